// Skinny bf16 GEMMs on the matrix cores for decoding: Y[M, N] = X[M, K] . W[N, K]^T with few
// rows (M <= 32: one token of each of a batch of streams), the shape of every projection of a
// decode step (code/lema/model.py:168-179, 85-94, the head). Such a product reads W once and is
// bound by that read; a workgroup streams a block of 16 * CT rows of W with its 8 wavefronts
// splitting K, each wavefront running v_mfma_f32_16x16x32_bf16 on 16-byte fragments loaded
// straight from memory (no LDS staging: X is a few KB and stays in L2), and the partial sums
// are reduced through LDS.
//
// Epilogues (a launch can hold up to three weight segments over the same x, e.g. a layer's q,
// k and v projections):
//   plain   Y rounded to bf16, optionally added to a bf16 residual (the MLP's down projection
//           and the residual add of Block.forward, code/lema/model.py:229-232);
//   pack    the q or k projection straight to codes (code/lema/attention.py:82-97): bit j of a
//           head's code is (bf16(z_j) >= 0), the sign of the value the unfused path would have
//           stored -- the projection's output never goes to HBM. A block covers 16 columns and
//           writes the bytes of each code its columns hold (d a multiple of 8), or whole heads;
//   swiglu  silu(x . gate^T) * (x . up^T) with the same bf16 roundings as SwiGLU.forward's
//           ops (code/lema/model.py:85-94): the block computes 16 columns of both.
// A swiglu launch can also take the MLP's pre-norm (Block.forward's norm2 with the attention's
// residual add, code/lema/model.py:229-232): every block then forms the normalised rows
// itself, with the stand-alone norm kernel's arithmetic (norm_row.h), into LDS and multiplies
// those; block 0 also writes x + d, the MLP's residual. That saves the norm's launch. A q/k/v
// launch takes the attention's pre-norm the same way (norm1, no addend): batch-16 decode steps
// of the 24-layer LM went 1.428 -> 1.391 ms.
//
// Operand layout of v_mfma_f32_16x16x32_bf16 (checked on the device): lane l holds A row l%16
// and B column l%16, k = 8 * (l / 16) + j, j < 8; the result's register r of lane l is row
// 4 * (l / 16) + r, column l % 16.
#include <type_traits>

#include "lema_internal.h"
#include "norm_row.h"

namespace lema {
namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

constexpr int kSkThreads = 512;
constexpr int kSkWaves = kSkThreads / 64;
constexpr int kSkStepK = 32 * kSkWaves;  // row elements that give every wavefront one K-step
constexpr int kSkNormMaxK = 8 * kSkStepK;  // longest rows of a fused pre-norm, held in registers

// One weight segment of a launch: its blocks cover N output columns of x . w^T with one
// epilogue. A launch holds up to three segments sharing x (the q, k and v projections of a
// layer in one launch).
enum SkMode : int32_t { kSkPlain = 0, kSkPack = 1, kSkSwiglu = 2 };

struct SkSegment {
  const uint16_t* w;   // [N, K]
  const uint16_t* w2;  // swiglu: the up projection [N, K] (w is the gate)
  void* out;           // plain / swiglu: bf16 [M, ldy]; pack: codes
  const uint16_t* res; // plain: optional bf16 [M, ldy] residual, out = bf16(res + bf16(sum))
  int64_t ldy;
  int32_t N, mode, code_bytes;
};

// A product on few blocks leaves CUs idle, and each block's weight read is bound by what its
// CU keeps in flight (measured at M = 1, K = 1536: 96 and 192 blocks of 16 columns both take
// 3.9 us). A launch of plain segments only (16-column tiles) with at most kNarrowMaxN columns
// therefore takes blocks of 8 columns, the other half of each matrix-core tile idle. A launch
// with packed segments (q/k/v) already has three segments' blocks and keeps 16 columns.
constexpr int kNarrowCols = 8;
constexpr int kNarrowMaxN = 256 * kNarrowCols;

struct SkinnyArgs {
  const uint16_t* x;
  int64_t ldx, ldw;
  int32_t M, K;
  int32_t d, T;  // pack: bits per code (one head), positions per stream (row m = (b, t))
  int32_t nseg;
  SkSegment seg[3];
  // fused pre-norm (nw non-null): x is the residual stream, nd the addend (or null), rows of
  // K; the product's input is norm(x + nd) * nw, and ns receives x + nd (rows of K)
  const uint16_t* nd;
  const uint16_t* nw;
  uint16_t* ns;
  float eps;
};

// What the kernel gets of it: two lines of 64 bytes of arguments, the first one all that a plain
// product needs. The argument lines are cold at every launch, and the weights' loads wait for
// them (in five lines of 64 bytes, as they were before, every launch took 0.3 to 0.5 us more).
struct SkDevice {
  const uint16_t* x;
  const uint16_t* w;
  void* out;
  const uint16_t* add;   // plain: the residual or null; pre-norm: the addend or null
  uint32_t ldx8, ldw8;   // row strides of x and the weights, in 8 elements: their low 32 bits
  int32_t K, N;
  int64_t ldy;
  uint32_t flags;        // mode | segments << 2 | code bytes << 4 | columns per block << 8 | M << 16
                         // | the strides' next 5 bits << 22 (x) and << 27 (weights)
  int32_t blocks;        // of the first segment, and of the second
  const uint16_t* w1;    // the second segment's, or swiglu's up
  const uint16_t* w2;    // the third segment's: plain, Nv columns
  void* out1;
  void* out2;
  const uint16_t* nw;
  uint16_t* ns;
  float eps;
  int32_t d, T, Nv;
};
static_assert(sizeof(SkDevice) == 128, "two lines");

__device__ __forceinline__ uint32_t f32_to_bf16_bits(float f) {
  const uint32_t b = __float_as_uint(f);
  if ((b & 0x7F800000u) == 0x7F800000u && (b & 0x007FFFFFu) != 0) return 0x7FC0u;
  return (b + 0x7FFFu + ((b >> 16) & 1u)) >> 16;
}
__device__ __forceinline__ float bf16_bits_to_f32(uint32_t h) { return __uint_as_float(h << 16); }

// (bf16(z) >= 0) as a float comparison: -0 -> true, NaN -> false.
__device__ __forceinline__ bool bf16_nonneg(float z) {
  return bf16_bits_to_f32(f32_to_bf16_bits(z)) >= 0.0f;
}

// Exchanges the values of lanes 8 apart in each row of 16 lanes.
__device__ __forceinline__ u32x4 swap_halves(u32x4 v) {
  u32x4 r;
#pragma unroll
  for (int i = 0; i < 4; ++i)
    r[i] = static_cast<uint32_t>(__builtin_amdgcn_mov_dpp(static_cast<int>(v[i]), 0x128, 0xf, 0xf, true));
  return r;
}

// A block owns `cols` columns: 16 * CT, or 8 for a narrow plain segment (swiglu: 16 columns
// of the gate and the same 16 of up). kNorm: 0 = x as it is, 1 = norm(x), 2 = norm(x + nd).
//
// Bound: the block's weight read, by the bytes its CU has in flight. So no load is conditional:
// lanes without a column or row of their own, and steps past a wavefront's share, read
// in-bounds elements whose products nothing uses. With a load per branch the compiler waited
// for every load of a group of 4 steps before its products and issued the next group after
// them. U is the K-steps of a group (kHalf: pairs of steps). A wavefront whose share is more than
// a group (kMore) issues the next group's loads before the current one's products, so it has
// one to two groups in flight. With a pre-norm one group is all of its share (3, 4, 6 or 8 steps
// for K of up to 768, 1024, 1536 or 2048; gate and up beyond 1536 take two of 4, whose registers
// leave room for a second workgroup: K 1792, 16 rows 22.0 -> 18.6 us), and the weights' loads are
// issued before the pre-norm's arithmetic and arrive meanwhile. Steps past the share cost a load each, and a second
// group's registers keep other workgroups off the CU: K = 768, N = 50304 (3 steps) took
// 22.6 us at M = 1 and 42.6 at M = 17 with groups of 4 and room for two, 14.8 and 24.4 now
// (16.4 and 27.4 with every load conditional).
//
// kHalf: a narrow block (8 columns) of at most 8 rows loads a second K-step into the matrix
// tile's idle quarters: columns and rows 8..15 are the same columns and rows one step on. Half
// the load instructions (the lanes past the block's columns would repeat others' loads at the
// same cost). The second step is multiplied after the first, both operands' halves exchanged by
// data-parallel moves, so a column adds its products in the order of a full tile and its bits
// don't depend on how many rows the call has (the two steps summed apart and added at the
// end differed from that in the last places, and a decoder's logits with them).
//
// Measured, launches in a graph over weights from HBM, before and now: M = 1, K = 1536,
// N = 1536 4.60 and 3.71 us, N = 4096 5.49 and 4.71, N = 8192 8.26 and 6.92; K = 4096, N = 1536
// 6.96 and 5.16; M = 16, N = 8192 10.9 and 8.9. (Half-filled tiles whose steps were summed apart:
// 3.64 and 5.14.)
template <int MT, int CT, int kNorm, int U, bool kHalf, bool kMore>
__global__ __launch_bounds__(kSkThreads, MT * CT <= 2 && (kNorm != 0 ? U <= 6 : !kMore || U <= 4) ? 4 : 2) void skinny_kernel(SkDevice a) {
  constexpr int kSteps = (kSkStepK * U * (kMore ? 2 : 1) + 511) / 512;  // the norm's, of 512 elements
  static_assert(!kHalf || (MT == 1 && CT == 1 && kNorm == 0), "a half-filled tile");
  __shared__ float part[kSkWaves][MT * 16][CT * 16 + 1];
  extern __shared__ __align__(16) uint16_t xs[];  // kNorm: the normalised rows, stride K + 8
  const int M = (a.flags >> 16) & 0x3F, cols = (a.flags >> 8) & 0xFF, code_bytes = (a.flags >> 4) & 0xF;
  int mode = a.flags & 3, N = a.N, bid = blockIdx.x;
  const uint16_t* wbase = a.w;
  void* dst = a.out;
  if (((a.flags >> 2) & 3) == 3) {  // q, k and v
    const bool s1 = bid >= a.blocks, s2 = bid >= 2 * a.blocks;
    wbase = s2 ? a.w2 : s1 ? a.w1 : wbase;
    dst = s2 ? a.out2 : s1 ? a.out1 : dst;
    mode = s2 ? kSkPlain : mode;
    N = s2 ? a.Nv : N;
    bid -= s2 ? 2 * a.blocks : s1 ? a.blocks : 0;
  }
  const bool glu = mode == kSkSwiglu;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), l = threadIdx.x & 63;
  const int64_t ldx = (static_cast<int64_t>((a.flags >> 22) & 31) << 32 | a.ldx8) * 8;
  const int64_t ldw = (static_cast<int64_t>(a.flags >> 27) << 32 | a.ldw8) * 8;
  const int n0 = bid * cols;
  const int ksteps = a.K / 32;
  const int per = (ksteps + kSkWaves - 1) / kSkWaves;
  const int s0 = wave * per;
  const int s1 = s0 + per < ksteps ? s0 + per : ksteps;
  // the step (kHalf: the two steps) that loads past the share repeat
  const int last = s1 > (kHalf ? 2 : 1) ? s1 - (kHalf ? 2 : 1) : 0;
  constexpr int kGroup = kHalf ? 2 * U : U;  // K-steps of a group
  const int r16 = l & 15, kg = (l >> 4) * 8;

  const uint16_t* wp[CT];
#pragma unroll
  for (int ct = 0; ct < CT; ++ct) {
    // column of the block; a lane past the block's or the segment's columns takes its first
    const int c = kHalf ? r16 & 7 : glu ? r16 : 16 * ct + r16;
    const int n = c < cols && n0 + c < N ? n0 + c : n0;
    const uint16_t* base = (glu && ct == 1) ? a.w1 : wbase;
    wp[ct] = base + static_cast<int64_t>(n) * ldw + kg + (kHalf ? (r16 >> 3) * 32 : 0);
  }
  // fragments as four 32-bit words: carried through the loop below as bf16 vectors, the compiler
  // took them apart into elements and reused half of one fragment's registers for an address
  typedef u32x4 WFrag[U][CT];
  typedef u32x4 XFrag[U][MT];
  // the step that load u of the group at s begins with, in bounds
  auto step_at = [&](int s, int u) __attribute__((always_inline)) {
    if constexpr (kHalf) return s + 2 * u < last ? s + 2 * u : last;
    return s + u < s1 ? s + u : last;
  };
  auto load_w = [&](WFrag& f, int s) __attribute__((always_inline)) {
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int at = step_at(s, u) * 32;
#pragma unroll
      for (int ct = 0; ct < CT; ++ct) f[u][ct] = *reinterpret_cast<const u32x4*>(wp[ct] + at);
    }
  };
  WFrag wa;
  const uint16_t* xp[MT];
  if constexpr (kNorm != 0) {
    // rows m and m + 8 of x by wavefront m, into LDS (a stride of K + 8 puts the 16 rows a
    // fragment load reads in different banks)
    const int xst = a.K + 8;
    auto rows = [&](int m, auto issue) __attribute__((always_inline)) {
      const uint16_t* xr[2];
      const uint16_t* dr[2];
      uint16_t* sr[2];
      const int n = m + kSkWaves < M ? 2 : 1;
#pragma unroll
      for (int r = 0; r < 2; ++r) {
        const int64_t mr = m + r * kSkWaves < M ? m + r * kSkWaves : m;
        xr[r] = a.x + mr * ldx;
        dr[r] = kNorm == 2 ? a.add + mr * a.K : nullptr;
        sr[r] = kNorm == 2 && blockIdx.x == 0 ? a.ns + mr * a.K : nullptr;
      }
      auto put = [&](int r, int e, u32x4 h) __attribute__((always_inline)) {
        *reinterpret_cast<u32x4*>(xs + (m + r * kSkWaves) * xst + e) = h;
      };
      auto loaded = [&]() __attribute__((always_inline)) {
        if constexpr (decltype(issue)::value) {
          __builtin_amdgcn_sched_barrier(0);  // the rows' loads first: they are waited for first
          load_w(wa, s0);
          __builtin_amdgcn_sched_barrier(0);
        }
      };
      norm_rows<2, kSteps, kNorm == 2>(xr, dr, n, a.nw, a.eps, a.K, l, sr, loaded, put);
    };
    if (wave < M)
      rows(wave, std::true_type{});
    else
      load_w(wa, s0);
    if constexpr (MT == 2)
      if (wave + 2 * kSkWaves < M) rows(wave + 2 * kSkWaves, std::false_type{});
    __syncthreads();
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) {
      const int m = 16 * mt + r16;
      xp[mt] = xs + (m < M ? m : 0) * xst + kg;
    }
  } else {
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) {
      const int m = kHalf ? r16 & 7 : 16 * mt + r16;
      xp[mt] = a.x + static_cast<int64_t>(m < M ? m : 0) * ldx + kg + (kHalf ? (r16 >> 3) * 32 : 0);
    }
    load_w(wa, s0);
  }

  f32x4 acc[MT][CT];
#pragma unroll
  for (int mt = 0; mt < MT; ++mt)
#pragma unroll
    for (int ct = 0; ct < CT; ++ct) acc[mt][ct] = f32x4{0.f, 0.f, 0.f, 0.f};
  auto load_x = [&](XFrag& f, int s) __attribute__((always_inline)) {
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int at = step_at(s, u) * 32;
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) f[u][mt] = *reinterpret_cast<const u32x4*>(xp[mt] + at);
    }
  };
  auto product = [&](int mt, int ct, u32x4 x, u32x4 w) __attribute__((always_inline)) {
    acc[mt][ct] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, x), __builtin_bit_cast(bf16x8, w),
                                                          acc[mt][ct], 0, 0, 0);
  };
  // `end`: the share may end inside the group. Steps past it are left out, with x from memory; with
  // x from LDS they multiply zeros (both factors, so that a stray infinity adds nothing): a
  // branch would put each fragment's LDS read behind the product before it
  auto products = [&](WFrag& w, XFrag& x, int s, bool end) __attribute__((always_inline)) {
    if (kNorm != 0 && end) {
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const bool in = s + u < s1;
#pragma unroll
        for (int ct = 0; ct < CT; ++ct) w[u][ct] = in ? w[u][ct] : u32x4{0u, 0u, 0u, 0u};
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) x[u][mt] = in ? x[u][mt] : u32x4{0u, 0u, 0u, 0u};
      }
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      if constexpr (kHalf) {
        const int at = s + 2 * u;  // the same in every lane, as s1 and last
        // an odd share's last step was loaded as the second of its pair
        if (!end || (at < s1 && at <= last)) product(0, 0, x[u][0], w[u][0]);
        // the swaps take copies as far as the compiler knows: with both products reading the same
        // fragments it reused two of a fragment's registers before the first one had read them
        asm("" : "+v"(x[u][0]), "+v"(w[u][0]));
        if (!end || (at < s1 && (at + 1 < s1 || at > last))) product(0, 0, swap_halves(x[u][0]), swap_halves(w[u][0]));
      } else {
        if (kNorm == 0 && end && s + u >= s1) break;  // the same in every lane
#pragma unroll
        for (int mt = 0; mt < MT; ++mt)
#pragma unroll
          for (int ct = 0; ct < CT; ++ct) product(mt, ct, x[u][mt], w[u][ct]);
      }
    }
  };
  XFrag xa;
  load_x(xa, s0);
  if constexpr (!kMore) {
    // no load moves past this into the branch of the product that uses it
    if constexpr (kNorm == 0) asm volatile("" ::: "memory");
    products(wa, xa, s0, true);
  } else {
    WFrag wb;
    XFrag xb;
    int s = s0;
    for (;;) {  // two groups a trip, so that neither is copied
      if (s + kGroup >= s1) {
        products(wa, xa, s, true);
        break;
      }
      load_w(wb, s + kGroup);
      load_x(xb, s + kGroup);
      products(wa, xa, s, false);
      s += kGroup;
      if (s + kGroup >= s1) {
        products(wb, xb, s, true);
        break;
      }
      load_w(wa, s + kGroup);
      load_x(xa, s + kGroup);
      products(wb, xb, s, false);
      s += kGroup;
    }
  }
#pragma unroll
  for (int mt = 0; mt < MT; ++mt)
#pragma unroll
    for (int ct = 0; ct < CT; ++ct)
#pragma unroll
      for (int r = 0; r < 4; ++r) part[wave][16 * mt + 4 * (l >> 4) + r][16 * ct + r16] = acc[mt][ct][r];
  __syncthreads();

  constexpr int kRows = MT * 16, kCols = CT * 16;
  constexpr int kPer = (kRows * kCols + kSkThreads - 1) / kSkThreads;
  float sums[kPer];
#pragma unroll
  for (int i = 0; i < kPer; ++i) {
    const int e = threadIdx.x + i * kSkThreads;
    sums[i] = 0.f;
    if (e < kRows * kCols) {
      const int row = e / kCols, col = e - (e / kCols) * kCols;
#pragma unroll
      for (int wv = 0; wv < kSkWaves; ++wv) sums[i] += part[wv][row][col];
    }
  }
  if (mode == kSkPlain) {
    uint16_t* y = static_cast<uint16_t*>(dst);
#pragma unroll
    for (int i = 0; i < kPer; ++i) {
      const int e = threadIdx.x + i * kSkThreads;
      const int row = e / kCols, col = e - (e / kCols) * kCols;
      if (e < kRows * kCols && row < M && col < cols && n0 + col < N) {
        const int64_t at = static_cast<int64_t>(row) * a.ldy + n0 + col;
        uint32_t out = f32_to_bf16_bits(sums[i]);
        if (kNorm == 0 && a.add != nullptr) out = f32_to_bf16_bits(bf16_bits_to_f32(a.add[at]) + bf16_bits_to_f32(out));
        y[at] = static_cast<uint16_t>(out);
      }
    }
    return;
  }
  if constexpr (CT == 2) {
    if (glu) {  // out = silu(gate) * up, the silu rounded to bf16 first; up is 16 lanes on
      uint16_t* y = static_cast<uint16_t*>(dst);
#pragma unroll
      for (int i = 0; i < kPer; ++i) {
        const int e = threadIdx.x + i * kSkThreads;
        const int row = e / kCols, c = e % kCols;
        const float u = bf16_bits_to_f32(f32_to_bf16_bits(__shfl(sums[i], l | 16)));
        if (c >= 16 || row >= M || n0 + c >= N) continue;
        const float g = bf16_bits_to_f32(f32_to_bf16_bits(sums[i]));
        const float sl = bf16_bits_to_f32(f32_to_bf16_bits(g / (1.0f + expf(-g))));
        y[static_cast<int64_t>(row) * a.ldy + n0 + c] = static_cast<uint16_t>(f32_to_bf16_bits(sl * u));
      }
      return;
    }
  }
  if constexpr (CT == 1) {
    if (a.d % 8 == 0) {
      // Heads of whole bytes: a ballot gives a row's 16 bits to its 16 lanes, and the lanes of
      // columns 0 and 8 write a byte of a code each; the one with the head's last byte also
      // clears the code's bytes above d. (Through LDS, one thread put a row's bits together
      // from 16 reads, two barriers later.)
      const int H = N / a.d;
#pragma unroll
      for (int i = 0; i < kPer; ++i) {
        const int e = threadIdx.x + i * kSkThreads;
        const uint64_t bal = __ballot(bf16_nonneg(sums[i]));
        const int row = e / kCols, c = e % kCols, n = n0 + c;
        if (e >= kRows * kCols || (c & 7) != 0 || row >= M || n >= N) continue;
        const int h = n / a.d, k = (n - h * a.d) / 8;
        const int b = row / a.T, t = row - b * a.T;
        uint8_t* w8 = static_cast<uint8_t*>(dst) + ((static_cast<int64_t>(b) * H + h) * a.T + t) * code_bytes;
        w8[k] = static_cast<uint8_t>(bal >> l);
        if (8 * k + 8 == a.d)
          for (int z = k + 1; z < code_bytes; ++z) w8[z] = 0;
      }
      return;
    }
  }
  __syncthreads();  // every partial is read: the block's sums go to part[0]
#pragma unroll
  for (int i = 0; i < kPer; ++i) {
    const int e = threadIdx.x + i * kSkThreads;
    if (e < kRows * kCols) part[0][e / kCols][e - (e / kCols) * kCols] = sums[i];
  }
  __syncthreads();
  // whole heads of other widths
  const int H = N / a.d;
  const int h0 = n0 / a.d;
  const int h1 = min((n0 + cols - 1) / a.d, H - 1);
  const int nh = h1 - h0 + 1;
  for (int e = threadIdx.x; e < kRows * nh; e += kSkThreads) {
    const int row = e / nh, h = h0 + (e - (e / nh) * nh);
    if (row >= M) continue;
    const int c_lo = max(n0, h * a.d), c_hi = min(n0 + cols, (h + 1) * a.d);
    uint64_t code = 0;
    for (int n = c_lo; n < c_hi; ++n)
      if (bf16_nonneg(part[0][row][n - n0])) code |= uint64_t(1) << (n - h * a.d);
    const int64_t b = row / a.T, t = row - (row / a.T) * a.T;
    const int64_t at = (b * H + h) * a.T + t;
    if (code_bytes == 4)
      static_cast<uint32_t*>(dst)[at] = static_cast<uint32_t>(code);
    else
      static_cast<uint64_t*>(dst)[at] = code;
  }
}

template <int CT>
int launch_skinny(SkinnyArgs& a, hipStream_t st) {
  bool all_plain = true;
  for (int j = 0; j < a.nseg; ++j) all_plain = all_plain && a.seg[j].mode == kSkPlain;
  const SkSegment& s0 = a.seg[0];
  const bool narrow = CT == 1 && all_plain && s0.N <= kNarrowMaxN;
  const int cols = s0.mode == kSkSwiglu ? 16 : narrow ? kNarrowCols : 16 * CT;
  int blocks = 0;
  for (int i = 0; i < a.nseg; ++i) blocks += (a.seg[i].N + cols - 1) / cols;
  SkDevice g{};
  g.x = a.x;
  g.w = s0.w;
  g.out = s0.out;
  g.add = a.nw != nullptr ? a.nd : s0.res;
  // 37 bits hold any stride that has a second row in memory; that of a single row is never used
  g.ldx8 = static_cast<uint32_t>(a.ldx / 8);
  g.ldw8 = static_cast<uint32_t>(a.ldw / 8);
  g.K = a.K;
  g.N = s0.N;
  g.ldy = a.nseg == 3 ? a.seg[2].ldy : s0.ldy;
  g.flags = static_cast<uint32_t>(s0.mode) | static_cast<uint32_t>(a.nseg) << 2 |
            static_cast<uint32_t>(s0.code_bytes) << 4 | static_cast<uint32_t>(cols) << 8 |
            static_cast<uint32_t>(a.M) << 16 | static_cast<uint32_t>(a.ldx >> 35 & 31) << 22 |
            static_cast<uint32_t>(a.ldw >> 35 & 31) << 27;
  g.blocks = (s0.N + cols - 1) / cols;
  g.w1 = a.nseg == 3 ? a.seg[1].w : s0.w2;
  g.w2 = a.seg[2].w;
  g.out1 = a.seg[1].out;
  g.out2 = a.seg[2].out;
  g.nw = a.nw;
  g.ns = a.ns;
  g.eps = a.eps;
  g.d = a.d;
  g.T = a.T;
  g.Nv = a.seg[2].N;
  const dim3 grid(blocks), block(kSkThreads);
  const size_t lds = a.nw != nullptr ? static_cast<size_t>(a.M) * (a.K + 8) * sizeof(uint16_t) : 0;
  void (*kernel)(SkDevice) = nullptr;
  const int per = (a.K / 32 + kSkWaves - 1) / kSkWaves;  // K-steps of a wavefront
  if (a.nw != nullptr) {  // the normalised rows in LDS (checked to fit by the entry point)
    auto pick_u = [&](auto mt, auto norm) {
      constexpr int MT = decltype(mt)::value, kNorm = decltype(norm)::value;
      if constexpr (CT <= 2) {  // whole-head codes of other widths (CT 3) are rare: two sizes
        if (per <= 3) return skinny_kernel<MT, CT, kNorm, 3, false, false>;
        if (per <= 4) return skinny_kernel<MT, CT, kNorm, 4, false, false>;
      }
      if (per <= 6) return skinny_kernel<MT, CT, kNorm, 6, false, false>;
      if constexpr (CT == 2)
        return skinny_kernel<MT, CT, kNorm, 4, false, true>;
      else
        return skinny_kernel<MT, CT, kNorm, 8, false, false>;
    };
    auto pick = [&](auto mt) {
      return a.nd != nullptr ? pick_u(mt, std::integral_constant<int, 2>{}) : pick_u(mt, std::integral_constant<int, 1>{});
    };
    kernel = a.M <= 16 ? pick(std::integral_constant<int, 1>{}) : pick(std::integral_constant<int, 2>{});
  } else {
    // A share of up to 6 steps in one group; longer ones in groups of 4, or of 6 where that divides
    // the share as well and two groups' registers still leave room for a second workgroup.
    auto waste = [](int n, int u) { return (n + u - 1) / u * u - n; };  // loads past a share of n
    auto pick = [&](auto mt) {
      constexpr int MT = decltype(mt)::value;
      if constexpr (CT <= 2) {
        if (per <= 2) return skinny_kernel<MT, CT, 0, 2, false, false>;
      }
      if (per <= 3) return skinny_kernel<MT, CT, 0, 3, false, false>;
      if (per <= 4) return skinny_kernel<MT, CT, 0, 4, false, false>;
      if (per <= 6) return skinny_kernel<MT, CT, 0, 6, false, false>;
      if constexpr (MT * CT == 1) {
        if (waste(per, 6) <= waste(per, 4)) return skinny_kernel<MT, CT, 0, 6, false, true>;
      }
      return skinny_kernel<MT, CT, 0, 4, false, true>;
    };
    kernel = a.M <= 16 ? pick(std::integral_constant<int, 1>{}) : pick(std::integral_constant<int, 2>{});
    if constexpr (CT == 1) {
      const int half = (per + 1) / 2;  // pairs of steps
      if (narrow && a.M <= 8 && a.K >= 64)
        kernel = half <= 2   ? skinny_kernel<1, 1, 0, 2, true, false>
                 : half <= 3 ? skinny_kernel<1, 1, 0, 3, true, false>
                 : half <= 4 ? skinny_kernel<1, 1, 0, 4, true, false>
                 : waste(half, 4) <= waste(half, 3) ? skinny_kernel<1, 1, 0, 4, true, true>
                                                    : skinny_kernel<1, 1, 0, 3, true, true>;
    }
  }
  kernel<<<grid, block, lds, st>>>(g);
  return launch_status("skinny_kernel");
}

int launch_ct(SkinnyArgs& a, int ct, hipStream_t st) {
  switch (ct) {
    case 1: return launch_skinny<1>(a, st);
    case 2: return launch_skinny<2>(a, st);
    default: return launch_skinny<3>(a, st);
  }
}

int check_skinny(const void* x, int64_t ldx, int64_t ldw, int64_t M, int64_t K) {
  LEMA_REQUIRE(M >= 1 && M <= 32, "skinny products take 1..32 rows, got %lld", (long long)M);
  LEMA_REQUIRE(K >= 32 && K % 32 == 0 && K < (int64_t(1) << 30), "K=%lld must be a multiple of 32",
               (long long)K);
  LEMA_REQUIRE(ldx >= K && ldw >= K && ldx % 8 == 0 && ldw % 8 == 0,
               "row strides must be >= K and multiples of 8");
  LEMA_REQUIRE(x != nullptr && aligned(x, 16), "x must be a 16-byte aligned device pointer");
  return LEMA_OK;
}

int check_weight(const void* w, int64_t N) {
  LEMA_REQUIRE(w != nullptr && aligned(w, 16), "weights must be 16-byte aligned device pointers");
  LEMA_REQUIRE(N >= 1 && N < (int64_t(1) << 30), "N=%lld", (long long)N);
  return LEMA_OK;
}

// Column tiles per block for codes of d bits: one (16 columns, a head split over blocks
// writes its bytes from each) when d is a multiple of 8, else the least multiple of 16 (up to
// 48) holding whole heads, or 0. More blocks of fewer weight rows: the q and k projections of
// 64-bit heads ran on 24 blocks of 64 rows each.
int pack_ct(int32_t d) {
  if (d % 8 == 0) return 1;
  for (int c = 1; c <= 3; ++c)
    if ((16 * c) % d == 0) return c;
  return 0;
}

}  // namespace
}  // namespace lema

using namespace lema;

extern "C" int lema_skinny_gemm_bf16(const void* x, int64_t ldx, const void* w, int64_t ldw,
                                     void* y, int64_t ldy, int64_t M, int64_t N, int64_t K,
                                     void* stream) {
  clear_error();
  if (int rc = check_skinny(x, ldx, ldw, M, K)) return rc;
  if (int rc = check_weight(w, N)) return rc;
  LEMA_REQUIRE(y != nullptr && ldy >= N, "bad output");
  SkinnyArgs a{};
  a.x = static_cast<const uint16_t*>(x);
  a.ldx = ldx;
  a.ldw = ldw;
  a.M = static_cast<int32_t>(M);
  a.K = static_cast<int32_t>(K);
  a.nseg = 1;
  a.seg[0] = SkSegment{static_cast<const uint16_t*>(w), nullptr, y, nullptr, ldy,
                       static_cast<int32_t>(N), kSkPlain, 0};
  return launch_ct(a, 1, static_cast<hipStream_t>(stream));
}

extern "C" int lema_skinny_gemm_add_bf16(const void* x, int64_t ldx, const void* w, int64_t ldw,
                                         const void* r, void* y, int64_t ldy, int64_t M, int64_t N,
                                         int64_t K, void* stream) {
  clear_error();
  if (int rc = check_skinny(x, ldx, ldw, M, K)) return rc;
  if (int rc = check_weight(w, N)) return rc;
  LEMA_REQUIRE(y != nullptr && r != nullptr && ldy >= N, "bad output or residual");
  SkinnyArgs a{};
  a.x = static_cast<const uint16_t*>(x);
  a.ldx = ldx;
  a.ldw = ldw;
  a.M = static_cast<int32_t>(M);
  a.K = static_cast<int32_t>(K);
  a.nseg = 1;
  a.seg[0] = SkSegment{static_cast<const uint16_t*>(w), nullptr, y,
                       static_cast<const uint16_t*>(r), ldy, static_cast<int32_t>(N), kSkPlain, 0};
  return launch_ct(a, 1, static_cast<hipStream_t>(stream));
}

extern "C" int lema_skinny_pack_bf16(const void* x, int64_t ldx, const void* w, int64_t ldw,
                                     int64_t M, int64_t N, int64_t K, int32_t d, int64_t T,
                                     void* codes, int32_t code_bytes, void* stream) {
  clear_error();
  if (int rc = check_skinny(x, ldx, ldw, M, K)) return rc;
  if (int rc = check_weight(w, N)) return rc;
  LEMA_REQUIRE(d >= 1 && d <= 64 && N % d == 0, "head width %d must divide N=%lld", d, (long long)N);
  LEMA_REQUIRE(code_bytes == 8 || (code_bytes == 4 && d <= 32), "code_bytes %d for %d-bit codes",
               code_bytes, d);
  LEMA_REQUIRE(T >= 1 && M % T == 0, "rows %lld are not streams x %lld positions", (long long)M,
               (long long)T);
  LEMA_REQUIRE(codes != nullptr && aligned(codes, code_bytes), "bad code pointer");
  const int ct = pack_ct(d);
  LEMA_REQUIRE(ct > 0, "head width %d does not tile 16..64 columns", d);
  SkinnyArgs a{};
  a.x = static_cast<const uint16_t*>(x);
  a.ldx = ldx;
  a.ldw = ldw;
  a.M = static_cast<int32_t>(M);
  a.K = static_cast<int32_t>(K);
  a.d = d;
  a.T = static_cast<int32_t>(T);
  a.nseg = 1;
  a.seg[0] = SkSegment{static_cast<const uint16_t*>(w), nullptr, codes, nullptr, 0,
                       static_cast<int32_t>(N), kSkPack, code_bytes};
  return launch_ct(a, ct, static_cast<hipStream_t>(stream));
}

namespace lema {
namespace {

// The checks and the three segments of a q/k/v launch; `ct` receives its block width.
int qkv_args(SkinnyArgs& a, int& ct, const void* x, int64_t ldx, const void* wq, const void* wk,
             const void* wv, int64_t ldw, int64_t M, int64_t Nqk, int64_t Nv, int64_t K,
             int32_t d, int64_t T, void* qcodes, void* kcodes, int32_t code_bytes, void* v) {
  if (int rc = check_skinny(x, ldx, ldw, M, K)) return rc;
  if (int rc = check_weight(wq, Nqk)) return rc;
  if (int rc = check_weight(wk, Nqk)) return rc;
  if (int rc = check_weight(wv, Nv)) return rc;
  LEMA_REQUIRE(d >= 1 && d <= 64 && Nqk % d == 0, "head width %d must divide %lld", d,
               (long long)Nqk);
  LEMA_REQUIRE(code_bytes == 8 || (code_bytes == 4 && d <= 32), "code_bytes %d for %d-bit codes",
               code_bytes, d);
  LEMA_REQUIRE(T >= 1 && M % T == 0, "rows %lld are not streams x %lld positions", (long long)M,
               (long long)T);
  LEMA_REQUIRE(qcodes && kcodes && aligned(qcodes, code_bytes) && aligned(kcodes, code_bytes) &&
                   v != nullptr, "bad output pointer");
  ct = pack_ct(d);
  LEMA_REQUIRE(ct > 0, "head width %d does not tile 16..64 columns", d);
  a.x = static_cast<const uint16_t*>(x);
  a.ldx = ldx;
  a.ldw = ldw;
  a.M = static_cast<int32_t>(M);
  a.K = static_cast<int32_t>(K);
  a.d = d;
  a.T = static_cast<int32_t>(T);
  a.nseg = 3;
  a.seg[0] = SkSegment{static_cast<const uint16_t*>(wq), nullptr, qcodes, nullptr, 0,
                       static_cast<int32_t>(Nqk), kSkPack, code_bytes};
  a.seg[1] = SkSegment{static_cast<const uint16_t*>(wk), nullptr, kcodes, nullptr, 0,
                       static_cast<int32_t>(Nqk), kSkPack, code_bytes};
  a.seg[2] = SkSegment{static_cast<const uint16_t*>(wv), nullptr, v, nullptr, Nv,
                       static_cast<int32_t>(Nv), kSkPlain, 0};
  return LEMA_OK;
}

}  // namespace
}  // namespace lema

extern "C" int lema_skinny_qkv_bf16(const void* x, int64_t ldx, const void* wq, const void* wk,
                                    const void* wv, int64_t ldw, int64_t M, int64_t Nqk,
                                    int64_t Nv, int64_t K, int32_t d, int64_t T, void* qcodes,
                                    void* kcodes, int32_t code_bytes, void* v, void* stream) {
  clear_error();
  SkinnyArgs a{};
  int ct = 0;
  if (int rc = qkv_args(a, ct, x, ldx, wq, wk, wv, ldw, M, Nqk, Nv, K, d, T, qcodes, kcodes,
                        code_bytes, v))
    return rc;
  return launch_ct(a, ct, static_cast<hipStream_t>(stream));
}

// The attention's pre-norm inside the q/k/v launch (Block.gpu_pre: norm1, then the
// projections, code/lema/model.py:224-227): every block normalises the rows of x (contiguous,
// K elements) into LDS with the stand-alone norm kernel's arithmetic and multiplies those, so
// the codes and v equal lema_rmsnorm_bf16 followed by lema_skinny_qkv_bf16 with one launch
// fewer.
extern "C" int lema_skinny_norm_qkv_bf16(const void* x, const void* nw, float eps,
                                         const void* wq, const void* wk, const void* wv,
                                         int64_t ldw, int64_t M, int64_t Nqk, int64_t Nv,
                                         int64_t K, int32_t d, int64_t T, void* qcodes,
                                         void* kcodes, int32_t code_bytes, void* v,
                                         void* stream) {
  clear_error();
  SkinnyArgs a{};
  int ct = 0;
  if (int rc = qkv_args(a, ct, x, K, wq, wk, wv, ldw, M, Nqk, Nv, K, d, T, qcodes, kcodes,
                        code_bytes, v))
    return rc;
  LEMA_REQUIRE(K <= kSkNormMaxK, "the fused norm takes rows of at most %d elements, got K=%lld",
               kSkNormMaxK, (long long)K);
  // LDS: the rows (M x (K + 8) bf16) next to the partial sums (8 x 16 or 32 rows x 16 ct + 1)
  const int64_t lds = M * (K + 8) * 2 + kSkWaves * (M <= 16 ? 16 : 32) * (16 * ct + 1) * 4;
  LEMA_REQUIRE(lds <= 160 * 1024, "%lld rows of %lld do not fit the LDS of a workgroup",
               (long long)M, (long long)K);
  LEMA_REQUIRE(nw != nullptr && aligned(nw, 16), "norm weight must be a 16-byte aligned device pointer");
  a.nd = nullptr;
  a.nw = static_cast<const uint16_t*>(nw);
  a.ns = nullptr;
  a.eps = eps;
  return launch_ct(a, ct, static_cast<hipStream_t>(stream));
}

extern "C" int lema_skinny_swiglu_bf16(const void* x, int64_t ldx, const void* wg, const void* wu,
                                       int64_t ldw, int64_t M, int64_t N, int64_t K, void* out,
                                       void* stream) {
  clear_error();
  if (int rc = check_skinny(x, ldx, ldw, M, K)) return rc;
  if (int rc = check_weight(wg, N)) return rc;
  if (int rc = check_weight(wu, N)) return rc;
  LEMA_REQUIRE(out != nullptr, "bad output pointer");
  SkinnyArgs a{};
  a.x = static_cast<const uint16_t*>(x);
  a.ldx = ldx;
  a.ldw = ldw;
  a.M = static_cast<int32_t>(M);
  a.K = static_cast<int32_t>(K);
  a.nseg = 1;
  a.seg[0] = SkSegment{static_cast<const uint16_t*>(wg), static_cast<const uint16_t*>(wu), out,
                       nullptr, N, static_cast<int32_t>(N), kSkSwiglu, 0};
  return launch_ct(a, 2, static_cast<hipStream_t>(stream));
}

extern "C" int lema_skinny_norm_swiglu_bf16(const void* x, const void* d, const void* nw,
                                            float eps, void* x_out, const void* wg,
                                            const void* wu, int64_t ldw, int64_t M, int64_t N,
                                            int64_t K, void* out, void* stream) {
  clear_error();
  if (int rc = check_skinny(x, K, ldw, M, K)) return rc;
  if (int rc = check_weight(wg, N)) return rc;
  if (int rc = check_weight(wu, N)) return rc;
  LEMA_REQUIRE(out != nullptr, "bad output pointer");
  LEMA_REQUIRE(K <= kSkNormMaxK, "the fused norm takes rows of at most %d elements, got K=%lld",
               kSkNormMaxK, (long long)K);
  // LDS: the rows (M x (K + 8) bf16) next to the partial sums (8 x 16 or 32 rows x 33 floats)
  const int64_t lds = M * (K + 8) * 2 + kSkWaves * (M <= 16 ? 16 : 32) * 33 * 4;
  LEMA_REQUIRE(lds <= 160 * 1024, "%lld rows of %lld do not fit the LDS of a workgroup",
               (long long)M, (long long)K);
  LEMA_REQUIRE(nw != nullptr && aligned(nw, 16), "norm weight must be a 16-byte aligned device pointer");
  LEMA_REQUIRE(d == nullptr || (aligned(d, 16) && x_out != nullptr && aligned(x_out, 16) &&
                                x_out != x && x_out != d),
               "the addend needs a 16-byte aligned output for x + d that is neither input");
  SkinnyArgs a{};
  a.x = static_cast<const uint16_t*>(x);
  a.ldx = K;
  a.ldw = ldw;
  a.M = static_cast<int32_t>(M);
  a.K = static_cast<int32_t>(K);
  a.nseg = 1;
  a.seg[0] = SkSegment{static_cast<const uint16_t*>(wg), static_cast<const uint16_t*>(wu), out,
                       nullptr, N, static_cast<int32_t>(N), kSkSwiglu, 0};
  a.nd = static_cast<const uint16_t*>(d);
  a.nw = static_cast<const uint16_t*>(nw);
  a.ns = static_cast<uint16_t*>(x_out);
  a.eps = eps;
  return launch_ct(a, 2, static_cast<hipStream_t>(stream));
}
