// The gradient of the value gather y = v[src] * (src >= 0) (code/lema/attention.py:146-158):
// gv[row, j] = sum of gy[row, i] over the queries i with src[row, i] = j.
//
// Bound: reading gy and src once and writing gv once. As tensor operations (mask, widened and
// expanded indices, zero fill, scatter-add) the same gradient makes six passes, the last of
// them one atomic per element, rounded to the value dtype at every addition. Here a workgroup
// owns R consecutive source rows of one row of streams and no float is ever added atomically:
//   scan    every index i after the rows' first position is read (a query only reads an
//           earlier position), and those that point into the rows are listed in LDS;
//   sort    the list is counted, scanned and placed by source row (integers, in LDS);
//   reduce  the sorted list is cut into equal runs, one per group of lanes (one lane per piece
//           of a value row, 8 rows in flight), each summed in fp32 in list order. A run's
//           first sum may belong to a source row that began in an earlier run; it goes to LDS
//           and the run where that row began adds it, so a source row that very many queries
//           read is spread over the workgroup.
// Every row of gv is written once, zeros included. A list that fills up before the scan ends is
// reduced at once and the rows then accumulate in gv (rounded once per list, in 16-bit types).
// The scan reads O(T^2 / R) indices from L2, 4 bytes each: at T = 100,000 and R = 1024 about
// 49 per index against the 48 to 256 bytes of its gy row. It counts 6144 indices behind one
// barrier before it lists them: with two barriers for every batch or two of 1024, one row of
// 131,072 positions (d_v 24 bf16) took 104 us where 39 are now.
//
// A missed query's row is multiplied by zero and added to source row 0: nothing, unless it holds
// an infinity or NaN, which make that column of gv[row, 0] NaN. A second kernel reads the missed
// rows and stores those NaNs, after the first has written the sums.
//
// Measured (MI355X), B2 H64 T8001 d_v 24 bf16 on projection views: 43 us and 17 us for the missed
// rows (48.8 and 18.7 with each row of streams on its own XCD), against 590 us for the tensor
// operations; B1 H8 T4096 d_v 64 fp32: 12.0 and 4.0 us against 88.
#include "lema_internal.h"

#include <hip/hip_fp16.h>

namespace lema {
namespace {

constexpr int kGgThreads = 256;
constexpr int kGgRows = 1024;            // most source rows per workgroup
constexpr int kGgBatch = 4 * kGgThreads; // indices of a 16-byte load by every thread
// Entries of the list: a list that is reduced early has no room for a batch, so it holds over 1536;
// every LDS array of 4 workgroups fits a CU's 160 KB.
constexpr int kGgList = 2560;
constexpr int kGgFlight = 8;             // gy rows in flight per group of lanes
constexpr int kGgSliceT = 16384;         // shorter rows' lists are short whoever reads what
constexpr int kGgSpan = 6;               // batches of indices whose loads are issued together
constexpr int kMissPositions = 256;      // positions per workgroup of the miss kernel

struct GradArgs {
  const uint8_t* gy;
  const int32_t* src;  // [N, T]
  uint8_t* gv;         // [N, T, dv]
  int64_t N, H, T;
  int64_t sb, sh, st;  // strides of gy, bytes
  int64_t row_bytes;
  int32_t pieces;      // pieces per value row, or a slice of one
  int32_t R, nch;      // source rows per workgroup, workgroups per row and slice
  int32_t slices;      // slices of a value row's columns, a workgroup each
  int32_t order;       // of the workgroups (gg_item)
  FastDiv pdiv;        // division by `pieces`
};

// (row, part) of workgroup v, of `parts` per row. Workgroup v runs on XCD v % 8.
//   kGgGroups  N a multiple of 64: rows 8g..8g+7 belong to XCD g % 8, which takes a part of all 8
//              back to back: where gy interleaves the rows (a projection view), their pieces of
//              each line are then read through one L2
//   kGgRowXcd  N a multiple of 8: row r runs on XCD r % 8, whose L2 keeps its indices
//   kGgSpread  any other N: a row's parts go round the XCDs. Bound to an XCD each, the rows left
//              8 - N of the XCDs idle for N < 8 (N = 1: all but 32 CUs)
// First parts first: they have the most indices to scan.
constexpr int kGgSpread = 0, kGgRowXcd = 1, kGgGroups = 2;
__device__ __forceinline__ void gg_item(int order, int64_t N, int parts, int v, int64_t& row, int& part) {
  if (order == kGgSpread) {
    part = v / static_cast<int>(N);
    row = v - part * static_cast<int>(N);
    return;
  }
  const int xcd = v % kNumXcd, k = v / kNumXcd;
  if (order == kGgGroups) {
    const int per = kNumXcd * parts;
    part = (k % per) / kNumXcd;
    row = (static_cast<int64_t>(k / per) * kNumXcd + xcd) * kNumXcd + (k % per) % kNumXcd;
  } else {
    part = k % parts;
    row = static_cast<int64_t>(k / parts) * kNumXcd + xcd;
  }
}

// VEC bytes of a row as 32-bit words (one 16-bit word for VEC = 2).
template <int VEC>
struct GgRaw {
  uint32_t w[VEC >= 4 ? VEC / 4 : 1];
};
template <int VEC>
__device__ __forceinline__ GgRaw<VEC> gg_load(const uint8_t* p) {
  GgRaw<VEC> r;
  if constexpr (VEC == 16) {
    const u32x4 v = *reinterpret_cast<const u32x4*>(p);
    r.w[0] = v.x; r.w[1] = v.y; r.w[2] = v.z; r.w[3] = v.w;
  } else if constexpr (VEC == 8) {
    const u32x2 v = *reinterpret_cast<const u32x2*>(p);
    r.w[0] = v.x; r.w[1] = v.y;
  } else if constexpr (VEC == 4) {
    r.w[0] = *reinterpret_cast<const uint32_t*>(p);
  } else {
    r.w[0] = *reinterpret_cast<const uint16_t*>(p);
  }
  return r;
}
template <int VEC>
__device__ __forceinline__ void gg_store(uint8_t* p, const GgRaw<VEC>& r) {
  if constexpr (VEC == 16)
    *reinterpret_cast<u32x4*>(p) = u32x4{r.w[0], r.w[1], r.w[2], r.w[3]};
  else if constexpr (VEC == 8)
    *reinterpret_cast<u32x2*>(p) = u32x2{r.w[0], r.w[1]};
  else if constexpr (VEC == 4)
    *reinterpret_cast<uint32_t*>(p) = r.w[0];
  else
    *reinterpret_cast<uint16_t*>(p) = static_cast<uint16_t>(r.w[0]);
}

template <int DTYPE>
__device__ __forceinline__ float gg_to_f32(uint32_t h) {
  if constexpr (DTYPE == LEMA_BF16) {
    return __uint_as_float(h << 16);
  } else {
    return __half2float(__ushort_as_half(static_cast<unsigned short>(h)));
  }
}
// Round to nearest even, NaN to a quiet NaN.
template <int DTYPE>
__device__ __forceinline__ uint32_t gg_from_f32(float f) {
  if constexpr (DTYPE == LEMA_BF16) {
    const uint32_t b = __float_as_uint(f);
    if ((b & 0x7F800000u) == 0x7F800000u && (b & 0x007FFFFFu) != 0) return 0x7FC0u;
    return (b + 0x7FFFu + ((b >> 16) & 1u)) >> 16;
  } else {
    return __half_as_ushort(__float2half_rn(f));
  }
}

template <int DTYPE, int VEC>
struct GgPiece {
  static constexpr int kElems = DTYPE == LEMA_F32 ? VEC / 4 : VEC / 2;
  static __device__ __forceinline__ void add(float (&acc)[kElems], const GgRaw<VEC>& r) {
#pragma unroll
    for (int k = 0; k < kElems; ++k) {
      if constexpr (DTYPE == LEMA_F32)
        acc[k] += __uint_as_float(r.w[k]);
      else
        acc[k] += gg_to_f32<DTYPE>((r.w[k >> 1] >> (16 * (k & 1))) & 0xFFFFu);
    }
  }
  static __device__ __forceinline__ GgRaw<VEC> round(const float (&acc)[kElems]) {
    GgRaw<VEC> r;
#pragma unroll
    for (int k = 0; k < (VEC >= 4 ? VEC / 4 : 1); ++k) {
      if constexpr (DTYPE == LEMA_F32) {
        r.w[k] = __float_as_uint(acc[k]);
      } else {
        r.w[k] = gg_from_f32<DTYPE>(acc[VEC >= 4 ? 2 * k : k]);
        if constexpr (VEC >= 4) r.w[k] |= gg_from_f32<DTYPE>(acc[2 * k + 1]) << 16;
      }
    }
    return r;
  }
  // Does element k hold an infinity or NaN?
  static __device__ __forceinline__ bool odd(const GgRaw<VEC>& r, int k) {
    if constexpr (DTYPE == LEMA_F32) return (r.w[k] & 0x7F800000u) == 0x7F800000u;
    const uint32_t e = DTYPE == LEMA_BF16 ? 0x7F80u : 0x7C00u;
    return ((r.w[k >> 1] >> (16 * (k & 1))) & e) == e;
  }
};

struct GradLds {
  alignas(16) int32_t list_i[kGgList];   // listed queries
  uint16_t list_j[kGgList];              // and the source rows they read, less the first
  int32_t perm_i[kGgList];               // the same sorted by source row
  uint16_t perm_j[kGgList];
  int32_t end[kGgRows];                  // counts, then cursors: where a source row's run ends
  int32_t wave_sum[kGgThreads / 64];
  int32_t incoming[3];                   // entries that the current span of indices adds
};
// A run's first sum when its row began in an earlier run, [element][thread]: the list's storage,
// dead once it is sorted.
static_assert(sizeof(int32_t) * kGgList >= sizeof(float) * 8 * kGgThreads, "the runs' first sums");

// 16-byte pieces take 155 registers, 3 workgroups per CU: held to 128 a few were spilled, and the
// scratch made every launch wait.
template <int DTYPE, int VEC>
__global__ __launch_bounds__(kGgThreads, VEC == 16 ? 3 : 4) void gather_grad_kernel(GradArgs a) {
  typedef GgPiece<DTYPE, VEC> P;
  constexpr int E = P::kElems;
  __shared__ GradLds s;
  const int t = threadIdx.x, lane = t & 63;
  int64_t row;
  int part_no;
  gg_item(a.order, a.N, a.nch * a.slices, blockIdx.x, row, part_no);
  const int64_t slice0 = static_cast<int64_t>(part_no % a.slices) * a.pieces * VEC;  // bytes
  const int64_t j0 = static_cast<int64_t>(part_no / a.slices) * a.R;
  const int rows = static_cast<int>(a.T - j0 < a.R ? a.T - j0 : a.R);
  const int32_t* src = a.src + row * a.T;
  const int64_t b = row / a.H, h = row - (row / a.H) * a.H;
  const uint8_t* gy = a.gy + b * a.sb + h * a.sh + slice0;
  uint8_t* gv = a.gv + (row * a.T + j0) * a.row_bytes + slice0;
  float* part = reinterpret_cast<float*>(s.list_i);

  bool accumulate = false;  // gv's rows hold earlier lists' sums
  // Sort the listed queries by source row and add their gy rows up (all threads).
  auto reduce_list = [&](int n, bool last) {
    __syncthreads();
    for (int x = t; x < kGgRows; x += kGgThreads) s.end[x] = 0;
    __syncthreads();
    for (int e = t; e < n; e += kGgThreads) atomicAdd(&s.end[s.list_j[e]], 1);
    __syncthreads();
    int c[kGgRows / kGgThreads], sum = 0;
#pragma unroll
    for (int u = 0; u < kGgRows / kGgThreads; ++u) {
      c[u] = s.end[t * (kGgRows / kGgThreads) + u];
      sum += c[u];
    }
    int inc = sum;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const int up = __shfl_up(inc, o);
      if (lane >= o) inc += up;
    }
    if (lane == 63) s.wave_sum[t >> 6] = inc;
    __syncthreads();
    int at = inc - sum;
    for (int w = 0; w < (t >> 6); ++w) at += s.wave_sum[w];
#pragma unroll
    for (int u = 0; u < kGgRows / kGgThreads; ++u) {
      s.end[t * (kGgRows / kGgThreads) + u] = at;
      at += c[u];
    }
    __syncthreads();
    for (int e = t; e < n; e += kGgThreads) {
      const int j = s.list_j[e];
      const int p = atomicAdd(&s.end[j], 1);
      s.perm_i[p] = s.list_i[e];
      s.perm_j[p] = static_cast<uint16_t>(j);
    }
    __syncthreads();  // sorted; end[j] is where row j's run ends, and the list is dead
    if (!accumulate) {  // rows no query reads (all rows, when more lists follow) start at zero
      const GgRaw<VEC> zero{};
      for (uint32_t x = t; x < static_cast<uint32_t>(rows) * a.pieces; x += kGgThreads) {
        const int j = static_cast<int>(a.pdiv.div(x));
        if (!last || s.end[j] == (j > 0 ? s.end[j - 1] : 0))
          gg_store<VEC>(gv + j * a.row_bytes + (x - static_cast<uint32_t>(j) * a.pieces) * VEC, zero);
      }
      if (!last) {
        accumulate = true;
        __syncthreads();
      }
    }
    for (int p0 = 0; p0 < a.pieces; p0 += kGgThreads) {  // columns of kGgThreads pieces
      const int pt = a.pieces - p0 < kGgThreads ? a.pieces - p0 : kGgThreads;
      const int G = kGgThreads / pt;
      const int g = t / pt, col = p0 + t - g * pt;
      const int per = (n + G - 1) / G;
      const int e0 = g * per < n ? g * per : n, e1 = e0 + per < n ? e0 + per : n;
      const uint8_t* gyc = gy + static_cast<int64_t>(col) * VEC;
      auto write = [&](int j, float (&acc)[E]) {
        uint8_t* to = gv + j * a.row_bytes + static_cast<int64_t>(col) * VEC;
        if (accumulate) P::add(acc, gg_load<VEC>(to));
        gg_store<VEC>(to, P::round(acc));
      };
      float acc[E];
#pragma unroll
      for (int u = 0; u < E; ++u) acc[u] = 0.0f;
      int cur = -1;
      bool pending = false;
      if (g < G && e0 < e1) {
        cur = s.perm_j[e0];
        bool head = e0 > 0 && s.perm_j[e0 - 1] == cur;  // the row began in an earlier run
        for (int e = e0; e < e1; e += kGgFlight) {
          GgRaw<VEC> raw[kGgFlight];
          int jj[kGgFlight];
#pragma unroll
          for (int u = 0; u < kGgFlight; ++u) {
            const int x = e + u < e1 ? e + u : e1 - 1;  // past the run: its last row again
            jj[u] = s.perm_j[x];
            raw[u] = gg_load<VEC>(gyc + static_cast<int64_t>(s.perm_i[x]) * a.st);
          }
#pragma unroll
          for (int u = 0; u < kGgFlight; ++u) {
            if (e + u >= e1) break;
            if (jj[u] != cur) {
              if (head) {
#pragma unroll
                for (int v = 0; v < E; ++v) part[v * kGgThreads + t] = acc[v];
              } else {
                write(cur, acc);
              }
#pragma unroll
              for (int v = 0; v < E; ++v) acc[v] = 0.0f;
              cur = jj[u];
              head = false;
            }
            P::add(acc, raw[u]);
          }
        }
        if (head) {
#pragma unroll
          for (int v = 0; v < E; ++v) part[v * kGgThreads + t] = acc[v];
        } else if (e1 < n && s.perm_j[e1] == cur) {
          pending = true;  // the row goes on in the next runs
        } else {
          write(cur, acc);
        }
      }
      __syncthreads();
      if (pending) {
        for (int g2 = g + 1; g2 < G && g2 * per < n && s.perm_j[g2 * per] == cur; ++g2)
#pragma unroll
          for (int v = 0; v < E; ++v) acc[v] += part[v * kGgThreads + t + (g2 - g) * pt];
        write(cur, acc);
      }
      __syncthreads();
    }
  };

  if (t < 3) s.incoming[t] = 0;
  __syncthreads();
  const uint32_t first_j = static_cast<uint32_t>(j0), n_j = static_cast<uint32_t>(rows);
  auto in = [&](int32_t x) { return static_cast<uint32_t>(x) - first_j < n_j; };  // a miss is no row either
  // four consecutive indices from i on, 16-byte aligned where they all lie in the row
  auto load4 = [&](int64_t i, int32_t (&x)[4]) {
    if (i >= 0 && i + 3 < a.T) {
      const u32x4 v = *reinterpret_cast<const u32x4*>(src + i);
      x[0] = v.x; x[1] = v.y; x[2] = v.z; x[3] = v.w;
    } else {
#pragma unroll
      for (int u = 0; u < 4; ++u) x[u] = i + u >= 0 && i + u < a.T ? src[i + u] : -1;
    }
  };
  // bit 4q + u: x[q][u] points into the rows
  auto mask_of = [&](const auto& x) {
    constexpr int Q = sizeof(x) / sizeof(x[0]);
    static_assert(4 * Q <= 32, "a bit each");
    uint32_t m = 0;
#pragma unroll
    for (int q = 0; q < Q; ++q)
#pragma unroll
      for (int u = 0; u < 4; ++u) m |= in(x[q][u]) ? 1u << (4 * q + u) : 0u;
    return m;
  };
  // The list's places of the indices of mask m: `before` those of the threads ahead of this one, in
  // all threads together `all`. A wavefront's places follow its turn at the counter, a thread's
  // those of the lanes below it.
  int turn = 0;
  auto places = [&](uint32_t m, int& before, int& all) {
    const int c = __popc(m);
    int inc = c;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const int up = __shfl_up(inc, o);
      if (lane >= o) inc += up;
    }
    int old = 0;
    if (lane == 63 && inc != 0) old = atomicAdd(&s.incoming[turn], inc);
    before = __shfl(old, 63) + inc - c;
    __syncthreads();
    all = s.incoming[turn];
    // the counter before this one: read before the last barrier, used after the next
    if (t == 0) s.incoming[turn == 0 ? 2 : turn - 1] = 0;
    turn = turn == 2 ? 0 : turn + 1;
  };
  auto list = [&](int64_t i0, const auto& x, uint32_t m, int p) {
    constexpr int Q = sizeof(x) / sizeof(x[0]);
    if (m == 0) return;
#pragma unroll
    for (int q = 0; q < Q; ++q)
#pragma unroll
      for (int u = 0; u < 4; ++u)
        if (m >> (4 * q + u) & 1u) {
          s.list_i[p] = static_cast<int32_t>(i0 + q * kGgBatch + 4 * t + u);
          s.list_j[p] = static_cast<uint16_t>(x[q][u] - static_cast<int32_t>(j0));
          ++p;
        }
  };
  // A span of indices is counted before it is listed, so one barrier tells whether it fits; one
  // that does not is listed by batches as far as there is room. (With a look at the list's
  // room for every batch or two, rows of 131,072 spent most of the scan in barriers.) Indices
  // at or before the first source row read rows below it, so the scan may begin up to three
  // early, on a 16-byte boundary.
  const int skew = static_cast<int>((reinterpret_cast<uintptr_t>(src + j0 + 1) & 15) / 4);
  int64_t i0 = j0 + 1 - skew;
  int listed = 0;  // entries of the list
  bool full;
  do {
    full = false;
    while (!full && i0 < a.T) {
      int32_t x[kGgSpan][4];
#pragma unroll
      for (int q = 0; q < kGgSpan; ++q) load4(i0 + q * kGgBatch + 4 * t, x[q]);
      const uint32_t m = mask_of(x);
      int before, more;
      places(m, before, more);
      if (listed + more <= kGgList) {
        list(i0, x, m, listed + before);
        listed += more;
        i0 += kGgSpan * kGgBatch;
        continue;
      }
      for (int q = 0; q < kGgSpan && !full && i0 < a.T; ++q) {
        int32_t y[1][4];
        load4(i0 + 4 * t, y[0]);
        const uint32_t my = mask_of(y);
        places(my, before, more);
        full = listed + more > kGgList;
        if (!full) {
          list(i0, y, my, listed + before);
          listed += more;
          i0 += kGgBatch;
        }
      }
    }
    reduce_list(listed, !full);
    listed = 0;
  } while (full);
}

// Missed queries: an infinity or NaN in such a row of gy makes its column of gv[row, 0] NaN
// (0 * inf). One workgroup per kMissPositions positions of a row; the sums are in place.
template <int DTYPE, int VEC>
__global__ __launch_bounds__(kGgThreads) void gather_grad_miss_kernel(GradArgs a, int32_t nch) {
  typedef GgPiece<DTYPE, VEC> P;
  __shared__ int32_t miss[kMissPositions];
  __shared__ int32_t count;
  const int t = threadIdx.x, lane = t & 63;
  int64_t row;
  int part_no;
  gg_item(a.order, a.N, nch, blockIdx.x, row, part_no);
  if (t == 0) count = 0;
  __syncthreads();
  const int64_t i = static_cast<int64_t>(part_no) * kMissPositions + t;
  const bool in = i < a.T && a.src[row * a.T + i] < 0;
  const unsigned long long bal = __ballot(in);
  int base = 0;
  if (lane == 0 && bal != 0) base = atomicAdd(&count, __popcll(bal));
  base = __shfl(base, 0);
  if (in) miss[base + __popcll(bal & ((1ull << lane) - 1ull))] = static_cast<int32_t>(i);
  __syncthreads();
  const int n = count;
  const int64_t b = row / a.H, h = row - (row / a.H) * a.H;
  const uint8_t* gy = a.gy + b * a.sb + h * a.sh;
  for (int p0 = 0; p0 < a.pieces; p0 += kGgThreads) {
    const int pt = a.pieces - p0 < kGgThreads ? a.pieces - p0 : kGgThreads;
    const int G = kGgThreads / pt;
    const int g = t / pt, col = p0 + t - g * pt;
    if (g >= G) continue;
    for (int e = g; e < n; e += kGgFlight * G) {
      GgRaw<VEC> raw[kGgFlight];
#pragma unroll
      for (int u = 0; u < kGgFlight; ++u) {
        const int x = e + u * G < n ? e + u * G : e;
        raw[u] = gg_load<VEC>(gy + static_cast<int64_t>(miss[x]) * a.st + static_cast<int64_t>(col) * VEC);
      }
#pragma unroll
      for (int u = 0; u < kGgFlight; ++u)
#pragma unroll
        for (int v = 0; v < P::kElems; ++v)
          if (P::odd(raw[u], v)) {
            uint8_t* to = a.gv + row * a.T * a.row_bytes + static_cast<int64_t>(col) * VEC;
            if constexpr (DTYPE == LEMA_F32)
              reinterpret_cast<uint32_t*>(to)[v] = 0x7FC00000u;
            else
              reinterpret_cast<uint16_t*>(to)[v] = DTYPE == LEMA_BF16 ? 0x7FC0u : 0x7E00u;
          }
    }
  }
}

template <int DTYPE, int VEC>
int launch_grad(GradArgs& a, hipStream_t st) {
  // While the launch has under 4 workgroups per CU: value rows in slices of at least 128 bytes (a
  // workgroup lists and sorts for its slice alone, but where all queries read a few source rows it
  // is one workgroup's loads that bound the launch: one row of 131,072 queries of the first
  // 3 rows, d_v 64 fp32, 1420 us whole, 1016 in two slices), then fewer source rows.
  const int32_t row_pieces = a.pieces;
  const FastDiv row_pdiv = a.pdiv;
  a.R = kGgRows;
  a.slices = 1;
  auto few = [&] { return a.N * ((a.T + a.R - 1) / a.R) * a.slices < 1024; };
  while (a.T >= kGgSliceT && a.pieces % 2 == 0 && a.pieces * VEC >= 256 && few()) {
    a.slices *= 2;
    a.pieces /= 2;
  }
  // and no more pieces than 32 bits count
  while (a.R > 64 && (few() || static_cast<int64_t>(a.R) * a.pieces >= (int64_t(1) << 31))) a.R /= 2;
  const int64_t nch = (a.T + a.R - 1) / a.R;
  const int64_t mch = (a.T + kMissPositions - 1) / kMissPositions;
  LEMA_REQUIRE(a.N < (int64_t(1) << 31) && a.N * mch < (int64_t(1) << 31) && a.N * nch * a.slices < (int64_t(1) << 31),
               "too many rows x positions");
  a.nch = static_cast<int32_t>(nch);
  a.pdiv = FastDiv(static_cast<uint32_t>(a.pieces));
  a.order = a.N % 64 == 0 ? kGgGroups : a.N % kNumXcd == 0 ? kGgRowXcd : kGgSpread;
  gather_grad_kernel<DTYPE, VEC><<<dim3(a.N * nch * a.slices), dim3(kGgThreads), 0, st>>>(a);
  if (int rc = launch_status("gather_grad_kernel")) return rc;
  a.pieces = row_pieces;
  a.pdiv = row_pdiv;
  gather_grad_miss_kernel<DTYPE, VEC>
      <<<dim3(a.N * mch), dim3(kGgThreads), 0, st>>>(a, static_cast<int32_t>(mch));
  return launch_status("gather_grad_miss_kernel");
}

template <int DTYPE>
int launch_grad_vec(GradArgs& a, int vec, hipStream_t st) {
  switch (vec) {
    case 16: return launch_grad<DTYPE, 16>(a, st);
    case 8: return launch_grad<DTYPE, 8>(a, st);
    case 4: return launch_grad<DTYPE, 4>(a, st);
    default:
      if constexpr (DTYPE != LEMA_F32) return launch_grad<DTYPE, 2>(a, st);
      set_error("internal: piece size %d", vec);
      return LEMA_BAD_ARG;
  }
}

}  // namespace
}  // namespace lema

using namespace lema;

extern "C" int lema_gather_grad(const void* gy, int32_t dtype, int64_t B, int64_t H, int64_t T,
                                int64_t dv, int64_t gy_sb, int64_t gy_sh, int64_t gy_st,
                                const int32_t* src, void* gv, void* stream) {
  clear_error();
  const int es = dtype_size(dtype);
  LEMA_REQUIRE(es > 0, "unknown value dtype %d", dtype);
  LEMA_REQUIRE(B >= 0 && H >= 0 && T >= 0 && dv >= 0, "negative shape");
  if (B * H * T * dv == 0) return LEMA_OK;
  LEMA_REQUIRE(T < (int64_t(1) << 30), "T=%lld exceeds the resolver's positions", (long long)T);
  LEMA_REQUIRE(gy != nullptr && src != nullptr && gv != nullptr && aligned(src, 4),
               "gy, src and gv must be device pointers");
  // the largest piece that divides the row and every offset of gy and gv
  int vec = 16;
  const int64_t rb = dv * es;
  while (vec > 1 && (rb % vec || gy_sb * es % vec || gy_sh * es % vec || gy_st * es % vec ||
                     !aligned(gy, vec) || !aligned(gv, vec)))
    vec /= 2;
  LEMA_REQUIRE(vec >= es, "gradient rows not aligned to the element size");
  // the gather's rows have at most 2^20 pieces, of 16 bytes at most: 2^23 of 2 bytes
  LEMA_REQUIRE(rb / vec <= (int64_t(1) << 23), "value rows too long (%lld elements)", (long long)dv);
  GradArgs a{};
  a.gy = static_cast<const uint8_t*>(gy);
  a.src = src;
  a.gv = static_cast<uint8_t*>(gv);
  a.N = B * H;
  a.H = H;
  a.T = T;
  a.sb = gy_sb * es;
  a.sh = gy_sh * es;
  a.st = gy_st * es;
  a.row_bytes = rb;
  a.pieces = static_cast<int32_t>(rb / vec);
  a.pdiv = FastDiv(static_cast<uint32_t>(a.pieces));
  hipStream_t st = static_cast<hipStream_t>(stream);
  switch (dtype) {
    case LEMA_F32: return launch_grad_vec<LEMA_F32>(a, vec, st);
    case LEMA_F16: return launch_grad_vec<LEMA_F16>(a, vec, st);
    default: return launch_grad_vec<LEMA_BF16>(a, vec, st);
  }
}
