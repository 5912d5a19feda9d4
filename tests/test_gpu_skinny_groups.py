"""The skinny products where their load groups, tile halves and epilogues can go wrong: K shares
that end inside a group, wavefronts without a share, up to 8 and more rows (a half-filled tile
holds a second K-step up to 8), infinities past a share's end, heads split over blocks at every
byte. Needs a GPU."""
import pytest
import torch

from latest_exact_match_attention_amd import _lib

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def dev():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    return torch.device("cuda", 0)


def _product(x, w):
    M, K = x.shape
    y = torch.empty((M, w.shape[0]), dtype=x.dtype, device=x.device)
    _lib.check(_lib.lib().lema_skinny_gemm_bf16(
        x.data_ptr(), K, w.data_ptr(), K, y.data_ptr(), w.shape[0], M, w.shape[0], K,
        _lib.stream_of(x)))
    return y


@pytest.mark.parametrize("M", [1, 7, 8, 9, 16, 17, 32])
@pytest.mark.parametrize("N", [5, 24, 2048, 2056])
@pytest.mark.parametrize("K", [32, 64, 96, 448, 768, 1536, 1568, 1792, 3072, 4096, 6400])
def test_shares(dev, M, N, K):
    g = torch.Generator(device=dev).manual_seed(M + N + K)
    x = torch.randn((M, K), device=dev, generator=g).to(torch.bfloat16)
    w = (torch.randn((N, K), device=dev, generator=g) * K ** -0.5).to(torch.bfloat16)
    ref = x.double() @ w.double().T
    size = x.double().abs() @ w.double().abs().T
    # one rounding to bf16, and fp32 sums of K products
    bound = 2.0 ** -8 * ref.abs() + K * 2.0 ** -24 * size
    assert float(((_product(x, w).double() - ref).abs() - bound).max()) <= 0.0


@pytest.mark.parametrize("K", [32, 64, 96, 256, 288, 512, 768, 1536, 1568, 2816, 4096, 6144])
@pytest.mark.parametrize("N", [5, 24, 1536, 2048])
def test_bits_do_not_depend_on_the_other_rows(dev, N, K):
    """A row's products are added in one order, whatever the number of rows: up to 8 of them in a
    half-filled tile, 9 and more in a full one, 17 and more in two."""
    g = torch.Generator(device=dev).manual_seed(N + K)
    x = torch.randn((17, K), device=dev, generator=g).to(torch.bfloat16)
    w = (torch.randn((N, K), device=dev, generator=g) * K ** -0.5).to(torch.bfloat16)
    want = _product(x[:9], w)
    for M in (1, 3, 8):
        assert torch.equal(_product(x[:M].contiguous(), w), want[:M]), M
    assert torch.equal(_product(x, w)[:9], want)


def test_an_infinity_stays_in_its_products(dev):
    """An infinity in the last column of x or a weight touches its own row or column alone."""
    for K in (1536, 1792, 2048):
        x = torch.ones((3, K), device=dev, dtype=torch.bfloat16)
        w = torch.ones((64, K), device=dev, dtype=torch.bfloat16)
        x[1, K - 1] = float("inf")
        w[5, K - 1] = float("-inf")
        y = _product(x, w).float()
        want = x.float() @ w.float().T
        assert torch.equal(torch.isnan(y), torch.isnan(want))
        assert torch.equal(y.nan_to_num(1.0, 2.0, 3.0), want.nan_to_num(1.0, 2.0, 3.0))


@pytest.mark.parametrize("M", [1, 8, 16, 31])
@pytest.mark.parametrize("d,cb", [(8, 4), (24, 4), (24, 8), (32, 4), (40, 8), (56, 8), (64, 8), (4, 4), (12, 8)])
def test_code_bytes(dev, M, d, cb):
    """Every byte of a code, those above d cleared, for heads that blocks split and hold."""
    H, K = 6, 256
    g = torch.Generator(device=dev).manual_seed(d + M)
    # integer products: the signs are exact
    x = torch.randint(-3, 4, (M, K), device=dev, generator=g).to(torch.bfloat16)
    w = torch.randint(-3, 4, (H * d, K), device=dev, generator=g).to(torch.bfloat16)
    z = x.double() @ w.double().T
    want = ((z.view(M, H, d) >= 0).long() << torch.arange(d, device=dev)).sum(-1).t()
    codes = torch.full((H, M), -1, dtype=torch.int32 if cb == 4 else torch.int64, device=dev)
    _lib.check(_lib.lib().lema_skinny_pack_bf16(x.data_ptr(), K, w.data_ptr(), K, M, H * d, K, d, M,
                                                codes.data_ptr(), cb, _lib.stream_of(x)))
    got = codes.long() & 0xFFFFFFFF if cb == 4 else codes
    assert torch.equal(got, want)


@pytest.mark.parametrize("K", [32, 256, 768, 800, 1024, 1056, 1536, 1568, 2048])
@pytest.mark.parametrize("M", [1, 9, 17])
@pytest.mark.parametrize("with_d", [False, True])
def test_norm_shares(dev, K, M, with_d):
    """A fused pre-norm's product at every size of its load group, each from its shortest to its
    longest rows, against the norm in 64 bits and the product of its bf16 rows in fp32 sums."""
    g = torch.Generator(device=dev).manual_seed(K + M)
    x, d = (torch.randn((M, K), device=dev, generator=g).to(torch.bfloat16) for _ in range(2))
    nw = (1 + 0.1 * torch.randn(K, device=dev, generator=g)).to(torch.bfloat16)
    wg, wu = ((torch.randn((48, K), device=dev, generator=g) * K ** -0.5).to(torch.bfloat16) for _ in range(2))
    out, h, xo = (torch.empty(s, device=dev, dtype=torch.bfloat16) for s in ((M, 48), (M, K), (M, K)))
    L, st, dp = _lib.lib(), _lib.stream_of(x), d.data_ptr() if with_d else None
    _lib.check(L.lema_skinny_norm_swiglu_bf16(x.data_ptr(), dp, nw.data_ptr(), 1e-5, xo.data_ptr(), wg.data_ptr(),
                                              wu.data_ptr(), K, M, 48, K, out.data_ptr(), st))
    _lib.check(L.lema_rmsnorm_bf16(x.data_ptr(), dp, nw.data_ptr(), 1e-5, M, K, xo.data_ptr() if with_d else None,
                                   h.data_ptr(), st))
    s = (x + d if with_d else x).double()
    want_h = s * torch.rsqrt(s.square().mean(-1, keepdim=True) + 1e-5) * nw.double()
    assert float((h.double() - want_h).abs().sub(2.0 ** -8 * want_h.abs() * (1 + 2.0 ** -12)).max()) <= 0.0
    want = torch.empty_like(out)
    _lib.check(L.lema_skinny_swiglu_bf16(h.data_ptr(), K, wg.data_ptr(), wu.data_ptr(), K, M, 48, K,
                                         want.data_ptr(), st))
    assert torch.equal(out, want)      # the same rows, sums in the same order
    gate, up = h.double() @ wg.double().T, h.double() @ wu.double().T
    ref = torch.nn.functional.silu(gate) * up
    # gate, up, the silu and the result each rounded to bf16; the silu's slope is at most 1.1
    bound = 2.0 ** -8 * (1.1 * gate.abs() * up.abs() + 3.1 * ref.abs()) * 1.01 + 1e-6
    assert float(((out.double() - ref).abs() - bound).max()) <= 0.0


def test_rows_far_apart(dev):
    """Row strides past 2^35 elements: two rows of x, and two of a weight, 64 GiB apart."""
    ld, K = (1 << 35) + 8, 64
    if torch.cuda.mem_get_info(dev)[0] < 2 * ld + (8 << 30):
        pytest.skip("needs 72 GiB of free memory")
    far = torch.empty(ld + K, dtype=torch.bfloat16, device=dev)
    rows = torch.randn((2, K), device=dev).to(torch.bfloat16)
    far[:K], far[ld:] = rows[0], rows[1]
    near = torch.randn((2, K), device=dev).to(torch.bfloat16)
    y = torch.empty((2, 2), dtype=torch.bfloat16, device=dev)
    for x, w, ldx, ldw, want in ((far, near, ld, K, _product(rows, near)), (near, far, K, ld, _product(near, rows))):
        _lib.check(_lib.lib().lema_skinny_gemm_bf16(x.data_ptr(), ldx, w.data_ptr(), ldw, y.data_ptr(), 2, 2, 2, K,
                                                    _lib.stream_of(y)))
        assert torch.equal(y, want)
