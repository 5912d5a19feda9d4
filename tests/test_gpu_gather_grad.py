"""The gradient of the value gather: lema_gather_grad against the sum in 64 bits, for every
dtype, piece size and stride form, for source rows that one, few or nearly all queries read
(lists that fill up before the scan ends), and for the ways a backward can be asked for that
keep the tensor operations. Needs a GPU."""
import pytest
import torch

import latest_exact_match_attention_amd as lema

pytestmark = pytest.mark.gpu

# relative to the sum of |gy| that a gradient element adds up: fp32 additions in any order (a
# few thousand terms at most are read one after another), and half a unit in the last place
# for every rounding to a 16-bit result: one, plus one for every list that was reduced before
# the scan's end, each of which held more than 1536 queries
FP32 = 2e-5
HALF_ULP = {torch.float32: 0.0, torch.float16: 2.0 ** -11, torch.bfloat16: 2.0 ** -8}


@pytest.fixture(scope="module")
def dev():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    return torch.device("cuda", 0)


def _codes(kind, rows, T, g):
    r = lambda n: torch.randint(0, n, (rows, T), generator=g)  # noqa: E731
    if kind == "few":        # 5 codes: runs of queries between two keys
        return r(5), r(5)
    if kind == "many":       # mostly misses
        return r(40 * T + 1), r(40 * T + 1)
    if kind == "first":      # every key but the first ones is new: all queries read 3 rows
        kc = torch.arange(T).expand(rows, T).clone() + 100
        kc[:, :min(3, T)] = torch.arange(min(3, T))
        return r(3), kc
    kc = torch.arange(T).expand(rows, T).clone()   # "spread": all queries read the first
    return r(min(T, 1500)), kc                      # 1500 rows


def _view(x, form):
    """x [B, H, T, d] in another memory order with the same values."""
    if form == "projection":
        return x.transpose(1, 2).contiguous().transpose(1, 2)
    if form == "offset":      # rows that no piece above the element size divides
        B, H, T, d = x.shape
        base = torch.empty((B, H, T, d + 1), dtype=x.dtype, device=x.device)
        base[..., 1:] = x
        return base[..., 1:]
    if form == "columns":     # the last dim strided: copied first
        return x.transpose(2, 3).contiguous().transpose(2, 3)
    return x


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
@pytest.mark.parametrize("kind,B,H,T,dv,form", [
    ("few", 1, 1, 1, 8, "plain"), ("few", 1, 3, 2, 1, "plain"), ("few", 2, 5, 63, 24, "projection"),
    ("few", 1, 2, 1025, 33, "plain"), ("many", 1, 9, 257, 64, "offset"),
    ("many", 2, 64, 3000, 24, "projection"), ("first", 1, 8, 5000, 16, "plain"),
    ("first", 1, 1, 9001, 520, "projection"), ("spread", 2, 3, 20000, 8, "plain"),
    ("spread", 1, 128, 9000, 4, "projection"), ("few", 1, 2, 700, 1100, "columns"),
    # rows that don't fill the XCDs: their parts go round them
    ("few", 1, 1, 40001, 8, "plain"), ("many", 1, 7, 5003, 24, "projection"), ("spread", 3, 3, 2600, 16, "plain"),
    ("few", 1, 12, 1500, 24, "projection"), ("first", 1, 8, 2050, 8, "offset"),
    # long enough for slices of the columns: 2, 4 and a row that none divides
    ("few", 1, 1, 16384, 64, "plain"), ("first", 1, 2, 17000, 128, "projection"), ("many", 1, 1, 16400, 260, "plain"),
    ("few", 1, 1, 16390, 65, "plain"),
])
def test_gradient_is_the_sum(dev, dtype, kind, B, H, T, dv, form):
    g = torch.Generator().manual_seed(T + dv)
    qc, kc = (c.view(B, H, T).to(dev) for c in _codes(kind, B * H, T, g))
    v = torch.randn((B, H, T, dv), generator=g).to(dev, dtype).requires_grad_(True)
    gy = _view(torch.randn((B, H, T, dv), generator=g).to(dev, dtype), form)
    y = lema.attention._LemaGather.apply(qc, kc, v)
    (gv,) = torch.autograd.grad(y, v, gy)
    assert gv.shape == v.shape and gv.dtype == dtype and gv.is_contiguous()
    src = lema.lema_from_codes(qc, kc, v.detach(), return_src=True)[1].long()
    idx = src.clamp_min(0).unsqueeze(-1).expand(B, H, T, dv)
    terms = gy.double() * (src >= 0).unsqueeze(-1)
    zero = torch.zeros((B, H, T, dv), dtype=torch.float64, device=dev)
    want, size = zero.scatter_add(2, idx, terms), zero.scatter_add(2, idx, terms.abs())
    bound = (FP32 + HALF_ULP[dtype] * (1 + T // 1536)) * size
    assert float(((gv.double() - want).abs() - bound).max()) <= 0.0


def test_gradient_of_an_expanded_gy(dev):
    qc = torch.randint(0, 4, (2, 3, 500), device=dev)
    v = torch.randn((2, 3, 500, 16), device=dev, requires_grad=True)
    lema.attention._LemaGather.apply(qc, qc, v).sum().backward()
    src = lema.lema_from_codes(qc, qc, v.detach(), return_src=True)[1].long()
    want = torch.zeros((2, 3, 500), device=dev).scatter_add_(2, src.clamp_min(0), (src >= 0).float())
    assert torch.equal(v.grad, want.unsqueeze(-1).expand_as(v))


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_infinities_and_nans(dev, dtype):
    """A hit's infinity or NaN goes to its source row; a missed query's makes its column of the
    first row NaN, as gy * 0 added to it does."""
    T, dv = 600, 24
    kc = torch.arange(T, device=dev).view(1, 1, T)
    qc = kc - 1                    # query i reads row i - 1; query 0 reads nothing
    qc = qc.clone()
    qc[..., 300:] = T + 5          # misses
    gy = torch.zeros((1, 1, T, dv), device=dev, dtype=dtype)
    gy[0, 0, 10, 3], gy[0, 0, 20, 4] = float("inf"), float("nan")
    gy[0, 0, 400, 5], gy[0, 0, 599, 23], gy[0, 0, 450, 6] = float("-inf"), float("nan"), 7.0
    v = torch.zeros((1, 1, T, dv), device=dev, dtype=dtype, requires_grad=True)
    y = lema.attention._LemaGather.apply(qc, kc, v)
    (got,) = torch.autograd.grad(y, v, gy, retain_graph=True)
    with torch.enable_grad():      # the tensor operations
        (want,) = torch.autograd.grad(y, v, gy.clone().requires_grad_(True), create_graph=True)
    assert torch.equal(torch.isnan(got), torch.isnan(want))
    assert torch.equal(got.nan_to_num(0.0), want.nan_to_num(0.0))


def test_other_backwards_keep_composing(dev):
    qc = torch.randint(0, 6, (1, 2, 40), device=dev)
    v = torch.randn((1, 2, 40, 8), device=dev, requires_grad=True)
    y = lema.attention._LemaGather.apply(qc, qc, v)
    gs = torch.randn((3,) + y.shape, device=dev)
    each = [torch.autograd.grad(y, v, x, retain_graph=True)[0] for x in gs]
    for ask in (lambda: torch.autograd.grad(y, v, gs, is_grads_batched=True, retain_graph=True),
                lambda: torch.func.vmap(
                    lambda x: torch.autograd.grad(y, v, x, retain_graph=True)[0])(gs)):
        with pytest.raises(RuntimeError):   # refused, not computed from one of them
            ask()
    gy = gs[0].clone().requires_grad_(True)          # double backward: the gather itself
    (gv,) = torch.autograd.grad(y, v, gy, create_graph=True)
    (ggy,) = torch.autograd.grad(gv, gy, gs[1])
    torch.testing.assert_close(ggy, lema.lema_from_codes(qc, qc, gs[1]))
    import torch.autograd.forward_ad as fw
    with fw.dual_level():
        dual = torch.autograd.grad(y, v, fw.make_dual(gs[0], gs[1]), retain_graph=True)[0]
        torch.testing.assert_close(fw.unpack_dual(dual).tangent, each[1])
    with torch.autograd.graph.save_on_cpu():
        y2 = lema.attention._LemaGather.apply(qc, qc, v)
    torch.testing.assert_close(torch.autograd.grad(y2, v, gs[2])[0], each[2])


@pytest.mark.parametrize("kind", ["first", "few"])
def test_deterministic_algorithms(dev, kind):
    """Under the switch the gradient is the tensor operations' own, bit for bit, every time."""
    N, T, dv = 2, 9001, 24
    g = torch.Generator().manual_seed(7)
    qc, kc = (c.view(1, N, T).to(dev) for c in _codes(kind, N, T, g))
    v = torch.randn((1, N, T, dv), generator=g).to(dev).requires_grad_(True)
    gy = torch.randn((1, N, T, dv), generator=g).to(dev)
    y = lema.attention._LemaGather.apply(qc, kc, v)
    src = lema.lema_from_codes(qc, kc, v.detach(), return_src=True)[1].long()
    idx = src.clamp_min(0).unsqueeze(-1).expand(1, N, T, dv)
    torch.use_deterministic_algorithms(True)
    try:
        want = torch.zeros_like(gy).scatter_add_(2, idx, gy * (src >= 0).unsqueeze(-1))
        for _ in range(2):
            (gv,) = torch.autograd.grad(y, v, gy, retain_graph=True)
            assert torch.equal(gv, want)
    finally:
        torch.use_deterministic_algorithms(False)


@pytest.mark.parametrize("kept", [torch.int64, torch.int16])
def test_indices_that_a_hook_keeps_in_another_type(dev, kept):
    """Saved-tensor hooks may bring the indices back wider or narrower than they were saved."""
    qc = torch.randint(0, 6, (1, 2, 900), device=dev)
    v = torch.randn((1, 2, 900, 8), device=dev, requires_grad=True)
    gy = torch.randn((1, 2, 900, 8), device=dev)
    (want,) = torch.autograd.grad(lema.attention._LemaGather.apply(qc, qc, v), v, gy)
    with torch.autograd.graph.saved_tensors_hooks(lambda x: x.to(kept), lambda x: x):
        y = lema.attention._LemaGather.apply(qc, qc, v)
    (got,) = torch.autograd.grad(y, v, gy)
    # a row's sum in another order: fp32, at most 900 terms
    torch.testing.assert_close(got, want, rtol=1e-4, atol=1e-4)


def test_rows_as_wide_as_the_forward_takes(dev):
    """Value rows of 2^20 and more elements have a gradient too, in pieces of 16 and of 4 bytes."""
    dv = (1 << 20) + 8
    for at in (0, 1):                                # gy's rows on and off a 16-byte boundary
        qc = torch.zeros((1, 1, 3), dtype=torch.int32, device=dev)
        v = torch.randn((1, 1, 3, dv), device=dev, requires_grad=True)
        gy = torch.randn((1, 1, 3, dv + 4), device=dev)[..., at:at + dv]
        (gv,) = torch.autograd.grad(lema.attention._LemaGather.apply(qc, qc, v), v, gy)
        want = torch.stack([gy[0, 0, 1], gy[0, 0, 2], torch.zeros_like(gy[0, 0, 0])])
        assert torch.equal(gv[0, 0], want), at       # query 1 reads row 0, query 2 row 1


def test_the_longest_rows_keep_the_tensor_operations(dev, monkeypatch):
    """Rows from attention.GRAD_KERNEL_T on take the tensor operations, shorter ones the kernel."""
    qc = torch.randint(0, 6, (1, 2, 300), device=dev)
    v = torch.randn((1, 2, 300, 8), device=dev, requires_grad=True)
    gy = torch.randn((1, 2, 300, 8), device=dev)
    y = lema.attention._LemaGather.apply(qc, qc, v)
    calls = []
    check = lema.attention._lib.check
    monkeypatch.setattr(lema.attention._lib, "check", lambda rc: (calls.append(rc), check(rc)))
    both = []
    for line, kernel in ((301, 1), (300, 0)):
        monkeypatch.setattr(lema.attention, "GRAD_KERNEL_T", line)
        calls.clear()
        both.append(torch.autograd.grad(y, v, gy, retain_graph=True)[0])
        assert len(calls) == kernel, line
    torch.testing.assert_close(both[0], both[1], rtol=1e-4, atol=1e-4)  # sums in another order
