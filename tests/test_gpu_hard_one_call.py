"""lema_hard's single library call against pack_codes followed by lema_from_codes, byte for byte,
over the layouts, widths and dtypes it takes and the ones it leaves to them; the errors of the
calls it does not take. Needs a GPU."""
import pytest
import torch

import latest_exact_match_attention_amd as lema
from latest_exact_match_attention_amd import attention

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def dev():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    return torch.device("cuda", 0)


def _z(form, B, H, T, D, dtype, dev, g):
    """Pre-activations whose codes recur: one of 5 sign rows per position."""
    book = torch.randn((5, D), generator=g)
    z = (book[torch.randint(0, 5, (B, H, T), generator=g)]).to(dev, dtype)
    if form == "projection":
        return z.transpose(1, 2).contiguous().transpose(1, 2)
    if form == "unaligned":            # every row starts off a 16-byte boundary
        base = torch.empty(z.numel() + 1, dtype=dtype, device=dev)
        base[1:] = z.reshape(-1)
        return base[1:].view(z.shape)
    if form == "gaps":                 # rows apart in memory
        base = torch.empty((B, H, T, D + 3), dtype=dtype, device=dev)
        base[..., :D] = z
        return base[..., :D]
    if form == "shared":               # one head's rows for all
        return z[:, :1].expand(B, H, T, D)
    if form == "columns":              # the last dim strided: packed after a copy
        return z.transpose(2, 3).contiguous().transpose(2, 3)
    return z


FORMS = ["plain", "projection", "unaligned", "gaps", "shared", "columns"]


@pytest.mark.parametrize("qf", FORMS)
@pytest.mark.parametrize("kf", FORMS)
@pytest.mark.parametrize("B,H,T,D,dv,dt,vt", [
    (1, 1, 1, 1, 1, torch.float32, torch.float32), (2, 3, 65, 8, 24, torch.bfloat16, torch.bfloat16),
    (1, 64, 130, 24, 33, torch.float16, torch.float32), (2, 5, 1030, 33, 16, torch.float32, torch.float16),
    (1, 2, 300, 64, 64, torch.bfloat16, torch.bfloat16),
])
def test_one_call_equals_the_steps(dev, qf, kf, B, H, T, D, dv, dt, vt):
    g = torch.Generator().manual_seed(T + D)
    q, k = _z(qf, B, H, T, D, dt, dev, g), _z(kf, B, H, T, D, dt, dev, g)
    v = torch.randn((B, T, H, dv), generator=g).to(dev, vt).transpose(1, 2)
    ct = attention.code_dtype_for(D)
    want = lema.lema_from_codes(lema.pack_codes(q, ct), lema.pack_codes(k, ct), v)
    got = lema.lema_hard(q, k, v)
    assert torch.equal(got, want) and got.stride() == want.stride()
    vg = v.detach().requires_grad_(True)
    y = lema.lema_hard(q.clone().requires_grad_(True), k, vg)
    assert torch.equal(y, want)
    (gv,) = torch.autograd.grad(y, vg, torch.ones_like(y))
    assert gv.shape == v.shape


def test_long_rows_and_mixed_dtypes(dev):
    g = torch.Generator().manual_seed(5)
    T = 66 * 1024 + 3                              # chunk summaries
    q, k = (_z("plain", 1, 2, T, 40, torch.bfloat16, dev, g) for _ in range(2))
    v = torch.randn((1, 2, T, 8), device=dev)
    want = lema.lema_from_codes(lema.pack_codes(q), lema.pack_codes(k), v)
    assert torch.equal(lema.lema_hard(q, k, v), want)
    assert torch.equal(lema.lema_hard(q.float(), k, v), want)   # two calls' dtypes


def test_refusals_are_the_steps_own(dev):
    q = torch.randn((1, 2, 8, 16), device=dev)
    v = torch.randn((1, 2, 8, 4), device=dev)
    with pytest.raises(ValueError):
        lema.lema_hard(torch.randn((1, 2, 8, 65), device=dev), torch.randn((1, 2, 8, 65), device=dev), v)
    with pytest.raises((ValueError, RuntimeError)):
        lema.lema_hard(q, q[:, :, :7], v)
    with pytest.raises(ValueError):
        lema.lema_hard(q, q, v[:, :, :7])
    with pytest.raises(TypeError):
        lema.lema_hard(q.double(), q.double(), v)
    with pytest.raises(TypeError):
        lema.lema_hard(q.cpu(), q.cpu(), v.cpu())
    assert lema.lema_hard(q[:, :, :0], q[:, :, :0], v[:, :, :0]).shape == (1, 2, 0, 4)
