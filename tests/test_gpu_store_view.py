"""Exchanges whose values are a strided [B, H, T, d] view, read in place, against the same call
with contiguous values: outputs, counts and the table's entries, on the chunked and the bulk
path, for 8- and 16-byte pieces. Needs a GPU."""
import pytest
import torch

from latest_exact_match_attention_amd.cache import HashStore, LayerStore

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def dev():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    return torch.device("cuda", 0)


def _entries(store):
    group, code, rows = store.dump()
    key = sorted(zip(group.tolist(), code.tolist(), map(bytes, rows.cpu().numpy())))
    return key


def _view(v, form):
    if form == "projection":
        return v.transpose(1, 2).contiguous().transpose(1, 2)
    if form == "gaps":                  # 8 bytes between rows: no 16-byte pieces
        B, H, T, d = v.shape
        base = torch.empty((B, H, T, d + 8 // v.element_size()), dtype=v.dtype, device=v.device)
        base[..., :d] = v
        return base[..., :d]
    if form == "offset":                # the pointer 8 bytes off
        n = 8 // v.element_size()
        base = torch.empty(v.numel() + n, dtype=v.dtype, device=v.device)
        base[n:] = v.transpose(1, 2).reshape(-1)
        B, H, T, d = v.shape
        return base[n:].view(B, T, H, d).transpose(1, 2)
    if form == "shared":                # one stream's values for all
        return v[:1].expand(v.shape)
    return v.transpose(2, 3).contiguous().transpose(2, 3)     # the last dim strided: copied


@pytest.mark.parametrize("form", ["projection", "gaps", "offset", "shared", "columns"])
@pytest.mark.parametrize("B,H,T,d,dt", [
    (2, 3, 2, 8, torch.float32), (2, 5, 300, 24, torch.bfloat16), (1, 3, 1500, 4, torch.float16),
    (3, 7, 1025, 64, torch.bfloat16), (1, 2, 33000, 16, torch.bfloat16), (4, 40, 1100, 24, torch.float16),
])
def test_view_equals_contiguous(dev, form, B, H, T, d, dt):
    g = torch.Generator().manual_seed(T + d)
    P = B * H
    kc = torch.randint(0, max(2, T // 2), (2, B, H, T), generator=g).to(dev)
    qc = torch.randint(0, max(2, T), (2, B, H, T), generator=g).to(dev)
    stores = [HashStore(d, groups=P, dtype=dt, capacity=2 * P * T, device=dev) for _ in range(2)]
    layers = [LayerStore(s, 0, P) for s in stores]
    for i in range(2):
        v = _view(torch.randn((B, H, T, d), generator=g).to(dev, dt), form)
        got = layers[0].exchange(qc[i], kc[i], v)
        want = layers[1].exchange(qc[i], kc[i], v.contiguous())
        assert torch.equal(got, want) and got.is_contiguous()
    assert torch.equal(stores[0].counts, stores[1].counts)
    assert _entries(stores[0]) == _entries(stores[1])


def test_results_over_the_values_memory(dev):
    """A caller's buffer that the values view lies in still gets the exchange of the old values."""
    g = torch.Generator().manual_seed(3)
    B, H, T, d = 2, 4, 50, 8
    kc = torch.randint(0, 9, (B, H, T), generator=g).to(dev)
    base = torch.randn((B, T, H, d), generator=g).to(dev)
    a, b = (HashStore(d, groups=B * H, dtype=torch.float32, capacity=4096, device=dev) for _ in range(2))
    want = torch.empty((B, H, T, d), device=dev)
    a.exchange(kc, kc, base.transpose(1, 2).contiguous(), want, T, 0)
    out = base.view(B, H, T, d)
    b.exchange(kc, kc, base.transpose(1, 2), out, T, 0)
    assert torch.equal(out, want)
    assert _entries(a) == _entries(b)


def test_a_view_that_carries_a_sign(dev):
    """A negated or conjugated view's signs are not in memory: such values are copied first."""
    g = torch.Generator().manual_seed(4)
    B, H, T, d = 1, 2, 40, 8
    kc = torch.randint(0, 9, (B, H, T), generator=g).to(dev)
    z = torch.randn((B, T, H, d), generator=g, dtype=torch.complex64).to(dev)
    for x in (torch._neg_view(z.real.contiguous()).transpose(1, 2), z.conj().transpose(1, 2)):
        a, b = (HashStore(d * x.element_size() // 4, groups=B * H, dtype=torch.float32, capacity=4096, device=dev)
                for _ in range(2))
        want, got = (torch.empty((B, H, T, d), dtype=x.dtype, device=dev) for _ in range(2))
        a.exchange(kc, kc, x.resolve_neg().resolve_conj().contiguous(), want, T, 0)
        b.exchange(kc, kc, x, got, T, 0)
        assert torch.equal(got, want)
        assert _entries(a) == _entries(b)


def test_results_over_part_of_the_values_memory(dev):
    """Overlap is a matter of addresses: tensors that share memory may have storages of their own."""
    g = torch.Generator().manual_seed(5)
    B, H, T, d = 2, 4, 700, 8
    n = B * H * T * d
    kc = torch.randint(0, 9, (B, H, T), generator=g).to(dev)
    buf = torch.randn(n + 64, generator=g).to(dev)
    values = buf[:n].view(B, T, H, d).transpose(1, 2)
    out = torch.from_dlpack(buf[64:].view(B, H, T, d))
    assert out.untyped_storage().data_ptr() != values.untyped_storage().data_ptr()
    a, b = (HashStore(d, groups=B * H, dtype=torch.float32, capacity=1 << 14, device=dev) for _ in range(2))
    want = torch.empty((B, H, T, d), device=dev)
    a.exchange(kc, kc, values.contiguous(), want, T, 0)
    b.exchange(kc, kc, values, out, T, 0)
    assert torch.equal(out, want)
    assert _entries(a) == _entries(b)
