"""What surrounds latent attention's products in fewer launches, against the separate operations (the same arithmetic: the same bits): the norms and
the cache row, with and without the expanded rows, slots that write nothing, turned queries in place; and sigmoid gates 16 bytes at a time."""

import pytest
import torch

from llmctl.ops import hybrid as hops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("T,H,nq,rk,dr,rot", [(1, 2, 24, 16, 8, 8), (16, 16, 1024, 512, 64, 64), (33, 3, 257, 300, 40, 24), (200, 4, 8, 64, 0, 0)])
@pytest.mark.parametrize("inter", [False, True])
@pytest.mark.parametrize("expand", [False, True])
def test_latent_prep(T, H, nq, rk, dr, rot, inter, dtype, expand):
    g = torch.Generator(device="cuda").manual_seed(T + rk)
    r = lambda *s: torch.randn(*s, generator=g, device="cuda")
    z = r(T, nq + rk + dr + 24).to(dtype)
    qw, kw, freq = r(nq), r(rk), torch.rand(rot // 2, generator=g, device="cuda")
    pos = torch.randint(0, 5000, (T,), generator=g, device="cuda", dtype=torch.int32)
    slots = torch.randperm(T + 9, generator=g, device="cuda")[:T]
    if not expand and T > 1:
        slots[T // 2] = -1
    caches = [torch.zeros((T + 9 + 3) // 4, 4, rk + dr, device="cuda", dtype=dtype) for _ in range(2)]
    rows = torch.full((T, H, 12 + dr), 7.0, device="cuda", dtype=dtype) if expand else None
    cq, lat = hops.latent_prep(z, qw, kw, dr, 1e-5, pos, freq, rot, caches[0], slots, inter, 1.25, rows, 12)
    hops.latent_kv_write(z[:, nq:nq + rk + dr], kw, 1e-5, pos, freq, rot, caches[1], slots, inter, 1.25)
    assert torch.equal(caches[0], caches[1])
    assert torch.equal(cq, hops.rmsnorm_cols(z[:, :nq], qw, 1e-5, nq, dtype))
    if expand:
        want = caches[1].view(-1, rk + dr)[slots]
        assert torch.equal(lat, want) and torch.equal(rows[:, :, 12:], want[:, None, rk:].expand(T, H, dr)) and (rows[:, :, :12] == 7).all()
    else:
        assert lat is None
    q = r(T, H, 20 + dr).to(dtype)
    want = hops.latent_q_assemble(q[:, :, :20], q, pos, freq, rot, 20, inter, 1.25)
    assert torch.equal(hops.rotary_tail_(q, pos, freq, rot, 20, inter, 1.25), want)


@pytest.mark.parametrize("T,H,nq,rk,dr,rot", [(1, 1, 8, 8, 8, 2), (9, 5, 2048, 2040, 64, 64), (5, 3, 2056, 512, 72, 70), (3, 2, 4096, 4088, 520, 514), (2, 1, 64, 4104, 8, 8)])
@pytest.mark.parametrize("expand", [False, True])
def test_latent_prep_of_rows_in_8s(T, H, nq, rk, dr, rot, expand):
    """Expanded rows whose key columns start on 16 bytes; one and two chunks a thread, and rows too long for them."""
    g = torch.Generator(device="cuda").manual_seed(T + rk)
    r = lambda *s: torch.randn(*s, generator=g, device="cuda")
    z = r(T, nq + rk + dr + 16).bfloat16()
    qw, kw, freq = r(nq), r(rk), torch.rand(rot // 2, generator=g, device="cuda")
    pos = torch.randint(0, 5000, (T,), generator=g, device="cuda", dtype=torch.int32)
    slots = torch.randperm(T + 9, generator=g, device="cuda")[:T]
    if not expand and T > 1:
        slots[T // 2] = -1
    caches = [torch.zeros((T + 9 + 3) // 4, 4, rk + dr, device="cuda", dtype=torch.bfloat16) for _ in range(2)]
    rows = torch.full((T, H, 16 + dr), 7.0, device="cuda", dtype=torch.bfloat16) if expand else None
    for inter in (False, True):
        cq, lat = hops.latent_prep(z, qw, kw, dr, 1e-5, pos, freq, rot, caches[0], slots, inter, 1.25, rows, 8)
        hops.latent_kv_write(z[:, nq:nq + rk + dr], kw, 1e-5, pos, freq, rot, caches[1], slots, inter, 1.25)
        assert torch.equal(caches[0], caches[1]) and torch.equal(cq, hops.rmsnorm_cols(z[:, :nq], qw, 1e-5, nq, torch.bfloat16))
        if expand:
            want = caches[1].view(-1, rk + dr)[slots]
            assert torch.equal(lat, want) and torch.equal(rows[:, :, 8:8 + dr], want[:, None, rk:].expand(T, H, dr))
            assert (rows[:, :, :8] == 7).all() and (rows[:, :, 8 + dr:] == 7).all()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("T,W,per", [(1, 8, 1), (5, 2048, 1), (33, 264, 1), (5, 256, 128), (7, 96, 8), (3, 96, 4), (9, 36, 12), (3, 30, 1)])
@pytest.mark.parametrize("off", [0, 2, 8])
def test_gates(T, W, per, dtype, off):
    g = torch.Generator(device="cuda").manual_seed(T + W)
    o = torch.randn(T, W, generator=g, device="cuda").to(dtype)
    gate = torch.randn(T, W // per + 16, generator=g, device="cuda").to(dtype)[:, off:off + W // per]
    got = hops.sigmoid_gate_mul(o, gate)
    want = (o.double() * torch.sigmoid(gate.double().repeat_interleave(per, 1)))
    # expf, an fp32 division and a product: a few ulp, then one rounding
    assert ((got.double() - want).abs() <= (2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -20) * want.abs() + 1e-30).all()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("T,W,per", [(64, 2048, 1), (65, 2048, 1), (257, 1032, 1), (700, 256, 128), (1400, 96, 8), (1400, 96, 4), (4000, 36, 12), (4500, 30, 1)])
@pytest.mark.parametrize("off", [0, 2, 8])
def test_gates_of_many_rows(T, W, per, dtype, off):
    """Sixteen bytes a thread, past 2^17 elements."""
    test_gates(T, W, per, dtype, off)
