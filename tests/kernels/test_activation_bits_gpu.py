"""Activations of rounded results, in the epilogues of products and in passes, against float64: not further off than the forms with the mathematical library's functions.
(A weight that is the identity, or several of them, makes a product's sums chosen numbers.)"""
import pytest
import torch

pytestmark = pytest.mark.gpu
N = 256


def _numbers():
    x = torch.arange(1 << 16, dtype=torch.int32).to(torch.int16).view(torch.bfloat16).view(N, N)
    return torch.where(x.isfinite(), x, torch.zeros_like(x)).cuda()


def _eye():
    return torch.eye(N, device="cuda", dtype=torch.bfloat16)


def _gelu(x):
    return torch.special.ndtr(x.double()) * x.double()


def _check_gelu(x, got):
    """One rounding to bf16 (2^-8) of what is within 7.3e-8 |x| of the exact value; subnormal results lose no more than a step of theirs."""
    want = _gelu(x)
    err = 7.5e-8 * x.double().abs()
    assert got.dtype == torch.bfloat16 and bool(((got.double() - want).abs() <= 2.0**-8 * want.abs() + 1.01 * err + 2.0**-133).all())


def test_gelu_of_every_number():
    from llmctl.ops import hybrid as hops
    from llmctl.ops._lib import native

    x, one = _numbers(), _eye()
    _check_gelu(x, hops.act_any(x, "gelu"))
    odd = torch.cat([x, x], 1)[:, 1:N + 1]  # (element by element)
    _check_gelu(odd, hops.act_any(odd, "gelu"))
    for form in (1, 2):
        _check_gelu(x, native().gemm_rows(x, one, None, form, 1, 1))
    _check_gelu(x, native().gemm_rows(torch.cat([x, torch.zeros_like(x)], 1), torch.cat([one, one], 1), None, 1, 2, 1))
    inf = torch.tensor([float("inf"), float("-inf"), float("nan")], device="cuda").bfloat16().repeat(8)[None]
    got = hops.act_any(inf, "gelu")[0, :3]
    assert got[0] == float("inf") and got[1].isnan() and got[2].isnan()  # (as 0.5 x (1 + erf) has it)


def test_gelu_of_fp32_sums():
    """16 million sums of 24 bits, as three bf16 numbers each: some 2000 of them are so near to the middle between two bf16 numbers that 1.5e-7 |x| too much would show (erff's form: 1.2e-7)."""
    from llmctl.ops._lib import native

    g = torch.Generator(device="cuda").manual_seed(0)
    for _ in range(8):
        x = torch.randn(8192, N, generator=g, device="cuda")
        hi = x.bfloat16()
        mid = (x - hi.float()).bfloat16()
        lo = (x - hi.float() - mid.float()).bfloat16()
        got = native().gemm_rows(torch.cat([hi, mid, lo], 1), torch.cat([_eye()] * 3, 1), None, 1, 1, 1)
        exact = _gelu(x)
        half = 2.0 ** (exact.abs().log2().floor() - 8)  # of a step of bf16
        assert bool(((got.double() - exact).abs() <= half + 7.5e-8 * x.double().abs()).all())


def _experts(x, act):
    """Rows of many on either kind of tiles, and of few, whose kernel takes the first projection's sums as they are: here exact bf16 numbers."""
    from llmctl.ops import hybrid as hops

    one = _eye()
    up = torch.cat([one, one])[None] if act == "swiglu" else one[None]
    nat, idx, w = hops.native_hybrid(), torch.zeros(N, 1, device="cuda", dtype=torch.int32), torch.ones(N, 1, device="cuda")
    call = lambda a, b, form: nat.moe_experts(x[a:b], idx[a:b], w[a:b], [up], [one[None]], hops._EXPERT_ACTS[act], None, None, form).bfloat16()
    return [call(0, N, 1), call(0, N, 2)], torch.cat([call(i, i + 64, 0) for i in range(0, N, 64)])


def test_gelu_of_experts():
    x = _numbers()
    many, few = _experts(x, "gelu")
    assert all(torch.equal(y, few) for y in many)
    _check_gelu(x, few)


def test_silu_of_experts():
    x = _numbers()
    many, few = _experts(torch.where(x.abs() < 2.0**63, x, torch.zeros_like(x)), "swiglu")  # (their squares are finite)
    assert all(torch.equal(y, few) for y in many)


@pytest.mark.parametrize("each", [True, False])
def test_gates_of_attention(each):
    """Every number as a gate: what the pass after the attention gives, prompts and decode rows whose splits a merge joins."""
    from llmctl.ops import hybrid as hops

    H, R, T = 2, 128, N
    g = torch.Generator(device="cuda").manual_seed(0)
    r = lambda *s: torch.randn(*s, generator=g, device="cuda").bfloat16()
    cache, bt = r(T * 8, 16, R), torch.arange(T * 8, device="cuda", dtype=torch.int32).view(T, 8)
    gate = _numbers() if each else _numbers()[:, :H]
    for col in range(0, 1 if each else N, H):
        if not each:
            gate = _numbers()[:, col:col + H]
        qa, one = r(T, H, R), torch.full((T,), 128, device="cuda", dtype=torch.int32)
        cu = torch.tensor([0, T // 2, T], device="cuda", dtype=torch.int32)
        calls = [lambda **kw: hops.latent_attention_decode(qa, cache, bt, one, hops.NO_LIMIT, None, 0.1, R, max_ctx=128, **kw),
                 lambda **kw: hops.latent_attention_prefill(qa, cache, bt[:2], cu, one[:2], hops.NO_LIMIT, None, 0.1, R, T // 2, **kw)]
        for call in calls:
            assert torch.equal(call(gate=gate).reshape(T, -1), hops.sigmoid_gate_mul(call().reshape(T, -1), gate))
