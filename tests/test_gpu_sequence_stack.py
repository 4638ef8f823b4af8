"""The Pairformer sequence stack as one native call (``bmx_sequence_stack_fwd``)
against the fp32 oracle layer evaluated in fp64."""

import pytest
import torch

from boltz_lumi_amd import _native, layers, pairformer
from oracle import boltz_ref as R

pytestmark = pytest.mark.gpu


def _layer(dev):
    ref = R.randomize(R.PairformerLayer(), generator=torch.Generator().manual_seed(2)).eval()
    mine = layers.PairformerLayer()
    mine.load_state_dict(ref.state_dict())
    return ref.double().to(dev), mine.to(dev).eval()


def _want(ref, s, bias, mask):
    s, att = s.double(), ref.attention
    sn = ref.pre_norm_s(s)
    b, n = s.shape[:2]
    q, k, v = (lin(sn).view(b, n, 16, 24).transpose(1, 2).contiguous() for lin in (att.proj_q, att.proj_k, att.proj_v))
    logits = torch.matmul(q, k.transpose(2, 3).contiguous()) / 24 ** 0.5 + bias.double()
    logits = logits + ((1 - mask.double()) * -att.inf)[:, None, None, :]
    o = torch.matmul(torch.softmax(logits, -1), v).transpose(1, 2).reshape(b, n, 384)
    s = s + att.proj_o(torch.sigmoid(att.proj_g(sn)) * o)
    return s + ref.transition_s(s)


# one row, partial and full 32-row tiles, 128 keys (two-tile and four-tile attention), one and two column
# tiles per block (700 tiles), odd key counts (bias rows at any alignment), batches, the last row count of
# the native call and the first of torch's GEMMs
@pytest.mark.parametrize("b,n", [(1, 1), (1, 31), (1, 32), (1, 33), (1, 117), (1, 128), (1, 129), (2, 63), (3, 150),
                                 (1, 450), (1, 497), (1, 767), (1, 1134), (1, 1280), (20, 64), (1, 1281),
                                 (21, 64)])
def test_sequence_stack_rows(gpu, b, n):
    ref, mine = _layer(gpu)
    g = torch.Generator().manual_seed(n)
    s = torch.randn(b, n, 384, generator=g).to(gpu)
    bias = torch.randn(b, 16, n, n, generator=g).to(gpu)
    mask = torch.ones(b, n, device=gpu)
    if n > 8:
        mask[0, -5:] = 0
    z = torch.zeros(b, n, n, 128, device=gpu)
    calls, real = [], _native.call
    with torch.inference_mode(), pytest.MonkeyPatch.context() as mp:
        mp.setattr(_native, "call", lambda name, *args: calls.append(name) or real(name, *args))
        s0 = s.clone()
        got = pairformer.sequence_stack(mine, s, z, mask, pair_bias=bias)
        again = pairformer.sequence_stack(mine, s, z, mask, pair_bias=bias)
        want = _want(ref, s, bias, mask)
        # the same stack on torch's fp32 GEMMs: the native one may be no further off
        mp.setattr(pairformer, "_native_sequence_params", lambda *_: None)
        torch_path = pairformer.sequence_stack(mine, s, z, mask, pair_bias=bias)
    native = b * n <= pairformer.SEQUENCE_MAX_ROWS
    assert calls.count("bmx_sequence_stack_fwd") == (2 if native else 0)
    assert torch.equal(got, again) and torch.equal(s, s0)
    err, err_torch = (((x.double() - want).norm() / want.norm()).item() for x in (got, torch_path))
    print(f"b={b} n={n}: {err:.2e}, torch {err_torch:.2e}", flush=True)
    assert err <= max(err_torch, 2**-23)  # an ulp of the outputs: what one rounding more may cost


def test_sequence_stack_keeps_other_cases(gpu):
    """A hooked transition and a changed weight: torch's
    path for the first, a repack for the second."""
    ref, mine = _layer(gpu)
    s, bias = torch.randn(1, 40, 384, device=gpu), torch.randn(1, 16, 40, 40, device=gpu)
    z, mask = torch.zeros(1, 40, 40, 128, device=gpu), torch.ones(1, 40, device=gpu)
    calls, real = [], _native.call
    with torch.inference_mode(), pytest.MonkeyPatch.context() as mp:
        mp.setattr(_native, "call", lambda name, *args: calls.append(name) or real(name, *args))
        handle = mine.transition_s.register_forward_hook(lambda *_: None)
        got = pairformer.sequence_stack(mine, s, z, mask, pair_bias=bias)
        handle.remove()
        assert "bmx_sequence_stack_fwd" not in calls
        assert torch.allclose(got.double(), _want(ref, s, bias, mask), atol=1e-4, rtol=1e-4)
        pairformer.sequence_stack(mine, s, z, mask, pair_bias=bias)
    with torch.no_grad():
        for m in (ref, mine):
            m.transition_s.fc2.weight.mul_(1.25)
    with torch.inference_mode():
        got = pairformer.sequence_stack(mine, s, z, mask, pair_bias=bias)
        assert torch.allclose(got.double(), _want(ref, s, bias, mask), atol=1e-4, rtol=1e-4)


def test_sequence_stack_odd_offsets(gpu):
    """Contiguous fp32 activations and parameters at a 4-byte storage offset
    (views of one flat buffer): the same result as at an aligned one."""

    def offset(t):
        return torch.empty(t.numel() + 1, device=gpu)[1:].view(t.shape).copy_(t)

    _, mine = _layer(gpu)
    s, bias = torch.randn(1, 40, 384, device=gpu), torch.randn(1, 16, 40, 40, device=gpu)
    z, mask = torch.zeros(1, 40, 40, 128, device=gpu), torch.ones(1, 40, device=gpu)
    with torch.inference_mode():
        want = pairformer.sequence_stack(mine, s, z, mask, pair_bias=bias)
    with torch.no_grad():
        for module in mine.modules():
            for name, p in list(module.named_parameters(recurse=False)):
                setattr(module, name, torch.nn.Parameter(offset(p), requires_grad=False))
        got = pairformer.sequence_stack(mine, offset(s), z, mask, pair_bias=bias)
    assert torch.equal(got, want)


def test_sequence_stack_silu(gpu):
    """silu(v) * g alone in the output (one nonzero weight per row, no residual)
    for v down to -80: as exact as fp32 operations give it. A fast exponential's
    argument error grows with |v|."""
    _, mine = _layer(gpu)
    tr, v = mine.transition_s, -torch.arange(8, 8 + 384, device=gpu) * 0.2
    scale = torch.exp2(torch.round(-v * 1.4427))  # a power of two: the product's rounding alone
    with torch.no_grad():
        for p in (mine.attention.proj_o.weight, tr.norm.weight, tr.fc1.weight, tr.fc2.weight, tr.fc3.weight):
            p.zero_()
        tr.norm.bias.fill_(1)
        tr.fc1.weight[:384, 0] = v
        tr.fc2.weight[:384, 0] = scale
        tr.fc3.weight[:, :384] = torch.eye(384, device=gpu)
    calls, real = [], _native.call
    with torch.inference_mode(), pytest.MonkeyPatch.context() as mp:
        mp.setattr(_native, "call", lambda name, *args: calls.append(name) or real(name, *args))
        got = pairformer.sequence_stack(mine, torch.zeros(1, 40, 384, device=gpu),
                                        torch.zeros(1, 40, 40, 128, device=gpu), torch.ones(1, 40, device=gpu),
                                        pair_bias=torch.zeros(1, 16, 40, 40, device=gpu))
    assert "bmx_sequence_stack_fwd" in calls
    want = torch.nn.functional.silu(v.double()) * scale.double()
    err = ((got.double() - want) / want).abs().max().item()
    print(f"silu error {err:.2e}", flush=True)
    assert err < 6 * 2**-24  # exp: 1 ulp; sum, quotient and product: half an ulp each
