"""The token transformer as one native call (``bmx_token_stack_fwd``, up to
1024 rows of a prepacked bias) against the fp32 oracle stack."""

import copy

import pytest
import torch
import torch.nn.utils.parametrize as parametrize
from torch import nn

from boltz_lumi_amd import _native, adapters, diffusion, ops
from boltz_lumi_amd.pair_bias import prepare_token_bias
from oracle import boltz_ref as R

pytestmark = pytest.mark.gpu

DEPTH, HEADS, WIDTH = 3, 16, 768


def _stack(dev, biased=False, heads=HEADS, width=WIDTH):
    ref = R.DiffusionTransformer(DEPTH, heads, width, width)
    if biased:  # every bias the call can carry, an s_norm with a bias among them
        ref.layers[1].adaln.s_norm = nn.LayerNorm(WIDTH)
        for layer in ref.layers:
            tr = layer.transition
            tr.swish_gate[0] = nn.Linear(WIDTH, 4 * WIDTH)
            tr.b_to_a = nn.Linear(2 * WIDTH, WIDTH)
            layer.pair_bias_attn.proj_o = nn.Linear(WIDTH, WIDTH)
    ref = R.randomize(ref, std=0.04, generator=torch.Generator().manual_seed(3)).to(dev).eval()
    host = nn.Module()
    host.structure_module = nn.Module()
    host.structure_module.score_model = nn.Module()
    host.structure_module.score_model.token_transformer = copy.deepcopy(ref)
    adapters.install(host, require_boltz2=False)
    return ref, host.structure_module.score_model.token_transformer


def _run(stack, ref, dev, structures, samples, n, calls, pack=prepare_token_bias):
    g = torch.Generator().manual_seed(n)
    b = structures * samples
    att = ref.layers[0].pair_bias_attn
    a, s = torch.randn(b, n, att.c_s, generator=g).to(dev), torch.randn(b, n, att.c_s, generator=g).to(dev)
    bias = torch.randn(structures, n, n, DEPTH * att.num_heads, generator=g).to(dev)
    mask = torch.ones(b, n, device=dev)
    if n > 4:
        mask[0, -3:] = 0
    a0 = a.clone()
    real = _native.call
    with torch.inference_mode(), pytest.MonkeyPatch.context() as mp:
        mp.setattr(_native, "call", lambda name, *args: calls.append(name) or real(name, *args))
        got = stack(a, s, pack(bias), mask, None, samples)
        again = stack(a, s, pack(bias), mask, None, samples)
        want = ref(a, s, bias, mask, None, samples)
    assert torch.equal(a, a0) and torch.equal(got, again)
    return ((got - want).double().norm() / want.double().norm()).item(), (got - want).abs().max() / want.abs().max()


# one row, partial and full 32-row tiles, both tile widths (768 tiles is the line), the fp32 and the
# split-bf16 attention (256 keys), several structures and samples, the last row count taken (1024) and
# the first one left to the library's GEMMs
@pytest.mark.parametrize("structures,samples,n", [(1, 1, 1), (1, 1, 31), (1, 5, 13), (2, 2, 64), (1, 1, 255), (1, 1, 256),
                                                  (1, 3, 257), (2, 2, 256), (1, 1, 1024), (1, 5, 205)])
def test_token_stack_rows(gpu, structures, samples, n):
    ref, stack = _stack(gpu)
    calls = []
    rel, mx = _run(stack, ref, gpu, structures, samples, n, calls)
    native = structures * samples * n <= diffusion.TOKEN_STACK_MAX_ROWS
    assert calls.count("bmx_token_stack_fwd") == (2 if native else 0)
    # split products: 2^-16 relative each, as the per-layer path (its bar is 1e-4 too)
    assert rel < 3e-5 and mx < 1e-4


def test_token_stack_biases_and_updates(gpu):
    ref, stack = _stack(gpu, biased=True)
    calls = []
    rel, mx = _run(stack, ref, gpu, 1, 2, 40, calls)
    assert "bmx_token_stack_fwd" in calls and rel < 3e-5 and mx < 1e-4
    with torch.no_grad():  # an in-place update repacks
        for m in (ref, stack):
            m.layers[2].transition.b_to_a.weight.mul_(1.5)
    rel, mx = _run(stack, ref, gpu, 1, 2, 40, calls)
    assert rel < 3e-5 and mx < 1e-4


def test_token_stack_leaves_other_cases(gpu):
    """A memoised projection, a hooked proj_o, exact fp32 linears and an
    unpacked bias keep the per-layer path."""
    ref, stack = _stack(gpu)
    calls = []
    lin = stack.layers[1].adaln.s_scale
    lin.forward = lambda x, f=type(lin).forward, m=lin: f(m, x)
    rel, mx = _run(stack, ref, gpu, 1, 1, 40, calls)
    del lin.forward
    assert rel < 3e-5 and mx < 1e-4
    handle = stack.layers[1].pair_bias_attn.proj_o.register_forward_hook(lambda *_: None)
    rel, mx = _run(stack, ref, gpu, 1, 1, 40, calls)
    handle.remove()
    assert rel < 3e-5 and mx < 1e-4
    before = ops.exact_fp32_linears(True)
    try:
        rel, mx = _run(stack, ref, gpu, 1, 1, 40, calls)
    finally:
        ops.exact_fp32_linears(before)
    assert rel < 1e-5
    for n in (1, 2, 40):  # upstream's layout; at one token it is the packed one
        rel, mx = _run(stack, ref, gpu, 1, 1, n, calls if n > 1 else [], pack=lambda bias: bias)
        assert rel < 3e-5 and mx < 1e-4
    assert "bmx_token_stack_fwd" not in calls


class _Doubled(nn.Module):
    def forward(self, w):
        return 2 * w


@pytest.mark.parametrize("path", ["pair_bias_attn.proj_q", "transition.swish_gate.0", "transition.b_to_a"])
def test_token_stack_computed_weights(gpu, path):
    """A parametrized linear keeps the per-layer path, which follows its
    parameter from call to call."""
    ref, stack = _stack(gpu)
    calls = []
    wrapped, plain = stack.layers[1].get_submodule(path), ref.layers[1].get_submodule(path)
    parametrize.register_parametrization(wrapped, "weight", _Doubled())
    with torch.no_grad():
        plain.weight.mul_(2)
    for _ in range(2):
        rel, mx = _run(stack, ref, gpu, 1, 1, 40, calls)
        assert rel < 3e-5 and mx < 1e-4
        with torch.no_grad():
            plain.weight.mul_(-0.75)
            wrapped.parametrizations.weight.original.mul_(-0.75)
    assert "bmx_token_stack_fwd" not in calls


def test_token_stack_wide_rows(gpu):
    """32 heads of 48 (1536 channels) are wider than the call's rows."""
    ref, stack = _stack(gpu, heads=32, width=1536)
    calls = []
    rel, mx = _run(stack, ref, gpu, 1, 1, 40, calls)
    assert rel < 3e-5 and mx < 1e-4 and "bmx_token_stack_fwd" not in calls
