"""Which modules and calls the stacks' one-call paths accept (CPU: the guards
read modules and shapes, nothing is launched)."""

import copy

import pytest
import torch
import torch.nn.utils.parametrize as parametrize
from torch import nn

from boltz_lumi_amd import adapters, diffusion
from oracle import boltz_ref as R


class Doubled(nn.Module):
    def forward(self, w):
        return 2 * w


def token_stack(heads=16, width=768, depth=1):
    host = nn.Module()
    host.structure_module = nn.Module()
    host.structure_module.score_model = nn.Module()
    host.structure_module.score_model.token_transformer = R.DiffusionTransformer(depth, heads, width, width).eval()
    adapters.install(host, require_boltz2=False, require_device=False)
    return host.structure_module.score_model.token_transformer


def accepted(layer, width=768):
    with torch.inference_mode():
        return diffusion._stack_layer(layer, width)


def test_token_stack_takes_stored_weights_only():
    """A computed weight (parametrize) is no parameter of its module: the pack's
    cache key could not follow it, so the layer keeps the per-layer path; every
    weight and bias of an accepted layer is among its pack's sources."""
    layer = token_stack().layers[0]
    sources = accepted(layer)[-1]
    # the pair bias's projection (a rearrangement) has no parameters; every other parameter is packed
    assert {id(p) for p in sources} == {id(p) for p in layer.parameters()}
    att, tr = layer.pair_bias_attn, layer.transition
    for owner, name in ((att, "proj_q"), (att, "proj_o"), (tr.swish_gate, "0"), (tr, "b_to_a"), (tr, "a_to_b"),
                        (layer.adaln, "s_scale"), (layer.adaln, "s_norm")):
        kept = getattr(owner, name)
        wrapped = copy.deepcopy(kept)
        parametrize.register_parametrization(wrapped, "weight", Doubled())
        setattr(owner, name, wrapped)
        assert accepted(layer) is None, name
        setattr(owner, name, kept)
    assert accepted(layer) is not None


@pytest.mark.parametrize("heads,width,taken", [(16, 768, True), (32, 32 * 32, True), (32, 32 * 48, False),
                                               (22, 22 * 48, False)])
def test_token_stack_width_limit(heads, width, taken):
    """The call takes rows of at most 1024; wider layers, which AttentionPairBias
    alone would allow (64 heads of 48), keep the per-layer path."""
    layer = token_stack(heads, width).layers[0]
    assert (accepted(layer, width) is not None) == taken
