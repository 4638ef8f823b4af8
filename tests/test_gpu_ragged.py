"""Triangle modules where n falls between the tiles: the contraction's 64-,
128- and 256-wide tiles with the last ones cut at the planes' end, the
attention core's query blocks past the written rows and its leftover columns,
each against the fp32 oracle on the GPU."""

import pytest
import torch

from boltz_lumi_amd import layers, ops
from oracle import boltz_ref as R

pytestmark = pytest.mark.gpu


def _pair(n, seed, dev):
    g = torch.Generator().manual_seed(seed)
    z = torch.randn(1, n, n, 128, generator=g).to(dev)
    tok = torch.ones(1, n)
    if n > 8:
        tok[:, torch.randperm(n, generator=g)[: n // 16]] = 0
    return z, (tok[:, :, None] * tok[:, None, :]).to(dev)


def _check(mine, ref, z, mask, dev):
    R.randomize(ref, generator=torch.Generator().manual_seed(1))
    mine.load_state_dict(ref.state_dict())
    mine, ref = mine.to(dev).eval(), ref.to(dev).eval()
    n = z.shape[1]
    # a workspace full of NaN bit patterns: nothing unwritten may reach the output
    ws = ops.new_workspace(n, dev)
    ws.fill_(255)
    with torch.inference_mode():
        got = mine(z, mask, workspace=ws).float()
    with torch.no_grad():
        want = ref(z, mask)
    err = ((got - want).abs().max() / want.abs().max()).item()
    assert err < 2e-2, (n, err)  # the bf16 kernels' bar


# np = round_up(n, 64): 64-wide tiles (one and four), 128-wide ones exact and cut, 256-wide ones exact,
# with one 64-wide, one 128-wide and one 192-wide edge
@pytest.mark.parametrize("n", [5, 64, 127, 130, 192, 250, 312, 450, 512, 640, 641, 833, 895, 960])
@pytest.mark.parametrize("outgoing", [True, False])
def test_trimul_between_tiles(gpu, n, outgoing):
    name = "TriangleMultiplicationOutgoing" if outgoing else "TriangleMultiplicationIncoming"
    z, mask = _pair(n, n, gpu)
    _check(getattr(layers, name)(), getattr(R, name)(), z, mask, gpu)


# 1 .. 5 query tiles of 128: 4 to 20 columns over the 8 XCDs, query blocks that end past the written rows
@pytest.mark.parametrize("n", [3, 64, 65, 129, 193, 300, 321, 390, 577])
@pytest.mark.parametrize("starting", [True, False])
def test_triattn_between_tiles(gpu, n, starting):
    z, mask = _pair(n, n, gpu)
    if starting:
        _check(layers.TriangleAttention(), R.TriangleAttention(128, 32, 4, starting=True), z, mask, gpu)
    else:
        _check(layers.TriangleAttentionEndingNode(), R.TriangleAttentionEndingNode(128, 32, 4), z, mask, gpu)
