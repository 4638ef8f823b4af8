"""The pair transition's 32-, 64- and 128-row tiles at their edges and around the
row counts where the tile changes (two blocks per CU of 32 and of 64 rows),
with and without the fused pair bias, against the fp32 oracle and against
the same rows inside a larger call."""

import pytest
import torch

from boltz_lumi_amd import layers, ops
from oracle import boltz_ref as R

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows", [1, 31, 33, 1000, "32x2cu", "32x2cu+1", "64x2cu", "64x2cu+1"])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_transition_tiles(gpu, rows, dtype):
    if isinstance(rows, str):
        base, _, more = rows.partition("+")
        rows = int(base.split("x")[0]) * 2 * torch.cuda.get_device_properties(gpu).multi_processor_count + int(more or 0)
    g = torch.Generator().manual_seed(4)
    ref = R.randomize(R.Transition(128, 512), generator=g).to(gpu).eval()
    mine = layers.Transition().to(gpu).eval()
    mine.load_state_dict(ref.state_dict())
    proj = R.randomize(R.AttentionPairBias(384, 128, 16), generator=g).to(gpu).eval().proj_z
    big = 64 * 2 * torch.cuda.get_device_properties(gpu).multi_processor_count + 200  # 128-row tiles
    x = torch.randn(big, 128, generator=g).to(gpu).to(dtype)
    with torch.inference_mode():
        want = ref(x[:rows].float())
        got = mine(x[:rows].contiguous(), out_mode=ops.OUT_F32)
        whole = mine(x, out_mode=ops.OUT_F32)[:rows]
        assert ((got - want).abs().max() / want.abs().max()).item() < 2e-2
        assert torch.equal(got, whole)  # a row's arithmetic does not depend on the tile
        bias = torch.empty(16, rows, device=gpu)
        out = ops.pair_transition(mine, x[:rows].contiguous(), ops.OUT_RESIDUAL, pair_bias=(proj[0], proj[1], bias))
        assert torch.equal(out, x[:rows].float() + got)
        pb = proj[1](proj[0](out)).t()
        assert ((bias - pb).abs().max() / pb.abs().max()).item() < 1e-4
