"""fp32-mode triangle attention's projection kernel at the edges of its 64-pair
tiles, in blocks of rows, with and without a mask, against the oracle module
in fp32 on the GPU."""

import pytest
import torch

from boltz_lumi_amd import ops
from oracle import boltz_ref as R

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 2, 31, 63, 64, 65, 129, 200])
@pytest.mark.parametrize("starting", [True, False])
@pytest.mark.parametrize("masked", [None, "tokens", "random"])
def test_fp32_projection_edges(gpu, n, starting, masked):
    g = torch.Generator().manual_seed(n + 3 * starting)
    cls = R.TriangleAttention if starting else R.TriangleAttentionEndingNode
    layer = R.randomize(cls(128, 32, 4), generator=g).to(gpu).eval()
    x = torch.randn(n, n, 128, generator=g).to(gpu)
    mask = None
    if masked == "tokens":  # padded tokens: closed rows too
        tok = torch.ones(n)
        tok[n - n // 5:] = 0
        mask = (tok[:, None] * tok[None, :]).to(gpu)
    elif masked == "random":
        mask = (torch.rand(n, n, generator=g) > 0.3).float().to(gpu)
    with torch.inference_mode():
        got = ops.triattn_fp32(layer, x, mask, starting)
        blocked = ops.triattn_fp32(layer, x, mask, starting, block_rows=max(1, n // 3))
        want = layer(x[None], None if mask is None else mask[None])[0]
    assert torch.isfinite(got).all()
    # the same products row by row; linear_o's library GEMM sums its 128 fp32 products in an order that depends on
    # its shape (2^-24 each)
    assert (got - blocked).abs().max() / got.abs().max() < 1e-6
    err = ((got - want).abs().max() / want.abs().max()).item()
    assert err < 1e-4, err  # split products: 2^-16 relative each


@pytest.mark.parametrize("n,scale,closed", [(97, 1.0, 70), (97, 1.0, 33), (130, 200.0, 0), (130, 200.0, 5), (1090, 1.0, 3)])
def test_fp32_attention_offsets(gpu, n, scale, closed):
    """The attention's shared offset comes from the first 32 keys: keys closed
    before the open ones, scores far above the first keys' (a triangle bias of
    hundreds), and more than one group of query tiles."""
    g = torch.Generator().manual_seed(n + closed)
    layer = R.randomize(R.TriangleAttention(128, 32, 4), generator=g).to(gpu).eval()
    x = torch.randn(n, n, 128, generator=g).to(gpu)
    with torch.no_grad():
        layer.linear.weight.mul_(scale)
    mask = torch.ones(n, n, device=gpu)
    mask[::3, :closed] = 0
    with torch.inference_mode():
        got = ops.triattn_fp32(layer, x, mask, True)
        want = layer(x[None], mask[None], chunk_size=64)[0]
        top = layer.linear(layer.layer_norm(x)).abs().max().item()
    err = ((got - want).abs().max() / want.abs().max()).item()
    print(f"n={n} scale={scale} closed={closed}: largest bias {top:.1f}, error {err:.2e}", flush=True)
    assert scale == 1.0 or top > 100
    # split products: 2^-16 relative each; an error of a score is a relative error of its probability
    assert err < max(1e-4, 2 * 2**-16 * top)


@pytest.mark.parametrize("rows", [1, 63, 64, 65, 127, 40000])
@pytest.mark.parametrize("in_place", [True, False])
def test_linear128(gpu, rows, in_place):
    from boltz_lumi_amd import _native as N

    g = torch.Generator().manual_seed(rows)
    x, w, b = (torch.randn(*s, generator=g).to(gpu) for s in ((rows + 1, 128), (128, 128), (128,)))
    want = torch.nn.functional.linear(x.double(), w.double(), b.double())
    out = x.clone() if in_place else torch.full_like(x, 7.0)
    src = out if in_place else x
    N.call("bmx_linear128_f32_fwd", src.data_ptr(), rows, w.data_ptr(), b.data_ptr(), out.data_ptr(),
           torch.cuda.current_stream().cuda_stream)
    # 128 fp32 products and sums: 128 * 2^-24 of the sum of magnitudes at most
    bound = 128 * 2**-24 * (x.double().abs() @ w.double().abs().t() + b.double().abs())
    assert ((out.double() - want).abs() <= bound)[:rows].all()
    assert torch.equal(out[rows], x[rows] if in_place else torch.full_like(x[rows], 7.0))  # the row past the end
