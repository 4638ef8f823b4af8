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
    # Blocks of an even number of rows pair the rows as one pass does: the same values. A block of one row shares the
    # offset of the scores with no other, so they round otherwise by some 2^-24, and a probability whose high or low
    # part then rounds to the other side keeps another residue: 2^-18 relative on each side.
    apart = ((got - blocked).abs().max() / got.abs().max()).item()
    assert apart == 0 if n // 3 > 1 else apart < 2**-17
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


def _separate_passes(layer, x, mask):
    """The same attention from separate passes: LayerNorm split operand, library
    GEMM of the folded weights, general split-bf16 attention, fp32 output GEMM."""
    n, mha, ln = x.shape[0], layer.mha, layer.layer_norm
    lins = (mha.linear_q, mha.linear_k, mha.linear_v, mha.linear_g, layer.linear)
    w = torch.cat([lin.weight for lin in lins] + [x.new_zeros(60, 128)])  # a multiple of 64 outputs
    b = torch.cat([lin.bias if lin.bias is not None else x.new_zeros(lin.out_features) for lin in lins]
                  + [x.new_zeros(60)]) + w @ ln.bias
    proj = ops.mm_split(ops.layernorm_split3(x.view(-1, 128), ln.eps), ops._x3_weight(w * ln.weight, b)).view(n, n, -1)
    q, k, v, g = proj[..., :512].split(128, dim=-1)
    bias = proj[..., 512:516].permute(2, 0, 1).contiguous()
    o = ops.seq_attention_batched(q, k, v, bias[None], mask, g, layer.inf, bias_div=n, split=True)
    return torch.nn.functional.linear(o, mha.linear_o.weight, mha.linear_o.bias)


@pytest.mark.parametrize("n", [17, 40, 97, 200])
def test_fp32_error_against_separate_passes(gpu, n):
    """No further from 64 bits than the passes that the kernels replace (the
    whole-number offset of the scores costs the largest probability its exact 1;
    the projection's fourth product, low by low, gives more back)."""
    g = torch.Generator().manual_seed(n)
    layer = R.TriangleAttention(128, 32, 4).eval()
    with torch.no_grad():
        for name, p in layer.named_parameters():
            r = torch.randn(p.shape, generator=g)
            p.copy_(1 + 0.08 * r if "norm" in name and name.endswith("weight")
                    else r / p.shape[1] ** 0.5 if p.dim() == 2 else 0.08 * r)
    layer, x, mask = layer.to(gpu), torch.randn(n, n, 128, generator=g).to(gpu), torch.ones(n, n, device=gpu)
    with torch.inference_mode():
        got, separate = ops.triattn_fp32(layer, x, mask, True), _separate_passes(layer, x, mask)
        want = layer.double()(x.double()[None], mask.double()[None])[0]
    err, err_separate = (((y.double() - want).norm() / want.norm()).item() for y in (got, separate))
    print(f"n={n}: {err:.3e}, separate passes {err_separate:.3e}", flush=True)
    assert err <= err_separate < 2e-5
