"""Which modules and calls the stacks' one-call paths accept (CPU: the guards
read modules and shapes, nothing is launched)."""

import copy

import pytest
import torch
import torch.nn.utils.parametrize as parametrize
from torch import nn

from boltz_lumi_amd import _native, adapters, diffusion, layers, ops, pairformer
from boltz_lumi_amd.pair_bias import prepare_token_bias
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


class Calls:
    """``ops`` on CPU tensors with every native call recorded instead of made."""

    def __init__(self, monkeypatch, devices=False):
        if not _native.lib_path().exists():
            pytest.skip("libbmx.so not built")
        self.made = []
        monkeypatch.setattr(_native, "call", lambda name, *args: self.made.append((name, args)))
        if not devices:
            monkeypatch.setattr(ops, "_cuda", lambda *_: None)
        monkeypatch.setattr(ops, "_stream", lambda _: 0)

    def __getitem__(self, name):
        return [args for made, args in self.made if made == name]


def offset(t):
    """``t``'s values as a contiguous view at a 4-byte storage offset."""
    flat = torch.empty(t.numel() + 4)
    start = next(i for i in range(1, 5) if (flat.data_ptr() + 4 * i) % 16 == 4)
    return flat[start:start + t.numel()].view(t.shape).copy_(t)


def sequence_layer():
    layer = layers.PairformerLayer().eval()
    for p in layer.parameters():
        p.requires_grad_(False)
    return layer


def sequence_call(layer, s):
    b, n = s.shape[:2]
    params, hidden = pairformer._native_sequence_params(layer, s.device)
    return ops.sequence_stack(s, params, 1e-5, 1e-5, torch.zeros(b, 16, n, n), torch.ones(b, n), 16, hidden, 1e6)


def test_sequence_stack_operands_are_aligned(monkeypatch):
    """Contiguous parameters and activations at any storage offset: what the call
    gets is 16-byte aligned."""
    layer, s = sequence_layer(), offset(torch.randn(1, 5, 384))
    with torch.no_grad():
        for module in layer.modules():
            for name, p in list(module.named_parameters(recurse=False)):
                setattr(module, name, nn.Parameter(offset(p), requires_grad=False))
    assert all(p.data_ptr() % 16 == 4 for p in layer.attention.parameters())
    calls = Calls(monkeypatch)
    with torch.inference_mode():
        sequence_call(layer, s)
    assert len(calls["bmx_f32_pack"]) == 8 and all(args[0] % 16 == 0 for args in calls["bmx_f32_pack"])
    (args,) = calls["bmx_sequence_stack_fwd"]
    assert args[0] % 16 == 0 and all((p or 0) % 16 == 0 for p in args[6])


def test_sequence_stack_limits():
    """What the call refuses (an eps of 0) and rows past its line keep torch's path."""
    layer = sequence_layer()
    for norm in (layer.pre_norm_s, layer.transition_s.norm):
        kept, norm.eps = norm.eps, 0.0
        assert pairformer._native_sequence_params(layer, torch.device("cpu")) is None
        norm.eps = kept
    line = pairformer.SEQUENCE_MAX_ROWS
    for b, n, native in ((1, 1, True), (1, line, True), (line // 64, 64, True), (line, 1, True), (0, 5, False), (5, 0, False),
                         (1, line + 1, False), (line // 64 + 1, 64, False), (65536, 32, False)):
        assert pairformer._native_sequence_rows(b, n) == native, (b, n)


def test_packs_refuse_host_weights(monkeypatch):
    """The packs hand raw addresses to a kernel: host tensors are refused."""
    calls = Calls(monkeypatch, devices=True)
    with pytest.raises(RuntimeError, match="CUDA"):
        ops.x3_pack(torch.empty(2 * 32 * 64, dtype=torch.bfloat16), 0, torch.zeros(32, 64))
    with pytest.raises(RuntimeError, match="CUDA"):
        ops.f32_pack(32, 64, (0, 1, torch.zeros(32, 64)))
    assert not calls.made


def test_packs_refuse_what_does_not_fit(monkeypatch):
    """A weight whose 32-row tiles lie past the packed operand, or of another
    width, is refused before the kernel writes; the last tile that fits is not."""
    calls = Calls(monkeypatch)
    out = torch.empty(2 * 96 * 64, dtype=torch.bfloat16)  # three tiles of 32 x 64
    ops.x3_pack(out, 1, torch.zeros(64, 64))
    ops.x3_pack(out, 0, torch.zeros(64, 64), tile_stride=2, col_scale=torch.ones(64))
    ops.f32_pack(96, 64, (0, 2, torch.zeros(64, 64)), (1, 1, torch.zeros(32, 64)))
    assert len(calls.made) == 4
    for tile0, stride, rows, cols, scale in ((2, 1, 64, 64, None), (1, 2, 64, 64, None), (0, 1, 96, 96, None),
                                             (0, 1, 33, 64, None), (0, 1, 32, 64, 32)):
        with pytest.raises(RuntimeError):
            ops.x3_pack(out, tile0, torch.zeros(rows, cols), stride, None if scale is None else torch.ones(scale))
    for tile0, stride, rows, cols in ((2, 1, 64, 64), (1, 2, 64, 64), (0, 1, 32, 96), (0, 1, 33, 64)):
        with pytest.raises(RuntimeError):
            ops.f32_pack(96, 64, (tile0, stride, torch.zeros(rows, cols)))
    assert len(calls.made) == 4


@pytest.mark.parametrize("path", ["pair_bias_attn.proj_k", "transition.a_to_b", "output_projection_linear"])
def test_token_stack_refuses_mismatched_projections(monkeypatch, path):
    """A projection of another output width fills only a part of its pack: it
    is refused, as the per-layer path's GEMM refuses it."""
    layer = token_stack().layers[0]
    Calls(monkeypatch)
    *parents, name = path.split(".")
    owner = layer.get_submodule(".".join(parents))
    kept = getattr(owner, name)
    narrow = nn.Linear(kept.in_features, kept.out_features - 32, bias=kept.bias is not None)
    narrow.out_features = kept.out_features
    setattr(owner, name, narrow)
    if path == "output_projection_linear":
        layer.output_projection[0] = narrow
    with torch.inference_mode(), pytest.raises(RuntimeError, match="does not match"):
        diffusion._stack_pack(layer, 768, 1536)


def fp32_call(module, x, mask, starting, rows=None):
    n = x.shape[0]
    with torch.inference_mode():
        return ops._triattn_fp32_split(module, x, mask, starting, n if rows is None else rows)


def test_fp32_triangle_attention_refuses_host_tensors(monkeypatch):
    calls = Calls(monkeypatch, devices=True)
    layer = R.TriangleAttention(128, 32, 4).eval()
    with pytest.raises(RuntimeError, match="CUDA"):
        fp32_call(layer, torch.zeros(5, 5, 128), None, True)
    assert not calls.made


def test_fp32_triangle_attention_masks(monkeypatch):
    """[N, N], or one row for all rows of the frame (x's columns for the ending
    node); the kernel reads N x N values. Other shapes are refused."""
    calls = Calls(monkeypatch)
    seen = []
    real = ops._triattn_fp32_native
    monkeypatch.setattr(ops, "_triattn_fp32_native", lambda m, w, x, mask, *a: seen.append(mask) or real(m, w, x, mask, *a))
    n, row = 5, torch.rand(5)
    for starting in (True, False):
        layer = (R.TriangleAttention if starting else R.TriangleAttentionEndingNode)(128, 32, 4).eval()
        x = torch.zeros(n, n, 128)
        for mask in (torch.rand(n, n), torch.rand(n, n) > 0.5, row[None] if starting else row[:, None]):
            fp32_call(layer, x, mask, starting)
            got = seen.pop()
            assert got.dtype == torch.float32 and got.is_contiguous() and torch.equal(got, mask.float().expand(n, n))
        made = len(calls.made)
        for mask in (row, torch.rand(n, n + 1), torch.rand(n + 1, n), row[:, None] if starting else row[None],
                     torch.rand(1, n, n)):
            with pytest.raises(RuntimeError, match="mask"):
                fp32_call(layer, x, mask, starting)
        assert len(calls.made) == made


def test_fp32_triangle_attention_refuses_other_widths(monkeypatch):
    calls = Calls(monkeypatch)
    x = torch.zeros(5, 5, 128)
    for path, module in (("mha.linear_k", nn.Linear(128, 96, bias=False)), ("linear", nn.Linear(128, 3, bias=False)),
                         ("mha.linear_o", nn.Linear(96, 128)), ("layer_norm", nn.LayerNorm(64))):
        layer = R.TriangleAttention(128, 32, 4).eval()
        *parents, name = path.split(".")
        setattr(layer.get_submodule(".".join(parents)), name, module)
        with pytest.raises(RuntimeError, match="expected"):
            fp32_call(layer, x, None, True)
    assert not [name for name, _ in calls.made if name != "bmx_x3_pack"]


@pytest.mark.parametrize("n,rows", [(9, 9), (9, 4), (9, 1)])
def test_fp32_triangle_attention_packs_once_per_call(monkeypatch, n, rows):
    """Inference-tensor weights carry no version counter, so every call packs
    them again: once, however many blocks of rows it runs in."""
    calls = Calls(monkeypatch)
    with torch.inference_mode():
        layer = R.TriangleAttention(128, 32, 4).eval()
        for _ in range(2):
            calls.made.clear()
            ops._triattn_fp32_split(layer, torch.zeros(n, n, 128), None, True, rows)
            assert len(calls["bmx_x3_pack"]) == 4
            assert len(calls["bmx_linear128_f32_fwd"]) == -(-n // rows)


def test_token_stack_bias_layout(monkeypatch):
    """Only a bias as ``prepare_token_bias`` packs it goes to the call, which
    reads it as dense [heads, N, N] elements; another one is seen before the
    layers are looked at."""
    stack, n = token_stack(depth=2), 6
    Calls(monkeypatch)
    walked, given = [], []
    real = diffusion._stack_layer
    monkeypatch.setattr(diffusion, "_stack_layer", lambda *a: walked.append(1) or real(*a))
    monkeypatch.setattr(diffusion, "_stack_pack", lambda *_: (None,) * 10)
    monkeypatch.setattr(ops, "token_stack", lambda a, s, addresses, *_: given.append(addresses[10::11]) or a)
    a, mask = torch.zeros(2, n, 768), torch.ones(2, n)
    raw = torch.randn(1, n, n, 32)

    def call(bias):
        walked.clear()
        given.clear()
        with torch.inference_mode():
            diffusion._native_stack(list(stack.layers), a, a, bias.view(1, n, n, 2, 16), mask, 2)
        return bool(given), len(walked)

    packed = prepare_token_bias(raw)
    assert call(packed) == (True, 2)
    assert given[0] == [packed.data_ptr(), packed.data_ptr() + 4 * 16 * n * n]
    for other in (raw, raw.transpose(1, 2).contiguous().transpose(1, 2), packed.transpose(1, 2), packed.double()):
        assert call(other) == (False, 0)
