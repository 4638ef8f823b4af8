"""Timed cases of the framework's public entry points.

A case is a dict of plain values.  ``prepare`` builds what a user's program
holds before the call (modules with weights, activations, masks, biases, all on
the GPU and all from the seed), ``run`` is one pass through the public entry
points, ``exact`` the same outputs from plain torch in 64 bits, ``work`` the
bytes and operations that one pass cannot do without.

Kinds of case:
  layer       boltz_lumi_amd.layers.PairformerLayer: one trunk block, whole
  triattn     layers.TriangleAttention / TriangleAttentionEndingNode, bf16 out
  triattn32   the installed TriangleAttention in fp32 mode (autocast off)
  trimul      layers.TriangleMultiplicationOutgoing / Incoming, bf16 out
  transition  layers.Transition, the 128 -> 512 -> 128 pair instance, bf16 out
  tokens      the score model's DiffusionTransformer after install(): layers of
              AdaLN, pair-biased attention (16 x 48) and conditioned transition
  atoms       the score model's AtomTransformer after install(): windows of 32
              query atoms over 128 key atoms (4 x 32), 3 layers

Everything here is inference: the framework runs no backward of its own (under
grad its modules call the upstream forward).
"""

import math

import torch
from torch import nn
import torch.nn.functional as F

from boltz_lumi_amd import adapters, layers
from boltz_lumi_amd.pair_bias import prepare_token_bias, prepare_window_bias

C = 128                       # pair channels
C_S, HEADS_S = 384, 16        # single channels and heads of the sequence stack
D_TOK, HEADS_TOK = 768, 16    # token transformer
D_ATOM, HEADS_ATOM, ATOM_LAYERS = 128, 4, 3
WINDOW, KEYS = 32, 128        # atom transformer: queries and keys of a window
LAYER_MAX_N, FP32_MAX_N = 1134, 576


# --------------------------------------------------------------------- cases


def listed():
    return [
        # a small target (117 tokens, the last 3 padded): a trunk block where latency and launches count
        {"name": "layer_n117", "kind": "layer", "n": 117, "pad": 3},
        # an ordinary single chain, no padding, an odd size
        {"name": "layer_n312", "kind": "layer", "n": 312, "pad": 0},
        # the largest published target of the trunk (1134 tokens, ragged against every tile)
        {"name": "layer_n1134", "kind": "layer", "n": 1134, "pad": 3},
        # triangle attention of a padded batch element: the last 10% of the tokens are padding
        {"name": "triattn_start_n512", "kind": "triattn", "n": 512, "pad": 51, "starting": True},
        # the headline trunk size, the transposed direction
        {"name": "triattn_end_n1024", "kind": "triattn", "n": 1024, "pad": 0, "starting": False},
        # fp32 mode, as a user without autocast runs it
        {"name": "triattn32_start_n576", "kind": "triattn32", "n": 576, "pad": 3, "starting": True},
        # triangle multiplication with 5% of the tokens masked anywhere
        {"name": "trimul_out_n768", "kind": "trimul", "n": 768, "masked": 38, "outgoing": True},
        # ... and of an ordinary chain, the other direction
        {"name": "trimul_in_n312", "kind": "trimul", "n": 312, "masked": 0, "outgoing": False},
        # the pair transition alone (MSA and trunk blocks call it as a module too)
        {"name": "transition_n1024", "kind": "transition", "n": 1024},
        # two blocks of the denoiser's token transformer at the sampler's full load: 5 samples of 1024 tokens
        {"name": "tokens_5x1024", "kind": "tokens", "n": 1024, "samples": 5, "depth": 2, "pad": 0},
        # the whole 24-block token transformer for one sample of a small target
        {"name": "tokens24_1x117", "kind": "tokens", "n": 117, "samples": 1, "depth": 24, "pad": 3},
        # the atom encoder / decoder stack: 5 samples of 8192 atoms
        {"name": "atoms_5x8192", "kind": "atoms", "atoms": 8192, "samples": 5},
    ]


def _log_int(rng, lo, hi):
    return min(hi, max(lo, round(math.exp(rng.uniform(math.log(lo), math.log(hi))))))


def draw(rng):
    kind = rng.choice(["layer", "layer", "triattn", "triattn", "triattn32", "trimul", "trimul", "transition", "tokens",
                       "tokens", "atoms"])
    if kind == "layer":
        n = _log_int(rng, 17, LAYER_MAX_N)
        return {"kind": kind, "n": n, "pad": rng.choice([0, 3, n // 10])}
    if kind == "triattn":
        n = _log_int(rng, 17, LAYER_MAX_N)
        return {"kind": kind, "n": n, "pad": rng.choice([0, 3, n // 10]), "starting": rng.random() < 0.5}
    if kind == "triattn32":
        n = _log_int(rng, 17, FP32_MAX_N)
        return {"kind": kind, "n": n, "pad": rng.choice([0, 3]), "starting": rng.random() < 0.5}
    if kind == "trimul":
        n = _log_int(rng, 17, LAYER_MAX_N)
        return {"kind": kind, "n": n, "masked": rng.choice([0, n // 20]), "outgoing": rng.random() < 0.5}
    if kind == "transition":
        return {"kind": kind, "n": _log_int(rng, 17, LAYER_MAX_N)}
    if kind == "tokens":
        n = _log_int(rng, 17, 1024)
        return {"kind": kind, "n": n, "samples": rng.choice([1, 5]), "depth": 2, "pad": rng.choice([0, 3])}
    return {"kind": "atoms", "atoms": WINDOW * _log_int(rng, 8, 256), "samples": rng.choice([1, 5])}


# ------------------------------------------------------- modules and inputs


class DiffusionTransformerLayer(nn.Module):
    """Parameters of Boltz's layer of the same name; install() gives it its forward."""

    def __init__(self, heads, dim):
        super().__init__()
        self.adaln = layers.AdaLN(dim, dim)
        self.pair_bias_attn = layers.AttentionPairBias(c_s=dim, num_heads=heads, compute_pair_bias=False)
        self.output_projection_linear = nn.Linear(dim, dim)
        self.output_projection = nn.Sequential(self.output_projection_linear, nn.Sigmoid())
        self.transition = layers.ConditionedTransitionBlock(dim, dim)
        self.post_lnorm = nn.Identity()


class DiffusionTransformer(nn.Module):
    def __init__(self, depth, heads, dim):
        super().__init__()
        self.layers = nn.ModuleList([DiffusionTransformerLayer(heads, dim) for _ in range(depth)])


class AtomTransformer(nn.Module):
    def __init__(self):
        super().__init__()
        self.attn_window_queries, self.attn_window_keys = WINDOW, KEYS
        self.diffusion_transformer = DiffusionTransformer(ATOM_LAYERS, HEADS_ATOM, D_ATOM)


class Boltz2(nn.Module):
    """A model with one module at its Boltz path, for install()."""

    def __init__(self, path, module):
        super().__init__()
        at = self
        *parents, last = path.split(".")
        for name in parents:
            child = nn.Module()
            setattr(at, name, child)
            at = child
        setattr(at, last, module)


def _device():
    return torch.device("cuda", torch.cuda.current_device()) if torch.cuda.is_available() else torch.device("cpu")


def _module(case):
    kind = case["kind"]
    if kind == "layer":
        return layers.PairformerLayer(C_S, C, HEADS_S)
    if kind in ("triattn", "triattn32"):
        return layers.TriangleAttention() if case["starting"] else layers.TriangleAttentionEndingNode()
    if kind == "trimul":
        return layers.TriangleMultiplicationOutgoing() if case["outgoing"] else layers.TriangleMultiplicationIncoming()
    if kind == "transition":
        return layers.Transition()
    if kind == "tokens":
        return DiffusionTransformer(case["depth"], HEADS_TOK, D_TOK)
    return AtomTransformer()


def _weights(module, g, dev):
    """Weights N(0, 1 / fan_in), norm weights N(1, 0.08), vectors N(0, 0.08): a
    trained network's scale, so that stacks of residual blocks stay bounded."""
    with torch.no_grad():
        for name, p in module.named_parameters():
            r = torch.randn(p.shape, generator=g, device=dev)
            if "norm" in name and name.endswith("weight"):
                p.copy_(1 + 0.08 * r)
            elif p.dim() == 2:
                p.copy_(r / math.sqrt(p.shape[1]))
            else:
                p.copy_(0.08 * r)
    return module


def _token_mask(n, pad, dev):
    m = torch.ones(1, n, device=dev)
    if pad:
        m[:, n - pad:] = 0
    return m


def _inputs(case, seed):
    """(module, inputs) on the device, from the seed alone."""
    dev = _device()
    g = torch.Generator(device=dev).manual_seed(int(seed))
    kind = case["kind"]

    def rand(*shape):
        return torch.randn(shape, generator=g, device=dev)

    with torch.device(dev):
        module = _module(case).eval()
    _weights(module, g, dev)
    t = {}
    if kind == "layer":
        n = case["n"]
        t["mask"] = _token_mask(n, case["pad"], dev)
        t["pair_mask"] = t["mask"][:, :, None] * t["mask"][:, None, :]
        t["z"], t["s"] = rand(1, n, n, C), rand(1, n, C_S)
    elif kind in ("triattn", "triattn32", "trimul"):
        n = case["n"]
        m = _token_mask(n, case.get("pad", 0), dev)
        if case.get("masked"):
            m[:, torch.randperm(n, generator=g, device=dev)[:case["masked"]]] = 0
        t["pair_mask"] = m[:, :, None] * m[:, None, :]
        t["z"] = rand(1, n, n, C)
    elif kind == "transition":
        t["z"] = rand(1, case["n"], case["n"], C)
    elif kind == "tokens":
        n, b = case["n"], case["samples"]
        t["a"], t["s"] = rand(b, n, D_TOK), rand(b, n, D_TOK)
        t["bias"] = rand(1, n, n, case["depth"] * HEADS_TOK)
        t["mask"] = _token_mask(n, case["pad"], dev).expand(b, n).contiguous()
    else:
        n, b = case["atoms"], case["samples"]
        t["q"], t["c"] = rand(b, n, D_ATOM), rand(b, n, D_ATOM)
        t["bias"] = rand(1, n // WINDOW, WINDOW, KEYS, ATOM_LAYERS * HEADS_ATOM)
        t["mask"] = torch.ones(b, n, device=dev)
    return module, t


def _key_windows(x):
    """[B, N, D] atom rows to [B, N / 32, 128, D]: the 128 atoms centred on each
    window of 32, zero rows past the ends (Boltz's single_to_keys)."""
    side = (KEYS - WINDOW) // 2
    return F.pad(x, (0, 0, side, side)).unfold(1, KEYS, WINDOW).transpose(2, 3)


def prepare(case, seed):
    module, t = _inputs(case, seed)
    kind = case["kind"]
    if kind == "triattn32":
        adapters.install(Boltz2("pairformer_module.tri_att", module))
    elif kind == "tokens":
        adapters.install(Boltz2("structure_module.score_model.token_transformer", module))
        t["bias"] = prepare_token_bias(t["bias"])  # as the sampler stores it, once per sampling call
    elif kind == "atoms":
        adapters.install(Boltz2("structure_module.score_model.atom_encoder", module))
        t["bias"] = prepare_window_bias(t["bias"])

    def to_keys(x):
        return _key_windows(x)

    return {"case": case, "module": module, "t": t, "to_keys": to_keys}


def run(state):
    case, m, t = state["case"], state["module"], state["t"]
    kind = case["kind"]
    with torch.inference_mode():
        if kind == "layer":
            s, z = m(t["s"], t["z"], t["mask"], t["pair_mask"])
            return {"s": s, "z": z}
        if kind in ("triattn", "triattn32", "trimul"):
            return m(t["z"], t["pair_mask"])
        if kind == "transition":
            return m(t["z"])
        if kind == "tokens":
            return m(t["a"], t["s"], t["bias"], t["mask"], multiplicity=case["samples"])
        return m(t["q"], t["c"], t["bias"], state["to_keys"], t["mask"], multiplicity=case["samples"])


# -------------------------------------------------------------- work, limits


def _attn_flops(n):
    return 512 * n**3 + 164864 * n * n


def _mul_flops(n):
    return 256 * n**3 + 196608 * n * n


def work(case):
    kind = case["kind"]
    if kind == "layer":
        n = case["n"]
        seq = 2 * n * C_S * (5 * C_S + 3 * 4 * C_S) + 4 * C_S * n * n
        flops = 2 * _attn_flops(n) + 2 * _mul_flops(n) + 2 * C * (12 * C + HEADS_S) * n * n + seq
        return {"bytes": n * n * (2 * 4 * C + 4) + 2 * 4 * C_S * n + 4 * (17 * C_S * C_S + 24 * C * C), "flops": flops}
    if kind in ("triattn", "trimul"):
        n = case["n"]
        return {"bytes": n * n * (4 * C + 4 + 2 * C) + 4 * 6 * C * C,
                "flops": _attn_flops(n) if kind == "triattn" else _mul_flops(n)}
    if kind == "triattn32":
        n = case["n"]
        return {"bytes": n * n * (8 * C + 4) + 4 * 6 * C * C, "flops": _attn_flops(n)}
    if kind == "transition":
        n = case["n"]
        return {"bytes": n * n * 6 * C + 4 * 12 * C * C, "flops": 24 * C * C * n * n}
    if kind == "tokens":
        n, b, d, depth = case["n"], case["samples"], D_TOK, case["depth"]
        per_layer = 2 * b * n * d * d * (4 + 2 + 4 + 1 + 6 + 2) + 4 * b * d * n * n
        return {"bytes": 4 * (3 * b * n * d + b * n + depth * (HEADS_TOK * n * n + 19 * d * d)),
                "flops": depth * per_layer}
    n, b, d = case["atoms"], case["samples"], D_ATOM
    per_layer = 2 * b * n * d * d * (4 + 2 + 4 + 1 + 6 + 2) + 4 * b * d * n * KEYS
    return {"bytes": 4 * (3 * b * n * d + b * n + ATOM_LAYERS * (HEADS_ATOM * n * KEYS + 19 * d * d)),
            "flops": ATOM_LAYERS * per_layer}


def tolerance(case):
    return TOLERANCE[case["kind"]]


# About four times what each path differs from ``exact`` by, over the listed and
# drawn sizes (2-norm / largest): layer z 4.7e-3 / 3.2e-2, triattn 4.8e-3 / 5.4e-2,
# trimul 5.5e-3 / 5.1e-2 and transition 4.5e-3 / 3.0e-2 (bf16 products and
# operands); the fp32 modes, whose products are split bf16, triattn32
# 8.3e-6 / 7.8e-5, tokens 6.9e-6 / 4.5e-5 (24 blocks 1.4e-5 / 6.6e-5), atoms
# 8.2e-6 / 8.0e-5.
TOLERANCE = {
    "layer": {"rel": 1.8e-2, "max": 0.13},
    "triattn": {"rel": 1.9e-2, "max": 0.22},
    "trimul": {"rel": 2.2e-2, "max": 0.2},
    "transition": {"rel": 1.8e-2, "max": 0.12},
    "triattn32": {"rel": 3.3e-5, "max": 3.1e-4},
    "tokens": {"rel": 5.5e-5, "max": 2.6e-4},
    "atoms": {"rel": 3.3e-5, "max": 3.2e-4},
}


# --------------------------------------------------------------------- exact


def _rows(x, f, rows):
    """``f`` over blocks of ``rows`` leading rows of ``x`` in 64 bits."""
    return torch.cat([f(x[i:i + rows].double()) for i in range(0, x.shape[0], rows)])


def _lin(x, linear):
    return F.linear(x, linear.weight.double(), None if linear.bias is None else linear.bias.double())


def _norm(x, m, eps=None):
    w = getattr(m, "weight", None)
    b = getattr(m, "bias", None)
    return F.layer_norm(x, x.shape[-1:], None if w is None else w.double(), None if b is None else b.double(),
                        m.eps if eps is None else eps)


def _block(n, columns):
    """Rows of an [n, n, columns] 64-bit frame that make at most 128 MB."""
    return max(1, (1 << 24) // (n * columns))


def _exact_trimul(m, x, mask, outgoing):
    n = x.shape[0]
    rows = _block(n, 4 * C)

    def gated(xb, mb):
        xn = _norm(xb, m.norm_in)
        return _lin(xn, m.p_in) * torch.sigmoid(_lin(xn, m.g_in)) * mb[..., None]

    a = torch.empty(C, n, n, device=x.device, dtype=torch.float64)
    b = torch.empty_like(a)
    for i in range(0, n, rows):
        p = gated(x[i:i + rows].double(), mask[i:i + rows].double())
        a[:, i:i + rows], b[:, i:i + rows] = p[..., :C].permute(2, 0, 1), p[..., C:].permute(2, 0, 1)
    for c in range(C):
        a[c] = a[c] @ b[c].t().contiguous() if outgoing else a[c].t().contiguous() @ b[c]
    del b
    out = torch.empty(n, n, C, device=x.device, dtype=torch.float64)
    for i in range(0, n, rows):
        o = _norm(a[:, i:i + rows].permute(1, 2, 0).contiguous(), m.norm_out)
        xn = _norm(x[i:i + rows].double(), m.norm_in)
        out[i:i + rows] = _lin(o, m.p_out) * torch.sigmoid(_lin(xn, m.g_out))
    return out


def _exact_triattn(m, x, mask, starting):
    if not starting:
        x, mask = x.transpose(0, 1).contiguous(), mask.transpose(0, 1).contiguous()
    n, h, d = x.shape[0], m.no_heads, m.c_hidden
    bias = torch.empty(h, n, n, device=x.device, dtype=torch.float64)
    rows = _block(n, 4 * C)
    for i in range(0, n, rows):
        bias[:, i:i + rows] = _lin(_norm(x[i:i + rows].double(), m.layer_norm), m.linear).permute(2, 0, 1)
    out = torch.empty(n, n, C, device=x.device, dtype=torch.float64)
    rows = max(1, min(rows, (1 << 24) // (h * n * n)))
    for i in range(0, n, rows):
        xn = _norm(x[i:i + rows].double(), m.layer_norm)
        r = xn.shape[0]
        q, k, v = (_lin(xn, lin).view(r, n, h, d).transpose(1, 2).contiguous()
                   for lin in (m.mha.linear_q, m.mha.linear_k, m.mha.linear_v))
        sc = torch.matmul(q / math.sqrt(d), k.transpose(2, 3).contiguous())
        mb = mask[i:i + rows].double()
        closed = (mb == 0).all(-1)
        sc = sc + bias + (m.inf * (mb - 1))[:, None, None, :]
        # a row with every key closed: in 32 bits the mask term swamps its scores, and its softmax is uniform
        sc[closed] = 0
        o = torch.matmul(torch.softmax(sc, -1), v).transpose(1, 2).reshape(r, n, C)
        out[i:i + rows] = _lin(o * torch.sigmoid(_lin(xn, m.mha.linear_g)), m.mha.linear_o)
    return out if starting else out.transpose(0, 1).contiguous()


def _exact_transition(m, x):
    def f(xb):
        xn = _norm(xb, m.norm)
        return _lin(F.silu(_lin(xn, m.fc1)) * _lin(xn, m.fc2), m.fc3)

    flat = x.reshape(-1, x.shape[-1])
    return _rows(flat, f, 1 << 14).view(x.shape)


def _exact_attention(m, s, k_in, bias, mask):
    """AttentionPairBias after its input norm: s [B, Q, D], k_in [B, K, D], bias [B or 1, H, Q, K], mask [B, K]."""
    b, h, d = s.shape[0], m.num_heads, m.head_dim

    def heads(x, lin):
        return _lin(x, lin).view(b, -1, h, d).transpose(1, 2).contiguous()

    q, k, v = heads(s, m.proj_q), heads(k_in, m.proj_k), heads(k_in, m.proj_v)
    sc = torch.matmul(q, k.transpose(2, 3).contiguous()) / math.sqrt(d) + bias
    sc = sc + ((1 - mask.double()) * -m.inf)[:, None, None, :]
    o = torch.matmul(torch.softmax(sc, -1), v).transpose(1, 2).reshape(s.shape)
    return _lin(torch.sigmoid(_lin(s, m.proj_g)) * o, m.proj_o)


def _exact_layer(m, t):
    mask = t["pair_mask"][0]
    z = t["z"][0].double()
    z = z + _exact_trimul(m.tri_mul_out, z, mask, True)
    z = z + _exact_trimul(m.tri_mul_in, z, mask, False)
    z = z + _exact_triattn(m.tri_att_start, z, mask, True)
    z = z + _exact_triattn(m.tri_att_end, z, mask, False)
    z = z + _exact_transition(m.transition_z, z)
    att = m.attention
    bias = _rows(z, lambda zb: _lin(_norm(zb, att.proj_z[0]), att.proj_z[1]), _block(z.shape[0], C))
    s = t["s"].double()
    sn = _norm(s, m.pre_norm_s)
    s = s + _exact_attention(att, sn, sn, bias.permute(2, 0, 1)[None], t["mask"])
    s = s + _exact_transition(m.transition_s, s)
    return {"s": s, "z": z[None]}


def _exact_adaln(m, a, s):
    sn = _norm(s, m.s_norm)
    return torch.sigmoid(_lin(sn, m.s_scale)) * _norm(a, m.a_norm) + _lin(sn, m.s_bias)


def _exact_diffusion_layer(layer, a, s, bias, mask, gather=None):
    """bias [B or 1, H, Q, K]; ``gather``: the key rows of the attention's input (None: the input itself)."""
    b = _exact_adaln(layer.adaln, a, s)
    b = _exact_attention(layer.pair_bias_attn, b, b if gather is None else gather(b), bias, mask)
    a = a + torch.sigmoid(_lin(s, layer.output_projection_linear)) * b
    tr = layer.transition
    x = _exact_adaln(tr.adaln, a, s)
    u, g = _lin(x, tr.swish_gate[0]).chunk(2, -1)
    y = _lin(F.silu(g) * u * _lin(x, tr.a_to_b), tr.b_to_a)
    return a + torch.sigmoid(_lin(s, tr.output_projection[0])) * y


def _exact_tokens(m, t):
    out = torch.empty_like(t["a"], dtype=torch.float64)
    for b in range(out.shape[0]):
        a, s, mask = t["a"][b:b + 1].double(), t["s"][b:b + 1].double(), t["mask"][b:b + 1]
        for i, layer in enumerate(m.layers):
            bias = t["bias"][..., i * HEADS_TOK:(i + 1) * HEADS_TOK].double().permute(0, 3, 1, 2)
            a = _exact_diffusion_layer(layer, a, s, bias, mask)
        out[b] = a[0]
    return out


def _exact_atoms(m, t):
    stack = m.diffusion_transformer.layers
    out = torch.empty_like(t["q"], dtype=torch.float64)
    for b in range(out.shape[0]):
        n = out.shape[1]
        nw = n // WINDOW
        a, s = t["q"][b].double().view(nw, WINDOW, -1), t["c"][b].double().view(nw, WINDOW, -1)
        mask = _key_windows(t["mask"][b].view(1, n, 1)).reshape(nw, KEYS)

        def gather(x):
            return _key_windows(x.reshape(1, n, -1)).reshape(nw, KEYS, -1).contiguous()

        for i, layer in enumerate(stack):
            bias = t["bias"][0, ..., i * HEADS_ATOM:(i + 1) * HEADS_ATOM].double().permute(0, 3, 1, 2)
            a = _exact_diffusion_layer(layer, a, s, bias, mask, gather)
        out[b] = a.reshape(n, -1)
    return out


def exact(case, seed):
    module, t = _inputs(case, seed)
    kind = case["kind"]
    with torch.no_grad():
        if kind == "layer":
            return _exact_layer(module, t)
        if kind in ("triattn", "triattn32"):
            return _exact_triattn(module, t["z"][0], t["pair_mask"][0], case["starting"])[None]
        if kind == "trimul":
            return _exact_trimul(module, t["z"][0], t["pair_mask"][0], case["outgoing"])[None]
        if kind == "transition":
            return _exact_transition(module, t["z"])
        if kind == "tokens":
            return _exact_tokens(module, t)
        return _exact_atoms(module, t)
