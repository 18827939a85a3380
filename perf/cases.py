"""The Pairformer path's work as a caller runs it: the sublayers one at a time,
whole blocks of the three ports and a short trunk, from peptide-sized inputs
to 2048 tokens.

Token counts are those of real complexes, so most are no multiple of anything
(245, 499, 952 and 1003 tokens are complexes the reference reports on); a
caller who pads buckets to 256 or 1024 leaves a masked tail. The pair track
runs in bfloat16 with float32 where a port asks for it (Protenix's "highest"
precision, Boltz-2's single track). Every call is forward only: the framework
has no backward.

``exact`` restates each call in float64 with plain torch.
"""

from __future__ import annotations

import math

import torch

from foldjax_amd import boltz2, openfold3, protenix
from foldjax_amd import params as P
from foldjax_amd.pairformer import PairformerLayerWeights

DEVICE = "cuda"
DTYPES = {"bf16": torch.bfloat16, "fp32": torch.float32}
HEADS_S = 16  # heads of the single track
C_S = 384  # its width


def listed():
    return [
        # a call at a time on a peptide: launches and host time are all there is
        {"name": "triattn_start_n37_bf16", "op": "triattn", "n": 37, "real": 37, "dtype": "bf16", "first": True,
         "c_z": 128, "heads": 4},
        # the reference's float32 check of tri-mul, at its size
        {"name": "trimul_out_n256_fp32", "op": "trimul", "n": 256, "real": 256, "dtype": "fp32", "first": True,
         "c_z": 128, "c_h": 128},
        # tri-mul of a complex run at its own length
        {"name": "trimul_in_n1003_bf16", "op": "trimul", "n": 1003, "real": 1003, "dtype": "bf16", "first": False,
         "c_z": 128, "c_h": 128},
        # tri-attn of a complex run at its own length
        {"name": "triattn_end_n952_bf16", "op": "triattn", "n": 952, "real": 952, "dtype": "bf16", "first": False,
         "c_z": 128, "heads": 4},
        # the attention core alone: the call that replaces the fused-kernel backend inside a caller's own module
        {"name": "core_n499_bf16", "op": "core", "n": 499, "real": 450, "dtype": "bf16", "heads": 4},
        # the single track's attention, float32 over a bfloat16 pair tensor
        {"name": "single_n1003_fp32", "op": "single", "n": 1003, "real": 1003, "dtype": "fp32"},
        # the 384-wide pair track (OpenDDE)
        {"name": "trimul_out_n245_c384_bf16", "op": "trimul", "n": 245, "real": 245, "dtype": "bf16", "first": True,
         "c_z": 384, "c_h": 384},
        # the template stack's pair block: 64 channels, no single track
        {"name": "template_n499_bf16", "op": "template", "n": 499, "real": 499, "dtype": "bf16"},
        # a Protenix block in float32, token count unpadded
        {"name": "protenix_n245_fp32", "op": "block", "port": "protenix", "n": 245, "real": 245, "dtype": "fp32",
         "single": "fp32"},
        # a short trunk on a small input: many launches, little work in each
        {"name": "trunk4_n77_bf16", "op": "trunk", "n": 77, "real": 77, "layers": 4},
        # the usual bucket with a masked tail
        {"name": "boltz2_n1024_bf16", "op": "block", "port": "boltz2", "n": 1024, "real": 973, "dtype": "bf16",
         "single": "fp32"},
        # one layer of a long-context trunk
        {"name": "boltz2_n2048_bf16", "op": "block", "port": "boltz2", "n": 2048, "real": 2048, "dtype": "bf16",
         "single": "fp32"},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    op = rng.choice(["trimul", "triattn", "transition", "single", "core", "wide", "template", "trunk", "boltz2",
                     "protenix", "openfold3"])
    hi = {"trimul": 2048, "triattn": 2048, "transition": 1536, "single": 1536, "core": 1024, "wide": 512,
          "template": 1024, "trunk": 320, "boltz2": 1536, "protenix": 1024, "openfold3": 1536}[op]
    n = _log_int(rng, 16, hi)
    if rng.random() < 0.25:  # a caller that pads to buckets
        n = min(hi, (n + 63) // 64 * 64)
    # half of the calls carry a masked tail of up to a tenth
    real = n if rng.random() < 0.5 else max(1, n - rng.randint(1, max(1, n // 10)))
    first = rng.random() < 0.5
    fp32 = rng.random() < 0.25 and n <= 640
    dt = "fp32" if fp32 else "bf16"
    if op == "trimul":
        return {"op": op, "n": n, "real": real, "dtype": dt, "first": first, "c_z": 128, "c_h": 128}
    if op == "triattn":
        # float32 rows whose every key is masked have no defined softmax: no tail
        return {"op": op, "n": n, "real": n if fp32 else real, "dtype": dt, "first": first, "c_z": 128, "heads": 4}
    if op == "transition":
        return {"op": op, "n": n, "real": real, "dtype": dt, "c_z": rng.choice([128, 128, 64])}
    if op == "single":
        return {"op": op, "n": n, "real": real, "dtype": rng.choice(["fp32", "bf16"])}
    if op == "core":
        return {"op": op, "n": n, "real": real, "dtype": "bf16", "heads": 4}
    if op == "wide":
        if rng.random() < 0.5:
            return {"op": "trimul", "n": n, "real": real, "dtype": "bf16", "first": first, "c_z": 384, "c_h": 384}
        return {"op": "triattn", "n": n, "real": real, "dtype": "bf16", "first": first, "c_z": 384, "heads": 12}
    if op == "template":
        return {"op": op, "n": n, "real": real, "dtype": "bf16"}
    if op == "trunk":
        return {"op": op, "n": n, "real": real, "layers": rng.randint(2, 4)}
    if op == "boltz2":
        return {"op": "block", "port": op, "n": n, "real": real, "dtype": "bf16", "single": "fp32"}
    if op == "protenix":
        return {"op": "block", "port": op, "n": n, "real": real, "dtype": dt, "single": dt}
    return {"op": "block", "port": op, "n": n, "real": real, "dtype": "bf16", "single": "bf16"}


# ------------------------------------------------------------------ inputs


class _Draw:
    """Seeded values on the GPU: activations N(0,1), Glorot-uniform linears,
    LayerNorm affines near (1, 0)."""

    def __init__(self, seed):
        self.g = torch.Generator(device=DEVICE)
        self.g.manual_seed(seed)

    def normal(self, *shape):
        return torch.randn(*shape, generator=self.g, device=DEVICE)

    def linear(self, out_f, in_f, bias=False):
        lim = math.sqrt(6.0 / (in_f + out_f))
        w = (2.0 * torch.rand(out_f, in_f, generator=self.g, device=DEVICE) - 1.0) * lim
        return P.LinearParams(w, 0.1 * self.normal(out_f) if bias else None)

    def ln(self, c):
        return P.LayerNormParams(1.0 + 0.1 * self.normal(c), 0.1 * self.normal(c))

    def trimul(self, c_z, c_h):
        return P.ProtenixTriangleMultiplicationParams(
            layer_norm_in=self.ln(c_z), layer_norm_out=self.ln(c_h),
            linear_a_p=self.linear(c_h, c_z), linear_a_g=self.linear(c_h, c_z),
            linear_b_p=self.linear(c_h, c_z), linear_b_g=self.linear(c_h, c_z),
            linear_z=self.linear(c_z, c_h), linear_g=self.linear(c_z, c_z))

    def triattn(self, c_z, heads):
        hd = 32 * heads
        att = P.AttentionParams(self.linear(hd, c_z), self.linear(hd, c_z), self.linear(hd, c_z),
                                self.linear(c_z, hd), self.linear(hd, c_z))
        return P.ProtenixTriangleAttentionParams(self.ln(c_z), self.linear(heads, c_z), att)

    def transition(self, c):
        return P.ProtenixTransitionParams(self.ln(c), self.linear(4 * c, c), self.linear(4 * c, c),
                                          self.linear(c, 4 * c))

    def single(self):
        att = P.AttentionParams(self.linear(C_S, C_S, bias=True), self.linear(C_S, C_S), self.linear(C_S, C_S),
                                self.linear(C_S, C_S), self.linear(C_S, C_S))
        return P.ProtenixAttentionPairBiasParams(layernorm_a=self.ln(C_S), layernorm_kv=None, attention=att,
                                                 layernorm_z=self.ln(128), linear_z=self.linear(HEADS_S, 128))

    def block(self, c_z=128, c_h=128, with_single=True):
        return P.ProtenixPairformerBlockParams(
            tri_mul_out=self.trimul(c_z, c_h), tri_mul_in=self.trimul(c_z, c_h),
            tri_att_start=self.triattn(c_z, 4), tri_att_end=self.triattn(c_z, 4),
            pair_transition=self.transition(c_z),
            attention_pair_bias=self.single() if with_single else None,
            single_transition=self.transition(C_S) if with_single else None)


def _round(tree, dtype):
    """The tree's tensors rounded through ``dtype`` (the values a packed weight
    holds), as float64."""
    if isinstance(tree, torch.Tensor):
        return tree.to(dtype).double()
    if isinstance(tree, tuple):
        vals = [_round(v, dtype) for v in tree]
        return type(tree)(*vals) if hasattr(tree, "_fields") else tuple(vals)
    return tree


def _inputs(case, seed):
    """(activations and masks in the case's dtypes, weight containers in float32)."""
    d, n, op = _Draw(seed), case["n"], case["op"]
    dt = DTYPES[case.get("dtype", "bf16")]
    sdt = DTYPES[case.get("single", case.get("dtype", "fp32"))] if op != "trunk" else torch.float32
    tok = (torch.arange(n, device=DEVICE) < case["real"]).float()
    x = {"tok": tok, "pair": torch.outer(tok, tok)[None]}
    if op == "trimul":
        x["z"] = d.normal(1, n, n, case["c_z"]).to(dt)
        w = d.trimul(case["c_z"], case["c_h"])
    elif op == "triattn":
        x["z"] = d.normal(1, n, n, case["c_z"]).to(dt)
        w = d.triattn(case["c_z"], case["heads"])
    elif op == "transition":
        x["z"] = d.normal(1, n, n, case["c_z"]).to(dt)
        w = d.transition(case["c_z"])
    elif op == "single":
        x["z"] = d.normal(1, n, n, 128).to(torch.bfloat16)
        x["s"] = d.normal(1, n, C_S).to(dt)
        w = d.single()
    elif op == "core":
        h = case["heads"]
        for k in ("q", "k", "v"):
            x[k] = d.normal(1, n, h, n, 32).to(dt)
        x["bias"] = d.normal(1, 1, h, n, n).to(dt)
        x["mask_bias"] = (1e9 * (tok - 1.0)).expand(1, n, n).reshape(1, n, 1, 1, n).contiguous()
        w = None
    elif op == "template":
        x["z"] = d.normal(1, n, n, 64).to(dt)
        w = d.block(64, 128, with_single=False)
    else:
        x["z"] = d.normal(1, n, n, 128).to(dt)
        x["s"] = d.normal(1, n, C_S).to(sdt)
        w = [d.block() for _ in range(case.get("layers", 1))]
    x["pair"] = x["pair"].to(dt)
    return x, w, dt, sdt


def prepare(case, seed):
    x, w, dt, sdt = _inputs(case, seed)
    op = case["op"]
    if op == "trimul":
        w = P.pack_trimul_torch(w, dt, DEVICE)
    elif op == "triattn":
        w = P.pack_triattn_protenix(w, dt, DEVICE)
    elif op == "transition":
        w = P.pack_transition_torch(w, dt, DEVICE)
    elif op == "single":
        w = P.pack_single_attention_protenix(w, dt, DEVICE)
    elif op == "template":
        w = PairformerLayerWeights.from_protenix(w, dt, DEVICE)
    elif op == "block":
        w = PairformerLayerWeights.from_protenix(w[0], dt, DEVICE, single_dtype=sdt)
    elif op == "trunk":
        w = boltz2.stack_layer_params([PairformerLayerWeights.from_protenix(b, dt, DEVICE, single_dtype=sdt)
                                       for b in w])
    x["tok"] = x["tok"][None].to(sdt)
    return dict(x, case=case, w=w)


def run(state):
    c, w = state["case"], state["w"]
    op = c["op"]
    if op == "trimul":
        return boltz2.triangle_multiplication_forward(w, state["z"], state["pair"],
                                                      "outgoing" if c["first"] else "incoming")
    if op == "triattn":
        return boltz2.triangle_attention_forward(w, state["z"], state["pair"], starting=c["first"])
    if op == "transition":
        return openfold3.swiglu_transition(state["z"], w, mask=state["pair"])
    if op == "single":
        return openfold3.attention_pair_bias(state["s"], state["z"], w, no_heads=HEADS_S, mask=state["tok"],
                                             residual=state["s"])
    if op == "core":
        return boltz2.hip_attention_core(state["q"], state["k"], state["v"], state["bias"], state["mask_bias"],
                                         scale=32 ** -0.5)
    if op == "template":
        return protenix.pairformer_block(None, state["z"], state["pair"], w)[1]
    if op == "trunk":
        return boltz2.pairformer_module_forward({"layers": w}, state["s"], state["z"], state["tok"], state["pair"])
    if c["port"] == "protenix":
        return protenix.pairformer_block(state["s"], state["z"], state["pair"], w)
    if c["port"] == "openfold3":
        return openfold3.pairformer_block(state["s"], state["z"], w, single_mask=state["tok"],
                                          pair_mask=state["pair"], no_heads_pair=4, no_heads_pair_bias=HEADS_S)
    return boltz2.pairformer_layer_forward(w, state["s"], state["z"], state["tok"], state["pair"])


# -------------------------------------------------------------------- work


def _trimul_flops(n, c_z, c_h):
    return 2.0 * n**3 * c_h + 2.0 * n * n * (4 * c_z * c_h + c_h * c_z + c_z * c_z)


def _triattn_flops(n, c_z, heads):
    return 4.0 * n**3 * 32 * heads + 2.0 * n * n * c_z * (5 * 32 * heads + heads)


def _single_flops(n):
    return 2.0 * n * C_S * C_S * 5 + 4.0 * n * n * C_S + 2.0 * n * n * 128 * HEADS_S


def _block_flops(n, c_z=128, with_single=True):
    f = 2 * _trimul_flops(n, c_z, 128) + 2 * _triattn_flops(n, c_z, 4) + 24.0 * n * n * c_z * c_z
    return f + (_single_flops(n) + 24.0 * n * C_S * C_S if with_single else 0.0)


def work(case):
    """One pass's flops, and its inputs read once plus its outputs written once."""
    n, op = case["n"], case["op"]
    es = 4 if case.get("dtype") == "fp32" else 2
    if op == "trimul":
        cz, ch = case["c_z"], case["c_h"]
        return {"flops": _trimul_flops(n, cz, ch), "bytes": es * (n * n * (2 * cz + 1) + 5 * cz * ch + cz * cz)}
    if op == "triattn":
        cz, hd = case["c_z"], 32 * case["heads"]
        return {"flops": _triattn_flops(n, cz, case["heads"]), "bytes": es * (n * n * (2 * cz + 1) + 5 * cz * hd)}
    if op == "transition":
        cz = case["c_z"]
        return {"flops": 24.0 * n * n * cz * cz, "bytes": es * (n * n * (2 * cz + 1) + 12 * cz * cz)}
    if op == "single":
        return {"flops": _single_flops(n), "bytes": 2 * n * n * 128 + es * (2 * n * C_S + 5 * C_S * C_S)}
    if op == "core":
        h = case["heads"]
        return {"flops": 4.0 * n**3 * 32 * h, "bytes": 2 * (4 * n * n * 32 * h + h * n * n) + 4 * n * n}
    if op == "template":
        return {"flops": _block_flops(n, 64, False), "bytes": 2 * n * n * (2 * 64 + 1)}
    layers = case.get("layers", 1)
    ss = 2 if case.get("single") == "bf16" else 4
    weights = 22 * 128 * 128 * es + 17 * C_S * C_S * ss
    return {"flops": layers * _block_flops(n), "bytes": es * n * n * 257 + ss * 2 * n * C_S + layers * weights}


def tolerance(case):
    """About four times the relative error of one call against ``exact``: 16-bit
    activations leave 4 to 8e-3 in a sublayer or a block and 1.2e-2 after four
    layers, float32 1 to 8e-7 (the hardware's exp2 and reciprocal included)."""
    if case.get("dtype", "bf16") == "fp32":
        return {"rel": 3e-6}
    return {"rel": 4e-2 if case["op"] == "trunk" else 2.5e-2}


# ------------------------------------------------------------------- exact


def _ln(x, p, eps=1e-5):
    m = x.mean(-1, keepdim=True)
    d = x - m
    return d / torch.sqrt((d * d).mean(-1, keepdim=True) + eps) * p.weight + p.bias


def _lin(x, p):
    y = x @ p.weight.t().contiguous()
    return y if p.bias is None else y + p.bias


def _rows(n, bytes_per_row, budget=4e9):
    return max(1, min(n, int(budget / bytes_per_row)))


def _x_trimul(z, pair, w, outgoing):
    """z [N, N, c], pair [N, N]; 32 channels of the contraction at a time."""
    n, ch = z.shape[0], w.linear_a_p.weight.shape[0]
    x = _ln(z, w.layer_norm_in)
    o = torch.empty(n, n, ch, dtype=torch.float64, device=z.device)
    for c0 in range(0, ch, 32):
        part = lambda p: P.LinearParams(p.weight[c0:c0 + 32], None)  # noqa: E731
        a = _lin(x, part(w.linear_a_p)) * torch.sigmoid(_lin(x, part(w.linear_a_g))) * pair[..., None]
        b = _lin(x, part(w.linear_b_p)) * torch.sigmoid(_lin(x, part(w.linear_b_g))) * pair[..., None]
        if outgoing:  # sum_k a[i, k] b[j, k]
            a, b = a.permute(2, 0, 1).contiguous(), b.permute(2, 1, 0).contiguous()
        else:  # sum_k a[k, i] b[k, j]
            a, b = a.permute(2, 1, 0).contiguous(), b.permute(2, 0, 1).contiguous()
        o[..., c0:c0 + 32] = torch.bmm(a, b).permute(1, 2, 0)
    return _lin(_ln(o, w.layer_norm_out), w.linear_z) * torch.sigmoid(_lin(x, w.linear_g))


def _x_core(q, k, v, bias, mask_bias, scale):
    """q, k, v [R, H, N, 32]; bias [H, N, N]; mask_bias [R, N]."""
    out = torch.empty_like(q)
    step = _rows(q.shape[0], q.shape[1] * q.shape[2] ** 2 * 24)
    for r in range(0, q.shape[0], step):
        s = torch.matmul(q[r:r + step] * scale, k[r:r + step].transpose(-1, -2).contiguous())
        s += bias
        s += mask_bias[r:r + step, None, None, :]
        out[r:r + step] = torch.matmul(torch.softmax(s, -1), v[r:r + step])
    return out


def _x_triattn(z, pair, w, starting, inf=1e9):
    if not starting:
        z, pair = z.transpose(0, 1).contiguous(), pair.t().contiguous()
    n, heads = z.shape[0], w.linear.weight.shape[0]
    x = _ln(z, w.layer_norm)
    split = lambda t: t.reshape(n, n, heads, 32).permute(0, 2, 1, 3).contiguous()  # noqa: E731
    a = w.attention
    o = _x_core(split(_lin(x, a.linear_q)), split(_lin(x, a.linear_k)), split(_lin(x, a.linear_v)),
                _lin(x, w.linear).permute(2, 0, 1).contiguous(), inf * (pair - 1.0), 32 ** -0.5)
    o = o.permute(0, 2, 1, 3).reshape(n, n, 32 * heads) * torch.sigmoid(_lin(x, a.linear_g))
    y = _lin(o, a.linear_o)
    return y if starting else y.transpose(0, 1)


def _x_transition(z, w):
    flat = z.reshape(-1, z.shape[-1])
    out = torch.empty_like(flat)
    step = _rows(flat.shape[0], flat.shape[1] * 4 * 8 * 4)
    for r in range(0, flat.shape[0], step):
        x = _ln(flat[r:r + step], w.layer_norm)
        a = _lin(x, w.linear_a)
        out[r:r + step] = _lin(a * torch.sigmoid(a) * _lin(x, w.linear_b), w.linear_out)
    return out.reshape(z.shape)


def _x_single(s, z, tok, w, inf):
    """s [N, c_s], z [N, N, 128], tok [N]: the update."""
    n, dh = s.shape[0], C_S // HEADS_S
    x = _ln(s, w.layernorm_a)
    a = w.attention
    split = lambda t: t.reshape(n, HEADS_S, dh).permute(1, 0, 2).contiguous()  # noqa: E731
    q, k, v = split(_lin(x, a.linear_q)), split(_lin(x, a.linear_k)), split(_lin(x, a.linear_v))
    sc = torch.bmm(q * dh ** -0.5, k.transpose(-1, -2).contiguous())
    sc += _lin(_ln(z, w.layernorm_z), w.linear_z).permute(2, 0, 1)
    sc += inf * (tok - 1.0)
    o = torch.bmm(torch.softmax(sc, -1), v).permute(1, 0, 2).reshape(n, C_S)
    return _lin(o * torch.sigmoid(_lin(x, a.linear_g)), a.linear_o)


def _x_block(s, z, tok, pair, wz, ws, port):
    """One block; wz and ws hold the pair track's and the single track's weights."""
    gate = pair if port == "protenix" else None

    def add(z, u):
        z = z + u
        return z if gate is None else z * gate[..., None]

    z = add(z, _x_trimul(z, pair, wz.tri_mul_out, True))
    z = add(z, _x_trimul(z, pair, wz.tri_mul_in, False))
    z = add(z, _x_triattn(z, pair, wz.tri_att_start, True))
    z = add(z, _x_triattn(z, pair, wz.tri_att_end, False))
    u = _x_transition(z, wz.pair_transition)
    z = add(z, u * pair[..., None] if port == "openfold3" else u)
    if s is None:
        return None, z
    valid = tok[:, None] if port == "protenix" else torch.ones_like(tok)[:, None]
    s = (s + _x_single(s, z, tok, ws.attention_pair_bias, {"boltz2": 1e6, "protenix": 1e10, "openfold3": 1e9}[port])
         ) * valid
    u = _x_transition(s, ws.single_transition)
    s = (s + (u * tok[:, None] if port == "openfold3" else u)) * valid
    return s, z


def exact(case, seed):
    x, w, dt, sdt = _inputs(case, seed)
    op = case["op"]
    z = x["z"][0].double() if "z" in x else None
    s = x["s"][0].double() if "s" in x else None
    tok, pair = x["tok"].double(), x["pair"][0].double()
    if op == "trimul":
        return _x_trimul(z, pair, _round(w, dt), case["first"])[None]
    if op == "triattn":
        return _x_triattn(z, pair, _round(w, dt), case["first"])[None]
    if op == "transition":
        return (_x_transition(z, _round(w, dt)) * pair[..., None])[None]
    if op == "single":
        return (s + _x_single(s, z, tok, _round(w, dt), 1e9))[None]
    if op == "core":
        return _x_core(x["q"][0].double(), x["k"][0].double(), x["v"][0].double(), x["bias"][0, 0].double(),
                       x["mask_bias"].reshape(case["n"], case["n"]).double(), 32 ** -0.5)[None]
    if op == "template":
        return _x_block(None, z, tok, pair, _round(w, dt), None, "protenix")[1][None]
    for b in w:
        s, z = _x_block(s, z, tok, pair, _round(b, dt), _round(b, sdt), case.get("port", "boltz2"))
    return s[None], z[None]
