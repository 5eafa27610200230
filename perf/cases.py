"""The work that users of this package have it do, as measurable cases.

A case is a dict of plain values: ``kind`` (which entry point), the sizes and
the arithmetic (``mode``):

* ``amp``: float32 tensors under bf16 autocast, the trunk's inference mode
  (float32 residual stream, bf16 module arithmetic);
* ``bf16``: bf16 tensors;
* ``fp32``: float32 arithmetic, TF32 not allowed;
* ``tf32``: float32 tensors with ``torch.backends.cuda.matmul.allow_tf32``,
  the reference's inference default.

``prepare`` makes the inputs and the module, ``run`` calls the module once as
a program would, ``exact`` is the same update in float64 by plain torch.
"""

import math

import torch
import torch.nn.functional as F

from opendde_amd.layer_norm import FusedLayerNorm
from opendde_amd.outer_product_mean import OuterProductMean
from opendde_amd.pairformer import PairformerStack, Transition
from opendde_amd.triangular import (TriangleAttention, TriangleMultiplicationIncoming,
                                    TriangleMultiplicationOutgoing)

DEV = "cuda"
HEAD_DIM = 32
SINGLE_HEADS = 16
C_SINGLE = 384
C_MSA, C_OPM = 64, 32
EPS = 1e-5


def listed():
    return [
        # a short peptide through one trunk block: launches and latency
        {"name": "block_n40_amp", "kind": "stack", "n": 40, "c": 128, "c_s": 384, "blocks": 1,
         "pads": 0, "mode": "amp", "inplace": False},
        # a small protein in float32 arithmetic, one trunk block
        {"name": "block_n128_fp32", "kind": "stack", "n": 128, "c": 128, "c_s": 384, "blocks": 1,
         "pads": 0, "mode": "fp32", "inplace": False},
        # the trunk at its usual crop of large complexes, in place over a copy of the recycled z
        {"name": "stack2_n1024_amp", "kind": "stack", "n": 1024, "c": 128, "c_s": 384, "blocks": 2,
         "pads": 51, "mode": "amp", "inplace": True},
        # one attention layer of a medium complex with a tenth of its tokens padded
        {"name": "triatt_start_n384_bf16", "kind": "triatt", "n": 384, "c": 128, "starting": True,
         "pads": 38, "mode": "bf16"},
        # one multiplication layer of a larger complex
        {"name": "trimul_out_n768_bf16", "kind": "trimul", "n": 768, "c": 128, "outgoing": True,
         "pads": 0, "mode": "bf16"},
        # the default precision (float32, TF32 allowed) at an unpadded, ragged length
        {"name": "triatt_end_n509_tf32", "kind": "triatt", "n": 509, "c": 128, "starting": False,
         "pads": 0, "mode": "tf32"},
        # full float32 products at a ragged length
        {"name": "trimul_in_n300_fp32", "kind": "trimul", "n": 300, "c": 128, "outgoing": False,
         "pads": 15, "mode": "fp32"},
        # the shipped model's pair width (c_z 384, 12 heads, hidden 384), layer by layer
        {"name": "triatt_start_n640_c384_amp", "kind": "triatt", "n": 640, "c": 384,
         "starting": True, "pads": 32, "mode": "amp"},
        {"name": "trimul_in_n517_c384_amp", "kind": "trimul", "n": 517, "c": 384,
         "outgoing": False, "pads": 0, "mode": "amp"},
        {"name": "transition_n512_c384_amp", "kind": "transition", "n": 512, "c": 384,
         "mode": "amp"},
        # the standalone LayerNorm of the pair tensor, forward and backward
        {"name": "layer_norm_1048576x128_bf16", "kind": "layer_norm", "rows": 1048576, "c": 128,
         "mode": "bf16"},
        # the MSA module's outer product mean at its usual depth
        {"name": "opm_s1280_n384_amp", "kind": "opm", "seqs": 1280, "n": 384, "c": 128,
         "mode": "amp"},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["triatt", "triatt", "trimul", "trimul", "transition", "stack",
                       "layer_norm", "opm"])
    if kind == "layer_norm":
        # widths of the model's tracks and others, whole vectors and not
        c = rng.choice([64, 128, 384, rng.randint(17, 1024)])
        return {"kind": kind, "rows": _log_int(rng, 500, min(1048576, 134217728 // c)), "c": c,
                "mode": rng.choice(["bf16", "fp32"])}
    if kind == "opm":
        return {"kind": kind, "seqs": _log_int(rng, 16, 1280), "n": _log_int(rng, 24, 512),
                "c": rng.choice([128, 384]), "mode": "amp"}
    mode = rng.choice(["amp", "amp", "bf16", "tf32", "fp32"])
    c = rng.choice([64, 128, 128, 384])
    if kind == "transition":
        top = 512 if c == 384 else 1024
        if mode in ("tf32", "fp32"):
            top //= 2
        return {"kind": kind, "n": _log_int(rng, 16, top), "c": c, "mode": mode}
    top = 640 if c == 384 else 1024
    if mode in ("tf32", "fp32"):
        top = top * 5 // 8
    if kind == "stack":
        top //= 2
        n = _log_int(rng, 16, top)
        return {"kind": kind, "n": n, "c": c, "c_s": 0 if c == 64 else 384,
                "blocks": rng.choice([1, 2]), "pads": rng.choice([0, n // 20]), "mode": mode
                if mode != "bf16" else "amp", "inplace": rng.random() < 0.5}
    n = _log_int(rng, 16, top)
    side = "starting" if kind == "triatt" else "outgoing"
    return {"kind": kind, "n": n, "c": c, side: rng.random() < 0.5,
            "pads": rng.choice([0, n // 20, n // 10]), "mode": mode}


# ---------------------------------------------------------------------------
# inputs and modules
# ---------------------------------------------------------------------------


def _module(case):
    kind, c = case["kind"], case.get("c")
    if kind == "triatt":
        return TriangleAttention(c, HEAD_DIM, c // HEAD_DIM, starting=case["starting"])
    if kind == "trimul":
        cls = (TriangleMultiplicationOutgoing if case["outgoing"]
               else TriangleMultiplicationIncoming)
        return cls(c_z=c, c_hidden=c)
    if kind == "transition":
        return Transition(c_in=c, n=4)
    if kind == "layer_norm":
        return FusedLayerNorm(c)
    if kind == "opm":
        return OuterProductMean(C_MSA, c, C_OPM)
    return PairformerStack(n_blocks=case["blocks"], n_heads=SINGLE_HEADS, c_z=c,
                           c_s=case["c_s"], hidden_scale_up=True)


def _fill(module, gen):
    """Weights of the scale that training gives: unit-variance linear outputs,
    LayerNorm gains near one."""
    with torch.no_grad():
        for _, p in sorted(module.named_parameters()):
            if p.dim() == 1:
                p.copy_(torch.randn(p.shape, generator=gen, device=DEV) * 0.1
                        + (1.0 if (p == 1).all() else 0.0))
            else:
                p.copy_(torch.randn(p.shape, generator=gen, device=DEV) / math.sqrt(p.shape[1]))


def _inputs(case, gen):
    def normal(*shape):
        return torch.randn(*shape, generator=gen, device=DEV)

    kind, c = case["kind"], case["c"]
    bf = torch.bfloat16 if case["mode"] == "bf16" else torch.float32
    if kind == "layer_norm":
        return {"x": (normal(case["rows"], c) * 2 + 0.3).to(bf), "dy": normal(case["rows"], c).to(bf)}
    if kind == "opm":
        s, n = case["seqs"], case["n"]
        return {"m": normal(s, n, C_MSA),
                "mask": (torch.rand(s, n, generator=gen, device=DEV) > 0.1).float()}
    n = case["n"]
    x = {"z": normal(n, n, c).to(bf)}
    if kind == "transition":
        return x
    t = torch.ones(n, device=DEV)
    if case["pads"]:
        t[torch.randperm(n, generator=gen, device=DEV)[:case["pads"]]] = 0.0
    x["mask"] = t[:, None] * t[None, :]
    if kind == "stack" and case["c_s"]:
        x["s"] = normal(n, case["c_s"])
    return x


def prepare(case, seed):
    gen = torch.Generator(DEV).manual_seed(seed)
    module = _module(case).to(DEV).eval()
    _fill(module, gen)
    state = _inputs(case, gen)
    if case["kind"] == "layer_norm":
        state["x"].requires_grad_()
    else:
        module.requires_grad_(False)
    state["case"], state["module"] = case, module
    return state


# ---------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------


def run(state):
    case, mod = state["case"], state["module"]
    kind = case["kind"]
    if kind == "layer_norm":
        y = mod(state["x"])
        grads = torch.autograd.grad(y, (state["x"], mod.weight, mod.bias), state["dy"])
        return {"y": y, "grad_x": grads[0], "grad_w": grads[1], "grad_b": grads[2]}
    torch.backends.cuda.matmul.allow_tf32 = case["mode"] == "tf32"
    with torch.no_grad(), torch.autocast("cuda", dtype=torch.bfloat16,
                                         enabled=case["mode"] == "amp"):
        if kind == "triatt":
            return mod(state["z"], state["mask"], triangle_attention="hip")
        if kind == "trimul":
            return mod(state["z"], state["mask"], triangle_multiplicative="hip")
        if kind == "transition":
            return mod.hip_apply(state["z"])
        if kind == "opm":
            return mod(state["m"], state["mask"], kernel="hip")
        z = state["z"].clone() if case["inplace"] else state["z"]
        s, z = mod(state.get("s"), z, state["mask"], triangle_multiplicative="hip",
                   triangle_attention="hip", inplace_safe=case["inplace"])
        return {"z": z} if s is None else {"s": s, "z": z}


# ---------------------------------------------------------------------------
# bytes and operations that a pass cannot do without
# ---------------------------------------------------------------------------


def _linear_flops(kind, n, c):
    if kind == "triatt":
        return 2 * n * n * c * (5 * c + c // HEAD_DIM)
    return 2 * n * n * 6 * c * c if kind == "trimul" else 2 * n * n * 12 * c * c


def work(case):
    kind, c = case["kind"], case["c"]
    size = 2 if case["mode"] == "bf16" else 4
    if kind == "layer_norm":
        e = case["rows"] * c
        # x and dy read, y and dx written once; the statistics are the layer's own
        return {"bytes": 4 * e * size, "flops": 20 * e}
    if kind == "opm":
        s, n = case["seqs"], case["n"]
        return {"bytes": s * n * (C_MSA + 1) * 4 + n * n * c * 2,
                "flops": 2 * s * n * C_MSA * 2 * C_OPM + 2 * s * n * n * C_OPM ** 2
                + 2 * n * n * C_OPM ** 2 * c}
    n = case["n"]
    z = 2 * n * n * c * size
    if kind == "transition":
        return {"bytes": z + 12 * c * c * 4, "flops": _linear_flops(kind, n, c)}
    z += n * n * 4
    if kind == "triatt":
        return {"bytes": z, "flops": 4 * n ** 3 * c + _linear_flops(kind, n, c)}
    if kind == "trimul":
        return {"bytes": z, "flops": 2 * n ** 3 * c + _linear_flops(kind, n, c)}
    block = 12 * n ** 3 * c + sum(k * _linear_flops(m, n, c) for m, k in
                                  (("triatt", 2), ("trimul", 2), ("transition", 1)))
    if case["c_s"]:
        cs = case["c_s"]
        block += 2 * n * n * c * SINGLE_HEADS + 34 * n * cs * cs + 4 * n * n * cs
    weights = case["blocks"] * (4 * 36 * c * c + (4 * 17 * case["c_s"] ** 2))
    return {"bytes": z + weights + 2 * n * case["c_s"] * 4, "flops": case["blocks"] * block}


def tolerance(case):
    # About four times the float32 and three-part errors measured against
    # exact() (4.9e-7 and 9.2e-6 in norm; 1.7e-3 for the bf16 LayerNorm), and
    # about twice the bf16 modules' (4.0e-3 to 5.5e-3).
    mode, kind = case["mode"], case["kind"]
    if kind == "layer_norm":
        return {"rel": 7e-3, "max": 5e-2} if mode == "bf16" else {"rel": 2e-6, "max": 2e-4}
    if kind == "stack":
        # the residual stream carries the input, so rounding in the updates counts for less
        return {"amp": {"rel": 1.2e-2, "max": 0.3}, "tf32": {"rel": 5e-5, "max": 2e-3},
                "fp32": {"rel": 4e-6, "max": 2e-4}}[mode]
    return {"amp": {"rel": 1.2e-2, "max": 0.2}, "bf16": {"rel": 1.2e-2, "max": 0.2},
            "tf32": {"rel": 5e-5, "max": 2e-3}, "fp32": {"rel": 4e-6, "max": 2e-4}}[mode]


# ---------------------------------------------------------------------------
# the same in float64
# ---------------------------------------------------------------------------


def _ln(x, p, name):
    return F.layer_norm(x, (x.shape[-1],), p[name + ".weight"], p[name + ".bias"], EPS)


def _rows(n, per_row, most=1 << 28):
    step = max(1, most // max(1, per_row))
    return ((i, min(n, i + step)) for i in range(0, n, step))


def _exact_triatt(z, mask, p, starting):
    if not starting:
        return _exact_triatt(z.transpose(0, 1), mask.t(), p, True).transpose(0, 1)
    n, c = z.shape[0], z.shape[-1]
    h = p["linear.weight"].shape[0]
    bias = torch.cat([_ln(z[a:b], p, "layer_norm") @ p["linear.weight"].t()
                      for a, b in _rows(n, n * c)]).permute(2, 0, 1)
    out = torch.empty(n, n, c, dtype=z.dtype, device=z.device)
    for a, b in _rows(n, n * n * h):
        y = _ln(z[a:b], p, "layer_norm")

        def heads(name):
            t = y @ p["mha.linear_%s.weight" % name].t()
            return t.view(b - a, n, h, HEAD_DIM).permute(0, 2, 1, 3).contiguous()

        q, k, v = heads("q"), heads("k"), heads("v")
        s = q @ k.transpose(-1, -2).contiguous() / math.sqrt(HEAD_DIM) + bias
        keep = mask[a:b] != 0
        # a row without any key to keep averages over all of them
        drop = ~keep & keep.any(-1, keepdim=True)
        s.masked_fill_(drop[:, None, None, :], -math.inf)
        s.masked_fill_(~keep.any(-1)[:, None, None, None], 0.0)
        o = (torch.softmax(s, -1) @ v).permute(0, 2, 1, 3).reshape(b - a, n, c)
        o = o * torch.sigmoid(y @ p["mha.linear_g.weight"].t())
        out[a:b] = o @ p["mha.linear_o.weight"].t()
    return out


def _exact_trimul(z, mask, p, outgoing):
    n, c = z.shape[0], z.shape[-1]
    ch = p["linear_a_p.weight"].shape[0]
    ab = torch.empty(2, ch, n, n, dtype=z.dtype, device=z.device)
    for a, b in _rows(n, n * c * 2):
        y = _ln(z[a:b], p, "layer_norm_in")
        for i, side in enumerate("ab"):
            t = torch.sigmoid(y @ p["linear_%s_g.weight" % side].t())
            t = t * (y @ p["linear_%s_p.weight" % side].t()) * mask[a:b, :, None]
            ab[i, :, a:b] = t.permute(2, 0, 1)
    a_, b_ = (ab[0], ab[1].transpose(1, 2)) if outgoing else (ab[0].transpose(1, 2), ab[1])
    x = torch.bmm(a_.contiguous(), b_.contiguous())
    out = torch.empty(n, n, z.shape[-1], dtype=z.dtype, device=z.device)
    for a, b in _rows(n, n * c * 2):
        y = _ln(z[a:b], p, "layer_norm_in")
        t = _ln(x[:, a:b].permute(1, 2, 0), p, "layer_norm_out") @ p["linear_z.weight"].t()
        out[a:b] = t * torch.sigmoid(y @ p["linear_g.weight"].t())
    return out


def _exact_transition(x, p):
    rows = x.reshape(-1, x.shape[-1])
    out = torch.empty_like(rows)
    for a, b in _rows(rows.shape[0], rows.shape[1] * 8):
        y = _ln(rows[a:b], p, "layernorm1")
        h = F.silu(y @ p["linear_no_bias_a.weight"].t()) * (y @ p["linear_no_bias_b.weight"].t())
        out[a:b] = h @ p["linear_no_bias.weight"].t()
    return out.view(x.shape)


def _exact_single(s, z, p):
    a = _ln(s, p, "layernorm_a")
    n, c = a.shape
    bias = torch.cat([_ln(z[i:j], p, "layernorm_z") @ p["linear_nobias_z.weight"].t()
                      for i, j in _rows(n, n * z.shape[-1])]).permute(2, 0, 1)

    def heads(name, b=None):
        t = F.linear(a, p["attention.linear_%s.weight" % name], b)
        return t.view(n, SINGLE_HEADS, -1).transpose(0, 1).contiguous()

    q, k, v = heads("q", p["attention.linear_q.bias"]), heads("k"), heads("v")
    w = torch.softmax(q @ k.transpose(1, 2).contiguous() / math.sqrt(c // SINGLE_HEADS) + bias, -1)
    o = (w @ v).transpose(0, 1).reshape(n, c)
    o = o * torch.sigmoid(a @ p["attention.linear_g.weight"].t())
    return o @ p["attention.linear_o.weight"].t()


def _part(p, prefix):
    return {k[len(prefix):]: v for k, v in p.items() if k.startswith(prefix)}


def exact(case, seed):
    state = prepare(case, seed)
    p = {k: v.detach().double() for k, v in state["module"].named_parameters()}
    x = {k: v.detach().double() for k, v in state.items() if torch.is_tensor(v)}
    kind = case["kind"]
    torch.backends.cuda.matmul.allow_tf32 = False
    if kind == "layer_norm":
        if case["mode"] == "bf16":  # the layer hands its kernels the parameters in x's type
            p = {k: v.to(torch.bfloat16).double() for k, v in p.items()}
        leaves = [t.requires_grad_() for t in (x["x"], p["weight"], p["bias"])]
        y = F.layer_norm(leaves[0], (case["c"],), leaves[1], leaves[2], EPS)
        g = torch.autograd.grad(y, leaves, x["dy"])
        return {"y": y.detach(), "grad_x": g[0], "grad_w": g[1], "grad_b": g[2]}
    with torch.no_grad():
        if kind == "triatt":
            return _exact_triatt(x["z"], x["mask"], p, case["starting"])
        if kind == "trimul":
            return _exact_trimul(x["z"], x["mask"], p, case["outgoing"])
        if kind == "transition":
            return _exact_transition(x["z"], p)
        if kind == "opm":
            y = _ln(x["m"], p, "layer_norm")
            a, b = (F.linear(y, p["linear_%d.weight" % i]) * x["mask"][..., None] for i in (1, 2))
            n, c = case["n"], case["c"]
            a = a.permute(1, 2, 0).reshape(n * C_OPM, -1).contiguous()
            b = b.permute(0, 1, 2).reshape(-1, n * C_OPM).contiguous()
            norm = x["mask"].t().contiguous() @ x["mask"] + 1e-3
            out = torch.empty(n, n, c, dtype=a.dtype, device=DEV)
            for i, j in _rows(n, n * C_OPM ** 2):
                o = (a[i * C_OPM:j * C_OPM] @ b).view(j - i, C_OPM, n, C_OPM).transpose(1, 2)
                o = o.reshape(j - i, n, -1) @ p["linear_out.weight"].t() + p["linear_out.bias"]
                out[i:j] = o / norm[i:j, :, None]
            return out
        s, z, mask = x.get("s"), x["z"], x["mask"]
        for i in range(case["blocks"]):
            q = _part(p, "blocks.%d." % i)
            z = z + _exact_trimul(z, mask, _part(q, "tri_mul_out."), True)
            z = z + _exact_trimul(z, mask, _part(q, "tri_mul_in."), False)
            z = z + _exact_triatt(z, mask, _part(q, "tri_att_start."), True)
            z = z + _exact_triatt(z, mask, _part(q, "tri_att_end."), False)
            z = z + _exact_transition(z, _part(q, "pair_transition."))
            if s is not None:
                s = s + _exact_single(s, z, _part(q, "attention_pair_bias."))
                s = s + _exact_transition(s, _part(q, "single_transition."))
        return {"z": z} if s is None else {"s": s, "z": z}
