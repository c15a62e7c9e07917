"""The work this framework does for its users, as cases that can be prepared, run and checked.

A case is a dict of plain values.  Its ``op`` names the entry point a program calls:

* ``trimul_fn``   ``ops.triangle_multiplicative_update``: one operator, weights as tensors
* ``attn_fn``     ``ops.triangle_attention``: the attention core on a caller's own q, k, v
* ``single_fn``   ``ops.attention_pair_bias``: the single track's attention
* ``trimul``      ``TriangleMultiplication`` on padded device tensors (the module classes)
* ``triatt``      ``TriangleAttention`` on padded device tensors with ``n_valid``
* ``layers``      ``PairformerModule``: whole Pairformer blocks on unpadded device tensors
* ``template``    ``PairformerModule`` without the single track at c_z = 64, a batch of templates
* ``msa``         ``MSAModule``: one block of the MSA stack
* ``diffusion``   ``DiffusionPairConditioning``: the pair side of the diffusion conditioning

Inference only: the framework has no backward pass.  Sizes are token counts ``n`` (and MSA
depths); ``tail`` tokens at the end are masked.  ``operand`` is the 16-bit matrix operand type
and ``fast`` the block-fp8 mode.
"""
from __future__ import annotations

import math
import random
from typing import Dict, List, Optional

import torch
import torch.nn.functional as F

import tt_boltz_amd as pf
from tt_boltz_amd import ops, synthetic

HEADS, HEAD_DIM = 4, 32          # triangle attention
S_HEADS, S_DIM, C_S = 16, 24, 384   # single track
MSA_HEADS, C_M, OPM_HIDDEN = 8, 64, 32
DIFF_LAYERS = 24                 # token-transformer layers whose biases are computed at once


def listed() -> List[dict]:
    return [
        # a peptide through one operator: launches and latency count, nothing else
        {"name": "trimul_fn_45", "op": "trimul_fn", "n": 45, "tail": 4, "direction": "outgoing", "operand": "fp16"},
        # a small protein through two whole blocks
        {"name": "layers_118", "op": "layers", "n": 118, "tail": 0, "blocks": 2, "operand": "fp16", "fast": False},
        # an ordinary protein padded by its caller to a bucket, odd length
        {"name": "layers_301", "op": "layers", "n": 301, "tail": 22, "blocks": 2, "operand": "fp16", "fast": False},
        # the largest complexes of the ordinary mode
        {"name": "layers_1024", "op": "layers", "n": 1024, "tail": 0, "blocks": 1, "operand": "fp16", "fast": False},
        # the block-fp8 mode (its sizes are padded to 128)
        {"name": "layers_fast_620", "op": "layers", "n": 620, "tail": 0, "blocks": 1, "operand": "fp16", "fast": True},
        # one operator of the module classes, in the benchmark's size and with its masked tail
        {"name": "trimul_512", "op": "trimul", "n": 512, "tail": 51, "direction": "incoming", "operand": "fp16"},
        # the ending-node attention on a padded size, bf16 operands
        {"name": "triatt_768", "op": "triatt", "n": 725, "tail": 0, "ending": True, "operand": "bf16"},
        # the attention core called with the caller's own fp32 q, k, v
        {"name": "attn_fn_384", "op": "attn_fn", "n": 384, "tail": 17, "operand": "fp16"},
        # the single track's attention called alone, odd length
        {"name": "single_fn_413", "op": "single_fn", "n": 413, "tail": 13, "operand": "fp16"},
        # an MSA block: ordinary depth and length
        {"name": "msa_350x777", "op": "msa", "n": 350, "tail": 0, "depth": 777, "operand": "fp16"},
        # the template stack: four templates, two blocks
        {"name": "template_4x250", "op": "template", "n": 250, "tail": 0, "batch": 4, "operand": "fp16"},
        # the pair side of the diffusion conditioning, once per sampled structure
        {"name": "diffusion_450", "op": "diffusion", "n": 450, "tail": 0, "operand": "fp16"},
    ]


def _log_int(rng: random.Random, lo: int, hi: int) -> int:
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng: random.Random) -> dict:
    op = rng.choice(["trimul_fn", "attn_fn", "single_fn", "trimul", "triatt", "layers", "layers", "template", "msa",
                     "diffusion"])
    hi = {"trimul_fn": 900, "attn_fn": 700, "single_fn": 900, "trimul": 900, "triatt": 800, "layers": 640,
          "template": 300, "msa": 450, "diffusion": 640}[op]
    n = _log_int(rng, 34, hi)
    case = {"op": op, "n": n, "tail": rng.choice([0, 0, n // 10]), "operand": rng.choice(["fp16", "fp16", "bf16"])}
    if op in ("trimul_fn", "trimul"):
        case["direction"] = rng.choice(["outgoing", "incoming"])
    elif op == "triatt":
        case["ending"] = rng.random() < 0.5
    elif op == "layers":
        case["blocks"], case["fast"] = rng.choice([1, 2]), rng.random() < 0.25
    elif op == "template":
        case["batch"] = rng.choice([1, 2, 4])
    elif op == "msa":
        case["depth"] = _log_int(rng, 8, 1024)
    return case


# --------------------------------------------------------------------------------------
# inputs and weights, from the seed alone
# --------------------------------------------------------------------------------------
class _Source:
    def __init__(self, seed: int):
        self.g = torch.Generator(device="cuda").manual_seed(1000003 * seed + 17)

    def normal(self, *shape: int) -> torch.Tensor:
        return torch.randn(shape, generator=self.g, device="cuda")

    def uniform(self, *shape: int) -> torch.Tensor:
        return torch.rand(shape, generator=self.g, device="cuda")

    def weights(self, shapes: Dict[str, tuple]) -> Dict[str, torch.Tensor]:
        """Xavier-uniform matrices, LayerNorm weights about 1, small biases."""
        out = {}
        for key in sorted(shapes):
            shape = shapes[key]
            u = self.uniform(*shape) * 2 - 1
            if len(shape) == 2:
                out[key] = u * (6.0 / (shape[0] + shape[1])) ** 0.5
            else:
                out[key] = 0.1 * u + (1.0 if key.endswith(".weight") else 0.0)
        return out

    def pair(self, batch: int, n: int, c: int) -> torch.Tensor:
        """A pair representation: its channels have means of their own."""
        return self.normal(batch, n, n, c) + 0.5 * self.normal(c)


def _sub(w: Dict[str, torch.Tensor], prefix: str) -> Dict[str, torch.Tensor]:
    return {k[len(prefix):]: v for k, v in w.items() if k.startswith(prefix)}


def _one(prefix: str, c_z: int = 128) -> Dict[str, tuple]:
    """The shapes of one operator of a Pairformer block, without its prefix."""
    return {k[len(prefix):]: v for k, v in synthetic.layer_shapes(c_z).items() if k.startswith(prefix)}


def _blocks(n: int, **kw) -> Dict[str, tuple]:
    return {f"layers.{i}.{k}": v for i in range(n) for k, v in synthetic.layer_shapes(**kw).items()}


def _token_mask(case: dict, batch: int = 1) -> torch.Tensor:
    m = torch.ones((batch, case["n"]), device="cuda")
    if case["tail"]:
        m[:, case["n"] - case["tail"]:] = 0.0
    return m


def _inputs(case: dict, seed: int) -> dict:
    src, op, n = _Source(seed), case["op"], case["n"]
    m = _token_mask(case, case.get("batch", 1))
    d = {"mask": m, "pair_mask": m[:, :, None] * m[:, None, :]}
    if op in ("trimul_fn", "trimul"):
        d["w"] = src.weights(_one("tri_mul_out."))
        d["z"] = src.pair(1, n, 128)
    elif op == "triatt":
        d["w"] = src.weights(_one("tri_att_start."))
        d["z"] = src.pair(1, n, 128)
    elif op == "attn_fn":
        for k in ("q", "k", "v"):
            d[k] = src.normal(1, n, HEADS, n, HEAD_DIM)
        d["bias"] = src.normal(1, 1, HEADS, n, n)
        d["key_mask"] = (m[:, None, :] * torch.ones((1, n, 1), device="cuda")).view(1, n, 1, 1, n) > 0
    elif op == "single_fn":
        d["w"] = src.weights(_one("attention."))
        d["s"], d["z"] = src.normal(1, n, C_S), src.pair(1, n, 128)
    elif op == "layers":
        d["w"] = src.weights(_blocks(case["blocks"]))
        d["s"], d["z"] = src.normal(1, n, C_S), src.pair(1, n, 128)
    elif op == "template":
        d["w"] = src.weights(_blocks(2, c_z=64, transform_s=False))
        d["z"] = src.pair(case["batch"], n, 64)
    elif op == "msa":
        depth = case["depth"]
        d["w"] = src.weights(synthetic.msa_module_shapes(1))
        d["z"], d["emb"] = src.pair(1, n, 128), src.normal(1, n, C_S)
        rows = torch.ones((1, depth, 1), device="cuda")
        rows[:, depth - depth // 16:] = 0.0   # the alignment's own padding rows
        d["feats"] = {"msa": (src.uniform(1, depth, n) * 33).long(),
                      "has_deletion": (src.uniform(1, depth, n) < 0.1).float(),
                      "deletion_value": src.uniform(1, depth, n) * (src.uniform(1, depth, n) < 0.1),
                      "msa_paired": (src.uniform(1, depth, n) < 0.3).float(),
                      "msa_mask": rows * m[:, None, :], "token_pad_mask": m}
    elif op == "diffusion":
        d["w"] = src.weights(synthetic.diffusion_pair_shapes(depth=DIFF_LAYERS))
        d["z"], d["rel"] = src.pair(1, n, 128), src.normal(1, n, n, 128)
    else:
        raise ValueError(f"unknown op {op!r}")
    return d


def _padded(z: torch.Tensor, n_pad: int) -> torch.Tensor:
    b, n = z.shape[:2]
    out = torch.zeros((b, n_pad, n_pad) + tuple(z.shape[3:]), dtype=z.dtype, device="cuda")
    out[:, :n, :n] = z
    return out


def prepare(case: dict, seed: int) -> dict:
    op, d = case["op"], _inputs(case, seed)
    opt = pf.Options(operand=case["operand"])
    st = {"case": case, "d": d}
    if op in ("trimul", "triatt"):
        n_pad = -(-case["n"] // 64) * 64
        st["z"], st["mask"] = _padded(d["z"], n_pad), _padded(d["pair_mask"], n_pad)
        if op == "trimul":
            mod = pf.TriangleMultiplication(case["direction"] == "incoming", d["w"], opt)
        else:
            w = {(k[4:] if k.startswith("mha.") else k): v for k, v in d["w"].items()}
            mod = pf.TriangleAttention(HEAD_DIM, HEADS, case["ending"], w, opt)
        st["mod"], st["out"] = mod, torch.empty_like(st["z"])
        st["ws"] = ops.workspace(mod.workspace_bytes(1, n_pad), st["z"].device)
    elif op in ("layers", "template"):
        pf.set_fast_mode(bool(case.get("fast")))
        if op == "layers":
            mod = pf.PairformerModule(case["blocks"], HEAD_DIM, HEADS, S_DIM, S_HEADS, True, options=opt)
        else:
            mod = pf.PairformerModule(2, HEAD_DIM, HEADS, None, None, False, options=opt)
        mod.load_state_dict(d["w"])
        pf.set_fast_mode(False)
        st["mod"] = mod
    elif op == "msa":
        st["mod"] = pf.MSAModule(1, 32, MSA_HEADS, HEAD_DIM, HEADS, options=opt)
        st["mod"].load_state_dict(d["w"])
    elif op == "diffusion":
        st["mod"] = pf.DiffusionPairConditioning(DIFF_LAYERS, options=opt)
        st["mod"].load_state_dict(d["w"])
    return st


def run(state: dict):
    case, d = state["case"], state["d"]
    op = case["op"]
    if op == "trimul_fn":
        w = d["w"]
        return ops.triangle_multiplicative_update(
            d["z"], case["direction"], d["pair_mask"], w["norm_in.weight"], w["norm_in.bias"], w["p_in.weight"],
            w["g_in.weight"], w["norm_out.weight"], w["norm_out.bias"], w["p_out.weight"], w["g_out.weight"],
            variant=case["operand"])
    if op == "attn_fn":
        return ops.triangle_attention(d["q"], d["k"], d["v"], d["bias"], d["key_mask"], variant=case["operand"])
    if op == "single_fn":
        return ops.attention_pair_bias(d["s"], d["z"], d["mask"], d["s"], d["w"], S_HEADS, variant=case["operand"])
    if op == "trimul":
        return state["mod"](state["z"], state["mask"], out=state["out"], ws=state["ws"])
    if op == "triatt":
        return state["mod"](state["z"], state["mask"], out=state["out"], ws=state["ws"], n_valid=case["n"])
    if op == "layers":
        return state["mod"](d["s"], d["z"], mask=d["mask"], pair_mask=d["pair_mask"])
    if op == "template":
        return state["mod"](None, d["z"], pair_mask=d["pair_mask"])[1]
    if op == "msa":
        return state["mod"](d["z"], d["emb"], d["feats"])
    return state["mod"](d["z"], d["rel"])


# --------------------------------------------------------------------------------------
# the work a case cannot do without
# --------------------------------------------------------------------------------------
def _pair_flops(n: int, c: int, batch: int = 1) -> float:
    """Both triangle multiplications, both triangle attentions and the transition."""
    hd = HEADS * HEAD_DIM
    tm = 12.0 * n * n * c * c + 2.0 * n ** 3 * c
    ta = 10.0 * n * n * c * hd + 2.0 * n * n * c * HEADS + 4.0 * n ** 3 * hd
    return batch * (2 * tm + 2 * ta + 24.0 * n * n * c * c)


def _single_flops(n: int) -> float:
    return 2.0 * n * n * 128 * S_HEADS + 10.0 * n * C_S * C_S + 4.0 * n * n * C_S


def work(case: dict) -> dict:
    """Every input read once and every output written once; 2 operations a multiply-add."""
    op, n = case["op"], case["n"]
    z = 4.0 * n * n * 128
    if op in ("trimul_fn", "trimul"):
        return {"bytes": 2 * z + 4.0 * n * n, "flops": 12.0 * n * n * 128 * 128 + 2.0 * n ** 3 * 128}
    if op == "triatt":
        return {"bytes": 2 * z + 4.0 * n * n,
                "flops": 10.0 * n * n * 128 * 128 + 2.0 * n * n * 128 * HEADS + 4.0 * n ** 3 * 128}
    if op == "attn_fn":
        return {"bytes": 4 * z + 4.0 * HEADS * n * n + 1.0 * n * n, "flops": 4.0 * n ** 3 * 128}
    if op == "single_fn":
        return {"bytes": z + 8.0 * n * C_S + 20.0 * C_S * C_S, "flops": _single_flops(n)}
    if op == "layers":
        nb = case["blocks"]
        weights = 4.0 * sum(math.prod(s) for s in synthetic.layer_shapes().values())
        per = _pair_flops(n, 128) + _single_flops(n) + 24.0 * n * C_S * C_S
        return {"bytes": 2 * z + 8.0 * n * C_S + 4.0 * n * n + nb * weights, "flops": nb * per}
    if op == "template":
        b = case["batch"]
        return {"bytes": b * (8.0 * n * n * 64 + 4.0 * n * n), "flops": 2 * _pair_flops(n, 64, b)}
    if op == "msa":
        s = case["depth"]
        pwa = 2.0 * n * n * 128 * MSA_HEADS + 6.0 * s * n * C_M * 256 + 2.0 * s * n * n * 256
        tr = 24.0 * s * n * C_M * C_M
        opm = 4.0 * s * n * C_M * OPM_HIDDEN + 2.0 * s * (n * OPM_HIDDEN) ** 2 + 2.0 * n * n * OPM_HIDDEN ** 2 * 128
        return {"bytes": 2 * z + 4.0 * n * C_S + 24.0 * s * n, "flops": pwa + tr + opm + _pair_flops(n, 128)}
    bias = n * n * DIFF_LAYERS * 16
    return {"bytes": 3 * z + 4.0 * bias,
            "flops": 2.0 * n * n * 256 * 128 + 2 * 12.0 * n * n * 128 * 128 + 2.0 * 128 * bias}


def tolerance(case: dict):
    """About four times the distance from the 64-bit results: single operators in fp16 measured
    3.6e-4 to 7.7e-4 (their updates alone are returned), whole blocks 1.4e-4 to 6.4e-4, bf16 eight
    times those (3.0e-3 on the attention).  The block-fp8 blocks are 5.4e-2 to 6.2e-2 off, nearly
    all of it the format's own; what two implementations of it re-round differently is of that
    order.  The largest single differences are bounded by the bar of the parity tests."""
    if case.get("fast"):
        return {"rel": 0.06}
    return {"rel": 2.5e-3, "max": 2e-2} if case["operand"] == "fp16" else {"rel": 1.5e-2, "max": 0.15}


# --------------------------------------------------------------------------------------
# the same in 64 bits, by torch alone
# --------------------------------------------------------------------------------------
def _ln(x: torch.Tensor, w: torch.Tensor, b: torch.Tensor) -> torch.Tensor:
    return F.layer_norm(x, (x.shape[-1],), w, b, 1e-5)


def _trimul64(z, pm, w, incoming):
    x = _ln(z, w["norm_in.weight"], w["norm_in.bias"])
    ab = (x @ w["p_in.weight"].T) * torch.sigmoid(x @ w["g_in.weight"].T) * pm[..., None]
    a, b = ab.permute(0, 3, 1, 2).chunk(2, dim=1)
    if incoming:
        a, b = a.transpose(2, 3), b.transpose(2, 3)
    t = torch.matmul(a.contiguous(), b.transpose(2, 3).contiguous()).permute(0, 2, 3, 1)
    t = _ln(t, w["norm_out.weight"], w["norm_out.bias"]) @ w["p_out.weight"].T
    return t * torch.sigmoid(x @ w["g_out.weight"].T)


def _softmax_masked(a, key_mask, inf):
    """softmax(a + inf * (mask - 1)) as the 32-bit sum has it: where every key of a row is masked
    by the larger constant the logits vanish beside it, and the row is a plain mean."""
    if inf == 1e9:
        none = (key_mask.sum(-1, keepdim=True) == 0).to(a.dtype)
        a = a * (1 - none)
        key_mask = torch.maximum(key_mask, none)
    return torch.softmax(a + inf * (key_mask - 1), dim=-1)


def _attend64(q, k, v, bias, key_mask):
    """q, k, v [B,I,H,J,D] (q scaled), bias [B,H,J,K], key_mask [B,I,K]; rows in chunks."""
    out = torch.empty_like(q)
    step = max(1, (1 << 28) // (q.shape[0] * q.shape[2] * q.shape[3] * k.shape[3]))
    for r in range(0, q.shape[1], step):
        s = slice(r, r + step)
        a = torch.matmul(q[:, s], k[:, s].transpose(-1, -2).contiguous()) + bias[:, None]
        out[:, s] = torch.matmul(_softmax_masked(a, key_mask[:, s, None, None], 1e9), v[:, s])
    return out


def _triatt64(z, pm, w, ending, n=None):
    """``n``: only the first n tokens are keys, the others padding (None = all)."""
    if ending:
        z, pm = z.transpose(1, 2), pm.transpose(1, 2)
    x = _ln(z, w["layer_norm.weight"], w["layer_norm.bias"])
    heads = lambda k: (x @ w[k].T).unflatten(-1, (HEADS, HEAD_DIM)).transpose(2, 3).contiguous()  # noqa: E731
    q, k, v = (heads(f"mha.linear_{c}.weight") for c in "qkv")
    bias = (x @ w["linear.weight"].T).permute(0, 3, 1, 2)[..., :n].contiguous()
    k, v, pm = k[..., :n, :].contiguous(), v[..., :n, :].contiguous(), pm[..., :n]
    o = _attend64(q * HEAD_DIM ** -0.5, k, v, bias, pm).transpose(2, 3).flatten(-2)
    o = (o * torch.sigmoid(x @ w["mha.linear_g.weight"].T)) @ w["mha.linear_o.weight"].T
    return o.transpose(1, 2) if ending else o


def _transition64(x, w):
    x = _ln(x, w["norm.weight"], w["norm.bias"])
    return (F.silu(x @ w["fc1.weight"].T) * (x @ w["fc2.weight"].T)) @ w["fc3.weight"].T


def _single64(s, k_in, z, mask, w):
    split = lambda t: t.unflatten(-1, (S_HEADS, S_DIM)).transpose(1, 2).contiguous()  # noqa: E731
    q = split(s @ w["proj_q.weight"].T + w["proj_q.bias"])
    k, v = split(k_in @ w["proj_k.weight"].T), split(k_in @ w["proj_v.weight"].T)
    bias = (_ln(z, w["proj_z.0.weight"], w["proj_z.0.bias"]) @ w["proj_z.1.weight"].T).permute(0, 3, 1, 2)
    a = torch.matmul(q, k.transpose(-1, -2).contiguous()) * S_DIM ** -0.5 + bias
    o = torch.matmul(_softmax_masked(a, mask[:, None, None], 1e6), v).transpose(1, 2).flatten(-2)
    return (torch.sigmoid(s @ w["proj_g.weight"].T) * o) @ w["proj_o.weight"].T


def _layer64(s, z, mask, pm, w):
    z = z + _trimul64(z, pm, _sub(w, "tri_mul_out."), False)
    z = z + _trimul64(z, pm, _sub(w, "tri_mul_in."), True)
    z = z + _triatt64(z, pm, _sub(w, "tri_att_start."), False)
    z = z + _triatt64(z, pm, _sub(w, "tri_att_end."), True)
    z = z + _transition64(z, _sub(w, "transition_z."))
    if s is not None:
        sn = _ln(s, w["pre_norm_s.weight"], w["pre_norm_s.bias"])
        s = s + _single64(sn, sn, z, mask, _sub(w, "attention."))
        s = s + _transition64(s, _sub(w, "transition_s."))
    return s, z


def _msa64(z, emb, f, w):
    m = w["msa_proj.weight"].T[f["msa"].long()]
    for i, k in enumerate(("has_deletion", "deletion_value", "msa_paired")):
        m = m + f[k][..., None] * w["msa_proj.weight"][:, 33 + i]
    m = m + (emb @ w["s_proj.weight"].T)[:, None]
    tok = f["token_pad_mask"]
    pm = tok[:, :, None] * tok[:, None, :]
    w = _sub(w, "layers.0.")
    p = _sub(w, "pair_weighted_averaging.")
    mn = _ln(m, p["norm_m.weight"], p["norm_m.bias"])
    a = (_ln(z, p["norm_z.weight"], p["norm_z.bias"]) @ p["proj_z.weight"].T).permute(0, 3, 1, 2)
    a = _softmax_masked(a, pm[:, None], 1e6)
    v = (mn @ p["proj_m.weight"].T).unflatten(-1, (MSA_HEADS, 32))          # b s j h d
    v = v.permute(0, 3, 2, 1, 4).flatten(-2).contiguous()                   # b h j (s d)
    o = torch.matmul(a, v).unflatten(-1, (-1, 32)).permute(0, 3, 2, 1, 4).flatten(-2)
    m = m + (torch.sigmoid(mn @ p["proj_g.weight"].T) * o) @ p["proj_o.weight"].T
    m = m + _transition64(m, _sub(w, "msa_transition."))
    p = _sub(w, "outer_product_mean.")
    mn = _ln(m, p["norm.weight"], p["norm.bias"])
    mk = f["msa_mask"]
    a, b = ((mn @ p[f"proj_{c}.weight"].T) * mk[..., None] for c in "ab")
    n = z.shape[1]
    t = torch.matmul(a.flatten(2).transpose(1, 2).contiguous(), b.flatten(2))
    t = t.view(1, n, OPM_HIDDEN, n, OPM_HIDDEN).permute(0, 1, 3, 2, 4).flatten(-2)
    t = t / torch.matmul(mk.transpose(1, 2).contiguous(), mk).clamp(min=1)[..., None]
    z = z + t @ p["proj_o.weight"].T + p["proj_o.bias"]
    return _layer64(None, z, None, pm, _sub(w, "pairformer_layer."))[1]


def _to64(v):
    if isinstance(v, dict):
        return {k: _to64(x) for k, x in v.items()}
    return v.double()


def exact(case: dict, seed: int) -> Optional[object]:
    op = case["op"]
    d = _inputs(case, seed)
    d = {k: (_to64(v) if k != "key_mask" else v.double().view(1, case["n"], case["n"])) for k, v in d.items()}
    w = d.get("w")
    if op in ("trimul", "triatt"):   # the module classes work on padded tensors
        n_pad = -(-case["n"] // 64) * 64
        d["z"], d["pair_mask"] = _padded(d["z"], n_pad), _padded(d["pair_mask"], n_pad)
    if op in ("trimul_fn", "trimul"):
        return _trimul64(d["z"], d["pair_mask"], w, case["direction"] == "incoming")
    if op == "triatt":
        return _triatt64(d["z"], d["pair_mask"], w, case["ending"], case["n"])
    if op == "attn_fn":
        return _attend64(d["q"] * HEAD_DIM ** -0.5, d["k"], d["v"], d["bias"][:, 0], d["key_mask"])
    if op == "single_fn":
        return _single64(d["s"], d["s"], d["z"], d["mask"], w)
    if op == "layers":
        s, z = d["s"], d["z"]
        for i in range(case["blocks"]):
            s, z = _layer64(s, z, d["mask"], d["pair_mask"], _sub(w, f"layers.{i}."))
        return s, z
    if op == "template":
        z = d["z"]
        for i in range(2):
            z = _layer64(None, z, None, d["pair_mask"], _sub(w, f"layers.{i}."))[1]
        return z
    if op == "msa":
        return _msa64(d["z"], d["emb"], d["feats"], w)
    p = _sub(w, "pairwise_conditioner.")
    x = torch.cat((d["z"], d["rel"]), dim=-1)
    z = _ln(x, p["dim_pairwise_init_proj.0.weight"], p["dim_pairwise_init_proj.0.bias"])
    z = z @ p["dim_pairwise_init_proj.1.weight"].T
    for i in range(2):
        z = z + _transition64(z, _sub(p, f"transitions.{i}."))
    t = [_ln(z, w[f"token_trans_proj_z.{l}.0.weight"], w[f"token_trans_proj_z.{l}.0.bias"])
         @ w[f"token_trans_proj_z.{l}.1.weight"].T for l in range(DIFF_LAYERS)]
    return z, torch.cat(t, dim=-1)
