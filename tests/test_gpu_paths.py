"""GPU parity of the kernels' size- and data-dependent branches, at the sizes where they change.

Same tolerance as the parity tests (errors over the reference output's RMS: max 2e-2, mean 2e-3),
against the fp32 oracle.
"""
import pytest
import torch

from oracle import msa_ref, pairformer_ref as ref
from tt_boltz_amd import ops, pairformer
from test_gpu_fast import F32_MAX, F32_MEAN, _mx8_trimul_w, check as check_fast
from test_gpu_parity import _inputs, _msa_sub, _sub_w, check

pytestmark = pytest.mark.gpu


# ------------------------------------------------------------------------------ attention core
@pytest.mark.parametrize("shift", [-24.0, -6.0, 0.0, 12.0, 24.0])
@pytest.mark.parametrize("first_masked", [128, 127, 33, 32, 31])
def test_attention_reference_and_mask_tiles(gpu, shift, first_masked):
    """Tiles ahead of a row's first masked key run without the mask / reference fold while 0 serves
    as the softmax reference.  ``first_masked`` puts that key on both sides of a 32-key tile's
    edge; ``shift`` moves the logits of the first tile below the sum that accepts 0, of later tiles
    above the one that forces a rescale, and both ways at once over the rows.  (|logit| stays below
    32, half of the fp32 spacing at 1e9: beyond it the reference's own fully masked row is not
    the plain mean that its additive mask stands for.)"""
    g = torch.Generator().manual_seed(11)
    B, N, H, D = 1, 128, 4, 32
    q, k, v = (torch.randn((B, N, H, N, D), generator=g) for _ in range(3))
    bias = torch.randn((B, 1, H, N, N), generator=g)
    bias[..., :40] += shift
    bias[:, :, 1, :, 64:] -= shift
    mask = torch.ones((B, N, 1, 1, N))
    mask[..., first_masked:] = 0.0
    mask[:, 7, ..., 3] = 0.0     # one row with a masked key in its first tile
    mask[:, 9] = 0.0             # a fully masked row
    want = ref.triangle_attention_core(q, k, v, bias, mask, D ** -0.5)
    got = ops.triangle_attention(q.to(gpu), k.to(gpu), v.to(gpu), bias.to(gpu), mask.to(gpu))
    check(f"attention shift={shift} first_masked={first_masked}", got, want)


@pytest.mark.parametrize("level", [11.8, 7.8, 0.0, -3.0, -6.0, -9.5, -12.0])
@pytest.mark.parametrize("depth", [8.0, 12.2, 15.2])
@pytest.mark.parametrize("n_first", [32, 16, 1])
def test_attention_small_weights(gpu, level, depth, n_first):
    """Keys ``depth`` log2 units below a row's largest logits keep their share wherever the logits as a
    whole lie.  ``n_first`` of the first 32 keys have ``level``, all others ``depth`` less; v marks
    the others, so the output is their share alone.  A weight is rounded to fp16 with the largest at
    1 or above: half a spacing of subnormals, 2^-25, beside 2^-depth, and 2^-11 each for the sum and
    the output."""
    N, H, D, ln2 = 512, 4, 32, 0.6931471805599453
    q = torch.zeros((1, N, H, N, D), device=gpu)
    bias = torch.full((1, 1, H, N, N), (level - depth) * ln2, device=gpu)
    bias[..., :n_first] = level * ln2
    v = torch.ones_like(q)
    v[:, :, :, :n_first] = 0.0
    got = ops.triangle_attention(q, q, v, bias).double()
    small = (N - n_first) * 2.0 ** -depth
    want = small / (small + n_first)
    bar = 2.0 ** (depth - 25) + 2.0 ** -10
    assert ((got - want).abs().max() / want).item() < bar


# ------------------------------------------------------------------------------ trimul
@pytest.mark.parametrize("B,N", [(1, 64), (1, 192), (1, 256), (1, 320), (2, 64), (2, 320)])
@pytest.mark.parametrize("incoming", [False, True])
@pytest.mark.parametrize("plain", [False, True])
def test_trimul_direct(gpu, B, N, incoming, plain):
    """The register-weight kernels with one group of 64 positions per workgroup and with several,
    on both sides of the line between the residual MFMA and the mean correction (N = 256 / 320),
    with plain weights, for a batch, and with the three ways of adding the residual."""
    w = _sub_w(5, "tri_mul_in" if incoming else "tri_mul_out")
    z = torch.cat([_inputs(N, 5 + b)[1] for b in range(B)])
    pm = torch.cat([_inputs(N, 5 + b, pad_tail=7, rand_mask=True)[3] for b in range(B)])
    opt = pairformer.Options(weight_residuals=not plain, mean_correction=not plain)
    mod = pairformer.TriangleMultiplication(incoming, w, opt)
    want = ref.triangle_multiplication(z.to(gpu), pm.to(gpu), {k: v.to(gpu) for k, v in w.items()},
                                       "incoming" if incoming else "outgoing")
    zd, pd = z.to(gpu), pm.to(gpu).contiguous()
    update = mod(zd, pd)
    check("trimul update", update, want)
    other = torch.ones_like(zd)
    check("trimul out += update", mod(zd, pd, out=other, accumulate=True) - 1.0, want)
    inplace = zd.clone()
    mod(inplace, pd, out=inplace, accumulate=True)
    # the same update added to z: one fp32 rounding of the sum apart
    assert (inplace - (zd + update)).abs().max() <= 2.0 ** -22 * (zd.abs().max() + update.abs().max())


@pytest.mark.parametrize("B,N", [(1, 64), (2, 128), (3, 128), (1, 192)])
def test_trimul_c64_direct_line(gpu, B, N):
    """c_z = 64 on both sides of the line between the direct and the persistent kernels (512 groups
    of 64 positions on 256 CUs)."""
    from tt_boltz_amd import synthetic
    w = ref.sub(synthetic.draw({k: v for k, v in synthetic.layer_shapes(64).items() if k.startswith("tri_mul_out.")},
                               6), "tri_mul_out")
    g = torch.Generator().manual_seed(N + B)
    z = torch.randn((B, N, N, 64), generator=g)
    pm = (torch.rand((B, N, N), generator=g) > 0.1).float()
    want = ref.triangle_multiplication(z, pm, w, "outgoing")
    got = pairformer.TriangleMultiplication(False, w)(z.to(gpu), pm.to(gpu))
    check(f"trimul c64 B={B} N={N}", got, want)


# ------------------------------------------------------------------------------ triangle attention
@pytest.mark.parametrize("B,N", [(1, 64), (1, 256), (1, 320), (2, 192)])
@pytest.mark.parametrize("ending", [False, True])
@pytest.mark.parametrize("plain", [False, True])
def test_triatt_direct(gpu, B, N, ending, plain):
    """The projections with one group of 64 positions per workgroup and with several, on both sides
    of the line between the residual MFMA and the mean correction (N = 256 / 320), with plain
    weights, for a batch, with padded keys, and with the three ways of adding the residual."""
    w = _sub_w(5, "tri_att_end" if ending else "tri_att_start")
    wm = {(k[4:] if k.startswith("mha.") else k): v for k, v in w.items()}
    n = N - 9
    z = torch.zeros((B, N, N, 128))
    pm = torch.zeros((B, N, N))
    for b in range(B):
        _, zb, _, pmb = _inputs(n, 5 + b, pad_tail=7, rand_mask=True)
        z[b, :n, :n], pm[b, :n, :n] = zb[0], pmb[0]
    opt = pairformer.Options(weight_residuals=not plain, mean_correction=not plain)
    mod = pairformer.TriangleAttention(32, 4, ending, wm, opt)
    want = ref.triangle_attention(z[:, :n, :n].to(gpu), pm[:, :n, :n].to(gpu), {k: v.to(gpu) for k, v in w.items()},
                                  not ending)
    zd, pd = z.to(gpu), pm.to(gpu).contiguous()
    update = mod(zd, pd, n_valid=n)
    check("triatt update", update[:, :n, :n], want)
    other = torch.ones_like(zd)
    check("triatt out += update", mod(zd, pd, out=other, accumulate=True, n_valid=n)[:, :n, :n] - 1.0, want)
    inplace = zd.clone()
    mod(inplace, pd, out=inplace, accumulate=True, n_valid=n)
    # the same update added to z: one fp32 rounding of the sum apart
    assert (inplace - (zd + update)).abs().max() <= 2.0 ** -22 * (zd.abs().max() + update.abs().max())


@pytest.mark.parametrize("B,N", [(1, 192), (3, 192)])
@pytest.mark.parametrize("ending", [False, True])
def test_triatt_c64_groups(gpu, B, N, ending):
    """c_z = 64 with several groups of 64 positions per workgroup and an uneven last round (576 and 1728
    groups on 256 CUs), padded keys, out of place and in place."""
    from tt_boltz_amd import synthetic
    prefix = "tri_att_end" if ending else "tri_att_start"
    w = ref.sub(synthetic.draw({k: v for k, v in synthetic.layer_shapes(64, transform_s=False).items()
                                if k.startswith(prefix + ".")}, 6), prefix)
    mod = pairformer.TriangleAttention(32, 4, ending, {(k[4:] if k.startswith("mha.") else k): v for k, v in w.items()})
    g = torch.Generator().manual_seed(N + B)
    n = N - 9
    z, pm = torch.zeros((B, N, N, 64)), torch.zeros((B, N, N))
    z[:, :n, :n] = torch.randn((B, n, n, 64), generator=g)
    pm[:, :n, :n] = (torch.rand((B, n, n), generator=g) > 0.1).float()
    want = ref.triangle_attention(z[:, :n, :n].to(gpu), pm[:, :n, :n].to(gpu), {k: v.to(gpu) for k, v in w.items()},
                                  not ending)
    zd, pd = z.to(gpu), pm.to(gpu)
    update = mod(zd, pd, n_valid=n)
    check("triatt c64 update", update[:, :n, :n], want)
    inplace = zd.clone()
    mod(inplace, pd, out=inplace, accumulate=True, n_valid=n)
    # the same update added to z: one fp32 rounding of the sum apart
    assert (inplace - (zd + update)).abs().max() <= 2.0 ** -22 * (zd.abs().max() + update.abs().max())


def test_template_stack_groups(gpu):
    """Two templates of 200 tokens through the c_z = 64 stack: eight groups per workgroup."""
    from tt_boltz_amd import synthetic
    N = 200
    w = synthetic.stack_weights(2, 44, c_z=64, transform_s=False)
    z = torch.randn((2, N, N, 64), generator=torch.Generator().manual_seed(45))
    m = torch.ones((2, N))
    m[0, 181:], m[1, 190:] = 0, 0
    pm = m[:, :, None] * m[:, None, :]
    want = torch.cat([ref.pairformer_stack(None, z[b:b + 1].to(gpu), None, pm[b:b + 1].to(gpu),
                                           {k: v.to(gpu) for k, v in w.items()}, 2)[1] for b in range(2)])
    mod = pairformer.PairformerModule(2, 32, 4, None, None, False)
    mod.load_state_dict(w)
    _, got = mod(None, z.to(gpu), pair_mask=pm.to(gpu))
    check("template stack", got, want)


# ------------------------------------------------------------------------------ boundary padding
@pytest.mark.parametrize("N,n_pad", [(1, 64), (45, 64), (64, 64), (130, 192)])
@pytest.mark.parametrize("form", ["plain", "transposed", "sliced", "offset", "expanded", "half", "grad"])
@pytest.mark.parametrize("shape,dims", [("BNNC", (1, 2)), ("BNC", (1,)), ("BNHND", (1, 3)), ("BNN", (1, 2)),
                                        ("BSN", (2,)), ("BN", (1,))])
def test_padded(gpu, N, n_pad, form, shape, dims):
    """The padding kernel against a fill and a copy, exactly: every layout it takes (strides,
    misaligned data, one channel, an odd channel count, nothing to pad) and what is left to torch."""
    size = [{"B": 2, "N": N, "C": 20, "H": 3, "D": 5, "S": 7}[c] for c in shape]
    g = torch.Generator(device=gpu).manual_seed(N)
    x = torch.randn(size, generator=g, device=gpu)
    if form == "transposed":
        d = 2 if len(size) > 2 else 1
        x = x.transpose(d - 1, d).contiguous().transpose(d - 1, d)
    elif form == "sliced":
        x = torch.randn([n + 3 for n in size], generator=g, device=gpu)[tuple(slice(2, 2 + n) for n in size)]
    elif form == "offset":
        x = torch.randn(x.numel() + 1, generator=g, device=gpu)[1:].view(size)
    elif form == "expanded":
        x = x[:1].expand(size)
    elif form == "half":
        x = x.half()
    elif form == "grad":
        x.requires_grad_(True)
    got = ops.padded(x, n_pad, x.device, dims)
    want = torch.zeros([n_pad if d in dims else n for d, n in enumerate(size)], device=gpu)
    want[tuple(slice(0, n) for n in size)] = x.detach().float()
    assert got.is_contiguous() and got.dtype == torch.float32 and torch.equal(got, want)


@pytest.mark.parametrize("copy", ["pad_pair", "to_device_padded"])
def test_padded_copies_under_torch_transforms(gpu, copy):
    """A forward-mode tangent is padded along, and traces replay the padding on another input."""
    from torch.autograd import forward_ad
    from torch.fx.experimental.proxy_tensor import make_fx
    fn = (lambda t: ops.pad_pair(t, 64)) if copy == "pad_pair" else \
        (lambda t: ops.to_device_padded(t, 64, t.device, True))
    z, other = torch.randn((2, 1, 45, 45, 8), generator=torch.Generator().manual_seed(1)).to(gpu)
    want = torch.nn.functional.pad(other, (0, 0, 0, 19, 0, 19))
    with forward_ad.dual_level():
        out = forward_ad.unpack_dual(fn(forward_ad.make_dual(z, other)))
        assert torch.equal(out.tangent, want)
    assert torch.equal(torch.jit.trace(fn, z, check_trace=False)(other), want)
    assert torch.equal(make_fx(fn)(z)(other), want)


# ------------------------------------------------------------------------------ single track
@pytest.mark.parametrize("B,N", [(1, 33), (1, 64), (2, 100), (1, 413)])
@pytest.mark.parametrize("masked", [False, True])
@pytest.mark.parametrize("fast", [False, True])
def test_attention_pair_bias_unpadded(gpu, B, N, masked, fast):
    """The pair bias read from an unpadded z (odd row lengths, a batch) against the same call on a
    padded z: identical bits."""
    w = {k: v for k, v in _sub_w(9, "attention").items()}
    g = torch.Generator().manual_seed(N)
    s, z = torch.randn((B, N, 384), generator=g).to(gpu), torch.randn((B, N, N, 128), generator=g).to(gpu)
    mask = (torch.rand((B, N), generator=g) > 0.2).float().to(gpu) if masked else None
    got = ops.attention_pair_bias(s, z, mask, s, w, fast=fast)
    n_pad = ops.padded_len(N)
    sp, zp = ops.padded(s, n_pad, s.device, (1,)), ops.pad_pair(z, n_pad)
    mp = torch.zeros((B, n_pad), device=gpu)
    mp[:, :N] = 1.0 if mask is None else mask
    ws = ops.workspace(ops.apb_workspace_bytes(B, n_pad, 384, 16), gpu)
    out = torch.empty_like(sp)
    ops.launch_apb(sp, sp, zp, mp, out, ops.convert_weights(w, gpu), 16, ws, accumulate=False, n_valid=N, fast=fast)
    assert torch.equal(got, out[:, :N])
    if not fast:
        check("attention_pair_bias", got, ref.attention_pair_bias(s.cpu(), z.cpu(), torch.ones((B, N)) if mask is None
                                                                  else mask.cpu(), s.cpu(), w))


# ------------------------------------------------------------------------------ alignment
def _odd(t):
    """A contiguous copy of ``t`` that begins 4 bytes past a 16-byte boundary."""
    out = torch.empty(t.numel() + 1, dtype=t.dtype, device=t.device)[1:].view(t.shape)
    return out.copy_(t)


@pytest.mark.parametrize("op", ["apb", "trimul", "triatt", "token_bias", "cond_proj", "pwa"])
@pytest.mark.parametrize("N", [50, 64])
def test_caller_arrays_at_odd_addresses(gpu, op, N):
    """A z read where it is and LayerNorm vectors off 16-byte boundaries: identical bits."""
    g = torch.Generator().manual_seed(N)
    z = torch.randn((1, N, N, 128), generator=g).to(gpu)
    sub = {"apb": "attention", "trimul": "tri_mul_out", "triatt": "tri_att_start"}
    if op in sub:
        w = ops.convert_weights(_sub_w(31, sub[op]), gpu, strip="mha.")
    elif op == "pwa":
        w = ops.convert_weights({k: v.to(gpu) for k, v in _msa_sub(5, "pair_weighted_averaging").items()}, gpu)
    else:
        c = 256 if op == "cond_proj" else 4 * 128
        w = {"w": 1 + 0.1 * torch.randn(c, generator=g).to(gpu), "b": 0.1 * torch.randn(c, generator=g).to(gpu)}
        rows = (0.1 * torch.randn((128, 256 if op == "cond_proj" else 128), generator=g)).half().to(gpu)
    zp = ops.pad_pair(z, 64)

    def run(w, z):
        if op == "apb":
            s = torch.randn((1, N, 384), generator=torch.Generator().manual_seed(3)).to(gpu)
            return ops.attention_pair_bias(s, z, None, s, w)
        if op == "trimul":
            out, ws = torch.empty_like(zp), ops.workspace(ops.trimul_workspace_bytes(1, 64), gpu)
            ops.launch_trimul(zp, out, None, w, 0, ws, False)
        elif op == "triatt":
            out, ws = torch.empty_like(zp), ops.workspace(ops.triatt_workspace_bytes(1, 64), gpu)
            ops.launch_triatt(zp, out, None, w, False, ws, False, n_valid=N)
        elif op == "token_bias":
            out = torch.empty((N * N, 128), device=gpu)
            ops.launch_token_pair_bias(z, w["w"], w["b"], rows, out, 4, 32, 0, 1.0)
        elif op == "cond_proj":
            out = torch.empty((N * N, 128), device=gpu)
            ops.launch_pair_cond_proj(z, 2 * z, w["w"], w["b"], rows, out)
        else:
            m = torch.randn((1, 5, 64, 64), generator=torch.Generator().manual_seed(4)).to(gpu)
            out, ws = torch.empty_like(m), ops.workspace(ops.pwa_workspace_bytes(1, 5, 64), gpu)
            ops.launch_pwa(m, zp, None, out, w, ws, accumulate=False)
        return out
    want = run(w, z)
    got = run({k: _odd(v) if v.dim() == 1 and v.dtype == torch.float32 else v for k, v in w.items()}, _odd(z))
    assert torch.equal(got, want)


# ------------------------------------------------------------------------------ pair transition
@pytest.mark.parametrize("rows", [1, 31, 33, 64, 65, 16384, 16385])
@pytest.mark.parametrize("hidden", [128, 512])
@pytest.mark.parametrize("accumulate", [False, True])
def test_transition_split(gpu, rows, hidden, accumulate):
    """The hidden-split transition up to one workgroup of 64 pairs per CU (16384 on 256 CUs) and the
    one-chain kernel just above: partial tiles, an odd number of tiles, two blocks per half and
    more."""
    from tt_boltz_amd import synthetic
    shapes = {"norm.weight": (128,), "norm.bias": (128,), "fc1.weight": (hidden, 128), "fc2.weight": (hidden, 128),
              "fc3.weight": (128, hidden)}
    raw = synthetic.draw(shapes, 13)
    w = ops.convert_weights(raw, gpu)
    w["fc3.weight.lo"] = ops.opw_lo(raw["fc3.weight"], gpu)
    x = torch.randn((rows, 128), generator=torch.Generator().manual_seed(rows))
    xd = torch.cat([x, torch.full((64, 128), 7.0)]).to(gpu)   # guard rows behind the last one
    out = xd.clone()
    ops.launch_transition(xd[:rows], out[:rows], w, None, accumulate)
    want = ref.transition(x, raw)
    check("transition", out[:rows] - x.to(gpu) if accumulate else out[:rows], want)
    assert torch.equal(out[rows:], xd[rows:])


@pytest.mark.parametrize("rows", [1, 63, 64, 65, 32 * 1031])
@pytest.mark.parametrize("hidden", [256, 512])
@pytest.mark.parametrize("mode", ["update", "accumulate", "inplace", "corrected"])
def test_transition_direct(gpu, rows, hidden, mode):
    """The register-weight transition: partial groups of 64 rows, more groups than CUs, the residual
    from another tensor and in place, and the mean correction (all rows are its sample up to 8192)."""
    from tt_boltz_amd import synthetic
    shapes = {"norm.weight": (128,), "norm.bias": (128,), "fc1.weight": (hidden, 128), "fc2.weight": (hidden, 128),
              "fc3.weight": (128, hidden)}
    raw = synthetic.draw(shapes, 17)
    w = ops.convert_weights(raw, gpu)
    x = torch.randn((rows, 128), generator=torch.Generator().manual_seed(rows))
    want = ref.transition(x, raw)
    xd = torch.cat([x, torch.full((64, 128), 7.0)]).to(gpu)   # guard rows behind the last one
    if mode == "corrected":
        w["fc3.weight.lo"] = ops.opw_lo(raw["fc3.weight"], gpu)
        ws = ops.workspace(ops.transition_workspace_bytes(rows, 128, hidden), gpu)
        out = torch.full_like(xd, 3.0)
        ops.launch_transition(xd[:rows], out[:rows], w, ws, False, fc3_mean_fix=True)
        check("transition corrected", out[:rows], want)
        assert (out[rows:] == 3.0).all()
        return
    out = xd if mode == "inplace" else torch.full_like(xd, 3.0)
    keep = out[rows:].clone()
    ops.launch_transition(xd[:rows], out[:rows], w, None, mode != "update")
    base = {"update": 0.0, "accumulate": 3.0, "inplace": x.to(gpu)}[mode]
    check(f"transition {mode}", out[:rows] - base, want)
    assert torch.equal(out[rows:], keep)


@pytest.mark.parametrize("N,mean_fix", [(320, False), (384, True)])
def test_transition_residual_line(gpu, N, mean_fix):
    """The module takes the fc3 residual as hi + lo up to 400 pairs per CU (102400 on 256 CUs) and
    through the mean correction above."""
    mod = pairformer.Transition(_sub_w(13, "transition_z"))
    z = torch.randn((1, N, N, 128), generator=torch.Generator().manual_seed(N)).to(gpu)
    want = torch.empty_like(z)
    ws = ops.workspace(mod.workspace_bytes(N * N), gpu)
    ops.launch_transition(z, want, mod.w, ws, False, fc3_mean_fix=mean_fix)
    other = torch.empty_like(z)
    ops.launch_transition(z, other, mod.w, ws, False, fc3_mean_fix=not mean_fix)
    assert torch.equal(mod(z), want) and not torch.equal(want, other)


@pytest.mark.parametrize("B,N", [(1, 64), (2, 96), (1, 352)])
def test_transition_direct_pair_bias(gpu, B, N):
    """The pair bias of the updated rows from the same kernel against the bias kernel on them (odd
    numbers of 32-row tiles, a batch)."""
    w = ops.convert_weights(_sub_w(21, "transition_z"), gpu)
    wa = ops.convert_weights(_sub_w(22, "attention"), gpu)
    g = torch.Generator().manual_seed(N)
    z = torch.randn((B, N, N, 128), generator=g).to(gpu)
    s = torch.randn((B, N, 384), generator=g).to(gpu)
    n = ops.apb_workspace_bytes(B, N, 384, 16)
    ws = [ops.workspace(n, gpu).fill_(0) for _ in range(2)]
    out = torch.empty_like(z)
    ops.launch_transition(z, out, w, None, False, pair_bias=(s, wa, 16, ws[0], 1e-5))
    ops.launch_apb(s, s, out, None, s, wa, 16, ws[1], False, part="bias")
    start = 5 * B * N * 384 * 4
    got, want = (t[start:start + B * 16 * N * N * 4].view(torch.float32) for t in ws)
    # one LayerNorm each, summed in another order: op_t rounding ties aside the bits agree
    check("fused pair bias", got, want, max_tol=5e-3, mean_tol=1e-4)


# ------------------------------------------------------------------------------ fast-mode trimul
@pytest.mark.parametrize("B,N", [(1, 128), (2, 128), (1, 384), (1, 512)])
@pytest.mark.parametrize("incoming", [False, True])
@pytest.mark.parametrize("masked", [False, True])
def test_trimul_mx8_groups(gpu, B, N, incoming, masked):
    """One group of 128 positions per workgroup and several, a batch, no mask and one with single
    masked pairs everywhere; the tolerances of the fast-mode parity tests."""
    w = _sub_w(5, "tri_mul_in" if incoming else "tri_mul_out")
    z = torch.cat([_inputs(N, 5 + b)[1] for b in range(B)])
    pm = torch.cat([_inputs(N, 5 + b, pad_tail=7, rand_mask=True)[3] for b in range(B)])
    pm = pm if masked else torch.ones_like(pm)
    wd = _mx8_trimul_w(w, gpu)
    zd, out = z.to(gpu), torch.empty_like(z, device=gpu)
    ws = ops.workspace(ops.trimul_mx8_workspace_bytes(B, N), gpu)
    ops.launch_trimul_mx8(zd, out, pm.to(gpu).contiguous() if masked else None, wd, int(incoming), ws,
                          accumulate=False)
    want = ref.triangle_multiplication(zd, pm.to(gpu), {k: v.to(gpu) for k, v in w.items()},
                                       "incoming" if incoming else "outgoing")
    check_fast("trimul mx8", out, want, F32_MAX, F32_MEAN)


# ------------------------------------------------------------------------------ diffusion conditioning
@pytest.mark.parametrize("N", [1, 7, 8, 13, 131])
@pytest.mark.parametrize("depth,heads", [(1, 32), (24, 16), (16, 32), (4, 24)])
@pytest.mark.parametrize("layout", [0, 1])
def test_token_bias_blocks(gpu, N, depth, heads, layout):
    """One to sixteen output blocks (some waves with two), layers that end inside a block, partial
    and several groups of 64 pairs, both layouts."""
    from tt_boltz_amd.diffusion import TokenTransformerPairBias
    g = torch.Generator().manual_seed(N)
    w = {}
    for l in range(depth):
        w[f"token_trans_proj_z.{l}.0.weight"] = 1 + 0.1 * torch.randn(128, generator=g)
        w[f"token_trans_proj_z.{l}.0.bias"] = 0.1 * torch.randn(128, generator=g)
        w[f"token_trans_proj_z.{l}.1.weight"] = 0.1 * torch.randn((heads, 128), generator=g)
    z = torch.randn((1, N, N, 128), generator=g)
    from oracle import diffusion_ref
    want = 0.5 * diffusion_ref.token_trans_bias(z, w, depth)
    M = depth * heads
    buf = torch.full((N * N * M + 64,), 7.0, device=gpu)   # guard values behind the output
    out = buf[:N * N * M].view(*((1, N, N, M) if layout == 0 else (M, 1, N, N)))
    TokenTransformerPairBias(depth, w)(z.to(gpu), layout, 0.5, out)
    check("token bias", out if layout == 0 else out.permute(1, 2, 3, 0), want)
    assert (buf[N * N * M:] == 7.0).all()


@pytest.mark.parametrize("rows", [1, 63, 64, 65, 64 * 256 + 1])
def test_cond_proj_groups(gpu, rows):
    """Partial and several groups of 64 pairs."""
    from oracle.pairformer_ref import layer_norm, linear
    g = torch.Generator().manual_seed(rows)
    z, r = (torch.randn((rows, 128), generator=g) for _ in range(2))
    lw, lb = 1 + 0.1 * torch.randn(256, generator=g), 0.1 * torch.randn(256, generator=g)
    w = 0.1 * torch.randn((128, 256), generator=g)
    want = linear(layer_norm(torch.cat((z, r), -1), lw, lb), w)
    out = torch.full((rows + 64, 128), 7.0, device=gpu)
    ops.launch_pair_cond_proj(z.to(gpu), r.to(gpu), lw.to(gpu), lb.to(gpu), ops.opw(w, gpu), out[:rows])
    check("cond proj", out[:rows], want)
    assert (out[rows:] == 7.0).all()


@pytest.mark.parametrize("B,S,N", [(1, 1, 64), (1, 31, 128), (2, 33, 64), (1, 700, 192)])
@pytest.mark.parametrize("masked", [False, True])
def test_pair_weighted_averaging_groups(gpu, B, S, N, masked):
    """One and several groups of 64 tokens and tiles of 32 sequences a workgroup, remainders of
    sequences, batches; into another tensor and in place."""
    w = {k: v.to(gpu) for k, v in _msa_sub(5, "pair_weighted_averaging").items()}
    g = torch.Generator().manual_seed(S + N)
    m = torch.randn((B, S, N, 64), generator=g).to(gpu)
    z = torch.randn((B, N, N, 128), generator=g).to(gpu)
    pm = torch.ones((B, N, N), device=gpu)
    if masked:
        pm[:, :, N - 13:] = 0
    want = msa_ref.pair_weighted_averaging(m, z, pm, w)
    wd = ops.convert_weights(w, gpu, ops.DEFAULT_VARIANT)
    ws = ops.workspace(ops.pwa_workspace_bytes(B, S, N), gpu)
    out = torch.full((B * S * N + 64, 64), 7.0, device=gpu)
    dst = out[:B * S * N].view_as(m)
    ops.launch_pwa(m, z, pm if masked else None, dst, wd, ws, accumulate=False)
    check(f"pwa B={B} S={S} N={N}", dst, want)
    assert (out[B * S * N:] == 7.0).all()
    want = m + dst
    ops.launch_pwa(m, z, pm if masked else None, m, wd, ws)
    assert torch.equal(m, want)
