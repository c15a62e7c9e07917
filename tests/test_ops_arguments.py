"""What the fused-op wrappers hand to the library, for arguments in shapes other than the call's own.

On the CPU, with the library recorded in place of being called: every tensor has to be of the call's
size (the kernels read that much from its pointer), broadcast as torch broadcasts, or refused.
"""
import pytest
import torch

from tt_boltz_amd import _lib, msa, ops


class Recorder:
    """Stands for the library: keeps the tensors behind the pointers, the calls and their arguments."""

    def __init__(self, monkeypatch):
        self.tensors, self.calls = {}, []
        monkeypatch.setattr(ops, "_require_gpu", lambda *ts: torch.device("cpu"))
        monkeypatch.setattr(ops, "_stream", lambda: 0)
        monkeypatch.setattr(ops, "_ptr", self.ptr)
        monkeypatch.setattr(_lib, "load", lambda *a: self)

    def ptr(self, t):
        if t is None:
            return None
        assert t.is_contiguous()
        self.tensors[t.data_ptr()] = t
        return t.data_ptr()

    def __getattr__(self, name):
        def call(*args):
            if name.endswith("workspace_size"):
                return 64
            self.calls.append((name, args))
            return 0
        return call


@pytest.fixture
def lib(monkeypatch):
    return Recorder(monkeypatch)


# ------------------------------------------------------------------------------ triangle attention
@pytest.mark.parametrize("N", [50, 64])
@pytest.mark.parametrize("shape", ["batch", "heads", "rows", "channels"])
def test_triangle_attention_broadcasts_k_and_v(lib, N, shape):
    B, H, D = 2, 4, 32
    g = torch.Generator().manual_seed(1)
    size = {"batch": (1, N, H, N, D), "heads": (B, N, 1, N, D), "rows": (B, 1, H, N, D), "channels": (B, N, H, N, 1)}[shape]
    q = torch.randn((B, N, H, N, D), generator=g)
    k, v = torch.randn(size, generator=g), torch.randn(size, generator=g)
    ops.triangle_attention(q, k, v, torch.zeros((B, 1, H, N, N)))
    (name, args), = lib.calls
    assert name == "pf_tri_attention"
    for given, ptr in zip((q, k, v), args):
        got = lib.tensors[ptr]
        assert got.shape == (B, 64, H, 64, D)
        assert torch.equal(got[:, :N, :, :N], given.expand(B, N, H, N, D))
        assert got[:, N:].abs().sum() == 0 and got[:, :, :, N:].abs().sum() == 0


@pytest.mark.parametrize("N", [50, 64])
@pytest.mark.parametrize("size", [(3, None, 4, None, 32), (2, 7, 4, None, 32), (2, None, 2, None, 32),
                                  (2, None, 4, None, 16)])
def test_triangle_attention_refuses_other_shapes(lib, N, size):
    q = torch.zeros((2, N, 4, N, 32))
    other = torch.zeros([N if n is None else n for n in size])
    for k, v in ((other, q), (q, other)):
        with pytest.raises(RuntimeError):
            ops.triangle_attention(q, k, v, torch.zeros((2, 1, 4, N, N)))
    assert not lib.calls


# ------------------------------------------------------------------------------ single track
def _apb(B, N, k_in=None, z=None, mask=None):
    g = torch.Generator().manual_seed(2)
    w = {f"proj_{k}.weight": torch.randn((384, 384), generator=g) for k in "qkvgo"}
    w.update({"proj_q.bias": torch.zeros(384), "proj_z.0.weight": torch.ones(128), "proj_z.0.bias": torch.zeros(128),
              "proj_z.1.weight": torch.randn((16, 128), generator=g)})
    s = torch.randn((B, N, 384), generator=g)
    z = torch.randn((B, N, N, 128), generator=g) if z is None else z
    return ops.attention_pair_bias(s, z, mask, s if k_in is None else k_in, w)


def _apb_args_of(lib):
    (name, args), = lib.calls
    assert name == "pf_apb_fwd_unpadded"
    return args[0]._obj, args[1]


@pytest.mark.parametrize("N", [50, 64])
@pytest.mark.parametrize("size", [(1, None, 384), (2, 1, 384), (2, None, 1)])
def test_attention_pair_bias_broadcasts_k_in(lib, N, size):
    k_in = torch.randn([N if n is None else n for n in size])
    _apb(2, N, k_in)
    a, _ = _apb_args_of(lib)
    got = lib.tensors[a.k_in]
    assert got.shape == (2, 64, 384)
    assert torch.equal(got[:, :N], k_in.expand(2, N, 384)) and got[:, N:].abs().sum() == 0


@pytest.mark.parametrize("N", [50, 64])
@pytest.mark.parametrize("size", [(3, None, 384), (2, 40, 384), (2, 80, 384), (2, None, 383)])
def test_attention_pair_bias_refuses_other_k_in(lib, N, size):
    with pytest.raises(RuntimeError):
        _apb(2, N, torch.zeros([N if n is None else n for n in size]))
    assert not lib.calls


@pytest.mark.parametrize("N", [50, 64])
@pytest.mark.parametrize("size", [(1, None), (None,), (2, 1), (1, 2, None)])
def test_attention_pair_bias_broadcasts_mask(lib, N, size):
    mask = torch.ones([N if n is None else n for n in size])
    _apb(2, N, mask=mask)
    a, _ = _apb_args_of(lib)
    assert torch.equal(lib.tensors[a.mask], torch.nn.functional.pad(torch.ones(2, N), (0, 64 - N)))


# ------------------------------------------------------------------------------ padded copies
PAIR_COPIES = {"pad_pair": lambda z, n: ops.pad_pair(z, n),
               # (a CPU tensor takes another path there: the meta device stands for the GPU)
               "to_device_padded": lambda z, n: ops.to_device_padded(z, n, z.device, True)}


@pytest.mark.parametrize("copy", PAIR_COPIES)
@pytest.mark.parametrize("size", [(1, 50, 40, 8), (1, 40, 50, 8), (1, 65, 65, 8), (1, 1, 50, 8)])
def test_pair_copies_refuse_what_is_not_square(copy, size):
    z = torch.ones(size, device="cpu" if copy == "pad_pair" else "meta")
    with pytest.raises(RuntimeError):
        PAIR_COPIES[copy](z, 64)


def test_pad_pair_broadcasts_one_column():
    z = torch.randn((2, 50, 1, 8))
    got = ops.pad_pair(z, 64)
    assert torch.equal(got, torch.nn.functional.pad(z.expand(2, 50, 50, 8), (0, 0, 0, 14, 0, 14)))
    assert ops.to_device_padded(z.to("meta"), 64, torch.device("meta"), True).shape == (2, 64, 64, 8)


@pytest.mark.parametrize("N", [50, 64])
def test_triangle_multiplication_refuses_what_is_not_square(lib, N):
    for size in ((1, N, N - 10, 128), (1, N, N + 1, 128)):
        with pytest.raises(RuntimeError):
            ops.triangle_multiplicative_update(torch.ones(size))
    assert not lib.calls


@pytest.mark.parametrize("N", [50, 64])
def test_attention_pair_bias_reads_z_of_its_own_length(lib, N):
    z = torch.randn((2, N, N, 128))
    _apb(2, N, z=z)
    a, z_n = _apb_args_of(lib)
    assert z_n == N and lib.tensors[a.z] is z   # unpadded, where it is


@pytest.mark.parametrize("N", [50, 64])
@pytest.mark.parametrize("tokens", [40, 1, 60])
def test_attention_pair_bias_pads_z_of_other_tokens(lib, N, tokens):
    """As the padded copy always was: zeros past z's own tokens, in the s grid's row length."""
    z = torch.randn((2, tokens, tokens, 128))
    _apb(2, N, z=z)
    a, z_n = _apb_args_of(lib)
    pad = 64 - tokens
    assert z_n == 64
    assert torch.equal(lib.tensors[a.z], torch.nn.functional.pad(z, (0, 0, 0, pad, 0, pad)))


@pytest.mark.parametrize("N", [50, 64])
def test_attention_pair_bias_broadcasts_z(lib, N):
    z = torch.randn((1, N, N, 128))
    _apb(2, N, z=z)
    a, z_n = _apb_args_of(lib)
    assert z_n == N and torch.equal(lib.tensors[a.z], z.expand(2, N, N, 128))


@pytest.mark.parametrize("N", [50, 64])
@pytest.mark.parametrize("size", [(2, 65, 65, 128), (2, 50, 40, 128), (3, 50, 50, 128), (2, 64, 64, 64)])
def test_attention_pair_bias_refuses_other_z(lib, N, size):
    with pytest.raises(RuntimeError):
        _apb(2, N, z=torch.zeros(size))
    assert not lib.calls


# ------------------------------------------------------------------------------ MSA inputs
def _msa_inputs(emb, B=2, S=3, N=50):
    feats = {k: torch.ones((B, S, N)) for k in ("has_deletion", "deletion_value", "msa_paired", "msa_mask")}
    feats["msa"] = torch.zeros((B, S, N), dtype=torch.int64)
    return msa.device_inputs(emb, feats, 64, torch.device("cpu"))


@pytest.mark.parametrize("size", [(2, 50, 6), (1, 50, 6), (50, 6), (2, 1, 6), (1, 2, 50, 6)])
def test_msa_inputs_broadcast_emb(size):
    emb = torch.randn(size)
    got = _msa_inputs(emb)["emb"]
    want = emb if emb.dim() < 4 else emb[0]
    assert torch.equal(got, torch.nn.functional.pad(want.expand(2, 50, 6), (0, 0, 0, 14)))


@pytest.mark.parametrize("size", [(2, 40, 6), (2, 60, 6), (3, 50, 6)])
def test_msa_inputs_refuse_other_emb(size):
    with pytest.raises(RuntimeError):
        _msa_inputs(torch.ones(size))


# ------------------------------------------------------------------------------ size-1 dimensions
def test_size_one_dimensions_may_differ_where_nothing_is_padded(lib):
    """At N = 64 the kernels read the caller's memory as it is: an unbatched z or k_in, a mask with
    dimensions of size 1 between."""
    N = 64
    z, k_in, mask = torch.randn((N, N, 128)), torch.randn((1, 1, N, 384)), torch.ones((1, 1, 1, N))
    _apb(1, N, k_in, z, mask)
    a, z_n = _apb_args_of(lib)
    assert z_n == N and torch.equal(lib.tensors[a.z], z[None])
    assert torch.equal(lib.tensors[a.k_in], k_in[0]) and torch.equal(lib.tensors[a.mask], mask[0, 0])
    lib.calls.clear()
    _apb(2, N, mask=torch.arange(2.0 * N).view(2, 1, N))
    a, _ = _apb_args_of(lib)
    assert torch.equal(lib.tensors[a.mask], torch.arange(2.0 * N).view(2, N))


def test_size_one_dimensions_where_padding_refuses_them(lib):
    for z, mask in ((torch.zeros((50, 50, 128)), None), (None, torch.ones((2, 1, 50)))):
        with pytest.raises((RuntimeError, ValueError)):
            _apb(1 if z is not None else 2, 50, z=z, mask=mask)
    assert not lib.calls
