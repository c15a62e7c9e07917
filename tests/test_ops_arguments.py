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
