"""NF4 quantisation on the GPU (csrc/nf4_quantize.hip): the bytes and scales of
quant.py's torch steps, bit for bit."""

import pytest
import torch

from ttspipe_amd import quant


def test_quantize_bins_hold_one_midpoint_each():
    """What nf4_quantize.hip's 64 bins over [-1, 1] rest on: at most one
    midpoint a bin, none within 1e-3 of an edge (a bin index is rounded by a
    few 1e-7)."""
    code = torch.tensor(quant.NF4_CODE, dtype=torch.float64)
    t = ((code[:-1] + code[1:]) / 2 + 1) * 32
    assert len(set(t.long().tolist())) == 15
    frac = t - t.floor()
    assert float(torch.minimum(frac, 1 - frac).min()) * 2 / 64 > 1e-3


def _same(a, b):
    assert (a is None) == (b is None)
    if a is not None:
        assert a.shape == b.shape and a.dtype == b.dtype and a.device == b.device
        nan = torch.isnan(a.float())
        assert torch.equal(nan, torch.isnan(b.float())) and torch.equal(a[~nan], b[~nan])


@pytest.mark.gpu
@pytest.mark.parametrize("n,bs", [(2, 64), (62, 64), (64, 64), (130, 128), (512, 512), (514, 64), (2048, 256),
                                  (8192 * 4 + 1026, 64), (9728 * 256, 64), (1 << 20, 128), (100 * 512, 512)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("nested", [True, False])
def test_quantize_kernel_equals_the_torch_steps(monkeypatch, n, bs, dtype, nested):
    """Sizes at and around a lane's, a wave's and a workgroup's elements, whole
    and ragged blocks; among the blocks one of zeros, one with a NaN, one with
    an infinity, one of subnormals, and values on the code midpoints."""
    g = torch.Generator(device="cuda").manual_seed(n + bs)
    w = (torch.randn(n, generator=g, device="cuda") * 0.02)
    code = torch.tensor(quant.NF4_CODE, device="cuda")
    if n >= 8 * bs:
        w[bs:2 * bs] = 0
        w[2 * bs + 3] = float("nan")
        w[3 * bs + 5] = -float("inf")
        w[4 * bs:5 * bs] *= 1e-38
        w[5 * bs:5 * bs + 15] = (code[:-1] + code[1:]) / 2
        w[5 * bs + 15] = 1.0
        w[5 * bs + 16:6 * bs].clamp_(-1, 1)
    w = w.to(dtype)
    assert quant._kernel_serves(w, w, bs)
    packed, state = quant.quantize_4bit(w.view(2, -1), bs, compress_statistics=nested)
    monkeypatch.setattr(quant, "_kernel_serves", lambda *a: False)
    packed_t, state_t = quant.quantize_4bit(w.view(2, -1), bs, compress_statistics=nested)
    assert torch.equal(packed, packed_t) and state.shape == state_t.shape
    _same(state.absmax, state_t.absmax)
    _same(state.code, state_t.code)
    _same(state.offset, state_t.offset)
    if nested:
        _same(state.state2.absmax, state_t.state2.absmax)
        _same(state.state2.code, state_t.state2.code)


@pytest.mark.gpu
def test_quantize_forms_the_kernel_leaves_to_torch():
    """Gradients, other dtypes, wide blocks and misaligned views keep the torch steps."""
    w = torch.randn(4096, device="cuda")
    assert not quant._kernel_serves(w.double(), w.double(), 64) and not quant._kernel_serves(w, w, 1024)
    assert not quant._kernel_serves(w, w[1:], 64)
    p = torch.nn.Parameter(w)
    assert not quant._kernel_serves(p, p.view(-1), 64)
    with torch.no_grad():
        assert quant._kernel_serves(p, p.view(-1), 64)
    a, b = quant.quantize_4bit(w[2:2050], 64), quant.quantize_4bit(w[2:2050].clone(), 64)  # misaligned, aligned
    assert torch.equal(a[0], b[0]) and torch.equal(a[1].absmax, b[1].absmax)


@pytest.mark.gpu
@pytest.mark.parametrize("nested", [True, False])
def test_quantize_without_the_library_runs_the_torch_steps(monkeypatch, tmp_path, nested):
    """A weight on the GPU is quantised to the same bytes where the library is
    not built (or not shipped)."""
    from ttspipe_amd import _lib

    w = torch.randn(64, 128, generator=torch.Generator(device="cuda").manual_seed(3), device="cuda").bfloat16()
    packed, state = quant.quantize_4bit(w, 64, compress_statistics=nested)
    monkeypatch.setattr(_lib, "_lib", None)
    monkeypatch.setattr(_lib, "LIB_PATH", tmp_path / "libttsp_hip.so")
    packed_t, state_t = quant.quantize_4bit(w, 64, compress_statistics=nested)
    assert torch.equal(packed, packed_t)
    _same(state.absmax, state_t.absmax)
    _same(state.offset, state_t.offset)


@pytest.mark.gpu
def test_quantize_reads_a_lazily_negated_weight_as_its_values():
    w = torch.randn(64, 128, generator=torch.Generator(device="cuda").manual_seed(5), device="cuda")
    lazy = torch._neg_view(w)
    assert lazy.is_neg() and lazy.data_ptr() == w.data_ptr()
    packed, state = quant.quantize_4bit(lazy)
    packed_n, state_n = quant.quantize_4bit((-w).contiguous())
    assert torch.equal(packed, packed_n)
    _same(state.absmax, state_n.absmax)


@pytest.mark.gpu
def test_quantize_steps_are_seen_by_modes_and_tangents():
    """Under a dispatch mode every step goes through it, and a forward-mode
    tangent reaches the scales: the torch steps run, with the same bytes."""
    from torch.autograd import forward_ad
    from torch.utils._python_dispatch import TorchDispatchMode

    class Names(TorchDispatchMode):
        seen: list = []

        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            self.seen.append(str(func))
            return func(*args, **(kwargs or {}))

    w = torch.randn(64, 128, generator=torch.Generator(device="cuda").manual_seed(7), device="cuda")
    packed, state = quant.quantize_4bit(w)
    with Names() as names:
        packed_m, state_m = quant.quantize_4bit(w)
    assert any("bucketize" in s for s in names.seen)
    assert torch.equal(packed, packed_m) and torch.equal(state.absmax, state_m.absmax)
    with forward_ad.dual_level():
        packed_d, state_d = quant.quantize_4bit(forward_ad.make_dual(w, torch.ones_like(w)))
        absmax, tangent = forward_ad.unpack_dual(state_d.absmax)
        assert torch.equal(packed, packed_d) and torch.equal(state.absmax, absmax)
        assert torch.equal(tangent, w.view(-1, 64).gather(1, w.view(-1, 64).abs().argmax(1, keepdim=True))[:, 0].sign())
