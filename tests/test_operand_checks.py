"""What the modules hand to the library as raw pointers is checked before the library is entered.  Runs without a GPU: CPU
tensors that say they are on one, and a library that records its calls."""
import pytest
import torch
import torch.autograd.forward_ad as forward_ad

from sla_amd import SageSparseLinearAttention, SparseLinearAttention, _lib, module


class _OnGpu(torch.Tensor):
    """A CPU tensor that says it is on the GPU (the stub library never reads it)."""

    is_cuda = property(lambda self: True)


class _Library:
    def __init__(self):
        self.calls = []

    def __getattr__(self, name):
        if name == "sla_workspace_bytes":
            return lambda *a: 4096

        def entry(*args):
            self.calls.append(name)
            return 0
        return entry


@pytest.fixture
def library(monkeypatch):
    lib = _Library()
    monkeypatch.setattr(_lib, "load", lambda: lib)
    monkeypatch.setattr(_lib, "stream_ptr", lambda dev: 0)
    _lib.workspace_bytes.cache_clear()
    module._plan.cache_clear()
    yield lib
    _lib.workspace_bytes.cache_clear()
    module._plan.cache_clear()


def _operands(*shape, dtype=torch.bfloat16):
    return [torch.zeros(shape, dtype=dtype).as_subclass(_OnGpu) for _ in range(3)]


def _on_gpu(mod):
    for name in ("weight", "bias"):
        p = getattr(mod.proj_l, name)
        del mod.proj_l._parameters[name]
        setattr(mod.proj_l, name, p.detach().as_subclass(_OnGpu))
    return mod


def _modules():
    return [SparseLinearAttention(64, 0.5), SparseLinearAttention(64, 0.5, linear_mode="complement"),
            SageSparseLinearAttention(64, 0.5)]


@pytest.mark.parametrize("which", [0, 2])
def test_accepted_operands_reach_the_library(library, which):
    mod = _on_gpu(_modules()[which])
    with torch.no_grad():
        mod(*_operands(1, 2, 128, 64))
        if which == 0:
            mod.forward_packed(torch.zeros(1, 128, 3, 2, 64, dtype=torch.bfloat16).as_subclass(_OnGpu))
    assert library.calls


@pytest.mark.parametrize("grad", [False, True])
@pytest.mark.parametrize("which", range(3))
@pytest.mark.parametrize("left", ["weight", "bias"])
def test_a_projection_left_on_the_cpu_is_refused(library, which, grad, left):
    mod = _on_gpu(_modules()[which])
    setattr(mod.proj_l, left, torch.zeros(64, 64) if left == "weight" else torch.zeros(64))
    ops = _operands(1, 2, 128, 64)
    if grad:
        ops = [t.requires_grad_(True) for t in ops]
    with torch.set_grad_enabled(grad), pytest.raises(RuntimeError, match="on the GPU only"):
        mod(*ops)
    if which == 0:
        packed = torch.zeros(1, 128, 3, 2, 64, dtype=torch.bfloat16).as_subclass(_OnGpu).requires_grad_(grad)
        with torch.set_grad_enabled(grad), pytest.raises(RuntimeError, match="on the GPU only"):
            mod.forward_packed(packed)
    assert not library.calls


@pytest.mark.parametrize("grad", [False, True])
def test_packed_activations_on_the_cpu_are_refused(library, grad):
    mod = _on_gpu(SparseLinearAttention(64, 0.5))
    with torch.set_grad_enabled(grad), pytest.raises(RuntimeError, match="on the GPU only"):
        mod.forward_packed(torch.zeros(1, 128, 3, 2, 64, dtype=torch.bfloat16).requires_grad_(grad))
    assert not library.calls


@pytest.mark.parametrize("grad", [False, True])
@pytest.mark.parametrize("which", range(3))
@pytest.mark.parametrize("operand,shape", [(1, (1, 1, 128, 64)), (1, (1, 2, 64, 64)), (2, (1, 1, 128, 64)), (2, (1, 2, 64, 64)),
                                           (1, (1, 2, 256, 64)), (2, (1, 2, 128, 128))])
def test_operands_of_different_shapes_are_refused(library, which, grad, operand, shape):
    """Fewer key heads, shorter or longer keys or values: every size is taken from q, so k and v would be read past their end."""
    mod = _on_gpu(_modules()[which])
    ops = _operands(1, 2, 128, 64)
    ops[operand] = torch.zeros(shape, dtype=torch.bfloat16).as_subclass(_OnGpu)
    if grad:
        ops = [t.requires_grad_(True) for t in ops]
    with torch.set_grad_enabled(grad), pytest.raises(AssertionError, match="same shape"):
        mod(*ops)
    assert not library.calls


@pytest.mark.parametrize("which", range(3))
@pytest.mark.parametrize("weight,bias", [(torch.zeros(64, 64, dtype=torch.bfloat16), torch.zeros(64)),
                                         (torch.zeros(64, 64), torch.zeros(64, dtype=torch.float16)),
                                         (torch.zeros(128, 128), torch.zeros(128)), (torch.zeros(64, 64), torch.zeros(32))])
def test_a_projection_of_another_type_or_size_is_refused(library, which, weight, bias):
    """The kernels read D x D and D values of 32 bits."""
    mod = _on_gpu(_modules()[which])
    mod.proj_l.weight, mod.proj_l.bias = weight.as_subclass(_OnGpu), bias.as_subclass(_OnGpu)
    with torch.no_grad(), pytest.raises(ValueError, match="proj_l"):
        mod(*_operands(1, 2, 128, 64))
    if which == 0:
        with torch.no_grad(), pytest.raises(ValueError, match="proj_l"):
            mod.forward_packed(torch.zeros(1, 128, 3, 2, 64, dtype=torch.bfloat16).as_subclass(_OnGpu))
    assert not library.calls


@pytest.mark.parametrize("grad", [False, True])
@pytest.mark.parametrize("shape", [(1, 128, 4, 2, 64), (1, 128, 2, 2, 64)])
def test_a_packed_tensor_has_three_parts(library, grad, shape):
    """Inference, which does not enter the autograd function, refuses what training refuses."""
    mod = _on_gpu(SparseLinearAttention(shape[-1], 0.5))
    packed = torch.zeros(shape, dtype=torch.bfloat16).as_subclass(_OnGpu).requires_grad_(grad)
    with torch.set_grad_enabled(grad), pytest.raises(AssertionError, match="packed"):
        mod.forward_packed(packed)
    assert not library.calls


@pytest.mark.parametrize("no_grad", [False, True])
@pytest.mark.parametrize("packed", [False, True])
def test_forward_mode_tangents_are_refused(library, monkeypatch, packed, no_grad):
    """There is no jvp: dual inputs raise as with any such autograd function, also where nothing asks for a gradient, instead
    of giving an output without its tangent."""
    monkeypatch.setattr(_lib, "require_gpu", lambda *t: None)
    mod = SparseLinearAttention(64, 0.5).requires_grad_(False)
    shape = (1, 128, 3, 2, 64) if packed else (1, 2, 128, 64)
    x, y, dx = (torch.randn(shape).bfloat16() for _ in range(3))
    with torch.set_grad_enabled(not no_grad), forward_ad.dual_level():
        dual = forward_ad.make_dual(x, dx)
        with pytest.raises(NotImplementedError, match="jvp"):
            mod.forward_packed(dual) if packed else mod(dual, y, y)
        out = mod.forward_packed(x) if packed else mod(x, y, y)       # (no tangent: nothing to lose)
    assert out.shape == ((1, 128, 2, 64) if packed else shape)


@pytest.mark.parametrize("packed", [False, True])
def test_a_trace_records_the_operator(library, monkeypatch, packed):
    """A traced inference call runs the library again; recorded below the operator it would be its uninitialised buffers."""
    monkeypatch.setattr(_lib, "require_gpu", lambda *t: None)
    mod = SparseLinearAttention(64, 0.5).requires_grad_(False)
    x = torch.randn((1, 128, 3, 2, 64) if packed else (1, 2, 128, 64)).bfloat16()
    traced = torch.jit.trace(lambda x: mod.forward_packed(x) if packed else mod(x, x, x), (x,), check_trace=False)
    library.calls.clear()
    traced(x)
    assert library.calls == ["sla_module_fwd"]
