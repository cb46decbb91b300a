"""csrc/host.cpp: what it leaves to the Python checks, and calls that it must not take."""
import pytest
import torch


def _host():
    from t2fw_amd import _lib
    return _lib.host()


def _ins(B=2, T=3, D=4, K=5, device="cpu", dtype=torch.float32):
    t = lambda *s: torch.ones(s, device=device, dtype=dtype)
    return [t(B, T, D), t(B, T, D), t(B, T, K), t(B, T, K), t(B, T, K), t(B, D, K)]


def test_host_memory_and_other_objects_are_left_to_the_python_checks():
    assert _host().lfw_shape(*_ins(), False) is None
    assert _host().lfw_shape(*_ins()[:5], None, False) is None
    assert _host().lfw_step(*(t[:, 0] for t in _ins()[:5]), _ins()[5], None, True, 0) is None


def test_calls_with_other_arguments_raise():
    with pytest.raises(RuntimeError):
        _host().lfw_shape(*_ins())
    with pytest.raises(RuntimeError):
        _host().block_copy(b"", (), (), 0, 0)
    with pytest.raises(RuntimeError):
        _host().block_copy(bytes(7), (torch.ones(64),), (torch.ones(64),), 0, 0)
    with pytest.raises(RuntimeError):
        _host().gate_forward(None, None, None, None, 0, 0)
    with pytest.raises(TypeError):
        _host().gate_forward(torch.ones(1), torch.ones(1), None, None, "0", 0)


@pytest.mark.gpu
@pytest.mark.parametrize("heads", [False, True])
def test_shapes_that_fit_and_those_that_do_not(heads):
    ins = _ins(device="cuda")
    if heads:
        ins = [t.unsqueeze(2) for t in ins[:5]] + [ins[5].unsqueeze(1)]
    shape = lambda *a: _host().lfw_shape(*a, heads)
    assert shape(*ins) == (2, 3, 1, 4, 5)
    for i in range(6):
        for other in (ins[i].half(), ins[i].cpu(), ins[i][:1], ins[i].unsqueeze(0), ins[i].transpose(0, 1), torch.cat([ins[i]] * 2, -1)[..., ::2]):
            assert shape(*ins[:i], other, *ins[i + 1:]) is None, i


@pytest.mark.gpu
def test_step_returns_the_callers_tensors():
    from t2fw_amd.functional_lfw import lfw_step
    x, f, q, k, fk, s = [t[:, 0].contiguous() if t.dim() == 3 and i < 5 else t for i, t in enumerate(_ins(device="cuda"))]
    out = torch.empty_like(x)
    got, state = lfw_step(x, f, q, k, fk, s, out=out)
    assert got is out and state is s
    got, state = lfw_step(x, f, q, k, fk, s, inplace=False)
    assert state is not s and torch.equal(s, torch.full_like(s, 2.0)) and torch.equal(state, torch.full_like(s, 3.0))
    for bad in (dict(x=x[:1]), dict(f=f.half()), dict(state=s[:, :3])):
        with pytest.raises((AssertionError, RuntimeError)):
            lfw_step(**{**dict(x=x, f=f, query=q, key=k, f_key=fk, state=s), **bad})


class _Marked(torch.Tensor):
    """a tensor subclass with torch's own behaviour"""


@pytest.mark.gpu
def test_results_keep_the_tensor_subclass_of_their_inputs():
    from t2fw_amd import LFWFunction
    from t2fw_amd.functional_dfw import DFWFunction
    from t2fw_amd.functional_lfw import lfw_step, sigmoid_gates
    ins = _ins(device="cuda")
    marked = lambda ts: [t.as_subclass(_Marked) for t in ts]
    assert [type(t) for t in LFWFunction.apply(*ins)] == [torch.Tensor] * 2
    assert [type(t) for t in LFWFunction.apply(*marked(ins))] == [_Marked] * 2
    assert [type(t) for t in sigmoid_gates(*marked(ins[1:3]))] == [_Marked] * 2
    assert [type(t) for t in lfw_step(*marked([t[:, 0].contiguous() for t in ins[:5]] + ins[5:]))] == [_Marked] * 2
    for D in (64, 128):
        q, v, s = torch.ones(2, 3, 64, device="cuda"), torch.ones(2, 3, D, device="cuda"), torch.ones(2, D, 64, device="cuda")
        assert [type(t) for t in DFWFunction.apply(*marked([q, q, v, s]))] == [_Marked] * 2
    param = [torch.nn.Parameter(t) for t in ins]
    assert [type(t) for t in LFWFunction.apply(*param)] == [torch.Tensor] * 2


class _Learned(torch.nn.Parameter):
    """of torch's operations on it a plain tensor comes, as of any parameter"""


class _Noted(torch.Tensor):
    """a tensor subclass that hands something on through torch.empty_like"""

    @classmethod
    def __torch_function__(cls, func, types, args=(), kwargs=None):
        res = super().__torch_function__(func, types, args, kwargs or {})
        if func is torch.empty_like:
            res.note = args[0].note
        return res


@pytest.mark.gpu
def test_subclasses_through_torch_empty_like():
    """What a call returns in the place of its own tensors is theirs, what it allocates is what torch.empty_like gives."""
    from t2fw_amd import LFWFunction
    from t2fw_amd.functional_dfw import DFWFunction
    from t2fw_amd.functional_lfw import lfw_step, sigmoid_gates
    ins = _ins(device="cuda")
    step = [t[:, 0].contiguous().as_subclass(_Marked) for t in ins[:5]] + [ins[5].clone().as_subclass(_Marked)]
    out, f, fk = torch.empty_like(step[0]), torch.empty_like(step[1]), torch.empty_like(step[4])
    got, state = lfw_step(*step, out=out)
    assert got is out and state is step[5]
    got = sigmoid_gates(step[1], step[4], out_f=f, out_fk=fk)
    assert got[0] is f and got[1] is fk
    learned = [_Learned(t) for t in ins]
    assert [type(t) for t in LFWFunction.apply(*learned)] == [torch.Tensor] * 2
    assert [type(t) for t in lfw_step(*[_Learned(t.as_subclass(torch.Tensor)) for t in step], inplace=False)] == [torch.Tensor] * 2
    noted = [t.as_subclass(_Noted) for t in ins]
    for i, t in enumerate(noted):
        t.note = i
    assert [t.note for t in LFWFunction.apply(*noted)] == [0, 5]
    for D in (64, 128):
        q, v, s = torch.ones(2, 3, 64, device="cuda"), torch.ones(2, 3, D, device="cuda"), torch.ones(2, D, 64, device="cuda")
        noted = [t.as_subclass(_Noted) for t in (q, q.clone(), v, s)]
        for i, t in enumerate(noted):
            t.note = i
        assert [t.note for t in DFWFunction.apply(*noted)] == [2, 3]


def _traced_calls():
    from t2fw_amd import LFWFunction, LFWHeadsFunction
    from t2fw_amd.functional_dfw import DFWFunction
    from t2fw_amd.functional_lfw import LFWGatedFunction, lfw_step, sigmoid_gates
    ones = lambda *s, dtype=torch.float32: torch.ones(s, device="cuda", dtype=dtype)
    delta = lambda D: [ones(2, 3, 64), ones(2, 3, 64), ones(2, 3, D), ones(2, D, 64)]
    lfw = _ins(device="cuda")
    return {
        "LFWFunction": (LFWFunction.apply, lfw),
        "LFWFunction, matrix cores": (LFWFunction.apply, _ins(2, 70, 64, 64, "cuda", torch.float16)),
        "LFWFunction, blocks": (LFWFunction.apply, _ins(2, 3, 128, 64, "cuda", torch.float16)),
        "LFWGatedFunction": (LFWGatedFunction.apply, lfw),
        "LFWHeadsFunction": (LFWHeadsFunction.apply, [t.unsqueeze(2) for t in lfw[:5]] + [lfw[5].unsqueeze(1)]),
        "lfw_step": (lfw_step, [t[:, 0].contiguous() for t in lfw[:5]] + [lfw[5]]),
        "sigmoid_gates": (sigmoid_gates, [lfw[1], lfw[4]]),
        "DFWFunction": (DFWFunction.apply, delta(64)),
        "DFWFunction, blocks": (DFWFunction.apply, delta(128)),
        "DFWFunction, per step": (DFWFunction.apply, delta(5)),
    }


@pytest.mark.gpu
@pytest.mark.parametrize("loaded", [False, True])
@pytest.mark.parametrize("grad", [False, True])
@pytest.mark.parametrize("name", ["LFWFunction", "LFWFunction, matrix cores", "LFWFunction, blocks", "LFWGatedFunction", "LFWHeadsFunction",
                                  "lfw_step", "sigmoid_gates", "DFWFunction", "DFWFunction, blocks", "DFWFunction, per step"])
def test_calls_are_not_traced(name, grad, loaded, monkeypatch):
    """What torch.compile makes of a call that runs by itself, before and after the library is loaded: an error of its tracing,
    as these calls can't be traced (no stream is known there, and the host module and ctypes are closed to it).  The host
    module isn't reached while a call is traced."""
    from t2fw_amd import _lib
    call, ins = _traced_calls()[name]
    fn = lambda *a: call(*a)
    if grad and name not in ("lfw_step", "sigmoid_gates"):
        ins[0].requires_grad_()
    for t in fn(*ins):
        assert t.is_cuda
    torch.cuda.synchronize()
    monkeypatch.setattr(_lib, "loaded", lambda: loaded)
    torch._dynamo.reset()
    try:
        with pytest.raises(torch._dynamo.exc.Unsupported, match="Dynamo does not know how to trace"):
            torch.compile(fn, backend="eager", fullgraph=True)(*ins)
        torch._dynamo.reset()
        with pytest.raises(AttributeError, match="'torch.Stream' object has no attribute 'cuda_stream'"):
            torch.compile(fn, backend="eager")(*ins)
    finally:
        torch._dynamo.reset()
