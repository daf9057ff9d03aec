"""Calls that somebody else takes part in (a tracer, a transform, a mode, autograd) keep to torch's dispatcher, where
those work; the launchers that go past it are for the others."""
import pytest
import torch
import torch.autograd.forward_ad as fwd
from torch._subclasses.fake_tensor import FakeTensorMode
from torch.fx.experimental.proxy_tensor import make_fx
from torch.overrides import TorchFunctionMode

from open_ommx_serve_amd.attention import _hip
from open_ommx_serve_amd.attention import reference_op as R
from open_ommx_serve_amd.synth import build_decode_case


class _Mode(TorchFunctionMode):
    def __torch_function__(self, fn, types, args=(), kwargs=None):
        return fn(*args, **(kwargs or {}))


class _Sub(torch.Tensor):
    pass


def _in_mode(f, t):
    with _Mode():
        f(t)


def _dual(f, t):
    with fwd.dual_level():
        f(fwd.make_dual(t, t))


def _fake(f, t):
    with FakeTensorMode():
        f(torch.zeros(3))


OBSERVERS = {
    "jit.trace": lambda f, t: torch.jit.trace(f, (t,), check_trace=False),
    "make_fx": lambda f, t: make_fx(f)(t),
    "vmap": lambda f, t: torch.vmap(f)(t),
    "grad": lambda f, t: torch.func.grad(lambda x: f(x).sum())(t),
    "jvp": lambda f, t: torch.func.jvp(f, (t,), (t,)),
    "functionalize": lambda f, t: torch.func.functionalize(f)(t),
    "dual": _dual,
    "fake": _fake,
    "function mode": _in_mode,
    "subclass": lambda f, t: f(t.as_subclass(_Sub)),
    "requires grad": lambda f, t: f(t.clone().requires_grad_()),
}


@pytest.mark.parametrize("how", OBSERVERS)
def test_an_observed_call_is_not_plain(how):
    plain, seen, ordinary = _hip.host().plain, [], torch.zeros(3)

    def f(x):
        seen.append((plain(x), plain(None, ordinary, x)))
        return x + 1

    OBSERVERS[how](f, torch.ones(3))
    assert seen == [(False, False)]


def test_an_ordinary_call_is_plain():
    plain, t = _hip.host().plain, torch.zeros(3)
    assert plain() and plain(t) and plain(t, None, t[1:])
    with torch.no_grad():
        assert plain(t.clone().requires_grad_())
    with torch.inference_mode():
        assert plain(torch.zeros(3))
    with torch.autocast("cpu", dtype=torch.bfloat16):
        assert plain(t)


def _case():
    case = build_decode_case([300, 150], seed=5)
    planes = dict(case.planes) | {"outliers_per_vector": case.outliers_per_vector, "page_size": case.page_size,
                                  "k_format": "i2f4", "outlier_repr": "bitmap", "kv_outlier_map": True,
                                  "kv_int8_scale": True}

    def decode(q):
        return R.ommx_paged_decode(q, planes, case.k_tail, case.v_tail, case.b_tail_len, case.b_seq_len,
                                   sm_scale=case.sm_scale, req_to_token=case.req_to_token,
                                   req_to_group=case.req_to_group, max_seq_len=300,
                                   max_tail_len=int(case.k_tail.shape[1]))[0]
    return case.q, decode


@pytest.mark.gpu
def test_a_traced_decode_holds_the_op():
    q, decode = _case()
    traced = torch.jit.trace(decode, (q,), check_trace=False)
    assert "ommx_gpu_serve::paged_decode" in str(traced.graph)
    other = q.flip(0).contiguous()
    assert torch.equal(traced(other), decode(other)) and not torch.equal(decode(other), decode(q))
