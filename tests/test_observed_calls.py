"""Calls that somebody else takes part in (a tracer, a transform, a mode, autograd) keep to torch's dispatcher, where
those work; the launchers that go past it are for the others."""
import pytest
import torch
import torch.autograd.forward_ad as fwd
from torch._subclasses.fake_tensor import FakeTensorMode
from torch.fx.experimental.proxy_tensor import make_fx
from torch.overrides import TorchFunctionMode

from open_ommx_serve_amd.attention import MultiSeqKVPool, _hip
from open_ommx_serve_amd.attention import reference_op as R
from open_ommx_serve_amd.integration.vllm.backend import causal_prefill_attention
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


def _case(**kw):
    case = build_decode_case([300, 150], seed=5)
    planes = dict(case.planes) | {"outliers_per_vector": case.outliers_per_vector, "page_size": case.page_size,
                                  "k_format": "i2f4", "outlier_repr": "bitmap", "kv_outlier_map": True,
                                  "kv_int8_scale": True}

    def decode(q):
        return R.ommx_paged_decode(q, planes, case.k_tail, case.v_tail, case.b_tail_len, case.b_seq_len,
                                   sm_scale=case.sm_scale, req_to_token=case.req_to_token,
                                   req_to_group=case.req_to_group, max_seq_len=300,
                                   max_tail_len=int(case.k_tail.shape[1]), **kw)[0]
    return case.q, decode


@pytest.mark.gpu
def test_a_traced_decode_holds_the_op():
    q, decode = _case()
    traced = torch.jit.trace(decode, (q,), check_trace=False)
    assert "ommx_gpu_serve::paged_decode" in str(traced.graph)
    other = q.flip(0).contiguous()
    assert torch.equal(traced(other), decode(other)) and not torch.equal(decode(other), decode(q))


def _prompt(n=70, D=64):
    g = torch.Generator(device="cuda").manual_seed(3)
    return [torch.randn(n, h, D, generator=g, device="cuda").to(torch.bfloat16) for h in (4, 2, 2)]


@pytest.mark.gpu
@pytest.mark.parametrize("which", ["q", "k", "v", "qkv"])
def test_prompt_attention_has_its_gradient(which):
    rows = _prompt()
    w = torch.randn(70, 4, 64, generator=torch.Generator(device="cuda").manual_seed(8), device="cuda")
    leaves = [t.clone().requires_grad_("qkv"[i] in which) for i, t in enumerate(rows)]
    out = causal_prefill_attention(*leaves, [0, 30, 70], 0.125, 2)
    (out * w).sum().backward()
    own = [t.clone().requires_grad_() for t in rows]
    for a, b in ((0, 30), (30, 70)):
        q, k, v = (t[a:b].transpose(0, 1).repeat_interleave(4 // t.shape[1], 0).unsqueeze(0).float() for t in own)
        o = torch.nn.functional.scaled_dot_product_attention(q, k, v, is_causal=True, scale=0.125)
        (o[0].transpose(0, 1) * w[a:b]).sum().backward()
    for leaf, want in zip(leaves, own):
        if not leaf.requires_grad:
            assert leaf.grad is None
            continue
        # The same library calls: their order of summation may differ, which moves a bf16 gradient, and each of
        # the two heads' that it sums, by one unit (2^-8 of a value no larger than twice the largest here).
        assert (leaf.grad.float() - want.grad.float()).abs().max() <= 3 * 2.0 ** -7 * want.grad.float().abs().max()
    with torch.no_grad():
        assert _hip.host().prefill(*leaves, torch.empty_like(w), [0, 30, 70], 0.125)


@pytest.mark.gpu
def test_prompt_attention_under_a_tracer_and_fake_tensors():
    q, k, v = _prompt()
    traced = torch.jit.trace(lambda q: causal_prefill_attention(q, k, v, [0, 70], 0.125, 2), (q,), check_trace=False)
    other = q.flip(0).contiguous()
    want = causal_prefill_attention(other, k, v, [0, 70], 0.125, 2)
    assert (traced(other) - want).abs().max() <= 1e-5
    with FakeTensorMode() as mode:
        out = causal_prefill_attention(*(mode.from_tensor(t) for t in (q, k, v)), [0, 70], 0.125, 2)
    assert out.shape == q.shape and out.dtype == torch.float32


@pytest.mark.gpu
def test_a_pool_decode_leaves_observed_calls_to_the_op():
    win_rows = 200
    pool = MultiSeqKVPool(128, 2, 1, win_rows, outliers_per_vector=6, outlier_repr="bitmap", use_pow2=True)
    g = torch.Generator(device="cuda").manual_seed(4)
    K, V, q = (torch.randn(n, h, 128, generator=g, device="cuda").to(torch.bfloat16)
               for n, h in ((150, 2), (150, 2), (1, 8)))
    pool.append_block(0, K, V)
    rows, seq = torch.tensor([0], device="cuda"), torch.tensor([150], device="cuda")
    packed = torch.tensor([pool.window.packed_len(150)], dtype=torch.int32, device="cuda")
    tables = (pool.pool_planes()["req_to_token"], pool.pool_planes()["req_to_group"])
    out = torch.empty(1, 8, 128, device="cuda")

    def decode(q, out):
        return pool.decode_into(q, out, rows, seq, packed, tables, sm_scale=0.09, max_seq_len=150)

    assert decode(q, out)
    kept = out.clone()
    out.fill_(5.0)
    assert not decode(q.clone().requires_grad_(), out) and not decode(q, torch.empty_like(out).requires_grad_())
    assert bool((out == 5.0).all())
    with torch.no_grad():
        assert decode(q.clone().requires_grad_(), out)
    assert torch.equal(out, kept)


@pytest.mark.gpu
def test_a_tensor_written_by_a_launch_is_a_new_version():
    """Autograd refuses a backward pass whose saved tensor has been overwritten since."""
    def overwritten(shape, write):
        t, x = torch.ones(shape, device="cuda"), torch.ones(shape, device="cuda", requires_grad=True)
        loss = (x * t).sum()
        with torch.no_grad():
            write(t)
        with pytest.raises(RuntimeError, match="modified by an inplace operation"):
            loss.backward()
        with torch.inference_mode():
            write(torch.ones(shape, device="cuda"))

    q, _ = _case()
    overwritten(q.shape, lambda t: _case(out=t)[1](q))
    overwritten(q.shape[:2], lambda t: _case(lse_out=t)[1](q))
    rows = _prompt()
    overwritten(rows[0].shape, lambda t: _hip.host().prefill(*rows, t, [0, 70], 0.125))
