"""Short decode calls, served by four waves on one kv head of one split (csrc/ommx_decode_team.hip), with their merge inside the
launch or as one of its own: edges of groups, steps, shares and states, against the oracle; the same call again, from a graph and
beside others on its own bits."""
import pytest
import torch

import oracle.ommx_oracle as O
from open_ommx_serve_amd.attention import _hip
from open_ommx_serve_amd.attention.paged_decode import ommx_paged_decode_attention_canonical
from open_ommx_serve_amd.synth import build_decode_case

pytestmark = pytest.mark.gpu


def _outputs(case):
    B, Hq, D = case.q.shape
    return (torch.full((B, Hq, D), float("nan"), dtype=torch.float32, device=case.q.device),
            torch.full((B, Hq), float("nan"), dtype=torch.float32, device=case.q.device))


def _run(case, **over):
    o, lse = _outputs(case)
    ommx_paged_decode_attention_canonical(*case.decode_args(o, lse), **{**case.decode_kwargs(), **over})
    return o.cpu(), lse.cpu()


def _oracle(case):
    planes = {k: (v.cpu() if torch.is_tensor(v) else v) for k, v in case.planes.items()}
    return O.decode_reference(case.q.cpu(), planes | {"outliers_per_vector": case.outliers_per_vector},
                              case.k_tail.cpu(), case.v_tail.cpu(), case.b_tail_len.tolist(), case.req_to_token.cpu(),
                              case.req_to_group.cpu(), case.b_seq_len.tolist(), sm_scale=case.sm_scale,
                              page_size=case.page_size)


def _close(got, want, what):
    # the bounds of every decode test: f16 rounding of weights and outlier entries, fp32 sums
    (o, lse), (wo, wl) = got, want
    assert torch.isfinite(o).all(), what
    err = (o.double() - wo.double()).abs()
    assert err.max().item() <= 2e-3 and err.mean().item() <= 2e-4, (what, err.max().item())
    fin = torch.isfinite(wl)
    assert torch.equal(torch.isfinite(lse), fin), what
    assert not fin.any() or (lse.double()[fin] - wl.double()[fin]).abs().max().item() <= 2e-3, what


SHAPES = [(32, 8, 128, {}), (64, 8, 128, {}), (8, 1, 128, dict(outlier_repr="relidx7")), (16, 8, 128, dict(outlier_repr="relidx7")),
          (4, 4, 128, {}), (32, 8, 64, {}), (4, 2, 64, {}), (32, 8, 128, dict(kv_outlier_map=False)),
          (64, 8, 128, dict(kv_outlier_map=False, outlier_repr="relidx7")), (8, 8, 64, dict(kv_outlier_map=False))]


@pytest.mark.parametrize("hq,hkv,D,kw", SHAPES)
@pytest.mark.parametrize("lens", [[7], [72], [104], [105], [136], [167], [2072], [4136], [9, 72, 100], [72, 9, 136, 700, 40],
                                  [40 + 33 * i for i in range(17)], [72] * 63 + [1]], ids=lambda l: f"{len(l)}x{max(l)}")
def test_edges_of_groups_and_shares(hq, hkv, D, kw, lens):
    """No packed token, one group, a step of one and of two groups, 32 steps and more; requests without any beside others."""
    case = build_decode_case(lens, q_heads=hq, kv_heads=hkv, head_dim=D, seed=len(lens) + max(lens), permute_tables=True,
                             sparse_frac=0.005, **kw)
    want = _oracle(case)
    _close(_run(case), want, "as told")
    _close(_run(case, max_seq_len=int(case.b_seq_len.max()) + 1000), want, "longer than it is")
    # a hint that says too little: splits take more groups each
    _close(_run(case, max_seq_len=64), want, "shorter than it is")


@pytest.mark.parametrize("hq,hkv,D,kw", SHAPES)
@pytest.mark.parametrize("lens", [[7], [104], [167], [4136], [9, 72, 100], [72, 9, 136, 700, 40]], ids=lambda l: f"{len(l)}x{max(l)}")
def test_without_a_tail(hq, hkv, D, kw, lens):
    """Packed tokens alone, as a range of groups is attended: nobody attends a tail, and a request may hold nothing at all."""
    case = build_decode_case(lens, q_heads=hq, kv_heads=hkv, head_dim=D, seed=len(lens) + max(lens), permute_tables=True,
                             sparse_frac=0.005, **kw)
    case.b_tail_len.zero_()
    want = _oracle(case)
    _close(_run(case, max_tail_len=0), want, "as told")
    _close(_run(case, max_tail_len=0, max_seq_len=int(case.b_seq_len.max()) + 1000), want, "longer than it is")
    outs = _outputs(case)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        ommx_paged_decode_attention_canonical(*case.decode_args(*outs), **{**case.decode_kwargs(), "max_tail_len": 0})
    for _ in range(2):
        for t in outs:
            t.fill_(float("nan"))
        graph.replay()
        _close([t.cpu() for t in outs], want, "captured")


def test_tables_are_not_read_past_their_rows():
    """The hint says more groups than the tables have entries: what lies behind a row is another request's, or nobody's."""
    case = build_decode_case([700, 135], seed=3, permute_tables=True)
    err = torch.zeros(1, dtype=torch.int32, device=case.q.device)
    _close(_run(case, max_seq_len=3000, err_flag=err), _oracle(case), "")
    one = build_decode_case([700], seed=3, permute_tables=True)
    _close(_run(one, max_seq_len=2000, err_flag=err), _oracle(one), "")
    assert int(err.item()) == 0


@pytest.mark.parametrize("hq,hkv,D", [(32, 8, 128), (64, 8, 128), (32, 8, 64)])
def test_the_same_bits_again_in_memory_of_other_calls(hq, hkv, D):
    """Calls of several shapes one behind another, in scratch that calls before or other tensors had; bits stay."""
    cases = [build_decode_case(l, q_heads=hq, kv_heads=hkv, head_dim=D, seed=5, permute_tables=True, sparse_frac=0.005)
             for l in ([1000], [300, 90, 500], [72], [9], [100 + 40 * i for i in range(8)])]
    first = [_run(c) for c in cases]
    for c, f in zip(cases, first):
        _close(f, _oracle(c), "")
    for turn in range(30):
        junk = torch.full((1 << 20,), [0, -1, 0x7F][turn % 3], dtype=torch.int8, device="cuda")
        del junk
        for i in ((turn * 7 + k) % len(cases) for k in range(len(cases))):
            o, lse = _run(cases[i])
            assert torch.equal(o, first[i][0]) and torch.equal(lse, first[i][1]), (turn, i)


@pytest.mark.parametrize("lens,mib", [([1000], 1), ([300, 90, 500], 1), ([97 + 86 * i for i in range(8)], 4)])
def test_the_merge_counts_over_whatever_its_scratch_holds(lens, mib):
    """A pool of its own holds one free block, so a call's scratch is cut from its front: filled beforehand with zeros, ones, words
    above the call's number, which have to come down to it, and words of an earlier call.  Read back, the counts lie there, a word on
    a line of 64 bytes for each request and kv head, all under one number, the lines' other words as they were filled."""
    case = build_decode_case(lens, q_heads=32, kv_heads=8, head_dim=128, seed=5, permute_tables=True, sparse_frac=0.005)
    want = _run(case)
    pool, number = torch.cuda.MemPool(), 0
    for left in ("zeros", "ones", "just above", "far above", "an earlier call's"):
        fill = {"zeros": 0, "ones": 2 ** 64 - 1, "just above": (number + 2) << 8 | 3, "far above": (number + 2 ** 20) << 8 | 17,
                "an earlier call's": number << 8 | 255}[left]
        o, lse = _outputs(case)
        with torch.cuda.use_mem_pool(pool):
            block = torch.empty(mib << 17, dtype=torch.int64, device="cuda")
            at = block.data_ptr()
            block.fill_(fill - 2 ** 64 if fill >= 2 ** 63 else fill)
            del block
            ommx_paged_decode_attention_canonical(*case.decode_args(o, lse), **case.decode_kwargs())
            block = torch.empty(mib << 17, dtype=torch.int64, device="cuda")
        assert block.data_ptr() == at, left
        lines = block.cpu().numpy().view("uint64").reshape(-1, 8)
        first = lines[:, 0]
        # (a call's number has 0xFF and zeros on top: no state or lse looks like it)
        found = first[(lines[:, 1:] == fill).all(1) & (first != fill) & (first >> 48 >= 0xFF00) & (first >> 48 < 0xFF80)]
        assert len(found) == len(lens) * 8 and len(set(found.tolist())) <= len(lens), left
        numbers = set((found >> 8).tolist())
        assert len(numbers) == 1 and min(numbers) > number, left
        number = int(min(numbers))
        assert torch.equal(o.cpu(), want[0]) and torch.equal(lse.cpu(), want[1]), left
        del block


OPTIONS = [(32, 8, 128, {}), (64, 8, 128, dict(outlier_repr="relidx7")), (32, 8, 64, {}), (64, 8, 128, dict(kv_outlier_map=False))]


@pytest.mark.parametrize("hq,hkv,D,kw", OPTIONS)
@pytest.mark.parametrize("lens", [[1000], [900, 40, 330]], ids=lambda l: f"{len(l)}x{max(l)}")
def test_caps_large_queries_and_large_steps(hq, hkv, D, kw, lens):
    """Options that take a branch of their own: a cap, query elements of several hundred in some waves' channels (the bounds of the same
    test of the one-wave kernel), steps beyond the f16 operands, held and reported."""
    def case_of(**over):
        return build_decode_case(lens, q_heads=hq, kv_heads=hkv, head_dim=D, seed=31, permute_tables=True,
                                 **{"sparse_frac": 0.005, **kw, **over})
    case = case_of()
    err = torch.zeros(1, dtype=torch.int32, device="cuda")
    plain = _run(case, logit_cap=4.0, _force_reference_kernel=True)
    assert not torch.allclose(plain[0], _run(case, _force_reference_kernel=True)[0], atol=1e-2)
    _close(_run(case, logit_cap=4.0, err_flag=err), (plain[0], plain[1]), "cap")
    q = case.q.float().cpu()
    where = torch.randperm(q.numel(), generator=torch.Generator().manual_seed(7))[:20]
    q.view(-1)[where] = torch.tensor([300.0, -512.0, 1000.0, -776.0, 256.0] * 4)
    case.q.copy_(q.to(case.q.dtype))
    want = _oracle(case)
    (o, lse), (wo, wl) = _run(case, err_flag=err), want
    d = (o.double() - wo).abs()
    assert d.max().item() <= 2e-3 and d.mean().item() <= 2e-4, d.max().item()
    assert ((lse.double() - wl).abs() <= 2e-3 + 1e-5 * wl.abs()).all()
    assert int(err.item()) == 0
    case = case_of(sparse_frac=0.02, sparse_gain=40.0, outlier_gain=150.0)
    exps = case.planes["k_scale"].to(torch.int32)
    assert int((exps >= 6).sum()) > 50 and int(exps.max()) <= 15
    (o, lse), (wo, wl) = _run(case, err_flag=err), _oracle(case)
    d = (o.double() - wo).abs()
    assert d.max().item() <= 2e-3 and d.mean().item() <= 2e-4, d.max().item()
    assert ((lse.double() - wl).abs() <= 2e-3 + 2e-6 * wl.abs()).all()
    assert int(err.item()) == 0
    for name in ("k_scale", "v_scale"):
        case = case_of()
        case.planes[name].view(-1)[5::97] = 17
        err.zero_()
        o, _ = _run(case, err_flag=err)
        assert torch.isfinite(o).all() and int(err.item()) & _hip.ERR_VALUE_RANGE, name


def test_captured_calls_replay_like_eager_ones():
    """Under capture the merge is a launch of its own: the same states in another order of sums (fp32 rounding)."""
    cases = [build_decode_case(l, seed=6, permute_tables=True, sparse_frac=0.005) for l in ([1000], [300, 90, 500])]
    eager = [_run(c) for c in cases]
    outs = [_outputs(c) for c in cases]
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        for c, (o, lse) in zip(cases, outs):
            ommx_paged_decode_attention_canonical(*c.decode_args(o, lse), **c.decode_kwargs())
    for turn in range(4):
        for o, lse in outs:
            o.fill_(float("nan"))
            lse.fill_(float("nan"))
        graph.replay()
        again = [_run(c) for c in cases]                     # eager work between the replays
        for (o, lse), (wo, wl), a in zip(outs, eager, again):
            assert (o.cpu() - wo).abs().max().item() <= 2e-6 * max(1.0, wo.abs().max().item()), turn
            assert (lse.cpu() - wl).abs().max().item() <= 1e-5
            assert torch.equal(a[0], wo)


@pytest.mark.parametrize("where", ["o in q", "lse in q", "o in the tail rows", "o in a plane", "o around q"])
@pytest.mark.parametrize("lens,hq,hkv,D", [([1000], 32, 8, 128), ([300, 90, 500], 64, 8, 128), ([700, 330], 8, 4, 64)])
def test_results_that_lie_in_what_the_call_reads(where, lens, hq, hkv, D):
    """The merge is a launch of its own then, behind everything that reads: on the bits of one under capture, which the merge
    inside the launch (sums in another order) does not have."""
    case = build_decode_case(lens, q_heads=hq, kv_heads=hkv, head_dim=D, seed=10, permute_tables=True, sparse_frac=0.005)
    apart, outs = _run(case), _outputs(case)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        ommx_paged_decode_attention_canonical(*case.decode_args(*outs), **case.decode_kwargs())
    graph.replay()
    want = [t.cpu() for t in outs]
    assert not torch.equal(apart[0], want[0])
    B = len(lens)
    o, lse = _outputs(case)
    floats = torch.zeros(4 * B * hq * D, device="cuda")
    if where == "o around q":                            # rows of one buffer, each head's q behind its result
        rows = floats[:B * hq * 2 * D].view(B, hq, 2, D)
        o, q = rows[:, :, 0], rows[:, :, 1].view(torch.bfloat16)[..., :D]
        case.q = q.copy_(case.q)
    elif where in ("o in q", "lse in q"):
        q = floats[:B * hq * D].view(torch.bfloat16)[:B * hq * D].view(B, hq, D)
        if where == "o in q":
            o = floats[:B * hq * D].view(B, hq, D)
        else:
            lse = floats[:B * hq].view(B, hq)
        case.q = q.copy_(case.q)
    else:
        name = "k_tail" if where == "o in the tail rows" else "k_base"
        source = case.k_tail if name == "k_tail" else case.planes[name]
        assert source.nbytes >= o.nbytes
        held = source.clone()
        o = held.view(-1).view(torch.float32)[:o.numel()].view(B, hq, D)
        if name == "k_tail":
            case.k_tail = held
        else:
            case.planes[name] = held
    ommx_paged_decode_attention_canonical(*case.decode_args(o, lse), **case.decode_kwargs())
    assert torch.equal(o.cpu(), want[0]) and torch.equal(lse.cpu(), want[1])


def test_two_streams_at_once():
    """Calls under way together have scratch of their own."""
    cases = [build_decode_case(l, seed=8, permute_tables=True) for l in ([1000], [400, 90, 600])]
    want = [_run(c) for c in cases]
    streams = [torch.cuda.Stream() for _ in cases]
    outs = [[_outputs(c) for _ in range(25)] for c in cases]
    torch.cuda.synchronize()
    for i in range(25):
        for c, s, os in zip(cases, streams, outs):
            with torch.cuda.stream(s):
                ommx_paged_decode_attention_canonical(*c.decode_args(*os[i]), **c.decode_kwargs())
    torch.cuda.synchronize()
    for os, (wo, wl) in zip(outs, want):
        for o, lse in os:
            assert torch.equal(o.cpu(), wo) and torch.equal(lse.cpu(), wl)


def test_an_id_outside_its_plane_is_reported():
    case = build_decode_case([700], seed=9, permute_tables=True)
    err = torch.zeros(1, dtype=torch.int32, device=case.q.device)
    case.req_to_group[0, 5] = 1 << 20
    _run(case, err_flag=err)
    torch.cuda.synchronize()
    assert int(err.item()) == _hip.ERR_TABLE_RANGE
