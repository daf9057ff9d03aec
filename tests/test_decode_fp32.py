"""Decode of 64-channel heads with position streams (csrc/ommx_decode_fp32.hip): edges of groups, pieces, steps and shares against the
oracle, every form that its rule takes, and streams that no store writes as the plain kernel reads them."""
import pytest
import torch

import oracle.ommx_oracle as O
from open_ommx_serve_amd.attention import _hip
from open_ommx_serve_amd.attention.paged_decode import ommx_paged_decode_attention_canonical
from open_ommx_serve_amd.synth import build_decode_case

pytestmark = pytest.mark.gpu
U = 2.0 ** -24


def _run(case, **over):
    B, Hq, D = case.q.shape
    o = torch.full((B, Hq, D), float("nan"), dtype=torch.float32, device=case.q.device)
    lse = torch.full((B, Hq), float("nan"), dtype=torch.float32, device=case.q.device)
    ommx_paged_decode_attention_canonical(*case.decode_args(o, lse), **{**case.decode_kwargs(), **over})
    return o.cpu(), lse.cpu()


def _host(case):
    planes = {k: (v.cpu() if torch.is_tensor(v) else v) for k, v in case.planes.items()}
    return planes | {"outliers_per_vector": case.outliers_per_vector}


def _oracle(case):
    return O.decode_reference(case.q.cpu(), _host(case), case.k_tail.cpu(), case.v_tail.cpu(), case.b_tail_len.tolist(),
                              case.req_to_token.cpu(), case.req_to_group.cpu(), case.b_seq_len.tolist(), sm_scale=case.sm_scale,
                              page_size=case.page_size)


def _bounds(case):
    """fp32 sums: a logit is off by at most (a chain of 16, three more additions, the scale and what exp and log add: 24) units
    of the sum of its products' sizes, an output by twice that and 64 units for its own sums, times the largest V."""
    planes, q, a, v = _host(case), case.q.cpu().float(), 1.0, 1.0
    for b, n in enumerate(case.b_seq_len.tolist()):
        K, V = O.gather_request(planes, case.req_to_token[b].cpu(), case.req_to_group[b].cpu(), n, page_size=case.page_size)
        t = int(case.b_tail_len[b])
        K = torch.cat([K, case.k_tail[b, :t].cpu().float()]).abs().repeat_interleave(q.shape[1] // case.kv_heads, 1)
        if K.shape[0]:
            a = max(a, float(torch.einsum("thd,hd->th", K, q[b].abs()).max()) * case.sm_scale)
            v = max(v, float(V.abs().max()) if n else 1.0, float(case.v_tail[b].abs().max()))
    return (48 * a + 64) * U * v, 24 * a * U


def _close(got, want, bounds, what=""):
    (o, lse), (wo, wl), (bo, bl) = got, want, bounds
    assert torch.isfinite(o).all(), what
    assert (o.double() - wo.double()).abs().max().item() <= bo, what
    fin = torch.isfinite(wl)
    assert torch.equal(torch.isfinite(lse), fin), what
    assert (lse.double()[fin] - wl.double()[fin]).abs().max().item() <= bl, what


# (tokens a group, channels a V vector, outliers, own map)
RECIPES = [(32, 32, 6, True), (32, 64, 5, False), (64, 64, 6, False), (64, 32, 9, True), (128, 64, 10, True), (128, 32, 7, False),
           (128, 64, 3, True), (32, 32, 1, True)]
LENS = ([7], [72], [73], [168], [169], [200], [232], [1500], [9, 300, 168], [40 + 65 * i for i in range(20)], [72] * 63 + [400],
        [168 + i for i in range(66)])


@pytest.mark.parametrize("gt,gc,k,own_map", RECIPES)
@pytest.mark.parametrize("lens", LENS, ids=lambda l: f"{len(l)}x{max(l)}")
def test_edges_of_groups_steps_and_shares(gt, gc, k, own_map, lens):
    """No packed token, one group, a step and a step more; one request, several in shares, more than a wave's lanes."""
    hq, hkv = ((8, 2), (4, 4), (2, 1), (12, 3))[(len(lens) + gt // 32 + k) % 4]
    case = build_decode_case(lens, q_heads=hq, kv_heads=hkv, head_dim=64, seed=len(lens) + max(lens), permute_tables=True,
                             sparse_frac=0.01, outlier_repr="relidx7", outliers_per_vector=k, kv_outlier_map=own_map, group_tokens=gt,
                             group_channels=gc)
    want, bounds = _oracle(case), _bounds(case)
    _close(_run(case), want, bounds)
    _close(_run(case, num_kv_splits=3), want, bounds, "fixed splits")


@pytest.mark.parametrize("gt,gc,k,own_map", RECIPES)
def test_options_of_a_call(gt, gc, k, own_map):
    """int64 tables, lengths inside a group and a page, a cap, queries and steps of any size; the plain kernel beside."""
    case = build_decode_case([1000, 333, 40], q_heads=8, kv_heads=2, head_dim=64, seed=gt + k, permute_tables=True, sparse_frac=0.01,
                             outlier_repr="relidx7", outliers_per_vector=k, kv_outlier_map=own_map, group_tokens=gt, group_channels=gc,
                             table_dtype=torch.int64)
    case.b_seq_len -= torch.tensor([45, 17, 0], dtype=torch.int32, device="cuda")
    case.b_seq_len.clamp_(min=0)
    bounds = _bounds(case)
    _close(_run(case), _oracle(case), bounds)
    plain = _run(case, logit_cap=5.0, _force_reference_kernel=True)
    _close(_run(case, logit_cap=5.0), plain, bounds, "cap")
    case.q *= 300.0
    _close(_run(case), _oracle(case), _bounds(case), "large queries")
    case.q /= 300.0 * 2.0 ** 30
    case.planes["k_scale"] += 30                        # steps far above what a 16-bit operand holds
    _close(_run(case), _run(case, _force_reference_kernel=True), _bounds(case), "large steps")


@pytest.mark.parametrize("gt,gc,k,own_map", RECIPES)
def test_any_bytes_in_the_index_plane(gt, gc, k, own_map):
    """Positions outside the group, out of order and named twice: as the plain kernel has them, and nothing else is touched."""
    case = build_decode_case([700, 200], q_heads=8, kv_heads=2, head_dim=64, seed=gt + k, permute_tables=True, outlier_repr="relidx7",
                             outliers_per_vector=k, kv_outlier_map=own_map, group_tokens=gt, group_channels=gc)
    gen = torch.Generator(device="cuda").manual_seed(gt + k)
    ix = case.planes["k_oidx"]
    ix.copy_(torch.randint(0, 256, ix.shape, generator=gen, device="cuda", dtype=torch.uint8))
    ix[::3] &= 0x11                                      # many positions twice
    got, want = _run(case), _run(case, _force_reference_kernel=True)
    bo = bl = 0.0
    for b in range(2):                                   # (values as large as the largest outlier)
        top = 64 * 64 * float(case.q.abs().max()) * case.sm_scale
        bo, bl = max(bo, (48 * top + 64) * U * 8), max(bl, 24 * top * U)
    _close(got, want, (bo, bl))


def test_the_same_bits_on_another_stream_and_from_a_graph():
    case = build_decode_case([900, 300], q_heads=8, kv_heads=2, head_dim=64, seed=4, permute_tables=True, outlier_repr="relidx7")
    first = _run(case)
    B, Hq, D = case.q.shape
    o, lse = torch.empty(B, Hq, D, device="cuda"), torch.empty(B, Hq, device="cuda")
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        ommx_paged_decode_attention_canonical(*case.decode_args(o, lse), **case.decode_kwargs())
    for _ in range(3):
        o.fill_(float("nan"))
        graph.replay()
        with torch.cuda.stream(torch.cuda.Stream()):
            again = _run(case)
        torch.cuda.synchronize()
        assert torch.equal(o.cpu(), first[0]) and torch.equal(lse.cpu(), first[1])
        assert torch.equal(again[0], first[0]) and torch.equal(again[1], first[1])


def test_an_id_outside_its_plane_is_reported():
    case = build_decode_case([700], q_heads=8, kv_heads=2, head_dim=64, seed=9, permute_tables=True, outlier_repr="relidx7")
    err = torch.zeros(1, dtype=torch.int32, device="cuda")
    case.req_to_token[0, 5] = 1 << 20
    _run(case, err_flag=err)
    assert int(err.item()) == _hip.ERR_TABLE_RANGE
