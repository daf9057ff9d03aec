"""Batches whose packed groups are dealt out in equal shares (no split count asked for): the edges of the
search -- as many requests as a lane or a wave of lanes holds, one request that takes nearly all of the groups,
requests with none, a length hint below the real length -- for every kernel that takes shares, against the oracle."""
import pytest
import torch

import oracle.ommx_oracle as O
from open_ommx_serve_amd.attention import MultiSeqKVPool, WindowSpec
from open_ommx_serve_amd.attention.paged_decode import ommx_paged_decode_attention_canonical
from open_ommx_serve_amd.synth import build_decode_case

pytestmark = pytest.mark.gpu
LEVER = dict(group_tokens=64, group_channels=64, outliers_per_vector=10, outlier_repr="relidx7")
LEVER6 = dict(LEVER, outliers_per_vector=6, kv_outlier_map=False)
PAPER10 = dict(group_tokens=128, group_channels=128, outliers_per_vector=10, outlier_repr="relidx7")
PAPER = dict(group_tokens=128, group_channels=128, outlier_repr="relidx7")


def _run(case, **over):
    B, Hq, D = case.q.shape
    o = torch.full((B, Hq, D), float("nan"), dtype=torch.float32, device=case.q.device)
    lse = torch.full((B, Hq), float("nan"), dtype=torch.float32, device=case.q.device)
    ommx_paged_decode_attention_canonical(*case.decode_args(o, lse), **{**case.decode_kwargs(), **over})
    return o.cpu(), lse.cpu()


def _close(got, want, what):
    (o, lse), (wo, wl) = got, want
    assert torch.isfinite(o).all(), what
    err = (o.double() - wo.double()).abs()
    assert err.max().item() <= 2e-3 and err.mean().item() <= 2e-4, (what, err.max().item())
    fin = torch.isfinite(wl)
    assert torch.equal(torch.isfinite(lse), fin), what
    assert (lse.double()[fin] - wl.double()[fin]).abs().max().item() <= 2e-3, what


def _oracle(case):
    planes = {k: (v.cpu() if torch.is_tensor(v) else v) for k, v in case.planes.items()}
    return O.decode_reference(case.q.cpu(), planes | {"outliers_per_vector": case.outliers_per_vector},
                              case.k_tail.cpu(), case.v_tail.cpu(), case.b_tail_len.tolist(), case.req_to_token.cpu(),
                              case.req_to_group.cpu(), case.b_seq_len.tolist(), sm_scale=case.sm_scale,
                              page_size=case.page_size)


@pytest.mark.parametrize("hq,hkv,D,kw,lens", [
    (32, 8, 128, {}, [3300, 3300]),                                       # pairs, two requests
    (32, 8, 128, {}, [9, 7000]),                                          # one request without groups
    (32, 8, 128, {}, [200 + 7 * i for i in range(63)]),
    (32, 8, 128, {}, [900] + [72] * 62 + [9]),                            # B = 64: one lane each
    (32, 8, 128, {}, [72] * 40 + [1500] + [9] * 24),                      # B = 65: four requests a lane
    (32, 8, 128, {}, [104] * 255 + [700]),                                # as many requests as shares
    (32, 8, 128, {}, [136] * 257),                                        # more than a wave can search
    (64, 8, 128, {}, [40, 2500, 777, 3000, 72]),
    (64, 8, 128, dict(outlier_repr="relidx7"), [150 + i for i in range(66)]),
    (8, 1, 128, {}, [17000, 33000, 100]),                                 # more than 256 states of one request
    (4, 4, 128, {}, [5000, 4000]),
    (32, 8, 64, {}, [72, 9000, 5000]),                                    # head_dim 64: pairs of kv heads
    (16, 4, 64, {}, [300 + i for i in range(65)]),
    (32, 8, 128, LEVER, [5000, 9, 9000]),                                 # ten outliers of 64 tokens: the plain kernel
    (32, 8, 128, PAPER, [400 + 5 * i for i in range(66)]),                # more requests than longer groups are dealt out for
    (32, 8, 128, LEVER6, [5000, 9, 9000]),                                # pieces of longer groups
    (64, 8, 128, LEVER6, [300 + 37 * i for i in range(64)]),
    (8, 1, 128, PAPER10, [9000, 131, 20000]),
    (32, 8, 128, PAPER10, [2100 + 67 * i for i in range(20)]),
    (64, 8, 128, dict(PAPER10, group_channels=64), [6000, 9, 170, 4000]),
])
def test_shares_against_the_oracle(hq, hkv, D, kw, lens):
    case = build_decode_case(lens, q_heads=hq, kv_heads=hkv, head_dim=D, seed=77, permute_tables=True,
                             sparse_frac=0.005, **kw)
    want = _oracle(case)
    longest = max(case.b_seq_len.tolist())
    got = _run(case, max_seq_len=longest)
    _close(got, want, "shares")
    _close(_run(case, num_kv_splits=7), want, "fixed splits")
    _close(_run(case, max_seq_len=2 * longest + 5000), want, "a generous length hint")
    _close(_run(case, max_seq_len=max(1, longest * 2 // 3)), want, "a hint below the longest request")
    again = _run(case, max_seq_len=longest)
    assert torch.equal(got[0], again[0]) and torch.equal(got[1], again[1])


@pytest.mark.parametrize("lens", [[2500 - 31 * i for i in range(3)], [100 + 5 * i for i in range(65)]])
def test_shares_over_a_row_history(lens):
    """The serving pool's call (tails read from the ring, bf16 out) against gathered tails and fixed splits."""
    B, H, D, Hq = len(lens), 8, 128, 32
    pool = MultiSeqKVPool(D, H, B, 2600, window=WindowSpec(), device="cuda", kv_ring=True, outliers_per_vector=6,
                          outlier_repr="bitmap", use_pow2=True)
    g = torch.Generator(device="cuda").manual_seed(5)
    for r, n in enumerate(lens):
        pool.append_block(r, *(torch.randn(n, H, D, generator=g, device="cuda").to(torch.bfloat16) for _ in range(2)))
    q = torch.randn(B, Hq, D, generator=g, device="cuda").to(torch.bfloat16)
    d = pool.decode_inputs_batched(range(B))
    p, want = d["planes"], torch.empty(B, Hq, D, dtype=torch.float32, device="cuda")
    ommx_paged_decode_attention_canonical(
        q, p["k_base"], p["k_scale"], p["k_zp"], None, p["k_oval"], p["v_main"], p["v_scale"], p["v_zp"], d["k_tail"],
        d["v_tail"], d["b_tail_len"], want, torch.empty(B, Hq, device="cuda"), d["req_to_token"], d["req_to_group"],
        d["b_seq_len"], sm_scale=D ** -0.5, page_size=16, k_outliers_per_vector=6, bitmap_read=True, k_obmp=p["k_obmp"],
        k_fp4_mapscale=p["k_fp4_mapscale"], k_fp4_mapcenter=p["k_fp4_mapcenter"], kv_outlier_map=True,
        kv_int8_scale=True, num_kv_splits=3)
    out = torch.zeros(B, Hq, D, dtype=torch.bfloat16, device="cuda")
    assert pool.decode_into(q, out, torch.arange(B, device="cuda"), torch.tensor(lens, device="cuda"), d["b_seq_len"],
                            (d["req_to_token"], d["req_to_group"]), sm_scale=D ** -0.5, max_seq_len=d["max_seq_len"])
    assert (out.float() - want).abs().max().item() <= 2.0 ** -8 * want.abs().max().item() + 1e-4


@pytest.mark.parametrize("hq,hkv,D,kw,recent", [
    (32, 8, 128, {}, 32), (64, 8, 128, {}, 32), (4, 4, 128, {}, 130), (8, 1, 128, dict(outlier_repr="relidx7"), 32),
    (32, 8, 64, {}, 32), (8, 8, 64, {}, 150), (16, 4, 128, dict(group_tokens=128, group_channels=64, outlier_repr="relidx7"), 32),
])
def test_tail_rows_beside_the_splits(hq, hkv, D, kw, recent):
    """The tail in four parts as states of its own: no rows, fewer rows than parts, parts of one and of two blocks of 16
    and one row more, several passes of 32; one request (fixed splits) and many (shares); rows that cannot be read 16
    bytes at a time take the other merge."""
    win = WindowSpec(recent_window=recent, group_tokens=kw.get("group_tokens", 32))
    for seqs in ([2000], [2000, 900, 3000, 700, 2500, 1500]):
        case = build_decode_case(seqs, q_heads=hq, kv_heads=hkv, head_dim=D, seed=91, permute_tables=True,
                                 sparse_frac=0.005, window=win, **kw)
        T = case.k_tail.shape[1]
        for lens in ([0, 1, 3, 15, 16, 17], [31, 32, 33, 63, 64, 65], [T, T - 1, 70, 128, 129, 2]):
            lens = [min(n, T) for n in lens][:len(seqs)]
            case.b_tail_len.copy_(torch.tensor(lens, dtype=torch.int32))
            want = _oracle(case)
            longest = max(case.b_seq_len.tolist())
            _close(_run(case, max_seq_len=longest), want, f"tails {lens}")
            _close(_run(case, max_seq_len=longest, num_kv_splits=400), want, f"tails {lens}, 400 splits")
        odd = torch.empty(case.v_tail.numel() + 1, dtype=case.v_tail.dtype, device=case.v_tail.device)[1:].view_as(case.v_tail)
        odd.copy_(case.v_tail)
        case.v_tail = odd
        _close(_run(case, max_seq_len=longest), want, "V rows at an odd address")
