"""The store kernel of the signed power-of-two recipes beside the serving one, bit for bit against
the oracle: every vector length it is built for, heads narrower and wider than the tuned one, both
outlier counts and maps, blocks of heavy ties (the outlier sets of the two ends then overlap), constant
vectors, permuted destinations, and what it reports."""
import numpy as np
import pytest
import torch

import oracle.ommx_oracle as O
from conftest import bits_of
from open_ommx_serve_amd.attention import _hip, ommx_pack_kv_canonical_block
from open_ommx_serve_amd.attention.pack import alloc_planes, store_pack_into
from open_ommx_serve_amd.synth import synth_kv

pytestmark = pytest.mark.gpu
ZERO_SIGN_FREE = ("k_zp", "v_zp", "k_fp4_mapcenter")


def _names(recipe):
    names = ["k_base", "k_scale", "k_zp", "k_oval", "v_main", "v_scale", "v_zp",
             "k_obmp" if recipe["outlier_repr"] == "bitmap" else "k_oidx"]
    return names + (["k_fp4_mapscale", "k_fp4_mapcenter"] if recipe.get("kv_outlier_map", True) else [])


def _same(got, want, names):
    for n in names:
        a, b = got[n], want[n]
        if n in ZERO_SIGN_FREE:                       # (a zero's sign is open where zeros of both signs tie)
            a, b = a.float().cpu() + 0.0, b.float().cpu() + 0.0
        assert np.array_equal(bits_of(a), bits_of(b)), n


@pytest.mark.parametrize("gt,gc,D,k,repr_,own_map", [
    (32, 32, 64, 6, "bitmap", True), (32, 32, 128, 6, "relidx7", False), (32, 32, 32, 10, "relidx7", True),
    (64, 64, 128, 6, "relidx7", False), (64, 32, 64, 10, "bitmap", True), (64, 64, 256, 6, "bitmap", True),
    (128, 128, 128, 10, "relidx7", True), (128, 64, 64, 6, "bitmap", False), (128, 128, 256, 10, "bitmap", False),
    (128, 32, 96, 10, "relidx7", True)])
def test_long_group_store_is_bit_exact(gt, gc, D, k, repr_, own_map):
    T, H = 4 * gt, 3
    K, V = synth_kv(T, H, D, seed=gt + D + k, sparse_frac=0.01)
    g = torch.Generator().manual_seed(gt)
    few = torch.tensor([-3.0, -1.0, 1.0, 0.0, -0.0, 0.5, -0.5, 2.0])
    K[:gt] = few[torch.randint(0, len(few), (gt, H, D), generator=g)].to(torch.bfloat16)      # heavy ties
    K[gt:2 * gt, 0] = 1.5                                                                     # constant vectors
    K[gt:2 * gt, 1] = few[torch.randint(2, 5, (gt, D), generator=g)].to(torch.bfloat16)       # hardly two values
    V[:gt, :, :gc] = -2.25
    recipe = dict(outliers_per_vector=k, outlier_repr=repr_, outlier_select="signed", use_pow2=True,
                  kv_outlier_map=own_map, group_tokens=gt, group_channels=gc)
    want = O.pack_kv(K, V, **recipe)
    _same(ommx_pack_kv_canonical_block(K.cuda(), V.cuda(), **recipe), want, _names(recipe))

    # the same block through a source permutation into permuted slots
    rows = torch.randperm(T, generator=g)
    pages, groups = torch.randperm(T // 16, generator=g), torch.randperm(T // gt, generator=g)
    planes = alloc_planes(T // 16, T // gt, H, D, outliers_per_vector=k, outlier_repr=repr_, kv_outlier_map=own_map,
                          group_tokens=gt, group_channels=gc, device="cuda")
    shuffled_k, shuffled_v = torch.empty_like(K), torch.empty_like(V)
    shuffled_k[rows], shuffled_v[rows] = K, V
    store_pack_into(shuffled_k.cuda(), shuffled_v.cuda(), planes, src_rows=rows.int().cuda(),
                    dst_pages=pages.int().cuda(), dst_groups=groups.int().cuda(), outliers_per_vector=k,
                    outlier_repr=repr_, group_tokens=gt, group_channels=gc)
    _same({n: planes[n][(pages if n in ("k_base", "v_main", "v_scale", "v_zp") else groups).cuda()]
           for n in _names(recipe)}, want, _names(recipe))


@pytest.mark.parametrize("gt,k", [(32, 10), (64, 6), (128, 10)])
@pytest.mark.parametrize("where,error", [("K", ValueError), ("V", ValueError)])
def test_long_group_store_reports_values_that_are_not_finite(gt, k, where, error):
    K, V = synth_kv(2 * gt, 2, 128, seed=5)
    (K if where == "K" else V)[gt + 3, 1, 77] = float("inf")
    with pytest.raises(error):
        ommx_pack_kv_canonical_block(K.cuda(), V.cuda(), outliers_per_vector=k, outlier_repr="relidx7",
                                     outlier_select="signed", use_pow2=True, group_tokens=gt)


@pytest.mark.parametrize("gt,gc,D,k", [(32, 32, 64, 6), (32, 128, 128, 6), (64, 64, 192, 10), (64, 128, 256, 6), (64, 32, 32, 6),
                                       (128, 32, 96, 10), (128, 128, 128, 6)])
@pytest.mark.parametrize("shift", [0, 1])
def test_v_vectors_of_any_alignment_and_range(gt, gc, D, k, shift):
    """V vectors shared by several lanes: rows that are not 16-byte aligned, zero points so far from their step that the
    code takes the two-step way, and denormal vectors, beside ordinary ones in the same wave."""
    T, H = 2 * gt, 2
    K, V = synth_kv(T, H, D, seed=gt + gc + D, sparse_frac=0.01)
    V[1::5, 0, :gc] = 3e38                               # 2^-e * zero point overflows
    V[2::7, 1, D - gc:] = torch.linspace(0, 6e-39, gc).to(torch.bfloat16)
    V[3, :, :gc] = torch.tensor([-0.0, 0.0, 2e-38, -2e-38]).repeat(gc // 4).to(torch.bfloat16)
    recipe = dict(outliers_per_vector=k, outlier_repr="relidx7", outlier_select="signed", use_pow2=True,
                  group_tokens=gt, group_channels=gc)
    want = O.pack_kv(K, V, **recipe)
    wide_k, wide_v = (torch.zeros(T, H, D + 2 * shift, dtype=torch.bfloat16, device="cuda") for _ in range(2))
    k_in, v_in = wide_k[:, :, shift:shift + D], wide_v[:, :, shift:shift + D]
    k_in.copy_(K)
    v_in.copy_(V)
    _same(ommx_pack_kv_canonical_block(k_in, v_in, **recipe), want, _names(recipe))


@pytest.mark.parametrize("gt,gc,D,k", [(32, 32, 64, 6), (64, 64, 128, 6), (64, 32, 96, 10), (128, 128, 128, 10), (128, 64, 64, 6)])
@pytest.mark.parametrize("ps", [1, 2, 32])
def test_tokens_of_a_pair_on_pages_of_any_size(gt, gc, D, k, ps):
    """Codes of two tokens are written together: pages of one token, of one pair and of a whole 32-token group in a shuffled
    order, K rows that cannot be read 16 bytes at a time (a view one element into its storage)."""
    T, H = 3 * gt, 2
    K, V = synth_kv(T, H, D, seed=gt + D + k + ps, sparse_frac=0.01)
    recipe = dict(outliers_per_vector=k, outlier_repr="relidx7", kv_outlier_map=True, group_tokens=gt, group_channels=gc)
    want = O.pack_kv(K, V, outlier_select="signed", use_pow2=True, **recipe)
    pages = torch.randperm(T // ps, generator=torch.Generator().manual_seed(ps))
    shifted = torch.empty(T * H * D + 1, dtype=torch.bfloat16, device="cuda")
    shifted[1:] = K.cuda().flatten()
    for rows in (K.cuda(), shifted[1:].view(T, H, D)):
        planes = alloc_planes(T // ps, T // gt, H, D, device="cuda", page_size=ps, **recipe)
        store_pack_into(rows, V.cuda(), planes, page_size=ps, dst_pages=pages.int().cuda(), outliers_per_vector=k,
                        outlier_repr="relidx7", group_tokens=gt, group_channels=gc)
        for n in ("k_base", "v_main", "v_scale", "v_zp"):
            got = planes[n].cpu()[pages].reshape(T, H, -1)
            assert np.array_equal(bits_of(got), bits_of(want[n].reshape(T, H, -1))), n
        for n in ("k_scale", "k_zp", "k_oval", "k_oidx", "k_fp4_mapscale", "k_fp4_mapcenter"):
            assert np.array_equal(bits_of(planes[n].cpu()), bits_of(want[n])), n


@pytest.mark.parametrize("gt,gc,D,k,rep", [(32, 32, 64, 6, "bitmap"), (64, 64, 128, 6, "bitmap"), (64, 32, 96, 10, "bitmap"),
                                           (32, 32, 64, 6, "relidx7"), (64, 64, 128, 6, "relidx7"), (128, 128, 128, 10, "relidx7")])
def test_positions_taken_from_both_ends_keep_codes_and_positions_together(gt, gc, D, k, rep):
    """A channel of 3e9 but for k/2 - 1 tokens: the lanes of the largest count as 1e9 for the smallest, so one of them is taken
    twice and a slot is left over, which is reported.  Codes stay beside the positions they belong to."""
    half, low = k // 2, [7, 19, 20, 31][:k // 2 - 1]
    K, V = synth_kv(gt, 2, D, seed=5)
    K[:, 1, 3] = 3e9
    K[low, 1, 3] = -3e9
    planes = alloc_planes(gt // 16, 1, 2, D, device="cuda", outliers_per_vector=k, outlier_repr=rep, group_tokens=gt, group_channels=gc)
    err = torch.zeros(1, dtype=torch.int32, device="cuda")
    store_pack_into(K.cuda(), V.cuda(), planes, err_flag=err, outliers_per_vector=k, outlier_repr=rep, group_tokens=gt, group_channels=gc)
    assert int(err.item()) & _hip.ERR_UNDERFILLED
    index = planes["k_obmp" if rep == "bitmap" else "k_oidx"][0, 1, 3].tolist()
    bits = sum(b << (8 * i) for i, b in enumerate(index))
    want = [*range(half), *low]
    if rep == "bitmap":
        assert [i for i in range(gt) if bits >> i & 1] == want
    else:
        assert [bits >> (7 * s) & 127 for s in range(k)] == [*want, want[-1]]
    codes = [planes["k_oval"][0, 1, 3, s // 2].item() >> (4 * (s & 1)) & 15 for s in range(k)]
    assert len(set(codes[1:half])) == 1 and len(set(codes[half:k - 1])) == 1 and codes[1] != codes[half]
