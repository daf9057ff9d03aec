"""The prompt-attention kernel against causal softmax in fp64: request lengths around the 32-row
wave, the 64-key and the 128-row tile, empty requests, rows that start past zero, every head
grouping, both output types, and a batch whose tile list takes more than one launch."""
import math
from types import SimpleNamespace as NS

import pytest
import torch

from open_ommx_serve_amd.attention import _hip
from open_ommx_serve_amd.integration.vllm import backend
from open_ommx_serve_amd.integration.vllm.backend import causal_prefill_attention

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _rows(n, H, D, seed):
    return torch.randn(n, H, D, generator=torch.Generator(device=DEV).manual_seed(seed), device=DEV).to(torch.bfloat16)


def _reference(q, k, v, starts, scale):
    out = torch.full(q.shape, float("nan"), dtype=torch.float64, device=DEV)
    rep = q.shape[1] // k.shape[1]
    for a, b in zip(starts, starts[1:]):
        Q, K, V = (t[a:b].double().transpose(0, 1).contiguous() for t in (q, k, v))
        K, V = K.repeat_interleave(rep, 0), V.repeat_interleave(rep, 0)
        s = Q @ K.transpose(1, 2).contiguous() * scale
        s = s.masked_fill(torch.ones(b - a, b - a, dtype=torch.bool, device=DEV).triu(1), -float("inf"))
        out[a:b] = (s.softmax(-1) @ V).transpose(0, 1)
    return out


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("hq,hkv", [(4, 4), (8, 2), (8, 1), (6, 2)])
@pytest.mark.parametrize("starts", [
    [0, 1], [0, 31, 63, 64], [0, 32, 97], [2, 65, 65, 129], [0, 127, 255], [0, 128, 257], [0, 700], [5, 6, 390]])
def test_prompt_attention_matches_causal_softmax(D, hq, hkv, starts):
    n = starts[-1] + 3
    q, k, v = _rows(n, hq, D, 1), _rows(n, hkv, D, 2), _rows(n, hkv, D, 3)
    k[:, :, :3] *= 12
    want = _reference(q, k, v, starts, D ** -0.5)
    out = torch.full((n, hq, D), 7.0, device=DEV)
    assert _hip.host().prefill(q, k, v, out, starts, D ** -0.5)
    live = slice(starts[0], starts[-1])
    assert (out[live].double() - want[live]).abs().max().item() <= 1e-5
    assert bool((out[:starts[0]] == 7).all()) and bool((out[starts[-1]:] == 7).all())     # other rows untouched
    half = torch.empty(n, hq, D, dtype=torch.bfloat16, device=DEV)
    assert _hip.host().prefill(q, k, v, half, starts, D ** -0.5)
    assert torch.equal(half[live], out[live].to(torch.bfloat16))


def test_more_tiles_than_one_launch_lists():
    starts = [*range(0, 330 * 3 + 1, 3)]                       # 330 requests of three rows
    q, k, v = _rows(starts[-1], 2, 64, 4), _rows(starts[-1], 1, 64, 5), _rows(starts[-1], 1, 64, 6)
    got = causal_prefill_attention(q, k, v, starts, 0.125, 2)
    assert (got.double() - _reference(q, k, v, starts, 0.125)).abs().max().item() <= 1e-5


@pytest.mark.parametrize("dtype,D", [(torch.float32, 128), (torch.bfloat16, 96)])
def test_rows_the_kernel_does_not_take_still_run(dtype, D):
    q, k, v = (_rows(70, h, D, h).to(dtype) for h in (4, 2, 2))
    out = torch.empty(70, 4, D, device=DEV)
    assert not _hip.host().prefill(q, k, v, out, [0, 70], D ** -0.5)
    got = causal_prefill_attention(q, k, v, [0, 70], D ** -0.5, 2)
    assert (got.double() - _reference(q, k, v, [0, 70], D ** -0.5)).abs().max().item() <= 2e-5


@pytest.mark.parametrize("D,hq,hkv,starts", [
    (128, 64, 8, [0, 1025]), (128, 96, 32, [3, 1412]), (64, 64, 16, [0, 1024, 1090, 2300]), (128, 64, 64, [0, 1087])])
def test_long_prompts_in_two_wave_groups(D, hq, hkv, starts):
    """Enough long tiles for the two-group kernel: groups on two q heads and (odd or single q heads) on two row blocks."""
    n = starts[-1] + 3
    q, k, v = _rows(n, hq, D, 1), _rows(n, hkv, D, 2), _rows(n, hkv, D, 3)
    k[:, :, :3] *= 12
    out = torch.full((n, hq, D), 7.0, device=DEV)
    assert _hip.host().prefill(q, k, v, out, starts, D ** -0.5)
    live = slice(starts[0], starts[-1])
    for h in range(0, hq, hq // hkv):
        heads = slice(h, h + hq // hkv)
        kv = slice(h // (hq // hkv), h // (hq // hkv) + 1)
        want = _reference(q[:, heads], k[:, kv], v[:, kv], starts, D ** -0.5)
        assert (out[live, heads].double() - want[live]).abs().max().item() <= 1e-5
    assert bool((out[:starts[0]] == 7).all()) and bool((out[starts[-1]:] == 7).all())


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("hq,hkv,lens", [(32, 8, [1100] + [100] * 7), (16, 4, [1500, 300, 1, 300, 128]), (8, 1, [33, 4000, 100])])
def test_a_long_prompt_beside_short_ones(D, hq, hkv, lens):
    """More workgroups than compute units, the long prompt's first, keys split between two wave groups in all of them."""
    starts = [2]
    for n in lens:
        starts.append(starts[-1] + n)
    n = starts[-1] + 3
    assert _hip.host().prefill_form(starts, hq, D) == 1 and sum(-(-x // 128) for x in lens) * hq > 256
    q, k, v = _rows(n, hq, D, 1), _rows(n, hkv, D, 2), _rows(n, hkv, D, 3)
    k[:, :, :3] *= 12
    out = torch.full((n, hq, D), 7.0, device=DEV)
    assert _hip.host().prefill(q, k, v, out, starts, D ** -0.5)
    live = slice(starts[0], starts[-1])
    for h in range(0, hq, hq // hkv):
        heads, kv = slice(h, h + hq // hkv), slice(h // (hq // hkv), h // (hq // hkv) + 1)
        want = _reference(q[:, heads], k[:, kv], v[:, kv], starts, D ** -0.5)
        assert (out[live, heads].double() - want[live]).abs().max().item() <= 1e-5
    assert bool((out[:starts[0]] == 7).all()) and bool((out[starts[-1]:] == 7).all())


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("starts", [[0, 257], [0, 321], [3, 387, 388, 700], [0, 1, 64, 449]])
@pytest.mark.parametrize("case", ["plain", "no f16", "weightless", "infinite"])
def test_keys_split_between_two_wave_groups(D, starts, case):
    """Few workgroups with tiles of five and more: odd and even numbers of 64-key tiles, requests of one among them, and in
    the second group's tiles V that is no f16, keys without weight (a row may have no other there), V that is no number."""
    n, hq, hkv = starts[-1] + 3, 8, 2
    q, k, v = _rows(n, hq, D, 1), _rows(n, hkv, D, 2), _rows(n, hkv, D, 3)
    k[:, :, :3] *= 12
    for a, b in zip(starts, starts[1:]):
        if case == "no f16":
            v[a + 64:b:2, :, 5] = 1e4
        elif case == "weightless":
            q[a:b, :, 7], k[a:b, :, 7] = 1e20, 0.0
            for t in range(a + 64, b, 128):
                k[t:min(t + 64, b), :, 7] = -1e20              # scores of -1e40, -inf in fp32
        elif case == "infinite" and b - a > 70:
            v[a + 70, :, 9] = float("inf")
    out = torch.full((n, hq, D), 7.0, device=DEV)
    assert _hip.host().prefill(q, k, v, out, starts, D ** -0.5)
    if case == "infinite":
        for a, b in zip(starts, starts[1:]):
            if b - a > 70:
                assert bool((out[a + 70:b, :, 9] == float("inf")).all())
                v[a + 70, :, 9] = out[a + 70:b, :, 9] = 0.0
    live = slice(starts[0], starts[-1])
    want = _reference(q, k, v, starts, D ** -0.5)
    if case == "infinite":
        for a, b in zip(starts, starts[1:]):
            if b - a > 70:
                want[a + 70:b, :, 9] = 0.0
    # fp32 sums of up to n weights, relative to the largest value of the channel
    bound = 1e-5 * max(1.0, v[live].abs().max().item() / 8)
    assert (out[live].double() - want[live]).abs().max().item() <= bound
    assert bool((out[:starts[0]] == 7).all()) and bool((out[starts[-1]:] == 7).all())


@pytest.mark.parametrize("hq,hkv,n", [(4, 2, 201), (64, 8, 1025)])       # one wave group, two
@pytest.mark.parametrize("case", ["tiny", "huge", "some", "edges"])
def test_values_that_are_no_f16(case, hq, hkv, n):
    """V elements outside 2^-22..256 take their tile through the three-piece path."""
    D = 128
    q, k, v = _rows(n, hq, D, 1), _rows(n, hkv, D, 2), _rows(n, hkv, D, 3)
    if case == "tiny":
        v *= 2.0 ** -40
    elif case == "huge":
        v *= 2.0 ** 20
    elif case == "some":
        v[70, :, 5], v[n - 1, :, 127], v[64, 0, 0] = 1e4, 2.0 ** -30, 0.0
    else:       # the last values on either side of both ends
        top = torch.tensor([0x4380, 0x437F, 0x3480, 0x347F, 0x0001, -0x7F00 - 0x80 + 0x4380], dtype=torch.int16, device=DEV)
        v[5, :, :6] = top.view(torch.bfloat16)
        v[130, :, 6:10] = top[1:3].repeat(2).view(torch.bfloat16)          # a tile with exact ends only
    out = torch.empty(n, hq, D, device=DEV)
    assert _hip.host().prefill(q, k, v, out, [0, n], D ** -0.5)
    rep = hq // hkv
    for h in range(0, hq, rep):
        want = _reference(q[:, h:h + rep], k[:, h // rep:h // rep + 1], v[:, h // rep:h // rep + 1], [0, n], D ** -0.5)
        # fp32 sums of up to n weights, relative to the largest value of the channel
        bound = 2e-6 * v[:, h // rep].double().abs().amax(0)
        assert bool(((out[:, h:h + rep].double() - want).abs() <= bound + 1e-44).all())


def test_an_infinite_value_stays_with_its_tile():
    n, D = 1025, 128
    q, k, v = _rows(n, 64, D, 1), _rows(n, 8, D, 2), _rows(n, 8, D, 3)
    clean = torch.empty(n, 64, D, device=DEV)
    assert _hip.host().prefill(q, k, v, clean, [0, n], D ** -0.5)
    v[400, :, 9] = float("inf")
    out = torch.empty(n, 64, D, device=DEV)
    assert _hip.host().prefill(q, k, v, out, [0, n], D ** -0.5)
    assert torch.equal(out[:384], clean[:384])                             # rows before the 64-key tile of row 400
    assert not bool(torch.isfinite(out[400:, :, 9]).any())
    other = torch.arange(D, device=DEV) != 9
    assert (out[:, :, other] - clean[:, :, other]).abs().max().item() <= 1e-5


@pytest.mark.parametrize("D,hq,hkv,n", [(128, 4, 2, 100), (64, 4, 4, 700), (128, 64, 8, 1025), (64, 96, 32, 1412)])
@pytest.mark.parametrize("gap", [12, 16, 20, 24])
@pytest.mark.parametrize("sink_v", [0.0, 2.0 ** -12])
def test_rows_made_of_small_weights(D, hq, hkv, n, gap, sink_v):
    """A key with next to no V that outweighs every other 2^gap times: the output is the small weights' share."""
    q, k, v = _rows(n, hq, D, 1), _rows(n, hkv, D, 2), _rows(n, hkv, D, 3)
    scale = D ** -0.5
    q[:, :, 0], k[:, :, 0], k[0] = 8.0, 0.0, 0.0
    k[0, :, 0] = gap * math.log(2.0) / (8.0 * scale)
    v[0] *= sink_v
    v[n // 2, :, 3] = 1e-9 if gap == 20 else 0.5                # with and without a tile of its own path
    out = torch.empty(n, hq, D, device=DEV)
    assert _hip.host().prefill(q, k, v, out, [0, n], scale)
    rep = hq // hkv
    for h in range(0, hq, rep):
        want = _reference(q[:, h:h + rep], k[:, h // rep:h // rep + 1], v[:, h // rep:h // rep + 1], [0, n], scale)[1:]
        err = (out[1:, h:h + rep].double() - want).norm(dim=-1) / want.norm(dim=-1)
        # Scores of up to 2^5 are rounded to 2^-20 twice (the sum, exp2's argument), which moves a weight by
        # ln 2 of that; 2^-21 is left of the split; fp32 sums of up to 1412 terms add less than 2^-20.
        assert err.max().item() <= 2.0 ** -18, (h, err.max().item())


@pytest.mark.parametrize("D,hq,hkv,starts", [(64, 4, 2, [0, 201]), (128, 4, 4, [3, 90, 300]), (128, 64, 8, [0, 1025])])
def test_values_that_are_no_numbers_reach_the_rows_from_theirs_on(D, hq, hkv, starts):
    n, inf = starts[-1], float("inf")
    q, k, v = _rows(n, hq, D, 1), _rows(n, hkv, D, 2), _rows(n, hkv, D, 3)
    clean = torch.zeros(n, hq, D, device=DEV)
    assert _hip.host().prefill(q, k, v, clean, starts, D ** -0.5)
    want = clean.clone()
    t0 = starts[-2]
    v[t0 + 70, :, 9], v[t0 + 75, :, 9] = inf, inf
    v[t0 + 64, :, D - 1], v[t0 + 130, :, D - 1] = -inf, inf
    v[t0, 0, 0] = float("nan")
    v[t0 + 127, :, 33], v[t0 + 128, :, 33] = float("nan"), -inf
    want[t0 + 70:, :, 9] = inf
    want[t0 + 64:t0 + 130, :, D - 1] = -inf
    want[t0 + 130:, :, D - 1] = float("nan")
    want[t0:, :hq // hkv, 0] = float("nan")
    want[t0 + 127:, :, 33] = float("nan")
    for dtype in (torch.float32, torch.bfloat16):
        out = torch.zeros(n, hq, D, dtype=dtype, device=DEV)
        assert _hip.host().prefill(q, k, v, out, starts, D ** -0.5)
        # (tiles with such a value take the path of three bf16 pieces: fp32 sums in another order)
        torch.testing.assert_close(out.float(), want.to(dtype).float(), rtol=2.0 ** -7 if dtype == torch.bfloat16 else 0,
                                   atol=1e-5, equal_nan=True)


@pytest.mark.parametrize("where", ["q", "k", "v", "fused", "shifted q"])
def test_an_output_in_the_memory_of_the_inputs(where):
    n, H, D = 700, 4, 64
    fused = _rows(n, 4 * H, D, 1)
    q, k, v = fused[:, :H], fused[:, H:2 * H], fused[:, 2 * H:3 * H]
    q, k, v = (t if where == "fused" else t.contiguous() for t in (q, k, v))
    if where == "shifted q":
        q = torch.cat([q, q[:1]])[:n]
        out = q.as_strided((n - 1, H, D), q.stride(), H * D)
        q, k, v = q[:n - 1], k[:n - 1], v[:n - 1]
    else:
        out = fused[:, 3 * H:] if where == "fused" else {"q": q, "k": k, "v": v}[where]
    n = out.shape[0]
    want = torch.empty(n, H, D, dtype=torch.bfloat16, device=DEV)
    assert _hip.host().prefill(q, k, v, want, [0, n], 0.125)
    impl = backend.OMMXCanonicalImpl(H, D, 0.125, H)
    backend.reset_worker_state(graph=False, batched=False, batched_graph=False)
    backend.OMMXCanonicalMetadataBuilder().build(0, NS(seq_lens_cpu=[n], query_start_loc_cpu=[0, n],
                                                       block_table_tensor=torch.tensor([[3, 4]])))
    impl.forward(NS(), q, k, v, None, None, out)
    backend.reset_worker_state()
    assert torch.equal(out, want)
