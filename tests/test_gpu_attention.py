"""tars_attention (opentars_amd.ops.attention) against the oracle's three ops per head, bit for bit:
fdot_nt of the head's q rows with its K head's rows, the causal softmax, fdot_nn with the V rows
(the reference's lowering, tars_mini/llm.py:736-746), and the last head's scores and
probabilities in the shared rows. The shapes cover the three forms: the split form (up to 4 query
rows per K / V head group: Qwen3 decode with 2 query heads per K / V head, Gemma-style 4, 2- to 4-row
chunks, long contexts), prompt rows (16 query rows of a head per workgroup: 5 rows and more, or
probabilities past the split form's LDS) and one workgroup per head (one row of a stream without a
scratch, V rows 128 MiB or more apart). Needs a gfx950 GPU."""
from __future__ import annotations

import ctypes

import numpy as np
import pytest
import torch

from attention_data import plant_attention_specials
from oracle import golden as G
from oracle import numerics as F
from oracle import rowops as R
from opentars_amd import ops
from opentars_amd.build import LIB
from opentars_amd.contract import OUT_BF16, OUT_FP32, OUT_INT8

pytestmark = pytest.mark.gpu
f32 = np.float32


def bits(a) -> np.ndarray:
    a = np.asarray(a)
    return a.view(np.uint32) if a.dtype == f32 else a.view(np.uint16) if a.itemsize == 2 else a.view(np.uint8)


def oracle_attention(q, kc, vval, heads, kv_heads, hd, causal_k, out, osc):
    """Per head in order: scores, causal softmax, P V, converted; the last head's scores and
    probabilities (what the shared buffers hold at the end)."""
    M, nk = q.shape[0], kc.shape[0]
    grp = heads // kv_heads
    valid = [min(nk, causal_k + m) if causal_k > 0 else nk for m in range(M)]
    att = []
    for h in range(heads):
        kv = h // grp
        s = R.fdot_nt(q[:, h * hd:(h + 1) * hd], kc[:, kv * hd:(kv + 1) * hd])
        p = R.softmax_rows_causal(s, valid)
        att.append(G.convert(R.fdot_nn(p, vval[:, kv * hd:(kv + 1) * hd]), out, osc))
    return np.concatenate(att, axis=1), s, p


def layer(seed, heads, kv_heads, hd, M, t0, v_fp16, specials):
    rng = np.random.default_rng(seed)
    nk = (t0 + M + 15) // 16 * 16
    q = rng.normal(0, 0.3, (M, heads * hd)).astype(f32)
    kc = rng.normal(0, 1, (nk, kv_heads * hd)).astype(f32)
    vv = rng.normal(0, 1, (nk, kv_heads * hd)).astype(f32)
    if specials:
        plant_attention_specials(rng, q, kc, vv, kv_heads, hd, v_fp16)
    vdev = vv.astype(np.float16).view(np.uint16) if v_fp16 else vv
    vval = F.from_fp16_bits(vdev) if v_fp16 else vv
    return q, kc, vdev, vval, nk


def run_case(heads, kv_heads, hd, M, t0, v_fp16, out, specials=False):
    q, kc, vdev, vval, nk = layer(heads * 1000 + hd + M * 7 + t0, heads, kv_heads, hd, M, t0, v_fp16, specials)
    osc = f32(4.0) if out == OUT_INT8 else None
    sc = torch.full((M, nk), float("nan"), device="cuda")
    pr = torch.full((M, nk), float("nan"), device="cuda")
    got = ops.attention(q, kc, vdev, heads, kv_heads, causal_k=t0 + 1, v_fp16=v_fp16, out=out, out_scale=osc,
                        sc=sc, pr=pr)
    want, s_last, p_last = oracle_attention(q, kc, vval, heads, kv_heads, hd, t0 + 1, out, osc)
    g, w = bits(got), bits(want)
    bad = np.argwhere(g != w)
    assert len(bad) == 0, f"att: {len(bad)} differ, first at {tuple(bad[0])}: {g[tuple(bad[0])]:#x} vs {w[tuple(bad[0])]:#x}"
    assert np.array_equal(bits(sc.cpu().numpy()), bits(s_last)), "last head's scores"
    assert np.array_equal(bits(pr.cpu().numpy()), bits(p_last)), "last head's probabilities"


CASES = [
    (16, 8, 128, 1, 250, False, OUT_FP32),   # Qwen3-0.6B decode: split, 2 query heads per K / V head
    (4, 1, 256, 1, 37, True, OUT_FP32),      # head size 256, fp16 V, 4 query heads per K / V head
    (8, 4, 64, 2, 100, False, OUT_BF16),     # a 2-row chunk: 4 query rows per group
    (6, 6, 128, 3, 60, False, OUT_INT8),     # 3 rows, no sharing
    (2, 1, 128, 4, 500, False, OUT_FP32),    # 4 rows: the group split back to single heads
    (2, 1, 64, 5, 30, False, OUT_FP32),      # 5 rows: the prompt-row kernel
    (2, 1, 64, 1, 2000, True, OUT_FP32),     # 2016 keys: 63 scores workgroups per head
    (2, 2, 128, 1, 4070, False, OUT_FP32),   # 4080 keys, the most any form takes
    (4, 2, 128, 2, 3000, False, OUT_FP32),   # probabilities past the split form's LDS: the prompt-row kernel
    (3, 3, 64, 1, 0, False, OUT_FP32),       # the first position: one valid key of 16
]


@pytest.mark.parametrize("heads,kv_heads,hd,M,t0,v_fp16,out", CASES)
def test_attention_matches_the_oracle(heads, kv_heads, hd, M, t0, v_fp16, out):
    run_case(heads, kv_heads, hd, M, t0, v_fp16, out)


@pytest.mark.parametrize("heads,kv_heads,hd,M,t0,v_fp16", [
    (16, 8, 128, 1, 250, False),
    (4, 2, 128, 2, 40, False),
    (2, 1, 64, 1, 300, True),
    (2, 1, 256, 1, 20, False),
    (2, 1, 64, 5, 30, False),
])
def test_attention_with_values_the_flushes_change(heads, kv_heads, hd, M, t0, v_fp16):
    run_case(heads, kv_heads, hd, M, t0, v_fp16, OUT_FP32, specials=True)


# the split form at the edges of its P V stages (64 keys, read in halves; 2, 4 or 8 stages ahead) and of the
# scores' key chunks, 1 to 4 query rows per group (key counts are multiples of 4), with scores spread so far that probabilities underflow to
# subnormal products and zeros; bit for bit, so no tolerance
@pytest.mark.parametrize("nk,M,grp,v_fp16,specials", [
    (4, 1, 1, False, False), (8, 2, 2, True, False), (28, 1, 2, False, True), (36, 3, 1, True, True),
    (60, 1, 4, False, False), (64, 2, 1, False, True), (68, 1, 2, True, False), (124, 4, 1, False, True),
    (128, 1, 4, True, True), (132, 1, 1, False, False), (252, 2, 2, False, True), (256, 1, 2, True, True),
    (260, 3, 1, False, False), (508, 1, 2, True, True), (512, 4, 1, False, True), (516, 1, 4, False, True),
    (580, 1, 2, False, True), (1028, 2, 1, True, True), (2052, 1, 1, False, True), (1092, 1, 2, True, False),
])
def test_split_attention_at_the_stage_edges(nk, M, grp, v_fp16, specials):
    rng = np.random.default_rng(nk * 8 + M)
    kv_heads, hd = 2, 64
    heads = kv_heads * grp
    q = rng.normal(0, 4.0, (M, heads * hd)).astype(f32)
    kc = rng.normal(0, 1.5, (nk, kv_heads * hd)).astype(f32)
    vv = rng.normal(0, 1, (nk, kv_heads * hd)).astype(f32)
    if specials and nk >= 16:
        plant_attention_specials(rng, q, kc, vv, kv_heads, hd, v_fp16)
    vdev = vv.astype(np.float16).view(np.uint16) if v_fp16 else vv
    vval = F.from_fp16_bits(vdev) if v_fp16 else vv
    for causal_k in (0, max(1, nk - M + 1)):
        got = ops.attention(q, kc, vdev, heads, kv_heads, causal_k=causal_k, v_fp16=v_fp16)
        want, _, _ = oracle_attention(q, kc, vval, heads, kv_heads, hd, causal_k, OUT_FP32, None)
        bad = np.argwhere(bits(got) != bits(want))
        assert len(bad) == 0, f"causal_k={causal_k}: {len(bad)} differ, first at {tuple(bad[0])}"


# prompt rows (16 query rows per workgroup): one row of a tile, whole and partial tiles, every head size
# and V format, both sides of the key count past which a tile holds 8 rows (2544 keys)
PROMPT_CASES = [
    (16, 8, 128, 5, 60, False, OUT_INT8, False),
    (2, 1, 64, 16, 0, False, OUT_FP32, False),
    (8, 4, 64, 17, 3, True, OUT_BF16, False),
    (3, 3, 128, 33, 100, False, OUT_FP32, True),
    (2, 1, 256, 40, 30, True, OUT_FP32, True),
    (8, 8, 256, 18, 7, False, OUT_FP32, True),
    (2, 2, 64, 20, 2520, False, OUT_FP32, False),
    (1, 1, 64, 9, 2540, False, OUT_FP32, True),
    (1, 1, 128, 23, 4050, True, OUT_FP32, False),
]


@pytest.mark.parametrize("heads,kv_heads,hd,M,t0,v_fp16,out,specials", PROMPT_CASES)
def test_attention_of_prompt_rows(heads, kv_heads, hd, M, t0, v_fp16, out, specials):
    run_case(heads, kv_heads, hd, M, t0, v_fp16, out, specials)


@pytest.mark.parametrize("v_fp16", [False, True])
def test_masked_keys_of_prompt_rows_that_change_a_sum(v_fp16):
    """Keys no row of a tile sees still take part in P V with probability +0: an infinite V element
    there makes NaN, and a sum that was flushed to -0 becomes +0 (or stays -0, by the V signs)."""
    M, nk, hd, causal_k = 40, 160, 64, 20
    rng = np.random.default_rng(5)
    q, kc, vv = (rng.normal(0, 0.5, s).astype(f32) for s in ((M, hd), (nk, hd), (nk, hd)))
    kc[1] = kc[0]
    vv[nk - 1, 7] = np.inf                              # masked for every row
    vv[causal_k + 30, 9] = np.nan                       # masked for the first rows only
    if not v_fp16:                                      # p0 v0 + p1 v1 = -2^-126 p, flushed to -0
        vv[0, 3:5], vv[1, 3:5] = f32(2.0 ** -103) * f32(1 - 2.0 ** -23), -f32(2.0 ** -103)
        vv[2:causal_k + M, 3:5] = -0.0
        vv[causal_k + M:, 3], vv[causal_k + M:, 4] = 1.0, -1.0
    vdev = vv.astype(np.float16).view(np.uint16) if v_fp16 else vv
    vval = F.from_fp16_bits(vdev) if v_fp16 else vv
    got = ops.attention(q, kc, vdev, 1, 1, causal_k=causal_k, v_fp16=v_fp16)
    want = oracle_attention(q, kc, vval, 1, 1, hd, causal_k, OUT_FP32, None)[0]
    if not v_fp16:
        assert np.all(bits(want[:, 3]) == 0) and np.all(bits(want[:, 4]) == 0x80000000)
    assert np.array_equal(bits(got), bits(want))


@pytest.mark.parametrize("M,nk,hd", [(2, 48, 128), (4, 100, 64), (5, 48, 128), (40, 100, 64), (33, 64, 256)])
@pytest.mark.parametrize("causal_k", [2 ** 31 - 1, 2 ** 31 - 3])
def test_causal_k_near_the_largest_int_is_no_mask(M, nk, hd, causal_k):
    """min(nk, causal_k + m) is nk for every row, whatever causal_k + m is in 32 bits: the same as causal_k = 0,
    the scores and probabilities with it. The split form (2 and 4 rows) and prompt rows."""
    rng = np.random.default_rng(M)
    q, kc, vv = (rng.normal(0, 0.5, s).astype(f32) for s in ((M, 2 * hd), (nk, hd), (nk, hd)))
    sc, pr = (torch.full((M, nk), float("nan"), device="cuda") for _ in range(2))
    got = ops.attention(q, kc, vv, 2, 1, causal_k=causal_k, sc=sc, pr=pr)
    want, s_last, p_last = oracle_attention(q, kc, vv, 2, 1, hd, 0, OUT_FP32, None)
    assert np.array_equal(bits(got), bits(want))
    assert np.array_equal(bits(sc.cpu().numpy()), bits(s_last))
    assert np.array_equal(bits(pr.cpu().numpy()), bits(p_last))


def test_attention_twice_in_a_row_and_without_the_shared_rows():
    """Two calls on one stream share the device scratch: the second (fewer keys, other heads)
    must not see the first's scores; sc / pr left out."""
    for heads, kv_heads, t0 in ((16, 8, 250), (4, 2, 40)):
        q, kc, vdev, vval, nk = layer(t0, heads, kv_heads, 128, 1, t0, False, False)
        got = ops.attention(q, kc, vdev, heads, kv_heads, causal_k=t0 + 1)
        want = oracle_attention(q, kc, vval, heads, kv_heads, 128, t0 + 1, OUT_FP32, None)[0]
        assert np.array_equal(bits(got), bits(want))


def test_attention_on_two_streams_at_once():
    """Calls on two streams overlap in time: each stream's split form has its own scores scratch,
    so every call's output matches the oracle (one shared scratch would mix their scores)."""
    data = []
    for i, (heads, kv_heads, t0) in enumerate(((16, 8, 250), (16, 8, 170))):
        q, kc, vdev, vval, nk = layer(700 + i, heads, kv_heads, 128, 1, t0, False, False)
        want = oracle_attention(q, kc, vval, heads, kv_heads, 128, t0 + 1, OUT_FP32, None)[0]
        dev = [torch.from_numpy(np.ascontiguousarray(a)).cuda() for a in (q, kc, vdev)]
        data.append((dev, want, heads, kv_heads, t0))
    streams = [torch.cuda.Stream(), torch.cuda.Stream()]
    outs = [[], []]
    torch.cuda.synchronize()
    for rep in range(16):
        for j in (0, 1):
            (q, kc, v), _, heads, kv_heads, t0 = data[j]
            with torch.cuda.stream(streams[j]):
                att = torch.empty((1, heads * 128), dtype=torch.float32, device="cuda")
                ops.attention(q, kc, v, heads, kv_heads, causal_k=t0 + 1, att=att)
                outs[j].append(att)
    torch.cuda.synchronize()
    for j in (0, 1):
        for rep, att in enumerate(outs[j]):
            assert np.array_equal(bits(att.cpu().numpy()), bits(data[j][1])), f"stream {j}, call {rep}"


def graph_nodes(g: torch.cuda.CUDAGraph) -> int:
    n = ctypes.c_size_t(0)
    assert ctypes.CDLL(str(LIB)).hipGraphGetNodes(ctypes.c_void_p(g.raw_cuda_graph()), None, ctypes.byref(n)) == 0
    return n.value


# without a scratch: one workgroup per head for one row (up to 64 keys, up to 128, and more take different numbers of
# keys at a time), the prompt-row kernel for 3
@pytest.mark.parametrize("heads,kv_heads,hd,M,t0,v_fp16,specials", [
    (4, 2, 128, 1, 40, False, True), (2, 1, 64, 1, 100, True, True), (2, 2, 256, 1, 60, False, False),
    (8, 1, 64, 1, 300, False, True), (2, 1, 256, 1, 250, True, True), (2, 1, 128, 1, 2100, True, False),
    (2, 1, 128, 1, 4070, False, False), (4, 2, 128, 3, 60, False, True),
])
def test_first_attention_of_a_stream_inside_a_graph_capture(heads, kv_heads, hd, M, t0, v_fp16, specials):
    """A stream whose first attention call is captured gets no scratch (nothing is allocated under capture): one
    kernel instead of the split form's two. Every replay equals the oracle, with eager calls between them."""
    q, kc, vdev, vval, nk = layer(900 + t0 + hd, heads, kv_heads, hd, M, t0, v_fp16, specials)
    want, s_last, p_last = oracle_attention(q, kc, vval, heads, kv_heads, hd, t0 + 1, OUT_FP32, None)
    dq, dk, dv = (torch.from_numpy(np.ascontiguousarray(a)).cuda() for a in (q, kc, vdev.view(np.int16) if v_fp16 else vdev))
    att = torch.empty((M, heads * hd), device="cuda")
    sc, pr = torch.empty((M, nk), device="cuda"), torch.empty((M, nk), device="cuda")
    hip, handle = ctypes.CDLL(str(LIB)), ctypes.c_void_p()
    assert hip.hipStreamCreate(ctypes.byref(handle)) == 0   # torch's own streams come from a pool: another test's, perhaps
    stream = torch.cuda.ExternalStream(handle.value)
    g = torch.cuda.CUDAGraph(keep_graph=True)
    with torch.cuda.graph(g, stream=stream):
        ops.attention(dq, dk, dv, heads, kv_heads, causal_k=t0 + 1, v_fp16=v_fp16, att=att, sc=sc, pr=pr)
    assert graph_nodes(g) == 1
    for rep in range(3):
        for t in (att, sc, pr):
            t.fill_(float("nan"))
        eager = ops.attention(dq, dk, dv, heads, kv_heads, causal_k=t0 + 1, v_fp16=v_fp16)
        g.replay()
        torch.cuda.synchronize()
        for t, w in ((att, want), (sc, s_last), (pr, p_last), (eager, want)):
            assert np.array_equal(bits(t.cpu().numpy()), bits(w)), f"replay {rep}"
    del g
    assert hip.hipStreamDestroy(handle) == 0


def test_rows_of_v_128_mib_apart():
    """V row strides past the prompt-row kernel's 32-bit offsets: one workgroup per head, its rows one after another."""
    heads, hd, M, nk, causal_k = 2, 64, 6, 6, 2
    rng = np.random.default_rng(8)
    q, kc, vv = (rng.normal(0, 0.5, s).astype(f32) for s in ((M, heads * hd), (nk, hd), (nk, hd)))
    v = torch.empty(((nk - 1) << 25) + hd, device="cuda").as_strided((nk, hd), (1 << 25, 1))
    v.copy_(torch.from_numpy(vv))
    sc, pr = torch.empty((M, nk + 2), device="cuda")[:, :nk], torch.empty((M, nk + 2), device="cuda")[:, :nk]
    att = ops.attention(torch.from_numpy(q).cuda(), torch.from_numpy(kc).cuda(), v, heads, 1, causal_k=causal_k, sc=sc, pr=pr)
    want, s_last, p_last = oracle_attention(q, kc, vv, heads, 1, hd, causal_k, OUT_FP32, None)
    for t, w in ((att, want), (sc, s_last), (pr, p_last)):
        assert np.array_equal(bits(t.cpu().numpy()), bits(w))


def test_attention_refusals():
    q = torch.zeros((1, 256), device="cuda")
    kc = torch.zeros((32, 128), device="cuda")
    with pytest.raises(ops.TarsError):
        ops.attention(q, kc, kc, 2, 1, att=q)                   # the output is the q rows
    with pytest.raises(ValueError):
        ops.attention(q, kc, kc, 3, 1)                          # 3 heads over 256 columns
    with pytest.raises(ops.TarsError):
        ops.attention(torch.zeros((1, 96), device="cuda"), torch.zeros((32, 48), device="cuda"),
                      torch.zeros((32, 48), device="cuda"), 2, 1)   # head size 48


def test_zero_wide_heads_are_refused_by_the_library():
    q, kc = torch.zeros((1, 0), device="cuda"), torch.zeros((32, 0), device="cuda")
    with pytest.raises(ops.TarsError):
        ops.attention(q, kc, kc, 2, 1)
