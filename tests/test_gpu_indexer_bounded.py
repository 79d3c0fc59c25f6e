"""The fused indexer's bounded path (64 heads of 128 dims) at the sizes where its forms change: few queries a batch
(a workgroup per query), rows counted by the recomputation or by a histogram launch, and top-k lists that fall into one
segment of a row; indices against the oracle, bit for bit."""
import numpy as np
import pytest
import torch

import oracle
from kernelswift_amd import ops, workloads
from tests.test_gpu_indexer import _bounded_scores_gpu

pytestmark = pytest.mark.gpu

_u16 = workloads.bf16_bits


def _check(device, q, k, w, k_top, causal, start_pos, ratio=1, offset=0, rows=None):
    tab = workloads.freqs_table(64, max(k.shape[1], start_pos + q.shape[1]) + 1)
    got = ops.indexer(q.to(device), k.to(device), w.to(device), tab.to(device), k_top, causal, start_pos, ratio, offset,
                      0, 64, True).cpu().numpy().astype(np.int64)
    for b in range(q.shape[0]):
        want = oracle.indexer(_u16(q[b:b + 1]), _u16(k[b:b + 1]), w[b:b + 1].numpy() if w.dtype == torch.float32
                              else _u16(w[b:b + 1]), tab.numpy(), k_top, causal, start_pos, ratio, offset, 0, 64, True)
        np.testing.assert_array_equal(got[b:b + 1], want)


# one to five queries (the few-queries form up to four); one key, a partial group of 64, a partial last workgroup;
# 8192 and 8193 columns (counted by the recomputation / by the histogram launch); causal limits inside a group and before
# the row's later groups
@pytest.mark.parametrize("B,S,T,k_top,causal,start,ratio", [
    (1, 1, 1, 1, False, 0, 1), (2, 1, 63, 64, False, 0, 1), (3, 2, 65, 32, True, 30, 1), (1, 4, 511, 100, True, 508, 1),
    (2, 3, 1025, 512, False, 700, 1), (1, 1, 8192, 512, False, 8191, 1), (1, 2, 8193, 2048, True, 8191, 1),
    (1, 5, 8193, 700, True, 4000, 1), (2, 1, 5000, 300, True, 4399, 2), (1, 4, 600, 64, True, 0, 3)])
def test_few_queries(device, B, S, T, k_top, causal, start, ratio):
    g = torch.Generator().manual_seed(B * 7 + S * T)
    q = torch.randn(B, S, 64, 128, generator=g).bfloat16()
    k = torch.randn(B, T, 128, generator=g).bfloat16()
    w = torch.randn(B, S, 64, generator=g) / 8
    print(f"[case] few queries B={B} S={S} T={T} k={k_top} causal={causal} start={start}", flush=True)
    _check(device, q, k, w, k_top, causal, start, ratio, offset=5)


def test_few_queries_several_groups_per_wave(device):
    g = torch.Generator().manual_seed(2)
    q = torch.randn(24, 4, 64, 128, generator=g).bfloat16()
    k = torch.randn(24, 16000, 128, generator=g).bfloat16()
    w = torch.randn(24, 4, 64, generator=g) / 8
    print("[case] few queries, several groups per wave", flush=True)
    tab = workloads.freqs_table(64, 16001)
    got = ops.indexer(q.to(device), k.to(device), w.to(device), tab.to(device), 256, True, 15996, 1, 0, 0, 64, True)
    for b in (0, 23):  # the oracle on the first and last batch
        want = oracle.indexer(_u16(q[b:b + 1]), _u16(k[b:b + 1]), w[b:b + 1].numpy(), tab.numpy(), 256, True, 15996, 1, 0,
                              0, 64, True)
        np.testing.assert_array_equal(got[b:b + 1].cpu().numpy().astype(np.int64), want)


# the whole top k in one segment of the row (keys parallel to the queries there): its list outgrows the threads that read
# it, and at T = 12000 with k = 2048 the others stay empty
@pytest.mark.parametrize("S,T,k_top,lo", [(64, 12000, 2048, 8200), (3, 8192, 1500, 4096), (130, 4000, 1024, 2900)])
def test_top_k_in_one_segment(device, S, T, k_top, lo):
    g = torch.Generator().manual_seed(S + T)
    q = torch.randn(1, S, 64, 128, generator=g)
    q[..., 64:] = torch.randn(128 - 64, generator=g)  # the unrotated half, shared by every query and head
    k = torch.randn(1, T, 128, generator=g) * 0.25
    k[0, lo:lo + k_top, 64:] += q[0, 0, 0, 64:] * 2
    q, k = q.bfloat16(), k.bfloat16()
    w = torch.rand(1, S, 64, generator=g) / 8
    print(f"[case] top k in one segment S={S} T={T} k={k_top}", flush=True)
    rows = slice(0, min(S, 4))
    tab = workloads.freqs_table(64, T + 1)
    got = ops.indexer(q.to(device), k.to(device), w.to(device), tab.to(device), k_top, False, 0, 1, 0, 0, 64, True)
    want = oracle.indexer(_u16(q[:, rows]), _u16(k), w[:, rows].numpy(), tab.numpy(), k_top, False, 0, 1, 0, 0, 64, True)
    np.testing.assert_array_equal(got[:, rows].cpu().numpy().astype(np.int64), want)
    assert ((want >= lo) & (want < lo + k_top)).mean() > 0.9


# bf16 head weights: products and scores rounded to bf16, so that many scores tie and the order rests on the columns
@pytest.mark.parametrize("B,S,T,k_top,causal,start,scale", [
    (1, 24, 3000, 512, True, 2976, 1.0), (2, 1, 9000, 512, False, 8999, 1.0), (2, 3, 700, 700, True, 100, 1.0),
    (1, 40, 750, 512, True, 0, 1.0), (1, 9, 2048, 300, False, 0, 2.0 ** -60), (1, 9, 2048, 300, False, 0, 2.0 ** 40)])
def test_bf16_weights(device, B, S, T, k_top, causal, start, scale):
    g = torch.Generator().manual_seed(B + S * T)
    q = (torch.randn(B, S, 64, 128, generator=g) * scale).bfloat16()
    k = torch.randn(B, T, 128, generator=g).bfloat16()
    w = (torch.randn(B, S, 64, generator=g) * 0.05)
    w[:, :, ::9] = 0.0
    print(f"[case] bf16 weights B={B} S={S} T={T} k={k_top} causal={causal} scale={scale}", flush=True)
    _check(device, q, k, w.bfloat16(), k_top, causal, start)


@pytest.mark.parametrize("wbf", [False, True])
def test_equal_keys_and_tiny_weights(device, wbf):
    # every key the same row (every score ties: the columns decide), and weights from subnormal to large
    g = torch.Generator().manual_seed(6)
    q = torch.randn(1, 6, 64, 128, generator=g).bfloat16()
    k = torch.randn(1, 1, 128, generator=g).expand(1, 5000, 128).contiguous().bfloat16()
    w = torch.randn(1, 6, 64, generator=g)
    w[0, 1] = 0.0
    w[0, 2] *= 2.0 ** -130
    w[0, 3] *= 2.0 ** -115
    w[0, 4] *= 2.0 ** 60
    print(f"[case] equal keys, weights of all magnitudes, bf16={wbf}", flush=True)
    _check(device, q, k, w.bfloat16() if wbf else w, 600, False, 0)
    k = torch.randn(1, 1500, 128, generator=g).bfloat16()
    _check(device, q, k, w.bfloat16() if wbf else w, 600, False, 0)


# rows of one segment (at most 1024 keys), ranked by the recomputation: with every column recomputed (k near the row's
# length, causal prompts) and with a threshold; edges of the two columns per thread, tiles of 16, rows without a live key
@pytest.mark.parametrize("wbf", [False, True])
@pytest.mark.parametrize("B,S,T,k_top,causal,start,ratio", [
    (1, 6, 1, 1, False, 0, 1), (1, 7, 17, 16, False, 0, 1), (2, 40, 33, 12, True, 0, 1), (1, 9, 512, 512, False, 0, 1),
    (1, 9, 513, 40, False, 0, 1), (1, 6, 1023, 1000, False, 0, 1), (1, 6, 1024, 100, False, 0, 1),
    (1, 6, 1025, 1000, False, 0, 1), (1, 70, 600, 512, True, 531, 1), (1, 300, 75, 64, True, 0, 4)])
def test_one_segment_rows(device, wbf, B, S, T, k_top, causal, start, ratio):
    g = torch.Generator().manual_seed(B + S * T + k_top)
    q = torch.randn(B, S, 64, 128, generator=g).bfloat16()
    k = torch.randn(B, T, 128, generator=g).bfloat16()
    w = torch.randn(B, S, 64, generator=g) / 8
    w[:, ::3, ::5] = 0.0
    print(f"[case] one segment B={B} S={S} T={T} k={k_top} causal={causal} start={start} bf16={wbf}", flush=True)
    _check(device, q, k, w.bfloat16() if wbf else w, k_top, causal, start, ratio, offset=3)


@pytest.mark.parametrize("wbf", [False, True])
@pytest.mark.parametrize("k_top", [90, 600])
def test_one_segment_rows_ties_and_range(device, wbf, k_top):
    g = torch.Generator().manual_seed(k_top)
    w = torch.randn(1, 5, 64, generator=g) * 0.05
    w[0, 1] = 0.0                                          # every score zero: the columns decide (and the merge sort)
    q = torch.randn(1, 5, 64, 128, generator=g)
    k = torch.randn(1, 700, 128, generator=g)
    k[0, 300:] = k[0, :1]                                  # 400 equal keys
    print(f"[case] one segment, ties, k={k_top} bf16={wbf}", flush=True)
    _check(device, q.bfloat16(), k.bfloat16(), w.bfloat16() if wbf else w, k_top, False, 0)
    # integers: dots on bf16 midpoints; norms past the overflow guard: no end certifies a score
    q, k = torch.randint(-4, 5, q.shape, generator=g).float(), torch.randint(-4, 5, k.shape, generator=g).float()
    print(f"[case] one segment, midpoints, k={k_top} bf16={wbf}", flush=True)
    _check(device, q.bfloat16(), k.bfloat16(), w.bfloat16() if wbf else w, k_top, False, 0)
    print(f"[case] one segment, overflow guard, k={k_top} bf16={wbf}", flush=True)
    _check(device, (q * 2.0 ** 59).bfloat16(), (k * 2.0 ** 59).bfloat16(), w.bfloat16() if wbf else w, k_top, False, 0)


# rows whose every score is recomputed: the recomputation rotates the queries and scales the weights itself; rotated ranges
# at either end, inside, of all dims and none, rotated and plain keys, a scale that is not a power of two
@pytest.mark.parametrize("rs,rd,rope_k,wbf,scale", [
    (0, 64, True, True, 0.0127), (64, 64, False, True, -0.0127), (64, 64, False, False, 0.0127), (24, 96, True, False, 1.0),
    (0, 128, False, True, 1.0), (0, 0, False, False, 0.3)])
def test_one_segment_prepares_queries(device, rs, rd, rope_k, wbf, scale):
    g = torch.Generator().manual_seed(rs + rd)
    B, S, T, start = 2, 37, 90, 300
    q = torch.randn(B, S, 64, 128, generator=g).bfloat16()
    cache = torch.randn(B, T + 7, 128, generator=g).bfloat16()
    w = torch.randn(B, S, 64, generator=g)
    w = w.bfloat16() if wbf else w
    tab = workloads.freqs_table(max(rd, 2), start + S + 1)
    print(f"[case] recomputation prepares queries rope {rs}+{rd} keys={rope_k} bf16={wbf}", flush=True)
    got = ops.indexer(q.to(device), cache.to(device), w.to(device), tab.to(device), 80, True, start, 4, 11, rs, rd, rope_k,
                      T=T, w_scale=scale).cpu().numpy().astype(np.int64)
    ws = w * scale
    for b in range(B):
        want = oracle.indexer(_u16(q[b:b + 1]), _u16(cache[b:b + 1, :T].contiguous()), _u16(ws[b:b + 1]) if wbf else
                              ws[b:b + 1].numpy(), tab.numpy(), 80, True, start, 4, 11, rs, rd, rope_k)
        np.testing.assert_array_equal(got[b:b + 1], want)


# infinite scores of finite inputs: they rank first (+inf) and last (-inf), among themselves by column.  One segment with
# every column recomputed and with a threshold, lists over short causal prefixes and long rows; "dots": one head's dot
# rounds to +inf; "weights": the weighted dot overflows
@pytest.mark.parametrize("wbf", [False, True])
@pytest.mark.parametrize("how", ["dots", "weights"])
@pytest.mark.parametrize("S,T,k_top,causal,start,share", [
    (9, 100, 100, False, 0, 0.1), (6, 250, 100, False, 0, 0.7), (7, 1024, 700, False, 0, 0.2), (8, 3000, 512, True, 120, 0.3),
    (6, 3000, 300, False, 0, 0.95), (3, 9000, 600, False, 0, 0.04)])
def test_infinite_scores(device, wbf, how, S, T, k_top, causal, start, share):
    g = torch.Generator().manual_seed(T + k_top)
    q = torch.randn(1, S, 64, 128, generator=g)
    k = torch.randn(1, T, 128, generator=g)
    w = torch.randn(1, S, 64, generator=g) / 8
    w[0, :, 0] = torch.where(torch.arange(S) % 3 == 0, 1.0, -1.0)
    rows = torch.rand(T, generator=g) < share
    k[0, rows, 64:] = 2.0 ** (62 if how == "dots" else 10)  # the unrotated half
    q[0, :, 0, 64:] = 2.0 ** (62 if how == "dots" else 10)  # head 0: dot 2^130 (bf16 infinity) or 2^26
    if how == "weights":
        w[0, :, 0] *= 2.0 ** 105
    print(f"[case] infinite scores {how} S={S} T={T} k={k_top} causal={causal} bf16={wbf}", flush=True)
    _check(device, q.bfloat16(), k.bfloat16(), w.bfloat16() if wbf else w, k_top, causal, start)


# dots in bf16's subnormal range under large weights, where a rounding moves a dot by a whole step however small it is: the
# first columns' dots lie 2^-155 above a tie (5 steps, 4 by the MFMA sum), which beats the 4.5 steps of the next columns
@pytest.mark.parametrize("wbf", [False, True])
@pytest.mark.parametrize("S,T", [(3, 600), (20, 600), (2, 9000), (12, 2500)])
def test_subnormal_dots_large_weights(device, wbf, S, T):
    n = 100
    q = torch.zeros(1, S, 64, 128)
    k = torch.zeros(1, T, 128)
    w = torch.full((1, S, 64), 2.0 ** -10)
    q[0, :, 0, 64], q[0, :, 0, 65], q[0, :, 1, 66] = 2.0 ** -66, 2.0 ** -78, 2.0 ** -66
    w[0, :, 0], w[0, :, 1] = 2.0 ** 40, 2.0 ** 39
    k[0, 50:50 + n, 64], k[0, 50:50 + n, 65] = 4.5 * 2.0 ** -67, 2.0 ** -77
    k[0, 300:300 + 2 * n, 64], k[0, 300:300 + 2 * n, 66] = 4.0 * 2.0 ** -67, 2.0 ** -67
    print(f"[case] subnormal dots, large weights S={S} T={T} bf16={wbf}", flush=True)
    _check(device, q.bfloat16(), k.bfloat16(), w.bfloat16() if wbf else w, n, False, 0)


# more tied scores than the ranking takes in LDS: the whole-row selection over the lists, in the workspace (at most 8192
# columns) and over the rows' own scores and bounds (more); a ragged last segment, causal prefixes inside a segment
@pytest.mark.parametrize("S,T,k_top,causal,start", [
    (5, 8192, 700, False, 0), (6, 9001, 2048, False, 0), (5, 20000, 1000, True, 17300), (3, 32768, 2048, False, 0),
    (300, 8200, 64, False, 0)])
def test_long_lists_of_ties(device, S, T, k_top, causal, start):
    g = torch.Generator().manual_seed(T)
    q = torch.randn(1, S, 64, 128, generator=g).abs().bfloat16()
    k = torch.randn(1, T, 128, generator=g)
    tied = torch.rand(T, generator=g) < 0.7
    k[0, tied] = torch.randn(1, 128, generator=g).abs() * 3  # ahead of most others
    k[0, :, :64] = 0.0                                       # nothing that the rotation changes
    w = torch.rand(1, S, 64, generator=g) / 8
    rows = slice(0, 6)
    print(f"[case] long lists of ties S={S} T={T} k={k_top} causal={causal}", flush=True)
    tab = workloads.freqs_table(64, T + 1)
    k = k.bfloat16()
    got = ops.indexer(q.to(device), k.to(device), w.to(device), tab.to(device), k_top, causal, start, 1, 0, 0, 64, True)
    want = oracle.indexer(_u16(q[:, rows]), _u16(k), w[:, rows].numpy(), tab.numpy(), k_top, causal, start, 1, 0, 0, 64, True)
    np.testing.assert_array_equal(got[:, rows].cpu().numpy().astype(np.int64), want)


# the bound itself, score by score, in the few-queries form (up to four queries) and the other one: |exact - S| <= U with
# U > 0; "subnormal": dots around the smallest bf16 steps under large weights
@pytest.mark.parametrize("dist", ["normal", "midpoints", "scaled", "subnormal"])
@pytest.mark.parametrize("S,T", [(1, 700), (4, 1100), (40, 1200)])
def test_bounds_contain_exact_scores(device, dist, S, T):
    g = torch.Generator().manual_seed(S + T)
    q, k = torch.randn(1, S, 64, 128, generator=g), torch.randn(1, T, 128, generator=g)
    w = torch.randn(1, S, 64, generator=g) / 8
    if dist == "midpoints":
        q, k = torch.randint(-3, 4, q.shape, generator=g).float(), torch.randint(-3, 4, k.shape, generator=g).float()
    elif dist == "scaled":
        q = q * torch.exp2(torch.randint(-8, 9, (1, S, 64, 1), generator=g).float())
        w = w * torch.exp2(torch.randint(-100, 60, (1, S, 64), generator=g).float())
    elif dist == "subnormal":
        q, k, w = q * 2.0 ** -66, k * 2.0 ** -69, w * 2.0 ** 33
    q, k = q.bfloat16(), k.bfloat16()
    print(f"[case] bounds contain exact scores {dist} S={S} T={T}", flush=True)
    got, u = _bounded_scores_gpu(q, k, w, T)  # every column is live
    want = oracle.indexer_scores(_u16(q), _u16(k), w.numpy(), True, T).astype(np.float64)
    assert (u > 0).all() and np.isfinite(u).all()
    assert (np.abs(want - got) <= u).all()
