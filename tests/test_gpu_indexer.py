"""GPU parity: indexer RoPE, exact scores and fused top-k vs the canonical CPU oracle (bit-exact).

Scores are compared bit for bit (float32 patterns), indices exactly, at the BASELINE.json shapes
(configs 2 and 4) and on small shapes that stress the exact-rounding path (integer-valued inputs whose
dots land exactly on bf16 midpoints, heavy-tailed data, wide dynamic range)."""
import numpy as np
import pytest
import torch

import oracle
from kernelswift_amd import ops, workloads
from kernelswift_amd import _lib

pytestmark = pytest.mark.gpu

bits = workloads.bf16_bits
BOUND_C = 13.0  # the interval constant derived for the MFMA accumulation (checked against the library below)


def test_bound_constant_is_the_derived_one(device):
    lib = _lib.load()
    assert lib.ks_dbg_score_bound_c() == BOUND_C
    # 64-dim dots (8 accumulation steps, tests/test_mfma_model.py::test_error_bound_of_64_dim_dots)
    assert lib.ks_dbg_score_bound_c_d(128) == BOUND_C and lib.ks_dbg_score_bound_c_d(64) == 9.0


def _u16(t):
    return bits(t)


def test_rope_bit_exact_first_and_last_segments(device):
    g = torch.Generator().manual_seed(1)
    q = torch.randn(2, 33, 4, 128, generator=g).bfloat16()
    tab = workloads.freqs_table(64, 4096)
    for rs, pos0 in [(0, 0), (64, 1000), (32, 7)]:
        print(f"[case] rope rope_start={rs} pos0={pos0}", flush=True)
        x = q.to(device)
        ops.rope_inplace(x, tab.to(device), rope_start=rs, pos0=pos0)
        torch.cuda.synchronize()
        want = oracle.rope_bf16(_u16(q), tab.numpy(), rs, 64, pos0)
        np.testing.assert_array_equal(_u16(x), want)


@pytest.mark.parametrize("scale", [2.0 ** -128, 2.0 ** -120, 2.0 ** 126])
def test_rope_bit_exact_extreme_magnitudes(device, scale):
    # rotated values in the subnormal range (the fp32 products and sums, and the bf16 results) and at the top
    # of the range (sums that overflow to infinity): the RNE conversion must match the oracle's bit for bit
    g = torch.Generator().manual_seed(3)
    q = (torch.randn(2, 17, 4, 128, generator=g) * scale).bfloat16()
    tab = workloads.freqs_table(64, 4096)
    print(f"[case] rope scale=2^{np.log2(scale):.0f}", flush=True)
    x = q.to(device)
    ops.rope_inplace(x, tab.to(device), rope_start=0, pos0=5)
    torch.cuda.synchronize()
    want = oracle.rope_bf16(_u16(q), tab.numpy(), 0, 64, 5)
    np.testing.assert_array_equal(_u16(x), want)


def test_row_stats(device):
    g = torch.Generator().manual_seed(2)
    x = torch.randn(300, 128, generator=g).bfloat16()
    x[5] = 0
    x[7, :100] = 0
    x[9, 3] = 1e-30
    print("[case] row stats", flush=True)
    n, s = ops.indexer_row_stats(x.to(device))
    n, s = n.cpu().numpy(), s.cpu().numpy()
    xf = oracle.bf16_to_f32(_u16(x)).astype(np.float64)
    true_n = np.sqrt((xf ** 2).sum(1))
    assert np.all(n >= true_n) and np.all(n <= true_n * (1 + 2 ** -10) + 1e-38)
    assert n[5] == 0 and s[5] == 0
    lsb = np.array([min([oracle_lsb(v) for v in _u16(x)[r] if v & 0x7FFF] or [0]) for r in range(300)])
    top = np.array([int(np.frexp(v)[1]) if v > 0 else 0 for v in n])
    np.testing.assert_array_equal(s[n > 0], (top - lsb)[n > 0])


def test_row_stats_past_the_range_of_squares(device):
    # rows whose squares leave the fp32 range: the norm stays an upper bound, and an infinite one claims no span
    g = torch.Generator().manual_seed(3)
    for D in (64, 128):
        x = torch.randn(40, D, generator=g)
        e = torch.tensor([2.0 ** i for i in range(-132, 124, 7)][:37])
        x[:37] *= e[:, None]
        x[37] = 2.0 ** -133
        x[38] = 2.0 ** 64
        x[39] = 0.0
        x = x.bfloat16()
        print(f"[case] row stats past the range of squares D={D}", flush=True)
        n, s = ops.indexer_row_stats(x.to(device))
        n, s = n.cpu().double(), s.cpu()
        true = x.double().pow(2).sum(1).sqrt()
        big = true > 2.0 ** -60
        assert (n >= true).all() and ((n[big] <= true[big] * (1 + 2 ** -10)) | torch.isinf(n[big])).all()
        assert n[39] == 0 and s[39] == 0
        assert (s[n == float("inf")] == 1024).all() and (n == float("inf")).any()


# dots on bf16 midpoints that a third, far smaller product decides, in rows whose squares leave the fp32 range: past it
# (infinite norms, span unknown) and below it (norms that would come out as zero)
@pytest.mark.parametrize("qe,ke", [(65, 0), (0, 65), (-80, 70), (70, -80), (-80, -30), (66, 40)])
@pytest.mark.parametrize("B,S,T,H,D", [(1, 2, 300, 64, 128), (1, 9, 300, 64, 128), (1, 9, 1500, 64, 128), (1, 9, 300, 32, 128),
                                       (1, 9, 300, 16, 64)])
def test_indexer_midpoints_of_extreme_rows(device, qe, ke, B, S, T, H, D):
    q = torch.zeros(B, S, H, D)
    k = torch.zeros(B, T, D)
    o = D - 8  # unrotated dims
    q[..., 0, o], q[..., 0, o + 1], q[..., 0, o + 2] = 2.0 ** qe, 2.0 ** (qe - 8), 2.0 ** (qe - 30)
    sign = torch.randint(-1, 2, (B, T), generator=torch.Generator().manual_seed(T)).float()
    k[..., o], k[..., o + 1], k[..., o + 2] = 2.0 ** ke, 2.0 ** ke, 2.0 ** (ke - 15) * sign
    w = torch.ones(B, S, H)
    q, k, k_top = q.bfloat16(), k.bfloat16(), 120
    tab = workloads.freqs_table(32, T + S)
    print(f"[case] midpoints of extreme rows 2^{qe} 2^{ke} {B, S, T, H, D}", flush=True)
    got = ops.indexer(q.to(device), k.to(device), w.to(device), tab.to(device), k_top, False, 0, 1, 0, 0, 32, True)
    want = oracle.indexer(_u16(q), _u16(k), w.numpy(), tab.numpy(), k_top, False, 0, 1, 0, 0, 32, True)
    np.testing.assert_array_equal(got.cpu().numpy().astype(np.int64), want)


def oracle_lsb(b):
    e = (int(b) >> 7) & 0xFF
    return -133 if e == 0 else e - 134


def _scores_gpu(q, k, w, causal, start_pos, ratio=1, bound_c=None):
    """Exact-score kernel through the C ABI; returns (scores, [recomputed, unresolved])."""
    qd, kd, wd = q.to("cuda"), k.to("cuda"), w.to("cuda")
    (qn, qs), (kn, ks_) = ops.indexer_row_stats(qd), ops.indexer_row_stats(kd)
    B, S, H, D = q.shape
    T = k.shape[1]
    out = torch.empty(B, S, T, dtype=torch.float32, device="cuda")
    st = torch.zeros(2, dtype=torch.int32, device="cuda")
    lib = _lib.load()
    rc = lib.ks_dbg_indexer_scores(qd.data_ptr(), kd.data_ptr(), wd.data_ptr(), 1 if w.dtype == torch.bfloat16 else 0,
                                   qn.data_ptr(), qs.data_ptr(), kn.data_ptr(), ks_.data_ptr(), out.data_ptr(),
                                   B, S, H, D, T, T, 1 if causal else 0, start_pos, ratio,
                                   BOUND_C if bound_c is None else bound_c, st.data_ptr(),
                                   torch.cuda.current_stream().cuda_stream)
    _lib.check(rc, "ks_dbg_indexer_scores")
    torch.cuda.synchronize()
    return out.cpu().numpy(), st.cpu().numpy()


def _oracle_scores(q, k, w, causal, start_pos, ratio=1):
    wn = _u16(w) if w.dtype == torch.bfloat16 else w.numpy()
    return oracle.indexer_scores(_u16(q), _u16(k), wn, causal, start_pos, ratio)


@pytest.mark.parametrize("D", [128, 64])
@pytest.mark.parametrize("H", [16, 32, 64])
@pytest.mark.parametrize("w_bf16", [False, True])
def test_scores_small_bit_exact(device, H, w_bf16, D):
    g = torch.Generator().manual_seed(H + w_bf16 + D)
    B, S, T = 2, 9, 300
    q = torch.randn(B, S, H, D, generator=g).bfloat16()
    k = torch.randn(B, T, D, generator=g).bfloat16()
    w = torch.randn(B, S, H, generator=g) / 8
    if w_bf16:
        w = w.bfloat16()
    print(f"[case] scores small H={H} D={D} w_bf16={w_bf16}", flush=True)
    got, st = _scores_gpu(q, k, w, True, T - S)
    want = _oracle_scores(q, k, w, True, T - S)
    np.testing.assert_array_equal(got.view(np.uint32), want.view(np.uint32))
    assert st[1] == 0


@pytest.mark.parametrize("D", [128, 64])
@pytest.mark.parametrize("H", [16, 32, 64])
@pytest.mark.parametrize("w_bf16", [False, True])
def test_scores_every_dot_deferred(device, H, w_bf16, D):
    # a huge error-bound constant makes every positive dot a near-tie: every key of every tile is deferred,
    # the per-wave entry list fills to capacity and each flush runs the exact path on all of its dots
    g = torch.Generator().manual_seed(7 * H + w_bf16 + D)
    B, S, T = 1, 11, 530
    q = torch.randn(B, S, H, D, generator=g).bfloat16()
    k = torch.randn(B, T, D, generator=g).bfloat16()
    w = torch.randn(B, S, H, generator=g) / 8
    if w_bf16:
        w = w.bfloat16()
    print(f"[case] scores all deferred H={H} D={D} w_bf16={w_bf16}", flush=True)
    got, st = _scores_gpu(q, k, w, True, T - S, bound_c=1e6)
    want = _oracle_scores(q, k, w, True, T - S)
    np.testing.assert_array_equal(got.view(np.uint32), want.view(np.uint32))
    assert st[0] > S * H * T // 4 and st[1] == 0


@pytest.mark.parametrize("D", [128, 64])
def test_scores_midpoint_ties_exact_path(device, D):
    # small-integer inputs: every dot is an integer computed exactly by the MFMA; odd values above 256
    # sit exactly on bf16 midpoints, so ties-to-even must come from the exact recomputation
    g = torch.Generator().manual_seed(7)
    q = torch.randint(-3, 4, (1, 8, 64, D), generator=g).bfloat16()
    k = torch.randint(-3, 4, (1, 512, D), generator=g).bfloat16()
    w = torch.randn(1, 8, 64, generator=g) / 8
    print("[case] scores integer midpoints", flush=True)
    got, st = _scores_gpu(q, k, w, False, 0)
    want = _oracle_scores(q, k, w, False, 0)
    np.testing.assert_array_equal(got.view(np.uint32), want.view(np.uint32))
    assert st[0] > 0 and st[1] == 0


@pytest.mark.parametrize("dist", ["heavy", "scaled", "tiny"])
def test_scores_adversarial_distributions(device, dist):
    g = torch.Generator().manual_seed(11)
    q = torch.randn(1, 16, 64, 128, generator=g)
    k = torch.randn(1, 1024, 128, generator=g)
    if dist == "heavy":  # heavy tails (x^3), tiny values flushed so rows stay inside the exact range
        q, k = q ** 3, k ** 3
        q = torch.where(q.abs() < 1e-3, torch.zeros_like(q), q)
        k = torch.where(k.abs() < 1e-3, torch.zeros_like(k), k)
    elif dist == "scaled":
        q = q * torch.exp2(torch.randint(-8, 9, (1, 16, 64, 1), generator=g).float())
        k = k * torch.exp2(torch.randint(-8, 9, (1, 1024, 1), generator=g).float())
    else:  # values near 0 mixed with O(1): wide dynamic range inside rows
        q = q * torch.exp2(torch.randint(-30, 1, q.shape, generator=g).float())
    q, k = q.bfloat16(), k.bfloat16()
    w = torch.randn(1, 16, 64, generator=g) / 8
    print(f"[case] scores adversarial {dist}", flush=True)
    got, st = _scores_gpu(q, k, w, True, 1024 - 16)
    want = _oracle_scores(q, k, w, True, 1024 - 16)
    np.testing.assert_array_equal(got.view(np.uint32), want.view(np.uint32))
    assert st[1] == 0


def test_scores_outside_double_range_exact(device):
    # x^3 of N(0,1) without flushing: row magnitudes span up to ~2^90, beyond the double-precision paths
    # (span_q + span_k <= 84); such near-tie dots go through the integer accumulator and every score must
    # still be the oracle's, bit for bit
    g = torch.Generator().manual_seed(11)
    q = (torch.randn(1, 16, 64, 128, generator=g) ** 3).bfloat16()
    k = (torch.randn(1, 1024, 128, generator=g) ** 3).bfloat16()
    w = torch.randn(1, 16, 64, generator=g) / 8
    print("[case] scores outside the double-precision range", flush=True)
    got, st = _scores_gpu(q, k, w, True, 1024 - 16)
    want = _oracle_scores(q, k, w, True, 1024 - 16)
    mism = int((got.view(np.uint32) != want.view(np.uint32)).sum())
    print(f"[info] integer-accumulator dots {int(st[1])}, mismatching scores {mism}", flush=True)
    assert st[1] > 0
    assert mism == 0


def _extreme_rows(rng, n, D):
    """Rows of bf16 bit patterns with extreme dynamic range: normals from 2^-126 to 2^120, subnormals, zeros,
    exact cancellation and near-midpoint sums."""
    rows_q, rows_k = [], []
    for i in range(n):
        kind = i % 6
        if kind == 0:  # any exponent
            q = rng.choice([-1.0, 1.0], D) * (1 + rng.random(D)) * 2.0 ** rng.integers(-126, 60, D)
            k = rng.choice([-1.0, 1.0], D) * (1 + rng.random(D)) * 2.0 ** rng.integers(-126, 60, D)
        elif kind == 1:  # bf16 subnormals next to normals
            q = rng.standard_normal(D) * 2.0 ** rng.integers(-140, -120, D)
            k = rng.standard_normal(D) * 2.0 ** rng.integers(-10, 10, D)
        elif kind == 2:  # exact cancellation: the result is 0 or one tiny product
            q = rng.standard_normal(D) * 2.0 ** rng.integers(-20, 20, D)
            k = rng.standard_normal(D)
            q[D // 2:] = -q[:D // 2]
            k[D // 2:] = k[:D // 2]
            q[-1] = 2.0 ** -100 * rng.choice([0.0, 1.0])
        elif kind == 3:  # a bf16 midpoint from large terms, decided by a term 2^-90 times smaller
            q = np.zeros(D)
            k = np.zeros(D)
            q[0], k[0] = 1.0, 1.0
            q[1], k[1] = 2.0 ** -8, 1.0
            q[2], k[2] = rng.choice([-1.0, 1.0]) * 2.0 ** -50, 2.0 ** -48
        elif kind == 4:  # results beyond the bf16 range (infinity) and just inside it
            q = rng.choice([-1.0, 1.0], D) * 2.0 ** rng.integers(55, 64, D)
            k = np.abs(q) * np.sign(q) * rng.choice([0.5, 1.0], D)
        else:  # results in the bf16 subnormal range
            q = rng.standard_normal(D) * 2.0 ** -70
            k = rng.standard_normal(D) * 2.0 ** -62
        rows_q.append(q)
        rows_k.append(k)
    f = lambda x: torch.from_numpy(np.asarray(x, np.float32)).bfloat16()
    return f(np.stack(rows_q)), f(np.stack(rows_k))


@pytest.mark.parametrize("D", [128, 64])
@pytest.mark.parametrize("parts", [2, 4])
def test_exact_dot_integer_accumulator(device, D, parts):
    # the integer-accumulator exact dot (the path beyond the double-precision spans) against the oracle's
    # big-integer dot, on rows of extreme dynamic range, subnormals, exact cancellation and overflow
    rng = np.random.default_rng(D + parts)
    q, k = _extreme_rows(rng, 600, D)
    print(f"[case] integer-accumulator exact dot D={D} parts={parts}", flush=True)
    qd, kd = q.to(device), k.to(device)
    out = torch.empty(q.shape[0], dtype=torch.int16, device=device)
    _lib.check(_lib.load().ks_dbg_exact_dot_wide(qd.data_ptr(), kd.data_ptr(), out.data_ptr(), q.shape[0], D, parts,
                                                 torch.cuda.current_stream().cuda_stream), "exact dot")
    got = out.cpu().numpy().view(np.uint16)
    qb, kb = _u16(q), _u16(k)
    want = np.array([oracle.dot_exact(qb[i], kb[i]) for i in range(q.shape[0])], np.uint16)
    np.testing.assert_array_equal(got, want)


def _adversarial_key_pair():
    """Key 1's dot with the query is a dot whose MFMA accumulation lands above the bf16 midpoint 1 + 2^-8
    while the exact value lies below it (tests/mfma_model.py: the earlier constant 3 certified the wrong
    value); key 0's dot is exactly 1.0.  Exactly, both score alike and key 0 ranks first."""
    from tests.test_mfma_model import adversarial_rows
    qb, kb = adversarial_rows(22)
    q = torch.from_numpy(qb.view(np.int16)).view(torch.bfloat16)
    k1 = torch.from_numpy(kb.view(np.int16)).view(torch.bfloat16)
    k0 = torch.zeros(128, dtype=torch.bfloat16)
    k0[0] = 1.0  # q[0] = 1: dot exactly 1
    return q, k0, k1


def test_scores_adversarial_accumulation(device):
    q1, k0, k1 = _adversarial_key_pair()
    g = torch.Generator().manual_seed(5)
    S, H, T = 4, 64, 64
    q = torch.randn(1, S, H, 128, generator=g).bfloat16()
    q[0, :, :] = q1  # every head of query 0: the adversarial row
    k = torch.randn(1, T, 128, generator=g).bfloat16()
    k[0, 0], k[0, 1] = k0, k1
    w = (torch.rand(1, S, H, generator=g) + 0.5) / 8
    print("[case] scores adversarial accumulation", flush=True)
    got, st = _scores_gpu(q, k, w, False, 0)
    want = _oracle_scores(q, k, w, False, 0)
    np.testing.assert_array_equal(got.view(np.uint32), want.view(np.uint32))
    assert got[0, 0, 0] == got[0, 0, 1]  # the two keys tie exactly


@pytest.mark.parametrize("H", [16, 64])
def test_scores_adversarial_accumulation_64_dim(device, H):
    # the 64-dim adversarial row (its MFMA accumulation rounds past the bf16 midpoint) through the public exact
    # score entry, which takes the 64-dim constant: scores bit-exact against the oracle, both weight formats
    from tests.test_mfma_model import adversarial_rows
    qb, kb = adversarial_rows(13, 64)
    q1 = torch.from_numpy(qb.view(np.int16)).view(torch.bfloat16)
    k1 = torch.from_numpy(kb.view(np.int16)).view(torch.bfloat16)
    g = torch.Generator().manual_seed(7)
    S, T = 4, 96
    q = torch.randn(1, S, H, 64, generator=g).bfloat16()
    q[0, 0, :] = q1
    k = torch.randn(1, T, 64, generator=g).bfloat16()
    k[0, 0] = 0
    k[0, 0, 0] = 1.0  # dot with q1 exactly 1
    k[0, 1] = k1
    print(f"[case] scores adversarial accumulation D=64 H={H}", flush=True)
    for w in ((torch.rand(1, S, H, generator=g) + 0.5) / 8, ((torch.rand(1, S, H, generator=g) + 0.5) / 8).bfloat16()):
        got = ops.indexer_scores(q.to(device), k.to(device), w.to(device), False, 0, 1).cpu().numpy()
        want = _oracle_scores(q, k, w, False, 0)
        np.testing.assert_array_equal(got.view(np.uint32), want.view(np.uint32))


@pytest.mark.parametrize("path", [1, 2])
def test_indexer_adversarial_accumulation(device, path):
    # the same pair inside the fused indexer (no RoPE, so the rows stay as constructed): exact scores tie,
    # so key 0 must come first, on the exact path and on the bounded path (recomputation in the top-k)
    q1, k0, k1 = _adversarial_key_pair()
    g = torch.Generator().manual_seed(6)
    S, H, T = 8, 64, 512
    q = torch.randn(1, S, H, 128, generator=g).bfloat16() * 0.25
    q[0, :, :] = q1
    k = torch.randn(1, T, 128, generator=g).bfloat16() * 0.25
    k[0, 0], k[0, 1] = k0, k1
    w = (torch.rand(1, S, H, generator=g) + 0.5) / 8
    print(f"[case] indexer adversarial accumulation path={path}", flush=True)
    B = 1
    qd, kd, wd = q.to(device), k.to(device), w.to(device)
    ws = torch.empty(ops.indexer_workspace_size(B, S, H, 128, T), dtype=torch.uint8, device=device)
    out = torch.empty(B, S, 16, dtype=torch.int32, device=device)
    rc = _lib.load().ks_dbg_indexer(qd.data_ptr(), kd.data_ptr(), wd.data_ptr(), 0, None, 0, 0, 0, 0, 16, 0, 0, 1, 0,
                                    out.data_ptr(), 0, B, S, H, 128, T, T, ws.data_ptr(), ws.numel(),
                                    torch.cuda.current_stream().cuda_stream, BOUND_C, None, path)
    _lib.check(rc, "ks_dbg_indexer")
    got = out.cpu().numpy().astype(np.int64)
    want = oracle.indexer(_u16(q), _u16(k), w.numpy(), np.zeros((1, 1, 2), np.float32), 16, False, 0, 1, 0, 0, 0,
                          False)
    np.testing.assert_array_equal(got, want)
    assert got[0, 0, 0] == 0 and got[0, 0, 1] == 1


def test_scores_norms_beyond_overflow_guard(device):
    # rows whose norm product reaches 2^126 (the MFMA could overflow): every dot of such a wave is
    # recomputed exactly; sparse rows keep the exact dots finite
    g = torch.Generator().manual_seed(9)
    S, H, T = 3, 16, 96
    q = torch.zeros(1, S, H, 128)
    k = torch.randn(1, T, 128, generator=g)
    idx = torch.randint(0, 128, (S, H, 3), generator=g)
    for s in range(S):
        for h in range(H):
            q[0, s, h, idx[s, h]] = torch.randn(3, generator=g) * 2.0 ** 62
    k[0, ::7] = k[0, ::7] * 2.0 ** 62
    q, k = q.bfloat16(), k.bfloat16()
    w = (torch.rand(1, S, H, generator=g) + 0.5) * 2.0 ** -30
    print("[case] scores beyond the overflow guard", flush=True)
    got, st = _scores_gpu(q, k, w, False, 0)
    want = _oracle_scores(q, k, w, False, 0)
    np.testing.assert_array_equal(got.view(np.uint32), want.view(np.uint32))


@pytest.mark.parametrize("cfg", [2, 4])
def test_indexer_config_bit_exact(device, cfg):
    w = workloads.CONFIGS[cfg]("cpu")
    t, p = w.tensors, w.params
    print(f"[case] indexer config {cfg}", flush=True)
    d = {n: v.to(device) for n, v in t.items()}
    got = ops.indexer(d["q"], d["k"], d["w"], d["freqs"], p["k_top"], p["causal"], p["start_pos"], p["ratio"],
                      p["offset"], p["rope_start"], p["rope_dim"], p["rope_k"])
    torch.cuda.synchronize()
    want = oracle.indexer(_u16(t["q"]), _u16(t["k"]), t["w"].numpy(), t["freqs"].numpy(), p["k_top"], p["causal"],
                          p["start_pos"], p["ratio"], p["offset"], p["rope_start"], p["rope_dim"], p["rope_k"])
    g = got.cpu().numpy().astype(np.int64)
    assert g.shape == want.shape
    mism = int((g != want).sum())
    assert mism == 0, f"{mism} mismatching indices"


def test_indexer_scores_config2_bit_exact(device):
    w = workloads.CONFIGS[2]("cpu")
    t, p = w.tensors, w.params
    qr = oracle.rope_bf16(_u16(t["q"]), t["freqs"].numpy(), 0, 64, p["start_pos"])
    kr = oracle.rope_bf16(_u16(t["k"]).reshape(1, 4096, 1, 128), t["freqs"].numpy(), 0, 64, 0).reshape(1, 4096, 128)
    q = torch.from_numpy(qr.view(np.int16)).view(torch.bfloat16)
    k = torch.from_numpy(kr.view(np.int16)).view(torch.bfloat16)
    print("[case] scores config 2", flush=True)
    got, st = _scores_gpu(q, k, t["w"], True, p["start_pos"])
    want = oracle.indexer_scores(qr, kr, t["w"].numpy(), True, p["start_pos"])
    np.testing.assert_array_equal(got.view(np.uint32), want.view(np.uint32))
    print(f"[info] exact recomputations: {int(st[0])} of {128 * 64 * 4096} dots", flush=True)
    assert st[1] == 0


def test_indexer_baseline_semantics_ratio4_bf16_weights(device):
    # the reference's own example semantics: start_pos = 0 masking with compress ratio 4, bf16 weights,
    # RoPE on the trailing dims of q only, int64 output with -1 and offset
    g = torch.Generator().manual_seed(5)
    B, S, H, T = 2, 64, 16, 16
    q = torch.randn(B, S, H, 128, generator=g).bfloat16()
    k = torch.randn(B, T, 128, generator=g).bfloat16()
    w = (torch.randn(B, S, H, generator=g) * 0.1).bfloat16()
    tab = workloads.freqs_table(32, 256)
    print("[case] indexer baseline semantics", flush=True)
    got = ops.indexer(q.to(device), k.to(device), w.to(device), tab.to(device), 128, True, 0, 4, 9, 96, 32, False,
                      out_dtype=torch.int64)
    torch.cuda.synchronize()
    want = oracle.indexer(_u16(q), _u16(k), _u16(w), tab.numpy(), 128, True, 0, 4, 9, 96, 32, False)
    np.testing.assert_array_equal(got.cpu().numpy(), want)


def _indexer_vs_oracle(q, k, w, tab, k_top, causal, start_pos, ratio, offset, rs, rd, rope_k, T, cache_rows=None):
    """ks_indexer (one RoPE/statistics launch over q and every batch's k, scores, top-k) vs the oracle.
    cache_rows > T gives k as a batch-strided view of a larger cache (batch stride cache_rows rows)."""
    B, S, H, D = q.shape
    kd = k.to("cuda")
    if cache_rows is not None:
        cache = torch.zeros(B, cache_rows, D, dtype=torch.bfloat16, device="cuda")
        cache[:, :T] = kd
        kd = cache[:, :T]
    got = ops.indexer(q.to("cuda"), kd, w.to("cuda"), tab.to("cuda"), k_top, causal, start_pos, ratio, offset, rs,
                      rd, rope_k)
    torch.cuda.synchronize()
    wn = _u16(w) if w.dtype == torch.bfloat16 else w.numpy()
    want = oracle.indexer(_u16(q), _u16(k), wn, tab.numpy(), k_top, causal, start_pos, ratio, offset, rs, rd, rope_k)
    np.testing.assert_array_equal(got.cpu().numpy().astype(np.int64), want)


@pytest.mark.parametrize("D,rs,rd,rope_k,w_bf16,cache_rows", [(128, 0, 64, True, False, 700),
                                                              (64, 32, 32, False, True, None),
                                                              (128, 64, 64, True, True, 301),
                                                              (128, 0, 0, False, False, 512)])
def test_indexer_prep_layouts(device, D, rs, rd, rope_k, w_bf16, cache_rows):
    g = torch.Generator().manual_seed(D + rs + rd)
    B, S, H, T = 2, 9, 64, 300
    q = torch.randn(B, S, H, D, generator=g).bfloat16()
    k = torch.randn(B, T, D, generator=g).bfloat16()
    w = torch.randn(B, S, H, generator=g) / 8
    if w_bf16:
        w = w.bfloat16()
    tab = workloads.freqs_table(max(rd, 2), 512)
    print(f"[case] indexer D={D} rope=[{rs},{rs + rd}) rope_k={rope_k} w_bf16={w_bf16} cache_rows={cache_rows}",
          flush=True)
    _indexer_vs_oracle(q, k, w, tab, 64, True, T - S, 1, 0, rs, rd, rope_k, T, cache_rows)


@pytest.mark.parametrize("dist", ["scaled", "tiny", "midpoints"])
def test_indexer_adversarial(device, dist):
    g = torch.Generator().manual_seed(21)
    q = torch.randn(1, 16, 64, 128, generator=g)
    k = torch.randn(1, 1024, 128, generator=g)
    if dist == "scaled":
        q = q * torch.exp2(torch.randint(-8, 9, (1, 16, 64, 1), generator=g).float())
        k = k * torch.exp2(torch.randint(-8, 9, (1, 1024, 1), generator=g).float())
    elif dist == "tiny":
        q = q * torch.exp2(torch.randint(-30, 1, q.shape, generator=g).float())
    else:  # integer inputs: many dots on exact bf16 midpoints before RoPE, many tied scores
        q = torch.randint(-3, 4, q.shape, generator=g).float()
        k = torch.randint(-3, 4, k.shape, generator=g).float()
    q, k = q.bfloat16(), k.bfloat16()
    w = torch.randn(1, 16, 64, generator=g) / 8
    tab = workloads.freqs_table(64, 2048)
    print(f"[case] indexer adversarial {dist}", flush=True)
    _indexer_vs_oracle(q, k, w, tab, 256, True, 1024 - 16, 1, 0, 0, 64, True, 1024)


def _dbg_indexer(q, k, w, tab, k_top, causal, start_pos, path, bound_c=None, T=None):
    """ks_dbg_indexer: path 1 = exact scores, 2 = bounded scores with exact recomputation in the top-k.
    Returns (indices, [exact dot recomputations, dots outside the exact range])."""
    B, S, H, D = q.shape
    T = k.shape[1] if T is None else T
    qd, kd, wd, td = q.to("cuda"), k.to("cuda"), w.to("cuda"), tab.to("cuda")
    ws = torch.empty(ops.indexer_workspace_size(B, S, H, D, T), dtype=torch.uint8, device="cuda")
    kk = min(k_top, T)
    out = torch.empty(B, S, kk, dtype=torch.int32, device="cuda")
    st = torch.zeros(2, dtype=torch.int32, device="cuda")
    rc = _lib.load().ks_dbg_indexer(qd.data_ptr(), kd.data_ptr(), wd.data_ptr(), 0, td.data_ptr(), tab.shape[0], 0, 64,
                                    1, k_top, 1 if causal else 0, start_pos, 1, 0, out.data_ptr(), 0, B, S, H, D, T, T,
                                    ws.data_ptr(), ws.numel(), torch.cuda.current_stream().cuda_stream,
                                    BOUND_C if bound_c is None else bound_c, st.data_ptr(), path)
    _lib.check(rc, "ks_dbg_indexer")
    torch.cuda.synchronize()
    return out.cpu().numpy().astype(np.int64), st.cpu().numpy()


@pytest.mark.parametrize("S,T,k_top,start_pos", [(24, 3000, 64, 2976), (7, 700, 700, 0), (33, 1500, 512, 4000)])
def test_indexer_bounded_recompute_everything(device, S, T, k_top, start_pos):
    # a huge interval constant makes every positive dot a near tie: every score carries a bound, every key
    # reaching the threshold is recomputed (the list is refilled in several batches), and the exact dots go
    # through the double-precision path; the result must still be the oracle's, bit for bit
    g = torch.Generator().manual_seed(S + T)
    q = torch.randn(1, S, 64, 128, generator=g).bfloat16()
    k = torch.randn(1, T, 128, generator=g).bfloat16()
    w = torch.randn(1, S, 64, generator=g) / 8
    tab = workloads.freqs_table(64, max(T, start_pos + S) + 1)
    causal = start_pos < 4000
    sp = start_pos if causal else 0
    print(f"[case] bounded recompute-all S={S} T={T} k={k_top} causal={causal}", flush=True)
    got, st = _dbg_indexer(q, k, w, tab, k_top, causal, sp, 2, bound_c=1e6)
    want = oracle.indexer(_u16(q), _u16(k), w.numpy(), tab.numpy(), k_top, causal, sp, 1, 0, 0, 64, True)
    np.testing.assert_array_equal(got, want)
    assert st[0] > 0 and st[1] == 0


def test_indexer_bounded_norms_beyond_overflow_guard(device):
    # the bounded path on rows whose norm products reach 2^126 (the MFMA could overflow): the score kernel gives
    # such waves infinite bounds, and the recomputation takes every dot of a tile whose key block reaches the
    # guard as a near tie and computes it exactly
    g = torch.Generator().manual_seed(19)
    S, T = 4, 160
    q = torch.zeros(1, S, 64, 128)
    idx = torch.randint(0, 128, (S, 64, 3), generator=g)
    for s in range(S):
        for h in range(64):
            q[0, s, h, idx[s, h]] = torch.randn(3, generator=g) * 2.0 ** 62
    k = torch.randn(1, T, 128, generator=g)
    k[0, ::7] = k[0, ::7] * 2.0 ** 62
    q, k = q.bfloat16(), k.bfloat16()
    w = (torch.rand(1, S, 64, generator=g) + 0.5) * 2.0 ** -30
    tab = workloads.freqs_table(64, T + 1)
    print("[case] bounded path beyond the overflow guard", flush=True)
    got, st = _dbg_indexer(q, k, w, tab, 32, False, 0, 2)
    want = oracle.indexer(_u16(q), _u16(k), w.numpy(), tab.numpy(), 32, False, 0, 1, 0, 0, 64, True)
    np.testing.assert_array_equal(got, want)
    assert st[0] > 0


def _bounded_scores_gpu(q, k, w, start_pos):
    """Bound-mode score kernel through the diagnostic export (causal): returns (scores, bounds)."""
    qd, kd, wd = q.to("cuda"), k.to("cuda"), w.to("cuda")
    (qn, qs), (kn, ks_) = ops.indexer_row_stats(qd), ops.indexer_row_stats(kd)
    B, S, H, D = q.shape
    T = k.shape[1]
    lib = _lib.load()
    out = torch.empty(B, S, T, dtype=torch.float32, device="cuda")
    bnd = torch.empty(B, S, T, dtype=torch.float32, device="cuda")
    kmax = torch.empty(B, (T + 255) // 256, dtype=torch.float32, device="cuda")
    part = torch.zeros(lib.ks_dbg_topk_bounded_slots(B * S, T), dtype=torch.int64, device="cuda")
    rc = lib.ks_dbg_indexer_scores_bounded(qd.data_ptr(), kd.data_ptr(), wd.data_ptr(), qn.data_ptr(), qs.data_ptr(),
                                           kn.data_ptr(), ks_.data_ptr(), out.data_ptr(), bnd.data_ptr(),
                                           kmax.data_ptr(), part.data_ptr(), B, S, T, 1, start_pos,
                                           torch.cuda.current_stream().cuda_stream)
    _lib.check(rc, "ks_dbg_indexer_scores_bounded")
    torch.cuda.synchronize()
    return out.cpu().numpy(), bnd.cpu().numpy()


@pytest.mark.parametrize("dist,S,T", [("normal", 16, 768), ("scaled", 16, 768), ("midpoints", 16, 768),
                                      ("heavy", 16, 768), ("adversarial", 16, 768), ("normal", 136, 4096)])
def test_bounded_scores_contain_exact(device, dist, S, T):
    # the bound-mode score kernel's contract, checked score by score against the oracle's exact scores on the
    # valid (unmasked) columns: U >= 0, the stored score exact (bit for bit) where U = 0, |exact - S| <= U elsewhere.  The last
    # shape's grid (17 query groups x 16 key blocks) exceeds one round of the GPU.
    g = torch.Generator().manual_seed(41 + S)
    q = torch.randn(1, S, 64, 128, generator=g)
    k = torch.randn(1, T, 128, generator=g)
    if dist == "scaled":
        q = q * torch.exp2(torch.randint(-8, 9, (1, S, 64, 1), generator=g).float())
        k = k * torch.exp2(torch.randint(-8, 9, (1, T, 1), generator=g).float())
    elif dist == "midpoints":
        q = torch.randint(-3, 4, q.shape, generator=g).float()
        k = torch.randint(-3, 4, k.shape, generator=g).float()
    elif dist == "heavy":
        q, k = q ** 3, k ** 3
        q = torch.where(q.abs() < 1e-3, torch.zeros_like(q), q)
        k = torch.where(k.abs() < 1e-3, torch.zeros_like(k), k)
    q, k = q.bfloat16(), k.bfloat16()
    w = torch.randn(1, S, 64, generator=g) / 8
    if dist == "adversarial":  # the MFMA-accumulation pair of test_scores_adversarial_accumulation in query 0
        q1, k0, k1 = _adversarial_key_pair()
        q[0, 0, :] = q1
        k[0, T - 40], k[0, T - 39] = k0, k1
        w[0, 0] = w[0, 0].abs() + 0.0625
    start_pos = T - S
    print(f"[case] bounded scores contain exact {dist} S={S} T={T}", flush=True)
    got, u = _bounded_scores_gpu(q, k, w, start_pos)
    want = _oracle_scores(q, k, w, True, start_pos)
    valid = np.isfinite(want)  # the causal mask; masked columns hold -inf and no bound (never read)
    assert np.array_equal(np.isfinite(got), valid) and (got[~valid] == -np.inf).all()
    assert (u[valid] >= 0).all()
    tight = valid & (u == 0)
    np.testing.assert_array_equal(got[tight].view(np.uint32), want[tight].view(np.uint32))
    loose = valid & (u > 0) & np.isfinite(u)
    err = np.abs(want[loose].astype(np.float64) - got[loose].astype(np.float64))
    assert (err <= u[loose].astype(np.float64)).all()
    print(f"[info] {int(loose.sum())} of {int(valid.sum())} scores bounded (U > 0)", flush=True)


@pytest.mark.parametrize("dist", ["normal", "scaled", "midpoints"])
def test_indexer_bounded_equals_exact_path(device, dist):
    # the two score paths select identical indices (and both equal the oracle's)
    g = torch.Generator().manual_seed(31)
    q = torch.randn(2, 20, 64, 128, generator=g)
    k = torch.randn(2, 2048, 128, generator=g)
    if dist == "scaled":
        q = q * torch.exp2(torch.randint(-6, 7, (2, 20, 64, 1), generator=g).float())
        k = k * torch.exp2(torch.randint(-6, 7, (2, 2048, 1), generator=g).float())
    elif dist == "midpoints":
        q = torch.randint(-3, 4, q.shape, generator=g).float()
        k = torch.randint(-3, 4, k.shape, generator=g).float()
    q, k = q.bfloat16(), k.bfloat16()
    w = torch.randn(2, 20, 64, generator=g) / 8
    tab = workloads.freqs_table(64, 2048)
    print(f"[case] bounded vs exact path {dist}", flush=True)
    exact, _ = _dbg_indexer(q, k, w, tab, 512, True, 2048 - 20, 1)
    bounded, st = _dbg_indexer(q, k, w, tab, 512, True, 2048 - 20, 2)
    np.testing.assert_array_equal(bounded, exact)
    want = oracle.indexer(_u16(q), _u16(k), w.numpy(), tab.numpy(), 512, True, 2048 - 20, 1, 0, 0, 64, True)
    np.testing.assert_array_equal(bounded, want)
    print(f"[info] bounded path: {int(st[0])} exact dot recomputations", flush=True)


# Rows too few to fill the GPU: column slices for the threshold's bucket counts and several recomputation
# segments per row, appending to one list per row: causal rows whose valid prefix ends inside the first slice
# (later slices and segments empty, masked tail), a prefix ending inside the second slice, slices of unequal
# width (T = 5000), and all-equal scores, whose order is decided by the column alone: every key lands in one
# bucket of the rank store (the merge sort takes over at T = 8192, the list's capacity), and past the capacity
# (T = 9000) the whole-row selection does.
@pytest.mark.parametrize("S,T,k_top,start_pos,causal,zero_q", [(8, 4096, 256, 0, True, False),
                                                              (6, 4096, 256, 1490, True, False),
                                                              (5, 5000, 300, 0, False, False),
                                                              (4, 8192, 512, 0, False, True),
                                                              (3, 9000, 512, 0, False, True)])
def test_indexer_split_topk(device, S, T, k_top, start_pos, causal, zero_q):
    g = torch.Generator().manual_seed(S * T + k_top)
    q = torch.randn(1, S, 64, 128, generator=g)
    if zero_q:
        q = torch.zeros_like(q)
    q = q.bfloat16()
    k = torch.randn(1, T, 128, generator=g).bfloat16()
    w = torch.randn(1, S, 64, generator=g) / 8
    tab = workloads.freqs_table(64, max(T, start_pos + S) + 1)
    print(f"[case] split top-k S={S} T={T} k={k_top} start={start_pos} causal={causal} zero_q={zero_q}", flush=True)
    got, _ = _dbg_indexer(q, k, w, tab, k_top, causal, start_pos, 2)
    want = oracle.indexer(_u16(q), _u16(k), w.numpy(), tab.numpy(), k_top, causal, start_pos, 1, 0, 0, 64, True)
    np.testing.assert_array_equal(got, want)
    if zero_q:
        assert np.array_equal(got[0, 0], np.arange(k_top))


# Grids of several score workgroups per CU: batches, a query count that leaves idle waves in the last
# group, a partial last key block, with and without the XCD tiling of the workgroups (180 per batch is not
# a multiple of 8; 256 is), causal, and rows short enough for the split top-k.
@pytest.mark.parametrize("B,S,T", [(4, 36, 9000), (2, 64, 8100)])
def test_indexer_multi_item_grids(device, B, S, T):
    g = torch.Generator().manual_seed(B * S + T)
    q = torch.randn(B, S, 64, 128, generator=g).bfloat16()
    k = torch.randn(B, T, 128, generator=g).bfloat16()
    w = torch.randn(B, S, 64, generator=g) / 8
    tab = workloads.freqs_table(64, T + 1)
    k_top, start_pos = 300, T - S
    print(f"[case] multi-item grid B={B} S={S} T={T}", flush=True)
    got = ops.indexer(q.to(device), k.to(device), w.to(device), tab.to(device), k_top, True, start_pos, 1, 0, 0, 64,
                      True)
    torch.cuda.synchronize()
    want = oracle.indexer(_u16(q), _u16(k), w.numpy(), tab.numpy(), k_top, True, start_pos, 1, 0, 0, 64, True)
    np.testing.assert_array_equal(got.cpu().numpy().astype(np.int64), want)


@pytest.mark.parametrize("H,D,w_bf16", [(16, 64, True), (64, 128, False), (32, 128, True), (64, 128, True)])
def test_indexer_weight_scale(device, H, D, w_bf16):
    # w_scale (ks_indexer_scaled, the drop-in's weights_proj(x) * scale): the same indices as the weights multiplied
    # by torch first, with a scale that is not a power of two (so the product's rounding matters); 64 heads of 128
    # with fp32 weights take the bounded path, whose recomputation reads the scaled weights too
    g = torch.Generator().manual_seed(H + D + w_bf16)
    B, S, T = 2, 24, 700
    q = torch.randn(B, S, H, D, generator=g).bfloat16().to(device)
    k = torch.randn(B, T, D, generator=g).bfloat16().to(device)
    w = (torch.randn(B, S, H, generator=g) / 8).to(device)
    if w_bf16:
        w = w.bfloat16()
    tab = workloads.freqs_table(64, 1024).to(device)
    scale = 128 ** -0.5 * 48 ** -0.5
    print(f"[case] indexer w_scale H={H} D={D} w_bf16={w_bf16}", flush=True)
    got = ops.indexer(q, k, w, tab, 128, True, T - S, rope_start=0, rope_dim=64, w_scale=scale)
    want = ops.indexer(q, k, (w * scale).contiguous(), tab, 128, True, T - S, rope_start=0, rope_dim=64)
    torch.cuda.synchronize()
    assert torch.equal(got, want)
    # a negative scale selects other keys: the scale is applied, not dropped
    neg = ops.indexer(q, k, w, tab, 128, True, T - S, rope_start=0, rope_dim=64, w_scale=-scale)
    assert torch.equal(neg, ops.indexer(q, k, (w * -scale).contiguous(), tab, 128, True, T - S, rope_start=0,
                                        rope_dim=64))
    assert not torch.equal(neg, want)
    # the torch operator takes the same argument
    tops = _lib.torch_ops()
    got2 = tops.indexer(q, k, w, tab, 128, True, T - S, 1, 0, 0, 64, True, False, None, w_scale=scale)
    assert torch.equal(got2, want)


@pytest.mark.parametrize("D,rs,rd,rope_k,w_bf16,causal", [(64, 32, 32, False, True, True),
                                                         (64, 16, 32, True, False, True),
                                                         (64, 0, 0, False, True, True),
                                                         (128, 0, 64, True, True, True),
                                                         (128, 40, 64, False, False, True),
                                                         (128, 24, 96, True, True, False)])
def test_indexer_16_heads_rope_layouts(device, D, rs, rd, rope_k, w_bf16, causal):
    # the fused indexer at 16 heads (the exact path with its per-dot half-widths): rotated ranges that start inside
    # a 32-element fragment or straddle two, none at all, rotated keys, fp32 and bf16 weights, causal and not (an
    # offset and a start position past zero), bit for bit against the oracle
    g = torch.Generator().manual_seed(D + rs + rd + rope_k)
    B, S, H, T = 2, 40, 16, 700
    q = torch.randn(B, S, H, D, generator=g).bfloat16()
    k = torch.randn(B, T, D, generator=g).bfloat16()
    w = torch.randn(B, S, H, generator=g) / 8
    if w_bf16:
        w = w.bfloat16()
    tab = workloads.freqs_table(max(rd, 2), 1024)
    start = T - S if causal else 123
    print(f"[case] indexer 16 heads D={D} rope=[{rs},{rs + rd}) rope_k={rope_k} w_bf16={w_bf16} causal={causal}",
          flush=True)
    _indexer_vs_oracle(q, k, w, tab, 96, causal, start, 1, 0 if causal else 5, rs, rd, rope_k, T)


@pytest.mark.parametrize("D,rs,rd", [(64, 32, 32), (128, 64, 64)])
def test_indexer_16_heads_split_rows_wide_range(device, D, rs, rd):
    # the fused indexer's exact path with a 32-aligned rotated range: the row preparation writes only q's rotated
    # dims and the score kernel reads the others from the caller's rows.  Cubed normals (row spans past the double-
    # precision paths) send near-tie dots through the wide-range and integer-accumulator recomputations, which read
    # q from memory on both sides of the split; every index must be the oracle's
    g = torch.Generator().manual_seed(D + 7)
    B, S, H, T = 1, 24, 16, 600
    q = (torch.randn(B, S, H, D, generator=g) ** 3).bfloat16()
    k = (torch.randn(B, T, D, generator=g) ** 3).bfloat16()
    w = torch.randn(B, S, H, generator=g) / 8
    tab = workloads.freqs_table(rd, 1024)
    k_top, start = 64, T - S
    qd, kd, wd, td = q.to("cuda"), k.to("cuda"), w.to("cuda"), tab.to("cuda")
    ws = torch.empty(ops.indexer_workspace_size(B, S, H, D, T), dtype=torch.uint8, device="cuda")
    out = torch.empty(B, S, k_top, dtype=torch.int32, device="cuda")
    st = torch.zeros(2, dtype=torch.int32, device="cuda")
    print(f"[case] indexer 16 heads split rows D={D} rope=[{rs},{rs + rd}) cubed normals", flush=True)
    _lib.check(_lib.load().ks_dbg_indexer(qd.data_ptr(), kd.data_ptr(), wd.data_ptr(), 0, td.data_ptr(), tab.shape[0],
                                          rs, rd, 0, k_top, 1, start, 1, 0, out.data_ptr(), 0, B, S, H, D, T, T,
                                          ws.data_ptr(), ws.numel(), torch.cuda.current_stream().cuda_stream,
                                          BOUND_C, st.data_ptr(), 1), "ks_dbg_indexer")
    torch.cuda.synchronize()
    want = oracle.indexer(_u16(q), _u16(k), w.numpy(), tab.numpy(), k_top, True, start, 1, 0, rs, rd, False)
    print(f"[info] exact dots {int(st[0])}, integer-accumulator dots {int(st[1])}", flush=True)
    assert st[1] > 0
    np.testing.assert_array_equal(out.cpu().numpy().astype(np.int64), want)
