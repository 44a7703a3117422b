"""GPU parity of the RaBitQ 1-bit encode / estimate / search against the CPU
oracle: codes, factors, estimates, candidate sets, reranked order and exact
scores are all bit-exact."""
import numpy as np
import pytest
import torch

from oracle import rabitq as orq
from oracle.numerics import f16_bits
from tests.helpers import from_torch

pytestmark = pytest.mark.gpu


def _f16(a_bits: np.ndarray) -> torch.Tensor:
    return torch.from_numpy(a_bits.view(np.int16)).view(torch.float16).cuda()


def _bits(t: torch.Tensor) -> np.ndarray:
    return from_torch(t.view(torch.int16)).view(np.uint16)


def _signs(seed=42):
    s = orq.srht_signs(seed)
    return s, torch.from_numpy(s).cuda()


def test_encode_bit_exact(rng):
    s_np, s_t = _signs(7)
    keys = np.concatenate([
        orq.clustered_unit_keys(rng, 3000, 16),
        f16_bits((rng.standard_normal((500, 128)) * 30).astype(np.float32)),
        np.zeros((2, 128), np.uint16),                                  # zero vector: corr 0
        f16_bits(np.full((1, 128), 60000.0, np.float32)),               # near fp16 max
        f16_bits(np.where(np.arange(128) == 5, 1.0, 0.0)[None].astype(np.float32)),
    ])
    codes, fac = orq.encode(keys, s_np)
    gc, gf = __import__("zoomkv_revision_amd.rabitq", fromlist=["x"]).rabitq_encode(_f16(keys), s_t)
    assert np.array_equal(from_torch(gc), codes)
    assert np.array_equal(_bits(gf), fac)


@pytest.mark.parametrize("n", [1, 63, 64, 65, 130])
def test_encode_tile_edges_and_nonfinite_rows(rng, n):
    """A partial tile of 64 rows, and rows with infinities and NaNs: codes as
    the oracle's (y >= 0 is false for a NaN), factors equal or both NaN."""
    from zoomkv_revision_amd.rabitq import rabitq_encode
    s_np, s_t = _signs(11)
    x = (rng.standard_normal((n, 128)) * 3).astype(np.float32)
    x[0, 17] = np.inf                                        # one infinity: no NaN in y
    if n > 60:
        x[1, 3], x[1, 90] = -np.inf, np.inf                  # two: some y are NaN
        x[2, [5, 6, 7, 101]] = np.inf
        x[3, 64] = np.nan
        x[4, 64], x[4, 9] = np.nan, -np.inf
        x[n - 1] = -0.0
    keys = f16_bits(x)
    with np.errstate(invalid="ignore"):
        codes, fac = orq.encode(keys, s_np)
    gc, gf = rabitq_encode(_f16(keys), s_t)
    assert np.array_equal(from_torch(gc), codes)
    got, want = _bits(gf), fac
    nan = np.isnan(want.view(np.float16))
    assert np.array_equal(np.isnan(got.view(np.float16)), nan)
    assert np.array_equal(got[~nan], want[~nan])


def test_encode_strided_rows(rng):
    from zoomkv_revision_amd.rabitq import rabitq_encode
    s_np, s_t = _signs(3)
    big = orq.clustered_unit_keys(rng, 2 * 700, 8).reshape(700, 256)   # rows of 256, use first 128
    t = _f16(big)[:, :128]
    gc, gf = rabitq_encode(t, s_t)
    codes, fac = orq.encode(np.ascontiguousarray(big[:, :128]), s_np)
    assert np.array_equal(from_torch(gc), codes) and np.array_equal(_bits(gf), fac)


def test_estimate_bit_exact(rng):
    from zoomkv_revision_amd.rabitq import rabitq_encode, rabitq_estimate
    s_np, s_t = _signs()
    keys = orq.clustered_unit_keys(rng, 5000, 32)
    qs = orq.clustered_unit_keys(rng, 7, 32)
    ck, fk = orq.encode(keys, s_np)
    cq, fq = orq.encode(qs, s_np)
    got = rabitq_estimate(*rabitq_encode(_f16(qs), s_t), *rabitq_encode(_f16(keys), s_t))
    ref = orq.estimate(cq, fq, ck, fk)
    assert np.array_equal(from_torch(got).view(np.uint32), ref.view(np.uint32))


def _check_search(rng, P, Q, N, topk, seed=42, dup=None):
    from zoomkv_revision_amd.rabitq import rabitq_encode, rabitq_search
    s_np, s_t = _signs(seed)
    keys = [orq.clustered_unit_keys(rng, N if dup is None else dup, 16) for _ in range(P)]
    if dup is not None:               # many identical keys: ties everywhere
        keys = [k[rng.integers(0, dup, size=N)] for k in keys]
    qs = [orq.clustered_unit_keys(rng, Q, 16) for _ in range(P)]
    kt = _f16(np.stack(keys))
    codes, fac = rabitq_encode(kt, s_t)
    cand, fidx, fsc = rabitq_search(_f16(np.stack(qs)), kt, codes, fac, s_t, topk)
    cand, fidx, fsc = from_torch(cand), from_torch(fidx), from_torch(fsc)
    for p in range(P):
        ck, fk = orq.encode(keys[p], s_np)
        rc, ri, rs = orq.search(qs[p], keys[p], ck, fk, s_np, topk)
        assert np.array_equal(cand[p], rc), f"pool {p}: candidate set"
        assert np.array_equal(fidx[p], ri), f"pool {p}: reranked order"
        assert np.array_equal(fsc[p].view(np.uint32), rs.view(np.uint32)), f"pool {p}: exact scores"


@pytest.mark.parametrize("P,Q,N,topk", [
    (1, 4, 20000, 256),        # 3 slices, last one partial
    (2, 3, 8192, 256),         # exactly one slice
    (1, 2, 8192 + 100, 256),   # last slice shorter than topk: padded candidates
    (1, 3, 300, 256),          # one slice, radix path
    (1, 2, 256, 256),          # topk == n
    (3, 2, 5000, 1),           # topk 1
    (1, 2, 40000, 100),        # non power-of-two topk
    (1, 1, 4000, 1000),        # topk near the limit
])
def test_search_bit_exact(rng, P, Q, N, topk):
    _check_search(rng, P, Q, N, topk)


def test_search_ties_go_to_lower_index(rng):
    _check_search(rng, 1, 4, 30000, 256, dup=40)


@pytest.mark.parametrize("P,Q,N,topk", [
    (1, 2, 65536, 1024),       # 8 slices x topk 1024 = the 8192-candidate limit
    (1, 3, 3000, 256),
    (2, 2, 2048, 300),
])
def test_search_more_sizes(rng, P, Q, N, topk):
    _check_search(rng, P, Q, N, topk)


@pytest.mark.parametrize("P,Q,N,topk", [
    (1, 3, 16384, 100),        # filter path, 64 lists: one select pass
    (2, 2, 200000, 256),       # 782 lists: 8 passes
    (1, 2, 524288, 300),       # 2048 lists: 16 passes, the filter path's largest pool
    (1, 2, 600000, 64),        # beyond it: the sliced path
])
def test_search_filter_path_passes(rng, P, Q, N, topk):
    _check_search(rng, P, Q, N, topk)


def test_search_all_keys_equal(rng):
    """Every key identical: every estimate ties, and the top-k are the lowest
    indices."""
    _check_search(rng, 1, 2, 20000, 256, dup=1)


def test_search_few_planted_winners(rng):
    """The query itself planted at 32 spread positions: those 32 keys lead the
    candidates, the other 224 come from the clustered rest."""
    from zoomkv_revision_amd.rabitq import rabitq_encode, rabitq_search
    s_np, s_t = _signs()
    n, topk = 50000, 256
    keys = orq.clustered_unit_keys(rng, n, 16)
    qs = orq.clustered_unit_keys(rng, 1, 16)
    keys[[s * n // 2048 for s in range(32)]] = qs[0]
    kt = _f16(keys)
    codes, fac = rabitq_encode(kt, s_t)
    cand, fidx, fsc = (from_torch(t) for t in rabitq_search(_f16(qs), kt, codes, fac, s_t, topk))
    ck, fk = orq.encode(keys, s_np)
    rc, ri, rs = orq.search(qs, keys, ck, fk, s_np, topk)
    assert set([s * n // 2048 for s in range(32)]) <= set(cand[0].tolist())
    assert np.array_equal(cand, rc) and np.array_equal(fidx, ri)
    assert np.array_equal(fsc.view(np.uint32), rs.view(np.uint32))


def test_search_into_preallocated_outputs(rng):
    """out= writes the same bits into the caller's tensors, call after call."""
    from zoomkv_revision_amd.rabitq import rabitq_encode, rabitq_search, search_workspace
    _, s_t = _signs()
    n, nq, topk = 40000, 3, 128
    kt = _f16(orq.clustered_unit_keys(rng, n, 16))
    qt = _f16(orq.clustered_unit_keys(rng, nq, 16))
    codes, fac = rabitq_encode(kt, s_t)
    ref = rabitq_search(qt, kt, codes, fac, s_t, topk)
    ws = search_workspace(1, nq, n, topk, qt.device)
    outs = (torch.full((nq, topk), -7, dtype=torch.int64, device=qt.device),
            torch.full((nq, topk), -7, dtype=torch.int64, device=qt.device),
            torch.full((nq, topk), float("nan"), device=qt.device))
    for _ in range(2):
        got = rabitq_search(qt, kt, codes, fac, s_t, topk, workspace=ws, out=outs)
        for a, b, o in zip(got, ref, outs):
            assert a.data_ptr() == o.data_ptr()
            assert torch.equal(a.view(torch.int32) if a.dtype == torch.float32 else a,
                               b.view(torch.int32) if b.dtype == torch.float32 else b)


def test_search_c4_full_size(rng):
    """131072 clustered unit keys, 64 queries, top-256;
    8 of the 64 queries checked against the oracle, all 64 against invariants."""
    from zoomkv_revision_amd.rabitq import rabitq_encode, rabitq_search
    s_np, s_t = _signs()
    keys = orq.clustered_unit_keys(rng, 131072, 64)
    qs = orq.clustered_unit_keys(rng, 64, 64)
    kt = _f16(keys)
    codes, fac = rabitq_encode(kt, s_t)
    cand, fidx, fsc = (from_torch(t) for t in rabitq_search(_f16(qs), kt, codes, fac, s_t, 256))
    ck, fk = orq.encode(keys, s_np)
    assert np.array_equal(from_torch(codes), ck)
    for i in range(0, 64, 8):
        rc, ri, rs = orq.search(qs[i:i + 1], keys, ck, fk, s_np, 256)
        assert np.array_equal(cand[i], rc[0]) and np.array_equal(fidx[i], ri[0])
        assert np.array_equal(fsc[i].view(np.uint32), rs[0].view(np.uint32))
    assert np.all(np.diff(cand, axis=-1) > 0)
    assert np.all(np.diff(fsc, axis=-1) <= 0)
    assert np.array_equal(np.sort(fidx, axis=-1), cand)


@pytest.mark.parametrize("N,topk", [(131072, 256), (20000, 256)])
def test_search_query_encode_in_workspace(rng, N, topk):
    """The search encodes its queries into the workspace's first two regions
    (codes [P*Q, 16] at byte 0, factors [P*Q, 2] fp16 at the next 256-byte
    boundary).  Both paths' encodes equal the oracle's, bits included: the
    filter path's prep kernel encodes across the lanes of one wave, and a
    wrong factor would not show in the results (it scales every estimate of
    its query alike)."""
    from zoomkv_revision_amd.rabitq import rabitq_encode, rabitq_search, search_workspace
    s_np, s_t = _signs()
    P, Q = 2, 5
    keys = orq.clustered_unit_keys(rng, N, 16)
    qs = np.concatenate([orq.clustered_unit_keys(rng, P * Q - 2, 16),
                         f16_bits((rng.standard_normal((1, 128)) * 300).astype(np.float32)),
                         np.zeros((1, 128), np.uint16)])                    # large norm; zero vector
    kt = _f16(np.stack([keys, keys]))
    codes, fac = rabitq_encode(kt, s_t)
    ws = search_workspace(P, Q, N, topk, "cuda")
    ws.fill_(0xAB)
    rabitq_search(_f16(qs.reshape(P, Q, 128)), kt, codes, fac, s_t, topk, workspace=ws)
    torch.cuda.synchronize()
    w = from_torch(ws)
    off = (P * Q * 16 + 255) // 256 * 256
    cq, fq = orq.encode(qs, s_np)
    assert np.array_equal(w[:P * Q * 16].reshape(P * Q, 16), cq)
    assert np.array_equal(w[off:off + P * Q * 4].view(np.uint16).reshape(P * Q, 2), fq)


def test_search_rejects_bad_sizes():
    from zoomkv_revision_amd.rabitq import rabitq_search
    s = torch.ones(128, device="cuda")
    k = torch.zeros(100, 128, dtype=torch.float16, device="cuda")
    c = torch.zeros(100, 16, dtype=torch.uint8, device="cuda")
    f = torch.zeros(100, 2, dtype=torch.float16, device="cuda")
    with pytest.raises(AssertionError):
        rabitq_search(torch.zeros(2, 128, dtype=torch.float16, device="cuda"), k, c, f, s, 101)
    big = torch.zeros(2000, 128, dtype=torch.float16, device="cuda")
    with pytest.raises(RuntimeError, match="topk"):                      # topk above 1024
        rabitq_search(torch.zeros(1, 128, dtype=torch.float16, device="cuda"), big,
                      torch.zeros(big.shape[0], 16, dtype=torch.uint8, device="cuda"),
                      torch.zeros(big.shape[0], 2, dtype=torch.float16, device="cuda"), s, 1025)


def _filter_premise(est_row, n, topk):
    """For the filter path's plan, from the oracle's estimates of one query:
    the number of keys reaching the threshold and the fullest 256-key list's
    count.  Plan: s = min(n, 2048) sample keys, 64 runs of 32 consecutive
    keys starting at multiples of n // 64 (every key when n < 2048);
    m = ceil(4 k s / n), at least 8; tau = the lower edge of the bin holding
    the m-th largest sample among 4096 bins of width 2^shift over the samples'
    [min, max] (shift = bit length of max - min, less 12, at least 0);
    lists hold 15 entries."""
    from oracle.select import ordered_key
    keys = ordered_key(est_row).astype(np.int64)
    s = min(n, 2048)
    i = np.arange(s)
    sk = keys[(i >> 5) * (n // 64) + (i & 31)] if s == 2048 else keys
    m = min(s, max(8, -(-4 * topk * s // n)))
    lo, hi = int(sk.min()), int(sk.max())
    shift = max((hi - lo).bit_length() - 12, 0)
    mth = int(np.sort(sk)[::-1][m - 1])
    tau = lo + (((mth - lo) >> shift) << shift)
    hit = keys >= tau
    per_list = np.add.reduceat(hit.astype(np.int64), np.arange(0, n, 256))
    return int(hit.sum()), int(per_list.max())


def _check_planted(rng, n, topk, planted_rows, Q=2, dup=None, premise=None):
    """Search where the first query is planted at `planted_rows` (its copies
    estimate highest, all equal); compare everything with the oracle.
    ``premise(hits, fullest_slice)`` checks which select path the first query
    takes."""
    from zoomkv_revision_amd.rabitq import rabitq_encode, rabitq_search
    s_np, s_t = _signs()
    keys = orq.clustered_unit_keys(rng, n if dup is None else dup, 16)
    if dup is not None:
        keys = keys[rng.integers(0, dup, size=n)]
    qs = orq.clustered_unit_keys(rng, Q, 16)
    keys[planted_rows] = qs[0]
    kt = _f16(keys)
    codes, fac = rabitq_encode(kt, s_t)
    cand, fidx, fsc = (from_torch(t) for t in rabitq_search(_f16(qs), kt, codes, fac, s_t, topk))
    ck, fk = orq.encode(keys, s_np)
    if premise is not None:
        cq, fq = orq.encode(qs[:1], s_np)
        assert premise(*_filter_premise(orq.estimate(cq, fq, ck, fk)[0], n, topk))
    rc, ri, rs = orq.search(qs, keys, ck, fk, s_np, topk)
    assert np.array_equal(cand, rc), "candidate set"
    assert np.array_equal(fidx, ri), "reranked order"
    assert np.array_equal(fsc.view(np.uint32), rs.view(np.uint32)), "exact scores"
    return cand


def test_search_filter_path_tau_above_the_kth_key(rng):
    """131072 keys, top-256: tau comes from the 16th largest of 2048 samples
    (64 runs of 32 keys every 2048).  200 copies of the query sit at
    sampled positions, so tau falls in their estimate's bin and fewer than k
    keys reach it: the select kernel takes its exact full-pool path."""
    t = np.arange(200)
    rows = (t % 64) * 2048 + (t // 64) * 5
    cand = _check_planted(rng, 131072, 256, rows, premise=lambda hits, full: hits < 256)
    assert set(rows.tolist()) <= set(cand[0].tolist())


def test_search_filter_path_overflowing_slice(rng):
    """40 consecutive copies of the query fill one 256-key list beyond its
    15 entries: the select kernel detects the overflow and takes its exact
    full-pool path."""
    _check_planted(rng, 65536, 200, np.arange(1024, 1064), premise=lambda hits, full: full > 15)


def test_search_filter_path_ties(rng):
    """Only 40 distinct keys among 131072 (every estimate ties with ~3300
    others) and only 2 distinct among 40000: ties at the threshold and at the
    k-th key go to the lowest indices, on the filter path (lists hold all of
    the >= 256 keys at or above tau) and on the full-pool path."""
    _check_planted(rng, 131072, 256, np.arange(0), dup=40,
                   premise=lambda hits, full: 256 <= hits <= 4096 and full <= 15)
    _check_planted(rng, 40000, 100, np.arange(0), dup=2, premise=lambda hits, full: full > 15)


def test_search_filter_path_beyond_compaction(rng):
    """262144 keys, top-1024: 4281 keys reach tau, more than the 4096 entries
    the select kernel compacts into LDS, with every list within its 15
    entries: the kernel selects and places them from its registers."""
    _check_planted(rng, 262144, 1024, np.arange(0), premise=lambda hits, full: 4096 < hits and full <= 15)


def test_search_filter_path_negative_tau(rng):
    """One cluster and queries opposite its keys: the 256th largest estimate,
    and so tau, is negative, where the filter re-checks its hits with the
    exact keys instead of taking the float compare's mask as it is."""
    from zoomkv_revision_amd.rabitq import rabitq_encode, rabitq_search
    s_np, s_t = _signs()
    n, topk = 131072, 256
    keys = orq.clustered_unit_keys(rng, n, 1)
    qs = keys[:2] ^ np.uint16(0x8000)
    ck, fk = orq.encode(keys, s_np)
    cq, fq = orq.encode(qs, s_np)
    est = orq.estimate(cq, fq, ck, fk)
    for row in est:
        assert np.sort(row)[-topk] < 0
        hits, full = _filter_premise(row, n, topk)
        assert hits >= topk and full <= 15
    kt = _f16(keys)
    codes, fac = rabitq_encode(kt, s_t)
    cand, fidx, fsc = (from_torch(t) for t in rabitq_search(_f16(qs), kt, codes, fac, s_t, topk))
    rc, ri, rs = orq.search(qs, keys, ck, fk, s_np, topk)
    assert np.array_equal(cand, rc), "candidate set"
    assert np.array_equal(fidx, ri), "reranked order"
    assert np.array_equal(fsc.view(np.uint32), rs.view(np.uint32)), "exact scores"


def test_search_plan_reads_current_contents(rng):
    """A SearchPlan checks its buffers once; each run searches what they hold
    then (queries rewritten in place between runs) with rabitq_search's bits."""
    from zoomkv_revision_amd.rabitq import SearchPlan, rabitq_encode, rabitq_search
    _, s_t = _signs()
    n, nq, topk = 40000, 4, 64
    kt = _f16(orq.clustered_unit_keys(rng, n, 16))
    codes, fac = rabitq_encode(kt, s_t)
    q_buf = torch.empty(nq, 128, dtype=torch.float16, device=kt.device)
    plan = SearchPlan(q_buf, kt, codes, fac, s_t, topk)
    for _ in range(2):
        qt = _f16(orq.clustered_unit_keys(rng, nq, 16))
        q_buf.copy_(qt)
        got = plan.run()
        ref = rabitq_search(qt, kt, codes, fac, s_t, topk)
        for a, b in zip(got, ref):
            assert torch.equal(a.view(torch.int32) if a.dtype == torch.float32 else a,
                               b.view(torch.int32) if b.dtype == torch.float32 else b)


def test_search_plan_rejects_operands_it_would_copy(rng):
    from zoomkv_revision_amd.rabitq import SearchPlan, rabitq_encode
    _, s_t = _signs()
    kt = _f16(orq.clustered_unit_keys(rng, 4096, 8))
    codes, fac = rabitq_encode(kt, s_t)
    q = torch.zeros(128, 6, dtype=torch.float16, device=kt.device).t()   # non-contiguous [6, 128]
    with pytest.raises(AssertionError, match="in place"):
        SearchPlan(q, kt, codes, fac, s_t, 16)
