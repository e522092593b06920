"""GPU parity of the bound kernels against the oracle, through the C ABI.

Integer work: every value must be bit-identical to the oracle's restatement
of bound_flowshop::bornes_calculer on the same node."""
import numpy as np
import pytest

import oracle
import wsbb_amd

pytestmark = pytest.mark.gpu


def edge_nodes(n, rng):
    """root, leaves, one free job, prefix-only and suffix-only nodes."""
    perms, l1s, l2s = [], [], []

    def add(perm, l1, l2):
        perms.append(perm)
        l1s.append(l1)
        l2s.append(l2)

    ident = np.arange(n)
    add(ident, -1, n)                           # root
    for _ in range(8):
        perm = rng.permutation(n)
        l1 = int(rng.integers(-1, n))
        add(perm, l1, l1 + 1)                   # leaf
        l1 = int(rng.integers(-1, n - 1))
        add(perm, l1, l1 + 2)                   # one free job
        add(perm, int(rng.integers(-1, n - 1)), n)  # no suffix
        add(perm, -1, int(rng.integers(1, n + 1)))  # no prefix
    permT = np.array(perms, np.uint8).T.copy()
    return permT, np.array(l1s, np.int32), np.array(l2s, np.int32)


def cases():
    rng = np.random.default_rng(0)
    out = [("ta001_20x5", oracle.taillard(1)[3]), ("ta011_20x10", oracle.taillard(11)[3]),
           ("ta021_20x20", oracle.taillard(21)[3]), ("ta051_50x20", oracle.taillard(51)[3]),
           ("ta081_100x20", oracle.taillard(81)[3]),
           ("corr_50x10", oracle.generate_correlated(50, 10, 5)),
           ("ties_30x6", rng.integers(1, 4, size=(6, 30)).astype(np.int32)),
           ("max_128x24", rng.integers(1, 100, size=(24, 128)).astype(np.int32)),
           # bound values beyond 2^14: the int16 two-node form does not apply
           ("big_p_20x10", rng.integers(1, 3000, size=(10, 20)).astype(np.int32)),
           ("tiny_3x2", rng.integers(1, 10, size=(2, 3)).astype(np.int32))]
    return out


def batch_for(n, N, seed):
    permT, l1, l2 = oracle.random_nodes(n, N, seed)
    e = edge_nodes(n, np.random.default_rng(seed))
    return (np.concatenate([permT, e[0]], axis=1), np.concatenate([l1, e[1]]),
            np.concatenate([l2, e[2]]))


@pytest.mark.parametrize("name,p", cases(), ids=[c[0] for c in cases()])
def test_lb2_lb1_parity(name, p):
    m, n = p.shape
    o = oracle.Oracle(p)
    N = 3000 if n <= 50 else 1000
    permT, l1, l2 = batch_for(n, N, 0x5EED)
    ref = o.bound_batch(permT, l1, l2, kind=oracle.LB2, threads=8)
    with wsbb_amd.Engine(p) as eng:
        # both the two-node int16 form (when the instance fits) and the int32 form
        for int16 in (2, 0):
            eng.set_int16(int16)
            for groups in (1, 2, 4):
                eng.set_launch(groups=groups)
                got = eng.bound(permT, l1, l2, kind=wsbb_amd.LB2)
                bad = np.nonzero(got != ref)[0]
                assert bad.size == 0, (int16, groups, bad[:5], got[bad[:5]], ref[bad[:5]])
        eng.set_int16(1)
        eng.set_launch(groups=0)
        got1 = eng.bound(permT, l1, l2, kind=wsbb_amd.LB1)
        ref1 = o.bound_batch(permT, l1, l2, kind=oracle.LB1, threads=8)
        assert np.array_equal(got1, ref1)
        leaf = (l2 - l1) == 1
        assert (got1[~leaf] <= ref[~leaf]).all() or m < 2


@pytest.mark.parametrize("tid", [11, 51])
def test_pair_values_argmax_best_subset(tid):
    p = oracle.taillard(tid)[3]
    m, n = p.shape
    o = oracle.Oracle(p)
    permT, l1, l2 = oracle.random_nodes(n, 700, 42)
    rng = np.random.default_rng(1)
    with wsbb_amd.Engine(p) as eng:
        P = eng.P
        res = eng.bound(permT, l1, l2, argmax=True, pairv=True, feat=True)
        for k in range(0, 700, 7):
            perm = permT[:, k].astype(np.int32)
            lb, v = o.pair_values(perm, l1[k], l2[k])
            assert res["bound"][k] == lb
            assert np.array_equal(res["pairv"][:, k], v)
            assert res["argmax"][k] == int(np.argmax(v))
            # features: head, tail, remaining work per machine (scaled)
            r, q = o.heads_tails(perm, l1[k], l2[k])
            t = o.tables()
            d1, d2 = l1[k] + 1, n - l2[k]
            head = r if d1 else t["R0"]
            tail = q if d2 else t["Q0"]
            rem = p[:, perm[l1[k] + 1:l2[k]]].sum(axis=1)
            f = res["feat"][:, k].reshape(5, m)
            scale = int(p.max(axis=0).sum() + p.max(axis=1).sum())  # path bound
            for row, ref in zip(f, [head, tail, rem, head + rem, rem + tail]):
                assert np.allclose(row * scale, ref, rtol=1e-5, atol=1e-3)
        # early exit against an incumbent
        best = rng.integers(500, 5000, size=700).astype(np.int32)
        for k in range(0, 700, 13):
            got = eng.bound(permT[:, k:k + 1], l1[k:k + 1], l2[k:k + 1], best=int(best[k]))[0]
            assert got == o.bound(permT[:, k].astype(np.int32), l1[k], l2[k], best=int(best[k]))
        # pair subsets
        nsw = (P + 31) // 32
        selb = rng.random((P, 700)) < 0.1
        sel = np.zeros((nsw, 700), np.uint32)
        for s in range(P):
            sel[s // 32] |= (selb[s].astype(np.uint32) << np.uint32(s % 32))
        got = eng.bound(permT, l1, l2, sel=sel)
        for k in range(0, 700, 5):
            ref = o.bound_subset(permT[:, k].astype(np.int32), l1[k], l2[k],
                                 selb[:, k].astype(np.uint8))
            assert got[k] == ref


def test_full_size_batch_50x20():
    """2^20 nodes of the 50x20 batched workload: full parity on a 2^15
    sample (oracle), properties on all nodes, and run-to-run determinism."""
    p = oracle.taillard(51)[3]
    n = p.shape[1]
    N = 1 << 20
    permT, l1, l2 = wsbb_amd.random_nodes(n, N, 0x5EED)
    o = oracle.Oracle(p)
    with wsbb_amd.Engine(p) as eng:
        lb2 = eng.bound(permT, l1, l2)
        lb2b = eng.bound(permT, l1, l2)
        lb1 = eng.bound(permT, l1, l2, kind=wsbb_amd.LB1)
    assert np.array_equal(lb2, lb2b)
    assert (lb1 <= lb2).all() and (lb2 > 0).all()
    idx = np.random.default_rng(3).choice(N, 1 << 15, replace=False)
    ref = o.bound_batch(permT[:, idx], l1[idx], l2[idx], threads=16)
    assert np.array_equal(lb2[idx], ref)


def test_device_resident_api_matches_host_api():
    p = oracle.taillard(21)[3]
    n = p.shape[1]
    N = 5000
    permT, l1, l2 = oracle.random_nodes(n, N, 7)
    with wsbb_amd.Engine(p) as eng:
        host = eng.bound(permT, l1, l2)
        dp, d1, d2, do = (eng.malloc(permT.nbytes), eng.malloc(4 * N), eng.malloc(4 * N),
                          eng.malloc(4 * N))
        try:
            eng.h2d(dp, permT)
            eng.h2d(d1, l1)
            eng.h2d(d2, l2)
            eng.bound_device(dp, d1, d2, N, do)
            eng.synchronize()
            dev = eng.d2h(np.zeros(N, np.int32), do)
        finally:
            for d in (dp, d1, d2, do):
                eng.free(d)
    assert np.array_equal(host, dev)


def test_invalid_nodes_are_rejected_on_the_host():
    p = oracle.taillard(1)[3]
    with wsbb_amd.Engine(p) as eng:
        permT, l1, l2 = oracle.random_nodes(20, 10, 1)
        bad = permT.copy()
        bad[0, 0] = 20
        with pytest.raises(wsbb_amd.WsbbError):
            eng.bound(bad, l1, l2)
        bl = l2.copy()
        bl[3] = l1[3]
        with pytest.raises(wsbb_amd.WsbbError):
            eng.bound(permT, l1, bl)


@pytest.mark.parametrize("n,m", [(2, 2), (10, 3), (20, 24), (30, 7), (31, 8), (32, 9), (33, 12),
                                 (62, 13), (63, 16), (64, 17), (65, 5), (94, 20), (95, 21), (96, 6),
                                 (97, 4), (126, 10), (127, 11), (128, 3)])
def test_lb2_matrix_core_operand_edges(n, m):
    """Job counts at the edges of the 32-wide operands (two constant columns
    after the jobs), machine counts at those of the padded rows, batches at
    the tiles' edges, and times at 127, the largest the form takes; 128 and
    126 + 2 jobs fall back to the scan.  Whole numbers: equal."""
    rng = np.random.default_rng(n * 100 + m)
    p = rng.integers(0, 128, size=(m, n)).astype(np.int32)
    p[rng.integers(m), rng.integers(n)] = 127
    big = p.copy()
    big[0, 0] = 128
    for q in (p, big):
        o = oracle.Oracle(q)
        with wsbb_amd.Engine(q) as eng:
            for N in (1, 63, 129, 700):
                permT, l1, l2 = batch_for(n, N, N)
                ref = o.bound_batch(permT, l1, l2, kind=oracle.LB2, threads=8)
                for groups in (1, 2, 4, 8):
                    eng.set_launch(groups=groups)
                    assert np.array_equal(eng.bound(permT, l1, l2), ref), (N, groups)


@pytest.mark.parametrize("tid,N", [(51, 140_001), (71, 70_003), (21, 140_001)])
def test_lb2_large_batches_in_several_launches(tid, N):
    """Batches large enough for 128-node tiles (50 and 100 jobs) and one wave
    per tile (20 jobs), whole and under a block cap."""
    p = oracle.taillard(tid)[3]
    n = p.shape[1]
    permT, l1, l2 = wsbb_amd.random_nodes(n, N, 11)
    idx = np.r_[0:200, N - 200:N, np.random.default_rng(5).choice(N, 3000, replace=False)]
    ref = oracle.Oracle(p).bound_batch(permT[:, idx], l1[idx], l2[idx], threads=16)
    with wsbb_amd.Engine(p) as eng:
        got = eng.bound(permT, l1, l2)
        eng.set_launch(groups=0, grid_blocks=100)
        assert np.array_equal(eng.bound(permT, l1, l2), got)
    assert np.array_equal(got[idx], ref)


@pytest.mark.gpu
@pytest.mark.parametrize("kind", [oracle.LB2, oracle.LB1])
def test_host_batches_about_the_in_place_limit(kind):
    """Host batches that the kernel reads in place (20 jobs: up to 32768
    nodes), just above it, and small ones after large ones on one engine."""
    p = oracle.taillard(11)[3]
    n = p.shape[1]
    ref = oracle.Oracle(p)
    with wsbb_amd.Engine(p) as eng:
        for seed, N in enumerate((1, 32768, 65, 32769, 32767, 3)):
            permT, l1, l2 = wsbb_amd.random_nodes(n, N, 100 + seed)
            idx = np.unique(np.r_[0:min(N, 300), max(0, N - 300):N])
            want = ref.bound_batch(permT[:, idx], l1[idx], l2[idx], kind=kind, threads=16)
            assert np.array_equal(eng.bound(permT, l1, l2, kind=kind)[idx], want), (seed, N)
            bad = permT.copy()
            bad[n - 1, N - 1] = n
            with pytest.raises(wsbb_amd.WsbbError, match=f"index {n * N - 1}"):
                eng.bound(bad, l1, l2, kind=kind)


@pytest.mark.parametrize("n,m,scale", [(20, 5, 1), (50, 20, 1), (100, 3, 1), (20, 10, 9)])
def test_device_batch_leaves_out_nodes_with_impossible_limits(n, m, scale):
    """Limits in device memory that no node can have, among ordinary ones: the
    kernels (matrix cores, both scans, LB1) leave those nodes out and bound the
    others; times beyond a signed byte take the scan."""
    p = scale * np.random.default_rng(n).integers(1, 100, size=(m, n)).astype(np.int32)
    o = oracle.Oracle(p)
    big = 2**31 - 1
    wrong = [(-2, n), (-1, n + 1), (3, 3), (n, n), (5, 4), (n - 1, 0), (big, big), (-big - 1, big),
             (big, -big - 1), (0, big), (-big, 1), (n + 40, n + 41)]
    with wsbb_amd.Engine(p) as eng:
        for N in (1, 200, 1025):
            permT, l1, l2 = wsbb_amd.random_nodes(n, N, N)
            at = np.random.default_rng(N).permutation(N)[:max(1, N // 3)]
            ok = np.ones(N, bool)
            ok[at] = False
            b1, b2 = l1.copy(), l2.copy()
            for i, k in enumerate(at):
                b1[k], b2[k] = wrong[i % len(wrong)]
            d = [eng.malloc(permT.nbytes)] + [eng.malloc(4 * N) for _ in range(3)]
            for buf, a in zip(d, (permT, b1, b2)):
                eng.h2d(buf, a)
            for kind in (wsbb_amd.LB2, wsbb_amd.LB1):
                ref = np.full(N, -7, np.int32)
                ref[ok] = o.bound_batch(permT, l1, l2, kind=kind, threads=8)[ok]
                for int16 in (1, 2):
                    eng.set_int16(int16)
                    eng.h2d(d[3], np.full(N, -7, np.int32))
                    eng.bound_device(d[0], d[1], d[2], N, d[3], kind=kind)
                    got = np.zeros(N, np.int32)
                    eng.d2h(got, d[3])
                    assert np.array_equal(got, ref), (N, kind, int16)
            for buf in d:
                eng.free(buf)


@pytest.mark.parametrize("n,m,scale,groups", [(20, 24, 1, [1, 2, 4]), (50, 5, 1, [1, 2]), (100, 5, 1, [1]),
                                              (20, 20, 9, [1, 2, 4]), (20, 5, 9, [1, 2, 4, 8, 16])])
def test_autotune_times_the_shapes_it_lists(n, m, scale, groups):
    """Every shape once: the waves that can split a tile's pairs, under each
    grid only for the scans (times beyond a signed byte), whose blocks loop."""
    p = scale * np.random.default_rng(n).integers(1, 100, size=(m, n)).astype(np.int32)
    permT, l1, l2 = wsbb_amd.random_nodes(n, 2000, 1)
    ref = oracle.Oracle(p).bound_batch(permT, l1, l2, threads=8)
    with wsbb_amd.Engine(p) as eng:
        for _ in range(2):  # the second finds the first's choice in place
            shapes = eng.autotune(2000, reps=50)
            assert len(set(s[:2] for s in shapes)) == len(shapes)
            assert sorted(set(s[0] for s in shapes)) == groups
            assert len(set(s[1] for s in shapes)) == (1 if scale == 1 else 3)
            ms = {s[0]: s[2] for s in shapes}
            if n == 20 and scale == 1:  # 32 tiles of 276 pairs: one wave a tile is what it says
                assert ms[1] > 1.2 * ms[4], ms
            assert np.array_equal(eng.bound(permT, l1, l2), ref)


def device_us(eng, permT, l1, l2, reps=10):
    """Bounds of a resident batch and the least of five timings of a pass."""
    N = l1.shape[0]
    d = [eng.malloc(permT.nbytes)] + [eng.malloc(4 * N) for _ in range(3)]
    for buf, a in zip(d, (permT, l1, l2)):
        eng.h2d(buf, a)
    eng.bound_device(d[0], d[1], d[2], N, d[3])
    times = []
    for _ in range(5):
        eng.timer_start()
        for _ in range(reps):
            eng.bound_device(d[0], d[1], d[2], N, d[3])
        times.append(eng.timer_stop() / reps * 1e3)
    out = np.zeros(N, np.int32)
    eng.d2h(out, d[3])
    for buf in d:
        eng.free(buf)
    return out, min(times)


def test_large_batches_about_32_jobs():
    """31 and 32 jobs have one row tile, as 30, and two column blocks: their
    large batches stay on 64-node tiles, and cost little more."""
    N, us = 300_001, {}
    for n in (30, 31, 32):
        p = np.random.default_rng(n).integers(1, 100, size=(20, n)).astype(np.int32)
        permT, l1, l2 = wsbb_amd.random_nodes(n, N, n)
        with wsbb_amd.Engine(p) as eng:
            out, us[n] = device_us(eng, permT, l1, l2)
        idx = np.r_[0:300, N - 300:N, np.random.default_rng(1).choice(N, 2000, replace=False)]
        assert np.array_equal(out[idx], oracle.Oracle(p).bound_batch(permT[:, idx], l1[idx], l2[idx], threads=8))
    # 97, 113 and 115 us; on 128-node tiles 179 and 182
    assert max(us[31], us[32]) < 1.4 * us[30], us


def test_large_batches_of_three_row_tiles():
    """65 to 94 jobs: large batches stay on 64-node tiles, and 90 jobs cost no
    more than 100, which fill a block's four waves."""
    N, us = 300_001, {}
    for n in (65, 90, 94, 100):
        p = np.random.default_rng(n).integers(1, 100, size=(5, n)).astype(np.int32)
        permT, l1, l2 = wsbb_amd.random_nodes(n, N, n)
        with wsbb_amd.Engine(p) as eng:
            out, us[n] = device_us(eng, permT, l1, l2)
        idx = np.r_[0:300, N - 300:N, np.random.default_rng(1).choice(N, 2000, replace=False)]
        assert np.array_equal(out[idx], oracle.Oracle(p).bound_batch(permT[:, idx], l1[idx], l2[idx], threads=8))
    # 123 and 137 us; on 128-node tiles 90 jobs take 165
    assert us[90] < 1.05 * us[100], us


@pytest.mark.parametrize("n,m,N,faster", [
    # the scans' side and the matrix cores' at the rule's sizes, pairs and jobs
    (11, 3, 98_303, False), (11, 3, 98_304, False), (11, 4, 262_143, False), (11, 3, 262_144, False),
    (8, 4, 300_001, True), (5, 2, 524_288, True), (11, 3, 1 << 20, True), (11, 6, 1 << 20, False),
    (33, 3, 1 << 20, True), (65, 3, 1 << 20, True), (96, 5, 1 << 20, True), (97, 3, 300_001, False),
    (21, 2, 524_287, False), (31, 3, 1 << 20, False), (8, 3, 49_152, False), (95, 5, 200_001, True)])
def test_large_batches_of_few_pairs(n, m, N, faster):
    """Both forms of plain LB2 on the same resident batch, against the oracle
    on a sample; where the rule's measurements say that the scans are clearly
    faster (by 12% and more), the call is as fast as they are."""
    p = np.random.default_rng(100 * n + m).integers(1, 100, size=(m, n)).astype(np.int32)
    permT, l1, l2 = wsbb_amd.random_nodes(n, N, 3)
    idx = np.r_[0:300, N - 300:N, np.random.default_rng(1).choice(N, 3000, replace=False)]
    ref = oracle.Oracle(p).bound_batch(permT[:, idx], l1[idx], l2[idx], threads=8)
    with wsbb_amd.Engine(p) as eng:
        out, us = device_us(eng, permT, l1, l2)
        eng.set_int16(2)
        scan, scan_us = device_us(eng, permT, l1, l2)
        eng.set_int16(0)
        other, _ = device_us(eng, permT, l1, l2, reps=1)
    assert np.array_equal(out[idx], ref)
    assert np.array_equal(out, scan) and np.array_equal(out, other)
    if faster:
        assert us < 1.07 * scan_us, (us, scan_us)


def test_first_small_batch_of_an_engine_allocates_no_staging():
    """A new engine's first 64-node call costs about what its next ones do
    (the pinned staging is the device's); making staging for it took as long
    again as the call."""
    import time

    p = oracle.taillard(1)[3]
    nodes = wsbb_amd.random_nodes(20, 64, 1)
    ref = oracle.Oracle(p).bound_batch(*nodes)
    first, later = [], []
    for _ in range(41):
        with wsbb_amd.Engine(p) as eng:
            eng.synchronize()
            for times in (first, later):
                t = time.perf_counter()
                got = eng.bound(*nodes)
                times.append(time.perf_counter() - t)
                assert np.array_equal(got, ref)
    assert np.median(first) < 1.5 * np.median(later), (np.median(first), np.median(later))


def test_small_batches_of_engines_on_threads():
    """Calls of several threads' engines overlap: one stages in the device's
    buffer, the others in their own."""
    import threading

    ps = [oracle.taillard(t)[3] for t in (1, 11, 21, 51)]
    wrong = []

    def work(i):
        p = ps[i]
        n = p.shape[1]
        with wsbb_amd.Engine(p) as eng:
            for rep in range(60):
                N = (1, 64, 4096, 15000)[(i + rep) % 4]
                permT, l1, l2 = wsbb_amd.random_nodes(n, N, 10 * i + rep)
                pick = np.unique(np.r_[0:min(N, 40), max(0, N - 40):N])
                want = oracle.Oracle(p).bound_batch(permT[:, pick], l1[pick], l2[pick])
                if not np.array_equal(eng.bound(permT, l1, l2)[pick], want):
                    wrong.append((i, rep, N))

    threads = [threading.Thread(target=work, args=(i,)) for i in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not wrong


@pytest.mark.parametrize("n", [31, 32, 33, 62, 64, 65, 94, 96, 97])
@pytest.mark.parametrize("m", [8, 16, 24])
def test_lb2_large_batches_at_operand_edges(n, m):
    """Batches large enough for one wave a row tile (every size) and for
    128-node tiles (two row tiles, three with four column blocks, four) at
    the edges of the operands, the last tile partial."""
    N = 131_137
    p = np.random.default_rng(n * m).integers(0, 128, size=(m, n)).astype(np.int32)
    permT, l1, l2 = wsbb_amd.random_nodes(n, N, n + m)
    idx = np.r_[0:200, N - 200:N, np.random.default_rng(7).choice(N, 1500, replace=False)]
    ref = oracle.Oracle(p).bound_batch(permT[:, idx], l1[idx], l2[idx], threads=8)
    with wsbb_amd.Engine(p) as eng:
        assert np.array_equal(eng.bound(permT, l1, l2)[idx], ref)
