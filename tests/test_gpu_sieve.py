"""The sieved plain path (int8 score pass, exact scores of its candidates) against the CPU
oracle: matches of pairs at block and tile edges, uneven sizes, minimum scores and ratios on
both sides of the rule that takes the path, rows the int8 form holds badly (large components,
negative components, norms other than one), equal scores, and sets that overflow the candidate
lists.  Matches are whole numbers: they equal the oracle's."""
import ctypes as C

import numpy as np
import pytest

import v3dmatch
from oracle import oracle
from v3dmatch import synth

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def matcher():
    m = v3dmatch.SIFT_Matching(0)
    m.enableRoundingWarning(False)
    m.allocate(4096, 4096)
    yield m
    m.close()


def _unit(x):
    return (x / np.linalg.norm(x, axis=1, keepdims=True)).astype(np.float32)


def _same(m, L, R, min_score, min_ratio):
    m.setLeftFeatures(L.shape[0], L)
    m.setRightFeatures(R.shape[0], R)
    got = m.find_putative_matches_array(min_score, min_ratio)
    assert np.array_equal(got, oracle.find_putative_matches(L, R, min_score, min_ratio))


@pytest.mark.parametrize("nL,nR", [(32, 32), (32, 4096), (4096, 32), (96, 160), (128, 512), (512, 128), (544, 1056),
                                   (2016, 2080), (4096, 4096)])
@pytest.mark.parametrize("min_score,min_ratio", [(0.9, 0.8), (0.85, 0.7), (0.8, -1.0), (0.75, 0.9), (0.2, 0.8)])
def test_sizes(matcher, nL, nR, min_score, min_ratio):
    print(f"case sieve {nL} x {nR} min {min_score} ratio {min_ratio}", flush=True)
    a, b, _ = synth.make_pair(nL, nR, 0.4, config=7, pair=nL + nR)
    _same(matcher, synth.dequantise(a), synth.dequantise(b), min_score, min_ratio)


@pytest.mark.parametrize("kind", ["sparse", "signed", "norms", "ties"])
def test_rows(matcher, kind):
    """sparse: components up to 1 (the int8 rows clip); signed: both signs; norms: 2^-3 to 1.9;
    ties: equal rows on both sides."""
    print(f"case sieve rows {kind}", flush=True)
    rng = np.random.default_rng(3)
    n = 640
    if kind == "sparse":
        L = np.zeros((n, 128), np.float32)
        for i in range(n):
            L[i, rng.choice(128, 3, replace=False)] = rng.uniform(0.3, 1.0, 3)
        L = _unit(L)
    else:
        L = _unit(rng.standard_normal((n, 128)))
    R = _unit(L[rng.permutation(n)] + 0.02 * rng.standard_normal((n, 128)))
    if kind == "norms":
        L = L * rng.uniform(0.125, 1.9, (n, 1)).astype(np.float32)
        R = R * rng.uniform(0.125, 1.9, (n, 1)).astype(np.float32)
    if kind == "ties":
        R[200:232] = R[100]
        L[300:340] = L[17]
        R[5] = L[17]
        R[630] = L[17]
    for ms, mr in ((0.9, 0.8), (0.8, -1.0), (0.8, 0.95)):
        _same(matcher, L, R, ms, mr)


@pytest.mark.parametrize("share", [0.3, 1.0])
def test_flooded_lists(matcher, share):
    """Nearly equal rows: every pair of them is a candidate and the lists overflow."""
    print(f"case sieve flooded {share}", flush=True)
    rng = np.random.default_rng(4)
    n = 1024
    a, b, _ = synth.make_pair(n, n, 0.4, config=7, pair=3)
    L, R = synth.dequantise(a), synth.dequantise(b)
    k = int(share * n)
    c = _unit(np.abs(rng.standard_normal((1, 128))))
    L[:k] = _unit(c + 0.01 * rng.standard_normal((k, 128)))
    R[n - k:] = _unit(c + 0.01 * rng.standard_normal((k, 128)))
    _same(matcher, L, R, 0.9, 0.8)
    assert matcher.stats()["nRechecked"] > 0
    _same(matcher, L, R, 0.9, -1.0)


def test_timing_leaves_no_state(matcher):
    print("case sieve timing", flush=True)
    a, b, _ = synth.make_pair(1024, 992, 0.4, config=7, pair=9)
    L, R = synth.dequantise(a), synth.dequantise(b)
    _same(matcher, L, R, 0.9, 0.8)
    assert matcher.time_dominant_kernel(3) > 0
    _same(matcher, L, R, 0.9, 0.8)


SIZES = [(33, 70), (512, 31), (256, 256), (300, 1700), (1056, 96), (32, 32), (640, 513), (513, 2080)]


@pytest.mark.parametrize("dtype", ["u8", "f32"])
@pytest.mark.parametrize("cache", [False, True])
def test_batch(dtype, cache):
    """Uneven pairs, with minimum scores that take the sieve and one that does not, in turn on
    one batch (runs, graph replays, and rows made by every run or kept)."""
    images = []
    for p, (nL, nR) in enumerate(SIZES):
        images += list(synth.make_pair(nL, nR, 0.5, config=3, pair=700 + p)[:2])
    left = np.arange(0, 2 * len(SIZES), 2, dtype=np.int32)
    rows = np.concatenate(images if dtype == "u8" else [synth.dequantise(q) for q in images])
    m = v3dmatch.SIFT_Matching(0)
    m.batch_set_images([len(q) for q in images], rows)
    m.batch_set_pairs(left, left + 1)
    m.set_derived_cache(cache)
    for ms, mr in ((0.9, 0.8), (0.2, 0.8), (0.85, -1.0), (0.9, 0.8), (0.2, 0.8)):
        print(f"case sieve batch {dtype} cache {cache} min {ms} ratio {mr}", flush=True)
        got = m.batch_match(ms, mr)
        for p in range(len(SIZES)):
            L, R = (synth.dequantise(images[2 * p + k][:len(images[2 * p + k]) // 32 * 32]) for k in (0, 1))
            want = oracle.find_putative_matches(L, R, ms, mr) if len(L) and len(R) else np.zeros((0, 2), np.int32)
            assert np.array_equal(np.asarray(got[p]).reshape(-1, 2), want.reshape(-1, 2)), (p, ms, mr)
    m.close()


@pytest.mark.parametrize("scale", [1.0, 1e-8, 1e-20, 1e12])
@pytest.mark.parametrize("threshold", [0.0, 1e-3, 1.5, 40.0])
def test_guided_mask(matcher_guided, scale, threshold):
    """The epipolar mask at scales of F that take the comparison of products and that leave
    single pairs or every pair to the division, on positions of which some lie on the lines."""
    print(f"case guided mask scale {scale} threshold {threshold}", flush=True)
    m = matcher_guided
    rng = np.random.default_rng(12)
    nL, nR = 352, 288
    a, b, _ = synth.make_pair(nL, nR, 0.5, config=7, pair=44)
    L, R = synth.dequantise(a), synth.dequantise(b)
    lxy = rng.uniform(0, 1000, (nL, 2)).astype(np.float32)
    rxy = rng.uniform(0, 1000, (nR, 2)).astype(np.float32)
    rxy[::3, 1] = lxy[:len(rxy[::3]), 1]                    # on the lines of a sideways motion
    F = np.array([[0, 0, 0], [0, 0, -1.0], [0, 1.0, 0]]) + 1e-4 * rng.standard_normal((3, 3))
    m.setLeftFeatures(nL, L)
    m.setRightFeatures(nR, R)
    m.find_putative_matches_array(0.9, 0.8)
    S = oracle.scores(L, R)
    for min_score in (0.9, 0.2):
        got = m.run_guided_array(False, scale * F, threshold, lxy, rxy, min_score, -1.0)
        want = oracle.guided(S, 0, scale * F, np.float32(threshold), lxy, rxy, min_score, -1.0)
        assert np.array_equal(got, want)


@pytest.fixture(scope="module")
def matcher_guided():
    m = v3dmatch.SIFT_Matching(0)
    m.enableRoundingWarning(False)
    m.allocate(512, 512, True)
    yield m
    m.close()


@pytest.mark.parametrize("first", [0xfffffffe, 0xffffffff])
@pytest.mark.parametrize("order", ["left right", "right left", "left right left", "right left right"])
def test_upload_counters_wrap(first, order):
    """The sets' largest norms are kept under the number of the upload; past its 32-bit wrap each
    side still has its own.  The side uploaded second holds rows whose int8 rounding errors all
    point the same way, the other side rows that int8 holds exactly, and the scores lie within
    those errors above the minimum: with a norm of 0 for the exact side the bound would drop them."""
    print(f"case sieve upload counter {first} order {order}", flush=True)
    rng = np.random.default_rng(8)
    n = 512
    X = np.rint(256 * _unit(rng.gamma(0.5, 1.0, (n, 128)))).clip(0, 120)
    X = (X / 256).astype(np.float32)
    Y = np.empty_like(X)
    for i in range(n):  # the largest multiple of row i below a score of 0.903
        for a in np.linspace(0.8, 1.3, 201):
            y = ((np.floor(a * 256 * X[i]) + 0.45) / 256).astype(np.float32)
            if float(y @ X[i]) > 0.903:
                break
            Y[i] = y
    L, R = (X, Y) if order.split()[0] == "left" else (Y, X)
    m = v3dmatch.SIFT_Matching(0)
    m.enableRoundingWarning(False)
    m.allocate(n, n)
    m.debug_prep_epoch(first)
    for side in order.split():
        (m.setLeftFeatures if side == "left" else m.setRightFeatures)(n, L if side == "left" else R)
    want = oracle.find_putative_matches(L, R, 0.9, -1.0)
    assert len(want) > 100 and np.array_equal(m.find_putative_matches_array(0.9, -1.0), want)
    with pytest.raises(v3dmatch.V3DMError):
        m.debug_prep_epoch(0)
    m.close()


@pytest.mark.parametrize("cache", [False, True])
@pytest.mark.parametrize("dtype", ["u8", "f32"])
def test_batch_tunes_the_pass_it_takes(dtype, cache):
    """A run that takes the sieve times no candidate of the full pass and still reports its
    setting; the first run that takes the pass tunes it, also after sieved runs of the same pairs,
    and every result is the oracle's."""
    print(f"case batch tuning with the sieve {dtype} cache {cache}", flush=True)
    images = []
    for p, (nL, nR) in enumerate(SIZES):
        images += list(synth.make_pair(nL, nR, 0.5, config=3, pair=800 + p)[:2])
    left = np.arange(0, 2 * len(SIZES), 2, dtype=np.int32)
    m = v3dmatch.SIFT_Matching(0)
    m.batch_set_images([len(q) for q in images],
                       np.concatenate(images if dtype == "u8" else [synth.dequantise(q) for q in images]))
    m.batch_set_pairs(left, left + 1)
    m.set_derived_cache(cache)
    for ms, mr, timed in ((0.9, 0.8, False), (0.9, 0.8, False), (0.2, 0.8, True), (0.9, 0.8, True), (0.2, 0.8, True)):
        got = m.batch_match(ms, mr)
        t = m.batch_get_tuning(v3dmatch.PREC_FP32)
        assert (t["pass_ms"] > 0) == timed and t["tiles_per_item"] > 0 and t["grid"] > 0 and t["items"] > 0
        for p in range(len(SIZES)):
            L, R = (synth.dequantise(images[2 * p + k][:len(images[2 * p + k]) // 32 * 32]) for k in (0, 1))
            want = oracle.find_putative_matches(L, R, ms, mr) if len(L) and len(R) else np.zeros((0, 2), np.int32)
            assert np.array_equal(np.asarray(got[p]).reshape(-1, 2), want.reshape(-1, 2)), (p, ms, mr)
    assert m.batch_time_dominant_kernel(2) > 0
    m.close()


def _many_candidates(kind, n):
    """Sets that the sieve gives to the full pass: clusters of nearly equal rows (spread over the
    sets, or in one run on each side), rows with two large components among SIFT rows, and rows of
    few large components throughout."""
    rng = np.random.default_rng(21)
    a, b, _ = synth.make_pair(n, n - 64, 0.4, config=7, pair=5)
    L, R = synth.dequantise(a).copy(), synth.dequantise(b).copy()
    if kind in ("spread", "runs", "whole"):
        k = n - 64 if kind == "whole" else n // 3
        c = _unit(np.abs(rng.standard_normal((1, 128))))
        i = rng.permutation(n)[:k] if kind == "spread" else np.arange(k)
        j = rng.permutation(n - 64)[:k] if kind == "spread" else np.arange(n - 64 - k, n - 64)
        L[i], R[j] = (_unit(c + 0.03 * rng.standard_normal((k, 128))) for _ in range(2))
    elif kind == "spikes":
        for X in (L, R):
            X[::32] = 0
            X[::32, 3], X[::32, 9] = 0.8, 0.6
    else:
        L, R = (_unit(np.maximum(rng.standard_normal((m, 128)) - 1.3, 0) + 1e-6) for m in (n, n - 64))
        R[:n // 4] = _unit(L[:n // 4] + 0.02 * np.abs(rng.standard_normal((n // 4, 128))))
    return L, R


KINDS = ["spread", "runs", "whole", "spikes", "large"]


@pytest.mark.parametrize("kind", KINDS)
@pytest.mark.parametrize("n", [512, 2080, 4064])
def test_many_candidates(kind, n):
    """Matches, decisions, the guided call behind them and the next ordinary call."""
    print(f"case sieve given up {kind} {n}", flush=True)
    L, R = _many_candidates(kind, n)
    m = v3dmatch.SIFT_Matching(0)
    m.enableRoundingWarning(False)
    m.allocate(n, n, True)
    S = oracle.scores(L, R)
    for ms, mr in ((0.9, 0.8), (0.9, -1.0)):
        _same(m, L, R, ms, mr)
        cm, rm = m.get_maxima()
        assert np.array_equal(cm, oracle.column_maxima(S, ms, mr))
        assert np.array_equal(rm, oracle.row_maxima(S, ms, mr))
    rng = np.random.default_rng(22)
    lxy, rxy = (rng.uniform(0, 1000, (len(X), 2)).astype(np.float32) for X in (L, R))
    H = np.eye(3)
    for t in (900.0, 400.0):  # the second call's mask adds to the first's
        got = m.run_guided_array(True, H, t, lxy, rxy, 0.9, 0.95)
    assert np.array_equal(got, oracle.guided(S, 1, H, np.float32(400.0), lxy, rxy, 0.9, 0.95))
    a, b, _ = synth.make_pair(n, n, 0.4, config=7, pair=6)
    _same(m, synth.dequantise(a), synth.dequantise(b), 0.9, 0.8)
    m.close()


@pytest.mark.parametrize("kind", KINDS + ["sift"])
@pytest.mark.parametrize("when", ["before", "after"])
def test_many_candidates_on_the_device(kind, when):
    """The same with the result read on the device: whole on the stream after an asynchronous call
    when the caller has the pointers (before), and when it asks for them (after); sets of settings
    that change between the call and the reading do not reach it."""
    print(f"case sieve given up, device results {kind} {when}", flush=True)
    n = 2080
    if kind == "sift":
        a, b, _ = synth.make_pair(n, n, 0.4, config=7, pair=5)
        L, R = synth.dequantise(a), synth.dequantise(b)
    else:
        L, R = _many_candidates(kind, n)
    rt = C.CDLL("libamdhip64.so")
    rt.hipMemcpy.argtypes = [C.c_void_p, C.c_void_p, C.c_size_t, C.c_int]
    m = v3dmatch.SIFT_Matching(0)
    m.enableRoundingWarning(False)
    m.allocate(n, n)
    pairs, counts = C.c_void_p(), C.c_void_p()

    def pointers():
        assert m._lib.v3dm_device_results(m._h, C.byref(pairs), C.byref(counts)) == 0

    if when == "before":
        pointers()
    for ms, mr in ((0.9, 0.8), (0.9, -1.0), (0.9, 0.8)):
        m.setLeftFeatures(len(L), L)
        m.setRightFeatures(len(R), R)
        m.find_async(ms, mr)
        m.set_certification(0.25)
        if when == "after":
            pointers()
        m.synchronize()
        m.set_certification(2.0 ** -15)
        cnt = np.zeros(1, np.int32)
        assert rt.hipMemcpy(cnt.ctypes.data, counts, 4, 2) == 0
        got = np.zeros((int(cnt[0]), 2), np.int32)
        if len(got):
            assert rt.hipMemcpy(got.ctypes.data, pairs, got.nbytes, 2) == 0
        want = oracle.find_putative_matches(L, R, ms, mr)
        assert np.array_equal(got, want.reshape(-1, 2))
        assert np.array_equal(np.asarray(m.get_matches()).reshape(-1, 2), want.reshape(-1, 2))
    m.close()


def _flooded_images(large, seed):
    """uint8 images of uneven pairs, some of nearly equal rows on both sides: a small pair, whose
    features are listed and re-checked within the bound, and with `large` pairs past it."""
    rng = np.random.default_rng(seed)
    images, shares = [], []
    sizes = [(300, 700), (512, 480), (640, 513), (32, 32)] + ([(2080, 2048), (1504, 1700)] if large else [])
    for p, (nL, nR) in enumerate(sizes):
        a, b, _ = synth.make_pair(nL, nR, 0.5, config=3, pair=seed + p)
        share = {1: 1.0, 4: 0.4, 5: 1.0}.get(p, 0.0)
        c = synth.dequantise(a[:1])
        out = []
        for q in (a.copy(), b.copy()):
            k = int(share * len(q))
            at = rng.permutation(len(q))[:k]
            q[at] = np.rint(512 * _unit(np.abs(c + 0.02 * rng.standard_normal((k, 128))))).clip(0, 255)
            out.append(q)
        images += out
        shares.append(share)
    return images, shares


def _oracle_batch(images, min_score, min_ratio):
    want = []
    for p in range(len(images) // 2):
        L, R = (synth.dequantise(q[:len(q) // 32 * 32]) for q in images[2 * p:2 * p + 2])
        want.append(oracle.find_putative_matches(L, R, min_score, min_ratio).reshape(-1, 2))
    return want


@pytest.mark.parametrize("large", [False, True])
@pytest.mark.parametrize("dtype", ["u8", "f32"])
@pytest.mark.parametrize("cache", [False, True])
@pytest.mark.parametrize("mode", ["fp32", "learned"])
def test_batch_many_candidates(large, dtype, cache, mode):
    """Batches with flooded pairs, in the plain form and as the pairs that a learned run hands over
    (a constant code): the oracle's matches from the first run, from graph replays, without graphs,
    with thresholds that take the full pass in between, and with settings changed between a run
    and its reading."""
    from v3dmatch import learned
    print(f"case batch flooded large {large} {dtype} cache {cache} {mode}", flush=True)
    images, shares = _flooded_images(large, 900)
    left = np.arange(0, len(images), 2, dtype=np.int32)
    m = v3dmatch.SIFT_Matching(0)
    m.batch_set_images([len(q) for q in images],
                       np.concatenate(images if dtype == "u8" else [synth.dequantise(q) for q in images]))
    m.batch_set_pairs(left, left + 1)
    m.set_derived_cache(cache)
    if mode == "learned":
        net = learned.Network(m)
        params = learned.init_params(3)
        params["W2"][:] = 0.0
        params["b2"][:] = 1.0
        net.set_params(params)
        net.set_code_scale(60.0)
        m.set_learned_topk(1)
        m.set_fallback(128, 1.0)
        m.set_precision(v3dmatch.PREC_LEARNED)
    handed = 0
    for ms, mr, graph in ((0.9, -1.0, True), (0.9, 0.8, True), (0.9, -1.0, True), (0.2, -1.0, True),
                          (0.9, -1.0, False), (0.9, -1.0, True)):
        m.batch_use_graph(graph)
        m.batch_match_async(ms, mr)
        m.set_certification(0.25)
        offs, pairs = m.batch_get_matches()
        again = m.batch_get_matches()
        m.set_certification(2.0 ** -15)
        assert np.array_equal(offs, again[0]) and np.array_equal(pairs, again[1])
        flags = m.batch_get_fallback() if mode == "learned" else np.ones(len(left), int)
        handed += int(flags.sum())
        for p, w in enumerate(_oracle_batch(images, ms, mr)):
            if flags[p]:
                assert np.array_equal(pairs[offs[p]:offs[p + 1]], w), (p, ms, mr, graph)
    assert handed >= 6 * len(left) // 2
    if mode == "fp32":
        assert m.batch_time_dominant_kernel(2) > 0
        got = m.batch_match(0.9, -1.0)
        assert all(np.array_equal(g, w) for g, w in zip(got, _oracle_batch(images, 0.9, -1.0)))
    m.close()


def test_batch_long_lists():
    """Pairs large enough that a wave's run of right tiles holds more candidates than a single pair's
    lists do (a small cluster on both sides), against the exact decisions of one pair."""
    n, share = 12288, 0.045
    print(f"case batch long lists {n} share {share}", flush=True)
    rng = np.random.default_rng(31)
    a, b, _ = synth.make_pair(n, n, 0.4, config=3, pair=950)
    c = synth.dequantise(a[:1])
    images = []
    for q in (a.copy(), b.copy()):
        k = int(share * n)
        q[rng.permutation(n)[:k]] = np.rint(512 * _unit(np.abs(c + 0.02 * rng.standard_normal((k, 128))))).clip(0, 255)
        images.append(q)
    one = v3dmatch.SIFT_Matching(0)
    one.allocate(n, n)
    one.set_left_u8(images[0])
    one.set_right_u8(images[1])
    one.set_certification(0.0)
    want = one.find_putative_matches_array(0.9, 0.8)
    assert one.stats()["nRechecked"] == 2 * n
    one.close()
    m = v3dmatch.SIFT_Matching(0)
    m.batch_set_images([n, n], np.concatenate(images))
    m.batch_set_pairs([0] * 16, [1] * 16)
    for _ in range(2):
        for got in m.batch_match(0.9, 0.8):
            assert np.array_equal(got, want)
    m.close()
