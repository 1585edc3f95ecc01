"""GPU tests of the plain form's score pass on FP16 parts (csrc/v3dm_split.hip) against the
oracle at the edges of its tiles (32 right features, 32-feature column blocks, 256-feature
work-groups, splits of the right features), at the edge of its range rule (row norms of 0 or
in [2^-10, 2); any other set takes the FP32 instruction), for every source of the rows, and
with thresholds that make it look for every position.

The match set and the per-feature decisions must equal the oracle's.  The pass's scores must
lie within 2^-18 |q| |c| of FP64: parts that keep 2^-22 of each component and a dropped
product of 2^-22, 24 FP32 accumulations of at most 2^-23 each: 3 * 2^-22 + 24 * 2^-23 < 2^-18
(v3dm_split.h), and 2^-39 sqrt(128) (|q| + |c|) from the smallest FP16 number.
"""
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
    m.allocate(2304, 2304)
    yield m
    m.close()


def _pair(nL, nR, seed):
    qL, qR, _ = synth.make_pair(nL, nR, 0.5, config=1, pair=seed)
    return synth.dequantise(qL), synth.dequantise(qR)


def _check(m, L, R, min_score=0.9, min_ratio=0.8):
    got = m.find_putative_matches_array(min_score, min_ratio)
    assert np.array_equal(got, oracle.find_putative_matches(L, R, min_score, min_ratio))
    cm, rm = m.get_maxima()
    S = oracle.scores(L, R)
    assert np.array_equal(cm, oracle.column_maxima(S, min_score, min_ratio))
    assert np.array_equal(rm, oracle.row_maxima(S, min_score, min_ratio))
    return got


def _set(m, L, R):
    m.setLeftFeatures(L.shape[0], L)
    m.setRightFeatures(R.shape[0], R)


@pytest.mark.parametrize("nL,nR", [(32, 32), (64, 32), (32, 64), (96, 96), (224, 64), (256, 2304), (288, 32),
                                   (320, 992), (2304, 32), (2272, 2080)])
@pytest.mark.parametrize("min_score,min_ratio", [(0.9, 0.8), (-2.0, -1.0), (0.4, 0.99)])
def test_tile_edges(matcher, nL, nR, min_score, min_ratio):
    L, R = _pair(nL, nR, nL + nR)
    _set(matcher, L, R)
    _check(matcher, L, R, min_score, min_ratio)


@pytest.mark.parametrize("factor", [2.0 ** -9, 2.0 ** -11, 1.875, 2.5, 2.0 ** -70, 2.0 ** 40])
@pytest.mark.parametrize("both", [True, False])
def test_range_rule(matcher, factor, both):
    """Scaled sets on both sides of the range rule (2^-11, 2.5, 2^-70 and 2^40 are outside)."""
    L, R = _pair(352, 416, 3)
    L = (L * np.float32(factor)).astype(np.float32)
    R = (R * np.float32(factor)).astype(np.float32) if both else R
    _set(matcher, L, R)
    scale = factor * factor if both else factor
    _check(matcher, L, R, 0.9 * scale, -1.0)
    _check(matcher, L, R, 0.9, 0.8)


@pytest.mark.parametrize("row", ["nan", "inf", "zero", "tiny"])
def test_special_rows(matcher, row):
    L, R = _pair(96, 128, 4)
    value = {"nan": np.nan, "inf": np.inf, "zero": 0.0, "tiny": 1e-20}[row]
    L[17], R[40] = value, value
    _set(matcher, L, R)
    _check(matcher, L, R)


def test_equal_rows(matcher):
    """Exact duplicates: the first index of an ascending scan, and no match under a ratio."""
    L, R = _pair(160, 192, 5)
    L[33:64] = L[32]
    R[64:192:32] = R[5]
    R[100] = L[32]
    _set(matcher, L, R)
    _check(matcher, L, R, 0.5, -1.0)
    _check(matcher, L, R)


@pytest.mark.parametrize("source", ["device", "device_odd", "pinned", "u8"])
@pytest.mark.parametrize("n", [32, 288, 2080])
def test_row_sources(matcher, source, n):
    """The rows read from device memory, from a device address aligned to 4 bytes only, from
    pinned host memory handed over as a device pointer, and from uint8 components."""
    qL, qR, _ = synth.make_pair(n, n, 0.5, config=1, pair=n)
    L, R = synth.dequantise(qL), synth.dequantise(qR)
    if source == "u8":
        matcher.set_left_u8(qL)
        matcher.set_right_u8(qR)
        _check(matcher, L, R)
        return
    rt = C.CDLL("libamdhip64.so")
    rt.hipMalloc.argtypes = rt.hipHostMalloc.argtypes = [C.POINTER(C.c_void_p), C.c_size_t]
    rt.hipHostMalloc.argtypes = [C.POINTER(C.c_void_p), C.c_size_t, C.c_uint]
    rt.hipMemcpy.argtypes = [C.c_void_p, C.c_void_p, C.c_size_t, C.c_int]
    rt.hipFree.argtypes = rt.hipHostFree.argtypes = [C.c_void_p]
    held = []
    for a, put in ((L, matcher.set_left_device), (R, matcher.set_right_device)):
        p = C.c_void_p()
        assert (rt.hipHostMalloc(C.byref(p), a.nbytes + 16, 0) if source == "pinned"
                else rt.hipMalloc(C.byref(p), a.nbytes + 16)) == 0
        at = p.value + (4 if source == "device_odd" else 0)
        assert rt.hipMemcpy(at, a.ctypes.data, a.nbytes, 0 if source == "pinned" else 1) == 0
        put(n, at)
        held.append(p)
    _check(matcher, L, R)
    for p in held:
        (rt.hipHostFree if source == "pinned" else rt.hipFree)(p)


@pytest.mark.parametrize("kind", ["sift", "spread", "signed", "sparse"])
def test_score_error(matcher, kind):
    rng = np.random.default_rng(9)
    L, R = _pair(1024, 1024, 6)
    if kind == "spread":  # norms over the whole range
        L = L * np.exp2(rng.uniform(-9.9, 0.9, (1024, 1))).astype(np.float32)
        R = R * np.exp2(rng.uniform(-9.9, 0.9, (1024, 1))).astype(np.float32)
    elif kind == "signed":
        L, R = (rng.standard_cauchy((1024, 128)) for _ in range(2))
    elif kind == "sparse":
        L, R = L * (rng.random(L.shape) < 0.1) + 1e-5, R * (rng.random(R.shape) < 0.1) + 1e-5
    if kind in ("signed", "sparse"):
        L, R = (x / np.linalg.norm(x, axis=1, keepdims=True) for x in (L, R))
    L, R = L.astype(np.float32), R.astype(np.float32)
    _set(matcher, L, R)
    got = matcher.score_block(v3dmatch.PREC_FP32, 1024, 1024).astype(np.float64)
    nq = np.linalg.norm(L.astype(np.float64), axis=1)[:, None]
    nc = np.linalg.norm(R.astype(np.float64), axis=1)[None, :]
    err = np.abs(got - L.astype(np.float64) @ R.astype(np.float64).T)
    assert (err <= 2.0 ** -18 * nq * nc + 2.0 ** -39 * np.sqrt(128) * (nq + nc)).all()


def _batch(sizes, seed):
    images = []
    for p, (nL, nR) in enumerate(sizes):
        qL, qR, _ = synth.make_pair(nL, nR, 0.5, config=3, pair=100 * seed + p)
        images += [qL, qR]
    left = np.arange(0, 2 * len(sizes), 2, dtype=np.int32)
    return images, left, left + 1


def _want(images, left, right, min_score, min_ratio):
    out = []
    for a, b in zip(left, right):
        L, R = images[a][:len(images[a]) // 32 * 32], images[b][:len(images[b]) // 32 * 32]
        out.append(oracle.find_putative_matches(L, R, min_score, min_ratio) if len(L) and len(R)
                   else np.zeros((0, 2), np.int32))
    return out


SIZES = [(33, 70), (512, 31), (256, 256), (300, 1700), (1056, 96), (32, 32), (640, 513)]


@pytest.mark.parametrize("dtype", ["u8", "f32", "f32_wide", "f32_nan"])
@pytest.mark.parametrize("rows", [128, 256])
def test_batch_split(dtype, rows):
    """Batches of uint8 images (integer rows), of FP32 images (split rows), and of images with
    rows outside the range (the FP32 instruction), in both work-group shapes, with the rows made
    by every run and kept."""
    qs, left, right = _batch(SIZES, 1)
    images = [synth.dequantise(q) for q in qs]
    if dtype == "f32_wide":
        images[3] = images[3] * np.float32(2.0 ** 30)
    elif dtype == "f32_nan":
        images[4][7] = np.nan
    m = v3dmatch.SIFT_Matching(0)
    m.batch_set_images([len(q) for q in qs], np.concatenate(qs if dtype == "u8" else images))
    m.batch_set_pairs(left, right)
    m.batch_set_tile_shape(v3dmatch.PREC_FP32, rows)
    for cache in (False, True):
        m.set_derived_cache(cache)
        for tiles, score, ratio in ((1, 0.9, 0.8), (3, 0.9, 0.8), (3, -2.0, -1.0)):
            m.batch_set_tuning(False, v3dmatch.PREC_FP32, tiles, 64)
            for got, want in zip(m.batch_match(score, ratio), _want(images, left, right, score, ratio)):
                assert np.array_equal(got, want)
    m.close()


@pytest.mark.parametrize("dtype", ["u8", "f32"])
@pytest.mark.parametrize("cache", [False, True])
@pytest.mark.parametrize("plain_first", [False, True])
def test_batch_fallback_split(dtype, cache, plain_first):
    """The pairs that a learned run hands to the plain form (a constant code with one
    candidate per query) get the exact matches, with the sieve's rows made for them alone or left
    by a plain run of the same images (the full pass: test_batch_fallback_full_pass)."""
    from v3dmatch import learned
    qs, left, right = _batch(SIZES, 2)
    images = [synth.dequantise(q) for q in qs]
    m = v3dmatch.SIFT_Matching(0)
    m.batch_set_images([len(q) for q in qs], np.concatenate(qs if dtype == "u8" else images))
    m.batch_set_pairs(left, right)
    m.set_derived_cache(cache)
    net = learned.Network(m)
    params = learned.init_params(3)
    params["W2"][:] = 0.0  # the same code for every descriptor: its candidates are arbitrary
    params["b2"][:] = 1.0
    net.set_params(params)
    net.set_code_scale(60.0)
    m.set_learned_topk(1)
    m.set_fallback(128, 1.0)
    want = _want(images, left, right, 0.9, 0.8)
    for mode in ([v3dmatch.PREC_FP32] if plain_first else []) + [v3dmatch.PREC_LEARNED] * 2:
        m.set_precision(mode)
        res = m.batch_match(0.9, 0.8)
        flags = m.batch_get_fallback() if mode == v3dmatch.PREC_LEARNED else np.ones(len(want), int)
        for p, w in enumerate(want):
            if flags[p]:
                assert np.array_equal(res[p], w)
    assert flags.sum() >= 1
    m.close()


@pytest.mark.parametrize("tiles", [64, 1 << 30])
def test_batch_image_of_many_rows(tiles):
    """An image whose split rows span more than 4 GiB: features past row 2^23 are scored by their
    own rows (the zero rows between score 0 and change no decision).  One work unit's tiles are
    bounded whatever the caller asks for."""
    n, far = 2 ** 23 + 96, 2 ** 23
    qL, qR, _ = synth.make_pair(96, 96, 0.6, config=1, pair=71)
    _, near, _ = synth.make_pair(96, 96, 0.6, config=1, pair=72)
    L, R = synth.dequantise(qL), np.concatenate([synth.dequantise(near), synth.dequantise(qR)])
    rows = np.zeros((96 + n, 128), np.float32)
    rows[:96], rows[96:192], rows[96 + far:] = L, R[:96], R[96:]
    m = v3dmatch.SIFT_Matching(0)
    m.batch_set_images([96, n], rows)
    del rows
    m.batch_set_pairs([0], [1])
    m.batch_set_tuning(False, v3dmatch.PREC_FP32, tiles, 512)
    print(f"case split image of 2^23 + 96 rows, {tiles} tiles an item", flush=True)
    got = m.batch_match(0.2, 0.8)[0]
    m.close()
    want = oracle.find_putative_matches(L, R, 0.2, 0.8)
    want[:, 1] += np.where(want[:, 1] >= 96, far - 96, 0)
    assert len(want) > 20 and np.array_equal(got, want)


@pytest.mark.parametrize("capacity", [96, 384, 2085])
def test_u8_odd_capacity(capacity):
    """uint8 pairs of a handle whose buffers hold an odd number of 128-row blocks, at thresholds
    that take the full pass on integer rows: its last work-group loads whole blocks of scales."""
    print(f"case integer rows, capacity {capacity}", flush=True)
    m = v3dmatch.SIFT_Matching(0)
    m.enableRoundingWarning(False)
    m.allocate(capacity, capacity)
    n = capacity // 32 * 32
    qL, qR, _ = synth.make_pair(n, n, 0.5, config=1, pair=capacity)
    m.set_left_u8(qL)
    m.set_right_u8(qR)
    _check(m, synth.dequantise(qL), synth.dequantise(qR), 0.4, 0.99)
    _check(m, synth.dequantise(qL), synth.dequantise(qR), -2.0, -1.0)
    m.close()


@pytest.mark.parametrize("n,copies", [(256, 33), (1536, 1001), (4096, 3001), (2304, 2304)])
@pytest.mark.parametrize("guided", [False, True])
def test_many_open_queries(n, copies, guided):
    """Exact copies score 1, which the certified rule leaves open: re-checks of one, four and eight
    queries a unit, with a partial last group, and with removed pairs of a guided call."""
    print(f"case open queries {copies} of {n} guided {guided}", flush=True)
    L, R = _pair(n, n, 12)
    R[:copies] = L[np.random.default_rng(5).permutation(n)[:copies]]
    m = v3dmatch.SIFT_Matching(0)
    m.enableRoundingWarning(False)
    m.allocate(n, n, guided)
    _set(m, L, R)
    got = m.find_putative_matches_array(0.2, 0.8)
    S = oracle.scores(L, R)
    assert np.array_equal(got, oracle.find_putative_matches(L, R, 0.2, 0.8))
    assert m.stats()["nRechecked"] >= 2 * copies
    if guided:
        rng = np.random.default_rng(6)
        lxy, rxy = (rng.uniform(0, 1000, (n, 2)).astype(np.float32) for _ in range(2))
        H = np.eye(3)
        got = m.run_guided_array(True, H, 600.0, lxy, rxy, 0.2, 0.8)
        assert np.array_equal(got, oracle.guided(S, 1, H, np.float32(600.0), lxy, rxy, 0.2, 0.8))
    m.set_certification(0.0)
    assert np.array_equal(m.find_putative_matches_array(0.9, 0.8), oracle.find_putative_matches(L, R, 0.9, 0.8))
    assert m.stats()["nRechecked"] == 2 * n
    m.close()


# Thresholds that the sieve refuses (v3dm_sieve.h): these tests run the full pass.
FULL = [(0.4, 0.99), (0.2, 0.8)]


@pytest.mark.parametrize("nL,nR", [(32, 32), (64, 288), (288, 64), (256, 256), (544, 1056), (2272, 2080)])
@pytest.mark.parametrize("min_score,min_ratio", FULL + [(-2.0, -1.0)])
@pytest.mark.parametrize("sides", ["both", "left"])
def test_u8_full_pass(matcher, nL, nR, min_score, min_ratio, sides):
    """uint8 sets in the full pass: integer rows where both sides are uint8, split rows made from
    dequantised rows where one is."""
    print(f"case full pass u8 {sides} {nL} x {nR} min {min_score} ratio {min_ratio}", flush=True)
    qL, qR, _ = synth.make_pair(nL, nR, 0.5, config=1, pair=nL + 3 * nR)
    L, R = synth.dequantise(qL), synth.dequantise(qR)
    matcher.set_left_u8(qL)
    if sides == "both":
        matcher.set_right_u8(qR)
    else:
        matcher.setRightFeatures(nR, R)
    _check(matcher, L, R, min_score, min_ratio)


@pytest.mark.parametrize("dtype", ["u8", "f32"])
@pytest.mark.parametrize("cache", [False, True])
@pytest.mark.parametrize("plain_first", [False, True])
def test_batch_fallback_full_pass(dtype, cache, plain_first):
    """test_batch_fallback_split at thresholds that refuse the sieve: the handed-over pairs' rows,
    the pass over their listed items, the masked merge and the re-check, with the split rows made
    for them alone or left by a plain run of the same images, and in turn with the sieve."""
    from v3dmatch import learned
    qs, left, right = _batch(SIZES, 2)
    images = [synth.dequantise(q) for q in qs]
    m = v3dmatch.SIFT_Matching(0)
    m.batch_set_images([len(q) for q in qs], np.concatenate(qs if dtype == "u8" else images))
    m.batch_set_pairs(left, right)
    m.set_derived_cache(cache)
    net = learned.Network(m)
    params = learned.init_params(3)
    params["W2"][:] = 0.0  # the same code for every descriptor: its candidates are arbitrary
    params["b2"][:] = 1.0
    net.set_params(params)
    net.set_code_scale(60.0)
    m.set_learned_topk(1)
    m.set_fallback(128, 1.0)
    for score, ratio in FULL + [(0.9, 0.8)] + FULL:
        print(f"case fallback full pass {dtype} cache {cache} first {plain_first} min {score} ratio {ratio}", flush=True)
        want = _want(images, left, right, score, ratio)
        for mode in ([v3dmatch.PREC_FP32] if plain_first else []) + [v3dmatch.PREC_LEARNED] * 2:
            m.set_precision(mode)
            res = m.batch_match(score, ratio)
            flags = m.batch_get_fallback() if mode == v3dmatch.PREC_LEARNED else np.ones(len(want), int)
            for p, w in enumerate(want):
                if flags[p]:
                    assert np.array_equal(res[p], w), (p, score, ratio, mode)
        assert flags.sum() >= 1
    m.close()


@pytest.mark.parametrize("dtype", ["u8", "f32"])
@pytest.mark.parametrize("rows", [128, 256])
def test_batch_shapes_full_pass(dtype, rows):
    """Work-group shapes, items and grids of the full pass, at thresholds where a run takes it."""
    qs, left, right = _batch(SIZES, 4)
    images = [synth.dequantise(q) for q in qs]
    m = v3dmatch.SIFT_Matching(0)
    m.batch_set_images([len(q) for q in qs], np.concatenate(qs if dtype == "u8" else images))
    m.batch_set_pairs(left, right)
    m.batch_set_tile_shape(v3dmatch.PREC_FP32, rows)
    for score, ratio in FULL:
        want = _want(images, left, right, score, ratio)
        for tiles, grid in ((0, 0), (1, 7), (5, 300), (64, 1024)):
            print(f"case full pass {dtype} rows {rows} tiles {tiles} grid {grid} min {score}", flush=True)
            m.batch_set_tuning(False, v3dmatch.PREC_FP32, tiles, grid)
            for got, w in zip(m.batch_match(score, ratio), want):
                assert np.array_equal(got, w)
            assert m.batch_get_tile_shape(v3dmatch.PREC_FP32)["query_rows"] == rows
    m.close()
