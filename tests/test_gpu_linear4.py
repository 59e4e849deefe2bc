"""uint4 group-64 projection routes on the GPU (tessery test_kernels.py:55-81, 421-516, 648-776):
float64 accuracy at atol = rtol = 5e-5, the expected route partition, bit-identical results
between routes over the same rows, and rows outside a route's region left untouched."""

import numpy as np
import pytest

from oracle import quant4 as ref
from tessery_amd.workloads import bf16_values, bf16_words
from tests.conftest import GOLDEN
from tests.test_gpu_attention import run

pytestmark = pytest.mark.gpu


def make(seed, m, n, k, cancellation=False):
    rng = np.random.default_rng(seed)
    codes = rng.integers(0, 16, size=(n, k), dtype=np.uint32)
    x = rng.normal(size=(m, k)).astype(np.float32)
    if cancellation:
        codes[:, 1::2] = codes[:, ::2]
        x[:, ::2], x[:, 1::2] = 1.0, -1.0
    scales = bf16_words(rng.uniform(0.01, 0.2, size=(n, k // 64)))
    biases = bf16_words(rng.uniform(-1, 0.1, size=(n, k // 64)))
    return x, ref.pack(codes), scales, biases


def project(engine, arrays, m, n, k, out=None):
    bufs = [engine.upload(a) for a in arrays]
    bufs.append(engine.upload(out) if out is not None else engine.buffer(m * n * 4))
    try:
        with engine.command():
            engine._linear4(bufs, rows=m, cols=n, k=k)
        shape = out.shape if out is not None else (m, n)
        return engine.read(bufs[-1], shape)
    finally:
        for b in bufs:
            b.close()


def test_fixture_and_known_answer(runtime):
    f = np.load(GOLDEN / "linear4_small.npz")
    got = project(runtime, [f["x"], f["packed"], f["scales"], f["biases"]], 7, 64, 128)
    np.testing.assert_allclose(got, f["expected"], atol=5e-5, rtol=5e-5)
    # scale 0.125 bias -0.5 (test_kernels.py:55-81) through the scalar route
    rng = np.random.default_rng(1)
    code = rng.integers(0, 16, size=(8, 128), dtype=np.uint32)
    x = rng.normal(size=(3, 128)).astype(np.float32)
    arrays = [x, ref.pack(code), bf16_words(np.full((8, 2), 0.125)), bf16_words(np.full((8, 2), -0.5))]
    got = run(runtime, "linear4", arrays, (3, 8), threads=8 * 32, group_size=32, rows=3, cols=8, k=128)
    np.testing.assert_allclose(got, x @ (code * 0.125 - 0.5).T, atol=1e-5, rtol=1e-5)


@pytest.mark.parametrize("m,n,k", [(m, 64, k) for m in (1, 2, 7, 8, 9, 12, 15, 16, 17, 31)
                                   for k in (64, 1024, 3072)] + [(7, 33, 128)])
def test_tiled_accuracy_and_route(runtime, m, n, k):
    x, packed, scales, biases = make(417, m, n, k)
    got = project(runtime, [x, packed, scales, biases], m, n, k)
    np.testing.assert_allclose(got, ref.linear4(x, packed, scales, biases), atol=5e-5, rtol=5e-5)
    expected = {"linear4": 1}
    if m >= 5 and n % 32 == 0:
        expected = {}
        if m >= 8:
            expected["linear4_tiled"] = 1
        if m % 8:
            expected["linear4" if m % 8 <= 4 else "linear4_tail"] = 1
    assert runtime.diagnostics()["dispatches"] == expected


@pytest.mark.parametrize("m,n,k", [(16, 1024, 1024), (32, 2048, 1024), (16, 3072, 1024),
                                   (32, 1024, 2048), (32, 1024, 3072), (4096, 1024, 1024)])
@pytest.mark.parametrize("pattern", ["random", "cancellation"])
def test_large_tiles_f64_and_bitwise_between_routes(runtime, m, n, k, pattern):
    arrays = list(make(821, m, n, k, pattern == "cancellation"))
    previous = run(runtime, "linear4_tiled", arrays, (m, n), threads=(m // 8) * (n // 32) * 128,
                   group_size=128, rows=m, cols=n, k=k)
    actual = run(runtime, "linear4_16x32_k64", arrays, (m, n), threads=(m // 16) * (n // 32) * 256,
                 group_size=256, rows=m, cols=n, k=k)
    np.testing.assert_allclose(actual, ref.linear4(*arrays), atol=5e-5, rtol=5e-5)
    np.testing.assert_array_equal(actual, previous)


@pytest.mark.parametrize("m", [17, 23, 24, 25, 31, 40, 128, 129, 257])
@pytest.mark.parametrize("n,k", [(1024, 1024), (2048, 1024), (1024, 3072)])
def test_mixed_partition_matches_f64_and_previous_routes(runtime, m, n, k):
    arrays = list(make(481 + m, m, n, k))
    sentinel = np.full((m, n), np.nan, np.float32)
    actual = project(runtime, arrays, m, n, k, out=sentinel)
    np.testing.assert_allclose(actual, ref.linear4(*arrays), atol=5e-5, rtol=5e-5)
    bufs = [runtime.upload(a) for a in arrays] + [runtime.upload(sentinel)]
    try:
        with runtime.command():
            runtime._dispatch("linear4_tiled", bufs, threads=(m // 8) * (n // 32) * 128,
                              group_size=128, rows=m, cols=n, k=k)
            if m % 8:
                small = m % 8 <= 4
                runtime._dispatch("linear4" if small else "linear4_tail", bufs,
                                  threads=n * 32 if small else (n // 32) * 128,
                                  group_size=32 if small else 128, n=m // 8 * 8, rows=m, cols=n, k=k)
        previous = runtime.read(bufs[-1], (m, n))
    finally:
        for b in bufs:
            b.close()
    np.testing.assert_array_equal(actual, previous)


@pytest.mark.parametrize("m", [2, 3, 4])
def test_small_row_routes_and_output_guard(runtime, m):
    n, k = 1024, 1024
    arrays = list(make(2030 + m, m, n, k))
    sentinel = np.full((m + 2, n), np.nan, np.float32)
    got = project(runtime, arrays, m, n, k, out=sentinel)
    assert np.isnan(got[m:]).all()
    np.testing.assert_allclose(got[:m], ref.linear4(*arrays), atol=5e-5, rtol=5e-5)
    assert runtime.diagnostics()["dispatches"] == {"linear4_small3" if m == 3 else "linear4": 1}


def test_eight_row_offset_preserves_surrounding_rows(runtime):
    m, n, k = 32, 32, 64
    arrays = [np.ones((m, k), np.float32), np.full((n, k // 8), 0x11111111, np.uint32),
              bf16_words(np.ones((n, 1))), bf16_words(np.zeros((n, 1)))]
    bufs = [runtime.upload(a) for a in arrays] + [runtime.upload(np.full((m, n), np.nan, np.float32))]
    try:
        with runtime.command():
            runtime._dispatch("linear4_tiled", bufs, threads=128, group_size=128, n=16, rows=m,
                              cols=n, k=k)
        out = runtime.read(bufs[-1], (m, n))
    finally:
        for b in bufs:
            b.close()
    assert np.isnan(out[:16]).all() and np.isnan(out[24:]).all()
    np.testing.assert_array_equal(out[16:24], 64)


@pytest.mark.parametrize("m,n,k", [(1024, 2048, 1024), (1100, 1024, 2048), (2048, 1024, 1024),
                                   (4096, 3072, 1024), (2050, 1024, 3072),
                                   (2176, 128, 64), (4097, 2048, 1024)])
def test_large_batch_fp16_mfma_path(runtime, m, n, k):
    """From 1024 rows the projection runs on fp16 MFMA over row-scaled hi + lo halves of x. Row
    magnitudes spread over 2^-20 .. 2^20, a zero row, rows near fp32's smallest and largest
    normal values (beyond fp16's range): every output stays within fp32-grade error of the
    float64 product, measured against sum_k |x| |w| of the same element."""
    x, packed, scales, biases = make(907 + m + n, m, n, k)
    rng = np.random.default_rng(m)
    x[5:] *= np.exp2(rng.integers(-20, 21, m - 5)).astype(np.float32)[:, None]
    x[0] = 0.0
    x[1] *= np.float32(1e-36)
    x[2] *= np.float32(1e6)
    x[3] *= np.float32(1e34)
    got = project(runtime, [x, packed, scales, biases], m, n, k)
    w = ref.dequantize(packed, scales, biases, k)
    want = x.astype(np.float64) @ w.T
    bound = np.abs(x).astype(np.float64) @ np.abs(w).T
    assert np.isfinite(got).all()
    err = np.abs(got - want)
    assert np.all(err <= 2e-6 * bound + 1e-37), float((err / (bound + 1e-300)).max())
    assert not np.any(got[0])


# Rows and columns at the edges of the 32 x 32 tiles, one to four of them a workgroup (up to 256
# tiles, up to 512, more), and K of 1, 3, 7, 17 and 48 groups: fewer than the eight partitions,
# uneven ones, odd counts (scales and biases at both parities of a dword).
@pytest.mark.parametrize("m,n,k", [(1, 8, 64), (31, 33, 192), (32, 96, 448), (33, 160, 1088),
                                   (65, 1056, 1088), (257, 1024, 3072), (255, 1031, 64),
                                   (289, 2080, 448), (1023, 128, 192), (1030, 1056, 192)])
def test_split_bf16_rows_kernel_at_its_edges(runtime, m, n, k):
    """Every output within 1e-6 of sum_k |x| |w| of float64 (fp32 sums of exact products: an error
    of a few 2^-24 a partial sum, at most 96 of them), rows past the range untouched; row
    magnitudes spread over 2^-20 .. 2^20."""
    x, packed, scales, biases = make(55 + m + k, m, n, k)
    x *= np.exp2(np.random.default_rng(m).integers(-20, 21, m)).astype(np.float32)[:, None]
    got = project(runtime, [x, packed, scales, biases], m, n, k,
                  out=np.full((m + 1, n), np.nan, np.float32))
    assert np.isnan(got[m:]).all()
    w = ref.dequantize(packed, scales, biases, k)
    err = np.abs(got[:m] - x.astype(np.float64) @ w.T)
    bound = 1e-6 * (np.abs(x).astype(np.float64) @ np.abs(w).T)
    assert np.all(err <= bound), float((err / bound).max())


@pytest.mark.parametrize("m,seq_of_ops", [(24, "norm"), (77, "norm"), (24, "add"), (308, "add"),
                                          (37, "gated"), (24, "gated"), (200, "gated")])
def test_projections_beside_each_other_keep_their_bits(runtime, m, seq_of_ops):
    """q, k and v (and gate, up, silu_gate, down) queued in one command, after the norm that makes
    their input, run as fewer launches than queued one by one, on activations that the launch
    before split; every buffer holds the bits of separate commands."""
    hidden, inter = 1024, 3072
    rng = np.random.default_rng(m)
    x, r = [rng.normal(size=(m, hidden)).astype(np.float32) for _ in range(2)]
    gamma = bf16_words(rng.uniform(0.5, 1.5, hidden))

    def weights(n, k):
        return [ref.pack(rng.integers(0, 16, size=(n, k), dtype=np.uint32)),
                bf16_words(rng.uniform(0.01, 0.2, size=(n, k // 64)) / 8),
                bf16_words(rng.uniform(-1, 0.1, size=(n, k // 64)) / 8)]

    sets = ([weights(inter, hidden), weights(inter, hidden), weights(hidden, inter)]
            if seq_of_ops == "gated" else [weights(n, hidden) for n in (2048, 1024, 1024)])
    results = []
    for separate in (False, True):
        bufs = [runtime.upload(a) for a in (x, r, gamma)]
        wb = [[runtime.upload(a) for a in w] for w in sets]
        h = runtime.buffer(x.nbytes)
        outs = [runtime.buffer(m * w[0].shape[0] * 4) for w in sets]
        steps = []
        if seq_of_ops == "add":
            steps.append(lambda: runtime._dispatch("add", [bufs[0], bufs[1], bufs[0]],
                                                   threads=x.size, n=x.size))
        steps.append(lambda: runtime._dispatch("rms_norm", [bufs[0], bufs[2], h], threads=m * 32,
                                               group_size=32, cols=hidden, eps=1e-6))
        if seq_of_ops == "gated":
            steps.append(lambda: runtime._gated4([h, *wb[0], *wb[1], outs[0], outs[1]], rows=m,
                                                 cols=inter, k=hidden))
            steps.append(lambda: runtime._linear4([outs[0], *wb[2], outs[2]], rows=m, cols=hidden,
                                                  k=inter))
        else:
            for w, out, a in zip(wb, outs, sets):
                steps.append(lambda w=w, out=out, a=a: runtime._linear4(
                    [h, *w, out], rows=m, cols=a[0].shape[0], k=hidden))
        if separate:
            for step in steps:
                with runtime.command():
                    step()
        else:
            with runtime.command():
                for step in steps:
                    step()
        results.append([runtime.read(h, x.shape), *(runtime.read(o, (m, a[0].shape[0]))
                                                    for o, a in zip(outs, sets))])
        for b in [*bufs, *(b for w in wb for b in w), h, *outs]:
            b.close()
    for together, alone in zip(*results):
        np.testing.assert_array_equal(together, alone)
    xs = x.astype(np.float64) + (r if seq_of_ops == "add" else 0)
    want = xs / np.sqrt((xs * xs).mean(-1, keepdims=True) + 1e-6) * bf16_values(gamma)
    np.testing.assert_allclose(results[0][0], want, atol=1e-5, rtol=1e-5)


# Codes at one end of their range, or near it, against a bias that all but cancels them: w is far
# smaller than scale * code and bias. One to four column blocks a workgroup.
@pytest.mark.parametrize("m", [24, 300, 700])
@pytest.mark.parametrize("code,bias,odd", [(0, 2.0**-12, None), (15, -15 + 2.0**-4, None),
                                           (3, -3 + 2.0**-6, None), (12, -12 - 2.0**-4, None), (5, -5.0, None),
                                           (0, 2.0**-12, 15), (15, -15 + 2.0**-4, 0)])
def test_groups_whose_bias_cancels_their_codes(runtime, m, code, bias, odd):
    """Within 1e-6 of sum_k |x| |w| of float64, as for any other weights; `odd`: one code of another
    value per group, where x is zero. Scales of both signs and several magnitudes."""
    n, k = 1056, 448
    rng = np.random.default_rng(m + code)
    x = rng.normal(size=(m, k)).astype(np.float32)
    codes = np.full((n, k), code, np.uint32)
    if odd is not None:
        codes[:, 7::64] = odd
        x[:, 7::64] = 0.0
    scale = np.exp2(rng.integers(-12, 5, size=(n, k // 64))) * rng.choice((-1.0, 1.0), (n, k // 64))
    packed, scales, biases = ref.pack(codes), bf16_words(scale), bf16_words(scale * bias)
    got = project(runtime, [x, packed, scales, biases], m, n, k)
    w = ref.dequantize(packed, scales, biases, k)
    err = np.abs(got - x.astype(np.float64) @ w.T)
    bound = 1e-6 * (np.abs(x).astype(np.float64) @ np.abs(w).T)
    assert np.all(err <= bound), float((err / bound).max())


def test_bias_term_keeps_every_product_of_its_terms(runtime):
    """x and w whose second and third bf16 terms are as large as they get, all of one sign: the
    products of those terms are 2^-21 of the result. The sums here are exact up to a few roundings
    of the result (2^-24 each)."""
    m, n, k = 24, 64, 512
    x = np.full((m, k), 0x3f80ffff, np.uint32).view(np.float32)
    scales = bf16_words(np.full((n, k // 64), 2.0**-26))
    biases = bf16_words(np.full((n, k // 64), -1.0078125))
    packed = ref.pack(np.full((n, k), 15, np.uint32))
    got = project(runtime, [x, packed, scales, biases], m, n, k)
    want = x.astype(np.float64) @ ref.dequantize(packed, scales, biases, k).T
    assert np.all(np.abs(got - want) <= 2.5e-7 * np.abs(want)), float(np.abs(got / want - 1).max())


@pytest.mark.parametrize("m", [24, 300, 700])
def test_non_finite_activations_and_scales_give_what_fp32_gives(runtime, m):
    """An infinite or NaN activation makes its row, and a non-finite scale or bias its column, what
    sums of fp32 products give: infinities where no NaN and no opposite infinity takes part."""
    n, k = 1056, 448
    x, packed, scales, biases = make(m, m, n, k)
    x[1, 5], x[4, 100], x[m - 1, k - 1] = np.inf, np.nan, -np.inf
    scales[7, 2], biases[33, 0], biases[n - 1, 1] = 0x7f80, 0xff80, 0x7fc0
    got = project(runtime, [x, packed, scales, biases], m, n, k)
    with np.errstate(invalid="ignore"):
        codes = ((packed[:, :, None] >> np.arange(0, 32, 4, dtype=np.uint32)) & 15).reshape(n, k)
        w = (codes * np.repeat(bf16_values(scales), 64, 1)
             + np.repeat(bf16_values(biases), 64, 1)).astype(np.float64)
        special = np.zeros((m, n), bool)
        special[[1, 4, m - 1]] = True
        special[:, [7, 33, n - 1]] = True
        for r, c in zip(*np.nonzero(special)):
            want = np.float32(np.sum(x[r].astype(np.float64) * w[c]))
            assert (np.isnan(want) and np.isnan(got[r, c])) or got[r, c] == want, (r, c, got[r, c])
    rows, cols = ~special.all(1), ~special.all(0)
    np.testing.assert_allclose(got[rows][:, cols], x[rows].astype(np.float64) @ w[cols].T,
                               atol=2e-4, rtol=5e-5)


@pytest.mark.parametrize("k", [8192, 8256])
def test_large_batch_beyond_the_fp16_kernels_k(runtime, k):
    """From 1024 rows on, the longest K the fp16-MFMA kernel's scale words leave room for, and the next
    one, which the split-bf16 kernel takes (in row ranges that fit the planes scratch)."""
    m, n = 1024, 128
    x, packed, scales, biases = make(k, m, n, k)
    got = project(runtime, [x, packed, scales, biases], m, n, k)
    w = ref.dequantize(packed, scales, biases, k)
    err = np.abs(got - x.astype(np.float64) @ w.T)
    bound = 2e-6 * (np.abs(x).astype(np.float64) @ np.abs(w).T)
    assert np.all(err <= bound), float((err / bound).max())


@pytest.mark.parametrize("m", [1024, 1029, 4096])
@pytest.mark.parametrize("chain", ["norm", "add", "gated", "overwritten", "dense", "longer"])
def test_row_scales_left_for_large_projections_keep_their_bits(runtime, m, chain):
    """From 1024 rows a norm, and the first projection of an input, leave the row scales of that input
    for the projections after them. Queued in one command, every buffer holds the bits of a command
    for each launch: q, k and v after a norm, alone or with the add before it, or over more rows than
    they project; gate, up, silu_gate, down; with their input written anew in between; with a dense
    projection in between, which keeps its partial sums where the scales are. Rows from 2^-20 to 2^10
    with an eps of 1e-2, so that the normalized rows, and their scales, differ as much."""
    k, rows = 576, m + 71 if chain == "longer" else m
    rng = np.random.default_rng(m)
    x, r = [rng.normal(size=(rows, k)).astype(np.float32)
            * np.exp2(rng.integers(-20, 11, (rows, 1))).astype(np.float32) for _ in range(2)]
    z = rng.normal(size=(m, 128)).astype(np.float32) * np.exp2(rng.integers(-8, 9, (m, 1))).astype(np.float32)
    dense = [rng.normal(size=s).astype(np.float32) for s in ((65, 1536), (384, 1536))]
    gamma = bf16_words(rng.uniform(0.5, 1.5, k))

    def weights(n, width):
        return [ref.pack(rng.integers(0, 16, size=(n, width), dtype=np.uint32)),
                bf16_words(rng.uniform(0.01, 0.2, size=(n, width // 64)) / 8),
                bf16_words(rng.uniform(-1, 0.1, size=(n, width // 64)) / 8)]

    widths = {"gated": [(640, k), (640, k), (k, 640)], "overwritten": [(256, k), (k, 128), (128, k)]}
    sets = [weights(*s) for s in widths.get(chain, [(256, k), (128, k), (128, k)])]
    results = []
    for separate in (False, True):
        xb, rb, zb, gb = [runtime.upload(a) for a in (x, r, z, gamma)]
        wb = [[runtime.upload(a) for a in w] for w in sets]
        db = [runtime.upload(a) for a in dense] + [runtime.buffer(65 * 384 * 4)]
        h = runtime.buffer(x.nbytes)
        outs = [runtime.buffer(m * w[0].shape[0] * 4) for w in sets]

        def project(i, src, dst):
            n, words = sets[i][0].shape
            return lambda: runtime._linear4([src, *wb[i], dst], rows=m, cols=n, k=8 * words)

        steps = [lambda: runtime._dispatch("rms_norm", [xb, gb, h], threads=rows * 32, group_size=32,
                                           cols=k, eps=1e-2)]
        if chain == "add":
            steps.insert(0, lambda: runtime._dispatch("add", [xb, rb, xb], threads=x.size, n=x.size))
        if chain == "gated":
            steps += [project(0, h, outs[0]), project(1, h, outs[1]),
                      lambda: runtime._dispatch("silu_gate", outs[:2], threads=m * 640, n=m * 640),
                      project(2, outs[0], outs[2])]
        elif chain == "overwritten":
            steps += [project(0, h, outs[0]), project(1, zb, h), project(2, h, outs[2])]
        else:
            steps += [project(i, h, outs[i]) for i in range(3)]
        if chain == "dense":
            steps.insert(2, lambda: runtime._dispatch("matmul_f32", db, threads=68 // 4 * 384 * 32,
                                                      group_size=32, rows=65, cols=384, k=1536))
        if separate:
            for step in steps:
                with runtime.command():
                    step()
        else:
            with runtime.command():
                for step in steps:
                    step()
        results.append([runtime.read(h, x.shape), runtime.read(db[2], (65, 384)),
                        *(runtime.read(o, (m, w[0].shape[0])) for o, w in zip(outs, sets))])
        for b in [xb, rb, zb, gb, h, *db, *outs, *(b for w in wb for b in w)]:
            b.close()
    for together, alone in zip(*results):
        np.testing.assert_array_equal(together, alone)
    if chain != "gated":  # the last projection, of the input as it was by then
        w = ref.dequantize(*sets[2], k)
        hd = results[0][0][:m].astype(np.float64)
        err = np.abs(results[0][4] - hd @ w.T)
        assert np.all(err <= 2e-6 * (np.abs(hd) @ np.abs(w).T) + 1e-37)


@pytest.mark.parametrize("m,n,k", [(1000, 64, 8192), (1023, 40, 4096), (1056, 72, 8192)])
def test_wide_inputs_beyond_one_planes_scratch_keep_their_bits(runtime, m, n, k):
    """Inputs whose split form exceeds the scratch of the usual ones (one range in the wide scratch; the
    last more than that holds): rows hold the bits of launches of their own, within 2e-6 of
    sum_k |x| |w| of float64."""
    x, packed, scales, biases = make(m, m, n, k)
    got = project(runtime, [x, packed, scales, biases], m, n, k,
                  out=np.full((m + 1, n), np.nan, np.float32))
    assert np.isnan(got[m:]).all()
    for rows in (slice(0, 96), slice(m - 50, m)):
        alone = project(runtime, [x[rows], packed, scales, biases], len(x[rows]), n, k)
        np.testing.assert_array_equal(got[:m][rows], alone)
    w = ref.dequantize(packed, scales, biases, k)
    err = np.abs(got[:m] - x.astype(np.float64) @ w.T)
    assert np.all(err <= 2e-6 * (np.abs(x).astype(np.float64) @ np.abs(w).T))


@pytest.mark.parametrize("m", [24, 300, 700])
def test_groups_without_scale(runtime, m):
    """Scale 0, with and without a bias (a group of equal or zero weights): z is 0 or 15, and the bias
    alone counts."""
    n, k = 1056, 448
    x, packed, scales, biases = make(m, m, n, k)
    scales[::2, 1:4] = 0
    scales[1::3, 2] = 0x8000
    biases[::4, 1:3] = 0
    got = project(runtime, [x, packed, scales, biases], m, n, k)
    w = ref.dequantize(packed, scales, biases, k)
    err = np.abs(got - x.astype(np.float64) @ w.T)
    assert np.all(err <= 1e-6 * (np.abs(x).astype(np.float64) @ np.abs(w).T))
