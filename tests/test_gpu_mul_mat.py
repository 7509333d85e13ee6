"""H3 parity: trc_hip_mul_mat_f32 (FP32 MFMA) against the oracle.

Reference semantics: compute_mul_mat (src/backends/cpu/trc_cpu_ops.cpp:182-216).
Bar (written here, from the benchmark's tolerance): for every dst row r (one
ne0-run), max_i |y_ri - yhat_ri| / ||yhat_r||_2 <= 1e-4, where yhat is the oracle.
The reference's own goldens additionally hold at their atol 1e-4 / rtol 1e-3.
"""
import numpy as np
import pytest

import oracle_lib as O
from conftest import GOLDEN, announce
from gpu_util import Dev, Stream, empty, gpu_mul_mat, launches
from traincpp_amd import hip as H
from traincpp_amd import synth

pytestmark = pytest.mark.gpu

TOL = 1e-4


def g(name):
    return np.load(GOLDEN / f"{name}.npy", allow_pickle=False)


def as4(a):
    return a.reshape((1,) * (4 - a.ndim) + a.shape)


def ramp(n):
    """The conformance tests' input ramp (tests/test_backend_conformance.cpp:130-135)."""
    i = np.arange(n)
    return ((i % 17) - 8).astype(np.float32) * np.float32(0.25)


def t01(x):
    return np.swapaxes(x, 2, 3)


def run_views(A, a_view_fn, B, b_view_fn):
    """Uploads the base arrays, runs the GPU on the views, returns (gpu, oracle)."""
    da, db = Dev(A), Dev(B)
    av, bv = a_view_fn(da.base), b_view_fn(db.base)
    got = gpu_mul_mat(da, av, db, bv)
    want = O.mul_mat(av, bv, threads=8)
    da.free()
    db.free()
    return got, want


@pytest.mark.parametrize("case", ["mul_mat", "mul_mat_batch", "mul_mat_batch_bcast_div", "mul_mat_batch_tile"])
def test_reference_goldens(hip, case):
    announce(f"mul_mat golden {case}")
    a, b, want = as4(g(f"{case}_in0")), as4(g(f"{case}_in1")), g(f"{case}_out")
    got, orc = run_views(a, lambda x: x, b, lambda x: x)
    assert np.all(np.abs(got - want) <= 1e-4 + 1e-3 * np.abs(want))
    assert O.row_l2_error(got, orc) <= TOL


# The conformance suite's mul_mat cases (tests/test_backend_conformance.cpp:455-553,928-934):
# (a base shape in ggml order, transpose a?, b base shape, transpose b?)
CONFORMANCE = {
    "basic": ((5, 3, 1, 1), False, (5, 4, 1, 1), False),
    "transposed_a": ((3, 5, 1, 1), True, (5, 4, 1, 1), False),
    "transposed_b": ((5, 3, 1, 1), False, (4, 5, 1, 1), True),
    "tile_boundary": ((33, 70, 1, 1), False, (33, 66, 1, 1), False),
    "batch": ((5, 3, 1, 1), False, (5, 4, 2, 3), False),
    "batch_bcast_div": ((5, 3, 2, 1), False, (5, 4, 4, 1), False),
    "batch_transposed": ((3, 5, 2, 2), True, (4, 5, 2, 2), True),
    "batch_tile_boundary": ((33, 70, 1, 1), False, (33, 66, 2, 2), False),
    "grid_batch_z": ((8, 4, 1, 1), False, (8, 4, 65, 1), False),
}


@pytest.mark.parametrize("name", list(CONFORMANCE))
def test_conformance_cases(hip, name):
    ane, ta, bne, tb = CONFORMANCE[name]
    announce(f"mul_mat conformance {name}")
    A = ramp(int(np.prod(ane))).reshape(ane[::-1])
    B = ramp(int(np.prod(bne))).reshape(bne[::-1])
    got, want = run_views(A, t01 if ta else (lambda x: x), B, t01 if tb else (lambda x: x))
    # the conformance tolerance (test_backend_conformance.cpp:107) and the benchmark bar
    assert np.all(np.abs(got - want) <= 1e-5 + 2e-4 * np.abs(want))
    assert O.row_l2_error(got, want) <= TOL


@pytest.mark.parametrize("case", ["grad_mul_mat_batch", "grad_mul_mat_batch_div"])
def test_backward_goldens(hip, case):
    """dA = transpose(mul_mat(transpose(dY), transpose(B))) (+ plane sum) and
    dB = mul_mat(transpose(A), dY) (src/core/trc_autograd.cpp:487-503) on the GPU."""
    announce(f"mul_mat backward golden {case}")
    A, B = as4(g(f"{case}_in0")), as4(g(f"{case}_in1"))
    Y, _ = run_views(A, lambda x: x, B, lambda x: x)
    dY = (2.0 * Y).astype(np.float32)
    dA_t, _ = run_views(dY, t01, B, t01)
    dA_full = t01(dA_t)
    a3, a2, b3, b2 = A.shape[0], A.shape[1], B.shape[0], B.shape[1]
    dA = dA_full.reshape(b3 // a3, a3, b2 // a2, a2, *dA_full.shape[2:]).sum(axis=(0, 2))
    dB, _ = run_views(A, t01, dY, lambda x: x)
    for got, name in ((dA, "grad0"), (dB, "grad1")):
        want = g(f"{case}_{name}")
        assert np.all(np.abs(got - want) <= 1e-4 + 1e-3 * np.abs(want)), name


@pytest.mark.parametrize("shape", [
    # K, M, N, b2, b3, a2, a3
    (1, 1, 1, 1, 1, 1, 1), (2, 33, 31, 1, 1, 1, 1), (17, 65, 129, 1, 1, 1, 1), (100, 130, 70, 3, 2, 3, 1),
    (256, 256, 256, 1, 1, 1, 1), (513, 200, 300, 2, 1, 1, 1), (64, 128, 128, 4, 2, 2, 2), (7, 9, 11, 6, 1, 3, 1),
    # 128 or more 128x128 tiles but under 512 and K >= 1024: K in two parts that
    # meet in dst (partial tiles, K not a multiple of the slab, two planes)
    (2500, 2000, 1000, 1, 1, 1, 1), (1030, 1000, 1000, 1, 1, 2, 1),
    # the same with whole tiles and slabs (double-buffered slabs): broadcast
    # planes, and 8 planes (each plane's tiles on one XCD)
    (1024, 1024, 512, 4, 1, 2, 1), (1088, 512, 512, 8, 1, 1, 1),
    # 512 or more whole 128x128 tiles, K whole (double-buffered slabs)
    (64, 4096, 2048, 1, 1, 1, 1),
    # plane counts that are a multiple of 8 (each plane's tiles on one XCD):
    # ragged 64x64 tiles over 8 planes, ragged 128x128 tiles over 64 planes
    (33, 70, 90, 4, 2, 1, 1), (40, 300, 300, 8, 8, 1, 1),
])
@pytest.mark.parametrize("layout", ["kk", "tk", "kt", "tt", "gen"])
def test_random_shapes_and_layouts(hip, shape, layout):
    K, M, N, b2, b3, a2, a3 = shape
    rng = np.random.default_rng(K * 7 + M * 3 + N)
    announce(f"mul_mat random {shape} {layout}")
    if layout == "gen":
        # every-other-element views: nb0 = 8 forces the scalar (generic) loaders
        A = rng.standard_normal((a3, a2, M, 2 * K)).astype(np.float32)
        B = rng.standard_normal((b3 * a3, b2 * a2, N, 2 * K)).astype(np.float32)
        got, want = run_views(A, lambda x: x[..., ::2], B, lambda x: x[..., ::2])
    else:
        ta, tb = layout[0] == "t", layout[1] == "t"
        A = rng.standard_normal((a3, a2, K, M) if ta else (a3, a2, M, K)).astype(np.float32)
        B = rng.standard_normal((b3 * a3, b2 * a2, K, N) if tb else (b3 * a3, b2 * a2, N, K)).astype(np.float32)
        got, want = run_views(A, t01 if ta else (lambda x: x), B, t01 if tb else (lambda x: x))
    assert O.row_l2_error(got, want) <= TOL


def sampled_oracle_cols(av, bv, cols):
    """Oracle values of dst columns `cols` (dst rows in the row-L2 metric)."""
    pa, ane, anb = O.base_ptr_and_meta(av)
    pb, bne, bnb = O.base_ptr_and_meta(bv)
    dne = [ane[1], bne[1], bne[2], bne[3]]
    out = np.zeros((dne[3], dne[2], dne[1], dne[0]), dtype=np.float32)
    _, _, dnb = O.base_ptr_and_meta(out)
    for j in cols:
        rc = O.oracle().orc_mul_mat_cols(pa, O.NE(*ane), O.NB(*anb), pb, O.NE(*bne), O.NB(*bnb), out.ctypes.data,
                                         O.NE(*dne), O.NB(*dnb), int(j), int(j) + 1, 8)
        assert rc == 0
    return out[:, :, cols, :]


def config3_inputs():
    t = 7  # Q5_1 weights, dequantized on the GPU exactly as the oracle does
    n = 4096 * 4096 // 32
    raw = synth.block_bytes(synth.quant_blocks(t, n, synth.config_seed(3, 0)))
    W = O.dequant(t, raw, threads=8).reshape(1, 1, 4096, 4096)
    X = synth.normal(synth.config_seed(3, 1), 4096 * 512).reshape(1, 1, 512, 4096)
    dY = synth.normal(synth.config_seed(3, 2), 4096 * 512, 0.0, 1e-2).reshape(1, 1, 512, 4096)
    return W, X, dY


# sampled dst rows (ne1 indices) at full size: tile edges, both ends and a stride
COLS = sorted({0, 1, 31, 32, 63, 64, 127, 128, 200, 255, 256, 383, 384, 510, 511, *range(5, 512, 37)})


def sums_error(got, av, bv):
    """Every dst element enters two float64 checksums that the operands fix:
    sum_j dst[i, j] = sum_k a[k, i] * (sum_j b[k, j]) and
    sum_i dst[i, j] = sum_k (sum_i a[k, i]) * b[k, j], per plane (a's planes by the
    ggml modulo broadcast). Returns the larger row-L2-normalised error of the two;
    a wrong or missing tile anywhere moves one of them far above FP32 rounding."""
    ne3, ne2 = got.shape[0], got.shape[1]
    worst = 0.0
    for i3 in range(ne3):
        for i2 in range(ne2):
            a = np.asarray(av[i3 % av.shape[0], i2 % av.shape[1]], dtype=np.float64)  # [M, K]
            b = np.asarray(bv[i3, i2], dtype=np.float64)                              # [N, K]
            d = np.asarray(got[i3, i2], dtype=np.float64)                             # [N, M]
            s_i, r_i = d.sum(axis=0), a @ b.sum(axis=0)
            s_j, r_j = d.sum(axis=1), b @ a.sum(axis=0)
            for s, r in ((s_i, r_i), (s_j, r_j)):
                worst = max(worst, float(np.abs(s - r).max() / max(np.linalg.norm(r), 1e-30)))
    return worst


@pytest.fixture(scope="module")
def cfg3():
    return config3_inputs()


@pytest.mark.parametrize("product", ["Y=W.X", "dX=W^T.dY", "dW^T=dY^T.X^T"])
def test_config3_full_size(hip, cfg3, product):
    """The linear layer's three products at 4096 x 4096 x 512, checked on sampled
    dst rows against the oracle."""
    W, X, dY = cfg3
    announce(f"mul_mat cfg3 {product}")
    if product == "Y=W.X":
        A, af, B, bf, cols = W, (lambda x: x), X, (lambda x: x), COLS
    elif product == "dX=W^T.dY":
        A, af, B, bf, cols = W, t01, dY, (lambda x: x), COLS
    else:
        A, af, B, bf, cols = dY, t01, X, t01, [0, 1, 4095, 1000, 2048]
    da, db = Dev(A), Dev(B)
    av, bv = af(da.base), bf(db.base)
    got = gpu_mul_mat(da, av, db, bv)
    want = sampled_oracle_cols(av, bv, cols)
    assert O.row_l2_error(got[:, :, cols, :], want) <= TOL
    assert np.isfinite(got).all()
    assert sums_error(got, av, bv) <= 1e-5
    da.free()
    db.free()


def test_config4_broadcast_permuted(hip):
    """src0 ne=[128,1024,8,4] x src1 = permute(base[128,32,512,4], 0,2,1,3)
    (ne=[128,512,32,4], nb1 > nb2), planes broadcast (i2%8, i3%4)."""
    announce("mul_mat cfg4")
    A = synth.normal(synth.config_seed(4, 0), 128 * 1024 * 8 * 4).reshape(4, 8, 1024, 128)
    base = synth.normal(synth.config_seed(4, 1), 128 * 32 * 512 * 4).reshape(4, 512, 32, 128)
    da, db = Dev(A), Dev(base)
    bv = np.swapaxes(db.base, 1, 2)  # ggml permute(0,2,1,3)
    ne, nb = O.view_meta(bv)
    assert ne == [128, 512, 32, 4] and nb == [4, 16384, 512, 8388608]
    got = gpu_mul_mat(da, da.base, db, bv)
    cols = [0, 7, 31, 32, 255, 256, 300, 480, 511]
    want = sampled_oracle_cols(da.base, bv, cols)
    assert O.row_l2_error(got[:, :, cols, :], want) <= TOL
    assert sums_error(got, da.base, bv) <= 1e-5
    da.free()
    db.free()


def test_split_products_on_two_streams(hip):
    """K split in two (K >= 1024, 128 to 511 tiles of 128 x 128): the waves holding
    one block in the two parts meet in dst through ticket words kept with the
    stream's workspace, which every launch leaves clear. Two such products
    alternate on two streams, 20 calls each, so that they overlap on the GPU and
    each stream needs its own words: one with whole tiles (double-buffered
    slabs), one with ragged tiles. Each result equals, bit for bit, the same
    product run twice more on the null stream, and matches the oracle."""
    streams = [Stream(), Stream()]
    cases = []
    for c, (K, M, N) in enumerate([(1024, 2048, 1024), (1100, 2000, 1000)]):  # 16 x 8 tiles each
        A = synth.normal(940 + c, K * M).reshape(1, 1, M, K)
        B = synth.normal(950 + c, K * N).reshape(1, 1, N, K) * np.float32(10.0 ** c)
        cases.append((A, B, Dev(A), Dev(B), empty((1, 1, N, M))))
    announce("mul_mat K split, two streams")
    for _ in range(20):
        for c, (A, B, da, db, dd) in enumerate(cases):
            H.mul_mat_f32(da.tensor(), db.tensor(), dd.tensor(), streams[c].handle)
    for st in streams:
        H.sync(st.handle)
    for A, B, da, db, dd in cases:
        got = dd.read()
        for _ in range(2):
            alone = gpu_mul_mat(da, da.base, db, db.base)
            assert np.array_equal(got.view(np.uint32), alone.view(np.uint32))
        assert O.row_l2_error(got, O.mul_mat(A, B, threads=8)) <= TOL
        for dv in (da, db, dd):
            dv.free()
    for st in streams:
        st.close()


def test_shape_errors_are_rejected(hip):
    a = empty((1, 1, 4, 8))
    b = empty((1, 1, 4, 6))
    d = empty((1, 1, 4, 4))
    with pytest.raises(H.HipError) as e:
        H.mul_mat_f32(a.tensor(), b.tensor(), d.tensor())  # K 8 vs 6
    assert e.value.code == H.E_SHAPE
    b2 = empty((1, 3, 4, 8))
    a2 = empty((1, 2, 4, 8))
    d2 = empty((1, 3, 4, 4))
    with pytest.raises(H.HipError) as e:
        H.mul_mat_f32(a2.tensor(), b2.tensor(), d2.tensor())  # 3 % 2 != 0
    assert e.value.code == H.E_SHAPE
    # dst sharing bytes with an operand
    buf = empty((1, 1, 8, 8))  # a: K = 8, M = 8
    b3 = empty((1, 1, 6, 8))   # b: K = 8, N = 6
    with pytest.raises(H.HipError) as e:
        H.mul_mat_f32(buf.tensor(), b3.tensor(), H.tensor(buf.ptr + 16, [8, 6, 1, 1], H.contiguous_nb([8, 6, 1, 1])))
    assert e.value.code == H.E_SHAPE
    with pytest.raises(H.HipError) as e:
        H.mul_mat_f32(buf.tensor(), b3.tensor(), H.tensor(b3.ptr, [8, 6, 1, 1], H.contiguous_nb([8, 6, 1, 1])))
    assert e.value.code == H.E_SHAPE
    for t in (buf, b3):
        t.free()


# ---------------------------------------------------------------- few columns (N <= 64)

@pytest.fixture(scope="module")
def cfg0_w():
    """Configuration 0's weight: the Q8_0 blocks of a 4096 x 4096 tensor as the GGUF
    warm start turns them into F32 (src/io/trc_gguf.cpp:1082-1088), here by the oracle."""
    n = 4096 * 4096 // 32
    raw = synth.block_bytes(synth.quant_blocks(H.TYPE_Q8_0, n, synth.config_seed(0, 8)))
    return O.dequant(H.TYPE_Q8_0, raw, threads=8).reshape(1, 1, 4096, 4096)


@pytest.mark.parametrize("N", [1, 2, 3, 5, 7, 8, 16, 32, 64])
@pytest.mark.parametrize("layout", ["contiguous", "transposed"])
def test_config0_f32_few_columns(hip, cfg0_w, N, layout):
    """mul_mat(W F32 [4096, 4096], X [4096, N]) at configuration 0's size, every dst
    element against the oracle: X k-contiguous, or X = transpose(base[N, 4096])
    (k strided, the layout of a transposed activation view)."""
    announce(f"mul_mat cfg0 F32 N={N} {layout}")
    X = synth.normal(synth.config_seed(0, 100 + N), 4096 * N)
    if layout == "contiguous":
        got, want = run_views(cfg0_w, lambda x: x, X.reshape(1, 1, N, 4096), lambda x: x)
    else:
        got, want = run_views(cfg0_w, lambda x: x, X.reshape(1, 1, 4096, N), t01)
    assert got.shape == (1, 1, N, 4096)
    assert O.row_l2_error(got, want) <= TOL


@pytest.mark.parametrize("K,M,N", [(512, 16, 1), (4096, 48, 5), (4096, 4096, 8), (1028, 70, 12), (2048, 33, 40)])
def test_few_columns_one_hot(hip, K, M, N):
    """W rows with a single 1 at k = kmap[i] and X[j, k] = 1000 j + k: every output
    is one X element times 1 plus exact zeros, so it must equal 1000 j + kmap[i]
    bit for bit. A wrong lane-to-(column, k) mapping in the few-column loads shows
    up here as the value of the (column, k) that was read instead."""
    announce(f"mul_mat one-hot K={K} M={M} N={N}")
    kmap = (np.arange(M) * 131 + 7) % K
    W = np.zeros((1, 1, M, K), np.float32)
    W[0, 0, np.arange(M), kmap] = 1.0
    X = (1000.0 * np.arange(N)[:, None] + np.arange(K)[None, :]).astype(np.float32).reshape(1, 1, N, K)
    a, b = Dev(W), Dev(X)
    got = gpu_mul_mat(a, W, b, X)
    want = (1000.0 * np.arange(N)[:, None] + kmap[None, :]).astype(np.float32).reshape(1, 1, N, M)
    assert np.array_equal(got, want)
    a.free()
    b.free()


def test_config0_f32_deterministic(hip, cfg0_w):
    """The waves' partial sums meet in a fixed order: two runs give the same bits."""
    announce("mul_mat cfg0 F32 N=8 twice")
    X = synth.normal(synth.config_seed(0, 108), 4096 * 8).reshape(1, 1, 8, 4096)
    a, _ = run_views(cfg0_w, lambda x: x, X, lambda x: x)
    b, _ = run_views(cfg0_w, lambda x: x, X, lambda x: x)
    assert np.array_equal(a.view(np.uint32), b.view(np.uint32))


@pytest.mark.parametrize("shape", [
    # K, M, N, b2, b3, a2, a3: ragged row blocks, K not a multiple of the 32-wide chunk,
    # fewer chunks than waves, every column-group count, broadcast planes
    (4, 1, 1, 1, 1, 1, 1), (36, 17, 5, 1, 1, 1, 1), (100, 33, 16, 1, 1, 1, 1), (512, 70, 17, 1, 1, 1, 1),
    (1028, 250, 33, 1, 1, 1, 1), (2048, 300, 48, 1, 1, 1, 1), (260, 129, 64, 1, 1, 1, 1),
    (128, 64, 8, 4, 2, 2, 1), (96, 48, 24, 6, 1, 3, 1), (64, 40, 64, 2, 2, 1, 2),
    (1000, 77, 7, 1, 1, 1, 1), (4100, 33, 6, 2, 1, 1, 1),
])
@pytest.mark.parametrize("layout", ["kk", "kt", "kgen", "kmis"])
def test_few_columns_shapes(hip, shape, layout):
    """The few-column path (N <= 64, W k-contiguous) on ragged shapes and planes, with
    X k-contiguous (kk), transposed (kt), every other element (kgen) or 4 bytes off
    16-byte alignment (kmis: read element by element)."""
    K, M, N, b2, b3, a2, a3 = shape
    rng = np.random.default_rng(K * 11 + M * 5 + N)
    announce(f"mul_mat few columns {shape} {layout}")
    A = rng.standard_normal((a3, a2, M, K)).astype(np.float32)
    if layout == "kk":
        B = rng.standard_normal((b3 * a3, b2 * a2, N, K)).astype(np.float32)
        got, want = run_views(A, lambda x: x, B, lambda x: x)
    elif layout == "kt":
        B = rng.standard_normal((b3 * a3, b2 * a2, K, N)).astype(np.float32)
        got, want = run_views(A, lambda x: x, B, t01)
    elif layout == "kgen":
        B = rng.standard_normal((b3 * a3, b2 * a2, N, 2 * K)).astype(np.float32)
        got, want = run_views(A, lambda x: x, B, lambda x: x[..., ::2])
    else:
        B = rng.standard_normal((b3 * a3, b2 * a2, N, K + 1)).astype(np.float32)
        got, want = run_views(A, lambda x: x, B, lambda x: x[..., 1:])
    assert O.row_l2_error(got, want) <= TOL


# ---------------------------------------------------------------- dst += mul_mat (trc_hip_mul_mat_acc_f32)

def _acc_run(A, a_view_fn, B, b_view_fn, D0):
    """GPU d0 + mul_mat(a, b) through the accumulate entry, and mul_mat(a, b) alone."""
    da, db, dd = Dev(A), Dev(B), Dev(D0)
    av, bv = a_view_fn(da.base), b_view_fn(db.base)
    H.mul_mat_acc_f32(da.tensor(av), db.tensor(bv), dd.tensor())
    H.sync()
    got = dd.read()
    mm = gpu_mul_mat(da, av, db, bv)
    for d in (da, db, dd):
        d.free()
    return got, mm, av, bv


@pytest.mark.parametrize("shape", [
    # (K, M, N, a transposed, b transposed): the gradient of configuration 3's weight as
    # the plugin fuses it (mul_mat(X^T, dY^T) into W's accumulator), smaller transposed
    # products, and the few-column kernel
    (512, 4096, 4096, True, True), (128, 1024, 768, True, True), (300, 130, 70, False, True),
    (4096, 4096, 8, False, False), (1000, 77, 7, False, False), (96, 48, 40, True, False),
    # 512 whole tiles with k-contiguous operands (double-buffered slabs)
    (256, 4096, 2048, False, False), (64, 4096, 2048, False, True), (96, 4096, 2048, True, False),
])
def test_mul_mat_acc_adds_the_product(hip, shape):
    """Each element gets the product's float sum, then one float add into dst: the
    result equals numpy float32 d0 + (the GPU's mul_mat of the same operands) bit for
    bit, on shapes whose plain product keeps K whole, as these do."""
    K, M, N, at, bt = shape
    announce(f"mul_mat_acc K={K} M={M} N={N} a{'T' if at else ''} b{'T' if bt else ''}")
    A = synth.normal(900 + K, K * M).reshape(1, 1, K, M) if at else synth.normal(900 + K, K * M).reshape(1, 1, M, K)
    B = synth.normal(901 + N, K * N).reshape(1, 1, K, N) if bt else synth.normal(901 + N, K * N).reshape(1, 1, N, K)
    D0 = synth.normal(902 + M, M * N).reshape(1, 1, N, M)
    got, mm, av, bv = _acc_run(A, t01 if at else (lambda x: x), B, t01 if bt else (lambda x: x), D0)
    assert np.array_equal(got.view(np.uint32), (D0 + mm).view(np.uint32))
    if K * M * N <= 64 << 20:
        assert O.row_l2_error(mm, O.mul_mat(av, bv, threads=8)) <= TOL


def test_mul_mat_acc_keeps_k_whole(hip):
    """Configuration 3's forward shape, whose plain product sums K in two parts that
    meet in dst: added into dst it keeps K whole (d + a + b would round differently
    from d + (a + b)), and is checked against d0 + the oracle's product."""
    announce("mul_mat_acc configuration 3 forward shape")
    K, M, N = 4096, 4096, 512
    W = synth.normal(910, K * M).reshape(1, 1, M, K)
    X = synth.normal(911, K * N).reshape(1, 1, N, K)
    D0 = synth.normal(912, M * N).reshape(1, 1, N, M)
    got, _, av, bv = _acc_run(W, lambda x: x, X, lambda x: x, D0)
    cols = np.arange(0, N, 37)
    want = D0[:, :, cols, :] + O.mul_mat(av, np.ascontiguousarray(bv[:, :, cols, :]), threads=8)
    assert O.row_l2_error(got[:, :, cols, :], want) <= TOL
    again, _, _, _ = _acc_run(W, lambda x: x, X, lambda x: x, D0)
    assert np.array_equal(got.view(np.uint32), again.view(np.uint32))


def test_mul_mat_acc_rejects_overlap(hip):
    buf = empty((1, 1, 8, 8))
    b3 = empty((1, 1, 6, 8))
    with pytest.raises(H.HipError) as e:
        H.mul_mat_acc_f32(buf.tensor(), b3.tensor(), H.tensor(buf.ptr + 16, [8, 6, 1, 1], H.contiguous_nb([8, 6, 1, 1])))
    assert e.value.code == H.E_SHAPE
    for t in (buf, b3):
        t.free()


# ---------------------------------------------------------------- bf16 tiles (csrc/hip/mm_bf3.h)

def _f64(av, bv):
    a, b = np.asarray(av, np.float64), np.asarray(bv, np.float64)
    r3, r2 = b.shape[0] // a.shape[0], b.shape[1] // a.shape[1]
    return b @ np.swapaxes(np.tile(a, (r3, r2, 1, 1)), 2, 3)


def _rel(got, want):
    return float(np.linalg.norm(got.astype(np.float64) - want) / np.linalg.norm(want))


@pytest.mark.parametrize("shape", [
    # (K, M, N, planes): last slabs of 1, 16, 17 and 31 k and a whole one; parts of K
    # from 1 to 8; last column tiles of 1, 64, 65 and 128; rows of 1, 3 and 127 past a tile
    (1025, 257, 129, 1), (2064, 515, 192, 1), (4113, 383, 193, 1), (3103, 129, 70, 1), (2048, 256, 256, 1),
    (8192, 131, 65, 1), (515, 130, 131, 3), (1056, 128, 128, 8), (160, 1300, 1100, 7),
])
@pytest.mark.parametrize("layout", ["kk", "tk", "kt", "tt", "odd", "gen"])
def test_bf16_tiles_against_float64(hip, shape, layout):
    """Every element against float64: the 2-norm of the error stays below that of K
    floats added one after another, sqrt(K) half ulps of the result for normal
    inputs (2^-25 sqrt(K)). odd: rows 4 bytes off 16-byte alignment; gen: every other
    element along both dimensions."""
    K, M, N, P = shape
    rng = np.random.default_rng(K + M + N)
    announce(f"mul_mat bf16 tiles {shape} {layout}")
    if layout == "odd":
        A, B = (rng.standard_normal((1, P, r, K + 3)).astype(np.float32) for r in (M, N))
        af = bf = lambda x: x[..., 3:]
    elif layout == "gen":
        A, B = (rng.standard_normal((1, P, r, 2 * K)).astype(np.float32) for r in (2 * M, N))
        af, bf = (lambda x: x[:, :, ::2, ::2]), (lambda x: x[..., ::2])
    else:
        ta, tb = layout[0] == "t", layout[1] == "t"
        A = rng.standard_normal((1, P, K, M) if ta else (1, P, M, K)).astype(np.float32)
        B = rng.standard_normal((1, P, K, N) if tb else (1, P, N, K)).astype(np.float32)
        af, bf = (t01 if ta else (lambda x: x)), (t01 if tb else (lambda x: x))
    da, db = Dev(A), Dev(B)
    got = gpu_mul_mat(da, af(da.base), db, bf(db.base))
    da.free()
    db.free()
    assert _rel(got, _f64(af(A), bf(B))) <= 2.0 ** -25 * np.sqrt(K)


# one shape per way the parts of K come together: K whole on 8-wave and 4-wave
# workgroups, two parts in dst, more in slots (of one and of two planes)
BF16_ROUTES = [((1024, 2560, 1280, 1), "whole8"), ((128, 2048, 512, 8), "whole4"), ((1024, 2048, 1024, 1), "pair"),
               ((4096, 512, 200, 1), "slots"), ((640, 1024, 512, 2), "slots")]


@pytest.mark.parametrize("shape,route", BF16_ROUTES)
def test_bf16_tiles_special_values(hip, shape, route):
    """Infinities, NaNs, values that round to infinity as bf16, subnormals and values
    near them, each in rows and columns of their own: results are float64's (not finite where it is not, equal to float rounding elsewhere), and
    the other rows' bits are what they are without them, in tiles that hold none."""
    K, M, N, P = shape
    rng = np.random.default_rng(7 * K + M)
    announce(f"mul_mat bf16 tiles special values {shape}")
    A = rng.standard_normal((1, P, M, K)).astype(np.float32)
    B = rng.standard_normal((1, P, N, K)).astype(np.float32)
    clean = (A.copy(), B.copy())
    A[0, 0, 3, 5] = np.inf
    A[0, 0, 4, K - 1] = np.nan
    A[0, 0, 5] = 0
    A[0, 0, 5, K // 2] = np.float32(3.4e38)       # infinity as bf16; finite times the column below
    B[0, 0, :, K // 2] = np.clip(B[0, 0, :, K // 2], -0.9, 0.9)
    clean[1][0, 0, :, K // 2] = B[0, 0, :, K // 2]
    A[0, 0, 6] = (rng.standard_normal(K) * 1e-38).astype(np.float32)
    A[0, 0, 7] = (rng.standard_normal(K) * 1e-41).astype(np.float32)
    B[0, 0, 2] *= np.float32(1e20)
    clean[1][0, 0, 2] = B[0, 0, 2]
    B[0, 0, 9, 0] = -np.inf
    clean[1][0, 0, 9] = B[0, 0, 9]
    da, db, dc = Dev(A), Dev(B), Dev(clean[0])
    out = empty((1, P, N, M))
    assert bf16_route(da.tensor(), db.tensor(), out.tensor()) == route
    out.free()
    got = gpu_mul_mat(da, A, db, B)
    plain = gpu_mul_mat(dc, clean[0], db, B)
    with np.errstate(invalid="ignore", over="ignore"):
        want = _f64(A[:, :1], B[:, :1])[0, 0]     # [N, M]
        w32 = want.astype(np.float32)
    g = got[0, 0]
    assert np.array_equal(np.isnan(g), np.isnan(w32))
    assert np.array_equal(g[np.isinf(w32)], w32[np.isinf(w32)])
    ok = np.isfinite(w32)
    a, b = (np.abs(np.nan_to_num(x[0, 0], posinf=0, neginf=0).astype(np.float64)) for x in (A, B))
    scale = b @ a.T
    # K additions of half an ulp each, and half the smallest subnormal for each
    bound = K * (2.0 ** -24 * scale + 2.0 ** -150)
    assert np.all(np.abs(g[ok].astype(np.float64) - want[ok]) <= bound[ok])
    # beyond the first tiles' rows nothing has changed
    assert np.array_equal(got[:, :, :, 128:].view(np.uint32), plain[:, :, :, 128:].view(np.uint32))
    for d in (da, db, dc):
        d.free()


@pytest.mark.parametrize("shape,route", BF16_ROUTES)
def test_bf16_tiles_integers_are_exact(hip, shape, route):
    """Integer operands whose sums stay under 2^24: every sum is exact in float, so
    the bits are those of any order of adding."""
    K, M, N, P = shape
    rng = np.random.default_rng(K)
    announce(f"mul_mat bf16 tiles integers {shape}")
    A = rng.integers(-60, 61, (1, P, M, K)).astype(np.float32)
    B = rng.integers(-60, 61, (1, P, N, K)).astype(np.float32)
    A[0, 0, 0], B[0, 0, 0] = 0, 0
    A[0, 0, 0, K // 3], B[0, 0, 0, K // 3] = 1, 16777215.0
    da, db, out = Dev(A), Dev(B), empty((1, P, N, M))
    assert bf16_route(da.tensor(), db.tensor(), out.tensor()) == route
    out.free()
    got = gpu_mul_mat(da, A, db, B)
    da.free()
    db.free()
    want = _f64(A, B)
    small = np.abs(want) < 2 ** 24
    small[0, 0, 0, 1:] = False                    # that column's other sums pass 2^24
    assert small.mean() > 0.99
    assert np.array_equal(got[small], want[small].astype(np.float32))


def test_bf16_tiles_without_a_workspace(hip):
    """Where a stream has no workspace and none may be made (eight other streams hold
    the device's, or the stream is under capture), the parts of K run one launch
    after another: the same bits as when they meet."""
    import ctypes as C

    from gpu_util import runtime
    rt = runtime()
    announce("mul_mat bf16 tiles, nine streams and capture")
    cases = []
    for K, M, N in [(2048, 512, 200), (1024, 2048, 1024)]:
        A, B = synth.normal(960 + M, K * M).reshape(1, 1, M, K), synth.normal(961 + N, K * N).reshape(1, 1, N, K)
        cases.append((Dev(A), Dev(B), empty((1, 1, N, M))))
    H.qmatvec_release_stream(None)
    live = [Stream() for _ in range(10)]
    refs = []
    for s in live:
        for c, (a, b, d) in enumerate(cases):
            H.mul_mat_f32(a.tensor(), b.tensor(), d.tensor(), s.handle)
            H.sync(s.handle)
            got = d.read().copy()
            if len(refs) <= c:
                refs.append(got)
                assert _rel(got, _f64(a.base, b.base)) <= 2.0 ** -25 * np.sqrt(a.base.shape[3])
            assert np.array_equal(got.view(np.uint32), refs[c].view(np.uint32))
    for s in live:
        s.close()
    s = Stream()
    graph, gexec = C.c_void_p(), C.c_void_p()
    assert rt.hipStreamBeginCapture(C.c_void_p(s.handle), 0) == 0
    try:
        for a, b, d in cases:
            H.mul_mat_f32(a.tensor(), b.tensor(), d.tensor(), s.handle)
    finally:
        rc = rt.hipStreamEndCapture(C.c_void_p(s.handle), C.byref(graph))
    assert rc == 0
    assert rt.hipGraphInstantiate(C.byref(gexec), graph, None, None, 0) == 0
    for _ in range(3):
        for a, b, d in cases:
            H.fill_f32(d.ptr, float("nan"), d.base.size)
        H.sync()
        assert rt.hipGraphLaunch(gexec, C.c_void_p(s.handle)) == 0
        H.sync(s.handle)
        for (a, b, d), ref in zip(cases, refs):
            assert np.array_equal(d.read().view(np.uint32), ref.view(np.uint32))
            H.mul_mat_f32(a.tensor(), b.tensor(), d.tensor(), s.handle)  # eager, between the replays
            H.sync(s.handle)
            assert np.array_equal(d.read().view(np.uint32), ref.view(np.uint32))
    rt.hipGraphExecDestroy(gexec)
    rt.hipGraphDestroy(graph)
    s.close()
    for a, b, d in cases:
        for x in (a, b, d):
            x.free()


def bf16_route(a, b, d, acc=False):
    """How a product on 256-CU devices is launched: "whole8" or "whole4" (bf16 tiles, K
    whole, workgroups of 8 or 4 waves), "pair" (K in two parts that meet in dst), "slots"
    (more parts), or "fp32" (another grid). From 512 tiles of 128 x 128 on the FP32
    tiles' grid is that of "whole4": shapes here have fewer."""
    f = H.mul_mat_acc_f32 if acc else H.mul_mat_f32
    (grid, block), = launches(lambda s: f(a, b, d, s))
    tiles = -(-d.ne[0] // 128) * -(-d.ne[1] // 128) * d.ne[2] * d.ne[3]
    if grid % tiles or (block == 256) != (grid == tiles and tiles > 256):
        return "fp32"
    return {1: "whole4" if block == 256 else "whole8", 2: "pair"}.get(grid // tiles, "slots")


@pytest.mark.parametrize("which", ["src0", "src1"])
@pytest.mark.parametrize("shape", [
    # (K, M, N, accumulated, route): rows of 1, 2 and 3 past a multiple of four
    (1056, 1409, 1410, False, "whole8"), (200, 2689, 2690, False, "whole4"), (1000, 1409, 1411, True, "whole8"),
    (1056, 1281, 1283, False, "pair"), (1056, 777, 130, False, "slots"),
])
def test_transposed_operands_ignore_what_follows_their_rows(hip, shape, which):
    """A transposed view of a wider buffer whose row count is no multiple of four: the
    loads of four rows reach into the columns after the view. Nothing there may matter,
    NaN, infinity or subnormal: the bits are those with zeros there."""
    K, M, N, acc, route = shape
    announce(f"mul_mat transposed view with padding {shape} {which}")
    rng = np.random.default_rng(K + M)
    A, B = (rng.standard_normal((1, 1, K, r + 3)).astype(np.float32) for r in (M, N))
    out, bits = empty((1, 1, N, M)), []
    for pad in (0.0, np.nan, np.inf, 1e-40):
        (A if which == "src0" else B)[..., -3:] = pad
        da, db = Dev(A), Dev(B)
        ta, tb = da.tensor(t01(A[..., :M])), db.tensor(t01(B[..., :N]))
        H.fill_f32(out.ptr, 0.0, M * N)
        (H.mul_mat_acc_f32 if acc else H.mul_mat_f32)(ta, tb, out.tensor())
        H.sync()
        bits.append(out.read().view(np.uint32))
        if pad == 0.0:
            assert bf16_route(ta, tb, out.tensor(), acc) == route
            assert _rel(bits[0].view(np.float32), _f64(t01(A[..., :M]), t01(B[..., :N]))) <= 2.0 ** -25 * np.sqrt(K)
        da.free()
        db.free()
    out.free()
    assert all(np.array_equal(bits[0], x) for x in bits[1:])


def laid(x, layout):
    """(a buffer, the view of it that is x) with x's rows along k ("k"), its columns
    ("t": a transposed view), rows along k off 16-byte alignment ("odd"), or neither
    ("gen": every other element along both)."""
    if layout == "t":
        base = np.ascontiguousarray(t01(x))
        return base, t01(base)
    if layout == "odd":
        base = np.zeros(x.shape[:3] + (x.shape[3] + 3,), np.float32)
        view = base[..., 3:]
    elif layout == "gen":
        base = np.zeros(x.shape[:2] + (2 * x.shape[2], 2 * x.shape[3]), np.float32)
        view = base[:, :, ::2, ::2]
    else:
        return x, x
    view[:] = x
    return base, view


def bf16_run(A, B, layouts, acc, route, D=None):
    """The product (added into D, or into zeros, where acc) of A and B laid out as
    given, whose launch is asserted to be `route`."""
    (ab, av), (bb, bv) = laid(A, layouts[0]), laid(B, layouts[1])
    da, db, out = Dev(ab), Dev(bb), empty((1, B.shape[1], B.shape[2], A.shape[2]))
    ta, tb, td = da.tensor(av), db.tensor(bv), out.tensor()
    assert bf16_route(ta, tb, td, acc) == route
    out.buf.upload(out.base if D is None else D)
    (H.mul_mat_acc_f32 if acc else H.mul_mat_f32)(ta, tb, td)
    H.sync()
    got = out.read()
    for d in (da, db, out):
        d.free()
    return got


# (K, M, N, accumulated, route): one shape for each way the parts of K come together
BF16_ONE_EACH = [(1056, 1409, 1410, False, "whole8"), (200, 2689, 2690, False, "whole4"), (1000, 1409, 1411, True, "whole8"),
                 (200, 2691, 2689, True, "whole4"), (1056, 1281, 1283, False, "pair"), (1056, 777, 130, False, "slots")]


@pytest.mark.parametrize("layouts", ["k,k", "t,k", "k,t", "t,t", "odd,odd", "gen,gen"])
@pytest.mark.parametrize("shape", BF16_ONE_EACH)
def test_bf16_tiles_not_finite(hip, shape, layouts):
    """The second pass, with the FP32 instructions, that a tile makes for a result that
    is not finite on the bf16 ones: in the first and the last rows and columns of tiles,
    with a last slab that is not whole, a last column tile under half full, every
    loader, and added to dst. Infinities, NaNs, operands from 2^104 and sums from 2^80
    on come out as float64's within K float roundings; tiles without any keep their bits."""
    K, M, N, acc, route = shape
    announce(f"mul_mat bf16 tiles not finite {shape} {layouts}")
    rng = np.random.default_rng(K + 3 * M)
    A, B, D = (rng.standard_normal((1, 1, r, c)).astype(np.float32) for r, c in ((M, K), (N, K), (N, M)))
    B[..., K // 2] = np.clip(B[..., K // 2], -0.9, 0.9)
    plain = bf16_run(A, B, layouts.split(","), acc, route, D)
    for i in (0, M - 8):
        A[0, 0, i, 5] = np.inf
        A[0, 0, i + 1, K - 1] = np.nan
        A[0, 0, i + 2] = 0
        A[0, 0, i + 2, K // 2] = 3.4e38                # infinity as bf16; finite times the column above
        A[0, 0, i + 3, K - 2] = -1e32                  # infinity times 2^24
        A[0, 0, i + 4] *= np.float32(1e25)
        A[0, 0, i + 5] *= np.float32(1e-41)
    B[0, 0, N - 1, 3] = -np.inf
    got = bf16_run(A, B, layouts.split(","), acc, route, D)
    with np.errstate(invalid="ignore", over="ignore"):
        want = _f64(A, B) + (D if acc else 0)
        w32 = want.astype(np.float32)
    assert np.array_equal(np.isnan(got), np.isnan(w32))
    assert np.array_equal(got[np.isinf(w32)], w32[np.isinf(w32)])
    ok = np.isfinite(w32)
    a, b = (np.abs(np.nan_to_num(x, posinf=0, neginf=0).astype(np.float64)) for x in (A, B))
    # K additions of half an ulp each (and the one into dst), and half the smallest subnormal for each
    bound = K * (2.0 ** -24 * _f64(a, b) + 2.0 ** -150) + (2.0 ** -24 * np.abs(D) if acc else 0)
    assert np.all(np.abs(got[ok].astype(np.float64) - want[ok]) <= bound[ok])
    mid = (slice(None), slice(None), slice(0, (N - 1) // 128 * 128), slice(128, (M - 8) // 128 * 128))
    assert got[mid].size and np.array_equal(got[mid].view(np.uint32), plain[mid].view(np.uint32))


def test_bf16_tiles_long_sums_do_not_drift(hip):
    """16384 positive products in one part of K: the error of K / 16 roundings of half an
    ulp at most, which add up like a random walk (2-norm under sqrt(K / 16) half ulps),
    and not in one direction (a loss of a hundredth of each rounding would move the mean
    by 2^-24 K / 16 / 100 / 2, 5 half ulps)."""
    K, M, N = 16384, 1409, 1410
    announce("mul_mat bf16 tiles long positive sums")
    rng = np.random.default_rng(23)
    A, B = (rng.random((1, 1, r, K), dtype=np.float32) for r in (M, N))
    got = bf16_run(A, B, "kk", True, "whole8")[:, :, -200:, -200:]
    want = _f64(A[:, :, -200:], B[:, :, -200:])
    err = got - want
    assert np.linalg.norm(err) / np.linalg.norm(want) <= 2.0 ** -24 * np.sqrt(K / 16)
    assert abs(err.mean()) / want.mean() <= 4 * 2.0 ** -24


@pytest.mark.parametrize("layouts", ["kk", "tt"])
@pytest.mark.parametrize("shape", BF16_ONE_EACH)
def test_bf16_tiles_small_values(hip, shape, layouts):
    """Operands down to the smallest float take the same way as any other: scaled by
    powers of two, normal floats near 2^-115 give the scaled result's bits, and
    integer multiples of powers of two whose sums a float holds give exact sums where
    the operand, its products or the results are subnormal."""
    K, M, N, acc, route = shape
    announce(f"mul_mat bf16 tiles small values {shape} {layouts}")
    rng = np.random.default_rng(K + N)
    A, B = ((1 + rng.random((1, 1, r, K))).astype(np.float32) * rng.choice([-1, 1], (1, 1, r, K)).astype(np.float32)
            for r in (M, N))
    run = lambda a, b: bf16_run(a.astype(np.float32), b.astype(np.float32), layouts, acc, route)
    plain = run(A, B)
    assert np.array_equal(run(A * 2.0 ** -115, B * 2.0 ** 60).view(np.uint32), np.ldexp(plain, -55).view(np.uint32))
    assert np.array_equal(run(A * 2.0 ** 30, B * 2.0 ** -120).view(np.uint32), np.ldexp(plain, -90).view(np.uint32))
    A, B = (rng.integers(-40, 41, (1, 1, r, K)).astype(np.float64) for r in (M, N))
    want = _f64(A, B)
    assert np.abs(want).max() < 2 ** 22
    for ea, eb in [(-149, 40), (20, -149), (-70, -79), (-140, 5)]:  # the last two: results of 2^-149 and 2^-135 up
        assert np.array_equal(run(A * 2.0 ** ea, B * 2.0 ** eb), (want * 2.0 ** (ea + eb)).astype(np.float32))


@pytest.mark.parametrize("acc", [False, True], ids=["plain", "acc"])
@pytest.mark.parametrize("layouts", ["kk", "tt", "gen"])
def test_outer_product_is_rounded_once(hip, layouts, acc):
    """K = 1 (the weight gradient of one token): every element is one float product,
    with the bits numpy's float32 product has."""
    M, N = 4096, 4100
    announce(f"mul_mat outer product {layouts} {'acc' if acc else ''}")
    rng = np.random.default_rng(17)
    A, B = (rng.standard_normal((1, 1, r, 1)).astype(np.float32) for r in (M, N))
    (ab, av), (bb, bv) = (laid(x, "gen" if layouts == "gen" else layouts[0]) for x in (A, B))
    da, db, out = Dev(ab), Dev(bb), empty((1, 1, N, M))
    (H.mul_mat_acc_f32 if acc else H.mul_mat_f32)(da.tensor(av), db.tensor(bv), out.tensor())
    H.sync()
    got = out.read()[0, 0]
    for d in (da, db, out):
        d.free()
    assert np.array_equal(got, B[0, 0] * A[0, 0].T)


@pytest.mark.parametrize("case", [
    # (K, M, N, layouts, route): few slabs against one strided operand are faster on the
    # FP32 tiles, many, or two such operands, on the bf16 tiles
    (512, 1024, 1024, "gen,k", "fp32"), (512, 512, 512, "t,gen", "fp32"), (128, 2048, 2048, "gen,k", "fp32"),
    (4096, 256, 256, "gen,k", "slots"), (1056, 1281, 1283, "gen,gen", "pair"), (512, 2048, 2048, "k,gen", "whole8"),
])
def test_strided_operands_choose_their_tiles(hip, case):
    K, M, N, layouts, route = case
    announce(f"mul_mat strided operands {case}")
    A, B = synth.normal(990 + K, K * M).reshape(1, 1, M, K), synth.normal(991 + N, K * N).reshape(1, 1, N, K)
    got = bf16_run(A, B, layouts.split(","), False, route)
    assert _rel(got, _f64(A, B)) <= 2.0 ** -25 * np.sqrt(K)


# ---------------------------------------------------------------- strides of tens of megabytes

@pytest.mark.parametrize("acc", [False, True], ids=["plain", "acc"])
@pytest.mark.parametrize("shape", [(1024, 4096, 5), (1024, 2000, 2)])
def test_dst_columns_far_apart(hip, shape, acc):
    """Few dst columns 100 MB and more apart: the kernels form offsets for up to 28
    columns, and those of columns that are not there pass 2^31 and 2^32. Nothing but
    the columns is written, and they hold the product."""
    K, M, N = shape
    stride = 400_000_000 // (N - 1)                    # bytes; 27 of them pass 2^31 (N = 2: 2^32 too)
    announce(f"mul_mat dst columns {stride} bytes apart {shape} {'acc' if acc else ''}")
    A = synth.normal(980 + N, K * M).reshape(1, 1, K, M)   # row-contiguous: tiles, not the few-column kernel
    B = synth.normal(981 + N, K * N).reshape(1, 1, N, K)
    da, db = Dev(A), Dev(B)
    total = stride // 4 * (N - 1) + M
    buf = H.DeviceBuffer(4 * total)
    H.fill_f32(buf.ptr, 0.5, total)
    d = H.tensor(buf.ptr, [M, N, 1, 1], [4, stride, stride * N, stride * N])
    (H.mul_mat_acc_f32 if acc else H.mul_mat_f32)(da.tensor(t01(A)), db.tensor(), d)
    H.sync()
    out = buf.download(np.empty(total, np.float32))
    for x in (da, db, buf):
        x.free()
    cols = [out[j * (stride // 4):j * (stride // 4) + M] for j in range(N)]
    got = np.stack(cols)[None, None]
    want = O.mul_mat(t01(A), B, threads=8)
    assert O.row_l2_error(got, want + np.float32(0.5) if acc else want) <= TOL
    for c in cols:
        c[:] = 0.5
    assert np.all(out == np.float32(0.5))


def test_operand_rows_far_apart(hip):
    """A transposed operand with 80 MB from one k to the next: the loads form offsets
    up to the end of the last slab of 32 k, past 2^31."""
    K, M, N, stride = 20, 4096, 4096, 80_000_000
    announce("mul_mat src0 with k 80 MB apart")
    A, B = synth.normal(985, K * M).reshape(K, M), synth.normal(986, K * N).reshape(1, 1, N, K)
    buf = H.DeviceBuffer(stride * (K - 1) + 4 * M)
    for k in range(K):
        H.check(H.load().trc_hip_h2d(buf.ptr + k * stride, A[k].ctypes.data, 4 * M, None))
    db, out = Dev(B), empty((1, 1, N, M))
    H.mul_mat_f32(H.tensor(buf.ptr, [K, M, 1, 1], [stride, 4, 4 * M, 4 * M]), db.tensor(), out.tensor())
    H.sync()
    got = out.read()
    for x in (buf, db, out):
        x.free()
    assert O.row_l2_error(got, O.mul_mat(t01(A[None, None]), B, threads=8)) <= TOL


# ---------------------------------------------------------------- more workgroups than a launch takes

@pytest.mark.parametrize("case", [
    # (K, M, N, src0 planes, src1 planes): the few-column kernel's limit of 4.2 million
    # workgroups and the tiles' of 16.8 million, the planes along either dimension
    (4, 1, 1, (2, 3), (700000, 6)), (4, 1, 1, (1, 2), (1, 4200002)), (4, 1, 3, (1, 5000000), (1, 5000000)),
    (1, 1, 1, (2, 3), (2800000, 6)), (1, 1, 1, (1, 1), (1, 16777300)), (1, 1, 1, (8400000, 1), (8400000, 2)),
])
@pytest.mark.parametrize("acc", [False, True], ids=["plain", "acc"])
def test_more_planes_than_one_launch_takes(hip, case, acc):
    K, M, N, (a3, a2), (b3, b2) = case
    announce(f"mul_mat planes past one launch {case}")
    rng = np.random.default_rng(K + b3)
    A = rng.integers(-8, 9, (a3, a2, M, K)).astype(np.float32)
    B = rng.integers(-8, 9, (b3, b2, N, K)).astype(np.float32)
    D = rng.integers(-8, 9, (b3, b2, N, M)).astype(np.float32)
    da, db, out = Dev(A), Dev(B), Dev(D)
    (H.mul_mat_acc_f32 if acc else H.mul_mat_f32)(da.tensor(), db.tensor(), out.tensor())
    H.sync()
    got = out.read()
    for d in (da, db, out):
        d.free()
    want = (B[..., :, None, :] * np.tile(A, (b3 // a3, b2 // a2, 1, 1))[..., None, :, :]).sum(-1)
    assert np.array_equal(got, want + D if acc else want)


def test_more_rows_than_one_launch_takes(hip):
    """A src0 of 67.2 million rows of 4: 4.2 million workgroups of 16 rows."""
    K, M, N = 4, 67_200_000, 2
    announce(f"mul_mat rows past one launch {M}")
    rng = np.random.default_rng(29)
    A = rng.integers(-8, 9, (1, 1, M, K), dtype=np.int8).astype(np.float32)
    B = rng.integers(-8, 9, (1, 1, N, K)).astype(np.float32)
    da, db = Dev(A), Dev(B)
    got = gpu_mul_mat(da, A, db, B)
    da.free()
    db.free()
    assert np.array_equal(got[0, 0], B[0, 0] @ A[0, 0].T)
