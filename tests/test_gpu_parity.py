"""GPU parity tests: every kernel, called through the gpu* C ABI, against the CPU
oracle on the same seeded inputs; reference golden vectors; size-independent
properties at the full benchmark shapes.

Bars: bit-exact for relu / transpose / reduce_outer / integer GEMM; <= 1 ulp for
SiLU (f32); |d| <= 1e-3 |ref| + 2^-24 for f16 softmax (2^-24 = one f16 subnormal
step, the output type's absolute resolution) and 1e-3 relative for row sums;
max|d| <= 5e-3 max|ref| for the GEMMs.
"""
import json
import os

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

HERE = os.path.dirname(os.path.abspath(__file__))
with open(os.path.join(HERE, "golden", "reference_vectors.json")) as f:
    GOLD = json.load(f)


def arr(v, shape=None):
    a = np.asarray(v, np.float32)
    return a.reshape(shape) if shape else a


def say(msg):
    print("[case] " + msg, flush=True)


# =============================== ReLU =====================================
def test_relu_golden_and_specials(host, orc, stream):
    g = GOLD["relu_f32_4x5_spirv"]
    assert np.array_equal(host.relu(stream, arr(g["input"], g["shape"])), arr(g["expected"], g["shape"]))
    x = np.array([0x7fc00001, 0xffc12345, 0x80000000, 0, 1, 0x80000001, 0x7f800000, 0xff800000, 0x7f800001],
                 np.uint32).view(np.float32)
    assert np.array_equal(host.relu(stream, x).view(np.uint32), orc.relu_f32(x).view(np.uint32))


@pytest.mark.parametrize("n", [1, 3, 4095, 4096, 4097, 100003, 1 << 20])
def test_relu_ragged_sizes(host, orc, stream, n):
    say("relu n=%d" % n)
    x = orc.fill_uniform(n, "f32", 20241 + n % 7, -1.0, 1.0)
    assert np.array_equal(host.relu(stream, x).view(np.uint32), orc.relu_f32(x).view(np.uint32))


def test_relu_config_4096x4096(host, orc, stream):
    x = orc.fill_uniform(4096 * 4096, "f32", 20241, -1.0, 1.0).reshape(4096, 4096)
    assert np.array_equal(host.relu(stream, x).view(np.uint32), orc.relu_f32(x).view(np.uint32))


def test_relu_every_f32_pattern(host, stream):
    """All 2^32 bit patterns against the closed form (x if x > 0 or NaN else +0)."""
    chunk = 1 << 27
    for base in range(0, 1 << 32, chunk):
        if base % (1 << 30) == 0:
            say("relu sweep base=0x%08x" % base)
        u = np.arange(base, base + chunk, dtype=np.uint32)
        got = host.relu(stream, u.view(np.float32)).view(np.uint32)
        keep = (u.view(np.int32) > 0) | (u > np.uint32(0xff800000))
        assert np.array_equal(got, np.where(keep, u, np.uint32(0)))


@pytest.mark.parametrize("dtype", ["f16", "bf16"])
def test_relu_every_16bit_pattern(host, orc, stream, dtype):
    x = np.tile(np.arange(65536, dtype=np.uint16), 3)[:-5]  # unaligned tail
    assert np.array_equal(host.relu(stream, x, dtype), orc.relu_16(x, dtype))


# =============================== SiLU =====================================
def test_silu_within_one_ulp(host, orc, stream):
    x = np.concatenate([
        orc.fill_uniform(1 << 20, "f32", 20251, -8.0, 8.0),
        orc.fill_uniform(1 << 18, "f32", 1, -110.0, 110.0),
        orc.fill_bits(1 << 18, "f32", 2).view(np.float32),
        np.array([0.0, -0.0, 1.3, np.inf, -np.inf, 88.0, -88.0, 88.72, 88.73, -103.9, -104.0, 1e-45, -1e-45, 1e38,
                  -1e38], np.float32),
        np.array([0x7fc00000], np.uint32).view(np.float32)])
    got, ref = host.silu(stream, x), orc.silu_f32(x)
    nan = np.isnan(ref)
    assert np.array_equal(np.isnan(got), nan)
    d = orc.ulp_distance_f32(got[~nan], ref[~nan])
    say("silu max ulp distance %d, exact %d of %d" % (d.max(), int((d == 0).sum()), d.size))
    assert d.max() <= 1
    assert host.silu(stream, np.array([0.0], np.float32))[0] == 0.0


def test_silu_same_bits_as_the_oracle_on_ordinary_inputs(host, orc, stream):
    """|x| < 64 takes the kernel's straight-line form (exp without its special cases, the reciprocal
    as an explicit refinement sequence): the same bits as libm's expf and an IEEE division, on every
    f32 in [1, 2) (2^23 consecutive values) and on 8 Mi values spread over (-64, 64)."""
    sweep = np.arange(0x3f800000, 0x40000000, dtype=np.uint32).view(np.float32)
    spread = orc.fill_uniform(1 << 23, "f32", 77, -63.99, 63.99)
    for name, x in (("every f32 in [1,2)", sweep), ("-every f32 in [1,2)", -sweep), ("uniform(-64,64)", spread)):
        say("silu bit-exact: " + name)
        assert np.array_equal(host.silu(stream, x).view(np.uint32), orc.silu_f32(x).view(np.uint32)), name


def test_silu_benchmark_shape(host, orc, stream):
    x = orc.fill_uniform(512 * 640 * 20 * 15, "f32", 20251, -8.0, 8.0)
    got, ref = host.silu(stream, x), orc.silu_f32(x)
    assert orc.ulp_distance_f32(got, ref).max() <= 1


# ============================ exp, maximum ================================
def test_exp_same_bits_as_libm(host, orc, stream):
    """WG/math_exp.mlir: math.exp against the CPU loop's libm call -- the test's own input range
    (-0.5, 0.5), the whole finite range, and the special values."""
    for name, x in (("reference range", orc.fill_uniform(256 * 256, "f32", 31, -0.5, 0.5)),
                    ("(-110, 110)", orc.fill_uniform(1 << 21, "f32", 32, -110.0, 110.0)),
                    ("(-64, 64) ragged", orc.fill_uniform((1 << 20) + 13, "f32", 33, -63.9, 63.9))):
        say("exp: " + name)
        assert np.array_equal(host.exp(stream, x).view(np.uint32), orc.expf_n(x).view(np.uint32)), name
    special = np.array([0.0, -0.0, np.inf, -np.inf, 88.72, 88.73, -103.9, -104.0, 1e-45, -1e-45, 1e38, -1e38, 64.0, -64.0],
                       np.float32)
    assert np.array_equal(host.exp(stream, special).view(np.uint32), orc.expf_n(special).view(np.uint32))
    assert np.isnan(host.exp(stream, np.array([np.nan], np.float32))[0])


def test_maximum_matches_the_oracle(host, orc, stream):
    """WG/arith_maximumf.mlir: bit for bit where no operand is NaN, NaN where one is."""
    a, b = orc.fill_uniform(256 * 256, "f32", 41, -0.5, 0.5), orc.fill_uniform(256 * 256, "f32", 42, -0.5, 0.5)
    assert np.array_equal(host.maximum(stream, a, b), np.maximum(a, b))
    n = (1 << 20) + 7
    a, b = orc.fill_bits(n, "f32", 43).view(np.float32).copy(), orc.fill_bits(n, "f32", 44).view(np.float32).copy()
    a[:8] = [0.0, -0.0, -0.0, np.inf, -np.inf, np.nan, 1.0, np.nan]
    b[:8] = [-0.0, 0.0, -0.0, 1.0, -1.0, 1.0, np.nan, np.nan]
    got, ref = host.maximum(stream, a, b), orc.maximum_f32(a, b)
    nan = np.isnan(ref)
    assert np.array_equal(np.isnan(got), nan) and nan[5] and nan[6] and nan[7]
    assert np.array_equal(got[~nan].view(np.uint32), ref[~nan].view(np.uint32))


# =============================== Softmax ==================================
def close_16(orc, got_bits, ref_bits, dtype):
    got, ref = orc.to_float(got_bits, dtype), orc.to_float(ref_bits, dtype)
    quantum = 2.0 ** -24 if dtype == "f16" else 0.0
    rtol = 1e-3 if dtype == "f16" else 2.0 ** -7  # bf16: one unit in the last place
    return np.all(np.abs(got - ref) <= rtol * np.abs(ref) + quantum)


@pytest.mark.parametrize("key", ["softmax_f32_10x20", "softmax_f32_10x20_spirv"])
def test_softmax_golden(host, orc, stream, key):
    g = GOLD[key]
    got = host.softmax(stream, arr(g["input"], g["shape"]), "f32")
    want = arr(g["expected"], g["shape"])
    assert np.max(np.abs(got - want) / want) < 2e-5
    assert orc.allclose_f32(got, want)


def test_softmax_config_f16_16384x1024(host, orc, stream):
    x = orc.fill_normal(16384 * 1024, "f16", 20242, 0.0, 2.0).reshape(16384, 1024)
    got, ref = host.softmax(stream, x, "f16"), orc.softmax_16(x, "f16")
    assert close_16(orc, got, ref, "f16")
    assert orc.allclose_f32(orc.half_to_float(got), orc.softmax_f32(orc.half_to_float(x)))
    sums = orc.half_to_float(got).sum(axis=1, dtype=np.float64)
    assert np.max(np.abs(sums - 1.0)) < 2e-3  # 1024 outputs each rounded to f16


@pytest.mark.parametrize("rows,cols", [(1, 1), (3, 7), (5, 8), (16, 2000), (64, 2000), (7, 1000), (9, 512), (4, 4096),
                                       (3, 5000), (2, 65536 + 8), (1025, 64), (6, 1016),
                                       (16385, 24), (20001, 8)])  # two rows per wavefront, odd row counts
@pytest.mark.parametrize("dtype", ["f16", "f32"])
def test_softmax_shapes(host, orc, stream, rows, cols, dtype):
    say("softmax %s %dx%d" % (dtype, rows, cols))
    x = orc.fill_normal(rows * cols, dtype, rows * 131 + cols, 0.0, 2.0).reshape(rows, cols)
    got = host.softmax(stream, x, dtype)
    if dtype == "f32":
        ref = orc.softmax_f32(x)
        assert np.all(np.abs(got - ref) <= 1e-3 * np.abs(ref))
        assert np.max(np.abs(got - ref) / np.maximum(ref, 1e-30)) < 5e-5
    else:
        assert close_16(orc, got, orc.softmax_16(x, "f16"), "f16")


def test_softmax_bf16_and_exact_rows(host, orc, stream):
    x = orc.fill_normal(64 * 1024, "bf16", 9, 0.0, 2.0).reshape(64, 1024)
    assert close_16(orc, host.softmax(stream, x, "bf16"), orc.softmax_16(x, "bf16"), "bf16")
    eq = orc.float_to_half(np.full((8, 1024), 3.3, np.float32))
    assert np.all(host.softmax(stream, eq, "f16") == 0x1400)  # exactly 2^-10
    # a row of -inf-free extremes: one dominant element
    x = np.full((4, 1024), -20.0, np.float32)
    x[:, 5] = 20.0
    got = host.softmax(stream, x, "f32")
    assert np.all(got[:, 5] == 1.0) and got.sum() == 4.0


@pytest.mark.parametrize("rows,cols", [(3, 5000), (2, 65536 + 8), (5, 4097), (2, 300001)])
def test_softmax_long_rows_streaming_form(host, orc, stream, rows, cols):
    """Rows beyond 4096 columns take the running (max, sum) form of WG/softmax_intra_sg_cross_lane.mlir:135-175;
    checked against the reference's scalar three-pass loop (:85-117) and the benchmark form, on random
    rows, on a ramp whose maximum moves with every vector (every partial sum is rescaled again and
    again), on its mirror image, and on one huge element at the very end."""
    say("softmax streaming %dx%d" % (rows, cols))
    x = orc.fill_normal(rows * cols, "f32", 81 + cols % 7, 0.0, 2.0).reshape(rows, cols).copy()
    x[0] = np.linspace(-40.0, 30.0, cols, dtype=np.float32)  # outputs stay normal f32 numbers (the hardware exp flushes subnormal results)
    x[1] = x[0][::-1]
    if rows > 2:
        x[2, -1] = 60.0
    got = host.softmax(stream, x, "f32")
    for ref in (orc.softmax_f32(x, three_pass=True), orc.softmax_f32(x)):
        assert np.all(np.abs(got - ref) <= 1e-3 * np.abs(ref))  # the stated bar
    # the sequential f32 sum of the reference loop carries up to ~2e-4 of rounding over 300 001 addends (it
    # differs by that much between a row and its mirror image); against the exact row sum the kernel is tighter
    assert np.max(np.abs(got.sum(axis=1, dtype=np.float64) - 1.0)) < 2e-5
    xh = orc.from_float(x, "f16")
    assert close_16(orc, host.softmax(stream, xh, "f16"), orc.softmax_16(xh, "f16"), "f16")


@pytest.mark.parametrize("cols,path", [(1024, "registers"), (2000, "lds"), (5000, "streamed")])
def test_softmax_reciprocal_deviation_is_one_rounding(host, orc, stream, cols, path):
    """The kernel multiplies by one reciprocal per row where the reference divides per element.  What that may
    cost, pinned on each of the kernel's three paths: an f16 output is the oracle's divided result or its
    neighbour (one unit in the last place), and all but a small fraction are the same bits."""
    say("softmax reciprocal deviation, %s path, cols=%d" % (path, cols))
    x = orc.fill_normal(64 * cols, "f16", 4242 + cols, 0.0, 2.0).reshape(64, cols)
    got, ref = host.softmax(stream, x, "f16"), orc.softmax_16(x, "f16")
    steps = np.abs(got.astype(np.int32) - ref.astype(np.int32))  # positive f16 bit patterns are ordered like their values
    assert steps.max() <= 1
    assert np.mean(steps == 0) > 0.98


@pytest.mark.parametrize("dtype,cols", [("f32", 20), ("f32", 512), ("f16", 1024), ("f32", 3000), ("f16", 4096),
                                        ("f32", 5000), ("f16", 70000)])
def test_softmax_nan_and_infinite_rows(host, orc, stream, dtype, cols):
    """Rows the benchmark's inputs never hold, on every path of the kernel (registers, LDS, streamed):
    a NaN anywhere makes its whole row NaN (arith.maximumf and the sum both carry it), a row of
    nothing but -inf is 0/0 = NaN because the running maximum starts at -3.40282347e38 rather than
    -inf, +inf in a row gives inf - inf = NaN, and a -inf among finite values is an exact zero."""
    say("softmax special rows %s cols=%d" % (dtype, cols))
    x = orc.to_float(orc.fill_normal(6 * cols, dtype, 71, 0.0, 2.0), dtype).reshape(6, cols).copy()
    x[1, cols // 3] = np.nan
    x[2, :] = -np.inf
    x[3, cols - 1] = np.inf
    x[4, 0] = -np.inf
    x[5, :] = -3.0e38 if dtype == "f32" else -65504.0
    xin = x if dtype == "f32" else orc.from_float(x, dtype)
    got = orc.to_float(host.softmax(stream, xin, dtype), dtype)
    ref = orc.softmax_f32(x) if dtype == "f32" else orc.to_float(orc.softmax_16(xin, dtype), dtype)
    assert np.array_equal(np.isnan(got), np.isnan(ref))
    assert np.isnan(ref[1]).all() and np.isnan(ref[2]).all() and np.isnan(ref[3]).all() and not np.isnan(ref[[0, 4, 5]]).any()
    assert got[4, 0] == 0.0
    ok = ~np.isnan(ref)
    assert np.all(np.abs(got[ok] - ref[ok]) <= 1e-3 * np.abs(ref[ok]) + (2.0 ** -24 if dtype == "f16" else 0.0))


@pytest.mark.parametrize("dtype", ["f32", "f16", "bf16"])
@pytest.mark.parametrize("rows,pieces", [(40001, 0.75), (40001, 1), (70000, 4), (70000, 4.25), (9001, 8.75), (9001, 16.5),
                                         (4500, 32.25), (4500, 63.75), (2049, 64.25), (2049, 129.5), (2048, 256), (2047, 255.75),
                                         (3000, 256.25), (3, 1023.75), (5, 1024.25), (5, 3072.5), (3, 4095.75), (2, 4096.25)])
def test_softmax_rows_of_any_length_and_address(host, orc, stream, rows, pieces, dtype):
    """Rows at the edges of the kernel's splits (16-byte pieces per row: less than one, a lane's four, a wavefront's
    256, a workgroup's 1024, 2048 and 4096), from buffers that start one element behind a 16-byte boundary, and the
    elements on either side of the result untouched.  Tolerances: those of test_softmax_shapes; bf16 outputs are
    the oracle's value or its neighbour (one rounding, 2^-8, of quotients that differ by f32 roundings)."""
    per, width = (4, 4) if dtype == "f32" else (8, 2)
    cols = int(pieces * per)
    say("softmax %s %dx%d, unaligned" % (dtype, rows, cols))
    x = orc.fill_normal(rows * cols, dtype, rows + cols, 0.0, 2.0)
    raw = np.zeros(rows * cols + 2, x.dtype)
    raw[1:-1] = x
    d_in, d_out = stream.to_device(raw), stream.to_device(np.full_like(raw, 7))
    stream.launch("imex_softmax_" + dtype, [rows, cols], [host.Ptr(d_in + width), host.Ptr(d_out + width), rows, cols])
    stream.wait()
    got = stream.from_device(d_out, (rows * cols + 2,), raw.dtype)
    stream.free(d_in), stream.free(d_out)
    assert got[0] == 7 and got[-1] == 7
    got, x = got[1:-1].reshape(rows, cols), x.reshape(rows, cols)
    if dtype == "f32":
        ref = orc.softmax_f32(x)
        assert np.max(np.abs(got - ref) / np.maximum(ref, 1e-30)) < 5e-5
    elif dtype == "f16":
        assert close_16(orc, got, orc.softmax_16(x, "f16"), "f16")
    else:
        ref = orc.softmax_16(x, "bf16")
        assert np.max(np.abs(got.astype(np.int32) - ref.astype(np.int32))) <= 1


@pytest.mark.parametrize("dtype", ["f32", "f16", "bf16"])
@pytest.mark.parametrize("rows,pieces", [(2500, 0.5), (700, 20.25), (1500, 65), (20003, 96), (300, 100.5), (1023, 129), (1024, 129),
                                         (40, 300), (7, 641), (5, 1025), (4, 1537), (3, 2049), (3, 4096), (2, 4100)])
def test_softmax_forms_by_their_own_names(host, orc, stream, rows, pieces, dtype):
    """The operator itself and its _shared form, each by its own name under its own launch shape and on two workgroups
    that walk all rows (a C caller need not take the advice of imexHipKernelVariant).  Tolerances: those of
    test_softmax_rows_of_any_length_and_address."""
    cols = int(pieces * (4 if dtype == "f32" else 8))
    x = orc.fill_normal(rows * cols, dtype, 3 * rows + cols, 0.0, 2.0).reshape(rows, cols)
    ref = orc.softmax_f32(x) if dtype == "f32" else orc.softmax_16(x, dtype)
    blank = np.zeros_like(x)
    d_in, d_out = stream.to_device(x), stream.alloc(x.nbytes)
    for name in ("imex_softmax_" + dtype, "imex_softmax_%s_shared" % dtype):
        grid, block, _ = host.launch_shape(name, [rows, cols])
        for g in (grid, (2, 1, 1)):
            say("%s %dx%d grid %s block %s" % (name, rows, cols, g, block))
            stream.copy(d_out, blank.ctypes.data, x.nbytes)
            stream.launch(name, [rows, cols], [d_in, d_out, rows, cols], grid=g, block=block)
            stream.wait()
            got = stream.from_device(d_out, (rows, cols), x.dtype)
            if dtype == "f32":
                assert np.max(np.abs(got - ref) / np.maximum(ref, 1e-30)) < 5e-5
            elif dtype == "f16":
                assert close_16(orc, got, ref, "f16")
            else:
                assert np.max(np.abs(got.astype(np.int32) - ref.astype(np.int32))) <= 1
    stream.free(d_in), stream.free(d_out)


@pytest.mark.parametrize("rows,cols", [(1000, 1024), (1000, 1016), (37, 1024), (4097, 1024), (5, 8)])
def test_softmax_f16_rows_in_registers_any_grid(host, orc, stream, rows, cols):
    """The f16 register path walks its rows with the next row's loads in flight: a wavefront that takes one
    row, two, three (odd and even trip counts of the two-row loop) or a few hundred gives the same bits as
    the catalogue's grid, for whole 1024-column rows and for rows that leave lanes without a vector."""
    say("softmax f16 walk %dx%d" % (rows, cols))
    x = orc.fill_normal(rows * cols, "f16", 7 * rows + cols, 0.0, 2.0).reshape(rows, cols)
    x[rows // 2, cols // 2] = 0x7E00  # a NaN row in the middle of a walk
    ref = orc.softmax_16(x, "f16")
    want = host.softmax(stream, x, "f16")
    nan = np.isnan(orc.half_to_float(ref))
    assert np.array_equal(np.isnan(orc.half_to_float(want)), nan) and nan[rows // 2].all() and nan.sum() == cols
    ok = ~nan
    assert close_16(orc, want[ok], ref[ok], "f16")
    for grid in (1, 2, -(-rows // 12), -(-rows // 8), -(-rows // 4) + 3):
        d_in, d_out = stream.to_device(x), stream.alloc(rows * cols * 2)
        stream.launch("imex_softmax_f16", [rows, cols], [d_in, d_out, rows, cols], grid=(grid, 1, 1))
        stream.wait()
        got = stream.from_device(d_out, (rows, cols), np.uint16)
        stream.free(d_in), stream.free(d_out)
        assert np.array_equal(got[ok], want[ok]) and np.isnan(orc.half_to_float(got[~ok])).all(), grid


# =============================== Reductions ================================
def test_rowsum_golden_and_exact(host, orc, stream):
    g = GOLD["sum_f32_10x20"]
    x = arr(g["input"], g["shape"])
    assert np.array_equal(host.rowsum(stream, x), np.full(10, 210.0, np.float32))
    assert host.rowsum(stream, x.reshape(1, 200))[0] == 2100.0
    g = GOLD["wg_reduction_rows"]
    x = np.repeat(np.arange(8, dtype=np.float32)[:, None], 256, axis=1)
    assert list(host.rowsum(stream, x)) == g["expected"]
    assert host.rowsum(stream, np.ones((1, 65536), np.float32))[0] == 65536.0
    # integer-valued inputs: any summation order is exact
    for rows, cols in [(37, 1000), (5, 8192), (3, 4099), (130, 2048), (2, 2052), (9, 1)]:
        xi = orc.fill_int(rows * cols, "f32", rows + cols, -8, 8).reshape(rows, cols)
        assert np.array_equal(host.rowsum(stream, xi, init=3.0), orc.rowsum_f32(xi, init=3.0)), (rows, cols)


@pytest.mark.parametrize("cols", [1, 3, 4, 5, 63, 64, 65, 129, 256, 511, 513, 1023, 1024, 1025, 1030, 2049, 3001, 4096, 4099])
def test_row_sums_of_any_length_and_address(host, orc, stream, cols):
    """Rows at the edges of the lane groups (four 16-byte pieces a lane, 4 .. 64 lanes) and of the longer forms, from a
    buffer that starts one element behind a 16-byte boundary.  Integer values: the sums are exact in any order."""
    rows = 333
    x = orc.fill_int(rows * cols, "f32", cols, -8, 8)
    d_in, d_out = stream.to_device(np.concatenate([np.float32([np.nan]), x, np.float32([np.nan])])), stream.alloc(rows * 4)
    x = x.reshape(rows, cols)
    for name, rest, want in (("rowsum", [3.0], orc.rowsum_f32(x, init=3.0)), ("rowmean", [], orc.rowmean_f32(x))):
        stream.launch("imex_%s_f32" % name, [rows, cols], [host.Ptr(d_in + 4), d_out, rows, cols, *rest])
        stream.wait()
        assert np.array_equal(stream.from_device(d_out, (rows,), np.float32), want), name
    stream.free(d_in), stream.free(d_out)


@pytest.mark.parametrize("cols", [4, 63, 129, 300, 1023])
def test_short_row_sums_walk(host, orc, stream, cols):
    """The forms whose lanes share a wavefront, on three workgroups that walk all rows.  Integer values: exact sums."""
    rows = 1501
    x = orc.fill_int(rows * cols, "f32", cols, -8, 8).reshape(rows, cols)
    d_in, d_out = stream.to_device(x), stream.alloc(rows * 4)
    for name, rest, want in (("rowsum", [3.0], orc.rowsum_f32(x, init=3.0)), ("rowmean", [], orc.rowmean_f32(x))):
        say("%s %dx%d, three workgroups" % (name, rows, cols))
        stream.launch("imex_%s_f32_short" % name, [rows, cols], [d_in, d_out, rows, cols, *rest], grid=(3, 1, 1))
        stream.wait()
        assert np.array_equal(stream.from_device(d_out, (rows,), np.float32), want), name
    stream.free(d_in), stream.free(d_out)


def test_rowsum_config_8192x8192(host, orc, stream):
    x = orc.fill_uniform(8192 * 8192, "f32", 20243, 0.0, 1.0).reshape(8192, 8192)
    got, ref = host.rowsum(stream, x), orc.rowsum_f32(x)
    assert np.max(np.abs(got - ref) / np.abs(ref)) <= 1e-3
    exact = x.sum(axis=1, dtype=np.float64)
    say("rowsum rel err vs f64: kernel %.2e, sequential oracle %.2e" %
        (np.max(np.abs(got - exact) / exact), np.max(np.abs(ref - exact) / exact)))
    assert np.max(np.abs(got - exact) / exact) < 1e-5


@pytest.mark.parametrize("dtype", ["f16", "bf16"])
def test_silu_sixteen_bit(host, orc, stream, dtype):
    """benchmarks/silu/silu.dtypes.in lists f16: widen, the f32 chain, one rounding -- same bits as the oracle.
    Every 16-bit pattern once (NaNs compared as NaNs), then the benchmark's 1x1024x40x30 and a large ragged size."""
    every = np.arange(65536, dtype=np.uint16)
    got, ref = host.silu(stream, every, dtype), orc.silu_16(every, dtype)
    gf, rf = orc.to_float(got, dtype), orc.to_float(ref, dtype)
    nan = np.isnan(rf)
    assert np.array_equal(np.isnan(gf), nan) and np.array_equal(got[~nan], ref[~nan])
    for n in (1024 * 40 * 30, (1 << 22) + 4099):
        x = orc.fill_uniform(n, dtype, 304, -8.0, 8.0)
        assert np.array_equal(host.silu(stream, x, dtype), orc.silu_16(x, dtype)), n


@pytest.mark.parametrize("dtype", ["f16", "bf16"])
@pytest.mark.parametrize("shape", [(32, 16, 64, 64), (10, 24), (7, 1023), (3, 512 * 4096 + 16), (5, 512 * 2048 + 3)])
def test_reduce_outer_sixteen_bit(host, orc, stream, dtype, shape):
    """benchmarks/reduce/reduce.dtypes.in lists f16 and bf16: f32 accumulation in slice order, one rounding."""
    x = orc.fill_uniform(int(np.prod(shape)), dtype, 305, -1.0, 1.0).reshape(shape)
    got = host.reduce_outer(stream, x, init=0.25, dtype=dtype)
    assert np.array_equal(got, orc.reduce_outer_16(x, dtype, init=0.25))


def test_rowmean(host, orc, stream):
    """Mean over the last dimension (WG/reduction_4D_3D_mean_intra_sg_intra_lane.mlir: 1x24x1024x64,
    uniform(-1,1) inputs, checked there against the sequential CPU loop with allclose)."""
    x = orc.fill_uniform(24 * 1024 * 64, "f32", 79, -1.0, 1.0).reshape(24 * 1024, 64)
    got, ref = host.rowmean(stream, x), orc.rowmean_f32(x)
    assert np.all(np.abs(got - ref) <= 1e-4 + 1e-3 * np.abs(ref))   # the reference's allclose
    assert np.max(np.abs(got - ref)) <= 2e-7                          # and far inside it
    # integer-valued rows: the sum is exact in any order, so the mean is the oracle's bits
    for rows, cols in ((7, 64), (5, 3000), (1000, 96), (3, 1)):
        m = orc.fill_int(rows * cols, "f32", 80, -8, 8).reshape(rows, cols)
        assert np.array_equal(host.rowmean(stream, m), orc.rowmean_f32(m)), (rows, cols)


@pytest.mark.parametrize("shape", [(32, 16, 64, 64), (10, 20), (7, 1023), (33, 4100), (1, 5), (3, 1, 9),
                                   (5, 512 * 2048 + 4), (3, 512 * 4096 + 1028), (2, 512 * 8192 + 8), (6, 512 * 2048 + 3)])
def test_reduce_outer_bit_exact(host, orc, stream, shape):
    """The catalogue's choice: the operator's own form with 16 and 32 KiB of a slice per workgroup and a ragged last one for
    3 and 2 slices of whole vectors, a lane per vector or output for the other large ones, column chains for the tall."""
    x = orc.fill_uniform(int(np.prod(shape)), "f32", 77, -1.0, 1.0).reshape(shape)
    got, ref = host.reduce_outer(stream, x, init=0.25), orc.reduce_outer_f32(x, init=0.25)
    assert np.array_equal(got.view(np.uint32), ref.view(np.uint32))


@pytest.mark.parametrize("dtype", ["f32", "f16", "bf16"])
@pytest.mark.parametrize("outer,inner,chosen", [(3, 2 * 512 + 1.25, True), (4, 2 * 512, True), (5, 4 * 512 + 3, True), (2, 8 * 512 + 1, True),
                                                (6, 2.5 * 512, True), (5, 2 * 512 + 0.25, False), (7, 300.125, False),
                                                (130, 0.5, False), (10, 0.03125, False)])
def test_reduce_outer_own_launch(host, orc, stream, dtype, outer, inner, chosen):
    """The operator's own kernel under its own launch; `inner` counts a workgroup's row of 256 16-byte vectors.  What the
    catalogue leaves to it (slices of 4 MiB and more for up to four of them, of 5 MiB, 16-bit: 8 MiB, beyond that): two, four
    and eight vectors per lane, with a whole and a ragged last workgroup; and what it gives to the other forms."""
    name, vec = "imex_reduce_outer_" + dtype, 4 if dtype == "f32" else 8
    cols = int(inner * 256 * vec) + (1 if inner % 1 == 0.125 else 0)  # (0.125: no whole vectors)
    if chosen and (dtype == "f32" or inner != 2.5 * 512):
        assert host.variant(name, [outer, cols]) == name
    x = orc.fill_uniform(outer * cols, dtype, 94, -1.0, 1.0).reshape(outer, cols)
    want = orc.reduce_outer_f32(x if dtype == "f32" else orc.to_float(x, dtype), 0.25)
    want = want if dtype == "f32" else orc.from_float(want, dtype)
    fill = np.full(cols + 64, 3, x.dtype)
    d_in, d_out = stream.to_device(x), stream.alloc(fill.nbytes)
    grid, block, _ = host.launch_shape(name, [outer, cols])
    for g in (grid, (5, 1, 1)):
        say("%s %dx%d, grid %s" % (name, outer, cols, g))
        stream.copy(d_out, fill.ctypes.data, fill.nbytes)
        stream.launch(name, [outer, cols], [d_in, d_out, outer, cols, 0.25], grid=g, block=block)
        stream.wait()
        got = stream.from_device(d_out, fill.shape, fill.dtype)
        assert np.array_equal(got[:cols], want), (name, g)
        assert np.all(got[cols:] == 3), (name, g)
    stream.free(d_in), stream.free(d_out)


@pytest.mark.parametrize("form", ["_tall", "_deep"])
@pytest.mark.parametrize("dtype", ["f32", "f16", "bf16"])
@pytest.mark.parametrize("outer,inner", [(1, 8), (16, 1), (17, 65), (63, 40), (64, 130), (65, 1032), (129, 67), (520, 8),
                                         (577, 2049), (0, 16)])
def test_reduce_outer_forms_bit_exact(host, orc, stream, form, dtype, outer, inner):
    """Both further forms of the outer-dimension sum around their rings (16 slices; chunks of 64, eight of them) and
    segments (32 / 64 columns, 256 lanes), with and without whole 16-byte vectors: the slices are added in order, so
    the result is the oracle's bit for bit; nothing behind it is written, and any grid computes it."""
    x = orc.fill_uniform(max(outer * inner, 1), dtype, 91, -1.0, 1.0)[:outer * inner].reshape(outer, inner)
    want = orc.reduce_outer_f32(orc.to_float(x, dtype) if dtype != "f32" else x, 0.25) if outer else None
    want = np.full(inner, 0.25, np.float32) if want is None else want
    want = want if dtype == "f32" else orc.from_float(want, dtype)
    fill = np.full(inner + 256, 3, x.dtype)
    name = "imex_reduce_outer_" + dtype + form
    d_in, d_out = stream.to_device(x), stream.to_device(fill)
    for grid in (None, (2, 1, 1)):
        stream.copy(d_out, fill.ctypes.data, fill.nbytes)
        stream.launch(name, [outer, inner], [d_in, d_out, outer, inner, 0.25], grid=grid)
        stream.wait()
        got = stream.from_device(d_out, fill.shape, fill.dtype)
        assert np.array_equal(got[:inner], want), (name, outer, inner, grid)
        assert np.array_equal(got[inner:], fill[inner:]), (name, outer, inner, grid)
    stream.free(d_in)
    stream.free(d_out)


@pytest.mark.parametrize("form", ["_tall", "_deep"])
@pytest.mark.parametrize("dtype", ["f32", "f16", "bf16"])
@pytest.mark.parametrize("outer,inner", [(1, 4104), (2, 520), (131, 520)])
def test_reduce_outer_forms_at_any_address(host, orc, stream, form, dtype, outer, inner):
    """Slices of whole 16-byte vectors in a buffer that starts one element behind a 16-byte boundary, and a result that
    does: the loops that stand in for the vector forms add in the same order."""
    width = 4 if dtype == "f32" else 2
    x = orc.fill_uniform(outer * inner, dtype, 92, -1.0, 1.0)
    wide = (x if dtype == "f32" else orc.to_float(x, dtype)).reshape(outer, inner)
    want = orc.reduce_outer_f32(wide, 0.25)
    want = want if dtype == "f32" else orc.from_float(want, dtype)
    name = "imex_reduce_outer_" + dtype + form
    for shift_in, shift_out in ((1, 0), (0, 1), (1, 1)):
        say("%s %dx%d, bases %d and %d elements off" % (name, outer, inner, shift_in, shift_out))
        fill = np.full(inner + 2, 3, x.dtype)
        d_in = stream.to_device(np.concatenate([np.zeros(shift_in, x.dtype), x]))
        d_out = stream.to_device(fill)
        stream.launch(name, [outer, inner], [host.Ptr(d_in + shift_in * width), host.Ptr(d_out + shift_out * width), outer, inner, 0.25])
        stream.wait()
        got = stream.from_device(d_out, fill.shape, fill.dtype)
        stream.free(d_in), stream.free(d_out)
        assert np.array_equal(got[shift_out:shift_out + inner], want), (name, shift_in, shift_out)
        assert np.all(got[:shift_out] == 3) and np.all(got[shift_out + inner:] == 3)


def test_reduce_outer_benchmark_shape_and_any_grid(host, orc, stream):
    """32x16x512x512 (the reference suite's reduce shape, README.md:335): integer-valued inputs
    make the sum exact; then the same kernel on a grid of 7 workgroups, which must stride."""
    import ctypes as C
    outer, inner = 32, 16 * 512 * 512
    x = orc.fill_int(outer * inner, "f32", 78, -8, 8).reshape(outer, inner)
    got = host.reduce_outer(stream, x, init=1.0)
    assert np.array_equal(got, 1.0 + x.sum(axis=0, dtype=np.float64).astype(np.float32))
    small = x[:, :300000]
    small = np.ascontiguousarray(small)
    d_in, d_out = stream.to_device(small), stream.alloc(small.shape[1] * 4)
    fn = stream.kernel("imex_reduce_outer_f32")
    descs, keep = host._pack_params([d_in, d_out, outer, small.shape[1], 1.0])
    stream.rt.gpuLaunchKernel(stream.handle, fn, 7, 1, 1, 256, 1, 1, 0, C.cast(descs, C.c_void_p), None)
    stream.wait()
    out = stream.from_device(d_out, (small.shape[1],), np.float32)
    stream.free(d_in)
    stream.free(d_out)
    assert np.array_equal(out, 1.0 + small.sum(axis=0, dtype=np.float64).astype(np.float32))


@pytest.mark.parametrize("grid", [(3, 1, 1), (100000, 1, 1)])
def test_streaming_kernels_any_grid(host, orc, stream, grid):
    """relu, silu, softmax, row sum and the fused chain stride over their work: a grid much
    smaller or much larger than the catalogue's gives the same bits."""
    n = 3 * 4096 * 5 + 77
    x = orc.fill_uniform(n, "f32", 91, -3, 3)
    for kernel, ref in (("imex_relu_f32", orc.relu_f32(x)), ("imex_silu_f32", orc.silu_f32(x))):
        d_in, d_out = stream.to_device(x), stream.alloc(n * 4)
        stream.launch(kernel, [n], [d_in, d_out, n], grid=grid)
        stream.wait()
        got = stream.from_device(d_out, (n,), np.float32)
        stream.free(d_in), stream.free(d_out)
        assert np.array_equal(got.view(np.uint32), ref.view(np.uint32)), kernel
    for rows, cols in ((37, 3000), (1000, 300)):
        m = orc.fill_int(rows * cols, "f32", 92, -8, 8).reshape(rows, cols)
        d_in, d_out = stream.to_device(m), stream.alloc(rows * 4)
        stream.launch("imex_rowsum_f32", [rows, cols], [d_in, d_out, rows, cols, 2.0], grid=grid)
        stream.wait()
        got = stream.from_device(d_out, (rows,), np.float32)
        stream.free(d_in), stream.free(d_out)
        assert np.array_equal(got, 2.0 + m.sum(axis=1, dtype=np.float64).astype(np.float32)), (rows, cols)
    a = np.abs(orc.fill_uniform(n, "f32", 93, -3, 3)) + 0.5
    d_a, d_b, d_out = stream.to_device(x), stream.to_device(a), stream.alloc(n * 4)
    stream.launch("imex_loop_fusion_f32", [n], [d_a, d_b, d_out, n], grid=grid)
    stream.wait()
    got = stream.from_device(d_out, (n,), np.float32)
    for p in (d_a, d_b, d_out):
        stream.free(p)
    assert np.array_equal(got.view(np.uint32), orc.loop_fusion_f32(x, a).view(np.uint32))


@pytest.mark.parametrize("kind,dtype", [("relu", "f32"), ("relu", "bf16"), ("silu", "f32"), ("silu", "f16"), ("silu", "bf16"),
                                        ("exp", "f32"), ("maximum", "f32"), ("loop_fusion", "f32"), ("loop_fusion", "f16"),
                                        ("loop_fusion", "bf16")])
def test_last_block_of_a_tensor(host, orc, stream, kind, dtype):
    """Tensors that end inside a block of four vectors per lane: fewer elements than a vector, a wavefront's vectors and one
    more, all but one element, whole blocks; NaN and infinities behind them, nothing written there; against the oracle."""
    wide = lambda t: t if dtype == "f32" else orc.to_float(t, dtype)
    narrow = lambda t: t if dtype == "f32" else orc.from_float(t, dtype)
    ops = {"relu": lambda a, b: orc.relu_f32(a) if dtype == "f32" else orc.relu_16(a, dtype),
           "silu": lambda a, b: orc.silu_f32(a) if dtype == "f32" else orc.silu_16(a, dtype),
           "exp": lambda a, b: orc.expf_n(a), "maximum": lambda a, b: orc.maximum_f32(a, b),
           "loop_fusion": lambda a, b: narrow(orc.loop_fusion_f32(wide(a), wide(b)))}
    per, block, whole = (4, 4096, 1 << 22) if dtype == "f32" else (8, 8192, 1 << 22)
    two, size, tail = kind in ("maximum", "loop_fusion"), whole + 2 * block, 3 * block
    a = orc.fill_uniform(size, dtype, 33, 0.5, 6.0) if kind == "loop_fusion" else orc.fill_uniform(size, dtype, 33, -6.0, 6.0)
    b = orc.fill_uniform(size, dtype, 34, -3.0, 3.0)
    for past in (0, 1, per - 1, per, 64 * per, 65 * per, 256 * per + 3, block - per, block - 1, block):
        n = whole + past
        say("%s %s, %d elements" % (kind, dtype, n))
        beside = narrow(np.resize(np.float32([np.nan, -np.inf, -1.0]), 64))
        ins = [np.concatenate([t[:n], beside]) for t in ((a, b) if two else (a,))]
        bufs, d_out = [stream.to_device(t) for t in ins], stream.to_device(np.full(n + 64, 3, a.dtype))
        stream.launch("imex_%s_%s" % (kind, dtype), [n], bufs + [d_out, n])
        stream.wait()
        got = stream.from_device(d_out, (n + 64,), a.dtype)
        for p in bufs + [d_out]:
            stream.free(p)
        bits = np.uint32 if dtype == "f32" else np.uint16
        want = ops[kind](a[n - tail:n].copy(), b[n - tail:n].copy())
        assert np.array_equal(got[n - tail:n].view(bits), want.view(bits)), past
        assert np.all(got[n:] == 3), past


# =============================== Transpose =================================
def test_transpose_golden(host, orc, stream):
    g = GOLD["transpose_f32_10x20"]
    assert np.array_equal(host.transpose2d(stream, arr(g["input"], g["shape"])), arr(g["expected"], [20, 10]))
    g = GOLD["transpose_bf16_10x20"]
    xb = orc.float_to_bfloat(arr(g["input"], g["shape"]))
    assert np.array_equal(orc.bfloat_to_float(host.transpose2d(stream, xb)), arr(g["expected"], [20, 10]))


@pytest.mark.parametrize("rows,cols", [(1, 1), (64, 64), (128, 136), (1024, 1024), (63, 65), (8, 2000), (200, 8),
                                       (72, 520), (1000, 3), (257, 129)])
@pytest.mark.parametrize("dtype", ["bf16", "f32"])
def test_transpose_shapes_bit_exact(host, orc, stream, rows, cols, dtype):
    say("transpose %s %dx%d" % (dtype, rows, cols))
    x = orc.fill_bits(rows * cols, dtype, 20244 + rows).reshape(rows, cols)
    got = host.transpose2d(stream, x)
    assert np.array_equal(got, orc.transpose2d(x))
    assert np.array_equal(host.transpose2d(stream, got), x)  # involution


def test_transpose_config_sizes(host, orc, stream):
    x = orc.fill_bits(8192 * 8192, "bf16", 20244).reshape(8192, 8192)
    got = host.transpose2d(stream, x)
    assert np.array_equal(got, x.T)
    # index-encoded input: every element lands where its index says
    idx = np.arange(4096 * 4096, dtype=np.uint32).reshape(4096, 4096)
    assert np.array_equal(host.transpose2d(stream, idx), idx.T)
    y = orc.fill_bits(4096 * 4096, "f32", 20245).reshape(4096, 4096)
    assert np.array_equal(host.transpose2d(stream, y), orc.transpose2d(y))


@pytest.mark.parametrize("rows,cols", [(4104, 4120), (8200, 2056), (300, 65544)])
@pytest.mark.parametrize("dtype", ["bf16", "f32"])
def test_transpose_large_tiles_ragged(host, orc, stream, rows, cols, dtype):
    """From 2^24 elements the kernels use 128 x 128 (32-bit) / 256 x 128 (16-bit)
    tiles; these shapes end in partial tiles on both sides."""
    x = orc.fill_bits(rows * cols, dtype, 20244 + cols).reshape(rows, cols)
    got = host.transpose2d(stream, x)
    assert np.array_equal(got, x.T)


@pytest.mark.parametrize("rows,planes,cols", [(8, 1, 9), (9, 1, 8), (4, 1, 5), (7, 1, 300), (256, 1, 65), (257, 1, 64), (255, 3, 63),
                                              (264, 1, 1001), (1001, 1, 264), (129, 2, 33), (513, 5, 191), (4097, 1, 4001)])
@pytest.mark.parametrize("dtype", ["bf16", "f32"])
def test_transpose_of_any_size_and_address(host, orc, stream, rows, planes, cols, dtype):
    """Sizes at the edges of the blocks and tiles for rows that are no whole 16-byte vectors, from buffers that start
    one element behind a 16-byte boundary; both kernels of the operator, the elements around the result untouched."""
    n, width, bits = rows * planes * cols, 4 if dtype == "f32" else 2, 32 if dtype == "f32" else 16
    say("transpose %s %dx%dx%d, unaligned" % (dtype, rows, planes, cols))
    raw = orc.fill_bits(n + 2, dtype, rows + cols).view(np.uint32 if dtype == "f32" else np.uint16)
    want = raw[1:-1].reshape(rows, planes, cols).transpose(2, 1, 0)
    dims = [rows, cols] if planes == 1 else [rows, planes, cols]
    name = "imex_transpose%dd_b%d" % (len(dims), bits)
    for grid in (None, (3, 1, 1)):  # the catalogue's choice; the operator itself, its workgroups walking the tiles
        d_in, d_out = stream.to_device(raw), stream.to_device(np.full_like(raw, 7))
        stream.launch(name, dims, [host.Ptr(d_in + width), host.Ptr(d_out + width), *dims], grid=grid)
        stream.wait()
        got = stream.from_device(d_out, raw.shape, raw.dtype)
        stream.free(d_in), stream.free(d_out)
        assert got[0] == 7 and got[-1] == 7
        assert np.array_equal(got[1:-1].reshape(want.shape), want)


@pytest.mark.parametrize("rows,planes,cols,bits,form", [
    (4104, 1, 4120, 16, "_any"), (4128, 1, 4120, 16, ""), (4128, 1, 24, 16, ""), (2184, 1, 16, 16, ""), (2056, 1, 16, 16, "_any"),
    (4100, 1, 4104, 32, "_any"), (4112, 1, 4120, 32, ""), (40, 7, 104, 16, "_any"), (32, 7, 104, 16, ""),
    (20, 3, 68, 32, "_any"), (16, 3, 68, 32, "")])
def test_transpose_by_lines_of_the_result(host, orc, stream, rows, planes, cols, bits, form):
    """Whole 16-byte vectors: results whose rows are whole 64 bytes, or few and long, by the operator's own kernel; the
    elements around the result untouched."""
    dims = [rows, cols] if planes == 1 else [rows, planes, cols]
    name = "imex_transpose%dd_b%d" % (len(dims), bits)
    assert host.variant(name, dims) == name + form
    say("%s %r by its lines" % (name, dims))
    x = orc.fill_bits(rows * planes * cols, "f32" if bits == 32 else "bf16", rows).view(np.uint32 if bits == 32 else np.uint16)
    d_in, d_out = stream.to_device(x), stream.to_device(np.full(x.size + 64, 7, x.dtype))
    stream.launch(name, dims, [d_in, host.Ptr(d_out + 32 * x.itemsize), *dims])
    stream.wait()
    got = stream.from_device(d_out, (x.size + 64,), x.dtype)
    stream.free(d_in), stream.free(d_out)
    assert np.all(got[:32] == 7) and np.all(got[-32:] == 7)
    assert np.array_equal(got[32:-32].reshape(dims[::-1]), x.reshape(dims).transpose(*range(len(dims))[::-1]))


@pytest.mark.parametrize("rows,cols", [(4096, 4224), (128, 131072), (8192, 4096)])
def test_transpose_b32_whole_tiles_pipelined(host, orc, stream, rows, cols):
    """32-bit problems made of whole 128 x 128 tiles: at most 512 workgroups, each walking two or more tiles
    with the next tile's loads issued before the current tile is written (an odd and an even number of tiles
    per workgroup, a single tile row)."""
    x = np.arange(rows * cols, dtype=np.uint32).reshape(rows, cols)
    assert np.array_equal(host.transpose2d(stream, x), x.T)


def test_transpose3d_b32_whole_tiles_pipelined(host, orc, stream):
    shape = (256, 64, 1024)
    x = np.arange(int(np.prod(shape)), dtype=np.uint32).reshape(shape)
    assert np.array_equal(host.transpose3d(stream, x), x.transpose(2, 1, 0))


def test_transpose_any_grid(host, orc, stream):
    """Workgroups stride over the tiles: a grid smaller or larger than one workgroup
    per tile gives the same result."""
    import ctypes as C
    for name, np_t, rows, cols in [("imex_transpose2d_b32", np.uint32, 4096, 4104), ("imex_transpose2d_b16", np.uint16, 520, 264),
                                   ("imex_transpose2d_b32", np.uint32, 4096, 4096)]:
        x = np.arange(rows * cols, dtype=np.uint64).astype(np_t).reshape(rows, cols)
        for grid in [(3, 1, 1), (7, 5, 2), (40, 30, 1)]:
            d_in, d_out = stream.to_device(x), stream.alloc(x.nbytes)
            fn = stream.kernel(name)
            descs, keep = host._pack_params([d_in, d_out, rows, cols])
            stream.rt.gpuLaunchKernel(stream.handle, fn, grid[0], grid[1], grid[2], 256, 1, 1, 0,
                                      C.cast(descs, C.c_void_p), None)
            stream.wait()
            got = stream.from_device(d_out, (cols, rows), np_t)
            stream.free(d_in)
            stream.free(d_out)
            assert np.array_equal(got, x.T), (name, grid)


@pytest.mark.parametrize("shape", [(16, 96, 96), (96, 7, 96), (5, 3, 9), (64, 2, 72), (520, 64, 512)])
def test_transpose3d(host, orc, stream, shape):
    n = int(np.prod(shape))
    x32 = orc.fill_bits(n, "f32", 5).reshape(shape)
    assert np.array_equal(host.transpose3d(stream, x32), orc.transpose3d(x32))
    x16 = orc.fill_bits(n, "f16", 6).reshape(shape)
    assert np.array_equal(host.transpose3d(stream, x16), x16.transpose(2, 1, 0))


# ========================= fused element-wise chains ========================
@pytest.mark.parametrize("shape", [(512, 1024), (7, 13), (1, 4097), (300, 1000)])
def test_loop_fusion_f32_bit_exact(host, orc, stream, shape):
    """kLoopFusion: the device logf is the host libm's algorithm, every op is a
    separately rounded f32 one, so the result is the oracle's bit for bit."""
    n = int(np.prod(shape))
    a = orc.fill_uniform(n, "f32", 41, 0.01, 40.0).reshape(shape)
    b = orc.fill_uniform(n, "f32", 42, -5.0, 5.0).reshape(shape)
    a.flat[:6] = [3.3, 1.0, 1e-40, 0.0, np.inf, 0.99999994]
    got = host.loop_fusion(stream, a, b)
    want = orc.loop_fusion_f32(a, b)
    assert np.array_equal(got.view(np.uint32), want.view(np.uint32))


def test_loop_fusion_logf_sweep(host, orc, stream):
    """b = 0 and exact cancellation aside, out + a = log a: sweep log over 16M bit
    patterns of the whole positive range through the fused kernel."""
    bits = (np.arange(1 << 24, dtype=np.uint64) * 127 + 1).astype(np.uint32) % np.uint32(0x7f800000)
    a = bits.view(np.float32)
    b = np.zeros_like(a)
    got = host.loop_fusion(stream, a, b)
    want = orc.loop_fusion_f32(a, b)
    assert np.array_equal(got.view(np.uint32), want.view(np.uint32))


def test_empty_inputs_every_operator(host, stream):
    """Tensors with a zero extent: nothing is launched (a grid of zero workgroups is not a launch), results have
    the right shape, a row sum over no columns is the initial value and a product over K = 0 is all zeros."""
    f = np.float32
    assert host.relu(stream, np.zeros((0,), f)).shape == (0,)
    assert host.silu(stream, np.zeros((0,), f)).shape == (0,)
    assert host.softmax(stream, np.zeros((0, 16), f), "f32").shape == (0, 16)
    assert host.softmax(stream, np.zeros((4, 0), f), "f32").shape == (4, 0)
    assert host.rowsum(stream, np.zeros((0, 16), f)).shape == (0,)
    assert np.array_equal(host.rowsum(stream, np.zeros((5, 0), f)), np.zeros(5, f))
    assert host.transpose2d(stream, np.zeros((0, 7), f)).shape == (7, 0)
    assert host.transpose2d(stream, np.zeros((7, 0), f)).shape == (0, 7)
    assert host.gemm(stream, np.zeros((0, 8), np.uint16), np.zeros((8, 16), np.uint16)).shape == (0, 16)
    assert np.array_equal(host.gemm(stream, np.zeros((4, 0), np.uint16), np.zeros((0, 16), np.uint16)), np.zeros((4, 16), f))


def test_fused_chains_empty_and_single(host, orc, stream):
    empty = np.zeros((0,), np.float32)
    assert host.loop_fusion(stream, empty, empty).shape == (0,)
    one = host.loop_fusion(stream, np.float32([2.5]), np.float32([-1.5]))
    assert np.array_equal(one, orc.loop_fusion_f32(np.float32([2.5]), np.float32([-1.5])))
    no_rows = host.input_fusion(stream, np.zeros((0, 12), np.float32), np.zeros((0, 12), np.float32))
    assert np.array_equal(no_rows.view(np.uint32), np.zeros(12, np.uint32))  # a sum over nothing: +0.0
    col = host.input_fusion(stream, np.float32([[1.0], [-2.0], [3.0]]), np.float32([[0.5], [2.0], [8.0]]))
    assert np.array_equal(col, orc.input_fusion_f32(np.float32([[1.0], [-2.0], [3.0]]), np.float32([[0.5], [2.0], [8.0]])))


@pytest.mark.parametrize("dtype", ["f16", "bf16"])
def test_loop_fusion_16bit(host, orc, stream, dtype):
    n = 512 * 1024 + 77
    a = orc.fill_uniform(n, dtype, 43, 0.05, 30.0)
    b = orc.fill_uniform(n, dtype, 44, -5.0, 5.0)
    got = orc.to_float(host.loop_fusion(stream, a, b, dtype), dtype)
    # widen, f32 chain, one rounding at the end
    want = orc.to_float(orc.from_float(orc.loop_fusion_f32(orc.to_float(a, dtype), orc.to_float(b, dtype)), dtype), dtype)
    assert np.array_equal(got, want)


@pytest.mark.parametrize("n", [1 << 16, (1 << 22) + 8192 + 5])
@pytest.mark.parametrize("dtype", ["f16", "bf16"])
def test_loop_fusion_16bit_every_logarithm(host, orc, stream, dtype, n):
    """Every 16-bit pattern under the logarithm, in order, so that whole wavefronts hold ordinary numbers and others zeros,
    infinities, NaN and negative ones; with one and with four vectors per lane and a tail: the oracle's bits (of a NaN,
    that it is one)."""
    a = np.resize(np.arange(1 << 16, dtype=np.uint16), n)
    b = orc.fill_uniform(n, dtype, 49, -2.0, 2.0)
    got = orc.to_float(host.loop_fusion(stream, a, b, dtype), dtype)
    want = orc.to_float(orc.from_float(orc.loop_fusion_f32(orc.to_float(a, dtype), orc.to_float(b, dtype)), dtype), dtype)
    assert np.array_equal(np.isnan(got), np.isnan(want))
    assert np.array_equal(got.view(np.uint32)[~np.isnan(want)], want.view(np.uint32)[~np.isnan(want)])


# The catalogue's choice: the operator's own launch for (9, 5) and (513, 4), column chains for the others, (2049, 4098) with
# rows that are no whole vectors.  (The operator's own launch at such sizes: test_input_fusion_own_launch.)
@pytest.mark.parametrize("shape", [(512, 1024), (9, 5), (1000, 300), (3, 2049), (1500, 36), (513, 4), (2048, 4096),
                                   (2500, 4100), (2049, 4098)])
def test_input_fusion_f32_bit_exact(host, orc, stream, shape):
    """kInputFusion: column sums in row order from +0.0, as the reference adds them."""
    n = int(np.prod(shape))
    a = orc.fill_uniform(n, "f32", 45, -5.0, 5.0).reshape(shape)
    b = orc.fill_uniform(n, "f32", 46, 0.01, 40.0).reshape(shape)
    got = host.input_fusion(stream, a, b)
    want = orc.input_fusion_f32(a, b)
    assert got.shape == (shape[1],)
    assert np.array_equal(got.view(np.uint32), want.view(np.uint32))


@pytest.mark.parametrize("shape", [(512, 1024), (700, 41), (2048, 8192), (2100, 8200)])
@pytest.mark.parametrize("dtype", ["f16", "bf16"])
def test_input_fusion_16bit(host, orc, stream, dtype, shape):
    rows, cols = shape
    a = orc.fill_uniform(rows * cols, dtype, 47, -2.0, 2.0).reshape(rows, cols)
    b = orc.fill_uniform(rows * cols, dtype, 48, 0.5, 4.0).reshape(rows, cols)
    got = orc.to_float(host.input_fusion(stream, a, b, dtype), dtype)
    want = orc.to_float(orc.from_float(orc.input_fusion_f32(orc.to_float(a, dtype), orc.to_float(b, dtype)), dtype), dtype)
    assert np.array_equal(got, want)


@pytest.mark.parametrize("dtype", ["f32", "f16", "bf16"])
@pytest.mark.parametrize("rows,cols", [(100, 500), (127, 2047), (3, 17000), (20, 37008), (9, 5), (512, 1024), (700, 41), (1000, 300),
                                       (1500, 36), (513, 4), (65, 4097), (1030, 5000), (33, 9001), (33, 25520), (129, 33001),
                                       (2048, 8192), (2500, 8200), (2049, 8202)])
def test_input_fusion_own_launch(host, orc, stream, dtype, rows, cols):
    """The operator's own kernel under its own launch, on the catalogue's grid and on three workgroups, where the catalogue
    leaves a problem to it (the first four) and where it takes the chains: four columns per workgroup with 320 lanes and
    with 256 (one group of tiles, several, partial ones), blocks of 8, 16, 32 and 64 columns, segments of 128 bytes for
    many rows."""
    name = "imex_input_fusion_" + dtype
    if (rows, cols) in ((100, 500), (127, 2047), (3, 17000), (20, 37008)):
        assert host.variant(name, [rows, cols]) == name
    wide = lambda t: t if dtype == "f32" else orc.to_float(t, dtype)
    a = orc.fill_uniform(rows * cols, dtype, 65, -5.0, 5.0).reshape(rows, cols)
    b = orc.fill_uniform(rows * cols, dtype, 66, 0.01, 40.0).reshape(rows, cols)
    want = orc.input_fusion_f32(wide(a), wide(b))
    want = want if dtype == "f32" else orc.from_float(want, dtype)
    fill = np.full(cols + 16, 3, a.dtype)
    d_a, d_b, d_out = stream.to_device(a), stream.to_device(b), stream.to_device(fill)
    grid, block, _ = host.launch_shape(name, [rows, cols])
    for launch in ((grid, block), ((3, 1, 1), block), (grid, (256, 1, 1))):
        say("%s %dx%d, %s" % (name, rows, cols, launch))
        stream.copy(d_out, fill.ctypes.data, fill.nbytes)
        stream.launch(name, [rows, cols], [d_a, d_b, d_out, rows, cols], grid=launch[0], block=launch[1])
        stream.wait()
        got = stream.from_device(d_out, fill.shape, fill.dtype)
        assert np.array_equal(got[:cols], want), (name, launch)
        assert np.all(got[cols:] == 3), (name, launch)
    for p in (d_a, d_b, d_out):
        stream.free(p)


@pytest.mark.parametrize("shape,block", [((600, 520), 320), ((2048, 4160), 576), ((2048, 4160), 256), ((600, 520), 256)])
def test_input_fusion_any_grid(host, orc, stream, shape, block):
    """Workgroups stride over the blocks of columns in every form of the kernel (the narrow and the wide
    streaming form, and the 256-lane form a launch with 256 lanes always gets): a grid of a few
    workgroups gives the same bits as the catalogue's."""
    import ctypes as C
    rows, cols = shape
    a = orc.fill_uniform(rows * cols, "f32", 51, -5.0, 5.0).reshape(shape)
    b = orc.fill_uniform(rows * cols, "f32", 52, 0.01, 40.0).reshape(shape)
    want = orc.input_fusion_f32(a, b)
    d_a, d_b, d_out = stream.to_device(a), stream.to_device(b), stream.alloc(cols * 4)
    fn = stream.kernel("imex_input_fusion_f32")
    descs, keep = host._pack_params([d_a, d_b, d_out, rows, cols])
    for grid in (1, 7):
        stream.memset(d_out, 0x7fc00000, cols, 32)
        stream.rt.gpuLaunchKernel(stream.handle, fn, grid, 1, 1, block, 1, 1, 0, C.cast(descs, C.c_void_p), None)
        stream.wait()
        got = stream.from_device(d_out, (cols,), np.float32)
        assert np.array_equal(got.view(np.uint32), want.view(np.uint32)), (shape, block, grid)
    for p in (d_a, d_b, d_out):
        stream.free(p)


@pytest.mark.parametrize("dtype", ["f32", "f16", "bf16"])
@pytest.mark.parametrize("rows,segments,extra", [(1, 1, 0), (255, 1, 1), (256, 3, -1), (257, 256, 0), (1000, 256, -7),
                                                 (127, 256, 1), (129, 512, 0), (271, 511, 3), (128, 512, 1),
                                                 (513, 515, 5), (64, 1024, 9), (0, 4, 0), (63, 1030, 3), (65, 1030, 1),
                                                 (128, 1025, 0), (200, 1100, 5), (321, 1025, -1)])
def test_column_chains_bit_exact(host, orc, stream, dtype, rows, segments, extra):
    """The fused chain and the plain sum down the columns around the tiles of rows (256 and 128; 64 beyond 1024 32-byte
    segments in a row, where every step of the adder's loop hands a tile over) and the widths of a workgroup's segment (32,
    64 and 128 bytes: up to 256, up to 512 and more segments), with buffers on and one element off the 16-byte grid, on the catalogue's grid, on five workgroups and with lanes that the chains do not
    take: the additions are in row order, so the results are the oracle's bits.  Zeros, infinities, NaN, negative and
    subnormal numbers stand under the logarithm of some columns."""
    width = 4 if dtype == "f32" else 2
    cols = segments * (32 // width) + extra
    wide = lambda t: t if dtype == "f32" else orc.to_float(t, dtype)
    narrow = lambda t: t if dtype == "f32" else orc.from_float(t, dtype)
    a = orc.fill_uniform(max(rows * cols, 1), dtype, 53, -5.0, 5.0)[:rows * cols].reshape(rows, cols)
    b = orc.fill_uniform(max(rows * cols, 1), dtype, 54, 0.01, 40.0)[:rows * cols].reshape(rows, cols)
    if rows > 2 and cols > 16:
        b[rows // 2, :6] = narrow(np.float32([0.0, -0.0, np.inf, -3.0, np.nan, 1e-40]))
        b[-1, -2:] = narrow(np.float32([1e-39, 1.0]))
    zeros = lambda init: np.full(cols, init, np.float32)
    want = {"input_fusion": narrow(orc.input_fusion_f32(wide(a), wide(b)) if rows else zeros(0.0)),
            "reduce_outer": narrow(orc.reduce_outer_f32(wide(a), 0.25) if rows else zeros(0.25))}
    for shift in (0, 1):
        at = lambda t: stream.to_device(np.concatenate([np.zeros(shift, t.dtype), t.ravel(), np.zeros(8, t.dtype)]))
        d_a, d_b = at(a), at(b)
        fill = np.full(cols + 16, 3, a.dtype)
        d_out = stream.to_device(fill)
        p_a, p_b, p_out = (host.Ptr(p + shift * width) for p in (d_a, d_b, d_out))
        for op, args in (("input_fusion", [p_a, p_b, p_out, rows, cols]), ("reduce_outer", [p_a, p_out, rows, cols, 0.25])):
            name = "imex_%s_%s_tall" % (op, dtype)
            for launch in ({}, {"grid": (5, 1, 1)}, {"block": (256, 1, 1)}):
                say("%s %dx%d, %d off, %s" % (name, rows, cols, shift, launch))
                stream.copy(d_out, fill.ctypes.data, fill.nbytes)
                stream.launch(name, [rows, cols], args, **launch)
                stream.wait()
                got = stream.from_device(d_out, fill.shape, fill.dtype)
                res, ref = wide(got[shift:shift + cols]), wide(want[op])
                assert np.array_equal(np.isnan(res), np.isnan(ref)), (name, launch)
                assert np.array_equal(got[shift:shift + cols][~np.isnan(ref)], want[op][~np.isnan(ref)]), (name, launch)
                assert np.all(got[:shift] == 3) and np.all(got[shift + cols:] == 3), (name, launch)
        for p in (d_a, d_b, d_out):
            stream.free(p)


@pytest.mark.parametrize("dtype", ["f32", "f16", "bf16"])
@pytest.mark.parametrize("segments,extra", [(288, 1), (384, 0), (512, 0)])
def test_column_chains_tiles_ahead(host, orc, stream, dtype, segments, extra):
    """Sums of 64-byte segments over 1 .. 9 tiles of 128 rows and last tiles that end on and beside the sixteen rows that are
    added at a time; rows of whole 4 KiB too.  The oracle's bits, also with a sum of -0 behind which the padding of the last sixteen rows must leave no trace."""
    cols = segments * (32 // (4 if dtype == "f32" else 2)) + extra
    wide = lambda t: t if dtype == "f32" else orc.to_float(t, dtype)
    narrow = lambda t: t if dtype == "f32" else orc.from_float(t, dtype)
    a = orc.fill_uniform(1153 * cols, dtype, 63, -5.0, 5.0).reshape(1153, cols)
    a[:, 5] = narrow(np.full(1, -0.0, np.float32))
    d_in, d_out = stream.to_device(a), stream.alloc(cols * a.itemsize)
    for rows in (1, 128, 143, 257, 384, 385, 400, 511, 513, 640, 769, 1000, 1153):
        say("%d x %d" % (rows, cols))
        for grid in (None, (7, 1, 1)):
            stream.launch("imex_reduce_outer_%s_tall" % dtype, [rows, cols], [d_in, d_out, rows, cols, -0.0], grid=grid)
            stream.wait()
            got = stream.from_device(d_out, (cols,), a.dtype)
            want = narrow(orc.reduce_outer_f32(wide(a[:rows]), -0.0))
            assert np.array_equal(got.view(np.uint8), want.view(np.uint8)), (rows, grid)
    stream.free(d_in), stream.free(d_out)


@pytest.mark.parametrize("dtype", ["f32", "f16", "bf16"])
@pytest.mark.parametrize("segments,extra", [(399, 3), (512, 0)])
def test_column_chains_from_memory(host, orc, stream, dtype, segments, extra):
    """The same from 84 MiB on, where three tiles are in flight: on both sides of the line, every number of tiles modulo the
    four of the ring, last tiles that end on and beside sixteen rows.  The oracle's bits."""
    cols = segments * (32 // (4 if dtype == "f32" else 2)) + extra
    wide = lambda t: t if dtype == "f32" else orc.to_float(t, dtype)
    narrow = lambda t: t if dtype == "f32" else orc.from_float(t, dtype)
    first = -(-(84 << 20) // (cols * (4 if dtype == "f32" else 2)))
    tiles = -(-first // 128)
    most = (tiles + 4) * 128
    a = orc.fill_uniform(most * cols, dtype, 64, -5.0, 5.0).reshape(most, cols)
    d_in, d_out = stream.to_device(a), stream.alloc(cols * a.itemsize)
    for rows in (first - 1, first, tiles * 128, tiles * 128 + 1, tiles * 128 + 144, tiles * 128 + 257, most - 1, most):
        say("%d x %d" % (rows, cols))
        for grid in (None, (7, 1, 1)):
            stream.launch("imex_reduce_outer_%s_tall" % dtype, [rows, cols], [d_in, d_out, rows, cols, 0.25], grid=grid)
            stream.wait()
            got = stream.from_device(d_out, (cols,), a.dtype)
            want = narrow(orc.reduce_outer_f32(wide(a[:rows]), 0.25))
            assert np.array_equal(got.view(np.uint8), want.view(np.uint8)), (rows, grid)
    stream.free(d_in), stream.free(d_out)


@pytest.mark.parametrize("dtype", ["f32", "f16", "bf16"])
@pytest.mark.parametrize("rows,cols", [(150, 41), (130, 2100), (40, 5000), (129, 3)])
def test_input_fusion_with_any_block(host, orc, stream, dtype, rows, cols):
    """Launches with fewer lanes than a form's tiles are filled by, with a number that no form asks for, and on two
    workgroups: the oracle's bits, also for the numbers that libm does not send down its main path."""
    wide = lambda t: t if dtype == "f32" else orc.to_float(t, dtype)
    narrow = lambda t: t if dtype == "f32" else orc.from_float(t, dtype)
    a = orc.fill_uniform(rows * cols, dtype, 57, -5.0, 5.0).reshape(rows, cols)
    b = orc.fill_uniform(rows * cols, dtype, 58, 0.01, 40.0).reshape(rows, cols)
    b[rows // 2, :2] = narrow(np.float32([0.0, np.inf]))
    want = narrow(orc.input_fusion_f32(wide(a), wide(b)))
    d_a, d_b, d_out = stream.to_device(a), stream.to_device(b), stream.alloc(cols * a.itemsize)
    junk = orc.fill_uniform(cols, dtype, 59, 100.0, 200.0)
    for form in ("", "_tall"):
        for lanes in (1, 8, 64, 192, 255, 384, 512):
            for grid in (None, (2, 1, 1)):
                name = "imex_input_fusion_" + dtype + form
                stream.copy(d_out, junk.ctypes.data, junk.nbytes)
                stream.launch(name, [rows, cols], [d_a, d_b, d_out, rows, cols], grid=grid, block=(lanes, 1, 1))
                stream.wait()
                got = stream.from_device(d_out, (cols,), a.dtype)
                assert np.array_equal(got, want), (name, lanes, grid)
    for p in (d_a, d_b, d_out):
        stream.free(p)


@pytest.mark.parametrize("dtype,rows,cols", [("f32", 73, (1 << 20) + 5), ("f16", 30, (1 << 21) + 3), ("bf16", 66, (1 << 21) + 8)])
def test_column_chains_rows_of_4_mib(host, orc, stream, dtype, rows, cols):
    """Rows of 4 MiB and more, in one and in two tiles of 64 rows: offsets inside a tile pass 2^28."""
    wide = lambda t: t if dtype == "f32" else orc.to_float(t, dtype)
    narrow = lambda t: t if dtype == "f32" else orc.from_float(t, dtype)
    assert host.variant("imex_input_fusion_" + dtype, [rows, cols]) == "imex_input_fusion_%s_tall" % dtype
    a = orc.fill_uniform(rows * cols, dtype, 61, -5.0, 5.0).reshape(rows, cols)
    b = orc.fill_uniform(rows * cols, dtype, 62, 0.01, 40.0).reshape(rows, cols)
    assert np.array_equal(host.input_fusion(stream, a, b, dtype), narrow(orc.input_fusion_f32(wide(a), wide(b))))
    d_in, d_out = stream.to_device(a), stream.alloc(cols * a.itemsize)
    stream.launch("imex_reduce_outer_%s_tall" % dtype, [rows, cols], [d_in, d_out, rows, cols, 0.25], grid=(1000, 1, 1))
    stream.wait()
    got = stream.from_device(d_out, (cols,), a.dtype)
    stream.free(d_in), stream.free(d_out)
    assert np.array_equal(got, narrow(orc.reduce_outer_f32(wide(a), 0.25)))


@pytest.mark.parametrize("dtype", ["f32", "f16", "bf16"])
@pytest.mark.parametrize("cols", range(1, 17))
def test_reduce_outer_narrow_rows(host, orc, stream, dtype, cols):
    """Rows of less than a 32-byte segment, down to one element: by the catalogue's choice, which takes the chains for tall
    ones, and by the chains themselves, with matrices of less than 8 bytes, lanes that start inside another's columns, loads
    that run past a row and the matrix's end in the middle of a tile and behind it; on and off the 16-byte grid; the
    oracle's bits, and nothing written beside them."""
    name, width = "imex_reduce_outer_" + dtype, 4 if dtype == "f32" else 2
    assert host.variant(name, [8192, cols]) == name + "_tall"
    for rows in (1, 2, 3, 5, 255, 256, 257, 258, 259, 700, 8195):
        x = orc.fill_uniform(rows * cols, dtype, 93, -1.0, 1.0)
        want = orc.reduce_outer_f32((x if dtype == "f32" else orc.to_float(x, dtype)).reshape(rows, cols), 0.25)
        want = want if dtype == "f32" else orc.from_float(want, dtype)
        for shift in (0, 1):
            # NaN in front of the matrix and behind it: what is read past its ends must not be added
            nan = np.full(8, np.nan, np.float32) if dtype == "f32" else np.full(8, 0x7fff, np.uint16)
            d_in = stream.to_device(np.concatenate([nan[:shift], x, nan]))
            fill = np.full(cols + 8, 3, x.dtype)
            for form in ("", "_tall"):
                d_out = stream.to_device(fill)
                stream.launch(name + form, [rows, cols], [host.Ptr(d_in + shift * width), host.Ptr(d_out + shift * width), rows, cols, 0.25])
                stream.wait()
                got = stream.from_device(d_out, fill.shape, fill.dtype)
                stream.free(d_out)
                assert np.array_equal(got[shift:shift + cols], want), (name + form, rows, shift)
                assert np.all(got[:shift] == 3) and np.all(got[shift + cols:] == 3), (name + form, rows, shift)
            stream.free(d_in)


@pytest.mark.parametrize("dtype", ["f32", "f16", "bf16"])
@pytest.mark.parametrize("cols", range(1, 17))
def test_input_fusion_narrow_rows(host, orc, stream, dtype, cols):
    """The same for the fused chain: rows of less than a segment, by the catalogue's choice, chains from 128 rows on (16-bit
    rows of less than a segment: 256), and by the chains themselves; infinities and NaN stand beside the matrices and a zero under the last logarithm."""
    name, width = "imex_input_fusion_" + dtype, 4 if dtype == "f32" else 2
    line = 256 if width * cols < 32 and width == 2 else 128
    assert host.variant(name, [line - 1, cols]) == name and host.variant(name, [line, cols]) == name + "_tall"
    narrow = lambda t: t if dtype == "f32" else orc.from_float(t, dtype)
    wide = lambda t: (t if dtype == "f32" else orc.to_float(t, dtype)).reshape(-1, cols)
    for rows in (1, 2, 3, 5, 255, 256, 257, 258, 259, 700, 8195):
        a = orc.fill_uniform(rows * cols, dtype, 95, -5.0, 5.0)
        b = orc.fill_uniform(rows * cols, dtype, 96, 0.01, 40.0)
        b[-1:] = narrow(np.zeros(1, np.float32))
        want = narrow(orc.input_fusion_f32(wide(a), wide(b)))
        for shift in (0, 1):
            beside = narrow(np.resize(np.float32([np.nan, -np.inf, -1.0]), 8))
            d_a, d_b = (stream.to_device(np.concatenate([beside[:shift], t, beside])) for t in (a, b))
            fill = np.full(cols + 8, 3, a.dtype)
            for form in ("", "_tall"):
                d_out = stream.to_device(fill)
                stream.launch(name + form, [rows, cols], [host.Ptr(p + shift * width) for p in (d_a, d_b, d_out)] + [rows, cols])
                stream.wait()
                got = stream.from_device(d_out, fill.shape, fill.dtype)
                stream.free(d_out)
                assert np.array_equal(got[shift:shift + cols], want), (name + form, rows, shift)
                assert np.all(got[:shift] == 3) and np.all(got[shift + cols:] == 3), (name + form, rows, shift)
            stream.free(d_a), stream.free(d_b)


@pytest.mark.parametrize("dtype", ["f32", "f16", "bf16"])
def test_input_fusion_half_segments(host, orc, stream, dtype):
    """Segments of 16 bytes, on both sides of the lines in rows and columns: tiles of 512 rows, whole, one row more and one
    fewer; rows that are no whole segments, at any element's address; the elements around the result untouched."""
    width, line = (4, 4096) if dtype == "f32" else (2, 2048)
    least, most, name = 32 // width, 4096 // width, "imex_input_fusion_" + dtype
    wide = lambda t: t if dtype == "f32" else orc.to_float(t, dtype)
    narrow = lambda t: t if dtype == "f32" else orc.from_float(t, dtype)
    for rows in (line - 1, line, line + 1, line + 511):
        for cols in (least - 1, least, least + 1, 5 * least + 3, most, most + 1):
            assert host.variant(name, [rows, cols]) == name + "_tall"
            half = rows >= line and least <= cols <= most
            assert host.launch_shape(name + "_tall", [rows, cols])[0][0] == -(-cols // (16 // width if half else 32 // width))
            say("%s %dx%d" % (name, rows, cols))
            a = orc.fill_uniform(rows * cols, dtype, 97, -5.0, 5.0)
            b = orc.fill_uniform(rows * cols, dtype, 98, 0.01, 40.0)
            want = narrow(orc.input_fusion_f32(wide(a).reshape(rows, cols), wide(b).reshape(rows, cols)))
            beside = narrow(np.full(1, np.nan, np.float32))
            d_a, d_b = (stream.to_device(np.concatenate([beside, t, beside])) for t in (a, b))
            d_out = stream.to_device(np.full(cols + 2, 3, a.dtype))
            stream.launch(name, [rows, cols], [host.Ptr(p + width) for p in (d_a, d_b, d_out)] + [rows, cols])
            stream.wait()
            got = stream.from_device(d_out, (cols + 2,), a.dtype)
            for p in (d_a, d_b, d_out):
                stream.free(p)
            assert np.array_equal(got[1:-1], want) and got[0] == 3 and got[-1] == 3


@pytest.mark.parametrize("dtype", ["f32", "f16", "bf16"])
@pytest.mark.parametrize("rows,segments,extra", [(300, 3, 1), (140, 300, -3), (130, 514, 7), (70, 1030, 5)])
def test_column_chains_in_place(host, orc, stream, dtype, rows, segments, extra):
    """A result that lies in the first or the last row of its own matrix.  On one workgroup the last block of columns, which
    starts inside the one before it, is walked after that one's sums are stored: they must not come back into its own."""
    width = 4 if dtype == "f32" else 2
    cols = segments * (32 // width) + extra
    wide = lambda t: t if dtype == "f32" else orc.to_float(t, dtype)
    narrow = lambda t: t if dtype == "f32" else orc.from_float(t, dtype)
    a = orc.fill_uniform(rows * cols, dtype, 55, -5.0, 5.0).reshape(rows, cols)
    b = orc.fill_uniform(rows * cols, dtype, 56, 0.01, 40.0).reshape(rows, cols)
    d_a, d_b = stream.to_device(a), stream.to_device(b)
    want = {"input_fusion": narrow(orc.input_fusion_f32(wide(a), wide(b))), "reduce_outer": narrow(orc.reduce_outer_f32(wide(a), 0.25))}
    for grid in ((1, 1, 1), None):
        for row in (0, rows - 1):
            out = host.Ptr(d_a + row * cols * width)
            for op, args in (("input_fusion", [d_a, d_b, out, rows, cols]), ("reduce_outer", [d_a, out, rows, cols, 0.25])):
                say("%s %s %dx%d, row %d, grid %s" % (op, dtype, rows, cols, row, grid))
                stream.copy(d_a, a.ctypes.data, a.nbytes)
                stream.launch("imex_%s_%s_tall" % (op, dtype), [rows, cols], args, grid=grid)
                stream.wait()
                got = stream.from_device(d_a, a.shape, a.dtype)
                assert np.array_equal(got[row], want[op]), (op, row, grid)
                assert np.array_equal(np.delete(got, row, 0), np.delete(a, row, 0)), (op, row, grid)
    for p in (d_a, d_b):
        stream.free(p)


# ============================ flash attention ===============================
def attention_close(got_bits, ref_bits, orc):
    """The reference checks its kernel with allclose (atol 1e-4, rtol 1e-3) on a constant
    input.  On random inputs the kernel (P truncated to f16 before normalisation, keys
    in blocks) and the CPU loop (P truncated after normalisation, keys in order) differ
    by f16 roundings of P, each <= 2^-11 relative: |d| <= 2^-10 * max|V| plus one f16
    output rounding."""
    got, ref = orc.half_to_float(got_bits), orc.half_to_float(ref_bits)
    return np.max(np.abs(got - ref)) <= 2.0 ** -10 + 2.0 ** -11 * np.max(np.abs(ref))


@pytest.mark.parametrize("zh,n_ctx", [(1, 128), (3, 256), (2, 1024), (2, 100), (1, 64)])
def test_flash_attention_vs_oracle(host, orc, stream, zh, n_ctx):
    n = zh * n_ctx
    q = orc.fill_uniform(n * 64, "f16", 51, -1, 1).reshape(n, 64)
    k = orc.fill_uniform(n * 64, "f16", 52, -1, 1).reshape(n, 64)
    v = orc.fill_uniform(n * 64, "f16", 53, -1, 1).reshape(n, 64)
    got = host.flash_attention(stream, q, k, v, zh, n_ctx, 0.5)
    rows = np.arange(n) if n <= 512 else np.unique(np.concatenate([np.arange(0, n, 37), [n_ctx - 1, n_ctx, n - 1]]))
    ref = orc.flash_attention_rows(q, k, v, n_ctx, 0.5, rows)
    assert attention_close(got[rows], ref, orc)


def test_flash_attention_sixteen_heads(host, orc, stream):
    """16 x 1024 x 64 with the scale 0.350097656 of the reference's second attention
    test (WG/flash_attention_fwd_ov_with_arrray_len_1k.mlir:22,40; inputs there are
    uniform(-1,1), checked against a natural-exp softmax)."""
    zh, n_ctx, scale = 16, 1024, 0.350097656
    n = zh * n_ctx
    q = orc.fill_uniform(n * 64, "f16", 61, -1, 1).reshape(n, 64)
    k = orc.fill_uniform(n * 64, "f16", 62, -1, 1).reshape(n, 64)
    v = orc.fill_uniform(n * 64, "f16", 63, -1, 1).reshape(n, 64)
    got = host.flash_attention(stream, q, k, v, zh, n_ctx, scale)
    rows = np.unique(np.concatenate([np.arange(0, n, 211), [1023, 1024, n - 1]]))
    assert attention_close(got[rows], orc.flash_attention_rows(q, k, v, n_ctx, scale, rows), orc)


@pytest.mark.parametrize("zh,n_ctx,scale", [(3, 512, 0.5), (2, 256, 4.0), (1, 2048, 0.125)])
def test_flash_attention_every_tiling(host, orc, stream, zh, n_ctx, scale):
    """64, 128 and 256 queries per workgroup (2, 4, 8 query blocks x 4, 2, 1 key groups; ring of
    2, 4, 8 stages) and 256 queries as sixteen wavefronts (8 x 2, ring of 4): each against the
    oracle, on the same inputs."""
    n = zh * n_ctx
    q = orc.fill_uniform(n * 64, "f16", 71, -2, 2).reshape(n, 64)
    k = orc.fill_uniform(n * 64, "f16", 72, -2, 2).reshape(n, 64)
    v = orc.fill_uniform(n * 64, "f16", 73, -1, 1).reshape(n, 64)
    rows = np.unique(np.concatenate([np.arange(0, n, 7), [n_ctx - 1, n - 1]]))
    ref = orc.flash_attention_rows(q, k, v, n_ctx, scale, rows)
    for queries, threads in ((64, 512), (128, 512), (256, 512), (256, 1024)):
        say("attention %dx%d, %d queries per workgroup of %d threads" % (zh, n_ctx, queries, threads))
        got = host.flash_attention(stream, q, k, v, zh, n_ctx, scale, queries_per_workgroup=queries, threads=threads)
        assert attention_close(got[rows], ref, orc), (queries, threads)


@pytest.mark.parametrize("zh,n_ctx,scale", [(2, 100, 0.5), (3, 1000, 0.125), (2, 257, 1.0), (1, 5, 0.5), (5, 333, 2.0),
                                             (1, 193, 0.5), (2, 64, 0.5)])
def test_flash_attention_ragged_context(host, orc, stream, zh, n_ctx, scale):
    """N_CTX that divides none of the tiles: padded queries are not stored, padded keys get a
    score of -inf; key groups that see no key at all (short heads) merge as empty.  Every
    tiling, every row, against the oracle; the rows behind Out stay untouched."""
    n = zh * n_ctx
    q = orc.fill_uniform(n * 64, "f16", 81, -2, 2).reshape(n, 64)
    k = orc.fill_uniform(n * 64, "f16", 82, -2, 2).reshape(n, 64)
    v = orc.fill_uniform(n * 64, "f16", 83, -1, 1).reshape(n, 64)
    rows = np.arange(n) if n <= 1200 else np.unique(np.concatenate([np.arange(0, n, 3), [n_ctx - 1, n_ctx, n - 1]]))
    ref = orc.flash_attention_rows(q, k, v, n_ctx, scale, rows)
    got = host.flash_attention(stream, q, k, v, zh, n_ctx, scale)
    assert attention_close(got[rows], ref, orc), "catalogue launch"
    for queries, threads in ((64, 512), (128, 512), (256, 512), (256, 1024)):
        say("attention %dx%d ragged, %d queries per workgroup of %d threads" % (zh, n_ctx, queries, threads))
        guard = np.full((n + 256, 64), 0x7e01, np.uint16)
        d_q, d_k, d_v, d_o = (stream.to_device(t) for t in (q, k, v, guard))
        grid = (-(-n_ctx // queries), zh, 1)
        stream.launch("imex_flash_attention_fwd_f16", [zh, n_ctx], [d_q, d_k, d_v, d_o, float(scale), zh, n_ctx],
                      grid=grid, block=(threads, 1, 1))
        stream.wait()
        out = stream.from_device(d_o, (n + 256, 64), np.uint16)
        for p in (d_q, d_k, d_v, d_o):
            stream.free(p)
        assert np.all(out[n:] == 0x7e01), (queries, threads, "wrote behind Out")
        assert attention_close(out[rows], ref, orc), (queries, threads)


@pytest.mark.parametrize("queries", [32, 64, 128, 256])
@pytest.mark.parametrize("zh,n_ctx", [(1, 1), (2, 33), (3, 255), (2, 512), (1, 769), (2, 1537)])
def test_flash_attention_one_tiling(host, orc, stream, queries, zh, n_ctx):
    """The kernels with one tiling each: fewer keys than key groups, one more than a tile, one fewer than a block of
    256, whole blocks, several blocks with a ragged last one; every row, and the rows behind Out untouched."""
    n = zh * n_ctx
    q = orc.fill_uniform(n * 64, "f16", 87, -2, 2).reshape(n, 64)
    k = orc.fill_uniform(n * 64, "f16", 88, -2, 2).reshape(n, 64)
    v = orc.fill_uniform(n * 64, "f16", 89, -1, 1).reshape(n, 64)
    rows = np.arange(n) if n <= 1200 else np.unique(np.concatenate([np.arange(0, n, 5), [n_ctx - 1, n_ctx % n, n - 1]]))
    guard = np.full((n + 256, 64), 0x7e01, np.uint16)
    d_q, d_k, d_v, d_o = (stream.to_device(t) for t in (q, k, v, guard))
    say("attention %dx%d, %d queries per workgroup" % (zh, n_ctx, queries))
    stream.launch("imex_flash_attention_fwd_f16_q%d" % queries, [zh, n_ctx], [d_q, d_k, d_v, d_o, 0.5, zh, n_ctx])
    stream.wait()
    out = stream.from_device(d_o, (n + 256, 64), np.uint16)
    for p in (d_q, d_k, d_v, d_o):
        stream.free(p)
    assert np.all(out[n:] == 0x7e01), "wrote behind Out"
    assert attention_close(out[rows], orc.flash_attention_rows(q, k, v, n_ctx, 0.5, rows), orc)


@pytest.mark.parametrize("zh,n_ctx,tiling", [
    (1, 31, "_q32"), (1, 32, "_q32"), (7, 225, "_q32"), (256, 32, "_q32"), (16, 512, "_q32"), (32, 256, "_q32"),  # to 256
    (4, 2048, "_q32"), (1, 3169, "_q32"), (17, 500, ""), (257, 32, ""), (16, 768, "_q64"), (48, 333, "_q128"),
    (100, 333, "_q256"), (2, 8000, "_q64"), (16, 600, "_q64"), (20, 641, "")])
def test_flash_attention_tiling_by_size(host, orc, stream, zh, n_ctx, tiling):
    """The tiling that the catalogue takes on both sides of its lines; wavefronts without a tile, with one that is ragged,
    with several; infinite keys (scores of -inf for whole tiles) and values beside it: the rows behind Out untouched."""
    name = "imex_flash_attention_fwd_f16"
    assert host.variant(name, [zh, n_ctx]) == name + tiling
    n = zh * n_ctx
    q, k, v = (orc.fill_uniform(n * 64, "f16", seed, lo, hi).reshape(n, 64)
               for seed, lo, hi in ((90, 0.25, 2), (91, -2, 2), (92, -1, 1)))
    head = np.arange(n).reshape(zh, n_ctx)[-1]
    k[head[:-1][head[:-1] % 3 != 0], 5] = 0xfc00  # -inf times a positive query
    v[head[0], 9] = 0x7c00
    rows = np.unique(np.concatenate([np.arange(0, n, max(1, n // 200)), head[:40], head[-40:]]))
    guard = np.full((n + 256, 64), 0x7e01, np.uint16)
    d_q, d_k, d_v, d_o = (stream.to_device(t) for t in (q, k, v, guard))
    say("attention %dx%d by size" % (zh, n_ctx))
    stream.launch(name, [zh, n_ctx], [d_q, d_k, d_v, d_o, 0.5, zh, n_ctx])
    stream.wait()
    out = stream.from_device(d_o, (n + 256, 64), np.uint16)
    for p in (d_q, d_k, d_v, d_o):
        stream.free(p)
    assert np.all(out[n:] == 0x7e01), "wrote behind Out"
    got, ref = orc.half_to_float(out[rows]), orc.half_to_float(orc.flash_attention_rows(q, k, v, n_ctx, 0.5, rows))
    ok = np.isfinite(ref)
    assert np.array_equal(np.isfinite(got), ok) and np.all(ok[:, :9]) and np.all(ok[:, 10:])
    assert np.max(np.abs(got[ok] - ref[ok])) <= 2.0 ** -10 + 2.0 ** -11 * np.max(np.abs(ref[ok]))


@pytest.mark.parametrize("queries", [32, 64, 128, 256])
@pytest.mark.parametrize("order", ["up", "down", "jumps"])
@pytest.mark.parametrize("zh,n_ctx", [(1, 769), (3, 1000), (2, 2080)])
def test_flash_attention_moving_maximum(host, orc, stream, zh, n_ctx, order, queries):
    """Scores that grow by less than a factor of 2^8 from tile to tile, so that every tile rescales what the ones before it
    left, that fall, so that none but the first does, and that jump from key to key, in the kernels with one tiling each;
    workgroups that 8 does not divide."""
    n = zh * n_ctx
    q = orc.fill_uniform(n * 64, "f16", 93, -0.5, 0.5).reshape(n, 64)
    k = orc.fill_uniform(n * 64, "f16", 94, -0.5, 0.5).reshape(n, 64)
    v = orc.fill_uniform(n * 64, "f16", 95, -1, 1).reshape(n, 64)
    q[:, 0] = 0x4000  # 2.0
    at = np.arange(n) % n_ctx
    ramp = {"up": at / 64.0, "down": -at / 64.0, "jumps": 40.0 * ((at * 7919) % 13 == 0) - 20.0}[order]
    k[:, 0] = ramp.astype(np.float16).view(np.uint16)
    say("attention %dx%d %s, %d queries per workgroup" % (zh, n_ctx, order, queries))
    d_q, d_k, d_v, d_o = (stream.to_device(t) for t in (q, k, v, np.zeros_like(q)))
    stream.launch("imex_flash_attention_fwd_f16_q%d" % queries, [zh, n_ctx], [d_q, d_k, d_v, d_o, 0.5, zh, n_ctx])
    stream.wait()
    got = stream.from_device(d_o, q.shape, np.uint16)
    for p in (d_q, d_k, d_v, d_o):
        stream.free(p)
    rows = np.unique(np.concatenate([np.arange(0, n, 11), [n_ctx - 1, n - 1]]))
    assert attention_close(got[rows], orc.flash_attention_rows(q, k, v, n_ctx, 0.5, rows), orc)


@pytest.mark.parametrize("queries", [32, 64, 128, 256])
def test_flash_attention_error_against_64_bits(host, orc, stream, queries):
    """P is rounded to f16 against the running maximum, so that the largest weights are 1 and just below it, where f16 is
    finest: 2-norms of the error of 2.4e-4 .. 2.7e-4, of which 2.0e-4 is the result's own rounding.  Against a reference
    that lags the maximum it is 2.9e-4."""
    n = 2048
    q, k, v = (orc.fill_uniform(n * 64, "f16", seed, -1, 1).reshape(n, 64) for seed in (101, 102, 103))
    d_q, d_k, d_v, d_o = (stream.to_device(t) for t in (q, k, v, np.zeros_like(q)))
    stream.launch("imex_flash_attention_fwd_f16_q%d" % queries, [1, n], [d_q, d_k, d_v, d_o, 0.5, 1, n])
    stream.wait()
    got = orc.half_to_float(stream.from_device(d_o, q.shape, np.uint16)).astype(np.float64)
    for p in (d_q, d_k, d_v, d_o):
        stream.free(p)
    q, k, v = (orc.half_to_float(t).astype(np.float64) for t in (q, k, v))
    s = 0.5 * (q @ k.T)
    p = np.exp(s - s.max(1, keepdims=True))
    want = p @ v / p.sum(1, keepdims=True)
    assert np.linalg.norm(got - want) <= 2.75e-4 * np.linalg.norm(want)


@pytest.mark.parametrize("queries", [32, 64, 128, 256])
def test_flash_attention_one_tiling_at_any_address(host, orc, stream, queries):
    """A tensor that starts one element behind a 16-byte boundary takes the reference loop of the same kernel."""
    zh, n_ctx = 2, 130
    n = zh * n_ctx
    q, k, v = (orc.fill_uniform(n * 64, "f16", seed, -1, 1).reshape(n, 64) for seed in (87, 88, 89))
    want = orc.flash_attention_rows(q, k, v, n_ctx, 0.5, np.arange(n))
    for which in range(4):
        say("attention, %d queries per workgroup, tensor %d off the 16-byte grid" % (queries, which))
        host_bufs = [q.ravel(), k.ravel(), v.ravel(), np.full(n * 64, 0x7e01, np.uint16)]
        host_bufs = [np.concatenate([np.zeros(int(i == which), np.uint16), t]) for i, t in enumerate(host_bufs)]
        bufs = [stream.to_device(t) for t in host_bufs]
        stream.launch("imex_flash_attention_fwd_f16_q%d" % queries, [zh, n_ctx],
                      [host.Ptr(p + 2 * (i == which)) for i, p in enumerate(bufs)] + [0.5, zh, n_ctx])
        stream.wait()
        out = stream.from_device(bufs[3], host_bufs[3].shape, np.uint16)[int(which == 3):].reshape(n, 64)
        for p in bufs:
            stream.free(p)
        assert attention_close(out, want, orc)


def test_flash_attention_negative_scale_takes_the_reference_loop(host, orc, stream):
    """The tiled path takes the row maximum before scaling, which needs a positive scale; any
    other scale runs the one-lane-per-query loop of the same kernel."""
    zh, n_ctx = 2, 256
    n = zh * n_ctx
    q = orc.fill_uniform(n * 64, "f16", 84, -1, 1).reshape(n, 64)
    k = orc.fill_uniform(n * 64, "f16", 85, -1, 1).reshape(n, 64)
    v = orc.fill_uniform(n * 64, "f16", 86, -1, 1).reshape(n, 64)
    rows = np.arange(0, n, 3)
    got = host.flash_attention(stream, q, k, v, zh, n_ctx, -0.5)
    assert attention_close(got[rows], orc.flash_attention_rows(q, k, v, n_ctx, -0.5, rows), orc)


@pytest.mark.parametrize("zh", [8, 16])
def test_flash_attention_catalogue_picks_wide_tilings(host, orc, stream, zh):
    """N_CTX = 4096 with 8 and 16 heads: the catalogue launches 128- and 256-query workgroups
    (16 heads is the reference's flash_attention_fwd_ov_with_arrray_len_4k.mlir shape)."""
    n_ctx = 4096
    grid, block, _ = host.launch_shape("imex_flash_attention_fwd_f16", [zh, n_ctx])
    assert grid == (n_ctx // (16 * zh), zh, 1) and block == ((1024 if zh == 16 else 512), 1, 1)
    n = zh * n_ctx
    q = orc.fill_uniform(n * 64, "f16", 74, -1, 1).reshape(n, 64)
    k = orc.fill_uniform(n * 64, "f16", 75, -1, 1).reshape(n, 64)
    v = orc.fill_uniform(n * 64, "f16", 76, -1, 1).reshape(n, 64)
    got = host.flash_attention(stream, q, k, v, zh, n_ctx, 0.5)
    rows = np.unique(np.concatenate([np.arange(0, n, 2999), [255, 256, n_ctx - 1, n_ctx, n - 1]]))
    assert attention_close(got[rows], orc.flash_attention_rows(q, k, v, n_ctx, 0.5, rows), orc)


def test_flash_attention_sharp_scores(host, orc, stream):
    """Large score range (scale 4, |q.k| up to ~20): the running max changes from block
    to block and the rescaling of the accumulator is exercised."""
    zh, n_ctx = 2, 512
    n = zh * n_ctx
    q = orc.fill_uniform(n * 64, "f16", 54, -2, 2).reshape(n, 64)
    k = orc.fill_uniform(n * 64, "f16", 55, -2, 2).reshape(n, 64)
    v = orc.fill_uniform(n * 64, "f16", 56, -1, 1).reshape(n, 64)
    got = host.flash_attention(stream, q, k, v, zh, n_ctx, 4.0)
    rows = np.arange(0, n, 5)
    assert attention_close(got[rows], orc.flash_attention_rows(q, k, v, n_ctx, 4.0, rows), orc)


def test_flash_attention_reference_config(host, orc, stream):
    """Z = 2, H = 2, N_CTX = 4096, D = 64, scale 0.5 (flash_attention_fwd.mlir:449-454):
    the reference's own constant input exactly, then random inputs on sampled rows."""
    zh, n_ctx = 4, 4096
    n = zh * n_ctx
    const = orc.from_float(np.full((n, 64), 0.625, np.float32), "f16")
    out = host.flash_attention(stream, const, const, const, zh, n_ctx, 0.5)
    assert np.all(orc.half_to_float(out) == 0.625)
    q = orc.fill_uniform(n * 64, "f16", 57, -1, 1).reshape(n, 64)
    k = orc.fill_uniform(n * 64, "f16", 58, -1, 1).reshape(n, 64)
    v = orc.fill_uniform(n * 64, "f16", 59, -1, 1).reshape(n, 64)
    got = host.flash_attention(stream, q, k, v, zh, n_ctx, 0.5)
    rows = np.array([0, 1, 63, 64, 4095, 4096, 5000, 8191, 8192, 12287, 12288, 16383])
    ref = orc.flash_attention_rows(q, k, v, n_ctx, 0.5, rows)
    assert attention_close(got[rows], ref, orc)
    # permuting the keys (and values with them) of one head leaves its outputs unchanged up to rounding
    perm = np.random.default_rng(3).permutation(n_ctx)
    k2, v2 = k.copy(), v.copy()
    k2[:n_ctx], v2[:n_ctx] = k[:n_ctx][perm], v[:n_ctx][perm]
    got2 = host.flash_attention(stream, q, k2, v2, zh, n_ctx, 0.5)
    assert attention_close(got2[:n_ctx], got[:n_ctx], orc)
    assert np.array_equal(got2[n_ctx:], got[n_ctx:])


# =============================== GEMM ======================================
def gemm_close(got, ref):
    return np.max(np.abs(got - ref)) <= 5e-3 * np.max(np.abs(ref))


def test_gemm_golden_3x3(host, orc, stream):
    g = GOLD["gemm_f16_acc_f32_3x3"]
    a, b = orc.float_to_half(arr(g["A"], [3, 3])), orc.float_to_half(arr(g["B"], [3, 3]))
    c = host.gemm(stream, a, b, c=arr(g["C0"], [3, 3]), ab_dtype="f16")
    assert orc.allclose_f32(c, arr(g["expected"], [3, 3]))
    assert np.array_equal(c, orc.gemm(a, b, "f16", c=arr(g["C0"], [3, 3])))  # scalar path: same order, bit-exact
    g = GOLD["gemm_bf16_acc_f32_3x3"]
    a, b = orc.float_to_bfloat(arr(g["A"], [3, 3])), orc.float_to_bfloat(arr(g["B"], [3, 3]))
    c = host.gemm(stream, a, b, c=arr(g["C0"], [3, 3]), ab_dtype="bf16")
    assert np.max(np.abs(c.ravel() - arr(g["expected"]))) < 6e-5
    g = GOLD["dot_f16_acc_f32_8x16x32"]
    a = orc.float_to_half(np.full((8, 16), 1.0, np.float32))
    b = orc.float_to_half(np.full((16, 32), 2.0, np.float32))
    out = host.gemm(stream, a, b, ab_dtype="f16", out_dtype="f16")
    assert np.all(orc.half_to_float(out) == g["expected_fill"])


@pytest.mark.parametrize("M,N,K", [(5, 7, 9), (100, 36, 130), (256, 256, 20), (256, 256, 44), (255, 252, 64), (17, 300, 64),
                                   (300, 260, 50), (129, 129, 17)])
@pytest.mark.parametrize("dtype", ["f16", "bf16"])
def test_gemm_untileable_shapes_bit_exact(host, orc, stream, M, N, K, dtype):
    """K not a multiple of 8 or N not a multiple of 8: the vector-ALU path (128 x 128 tiles, sixteen k at a
    time), which accumulates every output in the oracle's order."""
    a = orc.fill_uniform(M * K, dtype, 1, -1, 1).reshape(M, K)
    b = orc.fill_uniform(K * N, dtype, 2, -1, 1).reshape(K, N)
    assert np.array_equal(host.gemm(stream, a, b, ab_dtype=dtype), orc.gemm(a, b, dtype))


def test_gemm_untileable_special_values(host, orc, stream):
    """The vector-ALU path pads its tiles with zeros beyond M, N and K; infinities, NaNs and negative zeros
    in the operands must come out as in the sequential loop, which never sees the padding."""
    M, N, K = 70, 37, 21
    a = orc.fill_uniform(M * K, "f16", 3, -1, 1).reshape(M, K)
    b = orc.fill_uniform(K * N, "f16", 4, -1, 1).reshape(K, N)
    a[3, 5], a[9, 20], a[60, 0], a[69, 20] = 0x7c00, 0xfc00, 0x7e00, 0x7c00      # +inf, -inf, NaN, +inf
    b[20, 36], b[0, 0] = 0x7c00, 0xfc00
    a[11, :] = 0x8000                                                         # a row of -0.0
    got, want = host.gemm(stream, a, b, ab_dtype="f16"), orc.gemm(a, b, "f16")
    assert np.array_equal(np.isnan(got), np.isnan(want))
    ok = ~np.isnan(want)
    assert np.array_equal(got.view(np.uint32)[ok], want.view(np.uint32)[ok])


@pytest.mark.parametrize("dtype", ["f16", "bf16"])
def test_gemm_tiled_identity_and_layout(host, orc, stream, dtype):
    """B = I gives C = A exactly; A[i,j] = j patterns expose any fragment-layout mistake."""
    M, N, K = 512, 512, 512
    a = orc.fill_uniform(M * K, dtype, 3, -1, 1).reshape(M, K)
    eye = orc.from_float(np.eye(K, dtype=np.float32), dtype)
    assert np.array_equal(host.gemm(stream, a, eye, ab_dtype=dtype), orc.to_float(a, dtype))
    # A = I: C = B exactly (exercises the B transpose-in-registers path)
    b = orc.fill_uniform(K * N, dtype, 4, -1, 1).reshape(K, N)
    assert np.array_equal(host.gemm(stream, eye, b, ab_dtype=dtype), orc.to_float(b, dtype))
    # a single non-zero k picks out one row of B scaled by a column of A
    a1 = np.zeros((M, K), np.float32)
    a1[:, 77] = np.arange(M) % 16
    got = host.gemm(stream, orc.from_float(a1, dtype), b, ab_dtype=dtype)
    assert np.array_equal(got, np.outer(a1[:, 77], orc.to_float(b, dtype)[77]).astype(np.float32))


@pytest.mark.parametrize("dtype,M,N,K", [("f16", 512, 768, 4096), ("bf16", 256, 1024, 1024), ("f16", 1024, 256, 64),
                                           ("f16", 256, 256, 32), ("bf16", 512, 256, 96), ("f16", 256, 512, 160)])
def test_gemm_tiled_small_integers_exact(host, orc, stream, dtype, M, N, K):
    """|a|,|b| <= 4: every partial sum is an integer below 2^24, so any
    accumulation order gives the same f32 bits as the integer product."""
    a = orc.fill_int(M * K, dtype, 5, -4, 4).reshape(M, K)
    b = orc.fill_int(K * N, dtype, 6, -4, 4).reshape(K, N)
    want = orc.to_float(a, dtype).astype(np.int64) @ orc.to_float(b, dtype).astype(np.int64)
    got = host.gemm(stream, a, b, ab_dtype=dtype)
    assert np.array_equal(got.astype(np.int64), want)


@pytest.mark.parametrize("which", ["plain", "ta", "tb", "acc", "mlp"])
@pytest.mark.parametrize("M,N,K", [(256, 256, 8), (256, 256, 16), (256, 256, 48), (300, 520, 40), (512, 256, 4096 + 24),
                                   (64, 72, 104), (1000, 264, 72)])
def test_gemm_partial_last_k_step(host, orc, stream, which, M, N, K):
    """K a multiple of 8 but not of the 32-wide step: the MFMA path pads the last step with zeros on the
    way into LDS.  Integer operands give the exact product in any order, so any stale or foreign value
    that got multiplied in would show; every operand layout and an epilogue with its own loads."""
    say("gemm partial K step %s %dx%dx%d" % (which, M, N, K))
    if which == "ta" and M % 8:
        M = (M + 7) // 8 * 8
    dtype = "bf16" if which == "mlp" else "f16"
    a = orc.fill_int(M * K, dtype, 91, -4, 4).reshape(M, K)
    b = orc.fill_int(K * N, dtype, 92, -4, 4).reshape(K, N)
    want = orc.to_float(a, dtype).astype(np.int64) @ orc.to_float(b, dtype).astype(np.int64)
    if which == "plain":
        got = _gemm_guarded(host, stream, "imex_gemm_f16_f16_f32", a, b, M, N, K)
    elif which == "ta":
        got = _gemm_guarded(host, stream, "imex_gemm_f16_f16_f32_ta", np.ascontiguousarray(a.T), b, M, N, K)
    elif which == "tb":
        got = _gemm_guarded(host, stream, "imex_gemm_f16_f16_f32_tb", a, np.ascontiguousarray(b.T), M, N, K)
    elif which == "acc":
        c0 = orc.fill_int(M * N, "f32", 93, -1000, 1000).reshape(M, N)
        got = host.gemm(stream, a, b, c=c0, ab_dtype="f16")
        want = want + c0.astype(np.int64)
    else:
        bias = orc.fill_int(N, "f32", 94, -3, 3)
        out = _gemm_guarded(host, stream, "imex_gemm_bf16_bias_silu_bf16", a, b, M, N, K, extra=(bias,), out_np=np.uint16)
        ref = orc.bfloat_to_float(orc.bias_silu_bf16(want.astype(np.float32), bias))
        assert np.max(np.abs(orc.bfloat_to_float(out) - ref)) <= 2.0 ** -7 * np.max(np.abs(ref)) + 1e-6
        return
    assert np.array_equal(got.astype(np.int64), want)


@pytest.mark.parametrize("dtype,M,N,K", [("f16", 256, 256, 32), ("bf16", 256, 512, 96), ("f16", 512, 256, 224)])
def test_gemm_tiled_short_k_random(host, orc, stream, dtype, M, N, K):
    """K shorter than the copy pipeline is deep (1, 3 and 7 steps of 32): the
    prologue and the clamped tail copies must not disturb the result."""
    a = orc.fill_uniform(M * K, dtype, 11, -1, 1).reshape(M, K)
    b = orc.fill_uniform(K * N, dtype, 12, -1, 1).reshape(K, N)
    assert gemm_close(host.gemm(stream, a, b, ab_dtype=dtype), orc.gemm(a, b, dtype))


def _gemm_guarded(host, stream, name, sa, sb, M, N, K, extra=(), out_np=np.float32):
    """Launch a GEMM kernel on an output buffer with 256 guard rows behind it; returns the
    [M,N] result after checking that the guard rows kept their fill."""
    guard = 256
    fill = np.full((M + guard, N), 0x7fc1 if out_np == np.uint16 else np.float32(-12345.5), out_np)
    d_a, d_b, d_c = stream.to_device(sa), stream.to_device(sb), stream.to_device(fill)
    extras = [stream.to_device(e) for e in extra]
    try:
        stream.launch(name, [M, N, K], [d_a, d_b] + extras + [d_c, M, N, K])
        stream.wait()
        out = stream.from_device(d_c, (M + guard, N), out_np)
    finally:
        for p in [d_a, d_b, d_c] + extras:
            stream.free(p)
    assert np.array_equal(out[M:], fill[M:]), "%s wrote past row %d" % (name, M)
    return out[:M]


@pytest.mark.parametrize("M,N,K", [(255, 256, 64), (1, 8, 32), (300, 520, 96), (257, 264, 1024), (4000, 1000, 128),
                                   (31, 4104, 64)])
def test_gemm_ragged_tiles(host, orc, stream, M, N, K):
    """M and N that do not divide the 256 x 256 tile (K % 32 == 0, N % 8 == 0): the MFMA path with
    edge tiles.  Integer operands give the exact product in any order; random ones the 5e-3 bar;
    nothing is stored outside C."""
    say("gemm ragged %dx%dx%d" % (M, N, K))
    a = orc.fill_int(M * K, "f16", 5, -4, 4).reshape(M, K)
    b = orc.fill_int(K * N, "f16", 6, -4, 4).reshape(K, N)
    want = orc.to_float(a, "f16").astype(np.int64) @ orc.to_float(b, "f16").astype(np.int64)
    got = _gemm_guarded(host, stream, "imex_gemm_f16_f16_f32", a, b, M, N, K)
    assert np.array_equal(got.astype(np.int64), want)
    a = orc.fill_uniform(M * K, "bf16", 13, -1, 1).reshape(M, K)
    b = orc.fill_uniform(K * N, "bf16", 14, -1, 1).reshape(K, N)
    rows = np.unique(np.concatenate([np.arange(0, M, 61), [M - 1]]))
    got = _gemm_guarded(host, stream, "imex_gemm_bf16_bf16_f32", a, b, M, N, K)
    assert gemm_close(got[rows], orc.gemm_rows(a, b, rows, "bf16"))
    # fused bias + SiLU epilogue and the f16-output one on the same ragged shape
    bias = orc.fill_normal(N, "f32", 15, 0.0, 0.1)
    fused = _gemm_guarded(host, stream, "imex_gemm_bf16_bias_silu_bf16", a, b, M, N, K, extra=(bias,), out_np=np.uint16)
    ref = orc.bfloat_to_float(orc.bias_silu_bf16(orc.gemm_rows(a, b, rows, "bf16"), bias))
    assert np.max(np.abs(orc.bfloat_to_float(fused)[rows] - ref)) <= 5e-3 * np.max(np.abs(ref)) + 2.0 ** -9


@pytest.mark.parametrize("tile", ["", "_t256x128", "_t128", "_t128x64", "_t128x64s", "_t64", "_t32", "_t16", "_t16x32", "_t16x16"])
@pytest.mark.parametrize("M,N,K", [(1, 8, 8), (64, 64, 256), (127, 136, 72), (129, 264, 520), (520, 72, 1032)])
def test_gemm_every_tile_integers_exact(host, orc, stream, tile, M, N, K):
    """Each tile size (\"\": 256 x 256) on shapes below, at and beyond its edges in M, N and K, for every operand
    layout and epilogue.  Integer operands give the exact f32 sum in any order; results rounded to a 16-bit type
    are that sum's rounding (f16; |sum| < 2048 with K <= 1032 and |a b| <= 1) or within the bias + SiLU bar."""
    say("gemm tile %s %dx%dx%d" % (tile or "_t256", M, N, K))
    Mt = (M + 7) // 8 * 8
    for which in ("plain", "acc", "ta", "tb", "f16", "mlp"):
        m, dtype = (Mt if which == "ta" else M), "bf16" if which in ("mlp", "acc") else "f16"
        a = orc.fill_int(m * K, dtype, 95, -1, 1).reshape(m, K)
        b = orc.fill_int(K * N, dtype, 96, -1, 1).reshape(K, N)
        want = orc.to_float(a, dtype).astype(np.int64) @ orc.to_float(b, dtype).astype(np.int64)
        name = {"plain": "f16_f16_f32", "acc": "bf16_bf16_f32_acc", "ta": "f16_f16_f32_ta", "tb": "f16_f16_f32_tb",
                "f16": "f16_f16_f16", "mlp": "bf16_bias_silu_bf16"}[which]
        name = "imex_gemm_" + name + tile
        bias = orc.fill_int(N, "f32", 97, -3, 3)
        c0 = np.full((m + 256, N), 7, np.uint16 if which in ("f16", "mlp") else np.float32)
        bufs = [stream.to_device(np.ascontiguousarray(a.T) if which == "ta" else a),
                stream.to_device(np.ascontiguousarray(b.T) if which == "tb" else b)]
        bufs += [stream.to_device(bias)] if which == "mlp" else []
        bufs.append(stream.to_device(c0))
        stream.launch(name, [m, N, K], bufs + [m, N, K], grid=host.launch_shape(name, [m, N, K])[0])
        stream.wait()
        got = stream.from_device(bufs[-1], c0.shape, c0.dtype)
        for p in bufs:
            stream.free(p)
        assert np.array_equal(got[m:], c0[m:]), "%s wrote past row %d" % (name, m)
        if which == "mlp":
            ref = orc.bfloat_to_float(orc.bias_silu_bf16(want.astype(np.float32), bias))
            assert np.max(np.abs(orc.bfloat_to_float(got[:m]) - ref)) <= 2.0 ** -7 * np.max(np.abs(ref)) + 1e-6
        elif which == "f16":
            assert np.array_equal(orc.half_to_float(got[:m]).astype(np.int64), want), name
        else:
            assert np.array_equal(got[:m].astype(np.int64), want + (7 if which == "acc" else 0)), name


@pytest.mark.parametrize("tile", ["_u128", "_u64"])
@pytest.mark.parametrize("M,N,K", [(8, 8, 8), (9, 11, 13), (64, 64, 64), (63, 65, 71), (129, 67, 257), (130, 255, 65),
                                   (201, 129, 579)])
def test_gemm_unaligned_rows(host, orc, stream, tile, M, N, K):
    """Rows that are not 16-byte aligned on the matrix cores: shapes below, at and beyond the tiles' edges in M, N and
    K, every operand layout and epilogue.  Integer operands give the exact f32 sum in any order; an infinity in the
    row (k row) that follows reaches nothing but its own results, as it would if a piece beyond K were multiplied by
    something; nothing is stored outside C."""
    say("gemm unaligned %s %dx%dx%d" % (tile, M, N, K))
    for which in ("plain", "acc", "ta", "tb", "f16", "mlp"):
        dtype = "bf16" if which in ("mlp", "acc") else "f16"
        a = orc.fill_int(M * K, dtype, 95, -1, 1).reshape(M, K)
        b = orc.fill_int(K * N, dtype, 96, -1, 1).reshape(K, N)
        a[M - 1, 0] = b[0, N - 1] = 0x7f80 if dtype == "bf16" else 0x7c00
        fa, fb = orc.to_float(a, dtype).astype(np.float64), orc.to_float(b, dtype).astype(np.float64)
        with np.errstate(invalid="ignore"):
            want = fa[:-1, :] @ fb[:, :-1]
        name = {"plain": "f16_f16_f32", "acc": "bf16_bf16_f32_acc", "ta": "f16_f16_f32_ta", "tb": "f16_f16_f32_tb",
                "f16": "f16_f16_f16", "mlp": "bf16_bias_silu_bf16"}[which]
        name = "imex_gemm_" + name + tile
        bias = orc.fill_int(N, "f32", 97, -3, 3)
        c0 = np.full((M + 256, N), 7, np.uint16 if which in ("f16", "mlp") else np.float32)
        bufs = [stream.to_device(np.ascontiguousarray(a.T) if which == "ta" else a),
                stream.to_device(np.ascontiguousarray(b.T) if which == "tb" else b)]
        bufs += [stream.to_device(bias)] if which == "mlp" else []
        bufs.append(stream.to_device(c0))
        stream.launch(name, [M, N, K], bufs + [M, N, K])
        stream.wait()
        got = stream.from_device(bufs[-1], c0.shape, c0.dtype)
        for p in bufs:
            stream.free(p)
        assert np.array_equal(got[M:], c0[M:]), "%s wrote past row %d" % (name, M)
        got = got[:M - 1, :N - 1]
        if which == "mlp":
            ref = orc.bfloat_to_float(orc.bias_silu_bf16(np.ascontiguousarray(want, np.float32), bias[:-1]))
            assert np.max(np.abs(orc.bfloat_to_float(got) - ref)) <= 2.0 ** -7 * np.max(np.abs(ref)) + 1e-6
        elif which == "f16":
            assert np.array_equal(orc.half_to_float(np.ascontiguousarray(got)), want), name
        else:
            assert np.array_equal(got, want + (7 if which == "acc" else 0)), name


@pytest.mark.parametrize("tile,M,N,K", [("_u64", 67, 131, 257), ("_u64", 65, 71, 128), ("_u128", 135, 257, 193), ("_u128", 9, 13, 64)])
def test_gemm_unaligned_last_pieces(host, orc, stream, tile, M, N, K):
    """A strided operand's pieces at the end of a row run into the next one: infinities at the front of every row reach the
    results of those columns (rows, for A stored [K,M]) only.  Integer operands, exact sums."""
    inf = 0x7c00
    for which in ("plain", "ta"):
        a = orc.fill_int(M * K, "f16", 95, -1, 1).reshape(M, K)
        b = orc.fill_int(K * N, "f16", 96, -1, 1).reshape(K, N)
        b[:, :7] = inf
        if which == "ta":
            a[:7] = inf
        fa, fb = orc.to_float(a, "f16").astype(np.float64), orc.to_float(b, "f16").astype(np.float64)
        first = 7 if which == "ta" else 0
        name = "imex_gemm_f16_f16_f32" + ("_ta" if which == "ta" else "") + tile
        got = _gemm_guarded(host, stream, name, np.ascontiguousarray(a.T) if which == "ta" else a, b, M, N, K)
        assert np.array_equal(got[first:, 7:], fa[first:] @ fb[:, 7:]), name


@pytest.mark.parametrize("tile,M,N,K", [("_t128", 260, 392, 136), ("_t128x64", 260, 200, 136), ("_t64", 136, 200, 264),
                                        ("_t32", 104, 136, 264), ("_t16", 40, 200, 520), ("_u128", 259, 391, 135),
                                        ("_t256x128", 520, 264, 136), ("_t16x32", 40, 104, 520), ("_t16x16", 24, 56, 776),
                                        ("_u64", 135, 199, 263)])
def test_gemm_tiles_walk_and_any_address(host, orc, stream, tile, M, N, K):
    """The kernels with one tile size on two workgroups that walk all tiles (their LDS and their partial tiles are used
    again), and with each operand's and the result's base one element behind a 16-byte boundary (the aligned forms take
    their vector-ALU loop there).  Integer operands give the exact f32 sum in any order."""
    for which in ("plain", "acc", "ta", "tb"):
        name = "imex_gemm_" + {"plain": "f16_f16_f32", "acc": "f16_f16_f32_acc", "ta": "f16_f16_f32_ta", "tb": "f16_f16_f32_tb"}[which] + tile
        m = (M + 7) // 8 * 8 if which == "ta" and tile[1] == "t" else M
        a, b = orc.fill_int(m * K, "f16", 95, -3, 3).reshape(m, K), orc.fill_int(K * N, "f16", 96, -3, 3).reshape(K, N)
        want = orc.half_to_float(a).astype(np.int64) @ orc.half_to_float(b).astype(np.int64) + (7 if which == "acc" else 0)
        ins = [(a.T if which == "ta" else a).ravel(), (b.T if which == "tb" else b).ravel(), np.full(m * N, 7, np.float32)]
        full = host.launch_shape(name, [m, N, K])[0]
        for shifted, grid in ((None, (2, 1, 1)), (0, full), (1, full), (2, full)):
            say("%s %dx%dx%d grid %s, buffer %s off the 16-byte grid" % (name, m, N, K, grid, shifted))
            padded = [np.concatenate([np.zeros(int(i == shifted), t.dtype), t, np.full(64, 9, t.dtype)]) for i, t in enumerate(ins)]
            bufs = [stream.to_device(t) for t in padded]
            stream.launch(name, [m, N, K], [host.Ptr(p + t.itemsize * (i == shifted)) for i, (p, t) in enumerate(zip(bufs, ins))] + [m, N, K],
                          grid=grid)
            stream.wait()
            got = stream.from_device(bufs[2], padded[2].shape, np.float32)[int(shifted == 2):]
            for p in bufs:
                stream.free(p)
            assert np.array_equal(got[:m * N].reshape(m, N).astype(np.int64), want), (name, shifted, grid)
            assert np.all(got[m * N:] == 9), (name, shifted, grid)


@pytest.mark.parametrize("tile", ["_u32", "_u16x32", "_u16x16"])
@pytest.mark.parametrize("M,N,K", [(8, 8, 8), (9, 11, 13), (16, 32, 256), (15, 17, 255), (33, 65, 129), (17, 31, 257), (65, 129, 600)])
def test_gemm_unaligned_narrow_tiles(host, orc, stream, tile, M, N, K):
    """The same for the narrow tiles, around their sizes and their steps of 128 and 256 k, and walked by two workgroups."""
    test_gemm_unaligned_rows(host, orc, stream, tile, M, N, K)
    test_gemm_unaligned_last_pieces(host, orc, stream, tile, M, N, K)
    if K > 256:
        test_gemm_tiles_walk_and_any_address(host, orc, stream, tile, M, N, K)


@pytest.mark.parametrize("tile", ["_t128x64", "_t128x64s", "_t64", "_t32", "_t16", "_t16x32", "_t16x16"])
@pytest.mark.parametrize("M,N,K", [(40, 232, 4104), (8, 2120, 1416), (1000, 24, 2568), (264, 72, 3592), (336, 96, 2568)])
def test_gemm_workgroups_that_fetch(host, orc, stream, tile, M, N, K):
    """Launches with workgroups that have no tile and fetch what the others read: one and several bands of tile rows for an
    XCD, bands that it shares with the next, tiles that eight does not divide, ragged edges.  Integer operands, exact sums;
    bias and SiLU of such a sum within the rounding of the 16-bit result."""
    for which in ("plain", "acc", "ta", "tb", "f16", "silu"):
        kind = {"plain": "bf16_bf16_f32", "acc": "f16_f16_f32_acc", "ta": "f16_f16_f32_ta", "tb": "f16_f16_f32_tb",
                "f16": "f16_f16_f16", "silu": "bf16_bias_silu_bf16"}[which]
        name, dtype = "imex_gemm_" + kind + tile, "bf16" if which in ("plain", "silu") else "f16"
        n = N - 3 if which == "tb" else N
        assert host.launch_shape(name, [M, n, K])[0][0] == 256
        a, b = orc.fill_int(M * K, dtype, 95, -1, 1).reshape(M, K), orc.fill_int(K * n, dtype, 96, -1, 1).reshape(K, n)
        want = (orc.to_float(a, dtype) @ orc.to_float(b, dtype)).astype(np.int64) + (7 if which == "acc" else 0)
        fill = np.full((M + 4, n), 7, np.uint16 if which in ("f16", "silu") else np.float32)
        bufs = [stream.to_device(np.ascontiguousarray(a.T) if which == "ta" else a),
                stream.to_device(np.ascontiguousarray(b.T) if which == "tb" else b), stream.to_device(fill)]
        if which == "silu":
            bias = np.arange(n, dtype=np.float32) % 9 - 4
            bufs.insert(2, stream.to_device(bias))
            x = want + bias.astype(np.float64)
            want = x / (1 + np.exp(-x))
        for grid in (None, (256, 1, 1), (331, 1, 1)):
            stream.copy(bufs[-1], fill.ctypes.data, fill.nbytes)
            stream.launch(name, [M, n, K], bufs + [M, n, K], grid=grid or host.launch_shape(name, [M, n, K])[0])
            stream.wait()
            got = stream.from_device(bufs[-1], fill.shape, fill.dtype)
            if which == "silu":  # half an ulp of the result, and what the f32 exponential and quotient lose
                assert np.all(np.abs(orc.to_float(got[:M], dtype) - want) <= 2.0 ** -8 * np.abs(want) + 1e-30), (name, grid)
            else:
                sums = orc.half_to_float(got[:M]) if which == "f16" else got[:M]
                assert np.array_equal(sums.astype(np.int64), want), (name, grid)
            assert np.array_equal(got[M:], fill[M:]), (name, grid)
        for p in bufs:
            stream.free(p)


@pytest.mark.parametrize("which", ["", "_ta", "_tb"])
def test_gemm_unaligned_rows_chosen(host, orc, stream, which):
    """What the operator takes at an ordinary odd size, random operands: against 64 bits within the rounding of 32-bit
    sums, (K + 1) half-ulps of the sum of magnitudes in any order."""
    M, N, K = 301, 517, 259
    name = "imex_gemm_f16_f16_f32" + which
    assert host.variant(name, [M, N, K]) != name
    a = orc.fill_uniform(M * K, "f16", 98, -1, 1).reshape(M, K)
    b = orc.fill_uniform(K * N, "f16", 99, -1, 1).reshape(K, N)
    fa, fb = orc.to_float(a, "f16").astype(np.float64), orc.to_float(b, "f16").astype(np.float64)
    sa, sb = (np.ascontiguousarray(a.T) if which == "_ta" else a), (np.ascontiguousarray(b.T) if which == "_tb" else b)
    got = _gemm_guarded(host, stream, name, sa, sb, M, N, K)
    assert np.all(np.abs(got - fa @ fb) <= (K + 1) * 2.0 ** -24 * (np.abs(fa) @ np.abs(fb)))


@pytest.mark.parametrize("which,M,N,K", [("ta", 248, 264, 64), ("ta", 8, 8, 32), ("tb", 100, 37, 64), ("tb", 300, 515, 96)])
def test_gemm_ragged_tiles_transposed_operands(host, orc, stream, which, M, N, K):
    """Edge tiles with A stored [K,M] (M % 8 == 0) or B stored [N,K] (any N)."""
    a = orc.fill_int(M * K, "f16", 33, -4, 4).reshape(M, K)
    b = orc.fill_int(K * N, "f16", 34, -4, 4).reshape(K, N)
    sa, sb = (np.ascontiguousarray(a.T), b) if which == "ta" else (a, np.ascontiguousarray(b.T))
    want = orc.to_float(a, "f16").astype(np.int64) @ orc.to_float(b, "f16").astype(np.int64)
    got = _gemm_guarded(host, stream, "imex_gemm_f16_f16_f32_" + which, sa, sb, M, N, K)
    assert np.array_equal(got.astype(np.int64), want)


def test_gemm_launch_shape_slack(host, orc, stream):
    """A grid with more or fewer workgroups than tiles (MFMA path: the workgroups stride
    over the tiles) or fewer workgroups than tiles (vector-ALU path) still
    computes every element once."""
    import ctypes as C
    for (M, N, K, grid) in [(256, 256, 64, 9), (100, 36, 130, 2), (1024, 768, 96, 5), (1000, 520, 64, 1)]:
        a = orc.fill_uniform(M * K, "f16", 21, -1, 1).reshape(M, K)
        b = orc.fill_uniform(K * N, "f16", 22, -1, 1).reshape(K, N)
        d_a, d_b, d_c = stream.to_device(a), stream.to_device(b), stream.alloc(M * N * 4)
        fn = stream.kernel("imex_gemm_f16_f16_f32")
        descs, keep = host._pack_params([d_a, d_b, d_c, M, N, K])
        stream.rt.gpuLaunchKernel(stream.handle, fn, grid, 1, 1, 512, 1, 1, 0, C.cast(descs, C.c_void_p), None)
        stream.wait()
        got = stream.from_device(d_c, (M, N), np.float32)
        assert gemm_close(got, orc.gemm(a, b, "f16"))
        for p in (d_a, d_b, d_c):
            stream.free(p)


def test_gemm_config_f16_4096(host, orc, stream):
    M = N = K = 4096
    a = orc.fill_uniform(M * K, "f16", 20246, -1, 1).reshape(M, K)
    b = orc.fill_uniform(K * N, "f16", 20247, -1, 1).reshape(K, N)
    got = host.gemm(stream, a, b, ab_dtype="f16")
    rows = np.array(sorted(set(list(range(0, 4096, 97)) + [1, 255, 256, 2047, 4095])))
    ref = orc.gemm_rows(a, b, rows, "f16")
    err = np.max(np.abs(got[rows] - ref)) / np.max(np.abs(ref))
    say("gemm f16 4096^3: max|d|/max|ref| = %.3e over %d rows" % (err, rows.size))
    assert err <= 5e-3
    # the remaining rows: linearity / checksum  (1^T C) == (1^T A) B in f64
    colsum = got.sum(axis=0, dtype=np.float64)
    want = orc.half_to_float(a).sum(axis=0, dtype=np.float64) @ orc.half_to_float(b).astype(np.float64)
    assert np.max(np.abs(colsum - want)) <= 1e-3 * np.max(np.abs(want)) + 0.05
    # accumulate variant and the reference-signature entry point give C0 + A.B
    c0 = orc.fill_uniform(M * N, "f32", 1, -1, 1).reshape(M, N)
    acc = host.gemm(stream, a, b, c=c0, ab_dtype="f16")
    assert np.max(np.abs(acc - (c0 + got))) <= 1e-4
    d_a, d_b, d_c = stream.to_device(a), stream.to_device(b), stream.to_device(c0)
    fn = stream.kernel("imex_gemm_4kx4kx4k_f16_f16_f32")
    descs, keep = host._pack_params([d_a, d_b, d_c])
    import ctypes as C
    stream.rt.gpuLaunchKernel(stream.handle, fn, 16, 16, 1, 512, 1, 1, 0, C.cast(descs, C.c_void_p), None)
    stream.wait()
    fixed = stream.from_device(d_c, (M, N), np.float32)
    for p in (d_a, d_b, d_c):
        stream.free(p)
    assert np.array_equal(fixed, acc)


@pytest.mark.parametrize("which", ["ta", "tb"])
def test_gemm_transposed_operands(host, orc, stream, which):
    """A stored [K,M] / B stored [N,K] (WG/gemm_4kx4kx4k_transpose_{a,b}.mlir): same
    product as the plain layout; checked the way the reference does, against the
    plain GEMM of the un-transposed copies."""
    kw = {"trans_a": True} if which == "ta" else {"trans_b": True}

    def stored(a, b):
        return (np.ascontiguousarray(a.T), b) if which == "ta" else (a, np.ascontiguousarray(b.T))

    # vector-ALU path: bit-exact against the sequential oracle
    for (M, N, K) in [(5, 7, 9), (100, 36, 130), (300, 260, 50)]:
        a = orc.fill_uniform(M * K, "f16", 31, -1, 1).reshape(M, K)
        b = orc.fill_uniform(K * N, "f16", 32, -1, 1).reshape(K, N)
        sa, sb = stored(a, b)
        assert np.array_equal(host.gemm(stream, sa, sb, **kw), orc.gemm(a, b, "f16"))
    # tiled path: integer operands are exact in any order; non-square so a swapped M/N/K shows
    for (M, N, K) in [(256, 512, 96), (768, 256, 1024)]:
        a = orc.fill_int(M * K, "f16", 33, -4, 4).reshape(M, K)
        b = orc.fill_int(K * N, "f16", 34, -4, 4).reshape(K, N)
        sa, sb = stored(a, b)
        want = orc.to_float(a, "f16").astype(np.int64) @ orc.to_float(b, "f16").astype(np.int64)
        assert np.array_equal(host.gemm(stream, sa, sb, **kw).astype(np.int64), want)
    # layout probes: identity on the transposed side returns the other operand exactly
    M = N = K = 512
    x = orc.fill_uniform(M * K, "f16", 35, -1, 1).reshape(M, K)
    eye = orc.from_float(np.eye(K, dtype=np.float32), "f16")
    if which == "ta":
        assert np.array_equal(host.gemm(stream, np.ascontiguousarray(x.T), eye, **kw), orc.to_float(x, "f16"))
    else:
        assert np.array_equal(host.gemm(stream, eye, np.ascontiguousarray(x.T), **kw), orc.to_float(x, "f16"))
    # random operands at the reference's size and range (-0.5, 0.5), sampled rows + column checksum
    M = N = K = 4096
    a = orc.fill_uniform(M * K, "f16", 36, -0.5, 0.5).reshape(M, K)
    b = orc.fill_uniform(K * N, "f16", 37, -0.5, 0.5).reshape(K, N)
    sa, sb = stored(a, b)
    got = host.gemm(stream, sa, sb, **kw)
    rows = np.array([0, 1, 255, 256, 1999, 4095])
    assert gemm_close(got[rows], orc.gemm_rows(a, b, rows, "f16"))
    colsum = got.sum(axis=0, dtype=np.float64)
    want = orc.half_to_float(a).sum(axis=0, dtype=np.float64) @ orc.half_to_float(b).astype(np.float64)
    assert np.max(np.abs(colsum - want)) <= 1e-3 * np.max(np.abs(want)) + 0.05
    # the reference-signature entry point accumulates onto C
    import ctypes as C
    c0 = orc.fill_uniform(M * N, "f32", 38, -1, 1).reshape(M, N)
    d_a, d_b, d_c = stream.to_device(sa), stream.to_device(sb), stream.to_device(c0)
    fn = stream.kernel("imex_gemm_4kx4kx4k_transpose_a" if which == "ta" else "imex_gemm_4kx4kx4k_transpose_b")
    descs, keep = host._pack_params([d_a, d_b, d_c])
    stream.rt.gpuLaunchKernel(stream.handle, fn, 16, 16, 1, 512, 1, 1, 0, C.cast(descs, C.c_void_p), None)
    stream.wait()
    fixed = stream.from_device(d_c, (M, N), np.float32)
    for p in (d_a, d_b, d_c):
        stream.free(p)
    assert np.max(np.abs(fixed - (c0 + got))) <= 1e-4


def _launch_raw(host, stream, name, args, grid, block=(512, 1, 1)):
    """gpuLaunchKernel with an explicit launch shape (the reference's own, for the fixed-shape entries)."""
    import ctypes as C
    fn = stream.kernel(name)
    descs, keep = host._pack_params(args)
    stream.rt.gpuLaunchKernel(stream.handle, fn, grid[0], grid[1], grid[2], block[0], block[1], block[2], 0,
                              C.cast(descs, C.c_void_p), None)
    stream.wait()
    del keep


def _column_checksum_f64(a_f32, b_f32):
    """(1^T A) B in f64, in column panels so that B is never held whole as f64."""
    s = a_f32.sum(axis=0, dtype=np.float64)
    out = np.empty(b_f32.shape[1], np.float64)
    for n0 in range(0, b_f32.shape[1], 1024):
        out[n0:n0 + 1024] = s @ b_f32[:, n0:n0 + 1024].astype(np.float64)
    return out


STRIDED_ROWS_4096 = np.array(sorted(set(list(range(0, 4096, 97)) + [1, 127, 128, 255, 256, 2047, 2048, 4095])))


def test_gemm_config_mlp_bf16_bias_silu(host, orc, stream):
    M, K, N = 4096, 4096, 11008
    a = orc.fill_normal(M * K, "bf16", 20248, 0.0, 1.0).reshape(M, K)
    b = orc.fill_normal(K * N, "bf16", 20249, 0.0, 0.02).reshape(K, N)
    bias = orc.fill_normal(N, "f32", 20250, 0.0, 0.1)
    got = orc.bfloat_to_float(host.gemm_bias_silu(stream, a, b, bias))
    rows = STRIDED_ROWS_4096  # a stride of 97 lands in every 128-row wavefront block of every 256-row tile
    acc = orc.gemm_rows(a, b, rows, "bf16")
    ref = orc.bfloat_to_float(orc.bias_silu_bf16(acc, bias))
    err = np.max(np.abs(got[rows] - ref)) / np.max(np.abs(ref))
    say("mlp gemm: max|d|/max|ref| = %.3e over %d rows" % (err, rows.size))
    assert err <= 5e-3
    # element-wise: within one bf16 step wherever the value is not tiny
    big = np.abs(ref) > 1e-2
    assert np.max(np.abs(got[rows][big] - ref[big]) / np.abs(ref[big])) <= 2.0 ** -7
    # plain bf16 GEMM with f32 output: the same rows, and every column's sum against (1^T A) B in f64
    plain = host.gemm(stream, a, b, ab_dtype="bf16")
    assert gemm_close(plain[rows], acc)
    want = _column_checksum_f64(orc.bfloat_to_float(a), orc.bfloat_to_float(b))
    assert np.max(np.abs(plain.sum(axis=0, dtype=np.float64) - want)) <= 1e-3 * np.max(np.abs(want)) + 0.05
    # the whole fused output against the epilogue applied (in f64) to that checked f32 product:
    # every element within one bf16 step, so no tile, wavefront block or column strip is left out
    v = plain.astype(np.float64) + bias.astype(np.float64)[None, :]
    want = v / (1.0 + np.exp(-v))
    del v
    d = np.abs(got - want)
    assert np.all(d <= 2.0 ** -7 * np.abs(want) + 1e-6), "fused epilogue differs at %s" % (np.argwhere(d > 2.0 ** -7 * np.abs(want) + 1e-6)[:4],)


def _streamk_against_plain(host, orc, a, b, bias, stream, **kw):
    """The stream-K kernel against the one-workgroup-per-tile kernel on the same operands: the f32 sums
    of a split tile are added in another order (partials, then the finisher's own), so the bf16 results
    agree to a rounding step of the output type, and mostly bit for bit."""
    plain = host.gemm_bias_silu(stream, a, b, bias)
    got = host.gemm_bias_silu(stream, a, b, bias, streamk=True, **kw)
    p, g = orc.bfloat_to_float(plain), orc.bfloat_to_float(got)
    assert np.array_equal(np.isnan(p), np.isnan(g))
    d = np.abs(p - g)
    # a step of the output type, plus the f32 rounding of a sum of K products where the sum nearly cancels
    bad = d > 2.0 ** -7 * np.abs(p) + 1e-4
    assert not bad.any(), (np.argwhere(bad)[:4], p[bad][:4], g[bad][:4])
    return float(np.mean(plain == got))


@pytest.mark.parametrize("M,N,K,grid", [
    (512, 768, 256, None),        # 6 tiles, 4 slabs of 64 k each: one workgroup per tile, nothing to split
    (512, 768, 4096, None),       # 6 tiles over 24 workgroups: every tile split four ways
    (1024, 1280, 2048, (7, 1, 1)),    # 20 tiles on 7 workgroups: two full rounds, 6 tiles dealt out over 7
    (1000, 520, 1024, (5, 1, 1)),     # ragged edge tiles, 12 tiles on 5 workgroups
    (256, 256, 8192, (16, 1, 1)),     # one tile, sixteen parts: a finisher with fifteen partners
    (300, 264, 192, (64, 1, 1)),      # more workgroups than slabs: most ranges are empty
    (512, 512, 96, (3, 1, 1)),        # K % 64 != 0: the kernel takes the ordinary path and ignores the workspace
])
def test_gemm_streamk_small_shapes(host, orc, stream, M, N, K, grid):
    say("stream-K %dx%dx%d grid %s" % (M, N, K, grid))
    a = orc.fill_normal(M * K, "bf16", 31, 0.0, 1.0).reshape(M, K)
    b = orc.fill_normal(K * N, "bf16", 32, 0.0, 0.05).reshape(K, N)
    bias = orc.fill_normal(N, "f32", 33, 0.0, 0.1)
    _streamk_against_plain(host, orc, a, b, bias, stream, grid=grid)
    # integer operands: every order of additions gives the same f32 sums, so the two kernels agree bit for bit
    a = orc.fill_int(M * K, "bf16", 34, -2, 2).reshape(M, K)
    b = orc.fill_int(K * N, "bf16", 35, -2, 2).reshape(K, N)
    assert _streamk_against_plain(host, orc, a, b, np.zeros(N, np.float32), stream, grid=grid) == 1.0
    # ... and twice in a row on one workspace with consecutive epochs (flags of the first launch are stale)
    assert _streamk_against_plain(host, orc, a, b, np.zeros(N, np.float32), stream, grid=grid) == 1.0


def test_gemm_streamk_impatient_finisher(host, orc, stream):
    """A finishing workgroup that is allowed a single look at its partners' flags mostly finds them unset
    and computes the missing slabs itself: the same results, and the kernel ends either way."""
    M, N, K = 768, 512, 4096
    a = orc.fill_int(M * K, "bf16", 36, -2, 2).reshape(M, K)
    b = orc.fill_int(K * N, "bf16", 37, -2, 2).reshape(K, N)
    bias = orc.fill_normal(N, "f32", 38, 0.0, 0.1)
    for grid in ((24, 1, 1), (5, 1, 1)):
        assert _streamk_against_plain(host, orc, a, b, bias, stream, grid=grid, spin_limit=1) == 1.0


def test_gemm_streamk_config_mlp(host, orc, stream):
    """The MLP configuration: 688 tiles on 256 workgroups, two full rounds and 176 tiles dealt out."""
    M, K, N = 4096, 4096, 11008
    a = orc.fill_normal(M * K, "bf16", 20248, 0.0, 1.0).reshape(M, K)
    b = orc.fill_normal(K * N, "bf16", 20249, 0.0, 0.02).reshape(K, N)
    bias = orc.fill_normal(N, "f32", 20250, 0.0, 0.1)
    assert host.launch_shape("imex_gemm_bf16_bias_silu_bf16_streamk", [M, N, K])[0] == (256, 1, 1)
    same = _streamk_against_plain(host, orc, a, b, bias, stream)
    say("stream-K MLP: %.4f of the outputs bit-identical to the plain kernel" % same)
    assert same > 0.95


def test_gemm_split_k_operator_entry(host, orc, stream):
    """imexHipGemmBiasSiluBf16SplitK (include/imex_hip_ops.h): the K-splitting kernel behind one call that
    sizes, allocates and stamps the workspace itself -- a few-tile, deep-K problem, then a larger one (the
    workspace grows), then the first again; each against the one-workgroup-per-tile kernel."""
    ops = host.ops()
    for M, N, K in ((512, 512, 8192), (1024, 1280, 4096), (512, 512, 8192)):
        say("split-K operator entry %dx%dx%d" % (M, N, K))
        a = orc.fill_int(M * K, "bf16", 71, -2, 2).reshape(M, K)
        b = orc.fill_int(K * N, "bf16", 72, -2, 2).reshape(K, N)
        bias = orc.fill_normal(N, "f32", 73, 0.0, 0.1)
        d_a, d_b, d_bias = stream.to_device(a), stream.to_device(b), stream.to_device(bias)
        d_o = stream.to_device(np.full((M, N), 0x7FC1, np.uint16))
        rc = ops.imexHipGemmBiasSiluBf16SplitK(stream.handle, int(d_a), int(d_b), int(d_bias), int(d_o), M, N, K)
        assert rc == 0, ops.imexHipOpsLastError()
        stream.wait()
        got = stream.from_device(d_o, (M, N), np.uint16)
        for p in (d_a, d_b, d_bias, d_o):
            stream.free(p)
        # integer operands: the f32 sums are exact in any order, so the two kernels agree bit for bit
        assert np.array_equal(got, host.gemm_bias_silu(stream, a, b, bias)), (M, N, K)
    assert ops.imexHipGemmBiasSiluBf16SplitK(None, None, None, None, None, 256, 256, 64) == -1
    assert b"queue" in ops.imexHipOpsLastError()


def test_gemm_reference_bias_kernel_4096(host, orc, stream):
    """WG/gemm_4kx4kx4k_f16_f16_f32_bias.mlir:77-116: kernel arguments (bias, C, A, B), grid 16 x 16,
    C = bias[n] + (C + A.B); checked as the test itself does (:160-172): the f32 GEMM onto the initial C,
    then C_ref[i,j] += bias[j].  The initial C is not zero here, so the accumulate is visible."""
    M = N = K = 4096
    a = orc.fill_uniform(M * K, "f16", 61, -0.5, 0.5).reshape(M, K)
    b = orc.fill_uniform(K * N, "f16", 62, -0.5, 0.5).reshape(K, N)
    c0 = orc.fill_uniform(M * N, "f32", 63, -1.0, 1.0).reshape(M, N)
    bias = orc.fill_uniform(N, "f32", 64, -1.0, 1.0)
    d_bias, d_c, d_a, d_b = (stream.to_device(t) for t in (bias, c0, a, b))
    try:
        _launch_raw(host, stream, "imex_gemm_4kx4kx4k_f16_f16_f32_bias", [d_bias, d_c, d_a, d_b], (16, 16, 1))
        got = stream.from_device(d_c, (M, N), np.float32)
        assert np.array_equal(stream.from_device(d_bias, (N,), np.float32), bias)
    finally:
        for p in (d_bias, d_c, d_a, d_b):
            stream.free(p)
    rows = STRIDED_ROWS_4096
    # oracle: the i-k-j loop accumulates onto C0's rows, then the bias loop
    ref = orc.bias_add_rows(orc.gemm_rows(a, b, rows, "f16", c0_rows=c0[rows]), bias)
    err = np.max(np.abs(got[rows] - ref)) / np.max(np.abs(ref))
    say("bias gemm 4096^3: max|d|/max|ref| = %.3e over %d rows" % (err, rows.size))
    assert err <= 5e-3
    assert orc.allclose_f32(got[rows], ref)  # the reference's own check (atol 1e-4, rtol 1e-3)
    # every column: 1^T C = (1^T A) B + 1^T C0 + M bias[n], in f64
    want = (_column_checksum_f64(orc.half_to_float(a), orc.half_to_float(b)) + c0.sum(axis=0, dtype=np.float64)
            + M * bias.astype(np.float64))
    assert np.max(np.abs(got.sum(axis=0, dtype=np.float64) - want)) <= 1e-3 * np.max(np.abs(want)) + 0.05
    # and every element against the accumulate kernel plus the bias (two roundings apart at most)
    acc = host.gemm(stream, a, b, c=c0, ab_dtype="f16")
    assert np.max(np.abs(got - (acc + bias[None, :]))) <= 1e-5


@pytest.mark.parametrize("dtype,M,N,K", [("bf16", 512, 512, 96), ("bf16", 300, 520, 1024), ("f16", 768, 256, 4096)])
def test_gemm_tiled_accumulate_integers_exact(host, orc, stream, dtype, M, N, K):
    """C += A.B on the MFMA path with integer operands and an integer C0: exact in any order."""
    a = orc.fill_int(M * K, dtype, 41, -4, 4).reshape(M, K)
    b = orc.fill_int(K * N, dtype, 42, -4, 4).reshape(K, N)
    c0 = orc.fill_int(M * N, "f32", 43, -1000, 1000).reshape(M, N)
    want = orc.to_float(a, dtype).astype(np.int64) @ orc.to_float(b, dtype).astype(np.int64) + c0.astype(np.int64)
    got = host.gemm(stream, a, b, c=c0, ab_dtype=dtype)
    assert np.array_equal(got.astype(np.int64), want)


def test_gemm_f16_output_4096(host, orc, stream):
    """WG/gemm_4kx4kx4k_f16_f16_f16.mlir at its own size: f32 accumulation, one rounding to f16."""
    M = N = K = 4096
    a = orc.fill_uniform(M * K, "f16", 65, -0.5, 0.5).reshape(M, K)
    b = orc.fill_uniform(K * N, "f16", 66, -0.5, 0.5).reshape(K, N)
    got = orc.half_to_float(host.gemm(stream, a, b, ab_dtype="f16", out_dtype="f16"))
    rows = STRIDED_ROWS_4096
    ref = orc.half_to_float(orc.float_to_half(orc.gemm_rows(a, b, rows, "f16")))
    assert gemm_close(got[rows], ref)
    want = _column_checksum_f64(orc.half_to_float(a), orc.half_to_float(b))
    # 4096 roundings to f16 per column, each below 2^-11 relative
    assert np.max(np.abs(got.sum(axis=0, dtype=np.float64) - want)) <= 2e-3 * np.max(np.abs(want)) + 0.5


def test_gemm_f16_output_variant(host, orc, stream):
    M, N, K = 512, 256, 256
    a = orc.fill_uniform(M * K, "f16", 8, -1, 1).reshape(M, K)
    b = orc.fill_uniform(K * N, "f16", 9, -1, 1).reshape(K, N)
    got = orc.half_to_float(host.gemm(stream, a, b, ab_dtype="f16", out_dtype="f16"))
    ref = orc.gemm(a, b, "f16", out_round="f16")
    assert gemm_close(got, ref)


# ==================== MFMA ceiling measurement kernel ======================
def _ceiling_lds_f16(workgroup, mode):
    """The f16 operands imex_mfma_lds_ceiling_f16 writes into LDS, as (4096 slots, 8)."""
    with np.errstate(over="ignore"):
        i = np.arange(16384, dtype=np.uint32)
        x = (i + np.uint32(workgroup * 7919)) * np.uint32(2654435761)
        x ^= x >> np.uint32(15)
        x *= np.uint32(2246822519)
        x ^= x >> np.uint32(13)
    if mode == 2:
        lo = (x & np.uint32(0x83ff)) | (((x >> np.uint32(10)) % np.uint32(15)) << np.uint32(10))
        hi = ((x >> np.uint32(16)) & np.uint32(0x83ff)) | (((x >> np.uint32(26)) % np.uint32(15)) << np.uint32(10))
    else:
        half = lambda h: (h.astype(np.float32) * np.float32(1.0 / 32768.0) - np.float32(1.0)).astype(np.float16).view(np.uint16).astype(np.uint32)
        lo, hi = half(x & np.uint32(0xffff)), half(x >> np.uint32(16))
    words = lo | (hi << np.uint32(16))
    return words.view(np.uint16).view(np.float16).astype(np.float64).reshape(4096, 8)


@pytest.mark.parametrize("mode", [0, 2])
def test_mfma_ceiling_kernel_computes_what_it_says(host, stream, mode):
    """No oracle and no reference counterpart: the expected sums follow from the published
    operand / accumulator lane layout of MFMA 16x16x32 (A[m = l%16][k = 8(l/16)..+8],
    B likewise in n, C[4(l/16) + r][l%16] in register r), in f64."""
    iters, groups = 5, 3
    say("mfma ceiling probe: %d workgroups x %d steps" % (groups, iters))
    got = host.mfma_lds_ceiling(stream, groups, iters, mode=mode)
    assert got.shape == (groups, 512)
    l = np.arange(64)
    rows = 4 * (l[:, None] // 16) + np.arange(4)[None, :]                      # [lane, r]
    for g in range(groups):
        slots = _ceiling_lds_f16(g, mode)
        for w in range(8):
            lane = w * 64 + l
            total = np.zeros(64)
            for it in range(iters):
                off = (it & 63) * 64
                frag = lambda base: slots[(lane + off + base) & 4095]          # [64 lanes, 8 k]
                def tile(f):                                                     # -> [16, 32]
                    t = np.zeros((16, 32))
                    for k8 in range(4):
                        t[:, 8 * k8:8 * k8 + 8] = f[16 * k8:16 * k8 + 16]
                    return t
                for i in range(8):
                    A = tile(frag(i * 256))
                    for j in range(4):
                        Bt = tile(frag(2048 + j * 256))                          # [n, k]
                        Cm = A @ Bt.T
                        total += Cm[rows, (l % 16)[:, None]].sum(axis=1)
            want = total
            have = got[g, w * 64:(w + 1) * 64].astype(np.float64)
            assert np.all(np.abs(have - want) <= 1e-4 * np.abs(want).max() + 1e-4), (g, w)
    assert not np.any(host.mfma_lds_ceiling(stream, 2, 7, mode=1))
    assert host.mfma_lds_ceiling(stream, 1, 0).shape == (1, 512) and not np.any(host.mfma_lds_ceiling(stream, 1, 0))


# =============================== Launches by kept plans =====================
@pytest.mark.parametrize("rows,cols", [(64, 2000), (3, 77), (200, 512)])
def test_kept_plans_hold_each_operator_to_its_own_bar(host, orc, stream, rows, cols):
    """Stream.launch twice per operator and size, with other buffers the second time, so that the second launch packs its
    arguments for a plan that is kept: every result within the operator's own bar, exact where the operator is."""
    n, k8 = rows * cols, (cols + 7) // 8 * 8
    for seed in (501, 502):
        f = orc.fill_uniform(n, "f32", seed, 0.5, 2.0).reshape(rows, cols)
        h = orc.fill_normal(n, "f16", seed, 0.0, 2.0).reshape(rows, cols)
        g = orc.fill_uniform(n, "f32", seed + 10, -3.0, 3.0).reshape(rows, cols)
        a = orc.fill_uniform(rows * k8, "f16", seed, -1.0, 1.0).reshape(rows, k8)
        b = orc.fill_uniform(k8 * 64, "f16", seed + 10, -1.0, 1.0).reshape(k8, 64)
        exact = orc.half_to_float(a).astype(np.float64) @ orc.half_to_float(b).astype(np.float64)
        sums = f.astype(np.float64).sum(axis=1)
        bits = lambda want: (lambda got: np.array_equal(got.view(np.uint32 if got.itemsize == 4 else np.uint16),
                                                        want.view(np.uint32 if want.itemsize == 4 else np.uint16)))
        for name, dims, ins, out, rest, ok in (
                ("imex_relu_f32", [n], [g], (n,), [n], bits(orc.relu_f32(g.ravel()))),
                ("imex_silu_f16", [n], [h], (n,), [n], bits(orc.silu_16(h.ravel(), "f16"))),
                ("imex_softmax_f16", [rows, cols], [h], (rows, cols), [rows, cols],
                 lambda got: close_16(orc, got, orc.softmax_16(h, "f16"), "f16")),
                # f32 sums of positive terms: `cols` roundings of at most 2^-24 each
                ("imex_rowsum_f32", [rows, cols], [f], (rows,), [rows, cols, 0.0],
                 lambda got: np.all(np.abs(got - sums) <= cols * 2.0 ** -24 * sums)),
                ("imex_reduce_outer_f32", [rows, cols], [g], (cols,), [rows, cols, 0.25], bits(orc.reduce_outer_f32(g, 0.25))),
                ("imex_transpose2d_b16", [rows, cols], [h], (cols, rows), [rows, cols], bits(orc.transpose2d(h))),
                ("imex_loop_fusion_f32", [n], [f, g], (n,), [n], bits(orc.loop_fusion_f32(f.ravel(), g.ravel()))),
                # k8 additions, each rounded by at most 2^-24 of a partial sum; those of uniform products stay below sqrt(k8)
                ("imex_gemm_f16_f16_f32", [rows, 64, k8], [a, b], (rows, 64), [rows, 64, k8],
                 lambda got: np.max(np.abs(got - exact)) <= k8 ** 1.5 * 2.0 ** -24)):
            say("%s %s, seed %d" % (name, dims, seed))
            dtype = np.uint16 if name.endswith(("f16", "b16")) else np.float32
            blank = np.full(out, 7, dtype)
            bufs = [stream.to_device(t) for t in ins] + [stream.to_device(blank)]
            stream.launch(name, dims, bufs + rest)
            stream.wait()
            got = stream.from_device(bufs[-1], out, dtype)
            for p in bufs:
                stream.free(p)
            assert ok(got), (name, seed)
