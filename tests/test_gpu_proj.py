"""Row projections on the device (y = x . W^T, F16 weights, F32 rows) against
the CPU oracle's restatement of the reference matmul, through the C ABI.

The device sums in a different order (matrix-core tiles of 32 inputs, F32
accumulation) and feeds each activation as two half-precision terms, so the
results agree to F32 rounding, not bit for bit.  Tolerance, per output: 3e-7 *
sqrt(n_in) * sum_k |x_k w_k| (a few F32 ulps of the magnitudes summed, growing
like a random walk with the length of the sum), which is also what separates
the reference's own SIMD variants from its scalar loop."""
import ctypes as C

import numpy as np
import pytest

import oracle
from wayruntime_amd import hipattn, synth

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def _device():
    hipattn.init()
    yield


def _w16(seed, n_out, n_in, std):
    return synth.f32_to_f16_trunc(synth.normal(seed, (n_out, n_in), std=std))


def _widen(w16):
    # IEEE binary16 -> float64, the same values the reference's decoder yields
    return np.ascontiguousarray(w16).view(np.float16).astype(np.float64)


def _check(got, x, w16, what):
    want = oracle.matmul_w16(x, w16)
    mag = np.abs(x.astype(np.float64)) @ np.abs(_widen(w16)).T
    tol = 3e-7 * np.sqrt(x.shape[1]) * mag + 1e-37
    err = np.abs(got.astype(np.float64) - want.astype(np.float64))
    assert not np.isnan(got).any(), what
    assert np.all(err <= tol), f"{what}: worst err/tol = {np.max(err / tol):.3f}"


@pytest.mark.parametrize("rows,n_in,n_out,std", [
    (1, 1024, 4096, 0.02),        # Qwen3-0.6B: wq, wk, wv stacked
    (1, 2048, 1024, 0.02),        # wo
    (16, 1024, 3072, 0.02),       # a full batch through an FFN-sized weight
    (9, 96, 48, 0.5),             # three input tiles: no full batch of eight, tail loop only
    (3, 320, 16, 1.0),            # ten input tiles: one batch and a tail; a single output tile
    (8, 32, 64, 1.0),             # one input tile
    (17, 512, 80, 0.1),           # rows pad to four groups of eight; outputs not a multiple of 64
    (300, 256, 128, 0.1),         # prefill-sized rows: the register GEMM, 32 x 32 tiles, inputs split over four waves
    (64, 96, 48, 0.5),            # ... its smallest row count; three input tiles (a wave with none), three output tiles
    (100, 160, 80, 0.3),          # ... a last row group of four rows, five input tiles
    (300, 160, 2512, 0.2),        # ... 64 x 32 tiles, a partial last tile both ways
    (4102, 64, 32, 1.0),          # more rows than one launch takes: 4096 + a six-row launch
    (500, 96, 4112, 0.3),         # LDS-staged GEMM, 128 x 64 tiles, pipelined reads: partial panels, odd input tiles
    (500, 32, 4112, 0.5),         # ... a single input tile
    (500, 128, 4112, 0.3),        # ... an even number of them
    (1000, 1056, 4112, 0.02),     # ... the plain 128 x 64 tile (two workgroups per CU), 33 input tiles
    (1000, 96, 8208, 0.3),        # LDS-staged GEMM, 128 x 128 tiles: partial output and row panels, three input tiles
    (1536, 64, 6144, 0.3),        # ... 576 such tiles would fill 1.1 rounds: the 128 x 64 tile takes over
    (1000, 32, 8208, 0.5),        # ... a single input tile (the ring's prologue covers the whole product)
    (2040, 96, 4112, 0.3),        # LDS-staged GEMM, eight waves, 256 x 128 tiles: partial panels, three input tiles
    (2040, 32, 4112, 0.5),        # ... a single input tile
    (500, 1088, 4112, 0.02),      # ... 34 input tiles, partial panels
    (2047, 2048, 1024, 0.02),     # the output projection of a 2047-token prompt (Qwen3-0.6B): one 128 x 64 tile per CU,
                                  # two sets of waves halving the input range
    (2047, 3072, 1024, 0.02),     # ... its down projection, 96 input tiles
    (2000, 2112, 1040, 0.02),     # ... partial panels both ways, 66 input tiles
    (2000, 2080, 1040, 0.02),     # ... an odd number of input tiles: one set of waves takes the whole range
    (1000, 2048, 1040, 0.02),     # too few LDS tiles for the chip: the register GEMM with a long contraction
])
def test_projection_shapes_vs_oracle(rows, n_in, n_out, std):
    print("proj", rows, n_in, n_out, flush=True)
    x = synth.normal(rows * 7 + n_in, (rows, n_in))
    w16 = _w16(n_out + 3, n_out, n_in, std)
    w = hipattn.Weight([w16])
    _check(w.rows(x), x, w16, f"{rows}x{n_in}x{n_out}")
    w.close()


@pytest.mark.parametrize("rows,n_in,n_out", [(2047, 2048, 1024), (2000, 2112, 1040), (1000, 2048, 1040)])
def test_repeated_launches_give_the_same_bits(rows, n_in, n_out):
    # no sum in these kernels depends on the order in which waves or workgroups finish
    print("proj repeat", rows, n_in, n_out, flush=True)
    x = synth.normal(5, (rows, n_in))
    w16 = _w16(6, n_out, n_in, 0.02)
    w = hipattn.Weight([w16])
    first = w.rows(x)
    for _ in range(4):
        assert w.rows(x).tobytes() == first.tobytes()
    w.close()


def test_stacked_parts_equal_separate_weights():
    n_in = 1024
    parts = [_w16(11, 2048, n_in, 0.02), _w16(12, 1024, n_in, 0.02), _w16(13, 1024, n_in, 0.02)]
    x = synth.normal(14, (2, n_in))
    stacked = hipattn.Weight(parts)
    y = stacked.rows(x)
    assert y.shape == (2, 4096)
    off = 0
    for p in parts:
        single = hipattn.Weight([p])
        assert np.array_equal(single.rows(x), y[:, off:off + p.shape[0]])
        off += p.shape[0]
        single.close()
    stacked.close()


def test_small_integers_are_exact():
    # every product and partial sum is exact in F32 and the half-precision split
    # of a small integer has no low term: any correct implementation gives the
    # integer result bit for bit, a wrong tile or lane mapping cannot
    rng = np.random.default_rng(9)
    rows, n_in, n_out = 5, 160, 48
    xi = rng.integers(-8, 9, size=(rows, n_in))
    wi = rng.integers(-8, 9, size=(n_out, n_in))
    w16 = np.array([oracle.f32_to_f16(float(v)) for v in range(-8, 9)], dtype=np.uint16)[wi + 8]
    w = hipattn.Weight([w16])
    got = w.rows(xi.astype(np.float32))
    assert np.array_equal(got, (xi @ wi.T).astype(np.float32))
    w.close()


def test_row_magnitudes_do_not_matter():
    # rows of very different scale in one call, and one row whose entries span
    # fourteen orders of magnitude: the per-row power-of-two scaling and the
    # scaled low term keep F32-level accuracy (reference: float64)
    n_in, n_out = 256, 32
    x = synth.normal(21, (5, n_in))
    x[0] *= np.float32(1e-20)
    x[1] *= np.float32(1e20)
    x[2, 1:] *= np.float32(5e-5)         # one entry of order 1, the rest tiny
    x[3] = 0.0
    x[4, ::2] *= np.float32(1e-14)
    w16 = _w16(22, n_out, n_in, 0.5)
    w = hipattn.Weight([w16])
    got = w.rows(x).astype(np.float64)
    wf = _widen(w16)
    want = x.astype(np.float64) @ wf.T
    mag = np.abs(x.astype(np.float64)) @ np.abs(wf).T
    assert np.all(got[3] == 0.0)
    assert np.all(np.abs(got - want) <= 3e-7 * np.sqrt(n_in) * mag + 1e-37)
    w.close()


@pytest.mark.parametrize("rows,n_in,n_out", [
    (6, 128, 64), (70, 128, 64),    # the row kernel and the register-tiled one
    (1000, 2048, 1040),             # a GEMM-sized launch
])
def test_device_form_with_strides_and_residual_add(rows, n_in, n_out):
    ldx, ldy = n_in + 32, n_out + 8
    x = synth.normal(31, (rows, ldx))
    add = synth.normal(32, (rows, ldy))
    w16 = _w16(33, n_out, n_in, 0.2)
    w = hipattn.Weight([w16])
    xd = hipattn.DeviceBuffer.from_host(x)
    ad = hipattn.DeviceBuffer.from_host(add)
    yd = hipattn.DeviceBuffer.from_host(np.full((rows, ldy), 7.0, dtype=np.float32))
    w.rows_dev(rows, xd, ldx, yd, ldy, add_dev=ad)
    hipattn.sync()
    y = yd.to_host((rows, ldy))
    plain = w.rows(np.ascontiguousarray(x[:, :n_in]))
    assert np.array_equal(y[:, :n_out], plain + add[:, :n_out])
    assert np.all(y[:, n_out:] == 7.0)              # padding columns are not touched
    # in place: the residual is the output buffer (the device walk's h += W . x)
    w.rows_dev(rows, xd, ldx, ad, ldy, add_dev=ad)
    hipattn.sync()
    y2 = ad.to_host((rows, ldy))
    assert np.array_equal(y2[:, :n_out], y[:, :n_out]) and np.array_equal(y2[:, n_out:], add[:, n_out:])
    for b in (xd, ad, yd):
        b.free()
    w.close()


def test_error_contract():
    lib = hipattn.lib()
    h = C.c_void_p()
    good = _w16(41, 16, 32, 1.0)
    ptrs = (C.c_void_p * 1)(good.ctypes.data)

    def create(rows, n_in):
        return lib.wr_hip_proj_weight_create(1, ptrs, (C.c_uint32 * 1)(rows), n_in, C.byref(h))

    assert create(16, 31) == hipattn.ERR_INVAL           # inputs not a multiple of 32
    assert create(8, 32) == hipattn.ERR_INVAL            # outputs not a multiple of 16
    assert create(0, 32) == hipattn.ERR_INVAL
    assert lib.wr_hip_proj_weight_create(0, ptrs, (C.c_uint32 * 1)(16), 32, C.byref(h)) == hipattn.ERR_INVAL
    assert lib.wr_hip_proj_weight_create(1, None, (C.c_uint32 * 1)(16), 32, C.byref(h)) == hipattn.ERR_INVAL
    assert create(16, 32) == hipattn.OK
    x = np.zeros((1, 32), dtype=np.float32)
    y = np.zeros((1, 16), dtype=np.float32)
    assert lib.wr_hip_proj_rows(h, 1, None, y.ctypes.data) == hipattn.ERR_INVAL
    assert lib.wr_hip_proj_rows(None, 1, x.ctypes.data, y.ctypes.data) == hipattn.ERR_INVAL
    assert lib.wr_hip_proj_rows(h, 0, x.ctypes.data, y.ctypes.data) == hipattn.OK     # nothing to do
    lib.wr_hip_proj_weight_destroy(h)


def test_fused_sources_equal_the_separate_steps():
    # rmsnorm -> projection and swiglu -> projection in one call each must give
    # the bits of the separate row step followed by the plain projection
    lib = hipattn.lib()
    rows, n_in, n_out = 11, 256, 96
    x = synth.normal(51, (rows, n_in), std=2.0)
    nw = synth.normal(52, (n_in,)) * np.float32(0.2) + np.float32(1.0)
    gu = synth.normal(53, (rows, 2 * n_in), std=2.0)
    add = synth.normal(54, (rows, n_out))
    w16 = _w16(55, n_out, n_in, 0.1)
    w = hipattn.Weight([w16])
    D = hipattn.DeviceBuffer
    xd, nwd, gud, addd = D.from_host(x), D.from_host(nw), D.from_host(gu), D.from_host(add)
    tmp, y1, y2 = D(rows * n_in * 4), D(rows * n_out * 4), D(rows * n_out * 4)
    eps = 1e-6
    # norm
    assert lib.wr_hip_rows_rmsnorm_dev(xd.p, n_in, nwd.p, n_in, tmp.p, n_in, rows, n_in, eps) == hipattn.OK
    w.rows_dev(rows, tmp, n_in, y1, n_out, add_dev=addd)
    assert lib.wr_hip_proj_rows_norm_dev(w.h, rows, xd.p, n_in, nwd.p, eps, addd.p, y2.p, n_out) == hipattn.OK
    hipattn.sync()
    a, b = y1.to_host((rows, n_out)), y2.to_host((rows, n_out))
    assert a.tobytes() == b.tobytes()
    want = oracle.matmul_w16(oracle.rmsnorm(x, nw, eps), w16) + add
    assert np.max(np.abs(b - want)) <= 1e-5 * np.max(np.abs(want))
    # swiglu
    assert lib.wr_hip_rows_swiglu_dev(gud.p, 2 * n_in, tmp.p, n_in, rows, n_in) == hipattn.OK
    w.rows_dev(rows, tmp, n_in, y1, n_out)
    assert lib.wr_hip_proj_rows_swiglu_dev(w.h, rows, gud.p, 2 * n_in, None, y2.p, n_out) == hipattn.OK
    hipattn.sync()
    a, b = y1.to_host((rows, n_out)), y2.to_host((rows, n_out))
    assert a.tobytes() == b.tobytes()
    want = oracle.matmul_w16(oracle.silu_mul(np.ascontiguousarray(gu[:, :n_in]),
                                             np.ascontiguousarray(gu[:, n_in:])), w16)
    assert np.max(np.abs(b - want)) <= 1e-5 * np.max(np.abs(want))
    # contracts: missing norm vector, gate/up stride too small
    assert lib.wr_hip_proj_rows_norm_dev(w.h, rows, xd.p, n_in, None, eps, None, y2.p, n_out) == hipattn.ERR_INVAL
    assert lib.wr_hip_proj_rows_swiglu_dev(w.h, rows, gud.p, n_in, None, y2.p, n_out) == hipattn.ERR_INVAL
    for d in (xd, nwd, gud, addd, tmp, y1, y2):
        d.free()
    w.close()


@pytest.mark.parametrize("n_in", [256, 1056, 2080, 4128])
def test_fused_sources_with_many_rows(n_in):
    # 64 rows and more: the fragment kernel that takes a row group per workgroup
    # (values held in registers up to 4096 inputs, re-read beyond) and the GEMM
    # kernels.  The row sums of the norm are formed in another order than in the
    # separate row step, so the comparison is with the oracle, to rounding; the
    # gated activation has no sum and stays bit-identical to the separate steps.
    lib = hipattn.lib()
    rows, n_out = 77, 48
    x = synth.normal(61 + n_in, (rows, n_in), std=2.0)
    nw = synth.normal(62, (n_in,)) * np.float32(0.2) + np.float32(1.0)
    gu = synth.normal(63 + n_in, (rows, 2 * n_in), std=2.0)
    add = synth.normal(64, (rows, n_out))
    w16 = _w16(65, n_out, n_in, 0.1)
    w = hipattn.Weight([w16])
    D = hipattn.DeviceBuffer
    xd, nwd, gud, addd = D.from_host(x), D.from_host(nw), D.from_host(gu), D.from_host(add)
    tmp, y1, y2 = D(rows * n_in * 4), D(rows * n_out * 4), D(rows * n_out * 4)
    eps = 1e-6
    assert lib.wr_hip_proj_rows_norm_dev(w.h, rows, xd.p, n_in, nwd.p, eps, addd.p, y2.p, n_out) == hipattn.OK
    hipattn.sync()
    got = y2.to_host((rows, n_out))
    normed = oracle.rmsnorm(x, nw, eps)
    want = oracle.matmul_w16(normed, w16) + add
    mag = np.abs(normed.astype(np.float64)) @ np.abs(_widen(w16)).T + np.abs(add)
    assert np.all(np.abs(got - want) <= 1e-6 * np.sqrt(n_in) * mag)
    assert lib.wr_hip_rows_swiglu_dev(gud.p, 2 * n_in, tmp.p, n_in, rows, n_in) == hipattn.OK
    w.rows_dev(rows, tmp, n_in, y1, n_out)
    assert lib.wr_hip_proj_rows_swiglu_dev(w.h, rows, gud.p, 2 * n_in, None, y2.p, n_out) == hipattn.OK
    hipattn.sync()
    a, b = y1.to_host((rows, n_out)), y2.to_host((rows, n_out))
    assert a.tobytes() == b.tobytes()
    act = oracle.silu_mul(np.ascontiguousarray(gu[:, :n_in]), np.ascontiguousarray(gu[:, n_in:]))
    _check(b, act, w16, f"swiglu {n_in}")
    for d in (xd, nwd, gud, addd, tmp, y1, y2):
        d.free()
    w.close()


@pytest.mark.parametrize("n_in,n_out", [(1024, 4096), (3072, 1024), (2048, 48), (14336, 64), (96, 16)])
def test_one_row_equals_its_row_of_two(n_in, n_out):
    # A single row takes the kernel that builds its operand terms in LDS; two rows
    # take the fragment launch and then the product.  Same values, same order of
    # every sum: the row's bits must not depend on the company it keeps (the
    # reference's batch contract, src/core/batch.c:15-19).  All three sources.
    lib = hipattn.lib()
    x = synth.normal(71 + n_in, (2, n_in), std=2.0)
    nw = synth.normal(72, (n_in,)) * np.float32(0.2) + np.float32(1.0)
    gu = synth.normal(73 + n_in, (2, 2 * n_in), std=2.0)
    add = synth.normal(74, (2, n_out))
    w16 = _w16(75, n_out, n_in, 0.1)
    w = hipattn.Weight([w16])
    D = hipattn.DeviceBuffer
    xd, nwd, gud, addd = D.from_host(x), D.from_host(nw), D.from_host(gu), D.from_host(add)
    y1, y2 = D(n_out * 4), D(2 * n_out * 4)
    eps = 1e-6
    for what, one, two in (
        ("plain", lambda: w.rows_dev(1, xd, n_in, y1, n_out, add_dev=addd),
         lambda: w.rows_dev(2, xd, n_in, y2, n_out, add_dev=addd)),
        ("norm", lambda: lib.wr_hip_proj_rows_norm_dev(w.h, 1, xd.p, n_in, nwd.p, eps, None, y1.p, n_out),
         lambda: lib.wr_hip_proj_rows_norm_dev(w.h, 2, xd.p, n_in, nwd.p, eps, None, y2.p, n_out)),
        ("swiglu", lambda: lib.wr_hip_proj_rows_swiglu_dev(w.h, 1, gud.p, 2 * n_in, None, y1.p, n_out),
         lambda: lib.wr_hip_proj_rows_swiglu_dev(w.h, 2, gud.p, 2 * n_in, None, y2.p, n_out)),
    ):
        assert one() in (None, hipattn.OK) and two() in (None, hipattn.OK)
        hipattn.sync()
        a, b = y1.to_host((1, n_out)), y2.to_host((2, n_out))
        assert a[0].tobytes() == b[0].tobytes(), what
    _check(w.rows(x[:1]), x[:1], w16, "one row")
    for d in (xd, nwd, gud, addd, y1, y2):
        d.free()
    w.close()


@pytest.mark.parametrize("rows", [1, 11, 70])
def test_geglu_source(rows):
    # gelu_tanh(gate) * up feeding a projection (Gemma's FFN), against the closed
    # form in float64; one row, a few rows and a prefill-sized count take three
    # different fragment paths
    lib = hipattn.lib()
    n_in, n_out = 256, 48
    gu = synth.normal(95 + rows, (rows, 2 * n_in), std=2.0)
    w16 = _w16(96, n_out, n_in, 0.1)
    w = hipattn.Weight([w16])
    D = hipattn.DeviceBuffer
    gud, y = D.from_host(gu), D(rows * n_out * 4)
    assert lib.wr_hip_proj_rows_geglu_dev(w.h, rows, gud.p, 2 * n_in, None, y.p, n_out) == hipattn.OK
    hipattn.sync()
    g, u = gu[:, :n_in].astype(np.float64), gu[:, n_in:].astype(np.float64)
    act = 0.5 * g * (1.0 + np.tanh(0.7978845608 * (g + 0.044715 * g ** 3))) * u
    want = act @ _widen(w16).T
    got = y.to_host((rows, n_out)).astype(np.float64)
    mag = np.abs(act) @ np.abs(_widen(w16)).T
    assert np.all(np.abs(got - want) <= 2e-6 * np.sqrt(n_in) * mag + 1e-30)
    gud.free()
    y.free()
    w.close()


def test_projection_random_shapes():
    # a seeded sweep over row counts, input and output widths that crosses every
    # kernel-selection boundary (1 row, 2-63 rows, the four GEMM tilings, more
    # rows than a launch takes), checked against the oracle like the fixed cases
    rng = np.random.default_rng(20240607)
    row_choices = [1, 2, 7, 8, 9, 16, 17, 40, 63, 64, 65, 127, 128, 129, 500, 1023, 1025, 2047, 4096, 4100]
    done = 0
    for case in range(28):
        rows = int(rng.choice(row_choices))
        n_in = 32 * int(rng.integers(1, 40))
        budget = max(16, int(2.5e8 / (rows * n_in)) // 16 * 16)
        n_out = 16 * int(rng.integers(1, min(520, budget // 16) + 1))
        print("random proj", case, rows, n_in, n_out, flush=True)
        x = synth.normal(1000 + case, (rows, n_in), std=float(rng.choice([0.01, 1.0, 30.0])))
        w16 = _w16(2000 + case, n_out, n_in, 0.2)
        w = hipattn.Weight([w16])
        _check(w.rows(x), x, w16, f"case {case}: {rows}x{n_in}x{n_out}")
        w.close()
        done += 1
    assert done == 28


@pytest.mark.parametrize("rows,n_in,n_out", [
    (17, 1024, 4096),             # (each workgroup makes its own fragments; whole shares in one turn of eight)
    (48, 2080, 16),               # register tiles of 16 x 8: one output tile, 65 input tiles (a wave with one more than the others)
    (17, 1056, 1360),             # ... 255 of them, the last row group of one row
    (31, 32, 48),                 # ... a single input tile: three waves with none
    (31, 800, 48),                # ... 25: six and seven k-steps a wave, less than a turn
    (256, 3104, 80),              # ... the last row count whose fragments are made row by row
    (256, 3072, 80),              # (each workgroup makes its own)
    (17, 800, 1392),              # 16 x 16: 87 by 2, the last row group of one row
    (300, 256, 144),              # ... a row group past the end
    (48, 2080, 1392),             # 32 x 16 tiles
    (31, 1056, 3488),             # ... 109 by 2, 33 input tiles
    (20, 800, 7296),              # 32 x 32: fewer row groups than a tile has
    (17, 1056, 8208),             # 64 x 32: likewise, a last run of one output tile
    (49, 800, 4112),              # ... and 25 input tiles,
    (250, 1056, 4112),            # ... 33, row groups past the end
    (257, 288, 1040),             # ... fragments by row groups
    (130, 1088, 9872),            # LDS tiles with two sets of waves and too few workgroups for all CUs
    (2047, 64, 1040),             # LDS tiles whose panels are shared out over few XCDs: 9 by 32 of them
    (4095, 96, 528),              # ... 5 by 64
    (1100, 64, 8208),             # ... the outputs over all eight: 33 by 18
])
def test_products_of_a_short_prompt(rows, n_in, n_out):
    print("proj short prompt", rows, n_in, n_out, flush=True)
    x, w16 = synth.normal(rows * 7 + n_in, (rows, n_in)), _w16(n_out + 3, n_out, n_in, 0.05)
    w = hipattn.Weight([w16])
    got = w.rows(x)
    _check(got, x, w16, f"{rows}x{n_in}x{n_out}")
    assert w.rows(x).tobytes() == got.tobytes()
    w.close()


@pytest.mark.parametrize("rows", [20, 270])
@pytest.mark.parametrize("n_in", [256, 1056, 2080, 4128])
def test_normed_and_gated_rows_by_rows_and_by_groups(rows, n_in):
    # the two fragment kernels a product of many rows may take, all forms of each
    lib, D, n_out, eps = hipattn.lib(), hipattn.DeviceBuffer, 48, 1e-6
    x, gu = synth.normal(161 + n_in, (rows, n_in), std=2.0), synth.normal(163 + n_in, (rows, 2 * n_in), std=2.0)
    nw, w16 = synth.normal(162, (n_in,)) * np.float32(0.2) + np.float32(1.0), _w16(165, n_out, n_in, 0.1)
    w, xd, nwd, gud, y = hipattn.Weight([w16]), D.from_host(x), D.from_host(nw), D.from_host(gu), D(rows * n_out * 4)
    assert lib.wr_hip_proj_rows_norm_dev(w.h, rows, xd.p, n_in, nwd.p, eps, None, y.p, n_out) == hipattn.OK
    normed = oracle.rmsnorm(x, nw, eps)
    mag = np.abs(normed.astype(np.float64)) @ np.abs(_widen(w16)).T
    assert np.all(np.abs(y.to_host((rows, n_out)) - oracle.matmul_w16(normed, w16)) <= 1e-6 * np.sqrt(n_in) * mag)
    assert lib.wr_hip_proj_rows_swiglu_dev(w.h, rows, gud.p, 2 * n_in, None, y.p, n_out) == hipattn.OK
    act = oracle.silu_mul(np.ascontiguousarray(gu[:, :n_in]), np.ascontiguousarray(gu[:, n_in:]))
    _check(y.to_host((rows, n_out)), act, w16, f"swiglu {rows} {n_in}")
    for d in (xd, nwd, gud, y):
        d.free()
    w.close()


@pytest.mark.parametrize("rows,n_in,n_out", [
    (2, 512, 16), (16, 512, 8176),                   # one tile; three tiles a workgroup, 511 of them
    (8, 1024, 16368), (16, 1024, 4112),              # four, 1023 of them; three, 257
    (9, 1536, 4112), (5, 1536, 8192),                # two tiles a workgroup, the last with one; the most for it
    (16, 2048, 2064), (11, 2560, 48), (16, 3072, 1024), (9, 1024, 1024),
    (17, 1024, 4096), (41, 2048, 656),               # more than a decode step's rows: the last group of one row
    (16, 640, 4112), (9, 640, 4096), (9, 4224, 4112), (3, 5120, 3280),   # inputs none takes: 32 x 16 tiles, 16 x 8, streams
])
def test_rows_whose_workgroups_make_their_own_terms(rows, n_in, n_out):
    # Every row has the bits of the row alone (up to sixteen of them) and of the same
    # rows on an address that only the separate fragment launch takes, plain and
    # normalised, with a residual.  Row 1 is zero, a row holds magnitudes down to
    # where either term rounds away, one an infinity and one a NaN.
    print("own terms", rows, n_in, n_out, flush=True)
    lib, D, eps = hipattn.lib(), hipattn.DeviceBuffer, 1e-6
    x = synth.normal(211 + n_in, (rows, n_in), std=2.0)
    x[1] = 0.0
    x[0, 7::5] *= np.float32(2.0) ** -np.arange(len(x[0, 7::5]), dtype=np.float32).clip(0, 60)
    if rows > 4:
        x[3, 11], x[4, n_in - 1] = np.inf, np.nan
    nw, w16 = synth.normal(212, (n_in,)) * np.float32(0.2) + np.float32(1.0), _w16(213, n_out, n_in, 0.1)
    add = synth.normal(214, (rows, n_out))
    w, xd, nwd, addd = hipattn.Weight([w16]), D.from_host(x), D.from_host(nw), D.from_host(add)
    off = D.from_host(np.concatenate([np.zeros(1, np.float32), x.ravel()]))
    y, ya, y1 = D(rows * n_out * 4), D(rows * n_out * 4), D(n_out * 4)

    def run(norm, n, xp, addp, yp):
        if norm:
            return lib.wr_hip_proj_rows_norm_dev(w.h, n, xp, n_in, nwd.p, eps, addp, yp, n_out)
        return lib.wr_hip_proj_rows_dev(w.h, n, xp, n_in, addp, yp, n_out)

    finite = [i for i in range(rows) if np.isfinite(x[i]).all()]
    for norm in (False, True):
        assert run(norm, rows, xd.p, addd.p, y.p) == hipattn.OK
        assert run(norm, rows, off.p + 4, addd.p, ya.p) == hipattn.OK
        got, apart = y.to_host((rows, n_out)), ya.to_host((rows, n_out))
        assert got.tobytes() == apart.tobytes(), f"norm {norm}: not the bits of the separate fragments"
        src = oracle.rmsnorm(x, nw, eps) if norm else x
        src, got_f = src[finite], got[finite]
        want = oracle.matmul_w16(src, w16) + add[finite]
        mag = np.abs(src.astype(np.float64)) @ np.abs(_widen(w16)).T + np.abs(add[finite])
        assert np.all(np.abs(got_f - want) <= 1e-6 * np.sqrt(n_in) * mag)
        for i in range(min(rows, 16) if rows <= 16 else 0):
            assert run(norm, 1, xd.p + i * n_in * 4, addd.p + i * n_out * 4, y1.p) == hipattn.OK
            assert got[i].tobytes() == y1.to_host((n_out,)).tobytes(), f"norm {norm} row {i}"
    if n_in == n_out:
        assert run(False, rows, xd.p, None, ya.p) == hipattn.OK
        apart = ya.to_host((rows, n_out))
        assert run(False, rows, xd.p, None, xd.p) == hipattn.OK
        assert xd.to_host((rows, n_out)).tobytes() == apart.tobytes()
    for d in (xd, nwd, addd, off, y, ya, y1):
        d.free()
    w.close()


@pytest.mark.parametrize("rows,n_in,ffn", [
    (1, 1024, 3072), (1, 96, 48), (1, 3104, 8208),                # one row: four waves a pair, none shared, two, an odd count
    (1, 1024, 1040), (1, 768, 16), (1, 1536, 2048), (1, 320, 528),    # ... eight gates with their values, batches of eight and four, rests
    (1, 15360, 2064), (1, 15360, 32), (1, 15392, 32),             # ... more than 64 KiB of LDS, the most inputs, fragments apart
    (2, 512, 16), (16, 1024, 3072), (8, 1536, 2064), (9, 512, 4080),   # workgroups that make their own terms: a pair, two
    (24, 1024, 1024), (20, 1024, 2048), (17, 2048, 528), (100, 512, 272),    # ... more than two row groups, the last ones short
    (17, 1024, 2736), (17, 1024, 2752), (40, 1024, 3264), (40, 512, 3280), (33, 1536, 2064),    # ... up to one a CU, two, more, no such form
    (5, 1056, 528), (16, 160, 48), (16, 1024, 16400),             # a wave per pair of tiles, inputs split and not
    (17, 1056, 528), (17, 800, 1376), (100, 288, 2064), (17, 800, 2736), (17, 1056, 4128),    # register tiles of 32 x 8, 32 x 16 (two), 32 x 32, 64 x 32
    (130, 1088, 4944), (200, 1056, 8208),                         # LDS tiles of 128 x 64 (few, two sets of waves; two a CU)
    (300, 1024, 4112), (700, 2048, 2064), (700, 1056, 2064),      # LDS tiles of 128 x 64 (two and more a CU; one, two sets of waves; one)
    (1030, 288, 6160), (2050, 288, 4112),                         # of 128 x 128, of 256 x 128
])
def test_gates_and_values_in_one_product_equal_product_then_activation(rows, n_in, ffn):
    # act(gate) * value from the product itself has the bits of the product followed
    # by the activation's own step, SiLU directly and GELU through the next product,
    # normalised or not; nothing is written beyond ffn.
    print("gated", rows, n_in, ffn, flush=True)
    lib, D, eps, n2 = hipattn.lib(), hipattn.DeviceBuffer, 1e-6, 32
    x = synth.normal(221 + n_in, (rows, n_in), std=2.0)
    nw = synth.normal(222, (n_in,)) * np.float32(0.2) + np.float32(1.0)
    w, wd = hipattn.Weight([_w16(223, ffn, n_in, 0.1), _w16(224, ffn, n_in, 0.1)]), None
    xd, nwd, gu = D.from_host(x), D.from_host(nw), D(rows * 2 * ffn * 4)
    act, ld = D(rows * ffn * 4), ffn + 4
    fill = np.full((rows, ld), 7.0, dtype=np.float32)
    got = D.from_host(fill)
    if ffn % 32 == 0:
        wd = hipattn.Weight([_w16(225, n2, ffn, 0.1)])
        ya, yb = D(rows * n2 * 4), D(rows * n2 * 4)
    for norm in (True, False):
        if norm:
            assert lib.wr_hip_proj_rows_norm_dev(w.h, rows, xd.p, n_in, nwd.p, eps, None, gu.p, 2 * ffn) == hipattn.OK
        else:
            w.rows_dev(rows, xd, n_in, gu, 2 * ffn)
        assert lib.wr_hip_rows_swiglu_dev(gu.p, 2 * ffn, act.p, ffn, rows, ffn) == hipattn.OK
        assert lib.wr_hip_proj_rows_gated_dev(w.h, rows, xd.p, n_in, nwd.p if norm else None, eps, 0, got.p, ld) == hipattn.OK
        g = got.to_host((rows, ld))
        assert np.isfinite(g).all() and g[:, :ffn].tobytes() == act.to_host((rows, ffn)).tobytes(), f"norm {norm}"
        assert np.all(g[:, ffn:] == 7.0)
        if wd:
            assert lib.wr_hip_proj_rows_geglu_dev(wd.h, rows, gu.p, 2 * ffn, None, ya.p, n2) == hipattn.OK
            assert lib.wr_hip_proj_rows_gated_dev(w.h, rows, xd.p, n_in, nwd.p if norm else None, eps, 1, act.p, ffn) == hipattn.OK
            wd.rows_dev(rows, act, ffn, yb, n2)
            assert ya.to_host((rows, n2)).tobytes() == yb.to_host((rows, n2)).tobytes(), f"norm {norm} gelu"
    assert lib.wr_hip_proj_rows_gated_dev(w.h, rows, xd.p, n_in, None, eps, 0, got.p, ffn - 4) == hipattn.ERR_INVAL
    assert lib.wr_hip_proj_rows_gated_dev(w.h, rows, xd.p, n_in, None, eps, 0, got.p + 4, ld) == hipattn.ERR_INVAL
    assert lib.wr_hip_proj_rows_gated_dev(w.h, 0, xd.p, n_in, None, eps, 0, got.p, ld) == hipattn.OK
    for d in (xd, nwd, gu, act, got) + ((ya, yb) if wd else ()):
        d.free()
    for h in (w, wd):
        if h:
            h.close()


@pytest.mark.parametrize("rows", [1, 2, 16, 20])
@pytest.mark.parametrize("n", [1024, 4096])
def test_result_over_its_own_input(rows, n):
    # every source, written over the rows it came from: the bits of the result beside them
    lib, D, eps = hipattn.lib(), hipattn.DeviceBuffer, 1e-6
    print("in place", rows, n, flush=True)
    x, two = synth.normal(231, (rows, n), std=2.0), synth.normal(232, (rows, 2 * n), std=2.0)
    nw = D.from_host(synth.normal(233, (n,)) * np.float32(0.2) + np.float32(1.0))
    w, wg = hipattn.Weight([_w16(234, n, n, 0.1)]), hipattn.Weight([_w16(235, n, n, 0.1), _w16(236, n, n, 0.1)])
    for form in ("plain", "norm", "gated", "gated norm", "swiglu"):
        src = two if form == "swiglu" else x
        xd, y = D.from_host(src), D(rows * 2 * n * 4)

        def run(to, ld):
            if form == "plain":
                return lib.wr_hip_proj_rows_dev(w.h, rows, xd.p, n, None, to, ld)
            if form == "norm":
                return lib.wr_hip_proj_rows_norm_dev(w.h, rows, xd.p, n, nw.p, eps, None, to, ld)
            if form == "swiglu":
                return lib.wr_hip_proj_rows_swiglu_dev(w.h, rows, xd.p, 2 * n, None, to, ld)
            return lib.wr_hip_proj_rows_gated_dev(wg.h, rows, xd.p, n, nw.p if "norm" in form else None, eps, 0, to, ld)

        ld = src.shape[1]
        assert run(y.p, ld) == hipattn.OK
        want = y.to_host((rows, ld))[:, :n].copy()
        at = n if form == "swiglu" else 0                  # (over the second half, the gated values)
        assert run(xd.p + at * 4, ld) == hipattn.OK
        assert xd.to_host((rows, ld))[:, at:at + n].tobytes() == want.tobytes(), form
        for d in (xd, y):
            d.free()
    nw.free()
    w.close()
    wg.close()


def test_gated_product_refuses_an_odd_number_of_tiles():
    w = hipattn.Weight([_w16(226, 48, 64, 0.1)])
    b = hipattn.DeviceBuffer(4096)
    assert hipattn.lib().wr_hip_proj_rows_gated_dev(w.h, 1, b.p, 64, None, 1e-6, 0, b.p, 24) == hipattn.ERR_INVAL
    b.free()
    w.close()


@pytest.mark.parametrize("n_out,n_in", [(16, 32), (208, 1024), (48, 1056), (32, 4096)])
def test_embedding_rows(n_out, n_in):
    """Rows of a weight by token, beyond one launch's arguments: the table's values, times the scale."""
    rng = np.random.default_rng(n_in)
    table = (rng.standard_normal((n_out, n_in)) * 2.0 ** rng.integers(-24, 4, (n_out, 1))).astype(np.float16)
    w = hipattn.Weight([table.view(np.uint16)])
    lib = hipattn.lib()
    for rows, scale in ((1, 1.0), (17, 45.25), (960, 1.0), (961, 0.5), (2047, 1.0)):
        ld = n_in + 4
        tokens = rng.integers(0, n_out, rows).astype(np.uint32)
        out = hipattn.DeviceBuffer.from_host(np.full((rows, ld), 7.0, dtype=np.float32))
        assert lib.wr_hip_proj_embed_dev(w.h, rows, tokens.ctypes.data_as(C.POINTER(C.c_uint32)), scale, out.p, ld) == hipattn.OK
        got = out.to_host((rows, ld))
        assert np.array_equal(got[:, :n_in], table[tokens].astype(np.float32) * np.float32(scale)), rows
        assert np.all(got[:, n_in:] == 7.0)
        tokens[rows // 2] = n_out
        assert lib.wr_hip_proj_embed_dev(w.h, rows, tokens.ctypes.data_as(C.POINTER(C.c_uint32)), scale, out.p, ld) == hipattn.ERR_INVAL
        out.free()
    w.close()


@pytest.mark.parametrize("n_in", [512, 1024, 1536, 2048, 2560, 3072])
def test_rows_of_a_few_equal_the_row_alone(n_in):
    # The kernel that makes its own operand terms takes four rows to a workgroup of a narrow
    # weight and eight of a wider one: on either side of a workgroup's rows, and where the two
    # meet (256 compute units, 64 tiles: 16 rows; 68 tiles: 12), the bits are those of a row alone.
    lib = hipattn.lib()
    D = hipattn.DeviceBuffer
    for n_out in (1024, 1088):
        x = synth.normal(81 + n_in, (17, n_in), std=2.0)
        nw = synth.normal(82, (n_in,)) * np.float32(0.2) + np.float32(1.0)
        add = synth.normal(83, (17, n_out))
        w = hipattn.Weight([_w16(84, n_out, n_in, 0.1)])
        xd, nwd, addd, y = D.from_host(x), D.from_host(nw), D.from_host(add), D(17 * n_out * 4)
        for norm in (False, True):
            def call(at, rows):
                xp, ap = xd.p + at * n_in * 4, addd.p + at * n_out * 4
                if norm:
                    rc = lib.wr_hip_proj_rows_norm_dev(w.h, rows, xp, n_in, nwd.p, 1e-6, ap, y.p, n_out)
                else:
                    rc = lib.wr_hip_proj_rows_dev(w.h, rows, xp, n_in, ap, y.p, n_out)
                assert rc == hipattn.OK
                hipattn.sync()
                return y.to_host((17, n_out))[:rows].copy()
            alone = np.concatenate([call(i, 1) for i in range(16)])
            for at, rows in ((0, 2), (3, 3), (1, 4), (2, 5), (4, 7), (0, 8), (5, 9), (1, 12), (0, 13), (0, 15), (0, 16)):
                print("rows", n_in, n_out, norm, at, rows, flush=True)
                assert call(at, rows).tobytes() == alone[at:at + rows].tobytes()
        for d in (xd, nwd, addd, y):
            d.free()
        w.close()


@pytest.mark.parametrize("n_in,n_out", [(96, 32768), (1024, 32912), (64, 32800), (256, 144)])
def test_rows_of_a_product_into_host_memory(n_in, n_out):
    # One row, weights that a wave takes alone (ragged ends of a workgroup's 128 outputs among
    # them) and a narrow one: the bits of the product in device memory, and nothing beside the rows.
    lib = hipattn.lib()
    D = hipattn.DeviceBuffer
    x = synth.normal(91 + n_in, (17, n_in), std=2.0)
    nw = synth.normal(92, (n_in,)) * np.float32(0.2) + np.float32(1.0)
    w = hipattn.Weight([_w16(93, n_out, n_in, 0.1)])
    xd, nwd, y = D.from_host(x), D.from_host(nw), D(17 * n_out * 4)
    places = [lib.wr_hip_attn_host_alloc((n_out + 4) * 4) for _ in range(16)]
    rows = [np.ctypeslib.as_array(C.cast(p, C.POINTER(C.c_float)), shape=(n_out + 4,)) for p in places]
    dst = (C.c_void_p * 16)(*places)
    for n in (1, 2, 3, 7, 8, 9, 13, 16):
        for r in rows:
            r[:] = 7.0
        assert lib.wr_hip_proj_rows_norm_dev(w.h, n, xd.p, n_in, nwd.p, 1e-6, None, y.p, n_out) == hipattn.OK
        hipattn.sync()
        want = y.to_host((17, n_out))[:n]
        print("rows down", n_in, n_out, n, flush=True)
        assert lib.wr_hip_proj_rows_norm_down(w.h, n, xd.p, n_in, nwd.p, 1e-6, dst, y.p) == hipattn.OK
        for i, r in enumerate(rows):
            assert np.array_equal(r[:n_out], want[i]) if i < n else np.all(r == 7.0)
            assert np.all(r[n_out:] == 7.0)
    down = lib.wr_hip_proj_rows_norm_down
    assert down(w.h, 17, xd.p, n_in, nwd.p, 1e-6, dst, y.p) == hipattn.ERR_LIMIT
    assert down(w.h, 2, xd.p, n_in, None, 1e-6, dst, y.p) == hipattn.ERR_INVAL
    assert down(w.h, 2, xd.p, n_in, nwd.p, 1e-6, dst, None) == hipattn.ERR_INVAL
    assert down(w.h, 1, xd.p, n_in, nwd.p, 1e-6, dst, None) == hipattn.OK           # one row needs no memory of the caller's
    assert lib.wr_hip_proj_rows_norm_dev(w.h, 1, xd.p, n_in, nwd.p, 1e-6, None, y.p, n_out) == hipattn.OK
    hipattn.sync()
    assert np.array_equal(rows[0][:n_out], y.to_host((17, n_out))[0])
    assert down(w.h, 2, xd.p, n_in, nwd.p, 1e-6, (C.c_void_p * 2)(places[0], places[1] + 4), y.p) == hipattn.ERR_INVAL
    assert down(w.h, 0, xd.p, n_in, nwd.p, 1e-6, dst, y.p) == hipattn.OK
    for p in places:
        lib.wr_hip_attn_host_free(p)
    for d in (xd, nwd, y):
        d.free()
    w.close()
