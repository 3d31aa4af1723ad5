"""The matrix products of mixer-stack models by themselves, through the C ABI: every
kernel the row and output counts can select, every place an output can go, against
numpy on the same (bfloat16-exact) operands."""
import ctypes as C

import numpy as np
import pytest

from tests import mixer_oracle as O
from wayruntime_amd import hipattn

pytestmark = pytest.mark.gpu

ROWS_F32, ROWS, FRAG, SPLIT, GATED, SPLIT_GATED = range(6)
u32, vp = C.c_uint32, C.c_void_p


class Gemm(C.Structure):
    _fields_ = [("w", vp), ("x", vp), ("x_kt", u32), ("x_kt_z", u32), ("rows", u32), ("group_expert", vp),
                ("tile_groups", u32), ("out", u32), ("y_f32", vp), ("y_act", vp), ("ldy", u32), ("h", vp), ("h_kt", u32),
                ("col_z", u32), ("n_split", u32), ("silu_end", u32), ("sigmoid_end", u32), ("relu2", u32), ("scale", C.c_float),
                ("tanh_end", u32), ("gelu", u32), ("x_kt0", u32), ("bias", vp), ("limit", C.c_float), ("slope", C.c_float),
                ("up_bias", C.c_float), ("x_perm", vp), ("h_kt0", u32), ("x_scale", vp)]


@pytest.fixture(scope="module")
def lib():
    hipattn.init(0)
    lib = hipattn.lib()
    lib.wr_hip_mix_mat_create.argtypes = [u32, u32, u32, vp, C.POINTER(vp)]
    lib.wr_hip_mix_mat_destroy.argtypes = [vp]
    lib.wr_hip_mix_mat_destroy.restype = None
    lib.wr_hip_mix_gemm_run.argtypes = [C.c_int, C.POINTER(Gemm)]
    return lib


def frag(x):
    """[rows][K] -> operand order [rows/16][K/32][64][8], rows padded with NaN (nobody may use them)."""
    r = -(-x.shape[0] // 16) * 16
    p = np.full((r, x.shape[1]), np.nan, dtype=np.float32)
    p[:len(x)] = x
    return np.ascontiguousarray(p.reshape(r // 16, 16, -1, 4, 8).transpose(0, 2, 3, 1, 4))


def unfrag(f, rows, K):
    return f.reshape(-1, K // 32, 4, 16, 8).transpose(0, 3, 1, 2, 4).reshape(-1, K)[:rows]


class Run:
    def __init__(self, lib, f32, batch, N, K, rows, seed=0):
        rng = np.random.default_rng(seed)
        self.lib, self.f32, self.N, self.K, self.rows = lib, f32, N, K, rows
        self.bits = O.f32_to_bf16(rng.standard_normal((batch, N, K), dtype=np.float32) / np.float32(np.sqrt(K)))
        self.w = O.bf16_to_f32(self.bits)
        self.h = vp()
        assert lib.wr_hip_mix_mat_create(batch, N, K, self.bits.ctypes.data, C.byref(self.h)) == 0
        self.rng = rng

    def act(self, rows, K):
        x = self.rng.standard_normal((rows, K), dtype=np.float32)
        return x if self.f32 else O.bf16_to_f32(O.f32_to_bf16(x))

    def up(self, x):
        f = frag(x)
        return hipattn.DeviceBuffer.from_host(f if self.f32 else O.f32_to_bf16(np.nan_to_num(f, nan=0.0)) +
                                              np.where(np.isnan(f), np.uint16(0x7FC0), np.uint16(0)).astype(np.uint16))

    def go(self, x, **kw):
        g = Gemm(w=self.h, x=x.p, x_kt=kw.pop("x_kt", self.K // 32), rows=kw.pop("rows", self.rows), **kw)
        assert self.lib.wr_hip_mix_gemm_run(int(self.f32), C.byref(g)) == 0
        hipattn.sync()

    def frag_down(self, buf, rows, K):
        n = -(-rows // 16) * 16 * K
        if self.f32:
            return unfrag(buf.to_host((n,)), rows, K)
        b = buf.to_host((n // 2,)).view(np.uint16)
        return unfrag(O.bf16_to_f32(b), rows, K)

    def close(self, got, want, eight_bits=False):
        tol = 2.0 ** -7 if eight_bits and not self.f32 else 2e-5
        assert np.isfinite(got).all()
        err = np.abs(got - want).max() / max(1.0, np.abs(want).max())
        assert err < tol, err

    def end(self):
        self.lib.wr_hip_mix_mat_destroy(self.h)


# (outputs, inputs, rows): what each picks among the streaming kernels and the three LDS-staged tiles
SHAPES = [(16, 32, 1), (48, 800, 5), (64, 1504, 16), (6400, 736, 9), (48, 96, 7), (32, 416, 16), (4096, 64, 3), (80, 4096, 16), (64, 64, 17), (96, 160, 33), (160, 96, 70),
          (1024, 512, 200), (8192, 96, 256), (16384, 64, 250), (16384, 64, 600), (2064, 352, 1100)]


@pytest.mark.parametrize("f32", [False, True])
@pytest.mark.parametrize("N,K,rows", SHAPES)
def test_rows_out(lib, f32, N, K, rows):
    r = Run(lib, f32, 1, N, K, rows)
    x = r.act(rows, K)
    y = hipattn.DeviceBuffer(rows * N * 4)
    xd = r.up(x)
    want = x.astype(np.float64) @ r.w[0].T.astype(np.float64)
    r.go(xd, out=ROWS_F32, y_f32=y.p, ldy=N, scale=0.5)
    r.close(y.to_host((rows, N)), 0.5 * want)
    silu, sig = N // 2 + 3, N - 5                          # ends inside a tile
    r.go(xd, out=ROWS_F32, y_f32=y.p, ldy=N, silu_end=silu, sigmoid_end=sig)
    act = want.copy()
    act[:, :silu] = O.silu(want[:, :silu])
    act[:, silu:sig] = O.sigmoid(want[:, silu:sig])
    r.close(y.to_host((rows, N)), act)
    r.go(xd, out=ROWS_F32, y_f32=y.p, ldy=N, silu_end=N // 4, tanh_end=N - 7)
    act = want.copy()
    act[:, :N // 4] = O.silu(want[:, :N // 4])
    act[:, N // 4:N - 7] = np.tanh(want[:, N // 4:N - 7])
    r.close(y.to_host((rows, N)), act)
    bias = r.rng.standard_normal(N).astype(np.float32)
    bd = hipattn.DeviceBuffer.from_host(bias)
    r.go(xd, out=ROWS_F32, y_f32=y.p, ldy=N, bias=bd.p)
    r.close(y.to_host((rows, N)), want + bias)
    r.end()
    for b in (y, xd, bd):
        b.free()


@pytest.mark.parametrize("f32", [False, True])
@pytest.mark.parametrize("N,K,rows", [(64, 96, 1), (128, 64, 20), (512, 64, 90), (16384, 32, 300)])
def test_frag_split_and_gated_out(lib, f32, N, K, rows):
    r = Run(lib, f32, 1, N, K, rows)
    x = r.act(rows, K)
    xd = r.up(x)
    want = x.astype(np.float64) @ r.w[0].T.astype(np.float64)
    esize = 4 if f32 else 2
    h = hipattn.DeviceBuffer(-(-rows // 16) * 16 * N * esize)
    r.go(xd, out=FRAG, h=h.p, h_kt=N // 32, relu2=1)
    r.close(r.frag_down(h, rows, N), np.maximum(want, 0) ** 2, eight_bits=True)
    split = N // 2 // 32 * 32
    y = hipattn.DeviceBuffer(rows * (N - split) * 4)
    r.go(xd, out=SPLIT, h=h.p, h_kt=split // 32, n_split=split, y_f32=y.p, ldy=N - split)
    r.close(r.frag_down(h, rows, split), want[:, :split], eight_bits=True)
    r.close(y.to_host((rows, N - split)), want[:, split:])
    r.go(xd, out=GATED, h=h.p, h_kt=N // 64)
    t = want.reshape(rows, N // 32, 2, 16)
    r.close(r.frag_down(h, rows, N // 2), (O.silu(t[:, :, 0]) * t[:, :, 1]).reshape(rows, -1), eight_bits=True)
    r.go(xd, out=GATED, h=h.p, h_kt=N // 64, gelu=1)
    r.close(r.frag_down(h, rows, N // 2), (O.gelu_tanh(t[:, :, 0]) * t[:, :, 1]).reshape(rows, -1), eight_bits=True)

    def clamped(g, u, limit, slope, more):
        g = np.minimum(g, limit)
        return g * O.sigmoid(slope * g) * (np.clip(u, -limit, limit) + more)
    for limit in (0.3, 5.0):
        r.go(xd, out=GATED, h=h.p, h_kt=N // 64, limit=limit, slope=1.5, up_bias=0.75)
        r.close(r.frag_down(h, rows, N // 2), clamped(t[:, :, 0], t[:, :, 1], limit, 1.5, 0.75).reshape(rows, -1), eight_bits=True)
    # rows ahead of the gated outputs
    for split in (32, N // 2 // 32 * 32):
        r.go(xd, out=SPLIT_GATED, h=h.p, h_kt=(N - split) // 64 + 1, n_split=split, y_f32=y.p, ldy=split, limit=0.6, slope=2.0, up_bias=1.0)
        r.close(y.to_host((rows, split)), want[:, :split])
        u = want[:, split:].reshape(rows, -1, 2, 16)
        got = r.frag_down(h, rows, ((N - split) // 64 + 1) * 32)[:, :(N - split) // 2]
        r.close(got, clamped(u[:, :, 0], u[:, :, 1], 0.6, 2.0, 1.0).reshape(rows, -1), eight_bits=True)
    # those rows with a bias and an activation, the gated outputs behind three input tiles of a wider operand
    split, silu, tiles = N // 2 // 32 * 32, 27, (N - N // 2 // 32 * 32) // 64 + 4
    bias = np.pad(r.rng.standard_normal(split).astype(np.float32), (0, N - split), constant_values=np.nan)
    bd, wide = hipattn.DeviceBuffer.from_host(bias), hipattn.DeviceBuffer.from_host(np.full((-(-rows // 16) * 16, tiles * 32), 3.0, np.float32))
    r.go(xd, out=SPLIT_GATED, h=wide.p, h_kt=tiles, h_kt0=3, n_split=split, y_f32=y.p, ldy=split, bias=bd.p, silu_end=silu)
    v = want[:, :split] + bias[:split]
    r.close(y.to_host((rows, split)), np.concatenate([O.silu(v[:, :silu]), v[:, silu:]], axis=1))
    got, u = r.frag_down(wide, rows, tiles * 32), want[:, split:].reshape(rows, -1, 2, 16)
    r.close(got[:, 96:96 + (N - split) // 2], (O.silu(u[:, :, 0]) * u[:, :, 1]).reshape(rows, -1), eight_bits=True)
    blank = 3.0 if f32 else O.bf16_to_f32(np.full(2, 3.0, np.float32).view(np.uint16)[1::2])[0]
    assert set(np.unique(got[:, :96])) <= {blank, np.float32(0)}
    r.end()
    for b in (y, xd, h, bd, wide):
        b.free()


@pytest.mark.parametrize("f32", [False, True])
@pytest.mark.parametrize("batch,N,K,rows", [(3, 64, 32, 1), (5, 32, 96, 40), (40, 512, 64, 300), (2, 128, 64, 130), (4, 1040, 352, 300), (8, 528, 64, 500), (2, 2080, 352, 700),
                                            (6, 1040, 96, 300)])
def test_batch_of_matrices(lib, f32, batch, N, K, rows):
    # matrix z takes its own input columns and writes its own output columns
    r = Run(lib, f32, batch, N, K, rows)
    x = r.act(rows, batch * K)
    xd = r.up(x)
    h = hipattn.DeviceBuffer(-(-rows // 16) * 16 * N * batch * (4 if f32 else 2))
    r.go(xd, x_kt=batch * K // 32, x_kt_z=K // 32, out=FRAG, h=h.p, h_kt=batch * N // 32, col_z=N)
    want = np.einsum("rzk,znk->rzn", x.reshape(rows, batch, K).astype(np.float64), r.w.astype(np.float64)).reshape(rows, -1)
    r.close(r.frag_down(h, rows, batch * N), want, eight_bits=True)
    # and to columns of shared 32-bit rows, from inputs that start further in
    x = r.act(rows, (batch + 1) * K)
    xd2, y = r.up(x), hipattn.DeviceBuffer(rows * batch * N * 4)
    r.go(xd2, x_kt=(batch + 1) * K // 32, x_kt_z=K // 32, x_kt0=K // 32, out=ROWS_F32, y_f32=y.p, ldy=batch * N, col_z=N)
    x = x.reshape(rows, batch + 1, K)[:, 1:]
    r.close(y.to_host((rows, batch * N)), np.einsum("rzk,znk->rzn", x.astype(np.float64), r.w.astype(np.float64)).reshape(rows, -1))
    r.end()
    for b in (xd, xd2, h, y):
        b.free()


# whose tiles an XCD takes side by side, and beside them inputs and batches for which it does not: launches of fewer workgroups than XCDs, of a few more, of many and a rest; one tile to
# a workgroup, two, two workgroups to a tile, batches
@pytest.mark.parametrize("batch,N,K,rows", [(1, 16, 1024, 1), (1, 144, 1024, 16), (1, 6160, 1024, 9), (1, 14416, 2048, 16), (1, 48, 4096, 3), (1, 1104, 4096, 2),
                                            (3, 2064, 1024, 5), (3, 2064, 2048, 16), (8, 1040, 4096, 7), (16, 512, 2048, 16), (1, 4112, 3072, 16)])
def test_tiles_by_region(lib, batch, N, K, rows):
    r = Run(lib, False, batch, N, K, rows)
    x = r.act(rows, batch * K)
    xd, y = r.up(x), hipattn.DeviceBuffer(rows * batch * N * 4)
    r.go(xd, x_kt=batch * K // 32, x_kt_z=K // 32, out=ROWS_F32, y_f32=y.p, ldy=batch * N, col_z=N)
    want = np.stack([x.reshape(rows, batch, K)[:, z].astype(np.float64) @ r.w[z].T.astype(np.float64) for z in range(batch)], 1)
    r.close(y.to_host((rows, batch * N)), want.reshape(rows, -1))
    r.end()
    for b in (xd, y):
        b.free()


# (batch, outputs, small one's outputs and inputs, rows): one launch where both are of sixteen rows at most and the second is small; else two.
# Inputs a multiple of 1024 wide: the launch's items by region, of a multiple of eight workgroups and not, of eight and of four waves; odd
# numbers of the small one's tiles; small ones that alone are two workgroups' or would be in tiles of two; a gated first.
@pytest.mark.parametrize("f32", [False, True])
@pytest.mark.parametrize("batch,N,K,n,k,rows,gated", [(4, 1536, 288, 64, 288, 16, 0), (1, 6144, 512, 16, 96, 1, 0), (3, 2064, 1056, 48, 2048, 7, 0),
                                                      (2, 3088, 2080, 32, 4128, 5, 0), (4, 1536, 288, 64, 2080, 9, 0), (4, 1536, 256, 64, 288, 3, 0),
                                                      (4, 1520, 288, 64, 288, 16, 0), (4, 1536, 288, 400, 288, 16, 0), (4, 1536, 288, 64, 288, 17, 0),
                                                      (4, 2048, 2048, 64, 2048, 16, 0), (4, 1552, 1024, 48, 1024, 13, 0), (3, 2064, 1024, 16, 2080, 16, 0),
                                                      (2, 3088, 3072, 80, 3072, 6, 0), (1, 6160, 4096, 32, 2048, 16, 0), (1, 6160, 1024, 32, 4096, 16, 0),
                                                      (1, 2048, 1024, 64, 1024, 9, 1), (1, 2048, 4096, 64, 2080, 16, 1), (1, 2048, 1056, 16, 1056, 1, 1)])
def test_two_products(lib, f32, batch, N, K, n, k, rows, gated):
    lib.wr_hip_mix_gemm_run_two.argtypes = [C.c_int, C.POINTER(Gemm), C.POINTER(Gemm)]
    r, q = Run(lib, f32, batch, N, K, rows), Run(lib, f32, 1, n, k, rows, seed=1)
    x, u = r.act(rows, batch * K), q.act(rows, k)
    xd, ud = r.up(x), q.up(u)
    first = -(-rows // 16) * 16 * N // 2 * (4 if f32 else 2) if gated else rows * batch * N * 4
    second = -(-rows // 16) * 16 * (n + 31) // 32 * 32 * (4 if f32 else 2)
    y, h, y2, h2 = [hipattn.DeviceBuffer.from_host(np.full(size, 7, np.uint8)) for size in (first, second) * 2]

    def pair(y, h):
        a = Gemm(w=r.h, x=xd.p, x_kt=batch * K // 32, x_kt_z=K // 32, rows=rows, out=ROWS_F32, y_f32=y.p, ldy=batch * N, col_z=N)
        if gated:
            a = Gemm(w=r.h, x=xd.p, x_kt=K // 32, rows=rows, out=GATED, h=y.p, h_kt=N // 64)
        return a, Gemm(w=q.h, x=ud.p, x_kt=k // 32, rows=rows, out=FRAG, h=h.p, h_kt=(n + 31) // 32, tanh_end=n)

    for which in (0, 1):                                   # refused whole, whichever of the two it is
        bad = pair(y, h)
        bad[which].rows = 0
        assert lib.wr_hip_mix_gemm_run_two(int(f32), C.byref(bad[0]), C.byref(bad[1])) == hipattn.ERR_INVAL
        hipattn.sync()
        assert (y.to_host((first,), np.uint8) == 7).all() and (h.to_host((second,), np.uint8) == 7).all()
    a, b = pair(y, h)
    assert lib.wr_hip_mix_gemm_run_two(int(f32), C.byref(a), C.byref(b)) == 0
    hipattn.sync()
    want = np.stack([x.reshape(rows, batch, K)[:, z].astype(np.float64) @ r.w[z].T.astype(np.float64) for z in range(batch)], 1).reshape(rows, -1)
    if gated:
        t = want.reshape(rows, N // 32, 2, 16)
        r.close(r.frag_down(y, rows, N // 2), (O.silu(t[:, :, 0]) * t[:, :, 1]).reshape(rows, -1), eight_bits=True)
    else:
        r.close(y.to_host((rows, batch * N)), want)
    q.close(q.frag_down(h, rows, (n + 31) // 32 * 32)[:, :n], np.tanh(u.astype(np.float64) @ q.w[0].T.astype(np.float64)), eight_bits=True)
    for g in pair(y2, h2):                                 # the bits of two calls
        assert lib.wr_hip_mix_gemm_run(int(f32), C.byref(g)) == 0
    hipattn.sync()
    assert np.array_equal(y.to_host((first,), np.uint8), y2.to_host((first,), np.uint8))
    assert np.array_equal(h.to_host((second,), np.uint8), h2.to_host((second,), np.uint8))
    r.end(), q.end()
    for d in (xd, ud, y, h, y2, h2):
        d.free()


# ... in tiles of 256 outputs by 128 and 256 rows, the matrices on all XCDs and on one each (batches of 16 and more that eight divides)
@pytest.mark.parametrize("batch,N,K,rows", [(2, 7584, 2080, 400), (4, 7712, 2080, 130), (8, 4000, 2080, 130), (3, 6688, 2080, 280),
                                            (2, 7328, 1056, 910), (4, 7328, 1056, 400), (8, 7584, 1056, 130), (3, 6560, 1056, 670),
                                            (16, 1952, 2080, 200), (24, 1952, 1056, 400), (20, 1952, 1056, 200)])
def test_batch_of_matrices_in_wide_tiles(lib, batch, N, K, rows):
    r = Run(lib, False, batch, N, K, rows)
    x = r.act(rows, (batch + 1) * K)
    xd, h = r.up(x), hipattn.DeviceBuffer(-(-rows // 16) * 16 * N * batch * 2)
    y = hipattn.DeviceBuffer(rows * batch * N * 4)
    place = dict(x_kt=(batch + 1) * K // 32, x_kt_z=K // 32, x_kt0=K // 32, col_z=N)
    want = np.concatenate([x[:, (z + 1) * K:(z + 2) * K].astype(np.float64) @ r.w[z].T.astype(np.float64) for z in range(batch)], axis=1)
    r.go(xd, out=FRAG, h=h.p, h_kt=batch * N // 32, **place)
    r.close(r.frag_down(h, rows, batch * N), want, eight_bits=True)
    r.go(xd, out=ROWS_F32, y_f32=y.p, ldy=batch * N, **place)
    r.close(y.to_host((rows, batch * N)), want)
    r.end()
    for b in (xd, h, y):
        b.free()


# every tile the rule picks among: register tiles of 1 x 1, 1 x 2, 2 x 1 (gated outputs), 2 x 2, 2 x 3, 2 x 4, 4 x 3, 4 x 4 (outputs x rows,
# sixteens; gated outputs take even ones), LDS tiles of 64, 128 and 256 rows.  Input ranges that leave waves without
# k-steps (96), that are less than a turn of eight and a turn and a rest of four (800), and that split unevenly with
# a rest behind whole turns (1056), and two that two sets of waves halve, an
# odd number of k-steps each and an even one (2112, 2176; tiles of 64 and 128 rows).
@pytest.mark.parametrize("N,rows,K", [(n, r, k) for n, r in [(48, 17), (512, 64), (1088, 50), (1088, 130), (2112, 100), (2816, 100),
                                                             (2112, 300), (6208, 100), (6208, 511), (12352, 511),
                                                             (12352, 700)] for k in (96, 800, 1056)] +
                         [(2112, 700, 2112), (2112, 1100, 2112), (2112, 1100, 2176), (2112, 700, 2176)])
def test_every_tile_of_many_rows(lib, N, K, rows):
    r = Run(lib, False, 1, N, K, rows)
    x = r.act(rows, K)
    xd, y = r.up(x), hipattn.DeviceBuffer(rows * N * 4)
    want = x.astype(np.float64) @ r.w[0].T.astype(np.float64)
    r.go(xd, out=ROWS_F32, y_f32=y.p, ldy=N)
    r.close(y.to_host((rows, N)), want)
    if N % 64 == 0:
        h = hipattn.DeviceBuffer(-(-rows // 16) * 16 * N)
        r.go(xd, out=GATED, h=h.p, h_kt=N // 64)
        t = want.reshape(rows, N // 32, 2, 16)
        r.close(r.frag_down(h, rows, N // 2), (O.silu(t[:, :, 0]) * t[:, :, 1]).reshape(rows, -1), eight_bits=True)
        h.free()
    r.end()
    for b in (xd, y):
        b.free()


# tiles of 256 outputs by 256 and 128 rows: odd and even numbers of k-steps, a last tile of outputs that is not full, gated and not
@pytest.mark.parametrize("N,rows,K", [(32768 + 64, 400, 1056), (16384 + 64, 1000, 2048), (4144, 1800, 2080), (4096 + 64, 2047, 4160)])
def test_pipelined_tiles_of_many_rows(lib, N, rows, K):
    r = Run(lib, False, 1, N, K, rows)
    x = r.act(rows, K)
    xd, y = r.up(x), hipattn.DeviceBuffer(rows * N * 4)
    r.go(xd, out=ROWS_F32, y_f32=y.p, ldy=N)
    want = x.astype(np.float64) @ r.w[0].T.astype(np.float64)
    r.close(y.to_host((rows, N)), want)
    if N % 64 == 0:
        h = hipattn.DeviceBuffer(-(-rows // 16) * 16 * N)
        r.go(xd, out=GATED, h=h.p, h_kt=N // 64)
        t = want.reshape(rows, N // 32, 2, 16)
        r.close(r.frag_down(h, rows, N // 2), (O.silu(t[:, :, 0]) * t[:, :, 1]).reshape(rows, -1), eight_bits=True)
        h.free()
    r.end()
    for b in (xd, y):
        b.free()


@pytest.mark.parametrize("N,K", [(16, 4096), (2048, 4128), (80, 8192), (2064, 4096), (48, 4064)])
def test_two_workgroups_to_a_tile(lib, N, K):
    # narrow weights over long inputs, up to sixteen rows: one tile, as many as a launch holds, an odd number of k-steps;
    # one tile more and one k-step less, which a single workgroup takes.  A row's bits are its own whatever rows go with
    # it and whichever workgroup is last, sixteen launches over; every destination (gated outputs take no such tile), with
    # bias, activations and a factor.
    r = Run(lib, False, 1, N, K, 16)
    x = r.act(16, K)
    xd, y, y1 = r.up(x), hipattn.DeviceBuffer(16 * N * 4), hipattn.DeviceBuffer(N * 4)
    want = x.astype(np.float64) @ r.w[0].T.astype(np.float64)
    r.go(xd, out=ROWS_F32, y_f32=y.p, ldy=N)
    got = y.to_host((16, N))
    r.close(got, want)
    for i in range(16):
        one = r.up(x[i:i + 1])
        r.go(one, rows=1, out=ROWS_F32, y_f32=y1.p, ldy=N)
        assert y1.to_host((N,)).tobytes() == got[i].tobytes(), f"row {i}"
        one.free()
    if N % 32 == 0:
        h = hipattn.DeviceBuffer(16 * N * 2)
        r.go(xd, out=FRAG, h=h.p, h_kt=N // 32, relu2=1)
        r.close(r.frag_down(h, 16, N), np.maximum(want, 0) ** 2, eight_bits=True)
        split = N // 2 // 32 * 32
        r.go(xd, out=SPLIT, h=h.p, h_kt=split // 32, n_split=split, y_f32=y.p, ldy=N - split)
        r.close(r.frag_down(h, 16, split), want[:, :split], eight_bits=True)
        r.close(y.to_host((16, N - split)), want[:, split:])
        h.free()
    bias = r.rng.standard_normal(N).astype(np.float32)
    bd, ya, ld = hipattn.DeviceBuffer.from_host(bias), hipattn.DeviceBuffer(16 * (N + 8) * 2), N + 8
    r.go(xd, out=ROWS, y_act=ya.p, ldy=ld, bias=bd.p, silu_end=N // 3, scale=0.5)
    v = want + bias
    got = O.bf16_to_f32(ya.to_host((16 * ld // 2,)).view(np.uint16)).reshape(16, ld)[:, :N]
    r.close(got, 0.5 * np.concatenate([O.silu(v[:, :N // 3]), v[:, N // 3:]], axis=1), eight_bits=True)
    r.go(xd, out=ROWS_F32, y_f32=y.p, ldy=N, bias=bd.p, silu_end=N // 4, tanh_end=N - 7)
    v = np.concatenate([O.silu(v[:, :N // 4]), np.tanh(v[:, N // 4:N - 7]), v[:, N - 7:]], axis=1)
    r.close(y.to_host((16, N)), v)
    r.end()
    for b in (xd, y, y1, bd, ya):
        b.free()


@pytest.mark.parametrize("N,K,runs_each,spare,experts", [
    (64, 352, 1, 1, 3), (2080, 96, 1, 1, 3),                   # few rows an expert: a stream of the weights
    (64, 352, 1, 0, 3), (2080, 96, 1, 0, 3),                   # as many runs as experts, tiles of 128 rows
    (64, 352, 3, 0, 3), (2080, 96, 3, 0, 3), (1056, 32, 2, 0, 3), (64, 352, 2, 0, 3),    # ... and more than that
    (144, 2080, 1, 1, 60), (144, 2016, 1, 1, 60),              # narrow weights, a tile to a CU; one input tile fewer
])
def test_runs_whose_last_groups_hold_no_pair(lib, N, K, runs_each, spare, experts):
    # runs of eight groups per expert, the last one's rest and whole runs behind them empty, as routing leaves them
    r = Run(lib, False, experts, N, K, 0)
    which = np.full(8 * (experts * runs_each + spare), -1, dtype=np.int32)
    for e in range(experts):
        n = 8 * (runs_each - 1) + (1, 4, 7)[e % 3]         # groups that hold pairs
        which[8 * runs_each * e:8 * runs_each * e + n] = e
    rows, live = 16 * len(which), np.repeat(which, 16) >= 0
    x = r.act(rows, K)
    xd, gd = r.up(x), hipattn.DeviceBuffer.from_host(which.view(np.float32))
    y = hipattn.DeviceBuffer(rows * N * 4)
    r.go(xd, rows=rows, group_expert=gd.p, tile_groups=8, out=ROWS_F32, y_f32=y.p, ldy=N)
    want = np.concatenate([x[16 * g:16 * g + 16].astype(np.float64) @ r.w[e].T.astype(np.float64) for g, e in enumerate(which) if e >= 0])
    r.close(y.to_host((rows, N))[live], want)
    r.end()
    for b in (xd, gd, y):
        b.free()


# up to 48, 64 and 80 rows an expert; runs by XCD or not; tiles beyond
@pytest.mark.parametrize("experts,spare", [(8, 3), (8, 4), (15, 5), (15, 6), (20, 7), (20, 10)])
@pytest.mark.parametrize("N,K", [(64, 1024), (64, 1056), (1536, 544), (1568, 544), (96, 64), (32, 2080), (2048, 544)])
def test_runs_of_every_length(lib, experts, spare, N, K):
    # a run of one to eight groups with rows: workgroups of four and of eight groups, an XCD to a run and runs dealt out
    r = Run(lib, False, experts, N, K, 0)
    runs = experts + spare
    which = np.full(8 * runs, -1, dtype=np.int32)
    for e in range(experts):
        which[8 * e:8 * e + 1 + (5 * e) % 8] = e
    rows, live = 16 * len(which), np.repeat(which, 16) >= 0
    x = r.act(rows, K)
    xd, gd = r.up(x), hipattn.DeviceBuffer.from_host(which.view(np.float32))
    y, h = hipattn.DeviceBuffer(rows * N * 4), hipattn.DeviceBuffer(rows * (N // 32 * 16 + 32) * 2)
    r.go(xd, rows=rows, group_expert=gd.p, tile_groups=8, out=ROWS_F32, y_f32=y.p, ldy=N)
    want = np.concatenate([x[16 * g:16 * g + 16].astype(np.float64) @ r.w[e].T.astype(np.float64) for g, e in enumerate(which) if e >= 0])
    r.close(y.to_host((rows, N))[live], want)
    factor = r.rng.uniform(0, 2, rows).astype(np.float32)
    fd = hipattn.DeviceBuffer.from_host(factor)
    if N % 64 == 0:
        r.go(xd, rows=rows, group_expert=gd.p, tile_groups=8, out=GATED, h=h.p, h_kt=N // 64, x_scale=fd.p)
        t = (want * factor[live][:, None]).reshape(len(want), N // 32, 2, 16)
        r.close(r.frag_down(h, rows, N // 2)[live], (O.silu(t[:, :, 0]) * t[:, :, 1]).reshape(len(want), -1), eight_bits=True)
    r.end()
    for b in (xd, gd, y, h, fd):
        b.free()


@pytest.mark.parametrize("N,K", [(1024, 544), (1040, 96), (512, 32), (1024, 512), (528, 2080)])
def test_groups_of_an_expert_that_stand_together(lib, N, K):
    # single groups in any order, a negative one among them; rows in order and picked one by one, of inputs that are the
    # whole of their rows (brought together first) and of a part: each group's bits are those of the group by itself
    experts = 5
    r = Run(lib, False, experts, N, K, 0)
    which = np.array([0] * 9 + [1, -1, 1, 1, 3, 2, 2, 2] + [4] * 5 + [-1, -1, 0, 0, 3, 3, 3, 3, 4, 0, 1], dtype=np.int32)
    rows, live = 16 * len(which), np.repeat(which, 16) >= 0
    x = r.act(rows, K)
    xd, gd = r.up(x), hipattn.DeviceBuffer.from_host(which.view(np.float32))
    y, y1 = hipattn.DeviceBuffer.from_host(np.full((rows, N), 7.0, dtype=np.float32)), hipattn.DeviceBuffer(16 * N * 4)
    r.go(xd, rows=rows, group_expert=gd.p, tile_groups=1, out=ROWS_F32, y_f32=y.p, ldy=N)
    got = y.to_host((rows, N))
    want = np.concatenate([x[16 * g:16 * g + 16].astype(np.float64) @ r.w[e].T.astype(np.float64) for g, e in enumerate(which) if e >= 0])
    r.close(got[live], want)
    assert np.all(got[~live] == 7.0)
    for g, e in enumerate(which):
        if e < 0:
            continue
        one, ed = r.up(x[16 * g:16 * g + 16]), hipattn.DeviceBuffer.from_host(np.array([e], dtype=np.int32).view(np.float32))
        r.go(one, rows=16, group_expert=ed.p, tile_groups=1, out=ROWS_F32, y_f32=y1.p, ldy=N)
        assert y1.to_host((16, N)).tobytes() == got[16 * g:16 * g + 16].tobytes(), f"group {g}"
        one.free()
        ed.free()
    pick = r.rng.integers(0, 37, rows).astype(np.uint32)
    used = r.rng.random(rows) < 0.8
    pd = hipattn.DeviceBuffer.from_host(np.where(used, pick, np.uint32(0xFFFFFFFF)).astype(np.uint32).view(np.float32))
    few = r.act(37, K + 64)
    fd, whole = r.up(few), r.up(np.ascontiguousarray(few[:, 32:32 + K]))
    seen = live & used
    want = np.concatenate([few[pick[16 * g:16 * g + 16], 32:32 + K].astype(np.float64) @ r.w[max(e, 0)].T.astype(np.float64)
                           for g, e in enumerate(which)])[seen]
    r.go(whole, rows=rows, group_expert=gd.p, tile_groups=1, out=ROWS_F32, y_f32=y.p, ldy=N, x_perm=pd.p)
    got = y.to_host((rows, N))
    r.close(got[seen], want)
    assert np.all(got[~live] == 7.0)
    r.go(fd, rows=rows, group_expert=gd.p, tile_groups=1, out=ROWS_F32, y_f32=y.p, ldy=N, x_perm=pd.p, x_kt=K // 32 + 2, x_kt0=1)
    assert y.to_host((rows, N))[seen].tobytes() == got[seen].tobytes()
    r.end()
    for b in (xd, gd, y, y1, pd, fd, whole):
        b.free()


# weights of 64 MiB and more, a workgroup to eight (sixteen) tiles of an expert's outputs: k-steps and tiles that do and do
# not fill the last workgroup's turns, experts without rows, more runs or groups than a wave has lanes
LARGE = [(64, 1024, 512), (64, 1040, 544), (40, 1168, 800)]


@pytest.mark.parametrize("spare", [32, 64])
@pytest.mark.parametrize("experts,N,K", LARGE)
def test_large_experts_in_runs(lib, experts, N, K, spare):
    r = Run(lib, False, experts, N, K, 0)
    which = np.full((experts + spare, 8), -1, dtype=np.int32)
    for i in range(experts + 3):
        e = i if i < experts else i - experts                  # (three experts have a second run)
        if e % 9 != 4:
            which[i, :1 + (5 * i) % 8] = e
    which = which.reshape(-1)
    rows, live = 16 * len(which), np.repeat(which, 16) >= 0
    x = r.act(rows, K)
    xd, gd = r.up(x), hipattn.DeviceBuffer.from_host(which.view(np.float32))
    y, h = hipattn.DeviceBuffer.from_host(np.full((rows, N), 7.0, dtype=np.float32)), hipattn.DeviceBuffer(rows * (N // 32 * 16 + 32) * 2)
    r.go(xd, rows=rows, group_expert=gd.p, tile_groups=8, out=ROWS_F32, y_f32=y.p, ldy=N)
    want = np.concatenate([x[16 * g:16 * g + 16].astype(np.float64) @ r.w[e].T.astype(np.float64) for g, e in enumerate(which) if e >= 0])
    got = y.to_host((rows, N))
    r.close(got[live], want)
    assert np.all(got[np.repeat(which[::8], 128) < 0] == 7.0)      # (tiles write a run's empty groups too)
    if N % 64 == 0:
        factor = r.rng.uniform(0, 2, rows).astype(np.float32)
        fd = hipattn.DeviceBuffer.from_host(factor)
        r.go(xd, rows=rows, group_expert=gd.p, tile_groups=8, out=GATED, h=h.p, h_kt=N // 64, x_scale=fd.p)
        t = (want * factor[live][:, None]).reshape(len(want), N // 32, 2, 16)
        r.close(r.frag_down(h, rows, N // 2)[live], (O.silu(t[:, :, 0]) * t[:, :, 1]).reshape(len(want), -1), eight_bits=True)
        fd.free()
    r.end()
    for b in (xd, gd, y, h):
        b.free()


# the most runs that the stream takes, one more and twice as many: the rows are in the first runs and the last
@pytest.mark.parametrize("experts,N,K,runs", [(150, 512, 544, 256), (150, 512, 544, 257), (64, 1024, 544, 256), (64, 1024, 544, 257),
                                              (64, 1024, 544, 512), (64, 1024, 544, 513)])
def test_large_experts_in_many_runs(lib, experts, N, K, runs):
    r = Run(lib, False, experts, N, K, 0)
    which = np.full((runs, 8), -1, dtype=np.int32)
    for i in range(runs):
        if i < 3 or i >= runs - 60:
            which[i, :1 + (5 * i) % 8] = 7 * i % experts
    which = which.reshape(-1)
    rows, live = 16 * len(which), np.repeat(which, 16) >= 0
    x = r.act(rows, K)
    xd, gd = r.up(x), hipattn.DeviceBuffer.from_host(which.view(np.float32))
    y = hipattn.DeviceBuffer.from_host(np.full((rows, N), 7.0, dtype=np.float32))
    r.go(xd, rows=rows, group_expert=gd.p, tile_groups=8, out=ROWS_F32, y_f32=y.p, ldy=N)
    got = y.to_host((rows, N))
    r.close(got[live], np.concatenate([x[16 * g:16 * g + 16].astype(np.float64) @ r.w[e].T.astype(np.float64) for g, e in enumerate(which) if e >= 0]))
    assert np.all(got[np.repeat(which[::8], 128) < 0] == 7.0)
    r.end()
    for b in (xd, gd, y):
        b.free()


@pytest.mark.parametrize("order", ["together", "scattered"])
@pytest.mark.parametrize("experts,N,K", LARGE)
def test_large_experts_in_single_groups(lib, experts, N, K, order):
    # an expert's groups one after the other, up to nineteen, with gaps; and in an order that gives a piece to every group
    r = Run(lib, False, experts, N, K, 0)
    if order == "together":
        which = np.concatenate([np.repeat(e, (3, 1, 8, 0, 19, 2, 9)[e % 7]) for e in range(experts)] + [[-1, -1, 0, 0, 5, -1]])
        which[10] = -1
    else:
        which = np.arange(3 * experts) * 7 % experts
    which = which.astype(np.int32)
    rows, live = 16 * len(which), np.repeat(which, 16) >= 0
    x = r.act(rows, K)
    xd, gd = r.up(x), hipattn.DeviceBuffer.from_host(which.view(np.float32))
    y = hipattn.DeviceBuffer.from_host(np.full((rows, N), 7.0, dtype=np.float32))
    r.go(xd, rows=rows, group_expert=gd.p, tile_groups=1, out=ROWS_F32, y_f32=y.p, ldy=N)
    got = y.to_host((rows, N))
    r.close(got[live], np.concatenate([x[16 * g:16 * g + 16].astype(np.float64) @ r.w[e].T.astype(np.float64) for g, e in enumerate(which) if e >= 0]))
    assert np.all(got[~live] == 7.0)
    pick, used = r.rng.integers(0, 37, rows).astype(np.uint32), r.rng.random(rows) < 0.8
    pd = hipattn.DeviceBuffer.from_host(np.where(used, pick, np.uint32(0xFFFFFFFF)).astype(np.uint32).view(np.float32))
    few = r.act(37, K + 64)
    fd, seen = r.up(few), live & used
    r.go(fd, rows=rows, group_expert=gd.p, tile_groups=1, out=ROWS_F32, y_f32=y.p, ldy=N, x_perm=pd.p, x_kt=K // 32 + 2, x_kt0=1)
    got = y.to_host((rows, N))
    want = np.concatenate([few[pick[16 * g:16 * g + 16], 32:32 + K].astype(np.float64) @ r.w[max(e, 0)].T.astype(np.float64) for g, e in enumerate(which)])
    r.close(got[seen], want[seen])
    assert np.all(got[~live] == 7.0)
    r.end()
    for b in (xd, gd, y, pd, fd):
        b.free()


def test_picked_rows_of_a_recorded_product(lib):
    # A recorded product picks its rows by itself: it is one launch, none of the thread's own memory is in
    # the graph, and replays hold after a larger call has made that memory anew.
    experts, N, K = 2, 64, 64
    r = Run(lib, False, experts, N, K, 0)

    def inputs(groups):
        which = np.repeat(np.arange(experts), groups // experts).astype(np.int32)
        few = r.act(33, K)
        pick = r.rng.integers(0, 33, 16 * groups).astype(np.uint32)
        want = np.concatenate([few[pick[16 * g:16 * g + 16]].astype(np.float64) @ r.w[e].T.astype(np.float64) for g, e in enumerate(which)])
        y = hipattn.DeviceBuffer(16 * groups * N * 4)
        bufs = r.up(few), hipattn.DeviceBuffer.from_host(which.view(np.float32)), hipattn.DeviceBuffer.from_host(pick.view(np.float32)), y
        return bufs, Gemm(w=r.h, x=bufs[0].p, x_kt=K // 32, rows=16 * groups, group_expert=bufs[1].p, tile_groups=1, out=ROWS_F32,
                          y_f32=y.p, ldy=N, x_perm=bufs[2].p), want

    small, g, want = inputs(128)
    large, g2, want2 = inputs(4096)
    for _ in range(2):                                       # there is room for its rows from here on
        assert lib.wr_hip_mix_gemm_run(0, C.byref(g)) == 0
    hipattn.sync()
    eager = small[3].to_host((2048, N)).copy()
    r.close(eager, want)
    stream, graph, run, n = vp(lib.wr_hip_attn_stream()), vp(), vp(), C.c_size_t()
    assert lib.hipStreamBeginCapture(stream, 2) == 0         # relaxed
    rc = lib.wr_hip_mix_gemm_run(0, C.byref(g))
    assert lib.hipStreamEndCapture(stream, C.byref(graph)) == 0 and rc == 0
    assert lib.hipGraphGetNodes(graph, None, C.byref(n)) == 0 and n.value == 1
    assert lib.hipGraphInstantiate(C.byref(run), graph, None, None, C.c_size_t(0)) == 0
    for _ in range(3):
        assert lib.wr_hip_mix_gemm_run(0, C.byref(g2)) == 0
        hipattn.sync()
        r.close(large[3].to_host((65536, N)), want2)
        lib.wr_hip_attn_h2d(small[3].p, np.zeros((2048, N), np.float32).ctypes.data, eager.nbytes)
        assert lib.hipGraphLaunch(run, stream) == 0
        hipattn.sync()
        assert small[3].to_host((2048, N)).tobytes() == eager.tobytes()
    assert lib.hipGraphExecDestroy(run) == 0 and lib.hipGraphDestroy(graph) == 0
    r.end()
    for b in small + large:
        b.free()


def test_products_without_memory_for_picked_rows(lib):
    # The memory is optional: one refusal is one warning, the products after it do not ask again, and all are whole.
    experts, N, K, groups = 2, 64, 1024, 2048                 # 64 MiB of picked rows: more than any call before had
    r = Run(lib, False, experts, N, K, 0)
    which = np.repeat(np.arange(experts), groups // experts).astype(np.int32)
    few = r.act(33, K)
    pick = r.rng.integers(0, 33, 16 * groups).astype(np.uint32)
    want = np.concatenate([(few.astype(np.float64) @ r.w[e].T.astype(np.float64))[pick[which.repeat(16) == e]] for e in range(experts)])
    xd, gd, pd = r.up(few), hipattn.DeviceBuffer.from_host(which.view(np.float32)), hipattn.DeviceBuffer.from_host(pick.view(np.float32))
    y, said = hipattn.DeviceBuffer(16 * groups * N * 4), []
    log = C.CFUNCTYPE(None, C.c_int, C.c_char_p, vp)(lambda level, line, user: said.append((level, line)))
    lib.wr_hip_attn_set_log(log, None)
    lib.wr_hip_attn_set_alloc_failures(1000, 0)
    try:
        for call in range(6):
            if call == 3:
                lib.wr_hip_attn_set_alloc_failures(0, 0)
            r.go(xd, rows=16 * groups, group_expert=gd.p, tile_groups=1, out=ROWS_F32, y_f32=y.p, ldy=N, x_perm=pd.p)
            r.close(y.to_host((16 * groups, N)), want)
    finally:
        lib.wr_hip_attn_set_alloc_failures(0, 0)
        lib.wr_hip_attn_set_log(C.cast(None, type(log)), None)
    assert [level for level, _ in said] == [1] and b"picked rows" in said[0][1], said
    r.end()
    for b in (xd, gd, pd, y):
        b.free()


@pytest.mark.parametrize("f32", [False, True])
@pytest.mark.parametrize("N,K,tile", [(64, 96, 1), (48, 64, 8), (4096, 64, 8), (1024, 32, 1)])
def test_matrix_per_row_group(lib, f32, N, K, tile):
    experts = 4
    r = Run(lib, f32, experts, N, K, 0)
    which = np.repeat(np.array([2, 0, -1, 3, 2], dtype=np.int32), tile)
    rows = 16 * len(which)
    x = r.act(rows, K)
    xd, gd = r.up(x), hipattn.DeviceBuffer.from_host(which.view(np.float32))
    y = hipattn.DeviceBuffer.from_host(np.full((rows, N), 7.0, dtype=np.float32))
    r.go(xd, rows=rows, group_expert=gd.p, tile_groups=tile, out=ROWS_F32, y_f32=y.p, ldy=N)
    want = np.full((rows, N), 7.0)                          # groups nobody uses stay as they are
    for g, e in enumerate(which):
        if e >= 0:
            want[16 * g:16 * g + 16] = x[16 * g:16 * g + 16].astype(np.float64) @ r.w[e].T.astype(np.float64)
    r.close(y.to_host((rows, N)), want)
    # a factor per row, ahead of the gated units
    factor = r.rng.uniform(0, 2, rows).astype(np.float32)
    fd, h = hipattn.DeviceBuffer.from_host(factor), hipattn.DeviceBuffer(rows * (N // 32 * 16 + 32) * 4)
    if N % 64 == 0:
        r.go(xd, rows=rows, group_expert=gd.p, tile_groups=tile, out=GATED, h=h.p, h_kt=N // 64, x_scale=fd.p)
        t = (np.where(np.repeat(which, 16)[:, None] >= 0, want, 0) * factor[:, None]).reshape(rows, N // 32, 2, 16)
        live = np.repeat(which, 16) >= 0
        r.close(r.frag_down(h, rows, N // 2)[live], (O.silu(t[:, :, 0]) * t[:, :, 1]).reshape(rows, -1)[live], eight_bits=True)
    for b in (fd, h):
        b.free()
    if tile == 1:                                          # rows picked one by one out of fewer
        pick = r.rng.integers(0, 21, rows).astype(np.uint32)
        used = r.rng.random(rows) < 0.8
        few = r.act(21, K)
        fd = r.up(few)
        pd = hipattn.DeviceBuffer.from_host(np.where(used, pick, np.uint32(0xFFFFFFFF)).astype(np.uint32).view(np.float32))
        r.go(fd, rows=rows, group_expert=gd.p, tile_groups=1, out=ROWS_F32, y_f32=y.p, ldy=N, x_perm=pd.p)
        got = y.to_host((rows, N))
        for g, e in enumerate(which):
            for i in range(16 * g, 16 * g + 16):
                if e >= 0 and used[i]:
                    r.close(got[i], few[pick[i]].astype(np.float64) @ r.w[e].T.astype(np.float64))
        for b in (fd, pd):
            b.free()
    r.end()
    for b in (xd, gd, y):
        b.free()


class Resid(C.Structure):
    _fields_ = [("width", u32), ("eps", C.c_float), ("x", vp), ("y", vp), ("post", vp), ("add", vp), ("next", vp), ("gate", vp),
                ("slot", vp), ("top", u32), ("wanted", u32), ("h", vp), ("side", vp), ("ident", vp), ("shared", vp),
                ("pair_y", vp * 2), ("pair_post", vp * 2)]


class Seq(C.Structure):
    _fields_ = [("rows", u32), ("pos0", u32), ("slot", u32), ("buf_in", u32), ("buf_out", u32), ("n_pages", u32), ("pages", C.POINTER(u32))]


class StepOf:
    """A step of one request with these tokens."""

    def __init__(self, lib, tokens, vocab):
        pages = -(-len(tokens) // 64)
        lib.wr_hip_mix_pool_destroy.argtypes = lib.wr_hip_mix_step_destroy.argtypes = [vp]
        lib.wr_hip_mix_residual.argtypes = [vp, C.c_int, C.POINTER(Resid)]
        lib.wr_hip_mix_embed.argtypes = [vp, C.c_int, vp, u32, vp, C.c_float, C.c_float, vp, vp, vp, vp]
        self.lib, self.pool, self.h = lib, vp(), vp()
        assert lib.wr_hip_mix_pool_create(0, 1, (u32 * 1)(32), pages, 0, None, 1, C.byref(self.pool)) == 0
        assert lib.wr_hip_mix_step_create(pages, C.byref(self.h)) == 0
        seq = Seq(len(tokens), 0, 0, 0, 1, pages, (u32 * pages)(*range(pages)))
        assert lib.wr_hip_mix_step_set(self.h, self.pool, 1, C.byref(seq), (u32 * len(tokens))(*tokens), vocab, 0, None) == 0

    def end(self):
        hipattn.sync()
        self.lib.wr_hip_mix_step_destroy(self.h)
        self.lib.wr_hip_mix_pool_destroy(self.pool)


class Router(C.Structure):
    _fields_ = [("experts", u32), ("identity", u32), ("top", u32), ("groups", u32), ("keep", u32), ("softmax_all", u32), ("shared_gate", u32),
                ("scale", C.c_float), ("correction", vp), ("logistic", u32)]


# The choice with the order up to 32 rows, up to 64 where few are chosen of few, and before it beyond; pairs one by one and, past 2048, eight at a time: of whole turns of eight
# thousand, two less, one more, and of two turns and a rest; outputs a lane
# holds one, four and sixteen of; identity outputs; runs of one group and of eight.
@pytest.mark.parametrize("experts,identity,top,rows,run", [(64, 0, 6, 1, 1), (64, 0, 6, 32, 1), (64, 0, 6, 33, 1), (64, 0, 6, 64, 8), (64, 0, 1, 64, 1), (64, 0, 2, 40, 1), (64, 0, 2, 41, 1),
                                                           (100, 28, 1, 48, 1), (100, 28, 1, 49, 8), (64, 0, 8, 256, 1), (64, 0, 8, 257, 1), (60, 4, 2, 4095, 8),
                                                           (60, 0, 2, 4096, 8), (64, 0, 3, 2731, 8), (64, 0, 6, 2800, 8), (120, 8, 5, 40, 1), (300, 12, 9, 32, 2),
                                                           (300, 12, 9, 33, 2), (1000, 24, 64, 257, 1)])
def test_routes(lib, experts, identity, top, rows, run):
    lib.wr_hip_mix_route.argtypes = [vp, vp, u32, C.POINTER(Router), u32, vp, vp, vp, vp, vp, vp]
    lib.wr_hip_mix_route_groups.restype = u32
    outputs, rng = experts + identity, np.random.default_rng(rows)
    z = rng.standard_normal((rows, outputs), dtype=np.float32)
    groups = lib.wr_hip_mix_route_groups(rows, experts, top, run)
    s, zd = StepOf(lib, [0] * rows, 1), hipattn.DeviceBuffer.from_host(z)
    gate, side, weight, slot, perm, owner = [hipattn.DeviceBuffer.from_host(np.full(n, 7.0, np.float32))
                                             for n in (rows * top, rows * 2, groups * 16, rows * top, groups * 16, groups)]
    q = Router(experts=experts, identity=identity, top=top)
    for weighed in (weight.p, None):
        assert lib.wr_hip_mix_route(s.h, zd.p, outputs, C.byref(q), run, gate.p, side.p, weighed, slot.p, perm.p, owner.p) == 0
        hipattn.sync()
        g, at = gate.to_host((rows, top)), slot.to_host((rows, top)).view(np.uint32)
        row, expert = perm.to_host((groups * 16,)).view(np.uint32), owner.to_host((groups,)).view(np.int32)
        best = np.argsort(-z, axis=1, kind="stable")[:, :top]
        chosen = np.take_along_axis(z, best, axis=1).astype(np.float64)
        e = np.exp(chosen - chosen[:, :1])
        # differences of logits below 10 round by 2^-21; exp, the sum in turn and the quotient by a few 2^-24 each
        assert np.abs(g / (e / e.sum(axis=1, keepdims=True)) - 1).max() <= 2.0 ** -20 + (top + 8) * 2.0 ** -24
        real = best < experts
        assert (at[~real] == 0xFFFFFFFF).all() and len(set(at[real].tolist())) == real.sum()
        assert np.array_equal(row[at[real]], np.nonzero(real)[0]) and np.array_equal(expert[at[real] // 16], best[real])
        empty = np.ones(groups * 16, bool)
        empty[at[real]] = False
        assert (row[empty] == 0xFFFFFFFF).all() and (expert[empty.reshape(-1, 16).all(axis=1)] == -1).all()
        if weighed:
            w = weight.to_host((groups * 16,))
            assert np.array_equal(w[at[real]], g[real]) and not w[empty].any()
    s.end()
    for b in (zd, gate, side, weight, slot, perm, owner):
        b.free()


class Recurrence(C.Structure):
    _fields_ = [("heads", u32), ("dim", u32), ("rule", u32), ("gain", C.c_float), ("unit_eps", C.c_float), ("eps", C.c_float),
                ("out_scale", C.c_float), ("gate_silu", u32), ("w0", vp), ("u", vp), ("a_bias", vp), ("norm", vp), ("in_", vp),
                ("ld", u32), ("col_r", u32), ("col_k", u32), ("col_v", u32), ("col_a", u32), ("col_g", u32), ("w_decay", vp),
                ("low", vp), ("z", vp), ("h", vp), ("h_kt", u32), ("col_h", u32), ("vdim", u32), ("lower", vp)]


class Window(C.Structure):
    _fields_ = [("heads", u32), ("kv_heads", u32), ("dim", u32), ("dim_pad", u32), ("vdim", u32), ("vdim_pad", u32), ("rot_half", u32),
                ("window", u32), ("scale", C.c_float), ("out_scale", C.c_float), ("norm_values", u32), ("eps", C.c_float), ("maps", u32),
                ("neighbours", u32), ("softcap", C.c_float), ("diff", C.c_float), ("q_norm", vp), ("k_norm", vp), ("chunk", u32),
                ("gate_wide", u32), ("turn_values", vp)]


BONUS, DELTA, FORGET = range(3)


class Recur:
    """A recurrence (and, with `win`, a windowed layer beside it) over steps of requests that bring `rows` rows each."""

    def __init__(self, lib, f32, heads, dim, rank, rows, rule=DELTA, win=None, ld=None):
        self.lib, self.f32, self.rows = lib, f32, rows
        lib.wr_hip_mix_pool_destroy.argtypes = lib.wr_hip_mix_step_destroy.argtypes = [vp]
        lib.wr_hip_mix_pool_create.argtypes = [C.c_int, u32, vp, u32, u32, vp, u32, C.POINTER(vp)]
        lib.wr_hip_mix_recur.argtypes = [vp, vp, u32, C.c_int, C.POINTER(Recurrence)]
        lib.wr_hip_mix_window_append.argtypes = [vp, vp, u32, C.c_int, C.POINTER(Window), vp, u32, u32, u32, u32, vp, vp]
        lib.wr_hip_mix_window_append_recur.argtypes = lib.wr_hip_mix_window_append.argtypes + [u32, C.POINTER(Recurrence)]
        lib.wr_hip_mix_window_attend.argtypes = [vp, vp, u32, C.c_int, C.POINTER(Window), vp, vp, vp, u32, vp, u32]
        self.step, hd, self.total = vp(), heads * dim, sum(rows)
        self.padded = -(-self.total // 16) * 16
        self.e, self.kt, wide = 4 if f32 else 2, -(-hd // 32), -(-hd // 32) * 32
        self.pages, self.bufs, self.pools = [-(-3 * n // 64) for n in rows], [], []       # (room for three such steps)
        self.dims = (u32 * 1)(win.kv_heads * (win.maps * win.dim_pad + win.vdim_pad) if win else 32)
        self.state = (C.c_uint64 * 1)(hd * dim)
        assert lib.wr_hip_mix_step_create(sum(self.pages), C.byref(self.step)) == 0
        self.win, self.ld = win, ld or 5 * wide
        rng = self.rng = np.random.default_rng(dim + rank)
        self.r = Run(lib, f32, 1, -(-hd // 16) * 16, rank, self.total)
        self.h = self.fill(self.padded * self.kt * 32 * self.e)
        self.rec = Recurrence(heads=heads, dim=dim, rule=rule, unit_eps=1e-6, eps=1e-12, out_scale=1.0, gate_silu=0, ld=self.ld,
                              col_k=wide, col_v=2 * wide, col_a=3 * wide if rule == DELTA else 0, col_g=4 * wide, w_decay=self.r.h,
                              low=self.up(self.r.act(self.total, rank)), z=self.fill(self.padded * wide * 4).p, h=self.h.p, h_kt=self.kt,
                              w0=self.put(np.full(wide, -1.0)), u=self.put(np.ones(wide)), a_bias=self.put(np.full(wide, -100.0)),
                              norm=self.put(np.ones(wide)), in_=self.put(rng.standard_normal((self.total, self.ld))))

    def keep(self, b):
        self.bufs.append(b)
        return b

    def put(self, x):
        return self.keep(hipattn.DeviceBuffer.from_host(np.asarray(x, np.float32))).p

    def up(self, x):
        return self.keep(self.r.up(x)).p

    def fill(self, n):
        return self.keep(hipattn.DeviceBuffer.from_host(np.full(n, 0x3C, np.uint8)))

    def pool(self):
        p = vp()
        assert self.lib.wr_hip_mix_pool_create(int(self.f32), 1, self.dims, sum(self.pages), 1, self.state, len(self.rows), C.byref(p)) == 0
        self.pools.append(p)
        return p

    def set(self, pool, nth=0):
        seqs, page, lists = (Seq * len(self.rows))(), 0, []
        for i, n in enumerate(self.rows):
            lists.append((u32 * self.pages[i])(*range(page, page + self.pages[i])))
            seqs[i], page = Seq(n, nth * n, i, (nth + 1) % 2, nth % 2, self.pages[i], lists[-1]), page + self.pages[i]
        assert self.lib.wr_hip_mix_step_set(self.step, pool, len(self.rows), seqs, (u32 * self.total)(), 1, 0, None) == 0

    def out(self):
        hipattn.sync()
        return self.r.frag_down(self.h, self.total, self.kt * 32)

    def end(self):
        hipattn.sync()
        self.r.end()
        self.lib.wr_hip_mix_step_destroy(self.step)
        for p in self.pools:
            self.lib.wr_hip_mix_pool_destroy(p)
        for b in self.bufs:
            b.free()


# A decoded token's decays: one sum in the order of the low-rank product's outputs, over one to four tiles of them and whatever head size, as
# the rest of its tile and the next tiles lose a one beside 2^24 and what is added tile by tile does not.
@pytest.mark.parametrize("f32", [False, True])
@pytest.mark.parametrize("rule", [BONUS, DELTA])
@pytest.mark.parametrize("tiles", [1, 2, 3, 4])
@pytest.mark.parametrize("dim", [16, 30, 64, 65, 128, 200])
def test_decays_are_one_sum_in_order(lib, f32, rule, tiles, dim):
    heads, rank = 5, 32 * tiles
    t = Recur(lib, f32, heads, dim, rank, [3, 3], rule)
    w, low = np.zeros((1, t.r.N, rank), np.float32), np.zeros((6, rank), np.float32)
    w[:, :, [0, rank - 2, rank - 1]], low[[1, 4]] = [4096.0, 1.0, -4096.0], 1.0
    low[[[1], [4]], [0, rank - 1]] = 4096.0
    lib.wr_hip_mix_mat_destroy(t.r.h)
    assert lib.wr_hip_mix_mat_create(1, t.r.N, rank, O.f32_to_bf16(w).ctypes.data, C.byref(t.r.h)) == 0
    t.rec.w_decay, t.rec.low = t.r.h, t.up(low)
    # row 0 makes the state k v^T, row 1 lets it decay, row 2 reads w v + v': one channel a head
    x, at, wide = np.zeros((6, t.ld), np.float32), [0, 1, dim // 2, dim - 2, dim - 1], t.rec.col_k
    v0, v2 = np.where(np.arange(dim) % 2, -1.0, 1.0), np.ones(dim)
    for first in (0, 3):
        for h in range(heads):
            x[[first, first + 2], wide + h * dim + at[h]] = 1.0
            x[first + 2, h * dim + at[h]] = 1.0
            x[first, 2 * wide + h * dim:][:dim], x[first + 2, 2 * wide + h * dim:][:dim] = v0, v2
    t.rec.in_ = t.put(x)
    p = t.pool()
    t.set(p)
    assert lib.wr_hip_mix_recur(t.step, p, 0, int(f32), C.byref(t.rec)) == 0
    o = np.exp(-np.exp(-1.0)) ** (2 if rule == DELTA else 1) * v0 + v2     # (DELTA reads the state behind row 2's decay, of a product of zeros)
    want = 0.5 * np.tile(o / np.sqrt((o * o).mean()), heads)            # (the gate: logistic of 0)
    got = t.out()[[2, 5], :heads * dim]
    # bfloat16: half a unit in the last place of outputs below 1; 32 bits: sums of one product and a norm over 200, each rounded a few times
    assert np.abs(got - want).max() < (0.0 if f32 else 2.0 ** -9) + 2e-6, np.abs(got - want).max()
    t.end()


# Sixteen requests of 64 heads: more workgroups than find a place at once where rows are asked for ahead.  The bits of each request alone.
@pytest.mark.parametrize("f32", [False, True])
@pytest.mark.parametrize("rule", [BONUS, DELTA])
@pytest.mark.parametrize("dim,rank,rows", [(64, 64, 1), (40, 128, 3)])
def test_recurrence_of_many_workgroups(lib, f32, rule, dim, rank, rows):
    many, alone = Recur(lib, f32, 64, dim, rank, [rows] * 16, rule), Recur(lib, f32, 64, dim, rank, [rows], rule)
    x, low = many.rng.standard_normal((16 * rows, many.ld), dtype=np.float32), many.r.act(16 * rows, rank)
    many.rec.in_, many.rec.low = many.put(x), many.up(low)
    p, got = many.pool(), []
    for nth in (0, 1):
        many.set(p, nth)
        assert lib.wr_hip_mix_recur(many.step, p, 0, int(f32), C.byref(many.rec)) == 0
        got.append(many.out())
    for i in (0, 7, 15):
        at = slice(i * rows, (i + 1) * rows)
        alone.rec.in_, alone.rec.low = alone.put(x[at]), alone.up(low[at])
        p = alone.pool()
        for nth in (0, 1):
            alone.set(p, nth)
            assert lib.wr_hip_mix_recur(alone.step, p, 0, int(f32), C.byref(alone.rec)) == 0
            assert np.isfinite(got[nth][at]).all() and np.array_equal(alone.out(), got[nth][at]), (i, nth)
    many.end(), alone.end()


# The append and the recurrence of a step in one launch (bfloat16, DELTA, head sizes 33 to 64, ranks up to 128, no request of more than 16 rows, 8 a request where rows
# are not asked for ahead) and
# either side of each of these: the bits of the two calls, in rows, keys, values and states; refused whole, whichever of the two it is.
@pytest.mark.parametrize("f32,rule,dim,rank,rows,heads", [(False, DELTA, 64, 64, [1], 3), (False, DELTA, 33, 32, [1] * 16, 3), (False, DELTA, 64, 128, [16] * 16, 3),
                                                          (False, DELTA, 40, 96, [3, 1, 16], 3), (False, DELTA, 64, 160, [2, 1], 3), (False, DELTA, 32, 64, [2, 1], 3),
                                                          (False, DELTA, 65, 64, [2, 1], 3), (False, BONUS, 64, 64, [2, 1], 3), (False, DELTA, 64, 64, [2, 17], 3),
                                                          (True, DELTA, 64, 64, [2, 1], 3), (False, DELTA, 40, 64, [1] * 16, 64), (False, DELTA, 40, 64, [8] * 15 + [9], 64)])
def test_append_and_recurrence(lib, f32, rule, dim, rank, rows, heads):
    win = Window(heads=6, kv_heads=3, dim=40, dim_pad=64, vdim=24, vdim_pad=32, rot_half=8, window=1 << 20, scale=0.2, out_scale=1.0, eps=1e-6, maps=1)
    of_win = 6 * 40 + 3 * 40 + 3 * 24
    wide = -(-heads * dim // 32) * 32
    t = Recur(lib, f32, heads, dim, rank, rows, rule, win, 5 * wide + of_win + 4)
    angles = t.put(t.rng.uniform(-1, 1, (t.total, 8, 2)))
    cols, kt = (5 * wide, 5 * wide + 240, 5 * wide + 360), 6 * 64 // 32
    q, o = t.fill(t.padded * kt * 32 * t.e), t.fill(t.padded * 6 * t.e * 32)

    def step(pool, nth, together):
        t.set(pool, nth)
        head = (t.step, pool, 0, int(f32), C.byref(win), t.rec.in_, t.ld, *cols, angles, q.p)
        if together:
            assert lib.wr_hip_mix_window_append_recur(*head, 0, C.byref(t.rec)) == 0
        else:
            assert lib.wr_hip_mix_window_append(*head) == 0
            assert lib.wr_hip_mix_recur(t.step, pool, 0, int(f32), C.byref(t.rec)) == 0
        assert lib.wr_hip_mix_window_attend(t.step, pool, 0, int(f32), C.byref(win), q.p, None, None, 0, o.p, 6) == 0
        out = t.out()
        return [out] + [t.r.frag_down(b, t.total, n * 32) for b, n in ((q, kt), (o, 6))]

    one, two = t.pool(), t.pool()
    for nth in (0, 1):                                     # from nothing, then from what the first left
        for a, b in zip(step(one, nth, True), step(two, nth, False)):
            assert np.isfinite(a).all() and a.any() and np.array_equal(a, b), nth
    t.set(one, 2)
    clean = q.to_host((q.nbytes,), np.uint8), t.h.to_host((t.h.nbytes,), np.uint8)
    lib.wr_hip_attn_h2d(t.rec.in_, np.zeros((t.total, t.ld), np.float32).ctypes.data, t.total * t.ld * 4)
    for bad_win, bad_run in ((win, 1), (Window(), 0)):
        assert lib.wr_hip_mix_window_append_recur(t.step, one, 0, int(f32), C.byref(bad_win), t.rec.in_, t.ld, *cols, angles, q.p, bad_run,
                                                  C.byref(t.rec)) == hipattn.ERR_INVAL
        hipattn.sync()
        assert np.array_equal(q.to_host((q.nbytes,), np.uint8), clean[0]) and np.array_equal(t.h.to_host((t.h.nbytes,), np.uint8), clean[1])
    t.end()


# One row to a workgroup up to 599 rows (1791 with experts' rows) and wherever no fragment is written, four beyond; features
# that a workgroup holds in registers (4096) and more.
@pytest.mark.parametrize("f32", [False, True])
@pytest.mark.parametrize("width", [2048, 4200])
@pytest.mark.parametrize("kind", ["plain", "no_fragment", "no_norm", "pair", "embed", "experts"])
def test_row_steps_of_many_rows(lib, f32, width, kind):
    rng = np.random.default_rng(width)
    counts = (64, 1791, 1792, 1793) if kind == "experts" else (64, 599, 600, 601, 1501)
    most, wpad, top, vocab, eps = max(counts), -(-width // 32) * 32, 3, 50, 1e-6

    def rows(n):
        v = np.zeros((n, wpad), dtype=np.float32)
        v[:, :width] = rng.standard_normal((n, width), dtype=np.float32)
        return v

    def norm(v):
        v = v.astype(np.float64)
        return v / np.sqrt((v ** 2).sum(axis=-1, keepdims=True) / width + eps)

    up = hipattn.DeviceBuffer.from_host
    x0, y, add, post, nxt, post2 = rows(most), rows(most), rows(most), rows(1), rows(1), rows(2)
    pairs, table = [rows(most), rows(most)], O.f32_to_bf16(rng.standard_normal((vocab, width), dtype=np.float32))
    tokens, slot = rng.integers(0, vocab, most), rng.integers(0, most, (most, top)).astype(np.uint32)
    gate = rng.uniform(0, 1, (most, top)).astype(np.float32)
    slot[5, 1] = 0xFFFFFFFF                                    # left out
    want = x0.astype(np.float64)
    if kind == "embed":
        want = norm(O.bf16_to_f32(table)[tokens]) * post[:, :width]
        want = np.pad(want, ((0, 0), (0, wpad - width)))
    elif kind == "experts":
        g = np.where(slot == 0xFFFFFFFF, 0.0, gate).astype(np.float64)
        want = want + norm((g[:, :, None] * y[np.minimum(slot, most - 1)]).sum(axis=1)) * post
    else:
        want = want + (y if kind == "no_norm" else norm(y) * post) + add
        if kind == "pair":
            want = want + norm(pairs[0]) * post2[0] + norm(pairs[1]) * post2[1]
    yd, ad, pd, nd, td = up(y), up(add), up(post), up(nxt), up(table)
    qd, ppd, sd, gd = [up(p) for p in pairs], [up(post2[i:i + 1]) for i in range(2)], up(slot.view(np.float32)), up(gate)
    few = None
    for n in counts:
        s, xd = StepOf(lib, tokens[:n].tolist(), vocab), up(x0[:n])
        hd = hipattn.DeviceBuffer(-(-n // 16) * 16 * wpad * (4 if f32 else 2))
        if kind == "embed":
            assert lib.wr_hip_mix_embed(s.h, int(f32), td.p, width, pd.p, 1.0, eps, xd.p, None, nd.p, hd.p) == 0
        else:
            a = Resid(width=width, eps=eps, x=xd.p, y=yd.p, post=None if kind == "no_norm" else pd.p)
            if not kind.startswith("no_"):
                a.next, a.h = nd.p, hd.p
            if kind == "experts":
                a.gate, a.slot, a.top = gd.p, sd.p, top
            else:
                a.add = ad.p
            if kind == "pair":
                for i in range(2):
                    a.pair_y[i], a.pair_post[i] = qd[i].p, ppd[i].p
            assert lib.wr_hip_mix_residual(s.h, int(f32), C.byref(a)) == 0
        s.end()
        got = [xd.to_host((n, wpad))]
        scale = np.abs(want).max()
        assert np.abs(got[0] - want[:n]).max() < 2e-6 * scale, (kind, n)      # (32-bit sums of some thousand terms)
        if not kind.startswith("no_"):
            m = -(-n // 16) * 16 * wpad
            h = unfrag(hd.to_host((m,)) if f32 else O.bf16_to_f32(hd.to_host((m // 2,)).view(np.uint16)), n, wpad)
            ref = norm(want[:n]) * nxt
            assert np.abs(h - ref).max() < (2e-6 if f32 else 2.0 ** -8) * np.abs(ref).max(), (kind, n)
            got.append(h)
        few = few or got
        for a, b in zip(got, few):                             # a row's bits are its own from 64 rows on
            assert np.array_equal(a[:64], b), (kind, n)
        for b in (xd, hd):
            b.free()
    for b in (yd, ad, pd, nd, td, sd, gd, *qd, *ppd):
        b.free()


def test_refusals(lib):
    r = Run(lib, False, 1, 32, 32, 16)
    y = hipattn.DeviceBuffer(16 * 32 * 4)
    ok = dict(w=r.h, x=y.p, x_kt=1, rows=16, out=ROWS_F32, y_f32=y.p, ldy=32)
    for change in (dict(x_kt=0), dict(ldy=28), dict(ldy=33), dict(y_f32=None), dict(out=9), dict(rows=0), dict(w=None),
                   dict(out=FRAG, h=y.p, h_kt=0), dict(out=SPLIT, h=y.p, h_kt=1, n_split=8), dict(out=GATED), dict(x_kt0=1),
                   dict(out=GATED, h=y.p, h_kt=1, bias=y.p), dict(x_perm=y.p), dict(x_scale=y.p),
                   dict(out=GATED, h=y.p, h_kt=1, h_kt0=1), dict(out=SPLIT_GATED, h=y.p, h_kt=1, n_split=16)):
        assert lib.wr_hip_mix_gemm_run(0, C.byref(Gemm(**dict(ok, **change)))) == hipattn.ERR_INVAL, change
    h = vp()
    for shape in ((1, 8, 32), (1, 16, 16), (0, 16, 32)):
        assert lib.wr_hip_mix_mat_create(*shape, r.bits.ctypes.data, C.byref(h)) == hipattn.ERR_INVAL
    r.end()
    y.free()
