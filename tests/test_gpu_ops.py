"""GPU parity of every kernel behind the C ABI against the CPU oracle / golden vectors.

Tolerance (fp32): |gpu - ref| <= 1e-3 + 1e-4 * |ref| (max-abs 1e-3, rel 1e-4).  Paths whose arithmetic order matches jasmine exactly (per-column
reductions, elementwise trees) are additionally checked for bit-exactness.  bf16
attention: |gpu - fp32 ref| <= 2e-2 + 2e-2 * |ref|.
"""
import math

import numpy as np
import pytest

from jasmine_amd import expr as E
from oracle_lib import orc, fp, normal
from split_model import ATTENTION_BOUND, attention64, error, gemm_bound

pytestmark = pytest.mark.gpu


def close(a, b, atol=1e-3, rtol=1e-4):
    a, b = np.asarray(a, np.float64), np.asarray(b, np.float64)
    err = np.abs(a - b) - (atol + rtol * np.abs(b))
    assert a.shape == b.shape, (a.shape, b.shape)
    assert np.all(np.isfinite(a) == np.isfinite(b)), "non-finite mismatch"
    fin = np.isfinite(b)
    assert np.all(err[fin] <= 0), f"max abs err {np.max(np.abs(a - b)[fin]):.3g}"


def bitfrac(a, b):
    return float(np.mean(np.asarray(a, np.float32).view(np.uint32) == np.asarray(b, np.float32).view(np.uint32)))


# ---------------------------------------------------------------- expressions
GOLD_TREES = {
    0: lambda a, b: a + b,
    1: lambda a, b: a - b * 2,
    2: lambda a, b: a * b / (b + 3.0),
    3: lambda a, b: E.un("exp", a - b),
    4: lambda a, b: E.un("sigmoid", a * b),
    5: lambda a, b: (a > b) * a + (a < b) * b,
    6: lambda a, b: (a + b - a) * b / a,
    7: lambda a, b: a - E.const(1.5, E.F32),
    8: lambda a, b: 2 - a,
}


@pytest.fixture(params=[0, 1], ids=["interp", "jit"])
def ew_mode(jas, request):
    """Run an expression test through the interpreter kernel and through the specialised
    (hipRTC) kernel; the library default picks by output size."""
    prev = jas.lib.jas_ew_jit_mode(request.param)
    yield request.param
    jas.lib.jas_ew_jit_mode(prev)


def test_ew_golden(jas, ew_mode):
    g = np.load(__import__("os").path.join(__import__("os").path.dirname(__file__), "golden", "jasmine_golden.npz"))
    n = 0
    while f"expr{n}_id" in g:
        eid = int(g[f"expr{n}_id"])
        a_h, b_h, want = g[f"expr{n}_a"], g[f"expr{n}_b"], g[f"expr{n}_out"]
        da, db = jas.to_device(a_h), jas.to_device(b_h)
        if eid == 9:  # a.t() * 0.25 + b : transposed view of a
            tree = E.leaf(da, transposed=1) * 0.25 + E.leaf(db)
        else:
            tree = GOLD_TREES[eid](E.leaf(da), E.leaf(db))
        got = E.evaluate(jas, tree).astype(np.float32)
        close(got, want)
        if eid not in (3, 4):  # pure +-*/ and compares are bit-exact with jasmine
            assert bitfrac(got, want) == 1.0, (n, eid)
        n += 1
    assert n >= 13


@pytest.mark.parametrize("shape", [(64, 64), (33, 65), (1024, 1024), (8192, 1024)])
def test_ew_cfg2(jas, ew_mode, shape):
    R, Cc = shape
    a, b, c = normal(shape, 1, 0), normal(shape, 1, 1), normal(shape, 1, 2)
    want = np.zeros_like(a)
    orc.orc_cfg2_expr(fp(a), fp(b), fp(c), fp(want), a.size)
    da, db, dc = jas.to_device(a), jas.to_device(b), jas.to_device(c)
    A, B, C = E.leaf(da), E.leaf(db), E.leaf(dc)
    tree = A * B + 0.5 * C - E.un("tanh", A)
    assert tree.dtype == E.F64  # jasmine promotion through the double scalar
    got = E.evaluate(jas, tree, out_dtype=E.F32)
    close(got, want)
    # the +,-,* part follows jasmine's typed evaluation bit for bit; tanh's last ulp is the
    # platform libm's (glibc tanhf is not correctly rounded), so it is held to tolerance only
    part = E.evaluate(jas, A * B + 0.5 * C, out_dtype=E.F32)
    want_part = ((a * b).astype(np.float64) + 0.5 * c.astype(np.float64)).astype(np.float32)
    assert bitfrac(part, want_part) == 1.0


def test_ew_jasmine_view_and_modulo_semantics(jas, ew_mode):
    # jasmine views add offsets then the underlying mat_t wraps indices modulo its dims
    # (mat_view_t.hpp:28-38, mat_t.hpp:312-320), including the swapped offsets of a
    # transposed view with offsets.
    base = normal((5, 7), 2, 0)
    small = normal((2, 7), 2, 1)
    db, ds = __import__("jasmine_amd").to_device(base), __import__("jasmine_amd").to_device(small)

    def jas_get(m, r, c, roff, coff, t):
        a, bb = (c + coff, r + roff) if t else (r + roff, c + coff)
        return m[a % m.shape[0], bb % m.shape[1]]

    for (roff, coff, t, vr, vc) in [(1, 2, 0, 3, 4), (0, 0, 1, 7, 5), (1, 1, 1, 4, 3), (2, 3, 0, 6, 6)]:
        tree = E.leaf(db, roff=roff, coff=coff, transposed=t, vrows=vr, vcols=vc) + E.leaf(ds)
        out_r, out_c = max(vr, 2), max(vc, 7)
        want = np.array([[jas_get(base, i, j, roff, coff, t) + small[i % 2, j % 7] for j in range(out_c)]
                         for i in range(out_r)], np.float32)
        got = E.evaluate(jas, tree)
        assert got.shape == want.shape
        assert bitfrac(got, want) == 1.0, (roff, coff, t)


def test_ew_unary_and_pow(jas, ew_mode):
    x = normal((37, 41), 3, 0)
    dx = jas.to_device(x)
    X = E.leaf(dx)
    for op, fn in (("tanh", np.tanh), ("gelu", lambda v: 0.5 * v * (1 + np.tanh(0.7978845608028654 * (v + 0.044715 * v ** 3)))),
                   ("silu", lambda v: v / (1 + np.exp(-v))), ("neg", lambda v: -v)):
        close(E.evaluate(jas, E.un(op, X)), fn(x.astype(np.float64)).astype(np.float32), atol=2e-6, rtol=2e-6)
    sq = E.evaluate(jas, E.un("sqrt", E.un("pow", X, imm=2.0)))
    close(sq, np.abs(x), atol=1e-6, rtol=1e-6)


def test_ew_jit_equals_interpreter(jas):
    """The specialised kernel reproduces the interpreter bit for bit on mixed-type trees:
    int / float / double nodes, comparisons, every unary op, broadcast and strided views."""
    x = normal((67, 130), 4, 0)
    y = (np.abs(normal((67, 130), 4, 1)) + 0.25).astype(np.float32)
    r = normal((1, 130), 4, 2)
    xd = normal((67, 130), 4, 3).astype(np.float64)
    iv = (np.arange(67 * 130, dtype=np.int32).reshape(67, 130) % 11) - 5
    dx, dy, dr, dxd, di = (jas.to_device(v) for v in (x, y, r, xd, iv))
    X, Y, Rw, XD = E.leaf(dx), E.leaf(dy), E.leaf(dr), E.leaf(dxd, dtype=E.F64)
    I = E.leaf(di, dtype=E.I32)
    XT = E.leaf(dx, roff=3, coff=5, transposed=1, vrows=60, vcols=60)
    trees = [
        X * Y + 0.5 * Rw - E.un("tanh", X),
        (X > Y) * X + (X < Y) * Y / 3,
        E.un("exp", X - Rw) + E.un("sigmoid", X * 2.0) - E.un("silu", Y),
        E.un("gelu", X) * E.un("sqrt", Y) + E.un("pow", Y, imm=1.5),
        XD * X - E.un("exp", XD * 0.25) + E.un("neg", X),
        I * 3 + I / 2 - (I > 0) * X,
        E.un("gelu", XD) + E.un("tanh", XD) - E.un("sqrt", XD * XD),
    ]
    for k, t in enumerate(trees):
        for out_dt in (E.F32, t.dtype):
            jas.lib.jas_ew_jit_mode(0)
            a = E.evaluate(jas, t, out_dtype=out_dt)
            jas.lib.jas_ew_jit_mode(1)
            b = E.evaluate(jas, t, out_dtype=out_dt)
            jas.lib.jas_ew_jit_mode(2)
            assert a.shape == b.shape and a.dtype == b.dtype
            assert np.array_equal(a.view(np.uint8), b.view(np.uint8)), (k, out_dt)
    # transposed-offset view (general modulo addressing) against a dense leaf
    dsq = jas.to_device(np.ascontiguousarray(x[:60, :60]))  # keep the buffer alive while the leaf is used
    t = XT * 2.0 + E.leaf(dsq)
    jas.lib.jas_ew_jit_mode(0)
    a = E.evaluate(jas, t)
    jas.lib.jas_ew_jit_mode(1)
    b = E.evaluate(jas, t)
    jas.lib.jas_ew_jit_mode(2)
    assert np.array_equal(a.view(np.uint8), b.view(np.uint8))


def _rb(x):
    u = np.ascontiguousarray(x, np.float32).view(np.uint32).astype(np.uint64)
    return (((u + 0x7FFF + ((u >> 16) & 1)) >> 16)).astype(np.uint16)


def _wide(u16):
    return (u16.astype(np.uint32) << 16).view(np.float32)


def test_ew_bf16_leaves_and_nodes(jas):
    """bf16 leaves and nodes (mat_t<jas::bf16>): float operation then round to nearest even
    per node; interpreter and specialised kernel bit-identical; bf16 with an int constant stays
    bf16, with a float leaf it widens."""
    x, y = normal((300, 1030), 6, 0), normal((300, 1030), 6, 1)
    bx, by = _rb(x), _rb(y)
    dx, dy, df = jas.to_device(bx), jas.to_device(by), jas.to_device(y)
    X, Y, Fy = E.leaf(dx, dtype=E.BF16), E.leaf(dy, dtype=E.BF16), E.leaf(df)
    t = (X * Y + X) / (Y * 2 + 3) - (X > Y) * X
    assert t.dtype == E.BF16
    xf, yf = _wide(bx), _wide(by)
    r = lambda v: _wide(_rb(v))
    with np.errstate(all="ignore"):
        want = r(r(r(r(xf * yf) + xf) / r(r(yf * np.float32(2)) + np.float32(3))) - r((xf > yf).astype(np.float32) * xf))
    outs = []
    for mode in (0, 1):
        jas.lib.jas_ew_jit_mode(mode)
        try:
            outs.append(E.evaluate(jas, t))
        finally:
            jas.lib.jas_ew_jit_mode(2)
    assert outs[0].dtype == np.uint16
    assert np.array_equal(outs[0], outs[1])
    assert np.array_equal(_wide(outs[0]), want)
    mixed = X * Fy + E.un("exp", X * 0.5)  # float leaf and a double constant widen the tree
    assert mixed.dtype == E.F64
    got = []
    for mode in (0, 1):
        jas.lib.jas_ew_jit_mode(mode)
        try:
            got.append(E.evaluate(jas, mixed, out_dtype=E.BF16))
        finally:
            jas.lib.jas_ew_jit_mode(2)
    a, b = got
    assert np.array_equal(a, b)
    ref = (xf.astype(np.float64) * y.astype(np.float64) + np.exp(xf.astype(np.float64) * 0.5))
    assert np.all(np.abs(_wide(a) - ref) <= 2.0 ** -8 * np.abs(ref) + 1e-6)


def test_ew_rejects_bad_programs(jas):
    import ctypes as C
    from jasmine_amd.capi import Ins, Leaf, DeviceArray, lib
    out = DeviceArray((4, 4))
    prog = (Ins * 2)(Ins(1, 0, 0, 0, 1.0), Ins(2, 0, 0, 0, 0.0))  # const then ADD: stack underflow
    assert lib.jas_ew_eval(prog, 2, (Leaf * 1)(), 0, out.p, 0, 4, 4, None) == 1
    assert b"underflow" in lib.jas_last_error()


# ---------------------------------------------------------------- reductions
def test_reductions_bitexact(jas):
    g = np.load(__import__("os").path.join(__import__("os").path.dirname(__file__), "golden", "jasmine_golden.npz"))
    x = g["x"]
    R, Cc = x.shape
    dx = jas.to_device(x)
    lf = jas.leaf(dx)
    import ctypes as C
    for op, axis, name, n in ((0, 0, "hsum", R), (0, 1, "vsum", Cc), (1, 0, "hmax", R), (2, 1, "vmean", Cc),
                              (2, 0, "hmean", R)):
        out = jas.DeviceArray(n)
        jas.check(jas.lib.jas_reduce(C.byref(lf), op, axis, out.p, 0, None))
        assert bitfrac(out.numpy(), g[name]) == 1.0, name  # same sequential order as jasmine
    for op, k in ((0, 0), (1, 1), (2, 2)):
        out = jas.DeviceArray(1)
        jas.check(jas.lib.jas_reduce(C.byref(lf), op, 2, out.p, 0, None))
        close(out.numpy()[0], g["sum_max_mean"][k], atol=1e-5, rtol=1e-5)


# stage edges of the row form (16 KB over 16 / 8 / 4 / 1 lines per wave, from 4096 / 1024 /
# 256 lines) and of the column form (128 / 64 / 32 bytes of a row per wave), odd widths
# (4-byte loads), views with offsets and transposed ones, and short lines (under 64 elements)
@pytest.mark.parametrize("rows,cols,dt,roff,coff,t", [
    (4100, 260, "f4", 0, 0, 0), (4097, 255, "f4", 0, 0, 0), (1029, 516, "f4", 0, 0, 0), (257, 1028, "f4", 0, 0, 0),
    (1030, 1027, "f4", 0, 0, 0), (70, 4100, "f4", 0, 0, 0), (3, 9001, "f4", 0, 0, 0), (1030, 8200, "f4", 0, 0, 0),
    (300, 4100, "f4", 0, 4, 0), (300, 4101, "f4", 2, 3, 0), (515, 130, "f4", 0, 0, 1), (515, 132, "f4", 4, 0, 1),
    (2050, 130, "f8", 0, 0, 0), (131, 2051, "f8", 1, 1, 0), (4104, 72, "f8", 0, 0, 1), (300, 2064, "bf", 0, 0, 0),
    (300, 515, "bf", 0, 1, 0), (200, 40, "f4", 0, 0, 0), (40, 200, "f4", 0, 0, 0), (1, 70, "f4", 0, 0, 0), (70, 1, "f4", 0, 0, 0)])
def test_reductions_staged_bitexact(jas, rows, cols, dt, roff, coff, t):
    import ctypes as C
    x = normal((rows, cols), 7, rows + cols).astype(np.float64 if dt == "f8" else np.float32)
    x[rows // 2, cols // 3] = -np.inf  # max of a line with an infinity; sums stay finite elsewhere
    if dt == "bf":
        u = x.view(np.uint32) >> 16
        dx, x = jas.to_device(u.astype(np.uint16)), (u << 16).view(np.float32)
    else:
        dx = jas.to_device(x)
    # the logical view: the underlying (a, b) = (i + roff, j + coff), or (j + coff, i + roff) transposed
    v = x[coff:, roff:].T if t else x[roff:, coff:]
    lf = jas.leaf(dx, roff=roff, coff=coff, transposed=t, vrows=v.shape[0], vcols=v.shape[1])
    acc = x.dtype
    # a running sum / maximum in the accumulator type has jasmine's order: its last entry is the line's result
    sums = [np.add.accumulate(v, axis=1 - a, dtype=acc).take(-1, 1 - a) for a in (0, 1)]
    # a maximum starts from the type's lowest finite value (hmax, mat_express_t.hpp:619)
    maxs = [np.maximum(v.max(axis=1 - a), np.finfo(acc).min) for a in (0, 1)]
    total = np.add.accumulate(sums[0], dtype=acc)[-1]
    for op in (0, 1, 2):
        for axis in (0, 1, 2):
            n = (v.shape[0], v.shape[1], 1)[axis]
            want = maxs[axis] if op == 1 and axis < 2 else v.max() if op == 1 else sums[axis] if axis < 2 else total
            if op == 2:
                want = want / acc.type(v.size if axis == 2 else v.shape[1 - axis])
            out = jas.DeviceArray(n, acc)
            jas.check(jas.lib.jas_reduce(C.byref(lf), op, axis, out.p, 1 if dt == "f8" else 0, None))
            assert np.array_equal(out.numpy(), np.asarray(want, acc).reshape(n)), (op, axis)


@pytest.mark.parametrize("n_vec,length", [(3, 7), (5, 64), (4, 300), (2, 1000), (3, 2048), (2, 4099), (2, 8192),
                                          (1, 16384), (2, 20000)])
def test_row_ops(jas, n_vec, length):
    x = normal((n_vec, length), 4, length, std=2.0)
    dx, dy = jas.to_device(x), jas.DeviceArray((n_vec, length))
    want = np.zeros_like(x)
    jas.check(jas.lib.jas_softmax(dx.p, dy.p, n_vec, length, length, length, 1, None))
    orc.orc_hsoftmax(fp(x), n_vec, length, fp(want))
    close(dy.numpy(), want, atol=1e-6, rtol=1e-4)
    gam = normal(length, 4, 1, mean=1.0, std=0.1)
    bet = normal(length, 4, 2, std=0.1)
    dg, dbt = jas.to_device(gam), jas.to_device(bet)
    jas.check(jas.lib.jas_layernorm(dx.p, dy.p, n_vec, length, length, length, 1, 1e-5, dg.p, dbt.p, None))
    orc.orc_layernorm_rows(fp(x), n_vec, length, 1e-5, fp(gam), fp(bet), fp(want))
    close(dy.numpy(), want)
    jas.check(jas.lib.jas_rmsnorm(dx.p, dy.p, n_vec, length, length, length, 1, 1e-6, dg.p, None))
    orc.orc_rmsnorm_rows(fp(x), n_vec, length, 1e-6, fp(gam), fp(want))
    close(dy.numpy(), want)


def test_column_layernorm_jasmine(jas):
    # jasmine's layer_norm_net_t normalises each column of a feature-major [d, T] matrix, eps 0
    g = np.load(__import__("os").path.join(__import__("os").path.dirname(__file__), "golden", "jasmine_golden.npz"))
    x = g["x"]
    R, Cc = x.shape
    dx, dy = jas.to_device(x), jas.DeviceArray((R, Cc))
    jas.check(jas.lib.jas_layernorm(dx.p, dy.p, Cc, R, 1, 1, Cc, 0.0, None, None, None))
    close(dy.numpy(), g["layernorm_cols"], atol=1e-5, rtol=1e-5)
    jas.check(jas.lib.jas_softmax(dx.p, dy.p, R, Cc, Cc, Cc, 1, None))
    close(dy.numpy(), g["hsoftmax"], atol=1e-6, rtol=1e-5)


@pytest.mark.parametrize("mode", ["ln", "rms", "softmax"])
@pytest.mark.parametrize("R,Cc", [(512, 100), (130, 37), (1000, 64), (3, 5), (4096, 130), (5000, 64), (1000, 1024),
                                  (3000, 2048), (7, 1028)])
def test_column_row_ops(jas, mode, R, Cc):
    """Vectors down the columns of a row-major [R, Cc] matrix (element stride Cc): the
    column kernels against the oracle's row functions on the transposed matrix.  Column
    counts that are multiples of 4 take the 16-byte column-group kernel (8 vectors per
    workgroup below 1024 columns, 16 from 1024; elements held in registers up to 4096 / 2048
    rows, streamed past that: (5000, 64) and (3000, 2048)); the others the one-float form."""
    x = normal((R, Cc), 34, 0)
    xt = np.ascontiguousarray(x.T)
    gam, bet = normal(R, 34, 1), normal(R, 34, 2)
    want = np.zeros_like(xt)
    dx, dy, dg, db = jas.to_device(x), jas.DeviceArray((R, Cc)), jas.to_device(gam), jas.to_device(bet)
    if mode == "ln":
        orc.orc_layernorm_rows(fp(xt), Cc, R, 1e-5, fp(gam), fp(bet), fp(want))
        jas.check(jas.lib.jas_layernorm(dx.p, dy.p, Cc, R, 1, 1, Cc, 1e-5, dg.p, db.p, None))
    elif mode == "rms":
        orc.orc_rmsnorm_rows(fp(xt), Cc, R, 1e-6, fp(gam), fp(want))
        jas.check(jas.lib.jas_rmsnorm(dx.p, dy.p, Cc, R, 1, 1, Cc, 1e-6, dg.p, None))
    else:
        orc.orc_hsoftmax(fp(xt), Cc, R, fp(want))
        jas.check(jas.lib.jas_softmax(dx.p, dy.p, Cc, R, 1, 1, Cc, None))
    close(dy.numpy(), np.ascontiguousarray(want.T), atol=1e-5, rtol=1e-5)


def test_softmax_global(jas):
    x = normal((300, 517), 5, 0)
    dx, dy = jas.to_device(x), jas.DeviceArray(x.shape)
    jas.check(jas.lib.jas_softmax_global(dx.p, dy.p, x.size, None))
    want = np.zeros_like(x)
    orc.orc_softmax_global(fp(x), 300, 517, fp(want))
    close(dy.numpy(), want, atol=1e-9, rtol=1e-4)


def test_scratch_per_stream(jas):
    """Whole-matrix softmax keeps its partials in library scratch: calls queued on two
    streams without synchronising in between must not share it (one buffer per stream),
    including when one stream's buffer grows while the other's work is in flight."""
    import ctypes as C

    hip = C.CDLL("libamdhip64.so")
    sa, sb = C.c_void_p(), C.c_void_p()
    assert hip.hipStreamCreateWithFlags(C.byref(sa), 1) == 0  # non-blocking, default priority
    assert hip.hipStreamCreateWithFlags(C.byref(sb), 1) == 0
    xa, xb = normal((512, 2048), 6, 0), normal((1024, 4096), 6, 1)
    # float64 references: a sequential float sum over millions of terms drifts by ~1e-4
    wa, wb = (np.exp(x.astype(np.float64) - x.max()) for x in (xa, xb))
    wa, wb = wa / wa.sum(), wb / wb.sum()
    dxa, dxb = jas.to_device(xa), jas.to_device(xb)
    outs = [(jas.DeviceArray(xa.shape), jas.DeviceArray(xb.shape)) for _ in range(4)]
    for ya, yb in outs:
        jas.check(jas.lib.jas_softmax_global(dxa.p, ya.p, xa.size, sa))
        jas.check(jas.lib.jas_softmax_global(dxb.p, yb.p, xb.size, sb))
    assert hip.hipDeviceSynchronize() == 0
    for ya, yb in outs:
        close(ya.numpy(), wa, atol=0, rtol=1e-5)
        close(yb.numpy(), wb, atol=0, rtol=1e-5)
    # releasing a stream's scratch waits for its queued work; the next multi-pass call on it
    # allocates again, and a stream that never held scratch releases nothing
    for ya, _ in outs:
        jas.check(jas.lib.jas_softmax_global(dxa.p, ya.p, xa.size, sa))
    jas.check(jas.lib.jas_stream_release_scratch(sa))
    jas.check(jas.lib.jas_softmax_global(dxa.p, outs[0][0].p, xa.size, sa))
    jas.check(jas.lib.jas_stream_release_scratch(sa))
    jas.check(jas.lib.jas_stream_release_scratch(sa))
    for ya, _ in outs:
        close(ya.numpy(), wa, atol=0, rtol=1e-5)
    jas.check(jas.lib.jas_stream_release_scratch(sb))
    hip.hipStreamDestroy(sa)
    hip.hipStreamDestroy(sb)


# ---------------------------------------------------------------- GEMM
def _gemm_case(jas, M, N, K, ta=False, tb=False, col_c=False, bias_mode=0, act=0, acc=False, batch=1, seed=0):
    A = normal((batch, K, M) if ta else (batch, M, K), 10 + seed, 0)
    B = normal((batch, N, K) if tb else (batch, K, N), 10 + seed, 1)
    C0 = normal((batch, N, M) if col_c else (batch, M, N), 10 + seed, 2)
    bias = normal((batch, M if bias_mode == 1 else N), 10 + seed, 3)
    An = np.swapaxes(A, 1, 2) if ta else A
    Bn = np.swapaxes(B, 1, 2) if tb else B
    ref = np.einsum("bmk,bkn->bmn", An.astype(np.float64), Bn.astype(np.float64))
    if bias_mode == 1:
        ref += bias[:, :, None]
    elif bias_mode == 2:
        ref += bias[:, None, :]
    if act == 1:
        ref = np.where(ref > 0, ref, 0.0)
    elif act == 2:
        ref = 0.5 * ref * (1 + np.tanh(0.7978845608028654 * (ref + 0.044715 * ref ** 3)))
    if acc:
        ref += np.swapaxes(C0, 1, 2) if col_c else C0
    dA, dB, dC, dbias = jas.to_device(A), jas.to_device(B), jas.to_device(C0), jas.to_device(bias)
    as0, as1 = (1, M) if ta else (K, 1)
    bs0, bs1 = (1, K) if tb else (N, 1)
    cs0, cs1 = (1, M) if col_c else (N, 1)
    jas.check(jas.lib.jas_gemm(M, N, K, dA.p, as0, as1, dB.p, bs0, bs1, dC.p, cs0, cs1, dbias.p, bias_mode, act,
                               int(acc), batch, M * K, K * N, M * N, bias.shape[1], None))
    got = dC.numpy()
    if col_c:
        got = np.swapaxes(got, 1, 2)
    # fp32 accumulation of K products: scale the tolerance with sqrt(K) * |a||b|
    scale = np.sqrt(K) * 1.0
    close(got, ref.astype(np.float32), atol=1e-5 * scale + 1e-5, rtol=1e-5)


@pytest.mark.parametrize("M,N,K", [(1, 1, 1), (7, 5, 13), (128, 128, 16), (130, 257, 65), (512, 384, 1024),
                                   (256, 200, 4096)])
def test_gemm_shapes(jas, M, N, K):
    _gemm_case(jas, M, N, K)


@pytest.mark.parametrize("ta,tb,col_c", [(1, 0, 0), (0, 1, 0), (1, 1, 1), (0, 0, 1)])
def test_gemm_layouts(jas, ta, tb, col_c):
    _gemm_case(jas, 136, 72, 40, ta=bool(ta), tb=bool(tb), col_c=bool(col_c))
    _gemm_case(jas, 33, 17, 7, ta=bool(ta), tb=bool(tb), col_c=bool(col_c))


@pytest.mark.parametrize("bias_mode,act,acc,batch", [(1, 0, 0, 1), (2, 1, 0, 2), (1, 2, 1, 3), (0, 0, 1, 1)])
def test_gemm_epilogues(jas, bias_mode, act, acc, batch):
    _gemm_case(jas, 150, 90, 70, bias_mode=bias_mode, act=act, acc=bool(acc), batch=batch)


@pytest.mark.parametrize("ta,tb,col_c", [(0, 0, 0), (1, 0, 0), (0, 1, 0), (1, 1, 1), (0, 0, 1), (1, 0, 1)])
@pytest.mark.parametrize("bias_mode,acc,batch", [(0, 0, 1), (1, 0, 2), (2, 0, 1), (0, 1, 3)])
def test_gemm_library_sizes(jas, ta, tb, col_c, bias_mode, acc, batch):
    """Products of a few hundred rows and columns, single and batched: every operand
    layout, both bias modes, accumulation, batches; K of 200 and 129 leave a partial slab."""
    _gemm_case(jas, 300, 260, 200, ta=bool(ta), tb=bool(tb), col_c=bool(col_c), bias_mode=bias_mode, acc=bool(acc),
               batch=batch)
    _gemm_case(jas, 257, 513, 129, ta=bool(ta), tb=bool(tb), col_c=bool(col_c), bias_mode=bias_mode, acc=bool(acc),
               batch=batch, seed=1)


@pytest.mark.parametrize("ta,tb,col_c", [(0, 0, 0), (1, 1, 0), (0, 1, 1), (1, 0, 1)])
@pytest.mark.parametrize("M,N,K", [(4096, 4096, 40), (2048, 2100, 70), (1024, 1024, 1024)])
def test_gemm_dma_geometries(jas, ta, tb, col_c, M, N, K):
    """Large and middle-sized products over operand layouts, with ragged edges, partial K slabs,
    bias and accumulation."""
    _gemm_case(jas, M, N, K, ta=bool(ta), tb=bool(tb), col_c=bool(col_c), bias_mode=1, acc=True)


@pytest.mark.parametrize("M,N,K,act,rcol,bstride,ccol", [
    (512, 512, 512, 0, 0, 0, 0), (300, 260, 200, 1, 0, 0, 0), (257, 129, 129, 1, 1, 0, 0), (96, 70, 64, 0, 0, 3, 0),
    # 32 x 32 tiles by two waves: row-major and column-major C
    (1024, 1024, 256, 1, 0, 0, 0), (1024, 1024, 256, 0, 1, 0, 1),
    # 128 x 64 tiles: both C layouts
    (4096, 4096, 128, 0, 0, 0, 0), (4096, 4096, 128, 1, 1, 0, 1), (300, 516, 96, 1, 0, 0, 1)])
def test_gemm_residual(jas, M, N, K, act, rcol, bstride, ccol):
    """jas_gemm_residual: act(A B + bias) + R, against jas_gemm of the same operands followed by
    the residual added in fp32 (bit for bit: the same product, then the same two roundings).
    R row- or column-major, C row- or column-major; B with a padded row stride (3 extra
    floats), whose rows are not 16-byte aligned."""
    rng = np.random.default_rng(61)
    A = rng.standard_normal((M, K), dtype=np.float32)
    ldb = N + bstride
    B = rng.standard_normal((K, ldb), dtype=np.float32)
    bias = rng.standard_normal(M, dtype=np.float32)
    R = rng.standard_normal((M, N), dtype=np.float32)
    dA, dB, db = jas.to_device(A), jas.to_device(B), jas.to_device(bias)
    dR = jas.to_device(np.ascontiguousarray(R.T) if rcol else R)
    r0, r1 = (1, M) if rcol else (N, 1)
    c0, c1 = (1, M) if ccol else (N, 1)
    want, got = jas.DeviceArray((M, N)), jas.DeviceArray((M, N))
    jas.check(jas.lib.jas_gemm(M, N, K, dA.p, K, 1, dB.p, ldb, 1, want.p, c0, c1, db.p, 1, act, 0, 1, 0, 0, 0, 0, None))
    jas.check(jas.lib.jas_gemm_residual(M, N, K, dA.p, K, 1, dB.p, ldb, 1, got.p, c0, c1, db.p, 1, act, dR.p, r0, r1,
                                        None))
    w, g_ = want.numpy(), got.numpy()
    if ccol:  # the buffers hold C column-major
        w, g_ = w.reshape(N, M).T, g_.reshape(N, M).T
    assert np.array_equal(g_, w + R)


# every geometry of launch_split and launch_unpacked (gemm_split.hip) at its edges: partial tiles in both
# dimensions, K tails, K of less than a slab, rows that are not 16-byte aligned (odd leading
# dimensions), general strides (a step of 2 in both dimensions), both orders of C, batches
@pytest.mark.parametrize("M,N,K,batch", [
    (4100, 2050, 70, 1),    # 256 x 128, whole rounds
    (4097, 1023, 1057, 1),  # 128 x 64, long K
    (1537, 2049, 90, 1), (2100, 2050, 70, 1), (2100, 2050, 260, 1),  # 128 x 64, few slabs (64 x 64 split four ways)
    (1300, 1500, 90, 1), (350, 400, 140, 14),  # 64 x 64 in LDS, eight and four waves
    (1000, 1000, 100, 1), (1000, 1400, 170, 1), (1100, 1200, 100, 1),  # 64 x 64, 64 x 32 and, by two and four waves, 32 x 32
    (700, 900, 200, 1), (700, 900, 300, 1),  # 32 x 32 by four or two waves, 64 x 32
    (65, 33, 65, 40), (65, 33, 128, 1),  # K <= 128: 32 x 32, four waves
    (1023, 515, 333, 1),    # 64 x 32, four waves
    (600, 501, 257, 1),     # 64 x 32, eight waves
    (333, 450, 300, 1),     # 32 x 32, eight waves
    (33, 17, 4101, 1), (1, 1, 31, 1), (5, 300, 1, 2)])  # 32 x 16
@pytest.mark.parametrize("la,lb,lc", [(0, 0, 0), (0, 1, 1), (1, 0, 1), (1, 1, 0), (2, 0, 0), (0, 2, 1)])
def test_gemm_split_geometries(jas, M, N, K, batch, la, lb, lc):
    # layout 0: row-major, 1: column-major, 2: every second element of every second row
    def make(r, c, lay, sid):
        if lay == 2:
            buf = normal((batch, 2 * r, 2 * c), 31, sid)
            return buf, buf[:, ::2, ::2], (4 * c, 2), 4 * r * c
        buf = normal((batch, r, c) if lay == 0 else (batch, c, r), 31, sid)
        return buf, buf if lay == 0 else np.swapaxes(buf, 1, 2), (c, 1) if lay == 0 else (1, r), r * c

    Ab, A, (as0, as1), ab = make(M, K, la, 0)
    Bb, B, (bs0, bs1), bb = make(K, N, lb, 1)
    Cb, Cv, (cs0, cs1), cb = make(M, N, lc, 2)
    dA, dB, dC = jas.to_device(Ab), jas.to_device(Bb), jas.to_device(Cb)
    jas.check(jas.lib.jas_gemm(M, N, K, dA.p, as0, as1, dB.p, bs0, bs1, dC.p, cs0, cs1, None, 0, 0, 0, batch, ab, bb, cb, 0,
                               None))
    got = dC.numpy() if lc == 0 else np.swapaxes(dC.numpy(), 1, 2)
    want = A.astype(np.float64) @ B.astype(np.float64)
    # K products, each with at most one rounding of the running sum (2^-24 of it, below the sum
    # of magnitudes), and 2^-26 of each product left out by the split
    bound = (K + 2) * 2.0 ** -24 * (np.abs(A).astype(np.float64) @ np.abs(B).astype(np.float64))
    assert np.all(np.abs(got - want) <= bound + 1e-30), float(np.max(np.abs(got - want) / (bound + 1e-30)))
    # and the root mean square, which a lost product of two planes exceeds (test_split_model.py)
    assert error(got, want, np.sqrt(K)) <= gemm_bound(K), (error(got, want, np.sqrt(K)), gemm_bound(K))


@pytest.mark.parametrize("M,N,K", [(4096, 2048, 64), (1024, 4096, 1056), (2048, 1536, 96), (1000, 1000, 100),
                                   (96, 64, 640), (200, 90, 120)])
def test_gemm_split_range(jas, M, N, K):
    """Values outside the bf16 split's range: infinities, NaN, magnitudes that round to infinity
    in bf16, products that overflow, and operands so small that their parts underflow -- each
    in rows or columns of its own, next to ordinary ones."""
    A, B = normal((M, K), 32, 0), normal((K, N), 32, 1)
    A[3, 5], A[7, K - 1], B[2, 9] = np.inf, np.nan, -np.inf
    B[2, :9], B[2, 10:] = 0.5, 0.5                      # keep 0 * inf out of the other columns
    A[11] = 0.0
    A[11, 4] = 3.4e38                                   # rounds to infinity in bf16
    B[4] = np.where(np.arange(N) % 2, 0.25, -0.5)
    A[20] = 3e38                                        # overflows against B[:, 30], which sums to 16
    B[:, 30] = 16.0 / K
    A[33] *= np.float32(2.0 ** -118)                    # parts below the smallest bf16
    A[50] *= np.float32(2.0 ** -100)
    B[:, 40] *= np.float32(2.0 ** -20)
    dA, dB, dC = jas.to_device(A), jas.to_device(B), jas.DeviceArray((M, N))
    jas.check(jas.lib.jas_gemm(M, N, K, dA.p, K, 1, dB.p, N, 1, dC.p, N, 1, None, 0, 0, 0, 1, 0, 0, 0, 0, None))
    got = dC.numpy()
    with np.errstate(all="ignore"):
        want = A.astype(np.float64) @ B.astype(np.float64)
        mag = np.abs(A).astype(np.float64) @ np.abs(B).astype(np.float64)
    assert np.array_equal(np.isnan(got[[3, 7]]), np.isnan(want[[3, 7]]))
    assert np.array_equal(got[3][np.isinf(want[3])], want[3][np.isinf(want[3])])
    rows = np.setdiff1d(np.arange(M), [3, 7, 20])
    g, w, m = got[rows], want[rows], mag[rows]
    fin = np.isfinite(m)  # the column with -inf: an infinity or NaN everywhere
    assert np.all(fin[:, np.arange(N) != 9]) and not np.any(np.isfinite(g[:, 9][A[rows, 2] != 0]))
    # as above; fp32 sums of products of 2^-118 also round at the smallest denormal, 2^-149
    bound = (K + 2) * (2.0 ** -24 * m[fin] + 2.0 ** -149)
    assert np.all(np.abs(g[fin] - w[fin]) <= bound), float(np.max(np.abs(g[fin] - w[fin]) / bound))
    assert np.isinf(got[20, 30]) and got[20, 30] > 0


@pytest.mark.parametrize("M,N,K", [(4096, 2048, 64), (2050, 2100, 1056), (1030, 1900, 96), (1000, 1000, 100),
                                   (96, 64, 640), (200, 90, 120)])
def test_gemm_split_subnormal(jas, M, N, K):
    """Operands below 2^-110, subnormal ones and ones below the smallest bf16 among them, against
    partners large enough that their products are ordinary numbers, and next to ordinary
    operands; sums that cancel down to those products' size."""
    A, B = normal((M, K), 37, 0), normal((K, N), 37, 1)
    A[3] *= np.float32(2.0 ** -136)                      # a few bits above 2^-149
    A[5] = np.float32(2.0 ** -149)
    A[7] *= np.float32(2.0 ** -125)
    A[9] = 0
    A[9, ::2], A[9, 1::2] = np.float32(2.0 ** -120 * (1 + 2.0 ** -20)), np.float32(-2.0 ** -120)
    B[:, 2] *= np.float32(2.0 ** 100)
    B[:, 4] = np.float32(2.0 ** 60)
    B[:, 6] *= np.float32(2.0 ** -130)
    A[11] *= np.float32(2.0 ** 95)
    dA, dB, dC = jas.to_device(A), jas.to_device(B), jas.DeviceArray((M, N))
    jas.check(jas.lib.jas_gemm(M, N, K, dA.p, K, 1, dB.p, N, 1, dC.p, N, 1, None, 0, 0, 0, 1, 0, 0, 0, 0, None))
    got = dC.numpy()
    want = A.astype(np.float64) @ B.astype(np.float64)
    mag = np.abs(A).astype(np.float64) @ np.abs(B).astype(np.float64)
    assert np.any(A[3] != 0) and abs(want[5, 2]) > 2.0 ** -60
    fin = mag < 2.0 ** 127  # row 11 overflows against columns 2 and 4
    assert np.sum(~fin) == 2
    # each product's rounding and those of the running sum (2^-24, below the sum of magnitudes),
    # and of subnormal sums (2^-149)
    bound = (K + 2) * (2.0 ** -24 * mag[fin] + 2.0 ** -149)
    assert np.all(np.abs(got[fin] - want[fin]) <= bound), float(np.nanmax(np.abs(got[fin] - want[fin]) / bound))


@pytest.mark.parametrize("M,N,K", [(4096, 2048, 64), (2050, 2100, 1056), (1030, 1900, 96), (1000, 1000, 100),
                                   (96, 64, 640), (200, 90, 120)])
def test_gemm_split_one_lost_sum(jas, M, N, K):
    """A single product below the split's range in a tile of ordinary sums: column n is zero but for
    one element of 2^100, which row m alone meets with a number that has no bf16 part.  Rows and
    columns of zeros, whose sums are zero rightly, beside it."""
    A, B = normal((M, K), 38, 0), normal((K, N), 38, 1)
    m, n, k = M - 3, N // 2 + 1, K - 2
    A[::16], B[:, ::24] = 0, 0
    B[:, n], B[k, n], A[m, k] = 0, np.float32(2.0 ** 100), np.float32(1.25 * 2.0 ** -136)
    dA, dB, dC = jas.to_device(A), jas.to_device(B), jas.DeviceArray((M, N))
    jas.check(jas.lib.jas_gemm(M, N, K, dA.p, K, 1, dB.p, N, 1, dC.p, N, 1, None, 0, 0, 0, 1, 0, 0, 0, 0, None))
    got = dC.numpy()
    assert got[m, n] == np.float32(A[m, k]) * np.float32(B[k, n])
    want = A.astype(np.float64) @ B.astype(np.float64)
    bound = (K + 2) * 2.0 ** -24 * (np.abs(A).astype(np.float64) @ np.abs(B).astype(np.float64))  # as above
    assert np.all(np.abs(got - want) <= bound)


def test_gemm_dma_k_tail_padded_rows(jas):
    """K not a multiple of 4 with padded, K-contiguous rows: the tail slab reads element by
    element and zero-fills past K."""
    M, N, K, Kp = 300, 260, 147, 152
    A = np.zeros((M, Kp), np.float32)
    Bt = np.zeros((N, Kp), np.float32)
    A[:, :K] = normal((M, K), 36, 0)
    Bt[:, :K] = normal((N, K), 36, 1)
    A[:, K:] = np.nan  # padding must never be read
    Bt[:, K:] = np.nan
    dA, dB, dC = jas.to_device(A), jas.to_device(Bt), jas.DeviceArray((M, N))
    jas.check(jas.lib.jas_gemm(M, N, K, dA.p, Kp, 1, dB.p, 1, Kp, dC.p, N, 1, None, 0, 0, 0, 1, 0, 0, 0, 0, None))
    ref = A[:, :K].astype(np.float64) @ Bt[:, :K].astype(np.float64).T
    close(dC.numpy(), ref.astype(np.float32), atol=1e-5 * np.sqrt(K) + 1e-5, rtol=1e-5)


@pytest.mark.parametrize("N", [1, 2, 5, 8, 16])
@pytest.mark.parametrize("M,K", [(300, 64), (64, 100), (1000, 4096), (4096, 1024), (8200, 80), (25000, 64)])
def test_gemm_skinny(jas, M, N, K):
    # decode shape: W [M][K], tokens X [N][K] -> out [N][M] (token-major), via jas_gemm's skinny path
    W, X, b = normal((M, K), 20, 0), normal((N, K), 20, 1), normal(M, 20, 2)
    dW, dX, db, dO = jas.to_device(W), jas.to_device(X), jas.to_device(b), jas.DeviceArray((N, M))
    jas.check(jas.lib.jas_gemm(M, N, K, dW.p, K, 1, dX.p, 1, K, dO.p, 1, M, db.p, 1, 0, 0, 1, 0, 0, 0, 0, None))
    ref = X.astype(np.float64) @ W.astype(np.float64).T + b
    close(dO.numpy(), ref.astype(np.float32), atol=1e-5 * np.sqrt(K) + 1e-5, rtol=1e-5)


# ---------------------------------------------------------------- attention
@pytest.mark.parametrize("B,H,Sq,Sk,D,causal", [(2, 3, 100, 100, 64, 1), (1, 2, 64, 64, 32, 0), (2, 2, 70, 130, 128, 1),
                                                (1, 4, 200, 200, 128, 1), (1, 1, 1, 1, 64, 1), (2, 2, 37, 90, 64, 0),
                                                # non-causal with few query blocks: keys split over
                                                # work items and merged (ragged last split included)
                                                (1, 2, 100, 700, 64, 0), (2, 3, 130, 1000, 32, 0),
                                                (1, 1, 50, 513, 128, 0), (1, 2, 1, 300, 64, 0)])
def test_attn_prefill(jas, B, H, Sq, Sk, D, causal):
    Q, K, V = normal((B, H, Sq, D), 30, 0), normal((B, H, Sk, D), 30, 1), normal((B, H, Sk, D), 30, 2)
    want = np.zeros((B, H, Sq, D), np.float32)
    sc = 1 / math.sqrt(D)
    orc.orc_attention(fp(Q), fp(K), fp(V), fp(want), B, H, Sq, Sk, D, sc, causal)
    dq, dk, dv, do = jas.to_device(Q), jas.to_device(K), jas.to_device(V), jas.DeviceArray(Q.shape)
    jas.check(jas.lib.jas_attn_prefill(dq.p, dk.p, dv.p, do.p, B, H, Sq, Sk, D, H * Sq * D, Sq * D, D, H * Sk * D,
                                       Sk * D, D, H * Sq * D, Sq * D, D, sc, causal, 0, None))
    close(do.numpy(), want, atol=1e-5, rtol=1e-4)


@pytest.mark.parametrize("B,H,Sq,Sk,D,causal", [(2, 2, 96, 96, 64, 1), (1, 3, 70, 130, 128, 1), (2, 1, 64, 64, 32, 0),
                                                (1, 2, 200, 200, 128, 0), (1, 1, 1, 17, 64, 1),
                                                (1, 2, 77, 600, 128, 0), (2, 2, 64, 1024, 64, 0)])
def test_attn_prefill_bf16(jas, B, H, Sq, Sk, D, causal):
    """bf16 inputs on bf16 MFMA with fp32 accumulation and softmax; P is rounded to bf16 for
    the P.V product.  Held to 2e-2 abs + 2e-2 rel against the fp32 attention of the same
    (bf16-rounded) inputs."""
    Q, K, V = normal((B, H, Sq, D), 31, 0), normal((B, H, Sk, D), 31, 1), normal((B, H, Sk, D), 31, 2)

    def bf(x):  # round to nearest even bf16, as uint16
        u = x.astype(np.float32).view(np.uint32).astype(np.uint64)
        return ((u + 0x7FFF + ((u >> 16) & 1)) >> 16).astype(np.uint16)

    def unbf(u):
        return (u.astype(np.uint32) << 16).view(np.float32)

    Qb, Kb, Vb = bf(Q), bf(K), bf(V)
    sc = 1 / math.sqrt(D)
    want = np.zeros((B, H, Sq, D), np.float32)
    orc.orc_attention(fp(unbf(Qb)), fp(unbf(Kb)), fp(unbf(Vb)), fp(want), B, H, Sq, Sk, D, sc, causal)
    dq, dk, dv = jas.to_device(Qb), jas.to_device(Kb), jas.to_device(Vb)
    do = jas.DeviceArray((B, H, Sq, D), np.uint16)
    jas.check(jas.lib.jas_attn_prefill(dq.p, dk.p, dv.p, do.p, B, H, Sq, Sk, D, H * Sq * D, Sq * D, D, H * Sk * D,
                                       Sk * D, D, H * Sq * D, Sq * D, D, sc, causal, 3, None))
    close(unbf(do.numpy()), want, atol=2e-2, rtol=2e-2)


@pytest.mark.parametrize("B,H,Sq,Sk,D,dt", [(1, 2, 600, 600, 64, 0), (2, 3, 513, 700, 128, 0), (1, 2, 1030, 1030, 32, 0),
                                            (1, 2, 520, 520, 128, 3), (2, 1, 777, 800, 64, 3)])
def test_attn_prefill_long_causal(jas, B, H, Sq, Sk, D, dt):
    """Causal launches of four or more 128-query blocks (the heaviest-first work order over
    blocks of unequal cost), with Sk > Sq in two cases.  Two launches in a row with different
    inputs."""
    sc = 1 / math.sqrt(D)

    def bf(x):
        u = x.astype(np.float32).view(np.uint32).astype(np.uint64)
        return ((u + 0x7FFF + ((u >> 16) & 1)) >> 16).astype(np.uint16)

    def unbf(u):
        return (u.astype(np.uint32) << 16).view(np.float32)

    for rep in range(2):
        Q, K, V = (normal(sh, 33 + rep, i) for i, sh in enumerate(((B, H, Sq, D), (B, H, Sk, D), (B, H, Sk, D))))
        if dt:
            Q, K, V = (unbf(bf(x)) for x in (Q, K, V))
        want = np.zeros((B, H, Sq, D), np.float32)
        orc.orc_attention(fp(Q), fp(K), fp(V), fp(want), B, H, Sq, Sk, D, sc, 1)
        dq, dk, dv = (jas.to_device(bf(x) if dt else x) for x in (Q, K, V))
        do = jas.DeviceArray((B, H, Sq, D), np.uint16 if dt else np.float32)
        jas.check(jas.lib.jas_attn_prefill(dq.p, dk.p, dv.p, do.p, B, H, Sq, Sk, D, H * Sq * D, Sq * D, D, H * Sk * D,
                                           Sk * D, D, H * Sq * D, Sq * D, D, sc, 1, dt, None))
        if dt:
            close(unbf(do.numpy()), want, atol=2e-2, rtol=2e-2)
        else:
            close(do.numpy(), want, atol=1e-5, rtol=1e-4)


# flash_bf16_kernel (D = 128) with 32 queries per wave: not causal from 256 blocks of 128
# queries, causal from 1024; partial query blocks and key tiles
@pytest.mark.parametrize("B,H,Sq,Sk,causal", [(4, 33, 130, 130, 0), (2, 128, 65, 200, 0), (16, 33, 129, 193, 1), (32, 32, 33, 33, 1)])
def test_attn_prefill_bf16_wide(jas, B, H, Sq, Sk, causal):
    import ctypes as C
    D = 128

    def bf(shape, sid):
        x = normal(shape, 43, sid).view(np.uint32)
        u = ((x + 0x7FFF + ((x >> 16) & 1)) >> 16).astype(np.uint16)
        return u, (u.astype(np.uint32) << 16).view(np.float32)

    (qu, Q), (ku, K), (vu, V) = bf((B, H, Sq, D), 0), bf((B, H, Sk, D), 1), bf((B, H, Sk, D), 2)
    dq, dk, dv, do = jas.to_device(qu), jas.to_device(ku), jas.to_device(vu), jas.DeviceArray(Q.shape, np.uint16)
    qs, ks = (H * Sq * D, Sq * D, D), (H * Sk * D, Sk * D, D)
    jas.check(jas.lib.jas_attn_prefill(dq.p, dk.p, dv.p, do.p, B, H, Sq, Sk, D, *qs, *ks, *qs, C.c_float(1 / math.sqrt(D)),
                                       causal, 3, None))
    got = (do.numpy().astype(np.uint32) << 16).view(np.float32)
    for b, h in [(0, 0), (B - 1, H - 1), (B // 2, 7)]:
        want = _attention64(Q[b:b + 1, h:h + 1], K[b:b + 1, h:h + 1], V[b:b + 1, h:h + 1], causal)[0, 0]
        # probabilities and the output rounded to bf16 (2^-9 each), the row sum over the rounded ones
        assert np.abs(got[b, h] - want).max() <= 3 * 2.0 ** -9 * np.abs(V[b, h]).max()


def _attention64(Q, K, V, causal):
    """[B, H, S, D] attention in 64 bits, causal aligned to the last key; masked keys carry nothing."""
    Q, K, V = (x.astype(np.float64) for x in (Q, K, V))
    out = np.zeros(Q.shape)
    Sq, Sk = Q.shape[2], K.shape[2]
    with np.errstate(all="ignore"):
        for b, h, i in np.ndindex(*Q.shape[:3]):
            n = min(Sk, i + Sk - Sq + 1) if causal else Sk
            s = K[b, h, :n] @ Q[b, h, i] / math.sqrt(Q.shape[3])
            e = np.exp(s - s.max())
            out[b, h, i] = (e[:, None] * V[b, h, :n]).sum(0) / e.sum()
    return out


def _run_attention_f32(jas, Q, K, V, causal):
    import ctypes as C
    B, H, Sq, D = Q.shape
    Sk = K.shape[2]
    dq, dk, dv, do = jas.to_device(Q), jas.to_device(K), jas.to_device(V), jas.DeviceArray(Q.shape)
    qs, ks = (H * Sq * D, Sq * D, D), (H * Sk * D, Sk * D, D)
    jas.check(jas.lib.jas_attn_prefill(dq.p, dk.p, dv.p, do.p, B, H, Sq, Sk, D, *qs, *ks, *qs, C.c_float(1 / math.sqrt(D)),
                                       causal, 0, None))
    return do.numpy()


# both widths of flash_split_kernel (32 queries per wave from 256 blocks of 128; 16 below), the
# edges of its query blocks and key tiles, and its key split (few items, at least 256 keys)
@pytest.mark.parametrize("B,H,Sq,Sk,D,causal", [(8, 33, 97, 97, 32, 1), (16, 17, 65, 130, 64, 0), (4, 33, 129, 129, 64, 1),
                                                (3, 5, 63, 95, 128, 1), (1, 3, 130, 130, 128, 0), (1, 2, 17, 300, 64, 1),
                                                (1, 2, 70, 257, 32, 0), (1, 1, 1, 1, 64, 1)])
def test_attn_prefill_split(jas, B, H, Sq, Sk, D, causal):
    Q, K, V = normal((B, H, Sq, D), 41, 0), normal((B, H, Sk, D), 41, 1), normal((B, H, Sk, D), 41, 2)
    got = _run_attention_f32(jas, Q, K, V, causal)
    want = _attention64(Q, K, V, causal)
    # a score of magnitude sum |q||k| / sqrt(D) <= 12 here carries at most D roundings of 2^-24
    # of it, a probability that relative error twice (its own and its row sum's)
    bound = 2 * 12 * D * 2.0 ** -24 * np.abs(V).max()
    assert np.abs(got - want).max() <= bound, (np.abs(got - want).max(), bound)
    # and the root mean square over all heads, which a lost product exceeds (test_split_model.py)
    rms = np.sqrt(np.mean([error(got[b, h], *attention64(Q[b, h], K[b, h], V[b, h], causal)) ** 2
                           for b, h in np.ndindex(B, H)]))
    assert rms <= ATTENTION_BOUND, rms


@pytest.mark.parametrize("B,H,S,D", [(1, 2, 70, 64), (1, 1, 300, 32), (1, 1, 80, 128), (16, 17, 66, 64)])
def test_attn_prefill_split_range(jas, B, H, S, D):
    """Rows outside the bf16 split's range: infinities and NaN in Q, K and V, values of V whose
    parts underflow, and small Q against large K."""
    Q, K, V = (normal((B, H, S, D), 42, k) for k in range(3))
    Q[0, 0, 5, 3] = np.inf
    K[0, 0, 40, 0] = np.nan   # reaches queries 40 and up
    V[0, 0, 60, 1] = np.inf   # and 60 and up
    if B * H > 1:
        b, h = (0, 1) if B == 1 else (B - 1, H - 1)
        V[b, h] *= np.float32(2.0 ** -119)
        Q[b, h] *= np.float32(2.0 ** -112)
        K[b, h] *= np.float32(2.0 ** 112)
    got = _run_attention_f32(jas, Q, K, V, 1)
    want = _attention64(Q, K, V, 1)
    # row 5's one infinite query element gives infinite scores: no finite output
    assert np.array_equal(np.isfinite(got), np.isfinite(want))
    fin = np.isfinite(want)
    scale = np.broadcast_to(np.nanmax(np.where(np.isfinite(V), np.abs(V), np.nan), axis=(2, 3), keepdims=True), V.shape)
    # as above, and sums of products below 2^-126 round at 2^-149
    bound = 2 * 12 * D * 2.0 ** -24 * scale[fin] + S * 2.0 ** -149
    assert np.all(np.abs(got[fin] - want[fin]) <= bound), np.max(np.abs(got[fin] - want[fin]) / bound)


@pytest.mark.parametrize("B,H,S,D", [(1, 2, 70, 64), (1, 1, 300, 32), (1, 1, 80, 128), (16, 17, 66, 64)])
def test_attn_prefill_split_subnormal(jas, B, H, S, D):
    """Values of V below the smallest bf16 (2^-133), below 2^-110 and ordinary ones in columns of
    their own, and Q and K whose parts lie there."""
    Q, K, V = (normal((B, H, S, D), 44, k) for k in range(3))
    V[..., 0::4] *= np.float32(2.0 ** -140)
    V[..., 1::4] *= np.float32(2.0 ** -120)
    V[..., 2::4] *= np.float32(2.0 ** 90)
    Q *= np.float32(2.0 ** -108)
    K *= np.float32(2.0 ** 108)
    got = _run_attention_f32(jas, Q, K, V, 1)
    want = _attention64(Q, K, V, 1)
    # as in test_attn_prefill_split, for each column; the output rounds at 2^-149
    bound = 2 * 12 * D * 2.0 ** -24 * np.abs(V).max((0, 1, 2)) + 2.0 ** -149
    assert np.all(np.abs(want[..., 0::4]).max((0, 1, 2)) > 8 * 2.0 ** -149)
    assert np.all(np.abs(got - want) <= bound), np.max(np.abs(got - want) / bound)


@pytest.mark.parametrize("D", [32, 64, 128])
@pytest.mark.parametrize("dt", [0, 3])
def test_attn_prefill_key_split_nan(jas, D, dt):
    """NaN in launches whose keys are split over work items: a NaN key reaches every query of its
    head through the merge, a NaN query every element of its row, a NaN value its column."""
    import ctypes as C
    B, H, Sq, Sk = 1, 4, 40, 600
    x = [normal(sh, 45, k) for k, sh in enumerate(((B, H, Sq, D), (B, H, Sk, D), (B, H, Sk, D)))]
    x[1][0, 1, 450, 2] = np.nan
    x[0][0, 2, 5, 1] = np.nan
    x[2][0, 3, 333, 7] = np.nan
    if dt:  # the upper halves: bf16 numbers (truncated), NaN stays NaN
        x = [(v.view(np.uint32) >> 16).astype(np.uint16) for v in x]
    dq, dk, dv = (jas.to_device(v) for v in x)
    do = jas.DeviceArray((B, H, Sq, D), np.uint16 if dt else np.float32)
    qs, ks = (H * Sq * D, Sq * D, D), (H * Sk * D, Sk * D, D)
    jas.check(jas.lib.jas_attn_prefill(dq.p, dk.p, dv.p, do.p, B, H, Sq, Sk, D, *qs, *ks, *qs, C.c_float(1 / math.sqrt(D)),
                                       0, dt, None))
    got = (do.numpy().astype(np.uint32) << 16).view(np.float32) if dt else do.numpy()
    want = np.zeros((B, H, Sq, D), bool)
    want[0, 1] = True
    want[0, 2, 5] = True
    want[0, 3, :, 7] = True
    assert np.array_equal(np.isnan(got), want)


@pytest.mark.parametrize("D,dt,causal", [(64, 0, 1), (64, 3, 1), (128, 3, 0), (32, 3, 1), (128, 0, 0)])
def test_attn_prefill_growing_scores(jas, D, dt, causal):
    """Keys whose scale grows along the sequence, so the running row max keeps rising by more
    than the lazy-rescale threshold (2^8 in exponent units) deep into the key range: the
    accumulator is rescaled on late tiles, and probabilities above 1 (a stale base) are
    exercised in between.  Raw scores reach about 100 here, so the fp32 rounding of a score
    alone moves p by about 1e-5 relative: fp32 is held to 1e-4 abs (the configs' fp32 bound
    is 1e-3)."""
    B, H, S = 1, 2, 700
    sc = 1 / math.sqrt(D)
    Q = normal((B, H, S, D), 34, 0)
    K = normal((B, H, S, D), 34, 1) * (1 + np.arange(S, dtype=np.float32) / 64)[None, None, :, None]
    V = normal((B, H, S, D), 34, 2)

    def bf(x):
        u = x.astype(np.float32).view(np.uint32).astype(np.uint64)
        return ((u + 0x7FFF + ((u >> 16) & 1)) >> 16).astype(np.uint16)

    def unbf(u):
        return (u.astype(np.uint32) << 16).view(np.float32)

    if dt:
        Q, K, V = (unbf(bf(x)) for x in (Q, K, V))
    want = np.zeros((B, H, S, D), np.float32)
    orc.orc_attention(fp(Q), fp(K), fp(V), fp(want), B, H, S, S, D, sc, causal)
    dq, dk, dv = (jas.to_device(bf(x) if dt else x) for x in (Q, K, V))
    do = jas.DeviceArray((B, H, S, D), np.uint16 if dt else np.float32)
    jas.check(jas.lib.jas_attn_prefill(dq.p, dk.p, dv.p, do.p, B, H, S, S, D, H * S * D, S * D, D, H * S * D,
                                       S * D, D, H * S * D, S * D, D, sc, causal, dt, None))
    if dt:
        close(unbf(do.numpy()), want, atol=2e-2, rtol=2e-2)
    else:
        close(do.numpy(), want, atol=1e-4, rtol=1e-4)


@pytest.mark.parametrize("B,H,D,lens", [(2, 3, 64, (1, 37)), (3, 2, 128, (1000, 513, 64)), (1, 4, 32, (2049,)),
                                        (8, 12, 64, (1024,) * 8)])
def test_attn_decode(jas, B, H, D, lens):
    ctx = max(lens) + 5
    K, V = normal((B, H, ctx, D), 32, 0), normal((B, H, ctx, D), 32, 1)
    q = normal((B, H, 1, D), 32, 2)
    sc = 1 / math.sqrt(D)
    want = np.zeros((B, H, 1, D), np.float32)
    for b in range(B):
        L = lens[b]
        Kb, Vb = np.ascontiguousarray(K[b:b + 1, :, :L]), np.ascontiguousarray(V[b:b + 1, :, :L])
        o = np.zeros((1, H, 1, D), np.float32)
        orc.orc_attention(fp(np.ascontiguousarray(q[b:b + 1])), fp(Kb), fp(Vb), fp(o), 1, H, 1, L, D, sc, 1)
        want[b] = o[0]
    dq, dk, dv, do = jas.to_device(q), jas.to_device(K), jas.to_device(V), jas.DeviceArray((B, H, D))
    dl = jas.to_device(np.array(lens, np.int32))
    ws_bytes = jas.lib.jas_attn_decode_workspace(B, H, D, max(lens))
    ws = jas.DeviceArray(max(ws_bytes // 4, 1))
    jas.check(jas.lib.jas_attn_decode(dq.p, dk.p, dv.p, do.p, dl.p, B, H, D, max(lens), H * ctx * D, ctx * D, sc,
                                      ws.p, None))
    close(do.numpy(), want[:, :, 0], atol=1e-5, rtol=1e-4)


@pytest.mark.parametrize("B,H,D,lens,cap", [(2, 3, 64, (1, 37), 300), (3, 2, 128, (1000, 513, 64), 1100),
                                            (8, 12, 64, (1024, 0, 5, 129, 1024, 700, 1, 64), 1024),
                                            (2, 4, 32, (2049, 100), 2100)])
def test_attn_decode_poisoned_tail(jas, B, H, D, lens, cap):
    """Cache rows at and past each sequence's length hold NaN and Inf (the kernel's first
    tile is requested before the length is known, bounded only by the cache's row count
    max_len = cap): they must carry no weight.  Empty sequences (length 0) give zeros."""
    K, V = normal((B, H, cap, D), 33, 0), normal((B, H, cap, D), 33, 1)
    for b, L in enumerate(lens):
        K[b, :, L:] = np.nan
        V[b, :, L::2] = np.inf
        V[b, :, L + 1::2] = np.nan
    q = normal((B, H, 1, D), 33, 2)
    sc = 1 / math.sqrt(D)
    want = np.zeros((B, H, D), np.float32)
    for b, L in enumerate(lens):
        if L == 0:
            continue
        o = np.zeros((1, H, 1, D), np.float32)
        orc.orc_attention(fp(np.ascontiguousarray(q[b:b + 1])), fp(np.ascontiguousarray(K[b:b + 1, :, :L])),
                          fp(np.ascontiguousarray(V[b:b + 1, :, :L])), fp(o), 1, H, 1, L, D, sc, 1)
        want[b] = o[0, :, 0]
    dq, dk, dv, do = jas.to_device(q), jas.to_device(K), jas.to_device(V), jas.DeviceArray((B, H, D))
    dl = jas.to_device(np.array(lens, np.int32))
    ws = jas.DeviceArray(max(jas.lib.jas_attn_decode_workspace(B, H, D, cap) // 4, 1))
    for _ in range(2):  # the split-arrival counters are left at zero for the next call
        jas.check(jas.lib.jas_attn_decode(dq.p, dk.p, dv.p, do.p, dl.p, B, H, D, cap, H * cap * D, cap * D, sc,
                                          ws.p, None))
        got = do.numpy()
        assert np.all(np.isfinite(got))
        close(got, want, atol=1e-5, rtol=1e-4)


# ---------------------------------------------------------------- RoPE / embed / argmax / rng
def test_rope_jasmine(jas):
    for d, T in ((16, 6), (64, 33), (7, 5)):
        X = normal((d, T), 40, d)
        want = np.zeros_like(X)
        orc.orc_rope_jas(fp(X), d, T, fp(want))
        dx, dy = jas.to_device(X), jas.DeviceArray((d, T))
        jas.check(jas.lib.jas_rope_jasmine(dx.p, dy.p, d, T, None))
        close(dy.numpy(), want, atol=1e-6, rtol=1e-5)
    g = np.load(__import__("os").path.join(__import__("os").path.dirname(__file__), "golden", "jasmine_golden.npz"))
    dx, dy = jas.to_device(g["rope_x"]), jas.DeviceArray(g["rope_x"].shape)
    jas.check(jas.lib.jas_rope_jasmine(dx.p, dy.p, 16, 6, None))
    close(dy.numpy(), g["rope_y"], atol=1e-6, rtol=1e-5)


def test_rope_llama(jas):
    n, nh, dh = 5, 3, 128
    X = normal((n, nh * dh), 41, 0)
    pos = np.array([0, 1, 7, 1000, 2175], np.int32)
    want = X.copy()
    for t in range(n):
        for h in range(nh):
            seg = np.ascontiguousarray(want[t, h * dh:(h + 1) * dh])
            orc.orc_rope_llama(fp(seg), dh, int(pos[t]), 10000.0)
            want[t, h * dh:(h + 1) * dh] = seg
    dx, dp = jas.to_device(X), jas.to_device(pos)
    jas.check(jas.lib.jas_rope_llama(dx.p, dp.p, n, nh, dh, nh * dh, 10000.0, None))
    close(dx.numpy(), want, atol=1e-6, rtol=1e-6)


def test_hbm_read_probe(jas):
    """The bandwidth calibration reads its buffer and writes its 4-byte sink only when the
    folded data equal a fixed constant (seeded normal data do not); bad arguments are
    rejected before any launch."""
    n = 1 << 20
    buf = jas.DeviceArray((n,))
    jas.check(jas.lib.jas_fill_normal(buf.p, n, 7, 0, 0.0, 1.0, None))
    sink = jas.to_device(np.array([12345], np.uint32))
    for wgs, u, nt in ((1, 4, 1), (300, 8, 0), (2048, 8, 1)):
        jas.check(jas.lib.jas_hbm_read_probe(buf.p, 4 * n, wgs, u, nt, sink.p, None))
    jas.check(jas.lib.jas_synchronize(None))
    assert int(sink.numpy()[0]) == 12345
    for args in ((buf.p, 4 * n + 4, 64, 8, 1), (buf.p, 4 * n, 0, 8, 1), (buf.p, 4 * n, 64, 5, 1), (None, 4 * n, 64, 8, 1)):
        with pytest.raises(jas.JasError):
            jas.check(jas.lib.jas_hbm_read_probe(*args, sink.p, None))


def test_embed_argmax_fill(jas):
    V, d, n = 50, 16, 7
    wte, wpe = normal((V, d), 42, 0), normal((20, d), 42, 1)
    ids, pos = np.array([3, 0, 49, 7, 7, 12, 1], np.int32), np.arange(7, dtype=np.int32)
    dw, dp, di, dpo, do = jas.to_device(wte), jas.to_device(wpe), jas.to_device(ids), jas.to_device(pos), jas.DeviceArray((n, d))
    jas.check(jas.lib.jas_embed(dw.p, dp.p, di.p, dpo.p, do.p, n, d, None))
    assert bitfrac(do.numpy(), wte[ids] + wpe[pos]) == 1.0
    x = normal((4, 50257), 42, 2)
    x[1, 100] = x[1, 30000] = 50.0  # tie -> first index
    dx, da = jas.to_device(x), jas.DeviceArray(4, np.int32)
    jas.check(jas.lib.jas_argmax(dx.p, 4, 50257, 50257, da.p, None))
    assert list(da.numpy()) == [int(np.argmax(r)) for r in x]
    dn = jas.DeviceArray(100003)
    jas.check(jas.lib.jas_fill_normal(dn.p, 100003, 9, 3, 0.0, 0.02, None))
    close(dn.numpy(), normal(100003, 9, 3, std=0.02), atol=1e-7, rtol=1e-6)


@pytest.mark.parametrize("n,V,ld", [(1, 1, 1), (3, 4095, 4100), (16, 4097, 4097), (5, 32000, 32000), (16, 50257, 50260)])
def test_argmax_two_pass(jas, n, V, ld):
    """Ties resolve to the first index also when the tied values sit in different chunks
    (4096 elements per chunk) or on a chunk's first/last element; -inf rows give 0."""
    x = np.full((n, ld), np.nan, np.float32)
    x[:, :V] = normal((n, V), 7, n)
    if V > 4096:
        x[0, 4095] = x[0, 4096] = 80.0      # tie across the chunk boundary
    if n > 1:
        x[1, :V] = -np.inf
    if n > 2:
        x[2, V - 1] = 90.0                  # last element
    if n > 3:
        x[3, :V] = 1.0                      # all equal
    dx, da = jas.to_device(x), jas.DeviceArray(n, np.int32)
    jas.check(jas.lib.jas_argmax(dx.p, n, V, ld, da.p, None))
    assert list(da.numpy()) == [int(np.argmax(r[:V])) for r in x]


# ---------------------------------------------------------------- API support kernels
def test_leaf_assign_block_and_convert(jas):
    dst = np.zeros((7, 9), np.float32)
    dd = jas.to_device(dst)
    src = normal((3, 4), 5, 1).astype(np.float64)
    ds = jas.to_device(src)
    lf = jas.leaf(dd, roff=2, coff=3, vrows=3, vcols=4)
    jas.check(jas.lib.jas_leaf_assign(ds.p, 1,  # JAS_F64
                                           3, 4, __import__("ctypes").byref(lf), None))
    want = dst.copy()
    want[2:5, 3:7] = src.astype(np.float32)
    assert np.array_equal(dd.numpy(), want)


def test_causal_mask(jas):
    for dt, fn in ((np.float32, jas.lib.jas_causal_mask), (np.float64, jas.lib.jas_causal_mask_f64)):
        s = normal((6, 9), 5, 2).astype(dt)
        d = jas.to_device(s)
        ninf = __import__("ctypes").c_float(-np.inf) if dt == np.float32 else __import__("ctypes").c_double(-np.inf)
        jas.check(fn(d.p, 5, 8, 9, ninf, None))  # 5 x 8 block of a 6 x 9 matrix, ld 9
        want = s.copy()
        for i in range(5):
            want[i, i + 1:8] = -np.inf
        assert np.array_equal(d.numpy(), want)


@pytest.mark.parametrize("M,N,K", [(1, 1, 1), (17, 9, 33), (64, 80, 100), (130, 7, 257)])
def test_gemm_f64(jas, M, N, K):
    A, B = normal((M, K), 6, 1).astype(np.float64), normal((K, N), 6, 2).astype(np.float64)
    bias = normal(M, 6, 3).astype(np.float64)
    dA, dB, dbias, dC = jas.to_device(A), jas.to_device(B), jas.to_device(bias), jas.DeviceArray((M, N), np.float64)
    jas.check(jas.lib.jas_gemm_f64(M, N, K, dA.p, K, 1, dB.p, N, 1, dC.p, N, 1, dbias.p, 1, None))
    want = A @ B + bias[:, None]
    assert np.max(np.abs(dC.numpy() - want)) <= 1e-12 * (1 + np.max(np.abs(want))) * np.sqrt(K)


def test_rope_jasmine_f64(jas):
    d, T = 10, 7
    x = normal((d, T), 6, 4).astype(np.float64)
    dx, dy = jas.to_device(x), jas.DeviceArray((d, T), np.float64)
    jas.check(jas.lib.jas_rope_jasmine_f64(dx.p, dy.p, d, T, None))

    def entry(r, c):  # mat_RoPE_t::init in double (mat_RoPE_t.hpp:99-134)
        a = c / 10000.0 ** ((r // 2) / float(d))
        if r % 2 == c % 2:
            return np.cos(a)
        return -np.sin(a) if r % 2 == 0 else np.sin(a)

    want = np.zeros_like(x)
    for m in range(T):
        for i in range(d // 2):
            for r in range(2):
                want[2 * i + r, m] = entry(2 * i + r, 2 * m) * x[2 * i, m] + entry(2 * i + r, 2 * m + 1) * x[2 * i + 1, m]
    assert np.max(np.abs(dy.numpy() - want)) <= 1e-13


# ---------------------------------------------------------------- block pool behind mat_t
def test_pool_reuses_and_trims(jas):
    import ctypes as C
    lib = jas.lib
    a, b, c = C.c_void_p(), C.c_void_p(), C.c_void_p()
    jas.check(lib.jas_pool_alloc(C.byref(a), 1000))
    jas.check(lib.jas_pool_alloc(C.byref(b), 1000))
    assert a.value and b.value and a.value != b.value
    jas.check(lib.jas_pool_free(b))
    jas.check(lib.jas_pool_alloc(C.byref(c), 900))  # same rounded size (1 KiB): the cached block
    assert c.value == b.value
    with pytest.raises(jas.JasError):
        jas.check(lib.jas_pool_free(C.c_void_p(a.value + 4)))  # not a block of the pool
    jas.check(lib.jas_pool_free(a))
    jas.check(lib.jas_pool_free(c))
    n = C.c_size_t()
    jas.check(lib.jas_pool_trim(C.byref(n)))
    assert n.value >= 2048
    jas.check(lib.jas_pool_trim(C.byref(n)))
    assert n.value == 0


def test_gemm_library_is_deterministic(jas):
    """Two runs of a library-sized product give identical bits (no atomic reductions)."""
    M, N, K = 512, 384, 2048
    A, B = normal((M, K), 35, 0), normal((K, N), 35, 1)
    dA, dB = jas.to_device(A), jas.to_device(B)
    outs = []
    for _ in range(2):
        dC = jas.DeviceArray((M, N))
        jas.check(jas.lib.jas_gemm(M, N, K, dA.p, K, 1, dB.p, N, 1, dC.p, N, 1, None, 0, 0, 0, 1, 0, 0, 0, 0, None))
        outs.append(dC.numpy())
    assert np.array_equal(outs[0].view(np.uint32), outs[1].view(np.uint32))
