"""The kernels of the launcher's own forms (maize_amd/csrc/kernels/form_kernels.hip), launched by hand from their code object
at the sizes where they can go wrong: one element more or less than a tile, a K tile, a 16-byte chunk, a ring of K tiles;
rows and pointers on no grid; K ranges.  Against the oracle, to the bars of the registry kernels (test_gpu_gemm_ex.py,
test_gpu_gemm_f8.py)."""
import ctypes as C
import os

import numpy as np
import pytest

import maize_amd as mz
from maize_amd import _ffi

pytestmark = pytest.mark.gpu

HSACO = os.path.join(os.path.dirname(mz.LIB_PATH), "maize_forms_gfx950.hsaco")
NN, NT = mz.LAYOUT_NN, mz.LAYOUT_NT
TILES = {"32x128": (32, 128), "64x64": (64, 64), "64x128": (64, 128), "64x64w": (64, 64), "128x128": (128, 128)}
OPS = {"bf16": 0, "f16": 4, "e4m3": 8, "e5m2": 8 | 48, "e4m3e5m2": 8 | 32, "e5m2e4m3": 8 | 16}      # GemmArgs::epi


@pytest.fixture(scope="module")
def forms(ctx):
    with open(HSACO, "rb") as f:
        mod = ctx.load_module(f.read())
    yield mod
    mod.unload()


def operands(oracle, op, count, which, seed):
    rng = np.random.default_rng(seed)
    x = rng.random(count) * 2.0 - 1.0
    if op in ("bf16", "f16"):
        return oracle.bf16_bits_from_f64(x, oracle.BF16 if op == "bf16" else oracle.F16)
    fmt = op if len(op) == 4 else op[:4] if which == 0 else op[4:]
    return oracle.fp8_bits_from_f64(x, {"e4m3": oracle.E4M3, "e5m2": oracle.E5M2}[fmt])


def check_form(ctx, oracle, mod, op, tile, layout, m, n, k, ks=1, off=0, pad=0, alpha=1.0, beta=0.0, out_f32=False, batch=1):
    bm, bn = TILES[tile]
    name = f"maize_tile_{op}_{'nt' if layout == NT else 'nn'}_{tile}"
    esz = 2 if op in ("bf16", "f16") else 1
    brows, bcols = (n, k) if layout == NT else (k, n)
    lda, ldb, ldc = k + pad, bcols + pad, n + pad
    sa, sb, sc = m * lda + pad, brows * ldb + pad, m * ldc + pad
    a, b = operands(oracle, op, batch * sa, 0, 1), operands(oracle, op, batch * sb, 1, 2)
    c0 = np.random.default_rng(3).random(batch * sc + off).astype(np.float32) if out_f32 else operands(oracle, "f16" if op == "f16" else "bf16", batch * sc + off, 0, 3)
    place = lambda x: np.concatenate([np.zeros(off, x.dtype), x])
    da, db, dc = ctx.upload(place(a)), ctx.upload(place(b)), ctx.upload(c0)
    items = -(-m // bm) * -(-n // bn) * batch * ks
    ws = ctx.malloc(65536 + items * bm * bn * 4)
    ws.fill(0)
    args = _ffi.GemmArgsT(a=da.ptr + off * esz, arows=m, acols=k, b=db.ptr + off * esz, brows=brows, bcols=bcols,
                          c=dc.ptr + off * c0.itemsize, crows=m, ccols=n, stride_a=sa, stride_b=sb, stride_c=sc, batch=batch, layout=layout,
                          workspace=ws.ptr, ksplit=ks, lda=lda, ldb=ldb, ldc=ldc,
                          epi=OPS[op] | (1 if out_f32 else 0) | (2 if (alpha, beta) != (1.0, 0.0) else 0), alpha=alpha, beta=beta)
    print(f"form {name} {m}x{n}x{k} ks={ks} off={off} pad={pad} batch={batch} f32={out_f32} beta={beta}", flush=True)
    kern = mod.kernel(name)
    mz.api.LoadedKernel(ctx, mod, kern, (256, 1, 1)).launch((items, 1, 1), args)
    ctx.sync()
    got, left = dc.download(c0.dtype), ws.download(np.uint32, 16384)
    _ffi.check(_ffi.lib().maize_hip_kernel_release(kern))
    for x in (da, db, dc, ws):
        x.free()
    assert not left.any(), "ticket counters are not back at zero"
    assert np.array_equal(got[:off], c0[:off])
    elem = {"bf16": oracle.BF16, "f16": oracle.F16, "e4m3": oracle.E4M3, "e5m2": oracle.E5M2,
            "e4m3e5m2": (oracle.E4M3, oracle.E5M2), "e5m2e4m3": (oracle.E5M2, oracle.E4M3)}[op]
    for i in range(batch):
        gv, ov = got[off + i * sc:][:m * ldc].reshape(m, ldc), c0[off + i * sc:][:m * ldc].reshape(m, ldc)
        assert np.array_equal(gv[:, n:], ov[:, n:]), "wrote into C's row padding"
        ref, val, scale = oracle.ref_gemm_ex(a[i * sa:][:m * lda].copy(), b[i * sb:][:brows * ldb].copy(), m, n, k, layout=layout, lda=lda, ldb=ldb, alpha=alpha, beta=beta,
                                             c_old=None if beta == 0.0 else ov[:, :n].copy(), out_f32=out_f32, elem=elem)
        f8_unit = esz == 1 and not tile.endswith("w")              # (widened operands: the sums of the 16-bit kernels)
        if out_f32:
            tol = ((oracle.floor_coeff_f8(k) + 2.0 ** -23) if f8_unit else (k / 16.0 + 4.0) * 2.0 ** -24) * scale + 1e-45
            assert (np.abs(gv[:, :n].astype(np.float64) - val) <= tol).all()
        else:
            s = oracle.compare(gv[:, :n].copy(), ref, val, scale, k, elem=oracle.F16 if op == "f16" else oracle.BF16,
                               coeff=oracle.floor_coeff_f8(k) if f8_unit else None)
            assert s["n_fail"] == 0, s
            if esz == 2:
                oracle.assert_parity(s, name)


@pytest.mark.parametrize("layout", [NN, NT], ids=["nn", "nt"])
@pytest.mark.parametrize("op,tile", [(op, t) for op in OPS for t in TILES if (op not in ("bf16", "f16") or t != "64x64w")])
def test_tile_forms_at_their_edges(ctx, oracle, forms, op, tile, layout):
    bm, bn = TILES[tile]
    kt = 64 if op in ("bf16", "f16") else 128
    ch = kt // 8
    # K: the shortest, a chunk's and a K tile's edges, whole tiles only, and one entry around a full ring (at most 5 stages)
    for i, k in enumerate((ch, ch + 1, kt - 1, kt, kt + 1, 3 * kt, 4 * kt + ch, 5 * kt, 5 * kt + 1, 6 * kt + 3, 7 * kt, 8 * kt - 1)):
        check_form(ctx, oracle, forms, op, tile, layout, bm + (i % 3) - 1, bn + 1 - (i % 3), k, off=i % 2, pad=(0, 3, 8)[i % 3])
    check_form(ctx, oracle, forms, op, tile, layout, 1, ch, ch)
    check_form(ctx, oracle, forms, op, tile, layout, 2 * bm + 1, 9 * bn + 3, kt + 9, alpha=-1.25, beta=0.75)     # sweeps of 8 tile rows, ragged
    check_form(ctx, oracle, forms, op, tile, layout, 8 * bm + 5, 2 * bn - 1, kt, out_f32=True, alpha=0.5, beta=1.0, off=1)
    check_form(ctx, oracle, forms, op, tile, layout, bm + 1, bn + ch, 2 * kt + 5, batch=3, pad=1)
    for ks, k in ((2, 9 * kt), (3, 9 * kt + 1), (16, 64 * kt - 7)) if tile != "128x128" else ():                  # K ranges, the tail in the last
        check_form(ctx, oracle, forms, op, tile, layout, bm + 3, bn + 5, k, ks=ks, out_f32=ks == 3)


@pytest.mark.parametrize("layout", [NN, NT], ids=["nn", "nt"])
@pytest.mark.parametrize("ty,tile", [(ty, t) for ty in ("f32", "f64") for t in ("32x128", "64x64", "64x128", "128x128") if (ty, t) != ("f64", "128x128")])
def test_full_precision_forms_at_their_edges(ctx, oracle, forms, ty, tile, layout):
    bm, bn = TILES[tile]
    dt, kt = (np.float32, 32) if ty == "f32" else (np.float64, 16)
    es, ch = np.dtype(dt).itemsize, 16 // np.dtype(dt).itemsize

    def check(m, n, k, ks=1, off=0, pad=0, alpha=1.0, beta=0.0, batch=1):
        name = f"maize_tile_{ty}_{'nt' if layout == NT else 'nn'}_{tile}"
        print(f"form {name} {m}x{n}x{k} ks={ks} off={off} pad={pad} batch={batch} beta={beta}", flush=True)
        brows, bcols = (n, k) if layout == NT else (k, n)
        lda, ldb, ldc = k + pad, bcols + pad, n + pad
        sa, sb, sc = m * lda + pad, brows * ldb + pad, m * ldc + pad
        rng = np.random.default_rng(7)
        a, b, c0 = ((rng.random(off + batch * x) * 2 - 1).astype(dt) for x in (sa, sb, sc))
        da, db, dc = ctx.upload(a), ctx.upload(b), ctx.upload(c0)
        items = -(-m // bm) * -(-n // bn) * batch * ks
        ws = ctx.malloc(65536 + items * bm * bn * es)
        ws.fill(0)
        args = _ffi.GemmArgsT(a=da.ptr + off * es, arows=m, acols=k, b=db.ptr + off * es, brows=brows, bcols=bcols, c=dc.ptr + off * es,
                              crows=m, ccols=n, stride_a=sa, stride_b=sb, stride_c=sc, batch=batch, layout=layout, workspace=ws.ptr, ksplit=ks,
                              lda=lda, ldb=ldb, ldc=ldc, epi=2 if (alpha, beta) != (1.0, 0.0) else 0, alpha=alpha, beta=beta)
        kern = forms.kernel(name)
        mz.api.LoadedKernel(ctx, forms, kern, (256, 1, 1)).launch((items, 1, 1), args)
        ctx.sync()
        got, left = dc.download(dt), ws.download(np.uint32, 16384)
        _ffi.check(_ffi.lib().maize_hip_kernel_release(kern))
        for x in (da, db, dc, ws):
            x.free()
        assert not left.any(), "ticket counters are not back at zero"
        for i in range(batch):
            cut = lambda x, s, r, ld: x[off + i * s:][:r * ld].reshape(r, ld)
            gv, ov = cut(got, sc, m, ldc), cut(c0, sc, m, ldc)
            assert np.array_equal(gv[:, n:], ov[:, n:]), "wrote into C's row padding"
            hi, lo, ab = oracle.ref_gemm_wide(np.ascontiguousarray(cut(a, sa, m, lda)[:, :k]), np.ascontiguousarray(cut(b, sb, brows, ldb)[:, :bcols]), m, n, k, layout=layout)
            worst = oracle.check_wide(gv[:, :n], hi.reshape(m, n), lo.reshape(m, n), ab.reshape(m, n), k, alpha, beta, ov[:, :n])
            assert worst <= 1.0, worst

    # K: the shortest, a chunk's and a K tile's edges, whole tiles only, and one entry around a full ring (at most 5 stages)
    for i, k in enumerate((ch, ch + 1, kt - 1, kt, kt + 1, 3 * kt, 4 * kt + ch, 5 * kt, 5 * kt + 1, 6 * kt + 3, 7 * kt, 8 * kt - 1)):
        check(bm + (i % 3) - 1, bn + 1 - (i % 3), k, off=i % 2, pad=(0, 3, 8)[i % 3])
    check(1, ch, ch)
    check(2 * bm + 1, 9 * bn + 3, kt + 9, alpha=-1.25, beta=0.75)
    check(bm + 1, bn + ch, 2 * kt + 5, batch=3, pad=1)
    for ks, k in ((2, 9 * kt), (3, 9 * kt + 1), (16, 64 * kt - 7)) if tile != "128x128" else ():      # (never split)
        check(bm + 3, bn + 5, k, ks=ks)


@pytest.mark.parametrize("warm", [True, False], ids=["run-before", "first-call"])
def test_a_captured_form_in_k_ranges_equals_the_eager_one(ctx, warm):
    """A product whose form splits K, captured where the stream's workspace holds it and where the stream has none yet; between
    the replays a larger product runs on the stream and replaces the workspace.  Every replay has the bits of the eager call."""
    hip = _ffi.lib()                                          # (the HIP runtime's own functions, through the library that links it)

    def call(f, *args):
        assert getattr(hip, f)(*args) == 0, f

    cus = ctx.info()["compute_units"]
    m, n, k = 64, 64, 1999
    a, b = mz.gen.uniform_bf16(m * k, 5), mz.gen.uniform_bf16(k * n, 6)
    one = np.full(512 * 8192, 0x3F80, np.uint16)
    da, db, dla, dlb = ctx.upload(a), ctx.upload(b), ctx.upload(one), ctx.upload(np.concatenate([one, one]))
    dc, dlc = ctx.malloc(m * n * 4), ctx.malloc(512 * 1024 * 4)
    desc = mz.gemm_ex_desc(mz.Matrix(da, m, k), mz.Matrix(db, k, n), mz.Matrix(dc, m, n), out_type=mz.OUT_F32)
    larger = mz.gemm_ex_desc(mz.Matrix(dla, 512, 8192), mz.Matrix(dlb, 8192, 1024), mz.Matrix(dlc, 512, 1024), out_type=mz.OUT_F32)
    form, grows = mz.gemm_form(desc, cus), mz.gemm_form(larger, cus)
    assert form["ksplit"] > 1 and 2 * form["workspace_bytes"] < grows["workspace_bytes"], (form, grows)
    other = ctx.stream()
    ctx.gemm_bf16(desc, other)
    ctx.sync(other)
    want = dc.download(np.float32)
    fa, fb = ((x.astype(np.uint32) << 16).view(np.float32).astype(np.float64) for x in (a, b))
    fa, fb = fa.reshape(m, k), fb.reshape(k, n)
    assert (np.abs(want.reshape(m, n) - fa @ fb) <= (k / 16.0 + 4.0) * 2.0 ** -24 * (np.abs(fa) @ np.abs(fb))).all()
    s, graph, run = ctx.stream(), C.c_void_p(), C.c_void_p()
    if warm:
        ctx.gemm_bf16(desc, s)
        ctx.sync(s)
    call("hipStreamBeginCapture", s, 1)
    ctx.gemm_bf16(desc, s)
    call("hipStreamEndCapture", s, C.byref(graph))
    nodes = C.c_size_t()
    call("hipGraphGetNodes", graph, None, C.byref(nodes))
    assert nodes.value == 1
    call("hipGraphInstantiate", C.byref(run), graph, None, None, C.c_size_t(0))
    for i in range(3):
        dc.fill(0)
        ctx.sync()
        print(f"replay {i}", flush=True)
        call("hipGraphLaunch", run, s)
        ctx.sync(s)
        assert np.array_equal(dc.download(np.float32), want)
        ctx.gemm_bf16(larger, s)
        ctx.sync(s)
        assert (dlc.download(np.float32) == 8192.0).all()
    call("hipGraphExecDestroy", run)
    call("hipGraphDestroy", graph)
    ctx.stream_destroy(s)
    ctx.stream_destroy(other)
    for x in (da, db, dla, dlb, dc, dlc):
        x.free()


@pytest.mark.parametrize("layout", [NN, NT], ids=["nn", "nt"])
@pytest.mark.parametrize("op,tile", [("bf16", "32x128"), ("bf16", "64x64"), ("bf16", "64x128"), ("bf16", "128x128"), ("e4m3", "32x128"), ("e4m3", "64x64"),
                                     ("e4m3", "64x64w"), ("e4m3", "64x128"), ("e4m3", "128x128")])
def test_every_count_of_k_tiles(ctx, oracle, forms, op, tile, layout):
    """One K tile to two rounds of the three to five ring stages and a ragged one behind: each count of entries that the requests
    (one by one or in pairs), the one without a partner and the stage of the tail can meet.  128 x 128: with every row on a
    128-byte line (single requests) and with none there (pairs)."""
    bm, bn = TILES[tile]
    kt, es = (64, 2) if op == "bf16" else (128, 1)
    met = set()
    for entries in range(1, 13):
        # (a row-major B whose rows are no whole dwords makes its last whole K tile a tail: bn + 5 columns, but not bn + 4)
        for more, n in ((0, bn + 4), (9, bn + 5)) + (((0, bn + 5),) if layout == NN else ()):
            k = entries * kt + more
            tail = k % kt != 0 or (layout == NN and n * es % 4 != 0)
            met.add((entries - (1 if tail and not more else 0), tail))
            for lines in (True, False) if tile == "128x128" else (False,):
                check_form(ctx, oracle, forms, op, tile, layout, bm - 3, n, k, off=0 if lines else entries % 2, pad=-k % kt if lines else 1 - entries % 2 + more % 2)
    assert met >= {(nd, tail) for nd in range(1, 13) for tail in (False, True)}, met        # by direct loads, and whether a tail follows
