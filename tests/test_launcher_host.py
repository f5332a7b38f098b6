"""The launcher (maize_amd/csrc/shim.cpp) on a model of the HIP runtime (tests/cpu/fake_hip.cpp): what it allocates, frees and
launches, eagerly and while a stream is captured into a graph.  No device."""
import ctypes as C
import os
import subprocess
from types import SimpleNamespace

import pytest

import maize_amd as mz
from maize_amd import _ffi

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "maize_amd", "csrc")
STREAM, OTHER = C.c_void_p(0x1000), C.c_void_p(0x2000)


@pytest.fixture(scope="module")
def model(tmp_path_factory):
    so = tmp_path_factory.mktemp("model") / "libmodel.so"
    src = [os.path.join(CSRC, f) for f in ("shim.cpp", "dispatch.cpp", "forms.cpp")] + [os.path.join(ROOT, "tests", "cpu", "fake_hip.cpp")]
    subprocess.run(["g++", "-O1", "-std=c++17", "-fPIC", "-shared", "-Wl,-Bsymbolic", "-Wl,--no-undefined", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                    "-I" + os.path.join(ROOT, "include"), "-I" + CSRC, "-o", str(so)] + src, check=True)
    lib = C.CDLL(str(so))
    lib.fake_log.restype = lib.maize_hip_last_error.restype = C.c_char_p
    lib.fake_memory.argtypes = [C.c_size_t]
    return lib


class Device:
    """One context on the model."""

    def __init__(self, lib):
        self.lib, self.ctx = lib, C.c_void_p()
        lib.fake_memory(1 << 40)
        assert lib.maize_hip_ctx_create(0, C.byref(self.ctx)) == 0
        lib.fake_clear()

    def close(self):
        assert self.lib.maize_hip_ctx_destroy(self.ctx) == 0

    def events(self):
        """What was logged since the last call."""
        out = []
        for line in self.lib.fake_log().decode().splitlines():
            w = line.split()
            node = w[0] == "node"
            w = w[node:]
            if w[0] == "launch":
                out.append(SimpleNamespace(what="launch", node=node, stream=int(w[1]), kernel=w[2], grid=int(w[3]), ksplit=int(w[4]), workspace=int(w[5])))
            else:
                out.append(SimpleNamespace(what=w[0], node=node, at=int(w[1]), rest=[int(x) for x in w[2:]]))
        self.lib.fake_clear()
        return out

    def product(self, x, stream=STREAM):
        rc = self.lib.maize_hip_gemm_bf16_ex(self.ctx, C.byref(x), None, stream)
        assert rc == 0, (rc, self.lib.maize_hip_last_error())
        return self.events()

    def captured(self, x, stream=STREAM):
        self.lib.fake_capture(stream)
        ev = self.product(x, stream)
        assert self.lib.fake_end_capture(stream) == 1, "the capture was spoilt"
        return ev


@pytest.fixture
def dev(model):
    d = Device(model)
    yield d
    d.close()


def product(m, n, k, nt=False, in_type=mz.IN_BF16, batch=1, **how):
    brows, bcols = (n, k) if nt else (k, n)
    if batch > 1:
        how.update(stride_a=m * k, stride_b=k * n, stride_c=m * n)
    a, b, c = (mz.GlobalMatrix(p << 32, *s) for p, s in ((16, (m, k)), (32, (brows, bcols)), (48, (m, n))))
    return mz.gemm_ex_desc(a, b, c, layout=mz.LAYOUT_NT if nt else mz.LAYOUT_NN, batch=batch, in_type=in_type, **how)


def launches(events):
    return [e for e in events if e.what == "launch"]


# (the registry's kernel of the first needs scratch: it splits K; the second's needs none, its form 16.8 MB)
FEW_ROWS, GROWS = product(16, 14336, 4096), product(267, 4320, 3648, nt=True)


def test_a_buffer_that_a_graph_holds_is_not_freed_when_the_stream_needs_a_larger_one(dev):
    dev.product(FEW_ROWS)
    held = {e.workspace for e in launches(dev.captured(FEW_ROWS)) if e.workspace}
    assert held
    grown = dev.product(GROWS)
    assert launches(grown)[0].ksplit > 1 and any(e.what == "malloc" for e in grown), "the larger product was meant to need a larger buffer"
    assert not [e for e in grown if e.what == "free" and e.at in held]
    # ... the eager product that follows is off the graph's buffer, and a graph taken now holds the larger one
    assert not {e.workspace for e in launches(dev.product(FEW_ROWS))} & held
    held |= {e.workspace for e in launches(dev.captured(FEW_ROWS))}
    assert len(held) == 2
    assert not [e for e in dev.product(product(512, 1024, 16384)) if e.what == "free" and e.at in held]


def test_a_buffer_that_no_graph_holds_is_given_back(dev):
    first = launches(dev.product(FEW_ROWS))[0].workspace
    grown = dev.product(GROWS)
    assert [e.what for e in grown][:3] == ["wait", "free", "malloc"] and grown[1].at == first


def test_buffers_kept_for_graphs_go_with_the_stream_and_the_context(model):
    for close in ("stream", "context"):
        d = Device(model)
        made = []
        for stream in (STREAM, OTHER):
            for x in (FEW_ROWS, GROWS):
                made += [e.at for e in d.product(x, stream) if e.what == "malloc"]
                d.captured(x, stream)
        assert len(made) == 4
        gone = []
        if close == "stream":
            assert model.maize_hip_stream_destroy(d.ctx, STREAM) == 0
            gone = [e.at for e in d.events() if e.what == "free"]
            assert sorted(gone) == made[:2]
        d.close()
        assert sorted(gone + [e.at for e in d.events() if e.what == "free"]) == made


def route(events):
    return [(e.kernel, e.grid, e.ksplit) for e in launches(events)]


# a form in K ranges where the registry's kernel wants more scratch (packed copies), wants none, or is its twin; one without
# K ranges; a registry kernel in K ranges; and one with a reduce pass behind it
CAPTURED = [product(64, 64, 1999), GROWS, product(3, 4863, 4281), product(8, 7336, 4464, in_type=mz.IN_F32), product(150, 201, 333), FEW_ROWS, product(2048, 2048, 16384)]


@pytest.mark.parametrize("x", CAPTURED)
def test_a_captured_call_runs_what_the_eager_call_runs(model, x):
    """... with the same workspace where the stream has run it before, and with one of its own, zero before the graph first
    runs and not set by it, where it has not.  Neither spoils the capture."""
    warm, cold = Device(model), Device(model)
    eager = warm.product(x)
    again = warm.captured(x)
    assert route(again) == route(eager) and [e.what for e in again] == ["launch"] * len(again)
    assert [e.workspace for e in launches(again)] == [e.workspace for e in launches(eager)]
    first = cold.captured(x)
    assert route(first) == route(eager) and not model.fake_relaxed()
    for e in first:
        assert e.node == (e.what == "launch")
        if e.what == "set":
            assert e.at != STREAM.value and [f.at for f in first if f.what == "wait"] == [e.at]
    assert route(cold.product(x)) == route(eager)
    # grown within a capture: what earlier launches and the graph use stays
    cold.product(product(64, 64, 1999), OTHER)
    grown = cold.captured(x, OTHER)
    assert route(grown) == route(eager) and not [e for e in grown if e.what == "free"]
    warm.close()
    cold.close()


def test_growing_a_workspace_does_not_spoil_the_capture_of_another_stream(dev, model):
    model.fake_capture(OTHER)
    dev.product(FEW_ROWS)
    assert any(e.what == "free" for e in dev.product(GROWS))
    assert model.fake_end_capture(OTHER) == 1 and not model.fake_relaxed()


def test_a_product_whose_kernel_needs_no_device_memory_runs_when_there_is_none(dev, model):
    want = route(dev.product(GROWS))
    assert want[0][2] > 1                                        # a form in K ranges ...
    model.fake_memory(0)
    ran = launches(dev.product(GROWS, OTHER))
    assert len(ran) == 1 and ran[0].kernel == mz.gemm_plan(GROWS)["kernel"] and ran[0].workspace == 0
    assert model.hipGetLastError() == 0
    # ... one whose kernel needs scratch as well is an error, as it is for a kernel that is named
    assert model.maize_hip_gemm_bf16_ex(dev.ctx, C.byref(product(64, 64, 1999)), None, OTHER) == 2
    assert not launches(dev.events())


@pytest.mark.parametrize("x", [product(32768, 8, 9, batch=32768), product(1, 65536, 64, batch=32768, in_type=mz.IN_F32), product(32, 128, 64, batch=65535, in_type=mz.IN_F32),
                               product(4095 * 64, 64, 64, batch=4096, in_type=mz.IN_E4M3)])
def test_a_launch_stays_within_32_bits_of_work_items(dev, x):
    """Tiles that would make up 2^24 workgroups of 256, and a little fewer: the product runs, in a grid that a launch can have."""
    assert launches(dev.product(x))                              # (the model refuses what the runtime refuses)


# products that a form takes -- every tile, one K range and several, widened 8-bit operands, fp32 and fp64 -- and two that none takes
DESCRIBED = CAPTURED + [product(64, 64, 64), product(200, 1072, 368), product(544, 2472, 1112), product(1024, 3072, 1999), product(9, 2304, 2048), product(16, 14336, 4096, nt=True, in_type=mz.IN_E4M3),
                        product(128, 168, 296, in_type=mz.IN_E5M2_E4M3), product(1000, 1000, 1000, in_type=mz.IN_F64), product(1024, 4096, 4096, nt=True)]


@pytest.mark.parametrize("x", DESCRIBED)
def test_form_query_describes_the_launch(dev, x):
    form, plan, ran = mz.gemm_form(x), mz.gemm_plan(x), dev.product(x)
    first, bytes_ = launches(ran)[0], [e.rest[0] for e in ran if e.what == "malloc"]
    want = form or plan
    assert bytes_ == ([want["workspace_bytes"] * 3 // 2] if want["workspace_bytes"] else [])
    if form:
        assert (first.kernel, first.grid, max(1, first.ksplit)) == (form["kernel"], form["grid"][0], form["ksplit"])
        assert form["grid"][1:] == (1, 1) and form["block"] == (256, 1, 1) and len(launches(ran)) == 1
    else:
        assert first.grid == plan["grid"][0] * plan["grid"][1] * plan["grid"][2]


@pytest.mark.parametrize("x", [product(4453, 3712, 2432), product(816, 18448, 11456), product(1859, 8448, 9584, nt=True, in_type=mz.IN_E5M2), product(3191, 4992, 3840)])
def test_a_product_that_the_launcher_cuts_stays_cut(dev, x):
    """The cost model compares a form with the uncut kernel; the cut is 10 to 38 % ahead of the forms it had chosen here."""
    assert mz.gemm_tail_split(x) != (0, 0) and mz.gemm_form(x) is None
    ran = launches(dev.product(x))
    assert len(ran) >= 2 and all(e.kernel.startswith("maize_gemm_") for e in ran)


SLOWER_ON_A_FORM = [product(4624, 3360, 15632, nt=True), product(65, 8288, 14408), product(8936, 3368, 1024, in_type=mz.IN_E4M3, batch=8), product(781, 19008, 6656, nt=True),
                    product(192, 768, 5936, nt=True, batch=19), product(5904, 160, 1920, nt=True, batch=11), product(673, 13416, 14409, nt=True), product(768, 10432, 64, nt=True),
                    product(141, 4144, 6928, nt=True, in_type=mz.IN_F16, batch=4), product(128, 2752, 7040, nt=True, batch=11)]


@pytest.mark.parametrize("x", SLOWER_ON_A_FORM)
def test_products_that_a_form_slows_down_stay_on_the_registry_kernel(dev, x):
    """(25 to 84 % slower on the form that the model had chosen: operands beyond the L2s, one transposing copy taken for two, C
    written by a reduce pass that does not run, tiles at the edge that are split.)"""
    assert mz.gemm_form(x) is None and launches(dev.product(x))[-1].kernel.startswith("maize_")


SHORT_K = [product(7203, 17704, 16, in_type=mz.IN_F32), product(1280, 3216, 8, in_type=mz.IN_F32, batch=8), product(8544, 7372, 32, nt=True, in_type=mz.IN_F32),
           product(968, 4064, 112, in_type=mz.IN_F32, batch=32), product(4096, 15584, 32, nt=True, in_type=mz.IN_F64), product(240, 14280, 48, in_type=mz.IN_F64, batch=32)]


@pytest.mark.parametrize("x", SHORT_K)
def test_fp32_and_fp64_products_of_a_short_k_stay_on_the_registry_kernel(dev, x):
    """(8 to 23 % slower on the form: its tiles are the same, or nearly, and the ring is mostly prologue.)"""
    assert mz.gemm_form(x) is None
    ran = launches(dev.product(x))
    assert len(ran) == 1 and "_mt128_" in ran[0].kernel and ran[0].kernel == mz.gemm_plan(x)["kernel"]


@pytest.mark.parametrize("x", [product(7203, 17704, 15, in_type=mz.IN_F32), product(7203, 17702, 16, in_type=mz.IN_F32), product(1280, 3216, 8, in_type=mz.IN_F32, ldc=3217),
                               product(1280, 3216, 132, in_type=mz.IN_F32, batch=8), product(64, 3216, 16, in_type=mz.IN_F32), product(1024, 4096, 32, in_type=mz.IN_F64)])
def test_the_other_fp32_and_fp64_products_run_a_form(dev, x):
    """Rows that are no 16-byte material, a K tile more, fewer tiles."""
    assert "maize_tile_f" in mz.gemm_form(x)["kernel"]


def test_every_registry_kernel_has_a_cost(tmp_path):
    """A kernel whose name the cost model does not know would keep all its products; none does, and the table has a row for it."""
    src = tmp_path / "families.cpp"
    src.write_text(r'''
#include "forms.cpp"
using namespace maize;
int main() {
    for (uint32_t i = 0; i < kernel_count(); ++i) {
        const char* n = kernel_at(i).name;
        const FamilyOf f = family_of(n);
        const bool bits8 = std::strstr(n, "_e4m3") || std::strstr(n, "_e5m2");
        const bool rated = f.family == kWide || f.family == kAnyShape || f.family == kSkinnyNN || f.family == kSkinnyNT;
        if (f.family == kUnknown || (!rated && kRegistryCost[f.family][bits8].bm == 0u)) { std::puts(n); return 1; }
    }
    return 0;
}
''')
    exe = tmp_path / "families"
    subprocess.run(["g++", "-O1", "-std=c++17", "-I" + os.path.join(ROOT, "include"), "-I" + CSRC, "-o", str(exe), str(src), os.path.join(CSRC, "dispatch.cpp")], check=True)
    out = subprocess.run([str(exe)], capture_output=True, text=True)
    assert out.returncode == 0, out.stdout


def test_a_kernel_described_in_cpp_is_not_replaced_by_a_form(tmp_path):
    """include/maize_tile.hpp: a described mainloop launches its kernel also where the launcher, left the choice, would run a
    form (512 x 1024 x 1024)."""
    src = tmp_path / "described.cpp"
    src.write_text(r'''
#include <cstdio>
#include "maize_tile.hpp"
using namespace maize;
extern "C" const char* fake_log();
extern "C" void fake_memory(size_t);
int main() {
    fake_memory((size_t)1 << 40);
    Ctx ctx(0);
    const Matrix a = Matrix::make((BF16*)0x100000000, 512, 1024), b = Matrix::make((BF16*)0x200000000, 1024, 1024), c = Matrix::make((BF16*)0x300000000, 512, 1024);
    TracedKernel k = new_hip_kernel();
    k.with_launch_bounds_2d({256, 1});
    auto ring = k.alloc_aligned_shared<TilePair<Tile<BF16_128x64>, Tile<BF16_64x128>>, 4>(1024);
    const Wave wave{k.cx()};
    collective_aligned_row_panel_iter<128>(a, BlockX{k.cx()}).first.for_every_value([&](const RowPanel<128>& ap) {
        collective_aligned_col_panel_iter<128>(b, BlockY{k.cx()}).first.for_every_value([&](const ColPanel<128>& bp) {
            gemm_smem_multibuffer(Gfx950MfmaBf16F32_16x16x32{}, KTile<64>{}, ap, bp, ring, wave, 16).store(c);
        });
    });
    LoadedGemm g = k.finalize().compile(Gfx::Gfx950, ctx);
    g.launch();
    std::printf("%s\n%s", g.kernel_name().c_str(), fake_log());
}
''')
    exe = tmp_path / "described"
    cpp = [os.path.join(CSRC, f) for f in ("shim.cpp", "dispatch.cpp", "forms.cpp")] + [os.path.join(ROOT, "tests", "cpu", "fake_hip.cpp")]
    subprocess.run(["g++", "-O1", "-std=c++17", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include", "-I" + os.path.join(ROOT, "include"), "-I" + CSRC, "-o", str(exe), str(src)] + cpp, check=True)
    out = subprocess.run([str(exe)], capture_output=True, text=True, check=True).stdout
    assert mz.gemm_form(product(512, 1024, 1024)) is not None
    assert out.splitlines()[0] == "maize_gemm_bf16_t128_nn" and any(l.startswith("launch") and "maize_gemm_bf16_t128_nn" in l for l in out.splitlines()), out
