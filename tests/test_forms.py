"""The launcher's own forms without a device: what their code object contains, and the LDS layouts they add."""
import os
import random
import re
import shutil
import subprocess

import pytest

import maize_amd as mz

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HSACO = os.path.join(os.path.dirname(mz.LIB_PATH), "maize_forms_gfx950.hsaco")
OBJDUMP = shutil.which("llvm-objdump") or "/opt/rocm/llvm/bin/llvm-objdump"

MAPS = r"""
#include <cstdio>
#include <set>
#include "maps.hpp"
using namespace maize::maps;
// a pass (32 lanes, 8 bytes each) of a transposing read hits each of the 64 banks once
static bool free_of_conflicts(const unsigned (&off)[64]) {
    for (int p = 0; p < 64; p += 32) {
        std::set<unsigned> banks;
        for (int l = p; l < p + 32; ++l) for (unsigned b = 0; b < 8; b += 4) if (!banks.insert((off[l] + b) / 4 % 64).second) return false;
    }
    return true;
}
int main() {
    std::set<unsigned> seen, seen8;
    for (unsigned pc = 0; pc < 8; ++pc) for (unsigned l = 0; l < 64; ++l) {
        if (sk64_offset(sk64_piece_row(pc, l), sk64_piece_chunk(pc, l)) != pc * 1024 + l * 16 || !seen.insert(sk64_piece_row(pc, l) * 8 + sk64_piece_chunk(pc, l)).second) return 1;
        if (sk8s_offset(sk8s_piece_row(pc, l), sk8s_piece_chunk(pc, l)) != pc * 1024 + l * 16 || !seen8.insert(sk8s_piece_row(pc, l) * 4 + sk8s_piece_chunk(pc, l)).second) return 2;
    }
    for (unsigned cg = 0; cg < 4; ++cg) for (unsigned k = 0; k < 2; ++k) for (unsigned h = 0; h < 2; ++h) {
        unsigned off[64], off8[64];
        for (unsigned l = 0; l < 64; ++l) {
            const unsigned q = l & 15, g = l >> 4;
            off[l] = sk64_tr_offset(cg, 0, l) + 4096 * k + 512 * h;
            const unsigned row = 32 * k + 8 * g + 4 * h + q / 4, col = 16 * cg + 4 * (q % 4);
            if (off[l] != sk64_offset(row, col >> 3) + (col & 7) * 2) return 3;
            off8[l] = sk8s_tr_offset(cg, 0, 0, l) + 4096 * k + 512 * h;
            const unsigned row8 = 64 * k + 16 * g + 8 * h + q / 2, col8 = 16 * cg + 8 * (q % 2);
            if (off8[l] != sk8s_offset(row8, col8 >> 4) + (col8 & 15)) return 4;
        }
        if (!free_of_conflicts(off) || !free_of_conflicts(off8)) return 5;
    }
    // 4- and 8-byte elements, 64 and 128 columns: every chunk once, and the reads of a pass (64 or 32 lanes) on banks of their own
    for (unsigned es : {4u, 8u}) for (unsigned bn : {64u, 128u}) {
        const unsigned rb = es * bn, rows = 128 / es, ch = 16 / es;
        std::set<unsigned> all;
        for (unsigned pc = 0; pc < bn / 8; ++pc) for (unsigned l = 0; l < 64; ++l) {
            const unsigned row = we_piece_row(rb, pc, l), chunk = we_piece_chunk(es, rb, pc, l);
            if (we_offset(es, rb, row, chunk * ch) != pc * 1024 + l * 16 || row >= rows || chunk * 16 >= rb || !all.insert(row * 256 + chunk).second) return 7;
        }
        if (all.size() != bn * 8) return 8;
        for (unsigned cg = 0; cg < bn / 16; ++cg) for (unsigned kh = 0; kh < 2; ++kh) for (unsigned e = 0; e < ch; ++e) {
            std::set<unsigned> banks, cols;
            for (unsigned l = 0; l < 64; ++l) {
                if (es == 8 && l % 32 == 0) banks.clear();
                const unsigned off = we_read(es, rb, cg, l) + (kh * rows / 2 + e) * rb;
                if (off != we_offset(es, rb, kh * rows / 2 + ch * (l >> 4) + e, 16 * cg + we_column(es, l))) return 9;
                for (unsigned b = 0; b < es; b += 4) if (!banks.insert((off + b) / 4 % 64).second) return 10;
                cols.insert(we_column(es, l));
            }
            if (cols.size() != 16) return 11;
        }
    }
    return seen.size() == 64 * 8 && seen8.size() == 128 * 4 ? 0 : 6;
}
"""


def test_the_64_column_tiles_of_a_row_major_b_are_whole_and_free_of_bank_conflicts(tmp_path):
    src, exe = tmp_path / "maps.cpp", tmp_path / "maps"
    src.write_text(MAPS)
    subprocess.run(["g++", "-O1", "-std=c++17", "-I", os.path.join(ROOT, "maize_amd", "csrc", "kernels"), "-o", str(exe), str(src)], check=True)
    assert subprocess.run([str(exe)]).returncode == 0


LINES = r"""
#include "maps.hpp"
using namespace maize::maps;
// the K tiles of a row that reach into a second line, in rows of 1024 (none, every other, more)
static unsigned counted(unsigned long long start, unsigned long long pitch) {
    unsigned n = 0;
    for (unsigned r = 0; r < 1024; ++r) n += (start + r * pitch) % 128 != 0;
    return n == 0 ? 0 : n <= 512 ? 1 : 2;
}
int main() {
    for (unsigned pitch = 1; pitch < 600; ++pitch) if (off_lines(1u << 20, pitch, 0) != counted(1u << 20, pitch)) return 1;
    for (unsigned start = 1; start < 128; ++start) if (off_lines(start, 256, 0) == 0 || off_lines(0, 256, start) == 0) return 2;
    if (off_lines(128, 384, 1u << 30) != 0) return 3;
    // rows on lines: single requests, whatever a row-major B's do; N x K: half of the rows have to share lines
    for (unsigned b = 0; b < 3; ++b) if (in_pairs(false, 0, b) || !in_pairs(false, 1, b) || !in_pairs(false, 2, b)) return 4;
    for (unsigned a = 0; a < 3; ++a) for (unsigned b = 0; b < 3; ++b) if (in_pairs(true, a, b) != (a + b >= 2)) return 5;
    return 0;
}
"""


def test_tiles_of_128_by_128_ask_in_pairs_only_where_rows_share_lines(tmp_path):
    """Rows on 128-byte lines have nothing to share, and pairs then cost up to 5 %."""
    src, exe = tmp_path / "lines.cpp", tmp_path / "lines"
    src.write_text(LINES)
    kdir = os.path.join(ROOT, "maize_amd", "csrc", "kernels")
    subprocess.run(["g++", "-O1", "-std=c++17", "-I", kdir, "-o", str(exe), str(src)], check=True)
    assert subprocess.run([str(exe)]).returncode == 0
    text = open(os.path.join(kdir, "gemm_tile.hpp")).read()
    assert "const bool pairs = BY_LINES && maps::in_pairs(NT, off(p.a, lda, p.stride_a), off(p.b, ldb, p.stride_b));" in text
    assert re.search(r"\} else if \(pairs\) \{\s+constexpr bool PAIR = true;\s+constexpr int NS = RING;\s+#include \"gemm_tile_ring.hpp\"\s+\} else \{\s+constexpr bool PAIR = false;", text)


@pytest.mark.skipif(not (os.path.exists(OBJDUMP) and os.path.exists(HSACO)), reason="needs the ROCm llvm-objdump and the built code object")
def test_form_kernels_keep_to_registers_and_plain_stores():
    text = subprocess.run([OBJDUMP, "-d", "--mcpu=gfx950", HSACO], check=True, capture_output=True, text=True).stdout
    names = re.findall(r"^[0-9a-f]+ <(maize_[A-Za-z0-9_]+)>:", text, re.M)
    assert len(names) >= 40
    for banned in ("scratch_", "v_pk_add_f32", "v_pk_mul_f32", "v_pk_fma_f32", "s_dcache_" + "wb", "s_sto" + "re", "s_ato" + "mic"):
        assert "\t" + banned not in text, banned


@pytest.mark.skipif(not (os.path.exists(OBJDUMP) and os.path.exists(HSACO)), reason="needs the ROCm llvm-objdump and the built code object")
def test_no_register_that_a_fragment_read_is_still_filling_is_touched():
    """The fragment reads are assembly statements, so the compiler takes their registers as written at once: where it runs out
    of registers it may copy one before its data is there (128 x 128 tiles of 16-bit operands at two workgroups per compute
    unit did, and gave wrong results).  Every kernel must wait first."""
    text = subprocess.run([OBJDUMP, "-d", "--mcpu=gfx950", HSACO], check=True, capture_output=True, text=True).stdout

    def regs(s):
        return {(kind, i) for kind, lo, hi, one in re.findall(r"\b([va])(?:\[(\d+):(\d+)\]|(\d+)\b)", s)
                for i in (range(int(lo), int(hi) + 1) if lo else [int(one)])}

    kernel, filling, reads, early = None, set(), 0, []
    for line in text.splitlines():
        head = re.match(r"^[0-9a-f]+ <(maize_\w+)>:", line)
        if head:
            kernel, filling = head.group(1), set()
        ins = re.match(r"^\t(\S+)\s*(.*?)\s*//", line)
        if not ins:
            continue
        op, args = ins.groups()
        if op == "s_waitcnt" and "lgkmcnt(0)" in args:
            filling = set()
        elif not op.startswith("s_"):
            if regs(args) & filling:
                early.append((kernel, line.split("//")[0].strip()))
            if op.startswith("ds_read"):
                reads += 1
                filling |= regs(args.split(",")[0])
    assert reads > 1000 and not early, early[:8]


SIZE = {mz.IN_BF16: 2, mz.IN_F16: 2, mz.IN_E4M3: 1, mz.IN_E5M2: 1, mz.IN_E4M3_E5M2: 1, mz.IN_E5M2_E4M3: 1, mz.IN_F32: 4, mz.IN_F64: 8}
TAG = {mz.IN_BF16: "bf16", mz.IN_F16: "f16", mz.IN_E4M3: "e4m3", mz.IN_E5M2: "e5m2", mz.IN_E4M3_E5M2: "e4m3e5m2", mz.IN_E5M2_E4M3: "e5m2e4m3", mz.IN_F32: "f32", mz.IN_F64: "f64"}


def describe(m, n, k, nt=False, in_type=mz.IN_BF16, batch=1, **how):
    a, b, c = (mz.GlobalMatrix(p << 44, *s) for p, s in ((1, (m, k)), (2, (n, k) if nt else (k, n)), (3, (m, n))))
    return mz.gemm_ex_desc(a, b, c, layout=mz.LAYOUT_NT if nt else mz.LAYOUT_NN, batch=batch, in_type=in_type, stride_a=m * k, stride_b=k * n, stride_c=m * n, **how)


@pytest.mark.parametrize("seed", range(4))
def test_what_a_form_is_launched_with(seed):
    """Drawn products: the grid covers C once per K range and fits a launch, no range is empty, workspace and ticket counters hold
    what the kernel addresses, 8-bit operands are widened where the plan's kernel widens them and nowhere else, and the few-row
    kernels' K ranges are kept."""
    rng = random.Random(seed)
    taken = split = pinned = 0
    for i in range(3600):
        m, n, k = (max(1, int(2 ** rng.uniform(0, hi)) // g * g) for hi, g in ((rng.choice([6, 13]), rng.choice([1, 8])), (15, rng.choice([1, 8, 16, 64])), (14, rng.choice([1, 8, 16, 64]))))
        in_type, nt, batch, cus = rng.choice(list(SIZE)), rng.random() < 0.5, rng.choice([1, 1, 1, 3, 40]), rng.choice([256, 256, 304, 64, 1])
        if i >= 3000:                                            # few rows against a row-major B
            m, n, k, in_type, nt = rng.randint(1, 64), int(2 ** rng.uniform(8, 15)), 32 * rng.randint(8, 256), rng.choice([mz.IN_BF16, mz.IN_F16]), False
        x = describe(m, n, k, nt, in_type, batch)
        form, plan = mz.gemm_form(x, cus), mz.gemm_plan(x, compute_units=cus)
        if form is None:
            continue
        es = SIZE[in_type]
        got = re.fullmatch(r"maize_tile_([a-z0-9]+)_(nn|nt)_(\d+)x(\d+)(w?)", form["kernel"])
        assert got and got[1] == TAG[in_type] and got[2] == ("nt" if nt else "nn"), form
        bm, bn, ks = int(got[3]), int(got[4]), form["ksplit"]
        tiles, steps = -(-m // bm) * -(-n // bn) * batch, -(-k * es // 128)
        assert form["grid"] == (tiles * ks, 1, 1) and form["block"] == (256, 1, 1) and tiles * ks < 1 << 24
        assert bool(got[5]) == (es == 1 and "_wave32" in plan["kernel"])
        assert k * es >= 16 and (nt or n * es >= 16)
        taken += 1
        if ks == 1:
            assert form["workspace_bytes"] == 0
        else:
            per = -(-steps // ks)
            assert (ks - 1) * per < steps and tiles <= 16384
            assert form["workspace_bytes"] == 65536 + tiles * ks * bm * bn * (8 if es == 8 else 4) < 1 << 32
            split += 1
        if "_skinny_nn" in plan["kernel"] and es == 2:
            pinned += 1
            assert ks == max(1, plan["ksplit"]) and (ks == 1 or -(-(-(-k // 32)) // ks) * 32 == -(-steps // ks) * 64)
    assert taken > 1000 and split > 200 and pinned > 20, (taken, split, pinned)


@pytest.mark.parametrize("in_type", list(SIZE), ids=list(TAG.values()))
def test_where_no_form_can_run(in_type):
    """Less than one 16-byte chunk of K, or of a row of a row-major B; extents and leading dimensions of 2^21 elements."""
    ch = 16 // SIZE[in_type]
    for nt in (False, True):
        assert mz.gemm_form(describe(40, 50, ch, nt, in_type)) is not None
        assert ch == 1 or mz.gemm_form(describe(40, 50, ch - 1, nt, in_type)) is None
        assert (mz.gemm_form(describe(40, ch - 1, 50, nt, in_type)) is None) == (not nt)
        assert mz.gemm_form(describe(40, ch, 50, nt, in_type)) is not None
        for ld in ("lda", "ldb", "ldc"):
            assert mz.gemm_form(describe(40, 50, 60, nt, in_type, **{ld: (1 << 21) - 1})) is not None
            try:
                assert mz.gemm_form(describe(40, 50, 60, nt, in_type, **{ld: 1 << 21})) is None
            except mz.MaizeError:                                # (some are refused altogether: there is one fp64 kernel)
                assert in_type == mz.IN_F64


@pytest.mark.skipif(not (os.path.exists(OBJDUMP) and os.path.exists(HSACO)), reason="needs the ROCm llvm-objdump and the built code object")
def test_no_k_step_is_written_out_that_none_can_reach():
    """A ring's code: two K steps in the loop and one each for the last entries.  The loop ends with NS + 1 direct entries left, pairs
    (five stages) with five, and there may be a tail."""
    text = subprocess.run([OBJDUMP, "-d", "--mcpu=gfx950", HSACO], check=True, capture_output=True, text=True).stdout
    found = {}
    for line in text.splitlines():
        head = re.match(r"^[0-9a-f]+ <(maize_\w+)>:", line)
        if head:
            kernel = head.group(1)
            found[kernel] = 0
        elif "\tv_mfma_" in line:
            found[kernel] += 1
    for kernel, got in found.items():
        op, bm, bn, wide = re.fullmatch(r"maize_tile_([a-z0-9]+)_n[nt]_(\d+)x(\d+)(w?)", kernel).groups()
        if op in ("f32", "f64") or wide:
            continue
        step = int(bm) * int(bn) // 1024 * (2 if op in ("bf16", "f16") else 1)         # matrix instructions of a wave in a K tile
        last = {("32", "128"): [6], ("64", "64"): [7], ("64", "128"): [5], ("128", "128"): [6, 6]}[bm, bn]
        assert got == step * sum(2 + n for n in last), (kernel, got)
