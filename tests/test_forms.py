"""The launcher's own forms without a device: what their code object contains, and the LDS layouts they add."""
import os
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
