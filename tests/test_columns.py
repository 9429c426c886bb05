"""Index arithmetic of the fluid kernels (fortrancfd_amd/csrc/columns.hpp) on the host, for fields below and above
2^29 columns, where a byte offset from the start of a row no longer fits 32 bits: every address that a launch forms from its
slice's pointers and 32-bit offsets is the one that 64-bit indices give, and the slices cover the domain once."""
import subprocess

from fortrancfd_amd.build import CSRC

CHECK = r"""
#include <cstdio>
#include <initializer_list>
#include "columns.hpp"
using namespace fcfd;

// A stage update: every column is in one slice, and the offsets of its column, source and interface are what 64-bit
// indices give, counted from the slice's first block.  Columns are taken `step` apart.
static long stage(long nblk, long ncell, int lv, long most, long step) {
    const long S = ncell + 2 * lv;
    long bad = 0, next = 0;
    for_slices(int(nblk), S, most, [&](int b0, int n) {
        const StageSlice s = stage_slice(int(nblk), int(S), b0, n);
        const long first = long(s.first) * S, ffirst = long(s.first) * (ncell + 1);
        bad += first + s.col0 != next;
        next += s.ncol;
        bad += n > 1 && s.ncol > most;
        for (long k = 0; k < long(s.ncol); k = k + step < long(s.ncol) || k == long(s.ncol) - 1 ? k + step : long(s.ncol) - 1) {
            const unsigned c = s.col0 + unsigned(k);
            const int b = int(c / unsigned(S)), i = int(c - unsigned(b) * unsigned(S)) - lv;
            const long gb = s.first + b;                 // the block, and its source by 64-bit indices
            int sb, si, tb, ti;
            double sgn, tgn;
            ghost_source(s.left, s.right, int(ncell), b, i, sb, si, sgn);
            ghost_source(0, int(nblk - 1), int(ncell), int(gb), i, tb, ti, tgn);
            bad += sgn != tgn || s.first + sb != tb || si != ti;
            const unsigned sc = (unsigned(sb) * unsigned(S) + unsigned(lv + si)) * 8u;
            const unsigned fj = (unsigned(sb) * unsigned(ncell + 1) + unsigned(si)) * 8u;
            bad += first * 8 + long(sc) != (long(tb) * S + lv + ti) * 8;
            bad += ffirst * 8 + long(fj) != (long(tb) * (ncell + 1) + ti) * 8;
            bad += first * 8 + long(c * 8u) != (gb * S + lv + i) * 8;
        }
        return 0;
    });
    return bad + (next != nblk * S);
}

// The flux: every interface once, slices of blocks or of one block (as launch_flux makes them)
static long flux(long nblk, long ncell, int lv, long most) {
    const long S = ncell + 2 * lv, nif = ncell + 1;
    long bad = 0, next = 0;
    auto last = [&](long q0, long f0, long nb, long n) {        // the last interface of a launch
        const long g = nb * (n + 1) - 1;
        const unsigned bl = unsigned(g) / unsigned(n + 1), j = unsigned(g) - bl * unsigned(n + 1);
        const unsigned c0 = bl * unsigned(S) + unsigned(lv) + j - 1u;
        const long f = f0 + g, b = f / nif;
        bad += q0 * 8 + long((c0 + 3u) * 8u) != (b * S + lv + f % nif + 2) * 8;
        bad += f0 * 8 + long(unsigned(g) * 8u) != f * 8;
        bad += f0 != next;
        next = f + 1;
    };
    for_slices(int(nblk), S, most, [&](int b, int n) {
        if (S <= most) { last(b * S, b * nif, n, ncell); return 0; }
        return for_slices(int(nif), 1, most, [&](int j, int m) { last(b * S + j, b * nif + j, 1, m - 1); return 0; });
    });
    return bad + (next != nblk * nif);
}

int main() {
    long bad = 0, n = 0;
    for (int lv = 1; lv <= 4; ++lv) {
        // small domains in small slices, every column
        for (long ncell : {long(lv), lv + 1L, 17L, 64L})
            for (long nblk : {1L, 2L, 3L, 7L, 40L})
                for (long most : {1L, 20L, 64L, 200L, 1L << 28})
                    bad += stage(nblk, ncell, lv, most, 1), bad += lv == 3 ? flux(nblk, ncell, lv, most) : 0, ++n;
        // more than 2^29 columns (a stage's blocks are short there: longer ones do not fit the memory of a card)
        for (long ncell : {long(lv), 17L, 36L, 4096L})
            bad += stage(((1L << 29) + (1L << 20)) / (ncell + 2 * lv), ncell, lv, SLICE, 4999), ++n;
    }
    for (long ncell : {3L, 36L, 4096L}) bad += flux((3L << 28) / ncell, ncell, 3, SLICE), ++n;
    for (long ncell : {(1L << 28) - 6, (1L << 28) - 5, (1L << 29) + 77, (1L << 30) + 1}) bad += flux(1, ncell, 3, SLICE), ++n;
    std::printf("%ld domains, %ld wrong addresses\n", n, bad);
    return bad != 0;
}
"""


def test_addresses(tmp_path):
    src, exe = tmp_path / "check.cpp", tmp_path / "check"
    src.write_text(CHECK)
    subprocess.run(["g++", "-O1", "-std=c++17", f"-I{CSRC}", str(src), "-o", str(exe)], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True)
    print(r.stdout)
    assert r.returncode == 0, r.stdout
