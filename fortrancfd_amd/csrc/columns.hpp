// columns.hpp -- index arithmetic of the ghost-padded columns, for the kernels and the host.
//
// A kernel addresses row v of a field by a 64-bit pointer that is the same in all lanes (scalar registers) and a
// lane's offset in bytes, 32 bits wide: one instruction's address, where 64-bit offsets take two additions a lane
// and row.  A field may have 2^29 columns and more (4 GB a row).  Kernels whose columns grow with the lane start
// their pointers at the workgroup's first column (column_bytes); the flux and the stage update, which have no
// registers to spare for pointers of their own (formed in the kernel they cost 0.4 % and 1.2 % at 262,144 cells),
// are launched over slices of at most 2^28 columns.
#pragma once

#if defined(__HIPCC__)
#include <hip/hip_runtime.h>
#define FCFD_IDX __host__ __device__ inline
#else
#define FCFD_IDX static inline
#endif

namespace fcfd {

// Source column of padded column (b, i): interior -> itself; wall ghost (blocks left and right: the domain's
// first and last) -> mirrored interior cell with momentum negated (SRC/boundary.f90:152-199); block ghost ->
// the neighbour block's interior cell (SRC/block.f90:490-497).
FCFD_IDX void ghost_source(int left, int right, int ncell, int b, int i, int &sb, int &si, double &sgn) {
    sb = b; si = i; sgn = 1.0;
    if (i < 0) {
        if (b == left) { si = -i - 1; sgn = -1.0; }
        else { sb = b - 1; si = ncell + i; }
    } else if (i >= ncell) {
        if (b == right) { si = 2 * ncell - 1 - i; sgn = -1.0; }
        else { sb = b + 1; si = i - ncell; }
    }
}

// Offset of column c in a row that starts at column first <= c.
FCFD_IDX unsigned column_bytes(unsigned c, unsigned first) { return (c - first) * 8u; }

constexpr long SLICE = 1L << 28;

// f(b, n) over consecutive ranges of n blocks of `width` columns, at most `most` columns each (at least a block),
// until one fails (is not 0); its result.
template <class F>
auto for_slices(int nblk, long width, long most, F f) -> decltype(f(0, 0)) {
    const int per = width < most ? int(most / width < nblk ? most / width : nblk) : 1;
    decltype(f(0, 0)) e{};
    for (int b = 0; b < nblk && int(e) == 0; b += per) {
        e = f(b, nblk - b < per ? nblk - b : per);
        if (nblk - b <= per) break;
    }
    return e;
}

// A stage's slice of the blocks b .. b + n - 1: its fields start at block `first`, one block earlier where there is
// one (the first block's left ghosts read it), so that no offset is negative; its columns are col0 .. col0 + ncol - 1
// from there; left and right number the walls' blocks from there (-1 or beyond: not reached).
struct StageSlice {
    int first, left, right;
    unsigned col0, ncol;
};
FCFD_IDX StageSlice stage_slice(int nblk, int S, int b, int n) {
    const int first = b > 0 ? b - 1 : 0;
    return StageSlice{first, first == 0 ? 0 : -1, nblk - 1 - first, unsigned(b - first) * unsigned(S),
                      unsigned(n) * unsigned(S)};
}

}  // namespace fcfd
