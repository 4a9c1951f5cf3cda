// Batched Newton-Raphson kernel on the block form of the factorisation (blocks.hpp).
#pragma once

#include <hip/hip_runtime.h>

#include <cstddef>

namespace pfgpu_block {

struct BArgs {
    int n, nlev, nblev, m, zpair;
    int nlds, nspill;  // value pairs in LDS, and spilled ones, per instance
    int single_slack, ninst, max_iter, fresh, fdpf, chain;
    int nrow, njd, njc;  // Ybus rows assembled, jagged-diagonal columns, constant blocks
    int nent;            // off-diagonal Ybus entries of those rows
    int slack_x, slack_bus, nnzY;
    int sh_off, v_off;   // byte offsets in dynamic LDS: workgroup state; V of the instances (-1: read from memory)
    double tol, stall_tol, growth_tau;
    const int *bus_y, *tail_src;
    const int4* rows;        // {bus, pair word, CSC position and target word of the diagonal}
    const int* jd_ptr;       // [njd + 1]
    const int2* jd;          // {column bus, target word}
    const int* jd_pos;
    const int4 *jd_jidx, *row_jidx;
    const int *y_row, *y_ent;  // per CSC position: row bus; entry (jagged diagonals, then nent + row), -1: none
    const int* jc_dst;
    const int4* jc_jidx;
    const double* jc_val;
    // unit streams, the first unit of each wave, and the levels at which it has any ([wave][words])
    const int4 *fs, *bs;
    const int *f_at, *b_at;
    const unsigned long long *f_mask, *b_mask;
    int f_words, b_words;
    const double *Yjd, *Yrow;  // shared Ybus values in the order of jd and of rows' diagonals, or null
    const double* w;
    const double* Yx;
    long long y_stride;      // doubles between instances (0 = shared)
    const int *dptr, *dpos;
    const double* dval;
    const double* S;
    long long s_stride;
    double* V;               // [rows][n] complex
    double *Va, *Vm;         // per resident instance
    double* Vprev;           // V at the last assembly that a step followed (with Jx_last)
    void* Xg;                // spilled pairs [workgroup][nspill][G]
    int *iters, *status, *flags;
    double* Jx_last;
    long long jx_row;
    const int* imap;
    long long nrows;
    unsigned long long* phase_t;
    int* queue;
    long long ngroups;
};

// Workgroup state in dynamic LDS after the value pairs. Layout: part[waves][G], slack[G], flast[G],
// dval[G][kEdits][2] (doubles), then done, it, status, piv, grow [G], dent[G][kEdits], drow[G][kEdits],
// nd, d0 [G], ndone, grp (ints); kEdits Ybus edits of an instance are kept there.
constexpr int kEdits = 8;
constexpr size_t state_bytes(int G, int NT) {
    return ((size_t)(8 * G * (NT / 64 + 2 + 2 * kEdits) + 4 * (G * (7 + 2 * kEdits) + 2)) + 15) & ~(size_t)15;
}
// the kernel variant of a launch shape; lean: every value pair in LDS
const void* kernel(int fsize, int G, int NT, bool lean);
// issues the kernel (one launch, nothing else)
void launch(const BArgs& a, int fsize, int G, int NT, bool lean, int nblocks, size_t lds, hipStream_t stream);

}  // namespace pfgpu_block
