// Device programs of the interpreted register kernels (k_pass_reg, k_batch_reg).
//
// A pass's gates are split into stages: in each stage log2(A) tile bits are
// the register index of every thread's A amplitudes and the other tile bits
// the thread index. Between stages the tile moves through LDS. The program of
// a pass is one XPass record (where the amplitudes lie in the state and in
// LDS) followed by XOp records of one fixed size, so that the kernel loads the
// next record while it runs the current one. Everything the kernel would
// otherwise work out per workgroup is worked out here once: coefficients are
// in the amplitude type, register conditions are masks of registers or pairs,
// an uncontrolled X is a renaming of the two values of a tile bit that costs
// nothing, and in FP32 an uncontrolled unitary gate is a real rotation between
// phases:
//   U = diag(e0, e1) * [[1, t0], [t1, 1]] * diag(1, y)
// (rows exchanged where the off-diagonal entries are the larger ones). The
// rotation costs 4 multiply-adds per pair where U costs 16 (in FP64, 8 where
// the planner scaled both rows to an exact 1); the phases of all
// gates of a wave, with whatever else is diagonal there, are one factor per
// register.
#pragma once

#include <cstdint>
#include <vector>

#include "planner.hpp"

namespace hgm {

enum XKind : uint32_t {
    // gates on the register pairs (x, y) that differ in register bit `bit`
    X_DENSE = 0,       // 2x2 complex matrix m[0..7]
    X_DENSE_REAL = 1,  // real matrix m[0], m[2], m[4], m[6]
    X_ROT = 2,         // x + m0 y, y + m1 x; in FP64 x + (m0 + i m1) y, y + (m2 + i m3) x
    X_ROTS = 3,        // real rotations with m[2 b], m[2 b + 1] on every register bit b (up to 4)
    // under a condition on threads (tmask, tval): y, x; a 2x2 matrix; a real one
    X_SWAP = 4, X_DENSE_LANE = 5, X_REAL_LANE = 6,
    // and only on the pairs in pmask (bit k: the pair whose lower register is k)
    X_DENSE_MASK = 7, X_REAL_MASK = 8,
    // multiply registers by a factor, two doubles at m in either type: those whose bits in `pat` are all set, those
    // whose bit pat - X_PAT_CLEAR is clear, or (X_PAT_MASK) those in pmask
    X_PHASE = 9,
    // multiply every register by a factor of its own: A complex or A real values at word pmask of the pass's table
    X_VEC = 10, X_VEC_REAL = 11,
    X_REMAP = 12       // move to the next stage's registers through LDS (XMap in m)
};

enum XFlag : uint32_t {
    // consecutive phases on the same registers are multiplied into one factor
    // per lane, applied by the last of them; the product is FP64 in either
    // type: rounded to FP32 at every phase, all registers of a lane share its
    // error, and an adder's grows with its size (FP64 issues at the FP32 rate)
    X_FIRST = 1, X_LAST = 2,
    X_REAL = 4         // the whole group's factors are real
};

constexpr uint32_t X_PAT_CLEAR = 32, X_PAT_MASK = 255;

// One gate, phase or remap. It acts where (tile base & gmask) == gval and (the
// kinds above that take it, and phases) (thread & tmask) == tval.
template <class T>
struct XOp {
    uint8_t kind, bit, pat, flags;
    uint32_t pmask;
    uint32_t tmask, tval;
    uint64_t gmask, gval;
    T m[8];
};
static_assert(sizeof(XOp<float>) == 64 && sizeof(XOp<double>) == 96, "shared with the kernels");

// Where a stage's element (t, k) lies in LDS: thread index t with a zero
// inserted at each register bit (low[i]: the tile bits below it, ascending),
// swizzled, XOR the swizzled register bits sw[i] of k.
struct XMap {
    uint16_t low[5], sw[5];
    uint32_t pad[3];
};
static_assert(sizeof(XMap) == 32, "fits XOp<float>::m");

// Bits [from, from + popcount(mask)) of an index to state bit `to` on.
struct XRun {
    uint32_t mask;
    uint16_t from, to;
};

constexpr int kXBaseRuns = 18, kXLaneRuns = 10;

// Element (t, k) of tile number T is state amplitude
//   base_runs(T) | (lane_runs(t) ^ sflip) | (register bits of k ^ rflip)
struct XPass {
    int32_t n_ops, n_base, n_load, n_store;
    int64_t table;                    // byte offset of the factor table from this record
    int64_t pad[7];
    XMap first;                       // LDS map of the first stage
    uint64_t lbit[5], sbit[5];        // state bit of each register bit (load, store)
    uint64_t sflip, rflip;            // tile bits whose values are exchanged at the store: thread bits, register bits
    XRun base[kXBaseRuns], load[kXLaneRuns], store[kXLaneRuns];
};
static_assert(sizeof(XPass) % 64 == 0, "records after it stay aligned");

// Swizzle of LDS slots: the upper bits XOR-folded into the low F ones (32
// slots of 8 bytes or 16 of 16 bytes span the 256 bytes of the banks), so that
// lanes walking consecutive tile bits hit distinct banks. Linear, its own
// inverse.
template <int F>
#if defined(__HIPCC__)
__host__ __device__
#endif
constexpr uint32_t x_swizzle(uint32_t x) {
    constexpr uint32_t M = (1u << F) - 1;
    return x ^ ((x >> F) & M) ^ ((x >> (2 * F)) & M) ^ ((x >> (3 * F)) & M);
}

// Chooses the execution shape (plan.exec) and builds plan.xprog and
// plan.xlaunch: one launch per non-empty pass, or, unless pass_by_pass, whole
// runs of passes where the state fits one workgroup. A compact program has no
// factor tables and no rotations split off: at most one record per gate, phase
// and remap, so it is never larger than the plan's register program and its
// maps. Others may be: every gate on one qubit, 16 amplitudes per thread, takes
// 256 bytes in FP32 as a rotation and a factor per register, 64 compact, and 104
// there. Where memory is given (hgm_state_apply_noalloc, the serving budget) a
// program that does not fit is built compact.
void build_exec_program(Plan &plan, bool pass_by_pass, bool compact = false);

// A copy of a plan, which others may be using, with compact programs.
Plan compact_plan(const Plan &plan);

}  // namespace hgm
