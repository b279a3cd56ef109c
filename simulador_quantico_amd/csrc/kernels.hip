// gfx950 kernels of the t_GPU path: the interpreted register kernels, state
// set-up and copies, and readout.
#include "device.hpp"
#include "kernels.hpp"
#include "program.hpp"

#include <type_traits>

namespace hgm {

namespace {

// State accesses of a single-circuit pass, which reads and writes every
// amplitude once per pass: nontemporal (streaming) hint (interpreted random30
// FP64 609 -> 578 ms per step, Hadamard x3 at 30 qubits 53.6 -> 52.7 ms, on
// one box). The batched serving kernel keeps plain accesses: many of its
// states fit the last-level cache between steps.
template <class T>
__device__ __forceinline__ typename Vec<T>::type load_stream(const typename Vec<T>::type *p) {
    typedef T N __attribute__((ext_vector_type(2)));
    const N v = __builtin_nontemporal_load(reinterpret_cast<const N *>(p));
    return {v.x, v.y};
}
template <class T>
__device__ __forceinline__ void store_stream(typename Vec<T>::type *p, const typename Vec<T>::type &a) {
    typedef T N __attribute__((ext_vector_type(2)));
    const N v = {a.x, a.y};
    __builtin_nontemporal_store(v, reinterpret_cast<N *>(p));
}

// ---------------------------------------------------------------------------
// k_pass_reg: the register kernel. Each thread keeps A amplitudes of its tile
// in registers for the whole pass and runs the pass's program (program.hpp):
// gates act on register pairs, between stages the tile makes one round trip
// through LDS. HBM traffic per pass: one read and one write of every
// amplitude.
//
// What an interpreted gate costs beyond its multiply-adds is issue slots, so
// the program leaves nothing to work out per amplitude: a condition on tile
// bits skips the record (scalar), one on thread bits masks lanes (one
// divergent branch, no selected matrices), one on register bits is a mask of
// pairs; phases are gathered per lane and applied once per group; the next
// record's scalar loads are in flight while a record runs. A remap writes to
// the LDS slots the thread itself read last, so it needs one barrier, and none
// where a tile lies within a wave.

template <class T, int KIND>
__device__ __forceinline__ void pair_update(typename Vec<T>::type &x, typename Vec<T>::type &y, const T (&m)[8]) {
    using V = typename Vec<T>::type;
    const V p = x, q = y;
    if constexpr (KIND == X_DENSE) {
        x = cmul2<V, T>(m[0], m[1], p, m[2], m[3], q);
        y = cmul2<V, T>(m[4], m[5], p, m[6], m[7], q);
    } else if constexpr (KIND == X_DENSE_REAL) {
        x.x = m[0] * p.x + m[2] * q.x;
        x.y = m[0] * p.y + m[2] * q.y;
        y.x = m[4] * p.x + m[6] * q.x;
        y.y = m[4] * p.y + m[6] * q.y;
    } else if constexpr (KIND == X_ROT && sizeof(T) == 8) {
        x.x = p.x + m[0] * q.x - m[1] * q.y;
        x.y = p.y + m[0] * q.y + m[1] * q.x;
        y.x = q.x + m[2] * p.x - m[3] * p.y;
        y.y = q.y + m[2] * p.y + m[3] * p.x;
    } else {
        static_assert(KIND == X_ROT || KIND == X_ROTS);
        x.x = p.x + m[0] * q.x;
        x.y = p.y + m[0] * q.y;
        y.x = q.x + m[1] * p.x;
        y.y = q.y + m[1] * p.y;
    }
}

// Gates under a condition resolve it by selection: the matrix or the identity
// per lane (once per gate) and per pair.
template <class T, int A, int KIND, int BIT>
__device__ __forceinline__ void gate_bit(typename Vec<T>::type (&a)[A], const T (&m)[8], bool lane, uint32_t pmask) {
    constexpr bool kMask = KIND == X_DENSE_MASK || KIND == X_REAL_MASK;
    constexpr bool kCond = kMask || KIND == X_DENSE_LANE || KIND == X_REAL_LANE;
    constexpr bool kReal = KIND == X_REAL_LANE || KIND == X_REAL_MASK;
    T u[8];
    if constexpr (kCond) {
#pragma unroll
        for (int e = 0; e < 8; ++e) u[e] = lane ? m[e] : T(e == 0 || e == 6 ? 1 : 0);
    }
#pragma unroll
    for (int k = 0; k < A; ++k) {
        if (k & (1 << BIT)) continue;
        typename Vec<T>::type &x = a[k], &y = a[k | (1 << BIT)];
        if constexpr (KIND == X_SWAP) {
            const typename Vec<T>::type p = x;
            x.x = lane ? y.x : p.x;
            x.y = lane ? y.y : p.y;
            y.x = lane ? p.x : y.x;
            y.y = lane ? p.y : y.y;
        } else if constexpr (kMask) {
            const bool on = (pmask >> k) & 1u;
            T w[8];
#pragma unroll
            for (int e = 0; e < 8; ++e) w[e] = on ? u[e] : T(e == 0 || e == 6 ? 1 : 0);
            pair_update<T, kReal ? X_DENSE_REAL : X_DENSE>(x, y, w);
        } else if constexpr (kCond) {
            pair_update<T, kReal ? X_DENSE_REAL : X_DENSE>(x, y, u);
        } else {
            pair_update<T, KIND>(x, y, m);
        }
    }
}

// Dispatch on the runtime register bit (wave-uniform) to unrolled code; bits
// at log2(A) and above do not occur.
template <class T, int A, int KIND>
__device__ __forceinline__ void gate(typename Vec<T>::type (&a)[A], const T (&m)[8], int bit, bool lane = true,
                                     uint32_t pmask = 0) {
    switch (bit) {
        case 0: gate_bit<T, A, KIND, 0>(a, m, lane, pmask); break;
        case 1: if constexpr (A > 2) { gate_bit<T, A, KIND, 1>(a, m, lane, pmask); break; } __builtin_unreachable();
        case 2: if constexpr (A > 4) { gate_bit<T, A, KIND, 2>(a, m, lane, pmask); break; } __builtin_unreachable();
        case 3: if constexpr (A > 8) { gate_bit<T, A, KIND, 3>(a, m, lane, pmask); break; } __builtin_unreachable();
        case 4: if constexpr (A > 16) { gate_bit<T, A, KIND, 4>(a, m, lane, pmask); break; } __builtin_unreachable();
        default: __builtin_unreachable();
    }
}

// Multiplies the registers k with (k & BITS) == VAL by the lane's factor.
template <class T, int A, int BITS, int VAL>
__device__ __forceinline__ void phase_on(typename Vec<T>::type (&a)[A], T fr, T fi, bool real) {
    if constexpr (BITS < A) {
        if (real) {
#pragma unroll
            for (int k = 0; k < A; ++k)
                if ((k & BITS) == VAL) { a[k].x *= fr; a[k].y *= fr; }
        } else {
#pragma unroll
            for (int k = 0; k < A; ++k)
                if ((k & BITS) == VAL) a[k] = cmul<typename Vec<T>::type, T>(fr, fi, a[k]);
        }
    } else {
        __builtin_unreachable();
    }
}

template <class T, int A>
__device__ __forceinline__ void phase_apply(typename Vec<T>::type (&a)[A], T fr, T fi, bool real, uint32_t pat,
                                            uint32_t pmask) {
#define HGM_SET(S) case S: phase_on<T, A, S, S>(a, fr, fi, real); break;
#define HGM_CLEAR(B) case X_PAT_CLEAR + B: phase_on<T, A, (1 << B), 0>(a, fr, fi, real); break;
    switch (pat) {   // one or two register bits set: the phases of controlled phase gates
        HGM_CLEAR(0) HGM_CLEAR(1) HGM_CLEAR(2) HGM_CLEAR(3) HGM_CLEAR(4)
        HGM_SET(0) HGM_SET(1) HGM_SET(2) HGM_SET(3) HGM_SET(4) HGM_SET(5) HGM_SET(6) HGM_SET(8) HGM_SET(9)
        HGM_SET(10) HGM_SET(12) HGM_SET(16) HGM_SET(17) HGM_SET(18) HGM_SET(20) HGM_SET(24)
        default:
#pragma unroll
            for (int k = 0; k < A; ++k) {
                const bool on = (pmask >> k) & 1u;
                a[k] = cmul<typename Vec<T>::type, T>(on ? fr : T(1), on ? fi : T(0), a[k]);
            }
    }
#undef HGM_SET
#undef HGM_CLEAR
}

// Rotations on every register bit (up to 4), one after the other in straight
// line: one record, and one settling of the registers, for a layer of gates.
template <class T, int A>
__device__ __forceinline__ void rotations(typename Vec<T>::type (&a)[A], const T (&m)[8]) {
#pragma unroll
    for (int b = 0; b < 4 && (2 << b) <= A; ++b) {
        const T u[8] = {m[2 * b], m[2 * b + 1]};
#pragma unroll
        for (int k = 0; k < A; ++k)
            if (!((k >> b) & 1)) pair_update<T, X_ROTS>(a[k], a[k | (1 << b)], u);
    }
}

// Thread part of an LDS slot, in bytes: the thread index with a zero at every
// register bit, swizzled.
template <class T, int A>
__device__ __forceinline__ uint32_t lds_pos(uint32_t t, const XMap &m) {
    constexpr int L = A == 2 ? 1 : A == 4 ? 2 : A == 8 ? 3 : A == 16 ? 4 : 5;
    uint32_t x = t;
#pragma unroll
    for (int i = 0; i < L; ++i) x += x & ~(uint32_t)m.low[i];
    x = x_swizzle<sizeof(T) == 4 ? 5 : 4>(x) * (uint32_t)sizeof(typename Vec<T>::type);
    asm("" : "+v"(x));   // keeps the scaling here, once, instead of after the XOR with each register's part
    return x;
}

template <class T, int A>
__device__ __forceinline__ uint32_t lds_reg(int k, const XMap &m) {
    uint32_t x = 0;
#pragma unroll
    for (int i = 0; (1 << i) < A; ++i)
        if ((k >> i) & 1) x ^= m.sw[i];
    return x * (uint32_t)sizeof(typename Vec<T>::type);
}

__device__ __forceinline__ uint64_t run_bits(uint64_t v, const XRun &r) {
    return ((v >> r.from) & r.mask) << r.to;
}

// Deposit of v by runs; most deposits have up to 4, whose loads go out together.
__device__ __forceinline__ uint64_t deposit(uint64_t v, const XRun *__restrict__ runs, int n) {
    uint64_t x = run_bits(v, runs[0]) | run_bits(v, runs[1]) | run_bits(v, runs[2]) | run_bits(v, runs[3]);
    for (int i = 4; i < n; ++i) x |= run_bits(v, runs[i]);
    return x;
}

template <int A>
__device__ __forceinline__ uint64_t reg_bits(int k, const uint64_t *__restrict__ bit, uint64_t flip) {
#pragma unroll
    for (int i = 0; (1 << i) < A; ++i)
        if ((k >> i) & 1) flip ^= bit[i];
    return flip;
}

// Real (0) or imaginary (1) part of a phase record's factor.
__device__ __forceinline__ double phase_part(const XOp<double> &o, int part) { return o.m[part]; }
__device__ __forceinline__ double phase_part(const XOp<float> &o, int part) {
    return __hiloint2double(__float_as_int(o.m[2 * part + 1]), __float_as_int(o.m[2 * part]));
}

// Runs the records of a pass on the registers of one tile.
template <class T, int A>
__device__ __forceinline__ void run_program(typename Vec<T>::type (&a)[A], const XPass *__restrict__ xp, uint64_t base,
                                            unsigned char *lds, bool sync) {
    using V = typename Vec<T>::type;
    const uint32_t t = threadIdx.x;
    const XOp<T> *__restrict__ ops = reinterpret_cast<const XOp<T> *>(xp + 1);
    const T *__restrict__ table = reinterpret_cast<const T *>(reinterpret_cast<const char *>(xp) + xp->table);
    const int n = xp->n_ops;
    XMap cur = xp->first;
    uint32_t pos = lds_pos<T, A>(t, cur);
    double fr = 1, fi = 0;
    XOp<T> next = ops[0];
    for (int i = 0; i < n; ++i) {
        const XOp<T> o = next;
        next = ops[i + 1];   // the program ends with a spare record
        if (o.kind == X_REMAP) {
            XMap to;
            __builtin_memcpy(&to, o.m, sizeof to);
#pragma unroll
            for (int k = 0; k < A; ++k) *reinterpret_cast<V *>(lds + (pos ^ lds_reg<T, A>(k, cur))) = a[k];
            if (sync) __syncthreads();
            else __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
            pos = lds_pos<T, A>(t, to);
#pragma unroll
            for (int k = 0; k < A; ++k) a[k] = *reinterpret_cast<const V *>(lds + (pos ^ lds_reg<T, A>(k, to)));
            cur = to;
            continue;
        }
        const bool tile = (base & o.gmask) == o.gval;
        if (o.kind == X_PHASE) {
            if (!tile && (o.flags & (X_FIRST | X_LAST)) == (X_FIRST | X_LAST)) continue;
            const bool on = tile && (t & o.tmask) == o.tval;
            const double gr = on ? phase_part(o, 0) : 1.0, gi = on ? phase_part(o, 1) : 0.0;
            if (o.flags & X_FIRST) {
                fr = gr;
                fi = gi;
            } else if (o.flags & X_REAL) {
                fr *= gr;
            } else {
                const double r = fr * gr - fi * gi;
                fi = fr * gi + fi * gr;
                fr = r;
            }
            if (o.flags & X_LAST) phase_apply<T, A>(a, (T)fr, (T)fi, (o.flags & X_REAL) != 0, o.pat, o.pmask);
            continue;
        }
        if (!tile) continue;
        const auto lane = [&] { return (t & o.tmask) == o.tval; };
        switch (o.kind) {
            case X_ROTS: rotations<T, A>(a, o.m); break;
            case X_VEC: {
                const T *__restrict__ f = table + o.pmask;
#pragma unroll
                for (int k = 0; k < A; ++k) a[k] = cmul<V, T>(f[2 * k], f[2 * k + 1], a[k]);
                break;
            }
            case X_VEC_REAL: {
                const T *__restrict__ f = table + o.pmask;
#pragma unroll
                for (int k = 0; k < A; ++k) {
                    a[k].x *= f[k];
                    a[k].y *= f[k];
                }
                break;
            }
            case X_ROT: gate<T, A, X_ROT>(a, o.m, o.bit); break;
            case X_DENSE: gate<T, A, X_DENSE>(a, o.m, o.bit); break;
            case X_DENSE_REAL: gate<T, A, X_DENSE_REAL>(a, o.m, o.bit); break;
            case X_SWAP: gate<T, A, X_SWAP>(a, o.m, o.bit, lane()); break;
            case X_DENSE_LANE: gate<T, A, X_DENSE_LANE>(a, o.m, o.bit, lane()); break;
            case X_REAL_LANE: gate<T, A, X_REAL_LANE>(a, o.m, o.bit, lane()); break;
            case X_DENSE_MASK: gate<T, A, X_DENSE_MASK>(a, o.m, o.bit, lane(), o.pmask); break;
            case X_REAL_MASK: gate<T, A, X_REAL_MASK>(a, o.m, o.bit, lane(), o.pmask); break;
            default: __builtin_unreachable();
        }
    }
}

// Requests the program's cache lines (128 bytes each) into the L2, all at
// once: a program was copied to the device just before it runs, and read
// record by record its first reader would wait for memory at every line
// (default tuning: random layers at 13 qubits FP64 83 -> 55 us, QFT at 13
// qubits 48 -> 33). The first tiles of a state do it, the rest find the lines.
__device__ __forceinline__ uint32_t warm_program(const XPass *__restrict__ xp, uint32_t bytes, int64_t tile) {
    uint32_t v = 0;
    if (tile < 512)
        for (uint32_t o = threadIdx.x * 128; o < bytes; o += blockDim.x * 128)
            v |= *reinterpret_cast<const uint32_t *>(reinterpret_cast<const char *>(xp) + o);
    return v;
}

// How a pass reads and writes the state, and whether remaps need barriers.
constexpr uint32_t kStreamLoads = 1, kStreamStores = 2, kBarriers = 4;

template <class T, int A>
__global__ void __launch_bounds__(reg_kernel_max_threads(A, sizeof(typename Vec<T>::type)))
    k_pass_reg(typename Vec<T>::type *__restrict__ state, const int64_t *__restrict__ offs, const XPass *__restrict__ xp,
               uint32_t xp_bytes, int64_t n_tiles, uint32_t mode) {
    using V = typename Vec<T>::type;
    if (offs) state = reinterpret_cast<V *>(reinterpret_cast<char *>(state) + offs[blockIdx.y]);
    extern __shared__ __align__(16) unsigned char smem[];
    const uint32_t t = threadIdx.x;
    const uint32_t warm = warm_program(xp, xp_bytes, blockIdx.x);
    const uint64_t lt = deposit(t, xp->load, xp->n_load);
    const uint64_t st = deposit(t, xp->store, xp->n_store) ^ xp->sflip;
    for (int64_t tid = blockIdx.x; tid < n_tiles; tid += gridDim.x) {
        const uint64_t base = deposit((uint64_t)tid, xp->base, xp->n_base);
        V a[A];
        const V *src = state + (base | lt);
        if (mode & kStreamLoads) {
#pragma unroll
            for (int k = 0; k < A; ++k) a[k] = load_stream<T>(src + reg_bits<A>(k, xp->lbit, 0));
        } else {
#pragma unroll
            for (int k = 0; k < A; ++k) a[k] = src[reg_bits<A>(k, xp->lbit, 0)];
        }
        asm volatile("" ::"v"(warm));   // the loads are not dropped, and nothing waits for them before the state's
        run_program<T, A>(a, xp, base, smem, (mode & kBarriers) != 0);
        V *dst = state + (base | st);
        if (mode & kStreamStores) {
#pragma unroll
            for (int k = 0; k < A; ++k) store_stream<T>(dst + reg_bits<A>(k, xp->sbit, xp->rflip), a[k]);
        } else {
#pragma unroll
            for (int k = 0; k < A; ++k) dst[reg_bits<A>(k, xp->sbit, xp->rflip)] = a[k];
        }
        if (tid + gridDim.x < n_tiles) __syncthreads();   // the next tile writes LDS slots that others may still read
    }
}

// Batched register kernel: one launch runs one pass of each of many states
// (of any qubit count that shares the workgroup shape). Workgroup b belongs to
// the item whose tile range [tile_begin, next tile_begin) holds b; the items
// are sorted by tile_begin, so a binary search on tile-uniform values finds it.
// When the item asks for a readout, each tile also reduces its output (FP64
// sum of |a|^2, largest |a|^2 with the lowest index on ties) into
// partials[tile]; k_readout_final combines the tiles of a state.
template <class T, int A>
__global__ void __launch_bounds__(reg_kernel_max_threads(A, sizeof(typename Vec<T>::type))) k_batch_reg(const BatchItem *__restrict__ items,
                                                                          int n_items,
                                                                          const char *__restrict__ progs,
                                                                          char *__restrict__ states,
                                                                          char *__restrict__ parts) {
    using V = typename Vec<T>::type;
    extern __shared__ __align__(16) unsigned char smem[];
    __shared__ double red_s[16], red_m[16];
    __shared__ uint64_t red_i[16];
    const int t = threadIdx.x;
    const int64_t b = blockIdx.x;
    int lo = 0, hi = n_items - 1;
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (items[mid].tile_begin <= b) lo = mid; else hi = mid - 1;
    }
    const BatchItem &it = items[lo];
    V *__restrict__ state = reinterpret_cast<V *>(states + it.state_off);
    const XPass *__restrict__ xp = reinterpret_cast<const XPass *>(progs + it.xpass_off);
    const int64_t tid = b - it.tile_begin;
    const uint32_t warm = warm_program(xp, it.xpass_bytes, tid);
    const uint64_t base = deposit((uint64_t)tid, xp->base, xp->n_base);
    const uint64_t lt = deposit(t, xp->load, xp->n_load);
    V a[A];
#pragma unroll
    for (int k = 0; k < A; ++k) a[k] = state[(base | lt) + reg_bits<A>(k, xp->lbit, 0)];
    asm volatile("" ::"v"(warm));
    run_program<T, A>(a, xp, base, smem, it.sync != 0);
    const uint64_t to = base | (deposit(t, xp->store, xp->n_store) ^ xp->sflip);
#pragma unroll
    for (int k = 0; k < A; ++k) state[to + reg_bits<A>(k, xp->sbit, xp->rflip)] = a[k];
    if (it.partials_off < 0) return;
    double sum = 0.0, best = -1.0;
    uint64_t bi = ~uint64_t(0);
#pragma unroll
    for (int k = 0; k < A; ++k) {
        const double p = (double)a[k].x * (double)a[k].x + (double)a[k].y * (double)a[k].y;
        const uint64_t idx = to + reg_bits<A>(k, xp->sbit, xp->rflip);
        sum += p;
        if (p > best || (p == best && idx < bi)) { best = p; bi = idx; }
    }
    // lanes of a wave first (only lanes that exist: width = min(64, blockDim)), then waves in order
    const int width = blockDim.x < 64 ? (int)blockDim.x : 64;
    for (int off = width >> 1; off > 0; off >>= 1) {
        sum += __shfl_xor(sum, off, width);
        const double ob = __shfl_xor(best, off, width);
        const uint64_t oi = __shfl_xor(bi, off, width);
        if (ob > best || (ob == best && oi < bi)) { best = ob; bi = oi; }
    }
    if ((t & 63) == 0) { red_s[t >> 6] = sum; red_m[t >> 6] = best; red_i[t >> 6] = bi; }
    __syncthreads();
    if (t == 0) {
        const int waves = (blockDim.x + 63) >> 6;
        for (int w = 1; w < waves; ++w) {
            sum += red_s[w];
            if (red_m[w] > best || (red_m[w] == best && red_i[w] < bi)) { best = red_m[w]; bi = red_i[w]; }
        }
        ReadoutPartial r;
        r.sum = sum;
        r.pmax = best;
        r.idx = bi;
        r.pad = 0;
        reinterpret_cast<ReadoutPartial *>(parts + it.partials_off)[tid] = r;
    }
}

// One workgroup per task: combines a state's per-tile readout partials in
// tile order.
__global__ void __launch_bounds__(256) k_readout_final(const ReadoutTask *__restrict__ tasks) {
    __shared__ double ss[256], sm[256];
    __shared__ uint64_t si[256];
    const ReadoutTask &tk = tasks[blockIdx.x];
    double sum = 0.0, best = -1.0;
    uint64_t bi = ~uint64_t(0);
    for (int64_t i = threadIdx.x; i < tk.n; i += 256) {
        const ReadoutPartial p = tk.partials[i];
        sum += p.sum;
        if (p.pmax > best || (p.pmax == best && p.idx < bi)) { best = p.pmax; bi = p.idx; }
    }
    ss[threadIdx.x] = sum;
    sm[threadIdx.x] = best;
    si[threadIdx.x] = bi;
    __syncthreads();
    for (int w = 128; w > 0; w >>= 1) {
        if ((int)threadIdx.x < w) {
            ss[threadIdx.x] += ss[threadIdx.x + w];
            const double o = sm[threadIdx.x + w];
            const uint64_t oi = si[threadIdx.x + w];
            if (o > sm[threadIdx.x] || (o == sm[threadIdx.x] && oi < si[threadIdx.x])) { sm[threadIdx.x] = o; si[threadIdx.x] = oi; }
        }
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        ReadoutPartial r;
        r.sum = ss[0];
        r.pmax = sm[0];
        r.idx = si[0];
        r.pad = 0;
        *tk.out = r;
    }
}

// Plain streaming copy, 16 bytes per lane per iteration.
__global__ void __launch_bounds__(256) k_copy(uint4 *__restrict__ dst, const uint4 *__restrict__ src, uint64_t n16) {
    for (uint64_t i = blockIdx.x * (uint64_t)blockDim.x + threadIdx.x; i < n16; i += (uint64_t)gridDim.x * blockDim.x)
        dst[i] = src[i];
}

template <class T>
__global__ void k_set_basis(typename Vec<T>::type *state, uint64_t n, uint64_t index) {
    using V = typename Vec<T>::type;
    for (uint64_t i = blockIdx.x * (uint64_t)blockDim.x + threadIdx.x; i < n; i += (uint64_t)gridDim.x * blockDim.x) {
        V v;
        v.x = (i == index) ? T(1) : T(0);
        v.y = T(0);
        state[i] = v;
    }
}

// Reductions over a whole state read every amplitude once and write a few
// bytes, so they are bound by the bytes in flight: W amplitudes per 16-byte
// load, and U loads per lane issued before any of them is used. One 8-byte
// load per lane and iteration read a 4 GiB FP32 state at 3.6 TB/s (1200 us per
// sum), W = 2 and U = 8 at 6.1 (700 us; a copy moves 6.2). A lane takes every
// 256th vector of its block's U * 256, so it sees increasing indices.
template <class T, int W, int U, class F>
__device__ __forceinline__ void for_amps(const typename Vec<T>::type *state, uint64_t n, F fn) {
    typedef T Wide __attribute__((ext_vector_type(2 * W)));
    const Wide *p = reinterpret_cast<const Wide *>(state);
    const uint64_t nv = n / W, step = (uint64_t)gridDim.x * (256 * U);
    for (uint64_t v0 = blockIdx.x * (uint64_t)(256 * U) + threadIdx.x; v0 < nv; v0 += step) {
        Wide w[U];
#pragma unroll
        for (int u = 0; u < U; ++u) w[u] = p[v0 + u * 256];
#pragma unroll
        for (int u = 0; u < U; ++u)
#pragma unroll
            for (int j = 0; j < W; ++j) {
                const double x = w[u][2 * j], y = w[u][2 * j + 1];
                fn((v0 + u * 256) * W + j, x * x + y * y);
            }
    }
}

template <class T, int W, int U>
__global__ void __launch_bounds__(256) k_prob_halves(const typename Vec<T>::type *state, uint64_t n, int bit,
                                                      double *partial) {
    __shared__ double s0[4], s1[4];
    double a0 = 0, a1 = 0;
    const uint64_t sel = bit >= 0 ? uint64_t(1) << bit : 0;
    for_amps<T, W, U>(state, n, [&](uint64_t i, double p) {
        const bool one = (i & sel) != 0;
        a0 += one ? 0.0 : p;
        a1 += one ? p : 0.0;
    });
    for (int off = 32; off > 0; off >>= 1) {
        a0 += __shfl_xor(a0, off);
        a1 += __shfl_xor(a1, off);
    }
    if ((threadIdx.x & 63) == 0) { s0[threadIdx.x >> 6] = a0; s1[threadIdx.x >> 6] = a1; }
    __syncthreads();
    if (threadIdx.x == 0) {
        partial[2 * blockIdx.x] = (s0[0] + s0[1]) + (s0[2] + s0[3]);
        partial[2 * blockIdx.x + 1] = (s1[0] + s1[1]) + (s1[2] + s1[3]);
    }
}

template <class T, int W, int U>
__global__ void __launch_bounds__(256) k_argmax(const typename Vec<T>::type *state, uint64_t n, double *pmax,
                                                 uint64_t *pidx) {
    __shared__ double sm[4];
    __shared__ uint64_t si[4];
    double best = -1.0;
    uint64_t bi = ~uint64_t(0);
    for_amps<T, W, U>(state, n, [&](uint64_t i, double p) {
        if (p > best) { best = p; bi = i; }
    });
    for (int off = 32; off > 0; off >>= 1) {
        const double o = __shfl_xor(best, off);
        const uint64_t oi = __shfl_xor(bi, off);
        if (o > best || (o == best && oi < bi)) { best = o; bi = oi; }
    }
    if ((threadIdx.x & 63) == 0) { sm[threadIdx.x >> 6] = best; si[threadIdx.x >> 6] = bi; }
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int w = 1; w < 4; ++w)
            if (sm[w] > best || (sm[w] == best && si[w] < bi)) { best = sm[w]; bi = si[w]; }
        pmax[blockIdx.x] = best;
        pidx[blockIdx.x] = bi;
    }
}

// Per-block partials of the comparison of two states of any amplitude types:
// Re and Im of sum conj(a)*b, sum |a|^2, sum |b|^2 (FP64), and max |a - b|.
template <class TA, class TB>
__global__ void __launch_bounds__(256) k_compare(const typename Vec<TA>::type *a, const typename Vec<TB>::type *b,
                                                  uint64_t n, double *partial) {
    __shared__ double sh[5][256];
    double re = 0, im = 0, na = 0, nb = 0, mx = 0;
    for (uint64_t i = blockIdx.x * (uint64_t)blockDim.x + threadIdx.x; i < n; i += (uint64_t)gridDim.x * blockDim.x) {
        const double ar = a[i].x, ai = a[i].y, br = b[i].x, bi = b[i].y;
        re += ar * br + ai * bi;
        im += ar * bi - ai * br;
        na += ar * ar + ai * ai;
        nb += br * br + bi * bi;
        const double dr = ar - br, di = ai - bi;
        mx = fmax(mx, sqrt(dr * dr + di * di));
    }
    const int t = threadIdx.x;
    sh[0][t] = re; sh[1][t] = im; sh[2][t] = na; sh[3][t] = nb; sh[4][t] = mx;
    __syncthreads();
    for (int w = 128; w > 0; w >>= 1) {
        if (t < w) {
            for (int k = 0; k < 4; ++k) sh[k][t] += sh[k][t + w];
            sh[4][t] = fmax(sh[4][t], sh[4][t + w]);
        }
        __syncthreads();
    }
    if (t < 5) partial[5 * blockIdx.x + t] = sh[t][0];
}

template <class T>
__global__ void k_collapse(typename Vec<T>::type *state, uint64_t half, int bit, int outcome, double norm) {
    using V = typename Vec<T>::type;
    const uint64_t low = (uint64_t(1) << bit) - 1;
    for (uint64_t i = blockIdx.x * (uint64_t)blockDim.x + threadIdx.x; i < half; i += (uint64_t)gridDim.x * blockDim.x) {
        const uint64_t pos = ((i >> bit) << (bit + 1)) | (i & low);
        const V v = state[pos | (uint64_t(outcome) << bit)];
        V w;
        w.x = (T)((double)v.x / norm);
        w.y = (T)((double)v.y / norm);
        state[pos] = w;
        V z;
        z.x = T(0);
        z.y = T(0);
        state[pos | (uint64_t(1) << bit)] = z;
    }
}

int grid_for(uint64_t n, int block) {
    uint64_t g = (n + block - 1) / block;
    if (g > (uint64_t(1) << 24)) g = uint64_t(1) << 24;
    if (g > max_blocks(block)) g = max_blocks(block);
    if (g < 1) g = 1;
    return (int)g;
}

// The per-pass kernels' dynamic LDS limit, raised once per kernel (before the
// first launch, and before any stream capture that launches it).
template <class T, int A>
hipError_t pass_reg_attr() {
    static const hipError_t e =
        hipFuncSetAttribute((const void *)k_pass_reg<T, A>, hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
    return e;
}
template <class T>
hipError_t pass_attrs() {
    for (hipError_t e : {pass_reg_attr<T, 2>(), pass_reg_attr<T, 4>(), pass_reg_attr<T, 8>(),
                         pass_reg_attr<T, 16>(), pass_reg_attr<T, 32>()})
        if (e != hipSuccess) return e;
    return hipSuccess;
}

template <class T, int A>
hipError_t pass_reg(const StateSet &set, const XPass *xp, uint32_t xp_bytes, int64_t n_tiles, int B, size_t lds,
                    uint32_t mode, hipStream_t s) {
    pass_reg_attr<T, A>();
    const int64_t grid = tile_grid(n_tiles, B * set.count);
    hipLaunchKernelGGL((k_pass_reg<T, A>), dim3((unsigned)grid, (unsigned)set.count), dim3(B), lds, s,
                       reinterpret_cast<typename Vec<T>::type *>(set.first), set.offs, xp, xp_bytes, n_tiles, mode);
    return hipGetLastError();
}

template <class T>
hipError_t pass_reg_any(int A, const StateSet &state, const XPass *xp, uint32_t xp_bytes, int64_t n_tiles, int B, size_t lds,
                        uint32_t mode, hipStream_t s) {
    switch (A) {
        case 2: return pass_reg<T, 2>(state, xp, xp_bytes, n_tiles, B, lds, mode, s);
        case 4: return pass_reg<T, 4>(state, xp, xp_bytes, n_tiles, B, lds, mode, s);
        case 8: return pass_reg<T, 8>(state, xp, xp_bytes, n_tiles, B, lds, mode, s);
        case 16: return pass_reg<T, 16>(state, xp, xp_bytes, n_tiles, B, lds, mode, s);
        case 32: return pass_reg<T, 32>(state, xp, xp_bytes, n_tiles, B, lds, mode, s);
        default: return hipErrorInvalidValue;
    }
}

template <class T, int A>
hipError_t batch_reg(const BatchItem *items, int n_items, int64_t total_tiles, int B, size_t lds, char *arena,
                     hipStream_t s) {
    static bool attr_set = false;
    if (!attr_set) {
        hipFuncSetAttribute((const void *)k_batch_reg<T, A>, hipFuncAttributeMaxDynamicSharedMemorySize, 128 * 1024);
        attr_set = true;
    }
    hipLaunchKernelGGL((k_batch_reg<T, A>), dim3((unsigned)total_tiles), dim3(B), lds, s, items, n_items,
                       (const char *)arena, arena, arena);
    return hipGetLastError();
}

template <class T>
hipError_t batch_reg_any(int A, const BatchItem *items, int n_items, int64_t total_tiles, int B, size_t lds,
                         char *arena, hipStream_t s) {
    switch (A) {
        case 2: return batch_reg<T, 2>(items, n_items, total_tiles, B, lds, arena, s);
        case 4: return batch_reg<T, 4>(items, n_items, total_tiles, B, lds, arena, s);
        case 8: return batch_reg<T, 8>(items, n_items, total_tiles, B, lds, arena, s);
        case 16: return batch_reg<T, 16>(items, n_items, total_tiles, B, lds, arena, s);
        case 32: return batch_reg<T, 32>(items, n_items, total_tiles, B, lds, arena, s);
        default: return hipErrorInvalidValue;
    }
}

}  // namespace

hipError_t launch_pass_reg(int dtype, int qubits, const ExecShape &e, const StateSet &state, const XPass *xp,
                           uint32_t xp_bytes, size_t lds_bytes, hipStream_t s) {
    const size_t bytes = (size_t(1) << qubits) * amp_bytes(dtype) * (size_t)state.count;
    bool ld, st;
    state_streams(bytes, &ld, &st);
    const uint32_t mode = (ld ? kStreamLoads : 0) | (st ? kStreamStores : 0) | (e.sync ? kBarriers : 0);
    const int64_t n_tiles = int64_t(1) << (qubits - e.r);
    return dtype == HGM_C64 ? pass_reg_any<float>(e.A, state, xp, xp_bytes, n_tiles, e.B, lds_bytes, mode, s)
                            : pass_reg_any<double>(e.A, state, xp, xp_bytes, n_tiles, e.B, lds_bytes, mode, s);
}

hipError_t prepare_pass_kernels(int dtype) {
    const hipError_t e = prepare_pass_lds(dtype);
    return e != hipSuccess ? e : dtype == HGM_C64 ? pass_attrs<float>() : pass_attrs<double>();
}

hipError_t launch_copy(void *dst, const void *src, size_t bytes, hipStream_t s) {
    // one 16-byte element per thread over the whole buffer: a flat grid keeps
    // far more requests in flight than a grid-stride loop (6.2 vs 4.9 TB/s)
    const uint64_t n16 = bytes / 16;
    const int blk = 256;
    uint64_t g = (n16 + blk - 1) / blk;
    if (g > max_blocks(blk)) g = max_blocks(blk);
    if (g < 1) g = 1;
    hipLaunchKernelGGL(k_copy, dim3((unsigned)g), dim3(blk), 0, s, (uint4 *)dst, (const uint4 *)src, n16);
    return hipGetLastError();
}

hipError_t launch_set_basis(int dtype, void *state, uint64_t n, uint64_t index, hipStream_t s) {
    const int blk = 256, grid = grid_for(n, blk);
    if (dtype == HGM_C64) hipLaunchKernelGGL(k_set_basis<float>, dim3(grid), dim3(blk), 0, s, (float2 *)state, n, index);
    else hipLaunchKernelGGL(k_set_basis<double>, dim3(grid), dim3(blk), 0, s, (double2 *)state, n, index);
    return hipGetLastError();
}

namespace {

// Blocks and loads per lane of a whole-state reduction: 8 loads of 16 bytes
// when that gives every block at least one full round, else one load (more
// blocks at work); a borrowed FP32 state that is only 8-byte aligned is read
// one amplitude at a time.
template <class F>
hipError_t reduce_launch(int dtype, const void *state, uint64_t n, int blocks, F launch) {
    const bool f32 = dtype == HGM_C64;
    const int W = f32 && n >= 2 && (reinterpret_cast<uintptr_t>(state) & 15) == 0 ? 2 : 1;
    const bool deep = n / W >= (uint64_t)blocks * 256 * 8;
    using std::integral_constant;
    if (!f32) { if (deep) launch(double(), integral_constant<int, 1>(), integral_constant<int, 8>());
                else launch(double(), integral_constant<int, 1>(), integral_constant<int, 1>()); }
    else if (W == 2) { if (deep) launch(float(), integral_constant<int, 2>(), integral_constant<int, 8>());
                       else launch(float(), integral_constant<int, 2>(), integral_constant<int, 1>()); }
    else { if (deep) launch(float(), integral_constant<int, 1>(), integral_constant<int, 8>());
           else launch(float(), integral_constant<int, 1>(), integral_constant<int, 1>()); }
    return hipGetLastError();
}

}  // namespace

hipError_t launch_prob_halves(int dtype, const void *state, uint64_t n, int bit, double *partial, int blocks,
                              hipStream_t s) {
    return reduce_launch(dtype, state, n, blocks, [&](auto t, auto w, auto u) {
        using T = decltype(t);
        hipLaunchKernelGGL((k_prob_halves<T, w(), u()>), dim3(blocks), dim3(256), 0, s,
                           static_cast<const typename Vec<T>::type *>(state), n, bit, partial);
    });
}

hipError_t launch_argmax(int dtype, const void *state, uint64_t n, double *pmax, uint64_t *pidx, int blocks,
                         hipStream_t s) {
    return reduce_launch(dtype, state, n, blocks, [&](auto t, auto w, auto u) {
        using T = decltype(t);
        hipLaunchKernelGGL((k_argmax<T, w(), u()>), dim3(blocks), dim3(256), 0, s,
                           static_cast<const typename Vec<T>::type *>(state), n, pmax, pidx);
    });
}

hipError_t launch_compare(int dtype_a, const void *a, int dtype_b, const void *b, uint64_t n, double *partial,
                          int blocks, hipStream_t s) {
    const bool fa = dtype_a == HGM_C64, fb = dtype_b == HGM_C64;
    if (fa && fb)
        hipLaunchKernelGGL((k_compare<float, float>), dim3(blocks), dim3(256), 0, s, (const float2 *)a, (const float2 *)b, n, partial);
    else if (fa)
        hipLaunchKernelGGL((k_compare<float, double>), dim3(blocks), dim3(256), 0, s, (const float2 *)a, (const double2 *)b, n, partial);
    else if (fb)
        hipLaunchKernelGGL((k_compare<double, float>), dim3(blocks), dim3(256), 0, s, (const double2 *)a, (const float2 *)b, n, partial);
    else
        hipLaunchKernelGGL((k_compare<double, double>), dim3(blocks), dim3(256), 0, s, (const double2 *)a, (const double2 *)b, n, partial);
    return hipGetLastError();
}

hipError_t launch_collapse(int dtype, void *state, uint64_t n, int bit, int outcome, double norm, hipStream_t s) {
    const uint64_t half = n / 2;
    const int blk = 256, grid = grid_for(half, blk);
    if (dtype == HGM_C64)
        hipLaunchKernelGGL(k_collapse<float>, dim3(grid), dim3(blk), 0, s, (float2 *)state, half, bit, outcome, norm);
    else
        hipLaunchKernelGGL(k_collapse<double>, dim3(grid), dim3(blk), 0, s, (double2 *)state, half, bit, outcome, norm);
    return hipGetLastError();
}

hipError_t launch_batch_reg(int dtype, int A, int B, const BatchItem *items, int n_items, int64_t total_tiles,
                            size_t lds_bytes, void *arena, hipStream_t s) {
    if (n_items < 1 || total_tiles < 1 || B < 1 || (uint64_t)total_tiles > max_blocks(B) || B > reg_kernel_max_threads(A, amp_bytes(dtype)) ||
        !arena)
        return hipErrorInvalidValue;
    char *base = static_cast<char *>(arena);
    return dtype == HGM_C64 ? batch_reg_any<float>(A, items, n_items, total_tiles, B, lds_bytes, base, s)
                            : batch_reg_any<double>(A, items, n_items, total_tiles, B, lds_bytes, base, s);
}

hipError_t launch_readout_final(const ReadoutTask *tasks, int n_tasks, hipStream_t s) {
    if (n_tasks < 1) return hipSuccess;
    hipLaunchKernelGGL(k_readout_final, dim3((unsigned)n_tasks), dim3(256), 0, s, tasks);
    return hipGetLastError();
}

}  // namespace hgm
