// The LDS pass kernel.
//
// k_pass_lds: one workgroup per tile of 2^r amplitudes. The tile's local index
// L maps to the state index base | (L & cmask) | deposit(L >> c), where the
// low c bits stay contiguous (so a wave's loads cover runs of 2^c amplitudes)
// and deposit() scatters the remaining r-c tile bits onto the pass's chosen
// state-index bits through three 64-entry LDS tables. Thread t owns local
// indices t + k*B (k < 2R) for loading, storing and diagonal gates; for a
// pair-mixing gate it takes pairs t + k*B (k < R) and inserts a zero at the
// target's tile bit. Barriers are placed only where ownership changes.
#include "device.hpp"
#include "kernels.hpp"

namespace hgm {

namespace {

__device__ __forceinline__ uint64_t pdep64(uint64_t v, uint64_t mask) {
    uint64_t r = 0;
    for (uint64_t bb = 1; mask; bb <<= 1) {
        uint64_t lowbit = mask & (~mask + 1);
        if (v & bb) r |= lowbit;
        mask &= mask - 1;
    }
    return r;
}

template <class T>
__global__ void __launch_bounds__(1024) k_pass_lds(typename Vec<T>::type *__restrict__ state,
                                                   const DevOp *__restrict__ ops, int n_ops, PassArgs a) {
    using V = typename Vec<T>::type;
    extern __shared__ __align__(16) unsigned char smem[];
    uint64_t *dep = reinterpret_cast<uint64_t *>(smem);      // 3 tables of 64 entries
    V *tile = reinterpret_cast<V *>(smem + 3 * 64 * sizeof(uint64_t));

    const int t = threadIdx.x;
    const int hi_bits = a.r - a.c;
    for (int x = t; x < 192; x += blockDim.x) {
        const int tab = x >> 6, v = x & 63;
        uint64_t acc = 0;
        for (int j = 0; j < 6; ++j) {
            const int lb = tab * 6 + j;
            if (((v >> j) & 1) && lb < hi_bits) acc |= uint64_t(1) << a.local_pos[a.c + lb];
        }
        dep[x] = acc;
    }
    __syncthreads();

    const int B = a.B, R = a.R, c = a.c;
    const uint32_t cmask = (1u << c) - 1u;
    for (int64_t tid = blockIdx.x; tid < a.n_tiles; tid += gridDim.x) {
        const uint64_t base = pdep64((uint64_t)tid, a.nonlocal_mask);
        // load
        for (int k = 0; k < 2 * R; ++k) {
            const uint32_t L = (uint32_t)(t + k * B);
            const uint32_t h = L >> c;
            const uint64_t g = base | (L & cmask) | dep[h & 63] | dep[64 + ((h >> 6) & 63)] | dep[128 + ((h >> 12) & 63)];
            tile[L] = state[g];
        }
        bool last_pair = false;
        for (int i = 0; i < n_ops; ++i) {
            const DevOp &o = ops[i];
            if ((base & o.gmask) != o.gval) continue;   // tile-uniform
            const T m0r = (T)o.m[0], m0i = (T)o.m[1], m1r = (T)o.m[2], m1i = (T)o.m[3];
            const T m2r = (T)o.m[4], m2i = (T)o.m[5], m3r = (T)o.m[6], m3i = (T)o.m[7];
            if (o.kind == K_DENSE || o.kind == K_ANTI) {
                __syncthreads();
                const int tb = o.tbit;
                const uint32_t tmask = 1u << tb;
                for (int k = 0; k < R; ++k) {
                    const uint32_t p = (uint32_t)(t + k * B);
                    const uint32_t p0 = ((p >> tb) << (tb + 1)) | (p & (tmask - 1u));
                    const uint32_t p1 = p0 | tmask;
                    if ((p0 & o.lmask) != o.lval) continue;
                    const V x = tile[p0], y = tile[p1];
                    if (o.kind == K_DENSE) {
                        tile[p0] = cmul2<V, T>(m0r, m0i, x, m1r, m1i, y);
                        tile[p1] = cmul2<V, T>(m2r, m2i, x, m3r, m3i, y);
                    } else {
                        tile[p0] = cmul<V, T>(m1r, m1i, y);
                        tile[p1] = cmul<V, T>(m2r, m2i, x);
                    }
                }
                last_pair = true;
            } else {
                if (last_pair) { __syncthreads(); last_pair = false; }
                if (o.kind == K_DIAG) {
                    const int tb = o.tbit;
                    for (int k = 0; k < 2 * R; ++k) {
                        const uint32_t L = (uint32_t)(t + k * B);
                        if ((L & o.lmask) != o.lval) continue;
                        const bool one = (L >> tb) & 1u;
                        tile[L] = one ? cmul<V, T>(m3r, m3i, tile[L]) : cmul<V, T>(m0r, m0i, tile[L]);
                    }
                } else {   // K_DIAG_GLOBAL
                    const bool one = (base >> o.tbit) & 1u;
                    const T pr = one ? m3r : m0r, pi = one ? m3i : m0i;
                    for (int k = 0; k < 2 * R; ++k) {
                        const uint32_t L = (uint32_t)(t + k * B);
                        if ((L & o.lmask) != o.lval) continue;
                        tile[L] = cmul<V, T>(pr, pi, tile[L]);
                    }
                }
            }
        }
        if (last_pair) __syncthreads();
        // store
        for (int k = 0; k < 2 * R; ++k) {
            const uint32_t L = (uint32_t)(t + k * B);
            const uint32_t h = L >> c;
            const uint64_t g = base | (L & cmask) | dep[h & 63] | dep[64 + ((h >> 6) & 63)] | dep[128 + ((h >> 12) & 63)];
            state[g] = tile[L];
        }
        __syncthreads();   // the next tile reuses the LDS
    }
}

// The kernel's dynamic LDS limit, raised once (before the first launch, and
// before any stream capture that launches it).
template <class T>
hipError_t pass_lds_attr() {
    static const hipError_t e =
        hipFuncSetAttribute((const void *)k_pass_lds<T>, hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
    return e;
}
template <class T>
hipError_t pass_lds(void *state, const DevOp *ops, int n_ops, const PassArgs &a, hipStream_t s) {
    pass_lds_attr<T>();
    const size_t lds = 3 * 64 * sizeof(uint64_t) + (size_t(1) << a.r) * sizeof(typename Vec<T>::type);
    const int64_t grid = tile_grid(a.n_tiles, a.B);
    hipLaunchKernelGGL(k_pass_lds<T>, dim3((unsigned)grid), dim3(a.B), lds, s,
                       reinterpret_cast<typename Vec<T>::type *>(state), ops, n_ops, a);
    return hipGetLastError();
}

}  // namespace

hipError_t launch_pass_lds(int dtype, void *state, const DevOp *ops, int n_ops, const PassArgs &a, hipStream_t s) {
    return dtype == HGM_C64 ? pass_lds<float>(state, ops, n_ops, a, s) : pass_lds<double>(state, ops, n_ops, a, s);
}

hipError_t prepare_pass_lds(int dtype) { return dtype == HGM_C64 ? pass_lds_attr<float>() : pass_lds_attr<double>(); }

}  // namespace hgm
