// device_common.hpp -- device helpers shared by the HIP kernels (gfx950,
// wave64): ranking keys, wave primitives and the wavefront Top-M collector.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

#define ACC_WG 256                 // threads per workgroup (4 wavefronts)
#define ACC_WAVES (ACC_WG / 64)

// Ranking keys: a larger key ranks first.  High 32 bits: the score mapped to
// an order-preserving unsigned; low 32 bits: ~row, so on equal scores the
// lower row ranks first.  0 never occurs for a real row (row < 2^31).
__device__ __forceinline__ uint64_t dkey_i32(int32_t s, int32_t row) {
    return ((uint64_t)((uint32_t)s ^ 0x80000000u) << 32) | (uint64_t)(0xFFFFFFFFu - (uint32_t)row);
}
__device__ __forceinline__ uint32_t dordered_f32(float f) {
    uint32_t b = __float_as_uint(f == 0.0f ? 0.0f : f);
    return (b & 0x80000000u) ? ~b : (b | 0x80000000u);
}
__device__ __forceinline__ uint64_t dkey_f32(float s, int32_t row) {
    return ((uint64_t)dordered_f32(s) << 32) | (uint64_t)(0xFFFFFFFFu - (uint32_t)row);
}
__device__ __forceinline__ int32_t dkey_row(uint64_t k) { return (int32_t)(0xFFFFFFFFu - (uint32_t)k); }
__device__ __forceinline__ int32_t dkey_score_i32(uint64_t k) { return (int32_t)((uint32_t)(k >> 32) ^ 0x80000000u); }
__device__ __forceinline__ float dkey_score_f32(uint64_t k) {
    uint32_t o = (uint32_t)(k >> 32);
    uint32_t b = (o & 0x80000000u) ? (o & 0x7FFFFFFFu) : ~o;
    return __uint_as_float(b);
}

__device__ __forceinline__ int lane_id() { return (int)__lane_id(); }

// Orders LDS traffic between the lanes of one wavefront.  The fence names
// the LDS address space only: a wavefront's LDS operations complete in order,
// and a fence over all memory would also wait for every global load in flight
// (draining the prefetch rings of the streaming kernels).
__device__ __forceinline__ void wave_sync() {
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront", "local");
    __builtin_amdgcn_wave_barrier();
}

// Workgroup barrier for LDS only: waits for this wavefront's LDS operations,
// not for its global loads (a full barrier would also wait for the packet
// loads issued for the slices ahead).
__device__ __forceinline__ void lds_barrier() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// Maximum over the wavefront, valid in lane 63 (DPP steps: quad swaps,
// half-row and row mirrors, then the row 15 / row 31 broadcasts).
template <int CTRL, int ROWS>
__device__ __forceinline__ int32_t dpp_max_step(int32_t v) {
    return max(v, __builtin_amdgcn_update_dpp(v, v, CTRL, ROWS, 0xF, false));
}
template <int CTRL, int ROWS>
__device__ __forceinline__ uint32_t dpp_umax_step(uint32_t v) {
    return max(v, (uint32_t)__builtin_amdgcn_update_dpp((int)v, (int)v, CTRL, ROWS, 0xF, false));
}
// Unsigned maximum over the wavefront, returned to every lane.
__device__ __forceinline__ uint32_t wave_umax(uint32_t v) {
    v = dpp_umax_step<0xB1, 0xF>(v);
    v = dpp_umax_step<0x4E, 0xF>(v);
    v = dpp_umax_step<0x141, 0xF>(v);
    v = dpp_umax_step<0x140, 0xF>(v);
    v = dpp_umax_step<0x142, 0xA>(v);
    v = dpp_umax_step<0x143, 0xC>(v);
    return (uint32_t)__builtin_amdgcn_readlane((int)v, 63);
}
__device__ __forceinline__ int32_t wave_max_lane63(int32_t v) {
    v = dpp_max_step<0xB1, 0xF>(v);   // quad_perm [1,0,3,2]
    v = dpp_max_step<0x4E, 0xF>(v);   // quad_perm [2,3,0,1]
    v = dpp_max_step<0x141, 0xF>(v);  // row_half_mirror
    v = dpp_max_step<0x140, 0xF>(v);  // row_mirror
    v = dpp_max_step<0x142, 0xA>(v);  // row_bcast:15 into rows 1 and 3
    v = dpp_max_step<0x143, 0xC>(v);  // row_bcast:31 into rows 2 and 3
    return v;
}

// Inclusive prefix sum over the wavefront (DPP row shifts, then the row 15 /
// row 31 broadcasts: eight VALU steps against six LDS shuffles).
template <int CTRL, int ROWS>
__device__ __forceinline__ uint32_t dpp_add_step(uint32_t v) {
    return v + (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, CTRL, ROWS, 0xF, false);
}
__device__ __forceinline__ uint32_t wave_prefix_sum(uint32_t v) {
    // shifts by 1, 2, 4 and 8 inside the 16-lane rows (lanes without a source add 0)
    v = dpp_add_step<0x111, 0xF>(v);
    v = dpp_add_step<0x112, 0xF>(v);
    v = dpp_add_step<0x114, 0xF>(v);
    v = dpp_add_step<0x118, 0xF>(v);
    v = dpp_add_step<0x142, 0xA>(v);
    v = dpp_add_step<0x143, 0xC>(v);
    return v;
}

// p + the value of lane ^ S, S a power of two below 32: the rounding of p +
// __shfl_xor(p, S) without the LDS crossbar.  Lane ^ 4 is the quad reversal
// of the half-row mirror; lane ^ 16 comes from v_permlane16_swap, whose two
// results hold the even and the odd 16-lane rows.
template <int S>
__device__ __forceinline__ float xor_add(float p) {
    const int v = __float_as_int(p);
    if constexpr (S == 1) return p + __int_as_float(__builtin_amdgcn_update_dpp(v, v, 0xB1, 0xF, 0xF, false));
    if constexpr (S == 2) return p + __int_as_float(__builtin_amdgcn_update_dpp(v, v, 0x4E, 0xF, 0xF, false));
    if constexpr (S == 4) {
        const int t = __builtin_amdgcn_update_dpp(v, v, 0x1B, 0xF, 0xF, false);
        return p + __int_as_float(__builtin_amdgcn_update_dpp(t, t, 0x141, 0xF, 0xF, false));
    }
    if constexpr (S == 8) return p + __int_as_float(__builtin_amdgcn_update_dpp(v, v, 0x128, 0xF, 0xF, false));
    if constexpr (S == 16) {
        const auto r = __builtin_amdgcn_permlane16_swap((uint32_t)v, (uint32_t)v, false, false);
        return __uint_as_float(r[0]) + __uint_as_float(r[1]);
    }
    return p;
}
template <int G>
__device__ __forceinline__ float butterfly(float p) {
    if constexpr (G > 16) p = xor_add<16>(p);
    if constexpr (G > 8) p = xor_add<8>(p);
    if constexpr (G > 4) p = xor_add<4>(p);
    if constexpr (G > 2) p = xor_add<2>(p);
    return xor_add<1>(p);
}
// A bound that at least need of the U values per lane of the wavefront reach,
// and at most need + slack unless equal values force more (0 = no value;
// returns 0 when fewer than need are nonzero): bisection between the smallest
// lane maximum and the largest value, one comparison and scalar bit count per
// value and step (no LDS; about 100 cycles a step for U = 4).
template <int U>
__device__ __forceinline__ uint32_t wave_bound_u32(const uint32_t (&v)[U], int need, int slack) {
    uint32_t m = 0u;
#pragma unroll
    for (int u = 0; u < U; ++u) m = max(m, v[u]);
    auto count = [&](uint32_t t) {
        int c = 0;
#pragma unroll
        for (int u = 0; u < U; ++u) c += __popcll(__ballot(v[u] >= t));
        return c;
    };
    uint32_t hi = wave_umax(m), lo = max(~wave_umax(~m), 1u);
    int c = count(lo);
    if (c < need) {
        lo = 1u;
        c = count(lo);
        if (c < need) return 0u;
    }
    while (c > need + slack && hi > lo) {
        const uint32_t mid = lo + (hi - lo + 1u) / 2u;
        const int cm = count(mid);
        if (cm >= need) {
            lo = mid;
            c = cm;
        } else {
            hi = mid - 1u;
        }
    }
    return lo;
}

__device__ __forceinline__ int mbcnt64(uint64_t mask) {
    return (int)__builtin_amdgcn_mbcnt_hi((uint32_t)(mask >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)mask, 0u));
}

__device__ __forceinline__ uint64_t atomic_load_u64(const uint64_t *p) {
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

__device__ __forceinline__ uint64_t shfl_u64(uint64_t v, int src) {
    uint32_t lo = (uint32_t)__shfl((int)(uint32_t)v, src);
    uint32_t hi = (uint32_t)__shfl((int)(uint32_t)(v >> 32), src);
    return ((uint64_t)hi << 32) | lo;
}

__device__ __forceinline__ uint64_t readlane_u64(uint64_t v, int l) {  // l uniform
    return ((uint64_t)(uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(v >> 32), l) << 32) |
           (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)v, l);
}

__device__ __forceinline__ uint64_t shfl_xor_u64(uint64_t v, int m) {
    uint32_t lo = (uint32_t)__shfl_xor((int)(uint32_t)v, m);
    uint32_t hi = (uint32_t)__shfl_xor((int)(uint32_t)(v >> 32), m);
    return ((uint64_t)hi << 32) | lo;
}

// Bitonic sort, descending, of 64*R keys held in registers: element
// i = r*64 + lane lives in v[r] of that lane.  Stages with j >= 64 exchange
// slots inside a lane; the others exchange lanes with shfl_xor.
template <int R>
__device__ __forceinline__ void reg_sort_desc(uint64_t (&v)[R]) {
    const int lane = lane_id();
#pragma unroll
    for (int k = 2; k <= 64 * R; k <<= 1) {
#pragma unroll
        for (int j = k >> 1; j > 0; j >>= 1) {
            if (j >= 64) {
#pragma unroll
                for (int r = 0; r < R; ++r) {
                    const int rp = r ^ (j >> 6);
                    if (rp > r) {
                        const bool desc = ((r * 64 + lane) & k) == 0;
                        const uint64_t a = v[r], b = v[rp];
                        const bool sw = desc ? (a < b) : (a > b);
                        v[r] = sw ? b : a;
                        v[rp] = sw ? a : b;
                    }
                }
            } else {
                const bool lower = (lane & j) == 0;
#pragma unroll
                for (int r = 0; r < R; ++r) {
                    const uint64_t o = shfl_xor_u64(v[r], j);
                    const bool desc = ((r * 64 + lane) & k) == 0;
                    const bool take_max = lower == desc;
                    v[r] = take_max ? (v[r] > o ? v[r] : o) : (v[r] < o ? v[r] : o);
                }
            }
        }
    }
}

// Wavefront Top-M collector over an LDS buffer of cap = 64*R keys
// (M <= cap - 64).  All state is wave-uniform.  push() is called by all 64
// lanes together; each lane offers at most one key.  Appends go to LDS; a
// compaction reads the buffer into registers, sorts there and writes back the
// best M.
template <int R>
struct WaveTopM {
    static constexpr int cap = 64 * R;
    uint64_t *buf;
    int n, M;
    uint64_t thr;  // a key must be > thr to be kept (the M-th best once full)

    __device__ void init(uint64_t *b, int m) {
        buf = b;
        M = m;
        n = 0;
        thr = 0;
    }
    // Sort, keep the best M, set the admission threshold.
    __device__ void compact() {
        const int lane = lane_id();
        if (n <= 32) {
            // few keys: each finds its rank by counting the keys above it (equal
            // keys, should any occur, are ordered by lane), then moves there
            const uint64_t k = lane < n ? buf[lane] : 0ull;
            const uint32_t klo = (uint32_t)k, khi = (uint32_t)(k >> 32);
            int rank = 0;
            for (int j = 0; j < n; ++j) {
                const uint64_t kj = ((uint64_t)(uint32_t)__builtin_amdgcn_readlane((int)khi, j) << 32) |
                                    (uint32_t)__builtin_amdgcn_readlane((int)klo, j);
                rank += (kj > k || (kj == k && j < lane)) ? 1 : 0;
            }
            const int nn = n < M ? n : M;
            wave_sync();
            if (lane < n && rank < nn) buf[rank] = k;
            if (nn == M && M > 0) {
                const uint64_t bm = __ballot(lane < n && rank == M - 1);
                thr = shfl_u64(k, __builtin_ctzll(bm));
            }
            n = nn;
            wave_sync();
            return;
        }
        if (R > 1 && n <= 64) {  // one register of keys: a 64-key sort
            uint64_t w[1] = {lane < n ? buf[lane] : 0ull};
            reg_sort_desc<1>(w);
            n = n < M ? n : M;
            if (lane < n) buf[lane] = w[0];
            if (n == M && M > 0) thr = shfl_u64(w[0], M - 1);
            wave_sync();
            return;
        }
        uint64_t v[R];
#pragma unroll
        for (int r = 0; r < R; ++r) v[r] = (r * 64 + lane < n) ? buf[r * 64 + lane] : 0ull;
        reg_sort_desc<R>(v);
        n = n < M ? n : M;
#pragma unroll
        for (int r = 0; r < R; ++r)
            if (r * 64 + lane < n) buf[r * 64 + lane] = v[r];
        if (n == M && M > 0) {
            uint64_t t = 0;
#pragma unroll
            for (int r = 0; r < R; ++r)
                if (r == (M - 1) >> 6) t = v[r];
            thr = shfl_u64(t, (M - 1) & 63);
        }
        wave_sync();
    }
    __device__ void push(bool pred, uint64_t key) {
        pred = pred && key > thr;
        uint64_t mask = __ballot(pred);
        if (mask == 0) return;
        int c = __popcll(mask);
        if (n + c > cap) {
            compact();
            pred = pred && key > thr;
            mask = __ballot(pred);
            c = __popcll(mask);
        }
        if (pred) buf[n + mbcnt64(mask)] = key;
        wave_sync();
        n += c;
    }
};
