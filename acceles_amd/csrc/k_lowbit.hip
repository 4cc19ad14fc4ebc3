// k_lowbit.hip -- single-query low-bit kernels (three launches per query):
//   lowbit_slicemax  query quantization (quantify_util.py:31-49, 259) and the
//                    INT32 scores of the sliced packets (quantify_util.py:5-6,
//                    173-196; spmv_ucsr_top_k_multicore.hpp:195-355 on the
//                    FPGA); only the three largest of each 64-row slice (with
//                    many slices: the largest) are written;
//   lowbit_select    per partition: threshold = about its M-th best slice
//                    maximum (M distinct rows reach it, so no row below it can
//                    be in the partition's Top-M), the listed rows that reach
//                    it, exact rescan of the slices whose list may have
//                    dropped one, Top-M (quantify_util.py:173-196,
//                    host_spmv_ucsr.cpp:691-748) and FP32 rescoring of those
//                    rows (quantify_util.py:354-367);
//   lowbit_final_radix / lowbit_final
//                    the global Top-K of the rescored candidates;
//   lowbit_scores    INT32 scores of every row (parity checks).
// The streaming pass carries no selection state, so it runs at full
// occupancy with nothing but loads, decode and one wavefront max per slice.
#include "kernels_common.hpp"

#include <type_traits>

template <int E, bool SIGNED>
__device__ __forceinline__ int32_t slice_score(const LowbitArgs &a, const uint2 sl, const int8_t *qx) {
    const __amdgpu_buffer_rsrc_t rs = slice_rsrc(a.words, sl);
    int32_t acc = 0;
    for (int g0 = 0; g0 < (int)sl.y; g0 += E) {
        uint32_t w[E];
        load_group<E>(w, rs, g0);
        acc = decode_group<E, SIGNED>(w, min(E, (int)sl.y - g0), qx, a.col_bits, a.val_bits, acc);
    }
    return acc;
}

// The three largest of the lanes' scores and the lanes of the first two:
// (first, second, third, lane of first | lane of second << 8), in every lane.
__device__ __forceinline__ int4 top3(int32_t v) {
    const int lane = lane_id();
    int32_t m[3];
    int l[2];
#pragma unroll
    for (int i = 0; i < 3; ++i) {
        m[i] = __builtin_amdgcn_readlane(wave_max_lane63(v), 63);
        if (i < 2) {
            l[i] = __builtin_ctzll(__ballot(v == m[i]));
            v = lane == l[i] ? INT32_MIN : v;
        }
    }
    return make_int4(m[0], m[1], m[2], l[0] | (l[1] << 8));
}

// Work item blockIdx.x (a slice range of one partition): stop[s] = the three
// largest INT32 scores over the 64 lanes of slice s and the first two's
// lanes.  Padding lanes of a partition's last slice score 0, so that slice's
// may be too high; lowbit_select rescans it.  Without top3 only the largest
// is known, and lowbit_select rescans every slice that it needs.
//
// Bound: HBM (20,000,000 x 1024: 142 us, 6.5 TB/s of packets; 146 when 16 bytes
// per slice were written there too, 159 before the decode took four instructions
// per entry instead of six and the loads stayed in flight).  Small matrices: latency (400,000 x 500: 12.4 us, 13.4 before
// the first packets were loaded ahead of the query's quantization).
template <int E, bool SIGNED>
__global__ __launch_bounds__(LB_WG) void lowbit_slicemax(LowbitArgs a) {
    __shared__ __align__(16) int8_t qx[kMaxCols];
    __shared__ uint2 s_meta[LB_MAX_ITEM];
    __shared__ float red[LB_WAVES];
    const int4 item = a.items[blockIdx.x];
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)), lane = lane_id();
    // in order of use: the slices' metadata (into LDS) and the query, then the
    // first packets, whose latency covers the query's quantization (they
    // need the metadata of the wave's first two slices only, read here)
    const int nit = item.z - item.y;
    const uint2 m0 = a.slices[item.y + min((int)threadIdx.x, nit - 1)];
    float xr[kQueryRegs];
    load_query(a.x, a.cols, xr);
    const uint2 sl0 = a.slices[min(item.y + wave, item.z - 1)], sl1 = a.slices[min(item.y + wave + LB_WAVES, item.z - 1)];
    __builtin_amdgcn_sched_barrier(0);
    // Groups (E dwords per lane) of the wave's slices item.y + wave,
    // + LB_WAVES, ... stream through a ring of three register slots, two
    // groups ahead of the decoder.  Every load of the loop is unconditional
    // (through a buffer resource bounded by the slice, so loads past its end
    // return 0 and fetch nothing): a load whose result is merged into a loop
    // variable on only some paths is copied into place after a wait for all
    // outstanding loads, which would drain the ring.  A slot records the
    // group's slice, length and whether it ends the slice.
    constexpr int RING = 3;
    uint32_t w[RING][E];
    int ds[RING], dnd[RING];
    bool dend[RING], dval[RING];
    int ls = item.y + wave, lg = 0;  // load cursor
    uint2 lsl = ls < item.z ? sl0 : make_uint2(0u, 0u);
    // metadata of slice ls (head: before s_meta is published, at most the wave's second slice)
    auto meta = [&](bool head) { return ls >= item.z ? make_uint2(0u, 0u) : head ? sl1 : s_meta[ls - item.y]; };
    auto issue = [&](int slot, bool head) {
        const bool valid = ls < item.z;
        load_group<E>(w[slot], slice_rsrc(a.words, lsl), lg);
        __builtin_amdgcn_sched_barrier(0);  // keep the loads here: the scheduler would sink them to their use
        dval[slot] = valid;
        ds[slot] = ls;
        dnd[slot] = valid ? min(E, (int)lsl.y - lg) : 0;
        dend[slot] = valid && lg + E >= (int)lsl.y;
        if (valid) {
            if (dend[slot]) {
                ls += LB_WAVES;
                lg = 0;
                lsl = meta(head);
            } else {
                lg += E;
            }
        }
    };
    issue(0, true);
    issue(1, true);
    if ((int)threadIdx.x < nit) s_meta[threadIdx.x] = m0;
    for (int i = threadIdx.x + LB_WG; i < nit; i += LB_WG) s_meta[i] = a.slices[item.y + i];
    quantize_query_lds(a.x, a.cols, qx, red, nullptr, xr);  // its barriers also publish s_meta
    // the second issue may have moved on to the third slice
    if (ls >= item.y + wave + 2 * LB_WAVES) lsl = meta(false);
    int32_t acc = 0;
    bool done = false;
    while (!done) {
#pragma unroll
        for (int j = 0; j < RING; ++j) {
            if (done) break;
            if (!dval[j]) {
                done = true;
                break;
            }
            hold_group(w[j]);
            acc = decode_group<E, SIGNED>(w[j], dnd[j], qx, a.col_bits, a.val_bits, acc);
            if (dend[j]) {
                if (a.top3) {
                    const int4 t = top3(acc);
                    if (lane == 0) ((int4 *)a.stop)[ds[j]] = t;
                } else {
                    const int32_t t = wave_max_lane63(acc);
                    if (lane == 63) a.stop[ds[j]] = t;
                }
                acc = 0;
            }
            issue((j + 2) % RING, false);
        }
    }
}

// One workgroup of SEL_WG threads per partition p = blockIdx.x, after
// lowbit_slicemax.
// 1. ts: a score that M distinct rows reach, about the M-th largest of the
//    full slices' listed scores (radix selection that stops when at most kSlack
//    more reach it): every row of the partition's Top-M scores >= ts and lies
//    in a slice whose largest score is >= ts.
// 2. Of such a slice the two listed rows that reach ts go to an LDS key list.
//    If the third score reaches ts too (or the slice is not full), the slice
//    is rescanned exactly instead, CS slices at a time: their groups are
//    spread over all wavefronts (kU loads in flight per wavefront) and the
//    partial scores added into per-slice LDS sums, so long slices do not
//    serialize on one wavefront; rows >= ts are appended to the key list,
//    which is cut back to its best M whenever another chunk might not fit.
//    Where many slices would be, a query of zeros is looked for first: it
//    ranks the partition's rows in their order (400,000 x 500: 237 -> 27 us of
//    a call in 16 partitions, 1,984 -> 30 in one; a batch of such queries may
//    come here one by one).
// 3. The list's best M (by radix selection past 64), ranked by counting.  Past
//    kList slices to rescan or KCAP keys (heavy ties) each wavefront instead
//    rescans its share slice by slice into a wavefront Top-M collector.
// 4. Optional candidate output and the FP32 rescoring of the M rows.
//
// Bound: latency.  400,000 x 500 (196 slices, M = 16 per partition): 9.9 us;
// 15.1 when every slice that reaches ts was rescanned (16 slices, 5 us of
// decoding on one CU) after an exact threshold (3.6 us).  999,983 x 250: 9.1
// (before: 11.9), 20,000 x 500: 11.5 (17.2).
template <int E, bool SIGNED>
__global__ __launch_bounds__(SEL_WG) void lowbit_select(LowbitArgs a) {
    constexpr int V = 8;         // slice maxima per thread held in registers
    constexpr int kList = 2048;  // candidate slices listed in LDS
    constexpr int CS = 32;       // candidate slices per rescan chunk
    constexpr int kU = E <= 16 ? 3 : 2;  // groups in flight per wavefront (128 VGPRs at 16 waves)
    constexpr int KCAP = 4096;   // LDS key list (rows >= ts)
    constexpr int kSlack = 16;   // rows beyond M that may reach ts
    extern __shared__ __align__(16) unsigned char smem[];
    __shared__ __align__(16) int8_t qx[kMaxCols];
    __shared__ __align__(16) uint32_t s_hist[512];
    __shared__ int32_t s_list[kList];
    __shared__ uint2 s_lmeta[CS];
    __shared__ int32_t s_sum[CS * 64];
    __shared__ int s_ustart[CS + 1];
    __shared__ int s_n[SEL_WAVES];
    __shared__ int s_m, s_cnt, s_kn, s_tn, s_need[2];
    __shared__ uint32_t s_t32[2];
    __shared__ uint64_t s_t64[2];
    __shared__ __align__(16) uint64_t s_tmp[66], s_top[64];
    __shared__ uint2 s_rng[64];  // entry ranges of the rows in s_top
    float *red = (float *)smem;
    uint64_t *keys = (uint64_t *)(smem + 64);  // KCAP keys; the slow path's collectors reuse it
    float *xs = (float *)(smem + 64 + 8 * KCAP);  // FP32 query (rescoring)
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
    const int p = blockIdx.x;
    const int64_t s0 = a.part_slice[p];
    const int nsl = (int)(a.part_slice[p + 1] - s0);
    const int sw = a.top3 ? 4 : 1;  // dwords per slice
    const int32_t *stop = a.stop + s0 * sw;
    auto scores = [&](int i) {  // of slice i; without the top three second and third are unknown
        return a.top3 ? ((const int4 *)stop)[i] : make_int4(stop[i], INT32_MAX, INT32_MAX, 0);
    };
    const int32_t *perm = a.perm + s0 * 64;
    const bool regs = nsl <= V * SEL_WG, one = nsl <= SEL_WG;
    // the query and the thread's slices; one uniform test around loads with
    // clamped indices: they issue together (a per-element condition would
    // wait for each load)
    float xr[kQueryRegs];
    load_query(a.x, a.cols, xr);
    int4 st[V];
    int32_t r1 = -1, r2 = -1;  // one: the rows of the slice's two best scores
    auto load = [&](auto n, auto get) {
#pragma unroll
        for (int u = 0; u < V; ++u)
            st[u] = u < decltype(n)::value ? get(min(tid + u * SEL_WG, nsl - 1)) : make_int4(0, 0, 0, 0);
    };
    auto three = [&](int i) { return ((const int4 *)stop)[i]; };
    auto largest = [&](int i) { return make_int4(stop[i], INT32_MAX, INT32_MAX, 0); };
    if (nsl <= 0 || !regs) load(std::integral_constant<int, 0>(), three);
    else if (!a.top3) load(std::integral_constant<int, V>(), largest);
    else if (one) load(std::integral_constant<int, 1>(), three);
    else load(std::integral_constant<int, V>(), three);
    // every slice is full except a partition's last one
    const int nfull = nsl <= 0 || a.nvalid[s0 + nsl - 1] == 64 ? nsl : nsl - 1;
    if (tid == 0) {
        s_cnt = 0;
        s_kn = 0;
        s_tn = 0;
    }
#pragma unroll
    for (int u = 0; u < kQueryRegs; ++u)
        if (tid + u * SEL_WG < a.cols) xs[tid + u * SEL_WG] = xr[u];
    for (int c = tid + kQueryRegs * SEL_WG; c < a.cols; c += SEL_WG) xs[c] = a.x[c];
    if (one && nsl > 0) {  // in flight while the threshold is computed
        const int32_t *pr = perm + (size_t)min(tid, nsl - 1) * 64;
        r1 = pr[st[0].w & 63];
        r2 = pr[(st[0].w >> 8) & 63];
    }

    // 1. threshold (unsigned order: score ^ 2^31; key 0 = not a full slice).
    //    Up to SEL_WG slices: their three scores each (a partition of fewer
    //    than M slices has a threshold too), more: their largest.
    auto mkey = [](int32_t v, bool ok) -> uint32_t { return ok ? ((uint32_t)v ^ 0x80000000u) : 0u; };
    const uint32_t T = wg_radix_kth<uint32_t>(
        [&](auto fn) {
            if (one) {
                fn(mkey(st[0].x, tid < nfull));
                fn(mkey(st[0].y, a.top3 && tid < nfull));
                fn(mkey(st[0].z, a.top3 && tid < nfull));
            } else if (regs) {
#pragma unroll
                for (int u = 0; u < V; ++u) fn(mkey(st[u].x, tid + u * SEL_WG < nfull));
            } else {
                for (int i = tid; i < nsl; i += SEL_WG) fn(mkey(stop[(size_t)i * sw], i < nfull));
            }
        },
        a.M, s_hist, s_t32, s_need, kSlack);
    const int32_t ts = T == 0u ? INT32_MIN : (int32_t)(T ^ 0x80000000u);

    // 2. keys of the listed rows, slices to rescan
    auto slot = [&](int *count, bool ok) -> int {  // places in a list, for the lanes that are ok
        const uint64_t m = __ballot(ok);
        int base = 0;
        if (m != 0ull && lane == 0) base = atomicAdd(count, __popcll(m));
        return __builtin_amdgcn_readfirstlane(base) + mbcnt64(m);
    };
    auto offer = [&](int i, const int4 &t) {
        const bool cand = i < nsl && t.x >= ts;
        if (!__any(cand)) return;
        const bool again = cand && (i >= nfull || t.z >= ts), first = cand && !again, second = first && t.y >= ts;
        if (__any(again)) {
            const int j = slot(&s_cnt, again);
            if (again && j < kList) s_list[j] = i;
        }
        const int32_t *pr = perm + (size_t)i * 64;
        const int j1 = slot(&s_kn, first);
        if (first && j1 < KCAP) keys[j1] = dkey_i32(t.x, one ? r1 : pr[t.w & 63]);
        if (!__any(second)) return;
        const int j2 = slot(&s_kn, second);
        if (second && j2 < KCAP) keys[j2] = dkey_i32(t.y, one ? r2 : pr[(t.w >> 8) & 63]);
    };
    if (regs) {
#pragma unroll
        for (int u = 0; u < V; ++u)
            if (u * SEL_WG < nsl) offer(tid + u * SEL_WG, st[u]);
    } else {
        for (int b = 0; b < nsl; b += SEL_WG) offer(b + tid, scores(min(b + tid, nsl - 1)));
    }
    lds_barrier();
    const int ncand = s_cnt;
    int mcount = 0;
    // a query of zeros makes every row tie at 0: the partition's first M rows
    bool zero = false;
    if (a.part_row && (ncand > CS || s_kn > KCAP)) {
        if (tid == 0) s_m = 0;
        lds_barrier();
        bool any = false;
        for (int c = tid; c < a.cols; c += SEL_WG) any = any || xs[c] != 0.f;
        if (__any(any) && lane == 0) s_m = 1;
        lds_barrier();
        zero = s_m == 0;
    }
    if (!zero && (ncand > 0 || s_kn > KCAP)) quantize_query_lds(a.x, a.cols, qx, red, nullptr, xr);
    if (zero) {
        const int32_t row = a.part_row[p] + tid;
        mcount = min(a.M, (int)(a.part_row[p + 1] - a.part_row[p]));
        if (tid < mcount) {
            s_top[tid] = dkey_i32(0, row);
            if (a.K > 0) s_rng[tid] = make_uint2(a.ptr[row], a.ptr[row + 1]);
        }
        lds_barrier();
    } else if (ncand <= kList && s_kn <= KCAP) {
        // keeps the best M of the key list (all threads; the list is published)
        auto cut = [&](int n) -> int {
            const uint64_t Tk = wg_radix_kth<uint64_t>(
                [&](auto fn) {
                    for (int i = tid; i < n; i += SEL_WG) fn(keys[i]);
                },
                a.M, s_hist, s_t64, s_need);
            for (int i0 = 0; i0 < n; i0 += SEL_WG) {
                const int i = i0 + tid;
                const uint64_t k = i < n ? keys[i] : 0ull;
                const bool sel = k != 0ull && k >= Tk;
                const uint64_t m = __ballot(sel);
                if (m == 0) continue;
                int base = 0;
                if (lane == 0) base = atomicAdd(&s_tn, __popcll(m));
                base = __shfl(base, 0);
                const int j = base + mbcnt64(m);
                if (sel && j < 64) s_tmp[j] = k;  // j < M for distinct keys
            }
            lds_barrier();
            const int m = min(s_tn, a.M);
            lds_barrier();
            if (tid == 0) s_tn = 0;
            return m;
        };
        for (int cb = 0; cb < ncand; cb += CS) {
            const int cn = min(CS, ncand - cb);
            lds_barrier();  // metadata listed; the previous chunk's sums and keys in place
            if (s_kn > KCAP - CS * 64) {  // the next chunk might not fit: keep the best M
                const int m = cut(s_kn);
                if (tid < m) keys[tid] = s_tmp[tid];
                if (tid == 0) s_kn = m;
                lds_barrier();
            }
            for (int i = tid; i < CS * 64; i += SEL_WG) s_sum[i] = 0;
            if (wave == 0) {
                const uint2 sl = a.slices[s0 + s_list[cb + min(lane, cn - 1)]];
                if (lane < cn) s_lmeta[lane] = sl;
                const int ng = lane < cn ? ((int)sl.y + E - 1) / E : 0;
                const int inc = (int)wave_prefix_sum((uint32_t)ng);
                if (lane < CS) s_ustart[lane + 1] = inc;
                if (lane == 0) s_ustart[0] = 0;
            }
            constexpr int PR = CS / SEL_WAVES;  // slices each wavefront offers
            int32_t prow[PR];
#pragma unroll
            for (int r = 0; r < PR; ++r) {  // unconditional (clamped) lookups, masked after
                const int c = wave + r * SEL_WAVES;
                const int32_t v = perm[(size_t)s_list[cb + min(c, cn - 1)] * 64 + lane];
                prow[r] = c < cn ? v : -1;
            }
            lds_barrier();
            const int nu = s_ustart[cn];
            for (int u0 = wave * kU; u0 < nu; u0 += SEL_WAVES * kU) {
                uint32_t w[kU][E];
                int cu[kU], nd[kU];
#pragma unroll
                for (int t = 0; t < kU; ++t) {
                    const int u = u0 + t;
                    int c = -1, g0 = 0;
                    uint2 sl = make_uint2(0u, 0u);
                    if (u < nu) {
                        int lo = 0, hi = cn - 1;  // last c with s_ustart[c] <= u
                        while (lo < hi) {
                            const int mid = (lo + hi + 1) >> 1;
                            if (s_ustart[mid] <= u) lo = mid;
                            else hi = mid - 1;
                        }
                        c = lo;
                        g0 = (u - s_ustart[c]) * E;
                        sl = s_lmeta[c];
                    }
                    load_group<E>(w[t], slice_rsrc(a.words, sl), g0);
                    cu[t] = c;
                    nd[t] = c >= 0 ? min(E, (int)sl.y - g0) : 0;
                }
#pragma unroll
                for (int t = 0; t < kU; ++t) {
                    if (cu[t] < 0) continue;
                    const int32_t part = decode_group<E, SIGNED>(w[t], nd[t], qx, a.col_bits, a.val_bits, 0);
                    atomicAdd(&s_sum[cu[t] * 64 + lane], part);
                }
            }
            lds_barrier();
#pragma unroll
            for (int r = 0; r < PR; ++r) {
                const int c = wave + r * SEL_WAVES;
                if (c < cn) {
                    const int32_t sc = s_sum[c * 64 + lane];
                    const bool ok = prow[r] >= 0 && sc >= ts;
                    const uint64_t m = __ballot(ok);
                    if (m == 0) continue;
                    int base = 0;
                    if (lane == 0) base = atomicAdd(&s_kn, __popcll(m));
                    base = __shfl(base, 0);
                    if (ok) keys[base + mbcnt64(m)] = dkey_i32(sc, prow[r]);
                }
            }
        }
        lds_barrier();
        const int nk = s_kn;
        const uint64_t *src = keys;  // nk <= 64 keys, or the best M of more
        int n = nk;
        if (nk > 64) {
            n = cut(nk);
            src = s_tmp;
        }
        mcount = min(n, a.M);
        // rank by counting (keys are distinct), two keys per read; the rows'
        // entry ranges are in flight meanwhile
        uint64_t k = 0ull;
        uint2 rg = make_uint2(0u, 0u);
        if (tid < n) {
            k = src[tid];
            if (a.K > 0) rg = make_uint2(a.ptr[dkey_row(k)], a.ptr[dkey_row(k) + 1]);
        }
        if (tid == n) (nk > 64 ? s_tmp : keys)[n] = 0ull;
        lds_barrier();
        if (tid < n) {
            int rank = 0;
            for (int j = 0; j < n; j += 2) {
                const ulonglong2 o = *(const ulonglong2 *)(src + j);
                rank += (o.x > k) + (o.y > k);
            }
            if (rank < a.M) {
                s_top[rank] = k;
                s_rng[rank] = rg;
            }
        }
        lds_barrier();
    } else {
        uint64_t *colbuf = keys;
        WaveTopM<2> col;
        col.init(colbuf + wave * WaveTopM<2>::cap, a.M);
        for (int b = wave * 64; b < nsl; b += SEL_WG) {
            uint64_t mask = __ballot(b + lane < nsl && stop[(size_t)min(b + lane, nsl - 1) * sw] >= ts);
            while (mask) {
                const int l = __builtin_ctzll(mask);
                mask &= mask - 1;
                const int64_t s = s0 + b + l;
                const int32_t sc = slice_score<E, SIGNED>(a, a.slices[s], qx);
                const int32_t row = a.perm[s * 64 + lane];
                col.push(row >= 0 && sc >= ts, dkey_i32(sc, row));
            }
        }
        col.compact();
        if (lane == 0) s_n[wave] = col.n;
        lds_barrier();
        if (wave == 0) {
            wg_merge(col, colbuf, s_n, SEL_WAVES);
            if (lane < col.n) {  // col.n <= M <= 64, sorted
                const uint64_t k = col.buf[lane];
                s_top[lane] = k;
                if (a.K > 0) s_rng[lane] = make_uint2(a.ptr[dkey_row(k)], a.ptr[dkey_row(k) + 1]);
            }
            if (lane == 0) s_m = col.n;
        }
        lds_barrier();
        mcount = s_m;
    }
    const uint64_t *top = s_top;
    if (a.cand_rows_out) {
        for (int i = threadIdx.x; i < a.M; i += SEL_WG) {
            a.cand_rows_out[(size_t)p * a.M + i] = i < mcount ? dkey_row(top[i]) : -1;
            a.cand_scores_out[(size_t)p * a.M + i] = i < mcount ? dkey_score_i32(top[i]) : 0;
        }
    }
    if (a.K <= 0) return;

    // 4. FP32 rescoring of the partition's candidates (8 entries per lane in
    //    flight: a row has two to four per lane on average; the query from LDS)
    for (int base = 0; base < a.M; base += SEL_WG / a.G) {
        const int i = base + (int)threadIdx.x / a.G;
        const bool valid = i < mcount;
        const uint2 rg = valid ? s_rng[i] : make_uint2(0u, 0u);
        const float sc = group_dot_range<8>(a.idx, a.val, xs, rg.x, rg.y, a.G);
        if ((threadIdx.x & (a.G - 1)) == 0 && i < a.M)
            a.resc[(size_t)p * a.M + i] = valid ? dkey_f32(sc, dkey_row(top[i])) : 0ull;
    }
}

// One workgroup: the global Top-K of the split*M rescored candidates
// (split*M <= 4*64*R), ranks by merging sorted wavefront lists.
template <int R>
__global__ __launch_bounds__(ACC_WG) void lowbit_final(LowbitArgs a) {
    extern __shared__ __align__(16) unsigned char smem[];
    __shared__ int s_nz[ACC_WAVES];
    topk_by_rank<R>(a.resc, a.split * a.M, a.K, a.out, (uint64_t *)smem, s_nz);
}

// The same for K <= 256 by radix selection (split*M <= V*SEL_WG).
template <int V>
__global__ __launch_bounds__(SEL_WG) void lowbit_final_radix(LowbitArgs a) {
    __shared__ __align__(16) uint32_t lds[1036];
    topk_radix<V>(a.resc, a.split * a.M, a.K, a.out, lds);
}

// INT32 scores of every row (one work item per wavefront).

template <int E, bool SIGNED>
__global__ __launch_bounds__(ACC_WG) void lowbit_scores(ScoresArgs a) {
    __shared__ __align__(16) int8_t qx[kMaxCols];
    __shared__ float red[ACC_WAVES];
    quantize_query_lds(a.x, a.cols, qx, red);
    const int lane = lane_id();
    for (int64_t s = (int64_t)blockIdx.x * ACC_WAVES + (threadIdx.x >> 6); s < a.nslices;
         s += (int64_t)gridDim.x * ACC_WAVES) {
        const uint2 sl = a.slices[s];
        const __amdgpu_buffer_rsrc_t rs = slice_rsrc(a.words, sl);
        int32_t acc = 0;
        for (int g0 = 0; g0 < (int)sl.y; g0 += E) {
            uint32_t w[E];
            load_group<E>(w, rs, g0);
            acc = decode_group<E, SIGNED>(w, min(E, (int)sl.y - g0), qx, a.col_bits, a.val_bits, acc);
        }
        const int32_t row = a.perm[s * 64 + lane];
        if (row >= 0) a.y[row] = acc;
    }
}


template <bool SIGNED>
static lowbit_fn slicemax_for(int E) {
    switch (E) {
#define CASE(e) case e: return lowbit_slicemax<e, SIGNED>;
        CASE(10) CASE(11) CASE(12) CASE(13) CASE(14) CASE(15) CASE(16)
        CASE(17) CASE(18) CASE(19) CASE(20) CASE(21) CASE(22)
#undef CASE
        default: return nullptr;
    }
}

template <bool SIGNED>
static lowbit_fn select_for(int E) {
    switch (E) {
#define CASE(e) case e: return lowbit_select<e, SIGNED>;
        CASE(10) CASE(11) CASE(12) CASE(13) CASE(14) CASE(15) CASE(16)
        CASE(17) CASE(18) CASE(19) CASE(20) CASE(21) CASE(22)
#undef CASE
        default: return nullptr;
    }
}

template <bool SIGNED>
static scores_fn scores_for(int E) {
    switch (E) {
#define CASE(e) case e: return lowbit_scores<e, SIGNED>;
        CASE(10) CASE(11) CASE(12) CASE(13) CASE(14) CASE(15) CASE(16)
        CASE(17) CASE(18) CASE(19) CASE(20) CASE(21) CASE(22)
#undef CASE
        default: return nullptr;
    }
}

lowbit_fn get_lowbit_slicemax(int E, bool is_signed) {
    return is_signed ? slicemax_for<true>(E) : slicemax_for<false>(E);
}
lowbit_fn get_lowbit_select(int E, bool is_signed) { return is_signed ? select_for<true>(E) : select_for<false>(E); }
lowbit_fn get_lowbit_final_radix(int V) {
    return V <= 1 ? lowbit_final_radix<1> : V <= 2 ? lowbit_final_radix<2> : lowbit_final_radix<4>;
}
lowbit_fn get_lowbit_final(int R) {
    switch (R) {
        case 1: return lowbit_final<1>;
        case 2: return lowbit_final<2>;
        case 4: return lowbit_final<4>;
        case 8: return lowbit_final<8>;
        case 16: return lowbit_final<16>;
        default: return nullptr;
    }
}
scores_fn get_lowbit_scores(int E, bool is_signed) { return is_signed ? scores_for<true>(E) : scores_for<false>(E); }
