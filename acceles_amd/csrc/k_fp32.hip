// k_fp32.hip -- plain FP32 CSR path and FP64 exact scores:
//   fp32_spmv       FP32 CSR SpMV (cpu_mkl_baseline.cpp:261);
//   fp32_select_groups
//                   Top-K of its scores (cpu_mkl_baseline.cpp:128-149) from
//                   the three best keys of each group's rows (wavefronts or
//                   workgroups); together they are the plain FP32 CSR Top-K path
//                   (host_spmv_topk_csr_gpu.cu:171-231 is the GPU spec);
//   select_radix_pass / select_radix_final (K <= 256),
//   select_blocks / select_final (any K <= 960)
//                   Top-K of any score vector, and of a matrix with fewer
//                   than K groups' worth of rows;
//   spmv_fp64       FP64 exact scores for precision/recall reporting.
#include "kernels_common.hpp"

#include <algorithm>
#include <type_traits>

// ---------------------------------------------------------------------------
// FP32 CSR path
// ---------------------------------------------------------------------------

// y = A x with G lanes per row.  Lane g of a row sums its entries
// g, g+G, g+2G, ... in that order with fmaf, then an xor butterfly of plain
// adds.
//
// Bound: HBM, 6 bytes per entry; the LDS pipe is next (three LDS reads per
// entry slot).  A step is RS = B * 64/G rows, one contiguous range of
// entries; the steps are dealt to the wavefronts in turn, so that the
// wavefronts in flight read neighbouring entries.  A step's entries are read
// with 16-byte loads (whole cache lines, each byte once) into registers one
// step ahead, written to the wavefront's LDS area and summed from there in
// the G-lane order.  The loads go through buffer resources that end with the
// step's range, so they are unconditional (a conditional load is waited for
// before the next is issued) and fetch nothing else; past the range they
// leave zeros.  The row starts of a step are one load, two steps ahead, and
// reach the rows' lanes through LDS.  x is staged in LDS at offset 0, where a
// stored column is its address.
//
// The area: 896 entries at 6 bytes leave five workgroups per CU at 900
// columns.  2,000,000 x 900 (rows of 30-90, G = 16): 138 us, 5.2 TB/s; with
// areas of 768 / 1024 / 1536 entries 145 / 162 / 143 us; loading the rows'
// entries with 4-byte loads and 4-byte columns 286 us.  4,999,999 x 1024
// power-law rows (G = 8): 175 us (258 with such loads; under the profiler, which
// adds a tenth to this kernel, 196 against 211 with 768 entries and 232 with
// 1024: the other figures for these rows below are under it too).
// 100,000 x 500 (rows of 50-90, G = 32): 11.2 us (before: 15.3).
static constexpr int kFp32Stage = 896;   // entries per wavefront staged in LDS
static constexpr int kFp32Slack = 128;   // readable past them (the last batch of a row reads up to U*G - 1 further)
static constexpr int kFp32Area = kFp32Stage + kFp32Slack;

template <int G, int B>
struct SpmvShape {
    static constexpr int RPI = 64 / G;              // rows per block
    static constexpr int RS = B * RPI;              // rows per step
    static constexpr int NP = RS / 64 + 1;          // loads of its RS + 1 row starts
    // entries per lane in the first batch (of all blocks) and in one further
    // batch of a block: the slots past a row's end are wasted LDS reads
    // (power-law rows: 206 us with further batches of four, 196 with two)
    static constexpr int U = G >= 16 ? 3 : 4, kTail = 2;
    static constexpr int kWave = kFp32Area * 6 + NP * 256;  // LDS bytes of a wavefront
};

// B of a matrix of this mean row length: a mean step fills at most 85% of the
// staging area (row lengths vary; 75% and 95%, i.e. two and four blocks
// instead of three, were slower at 2,000,000 x 900: 145 and 188 against 141
// us), at most 4 blocks, so that a step's
// registers leave five wavefronts per SIMD.  One block less of three or four
// where a step two standard deviations above the mean would not fit: a step that
// exceeds the area waits for each of its blocks (power-law rows of 20 entries on
// average, 5M x 1024: three blocks 196 us, four 209, two 215).
int fp32_step_blocks(int G, double mean_row, double row_sd) {
    const int RPI = 64 / G;
    const double per_block = std::max(mean_row, 1.0) * RPI;
    const int B = std::max(1, (int)std::min(4.0, 0.85 * kFp32Stage / per_block));
    return B > 2 && B * per_block + 2.0 * row_sd * std::sqrt((double)B * RPI) > kFp32Stage ? B - 1 : B;
}

// With gmax, group w also leaves the three largest ranking keys of its rows
// (gmax[w] and the pair at gmax[group_pairs(groups) + 2w], 0 without such a row) for
// fp32_select_groups; a group is a wavefront, or with wg_groups a workgroup.
// Each lane of a row's group holds the row's sum, so lane
// g of the group takes block g's row: one update of a lane's best keys per step
// instead of one per block.  A key of 1 stands for a score whose order is 0 or 1 (a
// NaN of all ones).
template <int G, int B>
__global__ __launch_bounds__(ACC_WG) void fp32_spmv(const uint32_t *ptr, const colx_t *idx, const float *val,
                                                   const float *x, int rows, int cols, float *y, uint64_t *gmax,
                                                   int wg_groups) {
    using S = SpmvShape<G, B>;
    constexpr int RPI = S::RPI, RS = S::RS, NP = S::NP, U = S::U, kTail = S::kTail;
    static_assert(U * G <= kFp32Slack, "a batch stays in the slack");
    static_assert((kFp32Stage + 255) / 256 * 256 - kFp32Area <= kFp32Area / 2, "value loads end within the columns");
    static_assert((kFp32Stage + 511) / 512 * 512 >= kFp32Area, "the slack's columns are written (zeros)");
    static_assert(((kFp32Stage + 511) / 512 * 512 - kFp32Area) * 2 <= 256, "column loads end within the row starts");
    extern __shared__ __align__(16) unsigned char smem[];
    float *xs = (float *)smem;
    const uint32_t xs_bytes = ((uint32_t)cols * 4u + 15u) & ~15u;
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));  // uniform: steps and ranges stay scalar
    unsigned char *area = smem + xs_bytes + wave * S::kWave;  // this wavefront's
    float *sv = (float *)area;                                // staged values,
    colx_t *sc = (colx_t *)(area + kFp32Area * 4);            // columns
    uint32_t *sp = (uint32_t *)(area + kFp32Area * 6);        // and row starts of the step
    for (int c0 = 0; c0 < cols; c0 += 4 * ACC_WG) {  // four loads per thread issued together
        float t[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) t[u] = x[min(c0 + u * ACC_WG + (int)threadIdx.x, cols - 1)];
#pragma unroll
        for (int u = 0; u < 4; ++u)
            if (c0 + u * ACC_WG + (int)threadIdx.x < cols) xs[c0 + u * ACC_WG + threadIdx.x] = t[u];
    }
    const int lane = lane_id(), g = lane & (G - 1), grp = lane / G;
    __syncthreads();
    const int nsteps = (int)(((int64_t)rows + RS - 1) / RS);
    const int gw = blockIdx.x * ACC_WAVES + wave, nw = gridDim.x * ACC_WAVES;
    // the three best scores (ordered) and their rows of this lane so far
    uint32_t top = 0u, toprow = 0u, sec = 0u, secrow = 0u, thd = 0u, thdrow = 0u;

    typedef uint32_t v4 __attribute__((ext_vector_type(4)));
    constexpr int NV = (kFp32Stage + 255) / 256, NC = (kFp32Stage + 511) / 512;
    v4 lv[NV], lc[NC];
    auto load_starts = [&](int s, uint32_t (&p)[NP]) {  // row starts of step s (past the matrix: nnz)
        const int r0 = max(min(s, nsteps - 1), 0) * RS;
#pragma unroll
        for (int i = 0; i < NP; ++i) p[i] = ptr[(int)min((int64_t)r0 + i * 64 + lane, (int64_t)rows)];
    };
    auto first = [&](const uint32_t (&p)[NP]) { return (uint32_t)__builtin_amdgcn_readlane((int)p[0], 0); };
    auto last = [&](const uint32_t (&p)[NP]) { return (uint32_t)__builtin_amdgcn_readlane((int)p[RS / 64], RS % 64); };
    auto fits = [&](uint32_t b, uint32_t e) { return e - (b & ~7u) <= (uint32_t)kFp32Stage; };
    // the entries [b & ~7, e) into lv and lc (none of a range that exceeds the area)
    auto issue = [&](uint32_t b, uint32_t e) {
        const uint32_t sa = b & ~7u;
        const uint32_t cnt = fits(b, e) ? (e - sa + 7u) & ~7u : 0u;
        const __amdgpu_buffer_rsrc_t rv = __builtin_amdgcn_make_buffer_rsrc((void *)(val + sa), (short)0, (int)(cnt * 4u), 0x00020000);
        const __amdgpu_buffer_rsrc_t rc = __builtin_amdgcn_make_buffer_rsrc((void *)(idx + sa), (short)0, (int)(cnt * 2u), 0x00020000);
#pragma unroll
        for (int i = 0; i < NV; ++i) lv[i] = __builtin_amdgcn_raw_buffer_load_b128(rv, (i * 64 + lane) * 16, 0, 2 /* nt */);
#pragma unroll
        for (int i = 0; i < NC; ++i) lc[i] = __builtin_amdgcn_raw_buffer_load_b128(rc, (i * 64 + lane) * 16, 0, 2 /* nt */);
    };
    // The loads' last bytes (zeros: they cover more than the area) may fall on
    // what follows and is written after: the columns, then the row starts,
    // which are read before the area is staged again.
    auto stage = [&]() {
#pragma unroll
        for (int i = 0; i < NV; ++i) *(v4 *)(sv + (i * 64 + lane) * 4) = lv[i];
#pragma unroll
        for (int i = 0; i < NC; ++i)
            *(v4 *)(sc + (i * 64 + lane) * 8) = lc[i];
    };
    // Entries k .. of NT rows per lane, U per lane and row, added to p in order;
    // slots past a row's end read x[0], one address for all (power-law rows,
    // half of whose slots are: 212 -> 209 us) (base: the lane's first entry's
    // place in the area, n: entries of its row from there on).  All reads are issued before the first is used; the
    // empty asm keeps them out of the branches that the masked additions
    // would otherwise become.
    auto batch = [&](auto nt, auto nu, const uint32_t *base, const int *n, int k, float *p) {
        constexpr int NT = decltype(nt)::value, U = decltype(nu)::value;
        float a[NT][U], xv[NT][U];
        uint32_t c[NT][U];
#pragma unroll
        for (int t = 0; t < NT; ++t) {
            const uint32_t b = min(base[t] + (uint32_t)k, (uint32_t)kFp32Stage);
#pragma unroll
            for (int u = 0; u < U; ++u) {
                c[t][u] = sc[b + u * G];
                a[t][u] = sv[b + u * G];
            }
        }
#pragma unroll
        for (int t = 0; t < NT; ++t)
#pragma unroll
            for (int u = 0; u < U; ++u) xv[t][u] = x_at(xs, n[t] > k + u * G ? c[t][u] : (uint32_t)0);
#pragma unroll
        for (int t = 0; t < NT; ++t)
#pragma unroll
            for (int u = 0; u < U; ++u) asm volatile("" : "+v"(a[t][u]), "+v"(xv[t][u]));
#pragma unroll
        for (int t = 0; t < NT; ++t)
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const float f = __builtin_fmaf(a[t][u], xv[t][u], p[t]);
                p[t] = n[t] > k + u * G ? f : p[t];
            }
    };
    constexpr std::integral_constant<int, 1> one{};
    constexpr std::integral_constant<int, B> all{};
    constexpr std::integral_constant<int, U> un{};
    constexpr std::integral_constant<int, kTail> tail{};
    uint32_t pc[NP], pn[NP];  // row starts of this step and the next
    load_starts(gw, pc);
    load_starts(gw + nw, pn);
    issue(first(pc), last(pc));
    for (int s = gw; s < nsteps;) {  // (none for wavefronts past the last step)
        const uint32_t sa = first(pc) & ~7u;
        const bool staged = fits(first(pc), last(pc));
        stage();
#pragma unroll
        for (int i = 0; i < NP; ++i) sp[i * 64 + lane] = pc[i];
        const bool more = nw < nsteps - s;
        uint32_t pf[NP];
        load_starts(more ? s + nw + min(nw, nsteps - 1 - s - nw) : s, pf);  // the step after the next
        wave_sync();
        float p[B];
        uint32_t jb[B], je[B];
#pragma unroll
        for (int t = 0; t < B; ++t) {
            jb[t] = sp[t * RPI + grp];
            je[t] = sp[t * RPI + grp + 1];
            p[t] = 0.f;
        }
        if (!staged) {
            // a step of long rows: block by block, waiting for each block's
            // entries; a block that exceeds the area entry by entry, four per
            // lane together
#pragma unroll
            for (int t = 0; t < B; ++t) {
                const uint32_t b0 = (uint32_t)__builtin_amdgcn_readlane((int)jb[t], 0);
                const uint32_t b1 = (uint32_t)__builtin_amdgcn_readlane((int)je[t], 63);
                if (fits(b0, b1)) {
                    issue(b0, b1);
                    wave_sync();  // the block before has been read
                    stage();
                    wave_sync();
                    const uint32_t o = jb[t] - (b0 & ~7u) + g;
                    const int n = (int)(je[t] - jb[t]) - g;
                    for (int k = 0; __any(n > k); k += U * G) batch(one, un, &o, &n, k, &p[t]);
                    continue;
                }
                for (uint32_t j = jb[t] + g; j < je[t]; j += 4 * G) {
                    float v[4];
                    uint32_t c[4];
#pragma unroll
                    for (int u = 0; u < 4; ++u) {  // clamped into the row (j < je): the loads issue together
                        const uint32_t jj = min(j + u * G, je[t] - 1);
                        v[u] = __builtin_nontemporal_load(val + jj);
                        c[u] = __builtin_nontemporal_load(idx + jj);
                    }
#pragma unroll
                    for (int u = 0; u < 4; ++u)
                        if (j + u * G < je[t]) p[t] = __builtin_fmaf(v[u], x_at(xs, c[u]), p[t]);
                }
            }
        }
        // the next step's entries fly while this one is summed (none past the last step)
        issue(first(pn), more ? last(pn) : first(pn) & ~7u);
        if (staged) {
            uint32_t o[B];
            int n[B];
#pragma unroll
            for (int t = 0; t < B; ++t) {
                o[t] = jb[t] - sa + g;
                n[t] = (int)(je[t] - jb[t]) - g;
            }
            batch(all, un, o, n, 0, p);
            // longer rows, block by block
#pragma unroll
            for (int t = 0; t < B; ++t)
                for (int k = U * G; __any(n[t] > k); k += kTail * G) batch(one, tail, o + t, n + t, k, p + t);
        }
#pragma unroll
        for (int t = 0; t < B; ++t) p[t] = butterfly<G>(p[t]);
#pragma unroll
        for (int t0 = 0; t0 < B; t0 += G) {  // lane g of a group: block t0 + g
            float v = p[t0];
#pragma unroll
            for (int t = 1; t < G; ++t)
                if (t0 + t < B) v = g == t ? p[t0 + t] : v;
            const int64_t r = (int64_t)s * RS + (t0 + g) * RPI + grp;
            const bool mine = t0 + g < B && r < rows;
            if (mine) y[r] = v;
            // rows ascend, so an equal score keeps the lower row
            const uint32_t o = mine ? max(dordered_f32(v), 1u) : 0u;
            const bool b1 = o > top, b2 = o > sec, b3 = o > thd;
            thdrow = b2 ? secrow : b3 ? (uint32_t)r : thdrow;
            thd = max(thd, min(sec, o));
            secrow = b1 ? toprow : b2 ? (uint32_t)r : secrow;
            sec = max(sec, min(top, o));
            toprow = b1 ? (uint32_t)r : toprow;
            top = max(top, o);
        }
        if (!more) break;
        s += nw;
        wave_sync();  // the staged entries are read before the next step overwrites them
#pragma unroll
        for (int i = 0; i < NP; ++i) {
            pc[i] = pn[i];
            pn[i] = pf[i];
        }
    }
    if (gmax) {
        uint64_t best[3];
#pragma unroll
        for (int i = 0; i < 3; ++i) {
            const uint32_t m = wave_umax(top);
            const uint32_t lo = wave_umax(top == m ? 0xFFFFFFFFu - toprow : 0u);
            best[i] = m <= 1u ? (uint64_t)m : ((uint64_t)m << 32) | lo;
            if (top == m && 0xFFFFFFFFu - toprow == lo) {  // one lane: rows are distinct
                top = sec;
                toprow = secrow;
                sec = thd;
                secrow = thdrow;
            }
        }
        int w = gw, n = nw, t = lane;
        uint64_t key = lane == 0 ? best[0] : lane == 1 ? best[1] : best[2];
        if (wg_groups) {  // the workgroup's best of its wavefronts' keys, ranked by counting
            __shared__ uint64_t s_best[3 * ACC_WAVES];
            if (lane < 3) s_best[wave * 3 + lane] = key;
            __syncthreads();
            w = blockIdx.x;
            n = gridDim.x;
            t = 3;
            if (threadIdx.x < 3 * ACC_WAVES) {
                key = s_best[threadIdx.x];
                t = 0;
                for (int i = 0; i < 3 * ACC_WAVES; ++i)
                    t += s_best[i] > key || (s_best[i] == key && i < (int)threadIdx.x);  // equal: zeros and ones
            }
        }
        if (t < 3) gmax[t == 0 ? (size_t)w : group_pairs(n) + 2 * (size_t)w + t - 1] = key;
    }
}

// Top-K (K <= 960) of the scores y from the three largest keys of
// each group's rows (one workgroup): T, at most the K-th largest of
// the groups' best keys, is reached by K distinct rows, so every row of the
// Top-K has a key >= T and lies in one of the groups whose best reaches it (at
// most K + kSelSlack).  Their keys that reach T are listed in LDS; only a group
// whose third key exceeds T can hold more such rows and is read from y (the
// steps are dealt in turn, so neighbouring rows lie in different groups and
// hardly any is read).  Where the third key has T's score, all that is left of the
// group are rows of that score, and none after T's row: only its steps up to there
// are read (equal scores: every group's).  The listed keys are ranked.
//
// An order of rows that puts most of the best ones into the same groups
// leaves T too low.  Before many rows are read, and whenever more rows reach T
// than the list holds, T rises to the K-th best key listed and the listing
// starts again; after kSelRounds such rounds (scores that rise in the order of
// reading) a radix selection over the rows of those groups ends it.
//
// Bound: latency, and what one CU reads: at 2,000,000 rows and K = 100 it
// takes 9 us (at 100,000 rows 6), from wavefronts' instead of workgroups' keys
// 15 (10).  With two keys per wavefront, and some groups read in every call, it
// took 17 (11), reading all K groups' rows 53 (12 GB/s of scattered rows).
// Before it, two radix passes over all scores and a final one took 32 us, and
// above K = 256 the sorted lists of select_blocks and select_final 827 us
// (4,999,999 rows, K = 500; 16 us here).
// Equal scores (a query of zeros), us of the whole call, K = 100: 100,000 x 500
// 29, 2,000,000 x 900 154, 4,999,999 x 1024 191 -- any other query takes 17, 140
// and 179 --, before T rose and the reading ended at its row 38, 560 and 1205.
static constexpr int kSelList = 4096;  // keys listed in LDS
static constexpr int kSelSlack = 16;   // groups listed past the K-th, for one or two radix digits less
static constexpr int kSelRounds = 3;   // listings that overflowed
// Rows read before T rises: one round of loads of the workgroup, less than the
// rise takes.  Rows of a group whose three best keys are of one score and one
// step nearly all reach T and count more: they would have to be cut afterwards.
static constexpr uint32_t kSelRead = 16384, kSelDense = 16;

template <int V>
__global__ __launch_bounds__(1024) void fp32_select_groups(SelectGroupsArgs a) {
    extern __shared__ __align__(16) unsigned char smem[];
    __shared__ uint32_t hist[512];
    __shared__ uint64_t s_t[2];
    __shared__ int s_need[2], s_n, s_scans;
    __shared__ uint32_t s_rows;                      // rows to read, weighted
    __shared__ uint32_t s_scan[1024], s_last[1024];  // groups to read, up to this row
    __shared__ uint64_t s_below[1024];               // and the key below which their rows are not listed yet
    uint64_t *s_key = (uint64_t *)smem, *s_top = s_key + kSelList;  // kSelList, then 1024 keys
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
    const uint32_t nw = (uint32_t)a.nw, RS = (uint32_t)a.RS, rows = (uint32_t)a.rows;
    // all keys are loaded at once; the second and third ones arrive during the
    // radix selection of the best ones
    uint64_t k[V];
    ulonglong2 k23[V];
#pragma unroll
    for (int u = 0; u < V; ++u) k[u] = a.gmax[min((uint32_t)(tid + u * 1024), nw - 1u)];
#pragma unroll
    for (int u = 0; u < V; ++u) k23[u] = ((const ulonglong2 *)(a.gmax + group_pairs(a.nw)))[min((uint32_t)(tid + u * 1024), nw - 1u)];
#pragma unroll
    for (int u = 0; u < V; ++u)
        if ((uint32_t)(tid + u * 1024) >= nw) k[u] = 0ull;
    if (tid == 0) {
        s_n = 0;
        s_scans = 0;
        s_rows = 0u;
    }
    uint64_t T = wg_radix_kth<uint64_t>(
        [&](auto fn) {
#pragma unroll
            for (int u = 0; u < V; ++u) fn(k[u]);
        },
        a.K, hist, s_t, s_need, kSelSlack);
#pragma unroll
    for (int u = 0; u < V; ++u)  // not in the branches below, one wait each
        asm volatile("" : "+v"(k23[u].x), "+v"(k23[u].y));
    // fewer than K groups with rows, or keys of 1 among the best: every group is read
    const bool all = T <= 1ull;
    auto append = [&](uint64_t key) {
        const int j = atomicAdd(&s_n, 1);
        if (j < kSelList) s_key[j] = key;
    };
    const uint32_t L = (uint32_t)a.gsteps * RS;  // rows of a group
    // group w's keys that reach T (at most 3 * (K + kSelSlack) of all groups, which fit); a group to read
    auto list = [&](uint32_t w, uint64_t k1, uint64_t k2, uint64_t k3) {
        if (k1 < T) return;
        append(k1);
        if (k2 >= T) append(k2);
        if (k3 >= T) append(k3);
        if (k3 > T) {
            const int i = atomicAdd(&s_scans, 1);
            if (i < 1024) {  // K + kSelSlack of them at most: the keys are distinct
                s_scan[i] = w;
                s_below[i] = k3;
                // (T may be the lower end of a digit: its row then lies past the matrix)
                const uint32_t end = min((uint32_t)dkey_row(T), rows - 1u);
                const bool ties = (k3 >> 32) == (T >> 32);
                s_last[i] = ties ? end : rows - 1u;
                const uint32_t n = !ties ? L : (end / (nw * RS) + 1u) * RS * (k1 - k3 < RS ? kSelDense : 1u);
                atomicAdd(&s_rows, min(n, 1u << 20));  // (the sum of 1,024 of them fits)
            }
        }
    };
    // fn(key, i) for the rows of groups group(i), i = 0 .. nl-1, up to row
    // last(i) (0: no row).  A wavefront reads U rows per lane of C groups
    // together, and all wavefronts share a group's rows (20M x 1024: one group of
    // 15,600 rows read by one wavefront took 36 us, 5 now); the rows' places in a
    // group are the same for all groups.
    auto scan_by = [&](auto uu, auto cc, int nl, auto group, auto last, auto fn) {
        constexpr int U = decltype(uu)::value, C = decltype(cc)::value;
        const uint32_t nc = (uint32_t)(nl + C - 1) / C, items = nc * ((L + 64 * U - 1) / (64 * U));
        uint32_t off[U], off0 = 0u, cur = 0xFFFFFFFFu;
        for (uint32_t it = wave; it < items; it += 16) {
            const uint32_t jb = it / nc;
            const int c0 = (int)(it - jb * nc) * C;
            if (jb != cur) {
                cur = jb;
#pragma unroll
                for (int u = 0; u < U; ++u) {
                    const uint32_t j = (jb * U + u) * 64 + lane, st = j / RS;
                    off[u] = j < L ? st * nw * RS + (j - st * RS) : 0xFFFFFFFFu;
                }
                off0 = (uint32_t)__builtin_amdgcn_readfirstlane((int)off[0]);  // the first row's
            }
            uint32_t b[C], e[C];  // the groups' first rows, and one past the last to read
            bool any = false;
#pragma unroll
            for (int c = 0; c < C; ++c) {
                const int i = min(c0 + c, nl - 1);
                b[c] = group(i) * RS;
                e[c] = c0 + c < nl ? last(i) + 1u : 0u;
                any |= b[c] + off0 < e[c];
            }
            if (!any) continue;  // the same for the whole wavefront
            float v[C][U];
            uint32_t row[C][U];
#pragma unroll
            for (int c = 0; c < C; ++c)
#pragma unroll
                for (int u = 0; u < U; ++u) {
                    row[c][u] = off[u] != 0xFFFFFFFFu && b[c] + off[u] < e[c] ? b[c] + off[u] : 0xFFFFFFFFu;
                    v[c][u] = a.y[min(row[c][u], rows - 1u)];
                }
#pragma unroll
            for (int c = 0; c < C; ++c)
#pragma unroll
                for (int u = 0; u < U; ++u)
                    fn(row[c][u] < rows ? dkey_f32(v[c][u], (int32_t)row[c][u]) : 0ull, min(c0 + c, nl - 1));
        }
    };
    auto scan = [&](int nl, auto fn) {  // of the groups to read
        auto group = [&](int i) { return s_scan[i]; };
        auto last = [&](int i) { return s_last[i]; };
        if (L <= 64) scan_by(std::integral_constant<int, 1>(), std::integral_constant<int, 8>(), nl, group, last, fn);
        else scan_by(std::integral_constant<int, 8>(), std::integral_constant<int, 2>(), nl, group, last, fn);
    };
    if (!all) {
#pragma unroll
        for (int u = 0; u < V; ++u) list((uint32_t)(tid + u * 1024), k[u], k23[u].x, k23[u].y);
    }
    int nl = 0;  // keys listed before any row was read
    for (int over = -1; !all;) {  // -1: nothing read yet
        __syncthreads();
        nl = s_n;
        const int scans = min(s_scans, 1024);
        if (over >= 0 || s_rows <= kSelRead) {
            scan(scans, [&](uint64_t key, int i) {
                if (key >= T && key < s_below[i]) append(key);
            });
            __syncthreads();
            if (s_n <= kSelList || over == kSelRounds) break;
        }
        ++over;
        const int have = min(s_n, kSelList);
        T = wg_radix_kth<uint64_t>(
            [&](auto fn) {
                for (int i = tid; i < have; i += 1024) fn(s_key[i]);
            },
            a.K, hist, s_t, s_need);
        if (tid == 0) {
            s_n = 0;
            s_scans = 0;
            s_rows = 0u;
        }
        __syncthreads();
        for (uint32_t w = tid; w < nw; w += 1024) {
            const ulonglong2 k2 = ((const ulonglong2 *)(a.gmax + group_pairs(a.nw)))[w];
            list(w, a.gmax[w], k2.x, k2.y);
        }
    }
    if (all || s_n > kSelList) {
        // the K best of the listed keys and the rows of the groups to read (of every group)
        auto each = [&](auto fn) {
            for (int i = tid; i < nl; i += 1024) fn(s_key[i]);
            scan_by(
                std::integral_constant<int, 4>(), std::integral_constant<int, 1>(), all ? (int)nw : min(s_scans, 1024),
                [&](int i) { return all ? (uint32_t)i : s_scan[i]; }, [&](int i) { return all ? rows - 1u : s_last[i]; },
                [&](uint64_t key, int i) { fn(all || (key >= T && key < s_below[i]) ? key : 0ull); });
        };
        const uint64_t cut = wg_radix_kth<uint64_t>(each, a.K, hist, s_t, s_need);
        if (tid == 0) s_n = 0;
        __syncthreads();
        each([&](uint64_t key) {
            if (key != 0ull && key >= cut) {
                const int j = atomicAdd(&s_n, 1);
                if (j < 1024) s_top[j] = key;  // K of them at most: the keys are distinct
            }
        });
        __syncthreads();
        if (tid < min(s_n, 1024)) s_key[tid] = s_top[tid];
        __syncthreads();
    }
    int n = min(s_n, kSelList);
    if (n > 1024) {  // keep the best K
        const uint64_t cut = wg_radix_kth<uint64_t>(
            [&](auto fn) {
                for (int i = tid; i < n; i += 1024) fn(s_key[i]);
            },
            a.K, hist, s_t, s_need);
        if (tid == 0) s_n = 0;
        __syncthreads();
        for (int i = tid; i < n; i += 1024)
            if (s_key[i] >= cut) {
                const int j = atomicAdd(&s_n, 1);
                if (j < 1024) s_top[j] = s_key[i];
            }
        __syncthreads();
        n = min(s_n, 1024);
        if (tid < n) s_key[tid] = s_top[tid];
        __syncthreads();
    }
    int rank = 0;
    if (n <= 256) {  // ranks by counting: four lanes per key, two keys per read
        if (tid < 8) s_key[n + tid] = 0ull;
        __syncthreads();
        const int i = tid >> 2;
        const uint64_t mine = s_key[min(i, n)];
        for (int j = (tid & 3) * 2; j < n; j += 8) {
            const ulonglong2 o = *(const ulonglong2 *)(s_key + j);
            rank += (o.x > mine) + (o.y > mine);
        }
        rank += __builtin_amdgcn_update_dpp(0, rank, 0xB1, 0xF, 0xF, false);  // lane ^ 1
        rank += __builtin_amdgcn_update_dpp(0, rank, 0x4E, 0xF, 0xF, false);  // lane ^ 2
        if ((tid & 3) == 0 && i < n && rank < a.K) {
            acc_element e;
            e.value = dkey_score_f32(mine);
            e.index = dkey_row(mine);
            a.out[rank] = e;
        }
    } else {  // each wavefront sorts its keys; a key's rank: its places in the sorted lists
        uint64_t v[1] = {tid < n ? s_key[tid] : 0ull};
        reg_sort_desc<1>(v);
        s_top[tid] = v[0];
        __syncthreads();
        rank = lane;
        for (int w = 0; w * 64 < n; ++w) {
            if (w == wave) continue;
            int lo = 0, hi = 64;
            while (lo < hi) {
                const int mid = (lo + hi) >> 1;
                if (s_top[w * 64 + mid] > v[0]) lo = mid + 1;
                else hi = mid;
            }
            rank += lo;
        }
        const uint64_t mine = v[0];
        if (mine != 0ull && rank < a.K) {
            acc_element e;
            e.value = dkey_score_f32(mine);
            e.index = dkey_row(mine);
            a.out[rank] = e;
        }
    }
    for (int i = n + tid; i < a.K; i += 1024) {
        acc_element e;
        e.value = -__builtin_inff();
        e.index = -1;
        a.out[i] = e;
    }
}

select_groups_fn get_select_groups(int nw) { return nw <= 2048 ? fp32_select_groups<2> : fp32_select_groups<8>; }
size_t select_groups_lds() { return (size_t)(kSelList + 1024) * 8; }


template <int R>
__global__ __launch_bounds__(ACC_WG) void select_blocks(SelectArgs a) {
    extern __shared__ __align__(16) unsigned char smem[];
    __shared__ int s_n[ACC_WAVES];
    uint64_t *colbuf = (uint64_t *)smem;
    const int wave = threadIdx.x >> 6, lane = lane_id();
    const int64_t b0 = (int64_t)blockIdx.x * a.chunk;
    const int64_t b1 = min((int64_t)a.n, b0 + a.chunk);
    const int64_t q = (b1 - b0 + ACC_WAVES - 1) / ACC_WAVES;
    const int64_t w0 = b0 + wave * q, w1 = min(b1, w0 + q);
    WaveTopM<R> col;
    col.init(colbuf + wave * WaveTopM<R>::cap, a.K);
    // U scores per lane are loaded together (with the shared threshold) so one
    // memory latency covers 64*U keys
    constexpr int U = 8;
    for (int64_t i0 = w0; i0 < w1; i0 += 64 * U) {
        float v[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int64_t i = i0 + u * 64 + lane;
            v[u] = i < w1 ? __builtin_nontemporal_load(a.y + i) : 0.f;
        }
        const uint64_t g = atomic_load_u64(a.thr);
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int64_t i = i0 + u * 64 + lane;
            const bool valid = i < w1;
            const uint64_t key = valid ? dkey_f32(v[u], (int32_t)i) : 0ull;
            const uint64_t t = col.thr > g ? col.thr : g;
            col.push(valid && key > t, key);
        }
    }
    col.compact();
    if (lane == 0) s_n[wave] = col.n;
    __syncthreads();
    if (wave == 0) {
        wg_merge(col, colbuf, s_n, ACC_WAVES);
        publish_and_append(col, a.thr, a.cnt, a.cand);
    }
}

// Second launch (one workgroup): the final K of the appended candidates; the
// state is left zeroed for the next query.
template <int R>
__global__ __launch_bounds__(ACC_WG) void select_final(SelectArgs a) {
    extern __shared__ __align__(16) unsigned char smem[];
    __shared__ int s_n[ACC_WAVES];
    uint64_t *colbuf = (uint64_t *)smem;
    const int wave = threadIdx.x >> 6, lane = lane_id();
    const uint32_t n = *a.cnt;
    WaveTopM<R> col;
    col.init(colbuf + wave * WaveTopM<R>::cap, a.K);
    push_range(col, a.cand, n, (uint32_t)wave * 64, ACC_WG);
    col.compact();
    if (lane == 0) s_n[wave] = col.n;
    __syncthreads();
    if (wave == 0) {
        wg_merge(col, colbuf, s_n, ACC_WAVES);
        write_results(col, a.K, a.out);
        if (lane == 0) {
            *a.cnt = 0u;
            *a.thr = 0ull;
        }
    }
}

// Radix Top-K (K <= 256).  Pass: workgroup b keeps the K best keys of
// elements [b*V*ACC_WG, (b+1)*V*ACC_WG) of the input (FP32 scores keyed as
// (score, row i), or keys of an earlier pass) by radix selection and writes
// them to cand[b*K, (b+1)*K), zero-padded.  Passes repeat until the survivors
// fit one workgroup; then select_radix_final ranks them.
template <bool KEYS, int V>
__global__ __launch_bounds__(ACC_WG) void select_radix_pass(const void *in, int64_t n, int K, uint64_t *cand) {
    __shared__ uint32_t hist[512];
    __shared__ uint64_t s_t[2];
    __shared__ int s_need[2], s_n;
    const int tid = threadIdx.x, lane = tid & 63;
    const int64_t b0 = (int64_t)blockIdx.x * (V * ACC_WG);
    uint64_t k[V];
#pragma unroll
    for (int u = 0; u < V; ++u) {
        const int64_t i = b0 + tid + u * ACC_WG;
        if (KEYS) k[u] = i < n ? ((const uint64_t *)in)[i] : 0ull;
        else k[u] = i < n ? dkey_f32(__builtin_nontemporal_load((const float *)in + i), (int32_t)i) : 0ull;
    }
    if (tid == 0) s_n = 0;
    const uint64_t T = wg_radix_kth<uint64_t>(
        [&](auto fn) {
#pragma unroll
            for (int u = 0; u < V; ++u) fn(k[u]);
        },
        K, hist, s_t, s_need);
    uint64_t *dst = cand + (size_t)blockIdx.x * K;
#pragma unroll
    for (int u = 0; u < V; ++u) {
        const bool sel = k[u] != 0ull && k[u] >= T;
        const uint64_t m = __ballot(sel);
        if (m == 0) continue;
        int base = 0;
        if (lane == 0) base = atomicAdd(&s_n, __popcll(m));
        base = __shfl(base, 0);
        const int j = base + mbcnt64(m);
        if (sel && j < K) dst[j] = k[u];  // j < K for distinct keys
    }
    __syncthreads();
    for (int j = min(s_n, K) + tid; j < K; j += ACC_WG) dst[j] = 0ull;
}

template <int V>
__global__ __launch_bounds__(1024) void select_radix_final(const uint64_t *cand, int total, int K, acc_element *out) {
    __shared__ __align__(16) uint32_t lds[1036];
    topk_radix<V>(cand, total, K, out, lds);
}

// Zeroes the select state (a kernel rather than a memset, so the launch
// sequence can be captured in a graph).
__global__ void select_reset(uint64_t *thr, uint32_t *cnt) {
    if (threadIdx.x == 0) {
        *thr = 0ull;
        *cnt = 0u;
    }
}

// FP64 exact scores: 8 lanes per row, FP64 products and sums.

__global__ __launch_bounds__(ACC_WG) void spmv_fp64(const uint32_t *ptr, const colx_t *idx, const float *val,
                                                    const float *x, int rows, double *y) {
    const int lane8 = threadIdx.x & 7;
    for (int r = (blockIdx.x * ACC_WG + threadIdx.x) >> 3; r < ((rows + 31) & ~31); r += (gridDim.x * ACC_WG) >> 3) {
        double p = 0.0;
        if (r < rows)
            for (uint32_t j = ptr[r] + lane8; j < ptr[r + 1]; j += 8) p += (double)val[j] * (double)x_at(x, idx[j]);
        for (int s = 4; s >= 1; s >>= 1) p += __shfl_xor(p, s);
        if (r < rows && lane8 == 0) y[r] = p;
    }
}


template <int G>
static spmv_fn spmv_for(int B) {
    switch (B) {
        case 1: return fp32_spmv<G, 1>;
        case 2: return fp32_spmv<G, 2>;
        case 3: return fp32_spmv<G, 3>;
        case 4: return fp32_spmv<G, 4>;
        default: return nullptr;
    }
}

// LDS of an fp32_spmv<G, B> workgroup: x, then each wavefront's staging area.
size_t fp32_spmv_lds(int cols, int G, int B) {
    const size_t np = (size_t)(B * (64 / G)) / 64 + 1;
    return (((size_t)cols * 4 + 15) & ~(size_t)15) + ACC_WAVES * ((size_t)kFp32Area * 6 + np * 256);
}

spmv_fn get_fp32_spmv(int G, int B) {
    switch (G) {
        case 2: return spmv_for<2>(B);
        case 4: return spmv_for<4>(B);
        case 8: return spmv_for<8>(B);
        case 16: return spmv_for<16>(B);
        case 32: return spmv_for<32>(B);
        default: return nullptr;
    }
}
select_fn get_select_blocks(int R) {
    switch (R) {
        case 2: return select_blocks<2>;
        case 4: return select_blocks<4>;
        case 8: return select_blocks<8>;
        case 16: return select_blocks<16>;
        default: return nullptr;
    }
}
select_fn get_select_final(int R) {
    switch (R) {
        case 2: return select_final<2>;
        case 4: return select_final<4>;
        case 8: return select_final<8>;
        case 16: return select_final<16>;
        default: return nullptr;
    }
}
reset_fn get_select_reset() { return select_reset; }
radix_pass_fn get_select_radix_pass(bool keys, int V) {
    if (V == 8) return keys ? select_radix_pass<true, 8> : select_radix_pass<false, 8>;
    if (V == 32) return keys ? select_radix_pass<true, 32> : select_radix_pass<false, 32>;
    return nullptr;
}
radix_final_fn get_select_radix_final(int V) {
    switch (V) {
        case 1: return select_radix_final<1>;
        case 2: return select_radix_final<2>;
        case 4: return select_radix_final<4>;
        case 8: return select_radix_final<8>;
        case 16: return select_radix_final<16>;
        default: return nullptr;
    }
}
fp64_fn get_spmv_fp64() { return spmv_fp64; }
