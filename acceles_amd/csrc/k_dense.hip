// k_dense.hip -- the batched low-bit path around the matrix-core scores
// (pk_scores, k_pkmfma.hpp): query preparation, per-partition selection with
// FP32 rescoring, and the per-query Top-K.
//
// The INT32 stage-1 scores (quantify_util.py:173-196: exact integer dot of
// the quantized rows with the quantized query) of a block of queries come
// from v_mfma_i32_32x32x32_i8 over the slices' packets, expanded in LDS: at
// the densities of the embedding workloads (2-15% non-zeros) the matrix cores
// multiply a dense slice image faster than the vector ALUs decode (column,
// value) pairs once a pass serves tens of queries.  Integer arithmetic is
// exact, so the scores are the same integers as the packet kernels'.  Only
// the four best (score, row) keys of each (query, 64-row slice) leave the
// scores kernel; the per-partition selection derives its threshold from the
// slice maxima and rescans exactly the rare slice whose list may have
// dropped a qualifying row.
#include "kernels_common.hpp"

// 32-bit slice keys: (score + 2^25) << 6 | row_in_slice; a larger key is a
// higher score (equal scores: any fixed order will do, the lists are only a
// filter and every candidate is re-keyed by (score, row)).  0 = no row.
// |score| < 2^25 is checked on the host before the dense layout is used.
__device__ __forceinline__ int32_t tk_score(uint32_t k) { return (int32_t)(k >> 6) - (1 << 25); }
__device__ __forceinline__ int tk_rho(uint32_t k) { return (int)(k & 63u); }

// Exact INT32 score of this lane's row (row_in_slice = lane) of slice s for
// one query, decoded from the slice's packets with the entry width known
// only at run time: the lane's dwords stream through a 64-bit bit buffer,
// eight loads in flight, and every complete E-bit entry is taken off the
// bottom (the same number of entries on every lane, so no divergence).
// qx: the query's int8 values in LDS.
__device__ __forceinline__ int32_t slice_dot_packets(const DenseArgs &a, int64_t s, const int8_t *qx) {
    const uint2 sl = a.slices[s];
    const int cb = a.col_bits, vb = a.val_bits, E = cb + vb;
    const uint64_t emask = (1ull << E) - 1ull;
    const uint32_t cmask = (1u << cb) - 1u;
    const __amdgpu_buffer_rsrc_t rs = slice_rsrc(a.words, sl);
    const int lane = lane_id();
    uint64_t buf = 0ull;
    int nb = 0;
    int32_t acc = 0;
    for (int d0 = 0; d0 < (int)sl.y; d0 += 8) {
        uint32_t w[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) w[u] = __builtin_amdgcn_raw_buffer_load_b32(rs, ((d0 + u) * 64 + lane) * 4, 0, 0);
#pragma unroll
        for (int u = 0; u < 8; ++u) {
            buf |= (uint64_t)w[u] << nb;
            nb += 32;
            while (nb >= E) {
                const uint32_t e = (uint32_t)(buf & emask);
                buf >>= E;
                nb -= E;
                const int v = a.is_signed ? __builtin_amdgcn_sbfe(e, cb, vb) : (int)__builtin_amdgcn_ubfe(e, cb, vb);
                acc += v * (int)qx[e & cmask];
            }
        }
    }
    return acc;
}

// The same for one slot (slice * 64 + row in it) per lane, in any slices: 64
// scattered rows in about the time of one slice.
__device__ __forceinline__ int32_t slot_dot_packets(const DenseArgs &a, int64_t slot, const int8_t *qx) {
    const uint2 sl = a.slices[slot >> 6];
    const int cb = a.col_bits, vb = a.val_bits, E = cb + vb;
    const uint64_t emask = (1ull << E) - 1ull;
    const uint32_t cmask = (1u << cb) - 1u;
    const uint32_t *p = a.words + (size_t)sl.x * 64 + (uint32_t)(slot & 63);
    const int nd = (int)sl.y, end = (int)wave_umax(sl.y);
    uint32_t w[2][8];  // eight dwords are decoded while the next eight are loaded (words are padded past the last slice)
    auto load = [&](uint32_t (&v)[8], int d0) {
#pragma unroll
        for (int u = 0; u < 8; ++u) v[u] = p[(size_t)min(d0 + u, max(nd - 1, 0)) * 64];
    };
    uint64_t buf = 0ull;
    int nb = 0;
    int32_t acc = 0;
    load(w[0], 0);
    for (int d0 = 0; d0 < end; d0 += 8) {
        load(w[1], d0 + 8);
#pragma unroll
        for (int u = 0; u < 8; ++u) {
            buf |= (uint64_t)(d0 + u < nd ? w[0][u] : 0u) << nb;
            nb += 32;
            while (nb >= E) {
                const uint32_t e = (uint32_t)(buf & emask);
                buf >>= E;
                nb -= E;
                const int v = a.is_signed ? __builtin_amdgcn_sbfe(e, cb, vb) : (int)__builtin_amdgcn_ubfe(e, cb, vb);
                acc += v * (int)qx[e & cmask];
            }
        }
#pragma unroll
        for (int u = 0; u < 8; ++u) w[0][u] = w[1][u];
    }
    return acc;
}

// One workgroup per query slot of the padded batch: int8 quantization with
// the query's own scale (quantify_util.py:31-49, 259; the rule of the packet
// kernels), written in the B-operand layout, in plain order (rescans) and as
// the unsigned-8-bit offset correction.
__global__ __launch_bounds__(ACC_WG) void dense_prep(DenseArgs a) {
    __shared__ float red[ACC_WAVES];
    __shared__ int isum[ACC_WAVES];
    const int QB = 32 * a.NT;
    const int q = blockIdx.x, qb = q / QB, ql = q % QB, t = ql >> 5, j = ql & 31;
    const int wave = threadIdx.x >> 6, lane = lane_id();
    const bool valid = q < a.nq;
    const float *x = a.X + (size_t)(valid ? q : 0) * a.cols;
    // the first XR*ACC_WG columns are read once, with loads issued together
    // (clamped indices, masked after), and kept in registers for both passes
    constexpr int XR = 4;
    float xr[XR];
#pragma unroll
    for (int u = 0; u < XR; ++u) xr[u] = x[min((int)threadIdx.x + u * ACC_WG, a.cols - 1)];
    float m = 0.f;
#pragma unroll
    for (int u = 0; u < XR; ++u)
        if (valid && (int)threadIdx.x + u * ACC_WG < a.cols) m = fmaxf(m, fabsf(xr[u]));
    if (valid)
        for (int c = threadIdx.x + XR * ACC_WG; c < a.cols; c += ACC_WG) m = fmaxf(m, fabsf(x[c]));
    for (int o = 32; o > 0; o >>= 1) m = fmaxf(m, __shfl_xor(m, o));
    if (lane == 0) red[wave] = m;
    __syncthreads();
    float s = red[0];
    for (int w = 1; w < ACC_WAVES; ++w) s = fmaxf(s, red[w]);
    int sum = 0;
    for (int c = threadIdx.x, it = 0; c < a.cols_pad; c += ACC_WG, ++it) {
        int qv = 0;
        if (valid && c < a.cols && s > 0.f) {
            float xc = 0.f;
#pragma unroll
            for (int u = 0; u < XR; ++u)
                if (it == u) xc = xr[u];
            if (it >= XR) xc = x[c];
            const float qf = __fmul_rn(127.0f, __fdiv_rn(xc, s));
            qv = (int)__builtin_rintf(qf);
            qv = qv > 127 ? 127 : (qv < -128 ? -128 : qv);
        }
        const int kb = c >> 5, h = (c >> 4) & 1, bb = c & 15;
        a.qtab[(((size_t)qb * a.nkb + kb) * a.NT + t) * 1024 + (j + 32 * h) * 16 + bb] = (int8_t)qv;
        if (valid) a.qplain[(size_t)q * a.cols_pad + c] = (int8_t)qv;
        sum += qv;
    }
    for (int o = 32; o > 0; o >>= 1) sum += __shfl_xor(sum, o);
    if (lane == 0) isum[wave] = sum;
    __syncthreads();
    if (threadIdx.x == 0) {
        int tot = 0;
        for (int w = 0; w < ACC_WAVES; ++w) tot += isum[w];
        a.corr[q] = a.u8off ? 128 * tot : 0;
    }
}

// Copies the FP32 query (cols values) into this wavefront's LDS: eight
// clamped loads per lane are issued together per 512 columns (a loop of
// single loads would wait for each one before its LDS write).
__device__ __forceinline__ void stage_query(float *xs, const float *xq, int cols) {
    const int lane = lane_id();
    for (int c0 = 0; c0 < cols; c0 += 512) {
        float t[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) t[u] = xq[min(c0 + u * 64 + lane, cols - 1)];
#pragma unroll
        for (int u = 0; u < 8; ++u)
            if (c0 + u * 64 + lane < cols) xs[c0 + u * 64 + lane] = t[u];
    }
}

// FP32 rescoring of keys[0, nn) (ranking order, LDS) with their entry ranges
// (LDS) in the declared order, G lanes per row: a lane's U entries are at
// constant distances, so a row takes two addresses, and C rows per lane group
// are in flight (16 rows per round of loads: at G = 32 two rounds of eight
// rows took 5.7 us of the selection).  Loads past a row's end are
// masked; idx and val hold kRowPad entries past nnz.
template <int G>
__device__ __forceinline__ void rescore_rows(const DenseArgs &a, const uint64_t *keys, const uint2 *ranges, int nn,
                                             size_t base, const float *xs) {
    constexpr int groups = 64 / G, C = G >= 4 ? G / 4 : 1, U = G == 32 ? 3 : 6;
    static_assert(U * G <= kRowPad, "reads past the last row stay in the padding");
    const int lane = lane_id(), g = lane & (G - 1), grp = lane / G, M = a.M;
    for (int i0 = 0; i0 < M; i0 += groups * C) {
        uint32_t b[C], e[C];
        float out[C];
#pragma unroll
        for (int c = 0; c < C; ++c) {
            const int i = i0 + c * groups + grp;
            const uint2 rg = ranges[min(i, 63)];
            b[c] = i < nn ? rg.x + g : 0u;
            e[c] = i < nn ? rg.y : 0u;
            out[c] = 0.f;
        }
        for (;;) {
            bool any = false;
#pragma unroll
            for (int c = 0; c < C; ++c) any |= b[c] < e[c];
            if (!__any(any)) break;
            float v[C][U];
            uint32_t x[C][U];
#pragma unroll
            for (int c = 0; c < C; ++c) {
                const uint32_t at = min(b[c], e[c]);
                const float *pv = a.val + at;
                const colx_t *pc = a.idx + at;
#pragma unroll
                for (int u = 0; u < U; ++u) {
                    v[c][u] = pv[u * G];
                    x[c][u] = pc[u * G];
                }
            }
#pragma unroll
            for (int c = 0; c < C; ++c) {
#pragma unroll
                for (int u = 0; u < U; ++u) {
                    const float f = __builtin_fmaf(v[c][u], x_at(xs, x[c][u]), out[c]);
                    out[c] = b[c] + u * G < e[c] ? f : out[c];
                }
                b[c] += U * G;
            }
        }
#pragma unroll
        for (int c = 0; c < C; ++c) {
            const float sc = butterfly<G>(out[c]);
            const int i = i0 + c * groups + grp;
            if (g == 0 && i < M) a.resc[base + i] = i < nn ? dkey_f32(sc, dkey_row(keys[min(i, 63)])) : 0ull;
        }
    }
}

// Top-M of the n candidates k (lane i < n; ranked by counting) into keys, with
// their CSR entry ranges (in flight meanwhile), then the stage-1 outputs of
// this (query, partition) and the FP32 rescoring of those rows.
__device__ __forceinline__ void finish_rows(const DenseArgs &a, uint64_t k, int n, uint64_t *keys, uint2 *ranges, size_t base,
                                            const float *xs) {
    const int lane = lane_id(), M = a.M;
    uint2 rg = make_uint2(0u, 0u);
    if (a.out && n > 0) {  // out set: the CSR is present
        const int32_t r = lane < n ? dkey_row(k) : 0;
        rg = make_uint2(a.ptr[r], a.ptr[r + 1]);
    }
    int rank = 0;
    for (int j = 0; j < n; ++j) rank += readlane_u64(k, j) > k;  // distinct: one per row
    const int nn = min(n, M);
    if (lane < n && rank < nn) {
        keys[rank] = k;
        ranges[rank] = rg;
    }
    wave_sync();
    if (a.cand_rows_out)
        for (int i = lane; i < M; i += 64) {
            a.cand_rows_out[base + i] = i < nn ? dkey_row(keys[i]) : -1;
            a.cand_scores_out[base + i] = i < nn ? dkey_score_i32(keys[i]) : 0;
        }
    if (!a.out) return;
    switch (a.G) {
        case 2: return rescore_rows<2>(a, keys, ranges, nn, base, xs);
        case 4: return rescore_rows<4>(a, keys, ranges, nn, base, xs);
        case 8: return rescore_rows<8>(a, keys, ranges, nn, base, xs);
        case 16: return rescore_rows<16>(a, keys, ranges, nn, base, xs);
        default: return rescore_rows<32>(a, keys, ranges, nn, base, xs);
    }
}

// The query's int8 values into this wavefront's LDS (at most 1,024 columns, padded
// to whole dwords: one round trip); true if all are zero (padding of a batch).
__device__ __forceinline__ bool stage_qx(const DenseArgs &a, int q, int8_t *qx) {
    const uint32_t *src = (const uint32_t *)(a.qplain + (size_t)q * a.cols_pad);
    const int nd = a.cols_pad / 4, lane = lane_id();
    uint32_t v[4], any = 0u;
#pragma unroll
    for (int j = 0; j < 4; ++j) v[j] = src[min(j * 64 + lane, nd - 1)];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        if (j * 64 + lane < nd) ((uint32_t *)qx)[j * 64 + lane] = v[j];
        any |= v[j];
    }
    wave_sync();
    return !__any(any != 0u);
}

// The partition's n best rows for a query of zeros: every score is 0, so its first
// M; lane i < n: the i-th.
__device__ __forceinline__ uint64_t first_rows(const DenseArgs &a, int p, int &n) {
    const int32_t r0 = a.part_row[p];
    n = min(a.M, (int)(a.part_row[p + 1] - r0));
    return lane_id() < n ? dkey_i32(0, r0 + lane_id()) : 0ull;
}

// Candidates of one (query, partition) where more than 64 rows, or those of many
// slices besides the listed ones, may qualify (equal scores): k is left with the
// best of them (lane i < n: the i-th, or in no order as long as 64 hold them
// all), n returned.  nl: the number listed (keys of tk or above), in k up to 64;
// ts: the score that another row must reach; cand: 64 keys, then 384 dwords
// (LDS); qx, zero: stage_qx's.
// A row of a slice scores its fourth key's score at most, so with the M-th best
// key found so far only rows that this score would put above it are scored: of
// equal scores the lower rows.  64 of them at a time, of any slices.  G: blocks of
// 64 slices listed together; B: slices looked at together.
template <int G, int B>
__device__ __forceinline__ int select_rows(const DenseArgs &a, int q, int64_t s0, int nsl, int nvl, int nl, uint32_t tk,
                                           int32_t ts, uint64_t *cand, const int8_t *qx, bool zero, uint64_t &k) {
    const int lane = lane_id(), M = a.M;
    const uint4 *L = (const uint4 *)a.tk + (size_t)q * a.nslices + s0;
    const int32_t *perm = a.perm + s0 * 64;
    uint32_t *slots = (uint32_t *)(cand + 64);  // slots in the partition to score
    uint64_t *stage = cand + 64;                // before that, listed keys
    constexpr int kSlots = 384;
    // least: the M-th best so far; the pend keys above it wait in cand
    uint64_t least = 0ull, mask = 0ull;
    int pend = 0, nslots = 0, g = 0, b = -64;
    int c = 0, tot = 0, pos = 0, j0 = 0;  // listed keys of a group: a lane's, all, a lane's first place, the next to take
    uint32_t ke[4 * G];
    int32_t row[4 * G];
    uint4 l = make_uint4(0u, 0u, 0u, 0u);
    const bool every = ts == INT32_MIN;  // no bound: the lists hold fewer than M rows, every row is scored
    if (every) {
        g = nsl;
        b = 0;
    } else if (nl <= 64) {
        if (lane < nl) cand[lane] = k;
        pend = nl;
        g = nsl;
        if (nl >= M) {
            int rank = 0;
            for (int j = 0; j < nl; ++j) rank += readlane_u64(k, j) > k;
            least = readlane_u64(k, __builtin_ctzll(__ballot(lane < nl && rank == M - 1)));
        }
    }
    bool sorted = false;
    k = 0ull;
    for (;;) {
        uint64_t nk = 0ull;
        bool last = false, score = false;
        uint32_t slot = 0u;
        int ns = 64;
        if (every) {
            last = b >= nsl;
            score = !last;
            slot = (uint32_t)(b * 64 + lane);
            ++b;
        } else if (g < nsl) {  // the listed keys of 64 * G slices, 64 of them at a time
            if (j0 >= tot) {
#pragma unroll
                for (int u = 0; u < G; ++u) {
                    const int i = g + u * 64 + lane;
                    const uint4 v = L[min(i, nsl - 1)];
                    const int nv = i >= nsl ? 0 : i == nsl - 1 ? nvl : 64;
                    ke[4 * u] = tk_rho(v.x) < nv ? v.x : 0u;
                    ke[4 * u + 1] = tk_rho(v.y) < nv ? v.y : 0u;
                    ke[4 * u + 2] = tk_rho(v.z) < nv ? v.z : 0u;
                    ke[4 * u + 3] = tk_rho(v.w) < nv ? v.w : 0u;
                }
                // (the score of the M-th best: rows are looked up for what may pass it)
                const uint32_t lo = max(tk, least != 0ull ? (uint32_t)(dkey_score_i32(least) + (1 << 25)) << 6 : 0u);
                c = 0;
#pragma unroll
                for (int e = 0; e < 4 * G; ++e) {
                    const bool ok = ke[e] >= lo;
                    row[e] = perm[ok ? (size_t)(g + (e >> 2) * 64 + lane) * 64 + tk_rho(ke[e]) : 0];
                    ke[e] = ok ? ke[e] : 0u;
                }
#pragma unroll
                for (int e = 0; e < 4 * G; ++e) {
                    if (ke[e] != 0u && dkey_i32(tk_score(ke[e]), row[e]) <= least) ke[e] = 0u;
                    c += ke[e] != 0u ? 1 : 0;
                }
                const int incl = (int)wave_prefix_sum((uint32_t)c);
                pos = incl - c;
                tot = __builtin_amdgcn_readlane(incl, 63);
                j0 = 0;
            }
            if (tot > 0) {
                int at = pos - j0;
#pragma unroll
                for (int e = 0; e < 4 * G; ++e)
                    if (ke[e] != 0u) {
                        if (at >= 0 && at < 64) stage[at] = dkey_i32(tk_score(ke[e]), row[e]);
                        ++at;
                    }
                wave_sync();
                if (lane < tot - j0) nk = stage[lane];
                wave_sync();
            }
            j0 += 64;
            if (j0 >= tot) {
                g += 64 * G;
                tot = 0;
            }
        } else {
            // the rows that may qualify of the slices whose fourth key does
            while (nslots < 64 && (mask != 0ull || b + 64 < nsl)) {
                if (mask == 0ull) {
                    b += 64;
                    l = L[min(b + lane, nsl - 1)];
                    mask = __ballot(b + lane < nsl && l.w >= tk && dkey_i32(tk_score(l.w), 0) > least);
                    continue;
                }
                int sl[B];
                int32_t r[B];
                uint64_t rest = mask;
#pragma unroll
                for (int j = 0; j < B; ++j) {
                    sl[j] = rest ? __builtin_ctzll(rest) : -1;
                    rest &= rest - 1;
                }
#pragma unroll
                for (int j = 0; j < B; ++j) r[j] = perm[(size_t)(b + max(sl[j], 0)) * 64 + lane];
#pragma unroll
                for (int j = 0; j < B; ++j) {
                    if (sl[j] < 0 || nslots > kSlots - 64) continue;
                    mask &= mask - 1;
                    const uint32_t lw = (uint32_t)__builtin_amdgcn_readlane((int)l.w, sl[j]);
                    bool ok = r[j] >= 0 && dkey_i32(tk_score(lw), r[j]) > least;
                    if (!__any(ok)) continue;
                    ok = ok && lane != tk_rho(lw) && lane != tk_rho((uint32_t)__builtin_amdgcn_readlane((int)l.x, sl[j])) &&
                         lane != tk_rho((uint32_t)__builtin_amdgcn_readlane((int)l.y, sl[j])) &&
                         lane != tk_rho((uint32_t)__builtin_amdgcn_readlane((int)l.z, sl[j]));
                    const uint64_t m = __ballot(ok);
                    if (ok) slots[nslots + mbcnt64(m)] = (uint32_t)((b + sl[j]) * 64 + lane);
                    nslots += __popcll(m);
                }
            }
            wave_sync();
            ns = min(nslots, 64);
            last = ns == 0;
            score = !last;
            if (score) slot = slots[nslots - ns + min(lane, ns - 1)];  // the last 64 of them
            nslots -= ns;
        }
        if (score) {
            const int32_t r = perm[slot];
            const int32_t sc = zero ? 0 : every ? slice_dot_packets(a, s0 + b - 1, qx) : slot_dot_packets(a, s0 * 64 + slot, qx);
            if (lane < ns && r >= 0 && sc >= ts) nk = dkey_i32(sc, r);
        }
        uint64_t m = __ballot(nk > least);
        if (last && !sorted) {
            wave_sync();
            k = lane < pend ? cand[lane] : 0ull;
            return pend;
        }
        if (last || pend + __popcll(m) > 64) {
            wave_sync();
            uint64_t v[2] = {k, lane < pend ? cand[lane] : 0ull};
            reg_sort_desc<2>(v);
            k = v[0];
            sorted = true;
            if (last) return min(__popcll(__ballot(k != 0ull)), M);
            least = shfl_u64(k, M - 1);
            pend = 0;
            m = __ballot(nk > least);
            wave_sync();
        }
        if (nk > least) cand[pend + mbcnt64(m)] = nk;
        pend += __popcll(m);
    }
}

// One wavefront per (partition p = blockIdx.x, query q = blockIdx.y*4 + wave),
// for partitions of at most 64*U slices:
//  1. ts = a score that M distinct rows of the partition reach (INT32_MIN when
//     there are not M): at least M and, equal scores aside, at most M + kSlack
//     of the full slices' maxima reach it; up to 128 slices exactly M of their
//     whole lists (few maxima, or low ones, would make every list drop rows
//     that qualify: 400,000 x 500 in 64 partitions of 98 slices, M = 64, 64
//     queries: 160 -> 129 us of a call).  The partition's M-th best score is
//     >= ts, so no row below ts can be in its Top-M.
//  2. Every listed key of a real row scoring >= ts is a candidate; one prefix
//     sum places them, one gather finds their rows.  (Padding rows of the
//     partial slice score 0: its maximum is left out of step 1, their keys,
//     which may have displaced real rows from its list, of this step.)
//  3. A list whose fourth key still scores >= ts may have dropped a qualifying
//     row, none of a score above that key's.  The other rows of its slice are
//     scored exactly, unless M candidates score above that key (400,000 x 500,
//     100 queries: 64 -> 61 us of a call).
//  4. Top-M of the candidates by (score, row) (quantify_util.py:173-196 with
//     the lower-row tie rule), ranked by counting, then their FP32 rescoring
//     (out != null).  More than 64 candidates, or kRescans slices: select_rows.
//
// Bound: the memory requests of the rescoring (rows of a few cache lines each,
// anywhere in the CSR), about 0.4 ns per row.  400,000 x 500, 100 queries:
// 18.5 us; 22.9 when the rows of every listed key were looked up (784 per
// partition; now about 18), the threshold came from a 64-key sort through LDS
// and eight rows were rescored at a time.  1,000,000 x 500, 41 queries: 11.1
// us (26.2); 2,000,000 x 900, 256 queries: 65 (111).
template <int U>
__global__ __launch_bounds__(ACC_WG) void dense_select_regs(DenseArgs a) {
    constexpr int kSlack = 8, kRescans = 8;  // slices rescanned one after the other
    constexpr bool kExact = U <= 2;  // bound: the lists, not only the maxima
    extern __shared__ __align__(16) unsigned char smem[];
    const int wave = threadIdx.x >> 6, lane = lane_id();
    const int p = blockIdx.x, q = blockIdx.y * ACC_WAVES + wave;
    if (q >= a.nq) return;  // whole wavefront; no workgroup barrier below
    // per wavefront (2 KB): 64 candidates; 64 ranked keys and their entry
    // ranges, before that the slices to rescan or the slots to score
    uint64_t *cand = (uint64_t *)smem + wave * 256, *keys = cand + 64;
    uint2 *ranges = (uint2 *)(keys + 64);
    int8_t *qx = (int8_t *)(smem + ACC_WAVES * 256 * 8) + (size_t)wave * a.cols_pad;
    float *xs = (float *)(smem + ACC_WAVES * 256 * 8 + (size_t)ACC_WAVES * a.cols_pad) + (size_t)wave * a.cols_pad;
    const int64_t s0 = a.part_slice[p];
    const int nsl = (int)(a.part_slice[p + 1] - s0);
    const uint4 *L = (const uint4 *)a.tk + (size_t)q * a.nslices + s0;
    const int32_t *perm = a.perm + s0 * 64;
    const int M = a.M;
    const size_t base = ((size_t)q * a.split + p) * M;

    uint64_t k = 0ull;  // lane i < n: a candidate
    int n = 0;
    if (nsl > 0) {
        // unconditional loads (clamped into the partition, masked after) so
        // that the lists and the query for the rescoring arrive in one round
        // trip; a conditional load would be waited for on its own
        uint4 k4[U];
#pragma unroll
        for (int u = 0; u < U; ++u) k4[u] = L[min(u * 64 + lane, nsl - 1)];
        const int nvl = (int)a.nvalid[s0 + nsl - 1];  // every slice is full except a partition's last one
        if (a.out) stage_query(xs, a.X + (size_t)q * a.cols, a.cols);
        uint32_t t;
        {
            uint32_t v[kExact ? 4 * U : U];
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const int i = u * 64 + lane;
                if (i >= nsl) k4[u] = make_uint4(0u, 0u, 0u, 0u);
                const bool full = i < nsl - 1 || nvl == 64;
                v[u] = full ? k4[u].x : 0u;
                if constexpr (kExact) {
                    v[U + u] = full ? k4[u].y : 0u;
                    v[2 * U + u] = full ? k4[u].z : 0u;
                    v[3 * U + u] = full ? k4[u].w : 0u;
                }
            }
            t = wave_bound_u32(v, M, kExact ? 0 : kSlack);
        }
        // tk: the smallest list key of a score that reaches the bound (keys of
        // one score differ in the row); without a bound that of any row
        const uint32_t tk = max(t & ~63u, 64u);
        int c = 0, nr = 0;  // listed candidates of this lane, slices to rescan
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int nv = u * 64 + lane == nsl - 1 ? nvl : 64;
            const uint32_t ke[4] = {k4[u].x, k4[u].y, k4[u].z, k4[u].w};
#pragma unroll
            for (int e = 0; e < 4; ++e) c += tk_rho(ke[e]) < nv && ke[e] >= tk ? 1 : 0;
            nr += __popcll(__ballot(k4[u].w >= tk));
        }
        const int incl = (int)wave_prefix_sum((uint32_t)c);
        const int nl = __builtin_amdgcn_readlane(incl, 63);
        uint32_t listed = 0u;
        if (nl <= 64) {
            int pos = incl - c;
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const int nv = u * 64 + lane == nsl - 1 ? nvl : 64;
                const uint32_t ke[4] = {k4[u].x, k4[u].y, k4[u].z, k4[u].w};
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    if (tk_rho(ke[e]) < nv && ke[e] >= tk)
                        cand[pos++] = ((uint64_t)ke[e] << 32) | (uint32_t)((u * 64 + lane) * 64 + tk_rho(ke[e]));
            }
            wave_sync();
            n = nl;
            if (lane < n) {
                const uint64_t e = cand[lane];
                listed = (uint32_t)(e >> 32);
                k = dkey_i32(tk_score(listed), perm[(uint32_t)e]);
            }
        }
        const int32_t ts = t != 0u ? tk_score(t) : INT32_MIN;
        bool many = nl > 64 || nr > kRescans, zero = true;
        if (nr > 0 || many) zero = stage_qx(a, q, qx);
        if (nr > 0 && !many) {
            int i = 0;
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const uint64_t m = __ballot(k4[u].w >= tk);
                const int j = i + mbcnt64(m);
                if (k4[u].w >= tk && j < kRescans)
                    keys[j] = ((uint64_t)k4[u].w << 32) |
                              (uint32_t)((u * 64 + lane) << 18 | tk_rho(k4[u].z) << 12 | tk_rho(k4[u].y) << 6 | tk_rho(k4[u].x));
                i += __popcll(m);
            }
            wave_sync();
        }
        for (int j = 0; j < nr && !many; ++j) {  // slice by slice
            const uint64_t e = readlane_u64(keys[j], 0);
            const uint32_t lw = (uint32_t)(e >> 32), at = (uint32_t)e;
            // M listed candidates above its fourth key's score: no other row of it qualifies
            if (__popcll(__ballot(listed > (lw | 63u))) >= M) continue;
            const int s = (int)(at >> 18);
            const int32_t r = perm[(size_t)s * 64 + lane];
            const int32_t sc = slice_dot_packets(a, s0 + s, qx);
            const bool in_list = lane == (int)(at & 63u) || lane == (int)(at >> 6 & 63u) || lane == (int)(at >> 12 & 63u) ||
                                 lane == tk_rho(lw);
            const bool ok = r >= 0 && sc >= ts && !in_list;
            const uint64_t m = __ballot(ok);
            many = n + __popcll(m) > 64;
            if (ok && !many) cand[n + mbcnt64(m)] = dkey_i32(sc, r);
            n += many ? 0 : __popcll(m);
        }
        // (expected false: 20,000 x 500, 8 queries, 41.6 us of a call; 42.8 with
        // the block below laid out before the ordinary path)
        if (__builtin_expect(many, false)) {
            if (zero && a.part_row)
                k = first_rows(a, p, n);
            else
                n = select_rows<2, 8>(a, q, s0, nsl, nvl, nl, tk, ts, cand, qx, zero, k);
        } else if (nr > 0) {
            wave_sync();
            if (lane >= nl && lane < n) k = cand[lane];
        }
    }
    finish_rows(a, k, n, keys, ranges, base, xs);
}

// The same for partitions of any size: the threshold is the M-th best full-slice
// maximum (a sorted buffer of them), the lists are streamed twice (threshold,
// then candidates).  400,000 x 500 in one partition of 6,250 slices, 8 queries,
// M = 32: 158 -> 139 us of a call; queries of zeros 34,600 -> 44 (a collector
// was offered every row of each slice whose list was full of ties).
__global__ __launch_bounds__(ACC_WG) void dense_select(DenseArgs a) {
    extern __shared__ __align__(16) unsigned char smem[];
    const int wave = threadIdx.x >> 6, lane = lane_id();
    const int p = blockIdx.x, q = blockIdx.y * ACC_WAVES + wave;
    if (q >= a.nq) return;  // whole wavefront; no workgroup barrier below
    uint64_t *cand = (uint64_t *)smem + wave * 256, *keys = cand + 64;
    uint2 *ranges = (uint2 *)(keys + 64);
    int8_t *qx = (int8_t *)(smem + ACC_WAVES * 256 * 8) + (size_t)wave * a.cols_pad;
    float *xs = (float *)(smem + ACC_WAVES * 256 * 8 + (size_t)ACC_WAVES * a.cols_pad) + (size_t)wave * a.cols_pad;
    const int64_t s0 = a.part_slice[p];
    const int nsl = (int)(a.part_slice[p + 1] - s0);
    const uint4 *L = (const uint4 *)a.tk + (size_t)q * a.nslices + s0;
    const int M = a.M;

    uint64_t k = 0ull;
    int n = 0;
    const bool zero = nsl > 0 && stage_qx(a, q, qx);
    if (zero && a.part_row) {
        k = first_rows(a, p, n);
    } else if (nsl > 0) {
        const int nvl = (int)a.nvalid[s0 + nsl - 1];  // every slice is full except a partition's last one
        uint32_t t = 0u;
        {
            constexpr int U = 4;
            WaveTopM<2> ca;
            ca.init(cand, M);
            for (int b = 0; b < nsl; b += 64 * U) {
                uint32_t v[U];
#pragma unroll
                for (int u = 0; u < U; ++u) {
                    const int i = b + u * 64 + lane;
                    v[u] = i < nsl - 1 || (i == nsl - 1 && nvl == 64) ? L[i].x : 0u;
                }
                static_assert(U == 4, "four pushes below");
                ca.push(v[0] != 0u, ((uint64_t)v[0] << 32) | (uint32_t)(b + lane));
                ca.push(v[1] != 0u, ((uint64_t)v[1] << 32) | (uint32_t)(b + 64 + lane));
                ca.push(v[2] != 0u, ((uint64_t)v[2] << 32) | (uint32_t)(b + 128 + lane));
                ca.push(v[3] != 0u, ((uint64_t)v[3] << 32) | (uint32_t)(b + 192 + lane));
            }
            ca.compact();
            if (ca.n >= M) t = (uint32_t)(ca.buf[M - 1] >> 32);
        }
        wave_sync();
        n = select_rows<4, 16>(a, q, s0, nsl, nvl, 65, max(t & ~63u, 64u),
                               t != 0u ? tk_score(t) : INT32_MIN, cand, qx, zero, k);
    }
    if (a.out) stage_query(xs, a.X + (size_t)q * a.cols, a.cols);
    finish_rows(a, k, n, keys, ranges, ((size_t)q * a.split + p) * M, xs);
}

// One workgroup per query: each wavefront sorts a quarter of the query's
// split*M rescored keys in registers (64*R keys), the four sorted lists meet in
// LDS, and every key finds its rank in the union by binary search in the other
// three lists (keys are distinct: one per row).  Ranks below K[q] are written.
template <int R>
__global__ __launch_bounds__(ACC_WG) void batch_topk(DenseArgs a) {
    extern __shared__ __align__(16) unsigned char smem[];
    __shared__ int s_nz[ACC_WAVES];
    const int q = blockIdx.x;
    const int total = a.split * a.M;
    topk_by_rank<R>(a.resc + (size_t)q * total, total, a.K[q], a.out + (size_t)q * a.out_stride, (uint64_t *)smem, s_nz);
}

// The same for K <= 256 (total <= V * ACC_WG): radix selection of the K-th
// key, then ranks by counting.
template <int V>
__global__ __launch_bounds__(ACC_WG) void batch_topk_radix(DenseArgs a) {
    __shared__ __align__(16) uint32_t lds[1036];
    const int q = blockIdx.x;
    const int total = a.split * a.M;
    topk_radix<V>(a.resc + (size_t)q * total, total, a.K[q], a.out + (size_t)q * a.out_stride, lds);
}

dense_fn get_dense_prep() { return dense_prep; }
dense_fn get_dense_select(int64_t part_slices) {
    if (part_slices > 1024) return dense_select;
    if (part_slices <= 128) return part_slices <= 64 ? dense_select_regs<1> : dense_select_regs<2>;
    return part_slices <= 256 ? dense_select_regs<4> : part_slices <= 512 ? dense_select_regs<8> : dense_select_regs<16>;
}
dense_fn get_batch_topk_radix(int V) {
    switch (V) {
        case 1: return batch_topk_radix<1>;
        case 2: return batch_topk_radix<2>;
        case 4: return batch_topk_radix<4>;
        case 8: return batch_topk_radix<8>;
        case 16: return batch_topk_radix<16>;
        default: return nullptr;
    }
}
dense_fn get_batch_topk(int R) {
    switch (R) {
        case 1: return batch_topk<1>;
        case 2: return batch_topk<2>;
        case 4: return batch_topk<4>;
        case 8: return batch_topk<8>;
        case 16: return batch_topk<16>;
        default: return nullptr;
    }
}
