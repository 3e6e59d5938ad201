// Decode attention for one query position (src/models.rs:131-176, :228-256):
// RoPE on q and on the new key, the cache write, scores, softmax and the
// weighted sum of values in one kernel; a second, small kernel merges the
// splits when the timesteps are cut across several blocks.  gfx950, wave64.
//
// The softmax is computed in the running-maximum form: every group of lanes
// keeps (m, l, acc) = (largest score so far, sum of e^(s - m), sum of
// e^(s - m) v) and rescales when m grows; groups, waves and splits are merged
// by the same rule.  That is the function softmax(src/util.rs:49-65) followed
// by the weighted sum (:160-174); only the order of the roundings differs.
// Scores are kept in units of log2: t = (q.k) * log2(e) / sqrt(head_size), so
// that e^(s - m) is one v_exp_f32 of t - m (1 ulp; the scaling of the argument
// adds a relative error of about |s - m| * 6e-8 to a weight).
//
// Compiled with -ffp-contract=off; FMAs appear only where written as fmaf().
#include <stdlib.h>
#include <string.h>

#include <type_traits>

#include "l2_internal.h"
#include "lanes.h"

namespace {

template <int CTRL>
__device__ __forceinline__ float dpp_xchg(float v) {
    int r = __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), CTRL, 0xF, 0xF, true);
    return __builtin_bit_cast(float, r);
}

template <class T>
__device__ __forceinline__ T ld_at(const void *base, uint32_t byte_offset) {
    return *reinterpret_cast<const T *>(reinterpret_cast<const char *>(base) + byte_offset);
}

// Every kernel argument of a decode step, required in scalar registers at once: the arguments are cold in
// the scalar cache when a kernel starts, and loads placed where the values are first used follow each other
// (three round trips of some 0.3 us in front of the first cache row otherwise).
__device__ __forceinline__ void pin_args(const AttnDecode &A) {
    asm volatile("" ::"s"(A.q), "s"(A.k_new), "s"(A.v_new), "s"(A.kcache), "s"(A.vcache), "s"(A.cos_t), "s"(A.sin_t),
                 "s"(A.pos), "s"(A.dpos), "s"(A.out), "s"(A.scatter), "s"(A.part), "s"(A.n_heads), "s"(A.n_kv_heads),
                 "s"(A.ts), "s"(A.n_splits), "s"(A.max_splits));
}

constexpr float kNoScore = -1e30f; // "no timestep yet": finite, so that differences never give NaN

__device__ __forceinline__ float exp2_fast(float x) { return __builtin_amdgcn_exp2f(x); }

__device__ __forceinline__ float wave_sum(float v) {
    v += dpp_xchg<0xB1>(v);
    v += dpp_xchg<0x4E>(v);
    v += dpp_xchg<0x141>(v);
    v += dpp_xchg<0x140>(v);
    return lanes::rows_sum(v);
}

__device__ __forceinline__ float wave_max(float v) {
    v = fmaxf(v, dpp_xchg<0xB1>(v));
    v = fmaxf(v, dpp_xchg<0x4E>(v));
    v = fmaxf(v, dpp_xchg<0x141>(v));
    v = fmaxf(v, dpp_xchg<0x140>(v));
    return lanes::rows_max(v);
}

// Floats per row of the LDS tiles in which rows of lanes, waves and splits meet: the 128 partial outputs, then
// (m, l).  The outputs are stored four at a time (16-byte LDS stores), so a row starts on a 16-byte boundary.
constexpr int kCombRow = 128 + 4;
static_assert(kCombRow * sizeof(float) % 16 == 0, "rows of the merge tiles are written with 16-byte stores");

// Layout of a block: NWV waves x 4 rows of 16 lanes.  One row of lanes handles one timestep at a time, each lane 8
// of the 128 head dimensions of the key; a block covers 4 NWV timesteps per step and PD steps per tile, all of a
// tile's loads being issued before its arithmetic.
//
// A short context (n_splits == 1, QG = 1) is one block per query head and slice of 128 / DS output dimensions: every
// slice computes all scores, and reads and sums only its part of the values, so nothing has to be merged across blocks.  A
// single block per head leaves most CUs idle and is bound by what one CU can fetch (some 110 GB/s, 0.5 us per 100
// timesteps; asking for the next tile before this one's arithmetic changes nothing) and by the
// merge of its rows; eight slices read 9/16 of the bytes each and merge an eighth.  7B (32 kv heads), per token of 32
// layers, one block -> 8 slices: 1241 -> 1215 us at position 16, 1292 -> 1257 at 120; 13B (40 kv heads), 8 layers, 4
// slices: 566 -> 561 at 190, where 8 (320 blocks) took 570.  4 waves up to one tile of timesteps (position 16: 1215 us
// against 1227 with 8 waves), 8 beyond (190: 381 against 383 with 8 layers).  The query heads of one kv head (grouped-query
// attention, src/models.rs:142-145) are blocks of their own too: they read the same rows, out of one XCD's L2 where 8 divides the number
// of kv heads (blocks are dealt over the XCDs in turn, kv head by kv head; with 2 kv heads on four XCDs each), and a block has one chain of scores and sums instead of four or eight.  Whole layers, against a block for
// all heads of the kv head (in splits beyond 256), at 50, 100, 240 timesteps: 16 heads of 2 kv heads 22.8 / 24.1 / 27.4 ->
// 21.9 / 22.6 / 22.9 us, 32 of 4 28.3 / 29.8 / 31.8 -> 25.7 / 25.7 / 26.8, 64 of 8 at 500, 800 40.5 / 42.1 -> 37.7 / 38.7 (not taken for
// eight up to 256, see attn_launch_qg).
// Longer contexts are cut into splits of timesteps (DS = 1, 4 waves) that attn_combine_kernel merges; there all QG query heads
// of the kv head share each K and V load.
template <int QG, int NWV, int DS>
__global__ __launch_bounds__(NWV * 64) void attn_decode_kernel(const AttnDecode A) {
    constexpr int NT = NWV * 64, TSTEP = NWV * 4;
    constexpr int HS = 128, HALF = 64;
    constexpr int VD = HS / DS, VE = VD / 16; // head dimensions of the value that are this block's, and a lane's share
    static_assert(DS == 1 || QG == 1, "sliced: one head per block");
    constexpr int PD = QG >= 8 ? 2 : 4; // steps in flight and per pass through the phases (4 at 8 heads: over 256 registers, one block per CU, slower)
    __shared__ float qs[QG * HS];
    __shared__ float kvnew[2][HS];
    // With 4 or 8 query heads per kv head the four 16-lane rows of every wave hand their partial results
    // over through (dynamic) LDS: merging them with cross-row shuffles first takes 10 shuffles per head and
    // step, 160 at 8 heads, a fifth of the kernel at long contexts.
    constexpr bool kRowsInLds = QG * VE >= 32;
    constexpr int NR = kRowsInLds ? NWV * 4 : NWV; // partial results that meet in LDS
    __shared__ __align__(16) float comb_s[kRowsInLds ? 1 : NWV][QG][kCombRow];
    __shared__ float wts[QG][16], m_all[QG], den_all[QG];
    extern __shared__ __align__(16) float comb_d[]; // [NR][QG][kCombRow] when kRowsInLds
    float(*comb)[QG][kCombRow] = kRowsInLds ? reinterpret_cast<float(*)[QG][kCombRow]>(comb_d) : comb_s;
    pin_args(A);
    const int kvh = blockIdx.x, sp = DS > 1 ? 0 : blockIdx.y, slice = DS > 1 ? blockIdx.z : 0;
    // the block's first query head; sliced, one of the 1, 2, 4 or 8 of the kv head
    const int head = DS > 1 ? (kvh << (__builtin_ctz(A.n_heads) - __builtin_ctz(A.n_kv_heads))) + blockIdx.y : kvh * QG;
    const int pos = A.dpos ? A.dpos[0] : A.pos;
    const int t0 = sp * A.ts;
    if (t0 > pos) return;
    // The cached positions of this block; the new one, whose key and value are still to be written, is where the
    // sums of one row of lanes start from, in the block whose range ends with it.
    const int t1 = min(t0 + A.ts, pos);
    const bool owns_new = pos < t0 + A.ts;
    const int n = t1 - t0;
    const int kv_dim = A.n_kv_heads * HS;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int ds = lane & 15;            // dims [8 ds, 8 ds + 8)
    const int tl = wave * 4 + (lane >> 4); // this row's timestep within a step

    const float *__restrict__ kc = A.kcache;
    const float *__restrict__ vc = A.vcache;
    const uint32_t row_bytes = (uint32_t)kv_dim * 4u;
    const uint32_t lane_off = (uint32_t)(kvh * HS + ds * 8) * 4u;
    const int t_last = max(t1 - 1, t0);

    typedef float vec_v __attribute__((ext_vector_type(VE)));
    const uint32_t v_off = (uint32_t)(kvh * HS + slice * VD + ds * VE) * 4u;
    struct Step {
        float4 k0, k1;
        vec_v v;
    };
    // Unconditional loads: rows past the end re-read the last row.
    auto fetch = [&](int it, Step &d) {
        const int t = min(t0 + it * TSTEP + tl, t_last);
        const uint32_t row = __umul24(t, row_bytes), off = row + lane_off;
        d.k0 = ld_at<float4>(kc, off);
        d.k1 = ld_at<float4>(kc, off + 16);
        d.v = ld_at<vec_v>(vc, row + v_off);
    };
    // The small loads that the staging below needs go out first: loads return in
    // order, so behind the first tile's loads they would wait for all of them.
    // Every thread stages something (threads beyond the work repeat another
    // thread's element), so that no load can move into a branch further down.
    const float *ct = A.cos_t + (size_t)pos * HALF;
    const float *st = A.sin_t + (size_t)pos * HALF;
    constexpr int NQ = (QG * HALF + NT - 1) / NT;
    float qa[NQ], qb[NQ], qc[NQ], qsn[NQ];
#pragma unroll
    for (int r = 0; r < NQ; r++) {
        const int idx = (tid + r * NT) % (QG * HALF);
        const int j = idx >> 6, i = idx & 63;
        const float *qh = A.q + (size_t)(head + j) * HS;
        qa[r] = qh[i], qb[r] = qh[i + HALF];
        qc[r] = ct[i], qsn[r] = st[i];
    }
    const int hd = tid & 63;
    const float nk_a = A.k_new[(size_t)kvh * HS + hd], nk_b = A.k_new[(size_t)kvh * HS + hd + HALF];
    const float nv = A.v_new[(size_t)kvh * HS + (tid & 127)];
    const float nc = ct[hd], ns = st[hd];
    // Sliced, a thread has one output at most: where it goes is asked for here, not when it is there.
    int out_i = 0;
    if constexpr (DS > 1) {
        out_i = head * HS + slice * VD + tid % VD;
        const int32_t at = *((A.scatter ? A.scatter : reinterpret_cast<const int32_t *>(A.q)) + out_i);
        out_i = A.scatter ? at : out_i;
    }
    __builtin_amdgcn_sched_barrier(0);

    Step pipe[PD];
#pragma unroll
    for (int u = 0; u < PD; u++) fetch(u, pipe[u]); // first tile: in flight while q is staged
    __builtin_amdgcn_sched_barrier(0);

    // q with RoPE, src/models.rs:100-129 (the second half uses the rotated first half)
#pragma unroll
    for (int r = 0; r < NQ; r++) {
        const int idx = (tid + r * NT) % (QG * HALF);
        const int j = idx >> 6, i = idx & 63;
        const float first = qa[r] * qc[r] - qb[r] * qsn[r];
        qs[j * HS + i] = first;
        qs[j * HS + HALF + i] = qb[r] * qc[r] + first * qsn[r];
    }
    // the new key, rotated, and the new value; the block whose range ends at pos
    // also writes them to the cache (:236-249)
    {
        const float first = nk_a * nc - nk_b * ns;
        const float second = nk_b * nc + first * ns;
        kvnew[0][hd] = first;
        kvnew[0][hd + HALF] = second;
        kvnew[1][tid & 127] = nv;
        if (owns_new && (DS == 1 || blockIdx.y + slice == 0)) {
            if (tid < HALF) {
                float *kw = A.kcache + (size_t)pos * kv_dim + kvh * HS;
                kw[tid] = first;
                kw[tid + HALF] = second;
            } else if (tid >= 128 && tid < 256) {
                A.vcache[(size_t)pos * kv_dim + kvh * HS + (tid - 128)] = nv;
            }
        }
    }
    __syncthreads();

    // q in registers, except for 8 heads per kv head, where the registers go to the accumulators
    constexpr bool kQInLds = QG >= 8;
    float q[kQInLds ? 1 : QG][8];
    if constexpr (!kQInLds) {
#pragma unroll
        for (int j = 0; j < QG; j++) {
            const float4 a = *reinterpret_cast<const float4 *>(&qs[j * HS + ds * 8]);
            const float4 b = *reinterpret_cast<const float4 *>(&qs[j * HS + ds * 8 + 4]);
            q[j][0] = a.x, q[j][1] = a.y, q[j][2] = a.z, q[j][3] = a.w;
            q[j][4] = b.x, q[j][5] = b.y, q[j][6] = b.z, q[j][7] = b.w;
        }
    }
    // log2(e) / sqrt(head_size): src/models.rs:154 divides the score by sqrt(head_size)
    const float scale = 1.44269504088896340736f / sqrtf((float)HS);
    float m[QG], l[QG], acc[QG][VE];
#pragma unroll
    for (int j = 0; j < QG; j++) {
        float s = 0.f;
#pragma unroll
        for (int e = 0; e < 8; e++)
            s = fmaf(kQInLds ? qs[j * HS + ds * 8 + e] : q[kQInLds ? 0 : j][e], kvnew[0][ds * 8 + e], s);
        s += dpp_xchg<0xB1>(s);
        s += dpp_xchg<0x4E>(s);
        s += dpp_xchg<0x141>(s);
        s += dpp_xchg<0x140>(s);
        const bool mine = owns_new && tl == 0;
        m[j] = mine ? s * scale : kNoScore;
        l[j] = mine ? 1.f : 0.f;
#pragma unroll
        for (int e = 0; e < VE; e++) acc[j][e] = mine ? kvnew[1][slice * VD + ds * VE + e] : 0.f;
    }
    const int n_it = (n + TSTEP - 1) / TSTEP;
    const int n_tiles = (n_it + PD - 1) / PD;
    for (int tile = 0; tile < n_tiles; tile++) {
        if (tile > 0) { // all of the tile's loads, then its arithmetic
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int u = 0; u < PD; u++) fetch(tile * PD + u, pipe[u]);
            __builtin_amdgcn_sched_barrier(0);
        }
        // The tile's PD steps go through the phases together — all scores, one update of the running maxima,
        // all weights and weighted sums — so that the dependent chains of one step (dot product, four
        // cross-lane adds, exponential) interleave with those of the others: a block is often alone on its
        // CU, one wave per SIMD, and nothing else fills the gaps between dependent instructions.
        float k[PD][8], v[PD][VE];
        float sc[PD][QG];
        bool valid[PD];
        float mt[QG];
#pragma unroll
        for (int u = 0; u < PD; u++) {
            const int t = t0 + (tile * PD + u) * TSTEP + tl;
            valid[u] = t < t1;
            const Step &d = pipe[u];
            const float kk[8] = {d.k0.x, d.k0.y, d.k0.z, d.k0.w, d.k1.x, d.k1.y, d.k1.z, d.k1.w};
#pragma unroll
            for (int e = 0; e < 8; e++) k[u][e] = kk[e];
#pragma unroll
            for (int e = 0; e < VE; e++) v[u][e] = valid[u] ? d.v[e] : 0.f; // a row past the end may hold anything, NaN included
        }
#pragma unroll
        for (int j = 0; j < QG; j++) {
            float qj[8];
            if constexpr (kQInLds) { // one read of the head's q for all the steps of the tile
                const float4 a = *reinterpret_cast<const float4 *>(&qs[j * HS + ds * 8]);
                const float4 b = *reinterpret_cast<const float4 *>(&qs[j * HS + ds * 8 + 4]);
                qj[0] = a.x, qj[1] = a.y, qj[2] = a.z, qj[3] = a.w, qj[4] = b.x, qj[5] = b.y, qj[6] = b.z, qj[7] = b.w;
            } else {
#pragma unroll
                for (int e = 0; e < 8; e++) qj[e] = q[j][e];
            }
            float mj = kNoScore;
#pragma unroll
            for (int u = 0; u < PD; u++) {
                float s = 0.f;
#pragma unroll
                for (int e = 0; e < 8; e++) s = fmaf(qj[e], k[u][e], s);
                s += dpp_xchg<0xB1>(s);
                s += dpp_xchg<0x4E>(s);
                s += dpp_xchg<0x141>(s);
                s += dpp_xchg<0x140>(s);
                s = valid[u] ? s * scale : kNoScore;
                sc[u][j] = s;
                mj = fmaxf(mj, s);
            }
            mt[j] = mj;
        }
        bool grow = false;
#pragma unroll
        for (int j = 0; j < QG; j++) grow |= mt[j] > m[j];
        if (__any(grow)) { // some row's maximum moves: rescale what was summed so far
#pragma unroll
            for (int j = 0; j < QG; j++) {
                const float m_new = fmaxf(m[j], mt[j]);
                const float c = exp2_fast(m[j] - m_new);
                l[j] *= c;
#pragma unroll
                for (int e = 0; e < VE; e++) acc[j][e] *= c;
                m[j] = m_new;
            }
        }
#pragma unroll
        for (int u = 0; u < PD; u++) {
#pragma unroll
            for (int j = 0; j < QG; j++) {
                const float p = valid[u] ? exp2_fast(sc[u][j] - m[j]) : 0.f;
                l[j] += p;
#pragma unroll
                for (int e = 0; e < VE; e++) acc[j][e] = fmaf(p, v[u][e], acc[j][e]);
            }
        }
    }

    if constexpr (!kRowsInLds) {
        // merge the 4 rows of the wave (lanes 16 and 32 apart hold the same dims)
        auto merge = [&](auto both) __attribute__((always_inline)) {
#pragma unroll
            for (int j = 0; j < QG; j++) {
                const lanes::Both mb = both(m[j]), lb = both(l[j]);
                const float M = fmaxf(mb.lo, mb.hi);
                const float w1 = exp2_fast(mb.lo - M), w2 = exp2_fast(mb.hi - M);
                l[j] = lb.lo * w1 + lb.hi * w2;
#pragma unroll
                for (int e = 0; e < VE; e++) {
                    const lanes::Both a = both(acc[j][e]);
                    acc[j][e] = a.lo * w1 + a.hi * w2;
                }
                m[j] = M;
            }
        };
        merge([](float v) { return lanes::both16(v); });
        merge([](float v) { return lanes::both32(v); });
    }
    if (kRowsInLds || lane < 16) {
        const int slot = kRowsInLds ? wave * 4 + (lane >> 4) : wave;
#pragma unroll
        for (int j = 0; j < QG; j++) {
            vec_v a;
#pragma unroll
            for (int e = 0; e < VE; e++) a[e] = acc[j][e];
            *reinterpret_cast<vec_v *>(&comb[slot][j][ds * VE]) = a;
            if (ds == 0) {
                comb[slot][j][HS] = m[j];
                comb[slot][j][HS + 1] = l[j];
            }
        }
    }
    __syncthreads();
    if constexpr (kRowsInLds) {
        // weights of the 16 partial results of every head: one thread per (head, partial), a head per 16-lane row
        if (tid < QG * 16) {
            const int j = tid >> 4, e = tid & 15;
            const float me = comb[e][j][HS];
            float M = me;
            M = fmaxf(M, dpp_xchg<0xB1>(M));
            M = fmaxf(M, dpp_xchg<0x4E>(M));
            M = fmaxf(M, dpp_xchg<0x141>(M));
            M = fmaxf(M, dpp_xchg<0x140>(M));
            const float w = exp2_fast(me - M);
            float wl = w * comb[e][j][HS + 1];
            wl += dpp_xchg<0xB1>(wl);
            wl += dpp_xchg<0x4E>(wl);
            wl += dpp_xchg<0x141>(wl);
            wl += dpp_xchg<0x140>(wl);
            wts[j][e] = w;
            if (e == 0) {
                m_all[j] = M;
                den_all[j] = wl;
            }
        }
        __syncthreads();
    }
    // merge; one thread per (head, dim)
    for (int idx = tid; idx < QG * VD; idx += NT) {
        const int j = idx / VD, d = idx % VD, dv = slice * VD + d;
        float M, num = 0.f, den = 0.f;
        if constexpr (kRowsInLds) {
#pragma unroll
            for (int w = 0; w < NR; w++) num = fmaf(wts[j][w], comb[w][j][d], num);
            M = m_all[j];
            den = den_all[j];
        } else {
            M = comb[0][j][HS];
#pragma unroll
            for (int w = 1; w < NR; w++) M = fmaxf(M, comb[w][j][HS]);
#pragma unroll
            for (int w = 0; w < NR; w++) {
                const float e = exp2_fast(comb[w][j][HS] - M);
                num = fmaf(e, comb[w][j][d], num);
                den = fmaf(e, comb[w][j][HS + 1], den);
            }
        }
        const int h = head + j;
        if constexpr (DS > 1) {
            A.out[out_i] = num / den;
        } else {
            float *p = A.part + ((size_t)h * A.max_splits + sp) * (HS + 2);
            p[dv] = num;
            if (dv == 0) {
                p[HS] = M;
                p[HS + 1] = den;
            }
        }
    }
}

// The same decode step for grouped-query models (4 or 8 query heads per kv head) on the matrix cores, all in
// fp32 (v_mfma_f32_16x16x4_f32): the query heads of the kv head are columns of the tile, so a cache row
// costs the same whatever their number, and the dot products need no cross-lane sums.
//
// A wave takes tiles of 16 timesteps.  With lane = (i = lane % 16, kb = lane / 16):
//   S^T = K Q^T      A: lane (timestep i, kb) holds K[t][16 m + 4 kb + e], B: lane (head i, kb) holds
//                    Q[head][16 m + 4 kb + e]; MFMA step (m, e), m < 8, e < 4, contracts over those four d.
//                    The A operand is what a 16-byte load of the cache row gives: no LDS on the way.
//   C layout         lane (head j, kb), register r -> timestep 4 kb + r: the four lanes of a head hold its
//                    16 scores, the running maximum is shared by them, the running sum is per lane.
//   O^T += V^T P^T   MFMA step (r, c) contracts over timesteps 4 kb + r, the lane's own register r of P: the
//                    B operand needs no data movement.  A: lane (i, kb) holds V[4 kb + r][d] with
//                    d = 64 (c / 4) + 4 i + c % 4, again a 16-byte load as it stands.  The accumulator c,
//                    register r of lane (head j, kb) is O[head][64 (c / 4) + 16 kb + 4 r + c % 4].
// Two tiles per wave are in flight (all their loads issued before any arithmetic); the four waves of a block
// merge through LDS, the splits through attn_combine_kernel, as in the kernel above.
typedef float v4f __attribute__((ext_vector_type(4)));

template <int QG>
__global__ __launch_bounds__(256, 2) void attn_decode_mfma_kernel(const AttnDecode A) {
    constexpr int NWV = 4, NT = 256, TK = 16;
    constexpr int HS = 128, HALF = 64;
    static_assert(QG == 4 || QG == 8, "the query heads of a kv head fill part of the 16 columns of a tile");
    __shared__ float qs[QG * HS];
    __shared__ float kvnew[2][HS];
    __shared__ __align__(16) float comb[NWV][QG][kCombRow];
    pin_args(A);
    const int kvh = blockIdx.x, sp = blockIdx.y;
    const int pos = A.dpos ? A.dpos[0] : A.pos;
    const int t0 = sp * A.ts;
    if (t0 > pos) return;
    const int t1 = min(t0 + A.ts, pos + 1);
    const int n = t1 - t0;
    const int kv_dim = A.n_kv_heads * HS;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int li = lane & 15, kb = lane >> 4;

    const float *__restrict__ kc = A.kcache;
    const float *__restrict__ vc = A.vcache;
    const uint32_t row_bytes = (uint32_t)kv_dim * 4u;
    const int t_last = t1 - 1;
    const uint32_t k_lane = (uint32_t)(kvh * HS + 4 * kb) * 4u; // + 64 m bytes
    const uint32_t v_lane = (uint32_t)(kvh * HS + 4 * li) * 4u; // + 256 bytes for the second half of d

    struct Tile {
        float4 k[8]; // k[m]: K[t = li][16 m + 4 kb ..]
        float4 v[8]; // v[2 r + half]: V[t = 4 kb + r][64 half + 4 li ..]
    };
    // Unconditional loads: rows past the end re-read the last row (masked below).
    auto fetch = [&](int tile, Tile &d) {
        const int tb = t0 + tile * TK;
        const uint32_t ko = __umul24(min(tb + li, t_last), row_bytes) + k_lane;
#pragma unroll
        for (int m = 0; m < 8; m++) d.k[m] = ld_at<float4>(kc, ko + 64u * m);
#pragma unroll
        for (int r = 0; r < 4; r++) {
            const uint32_t vo = __umul24(min(tb + 4 * kb + r, t_last), row_bytes) + v_lane;
            d.v[2 * r] = ld_at<float4>(vc, vo);
            d.v[2 * r + 1] = ld_at<float4>(vc, vo + 256u);
        }
    };
    // The small loads that the staging needs go out first (loads return in order).
    const float *ct = A.cos_t + (size_t)pos * HALF;
    const float *st = A.sin_t + (size_t)pos * HALF;
    constexpr int NQ = (QG * HALF + NT - 1) / NT;
    float qa[NQ], qb[NQ], qc[NQ], qsn[NQ];
#pragma unroll
    for (int r = 0; r < NQ; r++) {
        const int idx = (tid + r * NT) % (QG * HALF);
        const int j = idx >> 6, i = idx & 63;
        const float *qh = A.q + (size_t)(kvh * QG + j) * HS;
        qa[r] = qh[i], qb[r] = qh[i + HALF];
        qc[r] = ct[i], qsn[r] = st[i];
    }
    // where this thread's outputs go when the step is not split: fetched now, used at the very end
    int sdst[QG * HS / NT];
    if constexpr (QG == 8) {
#pragma unroll
        for (int u = 0; u < QG * HS / NT; u++) {
            const int i = kvh * QG * HS + tid + u * NT;
            sdst[u] = (A.scatter && A.n_splits == 1) ? A.scatter[i] : i;
        }
    }
    const int hd = tid & 63;
    const float nk_a = A.k_new[(size_t)kvh * HS + hd], nk_b = A.k_new[(size_t)kvh * HS + hd + HALF];
    const float nv = A.v_new[(size_t)kvh * HS + (tid & 127)];
    const float nc = ct[hd], ns = st[hd];
    __builtin_amdgcn_sched_barrier(0);

    const int n_tiles = (n + TK - 1) / TK;
    Tile ta, tb2;
    fetch(wave, ta);
    fetch(wave + NWV, tb2);
    __builtin_amdgcn_sched_barrier(0);

    // q with RoPE, src/models.rs:100-129 (the second half uses the rotated first half)
#pragma unroll
    for (int r = 0; r < NQ; r++) {
        const int idx = (tid + r * NT) % (QG * HALF);
        const int j = idx >> 6, i = idx & 63;
        const float first = qa[r] * qc[r] - qb[r] * qsn[r];
        qs[j * HS + i] = first;
        qs[j * HS + HALF + i] = qb[r] * qc[r] + first * qsn[r];
    }
    // the new key, rotated, and the new value; the block whose range ends at pos also writes them to the
    // cache (:236-249)
    const bool owns_new = (t1 == pos + 1);
    {
        const float first = nk_a * nc - nk_b * ns;
        const float second = nk_b * nc + first * ns;
        kvnew[0][hd] = first;
        kvnew[0][hd + HALF] = second;
        kvnew[1][tid & 127] = nv;
        if (owns_new) {
            if (tid < HALF) {
                float *kw = A.kcache + (size_t)pos * kv_dim + kvh * HS;
                kw[tid] = first;
                kw[tid + HALF] = second;
            } else if (tid >= 128 && tid < 256) {
                A.vcache[(size_t)pos * kv_dim + kvh * HS + (tid - 128)] = nv;
            }
        }
    }
    __syncthreads();

    // B operands of the score MFMAs: this lane's head (columns beyond the QG heads are zero)
    float4 qf[8];
#pragma unroll
    for (int m = 0; m < 8; m++)
        qf[m] = li < QG ? *reinterpret_cast<const float4 *>(&qs[li * HS + 16 * m + 4 * kb]) : make_float4(0.f, 0.f, 0.f, 0.f);

    float m_run = kNoScore, l = 0.f;
    v4f acc[8];
#pragma unroll
    for (int c = 0; c < 8; c++) acc[c] = v4f{0.f, 0.f, 0.f, 0.f};
    // log2(e) / sqrt(head_size): src/models.rs:154 divides the score by sqrt(head_size)
    const float scale = 1.44269504088896340736f / sqrtf((float)HS);

    auto tile_math = [&](int tile, Tile &d) __attribute__((always_inline)) {
        const int tb = t0 + tile * TK;
        if (tb <= pos && pos < tb + TK) { // once per step: the row of the new position comes from LDS, not from the cache
            if (tb + li == pos) {
#pragma unroll
                for (int m = 0; m < 8; m++) d.k[m] = *reinterpret_cast<const float4 *>(&kvnew[0][16 * m + 4 * kb]);
            }
#pragma unroll
            for (int r = 0; r < 4; r++)
                if (tb + 4 * kb + r == pos) {
                    d.v[2 * r] = *reinterpret_cast<const float4 *>(&kvnew[1][4 * li]);
                    d.v[2 * r + 1] = *reinterpret_cast<const float4 *>(&kvnew[1][HALF + 4 * li]);
                }
        }
        // scores: two accumulators, so that consecutive MFMAs do not wait for each other
        v4f s0 = v4f{0.f, 0.f, 0.f, 0.f}, s1 = v4f{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int m = 0; m < 8; m += 2) {
            s0 = __builtin_amdgcn_mfma_f32_16x16x4f32(d.k[m].x, qf[m].x, s0, 0, 0, 0);
            s1 = __builtin_amdgcn_mfma_f32_16x16x4f32(d.k[m + 1].x, qf[m + 1].x, s1, 0, 0, 0);
            s0 = __builtin_amdgcn_mfma_f32_16x16x4f32(d.k[m].y, qf[m].y, s0, 0, 0, 0);
            s1 = __builtin_amdgcn_mfma_f32_16x16x4f32(d.k[m + 1].y, qf[m + 1].y, s1, 0, 0, 0);
            s0 = __builtin_amdgcn_mfma_f32_16x16x4f32(d.k[m].z, qf[m].z, s0, 0, 0, 0);
            s1 = __builtin_amdgcn_mfma_f32_16x16x4f32(d.k[m + 1].z, qf[m + 1].z, s1, 0, 0, 0);
            s0 = __builtin_amdgcn_mfma_f32_16x16x4f32(d.k[m].w, qf[m].w, s0, 0, 0, 0);
            s1 = __builtin_amdgcn_mfma_f32_16x16x4f32(d.k[m + 1].w, qf[m + 1].w, s1, 0, 0, 0);
        }
        float sc[4], p[4];
        float mx = kNoScore;
#pragma unroll
        for (int r = 0; r < 4; r++) {
            const bool valid = tb + 4 * kb + r <= t_last;
            sc[r] = valid ? (s0[r] + s1[r]) * scale : kNoScore;
            mx = fmaxf(mx, sc[r]);
        }
        if (__any(mx > m_run)) { // some head's maximum moves: agree on it among the head's four lanes, rescale
            mx = lanes::rows_max(mx);
            const float m_new = fmaxf(m_run, mx);
            const float c = exp2_fast(m_run - m_new);
            l *= c;
#pragma unroll
            for (int cc = 0; cc < 8; cc++) acc[cc] *= c;
            m_run = m_new;
        }
#pragma unroll
        for (int r = 0; r < 4; r++) {
            const bool valid = tb + 4 * kb + r <= t_last;
            p[r] = valid ? exp2_fast(sc[r] - m_run) : 0.f;
            l += p[r];
        }
        // weighted sums: eight independent accumulators
#pragma unroll
        for (int r = 0; r < 4; r++) {
            const float4 v0 = d.v[2 * r], v1 = d.v[2 * r + 1];
            acc[0] = __builtin_amdgcn_mfma_f32_16x16x4f32(v0.x, p[r], acc[0], 0, 0, 0);
            acc[1] = __builtin_amdgcn_mfma_f32_16x16x4f32(v0.y, p[r], acc[1], 0, 0, 0);
            acc[2] = __builtin_amdgcn_mfma_f32_16x16x4f32(v0.z, p[r], acc[2], 0, 0, 0);
            acc[3] = __builtin_amdgcn_mfma_f32_16x16x4f32(v0.w, p[r], acc[3], 0, 0, 0);
            acc[4] = __builtin_amdgcn_mfma_f32_16x16x4f32(v1.x, p[r], acc[4], 0, 0, 0);
            acc[5] = __builtin_amdgcn_mfma_f32_16x16x4f32(v1.y, p[r], acc[5], 0, 0, 0);
            acc[6] = __builtin_amdgcn_mfma_f32_16x16x4f32(v1.z, p[r], acc[6], 0, 0, 0);
            acc[7] = __builtin_amdgcn_mfma_f32_16x16x4f32(v1.w, p[r], acc[7], 0, 0, 0);
        }
    };
    // Tiles wave, wave + 4, ...: two buffers, each refilled right after its tile is done when the wave has a
    // further tile for it (a uniform branch; up to two tiles per wave, the usual case behind a long cache,
    // nothing is refilled).
    for (int tile = wave; tile < n_tiles; tile += 2 * NWV) {
        tile_math(tile, ta);
        if (tile + 2 * NWV < n_tiles) fetch(tile + 2 * NWV, ta);
        if (tile + NWV < n_tiles) {
            tile_math(tile + NWV, tb2);
            if (tile + 3 * NWV < n_tiles) fetch(tile + 3 * NWV, tb2);
        }
    }

    // this wave's (m, l, O) -> LDS.  The head's four lanes hold disjoint d: lane (j, kb), accumulators 0..3,
    // register r are d = 16 kb + 4 r + 0..3, accumulators 4..7 the same 64 further on.
    l = lanes::rows_sum(l);
    if (li < QG) {
#pragma unroll
        for (int r = 0; r < 4; r++) {
            *reinterpret_cast<float4 *>(&comb[wave][li][16 * kb + 4 * r]) = make_float4(acc[0][r], acc[1][r], acc[2][r], acc[3][r]);
            *reinterpret_cast<float4 *>(&comb[wave][li][HALF + 16 * kb + 4 * r]) =
                make_float4(acc[4][r], acc[5][r], acc[6][r], acc[7][r]);
        }
        if (kb == 0) {
            comb[wave][li][HS] = m_run;
            comb[wave][li][HS + 1] = l;
        }
    }
    __syncthreads();
    // merge the four waves; one thread per (head, dim), the passes unrolled so that their LDS reads overlap
    constexpr int NP = QG * HS / NT;
    float num[NP], den[NP], Mx[NP];
#pragma unroll
    for (int u = 0; u < NP; u++) {
        const int idx = tid + u * NT;
        const int j = idx >> 7, d = idx & 127;
        float M = comb[0][j][HS];
#pragma unroll
        for (int w = 1; w < NWV; w++) M = fmaxf(M, comb[w][j][HS]);
        float nu = 0.f, de = 0.f;
#pragma unroll
        for (int w = 0; w < NWV; w++) {
            const float e = exp2_fast(comb[w][j][HS] - M);
            nu = fmaf(e, comb[w][j][d], nu);
            de = fmaf(e, comb[w][j][HS + 1], de);
        }
        num[u] = nu, den[u] = de, Mx[u] = M;
    }
#pragma unroll
    for (int u = 0; u < NP; u++) {
        const int idx = tid + u * NT;
        const int j = idx >> 7, d = idx & 127;
        const int h = kvh * QG + j;
        if (QG == 8 && A.n_splits == 1) {
            A.out[sdst[u]] = num[u] / den[u];
            continue;
        }
        float *pp = A.part + ((size_t)h * A.max_splits + sp) * (HS + 2);
        pp[d] = num[u];
        if (d == 0) {
            pp[HS] = Mx[u];
            pp[HS + 1] = den[u];
        }
    }
}

// Attention for a chunk of B positions (prefill, src/models.rs:131-176 with B > 1).  Every cache row of
// the chunk is already written and q already rotated (rope_kv_kernel).  The same layout as the decode
// kernel, with the 8 "heads" of a block being 8 / QG query positions x the QG query heads of one kv head:
// the K and V rows a block streams are shared by 8 score/value streams instead of being re-read per query.
// Query j sees timesteps 0..pos[j] (causal within the chunk as well).
template <int QG>
__global__ __launch_bounds__(256) void attn_prefill_kernel(float *__restrict__ out, const float *__restrict__ q,
                                                            const float *__restrict__ kc, const float *__restrict__ vc,
                                                            const int32_t *__restrict__ pos,
                                                            const int32_t *__restrict__ scatter, int n_heads,
                                                            int n_kv_heads, int B) {
    constexpr int HS = 128, NQ = 8, QPB = NQ / QG, PD = 2, TSTEP = 16;
    __shared__ float qs[NQ * HS];
    __shared__ __align__(16) float comb[4][NQ][kCombRow];
    __shared__ int pj_s[NQ];
    const int kvh = blockIdx.x, qb = blockIdx.y;
    const int dim = n_heads * HS, kv_dim = n_kv_heads * HS;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int ds = lane & 15;
    const int tl = wave * 4 + (lane >> 4);
    // stream j: query qb * QPB + j / QG, head kvh * QG + j % QG
    if (tid < NQ) {
        const int qi = qb * QPB + tid / QG;
        pj_s[tid] = qi < B ? pos[qi] : -1;
    }
    for (int idx = tid; idx < NQ * HS; idx += 256) {
        const int j = idx >> 7, d = idx & 127;
        const int qi = min(qb * QPB + j / QG, B - 1);
        qs[idx] = q[(size_t)qi * dim + (kvh * QG + j % QG) * HS + d];
    }
    __syncthreads();
    int pj[NQ];
    int t_end = 0; // one past the last timestep any stream of the block sees
#pragma unroll
    for (int j = 0; j < NQ; j++) {
        pj[j] = pj_s[j];
        t_end = max(t_end, pj[j] + 1);
    }
    if (t_end == 0) return;
    const uint32_t row_bytes = (uint32_t)kv_dim * 4u;
    const uint32_t lane_off = (uint32_t)(kvh * HS + ds * 8) * 4u;
    struct Step {
        float4 k0, k1, v0, v1;
    };
    auto fetch = [&](int it, Step &d) {
        const int t = min(it * TSTEP + tl, t_end - 1);
        const uint32_t off = __umul24(t, row_bytes) + lane_off;
        d.k0 = ld_at<float4>(kc, off);
        d.k1 = ld_at<float4>(kc, off + 16);
        d.v0 = ld_at<float4>(vc, off);
        d.v1 = ld_at<float4>(vc, off + 16);
    };
    float m[NQ], l[NQ], acc[NQ][8];
#pragma unroll
    for (int j = 0; j < NQ; j++) {
        m[j] = kNoScore;
        l[j] = 0.f;
#pragma unroll
        for (int e = 0; e < 8; e++) acc[j][e] = 0.f;
    }
    const float scale = 1.44269504088896340736f / sqrtf((float)HS);
    const int n_it = (t_end + TSTEP - 1) / TSTEP;
    const int n_tiles = (n_it + PD - 1) / PD;
    Step pipe[PD];
    for (int tile = 0; tile < n_tiles; tile++) {
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int u = 0; u < PD; u++) fetch(tile * PD + u, pipe[u]);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int u = 0; u < PD; u++) {
            const int t = (tile * PD + u) * TSTEP + tl;
            const Step &d = pipe[u];
            const float k[8] = {d.k0.x, d.k0.y, d.k0.z, d.k0.w, d.k1.x, d.k1.y, d.k1.z, d.k1.w};
            float v[8] = {d.v0.x, d.v0.y, d.v0.z, d.v0.w, d.v1.x, d.v1.y, d.v1.z, d.v1.w};
#pragma unroll
            for (int e = 0; e < 8; e++) v[e] = t < t_end ? v[e] : 0.f; // rows past the end may hold anything
            float sc[NQ];
            bool grow = false;
#pragma unroll
            for (int j = 0; j < NQ; j++) {
                const float4 a = *reinterpret_cast<const float4 *>(&qs[j * HS + ds * 8]);
                const float4 b = *reinterpret_cast<const float4 *>(&qs[j * HS + ds * 8 + 4]);
                const float qj[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
                float s = 0.f;
#pragma unroll
                for (int e = 0; e < 8; e++) s = fmaf(qj[e], k[e], s);
                s += dpp_xchg<0xB1>(s);
                s += dpp_xchg<0x4E>(s);
                s += dpp_xchg<0x141>(s);
                s += dpp_xchg<0x140>(s);
                s = t <= pj[j] ? s * scale : kNoScore;
                sc[j] = s;
                grow |= s > m[j];
            }
            if (__any(grow)) {
#pragma unroll
                for (int j = 0; j < NQ; j++) {
                    const float m_new = fmaxf(m[j], sc[j]);
                    const float c = exp2_fast(m[j] - m_new);
                    l[j] *= c;
#pragma unroll
                    for (int e = 0; e < 8; e++) acc[j][e] *= c;
                    m[j] = m_new;
                }
            }
#pragma unroll
            for (int j = 0; j < NQ; j++) {
                const float p = t <= pj[j] ? exp2_fast(sc[j] - m[j]) : 0.f;
                l[j] += p;
#pragma unroll
                for (int e = 0; e < 8; e++) acc[j][e] = fmaf(p, v[e], acc[j][e]);
            }
        }
    }
#pragma unroll
    for (int step = 16; step <= 32; step *= 2) {
#pragma unroll
        for (int j = 0; j < NQ; j++) {
            const float mo = __shfl_xor(m[j], step);
            const float lo = __shfl_xor(l[j], step);
            const float M = fmaxf(m[j], mo);
            const float w1 = exp2_fast(m[j] - M), w2 = exp2_fast(mo - M);
            l[j] = l[j] * w1 + lo * w2;
#pragma unroll
            for (int e = 0; e < 8; e++) {
                const float ao = __shfl_xor(acc[j][e], step);
                acc[j][e] = acc[j][e] * w1 + ao * w2;
            }
            m[j] = M;
        }
    }
    if (lane < 16) {
#pragma unroll
        for (int j = 0; j < NQ; j++) {
            *reinterpret_cast<float4 *>(&comb[wave][j][ds * 8]) = make_float4(acc[j][0], acc[j][1], acc[j][2], acc[j][3]);
            *reinterpret_cast<float4 *>(&comb[wave][j][ds * 8 + 4]) =
                make_float4(acc[j][4], acc[j][5], acc[j][6], acc[j][7]);
            if (ds == 0) {
                comb[wave][j][HS] = m[j];
                comb[wave][j][HS + 1] = l[j];
            }
        }
    }
    __syncthreads();
    for (int idx = tid; idx < NQ * HS; idx += 256) {
        const int j = idx >> 7, d = idx & 127;
        const int qi = qb * QPB + j / QG;
        if (qi >= B) continue;
        float M = comb[0][j][HS];
#pragma unroll
        for (int w = 1; w < 4; w++) M = fmaxf(M, comb[w][j][HS]);
        float num = 0.f, den = 0.f;
#pragma unroll
        for (int w = 0; w < 4; w++) {
            const float e = exp2_fast(comb[w][j][HS] - M);
            num = fmaf(e, comb[w][j][d], num);
            den = fmaf(e, comb[w][j][HS + 1], den);
        }
        const int i = (kvh * QG + j % QG) * HS + d;
        const int dst = scatter ? scatter[i] : i;
        out[(size_t)qi * dim + dst] = num / den;
    }
}

// Column tile of block row y of n.  The work of a tile grows with its position, and blocks are dealt over the compute
// units in turn, `unit_rows` rows until every unit has one.  With up to two blocks per unit all are resident at once and
// the launch is as long as the unit with the most work, so the longest tiles get a unit to themselves and the others go
// in pairs of a long and a short one: 32 heads, 511 tokens 41.5 -> 37.1 us (against longest first, which pairs the longest
// with the middle).  Larger grids (unit_rows = 0) are worked off as units become free, longest first; dealing three per
// unit the same way gained nothing (299 tokens 27.0, 27.9).
__device__ __forceinline__ int column_tile(int y, int n, int unit_rows) {
    if (unit_rows == 0) return n - 1 - y;
    const int second = n - unit_rows; // rows of second blocks
    if (y >= unit_rows) return y - unit_rows;
    return n - 1 - (y < second ? unit_rows - second + y : y - second);
}

// Chunk attention on the matrix cores, all in fp32 (v_mfma_f32_16x16x4_f32): src/models.rs:131-176 with B > 1, causal per
// query over the cache rows 0..pos (every row of the chunk is already written, q is rotated), in the layout of attn_decode_mfma_kernel: a block owns 16 columns of one kv head, column
// n = (query ct*16/QG + n/QG, head kvh*QG + n%QG), its NWV waves take the tiles of 16 cache rows w, w + NWV, ...
// and merge through LDS at the end.  With lane = (i = lane % 16, kb = lane / 16):
//   S^T = K Q^T      A: lane (row i, kb) holds K[t][16 m + 4 kb + e] -- what a 16-byte load of the cache row leaves
//                    in the lane; B: lane (column i, kb) holds Q[column][16 m + 4 kb + e], eight 16-byte loads of
//                    the query's row, kept for the whole kernel.  Nothing passes through LDS on the way.
//   C layout         lane (column j, kb), register r -> row 4 kb + r: the lane masks the rows behind ITS column's
//                    position (causal per query); the four lanes of a column share its running maximum.
//   O^T += V^T P^T   contracts over the lane's own registers of P; A is a 16-byte load of the V row as it stands.
// 128 tokens of a 32-head model are 256 blocks, one per compute unit.  With CS = 2 a block owns two such sets of 16
// columns, so that a tile of K and V, which every block reads again from the L2, serves 32 columns instead of 16; their
// Q then lives in LDS.  One tile is in flight, its K and its V apart, in 158 (CS = 1) and 232 registers; two whole tiles in
// flight took 219 and did not fit with CS = 2.  Per launch, 64 heads on 8 kv heads: 777 tokens 129.8 us with two tiles in
// flight, 114.1 with one, 104.6 with CS = 2; 299 tokens 34.0, 30.1, 25.9; 32 heads: 511 tokens 37.7, 36.7, 32.3, 128
// tokens 8.6, 7.9.  (v_mfma_f32_16x16x4_f32 at its peak: 63 us for the first of these.)  (A form on 32 columns and tiles of 32 rows,
// v_mfma_f32_32x32x2_f32 with K and V turned through LDS, had half the blocks and took 16 to 31 us per chunk of a
// 512-token prompt where this one takes 11 to 19.)
//
// `keep`: which of a thread's outputs of each set are stored (comb and qs are LDS, qs of several sets only).
constexpr int kSetOutputs = 16 * 128 / 256; // of a thread, of a set of 16 columns in a block of 256
template <int QG, int NWV, int NP, int CS>
__device__ __forceinline__ void prefill_fp32(void *__restrict__ out, const float *__restrict__ q, const float *__restrict__ kc,
                                             const float *__restrict__ vc, const int32_t *__restrict__ pos,
                                             const int32_t *__restrict__ scatter, int n_heads, int n_kv_heads, int B, int max_pos,
                                             int unit_rows, float (*comb)[16][kCombRow], float4 (*qs)[8][64], const uint32_t (&keep)[CS]) {
    constexpr int NT = NWV * 64, TK = 16, HS = 128, HALF = 64, NC = 16, QPT = NC / QG;
    const int kvh = blockIdx.x, ct = column_tile(blockIdx.y, gridDim.y, unit_rows) * CS;
    const int dim = n_heads * HS, kv_dim = n_kv_heads * HS;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int li = lane & 15, kb = lane >> 4;
    const uint32_t row_bytes = (uint32_t)kv_dim * 4u;
    const uint32_t k_lane = (uint32_t)(kvh * HS + 4 * kb) * 4u; // + 64 m bytes
    const uint32_t v_lane = (uint32_t)(kvh * HS + 4 * li) * 4u; // + 256 bytes for the second half of d

    float4 k[8]; // k[m]: K[t = li][16 m + 4 kb ..]
    float4 v[8]; // v[2 r + half]: V[t = 4 kb + r][64 half + 4 li ..]
    // Unconditional loads: rows past the last one written re-read it (masked below).
    auto fetch_k = [&](int tile) __attribute__((always_inline)) {
        const uint32_t ko = __umul24(min(tile * TK + li, max_pos), row_bytes) + k_lane;
#pragma unroll
        for (int m = 0; m < 8; m++) k[m] = ld_at<float4>(kc, ko + 64u * m);
    };
    auto fetch_v = [&](int tile) __attribute__((always_inline)) {
#pragma unroll
        for (int r = 0; r < 4; r++) {
            const uint32_t vo = __umul24(min(tile * TK + 4 * kb + r, max_pos), row_bytes) + v_lane;
            v[2 * r] = ld_at<float4>(vc, vo);
            v[2 * r + 1] = ld_at<float4>(vc, vo + 256u);
        }
    };
    // this lane's column of each set: its query, its position, its B operands
    int my_pos[CS];
    float4 qf[8];
#pragma unroll
    for (int cs = 0; cs < CS; cs++) {
        const int my_qi = (ct + cs) * QPT + li / QG;
        my_pos[cs] = my_qi < B ? pos[my_qi] : -1;
        const float *qrow = q + (size_t)min(my_qi, B - 1) * dim + (size_t)(kvh * QG + li % QG) * HS + 4 * kb;
        if constexpr (CS == 1) {
#pragma unroll
            for (int m = 0; m < 8; m++) qf[m] = *reinterpret_cast<const float4 *>(qrow + 16 * m);
        } else {
#pragma unroll
            for (int m = 0; m < 8; m += NWV) qs[cs][m + wave][lane] = *reinterpret_cast<const float4 *>(qrow + 16 * (m + wave));
        }
    }
    fetch_k(wave);
    fetch_v(wave);
    // Where this thread's outputs go, asked for here and not when they are there: output u of a set is of head j % QG (see the
    // merge), which recurs.  7B, 16 / 64 / 128 tokens 6.6 / 7.8 / 9.7 -> 6.2 / 7.0 / 9.3 us, three planes and 64 tokens 10.1 -> 8.9.
    constexpr int PER = NT / HS, HEADS = QG > PER ? QG / PER : 1;
    int dst[HEADS];
#pragma unroll
    for (int u = 0; u < HEADS; u++) {
        const int i = (kvh * QG + (tid / HS + u * PER) % QG) * HS + tid % HS;
        dst[u] = scatter ? scatter[i] : i;
    }
    __builtin_amdgcn_sched_barrier(0);
    int t_end = my_pos[0] + 1; // the block's tiles end with the last row any of its columns sees
#pragma unroll
    for (int cs = 1; cs < CS; cs++) t_end = max(t_end, my_pos[cs] + 1);
#pragma unroll
    for (int off = 8; off > 0; off >>= 1) t_end = max(t_end, __shfl_xor(t_end, off));
    t_end = __builtin_amdgcn_readfirstlane(t_end);
    const int n_tiles = (t_end + TK - 1) / TK;

    struct Run {
        float m, l;
        v4f acc[8];
    };
    Run run[CS];
#pragma unroll
    for (int cs = 0; cs < CS; cs++) {
        run[cs].m = kNoScore, run[cs].l = 0.f;
#pragma unroll
        for (int c = 0; c < 8; c++) run[cs].acc[c] = v4f{0.f, 0.f, 0.f, 0.f};
    }
    const float scale = 1.44269504088896340736f / sqrtf((float)HS); // log2(e) / sqrt(head_size), src/models.rs:154
    if constexpr (CS > 1) __syncthreads();

    // A tile's scores, then its weighted sums.  K of the next tile is requested as soon as the scores have been taken and
    // V as soon as the sums have, so that each arrives behind the other's products.
    auto step = [&](int tile, auto last) __attribute__((always_inline)) {
        const int tb = tile * TK;
        float p[CS][4];
#pragma unroll
        for (int cs = 0; cs < CS; cs++) {
            if constexpr (CS > 1) {
#pragma unroll
                for (int m = 0; m < 8; m++) qf[m] = qs[cs][m][lane];
            }
            v4f s0 = v4f{0.f, 0.f, 0.f, 0.f}, s1 = v4f{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int m = 0; m < 8; m += 2) {
                s0 = __builtin_amdgcn_mfma_f32_16x16x4f32(k[m].x, qf[m].x, s0, 0, 0, 0);
                s1 = __builtin_amdgcn_mfma_f32_16x16x4f32(k[m + 1].x, qf[m + 1].x, s1, 0, 0, 0);
                s0 = __builtin_amdgcn_mfma_f32_16x16x4f32(k[m].y, qf[m].y, s0, 0, 0, 0);
                s1 = __builtin_amdgcn_mfma_f32_16x16x4f32(k[m + 1].y, qf[m + 1].y, s1, 0, 0, 0);
                s0 = __builtin_amdgcn_mfma_f32_16x16x4f32(k[m].z, qf[m].z, s0, 0, 0, 0);
                s1 = __builtin_amdgcn_mfma_f32_16x16x4f32(k[m + 1].z, qf[m + 1].z, s1, 0, 0, 0);
                s0 = __builtin_amdgcn_mfma_f32_16x16x4f32(k[m].w, qf[m].w, s0, 0, 0, 0);
                s1 = __builtin_amdgcn_mfma_f32_16x16x4f32(k[m + 1].w, qf[m + 1].w, s1, 0, 0, 0);
            }
            Run &R = run[cs];
            float sc[4];
            float mx = kNoScore;
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const bool valid = tb + 4 * kb + r <= my_pos[cs]; // causal: this column's query sees rows 0..pos
                sc[r] = valid ? (s0[r] + s1[r]) * scale : kNoScore;
                mx = fmaxf(mx, sc[r]);
            }
            if (__any(mx > R.m)) { // some column's maximum moves: agree on it among the column's four lanes, rescale
                mx = lanes::rows_max(mx);
                const float m_new = fmaxf(R.m, mx);
                const float c = exp2_fast(R.m - m_new);
                R.l *= c;
#pragma unroll
                for (int cc = 0; cc < 8; cc++) R.acc[cc] *= c;
                R.m = m_new;
            }
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const bool valid = tb + 4 * kb + r <= my_pos[cs];
                p[cs][r] = valid ? exp2_fast(sc[r] - R.m) : 0.f;
                R.l += p[cs][r];
            }
        }
        if (!last) fetch_k(tile + NWV);
#pragma unroll
        for (int cs = 0; cs < CS; cs++) {
            v4f(&acc)[8] = run[cs].acc;
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const float4 v0 = v[2 * r], v1 = v[2 * r + 1];
                const float pr = p[cs][r];
                acc[0] = __builtin_amdgcn_mfma_f32_16x16x4f32(v0.x, pr, acc[0], 0, 0, 0);
                acc[1] = __builtin_amdgcn_mfma_f32_16x16x4f32(v0.y, pr, acc[1], 0, 0, 0);
                acc[2] = __builtin_amdgcn_mfma_f32_16x16x4f32(v0.z, pr, acc[2], 0, 0, 0);
                acc[3] = __builtin_amdgcn_mfma_f32_16x16x4f32(v0.w, pr, acc[3], 0, 0, 0);
                acc[4] = __builtin_amdgcn_mfma_f32_16x16x4f32(v1.x, pr, acc[4], 0, 0, 0);
                acc[5] = __builtin_amdgcn_mfma_f32_16x16x4f32(v1.y, pr, acc[5], 0, 0, 0);
                acc[6] = __builtin_amdgcn_mfma_f32_16x16x4f32(v1.z, pr, acc[6], 0, 0, 0);
                acc[7] = __builtin_amdgcn_mfma_f32_16x16x4f32(v1.w, pr, acc[7], 0, 0, 0);
            }
        }
        if (!last) fetch_v(tile + NWV);
    };
    // The last tile apart: with a branch around the loads of the next tile these are copied, and waited for, where the branch
    // ends.  32 heads, 64 tokens behind 1500 rows 40.1 -> 36.3 us, 511 tokens 30.5 -> 29.6; 64 heads on 8 kv heads, 777 108.9 -> 105.5.
    int tile = wave;
    for (; tile + NWV < n_tiles; tile += NWV) step(tile, std::false_type());
    if (tile < n_tiles) step(tile, std::true_type());

#pragma unroll
    for (int cs = 0; cs < CS; cs++) {
        float l = run[cs].l;
        const v4f(&acc)[8] = run[cs].acc;
        if (cs > 0) __syncthreads(); // the set before has been read
        // this wave's (m, l, O) -> LDS: lane (column j, kb), accumulators 0..3, register r are d = 16 kb + 4 r + 0..3,
        // accumulators 4..7 the same 64 further on
        l = lanes::rows_sum(l);
#pragma unroll
        for (int r = 0; r < 4; r++) {
            *reinterpret_cast<float4 *>(&comb[wave][li][16 * kb + 4 * r]) = make_float4(acc[0][r], acc[1][r], acc[2][r], acc[3][r]);
            *reinterpret_cast<float4 *>(&comb[wave][li][HALF + 16 * kb + 4 * r]) =
                make_float4(acc[4][r], acc[5][r], acc[6][r], acc[7][r]);
        }
        if (kb == 0) {
            comb[wave][li][HS] = run[cs].m;
            comb[wave][li][HS + 1] = l;
        }
        __syncthreads();
        // merge the waves; the outputs go to their places in the consumer's order
        constexpr int NOUT = NC * HS / NT; // outputs per thread
#pragma unroll
        for (int u = 0; u < NOUT; u++) {
            const int idx = tid + u * NT;
            const int j = idx >> 7, d = idx & 127;
            const int qi = (ct + cs) * QPT + j / QG;
            float M = comb[0][j][HS];
#pragma unroll
            for (int w = 1; w < NWV; w++) M = fmaxf(M, comb[w][j][HS]);
            float nu = 0.f, de = 0.f;
#pragma unroll
            for (int w = 0; w < NWV; w++) {
                const float e = exp2_fast(comb[w][j][HS] - M);
                nu = fmaf(e, comb[w][j][d], nu);
                de = fmaf(e, comb[w][j][HS + 1], de);
            }
            if (qi < B && (keep[cs] >> u & 1)) {
                const int to = dst[u % HEADS];
                const float v = nu / de;
                if constexpr (NP == 1) {
                    reinterpret_cast<_Float16 *>(out)[(size_t)qi * dim + h16_slot(to)] = (_Float16)v;
                } else { // three bf16 numbers that add up to v exactly
                    uint16_t *o = reinterpret_cast<uint16_t *>(out) + (size_t)qi * NP * dim + b16_slot(to);
                    float left = v;
#pragma unroll
                    for (int p = 0; p < NP; p++) {
                        const uint32_t bits = __builtin_bit_cast(uint32_t, left) & 0xFFFF0000u;
                        o[(size_t)p * dim] = (uint16_t)(bits >> 16);
                        left -= __builtin_bit_cast(float, bits);
                    }
                }
            }
        }
    }
}

template <int QG, int CS>
__global__ __launch_bounds__(256, 2)
void attn_prefill_mfma16_kernel(void *__restrict__ out, const float *__restrict__ q, const float *__restrict__ kc,
                                const float *__restrict__ vc, const int32_t *__restrict__ pos,
                                const int32_t *__restrict__ scatter, int n_heads, int n_kv_heads, int B, int max_pos,
                                int unit_rows) {
    __shared__ __align__(16) float comb[4][16][kCombRow];
    __shared__ float4 qs[CS > 1 ? CS : 1][CS > 1 ? 8 : 1][64]; // several sets: their B operands
    constexpr uint32_t all = (1u << kSetOutputs) - 1;
    uint32_t keep[CS];
#pragma unroll
    for (int cs = 0; cs < CS; cs++) keep[cs] = all;
    prefill_fp32<QG, 4, 3, CS>(out, q, kc, vc, pos, scatter, n_heads, n_kv_heads, B, max_pos, unit_rows, comb,
                               reinterpret_cast<float4(*)[8][64]>(qs), keep);
}

typedef __bf16 b8 __attribute__((ext_vector_type(8)));
typedef __bf16 b2 __attribute__((ext_vector_type(2)));
typedef float v2f __attribute__((ext_vector_type(2)));

// Two fp32 numbers as three pairs of bf16 numbers each, whose sum they are: each rounded to nearest (one instruction for the pair),
// so that what it leaves has either sign.  What is left is one v_dot2_f32_bf16 of the pair with (-1, 0) or (0, -1).
struct Cut {
    uint32_t p[3];
    __device__ __forceinline__ Cut(float x, float y, uint32_t minus_lo, uint32_t minus_hi) {
#pragma unroll
        for (int k = 0; k < 3; k++) {
            p[k] = __builtin_bit_cast(uint32_t, __builtin_convertvector(v2f{x, y}, b2));
            if (k == 2) break;
            x = __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(b2, p[k]), __builtin_bit_cast(b2, minus_lo), x, false);
            y = __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(b2, p[k]), __builtin_bit_cast(b2, minus_hi), y, false);
        }
    }
};
struct Plane {
    uint32_t u[4];
    __device__ __forceinline__ b8 b() const { return __builtin_bit_cast(b8, *this); }
};

// The same for the fp16 mode (L2_PREFILL_MFMA), on v_mfma_f32_16x16x32_bf16 with every fp32 number as three bf16 numbers
// (sixteen times the rate of v_mfma_f32_16x16x4_f32): six products, down to the first by the third.  The second number is 2^-8 of
// the first at most and the third 2^-17, so the three products left out are 2^-24 of the whole at most, as an fp32 rounding is; of either
// sign, 2^-27.5 rms (2^-25.2).  (Cut off instead of rounded they are 2^-21.2 and all of one sign, 2^-24.7 on average.)  Relative rms
// error against fp64, 33 to 777 queries over 33 to 2040 rows, of that of the fp32 form: normal inputs 0.46 to 0.68, values of one sign
// 0.44 to 0.84, scores four times as sharp 0.52 to 0.70, nearly equal weights 0.35 to 0.93.  A number below 2^-102
// is held to 2^-126 at worst.  Blocks, columns and tiles are the fp32 form's, and a column's
// result depends on neither the other columns nor the number of sets: a pass gives the bits of the same tokens in several.
//   - Scores contract over 32 dimensions: a lane holds 16 m + 4 kb .. + 3 of two m, of K as of Q.
//   - The sums contract over the 16 rows of a tile, so one instruction takes two products: half its contraction is one plane of
//     V times one of the weights, half another.
//   - K, V and the weights are split by the wave that uses them, 7 vector instructions a pair of numbers (4 of them the dot
//     products of Cut; with masks and subtractions 11), Q once per block.
// What bounds it is the issue of vector instructions, most of them the splitting (half of a SIMD's cycles; the matrix unit's 28 %).
// Against the fp32 form, per launch: 32 heads, 16, 64, 128, 299, 511 tokens 5.5, 6.2, 8.0, 19.3, 29.6 -> 4.7, 5.2, 6.8, 15.6, 24.2 us;
// 128 tokens behind 384 17.2 -> 15.0, 64 behind 1500 36.3 -> 33.8; 64 heads on 8 kv heads, 128, 777 tokens 10.7, 105.5 -> 9.4, 79.8.
// Tiles of 32 rows, a product per instruction: 16, 128 and 777 of these tokens 6.0, 7.5 and 86.0; rescaling whenever a maximum
// moves: 511 and 777 tokens 26.0 and 83.7.
template <int QG, int CS>
__global__ __launch_bounds__(256, 2)
void attn_prefill_cut_kernel(void *__restrict__ out, const float *__restrict__ q, const float *__restrict__ kc,
                             const float *__restrict__ vc, const int32_t *__restrict__ pos,
                             const int32_t *__restrict__ scatter, int n_heads, int n_kv_heads, int B, int max_pos,
                             int unit_rows) {
    constexpr int NWV = 4, TK = 16, HS = 128, NC = 16, QPT = NC / QG;
    __shared__ __align__(16) float comb[NWV][NC][kCombRow];
    __shared__ float2 ml[CS][NWV][NC];
    __shared__ uint4 qs[CS][4][3][64]; // the columns' B operands: [set][32 dimensions][plane][lane]
    __shared__ int again;
    const int kvh = blockIdx.x, ct = column_tile(blockIdx.y, gridDim.y, unit_rows) * CS;
    const int dim = n_heads * HS, kv_dim = n_kv_heads * HS;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int li = lane & 15, kb = lane >> 4;
    const uint32_t row_bytes = (uint32_t)kv_dim * 4u;
    const uint32_t k_lane = (uint32_t)(kvh * HS + 4 * kb) * 4u; // + 64 m bytes
    const uint32_t v_lane = (uint32_t)(kvh * HS + 4 * li) * 4u; // + 256 bytes for the second half of d
    uint32_t minus_lo = 0x0000BF80u, minus_hi = 0xBF800000u; // (-1, 0) and (0, -1) as bf16, in registers
    asm volatile("" : "+s"(minus_lo), "+s"(minus_hi));
    // 32 dimensions of a row: four pairs of a, the next four of b
    auto cut8 = [&](const float4 a, const float4 b, Plane(&c)[3]) __attribute__((always_inline)) {
        const Cut w[4] = {{a.x, a.y, minus_lo, minus_hi}, {a.z, a.w, minus_lo, minus_hi}, {b.x, b.y, minus_lo, minus_hi}, {b.z, b.w, minus_lo, minus_hi}};
#pragma unroll
        for (int k = 0; k < 3; k++) c[k] = Plane{{w[0].p[k], w[1].p[k], w[2].p[k], w[3].p[k]}};
    };

    // Unconditional loads: rows past the last one written re-read it (masked below).
    float4 x[8]; // x[m]: K[t = li][16 m + 4 kb ..]
    float4 v[8]; // v[2 r + half]: V[t = 4 kb + r][64 half + 4 li ..]
    auto fetch_k = [&](int tile) __attribute__((always_inline)) {
        const uint32_t ko = __umul24(min(tile * TK + li, max_pos), row_bytes) + k_lane;
#pragma unroll
        for (int m = 0; m < 8; m++) x[m] = ld_at<float4>(kc, ko + 64u * m);
    };
    auto fetch_v = [&](int tile) __attribute__((always_inline)) {
#pragma unroll
        for (int r = 0; r < 4; r++) {
            const uint32_t vo = __umul24(min(tile * TK + 4 * kb + r, max_pos), row_bytes) + v_lane;
            v[2 * r] = ld_at<float4>(vc, vo);
            v[2 * r + 1] = ld_at<float4>(vc, vo + 256u);
        }
    };
    int my_pos[CS];
    float4 qa[CS], qb[CS];
#pragma unroll
    for (int cs = 0; cs < CS; cs++) {
        const int my_qi = (ct + cs) * QPT + li / QG;
        my_pos[cs] = my_qi < B ? pos[my_qi] : -1;
        // wave w cuts dimensions 32 w .. 32 w + 31
        const float *qrow = q + (size_t)min(my_qi, B - 1) * dim + (size_t)(kvh * QG + li % QG) * HS + 32 * wave + 4 * kb;
        qa[cs] = *reinterpret_cast<const float4 *>(qrow), qb[cs] = *reinterpret_cast<const float4 *>(qrow + 16);
    }
    fetch_k(wave);
    fetch_v(wave);
    constexpr int PER = NWV * 64 / HS, HEADS = QG > PER ? QG / PER : 1;
    int dst[HEADS]; // where this thread's outputs go (as in the kernel above)
#pragma unroll
    for (int u = 0; u < HEADS; u++) {
        const int i = (kvh * QG + (tid / HS + u * PER) % QG) * HS + tid % HS;
        dst[u] = scatter ? scatter[i] : i;
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int cs = 0; cs < CS; cs++) {
        Plane c[3];
        cut8(qa[cs], qb[cs], c);
#pragma unroll
        for (int k = 0; k < 3; k++) qs[cs][wave][k][lane] = make_uint4(c[k].u[0], c[k].u[1], c[k].u[2], c[k].u[3]);
    }
    if (tid == 0) again = 0;
    int t_end = my_pos[0] + 1; // the block's tiles end with the last row any of its columns sees
#pragma unroll
    for (int cs = 1; cs < CS; cs++) t_end = max(t_end, my_pos[cs] + 1);
#pragma unroll
    for (int off = 8; off > 0; off >>= 1) t_end = max(t_end, __shfl_xor(t_end, off));
    t_end = __builtin_amdgcn_readfirstlane(t_end);
    const int n_tiles = (t_end + TK - 1) / TK;

    float run_m[CS], run_l[CS];
    v4f acc[CS][8];
#pragma unroll
    for (int cs = 0; cs < CS; cs++) {
        run_m[cs] = kNoScore, run_l[cs] = 0.f;
#pragma unroll
        for (int c = 0; c < 8; c++) acc[cs][c] = v4f{0.f, 0.f, 0.f, 0.f};
    }
    const float scale = 1.44269504088896340736f / sqrtf((float)HS); // log2(e) / sqrt(head_size), src/models.rs:154
    float sign = 1.f;
    __syncthreads();

    // What is cut next goes between the products of what was cut before; K and V of the next tile are asked for when the last of
    // this one's has been cut.
    auto step = [&](int tile, auto last) __attribute__((always_inline)) {
        // Scores: K's planes times Q's, what is below the first planes' product summed apart.
        v4f s[CS], lo[CS];
        {
            Plane kp[2][3], q0[2][CS];
            auto ask = [&](int cs, int i, int k) __attribute__((always_inline)) {
                const uint4 u = qs[cs][i][k][lane];
                return Plane{{u.x, u.y, u.z, u.w}};
            };
            cut8(x[0], x[1], kp[0]);
#pragma unroll
            for (int cs = 0; cs < CS; cs++) q0[0][cs] = ask(cs, 0, 0), s[cs] = lo[cs] = v4f{0.f, 0.f, 0.f, 0.f};
            if (CS > 1) __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const Plane(&c)[3] = kp[i % 2];
                Plane q1[CS], q2[CS];
#pragma unroll
                for (int cs = 0; cs < CS; cs++) q1[cs] = ask(cs, i, 1);
#pragma unroll
                for (int cs = 0; cs < CS; cs++) q2[cs] = ask(cs, i, 2);
                if (i < 3) {
#pragma unroll
                    for (int cs = 0; cs < CS; cs++) q0[(i + 1) % 2][cs] = ask(cs, i + 1, 0);
                    cut8(x[2 * i + 2], x[2 * i + 3], kp[(i + 1) % 2]);
                }
#define L2_SCORES(D, KP, Q) _Pragma("unroll") for (int cs = 0; cs < CS; cs++) D[cs] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(c[KP].b(), Q[cs].b(), D[cs], 0, 0, 0)
                L2_SCORES(lo, 2, q0[i % 2]);
                L2_SCORES(s, 0, q0[i % 2]);
                L2_SCORES(lo, 1, q0[i % 2]);
                L2_SCORES(lo, 1, q1);
                L2_SCORES(lo, 0, q1);
                L2_SCORES(lo, 0, q2);
#undef L2_SCORES
                if (CS > 1 || i == 3) __builtin_amdgcn_sched_barrier(0);
                if (i == 2 && !last) fetch_k(tile + NWV);
            }
        }
        // Weights, their planes as the sums take them: (0, 2), (1, 1) and (0, 0)
        Plane pc[CS][3];
#pragma unroll
        for (int cs = 0; cs < CS; cs++) {
            float sc[4], mx = kNoScore;
            const int see = my_pos[cs] - tile * TK - 4 * kb; // causal: this column's query sees rows 0..pos
#pragma unroll
            for (int r = 0; r < 4; r++) {
                sc[r] = r <= see ? (s[cs][r] + lo[cs][r]) * scale : kNoScore;
                mx = fmaxf(mx, sc[r]);
            }
            // A maximum moves only by more than 8, for the column that it is of: weights of up to 2^8 lose nothing in fp32, and what
            // was summed is seldom rescaled.
            if (__any(mx > run_m[cs] + 8.f)) {
                mx = lanes::rows_max(mx); // the column's four lanes agree
                const float m_new = mx > run_m[cs] + 8.f ? mx : run_m[cs];
                const float c = exp2_fast(run_m[cs] - m_new);
                run_l[cs] *= c;
#pragma unroll
                for (int cc = 0; cc < 8; cc++) acc[cs][cc] *= c;
                run_m[cs] = m_new;
            }
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const float p = r <= see ? exp2_fast(sc[r] - run_m[cs]) : 0.f;
                run_l[cs] += p;
                sc[r] = p * sign;
            }
            const Cut a(sc[0], sc[1], minus_lo, minus_hi), b(sc[2], sc[3], minus_lo, minus_hi);
            pc[cs][0] = Plane{{a.p[0], b.p[0], a.p[2], b.p[2]}};
            pc[cs][1] = Plane{{a.p[1], b.p[1], a.p[1], b.p[1]}};
            pc[cs][2] = Plane{{a.p[0], b.p[0], a.p[0], b.p[0]}};
        }
        // V's planes times the weights', two products of 16 rows in one of 32: (2 0, 0 2), (1 1, 0 1), (1 0, 0 0).  Summed for the
        // tile and added with the rounding of the vector unit: the matrix unit's sums come out too small on average, so
        // every other tile's are taken negated.
        {
            Plane w[2][2]; // (2, 0) and (1, 0)
            v4f t[2][CS];
            auto cut = [&](int i) __attribute__((always_inline)) {
                const int h = i / 4, e = i % 4;
                const float4 r[4] = {v[h], v[2 + h], v[4 + h], v[6 + h]};
                const Cut a(reinterpret_cast<const float *>(&r[0])[e], reinterpret_cast<const float *>(&r[1])[e], minus_lo, minus_hi);
                const Cut b(reinterpret_cast<const float *>(&r[2])[e], reinterpret_cast<const float *>(&r[3])[e], minus_lo, minus_hi);
                w[i % 2][0] = Plane{{a.p[2], b.p[2], a.p[0], b.p[0]}};
                w[i % 2][1] = Plane{{a.p[1], b.p[1], a.p[0], b.p[0]}};
            };
            auto add = [&](int i) __attribute__((always_inline)) {
#pragma unroll
                for (int cs = 0; cs < CS; cs++)
#pragma unroll
                    for (int r = 0; r < 4; r++) acc[cs][i][r] = fmaf(t[i % 2][cs][r], sign, acc[cs][i][r]);
            };
            cut(0);
            if (CS > 1) __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int i = 0; i < 8; i++) {
                const Plane(&c)[2] = w[i % 2];
                if (i > 0) add(i - 1);
                if (i < 7) cut(i + 1);
#pragma unroll
                for (int cs = 0; cs < CS; cs++) t[i % 2][cs] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(c[0].b(), pc[cs][0].b(), v4f{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
#pragma unroll
                for (int cs = 0; cs < CS; cs++) t[i % 2][cs] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(c[1].b(), pc[cs][1].b(), t[i % 2][cs], 0, 0, 0);
#pragma unroll
                for (int cs = 0; cs < CS; cs++) t[i % 2][cs] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(c[1].b(), pc[cs][2].b(), t[i % 2][cs], 0, 0, 0);
                if (CS > 1 || i % 4 == 3) __builtin_amdgcn_sched_barrier(0);
                if (i == 6 && !last) fetch_v(tile + NWV);
            }
            add(7);
        }
        sign = -sign;
    };
    // The last tile apart: with a branch around the loads for the next one they are waited for at once.
    int tile = wave;
    for (; tile + NWV < n_tiles; tile += NWV) step(tile, std::false_type());
    if (tile < n_tiles) step(tile, std::true_type());

    // The waves agree on each column's maximum and sum, each scales its O by its share, and these add up in LDS.
    static_assert(NC * HS / (NWV * 64) == kSetOutputs && sizeof(qs) >= CS * 8 * 64 * sizeof(float4), "what prefill_fp32 takes over");
    uint32_t redo[CS] = {}; // this thread's outputs that are not finite
#pragma unroll
    for (int cs = 0; cs < CS; cs++) {
        const float l = lanes::rows_sum(run_l[cs]);
        if (kb == 0) ml[cs][wave][li] = make_float2(run_m[cs], l);
    }
    __syncthreads();
#pragma unroll
    for (int cs = 0; cs < CS; cs++) {
        float M = kNoScore, den = 0.f;
#pragma unroll
        for (int w = 0; w < NWV; w++) M = fmaxf(M, ml[cs][w][li].x);
#pragma unroll
        for (int w = 0; w < NWV; w++) den = fmaf(exp2_fast(ml[cs][w][li].x - M), ml[cs][w][li].y, den);
        const float share = exp2_fast(run_m[cs] - M) / den;
        if (cs > 0) __syncthreads(); // the set before has been read
#pragma unroll
        for (int c = 0; c < 8; c++) acc[cs][c] *= share;
#pragma unroll
        for (int r = 0; r < 4; r++) // register r of accumulators 0..3 is d = 16 kb + 4 r + 0..3, of 4..7 the same 64 further on
#pragma unroll
            for (int half = 0; half < 2; half++)
                *reinterpret_cast<float4 *>(&comb[wave][li][64 * half + 16 * kb + 4 * r]) =
                    make_float4(acc[cs][4 * half][r], acc[cs][4 * half + 1][r], acc[cs][4 * half + 2][r], acc[cs][4 * half + 3][r]);
        __syncthreads();
#pragma unroll
        for (int u = 0; u < NC * HS / (NWV * 64); u++) {
            const int j = tid / HS + u * PER, d = tid % HS, qi = (ct + cs) * QPT + j / QG;
            const float v = (comb[0][j][d] + comb[1][j][d]) + (comb[2][j][d] + comb[3][j][d]);
            if (qi < B) {
                reinterpret_cast<_Float16 *>(out)[(size_t)qi * dim + h16_slot(dst[u % HEADS])] = (_Float16)v;
                if (!__builtin_isfinite(v)) redo[cs] |= 1u << u;
            }
        }
        if (redo[cs]) again = 1;
    }
    // The planes of an infinity are not one (inf - inf), and one infinite term hides what the others add up to: outputs that are not
    // finite are taken from the fp32 form.
    __syncthreads();
    if (again)
        prefill_fp32<QG, NWV, 1, CS>(out, q, kc, vc, pos, scatter, n_heads, n_kv_heads, B, max_pos, unit_rows, comb,
                                     reinterpret_cast<float4(*)[8][64]>(qs), redo);
}

// Merge the splits of one q head: out = sum_s 2^(m_s - M) o_s / sum_s 2^(m_s - M) l_s.
// Every load goes out before anything is waited for (the partial outputs of this thread's splits, the
// (m_s, l_s) pairs, the scatter target: one round trip to memory instead of three); wave 0 then turns the
// (m_s, l_s) of up to 64 splits into weights and 4 groups of 128 threads sum the weighted partial outputs.  Compiled for 8,
// 16, 32 and 64 splits: a load per split that is not there costs as much as one that is (7B behind 1500 positions 462 -> 457 us
// per token of 8 layers, 70B behind 1000 and 4096 947 -> 944 and 983 -> 980).
template <int NU> // splits per thread: 4 NU of them over 4 groups
__global__ __launch_bounds__(512) void attn_combine_kernel(const AttnDecode A) {
    constexpr int HS = 128;
    pin_args(A);
    __shared__ float w[64];
    __shared__ float den_s;
    __shared__ float red[3][HS];
    const int h = blockIdx.x, tid = threadIdx.x, d = tid & 127, grp = tid >> 7;
    const int pos = A.dpos ? A.dpos[0] : A.pos;
    const int ns = min(A.n_splits, pos / A.ts + 1);
    const float *p = A.part + (size_t)h * A.max_splits * (HS + 2);
    float pv[NU];
#pragma unroll
    for (int u = 0; u < NU; u++) pv[u] = p[min(grp + 4 * u, ns - 1) * (HS + 2) + d]; // past the end: the last split again, unused
    const int i = h * HS + d;
    const int dst = A.scatter ? A.scatter[i] : i;
    const int sl = min(tid & 63, ns - 1);
    const float ms_r = p[sl * (HS + 2) + HS], ls_r = p[sl * (HS + 2) + HS + 1];
    if (tid < 64) {
        const bool on = tid < ns;
        const float ms = on ? ms_r : kNoScore;
        const float ls = on ? ls_r : 0.f;
        const float M = wave_max(ms);
        const float ws = on ? exp2_fast(ms - M) : 0.f;
        w[tid] = ws;
        const float den = wave_sum(ws * ls);
        if (tid == 0) den_s = den;
    }
    __syncthreads();
    float num = 0.f;
#pragma unroll
    for (int u = 0; u < NU; u++) num = fmaf(w[grp + 4 * u], pv[u], num); // w is 0 beyond the last split
    if (grp > 0) red[grp - 1][d] = num;
    __syncthreads();
    if (grp == 0) {
        num += red[0][d];
        num += red[1][d];
        num += red[2][d];
        A.out[dst] = num / den_s;
    }
}

template <int NWV, int DS>
int attn_launch_sliced(const AttnDecode &a, hipStream_t st) {
    l2_launch((attn_decode_kernel<1, NWV, DS>), dim3(a.n_kv_heads, a.n_heads / a.n_kv_heads, DS), dim3(NWV * 64), 0, st, a);
    L2_HIP(hipGetLastError());
    return L2_OK;
}

template <int QG>
int attn_launch_qg(const AttnDecode &a, hipStream_t st) {
    static const bool valu = []() {
        const char *v = getenv("L2_ATTN_IMPL");
        return v && !strcmp(v, "valu");
    }();
    // With eight query heads per kv head the first 256 timesteps stay on the matrix cores, although blocks of one head are faster (64 heads
    // of 8, 50 and 240 timesteps 37.0 / 42.0 us per layer, with blocks of one head 35.4 / 36.7): in other sums the texts that are sampled
    // from a model are others (of 20 of 60 tokens from 70B's widths three were), and short contexts are where texts are sampled.  It is
    // that and no rule of reproducibility: the form changes with the length, and with a captured step by the bucket's end.
    if (a.n_splits == 1 && (QG < 8 || valu || a.ts > kFewTimesteps)) { // slices of the head: as many as keep one block per CU
        const bool wide = a.pos >= 64, eight = a.n_heads * 8 <= cu_count();
        if (eight) return wide ? attn_launch_sliced<8, 8>(a, st) : attn_launch_sliced<4, 8>(a, st);
        return wide ? attn_launch_sliced<8, 4>(a, st) : attn_launch_sliced<4, 4>(a, st);
    }
    if constexpr (QG >= 4) {
        if (!valu) {
            l2_launch((attn_decode_mfma_kernel<QG>), dim3(a.n_kv_heads, a.n_splits), dim3(256), 0, st, a);
            L2_HIP(hipGetLastError());
            return L2_OK;
        }
    }
    constexpr size_t lds = QG >= 4 ? (size_t)16 * QG * kCombRow * sizeof(float) : 0; // the partial results of 16 rows
    if (lds > 48 * 1024) {
        static LdsLimit limit; // per instantiation
        L2_TRY(limit.ensure(reinterpret_cast<const void *>(attn_decode_kernel<QG, 4, 1>), lds));
    }
    l2_launch((attn_decode_kernel<QG, 4, 1>), dim3(a.n_kv_heads, a.n_splits), dim3(256), lds, st, a);
    L2_HIP(hipGetLastError());
    return L2_OK;
}

} // namespace

int attention_decode_launch(const AttnDecode &a, hipStream_t st) {
    const int qg = a.n_heads / a.n_kv_heads;
    if (a.ts < 64 || a.ts % 64 || a.n_splits < 1 || a.n_splits > a.max_splits || a.max_splits > 64)
        return l2_fail(L2_ERR_ARG, "attention: ts=%d splits=%d/%d", a.ts, a.n_splits, a.max_splits);
    switch (qg) {
        case 1: L2_TRY(attn_launch_qg<1>(a, st)); break;
        case 2: L2_TRY(attn_launch_qg<2>(a, st)); break;
        case 4: L2_TRY(attn_launch_qg<4>(a, st)); break;
        case 8: L2_TRY(attn_launch_qg<8>(a, st)); break;
        default: return l2_fail(L2_ERR_ARG, "attention: %d query heads per kv head (1, 2, 4 or 8)", qg);
    }
    if (a.n_splits > 1) {
        const auto combine = a.n_splits <= 8    ? attn_combine_kernel<2>
                             : a.n_splits <= 16 ? attn_combine_kernel<4>
                             : a.n_splits <= 32 ? attn_combine_kernel<8>
                                                : attn_combine_kernel<16>;
        l2_launch(combine, dim3(a.n_heads), dim3(512), 0, st, a);
        L2_HIP(hipGetLastError());
    }
    return L2_OK;
}

template <int QG>
static int prefill_qg(void *out, int planes, const float *q, const float *kc, const float *vc, const int32_t *pos,
                      const int32_t *scatter, int n_heads, int n_kv_heads, int max_pos, int B, hipStream_t st) {
    // 16 columns (queries x heads of the group) per block, or 32 where that still leaves two blocks per CU: with fewer
    // the longer blocks cost more than the shared tiles save (32 heads, 299 tokens: 18.6 us with 16, 19.7 with 32).  In the fp16
    // mode, which cuts a tile once for all its columns, from one block per CU on: 32 heads, 200 tokens (224 blocks of 32 columns) 10.2
    // with 16 and 12.1 with 32, 64 on 8 kv heads, 128 (256) 9.4 and 9.5, 40 heads, 200 (280) 13.9 and 13.8, 32 heads, 299 (320)
    // 17.5 and 15.6, 64 on 8, 777 106.8 and 79.8.
    const int sets = (B * QG + 15) / 16;
    const long pairs = (long)n_kv_heads * ((sets + 1) / 2);
    const bool two = planes == 1 ? pairs > cu_count() : pairs >= 2 * cu_count();
    const dim3 block(256), grid(n_kv_heads, two ? (sets + 1) / 2 : sets);
    const int cus = cu_count(), per_unit = cus / n_kv_heads, rows = (int)grid.y;
    const int unit_rows = cus % n_kv_heads == 0 && rows > per_unit && rows <= 2 * per_unit ? per_unit : 0; // see column_tile
#define L2_PREFILL_ATTN(...)                                                                                             \
    l2_launch((__VA_ARGS__), grid, block, 0, st, out, q, kc, vc, pos, scatter, n_heads, n_kv_heads, B, max_pos, unit_rows)
    switch (planes) {
        case 0: l2_launch(attn_prefill_kernel<QG>, dim3(n_kv_heads, (B * QG + 7) / 8), block, 0, st, (float *)out, q, kc, vc, pos, scatter, n_heads, n_kv_heads, B); break;
        case 1:
            if (two) L2_PREFILL_ATTN(attn_prefill_cut_kernel<QG, 2>);
            else L2_PREFILL_ATTN(attn_prefill_cut_kernel<QG, 1>);
            break;
        case 3:
            if (two) L2_PREFILL_ATTN(attn_prefill_mfma16_kernel<QG, 2>);
            else L2_PREFILL_ATTN(attn_prefill_mfma16_kernel<QG, 1>);
            break;
        default: return l2_fail(L2_ERR_ARG, "attention: %d planes", planes);
    }
#undef L2_PREFILL_ATTN
    L2_HIP(hipGetLastError());
    return L2_OK;
}

int attention_launch(void *out, int planes, const float *q, const float *kcache_l, const float *vcache_l,
                     const int32_t *pos, const int32_t *scatter, int n_heads, int n_kv_heads,
                     int head_size, int max_pos, int B, hipStream_t st) {
    if (head_size != 128) return l2_fail(L2_ERR_ARG, "attention: head_size=%d (128 only)", head_size);
    switch (n_heads / n_kv_heads) {
        case 1: return prefill_qg<1>(out, planes, q, kcache_l, vcache_l, pos, scatter, n_heads, n_kv_heads, max_pos, B, st);
        case 2: return prefill_qg<2>(out, planes, q, kcache_l, vcache_l, pos, scatter, n_heads, n_kv_heads, max_pos, B, st);
        case 4: return prefill_qg<4>(out, planes, q, kcache_l, vcache_l, pos, scatter, n_heads, n_kv_heads, max_pos, B, st);
        case 8: return prefill_qg<8>(out, planes, q, kcache_l, vcache_l, pos, scatter, n_heads, n_kv_heads, max_pos, B, st);
    }
    return l2_fail(L2_ERR_ARG, "attention: %d query heads per kv head (1, 2, 4 or 8)", n_heads / n_kv_heads);
}
