// Row-streaming form of the GPTQ 4-bit dequant matvec (gfx950, wave64).
//
// Same function, prologue and epilogues as the row-tile kernel in
// kernels_q4.hip; what differs is who walks what.  Here every lane owns ONE
// chunk of K (32 consecutive inputs) for the whole kernel and keeps that slice
// of x in registers, so the main loop reads nothing from LDS.  NWK = ceil(C/64)
// waves side by side cover a full row; S such wave groups ("streams") per block
// take rows s, s+S, s+2S, ... of the block's row range.  A stream keeps P rows
// in flight: the loads of row i+P are issued before row i is consumed, so once
// the pipe is primed the HBM stream and the dequant arithmetic overlap inside
// every wave rather than only across blocks.
//
// Reduction: four DPP adds fold a wave's 64 partials into 4 (one per 16-lane
// row); those go to a small double-buffered LDS tile [row][NWK*4]; after one
// barrier per tile of P*S rows, one thread per row adds them in a fixed order
// and runs the epilogue.  No atomics: results are bit-stable.
//
// Integer form (MODE 1, selected with L2_Q4_IMPL=idot; the fp32 form is the default).  The vector ALU is
// the co-bottleneck of the fp32 form (one FMA, one convert-equivalent and 3/8 of a mask per nibble).  The
// integer form quantises x once per block after staging, chunk by chunk, to 24-bit fixed point against a
// power-of-two step (delta = 2^(e-22), |x| < 2^e within the chunk) and stores it as six planes of balanced
// base-16 digits (-8..7), 8 digits per word in the nibble order of the weights.  A weight word XOR 0x88888888
// is the 8 signed nibbles n - 8, so v_dot8_i32_i4 multiplies one weight word with one digit word: 24
// instructions per 32 weights instead of ~76, exact integer sums, and
//   sum_k (n_k - z1) x_k = delta * (I - (z1 - 8) * sum_k q_k),  I = sum_d 16^d a_d.
// The quantisation error (2^-23 of the chunk maximum per element) is of the size of fp32 rounding.  Its
// quantisation prologue costs more than the shorter loop saves on the shapes measured, hence not the default.
#include <stdio.h>
#include <stdlib.h>
#include <string.h>

#include <type_traits>

#include "q4_common.h"

namespace {

using namespace q4;

constexpr int kPlaneWords = 28; // per chunk: 6 planes x 4 words, delta, sum of q, 2 pad

template <int CTRL>
__device__ __forceinline__ int dpp_xchg_i(int v) {
    return __builtin_amdgcn_update_dpp(0, v, CTRL, 0xF, 0xF, true);
}

// Quantise a staged vector (xs[c*36 + i], c < C, i < 32) in place into digit
// planes: word (c, d, j) at ((uint32_t*)xs)[c*28 + d*4 + j]; delta and sum(q)
// as floats at [c*28 + 24], [c*28 + 25].  Thread -> (chunk, word of 8 elements);
// the 4 threads of a chunk are adjacent lanes.  Outputs only ever land on
// inputs of lower chunks, which are consumed in earlier passes.
template <int NT>
__device__ __forceinline__ void quantize_in_place(float *xs, int C, int tid) {
    uint32_t *xw = reinterpret_cast<uint32_t *>(xs);
    const int n_words = C * 4;
    for (int base = 0; base < n_words; base += NT) {
        const int wi = base + tid;
        const bool ok = wi < n_words;
        const int c = wi >> 2, j = wi & 3;
        float v[8];
        if (ok) {
            const float4 a = *reinterpret_cast<const float4 *>(&xs[c * kChunkPad + j * 8]);
            const float4 b = *reinterpret_cast<const float4 *>(&xs[c * kChunkPad + j * 8 + 4]);
            v[0] = a.x, v[1] = a.y, v[2] = a.z, v[3] = a.w, v[4] = b.x, v[5] = b.y, v[6] = b.z, v[7] = b.w;
        } else {
#pragma unroll
            for (int e = 0; e < 8; e++) v[e] = 0.f;
        }
        float am = 0.f;
#pragma unroll
        for (int e = 0; e < 8; e++) am = fmaxf(am, fabsf(v[e]));
        am = fmaxf(am, dpp_xchg<0xB1>(am));
        am = fmaxf(am, dpp_xchg<0x4E>(am));
        // am < 2^(eb-126): step 2^(eb-148) keeps |x/step| < 2^22
        int eb = (int)((__builtin_bit_cast(uint32_t, am) >> 23) & 0xFFu);
        eb = eb < 22 ? 22 : eb;
        const float inv = __builtin_bit_cast(float, (uint32_t)(275 - eb) << 23);
        const float delta = __builtin_bit_cast(float, (uint32_t)(eb - 21) << 23);
        uint32_t u[8];
        int sq = 0;
#pragma unroll
        for (int e = 0; e < 8; e++) {
            const int q = (int)rintf(v[e] * inv);
            sq += q;
            u[e] = (uint32_t)(q + 0x888888);
        }
        sq += dpp_xchg_i<0xB1>(sq);
        sq += dpp_xchg_i<0x4E>(sq);
        uint32_t pw[6];
#pragma unroll
        for (int d = 0; d < 6; d++) {
            uint32_t w = 0;
#pragma unroll
            for (int e = 0; e < 8; e++) w |= ((u[e] >> (4 * d)) & 15u) << (4 * e);
            pw[d] = w ^ 0x88888888u; // unsigned digit - 8 as a signed nibble
        }
        __syncthreads(); // every input of this pass is in registers
        if (ok) {
#pragma unroll
            for (int d = 0; d < 6; d++) xw[c * kPlaneWords + d * 4 + j] = pw[d];
            if (j == 0) {
                xs[c * kPlaneWords + 24] = delta;
                xs[c * kPlaneWords + 25] = (float)sq;
            }
        }
        __syncthreads();
    }
}

// sum_k (n_k - 8) q_k over one chunk: 4 weight words against 6 digit planes.
__device__ __forceinline__ float chunk_idot(const uint4 w, const int (&xp)[24]) {
    const int w0 = (int)(w.x ^ 0x88888888u), w1 = (int)(w.y ^ 0x88888888u), w2 = (int)(w.z ^ 0x88888888u),
              w3 = (int)(w.w ^ 0x88888888u);
    int a[6];
#pragma unroll
    for (int d = 0; d < 6; d++) {
        int t = __builtin_amdgcn_sdot8(w0, xp[d * 4 + 0], 0, false);
        t = __builtin_amdgcn_sdot8(w1, xp[d * 4 + 1], t, false);
        t = __builtin_amdgcn_sdot8(w2, xp[d * 4 + 2], t, false);
        a[d] = __builtin_amdgcn_sdot8(w3, xp[d * 4 + 3], t, false);
    }
    const int lo = (((a[2] << 4) + a[1]) << 4) + a[0];
    const int hi = (((a[5] << 4) + a[4]) << 4) + a[3];
    return fmaf((float)hi, 4096.0f, (float)lo);
}

// A load of weights: read once per token and never again before some 40 GB of other weights have gone by,
// so it is marked non-temporal (no point in keeping the line in L2 or in the memory-side cache, where it
// would only push out what is re-read: x, the scales' neighbours, the next kernel's operands).  Measured on
// the 70B shapes: w1|w3 51.0 -> 45.8 us, w2 28.7 -> 25.7 us per launch.
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
template <class T>
__device__ __forceinline__ T ld_at(const void *base, uint32_t byte_offset) {
    const char *p = reinterpret_cast<const char *>(base) + byte_offset;
    if constexpr (sizeof(T) == 16)
        return __builtin_bit_cast(T, __builtin_nontemporal_load(reinterpret_cast<const u32x4 *>(p)));
    else
        return __builtin_nontemporal_load(reinterpret_cast<const T *>(p));
}

__device__ __forceinline__ void st_at(float *base, uint32_t byte_offset, float v) {
    *reinterpret_cast<float *>(reinterpret_cast<char *>(base) + byte_offset) = v;
}

// A uniform value, required in scalar registers where this is written: the load behind it is issued and
// waited for here rather than where the value is first used.  The value itself is not redefined (an asm
// output would hide from the compiler that a pointer is a kernel argument, i.e. global memory).
template <class T>
__device__ __forceinline__ T pin_s(T v) {
    asm volatile("" ::"s"(v));
    return v;
}

// The operands of one matrix of a launch.
struct MatOps {
    const uint4 *qweight;
    const int32_t *qzeros;
    const float *scales;
    float *y;
    int out;
};

// What a launch passes besides the leading arguments (see q4_stream_kernel).
struct StreamArgs {
    MatOps m[3];
    Q4Epi e;
    int groups, rows_per_block;
    float eps;
};

// A matrix's operands, in scalar registers.
__device__ __forceinline__ MatOps mat_ops(const MatOps &M) {
    MatOps o;
    o.qweight = pin_s(M.qweight);
    o.qzeros = pin_s(M.qzeros);
    o.scales = pin_s(M.scales);
    o.y = pin_s(M.y);
    o.out = pin_s(M.out);
    return o;
}

// What a thread holds of a vector on its way to LDS, NX pieces of four floats.  NX * 64 * NW pieces cover the
// longest vector of the kernel, so the staging has no loop, and past the vector's end a buffer load returns zeros,
// so it has no branch per piece either.  That is for the length of the code: a launch of 5 to 13 us runs its
// prologue once, from an instruction cache that does not hold it, and pays some 0.1 us per kilobyte.  With a guard
// per piece and a loop for what a first batch had left, the kernels were 2 to 4 KB longer and a 7B token took
// 1332 us, against 1301 in this form.
template <int NX>
struct XRegs {
    float4 v[NX], g[NX];
};

__device__ __forceinline__ float4 ld_bounded(__amdgpu_buffer_rsrc_t r, int byte_offset) {
    return __builtin_bit_cast(float4, __builtin_amdgcn_raw_buffer_load_b128(r, byte_offset, 0, 0));
}

__device__ __forceinline__ __amdgpu_buffer_rsrc_t bounded(const float *p, int n) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<float *>(p), 0, n * 4, 0x00020000);
}

template <int NW, int NX>
__device__ __forceinline__ void x_issue(const float *x, const float *wn, int in, int tid, XRegs<NX> &r) {
    const __amdgpu_buffer_rsrc_t rx = bounded(x, in);
#pragma unroll
    for (int u = 0; u < NX; u++) r.v[u] = ld_bounded(rx, (u * NW * 64 + tid) * 16);
    if (wn) {
        const __amdgpu_buffer_rsrc_t rg = bounded(wn, in);
#pragma unroll
        for (int u = 0; u < NX; u++) r.g[u] = ld_bounded(rg, (u * NW * 64 + tid) * 16);
    }
}

// The pieces into the padded chunks, with the sums of the chunks; returns the thread's share of sum(x^2).
// All slots are written (zeros past the vector's end).
template <int NWK, int NW, int NX>
__device__ __forceinline__ float x_stage(bool norm, int tid, XRegs<NX> &r, float *xs, float *xsum) {
    float ssq = 0.f;
    if (norm) {
#pragma unroll
        for (int u = 0; u < NX; u++) {
            float4 &v = r.v[u];
            ssq = fmaf(v.x, v.x, ssq);
            ssq = fmaf(v.y, v.y, ssq);
            ssq = fmaf(v.z, v.z, ssq);
            ssq = fmaf(v.w, v.w, ssq);
            v.x *= r.g[u].x;
            v.y *= r.g[u].y;
            v.z *= r.g[u].z;
            v.w *= r.g[u].w;
        }
    }
#pragma unroll
    for (int u = 0; u < NX; u++) {
        const int j4 = u * NW * 64 + tid;
        const float4 v = r.v[u];
        float s = (v.x + v.y) + (v.z + v.w);
        s += dpp_xchg<0xB1>(s);  // the 8 lanes that hold one chunk add up its sum: lanes ^1
        s += dpp_xchg<0x4E>(s);  // lanes ^2
        s += dpp_xchg<0x141>(s); // 7 - lane within each 8: the other quad
        if ((u + 1) * NW * 64 <= NWK * 512 || j4 < NWK * 512) {
            *reinterpret_cast<float4 *>(&xs[(j4 >> 3) * kChunkPad + (j4 & 7) * 4]) = v;
            xsum[j4 >> 3] = s; // the same value from all 8 lanes
        }
    }
    return ssq;
}

struct RowData {
    uint4 w;
    float s;
    int32_t z;
};

// A chunk's sum from those of its fours, in the association the block-wide staging uses (the tree of its three cross-lane
// adds), so that a form of the operator which takes the sum by itself gives the same bits.
__device__ __forceinline__ float chunk_sum(const float (&s4)[8]) {
    return ((s4[0] + s4[1]) + (s4[2] + s4[3])) + ((s4[7] + s4[6]) + (s4[5] + s4[4]));
}

// A lane's share of a row's dot product: scale times sum.  What a row's first addition across lanes rounds is written out here, since
// it is the row's last bit and every form of a launch must give the same: a row of the loop rounds the product, then the sum;
// one of those that stand behind the loop, the remainder of a block's rows, rounds once.
struct Share {
    float scale, sum;
    __device__ __forceinline__ float product() const {
#pragma clang fp contract(off)
        return scale * sum;
    }
    __device__ __forceinline__ float two_lanes(bool behind) const {
#pragma clang fp contract(off)
        const float other = dpp_xchg<0xB1>(scale * sum);
        return behind ? fmaf(scale, sum, other) : scale * sum + other;
    }
};

// The leading arguments are what the loads of x need: x of the launch's matrices (blocks0 and blocks1 of the grid belong to the
// first and second), the norm weights of the first, those of the others behind it, or null, and the inverse of g_index of the
// gathering form.  The dispatch puts them into scalar registers (-amdgpu-kernarg-preload-count), so x is asked for while the
// rest of the arguments, cold in the scalar cache, is still on its way.  In a chain of dependent kernels that is 0.15 us of each
// (8 MB 3.57 -> 3.43 us, 46 MB 10.08 -> 9.92); 8 layers of 7B, a token 378.6 -> 373.3 us.
//
// MODE 0: fp32 inner loop, x staged through LDS (rmsnorm prologue, several matrices, row pairs).
// MODE 1: integer-dot inner loop, x staged and quantised in LDS.
// MODE 2: fp32 inner loop, one matrix without rmsnorm: every wave loads its own slice of x (coalesced)
//         and turns it into the per-lane chunks through LDS of its own; no barrier before the first row.
// MODE 3: MODE 0, a block doing the work of two of half its waves (see two_in_one).
// GATHER (MODE 0, one matrix, no rmsnorm): x arrives in its natural order and the kernel applies the act-order
//         permutation itself, x[g_index[j]] (src/gptq.rs:99-122), for a caller with no producer to do it: x and the
//         inverse of g_index are requested together and every element is written straight to its place in the
//         staged chunks (the scatter a producer's epilogue would have done); the chunk sums are taken by the lanes.
template <int G, int NWK, int S, bool PAIR, int MODE, int P, bool GATHER = false>
__global__ __launch_bounds__(NWK *S * 64) void q4_stream_kernel(const float *x0, const float *x1, const float *x2, const float *wn0,
                                                                const int32_t *gidx, const int in, const int blocks0, const int blocks1,
                                                                const StreamArgs L) {
    constexpr bool IDOT = MODE == 1, DIRECT = MODE == 2, TWO = MODE == 3;
    static_assert(!GATHER || (MODE == 0 && !PAIR), "the gathering form takes one matrix through the block-wide staging");
    static_assert(!(DIRECT && PAIR), "the direct form takes one matrix");
    static_assert(!(TWO && PAIR), "two blocks in one: single rows");
    constexpr int NM = PAIR ? 2 : 1;
    constexpr int NW = NWK * S;
    constexpr int NWX = TWO ? NW / 2 : NW; // the waves that stage x (the sum of squares has the order of so many)
    // P rows (row pairs) are in flight per stream
    constexpr int TR = P * S;       // rows per reduction tile
    constexpr int PW = NWK * 4;     // partials per row
    constexpr int CPG = G / 32;     // chunks per group
    extern __shared__ float lds[];
    __shared__ float red[NW];
    __shared__ float part[2][TR][NM][PW];

    const int b = blockIdx.y;
    const int tid = threadIdx.x;
    const int lane = tid & 63;
    // the wave's number as a scalar: the row a wave works on, and with it the row's part of every address and
    // the shift that extracts its zero point, are then scalar arithmetic, off the vector ALU
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int kslice = wave % NWK;
    const int stream = wave / NWK;
    constexpr int NC = NWK * 64;                 // chunks the waves of a row cover
    constexpr int xstride = NC * kChunkPad + NC; // floats of LDS per staged vector
    constexpr int NX = (8 * NWK + NWX - 1) / NWX; // pieces of x per thread of the NWX waves that stage it
    const bool stages = NWX == NW || wave < NWX;

    // Which matrix the block's rows belong to.
    int rb = blockIdx.x, mi = 0;
    const float *x_of[2] = {x0, x1};
    if constexpr (!PAIR) {
        if (rb >= blocks0) {
            rb -= blocks0;
            mi = 1;
            x_of[0] = x1;
            if (rb >= blocks1) {
                rb -= blocks1;
                mi = 2;
                x_of[0] = x2;
            }
        }
    }
    const bool has_wn = wn0 != nullptr;

    // x first, then the first rows of the weights: loads return in order, and
    // the staging of x (a cache hit) must not queue behind rows that come from HBM.
    XRegs<NX> xr[DIRECT ? 1 : NM];
    float4 xd[DIRECT ? 8 : 1];
    int4 gi[GATHER ? NX : 1];
    if constexpr (GATHER) {
        const int n4 = in >> 2;
        const int4 *g4 = reinterpret_cast<const int4 *>(gidx);
#pragma unroll
        for (int u = 0; u < NX; u++) {
            const int j4 = u * (NW * 64) + tid;
            gi[u] = j4 < n4 ? g4[j4] : make_int4(0, 0, 0, 0);
        }
    }
    if constexpr (DIRECT) {
        // this wave's 64 chunks of x, 1 KB per load instruction (whole cache lines); past the end the last
        // 16 bytes are re-read and zeroed below
        const float4 *x4 = reinterpret_cast<const float4 *>(x0 + (size_t)b * in);
        const int n4 = in >> 2;
#pragma unroll
        for (int i = 0; i < 8; i++) xd[i] = x4[min(kslice * 512 + i * 64 + lane, n4 - 1)];
    } else if (stages) {
#pragma unroll
        for (int q = 0; q < NM; q++)
            x_issue<NWX, NX>(x_of[q] + (size_t)b * in, has_wn ? wn0 + (size_t)(mi + q) * in : nullptr, in, tid, xr[q]);
    }
    __builtin_amdgcn_sched_barrier(0);

    // Every other scalar operand is asked for at once, and pinned in SGPRs: a kernel's
    // arguments are cold in the scalar cache, a load that misses takes some 0.3 us, and loads the compiler
    // places where their values are first used follow each other (the matrix of this block, then its
    // pointers, then the row geometry: three round trips in front of the first weight load).
    const int groups = pin_s(L.groups);
    const int rows_per_block = pin_s(L.rows_per_block);
    const float eps = pin_s(L.eps);
    // epilogue operands, uniform for the block
    const int epi_kind = pin_s(L.e.kind);
    const int n_scatter = pin_s(L.e.n_scatter);
    const float *__restrict__ res = pin_s(L.e.res);
    const int32_t *__restrict__ sc_idx[3] = {pin_s(L.e.sc_idx[0]), pin_s(L.e.sc_idx[1]), pin_s(L.e.sc_idx[2])};
    float *__restrict__ sc_out[3] = {pin_s(L.e.sc_out[0]), pin_s(L.e.sc_out[1]), pin_s(L.e.sc_out[2])};
    MatOps mat[NM];
    if constexpr (PAIR) {
        mat[0] = mat_ops(L.m[0]);
        mat[1] = mat_ops(L.m[1]);
    } else {
        const MatOps m0 = mat_ops(L.m[0]), m1 = mat_ops(L.m[1]), m2 = mat_ops(L.m[2]);
        mat[0] = m0;
        if (mi > 0) {
            mat[0] = m1;
            if (mi > 1) mat[0] = m2;
        }
    }
    const int C = in >> 5;
    const int n_out = mat[0].out;
    const int row0 = rb * rows_per_block;
    const int row1 = min(row0 + rows_per_block, n_out);
    const int c = kslice * 64 + lane; // this lane's chunk, for good
    const bool has_chunk = c < C;

    // Row i of this stream is row0 + stream + i * S. Loads are unconditional so
    // that the loop body stays one basic block and every wait names only the
    // oldest row in flight: rows past the end re-read the block's last row and
    // lanes past the last chunk re-read the last chunk (their x is zero).
    const int cc = has_chunk ? c : C - 1;
    const int g = cc / CPG;
    const int last = row1 - 1;
    const uint4 *__restrict__ wq[NM];
    const float *__restrict__ sc[NM];
    const int32_t *__restrict__ zq[NM];
#pragma unroll
    for (int q = 0; q < NM; q++) {
        wq[q] = mat[q].qweight;
        sc[q] = mat[q].scales;
        zq[q] = mat[q].qzeros;
    }
    const uint32_t cc16 = (uint32_t)cc << 4, g4 = (uint32_t)g << 2; // the lane's part of the byte offsets
    auto fetch = [&](int i, RowData(&d)[NM]) {
        const int o = min(row0 + stream + i * S, last); // uniform: the row's part of an address is scalar work
#pragma unroll
        for (int q = 0; q < NM; q++) {
            d[q].w = ld_at<uint4>(reinterpret_cast<const char *>(wq[q]) + ((uint32_t)(o * C) << 4), cc16);
            d[q].s = ld_at<float>(reinterpret_cast<const char *>(sc[q]) + ((uint32_t)(o * groups) << 2), g4);
            d[q].z = ld_at<int32_t>(reinterpret_cast<const char *>(zq[q]) + ((uint32_t)((o >> 3) * groups) << 2), g4);
        }
    };

    if constexpr (!DIRECT) {
        // No wave of the block asks for weights before every wave has asked for its piece of x: a CU returns
        // loads in the order it received them, and a piece of x (a cache hit) requested behind another wave's
        // first rows (HBM) would hold up the staging of the whole block until those rows are in.
        if constexpr (NW > 1) __builtin_amdgcn_s_barrier();
    }
    __builtin_amdgcn_sched_barrier(0);
    // The first half of the rows in flight now, the rest once x is staged: HBM has something to do meanwhile, and x,
    // which has to cross the same memory pipe (another XCD wrote it), does not queue behind all of it.  Half
    // was best: 7B token 1275 us, 1294 with all rows of the pair first and 1311 with none; 13B of 20 layers 1246,
    // 1264 with all.
    constexpr int PRE = (P + 1) / 2;
    RowData pipe[P][NM];
#pragma unroll
    for (int u = 0; u < PRE; u++) fetch(u, pipe[u]);
    // What the epilogues read besides the sums (residual, scatter indices): by the thread that finishes the row,
    // once, before the first tile.  A load in each tile would be a wait in front of the tile's end, and as only the
    // finishing wave would issue it, that wave's counts of younger rows would be inexact.  Thread t finishes row t
    // of the block, and the row SPAN further on where a block has more rows than threads.  Operands that are absent
    // are not read (a dummy in their place was a cold line: 7B token 1275 us with it, 1264 without).
    constexpr int SPAN = NW * 64 / TR * TR;
    const size_t out_base = (size_t)b * n_out;
    const bool has_res = !PAIR && epi_kind == Q4_EPI_RESIDUAL;
    int eo = row0 + tid;
    float res_v = 0.f;
    uint32_t sidx[3] = {0, 0, 0};
    auto epi_fetch = [&]() __attribute__((always_inline)) {
        if (eo < row1) {
            if (has_res) res_v = res[out_base + eo];
#pragma unroll
            for (int t = 0; t < 3; t++)
                if (t < n_scatter) sidx[t] = (uint32_t)sc_idx[t][eo];
        }
    };
    __builtin_amdgcn_sched_barrier(0);

    // this lane's slice of x, for good: 32 floats, or 24 digit words + step + sum of q
    float x[NM][IDOT ? 1 : 32];
    int xp[NM][IDOT ? 24 : 1];
    float sx[NM];     // fp32 form: sum of the chunk's x; integer form: sum of its q
    float xdelta[NM]; // integer form: the chunk's step
    float ss = 1.0f;
    const bool norm = !DIRECT && has_wn;
    if constexpr (DIRECT) {
        // Turned through a region of LDS of the wave's own, from "lane l holds floats 4l..4l+3 of every 256"
        // to "lane l holds its chunk's 32": no block barrier (a wave's LDS accesses execute in order).
        float *xw = lds + wave * (64 * kChunkPad);
        const int n4 = in >> 2;
#pragma unroll
        for (int i = 0; i < 8; i++) {
            const int j4 = i * 64 + lane; // float4 index within the wave's slice
            const float4 v = kslice * 512 + j4 < n4 ? xd[i] : make_float4(0.f, 0.f, 0.f, 0.f);
            *reinterpret_cast<float4 *>(&xw[(j4 >> 3) * kChunkPad + (j4 & 7) * 4]) = v;
        }
        float t = 0.f, s4[8];
#pragma unroll
        for (int i = 0; i < 8; i++) {
            const float4 v = *reinterpret_cast<const float4 *>(&xw[lane * kChunkPad + 4 * i]);
            x[0][4 * i + 0] = v.x;
            x[0][4 * i + 1] = v.y;
            x[0][4 * i + 2] = v.z;
            x[0][4 * i + 3] = v.w;
            s4[i] = (v.x + v.y) + (v.z + v.w);
            t += s4[i];
        }
        // The operator by itself (nothing in its epilogue) runs these rows through the gathering form too: the same bits then
        if (NWK == 3 && epi_kind == Q4_EPI_STORE) t = chunk_sum(s4);
        sx[0] = t;
        xdelta[0] = 0.f;
    } else {
        // stage x for the whole block, then take this lane's chunk into registers
        float ssq = 0.f;
        if (stages) {
#pragma unroll
            for (int q = 0; q < NM; q++) {
                float *xs = lds + q * xstride;
                float p = 0.f;
                if constexpr (GATHER) {
                    const int n4 = in >> 2;
#pragma unroll
                    for (int u = 0; u < NX; u++) {
                        const int j4 = u * (NW * 64) + tid;
                        if (j4 < n4) { // element 4 j4 + e of x is input gi[u].e of the sorted rows
                            xs[(gi[u].x >> 5) * kChunkPad + (gi[u].x & 31)] = xr[q].v[u].x;
                            xs[(gi[u].y >> 5) * kChunkPad + (gi[u].y & 31)] = xr[q].v[u].y;
                            xs[(gi[u].z >> 5) * kChunkPad + (gi[u].z & 31)] = xr[q].v[u].z;
                            xs[(gi[u].w >> 5) * kChunkPad + (gi[u].w & 31)] = xr[q].v[u].w;
                        }
                    }
                } else {
                    p = x_stage<NWK, NWX, NX>(norm, tid, xr[q], xs, xs + NC * kChunkPad);
                }
                if (q == 0) ssq = p;
            }
            if (norm) {
                ssq = wave_sum(ssq);
                if (lane == 0) red[wave] = ssq;
            }
        }
        __syncthreads();
        if (norm) { // rmsnorm scale, src/models.rs:55-60
            float t = 0.f;
#pragma unroll
            for (int i = 0; i < NWX; i++) t += red[i];
            t /= (float)in;
            t += eps;
            ss = 1.0f / sqrtf(t);
        }
        if constexpr (IDOT) {
#pragma unroll
            for (int q = 0; q < NM; q++) quantize_in_place<NW * 64>(lds + q * xstride, C, tid);
        }
#pragma unroll
        for (int q = 0; q < NM; q++) {
            const float *xs = lds + q * xstride;
            xdelta[q] = 0.f;
            sx[q] = 0.f;
            if constexpr (IDOT) {
                if (has_chunk) {
                    const uint4 *p = reinterpret_cast<const uint4 *>(&xs[c * kPlaneWords]);
#pragma unroll
                    for (int i = 0; i < 6; i++) {
                        const uint4 v = p[i];
                        xp[q][4 * i + 0] = (int)v.x;
                        xp[q][4 * i + 1] = (int)v.y;
                        xp[q][4 * i + 2] = (int)v.z;
                        xp[q][4 * i + 3] = (int)v.w;
                    }
                    xdelta[q] = xs[c * kPlaneWords + 24];
                    sx[q] = xs[c * kPlaneWords + 25];
                } else {
#pragma unroll
                    for (int i = 0; i < 24; i++) xp[q][i] = 0;
                }
            } else {
                if (!GATHER || has_chunk) { // the staged form has zeros in the slots past the vector's end
                    const float4 *p = reinterpret_cast<const float4 *>(&xs[c * kChunkPad]);
#pragma unroll
                    for (int i = 0; i < 8; i++) {
                        const float4 v = p[i];
                        x[q][4 * i + 0] = v.x;
                        x[q][4 * i + 1] = v.y;
                        x[q][4 * i + 2] = v.z;
                        x[q][4 * i + 3] = v.w;
                    }
                    if constexpr (GATHER) {
                        float s4[8];
#pragma unroll
                        for (int k = 0; k < 8; k++)
                            s4[k] = (x[q][4 * k] + x[q][4 * k + 1]) + (x[q][4 * k + 2] + x[q][4 * k + 3]);
                        sx[q] = chunk_sum(s4);
                    } else {
                        sx[q] = xs[NC * kChunkPad + c];
                    }
                } else {
#pragma unroll
                    for (int i = 0; i < 32; i++) x[q][i] = 0.f;
                }
            }
        }
    }

    float nsx[NM];
#pragma unroll
    for (int q = 0; q < NM; q++) nsx[q] = -sx[q];
    const int n_rows = row1 - row0;
    // Steps of the longest stream; whole tiles of P steps run in the loop, what is left runs once after it,
    // straight-line and without refills, so that the loop body stays one block (and its waits exact).
    const int n_steps = (n_rows + S - 1) / S;
    const int n_full = n_steps / P;
    const int n_rem = n_steps - n_full * P;
    int buf = 0;
    // A block that does the work of two: the rows of each half that would stand behind the loop of a block of their own.
    const int row_half = row0 + rows_per_block / 2;
    auto behind = [](int rows) { return (rows + S / 2 - 1) / (P * S / 2) * (P * S / 2); };
    const int behind0 = TWO ? behind(min(rows_per_block / 2, n_rows)) : 0, behind1 = TWO ? behind(max(row1 - row_half, 0)) : 0;
    auto is_behind = [&](int o) { return o >= row_half ? o - row_half >= behind1 : o - row0 >= behind0; };
    // The second half of the rows, and a wait for the first, which arrived while x was staged.  The compiler's wait
    // counts inside the loop are then those of the steady state alone: vmcnt leaves the P - 1 younger rows in
    // flight.  Otherwise the issue order of the prologue leaks into the loop's waits.
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int u = PRE; u < P; u++) fetch(u, pipe[u]);
    __builtin_amdgcn_sched_barrier(0);
    constexpr int YOUNGER = (P - PRE) * NM * 3;
    static_assert(YOUNGER < 64, "vmcnt");
    __builtin_amdgcn_s_waitcnt(0x0F70 | (YOUNGER & 15) | (YOUNGER >> 4) << 14); // expcnt and lgkmcnt untouched
    epi_fetch();
    float *__restrict__ const yout = mat[0].y;

    // one row (row pair) of this stream: the lane's share of its dot product, a scale times the sum of the chunk
    auto row_dot = [&](int o, const RowData(&d)[NM], Share(&p)[NM]) __attribute__((always_inline)) {
#pragma unroll
        for (int q = 0; q < NM; q++) {
            const int zn = (int)(((uint32_t)d[q].z >> (4 * (o & 7))) & 15u);
            if constexpr (IDOT)
                p[q] = {d[q].s * xdelta[q], fmaf(-(float)(zn - 7), sx[q], chunk_idot(d[q].w, xp[q]))};
            else // -(zn + 1) sx as one FMA on the converted nibble (the same real number, rounded once either way)
                p[q] = {d[q].s, fmaf(chunk_dot(d[q].w, x[q]), 512.0f, fmaf((float)zn, nsx[q], nsx[q]))};
        }
    };
    // 64 partials -> 4 (one per 16-lane row) -> the tile's slot for this row; two_lanes: the first addition has been done
    auto row_fold = [&](int u, const float(&pr)[NM], auto two_lanes) __attribute__((always_inline)) {
#pragma unroll
        for (int q = 0; q < NM; q++) {
            float v = pr[q];
            if (!two_lanes) v += dpp_xchg<0xB1>(v);
            v += dpp_xchg<0x4E>(v);
            v += dpp_xchg<0x141>(v);
            v += dpp_xchg<0x140>(v);
            if ((lane & 15) == 0) part[buf][u * S + stream][q][kslice * 4 + (lane >> 4)] = v;
        }
    };
    // one thread per row of the tile: fixed-order sum of the partials, then the epilogue
    auto tile_finish = [&](int r) __attribute__((always_inline)) {
        float sum[NM];
#pragma unroll
        for (int q = 0; q < NM; q++) {
            float a = 0.f;
#pragma unroll
            for (int k = 0; k < PW; k++) a += part[buf][r][q][k];
            sum[q] = a;
        }
        float v = sum[0] * ss;
        if (PAIR) { // silu(w1 x) * (w3 x), src/models.rs:92-98
            const float u2 = sum[NM - 1] * ss;
            v = v * (1.0f / (1.0f + expf(-v)));
            v = v * u2;
        } else if (epi_kind == Q4_EPI_RESIDUAL) {
            v = res_v + v;
        }
        if (epi_kind != Q4_EPI_SCATTER_ONLY) yout[out_base + eo] = v;
#pragma unroll
        for (int t = 0; t < 3; t++)
            if (t < n_scatter) st_at(sc_out[t], ((uint32_t)out_base + sidx[t]) << 2, v); // 32-bit offset: nothing widens the loaded index
    };

    int r = tid; // the thread's row within the tile, if 0 <= r < TR
    for (int tile = 0; tile < n_full; tile++) {
#pragma unroll
        for (int u = 0; u < P; u++) {
            const int i = tile * P + u, o = row0 + stream + i * S;
            Share p[NM];
            row_dot(o, pipe[u], p);
            float pr[NM];
#pragma unroll
            for (int q = 0; q < NM; q++) pr[q] = TWO ? p[q].two_lanes(is_behind(o)) : p[q].product();
            // Refill this slot with row i + P, after its last use and not before:
            // a load hoisted above the row's arithmetic makes the compiler copy
            // live registers of the other slots, and each copy waits on its load.
            // The empty statements pin the row's result before the loads and
            // the loads before what follows.
            if constexpr (NM == 2) asm volatile("" : "+v"(pr[0]), "+v"(pr[NM - 1])::"memory");
            else asm volatile("" : "+v"(pr[0])::"memory");
            __builtin_amdgcn_sched_barrier(0);
            fetch(i + P, pipe[u]);
            __builtin_amdgcn_sched_barrier(0);
            row_fold(u, pr, std::bool_constant<TWO>());
        }
        __syncthreads();
        if ((unsigned)r < (unsigned)TR && eo < row1) tile_finish(r);
        buf ^= 1;
        r -= TR;
        if ((tile + 1) % (SPAN / TR) == 0) { // a block of more rows than threads: the next SPAN of them
            eo += SPAN;
            r = tid;
            epi_fetch();
        }
    }
    if (n_rem > 0) { // the rows already in the pipe: no refill, nothing younger to leave in flight
#pragma unroll
        for (int u = 0; u < P - 1; u++) {
            if (u < n_rem) {
                const int o = row0 + stream + (n_full * P + u) * S;
                Share p[NM];
                row_dot(o, pipe[u], p);
                float pr[NM];
#pragma unroll
                for (int q = 0; q < NM; q++) pr[q] = p[q].two_lanes(!TWO || is_behind(o));
                row_fold(u, pr, std::true_type());
            }
        }
        __syncthreads();
        if ((unsigned)r < (unsigned)TR && eo < row1) tile_finish(r);
    }
}

static long total_rows(const Q4Launch &L) {
    long rows = 0;
    for (int i = 0; i < (L.pair ? 1 : L.n_mats); i++) rows += L.m[i].out;
    return rows;
}

// Rows per block for a block of NW waves and tiles of TR rows: a whole number of rounds over the CUs, as
// many blocks per CU as 16 waves and the LDS allow (one for a row pair); every block gets the same number of
// rows; several matrices round up separately and the grid stays within one round.
static int plan_rows(const Q4Launch &L, int NW, int TR, size_t lds, bool pair, int *total_out) {
    int per_cu = 16 / NW;
    if (pair) per_cu = 1; // w1|w3: one block per CU measured faster than two (7B: 13.1 -> 12.4 us, 722 -> 733 tok/s)
    if (per_cu < 1) per_cu = 1;
    const int by_lds = (int)((150 * 1024) / (lds + 4 * 1024));
    if (per_cu > by_lds) per_cu = by_lds < 1 ? 1 : by_lds;
    const int nm = pair ? 1 : L.n_mats;
    const long rows = total_rows(L);
    const long slots = (long)cu_count() * per_cu;
    int rpb = (int)((rows + slots - 1) / slots);
    if (rpb < TR) rpb = TR;
    int total = 0;
    for (;;) {
        total = 0;
        for (int i = 0; i < nm; i++) total += (L.m[i].out + rpb - 1) / rpb;
        if (total <= slots || rpb >= rows) break;
        rpb++;
    }
    if (total_out) *total_out = total;
    return rpb;
}

static size_t staging_lds(int NWK, bool pair) { return (size_t)NWK * 64 * (kChunkPad + 1) * sizeof(float) * (pair ? 2 : 1); }

// Whether a launch in blocks of S streams with P rows in flight has no rows behind the loop (whose last bit is another).
static bool whole_tiles(const Q4Launch &L, int NWK, int S, int P) {
    const int rpb = plan_rows(L, NWK * S, P * S, staging_lds(NWK, false), false, nullptr);
    for (int i = 0; i < L.n_mats; i++) {
        const int out = L.m[i].out, last = out - (out - 1) / rpb * rpb;
        if ((last + S - 1) / S % P || (out > rpb && (rpb + S - 1) / S % P)) return false;
    }
    return true;
}

// Whether two blocks of eight waves (rows of two) run as one of sixteen.  A CU returns loads in the order it received them, so of two
// blocks on a CU the second has its x behind the first rows of the other's weights: with time stamps in 7B's q|k|v the one had x
// staged 1.2 us after the launch and was through at 5.2, the other at 2.3 and 6.4.  In one block all of x is asked for in front of all
// weights: 8 layers of 7B, a token 378 -> 371 us, q|k|v 4.2 of them, wo 1.8.  So where CUs would get two of them; not for several
// columns, which are more blocks than a CU holds at once.  A row is the same bits either way: the sum of squares is taken by eight
// waves, and the rows that stand behind the loop in a block of eight waves keep that rounding.
static bool two_in_one(const Q4Launch &L) {
    if (L.batch != 1 || (!L.m[0].wn && L.e.kind != Q4_EPI_RESIDUAL)) return false;
    int total = 0, halves = 0;
    const int rpb = plan_rows(L, 8, 8, staging_lds(2, false), false, &total);
    for (int i = 0; i < L.n_mats; i++) halves += (L.m[i].out + 2 * rpb - 1) / (2 * rpb);
    return total > cu_count() && halves <= cu_count();
}

template <int G, int NWK, int S, bool PAIR, int MODE, int P = (PAIR ? 2 : 4), bool GATHER = false>
int launch_s(Q4Launch &L, hipStream_t stream) {
    constexpr int NW = NWK * S;
    constexpr int TR = P * S;
    constexpr bool TWO = MODE == 3;
    const size_t lds = MODE == 2 ? (size_t)NW * 64 * kChunkPad * sizeof(float)
                                 : staging_lds(NWK, PAIR);
    if (lds + 8 * 1024 > 160 * 1024) return l2_fail(L2_ERR_ARG, "q4 matvec: in=%d needs %zu B of LDS", L.in, lds);
    int total = 0;
    const int rpb = TWO ? 2 * plan_rows(L, NW / 2, TR / 2, lds, PAIR, nullptr) : plan_rows(L, NW, TR, lds, PAIR, &total);
    if (TWO)
        for (int i = 0; i < L.n_mats; i++) total += (L.m[i].out + rpb - 1) / rpb;
    L.rows_per_block = rpb;
    for (int i = 0; i < L.n_mats; i++) L.m[i].row_blocks = (L.m[i].out + rpb - 1) / rpb;
    auto kern = q4_stream_kernel<G, NWK, S, PAIR, MODE, P, GATHER>;
    if (g_q4_name.armed) {
        g_q4_name.armed = false;
        snprintf(g_q4_name.buf, (size_t)g_q4_name.cap, "q4_stream_kernel<%d, %d, %d, %s, %d, %d, %s>", G, NWK, S,
                 PAIR ? "true" : "false", MODE, P, GATHER ? "true" : "false");
        g_q4_name.grid = total, g_q4_name.block = NW * 64, g_q4_name.rows_per_block = rpb, g_q4_name.lds = lds;
        if (MODE != 1) g_q4_name.rows = {TWO ? rpb / 2 : rpb, TWO ? TR / 2 : TR, TWO ? S / 2 : S, TWO ? NW / 2 : NW, MODE == 2};
        return L2_OK;
    }
    if (lds > 48 * 1024) {
        static LdsLimit limit; // per instantiation
        L2_TRY(limit.ensure(reinterpret_cast<const void *>(kern), lds));
    }
    for (int i = 1; i < L.n_mats; i++) // the kernel finds them behind those of the first
        if (L.m[i].wn != (L.m[0].wn ? L.m[0].wn + (size_t)i * L.in : nullptr)) return l2_fail(L2_ERR_ARG, "q4 matvec: norm weights apart");
    dim3 grid(total, L.batch), block(NW * 64);
    StreamArgs a{};
    for (int i = 0; i < L.n_mats; i++) a.m[i] = {L.m[i].qweight, L.m[i].qzeros, L.m[i].scales, L.m[i].y, L.m[i].out};
    a.e = L.e, a.groups = L.groups, a.rows_per_block = rpb, a.eps = L.eps;
    const Q4Mat *const m = L.m;
    if (g_q4_prof.armed) {
        g_q4_prof.armed = false;
        hipExtLaunchKernelGGL(kern, grid, block, lds, stream, g_q4_prof.start, g_q4_prof.stop, 0, m[0].x, m[1].x, m[2].x, m[0].wn, m[0].gidx, L.in,
                              m[0].row_blocks, m[1].row_blocks, a);
    } else {
        l2_launch(kern, grid, block, lds, stream, m[0].x, m[1].x, m[2].x, m[0].wn, m[0].gidx, L.in, m[0].row_blocks, m[1].row_blocks, a);
    }
    L2_HIP(hipGetLastError());
    return L2_OK;
}

// Rows in flight per stream (P) and streams per block (S) were measured per shape on whole decode steps.  Where the rows of a
// block are few (4096 and 11008 inputs: 4 to 8 rows per stream), fewer loads primed in front of x let x arrive sooner,
// and every instruction of the kernel waits for x: two rows at 4096 inputs (7B +1.2 %), three at 11008 (+0.9 %); priming all
// rows of the block is 15-20 % slower.  Blocks have a whole number of waves per SIMD: with 12 waves instead of 15 at 5120 inputs
// 13B's w1|w3 takes 17.3 us instead of 22.5 (9 waves 23.6, 6 waves 23.3) and wo 6.4 instead of 7.0.  16 waves with one pair of rows
// in flight against 8 with two at 8192 inputs: 70B's w1|w3 43.9 -> 42.6 (12 waves with one or two pairs 46.8, 44.1).
// 28672 -> 8192, two, three, four, five, six rows: 27.6 / 24.8 / 25.7 / 26.2 / 26.7 us; 13824 -> 5120, two rows or three: 11.0, 11.1.
//
// Few rows: a tile of P rows per stream is the least a block takes, so with the shapes above 1024 rows are 64 to 128 blocks, and
// a launch is as long as the serial work of one of them.  With one row in flight per stream (and, at up to 2048 inputs, eight
// streams) every CU has a block and a stream a row or two.  Cadence of the operator, before -> with the shape for few rows, us:
// 1024 inputs, 1024 rows 3.37 -> 3.24, 4096 rows 3.50, 3.68 (not taken); 4096 inputs, 1024 rows 3.45 -> 3.20, 1536 rows 3.55,
// 4.05 (not taken); 8192 inputs, 1024 rows 4.26 -> 3.98, 1536 rows 4.35, 4.70 (not taken).  The small model (1024 inputs, 2816
// hidden, three layers), per token 74.5 -> 69.5.
// Row pairs at up to 2048 inputs: eight streams of two pairs, 2048 -> 2 x 8192 87.3 -> 83.2 us per token of three layers.
//
// The gathering form has more to stage (x and where each of its elements goes) and nothing behind the sums, so it gains from more
// waves per block: 4096 inputs in one block of 16 waves per CU instead of two of 8, two rows in flight: 4096 rows 4.70 -> 4.35 us,
// 11008 rows 7.43 -> 6.76, 2048 rows 3.65, 4.02 (not taken); as a projection of the model the same shape loses (7B 287 -> 289 us
// per 8 layers); and several columns are more blocks than a CU holds at once, of which two of 8 waves overlap and one of 16 does not
// (4096 rows, 8, 16, 48 columns on host arrays 44.4 / 72.4 / 175 us, with 16 waves 47.7 / 79.5 / 198).  5120 inputs: two rows in flight up to 8192 rows, three beyond, instead of four: 1024 rows 4.65 -> 3.76, 5120 rows
// 5.79 -> 5.54, 13824 rows 10.05 -> 9.81.
//
// The rows here are those of all columns, so one column may take another shape than several of the same matrix, and the form
// without the gathering another than the one with it.  So that a column is the same bits all the same, the shapes of one matrix
// differ only where none of them has rows behind its loop: that is asked, or holds wherever the rows are whole eights (4096 inputs up
// to 1024 rows).  Up to 2048 inputs a matrix whose last block has eight rows (1032 of them) keeps four streams of four rows.
template <int G, int MODE>
int launch_sg(Q4Launch &L, hipStream_t stream) {
    const int nwk = (L.in / 32 + 63) / 64;
    const long rows = total_rows(L) * L.batch, cus = cu_count(); // every column has blocks of its own
    if constexpr (MODE == 2) { // only the shapes q4_stream_launch sends here
        if (!L.pair) switch (nwk) {
            case 3: return launch_s<G, 3, 4, false, MODE>(L, stream);
            case 7: return launch_s<G, 7, 2, false, MODE, 2>(L, stream);
            case 9: case 10: case 11: case 12: case 13: case 14: return launch_s<G, 14, 1, false, MODE, 3>(L, stream);
        }
    } else if (MODE == 0 && !L.pair && L.n_mats == 1 && L.m[0].gidx) {
        if constexpr (MODE == 0) switch (nwk) { // the gathering form, where one staging batch covers the vector
            case 1: return rows <= 8 * cus && whole_tiles(L, 1, 4, 4) ? launch_s<G, 1, 8, false, 0, 1, true>(L, stream) : launch_s<G, 1, 4, false, 0, 4, true>(L, stream);
            case 2:
                if (rows <= 4 * cus) return launch_s<G, 2, 4, false, 0, 1, true>(L, stream);
                if (L.batch <= 2 && rows > 8 * cus && whole_tiles(L, 2, 4, 2) && whole_tiles(L, 2, 8, 2)) return launch_s<G, 2, 8, false, 0, 2, true>(L, stream);
                return launch_s<G, 2, 4, false, 0, 2, true>(L, stream);
            case 3:
                if (rows <= 32 * cus && whole_tiles(L, 3, 4, 4) && whole_tiles(L, 3, 4, 2)) return launch_s<G, 3, 4, false, 0, 2, true>(L, stream);
                if (rows > 32 * cus && whole_tiles(L, 3, 4, 4) && whole_tiles(L, 3, 4, 3)) return launch_s<G, 3, 4, false, 0, 3, true>(L, stream);
                return launch_s<G, 3, 4, false, 0, 4, true>(L, stream);
            case 4: return rows <= 4 * cus && whole_tiles(L, 4, 4, 2) ? launch_s<G, 4, 4, false, 0, 1, true>(L, stream) : launch_s<G, 4, 4, false, 0, 2, true>(L, stream);
        }
    } else if (!L.pair) {
        switch (nwk) {
            case 1: return rows <= 8 * cus && whole_tiles(L, 1, 4, 4) ? launch_s<G, 1, 8, false, MODE, 1>(L, stream) : launch_s<G, 1, 4, false, MODE>(L, stream);
            case 2:
                if (rows <= 4 * cus) return launch_s<G, 2, 4, false, MODE, 1>(L, stream);
                if constexpr (MODE == 0)
                    if (two_in_one(L)) return launch_s<G, 2, 8, false, 3, 2>(L, stream);
                return launch_s<G, 2, 4, false, MODE, 2>(L, stream);
            case 3: return launch_s<G, 3, 4, false, MODE>(L, stream);
            case 4: return launch_s<G, 4, 4, false, MODE, 2>(L, stream); // 8192: rows of 4 KB; two in flight per stream measured faster than four (q|k|v 13.4 -> 12.2 us, wo 12.1 -> 10.9)
            case 5: case 6: return launch_s<G, 6, 2, false, MODE, 3>(L, stream);
            case 7: return launch_s<G, 7, 2, false, MODE, 5>(L, stream); // 13824 -> 5120: 20 rows per block in two tiles
            case 8: return launch_s<G, 8, 2, false, MODE>(L, stream);
            case 9: case 10: case 11: case 12: case 13: case 14: return launch_s<G, 14, 1, false, MODE>(L, stream);
        }
    } else {
        switch (nwk) {
            case 1: return launch_s<G, 1, 8, true, MODE, 2>(L, stream);
            case 2: return launch_s<G, 2, 4, true, MODE>(L, stream);
            case 3: return launch_s<G, 3, 4, true, MODE>(L, stream);
            case 4: return launch_s<G, 4, 4, true, MODE, 1>(L, stream);
        }
    }
    return l2_fail(L2_ERR_ARG, "q4 matvec (streaming): in=%d pair=%d has no kernel", L.in, L.pair);
}

} // namespace

int q4_stream_launch(Q4Launch &L, hipStream_t stream) {
    // L2_Q4_IMPL=idot selects the integer-dot form of the inner loop; the default is the fp32 form.
    static const bool fp32_form = []() {
        const char *v = getenv("L2_Q4_IMPL");
        return !(v && !strcmp(v, "idot"));
    }();
    // One matrix and no rmsnorm in front: x can reach the registers through LDS of each wave's own instead
    // of a block-wide staging with a barrier.  Measured per input width (cadence of the launch, block-wide
    // against per-wave): 28672: 30.3 -> 28.6 us; 13824: 14.2 -> 13.2; 5120: 9.0 -> 7.7; but 11008: 9.0 -> 9.5,
    // 8192: 11.6 -> 12.3, 4096 equal within the model.  The per-wave form is taken where it won: 3 and 7 waves
    // per row, and inputs too long to stage block-wide beside a second block.
    const int nwk = (L.in / 32 + 63) / 64;
    const bool direct = fp32_form && !L.pair && L.n_mats == 1 && L.m[0].wn == nullptr && L.m[0].gidx == nullptr &&
                        (L.in > 16384 || nwk == 3 || nwk == 7);
    if (direct) {
        switch (L.group_size) {
            case 32: return launch_sg<32, 2>(L, stream);
            case 64: return launch_sg<64, 2>(L, stream);
            case 128: return launch_sg<128, 2>(L, stream);
        }
    } else if (fp32_form) {
        switch (L.group_size) {
            case 32: return launch_sg<32, 0>(L, stream);
            case 64: return launch_sg<64, 0>(L, stream);
            case 128: return launch_sg<128, 0>(L, stream);
        }
    } else {
        switch (L.group_size) {
            case 32: return launch_sg<32, 1>(L, stream);
            case 64: return launch_sg<64, 1>(L, stream);
            case 128: return launch_sg<128, 1>(L, stream);
        }
    }
    return l2_fail(L2_ERR_ARG, "q4 matvec: group size %d (32, 64 or 128)", L.group_size);
}

static bool fp32_stream_form() {
    static const bool yes = []() {
        const char *v = getenv("L2_Q4_IMPL");
        return !(v && (!strcmp(v, "idot") || !strcmp(v, "tile")));
    }();
    return yes;
}

bool q4_gathers_in_kernel(const Q4Launch &L) {
    const int nwk = (L.in / 32 + 63) / 64;
    return fp32_stream_form() && !L.pair && L.n_mats == 1 && L.m[0].wn == nullptr && nwk <= 4 && L.in % 4 == 0 &&
           q4_stream_supports(L);
}

bool q4_stream_supports(const Q4Launch &L) {
    const int nwk = (L.in / 32 + 63) / 64;
    // the kernel addresses a matrix with 32-bit byte offsets and 24-bit row numbers
    for (int i = 0; i < L.n_mats; i++)
        if (L.m[i].out >= (1 << 24) || (size_t)L.m[i].out * (size_t)(L.in / 8) * 4 >= ((size_t)1 << 32)) return false;
    return L.pair ? nwk <= 4 : nwk <= 14;
}
