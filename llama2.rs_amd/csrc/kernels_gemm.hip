// QLinear::matvec<B> (src/gptq.rs:94-176) for a batch of columns on the matrix cores of gfx950 in fp32, the kernels that
// stand between two such products of a chunk, and the choice of how a product is cut (the fp16 product of the prefill
// mode L2_PREFILL_MFMA is in kernels_q4_gemm.hip).
//
//   Y[t][o] = sum_g s[o][g] * sum_{k in g} (nib(qweight[o],k) - z1[o][g]) X[t][k]
//
// fp32 activations, exactly: x = b0 + b1 + b2 with three bf16 numbers of 8 significant bits each, obtained by cutting x
// after its first, second and third byte of significand (all of x from 2^-109 on; below, what is under bf16's smallest number,
// 2^-133, is cut off).  The weights are integers n - z1 of at most five bits, exact in
// bf16, and so is every product that enters the fp32 accumulator (v_mfma_f32_16x16x32_bf16).  What is left is the sums:
//   - The matrix unit's sum of products and accumulator is not rounded to nearest; it comes out too small on average, whatever
//     its sign.  So every other group enters negated, weights and scale: the mean is below 1e-9.
//   - Of the three planes of a step the smallest is added first.
//   - The fp32 group scale is applied to the fp32 sum of each group, and these are added in runs of 8 to 16 groups, the runs to
//     each other, the slices of K in a tree: the error of a chain grows with its length.
// Relative rms error against fp64 over 1024..28672 inputs, 8..512 columns, of that of the matvec (kernels_q4_stream.hip): normal
// inputs 0.45 to 0.74, inputs all of one sign, where the matvec is better than elsewhere, 0.39 to 1.06 (1024 inputs, group 128).
//
// Against the matvec kernels run once per column, which read and dequantise the weights for each of them: 4096x11008,
// group 32, 61 columns 330 -> 30.2 us with everything around it.  Against the form before this one (activations and weights
// through registers, 32x32x16 tiles, two blocks of four waves per CU): that call 40.3 us; 16 columns of 13824x5120 33.7 -> 22.6;
// two layers of 7B, group 128, 16, 64, 299 columns 280 / 365 / 967 -> 222 / 328 / 930; 70B, group 64, 16 and 299 763 / 3593 ->
// 544 / 3350.
#include <algorithm>

#include "gemm_lds.h"

namespace {

typedef _Float16 h2 __attribute__((ext_vector_type(2)));
typedef _Float16 h8 __attribute__((ext_vector_type(8)));
typedef __bf16 b8 __attribute__((ext_vector_type(8)));
typedef __bf16 b2 __attribute__((ext_vector_type(2)));
typedef float v2f __attribute__((ext_vector_type(2)));

union Frag {
    uint4 q;
    uint32_t u[4];
    h8 h;
    b8 b;
    h2 p[4];
};

template <class T>
__device__ __forceinline__ T ld_at(const void *base, uint32_t byte_offset) {
    return *reinterpret_cast<const T *>(reinterpret_cast<const char *>(base) + byte_offset);
}

// bf16: sign (n - z1) in the order (0,2,4,6,1,3,5,7).  A nibble in the low half of a byte is n 2^-9 as an OCP E4M3 number; two
// at a time become fp32, one FMA each makes sign (n - z1) of it, and the upper halves of two results are the bf16 pair (the
// integers have at most five bits: nothing is cut off).
struct Dequant {
    float unit, z; // +-2^9, -+z1
    __device__ __forceinline__ void set(int zn, float sign) { unit = 512.0f * sign, z = (float)(zn + 1) * -sign; }
    // pair i of a word; i = 2 and 3 of the word shifted by 4
    __device__ __forceinline__ uint32_t pair(uint32_t masked, int i) const {
        const v2f v = i % 2 == 0 ? __builtin_amdgcn_cvt_pk_f32_fp8(masked, false) : __builtin_amdgcn_cvt_pk_f32_fp8(masked, true);
        return __builtin_amdgcn_perm(__builtin_bit_cast(uint32_t, fmaf(v.y, unit, z)), __builtin_bit_cast(uint32_t, fmaf(v.x, unit, z)), 0x07060302u);
    }
};

// ---- activations -------------------------------------------------------------------------------------------------

// Eight consecutive inputs of one token, as the GEMM's LDS tile wants them: NP planes of 16 bytes.
template <int NP>
struct Piece {
    uint4 q[NP];
};

template <int NP>
__device__ __forceinline__ Piece<NP> make_piece(const float (&v)[8]) {
    Piece<NP> r;
    if constexpr (NP == 1) {
        Frag f;
        f.p[0] = h2{(_Float16)v[0], (_Float16)v[4]};
        f.p[1] = h2{(_Float16)v[1], (_Float16)v[5]};
        f.p[2] = h2{(_Float16)v[2], (_Float16)v[6]};
        f.p[3] = h2{(_Float16)v[3], (_Float16)v[7]};
        r.q[0] = f.q;
    } else {
        constexpr int order[8] = {0, 2, 4, 6, 1, 3, 5, 7};
        uint32_t t[8];
#pragma unroll
        for (int e = 0; e < 8; e++) t[e] = __builtin_bit_cast(uint32_t, v[order[e]]);
#pragma unroll
        for (int p = 0; p < NP; p++) {
            Frag f;
#pragma unroll
            for (int i = 0; i < 4; i++) f.u[i] = __builtin_amdgcn_perm(t[2 * i + 1], t[2 * i], 0x07060302u);
            r.q[p] = f.q;
#pragma unroll
            for (int e = 0; e < 8; e++) // what the plane leaves over: exact
                t[e] = __builtin_bit_cast(uint32_t, __builtin_bit_cast(float, t[e]) - __builtin_bit_cast(float, t[e] & 0xFFFF0000u));
        }
    }
    return r;
}

// Plane p of token t: [t][p][in_p], in_p = the row padded to whole K steps.
template <int NP>
__device__ __forceinline__ void store_piece(void *out, size_t t, int in_p, int j8, const Piece<NP> &r) {
    uint4 *dst = reinterpret_cast<uint4 *>(reinterpret_cast<uint16_t *>(out) + t * NP * in_p);
#pragma unroll
    for (int p = 0; p < NP; p++) store_through(&dst[p * (in_p >> 3) + j8], r.q[p]);
}

// x[b][g_index[j]] -> planes: the gather of src/gptq.rs:110-114.  grid (pieces / 256, B, consumers).
template <int NP>
__global__ __launch_bounds__(256) void gemm_input_kernel(const GemmInput A, int n, int in_p) {
    const int b = blockIdx.y, c = blockIdx.z;
    const int j8 = blockIdx.x * 256 + threadIdx.x;
    if (j8 * 8 >= in_p) return;
    const float *x = A.x + (size_t)b * n;
    float v[8];
    if (j8 * 8 < n && !A.g_index[c]) { // no act-order: the model without quantisation
        const float4_any a = reinterpret_cast<const float4_any *>(x)[2 * j8], b4 = reinterpret_cast<const float4_any *>(x)[2 * j8 + 1];
        v[0] = a.x, v[1] = a.y, v[2] = a.z, v[3] = a.w, v[4] = b4.x, v[5] = b4.y, v[6] = b4.z, v[7] = b4.w;
#pragma unroll
        for (int e = 0; e < 8; e++) v[e] = __builtin_canonicalizef(v[e]); // a signalling NaN's first plane could be an infinity (dense_again)
    } else if (j8 * 8 < n) {
        const int4 g0 = reinterpret_cast<const int4 *>(A.g_index[c])[2 * j8], g1 = reinterpret_cast<const int4 *>(A.g_index[c])[2 * j8 + 1];
        const int g[8] = {g0.x, g0.y, g0.z, g0.w, g1.x, g1.y, g1.z, g1.w};
#pragma unroll
        for (int e = 0; e < 8; e++) v[e] = x[g[e]];
    } else {
#pragma unroll
        for (int e = 0; e < 8; e++) v[e] = 0.f;
    }
    store_piece<NP>(A.out[c], b, in_p, j8, make_piece<NP>(v));
}

// The same from x as the host has left it, in pinned memory or, from kWindowBytes (host.cpp) on, in device memory: read in order, 16 bytes per
// thread and load, and scattered to its places, so that every element crosses the bus once where it has to.  NP = 0: fp32, for the
// matvec kernels.  From device memory 6.8 us for the 0.9 MB of 16 columns of 13824 inputs.  From pinned memory what bounds it is the bus (48 GB/s, 18 us
// for the same; the scattered stores take a third of that, behind it), so a long x is launched for in two parts, one while the host
// brings the other.  A DMA engine reads at 65 GB/s, but a kernel behind a DMA starts 10 us late.
// With a column per block, read into LDS and permuted there, one compute unit's reads are the bound: one column of 28672 inputs
// 32.8 -> 39.3 us for the call, from pinned memory.
constexpr int kHostPieces = 2; // of 16 bytes per thread (four: 84 us for 16 columns of 13824x5120 from pinned memory, two 82)
template <int NP>
__global__ __launch_bounds__(256) void host_input_kernel(void *__restrict__ out, const float *__restrict__ x,
                                                         const int32_t *__restrict__ inv, int n, int in_p) {
    const int b = blockIdx.y, i0 = blockIdx.x * kHostPieces * 256 + threadIdx.x, n4 = n >> 2;
    const float4 *src = reinterpret_cast<const float4 *>(x + (size_t)b * n);
    float4 v[kHostPieces];
    int4 to[kHostPieces];
#pragma unroll
    for (int u = 0; u < kHostPieces; u++) {
        const int i = min(i0 + u * 256, n4 - 1); // past the end: the last piece again
        v[u] = src[i];
        to[u] = reinterpret_cast<const int4 *>(inv)[i];
    }
#pragma unroll
    for (int u = 0; u < kHostPieces; u++) {
        const float e[4] = {v[u].x, v[u].y, v[u].z, v[u].w};
        const int j[4] = {to[u].x, to[u].y, to[u].z, to[u].w};
#pragma unroll
        for (int k = 0; k < 4; k++) {
            if constexpr (NP == 0) {
                reinterpret_cast<float *>(out)[(size_t)b * n + j[k]] = e[k];
            } else if constexpr (NP == 1) {
                reinterpret_cast<_Float16 *>(out)[(size_t)b * in_p + h16_slot(j[k])] = (_Float16)e[k];
            } else {
                uint16_t *o = reinterpret_cast<uint16_t *>(out) + (size_t)b * NP * in_p + b16_slot(j[k]);
                float left = e[k];
#pragma unroll
                for (int p = 0; p < NP; p++) { // as make_piece cuts it
                    const uint32_t bits = __builtin_bit_cast(uint32_t, left) & 0xFFFF0000u;
                    o[(size_t)p * in_p] = (uint16_t)(bits >> 16);
                    left -= __builtin_bit_cast(float, bits);
                }
            }
        }
    }
    if (NP > 0 && n + i0 < in_p && i0 < 64) // the rest of the row's last K step
#pragma unroll
        for (int p = 0; p < NP; p++) reinterpret_cast<uint16_t *>(out)[((size_t)b * NP + p) * in_p + n + i0] = 0;
}

// ---- the GEMM ----------------------------------------------------------------------------------------------------

// Four consecutive outputs of column t: a partial tile of this K slice, or the result through the launch's epilogue.
__device__ __forceinline__ void finish4(const Q4Launch &L, int mi, const float *ss, float *ws, int KS, int ks, int partials,
                                        int t, int o, float4 v, int B) {
    const int n_out = L.m[mi].out;
    if (KS > 1 || partials) {
        store_through(reinterpret_cast<float4 *>(ws + ((size_t)ks * B + t) * n_out + o), v);
        return;
    }
    const float sc = ss ? ss[t] : 1.0f;
    v.x *= sc, v.y *= sc, v.z *= sc, v.w *= sc;
    const size_t at = (size_t)t * n_out + o;
    if (L.e.kind == Q4_EPI_RESIDUAL) {
        const float4 rr = *reinterpret_cast<const float4 *>(L.e.res + at);
        v.x += rr.x, v.y += rr.y, v.z += rr.z, v.w += rr.w;
    }
    *reinterpret_cast<float4_any *>(L.m[mi].y + at) = float4_any{v.x, v.y, v.z, v.w};
}

// LDS of a block of NW waves: three activation tiles of 64 k (three planes of 16 NT tokens), and for each wave three units of
// 128 k of its 32 rows' weights, scales and zero points.
template <int G, int NT, int NW>
struct TileLds {
    static constexpr int kPlane = 16 * NT * kStepRow, kTile = 3 * kPlane;
    static constexpr int kGroupLoads = G == 32 ? 2 : 1; // of 64 scales (zero points) per unit
    static constexpr int kWeights = 32 * 64, kScales = 256 * kGroupLoads;
    static constexpr int kUnit = kWeights + 2 * kScales;
    static constexpr size_t kSize = 3 * (size_t)kTile + (size_t)NW * 3 * kUnit;
};

// A wave owns 32 rows x 16 NT tokens, in tiles of 16 x 16 (v_mfma_f32_16x16x32_bf16); a block is NW waves side by side over the
// rows, on the same tokens.  What the K loop reads comes through LDS past the registers, as in the fp16 kernel
// (kernels_q4_gemm.hip, which explains the layout and the waits): tiles of 64 k two steps ahead, weights two units.  One
// barrier per step; a step is 6 NT pairs of MFMAs, with the dequantisation of the next one's weights and the folds of finished
// groups spread between them: some 230 instructions for 64 tokens, which the two waves of a SIMD issue at one per 4.9 cycles
// (2546 cycles per step of 7B's w1|w3 at 299 tokens before the scales and zero points came in tiles, 1536 of them MFMAs; what a
// SIMD can issue is 1624, the rest are waits).  Eight waves and 64 tokens take 133 KB of LDS, one
// block per CU, and 80 tokens (not with groups of 32) 154; four waves and 16 or 32 tokens, where weights are what is read, two or three.
//
// Lane (r = l % 16, kg = l / 16).  G >= 64: the lane's words of a step are 2 kg and 2 kg + 1, MFMA k takes one each.  G = 32: an
// MFMA must stay inside one group, so its words are kg and 4 + kg.
template <int G, int NT, int NW>
__device__ __forceinline__ void q4_tile(const Q4Launch &L, const XhList &xl, int in_p, const float *__restrict__ ss, float *__restrict__ ws,
                                        int KS, int partials, int rb, int ks, int t0, int B) {
    using S = TileLds<G, NT, NW>;
    constexpr int NP = 3, TN = 16 * NT, RB = 32 * NW;
    constexpr int KPG = G >= 64 ? G / 64 : 1; // K steps per group
    constexpr int GPS = G >= 64 ? 1 : 64 / G; // groups per K step
    extern __shared__ __align__(16) char lds[];
    int mi = 0;
    while (mi + 1 < L.n_mats && rb >= L.m[mi].row_blocks) {
        rb -= L.m[mi].row_blocks;
        mi++;
    }
    const int n_out = L.m[mi].out, groups = L.groups, in = L.in;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int r = lane & 15, kg = lane >> 4;
    const int obase = rb * RB + wave * 32;
    // this block's slice of K, in whole groups and whole K steps
    const int n_unit = in_p / (64 * KPG);
    const int it0 = (int)((long)n_unit * ks / KS) * KPG, it1 = (int)((long)n_unit * (ks + 1) / KS) * KPG, n_it = it1 - it0;

    const int row_tiles = (n_out + 31) >> 5; // of scales and zero points
    const uint32_t lds0 = lds_offset(lds), wave_at = 3 * S::kTile + wave * 3 * S::kUnit;
    const u4v xbuf = biased_buffer(xl.p[mi], (size_t)B * NP * in_p * 2), wbuf = biased_buffer(L.m[mi].qweight, (size_t)n_out * (in >> 1));
    const u4v sbuf = biased_buffer(L.m[mi].scales, (size_t)row_tiles * groups * 128), zbuf = biased_buffer(L.m[mi].qzeros, (size_t)row_tiles * groups * 16);
    constexpr int PIECES = NP * 2 * NT, XP = (PIECES + NW - 1) / NW; // 1 KB pieces of a tile: 8 tokens of a plane
    static_assert(XP <= 4, "the instruction's own offset has 12 bits");
    const int xfirst = min(wave * XP, PIECES - XP);
    uint32_t xoff[XP], woff[2];
#pragma unroll
    for (int i = 0; i < XP; i++) {
        const int p = (xfirst + i) / (2 * NT), t = (xfirst + i) % (2 * NT) * 8 + (lane >> 3);
        xoff[i] = ((uint32_t)min(t0 + t, B - 1) * NP + p) * (uint32_t)in_p * 2u + (((lane & 7) ^ piece_xor(t)) << 4) + kBias - i * 1024;
    }
#pragma unroll
    for (int i = 0; i < 2; i++) {
        const int row = i * 16 + (lane >> 2);
        woff[i] = (uint32_t)min(obase + row, n_out - 1) * (uint32_t)(in >> 1) + (((lane & 3) ^ ((row >> 2) & 3)) << 4) + kBias - i * 1024;
    }
    const int lane_group = G == 128 ? 0 : lane >> 5;
    const uint32_t group0 = (uint32_t)(min(obase >> 5, row_tiles - 1) * groups);
    const uint32_t soff = group0 * 128u + (lane & 31) * 4u + kBias - S::kWeights, zoff = group0 * 16u + (lane >> 3 & 3) * 4u + kBias - S::kWeights - S::kScales;
    uint32_t xr[2]; // where the lane reads a token's piece of MFMA k
#pragma unroll
    for (int k = 0; k < 2; k++) xr[k] = (uint32_t)r * kStepRow + (((G == 32 ? 4 * k + kg : 2 * kg + k) ^ piece_xor(r)) << 4);
    // ... and its words of a unit's first step (the second's: ^ 32)
    const int wsw = (r >> 2) & 3;
    const uint32_t wr0 = wave_at + r * 64 + (G == 32 ? (wsw << 4) + kg * 4 : (((kg >> 1) ^ wsw) << 4) + (kg & 1) * 8);
    const uint32_t sr = wave_at + S::kWeights + kg * 16, zr = wave_at + S::kWeights + S::kScales + r * 4;
    const int zsh = 4 * (r & 7);

    const uint32_t x_last = (uint32_t)(it1 - 1) * 128;
    uint32_t x_at = (uint32_t)it0 * 128, w_at = (uint32_t)it0 * 32; // what is requested next (requests past the slice's end are never read)
    auto fetch_x = [&](uint32_t tile, const int i) __attribute__((always_inline)) {
        LDS_LOAD("x4", lds0 + tile + xfirst * 1024, i * 1024, xbuf, xoff[i], x_at);
        if (i == XP - 1) x_at = min(x_at + 128, x_last);
    };
    constexpr int WL = 2 + 2 * S::kGroupLoads;
    auto fetch_w = [&](uint32_t unit, const int i) __attribute__((always_inline)) {
        const uint32_t to = lds0 + wave_at + unit;
        if (i < 2) {
            LDS_LOAD("x4", to, i * 1024, wbuf, woff[i], w_at);
        } else { // in % 64 = 32: the last step's second group is the first one again (its inputs are zero)
            const uint32_t g = min(w_at * 2 / G + lane_group + (i >= 4 ? 2 : 0), (uint32_t)groups - 1) * 128, z = g >> 3;
            if (i == 2) LDS_LOAD("", to, S::kWeights, sbuf, soff + g, 0);
            else if (i == 3) LDS_LOAD("", to, S::kWeights + S::kScales, zbuf, zoff + z, 0);
            else if (i == 4) LDS_LOAD("", to, S::kWeights + 256, sbuf, soff - 256 + g, 0);
            else LDS_LOAD("", to, S::kWeights + S::kScales + 256, zbuf, zoff - 256 + z, 0);
        }
        if (i == WL - 1) w_at += 64;
    };

    f4v top[NT][2], acc[NT][2], accg[NT][2]; // sums of the runs, of the current run, of the current group; two tiles of 16 rows
#pragma unroll
    for (int n = 0; n < NT; n++)
#pragma unroll
        for (int m = 0; m < 2; m++) top[n][m] = acc[n][m] = accg[n][m] = f4v{0.f, 0.f, 0.f, 0.f};
    f4v sv[GPS][2]; // scales of the group(s) that accg holds
#pragma unroll
    for (int g = 0; g < GPS; g++) sv[g][0] = sv[g][1] = f4v{0.f, 0.f, 0.f, 0.f};
    float sign = 1.0f; // G = 128: of this unit's group (every other group enters negated, weights and scale)
    auto negated = [](int par, int k) { return G == 32 ? k == 1 : G == 64 && par == 1; };

    Dequant dq[GPS][2];
    Frag aq[2][2][2]; // weights of this step and the next: [rows][k]
    uint32_t wd[2][2]; // packed weights of the next step
    int zw[GPS][2];
    Frag bq[4][NP];    // activations of four tiles of tokens
    auto read_w = [&](const int par, uint32_t unit) __attribute__((always_inline)) {
#pragma unroll
        for (int m = 0; m < 2; m++) {
            if constexpr (G == 32) {
#pragma unroll
                for (int k = 0; k < 2; k++) // piece 2 par + k of the row
                    wd[m][k] = *reinterpret_cast<const uint32_t *>(lds + (wr0 ^ ((2 * par + k) * 16)) + unit + m * 1024);
            } else {
                const uint2 v = *reinterpret_cast<const uint2 *>(lds + (wr0 ^ (par * 32)) + unit + m * 1024);
                wd[m][0] = v.x, wd[m][1] = v.y;
            }
#pragma unroll
            for (int g = 0; g < GPS; g++)
                if (G != 128 || par == 0)
                    zw[g][m] = *reinterpret_cast<const int *>(lds + zr + unit + (G == 128 ? 0 : (par * GPS + g) * 128) + m * 64);
        }
    };
    auto constants = [&](const int par, float sg) __attribute__((always_inline)) { // of a step with this parity
#pragma unroll
        for (int g = 0; g < GPS; g++)
#pragma unroll
            for (int m = 0; m < 2; m++) dq[g][m].set((zw[g][m] >> zsh) & 15, G == 128 ? sg : negated(par, g) ? -1.0f : 1.0f);
    };
    uint32_t masked = 0;
    auto dequant = [&](const int to, const int i) __attribute__((always_inline)) { // piece i of 16
        const int m = i >> 3, k = (i >> 2) & 1;
        if (i % 4 == 0) masked = wd[m][k] & 0x0F0F0F0Fu;
        if (i % 4 == 2) masked = (wd[m][k] >> 4) & 0x0F0F0F0Fu;
        aq[to][m][k].u[i % 4] = dq[G == 32 ? k : 0][m].pair(masked, i % 4);
    };
    // Tile t of a step: tokens n = t % NT, MFMA k = t / NT.  Its group, if it ended there, is folded LAG tiles later.
    constexpr int T = 2 * NT, AHEAD = T < 3 ? T : 3, LAG = NT < 2 ? 1 : 2;
    auto read_x = [&](const int par, const int t, uint32_t tile) __attribute__((always_inline)) {
#pragma unroll
        for (int p = 0; p < NP; p++)
            bq[(par * T + t) % 4][p].q = *reinterpret_cast<const uint4 *>(lds + xr[t / NT] + tile + p * S::kPlane + t % NT * 16 * kStepRow);
    };
    auto fold = [&](const int par, const int t) __attribute__((always_inline)) { // tile t of a step of this parity
        const int n = t % NT, k = t / NT;
        if (!(G == 32 || (k == 1 && (G == 64 || par == 1)))) return;
#pragma unroll
        for (int m = 0; m < 2; m++) {
#pragma unroll
            for (int e = 0; e < 4; e++) {
                const float s = sv[G == 32 ? k : 0][m][e];
                acc[n][m][e] = fmaf(negated(par, k) ? -s : s, accg[n][m][e], acc[n][m][e]);
            }
            asm volatile("" : "+v"(acc[n][m])); // here, and not where the compiler would rather have it
        }
    };
    uint32_t tile = 0, tile1 = S::kTile, tile2 = 2 * S::kTile; // this step's tile, the next one's, the one after it
    uint32_t unit = 0, unit1 = S::kUnit, unit2 = 2 * S::kUnit;
    auto k_step = [&](const int par) __attribute__((always_inline)) {
        if (G != 128 || par == 1) constants(par ^ 1, -sign); // of the next step
#pragma unroll
        for (int t = 0; t < T; t++) {
            const int n = t % NT, k = t / NT;
            if (t == T - AHEAD) {
                // The next tile: what this wave requested of it has landed, then what everybody has; and all reads of this one
                // have come back: its place is the next request's.
                asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(XP + (par == 1 ? WL : 0)) : "memory");
            }
            const int behind = (t + AHEAD) % T; // tiles since the barrier: the wave that is behind goes first
            if (T >= 4 && behind % (T / 4) == 0) asm volatile("s_setprio %0" ::"n"(3 - behind * 4 / T));
            read_x(t + AHEAD < T ? par : par ^ 1, (t + AHEAD) % T, t + AHEAD < T ? tile : tile1);
            fold(t < LAG ? par ^ 1 : par, (t + T - LAG) % T);
            const bool fresh = G == 32 || (k == 0 && (G == 64 || par == 0));
#pragma unroll
            for (int p = NP - 1; p >= 0; p--)
#pragma unroll
                for (int m = 0; m < 2; m++)
                    accg[n][m] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(aq[par][m][k].b, bq[(par * T + t) % 4][p].b,
                                                                         fresh && p == NP - 1 ? f4v{} : accg[n][m], 0, 0, 0);
#pragma unroll
            for (int i = t * 16 / T; i < (t + 1) * 16 / T; i++) dequant(par ^ 1, i);
            if (G == 32 ? t % NT == 0 : (t == NT && (G == 64 || par == 1))) { // scales of the group that ends with these tiles
#pragma unroll
                for (int m = 0; m < 2; m++) {
                    sv[G == 32 ? k : 0][m] = *reinterpret_cast<const f4v *>(lds + sr + unit + (G == 128 ? 0 : (par * GPS + (G == 32 ? k : 0)) * 128) + m * 64);
                    if (G == 128) sv[0][m] *= sign;
                }
            }
            // requests, one at a time: the weights two units ahead in front of the tile three steps ahead
            if (t >= T - AHEAD) {
                const int NL = XP + (par == 0 ? WL : 0), j = t - (T - AHEAD);
#pragma unroll
                for (int i = j * NL / AHEAD; i < (j + 1) * NL / AHEAD; i++) {
                    if (par == 0 && i < WL) fetch_w(unit2, i);
                    else fetch_x(tile, par == 0 ? i - WL : i);
                }
            }
            __builtin_amdgcn_sched_barrier(0);
        }
        read_w(par, unit1); // of the step after the next: the same half of the next unit
        const uint32_t free = tile;
        tile = tile1, tile1 = tile2, tile2 = free;
        if (par == 1) {
            const uint32_t free_unit = unit;
            unit = unit1, unit1 = unit2, unit2 = free_unit;
            sign = -sign;
        }
    };
    auto requests = [&](const int tiles, const int units) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < WL; i++) fetch_w(units * S::kUnit, i);
#pragma unroll
        for (int i = 0; i < XP; i++) fetch_x(tiles * S::kTile, i);
    };
    requests(0, 0);
    requests(1, 1);
#pragma unroll
    for (int i = 0; i < XP; i++) fetch_x(2 * S::kTile, i);
    asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"(2 * XP + WL) : "memory");
    read_w(0, 0);
    constants(0, sign);
#pragma unroll
    for (int i = 0; i < 16; i++) dequant(0, i);
    read_w(1, 0);
#pragma unroll
    for (int t = 0; t < AHEAD; t++) read_x(0, t, 0);

    auto finish_folds = [&](const int par) __attribute__((always_inline)) { // those still due behind a step; they add nothing again
#pragma unroll
        for (int t = T - LAG; t < T; t++) fold(par, t), accg[t % NT][0] = accg[t % NT][1] = f4v{0.f, 0.f, 0.f, 0.f};
    };
    const int n_full = n_it / 2 * 2;
    constexpr int kRunGroups = G == 32 ? 16 : G == 64 ? 10 : 8, kRunSteps = kRunGroups * KPG / GPS;
    const int runs = (n_it + kRunSteps - 1) / kRunSteps, run_len = (n_it / runs + 2) / 2 * 2;
    auto end_run = [&]() __attribute__((always_inline)) {
#pragma unroll
        for (int n = 0; n < NT; n++)
#pragma unroll
            for (int m = 0; m < 2; m++) top[n][m] += acc[n][m], acc[n][m] = f4v{0.f, 0.f, 0.f, 0.f};
    };
    int i = 0;
    for (;;) { // whole units, run by run
        for (const int end = min(i + run_len, n_full); i < end; i += 2) {
            k_step(0);
            k_step(1);
        }
        if (i >= n_full) break;
        finish_folds(1);
        end_run();
    }
    if (n_full < n_it) {
        k_step(0);
        finish_folds(0);
    } else {
        finish_folds(1);
    }
    end_run();
    asm volatile("s_waitcnt vmcnt(0)\n\ts_barrier" ::: "memory"); // the LDS is reused below

    size_t ws_base = 0;
    for (int i = 0; i < mi; i++) ws_base += (size_t)KS * B * L.m[i].out;
    // C layout: lane (column r = token, kg), register e -> row 4 kg + e.  Turned through LDS so that a store writes 128
    // contiguous bytes per token.
    constexpr int kTRow = 36, PASS = NT % 2 ? 16 : 32;
    float *tile_o = reinterpret_cast<float *>(lds) + wave * 32 * kTRow;
    const int tl = lane >> 3, oc = (lane & 7) * 4;
#pragma unroll
    for (int n0 = 0; n0 < NT; n0 += PASS / 16) {
#pragma unroll
        for (int n = 0; n < PASS / 16; n++)
#pragma unroll
            for (int m = 0; m < 2; m++) *reinterpret_cast<f4v *>(&tile_o[(n * 16 + r) * kTRow + m * 16 + kg * 4]) = top[n0 + n][m];
#pragma unroll
        for (int pass = 0; pass < PASS / 8; pass++) {
            const int tt = pass * 8 + tl;
            float4 v = *reinterpret_cast<const float4 *>(&tile_o[tt * kTRow + oc]);
            const int t = t0 + n0 * 16 + tt, o = obase + oc;
            if (t < B && o < n_out) finish4(L, mi, ss, ws + ws_base, KS, ks, partials, t, o, v, B);
        }
    }
}

// The first `whole` blocks take a tile each, row block (and slice) by row block, the others tiles of `width` columns of what is
// left, which may begin within a row block where they divide a whole tile.  The last tile of tokens takes as many 16s as it needs (48
// against 64: six layers of 7B, 33 and 48 tokens 1114 / 1131 -> 1046 / 1066 us, 299 2743 -> 2685, three of 70B, 44
// 1531 -> 1397; 13824x5120, 40 columns 36.4 -> 32.6).
template <int G, int NT, int NW>
__global__ __launch_bounds__(64 * NW, NT == 1 ? 3 : 2) void q4_tile_gemm_kernel(const Q4Launch L, const XhList xl, int in_p,
                                                              const float *__restrict__ ss, float *__restrict__ ws, int KS,
                                                              int t_tiles, int row_blocks, int whole, int width, int partials) {
    // an XCD gets all token tiles of a row block one behind the other: what runs on it at one time shares weights and tiles
    int rb, t0, n, B = L.batch;
    asm volatile("" : "+s"(B)); // read once, and not in front of every store again (0.5 % of 13B's prompts)
    if (NT < 4 || (int)blockIdx.x < whole) {
        const int work = xcd_item(blockIdx.x, whole);
        rb = work / t_tiles, t0 = (work - rb * t_tiles) * 16 * NT, n = B - t0;
    } else {
        const int per = (B + width - 1) / width, begun = whole / t_tiles;
        const int work = xcd_item(blockIdx.x - whole, gridDim.x - whole) + begun * per + (whole - begun * t_tiles) * (16 * NT / width);
        rb = work / per, t0 = (work - rb * per) * width, n = min(B - t0, width);
    }
    const int ks = rb / row_blocks;
    rb -= ks * row_blocks;
    switch (min((n + 15) >> 4, NT)) {
#define Q4_TILE(t) \
    case t: \
        if constexpr (t <= NT) q4_tile<G, t, NW>(L, xl, in_p, ss, ws, KS, partials, rb, ks, t0, B); \
        break
        Q4_TILE(1);
        Q4_TILE(2);
        Q4_TILE(3);
        Q4_TILE(4);
        Q4_TILE(5);
#undef Q4_TILE
    }
}

// Linear::matvec<B> of the model without quantisation (src/model.rs:22-31) for a batch: fp32 weights, fp32 activations,
// on the bf16 matrix cores.  The activations are three bf16 planes as above; the weights become three on the way in, each
// rounded to nearest, so that what a plane leaves over has either sign.  All nine products of a weight and an activation are
// taken, so a product is exact as long as both planes are: numbers below 2^-109 have bits below bf16's smallest, 2^-133, and
// enter as multiples of that.  That is 9 products at 2.5 PFLOP/s against one at the 157 TFLOP/s of v_mfma_f32_32x32x2_f32.  (The
// product of the third planes is up to 2^-32 of the whole, 2^-17 of the weight times 2^-15 of the activation.  Without it two layers
// of 7B's widths, 100 tokens with the logits, take 1287 us instead of 1332, but a term is then exact no more, which shows where
// larger ones cancel.)
//
// Sums: the product of the first planes, 16 bits, is all but 2^-7 of a weight times its activation.  These products of 32 inputs
// are summed from zero (one term alone: exactly) and the vector ALU adds them up, rounded to nearest; every other 32 inputs enter
// negated, as above; in runs and the runs to each other, the slices of K in a tree.  Runs of sqrt(steps / 2) and more
// make the two chains about equally long.  The other eight products go through the matrix unit from end to end: its rounding
// is of sums that are 2^-7 of the output's.
//
// Infinities and NaN: the planes of an infinity are not one (inf - inf), and a plane can be rounded to one.  A tile of 16 x 16 with
// a sum that is not finite is done again at the end with v_mfma_f32_16x16x4_f32, from the weights and what the planes stand for,
// unless its token holds a NaN anyway (attention hands one to every token behind it).  7B's w1, 100 columns, 106 us: with a NaN
// in one column 117, in all 187, with an infinity in one 181, in all 640 (one output at a time in the vector ALU: one column
// 2150 us, all 34 ms).
//
// A wave owns 16 rows x 16 NT tokens, a block 8 waves over the rows: a weight is read and split once for up to 128 tokens.
// Lane (row r = l % 16, kg = l / 16) loads 8 consecutive weights of each 32 inputs (a row's cache line, in two loads), four
// such pairs ahead, and splits 32 inputs ahead of the products; the activations of 64 inputs pass through LDS,
// double-buffered; the sums of the runs wait in LDS, which takes up all of it (NT = 8), so a compute unit has one block, and a launch
// of 172 leaves a third of them idle unless K is cut for it (gemm_shape).  What bounds it is the products
// and what issues beside them, one behind the other: a step of 64 inputs and 112 tokens is 480 instructions per wave, 126 of
// them products (2016 cycles), 96 the splitting, and two waves per SIMD take some 7000 cycles for it.
//
// Against products in v_mfma_f32_32x32x2_f32 (128 rows x 64 columns per block, every weight read for each): one layer of 7B's
// widths, 33, 64, 100, 200, 512 columns 332 / 347 / 557 / 1021 / 1818 -> 301 / 341 / 496 / 954 / 1652 us; w1|w3 alone at 99 columns
// 234 -> 214.  Without the three smallest products, and all six in one chain: 285 / 305 / 416 / 773 / 1330 us; but a sum of one term
// then errs by 3.9e-8 rms, 2.3e-7 at most, where fp32 errs by 2.5e-8 and 6.0e-8.
//
// Relative rms error against fp64, that product -> this one (the matvec), 100 columns of 1024 and of 4096 inputs: normal 9.1e-8 -> 6.9e-8
// (9.9e-8), 12.7e-8 -> 8.1e-8 (16.0e-8); one term 2.5e-8 in all; four terms 4.6e-8 -> 4.3e-8 (4.7e-8), 4.7e-8 -> 4.4e-8 (4.6e-8);
// one input 1e6 times the others 10.1e-8 -> 9.1e-8 (9.5e-8), 16.1e-8 -> 10.4e-8 (15.5e-8); all of one sign 3.4e-8 -> 3.8e-8 (3.4e-8),
// 3.5e-8 -> 3.4e-8 (3.6e-8).  11008 inputs, normal: 14e-8 -> 9.3e-8 (24e-8).
constexpr int kDenseWaves = 8, kDenseRows = 16 * kDenseWaves;
template <int NT>
struct DenseLds {
    static constexpr int kPlane = 16 * NT * kStepRow, kTile = 3 * kPlane;
    static constexpr int kTop = NT * 64 * (int)sizeof(f4v); // of a wave
    static constexpr int kSize = 2 * kTile + kDenseWaves * kTop;
};
static_assert(DenseLds<8>::kSize <= 160 * 1024, "LDS of a compute unit");

// A tile of 16 x 16 outputs over the inputs k0..k1-1 (whole 32) in fp32 products.  w, x: the lane's row and token, from its 8
// inputs of the first 32 on.  Every lane of the wave takes part.
__device__ __forceinline__ f4v dense_again(const float *w, const uint16_t *x, int in_p, int k0, int k1) {
    f4v sum{0.f, 0.f, 0.f, 0.f};
#pragma unroll 4
    for (int k = k0; k < k1; k += 32) {
        const float4 wv[2] = {*reinterpret_cast<const float4 *>(w + k), *reinterpret_cast<const float4 *>(w + k + 4)};
        Frag q[3];
#pragma unroll
        for (int p = 0; p < 3; p++) q[p].q = *reinterpret_cast<const uint4 *>(x + (size_t)p * in_p + k);
#pragma unroll
        for (int j = 0; j < 8; j++) {
            auto plane = [&](int p) { return __builtin_bit_cast(float, b16_slot(j) & 1 ? q[p].u[b16_slot(j) >> 1] & 0xFFFF0000u : q[p].u[b16_slot(j) >> 1] << 16); };
            const float hi = plane(0), v = __builtin_isfinite(hi) ? hi + (plane(1) + plane(2)) : hi;
            sum = __builtin_amdgcn_mfma_f32_16x16x4f32((&wv[j >> 2].x)[j & 3], v, sum, 0, 0, 0);
        }
    }
    return sum;
}

// Whether this lane's token has a NaN among the same inputs: then so are its outputs.  Every lane of the wave takes part.
__device__ __forceinline__ bool dense_nan(const uint16_t *x, int k0, int k1) {
    uint32_t most = 0;
#pragma unroll 8
    for (int k = k0; k < k1; k += 32) {
        Frag q;
        q.q = *reinterpret_cast<const uint4 *>(x + k);
#pragma unroll
        for (int i = 0; i < 4; i++) most = max(most, max(q.u[i] & 0x7FFFu, q.u[i] >> 16 & 0x7FFFu));
    }
    uint64_t any = __ballot(most > 0x7F80u); // of the four lanes that share the token
    any |= any >> 32;
    any |= any >> 16;
    return any >> (threadIdx.x & 15) & 1;
}

template <int NT>
__device__ __forceinline__ void dense_tile(const Q4Launch &L, const XhList &xl, int in_p, const float *__restrict__ ss, float *__restrict__ ws,
                                           int KS, int last, int partials, int rb, int ks, int t0) {
    using S = DenseLds<NT>;
    constexpr int NP = 3, TN = 16 * NT, THREADS = 64 * kDenseWaves;
    extern __shared__ __align__(16) char lds[];
    int mi = 0;
    while (mi + 1 < L.n_mats && rb >= L.m[mi].row_blocks) {
        rb -= L.m[mi].row_blocks;
        mi++;
    }
    const void *__restrict__ const xh = xl.p[mi];
    const void *__restrict__ const w = L.m[mi].qweight;
    const int n_out = L.m[mi].out, in = L.in, B = L.batch;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int r = lane & 15, kg = lane >> 4;
    const int obase = rb * kDenseRows + wave * 16;
    const int n_unit = in_p / 64;
    const int before = n_unit - last, equal = last ? KS - 1 : KS;
    const int it0 = ks < equal ? before * ks / equal : before, it1 = ks < equal ? before * (ks + 1) / equal : n_unit;

    // activations: pieces of 16 bytes, 8 to a token's 64 inputs in a plane
    constexpr int PIECES = NP * TN * 8, XP = (PIECES + THREADS - 1) / THREADS;
    uint32_t xoff[XP], xput[XP];
#pragma unroll
    for (int i = 0; i < XP; i++) {
        const int q = (tid + i * THREADS) % PIECES, t = (q >> 3) % TN, p = q / (8 * TN), j = q & 7; // some twice, if it does not divide
        xoff[i] = ((uint32_t)min(t0 + t, B - 1) * NP + p) * (uint32_t)in_p * 2u + j * 16u;
        xput[i] = (uint32_t)(p * S::kPlane + t * kStepRow + ((j ^ ((t >> 1) & 7)) << 4));
    }
    uint4 xr[XP];
    auto fetch_x = [&](int it) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < XP; i++) xr[i] = ld_at<uint4>(xh, xoff[i] + (uint32_t)min(it, it1 - 1) * 128u);
    };
    auto store_x = [&](uint32_t tile) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < XP; i++) *reinterpret_cast<uint4 *>(lds + tile + xput[i]) = xr[i];
    };
    uint32_t xread[2];
#pragma unroll
    for (int k = 0; k < 2; k++) xread[k] = (uint32_t)r * kStepRow + (((4 * k + kg) ^ ((r >> 1) & 7)) << 4);

    // weights: half h of the K steps is 32 inputs, 8 kg .. 8 kg + 7 the lane's.  Inputs beyond the row are zero in the
    // activations; their weights are the row's last ones again.
    struct Raw {
        float4 v[2];
    };
    const uint32_t wrow = (uint32_t)min(obase + r, n_out - 1) * (uint32_t)in * 4u;
    const int h_last = 2 * it1 - 1;
    auto fetch_w = [&](int h, Raw &d) __attribute__((always_inline)) {
        const uint32_t c = wrow + (uint32_t)min(min(h, h_last) * 32 + 8 * kg, in - 8) * 4u;
#pragma unroll
        for (int i = 0; i < 2; i++) d.v[i] = ld_at<float4>(w, c + 16u * i);
    };
    Raw raw[4];
    Frag a[2][NP], minus; // [half][plane]; the first plane of half 1, negated
    auto split = [&](const int from, const int half, const int i) __attribute__((always_inline)) { // a pair of weights, of four
        constexpr int order[8] = {0, 2, 4, 6, 1, 3, 5, 7}; // the activations' slots
        float x = (&raw[from].v[order[2 * i] >> 2].x)[order[2 * i] & 3], y = (&raw[from].v[order[2 * i + 1] >> 2].x)[order[2 * i + 1] & 3];
#pragma unroll
        for (int p = 0; p < NP; p++) {
            const uint32_t b = __builtin_bit_cast(uint32_t, __builtin_convertvector(v2f{x, y}, b2));
            a[half][p].u[i] = b;
            if (p == 0 && half == 1) minus.u[i] = b ^ 0x80008000u;
            if (p < NP - 1) x -= __builtin_bit_cast(float, b << 16), y -= __builtin_bit_cast(float, b & 0xFFFF0000u);
        }
    };

    // first x first: the products of 32 inputs, the sums of the current run and of the runs (this one in LDS, for want of
    // registers); all others
    f4v sum[4], run[NT], low[NT];
    f4v *const top = reinterpret_cast<f4v *>(lds + 2 * S::kTile + wave * S::kTop) + lane;
#pragma unroll
    for (int n = 0; n < NT; n++) run[n] = low[n] = top[64 * n] = f4v{0.f, 0.f, 0.f, 0.f};
    // The products of a half step go by pairs of token tiles, whose chains do not wait for each other.
    constexpr int PAIRS = (NT + 1) / 2;
    Frag b[4][NP];
    auto read_x = [&](const int pair, uint32_t tile) __attribute__((always_inline)) { // of the step's 2 PAIRS
#pragma unroll
        for (int u = 0; u < 2; u++) {
            const int n = pair % PAIRS * 2 + u;
            if (n < NT) {
#pragma unroll
                for (int p = 0; p < NP; p++)
                    b[(pair & 1) * 2 + u][p].q = *reinterpret_cast<const uint4 *>(lds + xread[pair / PAIRS] + tile + p * S::kPlane + n * 16 * kStepRow);
            }
        }
    };
    auto fold = [&](const int pair) __attribute__((always_inline)) {
#pragma unroll
        for (int u = 0; u < 2; u++) {
            const int n = pair % PAIRS * 2 + u;
            if (n < NT) {
                if (pair < PAIRS) run[n] += sum[(pair & 1) * 2 + u];
                else run[n] -= sum[(pair & 1) * 2 + u];
                asm volatile("" : "+v"(run[n])); // here, and not where the compiler would rather have it
            }
        }
    };
    int run_len = 1; // K steps per run
    while (4 * run_len * run_len < it1 - it0) run_len *= 2;
    int end = it0 + run_len;
    uint32_t tile = 0;
    auto step = [&](const int it, const int par) __attribute__((always_inline)) {
        store_x(tile ^ S::kTile);
        fetch_x(it + 2);
        read_x(0, tile);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int g = 0; g < 2 * PAIRS; g++) {
            const int k = g / PAIRS, next = (2 * par + k + 1) & 3; // the half whose weights are split meanwhile
            if (g + 1 < 2 * PAIRS) read_x(g + 1, tile);
            if (g > 0) fold(g - 1);
            constexpr int pa[8] = {2, 2, 1, 2, 1, 0, 1, 0}, pb[8] = {2, 1, 2, 0, 1, 2, 0, 1};
#pragma unroll
            for (int q = 0; q < 9; q++)
#pragma unroll
                for (int u = 0; u < 2; u++) {
                    const int at = (g & 1) * 2 + u, n = g % PAIRS * 2 + u;
                    if (n >= NT) continue;
                    if (q == 0) sum[at] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(k ? minus.b : a[k][0].b, b[at][0].b, f4v{}, 0, 0, 0);
                    else low[n] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[k][pa[q - 1]].b, b[at][pb[q - 1]].b, low[n], 0, 0, 0);
                }
#pragma unroll
            for (int i = g % PAIRS * 4 / PAIRS; i < (g % PAIRS + 1) * 4 / PAIRS; i++) split(next, k ^ 1, i);
            __builtin_amdgcn_sched_barrier(0);
            if (g % PAIRS == PAIRS - 1) { // after the last use of what was there: a load hoisted above it costs copies that wait for it
#pragma unroll
                for (int p = 0; p < NP; p++) asm volatile("" : "+v"(a[k ^ 1][p].b));
                if (k == 0) asm volatile("" : "+v"(minus.b));
                fetch_w(2 * it + k + 5, raw[next]);
                __builtin_amdgcn_sched_barrier(0);
            }
        }
        fold(2 * PAIRS - 1);
        if (it + 1 == end && end < it1) { // the last run stays in registers
            end += run_len;
#pragma unroll
            for (int n = 0; n < NT; n++) top[64 * n] += run[n], run[n] = f4v{0.f, 0.f, 0.f, 0.f};
        }
        __syncthreads();
        tile ^= S::kTile;
    };
    // the first requests, in the order of the loop, so that its waits are the steady state's
    fetch_x(it0);
    fetch_w(2 * it0, raw[0]);
    fetch_w(2 * it0 + 1, raw[1]);
    fetch_w(2 * it0 + 2, raw[2]);
    store_x(0);
    __builtin_amdgcn_sched_barrier(0);
    fetch_x(it0 + 1);
    __builtin_amdgcn_sched_barrier(0);
    fetch_w(2 * it0 + 3, raw[3]);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int i = 0; i < 4; i++) split(0, 0, i);
    __builtin_amdgcn_sched_barrier(0);
    fetch_w(2 * it0 + 4, raw[0]);
    __syncthreads();
    int it = it0;
    for (; it + 1 < it1; it += 2) step(it, 0), step(it + 1, 1);
    if (it < it1) step(it, 0);
#pragma unroll
    for (int n = 0; n < NT; n++) run[n] = top[64 * n] + (run[n] + low[n]);

    // C layout: lane (column r = token, kg), register e -> row 4 kg + e
    size_t ws_base = 0;
    for (int i = 0; i < mi; i++) ws_base += (size_t)KS * B * L.m[i].out;
    const int o = obase + 4 * kg;
    uint32_t again = 0; // the tiles of which this lane's part is not finite
#pragma unroll
    for (int n = 0; n < NT; n++) {
        const int t = t0 + n * 16 + r;
        if (t >= B || o >= n_out) continue;
        const f4v v = run[n];
        if (__builtin_isfinite((v[0] + v[1]) + (v[2] + v[3]))) finish4(L, mi, ss, ws + ws_base, KS, ks, partials, t, o, make_float4(v[0], v[1], v[2], v[3]), B);
        else again |= 1u << n;
    }
    if (!__any(again)) return;
    const float *const w_lane = reinterpret_cast<const float *>(w) + (size_t)min(obase + r, n_out - 1) * in + 8 * kg;
#pragma unroll 1
    for (int n = 0; n < NT; n++) {
        if (!__any(again >> n & 1)) continue;
        const int t = t0 + n * 16 + r;
        const uint16_t *const x_lane = reinterpret_cast<const uint16_t *>(xh) + (size_t)min(t, B - 1) * NP * in_p + 8 * kg;
        const int k0 = it0 * 64, k1 = min(it1 * 64, in);
        f4v v{NAN, NAN, NAN, NAN};
        const bool nan = dense_nan(x_lane, k0, k1);
        if (__any((again >> n & 1) && !nan)) v = dense_again(w_lane, x_lane, in_p, k0, k1);
        if (again >> n & 1) finish4(L, mi, ss, ws + ws_base, KS, ks, partials, t, o, make_float4(v[0], v[1], v[2], v[3]), B);
    }
}

// NT: the tiles of tokens of a block at most; the last one has as many as it needs.  The slices of K are equal, or the last one
// is `last` K steps: its blocks come behind all others.
template <int NT>
__global__ __launch_bounds__(64 * kDenseWaves, 2) void dense_gemm_kernel(const Q4Launch L, const XhList xl, int in_p,
                                                                         const float *__restrict__ ss, float *__restrict__ ws, int KS,
                                                                         int t_tiles, int last, int partials) {
    const int row_blocks = gridDim.x / (t_tiles * KS), front = last ? gridDim.x - row_blocks * t_tiles : gridDim.x;
    const int b = blockIdx.x;
    const int work = b < front ? xcd_item(b, front) : front + xcd_item(b - front, gridDim.x - front); // as in q4_tile_gemm_kernel
    int rb = work / t_tiles;
    const int t0 = (work - rb * t_tiles) * 16 * NT, need = min(NT, (L.batch - t0 + 15) / 16), ks = rb / row_blocks;
    rb -= ks * row_blocks;
    switch (need) {
#define DENSE_TILE(n) \
    case n: \
        if constexpr (n <= NT) dense_tile<n>(L, xl, in_p, ss, ws, KS, last, partials, rb, ks, t0); \
        break
        DENSE_TILE(1);
        DENSE_TILE(2);
        DENSE_TILE(3);
        DENSE_TILE(4);
        DENSE_TILE(5);
        DENSE_TILE(6);
        DENSE_TILE(7);
        DENSE_TILE(8);
#undef DENSE_TILE
    }
}

// ---- what follows a GEMM -----------------------------------------------------------------------------------------
//
// Partial tiles, and what these kernels write, go past the L2 (store_through): a GEMM of 7B's layers with 64 tokens leaves 8 to 16 MB
// of partial tiles in its last 3 us.  Six layers of 7B, 64 tokens: fp32 1243 -> 1205 us with the tiles, 1195 with all of them, fp16
// 991 -> 974, 128 tokens 1195 -> 1160; 4096x11008, group 32, 61 columns 35.1 -> 33.9.

// Sum of the K slices of four consecutive outputs, as a tree; every load goes out before the first add.  The kernels below are
// compiled for up to 2, 4, 8 and 16 slices: one that is not there costs a load all the same (four slices with four loads and with
// eight: 8192 outputs, 399 tokens 25.0 -> 22.0 us, 5120 outputs, 128 tokens 8.3 -> 7.6, 4096, 511 tokens 13.2 -> 12.6).
template <int N>
__device__ __forceinline__ float4 sum_slices_n(const float *p, size_t slice, int KS) {
    float4 part[N];
#pragma unroll
    for (int k = 0; k < N; k++) part[k] = *reinterpret_cast<const float4 *>(p + min(k, KS - 1) * slice);
#pragma unroll
    for (int k = 1; k < N; k++)
        if (k >= KS) part[k] = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
    for (int d = 1; d < N; d *= 2)
#pragma unroll
        for (int k = 0; k < N; k += 2 * d) part[k].x += part[k + d].x, part[k].y += part[k + d].y, part[k].z += part[k + d].z, part[k].w += part[k + d].w;
    return part[0];
}
__device__ __forceinline__ float4 sum_slices(const float *p, size_t slice, int KS) {
    if (KS <= 2) return sum_slices_n<2>(p, slice, KS);
    if (KS <= 8) return sum_slices_n<8>(p, slice, KS);
    return sum_slices_n<kMaxGemmSlices>(p, slice, KS);
}

// Adds the partial tiles of a launch of one matrix with several K slices and runs the epilogue (store or residual add); a thread
// owns four consecutive outputs of one token.  grid: (ceil(out / 1024), B).  With a launch's description for several matrices as
// its argument, read field by field, it was 0.4 to 0.9 us longer (8192x1024, 100 columns 20.8 -> 19.9 us for the call).
__global__ __launch_bounds__(256) void gemm_reduce_kernel(float *y, const float *ws, const float *res, const float *ss, int out, int B, int KS) {
    asm volatile("" ::"s"(y), "s"(ws), "s"(res), "s"(ss), "s"(out), "s"(B), "s"(KS)); // at once
    const int t = blockIdx.y, o = (blockIdx.x * 256 + threadIdx.x) * 4;
    if (o >= out) return;
    const size_t at = (size_t)t * out + o;
    float4 v = sum_slices(ws + at, (size_t)B * out, KS);
    if (ss) {
        const float sc = ss[t];
        v.x *= sc, v.y *= sc, v.z *= sc, v.w *= sc;
    }
    if (res) {
        const float4 r = *reinterpret_cast<const float4 *>(res + at);
        v.x += r.x, v.y += r.y, v.z += r.z, v.w += r.w;
    }
    *reinterpret_cast<float4_any *>(y + at) = float4_any{v.x, v.y, v.z, v.w};
}

// What follows a residual projection (wo, w2) of a chunk: add the partial tiles and the residual (src/models.rs:263-264,
// 283-285), store the new residual stream, take its rms scale (:55-60), and hand the stream times the norm weight to up
// to three consumers, each in its own act-order: permuted in LDS in fp32, so that the global stores are whole 16-byte
// pieces.  One block per token; at most kTrips x 4096 outputs.  What bounds it is a chain of latencies (loads, the block's
// sum, LDS, stores), so the consumers' orders are requested at the start, every consumer has an LDS row of its own where
// two blocks per CU fit, and the kernel is compiled per trips and slices: at 64 registers two blocks share a CU.
// 4096 outputs, 511 tokens 16.5 -> 12.2 us, 298 tokens in several slices 16.6 -> 12.7; 8192 outputs, 776 tokens 35.0 -> 26.0.
constexpr int kTrips = 4, kConsumers = 3;
template <int NP, int TRIPS, int SL>
__global__ __launch_bounds__(1024, TRIPS <= 2 && TRIPS * SL <= 8 ? 8 : 4) void gemm_residual_norm_kernel(const ResNormPrep A, int rows) {
    __shared__ float red[16];
    extern __shared__ __align__(16) float perm[]; // [rows][out]
    const int t = blockIdx.x, tid = threadIdx.x, n4 = A.out >> 2, n8 = A.out >> 3;
    const int in_p = gemm_padded(A.out);
    const size_t row = (size_t)t * A.out, slice = (size_t)A.B * A.out;
    float sq = 0.f;
    float4 v[TRIPS];
    int4 id[kConsumers][TRIPS]; // the consumers' orders: requested with the rest, not behind the barriers
#pragma unroll
    for (int k = 0; k < TRIPS; k++) {
        const int i4 = min(tid + k * 1024, n4 - 1);
#pragma unroll
        for (int c = 0; c < kConsumers; c++) {
            const int32_t *inv = A.inv[min(c, A.n - 1)];
            id[c][k] = inv ? *reinterpret_cast<const int4 *>(inv + 4 * i4) : make_int4(4 * i4, 4 * i4 + 1, 4 * i4 + 2, 4 * i4 + 3);
        }
    }
#pragma unroll
    for (int k = 0; k < TRIPS; k++) {
        const int i4 = tid + k * 1024;
        if (i4 >= n4) continue;
        const float4 g = *reinterpret_cast<const float4 *>(A.wn + 4 * i4);
        float4 w = *reinterpret_cast<const float4 *>(A.res + row + 4 * i4);
        if (A.ws) {
            const float4 a = sum_slices_n<SL>(A.ws + row + 4 * i4, slice, A.KS);
            w.x += a.x, w.y += a.y, w.z += a.z, w.w += a.w;
            store_through(reinterpret_cast<float4 *>(A.x + row + 4 * i4), w);
        }
        sq = fmaf(w.x, w.x, sq), sq = fmaf(w.y, w.y, sq), sq = fmaf(w.z, w.z, sq), sq = fmaf(w.w, w.w, sq);
        v[k] = make_float4(w.x * g.x, w.y * g.y, w.z * g.z, w.w * g.w);
    }
    for (int off = 32; off > 0; off >>= 1) sq += __shfl_xor(sq, off);
    if ((tid & 63) == 0) red[tid >> 6] = sq;
    for (int c0 = 0; c0 < A.n; c0 += rows) { // as many consumers at a time as the LDS has rows for
        if (c0 > 0) __syncthreads();         // the consumers before have been read out
#pragma unroll
        for (int c = 0; c < kConsumers; c++) {
            if (c < c0 || c >= min(c0 + rows, A.n)) continue;
            float *pc = perm + (size_t)(c - c0) * A.out;
#pragma unroll
            for (int k = 0; k < TRIPS; k++) {
                if (tid + k * 1024 >= n4) continue;
                pc[id[c][k].x] = v[k].x, pc[id[c][k].y] = v[k].y, pc[id[c][k].z] = v[k].z, pc[id[c][k].w] = v[k].w;
            }
        }
        __syncthreads();
        if (c0 == 0 && tid == 0) {
            float s = 0.f;
            for (int w = 0; w < 16; w++) s += red[w];
            s /= (float)A.out;
            s += A.eps;
            A.ss[t] = 1.0f / sqrtf(s);
        }
        for (int c = c0; c < min(c0 + rows, A.n); c++) {
            const float *pc = perm + (size_t)(c - c0) * A.out;
            for (int j8 = tid; j8 < (in_p >> 3); j8 += 1024) {
                float e[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
                if (j8 < n8) {
                    const float4 a = *reinterpret_cast<const float4 *>(&pc[8 * j8]), b = *reinterpret_cast<const float4 *>(&pc[8 * j8 + 4]);
                    e[0] = a.x, e[1] = a.y, e[2] = a.z, e[3] = a.w, e[4] = b.x, e[5] = b.y, e[6] = b.z, e[7] = b.w;
                }
                store_piece<NP>(A.out_h[c], t, in_p, j8, make_piece<NP>(e));
            }
        }
    }
}

// What follows the q|k|v projection of a chunk: add the partial tiles of the three matrices, apply the
// token's rms scale, rotate q and k (src/models.rs:100-129: the second half of a head uses the first half's ROTATED
// value), write q back and k and v into the cache rows of the tokens' positions (:236-249).  A thread takes four
// neighbouring pairs of a head, or four values of v, and no more: what bounds it is latency with few tokens and memory with many
// (50 MB at one slice and 511 tokens of 4096 + 2 x 4096), and blocks that loop over a token's row have one trip's loads in flight.
// One block per token -> this: 4096 + 2 x 4096, 16, 64, 399, 899 tokens 6.4 / 6.8 / 8.0 / 17.4 -> 4.0 / 4.7 / 7.6 / 15.1 us, 8192 + 2 x
// 1024, 64 and 776 tokens 7.4 / 14.0 -> 5.4 / 12.2.
template <int SL>
__global__ __launch_bounds__(512) void gemm_rope_kv_kernel(const RopeKvArgs A) {
    constexpr int HS = 128, HALF = 64;
    const int b = blockIdx.x;
    const int dim = A.n_heads * HS, kv_dim = A.n_kv_heads * HS;
    const int p = A.pos[b];
    const float ss = A.ss[b];
    const float *ct = A.cos_t + (size_t)p * HALF, *st = A.sin_t + (size_t)p * HALF;
    const float *wq = A.ws + (size_t)b * dim;
    const float *wk = A.ws + (size_t)A.KS * A.B * dim + (size_t)b * kv_dim;
    const float *wv = wk + (size_t)A.KS * A.B * kv_dim;
    const size_t sq = (size_t)A.B * dim, sk = (size_t)A.B * kv_dim;
    float *kc = A.kcache + (size_t)p * kv_dim, *vc = A.vcache + (size_t)p * kv_dim;
    const int nq = dim >> 3, nk = kv_dim >> 3, nv = kv_dim >> 2;
    const int idx = blockIdx.y * 512 + threadIdx.x;
    if (idx >= nq + nk + nv) return;
    if (idx >= nq + nk) {
        const int i = (idx - nq - nk) * 4;
        const float4 v = sum_slices_n<SL>(wv + i, sk, A.KS);
        store_through(reinterpret_cast<float4 *>(vc + i), make_float4(v.x * ss, v.y * ss, v.z * ss, v.w * ss));
        return;
    }
    const bool is_q = idx < nq;
    const int j = is_q ? idx : idx - nq, i = (j & 15) * 4, at = (j >> 4) * HS + i;
    const float4 c = *reinterpret_cast<const float4 *>(ct + i), s = *reinterpret_cast<const float4 *>(st + i);
    const float *src = (is_q ? wq : wk) + at;
    const size_t slice = is_q ? sq : sk;
    float4 x = sum_slices_n<SL>(src, slice, A.KS), y = sum_slices_n<SL>(src + HALF, slice, A.KS);
    x.x *= ss, x.y *= ss, x.z *= ss, x.w *= ss;
    y.x *= ss, y.y *= ss, y.z *= ss, y.w *= ss;
    const float4 f = make_float4(x.x * c.x - y.x * s.x, x.y * c.y - y.y * s.y, x.z * c.z - y.z * s.z, x.w * c.w - y.w * s.w);
    float *dst = (is_q ? A.q + (size_t)b * dim : kc) + at;
    store_through(reinterpret_cast<float4 *>(dst), f);
    store_through(reinterpret_cast<float4 *>(dst + HALF),
                  make_float4(y.x * c.x + f.x * s.x, y.y * c.y + f.y * s.y, y.z * c.z + f.z * s.z, y.w * c.w + f.w * s.w));
}

// The SiLU gate (src/models.rs:92-98) behind w1|w3 of a chunk: add the partial tiles of both, apply the token's rms
// scale, gate, and hand the row to w2 in its act-order (permuted in LDS, as fp16 where that is what w2 reads: 28672 values in fp32
// were all the LDS that one block per CU has).  One block per token, two trips' loads in flight; with few slices in 64
// registers, two blocks per CU: 11008 values, 511 tokens 13.6 -> 11.4 us.
template <int NP, int SL>
__global__ __launch_bounds__(1024, SL <= 2 ? 8 : 4) void gemm_silu_kernel(const SiluArgs A) {
    typedef std::conditional_t<NP == 1, _Float16, float> In;
    extern __shared__ __align__(16) char perm_lds[];
    In *const perm = reinterpret_cast<In *>(perm_lds); // [n]
    const int t = blockIdx.x, tid = threadIdx.x, n = A.n, in_p = gemm_padded(n), n4 = n >> 2;
    const size_t slice = (size_t)A.B * n, row = (size_t)t * n;
    const float ss = A.ss[t];
    constexpr int U = SL <= 2 ? 2 : 1;
    for (int i0 = tid; i0 < n4; i0 += U * 1024) {
        int4 id[U];
        float4 a[U], c[U];
#pragma unroll
        for (int u = 0; u < U; u++) {
            const int i4 = min(i0 + u * 1024, n4 - 1);
            id[u] = A.inv ? *reinterpret_cast<const int4 *>(A.inv + 4 * i4) : make_int4(4 * i4, 4 * i4 + 1, 4 * i4 + 2, 4 * i4 + 3);
            a[u] = sum_slices_n<SL>(A.ws + row + 4 * i4, slice, A.KS);
            c[u] = sum_slices_n<SL>(A.ws + A.KS * slice + row + 4 * i4, slice, A.KS);
        }
#pragma unroll
        for (int u = 0; u < U; u++) {
            if (u > 0 && i0 + u * 1024 >= n4) break;
            const float as[4] = {a[u].x, a[u].y, a[u].z, a[u].w}, cs[4] = {c[u].x, c[u].y, c[u].z, c[u].w};
            const int ids[4] = {id[u].x, id[u].y, id[u].z, id[u].w};
#pragma unroll
            for (int e = 0; e < 4; e++) {
                float s = as[e] * ss;
                s = s * (1.0f / (1.0f + expf(-s)));
                s = s * (cs[e] * ss);
                if constexpr (NP == 1) {
                    asm("" : "+v"(s)); // rounded to fp32 first, as ever
                    perm[h16_slot(ids[e])] = (_Float16)s;
                } else {
                    perm[ids[e]] = s;
                }
            }
        }
    }
    __syncthreads();
    for (int j8 = tid; j8 < (in_p >> 3); j8 += 1024) {
        if constexpr (NP == 1) { // as the GEMM wants them already
            Piece<NP> r{};
            if (8 * j8 < n) r.q[0] = *reinterpret_cast<const uint4 *>(&perm[8 * j8]);
            store_piece<NP>(A.out_h, t, in_p, j8, r);
        } else {
            float e[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
            if (8 * j8 < n) {
                const float4 a = *reinterpret_cast<const float4 *>(&perm[8 * j8]), b = *reinterpret_cast<const float4 *>(&perm[8 * j8 + 4]);
                e[0] = a.x, e[1] = a.y, e[2] = a.z, e[3] = a.w, e[4] = b.x, e[5] = b.y, e[6] = b.z, e[7] = b.w;
            }
            store_piece<NP>(A.out_h, t, in_p, j8, make_piece<NP>(e));
        }
    }
}

// A tile of 32 rows x 32 groups per block, turned through LDS.
__global__ __launch_bounds__(256) void group_tiles_kernel(const float *scales, const int32_t *qzeros, int out, int groups, float *scales_t, int32_t *zeros_t) {
    __shared__ float s[32][33];
    const int tile = blockIdx.x, g0 = blockIdx.y * 32, lo = threadIdx.x & 31, hi = threadIdx.x >> 5;
    for (int r = hi; r < 32; r += 8) {
        const int row = tile * 32 + r;
        s[r][lo] = row < out && g0 + lo < groups ? scales[(size_t)row * groups + g0 + lo] : 0.f;
    }
    __syncthreads();
    for (int g = hi; g < 32; g += 8)
        if (g0 + g < groups) scales_t[((size_t)tile * groups + g0 + g) * 32 + lo] = s[lo][g];
    const int z = tile * 4 + hi; // a word of eight rows
    if (hi < 4 && g0 + lo < groups) zeros_t[((size_t)tile * groups + g0 + lo) * 4 + hi] = z < out >> 3 ? qzeros[(size_t)z * groups + g0 + lo] : 0;
}

// ---- launchers ---------------------------------------------------------------------------------------------------

template <int G, int NT, int NW>
int ready_tile(size_t *lds) {
    *lds = std::max(TileLds<G, NT, NW>::kSize, (size_t)NW * 32 * 36 * sizeof(float));
    static LdsLimit limit; // per instantiation
    return limit.ensure(reinterpret_cast<const void *>(q4_tile_gemm_kernel<G, NT, NW>), *lds);
}

// How the blocks of a launch are dealt out (q4_tile_gemm_kernel), and what it takes in whole tiles of 64: a tile of w columns 0.4 + 0.15 w / 16.
struct TilePlan {
    int tokens, whole, width, blocks;
    float cost;
};

// One block per CU: what whole rounds of tiles leave over goes in the narrowest tiles with which it is one round of
// blocks.  Six layers of 7B, 32: 169, 250, 439 tokens 2239 / 2470 / 3871 ->
// 2120 / 2357 / 3635 us, four of 13B, 149 1964 -> 1881; 48: 299 and 511 tokens of 7B 2668 / 3971 -> 2632 /
// 3934, 179 of 70B 3251 -> 3196; 4096x11008, group 32, 130 columns 68.3 -> 58.7.  And where a last round is all there is, of any
// whole 16s, and tiles of 80 where those take less (a weight is dequantised once per tile): six layers of 7B, 149, 639 tokens 1931 / 4997 ->
// 1892 / 4905, four of 13B, 149, 399 in chunks of 256 1914 / 3501 -> 1729 / 3399, of 7B, group 32, 129 1391 -> 1341.
static TilePlan plan_tiles(int TN, int blocks_per_tile, int B, bool narrower) {
    auto cost = [](int w) { return 0.4f + 0.15f / 16 * w; };
    const int t_tiles = (B + TN - 1) / TN, tiles = blocks_per_tile * t_tiles, cus = cu_count();
    TilePlan p{TN, tiles, TN, tiles, (tiles + cus - 1) / cus * cost(t_tiles > 1 ? TN : (B + 15) / 16 * 16)};
    if (narrower && tiles % cus) {
        // Whole tiles for full rounds, to the tile where the narrower ones divide one (three layers of 70B, 750 tokens, where only then
        // those of 32 fit: 10690 -> 10440).
        const int rounds = tiles / cus * cus, begun = rounds / t_tiles;
        for (int w = TN - 16; w >= 16; w -= 16) {
            const int done = TN % w ? 0 : rounds % t_tiles, per = (B + w - 1) / w, at = begun * per + done * (TN / w), n = blocks_per_tile * per - at;
            const float c = tiles / cus * cost(TN) + cost(w);
            if (n <= cus && c < p.cost) p = {TN, begun * t_tiles + done, w, begun * t_tiles + done + n, c};
        }
    }
    return p;
}

static TilePlan plan_launch(const GemmShape &s, int group_size, int B) {
    const int all = s.row_blocks * s.slices;
    const TilePlan p = plan_tiles(s.tokens, all, B, s.tokens == 64);
    if (s.tokens < 64 || group_size < 64) return p; // (groups of 32 have more scales, and no LDS for 80)
    const TilePlan wide = plan_tiles(80, all, B, true);
    return wide.cost < 0.98f * p.cost ? wide : p;
}

template <int G, int NT, int NW>
int launch_tile(const Q4Launch &L, const XhList &xh, const float *ss, float *ws, const GemmShape &s, const TilePlan &p, int partials, hipStream_t st) {
    size_t lds = 0;
    L2_TRY((ready_tile<G, NT, NW>(&lds)));
    const int t_tiles = (L.batch + 16 * NT - 1) / (16 * NT);
    l2_launch(q4_tile_gemm_kernel<G, NT, NW>, dim3(p.blocks), dim3(64 * NW), lds, st, L, xh, gemm_padded(L.in), ss, ws, s.slices, t_tiles, s.row_blocks,
              p.whole, p.width, partials);
    L2_HIP(hipGetLastError());
    return L2_OK;
}

template <int G>
int ready_group() {
    size_t lds = 0;
    L2_TRY((ready_tile<G, 1, 4>(&lds)));
    L2_TRY((ready_tile<G, 2, 4>(&lds)));
    L2_TRY((ready_tile<G, 4, 8>(&lds)));
    if constexpr (G >= 64) L2_TRY((ready_tile<G, 5, 8>(&lds)));
    return L2_OK;
}

template <int G>
int launch_group(const Q4Launch &L, const XhList &xh, const float *ss, float *ws, const GemmShape &s, int partials, hipStream_t st) {
    const TilePlan p = plan_launch(s, G, L.batch);
    if constexpr (G >= 64)
        if (p.tokens == 80) return launch_tile<G, 5, 8>(L, xh, ss, ws, s, p, partials, st);
    if (p.tokens == 64) return launch_tile<G, 4, 8>(L, xh, ss, ws, s, p, partials, st);
    if (p.tokens == 32) return launch_tile<G, 2, 4>(L, xh, ss, ws, s, p, partials, st);
    return launch_tile<G, 1, 4>(L, xh, ss, ws, s, p, partials, st);
}

template <int NT>
int launch_dense(const Q4Launch &L, const XhList &xh, const float *ss, float *ws, const GemmShape &s, int partials, hipStream_t st) {
    static LdsLimit limit; // per instantiation
    const size_t lds = DenseLds<NT>::kSize;
    L2_TRY(limit.ensure(reinterpret_cast<const void *>(dense_gemm_kernel<NT>), lds));
    const int t_tiles = (L.batch + 16 * NT - 1) / (16 * NT);
    l2_launch(dense_gemm_kernel<NT>, dim3(s.row_blocks * t_tiles * s.slices), dim3(64 * kDenseWaves), lds, st, L, xh, gemm_padded(L.in), ss, ws, s.slices, t_tiles, s.last,
              partials);
    L2_HIP(hipGetLastError());
    return L2_OK;
}

int launch_fp32(Q4Launch &L, const XhList &xh, const float *ss, float *ws, const GemmShape &s, int partials, hipStream_t st) {
    for (int i = 0; i < L.n_mats; i++) L.m[i].row_blocks = (L.m[i].out + s.rows - 1) / s.rows;
    switch (L.group_size) {
        case 0:
            if (s.tokens == 128) return launch_dense<8>(L, xh, ss, ws, s, partials, st);
            if (s.tokens == 64) return launch_dense<4>(L, xh, ss, ws, s, partials, st);
            return launch_dense<2>(L, xh, ss, ws, s, partials, st);
        case 32: return launch_group<32>(L, xh, ss, ws, s, partials, st);
        case 64: return launch_group<64>(L, xh, ss, ws, s, partials, st);
        case 128: return launch_group<128>(L, xh, ss, ws, s, partials, st);
    }
    return l2_fail(L2_ERR_ARG, "q4 gemm: group size %d", L.group_size);
}

} // namespace

static int row_blocks(const Q4Launch &L, int rows) {
    int n = 0;
    for (int i = 0; i < L.n_mats; i++) n += (L.m[i].out + rows - 1) / rows;
    return n;
}

GemmShape gemm_shape(const Q4Launch &L, int slice_batch, int planes) {
    if (planes == 1) return gemm_shape_f16(L, slice_batch);
    GemmShape s{};
    const int B = L.batch;
    // inputs per slice, at least: 256, and from 4096 inputs on 512 (4096 -> 4096, group 128, 32 columns, 16 slices
    // 19.4 us, 8 17.0; 1024 inputs, 4 slices or 2, a three-layer prompt of 32: 140 or 153)
    const int shortest = L.in >= 4096 && L.group_size > 32 ? 512 : 256;
    auto slices = [&](int slots, int blocks, int most) { return std::max(1, std::min({slots / blocks, most, gemm_padded(L.in) / shortest})); };
    const int rows32 = row_blocks(L, 128), rows64 = row_blocks(L, 256), cus = cu_count();
    // The slices of K, of those that take `max_rounds` rounds of one block per CU at most, with the smallest cost: a block costs its
    // share of K, the first and last microseconds (4.5 % of 4096 inputs) and, with several slices, its partial tile, written and
    // read again (7.5 %).
    auto cheapest = [&](int blocks, int most, int max_rounds, float *its = nullptr) {
        const float per = 4096.0f / L.in;
        float best = 0.f;
        int slices = 1;
        for (int n = 1; n <= std::max(1, most) && (n == 1 || n * blocks <= max_rounds * cus); n++) {
            const int rounds = (n * blocks + cus - 1) / cus;
            const float cost = rounds * (1.0f / n + 0.045f * per) + (n > 1 ? 0.075f * per * n * blocks / cus : 0.f);
            if (n == 1 || cost < best) best = cost, slices = n;
        }
        if (its) *its = best;
        return slices;
    };
    if (L.group_size == 0) {
        // Blocks of 128 columns, so that a weight is read and split once; of 64 where those would leave half the CUs without a
        // block (four layers of 1024 inputs, 128 columns: 424 -> 363 us; 7B's widths keep 128: 64 columns at three quarters of
        // the CUs 530 -> 585).  128 inputs per slice at least (1024 inputs, 100 columns 367 us with 256, 348; with 64 349).
        const int blocks = rows32 * ((slice_batch + 127) / 128), n_unit = gemm_padded(L.in) / 64;
        float best = 0.f;
        s.slices = cheapest(blocks, std::min(kMaxGemmSlices, L.in / 128), 4, &best);
        // Or n equal slices and one of `last` steps of 64 inputs, of which the CUs that the last round of the others leaves take `each` in
        // their time, 2.9 steps (the 4.5 % above) to begin and end each: w1|w3 of 7B's widths, 172 row blocks, is one block per CU and
        // two thirds of the CUs in whole rows, 50 steps and three times 14 with it.  Two layers, 100 columns, with the logits 1341 -> 1286 us
        // (short slices of 12, 16, 18, 20 steps 1311 / 1316 / 1339 / 1365; four equal ones 1329); q|k|v in 26 + 26 + 12 steps for 32 + 32 another 10
        // (3 x 16 + 16 67 more, five equal ones 11 more).
        // Not for fewer slices than the equal ones, whose sums are shorter (2048 -> 17248, two for three: an error of 8.1e-8 for 7.8e-8; 4096 -> 22016, two
        // for one: 9.4e-8 for 9.9e-8, 4096 -> 11008, three for two: 8.8e-8 for 8.9e-8).
        // The 2.9 and the 0.97 are of that shape.  Whole layers of other widths, 17 to 800 columns, equal slices -> with it where it is taken: 2048 inputs
        // 5632 hidden, 17, 64, 400, 800 107 / 129 / 420 / 706 -> 101 / 122 / 407 / 687 us; 3072, 8192, 400 852 -> 821; 5120, 13824, 800 3696 -> 3695; 8192, 14336, 17, 64,
        // 130, 400, 800 518 / 626 / 1584 / 3185 / 5850 -> 511 / 620 / 1556 / 3134 / 5702.
        const float per = 4096.0f / L.in;
        for (int n = s.slices; n + 1 < kMaxGemmSlices && n * blocks <= 4 * cus; n++) {
            const int rounds = (n * blocks + cus - 1) / cus, idle = rounds * cus - n * blocks;
            if (!idle) continue;
            const int each = (blocks + idle - 1) / idle, last = (int)((n_unit - 2.9f * n * (each - 1)) / (n * each + 1));
            if (last < 2) continue;
            const float cost = rounds * ((float)(n_unit - last) / (n * n_unit) + 0.045f * per) + 0.075f * per * (n + 1) * blocks / cus;
            if (cost < 0.97f * best) best = cost, s.slices = n + 1, s.last = last;
        }
        s.tokens = B <= 32 ? 32 : B <= 64 || 2 * rows32 * ((B + 127) / 128) * s.slices <= cus ? 64 : 128;
        s.rows = 128, s.row_blocks = rows32;
        return s;
    }
    if (slice_batch <= 32) {
        // two blocks of 128 rows per CU (13824 -> 5120, 16 columns, 12 slices: 26 us; with three or four per CU 28)
        s.slices = slices(2 * cus, rows32, kMaxGemmSlices);
    } else {
        // one block of 256 rows x 64 columns per CU; two rounds of blocks is what the operator's fixed workspace holds
        s.slices = cheapest(rows64 * ((slice_batch + 63) / 64), std::min(slice_batch <= 64 ? kMaxGemmSlices : 8, L.in / shortest), 2);
    }
    // tiles of 32 columns and 128 rows too where wider blocks would leave half the CUs without one (six layers of 1024
    // inputs, group 64, 64 columns: 404 -> 380 us)
    const bool few = 2 * rows64 * ((B + 63) / 64) * s.slices <= cus;
    s.tokens = B <= 16 ? 16 : B <= 32 || few ? 32 : 64;
    s.rows = s.tokens == 64 ? 256 : 128;
    s.row_blocks = s.rows == 128 ? rows32 : rows64;
    return s;
}

GemmTiles gemm_tiles(const Q4Launch &L, int slice_batch, int planes, bool beside) {
    const GemmShape s = gemm_shape(L, slice_batch, planes);
    if (planes == 1) return gemm_tiles_f16(s, L.batch, beside);
    const TilePlan p = L.group_size ? plan_launch(s, L.group_size, L.batch) : plan_tiles(s.tokens, s.row_blocks * s.slices, L.batch, false);
    return {s.rows, p.tokens, s.slices, p.blocks, p.whole, p.width, s.last, p.whole % ((L.batch + p.tokens - 1) / p.tokens) > 0};
}

int gemm_launch(Q4Launch &L, const XhList &xh, const float *ss, float *ws, size_t ws_floats, int planes, int slice_batch,
                hipStream_t st, int *ks_out, bool beside) {
    if (L.n_mats < 1 || L.n_mats > 3 || L.pair) return l2_fail(L2_ERR_ARG, "q4 gemm: n_mats=%d pair=%d", L.n_mats, L.pair);
    if (L.in % 32 || (L.group_size && L.in % L.group_size) || L.batch < 1) return l2_fail(L2_ERR_ARG, "q4 gemm: in=%d batch=%d", L.in, L.batch);
    if (L.e.kind == Q4_EPI_SCATTER_ONLY || L.e.n_scatter) return l2_fail(L2_ERR_ARG, "q4 gemm: no scatter epilogue");
    long rows = 0;
    for (int i = 0; i < L.n_mats; i++) {
        if (L.m[i].out < 8 || L.m[i].out % 8 || (size_t)L.m[i].out * (L.group_size ? L.in / 8 : L.in) * 4 >= ((size_t)1 << 32))
            return l2_fail(L2_ERR_ARG, "q4 gemm: out=%d in=%d", L.m[i].out, L.in);
        rows += L.m[i].out;
    }
    const GemmShape s = gemm_shape(L, slice_batch, planes);
    const bool partials = ks_out;
    if (!partials && L.n_mats != 1) return l2_fail(L2_ERR_ARG, "q4 gemm: %d matrices without a consumer of their partial tiles", L.n_mats);
    if ((s.slices > 1 || partials) && (size_t)s.slices * L.batch * rows > ws_floats)
        return l2_fail(L2_ERR_ARG, "q4 gemm: %d slices of %d x %ld in a workspace of %zu", s.slices, L.batch, rows, ws_floats);
    if (planes == 1)
        L2_TRY(gemm_launch_f16(L, xh, ss, ws, s, partials, beside, st));
    else
        L2_TRY(launch_fp32(L, xh, ss, ws, s, partials, st));
    if (ks_out) {
        *ks_out = s.slices;
        return L2_OK;
    }
    if (s.slices > 1) {
        l2_launch(gemm_reduce_kernel, dim3((unsigned)((rows + 1023) / 1024), L.batch), dim3(256), 0, st, L.m[0].y, ws,
                           L.e.kind == Q4_EPI_RESIDUAL ? L.e.res : nullptr, ss, L.m[0].out, L.batch, s.slices);
        L2_HIP(hipGetLastError());
    }
    return L2_OK;
}

size_t group_tiles_floats(int out, int groups) { return (size_t)((out + 31) / 32) * groups * 36; }

int group_tiles_launch(const float *scales, const int32_t *qzeros, int out, int groups, float *tiles, hipStream_t st) {
    const int row_tiles = (out + 31) / 32;
    l2_launch(group_tiles_kernel, dim3(row_tiles, (groups + 31) / 32), dim3(256), 0, st, scales, qzeros, out, groups, tiles,
                       reinterpret_cast<int32_t *>(tiles + (size_t)row_tiles * groups * 32));
    L2_HIP(hipGetLastError());
    return L2_OK;
}

int gemm_warm_up(int group_size) {
    switch (group_size) {
        case 32: return ready_group<32>();
        case 64: return ready_group<64>();
        case 128: return ready_group<128>();
    }
    return l2_fail(L2_ERR_ARG, "q4 gemm: group size %d", group_size);
}

int gemm_input_launch(const GemmInput &A, int n, int B, int planes, hipStream_t st) {
    if (n % 32 || A.n < 1 || A.n > 3) return l2_fail(L2_ERR_ARG, "gemm input: n=%d, %d consumers", n, A.n);
    const int in_p = gemm_padded(n);
    const dim3 grid((in_p / 8 + 255) / 256, B, A.n);
    if (planes == 1)
        l2_launch(gemm_input_kernel<1>, grid, dim3(256), 0, st, A, n, in_p);
    else
        l2_launch(gemm_input_kernel<3>, grid, dim3(256), 0, st, A, n, in_p);
    L2_HIP(hipGetLastError());
    return L2_OK;
}

int host_input_launch(void *out, const float *x, const int32_t *inv, int n, int B, int planes, hipStream_t st) {
    if (n % 32 || n < 32 || B < 1 || !inv) return l2_fail(L2_ERR_ARG, "host input: n=%d, %d columns", n, B);
    const dim3 grid((n / 4 + kHostPieces * 256 - 1) / (kHostPieces * 256), B);
    switch (planes) {
        case 0: l2_launch(host_input_kernel<0>, grid, dim3(256), 0, st, out, x, inv, n, n); break;
        case 1: l2_launch(host_input_kernel<1>, grid, dim3(256), 0, st, out, x, inv, n, gemm_padded(n)); break;
        case 3: l2_launch(host_input_kernel<3>, grid, dim3(256), 0, st, out, x, inv, n, gemm_padded(n)); break;
        default: return l2_fail(L2_ERR_ARG, "host input: %d planes", planes);
    }
    L2_HIP(hipGetLastError());
    return L2_OK;
}

template <int NP, int TRIPS, int SL>
static int residual_norm(const ResNormPrep &A, hipStream_t st) {
    // every consumer a row of LDS where two blocks per CU (a token each) still fit
    const int rows = std::max(1, std::min(A.n, (int)(76 * 1024 / (A.out * sizeof(float)))));
    const size_t lds = (size_t)rows * A.out * sizeof(float);
    static LdsLimit limit(48 * 1024);
    L2_TRY(limit.ensure(reinterpret_cast<const void *>(gemm_residual_norm_kernel<NP, TRIPS, SL>), lds));
    l2_launch((gemm_residual_norm_kernel<NP, TRIPS, SL>), dim3(A.B), dim3(1024), lds, st, A, rows);
    L2_HIP(hipGetLastError());
    return L2_OK;
}
template <int NP, int TRIPS>
static int residual_norm(const ResNormPrep &A, hipStream_t st) {
    return A.KS == 1 ? residual_norm<NP, TRIPS, 1>(A, st) : A.KS <= 2 ? residual_norm<NP, TRIPS, 2>(A, st) : A.KS <= 4 ? residual_norm<NP, TRIPS, 4>(A, st) : A.KS <= 8 ? residual_norm<NP, TRIPS, 8>(A, st) : residual_norm<NP, TRIPS, kMaxGemmSlices>(A, st);
}
template <int NP>
static int residual_norm(const ResNormPrep &A, hipStream_t st) {
    return A.out <= 4096 ? residual_norm<NP, 1>(A, st) : A.out <= 8192 ? residual_norm<NP, 2>(A, st) : residual_norm<NP, kTrips>(A, st);
}

int gemm_residual_norm_launch(const ResNormPrep &A, int planes, hipStream_t st) {
    if (A.KS < 1 || A.KS > kMaxGemmSlices || A.out % 32 || A.out > kGemmMaxDim || A.n < 1 || A.n > 3)
        return l2_fail(L2_ERR_ARG, "residual epilogue: %d slices, %d outputs, %d consumers", A.KS, A.out, A.n);
    static_assert(kGemmMaxDim <= kTrips * 4096, "a thread keeps its part of the row in registers");
    return planes == 1 ? residual_norm<1>(A, st) : residual_norm<3>(A, st);
}

int gemm_rope_kv_launch(const RopeKvArgs &A, hipStream_t st) {
    if (A.KS < 1 || A.KS > kMaxGemmSlices || A.B < 1 || A.n_heads < A.n_kv_heads)
        return l2_fail(L2_ERR_ARG, "q|k|v epilogue: %d slices, %d tokens", A.KS, A.B);
    const dim3 grid(A.B, (A.n_heads * 16 + A.n_kv_heads * 48 + 511) / 512), block(512); // a thread per eight of q and k, four of v
    if (A.KS == 1) l2_launch(gemm_rope_kv_kernel<1>, grid, block, 0, st, A);
    else if (A.KS <= 2) l2_launch(gemm_rope_kv_kernel<2>, grid, block, 0, st, A);
    else if (A.KS <= 4) l2_launch(gemm_rope_kv_kernel<4>, grid, block, 0, st, A);
    else if (A.KS <= 8) l2_launch(gemm_rope_kv_kernel<8>, grid, block, 0, st, A);
    else l2_launch(gemm_rope_kv_kernel<kMaxGemmSlices>, grid, block, 0, st, A);
    L2_HIP(hipGetLastError());
    return L2_OK;
}

template <int NP, int SL>
static int silu(const SiluArgs &A, hipStream_t st) {
    const size_t lds = (size_t)A.n * (NP == 1 ? sizeof(_Float16) : sizeof(float));
    static LdsLimit limit(48 * 1024);
    L2_TRY(limit.ensure(reinterpret_cast<const void *>(gemm_silu_kernel<NP, SL>), lds));
    l2_launch((gemm_silu_kernel<NP, SL>), dim3(A.B), dim3(1024), lds, st, A);
    L2_HIP(hipGetLastError());
    return L2_OK;
}
template <int NP>
static int silu(const SiluArgs &A, hipStream_t st) {
    return A.KS == 1 ? silu<NP, 1>(A, st) : A.KS <= 2 ? silu<NP, 2>(A, st) : A.KS <= 4 ? silu<NP, 4>(A, st) : A.KS <= 8 ? silu<NP, 8>(A, st) : silu<NP, kMaxGemmSlices>(A, st);
}

int gemm_silu_launch(const SiluArgs &A, int planes, hipStream_t st) {
    if (A.KS < 1 || A.KS > kMaxGemmSlices || A.n % 32 || A.n > kGemmMaxHidden)
        return l2_fail(L2_ERR_ARG, "silu gate: %d slices, n=%d", A.KS, A.n);
    return planes == 1 ? silu<1>(A, st) : silu<3>(A, st);
}
