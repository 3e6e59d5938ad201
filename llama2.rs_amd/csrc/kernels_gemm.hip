// QLinear::matvec<B> (src/gptq.rs:94-176) for a batch of columns on the matrix cores of gfx950 in fp32, the kernels that
// stand between two such products of a chunk, and the choice of how a product is cut (the fp16 product of the prefill
// mode L2_PREFILL_MFMA is in kernels_q4_gemm.hip).
//
//   Y[t][o] = sum_g s[o][g] * sum_{k in g} (nib(qweight[o],k) - z1[o][g]) X[t][k]
//
// fp32 activations, exactly: x = b0 + b1 + b2 with three bf16 numbers of 8 significant bits each, obtained by cutting x
// after its first, second and third byte of significand.  The weights are integers n - z1 of at most five bits, exact in
// bf16, and so is every product that enters the fp32 accumulator (v_mfma_f32_32x32x16_bf16).  What is left is the sums:
//   - The matrix unit's sum of 16 products and the accumulator is not rounded to nearest; it comes out too small on
//     average, whatever its sign.  Left alone that adds up over K (28672 inputs in groups of 32: mean error -1.7e-7 of
//     the result's rms).  So every other group enters negated, weights and scale: the mean is below 1e-9.
//   - Of the three planes of a step the smallest is added first.
//   - The fp32 group scale is applied to the fp32 sum of each group, and these are added in runs of at most kRunGroups,
//     the runs to each other, the slices of K in a tree: the error of a chain grows with its length.
// Relative rms error against fp64 over 1024..28672 inputs, 8..512 columns, normal inputs: 0.49 to 0.95 of that of the
// matvec (kernels_q4_stream.hip) in every group size; inputs all of one sign, where the matvec is better than elsewhere,
// 0.42 to 1.36 (the largest at 4096 inputs in groups of 32, 512 columns).  One chain, largest plane first, no negation:
// 0.60 to 1.91 and 0.59 to 2.30.
//
// Against the matvec kernels run once per column, which read and dequantise the weights for each of them: 4096x11008,
// group 32, 61 columns 330 -> 40.4 us with everything around it; a 298-token prompt on 7B 230 -> 15.1 ms.
#include <algorithm>

#include "l2_internal.h"

namespace {

typedef float f16v __attribute__((ext_vector_type(16)));
typedef _Float16 h2 __attribute__((ext_vector_type(2)));
typedef _Float16 h8 __attribute__((ext_vector_type(8)));
typedef __bf16 b8 __attribute__((ext_vector_type(8)));
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

// bf16: sign (n - z1) 2^-9 in the order (0,2,4,6,1,3,5,7).  A nibble in the low half of a byte is n 2^-9 as an OCP E4M3
// number; two at a time become fp32, the zero point is subtracted there, and the upper halves of two results are the
// bf16 pair (the integers have at most five bits: nothing is cut off).
struct Dequant {
    float sign, z; // sign: 1 or -1
    static constexpr float kUnit = 0.001953125f; // 2^-9: value of the integer 1
    __device__ __forceinline__ Dequant(int zn, float sg) : sign(sg), z((float)(zn + 1) * (-kUnit * sg)) {}
    __device__ __forceinline__ uint32_t pair(v2f v) const {
        return __builtin_amdgcn_perm(__builtin_bit_cast(uint32_t, fmaf(v.y, sign, z)), __builtin_bit_cast(uint32_t, fmaf(v.x, sign, z)), 0x07060302u);
    }
    __device__ __forceinline__ Frag operator()(uint32_t w) const {
        const uint32_t l = w & 0x0F0F0F0Fu, h = (w >> 4) & 0x0F0F0F0Fu;
        Frag f;
        f.u[0] = pair(__builtin_amdgcn_cvt_pk_f32_fp8(l, false));
        f.u[1] = pair(__builtin_amdgcn_cvt_pk_f32_fp8(l, true));
        f.u[2] = pair(__builtin_amdgcn_cvt_pk_f32_fp8(h, false));
        f.u[3] = pair(__builtin_amdgcn_cvt_pk_f32_fp8(h, true));
        return f;
    }
    static __device__ __forceinline__ f16v mfma(const Frag &a, const Frag &b, f16v c) {
        return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a.b, b.b, c, 0, 0, 0);
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
    if constexpr (NP == kDensePlanes) {
        r.q[0] = __builtin_bit_cast(uint4, make_float4(v[0], v[1], v[2], v[3]));
        r.q[1] = __builtin_bit_cast(uint4, make_float4(v[4], v[5], v[6], v[7]));
    } else if constexpr (NP == 1) {
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

// Plane p of token t: [t][p][in_p], in_p = the row padded to whole K steps (fp32: [t][in_p]).
template <int NP>
__device__ __forceinline__ void store_piece(void *out, size_t t, int in_p, int j8, const Piece<NP> &r) {
    uint4 *dst = reinterpret_cast<uint4 *>(reinterpret_cast<uint16_t *>(out) + t * NP * in_p);
#pragma unroll
    for (int p = 0; p < NP; p++) dst[NP == kDensePlanes ? 2 * j8 + p : p * (in_p >> 3) + j8] = r.q[p];
}

// x[b][g_index[j]] * wn[g_index[j]] -> planes: the gather of src/gptq.rs:110-114 and the norm weight of
// src/models.rs:63-66 in one pass.  grid (pieces / 256, B, consumers).
template <int NP>
__global__ __launch_bounds__(256) void gemm_input_kernel(const GemmInput A, int n, int in_p) {
    const int b = blockIdx.y, c = blockIdx.z;
    const int j8 = blockIdx.x * 256 + threadIdx.x;
    if (j8 * 8 >= in_p) return;
    const float *x = A.x + (size_t)b * n;
    float v[8];
    if (j8 * 8 < n) {
        const int4 g0 = reinterpret_cast<const int4 *>(A.g_index[c])[2 * j8], g1 = reinterpret_cast<const int4 *>(A.g_index[c])[2 * j8 + 1];
        const int g[8] = {g0.x, g0.y, g0.z, g0.w, g1.x, g1.y, g1.z, g1.w};
#pragma unroll
        for (int e = 0; e < 8; e++) v[e] = x[g[e]];
        if (A.wn) {
#pragma unroll
            for (int e = 0; e < 8; e++) v[e] *= A.wn[g[e]];
        }
    } else {
#pragma unroll
        for (int e = 0; e < 8; e++) v[e] = 0.f;
    }
    store_piece<NP>(A.out[c], b, in_p, j8, make_piece<NP>(v));
}

// ---- the GEMM ----------------------------------------------------------------------------------------------------

// Four consecutive outputs of column t: a partial tile of this K slice, or the result through the launch's epilogue.
__device__ __forceinline__ void finish4(const Q4Launch &L, int mi, const float *ss, float *ws, int KS, int ks, int partials,
                                        int t, int o, float4 v) {
    const int n_out = L.m[mi].out;
    if (KS > 1 || partials) {
        *reinterpret_cast<float4 *>(ws + ((size_t)ks * L.batch + t) * n_out + o) = v;
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

constexpr int kRowHalves = 72; // halves per staged token row: 64 k + 8 (16-byte reads of 32 lanes stay conflict-free)

// A block is four waves side by side over the output rows, each with MT x NB tiles of 32 rows x 32 tokens, all of them
// on the same tokens: the activation tile (64 k) is staged in LDS once per block, double-buffered, and every 16 bytes a
// lane reads from it feed MT MFMAs.  (The LDS gives a compute unit some 150 B/ns: with MT = 1 the reads of the tile
// would hold the matrix pipes below 60 %.)  Weights are dequantised in registers, NB * NP times used.
//
// Lane (r = l % 32, h = l / 32) of a 32-row tile.  G >= 64: the lane loads inputs 32 h .. 32 h + 31 of every 64 of its
// row, MFMA step s takes word s.  G = 32: an MFMA step must stay inside one group, so the lane loads both groups of the
// 64 and step s takes word 2 (s % 2) + h of group s / 2.
template <int G, int MT, int NB>
__global__ __launch_bounds__(256, 2) void q4_tile_gemm_kernel(const Q4Launch L, const XhList xl, int in_p,
                                                              const float *__restrict__ ss, float *__restrict__ ws, int KS,
                                                              int t_tiles, int partials) {
    constexpr int NP = 3, TN = 32 * NB, RW = 32 * MT, RB = 4 * RW;
    constexpr int KPG = G >= 64 ? G / 64 : 1; // K steps per group
    constexpr int GPS = G >= 64 ? 1 : 64 / G; // groups per K step
    constexpr int WL = G >= 64 ? 1 : 2;       // 16-byte loads of weights per lane, row tile and K step
    constexpr int PIECES = NP * NB;           // 16-byte pieces of the activation tile per thread
    // K steps that weights are requested ahead (the activations: one): a step is 12 MT NB MFMAs, which cover the way
    // from memory; more would cost the registers of the second block per CU.
    constexpr int WR = 2, PW = 2;
    extern __shared__ __align__(16) uint16_t xs[]; // [2][NP][TN][kRowHalves]
    __shared__ float gsc[2][GPS][RB]; // scales of the group(s) of this K step and the next
    // Blocks are dealt round-robin over the 8 XCDs, each with an L2 of its own.  An XCD gets a contiguous range of the
    // work, all token tiles of a row block one behind the other: what runs on it at one time shares a few row blocks'
    // weights and the tiles' activations.
    const int n_blocks = gridDim.x, per_xcd = n_blocks >> 3, over = n_blocks & 7, xcd = blockIdx.x & 7;
    const int work = xcd * per_xcd + min(xcd, over) + (blockIdx.x >> 3);
    int rb = work / t_tiles, mi = 0;
    const int t0 = (work - rb * t_tiles) * TN;
    const int row_blocks = n_blocks / (t_tiles * KS), ks = rb / row_blocks;
    rb -= ks * row_blocks;
    while (mi + 1 < L.n_mats && rb >= L.m[mi].row_blocks) {
        rb -= L.m[mi].row_blocks;
        mi++;
    }
    // in registers for good: the loop must not ask for kernel arguments again
    const void *__restrict__ const xh = xl.p[mi];
    const void *__restrict__ const qw = L.m[mi].qweight;
    const void *__restrict__ const qz = L.m[mi].qzeros;
    const void *__restrict__ const qs = L.m[mi].scales;
    asm volatile("" ::"s"(xh), "s"(qw), "s"(qz), "s"(qs));
    const int n_out = L.m[mi].out, groups = L.groups, B = L.batch, C4 = L.in >> 5;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int r = lane & 31, h = lane >> 5;
    // this block's slice of K, in whole groups and whole K steps
    const int n_unit = in_p / (64 * KPG);
    const int it0 = (int)((long)n_unit * ks / KS) * KPG, it1 = (int)((long)n_unit * (ks + 1) / KS) * KPG;

    const int obase = rb * RB + wave * RW;
    uint32_t wrow[MT], zrow[MT]; // byte offsets of the lane's rows
    int zsh[MT];
#pragma unroll
    for (int mt = 0; mt < MT; mt++) {
        const int o = min(obase + mt * 32 + r, n_out - 1);
        wrow[mt] = (uint32_t)(o * C4) << 4;
        zrow[mt] = (uint32_t)((o >> 3) * groups) << 2;
        zsh[mt] = 4 * (o & 7);
    }
    const uint32_t srow = (uint32_t)(min(rb * RB + (tid & (RB - 1)), n_out - 1) * groups) << 2;

    struct WStage {
        uint4 w[MT][WL];
        int32_t z[MT][GPS];
    };
    auto fetch_w = [&](int it, WStage &d) __attribute__((always_inline)) {
        const int c = min(it, it1 - 1);
#pragma unroll
        for (int mt = 0; mt < MT; mt++) {
#pragma unroll
            for (int i = 0; i < WL; i++) // past the row's end (in % 64 = 32) the last chunk again: its inputs are zero
                d.w[mt][i] = ld_at<uint4>(qw, wrow[mt] + ((uint32_t)min(2 * c + (WL == 1 ? h : i), C4 - 1) << 4));
#pragma unroll
            for (int g = 0; g < GPS; g++)
                d.z[mt][g] = ld_at<int32_t>(qz, zrow[mt] + ((uint32_t)min(c * GPS / KPG + g, groups - 1) << 2));
        }
    };
    struct XStage {
        uint4 v[PIECES];
    };
    uint32_t xoff[NB];
#pragma unroll
    for (int p = 0; p < NB; p++) {
        const int idx = p * 256 + tid;
        xoff[p] = ((uint32_t)min(t0 + (idx >> 3), B - 1) * (uint32_t)(NP * in_p) + (idx & 7) * 8) * 2u;
    }
    auto fetch_x = [&](int it, XStage &d) __attribute__((always_inline)) {
        const uint32_t kb = (uint32_t)min(it, it1 - 1) * 128u;
#pragma unroll
        for (int q = 0; q < NP; q++)
#pragma unroll
            for (int p = 0; p < NB; p++) d.v[q * NB + p] = ld_at<uint4>(xh, xoff[p] + kb + (uint32_t)(q * in_p) * 2u);
    };
    auto store_x = [&](int buf, const XStage &d) __attribute__((always_inline)) {
#pragma unroll
        for (int q = 0; q < NP; q++)
#pragma unroll
            for (int p = 0; p < NB; p++) {
                const int idx = p * 256 + tid;
                *reinterpret_cast<uint4 *>(xs + ((size_t)(buf * NP + q) * TN + (idx >> 3)) * kRowHalves + (idx & 7) * 8) = d.v[q * NB + p];
            }
    };
    // scales of the group(s) that start with K step it, one row per thread; negative for the groups that enter negated
    auto negated = [](int slot, int g) __attribute__((always_inline)) { return (G < 64 ? g : slot) != 0; };
    auto fetch_s = [&](int it, float (&d)[GPS]) __attribute__((always_inline)) {
#pragma unroll
        for (int g = 0; g < GPS; g++) d[g] = ld_at<float>(qs, srow + ((uint32_t)min(it * GPS / KPG + g, groups - 1) << 2));
    };
    auto store_s = [&](int slot, const float (&d)[GPS]) __attribute__((always_inline)) {
#pragma unroll
        for (int g = 0; g < GPS; g++) gsc[slot][g][tid & (RB - 1)] = d[g] * (negated(slot, g) ? -1.0f / Dequant::kUnit : 1.0f / Dequant::kUnit);
    };

    f16v acc[MT][NB], accg[MT][NB];
#pragma unroll
    for (int mt = 0; mt < MT; mt++)
#pragma unroll
        for (int nb = 0; nb < NB; nb++)
#pragma unroll
            for (int i = 0; i < 16; i++) acc[mt][nb][i] = 0.f;

    WStage wr[WR];
    XStage xr;
    float sr[GPS];
    fetch_s(it0, sr);
    fetch_x(it0, xr);
#pragma unroll
    for (int j = 0; j < WR; j++) fetch_w(it0 + j, wr[j]);
    store_s(0, sr);
    store_x(0, xr);
    __syncthreads();

    // One K step; u = its number within a round of PW (slots of the rings and buffers, known where it is called).
    auto k_step = [&](const int it, const int u) __attribute__((always_inline)) {
        const int gpar = KPG == 2 ? ((it - it0) >> 1) & 1 : u; // buffer of this group's scales
        const bool first = KPG == 1 || u == 0, last = KPG == 1 || u == 1;
        fetch_x(it + 1, xr);
        if (first) fetch_s(it + KPG, sr);
        uint32_t wd[MT][4];
        int zw[MT][GPS];
#pragma unroll
        for (int mt = 0; mt < MT; mt++) {
            if constexpr (WL == 1) {
                wd[mt][0] = wr[u].w[mt][0].x, wd[mt][1] = wr[u].w[mt][0].y, wd[mt][2] = wr[u].w[mt][0].z, wd[mt][3] = wr[u].w[mt][0].w;
            } else {
#pragma unroll
                for (int i = 0; i < 2; i++) {
                    wd[mt][2 * i] = h ? wr[u].w[mt][i].y : wr[u].w[mt][i].x;
                    wd[mt][2 * i + 1] = h ? wr[u].w[mt][i].w : wr[u].w[mt][i].z;
                }
            }
#pragma unroll
            for (int g = 0; g < GPS; g++) zw[mt][g] = (wr[u].z[mt][g] >> zsh[mt]) & 15;
        }
#pragma unroll
        for (int mt = 0; mt < MT; mt++) // the slot's registers are free from here on, and not before
            asm volatile("" : "+v"(wd[mt][0]), "+v"(wd[mt][1]), "+v"(wd[mt][2]), "+v"(wd[mt][3])::"memory");
        __builtin_amdgcn_sched_barrier(0);
        fetch_w(it + WR, wr[u]);
        __builtin_amdgcn_sched_barrier(0);
        const uint16_t *xb = xs + (size_t)u * NP * TN * kRowHalves;
        __builtin_amdgcn_s_setprio(1);
#pragma unroll
        for (int s = 0; s < 4; s++) {
            const int piece = G >= 64 ? 4 * h + s : (s >> 1) * 4 + (s & 1) * 2 + h;
            Frag a[MT], b[NP][NB];
#pragma unroll
            for (int q = 0; q < NP; q++)
#pragma unroll
                for (int nb = 0; nb < NB; nb++)
                    b[q][nb].q = *reinterpret_cast<const uint4 *>(xb + ((size_t)q * TN + nb * 32 + r) * kRowHalves + piece * 8);
#pragma unroll
            for (int mt = 0; mt < MT; mt++) a[mt] = Dequant(zw[mt][G >= 64 ? 0 : s >> 1], negated(gpar, s >> 1) ? -1.0f : 1.0f)(wd[mt][s]);
            const bool zero = first && (G >= 64 ? s == 0 : (s & 1) == 0);
#pragma unroll
            for (int q = NP - 1; q >= 0; q--)
#pragma unroll
                for (int mt = 0; mt < MT; mt++)
#pragma unroll
                    for (int nb = 0; nb < NB; nb++)
                        accg[mt][nb] = Dequant::mfma(a[mt], b[q][nb], zero && q == NP - 1 ? f16v{} : accg[mt][nb]);
            if (G >= 64 ? (last && s == 3) : (s & 1) == 1) { // a group ends: its partial sum, scaled, joins the run
                const float *sc = gsc[gpar][G >= 64 ? 0 : s >> 1] + wave * RW;
#pragma unroll
                for (int mt = 0; mt < MT; mt++)
#pragma unroll
                    for (int k = 0; k < 4; k++) {
                        const float4 sv = *reinterpret_cast<const float4 *>(sc + mt * 32 + k * 8 + h * 4);
                        const float svv[4] = {sv.x, sv.y, sv.z, sv.w};
#pragma unroll
                        for (int nb = 0; nb < NB; nb++)
#pragma unroll
                            for (int e = 0; e < 4; e++)
                                acc[mt][nb][4 * k + e] = fmaf(svv[e], accg[mt][nb][4 * k + e], acc[mt][nb][4 * k + e]);
                    }
            }
        }
        __builtin_amdgcn_s_setprio(0);
        if (last) store_s(gpar ^ 1, sr);
        store_x(u ^ 1, xr);
        __syncthreads();
    };
    size_t ws_base = 0;
    for (int i = 0; i < mi; i++) ws_base += (size_t)KS * B * L.m[i].out;
    // Runs that have ended: their sum lies where the result goes, every lane's own elements.  (There are no registers for a
    // third set of tiles.  What it costs is this traffic: 4096 -> 22016 outputs, 512 columns, group 32, 45 MB a time; a layer
    // of 7B, 512 tokens, 0.88 -> 0.93 ms with runs of 64 groups, 0.98 with 32; 299 tokens, group 128 has one run.)
    float *const sums = KS > 1 || partials ? ws + ws_base + (size_t)ks * B * n_out : L.m[mi].y;
    auto each_sum = [&](auto &&f) __attribute__((always_inline)) {
#pragma unroll
        for (int mt = 0; mt < MT; mt++)
#pragma unroll
            for (int nb = 0; nb < NB; nb++)
#pragma unroll
                for (int k = 0; k < 4; k++) {
                    const int t = t0 + nb * 32 + r, o = obase + mt * 32 + k * 8 + h * 4;
                    if (t < B && o < n_out) f(*reinterpret_cast<float4_any *>(sums + (size_t)t * n_out + o), acc[mt][nb], 4 * k);
                }
    };
    const int n_it = it1 - it0;
    const int n_full = n_it / PW * PW;
    constexpr int kRunGroups = 64, kRunSteps = kRunGroups * KPG / GPS;
    const int runs = (n_it + kRunSteps - 1) / kRunSteps, run_len = (n_it / runs + PW) / PW * PW;
    int i = 0;
    for (;;) { // whole rounds of PW steps, run by run
        for (const int end = min(i + run_len, n_full); i < end; i += PW) {
#pragma unroll
            for (int u = 0; u < PW; u++) k_step(it0 + i + u, u);
        }
        if (i >= n_full) break;
        each_sum([&](float4_any &at, f16v &v, int k) __attribute__((always_inline)) {
            float4_any c{v[k], v[k + 1], v[k + 2], v[k + 3]};
            if (i > run_len) c += at;
            at = c;
            v[k] = v[k + 1] = v[k + 2] = v[k + 3] = 0.f;
        });
    }
#pragma unroll
    for (int u = 0; u < PW - 1; u++) // the rest straight-line: a loop left half-way copies ring registers, and waits
        if (n_full + u < n_it) k_step(it0 + n_full + u, u);
    if (n_full > run_len)
        each_sum([&](float4_any &at, f16v &v, int k) __attribute__((always_inline)) {
            const float4_any c = at;
            v[k] += c.x, v[k + 1] += c.y, v[k + 2] += c.z, v[k + 3] += c.w;
        });

    // C layout: lane (column r = token, h), register i -> row (i / 4) * 8 + h * 4 + i % 4.  Turned through LDS (the
    // activation buffers are free now) so that a store writes 128 contiguous bytes per token.
    constexpr int kTRow = 36;
    float *tile = reinterpret_cast<float *>(xs) + wave * 32 * kTRow;
    const int tl = lane >> 3, oc = (lane & 7) * 4;
#pragma unroll
    for (int mt = 0; mt < MT; mt++)
#pragma unroll
        for (int nb = 0; nb < NB; nb++) {
#pragma unroll
            for (int q = 0; q < 4; q++)
                *reinterpret_cast<float4 *>(&tile[r * kTRow + q * 8 + h * 4]) =
                    make_float4(acc[mt][nb][4 * q], acc[mt][nb][4 * q + 1], acc[mt][nb][4 * q + 2], acc[mt][nb][4 * q + 3]);
#pragma unroll
            for (int pass = 0; pass < 4; pass++) {
                const int tt = pass * 8 + tl;
                float4 v = *reinterpret_cast<const float4 *>(&tile[tt * kTRow + oc]);
                const int t = t0 + nb * 32 + tt, o = obase + mt * 32 + oc;
                if (t < B && o < n_out) finish4(L, mi, ss, ws + ws_base, KS, ks, partials, t, o, v);
            }
        }
}

// Linear::matvec<B> of the model without quantisation (src/model.rs:22-31) for a batch: fp32 weights, fp32 activations,
// fp32 products and sums (v_mfma_f32_32x32x2_f32, 157 TFLOP/s on this chip; it is what bounds the kernel, the loads hide
// behind it).  The matvec kernel once per column read the weights once per column: two layers of 7B's widths, 99 columns
// 16 -> 1 ms.
//
// A block is four waves of NB tiles of 32 rows x 32 columns, side by side over the rows.  Lane (r = l % 32, h = l / 32)
// loads inputs 16 h .. 16 h + 15 of every 32 of its row, 16 bytes at a time; step e of float4 i multiplies inputs 4 i + e
// and 16 + 4 i + e.  The activations' 32 inputs per column pass through LDS, double-buffered.
//
// Sums.  The matrix unit rounds once per product, and the error of a sum of n terms, each added to all before it, grows
// with n.  The matvec adds 64 lanes' shares in a tree, so that in / 64 products follow each other; to be no further from
// the exact sum than that, the products of a K step (of a part of it where the matvec's own chains are short) are summed
// from zero, the steps of a run are added to each other, and the runs; the slices of K follow in a tree (sum_slices_n).
// Runs of sqrt(steps / 2) and more make the two upper chains about equally long.  Relative rms error against fp64, normal
// inputs, matvec / this / one accumulator for the whole slice: 1024 inputs, 61 columns 1.00e-7 / 9.1e-8 / 2.1e-7; 4096,
// 128 columns 1.59e-7 / 1.27e-7 / 4.1e-7; 11008, 512 columns 2.44e-7 / 1.44e-7 / 9.4e-7.
// The sums take the registers of a second row tile (which would reuse every LDS read twice: the matrix unit is slow enough
// in fp32 for one).  Prompts, two row tiles and one accumulator / this: two layers of 7B's widths, 100 tokens 0.95-0.99 /
// 0.98 ms, 512 tokens 3.60 / 3.41; four layers of 1024 inputs, 33 tokens 0.29 / 0.31; one of 70B's widths, 64 tokens
// 1.09-1.13 / 1.12-1.17.
template <int NB, int FOLDS> // FOLDS: sums from zero per K step
__global__ __launch_bounds__(256, FOLDS == 4 ? 2 : 3) void dense_gemm_kernel(const Q4Launch L, const XhList xl, int in_p,
                                                            const float *__restrict__ ss, float *__restrict__ ws, int KS,
                                                            int t_tiles, int partials) {
    constexpr int TN = 32 * NB, RB = 128, kRow = 36; // floats per staged column: 32 + 4
    __shared__ __align__(16) float xs[4608]; // [2][TN][kRow], and the four output tiles of the epilogue
    static_assert(2 * TN * kRow <= 4608 && 4 * 32 * 36 <= 4608, "LDS");
    const int n_blocks = gridDim.x, per_xcd = n_blocks >> 3, over = n_blocks & 7, xcd = blockIdx.x & 7;
    const int work = xcd * per_xcd + min(xcd, over) + (blockIdx.x >> 3); // as in q4_tile_gemm_kernel
    int rb = work / t_tiles, mi = 0;
    const int t0 = (work - rb * t_tiles) * TN;
    const int row_blocks = n_blocks / (t_tiles * KS), ks = rb / row_blocks;
    rb -= ks * row_blocks;
    while (mi + 1 < L.n_mats && rb >= L.m[mi].row_blocks) {
        rb -= L.m[mi].row_blocks;
        mi++;
    }
    const void *__restrict__ const xh = xl.p[mi];
    const void *__restrict__ const w = L.m[mi].qweight;
    asm volatile("" ::"s"(xh), "s"(w));
    const int n_out = L.m[mi].out, in = L.in, B = L.batch;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int r = lane & 31, h = lane >> 5;
    const int n_unit = in / 32;
    const int it0 = (int)((long)n_unit * ks / KS), it1 = (int)((long)n_unit * (ks + 1) / KS);
    const int obase = rb * RB + wave * 32;
    const uint32_t wrow = ((uint32_t)min(obase + r, n_out - 1) * (uint32_t)in + 16 * h) * 4u;
    uint32_t xoff[NB];
#pragma unroll
    for (int p = 0; p < NB; p++) xoff[p] = ((uint32_t)min(t0 + p * 32 + (tid >> 3), B - 1) * (uint32_t)in_p + (tid & 7) * 4) * 4u;
    struct WStage {
        float4 w[4];
    };
    auto fetch_w = [&](int it, WStage &d) __attribute__((always_inline)) {
        const uint32_t c = (uint32_t)min(it, it1 - 1) * 128u;
#pragma unroll
        for (int i = 0; i < 4; i++) d.w[i] = ld_at<float4>(w, wrow + c + 16u * i);
    };
    float4 xr[NB];
    auto fetch_x = [&](int it) __attribute__((always_inline)) {
#pragma unroll
        for (int p = 0; p < NB; p++) xr[p] = ld_at<float4>(xh, xoff[p] + (uint32_t)min(it, it1 - 1) * 128u);
    };
    auto store_x = [&](int buf) __attribute__((always_inline)) {
#pragma unroll
        for (int p = 0; p < NB; p++) *reinterpret_cast<float4 *>(xs + (buf * TN + p * 32 + (tid >> 3)) * kRow + (tid & 7) * 4) = xr[p];
    };
    f16v run[NB], acc[NB];
#pragma unroll
    for (int nb = 0; nb < NB; nb++) run[nb] = acc[nb] = f16v{};
    int run_steps = 2; // K steps per run
    while (2 * run_steps * run_steps < it1 - it0) run_steps *= 2;
    WStage wr[2];
    fetch_x(it0);
    fetch_w(it0, wr[0]);
    store_x(0);
    __syncthreads();
    auto k_step = [&](const int it, const int u) __attribute__((always_inline)) {
        fetch_x(it + 1);
        fetch_w(it + 1, wr[u ^ 1]);
        __builtin_amdgcn_sched_barrier(0); // requested before this step's arithmetic, not behind it
        const float *xb = xs + u * TN * kRow;
        f16v even[NB]; // of four sums, pairs are added first
#pragma unroll
        for (int f = 0; f < FOLDS; f++) {
            constexpr int N = 4 / FOLDS;
            f16v sum[NB];
#pragma unroll
            for (int i = f * N; i < (f + 1) * N; i++) {
                float4 b[NB];
#pragma unroll
                for (int nb = 0; nb < NB; nb++) b[nb] = *reinterpret_cast<const float4 *>(xb + (nb * 32 + r) * kRow + 16 * h + 4 * i);
#pragma unroll
                for (int e = 0; e < 4; e++)
#pragma unroll
                    for (int nb = 0; nb < NB; nb++)
                        sum[nb] = __builtin_amdgcn_mfma_f32_32x32x2f32((&wr[u].w[i].x)[e], (&b[nb].x)[e],
                                                                       i == f * N && e == 0 ? f16v{} : sum[nb], 0, 0, 0);
            }
#pragma unroll
            for (int nb = 0; nb < NB; nb++) {
                if (FOLDS < 4) run[nb] += sum[nb];
                else if (f & 1) run[nb] += even[nb] + sum[nb];
                else even[nb] = sum[nb];
            }
        }
        store_x(u ^ 1);
        __syncthreads();
    };
    int it = it0;
    for (int end = it0 + run_steps; it + 1 < it1; it += 2) {
        k_step(it, 0);
        k_step(it + 1, 1);
        if (it + 2 == end) {
            end += run_steps;
#pragma unroll
            for (int nb = 0; nb < NB; nb++) acc[nb] += run[nb], run[nb] = f16v{};
        }
    }
    if (it < it1) k_step(it, 0);
#pragma unroll
    for (int nb = 0; nb < NB; nb++) acc[nb] += run[nb];

    size_t ws_base = 0;
    for (int i = 0; i < mi; i++) ws_base += (size_t)KS * B * L.m[i].out;
    float *tile = xs + wave * 32 * 36;
    const int tl = lane >> 3, oc = (lane & 7) * 4;
#pragma unroll
    for (int nb = 0; nb < NB; nb++) {
#pragma unroll
        for (int q = 0; q < 4; q++)
            *reinterpret_cast<float4 *>(&tile[r * 36 + q * 8 + h * 4]) =
                make_float4(acc[nb][4 * q], acc[nb][4 * q + 1], acc[nb][4 * q + 2], acc[nb][4 * q + 3]);
#pragma unroll
        for (int pass = 0; pass < 4; pass++) {
            const int tt = pass * 8 + tl;
            float4 v = *reinterpret_cast<const float4 *>(&tile[tt * 36 + oc]);
            const int t = t0 + nb * 32 + tt, o = obase + oc;
            if (t < B && o < n_out) finish4(L, mi, ss, ws + ws_base, KS, ks, partials, t, o, v);
        }
    }
}

// ---- what follows a GEMM -----------------------------------------------------------------------------------------

// Sum of the K slices of four consecutive outputs, as a tree; every load goes out before the first add.
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

// Adds the partial tiles of a launch with several K slices and runs the epilogue (store or residual add); a thread owns
// four consecutive outputs of one token.  grid: (ceil(sum_out / 1024), B); the matrices are laid end to end.
__global__ __launch_bounds__(256) void gemm_reduce_kernel(const Q4Launch L, const float *__restrict__ ss,
                                                          const float *__restrict__ ws, int KS) {
    const int t = blockIdx.y, B = L.batch;
    int o = (blockIdx.x * 256 + threadIdx.x) * 4, mi = 0;
    size_t ws_base = 0;
    while (mi + 1 < L.n_mats && o >= L.m[mi].out) {
        o -= L.m[mi].out;
        ws_base += (size_t)KS * B * L.m[mi].out;
        mi++;
    }
    const Q4Mat &M = L.m[mi];
    if (o >= M.out) return;
    const size_t at = (size_t)t * M.out + o;
    float4 v = sum_slices(ws + ws_base + at, (size_t)B * M.out, KS);
    if (ss) {
        const float sc = ss[t];
        v.x *= sc, v.y *= sc, v.z *= sc, v.w *= sc;
    }
    if (L.e.kind == Q4_EPI_RESIDUAL) {
        const float4 r = *reinterpret_cast<const float4 *>(L.e.res + at);
        v.x += r.x, v.y += r.y, v.z += r.z, v.w += r.w;
    }
    *reinterpret_cast<float4_any *>(M.y + at) = float4_any{v.x, v.y, v.z, v.w};
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
            *reinterpret_cast<float4 *>(A.x + row + 4 * i4) = w;
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
// value), write q back and k and v into the cache rows of the tokens' positions (:236-249).  One block per token; a thread
// takes four neighbouring pairs of a head, or four values of v.  Blocks of 512: at one slice the launch is bound by memory
// (50 MB in 12.3 us for 511 tokens of 4096 + 2 x 4096; 14.6 with blocks of 256, eight to a token).
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
    for (int idx = threadIdx.x; idx < nq + nk + nv; idx += 512) {
        if (idx >= nq + nk) {
            const int i = (idx - nq - nk) * 4;
            const float4 v = sum_slices_n<SL>(wv + i, sk, A.KS);
            *reinterpret_cast<float4 *>(vc + i) = make_float4(v.x * ss, v.y * ss, v.z * ss, v.w * ss);
            continue;
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
        *reinterpret_cast<float4 *>(dst) = f;
        *reinterpret_cast<float4 *>(dst + HALF) =
            make_float4(y.x * c.x + f.x * s.x, y.y * c.y + f.y * s.y, y.z * c.z + f.z * s.z, y.w * c.w + f.w * s.w);
    }
}

// The SiLU gate (src/models.rs:92-98) behind w1|w3 of a chunk: add the partial tiles of both, apply the token's rms
// scale, gate, and hand the row to w2 in its act-order (permuted in LDS).  One block per token; with few slices in 64
// registers, two blocks per CU: 11008 values, 511 tokens 13.6 -> 11.4 us.
template <int NP, int SL>
__global__ __launch_bounds__(1024, SL <= 2 ? 8 : 4) void gemm_silu_kernel(const SiluArgs A) {
    extern __shared__ __align__(16) float perm[]; // [n]
    const int t = blockIdx.x, tid = threadIdx.x, n = A.n, in_p = gemm_padded(n);
    const size_t slice = (size_t)A.B * n, row = (size_t)t * n;
    const float ss = A.ss[t];
    for (int i4 = tid; i4 < (n >> 2); i4 += 1024) {
        const int4 id = A.inv ? *reinterpret_cast<const int4 *>(A.inv + 4 * i4) : make_int4(4 * i4, 4 * i4 + 1, 4 * i4 + 2, 4 * i4 + 3);
        const float4 a = sum_slices_n<SL>(A.ws + row + 4 * i4, slice, A.KS);
        const float4 c = sum_slices_n<SL>(A.ws + A.KS * slice + row + 4 * i4, slice, A.KS);
        const float as[4] = {a.x, a.y, a.z, a.w}, cs[4] = {c.x, c.y, c.z, c.w};
        const int ids[4] = {id.x, id.y, id.z, id.w};
#pragma unroll
        for (int e = 0; e < 4; e++) {
            float s = as[e] * ss;
            s = s * (1.0f / (1.0f + expf(-s)));
            perm[ids[e]] = s * (cs[e] * ss);
        }
    }
    __syncthreads();
    for (int j8 = tid; j8 < (in_p >> 3); j8 += 1024) {
        float e[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
        if (8 * j8 < n) {
            const float4 a = *reinterpret_cast<const float4 *>(&perm[8 * j8]), b = *reinterpret_cast<const float4 *>(&perm[8 * j8 + 4]);
            e[0] = a.x, e[1] = a.y, e[2] = a.z, e[3] = a.w, e[4] = b.x, e[5] = b.y, e[6] = b.z, e[7] = b.w;
        }
        store_piece<NP>(A.out_h, t, in_p, j8, make_piece<NP>(e));
    }
}

// ---- launchers ---------------------------------------------------------------------------------------------------

template <int G, int MT, int NB>
int ready_tile(size_t *lds) {
    *lds = std::max((size_t)2 * 3 * 32 * NB * kRowHalves * 2, (size_t)4 * 32 * 36 * sizeof(float));
    static LdsLimit limit; // per instantiation
    return limit.ensure(reinterpret_cast<const void *>(q4_tile_gemm_kernel<G, MT, NB>), *lds);
}

template <int G, int MT, int NB>
int launch_tile(const Q4Launch &L, const XhList &xh, const float *ss, float *ws, int KS, int partials, int total, hipStream_t st) {
    size_t lds = 0;
    L2_TRY((ready_tile<G, MT, NB>(&lds)));
    const int t_tiles = (L.batch + 32 * NB - 1) / (32 * NB);
    hipLaunchKernelGGL((q4_tile_gemm_kernel<G, MT, NB>), dim3(total * t_tiles * KS), dim3(256), lds, st, L, xh, gemm_padded(L.in), ss, ws, KS, t_tiles, partials);
    L2_HIP(hipGetLastError());
    return L2_OK;
}

template <int G>
int ready_group() {
    size_t lds = 0;
    L2_TRY((ready_tile<G, 1, 1>(&lds)));
    L2_TRY((ready_tile<G, 1, 2>(&lds)));
    L2_TRY((ready_tile<G, 2, 2>(&lds)));
    return L2_OK;
}

template <int G>
int launch_group(Q4Launch &L, const XhList &xh, const float *ss, float *ws, const GemmShape &s, int partials, hipStream_t st) {
    for (int i = 0; i < L.n_mats; i++) L.m[i].row_blocks = (L.m[i].out + s.rows - 1) / s.rows;
    if (s.rows == 256)
        return launch_tile<G, 2, 2>(L, xh, ss, ws, s.slices, partials, s.row_blocks, st);
    if (s.tokens == 64) return launch_tile<G, 1, 2>(L, xh, ss, ws, s.slices, partials, s.row_blocks, st);
    return launch_tile<G, 1, 1>(L, xh, ss, ws, s.slices, partials, s.row_blocks, st);
}

int launch_fp32(Q4Launch &L, const XhList &xh, const float *ss, float *ws, const GemmShape &s, int partials, hipStream_t st) {
    switch (L.group_size) {
        case 32: return launch_group<32>(L, xh, ss, ws, s, partials, st);
        case 64: return launch_group<64>(L, xh, ss, ws, s, partials, st);
        case 128: return launch_group<128>(L, xh, ss, ws, s, partials, st);
    }
    return l2_fail(L2_ERR_ARG, "q4 gemm: group size %d", L.group_size);
}

int launch_dense(Q4Launch &L, const XhList &xh, const float *ss, float *ws, const GemmShape &s, int partials, hipStream_t st) {
    for (int i = 0; i < L.n_mats; i++) L.m[i].row_blocks = (L.m[i].out + s.rows - 1) / s.rows;
    const int t_tiles = (L.batch + s.tokens - 1) / s.tokens, in_p = gemm_padded(L.in);
    const dim3 grid(s.row_blocks * t_tiles * s.slices), block(256);
    auto launch = [&](void (*kernel)(Q4Launch, XhList, int, const float *, float *, int, int, int)) {
        hipLaunchKernelGGL(kernel, grid, block, 0, st, L, xh, in_p, ss, ws, s.slices, t_tiles, partials);
    };
    // products summed from zero: 32; 16 and 8 where the matvec's chains are so short that it would be nearer to the exact sum
    // (1024 inputs: 16s 1.01e-7 in eight slices and 1.09e-7 in one against its 1.00e-7)
    if (L.in >= 2560) launch(s.tokens == 64 ? dense_gemm_kernel<2, 1> : dense_gemm_kernel<1, 1>);
    else if (L.in >= 2048) launch(s.tokens == 64 ? dense_gemm_kernel<2, 2> : dense_gemm_kernel<1, 2>);
    else launch(s.tokens == 64 ? dense_gemm_kernel<2, 4> : dense_gemm_kernel<1, 4>);
    L2_HIP(hipGetLastError());
    return L2_OK;
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
    const int kstep = planes == kDensePlanes ? 32 : L.group_size > 64 ? L.group_size : 64, units = (gemm_padded(L.in) + kstep - 1) / kstep;
    auto slices = [&](int slots, int blocks, int most) { return std::max(1, std::min({slots / blocks, most, units / 2})); };
    // K slices: as many as keep the grid within one round of resident blocks.  Up to 32 columns the registers and the
    // LDS hold four blocks per CU of 128 rows, and the partial tiles are small; beyond, two of 256 rows (fp32 weights: three
    // of 128).  Where the rows are cut in 128s all the same (below), the grid is twice what was counted and may take a
    // second round: 11008 outputs, 61 columns are 688 blocks in 8 slices on 512 slots.
    const int rows32 = row_blocks(L, 128), rows64 = row_blocks(L, 256);
    if (slice_batch <= 32)
        s.slices = slices(4 * cu_count(), rows32, kMaxGemmSlices);
    else if (planes == kDensePlanes)
        s.slices = slices(3 * cu_count(), rows32 * ((slice_batch + 63) / 64), 8);
    else
        s.slices = slices(2 * cu_count(), rows64 * ((slice_batch + 63) / 64), 8);
    s.tokens = B <= 32 ? 32 : 64;
    // 256 rows reuse every 16 bytes read from the LDS twice; 128 where such blocks would be fewer than three to two CUs
    const int tiles = (B + s.tokens - 1) / s.tokens;
    s.rows = planes == kDensePlanes || s.tokens == 32 || rows64 * tiles * s.slices < 3 * cu_count() / 2 ? 128 : 256;
    s.row_blocks = s.rows == 128 ? rows32 : rows64;
    return s;
}

int gemm_launch(Q4Launch &L, const XhList &xh, const float *ss, float *ws, size_t ws_floats, int planes, int slice_batch,
                hipStream_t st, int *ks_out) {
    if (L.n_mats < 1 || L.n_mats > 3 || L.pair) return l2_fail(L2_ERR_ARG, "q4 gemm: n_mats=%d pair=%d", L.n_mats, L.pair);
    if (L.in % 32 || (planes != kDensePlanes && L.in % L.group_size) || L.batch < 1) return l2_fail(L2_ERR_ARG, "q4 gemm: in=%d batch=%d", L.in, L.batch);
    if (L.e.kind == Q4_EPI_SCATTER_ONLY || L.e.n_scatter) return l2_fail(L2_ERR_ARG, "q4 gemm: no scatter epilogue");
    long rows = 0;
    for (int i = 0; i < L.n_mats; i++) {
        if (L.m[i].out < 8 || L.m[i].out % 8 || (size_t)L.m[i].out * (planes == kDensePlanes ? L.in : L.in / 8) * 4 >= ((size_t)1 << 32))
            return l2_fail(L2_ERR_ARG, "q4 gemm: out=%d in=%d", L.m[i].out, L.in);
        rows += L.m[i].out;
    }
    const GemmShape s = gemm_shape(L, slice_batch, planes);
    // the fp32 kernel keeps its runs' sums where the result goes, which is where the residual lies
    const bool partials = ks_out || (planes == 3 && L.e.kind == Q4_EPI_RESIDUAL);
    if ((s.slices > 1 || partials) && (size_t)s.slices * L.batch * rows > ws_floats)
        return l2_fail(L2_ERR_ARG, "q4 gemm: %d slices of %d x %ld in a workspace of %zu", s.slices, L.batch, rows, ws_floats);
    if (planes == 1)
        L2_TRY(gemm_launch_f16(L, xh, ss, ws, s, partials, st));
    else if (planes == kDensePlanes)
        L2_TRY(launch_dense(L, xh, ss, ws, s, partials, st));
    else
        L2_TRY(launch_fp32(L, xh, ss, ws, s, partials, st));
    if (ks_out) {
        *ks_out = s.slices;
        return L2_OK;
    }
    if (s.slices > 1 || partials) {
        hipLaunchKernelGGL(gemm_reduce_kernel, dim3((unsigned)((rows + 1023) / 1024), L.batch), dim3(256), 0, st, L, ss, ws, s.slices);
        L2_HIP(hipGetLastError());
    }
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
        hipLaunchKernelGGL(gemm_input_kernel<1>, grid, dim3(256), 0, st, A, n, in_p);
    else
        hipLaunchKernelGGL(gemm_input_kernel<3>, grid, dim3(256), 0, st, A, n, in_p);
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
    hipLaunchKernelGGL((gemm_residual_norm_kernel<NP, TRIPS, SL>), dim3(A.B), dim3(1024), lds, st, A, rows);
    L2_HIP(hipGetLastError());
    return L2_OK;
}
template <int NP, int TRIPS>
static int residual_norm(const ResNormPrep &A, hipStream_t st) {
    return A.KS <= 2 ? residual_norm<NP, TRIPS, 2>(A, st) : A.KS <= 8 ? residual_norm<NP, TRIPS, 8>(A, st) : residual_norm<NP, TRIPS, kMaxGemmSlices>(A, st);
}
template <int NP>
static int residual_norm(const ResNormPrep &A, hipStream_t st) {
    return A.out <= 4096 ? residual_norm<NP, 1>(A, st) : A.out <= 8192 ? residual_norm<NP, 2>(A, st) : residual_norm<NP, kTrips>(A, st);
}

int gemm_residual_norm_launch(const ResNormPrep &A, int planes, hipStream_t st) {
    if (A.KS < 1 || A.KS > kMaxGemmSlices || A.out % 32 || A.out > kGemmMaxDim || A.n < 1 || A.n > 3)
        return l2_fail(L2_ERR_ARG, "residual epilogue: %d slices, %d outputs, %d consumers", A.KS, A.out, A.n);
    static_assert(kGemmMaxDim <= kTrips * 4096, "a thread keeps its part of the row in registers");
    return planes == 1 ? residual_norm<1>(A, st) : planes == kDensePlanes ? residual_norm<kDensePlanes>(A, st) : residual_norm<3>(A, st);
}

int gemm_rope_kv_launch(const RopeKvArgs &A, hipStream_t st) {
    if (A.KS < 1 || A.KS > kMaxGemmSlices || A.B < 1 || A.n_heads < A.n_kv_heads)
        return l2_fail(L2_ERR_ARG, "q|k|v epilogue: %d slices, %d tokens", A.KS, A.B);
    const dim3 grid(A.B), block(512);
    if (A.KS <= 2) hipLaunchKernelGGL(gemm_rope_kv_kernel<2>, grid, block, 0, st, A);
    else if (A.KS <= 8) hipLaunchKernelGGL(gemm_rope_kv_kernel<8>, grid, block, 0, st, A);
    else hipLaunchKernelGGL(gemm_rope_kv_kernel<kMaxGemmSlices>, grid, block, 0, st, A);
    L2_HIP(hipGetLastError());
    return L2_OK;
}

template <int NP, int SL>
static int silu(const SiluArgs &A, hipStream_t st) {
    const size_t lds = (size_t)A.n * sizeof(float);
    static LdsLimit limit(48 * 1024);
    L2_TRY(limit.ensure(reinterpret_cast<const void *>(gemm_silu_kernel<NP, SL>), lds));
    hipLaunchKernelGGL((gemm_silu_kernel<NP, SL>), dim3(A.B), dim3(1024), lds, st, A);
    L2_HIP(hipGetLastError());
    return L2_OK;
}
template <int NP>
static int silu(const SiluArgs &A, hipStream_t st) {
    return A.KS <= 2 ? silu<NP, 2>(A, st) : A.KS <= 8 ? silu<NP, 8>(A, st) : silu<NP, kMaxGemmSlices>(A, st);
}

int gemm_silu_launch(const SiluArgs &A, int planes, hipStream_t st) {
    if (A.KS < 1 || A.KS > kMaxGemmSlices || A.n % 32 || A.n > kGemmMaxHidden)
        return l2_fail(L2_ERR_ARG, "silu gate: %d slices, n=%d", A.KS, A.n);
    return planes == 1 ? silu<1>(A, st) : planes == kDensePlanes ? silu<kDensePlanes>(A, st) : silu<3>(A, st);
}
