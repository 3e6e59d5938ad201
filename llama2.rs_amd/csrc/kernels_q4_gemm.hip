// Batched-prefill form of the GPTQ 4-bit linear layer for gfx950: dequantise
// tiles of the packed weights to fp16 in registers and feed them to the matrix
// cores (v_mfma_f32_16x16x32_f16), fp32 accumulate.
//
//   Y[t][o] = sum_k W[o][k] * X[t][k],   W[o][k] = scales[o][k/G] * (nib(qweight[o],k) - z1[o][k/G])
//
// for a chunk of T tokens whose inputs the caller has already brought into this
// layer's g_index order, multiplied by the norm weight where one applies, and
// rounded to fp16 (kernels_gemm.hip).
//
// Tiling.  A wave owns 32 output rows and 16 NT tokens (its dequantised weights are reused for all of them); a block is 8 waves
// side by side over the rows with NT = 8 or 9, one per CU, or 4 waves with NT <= 4, two or three per CU.  K may be cut into KS
// slices; each writes its fp32 partial tile to a workspace and the consumer (or gemm_reduce_kernel) adds them in a fixed order.
//
// Memory.  Everything the K loop reads comes through LDS without touching a register (buffer_load ... lds): the activation
// tiles [tokens][64 k], which the block shares, and, for each wave alone, the packed weights, scales and zero points of its
// rows in units of 128 k (the latter two out of tiles of 32 rows, 144 bytes in two cache lines instead of 36: 64 tokens on six
// layers of 7B 986 -> 938 us).  Tiles are requested one unit ahead, weights two; the only waits are one vmcnt per kind and unit
// and ONE block barrier per unit.  16-byte pieces of a token (a row of weights) lie in the tile permuted by its number, so
// that the reads of 16 lanes meet 16 different banks; the lanes of the load permute their addresses accordingly.
//
// What bounds it, and what the layout of the loop answers (70B's w1|w3, 776 tokens: 928 -> 804 us, 7B's at 511 116 -> 107,
// before the scales and zero points came in tiles):
//   - A SIMD issues an instruction every 4 to 5 cycles from its two waves, and one wave alone gets half of that.  So the
//     vector work (dequantisation of the next step, fold of the group before) stands evenly between the MFMAs of both halves
//     of a step, operands are read from LDS four pairs of MFMAs ahead, and a wave's priority falls with its progress since
//     the last barrier: with equal priorities the older wave of a SIMD ran ahead and waited 30 % of the time at the barrier
//     (1862 cycles per step of 64 k; 1650 now, 1024 of them MFMAs; what a SIMD can issue is 1104, the rest are waits).
//   - Power, and with many tokens that is the bound: a kernel that takes fewer cycles runs at a lower clock.  By cycle stamps in the
//     kernel, launches back to back, 70B's w1|w3, 776 tokens, runs at 1.86 GHz, 7B's, 511, at 1.63 (by counters of a profiled pass,
//     with gaps between the launches, 1.83 and 1.97), all-zero activations at 2.4; nothing but MFMAs gives 1.8 PFLOP/s on such data
//     and 2.4 on zeros.  With 32x32x16 MFMAs a step takes 1512 cycles instead of 1658, and the clock falls to 1.57 GHz: 70B's prompt
//     14.11 -> 14.41 ms, 7B's 11.22 -> 11.55.  So what counts is the work per token: without the reads of activations from LDS the
//     launch would take 24 % less, without the folds 15, without the dequantisation 13.  Hence tiles of 144 tokens, as many as the
//     registers hold, where that makes fewer of them: 70B's 776 tokens 13.97 -> 13.18 ms, six layers of 7B, 280 tokens 1632 -> 1542 us,
//     699 2911 -> 2714, four of 13B, 280, 899 1594 / 3616 -> 1471 / 3518, three of 70B, 419 3196 -> 3052.
//
// Dequant.  (w >> 4i) & 0x000F000F | 0x64006400 is the fp16 pair (1024+n_i,
// 1024+n_{i+4}); subtracting 1024+z1 is exact.  The pairs come out as
// (n0,n4),(n1,n5),(n2,n6),(n3,n7), so X is stored with the same interleave
// inside every 8 consecutive k.  For G >= 64 the matrix cores see the exact
// integers n - z1 and the fp32 scale is applied to the fp32 partial sum of each
// group (one FMA per accumulator element and group), so the only rounding on
// the weight side is none at all; for G = 32 a step of 32 k would be a group,
// and the weights are multiplied by fp16(scale) before the MFMA.
#include "gemm_lds.h"
#include <algorithm>

namespace {

typedef _Float16 h2 __attribute__((ext_vector_type(2)));
typedef _Float16 h8 __attribute__((ext_vector_type(8)));

union A8 {
    h8 v;
    h2 p[4];
    uint32_t u[4];
};

// The constants of a lane's row and group, and the dequantisation of a packed word: 8 nibbles -> 8 fp16 values n - z1
// (exact), times `scale` if SCALED, in the pair order (0,4,1,5,2,6,3,7).  Nibbles 0 and 4 (and 2, 6 after one shift by 8)
// land in the low mantissa bits of the fp16 pair: 1024 + n.  Nibbles 1 and 5 (3, 7) are taken where they stand, four bits
// higher: 1024 + 16 n, and one packed FMA with 1/16 brings them to 64 + n, both exact.  9 instructions per word.
struct Dequant16 {
    uint32_t mask_lo, mask_hi, magic; // 0x000F000F, 0x00F000F0, 0x64006400: opaque, so that and + or is one instruction
    uint32_t c1024, c64;              // fp16 pairs -(1024 + 1), -(64 + 1)
    h2 neg_off, neg_off16;            // -(1024 + z1), -(64 + z1)
    __device__ __forceinline__ Dequant16() : mask_lo(0x000F000Fu), mask_hi(0x00F000F0u), magic(0x64006400u), c1024(0xE401E401u), c64(0xD410D410u) {
        asm("" : "+v"(mask_lo), "+v"(mask_hi), "+s"(magic), "+v"(c1024), "+v"(c64));
    }
    // z1 = zn + 1 in the mantissas of 1024 (steps of 1) and 64 (steps of 1/16)
    __device__ __forceinline__ void zero_point(uint32_t zn) {
        neg_off = __builtin_bit_cast(h2, __umul24(zn, 0x10001u) + c1024);
        neg_off16 = __builtin_bit_cast(h2, __umul24(zn, 0x100010u) + c64);
    }
    // pair i of a word; i = 2 and 3 of the word shifted by 8
    template <bool SCALED>
    __device__ __forceinline__ h2 pair(uint32_t w, int i, h2 scale) const {
        const h2 sixteenth = h2{(_Float16)0.0625f, (_Float16)0.0625f};
        const h2 v = i % 2 == 0 ? __builtin_bit_cast(h2, (w & mask_lo) | magic) + neg_off
                                : __builtin_elementwise_fma(__builtin_bit_cast(h2, (w & mask_hi) | magic), sixteenth, neg_off16);
        return SCALED ? v * scale : v;
    }
};

// LDS of a block of NW waves: four activation tiles, and for each wave three units of 128 k of its 32 rows' weights, scales
// and zero points.
template <int G, int NW>
struct GemmLds {
    static constexpr int kScaleLoads = G == 32 ? 2 : 1; // of 64 words per unit
    static constexpr int kWeights = 32 * 64, kScales = 256 * kScaleLoads;
    static constexpr int kUnit = kWeights + 2 * kScales;
    static constexpr size_t size(int tokens) { return (size_t)4 * tokens * kStepRow + (size_t)NW * 3 * kUnit; }
};

// 32 NW rows rb * 32 NW.. of the matrices of a launch against the 16 NT tokens t0.., K slice ks of KS.
template <int G, int NT, int NW>
__device__ __forceinline__ void q4_gemm_tile(const Q4Launch &L, const XhList &xh_list, const float *__restrict__ ss,
                                             float *__restrict__ ws, int KS, int partials, int rb, int ks, int t0) {
    using S = GemmLds<G, NW>;
    constexpr int TN = 16 * NT, kTile = TN * kStepRow;
    constexpr bool SA = G >= 64; // scale after the group's partial sum
    extern __shared__ __align__(16) char lds[];
    int mi = 0;
    while (mi + 1 < L.n_mats && rb >= L.m[mi].row_blocks) {
        rb -= L.m[mi].row_blocks;
        mi++;
    }
    const Q4Mat &M = L.m[mi];
    const int n_out = M.out, groups = L.groups, B = L.batch, in = L.in;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int r = lane & 15, kg = lane >> 4;
    const int obase = rb * (32 * NW) + wave * 32;
    // this block's slice of K, in units of 128
    const int n_units = in / 128;
    const int u0 = (int)((long)n_units * ks / KS), u1 = (int)((long)n_units * (ks + 1) / KS);

    const uint32_t lds0 = lds_offset(lds);
    const uint32_t wave_at = 4 * kTile + wave * 3 * S::kUnit; // of this wave's weights, scales and zero points

    // Where a lane's pieces come from.  A wave's 1 KB pieces of an activation tile follow each other in the LDS (fewer pieces
    // than waves: the last ones fetch the same), as do the parts of a unit: one base each, the rest in the instructions.
    constexpr int XP = (2 * NT + NW - 1) / NW;
    static_assert(XP <= 4, "the instruction's own offset has 12 bits");
    const int row_tiles = (n_out + 31) >> 5; // of scales and zero points
    const u4v xbuf = biased_buffer(xh_list.p[mi], (size_t)B * in * 2), wbuf = biased_buffer(M.qweight, (size_t)n_out * (in >> 1));
    const u4v sbuf = biased_buffer(M.scales, (size_t)row_tiles * groups * 128), zbuf = biased_buffer(M.qzeros, (size_t)row_tiles * groups * 16);
    const int xfirst = min(wave * XP, 2 * NT - XP);
    uint32_t xoff[XP], woff, soff, zoff;
#pragma unroll
    for (int i = 0; i < XP; i++) { // activations: 8 tokens of 128 bytes, a token's 16-byte pieces permuted by its number
        const int t = (xfirst + i) * 8 + (lane >> 3);
        xoff[i] = (uint32_t)min(t0 + t, B - 1) * (uint32_t)in * 2u + (((lane & 7) ^ piece_xor(t)) << 4) + kBias - i * 1024;
    }
    // weights: 16 rows of 64 bytes, permuted likewise, and 16 more (n_out is whole 32s; a wave beyond takes the last ones again)
    const int wrow = min(obase, n_out - 32);
    woff = (uint32_t)(wrow + (lane >> 2)) * (uint32_t)(in >> 1) + (((lane & 3) ^ (lane >> 4)) << 4) + kBias;
    const uint32_t w_half = (uint32_t)in * 8u - 1024;
    const uint32_t group0 = (uint32_t)(min(obase >> 5, row_tiles - 1) * groups) + (G == 128 ? 0 : lane >> 5); // two groups (G = 128: the same one again)
    soff = group0 * 128u + (lane & 31) * 4u + kBias - S::kWeights;
    zoff = group0 * 16u + (lane >> 3 & 3) * 4u + kBias - S::kWeights - S::kScales;
    // ... and where it reads them
    uint32_t xr[2]; // piece 2 kg + s of token r
#pragma unroll
    for (int s = 0; s < 2; s++) xr[s] = (uint32_t)r * kStepRow + (((2 * kg + s) ^ piece_xor(r)) << 4);
    // the second two of four tiles of 144 tokens lie beyond what an LDS read can have as a constant
    uint32_t xr_far[2] = {xr[0] + 2 * kTile, xr[1] + 2 * kTile};
    if constexpr (NT > 8) asm volatile("" : "+v"(xr_far[0]), "+v"(xr_far[1]));
    const uint32_t wr = wave_at + r * 64 + (((kg >> 1) ^ ((r >> 2) & 3)) << 4) + (kg & 1) * 8; // of a unit's first step; the second's: ^ 32
    const uint32_t sr = wave_at + S::kWeights + kg * 16, zr = wave_at + S::kWeights + ((G == 32 ? (kg >> 1) * 32 : 0) + r) * 4;
    const int zsh = 4 * (r & 7); // obase is a multiple of 8

    const uint32_t x_last = (uint32_t)u1 * 256 - 128, w_last = (uint32_t)(u1 - 1) * 64; // requests past the slice's end take its last piece again
    uint32_t x_at = (uint32_t)u0 * 256, w_at = (uint32_t)u0 * 64;                       // what is requested next
    constexpr int WL = 2 + 2 * S::kScaleLoads;
    auto fetch_x = [&](const int slot, const int i) __attribute__((always_inline)) { // piece i of XP
        LDS_LOAD("x4", lds0 + slot * kTile + xfirst * 1024, i * 1024, xbuf, xoff[i], x_at);
        if (i == XP - 1) x_at = min(x_at + 128, x_last);
    };
    auto fetch_w = [&](const uint32_t unit, const int i) __attribute__((always_inline)) { // piece i of WL
        const uint32_t s_at = w_at * (256 / G), z_at = s_at >> 3;
        const uint32_t to = lds0 + wave_at + unit;
        if (i < 2) LDS_LOAD("x4", to, i * 1024, wbuf, woff, w_at + i * w_half);
        else if (i == 2) LDS_LOAD("", to, S::kWeights, sbuf, soff, s_at);
        else if (i == 3) LDS_LOAD("", to, S::kWeights + S::kScales, zbuf, zoff, z_at);
        else if (i == 4) LDS_LOAD("", to, S::kWeights + 256, sbuf, soff - 256 + 2 * 128, s_at); // G = 32: the second step's groups
        else LDS_LOAD("", to, S::kWeights + S::kScales + 256, zbuf, zoff - 256 + 2 * 16, z_at);
        if (i == WL - 1) w_at = min(w_at + 64, w_last);
    };

    f4v acc[NT][2], accg[NT][2]; // running result of each tile of 16 tokens, two tiles of 16 rows; partial sums of the current group (SA)
#pragma unroll
    for (int n = 0; n < NT; n++)
#pragma unroll
        for (int m = 0; m < 2; m++) acc[n][m] = accg[n][m] = f4v{0.f, 0.f, 0.f, 0.f};
    f4v sv[2] = {}; // scales of the group that accg holds
    auto fold = [&](int n, int m) __attribute__((always_inline)) {
#pragma unroll
        for (int e = 0; e < 4; e++) acc[n][m][e] = fmaf(sv[m][e], accg[n][m][e], acc[n][m][e]);
        asm volatile("" : "+v"(acc[n][m])); // here, and not where the compiler would rather have it
    };

    Dequant16 dq[2];      // of the two rows of a lane
    A8 aq[2][2][2];       // weights of this step and the next: [rows][k]
    uint2 wd[2];          // packed weights of the next step,
    int zw[2];            // their zero points
    float sl[2] = {};     // and scales (G = 32)
    h2 s16[2] = {};
    h8 bq[8];             // activations of eight pairs of MFMAs
    auto read_w = [&](const int par, uint32_t unit) __attribute__((always_inline)) {
        const int gi = G == 128 ? 0 : G == 64 ? par * 128 : par * 256; // of the step's group
        uint32_t w_lds = wr;
        if constexpr (NT > 8) asm volatile("" : "+v"(w_lds)); // one register, not two
#pragma unroll
        for (int m = 0; m < 2; m++) {
            wd[m] = *reinterpret_cast<const uint2 *>(lds + (w_lds ^ (par * 32)) + unit + m * 1024);
            if (G != 128 || par == 0) zw[m] = *reinterpret_cast<const int *>(lds + zr + unit + S::kScales + gi + m * 64);
            if (!SA) sl[m] = *reinterpret_cast<const float *>(lds + zr + unit + gi + m * 64);
        }
    };
    auto constants = [&]() __attribute__((always_inline)) {
#pragma unroll
        for (int m = 0; m < 2; m++) {
            dq[m].zero_point((zw[m] >> zsh) & 15);
            if (!SA) s16[m] = h2{(_Float16)sl[m], (_Float16)sl[m]};
        }
    };
    auto dequant = [&](const int to, const int i) __attribute__((always_inline)) { // piece i of 16
        const int m = i >> 3, k = (i >> 2) & 1;
        uint32_t &w = k ? wd[m].y : wd[m].x;
        if (i % 4 == 2) w >>= 8;
        aq[to][m][k].p[i % 4] = dq[m].template pair<!SA>(w, i % 4, s16[m]);
    };

    // A step of 64 k is 2 NT pairs of MFMAs (two tiles of 16 rows with one of 16 tokens, 32 k), the first half of the token
    // tiles', then the others'.  Between them stands, evenly spread, what the vector unit has to do: the fold of the OTHER
    // tiles' finished group, the next step's weights.  Activations are read, and their registers dealt out, by the pairs' number
    // within the four steps of a round (2 NT is not a multiple of four where NT is odd).
    constexpr int T = 2 * NT, N0 = NT / 2, N1 = NT - N0, H = 2 * N0, AHEAD = 4;
    auto n_of = [](int t) { return t < H ? t % N0 : N0 + (t - H) % N1; };
    auto k_of = [](int t) { return t < H ? t / N0 : (t - H) / N1; };
    auto read_x = [&](const int u, const int t, const int tile) __attribute__((always_inline)) {
        const bool far = NT > 8 && tile >= 2 * kTile;
        bq[(u * T + t) % 8] = *reinterpret_cast<const h8 *>(lds + (far ? xr_far[k_of(t)] + tile - 2 * kTile : xr[k_of(t)] + tile) + n_of(t) * 16 * kStepRow);
    };
    uint32_t unit = 0, unit1 = S::kUnit, unit2 = 2 * S::kUnit; // this unit's place, the next one's and the one's after it
    // Step u of a round of four, which fixes the tiles' places.  Two steps (a unit) go between barriers; in the first of them
    // the two tiles of the next unit are requested, in the places of the one before, and the weights of the one after it.
    auto k_step = [&](const int u) __attribute__((always_inline)) {
        const int par = u & 1, tile = u * kTile, tile1 = (u + 1) % 4 * kTile;
        const bool first = G <= 64 || par == 0, last = G <= 64 || par == 1; // of its group
        const int gi = G == 64 ? par * 128 : 0;
        if (G != 128 || par == 1) constants(); // of the next step
#pragma unroll
        for (int t = 0; t < T; t++) {
            const int n = n_of(t), k = k_of(t);
            if (par == 1 && t == T - AHEAD) {
                // The next tiles: what this wave requested of them has landed, then what everybody has; and all reads of
                // this unit's have come back, so that they may be overwritten.
                asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(WL) : "memory");
            }
            const int behind = (par * T + t + AHEAD) % (2 * T); // MFMA pairs since the barrier
            if (behind % (T / 2) == 0) asm volatile("s_setprio %0" ::"n"(3 - behind / (T / 2)));
            if ((u * T + t) % 4 == 0) { // the next four pairs' activations, behind the arrival of these four's
                __builtin_amdgcn_s_waitcnt(0xC07F); // lgkmcnt(0)
#pragma unroll
                for (int i = t + 4; i < t + 8; i++) read_x(i < T ? u : u + 1, i < T ? i : i - T, i < T ? tile : tile1);
            }
#pragma unroll
            for (int m = 0; m < 2; m++) {
                f4v &c = SA ? accg[n][m] : acc[n][m];
                c = __builtin_amdgcn_mfma_f32_16x16x32_f16(aq[par][m][k].v, bq[(u * T + t) % 8], SA && first && k == 0 ? f4v{} : c, 0, 0, 0);
            }
            if (SA && (t < H ? first : last)) {
                const int j = t < H ? t : t - H, slots = t < H ? H : T - H, folds = t < H ? 2 * N1 : 2 * N0;
#pragma unroll
                for (int f = j * folds / slots; f < (j + 1) * folds / slots; f++) fold((t < H ? N0 : 0) + f / 2, f % 2);
            }
#pragma unroll
            for (int i = t * 16 / T; i < (t + 1) * 16 / T; i++) dequant(par ^ 1, i);
            // the scales of the group that ends with this step, once the folds above no longer need the one before's
#pragma unroll
            for (int m = 0; m < 2; m++)
                if (SA && last && t == (N0 == N1 ? H - 2 + m : H - 1)) sv[m] = *reinterpret_cast<const f4v *>(lds + sr + unit + gi + m * 64);
            if (par == 0) {
                // one request at a time: several in a row wait for the address unit
                constexpr int NL = 2 * XP + WL;
#pragma unroll
                for (int i = t * NL / T; i < (t + 1) * NL / T; i++) {
                    if (i < 2 * XP) fetch_x((u + 2 + i / XP) % 4, i % XP);
                    else fetch_w(unit2, i - 2 * XP);
                }
            }
            __builtin_amdgcn_sched_barrier(0);
        }
        if (par == 0) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(2 * XP + WL) : "memory"); // the next unit's weights
        read_w(par, unit1); // of the step after the next: the same half of the next unit
        if (par == 1) {
            const uint32_t free = unit;
            unit = unit1, unit1 = unit2, unit2 = free;
        }
    };
#pragma unroll
    for (int i = 0; i < WL; i++) fetch_w(0, i);
#pragma unroll
    for (int i = 0; i < 2 * XP; i++) fetch_x(i / XP, i % XP);
#pragma unroll
    for (int i = 0; i < WL; i++) fetch_w(S::kUnit, i);
    asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"(WL) : "memory");
    read_w(0, 0);
    constants();
#pragma unroll
    for (int i = 0; i < 16; i++) dequant(0, i);
    read_w(1, 0);
#pragma unroll
    for (int t = 0; t < 4; t++) read_x(0, t, 0);
    int u = u0;
    for (; u + 2 <= u1; u += 2) {
#pragma unroll
        for (int i = 0; i < 4; i++) k_step(i);
    }
    if (u < u1) k_step(0), k_step(1);
    if (SA) {
#pragma unroll
        for (int n = N0; n < NT; n++) fold(n, 0), fold(n, 1);
    }
    asm volatile("s_waitcnt vmcnt(0)\n\ts_barrier" ::: "memory"); // the LDS is reused below

    // C layout: lane (column r = token, kg), register i -> row 4 kg + i.  Stored as it stands, every store instruction would
    // touch 16 separate 64-byte pieces; instead each wave turns its 32 rows x 32 tokens through LDS (the activation buffers
    // are free now) so that a store instruction writes 8 tokens x 128 contiguous bytes.
    const Q4Epi &E = L.e;
    // workspace of matrix mi starts after those of the matrices before it
    size_t ws_base = 0;
    for (int i = 0; i < mi; i++) ws_base += (size_t)KS * B * L.m[i].out;
    constexpr int kTRow = 36; // floats per staged token row: 32 + 4 pad (16-byte reads of 8 lanes per token)
    float *tile_o = reinterpret_cast<float *>(lds) + wave * 32 * kTRow; // 4.5 KB per wave
    const int tl = lane >> 3, oc = (lane & 7) * 4; // read-back map: token within a pass of 8, 4 rows
#pragma unroll
    for (int nb = 0; nb < (NT + 1) / 2; nb++) {
#pragma unroll
        for (int i = 0; i < 4; i++)
            if (2 * nb + i / 2 < NT) *reinterpret_cast<f4v *>(&tile_o[(i / 2 * 16 + r) * kTRow + i % 2 * 16 + kg * 4]) = acc[2 * nb + i / 2][i % 2];
        // the wave reads what the wave wrote: no block barrier, the LDS queue of a wave is in order
#pragma unroll
        for (int pass = 0; pass < (2 * nb + 1 < NT ? 4 : 2); pass++) {
            const int tt = pass * 8 + tl;
            float4 v = *reinterpret_cast<const float4 *>(&tile_o[tt * kTRow + oc]);
            const int t = t0 + nb * 32 + tt;
            const int o = obase + oc;
            if (t >= B || o >= n_out) continue;
            const size_t row = (size_t)t * n_out;
            if (KS > 1 || partials) { // partial tile of this K slice
                float *at = ws + ws_base + ((size_t)ks * B + t) * n_out + o;
                if (partials > 1) __builtin_nontemporal_store(f4v{v.x, v.y, v.z, v.w}, reinterpret_cast<f4v *>(at));
                else store_through(reinterpret_cast<float4 *>(at), v);
                continue;
            }
            const float scale_t = ss ? ss[t] : 1.0f;
            v.x *= scale_t, v.y *= scale_t, v.z *= scale_t, v.w *= scale_t;
            if (E.kind == Q4_EPI_RESIDUAL) {
                const float4 rr = *reinterpret_cast<const float4 *>(E.res + row + o);
                v.x += rr.x;
                v.y += rr.y;
                v.z += rr.z;
                v.w += rr.w;
            }
            *reinterpret_cast<float4 *>(M.y + row + o) = v;
        }
    }
}

// One block per work item.  A unit is a row block and a slice of K.  The first `units` of them, and `extra` tiles of the next one, go in
// tiles of 16 NT tokens; what whole rounds of blocks leave over goes in tiles of `width`; then come the last tokens of the first units,
// where they are no more than half a tile and 64.  A tile takes as many 16s as it needs, two at least, and costs those and the
// dequantisation of its weights (128, 64, 32 tokens of 70B's w1: 119, 75, 62 us).
template <int G, int NT, int NW>
__global__ __launch_bounds__(64 * NW, NT > 4 ? 2 : 1) void q4_gemm_kernel(const Q4Launch L, const XhList xh, const float *__restrict__ ss,
                                                      float *__restrict__ ws, int KS, int partials, int row_blocks, int t_full, int units, int extra,
                                                      int width) {
    constexpr int TN = 16 * NT, CHUNK = 8;
    const int b = blockIdx.x, whole = units * t_full + extra, per = (L.batch + width - 1) / width;
    const int head = extra ? (L.batch - extra * TN + width - 1) / width : 0; // of the unit that has tiles of both kinds
    const int begun = units + (extra > 0), left = row_blocks * KS - begun, other = head + left * per;
    int unit, t0, n;
    if (b < whole) { // 8 row blocks at a time, token tile by token tile: what runs on an XCD shares tiles and weights
        int item = xcd_item(b, whole);
        const bool of_next = item >= units * t_full;
        const int next_tile = item - units * t_full;
        if (of_next) item = 0;
        const int first = item / (row_blocks * t_full) * row_blocks, c = (item -= first * t_full) / (CHUNK * t_full);
        const int of = min(CHUNK, min(row_blocks, units - first) - c * CHUNK), at = item - c * CHUNK * t_full, tt = at / of;
        unit = of_next ? units : first + c * CHUNK + at - tt * of, t0 = (of_next ? next_tile : tt) * TN, n = L.batch - t0;
    } else if (b < whole + other) {
        const int item = xcd_item(b - whole, other) - head, c = max(item, 0) / (CHUNK * per), of = min(CHUNK, max(left - c * CHUNK, 1));
        const int at = item - c * CHUNK * per, tt = at / of;
        if (item < 0) unit = units, t0 = extra * TN + (item + head) * width;
        else unit = begun + c * CHUNK + at - tt * of, t0 = tt * width;
        n = min(L.batch - t0, width);
    } else {
        unit = xcd_item(b - whole - other, gridDim.x - whole - other), t0 = t_full * TN, n = L.batch - t0;
    }
    const int ks = unit / row_blocks, rb = unit - ks * row_blocks;
    switch (min((n + 15) >> 4, NT)) { // tiles of 16 tokens that it takes
#define GEMM_TILE(t) \
    case t: \
        if constexpr (t <= NT) q4_gemm_tile<G, t, NW>(L, xh, ss, ws, KS, partials, rb, ks, t0); \
        break
        case 1:
        GEMM_TILE(2);
        GEMM_TILE(3);
        GEMM_TILE(4);
        GEMM_TILE(5);
        GEMM_TILE(6);
        GEMM_TILE(7);
        GEMM_TILE(8);
        GEMM_TILE(9);
#undef GEMM_TILE
    }
}

// How the blocks of a launch are dealt out (q4_gemm_kernel), with what it takes: a tile of w tokens 43 + 0.594 w (of 70B's w1: 62,
// 75 and 119 us for 32, 64 and 128).
struct GemmPlan {
    int tokens, t_full, units, extra, width, blocks;
    float cost;
};

// What whole rounds of tiles leave over goes in narrower ones, the narrowest with which these, and the last tokens of the other units,
// fit one round: 7B's w1|w3, 511 tokens, 344 tiles on 256 CUs 123 -> 112 us with 64; with 224 narrow tiles behind 64 left over (70B's, 776)
// they took 822 and whole tiles 804.  With several slices too: four layers of 13B, group 64, 399 tokens 2192 -> 2135, six of 7B, group 32, 249
// tokens 1656 -> 1610.  Of the blocks of four waves too, where some CUs have two and others one (two take twice as long as one):
// six layers of 7B, 64, 99, 128 tokens 918 / 1075 / 1120 -> 903 / 1047 / 1080, four of 13B, 128 1057 -> 1041; with more of them than
// two per CU whole tiles (70B, 179 1965 against 1978).  Of 32 to 112 tokens in steps of 16 against 96 and 64 alone: 70B's 776 13.47 ->
// 13.28 ms; six layers of 7B, 199, 511, 776 1330 / 2180 / 3260 -> 1298 / 2163 / 3230; four of 13B, 199 1280 -> 1230; 350 1735, 1740.
// None above 64 beside another pass, which has a use for the CUs that a round
// leaves: four layers of 13B, 300 and 399 tokens in chunks of 256 1359 / 1742 -> 1302 / 1713, six of 7B, 899 in chunks of 128 3891 -> 3812.
static GemmPlan plan_tiles(int TN, int all, int B, bool beside) {
    const int rest = B % TN, most = std::min(TN / 2, 64), t_full = B / TN + (rest > most), narrow = rest > 0 && rest <= most;
    const int tiles = all * t_full, cus = cu_count();
    auto tile_cost = [](int w) { return 43.f + 0.594f * w; };
    // whole tiles, and the last tokens' where a round leaves room
    const float whole = tile_cost(TN), last = narrow ? tile_cost(std::max((rest + 15) / 16 * 16, 32)) : 0.f;
    const int room = narrow && tiles % cus ? (cus - tiles % cus) * (int)(whole / last) : 0;
    GemmPlan p{TN, t_full, all, 0, TN, tiles + narrow * all,
               (tiles + cus - 1) / cus * whole + (narrow * all > room ? (narrow * all - room + cus - 1) / cus * last : 0.f)};
    if ((TN > 64 || (TN == 64 && tiles > cus && tiles < 2 * cus)) && tiles % cus) {
        // Whole tiles for full rounds: of these units, and `done` of the next one, without which those of 64 may not fit (three layers of
        // 70B, 399 tokens in chunks of 128: 2785 -> 2735).  With four waves none of the next one: 70B, 176 tokens 1405, with them 1433.
        const int rounds = tiles / cus * cus, begun = rounds / t_full, done = TN > 64 ? rounds % t_full : 0;
        for (int w = beside ? most : TN - 16; w >= 32; w -= 16) {
            const int n = (done ? (B - done * TN + w - 1) / w : 0) + (all - begun - (done > 0)) * ((B + w - 1) / w) + narrow * begun;
            const float cost = tiles / cus * whole + std::max(tile_cost(w), begun ? last : 0.f);
            if (n <= cus && cost < p.cost) p = {TN, t_full, begun, done, w, begun * t_full + done + n, cost};
        }
    }
    return p;
}

static GemmPlan plan_launch(const GemmShape &s, int B, bool beside) {
    const int all = s.row_blocks * s.slices;
    const GemmPlan p = plan_tiles(s.tokens, all, B, beside);
    if (s.tokens < 128) return p;
    // Tiles of 144 tokens where they take less (and not about the same: 7B, 899 tokens, a cost of 1.00, 3485 -> 3523 us for six layers).
    const GemmPlan wide = plan_tiles(144, all, B, beside);
    return wide.cost < 0.98f * p.cost ? wide : p;
}

template <int G, int NT, int NW>
int launch_gemm(Q4Launch &L, const XhList &xh, const float *ss, float *ws, const GemmShape &s, const GemmPlan &p, int partials, hipStream_t st) {
    constexpr int TN = 16 * NT;
    for (int i = 0; i < L.n_mats; i++) L.m[i].row_blocks = (L.m[i].out + 32 * NW - 1) / (32 * NW);
    // Partial tiles past the L2 (what a launch leaves dirty there is written back at its end, see store_through), and past the memory-side
    // cache too where they would fill it: up to 100 MB their consumer finds them there.  Above 16, 64, 100 MB: 7B, 511 tokens 11270 /
    // 11032 / 11038 us; six layers of 7B, 299, 699, 899 1700 / 2768 / 3570, 1666 / 2721 / 3537 and 1673 / 2720 / 3514; four of 13B, 249
    // 1364 / 1351 / 1346; none past it: 899 tokens of 13B 3606 -> 3631, 70B's 776 (178 MB of w1|w3) 13.39 -> 13.43 ms.
    size_t bytes = 0;
    for (int i = 0; i < L.n_mats; i++) bytes += (size_t)s.slices * L.batch * L.m[i].out * 4;
    if (partials && bytes > ((size_t)100 << 20)) partials = 2;
    const dim3 grid(p.blocks), block(64 * NW);
    // the tiles, or the output staging tiles of the epilogue (32 x 36 floats per wave)
    const size_t lds = std::max(GemmLds<G, NW>::size(TN), (size_t)NW * 32 * 36 * sizeof(float));
    static LdsLimit limit(48 * 1024);
    L2_TRY(limit.ensure(reinterpret_cast<const void *>(q4_gemm_kernel<G, NT, NW>), lds));
    l2_launch((q4_gemm_kernel<G, NT, NW>), grid, block, lds, st, L, xh, ss, ws, s.slices, partials, s.row_blocks, p.t_full, p.units, p.extra, p.width);
    L2_HIP(hipGetLastError());
    return L2_OK;
}

template <int G>
int launch_gemm_g(Q4Launch &L, const XhList &xh, const float *ss, float *ws, const GemmShape &s, int partials, bool beside, hipStream_t st) {
    const GemmPlan p = plan_launch(s, L.batch, beside);
    switch (p.tokens) {
        case 32: return launch_gemm<G, 2, 4>(L, xh, ss, ws, s, p, partials, st);
        case 64: return launch_gemm<G, 4, 4>(L, xh, ss, ws, s, p, partials, st);
        case 128: return launch_gemm<G, 8, 8>(L, xh, ss, ws, s, p, partials, st);
        case 144: return launch_gemm<G, 9, 8>(L, xh, ss, ws, s, p, partials, st);
    }
    return l2_fail(L2_ERR_ARG, "q4 gemm: token tile");
}

} // namespace

GemmShape gemm_shape_f16(const Q4Launch &L, int slice_batch) {
    GemmShape s{};
    const int B = L.batch;
    s.rows = 128;
    for (int i = 0; i < L.n_mats; i++) s.row_blocks += (L.m[i].out + 127) / 128;
    // K slices: as many as keep the grid within one round of 2 blocks per CU, of two units or more, at most 4; chunks of up
    // to 64 tokens, whose partial tiles are small, at most 8.  (More slices fill the chip when a launch runs alone, but every
    // one is a partial tile that the consumer reads back.  8 for 4, 32 tokens: two layers of 7B, group 128, 226 -> 202 us, of
    // 70B, group 64, 492 -> 450; 16: 210 and 456.)  They depend on the chunk and not on the pass: its bits must not.
    auto tile = [](int n) { return n >= 192 ? 128 : n > 32 ? 64 : 32; };
    const int t_tiles = (slice_batch + tile(slice_batch) - 1) / tile(slice_batch);
    s.slices = std::max(1, std::min({2 * cu_count() / (s.row_blocks * t_tiles), slice_batch <= 64 ? 8 : 4, L.in / 256}));
    // From 192 tokens on a block is 256 rows x 128 tokens, one per CU (every weight is dequantised once per 128 tokens instead
    // of twice, every token tile read once per 256 rows), where that gives work to at least half the CUs; below, or for a small
    // model, 128 rows x 64 tokens, two or three blocks per CU.  Two layers, 256 x 128 / 128 x 64, us: 7B, group 128, 192 tokens
    // 401 / 395, 250 431 / 450, 511 669 / 768; 13B 192 507 / 521; 70B, group 64, 250 1314 / 1371; dim 1024, 511 233 / 217.
    s.tokens = tile(B);
    if (s.tokens == 128) {
        int rows = 0;
        for (int i = 0; i < L.n_mats; i++) rows += (L.m[i].out + 255) / 256;
        if (rows * ((B + 127) / 128) * s.slices >= cu_count() / 2) s.rows = 256, s.row_blocks = rows;
        else s.tokens = 64;
    }
    return s;
}

GemmTiles gemm_tiles_f16(const GemmShape &s, int B, bool beside) {
    const GemmPlan p = plan_launch(s, B, beside);
    return {s.rows, p.tokens, s.slices, p.blocks, p.units * p.t_full + p.extra, p.width, B > p.t_full * p.tokens ? B - p.t_full * p.tokens : 0, p.extra > 0};
}

int gemm_launch_f16(Q4Launch &L, const XhList &xh, const float *ss, float *ws, const GemmShape &s, int partials, bool beside, hipStream_t st) {
    if (L.in % 128 != 0) return l2_fail(L2_ERR_ARG, "q4 gemm: in=%d must be a multiple of 128", L.in);
    if (L.group_size >= 64 && (L.in / L.group_size) % 2 != 0)
        return l2_fail(L2_ERR_ARG, "q4 gemm: in=%d is an odd number of groups of %d", L.in, L.group_size);
    for (int i = 0; i < L.n_mats; i++)
        if (L.m[i].out % 32 != 0) return l2_fail(L2_ERR_ARG, "q4 gemm: out=%d must be a multiple of 32", L.m[i].out);
    switch (L.group_size) {
        case 32: return launch_gemm_g<32>(L, xh, ss, ws, s, partials, beside, st);
        case 64: return launch_gemm_g<64>(L, xh, ss, ws, s, partials, beside, st);
        case 128: return launch_gemm_g<128>(L, xh, ss, ws, s, partials, beside, st);
    }
    return l2_fail(L2_ERR_ARG, "q4 gemm: group size %d", L.group_size);
}
