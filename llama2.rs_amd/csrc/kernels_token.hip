// All layers of a decode step (B = 1) in one launch: every compute unit holds one block for the whole step, and the vectors that
// layers hand on go from block to block through memory while the kernel runs (gfx950, wave64).
//
// Five vectors per layer are handed on: q|k|v, attention's output, the residual stream behind wo, the gated hidden vector and the
// residual stream behind w2.  A dependent launch spends some 3.5 us before its first FMA (the end of the one before it, arguments, x,
// staging); here a vector is in the other blocks' LDS 1.5 to 2.5 us after the last block has stored its part, and the weights of the
// next phase are on their way meanwhile.  Whole steps (kernel and classifier), the layers' own launches -> this, at position 30: three layers of 1024
// inputs 67.7 -> 51.2 us, four of 7B 219.7 -> 206.6, three of 13B 243 -> 227.9; 7B's 96 tokens 103.5 -> 95 ms, which is more, since the
// host's launches are not the kernels' length either.  What bounds it: a layer of 7B is 30 us, 18.5 of them in the rows of its four
// phases (w1|w3 at 5.9 TB/s, wo 3 us for 9 MB) and 11.5 between them: the exchanges, attention, and the 0.5 to 1.5 us by which blocks finish
// apart, all waiting for the last.  Rows that wait less (more of them asked for before x or as soon as it is there, wo's in front of
// attention's sums) take longer, because x, or q, is then behind them; so do keys and values brought into LDS before q is there:
// what attention takes behind 300 positions (3 us a layer more than behind 30) is what one compute unit can fetch.
//
// The exchange.  A place is "absent" (all ones, which as a float is one of the NaNs) until its value is stored; a consumer loads, at
// agent scope, until no place of its piece is absent.  The value is its own flag, every place is 4 bytes and stored once, so no order among
// stores is relied on.  Two sets of places are used in turn: a step's kernel empties the other one.
//   * A block stores a contiguous piece, and the consumer applies its act-order on the way into LDS.  With the order applied by the
//     producer, as the launches do it, every cache line has stores from 32 blocks while all blocks look at it: 4 us more per exchange.
//   * Loads of a compute unit return in the order in which they were asked for, so x is behind the weights that were asked for before it;
//     three rows per wave are.  Four: 7B 212.7 -> 222.
//   * Waits end: after `limit` looks (some 0.1 s) a wave gives up, says so, and the others follow; the host then does the steps again with
//     the layers' own launches.  That is for blocks that do not find room because others' kernels hold the device; blocks of one launch find
//     room together on an idle one, and the host keeps two of these kernels from running at once.
//
// The sums are those of the launches (kernels_q4_stream.hip, attn_decode_kernel), bit for bit: a lane has the same chunk, a row the same
// partial sums in the same order, the sum of squares is taken by as many waves, and rows that stand behind the loop of a launch are
// rounded as they are there (TokWalk::behind).  Which wave has a row does not matter to its bits.
#include <type_traits>

#include "q4_common.h"

namespace {

using namespace q4;

constexpr int kWaves = kTokenWaves, kThreads = kWaves * 64;
constexpr int kRows = kTokenRows;          // rows of a wave in flight
constexpr int HS = 128, HALF = 64;         // head size
constexpr float kNoScore = -1e30f;         // as in decode attention (kernels_attn.hip)
constexpr uint32_t kAbsent = 0xFFFFFFFFu;  // a value that has not been handed on yet
constexpr int kLooksPerCheck = 64;         // looks between two checks of whether to give up

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef uint16_t u16x4 __attribute__((ext_vector_type(4)));
typedef const __attribute__((address_space(4))) TokModel *ArgsPtr; // read through the scalar cache
typedef const __attribute__((address_space(4))) TokPhase *PhasePtr;
template <class T>
using Global = __attribute__((address_space(1))) T *;
typedef Global<float> Floats;
template <class T>
__device__ __forceinline__ Global<T> global(uint64_t address) {
    return (Global<T>)(uintptr_t)address;
}

__device__ __forceinline__ u32x4 load_agent(Floats p) { return __builtin_amdgcn_global_load_b128((Global<u32x4>)p, "agent"); }
__device__ __forceinline__ uint32_t load_agent1(Floats p) {
    return __hip_atomic_load((Global<uint32_t>)p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ bool is_there(u32x4 v) { return v.x != kAbsent && v.y != kAbsent && v.z != kAbsent && v.w != kAbsent; }

// A value handed on.  The pattern that means "absent" is a NaN; any other NaN stands for it.
__device__ __forceinline__ void hand_on(Floats p, float v) {
    uint32_t b = __builtin_bit_cast(uint32_t, v);
    if (b == kAbsent) b = 0x7FFFFFFFu;
    __hip_atomic_store((Global<uint32_t>)p, b, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Whether a wave that has looked `looks` times stops waiting: after `limit` looks, or because another one has.
__device__ __forceinline__ bool gives_up(ArgsPtr A, int looks) {
    if (looks >= A->limit) {
        __hip_atomic_store(global<int>(A->failed), 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __hip_atomic_store(global<int>(A->failed_host), 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
        return true;
    }
    return __builtin_amdgcn_readfirstlane(__hip_atomic_load(global<int>(A->failed), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) != 0;
}

struct RowData {
    u32x4 w;
    float s;
    int32_t z;
};

__device__ __forceinline__ float chunk_sum(const float (&s4)[8]) {
#pragma clang fp contract(off)
    return ((s4[0] + s4[1]) + (s4[2] + s4[3])) + ((s4[7] + s4[6]) + (s4[5] + s4[4]));
}

typedef const __attribute__((address_space(4))) TokWalk *WalkPtr;

// The lane's part of a row's addresses: its chunk of 32 nibbles and that chunk's group.
struct LaneAt {
    int w, g;
};
__device__ __forceinline__ LaneAt lane_at(const TokWalk &k, int gshift, int lane) {
    const int c = min(k.kslice * 64 + lane, k.C - 1);
    return {c << 4, (c >> gshift) << 2};
}

// A projection's arrays in one layer, as one buffer: a row is then a scalar offset and the lane a vector offset, with no 64-bit arithmetic.
struct Arrays {
    __amdgpu_buffer_rsrc_t r;
    int scales_at, zeros_at;
};
__device__ __forceinline__ Arrays arrays_of(ArgsPtr A, int mat, int l) {
    const auto *m = &A->m[mat];
    void *const p = (void *)(uintptr_t)(m->qweight + (uint64_t)l * m->stride);
    return {__builtin_amdgcn_make_buffer_rsrc(p, 0, -1, 0x00020000), (int)m->scales_at, (int)m->zeros_at};
}

constexpr int kOnce = 2; // non-temporal: weights are read once per token
__device__ __forceinline__ void fetch(const TokWalk &k, const Arrays &a, const LaneAt &at, int i, RowData &d) {
    const int o = min(k.first + i * k.stride, k.last);
    d.w = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(a.r, at.w, (int)((uint32_t)(o * k.C) << 4), kOnce));
    d.s = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(a.r, at.g, a.scales_at + ((o * k.groups) << 2), kOnce));
    d.z = (int32_t)__builtin_amdgcn_raw_buffer_load_b32(a.r, at.g, a.zeros_at + (((o >> 3) * k.groups) << 2), kOnce);
}

// The first rows.
__device__ __forceinline__ void ask(const TokWalk &k, const Arrays &a, const LaneAt &at, RowData (&pipe)[kRows]) {
#pragma unroll
    for (int u = 0; u < kRows; u++) {
        pipe[u] = RowData{}; // what was there is not kept
        if (u < k.steps) fetch(k, a, at, u, pipe[u]);
    }
}

// Where a thread's elements of the input go (places in LDS), and the norm weights of those: they do not depend on the step.
struct Places {
    u16x4 a[4], b[2];
    f32x4 g[2];
};
template <int PH>
__device__ __forceinline__ void places_of(ArgsPtr A, int l, int mat, int tid, Places &t) {
    constexpr bool kNorm = PH == TOK_QKV || PH == TOK_W13;
    const int n4 = A->phase[PH].n4;
    const auto order = [&](int i) { return (Global<const u16x4>)(global<const uint16_t>(A->slots[i]) + (size_t)l * (4 * n4)); };
    const Global<const u16x4> a = order(PH == TOK_QKV ? mat : PH == TOK_WO ? 6 : PH == TOK_W13 ? 3 : 5), b = order(4);
    const Global<const f32x4> g = (Global<const f32x4>)(global<const float>(PH == TOK_W13 ? A->rms_ffn : A->rms_att) + (size_t)l * A->dim);
#pragma unroll
    for (int u = 0; u < (PH == TOK_W2 ? 4 : 2); u++) {
        const int j4 = u * kThreads + tid;
        t.a[u] = u16x4{0, 0, 0, 0};
        if constexpr (kNorm) t.g[u] = f32x4{0.f, 0.f, 0.f, 0.f};
        if constexpr (PH == TOK_W13) t.b[u] = u16x4{0, 0, 0, 0};
        if (j4 < n4) {
            t.a[u] = a[j4];
            if constexpr (kNorm) t.g[u] = g[j4];
            if constexpr (PH == TOK_W13) t.b[u] = b[j4];
        }
    }
}

template <int DS>
__global__ __launch_bounds__(kThreads) void token_layers_kernel(const TokArgs S) {
    constexpr int VD = HS / DS, VE = VD / 16;
    extern __shared__ __align__(16) float lds[]; // staged x (two of them for w1|w3), then the rows' partial sums
    __shared__ __align__(16) float red[kWaves];
    __shared__ float qs[HS], kvnew[2][HS];
    __shared__ __align__(16) float comb[8][HS + 4];
    int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    uint64_t args = (uint64_t)(uintptr_t)S.model;
    ArgsPtr A = (ArgsPtr)(uintptr_t)args;
    const int n_layers = A->n_layers;

    // The block's part of attention: one query head's slice of the outputs, blocks dealt kv head by kv head.
    const int n_kv = A->n_kv_heads, qg = A->n_heads / n_kv;
    const int kvh = blockIdx.x % n_kv, jh = blockIdx.x / n_kv % qg, slice = blockIdx.x / n_kv / qg;
    const bool attends = slice < DS;
    const int head = kvh * qg + jh;
    float rot_c = 0.f, rot_s = 0.f;
    if (attends) {
        rot_c = global<const float>(A->cos_t)[(size_t)S.pos * HALF + lane];
        rot_s = global<const float>(A->sin_t)[(size_t)S.pos * HALF + lane];
    }

    // What this wave does in a phase.
    const auto walk_of = [&](int ph) __attribute__((always_inline)) {
        const WalkPtr p = (WalkPtr)(uintptr_t)A->walks + (ph * gridDim.x + blockIdx.x) * kWaves + wave;
        return TokWalk{p->mat, p->first, p->stride, p->last, p->steps, p->r0, p->n, p->part_row, p->kslice, p->C, p->groups, p->behind, p->behind_early, p->late, {}};
    };
    const auto at_of = [&](const TokWalk &k, int ph) __attribute__((always_inline)) { return lane_at(k, A->phase[ph].gshift, lane); };
    RowData pipe[kRows];
    Places places;
    TokWalk walk = walk_of(TOK_QKV);
    Arrays arrays = arrays_of(A, walk.mat, 0);
    places_of<TOK_QKV>(A, 0, walk.mat, tid, places);
    ask(walk, arrays, at_of(walk, TOK_QKV), pipe);
    // The step's token (as embed_kernel takes it), whose row of the table is the first layer's input.
    int token = S.src.token;
    if (S.src.tokens) token = S.src.tokens[0];
    else if (S.src.prev) token = (int)(S.src.prev[0] & 0xFFFFFFFFull);
    token = __builtin_amdgcn_readfirstlane(token);
    const Floats row0 = (Floats)S.emb + (size_t)token * A->dim;
    if (blockIdx.x == 0 && tid == 0) {
        if (S.src.prev) S.src.record[0] = token;
        if (S.amax) S.amax[0] = 0ull;
    }

    // The last threads finish the block's rows, one each; the residual stream of wo's and w2's rows stays in a register of theirs.
    float res = 0.f;
    {
        const TokWalk k = walk_of(TOK_WO);
        const int fin = tid - (kThreads - (k.n + 63) / 64 * 64);
        if (fin >= 0 && fin < k.n) res = row0[k.r0 + fin];
    }

    const auto phase = [&](auto which, const int l) __attribute__((always_inline)) {
        constexpr int PH = decltype(which)::value, NEXT = (PH + 1) & 3;
        constexpr bool kNorm = PH == TOK_QKV || PH == TOK_W13, kPair = PH == TOK_W13;
        // nothing that a phase computes from these is kept over all phases in registers
        asm volatile("" : "+v"(tid), "+v"(lane), "+s"(args));
        A = (ArgsPtr)(uintptr_t)args;
        const PhasePtr q = &A->phase[PH];
        const bool first = PH == TOK_QKV && l == 0, last = PH == TOK_W2 && l == n_layers - 1;
        const TokWalk k = walk, next = walk_of(NEXT);
        const Arrays arr = arrays, next_arr = arrays_of(A, next.mat, PH == TOK_W2 && !last ? l + 1 : l);
        const LaneAt next_at = at_of(next, NEXT);
        const int next_steps = last || (PH == TOK_QKV && next.late) ? 0 : next.steps;
        const Floats E = (Floats)S.handed + (size_t)l * A->layer_floats;
        float *const part = lds + A->part_at;
        const int dim = A->dim, n4 = q->n4, nwk = q->nwk, PW = nwk * 4, nwx = q->nwx, vec_floats = q->vec_floats;
        const int kslice = k.kslice;
        const LaneAt at = at_of(k, PH);
        // where the block's rows go
        const Floats out = last ? (Floats)S.x
                                : E + (PH == TOK_QKV ? A->at_qkv + (k.mat == 0 ? 0 : k.mat == 1 ? dim : dim + A->kv_dim)
                                       : PH == TOK_WO ? A->at_xm
                                       : PH == TOK_W13 ? A->at_hg
                                                       : A->layer_floats);
        asm volatile("" ::"s"(out));

        // x into LDS, in this phase's act-order, in chunks of 32 padded to 36.  It comes in its natural order: a block hands on a piece of
        // its own (with the order applied there, 32 blocks write into every cache line that all look at, some 4 us each time).
        float *const raw = lds + 2 * vec_floats;
        if constexpr (kNorm) {
            const Floats xp = first ? row0 : kPair ? E + A->at_xm : E;
            u32x4 v[2];
            for (int looks = 0;;) {
                bool ok = true;
#pragma unroll
                for (int u = 0; u < 2; u++) {
                    const int j4 = u * kThreads + tid;
                    v[u] = u32x4{0, 0, 0, 0};
                    if (j4 < n4) v[u] = load_agent(xp + 4 * j4);
                    ok = ok && is_there(v[u]);
                }
                if (__all(ok) || first) break;
                if (++looks % kLooksPerCheck == 0 && gives_up(A, looks)) break;
                __builtin_amdgcn_s_sleep(1);
            }
#pragma unroll
            for (int u = 0; u < 2; u++) {
                if (u * kThreads + tid < n4) {
                    const f32x4 f = __builtin_bit_cast(f32x4, v[u]);
#pragma unroll
                    for (int e = 0; e < 4; e++) {
                        const float w = f[e] * places.g[u][e];
                        lds[places.a[u][e]] = w;
                        raw[places.a[u][e]] = f[e];
                        if (kPair) lds[vec_floats + places.b[u][e]] = w;
                    }
                }
            }
        } else {
            const Floats xp = E + (PH == TOK_WO ? A->at_att : A->at_hg);
            const Global<const u16x4> to = (Global<const u16x4>)(global<const uint16_t>(A->slots[PH == TOK_WO ? 6 : 5]) + (size_t)l * (4 * n4));
            constexpr int kBatch = PH == TOK_WO ? 2 : 4;
            for (int base = 0; base < n4; base += kBatch * kThreads) {
                u32x4 v[kBatch];
                if (base > 0) {
#pragma unroll
                    for (int u = 0; u < kBatch; u++)
                        if (base + u * kThreads + tid < n4) places.a[u] = to[base + u * kThreads + tid];
                }
                for (int looks = 0;;) {
                    bool ok = true;
#pragma unroll
                    for (int u = 0; u < kBatch; u++) {
                        const int j4 = base + u * kThreads + tid;
                        v[u] = u32x4{0, 0, 0, 0};
                        if (j4 < n4) v[u] = load_agent(xp + 4 * j4);
                        ok = ok && is_there(v[u]);
                    }
                    if (__all(ok)) break;
                    if (++looks % kLooksPerCheck == 0 && gives_up(A, looks)) break;
                    __builtin_amdgcn_s_sleep(1);
                }
#pragma unroll
                for (int u = 0; u < kBatch; u++) {
                    if (base + u * kThreads + tid < n4) {
                        const f32x4 f = __builtin_bit_cast(f32x4, v[u]);
#pragma unroll
                        for (int e = 0; e < 4; e++) lds[places.a[u][e]] = f[e];
                    }
                }
            }
        }
        __syncthreads();
        if (kNorm && wave < nwx) { // the sum of squares, in the order of the launches that stage x by so many waves
            const int T = nwx * 64;
            float ssq = 0.f;
#pragma unroll
            for (int u = 0; u < 2; u++) {
                const int j4 = u * T + tid;
                if (j4 < n4) {
                    const float4 f = *reinterpret_cast<const float4 *>(&raw[(j4 >> 3) * kChunkPad + (j4 & 7) * 4]);
                    ssq = fmaf(f.x, f.x, ssq);
                    ssq = fmaf(f.y, f.y, ssq);
                    ssq = fmaf(f.z, f.z, ssq);
                    ssq = fmaf(f.w, f.w, ssq);
                }
            }
            ssq = wave_sum(ssq);
            if (lane == 0) red[wave] = ssq;
        }

        // the rows of the wave
        if (k.steps > 0) {
            float x[32], sx = 0.f;
            {
#pragma clang fp contract(off)
                const int c = kslice * 64 + lane;
                const float4 *p = reinterpret_cast<const float4 *>(&lds[(k.part_row > 0 ? vec_floats : 0) + c * kChunkPad]);
#pragma unroll
                for (int i = 0; i < 8; i++) {
                    const float4 v = p[i];
                    x[4 * i + 0] = v.x, x[4 * i + 1] = v.y, x[4 * i + 2] = v.z, x[4 * i + 3] = v.w;
                }
                if (kslice * 64 + 63 >= k.C) { // beyond the vector's end LDS holds anything
#pragma unroll
                    for (int i = 0; i < 32; i++) x[i] = c < k.C ? x[i] : 0.f;
                }
                float s4[8];
#pragma unroll
                for (int i = 0; i < 8; i++) s4[i] = (x[4 * i] + x[4 * i + 1]) + (x[4 * i + 2] + x[4 * i + 3]);
                if (!kNorm && q->direct) {
#pragma unroll
                    for (int i = 0; i < 8; i++) sx += s4[i];
                } else {
                    sx = chunk_sum(s4);
                }
            }
            const float nsx = -sx;
            float *to = part + (k.part_row + k.first - k.r0) * PW + kslice * 4 + (lane >> 4);
            const auto row = [&](int i, RowData &d, bool refill, auto whole) __attribute__((always_inline)) {
                const int o = k.first + i * k.stride;
                const int zn = (int)(((uint32_t)d.z >> (4 * (o & 7))) & 15u);
                const float sum = fmaf(chunk_dot(__builtin_bit_cast(uint4, d.w), x), 512.0f, fmaf((float)zn, nsx, nsx)), scale = d.s;
                const bool behind = !whole && ((k.behind >> i) & 1);
                float v;
                {
#pragma clang fp contract(off)
                    const float mine = scale * sum, other = dpp_xchg<0xB1>(mine);
                    v = behind ? fmaf(scale, sum, other) : mine + other;
                }
                asm volatile("" : "+v"(v)::"memory");
                __builtin_amdgcn_sched_barrier(0);
                if (refill) fetch(k, arr, at, i + kRows, d);
                __builtin_amdgcn_sched_barrier(0);
                v += dpp_xchg<0x4E>(v);
                v += dpp_xchg<0x141>(v);
                v += dpp_xchg<0x140>(v);
                *to = v; // the same from all 16 lanes
                to += k.stride * PW;
            };
            // The first rows are there as x is (loads return in order).  Said here, so that the compiler's counts in the loop are those of the
            // steady state: all but the oldest row stay in flight.
            __builtin_amdgcn_s_waitcnt(0x0F70);
            __builtin_amdgcn_s_setprio(3);
            int i = 0;
            const auto tiles = [&](auto whole) __attribute__((always_inline)) {
                for (; i + kRows < k.steps; i += kRows) {
#pragma unroll
                    for (int u = 0; u < kRows; u++) row(i + u, pipe[u], true, whole);
                    // waves that are behind first: else the oldest take the memory's time and the last run by themselves
                    if (i == 0) __builtin_amdgcn_s_setprio(2);
                    else if (i == kRows) __builtin_amdgcn_s_setprio(1);
                    else __builtin_amdgcn_s_setprio(0);
                }
            };
            if (k.behind_early)
                tiles(std::false_type());
            else
                tiles(std::true_type());
            // The last rows, and in their places the first ones of the next phase, which are there when its input is.
#pragma unroll
            for (int u = 0; u < kRows; u++) {
                if (i + u < k.steps) row(i + u, pipe[u], false, std::false_type());
                if (u < next_steps) fetch(next, next_arr, next_at, u, pipe[u]);
            }
            __builtin_amdgcn_s_setprio(0);
        } else if (next_steps > 0) {
            ask(next, next_arr, next_at, pipe);
        }
        walk = next, arrays = next_arr;
        __syncthreads();

        const int fin = tid - (kThreads - (k.n + 63) / 64 * 64);
        if (fin >= 0 && fin < k.n) {
            __builtin_amdgcn_s_setprio(3);
            // the row's partial sums in a fixed order; all that is read from LDS is asked for at once
            const float4 *const p0 = reinterpret_cast<const float4 *>(part + fin * PW), *const p1 = p0 + (kPair ? k.n * nwk : 0);
            float4 f0[4], f1[4], r4[kWaves / 4];
#pragma unroll
            for (int u = 0; u < 4; u++) {
                f0[u] = p0[min(u, nwk - 1)];
                if (kPair) f1[u] = p1[min(u, nwk - 1)];
                if (kNorm) r4[u] = *reinterpret_cast<const float4 *>(&red[4 * u]);
            }
            const auto add4 = [](float &a, const float4 &v, bool there) __attribute__((always_inline)) {
                float t = a + v.x;
                t += v.y;
                t += v.z;
                t += v.w;
                a = there ? t : a;
            };
            float ss = 1.0f, sum0 = 0.f, sum1 = 0.f, t = 0.f;
#pragma unroll
            for (int u = 0; u < 4; u++) {
                add4(sum0, f0[u], u < nwk);
                if (kPair) add4(sum1, f1[u], u < nwk);
                if (kNorm) add4(t, r4[u], 4 * u < nwx); // nwx is a multiple of four
            }
            for (int i = 4; i < nwk; i += 4) { // only rows of hidden inputs are longer
#pragma unroll
                for (int u = 0; u < 4; u++) f0[u] = p0[min(i + u, nwk - 1)];
#pragma unroll
                for (int u = 0; u < 4; u++) add4(sum0, f0[u], i + u < nwk);
            }
            if (kNorm) { // rmsnorm scale, src/models.rs:55-60
                t /= (float)dim;
                t += A->eps;
                ss = 1.0f / sqrtf(t);
            }
            float v = sum0 * ss;
            if constexpr (kPair) { // silu(w1 x) * (w3 x), src/models.rs:92-98
                const float u2 = sum1 * ss;
                v = v * (1.0f / (1.0f + expf(-v)));
                v = v * u2;
            } else if constexpr (PH != TOK_QKV) {
                v = res + v;
                res = v;
            }
            hand_on(out + (k.r0 + fin), v);
            __builtin_amdgcn_s_setprio(0);
        }
        if (PH != TOK_QKV && !last) places_of<NEXT>(A, PH == TOK_W2 ? l + 1 : l, next.mat, tid, places);
    };

    const auto attention = [&](const int l) __attribute__((always_inline)) {
        asm volatile("" : "+v"(tid), "+v"(lane), "+s"(args));
        A = (ArgsPtr)(uintptr_t)args;
        const Floats E = (Floats)S.handed + (size_t)l * A->layer_floats;
        // Attention of one query head over all timesteps, a slice of its outputs per block: the kernel of the sliced form in
        // kernels_attn.hip with as many waves, so that the sums are the same.
        const auto attend = [&](auto nwv) __attribute__((always_inline)) {
#pragma clang fp contract(off)
            constexpr int NWV = decltype(nwv)::value, TSTEP = NWV * 4, PD = 4;
            typedef float vec_v __attribute__((ext_vector_type(VE)));
            struct Step {
                f32x4 k0, k1;
                vec_v v;
            };
            const int ds = lane & 15, tl = wave * 4 + (lane >> 4);
            const int pos = S.pos;
            const Floats kc = (Floats)S.kcache + (size_t)l * A->cache_layer, vc = (Floats)S.vcache + (size_t)l * A->cache_layer;
            const uint32_t row_bytes = (uint32_t)A->kv_dim * 4u;
            const uint32_t lane_off = (uint32_t)(kvh * HS + ds * 8) * 4u, v_off = (uint32_t)(kvh * HS + slice * VD + ds * VE) * 4u;
            const int t_last = max(pos - 1, 0);
            const auto fetch_kv = [&](int it, Step &d) __attribute__((always_inline)) {
                const uint32_t row = __umul24(min(it * TSTEP + tl, t_last), row_bytes), off = row + lane_off;
                const Global<const char> k = (Global<const char>)kc, v = (Global<const char>)vc;
                d.k0 = *(Global<const f32x4>)(k + off);
                d.k1 = *(Global<const f32x4>)(k + off + 16);
                d.v = *(Global<const vec_v>)(v + (row + v_off));
            };
            places_of<TOK_WO>(A, l, 0, tid, places);
            if (wave >= NWV) { // nothing to do but to meet the others
                if (walk.late) ask(walk, arrays, at_of(walk, TOK_WO), pipe);
                __syncthreads();
                __syncthreads();
                return;
            }
            Step kv[PD];
#pragma unroll
            for (int u = 0; u < PD; u++) fetch_kv(u, kv[u]);
            if (wave < 3) { // the new query, key and value: RoPE (src/models.rs:100-129) and the cache's new row
                const Floats from = E + A->at_qkv + (wave == 0 ? head * HS : wave == 1 ? A->dim + kvh * HS : A->dim + A->kv_dim + kvh * HS) + lane;
                uint32_t b0, b1;
                for (int looks = 0;;) {
                    b0 = load_agent1(from), b1 = load_agent1(from + HALF);
                    if (__all(b0 != kAbsent && b1 != kAbsent)) break;
                    if (++looks % kLooksPerCheck == 0 && gives_up(A, looks)) break;
                    __builtin_amdgcn_s_sleep(1);
                }
                float first = __builtin_bit_cast(float, b0), second = __builtin_bit_cast(float, b1);
                if (wave < 2) {
                    const float a = first, b = second;
                    first = a * rot_c - b * rot_s;
                    second = b * rot_c + first * rot_s;
                }
                float *to = wave == 0 ? qs : kvnew[wave - 1];
                to[lane] = first;
                to[lane + HALF] = second;
                if (wave > 0 && jh + slice == 0) {
                    const Floats row = (wave == 1 ? kc : vc) + (size_t)pos * A->kv_dim + kvh * HS;
                    row[lane] = first;
                    row[lane + HALF] = second;
                }
            }
            __syncthreads();
            {
                float q8[8];
#pragma unroll
                for (int e = 0; e < 8; e++) q8[e] = qs[ds * 8 + e];
                const float scale = 1.44269504088896340736f / sqrtf((float)HS);
                float m, lsum, acc[VE];
                {
                    float s = 0.f;
#pragma unroll
                    for (int e = 0; e < 8; e++) s = fmaf(q8[e], kvnew[0][ds * 8 + e], s);
                    s += dpp_xchg<0xB1>(s);
                    s += dpp_xchg<0x4E>(s);
                    s += dpp_xchg<0x141>(s);
                    s += dpp_xchg<0x140>(s);
                    const bool mine = tl == 0;
                    m = mine ? s * scale : kNoScore;
                    lsum = mine ? 1.f : 0.f;
#pragma unroll
                    for (int e = 0; e < VE; e++) acc[e] = mine ? kvnew[1][slice * VD + ds * VE + e] : 0.f;
                }
                const int n_it = (pos + TSTEP - 1) / TSTEP, n_tiles = (n_it + PD - 1) / PD;
                for (int tile = 0; tile < n_tiles; tile++) {
                    if (tile > 0) {
                        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                        for (int u = 0; u < PD; u++) fetch_kv(tile * PD + u, kv[u]);
                        __builtin_amdgcn_sched_barrier(0);
                    }
                    float sc[PD], mt = kNoScore;
                    bool valid[PD];
#pragma unroll
                    for (int u = 0; u < PD; u++) {
                        valid[u] = (tile * PD + u) * TSTEP + tl < pos;
                        const float kk[8] = {kv[u].k0.x, kv[u].k0.y, kv[u].k0.z, kv[u].k0.w, kv[u].k1.x, kv[u].k1.y, kv[u].k1.z, kv[u].k1.w};
                        float s = 0.f;
#pragma unroll
                        for (int e = 0; e < 8; e++) s = fmaf(q8[e], kk[e], s);
                        s += dpp_xchg<0xB1>(s);
                        s += dpp_xchg<0x4E>(s);
                        s += dpp_xchg<0x141>(s);
                        s += dpp_xchg<0x140>(s);
                        s = valid[u] ? s * scale : kNoScore;
                        sc[u] = s;
                        mt = fmaxf(mt, s);
                    }
                    if (__any(mt > m)) {
                        const float m_new = fmaxf(m, mt), c = __builtin_amdgcn_exp2f(m - m_new);
                        lsum *= c;
#pragma unroll
                        for (int e = 0; e < VE; e++) acc[e] *= c;
                        m = m_new;
                    }
#pragma unroll
                    for (int u = 0; u < PD; u++) {
                        const float p = valid[u] ? __builtin_amdgcn_exp2f(sc[u] - m) : 0.f;
                        lsum += p;
#pragma unroll
                        for (int e = 0; e < VE; e++) acc[e] = fmaf(p, valid[u] ? kv[u].v[e] : 0.f, acc[e]);
                    }
                }
                const auto merge = [&](auto both) __attribute__((always_inline)) {
                    const lanes::Both mb = both(m), lb = both(lsum);
                    const float M = fmaxf(mb.lo, mb.hi);
                    const float w1 = __builtin_amdgcn_exp2f(mb.lo - M), w2 = __builtin_amdgcn_exp2f(mb.hi - M);
                    lsum = lb.lo * w1 + lb.hi * w2;
#pragma unroll
                    for (int e = 0; e < VE; e++) {
                        const lanes::Both a = both(acc[e]);
                        acc[e] = a.lo * w1 + a.hi * w2;
                    }
                    m = M;
                };
                merge([](float v) { return lanes::both16(v); });
                merge([](float v) { return lanes::both32(v); });
                if (walk.late) ask(walk, arrays, at_of(walk, TOK_WO), pipe);
                if (lane < 16) {
#pragma unroll
                    for (int e = 0; e < VE; e++) comb[wave][ds * VE + e] = acc[e];
                    if (ds == 0) comb[wave][HS] = m, comb[wave][HS + 1] = lsum;
                }
            }
            __syncthreads();
            if (tid < VD) {
                float M = comb[0][HS], num = 0.f, den = 0.f;
#pragma unroll
                for (int w = 1; w < NWV; w++) M = fmaxf(M, comb[w][HS]);
#pragma unroll
                for (int w = 0; w < NWV; w++) {
                    const float e = __builtin_amdgcn_exp2f(comb[w][HS] - M);
                    num = fmaf(e, comb[w][tid], num);
                    den = fmaf(e, comb[w][HS + 1], den);
                }
                hand_on(E + A->at_att + head * HS + slice * VD + tid, num / den);
            }
        };
        if (attends) {
            if (S.pos >= 64)
                attend(std::integral_constant<int, 8>());
            else
                attend(std::integral_constant<int, 4>());
        } else {
            places_of<TOK_WO>(A, l, 0, tid, places);
            if (walk.late) ask(walk, arrays, at_of(walk, TOK_WO), pipe);
        }
        if (wave >= 8) { // the same layer's places of the next step are made empty
            const Global<u32x4> clear = (Global<u32x4>)((Floats)S.clear + (size_t)l * A->layer_floats);
            const int n16 = A->layer_floats / 4, per = (n16 + gridDim.x - 1) / gridDim.x, end = min(n16, (int)(blockIdx.x + 1) * per);
            for (int i = blockIdx.x * per + tid - 8 * 64; i < end; i += 8 * 64) clear[i] = u32x4{kAbsent, kAbsent, kAbsent, kAbsent};
        }
    };

    for (int l = 0; l < n_layers; l++) {
        phase(std::integral_constant<int, TOK_QKV>(), l);
        attention(l);
        phase(std::integral_constant<int, TOK_WO>(), l);
        phase(std::integral_constant<int, TOK_W13>(), l);
        phase(std::integral_constant<int, TOK_W2>(), l);
    }
}

// out[i] = where element i of a staged vector stands: at inv[i], in chunks of 32 padded to 36.
__global__ void slots_kernel(uint16_t *out, const int32_t *inv, size_t n) {
    const size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x;
    if (i < n) out[i] = (uint16_t)((inv[i] >> 5) * kChunkPad + (inv[i] & 31));
}

} // namespace

int token_slots_launch(uint16_t *out, const int32_t *inv, size_t n, hipStream_t st) {
    l2_launch(slots_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, out, inv, n);
    L2_HIP(hipGetLastError());
    return L2_OK;
}

int token_layers_launch(const TokArgs &a, int grid, size_t lds, bool eight, hipStream_t st) {
    const auto kernel = eight ? token_layers_kernel<8> : token_layers_kernel<4>;
    static LdsLimit limit[2];
    L2_TRY(limit[eight].ensure(reinterpret_cast<const void *>(kernel), lds));
    l2_launch(kernel, dim3(grid), dim3(kThreads), lds, st, a);
    L2_HIP(hipGetLastError());
    return L2_OK;
}
