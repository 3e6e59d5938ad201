// Internal declarations shared by the host code and the kernel launchers.
// Not part of the C ABI (that is include/llama2_hip.h).
#pragma once

#include <hip/hip_runtime.h>
#include <hip/hip_ext.h>
#include <stddef.h>
#include <stdint.h>

#include <atomic>
#include <mutex>
#include <string>
#include <type_traits>
#include <vector>

#include "../../include/llama2_hip.h"
#include "../../include/llama2_hip_bench.h"

// Compute units of the current device (256 on MI355X); asked once.
inline int cu_count() {
    static int n = 0;
    if (n == 0) {
        int dev = 0;
        hipDeviceProp_t prop;
        if (hipGetDevice(&dev) == hipSuccess && hipGetDeviceProperties(&prop, dev) == hipSuccess)
            n = prop.multiProcessorCount;
        if (n <= 0) n = 256;
    }
    return n;
}

// Four floats at an address that a caller of the C ABI chose, aligned as a float is and no more.  gfx950 moves 16 bytes
// at any multiple of four, so a load or store through this is the same one instruction as through float4.
typedef float float4_any __attribute__((ext_vector_type(4), aligned(4)));

// 16 bytes (aligned) past the L2: what a launch leaves dirty there is written back at its end, with nothing else to do, and the
// kernels of a batch write megabytes in their last microseconds.  Not for single columns: the store's own way is longer, and that
// is what the end of a decode kernel waits for (7B token 2 to 3 % longer, 70B 5 %).  A store that the compiler knows (sc1 is what it
// makes of "agent"), and not a statement of assembly: data of such a store may come out of a matrix instruction, whose result is
// not there for another 10 wait states, and must not be overwritten for two behind it, neither of which the hardware sees to.
#if defined(__HIPCC__)
template <class T>
__device__ __forceinline__ void store_through(T *p, const T &v) {
    static_assert(sizeof(T) == 16, "one instruction");
    typedef uint32_t four __attribute__((ext_vector_type(4)));
    __builtin_amdgcn_global_store_b128((__attribute__((address_space(1))) four *)p, __builtin_bit_cast(four, v), "agent");
}
#endif

// ---- error plumbing -------------------------------------------------------
int l2_fail(int code, const char *fmt, ...) __attribute__((format(printf, 2, 3)));

#define L2_HIP(call)                                                                     \
    do {                                                                                 \
        hipError_t e_ = (call);                                                          \
        if (e_ != hipSuccess)                                                            \
            return l2_fail(L2_ERR_HIP, "%s: %s (%s:%d)", #call, hipGetErrorString(e_),   \
                           __FILE__, __LINE__);                                          \
    } while (0)

#define L2_TRY(call)            \
    do {                        \
        int rc_ = (call);       \
        if (rc_ != L2_OK) return rc_; \
    } while (0)

// A launch, whose error the next hipGetLastError gives.  hipLaunchKernel by itself: `kernel<<<...>>>` and hipLaunchKernelGGL leave the
// launch's shape with the runtime and fetch it back in a stub (a queued launch of nine arguments 2.65 us of the host, this 2.41).
template <class... P, class... A>
inline void l2_launch(void (*kernel)(P...), const dim3 &grid, const dim3 &block, size_t lds, hipStream_t stream, const A &...args) {
    static_assert(sizeof...(P) == sizeof...(A), "one value per parameter");
    [&](P... p) {
        void *at[] = {const_cast<void *>(static_cast<const void *>(&p))...};
        (void)hipLaunchKernel(reinterpret_cast<const void *>(kernel), grid, block, at, lds, stream);
    }(args...);
}

// A kernel's dynamic-LDS limit (hipFuncAttributeMaxDynamicSharedMemorySize), raised when a launch needs more than it
// was last raised to.  One of these per kernel (a function-local static at the launch site).  The attribute belongs to
// the kernel as loaded on ONE device, so what was raised is kept per device; model handles on different host threads
// share the launch sites, so the slow path is behind a mutex and the fast path reads an atomic.
struct LdsLimit {
    static constexpr int kMaxDevices = 64;
    std::atomic<size_t> raised[kMaxDevices];
    std::mutex mu;
    explicit LdsLimit(size_t initial = 0) {
        for (auto &r : raised) r.store(initial, std::memory_order_relaxed);
    }
    int ensure(const void *kernel, size_t bytes) {
        int dev = 0;
        L2_HIP(hipGetDevice(&dev));
        if (dev < 0 || dev >= kMaxDevices) return l2_fail(L2_ERR_HIP, "device %d: more devices than the launch tables hold", dev);
        if (bytes <= raised[dev].load(std::memory_order_acquire)) return L2_OK;
        std::lock_guard<std::mutex> lock(mu);
        if (bytes <= raised[dev].load(std::memory_order_relaxed)) return L2_OK;
        L2_HIP(hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes));
        raised[dev].store(bytes, std::memory_order_release);
        return L2_OK;
    }
};

// Position at which the prefill ladder 64/32/16/8/4/2 (src/inference.rs:78-127) leaves off.
int l2_prefill_ladder_end(int n_prompt);
// What the ladder computes: the cache rows of the positions before that (enqueued; waited for with `wait`).
int l2_prefill_ladder(l2_model *m, l2_state *s, const int32_t *prompt, int n_prompt, bool wait);

// One forward step for the sampler: the weights above of the logits at `pos`, in host memory that belongs to the model
// and stands until its next call.  more: another step of the caller's call follows (else the call's work is waited for).
struct SampleWeights {
    float *w;
    const unsigned long long *redo;
};
int l2_forward_weights(l2_model *m, l2_state *s, int32_t token, int32_t pos, float temperature, bool more, SampleWeights *out);

// ---- device views ---------------------------------------------------------

// One QLinear resident in device memory, `.bin` layout (src/gptq.rs:68-84),
// plus the inverse of g_index so that a producer can write its output straight
// into the order this layer reads it in.
struct DevQLinear {
    const uint4 *qweight = nullptr;   // [out][in/32] chunks of 32 nibbles
    const int32_t *qzeros = nullptr;  // [out/8][groups]
    const float *scales = nullptr;    // [out][groups]
    const int32_t *g_index = nullptr; // [in]
    const int32_t *inv_index = nullptr; // [in], inv_index[g_index[j]] = j
    // scales and zero points once more, in tiles of 32 rows (group_tiles_launch): what the GEMMs read
    const float *scales_t = nullptr;  // [out/32][groups][32]
    const int32_t *zeros_t = nullptr; // [out/32][groups][4]
    int in = 0, out = 0, groups = 0, group_size = 0;
    const float *dense = nullptr;     // the model without quantisation: Linear<IN,OUT>.w [out][in]; the rest null
};

// ---- q4 matvec launch description ------------------------------------------

enum {
    Q4_EPI_STORE = 0,       // y[b][o] = v (+ scatter targets)
    Q4_EPI_RESIDUAL = 1,    // v += res[b][o]; y[b][o] = v (+ scatter targets)
    Q4_EPI_SCATTER_ONLY = 2 // scatter targets only
};

struct Q4Mat {
    const uint4 *qweight;
    const int32_t *qzeros;
    const float *scales;
    const float *x;  // input already in this layer's g_index order: [B][in] (in its natural order if gidx is set)
    const int32_t *gidx; // null, or the INVERSE of this layer's g_index: x is in its natural order and the kernel puts
                         // x[b][i] where input gidx[i] of the sorted rows is read (one matrix, no rmsnorm)
    const float *wn; // rmsnorm weights in the same order, or null: x is used as it is (a launch's matrices have theirs one behind the other)
    float *y;        // [B][out]
    int out;
    int row_blocks;  // blocks of grid.x that belong to this matrix
};

struct Q4Epi {
    int kind;
    const float *res;          // Q4_EPI_RESIDUAL: [B][out] (may alias y)
    int n_scatter;             // 0..3
    const int32_t *sc_idx[3];  // inverse act-order permutation of a following layer
    float *sc_out[3];          // [B][out]: sc_out[t][b][sc_idx[t][o]] = v
};

struct Q4Launch {
    Q4Mat m[3];
    Q4Epi e;
    int n_mats;
    int in;      // shared by all matrices of one launch
    int groups;
    int group_size;
    int batch;
    int pair;    // 1: m[0], m[1] are w1, w3; v = silu(m0 row) * (m1 row)
    float eps;   // rmsnorm epsilon, used when wn is set
    int rows_per_block; // filled by the streaming launcher
};
// The launch description travels by value as the kernel's one argument: it must stay far inside the 4 KB a
// dispatch packet's argument block holds, and be plain data that a byte copy reproduces.
static_assert(sizeof(Q4Launch) <= 1024, "Q4Launch is passed by value as a kernel argument");
static_assert(std::is_trivially_copyable<Q4Launch>::value && std::is_standard_layout<Q4Launch>::value,
              "Q4Launch is copied byte for byte into the dispatch's argument block");

// When armed (profiling runs only), the next q4 launch goes out through
// hipExtLaunchKernel with these events, which then carry the dispatch's own
// begin and end timestamps rather than those of marker packets around it.
struct Q4ProfHook {
    hipEvent_t start = nullptr, stop = nullptr;
    bool armed = false;
};
extern thread_local Q4ProfHook g_q4_prof;

// How the streaming launch takes its rows: `unit` rows stand behind one another, tiles of `tile` of them, `streams` at once; a row of
// a unit that is not in a whole tile stands behind the loop.  nwx: waves that the sum of squares of x is taken by; direct: the
// chunk sums of x are taken by the lanes, one four behind the other.  unit 0: another kernel's.
struct RowPlan {
    int unit, tile, streams, nwx;
    bool direct;
};

// When armed, the next q4 launch is not launched: the launcher writes the name of the kernel it would run
// (as a profiler prints it, template arguments included) into buf and disarms the hook.
struct Q4NameHook {
    char *buf = nullptr;
    int cap = 0;
    bool armed = false;
    int grid = 0, block = 0, rows_per_block = 0; // what the launch would have been
    size_t lds = 0;
    RowPlan rows{};
};
extern thread_local Q4NameHook g_q4_name;

// Launch the fp32 dequant matvec for up to 3 matrices that share `in`
// (wq|wk|wv), or a (w1, w3) pair.  Fills row_blocks itself.
int q4_matvec_launch(Q4Launch &L, hipStream_t stream);
// The two forms of the kernel behind q4_matvec_launch.
int q4_stream_launch(Q4Launch &L, hipStream_t stream);
bool q4_stream_supports(const Q4Launch &L);
// Whether q4_matvec_launch would apply the act-order permutation itself for this launch if m[0].gidx were set (one
// matrix, no rmsnorm, the default fp32 streaming form, rows of at most four waves); otherwise the caller gathers.
bool q4_gathers_in_kernel(const Q4Launch &L);

// ---- batches through the matrix cores (kernels_gemm.hip) -----------------------
// `planes` is 1 (activations rounded to fp16) or 3 (fp32 activations as three exact bf16 planes).  The activations of
// a GEMM are [B][planes][gemm_padded(in)] 16-bit values in the layer's g_index order, zero beyond `in`.  A launch with
// group_size 0 has fp32 weights (the model without quantisation, always 3 planes).
constexpr int kMaxGemmSlices = 16;
constexpr int kGemmMaxDim = 16384, kGemmMaxHidden = 38912; // a row of floats in LDS
__host__ __device__ inline int gemm_padded(int in) { return (in + 63) / 64 * 64; }

// Scales and zero points of a QLinear in tiles of 32 rows (the last one filled up with zeros): `tiles` holds group_tiles_floats
// floats, scales [out/32][groups][32] and behind them qzeros [out/32][groups][4].  A wave of a GEMM takes one group of 32 rows at
// a time, which is one or two cache lines here and 36 of 128 bytes in the checkpoint's order, whose rows the matvec
// kernels want.  Six layers of 7B, group 128, 64 tokens: fp32 1201 -> 1132 us, fp16 986 -> 938; 7B's prompt of 512 11.19 -> 10.78 ms,
// 70B's of 777 13.92 -> 13.53; 4096x11008, group 32, 61 columns 33.8 -> 30.0 us.  They take 4.5 bytes per row and
// group beside the checkpoint's own: 7, 14 or 28 % of the packed weights with groups of 128, 64 or 32.  The launches of gemm_launch have both in this form.
size_t group_tiles_floats(int out, int groups);
int group_tiles_launch(const float *scales, const int32_t *qzeros, int out, int groups, float *tiles, hipStream_t st);

struct XhList {
    const void *p[3]; // activations per matrix of the launch
};
// How a launch is cut.  The results depend on `slices` and `last` alone, and these on slice_batch, the number of columns the
// caller's chunk has: a pass over several chunks then gives what the chunks one by one would have given.  last (fp32 weights): the
// K steps of 64 inputs of the last slice, which is shorter than the others; 0, and all are equal.
struct GemmShape {
    int rows, tokens, row_blocks, slices, last;
};
GemmShape gemm_shape(const Q4Launch &L, int slice_batch, int planes);
GemmShape gemm_shape_f16(const Q4Launch &L, int slice_batch);
// The tiles that a launch of this shape takes, for tests: rows and tokens of a block, slices of K, blocks, how many of them take whole
// tiles, the width of the tiles of what whole rounds leave over, the tokens behind the whole tiles of a row block where they have a
// narrower one of their own (fp16; with fp32 weights GemmShape's `last`), whether a row block has whole tiles and others.
struct GemmTiles {
    int rows, tokens, slices, blocks, whole, width, last, both;
};
GemmTiles gemm_tiles(const Q4Launch &L, int slice_batch, int planes, bool beside);
GemmTiles gemm_tiles_f16(const GemmShape &s, int B, bool beside);
// Y = X W^T for L.batch columns; ss (per column, may be null) scales them.  Epilogues: store, residual add.  ws:
// workspace for the K slices' partial tiles.  ks_out given: the kernel leaves its slices as partial tiles [KS][B][out]
// in ws (also when there is one), no reduction is launched, and *ks_out says how many there are.  beside: a launch on another
// stream runs at the same time and takes the CUs that this one leaves.
int gemm_launch(Q4Launch &L, const XhList &xh, const float *ss, float *ws, size_t ws_floats, int planes, int slice_batch,
                hipStream_t st, int *ks_out = nullptr, bool beside = false);
int gemm_launch_f16(Q4Launch &L, const XhList &xh, const float *ss, float *ws, const GemmShape &s, int partials, bool beside,
                    hipStream_t st);
// What a first launch for this group size does besides enqueueing (for callers under graph capture).
int gemm_warm_up(int group_size);

struct GemmInput {
    void *out[3];
    const int32_t *g_index[3];
    const float *x; // [B][n], natural order
    int n;          // consumers (1..3)
};
int gemm_input_launch(const GemmInput &A, int n, int B, int planes, hipStream_t st);
// x[B][n] in pinned host memory, brought into the order of `inv` (the inverse of g_index) in device memory: as `planes`, or as
// fp32 (planes 0).
int host_input_launch(void *out, const float *x, const int32_t *inv, int n, int B, int planes, hipStream_t st);

struct ResNormPrep {
    const float *ws;   // partial tiles [KS][B][out] of one matrix, or null: the stream is already complete
    int KS, B, out;
    const float *res;  // [B][out] residual stream in
    float *x;          // [B][out] residual stream out (may be res)
    float *ss;         // [B] rms scale of the new residual stream
    float eps;
    int n;             // consumers (1..3)
    const int32_t *inv[3]; // inverse act-order permutation of each consumer (null: none)
    const float *wn;       // [out] norm weight of the consumers' rmsnorm, in the order of the residual stream
    void *out_h[3];        // the consumers' activations
};
int gemm_residual_norm_launch(const ResNormPrep &A, int planes, hipStream_t st);

struct SiluArgs {
    const float *ws; // partial tiles of w1 and w3 laid end to end: [KS][B][n] each
    int KS, B, n;
    const float *ss; // [B] rms scale of the layer's input
    const int32_t *inv; // inverse act-order permutation of w2 (null: none)
    void *out_h;
};
int gemm_silu_launch(const SiluArgs &A, int planes, hipStream_t st);

struct RopeKvArgs {
    const float *ws;   // partial tiles of q, k, v laid end to end: [KS][B][dim], [KS][B][kv_dim], [KS][B][kv_dim]
    int KS, B;
    const float *ss;   // [B] rms scale of the layer's input
    const int32_t *pos;
    const float *cos_t, *sin_t;
    float *q;          // [B][dim] out
    float *kcache, *vcache; // the layer's cache: rows [pos][kv_dim]
    int n_heads, n_kv_heads; // head size 128
};
int gemm_rope_kv_launch(const RopeKvArgs &A, hipStream_t st);

// Slot of element j of a vector in the order of a GEMM's bf16 planes: (0,2,4,6,1,3,5,7) inside every 8.
__host__ __device__ inline int b16_slot(int j) {
    const int e = j & 7;
    return (j & ~7) | ((e >> 1) + 4 * (e & 1));
}
// Slot of element j of a vector in the fp16 pair-interleaved order: (0,4,1,5,2,6,3,7) inside every 8.
__host__ __device__ inline int h16_slot(int j) {
    const int e = j & 7;
    return (j & ~7) | (e < 4 ? 2 * e : 2 * (e - 4) + 1);
}

// ---- the other per-token kernels -------------------------------------------

struct ScatterTargets {
    const int32_t *inv[3];
    float *out[3];
    int n;
};

// Where the tokens of a forward pass come from: an array in device memory; one token given here; or, for a step of the
// greedy loop, the running maximum of the step before, which is recorded as that step's result.
struct TokenSource {
    const int32_t *tokens = nullptr;
    const unsigned long long *prev = nullptr;
    int32_t *record = nullptr;
    int32_t token = 0;
};
// x[b] = emb[token b], also delivered through t; clears the running argmax.
int embed_launch(float *x, const float *emb, const TokenSource &src, int dim, int B, const ScatterTargets &t,
                 unsigned long long *amax_key, hipStream_t st);
// For sampling at `temperature` > 0 behind a classifier whose running maximum is amax: with d_i = logits[i] / temperature -
// max_j(logits[j] / temperature), w[i] = expf(d_i), correctly rounded; where that lies so close to the boundary between
// two floats that another faithful expf may round it the other way, w[i] = d_i and bit i of `redo` is set.
int sample_weights_launch(float *w, unsigned long long *redo, const float *logits, int n, float temperature,
                          const unsigned long long *amax, hipStream_t st);
// *id = the index of the running maximum.
int index_launch(const unsigned long long *amax, int32_t *id, hipStream_t st);
// dst = src, n floats; for pieces of pinned host memory up to a megabyte: quicker than the copy engine, behind which a kernel starts
// late (the operator on host arrays, 4096x1024, 4, 16, 64 columns by themselves 22.7 / 38.4 / 104 us, with it 27.8 / 42.2 / 120).
int copy_launch(float *dst, const float *src, size_t n, hipStream_t st);
// k and v: the first n floats (a multiple of 4) of each of `layers` stretches of `stride` floats become zero.
int clear_rows_launch(float *k, float *v, int layers, size_t stride, size_t n, hipStream_t st);
int gather_launch(float *out, const float *x, const int32_t *g_index, int n, int B, hipStream_t st);
int rope_kv_launch(float *q, const float *k, const float *v, const int32_t *pos, const float *cos_t,
                   const float *sin_t, float *kcache_l, float *vcache_l, int n_heads, int n_kv_heads,
                   int head_size, int B, hipStream_t st);
// Batched attention over an already written cache: out[b][scatter[i]] for query b at pos[b]; fp32 (planes 0), or the
// planes that a GEMM over `dim` inputs reads.
int attention_launch(void *out, int planes, const float *q, const float *kcache_l, const float *vcache_l,
                     const int32_t *pos, const int32_t *scatter, int n_heads, int n_kv_heads,
                     int head_size, int max_pos, int B, hipStream_t st);

// Up to so many timesteps eight query heads per kv head go together (attn_launch_qg).
constexpr int kFewTimesteps = 256;
// Decode attention (one query) with RoPE and the cache write folded in.
struct AttnDecode {
    const float *q;      // [dim]    raw query of this step
    const float *k_new;  // [kv_dim] raw key
    const float *v_new;  // [kv_dim] value
    float *kcache, *vcache;          // this layer: [max_seq][kv_dim]
    const float *cos_t, *sin_t;      // [max_seq][head_size/2]
    int pos;                         // position of this step (the host knows it; no device read in front of the loads)
    const int32_t *dpos;             // if set, the position is read from here instead (a captured step serves many positions)
    float *out;                      // [dim], written through scatter
    const int32_t *scatter;
    float *part;                     // split workspace: [n_heads][max_splits][130]
    int n_heads, n_kv_heads;
    int ts;                          // timesteps per split (multiple of 64)
    int n_splits;                    // grid.y; 1 = no combine pass
    int max_splits;
};
int attention_decode_launch(const AttnDecode &a, hipStream_t st);

// A call is at work on its handle's device for its time, for which it keeps one of these (host.cpp: DeviceCalls).  Calls that others make
// count once.
struct WorkMark {
    int depth = 0;
    bool claims = false; // steps of the call are in token kernels
};
struct AtWork {
    int device;
    WorkMark *mark;
    explicit AtWork(l2_model *m);
    AtWork(int device, WorkMark *mark);
    ~AtWork();
    AtWork(const AtWork &) = delete;
};

// ---- all layers of a decode step in one launch (kernels_token.hip) ---------------------------

constexpr int kTokenWaves = 16; // of a block
constexpr int kTokenRows = 3;   // rows of a wave in flight
enum { TOK_QKV = 0, TOK_WO = 1, TOK_W13 = 2, TOK_W2 = 3 };

// A projection: its arrays in the first layer, and how far apart those of two layers are (addresses: bytes).
struct TokMat {
    uint64_t qweight;
    uint32_t scales_at, zeros_at; // from qweight
    uint64_t stride;
};
// What is the same for a phase of every layer and wave.
struct TokPhase {
    int n4, nwk, gshift;  // inputs / 4, waves per row, log2(chunks of 32 inputs per group)
    int nwx, vec_floats;  // rmsnorm: waves that the sum of squares is taken by; floats of LDS per staged vector
    int direct;           // chunk sums of x one four behind the other
};
// What a wave does in a phase, the same in every layer: rows first, first + stride, ... (`steps` of them, none beyond `last`) of
// projection `mat`, the chunks 64 kslice to 64 kslice + 63 of each; bit i of `behind`: step i is a row that stands behind the loop of the launch
// that does this by itself, where its last bit is another.  The block's rows are n from r0 on, this wave's partial sums stand from row part_row on.
struct TokWalk {
    int mat, first, stride, last, steps, r0, n, part_row, kslice, C, groups;
    uint32_t behind;
    int32_t behind_early;  // whether one of them is among the looped steps, before the last kTokenRows or fewer
    int32_t late;          // wo: the wave attends, and asks for its first rows behind that
    int32_t pad[2];
};
static_assert(sizeof(TokWalk) == 64, "one scalar load");
struct TokModel { // in device memory
    TokPhase phase[4];
    TokMat m[7];               // q, k, v, wo, w1, w3, w2
    uint64_t walks;            // [4][blocks][kTokenWaves]
    uint64_t slots[7];         // of q, k, v, w1, w3, w2, wo: [layers][inputs], 16 bits: where an input stands in LDS (token_slots_launch)
    uint64_t rms_att, rms_ffn; // [layers][dim]
    uint64_t cos_t, sin_t;
    uint64_t failed, failed_host; // set where a wait has been given up, in device and in pinned memory
    uint64_t cache_layer;      // floats of one layer's K
    int n_layers, dim, kv_dim, n_heads, n_kv_heads;
    int layer_floats, at_qkv, at_att, at_xm, at_hg; // places in a layer's stretch; the layer's input stands at its start
    int part_at;               // floats of LDS in front of the partial sums
    int limit;                 // looks after which a wait is given up
    float eps;
};
struct TokArgs {
    const TokModel *model;
    float *handed;             // [layers][layer_floats]: what blocks hand on in this step, every float absent (all ones) before
    float *clear;              // the same for the next step
    const float *emb;          // the embedding table: the step starts from its token's row
    TokenSource src;
    unsigned long long *amax;  // null, or a running maximum to clear
    float *x;                  // [dim] the residual stream behind the last layer
    float *kcache, *vcache;    // [layers][max_seq][kv_dim]
    int pos;
};
int token_slots_launch(uint16_t *out, const int32_t *inv, size_t n, hipStream_t st);
int token_layers_launch(const TokArgs &a, int grid, size_t lds, bool eight, hipStream_t st);
// logits = wcls (rmsnorm(x, wn)); folds (value, index) into amax_key when set.
// wn == nullptr: plain Linear::matvec of x.
int dense_matvec_launch(float *y, const float *w, const float *x, const float *wn, float eps, int in, int out,
                        unsigned long long *amax_key, hipStream_t st);
// The general form: y[b] = epilogue(w (rmsnorm?)(x[b])) for `batch` columns (see dense_matvec_kernel).
struct DenseMat {
    const float *w; // [out][in]
    float *y;       // [batch][out]
    int out;
};
struct DenseArgs {
    DenseMat m[3];
    int n_mats;          // 1..3, one behind the other
    bool gated;          // of two with as many rows: m[1].y = silu(m[0] x) * (m[1] x), and m[0].y is scratch of the same size
    const float *x;      // [batch][in]
    const float *wn;     // [in] or null: rmsnorm weight applied to x, with eps
    float eps;
    int in, batch;
    unsigned long long *amax; // null, or the running (value, index) maximum (one matrix, batch == 1)
    const float *res;    // null, or [batch][out] added to the result (may alias y; one matrix)
    const float *gate;   // null, or [batch][out]: result = silu(gate) * result (one matrix)
    int n_pass, rows;    // set by the launcher: the matrices' rows
};
int dense_launch(const DenseArgs &a, hipStream_t st);
// pos = dpos[0]; next = pos < n_prompt ? prompt[pos] : index(amax_key);
// out_ids[pos - pos0] = next; tok[0] = next; dpos[0] = pos + 1.
// With loop_params (device: {n_prompt, pos0}) those two come from there, so that one captured launch serves any loop.
int next_token_launch(const unsigned long long *amax_key, const int32_t *prompt, int n_prompt,
                      int32_t *dpos, int32_t *out_ids, int pos0, int32_t *tok, hipStream_t st,
                      const int32_t *loop_params = nullptr);
// p[0] = a; if (q) q[0] = b.  Scalars travel as kernel arguments, never as
// asynchronous copies from the caller's stack.
int set_i32_launch(int32_t *p, int32_t a, int32_t *q, int32_t b, hipStream_t st);
int fill_pattern_launch(float *p, size_t n, uint64_t seed, hipStream_t st);
