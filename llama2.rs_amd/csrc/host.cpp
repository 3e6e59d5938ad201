// Host side of the C ABI: checkpoint loading and upload (LlamaModel::from_file,
// src/lib.rs:45-104), RunState (src/models.rs:29-42), the layer schedule of
// transformer<B> (src/models.rs:178-298) and the greedy loop of generate
// (src/inference.rs:16-193), driving the HIP kernels.  Nothing here computes on
// the CPU except the one-time RoPE angle table and the synthetic-image
// generator.
#include <map>
#include <fcntl.h>
#include <math.h>
#include <stdarg.h>
#include <stdio.h>
#include <string.h>
#include <sys/mman.h>
#include <sys/stat.h>
#include <unistd.h>

#include <algorithm>
#include <chrono>
#include <mutex>
#include <numeric>
#include <thread>

#include "host_window.h"
#include "l2_internal.h"

// ---------------------------------------------------------------------------
// errors

static thread_local char g_err[512] = "";
thread_local Q4ProfHook g_q4_prof;
thread_local Q4NameHook g_q4_name;

int l2_fail(int code, const char *fmt, ...) {
    va_list ap;
    va_start(ap, fmt);
    vsnprintf(g_err, sizeof(g_err), fmt, ap);
    va_end(ap);
    return code;
}

extern "C" const char *l2_last_error(void) { return g_err; }

// ---------------------------------------------------------------------------
// dims, presets, sizes

static int64_t div_up(int64_t x, int64_t y) { return x / y + (x % y == 0 ? 0 : 1); }

static size_t qlinear_bytes(int in, int out, int g) {
    if (g == 0) return (size_t)out * in * 4; // dense Linear<IN,OUT> (src/model.rs:11-15)
    const size_t groups = (size_t)div_up(in, g);
    return (size_t)out * (in / 8) * 4 + (size_t)(out / 8) * groups * 4 + (size_t)out * groups * 4 +
           (size_t)in * 4;
}

static int check_dims(const l2_dims *d) {
    if (!d) return l2_fail(L2_ERR_ARG, "dims is null");
    if (d->dim <= 0 || d->hidden_dim <= 0 || d->n_layers <= 0 || d->n_heads <= 0 ||
        d->n_kv_heads <= 0 || d->vocab_size <= 0 || d->seq_len <= 0)
        return l2_fail(L2_ERR_ARG, "dims: non-positive field");
    // 0 is the build without quantisation (GROUPSIZE of src/constants.rs:58-61): every projection dense
    if (d->group_size != 0 && d->group_size != 32 && d->group_size != 64 && d->group_size != 128)
        return l2_fail(L2_ERR_ARG, "dims: group_size %d (32, 64, 128, or 0 for the model without quantisation)",
                       d->group_size);
    if (d->dim % d->n_heads || d->n_heads % d->n_kv_heads)
        return l2_fail(L2_ERR_ARG, "dims: heads do not divide");
    if (d->dim / d->n_heads != 128)
        return l2_fail(L2_ERR_ARG, "dims: head size %d (the kernels are built for 128)", d->dim / d->n_heads);
    if ((d->group_size && (d->dim % d->group_size || d->hidden_dim % d->group_size)) || d->dim % 32 ||
        d->hidden_dim % 32)
        return l2_fail(L2_ERR_ARG, "dims: dim and hidden_dim must be multiples of 32 and of the group size");
    return L2_OK;
}

extern "C" int l2_preset(const char *model_size, int group_size, l2_dims *out) {
    if (!model_size || !out) return l2_fail(L2_ERR_ARG, "l2_preset: null argument");
    l2_dims d;
    // src/constants.rs:7-41
    if (!strcmp(model_size, "7B"))
        d = {4096, 11008, 32, 32, 32, 32000, 2048, group_size};
    else if (!strcmp(model_size, "13B"))
        d = {5120, 13824, 40, 40, 40, 32000, 2048, group_size};
    else if (!strcmp(model_size, "70B"))
        d = {8192, 28672, 80, 64, 8, 32000, 2048, group_size};
    else
        return l2_fail(L2_ERR_ARG, "l2_preset: model size '%s' (7B, 13B or 70B)", model_size);
    L2_TRY(check_dims(&d));
    *out = d;
    return L2_OK;
}

extern "C" size_t l2_weights_bytes(const l2_dims *d) {
    if (!d || d->n_heads <= 0) return 0;
    const int hs = d->dim / d->n_heads;
    const int kv_dim = d->n_kv_heads * hs;
    const size_t L = (size_t)d->n_layers;
    const int G = d->group_size;
    size_t n = 4;
    n += (size_t)d->vocab_size * d->dim * 4;
    n += L * d->dim * 4;
    n += L * (2 * qlinear_bytes(d->dim, d->dim, G) + 2 * qlinear_bytes(d->dim, kv_dim, G));
    n += L * d->dim * 4;
    n += L * (2 * qlinear_bytes(d->dim, d->hidden_dim, G) + qlinear_bytes(d->hidden_dim, d->dim, G));
    n += (size_t)d->dim * 4;
    n += (size_t)d->seq_len * (hs / 2) * 4 * 2;
    n += (size_t)d->vocab_size * d->dim * 4;
    return n;
}

// ---------------------------------------------------------------------------
// synthetic image

namespace {

struct Rng { // splitmix64
    uint64_t s;
    explicit Rng(uint64_t seed) : s(seed) {}
    uint64_t next() {
        uint64_t z = (s += 0x9E3779B97F4A7C15ull);
        z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
        z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
        return z ^ (z >> 31);
    }
    double uniform() { return (double)(next() >> 11) * (1.0 / 9007199254740992.0); }
    float normal(float sigma) {
        double u1 = uniform(), u2 = uniform();
        if (u1 < 1e-300) u1 = 1e-300;
        return (float)(sigma * sqrt(-2.0 * log(u1)) * cos(6.283185307179586 * u2));
    }
};

// One tensor-sized job of the generator; jobs are independent so that threads
// can take them in any order and still produce the same bytes.
struct SynthJob {
    char *dst;
    size_t n; // elements
    int kind; // 0 random words, 1 scales, 2 normal(0.02), 3 g_index, 4 freq cos, 5 freq sin
    uint64_t seed;
    int a, b; // g_index: in, group_size; freq: seq_len, half
};

void run_job(const SynthJob &j) {
    Rng r(j.seed);
    switch (j.kind) {
        case 0: {
            uint32_t *p = (uint32_t *)j.dst;
            size_t i = 0;
            for (; i + 1 < j.n; i += 2) {
                const uint64_t v = r.next();
                p[i] = (uint32_t)v;
                p[i + 1] = (uint32_t)(v >> 32);
            }
            if (i < j.n) p[i] = (uint32_t)r.next();
            break;
        }
        case 1: {
            float *p = (float *)j.dst;
            for (size_t i = 0; i < j.n; i++) p[i] = (float)(0.002 + 0.018 * r.uniform());
            break;
        }
        case 2: {
            float *p = (float *)j.dst;
            for (size_t i = 0; i < j.n; i++) p[i] = r.normal(0.02f);
            break;
        }
        case 3: {
            // g_idx = shuffled i / group_size; g_index = stable argsort(g_idx)
            // (export.py:52,65)
            const int in = j.a, G = j.b;
            std::vector<int32_t> gidx(in);
            for (int i = 0; i < in; i++) gidx[i] = i / G;
            for (int i = in - 1; i > 0; i--) {
                const int k = (int)(r.next() % (uint64_t)(i + 1));
                std::swap(gidx[i], gidx[k]);
            }
            const int groups = (in + G - 1) / G;
            std::vector<int32_t> start(groups + 1, 0);
            for (int i = 0; i < in; i++) start[gidx[i] + 1]++;
            for (int g = 0; g < groups; g++) start[g + 1] += start[g];
            int32_t *p = (int32_t *)j.dst;
            for (int i = 0; i < in; i++) p[start[gidx[i]]++] = i;
            break;
        }
        case 4:
        case 5: {
            float *p = (float *)j.dst;
            const int half = j.b;
            for (int t = 0; t < j.a; t++)
                for (int i = 0; i < half; i++) {
                    const float f = 1.0f / powf(10000.0f, (float)(2 * i) / (float)(2 * half));
                    const float ang = (float)t * f;
                    p[(size_t)t * half + i] = j.kind == 4 ? cosf(ang) : sinf(ang);
                }
            break;
        }
    }
}

// Walk the image in struct order (src/gptq.rs:34-84), calling f(kind, ptr, elems, in, out).
struct Walker {
    const l2_dims &d;
    char *p;
    std::vector<SynthJob> jobs;
    uint64_t seed;
    uint64_t counter = 0;
    void add(int kind, size_t n, int a = 0, int b = 0) {
        // big tensors are cut into slices so that the threads stay balanced
        const size_t slice = (kind == 3 || kind == 4 || kind == 5) ? n : ((size_t)1 << 22);
        for (size_t off = 0; off < n; off += slice) {
            const size_t m = std::min(slice, n - off);
            jobs.push_back({p + off * 4, m, kind, seed * 0x100000001B3ull + (++counter) * 0x9E3779B97F4A7C15ull, a, b});
        }
        p += n * 4;
    }
    void qlinears(int in, int out) {
        const int G = d.group_size;
        if (G == 0) { // dense projections, N(0, 0.02) like the embedding
            for (int l = 0; l < d.n_layers; l++) add(2, (size_t)out * in);
            return;
        }
        const size_t groups = (size_t)div_up(in, G);
        for (int l = 0; l < d.n_layers; l++) {
            add(0, (size_t)out * (in / 8));
            add(0, (size_t)(out / 8) * groups);
            add(1, (size_t)out * groups);
            add(3, (size_t)in, in, G);
        }
    }
};

} // namespace

extern "C" int l2_synth_image(const l2_dims *d, uint64_t seed, void *buf, size_t nbytes) {
    L2_TRY(check_dims(d));
    if (!buf) return l2_fail(L2_ERR_ARG, "l2_synth_image: null buffer");
    if (nbytes != l2_weights_bytes(d))
        return l2_fail(L2_ERR_ARG, "l2_synth_image: buffer is %zu bytes, image is %zu", nbytes, l2_weights_bytes(d));
    const int hs = d->dim / d->n_heads, kv_dim = d->n_kv_heads * hs;
    Walker w{*d, (char *)buf, {}, seed};
    const float eps = 1e-5f;
    memcpy(w.p, &eps, 4);
    w.p += 4;
    w.add(2, (size_t)d->vocab_size * d->dim);
    w.add(2, (size_t)d->n_layers * d->dim);
    w.qlinears(d->dim, d->dim);
    w.qlinears(d->dim, kv_dim);
    w.qlinears(d->dim, kv_dim);
    w.qlinears(d->dim, d->dim);
    w.add(2, (size_t)d->n_layers * d->dim);
    w.qlinears(d->dim, d->hidden_dim);
    w.qlinears(d->hidden_dim, d->dim);
    w.qlinears(d->dim, d->hidden_dim);
    w.add(2, (size_t)d->dim);
    w.add(4, (size_t)d->seq_len * (hs / 2), d->seq_len, hs / 2);
    w.add(5, (size_t)d->seq_len * (hs / 2), d->seq_len, hs / 2);
    w.add(2, (size_t)d->vocab_size * d->dim);
    if ((size_t)(w.p - (char *)buf) != nbytes) return l2_fail(L2_ERR_ARG, "l2_synth_image: internal size mismatch");
    unsigned nt = std::thread::hardware_concurrency();
    if (nt == 0) nt = 1;
    if (nt > 16) nt = 16;
    std::vector<std::thread> th;
    for (unsigned t = 0; t < nt; t++)
        th.emplace_back([&, t]() {
            for (size_t i = t; i < w.jobs.size(); i += nt) run_job(w.jobs[i]);
        });
    for (auto &t : th) t.join();
    return L2_OK;
}

// ---------------------------------------------------------------------------
// model

// Scratch of the stand-alone operator on a batch: the activations as planes and the K slices' partial tiles.
struct OperatorBufs {
    void *planes = nullptr;
    float *ws = nullptr;
    size_t planes_bytes = 0, ws_floats = 0;
};

struct l2_model {
    l2_dims d{};
    l2_config cfg{};
    int max_seq = 0;
    int head_size = 0, kv_dim = 0;
    float rms_eps = 0.f;
    int prefill_mode = L2_PREFILL_FP32;
    hipStream_t stream = nullptr;

    char *dimage = nullptr; // device copy of the weights image (shifted to 128-byte alignment)
    const float *tok_emb = nullptr, *rms_att = nullptr, *rms_ffn = nullptr, *rms_final = nullptr,
                *wcls = nullptr;
    std::vector<DevQLinear> q[7]; // indexed by L2_WQ..L2_W3, then layer
    int32_t *dinv = nullptr;      // all inverse permutations
    float *dtiles = nullptr;      // scales and zero points of all projections in tiles of 32 rows
    float *rope_cos = nullptr, *rope_sin = nullptr; // [max_seq][head_size/2]

    float *dwn = nullptr;         // norm weights in consumer order: [L][5][dim] (q, k, v, w1, w3)
    float *attn_part = nullptr;   // split-KV workspace [n_heads][kMaxSplits][130]

    // forward scratch, sized for cap_B batch columns.  xq/xk/xv and x1/x3 hold
    // the raw residual stream in the input order of the named projection.
    int cap_B = 0;
    float *x = nullptr, *xq = nullptr, *xk = nullptr, *xv = nullptr, *qv = nullptr, *kv = nullptr,
          *vv = nullptr, *attg = nullptr, *x1 = nullptr, *x3 = nullptr, *hg = nullptr, *hd = nullptr,
          *logits = nullptr;
    // Buffers of a batch through the matrix cores (kernels_gemm.hip).  l2_prefill_chunks runs consecutive passes of a
    // prompt side by side, one layer apart, on lanes: lane 0 is the model's stream, every lane has buffers of its own.
    struct ChunkBufs {
        float *x = nullptr, *q = nullptr, *ss = nullptr, *ws = nullptr;
        void *h[3] = {nullptr, nullptr, nullptr}; // activations of up to three consumers, as planes
        size_t cap_B = 0, ws_floats = 0, h_bytes = 0;
    };
    int32_t *dtok = nullptr, *dpos = nullptr;
    // Running maxima (value, index) of the classifier: step n of a loop folds into slot n % 2, so that the embedding
    // kernel of step n + 1 can read one slot while it clears the other.
    unsigned long long *amax = nullptr;
    // Pinned host memory that kernels read and write directly: logits, token ids, ids and positions on their way in.  The
    // calls on one model are serialised and each waits for its work, so it is free between calls.
    struct HostStage {
        char *base = nullptr;
        float *logits = nullptr;               // [vocab]: logits, or the sampler's weights
        unsigned long long *redo = nullptr;    // one bit per vocabulary entry
        int32_t *ids = nullptr, *in = nullptr; // [max_seq] out; [2 * max(max_seq, 4096)] in
        volatile int *gave_up = nullptr;       // TokArgs::failed_host
        bool reading = false; // a copy from `in` may still be on its way: no call has waited since
    } hs;
    static constexpr int kMaxLanes = 4; // the process has four hardware queues
    int n_lanes = 2;
    hipStream_t extra_stream[kMaxLanes - 1] = {nullptr, nullptr, nullptr};
    ChunkBufs lane[kMaxLanes];
    int32_t *pf_ids = nullptr; // ids, then positions, of a batch or prompt
    int cap_pf = 0;
    std::vector<hipEvent_t> pf_ev[kMaxLanes];
    hipEvent_t pf_join = nullptr, step_done = nullptr, ahead[2] = {}; // ahead: steps_ahead
    int32_t *dprompt = nullptr, *dout_ids = nullptr;
    int cap_prompt = 0, cap_out = 0;
    // The decode step as a HIP graph (one per bucket of positions, kept in the state).  Off by default: a
    // replayed step takes the host out of the loop (one call per token instead of some 160), but the step is
    // bound by its kernels, not by their launches, and reading the position from device memory costs the
    // attention kernel a little (7B: 625 tok/s replayed, 629 launched).
    int32_t *dloop = nullptr;     // device {n_prompt, pos0} of the running loop, read by the captured next_token launch
    uint64_t buf_epoch = 1;       // bumped whenever a buffer a captured step points at is reallocated
    bool capturing = false;       // forward_enqueue: take the position from m->dpos, size attention for max_pos
    bool use_graph = false;
    // scratch for the operator-level entry points
    float *op_x = nullptr, *op_xg = nullptr, *op_y = nullptr;
    size_t op_cap = 0;
    OperatorBufs op_batch;
    // All layers of a decode step in one launch (kernels_token.hip).
    struct TokenKernel {
        bool on = false;
        bool skip = false;      // this call's steps are done again with the layers' own launches
        int gave_up = 0;        // calls that had to be
        int in_a_row = 0;       // the last ones, with no call between whose token kernels came through
        uint64_t steps = 0;     // launched so far
        int missing = 0, fail_in = 0; // l2_model_token_trouble
        TokModel *model = nullptr; // in device memory
        uint16_t *slots = nullptr;
        TokWalk *walks = nullptr;
        float *handed = nullptr; // two sets, used in turn: a step's kernel empties the other
        size_t set_floats = 0;
        int set = 0, grid = 0;
        size_t lds = 0;
        bool eight = false;
        int *failed = nullptr;
    } tok;
    uint64_t asked = 0; // times that a loop of steps has asked the runtime about the stream (kAskLaunches)
    int device = 0;
    WorkMark work;
    // per-launch event timing, on only inside l2_decode_profile
    struct ProfRec { int cls; hipEvent_t e0, e1; };
    bool prof_on = false;
    std::vector<ProfRec> prof;
};


enum { K_EMBED = 0, K_Q4_QKV, K_ROPE_KV, K_ATTENTION, K_Q4_WO, K_Q4_W13, K_Q4_W2, K_CLASSIFIER, K_NEXT_TOKEN,
       K_NCLASS };
static const char *const kClassNames[K_NCLASS] = {"embed", "q4_qkv", "rope_kv", "attention", "q4_wo",
                                                  "q4_w13", "q4_w2", "classifier", "next_token"};
static constexpr int kMaxSplits = 64;

// Time one launch (profiling runs only).  The q4 launches of the streaming form hand their events to the
// dispatch itself; everything else is bracketed by event records on the stream.  Events of a launch that
// failed, or that nobody recorded, are destroyed here and leave no record.
template <class F>
static int timed_launch(l2_model *m, int cls, F &&launch) {
    l2_model::ProfRec r{cls, nullptr, nullptr};
    auto drop = [&]() {
        if (r.e0) (void)hipEventDestroy(r.e0);
        if (r.e1) (void)hipEventDestroy(r.e1);
    };
    hipError_t e = hipEventCreate(&r.e0);
    if (e == hipSuccess) e = hipEventCreate(&r.e1);
    if (e != hipSuccess) {
        drop();
        return l2_fail(L2_ERR_HIP, "hipEventCreate: %s", hipGetErrorString(e));
    }
    const bool q4 = m->d.group_size != 0 &&
                    (cls == K_Q4_QKV || cls == K_Q4_WO || cls == K_Q4_W13 || cls == K_Q4_W2);
    int rc = L2_OK;
    bool recorded = true;
    if (q4) {
        g_q4_prof.start = r.e0;
        g_q4_prof.stop = r.e1;
        g_q4_prof.armed = true;
        rc = launch();
        recorded = !g_q4_prof.armed; // a form of the kernel that does not take the events leaves them armed
        g_q4_prof.armed = false;
    } else {
        e = hipEventRecord(r.e0, m->stream);
        if (e == hipSuccess) rc = launch();
        if (e == hipSuccess && rc == L2_OK) e = hipEventRecord(r.e1, m->stream);
        if (e != hipSuccess && rc == L2_OK) rc = l2_fail(L2_ERR_HIP, "hipEventRecord: %s", hipGetErrorString(e));
    }
    if (rc != L2_OK || !recorded) {
        drop();
        return rc;
    }
    m->prof.push_back(r);
    return L2_OK;
}

#define LAUNCH(cls_, call)                                                   \
    do {                                                                     \
        if (m->prof_on)                                                      \
            L2_TRY(timed_launch(m, (cls_), [&]() -> int { return (call); })); \
        else                                                                 \
            L2_TRY(call);                                                    \
    } while (0)

// The calls that are at work on a device.  Blocks of a token kernel wait for one another, so all of them have to find room, which two such
// kernels at once might not; and while one runs it leaves room for kernels of up to 32 registers alone, others get their next launch at the end
// of a step (1 ms at 7B).  So a step takes it only while no other call of this process is at work on the device; else it goes out as launches of its own, which
// those of others come between.  Side by side, ms a call, before there were token kernels / with one model at a time in them, whatever others do /
// so: two models of eight layers of 7B, 100 tokens each, 59 and 59 / 34 and 383 / 60 and 60; a prompt of 256 tokens beside such a loop 1.8 / 9.8 / 1.8; 40
// tokens of a small fp32 model beside it 5.4 / 23 / 3.7.
// Calls that overlap do so again as a rule: steps stay with launches for kShared behind.
struct DeviceCalls {
    static constexpr int kMaxDevices = 64;
    static constexpr std::chrono::milliseconds kShared{10};
    typedef std::chrono::steady_clock Clock;
    std::mutex mu;
    struct {
        int calls = 0;
        Clock::time_point shared_until;
    } dev[kMaxDevices];
    std::atomic<int> claims{0}; // calls that have steps in token kernels

    void enter(int device) {
        std::lock_guard<std::mutex> lock(mu);
        if (dev[device].calls++ > 0) dev[device].shared_until = Clock::now() + kShared;
    }
    void leave(int device) {
        std::lock_guard<std::mutex> lock(mu);
        if (--dev[device].calls > 0) dev[device].shared_until = Clock::now() + kShared;
    }
    // Work that is enqueued and not waited for, on a stream of the caller's.
    void pass_by(int device) {
        if (claims.load(std::memory_order_relaxed) == 0 || device < 0 || device >= kMaxDevices) return;
        std::lock_guard<std::mutex> lock(mu);
        dev[device].shared_until = Clock::now() + kShared;
    }
    // Whether the one call that asks may take a token kernel.
    bool alone(int device) {
        if (device < 0 || device >= kMaxDevices) return false;
        std::lock_guard<std::mutex> lock(mu);
        return dev[device].calls == 1 && Clock::now() >= dev[device].shared_until;
    }
};
static DeviceCalls device_calls;

AtWork::AtWork(int device, WorkMark *mark) : device(device), mark(mark) {
    if (device >= 0 && device < DeviceCalls::kMaxDevices && mark->depth++ == 0) device_calls.enter(device);
}
// Token kernels of the call have been waited for.
AtWork::~AtWork() {
    if (device < 0 || device >= DeviceCalls::kMaxDevices || --mark->depth > 0) return;
    if (mark->claims) device_calls.claims--, mark->claims = false;
    device_calls.leave(device);
}
AtWork::AtWork(l2_model *m) : AtWork(m->device, &m->work) {}

struct StepGraph {
    hipGraph_t graph = nullptr;
    hipGraphExec_t exec = nullptr;
    uint64_t epoch = 0;
};

struct l2_state {
    l2_model *m = nullptr;
    float *kcache = nullptr, *vcache = nullptr; // [L][max_seq][kv_dim]
    size_t elems = 0;
    int rows = 0; // rows [0, rows) of every layer may have been written since the last reset; the others are zero
    std::map<int, StepGraph> steps; // captured decode step per upper bound of the position
};

static void step_graph_drop(StepGraph &g);

struct l2_qlinear {
    DevQLinear q;
    void *bufs[6] = {}; // the five arrays, the group tiles
    hipStream_t stream = nullptr;
    float *x = nullptr, *xg = nullptr, *y = nullptr;
    int cap_B = 0;
    int device = 0; // that was current when the handle was made
    int mode = L2_PREFILL_FP32;
    OperatorBufs batch;
};

extern "C" int l2_device_count(void) {
    int n = 0;
    if (hipGetDeviceCount(&n) != hipSuccess) {
        (void)hipGetLastError();
        return 0;
    }
    return n;
}

static int require_device() {
    int n = 0;
    hipError_t e = hipGetDeviceCount(&n);
    if (e != hipSuccess || n < 1) {
        (void)hipGetLastError();
        return l2_fail(L2_ERR_HIP, "no HIP device available (%s)", e == hipSuccess ? "count is 0" : hipGetErrorString(e));
    }
    return L2_OK;
}

template <typename T>
static int dalloc(T **p, size_t n) {
    void *v = nullptr;
    hipError_t e = hipMalloc(&v, n * sizeof(T) ? n * sizeof(T) : 16);
    if (e != hipSuccess) return l2_fail(L2_ERR_HIP, "hipMalloc(%zu bytes): %s", n * sizeof(T), hipGetErrorString(e));
    *p = (T *)v;
    return L2_OK;
}

static void dfree(void *p) {
    if (p) (void)hipFree(p);
}

// Pinned host memory for the operator's calls on host arrays, shared by all handles: a call takes a slot for its time, so
// calls of several threads run side by side.  At most kKept idle slots are kept, and none once the last handle is gone.
struct HostSlot {
    static constexpr size_t kBytes = (size_t)1 << 20; // each of x and y
    char *base = nullptr;
    float *x = nullptr, *y = nullptr;
};
static struct HostSlots {
    static constexpr size_t kKept = 4;
    std::mutex mu;
    HostSlot idle[kKept];
    size_t n_idle = 0;
    int users = 0;

    void add_user() {
        std::lock_guard<std::mutex> lock(mu);
        users++;
    }
    void drop_user() {
        std::lock_guard<std::mutex> lock(mu);
        if (--users > 0) return;
        while (n_idle > 0) (void)hipHostFree(idle[--n_idle].base);
    }
    int take(HostSlot *out) {
        {
            std::lock_guard<std::mutex> lock(mu);
            if (n_idle > 0) {
                *out = idle[--n_idle];
                return L2_OK;
            }
        }
        void *p = nullptr;
        L2_HIP(hipHostMalloc(&p, 2 * HostSlot::kBytes, hipHostMallocCoherent | hipHostMallocPortable));
        out->base = (char *)p;
        out->x = (float *)p, out->y = (float *)(out->base + HostSlot::kBytes);
        return L2_OK;
    }
    void give(const HostSlot &s) {
        std::lock_guard<std::mutex> lock(mu);
        if (n_idle < kKept && users > 0)
            idle[n_idle++] = s;
        else
            (void)hipHostFree(s.base);
    }
} host_slots;

// Device memory that the host writes itself, over the bus (fine-grained; where all of the device's memory is mapped for the host, and with it
// the register that says when the writes are there, see window_written): x of a
// call on host arrays goes there, and the kernel that needs it reads it on the device.  Before, x went to pinned memory, and a kernel of its
// own brought it over, or read it from there while it was cut into planes: 4096x4096, one column, 20.4 -> 19.3 us; 13824x5120, 16
// columns 76.4 -> 70.2.  The host writes 45 GB/s this way (with the flush 16 KB 1.6 us, 64 KB 2.7, 864 KB 20.7), the kernels read the bus at some 32.
// At most kKept pieces of a device, for as long as the process runs (memory that others may have cached is not given back to be used as
// something else); a call that finds none free takes the way through pinned memory.
struct HostWindow {
    float *x = nullptr;
    volatile uint32_t *flush = nullptr;
};
static struct HostWindows {
    static constexpr int kKept = 4, kMaxDevices = 64;
    std::mutex mu;
    float *idle[kMaxDevices][kKept] = {};
    volatile uint32_t *flush[kMaxDevices] = {};
    int n_idle[kMaxDevices] = {}, made[kMaxDevices] = {};
    uint64_t taken = 0;

    // One for a handle of `device`, if that is the calling thread's current device too: another device's memory is not for its kernels
    // (pinned memory is every device's).
    HostWindow take(int device) {
        int current = -1;
        if (device < 0 || device >= kMaxDevices || hipGetDevice(&current) != hipSuccess || current != device) return {};
        std::lock_guard<std::mutex> lock(mu);
        if (n_idle[device] > 0) return taken++, HostWindow{idle[device][--n_idle[device]], flush[device]};
        if (made[device] >= kKept) return {};
        int mapped = 0;
        uint64_t address = 0; // the attribute is one, and is stored as such
        void *p = nullptr;
        if (hipDeviceGetAttribute(&mapped, hipDeviceAttributeIsLargeBar, device) != hipSuccess || !mapped ||
            hipDeviceGetAttribute(reinterpret_cast<int *>(&address), hipDeviceAttributeHdpMemFlushCntl, device) != hipSuccess || !address ||
            hipExtMallocWithFlags(&p, HostSlot::kBytes, hipDeviceMallocFinegrained) != hipSuccess) {
            (void)hipGetLastError();
            made[device] = kKept; // not here
            return {};
        }
        flush[device] = reinterpret_cast<volatile uint32_t *>((uintptr_t)address);
        made[device]++, taken++;
        return {(float *)p, flush[device]};
    }
    void give(int device, const HostWindow &w) {
        if (!w.x) return;
        std::lock_guard<std::mutex> lock(mu);
        idle[device][n_idle[device]++] = w.x;
    }
} host_windows;

static void invert_perm(const int32_t *g, int n, int32_t *inv, bool *ok) {
    std::fill(inv, inv + n, -1);
    for (int j = 0; j < n; j++) {
        const int32_t v = g[j];
        if (v < 0 || v >= n || inv[v] != -1) {
            *ok = false;
            return;
        }
        inv[v] = j;
    }
}

static constexpr size_t kImageShift = 124; // image offset 4 (first tensor) lands on a 128-byte boundary

// q's group tiles in the memory at `tiles`; returns how much of it they take.
static size_t make_group_tiles(DevQLinear &q, float *tiles) {
    q.scales_t = tiles;
    q.zeros_t = reinterpret_cast<const int32_t *>(tiles + (size_t)((q.out + 31) / 32) * q.groups * 32);
    return group_tiles_floats(q.out, q.groups);
}

static int token_kernel_setup(l2_model *m);

static int model_build(const char *weights, size_t nbytes, const l2_dims *dims, int max_seq, l2_model **out) {
    L2_TRY(check_dims(dims));
    if (!weights || !out) return l2_fail(L2_ERR_ARG, "null argument");
    if (nbytes != l2_weights_bytes(dims)) // src/lib.rs:97
        return l2_fail(L2_ERR_FORMAT, "weights are %zu bytes, the struct for these dims is %zu", nbytes,
                       l2_weights_bytes(dims));
    if (max_seq <= 0) max_seq = dims->seq_len;
    {   // the attention kernels address one layer's cache with 32-bit byte offsets
        const size_t layer_bytes = (size_t)max_seq * dims->n_kv_heads * (dims->dim / dims->n_heads) * 4;
        if (layer_bytes >= ((size_t)1 << 32))
            return l2_fail(L2_ERR_RANGE, "max_seq %d: one layer of the cache would be %zu bytes (below 4 GiB)", max_seq,
                           layer_bytes);
    }
    L2_TRY(require_device());
    int device = 0;
    L2_HIP(hipGetDevice(&device));
    WorkMark mark;
    const AtWork at_work(device, &mark);

    l2_model *m = new l2_model();
    host_slots.add_user();
    m->use_graph = getenv("L2_STEP_GRAPH") != nullptr; // also l2_model_set_step_graph
    if (const char *v = getenv("L2_PREFILL_LANES")) { // chunks of a prompt in flight at once (l2_prefill_chunks)
        const int n = atoi(v);
        if (n >= 1 && n <= l2_model::kMaxLanes) m->n_lanes = n;
    }
    m->d = *dims;
    m->max_seq = max_seq;
    m->head_size = dims->dim / dims->n_heads;
    m->kv_dim = dims->n_kv_heads * m->head_size;
    m->cfg = {dims->dim, dims->hidden_dim, dims->n_layers, dims->n_heads, dims->n_kv_heads,
              dims->vocab_size, dims->seq_len, 0};
    auto bail = [&](int rc) {
        l2_model_close(m);
        return rc;
    };
#define M_HIP(call)                                                                              \
    do {                                                                                         \
        hipError_t e_ = (call);                                                                  \
        if (e_ != hipSuccess)                                                                    \
            return bail(l2_fail(L2_ERR_HIP, "%s: %s", #call, hipGetErrorString(e_)));            \
    } while (0)
#define M_TRY(call)                    \
    do {                               \
        int rc_ = (call);              \
        if (rc_ != L2_OK) return bail(rc_); \
    } while (0)

    M_HIP(hipStreamCreate(&m->stream));
    M_TRY(dalloc(&m->dimage, nbytes + 256));
    char *dbase = m->dimage + kImageShift;
    // one pass over the host image, in 64 MiB pieces so that a mapped file is paged in as it goes
    for (size_t off = 0; off < nbytes; off += (size_t)64 << 20) {
        const size_t n = std::min((size_t)64 << 20, nbytes - off);
        M_HIP(hipMemcpy(dbase + off, weights + off, n, hipMemcpyHostToDevice));
    }

    // views, in struct order (src/gptq.rs:34-66)
    const int L = dims->n_layers, G = dims->group_size, dim = dims->dim, hid = dims->hidden_dim;
    size_t off = 0;
    memcpy(&m->rms_eps, weights, 4);
    off += 4;
    auto f32 = [&](size_t n) {
        const float *p = (const float *)(dbase + off);
        off += n * 4;
        return p;
    };
    size_t inv_total = 0;
    struct Pending { int proj, layer; size_t host_off; int in; size_t inv_off; };
    std::vector<Pending> pend;
    auto qblock = [&](int proj, int in, int outn) {
        m->q[proj].resize(L);
        if (G == 0) { // src/model.rs:36-67: the same field order, every projection a dense matrix
            for (int l = 0; l < L; l++) {
                DevQLinear &q = m->q[proj][l];
                q.in = in;
                q.out = outn;
                q.dense = (const float *)(dbase + off);
                off += (size_t)outn * in * 4;
            }
            return;
        }
        const int groups = (int)div_up(in, G);
        for (int l = 0; l < L; l++) {
            DevQLinear &q = m->q[proj][l];
            q.in = in;
            q.out = outn;
            q.groups = groups;
            q.group_size = G;
            q.qweight = (const uint4 *)(dbase + off);
            off += (size_t)outn * (in / 8) * 4;
            q.qzeros = (const int32_t *)(dbase + off);
            off += (size_t)(outn / 8) * groups * 4;
            q.scales = (const float *)(dbase + off);
            off += (size_t)outn * groups * 4;
            q.g_index = (const int32_t *)(dbase + off);
            pend.push_back({proj, l, off, in, inv_total});
            inv_total += (size_t)in;
            off += (size_t)in * 4;
        }
    };
    m->tok_emb = f32((size_t)dims->vocab_size * dim);
    m->rms_att = f32((size_t)L * dim);
    qblock(L2_WQ, dim, dim);
    qblock(L2_WK, dim, m->kv_dim);
    qblock(L2_WV, dim, m->kv_dim);
    qblock(L2_WO, dim, dim);
    m->rms_ffn = f32((size_t)L * dim);
    qblock(L2_W1, dim, hid);
    qblock(L2_W2, hid, dim);
    qblock(L2_W3, dim, hid);
    m->rms_final = f32((size_t)dim);
    off += (size_t)dims->seq_len * (m->head_size / 2) * 4 * 2; // deprecated tables, never read (src/models.rs:193-197)
    m->wcls = f32((size_t)dims->vocab_size * dim);
    if (off != nbytes) return bail(l2_fail(L2_ERR_FORMAT, "internal: walked %zu of %zu bytes", off, nbytes));

    // inverse act-order permutations (also validates every g_index)
    if (G != 0) {
        std::vector<int32_t> inv(inv_total);
        bool ok = true;
        for (const Pending &p : pend) {
            invert_perm((const int32_t *)(weights + p.host_off), p.in, inv.data() + p.inv_off, &ok);
            if (!ok)
                return bail(l2_fail(L2_ERR_FORMAT, "g_index of projection %d, layer %d is not a permutation of 0..%d",
                                    p.proj, p.layer, p.in - 1));
        }
        M_TRY(dalloc(&m->dinv, inv_total));
        M_HIP(hipMemcpy(m->dinv, inv.data(), inv_total * 4, hipMemcpyHostToDevice));
        for (const Pending &p : pend) m->q[p.proj][p.layer].inv_index = m->dinv + p.inv_off;
        size_t tiles = 0;
        for (const Pending &p : pend) tiles += group_tiles_floats(m->q[p.proj][p.layer].out, m->q[p.proj][p.layer].groups);
        M_TRY(dalloc(&m->dtiles, tiles));
        tiles = 0;
        for (const Pending &p : pend) tiles += make_group_tiles(m->q[p.proj][p.layer], m->dtiles + tiles);
        for (const Pending &p : pend) {
            const DevQLinear &q = m->q[p.proj][p.layer];
            M_TRY(group_tiles_launch(q.scales, q.qzeros, q.out, q.groups, const_cast<float *>(q.scales_t), m->stream));
        }
    }

    M_TRY(dalloc(&m->attn_part, (size_t)dims->n_heads * kMaxSplits * 130));
    // Norm weights re-ordered for each consumer of a normalised vector, so that the
    // matvec prologue reads them linearly: wn_c[j] = w[g_index_c[j]].
    if (G != 0) {
        const size_t per_layer = (size_t)5 * dim;
        std::vector<float> wn((size_t)L * per_layer);
        const float *att_h = (const float *)(weights + ((const char *)m->rms_att - dbase));
        const float *ffn_h = (const float *)(weights + ((const char *)m->rms_ffn - dbase));
        const int projs[5] = {L2_WQ, L2_WK, L2_WV, L2_W1, L2_W3};
        for (int l = 0; l < L; l++)
            for (int c = 0; c < 5; c++) {
                const float *src = (c < 3 ? att_h : ffn_h) + (size_t)l * dim;
                const int32_t *g = (const int32_t *)(weights + ((const char *)m->q[projs[c]][l].g_index - dbase));
                float *dst = wn.data() + l * per_layer + (size_t)c * dim;
                for (int j = 0; j < dim; j++) dst[j] = src[g[j]];
            }
        M_TRY(dalloc(&m->dwn, wn.size()));
        M_HIP(hipMemcpy(m->dwn, wn.data(), wn.size() * 4, hipMemcpyHostToDevice));
    }

    // RoPE angles exactly as the reference evaluates them per element
    // (src/models.rs:107-110), computed once with the host's libm.
    {
        const int half = m->head_size / 2;
        std::vector<float> c((size_t)max_seq * half), s((size_t)max_seq * half);
        for (int i = 0; i < half; i++) {
            const float freq = 1.0f / powf(10000.0f, ((float)((2 * i) % m->head_size)) / (float)m->head_size);
            for (int p = 0; p < max_seq; p++) {
                const float val = (float)p * freq;
                c[(size_t)p * half + i] = cosf(val);
                s[(size_t)p * half + i] = sinf(val);
            }
        }
        M_TRY(dalloc(&m->rope_cos, c.size()));
        M_TRY(dalloc(&m->rope_sin, s.size()));
        M_HIP(hipMemcpy(m->rope_cos, c.data(), c.size() * 4, hipMemcpyHostToDevice));
        M_HIP(hipMemcpy(m->rope_sin, s.data(), s.size() * 4, hipMemcpyHostToDevice));
    }
    M_TRY(dalloc(&m->amax, 2));
    {
        const size_t redo = ((size_t)dims->vocab_size * 4 + 255) / 256 * 256,
                     ids = redo + ((size_t)dims->vocab_size / 64 + 32) / 32 * 256,
                     in = ids + ((size_t)max_seq * 4 + 255) / 256 * 256, flag = in + (size_t)std::max(max_seq, 4096) * 8, end = flag + 256;
        void *p = nullptr;
        M_HIP(hipHostMalloc(&p, end, hipHostMallocCoherent));
        m->hs.base = (char *)p;
        m->hs.logits = (float *)m->hs.base;
        m->hs.redo = (unsigned long long *)(m->hs.base + redo);
        m->hs.ids = (int32_t *)(m->hs.base + ids);
        m->hs.in = (int32_t *)(m->hs.base + in);
        m->hs.gave_up = (volatile int *)(m->hs.base + flag);
        *m->hs.gave_up = 0;
    }
    m->device = device;
    M_TRY(token_kernel_setup(m));
    M_HIP(hipDeviceSynchronize());
#undef M_HIP
#undef M_TRY
    *out = m;
    return L2_OK;
}

extern "C" int l2_model_from_image(const void *weights, size_t nbytes, const l2_dims *dims, int max_seq,
                                   l2_model **out) {
    return model_build((const char *)weights, nbytes, dims, max_seq, out);
}

extern "C" int l2_model_open(const char *path, const l2_dims *expect, int max_seq, l2_model **out) {
    if (!path || !expect || !out) return l2_fail(L2_ERR_ARG, "l2_model_open: null argument");
    L2_TRY(check_dims(expect));
    const int fd = open(path, O_RDONLY);
    if (fd < 0) return l2_fail(L2_ERR_IO, "open %s: %s", path, strerror(errno));
    struct stat st;
    if (fstat(fd, &st) != 0) {
        close(fd);
        return l2_fail(L2_ERR_IO, "stat %s: %s", path, strerror(errno));
    }
    int32_t h[7];
    if (st.st_size < 28 || pread(fd, h, 28, 0) != 28) {
        close(fd);
        return l2_fail(L2_ERR_FORMAT, "%s: shorter than the 28-byte header", path);
    }
    // Config::load + check_static (src/constants.rs:94-119)
    l2_config cfg = {h[0], h[1], h[2], h[3], h[4], h[5] < 0 ? -h[5] : h[5], h[6], h[5] > 0};
    if (cfg.dim != expect->dim || cfg.hidden_dim != expect->hidden_dim || cfg.n_layers != expect->n_layers ||
        cfg.n_heads != expect->n_heads || cfg.vocab_size != expect->vocab_size) {
        close(fd);
        return l2_fail(L2_ERR_FORMAT,
                       "%s: header (dim %d, hidden %d, layers %d, heads %d, vocab %d) does not match the "
                       "expected (%d, %d, %d, %d, %d)",
                       path, cfg.dim, cfg.hidden_dim, cfg.n_layers, cfg.n_heads, cfg.vocab_size, expect->dim,
                       expect->hidden_dim, expect->n_layers, expect->n_heads, expect->vocab_size);
    }
    const size_t want = l2_weights_bytes(expect);
    if ((size_t)st.st_size - 28 != want) { // src/lib.rs:97
        close(fd);
        return l2_fail(L2_ERR_FORMAT, "%s: %zu bytes after the header, the struct for these dims is %zu", path,
                       (size_t)st.st_size - 28, want);
    }
    // The reference maps from byte 28 (src/lib.rs:95-96); mmap offsets must be
    // page aligned, so map from 0 and step over the header.
    void *map = mmap(nullptr, (size_t)st.st_size, PROT_READ, MAP_PRIVATE, fd, 0);
    close(fd);
    if (map == MAP_FAILED) return l2_fail(L2_ERR_IO, "mmap %s: %s", path, strerror(errno));
    (void)madvise(map, (size_t)st.st_size, MADV_SEQUENTIAL);
    const int rc = model_build((const char *)map + 28, want, expect, max_seq, out);
    munmap(map, (size_t)st.st_size);
    if (rc == L2_OK) (*out)->cfg = cfg;
    return rc;
}

extern "C" void l2_model_close(l2_model *m) {
    if (!m) return;
    if (m->stream) (void)hipStreamSynchronize(m->stream);
    for (hipStream_t es : m->extra_stream)
        if (es) (void)hipStreamSynchronize(es);
    void *ptrs[] = {m->dimage, m->dinv, m->dtiles, m->rope_cos, m->rope_sin, m->dwn, m->attn_part, m->x, m->xq, m->xk,
                    m->xv, m->qv, m->kv, m->vv, m->attg, m->x1, m->x3, m->hg, m->hd, m->logits, m->dtok, m->dpos, m->dloop,
                    m->amax, m->dprompt, m->dout_ids, m->op_x, m->op_xg, m->op_y, m->op_batch.planes, m->op_batch.ws,
                    m->tok.handed, m->tok.failed, m->tok.model, m->tok.slots, m->tok.walks};
    for (void *p : ptrs) dfree(p);
    for (auto &a : m->lane) {
        void *bufs[] = {a.x, a.q, a.ss, a.ws, a.h[0], a.h[1], a.h[2]};
        for (void *p : bufs) dfree(p);
    }
    dfree(m->pf_ids);
    for (auto &v : m->pf_ev)
        for (hipEvent_t e : v) (void)hipEventDestroy(e);
    if (m->pf_join) (void)hipEventDestroy(m->pf_join);
    if (m->step_done) (void)hipEventDestroy(m->step_done);
    for (hipEvent_t e : m->ahead)
        if (e) (void)hipEventDestroy(e);
    if (m->hs.base) (void)hipHostFree(m->hs.base);
    for (hipStream_t es : m->extra_stream)
        if (es) (void)hipStreamDestroy(es);
    if (m->stream) (void)hipStreamDestroy(m->stream);
    delete m;
    host_slots.drop_user();
}

extern "C" int l2_model_config(const l2_model *m, l2_config *out) {
    if (!m || !out) return l2_fail(L2_ERR_ARG, "null argument");
    *out = m->cfg;
    return L2_OK;
}

extern "C" int l2_model_dims(const l2_model *m, l2_dims *out) {
    if (!m || !out) return l2_fail(L2_ERR_ARG, "null argument");
    *out = m->d;
    return L2_OK;
}

extern "C" int l2_model_max_seq(const l2_model *m) { return m ? m->max_seq : 0; }

extern "C" int l2_prefill_supported(const l2_model *m) { return m ? 1 : 0; }

extern "C" int l2_model_set_step_graph(l2_model *m, int on) {
    if (!m) return l2_fail(L2_ERR_ARG, "null model");
    m->use_graph = on != 0;
    return L2_OK;
}

static bool q4_gemm_supports(int in, int out, int g) {
    return in % 128 == 0 && out % 32 == 0 && in % g == 0 && (g < 64 || (in / g) % 2 == 0);
}

extern "C" int l2_model_set_prefill_mode(l2_model *m, int mode) {
    if (!m) return l2_fail(L2_ERR_ARG, "null model");
    if (mode != L2_PREFILL_FP32 && mode != L2_PREFILL_MFMA && mode != L2_PREFILL_COLUMNS) return l2_fail(L2_ERR_ARG, "prefill mode %d", mode);
    if (mode == L2_PREFILL_MFMA && m->d.group_size == 0)
        return l2_fail(L2_ERR_ARG, "the MFMA prefill path is the quantised model's");
    const int G = m->d.group_size;
    if (mode == L2_PREFILL_MFMA && m->head_size != 128)
        return l2_fail(L2_ERR_ARG, "the MFMA prefill path is built for heads of 128 (this model: %d)", m->head_size);
    if (mode == L2_PREFILL_MFMA && !(q4_gemm_supports(m->d.dim, m->d.dim, G) && q4_gemm_supports(m->d.hidden_dim, m->kv_dim, G) &&
                                     q4_gemm_supports(m->d.dim, m->d.hidden_dim, G)))
        return l2_fail(L2_ERR_ARG, "the MFMA prefill path needs dim and hidden_dim to be multiples of 128 (of 2 groups for "
                                   "group sizes 64 and 128) and output sizes to be multiples of 32");
    m->prefill_mode = mode;
    return L2_OK;
}

// When a batch of fp32 columns goes through the matrix cores (three exact bf16 planes): from four columns on, and from
// where the arithmetic outweighs the launches around the product.  Anything less is columns of the vector-ALU matvec,
// each the bits of a single one.  Measured on the operator, matvec against GEMM: 4096x4096 13.7 against 13.9 us at 4
// columns, 22 against 14 at 8; 4096x1024 13.5 against 12.9 at 16; 1024x1024 13.0 against 13.9 at 48.
static bool gemm_pays(int B, double weights) { return B >= 4 && B * weights >= 6e7; }
// The same for the layers of a model (nine launches each instead of seven).  Three layers of 1024 inputs, 2816 hidden units,
// with the logits behind them, matvec against GEMM: 8 columns 228 against 256 us, 12 257 against 258, 16 284 against 260,
// 32 394 against 270, 48 514 against 300.
static bool gemm_pays_layer(int B, double weights) { return B >= 8 && B * weights >= 1.4e8; }

static double layer_weights(const l2_model *m) {
    return (double)m->d.dim * (2.0 * m->d.dim + 2.0 * m->kv_dim + 3.0 * m->d.hidden_dim);
}

// What a batch of B columns of this model is computed with: 0 = the matvec kernels column by column, 1 or 3 = the GEMM
// with that many planes of activations.
static int batch_planes(const l2_model *m, int B) {
    if (B < 2 || m->prefill_mode == L2_PREFILL_COLUMNS || m->d.dim > kGemmMaxDim || m->d.hidden_dim > kGemmMaxHidden) return 0;
    if (m->prefill_mode == L2_PREFILL_MFMA) return 1; // quantised models only
    if (!gemm_pays_layer(B, layer_weights(m))) return 0;
    return 3;
}

// The same for the stand-alone operator.
static int operator_planes(const DevQLinear &q, int B, int mode) {
    return mode != L2_PREFILL_COLUMNS && gemm_pays(B, (double)q.in * q.out) ? 3 : 0;
}

// Nothing may be running on either of the model's streams when a buffer they use is freed.
static int drain_streams(l2_model *m) {
    L2_HIP(hipStreamSynchronize(m->stream));
    for (hipStream_t es : m->extra_stream)
        if (es) L2_HIP(hipStreamSynchronize(es));
    return L2_OK;
}

static int ensure_batch(l2_model *m, int B) {
    if (B <= m->cap_B) return L2_OK;
    L2_TRY(drain_streams(m));
    m->buf_epoch++;
    float **bufs[] = {&m->x, &m->xq, &m->xk, &m->xv, &m->qv, &m->kv, &m->vv, &m->attg, &m->x1, &m->x3, &m->hg};
    for (float **b : bufs) {
        dfree(*b);
        *b = nullptr;
    }
    dfree(m->dtok);
    dfree(m->dpos);
    m->dtok = m->dpos = nullptr;
    m->cap_B = 0;
    const size_t dim = m->d.dim, hid = m->d.hidden_dim, kvd = m->kv_dim;
    L2_TRY(dalloc(&m->x, B * dim));
    L2_TRY(dalloc(&m->xq, B * dim));
    L2_TRY(dalloc(&m->xk, B * dim));
    L2_TRY(dalloc(&m->xv, B * dim));
    L2_TRY(dalloc(&m->qv, B * dim));
    L2_TRY(dalloc(&m->kv, B * kvd));
    L2_TRY(dalloc(&m->vv, B * kvd));
    L2_TRY(dalloc(&m->attg, B * dim));
    L2_TRY(dalloc(&m->x1, B * dim));
    L2_TRY(dalloc(&m->x3, B * dim));
    L2_TRY(dalloc(&m->hg, B * hid));
    if (m->d.group_size == 0) { // the dense model keeps w1's output beside the gated product
        dfree(m->hd);
        m->hd = nullptr;
        L2_TRY(dalloc(&m->hd, B * hid));
    }
    L2_TRY(dalloc(&m->dtok, (size_t)B));
    L2_TRY(dalloc(&m->dpos, (size_t)B));
    if (!m->logits) L2_TRY(dalloc(&m->logits, (size_t)m->d.vocab_size));
    if (!m->dloop) L2_TRY(dalloc(&m->dloop, (size_t)2));
    m->cap_B = B;
    return L2_OK;
}

// Device room for the ids and the positions of n tokens.
static int ensure_ids(l2_model *m, int n) {
    if (n <= m->cap_pf) return L2_OK;
    L2_TRY(drain_streams(m));
    dfree(m->pf_ids);
    m->pf_ids = nullptr, m->cap_pf = 0;
    L2_TRY(dalloc(&m->pf_ids, (size_t)n * 2));
    m->cap_pf = n;
    return L2_OK;
}

// ---------------------------------------------------------------------------
// state

extern "C" int l2_state_new(l2_model *m, l2_state **out) {
    if (!m || !out) return l2_fail(L2_ERR_ARG, "null argument");
    l2_state *s = new l2_state();
    s->m = m;
    s->elems = (size_t)m->d.n_layers * m->max_seq * m->kv_dim;
    int rc = dalloc(&s->kcache, s->elems);
    if (rc == L2_OK) rc = dalloc(&s->vcache, s->elems);
    if (rc != L2_OK) {
        l2_state_free(s);
        return rc;
    }
    s->rows = m->max_seq; // nothing is known of fresh memory
    rc = l2_state_reset(s);
    if (rc != L2_OK) {
        l2_state_free(s);
        return rc;
    }
    *out = s;
    return L2_OK;
}

extern "C" void l2_state_free(l2_state *s) {
    if (!s) return;
    if (s->m && s->m->stream) (void)hipStreamSynchronize(s->m->stream);
    for (auto &kv : s->steps) step_graph_drop(kv.second);
    dfree(s->kcache);
    dfree(s->vcache);
    delete s;
}

// Zeroes what has been written since the last reset, on the model's stream.
static int state_clear(l2_state *s) {
    const l2_model *m = s->m;
    L2_TRY(clear_rows_launch(s->kcache, s->vcache, m->d.n_layers, (size_t)m->max_seq * m->kv_dim, (size_t)s->rows * m->kv_dim, m->stream));
    s->rows = 0;
    return L2_OK;
}

extern "C" int l2_state_reset(l2_state *s) {
    if (!s) return l2_fail(L2_ERR_ARG, "null state");
    const AtWork at_work(s->m);
    L2_TRY(state_clear(s));
    L2_HIP(hipStreamSynchronize(s->m->stream));
    return L2_OK;
}

extern "C" int l2_state_read_kv(l2_state *s, int layer, int pos0, int npos, float *k_host, float *v_host) {
    if (!s || !k_host || !v_host) return l2_fail(L2_ERR_ARG, "null argument");
    const AtWork at_work(s->m);
    const l2_model *m = s->m;
    if (layer < 0 || layer >= m->d.n_layers || pos0 < 0 || npos < 0 || pos0 + npos > m->max_seq)
        return l2_fail(L2_ERR_RANGE, "read_kv: layer %d, positions [%d,%d)", layer, pos0, pos0 + npos);
    const size_t off = ((size_t)layer * m->max_seq + pos0) * m->kv_dim;
    L2_HIP(hipStreamSynchronize(m->stream));
    L2_HIP(hipMemcpy(k_host, s->kcache + off, (size_t)npos * m->kv_dim * 4, hipMemcpyDeviceToHost));
    L2_HIP(hipMemcpy(v_host, s->vcache + off, (size_t)npos * m->kv_dim * 4, hipMemcpyDeviceToHost));
    return L2_OK;
}

extern "C" int l2_state_write_kv(l2_state *s, int layer, int pos0, int npos, const float *k_host,
                                 const float *v_host) {
    if (!s || !k_host || !v_host) return l2_fail(L2_ERR_ARG, "null argument");
    const AtWork at_work(s->m);
    const l2_model *m = s->m;
    if (layer < 0 || layer >= m->d.n_layers || pos0 < 0 || npos < 0 || pos0 + npos > m->max_seq)
        return l2_fail(L2_ERR_RANGE, "write_kv: layer %d, positions [%d,%d)", layer, pos0, pos0 + npos);
    const size_t off = ((size_t)layer * m->max_seq + pos0) * m->kv_dim;
    s->rows = std::max(s->rows, pos0 + npos);
    L2_HIP(hipStreamSynchronize(m->stream));
    L2_HIP(hipMemcpy(s->kcache + off, k_host, (size_t)npos * m->kv_dim * 4, hipMemcpyHostToDevice));
    L2_HIP(hipMemcpy(s->vcache + off, v_host, (size_t)npos * m->kv_dim * 4, hipMemcpyHostToDevice));
    return L2_OK;
}

extern "C" int l2_state_fill_synthetic(l2_state *s, int pos0, int npos, uint64_t seed) {
    if (!s) return l2_fail(L2_ERR_ARG, "null state");
    const AtWork at_work(s->m);
    const l2_model *m = s->m;
    if (pos0 < 0 || npos < 0 || pos0 + npos > m->max_seq)
        return l2_fail(L2_ERR_RANGE, "fill: positions [%d,%d)", pos0, pos0 + npos);
    s->rows = std::max(s->rows, pos0 + npos);
    for (int l = 0; l < m->d.n_layers; l++) {
        const size_t off = ((size_t)l * m->max_seq + pos0) * m->kv_dim;
        const size_t n = (size_t)npos * m->kv_dim;
        L2_TRY(fill_pattern_launch(s->kcache + off, n, seed * 2654435761ull + 2 * l, m->stream));
        L2_TRY(fill_pattern_launch(s->vcache + off, n, seed * 2654435761ull + 2 * l + 1, m->stream));
    }
    L2_HIP(hipStreamSynchronize(m->stream));
    return L2_OK;
}

// ---------------------------------------------------------------------------
// operators

static Q4Mat mat_of(const DevQLinear &q, const float *x, const float *wn, float *y) {
    Q4Mat M{};
    M.qweight = q.dense ? reinterpret_cast<const uint4 *>(q.dense) : q.qweight;
    M.qzeros = q.qzeros;
    M.scales = q.scales;
    M.x = x;
    M.wn = wn;
    M.y = y;
    M.out = q.out;
    return M;
}

// The same for gemm_launch.
static Q4Mat gemm_mat_of(const DevQLinear &q, float *y) {
    Q4Mat M = mat_of(q, nullptr, nullptr, y);
    M.qzeros = q.zeros_t, M.scales = q.scales_t;
    return M;
}

static Q4Launch launch_of(const DevQLinear &q, int B, float eps) {
    Q4Launch L{};
    L.n_mats = 1;
    L.in = q.in;
    L.groups = q.groups;
    L.group_size = q.group_size;
    L.batch = B;
    L.eps = eps;
    L.e.kind = Q4_EPI_STORE;
    return L;
}

// y = W xg for one matrix, plain store.
static int q4_one(const DevQLinear &q, const float *xg, float *y, int B, hipStream_t st) {
    Q4Launch L = launch_of(q, B, 0.f);
    L.m[0] = mat_of(q, xg, nullptr, y);
    return q4_matvec_launch(L, st);
}

// Whether the matvec kernel can apply g_index itself.
static bool takes_natural_order(const DevQLinear &q) {
    Q4Launch L = launch_of(q, 1, 0.f);
    L.m[0] = mat_of(q, nullptr, nullptr, nullptr);
    return q4_gathers_in_kernel(L);
}

// QLinear::matvec<B> on x in its natural order (src/gptq.rs:94-176, the act-order gather of :99-122 included):
// one launch where the kernel can apply g_index itself, else a gather into xg_scratch and the matvec.
static int q4_one_natural(const DevQLinear &q, const float *x, float *xg_scratch, float *y, int B, hipStream_t st) {
    Q4Launch L = launch_of(q, B, 0.f);
    L.m[0] = mat_of(q, x, nullptr, y);
    if (q4_gathers_in_kernel(L)) {
        L.m[0].gidx = q.inv_index;
        return q4_matvec_launch(L, st);
    }
    L2_TRY(gather_launch(xg_scratch, x, q.g_index, q.in, B, st));
    return q4_one(q, xg_scratch, y, B, st);
}

// Whether n floats at a and m floats at b share any.
static bool ranges_overlap(const float *a, size_t n, const float *b, size_t m) {
    const uintptr_t a0 = (uintptr_t)a, b0 = (uintptr_t)b;
    return a0 < b0 + m * sizeof(float) && b0 < a0 + n * sizeof(float);
}

static int check_qlinear_shape(int in, int out, int g) {
    if (g != 32 && g != 64 && g != 128) return l2_fail(L2_ERR_ARG, "group size %d (32, 64 or 128)", g);
    if (in <= 0 || out <= 0 || in % 32 || in % g || out % 8)
        return l2_fail(L2_ERR_ARG, "QLinear %dx%d: in must be a multiple of 32 and of the group size, out of 8", in, out);
    return L2_OK;
}

static int qlinear_scratch(l2_qlinear *q, int B);
struct FixedScratch {
    float *xg;
    void *planes;
    float *ws;
};
static int scratch_ptr(FixedScratch *out);

// Workspace of a stand-alone batch: a launch takes several K slices only while all its blocks (at most 256 x 64 outputs
// each) are resident at once, two per CU.
static constexpr size_t kOperatorWsFloats = (size_t)512 * 256 * 64;

// The operator on a batch through the matrix cores, activations already in planes: GEMM, sum of the K slices.
static int gemm_operator(const DevQLinear &q, int B, float *y, int planes, void *xh, float *ws, size_t ws_floats, hipStream_t st) {
    Q4Launch L = launch_of(q, B, 0.f);
    L.m[0] = gemm_mat_of(q, y);
    XhList X{{xh, nullptr, nullptr}};
    return gemm_launch(L, X, nullptr, ws, ws_floats, planes, B, st);
}

// ... with x in device memory: gather + split into planes first.
static int gemm_operator_natural(const DevQLinear &q, const float *x, int B, float *y, int planes, void *xh, float *ws,
                                 size_t ws_floats, hipStream_t st) {
    GemmInput in{};
    in.out[0] = xh, in.g_index[0] = q.g_index, in.x = x, in.n = 1;
    L2_TRY(gemm_input_launch(in, q.in, B, planes, st));
    return gemm_operator(q, B, y, planes, xh, ws, ws_floats, st);
}

static int operator_bufs(OperatorBufs &b, const DevQLinear &q, int B, int planes, hipStream_t st) {
    Q4Launch L = launch_of(q, B, 0.f);
    L.m[0] = mat_of(q, nullptr, nullptr, nullptr);
    const int ks = gemm_shape(L, B, planes).slices;
    const size_t pb = (size_t)B * planes * gemm_padded(q.in) * 2, wf = ks > 1 ? (size_t)ks * B * q.out : 0;
    if (pb <= b.planes_bytes && wf <= b.ws_floats) return L2_OK;
    L2_HIP(hipStreamSynchronize(st));
    if (pb > b.planes_bytes) {
        dfree(b.planes);
        b.planes = nullptr, b.planes_bytes = 0;
        char *p = nullptr;
        L2_TRY(dalloc(&p, pb));
        b.planes = p, b.planes_bytes = pb;
    }
    if (wf > b.ws_floats) {
        dfree(b.ws);
        b.ws = nullptr, b.ws_floats = 0;
        L2_TRY(dalloc(&b.ws, wf));
        b.ws_floats = wf;
    }
    return L2_OK;
}

// Everything a later launch of this layer's operator would otherwise do on first use, done once here and waited
// for: the code object is loaded on this device, the kernel's dynamic-LDS limit is raised, the fixed scratch
// arrays' addresses are resolved.  A call made under stream capture afterwards only enqueues kernels.
static int qlinear_warm_up(l2_qlinear *q) {
    L2_TRY(qlinear_scratch(q, 1));
    FixedScratch fixed{};
    L2_TRY(scratch_ptr(&fixed));
    L2_HIP(hipMemsetAsync(q->x, 0, (size_t)q->q.in * 4, q->stream));
    L2_TRY(q4_one_natural(q->q, q->x, q->xg, q->y, 1, q->stream));   // one column, either entry point
    L2_TRY(gather_launch(q->xg, q->x, q->q.g_index, q->q.in, 1, q->stream));
    L2_TRY(q4_one(q->q, q->xg, q->y, 1, q->stream));                 // several columns on device memory
    L2_TRY(gemm_warm_up(q->q.group_size));                           // and what either runs for a batch
    L2_HIP(hipStreamSynchronize(q->stream));
    return L2_OK;
}

extern "C" int l2_qlinear_create(const int32_t *qweight, const int32_t *qzeros, const float *scales,
                                 const int32_t *g_index, int in, int out, int group_size, l2_qlinear **ql) {
    if (!qweight || !qzeros || !scales || !g_index || !ql) return l2_fail(L2_ERR_ARG, "null argument");
    L2_TRY(check_qlinear_shape(in, out, group_size));
    L2_TRY(require_device());
    int device = 0;
    L2_HIP(hipGetDevice(&device));
    WorkMark mark;
    const AtWork at_work(device, &mark);
    const int groups = (int)div_up(in, group_size);
    std::vector<int32_t> inv(in);
    bool ok = true;
    invert_perm(g_index, in, inv.data(), &ok);
    if (!ok) return l2_fail(L2_ERR_FORMAT, "g_index is not a permutation of 0..%d", in - 1);
    l2_qlinear *q = new l2_qlinear();
    host_slots.add_user();
    const size_t sizes[5] = {(size_t)out * (in / 8) * 4, (size_t)(out / 8) * groups * 4, (size_t)out * groups * 4,
                             (size_t)in * 4, (size_t)in * 4};
    const void *src[5] = {qweight, qzeros, scales, g_index, inv.data()};
    for (int i = 0; i < 5; i++) {
        hipError_t e = hipMalloc(&q->bufs[i], sizes[i]);
        if (e == hipSuccess) e = hipMemcpy(q->bufs[i], src[i], sizes[i], hipMemcpyHostToDevice);
        if (e != hipSuccess) {
            l2_qlinear_free(q);
            return l2_fail(L2_ERR_HIP, "upload of QLinear array %d: %s", i, hipGetErrorString(e));
        }
    }
    if (hipStreamCreate(&q->stream) != hipSuccess) {
        l2_qlinear_free(q);
        return l2_fail(L2_ERR_HIP, "hipStreamCreate failed");
    }
    q->q.qweight = (const uint4 *)q->bufs[0];
    q->q.qzeros = (const int32_t *)q->bufs[1];
    q->q.scales = (const float *)q->bufs[2];
    q->q.g_index = (const int32_t *)q->bufs[3];
    q->q.inv_index = (const int32_t *)q->bufs[4];
    q->q.in = in;
    q->q.out = out;
    q->q.groups = groups;
    q->q.group_size = group_size;
    q->device = device;
    float *tiles = nullptr;
    int rc = dalloc(&tiles, group_tiles_floats(out, groups));
    q->bufs[5] = tiles;
    if (rc == L2_OK) {
        make_group_tiles(q->q, tiles);
        rc = group_tiles_launch(q->q.scales, q->q.qzeros, out, groups, tiles, q->stream);
    }
    if (rc == L2_OK) rc = qlinear_warm_up(q);
    if (rc != L2_OK) {
        l2_qlinear_free(q);
        return rc;
    }
    *ql = q;
    return L2_OK;
}

extern "C" void l2_qlinear_free(l2_qlinear *q) {
    if (!q) return;
    if (q->stream) (void)hipStreamSynchronize(q->stream);
    for (void *p : q->bufs) dfree(p);
    dfree(q->x);
    dfree(q->xg);
    dfree(q->y);
    dfree(q->batch.planes);
    dfree(q->batch.ws);
    if (q->stream) (void)hipStreamDestroy(q->stream);
    delete q;
    host_slots.drop_user();
}

extern "C" int l2_qlinear_set_mode(l2_qlinear *q, int mode) {
    if (!q) return l2_fail(L2_ERR_ARG, "null qlinear");
    if (mode != L2_PREFILL_FP32 && mode != L2_PREFILL_COLUMNS) return l2_fail(L2_ERR_ARG, "operator mode %d", mode);
    q->mode = mode;
    return L2_OK;
}

static int qlinear_scratch(l2_qlinear *q, int B) {
    if (B <= q->cap_B) return L2_OK;
    dfree(q->x);
    dfree(q->xg);
    dfree(q->y);
    q->x = q->xg = q->y = nullptr;
    q->cap_B = 0;
    L2_TRY(dalloc(&q->x, (size_t)B * q->q.in));
    L2_TRY(dalloc(&q->xg, (size_t)B * q->q.in));
    L2_TRY(dalloc(&q->y, (size_t)B * q->q.out));
    q->cap_B = B;
    return L2_OK;
}

// From here on x in pinned memory comes in two parts, whose second kernel costs 3 us: 384 KB (24 columns of 4096 inputs) 57.4 us whole, 58.5 by
// halves, 512 KB 67.8 and 67.9, 768 KB 91.6 and 89.6, 884 KB (16 of 13824) 82.8 and 78.5; with the matvec that permutes x itself
// 50.1 and 50.5, 62.3 and 61.2, 85.7 and 83.4 for 24, 32 and 48 of 4096.
static constexpr size_t kSplitBytes = 512 * 1024;
// From here on an x that a kernel permutes is written into device memory, in one part.  In device memory, in pinned memory: 13824 inputs, 1, 3,
// 4, 6, 8, 10, 16 columns (54 to 864 KB) 28.7 and 27.1 us, 49.6 and 47.9, 42.9 and 41.7, 47.8 and 47.2, 52.0 and 53.5, 56.7 and 60.0, 70.3 and 76.0; 4096, 10, 20,
// 24, 32, 61 columns (160 to 976 KB) 37.4 and 34.9, 48.1 and 48.7, 52.7 and 54.4, 62.5 and 65.8, 97.1 and 102; 8192, 10, 12, 16 columns (320 to 512 KB) 36.3 and
// 35.8, 38.2 and 38.4, 41.9 and 45.0.  By halves it takes longer (13824, 16 columns 72.5; 4096, 61 columns 100): the host's writes take the time, and
// each part waits for its own.
static constexpr size_t kWindowBytes = 384 * 1024;

static int operator_enqueue(const DevQLinear &q, const float *dx, float *dxg, float *y, const OperatorBufs &bufs, int planes,
                            int B, hipStream_t st) {
    if (!planes) return q4_one_natural(q, dx, dxg, y, B, st);
    return gemm_operator_natural(q, dx, B, y, planes, bufs.planes, bufs.ws, bufs.ws_floats, st);
}

// x (host, natural order) -> gather through g_index -> matvec -> y (host).  Where x and y fit a slot of pinned memory, the last kernel
// writes y there, and x is in device memory (HostWindows) or in the slot, from where kernels fetch it.  In the slot, one 4096x4096 matvec
// 28-40 -> 19.6 us (pageable copies either way before); against a DMA from the slot and a gather on the device, 16 columns of 13824x5120
// 89 -> 82 us, 61 of 4096x4096 116 -> 107, one of 28672x1024 32.8 -> 26.8.
static int matvec_host(const DevQLinear &q, int device, float *dx, float *dxg, float *dy, OperatorBufs &bufs, int planes,
                       const float *x_host, int B, float *y_host, hipStream_t st) {
    if (planes) L2_TRY(operator_bufs(bufs, q, B, planes, st));
    const size_t xb = (size_t)B * q.in * 4, yb = (size_t)B * q.out * 4;
    if (xb > HostSlot::kBytes || yb > HostSlot::kBytes) {
        L2_HIP(hipMemcpyAsync(dx, x_host, xb, hipMemcpyHostToDevice, st));
        L2_TRY(operator_enqueue(q, dx, dxg, dy, bufs, planes, B, st));
        L2_HIP(hipMemcpyAsync(y_host, dy, yb, hipMemcpyDeviceToHost, st));
        L2_HIP(hipStreamSynchronize(st));
        return L2_OK;
    }
    HostSlot slot;
    L2_TRY(host_slots.take(&slot));
    const bool natural = !planes && takes_natural_order(q); // the matvec kernel gathers
    const bool direct = natural || xb >= kWindowBytes;
    const HostWindow window = direct ? host_windows.take(device) : HostWindow{};
    float *const x = window.x ? window.x : slot.x;
    auto call = [&]() -> int {
        // a long x in pinned memory in two parts: the host brings the second one while the first crosses the bus
        for (int b0 = 0, b1 = B > 1 && xb >= kSplitBytes && !window.x ? B / 2 : B; b0 < B; b0 = b1, b1 = B) {
            const size_t at = (size_t)b0 * q.in, n = (size_t)(b1 - b0) * q.in;
            memcpy(x + at, x_host + at, n * sizeof(float));
            if (window.x) window_written(window.flush);
            if (!natural)
                L2_TRY(host_input_launch(planes ? (char *)bufs.planes + (size_t)b0 * planes * gemm_padded(q.in) * 2 : (char *)(dxg + at),
                                         x + at, q.inv_index, q.in, b1 - b0, planes, st));
            else if (!window.x)
                L2_TRY(copy_launch(dx + at, x + at, n, st));
        }
        if (natural) return q4_one_natural(q, window.x ? window.x : dx, dxg, slot.y, B, st);
        if (!planes) return q4_one(q, dxg, slot.y, B, st);
        return gemm_operator(q, B, slot.y, planes, bufs.planes, bufs.ws, bufs.ws_floats, st);
    };
    int rc = call();
    const hipError_t e = hipStreamSynchronize(st);
    if (rc == L2_OK && e != hipSuccess) rc = l2_fail(L2_ERR_HIP, "matvec: %s", hipGetErrorString(e));
    if (rc == L2_OK) memcpy(y_host, slot.y, yb);
    host_slots.give(slot);
    host_windows.give(device, window);
    return rc;
}

extern "C" int l2_qlinear_matvec(l2_qlinear *q, const float *x_host, int B, float *y_host) {
    if (!q || !x_host || !y_host) return l2_fail(L2_ERR_ARG, "null argument");
    if (B < 1 || B > 4096) return l2_fail(L2_ERR_RANGE, "batch %d (1..4096)", B);
    WorkMark mark; // of the call, not the handle: none is inside another here
    const AtWork at_work(q->device, &mark);
    L2_TRY(qlinear_scratch(q, B));
    return matvec_host(q->q, q->device, q->x, q->xg, q->y, q->batch, operator_planes(q->q, B, q->mode), x_host, B, y_host, q->stream);
}

// ---- the same operator for callers that cannot allocate ---------------------------------------------
// (code under HIP graph capture, tight serving loops, harnesses that forbid hipMalloc).  What
// l2_qlinear_matvec needs beyond its input and output lives in fixed device arrays instead of hipMalloc'ed ones.
// Every GPU the library runs on holds its own copy of the arrays, at its own addresses, until the process ends.
// A few columns: x gathered into the layer's act-order.
static constexpr size_t kScratchFloats = L2_MATVEC_DEVICE_MAX_ELEMS; // 4 MiB
static __device__ __align__(256) float scratch[kScratchFloats];
// A batch: its activations as three 16-bit planes (rows padded to 64, so at most twice the elements) and partial tiles.
static __device__ __align__(256) uint16_t scratch_planes[2 * 3 * kScratchFloats]; // 12 MiB
static __device__ __align__(256) float scratch_ws[kOperatorWsFloats];             // 32 MiB

// The arrays' addresses on the current device.  `scratch` by name is a host-side stand-in, not a device
// address; the address is asked for once per device, with that device current, and kept.
static int scratch_ptr(FixedScratch *out) {
    static constexpr int kMaxDevices = 64;
    static FixedScratch ptrs[kMaxDevices] = {};
    static std::mutex mu;
    int dev = 0;
    L2_HIP(hipGetDevice(&dev));
    if (dev < 0 || dev >= kMaxDevices) return l2_fail(L2_ERR_HIP, "device %d: more devices than the scratch table holds", dev);
    std::lock_guard<std::mutex> lock(mu);
    if (!ptrs[dev].ws) {
        void *p[3] = {nullptr, nullptr, nullptr};
        L2_HIP(hipGetSymbolAddress(&p[0], HIP_SYMBOL(scratch)));
        L2_HIP(hipGetSymbolAddress(&p[1], HIP_SYMBOL(scratch_planes)));
        L2_HIP(hipGetSymbolAddress(&p[2], HIP_SYMBOL(scratch_ws)));
        if (!p[0] || !p[1] || !p[2]) return l2_fail(L2_ERR_HIP, "hipGetSymbolAddress(scratch) on device %d", dev);
        ptrs[dev] = {(float *)p[0], p[1], (float *)p[2]};
    }
    *out = ptrs[dev];
    return L2_OK;
}

extern "C" int l2_qlinear_matvec_device(l2_qlinear *q, const float *x_dev, int B, float *y_dev, void *hip_stream) {
    if (!q || !x_dev || !y_dev) return l2_fail(L2_ERR_ARG, "null argument");
    if (B < 1 || B > 4096) return l2_fail(L2_ERR_RANGE, "batch %d (1..4096)", B);
    if ((size_t)B * (size_t)q->q.in > kScratchFloats)
        return l2_fail(L2_ERR_RANGE, "B * in = %zu floats exceed the fixed scratch of %zu (no allocation is made here: "
                                     "use a smaller batch, or l2_qlinear_matvec)",
                       (size_t)B * (size_t)q->q.in, kScratchFloats);
    device_calls.pass_by(q->device);
    FixedScratch fixed{};
    L2_TRY(scratch_ptr(&fixed));
    hipStream_t st = (hipStream_t)hip_stream;
    // Every element of the scratch that is read has been written before by the same call: nothing of the
    // previous call's contents is read, so nothing needs clearing.
    if (operator_planes(q->q, B, q->mode))
        return gemm_operator_natural(q->q, x_dev, B, y_dev, 3, fixed.planes, fixed.ws, kOperatorWsFloats, st);
    // One column: the kernel applies the permutation while it stages x (one launch where the host's launch rate is what
    // counts: 9.7 -> 6.6 us per call at 8192x1024).  Its blocks read all of x while others write y already, so where y lies
    // over x, x is gathered by a launch in front.  Several columns are gathered once, rather than by every block of every column.
    if (B == 1 && !ranges_overlap(x_dev, q->q.in, y_dev, q->q.out)) return q4_one_natural(q->q, x_dev, fixed.xg, y_dev, 1, st);
    L2_TRY(gather_launch(fixed.xg, x_dev, q->q.g_index, q->q.in, B, st));
    return q4_one(q->q, fixed.xg, y_dev, B, st);
}

static int op_scratch(l2_model *m, size_t elems) {
    if (elems <= m->op_cap) return L2_OK;
    L2_HIP(hipStreamSynchronize(m->stream));
    dfree(m->op_x);
    dfree(m->op_xg);
    dfree(m->op_y);
    m->op_x = m->op_xg = m->op_y = nullptr;
    m->op_cap = 0;
    L2_TRY(dalloc(&m->op_x, elems));
    L2_TRY(dalloc(&m->op_xg, elems));
    L2_TRY(dalloc(&m->op_y, elems));
    m->op_cap = elems;
    return L2_OK;
}

extern "C" int l2_model_qmatvec(l2_model *m, int layer, int proj, const float *x_host, int B, float *y_host) {
    if (!m || !x_host || !y_host) return l2_fail(L2_ERR_ARG, "null argument");
    if (proj < 0 || proj > 6 || layer < 0 || layer >= m->d.n_layers)
        return l2_fail(L2_ERR_RANGE, "projection %d, layer %d", proj, layer);
    if (B < 1 || B > 4096) return l2_fail(L2_ERR_RANGE, "batch %d (1..4096)", B);
    const AtWork at_work(m);
    const DevQLinear &q = m->q[proj][layer];
    L2_TRY(op_scratch(m, (size_t)B * std::max(std::max(q.in, q.out), m->d.vocab_size)));
    if (q.dense) { // Linear::matvec<B> (src/model.rs:22-31)
        hipStream_t st = m->stream;
        L2_HIP(hipMemcpyAsync(m->op_x, x_host, (size_t)B * q.in * 4, hipMemcpyHostToDevice, st));
        if (operator_planes(q, B, m->prefill_mode)) {
            L2_TRY(operator_bufs(m->op_batch, q, B, 3, st));
            GemmInput in{};
            in.out[0] = m->op_batch.planes, in.x = m->op_x, in.n = 1;
            L2_TRY(gemm_input_launch(in, q.in, B, 3, st));
            Q4Launch L = launch_of(q, B, 0.f);
            L.m[0] = gemm_mat_of(q, m->op_y);
            L2_TRY(gemm_launch(L, XhList{{m->op_batch.planes, nullptr, nullptr}}, nullptr, m->op_batch.ws, m->op_batch.ws_floats, 3, B, st));
        } else {
            DenseArgs a{};
            a.m[0] = {q.dense, m->op_y, q.out}, a.n_mats = 1, a.x = m->op_x, a.in = q.in, a.batch = B;
            L2_TRY(dense_launch(a, st));
        }
        L2_HIP(hipMemcpyAsync(y_host, m->op_y, (size_t)B * q.out * 4, hipMemcpyDeviceToHost, st));
        L2_HIP(hipStreamSynchronize(st));
        return L2_OK;
    }
    const int planes = m->prefill_mode == L2_PREFILL_MFMA ? batch_planes(m, B) : operator_planes(q, B, m->prefill_mode);
    return matvec_host(q, m->device, m->op_x, m->op_xg, m->op_y, m->op_batch, planes, x_host, B, y_host, m->stream);
}

extern "C" int l2_model_classifier(l2_model *m, const float *x_host, float *y_host) {
    if (!m || !x_host || !y_host) return l2_fail(L2_ERR_ARG, "null argument");
    const AtWork at_work(m);
    L2_TRY(op_scratch(m, (size_t)std::max(m->d.dim, m->d.vocab_size)));
    L2_HIP(hipMemcpyAsync(m->op_x, x_host, (size_t)m->d.dim * 4, hipMemcpyHostToDevice, m->stream));
    L2_TRY(dense_matvec_launch(m->op_y, m->wcls, m->op_x, nullptr, 0.f, m->d.dim, m->d.vocab_size, nullptr, m->stream));
    L2_HIP(hipMemcpyAsync(y_host, m->op_y, (size_t)m->d.vocab_size * 4, hipMemcpyDeviceToHost, m->stream));
    L2_HIP(hipStreamSynchronize(m->stream));
    return L2_OK;
}

// ---------------------------------------------------------------------------
// transformer<B>

// How the timesteps of a decode step are cut across blocks: not at all in a short context, where each query head's dimensions
// are spread over blocks instead, which every one scans all keys for; splits cost their merge, a launch of their own.  Whole
// against in splits, us per layer, the median of three processes (whose launches differ by a us, and with them the splits' cost),
// models of 32 layers (64 heads: 12, 64 of 8: 24) and the presets, so that a layer's rows come from memory as a user's do:
//   one or two query heads per kv head: up to 640.  7B at 500, 620, 800, 1010 40.8 / 41.9 / 43.9 / 45.9 and 41.1 / 41.8 / 42.3 / 42.7; 24
//   heads 33.5 / 35.0 / 37.4 / 39.4 and 34.9 / 35.2 / 36.4 / 36.5, 16 26.0 / 28.2 / 30.8 / 32.5 and 29.4 / 29.9 / 30.6 / 31.0, 8 21.0 /
//   21.9 / 22.9 / 26.2 and 21.8 / 22.8 / 20.6 / 21.7, 4 21.5 / 22.2 / 23.5 / 24.4 and 22.4 / 23.5 / 23.1 / 23.1; 32 of 16 37.5 / 39.2 / 41.7 /
//   43.2 and 39.3 / 39.9 / 40.6 / 40.4, 16 of 8 24.0 / 24.6 / 26.4 / 29.0 and 24.9 / 24.5 / 24.8 / 25.5
//   above 32 kv heads, whose heads are four slices each: 512.  13B at 440, 500, 620, 800 57.0 / 57.4 / 58.7 / 61.7 and 57.0 / 56.9 / 57.0 /
//   58.3; 64 heads 100.0 / 101.2 / 102.8 / 105.6 and 101.3 / 102.8 / 104.0 / 104.7
//   four or eight, whose splits take longer (the matrix cores): 768 from 32 heads on.  70B at 620, 740, 800, 1010 98.7 / 98.4 / 99.5 / 100.4
//   and 99.3 / 99.3 / 99.1 / 99.3; 32 of 8 39.9 / 40.8 / 41.6 / 44.6 and 41.8 / 42.2 / 42.2 / 42.4; 1024 where these have at most 4 kv heads,
//   32 of 4 35.4 / 36.1 / 36.6 / 37.5 and 38.5 / 38.7 / 38.8 / 39.0.  Fewer heads: 896.  8 of 2 at 740, 860, 1010 22.0 / 22.8 / 23.4 and
//   22.5 / 22.5 / 22.6, in 3 layers, as long as their launches, 25.5 / 26.8 / 26.8 and 26.4 / 27.2 / 27.0; 8 of 1 22.4 / 23.1 / 23.7 and 22.7 /
//   22.7 / 23.0, 16 of 4 25.3 / 26.0 / 26.5 and 25.9 / 25.8 / 25.9
// Beyond that one block per CU where
// the context allows it, at least 64 timesteps each.  (Two per CU, the earlier rule, left some CUs with two blocks
// and the launch as long as those: 70B behind 4096 positions 18.6 -> 16.5 us per layer, 13B behind 1000 positions
// 16.7 -> 15.3, 7B unchanged; half a block per CU is slower everywhere.)
// The limits are where launches cross, on both sides of which a step was launches.  Where a model has the token kernel they are also where its
// steps go from one launch to five per layer, and one launch is the shorter by more than the splits give, right up to them: us a step as launches and
// in one, at 30, 300, 500 positions and shortly before the limit, then behind it: 8 layers of 7B 276 / 298 / 309 / 312 and 248 / 266 / 277 / 280, then
// 317; 6 of 13B 291 / 308 / - / 315 and 260 / 274 / - / 280, then 322; 6 of 2048 inputs, 16 heads on 4, 129 / 142 / 149 / 160 and 104 / 115 / 122 / 132,
// then 159; 6 of 4096, 32 on 8, 200 / 215 / 222 / 229 and 180 / 192 / 200 / 206, then 230; 3 of 1024, 8 on 2, 55 / 61 / 63 / 68 and 50 / 54 / 56 / 60, then 70.
// So one launch would still be the shorter some way behind them; how far has not been measured.  The limits move for both routes together, or a
// call that is done again as launches would give other bits.
static void attn_split_policy(int n_t, int n_heads, int n_kv_heads, int *ts_out, int *n_splits_out) {
    int whole = n_heads <= 2 * n_kv_heads ? (n_kv_heads > 32 ? 512 : 640) : n_heads < 32 ? 896 : n_kv_heads <= 4 ? 1024 : 768;
    if (n_heads == 8 * n_kv_heads && n_t <= kFewTimesteps) whole = kFewTimesteps;
    if (n_t <= whole) {
        *ts_out = whole;
        *n_splits_out = 1;
        return;
    }
    int want = (cu_count() + n_kv_heads - 1) / n_kv_heads;
    if (want > kMaxSplits) want = kMaxSplits;
    int ts = ((n_t + want - 1) / want + 63) / 64 * 64;
    if (ts < 64) ts = 64;
    *ts_out = ts;
    *n_splits_out = (n_t + ts - 1) / ts;
}

// Enqueue one forward pass for the B tokens of `src` at the positions dpos (device; B == 1 takes its position from
// max_pos).  max_pos is the largest position among them (sizes the attention
// scratch).  With want_logits the classifier and the running argmax follow.
//
// When B == 1 all layers are one launch where the token kernel can be taken
// (`whole`, below), else five per layer: q|k|v with the attention rmsnorm in
// front; attention with RoPE and the cache write folded in; wo with the
// residual add behind; w1|w3 with the ffn rmsnorm in front and the SiLU gate
// behind; w2 with the residual add behind.  Every producer writes its result
// in the input order (g_index) of whoever reads it next.
struct ForwardIn {
    TokenSource src;
    const int32_t *dpos = nullptr;
    float *logits = nullptr;             // B == 1: where the logits go, or null
    unsigned long long *amax = nullptr;  // and their running maximum
    bool whole = false;                  // B == 1: the caller asks token_gave_up behind its wait, so the token kernel may be taken
};
static int forward_enqueue_dense(l2_model *m, l2_state *s, int B, int max_pos, const ForwardIn &in);

static int check_position(const l2_model *m, int max_pos) {
    // No kernel clamps a position: the RoPE table and the cache end at max_seq (the reference panics on its
    // fixed [SEQ_LEN] arrays, src/models.rs:29-33).
    if (max_pos < 0 || max_pos >= m->max_seq)
        return l2_fail(L2_ERR_RANGE, "position %d outside 0..%d", max_pos, m->max_seq - 1);
    return L2_OK;
}

// Waits for everything on the model's stream; with `amax`, the index of that running maximum is in *id (pinned host
// memory) then.  (A number that a last kernel stores in pinned memory is seen 4 to 13 us earlier than a synchronisation
// returns, but what the runtime does at one is then left for the next call: l2_state_reset behind a pass 13 -> 44 us.)
static int wait_host(l2_model *m, const unsigned long long *amax, int32_t *id) {
    if (amax) L2_TRY(index_launch(amax, id, m->stream));
    L2_HIP(hipStreamSynchronize(m->stream));
    m->hs.reading = false;
    return L2_OK;
}

// Before hs.in is written: a call that enqueued a prompt and left without waiting (an error behind it) may have its copy
// from there in flight.
static int claim_host_ids(l2_model *m) {
    if (m->hs.reading) L2_HIP(hipStreamSynchronize(m->stream));
    m->hs.reading = true;
    return L2_OK;
}

// How the token kernel deals a model's rows over its blocks and waves.
struct TokenPlan {
    TokPhase phase[4] = {};
    std::vector<TokWalk> walks; // [4][grid][kTokenWaves]
    int grid = 0, part_at = 0;  // part_at: TokModel::part_at
    size_t lds = 0;
    bool eight = false;         // slices of a head: eight or four, as many as keep one block per CU

    // The last blocks have no rows, and hand nothing on that others wait for: tests of waits that are given up.  They are launched like the
    // others, for the kernel reads the table by its grid.
    void leave_out(int blocks) {
        for (int p = 0; p < 4; p++)
            for (int b = grid - blocks; b < grid; b++)
                for (int w = 0; w < kTokenWaves; w++) {
                    TokWalk &k = walks[((size_t)p * grid + b) * kTokenWaves + w];
                    k.steps = k.n = k.part_row = k.late = k.behind_early = 0, k.behind = 0;
                }
    }
};
// The launches of a layer's four kinds of matvec, for their plans alone.
static void layer_launches(const l2_dims &d, Q4Launch (&L)[4]) {
    static const float some[4] = {0.f, 0.f, 0.f, 0.f}; // pointers count as null or not
    const auto one = [&](Q4Launch &l, std::initializer_list<int> outs, int in, bool norm) {
        DevQLinear q;
        q.in = in, q.group_size = d.group_size, q.groups = in / d.group_size;
        l = launch_of(q, 1, 0.f);
        l.n_mats = 0;
        for (int out : outs) {
            q.out = out;
            l.m[l.n_mats++] = mat_of(q, some, norm ? some : nullptr, nullptr);
        }
    };
    for (auto &l : L) l = Q4Launch{};
    const int kvd = d.dim / d.n_heads * d.n_kv_heads;
    one(L[TOK_QKV], {d.dim, kvd, kvd}, d.dim, true);
    one(L[TOK_WO], {d.dim}, d.dim, false);
    one(L[TOK_W13], {d.hidden_dim, d.hidden_dim}, d.dim, true);
    one(L[TOK_W2], {d.dim}, d.hidden_dim, false);
    L[TOK_W13].pair = 1, L[TOK_W13].e.kind = Q4_EPI_SCATTER_ONLY;
    L[TOK_WO].e.kind = L[TOK_W2].e.kind = Q4_EPI_RESIDUAL;
}

// *ok: whether decode steps of such a model can go through the token kernel.
static int token_plan(const l2_dims &d, TokenPlan &t, bool *ok) {
    *ok = false;
    if (d.group_size == 0) return L2_OK;
    const int grid = t.grid = cu_count(), qg = d.n_heads / d.n_kv_heads;
    t.eight = d.n_heads * 8 <= grid;
    if (d.dim / d.n_heads != 128 || d.n_heads * (t.eight ? 8 : 4) > grid || (qg != 1 && qg != 2 && qg != 4 && qg != 8)) return L2_OK;
    Q4Launch L[4];
    layer_launches(d, L);
    t.walks.assign((size_t)4 * grid * kTokenWaves, TokWalk{});
    int part = 0;
    for (int p = 0; p < 4; p++) {
        char name[160];
        g_q4_name = Q4NameHook{};
        g_q4_name.buf = name, g_q4_name.cap = (int)sizeof name, g_q4_name.armed = true;
        const int rc = q4_matvec_launch(L[p], nullptr);
        const bool answered = !g_q4_name.armed;
        g_q4_name.armed = false;
        L2_TRY(rc);
        const RowPlan plan = g_q4_name.rows;
        if (!answered || plan.unit < 1) return L2_OK; // not the streaming fp32 form, whose sums the kernel repeats
        const bool norm = p == TOK_QKV || p == TOK_W13;
        const int in = L[p].in, C = in / 32, nwk = (C + 63) / 64, halves = p == TOK_W13 ? 2 : 1, n_mats = p == TOK_QKV ? 3 : 1;
        TokPhase &f = t.phase[p];
        f.n4 = in / 4, f.nwk = nwk, f.nwx = plan.nwx, f.direct = plan.direct, f.vec_floats = nwk * 64 * 36;
        f.gshift = L[p].group_size == 128 ? 2 : L[p].group_size == 64 ? 1 : 0;
        if (nwk > kTokenWaves || (norm && (nwk > 4 || f.nwx > kTokenWaves || f.nwx % 4 || nwk * 512 > 2 * f.nwx * 64))) return L2_OK;
        // every block gets the same number of rows; q, k and v round up separately
        long rows = 0;
        for (int i = 0; i < n_mats; i++) {
            rows += L[p].m[i].out;
            const uint64_t bytes = (uint64_t)L[p].m[i].out * (in / 2 + L[p].groups * 4 + L[p].groups / 2 + 1);
            if (bytes >= (uint64_t)1 << 31) return L2_OK; // a matrix's arrays are one buffer with 32-bit offsets
        }
        int rpb = (int)((rows + grid - 1) / grid);
        const auto blocks = [&](int i) { return (L[p].m[i].out + rpb - 1) / rpb; };
        if (n_mats == 3)
            while (blocks(0) + blocks(1) + blocks(2) > grid) rpb++;
        // wo, where a wave has few rows: those that do not attend have theirs there when attention is, and take more (`early` of a stream)
        const bool uneven = p == TOK_WO && nwk <= 8 && rpb <= 8 / nwk * (kTokenRows + 1);
        const int streams = uneven ? 8 / nwk : kTokenWaves / nwk / halves;
        const int early = uneven ? std::min((rpb + streams - 1) / streams, (rpb + 2 * streams - 1) / (2 * streams) + 1) : 0;
        // A wave's rows that are rounded as behind a loop are a mask of 32 bits.  The more rows a wave has, the less there is to gain: two layers behind
        // 280 positions, as launches and in one, with 27, 28 and 32 pairs of w1|w3 a wave (5120 inputs, 13824 hidden; 8192, 14336; 8192, 16384) 110.8 and 101.7
        // us, 137.1 and 133.0, 146.4 and 143.8; with 56 (70B, with the classifier) 337.6 and 338.6.
        if (rpb > kTokenWaves * 64 || rpb > 32 * streams) return L2_OK;
        const auto whole = [&](int n) { return (n + plan.streams - 1) / plan.tile * plan.tile; };
        for (int b = 0; b < grid; b++) {
            int rb = b, mi = 0;
            while (mi + 1 < n_mats && rb >= blocks(mi)) rb -= blocks(mi), mi++;
            const int out = L[p].m[mi].out;
            for (int w = 0; w < kTokenWaves; w++) {
                TokWalk &k = t.walks[((size_t)p * grid + b) * kTokenWaves + w];
                const int v = uneven ? w & 7 : w;
                int s = v / nwk;
                k.kslice = v % nwk;
                k.r0 = rb * rpb, k.n = std::max(0, std::min(rpb, out - k.r0));
                k.mat = p == TOK_QKV ? mi : p == TOK_WO ? 3 : p == TOK_W13 ? 4 : 6;
                if (halves == 2 && s >= streams) s -= streams, k.mat = 5, k.part_row = k.n; // the second half of the waves has w3
                // the rows that the wave's half has: all, or for wo the first and the rest
                const int from = uneven && w < 8 ? std::min(early * streams, k.n) : 0, to = uneven && w >= 8 ? std::min(early * streams, k.n) : k.n;
                k.first = k.r0 + from + s, k.stride = streams, k.last = std::max(k.r0 + k.n - 1, 0);
                k.steps = s < streams && to - from > s ? (to - from - s + streams - 1) / streams : 0;
                k.late = uneven && w < 8 && k.steps > 0;
                k.C = C, k.groups = L[p].groups;
                for (int i = 0; i < k.steps; i++) {
                    const int o = k.first + i * k.stride, u = o / plan.unit, n = std::min(plan.unit, out - u * plan.unit);
                    if (o - u * plan.unit < whole(n)) continue;
                    k.behind |= 1u << i;
                    if (i < (k.steps - 1) / kTokenRows * kTokenRows) k.behind_early = 1;
                }
            }
        }
        part = std::max(part, rpb * nwk * 4 * halves);
    }
    t.part_at = std::max(3 * t.phase[TOK_QKV].vec_floats, t.phase[TOK_W2].vec_floats);
    t.lds = ((size_t)t.part_at + part) * 4;
    *ok = t.lds + 8 * 1024 <= 160 * 1024;
    return L2_OK;
}

// Every place that a step hands values on through becomes absent.
static int token_kernel_clear(l2_model *m) {
    L2_HIP(hipMemsetAsync(m->tok.handed, 0xFF, 2 * m->tok.set_floats * 4, m->stream));
    L2_HIP(hipMemsetAsync(m->tok.failed, 0, 4, m->stream));
    return L2_OK;
}

static constexpr int kTokenLooks = 1 << 17; // some 0.1 s

static int token_kernel_setup(l2_model *m) {
    const l2_dims &d = m->d;
    l2_model::TokenKernel &t = m->tok;
    if (getenv("L2_Q4_IMPL") || getenv("L2_ATTN_IMPL") || getenv("L2_TOKEN_LAUNCHES")) return L2_OK; // other forms of the launches
    TokenPlan plan;
    bool ok = false;
    L2_TRY(token_plan(d, plan, &ok));
    if (!ok) return L2_OK;
    t.grid = plan.grid, t.lds = plan.lds, t.eight = plan.eight;
    TokModel a{};
    memcpy(a.phase, plan.phase, sizeof a.phase);
    a.part_at = plan.part_at;
    a.n_layers = d.n_layers, a.dim = d.dim, a.kv_dim = m->kv_dim, a.n_heads = d.n_heads, a.n_kv_heads = d.n_kv_heads;
    a.at_qkv = d.dim, a.at_att = a.at_qkv + d.dim + 2 * m->kv_dim, a.at_xm = a.at_att + d.dim, a.at_hg = a.at_xm + d.dim;
    a.layer_floats = a.at_hg + d.hidden_dim;
    a.cache_layer = (size_t)m->max_seq * m->kv_dim;
    a.eps = m->rms_eps;
    a.limit = kTokenLooks;
    t.set_floats = (size_t)d.n_layers * a.layer_floats;
    size_t n_orders = 0;
    for (const auto &proj : m->q)
        for (const DevQLinear &q : proj) n_orders += (size_t)q.in;
    L2_TRY(dalloc(&t.slots, n_orders));
    L2_TRY(token_slots_launch(t.slots, m->dinv, n_orders, m->stream));
    L2_TRY(dalloc(&t.walks, plan.walks.size()));
    L2_HIP(hipMemcpy(t.walks, plan.walks.data(), plan.walks.size() * sizeof(TokWalk), hipMemcpyHostToDevice));
    L2_TRY(dalloc(&t.handed, 2 * t.set_floats));
    L2_TRY(dalloc(&t.failed, (size_t)1));
    L2_TRY(dalloc(&t.model, (size_t)1));
    const auto at = [](const void *p) { return (uint64_t)(uintptr_t)p; };
    a.walks = at(t.walks), a.rms_att = at(m->rms_att), a.rms_ffn = at(m->rms_ffn);
    a.cos_t = at(m->rope_cos), a.sin_t = at(m->rope_sin);
    a.failed = at(t.failed), a.failed_host = at(const_cast<int *>(m->hs.gave_up));
    // The layers' arrays stand at equal distances in the image and among the orders; the kernel counts on it.
    const int order[7] = {L2_WQ, L2_WK, L2_WV, L2_WO, L2_W1, L2_W3, L2_W2}, consumer[7] = {L2_WQ, L2_WK, L2_WV, L2_W1, L2_W3, L2_W2, L2_WO};
    for (int i = 0; i < 7; i++) {
        const DevQLinear &q = m->q[order[i]][0];
        TokMat &w = a.m[i];
        w.qweight = at(q.qweight);
        w.scales_at = (uint32_t)(at(q.scales) - w.qweight), w.zeros_at = (uint32_t)(at(q.qzeros) - w.qweight);
        w.stride = d.n_layers > 1 ? at(m->q[order[i]][1].qweight) - w.qweight : 0;
        const int32_t *const first = m->q[consumer[i]][0].inv_index;
        a.slots[i] = at(t.slots + (first - m->dinv));
        for (int l = 0; l < d.n_layers; l++) {
            const DevQLinear &k = m->q[order[i]][l], &o = m->q[consumer[i]][l];
            const uint64_t base = w.qweight + l * w.stride;
            if (at(k.qweight) != base || at(k.scales) != base + w.scales_at || at(k.qzeros) != base + w.zeros_at ||
                o.inv_index != first + (size_t)l * o.in)
                return l2_fail(L2_ERR_FORMAT, "internal: layers at unequal distances");
        }
    }
    L2_HIP(hipMemcpy(t.model, &a, sizeof a, hipMemcpyHostToDevice));
    L2_TRY(token_kernel_clear(m));
    t.on = true;
    return L2_OK;
}

// Behind a wait for the stream: whether a token kernel gave up waiting (its blocks did not all find room on the device, which other
// processes share), so that the call's steps have to be done again.
static int token_gave_up(l2_model *m, bool *again) {
    *again = false;
    if (!m->tok.on || !*m->hs.gave_up) return L2_OK;
    L2_TRY(token_kernel_clear(m));
    L2_HIP(hipStreamSynchronize(m->stream));
    *m->hs.gave_up = 0;
    m->tok.gave_up++;
    // The device is others' to stay, then; a call now and then that had to wait too long does not count for ever.
    if (++m->tok.in_a_row >= 3) m->tok.on = false;
    *again = true;
    return L2_OK;
}

// Steps of a call: steps() enqueues them and waits.  Where a token kernel gave up they are done once more, with the layers' own launches.
// Whatever comes back, no token kernel of the call is on the stream then and nothing of the call is left for the next one.
template <class F>
static int token_tries(l2_model *m, F &&steps) {
    bool again = false;
    int rc = L2_OK;
    do {
        const uint64_t before = m->tok.steps;
        rc = steps();
        if (rc != L2_OK) { // some of them may be on their way
            if (m->tok.steps != before && hipStreamSynchronize(m->stream) == hipSuccess) (void)token_gave_up(m, &again);
            break;
        }
        rc = token_gave_up(m, &again);
        if (rc == L2_OK && !again && m->tok.steps != before) m->tok.in_a_row = 0;
        m->tok.skip = again;
    } while (rc == L2_OK && again);
    m->tok.skip = false;
    return rc;
}

static int forward_enqueue(l2_model *m, l2_state *s, int B, int max_pos, const ForwardIn &in) {
    L2_TRY(check_position(m, max_pos));
    s->rows = std::max(s->rows, max_pos + 1);
    if (m->d.group_size == 0) return forward_enqueue_dense(m, s, B, max_pos, in);
    const l2_dims &d = m->d;
    const int dim = d.dim, hid = d.hidden_dim, kvd = m->kv_dim, L = d.n_layers;
    hipStream_t st = m->stream;
    bool whole = in.whole && m->tok.on && !m->tok.skip && !m->capturing && !m->prof_on;
    if (whole) { // contexts that one query head's blocks take whole, see attn_launch_qg
        int ts = 0, n_splits = 0;
        attn_split_policy(max_pos + 1, d.n_heads, d.n_kv_heads, &ts, &n_splits);
        whole = n_splits == 1 && (d.n_heads < 8 * d.n_kv_heads || ts > kFewTimesteps) && device_calls.alone(m->device);
    }
    if (whole) {
        if (!m->work.claims) device_calls.claims++, m->work.claims = true;
        l2_model::TokenKernel &t = m->tok;
        float *const handed = t.handed + (t.set ? t.set_floats : 0), *const clear = t.handed + (t.set ? 0 : t.set_floats);
        const TokArgs a{t.model, handed, clear, m->tok_emb, in.src, in.amax, m->x, s->kcache, s->vcache, max_pos};
        L2_TRY(token_layers_launch(a, t.grid, t.lds, t.eight, st));
        t.set ^= 1, t.steps++;
        if (t.fail_in > 0 && --t.fail_in == 0) return l2_fail(L2_ERR_HIP, "a step that a test has fail");
        if (in.logits)
            L2_TRY(dense_matvec_launch(in.logits, m->wcls, m->x, m->rms_final, m->rms_eps, dim, d.vocab_size, in.amax, st));
        return L2_OK;
    }
    {   // :189-191
        ScatterTargets t{};
        t.n = 3;
        t.inv[0] = m->q[L2_WQ][0].inv_index, t.inv[1] = m->q[L2_WK][0].inv_index, t.inv[2] = m->q[L2_WV][0].inv_index;
        t.out[0] = m->xq, t.out[1] = m->xk, t.out[2] = m->xv;
        LAUNCH(K_EMBED, embed_launch(m->x, m->tok_emb, in.src, dim, B, t, in.amax, st));
    }
    for (int l = 0; l < L; l++) {
        const DevQLinear &wq = m->q[L2_WQ][l], &wk = m->q[L2_WK][l], &wv = m->q[L2_WV][l],
                         &wo = m->q[L2_WO][l], &w1 = m->q[L2_W1][l], &w2 = m->q[L2_W2][l],
                         &w3 = m->q[L2_W3][l];
        const float *wn = m->dwn + (size_t)l * 5 * dim;
        {   // attention rmsnorm (:217-219) + q, k, v (:224-226)
            Q4Launch Q = launch_of(wq, B, m->rms_eps);
            Q.m[0] = mat_of(wq, m->xq, wn + 0 * (size_t)dim, m->qv);
            Q.m[1] = mat_of(wk, m->xk, wn + 1 * (size_t)dim, m->kv);
            Q.m[2] = mat_of(wv, m->xv, wn + 2 * (size_t)dim, m->vv);
            Q.n_mats = 3;
            LAUNCH(K_Q4_QKV, q4_matvec_launch(Q, st));
        }
        float *kc = s->kcache + (size_t)l * m->max_seq * kvd;
        float *vc = s->vcache + (size_t)l * m->max_seq * kvd;
        if (B == 1) { // rope (:228-230), cache write (:236-249), attention (:250-256)
            AttnDecode a{};
            a.q = m->qv, a.k_new = m->kv, a.v_new = m->vv;
            a.kcache = kc, a.vcache = vc;
            a.cos_t = m->rope_cos, a.sin_t = m->rope_sin;
            a.pos = max_pos;
            a.dpos = m->capturing ? m->dpos : nullptr; // a captured step serves every position up to max_pos
            a.out = m->attg, a.scatter = wo.inv_index;
            a.part = m->attn_part;
            a.n_heads = d.n_heads, a.n_kv_heads = d.n_kv_heads;
            a.max_splits = kMaxSplits;
            attn_split_policy(max_pos + 1, d.n_heads, d.n_kv_heads, &a.ts, &a.n_splits);
            if (a.n_splits > kMaxSplits)
                return l2_fail(L2_ERR_RANGE, "attention: position %d needs %d splits", max_pos, a.n_splits);
            LAUNCH(K_ATTENTION, attention_decode_launch(a, st));
        } else {
            LAUNCH(K_ROPE_KV, rope_kv_launch(m->qv, m->kv, m->vv, in.dpos, m->rope_cos, m->rope_sin, kc, vc, d.n_heads,
                                             d.n_kv_heads, m->head_size, B, st));
            LAUNCH(K_ATTENTION, attention_launch(m->attg, 0, m->qv, kc, vc, in.dpos, wo.inv_index, d.n_heads,
                                                 d.n_kv_heads, m->head_size, max_pos, B, st));
        }
        {   // wo (:260) + residual (:263-264); the new x also goes out in w1's and w3's order
            Q4Launch Q = launch_of(wo, B, 0.f);
            Q.m[0] = mat_of(wo, m->attg, nullptr, m->x);
            Q.e.kind = Q4_EPI_RESIDUAL;
            Q.e.res = m->x;
            Q.e.n_scatter = 2;
            Q.e.sc_idx[0] = w1.inv_index, Q.e.sc_out[0] = m->x1;
            Q.e.sc_idx[1] = w3.inv_index, Q.e.sc_out[1] = m->x3;
            LAUNCH(K_Q4_WO, q4_matvec_launch(Q, st));
        }
        {   // ffn rmsnorm (:266) + w1 | w3 (:271-272) + silu gate (:274-276), in w2's order
            Q4Launch Q = launch_of(w1, B, m->rms_eps);
            Q.m[0] = mat_of(w1, m->x1, wn + 3 * (size_t)dim, nullptr);
            Q.m[1] = mat_of(w3, m->x3, wn + 4 * (size_t)dim, nullptr);
            Q.n_mats = 2;
            Q.pair = 1;
            Q.e.kind = Q4_EPI_SCATTER_ONLY;
            Q.e.n_scatter = 1;
            Q.e.sc_idx[0] = w2.inv_index, Q.e.sc_out[0] = m->hg;
            LAUNCH(K_Q4_W13, q4_matvec_launch(Q, st));
        }
        {   // w2 (:279) + residual (:283-285); the new x goes out in the next layer's q, k, v order
            Q4Launch Q = launch_of(w2, B, 0.f);
            Q.m[0] = mat_of(w2, m->hg, nullptr, m->x);
            Q.e.kind = Q4_EPI_RESIDUAL;
            Q.e.res = m->x;
            if (l + 1 < L) {
                Q.e.n_scatter = 3;
                Q.e.sc_idx[0] = m->q[L2_WQ][l + 1].inv_index, Q.e.sc_out[0] = m->xq;
                Q.e.sc_idx[1] = m->q[L2_WK][l + 1].inv_index, Q.e.sc_out[1] = m->xk;
                Q.e.sc_idx[2] = m->q[L2_WV][l + 1].inv_index, Q.e.sc_out[2] = m->xv;
            }
            LAUNCH(K_Q4_W2, q4_matvec_launch(Q, st));
        }
        (void)hid;
    }
    if (in.logits) // final rmsnorm + classifier (:288-297, B == 1 only) + running argmax
        LAUNCH(K_CLASSIFIER, dense_matvec_launch(in.logits, m->wcls, m->x, m->rms_final, m->rms_eps, dim,
                                                 d.vocab_size, in.amax, st));
    return L2_OK;
}

// The same schedule for the model without quantisation (TransformerWeights, src/model.rs:36-67):
// every projection is a dense matvec with its rmsnorm in front (q, k, v, w1, w3), the SiLU gate behind
// (w3) or the residual add behind (wo, w2).  No act-order, so nothing is scattered.
static int forward_enqueue_dense(l2_model *m, l2_state *s, int B, int max_pos, const ForwardIn &in) {
    const l2_dims &d = m->d;
    const int dim = d.dim, hid = d.hidden_dim, kvd = m->kv_dim, L = d.n_layers;
    hipStream_t st = m->stream;
    {
        ScatterTargets t{};
        LAUNCH(K_EMBED, embed_launch(m->x, m->tok_emb, in.src, dim, B, t, in.amax, st));
    }
    auto dense = [&](const DevQLinear &w, const float *x, float *y, const float *res) {
        DenseArgs a{};
        a.m[0] = {w.dense, y, w.out}, a.n_mats = 1, a.x = x, a.in = w.in, a.batch = B, a.res = res;
        return dense_launch(a, st);
    };
    auto normed = [&](std::initializer_list<DenseMat> mats, const float *wn, bool gated) {
        DenseArgs a{};
        for (const DenseMat &w : mats) a.m[a.n_mats++] = w;
        a.x = m->x, a.wn = wn, a.eps = m->rms_eps, a.in = dim, a.batch = B, a.gated = gated;
        return dense_launch(a, st);
    };
    for (int l = 0; l < L; l++) {
        const float *att_n = m->rms_att + (size_t)l * dim, *ffn_n = m->rms_ffn + (size_t)l * dim;
        const float *const wq = m->q[L2_WQ][l].dense, *const wk = m->q[L2_WK][l].dense, *const wv = m->q[L2_WV][l].dense;
        LAUNCH(K_Q4_QKV, normed({{wq, m->qv, dim}, {wk, m->kv, kvd}, {wv, m->vv, kvd}}, att_n, false)); // :217-226
        float *kc = s->kcache + (size_t)l * m->max_seq * kvd;
        float *vc = s->vcache + (size_t)l * m->max_seq * kvd;
        if (B == 1) {
            AttnDecode a{};
            a.q = m->qv, a.k_new = m->kv, a.v_new = m->vv;
            a.kcache = kc, a.vcache = vc;
            a.cos_t = m->rope_cos, a.sin_t = m->rope_sin;
            a.pos = max_pos;
            a.dpos = m->capturing ? m->dpos : nullptr; // a captured step serves every position up to max_pos
            a.out = m->attg, a.scatter = nullptr;
            a.part = m->attn_part;
            a.n_heads = d.n_heads, a.n_kv_heads = d.n_kv_heads;
            a.max_splits = kMaxSplits;
            attn_split_policy(max_pos + 1, d.n_heads, d.n_kv_heads, &a.ts, &a.n_splits);
            if (a.n_splits > kMaxSplits)
                return l2_fail(L2_ERR_RANGE, "attention: position %d needs %d splits", max_pos, a.n_splits);
            LAUNCH(K_ATTENTION, attention_decode_launch(a, st));
        } else {
            LAUNCH(K_ROPE_KV, rope_kv_launch(m->qv, m->kv, m->vv, in.dpos, m->rope_cos, m->rope_sin, kc, vc, d.n_heads,
                                             d.n_kv_heads, m->head_size, B, st));
            LAUNCH(K_ATTENTION, attention_launch(m->attg, 0, m->qv, kc, vc, in.dpos, nullptr, d.n_heads,
                                                 d.n_kv_heads, m->head_size, max_pos, B, st));
        }
        LAUNCH(K_Q4_WO, dense(m->q[L2_WO][l], m->attg, m->x, m->x));                                                        // :260-264
        LAUNCH(K_Q4_W13, normed({{m->q[L2_W1][l].dense, m->hd, hid}, {m->q[L2_W3][l].dense, m->hg, hid}}, ffn_n, true)); // :266-276
        LAUNCH(K_Q4_W2, dense(m->q[L2_W2][l], m->hg, m->x, m->x));                                                          // :279-285
    }
    if (in.logits)
        LAUNCH(K_CLASSIFIER, dense_matvec_launch(in.logits, m->wcls, m->x, m->rms_final, m->rms_eps, dim,
                                                 d.vocab_size, in.amax, st));
    return L2_OK;
}

// Sizes of the four launches of a layer (q|k|v, wo, w1|w3, w2), for gemm_shape.
static Q4Launch layer_launch(const l2_model *m, int i, int B) {
    const l2_dims &d = m->d;
    const int outs[4][3] = {{d.dim, m->kv_dim, m->kv_dim}, {d.dim, 0, 0}, {d.hidden_dim, d.hidden_dim, 0}, {d.dim, 0, 0}};
    Q4Launch L{};
    L.in = i == 3 ? d.hidden_dim : d.dim, L.group_size = d.group_size, L.batch = B;
    for (int k = 0; k < 3 && outs[i][k]; k++) L.m[L.n_mats++].out = outs[i][k];
    return L;
}

// Whether chunks of a and of b columns are cut into the same K slices in every launch of a layer.
static bool cut_alike(const l2_model *m, int a, int b, int planes) {
    for (int i = 0; i < 4 && a != b; i++) {
        const Q4Launch L = layer_launch(m, i, a);
        const GemmShape p = gemm_shape(L, a, planes), q = gemm_shape(L, b, planes);
        if (p.slices != q.slices || p.last != q.last) return false;
    }
    return true;
}

// Buffers of one lane for passes of B columns cut as slice_batch columns are.
static int ensure_lane(l2_model *m, int lane, int B, int slice_batch, int planes) {
    l2_model::ChunkBufs &b = m->lane[lane];
    const l2_dims &d = m->d;
    const size_t wide = gemm_padded(std::max(d.dim, d.hidden_dim));
    size_t ws = 0; // partial tiles of the widest launch
    for (int i = 0; i < 4; i++) {
        const Q4Launch L = layer_launch(m, i, B);
        size_t rows = 0;
        for (int k = 0; k < L.n_mats; k++) rows += L.m[k].out;
        ws = std::max(ws, (size_t)gemm_shape(L, slice_batch, planes).slices * B * rows);
    }
    const size_t hb = (size_t)B * planes * wide * 2;
    if ((size_t)B <= b.cap_B && ws <= b.ws_floats && hb <= b.h_bytes) return L2_OK;
    L2_TRY(drain_streams(m));
    if ((size_t)B > b.cap_B) {
        float **f[3] = {&b.x, &b.q, &b.ss};
        for (float **p : f) dfree(*p), *p = nullptr;
        b.cap_B = 0;
        L2_TRY(dalloc(&b.x, (size_t)B * d.dim));
        L2_TRY(dalloc(&b.q, (size_t)B * d.dim));
        L2_TRY(dalloc(&b.ss, (size_t)B));
        b.cap_B = B;
    }
    if (ws > b.ws_floats) {
        dfree(b.ws);
        b.ws = nullptr, b.ws_floats = 0;
        L2_TRY(dalloc(&b.ws, ws));
        b.ws_floats = ws;
    }
    if (hb > b.h_bytes) {
        for (void *&p : b.h) dfree(p), p = nullptr;
        b.h_bytes = 0;
        for (void *&p : b.h) {
            char *c = nullptr;
            L2_TRY(dalloc(&c, hb));
            p = c;
        }
        b.h_bytes = hb;
    }
    return L2_OK;
}

// A pass of B positions through the matrix cores: the same schedule as forward_enqueue, with every QLinear as a GEMM
// over the B columns and what stands between two of them as one kernel.  Logits are never produced here
// (src/models.rs:288).  The pass may be several of the caller's chunks (slice_batch columns each, see GemmShape).
//
// The buffers and the stream are the lane's.  What a pass needs from the ones before it is their cache rows of the same
// layer, so `before_attn[l]` (the event of the pass before) is waited for in front of the attention of layer l, behind
// the kernel that writes this pass's own rows of layer l, and `after_kv[l]` is recorded right there (either may be null).
static int forward_enqueue_gemm(l2_model *m, l2_state *s, int B, int max_pos, const int32_t *dtok, const int32_t *dpos,
                                int planes, int slice_batch, int lane, bool beside, const hipEvent_t *after_kv,
                                const hipEvent_t *before_attn) {
    L2_TRY(check_position(m, max_pos));
    s->rows = std::max(s->rows, max_pos + 1);
    const l2_dims &d = m->d;
    const int dim = d.dim, hid = d.hidden_dim, kvd = m->kv_dim, L = d.n_layers;
    const l2_model::ChunkBufs &b = m->lane[lane];
    const bool dense = d.group_size == 0;
    hipStream_t st = lane ? m->extra_stream[lane - 1] : m->stream;
    auto gemm = [&](Q4Launch &Q, const XhList &X, const float *ss, int *ks) {
        return gemm_launch(Q, X, ss, b.ws, b.ws_floats, planes, slice_batch, st, ks, beside);
    };
    // rms scale of the stream in b.x and the inputs of layer l's q, k and v; ks partial tiles are added first
    auto attn_inputs = [&](int l, int ks) {
        ResNormPrep R{};
        R.ws = ks ? b.ws : nullptr, R.KS = ks ? ks : 1, R.B = B, R.out = dim, R.res = b.x, R.x = b.x, R.ss = b.ss, R.eps = m->rms_eps;
        R.n = 3, R.wn = m->rms_att + (size_t)l * dim;
        for (int c = 0; c < 3; c++) R.inv[c] = m->q[L2_WQ + c][l].inv_index, R.out_h[c] = b.h[c];
        if (dense) R.n = 1; // no act-order: one input serves q, k and v
        return gemm_residual_norm_launch(R, planes, st);
    };
    {
        ScatterTargets t{};
        TokenSource src;
        src.tokens = dtok;
        L2_TRY(embed_launch(b.x, m->tok_emb, src, dim, B, t, nullptr, st));
        L2_TRY(attn_inputs(0, 0));
    }
    for (int l = 0; l < L; l++) {
        const DevQLinear &wq = m->q[L2_WQ][l], &wk = m->q[L2_WK][l], &wv = m->q[L2_WV][l],
                         &wo = m->q[L2_WO][l], &w1 = m->q[L2_W1][l], &w2 = m->q[L2_W2][l],
                         &w3 = m->q[L2_W3][l];
        float *kc = s->kcache + (size_t)l * m->max_seq * kvd;
        float *vc = s->vcache + (size_t)l * m->max_seq * kvd;
        {   // q, k, v: partial tiles; the kernel that adds them also applies the rms scale, RoPE and the cache write
            Q4Launch Q = launch_of(wq, B, m->rms_eps);
            Q.m[0] = gemm_mat_of(wq, nullptr);
            Q.m[1] = gemm_mat_of(wk, nullptr);
            Q.m[2] = gemm_mat_of(wv, nullptr);
            Q.n_mats = 3;
            RopeKvArgs R{};
            L2_TRY(gemm(Q, dense ? XhList{{b.h[0], b.h[0], b.h[0]}} : XhList{{b.h[0], b.h[1], b.h[2]}}, nullptr, &R.KS));
            R.ws = b.ws, R.B = B, R.ss = b.ss, R.pos = dpos, R.cos_t = m->rope_cos, R.sin_t = m->rope_sin;
            R.q = b.q, R.kcache = kc, R.vcache = vc, R.n_heads = d.n_heads, R.n_kv_heads = d.n_kv_heads;
            L2_TRY(gemm_rope_kv_launch(R, st));
        }
        // Wait first, record second: the event of this pass then stands for its own rows of layer l AND, through
        // the event it waited for, for those of every pass before it, so that a pass two or more lanes behind
        // needs to wait for its direct predecessor only.
        if (before_attn) L2_HIP(hipStreamWaitEvent(st, before_attn[l], 0));
        if (after_kv) L2_HIP(hipEventRecord(after_kv[l], st));
        L2_TRY(attention_launch(b.h[0], planes, b.q, kc, vc, dpos, wo.inv_index, d.n_heads, d.n_kv_heads, m->head_size,
                                max_pos, B, st));
        {   // wo: partial tiles, then residual + rms scale + the inputs of w1 and w3 in one kernel
            Q4Launch Q = launch_of(wo, B, 0.f);
            Q.m[0] = gemm_mat_of(wo, nullptr);
            ResNormPrep R{};
            L2_TRY(gemm(Q, XhList{{b.h[0], nullptr, nullptr}}, nullptr, &R.KS));
            R.ws = b.ws, R.B = B, R.out = dim, R.res = b.x, R.x = b.x, R.ss = b.ss, R.eps = m->rms_eps;
            R.n = dense ? 1 : 2, R.wn = m->rms_ffn + (size_t)l * dim;
            R.inv[0] = w1.inv_index, R.out_h[0] = b.h[0];
            R.inv[1] = w3.inv_index, R.out_h[1] = b.h[1];
            L2_TRY(gemm_residual_norm_launch(R, planes, st));
        }
        {   // w1 | w3, then the gate in w2's order
            Q4Launch Q = launch_of(w1, B, m->rms_eps);
            Q.m[0] = gemm_mat_of(w1, nullptr);
            Q.m[1] = gemm_mat_of(w3, nullptr);
            Q.n_mats = 2;
            SiluArgs S{};
            L2_TRY(gemm(Q, XhList{{b.h[0], dense ? b.h[0] : b.h[1], nullptr}}, nullptr, &S.KS));
            S.ws = b.ws, S.B = B, S.n = hid, S.ss = b.ss, S.inv = w2.inv_index, S.out_h = b.h[2];
            L2_TRY(gemm_silu_launch(S, planes, st));
        }
        {   // w2; the kernel that adds its tiles hands the next layer its q, k and v inputs
            Q4Launch Q = launch_of(w2, B, 0.f);
            Q.m[0] = gemm_mat_of(w2, b.x);
            int ks = 0;
            if (l + 1 < L) {
                L2_TRY(gemm(Q, XhList{{b.h[2], nullptr, nullptr}}, nullptr, &ks));
                L2_TRY(attn_inputs(l + 1, ks));
            } else {
                Q.e.kind = Q4_EPI_RESIDUAL;
                Q.e.res = b.x;
                L2_TRY(gemm(Q, XhList{{b.h[2], nullptr, nullptr}}, nullptr, nullptr));
            }
        }
    }
    return L2_OK;
}

// transformer<B> on the model's stream for B > 1 tokens and positions already in device memory.
static int forward_batch(l2_model *m, l2_state *s, int B, int max_pos, const int32_t *dtok, const int32_t *dpos) {
    const int planes = batch_planes(m, B);
    if (!planes) {
        ForwardIn in;
        in.src.tokens = dtok, in.dpos = dpos;
        return forward_enqueue(m, s, B, max_pos, in);
    }
    L2_TRY(ensure_lane(m, 0, B, B, planes));
    return forward_enqueue_gemm(m, s, B, max_pos, dtok, dpos, planes, B, 0, false, nullptr, nullptr);
}

static int check_tokens(const l2_model *m, const int32_t *tokens, const int32_t *pos, int B, int *max_pos) {
    int mp = 0;
    for (int b = 0; b < B; b++) {
        if (tokens[b] < 0 || tokens[b] >= m->d.vocab_size)
            return l2_fail(L2_ERR_RANGE, "token id %d outside 0..%d", tokens[b], m->d.vocab_size - 1);
        if (pos[b] < 0 || pos[b] >= m->max_seq)
            return l2_fail(L2_ERR_RANGE, "position %d outside 0..%d", pos[b], m->max_seq - 1);
        mp = std::max(mp, pos[b]);
    }
    *max_pos = mp;
    return L2_OK;
}

extern "C" int l2_forward(l2_model *m, l2_state *s, const int32_t *tokens, const int32_t *pos, int B,
                          float *logits_host) {
    if (!m || !s || !tokens || !pos) return l2_fail(L2_ERR_ARG, "null argument");
    if (s->m != m) return l2_fail(L2_ERR_ARG, "state belongs to another model");
    if (B < 1 || B > 4096) return l2_fail(L2_ERR_RANGE, "batch %d (1..4096)", B);
    const AtWork at_work(m);
    int max_pos = 0;
    L2_TRY(check_tokens(m, tokens, pos, B, &max_pos));
    L2_TRY(ensure_batch(m, B));
    if (B > 1) {
        L2_TRY(ensure_ids(m, B));
        L2_TRY(claim_host_ids(m));
        memcpy(m->hs.in, tokens, (size_t)B * 4);
        memcpy(m->hs.in + B, pos, (size_t)B * 4);
        L2_HIP(hipMemcpyAsync(m->pf_ids, m->hs.in, (size_t)B * 8, hipMemcpyHostToDevice, m->stream));
        L2_TRY(forward_batch(m, s, B, max_pos, m->pf_ids, m->pf_ids + B));
        return wait_host(m, nullptr, nullptr);
    }
    ForwardIn in;
    in.src.token = tokens[0], in.whole = true;
    in.logits = logits_host ? m->hs.logits : m->logits, in.amax = m->amax;
    L2_TRY(token_tries(m, [&]() -> int {
        L2_TRY(forward_enqueue(m, s, 1, max_pos, in));
        return wait_host(m, nullptr, nullptr);
    }));
    if (logits_host) memcpy(logits_host, m->hs.logits, (size_t)m->d.vocab_size * 4);
    return L2_OK;
}

int l2_forward_weights(l2_model *m, l2_state *s, int32_t token, int32_t pos, float temperature, bool more, SampleWeights *out) {
    if (s->m != m) return l2_fail(L2_ERR_ARG, "state belongs to another model");
    const AtWork at_work(m);
    int max_pos = 0;
    L2_TRY(check_tokens(m, &token, &pos, 1, &max_pos));
    L2_TRY(ensure_batch(m, 1));
    ForwardIn in;
    in.src.token = token, in.logits = m->logits, in.amax = m->amax, in.whole = true;
    L2_TRY(token_tries(m, [&]() -> int {
        L2_TRY(forward_enqueue(m, s, 1, pos, in));
        L2_TRY(sample_weights_launch(m->hs.logits, m->hs.redo, m->logits, m->d.vocab_size, temperature, m->amax, m->stream));
        if (!more) return wait_host(m, nullptr, nullptr);
        // an event is all that a step inside a call has to wait for (7B: 24 us less than for the stream)
        if (!m->step_done) L2_HIP(hipEventCreateWithFlags(&m->step_done, hipEventDisableTiming));
        L2_HIP(hipEventRecord(m->step_done, m->stream));
        L2_HIP(hipEventSynchronize(m->step_done));
        return L2_OK;
    }));
    *out = {m->hs.logits, m->hs.redo};
    return L2_OK;
}

// One pass over consecutive positions: whole chunks of the caller's that are cut into the same K slices.
struct PrefillPass {
    int first, n, slice_batch, planes;
};
// The lanes of l2_prefill_chunks: streams, events and buffers for `passes`, any of them on any lane.  (A longer chunk may be
// cut into more slices than a shorter one, so no single pass stands for all.)
static int ensure_prefill_pipeline(l2_model *m, int lanes, const std::vector<PrefillPass> &passes) {
    for (int i = 0; i + 1 < lanes; i++)
        if (!m->extra_stream[i]) L2_HIP(hipStreamCreate(&m->extra_stream[i])); // default priority, as the model's own
    if (!m->pf_join) L2_HIP(hipEventCreateWithFlags(&m->pf_join, hipEventDisableTiming));
    for (int i = 0; i < lanes; i++) {
        while ((int)m->pf_ev[i].size() < m->d.n_layers) {
            hipEvent_t e = nullptr;
            L2_HIP(hipEventCreateWithFlags(&e, hipEventDisableTiming));
            m->pf_ev[i].push_back(e);
        }
        for (size_t p = 0; p < passes.size(); p++) {
            const bool again = p > 0 && passes[p].n == passes[p - 1].n && passes[p].slice_batch == passes[p - 1].slice_batch;
            if (passes[p].planes && !again) L2_TRY(ensure_lane(m, i, passes[p].n, passes[p].slice_batch, passes[p].planes));
        }
    }
    return L2_OK;
}

static constexpr int kPassTokens = 512;

// prefill<A> (src/inference.rs:16-40) for a whole prompt: tokens[i] at position pos0 + i, in chunks of `chunk`, no
// logits.  Chunks that the GEMM cuts alike go through it together, up to kPassTokens at a time: a column's arithmetic
// does not depend on the columns beside it, so every chunk is what l2_forward computes for it, bit for bit, and the
// weights are read and dequantised once per pass.  Passes run on n_lanes streams, each with buffers of its own: a pass
// needs from its predecessor only the cache rows of the same layer (an event per layer), so every pass follows one layer
// behind the one before it and its kernels fill the compute units that the others' short launches leave idle.
static int prefill_chunks(l2_model *m, l2_state *s, const int32_t *tokens, int n, int pos0, int chunk, bool wait) {
    if (!m || !s || !tokens) return l2_fail(L2_ERR_ARG, "null argument");
    if (s->m != m) return l2_fail(L2_ERR_ARG, "state belongs to another model");
    const AtWork at_work(m);
    if (n < 1 || chunk < 1 || chunk > 4096) return l2_fail(L2_ERR_RANGE, "%d tokens in chunks of %d (1..4096)", n, chunk);
    if (pos0 < 0 || (long)pos0 + n > m->max_seq)
        return l2_fail(L2_ERR_RANGE, "positions %d..%ld outside 0..%d", pos0, (long)pos0 + n - 1, m->max_seq - 1);
    for (int i = 0; i < n; i++)
        if (tokens[i] < 0 || tokens[i] >= m->d.vocab_size)
            return l2_fail(L2_ERR_RANGE, "token id %d outside 0..%d", tokens[i], m->d.vocab_size - 1);
    std::vector<PrefillPass> passes;
    int rest = 0; // most columns of a chunk that the matvec kernels take
    for (int c0 = 0; c0 < n; c0 += chunk) {
        const int B = std::min(chunk, n - c0), p = batch_planes(m, B);
        if (!p) rest = std::max(rest, B);
        if (p && !passes.empty()) {
            PrefillPass &last = passes.back();
            if (last.planes == p && cut_alike(m, last.slice_batch, B, p) && last.n + B <= kPassTokens) {
                last.n += B;
                continue;
            }
        }
        passes.push_back({c0, B, B, p});
    }
    const int lanes = passes.size() > 1 ? m->n_lanes : 1;
    L2_TRY(ensure_batch(m, std::max(rest, 1)));
    L2_TRY(ensure_prefill_pipeline(m, lanes, passes));
    L2_TRY(ensure_ids(m, n));
    L2_TRY(claim_host_ids(m));
    memcpy(m->hs.in, tokens, (size_t)n * 4);
    for (int i = 0; i < n; i++) m->hs.in[n + i] = pos0 + i;
    const int32_t *dtok = m->pf_ids, *dpos = m->pf_ids + n;
    L2_HIP(hipMemcpyAsync(m->pf_ids, m->hs.in, (size_t)n * 8, hipMemcpyHostToDevice, m->stream));
    if (lanes > 1) { // the other lanes start behind what the model's stream has been given so far
        L2_HIP(hipEventRecord(m->pf_join, m->stream));
        for (int i = 0; i + 1 < lanes; i++) L2_HIP(hipStreamWaitEvent(m->extra_stream[i], m->pf_join, 0));
    }
    // Everything that is enqueued on the two streams; a failure half-way returns through the caller below, which
    // first waits for what earlier chunks already have in flight on either stream.
    // the model's stream waits for everything the other lanes have been given so far
    auto join_lanes = [&]() -> int {
        for (int i = 0; i + 1 < lanes; i++) {
            L2_HIP(hipEventRecord(m->pf_join, m->extra_stream[i]));
            L2_HIP(hipStreamWaitEvent(m->stream, m->pf_join, 0));
        }
        return L2_OK;
    };
    auto enqueue_all = [&]() -> int {
        const bool beside = lanes > 1 && std::count_if(passes.begin(), passes.end(), [](const PrefillPass &p) { return p.planes != 0; }) > 1;
        int c = 0; // GEMM passes so far
        for (const PrefillPass &p : passes) {
            const int max_pos = pos0 + p.first + p.n - 1;
            if (p.planes) {
                const int lane = c % lanes, before = (c + lanes - 1) % lanes;
                L2_TRY(forward_enqueue_gemm(m, s, p.n, max_pos, dtok + p.first, dpos + p.first, p.planes, p.slice_batch,
                                            lane, beside, passes.size() > 1 ? m->pf_ev[lane].data() : nullptr, c > 0 ? m->pf_ev[before].data() : nullptr));
                c++;
            } else {
                // few columns: the matvec kernels on the model's stream, behind everything
                L2_TRY(join_lanes());
                ForwardIn in;
                in.src.tokens = dtok + p.first, in.dpos = dpos + p.first;
                L2_TRY(forward_enqueue(m, s, p.n, max_pos, in));
            }
        }
        return join_lanes();
    };
    const int rc = enqueue_all();
    if (rc != L2_OK) {
        // kernels of earlier chunks may still be writing cache rows and chunk buffers on both streams: nothing
        // returns to the caller (who may reset the state or free the model next) before they are done.  The
        // error text of the failure that brought us here is kept.
        char keep[sizeof g_err];
        memcpy(keep, g_err, sizeof keep);
        (void)hipStreamSynchronize(m->stream);
        for (hipStream_t es : m->extra_stream)
            if (es) (void)hipStreamSynchronize(es);
        memcpy(g_err, keep, sizeof keep);
        return rc;
    }
    return wait ? wait_host(m, nullptr, nullptr) : L2_OK;
}

extern "C" int l2_prefill_chunks(l2_model *m, l2_state *s, const int32_t *tokens, int n, int pos0, int chunk) {
    return prefill_chunks(m, s, tokens, n, pos0, chunk, true);
}

static int steps_enqueue(l2_model *m, l2_state *s, int32_t first, int pos0, int n, const int32_t *prompt, int n_prompt);
static int steps_collect(l2_model *m, int pos0, int n, const int32_t *prompt, int n_prompt, int32_t *ids);
static int steps_run(l2_model *m, l2_state *s, int32_t first, int pos0, int n, const int32_t *prompt, int n_prompt, int32_t *ids);

extern "C" int l2_decode_greedy(l2_model *m, l2_state *s, int32_t token, int32_t pos, int32_t *next) {
    if (!m || !s || !next) return l2_fail(L2_ERR_ARG, "null argument");
    if (s->m != m) return l2_fail(L2_ERR_ARG, "state belongs to another model");
    const AtWork at_work(m);
    int max_pos = 0;
    L2_TRY(check_tokens(m, &token, &pos, 1, &max_pos));
    L2_TRY(ensure_batch(m, 1));
    return steps_run(m, s, token, pos, 1, nullptr, 0, next);
}

static int ensure_loop_buffers(l2_model *m, int n_prompt, int n_out) {
    if (n_prompt > m->cap_prompt) {
        L2_HIP(hipStreamSynchronize(m->stream));
        m->buf_epoch++;
        dfree(m->dprompt);
        m->dprompt = nullptr;
        m->cap_prompt = 0;
        L2_TRY(dalloc(&m->dprompt, (size_t)n_prompt));
        m->cap_prompt = n_prompt;
    }
    if (n_out > m->cap_out) {
        L2_HIP(hipStreamSynchronize(m->stream));
        m->buf_epoch++;
        dfree(m->dout_ids);
        m->dout_ids = nullptr;
        m->cap_out = 0;
        L2_TRY(dalloc(&m->dout_ids, (size_t)n_out));
        m->cap_out = n_out;
    }
    return L2_OK;
}

static void step_graph_drop(StepGraph &g) {
    if (g.exec) (void)hipGraphExecDestroy(g.exec);
    if (g.graph) (void)hipGraphDestroy(g.graph);
    g = StepGraph{};
}

// The captured form of the same step for every position below `upper`: the kernels read the position, the
// prompt length and the first position of the loop from device memory (m->dpos, m->dloop), attention is
// cut for `upper` timesteps and blocks beyond the current position leave at once.
static int step_graph_get(l2_model *m, l2_state *s, int upper, hipGraphExec_t *out) {
    StepGraph &g = s->steps[upper];
    if (g.exec && g.epoch == m->buf_epoch) {
        *out = g.exec;
        return L2_OK;
    }
    step_graph_drop(g);
    L2_HIP(hipStreamBeginCapture(m->stream, hipStreamCaptureModeRelaxed));
    m->capturing = true;
    ForwardIn in;
    in.src.tokens = m->dtok, in.logits = m->logits, in.amax = m->amax;
    const int rows = s->rows; // capturing writes nothing
    int rc = forward_enqueue(m, s, 1, upper - 1, in);
    s->rows = rows;
    if (rc == L2_OK)
        rc = next_token_launch(m->amax, m->dprompt, 0, m->dpos, m->dout_ids, 0, m->dtok, m->stream, m->dloop);
    m->capturing = false;
    hipGraph_t graph = nullptr;
    const hipError_t e = hipStreamEndCapture(m->stream, &graph);
    if (rc != L2_OK) {
        if (graph) (void)hipGraphDestroy(graph);
        return rc;
    }
    if (e != hipSuccess) return l2_fail(L2_ERR_HIP, "hipStreamEndCapture: %s", hipGetErrorString(e));
    g.graph = graph;
    const hipError_t e2 = hipGraphInstantiate(&g.exec, graph, nullptr, nullptr, 0);
    if (e2 != hipSuccess) {
        step_graph_drop(g);
        return l2_fail(L2_ERR_HIP, "hipGraphInstantiate: %s", hipGetErrorString(e2));
    }
    g.epoch = m->buf_epoch;
    *out = g.exec;
    return L2_OK;
}

// Positions are served in buckets [0, 256), [256, 512), [512, 1024), ...: one captured step each.
static int step_bucket(const l2_model *m, int pos) {
    long upper = 256;
    while (upper <= pos) upper *= 2;
    if (upper > m->max_seq) upper = m->max_seq;
    return (int)upper;
}

// The B = 1 loop (src/inference.rs:141-162) with everything on the device: n steps from token `first` at position pos0,
// each one's next token being prompt[pos] while that is inside the prompt, else the argmax.
//
// Launched: the embedding kernel of a step takes the step before's argmax itself and records it (in pinned host memory),
// so a step is its layers' launches, one in front and the classifier, or the token kernel and the classifier.  Forced tokens travel as kernel arguments.
// As graphs: see step_graph_get.
static constexpr int kAskLaunches = 128;
static constexpr double kAskWeights = 5e7; // a layer of 7B has 2e8 and takes 40 us
// Steps in token kernels leave little room for other calls' kernels (DeviceCalls), which may come at any time, so a loop has no more of them
// enqueued than 2 * steps_ahead, some 2 * kAheadUs; an event that is waited for every 4 ms costs some 1 us of each ms (7B 1053 -> 1054 us a step).
static constexpr double kAheadUs = 4000;
static int steps_ahead(const l2_model *m) {
    const double us = m->d.n_layers * (layer_weights(m) * 0.53 / 4.2e6 + 12) + (double)m->d.vocab_size * m->d.dim * 4 / 5e6;
    return std::max(2, (int)(kAheadUs / us));
}
static int steps_enqueue(l2_model *m, l2_state *s, int32_t first, int pos0, int n, const int32_t *prompt, int n_prompt) {
    if (m->use_graph && !m->prof_on) {
        L2_TRY(ensure_loop_buffers(m, std::max(n_prompt, 1), std::max(n, 1)));
        if (n_prompt > 0) {
            L2_TRY(claim_host_ids(m)); // a prefill before may still be reading its ids there
            memcpy(m->hs.in, prompt, (size_t)std::min(n_prompt, m->max_seq) * 4);
            L2_HIP(hipMemcpyAsync(m->dprompt, m->hs.in, (size_t)std::min(n_prompt, m->max_seq) * 4, hipMemcpyHostToDevice, m->stream));
        }
        L2_TRY(set_i32_launch(m->dtok, first, m->dpos, pos0, m->stream));
        L2_TRY(set_i32_launch(m->dloop, n_prompt, m->dloop + 1, pos0, m->stream));
        for (int pos = pos0; pos < pos0 + n; pos++) {
            L2_TRY(check_position(m, pos));
            hipGraphExec_t exec = nullptr;
            L2_TRY(step_graph_get(m, s, step_bucket(m, pos), &exec));
            s->rows = std::max(s->rows, pos + 1);
            L2_HIP(hipGraphLaunch(exec, m->stream));
        }
        return L2_OK;
    }
    // The runtime keeps a record of every launch until it is asked about the stream or has a thousand of them, and a loop of
    // so many launches behind a synchronisation is slow to enqueue in most processes (three layers of 1024 inputs, 48 steps:
    // 2.1 or 3.2 ms, 4.0 or 4.5 ms in all; 167 steps 14.0 or 14.5).  Asked about in between, the loop takes 4.04 and 14.1 ms in
    // every process.  That pays where a launch is too short to hide the enqueueing (an ask costs the GPU 5 us); not shortly
    // before the end, where the wait would meet it.
    const bool asks = layer_weights(m) < kAskWeights;
    int since = 0; // launches since it was asked
    const int ahead = steps_ahead(m);
    int in_ones = 0, records = 0;
    ForwardIn in;
    in.src.token = first, in.logits = m->logits, in.whole = true;
    for (int i = 0; i < n; i++) {
        const int pos = pos0 + i;
        in.amax = m->amax + (i & 1);
        const uint64_t in_one = m->tok.steps;
        L2_TRY(forward_enqueue(m, s, 1, pos, in));
        // by the route that this step has taken: the next one's may be another
        const int launches = m->tok.steps != in_one ? 2 : 5 * m->d.n_layers + 2, ask_steps = std::max(1, kAskLaunches / launches);
        since += launches;
        if (asks && since >= ask_steps * launches && i + ask_steps < n) {
            if (hipStreamQuery(m->stream) == hipErrorNotReady) (void)hipGetLastError();
            since = 0, m->asked++;
        }
        if (m->tok.steps != in_one && ++in_ones % ahead == 0 && i + 1 < n) {
            for (hipEvent_t &e : m->ahead)
                if (!e) L2_HIP(hipEventCreateWithFlags(&e, hipEventDisableTiming));
            L2_HIP(hipEventRecord(m->ahead[records & 1], m->stream));
            if (records++ > 0) L2_HIP(hipEventSynchronize(m->ahead[records & 1]));
        }
        in.src = TokenSource{};
        if (pos < n_prompt)
            in.src.token = prompt[pos];
        else
            in.src.prev = in.amax, in.src.record = m->hs.ids + i;
    }
    return L2_OK;
}

// Waits for the steps above and hands out every one's next token.
static int steps_collect(l2_model *m, int pos0, int n, const int32_t *prompt, int n_prompt, int32_t *ids) {
    if (n == 0) return wait_host(m, nullptr, nullptr);
    if (m->use_graph && !m->prof_on) {
        L2_HIP(hipMemcpyAsync(m->hs.ids, m->dout_ids, (size_t)n * 4, hipMemcpyDeviceToHost, m->stream));
        L2_TRY(wait_host(m, nullptr, nullptr));
    } else {
        const bool forced = pos0 + n - 1 < n_prompt;
        L2_TRY(wait_host(m, forced ? nullptr : m->amax + ((n - 1) & 1), m->hs.ids + n - 1));
        for (int i = 0; i < n && pos0 + i < n_prompt; i++) m->hs.ids[i] = prompt[pos0 + i];
    }
    if (ids) memcpy(ids, m->hs.ids, (size_t)n * 4);
    return L2_OK;
}

static int steps_run(l2_model *m, l2_state *s, int32_t first, int pos0, int n, const int32_t *prompt, int n_prompt, int32_t *ids) {
    return token_tries(m, [&]() -> int {
        L2_TRY(steps_enqueue(m, s, first, pos0, n, prompt, n_prompt));
        return steps_collect(m, pos0, n, prompt, n_prompt, ids);
    });
}

// Position at which prefill<64>, <32>, ... <2> (src/inference.rs:78-127) leave off for a prompt of n_prompt
// tokens: each takes chunks of A positions while pos + A < n_prompt (:24).
int l2_prefill_ladder_end(int n_prompt) {
    int pos = 0;
    for (int A = 64; A >= 2; A /= 2)
        while (pos + A < n_prompt) pos += A;
    return pos;
}

// The rungs of the ladder one behind the other are one prompt: the tokens START, prompt[0], ... (:29-33) at the
// positions before l2_prefill_ladder_end.  They go through in as few, evenly filled passes as kPassTokens allows.
int l2_prefill_ladder(l2_model *m, l2_state *s, const int32_t *prompt, int n_prompt, bool wait) {
    const int n = l2_prefill_ladder_end(n_prompt);
    if (n == 0) return L2_OK;
    std::vector<int32_t> toks((size_t)n);
    for (int i = 0; i < n; i++) toks[i] = i == 0 ? 1 : prompt[i - 1];
    const int passes = (n + kPassTokens - 1) / kPassTokens;
    return prefill_chunks(m, s, toks.data(), n, 0, (n + passes - 1) / passes, wait);
}

extern "C" int l2_generate_greedy(l2_model *m, l2_state *s, const int32_t *prompt, int n_prompt, int steps,
                                  int use_prefill, int32_t *out_ids, int *n_out, double *ms) {
    if (!m || !s || !out_ids || !n_out || (n_prompt > 0 && !prompt)) return l2_fail(L2_ERR_ARG, "null argument");
    if (s->m != m) return l2_fail(L2_ERR_ARG, "state belongs to another model");
    if (n_prompt < 0 || steps < 0) return l2_fail(L2_ERR_ARG, "negative count");
    if (steps > m->max_seq) return l2_fail(L2_ERR_RANGE, "steps %d exceeds the cache length %d", steps, m->max_seq);
    const AtWork at_work(m);
    // The ladder runs whatever `steps` is: a prompt it would carry past the cache is refused before any launch
    // (the reference panics there on its fixed [SEQ_LEN] arrays).
    if (use_prefill && l2_prefill_ladder_end(n_prompt) > m->max_seq)
        return l2_fail(L2_ERR_RANGE, "a prompt of %d tokens prefills %d positions, the cache holds %d", n_prompt,
                       l2_prefill_ladder_end(n_prompt), m->max_seq);
    for (int i = 0; i < n_prompt; i++)
        if (prompt[i] < 0 || prompt[i] >= m->d.vocab_size)
            return l2_fail(L2_ERR_RANGE, "prompt token %d outside 0..%d", prompt[i], m->d.vocab_size - 1);
    L2_TRY(state_clear(s)); // RunState::new per call (:59)
    L2_TRY(ensure_batch(m, 1));
    const auto t0 = std::chrono::steady_clock::now(); // :72
    int pos = 0;
    if (use_prefill) { // :78-127
        pos = l2_prefill_ladder_end(n_prompt);
        L2_TRY(l2_prefill_ladder(m, s, prompt, n_prompt, false));
    }
    const int32_t first = pos == 0 ? 1 : prompt[pos - 1]; // :128-132
    const int n = std::max(steps - pos, 0); // :141
    if (n > 0 && pos + n > m->max_seq) return l2_fail(L2_ERR_RANGE, "position %d outside 0..%d", pos + n - 1, m->max_seq - 1);
    L2_TRY(steps_run(m, s, first, pos, n, prompt, n_prompt, out_ids));
    const auto t1 = std::chrono::steady_clock::now(); // :192
    *n_out = n;
    if (ms) *ms = std::chrono::duration<double, std::milli>(t1 - t0).count();
    return L2_OK;
}

// ---------------------------------------------------------------------------
// measurement hooks

extern "C" int l2_qlinear_set_device(l2_qlinear *q, int device) {
    if (!q || device < 0) return l2_fail(L2_ERR_ARG, "bad argument");
    q->device = device;
    return L2_OK;
}

extern "C" int l2_host_windows_taken(uint64_t *n) {
    if (!n) return l2_fail(L2_ERR_ARG, "null argument");
    std::lock_guard<std::mutex> lock(host_windows.mu);
    *n = host_windows.taken;
    return L2_OK;
}

extern "C" int l2_qlinear_bench(l2_qlinear **qs, int n, int iters, float *ms_total) {
    if (!qs || n < 1 || iters < 1 || !ms_total) return l2_fail(L2_ERR_ARG, "bad argument");
    hipStream_t st = qs[0]->stream;
    for (int i = 0; i < n; i++) {
        if (!qs[i]) return l2_fail(L2_ERR_ARG, "null qlinear %d", i);
        L2_TRY(qlinear_scratch(qs[i], 1));
        L2_TRY(fill_pattern_launch(qs[i]->x, (size_t)qs[i]->q.in, 17 + i, st));
    }
    hipEvent_t e0, e1;
    L2_HIP(hipEventCreate(&e0));
    L2_HIP(hipEventCreate(&e1));
    for (int i = 0; i < n; i++) L2_TRY(q4_one_natural(qs[i]->q, qs[i]->x, qs[i]->xg, qs[i]->y, 1, st)); // warm-up
    L2_HIP(hipStreamSynchronize(st));
    L2_HIP(hipEventRecord(e0, st));
    for (int it = 0; it < iters; it++) { // the whole operator: x in its natural order -> y, the act-order gather included
        l2_qlinear *q = qs[it % n];
        L2_TRY(q4_one_natural(q->q, q->x, q->xg, q->y, 1, st));
    }
    L2_HIP(hipEventRecord(e1, st));
    L2_HIP(hipEventSynchronize(e1));
    L2_HIP(hipEventElapsedTime(ms_total, e0, e1));
    (void)hipEventDestroy(e0);
    (void)hipEventDestroy(e1);
    return L2_OK;
}

extern "C" int l2_qlinear_bench_dispatch(l2_qlinear **qs, int n, int iters, float *ms_sum) {
    if (!qs || n < 1 || iters < 1 || iters > 65536 || !ms_sum) return l2_fail(L2_ERR_ARG, "bad argument");
    hipStream_t st = qs[0]->stream;
    for (int i = 0; i < n; i++) {
        if (!qs[i]) return l2_fail(L2_ERR_ARG, "null qlinear %d", i);
        L2_TRY(qlinear_scratch(qs[i], 1));
        L2_TRY(fill_pattern_launch(qs[i]->x, (size_t)qs[i]->q.in, 17 + i, st));
    }
    for (int i = 0; i < n; i++) {
        Q4Launch probe = launch_of(qs[i]->q, 1, 0.f);
        probe.m[0] = mat_of(qs[i]->q, qs[i]->x, nullptr, qs[i]->y);
        if (!q4_gathers_in_kernel(probe))
            return l2_fail(L2_ERR_ARG, "dispatch timing covers the one-launch form of the operator only (in=%d)", qs[i]->q.in);
        L2_TRY(q4_one_natural(qs[i]->q, qs[i]->x, qs[i]->xg, qs[i]->y, 1, st)); // warm-up
    }
    L2_HIP(hipStreamSynchronize(st));
    std::vector<hipEvent_t> ev((size_t)iters * 2, nullptr);
    int rc = L2_OK;
    for (auto &e : ev)
        if (rc == L2_OK && hipEventCreate(&e) != hipSuccess) rc = l2_fail(L2_ERR_HIP, "hipEventCreate failed");
    int launched = 0;
    for (int it = 0; it < iters && rc == L2_OK; it++) {
        l2_qlinear *q = qs[it % n];
        g_q4_prof.start = ev[2 * (size_t)it];
        g_q4_prof.stop = ev[2 * (size_t)it + 1];
        g_q4_prof.armed = true;
        rc = q4_one_natural(q->q, q->x, q->xg, q->y, 1, st);
        if (rc == L2_OK && g_q4_prof.armed) rc = l2_fail(L2_ERR_ARG, "this form of the kernel takes no dispatch events");
        g_q4_prof.armed = false;
        if (rc == L2_OK) launched++;
    }
    const hipError_t es = hipStreamSynchronize(st);
    double sum = 0.0;
    for (int it = 0; it < launched && rc == L2_OK && es == hipSuccess; it++) {
        float ms = 0.f;
        if (hipEventElapsedTime(&ms, ev[2 * (size_t)it], ev[2 * (size_t)it + 1]) != hipSuccess)
            rc = l2_fail(L2_ERR_HIP, "hipEventElapsedTime failed on dispatch %d", it);
        sum += ms;
    }
    for (auto &e : ev)
        if (e) (void)hipEventDestroy(e);
    if (rc != L2_OK) return rc;
    if (es != hipSuccess) return l2_fail(L2_ERR_HIP, "matvec bench: %s", hipGetErrorString(es));
    *ms_sum = (float)sum;
    return L2_OK;
}

extern "C" int l2_qlinear_kernel(l2_qlinear *q, char *out, size_t cap) {
    if (!q || !out || cap < 2) return l2_fail(L2_ERR_ARG, "bad argument");
    out[0] = '\0';
    const float *some = (const float *)q->bufs[2]; // only null / non-null matters for the choice of kernel
    Q4Launch L = launch_of(q->q, 1, 0.f);
    L.m[0] = mat_of(q->q, some, nullptr, nullptr);
    if (q4_gathers_in_kernel(L)) L.m[0].gidx = q->q.inv_index;
    g_q4_name.buf = out;
    g_q4_name.cap = (int)cap;
    g_q4_name.armed = true;
    const int rc = q4_matvec_launch(L, q->stream);
    const bool answered = !g_q4_name.armed;
    g_q4_name.armed = false;
    L2_TRY(rc);
    if (!answered) return l2_fail(L2_ERR_ARG, "the launcher did not name its kernel");
    return L2_OK;
}

extern "C" int l2_decode_bench(l2_model *m, l2_state *s, int32_t token, int32_t pos, int n_tokens,
                               int32_t *out_ids, float *ms_total) {
    if (!m || !s || !ms_total || n_tokens < 1) return l2_fail(L2_ERR_ARG, "bad argument");
    if (s->m != m) return l2_fail(L2_ERR_ARG, "state belongs to another model");
    if (pos < 0 || pos + n_tokens > m->max_seq) return l2_fail(L2_ERR_RANGE, "positions [%d,%d) exceed the cache", pos, pos + n_tokens);
    if (token < 0 || token >= m->d.vocab_size) return l2_fail(L2_ERR_RANGE, "token %d", token);
    const AtWork at_work(m);
    L2_TRY(ensure_batch(m, 1));
    if (m->use_graph) { // capture (if need be) outside the timed region
        L2_TRY(ensure_loop_buffers(m, 1, n_tokens));
        hipGraphExec_t exec = nullptr;
        for (int b = step_bucket(m, pos);; b = step_bucket(m, b)) {
            L2_TRY(step_graph_get(m, s, b, &exec));
            if (b > pos + n_tokens - 1 || b >= m->max_seq) break;
        }
    }
    hipEvent_t e0, e1;
    L2_HIP(hipEventCreate(&e0));
    L2_HIP(hipEventCreate(&e1));
    L2_HIP(hipStreamSynchronize(m->stream));
    const int rc = token_tries(m, [&]() -> int {
        L2_HIP(hipEventRecord(e0, m->stream));
        L2_TRY(steps_enqueue(m, s, token, pos, n_tokens, nullptr, 0));
        L2_HIP(hipEventRecord(e1, m->stream));
        L2_HIP(hipEventSynchronize(e1));
        L2_HIP(hipEventElapsedTime(ms_total, e0, e1));
        return steps_collect(m, pos, n_tokens, nullptr, 0, out_ids);
    });
    (void)hipEventDestroy(e0);
    (void)hipEventDestroy(e1);
    return rc;
}

// Which kernel each q4 launch class of this model's decode step runs: "class=kernel;..." with the kernel's
// name as a profiler prints it (template arguments included).  Nothing is launched.
extern "C" int l2_model_q4_kernels(l2_model *m, char *out, size_t cap) {
    if (!m || !out || cap < 2) return l2_fail(L2_ERR_ARG, "bad argument");
    out[0] = '\0';
    if (m->d.group_size == 0) return L2_OK; // the model without quantisation has no q4 launches
    const int layer = 0;
    const DevQLinear &wq = m->q[L2_WQ][layer], &wk = m->q[L2_WK][layer], &wv = m->q[L2_WV][layer],
                     &wo = m->q[L2_WO][layer], &w1 = m->q[L2_W1][layer], &w2 = m->q[L2_W2][layer],
                     &w3 = m->q[L2_W3][layer];
    const float *some = (const float *)m->dimage; // only null / non-null matters for the choice of kernel
    struct { const char *cls; Q4Launch L; } items[4];
    items[0].cls = "q4_qkv";
    items[0].L = launch_of(wq, 1, m->rms_eps);
    items[0].L.m[0] = mat_of(wq, some, some, nullptr);
    items[0].L.m[1] = mat_of(wk, some, some, nullptr);
    items[0].L.m[2] = mat_of(wv, some, some, nullptr);
    items[0].L.n_mats = 3;
    items[1].cls = "q4_wo";
    items[1].L = launch_of(wo, 1, 0.f);
    items[1].L.m[0] = mat_of(wo, some, nullptr, nullptr);
    items[1].L.e.kind = Q4_EPI_RESIDUAL;
    items[2].cls = "q4_w13";
    items[2].L = launch_of(w1, 1, m->rms_eps);
    items[2].L.m[0] = mat_of(w1, some, some, nullptr);
    items[2].L.m[1] = mat_of(w3, some, some, nullptr);
    items[2].L.n_mats = 2;
    items[2].L.pair = 1;
    items[3].cls = "q4_w2";
    items[3].L = launch_of(w2, 1, 0.f);
    items[3].L.m[0] = mat_of(w2, some, nullptr, nullptr);
    items[3].L.e.kind = Q4_EPI_RESIDUAL;
    std::string all;
    for (auto &it : items) {
        char name[160] = "";
        g_q4_name.buf = name;
        g_q4_name.cap = (int)sizeof(name);
        g_q4_name.armed = true;
        const int rc = q4_matvec_launch(it.L, m->stream);
        const bool answered = !g_q4_name.armed;
        g_q4_name.armed = false;
        L2_TRY(rc);
        if (!answered) return l2_fail(L2_ERR_ARG, "the launcher of %s did not name its kernel", it.cls);
        all += std::string(it.cls) + "=" + name + ";";
    }
    if (all.size() + 1 > cap) return l2_fail(L2_ERR_ARG, "buffer of %zu bytes, %zu needed", cap, all.size() + 1);
    memcpy(out, all.c_str(), all.size() + 1);
    return L2_OK;
}

// What the q4 launcher would do for L: nothing is launched, only null / non-null pointers matter.
static int plan_of(Q4Launch &L, char *kernel, size_t cap, int32_t *geometry) {
    kernel[0] = '\0';
    g_q4_name = Q4NameHook{};
    g_q4_name.buf = kernel;
    g_q4_name.cap = (int)cap;
    g_q4_name.armed = true;
    const int rc = q4_matvec_launch(L, nullptr);
    const bool answered = !g_q4_name.armed;
    g_q4_name.armed = false;
    L2_TRY(rc);
    if (!answered) return l2_fail(L2_ERR_ARG, "the launcher did not name its kernel");
    geometry[0] = g_q4_name.grid, geometry[1] = g_q4_name.block, geometry[2] = g_q4_name.rows_per_block;
    geometry[3] = (int32_t)g_q4_name.lds;
    // every row of every matrix belongs to exactly one block, and the blocks of all matrices fit the grid
    long blocks = 0;
    for (int i = 0; i < (L.pair ? 1 : L.n_mats); i++) blocks += (L.m[i].out + geometry[2] - 1) / geometry[2];
    if (blocks != geometry[0]) return l2_fail(L2_ERR_ARG, "plan: %ld row blocks for a grid of %d", blocks, geometry[0]);
    return L2_OK;
}

extern "C" int l2_q4_plan(int in, const int32_t *out, int n_mats, int group_size, int pair, int norm, char *kernel,
                          size_t cap, int32_t *geometry) {
    if (!out || !kernel || cap < 2 || !geometry || n_mats < 1 || n_mats > 3) return l2_fail(L2_ERR_ARG, "bad argument");
    if (group_size != 32 && group_size != 64 && group_size != 128) return l2_fail(L2_ERR_ARG, "group size %d", group_size);
    if (in <= 0 || in % 32 || in % group_size) return l2_fail(L2_ERR_ARG, "in=%d", in);
    static const float dummy[4] = {0.f, 0.f, 0.f, 0.f};
    Q4Launch L{};
    L.n_mats = n_mats;
    L.in = in;
    L.groups = in / group_size;
    L.group_size = group_size;
    L.batch = 1;
    L.pair = pair ? 1 : 0;
    L.eps = 1e-5f;
    L.e.kind = pair ? Q4_EPI_SCATTER_ONLY : Q4_EPI_STORE;
    for (int i = 0; i < n_mats; i++) {
        if (out[i] <= 0 || out[i] % 8) return l2_fail(L2_ERR_ARG, "out[%d]=%d", i, out[i]);
        L.m[i].x = dummy;
        L.m[i].wn = norm ? dummy : nullptr;
        L.m[i].out = out[i];
    }
    return plan_of(L, kernel, cap, geometry);
}

extern "C" int l2_qlinear_plan(int in, int out, int group_size, int batch, int natural, char *kernel, size_t cap, int32_t *geometry) {
    if (!kernel || cap < 2 || !geometry || batch < 1 || batch > 4096) return l2_fail(L2_ERR_ARG, "bad argument");
    L2_TRY(check_qlinear_shape(in, out, group_size));
    static const float dummy[4] = {0.f, 0.f, 0.f, 0.f};
    static const int32_t order[4] = {0, 0, 0, 0};
    DevQLinear q;
    q.in = in, q.out = out, q.group_size = group_size, q.groups = in / group_size;
    Q4Launch L = launch_of(q, batch, 0.f);
    L.m[0] = mat_of(q, dummy, nullptr, nullptr);
    if (natural && !q4_gathers_in_kernel(L)) return l2_fail(L2_ERR_ARG, "in=%d: x is gathered in front", in);
    L.m[0].gidx = natural ? order : nullptr;
    return plan_of(L, kernel, cap, geometry);
}

extern "C" int l2_gemm_plan(int in, const int32_t *out, int n_mats, int group_size, int batch, int mode, int32_t *plan) {
    if (!out || !plan || n_mats < 1 || n_mats > 3 || batch < 1) return l2_fail(L2_ERR_ARG, "bad argument");
    if (mode != L2_PREFILL_FP32 && mode != L2_PREFILL_MFMA) return l2_fail(L2_ERR_ARG, "mode %d", mode);
    Q4Launch L{};
    L.n_mats = n_mats, L.in = in, L.batch = batch, L.group_size = group_size;
    if (group_size) L2_TRY(check_qlinear_shape(in, 8, group_size));
    else if (in < 32 || in % 32) return l2_fail(L2_ERR_ARG, "in=%d", in);
    L.groups = group_size ? in / group_size : 0;
    for (int i = 0; i < n_mats; i++) {
        if (out[i] <= 0 || out[i] % 8) return l2_fail(L2_ERR_ARG, "out[%d]=%d", i, out[i]);
        L.m[i].out = out[i];
    }
    if (mode == L2_PREFILL_MFMA && (!group_size || !q4_gemm_supports(in, 32, group_size))) return l2_fail(L2_ERR_ARG, "in=%d, groups of %d: not in fp16", in, group_size);
    const GemmTiles t = gemm_tiles(L, batch, mode == L2_PREFILL_MFMA ? 1 : 3, false);
    const int32_t all[8] = {t.rows, t.tokens, t.slices, t.blocks, t.whole, t.width, t.last, t.both};
    memcpy(plan, all, sizeof all);
    return L2_OK;
}

extern "C" int l2_model_token_trouble(l2_model *m, int missing, int looks, int fail_in) {
    if (!m || missing < 0 || looks < 1 || looks > kTokenLooks || fail_in < 0) return l2_fail(L2_ERR_ARG, "bad argument");
    if (!m->tok.model) return l2_fail(L2_ERR_ARG, "this model has no token kernel");
    if (missing >= m->tok.grid) return l2_fail(L2_ERR_ARG, "missing %d of %d blocks", missing, m->tok.grid);
    L2_HIP(hipStreamSynchronize(m->stream));
    L2_HIP(hipMemcpy((char *)m->tok.model + offsetof(TokModel, limit), &looks, sizeof looks, hipMemcpyHostToDevice));
    if (missing != m->tok.missing) {
        TokenPlan plan;
        bool ok = false;
        L2_TRY(token_plan(m->d, plan, &ok));
        plan.leave_out(missing);
        L2_HIP(hipMemcpy(m->tok.walks, plan.walks.data(), plan.walks.size() * sizeof(TokWalk), hipMemcpyHostToDevice));
    }
    m->tok.missing = missing, m->tok.fail_in = fail_in;
    return L2_OK;
}

extern "C" int l2_model_set_token_kernel(l2_model *m, int on, int missing, int looks) {
    if (!m || missing < 0 || looks < 1 || looks > kTokenLooks) return l2_fail(L2_ERR_ARG, "bad argument");
    if (!m->tok.model) return on ? l2_fail(L2_ERR_ARG, "this model has no token kernel") : L2_OK;
    L2_TRY(l2_model_token_trouble(m, missing, looks, 0));
    m->tok.on = on != 0, m->tok.gave_up = m->tok.in_a_row = 0;
    return L2_OK;
}

extern "C" int l2_model_token_kernel(const l2_model *m, int *on, int *gave_up) {
    if (!m || !on || !gave_up) return l2_fail(L2_ERR_ARG, "null argument");
    *on = m->tok.on, *gave_up = m->tok.gave_up;
    return L2_OK;
}

extern "C" int l2_model_token_steps(const l2_model *m, uint64_t *steps) {
    if (!m || !steps) return l2_fail(L2_ERR_ARG, "null argument");
    *steps = m->tok.steps;
    return L2_OK;
}

extern "C" int l2_model_asked(const l2_model *m, uint64_t *asked) {
    if (!m || !asked) return l2_fail(L2_ERR_ARG, "null argument");
    *asked = m->asked;
    return L2_OK;
}

extern "C" int l2_token_plan(const l2_dims *d, int32_t *walks, size_t cap, int32_t *info) {
    if (!d || !info) return l2_fail(L2_ERR_ARG, "null argument");
    L2_TRY(check_dims(d));
    TokenPlan t;
    bool ok = false;
    L2_TRY(token_plan(*d, t, &ok));
    info[0] = ok, info[1] = t.grid, info[2] = kTokenWaves, info[3] = (int32_t)t.lds;
    if (!ok || !walks) return L2_OK;
    const size_t n = t.walks.size() * (sizeof(TokWalk) / 4);
    if (cap < n) return l2_fail(L2_ERR_ARG, "room for %zu numbers, %zu needed", cap, n);
    memcpy(walks, t.walks.data(), n * 4);
    return L2_OK;
}

extern "C" int l2_token_rows(const l2_dims *d, int missing, int32_t *rows, size_t cap) {
    if (!d || !rows) return l2_fail(L2_ERR_ARG, "null argument");
    L2_TRY(check_dims(d));
    TokenPlan t;
    bool ok = false;
    L2_TRY(token_plan(*d, t, &ok));
    if (!ok || missing < 0 || missing >= t.grid) return l2_fail(L2_ERR_ARG, "missing %d of %d blocks", missing, ok ? t.grid : 0);
    if (cap < t.walks.size() * 4) return l2_fail(L2_ERR_ARG, "room for %zu numbers", cap);
    t.leave_out(missing);
    for (size_t i = 0; i < t.walks.size(); i++, rows += 4) {
        const TokWalk &k = t.walks[i];
        rows[0] = k.steps, rows[1] = k.r0, rows[2] = k.n, rows[3] = (t.part_at + (k.part_row + k.n) * t.phase[i / (t.walks.size() / 4)].nwk * 4) * 4;
    }
    return L2_OK;
}

extern "C" int l2_kernel_class_count(void) { return K_NCLASS; }

extern "C" const char *l2_kernel_class_name(int cls) { return cls >= 0 && cls < K_NCLASS ? kClassNames[cls] : ""; }

extern "C" int l2_decode_profile(l2_model *m, l2_state *s, int32_t token, int32_t pos, int n_tokens,
                                 float *ms_by_class, int32_t *launches_by_class) {
    if (!m || !s || !ms_by_class || !launches_by_class || n_tokens < 1) return l2_fail(L2_ERR_ARG, "bad argument");
    if (s->m != m) return l2_fail(L2_ERR_ARG, "state belongs to another model");
    if (pos < 0 || pos + n_tokens > m->max_seq) return l2_fail(L2_ERR_RANGE, "positions [%d,%d) exceed the cache", pos, pos + n_tokens);
    if (token < 0 || token >= m->d.vocab_size) return l2_fail(L2_ERR_RANGE, "token %d", token);
    const AtWork at_work(m);
    L2_TRY(ensure_batch(m, 1));
    L2_HIP(hipStreamSynchronize(m->stream));
    m->prof.clear();
    m->prof_on = true;
    int rc = steps_enqueue(m, s, token, pos, n_tokens, nullptr, 0);
    m->prof_on = false;
    hipError_t e = hipStreamSynchronize(m->stream);
    for (int c = 0; c < K_NCLASS; c++) {
        ms_by_class[c] = 0.f;
        launches_by_class[c] = 0;
    }
    for (auto &r : m->prof) {
        float ms = 0.f;
        if (rc == L2_OK && e == hipSuccess && r.e0 && r.e1 && hipEventElapsedTime(&ms, r.e0, r.e1) == hipSuccess) {
            ms_by_class[r.cls] += ms;
            launches_by_class[r.cls] += 1;
        }
        if (r.e0) (void)hipEventDestroy(r.e0);
        if (r.e1) (void)hipEventDestroy(r.e1);
    }
    m->prof.clear();
    if (rc != L2_OK) return rc;
    if (e != hipSuccess) return l2_fail(L2_ERR_HIP, "profile run: %s", hipGetErrorString(e));
    return L2_OK;
}

extern "C" int l2_copy_bench(size_t nbytes, int iters, float *ms_total) {
    if (!ms_total || nbytes < 16 || iters < 1) return l2_fail(L2_ERR_ARG, "bad argument");
    L2_TRY(require_device());
    char *a = nullptr, *b = nullptr;
    L2_TRY(dalloc(&a, nbytes));
    if (dalloc(&b, nbytes) != L2_OK) {
        dfree(a);
        return L2_ERR_HIP;
    }
    hipEvent_t e0, e1;
    (void)hipEventCreate(&e0);
    (void)hipEventCreate(&e1);
    (void)hipMemcpyAsync(b, a, nbytes, hipMemcpyDeviceToDevice, nullptr);
    (void)hipDeviceSynchronize();
    (void)hipEventRecord(e0, nullptr);
    for (int i = 0; i < iters; i++) (void)hipMemcpyAsync(b, a, nbytes, hipMemcpyDeviceToDevice, nullptr);
    (void)hipEventRecord(e1, nullptr);
    hipError_t e = hipEventSynchronize(e1);
    if (e == hipSuccess) e = hipEventElapsedTime(ms_total, e0, e1);
    (void)hipEventDestroy(e0);
    (void)hipEventDestroy(e1);
    dfree(a);
    dfree(b);
    if (e != hipSuccess) return l2_fail(L2_ERR_HIP, "copy bench: %s", hipGetErrorString(e));
    return L2_OK;
}
