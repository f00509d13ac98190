// C ABI for the individual kernels plus the HIP plumbing (memory, streams,
// events) a host without its own HIP bindings needs.  Every function checks
// its arguments, enqueues, and reports launch errors as VKH_ERR_HIP.
#include <dlfcn.h>
#include <math.h>
#include <stdio.h>
#include <string.h>

#include <algorithm>
#include <atomic>
#include <iterator>
#include <map>
#include <memory>
#include <mutex>
#include <tuple>
#include <vector>

#include "internal.hpp"

namespace vkh {

static thread_local char g_err[512] = "";

vkh_status fail(vkh_status st, const char *fmt, ...) {
    va_list ap;
    va_start(ap, fmt);
    vsnprintf(g_err, sizeof(g_err), fmt, ap);
    va_end(ap);
    return st;
}

vkh_status hip_fail(hipError_t e, const char *what) {
    if (e == hipErrorOutOfMemory || e == hipErrorMemoryAllocation)
        return fail(VKH_ERR_OUT_OF_MEMORY, "%s: %s", what, hipGetErrorString(e));
    return fail(VKH_ERR_HIP, "%s: %s", what, hipGetErrorString(e));
}

static std::atomic<uint64_t> g_allocations{0};
void note_allocation() { g_allocations.fetch_add(1, std::memory_order_relaxed); }

// RoPE tables for the standalone kernel entry points, cached per
// (device, seq_len, rotary_dim, theta) for the life of the process.
static vkh_status rope_table_cached(int seq_len, int rot, float theta, const float2 **out) {
    static std::mutex mu;
    static std::map<std::tuple<int, int, int, uint32_t>, float2 *> cache;
    int dev = 0;
    VKH_HIP(hipGetDevice(&dev));
    uint32_t tb;
    memcpy(&tb, &theta, 4);
    std::lock_guard<std::mutex> lk(mu);
    auto key = std::make_tuple(dev, seq_len, rot, tb);
    auto it = cache.find(key);
    if (it != cache.end()) { *out = it->second; return VKH_OK; }
    const int half = rot / 2;
    std::vector<float2> tab((size_t)seq_len * (half ? half : 1));
    if (half) rope_table_host(tab.data(), seq_len, rot, theta);
    float2 *d = nullptr;
    note_allocation();
    VKH_HIP(hipMalloc(&d, tab.size() * sizeof(float2)));
    VKH_HIP(hipMemcpy(d, tab.data(), tab.size() * sizeof(float2), hipMemcpyHostToDevice));
    cache[key] = d;
    *out = d;
    return VKH_OK;
}

// Scratch memory of the standalone entry points (gain partials, split-K
// partials, packed operands, parts of a split dK / dV): one buffer per (device,
// stream), grown on demand and reused, so a call does not allocate once its
// stream's buffer is large enough.  Calls on one stream are ordered by the stream;
// calls on different streams use different buffers, so no event is recorded or
// waited for per call (an event record costs a few microseconds of device time).
// Streams are told apart by hipStreamGetId, which is unique for the life of the
// process, so a stream created after another was destroyed never inherits its
// buffer.  The runtime that a process has loaded may be older than that function
// (torch brings its own), so it is looked up at run time; without it only the null
// stream, which is never destroyed, keeps a buffer.
//   * A buffer is replaced by one of at least twice its size (calls of varying
//     shapes settle) after its stream has drained; only calls on that stream wait.
//   * At most kMaxStreams buffers and kKeptTotal bytes are kept; room for another
//     stream is made by freeing the buffers that no call holds, after the device
//     has drained.
//   * What is not kept (calls of more than kLeaseMax, calls past kKeptTotal, streams
//     without an identity) is allocated in stream order and freed after the call.
constexpr size_t kLeaseMax = 256ull << 20, kKeptTotal = 1ull << 30;
class ScratchLease {
  public:
    ~ScratchLease() {
        if (own_) (void)hipFreeAsync(own_, st_);
    }
    vkh_status acquire(size_t bytes, hipStream_t st, void **out) {
        note_allocation();
        const vkh_status s = get(bytes, st, out);
        if (s != VKH_OK) (void)hipGetLastError();  // (an allocation's: the caller may do without)
        if (s != VKH_OK || own_) {
            lk_ = std::unique_lock<std::mutex>();
            buf_.reset();
        }
        return s;
    }

  private:
    struct Buf {
        std::mutex mu;  // held by a call until it has enqueued its work
        void *p = nullptr;
        size_t bytes = 0;
    };
    typedef std::pair<int, unsigned long long> Key;
    struct Kept {
        std::mutex mu;
        std::map<Key, std::shared_ptr<Buf>> per_stream;
        size_t total = 0;
    };
    static Kept &kept() {
        static Kept k;
        return k;
    }

    vkh_status get(size_t bytes, hipStream_t st, void **out) {
        static const auto stream_id =
            (hipError_t(*)(hipStream_t, unsigned long long *))dlsym(RTLD_DEFAULT, "hipStreamGetId");
        if (bytes > kLeaseMax || (!stream_id && st)) return in_order(bytes, st, out);
        Key key(0, 0);
        VKH_HIP(hipGetDevice(&key.first));
        if (stream_id) VKH_HIP(stream_id(st, &key.second));
        VKH_TRY(find(key));
        lk_ = std::unique_lock<std::mutex>(buf_->mu);
        if (buf_->bytes < bytes) {
            size_t nb = std::max({bytes, 2 * buf_->bytes, (size_t)1 << 20});
            nb = std::min(nb, kLeaseMax);
            if (!reserve(nb - buf_->bytes)) return in_order(bytes, st, out);
            hipError_t e = buf_->p ? hipStreamSynchronize(st) : hipSuccess;  // its earlier uses are done
            if (e == hipSuccess && buf_->p) e = hipFree(buf_->p);
            buf_->p = nullptr;
            note_allocation();
            if (e == hipSuccess) e = hipMalloc(&buf_->p, nb);
            if (e != hipSuccess) buf_->p = nullptr, give_back(nb);
            buf_->bytes = buf_->p ? nb : 0;
            if (e != hipSuccess) return hip_fail(e, "scratch");
        }
        *out = buf_->p;
        return VKH_OK;
    }

    vkh_status in_order(size_t bytes, hipStream_t st, void **out) {
        note_allocation();
        VKH_HIP(hipMallocAsync(&own_, bytes, st));
        st_ = st;
        *out = own_;
        return VKH_OK;
    }

    // buf_ = the stream's buffer (a new one is empty)
    vkh_status find(const Key &key) {
        constexpr size_t kMaxStreams = 64;
        std::vector<std::shared_ptr<Buf>> idle;
        {
            Kept &k = kept();
            std::lock_guard<std::mutex> lk(k.mu);
            auto it = k.per_stream.find(key);
            if (it == k.per_stream.end()) {
                if (k.per_stream.size() >= kMaxStreams)
                    for (auto i = k.per_stream.begin(); i != k.per_stream.end();) {
                        // no call holds it, and none can find it from here on
                        if (i->first.first == key.first && i->second.use_count() == 1) {
                            idle.push_back(i->second);
                            i = k.per_stream.erase(i);
                        } else {
                            ++i;
                        }
                    }
                it = k.per_stream.emplace(key, std::make_shared<Buf>()).first;
            }
            buf_ = it->second;
        }
        if (idle.empty()) return VKH_OK;
        const hipError_t e = hipDeviceSynchronize();
        for (auto &b : idle) {
            if (b->p) (void)hipFree(b->p);
            give_back(b->bytes);
        }
        VKH_HIP(e);
        return VKH_OK;
    }

    static bool reserve(size_t bytes) {
        Kept &k = kept();
        std::lock_guard<std::mutex> lk(k.mu);
        if (k.total + bytes > kKeptTotal) return false;
        k.total += bytes;
        return true;
    }
    static void give_back(size_t bytes) {
        Kept &k = kept();
        std::lock_guard<std::mutex> lk(k.mu);
        k.total -= bytes;
    }

    std::shared_ptr<Buf> buf_;
    std::unique_lock<std::mutex> lk_;  // (released before buf_ is)
    void *own_ = nullptr;              // of this call alone
    hipStream_t st_ = nullptr;
};

}  // namespace vkh

using namespace vkh;

#define CHECK_ARG(cond, msg)                                              \
    do {                                                                  \
        if (!(cond)) return fail(VKH_ERR_INVALID_ARGUMENT, "%s", msg);    \
    } while (0)

static inline hipStream_t S(vkh_stream s) { return (hipStream_t)s; }
static inline Precision PR(uint32_t p) { return p == VKH_PRECISION_BF16 ? Precision::BF16 : Precision::FP32; }

static AttnShape attn_shape(const vkh_attn_params *p) {
    AttnShape s;
    s.n_batch = p->n_batch ? (int)p->n_batch : 1;
    s.n_q = p->n_q; s.n_kv = p->n_kv; s.n_heads = p->n_heads; s.n_kv_heads = p->n_kv_heads;
    s.head_dim = p->head_dim; s.causal = p->causal ? 1 : 0; s.inv_sqrt_dim = p->inv_sqrt_dim;
    s.ragged = 1;
    return s;
}

static vkh_status check_attn(const vkh_attn_params *p) {
    CHECK_ARG(p, "null params");
    CHECK_ARG(p->n_heads && p->n_kv_heads && p->head_dim && p->n_q && p->n_kv, "zero attention dimension");
    CHECK_ARG(p->n_heads % p->n_kv_heads == 0, "n_heads % n_kv_heads != 0");
    CHECK_ARG(!p->causal || p->n_q <= p->n_kv, "causal attention needs n_q <= n_kv");
    CHECK_ARG(p->dtype <= VKH_BF16, "dtype");
    if (p->dtype == VKH_BF16 && p->head_dim != 64 && p->head_dim != 128)
        return fail(VKH_ERR_UNSUPPORTED, "bf16 attention supports head_dim 64 and 128");
    if (p->head_dim > 256) return fail(VKH_ERR_UNSUPPORTED, "head_dim > 256");
    return VKH_OK;
}

extern "C" {

const char *vkh_last_error(void) { return g_err; }

const char *vkh_build_info(void) { return "vkhip for gfx950 (MI355X), built with hipcc " __VERSION__; }

const char *vkh_status_name(vkh_status s) {
    switch (s) {
    case VKH_OK: return "Ok";
    case VKH_ERR_INVALID_ARGUMENT: return "InvalidArgument";
    case VKH_ERR_HIP: return "HipError";
    case VKH_ERR_OUT_OF_MEMORY: return "OutOfMemory";
    case VKH_ERR_UNSUPPORTED: return "Unsupported";
    case VKH_ERR_NO_DEVICE: return "NoDevice";
    case VKH_ERR_TOKEN_IDS_LEN: return "TokenIdsLen";
    case VKH_ERR_TARGET_LEN: return "TargetLen";
    case VKH_ERR_OUT_LOGITS_LEN: return "OutLogitsLen";
    case VKH_ERR_TOKEN_OUT_OF_RANGE: return "TokenOutOfRange";
    case VKH_ERR_EMBED_SHAPE: return "EmbedShape";
    case VKH_ERR_FINAL_NORM_SHAPE: return "FinalNormShape";
    case VKH_ERR_LM_HEAD_SHAPE: return "LmHeadShape";
    case VKH_ERR_LAYER_COUNT: return "LayerCount";
    case VKH_ERR_LAYER_N1_SHAPE: return "LayerN1Shape";
    case VKH_ERR_LAYER_Q_SHAPE: return "LayerQShape";
    case VKH_ERR_LAYER_K_SHAPE: return "LayerKShape";
    case VKH_ERR_LAYER_V_SHAPE: return "LayerVShape";
    case VKH_ERR_LAYER_O_SHAPE: return "LayerOShape";
    case VKH_ERR_LAYER_N2_SHAPE: return "LayerN2Shape";
    case VKH_ERR_LAYER_GATE_SHAPE: return "LayerGateShape";
    case VKH_ERR_LAYER_UP_SHAPE: return "LayerUpShape";
    case VKH_ERR_LAYER_DOWN_SHAPE: return "LayerDownShape";
    case VKH_ERR_LAYER_Q_NORM_SHAPE: return "LayerQNormShape";
    case VKH_ERR_LAYER_K_NORM_SHAPE: return "LayerKNormShape";
    case VKH_ERR_LORA_RANK_ZERO: return "LoraRankZero";
    case VKH_ERR_LORA_INIT_LEN: return "LoraInitLen";
    case VKH_ERR_INVALID_CHECKPOINT_MAGIC: return "InvalidCheckpointMagic";
    case VKH_ERR_UNSUPPORTED_CHECKPOINT_VERSION: return "UnsupportedCheckpointVersion";
    case VKH_ERR_CHECKPOINT_CONFIG_SIZE_MISMATCH: return "CheckpointConfigSizeMismatch";
    case VKH_ERR_CHECKPOINT_CONFIG_MISMATCH: return "CheckpointConfigMismatch";
    case VKH_ERR_END_OF_STREAM: return "EndOfStream";
    case VKH_ERR_INVALID_LORA_CHECKPOINT_MAGIC: return "InvalidLoraCheckpointMagic";
    case VKH_ERR_UNSUPPORTED_LORA_CHECKPOINT_VERSION: return "UnsupportedLoraCheckpointVersion";
    case VKH_ERR_LORA_CHECKPOINT_CONFIG_SIZE_MISMATCH: return "LoraCheckpointConfigSizeMismatch";
    case VKH_ERR_LORA_CHECKPOINT_CONFIG_MISMATCH: return "LoraCheckpointConfigMismatch";
    case VKH_ERR_LORA_CHECKPOINT_EMPTY: return "LoraCheckpointEmpty";
    case VKH_ERR_IO: return "IoError";
    case VKH_ERR_INPUT_IDS_LEN: return "InputIdsLen";
    case VKH_ERR_TARGET_IDS_LEN: return "TargetIdsLen";
    case VKH_ERR_BATCH_INDEX_OUT_OF_RANGE: return "BatchIndexOutOfRange";
    case VKH_ERR_EMPTY_DATASET: return "EmptyDataset";
    case VKH_ERR_DATASET_TOO_SHORT: return "DatasetTooShort";
    case VKH_ERR_BATCH_IDX_OUT_OF_RANGE: return "BatchIdxOutOfRange";
    case VKH_ERR_HIDDEN_DIM_EXCEEDS_MAX: return "HiddenDimExceedsMax";
    case VKH_ERR_X_DIM_MISMATCH: return "XDimMismatch";
    case VKH_ERR_TARGET_DIM_MISMATCH: return "TargetDimMismatch";
    case VKH_ERR_OUT_DIM_MISMATCH: return "OutDimMismatch";
    case VKH_ERR_BATCH_SIZE_NOT_CONFIGURED: return "BatchSizeNotConfigured";
    case VKH_ERR_BATCH_SIZE_EXCEEDS_MAX: return "BatchSizeExceedsMax";
    case VKH_ERR_X_BATCH_DIM_MISMATCH: return "XBatchDimMismatch";
    case VKH_ERR_TARGET_BATCH_DIM_MISMATCH: return "TargetBatchDimMismatch";
    case VKH_ERR_OUT_BATCH_DIM_MISMATCH: return "OutBatchDimMismatch";
    case VKH_ERR_OUTPUT_TOO_LARGE: return "OutputTooLarge";
    }
    return "Unknown";
}

// ── attention ──────────────────────────────────────────────────────────

vkh_status vkh_fa_forward(const vkh_attn_params *p, const void *q, const void *k, const void *v,
                          float *o, float *lse, vkh_stream stream) {
    VKH_TRY(check_attn(p));
    CHECK_ARG(q && k && v && o, "null pointer");
    const AttnShape s = attn_shape(p);
    const long ldq = (long)p->n_heads * p->head_dim, ldk = (long)p->n_kv_heads * p->head_dim;
    VKH_HIP(fa_forward(s, q, ldq, k, ldk, v, ldk, o, ldq, lse,
                       p->dtype == VKH_BF16 ? DType::BF16 : DType::F32, nullptr, 0, S(stream)));
    return VKH_OK;
}

vkh_status vkh_fa_bw_d(const vkh_attn_params *p, const float *o, const float *dout, float *d,
                       void *dout_bf16, vkh_stream stream) {
    VKH_TRY(check_attn(p));
    CHECK_ARG(o && dout && d, "null pointer");
    const AttnShape s = attn_shape(p);
    const long ld = (long)p->n_heads * p->head_dim;
    VKH_HIP(fa_bw_d(s, o, ld, dout, ld, d, p->dtype == VKH_BF16 ? (bf16 *)dout_bf16 : nullptr, ld,
                    S(stream)));
    return VKH_OK;
}

vkh_status vkh_fa_bw_d_bf16(const vkh_attn_params *p, const void *o_bf16, const void *dout_bf16,
                            float *d, vkh_stream stream) {
    VKH_TRY(check_attn(p));
    CHECK_ARG(o_bf16 && dout_bf16 && d, "null pointer");
    if (p->head_dim != 64 && p->head_dim != 128)
        return fail(VKH_ERR_UNSUPPORTED, "bf16 D preprocess needs head_dim 64 or 128");
    const AttnShape s = attn_shape(p);
    const long ld = (long)p->n_heads * p->head_dim;
    VKH_HIP(fa_bw_d_bf16(s, (const bf16 *)o_bf16, ld, (const bf16 *)dout_bf16, ld, d, S(stream)));
    return VKH_OK;
}

static AttnPtrs attn_ptrs(const vkh_attn_params *p, const void *q, const void *k, const void *v,
                          const void *dout, const float *lse, const float *d) {
    AttnPtrs a{};
    const long ldq = (long)p->n_heads * p->head_dim, ldk = (long)p->n_kv_heads * p->head_dim;
    a.q = q; a.ldq = ldq; a.k = k; a.ldk = ldk; a.v = v; a.ldv = ldk;
    a.dout = dout; a.lddo = ldq; a.lse = lse; a.d = (float *)d;
    a.lddq = ldq; a.lddk = ldk; a.lddv = ldk;
    a.dt = p->dtype == VKH_BF16 ? DType::BF16 : DType::F32;
    return a;
}

vkh_status vkh_fa_bw_dq(const vkh_attn_params *p, const void *q, const void *k, const void *v,
                        const void *dout, const float *lse, const float *d, float *dq,
                        vkh_stream stream) {
    VKH_TRY(check_attn(p));
    CHECK_ARG(q && k && v && dout && lse && d && dq, "null pointer");
    AttnPtrs a = attn_ptrs(p, q, k, v, dout, lse, d);
    a.dq = dq;
    VKH_HIP(fa_bw_dq(attn_shape(p), a, S(stream)));
    return VKH_OK;
}

// Scratch of a split dK / dV launch, where the grid asks for one (not under capture, nor
// where there is no memory for it).
static bool capturing(hipStream_t st);
static vkh_status attn_parts(const AttnShape &s, AttnPtrs &a, ScratchLease &lease, hipStream_t st) {
    const int parts = fa_bw_parts(s, a.dt);
    const size_t b = fa_bw_parts_ws_bytes(s, parts);
    if (!b || b > kLeaseMax || capturing(st)) return VKH_OK;
    void *w = nullptr;
    const vkh_status got = lease.acquire(b, st, &w);
    if (got == VKH_ERR_OUT_OF_MEMORY) return VKH_OK;
    VKH_TRY(got);
    a.split_ws = (float *)w;
    a.split_parts = parts;
    return VKH_OK;
}
// bf16 shapes that the recompute kernels' general form takes: all that the fused form's
// own recompute kernels do not, and those whose dK / dV grid is split.  (4 x 2048
// tokens, 16 / 8 heads of 64: 289 us on the dS workspace and dQ GEMM, 174 here.)
static bool attn_general(const AttnShape &s, const AttnPtrs &a) {
    return a.dt == DType::BF16 && (a.split_ws || !fa_bw_v4_ok(s)) && fa_bw_ragged_ok(s, a);
}

vkh_status vkh_fa_bw_dkv(const vkh_attn_params *p, const void *q, const void *k, const void *v,
                         const void *dout, const float *lse, const float *d, float *dk,
                         float *dv, vkh_stream stream) {
    VKH_TRY(check_attn(p));
    CHECK_ARG(q && k && v && dout && lse && d && dk && dv, "null pointer");
    AttnPtrs a = attn_ptrs(p, q, k, v, dout, lse, d);
    a.dk = dk;
    a.dv = dv;
    const AttnShape s = attn_shape(p);
    ScratchLease lease;
    VKH_TRY(attn_parts(s, a, lease, S(stream)));
    VKH_HIP(fa_bw_dkv(s, a, S(stream)));
    return VKH_OK;
}

size_t vkh_fa_backward_workspace_bytes(const vkh_attn_params *p) {
    if (!p || check_attn(p) != VKH_OK) return 0;
    const AttnShape s = attn_shape(p);
    // aligned operands of this shape (others allocate for their call)
    const float *al = (const float *)256;
    AttnPtrs a = attn_ptrs(p, al, al, al, al, al, al);
    a.dq = a.dk = a.dv = (float *)al;
    if (p->dtype != VKH_BF16 || !fa_bw_fused_ok(s) || attn_general(s, a)) return 0;
    return fa_bw_ws_bytes(s, fa_bw_v4_ok(s));
}

vkh_status vkh_fa_backward(const vkh_attn_params *p, const void *q, const void *k, const void *v,
                           const void *dout, const float *lse, const float *d, float *dq,
                           float *dk, float *dv, void *workspace, vkh_stream stream) {
    VKH_TRY(check_attn(p));
    CHECK_ARG(q && k && v && dout && lse && d && dq && dk && dv, "null pointer");
    AttnPtrs a = attn_ptrs(p, q, k, v, dout, lse, d);
    a.dq = dq;
    a.dk = dk;
    a.dv = dv;
    const AttnShape s = attn_shape(p);
    hipStream_t st = S(stream);
    ScratchLease lease;
    VKH_TRY(attn_parts(s, a, lease, st));
    if (p->dtype != VKH_BF16 || !fa_bw_fused_ok(s) || attn_general(s, a)) {
        VKH_HIP(fa_bw_dkv(s, a, st));
        VKH_HIP(fa_bw_dq(s, a, st));
        return VKH_OK;
    }
    // the fused form's own recompute kernels, or dS in a workspace (the caller's holds it
    // only where vkh_fa_backward_workspace_bytes says so)
    const bool v4 = fa_bw_v4_ok(s);
    const size_t wsb = fa_bw_ws_bytes(s, v4);
    const bool own = wsb && (!workspace || vkh_fa_backward_workspace_bytes(p) < wsb);
    void *ws = workspace;
    a.split_ws = nullptr;
    if (own) {
        note_allocation();
        VKH_HIP(hipMallocAsync(&ws, wsb, st));
    }
    const hipError_t e = fa_bw_fused(s, a, (bf16 *)ws, v4, st);
    if (own) (void)hipFreeAsync(ws, st);
    if (e != hipSuccess) return hip_fail(e, "fa_backward");
    return VKH_OK;
}

// The whole attention backward from bf16 O: the D preprocess and the two
// gradient kernels.  On the recompute path the dQ kernel forms D itself (no
// separate pass) and the dK/dV kernel reads it; other shapes run the D kernel
// and then vkh_fa_backward.
vkh_status vkh_fa_backward_from_o(const vkh_attn_params *p, const void *q, const void *k,
                                  const void *v, const void *o_bf16, const void *dout_bf16,
                                  const float *lse, float *d, float *dq, float *dk, float *dv,
                                  void *workspace, vkh_stream stream) {
    VKH_TRY(check_attn(p));
    CHECK_ARG(q && k && v && o_bf16 && dout_bf16 && lse && d && dq && dk && dv, "null pointer");
    if (p->dtype != VKH_BF16) return fail(VKH_ERR_INVALID_ARGUMENT, "fa_backward_from_o takes bf16 operands");
    const AttnShape s = attn_shape(p);
    AttnPtrs a = attn_ptrs(p, q, k, v, dout_bf16, lse, d);
    a.dq = dq;
    a.dk = dk;
    a.dv = dv;
    a.o16 = o_bf16;
    a.ldo16 = (long)p->n_heads * p->head_dim;
    {
        ScratchLease lease;
        VKH_TRY(attn_parts(s, a, lease, S(stream)));
        if (attn_general(s, a) && fa_bw_ragged(s, a, S(stream))) {
            VKH_HIP(hipGetLastError());
            return VKH_OK;
        }
    }
    a.split_ws = nullptr;
    if (fa_bw_fused_ok(s) && fa_bw_v4_ok(s)) {
        const hipError_t e = fa_bw_fused(s, a, nullptr, true, S(stream));
        if (e != hipSuccess) return hip_fail(e, "fa_backward_from_o");
        return VKH_OK;
    }
    VKH_TRY(vkh_fa_bw_d_bf16(p, o_bf16, dout_bf16, d, stream));
    return vkh_fa_backward(p, q, k, v, dout_bf16, lse, d, dq, dk, dv, workspace, stream);
}

// ── GEMMs ──────────────────────────────────────────────────────────────

static bool capturing(hipStream_t st) {
    hipStreamCaptureStatus cs = hipStreamCaptureStatusNone;
    if (hipStreamIsCapturing(st, &cs) != hipSuccess) {
        (void)hipGetLastError();
        return true;
    }
    return cs != hipStreamCaptureStatusNone;
}

// One contraction of a linear layer.  Operands that need a packed copy (fp32
// operands in the bf16 precision; rows that are not whole 16-byte chunks) go
// through the workspace to the DMA-staged kernels; while the stream is being
// captured, or where there is no memory for the workspace, they take the generic
// kernel, and the others a plan without a split: a graph outlives the call, so it
// holds no pointer into the stream's scratch (which a later call may replace).
// Against the generic kernel, forward / dx / dW: 2048 tokens, 2560 x 2560, fp32
// operands in bf16 products 55 / 55 / 63 us (645 / 443 / 351); bf16 operands of
// 2000 x 4100 x 4099 156 / 143 / 117 us (455 / 638 / 533); fp32 of 1000 x 1500 x 3001
// 131 / 130 / 117 us (205 / 156 / 211); 16 tokens, 1024 x 1024 mixed 15 / 15 / 8 us
// (41 / 29 / 7).
//
// Products of so few terms that the packing launch is most of the call stay on the
// generic kernel: sums of up to 64 terms onto 1.25 M outputs, of 32 onto 2.5 M, and of
// 128 where its 128 x 128 tiles fill the chip (mixed dW of 16 to 64 tokens, 1000 x 1000:
// 6.7 us against 8.1; 16 x 30000 over 96: 7.9 to 9.5 against 10.7 to 11.8).  Beyond,
// the packed form is: 2048 x 1024 over 64 8.8 against 11.3, 2048 x 4096 over 64 the same
// way; over 472 timed products of 1 to 300 terms this line is 1 % above the better form.
static bool few_terms(LinOp op, uint32_t M, uint32_t N, uint32_t K) {
    const uint32_t rows = op == LinOp::TN ? N : M, cols = op == LinOp::NT ? N : K,
                   terms = op == LinOp::NT ? K : op == LinOp::NN ? N : M;
    const double out = (double)rows * cols;
    return (terms <= 64 && out <= 1.25e6) || (terms <= 32 && out <= 2.5e6) ||
           (terms <= 128 && out <= 2.5e6 && (uint64_t)ceil_div(rows, 128) * ceil_div(cols, 128) >= 192);
}

static vkh_status linear(LinOp op, LinForm f, const void *a, const void *b, float *out, uint32_t M,
                         uint32_t N, uint32_t K, const char *what, hipStream_t st) {
    ScratchLease lease;
    GemmWs ws{nullptr, 0};
    const bool any = M && N && K, packs = any && lin_packs(op, f, a, b, M, N, K);
    const bool generic = !any || (packs && few_terms(op, M, N, K));
    if (!generic && !capturing(st)) {
        ws.bytes = lin_ws_bytes(op, f, a, b, M, N, K);
        const vkh_status got = ws.bytes ? lease.acquire(ws.bytes, st, &ws.p) : VKH_OK;
        if (got == VKH_ERR_OUT_OF_MEMORY) ws = GemmWs{nullptr, 0};
        else VKH_TRY(got);
    }
    if (generic || (packs && !ws.p)) {
        const Precision pr = f == LinForm::F32 ? Precision::FP32 : Precision::BF16;
        const DType dt = f == LinForm::BF16 ? DType::BF16 : DType::F32;
        const Mat ma{a, (long)(op == LinOp::NT ? K : N), dt}, mb{b, (long)K, dt};
        if (op == LinOp::NT) VKH_HIP(gemm_nt(pr, ma, mb, out, N, M, N, K, nullptr, 0, 1.f, 0.f, st));
        else if (op == LinOp::NN) VKH_HIP(gemm_nn(pr, ma, mb, out, K, M, N, K, 1.f, 0.f, st));
        else VKH_HIP(gemm_tn(pr, ma, mb, out, K, M, N, K, 1.f, 0.f, st));
        return VKH_OK;
    }
    const hipError_t e = lin_run(op, f, a, b, out, M, N, K, ws, st);
    if (e != hipSuccess) return hip_fail(e, what);
    return VKH_OK;
}
static inline LinForm form_of(uint32_t precision) {
    return PR(precision) == Precision::FP32 ? LinForm::F32 : LinForm::MIXED;
}

vkh_status vkh_matmul_nt(const float *x, const float *w, float *y, uint32_t M, uint32_t N,
                         uint32_t K, uint32_t precision, vkh_stream stream) {
    CHECK_ARG(x && w && y, "null pointer");
    return linear(LinOp::NT, form_of(precision), x, w, y, M, N, K, "matmul_nt", S(stream));
}

vkh_status vkh_linear_backward_dx(const float *dy, const float *w, float *dx, uint32_t M,
                                  uint32_t N, uint32_t K, uint32_t precision, vkh_stream stream) {
    CHECK_ARG(dy && w && dx, "null pointer");
    return linear(LinOp::NN, form_of(precision), dy, w, dx, M, N, K, "linear_backward_dx", S(stream));
}

vkh_status vkh_linear_backward_dw(const float *dy, const float *x, float *dw, uint32_t M,
                                  uint32_t N, uint32_t K, uint32_t precision, vkh_stream stream) {
    CHECK_ARG(dy && x && dw, "null pointer");
    return linear(LinOp::TN, form_of(precision), dy, x, dw, M, N, K, "linear_backward_dw", S(stream));
}

vkh_status vkh_matmul_nt_bf16(const void *x, const void *w, float *y, uint32_t M, uint32_t N,
                              uint32_t K, vkh_stream stream) {
    CHECK_ARG(x && w && y, "null pointer");
    return linear(LinOp::NT, LinForm::BF16, x, w, y, M, N, K, "matmul_nt_bf16", S(stream));
}

vkh_status vkh_gate_up_swiglu_bf16(const void *x, const void *w_gu, float *gu, void *gated,
                                   uint32_t M, uint32_t F, uint32_t K, vkh_stream stream) {
    CHECK_ARG(x && w_gu && gu && gated, "null pointer");
    CHECK_ARG(2ull * F < (1ull << 31), "F too large");
    hipStream_t st = S(stream);
    const hipError_t e = g16_gate_up_swiglu((const bf16 *)x, K, (const bf16 *)w_gu, K, gu, 2L * F,
                                            (bf16 *)gated, F, (int)M, (int)F, (int)K, st);
    if (e != hipErrorNotSupported) {
        VKH_HIP(e);
        return VKH_OK;
    }
    // the two-pass form: the [M, 2F] product, then the SwiGLU over its halves
    const vkh_status r = vkh_matmul_nt_bf16(x, w_gu, gu, M, 2 * F, K, stream);
    if (r != VKH_OK) return r;
    VKH_HIP(swiglu_forward(gu, 2L * F, gu + F, 2L * F, gated, F, DType::BF16, (int)M, (int)F, st));
    return VKH_OK;
}

vkh_status vkh_gate_up_swiglu(const float *x, const float *w_gu, float *gu, float *gated,
                              uint32_t M, uint32_t F, uint32_t K, int fused, vkh_stream stream) {
    CHECK_ARG(x && w_gu && gu && gated, "null pointer");
    CHECK_ARG(2ull * F < (1ull << 31), "F too large");
    hipStream_t st = S(stream);
    if (fused) {
        const hipError_t e = g32_gate_up_swiglu(x, K, w_gu, K, gu, 2L * F, gated, F, (int)M, (int)F,
                                                (int)K, st);
        if (e != hipErrorNotSupported) {
            VKH_HIP(e);
            return VKH_OK;
        }
    }
    const vkh_status r = vkh_matmul_nt(x, w_gu, gu, M, 2 * F, K, VKH_PRECISION_FP32, stream);
    if (r != VKH_OK) return r;
    VKH_HIP(swiglu_forward(gu, 2L * F, gu + F, 2L * F, gated, F, DType::F32, (int)M, (int)F, st));
    return VKH_OK;
}

vkh_status vkh_linear_backward_dx_bf16(const void *dy, const void *w, float *dx, uint32_t M,
                                       uint32_t N, uint32_t K, vkh_stream stream) {
    CHECK_ARG(dy && w && dx, "null pointer");
    return linear(LinOp::NN, LinForm::BF16, dy, w, dx, M, N, K, "linear_backward_dx_bf16", S(stream));
}

vkh_status vkh_linear_backward_dw_bf16(const void *dy, const void *x, float *dw, uint32_t M,
                                       uint32_t N, uint32_t K, vkh_stream stream) {
    CHECK_ARG(dy && x && dw, "null pointer");
    return linear(LinOp::TN, LinForm::BF16, dy, x, dw, M, N, K, "linear_backward_dw_bf16", S(stream));
}

// The rank-r products go through the fp32 GEMMs (their few-tile plans split the long
// sum; one block per column group walked it alone before, dA and dB 21 us each at 2048
// tokens and 2560 columns), and the rank-r update rides in the base product's epilogue
// instead of reading the output back (16 and 14 us): that layer, forward and backward
// at rank 16, 213 -> 157 us.  A captured stream (no scratch), no memory for the scratch and
// operands of 2 GiB keep the row and update kernels, with fp32 factors and products as well.  x A^T and dy B
// sum in at least the row kernel's eight partial sums.
constexpr int kLoraChains = 8;
vkh_status vkh_lora_forward(const float *x, const float *w, const float *a, const float *b,
                            float *y, float *inter, uint32_t M, uint32_t N, uint32_t K,
                            uint32_t r, float aor, uint32_t precision, vkh_stream stream) {
    CHECK_ARG(x && w && a && b && y && inter, "null pointer");
    CHECK_ARG(r > 0, "rank 0");
    const Precision pr = PR(precision);
    const LinForm form = form_of(precision);
    hipStream_t st = S(stream);
    LoraSegs sa, sb;
    sa.n = sb.n = 1;
    sa.s[0] = LoraSeg{0, (int)K, a, 1, (long)K, inter, (long)r};
    sb.s[0] = LoraSeg{0, (int)N, b, (long)r, 1, inter, (long)r};
    // fp32 factors and products where the shape allows
    if (lora_fast_ok(DType::F32, x, K, (int)r, sa) && lora_update_ok(y, N, (int)r, sb) && M) {
        const size_t wsb = std::max(lin_ws_bytes(LinOp::NT, form, x, w, M, N, K), g32_ws_bytes_for(M, r, K, kLoraChains));
        ScratchLease lease;
        void *sc = nullptr;
        bool tiled = !capturing(st) && lin_lora_ok(LinOp::NT, form, M, N, K, sb, (int)r);
        if (tiled && wsb) {
            const vkh_status got = lease.acquire(wsb, st, &sc);
            if (got == VKH_ERR_OUT_OF_MEMORY) tiled = false;
            else VKH_TRY(got);
        }
        if (!tiled) {
            VKH_TRY(linear(LinOp::NT, form, x, w, y, M, N, K, "lora_forward", st));
            VKH_HIP(lora_rows(DType::F32, x, K, (int)M, (int)r, sa, 1.f, st));
            VKH_HIP(lora_update(y, N, (int)M, (int)r, sb, aor, st));
            return VKH_OK;
        }
        const GemmWs ws{sc, wsb}, rows{sc, wsb, false, kLoraChains};
        VKH_HIP(g32_nt(x, K, a, K, inter, r, M, r, K, nullptr, 0, 1.f, 0.f, rows, st));
        VKH_HIP(lin_run(LinOp::NT, form, x, w, y, M, N, K, ws, st, &sb, (int)r, aor));
        return VKH_OK;
    }
    VKH_TRY(linear(LinOp::NT, form, x, w, y, M, N, K, "lora_forward", st));
    VKH_HIP(gemm_nt(pr, matf(x, K), matf(a, K), inter, r, M, r, K, nullptr, 0, 1.f, 0.f, st));
    VKH_HIP(gemm_nt(pr, matf(inter, r), matf(b, r), y, N, M, N, r, nullptr, 0, aor, 1.f, st));
    return VKH_OK;
}

vkh_status vkh_lora_backward(const float *dy, const float *x, const float *w, const float *a,
                             const float *b, const float *inter, float *dx, float *dA,
                             float *dB, uint32_t M, uint32_t N, uint32_t K, uint32_t r,
                             float aor, uint32_t precision, vkh_stream stream) {
    CHECK_ARG(dy && x && w && a && b && inter && dA && dB, "null pointer");
    CHECK_ARG(r > 0, "rank 0");
    const Precision pr = PR(precision);
    const LinForm form = form_of(precision);
    hipStream_t st = S(stream);
    LoraSegs sb, sa, sdA, sdB;
    sb.n = sa.n = sdA.n = sdB.n = 1;
    sb.s[0] = LoraSeg{0, (int)N, b, (long)r, 1, (float *)inter, (long)r};
    sa.s[0] = LoraSeg{0, (int)K, a, 1, (long)K, (float *)inter, (long)r};  // (u: dyB, set below)
    sdA.s[0] = LoraSeg{0, (int)K, nullptr, 1, 1, (float *)inter, (long)r, dA, 1, (long)K};
    sdB.s[0] = LoraSeg{0, (int)N, nullptr, 1, 1, (float *)inter, (long)r, dB, (long)r, 1};
    const size_t dyb_bytes = ((size_t)M * r * 4 + 511) / 256 * 256;
    const bool fast = lora_fast_ok(DType::F32, dy, N, (int)r, sb) && lora_fast_ok(DType::F32, x, K, (int)r, sdA) &&
                      lora_fast_ok(DType::F32, dy, N, (int)r, sdB) && M &&
                      (!dx || lora_update_ok(dx, K, (int)r, sa));
    bool tiled = fast && !capturing(st) && (!dx || lin_lora_ok(LinOp::NN, form, M, N, K, sa, (int)r));
    ScratchLease lease;
    void *sc = nullptr;
    size_t wsb = 0;
    if (tiled) {
        wsb = std::max({g32_ws_bytes_for(M, r, N, kLoraChains), g32_ws_bytes_for(r, K, M), g32_ws_bytes_for(N, r, M)});
        if (dx) wsb = std::max(wsb, lin_ws_bytes(LinOp::NN, form, dy, w, M, N, K));
        const vkh_status got = lease.acquire(dyb_bytes + wsb, st, &sc);
        if (got == VKH_ERR_OUT_OF_MEMORY) tiled = false;
        else VKH_TRY(got);
    }
    if (tiled) {  // fp32 factors and products
        float *dyB = (float *)sc;
        const GemmWs ws{wsb ? (char *)sc + dyb_bytes : nullptr, wsb}, rows{ws.p, wsb, false, kLoraChains};
        sa.s[0].u = dyB;
        VKH_HIP(g32_nn(dy, N, b, r, dyB, r, M, N, r, 1.f, 0.f, rows, st));
        if (dx) VKH_HIP(lin_run(LinOp::NN, form, dy, w, dx, M, N, K, ws, st, &sa, (int)r, aor));
        VKH_HIP(g32_tn(dyB, r, x, K, dA, K, M, r, K, aor, 0.f, ws, st));
        VKH_HIP(g32_tn(dy, N, inter, r, dB, r, M, N, r, aor, 0.f, ws, st));
        return VKH_OK;
    }
    float *dyB = nullptr;
    note_allocation();
    VKH_HIP(hipMallocAsync((void **)&dyB, dyb_bytes, st));
    vkh_status base = VKH_OK;  // of the base product
    hipError_t e;
    if (fast) {
        for (LoraSegs *g : {&sb, &sa, &sdA}) g->s[0].u = dyB;
        e = lora_rows(DType::F32, dy, N, (int)M, (int)r, sb, 1.f, st);
        if (e == hipSuccess && dx) base = linear(LinOp::NN, form, dy, w, dx, M, N, K, "lora_backward", st);
        if (e == hipSuccess && base == VKH_OK && dx) e = lora_update(dx, K, (int)M, (int)r, sa, aor, st);
        if (e == hipSuccess) e = lora_cols(DType::F32, x, K, (int)M, (int)r, sdA, aor, st);
        if (e == hipSuccess) e = lora_cols(DType::F32, dy, N, (int)M, (int)r, sdB, aor, st);
    } else {
        e = gemm_nn(pr, matf(dy, N), matf(b, r), dyB, r, M, N, r, 1.f, 0.f, st);
        if (e == hipSuccess && dx) base = linear(LinOp::NN, form, dy, w, dx, M, N, K, "lora_backward", st);
        if (e == hipSuccess && base == VKH_OK && dx) e = gemm_nn(pr, matf(dyB, r), matf(a, K), dx, K, M, r, K, aor, 1.f, st);
        if (e == hipSuccess) e = gemm_tn(pr, matf(dyB, r), matf(x, K), dA, K, M, r, K, aor, 0.f, st);
        if (e == hipSuccess) e = gemm_tn(pr, matf(dy, N), matf(inter, r), dB, r, M, N, r, aor, 0.f, st);
    }
    (void)hipFreeAsync(dyB, st);
    if (base != VKH_OK) return base;
    if (e != hipSuccess) return hip_fail(e, "lora_backward");
    return VKH_OK;
}

// The training step's grouped LoRA launches on bf16 activations: the segment
// lists come from lora_group_segs, as in the runner.
static vkh_status lora_group_args(const vkh_lora_adapter *ad, uint32_t na, uint32_t r,
                                  LoraAdapter (&out)[3]) {
    CHECK_ARG(ad && na >= 1 && na <= 3, "1 to 3 adapters");
    CHECK_ARG(r > 0, "rank 0");
    for (uint32_t i = 0; i < na; ++i) {
        const vkh_lora_adapter &a = ad[i];
        CHECK_ARG(a.a && a.b && a.inter && a.n && a.k, "adapter: null factor or buffer");
        out[i] = LoraAdapter{(long)a.col, (int)a.n, (int)a.k, a.a, a.b, a.inter, a.dyb, a.da, a.db};
    }
    return VKH_OK;
}

vkh_status vkh_lora_group_forward_bf16(const uint16_t *x, uint32_t ldx, uint32_t T, uint32_t r,
                                       float aor, const vkh_lora_adapter *adapters,
                                       uint32_t n_adapters, float *y, uint32_t ldy,
                                       vkh_stream stream) {
    CHECK_ARG(x && y, "null pointer");
    LoraAdapter ad[3];
    VKH_TRY(lora_group_args(adapters, n_adapters, r, ad));
    for (uint32_t i = 0; i < n_adapters; ++i)
        CHECK_ARG(ad[i].k <= (long)ldx && ad[i].col + ad[i].n <= (long)ldy, "adapter outside the rows");
    const LoraGroupSegs g = lora_group_segs(ad, (int)n_adapters, (int)r);
    if (!lora_fast_ok(DType::BF16, x, ldx, (int)r, g.fwd_rows) ||
        !lora_update_ok(y, ldy, (int)r, g.fwd_upd))
        return fail(VKH_ERR_UNSUPPORTED, "lora_group_forward_bf16: shape or alignment");
    hipStream_t st = S(stream);
    VKH_HIP(lora_rows(DType::BF16, x, ldx, (int)T, (int)r, g.fwd_rows, 1.f, st));
    VKH_HIP(lora_update(y, ldy, (int)T, (int)r, g.fwd_upd, aor, st));
    return VKH_OK;
}

vkh_status vkh_lora_group_backward_bf16(const uint16_t *dy, uint32_t lddy, const uint16_t *x,
                                        uint32_t ldx, uint32_t T, uint32_t r, float aor,
                                        const vkh_lora_adapter *adapters, uint32_t n_adapters,
                                        float *dx, uint32_t lddx, vkh_stream stream) {
    CHECK_ARG(dy && x, "null pointer");
    LoraAdapter ad[3];
    VKH_TRY(lora_group_args(adapters, n_adapters, r, ad));
    for (uint32_t i = 0; i < n_adapters; ++i) {
        CHECK_ARG(ad[i].dyb && ad[i].da && ad[i].db, "adapter: null dyb, da or db");
        CHECK_ARG(ad[i].k <= (long)ldx && ad[i].col + ad[i].n <= (long)lddy &&
                      (!dx || ad[i].k <= (long)lddx),
                  "adapter outside the rows");
    }
    const LoraGroupSegs g = lora_group_segs(ad, (int)n_adapters, (int)r);
    if (!lora_fast_ok(DType::BF16, dy, lddy, (int)r, g.bwd_rows) ||
        !lora_fast_ok(DType::BF16, x, ldx, (int)r, g.bwd_da) ||
        !lora_fast_ok(DType::BF16, dy, lddy, (int)r, g.bwd_db) ||
        (dx && !lora_update_ok(dx, lddx, (int)r, g.bwd_upd)))
        return fail(VKH_ERR_UNSUPPORTED, "lora_group_backward_bf16: shape or alignment");
    hipStream_t st = S(stream);
    VKH_HIP(lora_rows(DType::BF16, dy, lddy, (int)T, (int)r, g.bwd_rows, 1.f, st));
    VKH_HIP(lora_cols(DType::BF16, x, ldx, (int)T, (int)r, g.bwd_da, aor, st));
    VKH_HIP(lora_cols(DType::BF16, dy, lddy, (int)T, (int)r, g.bwd_db, aor, st));
    if (dx) VKH_HIP(lora_update(dx, lddx, (int)T, (int)r, g.bwd_upd, aor, st));
    return VKH_OK;
}

// ── CCE ────────────────────────────────────────────────────────────────

// Device memory of one head call: its scratch, and the packed copies of h and W
// that the DMA-staged products need (fp32 operands in the bf16 precision; rows
// that are not whole aligned 16-byte chunks).
extern "C++" {
namespace {
struct CceOperands {
    CceShape s;
    LinForm form;
    const void *h, *w;  // as the products read them, rows of s.hs()
    char *mem = nullptr;
    vkh_status set(const vkh_cce_params *p, const float *h0, const float *w0, size_t scratch,
                   hipStream_t st, char **scratch_out) {
        s = CceShape{(int)p->n, (int)p->vocab, (int)p->dim, p->z_loss_scale, p->label_smoothing};
        form = form_of(p->precision);
        h = h0;
        w = w0;
        const bool pack = form == LinForm::MIXED || s.D % 4 || ((uintptr_t)h0 & 15u) || ((uintptr_t)w0 & 15u);
        const size_t es = form == LinForm::MIXED ? 2 : 4;
        size_t hb = 0, wb = 0;
        if (pack) {
            s.ldh = lin_packed_ld(form, s.D);
            hb = (s.N * s.ldh * es + 255) / 256 * 256;
            wb = s.V * s.ldh * es;
        }
        scratch = (scratch + 255) / 256 * 256;
        note_allocation();
        VKH_HIP(hipMallocAsync((void **)&mem, scratch + hb + wb, st));
        *scratch_out = mem;
        if (!pack) return VKH_OK;
        void *hp = mem + scratch, *wp = mem + scratch + hb;
        const hipError_t e = lin_pack(form, h0, s.N, s.D, hp, w0, s.V, s.D, wp, st);
        h = hp;
        w = wp;
        if (e == hipSuccess) return VKH_OK;
        (void)hipFreeAsync(mem, st);
        return hip_fail(e, "cce operands");
    }
};
}  // namespace
}

// fp32 operands in bf16 products (2048 x 151936 x 1024) measured, forward and
// backward: 27.5 ms on the generic kernel that converts while staging, 3.0 ms with
// the operands packed once per call.  fp32 of 127 x 32003 x 768: 1.75 -> 0.27 ms,
// with padded dz rows, a split dh and the smaller logits tiles.
vkh_status vkh_cce_forward(const vkh_cce_params *p, const float *h, const float *w,
                           const uint32_t *targets, float *lse, float *loss_row,
                           float *loss_mean, vkh_stream stream) {
    CHECK_ARG(p && h && w && targets && lse, "null pointer");
    CHECK_ARG(p->n && p->vocab && p->dim, "zero dimension");
    hipStream_t st = S(stream);
    const CceShape sz{(int)p->n, (int)p->vocab, (int)p->dim, 0.f, 0.f};
    CceOperands o;
    char *work = nullptr;
    VKH_TRY(o.set(p, h, w, cce_work_floats(sz) * 4, st, &work));
    const hipError_t e =
        o.form == LinForm::F32
            ? cce_forward(o.s, (const float *)o.h, (const float *)o.w, targets, lse, loss_row, loss_mean, (float *)work, st)
            : cce_forward16(o.s, (const bf16 *)o.h, (const bf16 *)o.w, targets, lse, loss_row, loss_mean, (float *)work, st);
    (void)hipFreeAsync(o.mem, st);
    if (e != hipSuccess) return hip_fail(e, "cce_forward");
    return VKH_OK;
}

vkh_status vkh_cce_backward(const vkh_cce_params *p, const float *h, const float *w,
                            const uint32_t *targets, const float *lse, float *dh, float *dw,
                            uint32_t accumulate_dw, vkh_stream stream) {
    CHECK_ARG(p && h && w && targets && lse, "null pointer");
    CHECK_ARG(p->n && p->vocab && p->dim, "zero dimension");
    hipStream_t st = S(stream);
    const LinForm form = form_of(p->precision);
    const int N = (int)p->n, V = (int)p->vocab, D = (int)p->dim;
    const long ldz = lin_packed_ld(form, V);
    const size_t zb = (N * ldz * (form == LinForm::F32 ? 4 : 2) + 255) / 256 * 256;
    size_t wsb = 0;  // the products' split-K partials
    auto need = [&](int m, int n, int k) {
        wsb = std::max(wsb, form == LinForm::F32 ? g32_ws_bytes_for(m, n, k) : g16_ws_bytes_for(m, n, k));
    };
    if (dh) need(N, D, V);
    if (dw) need(V, D, N);
    CceOperands o;
    char *dz = nullptr;
    VKH_TRY(o.set(p, h, w, zb + wsb, st, &dz));
    if (ldz != V) o.s.ldz = ldz;
    const GemmWs ws{wsb ? dz + zb : nullptr, wsb};
    const float beta = accumulate_dw ? 1.f : 0.f;
    const hipError_t e =
        form == LinForm::F32
            ? cce_backward(o.s, (const float *)o.h, (const float *)o.w, targets, lse, (float *)dz, dh, dw, beta, ws, st)
            : cce_backward16(o.s, (const bf16 *)o.h, (const bf16 *)o.w, targets, lse, (bf16 *)dz, dh, dw, beta, ws, st);
    (void)hipFreeAsync(o.mem, st);
    if (e != hipSuccess) return hip_fail(e, "cce_backward");
    return VKH_OK;
}

// ── norms, rope, elementwise ───────────────────────────────────────────

vkh_status vkh_rmsnorm_forward(const float *x, const float *w, float *y, uint32_t n_rows,
                               uint32_t dim, float eps, uint32_t gq, vkh_stream stream) {
    CHECK_ARG(x && w && y, "null pointer");
    VKH_HIP(rmsnorm_forward(x, w, y, DType::F32, n_rows, dim, eps, gq ? 1 : 0, S(stream)));
    return VKH_OK;
}

vkh_status vkh_rmsnorm_backward(const float *dy, const float *x, const float *w, float *dx,
                                const float *residual, float *dw, uint32_t n_rows, uint32_t dim,
                                float eps, uint32_t gq, vkh_stream stream) {
    CHECK_ARG(dy && x && w && dx, "null pointer");
    if (dim > 4096) return fail(VKH_ERR_UNSUPPORTED, "rmsnorm_backward dim > 4096");
    hipStream_t st = S(stream);
    void *partial = nullptr;
    ScratchLease lease;
    VKH_TRY(lease.acquire(rmsnorm_partial_floats(n_rows, dim) * 4 + 16, st, &partial));
    hipError_t e = rmsnorm_backward(dy, x, w, dx, nullptr, residual, dw, (float *)partial, n_rows,
                                    dim, eps, gq ? 1 : 0, st);
    if (e != hipSuccess) return hip_fail(e, "rmsnorm_backward");
    return VKH_OK;
}

// ── the allocation-free RMSNorm backward ───────────────────────────────
// The gain-gradient partials (one row of `dim` floats per block of the
// backward kernel, at most 512 blocks and dim <= 4096) live in a fixed device
// array instead of the lease above, so a call allocates nothing (for callers
// under graph capture or in loops that must not call hipMalloc).  Each GPU
// holds its own copy for the life of the process; its device address is
// looked up once per device, at the first call on it, and only that address
// is handed to kernels.  Every block overwrites its whole partial row before
// the column sum reads it, so nothing needs clearing between calls.
//
// Calls share the array, so they are ordered like the lease's uses: an event
// per device (created with the address lookup; an event holds no device
// memory) is recorded after each call's launch, and a call on another stream
// first makes its stream wait for it.  While the caller's stream is being
// captured into a graph the event is neither waited for nor recorded (a
// captured stream may not wait on work outside its capture): the caller then
// orders the graph's launches against other uses of the array itself.
constexpr size_t kNoAllocPartialFloats = 512 * 4096;  // 8 MiB
static __device__ __align__(256) float scratch[kNoAllocPartialFloats];

namespace {
constexpr int kMaxDevices = 64;
struct NoAllocScratch {
    float *ptr = nullptr;      // the device address of `scratch` on this device
    hipEvent_t done = nullptr; // recorded after each uncaptured use
    hipStream_t last = nullptr;
    bool used = false;
};
std::mutex g_scratch_mu;
NoAllocScratch g_scratch[kMaxDevices];
}  // namespace

// Set-up of the current device's array (once per device, with the mutex held).
static vkh_status noalloc_scratch_setup(int dev) {
    NoAllocScratch &d = g_scratch[dev];
    if (d.ptr) return VKH_OK;
    void *p = nullptr;
    const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess) return hip_fail(e, "hipGetSymbolAddress(scratch)");
    if (!p) return fail(VKH_ERR_HIP, "hipGetSymbolAddress(scratch) returned null");
    VKH_HIP(hipEventCreateWithFlags(&d.done, hipEventDisableTiming | hipEventDisableSystemFence));
    d.ptr = (float *)p;
    return VKH_OK;
}

vkh_status vkh_rmsnorm_backward_noalloc(const float *dy, const float *x, const float *w,
                                        float *dx, const float *residual, float *dw,
                                        uint32_t n_rows, uint32_t dim, float eps, uint32_t gq,
                                        vkh_stream stream) {
    CHECK_ARG(dy && x && w && dx, "null pointer");
    if (dim > 4096) return fail(VKH_ERR_UNSUPPORTED, "rmsnorm_backward_noalloc: dim %u > 4096", dim);
    const size_t need = rmsnorm_partial_floats((int)n_rows, (int)dim);
    if (need > kNoAllocPartialFloats)
        return fail(VKH_ERR_UNSUPPORTED, "rmsnorm_backward_noalloc: %zu partial floats > %zu",
                    need, kNoAllocPartialFloats);
    int dev = 0;
    VKH_HIP(hipGetDevice(&dev));
    if (dev < 0 || dev >= kMaxDevices)
        return fail(VKH_ERR_UNSUPPORTED, "device index %d >= %d", dev, kMaxDevices);
    const hipStream_t st = S(stream);
    std::lock_guard<std::mutex> lk(g_scratch_mu);  // held while the call enqueues
    VKH_TRY(noalloc_scratch_setup(dev));
    NoAllocScratch &d = g_scratch[dev];
    hipStreamCaptureStatus cs = hipStreamCaptureStatusNone;
    VKH_HIP(hipStreamIsCapturing(st, &cs));
    const bool captured = cs != hipStreamCaptureStatusNone;
    if (!captured && d.used && d.last != st) VKH_HIP(hipStreamWaitEvent(st, d.done, 0));
    hipError_t e = rmsnorm_backward(dy, x, w, dx, nullptr, residual, dw, d.ptr, n_rows, dim, eps,
                                    gq ? 1 : 0, st);
    if (e != hipSuccess) return hip_fail(e, "rmsnorm_backward_noalloc");
    if (!captured) {
        VKH_HIP(hipEventRecord(d.done, st));
        d.used = true;
        d.last = st;
    }
    return VKH_OK;
}

uint64_t vkh_allocation_count(void) { return g_allocations.load(std::memory_order_relaxed); }

vkh_status vkh_swiglu_forward(const float *pg, const float *up, float *g, size_t n,
                              vkh_stream stream) {
    CHECK_ARG(pg && up && g, "null pointer");
    CHECK_ARG(n < (1ull << 31), "n too large");
    VKH_HIP(swiglu_forward(pg, (long)n, up, (long)n, g, (long)n, DType::F32, 1, (int)n, S(stream)));
    return VKH_OK;
}

vkh_status vkh_swiglu_backward(const float *dg, const float *pg, const float *up, float *dpg,
                               float *dup, size_t n, vkh_stream stream) {
    CHECK_ARG(dg && pg && up && dpg && dup, "null pointer");
    CHECK_ARG(n < (1ull << 31), "n too large");
    VKH_HIP(swiglu_backward(dg, (long)n, pg, (long)n, up, (long)n, dpg, (long)n, dup, (long)n,
                            DType::F32, 1, (int)n, S(stream)));
    return VKH_OK;
}

static vkh_status rope_common(const vkh_rope_params *p, const float *qi, float *qo,
                              const float *ki, float *ko, bool bw, vkh_stream stream) {
    CHECK_ARG(p && qi && qo && ki && ko, "null pointer");
    CHECK_ARG(p->rotary_dim <= p->head_dim && (p->rotary_dim % 2) == 0, "rotary_dim");
    const int seq = p->seq_len ? (int)p->seq_len : (int)p->n_pos;
    const float2 *tab = nullptr;
    VKH_TRY(rope_table_cached(seq, p->rotary_dim, p->theta_base, &tab));
    const long ldq = (long)p->n_q_heads * p->head_dim, ldk = (long)p->n_kv_heads * p->head_dim;
    VKH_HIP(qk_rope(qi, ldq, qo, ldq, ki, ldk, ko, ldk, p->n_pos, p->n_q_heads, p->n_kv_heads,
                    p->head_dim, p->rotary_dim, seq, tab, bw, S(stream)));
    return VKH_OK;
}

vkh_status vkh_qk_rope_forward(const vkh_rope_params *p, const float *q_in, float *q_out,
                               const float *k_in, float *k_out, vkh_stream stream) {
    return rope_common(p, q_in, q_out, k_in, k_out, false, stream);
}

vkh_status vkh_qk_rope_backward(const vkh_rope_params *p, const float *dq_out, float *dq_in,
                                const float *dk_out, float *dk_in, vkh_stream stream) {
    return rope_common(p, dq_out, dq_in, dk_out, dk_in, true, stream);
}

vkh_status vkh_qkv_project_bf16(const vkh_rope_params *p, uint32_t K, float eps, int qk_norm,
                                const void *x, const void *w, const float *wq, const float *wk,
                                float *y, void *out, int fused, vkh_stream stream) {
    CHECK_ARG(p && x && w && y && out, "null pointer");
    CHECK_ARG(!qk_norm || (wq && wk), "null norm gains");
    CHECK_ARG(p->rotary_dim <= p->head_dim && (p->rotary_dim % 2) == 0, "rotary_dim");
    QkvLayout L;
    L.n_rows = (int)p->n_pos; L.n_q_heads = (int)p->n_q_heads; L.n_kv_heads = (int)p->n_kv_heads;
    L.head_dim = (int)p->head_dim; L.seq_len = p->seq_len ? (int)p->seq_len : (int)p->n_pos;
    L.rotary_dim = (int)p->rotary_dim; L.theta = p->theta_base; L.eps = eps; L.qk_norm = qk_norm ? 1 : 0;
    const float2 *tab = nullptr;
    VKH_TRY(rope_table_cached(L.seq_len, L.rotary_dim, L.theta, &tab));
    const uint32_t N = (p->n_q_heads + 2 * p->n_kv_heads) * p->head_dim;
    hipStream_t st = S(stream);
    if (fused) {
        const hipError_t e = g16_qkv_norm_rope((const bf16 *)x, K, (const bf16 *)w, K, y, N, L.n_rows,
                                               (int)N, (int)K, L, wq, wk, (bf16 *)out, N, tab, st);
        if (e != hipErrorNotSupported) {
            VKH_HIP(e);
            return VKH_OK;
        }
    }
    const vkh_status r = vkh_matmul_nt_bf16(x, w, y, p->n_pos, N, K, stream);
    if (r != VKH_OK) return r;
    VKH_HIP(qkv_prepare_forward(L, y, N, wq, wk, out, N, DType::BF16, tab, st));
    return VKH_OK;
}

vkh_status vkh_qkv_project(const vkh_rope_params *p, uint32_t K, float eps, int qk_norm,
                           const float *x, const float *w, const float *wq, const float *wk,
                           float *y, float *out, int fused, vkh_stream stream) {
    CHECK_ARG(p && x && w && y && out, "null pointer");
    CHECK_ARG(!qk_norm || (wq && wk), "null norm gains");
    CHECK_ARG(p->rotary_dim <= p->head_dim && (p->rotary_dim % 2) == 0, "rotary_dim");
    QkvLayout L;
    L.n_rows = (int)p->n_pos; L.n_q_heads = (int)p->n_q_heads; L.n_kv_heads = (int)p->n_kv_heads;
    L.head_dim = (int)p->head_dim; L.seq_len = p->seq_len ? (int)p->seq_len : (int)p->n_pos;
    L.rotary_dim = (int)p->rotary_dim; L.theta = p->theta_base; L.eps = eps; L.qk_norm = qk_norm ? 1 : 0;
    const float2 *tab = nullptr;
    VKH_TRY(rope_table_cached(L.seq_len, L.rotary_dim, L.theta, &tab));
    const uint32_t N = (p->n_q_heads + 2 * p->n_kv_heads) * p->head_dim;
    hipStream_t st = S(stream);
    if (fused) {
        const hipError_t e = g32_qkv_norm_rope(x, K, w, K, y, N, L.n_rows, (int)N, (int)K, L, wq, wk,
                                               out, N, tab, st);
        if (e != hipErrorNotSupported) {
            VKH_HIP(e);
            return VKH_OK;
        }
    }
    const vkh_status r = vkh_matmul_nt(x, w, y, p->n_pos, N, K, VKH_PRECISION_FP32, stream);
    if (r != VKH_OK) return r;
    VKH_HIP(qkv_prepare_forward(L, y, N, wq, wk, out, N, DType::F32, tab, st));
    return VKH_OK;
}

vkh_status vkh_embed_lookup(const float *embed, const uint32_t *ids, float *out, uint32_t n_pos,
                            uint32_t dim, float scale, vkh_stream stream) {
    CHECK_ARG(embed && ids && out, "null pointer");
    VKH_HIP(embed_lookup(embed, ids, out, n_pos, dim, scale, S(stream)));
    return VKH_OK;
}

vkh_status vkh_embedding_backward(const float *dy, const uint32_t *ids, float *dE,
                                  uint32_t n_pos, uint32_t dim, uint32_t vocab,
                                  vkh_stream stream) {
    CHECK_ARG(dy && ids && dE, "null pointer");
    if (n_pos > (uint32_t)kEmbedBwMaxPos) return fail(VKH_ERR_UNSUPPORTED, "n_pos > %d", kEmbedBwMaxPos);
    // the owner kernels need no work buffer (no lease, no ordering event)
    hipError_t e = embedding_backward(dy, ids, dE, n_pos, dim, vocab, true, nullptr, S(stream));
    if (e != hipSuccess) return hip_fail(e, "embedding_backward");
    return VKH_OK;
}

vkh_status vkh_adam_step(float *param, const float *grad, float *m, float *v, size_t n, float lr,
                         float beta1, float beta2, float eps, uint32_t t, float wd,
                         vkh_stream stream) {
    CHECK_ARG(param && grad && m && v, "null pointer");
    CHECK_ARG(t >= 1, "t must be >= 1");
    const float tf = (float)t;
    VKH_HIP(adam_step(param, grad, m, v, n, lr, beta1, beta2, eps, 1.0f - powf(beta1, tf),
                      1.0f - powf(beta2, tf), wd, nullptr, S(stream)));
    return VKH_OK;
}

vkh_status vkh_add_in_place(float *dst, const float *src, size_t n, vkh_stream stream) {
    CHECK_ARG(dst && src, "null pointer");
    VKH_HIP(add_in_place(dst, src, n, S(stream)));
    return VKH_OK;
}

vkh_status vkh_vec_add(const float *a, const float *b, float *c, size_t n, vkh_stream stream) {
    CHECK_ARG(a && b && c, "null pointer");
    VKH_HIP(vec_add(a, b, c, n, S(stream)));
    return VKH_OK;
}

vkh_status vkh_scale(const float *in, float *out, size_t n, float s, vkh_stream stream) {
    CHECK_ARG(in && out, "null pointer");
    VKH_HIP(scale(in, out, n, s, S(stream)));
    return VKH_OK;
}

vkh_status vkh_cast_f32_to_bf16(const float *in, void *out, size_t n, vkh_stream stream) {
    CHECK_ARG(in && out, "null pointer");
    VKH_HIP(cast_f32_to_bf16(in, (bf16 *)out, n, S(stream)));
    return VKH_OK;
}

// ── plumbing ───────────────────────────────────────────────────────────

vkh_status vkh_device_count(int *count) {
    CHECK_ARG(count, "null pointer");
    *count = 0;
    hipError_t e = hipGetDeviceCount(count);
    if (e != hipSuccess) { *count = 0; return fail(VKH_ERR_NO_DEVICE, "%s", hipGetErrorString(e)); }
    return VKH_OK;
}
vkh_status vkh_set_device(int device) { VKH_HIP(hipSetDevice(device)); return VKH_OK; }
vkh_status vkh_malloc(void **ptr, size_t bytes) {
    CHECK_ARG(ptr, "null pointer");
    note_allocation();
    VKH_HIP(hipMalloc(ptr, bytes ? bytes : 1));
    return VKH_OK;
}
vkh_status vkh_free(void *ptr) { VKH_HIP(hipFree(ptr)); return VKH_OK; }
vkh_status vkh_memcpy_h2d(void *dst, const void *src, size_t bytes) {
    VKH_HIP(hipMemcpy(dst, src, bytes, hipMemcpyHostToDevice));
    return VKH_OK;
}
vkh_status vkh_memcpy_d2h(void *dst, const void *src, size_t bytes) {
    VKH_HIP(hipMemcpy(dst, src, bytes, hipMemcpyDeviceToHost));
    return VKH_OK;
}
vkh_status vkh_memset(void *ptr, int value, size_t bytes) {
    VKH_HIP(hipMemset(ptr, value, bytes));
    return VKH_OK;
}
vkh_status vkh_device_synchronize(void) { VKH_HIP(hipDeviceSynchronize()); return VKH_OK; }
vkh_status vkh_stream_create(vkh_stream *out) {
    CHECK_ARG(out, "null pointer");
    hipStream_t s;
    VKH_HIP(hipStreamCreateWithFlags(&s, hipStreamNonBlocking));
    *out = (vkh_stream)s;
    return VKH_OK;
}
vkh_status vkh_stream_destroy(vkh_stream s) { VKH_HIP(hipStreamDestroy(S(s))); return VKH_OK; }
vkh_status vkh_stream_synchronize(vkh_stream s) { VKH_HIP(hipStreamSynchronize(S(s))); return VKH_OK; }
vkh_status vkh_event_create(vkh_event *out) {
    CHECK_ARG(out, "null pointer");
    hipEvent_t e;
    VKH_HIP(hipEventCreate(&e));
    *out = (vkh_event)e;
    return VKH_OK;
}
vkh_status vkh_event_destroy(vkh_event e) { VKH_HIP(hipEventDestroy((hipEvent_t)e)); return VKH_OK; }
vkh_status vkh_event_record(vkh_event e, vkh_stream s) {
    VKH_HIP(hipEventRecord((hipEvent_t)e, S(s)));
    return VKH_OK;
}
vkh_status vkh_event_synchronize(vkh_event e) { VKH_HIP(hipEventSynchronize((hipEvent_t)e)); return VKH_OK; }
vkh_status vkh_event_elapsed_ms(vkh_event a, vkh_event b, float *ms) {
    CHECK_ARG(ms, "null pointer");
    VKH_HIP(hipEventElapsedTime(ms, (hipEvent_t)a, (hipEvent_t)b));
    return VKH_OK;
}

}  // extern "C"
