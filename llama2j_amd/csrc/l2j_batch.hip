// libllama2j_hip.so: several sequences at once (l2j_decode_greedy_batch, l2j_batch_matmul).
#include "l2j_internal.hpp"
#include "batch_kernels.hpp"
#include "batch_step.hpp"
#include "rows_kernels.hpp"
#include "rows.hpp"

#include <condition_variable>
#include <thread>

using namespace l2j;

bool l2j::matrix_shape(const l2j_config &cf, int tensor, int *rows, int *K)
{
    const int kvd = cf.dim / cf.n_heads * cf.n_kv_heads;
    switch (tensor) {
    case L2J_WQ: case L2J_WO: *rows = cf.dim; *K = cf.dim; return true;
    case L2J_WK: case L2J_WV: *rows = kvd; *K = cf.dim; return true;
    case L2J_W1: case L2J_W3: *rows = cf.hidden_dim; *K = cf.dim; return true;
    case L2J_W2: *rows = cf.dim; *K = cf.hidden_dim; return true;
    default: return false;
    }
}

// The tile-ordered copy of `tensor` for the batched path (rows % 16 == 0 and K % 256 == 0 checked by the caller; the
// caller holds the context's upload lock: an upload of the tensor marks the copy stale, invalidate_batch_tiles).
static int ensure_batch_tiles(l2j_ctx *c, int tensor)
{
    if (c->bt_done[tensor]) return L2J_OK;
    int rows = 0, K = 0;
    if (!matrix_shape(c->cfg, tensor, &rows, &K)) return fail(L2J_E_ARG, "not a matrix tensor");
    const QTensor &t = c->qt[tensor];
    if (t.groups_loaded < t.ngroups) return fail(L2J_E_STATE, "tensor not uploaded");
    const uint64_t n = (uint64_t)c->cfg.n_layers * rows * K;
    int rc;
    if (!c->bt_codes[tensor] && (rc = dev_alloc(&c->bt_codes[tensor], n))) return rc;
    if (!c->bt_gs[tensor] && (rc = dev_alloc(&c->bt_gs[tensor], n / 256))) return rc;
    const long n16 = (long)(n / 16);
    hipLaunchKernelGGL(k_btile, dim3((unsigned)((n16 + 255) / 256)), dim3(256), 0, c->stream, t.codes, t.gs, n16, rows, K, c->bt_codes[tensor],
                       c->bt_gs[tensor]);
    HIPCHK(hipGetLastError());
    c->bt_done[tensor] = true;
    return L2J_OK;
}

int l2j::ensure_batch_tiles(l2j_ctx *c)
{
    if (c->bt_ready) return L2J_OK;
    std::lock_guard<std::mutex> lock(c->upload_mu);
    for (int t : {L2J_WQ, L2J_WK, L2J_WV, L2J_WO, L2J_W1, L2J_W2, L2J_W3}) {
        const int trc = ensure_batch_tiles(c, t);
        if (trc) return trc;
    }
    c->bt_ready = true;
    return L2J_OK;
}

static QMat bqmat(const l2j_ctx *c, int t, uint64_t off)
{
    QMat m;
    m.codes = c->bt_codes[t];
    m.gs = c->bt_gs[t];
    m.off = (long)off;
    return m;
}

extern "C" {

int l2j_batch_matmul(l2j_ctx *c, int tensor, int layer, const float *x, float *y, int32_t groups_per_slice, int32_t rounds,
                     double *mean_us)
{
    return ctx_rc(c, [&]() -> int {
        std::lock_guard<std::mutex> forward_lock(g_forward_mu);
        if (!c || !x || !y) return fail(L2J_E_ARG, "null argument");
        int rows = 0, K = 0;
        if (!matrix_shape(c->cfg, tensor, &rows, &K)) return fail(L2J_E_ARG, "not a matrix tensor");
        if (layer < 0 || layer >= c->cfg.n_layers) return fail(L2J_E_ARG, "layer out of range");
        if (K % 256 || rows % 16) return fail(L2J_E_SIZE, "the batched matrix product needs rows of whole groups (K % 256 == 0) and rows % 16 == 0");
        (void)groups_per_slice;   // (the product picks its slices of K by the shape)
        HIPCHK(hipSetDevice(c->cfg.device));
        {
            std::lock_guard<std::mutex> lock(c->upload_mu);
            const int trc = ensure_batch_tiles(c, tensor);
            if (trc) return trc;
        }
        HIPCHK(prepare_dgemm(c));
        const int slices = product_slices(c, rows / 16, K / 256, kBatch);
        RowBufs rb;
        float *dx = nullptr, *dy = nullptr;
        hipEvent_t e0 = nullptr, e1 = nullptr;
        auto release = [&]() {
            (void)hipFree(dx); (void)hipFree(dy);
            rb.release();
            if (e0) (void)hipEventDestroy(e0);
            if (e1) (void)hipEventDestroy(e1);
        };
        hipError_t e = hipMalloc(reinterpret_cast<void **>(&dx), (size_t)kBatch * K * sizeof(float));
        if (e == hipSuccess) e = hipMalloc(reinterpret_cast<void **>(&dy), (size_t)kBatch * rows * sizeof(float));
        if (e == hipSuccess) e = rb.alloc(c, kBatch, false);
        if (e == hipSuccess) e = hipEventCreate(&e0);
        if (e == hipSuccess) e = hipEventCreate(&e1);
        if (e == hipSuccess) e = hipMemcpyAsync(dx, x, (size_t)kBatch * K * sizeof(float), hipMemcpyHostToDevice, c->stream);
        if (e == hipSuccess) {
            hipLaunchKernelGGL(k_rows_digits, dim3((unsigned)((kBatch * (K / 16) + 255) / 256)), dim3(256), 0, c->stream, dx, rb.dig, kBatch, K);
            const int n = std::max(1, (int)rounds);
            launch_dgemm(c, {tensor}, layer, rb.dig, kBatch, rb.part);   // warm
            (void)hipEventRecord(e0, c->stream);
            for (int i = 0; i < n; i++) launch_dgemm(c, {tensor}, layer, rb.dig, kBatch, rb.part);
            (void)hipEventRecord(e1, c->stream);
            hipLaunchKernelGGL(k_breduce, dim3(256), dim3(256), 0, c->stream, rb.part, dy, rows, slices);
            e = hipGetLastError();
            if (e == hipSuccess) e = hipMemcpyAsync(y, dy, (size_t)kBatch * rows * sizeof(float), hipMemcpyDeviceToHost, c->stream);
            if (e == hipSuccess) e = hipStreamSynchronize(c->stream);
            float ms = 0.0f;
            if (e == hipSuccess) e = hipEventElapsedTime(&ms, e0, e1);
            if (mean_us) *mean_us = (double)ms * 1e3 / n;
        }
        release();
        if (e != hipSuccess) return fail(e == hipErrorOutOfMemory ? L2J_E_OOM : L2J_E_HIP, std::string("batch matmul: ") + hipGetErrorString(e));
        return L2J_OK;
    }());
}

}  // extern "C"

// ---- several sequences at once ----------------------------------------------------------------------------------

// Device memory, pinned staging and the captured step of the batched decode.  The context owns one set, made by the first
// l2j_decode_greedy_batch and kept until l2j_destroy; a call that needs more (other sequence count, more steps, longer
// prompts) replaces it.  No call allocates or captures anything once the set fits.
struct l2j::BatchBufs {
    int nseq = 0, cap_steps = 0, cap_pstride = 0;   // what the buffers and the graph's kernel arguments are made for
    RowBufs r;                                      // a row per sequence
    float *logits = nullptr, *cls_part = nullptr;   // (sequence, vocab); the slices of the classifier
    float *xb = nullptr, *hb = nullptr;             // k_bstep: the inputs of Wo and W2,
    float *part[3] = {nullptr, nullptr, nullptr};   // the slices of its products
    float *kc = nullptr, *vc = nullptr;             // (sequence, layer, kv head, cap_steps, head_size)
    BatchState *st = nullptr;
    int *prompts = nullptr, *out = nullptr;         // (sequence, cap_pstride), (sequence, cap_steps)
    unsigned *done = nullptr;             // (1 + nseq) counters and
    unsigned long long *best = nullptr;   // (nseq, kNextParts) maxima of k_bnext
    unsigned *bar_ctr = nullptr;   // k_bstep: the counters of its grid barrier,
    int *fault = nullptr;          // the flag a bounded wait sets when it runs out,
    float *ssq = nullptr;          // the sums of squares behind the two norms of a layer,
    BStep *step_args = nullptr;    // its argument (fixed for the life of the buffers)
    int step_grid = 0;             // workgroups of k_bstep (0: the layers run as eight launches each)
    int fuse_opt = 0;              // option batch_fuse when the step was planned
    int h_fault = 0;
    int *h_pin = nullptr;   // pinned: every transfer of a call goes through it, as in the single-sequence loops
    // the logits of every step for a caller that wants them: kept here while later steps are computed, made by the first such call
    float *log_dev = nullptr, *log_pin = nullptr;   // log_slots steps on the device, one pinned
    int log_slots = 0;
    hipStream_t log_stream = nullptr;
    hipEvent_t log_step[kLogSlots] = {};            // the slot holds its step's logits
    BatchSamplers samplers;   // l2j_decode_sample_batch: a sampler per sequence (made by its first call)
    hipGraph_t graph = nullptr;
    hipGraphExec_t exec = nullptr;
    hipEvent_t e0 = nullptr, e1 = nullptr;
    // Slots for a call of `steps` steps: one a step up to kLogSlots, or as many as the device memory suffices for.
    hipError_t ensure_log(size_t step_floats, int steps)
    {
        hipError_t e = hipSuccess;
        const int want = std::min(steps, kLogSlots);
        if (log_slots < want) {
            (void)hipFree(log_dev);   // (no call is under way: nothing uses it)
            log_dev = nullptr; log_slots = 0;
            for (int n = want; n > 0; n /= 2) {
                e = hipMalloc(reinterpret_cast<void **>(&log_dev), n * step_floats * sizeof(float));
                if (e == hipSuccess) log_slots = n;
                if (e != hipErrorOutOfMemory) break;
                (void)hipGetLastError();   // (or the next launch would report it)
            }
        }
        if (e == hipSuccess && !log_pin) e = hipHostMalloc(reinterpret_cast<void **>(&log_pin), step_floats * sizeof(float), hipHostMallocDefault);
        if (e == hipSuccess && !log_stream) e = hipStreamCreateWithFlags(&log_stream, hipStreamNonBlocking);
        for (int i = 0; i < log_slots; i++)
            if (e == hipSuccess && !log_step[i]) e = hipEventCreateWithFlags(&log_step[i], hipEventDisableTiming);
        return e;
    }
    void release()
    {
        for (hipEvent_t ev : log_step)
            if (ev) (void)hipEventDestroy(ev);
        if (log_stream) (void)hipStreamDestroy(log_stream);
        (void)hipFree(log_dev);
        if (log_pin) (void)hipHostFree(log_pin);
        if (exec) (void)hipGraphExecDestroy(exec);
        if (graph) (void)hipGraphDestroy(graph);
        if (e0) (void)hipEventDestroy(e0);
        if (e1) (void)hipEventDestroy(e1);
        void *ps[] = {xb, hb, logits, cls_part, part[0], part[1], part[2], kc, vc, st, prompts, out, done, best, bar_ctr, fault, ssq, step_args};
        for (void *p : ps) (void)hipFree(p);
        r.release();
        free_batch_samplers(&samplers);
        if (h_pin) (void)hipHostFree(h_pin);
    }
};

void l2j::free_batch(l2j_ctx *c)
{
    if (c->batch) {
        c->batch->release();
        delete c->batch;
        c->batch = nullptr;
    }
    c->rows.release();
    for (int t = 0; t < L2J_TENSOR_COUNT; t++) {
        (void)hipFree(c->bt_codes[t]);
        (void)hipFree(c->bt_gs[t]);
        c->bt_codes[t] = nullptr; c->bt_gs[t] = nullptr; c->bt_done[t] = false;
    }
    c->bt_ready = false;
}

void l2j::invalidate_batch_tiles(l2j_ctx *c, int tensor)
{
    c->bt_done[tensor] = false;
    c->bt_ready = false;
}

namespace {

constexpr int kClsGps = 2;   // k_bgemm_f32: groups of 256 floats per slice of K

int batch_slices(int K) { return bg_slices(K); }
int cls_slices(int K) { return (K / 256 + kClsGps - 1) / kClsGps; }
size_t step_lds(int nseq) { return bg_lds_bytes(nseq, nseq / kBatch); }       // k_bstep: 256 threads per 16 sequences
size_t batch_lds_f32(int nseq) { return (size_t)nseq * (kClsGps * 256 + kXPad) * sizeof(float); }   // k_bgemm_f32: floats

// The product of one layer's matrices `tensors` (the same input, the same row length) as one argument of the one-launch step.
BGemm bgemm_args(l2j_ctx *c, std::initializer_list<int> tensors, int layer, const float *x, float *const *part)
{
    BGemm a{};
    int K = 0;
    for (int tensor : tensors) {
        int rows = 0;
        matrix_shape(c->cfg, tensor, &rows, &K);
        a.m[a.nmat] = bqmat(c, tensor, (uint64_t)layer * rows * K);
        a.rows[a.nmat] = rows; a.part[a.nmat] = part[a.nmat];
        a.nmat++;
    }
    a.K = K; a.x = x;
    return a;
}

// The workgroups per slice of K: at most gmax (all of a launch resident at once); every workgroup takes every gx-th tile of
// 16 rows, in batches of as many tiles as it has waves, so no more workgroups than the number of rounds needs.
int bgemm_shape(const BGemm &a, int gmax)
{
    int tiles = 0;
    for (int i = 0; i < a.nmat; i++) tiles += a.rows[i] / 16;
    const int g = std::max(1, std::min(gmax, tiles)), iters = (tiles + g - 1) / g;
    return (tiles + iters - 1) / iters;
}

// The grid of k_bstep: one workgroup per compute unit, all resident (by the runtime's count for the kernel and its LDS);
// 0 when the shape does not fit (a product with more slices of K than workgroups) or the option is off.
hipError_t plan_bstep(l2j_ctx *c, BatchBufs &b, int nseq)
{
    b.step_grid = 0;
    if (!c->opt[OPT_BATCH_FUSE]) return hipSuccess;
    const void *kernel = nseq == kBatch ? (const void *)k_bstep<1> : (const void *)k_bstep<2>;
    hipError_t e = hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)step_lds(nseq));
    if (e != hipSuccess) return e;
    int per_cu = 0;
    e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, kernel, kBgThreads * (nseq / kBatch), step_lds(nseq));
    if (e != hipSuccess) return e;
    if (per_cu < 1 || c->n_cu < batch_slices(c->cfg.hidden_dim) || c->n_cu < batch_slices(c->cfg.dim)) return hipSuccess;
    b.step_grid = c->n_cu;
    return hipSuccess;
}

// The argument of k_bstep for these buffers.
BStep bstep_args(l2j_ctx *c, BatchBufs &b, int max_pos, int nseq)
{
    const l2j_config &cf = c->cfg;
    BStep a{};
    a.g[BS_QKV] = bgemm_args(c, {L2J_WQ, L2J_WK, L2J_WV}, 0, b.r.xn, b.part);
    a.g[BS_WO] = bgemm_args(c, {L2J_WO}, 0, b.xb, b.part);
    a.g[BS_W13] = bgemm_args(c, {L2J_W1, L2J_W3}, 0, b.r.xn, b.part);
    a.g[BS_W2] = bgemm_args(c, {L2J_W2}, 0, b.hb, b.part);
    for (int k = 0; k < 4; k++) a.gx[k] = bgemm_shape(a.g[k], std::max(1, b.step_grid / batch_slices(a.g[k].K)));
    a.n_layers = cf.n_layers; a.nseq = nseq; a.dim = cf.dim; a.hidden = cf.hidden_dim; a.n_heads = cf.n_heads;
    a.kv_mul = cf.n_heads / cf.n_kv_heads; a.head_size = c->head_size; a.kv_dim = c->kv_dim;
    a.sqrt_hs = sqrtf((float)c->head_size);
    a.rope = c->rope; a.kc = b.kc; a.vc = b.vc; a.seq_stride = (long)cf.n_layers * max_pos * c->kv_dim; a.layer_stride = (long)max_pos * c->kv_dim; a.cap = max_pos; a.st = b.st;
    a.x = b.r.x; a.xn = b.r.xn; a.xb = b.xb; a.hb = b.hb; a.rmsw = c->rmsw; a.ssq = b.ssq;
    a.silu = c->silu; a.exact = (cf.flags & L2J_F_EXACT_SILU) ? 1 : 0;
    a.bar.ctr = b.bar_ctr; a.bar.fault = b.fault; a.bar.ngroups = kBarGroups; a.bar.maxspin = c->opt[OPT_BARRIER_SPINS];
    return a;
}

// All layers of a step in one launch.
void launch_bstep(l2j_ctx *c, BatchBufs &b, int nseq)
{
    const dim3 grid(b.step_grid), block(kBgThreads * (nseq / kBatch));
    const BStep *args = b.step_args;
    if (nseq == kBatch) hipLaunchKernelGGL(k_bstep<1>, grid, block, step_lds(nseq), c->stream, args);
    else hipLaunchKernelGGL(k_bstep<2>, grid, block, step_lds(nseq), c->stream, args);
}

// The classifier on one row per sequence (xn: after the final norm), the logits and the next tokens.
void launch_batch_tokens(l2j_ctx *c, BatchBufs &b, const float *xn)
{
    const l2j_config &cf = c->cfg;
    hipStream_t s = c->stream;
    BGemmF32 g{};
    g.w = c->wcls; g.rows = cf.vocab_size; g.K = cf.dim; g.x = xn; g.part = b.cls_part; g.gps = kClsGps;
    const dim3 cg((cf.vocab_size + kBgRowsPerWG - 1) / kBgRowsPerWG, cls_slices(cf.dim));
    if (b.nseq == kBatch) hipLaunchKernelGGL(k_bgemm_f32<1>, cg, dim3(kBgThreads), batch_lds_f32(b.nseq), s, g);
    else hipLaunchKernelGGL(k_bgemm_f32<2>, cg, dim3(kBgThreads), batch_lds_f32(b.nseq), s, g);
    BNext n{};
    n.part = b.cls_part; n.slices = cls_slices(cf.dim); n.vocab = cf.vocab_size; n.logits = b.logits; n.st = b.st; n.prompts = b.prompts;
    n.prompt_stride = b.cap_pstride; n.out_tokens = b.out; n.out_stride = b.cap_steps;
    n.best = b.best; n.done = b.done;
    hipLaunchKernelGGL(k_bnext, dim3(kNextParts, b.nseq), dim3(512), 0, s, n);
}

// One position of all sequences: embedding, the layers, the classifier, the next tokens.
void launch_batch_step(l2j_ctx *c, BatchBufs &b)
{
    const l2j_config &cf = c->cfg;
    const int dim = cf.dim, L = cf.n_layers, hs = c->head_size, kvd = c->kv_dim, nseq = b.nseq, cap = b.cap_steps;
    hipStream_t s = c->stream;
    if (b.step_grid > 0) {
        hipLaunchKernelGGL(k_bembed, dim3(nseq), dim3(256), 0, s, c->emb, b.st, b.r.x, dim, b.bar_ctr);
        hipLaunchKernelGGL(k_brms, dim3(nseq), dim3(1024), 0, s, b.r.x, c->rmsw, b.r.xn, dim);
        launch_bstep(c, b, nseq);
        hipLaunchKernelGGL(k_brms, dim3(nseq), dim3(1024), 0, s, b.r.x, c->rmsw + (size_t)2 * L * dim, b.r.xn, dim);   // the final norm
        launch_batch_tokens(c, b, b.r.xn);
        return;
    }
    RowNorm n{};
    n.emb = c->emb; n.nrows = nseq; n.x = b.r.x; n.dim = dim; n.dig = b.r.dig;
    n.tokens = b.st->token; n.w = c->rmsw;
    launch_norm(c, n, nseq);
    n.tokens = nullptr;
    n.part = b.r.part;
    for (int l = 0; l < L; l++) {
        BAttn t{};
        t.slices = launch_dgemm(c, {L2J_WQ, L2J_WK, L2J_WV}, l, b.r.dig, nseq, b.r.part);
        t.part = b.r.part; t.rope = c->rope;
        t.kc = b.kc + (size_t)l * cap * kvd; t.vc = b.vc + (size_t)l * cap * kvd;
        t.seq_stride = (long)L * cap * kvd; t.cap = cap; t.out = b.r.dig; t.st = b.st;
        t.kv_mul = c->kv_mul; t.kv_dim = kvd; t.dim = dim; t.sqrt_hs = sqrtf((float)hs);
        const dim3 ag(dim / 256, nseq);
        if (hs == 64) hipLaunchKernelGGL(k_battn<16>, ag, dim3(1024), 0, s, t);
        else if (hs == 128) hipLaunchKernelGGL(k_battn<32>, ag, dim3(512), 0, s, t);
        else hipLaunchKernelGGL(k_battn<64>, ag, dim3(256), 0, s, t);
        n.slices = launch_dgemm(c, {L2J_WO}, l, b.r.dig, nseq, b.r.part);
        n.per_slice = 0;
        n.w = c->rmsw + (size_t)(L + l) * dim;
        launch_norm(c, n, nseq);
        launch_ffn(c, l, b.r, nseq, n);
        // the residual, then the norm of what follows: the next layer's attention norm, or the final one (rmsw: att, ffn, final)
        n.w = c->rmsw + (l + 1 < L ? (size_t)(l + 1) * dim : (size_t)2 * L * dim);
        n.xn = l + 1 < L ? nullptr : b.r.xn;
        launch_norm(c, n, nseq);
    }
    launch_batch_tokens(c, b, b.r.xn);
}

int hip_rc(hipError_t e, const char *what)
{
    return fail(e == hipErrorOutOfMemory ? L2J_E_OOM : L2J_E_HIP, std::string("batched decode: ") + what + ": " + hipGetErrorString(e));
}

// The context's buffers for n_seq sequences over `steps` positions with prompts of up to `pstride` ids: kept when they fit.
int ensure_batch(l2j_ctx *c, int nseq, int steps, int pstride)
{
    BatchBufs *old = c->batch;
    if (old && old->nseq == nseq && old->cap_steps >= steps && old->cap_pstride >= pstride && old->fuse_opt == c->opt[OPT_BATCH_FUSE]) return L2J_OK;
    if (old) {
        hipError_t se = hipStreamSynchronize(c->stream);
        if (se != hipSuccess) return hip_rc(se, "synchronize");
        old->release();
        delete old;
        c->batch = nullptr;
    }
    const l2j_config &cf = c->cfg;
    const int dim = cf.dim, hidden = cf.hidden_dim, L = cf.n_layers, kvd = c->kv_dim, vocab = cf.vocab_size;
    const size_t cache_floats = (size_t)nseq * L * steps * kvd;
    BatchBufs *b = new (std::nothrow) BatchBufs();
    if (!b) return fail(L2J_E_OOM, "batched decode: host allocation failed");
    b->nseq = nseq; b->cap_steps = steps; b->cap_pstride = pstride; b->fuse_opt = c->opt[OPT_BATCH_FUSE];
    hipError_t e = hipSuccess;
    auto alloc = [&](auto **p, size_t n) {
        if (e == hipSuccess) e = hipMalloc(reinterpret_cast<void **>(p), n * sizeof(**p));
    };
    e = prepare_dgemm(c);
    if (e == hipSuccess) e = b->r.alloc(c, nseq, false);
    alloc(&b->logits, (size_t)nseq * vocab); alloc(&b->cls_part, (size_t)nseq * cls_slices(dim) * vocab);
    alloc(&b->kc, cache_floats); alloc(&b->vc, cache_floats);
    alloc(&b->st, 1); alloc(&b->prompts, (size_t)nseq * pstride); alloc(&b->out, (size_t)nseq * steps); alloc(&b->done, 1 + nseq);
    alloc(&b->best, (size_t)nseq * kNextParts);
    if (e == hipSuccess) e = plan_bstep(c, *b, nseq);
    if (e == hipSuccess && b->step_grid > 0) {
        const size_t part_floats = (size_t)nseq * std::max((size_t)batch_slices(dim) * hidden, (size_t)batch_slices(hidden) * dim);
        alloc(&b->xb, (size_t)nseq * dim); alloc(&b->hb, (size_t)nseq * hidden);
        for (int i = 0; i < 3; i++) alloc(&b->part[i], part_floats);
        alloc(&b->bar_ctr, (size_t)kBarStride); alloc(&b->fault, 1); alloc(&b->ssq, (size_t)2 * nseq * (dim / 256));
        if (e == hipSuccess) e = hipMemsetAsync(b->bar_ctr, 0, kBarStride * sizeof(unsigned), c->stream);
        if (e == hipSuccess) e = hipMemsetAsync(b->fault, 0, sizeof(int), c->stream);
        alloc(&b->step_args, 1);
    }
    if (e == hipSuccess && b->step_grid > 0) {
        const BStep a = bstep_args(c, *b, steps, nseq);
        e = copy_now(c, b->step_args, &a, sizeof(a), hipMemcpyHostToDevice);
    }
    if (e == hipSuccess) e = hipEventCreate(&b->e0);
    if (e == hipSuccess) e = hipEventCreate(&b->e1);
    const size_t state_ints = sizeof(BatchState) / sizeof(int), prompt_ints = (size_t)nseq * pstride, out_ints = (size_t)nseq * steps;
    if (e == hipSuccess) e = hipHostMalloc(reinterpret_cast<void **>(&b->h_pin), (state_ints + prompt_ints + out_ints) * sizeof(int), hipHostMallocDefault);
    if (e == hipSuccess) e = hipFuncSetAttribute((const void *)k_bgemm_f32<1>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)batch_lds_f32(kBatch));
    if (e == hipSuccess) e = hipFuncSetAttribute((const void *)k_bgemm_f32<2>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)batch_lds_f32(kMaxBatch));
    // one position as a graph: every kernel reads the position and the tokens from device memory, so the same nodes serve
    // every step of every call ("graph" = 0: the kernels are launched one by one, for tools that do not follow graph launches)
    if (e == hipSuccess && c->opt[OPT_GRAPH] != 0) {
        e = hipStreamBeginCapture(c->stream, hipStreamCaptureModeThreadLocal);
        if (e == hipSuccess) {
            launch_batch_step(c, *b);
            const hipError_t le = hipGetLastError();
            e = hipStreamEndCapture(c->stream, &b->graph);
            if (e == hipSuccess) e = le;
        }
        if (e == hipSuccess) e = hipGraphInstantiate(&b->exec, b->graph, nullptr, nullptr, 0);
    }
    if (e != hipSuccess) {
        b->release();
        delete b;
        return hip_rc(e, "set-up");
    }
    c->batch = b;
    return L2J_OK;
}

// The samplers of the sequences, as new Sampler(seeds[s], vocab_size) (J/Sampler.java:24-31) leaves them.
int seed_batch_samplers(l2j_ctx *c, BatchBufs &b, const int64_t *seeds)
{
    BatchSamplers &bs = b.samplers;
    if (!bs.ss) {
        const int rc = alloc_batch_samplers(c, b.nseq, &bs);
        if (rc) return rc;
    }
    SamplerState h[kMaxBatch] = {};
    for (int s = 0; s < b.nseq; s++) h[s].rng = ((unsigned long long)seeds[s] ^ kJavaRandMult) & kJavaRandMask;
    HIPCHK(hipMemcpyAsync(bs.ss, h, (size_t)b.nseq * sizeof(SamplerState), hipMemcpyHostToDevice, c->stream));
    for (int i = 0; i < 2; i++) {
        HIPCHK(hipMemsetAsync(bs.pi_prob[i], 0, (size_t)b.nseq * bs.pi_stride * sizeof(float), c->stream));
        HIPCHK(hipMemsetAsync(bs.pi_idx[i], 0, (size_t)b.nseq * bs.pi_stride * sizeof(int), c->stream));
    }
    HIPCHK(hipStreamSynchronize(c->stream));   // (h is pageable host memory)
    return L2J_OK;
}

// Brings the logits of the steps of one call to the caller's memory while later steps are computed, in a thread of its own:
// the copy into memory the caller has just been given (page faults included) takes about as long as a step of a small
// model.  The thread waits for a step on the host: a queue that waits for another one on the device (hipStreamWaitEvent) made the
// 100 kernels of a step 1 us longer each (1745 -> 1853 us per replay of a graph of 100 kernels, 1757 us with the copies alone).
// A process that may not start another thread (std::thread throws) has each step copied by offer() itself.
class LogTaker {
public:
    LogTaker(const BatchBufs &b_, float *out_, size_t step_floats_, int device_) : b(b_), out(out_), step_floats(step_floats_), device(device_)
    {
        if (!out) return;
        try {
            th = std::thread([this] { run(); });
        } catch (const std::exception &) {
        }
    }
    ~LogTaker()
    {
        if (!th.joinable()) return;
        {
            std::lock_guard<std::mutex> l(mu);
            stop = true;
        }
        cv.notify_all();
        th.join();
    }
    // the slot of step `pos` is free (or a copy has failed)
    void wait_slot(int pos)
    {
        std::unique_lock<std::mutex> l(mu);
        cv.wait(l, [&] { return err != hipSuccess || pos - taken < b.log_slots; });
    }
    // log_step of step `pos` has been recorded
    void offer(int pos)
    {
        if (!th.joinable()) {
            if (err == hipSuccess) err = take(pos);
            offered = taken = pos + 1;
            return;
        }
        {
            std::lock_guard<std::mutex> l(mu);
            offered = pos + 1;
        }
        cv.notify_all();
    }
    hipError_t wait_all()
    {
        std::unique_lock<std::mutex> l(mu);
        cv.wait(l, [&] { return err != hipSuccess || taken == offered; });
        return err;
    }

private:
    const BatchBufs &b;
    float *out;
    size_t step_floats;
    int device;
    std::mutex mu;
    std::condition_variable cv;
    int offered = 0, taken = 0;
    bool stop = false;
    hipError_t err = hipSuccess;
    std::thread th;

    hipError_t take(int pos)
    {
        const int slot = pos % b.log_slots;
        hipError_t e = hipEventSynchronize(b.log_step[slot]);
        if (e == hipSuccess) e = hipMemcpyAsync(b.log_pin, b.log_dev + slot * step_floats, step_floats * sizeof(float), hipMemcpyDeviceToHost, b.log_stream);
        if (e == hipSuccess) e = hipStreamSynchronize(b.log_stream);
        if (e == hipSuccess) memcpy(out + (size_t)pos * step_floats, b.log_pin, step_floats * sizeof(float));
        return e;
    }

    void run()
    {
        hipError_t e = hipSetDevice(device);
        for (int i = 0; ; i++) {
            {
                std::unique_lock<std::mutex> l(mu);
                if (e != hipSuccess) err = e;
                else cv.wait(l, [&] { return stop || offered > i; });
                if (err != hipSuccess || offered <= i) {
                    cv.notify_all();
                    return;
                }
            }
            e = take(i);
            {
                std::lock_guard<std::mutex> l(mu);
                if (e == hipSuccess) taken = i + 1;
            }
            cv.notify_all();
        }
    }
};

// logits_log: null, or steps x n_seq x vocab_size floats of the caller that receive the logits of every step.
// seeds: null (every unforced token is the argmax), or the seed of every sequence's sampler: unforced tokens are sampled as
// l2j_sample does at this temperature (not 0) and topp.
int decode_batch(l2j_ctx *c, const int32_t *prompts, const int32_t *n_prompt, int32_t n_seq, int32_t prompt_stride, int32_t steps,
                 int32_t *out_tokens, double *seconds, float *logits_log, float temperature = 0.0f, float topp = 0.0f,
                 const int64_t *seeds = nullptr)
{
    if (!c || !n_prompt || !out_tokens || (prompt_stride > 0 && !prompts) || prompt_stride < 0) return fail(L2J_E_ARG, "bad argument");
    if (!c->finalized) return fail(L2J_E_STATE, "decode before l2j_finalize");
    if (n_seq != kBatch && n_seq != kMaxBatch) return fail(L2J_E_ARG, "n_seq must be 16 or 32");
    const int nseq = n_seq;
    const l2j_config &cf = c->cfg;
    const int hs = c->head_size;
    if (cf.dim % 256 || cf.hidden_dim % 256 || c->kv_dim % 16 || cf.vocab_size % 16 || (hs != 64 && hs != 128 && hs != 256))
        return fail(L2J_E_SIZE, "batched decode needs dim and hidden_dim in whole groups of 256, kv_dim and vocab_size multiples of 16, "
                                "head_size 64, 128 or 256");
    if (steps <= 0 || steps > cf.seq_len) return fail(L2J_E_ARG, "steps must be 1..seq_len");
    for (int b = 0; b < nseq; b++) {
        if (n_prompt[b] < 0 || n_prompt[b] > prompt_stride) return fail(L2J_E_ARG, "n_prompt out of range");
        for (int i = 0; i < n_prompt[b]; i++)
            if (prompts[(size_t)b * prompt_stride + i] < 0 || prompts[(size_t)b * prompt_stride + i] >= cf.vocab_size)
                return fail(L2J_E_ARG, "prompt id out of range");
    }
    HIPCHK(hipSetDevice(cf.device));
    int rc = ensure_batch_tiles(c);   // the matrices once more, in the order the batched products read them
    if (rc) return rc;
    rc = ensure_batch(c, nseq, steps, std::max(1, (int)prompt_stride));
    if (rc) return rc;
    BatchBufs &b = *c->batch;
    const int vocab = cf.vocab_size, cap = b.cap_steps, pcap = b.cap_pstride;
    const size_t state_ints = sizeof(BatchState) / sizeof(int);
    unsigned cur = 0;   // bit s: the copy of its ProbIndex array that sequence s's last top-p step left
    if (seeds && (rc = seed_batch_samplers(c, b, seeds))) return rc;
    const size_t step_floats = (size_t)nseq * vocab;
    if (logits_log) {
        const hipError_t le = b.ensure_log(step_floats, steps);
        if (le != hipSuccess) return hip_rc(le, "logits of every step");
    }
    auto fail_hip = [&](hipError_t e, const char *what) {
        (void)hipStreamSynchronize(c->stream);
        if (b.log_stream) (void)hipStreamSynchronize(b.log_stream);
        return hip_rc(e, what);
    };
    // The positions whose input tokens are known for every sequence (BOS and the shortest prompt) are taken at once, nseq
    // sequences side by side: the weights are read once for up to kRowsMax rows instead of once per position.
    int known = steps;
    for (int i = 0; i < nseq; i++) known = std::min(known, n_prompt[i] + 1);
    if (known < 2 || b.step_grid > 0) known = 0;
    int per = std::min(known, kRowsMax / nseq);
    if (known > 0) {
        // room for the longest common prompt a call on these buffers may have: the next one allocates nothing
        int got = 0;
        rc = ensure_rows(c, std::min({cap, pcap + 1, kRowsMax / nseq}) * nseq, 2 * nseq, &got);
        if (rc == L2J_E_OOM) known = 0;   // (the loop takes these positions as well)
        else if (rc) return rc;
        per = std::min(per, got / nseq);
    }
    BatchState h{};
    h.pos = known > 0 && !logits_log ? known - 1 : 0;
    for (int i = 0; i < nseq; i++) { h.token[i] = 1; h.n_prompt[i] = n_prompt[i]; }   // BOS first (J/Run.java:612)
    h.log = logits_log ? b.log_dev : nullptr;
    h.log_slots = std::max(1, b.log_slots);
    memcpy(b.h_pin, &h, sizeof(h));
    memset(b.h_pin + state_ints, 0, (size_t)nseq * pcap * sizeof(int));
    for (int s = 0; s < nseq && prompt_stride > 0; s++)
        memcpy(b.h_pin + state_ints + (size_t)s * pcap, prompts + (size_t)s * prompt_stride, (size_t)n_prompt[s] * sizeof(int));
    int *h_rows = b.h_pin + state_ints + (size_t)nseq * pcap;   // input tokens of the known positions, position by position
    for (int t = 0; t < known; t++)
        for (int s = 0; s < nseq; s++) h_rows[t * nseq + s] = t == 0 ? 1 : prompts[(size_t)s * prompt_stride + t - 1];
    hipError_t e = hipMemcpyAsync(b.st, b.h_pin, sizeof(h), hipMemcpyHostToDevice, c->stream);
    if (e == hipSuccess) e = hipMemcpyAsync(b.prompts, b.h_pin + state_ints, (size_t)nseq * pcap * sizeof(int), hipMemcpyHostToDevice, c->stream);
    if (e == hipSuccess) e = hipMemsetAsync(b.done, 0, (1 + b.nseq) * sizeof(unsigned), c->stream);
    if (e != hipSuccess) return fail_hip(e, "state upload");
    LogTaker taker(b, logits_log, step_floats, cf.device);
    // after the logits of a position: kept for the caller, and J/Run.java:643-665 for the sequences whose prompt is used up
    // (the sampled token replaces the argmax k_bnext stored)
    auto after_logits = [&](int pos) {
        if (logits_log && e == hipSuccess) {
            e = hipEventRecord(b.log_step[pos % b.log_slots], c->stream);
            if (e == hipSuccess) taker.offer(pos);
        }
        if (seeds && e == hipSuccess) {
            unsigned active = 0;
            for (int s = 0; s < nseq; s++) active |= pos >= n_prompt[s] ? 1u << s : 0u;
            if (active) {
                e = launch_samplers(c, b.samplers, active, cur, b.logits, b.best, kNextParts, temperature, topp, b.st->token, b.out + pos, cap);
                if ((double)topp <= 0.999) cur ^= active;   // (a top-p step leaves the array in its other copy)
            }
        }
    };
    if (known > 0) {
        e = hipEventRecord(b.e0, c->stream);
        RowJob job{};
        job.nseg = nseq;
        job.kc = b.kc; job.vc = b.vc;
        job.seq_stride = (long)cf.n_layers * cap * c->kv_dim; job.layer_stride = (long)cap * c->kv_dim; job.head_stride = (long)cap * hs; job.row_stride = hs;
        for (int t0 = 0; t0 < known && e == hipSuccess; t0 += per) {
            job.pos0 = t0; job.T = std::min(per, known - t0);
            const bool last = t0 + job.T == known;
            job.norm_from = logits_log ? 0 : last ? (job.T - 1) * nseq : job.T * nseq;
            e = hipMemcpyAsync(c->rows.tokens, h_rows + (size_t)t0 * nseq, (size_t)job.T * nseq * sizeof(int), hipMemcpyHostToDevice, c->stream);
            if (e == hipSuccess) e = launch_rows(c, c->rows, job);
            for (int t = logits_log ? 0 : job.T - 1; t < job.T && (logits_log || last) && e == hipSuccess; t++) {
                if (logits_log) taker.wait_slot(t0 + t);
                launch_batch_tokens(c, b, c->rows.xn + (logits_log ? (size_t)t * nseq * cf.dim : 0));
                e = hipGetLastError();
                after_logits(t0 + t);
            }
        }
    }
    for (int pos = known; pos < steps && e == hipSuccess; pos++) {
        if (logits_log) taker.wait_slot(pos);
        if (b.exec) {
            e = hipGraphLaunch(b.exec, c->stream);
        } else {
            launch_batch_step(c, b);
            e = hipGetLastError();
        }
        after_logits(pos);
        if (pos == 0 && e == hipSuccess) e = hipEventRecord(b.e0, c->stream);   // the clock starts after the first step (J/Run.java:682-684)
    }
    if (e == hipSuccess) e = hipEventRecord(b.e1, c->stream);
    if (e == hipSuccess) e = hipMemcpyAsync(b.h_pin, b.out, (size_t)nseq * cap * sizeof(int), hipMemcpyDeviceToHost, c->stream);
    if (logits_log && e == hipSuccess) e = taker.wait_all();
    if (e == hipSuccess) e = hipStreamSynchronize(c->stream);
    if (e != hipSuccess) return fail_hip(e, "step");
    for (int s = 0; s < nseq; s++) {
        memcpy(out_tokens + (size_t)s * steps, b.h_pin + (size_t)s * cap, (size_t)steps * sizeof(int));
        if (known > 1 && !logits_log)   // (the outputs of the known positions but the last are the prompt's ids)
            memcpy(out_tokens + (size_t)s * steps, prompts + (size_t)s * prompt_stride, (size_t)(known - 1) * sizeof(int));
    }
    if (seeds) {   // the reference's exceptions, as in l2j_sample
        SamplerState h[kMaxBatch] = {};
        if ((e = copy_now(c, h, b.samplers.ss, (size_t)nseq * sizeof(SamplerState), hipMemcpyDeviceToHost)) != hipSuccess) return hip_rc(e, "sampler flags");
        int st = 0;
        for (int s = 0; s < nseq; s++) st |= h[s].nan;
        if (st & 1) return fail(L2J_E_ARG, "sampler: NaN among the logits (J/Sampler.java:88-90)");
        if (st & 2) return fail(L2J_E_ARG, "sampler: no probability reaches the top-p cutoff (ArrayIndexOutOfBoundsException at J/Sampler.java:119)");
    }
    if (b.step_grid > 0) {
        int fault = 0;
        if ((e = copy_now(c, &fault, b.fault, sizeof(int), hipMemcpyDeviceToHost)) != hipSuccess) return hip_rc(e, "fault flag");
        if (fault) {
            (void)hipMemsetAsync(b.fault, 0, sizeof(int), c->stream);
            return fail(L2J_E_HIP, "batched decode: a bounded wait at a grid barrier ran out (is another process using the GPU?); "
                                   "option batch_fuse = 0 runs the same step without grid barriers");
        }
    }
    float ms = 0.0f;
    if (steps > 1 && (e = hipEventElapsedTime(&ms, b.e0, b.e1)) != hipSuccess) return hip_rc(e, "timing");
    if (seconds) *seconds = (double)ms * 1e-3;
    return L2J_OK;
}

}  // namespace

extern "C" {

int l2j_release_batch(l2j_ctx *c)
{
    return ctx_rc(c, [&]() -> int {
        std::lock_guard<std::mutex> forward_lock(g_forward_mu);
        if (!c) return fail(L2J_E_ARG, "null context");
        HIPCHK(hipSetDevice(c->cfg.device));
        HIPCHK(hipStreamSynchronize(c->stream));
        std::lock_guard<std::mutex> lock(c->upload_mu);
        free_batch(c);
        return L2J_OK;
    }());
}

int l2j_decode_greedy_batch(l2j_ctx *c, const int32_t *prompts, const int32_t *n_prompt, int32_t n_seq, int32_t prompt_stride,
                            int32_t steps, int32_t *out_tokens, double *seconds)
{
    return ctx_rc(c, [&]() -> int {
        std::lock_guard<std::mutex> forward_lock(g_forward_mu);
        return decode_batch(c, prompts, n_prompt, n_seq, prompt_stride, steps, out_tokens, seconds, nullptr);
    }());
}

int l2j_decode_sample_batch(l2j_ctx *c, const int32_t *prompts, const int32_t *n_prompt, int32_t n_seq, int32_t prompt_stride,
                            int32_t steps, float temperature, float topp, const int64_t *rng_seeds, int32_t *out_tokens, double *seconds,
                            float *logits)
{
    return ctx_rc(c, [&]() -> int {
        std::lock_guard<std::mutex> forward_lock(g_forward_mu);
        const int rc = check_sampler_args(temperature, topp);
        if (rc) return rc;
        if (temperature != 0.0f && !rng_seeds) return fail(L2J_E_ARG, "null argument");
        return decode_batch(c, prompts, n_prompt, n_seq, prompt_stride, steps, out_tokens, seconds, logits, temperature, topp,
                            temperature != 0.0f ? rng_seeds : nullptr);   // (temperature 0: Sampler.argmax, J/Run.java:644-646)
    }());
}

int l2j_decode_greedy_batch_logits(l2j_ctx *c, const int32_t *prompts, const int32_t *n_prompt, int32_t n_seq, int32_t prompt_stride,
                                   int32_t steps, int32_t *out_tokens, float *logits)
{
    return ctx_rc(c, [&]() -> int {
        std::lock_guard<std::mutex> forward_lock(g_forward_mu);
        if (!logits) return fail(L2J_E_ARG, "null argument");
        return decode_batch(c, prompts, n_prompt, n_seq, prompt_stride, steps, out_tokens, nullptr, logits);
    }());
}

}  // extern "C"
