// libllama2j_hip.so: the products with many activation vectors (digit_gemm.hpp) and the forward pass of many positions at
// once: the prompt of one sequence (l2j_prefill), the common prompt positions of a batch.
#include "l2j_internal.hpp"
#include "rows_kernels.hpp"
#include "rows.hpp"

using namespace l2j;

namespace {

// The two shapes of k_dgemm: 256 rows of the matrix x 32 vectors per workgroup, two of which share a compute unit, and
// 512 x 64, one per compute unit.  Microseconds per group of 256: the only workgroup of its compute unit (alone), in a round that
// fills the slots (shared), in the rounds before the last (full); before the first and after the last group (start).  Fitted
// at the products of Llama-2-7B, the full rounds to the same products inside a forward pass of 1024 positions, where the clock is
// lower than in a short burst.  The pick against the best of all launches, over the four products with fifteen numbers of vectors
// from 33 to 1024, mean and largest excess: 110M shape 1.7 and 21 %, 7B 2.4 and 29, 13B 4.7 and 71, 70B widths 1.9 and 77.  (The
// largest: 700 vectors, where the row tiles are dealt unevenly to the eight XCDs and some take a second round, which the
// estimate does not see.)
struct Variant { int pt, nw, per_cu; double alone, shared, full, start; };
constexpr Variant kVariants[2] = {{1, 4, 2, 2.3, 3.8, 4.2, 4.3}, {2, 8, 1, 4.9, 7.2, 7.2, 7.7}};

}  // namespace

// How the product of `tiles16` 16-row tiles (rows of K = 256 ngroups) with `rows` vectors is launched: the variant and the
// groups per slice of K with the smallest estimate: rounds of workgroups over the compute units, and the slices' sums
// written and read again (0.2 us per MB).  It depends on the shape alone, so a shape always adds up in the same order.
DgPlan l2j::dgemm_plan(int n_cu, int tiles16, int ngroups, int rows)
{
    DgPlan best;
    double best_us = 0.0;
    for (int v = 0; v < 2; v++) {
        const Variant &k = kVariants[v];
        const int nrow = (tiles16 + 4 * k.nw - 1) / (4 * k.nw), ncol = (rows + 32 * k.pt - 1) / (32 * k.pt);
        for (int s = 1; s <= std::min(ngroups, max_slices(rows)); s++) {
            const int gps = (ngroups + s - 1) / s;
            if ((ngroups + gps - 1) / gps != s) continue;
            const long wgs = (long)nrow * ncol * s, slots = (long)n_cu * k.per_cu;
            const long full = wgs / slots, rest = wgs % slots;
            double us = full * (gps * k.full + k.start) + 0.2e-6 * s * rows * tiles16 * 64;
            if (rest > 0) {
                const double group = k.per_cu == 2 ? (rest <= n_cu ? k.alone : k.shared) : k.alone + (k.shared - k.alone) * rest / slots;
                us += gps * group + k.start;
            }
            if (best_us == 0.0 || us < best_us) {
                best_us = us;
                best.variant = v; best.gps = gps; best.slices = s; best.nrow = nrow; best.ncol = ncol;
            }
        }
    }
    return best;
}

hipError_t l2j::prepare_dgemm(l2j_ctx *c)
{
    if (c->dgemm_ready) return hipSuccess;
    hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void *>(k_dgemm<1, 4>), hipFuncAttributeMaxDynamicSharedMemorySize, (int)dgemm_lds<1>());
    if (e == hipSuccess) e = hipFuncSetAttribute(reinterpret_cast<const void *>(k_dgemm<2, 8>), hipFuncAttributeMaxDynamicSharedMemorySize, (int)dgemm_lds<2>());
    if (e == hipSuccess) e = hipFuncSetAttribute(reinterpret_cast<const void *>(k_rows_norm<false>), hipFuncAttributeMaxDynamicSharedMemorySize, 128 << 10);
    if (e == hipSuccess) e = hipFuncSetAttribute(reinterpret_cast<const void *>(k_rows_logits), hipFuncAttributeMaxDynamicSharedMemorySize, 128 << 10);
    if (e == hipSuccess) e = hipFuncSetAttribute(reinterpret_cast<const void *>(k_rows_attn<64, 2>), hipFuncAttributeMaxDynamicSharedMemorySize, (int)attn_lds(64, 2));
    if (e == hipSuccess) e = hipFuncSetAttribute(reinterpret_cast<const void *>(k_rows_attn<128, 1>), hipFuncAttributeMaxDynamicSharedMemorySize, (int)attn_lds(128, 1));
    if (e == hipSuccess) e = hipFuncSetAttribute(reinterpret_cast<const void *>(k_rows_attn<128, 2>), hipFuncAttributeMaxDynamicSharedMemorySize, (int)attn_lds(128, 2));
    if (e == hipSuccess) e = hipFuncSetAttribute(reinterpret_cast<const void *>(k_rows_attn<256, 1>), hipFuncAttributeMaxDynamicSharedMemorySize, (int)attn_lds(256, 1));
    if (e == hipSuccess) e = hipFuncSetAttribute(reinterpret_cast<const void *>(k_pflash<64, 16>), hipFuncAttributeMaxDynamicSharedMemorySize, (int)pflash_lds(64, 16));
    if (e == hipSuccess) e = hipFuncSetAttribute(reinterpret_cast<const void *>(k_pflash<128, 16>), hipFuncAttributeMaxDynamicSharedMemorySize, (int)pflash_lds(128, 16));
    if (e == hipSuccess) e = hipFuncSetAttribute(reinterpret_cast<const void *>(k_pflash<256, 8>), hipFuncAttributeMaxDynamicSharedMemorySize, (int)pflash_lds(256, 8));
    c->dgemm_ready = e == hipSuccess;
    return e;
}

// The product of one layer's matrices `tensors` (the same input) with `rows` vectors: (slices, rows, all their rows) into
// part.  Returns the number of slices.
int l2j::launch_dgemm(l2j_ctx *c, std::initializer_list<int> tensors, int layer, const Digits &x, int rows, float *part)
{
    DGemm a{};
    int K = 0, m = 0;
    for (int tensor : tensors) {
        int n = 0;
        matrix_shape(c->cfg, tensor, &n, &K);
        const uint64_t off = (uint64_t)layer * n * K;
        a.codes[m] = c->bt_codes[tensor] + off;
        a.gs[m] = c->bt_gs[tensor] + off / 256;
        a.tiles[m] = n / 16;
        a.ntiles += n / 16;
        m++;
    }
    a.ngroups = K / 256;
    a.x = x; a.npos = rows; a.out = part;
    for (int i = m; i < 3; i++) { a.codes[i] = a.codes[0]; a.gs[i] = a.gs[0]; }
    if (streams(a.ntiles, rows)) {
        const int slices = stream_slices(a.ngroups), share = std::max(1, c->n_cu / slices), ntile = a.ntiles / 2, iters = (ntile + share - 1) / share;
        a.gps = (a.ngroups + slices - 1) / slices;
        const dim3 grid((ntile + iters - 1) / iters, slices);
        const dim3 block(64 * kStreamWaves);
        if (rows <= 16 && iters == 1) hipLaunchKernelGGL((k_dstream<1, 1>), grid, block, dstream_lds<1>(), c->stream, a);
        else if (rows <= 16 && iters == 2) hipLaunchKernelGGL((k_dstream<1, 2>), grid, block, dstream_lds<1>(), c->stream, a);
        else if (rows <= 16) hipLaunchKernelGGL((k_dstream<1, 0>), grid, block, dstream_lds<1>(), c->stream, a);
        else if (iters == 1) hipLaunchKernelGGL((k_dstream<2, 1>), grid, block, dstream_lds<2>(), c->stream, a);
        else hipLaunchKernelGGL((k_dstream<2, 0>), grid, block, dstream_lds<2>(), c->stream, a);
        return slices;
    }
    const DgPlan p = dgemm_plan(c->n_cu, a.ntiles, a.ngroups, rows);
    a.gps = p.gps; a.ncol = p.ncol; a.nrow = p.nrow;
    const dim3 grid((unsigned)((p.nrow * p.slices + 7) / 8 * 8 * p.ncol));
    if (p.variant == 0) hipLaunchKernelGGL((k_dgemm<1, 4>), grid, dim3(256), dgemm_lds<1>(), c->stream, a);
    else hipLaunchKernelGGL((k_dgemm<2, 8>), grid, dim3(512), dgemm_lds<2>(), c->stream, a);
    return p.slices;
}

// The number of slices a product with these vectors leaves.
int l2j::product_slices(l2j_ctx *c, int tiles16, int ngroups, int rows)
{
    return streams(tiles16, rows) ? stream_slices(ngroups) : dgemm_plan(c->n_cu, tiles16, ngroups, rows).slices;
}

void l2j::launch_norm(l2j_ctx *c, const RowNorm &n, int rows)
{
    const int threads = std::min(1024, std::max(64, n.dim / 4));
    RowNorm a = n;
    a.together = rows >= kTogetherFrom && !n.xn ? rows : 0;
    const dim3 grid(a.together ? together_grid(rows, 1) : rows);
    if (n.per_slice > 0) hipLaunchKernelGGL(k_rows_norm<true>, grid, dim3(threads), (size_t)n.dim * sizeof(float), c->stream, a);
    else hipLaunchKernelGGL(k_rows_norm<false>, grid, dim3(threads), (size_t)n.dim * sizeof(float), c->stream, a);
}

static void launch_swiglu(l2j_ctx *c, const float *part, int slices, const Digits &o, int rows)
{
    const int hidden = c->cfg.hidden_dim, parts = (hidden + 1023) / 1024, together = rows >= kTogetherFrom;
    const dim3 grid = together ? dim3(together_grid(rows, parts)) : dim3(parts, rows);
    hipLaunchKernelGGL(k_rows_swiglu, grid, dim3(256), 0, c->stream, part, slices, o, rows, hidden, c->silu, (c->cfg.flags & L2J_F_EXACT_SILU) ? 1 : 0, together);
}

// W1 and W3 of the normed rows in b.dig, SwiGLU, W2: the slices in b.part, n.slices and n.per_slice what k_rows_norm then adds up.
void l2j::launch_ffn(l2j_ctx *c, int layer, const RowBufs &b, int rows, RowNorm &n)
{
    const int dim = c->cfg.dim, hidden = c->cfg.hidden_dim;
    n.per_slice = 0;
    if (!swiglu_in_products(c->n_cu, dim, hidden, rows)) {
        const int s13 = launch_dgemm(c, {L2J_W1, L2J_W3}, layer, b.dig, rows, b.part);
        launch_swiglu(c, b.part, s13, b.dig, rows);
        n.slices = launch_dgemm(c, {L2J_W2}, layer, b.dig, rows, b.part);
        return;
    }
    const uint64_t off = (uint64_t)layer * dim * hidden;
    DGemm a{};
    a.codes[0] = c->bt_codes[L2J_W1] + off; a.codes[1] = c->bt_codes[L2J_W3] + off; a.codes[2] = a.codes[0];
    a.gs[0] = c->bt_gs[L2J_W1] + off / 256; a.gs[1] = c->bt_gs[L2J_W3] + off / 256; a.gs[2] = a.gs[0];
    a.tiles[0] = a.tiles[1] = hidden / 16; a.ntiles = 2 * (hidden / 16);
    a.ngroups = a.gps = dim / 256;
    a.x = b.dig; a.npos = rows; a.out = b.act;
    a.silu = c->silu; a.exact = (c->cfg.flags & L2J_F_EXACT_SILU) ? 1 : 0;
    W2Rows d{};
    d.x = b.act; d.npos = rows; d.hidden = hidden; d.dim = dim;
    d.codes = c->bt_codes[L2J_W2] + off; d.gs = c->bt_gs[L2J_W2] + off / 256;
    d.out = b.part;
    const dim3 grid(dim / 32, hidden / 256);
    if (rows <= 16) {
        hipLaunchKernelGGL((k_dstream<1, 1, true>), dim3(hidden / 16), dim3(64 * kStreamWaves), dstream_lds<1>(), c->stream, a);
        hipLaunchKernelGGL(k_w2_rows<1>, grid, dim3(256), 0, c->stream, d);
    } else {
        hipLaunchKernelGGL((k_dstream<2, 1, true>), dim3(hidden / 16), dim3(64 * kStreamWaves), dstream_lds<2>(), c->stream, a);
        hipLaunchKernelGGL(k_w2_rows<2>, grid, dim3(512), 0, c->stream, d);
    }
    const int groups = hidden / 256, slices = stream_slices(groups);
    n.slices = 2 * groups;
    n.per_slice = 2 * ((groups + slices - 1) / slices);
}

void RowBufs::release()
{
    void *ps[] = {x, part, act, q, xb, xn, dig.d, dig.sx, dig.sum, tokens, pf_part, pf_cnt};
    for (void *p : ps) (void)hipFree(p);
    *this = RowBufs();
}

// Room for `rows` rows.  attention: also what the passes of many positions need.
hipError_t RowBufs::alloc(l2j_ctx *c, int rows, bool attention)
{
    const l2j_config &cf = c->cfg;
    const size_t dim = cf.dim, hidden = cf.hidden_dim, kvd = c->kv_dim, tiles = 2 * ((digit_tiles(rows) + 1) / 2);   // (whole workgroups of 64 rows)
    const size_t groups = std::max(dim, hidden) / 256;
    hipError_t e = hipSuccess;
    auto get = [&](auto **p, size_t n) {
        if (e == hipSuccess) e = hipMalloc(reinterpret_cast<void **>(p), n * sizeof(**p));
    };
    cap = rows;
    get(&x, rows * dim);
    get(&xn, rows * dim);
    get(&part, (size_t)max_slice_rows(rows, (int)groups) * std::max(2 * hidden, dim + 2 * kvd));
    if (swiglu_in_products(c->n_cu, cf.dim, cf.hidden_dim, 1)) get(&act, std::min(rows, kRowTile) * (hidden + hidden / 16));
    get(&dig.d, tiles * groups * (kDigitBytes / 16));
    get(&dig.sx, tiles * groups * 32);
    get(&dig.sum, tiles * groups * 32);
    if (attention) {
        get(&q, rows * dim);
        get(&xb, rows * dim);
        get(&tokens, (size_t)rows);
    }
    if (e != hipSuccess) release();
    return e;
}

// Blocks of 32 positions (the cache rows loaded once for 32) where pairs of blocks of 16 are an eighth more workgroups than compute
// units: a last round of them costs more than half-filled compute units do.  7B shape, us a launch with blocks of 16 -> 32: 520
// positions 58.6 -> 71.0 (272 pairs of blocks of 16: just past the 256 units), 560 76.4 -> 69.0 (288), 700 88.2 -> 79.5, 900 110.8 ->
// 100.1; whole passes of 1024 positions, four layers, ms: 7B 3.81 -> 3.77, 13B 5.91 -> 6.04, 70B widths 13.15 -> 13.10.
// Pairs of blocks unless one block per workgroup already leaves compute units idle.
template <int HS>
static void launch_attn(l2j_ctx *c, RowAttn t)
{
    const int units = c->cfg.n_heads / (256 / HS) * t.nseg;
    auto blocks = [&](int q) { return (t.T + q - 1) / q; };
    const bool two = HS < 256 && t.T > 16 && 8L * ((blocks(16) + 1) / 2) * units >= 9L * c->n_cu;
    const int n = blocks(two ? 32 : 16);
    t.paired = n * units > c->n_cu;
    const dim3 g((t.paired ? (n + 1) / 2 : n) * units), blk(64 * attn_waves(HS));
    if (two) hipLaunchKernelGGL((k_rows_attn<HS, HS < 256 ? 2 : 1>), g, blk, attn_lds(HS, 2), c->stream, t);
    else hipLaunchKernelGGL((k_rows_attn<HS, 1>), g, blk, attn_lds(HS, 1), c->stream, t);
}

// How the attention of T positions is launched: the keys of a block of 16 positions dealt to the waves of a workgroup (k_pflash,
// split: and to so many workgroups) where there are few blocks over many keys, else a wave per block (k_rows_attn).
struct RowAttnPlan { bool shared; int nqb, split; };

static RowAttnPlan attn_plan(const l2j_ctx *c, const RowJob &job, int T, int keys)
{
    RowAttnPlan p;
    p.nqb = (T + 15) / 16;
    p.split = 1;
    const int flash = c->opt[OPT_PREFILL_FLASH], heads = c->cfg.n_heads;
    const long waves = (long)heads * job.nseg * p.nqb;   // of a wave per block
    const bool far = (long)keys * job.row_stride > UINT32_MAX;   // (past the 32-bit offsets of k_rows_attn)
    p.shared = job.nseg == 1 && (far || (flash != 0 && (flash == 2 || (keys >= kSharedKeysFrom && waves < kSharedKeysBelow * c->n_cu))));
    const int opt = c->opt[OPT_PREFILL_SPLIT];
    if (p.shared && (opt > 0 || keys >= kSplitKeysFrom)) p.split = std::min(kPflashMaxSplit, std::max(1, opt > 0 ? opt : c->n_cu / (p.nqb * heads)));
    return p;
}

// The forward passes of job.T positions of job.nseg sequences: their k and v rows are left in the cache and, from row
// job.norm_from on (a whole position), the rows after the final norm in b.xn.
// Behind its keys and values the last layer is for those rows alone: nothing else reads the others.  (A layer in
// 32 of the 7B shape: 77 positions 7.06 -> 6.95 ms, 1024 positions 32.14 -> 31.49.)
hipError_t l2j::launch_rows(l2j_ctx *c, RowBufs &b, const RowJob &job)
{
    const l2j_config &cf = c->cfg;
    const int dim = cf.dim, L = cf.n_layers, hs = c->head_size, kvd = c->kv_dim, keys = job.pos0 + job.T;
    int rows = job.nseg * job.T, T = job.T;
    hipStream_t s = c->stream;
    const int first = std::min(job.norm_from / job.nseg, T);   // position from which on rows are wanted
    RowAttnPlan ap = attn_plan(c, job, T, keys), ap_last = attn_plan(c, job, std::max(1, T - first), keys);
    const int blocks = std::max(ap.split > 1 ? ap.nqb : 0, ap_last.split > 1 ? ap_last.nqb : 0);
    if (b.pf_blocks < blocks) {
        (void)hipFree(b.pf_part);
        (void)hipFree(b.pf_cnt);
        b.pf_part = nullptr; b.pf_cnt = nullptr; b.pf_blocks = 0;
        hipError_t e = hipMalloc(reinterpret_cast<void **>(&b.pf_part), (size_t)cf.n_heads * blocks * kPflashMaxSplit * (32 + 16 * hs) * sizeof(float));
        if (e == hipSuccess) e = hipMalloc(reinterpret_cast<void **>(&b.pf_cnt), (size_t)cf.n_heads * blocks * sizeof(unsigned));
        if (e == hipSuccess) e = hipMemsetAsync(b.pf_cnt, 0, (size_t)cf.n_heads * blocks * sizeof(unsigned), s);
        if (e == hipErrorOutOfMemory) {   // (the keys of a block in one workgroup then)
            (void)hipGetLastError();
            ap.split = ap_last.split = 1;
        } else if (e != hipSuccess) {
            return e;
        } else {
            b.pf_blocks = blocks;
        }
    }
    const int qkv_parts = std::min((dim + 2 * kvd + 1023) / 1024, std::max(1, 4 * c->n_cu / rows));   // (few rows: their columns over several workgroups)
    RowNorm n{};
    n.emb = c->emb; n.nrows = rows; n.x = b.x; n.dim = dim; n.dig = b.dig;
    n.tokens = b.tokens; n.w = c->rmsw;
    launch_norm(c, n, rows);
    n.tokens = nullptr;
    n.part = b.part;
    for (int l = 0; l < L; l++) {
        RowQkv k{};
        k.slices = launch_dgemm(c, {L2J_WQ, L2J_WK, L2J_WV}, l, b.dig, rows, b.part);
        k.part = b.part; k.nrows = rows; k.nseg = job.nseg; k.pos0 = job.pos0; k.rope = c->rope; k.q = b.q;
        k.kc = job.kc + l * job.layer_stride; k.vc = job.vc + l * job.layer_stride;
        k.seq_stride = job.seq_stride; k.head_stride = job.head_stride; k.row_stride = job.row_stride;
        k.dim = dim; k.kv_dim = kvd; k.head_size = hs;
        hipLaunchKernelGGL(k_rows_qkv, dim3(rows, qkv_parts), dim3(256), 0, s, k);
        const float *q = b.q;
        int pos0 = job.pos0;
        if (l + 1 == L) {   // the wanted positions alone, as rows from 0 on
            T -= first; rows = job.nseg * T; pos0 += first;
            if (rows == 0) break;
            q += (size_t)job.nseg * first * dim;
            n.x += (size_t)job.nseg * first * dim; n.nrows = rows;
            ap = ap_last;
        }
        RowAttn t{};
        t.q = q; t.kc = k.kc; t.vc = k.vc; t.seq_stride = k.seq_stride; t.head_stride = k.head_stride; t.row_stride = k.row_stride;
        t.out = b.xb; t.nseg = job.nseg; t.T = T; t.pos0 = pos0; t.n_heads = cf.n_heads; t.kv_mul = c->kv_mul; t.dim = dim;
        t.dig = b.dig; t.sqrt_hs = sqrtf((float)hs); t.pf_part = b.pf_part; t.pf_cnt = b.pf_cnt;
        if (ap.shared) {
            const dim3 g(cf.n_heads, ap.nqb, ap.split);
            if (hs == 64) hipLaunchKernelGGL((k_pflash<64, 16>), g, dim3(1024), pflash_lds(64, 16), s, t);
            else if (hs == 128) hipLaunchKernelGGL((k_pflash<128, 16>), g, dim3(1024), pflash_lds(128, 16), s, t);
            else hipLaunchKernelGGL((k_pflash<256, 8>), g, dim3(512), pflash_lds(256, 8), s, t);
            hipLaunchKernelGGL(k_rows_digits, dim3((unsigned)(((long)rows * (dim / 16) + 255) / 256)), dim3(256), 0, s, b.xb, b.dig, rows, dim);
        } else if (hs == 64) {
            launch_attn<64>(c, t);
        } else if (hs == 128) {
            launch_attn<128>(c, t);
        } else {
            launch_attn<256>(c, t);
        }
        n.slices = launch_dgemm(c, {L2J_WO}, l, b.dig, rows, b.part);
        n.per_slice = 0;
        n.w = c->rmsw + (size_t)(L + l) * dim;
        launch_norm(c, n, rows);
        launch_ffn(c, l, b, rows, n);
        // the residual, then the norm of what follows: the next layer's attention norm, or the final one (rmsw: att, ffn, final)
        if (l + 1 < L) {
            n.w = c->rmsw + (size_t)(l + 1) * dim;
            launch_norm(c, n, rows);
        } else {
            RowNorm f = n;
            f.w = c->rmsw + (size_t)2 * L * dim; f.xn = b.xn;
            launch_norm(c, f, rows);
        }
    }
    return hipGetLastError();
}

// Room in the context's buffers for passes of `rows` rows, or, where the device memory does not suffice, of half as many and so
// on down to `least` (passes of many rows are faster, but nothing needs them): *got, at most rows.
int l2j::ensure_rows(l2j_ctx *c, int rows, int least, int *got)
{
    const int rc = ensure_batch_tiles(c);
    if (rc) return rc;
    HIPCHK(prepare_dgemm(c));
    if (c->rows.cap < rows) {
        HIPCHK(hipStreamSynchronize(c->stream));
        c->rows.release();
        hipError_t e;
        for (int n = rows; (e = c->rows.alloc(c, n, true)) == hipErrorOutOfMemory; n = std::max(least, n / 2)) {
            (void)hipGetLastError();   // (or the next launch would report it)
            if (n <= least) break;
        }
        HIPCHK(e);
    }
    *got = std::min(rows, c->rows.cap);
    return L2J_OK;
}

// ---- l2j_prefill ----------------------------------------------------------------------------------------------------

int l2j::prefill_positions(l2j_ctx *c, const int32_t *tokens, int32_t n, int32_t pos0, float *logits, double *seconds, bool keep_logits)
{
    if (!c || !tokens) return fail(L2J_E_ARG, "null argument");
    if (!c->finalized) return fail(L2J_E_STATE, "prefill before l2j_finalize");
    const l2j_config &cf = c->cfg;
    const int hs = c->head_size, kvd = c->kv_dim;
    if (cf.dim % 256 || cf.hidden_dim % 256 || kvd % 16 || cf.vocab_size % 16 || (hs != 64 && hs != 128 && hs != 256))
        return fail(L2J_E_SIZE, "prefill needs dim and hidden_dim in whole groups of 256, kv_dim and vocab_size multiples of 16, "
                                "head_size 64, 128 or 256 (as the batched decode); take l2j_forward position by position");
    if (n <= 0 || pos0 < 0 || (long)pos0 + n > cf.seq_len) return fail(L2J_E_ARG, "positions pos0 .. pos0 + n - 1 must lie in 0 .. seq_len - 1");
    for (int i = 0; i < n; i++)
        if (tokens[i] < 0 || tokens[i] >= cf.vocab_size) return fail(L2J_E_ARG, "token id out of range");
    HIPCHK(hipSetDevice(cf.device));
    // passes of at most kRowsMax positions, as even as they come
    auto even = [&](int most) { const int npass = (n + most - 1) / most; return (n + npass - 1) / npass; };
    int got = 0;
    const int rc = ensure_rows(c, even(kRowsMax), std::min(n, kRowTile), &got);
    if (rc) return rc;
    const int per = even(got);
    RowBufs &b = c->rows;
    while ((int)c->events.size() < 2) {
        hipEvent_t ev;
        HIPCHK(hipEventCreate(&ev));
        c->events.push_back(ev);
    }
    RowJob job{};
    job.nseg = 1;
    job.kc = c->kcache; job.vc = c->vcache;
    job.layer_stride = (long)cf.seq_len * kvd; job.head_stride = hs; job.row_stride = kvd;   // (position, kv_dim) per layer
    for (int i = 0; i < n; i += per) {
        const int T = std::min(per, n - i);
        const bool last = i + T == n && keep_logits;
        if (i > 0) HIPCHK(hipStreamSynchronize(c->stream));   // (the staging memory is in use until the copy before is done)
        memcpy(c->h_tokens, tokens + i, (size_t)T * sizeof(int));
        HIPCHK(hipMemcpyAsync(b.tokens, c->h_tokens, (size_t)T * sizeof(int), hipMemcpyHostToDevice, c->stream));
        if (i == 0) HIPCHK(hipEventRecord(c->events[0], c->stream));
        job.T = T; job.pos0 = pos0 + i;
        job.norm_from = last ? T - 1 : T;   // the logits of the last position alone are wanted
        HIPCHK(launch_rows(c, b, job));
    }
    if (keep_logits) hipLaunchKernelGGL(k_rows_logits, dim3(8 * c->n_cu), dim3(256), (size_t)cf.dim * sizeof(float), c->stream, c->wcls, b.xn, c->logits, cf.dim, cf.vocab_size);
    HIPCHK(hipGetLastError());
    HIPCHK(hipEventRecord(c->events[1], c->stream));
    if (logits) HIPCHK(hipMemcpyAsync(logits, c->logits, (size_t)cf.vocab_size * sizeof(float), hipMemcpyDeviceToHost, c->stream));
    HIPCHK(hipStreamSynchronize(c->stream));
    float ms = 0.0f;
    HIPCHK(hipEventElapsedTime(&ms, c->events[0], c->events[1]));
    if (seconds) *seconds = (double)ms * 1e-3;
    return L2J_OK;
}

extern "C" {

int l2j_prefill(l2j_ctx *c, const int32_t *tokens, int32_t n, int32_t pos0, float *logits, double *seconds)
{
    return ctx_rc(c, [&]() -> int {
        std::lock_guard<std::mutex> forward_lock(g_forward_mu);
        return prefill_positions(c, tokens, n, pos0, logits, seconds);
    }());
}

}  // extern "C"
