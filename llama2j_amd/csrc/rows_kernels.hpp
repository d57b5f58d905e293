// Many positions in one pass over the weights: the kernels between the products of digit_gemm.hpp.  A row is one position
// of one sequence: row = t * nseg + seg is position pos0 + t of sequence seg (a prompt: nseg = 1; the prompts of a batch
// side by side: nseg sequences).
#pragma once

#include "batch_kernels.hpp"
#include "digit_gemm.hpp"

namespace l2j {

__device__ __forceinline__ void load16(const float *p, float (&v)[16])
{
#pragma unroll
    for (int q = 0; q < 4; q++) {
        const v4f f = reinterpret_cast<const v4f *>(p)[q];
#pragma unroll
        for (int e = 0; e < 4; e++) v[4 * q + e] = f[e];
    }
}

// Eight rows of a group of 256 share the 128-byte lines of its digits, 16 bytes each.  With `together` the workgroups of
// eight such rows run on one XCD (blockIdx % 8), one after the other, and its L2 puts the lines together; workgroup `id`
// takes row `row` of part `part` of `nparts` of the columns.  (A workgroup per row in order has the pieces of a line written
// through eight L2s.  7B shape, us, in order -> together, at 256 / 448 / 700 / 1024 rows: SwiGLU 14.5 / 23.1 / 33.2 / 48.7 -> 11.1 /
// 17.0 / 23.2 / 31.4; norm 8.2 / 12.4 / 16.3 / 23.1 -> 8.0 / 10.7 / 13.6 / 17.7.)
__host__ __device__ inline unsigned together_grid(int rows, int nparts) { return (unsigned)(((rows + 7) / 8 * nparts + 7) / 8 * 64); }

__device__ __forceinline__ void together_row(int id, int nparts, int *row, int *part)
{
    const int j = id >> 3, unit = (j >> 3) * 8 + (id & 7);
    *part = unit % nparts;
    *row = unit / nparts * 8 + (j & 7);
}

struct RowNorm {
    const float *emb;       // with tokens: the row's x is its token's row of the table (J/Run.java:72)
    const int *tokens;
    const float *part;      // else: x += the slices of a product (K/Accum.java:26-30)
    int slices, nrows;      // nrows: rows of the product's output
    int per_slice;          // 0, or part holds that many sums of each slice (of the last one what is left), `slices` in all (k_w2_rows)
    int together;           // 0: a workgroup per row in order, else the number of rows (together_row)
    float *x;               // (rows, dim)
    const float *w;         // norm weights
    int dim;
    Digits dig;             // the normed row as digits,
    float *xn;              // or, not null, as floats
};

// The slices of k_w2_rows: the sums of a slice are added up first, as k_dstream does within a workgroup.  At most 2 slices, n <= N sums, all
// loads in flight.
template <int N>
__device__ __forceinline__ v4f sum_in_slices(const float *__restrict__ part, int n, int per_slice, size_t stride)
{
    v4f v[N], t = {}, y;
#pragma unroll
    for (int i = 0; i < N; i++) v[i] = *reinterpret_cast<const v4f *>(part + min(i, n - 1) * stride);
    y = v[0];
#pragma unroll
    for (int i = 1; i < N; i++) {
        if (i < n) {
            if (i == per_slice) { t += y; y = v[i]; }
            else y += v[i];
        }
    }
    return t + y;
}

// x, then w * (ss * x), ss = 1 / sqrt(sum(x^2) / n + 1e-5) (K/RootMeanSquare.java:25-35, K/WeightNormalizeAndScale.java:73).
// One workgroup per row, four values per thread and step of 4096, kept in LDS (dim floats, each thread its own): a wave
// holds whole groups of 256 and writes their digits.  Bound by its chain of latencies (slices, sum over the workgroup,
// digits): the loads of the slices and of the first weights go out together.  32 rows of 4096 behind 4 or 11 slices
// 6.7 us, 13 of 768 behind 1 or 2 slices 3.5 (7.4 and 4.0 when sixteen lanes per group wrote the digits behind another barrier
// and the slices came four at a time).
// W2ROWS: the slices are those of k_w2_rows.
template <bool W2ROWS>
static __global__ void __launch_bounds__(1024) k_rows_norm(const RowNorm a)
{
    extern __shared__ __align__(16) float ln[];
    __shared__ float red[16];
    int row = blockIdx.x, part0 = 0;
    if (a.together) {
        together_row(blockIdx.x, 1, &row, &part0);
        if (row >= a.together) return;
    }
    const int tid = threadIdx.x, n4 = a.dim >> 2, nt = blockDim.x;
    v4f *x = reinterpret_cast<v4f *>(a.x + (size_t)row * a.dim), *l4 = reinterpret_cast<v4f *>(ln);
    const v4f *e = a.tokens ? reinterpret_cast<const v4f *>(a.emb + (size_t)a.tokens[row] * a.dim) : nullptr;
    const float *part = a.part + (size_t)row * a.dim;
    const size_t stride = (size_t)a.nrows * a.dim;
    const v4f *w = reinterpret_cast<const v4f *>(a.w);
    v4f w0 = w[tid];   // (no more threads than n4)
    float ssq = 0.0f;
    for (int i = tid; i < n4; i += nt) {
        v4f v;
        if (e) {
            v = e[i];
        } else {
            v = x[i];
            v4f t;
            if constexpr (!W2ROWS) t = sum_slices<v4f>(part + 4 * i, a.slices, stride);
            else if (a.slices <= 8) t = sum_in_slices<8>(part + 4 * i, a.slices, a.per_slice, stride);
            else t = sum_in_slices<16>(part + 4 * i, a.slices, a.per_slice, stride);
#pragma unroll
            for (int k = 0; k < 4; k++) v[k] = __fadd_rn(v[k], t[k]);
        }
        x[i] = v;
        l4[i] = v;
        ssq += (v[0] * v[0] + v[1] * v[1]) + (v[2] * v[2] + v[3] * v[3]);
    }
    ssq = block_sum(ssq, red, nt >> 6);
    const float ss = __fdiv_rn(1.0f, __fsqrt_rn(__fadd_rn(__fdiv_rn(ssq, (float)a.dim), 1e-5f)));
    for (int i = tid; i < n4; i += nt) {   // (each thread its own values; whole waves leave together: n4 % 64 == 0)
        if (i != tid) w0 = w[i];
        v4f v = l4[i];
#pragma unroll
        for (int k = 0; k < 4; k++) v[k] = __fmul_rn(w0[k], __fmul_rn(ss, v[k]));
        if (a.xn) reinterpret_cast<v4f *>(a.xn + (size_t)row * a.dim)[i] = v;
        else quantize_wave(a.dig, row, a.dim >> 8, i >> 6, tid & 63, v);
    }
}

struct RowQkv {
    const float *part;       // (slices, rows, dim + 2 kv_dim)
    int slices, nrows, nseg, pos0;
    const float2 *rope;      // (seq_len, head_size / 2) cos, sin
    float *q;                // (rows, dim)
    float *kc, *vc;          // + seg * seq_stride + kv head * head_stride + position * row_stride
    long seq_stride, head_stride, row_stride;
    int dim, kv_dim, head_size;
};

// q, k and v of a row: the slices added up, RoPE on the pairs of q and k (K/ApplyRope.java:74-90), k and v into the cache row
// (J/Run.java:95-99).  grid (rows, parts of the columns), two pairs per thread and step.
static __global__ void __launch_bounds__(256) k_rows_qkv(const RowQkv a)
{
    const int row = blockIdx.x, seg = row % a.nseg, pos = a.pos0 + row / a.nseg, cols = a.dim + 2 * a.kv_dim, hs = a.head_size;
    const size_t stride = (size_t)a.nrows * cols;
    const float *part = a.part + (size_t)row * cols;
    const float4 *rope = reinterpret_cast<const float4 *>(a.rope + (size_t)pos * (hs >> 1));
    for (int c = 4 * (threadIdx.x + 256 * blockIdx.y); c < cols; c += 1024 * gridDim.y) {
        const v4f t = sum_slices<v4f>(part + c, a.slices, stride);
        float4 v = make_float4(t[0], t[1], t[2], t[3]);
        const bool isq = c < a.dim, isk = !isq && c < a.dim + a.kv_dim;
        const int at = isq ? c : c - a.dim - (isk ? 0 : a.kv_dim);
        const int head = at / hs, idx = at - head * hs;
        if (isq || isk) {
            const float4 cs = rope[idx >> 2];
            const float r0 = __fsub_rn(__fmul_rn(v.x, cs.x), __fmul_rn(v.y, cs.y)), r1 = __fadd_rn(__fmul_rn(v.x, cs.y), __fmul_rn(v.y, cs.x));
            const float r2 = __fsub_rn(__fmul_rn(v.z, cs.z), __fmul_rn(v.w, cs.w)), r3 = __fadd_rn(__fmul_rn(v.z, cs.w), __fmul_rn(v.w, cs.z));
            v = make_float4(r0, r1, r2, r3);
        }
        float *o = isq ? a.q + (size_t)row * a.dim + c
                       : (isk ? a.kc : a.vc) + seg * a.seq_stride + head * a.head_stride + pos * a.row_stride + idx;
        *reinterpret_cast<float4 *>(o) = v;
    }
}

// (rows, K) floats as digits: sixteen values per thread.
static __global__ void __launch_bounds__(256) k_rows_digits(const float *__restrict__ x, Digits o, int rows, int K)
{
    const long i = (long)blockIdx.x * 256 + threadIdx.x;
    const int nc = K >> 4;
    if (i >= (long)rows * nc) return;   // (whole groups: sixteen lanes leave together)
    const int row = (int)(i / nc), c = (int)(i - (long)row * nc);
    float v[16];
    load16(x + (size_t)row * K + 16 * c, v);
    quantize_group(o, row, K >> 8, c >> 4, c & 15, v);
}

// silu(h1) * h3 with the reference's sigmoid table (K/Silu.java:72-74) as digits; part: (slices, rows, 2 hidden), h1 | h3.
// Workgroup (x, row), or together_row: four groups of 256, one per wave, four values per thread.
static __global__ void __launch_bounds__(256) k_rows_swiglu(const float *__restrict__ part, int slices, Digits o, int rows, int hidden,
                                                     const float *__restrict__ silu, int exact, int together)
{
    int row = blockIdx.y, cpart = blockIdx.x;
    if (together) together_row(blockIdx.x, (hidden + 1023) / 1024, &row, &cpart);
    const int col = cpart * 1024 + 4 * threadIdx.x;
    if (row >= rows || col >= hidden) return;   // (whole waves: hidden % 256 == 0)
    const size_t stride = (size_t)rows * 2 * hidden;
    const float *p = part + (size_t)row * 2 * hidden + col;
    const v4f h1 = sum_slices<v4f>(p, slices, stride), h3 = sum_slices<v4f>(p + hidden, slices, stride);
    v4f y;
#pragma unroll
    for (int e = 0; e < 4; e++) y[e] = __fmul_rn(h1[e], __fmul_rn(silu_sigma(silu, h1[e], exact), h3[e]));
    quantize_wave(o, row, hidden >> 8, col >> 8, threadIdx.x & 63, y);
}

// The product W2 for at most 16 NB vectors of floats, where a workgroup has one tile of 32 rows and one group of K: there a launch is its way
// in and out, and forming the group's digits once per tile costs less than a launch that stores them.
// A lane holds 16 consecutive activations of the vector and the k at which the matrix instruction takes them from it, so
// the digits never leave its registers: wave (T, m) has the 64 k of block T for vectors 16 m .. 16 m + 15, and only the groups' maxima
// and sums cross the waves.  The blocks' sums meet in LDS as integers.  What leaves are the sums of a group's two halves, each
// scaled for itself, and k_rows_norm adds them up slice by slice: bit for bit what k_rows_swiglu and k_dstream give, so that no result depends on
// which of the two ways a shape or a number of rows takes.
// Bound by its chain of latencies (activations, two barriers, codes); with SwiGLU at the end of W1 and W3 a layer takes 1.1 to 1.7 us less at
// 16 vectors and 1.5 to 2.3 at 32 than with a launch in between.  (One sum per group, of all 256 k at once, was 1.3 us a layer of the
// 110M shape less still, but rounded elsewhere: plain-sampled batches got other tokens.)
// grid (rows of W2 / 32, groups), 256 NB threads; out: (half of a group, vector, row of W2); vectors past npos count as zeros.
struct W2Rows {
    const float *x;          // (npos, hidden), behind it the sums of 16 consecutive ones (npos, hidden / 16)
    int npos, hidden, dim;
    const uint8_t *codes;    // W2 of the layer in tile order (DGemm)
    const float2 *gs;
    float *out;
};

template <int NB>
static __global__ void __launch_bounds__(256 * NB) k_w2_rows(const W2Rows a)
{
    __shared__ v4i red[2][4][2 * NB][64];   // high and low sums; block of 64 k; vectors and rows
    __shared__ unsigned s_max[4][16 * NB];
    __shared__ float s_sum[4][16 * NB], s_inv[16 * NB], s_tot[16 * NB];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), T = wave & 3, m = wave >> 2, n = lane & 15;
    const int tile = blockIdx.x, g = blockIdx.y, ngroups = a.hidden >> 8, row = 16 * m + n;
    const float *p = a.x + (size_t)min(row, a.npos - 1) * a.hidden + 256 * g + 64 * T + 16 * (lane >> 4);
    v4f v[4];
#pragma unroll
    for (int i = 0; i < 4; i++) v[i] = *reinterpret_cast<const v4f *>(p + 4 * i);
    float sum = a.x[(size_t)a.npos * a.hidden + (size_t)min(row, a.npos - 1) * (a.hidden >> 4) + 16 * g + 4 * T + (lane >> 4)];
    // the codes of the two tiles of 16 rows, on their way while the digits are formed
    const uint8_t *cb = a.codes + ((size_t)2 * tile * ngroups + g) * 4096 + 1024 * T + 16 * lane;
    v4i w[2];
#pragma unroll
    for (int r = 0; r < 2; r++) w[r] = *reinterpret_cast<const v4i *>(cb + (size_t)r * ngroups * 4096);
    const int blk = tid >> 7, l2 = (tid >> 1) & 63, e2 = 2 * (tid & 1);   // the sums that this thread finishes: block (vectors, rows), lane, two of its four
    const float2 rm = a.gs[((size_t)(2 * tile + (blk & 1)) * ngroups + g) * 16 + (l2 & 15)];
    float y[16];
    unsigned mx = 0;
#pragma unroll
    for (int i = 0; i < 4; i++)
#pragma unroll
        for (int e = 0; e < 4; e++) {
            y[4 * i + e] = row < a.npos ? v[i][e] : 0.0f;
            mx = max(mx, __float_as_uint(y[4 * i + e]) & 0x7fffffffu);   // (as bits: a NaN is the largest)
        }
    if (row >= a.npos) sum = 0.0f;
    sum += __shfl_xor(sum, 48);   // (the order of wave_sum in quantize_wave, where the four stand in a row of sixteen lanes: first and last, the two between)
    sum += __shfl_xor(sum, 16);
#pragma unroll
    for (int off = 16; off < 64; off <<= 1) mx = max(mx, (unsigned)__shfl_xor((int)mx, off));
    if (lane < 16) { s_max[T][row] = mx; s_sum[T][row] = sum; }
    __syncthreads();
    mx = max(max(s_max[0][row], s_max[1][row]), max(s_max[2][row], s_max[3][row]));
    float inv;
    const int s = digit_shift(mx, &inv);
    if (T == 0 && lane < 16) { s_inv[row] = inv; s_tot[row] = (s_sum[0][row] + s_sum[1][row]) + (s_sum[2][row] + s_sum[3][row]); }
    v4i x[4];
    make_digits(y, s, x);
#pragma unroll
    for (int r = 0; r < 2; r++) {
        const v4i zero = {0, 0, 0, 0};
        v4i hi = __builtin_amdgcn_mfma_i32_16x16x64_i8(x[0], w[r], zero, 0, 0, 0), lo = __builtin_amdgcn_mfma_i32_16x16x64_i8(x[2], w[r], zero, 0, 0, 0);
        hi <<= 8; lo <<= 8;
        red[0][T][2 * m + r][lane] = __builtin_amdgcn_mfma_i32_16x16x64_i8(x[1], w[r], hi, 0, 0, 0);
        red[1][T][2 * m + r][lane] = __builtin_amdgcn_mfma_i32_16x16x64_i8(x[3], w[r], lo, 0, 0, 0);
    }
    __syncthreads();
    const int first = 16 * (blk >> 1) + 4 * (l2 >> 4) + e2;
    float *o = a.out + ((size_t)2 * g * a.npos + first) * a.dim + 32 * tile + 16 * (blk & 1) + (l2 & 15);
#pragma unroll
    for (int h = 0; h < 2; h++) {
#pragma unroll
        for (int k = 0; k < 2; k++) {
            auto both = [&](int d) { return reinterpret_cast<const int *>(&red[d][2 * h][blk][l2])[e2 + k] + reinterpret_cast<const int *>(&red[d][2 * h + 1][blk][l2])[e2 + k]; };
            const int hi = both(0), lo = both(1);
            // (the power of two into the sum, and the offset with the first half, as k_dstream)
            if (first + k < a.npos)
                o[((size_t)h * a.npos + k) * a.dim] = fmaf(fmaf((float)hi, 65536.0f, (float)lo) * s_inv[first + k], rm.x, rm.y * (h ? 0.0f : s_tot[first + k]));
        }
    }
}

struct RowAttn {
    const float *q;          // (rows, dim), RoPE applied
    const float *kc, *vc;    // as RowQkv; the rows of this pass are stored
    long seq_stride, head_stride, row_stride;
    float *out;              // (rows, dim): k_pflash
    Digits dig;              // k_rows_attn
    int nseg, T, pos0;       // rows: T positions of nseg sequences
    int n_heads, kv_mul, dim;
    float sqrt_hs;
    int paired;              // k_rows_attn: two blocks per workgroup
    // k_pflash with the keys of a (head, block) pair split over gridDim.z workgroups (nseg = 1):
    float *pf_part;          // (head, block, z) x (16 maxima, 16 sums, 16 x head_size values): what each leaves for the last one
    unsigned *pf_cnt;        // (head, block): how many have; zero between launches
};

// Keys behind a query's position have weight 0, and 0 times a NaN or an infinity is a NaN.  Where a tile of 16 keys holds such
// values and reaches behind the position of some query of the block, the values go into the product as 0, and the sums of the
// queries that see one are set to NaN by this: flag[e]: 1 where the lane's value of key k0 + 4 g + e (one tile of the
// dimensions) is not finite, else 0.  (An infinity leaves a NaN as well: the norms and digits behind make it one in any case.)
__device__ __forceinline__ void see_not_finite(v4f &o, const float (&flag)[4], int key0, int qpos)
{
    v4f t = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int e = 0; e < 4; e++) t = __builtin_amdgcn_mfma_f32_16x16x4f32(flag[e], key0 + e <= qpos ? 1.0f : 0.0f, t, 0, 0, 0);
#pragma unroll
    for (int i = 0; i < 4; i++) o[i] = t[i] > 0.0f ? __builtin_nanf("") : o[i];
}

__device__ __forceinline__ bool finite(float v) { return (__float_as_uint(v) & 0x7f800000u) != 0x7f800000u; }

// Waves of a workgroup of k_rows_attn, and its dynamic LDS: per wave 16 QPW rows of HS floats (rows a bank apart), maxima and sums.
__host__ __device__ constexpr int attn_waves(int hs) { return hs == 256 ? 4 : 8; }
__host__ __device__ constexpr size_t attn_lds(int hs, int qpw) { return (size_t)attn_waves(hs) * 16 * qpw * (hs + 4 + 2) * sizeof(float); }

// Causal attention on the fp32 matrix cores, as k_pflash multiplies them.  A workgroup takes the HPG = 256 / HS heads whose
// outputs are one group of 256 of the next product's input, and two blocks of 16 QPW positions of one sequence, one after the
// other: block i from the front and block i from the back, so that every workgroup has as many keys to go through (a wave
// per block left the compute units of the first blocks idle behind the last: 142 us at 1024 positions of the 7B shape,
// head size 128, and 16 for the digits as a kernel of their own; now 117, of which the matrix cores need 65).  The KS = waves / HPG waves of a head take every KS-th tile of 16 keys
// with an online softmax each; their parts meet in LDS, where sixteen threads per position merge them into digits.
// QPW = 2: two positions per lane share every cache row loaded, where there are workgroups enough.
// grid: blocks (paired: half of them, rounded up) * nseg * n_heads / HPG.
// Tile u of the values holds the dimensions 64 (u / 4) + 4 m + u % 4, m = 0..15, so that a lane's four values of a cache
// row are one 16-byte load; the keys of the next tile are requested before this tile's are used up.
template <int HS, int QPW>
static __global__ void __launch_bounds__(64 * attn_waves(HS), HS > 128 ? 1 : 2) k_rows_attn(const RowAttn a)
{
    constexpr int U = HS / 16, HPG = 256 / HS, NW = attn_waves(HS), KS = NW / HPG, LD = HS + 4, Q = 16 * QPW;
    extern __shared__ __align__(16) float at_lds[];
    float *lm = at_lds + NW * Q * LD, *ll = lm + NW * Q;   // [wave][Q]
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int c = lane & 15, g = lane >> 4;
    const int units = a.n_heads / HPG * a.nseg, u0 = blockIdx.x % units;
    const int nblk = (a.T + Q - 1) / Q, front = (int)blockIdx.x / units, back = nblk - 1 - front;
    const int hg = u0 % (a.n_heads / HPG), seg = u0 / (a.n_heads / HPG), h = hg * HPG + wave / KS, kvh = h / a.kv_mul;
    const float *kc = a.kc + seg * a.seq_stride + kvh * a.head_stride, *vc = a.vc + seg * a.seq_stride + kvh * a.head_stride;
    const unsigned rs = (unsigned)a.row_stride;   // (uniform addresses and 32-bit offsets, in floats)
    for (int which = 0; which < (a.paired && front != back ? 2 : 1); which++) {
        const int qb = which ? front : back;
        int qpos[QPW];
        v4f qv[QPW][U], o[QPW][U];
        float m[QPW], l[QPW];
#pragma unroll
        for (int p = 0; p < QPW; p++) {
            const int tq = min(Q * qb + 16 * p + c, a.T - 1);        // (past the last position: that one again, not stored)
            qpos[p] = a.pos0 + tq;
            const float *qp = a.q + (size_t)(tq * a.nseg + seg) * a.dim + h * HS + 4 * g;
#pragma unroll
            for (int u = 0; u < U; u++) { qv[p][u] = *reinterpret_cast<const v4f *>(qp + 16 * u); o[p][u] = v4f{0.f, 0.f, 0.f, 0.f}; }
            m[p] = -3.0e38f; l[p] = 0.0f;
        }
        const int lastkey = a.pos0 + min(Q * (qb + 1) - 1, a.T - 1), ntiles = lastkey / 16 + 1;
        v4f kf[U];
        auto keys = [&](int t) {
            const unsigned off = (unsigned)min(16 * t + c, lastkey) * rs + 4 * g;
#pragma unroll
            for (int u = 0; u < U; u++) kf[u] = *reinterpret_cast<const v4f *>(kc + 16 * u + off);
        };
        keys(wave % KS);
        for (int t = wave % KS; t < ntiles; t += KS) {
            const int k0 = t * 16;
            v4f vf[4][U / 4];
#pragma unroll
            for (int e = 0; e < 4; e++) {
                const unsigned off = (unsigned)min(k0 + 4 * g + e, lastkey) * rs + 4 * c;
#pragma unroll
                for (int w = 0; w < U / 4; w++) vf[e][w] = *reinterpret_cast<const v4f *>(vc + 64 * w + off);
            }
            v4f st[QPW];
#pragma unroll
            for (int p = 0; p < QPW; p++) st[p] = v4f{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int u = 0; u < U; u++)
#pragma unroll
                for (int e = 0; e < 4; e++)
#pragma unroll
                    for (int p = 0; p < QPW; p++) st[p] = __builtin_amdgcn_mfma_f32_16x16x4f32(kf[u][e], qv[p][u][e], st[p], 0, 0, 0);
            keys(min(t + KS, ntiles - 1));
            __builtin_amdgcn_sched_barrier(0);
            float pr[QPW][4];
#pragma unroll
            for (int p = 0; p < QPW; p++) {
                float sv[4], tmax = -3.0e38f;
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    sv[e] = k0 + 4 * g + e <= qpos[p] ? __fdiv_rn(st[p][e], a.sqrt_hs) : -3.0e38f;
                    tmax = fmaxf(tmax, sv[e]);
                }
                tmax = fmaxf(tmax, __shfl_xor(tmax, 16));
                tmax = fmaxf(tmax, __shfl_xor(tmax, 32));
                const float mb = fmaxf(m[p], tmax), sc = expf(m[p] - mb);
                l[p] *= sc;
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    pr[p][e] = k0 + 4 * g + e <= qpos[p] ? expf(sv[e] - mb) : 0.0f;
                    l[p] += pr[p][e];
                }
#pragma unroll
                for (int u = 0; u < U; u++) o[p][u] *= sc;
                m[p] = mb;
            }
            if (k0 + 15 > a.pos0 + Q * qb) {   // (a key behind a position of the block)
                v4f z = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int u = 0; u < U; u++)
#pragma unroll
                    for (int e = 0; e < 4; e++) z[e] = fmaf(vf[e][u / 4][u % 4], 0.0f, z[e]);
                if (__any(!((z[0] + z[1]) + (z[2] + z[3]) == 0.0f))) {
#pragma unroll
                    for (int u = 0; u < U; u++) {
                        float flag[4];
#pragma unroll
                        for (int e = 0; e < 4; e++) {
                            const bool ok = finite(vf[e][u / 4][u % 4]);
                            flag[e] = ok ? 0.0f : 1.0f;
                            vf[e][u / 4][u % 4] = ok ? vf[e][u / 4][u % 4] : 0.0f;
                        }
#pragma unroll
                        for (int p = 0; p < QPW; p++) see_not_finite(o[p][u], flag, k0 + 4 * g, qpos[p]);
                        __builtin_amdgcn_sched_barrier(0);
                    }
                }
            }
#pragma unroll
            for (int e = 0; e < 4; e++)
#pragma unroll
                for (int u = 0; u < U; u++)
#pragma unroll
                    for (int p = 0; p < QPW; p++) o[p][u] = __builtin_amdgcn_mfma_f32_16x16x4f32(vf[e][u / 4][u % 4], pr[p][e], o[p][u], 0, 0, 0);
        }
        if (which) __syncthreads();   // (the block before has been read)
#pragma unroll
        for (int p = 0; p < QPW; p++) {
            l[p] += __shfl_xor(l[p], 16);
            l[p] += __shfl_xor(l[p], 32);
            if (g == 0) { lm[wave * Q + 16 * p + c] = m[p]; ll[wave * Q + 16 * p + c] = l[p]; }
            float *op = at_lds + (wave * Q + 16 * p + c) * LD + 16 * g;   // (element i of o[u]: m = 4 g + i)
#pragma unroll
            for (int w = 0; w < U / 4; w++)
#pragma unroll
                for (int i = 0; i < 4; i++)
                    *reinterpret_cast<v4f *>(op + 64 * w + 4 * i) = v4f{o[p][4 * w][i], o[p][4 * w + 1][i], o[p][4 * w + 2][i], o[p][4 * w + 3][i]};
        }
        __syncthreads();
        // position q, values 16 cc .. 16 cc + 15 of the group: of one head, whose KS parts are merged
        for (int i = threadIdx.x; i < Q * 16; i += 64 * NW) {
            const int q = i >> 4, cc = i & 15, t = Q * qb + q, w0 = 16 * cc / HS * KS, at = 16 * cc % HS;
            if (t >= a.T) continue;   // (sixteen threads at a time)
            float M = lm[w0 * Q + q], L = 0.0f, v[16] = {};
#pragma unroll
            for (int w = 1; w < KS; w++) M = fmaxf(M, lm[(w0 + w) * Q + q]);
#pragma unroll
            for (int w = 0; w < KS; w++) {   // (a wave without a tile has left maximum -3e38, sum 0 and values 0)
                const float wt = expf(lm[(w0 + w) * Q + q] - M);
                float x[16];
                load16(at_lds + ((w0 + w) * Q + q) * LD + at, x);
                L += wt * ll[(w0 + w) * Q + q];
#pragma unroll
                for (int k = 0; k < 16; k++) v[k] += wt * x[k];
            }
#pragma unroll
            for (int k = 0; k < 16; k++) v[k] = __fdiv_rn(v[k], L);
            quantize_group(a.dig, t * a.nseg + seg, a.dim >> 8, hg, cc, v);
        }
    }
}

// Attention of 16 consecutive positions of one sequence for one head on the fp32 matrix cores (after k_rows_qkv has stored
// their k and v): every cache row is fetched once for the 16 queries, instead of once per query.
//   scores, transposed: S^T (16 keys x 16 queries) = K (16 keys x HS) . Q^T (HS x 16 queries), HS / 4 v_mfma_f32_16x16x4_f32;
//     a lane (c = lane % 16, g = lane / 16) then holds S^T[key 4 g + e][query c], e = 0..3: the keys of a query lie in four
//     lanes, so a query's maximum is two cross-lane steps, and the same registers are the B operand of
//   values, transposed: O^T (HS x 16 queries) += V^T (HS x 16 keys) . P^T (16 keys x 16 queries), HS / 4 more;
//   online softmax over the tiles of 16 keys (K/AttentionLoop.java:29-54, K/ExpSumNormalize.java:25-38,
//     K/AccumWeightedValue.java restated as in k_battn), a query seeing the keys up to its own position.
// The waves of the workgroup take every WAVES-th tile of keys and merge their (maximum, sum, values) through LDS.
// The k index of a product may be permuted if both operands are: lane group g supplies the dimensions 16 u + 4 g + e
// (one 16-byte load per u) and the keys 4 g + e.
// grid: (n_heads, blocks of 16 positions, 1..4): z splits the tiles of keys over that many workgroups, the last of which to finish merges what the
// others left in device memory.  64 * WAVES threads; dynamic LDS: (32 WAVES + 16 WAVES HS) floats.
template <int HS, int WAVES>
__global__ void __launch_bounds__(64 * WAVES) k_pflash(const RowAttn a)
{
    constexpr int U = HS / 16;
    extern __shared__ __align__(16) float pf_lds[];
    float *wm = pf_lds;                  // [WAVES][16]
    float *wl = wm + WAVES * 16;         // [WAVES][16]
    float *wo = wl + WAVES * 16;         // [WAVES][HS / 4][16 queries][4]: dimension d of query q at (d / 4) * 64 + 4 q + d % 4
    __shared__ float ww[WAVES * 16], wM[16];
    __shared__ int s_last;
    const int h = blockIdx.x, qb = blockIdx.y * 16, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int c = lane & 15, g = lane >> 4;
    const int vrows = min(16, a.T - qb);   // (rows past the end repeat the last one: their output is not used)
    const int pos0 = a.pos0 + qb, kvh = h / a.kv_mul;
    const float *qp = a.q + (size_t)(qb + min(c, vrows - 1)) * a.dim + h * HS + 4 * g;
    float4 qv[U];
#pragma unroll
    for (int u = 0; u < U; u++) qv[u] = *reinterpret_cast<const float4 *>(qp + 16 * u);
    const int qpos = pos0 + min(c, vrows - 1), lastkey = pos0 + vrows - 1, ntiles = lastkey / 16 + 1;
    const float *kc = a.kc + kvh * a.head_stride, *vc = a.vc + kvh * a.head_stride;
    const long rs = a.row_stride;
    v4f o[U];
#pragma unroll
    for (int u = 0; u < U; u++) o[u] = v4f{0.f, 0.f, 0.f, 0.f};
    float m = -3.0e38f, l = 0.0f;
    // tile t of the keys goes to workgroup t % NS (z) and there to wave (t / NS) % WAVES: few tiles spread over the workgroups first
    const int NS = gridDim.z;
    const int mytiles = (ntiles - (int)blockIdx.z + NS - 1) / NS;   // of this workgroup
    const int nw = min(WAVES, mytiles);                              // waves that have any
    for (int t = blockIdx.z + NS * wave; t < ntiles; t += NS * WAVES) {
        const int k0 = t * 16;
        const float *krow = kc + (long)min(k0 + c, lastkey) * rs + 4 * g;   // (past the last key: that key again, left out below)
        float4 kf[U];
#pragma unroll
        for (int u = 0; u < U; u++) kf[u] = *reinterpret_cast<const float4 *>(krow + 16 * u);
        v4f32 st = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int u = 0; u < U; u++) {
            st = __builtin_amdgcn_mfma_f32_16x16x4f32(kf[u].x, qv[u].x, st, 0, 0, 0);
            st = __builtin_amdgcn_mfma_f32_16x16x4f32(kf[u].y, qv[u].y, st, 0, 0, 0);
            st = __builtin_amdgcn_mfma_f32_16x16x4f32(kf[u].z, qv[u].z, st, 0, 0, 0);
            st = __builtin_amdgcn_mfma_f32_16x16x4f32(kf[u].w, qv[u].w, st, 0, 0, 0);
        }
        float sv[4], tmax = -3.0e38f;
#pragma unroll
        for (int e = 0; e < 4; e++) {
            sv[e] = k0 + 4 * g + e <= qpos ? __fdiv_rn(st[e], a.sqrt_hs) : -3.0e38f;   // (a query sees the keys up to its own position)
            tmax = fmaxf(tmax, sv[e]);
        }
        tmax = fmaxf(tmax, __shfl_xor(tmax, 16));
        tmax = fmaxf(tmax, __shfl_xor(tmax, 32));
        const float mb = fmaxf(m, tmax), sc = expf(m - mb);
        float pr[4];
        l *= sc;
#pragma unroll
        for (int e = 0; e < 4; e++) {
            pr[e] = k0 + 4 * g + e <= qpos ? expf(sv[e] - mb) : 0.0f;
            l += pr[e];
        }
#pragma unroll
        for (int u = 0; u < U; u++) o[u] *= sc;
        m = mb;
        bool clean = true;
        if (k0 + 15 > pos0) {   // (as in k_rows_attn)
            float z = 0.0f;
#pragma unroll 1
            for (int e = 0; e < 4; e++) {
                const float *vrow = vc + (long)min(k0 + 4 * g + e, lastkey) * rs + c;
#pragma unroll
                for (int u = 0; u < U; u++) z = fmaf(vrow[16 * u], 0.0f, z);
            }
            clean = !__any(!(z == 0.0f));
            if (!clean) {
#pragma unroll
                for (int u = 0; u < U; u++) {
                    float flag[4];
#pragma unroll
                    for (int e = 0; e < 4; e++) flag[e] = finite(vc[(long)min(k0 + 4 * g + e, lastkey) * rs + c + 16 * u]) ? 0.0f : 1.0f;
                    see_not_finite(o[u], flag, k0 + 4 * g, qpos);
                    __builtin_amdgcn_sched_barrier(0);
                }
            }
        }
#pragma unroll
        for (int e = 0; e < 4; e++) {
            const float *vrow = vc + (long)min(k0 + 4 * g + e, lastkey) * rs + c;
#pragma unroll
            for (int u = 0; u < U; u++) {
                const float v = vrow[16 * u];
                o[u] = __builtin_amdgcn_mfma_f32_16x16x4f32(clean || finite(v) ? v : 0.0f, pr[e], o[u], 0, 0, 0);
            }
        }
    }
    l += __shfl_xor(l, 16);
    l += __shfl_xor(l, 32);
    if (g == 0) { wm[wave * 16 + c] = m; wl[wave * 16 + c] = l; }
    if (wave < nw) {   // (the waves without a tile have nothing to add)
#pragma unroll
        for (int u = 0; u < U; u++)   // (a lane's four dimensions 16 u + 4 g + e of query c as one 16-byte store, a wave's stores 1 KB in a row)
            *reinterpret_cast<v4f *>(&wo[wave * HS * 16 + (4 * u + g) * 64 + 4 * c]) = o[u];
    }
    __syncthreads();
    if (tid < 16 * WAVES) {   // weight of wave w's part in query q's sum: tid = w * 16 + q (a workgroup without any tile leaves
        const int q = tid & 15;   // maximum -3e38, sum 0 and values 0)
        float M = wm[q];
#pragma unroll
        for (int w = 1; w < WAVES; w++) M = fmaxf(M, wm[w * 16 + q]);
        ww[tid] = expf(wm[tid] - M);
        if (tid < 16) wM[tid] = M;
    }
    __syncthreads();
    if (NS == 1) {
        for (int idx = tid; idx < HS * 16; idx += 64 * WAVES) {   // the waves' parts of a query merged
            const int d = (idx >> 6) * 4 + (idx & 3), q = (idx >> 2) & 15;   // (neighbouring lanes read neighbouring words of LDS)
            float L = 0.0f, O = 0.0f;
#pragma unroll
            for (int w = 0; w < WAVES; w++) {
                if (w < nw) {
                    const float wt = ww[w * 16 + q];
                    L += wt * wl[w * 16 + q];
                    O += wt * wo[w * HS * 16 + idx];
                }
            }
            if (q < vrows) a.out[(long)(qb + q) * a.dim + h * HS + d] = __fdiv_rn(O, L);
        }
        return;
    }
    // The keys are split over NS workgroups: each leaves its maxima, sums and values (not yet divided) in device memory, and
    // the last one to do so merges them all.
    constexpr int PER = 32 + 16 * HS;
    const int pair = h * gridDim.y + blockIdx.y;
    float *mine = a.pf_part + ((long)pair * NS + blockIdx.z) * PER;
    for (int idx = tid; idx < HS * 16; idx += 64 * WAVES) {   // (values in the order they have in LDS)
        const int d = (idx >> 6) * 4 + (idx & 3), q = (idx >> 2) & 15;
        float L = 0.0f, O = 0.0f;
#pragma unroll
        for (int w = 0; w < WAVES; w++) {
            if (w < nw) {
                const float wt = ww[w * 16 + q];
                L += wt * wl[w * 16 + q];
                O += wt * wo[w * HS * 16 + idx];
            }
        }
        st_coh(mine + 32 + idx, O);
        if (d == 0) { st_coh(mine + q, wM[q]); st_coh(mine + 16 + q, L); }
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // (this thread's stores have arrived where the other workgroups read)
    __syncthreads();
    if (tid == 0) {
        const unsigned old = __hip_atomic_fetch_add(a.pf_cnt + pair, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        s_last = old + 1u == (unsigned)NS;
        if (s_last) __hip_atomic_store(a.pf_cnt + pair, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);   // (for the next launch)
    }
    __syncthreads();
    if (!s_last) return;
    const float *all = a.pf_part + (long)pair * NS * PER;
    for (int idx = tid; idx < HS * 16; idx += 64 * WAVES) {
        const int q = (idx >> 2) & 15;
        float mz[4], M = -3.0e38f;
#pragma unroll
        for (int z = 0; z < 4; z++) {
            mz[z] = z < NS ? ld_coh(all + (long)z * PER + q) : -3.0e38f;
            M = fmaxf(M, mz[z]);
        }
        float L = 0.0f, O = 0.0f;
#pragma unroll
        for (int z = 0; z < 4; z++) {
            if (z < NS) {
                const float wt = expf(mz[z] - M);
                L += wt * ld_coh(all + (long)z * PER + 16 + q);
                O += wt * ld_coh(all + (long)z * PER + 32 + idx);
            }
        }
        if (q < vrows) a.out[(long)(qb + q) * a.dim + h * HS + (idx >> 6) * 4 + (idx & 3)] = __fdiv_rn(O, L);
    }
}

// logits = W x for one row x (K/MatMul.java:37-60): a wave per row of the classifier.
static __global__ void __launch_bounds__(256) k_rows_logits(const float *__restrict__ w, const float *__restrict__ x, float *__restrict__ logits,
                                                     int dim, int vocab)
{
    extern __shared__ __align__(16) float lx[];
    const int n4 = dim >> 2, lane = threadIdx.x & 63;
    float4 *l4 = reinterpret_cast<float4 *>(lx);
    for (int i = threadIdx.x; i < n4; i += 256) l4[i] = reinterpret_cast<const float4 *>(x)[i];
    __syncthreads();
    for (int r = blockIdx.x * 4 + (threadIdx.x >> 6); r < vocab; r += 4 * gridDim.x) {
        const float4 *wr = reinterpret_cast<const float4 *>(w + (size_t)r * dim);
        float t = 0.0f;
#pragma unroll 8
        for (int i = lane; i < n4; i += 64) t += dot4(load_stream(wr + i), l4[i]);
        t = wave_sum(t);
        if (lane == 0) logits[r] = t;
    }
}

}  // namespace l2j
