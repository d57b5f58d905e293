// The token of a small model in one launch whose layers run on one XCD.
//
// A layer of a small model is five dependent phases of a few kilobytes to compute on, and what a token costs is the way of
// the vectors between them.  Handed from all 256 workgroups to all 256 (k_token), a vector of 288 or 768 floats takes 2.5 us a
// phase: 256 pollers queue for its few lines in memory.  Among the 32 workgroups of one XCD it takes 0.6: a plain store leaves
// the words in that XCD's L2, where the others' loads (past their L1) find them 0.22 us later.  So workgroups 8 i (the ones the
// dispatcher puts on the first XCD) run the layers, 1.3 TB/s from beyond its L2 being enough for up to some 8 MB a layer, and
// the others meanwhile mark the next token's vectors unwritten and load their rows of the classifier into registers.  They
// get the last vector through one workgroup per XCD, which passes it on inside its own L2.
//
// 15M shape (288, 768, six layers), us a token at positions 5 and 255: k_token 111 and 122, this 58 and 69; two layers 51 and 54 -> 24
// and 26.  (5.5 of these more when the classifier's workgroups requested rows past their own behind their last; 1.3 less with the
// exponentials and the scale of q in one rounding each, at 130 times the error of a far weight.)  What is left of a layer's 8.5 us, by time stamps: the hand-overs 0.5 to 0.6 us each, the stagers 0.3, a phase's
// multiply-adds and sums 0.45 (one wave per SIMD issues an instruction every five to six cycles), attention 1.0.
//
// Nothing depends on where the workgroups really run but the speed: a word that is not seen stays unwritten (kUnset), the
// bounded wait for it runs out and the host falls back to k_token.
//
// In a workgroup of the layers two waves (stagers) wait for the input of the next phase and put it into LDS; the other six hold
// the codes of all phases in registers, requested a layer ahead, and never wait for anything but these and the barrier
// that publishes the input (a wait of their own would be in order behind the requests: loads return in order).
#pragma once

#include "digit_gemm.hpp"
#include "phase_kernels.hpp"

namespace l2j {

constexpr int kXThreads = 512, kXStagers = 2, kXWaves = kXThreads / 64 - kXStagers, kXLanes = 64 * kXWaves;
constexpr int kXcds = 8;
constexpr int kXMaxSplits = 4;    // splits of a head's cache rows
constexpr int kXRowsAhead = 4;    // cache rows per 16 lanes requested ahead
constexpr int kXSplitRows = 4 * kXWaves * kXRowsAhead;   // cache rows per split before there are more splits

struct XcdArgs {
    TokenGeom g;
    int maxspin;
    int nsplit;      // at most this many splits per head
    float *mem;      // two sets of: the splits' results (layer, head, split) x (head_size + 4), the last vector once per XCD
    long mem_stride; // floats of one set
};

__host__ __device__ inline long xcd_part_floats(int n_layers, int n_heads, int nsplit, int head_size) { return (long)n_layers * n_heads * nsplit * (head_size + 4); }

// Lanes per row and chunks of 16 codes per lane: rows of dim codes (LD, CD), of hidden codes (LH, CH); lanes and float4s per row of
// the classifier (LC, FC).  One row per group of lanes and phase (W1 and W3: one of each): up to 384 x 768, the 15M shape.  (The 110M
// shape this way, three rows and six per group of lanes and up to eight chunks, takes 220 to 270 us a token, k_token 212 to 235:
// the multiply-adds of 7 MB a layer are too many for 32 compute units.)
struct XSmall {
    static constexpr int LD = 8, CD = 3, LH = 16, CH = 3, LC = 8, FC = 12;
};

// LDS of a workgroup, in floats.  An input vector of up to 16 NC floats: float4 (quarter q, chunk c) at q * NC + c, then the
// chunks' sums; the chunks past the vector hold zeros, so that no lane of a fold is masked.
template <class C>
struct XLds {
    static constexpr int ND = C::LD * C::CD, NH = C::LH * C::CH;   // chunks
    static constexpr int xd0 = 0, xd1 = xd0 + 17 * ND, xh = xd1 + 17 * ND;   // Wq Wk Wv and W1 W3; Wo; W2
    static constexpr int raw0 = (xh + 17 * NH + 3) / 4 * 4, raw1 = raw0 + 16 * ND;   // the residual stream before Wo and W2
    static constexpr int red = raw1 + 16 * ND;          // sums of squares: two per norm
    static constexpr int qkv = red + 4, acc = qkv + 3 * 64, ml = acc + 64 * kXWaves, silu = ml + 16, end = silu + kSiluTable;
    static_assert(xd1 % 4 == 0 && xh % 4 == 0 && 4 * end <= 65536, "");
};

// A pointer to global memory that says so: a choice by lane between generic ones becomes flat loads.
template <typename T>
using Global = __attribute__((address_space(1))) T *;

template <typename T>
__device__ __forceinline__ Global<T> pinned(T *p)   // (left alone, a choice by lane between fields of the argument becomes a load of the chosen field)
{
    Global<T> q = (Global<T>)p;
    asm volatile("" : "+s"(q));
    return q;
}

typedef const __attribute__((address_space(4))) XcdArgs *XcdArgsPtr;
__device__ __forceinline__ XcdArgsPtr xcd_args()   // (re-read where it is used, see token_args)
{
    XcdArgsPtr p = (XcdArgsPtr)__builtin_amdgcn_kernarg_segment_ptr();
    asm volatile("" : "+s"(p));
    return p;
}

// The codes and scales of one row per group of LP lanes, CP chunks of 16 per lane, in registers.
template <int LP, int CP>
struct XRow {
    static constexpr int NC = LP * CP;
    uint4 w[CP];
    float2 s[CP];

    // Where a lane's words of a row lie, in bytes from the layer's matrix and its scales (past the row: its last chunk, which
    // meets a zero).
    struct At {
        unsigned c[CP], s[CP];
        __device__ __forceinline__ void set(int row, int n, int cl)
        {
#pragma unroll
            for (int j = 0; j < CP; j++) {
                c[j] = (unsigned)row * (unsigned)n + 16u * (unsigned)min(cl + LP * j, (n >> 4) - 1);
                s[j] = c[j] >> 8 << 3;
            }
        }
    };

    __device__ __forceinline__ void request(Global<const uint8_t> codes, Global<const uint8_t> gs, const At &at)
    {
#pragma unroll
        for (int j = 0; j < CP; j++) {
            const v4u v = __builtin_nontemporal_load((Global<const v4u>)(codes + at.c[j]));
            w[j] = make_uint4(v.x, v.y, v.z, v.w);
        }
#pragma unroll
        for (int j = 0; j < CP; j++) {
            const v2f v = *(Global<const v2f>)(gs + at.s[j]);
            s[j] = make_float2(v.x, v.y);
        }
    }

    // the sum of the row, in all its lanes; a second row against the same values
    template <int N>
    static __device__ __forceinline__ void fold(const XRow *const (&rows)[N], const float *x, int cl, float (&acc)[N])
    {
        const float4 *x4 = reinterpret_cast<const float4 *>(x) + cl;
#pragma unroll
        for (int r = 0; r < N; r++) acc[r] = 0.0f;
#pragma unroll
        for (int j = 0; j < CP; j++) {
            const float4 v0 = x4[LP * j], v1 = x4[NC + LP * j], v2 = x4[2 * NC + LP * j], v3 = x4[3 * NC + LP * j];
            const float sx = (x + 16 * NC + cl)[LP * j];
#pragma unroll
            for (int r = 0; r < N; r++) acc[r] += fmaf(rows[r]->s[j].x, dot16(rows[r]->w[j], v0, v1, v2, v3), rows[r]->s[j].y * sx);
        }
#pragma unroll
        for (int r = 0; r < N; r++) {
            acc[r] += dpp_f<0xB1>(acc[r]);
            acc[r] += dpp_f<0x4E>(acc[r]);
            acc[r] += dpp_f<0x141>(acc[r]);   // row_half_mirror: eight lanes
            if (LP == 16) acc[r] += dpp_f<0x128>(acc[r]);
        }
    }
};

// The 16-byte words at p[0..N-1] once their producers have written all of them, requested together.
template <int N>
__device__ __forceinline__ void xwait(const float *const (&p)[N], float4 (&v)[N], const Poll &pl)
{
    int spins = 0;
    while (true) {
        if constexpr (N == 1) {
            v[0] = ld_coh16(p[0]);
        } else if constexpr (N == 2) {
            asm volatile("global_load_dwordx4 %0, %2, off sc1\n\tglobal_load_dwordx4 %1, %3, off sc1\n\ts_waitcnt vmcnt(0)"
                         : "=&v"(v[0]), "=&v"(v[1]) : "v"(p[0]), "v"(p[1]) : "memory");
        } else {
            static_assert(N == 4, "one, two or four words at a time");
            asm volatile("global_load_dwordx4 %0, %4, off sc1\n\tglobal_load_dwordx4 %1, %5, off sc1\n\t"
                         "global_load_dwordx4 %2, %6, off sc1\n\tglobal_load_dwordx4 %3, %7, off sc1\n\ts_waitcnt vmcnt(0)"
                         : "=&v"(v[0]), "=&v"(v[1]), "=&v"(v[2]), "=&v"(v[3]) : "v"(p[0]), "v"(p[1]), "v"(p[2]), "v"(p[3]) : "memory");
        }
        bool ok = true;
#pragma unroll
        for (int i = 0; i < N; i++) ok = ok && all_set(v[i]);
        if (ok) break;
        if (++spins > pl.maxspin || ((spins & 63) == 0 && ld_coh(pl.fault) != 0)) { st_coh(pl.fault, 1); break; }
    }
}

// A stager's words wl, wl + 128, ... of an input vector of up to 16 NC floats.
template <int NC>
struct XStage {
    static constexpr int N = (4 * NC + 64 * kXStagers - 1) / (64 * kXStagers);
    float4 g[N];   // the norm weights

    __device__ __forceinline__ void request(const float *w, int n, int wl)
    {
#pragma unroll
        for (int j = 0; j < N; j++) g[j] = reinterpret_cast<const float4 *>(w)[min(wl + 64 * kXStagers * j, (n >> 2) - 1)];
    }

    static __device__ __forceinline__ void clear_past(float *x, int n, int wl)
    {
        for (int i = wl; i < 4 * NC; i += 64 * kXStagers) {
            if (i < (n >> 2)) continue;
            reinterpret_cast<float4 *>(x)[(i & 3) * NC + (i >> 2)] = make_float4(0.f, 0.f, 0.f, 0.f);
            x[16 * NC + (i >> 2)] = 0.0f;
        }
    }

    // words into x (times the norm weights), as they came into raw (not null), their sum of squares into red
    template <bool NORM>
    __device__ __forceinline__ void put(const float4 (&v)[N], int n, int wl, float *x, float *raw, float *red) const
    {
        float ssq = 0.0f;
#pragma unroll
        for (int j = 0; j < N; j++) {
            const int i = wl + 64 * kXStagers * j;
            float4 f = v[j];
            const bool ok = i < (n >> 2);   // (whole quads)
            if (NORM) {
                const float t = (f.x * f.x + f.y * f.y) + (f.z * f.z + f.w * f.w);
                ssq += ok ? t : 0.0f;
                if (ok) reinterpret_cast<float4 *>(raw)[i] = f;
                f.x = __fmul_rn(g[j].x, f.x);
                f.y = __fmul_rn(g[j].y, f.y);
                f.z = __fmul_rn(g[j].z, f.z);
                f.w = __fmul_rn(g[j].w, f.w);
            }
            float s = (f.x + f.y) + (f.z + f.w);
            s += dpp_f<0xB1>(s);
            s += dpp_f<0x4E>(s);
            if (ok) {
                reinterpret_cast<float4 *>(x)[(i & 3) * NC + (i >> 2)] = f;
                if ((i & 3) == 0) x[16 * NC + (i >> 2)] = s;
            }
        }
        if (NORM) {
            ssq = wave_sum(ssq);
            if ((wl & 63) == 0) red[wl >> 6] = ssq;
        }
    }

    static __device__ __forceinline__ void words(const float *x, int n, int wl, float4 (&v)[N], const Poll &pl)
    {
        const float *p[N];
#pragma unroll
        for (int j = 0; j < N; j++) p[j] = x + 4 * min(wl + 64 * kXStagers * j, (n >> 2) - 1);
        xwait<N>(p, v, pl);
    }
};

// 1 / sqrt(sum x^2 / n + 1e-5) from the stagers' sums (K/RootMeanSquare.java:31-33): rn = 1 / n, and one step of Newton's method
// behind the instruction's result (eight instructions in every wave instead of some forty for two divisions and a root, and no
// less exact: against 64 bits 0.52 to 0.65 units of 2^-24, 1.95 at most, for the two divisions and the root 0.64 to 0.67 and 2.3);
// where the sum is infinite the step's 1 - a y^2 is no number, and the maximum keeps the instruction's 0
__device__ __forceinline__ float xcd_rms(const float *red, float rn)
{
    const float a = fmaf(red[0] + red[1], rn, 1e-5f), y = __builtin_amdgcn_rsqf(a);
    return fmaf(0.5f * y, fmaxf(fmaf(-a * y, y, 1.0f), -1.0f), y);
}

// q / b, r = 1 / b rounded: the quotient's residual folded back in (Markstein 1990).  The same word as the division for every q and the root
// of every head size up to 64; one that is not finite, which the residual is not either, is a NaN (and with it every score it enters or their sum).
__device__ __forceinline__ float quotient(float q, float b, float r)
{
    const float y = q * r;
    return fmaf(fmaf(-y, b, q), r, y);
}

// How the cache rows of a head are split at a length: splits, and rows of each.
__device__ __forceinline__ int xcd_splits(int len, int most, int &chunk)
{
    int n = (len + kXSplitRows - 1) / kXSplitRows;
    n = min(n, most);
    chunk = (len + n - 1) / n;
    return (len + chunk - 1) / chunk;
}

// The stagers of a workgroup of the layers: lanes wl = 0..127.
template <class C>
__device__ __forceinline__ void xcd_stage_layers(float *lds, int w, int wl, int token, int pos, int set)
{
    typedef XLds<C> M;
    XcdArgsPtr a = xcd_args();
    Poll pl;
    pl.on = 1; pl.maxspin = a->maxspin; pl.fault = a->g.fault;
    const int dim = a->g.dim, hid = a->g.hidden, hs = a->g.head_size, L = a->g.n_layers, nh = a->g.n_heads, nsplit = a->nsplit;
    const long so = set * a->g.set_stride, sd = a->g.sd, skv = a->g.skv, sh = a->g.sh;
    const float *x = a->g.x + so, *xb = a->g.xb + so, *hb = a->g.hb + so, *rmsw = a->g.rmsw;
    const float sqrt_hs = a->g.sqrt_hs, rs = __fdiv_rn(1.0f, sqrt_hs);
    int chunk;
    const int nact = xcd_splits(pos + 1, nsplit, chunk), head = w % nh;
    const bool item = w < nh * nact;
    // this lane's word of q, k and v of the head (sixteen each)
    const int which = wl >> 4, j4 = min(wl & 15, (hs >> 2) - 1);
    const float *qkv = (which == 0 ? a->g.q + head * hs : (which == 1 ? a->g.knew : a->g.vnew) + head / a->g.kv_mul * hs) + so + 4 * j4;
    const long qkv_step = which == 0 ? sd : skv;
    const float *part = a->mem + set * a->mem_stride;
    XStage<M::ND> st;
    XStage<M::NH> sh_;
    float4 v[st.N];
    st.request(rmsw, dim, wl);
#pragma unroll
    for (int j = 0; j < st.N; j++) v[j] = reinterpret_cast<const float4 *>(a->g.emb + (long)token * dim)[min(wl + 64 * kXStagers * j, (dim >> 2) - 1)];
    st.clear_past(lds + M::xd0, dim, wl);
    st.clear_past(lds + M::xd1, dim, wl);
    sh_.clear_past(lds + M::xh, hid, wl);
    for (int l = 0; l < L; l++) {
        if (l > 0) st.words(x + 2L * l * sd, dim, wl, v, pl);
        st.template put<true>(v, dim, wl, lds + M::xd0, lds + M::raw0, lds + M::red);
        __syncthreads();
        st.request(rmsw + (long)(L + l) * dim, dim, wl);
        if (item) {
            if (wl < 3 * 16) {
                const float *p[1] = {qkv + l * qkv_step};
                float4 q[1];
                xwait<1>(p, q, pl);
                if (which == 0) {   // (the scores' division by sqrt(head_size), K/AttentionLoop.java:48)
                    q[0].x = quotient(q[0].x, sqrt_hs, rs); q[0].y = quotient(q[0].y, sqrt_hs, rs);
                    q[0].z = quotient(q[0].z, sqrt_hs, rs); q[0].w = quotient(q[0].w, sqrt_hs, rs);
                }
                reinterpret_cast<float4 *>(lds + M::qkv)[16 * which + (wl & 15)] = q[0];
            }
            __syncthreads();
            __syncthreads();
        }
        if (nact == 1) {
            st.words(xb + l * sd, dim, wl, v, pl);
        } else {   // the splits' values, merged
#pragma unroll
            for (int j = 0; j < st.N; j++) {
                const int i = 4 * min(wl + 64 * kXStagers * j, (dim >> 2) - 1), h = i / hs;
                const float *hp = part + (long)(l * nh + h) * nsplit * (hs + 4);
                const int e = 4 + i - h * hs;
                float m = -3.402823466e+38f, sum = 0.0f;
                float4 o = make_float4(0.f, 0.f, 0.f, 0.f);
                for (int s = 0; s < nact; s += 2) {
                    const float *p0 = hp + s * (hs + 4), *p1 = hp + min(s + 1, nact - 1) * (hs + 4);
                    const float *p[4] = {p0, p0 + e, p1, p1 + e};
                    float4 q[4];
                    xwait<4>(p, q, pl);
                    const bool two = s + 1 < nact;
                    const float mb = fmaxf(m, two ? fmaxf(q[0].x, q[2].x) : q[0].x);
                    const float k = s > 0 ? expf(m - mb) : 0.0f, k0 = expf(q[0].x - mb), k1 = two ? expf(q[2].x - mb) : 0.0f;
                    sum = fmaf(q[2].y, k1, fmaf(q[0].y, k0, sum * k));
                    o.x = fmaf(q[3].x, k1, fmaf(q[1].x, k0, o.x * k));
                    o.y = fmaf(q[3].y, k1, fmaf(q[1].y, k0, o.y * k));
                    o.z = fmaf(q[3].z, k1, fmaf(q[1].z, k0, o.z * k));
                    o.w = fmaf(q[3].w, k1, fmaf(q[1].w, k0, o.w * k));
                    m = mb;
                }
                v[j] = make_float4(__fdiv_rn(o.x, sum), __fdiv_rn(o.y, sum), __fdiv_rn(o.z, sum), __fdiv_rn(o.w, sum));
                if (w == 0) *reinterpret_cast<float4 *>(const_cast<float *>(xb) + l * sd + i) = v[j];   // (for l2j_read)
            }
        }
        st.template put<false>(v, dim, wl, lds + M::xd1, nullptr, nullptr);
        __syncthreads();
        st.words(x + (2L * l + 1) * sd, dim, wl, v, pl);
        st.template put<true>(v, dim, wl, lds + M::xd0, lds + M::raw1, lds + M::red + 2);
        __syncthreads();
        st.request(rmsw + (long)min(l + 1, L - 1) * dim, dim, wl);
        {
            float4 h[sh_.N];
            sh_.words(hb + l * sh, hid, wl, h, pl);
            sh_.template put<false>(h, hid, wl, lds + M::xh, nullptr, nullptr);
        }
        __syncthreads();
    }
}

// The other waves: t = 0 .. kXLanes - 1.
template <class C>
__device__ __forceinline__ void xcd_layers(float *lds, int w, int nwork, int t, int pos, int set)
{
    typedef XLds<C> M;
    static_assert(C::LD == 8 && C::LH == 16, "the sums' exchanges between lanes");
    typedef XRow<C::LD, C::CD> RD;
    typedef XRow<C::LH, C::CH> RH;
    typedef Global<const uint8_t> Bytes;
    const int lane = t & 63, wave = __builtin_amdgcn_readfirstlane(t >> 6);
    const int gd = t / C::LD, cd = t % C::LD, gh = t / C::LH, ch = t % C::LH;
    int dim, hid, kvd, hs, L;
    long so, sd;
    {
        XcdArgsPtr a = xcd_args();
        dim = a->g.dim; hid = a->g.hidden; kvd = a->g.kv_dim; hs = a->g.head_size; L = a->g.n_layers;
        so = set * a->g.set_stride; sd = a->g.sd;
    }
    // This workgroup's rows, consecutive ones: pairs of rows of Wq, Wk and Wv one after the other, rows of W1 and W3, of Wo and
    // W2.  (A group of lanes without a row takes row 0 and drops the result.)
    RD rq, ro, r1, r3;
    RH r2;
    typename RD::At aq, ao, a13;
    typename RH::At a2;
    const int per13 = (hid + nwork - 1) / nwork, pero = (dim + nwork - 1) / nwork;
    const int pairs = (dim + 2 * kvd) >> 1, perq = 2 * ((pairs + nwork - 1) / nwork);
    const bool okq = gd < perq && w * perq + gd < 2 * pairs, ok13 = gd < per13 && w * per13 + gd < hid;
    const bool oko = gd < pero && w * pero + gd < dim, ok2 = gh < pero && w * pero + gh < dim;
    const int rowo = oko ? w * pero + gd : 0, row2 = ok2 ? w * pero + gh : 0, row13 = ok13 ? w * per13 + gd : 0;
    int rowq = okq ? w * perq + gd : 0;
    const bool isq = rowq < dim, isk = !isq && rowq < dim + kvd;
    rowq -= isq ? 0 : isk ? dim : dim + kvd;   // in its matrix
    aq.set(rowq, dim, cd);
    ao.set(rowo, dim, cd);
    a13.set(row13, dim, cd);
    a2.set(row2, hid, ch);
    float2 cs;   // K/ApplyRope.java:74-90: own * x + the other row of the pair * y
    {
        XcdArgsPtr a = xcd_args();
        const v2f c = ((Global<const v2f>)a->g.rope)[pos * (hs >> 1) + ((rowq % hs) >> 1)];
        cs = make_float2(c.x, (rowq & 1) ? c.y : -c.y);
    }
    auto request_q = [&](int l) {
        XcdArgsPtr a = xcd_args();
        const long fq = (long)l * dim * dim, fk = (long)l * kvd * dim;
        const Bytes cq = (Bytes)pinned(a->g.wq.codes) + fq, ck = (Bytes)pinned(a->g.wk.codes) + fk, cv = (Bytes)pinned(a->g.wv.codes) + fk;
        const Bytes sq = (Bytes)pinned(a->g.wq.gs) + (fq >> 8) * 8, sk = (Bytes)pinned(a->g.wk.gs) + (fk >> 8) * 8, sv = (Bytes)pinned(a->g.wv.gs) + (fk >> 8) * 8;
        rq.request(isq ? cq : isk ? ck : cv, isq ? sq : isk ? sk : sv, aq);
    };
    auto request_o = [&](int l) {
        XcdArgsPtr a = xcd_args();
        const long f = (long)l * dim * dim;
        ro.request((Bytes)a->g.wo.codes + f, (Bytes)a->g.wo.gs + (f >> 8) * 8, ao);
    };
    auto request_13 = [&](int l) {
        XcdArgsPtr a = xcd_args();
        const long f = (long)l * hid * dim;
        r1.request((Bytes)a->g.w1.codes + f, (Bytes)a->g.w1.gs + (f >> 8) * 8, a13);
        r3.request((Bytes)a->g.w3.codes + f, (Bytes)a->g.w3.gs + (f >> 8) * 8, a13);
    };
    auto request_2 = [&](int l) {
        XcdArgsPtr a = xcd_args();
        const long f = (long)l * hid * dim;
        r2.request((Bytes)a->g.w2.codes + f, (Bytes)a->g.w2.gs + (f >> 8) * 8, a2);
    };
    // Attention: sixteen lanes per cache row, four floats each.  Rows t0 .. t1 - 1 of the cache, and this token's where the split
    // reaches it.
    int chunk, head, split, kvcol, t0, t1;
    bool item, active, now;
    int nact;
    {
        XcdArgsPtr a = xcd_args();
        nact = xcd_splits(pos + 1, a->nsplit, chunk);
        head = w % a->g.n_heads; split = w / a->g.n_heads;
        item = w < a->g.n_heads * nact;
        active = 4 * (lane & 15) < hs;
        kvcol = head / a->g.kv_mul * hs + (active ? 4 * (lane & 15) : 0);
        t0 = split * chunk; t1 = min(pos, t0 + chunk);
        now = pos < t0 + chunk;
    }
    const int slot = 4 * wave + (lane >> 4);
    v4f k4[kXRowsAhead], v4[kXRowsAhead];
    auto request_kv = [&](int l, int tb) {
        XcdArgsPtr a = xcd_args();
        const long f = (long)l * a->g.seq_len * kvd;
        const Global<const float> kc = (Global<const float>)a->g.kcache + f, vc = (Global<const float>)a->g.vcache + f;
#pragma unroll
        for (int u = 0; u < kXRowsAhead; u++) {
            const unsigned at = (unsigned)(max(0, min(tb + slot + 4 * kXWaves * u, t1 - 1)) * kvd + kvcol);   // (past the split: its last row again, weight 0)
            k4[u] = __builtin_nontemporal_load((Global<const v4f>)(kc + at));
            v4[u] = __builtin_nontemporal_load((Global<const v4f>)(vc + at));
        }
    };

    request_q(0);
    if (item) request_kv(0, t0);
    request_o(0);
    request_13(0);
    request_2(0);
    {
        XcdArgsPtr a = xcd_args();
        for (int i = t; i < kSiluTable / 4; i += kXLanes) reinterpret_cast<v4f *>(lds + M::silu)[i] = ((Global<const v4f>)a->g.silu)[i];
    }
    const float rn = __fdiv_rn(1.0f, (float)dim);

    for (int l = 0; l < L; l++) {
        const int ln = min(l + 1, L - 1);   // (past the last layer: that one again, not used)
        __syncthreads();
        {
            float acc[1];
            RD::template fold<1>({&rq}, lds + M::xd0, cd, acc);
            XcdArgsPtr a = xcd_args();
            const float own = __fmul_rn(xcd_rms(lds + M::red, rn), acc[0]);
            const float other = dpp_f<0x128>(own);   // the other row of the pair: eight lanes on
            const float y = isq || isk ? __fadd_rn(__fmul_rn(own, cs.x), __fmul_rn(other, cs.y)) : own;
            const Global<float> q = (Global<float>)pinned(a->g.q) + so + l * sd, kn = (Global<float>)pinned(a->g.knew) + so + l * a->g.skv, vn = (Global<float>)pinned(a->g.vnew) + so + l * a->g.skv;
            const long row = ((long)l * a->g.seq_len + pos) * kvd;
            const Global<float> kc = (Global<float>)pinned(a->g.kcache) + row, vc = (Global<float>)pinned(a->g.vcache) + row;
            if (okq && cd == 0) {
                (isq ? q : isk ? kn : vn)[rowq] = y;
                if (!isq) (isk ? kc : vc)[rowq] = y;
            }
            request_q(ln);
        }
        if (item) {
            __syncthreads();
            // (lanes past the head read words that are not used: their results are selected, not their loads)
            const v4f *qkv = reinterpret_cast<const v4f *>(lds + M::qkv) + (lane & 15);
            const v4f q4 = qkv[0], kn = qkv[16], vn = qkv[32];
            auto score = [&](const v4f &k) {
                const float d = fmaf(q4[3], k[3], fmaf(q4[2], k[2], fmaf(q4[1], k[1], q4[0] * k[0])));
                return row16_sum(active ? d : 0.0f);
            };
            float m = -3.402823466e+38f, sum = 0.0f;
            v4f o = {0.f, 0.f, 0.f, 0.f};
            if (now && wave == 0) {   // this token's row: the first sixteen lanes
                m = readlane_f(score(kn), 0);
                sum = lane < 16 ? 1.0f : 0.0f;
#pragma unroll
                for (int e = 0; e < 4; e++) o[e] = lane < 16 ? vn[e] : 0.0f;
            }
            auto fold_rows = [&](int tb) {
                float sc[kXRowsAhead], mb = -3.402823466e+38f;
#pragma unroll
                for (int u = 0; u < kXRowsAhead; u++) {
                    sc[u] = -3.402823466e+38f;
                    if (tb + 4 * kXWaves * u + 4 * wave >= t1) continue;   // (uniform)
                    const float d = score(k4[u]);
                    sc[u] = tb + slot + 4 * kXWaves * u < t1 ? d : -3.402823466e+38f;
                    mb = fmaxf(mb, sc[u]);
                }
                mb = fmaxf(m, max_of_groups<16>(mb));
                // The four rows' weights and the rescaling factor with one exponential: sixteen lanes hold the same scores, so lanes 0 to 3 of
                // them take one row each, the others the maximum.
                const int j = lane & 15;
                const float w = expf((j == 0 ? sc[0] : j == 1 ? sc[1] : j == 2 ? sc[2] : j == 3 ? sc[3] : m) - mb);
                const float p4[kXRowsAhead] = {dpp_f<0x150>(w), dpp_f<0x151>(w), dpp_f<0x152>(w), dpp_f<0x153>(w)};   // row_newbcast
                const float k = readlane_f(w, 4);
                sum *= k;
                o *= k;
#pragma unroll
                for (int u = 0; u < kXRowsAhead; u++) {
                    if (tb + 4 * kXWaves * u + 4 * wave >= t1) continue;
                    const bool ok = tb + slot + 4 * kXWaves * u < t1;
                    const float p = ok ? p4[u] : 0.0f;
                    sum += p;
#pragma unroll
                    for (int e = 0; e < 4; e++) o[e] = fmaf(p, ok ? v4[u][e] : 0.0f, o[e]);   // K/AccumWeightedValue.java:48-62 (the repeated row may hold infinities)
                }
                m = mb;
            };
            if (t0 < t1) fold_rows(t0);
            for (int tb = t0 + kXSplitRows; tb < t1; tb += kXSplitRows) {
                request_kv(l, tb);
                fold_rows(tb);
            }
            request_kv(ln, t0);
            sum = sum_of_groups<16>(sum);
#pragma unroll
            for (int e = 0; e < 4; e++) o[e] = sum_of_groups<16>(o[e]);
            if (lane < 16) reinterpret_cast<v4f *>(lds + M::acc)[16 * wave + lane] = o;
            if (lane == 0) { lds[M::ml + 2 * wave] = m; lds[M::ml + 2 * wave + 1] = sum; }
            __syncthreads();
            if (wave == 0) {
                float ll[kXWaves], oo[kXWaves], top = -3.402823466e+38f, S = 0.0f, O = 0.0f;
                const float own = lds[M::ml + 2 * min(lane, kXWaves - 1)];   // the waves' maxima, one per lane
#pragma unroll
                for (int i = 0; i < kXWaves; i++) {
                    ll[i] = lds[M::ml + 2 * i + 1];
                    oo[i] = lds[M::acc + 64 * i + lane];
                    top = fmaxf(top, readlane_f(own, i));
                }
                const float w = expf(own - top);   // (a wave without rows: 0)
#pragma unroll
                for (int i = 0; i < kXWaves; i++) {
                    const float k = readlane_f(w, i);
                    S = fmaf(ll[i], k, S);
                    O = fmaf(oo[i], k, O);
                }
                XcdArgsPtr a = xcd_args();
                if (nact == 1) {
                    if (lane < hs) ((Global<float>)a->g.xb + so + l * sd + head * hs)[lane] = __fdiv_rn(O, S);
                } else {
                    const Global<float> part = (Global<float>)a->mem + set * a->mem_stride + ((long)(l * a->g.n_heads + head) * a->nsplit + split) * (hs + 4);
                    if (lane < hs) part[4 + lane] = O;
                    if (lane < 4) part[lane] = lane == 0 ? top : S;
                }
            }
        }
        __syncthreads();
        {
            float acc[1];
            RD::template fold<1>({&ro}, lds + M::xd1, cd, acc);
            const float y = __fadd_rn(lds[M::raw0 + rowo], acc[0]);   // K/Accum.java:26-30
            XcdArgsPtr a = xcd_args();
            if (oko && cd == 0) ((Global<float>)a->g.x + so + (2L * l + 1) * sd)[rowo] = y;
            request_o(ln);
        }
        __syncthreads();
        {
            float acc[2];
            RD::template fold<2>({&r1, &r3}, lds + M::xd0, cd, acc);
            XcdArgsPtr a = xcd_args();
            const float ss = xcd_rms(lds + M::red + 2, rn), h1 = __fmul_rn(ss, acc[0]), h3 = __fmul_rn(ss, acc[1]);
            const float y = __fmul_rn(h1, __fmul_rn(silu_sigma(lds + M::silu, h1, a->g.exact_silu), h3));   // K/Silu.java:72-74
            if (ok13 && cd == 0) ((Global<float>)a->g.hb + so + l * a->g.sh)[row13] = y;
            request_13(ln);
        }
        __syncthreads();
        {
            float acc[1];
            RH::template fold<1>({&r2}, lds + M::xh, ch, acc);
            const float y = __fadd_rn(lds[M::raw1 + row2], acc[0]);
            XcdArgsPtr a = xcd_args();
            if (ok2 && ch == 0) {
                const Global<float> o = (Global<float>)a->g.x + so + (2L * l + 2) * sd;
                if (l + 1 < L) o[row2] = y;
                else st_coh((float *)(o + row2), y);   // for the workgroups of the classifier, on the other XCDs
            }
            request_2(ln);
        }
    }
}

// The workgroups of the classifier: number id of ncls.
template <class C>
__device__ __forceinline__ void xcd_classifier(const XcdArgs &a, float *lds, int id, int ncls, int set)
{
    constexpr int NG = kXThreads / C::LC, NPRE = 3;
    static_assert(C::LC == 8, "the sums' exchanges between lanes");
    const TokenGeom &g = a.g;
    const int tid = threadIdx.x, dim = g.dim, n4 = dim >> 2, gc = tid / C::LC, cl = tid % C::LC, xcd = blockIdx.x % kXcds;
    const Poll pl{1, a.maxspin, g.fault};
    {   // the vectors of the token after this one
        const v4f uv = {__uint_as_float(kUnset), __uint_as_float(kUnset), __uint_as_float(kUnset), __uint_as_float(kUnset)};
        float4 *p0 = reinterpret_cast<float4 *>(g.x + (1 - set) * g.set_stride), *p1 = reinterpret_cast<float4 *>(a.mem + (1 - set) * a.mem_stride);
        const long n0 = g.set_stride >> 2, n = n0 + (a.mem_stride >> 2);
        for (long i = (long)id * kXThreads + tid; i < n; i += (long)ncls * kXThreads)
            asm volatile("global_store_dwordx4 %0, %1, off sc0 sc1\n\ts_nop 2" ::"v"(i < n0 ? p0 + i : p1 + (i - n0)), "v"(uv) : "memory");   // (wait states: a 16-byte store reads its data registers after it has issued)
    }
    const int per = (g.vocab + ncls - 1) / ncls, r0 = id * per, r1 = min(g.vocab, r0 + per);
    float4 w[NPRE][C::FC];
    auto request = [&](int i, int p) {
        const float4 *wr = reinterpret_cast<const float4 *>(g.wcls + (long)min(r0 + gc + p * NG, g.vocab - 1) * dim);
#pragma unroll
        for (int u = 0; u < C::FC; u++) w[i][u] = load_stream(wr + min(cl + C::LC * u, n4 - 1));
    };
#pragma unroll
    for (int i = 0; i < NPRE; i++) request(i, i);
    // the last vector: one workgroup of each XCD brings it there
    float *mine = a.mem + set * a.mem_stride + xcd_part_floats(g.n_layers, g.n_heads, a.nsplit, g.head_size) + xcd * g.sd;
    if (blockIdx.x / kXcds == 0 && tid < n4) {
        const float *p[1] = {g.x + set * g.set_stride + 2L * g.n_layers * g.sd + 4 * tid};
        float4 v[1];
        xwait<1>(p, v, pl);
        reinterpret_cast<float4 *>(mine)[tid] = v[0];
    }
    float4 *xs = reinterpret_cast<float4 *>(lds);
    const int nch = dim >> 4;
    float *sumx = lds + dim, *red = sumx + nch;
    const float ss = stage_vector_poll<1>(mine, dim, g.rmsw + 2L * g.n_layers * dim, xs, sumx, red, kXThreads, pl);
    float best_v = -__builtin_inff();
    int best_i = 0x7fffffff;
    for (int p0 = 0; r0 + p0 * NG < r1; p0 += NPRE) {
#pragma unroll
        for (int i = 0; i < NPRE; i++) {
            float acc = 0.0f;
#pragma unroll
            for (int u = 0; u < C::FC; u++) {
                const int c = cl + C::LC * u, cc = min(c, n4 - 1);
                const float t = dot4(w[i][u], xs[(cc & 3) * nch + (cc >> 2)]);
                acc += c < n4 ? t : 0.0f;
            }
            acc += dpp_f<0xB1>(acc);
            acc += dpp_f<0x4E>(acc);
            acc += dpp_f<0x141>(acc);   // (row_half_mirror: eight lanes)
            const int row = r0 + gc + (p0 + i) * NG;
            acc = __fmul_rn(ss, acc);
            if (row < r1 && cl == 0) {
                g.logits[row] = acc;
                if (better(acc, row, best_v, best_i)) { best_v = acc; best_i = row; }
            }
            if (r0 + (p0 + i + NPRE) * NG < r1) request(i, p0 + i + NPRE);   // (uniform)
        }
    }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
        const float ov = __shfl_xor(best_v, off);
        const int oi = __shfl_xor(best_i, off);
        if (better(ov, oi, best_v, best_i)) { best_v = ov; best_i = oi; }
    }
    __syncthreads();   // (the norm's sums have been read)
    float *bval = red;
    int *bidx = reinterpret_cast<int *>(red) + 16;
    if ((tid & 63) == 0) { bval[tid >> 6] = best_v; bidx[tid >> 6] = best_i; }
    __syncthreads();
    if (tid == 0) {
        for (int i = 1; i < kXThreads / 64; i++)
            if (better(bval[i], bidx[i], best_v, best_i)) { best_v = bval[i]; best_i = bidx[i]; }
        st_coh(g.cls_part + id, pack_max(best_v, best_i));
    }
}

template <class C>
static __global__ void __launch_bounds__(kXThreads, 2) k_xtoken(const XcdArgs a)
{
    __shared__ float4 smem4[XLds<C>::end / 4];
    float *lds = reinterpret_cast<float *>(smem4);
    const int token = a.g.st->token, pos = a.g.st->pos, set = a.g.st->epoch & 1;
    const int nwork = gridDim.x / kXcds, ncls = gridDim.x - nwork, xcd = blockIdx.x % kXcds, i = blockIdx.x / kXcds;
    if (xcd != 0) {
        xcd_classifier<C>(a, lds, i * (kXcds - 1) + xcd - 1, ncls, set);
        return;
    }
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    if (wave < kXWaves) xcd_layers<C>(lds, i, nwork, threadIdx.x, pos, set);
    else xcd_stage_layers<C>(lds, i, threadIdx.x - kXLanes, token, pos, set);
    if (i == 0) {
        ClsPhase cp{};
        cp.part = a.g.cls_part; cp.nparts = ncls; cp.st = a.g.st; cp.prompt = a.g.prompt; cp.out_tokens = a.g.out_tokens; cp.tstamp = a.g.tstamp;
        cp.poll = Poll{1, a.maxspin, a.g.fault};
        token_finish(cp, smem4);
    }
}

}  // namespace l2j
