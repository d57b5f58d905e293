// Products of the quantized matrices with many activation vectors on the int8 matrix cores.
//
// An fp32 activation is written as a fixed-point number: per vector and group of 256 (the weights' groups) a power of two
// 2^s brings the largest magnitude of the group into [2^29, 2^30), x = q * 2^-s with an integer q, and q is four signed
// digits to the base 256, which v_mfma_i32_16x16x64_i8 multiplies by the codes (less 128: signed bytes) and adds up
// exactly.  Every activation that is not 64 times smaller than the largest of its group keeps all 24 bits of its
// significand, and none is off by more than 2^-30 of that largest one; the sum over a group is exact, where a sum of fp32
// products rounds at every addition (K/MatMul.java:117-151 is the loop this restates).  Groups are added in fp32.
// Against three bf16 planes per activation (the exact cut this replaces): four products at twice the rate instead of
// three, and no conversion of the codes, whose bytes go into the matrix cores as they lie in memory.
#pragma once

#include "kernels.hpp"

#include <utility>

namespace l2j {

typedef int v4i __attribute__((ext_vector_type(4)));
typedef float v2f __attribute__((ext_vector_type(2)));

constexpr int kRowTile = 32;                       // activation vectors per tile: two MFMAs of 16
constexpr int kDigitBytes = 4 * 4 * 2 * 64 * 16;   // digits of a (tile, group): [digit][64 k][half of the tile][lane][16], most significant digit first

// The digits of `rows` activation vectors of length K, in the order the matrix cores take them, with the groups' scales
// 2^-s and sums.  Tiles of 32 vectors; the vectors past the last one hold anything finite.
struct Digits {
    uint4 *d;      // (tile, group) x kDigitBytes; lane l of a block of 64 k: vector l % 16 of the half, k = 16 (l / 16) + 0..15
    float *sx;     // (tile, group, 32): 2^-s (NaN: the group holds a NaN or an infinity)
    float *sum;    // (tile, group, 32): the sum of the group's activations
};

__host__ __device__ inline size_t digit_tiles(int rows) { return (size_t)(rows + kRowTile - 1) / kRowTile; }

// The exponent s for a group whose largest magnitude has the bits `amax` (sign cleared), and 2^-s.
__device__ __forceinline__ int digit_shift(unsigned amax, float *inv)
{
    // 2^e <= amax < 2^(e+1): s = 29 - e, no larger than 149 (below 2^-120 every float is a multiple of the step 2^-149)
    const int e = (int)(amax >> 23) - 127;
    const int s = min(29 - e, 149);
    *inv = amax >= 0x7f800000u ? __uint_as_float(0x7fc00000u) : amax == 0u ? 1.0f : ldexpf(1.0f, -s);
    return s;
}

// Sixteen consecutive activations of a vector as digits, x[d] their digits d (0: the most significant); s: the group's exponent.
__device__ __forceinline__ void make_digits(const float (&v)[16], int s, v4i (&x)[4])
{
    unsigned w[16];
#pragma unroll
    for (int i = 0; i < 16; i++) {
        // (a group with a NaN or an infinity: any digits, its scale is a NaN)
        const int q = (int)rintf(ldexpf(v[i], s));
        w[i] = ((unsigned)q + 0x80808080u) ^ 0x80808080u;   // byte d: digit d, -128 .. 127
    }
#pragma unroll
    for (int d = 0; d < 4; d++) {   // byte 3 - d of every word
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const unsigned sel = 0x0c0c0400u + (unsigned)((3 - d) * 0x0101u);
            const unsigned lo = __builtin_amdgcn_perm(w[4 * i + 1], w[4 * i], sel), hi = __builtin_amdgcn_perm(w[4 * i + 3], w[4 * i + 2], sel);
            x[d][i] = (int)__builtin_amdgcn_perm(hi, lo, 0x05040100u);
        }
    }
}

// Those of vector `row`, k = 16 c .. 16 c + 15 of group g, to their place.
__device__ __forceinline__ void store_digits(const Digits &o, int row, int ngroups, int g, int c, const float (&v)[16], int s)
{
    v4i x[4];
    make_digits(v, s, x);
    v4i *p = reinterpret_cast<v4i *>(o.d) + ((size_t)(row >> 5) * ngroups + g) * (kDigitBytes / 16) + (2 * (c >> 2) + ((row >> 4) & 1)) * 64 + (row & 15) + 16 * (c & 3);
#pragma unroll
    for (int d = 0; d < 4; d++) p[d * 8 * 64] = x[d];
}

// max and sum over the sixteen lanes that hold a group (lanes 16 n .. 16 n + 15)
__device__ __forceinline__ unsigned amax16(const float (&v)[16])
{
    unsigned m = 0;
#pragma unroll
    for (int i = 0; i < 16; i++) m = max(m, __float_as_uint(v[i]) & 0x7fffffffu);
#pragma unroll
    for (int off = 1; off < 16; off <<= 1) m = max(m, (unsigned)__shfl_xor((int)m, off));
    return m;
}

__device__ __forceinline__ float sum16(const float (&v)[16])
{
    float t = 0.0f;
#pragma unroll
    for (int i = 0; i < 16; i += 4) t += (v[i] + v[i + 1]) + (v[i + 2] + v[i + 3]);
    return row16_sum(t);
}

// A group of vector `row` held by sixteen lanes, sixteen activations each (lane % 16 = c): digits, scale and sum.
__device__ __forceinline__ void quantize_group(const Digits &o, int row, int ngroups, int g, int c, const float (&v)[16])
{
    float inv;
    const int s = digit_shift(amax16(v), &inv);
    const float t = sum16(v);
    store_digits(o, row, ngroups, g, c, v, s);
    if (c == 0) {
        const size_t at = ((size_t)(row >> 5) * ngroups + g) * 32 + (row & 31);
        o.sx[at] = inv;
        o.sum[at] = t;
    }
}

// A group of vector `row` held by the whole wave, four consecutive activations per lane (k = 4 lane ..): digits, scale and sum.
__device__ __forceinline__ void quantize_wave(const Digits &o, int row, int ngroups, int g, int lane, const v4f &v)
{
    unsigned m = 0;
#pragma unroll
    for (int i = 0; i < 4; i++) m = max(m, __float_as_uint(v[i]) & 0x7fffffffu);   // (as bits: a NaN is the largest)
    m = max(m, dpp_u<0xB1>(m));
    m = max(m, dpp_u<0x4E>(m));
    m = max(m, dpp_u<0x124>(m));
    m = max(m, dpp_u<0x128>(m));
    auto at = [&](int l) { return (unsigned)__builtin_amdgcn_readlane((int)m, l); };
    m = max(max(at(0), at(16)), max(at(32), at(48)));
    float inv;
    const int s = digit_shift(m, &inv);
    const float t = wave_sum((v[0] + v[1]) + (v[2] + v[3]));
    unsigned w[4];
#pragma unroll
    for (int i = 0; i < 4; i++) w[i] = ((unsigned)(int)rintf(ldexpf(v[i], s)) + 0x80808080u) ^ 0x80808080u;   // (as store_digits)
    const int c = lane >> 2;
    unsigned *p = reinterpret_cast<unsigned *>(o.d + ((size_t)(row >> 5) * ngroups + g) * (kDigitBytes / 16) + (2 * (c >> 2) + ((row >> 4) & 1)) * 64 + (row & 15) + 16 * (c & 3)) + (lane & 3);
    // (a transpose within four lanes, for one 16-byte store per lane instead of four of 4 bytes, gains nothing)
#pragma unroll
    for (int d = 0; d < 4; d++) {   // byte 3 - d of every word
        const unsigned sel = 0x0c0c0400u + (unsigned)((3 - d) * 0x0101u);
        p[d * 8 * 64 * 4] = __builtin_amdgcn_perm(__builtin_amdgcn_perm(w[3], w[2], sel), __builtin_amdgcn_perm(w[1], w[0], sel), 0x05040100u);
    }
    if (lane == 0) {
        const size_t q = ((size_t)(row >> 5) * ngroups + g) * 32 + (row & 31);
        o.sx[q] = inv;
        o.sum[q] = t;
    }
}

// The sum of a product's slices at consecutive columns (V: float2, v4f), added in slice order: up to four, or eight at a time,
// with all loads in flight (past the last slice: that one again, not added).
template <int N, class V>
__device__ __forceinline__ void add_slices(V &t, const float *__restrict__ part, int s0, int slices, size_t stride)
{
    V v[N];
#pragma unroll
    for (int i = 0; i < N; i++) v[i] = *reinterpret_cast<const V *>(part + min(s0 + i, slices - 1) * stride);
#pragma unroll
    for (int i = 0; i < N; i++)
        if (s0 + i < slices) t += v[i];
}

template <class V>
__device__ __forceinline__ V sum_slices(const float *__restrict__ part, int slices, size_t stride)
{
    V t = {};
    if (slices == 1) return t + *reinterpret_cast<const V *>(part);   // (-0 + 0 = +0, as the sum of several)
    if (slices <= 4) {
        add_slices<4>(t, part, 0, slices, stride);
    } else {
        for (int s = 0; s < slices; s += 8) add_slices<8>(t, part, s, slices, stride);
    }
    return t;
}

struct DGemm {
    const uint8_t *codes[3];   // the matrices of one layer in tile order (k_btile): codes less 128
    const float2 *gs[3];       // (rm, min + 128 rm) in tile order
    int tiles[3];              // 16-row tiles of each; the matrices' rows follow each other in the output
    int ntiles;                // all of them
    int ngroups;               // K / 256
    int gps;                   // groups per slice of K
    Digits x;
    int npos;                  // vectors
    float *out;                // (slice, npos, 16 * ntiles)
    int ncol, nrow;            // tiles of the grid: vectors, matrix rows
    const float *silu;         // k_dstream with SwiGLU: the sigmoid table, and whether to do without it
    int exact;
};

constexpr int kDgWaveRows = 64;   // matrix rows per wave

template <int PT> __host__ __device__ constexpr size_t dgemm_lds() { return (size_t)2 * PT * (kDigitBytes + 128); }

// f(0), ..., f(N - 1) with the numbers as constants
template <class F, int... I> __device__ __forceinline__ void unroll_seq(F &&f, std::integer_sequence<int, I...>) { (f(std::integral_constant<int, I>{}), ...); }
template <int N, class F> __device__ __forceinline__ void unroll(F &&f) { unroll_seq(f, std::make_integer_sequence<int, N>{}); }

// A load at a uniform address plus 32 bits per lane (held as such: the compiler otherwise keeps 64-bit sums in vector registers).
template <class T> __device__ __forceinline__ T load_at(const void *base, unsigned &off)
{
    typedef const __attribute__((address_space(1))) char *P;
    P p = (P)base;
    asm volatile("" : "+s"(p), "+v"(off));
    return *reinterpret_cast<const __attribute__((address_space(1))) T *>(p + off);
}

// The order in which unit u of NU (16 vectors against the wave's 64 rows) takes its sixteen fragments of digits: step j is digit
// dg_digit and block of 64 k dg_block.  First and third digits before second and fourth, each pair's sums being shifted in between;
// the first unit of a group begins, and the last one ends, with the two digits of a block of 64 k next to each other, so that the
// codes of a block are needed 24 matrix instructions after they were free to be requested instead of 12.
__device__ constexpr int dg_digit(int u, int nu, int j) { return u == 0 && j < 8 ? 2 * (j & 1) : u == nu - 1 && j >= 8 ? 1 + 2 * (j & 1) : (j >> 2) == 1 ? 2 : (j >> 2) == 2 ? 1 : j >> 2; }
__device__ constexpr int dg_block(int u, int nu, int j) { return u == 0 && j < 8 ? j >> 1 : u == nu - 1 && j >= 8 ? (j - 8) >> 1 : j & 3; }

// A workgroup takes 64 NW rows of the matrix x 32 PT vectors x one slice of K.  A wave holds the codes of its 64 rows of a
// group in registers (read once from memory, 1 KB per load) and multiplies them by the digits of the vectors, which the
// workgroup stages in LDS a group ahead (straight from memory: no registers, no writes of its own); the digits of an output are
// summed 256 * first + second in one accumulator, third and fourth in another.  (16 x 16 tiles: on random digits and codes of standard
// deviation 40, operands in registers, two waves per SIMD, v_mfma_i32_16x16x64_i8 sustains 4.0 POP/s over 40 ms and
// v_mfma_i32_32x32x32_i8 2.9: the clock drops under the matrix cores' load.)
// What a unit of 16 vectors leaves is converted, scaled and added between the matrix instructions of the next one, two vector
// instructions beside each: alone that many cost it 9 % (9.4 -> 10.2 ns each, two waves per SIMD), in a block of their own behind the
// matrix instructions, where both waves of a SIMD come at once behind a barrier, their whole time.  Inside passes of the 7B
// shape, us, Wq+Wk+Wv, Wo, W1+W3, W2: 1024 vectors 183 61.6 341 154 -> 179 60.0 329 148 (2.2 POP/s), 448 95.3 35.7 166 79.5 -> 93.5 35.5
// 160 78.1, 64 24.6 13.8 40.9 23.2 -> 24.4 14.3 41.3 22.9.  (The digits joined before the running sum, four operations less per row, were
// 1 to 1.5 % faster still, but rounded elsewhere.)  A group of 64 vectors then takes 11000 cycles at 1.9 GHz, 8192 of them
// matrix instructions; without the codes' loads 0.9 of the time, without the digits' 0.95.  Tried, no faster: codes a whole group ahead in
// a second set of registers (32 vectors: 3 % slower, it is bound by the codes' way through L2), workgroups that go on to
// another tile instead of ending, sums stored four rows at a time by way of LDS.
// dgemm_tile: the vectors' tile `col`, rows and slice `tile` of the launch.  NU: units of 16 vectors, 2 PT, or 1 of a tile of 32 whose second
// half is empty.  (The argument by value: behind a reference the addresses came out in vector registers.)
template <int PT, int NW, int NU>
__device__ __forceinline__ void dgemm_tile(const DGemm a, v4i *dg_lds, int tile, int col)
{
    constexpr int STAGE = PT * kDigitBytes / 16;            // 16-byte words of a group's digits
    constexpr int NT = 64 * NW, NST = STAGE / NT * NU / (2 * PT);   // words a thread stages per group,
    constexpr int U1 = NU > 1 ? 1 : 0, PER = (NST + NU - 1 - U1) / (NU - U1);   // in the units behind the first (of one: in it), so many in each, one a step
    // The wait at a group's end leaves sixteen loads under way and takes them for the next codes, which are requested from the last unit's tenth step on:
    // every word has to be requested before.
    static_assert(STAGE % NT == 0 && STAGE / NT * NU % (2 * PT) == 0 && PER <= 9, "digits would be read before they are staged");
    float *lsx = reinterpret_cast<float *>(dg_lds + 2 * STAGE);   // [2][32 PT]
    constexpr int RUN = NU == 2 * PT ? 64 : 128;             // the wave's q-th run of 64 words begins at (q NW + wave) RUN (one unit: the runs of the tile's first half)
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), s4 = lane >> 4, n = lane & 15;
    const int nslice = (a.ngroups + a.gps - 1) / a.gps;
    const int rt = __builtin_amdgcn_readfirstlane(tile / nslice), slice = tile - rt * nslice;
    const int g0 = slice * a.gps, g1 = min(g0 + a.gps, a.ngroups);
    // The wave's 64 rows lie in one matrix (with several matrices: rows % 64 == 0): its address is uniform.  (Rows past the
    // matrix's last tile of 16 repeat that tile and are not stored.)
    const int row0 = (rt * NW + wave) * kDgWaveRows;
    int t = min(row0 >> 4, a.ntiles - 1), m = 0, nt = a.tiles[0];
    if (t >= nt) { t -= nt; m = 1; nt = a.tiles[1]; if (t >= nt) { t -= nt; m = 2; nt = a.tiles[2]; } }
    const uint8_t *cm = m == 0 ? a.codes[0] : m == 1 ? a.codes[1] : a.codes[2];
    const float2 *sm = m == 0 ? a.gs[0] : m == 1 ? a.gs[1] : a.gs[2];
    const uint8_t *cp[4];
    const float2 *sp[4];
#pragma unroll
    for (int r = 0; r < 4; r++) {
        const size_t blk = (size_t)min(t + r, nt - 1) * a.ngroups + g0;
        cp[r] = cm + blk * 4096;
        sp[r] = sm + blk * 16;
    }
    unsigned co = lane * 16, n8 = n * 8, stage16 = (wave * RUN + lane) * 16;
    const v4i *xd = reinterpret_cast<const v4i *>(a.x.d) + ((size_t)col * PT * a.ngroups + g0) * (kDigitBytes / 16);
    const size_t xstep = (size_t)a.ngroups * (kDigitBytes / 16);   // 16-byte words between two tiles of vectors
    const float *xs = a.x.sx + ((size_t)col * PT * a.ngroups + g0) * 32;
    const int xt = tid & (32 * PT - 1);   // (every wave stages the scales: no branch in the loop)
    unsigned xso = ((xt >> 5) * a.ngroups * 32 + (xt & 31)) * 4;

    // codes of the first group
    v4i cw[4][4];
#pragma unroll
    for (int T = 0; T < 4; T++)
#pragma unroll
        for (int r = 0; r < 4; r++) cw[r][T] = load_at<v4i>(cp[r] + 1024 * T, co);
    // digits of the first group, its vectors' and its rows' scales
    float sx0, rm[4], rmp[4] = {0.f, 0.f, 0.f, 0.f};   // (rmp: the rows' scales of the group before)
    {
        v4i st[NST];
#pragma unroll
        for (int q = 0; q < NST; q++) st[q] = (xd + (q * NW * RUN / 2048) * xstep + q * NW * RUN % 2048)[stage16 / 16];
        sx0 = load_at<float>(xs, xso);
#pragma unroll
        for (int r = 0; r < 4; r++) rm[r] = load_at<float>(sp[r], n8);
#pragma unroll
        for (int q = 0; q < NST; q++) dg_lds[(q * NW + wave) * RUN + lane] = st[q];
    }
    // the groups' offsets times the sums of the activations: fp32 matrix cores, four groups at a time
    v4f f0[NU][4];
#pragma unroll
    for (int u = 0; u < NU; u++)
#pragma unroll
        for (int r = 0; r < 4; r++) f0[u][r] = v4f{0.f, 0.f, 0.f, 0.f};
    for (int g = g0; g < g1; g += 4) {
        const bool on = g + s4 < g1;
        const int gg = on ? s4 : 0;
        float b[4];
#pragma unroll
        for (int r = 0; r < 4; r++) { const float v = (sp[r] + (size_t)(g - g0) * 16)[gg * 16 + n].y; b[r] = on ? v : 0.0f; }
#pragma unroll
        for (int u = 0; u < NU; u++) {
            const float v = (a.x.sum + ((size_t)(col * PT + (u >> 1)) * a.ngroups + g) * 32 + 16 * (u & 1))[gg * 32 + n];
            const float s = on ? v : 0.0f;
#pragma unroll
            for (int r = 0; r < 4; r++) f0[u][r] = __builtin_amdgcn_mfma_f32_16x16x4f32(s, b[r], f0[u][r], 0, 0, 0);
        }
    }
    float f[NU][4][4];
#pragma unroll
    for (int u = 0; u < NU; u++)
#pragma unroll
        for (int r = 0; r < 4; r++)
#pragma unroll
            for (int e = 0; e < 4; e++) f[u][r][e] = f0[u][r][e];
    // Where 2^-s of some vector is so small that its product with a matrix's scale would lose bits (below 2^-126), all sums are kept
    // times 2^48 from that group on, unless a group of some vector is so large that this might carry its sum past the largest
    // float.  (2^-s into the sum of digits instead, as k_dstream has it, was one product more behind the matrix cores: W1 and W3
    // of the 7B shape with 1024 vectors 330 -> 336 us; the vectors looked through ahead 330 -> 335.)  Every wave holds the 2^-s of all
    // the workgroup's vectors, so all come to the same power.
    const bool live = col * PT * 32 + xt < a.npos;
    float up = 1.0f;
    bool large = false;
    auto keep = [&](float x, auto pending) {   // pending(): what the sums kept so far still lack
        x = live ? x : 1.0f;
        if (__any(!(x >= 0x1p-64f && x <= 0x1p20f))) {
            large |= __any(x > 0x1p20f) != 0;
            const float k = large ? 1.0f : __any(x < 0x1p-64f) ? 0x1p48f : up;
            if (k != up) {
                const float by = k > up ? 0x1p48f : 0x1p-48f;
                pending();
#pragma unroll
                for (int u = 0; u < NU; u++)
#pragma unroll
                    for (int r = 0; r < 4; r++)
#pragma unroll
                        for (int e = 0; e < 4; e++) f[u][r][e] *= by;
                up = k;
            }
        }
        return x * up;
    };
    lsx[xt] = keep(sx0, [] {});
    __syncthreads();
    __builtin_amdgcn_s_waitcnt(0x0f70);   // vmcnt(0): (a load under way here would be waited for in every round of the loop)

    // The accumulators of two units in turn, and what adding up a unit takes: 96 operations, six for each of four rows' four values.
    // The high and the low digits go into the running sum one after the other, the high ones times 65536 r_m: joined first, they would share
    // a factor sixteen powers of two nearer to 2^-126, and every sum round elsewhere.  Operation o of unit v, whose vectors' scales are sx
    // and whose rows' are r_m:
    v4i hi[2][4], lo[2][4];
#pragma unroll
    for (int k = 0; k < 2; k++)
#pragma unroll
        for (int r = 0; r < 4; r++) { hi[k][r] = v4i{0, 0, 0, 0}; lo[k][r] = v4i{0, 0, 0, 0}; }
    v4f sxp = {0.f, 0.f, 0.f, 0.f};   // the scales of the unit whose sums are still to be added
    float eh[4], el[4], mh[4], ml[4], rh;
    auto add_up = [&](auto oc, auto vc, const v4f &sx, const float (&r_m)[4]) __attribute__((always_inline)) {
        constexpr int o = oc.value, v = vc.value;
        if constexpr (o < 96) {
            constexpr int r = o / 24, what = o % 24 / 4, e = o % 4, k = v & 1;
            if constexpr (o % 24 == 0) rh = r_m[r] * 65536.0f;
            if constexpr (what == 0) eh[e] = (float)hi[k][r][e];
            else if constexpr (what == 1) mh[e] = rh * sx[e];
            else if constexpr (what == 2) el[e] = (float)lo[k][r][e];
            else if constexpr (what == 3) ml[e] = r_m[r] * sx[e];
            else if constexpr (what == 4) f[v][r][e] = fmaf(eh[e], mh[e], f[v][r][e]);
            else f[v][r][e] = fmaf(el[e], ml[e], f[v][r][e]);
        }
    };
    const unsigned lds0 = (unsigned)(uintptr_t)(__attribute__((address_space(3))) v4i *)dg_lds;
    const int ng = g1 - g0;
    for (int g = 0; g < ng; g++) {
        const v4i *cur = dg_lds + (g & 1) * STAGE + lane;
        const float *csx = lsx + (g & 1) * 32 * PT;
        const int gn = min(g + 1, ng - 1);                    // (past the last group: that group again, not used)
        const v4i *xn = xd + (size_t)gn * (kDigitBytes / 16);
        // The next group's digits on their way into the other buffer, a KB per wave and instruction (m0: where in LDS; the lanes'
        // 16 bytes follow each other).  Nothing the compiler counts: they come behind the codes of this group, which it waits for one by one,
        // and are waited for below.
        auto stage = [&](int q) __attribute__((always_inline)) {
            const v4i *from = xn + (q * NW * RUN / 2048) * xstep + q * NW * RUN % 2048;
            const unsigned to = lds0 + (((g + 1) & 1) * STAGE + q * NW * RUN + wave * RUN) * 16;
            asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" :: "s"(to), "v"(stage16), "s"(from) : "memory", "m0");
        };
        v4i x[4];   // fragments, three ahead of their use
        auto fragment = [&](int u, int j) __attribute__((always_inline)) {
            return cur[(u >> 1) * (kDigitBytes / 16) + dg_digit(u, NU, j) * 512 + (2 * dg_block(u, NU, j) + (u & 1)) * 64];
        };
        x[0] = fragment(0, 0); x[1] = fragment(0, 1); x[2] = fragment(0, 2);
        const float nsx = load_at<float>(xs + gn * 32, xso);
        float rmn[4];
#pragma unroll
        for (int r = 0; r < 4; r++) rmn[r] = load_at<float>(sp[r] + (size_t)gn * 16, n8);
        __builtin_amdgcn_sched_barrier(0);
        unroll<NU>([&](auto uc) __attribute__((always_inline)) {
            constexpr int u = uc.value, k = u & 1;
            typedef std::integral_constant<int, (u + NU - 1) % NU> Before;
            const v4f sx = *reinterpret_cast<const v4f *>(csx + 16 * u + 4 * s4);
            unroll<16>([&](auto jc) __attribute__((always_inline)) {
                constexpr int j = jc.value, d = dg_digit(u, NU, j), T = dg_block(u, NU, j), at = 16 * u + j;
                if constexpr (u >= U1 && j < PER && (u - U1) * PER + j < NST) stage((u - U1) * PER + j);
                if constexpr (at + 3 < 16 * NU) x[(at + 3) & 3] = fragment((at + 3) >> 4, (at + 3) & 15);
                unroll<4>([&](auto rc) __attribute__((always_inline)) {
                    constexpr int r = rc.value, i = 4 * j + r;
                    v4i &acc = (d & 2) ? lo[k][r] : hi[k][r];
                    acc = __builtin_amdgcn_mfma_i32_16x16x64_i8(x[at & 3], cw[r][T], !(d & 1) && T == 0 ? v4i{0, 0, 0, 0} : acc, 0, 0, 0);
                    // beside it the unit before (one unit: nothing, its sums are added up behind it), and the shifts between the digits of a pair:
                    // about two vector instructions each
                    constexpr int o = NU == 1 ? 96 : i < 16 ? 2 * i : i < 48 ? 16 + i : 2 * i - 32;
                    add_up(std::integral_constant<int, o>{}, Before{}, sxp, u == 0 ? rmp : rm);
                    if constexpr (i < 16 || i >= 48) add_up(std::integral_constant<int, o + 1>{}, Before{}, sxp, u == 0 ? rmp : rm);
                    if constexpr (u == 0 && j == 7) hi[k][r] <<= 8;
                    if constexpr (u != 0 && j >= 4 && j < 8) hi[k][j - 4][r] <<= 8;
                    if constexpr (u == NU - 1 && j == 8) lo[k][r] <<= 8;
                    if constexpr (u != NU - 1 && j >= 8 && j < 12) lo[k][j - 8][r] <<= 8;
                    __builtin_amdgcn_sched_barrier(0);
                });
                if constexpr (u == NU - 1 && j >= 8 && (j & 1)) {   // (the last use of these codes: the next group's in their place)
#pragma unroll
                    for (int r = 0; r < 4; r++) cw[r][T] = load_at<v4i>(cp[r] + (size_t)gn * 4096 + 1024 * T, co);
                }
            });
            sxp = sx;
            __builtin_amdgcn_sched_barrier(0);
        });
        if constexpr (NU == 1) unroll<96>([&](auto oc) __attribute__((always_inline)) { add_up(oc, std::integral_constant<int, 0>{}, sxp, rm); });
#pragma unroll
        for (int r = 0; r < 4; r++) { rmp[r] = rm[r]; rm[r] = rmn[r]; }
        lsx[((g + 1) & 1) * 32 * PT + xt] = keep(nsx, [&] {
            if constexpr (NU > 1) {
                unroll<96>([&](auto oc) __attribute__((always_inline)) { add_up(oc, std::integral_constant<int, NU - 1>{}, sxp, rmp); });
                sxp = v4f{0.f, 0.f, 0.f, 0.f};
            }
        });
        asm volatile("s_waitcnt vmcnt(16)" ::: "memory");   // (the staged digits: all but the sixteen loads of codes behind them)
        __syncthreads();
    }
    if constexpr (NU > 1) unroll<96>([&](auto oc) __attribute__((always_inline)) { add_up(oc, std::integral_constant<int, NU - 1>{}, sxp, rmp); });
    const int ldo = 16 * a.ntiles;
    const float down = up == 1.0f ? 1.0f : 0x1p-48f;
#pragma unroll
    for (int u = 0; u < NU; u++)
#pragma unroll
        for (int e = 0; e < 4; e++) {
            const int pos = (col * 2 * PT + u) * 16 + 4 * s4 + e;
            if (pos < a.npos) {
                float *o = a.out + ((size_t)slice * a.npos + pos) * ldo;
#pragma unroll
                for (int r = 0; r < 4; r++)
                    if (row0 + 16 * r + n < ldo) o[row0 + 16 * r + n] = f[u][r][e] * down;
            }
        }
}

// Of a last tile of 32 vectors whose second half is empty only the first unit is multiplied, and staged: a third of the work at 77 vectors
// had been for padding.  Wq+Wk+Wv, Wo, W1+W3, W2 inside passes of the 7B shape, us, 40 vectors 24.2 13.2 41.5 21.8 -> 21.2 12.2 35.4 19.4, 77 vectors
// 29.9 17.3 50.7 28.6 -> 27.2 16.4 47.6 25.7, 144 vectors 38.2 19.0 66.6 39.3 -> 35.8 18.5 61.2 36.0.  (The launches are picked as for whole tiles:
// within 2.3 % of the best on average; an estimate with half a tile in it does worse.)
template <int PT, int NW>
__global__ void __launch_bounds__(64 * NW, 2) k_dgemm(const DGemm a)
{
    extern __shared__ __align__(16) v4i dg_lds[];
    // The workgroups of an XCD (blockIdx % 8) take the same rows of the matrix against all vectors, one after the other.
    const int xcd = blockIdx.x & 7, i = blockIdx.x >> 3;
    const int row = __builtin_amdgcn_readfirstlane(i / a.ncol), tile = row * 8 + xcd, col = i - row * a.ncol;    // (tile: of rows and slices)
    if (tile >= a.nrow * ((a.ngroups + a.gps - 1) / a.gps)) return;
    if (PT == 1 && a.npos - 32 * col <= 16) dgemm_tile<PT, NW, PT == 1 ? 1 : 2 * PT>(a, dg_lds, tile, col);
    else dgemm_tile<PT, NW, 2 * PT>(a, dg_lds, tile, col);
}

// ---- at most 32 vectors: a decode step of a batch ---------------------------------------------------------------------

constexpr int kStreamWaves = 8, kStreamGroups = kStreamWaves / 2;   // groups per slice of K: two waves each
template <int NB> __host__ __device__ constexpr size_t dstream_lds() { return (size_t)2 * kStreamWaves * NB * 512 * sizeof(float); }

// With at most 32 vectors a product is bound by the codes' way from memory and, launch by launch, by the way in and out (7B shape, 32
// vectors: 57 us for the 208 MB of a layer's four products, 3.6 TB/s; 4.7 us of a launch are not tiles), and the digits are what is
// reused: a wave owns half a group of the slice (128 k) and keeps its digits of all 16 NB vectors in registers for the whole launch,
// while the codes of 32 matrix rows after another stream past, requested a tile ahead.  The waves' sums of a tile meet in LDS (two
// buffers in turn, one barrier per tile) and are added up while the next tile's products run.
// That order, request addresses that need no vector registers and the instantiation without the loop, W1 and W3 / Wq, Wk and Wv /
// W2 / Wo of the 7B shape: 22.4 -> 20.8, 15.2 -> 14.7, 14.8 -> 13.9, 8.1 -> 8.0 us, those of the 110M shape 5.0 -> 4.6.  Codes two tiles
// ahead instead: 3 to 5 % slower (the requests past the end, of which a workgroup with two tiles then makes two).
// TILES: the most tiles a workgroup has, 0 for any number.  One (every product of the 110M shape): no codes requested ahead, no copy of the
// loop to fetch.  Two, up to 16 vectors: no third request, which the loop makes for nothing (Wo of the 7B shape 6.9 -> 6.45 us,
// 24 steps of 16 sequences 52.5 -> 52.0 ms).
// Workgroup (blockIdx.x, slice blockIdx.y) of gridDim.x per slice: every gridDim.x-th tile of 32 rows (rows % 32 == 0).
// A row is added up in the same order at 16 and at 32 vectors: sampling from all of the distribution follows the last bits of the logits.
// (Waves with 16 of 32 vectors against a whole group, where a workgroup has one tile, convert half as many sums, step of 32
// sequences of the 110M shape 476 -> 462 us, but round them elsewhere: one plain-sampled batch in fifty got other tokens.)
// SWIGLU (one tile, one slice, matrices W1 and W3): a tile is 16 rows of W1 and the same rows of W3, and out is (npos, hidden):
// silu(h1) * h3 with the reference's sigmoid table (K/Silu.java:72-74); behind it (npos, hidden / 16): the sums of 16 consecutive ones.
template <int NB, int TILES, bool SWIGLU = false>
static __global__ void __launch_bounds__(64 * kStreamWaves, 2) k_dstream(const DGemm a)
{
    constexpr int NT = 2;   // blocks of 64 k per wave
    extern __shared__ __align__(16) float ds_lds[];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), s4 = lane >> 4, n = lane & 15;
    const int slice = blockIdx.y, g0 = slice * a.gps, ng = min(a.gps, a.ngroups - g0);
    const bool on = wave < 2 * ng;       // (a wave without a group multiplies the slice's last one by zero scales: no branch around loads)
    const int g = g0 + min(wave >> 1, ng - 1), hf = wave & 1, ntile = a.ntiles >> 1, step = gridDim.x;
    // this wave's k of the first tile of the first matrix, and how far from there the others lie (differences of addresses:
    // a choice between pointers would turn the loads into flat ones)
    const uint8_t *cb = a.codes[0] + (size_t)g * 4096 + 1024 * NT * hf;
    const float2 *sb = a.gs[0] + (size_t)g * 16;
    const long cd1 = a.codes[1] - a.codes[0], cd2 = a.codes[2] - a.codes[0], sd1 = a.gs[1] - a.gs[0], sd2 = a.gs[2] - a.gs[0];
    const int nt0 = a.tiles[0], nt1 = a.tiles[1];

    typedef const __attribute__((address_space(1))) uint8_t *CodePtr;
    unsigned lane16 = (unsigned)lane * 16;
    struct Codes { v4i w[2][NT]; float2 s[2]; };
    // the codes of this wave's k of tile t (past the end: the last tile again, not used), and the rows' scales
    auto request = [&](int t, Codes &c) {
        t = (SWIGLU ? 1 : 2) * min(t, ntile - 1);
        long cd = 0, sd = 0;
        if (!SWIGLU && t >= nt0) { t -= nt0; cd = cd1; sd = sd1; if (t >= nt1) { t -= nt1; cd = cd2; sd = sd2; } }
#pragma unroll
        for (int r = 0; r < 2; r++) c.s[r] = (sb + (SWIGLU ? (long)t * a.ngroups * 16 + r * sd1 : (long)(t + r) * a.ngroups * 16 + sd))[n];
        // Up to 16 vectors leave the registers for addresses, and scalar ones take longer to form: W1 and W3, W2, Wq Wk Wv and Wo (mean) of the
        // 7B shape 19.2 -> 18.6, 12.3 -> 11.9, 10.0 -> 9.8 us this way.
        if constexpr (NB == 1) {
#pragma unroll
            for (int T = 0; T < NT; T++)
#pragma unroll
                for (int r = 0; r < 2; r++)
                    c.w[r][T] = __builtin_nontemporal_load(reinterpret_cast<const v4i *>(cb + (SWIGLU ? (long)t * a.ngroups * 4096 + r * cd1 : (long)(t + r) * a.ngroups * 4096 + cd) + 1024 * T + (unsigned)lane * 16));
            return;
        }
        // (scalar bases and one register of offsets: addresses formed in vector registers took those of the codes two tiles on, and
        // every request waited for all codes under way)
        CodePtr p0 = (CodePtr)(cb + ((long)t * a.ngroups * 4096 + cd)), p1 = (CodePtr)(cb + (SWIGLU ? (long)t * a.ngroups * 4096 + cd1 : (long)(t + 1) * a.ngroups * 4096 + cd));
        asm volatile("" : "+s"(p0), "+s"(p1), "+v"(lane16));
#pragma unroll
        for (int T = 0; T < NT; T++) {
            c.w[0][T] = __builtin_nontemporal_load(reinterpret_cast<const __attribute__((address_space(1))) v4i *>(p0 + lane16 + 1024 * T));
            c.w[1][T] = __builtin_nontemporal_load(reinterpret_cast<const __attribute__((address_space(1))) v4i *>(p1 + lane16 + 1024 * T));
        }
    };

    Codes c0, c1;
    const int t0 = blockIdx.x;
    v4i dg[4][NB][NT];
    {
        const v4i *xp = reinterpret_cast<const v4i *>(a.x.d) + (size_t)g * (kDigitBytes / 16) + hf * NT * 128;
#pragma unroll
        for (int d = 0; d < 4; d++)
#pragma unroll
            for (int T = 0; T < NT; T++)
#pragma unroll
                for (int mt = 0; mt < NB; mt++) dg[d][mt][T] = (xp + ((d * 4 + T) * 2 + mt) * 64)[(unsigned)lane];
    }
    // The digits first: a wave's loads return in order, and the first tile needs all of the digits but only its own codes.  (Codes first: a step
    // of 16 and 32 sequences of the 110M shape 440 and 482 us for 411 and 476, of the 7B shape 2406 and 2910 for 2356 and 2885.)
    __builtin_amdgcn_sched_barrier(0);
    request(t0, c0);
    __builtin_amdgcn_sched_barrier(0);
    v4f sx[NB], sm[NB];
#pragma unroll
    for (int mt = 0; mt < NB; mt++) {
        sx[mt] = *reinterpret_cast<const v4f *>(a.x.sx + (size_t)g * 32 + 16 * mt + 4 * s4);
        sm[mt] = *reinterpret_cast<const v4f *>(a.x.sum + (size_t)g * 32 + 16 * mt + 4 * s4);
        if (!on) sx[mt] = v4f{0.f, 0.f, 0.f, 0.f};
        if (!on || hf) sm[mt] = v4f{0.f, 0.f, 0.f, 0.f};   // (the group's offset: by the first of its waves)
    }
    const int ldo = 16 * a.ntiles;
    float *out = a.out + (size_t)slice * a.npos * ldo;

    auto tile = [&](int buf, const Codes &c) {
        float *red = ds_lds + buf * kStreamWaves * NB * 512;
#pragma unroll
        for (int mt = 0; mt < NB; mt++)
#pragma unroll
            for (int r = 0; r < 2; r++) {
                v4i hi = {0, 0, 0, 0}, lo = {0, 0, 0, 0};
#pragma unroll
                for (int T = 0; T < NT; T++) {
                    hi = __builtin_amdgcn_mfma_i32_16x16x64_i8(dg[0][mt][T], c.w[r][T], hi, 0, 0, 0);
                    lo = __builtin_amdgcn_mfma_i32_16x16x64_i8(dg[2][mt][T], c.w[r][T], lo, 0, 0, 0);
                }
                hi <<= 8; lo <<= 8;
#pragma unroll
                for (int T = 0; T < NT; T++) {
                    hi = __builtin_amdgcn_mfma_i32_16x16x64_i8(dg[1][mt][T], c.w[r][T], hi, 0, 0, 0);
                    lo = __builtin_amdgcn_mfma_i32_16x16x64_i8(dg[3][mt][T], c.w[r][T], lo, 0, 0, 0);
                }
                v4f y;
#pragma unroll
                for (int e = 0; e < 4; e++)   // (the power of two into the sum, which takes it exactly: times the scale a small one would lose bits)
                    y[e] = fmaf(fmaf((float)hi[e], 65536.0f, (float)lo[e]) * sx[mt][e], c.s[r].x, c.s[r].y * sm[mt][e]);
                *reinterpret_cast<v4f *>(red + (((wave * NB + mt) * 2 + r) * 64 + lane) * 4) = y;
            }
    };
    // the tile's sums: NB x 2 blocks of 64 lanes x 4: NB values per thread
    struct Sums { float v[kStreamWaves][NB]; };
    auto read = [&](int buf, Sums &u) {
        const float *red = ds_lds + buf * kStreamWaves * NB * 512 + tid * NB;
#pragma unroll
        for (int w = 0; w < kStreamWaves; w++)
#pragma unroll
            for (int k = 0; k < NB; k++) u.v[w][k] = red[w * NB * 512 + k];
    };
    auto finish = [&](int tt, const Sums &u) {
        const int at = tid * NB, blk = at >> 8, l = (at >> 2) & 63, e = at & 3;
        const int row = 16 * (blk >> 1) + 4 * (l >> 4) + e;
        float *o = out + (size_t)row * ldo + 32 * tt + 16 * (blk & 1) + (l & 15);
#pragma unroll
        for (int k = 0; k < NB; k++) {
            float y = u.v[0][k];
#pragma unroll
            for (int w = 1; w < kStreamWaves; w++) y += u.v[w][k];
            if (row + k < a.npos) o[(size_t)k * ldo] = y;
        }
    };
    Sums u;
    int t = t0;
    if constexpr (SWIGLU) {
        static_assert(TILES == 1);
        tile(0, c0);
        __syncthreads();
        // thread: vectors and lane of a block of W1 and of the one of W3 beside it
        const int row = 16 * (tid >> 8) + 4 * ((tid >> 6) & 3) + (tid & 3), col = (tid >> 2) & 15;
        if (tid < 256 * NB && row < a.npos) {
            const float *red = ds_lds + (tid >> 8) * 512 + (tid & 255);
            float h1 = red[0], h3 = red[256];
#pragma unroll
            for (int w = 1; w < kStreamWaves; w++) {
                h1 += red[w * NB * 512];
                h3 += red[w * NB * 512 + 256];
            }
            const float m = silu_sigma(a.silu, h1, a.exact) * h3, y = h1 * m;
            a.out[(size_t)row * 16 * ntile + 16 * t + col] = y;
            // the sum of the sixteen, in the order (and with the first of two products unrounded, as the compiler contracts it there) of k_rows_swiglu
            float sum = fmaf(h1, m, __shfl_xor(y, 4));
#pragma unroll
            for (int off = 8; off < 64; off <<= 1) sum += __shfl_xor(sum, off);
            if (col == 0) a.out[(size_t)(a.npos * 16 + row) * ntile + t] = sum;
        }
        return;
    }
    if constexpr (TILES == 1) {
        tile(0, c0);
        __syncthreads();
        read(0, u);
        finish(t, u);
        return;
    }
    // The sums of a tile are read while the next one's products run.
    request(t + step, c1);
    __builtin_amdgcn_sched_barrier(0);   // (not moved behind the products, where it would find its registers free)
    tile(0, c0);
    __syncthreads();
    if constexpr (TILES == 2) {
        read(0, u);
        if (t + step >= ntile) {
            finish(t, u);
            return;
        }
        tile(1, c1);
        finish(t, u);
        __syncthreads();
        read(1, u);
        finish(t + step, u);
        return;
    }
    while (true) {
        read(0, u);
        if (t + step >= ntile) break;
        request(t + 2 * step, c0);
        __builtin_amdgcn_sched_barrier(0);
        tile(1, c1);
        finish(t, u);
        t += step;
        __syncthreads();
        read(1, u);
        if (t + step >= ntile) break;
        request(t + 2 * step, c1);
        __builtin_amdgcn_sched_barrier(0);
        tile(0, c0);
        finish(t, u);
        t += step;
        __syncthreads();
    }
    finish(t, u);
}

}  // namespace l2j
