// The forward pass of many positions at once: what l2j_rows.hip offers to the batched path.
#pragma once

#include <initializer_list>

#include "l2j_internal.hpp"
#include "digit_gemm.hpp"

namespace l2j {

constexpr int kRowsMax = 1024;   // rows of a pass
// Rows from which on the rows of a line of digits share an XCD (together_row): below, too few units of eight rows to keep eight XCDs evenly
// busy.  Whole passes, ms in order -> together, 256 and 1024 rows: 110M 0.911 -> 0.895 and 1.840 -> 1.804, 7B (four layers, as the others)
// 1.189 -> 1.179 and 3.882 -> 3.765, 13B 1.631 -> 1.617 and 6.174 -> 6.040, 70B widths 3.523 -> 3.472 and 13.29 -> 13.10; at 64 and 128
// rows within 2 % of each other.
constexpr int kTogetherFrom = 256;

struct DgPlan {
    int variant = 0, gps = 0, slices = 0, nrow = 0, ncol = 0;
};

struct RowNorm;

// k_dstream takes the products with at most 32 vectors (rows of the matrices in whole tiles of 32), k_dgemm the others.
inline bool streams(int tiles16, int rows) { return rows <= kRowTile && tiles16 % 2 == 0; }
inline int stream_slices(int ngroups) { return (ngroups + kStreamGroups - 1) / kStreamGroups; }

// Most slices of K k_dgemm cuts a product into: their sums are written and read again.
inline int max_slices(int rows) { return std::min(16, std::max(4, 1024 / std::max(1, rows))); }
// Most (slice, row) pairs of products of up to `cap` rows with rows of up to `ngroups` groups.
inline int max_slice_rows(int cap, int ngroups) { return std::max({std::min(16 * cap, 1024), 4 * cap, stream_slices(ngroups) * std::min(cap, kRowTile)}); }

// SwiGLU at the end of the product W1 and W3 and its digits at the beginning of W2 (k_dstream<NB, 1, true>, k_w2_rows) instead of a launch of
// its own: where W1 and W3 leave one slice, and both products are one round of the compute units: 16 rows of each of W1 and W3 a
// workgroup, 32 rows of W2 and one group of K, at most two slices of four groups, whose halves k_rows_norm adds up with all loads in flight.
// The bits are the same either way.  Step of twelve layers with 16 and 32 sequences, us, launch of its own -> this: 256 wide, hidden 256
// 334 398 -> 316 377, 256 x 2048 354 418 -> 336 393, 512 x 1536 370 436 -> 352 408, 768 x 2048 393 458 -> 376 437, 1024 x 1024 394 458 ->
// 376 434, 1024 x 2048 399 464 -> 386 446 (2000 ids).  (SwiGLU itself at the beginning of W2, by every tile, was 1.7 % slower than the
// launch: the sigmoid table's entries come one lane a cycle.)
inline bool swiglu_in_products(int n_cu, int dim, int hidden, int rows)
{
    return streams(dim / 16, rows) && stream_slices(dim / 256) == 1 && hidden / 16 <= n_cu && hidden / 256 <= 8 && dim / 32 * (hidden / 256) <= n_cu;
}

DgPlan dgemm_plan(int n_cu, int tiles16, int ngroups, int rows);
hipError_t prepare_dgemm(l2j_ctx *c);
int product_slices(l2j_ctx *c, int tiles16, int ngroups, int rows);
void launch_norm(l2j_ctx *c, const RowNorm &n, int rows);
int launch_dgemm(l2j_ctx *c, std::initializer_list<int> tensors, int layer, const Digits &x, int rows, float *part);
void launch_ffn(l2j_ctx *c, int layer, const RowBufs &b, int rows, RowNorm &n);

struct RowJob {
    int nseg, T, pos0;                                        // T positions from pos0 on of nseg sequences; b.tokens: their tokens
    float *kc, *vc;
    long seq_stride, layer_stride, head_stride, row_stride;   // of the cache, floats
    int norm_from;                                            // rows from here on (a multiple of nseg) are wanted after the final norm
};
int ensure_rows(l2j_ctx *c, int rows, int least, int *got);
hipError_t launch_rows(l2j_ctx *c, RowBufs &b, const RowJob &job);

// l2j_batch.hip
bool matrix_shape(const l2j_config &cf, int tensor, int *rows, int *K);
int ensure_batch_tiles(l2j_ctx *c);   // the tile-ordered copy of every matrix

// k_pflash (the keys of 16 positions shared by the waves of a workgroup, and from kSplitKeysFrom keys on by several workgroups)
// where k_rows_attn would have fewer than kSharedKeysBelow waves per compute unit for this many keys or more: 40 positions behind 1000
// of Llama-2-7B 5.0 against 5.8 ms, 128 behind 1000 7.2 against 7.6, 200 from 0 on 9.2 against 9.0, 400 from 0 on 15.3 against 14.7.
// At other shapes, ms never shared -> by this rule, 40 and 128 positions behind 1000: 110M (12 layers) 1.23 -> 0.70 and 1.33 -> 0.81, 13B
// (four layers) 0.86 -> 0.76 and 1.14 -> 1.24, 70B widths (four layers) 1.42 -> 1.38 and 2.11 -> 2.15.
// (kSplitKeysFrom lies below kSharedKeysFrom: it decides with option prefill_flash = 2 alone.)
constexpr int kSharedKeysFrom = 512, kSharedKeysBelow = 2, kSplitKeysFrom = 192, kPflashMaxSplit = 4;
inline size_t pflash_lds(int hs, int waves) { return (size_t)(32 * waves + 16 * waves * hs) * sizeof(float); }

}  // namespace l2j
