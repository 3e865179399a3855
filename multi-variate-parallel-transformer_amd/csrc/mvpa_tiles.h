// Small-tile bf16 GEMM for products with few rows of x (one decoding step, one short window), and
// what the stack executor launches around it.  Implemented in mvpa_tiles.hip.
#pragma once

#include "mvpa_common.h"

namespace mvpa {

// Where the columns of a plain product go: columns [0, n_y) to y; columns past n_y, if any, are the
// keys and then the values of ONE time step of every sample (n_kv columns each) and go straight into
// slot `slot` (or *head, read on the device) of the caches [B][Hkv][steps][C][Dh].
struct tile_out {
  bf16_t* y;
  int64_t ldy;
  int32_t n_y;
  int32_t n_kv, Dh, C;
  bf16_t *k, *v;
  int64_t stride_b, stride_g;      // elements, of k and v alike; a slot is C * Dh elements
  int32_t slot;
  const int32_t* head;
};

struct tile_gated {                // y = silu(x wg^T) * (x wu^T), w = gate rows [0, N) then up rows
  const bf16_t* w;
  bf16_t* y;
  int64_t ldw, ldy;
  int32_t N;
};

// RMSNorm inside the product: x holds raw rows, every output row is scaled by
// rsqrt(sum of its `parts` partial sums of squares / K + eps) before the gate (the norm's weight sits in
// the columns of the weights).  ss null: x is multiplied as it is.
struct tile_norm {
  const float* ss;
  int32_t parts;
  float eps;
};

// y0 = x w0^T (columns placed by `out`) and, if gated.w, the gated product on the same x.
// K a multiple of 64; 16-byte aligned rows.
int launch_tile_dual(const bf16_t* x, int64_t M, int64_t K, int64_t ldx, const bf16_t* w0, int64_t N0, int64_t ldw0,
                     const tile_out& out, const tile_gated& gated, const tile_norm& norm, hipStream_t s);

// y = x w^T where the tiles are the faster ones (tile_linear_pays; operands 16-byte aligned): few enough of them.
bool tile_linear_pays(int64_t M, int64_t N, int64_t K, int64_t ldx, int64_t ldw, int64_t ldy, const void* y);
int launch_tile_linear(const bf16_t* x, int64_t M, int64_t K, int64_t ldx, const bf16_t* w, int64_t N, int64_t ldw, bf16_t* y,
                       int64_t ldy, hipStream_t s);

// How a contraction is cut: columns [0, Ka) of x into `a` runs of per_a k-blocks, the rest (all of it where
// Ka is 0) into `b` runs of per_b.
struct tile_split {
  int32_t a, per_a, b, per_b, nkb_a;
  int total() const { return a + b; }
};
tile_split make_tile_split(int64_t M, int64_t N, int64_t K, int64_t Ka);

// Split-K product for the tail of a block: partial sums to P [a + b][M][N] (fp32).
int launch_tile_partial(const bf16_t* x, int64_t M, int64_t K, int64_t ldx, const bf16_t* w, int64_t N, int64_t ldw,
                        float* P, const tile_split& split, hipStream_t s);

// sum[m] = r[m] + the products of the two parts, each rounded to bf16 as a product of its own would be, then
// the sum once more; rows of N (a multiple of 8, at most 4096) columns; sum may be r.
// With norm: norm[m] = RMSNorm(sum[m]) * w.  With ss: ss[m] = the sum of squares of row m.
int launch_tail_reduce(const float* P, const tile_split& split, const bf16_t* r, bf16_t* sum, bf16_t* norm, const float* w,
                       float eps, float* ss, int64_t M, int64_t N, hipStream_t s);

// One new time step of keys and values, [B,Hkv,C,Dh] views (strides in elements, multiples of 8, unit last
// stride), into slot `slot` (or *head) of caches as in tile_out.  Implemented in mvpa_dense.hip.
int launch_append(const bf16_t* k_new, const bf16_t* v_new, bf16_t* k, bf16_t* v, const int32_t* head, int32_t slot,
                  int32_t B, int32_t Hkv, int32_t C, int32_t Dh, int64_t stride_b, int64_t stride_h, int64_t stride_c,
                  int64_t cache_stride_b, int64_t cache_stride_h, hipStream_t s);

}  // namespace mvpa
