// Row operations of the training path: backward of RMSNorm with the residual's gradient, and the gated
// activation of the MLP with its backward (models/mvpformer.py:132-147).
//
// All are bound by HBM: each input is read once and each result written once, where the tensor
// expressions they stand for walked fp32 copies of their operands (RMSNorm backward: a dozen passes).
// 6400 rows: norm backward with residual 768 columns 20 us, gate of 2048 columns 18 us (4.5 TB/s), its
// backward 23 us (5.6 TB/s).  A fine-tuning pass of twelve such blocks 21.8 -> 15.9 ms.
#include "mvpa_common.h"

namespace mvpa {
namespace train {

typedef __attribute__((ext_vector_type(4))) float f32x4;
typedef __attribute__((ext_vector_type(4))) uint32_t u32x4;
typedef __attribute__((ext_vector_type(2))) uint32_t u32x2;

constexpr int MAX_COLS = 4096;       // 16 chunks of 4 columns per lane
constexpr int MAX_GROUPS = 512;      // workgroups of the row pass = partial sums per column of the weight gradient

__device__ inline float wave_sum(float x) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) x += __shfl_xor(x, off);
  return x;
}

// four values as they lie in memory
__device__ inline f32x4 raw4(const float* p) { return *(const f32x4*)p; }
__device__ inline u32x2 raw4(const bf16_t* p) { return *(const u32x2*)p; }
__device__ inline void widen(f32x4 x, float (&v)[4]) {
#pragma unroll
  for (int i = 0; i < 4; ++i) v[i] = x[i];
}
__device__ inline void widen(u32x2 x, float (&v)[4]) {
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    v[2 * i] = __uint_as_float(x[i] << 16);
    v[2 * i + 1] = __uint_as_float(x[i] & 0xffff0000u);
  }
}
__device__ inline uint32_t pack2(float lo, float hi) { return (uint32_t)f32_to_bf16(lo) | ((uint32_t)f32_to_bf16(hi) << 16); }
__device__ inline void store4(float* p, const float (&v)[4]) { *(f32x4*)p = f32x4{v[0], v[1], v[2], v[3]}; }
__device__ inline void store4(bf16_t* p, const float (&v)[4]) { *(u32x2*)p = u32x2{pack2(v[0], v[1]), pack2(v[2], v[3])}; }

// four columns of a row, guarded at the end of the row where rows are not whole chunks
template <bool VEC, typename T>
__device__ inline void get4(const T* row, int c, int cols, float (&v)[4]) {
#pragma unroll
  for (int i = 0; i < 4; ++i) v[i] = 0.f;
  if (VEC) {
    if (c < cols) widen(raw4(row + c), v);
  } else {
#pragma unroll
    for (int i = 0; i < 4; ++i)
      if (c + i < cols) v[i] = io<T>::load(row + c + i);
  }
}
template <bool VEC, typename T>
__device__ inline void put4(T* row, int c, int cols, const float (&v)[4]) {
  if (VEC) {
    if (c < cols) store4(row + c, v);
  } else {
#pragma unroll
    for (int i = 0; i < 4; ++i)
      if (c + i < cols) io<T>::store(row + c + i, v[i]);
  }
}

// y = x r w with r = rsqrt(mean(x^2) + eps):   dx = r w dy - x r^3 mean(x w dy) (+ res),   dw = sum_rows dy x r
// A wave owns whole rows, a lane the same columns of each of them: the row is in registers between its
// two sums and its result, and the lane's share of dw stays there over all rows.  HBM bound.  512 workgroups:
// with one per four rows the partial sums of dw are as many bytes as a row operand.  AHEAD: the wave's next row, where
// there is one, is requested before the sums of this one, without a branch per chunk, behind which each load would be
// waited for by itself: with the sums of dw 18.6 -> 13.8 us for 6400 rows of 768 in bf16, 144 -> 79 for 65536.  Where that
// pays: launch_norm.
template <typename TX, typename TW, int NCH, bool VEC, bool AHEAD>
__global__ __launch_bounds__(256) void rmsnorm_backward_kernel(const TX* __restrict__ x, const TW* __restrict__ w,
                                                               const bf16_t* __restrict__ dy, const TX* __restrict__ res,
                                                               TX* __restrict__ dx, float* __restrict__ part,
                                                               int64_t rows, int cols, float eps) {
  __shared__ float red[3][256];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  float wv[NCH][4], acc[NCH][4];
#pragma unroll
  for (int i = 0; i < NCH; ++i) {
    get4<VEC>(w, (i * 64 + lane) * 4, cols, wv[i]);
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[i][j] = 0.f;
  }
  const float rcols = 1.f / (float)cols;
  // chunks beyond the row read its last four columns and count as zero
  static_assert(VEC || !AHEAD, "whole chunks");
  constexpr int NR = AHEAD ? NCH : 1;
  decltype(raw4(x)) x_raw[NR], r_raw[NR] = {};
  u32x2 g_raw[NR];
  auto request = [&](int64_t row) {
    if constexpr (AHEAD) {
#pragma unroll
      for (int i = 0; i < NCH; ++i) {
        const int64_t at = row * cols + min((i * 64 + lane) * 4, cols - 4);
        x_raw[i] = raw4(x + at);
        g_raw[i] = raw4(dy + at);
      }
      if (res)
#pragma unroll
        for (int i = 0; i < NCH; ++i) r_raw[i] = raw4(res + row * cols + min((i * 64 + lane) * 4, cols - 4));
    }
  };
  const int64_t first = (int64_t)blockIdx.x * 4 + wave, stride = (int64_t)gridDim.x * 4;
  if (first < rows) request(first);
  for (int64_t row = first; row < rows; row += stride) {
    float xv[NCH][4], gv[NCH][4], add[NR][4];
    float ss = 0.f, dot = 0.f;
#pragma unroll
    for (int i = 0; i < NCH; ++i) {
      const int c = (i * 64 + lane) * 4;
      if constexpr (AHEAD) {
        widen(x_raw[i], xv[i]);
        widen(g_raw[i], gv[i]);
        widen(r_raw[i], add[i]);
#pragma unroll
        for (int j = 0; j < 4; ++j)
          if (c >= cols) xv[i][j] = gv[i][j] = 0.f;
      } else {
        get4<VEC>(x + row * cols, c, cols, xv[i]);
        get4<VEC>(dy + row * cols, c, cols, gv[i]);
      }
    }
    if (row + stride < rows) request(row + stride);
#pragma unroll
    for (int i = 0; i < NCH; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        ss += xv[i][j] * xv[i][j];
        dot += xv[i][j] * (gv[i][j] * wv[i][j]);
      }
    ss = wave_sum(ss);
    dot = wave_sum(dot);
    const float r = rsqrtf(ss * rcols + eps), k = r * r * r * (dot * rcols);
#pragma unroll
    for (int i = 0; i < NCH; ++i) {
      const int c = (i * 64 + lane) * 4;
      if (dx) {
        float o[4], late[4] = {0.f, 0.f, 0.f, 0.f};
        if (!AHEAD && res) get4<VEC>(res + row * cols, c, cols, late);
#pragma unroll
        for (int j = 0; j < 4; ++j) o[j] = r * (gv[i][j] * wv[i][j]) - xv[i][j] * k + (AHEAD ? add[AHEAD ? i : 0][j] : late[j]);
        put4<VEC>(dx + row * cols, c, cols, o);
      }
#pragma unroll
      for (int j = 0; j < 4; ++j) acc[i][j] += gv[i][j] * xv[i][j] * r;
    }
  }
  if (!part) return;
#pragma unroll
  for (int i = 0; i < NCH; ++i) {
    __syncthreads();
    if (wave > 0)
#pragma unroll
      for (int j = 0; j < 4; ++j) red[wave - 1][lane * 4 + j] = acc[i][j];
    __syncthreads();
    if (wave == 0)
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int c = (i * 64 + lane) * 4 + j;
        const float s = (acc[i][j] + red[0][lane * 4 + j]) + (red[1][lane * 4 + j] + red[2][lane * 4 + j]);
        if (c < cols) part[(int64_t)blockIdx.x * cols + c] = s;
      }
  }
}

// column sums of part [n][cols]: 64 columns per workgroup, 16 of its waves each every 16th row
template <typename TW>
__global__ __launch_bounds__(1024) void column_sum_kernel(const float* __restrict__ part, TW* __restrict__ out, int n, int cols) {
  __shared__ float red[16][64];
  const int lane = threadIdx.x & 63, sub = threadIdx.x >> 6, c = blockIdx.x * 64 + lane;
  float s = 0.f;
  if (c < cols) {
#pragma unroll 8
    for (int i = sub; i < n; i += 16) s += part[(int64_t)i * cols + c];
  }
  red[sub][lane] = s;
  __syncthreads();
  if (sub == 0 && c < cols) {
#pragma unroll
    for (int i = 1; i < 16; ++i) s += red[i][lane];
    io<TW>::store(out + c, s);
  }
}

// part[group][c] = sum over the group's rows of dy x inv, for a norm whose row factors are known (the encoder's: its rows are
// the signal's, no gradient goes on).  Nothing is summed along a row, so a lane keeps four columns and walks down the
// rows, four of them requested together.  HBM bound: 6400 rows of 2610 21 us, 5 TB/s (rmsnorm_backward_kernel, which takes
// single elements of rows that do not start at 16-byte boundaries, 118).
constexpr int DW_GROUPS = 64, DW_ROWS = 4;
__global__ __launch_bounds__(256) void norm_dw_kernel(const float* __restrict__ x, const float* __restrict__ inv,
                                                      const bf16_t* __restrict__ dy, float* __restrict__ part, int64_t rows, int cols,
                                                      int64_t ldx, int64_t lddy) {
  __shared__ float red[3][256];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, c = (blockIdx.x * 64 + lane) * 4;
  const int at = min(c, (cols - 1) & ~3);           // lanes past the row: its last four columns, for nobody
  float acc[4] = {};
  const int64_t stride = (int64_t)gridDim.y * 4;
  for (int64_t row = (int64_t)blockIdx.y * 4 + wave; row < rows; row += stride * DW_ROWS) {
    f32x4 xr[DW_ROWS];
    u32x2 gr[DW_ROWS];
    float f[DW_ROWS];
#pragma unroll
    for (int i = 0; i < DW_ROWS; ++i) {
      const int64_t r = min(row + i * stride, rows - 1);
      xr[i] = raw4(x + r * ldx + at);
      gr[i] = raw4(dy + r * lddy + at);
      f[i] = inv[r];
    }
#pragma unroll
    for (int i = 0; i < DW_ROWS; ++i) {
      float v[4];
      widen(gr[i], v);
#pragma unroll
      for (int j = 0; j < 4; ++j) acc[j] += row + i * stride < rows ? v[j] * xr[i][j] * f[i] : 0.f;
    }
  }
  if (wave > 0) *(f32x4*)&red[wave - 1][lane * 4] = f32x4{acc[0], acc[1], acc[2], acc[3]};
  __syncthreads();
  if (wave > 0) return;
#pragma unroll
  for (int j = 0; j < 4; ++j)
    if (c + j < cols)
      part[(int64_t)blockIdx.y * cols + c + j] = (acc[j] + red[0][lane * 4 + j]) + (red[1][lane * 4 + j] + red[2][lane * 4 + j]);
}

// about 8 rows a wave or more
static int dw_groups(int64_t rows) { return (int)(rows >= 32 * DW_GROUPS ? DW_GROUPS : (rows + 31) / 32); }

__device__ inline void unpack8(u32x4 x, float (&v)[8]) {
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    v[2 * i] = __uint_as_float(x[i] << 16);
    v[2 * i + 1] = __uint_as_float(x[i] & 0xffff0000u);
  }
}
__device__ inline void load8(const bf16_t* p, float (&v)[8]) { unpack8(*(const u32x4*)p, v); }
__device__ inline void store8(bf16_t* p, const float (&v)[8]) {
  *(u32x4*)p = u32x4{pack2(v[0], v[1]), pack2(v[2], v[3]), pack2(v[4], v[5]), pack2(v[6], v[7])};
}

// The generative score's backward (models/mvpformer.py:749-764): step t + 1 of a against step t of b.
//   s = a.b / (|a|' |b|'),  |x|' = max(|x|, eps):   da = d (b / (|a|' |b|') - a s / (|a|' |a|)), db likewise,
// the norms not held at eps in the derivative, as torch.cosine_similarity has it; zeros for the step without a partner.  A wave
// owns a pair of rows and reads them twice, the second time from the caches.  HBM bound; as tensor operations on fp32
// copies the score and its backward were 45 launches, 330 us at B4 C64 T25 E768, of which this one takes 9 and the forward 5.
__global__ __launch_bounds__(256) void cosine_steps_backward_kernel(const bf16_t* __restrict__ a, const bf16_t* __restrict__ b,
                                                                    const float* __restrict__ d, bf16_t* __restrict__ da,
                                                                    bf16_t* __restrict__ db, int64_t rows, int64_t T, int64_t C,
                                                                    int cols, float eps) {
  const int64_t row = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (row >= rows) return;
  const int lane = threadIdx.x & 63;
  const int64_t bt = row / C, n = bt / T, t = bt - n * T;
  const bf16_t* ar = a + row * cols;
  bf16_t* dar = da ? da + row * cols : nullptr;
  if (t == 0) {                      // a's first step and b's last one
    bf16_t* dbr = db ? db + (row + (T - 1) * C) * cols : nullptr;
    for (int c = lane * 8; c < cols; c += 512) {
      if (dar) *(u32x4*)(dar + c) = u32x4{0u, 0u, 0u, 0u};
      if (dbr) *(u32x4*)(dbr + c) = u32x4{0u, 0u, 0u, 0u};
    }
    return;
  }
  const bf16_t* br = b + (row - C) * cols;
  bf16_t* dbr = db ? db + (row - C) * cols : nullptr;
  const float g = d[row - (n + 1) * C];
  float dot = 0.f, na = 0.f, nb = 0.f;
  for (int c = lane * 8; c < cols; c += 512) {
    float x[8], y[8];
    load8(ar + c, x);
    load8(br + c, y);
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      dot += x[i] * y[i];
      na += x[i] * x[i];
      nb += y[i] * y[i];
    }
  }
  dot = wave_sum(dot);
  na = sqrtf(wave_sum(na));
  nb = sqrtf(wave_sum(nb));
  // comparisons that are false for a NaN, whose row's gradients are NaN throughout (fmaxf would give eps)
  const float ia = 1.f / (na < eps ? eps : na), ib = 1.f / (nb < eps ? eps : nb);
  float s = dot * ia * ib;
  if (na == INFINITY || nb == INFINITY) {       // as the forward has it: the elements are divided first
    s = 0.f;
    for (int c = lane * 8; c < cols; c += 512) {
      float x[8], y[8];
      load8(ar + c, x);
      load8(br + c, y);
#pragma unroll
      for (int i = 0; i < 8; ++i) s += (x[i] * ia) * (y[i] * ib);
    }
    s = wave_sum(s);
  }
  const float cross = g * ia * ib, ca = na == 0.f ? 0.f : g * s * ia / na, cb = nb == 0.f ? 0.f : g * s * ib / nb;
  for (int c = lane * 8; c < cols; c += 512) {
    float x[8], y[8], o[8];
    load8(ar + c, x);
    load8(br + c, y);
    if (dar) {
#pragma unroll
      for (int i = 0; i < 8; ++i) o[i] = cross * y[i] - ca * x[i];
      store8(dar + c, o);
    }
    if (dbr) {
#pragma unroll
      for (int i = 0; i < 8; ++i) o[i] = cross * x[i] - cb * y[i];
      store8(dbr + c, o);
    }
  }
}

constexpr int GATE_ROWS = 4;         // rows per thread: their loads go out together

// out = silu(gate) up for rows [gate | up] of 2 n columns; a thread takes 8 columns of GATE_ROWS rows
__global__ __launch_bounds__(256) void silu_gate_kernel(const bf16_t* __restrict__ gu, bf16_t* __restrict__ out, int64_t rows, int n) {
  const int c = (blockIdx.y * 256 + threadIdx.x) * 8;
  if (c >= n) return;
#pragma unroll
  for (int i = 0; i < GATE_ROWS; ++i) {
    const int64_t row = (int64_t)blockIdx.x * GATE_ROWS + i;
    if (row >= rows) break;
    float g[8], u[8];
    load8(gu + row * 2 * n + c, g);
    load8(gu + row * 2 * n + n + c, u);
#pragma unroll
    for (int j = 0; j < 8; ++j) g[j] = silu_gate(g[j], u[j]);
    store8(out + row * n + c, g);
  }
}

// dgate = d up s (1 + gate (1 - s)), dup = d gate s, s the sigmoid of gate
__global__ __launch_bounds__(256) void silu_gate_backward_kernel(const bf16_t* __restrict__ gu, const bf16_t* __restrict__ d,
                                                                 bf16_t* __restrict__ dgu, int64_t rows, int n) {
  const int c = (blockIdx.y * 256 + threadIdx.x) * 8;
  if (c >= n) return;
#pragma unroll
  for (int i = 0; i < GATE_ROWS; ++i) {
    const int64_t row = (int64_t)blockIdx.x * GATE_ROWS + i;
    if (row >= rows) break;
    float g[8], u[8], dv[8];
    load8(gu + row * 2 * n + c, g);
    load8(gu + row * 2 * n + n + c, u);
    load8(d + row * n + c, dv);
#pragma unroll
    for (int j = 0; j < 8; ++j) silu_gate_gradients(g[j], u[j], dv[j], g[j], u[j]);
    store8(dgu + row * 2 * n + c, g);
    store8(dgu + row * 2 * n + n + c, u);
  }
}

// ---- stacked projection weights with low-rank adapters (layers/mvpa.py:43-62, 86-93) ----------
// out = [w_0 + scale b_0 a_0; w_1 + ...] over the parts of a projection and the gradients of a and b from that
// of out.  As tensor expressions a block's pair of projections is ten launches forward and twenty-six
// backward, none of which moves more than a megabyte: they cost a launch each.  Here one each way, sums in
// fp32 and one rounding.  Bound by the launch and a chain of loads.  Rank 8 on
// 1 024 of 1 280 rows of 768: 7.5 and 14 us; the training pass of twelve such blocks went from 13.8 to 11.9 ms.
struct lora_parts {
  mvpa_lora_part p[MVPA_LORA_PARTS];
};

constexpr int LORA_ROWS = 4;         // rows per workgroup of the stacked weight: a's columns are read once for them

// eight terms k0 .. of a row of b; whole rows of 16-byte chunks where VEC, zeros past the rank
template <bool VEC>
__device__ inline void lora_b8(const bf16_t* row, int k0, int r, float (&v)[8]) {
  if (VEC) {
    load8(row + k0, v);
  } else {
#pragma unroll
    for (int i = 0; i < 8; ++i) v[i] = k0 + i < r ? bf16_to_f32(row[k0 + i]) : 0.f;
  }
}

// a thread takes 8 columns of LORA_ROWS rows (groups of them along x, whose grid takes any number of them); blockIdx.z is
// the part.  VEC: r a multiple of 8
template <bool VEC>
__global__ __launch_bounds__(128) void lora_stack_kernel(lora_parts parts, bf16_t* __restrict__ out, int K, int r, float scale) {
  const mvpa_lora_part p = parts.p[blockIdx.z];
  const int row0 = blockIdx.x * LORA_ROWS, c = (blockIdx.y * 128 + threadIdx.x) * 8;
  if (row0 >= p.rows || c >= K) return;
  const bf16_t *w = (const bf16_t*)p.w, *a = (const bf16_t*)p.a, *b = (const bf16_t*)p.b;
  u32x4 wv[LORA_ROWS];               // requested first: the only operand that is not in a cache
#pragma unroll
  for (int i = 0; i < LORA_ROWS; ++i) wv[i] = *(const u32x4*)(w + (int64_t)min(row0 + i, p.rows - 1) * K + c);
  float acc[LORA_ROWS][8];
#pragma unroll
  for (int i = 0; i < LORA_ROWS; ++i)
#pragma unroll
    for (int j = 0; j < 8; ++j) acc[i][j] = 0.f;
  for (int k0 = 0; a && k0 < r; k0 += 8) {
    float bv[LORA_ROWS][8];
#pragma unroll
    for (int i = 0; i < LORA_ROWS; ++i) lora_b8<VEC>(b + (int64_t)min(row0 + i, p.rows - 1) * r, k0, r, bv[i]);
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      if (!VEC && k0 + k >= r) break;            // no zero times a row of a, which may be infinite
      float av[8];
      load8(a + (int64_t)(k0 + k) * K + c, av);
#pragma unroll
      for (int i = 0; i < LORA_ROWS; ++i)
#pragma unroll
        for (int j = 0; j < 8; ++j) acc[i][j] += bv[i][k] * av[j];
    }
  }
#pragma unroll
  for (int i = 0; i < LORA_ROWS; ++i) {
    if (row0 + i >= p.rows) break;
    float v[8];
    unpack8(wv[i], v);
#pragma unroll
    for (int j = 0; j < 8; ++j) v[j] += scale * acc[i][j];
    store8(out + (p.row0 + row0 + i) * (int64_t)K + c, v);
  }
}

// One launch for both gradients of every part: the first (K + 63) / 64 workgroups of a part sum
// da[k, c] = scale sum_rows b[row, k] d[row, c] over 64 columns each (32 row shares, merged through LDS), the
// rest take a row per wave for db[row, k] = scale sum_c d[row, c] a[k, c].  Eight of the r terms at a time.
// b's rows go through LDS, so that what a row costs is one load of d and many of them are in flight: with b
// read where it is used, 2 bytes at a time, the launch took 47 us.
constexpr int LORA_B_ROWS = 1024;    // rows of b in LDS at a time
template <bool VEC>
__global__ __launch_bounds__(1024) void lora_stack_backward_kernel(lora_parts parts, const bf16_t* __restrict__ d, int K, int r,
                                                                   float scale) {
  __shared__ float red[16][8][64];
  __shared__ __attribute__((aligned(16))) float bs[LORA_B_ROWS][8];
  const mvpa_lora_part p = parts.p[blockIdx.y];
  if (!p.a) return;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, col_groups = (K + 63) / 64;
  const bf16_t *a = (const bf16_t*)p.a, *b = (const bf16_t*)p.b;
  d += p.row0 * (int64_t)K;
  if ((int)blockIdx.x < col_groups) {
    if (!p.da) return;
    bf16_t* da = (bf16_t*)p.da;
    const int c = blockIdx.x * 64 + (lane & 31) * 2, share = wave * 2 + (lane >> 5);
    for (int k0 = 0; k0 < r; k0 += 8) {
      float acc[8][2];
#pragma unroll
      for (int i = 0; i < 8; ++i) acc[i][0] = acc[i][1] = 0.f;
      for (int first = 0; first < p.rows; first += LORA_B_ROWS) {
        const int n = min(p.rows - first, LORA_B_ROWS);
        __syncthreads();
        if ((int)threadIdx.x < n) {
          float v[8];
          lora_b8<VEC>(b + (int64_t)(first + threadIdx.x) * r, k0, r, v);
          store4(&bs[threadIdx.x][0], {v[0], v[1], v[2], v[3]});
          store4(&bs[threadIdx.x][4], {v[4], v[5], v[6], v[7]});
        }
        __syncthreads();
        if (c < K) {
#pragma unroll 8
          for (int row = share; row < n; row += 32) {
            const uint32_t x = *(const uint32_t*)(d + (int64_t)(first + row) * K + c);
            const float lo = __uint_as_float(x << 16), hi = __uint_as_float(x & 0xffff0000u);
#pragma unroll
            for (int i = 0; i < 8; ++i) {
              acc[i][0] += bs[row][i] * lo;
              acc[i][1] += bs[row][i] * hi;
            }
          }
        }
      }
      __syncthreads();
#pragma unroll
      for (int i = 0; i < 8; ++i) {
#pragma unroll
        for (int j = 0; j < 2; ++j) acc[i][j] += __shfl_xor(acc[i][j], 32);
        if (lane < 32) {
          red[wave][i][lane * 2] = acc[i][0];
          red[wave][i][lane * 2 + 1] = acc[i][1];
        }
      }
      __syncthreads();
      const int i = threadIdx.x >> 6, cc = blockIdx.x * 64 + lane;
      if (threadIdx.x < 512 && k0 + i < r && cc < K) {
        float s = 0.f;
#pragma unroll
        for (int g = 0; g < 16; ++g) s += red[g][i][lane];
        da[(int64_t)(k0 + i) * K + cc] = f32_to_bf16(scale * s);
      }
    }
    return;
  }
  if (!p.db) return;
  const int row = (blockIdx.x - col_groups) * 16 + wave;
  if (row >= p.rows) return;
  bf16_t* db = (bf16_t*)p.db;
  for (int k0 = 0; k0 < r; k0 += 8) {
    float acc[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) acc[i] = 0.f;
    for (int c = lane * 8; c < K; c += 512) {
      float x[8];
      load8(d + (int64_t)row * K + c, x);
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        float av[8];
        load8(a + (int64_t)min(k0 + i, r - 1) * K + c, av);
#pragma unroll
        for (int j = 0; j < 8; ++j) acc[i] += x[j] * av[j];
      }
    }
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const float s = wave_sum(acc[i]);
      if (lane == 0 && k0 + i < r) db[(int64_t)row * r + k0 + i] = f32_to_bf16(scale * s);
    }
  }
}

static int row_groups(int64_t rows) { return (int)(rows >= 4 * MAX_GROUPS ? MAX_GROUPS : (rows + 3) / 4); }

template <typename TX, typename TW>
static void launch_norm(const void* x, const void* w, const void* dy, const void* res, void* dx, float* part, int64_t rows,
                        int cols, float eps, bool vec, hipStream_t s) {
  auto go = [&](auto kern) {
    MVPA_LAUNCH(kern, dim3((unsigned)row_groups(rows)), dim3(256), 0, s, (const TX*)x, (const TW*)w, (const bf16_t*)dy,
                (const TX*)res, (TX*)dx, part, rows, cols, eps);
  };
  // The next row ahead: up to 1024 columns.  Up to 2048 in bf16 it takes the registers of a second row, and the waves of a
  // launch whose operands the caches hold wait less for memory than for each other.  us, rows as they come / ahead, dx
  // and dw, and with res: 1600 x 2048 13.3 / 19.6, 14.1 / 19.6; 6400 x 2048 28.9 / 33.6, 33.0 / 33.6; 16384 x 2048 50 / 57,
  // 61 / 57; 30000 x 2048 119 / 97, 157 / 97; 30000 x 1280 60 / 74, 74 / 74; 65536 x 1280 163 / 170, 218 / 170; 30000 x 1536
  // 87 / 86, 105 / 86.  In fp32, and wider, two rows do not fit the registers (2560 in fp32: 69 / 174).
  const bool far = sizeof(TX) == 2 && rows * cols >= (res ? 40000000 : 45000000) && (res || cols > 1408);
  if (!vec) {
    if (cols <= 1024) go(rmsnorm_backward_kernel<TX, TW, 4, false, false>);
    else go(rmsnorm_backward_kernel<TX, TW, 16, false, false>);
  } else if (cols <= 768) go(rmsnorm_backward_kernel<TX, TW, 3, true, true>);
  else if (cols <= 1024) go(rmsnorm_backward_kernel<TX, TW, 4, true, true>);
  else if (cols <= 2048 && far) go(rmsnorm_backward_kernel<TX, TW, 8, true, sizeof(TX) == 2>);
  else if (cols <= 2048) go(rmsnorm_backward_kernel<TX, TW, 8, true, false>);
  else go(rmsnorm_backward_kernel<TX, TW, 16, true, false>);
}

}  // namespace train
}  // namespace mvpa

using namespace mvpa;

extern "C" size_t mvpa_rmsnorm_backward_ws_bytes(int64_t rows, int32_t cols) {
  return rows > 0 && cols > 0 ? (size_t)train::row_groups(rows) * cols * sizeof(float) : 0;
}

extern "C" int mvpa_rmsnorm_backward(const void* x, const void* weight, const void* dy, const void* res, void* dx, void* dw,
                                     void* ws, int64_t rows, int32_t cols, float eps, int32_t x_f32, int32_t w_f32,
                                     void* stream) {
  if (!x || !weight || !dy || (!dx && !dw) || (dw && !ws)) return MVPA_ERR_NULL;
  if (rows <= 0 || cols <= 0) return MVPA_ERR_SHAPE;
  if (cols > train::MAX_COLS) return MVPA_ERR_UNSUPPORTED;
  const uintptr_t low = (uintptr_t)x | (uintptr_t)weight | (uintptr_t)dy | (uintptr_t)res | (uintptr_t)dx;
  const bool vec = cols % 4 == 0 && (low & 15) == 0;
  float* part = dw ? (float*)ws : nullptr;
  hipStream_t s = (hipStream_t)stream;
  if (x_f32 && w_f32) train::launch_norm<float, float>(x, weight, dy, res, dx, part, rows, cols, eps, vec, s);
  else if (x_f32) train::launch_norm<float, bf16_t>(x, weight, dy, res, dx, part, rows, cols, eps, vec, s);
  else if (w_f32) train::launch_norm<bf16_t, float>(x, weight, dy, res, dx, part, rows, cols, eps, vec, s);
  else train::launch_norm<bf16_t, bf16_t>(x, weight, dy, res, dx, part, rows, cols, eps, vec, s);
  if (dw) {
    const dim3 grid((unsigned)((cols + 63) / 64));
    const int n = train::row_groups(rows);
    if (w_f32) MVPA_LAUNCH(train::column_sum_kernel<float>, grid, dim3(1024), 0, s, part, (float*)dw, n, cols);
    else MVPA_LAUNCH(train::column_sum_kernel<bf16_t>, grid, dim3(1024), 0, s, part, (bf16_t*)dw, n, cols);
  }
  return take_launch_status();
}

extern "C" size_t mvpa_norm_dw_ws_bytes(int64_t rows, int32_t cols) {
  return rows > 0 && cols > 0 ? (size_t)train::dw_groups(rows) * cols * sizeof(float) : 0;
}

extern "C" int mvpa_norm_dw(const float* x, const float* inv, const void* dy, void* dw, void* ws, int64_t rows, int32_t cols,
                            int64_t ldx, int64_t lddy, int32_t w_f32, void* stream) {
  if (!x || !inv || !dy || !dw || !ws) return MVPA_ERR_NULL;
  const int64_t whole = ((int64_t)cols + 3) / 4 * 4;
  if (rows <= 0 || cols <= 0 || ldx < whole || lddy < whole) return MVPA_ERR_SHAPE;
  if ((ldx & 3) || (lddy & 3) || ((uintptr_t)x & 15) || ((uintptr_t)dy & 7)) return MVPA_ERR_ALIGN;
  const int n = train::dw_groups(rows);
  hipStream_t s = (hipStream_t)stream;
  MVPA_LAUNCH(train::norm_dw_kernel, dim3((unsigned)((cols + 255) / 256), (unsigned)n), dim3(256), 0, s, x, inv, (const bf16_t*)dy,
              (float*)ws, rows, cols, ldx, lddy);
  const dim3 grid((unsigned)((cols + 63) / 64));
  if (w_f32) MVPA_LAUNCH(train::column_sum_kernel<float>, grid, dim3(1024), 0, s, (const float*)ws, (float*)dw, n, cols);
  else MVPA_LAUNCH(train::column_sum_kernel<bf16_t>, grid, dim3(1024), 0, s, (const float*)ws, (bf16_t*)dw, n, cols);
  return take_launch_status();
}

static int gate_check(const void* a, const void* b, const void* c, int64_t rows, int32_t n) {
  if (!a || !b || !c) return MVPA_ERR_NULL;
  if (rows <= 0 || n <= 0 || n > (1 << 24) || rows > ((int64_t)1 << 31)) return MVPA_ERR_SHAPE;
  if (n % 8 != 0 || (((uintptr_t)a | (uintptr_t)b | (uintptr_t)c) & 15)) return MVPA_ERR_ALIGN;
  return MVPA_OK;
}

static dim3 gate_grid(int64_t rows, int32_t n) {
  return dim3((unsigned)((rows + train::GATE_ROWS - 1) / train::GATE_ROWS), (unsigned)((n + 2047) / 2048));
}

extern "C" int mvpa_silu_gate_bf16(const void* gu, void* out, int64_t rows, int32_t n, void* stream) {
  const int st = gate_check(gu, out, out, rows, n);
  if (st != MVPA_OK) return st;
  MVPA_LAUNCH(train::silu_gate_kernel, gate_grid(rows, n), dim3(256), 0, (hipStream_t)stream, (const bf16_t*)gu, (bf16_t*)out, rows, n);
  return take_launch_status();
}

extern "C" int mvpa_silu_gate_backward_bf16(const void* gu, const void* d, void* dgu, int64_t rows, int32_t n, void* stream) {
  const int st = gate_check(gu, d, dgu, rows, n);
  if (st != MVPA_OK) return st;
  MVPA_LAUNCH(train::silu_gate_backward_kernel, gate_grid(rows, n), dim3(256), 0, (hipStream_t)stream, (const bf16_t*)gu,
              (const bf16_t*)d, (bf16_t*)dgu, rows, n);
  return take_launch_status();
}

extern "C" int mvpa_cosine_steps_backward_bf16(const void* nxt, const void* pred, const float* d, void* d_nxt, void* d_pred, int64_t B,
                                               int64_t T, int64_t C, int32_t cols, float eps, void* stream) {
  if (!nxt || !pred || !d || (!d_nxt && !d_pred)) return MVPA_ERR_NULL;
  if (B <= 0 || T <= 1 || C <= 0 || cols <= 0 || T > ((int64_t)1 << 31) / C || B > ((int64_t)1 << 31) / (T * C)) return MVPA_ERR_SHAPE;
  if (cols % 8 != 0 || (((uintptr_t)nxt | (uintptr_t)pred | (uintptr_t)d_nxt | (uintptr_t)d_pred) & 15)) return MVPA_ERR_ALIGN;
  const int64_t rows = B * T * C;
  MVPA_LAUNCH(train::cosine_steps_backward_kernel, dim3((unsigned)((rows + 3) / 4)), dim3(256), 0, (hipStream_t)stream,
              (const bf16_t*)nxt, (const bf16_t*)pred, d, (bf16_t*)d_nxt, (bf16_t*)d_pred, rows, T, C, cols, eps);
  return take_launch_status();
}

// the parts' rows follow one another in the stacked weight; *rows: their sum, *most: the largest part
static int lora_check(const mvpa_lora_part* parts, int32_t n, int32_t K, int32_t r, const void* stacked, bool backward,
                      train::lora_parts& out, int32_t* most) {
  if (!parts || !stacked) return MVPA_ERR_NULL;
  if (n <= 0 || n > MVPA_LORA_PARTS || K <= 0 || r <= 0) return MVPA_ERR_SHAPE;
  if (K % 8 != 0 || ((uintptr_t)stacked & 15)) return MVPA_ERR_ALIGN;
  int64_t row0 = 0;
  *most = 0;
  for (int i = 0; i < n; ++i) {
    mvpa_lora_part p = parts[i];
    if (p.rows <= 0 || p.rows > MVPA_LORA_ROWS) return MVPA_ERR_SHAPE;
    if ((!backward && !p.w) || !p.a != !p.b) return MVPA_ERR_NULL;
    if ((((uintptr_t)p.a | (uintptr_t)p.b) & (r % 8 == 0 ? 15 : 1)) || ((uintptr_t)p.a & 15) || (!backward && ((uintptr_t)p.w & 15))) return MVPA_ERR_ALIGN;
    p.row0 = row0;
    row0 += p.rows;
    if (p.rows > *most) *most = p.rows;
    out.p[i] = p;
  }
  return MVPA_OK;
}

extern "C" int mvpa_lora_stack_bf16(const mvpa_lora_part* parts, int32_t n, int32_t K, int32_t r, float scale, void* out,
                                    void* stream) {
  train::lora_parts args;
  int32_t most;
  const int st = lora_check(parts, n, K, r, out, false, args, &most);
  if (st != MVPA_OK) return st;
  MVPA_LAUNCH(r % 8 == 0 ? train::lora_stack_kernel<true> : train::lora_stack_kernel<false>,
              dim3((unsigned)((most + train::LORA_ROWS - 1) / train::LORA_ROWS), (unsigned)((K + 1023) / 1024), (unsigned)n), dim3(128),
              0, (hipStream_t)stream, args, (bf16_t*)out, K, r, scale);
  return take_launch_status();
}

extern "C" int mvpa_lora_stack_backward_bf16(const mvpa_lora_part* parts, int32_t n, int32_t K, int32_t r, float scale,
                                             const void* d_out, void* stream) {
  train::lora_parts args;
  int32_t most;
  const int st = lora_check(parts, n, K, r, d_out, true, args, &most);
  if (st != MVPA_OK) return st;
  MVPA_LAUNCH(r % 8 == 0 ? train::lora_stack_backward_kernel<true> : train::lora_stack_backward_kernel<false>, dim3((unsigned)((K + 63) / 64 + (most + 15) / 16), (unsigned)n), dim3(1024), 0,
              (hipStream_t)stream, args, (const bf16_t*)d_out, K, r, scale);
  return take_launch_status();
}
