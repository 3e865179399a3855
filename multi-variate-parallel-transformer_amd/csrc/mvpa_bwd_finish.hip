// From the backward's fp32 results to the gradients of the operator's inputs (bf16, head size 64 or 128).
//
// mvpa_backward leaves the content share of dq, dk and dv in fp32 and the gradients G of the two bias
// tables [B,H,N,T], [B,H,N,C]; what autograd makes of attentions/attn.py:1305-1314 turns them into
//     dq          = dq_content + G_time k_time + G_chan k_chan          (per kv head, rows of its heads)
//     d k_time[j] = sum_rows G_time[:, j] (q + v),   d k_chan likewise with z
//     dv          = sum_rows G_time k_time = (column sums of G_time) k_time,  dz likewise,  du = sum_rows dq_content
// As tensor operations this is some twenty passes over the largest tensors of the backward (casts, two
// batched products each way, sums: 0.85 ms beside 1.7 ms of kernels at B4 H16 C64 T128).  Here nothing of G's size
// is written, and G is read
//   once, by finish_fused (below), where the sums of all table rows fit the registers of a workgroup: up to 640
//   columns of both tables, each rounded up to 64, at Dh 64 and 256 at Dh 128;
//   else twice:
//     finish_rows     128 query rows per workgroup: products with the tables on MFMA, dq to bf16 where the
//                     caller wants it, partial column sums of dq_content
//     finish_tables   128 table rows per workgroup over a share of the query rows: G^T q on MFMA (both
//                     operands by transposing LDS reads), column sums of G; fp32 partial results
//   finish_reduce   the partial results to dk_time, dk_chan; finish_biases: du, dv, dz
// Columns of G_time that the causal mask empties (j < T-1-tq) are skipped.  HBM bound: at that size, G being
// 400 MB of which 270 are read, 148 us in one read (3.6 TB/s with dq and q) and 187 + 189 in two.  dk and dv come rounded from
// the key pass; finish_kv rounds and adds them (60 us at that size) where each query head has parts of its own or
// the results lie over what the passes read.
#include "mvpa_mfma_tools.h"

namespace mvpa {
namespace fin {

constexpr int ROWS = 128;            // query rows per workgroup of finish_rows
constexpr int JB = 64;               // table rows per step of finish_rows
constexpr int TJ = 128, TN = 64;     // table rows per workgroup, query rows per step of finish_tables

struct fin_args {
  int32_t B, H, Hkv, T, C, N, kv_done;
  const bf16_t* q;
  int64_t q_sb, q_sh, q_sn;
  const bf16_t *bias_v, *bias_z, *k_time, *k_chan;
  const float *dq, *dk, *dv, *gt, *gc;
  bf16_t *dq_out, *dk_out, *dv_out;
  int64_t dq_sb, dq_sh, dq_sn, dk_sb, dk_sh, dk_sn, dv_sb, dv_sh, dv_sn;
  float *p_du, *p_tab, *p_col;       // partial results: [b,h][row tile][Dh], [part][T + C][Dh], [part][T + C]
  float* csum;                       // [Hkv][T + C] column sums of G
  bf16_t *du, *dvb, *dz, *dk_time, *dk_chan;
  int32_t kv_parts;                  // query heads whose partial dk, dv make one kv head's (1: summed already)
  int32_t tj_t, tj_c, n_split, split_len;   // column tiles of the two tables; row shares and their length
  int32_t fused;                     // finish_fused: n_split workgroups a head
};

// four consecutive fp32 of a table-gradient row as bf16; zeros past the end
__device__ inline bf16x4 load4(const float* row, int col, int cols, bool vec) {
  float v[4] = {0.f, 0.f, 0.f, 0.f};
  if (vec && col + 3 < cols) {
    const float4 x = *(const float4*)(row + col);
    v[0] = x.x; v[1] = x.y; v[2] = x.z; v[3] = x.w;
  } else {
#pragma unroll
    for (int i = 0; i < 4; ++i)
      if (col + i < cols) v[i] = row[col + i];
  }
  return bf16x4{(__bf16)v[0], (__bf16)v[1], (__bf16)v[2], (__bf16)v[3]};
}

// fragment of a [rows][columns] tile for a product contracted over its rows: column 32 mt + ln, rows
// 16 s + 8 rd + 4 hh + e in element 4 rd + e (row pitch ROWB, swizzle swz_v<DH>)
template <int DH>
struct tr_tile {
  static constexpr int ROWB = DH * 2;
  static __device__ inline bf16x8 frag(const unsigned char* tile, int s, int mt, int lane) {
    const int ln = lane & 31, hh = lane >> 5, e = (ln & 15) >> 2, aa = ln & 3, grp = ln >> 4, row0 = 4 * hh + e;
    const unsigned char* p = tile + (16 * s + row0) * ROWB + (((4 * mt + 2 * grp + (aa >> 1)) ^ swz_v<DH>(row0)) << 4) + ((aa & 1) << 3);
    const bf16x4 lo = el_bf16::read_tr(p), hi = el_bf16::read_tr(p + 8 * ROWB);
    return __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
  }
  static __device__ inline int offset(int row, int col) {          // byte offset of element (row, col), col a multiple of 4
    return row * ROWB + (((col >> 3) ^ swz_v<DH>(row)) << 4) + ((col & 4) << 1);
  }
};

template <int DH>
__global__ __launch_bounds__(256) void finish_rows_kernel(fin_args a) {
  constexpr int MT = DH / 32, ROWB = DH * 2, GP = JB + 8;
  __shared__ __attribute__((aligned(16))) bf16_t Gs[4][32 * GP];
  __shared__ __attribute__((aligned(16))) unsigned char Ts[JB * ROWB];
  __shared__ float red[256];
  const int tid = threadIdx.x, lane = tid & 63, ln = lane & 31, hh = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int bh = blockIdx.y, b = bh / a.H, h = bh % a.H, g = h / (a.H / a.Hkv);
  const int n0 = blockIdx.x * ROWS, nw = n0 + wave * 32;
  const int64_t rbase = (int64_t)bh * a.N;
  f32x16 acc[MT];
#pragma unroll
  for (int mt = 0; mt < MT; ++mt)
#pragma unroll
    for (int i = 0; i < 16; ++i) acc[mt][i] = 0.f;
  const int tq_hi = min(n0 + ROWS - 1, a.N - 1) / a.C;
#pragma unroll 1
  for (int which = 0; which < 2; ++which) {
    const float* G = which ? a.gc : a.gt;
    if (!G) continue;
    const int cols = which ? a.C : a.T;
    const bf16_t* tab = (which ? a.k_chan : a.k_time) + (int64_t)g * cols * DH;
    const bool vec = (cols & 3) == 0;
    const int j_first = which ? 0 : (a.T - 1 - tq_hi) / JB * JB;
#pragma unroll 1
    for (int j0 = j_first; j0 < cols; j0 += JB) {
      __syncthreads();
      // table rows j0 .. (shared), G rows of the wave (its own): 16 lanes x 4 columns, 4 rows at a time;
      // the four-column groups of 16 in the order 0 2 1 3, so that a lane's 8 operand elements are together
#pragma unroll
      for (int i = 0; i < JB * DH / 8 / 256; ++i) {
        const int c = i * 256 + tid, r = c / (DH / 8), ch = c % (DH / 8);
        u32x4 v = {0u, 0u, 0u, 0u};
        if (j0 + r < cols) v = *(const u32x4*)(tab + (int64_t)(j0 + r) * DH + ch * 8);
        *(u32x4*)(Ts + r * ROWB + ((ch ^ swz_v<DH>(r)) << 4)) = v;
      }
      const int c16 = lane & 15, grp4 = (c16 & 12) | ((c16 & 1) << 1) | ((c16 >> 1) & 1);
      bf16x4 gv[8];
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const int r = i * 4 + (lane >> 4), n = nw + r;
        gv[i] = n < a.N ? load4(G + (rbase + n) * cols, j0 + c16 * 4, cols, vec) : bf16x4{};
      }
#pragma unroll
      for (int i = 0; i < 8; ++i) *(bf16x4*)(&Gs[wave][(i * 4 + (lane >> 4)) * GP + grp4 * 4]) = gv[i];
      __syncthreads();
#pragma unroll
      for (int s = 0; s < JB / 16; ++s) {
        const bf16x8 gf = *(const bf16x8*)(&Gs[wave][ln * GP + s * 16 + hh * 8]);
#pragma unroll
        for (int mt = 0; mt < MT; ++mt)
          acc[mt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(tr_tile<DH>::frag(Ts, s, mt, lane), gf, acc[mt], 0, 0, 0);
      }
    }
  }
  // dq = content share + table shares; lane: row nw + ln, columns 32 mt + 8 a4 + 4 hh + 0..3
  const int n = nw + ln;
  if (n < a.N) {
    const float* src = a.dq + (rbase + n) * DH;
    bf16_t* dst = a.dq_out + b * a.dq_sb + h * a.dq_sh + (int64_t)n * a.dq_sn;
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
      for (int a4 = 0; a4 < 4; ++a4) {
        const int d = mt * 32 + a4 * 8 + hh * 4;
        const float4 c = *(const float4*)(src + d);
        *(bf16x4*)(dst + d) = bf16x4{(__bf16)(c.x + acc[mt][a4 * 4]), (__bf16)(c.y + acc[mt][a4 * 4 + 1]),
                                     (__bf16)(c.z + acc[mt][a4 * 4 + 2]), (__bf16)(c.w + acc[mt][a4 * 4 + 3])};
      }
  }
  // column sums of the content share (the rows are in the L2 by now)
  {
    const int d = tid % DH;
    float s = 0.f;
    for (int r = tid / DH; r < ROWS; r += 256 / DH)
      if (n0 + r < a.N) s += a.dq[(rbase + n0 + r) * DH + d];
    red[tid] = s;
    __syncthreads();
    if (tid < DH) {
#pragma unroll
      for (int i = 1; i < 256 / DH; ++i) s += red[tid + i * DH];
      a.p_du[((int64_t)bh * gridDim.x + blockIdx.x) * DH + d] = s;
    }
  }
}

// dk, dv: fp32 [B,Hkv,kv_parts,N,Dh] summed over the parts, to bf16 rows at the caller's strides
template <int DH>
__global__ __launch_bounds__(256) void finish_kv_kernel(fin_args a) {
  const int64_t per = (int64_t)a.B * a.Hkv * a.N * (DH / 8);
  int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  const bool is_v = i >= per;
  if (is_v) i -= per;
  if (i >= per) return;
  const int ch = (int)(i % (DH / 8));
  const int64_t r = i / (DH / 8);
  const int n = (int)(r % a.N), bg = (int)(r / a.N), b = bg / a.Hkv, g = bg % a.Hkv;
  const float* src = (is_v ? a.dv : a.dk) + ((int64_t)bg * a.kv_parts * a.N + n) * DH + ch * 8;
  bf16_t* dst = is_v ? a.dv_out + b * a.dv_sb + g * a.dv_sh + (int64_t)n * a.dv_sn
                     : a.dk_out + b * a.dk_sb + g * a.dk_sh + (int64_t)n * a.dk_sn;
  float4 x = *(const float4*)src, y = *(const float4*)(src + 4);
  for (int part = 1; part < a.kv_parts; ++part) {
    src += (int64_t)a.N * DH;
    const float4 x1 = *(const float4*)src, y1 = *(const float4*)(src + 4);
    x.x += x1.x; x.y += x1.y; x.z += x1.z; x.w += x1.w;
    y.x += y1.x; y.y += y1.y; y.z += y1.z; y.w += y1.w;
  }
  *(bf16x8*)(dst + ch * 8) = bf16x8{(__bf16)x.x, (__bf16)x.y, (__bf16)x.z, (__bf16)x.w,
                                    (__bf16)y.x, (__bf16)y.y, (__bf16)y.z, (__bf16)y.w};
}

template <int DH>
__global__ __launch_bounds__(256) void finish_tables_kernel(fin_args a) {
  constexpr int MT = DH / 32, GB = TJ * 2;           // bytes per G row in LDS
  __shared__ __attribute__((aligned(16))) unsigned char Gs[TN * GB];
  __shared__ __attribute__((aligned(16))) unsigned char Qs[TN * DH * 2];
  __shared__ float cred[8][TJ];
  const int tid = threadIdx.x, lane = tid & 63, ln = lane & 31, hh = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int tile = blockIdx.x, split = blockIdx.y, bh = blockIdx.z, b = bh / a.H, h = bh % a.H;
  const bool chan = tile >= a.tj_t;
  const float* G = chan ? a.gc : a.gt;
  const int cols = chan ? a.C : a.T, j0 = (chan ? tile - a.tj_t : tile) * TJ;
  const int row_out = (chan ? a.T : 0) + j0;          // first row of this tile in the [T + C] tables
  const bool vec = (cols & 3) == 0;
  const int64_t rbase = (int64_t)bh * a.N;
  const bf16_t* qbase = a.q + b * a.q_sb + h * a.q_sh;
  int lo = split * a.split_len, hi = min(lo + a.split_len, a.N);
  // query rows that reach a column of this tile: tq >= T-1-(j0+TJ-1)
  if (!chan) lo = max(lo, max(0, a.T - j0 - TJ) * a.C / TN * TN);
  f32x16 acc[MT];
#pragma unroll
  for (int mt = 0; mt < MT; ++mt)
#pragma unroll
    for (int i = 0; i < 16; ++i) acc[mt][i] = 0.f;
  float cs[4] = {0.f, 0.f, 0.f, 0.f};
  const int gc4 = (tid & 31) * 4, gr = tid >> 5;
  float4 gv[TN / 8];
  u32x4 qv[TN * DH / 8 / 256];
  auto request = [&](int n1) {
#pragma unroll
    for (int i = 0; i < TN / 8; ++i) {
      const int n = n1 + gr + 8 * i;
      gv[i] = make_float4(0.f, 0.f, 0.f, 0.f);
      if (n < hi && G) {
        const float* row = G + (rbase + n) * cols + j0;
        if (vec && j0 + gc4 + 3 < cols) gv[i] = *(const float4*)(row + gc4);
        else {
          if (j0 + gc4 < cols) gv[i].x = row[gc4];
          if (j0 + gc4 + 1 < cols) gv[i].y = row[gc4 + 1];
          if (j0 + gc4 + 2 < cols) gv[i].z = row[gc4 + 2];
          if (j0 + gc4 + 3 < cols) gv[i].w = row[gc4 + 3];
        }
      }
    }
#pragma unroll
    for (int i = 0; i < TN * DH / 8 / 256; ++i) {
      const int c = i * 256 + tid, r = c / (DH / 8), ch = c % (DH / 8);
      qv[i] = *(const u32x4*)(qbase + (int64_t)min(n1 + r, a.N - 1) * a.q_sn + ch * 8);   // G is 0 past the end
    }
  };
  if (lo < hi) request(lo);
#pragma unroll 1
  for (int n1 = lo; n1 < hi; n1 += TN) {
    __syncthreads();
#pragma unroll
    for (int i = 0; i < TN / 8; ++i) {
      cs[0] += gv[i].x; cs[1] += gv[i].y; cs[2] += gv[i].z; cs[3] += gv[i].w;
      *(bf16x4*)(Gs + tr_tile<128>::offset(gr + 8 * i, gc4)) =
          bf16x4{(__bf16)gv[i].x, (__bf16)gv[i].y, (__bf16)gv[i].z, (__bf16)gv[i].w};
    }
#pragma unroll
    for (int i = 0; i < TN * DH / 8 / 256; ++i) {
      const int c = i * 256 + tid, r = c / (DH / 8), ch = c % (DH / 8);
      *(u32x4*)(Qs + r * DH * 2 + ((ch ^ swz_v<DH>(r)) << 4)) = qv[i];
    }
    __syncthreads();
    if (n1 + TN < hi) request(n1 + TN);
#pragma unroll
    for (int s = 0; s < TN / 16; ++s) {
      const bf16x8 gf = tr_tile<128>::frag(Gs, s, wave, lane);
#pragma unroll
      for (int mt = 0; mt < MT; ++mt)
        acc[mt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(gf, tr_tile<DH>::frag(Qs, s, mt, lane), acc[mt], 0, 0, 0);
    }
  }
  const int64_t part = (int64_t)bh * a.n_split + split;
  float* P = a.p_tab + part * (a.T + a.C) * DH;
#pragma unroll
  for (int mt = 0; mt < MT; ++mt)
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const int j = wave * 32 + (i >> 2) * 8 + hh * 4 + (i & 3);
      if (j0 + j < cols) P[(int64_t)(row_out + j) * DH + mt * 32 + ln] = acc[mt][i];
    }
#pragma unroll
  for (int i = 0; i < 4; ++i) cred[gr][gc4 + i] = cs[i];
  __syncthreads();
  if (tid < TJ && j0 + tid < cols) {
    float s = 0.f;
#pragma unroll
    for (int i = 0; i < 8; ++i) s += cred[i][tid];
    a.p_col[part * (a.T + a.C) + row_out + tid] = s;
  }
}

// ---- both products of G in one read ------------------------------------------------------------
// A workgroup walks row tiles of one (b, h), `n_split` apart so that long and short rows of the causal mask are
// dealt evenly, and keeps the fp32 table sums of ALL columns in registers over them: 16 a lane and step of 64
// columns at Dh 64.  Per row tile and step a tile of G goes through LDS once, as bf16, and is read there twice:
// by rows for dq^T += table^T G^T and by columns for the tables' G^T q.  The next tile of G is in flight
// meanwhile, and a second workgroup on the CU covers the barriers.
constexpr int FR = 128, FC = 64;     // rows of a tile, columns of a step

// chunk swizzle of G rows of 128 bytes: 16 consecutive rows at one chunk (rows) and 8 rows x 4 chunks
// (transposing reads) both spread over all banks
__device__ inline int swz_g(int row) { return (((row >> 1) & 1) << 2) | ((row >> 2) & 3); }

template <int DH, int MAXS>
__global__ __launch_bounds__(256, DH == 64 && MAXS <= 4 ? 2 : 1) void finish_fused_kernel(fin_args a) {
  constexpr int MT = DH / 32, NT = MT / 2, ROWB = DH * 2, CPR = DH / 8, QL = FR * CPR / 256, GB = FC * 2;
  constexpr int C4 = DH / 4, CI = 32 * C4 / 64;      // float4 columns of a row; a lane's rows of its wave's 32
  constexpr bool EARLY = MAXS <= 4;                  // the content is requested a tile ahead where registers allow it
  extern __shared__ __attribute__((aligned(1024))) unsigned char smem[];
  // G, under the staged fp32 rows of dq; q; the rows of both tables, steps side by side
  unsigned char *Gs = smem, *Qs = smem + FR * DH * 4, *Ts = Qs + FR * ROWB;
  const int tid = threadIdx.x, lane = tid & 63, ln = lane & 31, hh = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int split = blockIdx.x, bh = blockIdx.y, b = bh / a.H, h = bh % a.H, g = h / (a.H / a.Hkv);
  const int time_steps = (a.T + FC - 1) / FC, s_end = a.gc ? time_steps + (a.C + FC - 1) / FC : time_steps;
  const int tiles = (a.N + FR - 1) / FR;
  const int64_t rbase = (int64_t)bh * a.N;
  const bf16_t* qbase = a.q + b * a.q_sb + h * a.q_sh;
  const int c16 = tid & 15, gr = tid >> 4;         // this thread's four columns of a step, its rows gr + 16 i
  // first step of a row tile: columns of G_time below T-1-tq are empty
  auto first_step = [&](int tile) {
    const int tq_hi = min(tile * FR + FR - 1, a.N - 1) / a.C;
    return a.gt ? (a.T - 1 - tq_hi) / FC : time_steps;
  };
  float4 gv[FR / 16];
  // the tile's part of G for step s
  auto request = [&](int tile, int s) {
    const bool chan = s >= time_steps;
    const int cols = chan ? a.C : a.T, j0 = (chan ? s - time_steps : s) * FC, j = j0 + c16 * 4;
    const float* G = (chan ? a.gc : a.gt) + (rbase + tile * FR) * cols + j0;
    const int rows = a.N - tile * FR;
    const uint32_t off = gr * cols + c16 * 4;
    if ((cols & 3) == 0) {
#pragma unroll
      for (int i = 0; i < FR / 16; ++i) {
        gv[i] = make_float4(0.f, 0.f, 0.f, 0.f);
        if (gr + 16 * i < rows && j < cols) gv[i] = *(const float4*)(G + (int64_t)16 * i * cols + off);
      }
    } else {
#pragma unroll
      for (int i = 0; i < FR / 16; ++i) {
        const float* p = G + (int64_t)16 * i * cols + off;
        const bool on = gr + 16 * i < rows;
        gv[i].x = on && j < cols ? p[0] : 0.f;
        gv[i].y = on && j + 1 < cols ? p[1] : 0.f;
        gv[i].z = on && j + 2 < cols ? p[2] : 0.f;
        gv[i].w = on && j + 3 < cols ? p[3] : 0.f;
      }
    }
  };
  // its rows of q, straight to LDS
  const uint32_t q_lds = (uint32_t)(uintptr_t)(LDS_PTR(unsigned char))Qs;
  auto request_q = [&](int tile) {
#pragma unroll
    for (int i = 0; i < QL; ++i) {
      const int c = i * 256 + tid, r = c / CPR, ch = (c % CPR) ^ swz_v<DH>(r);
      load_to_lds_16(qbase + (int64_t)min(tile * FR + r, a.N - 1) * a.q_sn + ch * 8,           // G is 0 past the end
                     __builtin_amdgcn_readfirstlane(q_lds + (i * 256 + wave * 64) * 16));
    }
  };
  for (int c = tid; c < s_end * FC * CPR; c += 256) {
    const int r = c / CPR, ch = c % CPR;
    const bool chan = r >= time_steps * FC;
    const int j = chan ? r - time_steps * FC : r, cols = chan ? a.C : a.T;
    u32x4 v = {0u, 0u, 0u, 0u};
    if (j < cols) v = *(const u32x4*)((chan ? a.k_chan : a.k_time) + ((int64_t)g * cols + j) * DH + ch * 8);
    *(u32x4*)(Ts + r * ROWB + ((ch ^ swz_v<DH>(r)) << 4)) = v;
  }
  f32x16 tab[MAXS][NT];
  float cs[MAXS][4];
  float4 dus = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
  for (int s = 0; s < MAXS; ++s) {
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
      for (int i = 0; i < 16; ++i) tab[s][t][i] = 0.f;
#pragma unroll
    for (int i = 0; i < 4; ++i) cs[s][i] = 0.f;
  }
  const int jt = wave & 1, dt = (wave >> 1) * NT;    // this wave's columns of a step and rows of the table sums' transpose
  // Addresses in LDS: every swizzle has a period of 16 rows, so that rows 16 i on are constants away.
  // G is written with the four-column groups of 16 in the order 0 2 1 3, so that a lane's 8 operand elements of
  // a row are together.
  const int col_w = ((c16 & 12) | ((c16 & 1) << 1) | ((c16 >> 1) & 1)) * 4;
  unsigned char* const g_write = Gs + gr * GB + (((col_w >> 3) ^ swz_g(gr)) << 4) + ((col_w & 4) << 1);
  const unsigned char* const g_row = Gs + (wave * 32 + ln) * GB;
  const int g_chunk = (hh ^ swz_g(ln)) << 4;
  const int tr_row = 4 * hh + ((ln & 15) >> 2), tr_chunk = 4 * jt + 2 * (ln >> 4) + ((ln & 3) >> 1);
  const unsigned char* const g_lo = Gs + tr_row * GB + ((ln & 1) << 3) + ((tr_chunk ^ swz_g(tr_row)) << 4);
  const unsigned char* const g_hi = Gs + (tr_row + 8) * GB + ((ln & 1) << 3) + ((tr_chunk ^ swz_g(tr_row + 8)) << 4);
  int s = 0, tile = split;
  if (tile < tiles) {
    s = first_step(tile);
    request_q(tile);
    if (s < s_end) request(tile, s);
  }
#pragma unroll 1
  while (tile < tiles) {
    // the content share of the wave's rows, a lane four columns of every 64 / C4-th of them
    float4 cont[CI];
    auto request_content = [&]() {
#pragma unroll
      for (int i = 0; i < CI; ++i) {
        const int row = tile * FR + wave * 32 + i * (64 / C4) + lane / C4;
        cont[i] = make_float4(0.f, 0.f, 0.f, 0.f);
        if (row < a.N) cont[i] = *(const float4*)(a.dq + (rbase + row) * DH + lane % C4 * 4);
      }
    };
    if (EARLY) request_content();
    f32x16 acc[MT];
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
      for (int i = 0; i < 16; ++i) acc[mt][i] = 0.f;
    const int next = tile + gridDim.x, next_s = next < tiles ? first_step(next) : s_end;
    bool fresh = true;
#pragma unroll 1
    for (; s < s_end; ++s) {
      __syncthreads();                               // everyone is done with the tiles before
#pragma unroll
      for (int i = 0; i < FR / 16; ++i)
        *(bf16x4*)(g_write + i * 16 * GB) = bf16x4{(__bf16)gv[i].x, (__bf16)gv[i].y, (__bf16)gv[i].z, (__bf16)gv[i].w};
#pragma unroll
      for (int ss = 0; ss < MAXS; ++ss)
        if (s == ss)
#pragma unroll
          for (int i = 0; i < FR / 16; ++i) {
            cs[ss][0] += gv[i].x; cs[ss][1] += gv[i].y; cs[ss][2] += gv[i].z; cs[ss][3] += gv[i].w;
          }
      if (fresh) wait_vmcnt_imm<0>();                // q is in LDS
      fresh = false;
      __syncthreads();
      {
        const bool more = s + 1 < s_end;
        if (more || next_s < s_end) request(more ? tile : next, more ? s + 1 : next_s);
      }
      const unsigned char* tab_rows = Ts + s * FC * ROWB;
#pragma unroll
      for (int k = 0; k < FC / 16; ++k) {
        const bf16x8 gf = *(const bf16x8*)(g_row + (g_chunk ^ (k << 5)));
#pragma unroll
        for (int mt = 0; mt < MT; ++mt)
          acc[mt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(tr_tile<DH>::frag(tab_rows, k, mt, lane), gf, acc[mt], 0, 0, 0);
      }
#pragma unroll
      for (int ss = 0; ss < MAXS; ++ss)
        if (s == ss) {
#pragma unroll
          for (int k = 0; k < FR / 16; ++k) {
            const bf16x4 lo = el_bf16::read_tr(g_lo + k * 16 * GB), hi = el_bf16::read_tr(g_hi + k * 16 * GB);
            const bf16x8 gf = __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
#pragma unroll
            for (int t = 0; t < NT; ++t)
              tab[ss][t] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(gf, tr_tile<DH>::frag(Qs, k, dt + t, lane), tab[ss][t], 0, 0, 0);
          }
        }
    }
    if (fresh && next_s < s_end) request(next, next_s);      // nothing to multiply here
    // dq = content share + table shares: the latter go by rows through LDS, over G and q
    if (!EARLY) request_content();
    __syncthreads();
    if (next < tiles) request_q(next);
    unsigned char* st = smem + wave * 32 * ROWB * 2;
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
      for (int a4 = 0; a4 < 4; ++a4)
        *(float4*)(st + ln * ROWB * 2 + (((8 * mt + 2 * a4 + hh) ^ (ln & (C4 - 1))) << 4)) =
            make_float4(acc[mt][a4 * 4], acc[mt][a4 * 4 + 1], acc[mt][a4 * 4 + 2], acc[mt][a4 * 4 + 3]);
    wave_lds_sync();
#pragma unroll
    for (int i = 0; i < CI; ++i) {
      const int r = i * (64 / C4) + lane / C4, row = tile * FR + wave * 32 + r;
      const float4 v = *(const float4*)(st + r * ROWB * 2 + (((lane % C4) ^ (r & (C4 - 1))) << 4)), c = cont[i];
      dus.x += c.x; dus.y += c.y; dus.z += c.z; dus.w += c.w;
      if (row < a.N)
        *(bf16x4*)(a.dq_out + b * a.dq_sb + h * a.dq_sh + (int64_t)row * a.dq_sn + lane % C4 * 4) =
            bf16x4{(__bf16)(c.x + v.x), (__bf16)(c.y + v.y), (__bf16)(c.z + v.z), (__bf16)(c.w + v.w)};
    }
    tile = next;
    s = next_s;
  }
  const int64_t part = (int64_t)bh * gridDim.x + split, rows = a.T + a.C;
  float* P = a.p_tab + part * rows * DH;
  float* red = (float*)smem;
#pragma unroll
  for (int ss = 0; ss < MAXS; ++ss) {
    const bool chan = ss >= time_steps;
    const int cols = chan ? a.C : a.T, j0 = (chan ? ss - time_steps : ss) * FC, row0 = chan ? a.T : 0;
    if (j0 >= cols) continue;
    // rows of the MFMA tile are LDS columns: undo the order of the four-column groups
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        const int j = j0 + jt * 32 + (i >> 3) * 16 + hh * 8 + ((i >> 2) & 1) * 4 + (i & 3);
        if (j < cols) P[(int64_t)(row0 + j) * DH + (dt + t) * 32 + ln] = tab[ss][t][i];
      }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < 4; ++i) red[gr * FC + c16 * 4 + i] = cs[ss][i];
    __syncthreads();
    if (tid < FC && j0 + tid < cols) {
      float sum = 0.f;
#pragma unroll
      for (int i = 0; i < 16; ++i) sum += red[i * FC + tid];
      a.p_col[part * rows + row0 + j0 + tid] = sum;
    }
  }
  __syncthreads();
  *(float4*)(red + (tid / C4) * DH + tid % C4 * 4) = dus;
  __syncthreads();
  if (tid < DH) {
    float sum = 0.f;
#pragma unroll
    for (int i = 0; i < 256 / C4; ++i) sum += red[i * DH + tid];
    a.p_du[part * DH + tid] = sum;
  }
}

// one workgroup per table row of a kv head, its threads' 256 / DH shares of the partial results merged through LDS
// (B4 C64 T25 H12/4, 336 parts: 14.6 -> 6 us against a share of one thread)
template <int DH>
__global__ __launch_bounds__(256) void finish_reduce_kernel(fin_args a) {
  constexpr int SHARES = 256 / DH;
  __shared__ float red[256], redc[SHARES];
  const int g = blockIdx.y, rows = a.T + a.C, j = blockIdx.x, d = threadIdx.x % DH, share = threadIdx.x / DH;
  const int grp = a.H / a.Hkv, np = grp * a.n_split;
  float s = 0.f, c = 0.f;
#pragma unroll 8
  for (int i = share; i < a.B * np; i += SHARES) {
    const int b = i / np, p = (b * a.H + g * grp) * a.n_split + i % np;
    s += a.p_tab[((int64_t)p * rows + j) * DH + d];
    c += a.p_col[(int64_t)p * rows + j];
  }
  red[threadIdx.x] = s;
  if (d == 0) redc[share] = c;
  __syncthreads();
  if (share > 0) return;
#pragma unroll
  for (int i = 1; i < SHARES; ++i) {
    s += red[i * DH + d];
    c += redc[i];
  }
  const bool chan = j >= a.T;
  s += c * bf16_to_f32((chan ? a.bias_z : a.bias_v)[g * DH + d]);
  bf16_t* dst = chan ? a.dk_chan + ((int64_t)g * a.C + j - a.T) * DH : a.dk_time + ((int64_t)g * a.T + j) * DH;
  dst[d] = f32_to_bf16(s);
  if (d == 0) a.csum[(int64_t)g * rows + j] = c;
}

// du, dv, dz of a kv head: blockIdx.y = 0, 1, 2
template <int DH>
__global__ __launch_bounds__(1024) void finish_biases_kernel(fin_args a, int row_tiles) {
  __shared__ float red[1024];
  const int g = blockIdx.x, d = threadIdx.x % DH, sub = threadIdx.x / DH;
  constexpr int SUBS = 1024 / DH;
  const int grp = a.H / a.Hkv;
  float s = 0.f;
  if (blockIdx.y == 0) {
    const int per = grp * row_tiles;
    for (int i = sub; i < a.B * per; i += SUBS)
      s += a.p_du[(((int64_t)(i / per) * a.H + g * grp) * row_tiles + i % per) * DH + d];
  } else {
    const bool chan = blockIdx.y == 2;
    const int cols = chan ? a.C : a.T;
    const bf16_t* tab = (chan ? a.k_chan : a.k_time) + (int64_t)g * cols * DH;
    const float* c = a.csum + (int64_t)g * (a.T + a.C) + (chan ? a.T : 0);
    for (int j = sub; j < cols; j += SUBS) s += c[j] * bf16_to_f32(tab[(int64_t)j * DH + d]);
  }
  red[threadIdx.x] = s;
  __syncthreads();
  if (sub == 0) {
#pragma unroll
    for (int i = 1; i < SUBS; ++i) s += red[threadIdx.x + i * DH];
    (blockIdx.y == 0 ? a.du : blockIdx.y == 1 ? a.dvb : a.dz)[g * DH + d] = f32_to_bf16(s);
  }
}

struct layout {
  int64_t used = 0;
  char* base;
  template <typename T> T* take(int64_t n) {
    T* p = base ? (T*)(base + used) : nullptr;
    used += (n * (int64_t)sizeof(T) + 255) & ~(int64_t)255;
    return p;
  }
};

// row shares of finish_tables: enough workgroups for two rounds of the chip, whole TN-row steps
static void row_split(const mvpa_bwd_args* b, int* n_split, int* len) {
  const int64_t N = (int64_t)b->T * b->C;
  const int tiles = (b->T + TJ - 1) / TJ + (b->C + TJ - 1) / TJ;
  int64_t s = 512 / ((int64_t)tiles * b->B * b->H);
  const int64_t most = (N + 4 * TN - 1) / (4 * TN);
  if (s > most) s = most;
  if (s < 1) s = 1;
  *len = (int)(((N + s - 1) / s + TN - 1) / TN * TN);
  *n_split = (int)((N + *len - 1) / *len);
}

// A workgroup of the key pass walks the query heads of a kv head one after the other.  Where its workgroups (counted
// as four key steps each) are less than two rounds of the chip, each query head gets its own, and finish_kv adds up their dk, dv.
// Forward and backward without / with, us: B4 C64 T25 H12/4 (112 workgroups) 240 / 197, B1 C64 T64 (64) 405 / 275,
// B4 C21 T100 (400) 490 / 425, B8 C32 T64 (512) 482 / 506, B32 C64 T25 (896) 1122 / 1215; Dh 128, H16/8: B1 C128 T128
// (256) 5036 / 4582, B1 C32 T192 (384) 952 / 972.
// Long walks at Dh 64 gain up to twice as many, the far kernel's workgroups with them: B2 C64 T256 (512) 2331 / 2003,
// B4 C40 T200 (800) 2845 / 2297, B4 C64 T256 (1024) 4670 / 3960, B8 C64 T128 (1024) 2800 / 2620, B16 C64 T64 (1024)
// 2018 / 2008, B6 C64 T256 (1536) 5870 / 6010, B8 C64 T256 (2048) 7810 / 8200.
// At Dh 128, H16/8, above 32 channels: B2 C64 T64 (256) 789 / 839, B8 C64 T25 (448) 873 / 954, B4 C40 T60 (480) 1296 / 1280; B2 C64 T100 (400) 1515 /
// 1475, B2 C64 T128 (512) 2053 / 2002, B1 C64 T256 (512) 3446 / 3201, B3 C64 T128 (768) 2875 / 3007.
static bool per_head(const mvpa_bwd_args* b) {
  const int64_t full = b->C <= 32 ? 512 : b->Dh == 64 ? (b->T >= 64 ? 1280 : 512) : b->T >= 96 ? 640 : 256;
  return b->H > b->Hkv && (int64_t)b->B * b->Hkv * ((b->T + 3) / 4) < full;
}

// dk and dv share no memory with what the passes read
static bool apart(const mvpa_bwd_args* a, const mvpa_bwd_grads* o) {
  struct span { uintptr_t lo, hi; };
  const int64_t N = (int64_t)a->T * a->C;
  auto rows = [&](const void* p, int heads, int64_t sb, int64_t sh, int64_t sn) {
    int64_t lo = 0, hi = a->Dh;
    for (const int64_t reach : {(a->B - 1) * sb, (heads - 1) * sh, (N - 1) * sn}) (reach < 0 ? lo : hi) += reach;
    return span{(uintptr_t)p + 2 * lo, (uintptr_t)p + 2 * hi};
  };
  auto flat = [](const void* p, int64_t bytes) { return span{(uintptr_t)p, (uintptr_t)p + (p ? bytes : 0)}; };
  const span outs[] = {rows(o->dk, a->Hkv, o->dk_stride_b, o->dk_stride_h, o->dk_stride_n),
                       rows(o->dv, a->Hkv, o->dv_stride_b, o->dv_stride_h, o->dv_stride_n)};
  const span ins[] = {rows(a->q, a->H, a->q_stride_b, a->q_stride_h, a->q_stride_n),
                      rows(a->k, a->Hkv, a->k_stride_b, a->k_stride_h, a->k_stride_n),
                      rows(a->v, a->Hkv, a->v_stride_b, a->v_stride_h, a->v_stride_n),
                      rows(a->o, a->H, a->o_stride_b, a->o_stride_h, a->o_stride_n),
                      rows(a->d_o, a->H, a->do_stride_b, a->do_stride_h, a->do_stride_n),
                      flat(a->lse, 4 * a->B * a->H * N), flat(a->bias_u, 2 * a->Hkv * a->Dh), flat(a->bias_v, 2 * a->Hkv * a->Dh),
                      flat(a->bias_z, 2 * a->Hkv * a->Dh), flat(a->k_time, 2ll * a->Hkv * a->T * a->Dh),
                      flat(a->k_chan, 2ll * a->Hkv * a->C * a->Dh), flat(a->chan_valid, (int64_t)a->B * a->C)};
  for (const span& x : outs)
    for (const span& y : ins)
      if (x.lo < y.hi && y.lo < x.hi) return false;
  return true;
}

// steps of 64 columns that finish_fused keeps sums for, 0 where they do not fit the registers
static int fused_steps(const mvpa_bwd_args* b) {
  const int steps = (b->T + FC - 1) / FC + (b->C + FC - 1) / FC;
  return steps <= 4 ? 4 : steps <= 10 && b->Dh == 64 ? 10 : 0;
}

static void lay_out(const mvpa_bwd_args* b, fin_args& f, mvpa_bwd_args& w, layout& l) {
  const int64_t N = (int64_t)b->T * b->C, bhn = (int64_t)b->B * b->H * N, bgn = (int64_t)b->B * b->Hkv * N, Dh = b->Dh;
  w = *b;
  w.dq = l.take<float>(bhn * Dh);
  f.kv_parts = per_head(b) ? b->H / b->Hkv : 1;
  w.dk = l.take<float>(bgn * f.kv_parts * Dh);
  w.dv = l.take<float>(bgn * f.kv_parts * Dh);
  w.dbias_time = l.take<float>(bhn * b->T);
  w.dbias_chan = l.take<float>(bhn * b->C);
  w.ws_delta = l.take<float>(bhn);
  w.ws_time = l.take<float>(bhn * b->T);
  w.ws_chan = l.take<float>(bhn * ((b->C + 3) / 4 * 4));
  w.ws_qu = l.take<bf16_t>(bhn * Dh);
  const int64_t row_tiles = (N + ROWS - 1) / ROWS;
  f.fused = fused_steps(b);
  int n_split, len = 0;
  if (f.fused) {
    const int64_t s = (Dh == 64 && f.fused == 4 ? 512 : 256) / ((int64_t)b->B * b->H);    // two workgroups a CU, one at Dh 128
    // as few as walk no more tiles each: 13 tiles take two rounds with 12 workgroups and with 7
    const int64_t each = s < 1 ? row_tiles : (row_tiles + s - 1) / s;
    n_split = (int)((row_tiles + each - 1) / each);
  } else {
    row_split(b, &n_split, &len);
  }
  f.n_split = n_split;
  f.split_len = len;
  f.tj_t = (b->T + TJ - 1) / TJ;
  f.tj_c = (b->C + TJ - 1) / TJ;
  const int64_t parts = (int64_t)b->B * b->H * n_split, rows = b->T + b->C;
  f.p_du = l.take<float>((int64_t)b->B * b->H * row_tiles * Dh);
  f.p_tab = l.take<float>(parts * rows * Dh);
  f.p_col = l.take<float>(parts * rows);
  f.csum = l.take<float>(b->Hkv * rows);
}

template <int DH>
static int launch_finish(const fin_args& f, hipStream_t s) {
  const int row_tiles = f.fused ? f.n_split : (f.N + ROWS - 1) / ROWS;
  if (f.fused) {
    const size_t lds = (size_t)FR * DH * 6 +
                       (size_t)((f.T + FC - 1) / FC + (f.C + FC - 1) / FC) * FC * DH * 2;
    auto kern = finish_fused_kernel<DH, 4>;
    if constexpr (DH == 64) kern = f.fused == 10 ? finish_fused_kernel<64, 10> : kern;
    want_dynamic_lds((const void*)kern, (int)lds);
    MVPA_LAUNCH(kern, dim3((unsigned)f.n_split, (unsigned)(f.B * f.H)), dim3(256), lds, s, f);
  } else {
    MVPA_LAUNCH(finish_rows_kernel<DH>, dim3((unsigned)row_tiles, (unsigned)(f.B * f.H)), dim3(256), 0, s, f);
    MVPA_LAUNCH(finish_tables_kernel<DH>, dim3((unsigned)(f.tj_t + f.tj_c), (unsigned)f.n_split, (unsigned)(f.B * f.H)),
                dim3(256), 0, s, f);
  }
  const int64_t kv = 2 * (int64_t)f.B * f.Hkv * f.N * (DH / 8);
  if (!f.kv_done) {
    MVPA_LAUNCH(finish_kv_kernel<DH>, dim3((unsigned)((kv + 255) / 256)), dim3(256), 0, s, f);
  }
  MVPA_LAUNCH(finish_reduce_kernel<DH>, dim3((unsigned)(f.T + f.C), (unsigned)f.Hkv), dim3(256), 0, s, f);
  MVPA_LAUNCH(finish_biases_kernel<DH>, dim3((unsigned)f.Hkv, 3), dim3(1024), 0, s, f, row_tiles);
  return take_launch_status();
}

}  // namespace fin
}  // namespace mvpa

using namespace mvpa;

extern "C" size_t mvpa_backward_full_ws_bytes(const mvpa_bwd_args* a) {
  if (!a || a->struct_size != sizeof(mvpa_bwd_args) || a->B <= 0 || a->H <= 0 || a->Hkv <= 0 || a->T <= 0 || a->C <= 0) return 0;
  fin::fin_args f;
  mvpa_bwd_args w;
  fin::layout l{0, nullptr};
  fin::lay_out(a, f, w, l);
  return (size_t)l.used;
}

extern "C" int mvpa_backward_full(const mvpa_bwd_args* a, const mvpa_bwd_grads* o, void* ws, size_t ws_bytes, void* stream) {
  if (!a || !o || !ws) return MVPA_ERR_NULL;
  if (a->struct_size != sizeof(mvpa_bwd_args) || o->struct_size != sizeof(mvpa_bwd_grads)) return MVPA_ERR_STRUCT;
  if (a->dtype != MVPA_BF16 || (a->Dh != 64 && a->Dh != 128)) return MVPA_ERR_UNSUPPORTED;
  if (!o->dq || !o->dk || !o->dv || !o->dbias_u || !o->dbias_v || !o->dbias_z || !o->dk_time || !o->dk_chan) return MVPA_ERR_NULL;
  if ((uintptr_t)ws & 255) return MVPA_ERR_ALIGN;
  if (((uintptr_t)o->dq | (uintptr_t)o->dk | (uintptr_t)o->dv) & 15) return MVPA_ERR_ALIGN;
  if ((o->dq_stride_b | o->dq_stride_h | o->dq_stride_n | o->dk_stride_b | o->dk_stride_h | o->dk_stride_n |
       o->dv_stride_b | o->dv_stride_h | o->dv_stride_n) & 7) return MVPA_ERR_ALIGN;
  fin::fin_args f = {};
  mvpa_bwd_args w;
  fin::layout l{0, (char*)ws};
  fin::lay_out(a, f, w, l);
  if ((size_t)l.used > ws_bytes) return MVPA_ERR_WS_SIZE;
  if (!mvpa_bwd_query_mfma_supported(&w)) return MVPA_ERR_UNSUPPORTED;
  // dk and dv from the key pass itself, unless parts of them are to be added or they lie where inputs are still read
  const mvpa_kv_out out{o->dk, o->dv, o->dk_stride_b, o->dk_stride_h, o->dk_stride_n, o->dv_stride_b, o->dv_stride_h, o->dv_stride_n};
  f.kv_done = f.kv_parts == 1 && fin::apart(a, o);
  const int st = mvpa_backward_checked(&w, (hipStream_t)stream, f.kv_parts > 1, f.kv_done ? &out : nullptr);
  if (st != MVPA_OK) return st;
  f.B = a->B; f.H = a->H; f.Hkv = a->Hkv; f.T = a->T; f.C = a->C; f.N = a->T * a->C;
  f.q = (const bf16_t*)a->q;
  f.q_sb = a->q_stride_b; f.q_sh = a->q_stride_h; f.q_sn = a->q_stride_n;
  f.bias_v = (const bf16_t*)a->bias_v; f.bias_z = (const bf16_t*)a->bias_z;
  f.k_time = (const bf16_t*)a->k_time; f.k_chan = (const bf16_t*)a->k_chan;
  f.dq = w.dq; f.dk = w.dk; f.dv = w.dv;
  // a bias term that is switched off takes no part in the forward: its table, its query bias and the query
  // get nothing through it
  f.gt = (a->flags & MVPA_FLAG_TIME_BIAS) ? w.dbias_time : nullptr;
  f.gc = (a->flags & MVPA_FLAG_CHAN_BIAS) ? w.dbias_chan : nullptr;
  f.dq_out = (bf16_t*)o->dq; f.dk_out = (bf16_t*)o->dk; f.dv_out = (bf16_t*)o->dv;
  f.dq_sb = o->dq_stride_b; f.dq_sh = o->dq_stride_h; f.dq_sn = o->dq_stride_n;
  f.dk_sb = o->dk_stride_b; f.dk_sh = o->dk_stride_h; f.dk_sn = o->dk_stride_n;
  f.dv_sb = o->dv_stride_b; f.dv_sh = o->dv_stride_h; f.dv_sn = o->dv_stride_n;
  f.du = (bf16_t*)o->dbias_u; f.dvb = (bf16_t*)o->dbias_v; f.dz = (bf16_t*)o->dbias_z;
  f.dk_time = (bf16_t*)o->dk_time; f.dk_chan = (bf16_t*)o->dk_chan;
  return a->Dh == 64 ? fin::launch_finish<64>(f, (hipStream_t)stream) : fin::launch_finish<128>(f, (hipStream_t)stream);
}
