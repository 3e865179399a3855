// Small-tile bf16 GEMM (y = x w^T): products whose x has few rows.
//
// The 256-row tiles of mvpa_dense.hip give such a product a handful of workgroups (525 rows x 768
// columns: 18 of them on 256 CUs, 50 us for 2 GFLOP).  Here a workgroup is 32 * WM rows of x by 64 rows
// of w, and a product with a long contraction and a narrow output is split over K as well.  The
// time of such a product is the latency of its chain of k-blocks, so the operands come through a ring
// of STAGES direct-to-LDS blocks of 64: STAGES - 1 blocks are in flight at any time, and the fragments of the next block are on
// their way from LDS while this one is multiplied (with a block's fragments read where its products stand, a few
// at a time: 32 rows of x, [768,2624] weights 9.8 -> 6.0 us, [2048,2048] 8.7 -> 5.8; 128 x 64 tiles 16.1 -> 13.6).
//   4 waves.  WM = 4: a wave owns 32 rows of x and all 64 columns.  WM = 2 / 1: two / four waves share
//   the rows and take 32 / 16 of every 64 k each, so that a wave holds two 32 x 32 tiles (for the gated
//   product: the gate and the up columns of an output); a product by itself on 64 rows, whose sums stay one chain, one a
//   wave.  128 columns: twice the waves.
//   The sums go through LDS by rows and every thread finishes and stores 16 bytes of a row: stored as the
//   products leave them, 8 or 16 bytes of each of 32 rows per instruction, the partial sums of 525 rows of 768
//   alone took 3 us.
//   Rows are 128 bytes with the 16-byte chunks XOR-swizzled as in mvpa_dense.hip.
#include "mvpa_tiles.h"

#include "mvpa_mfma_tools.h"

#include <type_traits>

namespace mvpa {

typedef __attribute__((ext_vector_type(4))) float f32x4;

constexpr int TL_BN = 64, TL_BK = 64, TL_ROWB = TL_BK * 2;
constexpr int TL_SUM = TL_BN * 4;                   // bytes of a row of sums: 16 chunks, XOR-swizzled by the row

template <int WM, int STAGES, int CT = 2, int BN = TL_BN>           // CT: tiles of 32 columns of a wave
struct tile_cfg {
  static constexpr int BM = 32 * WM, CW = BN / 32 / CT, NW = BN / 16, KH = NW / (WM * CW);
  static constexpr int XL = BM / 8 / NW, LPW = (BM + BN) / 8 / NW;          // 1 KiB loads per wave and block: of x, in all
  static constexpr int STAGE = (BM + BN) * TL_ROWB;
  static constexpr int LDS = STAGES * STAGE, SUMS = KH * BM * TL_SUM;       // SUMS: of 64 columns
  static_assert(WM * CW * KH == NW && XL * 8 * NW == BM && LPW * 8 * NW == BM + BN && BN / TL_BN * SUMS <= LDS,
                "four waves for every 64 columns, and their sums fit the ring");
};

// The tile's products over k-blocks [kb0, kb1), left in LDS for tile_sum.  wrow(r): which row of W feeds row r of
// the tile.
template <int WM, int STAGES, int CT = 2, int BN = TL_BN, typename WRow>
__device__ __forceinline__ void tile_product(unsigned char* lds, const bf16_t* __restrict__ X, int64_t ldx, int64_t m0,
                                             int64_t M, const bf16_t* __restrict__ W, int64_t ldw, WRow wrow,
                                             int kb0, int kb1) {
  using G = tile_cfg<WM, STAGES, CT, BN>;
  f32x16 acc[CT];
  const int tid = threadIdx.x, lane = tid & 63, ln = lane & 31, hh = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave % WM, wc = wave / WM % G::CW, kh = wave / (WM * G::CW);
  const uint32_t lds0 = (uint32_t)(uintptr_t)(LDS_PTR(unsigned char))lds;

  // load i of a wave: rows (wave + NW i) * 8 .. + 7 of the block, x rows first (i < XL), then w rows
  uint32_t off[G::LPW];
  {
    const int rsub = lane >> 3, phys = lane & 7;
#pragma unroll
    for (int i = 0; i < G::LPW; ++i) {
      const int row = (wave + G::NW * i) * 8 + rsub;
      const int chunk = (phys ^ ((row >> 1) & 7)) << 3;
      if (i < G::XL) {
        const int64_t m = m0 + row;
        off[i] = (uint32_t)((((m < M ? m : M - 1) - m0) * ldx + chunk) * 2);
      } else {
        off[i] = (uint32_t)((wrow(row - G::BM) * ldw + chunk) * 2);
      }
    }
  }
  const bf16_t* xs = X + m0 * ldx + (int64_t)kb0 * TL_BK;
  const bf16_t* ws = W + (int64_t)kb0 * TL_BK;
  uint32_t dst = lds0;
  auto issue = [&]() {
#pragma unroll
    for (int i = 0; i < G::LPW; ++i)
      load_to_lds_16(i < G::XL ? (const void*)xs : (const void*)ws, off[i], dst + (wave + G::NW * i) * 1024);
    xs += TL_BK;
    ws += TL_BK;
    dst = dst + G::STAGE == lds0 + G::LDS ? lds0 : dst + G::STAGE;
  };

#pragma unroll
  for (int j = 0; j < CT; ++j)
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[j][r] = 0.f;
  const int nkb = kb1 - kb0;
#pragma unroll
  for (int s = 0; s < STAGES; ++s)
    if (s < nkb) issue();

  constexpr int SL = 4 / G::KH;                     // 16-wide k-slices of a block per wave
  struct frags { bf16x8 x[SL], w[SL][CT]; };
  int frag[SL];
#pragma unroll
  for (int s = 0; s < SL; ++s) frag[s] = ln * TL_ROWB + (((2 * (kh * SL + s) + hh) ^ ((ln >> 1) & 7)) << 4);
  const unsigned char* st = lds;                    // the stage whose fragments are read next
  auto read = [&](frags& f) {
    const unsigned char* xb = st + wm * 32 * TL_ROWB;
    const unsigned char* wb = st + (G::BM + wc * CT * 32) * TL_ROWB;
#pragma unroll
    for (int s = 0; s < SL; ++s) {
      f.x[s] = *(const bf16x8*)(xb + frag[s]);
#pragma unroll
      for (int j = 0; j < CT; ++j) f.w[s][j] = *(const bf16x8*)(wb + j * 32 * TL_ROWB + frag[s]);
    }
    st = st + G::STAGE == lds + G::LDS ? lds : st + G::STAGE;
  };
  auto multiply = [&](const frags& f) {
#pragma unroll
    for (int s = 0; s < SL; ++s)
#pragma unroll
      for (int j = 0; j < CT; ++j) acc[j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(f.w[s][j], f.x[s], acc[j], 0, 0, 0);
  };
  // One step: block kb's fragments are in registers.  Behind the barrier block kb + 1 has landed (only the loads of
  // younger blocks are still out), and block kb is read by all: its stage takes block kb + STAGES.
  auto step = [&](const frags& now, frags& next) {
    wait_vmcnt_imm<(STAGES - 2) * G::LPW>();
    lds_barrier();
    issue();
    read(next);
    multiply(now);
  };
  frags fa, fb;
  const int steady = max(nkb - STAGES, 0), last = min(STAGES, nkb) - 1;
  if (last == STAGES - 1) wait_vmcnt_imm<(STAGES - 1) * G::LPW>();
  else wait_vmcnt_imm<0>();
  lds_barrier();
  read(fa);
  int kb = 0;
  for (; kb + 1 < steady; kb += 2) {
    step(fa, fb);
    step(fb, fa);
  }
  if (kb < steady) {
    step(fa, fb);
    fa = fb;
  }
  if (last & 1) fb = fa;                            // what is left: an even number of blocks behind this one from fa, an odd from fb
#pragma unroll
  for (int r = STAGES - 1; r >= 0; --r) {
    if (r > last) continue;
    if (r > 0) {
      // (r is a constant of every copy of the loop's body)
      static_assert(STAGES <= 6, "waits below");
      if (r == 5) wait_vmcnt_imm<4 * G::LPW>();
      else if (r == 4) wait_vmcnt_imm<3 * G::LPW>();
      else if (r == 3) wait_vmcnt_imm<2 * G::LPW>();
      else if (r == 2) wait_vmcnt_imm<G::LPW>();
      else wait_vmcnt_imm<0>();
      lds_barrier();
      read(r & 1 ? fa : fb);
    }
    multiply(r & 1 ? fb : fa);
  }
  // every wave's sums by rows of x, [64 columns of the tile][k part][BM rows] over the ring
  lds_barrier();
  unsigned char* sums = lds + (kh * G::BM + wm * 32 + ln) * TL_SUM;
#pragma unroll
  for (int j = 0; j < CT; ++j)
#pragma unroll
    for (int a4 = 0; a4 < 4; ++a4)
      *(float4*)(sums + (wc * CT + j) / 2 * G::SUMS + (((8 * ((wc * CT + j) & 1) + 2 * a4 + hh) ^ (ln & 15)) << 4)) =
          make_float4(acc[j][a4 * 4], acc[j][a4 * 4 + 1], acc[j][a4 * 4 + 2], acc[j][a4 * 4 + 3]);
  lds_barrier();
}

// four columns 4 c .. of row r of the tile, summed over the k parts
template <typename G>
__device__ __forceinline__ float4 tile_sum(const unsigned char* lds, int r, int c) {
  const unsigned char* p = lds + r * TL_SUM + ((c ^ (r & 15)) << 4);
  float4 v = *(const float4*)p;
#pragma unroll
  for (int k = 1; k < G::KH; ++k) {
    const float4 o = *(const float4*)(p + k * G::BM * TL_SUM);
    v.x += o.x; v.y += o.y; v.z += o.z; v.w += o.w;
  }
  return v;
}

// Workgroup id -> (column tile, row tile): ids equal mod 8 share an XCD and its L2; the row tiles of a
// column tile are neighbours there, so the panel of w enters one L2 once.
__device__ inline bool tile_coords(int id, int ct, int mt, int& col, int& row) {
  const int xcd = id & 7, s = id >> 3;
  col = (s / mt) * 8 + xcd;
  row = s % mt;
  return col < ct;
}

// What a row tile of WM * 32 rows does: the last one of `mt` where few rows are left takes a smaller one, in whose blocks x
// is less (525 rows: 13 of them are left to a fifth tile of 128).  Up to 32 rows from `least` tiles on: of two, the smaller one, whose
// waves split every block, is the last to end ([q/k/v | gate/up] of width 4096, 129 rows 90 us, 192 rows without it 78).  33 .. 64 rows
// from five tiles on; with fragments a block ahead it takes as long as a whole one there (us, [q/k/v | gate/up] of MVPFormer-S, as a tile of
// 128 / of 64: 560 rows 9.7 / 9.7, 832 14.1 / 13.9; the base model 832 70.7 / 74.3, 704 59.4 / 59.0; tail products 1 % either way).
template <int WM, int STAGES, typename F>
__device__ __forceinline__ void for_rows_left(int64_t rows, int mt, int least, F f) {
  if constexpr (WM == 4 && STAGES == 3) {
    if (rows <= 32 && mt >= least) f(std::integral_constant<int, 1>(), std::integral_constant<int, 6>());
    else if (rows <= 64 && mt > 4) f(std::integral_constant<int, 2>(), std::integral_constant<int, 4>());
    else f(std::integral_constant<int, 4>(), std::integral_constant<int, 3>());
    static_assert(tile_cfg<1, 6>::LDS <= tile_cfg<4, 3>::LDS && tile_cfg<2, 4>::LDS <= tile_cfg<4, 3>::LDS, "LDS of the launch");
  } else {
    f(std::integral_constant<int, WM>(), std::integral_constant<int, STAGES>());
  }
}

template <int WM, int STAGES, int BN>
__device__ __forceinline__ void tile_dual(unsigned char* tl_lds, const bf16_t* __restrict__ X, int64_t M, int K, int64_t ldx,
                                          const bf16_t* __restrict__ W0, int N0, int64_t ldw0, const tile_out& out,
                                          const tile_gated& gt, const tile_norm& nrm, int gated_ct, int col, int64_t m0) {
  using G = tile_cfg<WM, STAGES, 2, BN>;
  constexpr int PER = BN / TL_BN;                   // 256 threads finish 64 columns
  const int tid = threadIdx.x & 255, part = PER > 1 ? __builtin_amdgcn_readfirstlane(threadIdx.x >> 8) : 0;
  const bool gated = col < gated_ct;
  const int first = gated ? col * PER * 32 : (col - gated_ct) * BN, N = gated ? gt.N : N0;
  const int n0 = first + part * (gated ? 32 : TL_BN);
  // sums of squares of the rows this thread will finish: requested in front of the product, used behind it
  constexpr int ROWS = G::BM / 32;                  // every 64th row of the gated product, every 32nd of the plain one
  const int r0 = gated ? tid >> 2 : tid >> 3, dr = gated ? 64 : 32;
  float ss[ROWS];
#pragma unroll
  for (int i = 0; i < ROWS; ++i) ss[i] = nrm.ss ? nrm.ss[min(m0 + r0 + i * dr, M - 1) * nrm.parts] : 0.f;
  if (gated)
    tile_product<WM, STAGES, 2, BN>(tl_lds, X, ldx, m0, M, gt.w, gt.ldw, [&](int r) {
      return (int64_t)((r >> 5 & 1) * N + min(first + (r >> 6) * 32 + (r & 31), N - 1)); }, 0, K / TL_BK);
  else
    tile_product<WM, STAGES, 2, BN>(tl_lds, X, ldx, m0, M, W0, ldw0, [&](int r) { return (int64_t)min(first + r, N0 - 1); }, 0, K / TL_BK);
  tl_lds += part * G::SUMS;
#pragma unroll
  for (int i = 0; i < ROWS; ++i) asm volatile("" : "+v"(ss[i]));       // not before the product
  auto factor = [&](int i, int64_t m) {
    if (!nrm.ss) return 1.f;
    float s = ss[i];
    for (int p = 1; p < nrm.parts; ++p) s += nrm.ss[m * nrm.parts + p];
    return rsqrtf(s / (float)K + nrm.eps);
  };
  if (gated) {                                      // 8 outputs of a row per thread
    const int c = tid & 3, n = n0 + c * 8;
#pragma unroll
    for (int i = 0; i < (G::BM + 63) / 64; ++i) {
      const int r = r0 + i * 64;
      const int64_t m = m0 + r;
      if (r >= G::BM || m >= M || n >= N) continue;
      const float rn = factor(i, m);
      bf16x8 o;
#pragma unroll
      for (int q = 0; q < 2; ++q) {
        const float4 g4 = tile_sum<G>(tl_lds, r, 2 * c + q), u4 = tile_sum<G>(tl_lds, r, 8 + 2 * c + q);
        const float g[4] = {g4.x, g4.y, g4.z, g4.w}, u[4] = {u4.x, u4.y, u4.z, u4.w};
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const float x = g[e] * rn;
          o[4 * q + e] = (__bf16)(x / (1.f + __expf(-x)) * (u[e] * rn));
        }
      }
      *(bf16x8*)(gt.y + m * gt.ldy + n) = o;
    }
    return;
  }
  const int slot = out.k ? (out.head ? *out.head : out.slot) : 0, c = tid & 7, n = n0 + c * 8;
#pragma unroll
  for (int i = 0; i < ROWS; ++i) {
    const int r = r0 + i * 32;
    const int64_t m = m0 + r;
    if (m >= M || n >= N0) continue;
    bf16_t* dst;
    if (n < out.n_y) {
      dst = out.y + m * out.ldy + n;
    } else {
      const int o = n - out.n_y, is_v = o >= out.n_kv, e = is_v ? o - out.n_kv : o;
      const int g = e / out.Dh, d = e - g * out.Dh;
      const int b = (int)m / out.C, ch = (int)m - b * out.C;
      dst = (is_v ? out.v : out.k) + b * out.stride_b + g * out.stride_g + ((int64_t)slot * out.C + ch) * out.Dh + d;
    }
    const float rn = factor(i, m);
    const float4 lo = tile_sum<G>(tl_lds, r, 2 * c), hi = tile_sum<G>(tl_lds, r, 2 * c + 1);
    *(bf16x8*)dst = bf16x8{(__bf16)(lo.x * rn), (__bf16)(lo.y * rn), (__bf16)(lo.z * rn), (__bf16)(lo.w * rn),
                           (__bf16)(hi.x * rn), (__bf16)(hi.y * rn), (__bf16)(hi.z * rn), (__bf16)(hi.w * rn)};
  }
}

template <int WM, int STAGES, int BN>
__global__ __launch_bounds__(BN * 4) void tile_dual_kernel(const bf16_t* __restrict__ X, int64_t M, int K, int64_t ldx,
                                                        const bf16_t* __restrict__ W0, int N0, int64_t ldw0,
                                                        tile_out out, tile_gated gt, tile_norm nrm, int gated_ct,
                                                        int ct, int mt) {
  extern __shared__ __attribute__((aligned(1024))) unsigned char tl_lds[];
  int col, row;
  if (!tile_coords(blockIdx.x, ct, mt, col, row)) return;
  const int64_t m0 = (int64_t)row * 32 * WM;
  for_rows_left<WM, STAGES>(M - m0, mt, 3, [&](auto wm, auto stages) {
    tile_dual<wm(), stages(), BN>(tl_lds, X, M, K, ldx, W0, N0, ldw0, out, gt, nrm, gated_ct, col, m0);
  });
}

template <int WM, int STAGES, int BN>
__global__ __launch_bounds__(BN * 4) void tile_partial_kernel(const bf16_t* __restrict__ X, int64_t M, int K, int64_t ldx,
                                                           const bf16_t* __restrict__ W, int N, int64_t ldw,
                                                           float* __restrict__ P, tile_split sp, int ct, int mt, bool spread) {
  extern __shared__ __attribute__((aligned(1024))) unsigned char tl_lds[];
  // an XCD (ids equal mod 8) takes neighbours of one part, row tiles fastest: it reads that part's columns of x, not
  // all of them, and its panel of w once.  spread: parts of a column side by side, dealt over the XCDs
  const int splits = sp.a + sp.b, total = ct * splits * mt, per = (total + 7) / 8;
  int row, z, col;
  if (spread) {
    int cz;
    if (!tile_coords(blockIdx.x, ct * splits, mt, cz, row)) return;
    col = cz / splits;
    z = cz - col * splits;
  } else {
    const int id = (blockIdx.x & 7) * per + (blockIdx.x >> 3), cz = id / mt;
    if (id >= total) return;
    row = id - cz * mt;
    z = cz / ct;
    col = cz - z * ct;
  }
  const int kb0 = z < sp.a ? z * sp.per_a : sp.nkb_a + (z - sp.a) * sp.per_b;
  const int kb1 = z < sp.a ? min(kb0 + sp.per_a, sp.nkb_a) : min(kb0 + sp.per_b, K / TL_BK);
  const int64_t m0 = (int64_t)row * 32 * WM;
  // 256 threads finish 64 columns
  const int n0 = col * BN, part = BN > TL_BN ? __builtin_amdgcn_readfirstlane(threadIdx.x >> 8) : 0, c = threadIdx.x & 15;
  const int n = n0 + part * TL_BN + c * 4;
  for_rows_left<WM, STAGES>(M - m0, mt, 2, [&](auto wm, auto stages) {
    using G = tile_cfg<wm(), stages(), 2, BN>;
    tile_product<wm(), stages(), 2, BN>(tl_lds, X, ldx, m0, M, W, ldw, [&](int r) { return (int64_t)min(n0 + r, N - 1); }, kb0, kb1);
#pragma unroll
    for (int r = (threadIdx.x & 255) >> 4; r < G::BM; r += 16)
      if (m0 + r < M && n < N) *(float4*)(P + ((int64_t)z * M + m0 + r) * N + n) = tile_sum<G>(tl_lds + part * G::SUMS, r, c);
  });
}

// A product by itself: every output's sum is one chain over K, as in the large tiles (and the same bits)
template <int WM, int STAGES, int CT>
__global__ __launch_bounds__(256) void tile_linear_kernel(const bf16_t* __restrict__ X, int64_t M, int K, int64_t ldx,
                                                          const bf16_t* __restrict__ W, int N, int64_t ldw, bf16_t* __restrict__ Y,
                                                          int64_t ldy, int ct, int mt) {
  using G = tile_cfg<WM, STAGES, CT>;
  static_assert(G::KH == 1, "one chain");
  extern __shared__ __attribute__((aligned(1024))) unsigned char tl_lds[];
  // An eighth of the tiles to an XCD, row tiles fastest.  (A column of tiles to an XCD left seven of them idle where there is one:
  // [8,768] 9999 rows 15.8 -> 5.2 us, [64,4096] 16384 108 -> 22, and [768,2624] 1152 14.8 -> 11.4.)
  const int total = ct * mt, per = (total + 7) / 8, id = (blockIdx.x & 7) * per + (blockIdx.x >> 3), col = id / mt;
  if (id >= total) return;
  const int64_t m0 = (int64_t)(id - col * mt) * G::BM;
  const int n0 = col * TL_BN, c = threadIdx.x & 7, n = n0 + c * 8;
  tile_product<WM, STAGES, CT>(tl_lds, X, ldx, m0, M, W, ldw, [&](int r) { return (int64_t)min(n0 + r, N - 1); }, 0, K / TL_BK);
#pragma unroll
  for (int i = 0; i < G::BM / 32; ++i) {
    const int r = (threadIdx.x >> 3) + i * 32;
    if (m0 + r >= M || n >= N) continue;
    const float4 lo = tile_sum<G>(tl_lds, r, 2 * c), hi = tile_sum<G>(tl_lds, r, 2 * c + 1);
    *(bf16x8*)(Y + (m0 + r) * ldy + n) = bf16x8{(__bf16)lo.x, (__bf16)lo.y, (__bf16)lo.z, (__bf16)lo.w,
                                                (__bf16)hi.x, (__bf16)hi.y, (__bf16)hi.z, (__bf16)hi.w};
  }
}

// One workgroup per row, a wave per 512 columns: the partial sums of a split-K tail product, the residual, one rounding, and
// the RMSNorm that the next product wants, while the row is in registers (8 columns per lane and chunk).
// Bound by the trip to the sums, which other XCDs have just written, and with hundreds of rows by what is requested: all parts, the
// residual and the norm's weight are requested together, and nothing beside them.  TWO: the first split_a parts are a product
// of their own.  us, one part after the other and the weight behind the sums of squares / everything together for the next of 4, 6,
// 8, 9 parts in four waves a row / now: 64 rows of 768, 9 parts 3.6 / 3.6 / 3.2; 525, 4 parts 3.3 / 3.9 / 3.3; 1200, 2 parts 3.6 / 5.0 / 3.7; 128
// rows of 2048, 8 parts 3.65 / 3.6 / 3.6; 768 rows of 3072, 1 part 4.9 / 6.7 / 5.1.
template <int CHUNKS, int PARTS, bool TWO>
__global__ __launch_bounds__(256) void tail_reduce_kernel(const float* __restrict__ P, int split_a, const bf16_t* __restrict__ R,
                                                          bf16_t* __restrict__ S, bf16_t* __restrict__ Y, const float* __restrict__ w,
                                                          float eps, float* __restrict__ ss_out, int64_t M, int N) {
  __shared__ float red[4];
  const int64_t m = blockIdx.x;
  const int wave0 = __builtin_amdgcn_readfirstlane(threadIdx.x & ~63) * 8;
  float v[CHUNKS][8], ss = 0.f;
  f32x4 p[CHUNKS][PARTS][2], wr[CHUNKS][2];
  u32x4 rr[CHUNKS];
#pragma unroll
  for (int c = 0; c < CHUNKS; ++c) {                // lanes past the row: its last columns, for nobody
    if (c > 0 && wave0 + c * 2048 >= N) continue;   // (a whole wave: nothing)
    const int n = min((c * 256 + (int)threadIdx.x) * 8, N - 8);
    rr[c] = *(const u32x4*)(R + m * N + n);
#pragma unroll
    for (int z = 0; z < PARTS; ++z) {
      const float* at = P + ((int64_t)z * M + m) * N + n;
      p[c][z][0] = *(const f32x4*)at;
      p[c][z][1] = *(const f32x4*)(at + 4);
    }
    const float* at = (Y ? w : P) + n;              // without a norm: anything
    wr[c][0] = *(const f32x4*)at;
    wr[c][1] = *(const f32x4*)(at + 4);
  }
  __builtin_amdgcn_sched_barrier(0);                // every request first
  // without branches, behind which the loads would be put and waited for one by one
#pragma unroll
  for (int c = 0; c < CHUNKS; ++c) {
    if (c > 0 && wave0 + c * 2048 >= N) continue;
    const int n = (c * 256 + threadIdx.x) * 8;
    float a[8] = {}, b[8] = {};
#pragma unroll
    for (int z = 0; z < PARTS; ++z)
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const float x = p[c][z][i >> 2][i & 3];
        if (TWO) a[i] += z < split_a ? x : 0.f;
        b[i] += !TWO || z >= split_a ? x : 0.f;
      }
    bf16x8 o;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      v[c][i] = __uint_as_float(i & 1 ? rr[c][i >> 1] & 0xffff0000u : rr[c][i >> 1] << 16);
      v[c][i] += (float)(__bf16)b[i];
      if (TWO) v[c][i] += (float)(__bf16)a[i];
      o[i] = (__bf16)v[c][i];
      v[c][i] = (float)o[i];
      ss += n < N ? v[c][i] * v[c][i] : 0.f;
    }
    if (n < N) *(bf16x8*)(S + m * N + n) = o;
  }
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) ss += __shfl_xor(ss, off);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = ss;
  __syncthreads();
  float tot = red[0];
  for (int k = 1; k < (int)blockDim.x / 64; ++k) tot += red[k];
  if (ss_out && threadIdx.x == 0) ss_out[m] = tot;
  if (!Y) return;
  const float inv = rsqrtf(tot / (float)N + eps);
#pragma unroll
  for (int c = 0; c < CHUNKS; ++c) {
    const int n = (c * 256 + threadIdx.x) * 8;
    if (n < N) {
      bf16x8 o;
#pragma unroll
      for (int i = 0; i < 8; ++i) o[i] = (__bf16)(v[c][i] * inv * wr[c][i >> 2][i & 3]);
      *(bf16x8*)(Y + m * N + n) = o;
    }
  }
}

template <int CHUNKS, int PARTS = 9>                // at most 9 parts: make_tile_split
static auto tail_reduce_for(const tile_split& split) {
  if constexpr (PARTS > 1)
    if (split.total() < PARTS) return tail_reduce_for<CHUNKS, PARTS - 1>(split);
  return split.a ? tail_reduce_kernel<CHUNKS, PARTS, true> : tail_reduce_kernel<CHUNKS, PARTS, false>;
}

template <int WM, int STAGES, int BN = TL_BN>
static int launch_dual_t(const bf16_t* x, int64_t M, int64_t K, int64_t ldx, const bf16_t* w0, int64_t N0, int64_t ldw0,
                         const tile_out& out, const tile_gated& gated, const tile_norm& norm, hipStream_t s) {
  using G = tile_cfg<WM, STAGES, 2, BN>;
  auto kern = tile_dual_kernel<WM, STAGES, BN>;
  want_dynamic_lds((const void*)kern, G::LDS);
  const int gct = gated.w ? (gated.N + BN / 2 - 1) / (BN / 2) : 0;
  const int ct = gct + (w0 ? (int)((N0 + BN - 1) / BN) : 0), mt = (int)((M + G::BM - 1) / G::BM);
  MVPA_LAUNCH(kern, dim3((unsigned)((ct + 7) / 8 * 8 * mt)), dim3(G::NW * 64), G::LDS, s, x, M, (int)K, ldx, w0, (int)N0, ldw0,
              out, gated, norm, gct, ct, mt);
  return take_launch_status();
}

// The smallest tile that gives at most one workgroup a CU: what a product of few rows takes is its chain of blocks, and a
// block of 32 rows of x is 12 KB, of 64 16, of 128 24.  With more workgroups than CUs the panels of w are read again instead.
// [q/k/v | gate/up] of MVPFormer-S (74 columns of tiles), tiles of 32 / 64 / 128 rows, us: 32 rows 4.8 / 5.1 / 7.0, 64 4.8 /
// 5.4 / 7.1, 100 6.1 / 5.4 / 7.9, 192 6.7 / 5.5 / 7.8, 256 8.7 / 7.7 / 7.6, 400 11.8 / 10.0 / 9.3; of the base model (240): 32
// 15.0 / 14.8 / 16.2, 64 20.9 / 17.9 / 17.8, 100 26.6 / 22.7 / 19.2, 128 29.8 / 24.4 / 20.8.  Never more rows than there are: the
// workgroups would be as many (width 3072, 336 columns of tiles, 21 rows 24 / . / 31, 64 rows . / 27 / 32).
static int tile_rows(int64_t M, int64_t per_row_tile) {
  if (M <= 32 || (M + 31) / 32 * per_row_tile <= 256) return 32;
  return M <= 64 || (M + 63) / 64 * per_row_tile <= 256 ? 64 : 128;
}

int launch_tile_dual(const bf16_t* x, int64_t M, int64_t K, int64_t ldx, const bf16_t* w0, int64_t N0, int64_t ldw0,
                     const tile_out& out, const tile_gated& gated, const tile_norm& norm, hipStream_t s) {
  const int rows = tile_rows(M, (gated.w ? (gated.N + 31) / 32 : 0) + (w0 ? (N0 + TL_BN - 1) / TL_BN : 0));
  if (rows == 32) return launch_dual_t<1, 6>(x, M, K, ldx, w0, N0, ldw0, out, gated, norm, s);
  if (rows == 64) return launch_dual_t<2, 5>(x, M, K, ldx, w0, N0, ldw0, out, gated, norm, s);
  if (M <= 128) return launch_dual_t<4, 6>(x, M, K, ldx, w0, N0, ldw0, out, gated, norm, s);
  // Where a CU would hold two tiles of 128 x 64, which read the same x twice and share its LDS unevenly with CUs that hold one: one of
  // 128 x 128 on eight waves instead, as long as they are one a CU.  us, 64 / 128 columns: base model, 129 rows 24.4 / 20.4, 192 22.1 / 20.3, 256
  // 23.5 / 21.5; MVPFormer-S 385 9.8 / 9.6, 525 10.0 / 9.8, 768 10.9 / 10.5; one of 64 columns a CU: S 300 7.3 / 9.4.  Chains of a few
  // blocks keep the narrow ones (256 columns, 1200 rows 6.7 / 6.9).  More than one a CU: long chains whose last round is more than half
  // full, or of many rounds (base 300 rows, 1.4 rounds, 31.4 / 34.7, 512, 1.9, 41.8 / 39.7; width 4096 129, 1.7, 90 / 66, 640, 4.3, 184 / 174; S
  // 800, 1.0, 14.1 / 17.4, 1600, 1.9, 21.4 / 26.7).
  const int64_t cols = (gated.w ? (gated.N + 31) / 32 : 0) + (w0 ? (N0 + TL_BN - 1) / TL_BN : 0);
  const int64_t mt = (M + 127) / 128, wide = mt * ((gated.w ? (gated.N + 63) / 64 : 0) + (w0 ? (N0 + 127) / 128 : 0));
  if (mt * cols > 256 && K >= 8 * TL_BK && (wide <= 256 || (K >= 24 * TL_BK && ((wide - 1) % 256 >= 128 || wide > 5 * 256))))
    return launch_dual_t<4, 4, 128>(x, M, K, ldx, w0, N0, ldw0, out, gated, norm, s);
  return launch_dual_t<4, 3>(x, M, K, ldx, w0, N0, ldw0, out, gated, norm, s);
}

template <int WM, int STAGES, int CT>
static int launch_linear_t(const bf16_t* x, int64_t M, int64_t K, int64_t ldx, const bf16_t* w, int64_t N, int64_t ldw, bf16_t* y,
                           int64_t ldy, hipStream_t s) {
  using G = tile_cfg<WM, STAGES, CT>;
  auto kern = tile_linear_kernel<WM, STAGES, CT>;
  want_dynamic_lds((const void*)kern, G::LDS);
  const int ct = (int)((N + TL_BN - 1) / TL_BN), mt = (int)((M + G::BM - 1) / G::BM);
  MVPA_LAUNCH(kern, dim3((unsigned)((ct * mt + 7) / 8 * 8)), dim3(256), G::LDS, s, x, M, (int)K, ldx, w, (int)N, ldw, y, ldy, ct, mt);
  return take_launch_status();
}

// Where large tiles leave most CUs without work: up to one of these a CU, and below 512 rows, where large ones are not used, up to 288.
// us, large tiles (below 512 rows the 128 x 128 ones without a ring, from there the ones of pair_tile_rows) / these: [768,768] 129 rows 20.4 /
// 5.1, 525 8.0 / 7.2, 1600 8.1 / 7.2, 2500 8.2 / 8.4, 3000 (288 tiles) 8.2 / 11.1; [768,2624] 525 17.9 / 9.7, 2500 18.5 / 18.3, 3000 18.6 / 28;
// [2048,2048] 129 40.7 / 8.3, 800 15.7 / 12.1, 1152 (288) 17.1 / 19.0; [1280,768] 1600 (260) 8.5 / 9.7; [256,8192] 6000 (188) 70 / 61; [64,4096] 6000
// 26.5 / 13.5: of 64 columns and fewer they stay, half of a large tile would be empty.  Up to 128 rows keep the kernels of a
// step, whose sums are in another order, and not for their speed: [768,576] 64 rows 7.7 / 4.1, [768,2624] 11.8 / 9.2, [2048,2048] 128 14.4 /
// 7.9, 1 8.9 / 7.6; [1024,4096] 32 12.9 / 12.9, 1 11.1 / 12.7.
bool tile_linear_pays(int64_t M, int64_t N, int64_t K, int64_t ldx, int64_t ldw, int64_t ldy, const void* y) {
  const int64_t ct = (N + TL_BN - 1) / TL_BN, most = M >= 512 && N > TL_BN && K >= 128 ? 256 : 288;
  return M > 128 && K % TL_BK == 0 && N % 8 == 0 && ldy % 8 == 0 && ((uintptr_t)y & 15) == 0 && M < (1 << 20) && N < (1 << 20) &&
         K < (1 << 30) && 128 * ldx < (1 << 30) && N * ldw < ((int64_t)1 << 31) && (M + 127) / 128 * ct <= most;
}

int launch_tile_linear(const bf16_t* x, int64_t M, int64_t K, int64_t ldx, const bf16_t* w, int64_t N, int64_t ldw, bf16_t* y,
                       int64_t ldy, hipStream_t s) {
  if ((M + 63) / 64 * ((N + TL_BN - 1) / TL_BN) <= 256) return launch_linear_t<2, 5, 1>(x, M, K, ldx, w, N, ldw, y, ldy, s);
  return launch_linear_t<4, 3, 2>(x, M, K, ldx, w, N, ldw, y, ldy, s);
}

// Partial sums per output element: enough workgroups for every CU, about 4 k-blocks each or more, at most
// 8 or 9 (every one of them is 4 bytes written and read again per output element).  Never a little more than one
// workgroup a CU: a CU takes blocks at a fixed rate, and the 288 workgroups of the base model's 3 + 6 parts took as
// long as 512 (128 rows: 19.5 us, in 2 + 6 parts 14.5; 64 rows 14.4 and 10.1).
tile_split make_tile_split(int64_t M, int64_t N, int64_t K, int64_t Ka) {
  const int64_t wgs = ((N + TL_BN - 1) / TL_BN) * ((M + 127) / 128), nkb = K / TL_BK, na = Ka / TL_BK, nb = nkb - na;
  int64_t z = (256 + wgs / 2) / wgs;
  if (z > nkb / 4) z = nkb / 4;
  if (z > 8) z = 8;
  if (z < 1) z = 1;
  auto parts_of = [](int64_t n, int64_t per) { return (n + per - 1) / per; };
  int64_t per = parts_of(nkb, z);                   // blocks of the longest part
  while ((parts_of(na, per) + parts_of(nb, per)) * wgs > 256 && z > 2 && z * wgs <= 256 && per < nkb) ++per;
  tile_split sp;
  sp.nkb_a = (int32_t)na;
  sp.a = (int32_t)parts_of(na, per);
  sp.per_a = sp.a ? (int32_t)parts_of(na, sp.a) : 0;
  sp.b = (int32_t)parts_of(nb, per);
  sp.per_b = sp.b ? (int32_t)parts_of(nb, sp.b) : 0;
  if (sp.a) sp.a = (int32_t)parts_of(na, sp.per_a);
  if (sp.b) sp.b = (int32_t)parts_of(nb, sp.per_b);
  return sp;
}

template <int WM, int STAGES, int BN = TL_BN>
static int launch_partial_t(const bf16_t* x, int64_t M, int64_t K, int64_t ldx, const bf16_t* w, int64_t N, int64_t ldw,
                            float* P, const tile_split& sp, hipStream_t s) {
  using G = tile_cfg<WM, STAGES, 2, BN>;
  auto kern = tile_partial_kernel<WM, STAGES, BN>;
  want_dynamic_lds((const void*)kern, G::LDS);
  const int ct = (int)((N + BN - 1) / BN), mt = (int)((M + G::BM - 1) / G::BM);
  // A part's columns of x to an XCD, but for four row tiles of an x that the L2 of each (4 MB) holds as a whole.  Windows of
  // MVPFormer-S (2496 columns), part to an XCD / spread, us: 384 rows (three tiles) 343 / 351, 392 368 / 366, 416 370 / 369, 448 373 / 370, 480
  // 377 / 372, 512 375 / 367; four blocks of the base model (7680), 448 rows 412 / 411.
  const bool spread = mt == 4 && M * K * 2 <= (4 << 20);
  const int ids = spread ? (ct * sp.total() + 7) / 8 * 8 * mt : (ct * sp.total() * mt + 7) / 8 * 8;
  MVPA_LAUNCH(kern, dim3((unsigned)ids), dim3(G::NW * 64), G::LDS, s, x, M, (int)K, ldx, w, (int)N, ldw, P, sp, ct, mt, spread);
  return take_launch_status();
}

int launch_tile_partial(const bf16_t* x, int64_t M, int64_t K, int64_t ldx, const bf16_t* w, int64_t N, int64_t ldw,
                        float* P, const tile_split& splits, hipStream_t s) {
  // As above, but that tiles of 32 rows are for 32 rows alone: the chains are a part's few blocks.  Tail of MVPFormer-S (12
  // columns of tiles in up to 9 parts), tiles of 32 / 64 / 128 rows, us: 64 rows 4.3 / 4.3 / 5.3, 128 5.2 / 4.4 / 6.1, 192 7.2 / 5.8 /
  // 5.7; of the base model (32 in 8): 64 12.9 / 10.4 / 10.5, 100 16.7 / 13.0 / 11.8, 128 18.3 / 14.2 / 12.8.
  if (M <= 32) return launch_partial_t<1, 6>(x, M, K, ldx, w, N, ldw, P, splits, s);
  if (tile_rows(M, (N + TL_BN - 1) / TL_BN * splits.total()) <= 64) return launch_partial_t<2, 5>(x, M, K, ldx, w, N, ldw, P, splits, s);
  if (M <= 128) return launch_partial_t<4, 6>(x, M, K, ldx, w, N, ldw, P, splits, s);
  // As in launch_tile_dual.  us, 64 / 128 columns: base model, 300 rows in 3 parts 24.6 / 21.4, 525 in 2 35.1 / 29.5, 1200 76.7 / 54.7; width 3072,
  // 192 in 3 33.1 / 28.2, 768 99.6 / 71.8 (64 columns, fragments read where their products stand: 23.8, 32.8, 65.2, 30.5, 84.5);
  // MVPFormer-S, 641 in 4 9.0 / 8.5, but one a CU: 600 6.8 / 8.4, 1024 rows of the base model 42.7 / 51.9.
  const int64_t row_tiles = (M + 127) / 128 * splits.total();
  if (row_tiles * ((N + TL_BN - 1) / TL_BN) > 256 && row_tiles * ((N + 127) / 128) <= 256 && splits.per_b >= 8)
    return launch_partial_t<4, 4, 128>(x, M, K, ldx, w, N, ldw, P, splits, s);
  return launch_partial_t<4, 3>(x, M, K, ldx, w, N, ldw, P, splits, s);
}

int launch_tail_reduce(const float* P, const tile_split& split, const bf16_t* r, bf16_t* sum, bf16_t* norm, const float* w,
                       float eps, float* ss, int64_t M, int64_t N, hipStream_t s) {
  auto kern = N <= 2048 ? tail_reduce_for<1>(split) : tail_reduce_for<2>(split);
  const unsigned waves = N <= 2048 ? (unsigned)(N + 511) / 512 : 4;
  MVPA_LAUNCH(kern, dim3((unsigned)M), dim3(waves * 64), 0, s, P, split.a, r, sum, norm, w, eps, ss, M, (int)N);
  return take_launch_status();
}

}  // namespace mvpa
