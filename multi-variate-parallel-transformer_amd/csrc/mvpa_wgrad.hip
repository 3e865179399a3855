// Weight gradients: dW[N,K] = dY[M,N]^T X[M,K] in bf16 with fp32 sums (the backward of layers/mvpa.py:354-359, 400
// and of the MLP's projections, models/mvpformer.py:146).
//
// The output is small and the contraction long (MVPFormer-S, 6400 rows: 36 .. 162 tiles of 128 x 128 over 200
// blocks of 32 rows), so the tiles alone do not fill 256 CUs: the rows are dealt over `splits` workgroups per
// tile, fp32 partial tiles meet in a second kernel, or over two groups of waves of a workgroup that meet in LDS.  Both operands are contracted over their slow index: they go
// straight from memory to LDS as they lie, [32 rows][128 columns], and both MFMA operands come out of transposing
// LDS reads.  A group is 4 waves of 64 x 64 outputs (64 accumulator registers) on five 16 KiB stages of 32 rows, so
// that two share a CU and four blocks of each are on their way.  Per block one barrier, in front of its last half: that half's
// fragments are in registers, the barrier publishes the next block and frees this one's stage for the block five further on.
// Bound by the fragment reads (one per product).  With two stages of 64 rows, one block on its way, and an address formed by
// every lane for every request, both launches / now, us: [3456,768] over 6400 rows 56.1 / 53.5, 25600 175 / 165; [768,2624] 52.1 /
// 45.7, 161 / 129; [768,768] 21.9 / 21.8, 60 / 49.
#include "mvpa_mfma_tools.h"

namespace mvpa {
namespace wgrad {

constexpr int TILE = 128, KB = 32;               // outputs of a tile each way, rows of a block
constexpr int ROWB = TILE * 2, STAGE = 2 * KB * ROWB, STAGES = 5;
constexpr int LOADS = STAGE / 1024 / 4;          // 1 KiB requests per wave and block

struct args {
  const bf16_t *dy, *x;
  void* out;                                     // dW, or the partial tiles [splits][N][K]
  int64_t ldy, ldx, ldo;
  int32_t M, N, K, tiles_k, splits, blocks;      // blocks of rows in all
};

// fragment of a [32][128] tile contracted over its rows: column 32 c + lane's, rows 16 s + 8 rd + 4 hh + e
__device__ inline bf16x8 frag(const unsigned char* p, int s) {
  const bf16x4 lo = el_bf16::read_tr(p + 16 * s * ROWB), hi = el_bf16::read_tr(p + (16 * s + 8) * ROWB);
  return __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
}

template <int GROUPS, bool PARTIAL, bool FAR = false>
__global__ __launch_bounds__(256 * GROUPS, 2) void linear_wgrad_kernel(args a) {
  extern __shared__ __attribute__((aligned(1024))) unsigned char all_stages[];
  const int tid = threadIdx.x, lane = tid & 63, ln = lane & 31, hh = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6) & 3, group = __builtin_amdgcn_readfirstlane(tid >> 8);
  unsigned char* const smem = all_stages + group * STAGES * STAGE;
  // ids equal mod 8 run on one XCD: it gets neighbouring tiles of one share of the rows, which read the same
  // rows at about the same time
  const int total = gridDim.x, per = total / 8, more = total % 8, xcd = blockIdx.x & 7;
  const int id = xcd * per + min(xcd, more) + (int)(blockIdx.x >> 3);
  const int tiles = total / a.splits, split = id / tiles, tile = id % tiles;
  const int n0 = tile / a.tiles_k * TILE, k0 = tile % a.tiles_k * TILE;
  const int first = (int)((int64_t)a.blocks * split / a.splits), last = (int)((int64_t)a.blocks * (split + 1) / a.splits);
  const int count = (last - first + GROUPS - 1) / GROUPS;       // blocks of a group: first + group, + GROUPS ..
  const int64_t m_end = min((int64_t)last * KB, (int64_t)a.M);
  auto row_of = [&](int kb) { return (int64_t)(first + group + kb * GROUPS) * KB; };

  // requests of a wave: rows 4 wave + 16 i .. of dY and of X; lane: row lane / 16, chunk lane % 16
  const int row_l = lane >> 4, chunk = ((lane & 15) ^ swz_v<TILE>(row_l)) * 8;
  // columns past the end: any, their outputs are not stored
  const uint32_t col_y = (uint32_t)min(n0 + chunk, a.N - 8), col_x = (uint32_t)min(k0 + chunk, a.K - 8);
  const uint32_t off_y = (uint32_t)(row_l * (int)a.ldy + col_y) * 2, off_x = (uint32_t)(row_l * (int)a.ldx + col_x) * 2;
  const uint32_t lds0 = (uint32_t)(uintptr_t)(LDS_PTR(unsigned char))smem;
  // rows of a block that is whole: a uniform base and the lane's own offset, which does not change (addresses formed per
  // lane cost as many vector cycles as the products)
  auto request = [&](int kb, int stage) {
    const int64_t m0 = row_of(kb) + 4 * wave;
    const uint32_t dst = lds0 + stage * STAGE + 4 * wave * ROWB;
    if (!FAR && row_of(kb) + KB <= m_end) {
      const bf16_t *y = a.dy + m0 * a.ldy, *x = a.x + m0 * a.ldx;
#pragma unroll
      for (int i = 0; i < LOADS / 2; ++i) {
        load_to_lds_16(y + (int64_t)(16 * i) * a.ldy, off_y, dst + 16 * i * ROWB);
        load_to_lds_16(x + (int64_t)(16 * i) * a.ldx, off_x, dst + STAGE / 2 + 16 * i * ROWB);
      }
    } else if (FAR) {                            // rows farther apart than 32 bits of a block's bytes
#pragma unroll
      for (int i = 0; i < LOADS / 2; ++i) {
        const int64_t m = min(m0 + 16 * i + row_l, m_end - 1);
        load_to_lds_16(a.dy + m * a.ldy + col_y, dst + 16 * i * ROWB);
        load_to_lds_16(a.x + m * a.ldx + col_x, dst + STAGE / 2 + 16 * i * ROWB);
      }
    } else {                                     // the last row again where there are no more
      const int64_t m1 = min(m0, m_end - 1);
      const bf16_t *y = a.dy + m1 * a.ldy, *x = a.x + m1 * a.ldx;
#pragma unroll
      for (int i = 0; i < LOADS / 2; ++i) {
        const int r = (int)(min(m0 + 16 * i + row_l, m_end - 1) - m1);
        load_to_lds_16(y, (uint32_t)(r * (int)a.ldy + col_y) * 2, dst + 16 * i * ROWB);
        load_to_lds_16(x, (uint32_t)(r * (int)a.ldx + col_x) * 2, dst + STAGE / 2 + 16 * i * ROWB);
      }
    }
  };
  // a block that reaches past the last row: zeros there, in what this wave has requested itself
  auto cut = [&](int kb, int stage) {
    if (row_of(kb) + KB <= m_end) return;
#pragma unroll
    for (int i = 0; i < LOADS; ++i) {
      const int r = 4 * wave + 16 * (i % (LOADS / 2)) + row_l;
      if (row_of(kb) + r >= m_end)
        *(u32x4*)(smem + stage * STAGE + (i < LOADS / 2 ? 0 : STAGE / 2) + r * ROWB + (lane & 15) * 16) = u32x4{0u, 0u, 0u, 0u};
    }
  };

  const int wn = wave >> 1, wk = wave & 1, row0 = 4 * hh + ((ln & 15) >> 2);
  const unsigned char *pa[2], *pb[2];
#pragma unroll
  for (int c = 0; c < 2; ++c) {
    const int sub = 2 * (ln >> 4) + ((ln & 3) >> 1), base = row0 * ROWB + ((ln & 1) << 3);
    pa[c] = smem + base + (((4 * (2 * wn + c) + sub) ^ swz_v<TILE>(row0)) << 4);
    pb[c] = smem + STAGE / 2 + base + (((4 * (2 * wk + c) + sub) ^ swz_v<TILE>(row0)) << 4);
  }
  f32x16 acc[2][2];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.f;

#pragma unroll
  for (int b = 0; b < STAGES; ++b)
    if (b < count) request(b, b);
  if (count >= STAGES) wait_vmcnt_imm<(STAGES - 1) * LOADS>();
  else wait_vmcnt_imm<0>();
  cut(0, 0);
  lds_barrier();
  bf16x8 fa[2], fb[2];
#pragma unroll
  for (int c = 0; c < 2; ++c) {
    fa[c] = frag(pa[c], 0);
    fb[c] = frag(pb[c], 0);
  }
  int stage = 0;
#pragma unroll 1
  for (int kb = 0; kb < count; ++kb) {
    const int st = stage * STAGE, next = stage + 1 == STAGES ? 0 : stage + 1;
#pragma unroll
    for (int s = 0; s < KB / 16; ++s) {
      bf16x8 na[2], nb[2];
      if (s + 1 < KB / 16) {
#pragma unroll
        for (int c = 0; c < 2; ++c) {
          na[c] = frag(pa[c] + st, s + 1);
          nb[c] = frag(pb[c] + st, s + 1);
        }
      } else {
        // block kb + 1, requested STAGES - 1 blocks ago: younger ones stay out while there are STAGES - 2 of them
        if (kb + STAGES <= count) wait_vmcnt_imm<(STAGES - 2) * LOADS>();
        else wait_vmcnt_imm<0>();
        if (kb + 1 < count) cut(kb + 1, next);
        lds_barrier();
        if (kb + STAGES < count) request(kb + STAGES, stage);
#pragma unroll
        for (int c = 0; c < 2; ++c) {            // past the end: what lies there, for nobody
          na[c] = frag(pa[c] + next * STAGE, 0);
          nb[c] = frag(pb[c] + next * STAGE, 0);
        }
      }
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fa[i], fb[j], acc[i][j], 0, 0, 0);
#pragma unroll
      for (int c = 0; c < 2; ++c) {
        fa[c] = na[c];
        fb[c] = nb[c];
      }
    }
    stage = next;
  }
  if (GROUPS == 2) {                             // the second group's sums to the first, 64 KiB over the first's stages
    __syncthreads();
    float* merge = (float*)all_stages + wave * 64 * 64 + lane;
    if (group == 1) {
#pragma unroll
      for (int i = 0; i < 64; ++i) merge[i * 64] = acc[i >> 5][(i >> 4) & 1][i & 15];
    }
    __syncthreads();
    if (group == 1) return;
#pragma unroll
    for (int i = 0; i < 64; ++i) acc[i >> 5][(i >> 4) & 1][i & 15] += merge[i * 64];
  }
  // lane: column k0 + 64 wk + 32 j + ln of 16 rows
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const int k = k0 + 64 * wk + 32 * j + ln;
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        const int n = n0 + 64 * wn + 32 * i + (e >> 2) * 8 + hh * 4 + (e & 3);
        if (n < a.N && k < a.K) {
          if (PARTIAL) ((float*)a.out)[((int64_t)split * a.N + n) * a.K + k] = acc[i][j][e];
          else ((bf16_t*)a.out)[n * a.ldo + k] = f32_to_bf16(acc[i][j][e]);
        }
      }
    }
}

// The same on tiles of 256 x 128 (or 128 x 256) outputs: a workgroup of 8 waves of 64 x 64, alone on its CU, on a ring of three blocks of 64
// rows.  Two tiles of 128 x 128 a CU send 32 requests of 1 KiB for 32 rows where these send 24; a request takes 16 cycles of the CU's one address unit,
// 512 or 384 cycles beside 512 of products.  A block's requests follow its products one by one over three quarters of a block: sent together
// every wave stands in line for that unit.  Bound by the LDS now (fragments 256 cycles of 16 rows' 256 of products, the requests' rows 96).  us,
// both launches, tiles of 128 x 128 / these: [3456,768] over 3072 rows 30.0 / 29.0, 6400 47.4 / 43.6, 16000 111 / 89, 32768 208 / 171; [768,1728]
// 2560 21.1 / 22.6, 6400 28.8 / 28.4, 32768 111 / 93; [768,2624] 6400 37.4 / 36.1; [768,768] 16000 30.0 / 29.9; [2952,3384] 12260 387 / 303.
constexpr int WKB = 64, WSTAGES = 3;
template <int TN, int TK>
struct wide {
  static constexpr int STAGE = WKB * (TN + TK) * 2, LDS = WSTAGES * STAGE;
  static constexpr int Y_LOADS = WKB * TN * 2 / 1024 / 8, X_LOADS = WKB * TK * 2 / 1024 / 8, LOADS = Y_LOADS + X_LOADS;
  static_assert(TN * TK == 64 * 64 * 8 && LDS <= 160 * 1024, "eight waves, the LDS of a CU");
};
// chunks of 16 bytes of a row: a transposing read takes 64 bytes of four rows in a row, which cover all banks
__device__ inline int swz_wide(int row) { return (row & 3) << 2; }

template <int TN, int TK, bool PARTIAL>
__global__ __launch_bounds__(512) void linear_wgrad_wide_kernel(args a) {
  using G = wide<TN, TK>;
  constexpr int P = 4, WK = TK / 64;             // products of a slice of 16 rows, waves along the columns
  extern __shared__ __attribute__((aligned(1024))) unsigned char smem[];
  const int tid = threadIdx.x, lane = tid & 63, ln = lane & 31, hh = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), wn = wave / WK, wk = wave % WK;
  const int total = gridDim.x, per = total / 8, left = total % 8, xcd = blockIdx.x & 7;
  const int id = xcd * per + min(xcd, left) + (int)(blockIdx.x >> 3);          // as above
  const int tiles = total / a.splits, split = id / tiles, tile = id % tiles;
  const int n0 = tile / a.tiles_k * TN, k0 = tile % a.tiles_k * TK;
  const int first = (int)((int64_t)a.blocks * split / a.splits), last = (int)((int64_t)a.blocks * (split + 1) / a.splits);
  const int count = last - first;                // at least one block

  // request r of a wave: 1 KiB of the block of dY, then of X, as it lies; columns past the end: any, their outputs are not stored
  uint32_t off[G::LOADS];
  int row_of[G::LOADS];
  auto offset = [&](int r, int row) {
    const bool y = r < G::Y_LOADS;
    const int chunks = (y ? TN : TK) / 8, at = (wave + 8 * (y ? r : r - G::Y_LOADS)) * 64 + lane;
    const int col = (at % chunks ^ swz_wide(row_of[r])) * 8;
    return (uint32_t)(row * (int)(y ? a.ldy : a.ldx) + (y ? min(n0 + col, a.N - 8) : min(k0 + col, a.K - 8))) * 2;
  };
#pragma unroll
  for (int r = 0; r < G::LOADS; ++r) {
    const bool y = r < G::Y_LOADS;
    row_of[r] = ((wave + 8 * (y ? r : r - G::Y_LOADS)) * 64 + lane) / ((y ? TN : TK) / 8);
    off[r] = offset(r, row_of[r]);
  }
  const uint32_t lds0 = (uint32_t)(uintptr_t)(LDS_PTR(unsigned char))smem;
  int next = 0;                                  // block requested next; past the end the last one again, into a stage nobody reads
  uint32_t dst = lds0 + wave * 1024;
  const bf16_t *ys = a.dy + (int64_t)first * WKB * a.ldy, *xs = a.x + (int64_t)first * WKB * a.ldx;
  auto rows_in = [&](int kb) { return (int)min((int64_t)WKB, (int64_t)a.M - (int64_t)(first + kb) * WKB); };
  auto request = [&](int r) {
    const bool y = r < G::Y_LOADS;
    uint32_t o = off[r];
    const int rows = rows_in(next);
    if (rows < WKB) o = offset(r, min(row_of[r], rows - 1));                   // the last row again where there are no more
    load_to_lds_16(y ? ys : xs, o, dst + (y ? r * 8192 : WKB * TN * 2 + (r - G::Y_LOADS) * 8192));
  };
  auto next_block = [&]() {
    dst = dst + G::STAGE >= lds0 + G::LDS ? dst - (WSTAGES - 1) * G::STAGE : dst + G::STAGE;
    if (next + 1 < count) {
      ++next;
      ys += WKB * a.ldy;
      xs += WKB * a.ldx;
    }
  };
  // a block that reaches past the last row: zeros there, in what this wave has requested itself
  auto cut = [&](int kb, int stage) {
    const int rows = rows_in(kb);
    if (rows >= WKB) return;
#pragma unroll
    for (int r = 0; r < G::LOADS; ++r) {
      const int at = stage * G::STAGE + wave * 1024 + (r < G::Y_LOADS ? r * 8192 : WKB * TN * 2 + (r - G::Y_LOADS) * 8192) + lane * 16;
      if (row_of[r] >= rows) *(u32x4*)(smem + at) = u32x4{0u, 0u, 0u, 0u};
    }
  };

  // a lane's part of a fragment: rows 8 hh + (ln & 15) / 4 and four further on, of the lane's 4 of 32 columns
  const int row0 = 8 * hh + ((ln & 15) >> 2), sub = 2 * (ln >> 4) + ((ln & 3) >> 1);
  int ya[2], xa[2];
#pragma unroll
  for (int c = 0; c < 2; ++c) {
    ya[c] = row0 * TN * 2 + (((8 * wn + 4 * c + sub) ^ swz_wide(row0)) << 4) + ((ln & 1) << 3);
    xa[c] = WKB * TN * 2 + row0 * TK * 2 + (((8 * wk + 4 * c + sub) ^ swz_wide(row0)) << 4) + ((ln & 1) << 3);
  }
  auto read = [&](const unsigned char* p, int pitch) {
    const bf16x4 lo = el_bf16::read_tr(p), hi = el_bf16::read_tr(p + 4 * pitch);
    return __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
  };
  auto y_frag = [&](const unsigned char* st, int c, int sl) { return read(st + ya[c] + 16 * sl * TN * 2, TN * 2); };
  auto x_frag = [&](const unsigned char* st, int c, int sl) { return read(st + xa[c] + 16 * sl * TK * 2, TK * 2); };

#pragma unroll
  for (int b = 0; b < WSTAGES; ++b) {
#pragma unroll
    for (int r = 0; r < G::LOADS; ++r) request(r);
    next_block();
  }
  wait_vmcnt_imm<(WSTAGES - 1) * G::LOADS>();
  cut(0, 0);
  lds_barrier();
  bf16x8 fy[2][2], fx[2][2];                     // two slices' fragments
#pragma unroll
  for (int c = 0; c < 2; ++c) {
    fy[0][c] = y_frag(smem, c, 0);
    fx[0][c] = x_frag(smem, c, 0);
  }
  f32x16 acc[2][2];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.f;
  int stage = 0;
#pragma unroll 1
  for (int kb = 0; kb < count; ++kb) {
    const unsigned char* st = smem + stage * G::STAGE;
    // products of the fragments in f, between them those of the next slice are read and, for `turn` 0 .. 2 (the block's last slice, then two of
    // the block behind it), a block's requests sent
    auto products = [&](int f, int turn, int next_slice) __attribute__((always_inline)) {
#pragma unroll
      for (int q = 0; q < P; ++q) {
        const int i = q >> 1, j = q & 1;
        if (q < 2) fy[f ^ 1][q] = y_frag(st, q, next_slice);
        else fx[f ^ 1][q - 2] = x_frag(st, q - 2, next_slice);
        __builtin_amdgcn_sched_barrier(0);
        acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fy[f][i], fx[f][j], acc[i][j], 0, 0, 0);
        __builtin_amdgcn_sched_barrier(0);
        const int p = turn * P + q;
        if (p < 3 * P && (kb > 0 || turn == 0)) {
#pragma unroll
          for (int r = p * G::LOADS / (3 * P); r < (p + 1) * G::LOADS / (3 * P); ++r) request(r);
          if (p == 3 * P - 1) next_block();
        }
        __builtin_amdgcn_sched_barrier(0);
      }
    };
    products(0, 1, 1);
    products(1, 2, 2);
    products(0, 3, 3);
    // the next block has landed, and every fragment of this one is in registers: publish / free
    wait_vmcnt_imm<(WSTAGES - 2) * G::LOADS>();
    stage = stage + 1 == WSTAGES ? 0 : stage + 1;
    if (kb + 1 < count) cut(kb + 1, stage);
    lds_barrier();
    st = smem + stage * G::STAGE;                // past the end: what lies there, for nobody
    products(1, 0, 0);
  }
  wait_vmcnt_imm<0>();                           // (the requests past the end)
  // lane: column k0 + 64 wk + 32 j + ln of 16 rows
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const int k = k0 + 64 * wk + 32 * j + ln;
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        const int n = n0 + 64 * wn + 32 * i + (e >> 2) * 8 + hh * 4 + (e & 3);
        if (n < a.N && k < a.K) {
          if (PARTIAL) ((float*)a.out)[((int64_t)split * a.N + n) * a.K + k] = acc[i][j][e];
          else ((bf16_t*)a.out)[n * a.ldo + k] = f32_to_bf16(acc[i][j][e]);
        }
      }
    }
}

// dW = the sum of the partial tiles, a thread 8 columns of a row
__global__ __launch_bounds__(256) void linear_wgrad_reduce_kernel(const float* __restrict__ part, bf16_t* __restrict__ dw, int N, int K,
                                                                  int64_t ldo, int splits) {
  const int64_t i = ((int64_t)blockIdx.x * 256 + threadIdx.x) * 8, size = (int64_t)N * K;
  if (i >= size) return;
  float v[8] = {};
#pragma unroll 4
  for (int s = 0; s < splits; ++s) {
    const float4 lo = *(const float4*)(part + s * size + i), hi = *(const float4*)(part + s * size + i + 4);
    v[0] += lo.x; v[1] += lo.y; v[2] += lo.z; v[3] += lo.w;
    v[4] += hi.x; v[5] += hi.y; v[6] += hi.z; v[7] += hi.w;
  }
  *(bf16x8*)(dw + i / K * ldo + i % K) = bf16x8{(__bf16)v[0], (__bf16)v[1], (__bf16)v[2], (__bf16)v[3],
                                                (__bf16)v[4], (__bf16)v[5], (__bf16)v[6], (__bf16)v[7]};
}

static int tiles_of(int64_t N, int64_t K) { return (int)((N + TILE - 1) / TILE * ((K + TILE - 1) / TILE)); }

// How the rows are dealt, by what launches were seen to take (every plan of 132 shapes: the one chosen here is 0.5 % behind the best on
// average, 4 % with 0.6 us a block, 3 for a second launch and no more for a second group): a group of 4 waves 0.45 us a block
// where two share a CU and 0.4 alone, the second group's sums 2.5, partial results one launch, 0.15 a share and 2 x 4 bytes an
// output and share at 6 TB/s.  Both launches over 6400 rows, eight sets of them in
// turn, us (vendor library): [3456,768] 53 (73), [768,1728] 32 (49), [1280,768] 26 (42), [768,768] 22 (39).  Pairs of groups
// took 6 to 8 us off the last three.  ([3456,768] over 5120 rows 42.7 -> 46.5 us when blocks became 32 rows, 43.1 with these costs; 64 rows of
// [768,768] 7.65 -> 8.8 -> 7.75.)  The wide tiles: 0.64 us a block of 64 rows and 1 a round more; of 65 shapes from 570 to 32768 rows
// the plan chosen is 0.2 % behind the faster of the best plan on either tile (one 13 %: [240,2032] over 17880 rows, 37.5 / 33.0).  They are taken where
// that is a hundredth less, and of fewer than 128 columns on either side, whose tile is padding for the most part and which it flatters, a sixth less.  us, tiles
// of 128 x 128 / wide (what it says of them): [1728,8] over 33004 rows 28.3 / 31.0 (0.93), [24,3456] 15715 28.8 / 30.9 (0.87), [3456,32] 6150 15.3 / 16.1 (0.97),
// [1280,136] 16951 21.9 / 22.6 (1.00), [2624,8] 26490 33.0 / 33.2 (0.85); [5632,16] 12564 34.9 / 32.9 (0.83), [4096,24] 36759 62.2 / 56.9 (0.79).
struct plan {
  int groups, splits;
  int tn, tk;                                    // of the wide kernel; 0: tiles of 128 x 128
};
static plan plan_of(int64_t M, int64_t N, int64_t K) {
  const int64_t blocks = (M + KB - 1) / KB, tiles = tiles_of(N, K);
  plan best{1, 1, 0, 0};
  double best_us = 1e30;
  for (int groups = 1; groups <= 2; ++groups)
    for (int s = 1; s <= 32 && (s == 1 || (int64_t)s * groups <= blocks); ++s) {
      const int64_t slots = 512 / groups, rounds = (tiles * s + slots - 1) / slots, each = (blocks + s * groups - 1) / (s * groups);
      const int64_t last = (tiles * s - (rounds - 1) * slots) * groups;          // groups of the last round
      const double us = each * ((rounds - 1) * 0.45 + (last <= 256 ? 0.4 : 0.45)) + (groups - 1) * 2.5 +
                        (s > 1 ? 1.0 + 0.15 * s + 8e-6 * s * N * K / 6.0 : 0.0);
      if (us < best_us) {
        best_us = us;
        best = {groups, s, 0, 0};
      }
    }
  const int64_t wblocks = (M + WKB - 1) / WKB;
  best_us *= N < 128 || K < 128 ? 0.84 : 0.99;
  for (int t = 0; t < 2; ++t) {
    const int tn = t ? 128 : 256, tk = t ? 256 : 128;
    const int64_t wtiles = (N + tn - 1) / tn * ((K + tk - 1) / tk);
    for (int s = 1; s <= 32 && (s == 1 || s <= wblocks); ++s) {
      const int64_t rounds = (wtiles * s + 255) / 256, each = (wblocks + s - 1) / s;
      const double us = 1e-3 * wtiles * s + rounds * (each * 0.64 + 1.0) + (s > 1 ? 1.0 + 0.15 * s + 8e-6 * s * N * K / 6.0 : 0.0);
      if (us < best_us) {
        best_us = us;
        best = {1, s, tn, tk};
      }
    }
  }
  return best;
}

}  // namespace wgrad
}  // namespace mvpa

using namespace mvpa;

extern "C" size_t mvpa_linear_wgrad_ws_bytes(int64_t M, int64_t N, int64_t K) {
  if (M <= 0 || N <= 0 || K <= 0 || N > (1 << 20) || K > (1 << 20)) return 0;
  const int s = wgrad::plan_of(M, N, K).splits;
  return s == 1 ? 0 : (size_t)s * N * K * sizeof(float);
}

extern "C" int mvpa_linear_wgrad_bf16(const void* dy, const void* x, void* dw, int64_t M, int64_t N, int64_t K, int64_t lddy,
                                      int64_t ldx, int64_t lddw, void* ws, size_t ws_bytes, void* stream) {
  if (!dy || !x || !dw) return MVPA_ERR_NULL;
  if (M <= 0 || N <= 0 || K <= 0 || N > (1 << 20) || K > (1 << 20) || M > ((int64_t)1 << 30) || lddy < N || ldx < K || lddw < K)
    return MVPA_ERR_SHAPE;
  if ((N | K | lddy | ldx | lddw) % 8 != 0 || (((uintptr_t)dy | (uintptr_t)x | (uintptr_t)dw | (uintptr_t)ws) & 15)) return MVPA_ERR_ALIGN;
  const wgrad::plan p = wgrad::plan_of(M, N, K);
  const size_t need = p.splits == 1 ? 0 : (size_t)p.splits * N * K * sizeof(float);
  if (need > ws_bytes || (need && !ws)) return MVPA_ERR_WS_SIZE;
  // rows farther apart than 32 bits of a block's bytes: a handful of them fills the memory, any plan will do
  const bool far = lddy > (1 << 25) || ldx > (1 << 25), wide = p.tn && !far;
  const int tn = wide ? p.tn : wgrad::TILE, tk = wide ? p.tk : wgrad::TILE, kb = wide ? wgrad::WKB : wgrad::KB;
  wgrad::args a{(const bf16_t*)dy, (const bf16_t*)x, p.splits > 1 ? ws : dw, lddy, ldx, lddw, (int32_t)M, (int32_t)N, (int32_t)K,
                (int32_t)((K + tk - 1) / tk), p.splits, (int32_t)((M + kb - 1) / kb)};
  hipStream_t s = (hipStream_t)stream;
  const int groups = far ? 1 : p.groups;
  const unsigned grid = (unsigned)((N + tn - 1) / tn * ((K + tk - 1) / tk) * p.splits);
  if (wide) {
    auto kern = tn == 256 ? p.splits > 1 ? wgrad::linear_wgrad_wide_kernel<256, 128, true> : wgrad::linear_wgrad_wide_kernel<256, 128, false>
                          : p.splits > 1 ? wgrad::linear_wgrad_wide_kernel<128, 256, true> : wgrad::linear_wgrad_wide_kernel<128, 256, false>;
    const int lds = wgrad::wide<256, 128>::LDS;
    want_dynamic_lds((const void*)kern, lds);
    MVPA_LAUNCH(kern, dim3(grid), dim3(512), lds, s, a);
  } else {
    auto kern = far ? p.splits > 1 ? wgrad::linear_wgrad_kernel<1, true, true> : wgrad::linear_wgrad_kernel<1, false, true>
              : groups == 2 ? p.splits > 1 ? wgrad::linear_wgrad_kernel<2, true> : wgrad::linear_wgrad_kernel<2, false>
                              : p.splits > 1 ? wgrad::linear_wgrad_kernel<1, true> : wgrad::linear_wgrad_kernel<1, false>;
    const int lds = wgrad::STAGES * wgrad::STAGE * groups;
    want_dynamic_lds((const void*)kern, lds);
    MVPA_LAUNCH(kern, dim3(grid), dim3(256 * groups), lds, s, a);
  }
  if (p.splits > 1)
    MVPA_LAUNCH(wgrad::linear_wgrad_reduce_kernel, dim3((unsigned)((N * K / 8 + 255) / 256)), dim3(256), 0, s, (const float*)ws,
                (bf16_t*)dw, (int)N, (int)K, lddw, p.splits);
  return take_launch_status();
}
