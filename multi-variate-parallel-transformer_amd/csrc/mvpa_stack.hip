// The stack of parallel blocks as one call: a host-side sequence of the library's launches.
//
// A block is four or five short launches; driven one by one from the caller's language a window of 525
// rows or one step of a stream is bound by that caller (1.2 ms of host time for twelve blocks), not
// by the GPU.  Three sequences, by the number of rows:
//   many rows      [q/k/v | gate/up] on raw rows with ln_1 in the epilogue -> attention -> tail product
//                  with residual and the next norm's row statistics (mvpa_dense.hip, 256-row tiles)
//   few rows       [q/k/v | gate/up] on small tiles, of raw rows (ln_1 in the epilogue) or of normed ones ->
//                  attention -> split-K tail -> sum + residual + the row statistics or the normed rows
//                  that the next block wants (mvpa_tiles.hip)
//   a step         the latter with the new keys and values written straight into the caches by the
//                  product's epilogue, and the attention of the last time step only
//   a step of      norm -> [q/k/v | gate/up] on 256-row tiles -> keys and values into the caches -> attention of
//   many rows      the last time step -> tail product with residual
#include "mvpa_mfma_tools.h"
#include "mvpa_tiles.h"

namespace mvpa {

// The 256-row tiles are the better ones once [q/k/v | gate/up] is this many of them, the more the longer the
// contraction; a step's small tiles write the caches themselves and stand a little longer.  256-row against small
// tiles, us a pass of all blocks (four of the base model's) at so many tiles,
//   windows of MVPFormer-S   228 1454 : 1306, 247 1486 : 1418, 266 1718 : 1552, 285 1717 : 1658, 304 1751 : 1777,
//                            342 1874 : 2029; 266 at 37 channels 2077 : 1882
//   of the base model        360 1244 : 1009, 420 1264 : 1096, 480 1315 : 1261, 600 1575 : 1690, 720 1659 : 2045
//   steps of MVPFormer-S     228 2002 : 2005, 266 2218 : 2243, 304 2288 : 2552, 456 2804 : 3781
//   of the base model        300 1597 : 1376, 360 1616 : 1509, 420 1636 : 1694, 480 1676 : 1883
// (The lines were drawn when small tiles took up to a fifth more; those of windows lie early by as much.)
static int64_t many_tiles(int64_t E, bool step) { return (step ? 176 : 148) + E / 8; }

static int64_t up256(int64_t n) { return (n + 255) & ~(int64_t)255; }

struct stack_ws {
  char* base;
  int64_t used;
  void* take(int64_t bytes) {
    void* p = base ? base + used : nullptr;
    used += up256(bytes);
    return p;
  }
};

struct stack_plan {
  bool many, raw;                      // 256-row tiles; ln_1 inside the products
  int64_t rows, ld_qkv;
  tile_split split_k;
  int runs;
  bf16_t *qkv, *both, *hidden[2], *normed;
  float *partial, *sumsq[2];
  float *q_scale, *k_scale;
  void *k_fp8, *split;
  int32_t parts;
};

static bool stack_supported(const mvpa_stack_args* a) {
  if (a->E != a->H * a->Dh || a->E % 64 || a->inner <= 0 || a->inner % 64 || a->E > 4096) return false;
  if (a->Dh != 32 && a->Dh != 64 && a->Dh != 128) return false;
  if (a->C > 128) return false;
  const int64_t nw = (int64_t)a->E + 2 * a->Hkv * a->Dh;
  const int64_t widest = 2 * (int64_t)a->inner > nw ? 2 * (int64_t)a->inner : nw;
  if (widest * a->E >= ((int64_t)1 << 30) || (int64_t)a->E * (a->E + a->inner) >= ((int64_t)1 << 30)) return false;
  return true;
}

// Key runs of a step: a power of two, up to one workgroup per CU (the query tiles of a head are workgroups
// of their own up to 64 channels) and no run under 4 steps (us by runs 4 / 8 / 16: H12 C64 T64 12.6 / 11.2 / 16.9,
// H12 C21 T64 10.5 / 9.7 / 10, H16 C128 T110 Dh128 60 / 37 / 28, H16 C64 T110 Dh128 28 / 22 / 33); still two, of
// 8 steps and more, while the (b, h) pairs alone leave half the CUs idle (us in one / two: B8 H16 C64 T110 Dh128
// 216 / 87, T25 57 / 40, B8 H12 C64 T64 Dh64 40 / 28, T25 20.9 / 19.3).
static int default_runs(const mvpa_stack_args* a) {
  const int wgs = a->B * a->H * (a->C > 64 ? 1 : (a->C + 31) / 32);
  int n = 1;
  while (2 * n * wgs <= 256 && 8 * n <= a->T) n *= 2;
  if (n == 1 && 2 * a->B * a->H <= 256 && a->T >= 16) n = 2;
  while (n > 1 && (int64_t)(n - 1) * ((a->T + n - 1) / n) >= a->T) --n;      // no empty run
  return n;
}

static void stack_layout(const mvpa_stack_args* a, stack_plan& p, stack_ws& w) {
  const int64_t E = a->E, kv = (int64_t)a->Hkv * a->Dh, inner = a->inner;
  p.rows = (int64_t)a->B * a->C * (a->step ? 1 : a->T);
  p.raw = !a->step && a->sumsq;
  for (int i = 0; i < a->n_blocks; ++i) p.raw = p.raw && a->blocks[i].w_qkv_normed && a->blocks[i].w_gate_up_normed;
  const int64_t tiles = (p.rows + 255) / 256 * ((inner + 127) / 128 + (E + 2 * kv + 255) / 256);
  p.many = (p.raw || a->step) && tiles >= many_tiles(E, a->step) && p.rows >= 512 && E >= 128;
  p.ld_qkv = a->step && !p.many ? E : E + 2 * kv;
  p.qkv = (bf16_t*)w.take(p.rows * p.ld_qkv * 2);
  p.both = (bf16_t*)w.take(p.rows * (E + inner) * 2);
  p.hidden[0] = (bf16_t*)w.take(p.rows * E * 2);
  p.hidden[1] = p.normed = nullptr;
  p.sumsq[0] = p.sumsq[1] = nullptr;
  p.partial = nullptr;
  if (p.many && a->step) {
    p.hidden[1] = (bf16_t*)w.take(p.rows * E * 2);
    p.normed = (bf16_t*)w.take(p.rows * E * 2);
  } else if (p.many) {
    p.hidden[1] = (bf16_t*)w.take(p.rows * E * 2);
    p.parts = mvpa_linear_sumsq_parts(p.rows, E);
    for (int i = 0; i < 2; ++i) p.sumsq[i] = (float*)w.take(p.rows * p.parts * 4);
  } else {
    if (p.raw) p.sumsq[0] = (float*)w.take(p.rows * 4);
    else p.normed = (bf16_t*)w.take(p.rows * E * 2);
    p.split_k = make_tile_split(p.rows, E, E + inner, p.raw ? 0 : E);
    p.partial = (float*)w.take((int64_t)p.split_k.total() * p.rows * E * 4);
  }
  p.runs = 1;
  p.split = nullptr;
  if (a->step) {
    p.runs = default_runs(a);
    if (p.runs > 1) p.split = w.take((int64_t)p.runs * a->B * a->H * a->C * (a->Dh * 2 + 4));
  }
  p.q_scale = p.k_scale = nullptr;
  p.k_fp8 = nullptr;
  bool fp8 = false;
  for (int i = 0; i < a->n_blocks; ++i) fp8 |= (a->blocks[i].flags & MVPA_FLAG_FP8_QK) != 0;
  if (fp8) {
    p.q_scale = (float*)w.take(a->H * 4);
    p.k_scale = (float*)w.take(a->Hkv * 4);
    if (!a->step && a->C > 32 && (a->Dh == 64 || a->Dh == 128)) p.k_fp8 = w.take((int64_t)a->B * a->T * a->C * kv);
  }
}

static int stack_check(const mvpa_stack_args* a) {
  if (!a) return MVPA_ERR_NULL;
  if (a->struct_size != sizeof(mvpa_stack_args)) return MVPA_ERR_STRUCT;
  if (a->n_blocks <= 0 || a->B <= 0 || a->H <= 0 || a->Hkv <= 0 || a->E <= 0) return MVPA_ERR_SHAPE;
  if (a->T <= 0 || a->C <= 0) return MVPA_ERR_CTX;
  if (a->H % a->Hkv) return MVPA_ERR_HEAD_RATIO;
  if (!a->blocks) return MVPA_ERR_NULL;
  return stack_supported(a) ? MVPA_OK : MVPA_ERR_UNSUPPORTED;
}

}  // namespace mvpa

using namespace mvpa;

extern "C" size_t mvpa_stack_ws_bytes(const mvpa_stack_args* a) {
  if (stack_check(a) != MVPA_OK) return 0;
  stack_plan p;
  stack_ws w{nullptr, 0};
  stack_layout(a, p, w);
  return (size_t)w.used;
}

extern "C" int mvpa_stack_forward(const mvpa_stack_args* a, void* stream) {
  return mvpa_stack_forward_blocks(a, 0, a ? a->n_blocks : 0, stream);
}

extern "C" int mvpa_stack_forward_blocks(const mvpa_stack_args* a, int32_t first, int32_t end, void* stream) {
  int st = stack_check(a);
  if (st != MVPA_OK) return st;
  if (first < 0 || end <= first || end > a->n_blocks) return MVPA_ERR_SHAPE;
  if (!a->x || !a->y || !a->lnf_weight || !a->ws) return MVPA_ERR_NULL;
  if (((uintptr_t)a->ws & 255) || ((uintptr_t)a->x & 15) || ((uintptr_t)a->y & 15)) return MVPA_ERR_ALIGN;
  stack_plan p;
  stack_ws w{(char*)a->ws, 0};
  stack_layout(a, p, w);
  if ((size_t)w.used > a->ws_bytes) return MVPA_ERR_WS_SIZE;
  hipStream_t s = (hipStream_t)stream;
  const int64_t E = a->E, kv = (int64_t)a->Hkv * a->Dh, inner = a->inner, wide = E + inner, nw = E + 2 * kv;
  const int64_t n = a->step ? a->C : (int64_t)a->T * a->C;

  // the attention of a block, from p.qkv (and the caches) to the first E columns of p.both
  auto attend = [&](const mvpa_stack_block& blk) -> int {
    mvpa_fwd_args f = {};
    f.struct_size = sizeof(f);
    f.dtype = MVPA_BF16;
    f.kernel = MVPA_KERNEL_AUTO;
    f.flags = MVPA_FLAG_CAUSAL | MVPA_FLAG_TIME_BIAS | MVPA_FLAG_CHAN_BIAS |
              (blk.flags & (MVPA_FLAG_CONTENT | MVPA_FLAG_FP8_QK));
    f.B = a->B; f.H = a->H; f.Hkv = a->Hkv; f.T = a->T; f.C = a->C; f.Dh = a->Dh;
    f.window = blk.window;
    f.sm_scale = blk.sm_scale;
    const int64_t row = p.ld_qkv;
    f.q = p.qkv;
    f.q_stride_b = n * row; f.q_stride_h = a->Dh; f.q_stride_n = row;
    if (a->step) {
      f.flags |= MVPA_FLAG_LAST_STEP | (a->ring_head ? MVPA_FLAG_RING : 0);
      f.ring_head = a->ring_head;
      f.k = blk.k_cache;
      f.v = blk.v_cache;
      f.k_stride_b = f.v_stride_b = blk.cache_stride_b;
      f.k_stride_h = f.v_stride_h = blk.cache_stride_g;
      f.k_stride_n = f.v_stride_n = a->Dh;
    } else {
      f.k = p.qkv + E;
      f.v = p.qkv + E + kv;
      f.k_stride_b = f.v_stride_b = n * row;
      f.k_stride_h = f.v_stride_h = a->Dh;
      f.k_stride_n = f.v_stride_n = row;
    }
    f.o = p.both;
    f.o_stride_b = n * wide; f.o_stride_h = a->Dh; f.o_stride_n = wide;
    f.bias_u = blk.bias_u; f.bias_v = blk.bias_v; f.bias_z = blk.bias_z;
    f.k_time = blk.k_time; f.k_chan = blk.k_chan;
    f.chan_valid = blk.chan_valid;
    if (f.flags & MVPA_FLAG_FP8_QK) {
      f.fp8_q_scale = p.q_scale;
      f.fp8_k_scale = p.k_scale;
      f.k_fp8 = p.k_fp8;
      const int e = mvpa_fp8_prepare(&f, p.q_scale, p.k_scale, p.k_fp8, stream);
      if (e != MVPA_OK) return e;
    }
    if (a->step && p.runs > 1) {
      f.n_split = p.runs;
      f.split_ws = p.split;
    }
    return mvpa_forward(&f, stream);
  };

  if (p.many && a->step) {
    if (first == 0 && (st = mvpa_rmsnorm(a->x, a->blocks[0].ln_weight, p.normed, p.rows, (int32_t)E, E, E, a->blocks[0].ln_eps,
                                         MVPA_BF16, MVPA_BF16, stream)) != MVPA_OK) return st;
    for (int i = first; i < end; ++i) {
      const mvpa_stack_block& blk = a->blocks[i];
      const bool last = i + 1 == a->n_blocks;
      if ((st = mvpa_linear_bf16_dual(p.normed, blk.w_qkv, p.qkv, blk.w_gate_up, p.both + E, p.rows, nw, inner, E, E, E, nw,
                                      E, wide, stream)) != MVPA_OK) return st;
      if ((st = launch_append(p.qkv + E, p.qkv + E + kv, (bf16_t*)blk.k_cache, (bf16_t*)blk.v_cache, a->ring_head, a->T - 1,
                              a->B, a->Hkv, a->C, a->Dh, n * nw, a->Dh, nw, blk.cache_stride_b, blk.cache_stride_g,
                              s)) != MVPA_OK) return st;
      if ((st = attend(blk)) != MVPA_OK) return st;
      if ((st = mvpa_linear_bf16_residual(p.both, blk.w_tail, i ? p.hidden[(i - 1) & 1] : a->x, p.hidden[i & 1], p.rows, E, wide,
                                          wide, wide, E, E, stream)) != MVPA_OK) return st;
      if ((st = mvpa_rmsnorm(p.hidden[i & 1], last ? a->lnf_weight : a->blocks[i + 1].ln_weight, last ? a->y : p.normed, p.rows,
                             (int32_t)E, E, E, last ? a->lnf_eps : a->blocks[i + 1].ln_eps, MVPA_BF16, MVPA_BF16,
                             stream)) != MVPA_OK) return st;
    }
    return MVPA_OK;
  }
  if (p.many) {
    for (int i = first; i < end; ++i) {
      const mvpa_stack_block& blk = a->blocks[i];
      const bf16_t* x = i ? p.hidden[(i - 1) & 1] : (const bf16_t*)a->x;
      const float* ss = i ? p.sumsq[i & 1] : a->sumsq;
      const int32_t parts = i ? p.parts : 1;
      if ((st = mvpa_linear_bf16_dual_normed(x, blk.w_qkv_normed, p.qkv, blk.w_gate_up_normed, p.both + E, p.rows, nw,
                                             inner, E, E, E, nw, E, wide, ss, parts, blk.ln_eps,
                                             stream)) != MVPA_OK) return st;
      if ((st = attend(blk)) != MVPA_OK) return st;
      if ((st = mvpa_linear_bf16_residual_sumsq(p.both, blk.w_tail, x, p.hidden[i & 1], p.sumsq[(i + 1) & 1], p.rows, E, wide, wide,
                                                wide, E, E, stream)) != MVPA_OK) return st;
    }
    if (end < a->n_blocks) return MVPA_OK;
    return mvpa_rmsnorm(p.hidden[(end - 1) & 1], a->lnf_weight, a->y, p.rows, (int32_t)E, E, E, a->lnf_eps, MVPA_BF16, MVPA_BF16, stream);
  }

  if (first == 0 && !p.raw && (st = mvpa_rmsnorm(a->x, a->blocks[0].ln_weight, p.normed, p.rows, (int32_t)E, E, E, a->blocks[0].ln_eps, MVPA_BF16,
                         MVPA_BF16, stream)) != MVPA_OK) return st;
  for (int i = first; i < end; ++i) {
    const mvpa_stack_block& blk = a->blocks[i];
    const bf16_t* x = i ? p.hidden[0] : (const bf16_t*)a->x;
    tile_out out = {};
    out.y = p.qkv;
    out.ldy = a->step ? E : nw;
    out.n_y = (int32_t)(a->step ? E : nw);
    if (a->step) {
      out.n_kv = (int32_t)kv;
      out.Dh = a->Dh;
      out.C = a->C;
      out.k = (bf16_t*)blk.k_cache;
      out.v = (bf16_t*)blk.v_cache;
      out.stride_b = blk.cache_stride_b;
      out.stride_g = blk.cache_stride_g;
      out.slot = a->T - 1;
      out.head = a->ring_head;
    }
    const tile_gated gated{(const bf16_t*)(p.raw ? blk.w_gate_up_normed : blk.w_gate_up), p.both + E, E, wide, (int32_t)inner};
    const tile_norm norm{p.raw ? (i ? p.sumsq[0] : a->sumsq) : nullptr, 1, blk.ln_eps};
    if ((st = launch_tile_dual(p.raw ? x : p.normed, p.rows, E, E, (const bf16_t*)(p.raw ? blk.w_qkv_normed : blk.w_qkv), nw,
                               E, out, gated, norm, s)) != MVPA_OK) return st;
    if ((st = attend(blk)) != MVPA_OK) return st;
    if ((st = launch_tile_partial(p.both, p.rows, wide, wide, (const bf16_t*)blk.w_tail, E, wide, p.partial, p.split_k, s)) != MVPA_OK) return st;
    const bool last = i + 1 == a->n_blocks;
    if ((st = launch_tail_reduce(p.partial, p.split_k, x, p.hidden[0], last ? (bf16_t*)a->y : p.raw ? nullptr : p.normed,
                                 last ? a->lnf_weight : a->blocks[i + 1].ln_weight, last ? a->lnf_eps : a->blocks[i + 1].ln_eps,
                                 p.raw && !last ? p.sumsq[0] : nullptr, p.rows, E, s)) != MVPA_OK) return st;
  }
  return MVPA_OK;
}
