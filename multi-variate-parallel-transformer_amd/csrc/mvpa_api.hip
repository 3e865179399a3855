// Host side of the C ABI: argument validation, kernel selection, status strings.
// Nothing here touches device memory, so mvpa_validate / mvpa_select_kernel work on a machine
// without a GPU.
#include "mvpa_common.h"
#include "mvpa_mfma_tools.h"

extern "C" int mvpa_version(void) { return MVPA_ABI_VERSION; }

extern "C" const char* mvpa_error_string(int status) {
  switch (status) {
    case MVPA_OK: return "ok";
    case MVPA_ERR_NULL: return "required pointer is null";
    case MVPA_ERR_HEAD_DIM: return "head dim must be one of 16, 32, 64, 128";
    case MVPA_ERR_HEAD_RATIO: return "Q heads must be divisible by KV heads";
    case MVPA_ERR_CTX: return "time and channel context must be positive";
    case MVPA_ERR_SHAPE: return "bad shape (B, H must be positive; N must equal T*C)";
    case MVPA_ERR_DTYPE: return "unknown dtype or kernel selector";
    case MVPA_ERR_ALIGN: return "pointer or stride not aligned to 16 bytes";
    case MVPA_ERR_UNSUPPORTED: return "request not supported by the selected kernel";
    case MVPA_ERR_STRUCT: return "argument struct size does not match the library";
    case MVPA_ERR_LAUNCH: return "kernel launch failed";
    case MVPA_ERR_NONCAUSAL_BIAS: return "relative biases require the time-causal mask";
    case MVPA_ERR_WS_SIZE: return "request needs more workspace than the library's built-in array holds";
  }
  return "unknown status";
}

extern "C" int mvpa_validate(const mvpa_fwd_args* a) {
  if (!a) return MVPA_ERR_NULL;
  if (a->struct_size != sizeof(mvpa_fwd_args)) return MVPA_ERR_STRUCT;
  if (a->dtype != MVPA_F32 && a->dtype != MVPA_BF16 && a->dtype != MVPA_F16) return MVPA_ERR_DTYPE;
  if (a->kernel < MVPA_KERNEL_AUTO || a->kernel > MVPA_KERNEL_MFMA_SPLIT) return MVPA_ERR_DTYPE;
  if (a->Dh != 16 && a->Dh != 32 && a->Dh != 64 && a->Dh != 128) return MVPA_ERR_HEAD_DIM;
  if (a->B <= 0 || a->H <= 0 || a->Hkv <= 0) return MVPA_ERR_SHAPE;
  if (a->H % a->Hkv != 0) return MVPA_ERR_HEAD_RATIO;
  if (a->T <= 0 || a->C <= 0) return MVPA_ERR_CTX;
  if ((int64_t)a->T * a->C > (int64_t)1 << 24) return MVPA_ERR_SHAPE;
  if (a->window < 0) return MVPA_ERR_SHAPE;
  if (!a->q || !a->k || !a->v || !a->o) return MVPA_ERR_NULL;
  if (!a->bias_u || !a->bias_v || !a->bias_z || !a->k_time || !a->k_chan) return MVPA_ERR_NULL;
  if ((a->flags & (MVPA_FLAG_TIME_BIAS | MVPA_FLAG_CHAN_BIAS)) && !(a->flags & MVPA_FLAG_CAUSAL))
    return MVPA_ERR_NONCAUSAL_BIAS;
  if ((a->flags & MVPA_FLAG_LAST_STEP) && !(a->flags & MVPA_FLAG_CAUSAL)) return MVPA_ERR_UNSUPPORTED;
  const int64_t n = (int64_t)a->T * a->C;
  // a token stride smaller than Dh (or a head/batch stride of 0 with more than one head)
  // means the caller's N does not match T*C or the view is wrong
  if (a->q_stride_n < a->Dh || a->k_stride_n < a->Dh || a->v_stride_n < a->Dh ||
      a->o_stride_n < a->Dh)
    return MVPA_ERR_SHAPE;
  (void)n;
  if (a->flags & MVPA_FLAG_FP8_QK) {
    if (a->dtype != MVPA_BF16) return MVPA_ERR_UNSUPPORTED;
    if (!a->fp8_q_scale || !a->fp8_k_scale) return MVPA_ERR_NULL;
  }
  if (a->flags & MVPA_FLAG_RING) {
    if (!(a->flags & MVPA_FLAG_LAST_STEP)) return MVPA_ERR_UNSUPPORTED;
    if (!a->ring_head) return MVPA_ERR_NULL;
  }
  if (a->n_split < 0 || a->n_split > a->T) return MVPA_ERR_SHAPE;
  if (a->n_split > 1) {
    if (!(a->flags & MVPA_FLAG_LAST_STEP)) return MVPA_ERR_UNSUPPORTED;
    if (!a->split_ws) return MVPA_ERR_NULL;
    if ((uintptr_t)a->split_ws & 15) return MVPA_ERR_ALIGN;
    const int len = (a->T + a->n_split - 1) / a->n_split;
    if ((int64_t)(a->n_split - 1) * len >= a->T) return MVPA_ERR_SHAPE;   // an empty run
  }
  if (a->kernel == MVPA_KERNEL_MFMA_STEP && mvpa_mfma_supported(a) && !mvpa_mfma64_supported(a))
    return MVPA_ERR_UNSUPPORTED;
  if (a->kernel == MVPA_KERNEL_MFMA_SPLIT && mvpa_mfma_supported(a) && !mvpa_mfma128_supported(a))
    return MVPA_ERR_UNSUPPORTED;
  if (a->kernel >= MVPA_KERNEL_MFMA && !mvpa_mfma_supported(a)) {
    if (a->dtype == MVPA_BF16) {
      const uintptr_t p = (uintptr_t)a->q | (uintptr_t)a->k | (uintptr_t)a->v | (uintptr_t)a->o;
      const int64_t s = a->q_stride_b | a->q_stride_h | a->q_stride_n | a->k_stride_b |
                        a->k_stride_h | a->k_stride_n | a->v_stride_b | a->v_stride_h |
                        a->v_stride_n | a->o_stride_b | a->o_stride_h | a->o_stride_n;
      if ((p & 15) || (s & 7)) return MVPA_ERR_ALIGN;
    }
    return MVPA_ERR_UNSUPPORTED;
  }
  return MVPA_OK;
}

extern "C" size_t mvpa_split_ws_bytes(const mvpa_fwd_args* a) {
  if (!a || a->n_split <= 1) return 0;
  return (size_t)a->n_split * a->B * a->H * a->C * ((size_t)a->Dh * 2 + sizeof(float));
}

extern "C" int mvpa_debug_block_order(int32_t n_bh, int32_t n_tiles, int32_t heads_per_kv, int32_t* bh,
                                      int32_t* tile) {
  if (!bh || !tile) return MVPA_ERR_NULL;
  if (n_bh <= 0 || n_tiles <= 0 || heads_per_kv <= 0) return MVPA_ERR_SHAPE;
  for (int L = 0; L < n_bh * n_tiles; ++L) {
    int x, y;
    mvpa::map_block(L, n_bh, n_tiles, heads_per_kv, x, y);
    bh[L] = x;
    tile[L] = y;
  }
  return MVPA_OK;
}

extern "C" int mvpa_debug_walk_order(int32_t n_walks, int32_t n_items, int32_t slots, int32_t alone, int32_t* walk,
                                     int32_t* item) {
  if (!walk || !item) return MVPA_ERR_NULL;
  if (n_walks <= 0 || n_items <= 0 || slots <= 0 || alone < 0) return MVPA_ERR_SHAPE;
  for (int L = 0; L < n_walks * n_items; ++L) {
    int w, i;
    mvpa::deal_walks(L, n_walks, n_items, slots, alone, w, i);
    walk[L] = w;
    item[L] = i;
  }
  return MVPA_OK;
}

extern "C" int mvpa_select_kernel(const mvpa_fwd_args* a) {
  const int st = mvpa_validate(a);
  if (st != MVPA_OK) return st;
  if (a->kernel == MVPA_KERNEL_GENERIC) return MVPA_KERNEL_GENERIC;
  if (a->kernel >= MVPA_KERNEL_MFMA) return MVPA_KERNEL_MFMA;
  return mvpa_mfma_supported(a) ? MVPA_KERNEL_MFMA : MVPA_KERNEL_GENERIC;
}

extern "C" int mvpa_forward(const mvpa_fwd_args* a, void* stream) {
  const int sel = mvpa_select_kernel(a);
  if (sel < 0) return sel;
  if (sel == MVPA_KERNEL_MFMA) {
    hipStream_t st = (hipStream_t)stream;
    if (a->kernel == MVPA_KERNEL_MFMA_STEP) return mvpa_launch_mfma64(a, st);
    if (a->kernel == MVPA_KERNEL_MFMA_SPLIT) return mvpa_launch_mfma128(a, st);
    if (a->kernel == MVPA_KERNEL_MFMA) return mvpa_launch_mfma(a, st);
    // AUTO: the specialised builds where they are the faster ones.
    // Launches that leave the chip idle: the build whose waves split the keys of a query tile.  Its time follows the
    // number of its workgroups (B H T and the query tiles of a step), the other kernels' is one chain over the steps
    // until they fill the chip, so the line lies where the two meet (us, general : this).  Up to 32 channels and 64, by B H:
    // T 25 at 12 / 24 / 48 / 64 23.5 : 10.0, 23.7 : 12.8, 24.1 : 21.6, 24.2 : 26.9; T 32 at 48 / 64 27.9 : 24.0, 28.1 :
    // 32.2; T 64 at 12 / 24 / 48 50.1 : 19.1, 50.5 : 33.8, 51.8 : 58.1.  From T 80 on the general kernel's last step is no chain of
    // one wave, and tables of more than 64 rows leave this one a workgroup a CU: T 80 at 12 / 24 41.4 : 33.7, 42.5 : 64.7; T 96 at
    // 12 45.8 : 43.0; T 110 at 16 51.9 : 68.4; T 160 at 12 67.4 : 87.2; T 200 at 8 80.6 : 85.6; T 300 at 4 114 : 83.9; T 500
    // at 4 181 : 197; head size 32 T 100 at 16 35.0 : 32.9, T 200 at 8 57 : 47, T 250 at 8 68.4 : 66.6, T 500 at 4 122 : 160.
    // 33..64 channels, by workgroups, T 12 at 576 / 1152 17.3 : 13.5, 19.1 : 22.3; T 16 at 768 19.1 : 16.3; T 25
    // at 600 / 800 / 1200 23.2 : 16.9, 23.6 : 21.6, 25.9 : 26.7; T 40 at 960 29.5 : 35.4; Dh 32 at 768 / 1600 18.1 : 13.5,
    // 24.8 : 26.8.  Head size 128 has one workgroup per CU, the general kernel two from T 32, C21 by workgroups: T 32 at 1024 / 1280
    // 37.3 : 38.5, 48.2 : 48.1; T 48 at 1152 / 1536 51.4 : 50.5, 55.0 : 63.0; T 64 at 1024 / 1536 52.0 : 48.3, 63.3 : 69.5; T 100 at 1200 / 1600
    // 83 : 66, 79 : 86; T 128 at 1024 78 : 66; T 25 at 400 36 : 20.
    if (!(a->flags & MVPA_FLAG_LAST_STEP) && a->C <= (a->Dh == 128 ? 32 : 64) && mvpa_wave_supported(a)) {
      const int64_t wgs = (int64_t)a->B * a->H * ((a->C + 31) / 32) * a->T, T = a->T;
      int64_t most = 512;
      if (a->Dh == 128) most = T >= 32 ? 1200 : 24 * T > most ? 24 * T : most;
      else if (a->C > 32) most = T <= 32 ? 768 : most;
      else if (T >= (a->Dh == 32 ? 257 : 80)) most = 1200;
      else if (48 * T > most) most = 48 * T < 2048 ? 48 * T : 2048;
      if (wgs <= most) return mvpa_launch_wave(a, st);
    }
    // 65..128 channels at head size 64 or 128: the build of csrc/mvpa_mfma128.hip wins at every
    // length and channel count measured (Dh 128, B1 H16: C128 T 16 .. 1024 13 .. 20 % less time than
    // the general kernel, C 80 .. 100 21 .. 40 %; Dh 64, H16: B8 C117 T256 11.14 -> 8.58 ms,
    // B4 C128 T128 1.86 -> 1.34, B4 C80 T128 1.78 -> 1.21, B8 C128 T32 0.53 -> 0.38, B2 C128 T512
    // 9.99 -> 7.66 ms).
    if (mvpa_mfma128_supported(a) && a->C > 64) return mvpa_launch_mfma128(a, st);
    // The same build with two key tiles serves 33..64 channels: at head size 128 it wins too
    // (B1 H16 C64 T512 3.71 -> 2.87 ms, B4 C64 T64 0.42 -> 0.39); at head size 64 it loses to both
    // other builds (c2 0.49 against 0.40 and 0.38 ms: 8 products per wave and far step, one
    // workgroup per CU).
    if (mvpa_mfma128_supported(a) && a->Dh == 128) return mvpa_launch_mfma128(a, st);
    // Head size 64, 33..64 channels: the whole-time-step build pays for its window passes with a
    // cheaper far phase; against the general kernel it loses at 64 time steps (B4 H12 C64: 0.131
    // against 0.109 ms), is level at 128 and wins from there on (T 256: 6 %, T 512: 10 %), and
    // wins by 15 % when there are no window steps at all (content term off).
    if (mvpa_mfma64_supported(a) && (a->T >= 128 || !(a->flags & MVPA_FLAG_CONTENT))) return mvpa_launch_mfma64(a, st);
    return mvpa_launch_mfma(a, st);
  }
  if (a->flags & (MVPA_FLAG_FP8_QK | MVPA_FLAG_RING)) return MVPA_ERR_UNSUPPORTED;
  return mvpa_launch_generic(a, (hipStream_t)stream);
}
