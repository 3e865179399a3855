// Generic MVPA forward: one lane per query row, fp32 arithmetic throughout, any shape.
//
// This is the kernel behind the fp32 path (max-abs parity with the fp32 PyTorch MVPA,
// layers/mvpa.py:173-278) and behind every request the tiled bf16 MFMA kernel does not take
// (additive key bias, C > 128, content term without causal mask, ...).  It keeps the three
// score terms separate exactly as the reference sums them and uses expf, not a base-2
// shortcut, so that its rounding stays within a few ulp of torch.softmax.
//
// Work split: grid = (ceil(N/128), B*H); a workgroup owns 128 consecutive query tokens of one
// (b, h).  Key/value rows are staged through LDS 32 at a time as fp32 and broadcast to all
// lanes; the per-row channel table (q+z).e[j], j < C, is computed once into LDS.
#include "mvpa_common.h"

namespace mvpa {

constexpr int GEN_THREADS = 128;
constexpr int GEN_KT = 32;

template <typename T, int DH>
__global__ __launch_bounds__(GEN_THREADS) void mvpa_generic_kernel(mvpa_fwd_args a,
                                                                   int chan_table) {
  extern __shared__ float smem[];
  float* Ks = smem;                               // [KT][DH]
  float* Vs = Ks + GEN_KT * DH;                   // [KT][DH]
  float* Ss = Vs + GEN_KT * DH;                   // [KT][128] scores of the current tile
  float* Sc = Ss + GEN_KT * GEN_THREADS;          // [128][C+1] channel table (if chan_table)

  const int tid = threadIdx.x;
  const int T_ = a.T, C_ = a.C, N = a.T * a.C;
  const int b = blockIdx.y / a.H, h = blockIdx.y % a.H;
  const int g = h / (a.H / a.Hkv);
  const bool causal = a.flags & MVPA_FLAG_CAUSAL;
  const bool has_content = a.flags & MVPA_FLAG_CONTENT;
  const bool has_time = a.flags & MVPA_FLAG_TIME_BIAS;
  const bool has_chan = a.flags & MVPA_FLAG_CHAN_BIAS;

  // MVPA_FLAG_LAST_STEP: only the C queries of the last time step exist; rq is the row of q / o,
  // nq the query's place in the full sequence
  const bool last_only = a.flags & MVPA_FLAG_LAST_STEP;
  const int Nq = last_only ? C_ : N;
  const int nq_raw = blockIdx.x * GEN_THREADS + tid;
  const bool live = nq_raw < Nq;
  const int rq = live ? nq_raw : Nq - 1;          // clamp: dead lanes still take part in barriers
  const int nq = last_only ? (T_ - 1) * C_ + rq : rq;
  const int tq = nq / C_, cq = nq % C_;

  const T* qrow = (const T*)a.q + b * a.q_stride_b + h * a.q_stride_h + (int64_t)rq * a.q_stride_n;
  const T* kbase = (const T*)a.k + b * a.k_stride_b + g * a.k_stride_h;
  const T* vbase = (const T*)a.v + b * a.v_stride_b + g * a.v_stride_h;
  const T* bu = (const T*)a.bias_u + g * DH;
  const T* bv = (const T*)a.bias_v + g * DH;
  const T* bz = (const T*)a.bias_z + g * DH;
  const T* ktime = (const T*)a.k_time + (int64_t)g * T_ * DH;
  const T* kchan = (const T*)a.k_chan + (int64_t)g * C_ * DH;
  const uint8_t* valid = a.chan_valid ? a.chan_valid + (int64_t)b * C_ : nullptr;
  const float* kbias = a.key_bias ? a.key_bias + (int64_t)b * N : nullptr;

  float qu[DH];
#pragma unroll
  for (int d = 0; d < DH; ++d) qu[d] = io<T>::load(qrow + d) + io<T>::load(bu + d);

  // channel table: Sc[tid][j] = (q+z).e[j]
  const int sc_pitch = C_ + 1;
  if (has_chan && chan_table) {
    for (int j = 0; j < C_; ++j) {
      const T* e = kchan + (int64_t)j * DH;
      float s = 0.f;
#pragma unroll 8
      for (int d = 0; d < DH; ++d) s += (io<T>::load(qrow + d) + io<T>::load(bz + d)) * io<T>::load(e + d);
      Sc[tid * sc_pitch + j] = s;
    }
  }

  const int q_last = min(N - 1, (int)blockIdx.x * GEN_THREADS + GEN_THREADS - 1);
  const int hi = (causal && !last_only) ? (q_last / C_ + 1) * C_ : N;   // last step: every key

  float m = -INFINITY, l = 0.f;
  float acc[DH];
#pragma unroll
  for (int d = 0; d < DH; ++d) acc[d] = 0.f;
  int cur_tk = -1;
  float st = 0.f;

  for (int k0 = 0; k0 < hi; k0 += GEN_KT) {
    __syncthreads();
    for (int i = tid; i < GEN_KT * DH; i += GEN_THREADS) {
      const int kk = i / DH, d = i % DH;
      const int nk = k0 + kk;
      float kv = 0.f, vv = 0.f;
      if (nk < hi) {
        kv = io<T>::load(kbase + (int64_t)nk * a.k_stride_n + d);
        vv = io<T>::load(vbase + (int64_t)nk * a.v_stride_n + d);
      }
      Ks[i] = kv;
      Vs[i] = vv;
    }
    __syncthreads();

    float tmax = -INFINITY;
    for (int kk = 0; kk < GEN_KT; ++kk) {
      const int nk = k0 + kk;
      float x = -INFINITY;
      if (nk < hi) {
        const int tk = nk / C_, ck = nk - tk * C_;
        if (tk != cur_tk) {   // uniform across the workgroup: keys advance in lock step
          cur_tk = tk;
          st = 0.f;
          if (has_time && tk <= tq) {
            const T* r = ktime + (int64_t)time_row(tq, tk, T_) * DH;
#pragma unroll 8
            for (int d = 0; d < DH; ++d)
              st += (io<T>::load(qrow + d) + io<T>::load(bv + d)) * io<T>::load(r + d);
          }
        }
        const bool vis = causal_visible(tq, tk, causal) && (!valid || valid[ck] != 0);
        float sc = 0.f;
        if (has_chan) {
          const int j = chan_row(cq, ck, C_);
          if (chan_table) {
            sc = Sc[tid * sc_pitch + j];
          } else {
            const T* e = kchan + (int64_t)j * DH;
#pragma unroll 8
            for (int d = 0; d < DH; ++d)
              sc += (io<T>::load(qrow + d) + io<T>::load(bz + d)) * io<T>::load(e + d);
          }
        }
        float s = st + sc;
        const bool kept = has_content && content_kept(tq, tk, T_, a.window);
        if (__ballot(kept && vis) != 0ull) {   // wave-uniform skip of the content dot product
          float dot = 0.f;
          const float* kr = Ks + kk * DH;
#pragma unroll
          for (int d = 0; d < DH; ++d) dot += qu[d] * kr[d];
          if (kept) s += dot;
        }
        s *= a.sm_scale;
        if (kbias) s += kbias[nk];
        x = vis ? s : -INFINITY;
      }
      Ss[kk * GEN_THREADS + tid] = x;
      tmax = fmaxf(tmax, x);
    }

    const float m_new = fmaxf(m, tmax);
    if (m_new > -INFINITY) {
      const float alpha = (m == -INFINITY) ? 0.f : expf(m - m_new);
      l *= alpha;
#pragma unroll
      for (int d = 0; d < DH; ++d) acc[d] *= alpha;
      for (int kk = 0; kk < GEN_KT; ++kk) {
        const float x = Ss[kk * GEN_THREADS + tid];
        const float p = (x == -INFINITY) ? 0.f : expf(x - m_new);
        l += p;
        const float* vr = Vs + kk * DH;
#pragma unroll
        for (int d = 0; d < DH; ++d) acc[d] += p * vr[d];
      }
      m = m_new;
    }
  }

  if (live) {
    T* orow = (T*)a.o + b * a.o_stride_b + h * a.o_stride_h + (int64_t)rq * a.o_stride_n;
    const float inv = 1.f / l;
#pragma unroll
    for (int d = 0; d < DH; ++d) io<T>::store(orow + d, acc[d] * inv);
    if (a.lse) a.lse[((int64_t)b * a.H + h) * Nq + rq] = (m + logf(l)) * kLog2e;
  }
}

// -----------------------------------------------------------------------------------------
// The same operator on fp32 matrix instructions (v_mfma_f32_32x32x2_f32, exact fp32 products):
// what serves every generic request whose bias tables fit the LDS.  A workgroup owns 32 query
// tokens of one (b, h); its 8 waves take the 32-key tiles in turn, each with a soft-max state of
// its own, and merge through LDS at the end.  One lane per row (the kernel above) is a single
// dependent chain through every key and gives a small call 16 workgroups; here a wave sees an
// eighth of the keys and a call has N/32 workgroups per head.  Products are transposed as in the
// bf16 kernels (S^T = K Q^T, O^T = V^T P^T): a lane owns one query and the probabilities of a tile
// leave the first product in the operand layout of the second.  Both bias tables of the 32
// queries are formed once into LDS, [distance][query], and gathered per element.
// Bound: latency at the small end (B2 C8 T32 H4 Dh32: 211 -> 15 us), the fp32 matrix rate at the
// large one.
// -----------------------------------------------------------------------------------------
typedef __attribute__((ext_vector_type(16))) float gen_f32x16;
constexpr int TILE_WAVES = 8;

template <typename T> struct row4;        // 4 consecutive elements of a row as fp32
template <> struct row4<float> {
  __device__ static inline void load(const float* p, bool vec, float (&v)[4]) {
    if (vec) {
      const float4 x = *(const float4*)p;
      v[0] = x.x; v[1] = x.y; v[2] = x.z; v[3] = x.w;
    } else {
#pragma unroll
      for (int i = 0; i < 4; ++i) v[i] = p[i];
    }
  }
};
template <> struct row4<bf16_t> {
  __device__ static inline void load(const bf16_t* p, bool vec, float (&v)[4]) {
    if (vec) {
      const uint2 x = *(const uint2*)p;
      v[0] = __uint_as_float(x.x << 16); v[1] = __uint_as_float(x.x & 0xffff0000u);
      v[2] = __uint_as_float(x.y << 16); v[3] = __uint_as_float(x.y & 0xffff0000u);
    } else {
#pragma unroll
      for (int i = 0; i < 4; ++i) v[i] = bf16_to_f32(p[i]);
    }
  }
};
template <> struct row4<f16_t> {
  __device__ static inline void load(const f16_t* p, bool, float (&v)[4]) {
#pragma unroll
    for (int i = 0; i < 4; ++i) v[i] = (float)p[i];
  }
};

template <typename T, int DH>
__global__ __launch_bounds__(TILE_WAVES * 64) void mvpa_f32_tile_kernel(mvpa_fwd_args a, int vec_ok) {
  constexpr int HD = DH / 2;                // head dims of a lane: hh = 0 the first half, 1 the second
  constexpr int MT = (DH + 31) / 32;        // 32-wide output tiles
  extern __shared__ float smem[];

  const int tid = threadIdx.x, lane = tid & 63, ln = lane & 31, hh = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int T_ = a.T, C_ = a.C, N = a.T * a.C;
  const int b = blockIdx.y / a.H, h = blockIdx.y % a.H;
  const int g = h / (a.H / a.Hkv);
  const bool causal = a.flags & MVPA_FLAG_CAUSAL;
  const bool has_content = a.flags & MVPA_FLAG_CONTENT;
  const bool has_time = a.flags & MVPA_FLAG_TIME_BIAS;
  const bool has_chan = a.flags & MVPA_FLAG_CHAN_BIAS;
  const bool last_only = a.flags & MVPA_FLAG_LAST_STEP;
  const bool vec = vec_ok != 0;
  const int Nq = last_only ? C_ : N;
  const int q0 = blockIdx.x * 32;
  const int rq = min(q0 + ln, Nq - 1);      // rows past the end repeat the last one and are not stored
  const int base = last_only ? (T_ - 1) * C_ : 0;
  const int nq = base + rq;
  const int tq = nq / C_, cq = nq - tq * C_;
  const int tq_lo = (base + q0) / C_;
  const int tq_hi = (base + min(q0 + 31, Nq - 1)) / C_;

  const T* qrow = (const T*)a.q + b * a.q_stride_b + h * a.q_stride_h + (int64_t)rq * a.q_stride_n + hh * HD;
  const T* kbase = (const T*)a.k + b * a.k_stride_b + g * a.k_stride_h;
  const T* vbase = (const T*)a.v + b * a.v_stride_b + g * a.v_stride_h;
  const uint8_t* valid = a.chan_valid ? a.chan_valid + (int64_t)b * C_ : nullptr;
  const float* kbias = a.key_bias ? a.key_bias + (int64_t)b * N : nullptr;

  // tables: rows [0, nt32) of distance |tq - tk|, then rows of distance |cq - ck|, 32 queries each
  const int nt = has_time ? tq_hi + 1 : 0, nt32 = (nt + 31) & ~31;
  const int nc = has_chan ? C_ : 0, nc32 = (nc + 31) & ~31;
  float* St = smem;
  float* Sc = smem + nt32 * 32;

  float q[HD];
#pragma unroll
  for (int i = 0; i < HD; i += 4) {
    float v[4];
    row4<T>::load(qrow + i, vec, v);
#pragma unroll
    for (int e = 0; e < 4; ++e) q[i + e] = v[e];
  }
  for (int t = wave; t < (nt32 + nc32) / 32; t += TILE_WAVES) {
    const bool is_t = t < nt32 / 32;
    const int dist = (is_t ? t : t - nt32 / 32) * 32 + ln;
    const int row = is_t ? max(T_ - 1 - dist, 0) : max(C_ - 1 - dist, 0);
    const T* tab = (const T*)(is_t ? a.k_time : a.k_chan) + ((int64_t)g * (is_t ? T_ : C_) + row) * DH + hh * HD;
    const T* bias = (const T*)(is_t ? a.bias_v : a.bias_z) + g * DH + hh * HD;
    gen_f32x16 acc;
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[r] = 0.f;
#pragma unroll
    for (int i = 0; i < HD; i += 4) {
      float x[4], y[4];
      row4<T>::load(tab + i, vec, x);
      row4<T>::load(bias + i, vec, y);
#pragma unroll
      for (int e = 0; e < 4; ++e) acc = __builtin_amdgcn_mfma_f32_32x32x2f32(x[e], q[i + e] + y[e], acc, 0, 0, 0);
    }
#pragma unroll
    for (int r = 0; r < 16; ++r) smem[(t * 32 + (r >> 2) * 8 + hh * 4 + (r & 3)) * 32 + ln] = acc[r];
  }
#pragma unroll
  for (int i = 0; i < HD; i += 4) {
    float y[4];
    row4<T>::load((const T*)a.bias_u + g * DH + hh * HD + i, vec, y);
#pragma unroll
    for (int e = 0; e < 4; ++e) q[i + e] += y[e];
  }
  __syncthreads();

  const int hi = (causal && !last_only) ? (tq_hi + 1) * C_ : N;
  float m = -INFINITY, l = 0.f;
  gen_f32x16 acc[MT];
#pragma unroll
  for (int t = 0; t < MT; ++t)
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[t][r] = 0.f;

  for (int k0 = wave * 32; k0 < hi; k0 += TILE_WAVES * 32) {
    // V first: 16 rows of this half of the tile per output tile, in flight under the scores
    float vf[MT][16];
#pragma unroll
    for (int t = 0; t < MT; ++t)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int nk = min(k0 + (r >> 2) * 8 + hh * 4 + (r & 3), N - 1), d = t * 32 + ln;
        vf[t][r] = d < DH ? io<T>::load(vbase + (int64_t)nk * a.v_stride_n + d) : 0.f;
      }
    // content product, unless every pair of the tile is outside the window
    const int tk_lo = k0 / C_, tk_hi = min(k0 + 31, N - 1) / C_;
    const bool near = has_content && (a.window <= 0 || tq_hi == T_ - 1 ||
                                      (tq_lo - tk_hi <= a.window && tk_lo - tq_hi <= a.window));
    gen_f32x16 s;
#pragma unroll
    for (int r = 0; r < 16; ++r) s[r] = 0.f;
    if (near) {
      const T* krow = kbase + (int64_t)min(k0 + ln, N - 1) * a.k_stride_n + hh * HD;
#pragma unroll
      for (int i = 0; i < HD; i += 4) {
        float x[4];
        row4<T>::load(krow + i, vec, x);
#pragma unroll
        for (int e = 0; e < 4; ++e) s = __builtin_amdgcn_mfma_f32_32x32x2f32(x[e], q[i + e], s, 0, 0, 0);
      }
    }
    float tmax = -INFINITY;
    int tk = (k0 + hh * 4) / C_, ck = (k0 + hh * 4) - tk * C_;   // key of accumulator row 0, advanced below
    int prev = 0;
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const int off = (r >> 2) * 8 + (r & 3);
      ck += off - prev;
      prev = off;
      while (ck >= C_) {
        ck -= C_;
        ++tk;
      }
      const int nk = k0 + hh * 4 + off;
      const bool vis = nk < hi && causal_visible(tq, tk, causal) && (!valid || valid[ck] != 0);
      float x = -INFINITY;
      if (vis) {
        x = (has_time ? St[(tq - tk) * 32 + ln] : 0.f);
        if (has_chan) {
          const int dc = cq - ck;
          x += Sc[(dc < 0 ? -dc : dc) * 32 + ln];
        }
        if (has_content && content_kept(tq, tk, T_, a.window)) x += s[r];
        x *= a.sm_scale;
        if (kbias) x += kbias[nk];
      }
      s[r] = x;
      tmax = fmaxf(tmax, x);
    }
    tmax = fmaxf(tmax, __shfl_xor(tmax, 32));
    const float m_new = fmaxf(m, tmax);
    if (m_new > -INFINITY) {
      const float alpha = (m == -INFINITY) ? 0.f : expf(m - m_new);
      l *= alpha;
#pragma unroll
      for (int t = 0; t < MT; ++t)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[t][r] *= alpha;
      m = m_new;
    }
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      s[r] = (s[r] == -INFINITY) ? 0.f : expf(s[r] - m);
      l += s[r];
    }
#pragma unroll
    for (int t = 0; t < MT; ++t)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[t] = __builtin_amdgcn_mfma_f32_32x32x2f32(vf[t][r], s[r], acc[t], 0, 0, 0);
  }
  l += __shfl_xor(l, 32);                   // the two halves of a query's keys

  // merge of the waves' states: [wave][query] m, l and [wave][d][query] accumulators over the tables
  __syncthreads();
  float* Ml = smem;                                    // [waves][2][32]
  float* Ac = smem + TILE_WAVES * 64;                  // [waves][MT * 32][32]
  if (hh == 0) {
    Ml[wave * 64 + ln] = m;
    Ml[wave * 64 + 32 + ln] = l;
  }
#pragma unroll
  for (int t = 0; t < MT; ++t)
#pragma unroll
    for (int r = 0; r < 16; ++r)
      Ac[(wave * MT * 32 + t * 32 + (r >> 2) * 8 + hh * 4 + (r & 3)) * 32 + ln] = acc[t][r];
  __syncthreads();
  const int mq = tid & 31;                             // one query per lane, head dims over the rest
  float mm = -INFINITY;
#pragma unroll
  for (int w = 0; w < TILE_WAVES; ++w) mm = fmaxf(mm, Ml[w * 64 + mq]);
  float wgt[TILE_WAVES], ll = 0.f;
#pragma unroll
  for (int w = 0; w < TILE_WAVES; ++w) {
    const float mw = Ml[w * 64 + mq];
    wgt[w] = mw == -INFINITY ? 0.f : expf(mw - mm);
    ll += wgt[w] * Ml[w * 64 + 32 + mq];
  }
  const int row = q0 + mq;
  if (row >= Nq) return;
  const float inv = 1.f / ll;
  T* orow = (T*)a.o + b * a.o_stride_b + h * a.o_stride_h + (int64_t)row * a.o_stride_n;
  for (int d = tid >> 5; d < DH; d += TILE_WAVES * 2) {
    float v = 0.f;
#pragma unroll
    for (int w = 0; w < TILE_WAVES; ++w) v += wgt[w] * Ac[(w * MT * 32 + d) * 32 + mq];
    io<T>::store(orow + d, v * inv);
  }
  if (a.lse && tid < 32) a.lse[((int64_t)b * a.H + h) * Nq + row] = (mm + logf(ll)) * kLog2e;
}

__global__ void mvpa_debug_maps_kernel(int T_, int C_, int window, unsigned flags,
                                       const uint8_t* valid, int32_t* time_idx,
                                       int32_t* chan_idx, uint8_t* mask_bits) {
  const int N = T_ * C_;
  const int nk = blockIdx.x * blockDim.x + threadIdx.x;
  const int nq = blockIdx.y;
  if (nk >= N) return;
  const int tq = nq / C_, cq = nq % C_, tk = nk / C_, ck = nk % C_;
  const bool causal = flags & MVPA_FLAG_CAUSAL;
  const bool vis = causal_visible(tq, tk, causal) && (!valid || valid[ck] != 0);
  const bool kept = (flags & MVPA_FLAG_CONTENT) && content_kept(tq, tk, T_, window);
  const int64_t i = (int64_t)nq * N + nk;
  time_idx[i] = tk <= tq ? time_row(tq, tk, T_) : -1;
  chan_idx[i] = chan_row(cq, ck, C_);
  mask_bits[i] = (uint8_t)((vis ? 1 : 0) | (kept ? 2 : 0));
}

template <typename T, int DH>
static int launch_generic_t(const mvpa_fwd_args* a, hipStream_t stream) {
  const int rows = (a->flags & MVPA_FLAG_LAST_STEP) ? a->C : a->T * a->C;
  // the matrix-instruction kernel wherever its two tables (128 bytes per distance) fit the LDS, i.e.
  // up to about 1200 time steps and channels together; beyond that one lane per row
  const size_t tables = (size_t)(((a->T + 31) & ~31) + ((a->C + 31) & ~31)) * 32 * sizeof(float);
  const size_t merge = (size_t)TILE_WAVES * (64 + (DH + 31) / 32 * 1024) * sizeof(float);
  const size_t tile_lds = tables > merge ? tables : merge;
  if (tile_lds <= 156 * 1024) {
    const uintptr_t p = (uintptr_t)a->q | (uintptr_t)a->k | (uintptr_t)a->k_time | (uintptr_t)a->k_chan |
                        (uintptr_t)a->bias_u | (uintptr_t)a->bias_v | (uintptr_t)a->bias_z;
    const int64_t st = a->q_stride_b | a->q_stride_h | a->q_stride_n | a->k_stride_b | a->k_stride_h | a->k_stride_n;
    const int vec_ok = (p % (4 * sizeof(T))) == 0 && (st & 3) == 0;
    auto tk = mvpa_f32_tile_kernel<T, DH>;
    mvpa::want_dynamic_lds((const void*)tk, (int)tile_lds);
    MVPA_LAUNCH(tk, dim3((rows + 31) / 32, a->B * a->H), dim3(TILE_WAVES * 64), tile_lds, stream, *a, vec_ok);
    return mvpa::take_launch_status();
  }
  const size_t base = (size_t)(2 * GEN_KT * DH + GEN_KT * GEN_THREADS) * sizeof(float);
  const size_t table = (size_t)GEN_THREADS * (a->C + 1) * sizeof(float);
  const int chan_table = (base + table <= 150 * 1024) ? 1 : 0;
  const size_t lds = base + (chan_table ? table : 0);
  auto kern = mvpa_generic_kernel<T, DH>;
  mvpa::want_dynamic_lds((const void*)kern, (int)lds);
  dim3 grid((rows + GEN_THREADS - 1) / GEN_THREADS, a->B * a->H);
  MVPA_LAUNCH(kern, grid, dim3(GEN_THREADS), lds, stream, *a, chan_table);
  return mvpa::take_launch_status();
}

template <typename T>
static int launch_generic_dh(const mvpa_fwd_args* a, hipStream_t stream) {
  switch (a->Dh) {
    case 16: return launch_generic_t<T, 16>(a, stream);
    case 32: return launch_generic_t<T, 32>(a, stream);
    case 64: return launch_generic_t<T, 64>(a, stream);
    case 128: return launch_generic_t<T, 128>(a, stream);
  }
  return MVPA_ERR_HEAD_DIM;
}

}  // namespace mvpa

int mvpa_launch_generic(const mvpa_fwd_args* a, hipStream_t stream) {
  if (a->dtype == MVPA_F32) return mvpa::launch_generic_dh<float>(a, stream);
  if (a->dtype == MVPA_BF16) return mvpa::launch_generic_dh<mvpa::bf16_t>(a, stream);
  if (a->dtype == MVPA_F16) return mvpa::launch_generic_dh<mvpa::f16_t>(a, stream);
  return MVPA_ERR_DTYPE;
}

extern "C" int mvpa_debug_maps(int32_t T, int32_t C, int32_t window, uint32_t flags,
                               const uint8_t* chan_valid, int32_t* time_idx, int32_t* chan_idx,
                               uint8_t* mask_bits, void* stream) {
  if (!time_idx || !chan_idx || !mask_bits) return MVPA_ERR_NULL;
  if (T <= 0 || C <= 0) return MVPA_ERR_CTX;
  const int N = T * C;
  dim3 grid((N + 255) / 256, N);
  MVPA_LAUNCH(mvpa::mvpa_debug_maps_kernel, grid, dim3(256), 0, (hipStream_t)stream, T, C,
                     window, flags, chan_valid, time_idx, chan_idx, mask_bits);
  return mvpa::take_launch_status();
}
