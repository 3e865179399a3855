// MVPA forward for launches that do not fill the chip (bf16 or fp16): one decoding step, a short window.
//
// The tiled kernel of mvpa_mfma.hip lets a wave walk every key step of its queries behind a shared tile
// ring; with a few hundred query tiles in all, a launch lasts as long as that chain (25 steps x 0.8 us and
// 5 us of set-up for one window of 25 segments), whatever idles beside it.  Here the keys of ONE query
// tile - 32 channels of one time step - are dealt to the 8 waves of a workgroup, 32 keys at a time, each
// wave with a soft-max state of its own; the states are merged through LDS at the end.  Nothing is
// shared while the waves run, so there is no barrier between set-up and merge: a wave's K and V tiles go
// through 2 x 32 rows of LDS of its own, the next tile's are on their way while a tile is multiplied.
// Everything comes from memory as whole rows and becomes fragments on its way out of LDS - a fragment
// load straight from global memory touches 32 lines for one KiB, at about two cycles each (q, bias and
// table rows loaded that way took 8 us of a launch).  Arithmetic, roundings and operand layouts are
// those of mvpa_mfma.hip; steps outside the content window skip K and the product with it.
// Bound: the latency of set-up, of one or a few tiles per wave, and of the merge.  What hides it is a second
// workgroup on the CU, so head sizes up to 64 keep to 128 registers (at 64 one of them spills: 8 bytes of scratch a
// lane) and 80 KB (tables of up to 64 rows): (q + u),
// (q + v), (q + z) are formed once for all waves and stay in LDS, table rows go there directly, and addresses of a
// tile are one register each.  With 165 registers, one workgroup a CU, B1 H12 Hkv4 C21 T25 Dh64 took two rounds of
// an XCD's 32 CUs: 12.1 -> 9.9 us; C21 T64 23 -> 20.
#include "mvpa_mfma_tools.h"

namespace mvpa {

constexpr int WV_WAVES = 8;

template <int DH>
struct wave_cfg {
  static constexpr int KS = DH / 16, MT = DH / 32, ROWB = DH * 2, CHUNKS = DH / 8;
  static constexpr int TILE = 32 * ROWB, KV = 2 * TILE;           // one wave's K tile, then its V tile
  static constexpr int Q_BYTES = 32 * ROWB;                       // (q + u) * scale
  static constexpr int MERGE = WV_WAVES * (64 + DH * 33) * 4;     // m, l and accumulators of every wave
};

template <int DH, typename E>
__global__ __launch_bounds__(WV_WAVES * 64, DH == 128 ? 2 : 4) void mvpa_wave_kernel(mvpa_fwd_args a, step_geom geo) {
  using x8 = typename E::x8;
  using x4 = typename E::x4;
  using x2 = typename E::x2;
  using G = wave_cfg<DH>;
  constexpr int KS = G::KS, MT = G::MT, ROWB = G::ROWB, CHUNKS = G::CHUNKS;
  extern __shared__ __attribute__((aligned(1024))) unsigned char wv_lds[];

  const int tid = threadIdx.x, lane = tid & 63, ln = lane & 31, hh = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int C_ = a.C, W = a.window, nbh = a.B * a.H;
  const bool last_only = a.flags & MVPA_FLAG_LAST_STEP;
  const bool has_content = a.flags & MVPA_FLAG_CONTENT;
  const bool has_time = a.flags & MVPA_FLAG_TIME_BIAS;
  const bool has_chan = a.flags & MVPA_FLAG_CHAN_BIAS;
  const int qt = (C_ + 31) >> 5;                                  // query (and key) tiles of a time step

  // workgroup -> (b, h), query tile, and time step (latest = longest first) or run of key steps
  int bg, r2;
  if (!step_block(geo, bg, r2)) return;
  const int item = blockIdx.y, hg = qt == 1 ? item : qt == 2 ? item >> 1 : qt == 4 ? item >> 2 : (item * 43691) >> 17;
  const int tile = item - hg * qt;
  const int b = a.B == 1 ? 0 : bg / a.Hkv, g = bg - b * a.Hkv, h = g * geo.grp + hg, bh = b * a.H + h;
  const int n_split = last_only ? geo.runs : 1;
  const int run = last_only ? r2 : 0, t_lo = run * geo.len;
  const int tq = last_only ? a.T - 1 : a.T - 1 - r2;
  const int steps = last_only ? min(geo.len, a.T - t_lo) : tq + 1;
  const int cq = tile * 32 + ln;
  const bool ring = a.flags & MVPA_FLAG_RING;
  const int ring_rot = ring ? a.T - 1 - __builtin_amdgcn_readfirstlane(*a.ring_head) : 0;

  const bf16_t* qbase = (const bf16_t*)a.q + b * a.q_stride_b + h * a.q_stride_h +
                        (int64_t)(last_only ? 0 : tq * C_) * a.q_stride_n;
  const bf16_t* kbase = (const bf16_t*)a.k + b * a.k_stride_b + g * a.k_stride_h + (int64_t)t_lo * C_ * a.k_stride_n;
  const bf16_t* vbase = (const bf16_t*)a.v + b * a.v_stride_b + g * a.v_stride_h + (int64_t)t_lo * C_ * a.v_stride_n;
  const bf16_t* ktime = (const bf16_t*)a.k_time + (int64_t)g * a.T * DH;
  const bf16_t* kchan = (const bf16_t*)a.k_chan + (int64_t)g * C_ * DH;
  const uint8_t* valid = a.chan_valid ? a.chan_valid + (int64_t)b * C_ : nullptr;
  const float sc2 = a.sm_scale * kLog2e;

  // a wave keeps one key tile of the time step and takes every spr-th step (three tiles count as four)
  const int qt2 = qt <= 2 ? qt : 4;
  const int ct = wave & (qt2 - 1), spr = WV_WAVES / qt2;
  const int n_units = ct < qt ? steps : 0;
  // first step that keeps the content term (every step of the last time step does)
  const int near0 = !has_content ? a.T : (W <= 0 || tq == a.T - 1) ? 0 : max(0, tq - W);

  // 16-byte chunk i of a 32-row tile for this lane: row (64 i + lane) / CHUNKS, and where K / V rows keep it
  constexpr int NL = DH / 16;
  const auto row_of = [&](int i) { return (i * 64 + lane) / CHUNKS; };
  const auto chunk_of = [&](int i) { return (i * 64 + lane) % CHUNKS; };
  // bytes from the step's first row to this lane's chunk 0, and to the last row's; the NL chunks lie RPL rows apart
  constexpr int RPL = 64 / CHUNKS;
  uint32_t koff = (uint32_t)((ct * 32 + row_of(0)) * (int)a.k_stride_n + chunk_of(0) * 8) * 2u;
  uint32_t voff = (uint32_t)((ct * 32 + row_of(0)) * (int)a.v_stride_n + chunk_of(0) * 8) * 2u;
  uint32_t kend = (uint32_t)((C_ - 1) * (int)a.k_stride_n + chunk_of(0) * 8) * 2u;
  uint32_t vend = (uint32_t)((C_ - 1) * (int)a.v_stride_n + chunk_of(0) * 8) * 2u;
  u32x4 kr[NL], vr[NL];
  auto request = [&](int s) {
    asm volatile("" : "+v"(koff), "+v"(voff), "+v"(kend), "+v"(vend));   // (no 64-bit addresses held over the loop)
    if (s >= near0) {
      const char* ks = (const char*)(kbase + (int64_t)s * C_ * a.k_stride_n);
#pragma unroll
      for (int i = 0; i < NL; ++i) kr[i] = *(const u32x4*)(ks + min(koff + i * RPL * 2u * (uint32_t)a.k_stride_n, kend));
    }
    const char* vs = (const char*)(vbase + (int64_t)s * C_ * a.v_stride_n);
#pragma unroll
    for (int i = 0; i < NL; ++i) vr[i] = *(const u32x4*)(vs + min(voff + i * RPL * 2u * (uint32_t)a.v_stride_n, vend));
  };
  unsigned char* kl = wv_lds + wave * G::KV;
  unsigned char* vl = kl + G::TILE;
  auto put_k = [&](const u32x4 (&r)[NL]) {
#pragma unroll
    for (int i = 0; i < NL; ++i) *(u32x4*)(kl + row_of(i) * ROWB + ((chunk_of(i) ^ swz_k<DH>(row_of(i))) << 4)) = r[i];
  };
  // fragment ks of row ln: the chunk's bits lie above the row's, so one address serves all (k_frag ^ ks << 5)
  int k_frag = ln * ROWB + ((hh ^ swz_k<DH>(ln)) << 4);

  // ---- set-up.  Requests, in the order of their use: a chunk of the tile's q rows and of the three bias vectors
  // per thread, the table rows of the wave's first 32-row tile, the wave's first K and V tiles.
  constexpr int QCH = 32 * CHUNKS, QN = (QCH + WV_WAVES * 64 - 1) / (WV_WAVES * 64);
  static_assert(QN == 1, "a chunk of q per thread");
  const int q_row = min(tid / CHUNKS, 31), q_chunk = tid % CHUNKS;
  const u32x4 q_raw = *(const u32x4*)(qbase + (int64_t)min(tile * 32 + q_row, C_ - 1) * a.q_stride_n + q_chunk * 8);
  const u32x4 u_raw = *(const u32x4*)((const bf16_t*)a.bias_u + g * DH + q_chunk * 8);
  const u32x4 v_raw = *(const u32x4*)((const bf16_t*)a.bias_v + g * DH + q_chunk * 8);
  const u32x4 z_raw = *(const u32x4*)((const bf16_t*)a.bias_z + g * DH + q_chunk * 8);
  const int ch_rows = qt * 32, n_tasks = qt + (steps + 31) / 32;
  const uint32_t kl0 = (uint32_t)(uintptr_t)(LDS_PTR(unsigned char))wv_lds + wave * G::KV;
  auto request_rows = [&](int t) {                  // 32 table rows into the wave's K tile: channel tiles first, then time tiles
#pragma unroll
    for (int i = 0; i < NL; ++i) {
      const int tr = row_of(i);
      const bf16_t* row;
      if (t < qt) {
        row = kchan + (int64_t)min(t * 32 + tr, C_ - 1) * DH;
      } else {
        const int r = (t - qt) * 32 + tr;
        int j = last_only ? t_lo + r : time_row(tq, r, a.T);
        j += ring_rot;
        if (ring && j >= a.T) j -= a.T;
        row = ktime + (int64_t)min(j, a.T - 1) * DH;              // rows past the run: never used
      }
      load_to_lds_16(row + (chunk_of(i) ^ swz_k<DH>(tr)) * 8, kl0 + i * 1024);
    }
  };
  if (wave < n_tasks) request_rows(wave);
  int s = wave / qt2;
  if (s < n_units) request(s);
  __builtin_amdgcn_sched_barrier(0);
  // (q + bias) * scale of the tile, once for all waves: u for the key tiles; v and z, which the tables alone
  // need, where the first two waves will keep their V tiles
  unsigned char* ql = wv_lds + WV_WAVES * G::KV;
  unsigned char* qv = wv_lds + G::TILE;
  unsigned char* qz = qv + G::KV;
  if (QCH == WV_WAVES * 64 || tid < QCH) {
    const int at = q_row * ROWB + ((q_chunk ^ swz_k<DH>(q_row)) << 4);
    float f[8];
    E::unpack(q_raw, f);
    *(x8*)(ql + at) = qfrag_fma<E>(f, u_raw, sc2);
    *(x8*)(qv + at) = qfrag_fma<E>(f, v_raw, sc2);
    *(x8*)(qz + at) = qfrag_fma<E>(f, z_raw, sc2);
  }
  lds_barrier();
  float* Sc = (float*)(ql + G::Q_BYTES);
  float* St = Sc + ch_rows * 32;
  for (int t = wave; t < n_tasks; t += WV_WAVES) {
    const bool chan = t < qt;
    if (t != wave) request_rows(t);
    wait_vmcnt_imm<0>();
    wave_lds_sync();
    f32x16 acc;
#pragma unroll
    for (int i = 0; i < 16; ++i) acc[i] = 0.f;
    if (chan ? has_chan : has_time) {
#pragma unroll
      for (int ks = 0; ks < KS; ++ks)
        acc = E::mfma(*(const x8*)(kl + (k_frag ^ (ks << 5))), *(const x8*)((chan ? qz : qv) + (k_frag ^ (ks << 5))), acc, 0, 0, 0);
    }
    wave_lds_sync();
    float* dst = (chan ? Sc : St) + (chan ? t : t - qt) * 1024 + ln;
#pragma unroll
    for (int i = 0; i < 16; ++i) dst[((i >> 2) * 8 + hh * 4 + (i & 3)) * 32] = acc[i];
  }
  uint32_t kbits;                                   // bit 8(i/4) + i%4: this lane's key i exists and is present
  {
    const int ck = ct * 32 + ln;
    bool ok = ck < C_;
    if (valid) ok = ok && valid[min(ck, C_ - 1)] != 0;
    kbits = (uint32_t)__ballot(ok) >> (4 * hh);
  }
  lds_barrier();
  f32x16 Bc;
#pragma unroll
  for (int i = 0; i < 16; ++i) {
    const int d = cq - (ct * 32 + (i >> 2) * 8 + hh * 4 + (i & 3));
    const int dist = min(d < 0 ? -d : d, C_ - 1);   // (clamped only for padded queries and keys)
    const float v = Sc[(C_ - 1 - dist) * 32 + ln];
    Bc[i] = ((kbits >> ((i >> 2) * 8 + (i & 3))) & 1u) ? v : -INFINITY;
  }

  // ---- the wave's key tiles
  int v_frag;                                       // of output tile mt: v_frag ^ mt << 6
  {
    const int e = (ln & 15) >> 2, aa = ln & 3, grp = ln >> 4, row0 = 4 * hh + e;
    v_frag = row0 * ROWB + (((2 * grp + (aa >> 1)) ^ swz_v<DH>(row0)) << 4) + ((aa & 1) << 3);
  }
  float m_run = kMFloor, l_run = 0.f;
  f32x16 acc[MT];
#pragma unroll
  for (int mt = 0; mt < MT; ++mt)
#pragma unroll
    for (int i = 0; i < 16; ++i) acc[mt][i] = 0.f;

  for (; s < n_units; s += spr) {
    const bool near = s >= near0;
    asm volatile("" : "+v"(k_frag), "+v"(v_frag));   // (addresses formed where they are used: 128 registers)
    if (near) put_k(kr);
#pragma unroll
    for (int i = 0; i < NL; ++i) *(u32x4*)(vl + row_of(i) * ROWB + ((chunk_of(i) ^ swz_v<DH>(row_of(i))) << 4)) = vr[i];
    if (s + spr < n_units) request(s + spr);
    wave_lds_sync();
    f32x16 S = Bc;
    if (near) {
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) S = E::mfma(*(const x8*)(kl + (k_frag ^ (ks << 5))), *(const x8*)(ql + (k_frag ^ (ks << 5))), S, 0, 0, 0);
    }
    const float st = St[s * 32 + ln];
    float rmax = -INFINITY;
#pragma unroll
    for (int i = 0; i < 16; ++i) rmax = fmaxf(rmax, S[i]);
    const float cand = xhalf_max(rmax) + st;
    if (__ballot(cand > m_run + 8.f) != 0ull) {     // lazy reference point, as in mvpa_mfma.hip
      const float m_new = fmaxf(m_run, cand), alpha = fast_exp2(m_run - m_new);
      m_run = m_new;
      l_run *= alpha;
#pragma unroll
      for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (int i = 0; i < 16; ++i) acc[mt][i] *= alpha;
    }
    const float off = st - m_run;
#pragma unroll
    for (int i = 0; i < 16; ++i) S[i] = fast_exp2(S[i] + off);
    x8 P[2] = {E::pack(S, 0), E::pack(S, 8)};
#pragma unroll
    for (int p = 0; p < 2; ++p) {
      union { x8 v; x2 q[4]; } u;
      u.v = P[p];
#pragma unroll
      for (int j = 0; j < 4; ++j) l_run = E::add_pair(u.q[j], l_run);
    }
#pragma unroll
    for (int p = 0; p < 2; ++p)
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) {
        const unsigned char* vp = vl + (v_frag ^ (mt << 6)) + 16 * p * ROWB;
        const x4 lo = E::read_tr(vp), hi = E::read_tr(vp + 8 * ROWB);
        acc[mt] = E::mfma(__builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7), P[p], acc[mt], 0, 0, 0);
      }
    wave_lds_sync();
  }
  l_run += __shfl_xor(l_run, 32);                   // the two halves of the wave's keys

  // ---- merge: [wave][m | l][query], [wave][d][query] (pitch 33) over everything above
  lds_barrier();
  float* Ml = (float*)wv_lds;
  float* Ac = Ml + WV_WAVES * 64;
  if (hh == 0) {
    Ml[wave * 64 + ln] = m_run;
    Ml[wave * 64 + 32 + ln] = l_run;
  }
#pragma unroll
  for (int mt = 0; mt < MT; ++mt)
#pragma unroll
    for (int i = 0; i < 16; ++i) Ac[(wave * DH + mt * 32 + (i >> 2) * 8 + hh * 4 + (i & 3)) * 33 + ln] = acc[mt][i];
  lds_barrier();
  const int mq = tid >> 4, cm = tile * 32 + mq;     // 16 threads per query, DPT head dims each: whole rows leave
  float m = kMFloor, w[WV_WAVES], l = 0.f;
#pragma unroll
  for (int i = 0; i < WV_WAVES; ++i) m = fmaxf(m, Ml[i * 64 + mq]);
#pragma unroll
  for (int i = 0; i < WV_WAVES; ++i) {
    w[i] = fast_exp2(Ml[i * 64 + mq] - m);
    l += w[i] * Ml[i * 64 + 32 + mq];
  }
  if (cm >= C_) return;
  const float inv = 1.f / l;
  const int64_t n = (last_only ? 0 : (int64_t)tq * C_) + cm;
  const int64_t prow = ((int64_t)run * nbh + bh) * C_ + cm;       // row of the split workspace
  bf16_t* orow = n_split > 1 ? (bf16_t*)a.split_ws + prow * DH
                             : (bf16_t*)a.o + b * a.o_stride_b + h * a.o_stride_h + n * a.o_stride_n;
  constexpr int DPT = DH / 16;                      // head dims per thread
  const int d0 = (tid & 15) * DPT;
  typedef decltype(E::cvt(0.f)) el;
  el o[DPT];
#pragma unroll
  for (int d = 0; d < DPT; ++d) {
    float v = 0.f;
#pragma unroll
    for (int i = 0; i < WV_WAVES; ++i) v += w[i] * Ac[(i * DH + d0 + d) * 33 + mq];
    o[d] = E::cvt(v * inv);
  }
  __builtin_memcpy(orow + d0, o, sizeof(o));
  if ((tid & 15) == 0) {
    const float lse = m + log2f(l);
    if (n_split > 1) ((float*)((bf16_t*)a.split_ws + (int64_t)n_split * nbh * C_ * DH))[prow] = lse;
    else if (a.lse) a.lse[(int64_t)bh * (last_only ? (int64_t)C_ : (int64_t)a.T * C_) + n] = lse;
  }
}

template <int DH, typename E>
static int launch_wave_t(const mvpa_fwd_args* a, int lds, hipStream_t stream) {
  auto kern = mvpa_wave_kernel<DH, E>;
  want_dynamic_lds((const void*)kern, lds);
  const bool last = a->flags & MVPA_FLAG_LAST_STEP;
  const int n_split = last && a->n_split > 1 ? a->n_split : 1;
  const int grp = a->H / a->Hkv;
  step_geom geo = make_step_geom(a->B * a->Hkv, grp, last ? n_split : a->T, a->T);
  MVPA_LAUNCH(kern, step_grid(geo, grp * ((a->C + 31) / 32)), dim3(WV_WAVES * 64), lds, stream, *a, geo);
  return take_launch_status();
}

static int wave_lds_bytes(const mvpa_fwd_args* a) {
  const int steps = (a->flags & MVPA_FLAG_LAST_STEP) && a->n_split > 1 ? (a->T + a->n_split - 1) / a->n_split : a->T;
  const int rows = (a->C + 31) / 32 * 32 + (steps + 31) / 32 * 32;
  const int run = (WV_WAVES * 64 + 32) * a->Dh * 2 + rows * 128, merge = WV_WAVES * (64 + a->Dh * 33) * 4;
  return run > merge ? run : merge;
}

}  // namespace mvpa

// Shapes: those of the tiled kernel, without the fp8 content term, as long as the tables fit the LDS.
int mvpa_wave_supported(const mvpa_fwd_args* a) {
  const int64_t row = a->k_stride_n > a->v_stride_n ? a->k_stride_n : a->v_stride_n;
  return mvpa_mfma_supported(a) && !(a->flags & MVPA_FLAG_FP8_QK) && mvpa::wave_lds_bytes(a) <= 160 * 1024 &&
         row < ((int64_t)1 << 24);                 // 128 rows of a step, padded ones too, in 32 bits of bytes
}

int mvpa_launch_wave(const mvpa_fwd_args* a, hipStream_t stream) {
  using namespace mvpa;
  const int lds = wave_lds_bytes(a);
  const bool f16 = a->dtype == MVPA_F16;
  switch (a->Dh) {
    case 32: return f16 ? launch_wave_t<32, el_f16>(a, lds, stream) : launch_wave_t<32, el_bf16>(a, lds, stream);
    case 64: return f16 ? launch_wave_t<64, el_f16>(a, lds, stream) : launch_wave_t<64, el_bf16>(a, lds, stream);
    case 128: return f16 ? launch_wave_t<128, el_f16>(a, lds, stream) : launch_wave_t<128, el_bf16>(a, lds, stream);
  }
  return MVPA_ERR_UNSUPPORTED;
}
