// MVPA forward of one decoding step for 65..128 channels, its key steps cut into runs (bf16 or fp16).
//
// A workgroup is one run of key steps of one (b, h), 8 waves: four tiles of 32 queries x two halves of the
// 128 (padded) keys of a step, two waves per SIMD.  The wave-split kernel (mvpa_wave.hip) would read every
// K and V row four times here, once per query tile, and is bound by that traffic; the tiled kernel
// (mvpa_mfma.hip) reads them once but spends 20 us setting up for a run that takes 7.  This one keeps the
// shared ring and takes the set-up once through LDS: q, bias and table rows arrive as whole rows by
// direct-to-LDS loads (the same fragments loaded from global memory touch 32 lines per KiB: 56 such loads
// per wave took 8 us), each wave forms two 32-row tiles of the channel table and its share of the time
// table (the whole run's: no slabs later on).
//   LDS: the rows wait in the last stage of the ring, the channel tables of the four query tiles (64 KB) are
//   written over the other stages; step 0 goes into the last stage while the tables are gathered from.
//   DH 128: two stages of 64 KB, DH 64: three of 32 KB.
// Arithmetic, roundings and layouts as in mvpa_mfma.hip.
// B1 H16 Hkv8 C128 T110 Dh128 in 16 runs: 43 -> 25 us without the merge, a chain: 2.5 to the rows, 6 of tables and the first step's way,
// 1.8 a step (on 128 workgroups as on 256: products, exponentials and what lies between them, not memory), 4 of merge and stores.
#include "mvpa_mfma_tools.h"

#include <type_traits>

namespace mvpa {

typedef __attribute__((ext_vector_type(4))) float f32x4;

template <int DH>
struct step_cfg {
  static constexpr int KS = DH / 16, MT = DH / 32, ROWB = DH * 2, CHUNKS = DH / 8;
  static constexpr int TILE = 128 * ROWB, STAGE = 2 * TILE;       // K rows, then V rows
  static constexpr int TABLE = 4 * 128 * 32 * 4;                  // [query tile][distance][query]
  static constexpr int R = TABLE / STAGE + 1;
  static constexpr int RING = R * STAGE;
  static constexpr int LPW = TILE / 1024 / 8;                     // 1 KiB loads per wave and tile
  static_assert(8 * (512 + MT * 2048 + 32 * (ROWB / 2 + 16)) <= RING, "merge buffer and output rows");
  static_assert(256 * ROWB <= STAGE, "q and channel-table rows fit a stage");
};

template <int DH, typename E>
__global__ __launch_bounds__(512, 2) void mvpa_step_kernel(mvpa_fwd_args a, step_geom geo) {
  using x8 = typename E::x8;
  using x4 = typename E::x4;
  using x2 = typename E::x2;
  using G = step_cfg<DH>;
  constexpr int KS = G::KS, MT = G::MT, ROWB = G::ROWB, CHUNKS = G::CHUNKS;
  extern __shared__ __attribute__((aligned(1024))) unsigned char sp_lds[];
  float* St = (float*)(sp_lds + G::RING);                         // [query tile][step][query]

  const int tid = threadIdx.x, lane = tid & 63, ln = lane & 31, hh = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int qt = wave & 3, kp = wave >> 2;
  const int C_ = a.C, nbh = a.B * a.H;
  const bool has_time = a.flags & MVPA_FLAG_TIME_BIAS, has_chan = a.flags & MVPA_FLAG_CHAN_BIAS;
  int bg, run;
  if (!step_block(geo, bg, run)) return;
  const int b = a.B == 1 ? 0 : bg / a.Hkv, g = bg - b * a.Hkv, h = g * geo.grp + blockIdx.y, bh = b * a.H + h;
  const int n_split = geo.runs, t_lo = run * geo.len, steps = min(geo.len, a.T - t_lo), steps32 = (steps + 31) & ~31;
  const int cq = qt * 32 + ln;
  const bool ring = a.flags & MVPA_FLAG_RING;
  const int ring_rot = ring ? a.T - 1 - __builtin_amdgcn_readfirstlane(*a.ring_head) : 0;
  const bf16_t* qbase = (const bf16_t*)a.q + b * a.q_stride_b + h * a.q_stride_h;
  const bf16_t* kbase = (const bf16_t*)a.k + b * a.k_stride_b + g * a.k_stride_h + (int64_t)t_lo * C_ * a.k_stride_n;
  const bf16_t* vbase = (const bf16_t*)a.v + b * a.v_stride_b + g * a.v_stride_h + (int64_t)t_lo * C_ * a.v_stride_n;
  const uint8_t* valid = a.chan_valid ? a.chan_valid + (int64_t)b * C_ : nullptr;
  const float sc2 = a.sm_scale * kLog2e;

  // ---- set-up rows to LDS: q and the channel table (128 rows each) into the last stage, time-table rows of
  // the run and the three bias vectors behind the time scores.  A wave load is 64 chunks of 16 bytes.
  const uint32_t lds0 = (uint32_t)(uintptr_t)(LDS_PTR(unsigned char))sp_lds;
  unsigned char* rows_q = sp_lds + (G::R - 1) * G::STAGE;
  unsigned char* rows_e = rows_q + 128 * ROWB;
  unsigned char* rows_t = (unsigned char*)(St + 4 * steps32 * 32);
  unsigned char* rows_b = rows_t + steps32 * ROWB;                // u, v, z: one wave load
  auto lds_of = [&](const unsigned char* p) { return lds0 + (uint32_t)(p - sp_lds); };
#pragma unroll
  for (int i = 0; i < G::LPW; ++i) {
    const int li = wave + 8 * i, pc = li * 64 + lane, row = pc / CHUNKS, c = ((pc % CHUNKS) ^ swz_k<DH>(row)) * 8;
    load_to_lds_16(qbase + (int64_t)min(row, C_ - 1) * a.q_stride_n + c, lds_of(rows_q) + li * 1024);
    load_to_lds_16((const bf16_t*)a.k_chan + ((int64_t)g * C_ + min(row, C_ - 1)) * DH + c, lds_of(rows_e) + li * 1024);
  }
  for (int li = wave; li < steps32 * ROWB / 1024; li += 8) {
    const int pc = li * 64 + lane, row = pc / CHUNKS, c = ((pc % CHUNKS) ^ swz_k<DH>(row)) * 8;
    int j = t_lo + row;
    if (ring) {
      j += ring_rot;
      j = j >= a.T ? j - a.T : j;
    }
    load_to_lds_16((const bf16_t*)a.k_time + ((int64_t)g * a.T + min(j, a.T - 1)) * DH + c, lds_of(rows_t) + li * 1024);
  }
  if (wave == 0) {
    const int pc = lane, row = min(pc / CHUNKS, 2), c = (pc % CHUNKS) * 8;
    const bf16_t* src = (const bf16_t*)(row == 0 ? a.bias_u : row == 1 ? a.bias_v : a.bias_z) + g * DH + c;
    load_to_lds_16(src, lds_of(rows_b));
  }

  // ---- the ring
  uint32_t koff[G::LPW], voff[G::LPW];
#pragma unroll
  for (int i = 0; i < G::LPW; ++i) {
    const int pc = (wave + 8 * i) * 64 + lane, row = pc / CHUNKS, phys = pc % CHUNKS, rc = min(row, C_ - 1);
    koff[i] = (uint32_t)(rc * (int)a.k_stride_n + ((phys ^ swz_k<DH>(row)) << 3)) * 2;
    voff[i] = (uint32_t)(rc * (int)a.v_stride_n + ((phys ^ swz_v<DH>(row)) << 3)) * 2;
  }
  const int64_t kstep = (int64_t)C_ * a.k_stride_n, vstep = (int64_t)C_ * a.v_stride_n;
  const bf16_t *ks_next = kbase, *vs_next = vbase;               // of the step requested next
  uint32_t dst = lds0 + (G::R - 1) * G::STAGE;
  auto request = [&](int i) {                                     // 2 LPW of them are a step
    if (i < G::LPW) load_to_lds_16(ks_next, koff[i < G::LPW ? i : 0], dst + (wave + 8 * i) * 1024);
    else load_to_lds_16(vs_next, voff[i < G::LPW ? 0 : i - G::LPW], dst + G::TILE + (wave + 8 * (i - G::LPW)) * 1024);
  };
  auto next_step = [&]() {
    ks_next += kstep;
    vs_next += vstep;
    dst = dst + G::STAGE == lds0 + G::RING ? lds0 : dst + G::STAGE;
  };

  // ---- tables
  int k_row[KS];                                                  // fragment ks of row ln of a 32-row tile
#pragma unroll
  for (int ks = 0; ks < KS; ++ks) k_row[ks] = ln * ROWB + (((2 * ks + hh) ^ swz_k<DH>(ln)) << 4);
  wait_vmcnt_imm<0>();
  lds_barrier();
  x8 Qu[KS], Qv[KS];
  f32x16 c[2];
#pragma unroll
  for (int t = 0; t < 2; ++t)
#pragma unroll
    for (int i = 0; i < 16; ++i) c[t][i] = 0.f;
#pragma unroll
  for (int ks = 0; ks < KS; ++ks) {
    float f[8];
    E::unpack(*(const u32x4*)(rows_q + qt * 32 * ROWB + k_row[ks]), f);
    const unsigned char* bp = rows_b + ((2 * ks + hh) << 4);
    Qu[ks] = qfrag_fma<E>(f, *(const u32x4*)bp, sc2);
    Qv[ks] = qfrag_fma<E>(f, *(const u32x4*)(bp + ROWB), sc2);
    const x8 qz = qfrag_fma<E>(f, *(const u32x4*)(bp + 2 * ROWB), sc2);
    if (has_chan) {
#pragma unroll
      for (int t = 0; t < 2; ++t) c[t] = E::mfma(*(const x8*)(rows_e + (kp * 2 + t) * 32 * ROWB + k_row[ks]), qz, c[t], 0, 0, 0);
    }
  }
  float* tab = (float*)sp_lds + qt * 4096;
#pragma unroll
  for (int t = 0; t < 2; ++t)
#pragma unroll
    for (int i = 0; i < 16; ++i) tab[((kp * 2 + t) * 32 + (i >> 2) * 8 + hh * 4 + (i & 3)) * 32 + ln] = c[t][i];
  float* Stq = St + qt * steps32 * 32;
  for (int t0 = kp * 32; t0 < steps32; t0 += 64) {
    f32x16 s;
#pragma unroll
    for (int i = 0; i < 16; ++i) s[i] = 0.f;
    if (has_time) {
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) s = E::mfma(*(const x8*)(rows_t + t0 * ROWB + k_row[ks]), Qv[ks], s, 0, 0, 0);
    }
#pragma unroll
    for (int i = 0; i < 16; ++i) Stq[(t0 + (i >> 2) * 8 + hh * 4 + (i & 3)) * 32 + ln] = s[i];
  }
  uint32_t kbits[2];
#pragma unroll
  for (int t = 0; t < 2; ++t) {
    const int ck = (kp * 2 + t) * 32 + ln;
    bool ok = ck < C_;
    if (valid) ok = ok && valid[min(ck, C_ - 1)] != 0;
    kbits[t] = (uint32_t)__ballot(ok) >> (4 * hh);
  }
  lds_barrier();
#pragma unroll
  for (int i = 0; i < 2 * G::LPW; ++i) request(i);  // (everybody is done with the rows there)
  next_step();
  f32x16 Bc[2];
#pragma unroll
  for (int t = 0; t < 2; ++t)
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const int d = cq - ((kp * 2 + t) * 32 + (i >> 2) * 8 + hh * 4 + (i & 3));
      const float v = tab[(C_ - 1 - min(d < 0 ? -d : d, C_ - 1)) * 32 + ln];
      Bc[t][i] = ((kbits[t] >> ((i >> 2) * 8 + (i & 3))) & 1u) ? v : -INFINITY;
    }

  int v_lane[MT], k_lane[KS];
  {
    const int e = (ln & 15) >> 2, aa = ln & 3, grp = ln >> 4, row0 = 4 * hh + e;
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
      v_lane[mt] = G::TILE + (kp * 64 + row0) * ROWB + (((4 * mt + 2 * grp + (aa >> 1)) ^ swz_v<DH>(row0)) << 4) + ((aa & 1) << 3);
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) k_lane[ks] = (kp * 64 + ln) * ROWB + (((2 * ks + hh) ^ swz_k<DH>(ln)) << 4);
  }
  float m_run = kMFloor, l_run = 0.f;
  f32x16 acc[MT];
#pragma unroll
  for (int mt = 0; mt < MT; ++mt)
#pragma unroll
    for (int i = 0; i < 16; ++i) acc[mt][i] = 0.f;

  int stage = G::R - 1;
  for (int s = 0; s < steps; ++s) {
    // step s has landed; everybody is done with the stage that step s + 1 goes into (at s = 0: with the tables)
    wait_vmcnt_imm<0>();
    lds_barrier();
    const unsigned char* st_lds = sp_lds + stage * G::STAGE;
    stage = stage + 1 == G::R ? 0 : stage + 1;
    const bool more = s + 1 < steps;
    const float st = Stq[s * 32 + ln];
    // The next step's requests go out one behind a product: together in front of them (64 KiB at the CU's one address unit, 1024
    // cycles) every wave stood there first.  B1 H16 Hkv8 Dh128 with the merge, us: C100 T64 in 8 runs 28.4 -> 26.9, C128 T512 in 16
    // 90.4 -> 86.5, T16 in 2 26.2 -> 24.5, T110 in 16 31.0 -> 30.6.
    f32x16 S[2] = {Bc[0], Bc[1]};
    x8 kf[4];
#pragma unroll
    for (int p = 0; p < 3; ++p) kf[p] = *(const x8*)(st_lds + k_lane[p >> 1] + (p & 1) * 32 * ROWB);
#pragma unroll
    for (int p = 0; p < 2 * KS; ++p) {
      const int t = p & 1, ks = p >> 1;
      if (p + 3 < 2 * KS) kf[(p + 3) & 3] = *(const x8*)(st_lds + k_lane[(p + 3) >> 1] + ((p + 3) & 1) * 32 * ROWB);
      S[t] = E::mfma(kf[p & 3], Qu[ks], S[t], 0, 0, 0);
      __builtin_amdgcn_sched_barrier(0);
      if (more && p * 2 * G::LPW / (2 * KS) < (p + 1) * 2 * G::LPW / (2 * KS)) request(p * 2 * G::LPW / (2 * KS));
      __builtin_amdgcn_sched_barrier(0);
    }
    next_step();
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      float rmax = -INFINITY;
#pragma unroll
      for (int i = 0; i < 16; ++i) rmax = fmaxf(rmax, S[t][i]);
      const float cand = xhalf_max(rmax) + st;
      if (__ballot(cand > m_run + 8.f) != 0ull) {
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
      for (int i = 0; i < 16; ++i) S[t][i] = fast_exp2(S[t][i] + off);
      const x8 P[2] = {E::pack(S[t], 0), E::pack(S[t], 8)};
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
          const unsigned char* vp = st_lds + v_lane[mt] + (32 * t + 16 * p) * ROWB;
          const x4 lo = E::read_tr(vp), hi = E::read_tr(vp + 8 * ROWB);
          acc[mt] = E::mfma(__builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7), P[p], acc[mt], 0, 0, 0);
        }
    }
  }

  // ---- the two halves of the keys: each wave of a pair finishes half of the output columns (one of them all: 2.4 us)
  constexpr int HALF = MT / 2;
  lds_barrier();
  const int other = wave ^ 4;
  float* ml = (float*)sp_lds + lane;                              // [wave][m | l][lane]
  f32x4* give = (f32x4*)(sp_lds + 8 * 512) + lane;                // [wave][quad of the half][lane]
  ml[wave * 128] = m_run;
  ml[wave * 128 + 64] = l_run;
  auto hand_over = [&](auto first) {
#pragma unroll
    for (int q = 0; q < HALF * 4; ++q) {
      const f32x16& v = acc[first() + q / 4];
      give[(wave * HALF * 4 + q) * 64] = f32x4{v[q % 4 * 4], v[q % 4 * 4 + 1], v[q % 4 * 4 + 2], v[q % 4 * 4 + 3]};
    }
  };
  if (kp == 0) hand_over(std::integral_constant<int, HALF>());
  else hand_over(std::integral_constant<int, 0>());
  lds_barrier();
  const float m1 = ml[other * 128], m = fmaxf(m_run, m1), a0 = fast_exp2(m_run - m), a1 = fast_exp2(m1 - m);
  const float w0 = kp == 0 ? a0 : a1, w1 = kp == 0 ? a1 : a0;       // of the first half of the keys, of the second
  const float l1 = ml[other * 128 + 64];
  l_run = __builtin_fmaf(w0, kp == 0 ? l_run : l1, w1 * (kp == 0 ? l1 : l_run));
  const float ltot = l_run + __shfl_xor(l_run, 32);
  const float inv = 1.f / ltot;
  // through LDS, so that whole halves of rows leave
  constexpr int PITCH = HALF * 64 + 16, CPR = HALF * 4;
  unsigned char* stg = sp_lds + 8 * (512 + HALF * 4 * 1024) + wave * (32 * PITCH);
  auto finish = [&](auto first) {
#pragma unroll
    for (int q = 0; q < HALF * 4; ++q) {
      const f32x16& v = acc[first() + q / 4];
      const f32x4 o = give[(other * HALF * 4 + q) * 64];
      x4 w;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const float own = v[q % 4 * 4 + r];
        w[r] = E::cvt(__builtin_fmaf(w0, first() == 0 ? own : o[r], w1 * (first() == 0 ? o[r] : own)) * inv);
      }
      *(x4*)(stg + ln * PITCH + (q / 4 * 32 + q % 4 * 8 + hh * 4) * 2) = w;
    }
  };
  if (kp == 0) finish(std::integral_constant<int, 0>());
  else finish(std::integral_constant<int, HALF>());
  wave_lds_sync();
  const int64_t prow0 = ((int64_t)run * nbh + bh) * C_;           // rows of the split workspace
#pragma unroll
  for (int i = 0; i < 32 * CPR / 64; ++i) {
    const int row = (i * 64 + lane) / CPR, ch = (i * 64 + lane) % CPR;
    if (qt * 32 + row < C_)
      *(u32x4*)((bf16_t*)a.split_ws + (prow0 + qt * 32 + row) * DH + kp * HALF * 32 + ch * 8) = *(const u32x4*)(stg + row * PITCH + ch * 16);
  }
  if (kp == 0 && hh == 0 && cq < C_)
    ((float*)((bf16_t*)a.split_ws + (int64_t)n_split * nbh * C_ * DH))[prow0 + cq] = m + log2f(ltot);
}

template <int DH>
static int step_lds_bytes(const mvpa_fwd_args* a) {
  const int steps = (a->T + a->n_split - 1) / a->n_split;
  const int steps32 = (steps + 31) & ~31;
  return step_cfg<DH>::RING + 4 * steps32 * 128 + steps32 * step_cfg<DH>::ROWB + 1024;
}

template <int DH, typename E>
static int launch_step_t(const mvpa_fwd_args* a, hipStream_t stream) {
  auto kern = mvpa_step_kernel<DH, E>;
  const int lds = step_lds_bytes<DH>(a);
  want_dynamic_lds((const void*)kern, lds);
  const step_geom geo = make_step_geom(a->B * a->Hkv, a->H / a->Hkv, a->n_split, a->T);
  MVPA_LAUNCH(kern, step_grid(geo, geo.grp), dim3(512), lds, stream, *a, geo);
  return take_launch_status();
}

}  // namespace mvpa

// 65..128 channels, head size 64 or 128; runs whose time rows and scores fit beside the ring (32 steps at 128)
int mvpa_step_supported(const mvpa_fwd_args* a) {
  if (!mvpa_mfma_supported(a) || (a->flags & MVPA_FLAG_FP8_QK) || !(a->flags & MVPA_FLAG_CONTENT)) return 0;
  if (a->C <= 64 || (a->Dh != 64 && a->Dh != 128) || a->n_split <= 1) return 0;
  return (a->Dh == 64 ? mvpa::step_lds_bytes<64>(a) : mvpa::step_lds_bytes<128>(a)) <= 160 * 1024;
}

int mvpa_launch_step(const mvpa_fwd_args* a, hipStream_t stream) {
  using namespace mvpa;
  const bool f16 = a->dtype == MVPA_F16;
  if (a->Dh == 64) return f16 ? launch_step_t<64, el_f16>(a, stream) : launch_step_t<64, el_bf16>(a, stream);
  return f16 ? launch_step_t<128, el_f16>(a, stream) : launch_step_t<128, el_bf16>(a, stream);
}
