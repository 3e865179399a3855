// MVPA backward on MFMA (bf16, Dh = 64 or 128, up to 64 channels per launch, 128 in parts): the QUERY pass (the KEY pass follows below).
//
// Same tiling as the forward kernel: queries and keys are tiled by time step, a wave owns 32
// query channels of one time step, products are formed transposed (a lane owns one query), the
// channel-bias tile is built once per wave and used as the C operand of K Q^T, the time bias is
// one scalar per (query, key step) taken from 32-step slabs.  With the forward's base-2
// log-sum-exp L nothing is "online" here: per key step
//     S^T  = K (q+u)^T + Bc + st          (content product only inside the window)
//     P^T  = exp2(S^T - L)
//     dP^T = V dO^T
//     dS^T = P^T o (dP^T - delta) * scale,          delta = dO . O
//     dq^T += K^T dS^T                     (inside the window)
//     dbias_time[q, tk] = sum_ck dS,       dbias_chan[q, |cq-ck|] += dS.
// Outputs are those of mvpa_backward (include/mvpa_hip.h): the content share of dq and the two
// bias-table gradients.  For the key pass the workspace receives, in base-2 score units, -delta,
// the channel-table rows, (time bias - L) laid out [b,h,tq,tk,cq] and (q+u) * scale in bf16.
// K and V tiles come through a ring of LDS stages filled by direct-to-LDS loads; one copy of K serves the row
// fragments of K Q^T and the transposed ones of K^T dS^T; far key steps fetch V only.
#include "mvpa_common.h"

#include <type_traits>

namespace mvpa {
namespace bwdq {

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;
typedef __attribute__((ext_vector_type(4))) __bf16 bf16x4;
typedef __attribute__((ext_vector_type(2))) __bf16 bf16x2;
typedef __attribute__((ext_vector_type(2))) float f32x2;
typedef __attribute__((ext_vector_type(4))) float f32x4;
typedef __attribute__((ext_vector_type(16))) float f32x16;
typedef __attribute__((ext_vector_type(4))) uint32_t u32x4;

#define BWD_LDS_PTR(T) __attribute__((address_space(3))) T*

// Head dim DH is 64 or 128: KS = DH / 16 contraction blocks per product, MT = DH / 32 output tiles
// of the gradients, rows of ROWB = 2 DH bytes (CPR = DH / 8 chunks of 16 bytes) in the LDS tiles.
// floats of per-wave scratch in the query pass: a slab of 32 key steps' time-bias exponents [step][query] and of their
// gradients [query][step].  The channel table of the set-up ([64][32]) overlays them.
constexpr int WAVE_SCRATCH = 2048;
typedef float f32x4u __attribute__((ext_vector_type(4), aligned(4)));        // four floats at any float's address

__device__ inline void wave_sync_lds() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// workgroup barrier that orders LDS traffic only (global loads of the ring stay in flight)
__device__ inline void lds_barrier() {
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
}

// direct-to-LDS loads: lane L's 16 (4) bytes land at lds_base + 16 L (4 L).  Inline assembly so
// that the compiler does not drain the ring in front of later LDS reads; completion is awaited
// with wait_vmcnt_imm before the barrier that publishes a stage.
__device__ inline void dma16(const void* gptr, uint32_t lds_base) {
  lds_base = __builtin_amdgcn_readfirstlane(lds_base);    // uniform by construction; pins it to an SGPR
  asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off"
               :: "v"(gptr), "s"(lds_base) : "memory", "m0");
}
__device__ inline void dma4(const void* gptr, uint32_t lds_base) {
  lds_base = __builtin_amdgcn_readfirstlane(lds_base);
  asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dword %0, off"
               :: "v"(gptr), "s"(lds_base) : "memory", "m0");
}

template <int N>
__device__ inline void wait_vmcnt_imm() {
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}

__device__ inline bf16x8 as_frag(u32x4 v) {
  union { u32x4 u; bf16x8 b; } c;
  c.u = v;
  return c.b;
}

// 8 bf16 of a q row + bias, scaled, as an MFMA fragment
__device__ inline bf16x8 qfrag(u32x4 raw, u32x4 braw, float scale) {
  bf16x8 out;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const uint32_t w = raw[i], bw = braw[i];
    out[2 * i] = (__bf16)((__uint_as_float(w << 16) + __uint_as_float(bw << 16)) * scale);
    out[2 * i + 1] = (__bf16)((__uint_as_float(w & 0xffff0000u) + __uint_as_float(bw & 0xffff0000u)) * scale);
  }
  return out;
}

// 8 floats to a bf16 fragment, two per conversion instruction
__device__ inline bf16x8 pack8(const f32x16& v, int base) {
  union { bf16x8 f; bf16x2 q[4]; } out;
#pragma unroll
  for (int i = 0; i < 4; ++i)
    out.q[i] = __builtin_convertvector(f32x2{v[base + 2 * i], v[base + 2 * i + 1]}, bf16x2);
  return out.f;
}

// sum over a lane and its partner in the other half-wave, without a trip through the LDS crossbar
__device__ inline float xhalf_sum(float x) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}
__device__ inline float xhalf_max(float x) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}

// The 16-byte chunks of a row of 2 DH bytes are swizzled so that both kinds of reads of one copy are free of bank
// conflicts: a row fragment takes one chunk of 16 rows (256 bytes of banks: all its chunks at Dh 128, two rows' at Dh
// 64, differ), a transposing read four chunks of four rows (differ in bits 2, 3; at Dh 64 rows of one parity in bit 2).
template <int DH> __device__ inline int swz(int row) {
  return DH == 64 ? ((row >> 1) & 1) << 2 | ((row >> 2) & 3) : (row & 3) << 2 | ((row >> 2) & 3);
}

// ONE: the whole walk.  FAR, WIN: the steps before a wave's content window and those from it on, as a launch
// each, FAR first.  At Dh 128 a wave of the whole walk takes 420 registers and has its SIMD to itself: the far steps'
// LDS reads, products, reductions and table slabs simply add up (0.89 us a step of 2 x 64 queries at T 512, 0.25 of
// them products).  FAR alone fits in 256, and two waves cover each other's waits (1.2 us a step of 4 x 64 queries).
//
// At Dh 64 a workgroup is 4 waves and two of them share a CU (80 KB and 256 registers): a third of a workgroup's life
// at T 128 is set-up, slabs and epilogue, chains of waits that leave the CU idle if all its waves are in them at
// once.  B4 H16 C64, T 128 / 256 / 512, one workgroup of 8 waves with a barrier a step against this: 920 / 1243 /
// 2043 -> 735 / 1040 / 1730 us; B4 H12 C21 T25 53 -> 34 us.  The clock is what is left: the waits of a far step have
// gone from 1040 to 570 of 1770 -> 1350 cycles, and it falls from 2.25 to 1.9 GHz as they go.
enum query_phase { ONE, FAR, WIN };
template <int PHASE> constexpr int PHASE_WAVES = PHASE == FAR ? 8 : 4;
// The last time step keeps the content term at every key step, T steps where the others have window + 1.  At Dh 128
// with two key tiles it has a workgroup to itself, in which two waves share a query tile and take a key tile each (window
// launch at T 512, 128 channels, most of which was this chain: 1.15 -> 0.99 ms).  At Dh 64 the chain hides behind the
// rest, and the longer code takes what it gives (T 25: 70 -> 73 us, T 128 730, T 512 1690 either way).
template <int DH, int NCT, int PHASE> constexpr bool LAST_APART = DH == 128 && NCT == 2 && PHASE != FAR;
template <int DH, int NCT, int PHASE> __host__ __device__ inline int query_tiles(int T, bool content) {
  constexpr int TQW = PHASE_WAVES<PHASE> / NCT;
  return LAST_APART<DH, NCT, PHASE> && content ? (T - 1 + TQW - 1) / TQW + 1 : (T + TQW - 1) / TQW;
}
// waves per SIMD: at Dh 64 two workgroups share a CU
template <int DH, int PHASE> constexpr int PHASE_OCC = PHASE == FAR || DH == 64 ? 2 : 1;
// The ring holds three units of two tiles: V of two far steps, or V and K of a step with content.
template <int DH, int NCT> constexpr int TILE_BYTES = NCT * 32 * 2 * DH;
template <int DH, int NCT, int PHASE> constexpr int QUERY_LDS = 6 * TILE_BYTES<DH, NCT> + PHASE_WAVES<PHASE> * WAVE_SCRATCH * 4;

// One tile of query time steps of one (b, h).  LAST: the last time step alone.
template <int DH, int NCT, int PHASE, bool LAST>
__device__ __forceinline__ void query_walk(const mvpa_bwd_args& a, int q0, int k0, int accum, int bh, int tile) {
  constexpr int KS = DH / 16, MT = DH / 32, ROWB = 2 * DH, CPR = DH / 8;
  constexpr int NW = PHASE_WAVES<PHASE>;
  constexpr bool SOLO = PHASE_OCC<DH, PHASE> == 1;                // one wave per SIMD
  constexpr int CP = NCT * 32, TQW = NW / NCT, TILE = TILE_BYTES<DH, NCT>;
  static_assert(64 * 32 <= WAVE_SCRATCH && (1 + 32 * (CP + 1)) * 4 <= QUERY_LDS<DH, NCT, PHASE> / NW && MT * 4096 <= QUERY_LDS<DH, NCT, PHASE> / NW, "channel tables overlay the rest");
  constexpr int LPW = TILE / 1024 / NW;           // 1 KiB wave loads per wave and tile copy
  extern __shared__ __attribute__((aligned(1024))) unsigned char smem[];
  float* wave_base = (float*)(smem + 6 * TILE);

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int ln = lane & 31, hh = lane >> 5;
  constexpr int PC = CP + 1;                      // padded pitch of the epilogue's table
  float* Stb = wave_base + wave * WAVE_SCRATCH;           // [32 steps][32 queries] time-bias exponents of a slab
  float* Gtb = Stb + 1024;                                // [32 queries][32 steps] their gradients, in swizzled fours
  float* scr = Stb;                                       // before the first slab [64][32] channel table
  float* g_lane = Gtb + ln * 32;                          // step j of the slab at 4 ((j >> 2) ^ (ln & 7)) + (j & 3)
  const int g_swz = (ln & 7) << 2;

  const int T_ = a.T, C_ = a.C, W = a.window, N = a.T * a.C;
  const int CW = (C_ + 3) & ~3;                   // row pitch of the Ec tiles in the workspace
  const bool has_content = a.flags & MVPA_FLAG_CONTENT;
  const bool has_time = a.flags & MVPA_FLAG_TIME_BIAS;
  const bool has_chan = a.flags & MVPA_FLAG_CHAN_BIAS;
  const int b = bh / a.H, h = bh % a.H;
  const int g = h / (a.H / a.Hkv);
  const int tq_end = LAST_APART<DH, NCT, PHASE> && has_content ? T_ - 2 : T_ - 1;    // the last step of these tiles
  const int tq0 = LAST ? T_ - 1 : tile * TQW;
  const int tq_hi = LAST ? T_ - 1 : min(tq_end, tq0 + TQW - 1);
  const int tq = LAST ? T_ - 1 : tq0 + wave / NCT;
  const bool second = LAST && wave >= NCT;        // wave w and wave w + NCT take a key tile each
  const bool active = LAST || tq <= tq_hi;
  const int cqw0 = q0 + (wave % NCT) * 32;        // first query channel of this wave
  const int cq = cqw0 + ln;
  const bool qok = active && cq < C_;
  const int nq = active ? tq * C_ + min(cq, C_ - 1) : 0;
  const int64_t row = ((int64_t)b * a.H + h) * N + nq;

  const bf16_t* qrow = (const bf16_t*)a.q + b * a.q_stride_b + h * a.q_stride_h + (int64_t)nq * a.q_stride_n;
  const bf16_t* orow = (const bf16_t*)a.o + b * a.o_stride_b + h * a.o_stride_h + (int64_t)nq * a.o_stride_n;
  const bf16_t* drow = (const bf16_t*)a.d_o + b * a.do_stride_b + h * a.do_stride_h + (int64_t)nq * a.do_stride_n;
  const bf16_t* kbase = (const bf16_t*)a.k + b * a.k_stride_b + g * a.k_stride_h;
  const bf16_t* vbase = (const bf16_t*)a.v + b * a.v_stride_b + g * a.v_stride_h;
  const bf16_t* ktime = (const bf16_t*)a.k_time + (int64_t)g * T_ * DH;
  const bf16_t* kchan = (const bf16_t*)a.k_chan + (int64_t)g * C_ * DH;
  const bf16_t* bu = (const bf16_t*)a.bias_u + g * DH;
  const bf16_t* bv = (const bf16_t*)a.bias_v + g * DH;
  const bf16_t* bz = (const bf16_t*)a.bias_z + g * DH;
  const uint8_t* valid = a.chan_valid ? a.chan_valid + (int64_t)b * C_ : nullptr;
  const float sc2 = a.sm_scale * kLog2e;          // scores live in the base-2 domain

  // ---- the ring: per-wave source offsets (the swizzle is applied on the source side), prologue
  int k_off[LPW], v_off[LPW];
#pragma unroll
  for (int i = 0; i < LPW; ++i) {
    const int pc = (wave + NW * i) * 64 + lane;
    const int r = pc / CPR, phys = pc % CPR;
    const int rc = min(k0 + r, C_ - 1);           // key channels k0 .. of this launch
    k_off[i] = rc * (int)a.k_stride_n + ((phys ^ swz<DH>(r)) << 3);
    v_off[i] = rc * (int)a.v_stride_n + ((phys ^ swz<DH>(r)) << 3);
  }
  // first key step whose K is needed: the band of the earliest query step of the workgroup
  const int tk_near = LAST ? 0 : !has_content ? tq_hi + 1 : (W <= 0 || tq_hi == T_ - 1) ? 0 : max(0, tq0 - W);
  // this wave's far steps are those before far_end (none for the last time step, whose queries keep the content
  // term everywhere); the workgroup walks the key steps tk_lo .. tk_hi
  const int far_end = !active || LAST ? 0 : !has_content ? tq + 1 : (W <= 0 || tq == T_ - 1) ? 0 : max(0, tq - W);
  const int far_top = tq_hi == T_ - 1 ? T_ - 2 : tq_hi;           // FAR: the latest query step with far steps
  const int tk_lo = PHASE == WIN ? tk_near : 0;
  const int tk_hi = PHASE == FAR ? (far_top < tq0 ? -1 : far_top - W - 1) : tq_hi;
  const int tk_first = PHASE == WIN ? far_end : 0;                // slabs of 32 steps count from here
  const int far_lim = PHASE == FAR ? tk_hi + 1 : PHASE == WIN ? 0 : tk_near;       // steps before it are walked in pairs
  const uint32_t ring_lds = (uint32_t)(uintptr_t)(BWD_LDS_PTR(unsigned char))smem;
  auto issue_v = [&](int tk, uint32_t dst) {
    const bf16_t* vsrc = vbase + (int64_t)tk * C_ * a.v_stride_n;
#pragma unroll
    for (int i = 0; i < LPW; ++i) dma16(vsrc + v_off[i], dst + (wave + NW * i) * 1024);
  };
  auto next_unit = [&](int tk) { return PHASE != WIN && tk < far_lim ? min(tk + 2, far_lim) : tk + 1; };
  auto unit_loads = [&](int tk) { return tk > tk_hi ? 0 : PHASE != WIN && tk + 1 == far_lim ? LPW : 2 * LPW; };
  auto issue_unit = [&](int tk, int slot) {
    if (tk > tk_hi) return;
    const uint32_t st = ring_lds + slot * 2 * TILE;
    issue_v(tk, st);
    if (PHASE != WIN && tk < far_lim) {
      if (tk + 1 < far_lim) issue_v(tk + 1, st + TILE);
    } else {
      const bf16_t* ksrc = kbase + (int64_t)tk * C_ * a.k_stride_n;
#pragma unroll
      for (int i = 0; i < LPW; ++i) dma16(ksrc + k_off[i], st + TILE + (wave + NW * i) * 1024);
    }
  };
  issue_unit(tk_lo, 0);
  issue_unit(next_unit(tk_lo), 1);
  int slot = 0;
  // the stage of the unit of key step tk; requests the unit after the next one
  auto begin_unit = [&](int tk) __attribute__((always_inline)) -> const unsigned char* {
    const int before = slot == 0 ? 2 : slot - 1;
    if (PHASE != WIN && tk + 5 < far_lim) {       // far steps all around
      wait_vmcnt_imm<2 * LPW>();
      lds_barrier();                              // the unit is visible to all; everyone is done with the one before
      issue_v(tk + 4, ring_lds + before * 2 * TILE);
      issue_v(tk + 5, ring_lds + (before * 2 + 1) * TILE);
    } else {
      const int next = next_unit(tk), loads = unit_loads(next);   // these may be under way
      if (loads == 2 * LPW) wait_vmcnt_imm<2 * LPW>();
      else if (loads == LPW) wait_vmcnt_imm<LPW>();
      else wait_vmcnt_imm<0>();
      lds_barrier();
      issue_unit(next_unit(next), before);
    }
    const unsigned char* p = smem + slot * 2 * TILE;
    slot = slot == 2 ? 0 : slot + 1;
    return p;
  };

  // ---- set-up: operand fragments, delta, channel-bias tile
  bf16x8 dOf[KS];            // (q+u), (q+v) fragments are re-formed where needed, not kept
  f32x16 Ec[NCT];            // exp2(channel bias - mc): the far steps' probabilities up to a scalar
  float delta = 0.f, mc = -INFINITY, sumEc = 0.f;
  // every global load of the set-up goes out before the first use: one round trip, not one per
  // fragment.  The log-sum-exp is among them so that its wait does not fall into the loops, where
  // it would drain the whole ring (vmcnt 0) at every key step.
  u32x4 raw_[KS], draw_[KS], oraw_[KS], bz_[KS], bu_[KS];
  u32x4 er[KS][2];
  auto window_row = [&](int t) { return max(C_ - 1 - max(cqw0 + 31 - k0 - t * 32, k0 + t * 32 + 31 - cqw0), 0); };
  auto load_window = [&](int t) {
#pragma unroll
    for (int ks = 0; ks < KS; ++ks)
#pragma unroll
      for (int tt = 0; tt < 2; ++tt)
        er[ks][tt] = *(const u32x4*)(kchan + (int64_t)min(window_row(t) + tt * 32 + ln, C_ - 1) * DH + ks * 16 + hh * 8);
  };
  load_window(0);
#pragma unroll
  for (int ks = 0; ks < KS; ++ks) {
    const int d0 = ks * 16 + hh * 8;
    raw_[ks] = *(const u32x4*)(qrow + d0);
    draw_[ks] = *(const u32x4*)(drow + d0);
    oraw_[ks] = *(const u32x4*)(orow + d0);
    bz_[ks] = *(const u32x4*)(bz + d0);
    if (DH == 64) bu_[ks] = *(const u32x4*)(bu + d0);
  }
  const float lse = a.lse[row];
  uint64_t kmask;                                 // the (up to 64) key channels of this launch
  {
    const int ck = k0 + lane;
    bool ok = ck < C_ && lane < CP;
    if (valid) ok = ok && valid[min(ck, C_ - 1)] != 0;
    kmask = __ballot(ok);
  }
  asm volatile("" :: "v"(lse));
  {
    bf16x8 qz[KS];
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      const u32x4 raw = raw_[ks], draw = draw_[ks], oraw = oraw_[ks];
      qz[ks] = qfrag(raw, bz_[ks], sc2);
      dOf[ks] = as_frag(draw);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        delta += __uint_as_float(draw[i] << 16) * __uint_as_float(oraw[i] << 16);
        delta += __uint_as_float(draw[i] & 0xffff0000u) * __uint_as_float(oraw[i] & 0xffff0000u);
      }
    }
    delta = xhalf_sum(delta);
    // Channel-bias tile, one key tile at a time: the 32 queries of this wave and the 32 keys of
    // tile t are at most 63 channels apart in either direction, so the rows C-1-d of the table
    // (q+z).k_chan^T they need lie in a window of 64 rows starting at jlo.  That window goes
    // through the per-wave scratch ([64][32]), and Bc[key][q] = table[C-1-|cq-ck|][q] is
    // gathered from it; -inf where the key channel is padding or absent.
#pragma unroll
    for (int t = 0; t < NCT; ++t) {
      const int ck0 = k0 + t * 32, jlo = window_row(t);
      f32x16 sct[2];
#pragma unroll
      for (int tt = 0; tt < 2; ++tt)
#pragma unroll
        for (int i = 0; i < 16; ++i) sct[tt][i] = 0.f;
#pragma unroll
      for (int ks = 0; ks < KS; ++ks)
#pragma unroll
        for (int tt = 0; tt < 2; ++tt)
          sct[tt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(as_frag(er[ks][tt]), qz[ks], sct[tt], 0, 0, 0);
      if (t + 1 < NCT) load_window(t + 1);        // on their way while this tile is gathered
      if (!has_chan)
#pragma unroll
        for (int tt = 0; tt < 2; ++tt)
#pragma unroll
          for (int i = 0; i < 16; ++i) sct[tt][i] = 0.f;
      wave_sync_lds();                            // the previous tile's gather is done with the scratch
#pragma unroll
      for (int tt = 0; tt < 2; ++tt)
#pragma unroll
        for (int i = 0; i < 16; ++i) scr[(tt * 32 + (i >> 2) * 8 + hh * 4 + (i & 3)) * 32 + ln] = sct[tt][i];
      wave_sync_lds();
      // Row of the window for key ck = ck0 + c_i + 4hh: (C-1-jlo) - |cq - ck|, at most 62.  In floats, where the
      // absolute value is free; rows below 0 belong to padded queries and keys, for which any value does.
      const float top = (float)((C_ - 1 - jlo) * 32 + ln), dc = (float)(32 * (cq - ck0 - 4 * hh));
#pragma unroll
      for (int i = 0; i < 16; ++i) Ec[t][i] = scr[(int)fmaxf(top - fabsf(dc - (float)(32 * ((i >> 2) * 8 + (i & 3)))), 0.f)];
      if ((uint32_t)(kmask >> (t * 32)) != 0xffffffffu) {
        const uint32_t kbits = (uint32_t)(kmask >> (t * 32 + 4 * hh));
#pragma unroll
        for (int i = 0; i < 16; ++i) Ec[t][i] = ((kbits >> ((i >> 2) * 8 + (i & 3))) & 1u) ? Ec[t][i] : -INFINITY;
      }
    }
#pragma unroll
    for (int t = 0; t < NCT; ++t)
#pragma unroll
      for (int i = 0; i < 16; ++i) mc = fmaxf(mc, Ec[t][i]);
    mc = xhalf_max(mc);
    if (mc == -INFINITY) mc = 0.f;                // no valid key channel at all
#pragma unroll
    for (int t = 0; t < NCT; ++t)
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        Ec[t][i] = __builtin_amdgcn_exp2f(Ec[t][i] - mc);
        sumEc += Ec[t][i];
      }
    sumEc = xhalf_sum(sumEc);
    bf16x8 qu[KS];
    if constexpr (PHASE != WIN) {
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) {
        const int d0 = ks * 16 + hh * 8;
        qu[ks] = DH == 64 ? qfrag(raw_[ks], bu_[ks], sc2) : qfrag(*(const u32x4*)(qrow + d0), *(const u32x4*)(bu + d0), sc2);
      }
    }
    // for the key pass: (q+u) * scale, delta, and the tile exp2(channel bias - mc) by
    // [query][key channel]; and the rows of dbias_time that no key step reaches
    if (PHASE != WIN && qok && !second) {
      float* wc = a.ws_chan + row * CW + k0;      // rows of CW floats: 16-byte aligned for any C
#pragma unroll
      for (int t = 0; t < NCT; ++t)
#pragma unroll
        for (int a4 = 0; a4 < 4; ++a4) {
          const int ci = t * 32 + a4 * 8 + hh * 4;
          if (k0 + ci < CW)
            *(float4*)(wc + ci) = make_float4(Ec[t][a4 * 4], Ec[t][a4 * 4 + 1], Ec[t][a4 * 4 + 2], Ec[t][a4 * 4 + 3]);
        }
    }
    // the stores last: loads return behind the stores before them
    if (PHASE != WIN && qok && !second) {
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) *(bf16x8*)((bf16_t*)a.ws_qu + row * DH + ks * 16 + hh * 8) = qu[ks];
      if (hh == 0) a.ws_delta[row] = -delta;
    }
  }

  f32x16 dq[MT], dSc[NCT];
#pragma unroll
  for (int mt = 0; mt < MT; ++mt)
#pragma unroll
    for (int i = 0; i < 16; ++i) dq[mt][i] = 0.f;
#pragma unroll
  for (int t = 0; t < NCT; ++t)
#pragma unroll
    for (int i = 0; i < 16; ++i) dSc[t][i] = 0.f;

  // this wave's query rows are consecutive in memory; outputs are written a row at a time (the
  // two half-waves take alternate rows) so that each store covers one contiguous run
  const int cq0 = cqw0;
  const int nq_live = active ? max(0, min(32, C_ - cq0)) : 0;
  const int64_t wrow0 = ((int64_t)b * a.H + h) * N + (int64_t)(active ? tq : 0) * C_ + cq0;

  // the columns of dbias_time that no key step reaches (once: by the launch that does not add)
  if (PHASE != WIN && !accum)
    for (int q = lane >> 3; q < nq_live; q += 8) {
      float* dst = a.dbias_time + (wrow0 + q) * T_;
      const int n = T_ - 1 - tq;
      if (n >= 4)
        for (int j = 4 * (lane & 7); j < n; j += 32) *(f32x4u*)(dst + min(j, n - 4)) = f32x4u{0.f, 0.f, 0.f, 0.f};
      else if ((lane & 7) < n)
        dst[lane & 7] = 0.f;
    }

  // ---- loop-invariant fragment offsets
  int r_lane[KS], t_lane[MT];
  {
    const int e = (ln & 15) >> 2, aa = ln & 3, grp = ln >> 4;
    const int row0 = 4 * hh + e;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) r_lane[ks] = ln * ROWB + (((2 * ks + hh) ^ swz<DH>(ln)) << 4);
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
      t_lane[mt] = row0 * ROWB + (((4 * mt + 2 * grp + (aa >> 1)) ^ swz<DH>(row0)) << 4) + ((aa & 1) << 3);
  }
  auto tr_frag = [&](const unsigned char* tile_p, int t, int s, int mt) -> bf16x8 {
    const unsigned char* p = tile_p + (32 * t + 16 * s) * ROWB;   // eight rows on, bit 1 of the swizzle is the other
    const bf16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4bf16((BWD_LDS_PTR(bf16x4))(p + t_lane[mt]));
    const bf16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4bf16((BWD_LDS_PTR(bf16x4))(p + 8 * ROWB + (t_lane[mt] ^ 32)));
    return __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
  };

  // the first n floats of each of the first rows rows of a slab: eight lanes a row, four floats a lane; the last four
  // of a row overlap the ones before them with the same values
  auto store_rows = [&](int rows, int n, auto at, auto value) __attribute__((always_inline)) {
    int l = lane;
    asm volatile("" : "+v"(l));                    // the addresses are formed here, not kept in registers over the walk
    if (n >= 4) {
      const int c = min(4 * (l & 7), n - 4);
#pragma unroll
      for (int it = 0; it < 4; ++it) {
        const int r = it * 8 + (l >> 3);
        f32x4u v;
#pragma unroll
        for (int x = 0; x < 4; ++x) v[x] = value(r, c + x);
        if (r < rows && 4 * (l & 7) < n) *(f32x4u*)(at(r) + c) = v;
      }
    } else {
#pragma unroll 1
      for (int r = l >> 2; r < rows; r += 16)
        if ((l & 3) < n) at(r)[l & 3] = value(r, l & 3);
    }
  };

  // writes the gradients of the slab that started at key step tks, and its per-pair scalars for
  // the key pass (the exponent e = time bias - L + mc for pairs inside the window, else exp2(e))
  auto flush_slab = [&](int tks) __attribute__((always_inline)) {
    const int nj = min(32, (PHASE == FAR ? far_end : tq + 1) - tks);
    if (!second)
    store_rows(nj, min(32, C_ - cqw0), [&](int jj) { return a.ws_time + (((int64_t)bh * T_ + tq) * T_ + tks + jj) * C_ + cqw0; },
               [&](int jj, int q) {
                 const float e = Stb[jj * 32 + q];
                 const bool near_pair = has_content && (W <= 0 || tq - tks - jj <= W || tq == T_ - 1);
                 return near_pair ? e : __builtin_amdgcn_exp2f(e);
               });
    if (LAST && !second) return;                // the second wave adds up both waves' gradients
    const int j0 = time_row(tq, tks, T_);
    auto gradient = [&](int q, int jj) __attribute__((always_inline)) {
      const float* g = Gtb + q * 32 + (jj ^ ((q & 7) << 2));
      return (second ? g[0] + g[-NCT * WAVE_SCRATCH] : g[0]) * a.sm_scale;
    };
    if (!accum) {
      store_rows(nq_live, nj, [&](int q) { return a.dbias_time + (wrow0 + q) * T_ + j0; }, gradient);
    } else {
      // launches of one stream: the key parts add up.  An atomic add without a return value, not a load and a
      // store: nothing waits for the old value (every address has one writer)
#pragma unroll 8
      for (int it = 0; it < 16; ++it) {
        const int q = 2 * it + hh;
        const float g = gradient(q, ln);
        if (q < nq_live && ln < nj) atomicAdd(a.dbias_time + (wrow0 + q) * T_ + j0 + ln, g);
      }
    }
  };

  // Every 32 key steps: form the next slab of time-bias scores, write the finished one.  In this order: loads return
  // behind the stores before them.
  auto time_slab = [&](int tk) __attribute__((always_inline)) {
    if (((tk - tk_first) & 31) == 0) {
      f32x16 stc;
#pragma unroll
      for (int i = 0; i < 16; ++i) stc[i] = 0.f;
      if (has_time) {
        const int j = min(time_row(tq, tk, T_) + ln, T_ - 1);
        u32x4 rr[KS], qr[KS], br[KS];
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) {         // every load before the first use
          rr[ks] = *(const u32x4*)(ktime + (int64_t)j * DH + ks * 16 + hh * 8);
          qr[ks] = *(const u32x4*)(qrow + ks * 16 + hh * 8);
          br[ks] = *(const u32x4*)(bv + ks * 16 + hh * 8);
        }
#pragma unroll
        for (int ks = 0; ks < KS; ++ks)
          stc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(as_frag(rr[ks]), qfrag(qr[ks], br[ks], sc2), stc, 0, 0, 0);
      }
      if (tk > tk_first) {
        if constexpr (LAST) lds_barrier();
        else wave_sync_lds();
        flush_slab(tk - 32);
        if constexpr (LAST) lds_barrier();
        else wave_sync_lds();
      }
#pragma unroll
      for (int i = 0; i < 16; ++i) Stb[((i >> 2) * 8 + hh * 4 + (i & 3)) * 32 + ln] = stc[i] - lse + mc;
      wave_sync_lds();
    }
  };

  // A far key step (content term dropped): P^T = Ec et with et = exp2(time bias - L + mc) one
  // scalar per query, so with dP^T = V dO^T
  //     dbias_time[q, tk]  = et (sum_keys Ec dP - delta sumEc)
  //     dbias_chan share   = Ec (sum_tk et dP - delta sum_tk et)   (formed after the loop)
  // (all of them, like dS below, times the score scale where they are written)
  // costs two FMAs per element and no exponential per element.
  float esum = 0.f;
  // Every fragment is read before the first product: read where they are used, each waits out the LDS latency.
  auto far_read = [&](const unsigned char* Vrow, bf16x8 (&vf)[KS][NCT]) __attribute__((always_inline)) {
#pragma unroll
    for (int ks = 0; ks < KS; ++ks)
#pragma unroll
      for (int t = 0; t < NCT; ++t) vf[ks][t] = *(const bf16x8*)(Vrow + r_lane[ks] + t * 32 * ROWB);
  };
  auto far_products = [&](const bf16x8 (&vf)[KS][NCT], f32x16 (&dP)[NCT]) __attribute__((always_inline)) {
#pragma unroll
    for (int t = 0; t < NCT; ++t)
#pragma unroll
      for (int i = 0; i < 16; ++i) dP[t][i] = 0.f;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks)
#pragma unroll
      for (int t = 0; t < NCT; ++t) dP[t] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vf[ks][t], dOf[ks], dP[t], 0, 0, 0);
  };
  auto far_reduce = [&](const f32x16 (&dP)[NCT], float st, int tk) __attribute__((always_inline)) {
    const float et = __builtin_amdgcn_exp2f(st);
    float dot[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int t = 0; t < NCT; ++t)
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        dot[i & 3] += Ec[t][i] * dP[t][i];
        dSc[t][i] += et * dP[t][i];
      }
    esum += et;
    const float gt = et * (xhalf_sum((dot[0] + dot[1]) + (dot[2] + dot[3])) - delta * sumEc);
    g_lane[(tk & 31) ^ g_swz] = gt;               // both halves hold it: no branch
  };
  auto far_one = [&](const unsigned char* Vrow, int tk) __attribute__((always_inline)) {
    bf16x8 vf[KS][NCT];
    f32x16 dP[NCT];
    far_read(Vrow, vf);
    const float st = Stb[(tk & 31) * 32 + ln];
    __builtin_amdgcn_sched_barrier(0);
    far_products(vf, dP);
    far_reduce(dP, st, tk);
  };

  // A key step inside the content window
  f32x16 Bc[NCT];
  bf16x8 Qu[KS];
  auto near_step = [&](const unsigned char* Vrow, int tk) __attribute__((always_inline)) {
    Vrow += second ? 32 * ROWB : 0;
    const unsigned char* Krow = Vrow + TILE;
    const float off2 = Stb[((tk - tk_first) & 31) * 32 + ln];
    float gt = 0.f;
    // A branch between the tiles where a wave has 512 registers: without it the two are mixed, which takes 36 registers
    // more and their copies from the accumulation half (window launch at Dh 128, T 512, 128 channels: 1045 against 990 us).
    int tiles = NCT;
    if constexpr (SOLO) asm volatile("" : "+s"(tiles));
#pragma unroll
    for (int t = 0; t < NCT; ++t) {               // one key-channel tile at a time: fewer live tiles
      if (t > 0 && LAST) break;                   // tile 0 is this wave's
      if (t >= tiles) break;
      // A wave that has its SIMD to itself sends out every LDS read of a phase before the first product or
      // exponential of it: read where they are used, each pair of fragments waits out the LDS latency (last time
      // step of 512: 512 such steps, the longest chain of the launch; 4.92 -> 4.64 ms at B1 H16 C64 of 128 Dh128).
      // Two waves cover each other's waits (read ahead at Dh 64: 786 us and 16 registers spilled against 785).
      const unsigned char *Kt = Krow + t * 32 * ROWB, *Vt = Vrow + t * 32 * ROWB;
      bf16x8 kf[KS], vf[KS], kt[2][MT];
      if constexpr (SOLO) {
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) {
          kf[ks] = *(const bf16x8*)(Kt + r_lane[ks]);
          vf[ks] = *(const bf16x8*)(Vt + r_lane[ks]);
        }
        __builtin_amdgcn_sched_barrier(0);
      }
      f32x16 S = Bc[t], dP;
      // dP - delta: the subtraction is the product's C operand (16 registers more)
#pragma unroll
      for (int i = 0; i < 16; ++i) dP[i] = SOLO ? -delta : 0.f;
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) {
        S = __builtin_amdgcn_mfma_f32_32x32x16_bf16(SOLO ? kf[ks] : *(const bf16x8*)(Kt + r_lane[ks]), Qu[ks], S, 0, 0, 0);
        dP = __builtin_amdgcn_mfma_f32_32x32x16_bf16(SOLO ? vf[ks] : *(const bf16x8*)(Vt + r_lane[ks]), dOf[ks], dP, 0, 0, 0);
      }
      if constexpr (SOLO) {
#pragma unroll
        for (int s = 0; s < 2; ++s)
#pragma unroll
          for (int mt = 0; mt < MT; ++mt) kt[s][mt] = tr_frag(Krow, t, s, mt);
        __builtin_amdgcn_sched_barrier(0);
      }
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        const float p = __builtin_amdgcn_exp2f(S[i] + off2);        // masked keys: exp2(-inf) = 0
        const float ds = p * (SOLO ? dP[i] : dP[i] - delta);
        S[i] = ds;
        dSc[t][i] += ds;
        gt += ds;
      }
#pragma unroll
      for (int s = 0; s < 2; ++s) {
        const bf16x8 dsf = pack8(S, 8 * s);
#pragma unroll
        for (int mt = 0; mt < MT; ++mt)
          dq[mt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(SOLO ? kt[s][mt] : tr_frag(Krow, t, s, mt), dsf, dq[mt], 0, 0, 0);
      }
    }
    gt = xhalf_sum(gt);
    g_lane[((tk - tk_first) & 31) ^ g_swz] = gt;
  };

  // far steps first, then the steps inside the window; waves that are done keep the ring and the barriers going
  int tk = tk_lo;
  if constexpr (PHASE != WIN && !LAST) {
    // Two steps per barrier, two units on their way.  With a barrier a step the two waves of a SIMD read, multiply and
    // reduce at the same time, and the three add up (T 512, 128 channels of Dh 128: 2.80 ms a launch, 2.47 .. 2.56
    // with half the barriers).
    for (; tk < far_lim; tk += 2) {
      const unsigned char* Vrow = begin_unit(tk);
      if (tk >= far_end) continue;
      if ((tk & 31) == 0) time_slab(tk);
      if (PHASE == FAR || tk + 1 >= min(far_lim, far_end)) {
        far_one(Vrow, tk);
        if (tk + 1 < min(far_lim, far_end)) far_one(Vrow + TILE, tk + 1);
      } else {
        // the second step's products run while the first one's are reduced
        bf16x8 vf[KS][NCT];
        f32x16 dPa[NCT], dPb[NCT];
        far_read(Vrow, vf);
        const float sa = Stb[(tk & 31) * 32 + ln], sb = Stb[((tk & 31) + 1) * 32 + ln];
        __builtin_amdgcn_sched_barrier(0);
        far_products(vf, dPa);
        far_read(Vrow + TILE, vf);
        __builtin_amdgcn_sched_barrier(0);
        far_products(vf, dPb);
        far_reduce(dPa, sa, tk);
        far_reduce(dPb, sb, tk + 1);
      }
    }
    tk = far_lim;
  }
  if constexpr (PHASE == ONE && !LAST)
    for (; tk < far_end; ++tk) {                  // far for this wave, not for the workgroup
      const unsigned char* Vrow = begin_unit(tk);
      time_slab(tk);
      far_one(Vrow, tk);
    }
  // the far steps' share of the channel-table gradient; from here on the tile holds the bias
#pragma unroll
  for (int t = 0; t < NCT; ++t)
#pragma unroll
    for (int i = 0; i < 16; ++i) dSc[t][i] = Ec[t][i] * (dSc[t][i] - delta * esum);
  if constexpr (PHASE != FAR) {
  // Bc = log2(Ec): the table it was gathered from lies under the slabs by now (-inf where
  // Ec = 0: masked keys, and biases more than 126 octaves below the row's largest)
#pragma unroll
  for (int t = 0; t < NCT; ++t)
#pragma unroll
    for (int i = 0; i < 16; ++i) Bc[t][i] = __builtin_amdgcn_logf(Ec[t][i]);
  if (second) Bc[0] = Bc[NCT - 1];
#pragma unroll
  for (int ks = 0; ks < KS; ++ks)
    Qu[ks] = qfrag(*(const u32x4*)(qrow + ks * 16 + hh * 8), *(const u32x4*)(bu + ks * 16 + hh * 8), sc2);
  for (; tk <= tq_hi; ++tk) {
    const unsigned char* Vrow = begin_unit(tk);
    if (active && tk >= far_end && tk <= tq) {
      time_slab(tk);
      near_step(Vrow, tk);
    }
  }
  }

  if constexpr (LAST) lds_barrier();
  else wave_sync_lds();
  const int tk_end = PHASE == FAR ? far_end : tq + 1;
  if (active && tk_end > tk_first) flush_slab(tk_first + ((tk_end - 1 - tk_first) & ~31));
  lds_barrier();                                  // from here on the waves share out the whole of the LDS
  if (!active) return;

  // channel-table gradient: element (ck) of query cq goes to column C-1-|cq-ck|, so column
  // C-1-d collects the two key channels cq-d and cq+d (those of them that this launch holds).
  // The tile goes to a per-wave table [32 queries][PC] by local key channel, and each output row
  // is gathered from it (LDS float atomics for the scatter form were measured at ~0.3 us apiece).
  // The column behind the last channel, and the one before the first, is zero: key channels that this launch does
  // not hold.
  constexpr int SHARE = QUERY_LDS<DH, NCT, PHASE> / NW / 4;
  float* share = (float*)smem + wave * SHARE;
  float* tab = share - (second ? NCT * SHARE : 0) + 1;
#pragma unroll
  for (int t = 0; t < NCT; ++t) {
    if (t > 0 && LAST) break;
    const int col = second ? 32 : t * 32;
#pragma unroll
    for (int i = 0; i < 16; ++i) tab[ln * PC + col + (i >> 2) * 8 + hh * 4 + (i & 3)] = dSc[t][i] * a.sm_scale;
  }
  if (!second) {
    tab[ln * PC + CP] = 0.f;
    if (lane == 0) tab[-1] = 0.f;
  }
  // two waves of one query tile: the first stores the sum of their dq, the second the table of both
  if (second) {
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
      for (int i = 0; i < 16; ++i) share[(mt * 16 + i) * 64 + lane] = dq[mt][i];
  }
  if constexpr (LAST) lds_barrier();
  else wave_sync_lds();
  // dq^T[d][q]: this lane's query, d = 32mt + 8a4 + 4hh + 0..3
  if (PHASE != FAR && qok && !second) {
    const float* other = share + NCT * SHARE + lane;
    float* dqo = a.dq + row * DH;
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
      for (int a4 = 0; a4 < 4; ++a4)
      {
        float4* dst = (float4*)(dqo + mt * 32 + a4 * 8 + hh * 4);
        float v[4];
#pragma unroll
        for (int x = 0; x < 4; ++x) {
          v[x] = dq[mt][a4 * 4 + x];
          if (LAST) v[x] += other[(mt * 16 + a4 * 4 + x) * 64];
          v[x] *= a.sm_scale;
        }
        float4 val = make_float4(v[0], v[1], v[2], v[3]);
        if (accum) {
          const float4 old = *dst;
          val = make_float4(val.x + old.x, val.y + old.y, val.z + old.z, val.w + old.w);
        }
        *dst = val;
      }
  }
  if (LAST && !second) return;
  for (int c0 = 0; c0 < C_; c0 += 64) {
    const int col = c0 + lane;
    const int d = C_ - 1 - col;                   // this lane's column holds distance d
    const int lo = cqw0 - k0 - d, hi = d > 0 ? cqw0 - k0 + d : CP;           // local key channels of query 0 (d = 0: one)
    float* dst = a.dbias_chan + wrow0 * C_ + col;
    if (col < C_) {
#pragma unroll 8
      for (int q = 0; q < 32; ++q) {
        const float g = tab[q * PC + min(max(lo + q, -1), CP)] + tab[q * PC + min(max(hi + q, -1), CP)];
        if (q < nq_live) {
          if (accum || PHASE == WIN) atomicAdd(dst + q * C_, g);
          else dst[q * C_] = g;
        }
      }
    }
  }
}

template <int DH, int NCT, int PHASE>
__global__ __launch_bounds__((PHASE_WAVES<PHASE> * 64), (PHASE_OCC<DH, PHASE>)) void mvpa_bwd_query_mfma_kernel(mvpa_bwd_args a, int q0, int k0, int accum) {
  const bool has_content = a.flags & MVPA_FLAG_CONTENT;
  const int nt = query_tiles<DH, NCT, PHASE>(a.T, has_content);
  // blocks go round-robin over the 8 XCDs: keep the tiles of one (b,h) on one XCD (they walk the
  // same K and V in step, so its L2 serves all but the first), long tiles first.  The tile with
  // the last time step runs longest: all of those go first, or the last of them would end the launch alone.
  const int nbh = a.B * a.H;
  int bh, tile;
  {
    const int L = blockIdx.x;
    if (nt == 1) {
      bh = L;
      tile = 0;
    } else if (L < nbh) {
      bh = L;
      tile = nt - 1;
    } else {
      // (an XCD's first walk takes no turns; with / without: B1 H16/8 C64 T128 Dh128 1265 / 1247 us, B2 H16 C64 T64 Dh64 364 / 355)
      deal_walks(L - nbh, nbh, nt - 1, DH == 64 ? 64 : 32, 1, bh, tile);
      tile = nt - 2 - tile;
    }
  }
  if constexpr (LAST_APART<DH, NCT, PHASE>)
    if (has_content && tile == nt - 1) {
      query_walk<DH, NCT, PHASE, true>(a, q0, k0, accum, bh, tile);
      return;
    }
  query_walk<DH, NCT, PHASE, false>(a, q0, k0, accum, bh, tile);
}

}  // namespace bwdq
}  // namespace mvpa

// 1 if the MFMA query pass can serve these (already validated) arguments
int mvpa_bwd_query_mfma_supported(const mvpa_bwd_args* a) {
  if (a->dtype != MVPA_BF16 || (a->Dh != 64 && a->Dh != 128) || a->C > 128) return 0;
  if (!(a->flags & MVPA_FLAG_CAUSAL) || a->key_bias || !a->ws_qu) return 0;
  const uintptr_t p = (uintptr_t)a->q | (uintptr_t)a->k | (uintptr_t)a->v | (uintptr_t)a->o |
                      (uintptr_t)a->d_o | (uintptr_t)a->bias_u | (uintptr_t)a->bias_v |
                      (uintptr_t)a->bias_z | (uintptr_t)a->k_time | (uintptr_t)a->k_chan |
                      (uintptr_t)a->dq | (uintptr_t)a->ws_qu | (uintptr_t)a->ws_chan |
                      (uintptr_t)a->dk | (uintptr_t)a->dv;
  const int64_t s = a->q_stride_b | a->q_stride_h | a->q_stride_n | a->k_stride_b | a->k_stride_h |
                    a->k_stride_n | a->v_stride_b | a->v_stride_h | a->v_stride_n |
                    a->o_stride_b | a->o_stride_h | a->o_stride_n | a->do_stride_b |
                    a->do_stride_h | a->do_stride_n;
  if ((p & 15) || (s & 7)) return 0;
  // row offsets within one time step are kept in 32 bits inside the kernels
  const int64_t big = (int64_t)1 << 31;
  if (a->C * a->q_stride_n >= big || a->C * a->k_stride_n >= big || a->C * a->v_stride_n >= big ||
      a->C * a->do_stride_n >= big || a->q_stride_n < 0 || a->k_stride_n < 0 || a->v_stride_n < 0 ||
      a->do_stride_n < 0)
    return 0;
  return 1;
}

template <int DH, int NCT, int PHASE>
static void launch_query(const mvpa_bwd_args* a, hipStream_t stream, int q0, int k0, int accum) {
  using namespace mvpa::bwdq;
  constexpr int nw = PHASE_WAVES<PHASE>;
  const int nt = query_tiles<DH, NCT, PHASE>(a->T, a->flags & MVPA_FLAG_CONTENT);
  constexpr size_t lds = QUERY_LDS<DH, NCT, PHASE>;
  static_assert(lds <= 160 * 1024 / (DH == 64 ? 2 : 1), "query-pass ring exceeds the LDS");
  dim3 grid((unsigned)(nt * a->B * a->H));
  auto kern = mvpa_bwd_query_mfma_kernel<DH, NCT, PHASE>;
  mvpa::want_dynamic_lds((const void*)kern, (int)lds);
  MVPA_LAUNCH(kern, grid, dim3(nw * 64), lds, stream, *a, q0, k0, accum);
}

// ==========================================================================================
// The KEY pass: dk, dv.  A workgroup of 4 waves owns consecutive key time steps of one kv head, 2 with two
// channel tiles and 4 with one; a wave owns 32 key channels of one of them (its K and V rows stay in registers as MFMA B
// operands) and walks every query time step tq >= tk of every query head of the group, both
// query-channel tiles in turn.  Products are formed NON-transposed here, S[q][key] = (q+u) K^T,
// so that a lane owns one key and the contraction index of dv^T = dO^T P and dk^T = (q+u)^T dS
// is the register index.  With Ec[q][key] = exp2(channel bias - mc[q]) and, per (query, tk), one
// scalar from the query pass (the exponent e = time bias - L + mc inside the content window,
// exp2(e) outside it):
//     inside :  P = exp2((q+u) K^T + e) o Ec,  dP = dO V^T,  dS = P o (dP - delta[q])
//               dv^T[d][key] += dO^T[d][q] P[q][key],   dk^T[d][key] += (q+u)^T[d][q] dS[q][key]
//     outside:  P = exp2(e) Ec,                dv^T += dO^T P           (dk gets nothing)
// Per (head, tq) one ring stage holds dO, the Ec tile and the scalars, and for steps that are inside the window for
// some wave also (q+u) * scale and delta; direct-to-LDS loads fetch it one or two steps ahead.  The query steps are
// walked from the last one down and the workgroups of one (b, kv head) sit on one XCD: they then read the same stage
// data at about the same time and share it in L2.  MASKED: the query part holds fewer channels than its tiles, padded query rows are cut.
// ==========================================================================================
namespace mvpa {
namespace bwdq {

// Every wave of a workgroup reads the same stage (only the per-key-step scalars differ), and no wave has work on all of
// its steps: with a window of 10 a workgroup of two key steps walks 13 for 12, one of four 15.  At Dh 64 two
// workgroups share a CU, which one copy of dO and (q+u) a stage makes room for (67 KB; with copies for each kind of read
// 8 waves had the CU to themselves): B4 H16 C64 T128 404 -> 340 us, 315 with dv read at the start and not at the end;
// Dh 128, T 512, 32 of 128 channels 279 -> 240 us.  (dk read at the start as well: 250.)
constexpr int KEY_WAVES = 4;
template <int NCT> constexpr int KSTAGES = NCT == 2 ? 2 : 3;      // ring depth

// NEAR: the far steps are left to mvpa_bwd_far_kernel, which has written dv before.
template <int DH, int NCT, bool MASKED, bool NEAR>
__global__ __launch_bounds__(KEY_WAVES * 64, DH == 64 ? 2 : 1) void mvpa_bwd_key_mfma_kernel(mvpa_bwd_args a, mvpa_kv_out out, int k0, int q0, int accum, int per_head) {
  constexpr int KS = DH / 16, MT = DH / 32, ROWB = 2 * DH, CPR = DH / 8;
  constexpr int NW = KEY_WAVES;
  constexpr int CP = NCT * 32, KT = NW / NCT, TILE = CP * ROWB;
  constexpr int CS_BYTES = CP * CP * 4, SC_BYTES = (KT + 1) * 256;
  constexpr int STAGES = KSTAGES<NCT>, STAGE_BYTES = 2 * TILE + CS_BYTES + SC_BYTES;
  constexpr int LPW = TILE / 1024 / NW, CS_LPW = CS_BYTES / 1024 / NW;
  // direct-to-LDS loads per wave and step
  constexpr int LPS_FAR = LPW + CS_LPW + 1, LPS_NEAR = 2 * LPW + CS_LPW + 2;
  // stage layout: dO | Ec | scalars | (q+u)
  constexpr int OFF_DO = 0, OFF_EC = TILE, OFF_SC = TILE + CS_BYTES, OFF_QU = OFF_SC + SC_BYTES;
  extern __shared__ __attribute__((aligned(1024))) unsigned char smem[];

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int ln = lane & 31, hh = lane >> 5;
  const int ktw = wave / NCT, kt = wave % NCT;    // this wave's key step and key-channel tile
  const int T_ = a.T, C_ = a.C, W = a.window, N = a.T * a.C;
  const int CW = (C_ + 3) & ~3;                   // row pitch of the Ec tiles in the workspace
  const bool has_content = a.flags & MVPA_FLAG_CONTENT;
  // per_head: a workgroup takes one query head and dk, dv come per query head ([B,H,N,Dh])
  const int out_heads = per_head ? a.H : a.Hkv, nbg = a.B * out_heads, ntk = (T_ + KT - 1) / KT;
  int bg, tile;
  deal_walks(blockIdx.x, nbg, ntk, DH == 64 ? 64 : 32, 0, bg, tile);     // early key steps (most queries) first
  const int b = bg / out_heads, g = per_head ? bg % out_heads / (a.H / a.Hkv) : bg % out_heads;
  const int grp = per_head ? 1 : a.H / a.Hkv, h0 = per_head ? bg % out_heads : g * grp;
  const int tk0 = tile * KT;
  const int tk = tk0 + ktw;
  const bool wave_on = tk < T_;
  const int tkc = min(tk, T_ - 1);

  const int ck = k0 + kt * 32 + ln;               // key channels k0 .., query channels q0 .. in this launch
  const int ckl = kt * 32 + ln;                   // ... local to the launch
  // Lanes of key channels beyond C own columns of dk / dv that are never stored, and a product's
  // column depends on no other lane's operand: they need no masking.  Padded QUERY rows are the
  // contraction index of both gradient products; their probabilities are cut after packing, with
  // one mask per fragment dword (two queries) kept in registers (per-element predicates were
  // hoisted out of the loop as 32 lane masks and spilled the scalar registers).
  uint32_t qmask[NCT][8];
#pragma unroll
  for (int qt = 0; qt < NCT; ++qt)
#pragma unroll
    for (int w = 0; w < 8; ++w) {
      const int i = 2 * w;                        // elements i, i + 1 of the tile: queries qa, qa + 1
      const int qa = q0 + qt * 32 + (i >> 2) * 8 + hh * 4 + (i & 3);
      qmask[qt][w] = MASKED ? ((qa < C_ ? 0x0000ffffu : 0u) | (qa + 1 < C_ ? 0xffff0000u : 0u)) : 0xffffffffu;
    }
  auto cut = [&](bf16x8 f, int qt, int s) -> bf16x8 {
    if (!MASKED) return f;
    union { bf16x8 b; u32x4 u; } c;
    c.b = f;
#pragma unroll
    for (int w = 0; w < 4; ++w) c.u[w] &= qmask[qt][4 * s + w];
    return c.b;
  };
  const int64_t nk = (int64_t)tkc * C_ + min(ck, C_ - 1);
  const bf16_t* krow = (const bf16_t*)a.k + b * a.k_stride_b + g * a.k_stride_h + nk * a.k_stride_n;
  const bf16_t* vrow = (const bf16_t*)a.v + b * a.v_stride_b + g * a.v_stride_h + nk * a.v_stride_n;
  bf16x8 Kf[KS], Vf[KS];
#pragma unroll
  for (int ks = 0; ks < KS; ++ks) {
    Kf[ks] = as_frag(*(const u32x4*)(krow + ks * 16 + hh * 8));
    Vf[ks] = as_frag(*(const u32x4*)(vrow + ks * 16 + hh * 8));
  }

  // ---- the ring: per-wave source offsets (swizzles applied on the source side)
  int q_off[LPW], d_off[LPW], cs_off[CS_LPW];
#pragma unroll
  for (int i = 0; i < LPW; ++i) {
    const int pc = (wave + NW * i) * 64 + lane;
    const int r = pc / CPR, phys = pc % CPR;
    const int rc = min(q0 + r, C_ - 1);
    q_off[i] = rc * DH + ((phys ^ swz<DH>(r)) << 3);
    d_off[i] = rc * (int)a.do_stride_n + ((phys ^ swz<DH>(r)) << 3);
  }
  // the Ec tile [C][C] lands with a row pitch of CP floats
#pragma unroll
  for (int i = 0; i < CS_LPW; ++i) {
    const int pc = (wave + NW * i) * 64 + lane;   // 16-byte chunk: row pc / (CP/4), 4 columns
    const int r = min(q0 + pc / (CP / 4), C_ - 1), c4 = min((pc % (CP / 4)) * 4, max(CW - k0 - 4, 0));
    cs_off[i] = r * CW + k0 + c4;
  }
  const int sc_lane = min(q0 + lane, C_ - 1);
  const uint32_t ring_lds = (uint32_t)(uintptr_t)(BWD_LDS_PTR(unsigned char))smem;
  // a step is fetched in full when it lies inside the content window of one of the waves
  auto wg_near = [&](int tq) -> bool {
    return has_content && (W <= 0 || tq == T_ - 1 || tq - tk0 <= W + KT - 1);
  };
  // source pointers of the step the ring fetches next: re-based at each head, stepped down by
  // one query time step otherwise (the full address arithmetic per step cost as many scalar
  // instructions as a far step has vector ones)
  const bf16_t* p_do = nullptr;
  const bf16_t* p_qu = nullptr;
  const float* p_ec = nullptr;
  const float* p_sc = nullptr;
  const float* p_de = nullptr;
  const int64_t d_do = (int64_t)C_ * a.do_stride_n, d_sc = (int64_t)T_ * C_;
  const int d_ec = C_ * CW, d_qu = C_ * DH;
  auto rebase = [&](int hq) {
    const int h = h0 + hq;
    const int64_t bhq = (int64_t)b * a.H + h;
    const int64_t r0 = bhq * N + (int64_t)(T_ - 1) * C_;    // first query row of step T-1
    p_do = (const bf16_t*)a.d_o + b * a.do_stride_b + h * a.do_stride_h + (int64_t)(T_ - 1) * d_do;
    p_qu = (const bf16_t*)a.ws_qu + r0 * DH;
    p_ec = a.ws_chan + r0 * CW;
    p_sc = a.ws_time + ((bhq * T_ + (T_ - 1)) * T_ + tkc) * C_;
    p_de = a.ws_delta + r0;
  };
  auto issue_step = [&](int tq, int stage_idx) {
    const uint32_t st = ring_lds + stage_idx * STAGE_BYTES;
#pragma unroll
    for (int i = 0; i < LPW; ++i) dma16(p_do + d_off[i], st + OFF_DO + (wave + NW * i) * 1024);
#pragma unroll
    for (int i = 0; i < CS_LPW; ++i) dma16(p_ec + cs_off[i], st + OFF_EC + (wave + NW * i) * 1024);
    // per-query scalar of this wave's key step
    dma4(p_sc + sc_lane, st + OFF_SC + ktw * 256);
    if (wg_near(tq)) {
#pragma unroll
      for (int i = 0; i < LPW; ++i) dma16(p_qu + q_off[i], st + OFF_QU + (wave + NW * i) * 1024);
      dma4(p_de + sc_lane, st + OFF_SC + KT * 256);
    }
  };

  f32x16 dK[MT], dV[MT];
#pragma unroll
  for (int mt = 0; mt < MT; ++mt)
#pragma unroll
    for (int i = 0; i < 16; ++i) { dK[mt][i] = 0.f; dV[mt][i] = 0.f; }
  const int64_t out_row = ((int64_t)bg * N + (int64_t)tkc * C_ + ck) * DH;
  const bool stores = wave_on && ck < C_;
  if ((NEAR || accum) && stores)                  // launches of one stream: dv goes on from what is there
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
      for (int a4 = 0; a4 < 4; ++a4) {
        const float4 v = *(const float4*)(a.dv + out_row + mt * 32 + a4 * 8 + hh * 4);
        dV[mt][a4 * 4] = v.x; dV[mt][a4 * 4 + 1] = v.y; dV[mt][a4 * 4 + 2] = v.z; dV[mt][a4 * 4 + 3] = v.w;
      }

  int r_lane[KS], t_lane[MT];
  {
    const int e = (ln & 15) >> 2, aa = ln & 3, grp16 = ln >> 4;
    const int row0 = 4 * hh + e;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) r_lane[ks] = ln * ROWB + (((2 * ks + hh) ^ swz<DH>(ln)) << 4);
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
      t_lane[mt] = row0 * ROWB + (((4 * mt + 2 * grp16 + (aa >> 1)) ^ swz<DH>(row0)) << 4) + ((aa & 1) << 3);
  }
  auto tr_frag = [&](const unsigned char* tile_p, int qt, int s, int mt) -> bf16x8 {
    const unsigned char* p = tile_p + (32 * qt + 16 * s) * ROWB;  // eight rows on, bit 1 of the swizzle is the other
    const bf16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4bf16((BWD_LDS_PTR(bf16x4))(p + t_lane[mt]));
    const bf16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4bf16((BWD_LDS_PTR(bf16x4))(p + 8 * ROWB + (t_lane[mt] ^ 32)));
    return __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
  };

  // steps: query heads of the group, and for each the query steps T-1 .. tk0; NEAR: T-1, then top .. tk0,
  // top the last step in the window of one of the waves
  const int top = NEAR ? min(T_ - 2, tk0 + KT - 1 + W) : T_ - 2;
  const int span = top < tk0 ? 1 : top - tk0 + 2, nsteps = grp * span;
  int ihq = 0, itq = T_ - 1;                      // the step the ring fetches next
  rebase(0);
  auto next_issue = [&]() {
    if (--itq < tk0) {
      itq = T_ - 1;
      if (++ihq < grp) rebase(ihq);
    } else {
      p_do -= d_do;
      p_qu -= d_qu;
      p_ec -= d_ec;
      p_sc -= d_sc;
      p_de -= C_;
      if (NEAR && itq == T_ - 2) {                // over the steps that are far for every wave
        const int64_t n = T_ - 2 - top;
        p_do -= n * d_do;
        p_qu -= n * d_qu;
        p_ec -= n * d_ec;
        p_sc -= n * d_sc;
        p_de -= n * C_;
        itq = top;
      }
    }
  };
#pragma unroll
  for (int s = 0; s < STAGES - 1; ++s)
    if (s < nsteps) { issue_step(itq, s); next_issue(); }

  int stage = 0, it = 0, ring_tq = T_ - 1;        // ring_tq: query step of the stage handed out next
  // advances the ring by one step and returns the stage that holds its data
  auto ring_step = [&]() -> const unsigned char* {
    // the step has landed once only the loads of the one younger step are in flight
    const int next_tq = ring_tq - 1 < tk0 ? T_ - 1 : ring_tq == T_ - 1 ? top : ring_tq - 1;
    if (STAGES == 2 || it + 1 >= nsteps) wait_vmcnt_imm<0>();
    else if (wg_near(next_tq)) wait_vmcnt_imm<LPS_NEAR>();
    else wait_vmcnt_imm<LPS_FAR>();
    lds_barrier();            // this step's stage visible to all; the previous one is free
    if (it + STAGES - 1 < nsteps) { issue_step(itq, stage == 0 ? STAGES - 1 : stage - 1); next_issue(); }
    const unsigned char* base = smem + stage * STAGE_BYTES;
    stage = stage + 1 == STAGES ? 0 : stage + 1;
    ring_tq = next_tq;
    ++it;
    return base;
  };

  // ---- a query step outside the content window: P = Ec * exp2(e), dv only
  auto far_step = [&](const unsigned char* base) {
    const unsigned char* Do = base + OFF_DO;
    const float* Ecs = (const float*)(base + OFF_EC) + ckl;
    const float* ET = (const float*)(base + OFF_SC) + ktw * 64;
#pragma unroll
    for (int qt = 0; qt < NCT; ++qt) {
      f32x16 P;
#pragma unroll
      for (int a4 = 0; a4 < 4; ++a4) {
        const int rb = qt * 32 + a4 * 8 + hh * 4;              // query channels rb .. rb+3
        const float4 e4 = *(const float4*)(ET + rb);
        const float es[4] = {e4.x, e4.y, e4.z, e4.w};
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          P[a4 * 4 + j] = Ecs[(rb + j) * CP] * es[j];
        }
      }
#pragma unroll
      for (int s = 0; s < 2; ++s) {
        const bf16x8 pf = cut(pack8(P, 8 * s), qt, s);
#pragma unroll
        for (int mt = 0; mt < MT; ++mt)
          dV[mt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(tr_frag(Do, qt, s, mt), pf, dV[mt], 0, 0, 0);
      }
    }
  };

  // ---- a query step inside the content window
  auto near_step = [&](const unsigned char* base) {
    const unsigned char* Do = base + OFF_DO;
    const unsigned char* Qu = base + OFF_QU;
    const float* Ecs = (const float*)(base + OFF_EC) + ckl;
    const float* TL = (const float*)(base + OFF_SC) + ktw * 64;
    const float* De = (const float*)(base + OFF_SC) + KT * 64;
#pragma unroll
    for (int qt = 0; qt < NCT; ++qt) {
      // the exponent and -delta are the products' C operands; dk takes its factor 1 / log2(e) where it is written
      f32x16 S, dP;
#pragma unroll
      for (int a4 = 0; a4 < 4; ++a4) {
        const int rb = qt * 32 + a4 * 8 + hh * 4;
        const float4 tl = *(const float4*)(TL + rb);
        const float4 de = *(const float4*)(De + rb);
        S[a4 * 4] = tl.x; S[a4 * 4 + 1] = tl.y; S[a4 * 4 + 2] = tl.z; S[a4 * 4 + 3] = tl.w;
        dP[a4 * 4] = de.x; dP[a4 * 4 + 1] = de.y; dP[a4 * 4 + 2] = de.z; dP[a4 * 4 + 3] = de.w;
      }
      bf16x8 qf[KS], df[KS];
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) {
        qf[ks] = *(const bf16x8*)(Qu + r_lane[ks] + qt * 32 * ROWB);
        df[ks] = *(const bf16x8*)(Do + r_lane[ks] + qt * 32 * ROWB);
      }
      __builtin_amdgcn_sched_barrier(0);          // every read out before the first product
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) {
        S = __builtin_amdgcn_mfma_f32_32x32x16_bf16(qf[ks], Kf[ks], S, 0, 0, 0);
        dP = __builtin_amdgcn_mfma_f32_32x32x16_bf16(df[ks], Vf[ks], dP, 0, 0, 0);
      }
      float ec[16];
#pragma unroll
      for (int i = 0; i < 16; ++i) ec[i] = Ecs[(qt * 32 + (i >> 2) * 8 + hh * 4 + (i & 3)) * CP];
      __builtin_amdgcn_sched_barrier(0);
      f32x16& dS = dP;
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        S[i] = __builtin_amdgcn_exp2f(S[i]) * ec[i];
        dS[i] = S[i] * dP[i];
      }
#pragma unroll
      for (int s = 0; s < 2; ++s) {
        const bf16x8 pf = cut(pack8(S, 8 * s), qt, s);
        const bf16x8 sf = cut(pack8(dS, 8 * s), qt, s);
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) {
          dV[mt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(tr_frag(Do, qt, s, mt), pf, dV[mt], 0, 0, 0);
          dK[mt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(tr_frag(Qu, qt, s, mt), sf, dK[mt], 0, 0, 0);
        }
      }
    }
  };

  // this wave's steps of one head, walking down from tq = T-1: the last query step keeps the
  // content term, then the steps beyond the window, then the window, then the steps before tk
  int n_last = 0, n_far = 0, n_win = 0, n_over = 0;
  if (wave_on) {
    const int live = T_ - tk;
    if (NEAR) {
      const int win_top = min(T_ - 2, tk + W);
      n_last = 1;
      n_over = max(0, top - win_top);             // far for this wave, inside the window of another
      n_win = win_top - tk + 1;
    } else if (!has_content) n_far = live;
    else if (W <= 0) n_win = live;
    else {
      n_last = 1;
      n_far = max(0, live - 2 - W);
      n_win = live - 1 - n_far;
    }
  }
  const int n_idle = span - n_last - n_over - n_far - n_win;
  for (int hq = 0; hq < grp; ++hq) {
    for (int n = n_last; n > 0; --n) near_step(ring_step());
    if (NEAR) for (int n = n_over; n > 0; --n) (void)ring_step();
    else for (int n = n_far; n > 0; --n) far_step(ring_step());
    for (int n = n_win; n > 0; --n) near_step(ring_step());
    for (int n = n_idle; n > 0; --n) (void)ring_step();
  }

  // The last of the launches that add to these rows rounds them to the caller's dk and dv where there are such: a
  // lane swaps half of two runs of four columns with its partner and stores eight (a pass over the fp32 results took
  // 61 us at B4 H16 C64 T128).
  if (stores) {
    constexpr float f = 1.f / kLog2e;
    const int64_t n_out = (int64_t)tk * C_ + ck;
    bf16_t* dk_out = (bf16_t*)out.dk + b * out.dk_sb + g * out.dk_sh + n_out * out.dk_sn;
    bf16_t* dv_out = (bf16_t*)out.dv + b * out.dv_sb + g * out.dv_sh + n_out * out.dv_sn;
    auto store8 = [&](bf16_t* dst, const float (&x)[2][4]) {
      union { bf16x2 h[2]; uint32_t w[2]; } p[2];
#pragma unroll
      for (int r = 0; r < 2; ++r)
#pragma unroll
        for (int e = 0; e < 2; ++e) p[r].h[e] = __builtin_convertvector(f32x2{x[r][2 * e], x[r][2 * e + 1]}, bf16x2);
      const auto w0 = __builtin_amdgcn_permlane32_swap(p[0].w[0], p[1].w[0], false, false);
      const auto w1 = __builtin_amdgcn_permlane32_swap(p[0].w[1], p[1].w[1], false, false);
      *(u32x4*)dst = u32x4{w0[0], w1[0], w0[1], w1[1]};
    };
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
      for (int a2 = 0; a2 < 2; ++a2) {
        float vk[2][4], vv[2][4];
#pragma unroll
        for (int r = 0; r < 2; ++r)
#pragma unroll
          for (int x = 0; x < 4; ++x) {
            vk[r][x] = dK[mt][(2 * a2 + r) * 4 + x] * f;
            vv[r][x] = dV[mt][(2 * a2 + r) * 4 + x];
          }
        const int64_t d = out_row + mt * 32 + a2 * 16 + hh * 4;
        if (accum)                                // launches of one stream: the query parts add up
#pragma unroll
          for (int r = 0; r < 2; ++r) {
            const float4 ok = *(const float4*)(a.dk + d + 8 * r);
            vk[r][0] += ok.x; vk[r][1] += ok.y; vk[r][2] += ok.z; vk[r][3] += ok.w;
          }
        if (out.dk) {
          store8(dk_out + mt * 32 + a2 * 16 + hh * 8, vk);
          store8(dv_out + mt * 32 + a2 * 16 + hh * 8, vv);
        } else {
#pragma unroll
          for (int r = 0; r < 2; ++r) {
            *(float4*)(a.dk + d + 8 * r) = make_float4(vk[r][0], vk[r][1], vk[r][2], vk[r][3]);
            *(float4*)(a.dv + d + 8 * r) = make_float4(vv[r][0], vv[r][1], vv[r][2], vv[r][3]);
          }
        }
      }
  }
}


// ==========================================================================================
// The far share of dv: dv^T[d][key] += dO^T[d][q] Ec[q][ck] et[q][tk] over the (query, key) steps outside
// the content window, for 64 query and 64 key channels of a launch.  Nothing else of a far pair enters the key
// pass, so that a wave holds the dv tiles of FR key steps at once: per query step it reads the Ec tile and
// the dO fragments once for all of them.  In the key pass the wave of each key step reads both, three LDS
// cycles for one of the matrix cores: 1.4 us a step with 0.1 us of products at Dh 128.  (Key pass of B1 C128
// T512 Dh128 21.3 -> 11.5 ms, of B4 C64 T128 Dh64 820 -> 690 us; this kernel runs at 0.5 of the matrix cores'
// rate there.)  The scalars et of a key step are one register per 32 queries: lane n of a row of 16 holds the
// n-th query of the tile's register order, and the multiplication takes its operand from there by DPP.
// ==========================================================================================
constexpr int FR = 4;                                            // key steps per wave
template <int DH> constexpr int FAR_WAVES = DH == 64 ? 8 : 4;    // FR tiles of Dh 128 are 256 registers
template <int DH> constexpr int FAR_STAGES = DH == 64 ? 5 : 4;
template <int DH> constexpr int FAR_STAGE_BYTES = 64 * 2 * DH + 64 * 64 * 4 + FR * FAR_WAVES<DH> / 2 * 256;

// x * (the value of lane I of this lane's row of 16)
template <int I>
__device__ inline float times_row_lane(float x, float row) {
  return x * __uint_as_float((uint32_t)__builtin_amdgcn_update_dpp(0, (int)__float_as_uint(row), 0x150 + I, 0xf, 0xf, true));
}
template <int... I>
__device__ inline f32x16 times_row(const float (&x)[16], float row, std::integer_sequence<int, I...>) {
  f32x16 r;
  ((r[I] = times_row_lane<I>(x[I], row)), ...);
  return r;
}

template <int DH>
__global__ __launch_bounds__(FAR_WAVES<DH> * 64) void mvpa_bwd_far_kernel(mvpa_bwd_args a, int k0, int q0, int accum, int per_head) {
  constexpr int MT = DH / 32, ROWB = 2 * DH, CPR = DH / 8, CP = 64, NW = FAR_WAVES<DH>, KT = FR * NW / 2;
  constexpr int TILE = CP * ROWB, OFF_EC = TILE, OFF_SC = TILE + CP * CP * 4;
  constexpr int STAGES = FAR_STAGES<DH>, STAGE_BYTES = FAR_STAGE_BYTES<DH>;
  constexpr int LPW = TILE / 1024 / NW, CS_LPW = CP * CP * 4 / 1024 / NW, SC_LPW = KT / NW, LPS = LPW + CS_LPW + SC_LPW;
  extern __shared__ __attribute__((aligned(1024))) unsigned char smem[];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int ln = lane & 31, hh = lane >> 5;
  const int kt = wave & 1, set = wave >> 1;       // key-channel tile, and which FR key steps
  const int T_ = a.T, C_ = a.C, N = a.T * a.C, CW = (C_ + 3) & ~3;
  const int Wf = a.window, tq_top = T_ - 2;       // far: tq - tk > Wf and tq <= tq_top
  const int out_heads = per_head ? a.H : a.Hkv, nbg = a.B * out_heads;
  // the longest walks (early key steps) first, over all (b, kv head); those of one (b, kv head) on one XCD
  const int bg = blockIdx.x % nbg, tile = blockIdx.x / nbg;
  const int b = bg / out_heads, grp = per_head ? 1 : a.H / a.Hkv, h0 = bg % out_heads * grp;
  const int tk0 = tile * KT, tkw = tk0 + set * FR;
  const int span = max(0, tq_top - (tk0 + Wf)), nsteps = grp * span;   // query steps tq_top .. tk0 + Wf + 1

  int d_off[LPW], cs_off[CS_LPW], sc_off[SC_LPW];
#pragma unroll
  for (int i = 0; i < LPW; ++i) {
    const int pc = (wave + NW * i) * 64 + lane, r = pc / CPR, phys = pc % CPR;
    d_off[i] = min(q0 + r, C_ - 1) * (int)a.do_stride_n + ((phys ^ swz<DH>(r)) << 3);
  }
#pragma unroll
  for (int i = 0; i < CS_LPW; ++i) {
    const int pc = (wave + NW * i) * 64 + lane;
    cs_off[i] = min(q0 + pc / (CP / 4), C_ - 1) * CW + k0 + min((pc % (CP / 4)) * 4, max(CW - k0 - 4, 0));
  }
#pragma unroll
  for (int i = 0; i < SC_LPW; ++i) sc_off[i] = min(tk0 + wave + NW * i, T_ - 1) * C_ + min(q0 + lane, C_ - 1);
  const uint32_t ring_lds = (uint32_t)(uintptr_t)(BWD_LDS_PTR(unsigned char))smem;
  // source pointers of the step the ring fetches next: re-based at each head, stepped down otherwise
  const bf16_t* p_do = nullptr;
  const float *p_ec = nullptr, *p_sc = nullptr;
  const int64_t d_do = (int64_t)C_ * a.do_stride_n, d_sc = (int64_t)T_ * C_;
  const int d_ec = C_ * CW;
  int ihq = 0, itq = tq_top;
  auto rebase = [&]() {
    const int h = h0 + ihq;
    const int64_t bhq = (int64_t)b * a.H + h;
    p_do = (const bf16_t*)a.d_o + b * a.do_stride_b + h * a.do_stride_h + (int64_t)tq_top * d_do;
    p_ec = a.ws_chan + (bhq * N + (int64_t)tq_top * C_) * CW;
    p_sc = a.ws_time + (bhq * T_ + tq_top) * d_sc;
  };
  auto issue_next = [&](int stage_idx) {
    const uint32_t st = ring_lds + stage_idx * STAGE_BYTES;
#pragma unroll
    for (int i = 0; i < LPW; ++i) dma16(p_do + d_off[i], st + (wave + NW * i) * 1024);
#pragma unroll
    for (int i = 0; i < CS_LPW; ++i) dma16(p_ec + cs_off[i], st + OFF_EC + (wave + NW * i) * 1024);
#pragma unroll
    for (int i = 0; i < SC_LPW; ++i) dma4(p_sc + sc_off[i], st + OFF_SC + (wave + NW * i) * 256);
    if (--itq <= tk0 + Wf) {
      itq = tq_top;
      if (++ihq < grp) rebase();
    } else {
      p_do -= d_do;
      p_ec -= d_ec;
      p_sc -= d_sc;
    }
  };

  f32x16 dV[FR][MT];
#pragma unroll
  for (int r = 0; r < FR; ++r)
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
      for (int i = 0; i < 16; ++i) dV[r][mt][i] = 0.f;

  int t_lane[MT];
  {
    const int e = (ln & 15) >> 2, aa = ln & 3, grp16 = ln >> 4, row0 = 4 * hh + e;
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
      t_lane[mt] = row0 * ROWB + (((4 * mt + 2 * grp16 + (aa >> 1)) ^ swz<DH>(row0)) << 4) + ((aa & 1) << 3);
  }
  auto tr_frag = [&](const unsigned char* tile_p, int qt, int s, int mt) -> bf16x8 {
    const unsigned char* p = tile_p + (32 * qt + 16 * s) * ROWB;  // eight rows on, bit 1 of the swizzle is the other
    const bf16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4bf16((BWD_LDS_PTR(bf16x4))(p + t_lane[mt]));
    const bf16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4bf16((BWD_LDS_PTR(bf16x4))(p + 8 * ROWB + (t_lane[mt] ^ 32)));
    return __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
  };
  // the query whose scalar this lane holds: register n = lane & 15 of the product layout
  const int qn = (((lane & 15) >> 2) << 3) + hh * 4 + (lane & 3);
  uint32_t q_mask[2];
#pragma unroll
  for (int qt = 0; qt < 2; ++qt) q_mask[qt] = q0 + qt * 32 + qn < C_ ? 0xffffffffu : 0u;

  rebase();
#pragma unroll
  for (int s = 0; s < STAGES - 1; ++s)
    if (s < nsteps) issue_next(s);
  int stage = 0, tq = tq_top;
  for (int it = 0; it < nsteps; ++it) {
    // the step has landed once only the loads of the younger ones are in flight
    const int left = nsteps - 1 - it;
    if (left >= STAGES - 2) wait_vmcnt_imm<(STAGES - 2) * LPS>();
    else if (left >= 2) wait_vmcnt_imm<2 * LPS>();
    else if (left == 1) wait_vmcnt_imm<LPS>();
    else wait_vmcnt_imm<0>();
    lds_barrier();            // the stage visible to all; the previous one is free
    if (left >= STAGES - 1) issue_next(stage == 0 ? STAGES - 1 : stage - 1);
    const unsigned char* base = smem + stage * STAGE_BYTES;
    const float* Ecs = (const float*)(base + OFF_EC) + kt * 32 + ln;
    const float* Sc = (const float*)(base + OFF_SC) + set * FR * 64 + qn;
#pragma unroll
    for (int qt = 0; qt < 2; ++qt) {
      float ec[16], et[FR];
#pragma unroll
      for (int r = 0; r < FR; ++r) {
        // 0 for padded queries and for the pairs of this step that are not far (their slot holds something else)
        const uint32_t m = tq - (tkw + r) > Wf ? q_mask[qt] : 0u;
        et[r] = __uint_as_float(__float_as_uint(Sc[r * 64 + qt * 32]) & m);
      }
#pragma unroll
      for (int i = 0; i < 16; ++i) ec[i] = Ecs[(qt * 32 + (i >> 2) * 8 + hh * 4 + (i & 3)) * CP];
      bf16x8 df[2][MT];
#pragma unroll
      for (int s = 0; s < 2; ++s)
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) df[s][mt] = tr_frag(base, qt, s, mt);
#pragma unroll
      for (int r = 0; r < FR; ++r) {
        const f32x16 P = times_row(ec, et[r], std::make_integer_sequence<int, 16>{});
#pragma unroll
        for (int s = 0; s < 2; ++s) {
          const bf16x8 pf = pack8(P, 8 * s);
#pragma unroll
          for (int mt = 0; mt < MT; ++mt)
            dV[r][mt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(df[s][mt], pf, dV[r][mt], 0, 0, 0);
        }
      }
    }
    stage = stage + 1 == STAGES ? 0 : stage + 1;
    if (--tq <= tk0 + Wf) tq = tq_top;
  }

  const int ck = k0 + kt * 32 + ln;
#pragma unroll
  for (int r = 0; r < FR; ++r) {
    if (tkw + r >= T_ || ck >= C_) continue;
    float* o = a.dv + (((int64_t)bg * N) + (int64_t)(tkw + r) * C_ + ck) * DH;
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
      for (int a4 = 0; a4 < 4; ++a4) {
        float4* dst = (float4*)(o + mt * 32 + a4 * 8 + hh * 4);
        float4 v = make_float4(dV[r][mt][a4 * 4], dV[r][mt][a4 * 4 + 1], dV[r][mt][a4 * 4 + 2], dV[r][mt][a4 * 4 + 3]);
        if (accum) {
          const float4 old = *dst;
          v = make_float4(v.x + old.x, v.y + old.y, v.z + old.z, v.w + old.w);
        }
        *dst = v;
      }
  }
}

}  // namespace bwdq
}  // namespace mvpa

template <int DH>
static void launch_far(const mvpa_bwd_args* a, hipStream_t stream, int k0, int q0, int accum, int per_head) {
  using namespace mvpa::bwdq;
  constexpr int nw = FAR_WAVES<DH>, kt = FR * nw / 2;
  constexpr size_t lds = (size_t)FAR_STAGES<DH> * FAR_STAGE_BYTES<DH>;
  static_assert(lds <= 160 * 1024, "far-pass ring exceeds the LDS");
  dim3 grid((unsigned)(((a->T + kt - 1) / kt) * a->B * (per_head ? a->H : a->Hkv)));
  auto kern = mvpa_bwd_far_kernel<DH>;
  mvpa::want_dynamic_lds((const void*)kern, (int)lds);
  MVPA_LAUNCH(kern, grid, dim3(nw * 64), lds, stream, *a, k0, q0, accum, per_head);
}

template <int DH, int NCT, bool MASKED, bool NEAR>
static void launch_key(const mvpa_bwd_args* a, const mvpa_kv_out& out, hipStream_t stream, int k0, int q0, int accum, int per_head) {
  using namespace mvpa::bwdq;
  constexpr int nw = KEY_WAVES, cp = NCT * 32, kt = nw / NCT, ROWB = 2 * DH;
  static_assert((size_t)KSTAGES<NCT> * (2 * cp * ROWB + cp * cp * 4 + (kt + 1) * 256) <= 160 * 1024 / (DH == 64 ? 2 : 1), "key-pass ring exceeds the LDS");
  const size_t lds = (size_t)KSTAGES<NCT> * (2 * cp * ROWB + cp * cp * 4 + (kt + 1) * 256);
  dim3 grid((unsigned)(((a->T + kt - 1) / kt) * a->B * (per_head ? a->H : a->Hkv)));
  auto kern = mvpa_bwd_key_mfma_kernel<DH, NCT, MASKED, NEAR>;
  mvpa::want_dynamic_lds((const void*)kern, (int)lds);
  MVPA_LAUNCH(kern, grid, dim3(nw * 64), lds, stream, *a, out, k0, q0, accum, per_head);
}

// Both passes.  Up to 32 channels: one launch each with one channel tile per wave; up to 64: one
// launch each with two.  Beyond that the channels are taken in parts of 64: with the forward's
// log-sum-exp known, the contributions of disjoint key channels (to dq and the bias-table
// gradients) and of disjoint query channels (to dk, dv) simply add up, so every (query part, key
// part) pair is one query-pass launch followed by the key-pass launch that consumes its
// workspace; later launches add to what earlier ones wrote (one stream, hence ordered).
// A key-pass launch takes the (query part, key part) pair of a query-pass launch whole.  At Dh 128 it took quarters of 32 x 32 channels, a
// launch each, whose waves had half the products between two barriers (forward and backward, H16/8, us, quarters / whole: B1 C64 T25 286 / 192,
// B2 C64 T128 2228 / 2066, B1 C100 T40 1434 / 942, B1 C128 T128 4665 / 4195, T512 36.2 / 34.8 ms; three stages instead of two: the same).
// far steps of the longest walk from which the two phases of the query pass are a launch each (Dh 128): the
// set-up of a workgroup is paid twice.  Forward and backward, one launch / two, H16/8: B2 C128 T128 8.39 / 8.82 ms, B1
// C128 T200 9.01 / 9.10, B2 C64 T256 6.40 / 6.37, B1 C128 T300 17.1 / 17.0, T 512 36.4 / 35.8.
constexpr int SPLIT_STEPS = 256;
template <int DH>
static void launch_bwd_parts(const mvpa_bwd_args* a, hipStream_t stream, int per_head, const mvpa_kv_out* out) {
  using namespace mvpa::bwdq;
  const int C = a->C, T = a->T;
  // Far query steps (outside the content window and not the last step) in a kernel of their own where its
  // workgroups, of FAR_KT key steps (16 at Dh 64, 8 at Dh 128; 2 in the key pass), still fill the chip and its walks are long.  Forward and backward, far
  // kernel / without:
  // Dh 64, C 64, T 128: 384 workgroups 1327 / 1495 us, 256: 962 / 1022, 192: 793 / 850, 128: 667 / 589; T 256 of 256:
  // 1480 / 1648; T 64, C 40 of 192: 495 / 495; T 64 of 48: 315 / 272;
  // Dh 128, H16/8, C 64: T 64, 128 workgroups 502 / 453, T 72, 144: 613 / 571, T 80, 160: 688 / 660, T 90, 192: 766 / 780, T 64, 256: 840 / 876, T 128, 256:
  // 1155 / 1289; walks of at most 13 steps (T 25), 256: 541 / 518, 18: 639 / 621, 22: 737 / 725, 28 (C 100): 3169 / 3242.
  constexpr int FAR_KT = FR * FAR_WAVES<DH> / 2;
  const int64_t far_groups = (int64_t)a->B * (per_head ? a->H : a->Hkv) * ((T + FAR_KT - 1) / FAR_KT);
  const bool far = (a->flags & MVPA_FLAG_CONTENT) && a->window > 0 && C > 32 && T - 2 - a->window >= (DH == 64 ? 16 : 24) &&
                   far_groups >= 192;
  const bool split_query = DH == 128 && (a->flags & MVPA_FLAG_CONTENT) && a->window > 0 && T - 2 - a->window >= SPLIT_STEPS;
  auto key_launch = [&](auto near, auto tiles, int kk, int qq, int accum) {
    constexpr bool NEAR = decltype(near)::value;
    constexpr int NCT = decltype(tiles)::value, CP = NCT * 32;
    const mvpa_kv_out to = out && qq + CP >= C ? *out : mvpa_kv_out{};        // the last query part rounds
    const bool full = C - qq >= CP && C - kk >= CP;
    if (full) launch_key<DH, NCT, false, NEAR>(a, to, stream, kk, qq, accum, per_head);
    else launch_key<DH, NCT, true, NEAR>(a, to, stream, kk, qq, accum, per_head);
  };
  // Parts of up to 32 channels in tiles of 32, the existing ones alone; at Dh 64 where a launch on tiles of 64 is two rounds of two workgroups a CU.
  // Tiles of 64 / of 32, us: Dh 128, H16/8 B3 C65 T77 5048 / 4708, B2 C96 T40 1574 / 1429, B1 C80 T25 556 / 578; Dh 64, 480 workgroups (B2 H12 C96
  // T40) 684 / 698, 768 (B2 H12 C75 T64) 1009 / 1033, 960 (B4 H16 C65 T30) 805 / 772, 1200 (B1 H12 C90 T200) 3247 / 3074, 1404 (B3 H12 C65 T77) 1833 / 1645.
  const bool by_32 = DH == 128 || (int64_t)a->B * (per_head ? a->H : a->Hkv) * ((T + 1) / 2) >= 900;
  auto key_launches = [&](auto near, int q0, int k0, bool first_q) {
    if (!by_32 || (C - q0 > 32 && C - k0 > 32)) {
      key_launch(near, std::integral_constant<int, 2>{}, k0, q0, !first_q);
      return;
    }
    for (int kk = k0; kk < min(k0 + 64, C); kk += 32)
      for (int qq = q0; qq < min(q0 + 64, C); qq += 32)
        key_launch(near, std::integral_constant<int, 1>{}, kk, qq, !(first_q && qq == q0));
  };
  if (C <= 32) {
    launch_query<DH, 1, ONE>(a, stream, 0, 0, 0);
    const mvpa_kv_out to = out ? *out : mvpa_kv_out{};
    if (C == 32) launch_key<DH, 1, false, false>(a, to, stream, 0, 0, 0, per_head);
    else launch_key<DH, 1, true, false>(a, to, stream, 0, 0, 0, per_head);
  } else {
    const int parts = (C + 63) / 64;
    for (int kp = 0; kp < parts; ++kp)
      for (int qp = 0; qp < parts; ++qp) {
        if constexpr (DH == 128) {
          if (split_query) {
            launch_query<DH, 2, FAR>(a, stream, qp * 64, kp * 64, kp > 0);
            launch_query<DH, 2, WIN>(a, stream, qp * 64, kp * 64, kp > 0);
          }
        }
        if (!split_query) launch_query<DH, 2, ONE>(a, stream, qp * 64, kp * 64, kp > 0);
        if (far) launch_far<DH>(a, stream, kp * 64, qp * 64, qp > 0, per_head);
        if (far) key_launches(std::true_type{}, qp * 64, kp * 64, qp == 0);
        else key_launches(std::false_type{}, qp * 64, kp * 64, qp == 0);
      }
  }
}

int mvpa_launch_bwd_mfma(const mvpa_bwd_args* a, hipStream_t stream, int per_head, const mvpa_kv_out* out) {
  if (a->Dh == 64) launch_bwd_parts<64>(a, stream, per_head, out);
  else launch_bwd_parts<128>(a, stream, per_head, out);
  return mvpa::take_launch_status();
}
