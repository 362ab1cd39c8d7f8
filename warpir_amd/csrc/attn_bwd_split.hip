// attn_bwd_split.hip -- attention backward for launches too small to fill the
// chip (plain heads): the counterpart of attn_splitkv.hip for the dQ kernel
// (with its Dv and log2-LSE outputs) and the dK/dV kernel of
// warpir_amd.workloads, whose argument layouts these share.
//
// Bound by latency, not by a unit: with few blocks the tiled kernels take one
// wave's walk over all keys (or queries), ~0.9 us per 32 rows at one wave per
// SIMD.  A workgroup takes 32 query (key) rows and its four waves every fourth
// tile of the other side, loaded into the wave's own LDS slots (vmcnt waits, no
// barrier); the fp32 partial sums are added through LDS in wave order and
// rounded once.  Device time, tiled -> here: B1 H8 S512 D64 dQ 14.9 -> 8.0 us,
// dK/dV 17.5 -> 8.3 us; S1024 D128 31.9 -> 17.7 and 36.8 -> 19.9 us.
#include "wir_split.h"

namespace {

using wir::bf16;
using wir::bf16x8;
using wir::f32x4;
using wir::lds_f32x4;
using wir::lds_float;

struct dq_args {   // mha_bwd_dq_prep_*
  wir::gl<bf16> Q, K, V, dO, O;
  wir::gl<float> L;
  int N;
  wir::gl<bf16> dQ;
  wir::gl<float> Dv, L2;
};

struct dkdv_args {   // mha_bwd_dkdv_*
  wir::gl<bf16> Q, K, V, dO;
  wir::gl<float> L2, Dv;
  int N;
  wir::gl<bf16> dK, dV;
};

constexpr int WAVES = wir::SPLIT_WAVES, ROWS = wir::SPLIT_ROWS;

template <int D>
struct Scale {
  static constexpr double inv_sqrt = D == 64 ? 0.125 : 0.08838834764831845;
  static constexpr float s = (float)inv_sqrt, c = (float)(1.4426950408889634 * inv_sqrt);
};

// bf16 of `scale` times the waves' sum, rows row0.. of one head.
template <int D>
__device__ __forceinline__ void store_sum(const lds_float* part, const wir::gl<bf16>& g, int b, int h, int row0,
                                          float scale) {
  const wir::RowStore out(g, b, h, row0, D);
#pragma unroll
  for (int it = 0; it < ROWS * (D / 8) / (WAVES * 64); ++it) {
    const int idx = it * WAVES * 64 + threadIdx.x;
    const int row = idx / (D / 8), ch = idx % (D / 8);
    float acc[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) acc[j] = 0.f;
#pragma unroll
    for (int w = 0; w < WAVES; ++w) {
      const lds_float* p = part + (w * ROWS + row) * wir::split_pitch<D> + ch * 8;
      const f32x4 lo = *(const lds_f32x4*)p, hi = *(const lds_f32x4*)(p + 4);
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        acc[j] += lo[j];
        acc[4 + j] += hi[j];
      }
    }
    bf16x8 v;
#pragma unroll
    for (int j = 0; j < 8; ++j) v[j] = (bf16)(acc[j] * scale);
    out.put8(g, row, ch * 8, v);
  }
}

// Wait for this wave's oldest tile; `more`: another one (of STEP DMAs) is behind it.
template <int STEP>
__device__ __forceinline__ void wait_tile(bool more) {
  if (more)
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(STEP) : "memory");
  else
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
}

template <int D, int KT, bool CAUSAL>
__device__ __forceinline__ void dq_split(const dq_args& args) {
  typedef wir::STile<KT, D, wir::BOTH> TK;
  typedef wir::STile<KT, D, wir::ROWREAD> TV;
  constexpr int STEP = wir::Loader<TK, 1>::INSTR_PER_WAVE + wir::Loader<TV, 1>::INSTR_PER_WAVE;
  constexpr int SLOT = TK::BYTES + TV::BYTES;
  static_assert(STEP < 64 && ROWS * wir::split_pitch<D> * 4 <= 2 * SLOT, "the merge reuses the tiles' LDS");
  __shared__ __attribute__((aligned(1024))) char smem[WAVES * 2 * SLOT];
  int x, h, b;
  wir::split_program<CAUSAL, true>(x, h, b);
  const int row0 = x * ROWS, wave = wir::wave_id();
  const int tiles = ((CAUSAL ? min(args.N, row0 + ROWS) : args.N) + KT - 1) / KT;

  wir::RowFrags<32, 1, D / 16> q, d_o, o;
  wir::load_row_frags_global(q, args.Q, b, h, row0, 0);
  wir::load_row_frags_global(d_o, args.dO, b, h, row0, 0);
  wir::load_row_frags_global(o, args.O, b, h, row0, 0);
  wir::RVec<32, 32> lse, dvec;
  wir::load_rvec(lse, args.L, b, h, row0);
  char* own = smem + wave * 2 * SLOT;
  auto load = [&](int t, int slot) {
    wir::Loader<TK, 1>::template load<true, true>(own + slot * SLOT, args.K, b, h, t * KT, 0, 0);
    wir::Loader<TV, 1>::template load<true, true>(own + slot * SLOT + TK::BYTES, args.V, b, h, t * KT, 0, 0);
  };
  if (wave < tiles) load(wave, 0);
  if (wave + WAVES < tiles) load(wave + WAVES, 1);
  wir::row_dot(dvec, d_o, o);
  lse.v[0] *= 1.4426950408889634f;
  if (wave == 0) {
    wir::store_vec(args.Dv, dvec, b, h, row0, 0);
    wir::store_vec(args.L2, lse, b, h, row0, 0);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // (the loop counts DMAs only)
  }

  wir::RTile<32, 32, D> acc;
  wir::fill(acc, 0.f);
  int slot = 0;
  for (int t = wave; t < tiles; t += WAVES, slot ^= 1) {
    char *kt = own + slot * SLOT, *vt = kt + TK::BYTES;
    wir::RTile<32, 32, KT> s, dp;
    wir::BTile<32, 32, KT> ds;
    wait_tile<STEP>(t + WAVES < tiles);
    wir::mma_ABt_frags<32, 32, KT, TK, D / 16>(s, q, kt, 0);
    if (CAUSAL) wir::causal_mask<false>(s, s, row0, t * KT);
    wir::mma_ABt_frags<32, 32, KT, TV, D / 16>(dp, d_o, vt, 0);
#pragma unroll
    for (int cb = 0; cb < KT / 32; ++cb)
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        const float p = __builtin_amdgcn_exp2f(__builtin_fmaf(s.f[cb][0][i], Scale<D>::c, -lse.v[0]));
        s.f[cb][0][i] = p * (dp.f[cb][0][i] - dvec.v[0]);
      }
    wir::to_bf16(ds, s);
    wir::mma_rAB<32, 32, KT, D, TK>(acc, ds, kt, 0);
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");   // the slot is read: refill it
    if (t + 2 * WAVES < tiles) load(t + 2 * WAVES, slot);
  }
  wir::wait_vm_barrier<0>();
  lds_float* part = (lds_float*)wir::lds(smem);
  wir::put_partial<D>(part, acc, wave);
  wir::barrier();
  store_sum<D>(part, args.dQ, b, h, row0, Scale<D>::s);
}

template <int D, int QT, bool CAUSAL>
__device__ __forceinline__ void dkdv_split(const dkdv_args& args) {
  typedef wir::STile<QT, D, wir::BOTH> T;
  typedef wir::Loader<T, 1> Load;
  typedef wir::VecLoader<QT, 1> LoadVec;
  constexpr int STEP = 2 * Load::INSTR_PER_WAVE + 2;
  constexpr int VEC = 2 * T::BYTES, SLOT = VEC + 512;   // Q, dO, then 256 bytes each for the LSE and Dv
  constexpr int PART = WAVES * ROWS * wir::split_pitch<D>;
  static_assert(STEP < 64 && QT * 4 <= 256 && 2 * PART * 4 <= WAVES * 2 * SLOT, "the merge reuses the tiles' LDS");
  __shared__ __attribute__((aligned(1024))) char smem[WAVES * 2 * SLOT];
  int x, h, b;
  wir::split_program<CAUSAL, false>(x, h, b);
  const int row0 = x * ROWS, wave = wir::wave_id();
  const int first = (CAUSAL ? row0 / QT : 0) + wave, tiles = args.N / QT;

  wir::RowFrags<32, 1, D / 16> k, v;
  wir::load_row_frags_global(k, args.K, b, h, row0, 0);
  wir::load_row_frags_global(v, args.V, b, h, row0, 0);
  char* own = smem + wave * 2 * SLOT;
  auto load = [&](int t, int slot) {
    char* at = own + slot * SLOT;
    Load::template load<true, true>(at, args.Q, b, h, t * QT, 0, 0);
    Load::template load<true, true>(at + T::BYTES, args.dO, b, h, t * QT, 0, 0);
    LoadVec::template load<true>(at + VEC, args.L2, b, h, t * QT, 0);
    LoadVec::template load<true>(at + VEC + 256, args.Dv, b, h, t * QT, 0);
  };
  if (first < tiles) load(first, 0);
  if (first + WAVES < tiles) load(first + WAVES, 1);

  wir::RTile<32, 32, D> dk, dv;
  wir::fill(dk, 0.f);
  wir::fill(dv, 0.f);
  int slot = 0;
  for (int t = first; t < tiles; t += WAVES, slot ^= 1) {
    char *qt = own + slot * SLOT, *dot = qt + T::BYTES;
    wir::RTile<32, 32, QT> s, dp;
    wir::BTile<32, 32, QT> pb, ds;
    wir::CVec<32, QT> lse, dvec;
    wait_tile<STEP>(t + WAVES < tiles);
    wir::load_cvec_lds(lse, qt + VEC, 0);
    wir::load_cvec_lds(dvec, qt + VEC + 256, 0);
    wir::mma_ABt_frags<32, 32, QT, T, D / 16>(s, k, qt, 0);
    if (CAUSAL) wir::causal_mask<true>(s, s, row0, t * QT);
    wir::mma_ABt_frags<32, 32, QT, T, D / 16>(dp, v, dot, 0);
#pragma unroll
    for (int cb = 0; cb < QT / 32; ++cb)
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        const float p = __builtin_amdgcn_exp2f(__builtin_fmaf(s.f[cb][0][i], Scale<D>::c, -lse.v[cb][i]));
        dp.f[cb][0][i] = p * (dp.f[cb][0][i] - dvec.v[cb][i]);
        s.f[cb][0][i] = p;
      }
    wir::to_bf16(pb, s);
    wir::to_bf16(ds, dp);
    wir::mma_rAB<32, 32, QT, D, T>(dv, pb, dot, 0);
    wir::mma_rAB<32, 32, QT, D, T>(dk, ds, qt, 0);
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");   // the slot is read: refill it
    if (t + 2 * WAVES < tiles) load(t + 2 * WAVES, slot);
  }
  wir::wait_vm_barrier<0>();
  lds_float* part = (lds_float*)wir::lds(smem);
  wir::put_partial<D>(part, dk, wave);
  wir::put_partial<D>(part + PART, dv, wave);
  wir::barrier();
  store_sum<D>(part, args.dK, b, h, row0, Scale<D>::s);
  store_sum<D>(part + PART, args.dV, b, h, row0, 1.0f);
}

}  // namespace

WIR_SPLIT_KERNEL(wir_attn_dq_split_d64, dq_args, (dq_split<64, 64, false>))
WIR_SPLIT_KERNEL(wir_attn_dq_split_d64_causal, dq_args, (dq_split<64, 64, true>))
WIR_SPLIT_KERNEL(wir_attn_dq_split_d128, dq_args, (dq_split<128, 32, false>))
WIR_SPLIT_KERNEL(wir_attn_dq_split_d128_causal, dq_args, (dq_split<128, 32, true>))
WIR_SPLIT_KERNEL(wir_attn_dkdv_split_d64, dkdv_args, (dkdv_split<64, 64, false>))
WIR_SPLIT_KERNEL(wir_attn_dkdv_split_d64_causal, dkdv_args, (dkdv_split<64, 64, true>))
WIR_SPLIT_KERNEL(wir_attn_dkdv_split_d128, dkdv_args, (dkdv_split<128, 32, false>))
WIR_SPLIT_KERNEL(wir_attn_dkdv_split_d128_causal, dkdv_args, (dkdv_split<128, 32, true>))
