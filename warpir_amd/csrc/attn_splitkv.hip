// attn_splitkv.hip -- FlashAttention forward for launches too small to fill
// the chip: O and the natural-log LSE of Q, K, V [B, H, S, D], as
// warpir_amd.api.attention_forward.
//
// The tiled kernels give a wave 32 query rows and every key: with few query
// blocks most CUs are idle and the launch takes one wave's walk over all the
// keys, ~0.85 us per 64 of them, almost all of it the latency of the chain
// LDS read -> MFMA -> softmax -> MFMA at one wave per SIMD.  Here a workgroup
// takes 32 query rows and its four waves take every fourth key tile each, so
// four times the CUs work and the walk is a quarter as long; the waves'
// partial (m, l, O) are merged through LDS at the end.  Device time, tiled ->
// here: B1 H8 S512 D64 10.3 -> 6.0 us, D128 16.6 -> 9.7 us; B1 H8 S1024 D64
// 16.8 -> 9.2 us.
//
// Every wave loads its own K and V tiles into its own two LDS slots, so the
// loop has no barrier: vmcnt waits only.  The price is K and V going to LDS
// once per 32 query rows instead of once per 128, which is why the tiled
// kernels keep every launch that fills the chip (the L2s deliver ~20 TB/s,
// which this kernel reaches at about 40% of the MFMA rate).
//
// The softmax is the exact online one (a running maximum per wave, fp32 sums,
// probabilities rounded to bf16 for the second product), so its error is that
// of the exact tiled kernels; the merge rescales in fp32 and rounds O once.
#include "wir_split.h"

namespace {

using wir::bf16;
using wir::bf16x4;
using wir::bf16x8;
using wir::f32x4;
using wir::lds_f32x4;
using wir::lds_float;

// Arguments: the grouped-query forward's globals (HR = 1 for plain heads).
struct splitkv_args {
  wir::gl<bf16> Q, K, V;
  int N;    // keys (a multiple of 64)
  int HR;   // query heads per key/value head
  wir::gl<bf16> O;
  wir::gl<float> L;
};

constexpr int WAVES = wir::SPLIT_WAVES, ROWS = wir::SPLIT_ROWS;
constexpr float kLn2 = 0.6931471805599453f;

// Wait until at most `n` of this wave's DMAs are in flight (n = 3, 2, 1 or 0
// tiles' worth of STEP, wave-uniform).
template <int STEP>
__device__ __forceinline__ void wait_tiles(int n) {
  if (n >= 3)
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(3 * STEP) : "memory");
  else if (n == 2)
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(2 * STEP) : "memory");
  else if (n == 1)
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(STEP) : "memory");
  else
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
}

// One online-softmax step on the 32 x KT scores of a wave: m, l, o and the
// bf16 probabilities pb.  A row whose scores so far are all -inf keeps l = 0.
template <int KT, int D>
__device__ __forceinline__ void softmax_step(const wir::RTile<32, 32, KT>& s, float& m, float& l,
                                             wir::RTile<32, 32, D>& o, wir::BTile<32, 32, KT>& pb, float c) {
  float x[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) x[j] = s.f[0][0][j];
#pragma unroll
  for (int cb = 0; cb < KT / 32; ++cb)
#pragma unroll
    for (int i = cb == 0 ? 4 : 0; i < 16; ++i) x[i & 3] = fmaxf(x[i & 3], s.f[cb][0][i]);
  const float top = fmaxf(wir::lane_group_reduce<32>(fmaxf(fmaxf(x[0], x[1]), fmaxf(x[2], x[3])), wir::OpMax()), m);
  const float b = top == -__builtin_inff() ? 0.f : -top * c;   // subtracted from the scaled scores
  const float corr = __builtin_amdgcn_exp2f(__builtin_fmaf(m, c, b));
  m = top;
  float part[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int cb = 0; cb < KT / 32; ++cb)
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      bf16x4 v;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const float e = __builtin_amdgcn_exp2f(__builtin_fmaf(s.f[cb][0][4 * g + j], c, b));
        part[j] += e;
        v[j] = (bf16)e;
      }
      pb.f[cb][0][g] = v;
    }
  l = l * corr + wir::lane_group_reduce<32>((part[0] + part[1]) + (part[2] + part[3]), wir::OpAdd());
  if (__builtin_amdgcn_ballot_w64(corr != 1.0f) != 0) {
#pragma unroll
    for (int cb = 0; cb < D / 32; ++cb)
#pragma unroll
      for (int i = 0; i < 16; ++i) o.f[cb][0][i] *= corr;
  }
}

template <int D, int KT, bool CAUSAL>
__device__ __forceinline__ void splitkv(const splitkv_args& args) {
  typedef wir::STile<KT, D, wir::ROWREAD> TK;
  typedef wir::STile<KT, D, wir::TRREAD> TV;
  typedef wir::Loader<TK, 1> LoadK;
  typedef wir::Loader<TV, 1> LoadV;
  constexpr int STEP = LoadK::INSTR_PER_WAVE, SLOT = TK::BYTES + TV::BYTES;
  constexpr int PITCH = wir::split_pitch<D>;
  static_assert(LoadV::INSTR_PER_WAVE == STEP && 3 * STEP < 64, "vmcnt range");
  static_assert(WAVES * (ROWS * PITCH + 2 * ROWS) * 4 <= WAVES * 2 * SLOT, "the merge reuses the tiles' LDS");
  __shared__ __attribute__((aligned(1024))) char smem[WAVES * 2 * SLOT];

  int x, h, b;
  wir::split_program<CAUSAL, true>(x, h, b);
  const int hkv = h / args.HR;
  const int row0 = x * ROWS, wave = wir::wave_id();
  const int keys = CAUSAL ? min(args.N, row0 + ROWS) : args.N;
  const int tiles = (keys + KT - 1) / KT;
  const float c = (float)(1.4426950408889634 / (D == 64 ? 8.0 : 11.313708498984761));   // log2(e) / sqrt(D)

  wir::RowFrags<32, 1, D / 16> q;
  wir::load_row_frags_global(q, args.Q, b, h, row0, 0);
  char* own = smem + wave * 2 * SLOT;
  auto load = [&](int t, int slot) {
    LoadK::template load<true, true>(own + slot * SLOT, args.K, b, hkv, t * KT, 0, 0);
    LoadV::template load<true, true>(own + slot * SLOT + TK::BYTES, args.V, b, hkv, t * KT, 0, 0);
  };
  if (wave < tiles) load(wave, 0);
  if (wave + WAVES < tiles) load(wave + WAVES, 1);

  // the destination's arguments load under the first tiles' (at D = 128 keeping them costs more than
  // the wait at the end: S512 9.8 us against 9.6)
  wir::RowStore out;
  if constexpr (D == 64) out = wir::RowStore(args.O, b, h, row0, D);
  wir::RTile<32, 32, D> o;
  wir::fill(o, 0.f);
  float m = -__builtin_inff(), l = 0.f;
  int slot = 0;
  for (int t = wave; t < tiles; t += WAVES, slot ^= 1) {
    // this wave's DMAs in flight, oldest first: K_t, V_t and, if there is one, K and V of its next tile
    const int next = t + WAVES < tiles ? 2 : 0;
    wir::RTile<32, 32, KT> s;
    wir::BTile<32, 32, KT> pb;
    wait_tiles<STEP>(next + 1);
    wir::mma_ABt_frags<32, 32, KT, TK, D / 16>(s, q, own + slot * SLOT, 0);
    if (CAUSAL) wir::causal_mask<false>(s, s, row0, t * KT);
    softmax_step<KT, D>(s, m, l, o, pb, c);
    wait_tiles<STEP>(next);
    wir::mma_rAB<32, 32, KT, D, TV>(o, pb, own + slot * SLOT + TK::BYTES, 0);
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");   // the slot is read: refill it
    if (t + 2 * WAVES < tiles) load(t + 2 * WAVES, slot);
  }

  // merge: partial O of wave w at part[w][row][col], then m and l of every row
  wir::wait_vm_barrier<0>();
  lds_float* part = (lds_float*)wir::lds(smem);
  lds_float* ml = part + WAVES * ROWS * PITCH;
  wir::put_partial<D>(part, o, wave);
  const int lane = wir::lane_id(), lr = lane % 32, lh = lane / 32;
  if (lh == 0) {
    ml[wave * ROWS + lr] = m;
    ml[(WAVES + wave) * ROWS + lr] = l;
  }
  wir::barrier();

  if constexpr (D == 128) out = wir::RowStore(args.O, b, h, row0, D);
  float* lb = args.L.data + (long long)b * args.L.sb + (long long)h * args.L.sd;
  const int lse_rows = (unsigned)b < (unsigned)args.L.b && (unsigned)h < (unsigned)args.L.d ? args.L.r : 0;
#pragma unroll
  for (int it = 0; it < ROWS * (D / 8) / (WAVES * 64); ++it) {
    const int idx = it * WAVES * 64 + threadIdx.x;
    const int row = idx / (D / 8), ch = idx % (D / 8);
    float top = ml[row];
#pragma unroll
    for (int w = 1; w < WAVES; ++w) top = fmaxf(top, ml[w * ROWS + row]);
    const float base = -top * c;   // (a row of nothing but -inf scores gives NaN, as in the tiled kernels)
    float sum = 0.f, acc[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) acc[j] = 0.f;
#pragma unroll
    for (int w = 0; w < WAVES; ++w) {
      const float f = __builtin_amdgcn_exp2f(__builtin_fmaf(ml[w * ROWS + row], c, base));
      sum += f * ml[(WAVES + w) * ROWS + row];
      const lds_float* p = part + (w * ROWS + row) * PITCH + ch * 8;
      const f32x4 lo = *(const lds_f32x4*)p;
      const f32x4 hi = *(const lds_f32x4*)(p + 4);
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        acc[j] += f * lo[j];
        acc[4 + j] += f * hi[j];
      }
    }
    const float inv = 1.0f / sum;
    bf16x8 v;
#pragma unroll
    for (int j = 0; j < 8; ++j) v[j] = (bf16)(acc[j] * inv);
    out.put8(args.O, row, ch * 8, v);
    if (ch == 0 && row0 + row < lse_rows)
      lb[(long long)(row0 + row) * args.L.sr] = (top * c + __builtin_amdgcn_logf(sum)) * kLn2;
  }
}

}  // namespace

WIR_SPLIT_KERNEL(wir_attn_splitkv_d64, splitkv_args, (splitkv<64, 64, false>))
WIR_SPLIT_KERNEL(wir_attn_splitkv_d64_causal, splitkv_args, (splitkv<64, 64, true>))
WIR_SPLIT_KERNEL(wir_attn_splitkv_d128, splitkv_args, (splitkv<128, 32, false>))
WIR_SPLIT_KERNEL(wir_attn_splitkv_d128_causal, splitkv_args, (splitkv<128, 32, true>))
