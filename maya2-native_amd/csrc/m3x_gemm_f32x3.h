// The fp32 projection on the bf16 matrix cores, shared by the projections (gemm.hip) and the codec's convolutions
// (codec.hip).
#pragma once
#include "m3x_common.h"

// ELU (alpha 1). 16-bit storage: the hardware exp, exp(v) - 1 for v <= 0, absolute error ~1e-7, below the storage
// step of every value it produces. fp32 storage: expm1f, accurate to an ulp of the result near 0 as well.
template <int DT> __device__ __forceinline__ float elu(float v) {
  if constexpr (DT == M3X_F32) return v > 0.f ? v : expm1f(v);
  else return v > 0.f ? v : __expf(v) - 1.f;
}

// Workgroups from which the kernels below have the chip filled enough to beat the fp32 instructions with their K splits
// and smaller tiles (measurements at launch_linear_f32).
constexpr long F32X3_MIN_BLOCKS = 256;

// The conv epilogue: y = act(res + (acc + bias)), bias and res optional, act = ELU when use_elu.
struct F32Epi {
  const float* bias;
  const float* res;
  long ld_res;
  int use_elu;
};

// fp32 projections on the bf16 matrix cores. Each fp32 operand is the sum of three bf16 values, h = bf16(x),
// m = bf16(x - h), l = bf16(x - h - m) (8 significant bits each, 24 in all; exact from 2^-110 up, within 2^-134 below, where l
// and then m fall under bf16's smallest step), and x . w is summed as
// l_x h_w + h_x l_w + m_x m_w + m_x h_w + h_x m_w + h_x h_w in fp32, smallest terms first: six
// v_mfma_f32_16x16x32_bf16 a 16 x 16 x 32 step in place of eight v_mfma_f32_16x16x4_f32, 108 cycles instead of 259. The
// products left out (m l, l m, l l) are below 2^-25 of the whole, and the accumulators round six times per 32 products
// instead of eight: against 64 bits the relative error of a product of N(0, 1) rows is
// 2.3e-7 at K = 256 and 9.3e-7 at K = 3584, where the fp32 instructions give 2.9e-7 and 1.07e-6 (MI355X; about the
// same for ELU outputs, lower for rows with an offset).
//
// A workgroup of 4 waves (WR along the rows, 4 / WR along the columns) owns 16 RT WR rows, a wave 16 RT x 16 CT. Per k step
// every thread splits its share of both operands once and stores the three planes to LDS as fragments (a lane's 16 bytes in lane order; the
// activations' slots XOR-swizzled so that 4 threads of a row and 4 rows hit 16 bank groups), so the split's VALU work
// is shared by the four waves and each fragment read is one contiguous 1 KB. The next step's global loads are in
// flight while the current one multiplies; one small LDS buffer, so that several workgroups a CU overlap one's staging
// with another's products. Weights kept in registers as planes split at load time, double-buffered LDS and 8 waves
// a workgroup were each measured and no faster: the CU's L1 path, LDS and VALU are all about half busy.
//
// EPI 2 is m3x_conv_gemm's epilogue: bias, shortcut and ELU on the accumulators.
//
// Results that the split cannot give as fp32 would are taken from the fp32 instructions, element by element (redo_unsure):
// those that are not finite (an infinity or NaN in the operands, or a value that bf16(x) rounds to infinity), and those
// below 2^-48, where what the split loses of operands below 2^-110 (up to 2^-134 times the other operand's sum) may be more
// than fp32's rounding: x of 2^-126 N(0, 1) came out 2e-3 off, 2.9e-7 in fp32. A sum of exactly zero stands: it is a row of
// zeros or a cancellation (one in 10^7 to 10^8 sums, each of which would hold its launch up by a redone tile: 12.7 -> 16.3 us
// at 19200 x 64 x 256); if its operands are below 2^-110 all the same, it is off by up to the 2^-134 above, and operands
// below 2^-134, deep in fp32's subnormals, count as zero.
__device__ __forceinline__ void split_bf16x3(const f32x8& x, u16x8& h, u16x8& m, u16x8& l) {
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    const uint16_t a = f2bf(x.v[e]);
    const float r = x.v[e] - bf2f(a);
    const uint16_t b = f2bf(r);
    h.v[e] = a;
    m.v[e] = b;
    l.v[e] = f2bf(r - bf2f(b));
  }
}

// The six products of one k step of a weight tile (planes w) with RT row tiles (planes b), smallest terms first.
template <int RT>
__device__ __forceinline__ void mfma_x3(const u16x8 (&w)[3], const u16x8 (&b)[RT][3], f32x4_t (&acc)[RT]) {
  constexpr int PW[6] = {2, 0, 1, 1, 0, 0}, PX[6] = {0, 2, 1, 0, 1, 0};
#pragma unroll
  for (int i = 0; i < 6; ++i)
#pragma unroll
    for (int t = 0; t < RT; ++t) acc[t] = mfma16x16x32<M3X_BF16>(w[PW[i]], b[t][PX[i]], acc[t]);
}

// Whether a split sum may be worse than fp32's: it is not finite, or below 2^-48 and not zero.
constexpr uint32_t SPLIT_SMALL = (127 - 48) << 23;  // 2^-48 as bits
__device__ __forceinline__ bool split_unsure(float v) {
  const uint32_t a = __float_as_uint(v) & 0x7fffffffu;
  return a - SPLIT_SMALL >= 0x7f800000u - SPLIT_SMALL && a != 0;
}

// Such elements of a wave's CT x RT tiles, taken from the fp32 instructions (wt(a, s), xt(s, t): the fragments of k step s); the
// others keep their sums, so that an element depends on its own row and column alone. Called by a whole wave.
template <int CT, int RT, class WT, class XT>
__device__ __forceinline__ void redo_unsure(f32x4_t (&acc)[CT][RT], int ksteps, WT wt, XT xt) {
  // most tiles hold none, nor zeros: 1.5 operations an element (the magnitude from SPLIT_SMALL on, doubled)
  uint32_t far = 0;
#pragma unroll
  for (int a = 0; a < CT; ++a)
#pragma unroll
    for (int t = 0; t < RT; ++t)
#pragma unroll
      for (int r = 0; r < 4; ++r) far = max(far, (__float_as_uint(acc[a][t][r]) << 1) - (SPLIT_SMALL << 1));
  if (!__ballot(far >= (0x7f800000u - SPLIT_SMALL) << 1)) return;
#pragma unroll
  for (int a = 0; a < CT; ++a) {
    bool unsure = false;
#pragma unroll
    for (int t = 0; t < RT; ++t)
#pragma unroll
      for (int r = 0; r < 4; ++r) unsure |= split_unsure(acc[a][t][r]);
    if (!__ballot(unsure)) continue;
    f32x4_t f[RT];
#pragma unroll
    for (int t = 0; t < RT; ++t) f[t] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll 1
    for (int s = 0; s < ksteps; ++s) {
      const f32x8 w = wt(a, s);
#pragma unroll
      for (int t = 0; t < RT; ++t) f[t] = mfma16x16x32_f32(w, xt(s, t), f[t]);
    }
#pragma unroll
    for (int t = 0; t < RT; ++t)
#pragma unroll
      for (int r = 0; r < 4; ++r) acc[a][t][r] = split_unsure(acc[a][t][r]) ? f[t][r] : acc[a][t][r];
  }
}

template <int WR, int RT, int CT, int EPI>  // EPI 0: plain, 1: GELU, 2: the conv epilogue
__global__ __launch_bounds__(256) void linear_f32x3_kernel(const float* __restrict__ X, long ldx,
                                                           const float* __restrict__ Wp, float* Y, long ldy, int M,
                                                           int N, int K, int mblk, int nblk, F32Epi ep) {
  constexpr int XF = RT * WR, WF = CT * 4 / WR;  // fragments a step: activations, weights
  constexpr int XV = XF / 4, WV = (WF + 3) / 4;  // 8-float vectors a thread and step
  static_assert(XF % 4 == 0 && (WF % 4 == 0 || WF < 4), "a fragment a wave and round");
  __shared__ __align__(16) u16x8 lx[3][XF][64], lw[3][WF][64];

  int mb, nb;
  if (!xcd_block(mblk, nblk, mb, nb)) return;  // padding block: the whole workgroup leaves before any barrier

  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);  // wave-uniform: scalar branches around the MFMAs
  const int lane = tid & 63;
  const int li = lane & 15;
  const int lg = lane >> 4;
  const int wr = wave % WR, wc = wave / WR;
  const int ntiles = (N + 15) >> 4;
  const int m0 = mb * 16 * XF;
  const int t0 = nb * WF;
  const int ksteps = K >> 5;

  // activation vector v = tid + 256 j: k group v % 4 of row v / 4, so a row's 128 bytes are read by 4 neighbours; weight
  // vector v: lane v % 64 of fragment v / 64, as packed. Rows past M and tiles past N read a valid place (never stored).
  const float* xp[XV];
#pragma unroll
  for (int j = 0; j < XV; ++j) xp[j] = X + (long)min(m0 + (tid >> 2) + 64 * j, M - 1) * ldx + 8 * (tid & 3);
  const float* wp[WV];
#pragma unroll
  for (int j = 0; j < WV; ++j) wp[j] = Wp + (long)min(t0 + min(wave, WF - 1) + 4 * j, ntiles - 1) * ksteps * 512 + 8 * lane;
  f32x8 xv[XV], wv[WV];
  auto load = [&](int s) {
#pragma unroll
    for (int j = 0; j < XV; ++j) xv[j] = ldv<M3X_F32>(xp[j] + s * 32);
#pragma unroll
    for (int j = 0; j < WV; ++j) wv[j] = ldv<M3X_F32>(wp[j] + (long)s * 512);
  };
  const int xw = 16 * (tid & 3) + (((tid >> 2) & 15) ^ (4 * (tid & 3)));  // the vector's slot in its fragment
  auto store = [&]() {
#pragma unroll
    for (int j = 0; j < XV; ++j)
      split_bf16x3(xv[j], lx[0][wave + 4 * j][xw], lx[1][wave + 4 * j][xw], lx[2][wave + 4 * j][xw]);
#pragma unroll
    for (int j = 0; j < WV; ++j)
      if (WF >= 4 || wave < WF)  // wave-uniform
        split_bf16x3(wv[j], lw[0][wave + 4 * j][lane], lw[1][wave + 4 * j][lane], lw[2][wave + 4 * j][lane]);
  };
  f32x4_t acc[CT][RT];
#pragma unroll
  for (int a = 0; a < CT; ++a)
#pragma unroll
    for (int t = 0; t < RT; ++t) acc[a][t] = f32x4_t{0.f, 0.f, 0.f, 0.f};

  const int xs = 16 * lg + (li ^ (4 * lg));
  load(0);
  for (int s = 0; s < ksteps; ++s) {
    __syncthreads();  // every wave is done reading the previous step
    store();
    __syncthreads();
    if (s + 1 < ksteps) load(s + 1);
    u16x8 b[RT][3];
#pragma unroll
    for (int t = 0; t < RT; ++t)
#pragma unroll
      for (int p = 0; p < 3; ++p) b[t][p] = lx[p][wr * RT + t][xs];
#pragma unroll
    for (int a = 0; a < CT; ++a) {
      u16x8 w[3];
#pragma unroll
      for (int p = 0; p < 3; ++p) w[p] = lw[p][wc * CT + a][lane];
      mfma_x3<RT>(w, b, acc[a]);
    }
  }

  redo_unsure<CT, RT>(
      acc, ksteps,
      [&](int a, int s) {
        return ldv<M3X_F32>(Wp + ((long)min(t0 + wc * CT + a, ntiles - 1) * ksteps + s) * 512 + lane * 8);
      },
      [&](int s, int t) {
        return ldv<M3X_F32>(X + (long)min(m0 + 16 * (wr * RT + t) + li, M - 1) * ldx + s * 32 + 8 * lg);
      });

  const bool vec = (ldy & 3) == 0 && (((uintptr_t)Y) & 15) == 0;
#pragma unroll
  for (int t = 0; t < RT; ++t) {
    const int m = m0 + 16 * (wr * RT + t) + li;
    if (m >= M) continue;
#pragma unroll
    for (int a = 0; a < CT; ++a) {
      const int n = (t0 + wc * CT + a) * 16 + 4 * lg;
      float o[4];
      if constexpr (EPI == 2) {  // N % 16 == 0; ep.res may be Y (a lane reads its four values before it stores them)
        if (n >= N) continue;
        const float4 bb = ep.bias ? *reinterpret_cast<const float4*>(ep.bias + n) : make_float4(0.f, 0.f, 0.f, 0.f);
        const float4 rr =
            ep.res ? *reinterpret_cast<const float4*>(ep.res + (long)m * ep.ld_res + n) : make_float4(0.f, 0.f, 0.f, 0.f);
        const float bv[4] = {bb.x, bb.y, bb.z, bb.w}, rv[4] = {rr.x, rr.y, rr.z, rr.w};
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          float v = acc[a][t][r];
          if (ep.bias) v = v + bv[r];
          if (ep.res) v = rv[r] + v;
          o[r] = ep.use_elu ? elu<M3X_F32>(v) : v;
        }
      } else {
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const float v = acc[a][t][r];
          o[r] = EPI == 1 ? 0.5f * v * (1.0f + erff(v * 0.70710678118654752f)) : v;
        }
      }
      float* yp = Y + (long)m * ldy + n;
      if (vec && n + 3 < N) {
        *reinterpret_cast<float4*>(yp) = make_float4(o[0], o[1], o[2], o[3]);
      } else {
#pragma unroll
        for (int r = 0; r < 4; ++r)
          if (n + r < N) yp[r] = o[r];
      }
    }
  }
}
