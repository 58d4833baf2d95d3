// Mimi one-frame decode (serve/fast_codec.py StaticMimi, :32-277): the kernels around the projections and
// convolutions, which run as GEMMs on m3x_linear. Activations are time-major [rows = seat * T + t, channels] in
// 16-bit with fp32 arithmetic. Every stateful layer keeps one row per slot (the reference's conv_flat / kv /
// key_pos rows); several padding seats of a batch may name the one dummy slot, whose rows are scratch.
#include "m3x_common.h"
#include "m3x_gemm_f32x3.h"

// Stateful kernels split a seat's rows over workgroups (blockIdx.y); the chunk is at least the state's depth, so
// only chunk 0 reads the old state, and chunk 0 alone writes the new state after a barrier. A thread keeps at
// most CODEC_KEEP state values across that barrier.
constexpr int CODEC_THREADS = 256;
constexpr int CODEC_KEEP = 16;

// ---------------------------------------------------------------------------------------------------------
// RVQ decode (:134-149; transformers MimiSplitResidualVectorQuantizer.decode): out[b, :dim] = table_0[code_0]
// (the semantic codebook), out[b, dim:] = dt(table_1[code_1] + ... + table_{nq-1}[code_{nq-1}]) summed in fp32 in
// that order. A GEMM with [W_semantic | W_acoustic] then applies both 1x1 output projections and their sum.
// Codes outside [0, n_codes) are clamped into it (the reference's embedding lookup raises on them).
template <int DT>
__global__ __launch_bounds__(256) void rvq_decode_kernel(const int64_t* __restrict__ codes, long ld_codes,
                                                         const Elt<DT>* __restrict__ tables, Elt<DT>* __restrict__ out,
                                                         long ld_out, int nq, int n_codes, int dim) {
  const int b = blockIdx.x;
  const int64_t* c = codes + (long)b * ld_codes;
  auto code = [&](int q) -> long { return (long)min(max(c[q], (int64_t)0), (int64_t)(n_codes - 1)); };
  for (int d = threadIdx.x; d < dim; d += blockDim.x) {
    out[(long)b * ld_out + d] = tables[code(0) * dim + d];
    float s = 0.f;
    int q = 1;
    for (; q + 8 <= nq; q += 8) {  // eight rows' loads in flight, then added in codebook order
      Elt<DT> v[8];
#pragma unroll
      for (int u = 0; u < 8; ++u) v[u] = tables[((long)(q + u) * n_codes + code(q + u)) * dim + d];
#pragma unroll
      for (int u = 0; u < 8; ++u) s += E<DT>::to_f(v[u]);
    }
    for (; q < nq; ++q) s += E<DT>::to_f(tables[((long)q * n_codes + code(q)) * dim + d]);
    out[(long)b * ld_out + dim + d] = E<DT>::from_f(s);
  }
}

// ---------------------------------------------------------------------------------------------------------
// Upsample (:186-188 -> :112-130): depthwise transposed conv with kernel k <= 2 s, stride s, no bias, one input
// frame per seat: out[b * s + j, c] = x[b, c] w[c, j] + tail[slot, j, c] (j < k - s); the new tail[slot, j - s, c]
// = x[b, c] w[c, j] for j >= s. Each thread owns channels, so its tail reads precede its tail writes.
template <int DT>
__global__ __launch_bounds__(256) void dwconvt_kernel(const Elt<DT>* __restrict__ x, long ld_x,
                                                      const Elt<DT>* __restrict__ w, Elt<DT>* tail, long ld_tail,
                                                      const int64_t* __restrict__ slots, Elt<DT>* __restrict__ out,
                                                      int C, int k, int s) {
  const int b = blockIdx.x;
  Elt<DT>* tl = tail + slots[b] * ld_tail;  // [k - s][C]
  for (int c = threadIdx.x; c < C; c += blockDim.x) {
    const float xv = E<DT>::to_f(x[(long)b * ld_x + c]);
    for (int j = 0; j < s; ++j) {
      const float prev = j < k - s ? E<DT>::to_f(tl[(long)j * C + c]) : 0.f;
      out[((long)b * s + j) * C + c] = E<DT>::from_f(xv * E<DT>::to_f(w[(long)c * k + j]) + prev);
    }
    for (int j = s; j < k; ++j) tl[(long)(j - s) * C + c] = E<DT>::from_f(xv * E<DT>::to_f(w[(long)c * k + j]));
  }
}

// ---------------------------------------------------------------------------------------------------------
// Causal conv input as GEMM rows (:104-111): cols[b * T + t, j * C + c] = joined[t + j * dil][c], where joined =
// the slot's pad = (k - 1) * dil stored frames followed by act(x[b * T + 0 .. T)), act = ELU (alpha 1) when
// use_elu, the ELU module in front of the conv. The slot's state becomes joined's last pad frames (post-ELU, as
// the reference stores the conv's own input). Grid (B, ceil(T / chunk)), chunk >= pad; 8 channels per thread.
// cols == NULL only advances the history (after an m3x_conv_gemm that read it in place of the gathered rows).
template <int DT>
__device__ __forceinline__ V8<DT> joined8(const Elt<DT>* st, const Elt<DT>* x, long ld_x, long row0, int pad, int i,
                                         int c, int C, int use_elu) {
  if (i < pad) return ldv<DT>(st + (long)i * C + c);
  V8<DT> v = ldv<DT>(x + (row0 + i - pad) * ld_x + c);
  if (use_elu) {
#pragma unroll
    for (int e = 0; e < 8; ++e) v.v[e] = E<DT>::from_f(elu<DT>(E<DT>::to_f(v.v[e])));
  }
  return v;
}

template <int DT>
__global__ __launch_bounds__(CODEC_THREADS) void conv_gather_kernel(const Elt<DT>* __restrict__ x, long ld_x,
                                                                    Elt<DT>* state, long ld_state,
                                                                    const int64_t* __restrict__ slots,
                                                                    Elt<DT>* __restrict__ cols, long ld_cols, int T,
                                                                    int C, int k, int dil, int use_elu, int chunk) {
  const int b = blockIdx.x;
  const int t0 = blockIdx.y * chunk, t1 = min(T, t0 + chunk);
  const int pad = (k - 1) * dil;
  const long row0 = (long)b * T;
  Elt<DT>* st = pad ? state + slots[b] * ld_state : nullptr;  // [pad][C]
  const int cv = C / 8, kcv = k * cv;
  for (int e = threadIdx.x; cols && e < (t1 - t0) * kcv; e += CODEC_THREADS) {
    const int t = t0 + e / kcv;
    const int r = e - (t - t0) * kcv;
    const int j = r / cv, c = 8 * (r - j * cv);
    stv<DT>(cols + (row0 + t) * ld_cols + (long)j * C + c, joined8<DT>(st, x, ld_x, row0, pad, t + j * dil, c, C, use_elu));
  }
  if (!pad || blockIdx.y) return;
  V8<DT> keep[CODEC_KEEP / 8];  // constant indices: registers, not a private or LDS array
#pragma unroll
  for (int p = 0; p < CODEC_KEEP / 8; ++p) {
    const int e = threadIdx.x + CODEC_THREADS * p;
    if (e < pad * cv) keep[p] = joined8<DT>(st, x, ld_x, row0, pad, T + e / cv, 8 * (e % cv), C, use_elu);
  }
  __syncthreads();
#pragma unroll
  for (int p = 0; p < CODEC_KEEP / 8; ++p) {
    const int e = threadIdx.x + CODEC_THREADS * p;
    if (e < pad * cv) stv<DT>(st + 8 * e, keep[p]);
  }
}

// ---------------------------------------------------------------------------------------------------------
// Row op: out = act(res + scale * (g + bias)); bias, scale, res may be NULL; act = ELU (alpha 1) when use_elu.
// Serves the conv biases (with the resnet shortcut and the ELU that follows it) and the transformer's
// layer-scaled residuals. C % 8 == 0, 16-byte rows.
template <int DT>
__global__ __launch_bounds__(256) void rows_op_kernel(const Elt<DT>* __restrict__ g, long ld_g,
                                                      const Elt<DT>* __restrict__ bias,
                                                      const Elt<DT>* __restrict__ scale, const Elt<DT>* res,
                                                      long ld_res, Elt<DT>* out, long ld_out, int rows, int C,
                                                      int use_elu) {
  const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  const int cv = C / 8;
  if (i >= (long)rows * cv) return;
  const long r = i / cv;
  const int c = 8 * (int)(i - r * cv);
  const V8<DT> gv = ldv<DT>(g + r * ld_g + c);
  V8<DT> bv = zero_v8<DT>(), sv = zero_v8<DT>(), rv = zero_v8<DT>(), ov;
  if (bias) bv = ldv<DT>(bias + c);
  if (scale) sv = ldv<DT>(scale + c);
  if (res) rv = ldv<DT>(res + r * ld_res + c);
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    float v = E<DT>::to_f(gv.v[e]);
    if (bias) v = v + E<DT>::to_f(bv.v[e]);
    if (scale) v = E<DT>::to_f(sv.v[e]) * v;
    if (res) v = E<DT>::to_f(rv.v[e]) + v;
    if (use_elu) v = elu<DT>(v);
    ov.v[e] = E<DT>::from_f(v);
  }
  stv<DT>(out + r * ld_out + c, ov);
}

// ---------------------------------------------------------------------------------------------------------
// Layer-scaled residual then LayerNorm over rows of 512: h = dt(h + scale * a) (the arithmetic of m3x_rows_op),
// y = dt((h - mean) / sqrt(var + eps) * w + b) with fp32 statistics. One wave per row. Serves the decoder
// transformer's `h = h + layer_scale(a)` followed by the next LayerNorm (serve/fast_codec.py:181-182,172,182).
constexpr int RLN_N = 512;
template <int DT>
__global__ __launch_bounds__(256) void resid_ln_kernel(Elt<DT>* h, long ld_h, const Elt<DT>* __restrict__ a,
                                                       long ld_a, const Elt<DT>* __restrict__ scale,
                                                       const Elt<DT>* __restrict__ w, const Elt<DT>* __restrict__ b,
                                                       Elt<DT>* __restrict__ y, long ld_y, float eps, int rows) {
  const int row = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (row >= rows) return;  // a whole wave; the kernel has no block barrier
  const int c = 8 * (threadIdx.x & 63);
  const V8<DT> hv = ldv<DT>(h + row * ld_h + c), av = ldv<DT>(a + row * ld_a + c), sv = ldv<DT>(scale + c);
  const V8<DT> wv = ldv<DT>(w + c), bv = ldv<DT>(b + c);  // one round trip for every operand
  float v[8];
  V8<DT> ho;
  float sum = 0.f;
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    float t = E<DT>::to_f(sv.v[e]) * E<DT>::to_f(av.v[e]);
    t = E<DT>::to_f(hv.v[e]) + t;
    ho.v[e] = E<DT>::from_f(t);
    v[e] = E<DT>::to_f(ho.v[e]);
    sum += v[e];
  }
  stv<DT>(h + row * ld_h + c, ho);
  const float mean = xor32_sum(xor16_sum(group_sum<16>(sum))) / (float)RLN_N;
  float sq = 0.f;
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    v[e] = v[e] - mean;
    sq += v[e] * v[e];
  }
  const float inv = 1.f / sqrtf(xor32_sum(xor16_sum(group_sum<16>(sq))) / (float)RLN_N + eps);
  V8<DT> yo;
#pragma unroll
  for (int e = 0; e < 8; ++e) yo.v[e] = E<DT>::from_f(v[e] * inv * E<DT>::to_f(wv.v[e]) + E<DT>::to_f(bv.v[e]));
  stv<DT>(y + row * ld_y + c, yo);
}

// ---------------------------------------------------------------------------------------------------------
// Thin GEMM with the conv epilogue, for the SEANet convs with at most 128 output channels:
// y[m, n] = act(res[m, n] + (dt(x[m, :] . w[n, :]) + bias[n])) (m3x_linear's product, then m3x_rows_op's
// arithmetic), w packed by m3x_pack_weight, N = 16 NT, K % 32 == 0; bias and res optional, act = ELU when use_elu.
// Each wave owns 16 MT rows and the 16 NT columns of its column group (blockIdx.y; one group unless the rows alone
// make a small grid): the activation fragments are loaded straight into the MFMA's B operand (read once per column
// group), the weight fragments (cache resident) into A. A column group does not change any output's K order.
// Gathered form (G = 1): the conv's rows are read in place of a gathered copy. Row m = b * T + t, column
// kk = j * C + c of the product is joined[t + j * dil][c] (m3x_conv_gather's rows: the slot's pad stored frames,
// then x with ELU when pre_elu); the caller advances the history afterwards.
struct ConvSrc {
  const void* state;  // Elt<DT> rows
  long ld_state;
  const int64_t* slots;
  int T, C, dil, pad, pre_elu;
};

template <int DT, int NT, int MT, int G>
__global__ __launch_bounds__(256) void conv_gemm_kernel(const Elt<DT>* __restrict__ X, long ldx,
                                                        const Elt<DT>* __restrict__ Wp,
                                                        const Elt<DT>* __restrict__ bias, const Elt<DT>* res,
                                                        long ld_res, Elt<DT>* Y, long ldy, int M, int K,
                                                        int use_elu, ConvSrc cs) {
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int l = threadIdx.x & 63, li = l & 15, lg = l >> 4;
  const long m0 = ((long)blockIdx.x * 4 + wave) * (16 * MT);
  if (m0 >= M) return;  // wave-uniform
  {  // column group blockIdx.y: columns 16 NT y .. 16 NT (y + 1) - 1
    const int n0 = 16 * NT * (int)blockIdx.y;
    Wp += (long)n0 * K;  // NT tiles of K / 32 fragments of 512 elements
    if (bias) bias += n0;
    if (res) res += n0;
    Y += n0;
  }
  f32x4_t acc[NT][MT];
#pragma unroll
  for (int t = 0; t < NT; ++t)
#pragma unroll
    for (int j = 0; j < MT; ++j) acc[t][j] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  const int ks = K / 32;
  // the fragments of step s + 1 are in flight while step s multiplies
  V8<DT> a[2][NT], b[2][MT];
  // gathered form: each row's seat, time and history row
  long xrow0[MT];
  int tt[MT];
  const Elt<DT>* hist[MT];
#pragma unroll
  for (int j = 0; j < MT; ++j) {
    const long row = m0 + 16 * j + li;
    xrow0[j] = 0, tt[j] = 0, hist[j] = nullptr;
    if (G && row < M) {
      const long bs = row / cs.T;
      tt[j] = (int)(row - bs * cs.T);
      xrow0[j] = bs * cs.T;
      hist[j] = cs.pad ? (const Elt<DT>*)cs.state + cs.slots[bs] * cs.ld_state : nullptr;
    }
  }
  auto load = [&](int s, int buf) {
    const int kk = 32 * s + 8 * lg;
    const int tap = G ? kk / cs.C : 0, c = G ? kk - tap * cs.C : 0;
#pragma unroll
    for (int j = 0; j < MT; ++j) {
      const long row = m0 + 16 * j + li;
      b[buf][j] = zero_v8<DT>();
      if (row < M) {
        if (!G) {
          b[buf][j] = ldv<DT>(X + row * ldx + kk);
        } else {
          const int i = tt[j] + tap * cs.dil;
          if (i < cs.pad) {
            b[buf][j] = ldv<DT>(hist[j] + (long)i * cs.C + c);
          } else {
            b[buf][j] = ldv<DT>(X + (xrow0[j] + i - cs.pad) * ldx + c);
            if (cs.pre_elu) {
#pragma unroll
              for (int e = 0; e < 8; ++e) b[buf][j].v[e] = E<DT>::from_f(elu<DT>(E<DT>::to_f(b[buf][j].v[e])));
            }
          }
        }
      }
    }
#pragma unroll
    for (int t = 0; t < NT; ++t) a[buf][t] = ldv<DT>(Wp + ((long)t * ks + s) * 512 + 8 * l);
  };
  load(0, 0);
  for (int s = 0; s < ks; s += 2) {
    if (s + 1 < ks) load(s + 1, 1);
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
      for (int j = 0; j < MT; ++j) acc[t][j] = mfma_k32<DT>(a[0][t], b[0][j], acc[t][j]);
    if (s + 1 >= ks) break;
    if (s + 2 < ks) load(s + 2, 0);
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
      for (int j = 0; j < MT; ++j) acc[t][j] = mfma_k32<DT>(a[1][t], b[1][j], acc[t][j]);
  }
  // lane (li, lg) holds columns 16 t + 4 lg + r of row m0 + 16 j + li. res may be y itself (in place): every
  // residual and bias value of the lane is read before its first store.
#pragma unroll
  for (int j = 0; j < MT; ++j) {
    const long m = m0 + 16 * j + li;
    if (m >= M) continue;
    if constexpr (DT == M3X_F32) {
      float4 bb[NT], rr[NT];
#pragma unroll
      for (int t = 0; t < NT; ++t) {
        const int n = 16 * t + 4 * lg;
        bb[t] = bias ? *reinterpret_cast<const float4*>(bias + n) : make_float4(0.f, 0.f, 0.f, 0.f);
        rr[t] = res ? *reinterpret_cast<const float4*>(res + m * ld_res + n) : make_float4(0.f, 0.f, 0.f, 0.f);
      }
#pragma unroll
      for (int t = 0; t < NT; ++t) {
        const int n = 16 * t + 4 * lg;
        const float bv[4] = {bb[t].x, bb[t].y, bb[t].z, bb[t].w}, rv[4] = {rr[t].x, rr[t].y, rr[t].z, rr[t].w};
        float o[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          float v = acc[t][j][r];
          if (bias) v = v + bv[r];
          if (res) v = rv[r] + v;
          if (use_elu) v = elu<DT>(v);
          o[r] = v;
        }
        *reinterpret_cast<float4*>(Y + m * ldy + n) = make_float4(o[0], o[1], o[2], o[3]);
      }
    } else {
      uint2 bb[NT], rr[NT];
#pragma unroll
      for (int t = 0; t < NT; ++t) {
        const int n = 16 * t + 4 * lg;
        bb[t] = bias ? *reinterpret_cast<const uint2*>(bias + n) : uint2{0, 0};
        rr[t] = res ? *reinterpret_cast<const uint2*>(res + m * ld_res + n) : uint2{0, 0};
      }
#pragma unroll
      for (int t = 0; t < NT; ++t) {
        const int n = 16 * t + 4 * lg;
        const uint16_t* bv = reinterpret_cast<const uint16_t*>(&bb[t]);
        const uint16_t* rv = reinterpret_cast<const uint16_t*>(&rr[t]);
        uint16_t o[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          float v = rnd<DT>(acc[t][j][r]);
          if (bias) v = v + E<DT>::to_f(bv[r]);
          if (res) v = E<DT>::to_f(rv[r]) + v;
          if (use_elu) v = elu<DT>(v);
          o[r] = E<DT>::from_f(v);
        }
        *reinterpret_cast<uint2*>(Y + m * ldy + n) = *reinterpret_cast<const uint2*>(o);
      }
    }
  }
}

// The gathered fp32 conv on the bf16 matrix cores (m3x_gemm_f32x3.h's split and sums; the epilogue as conv_gemm_kernel).
// conv_gemm_kernel reads a row once per tap and repeats the ELU in front of the conv (about 30 instructions an element)
// each time, which bounds it. Here a workgroup owns 128 rows of one seat (blockIdx.x = seat x row block, rows past T
// are dropped) and the 16 CT columns of its column block; per 32 channels it loads the 128 + pad joined rows once,
// applies the ELU and splits them once into LDS, splits the TAPS x CT weight fragments beside them, and multiplies
// all taps from LDS: a tap's fragment is the same rows shifted by tap * dil (row r sits in slot r % 16, XOR-swizzled by
// its k group, of fragment r / 16, so 16 consecutive rows hit 16 bank groups wherever they start). The products add up
// channel block by channel block, taps within.
// 224 seats (MI355X, inside the frame, conv_gemm_kernel against it): 64 -> 32 channels of 1920 rows a seat 128 / 70 us,
// 128 -> 64 of 480 108 / 58, 256 -> 128 of 96 112 / 46. One seat: 4 workgroups 16.6 / 25.7 us, 15 workgroups 10.2 / 12.9, so
// it takes CX_MIN_BLOCKS of them.
constexpr int CX_ROWS = 128, CX_PAD = 16;  // rows a workgroup, most history frames
constexpr long CX_MIN_BLOCKS = 160;

template <int CT, int TAPS>
__global__ __launch_bounds__(256) void conv_x3_kernel(const float* __restrict__ X, long ldx,
                                                      const float* __restrict__ Wp, float* Y, long ldy, int rblk,
                                                      F32Epi ep, ConvSrc cs) {
  constexpr int RT = 2;                               // row tiles a wave: 4 waves x 32 rows
  constexpr int RF = (CX_ROWS + CX_PAD) / 16;         // row fragments in LDS
  constexpr int XV = (RF * 64 + 255) / 256;           // 8-float vectors a thread and channel block
  constexpr int WF = CT * TAPS, WV = (WF + 3) / 4;
  __shared__ __align__(16) u16x8 lx[3][RF][64], lw[3][WF][64];
  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);  // wave-uniform: scalar branches around the MFMAs
  const int lane = tid & 63;
  const int li = lane & 15;
  const int lg = lane >> 4;
  const int bs = blockIdx.x / rblk;
  const int t0 = (blockIdx.x - bs * rblk) * CX_ROWS;
  const int n0 = 16 * CT * blockIdx.y;
  const int cst = cs.C >> 5;       // channel blocks
  const int ks = TAPS * cst;
  const float* xs = X + ((long)bs * cs.T - cs.pad) * ldx;  // joined row i >= pad
  const float* hs = cs.pad ? (const float*)cs.state + cs.slots[bs] * cs.ld_state : X;
  const int rows = min(CX_ROWS, cs.T - t0) + cs.pad;       // joined rows t0 .. t0 + rows - 1
  const int lastw = min(3, (cs.T - t0 - 1) >> 5);          // the waves up to it hold live rows
  const float* wb = Wp + (long)(n0 >> 4) * ks * 512 + 8 * lane;

  f32x8 xv[XV], wv[WV];
  auto load = [&](int cb) {
#pragma unroll
    for (int j = 0; j < XV; ++j) {
      const int i = t0 + min((tid >> 2) + 64 * j, rows - 1);  // rows past the block repeat its last (never stored)
      const int c = 32 * cb + 8 * (tid & 3);
      xv[j] = ldv<M3X_F32>(i < cs.pad ? hs + (long)i * cs.C + c : xs + (long)i * ldx + c);
    }
#pragma unroll
    for (int j = 0; j < WV; ++j) {
      const int f = min(wave + 4 * j, WF - 1);  // [tap][tile]
      wv[j] = ldv<M3X_F32>(wb + ((long)(f % CT) * ks + (f / CT) * cst + cb) * 512);
    }
  };
  f32x4_t acc[CT][RT];
#pragma unroll
  for (int a = 0; a < CT; ++a)
#pragma unroll
    for (int t = 0; t < RT; ++t) acc[a][t] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  load(0);
  for (int cb = 0; cb < cst; ++cb) {
    __syncthreads();  // every wave is done reading the previous channels
#pragma unroll
    for (int j = 0; j < XV; ++j) {
      const int r = (tid >> 2) + 64 * j;
      // wave-uniform: the 16 rows that this wave stores, if a live wave reads them
      if (wave + 4 * j < RF && 16 * (wave + 4 * j) < 32 * (lastw + 1) + cs.pad) {
        if (cs.pre_elu && t0 + r >= cs.pad) {
#pragma unroll
          for (int e = 0; e < 8; ++e) xv[j].v[e] = elu<M3X_F32>(xv[j].v[e]);
        }
        const int s = 16 * (tid & 3) + ((r & 15) ^ (4 * (tid & 3)));
        split_bf16x3(xv[j], lx[0][r >> 4][s], lx[1][r >> 4][s], lx[2][r >> 4][s]);
      }
    }
#pragma unroll
    for (int j = 0; j < WV; ++j)
      if (wave + 4 * j < WF)  // wave-uniform
        split_bf16x3(wv[j], lw[0][wave + 4 * j][lane], lw[1][wave + 4 * j][lane], lw[2][wave + 4 * j][lane]);
    __syncthreads();
    if (cb + 1 < cst) load(cb + 1);
    if (wave > lastw) continue;
#pragma unroll
    for (int tap = 0; tap < TAPS; ++tap) {
      u16x8 b[RT][3];
#pragma unroll
      for (int t = 0; t < RT; ++t) {
        const int r = 16 * (wave * RT + t) + li + tap * cs.dil;
        const int s = 16 * lg + ((r & 15) ^ (4 * lg));
#pragma unroll
        for (int p = 0; p < 3; ++p) b[t][p] = lx[p][r >> 4][s];
      }
#pragma unroll
      for (int a = 0; a < CT; ++a) {
        u16x8 w[3];
#pragma unroll
        for (int p = 0; p < 3; ++p) w[p] = lw[p][tap * CT + a][lane];
        mfma_x3<RT>(w, b, acc[a]);
      }
    }
  }
  if (wave > lastw) return;  // rows past T, never stored (no barrier follows)
  redo_unsure<CT, RT>(
      acc, ks, [&](int a, int s) { return ldv<M3X_F32>(wb + ((long)a * ks + s) * 512); },
      [&](int s, int t) {
        const int tap = s / cst;
        const int i = t0 + min(16 * (wave * RT + t) + li + tap * cs.dil, rows - 1);
        const int c = 32 * (s - tap * cst) + 8 * lg;
        f32x8 x = ldv<M3X_F32>(i < cs.pad ? hs + (long)i * cs.C + c : xs + (long)i * ldx + c);
        if (cs.pre_elu && i >= cs.pad) {
#pragma unroll
          for (int e = 0; e < 8; ++e) x.v[e] = elu<M3X_F32>(x.v[e]);
        }
        return x;
      });
#pragma unroll
  for (int t = 0; t < RT; ++t) {
    const int tr = t0 + 16 * (wave * RT + t) + li;
    if (tr >= cs.T) continue;
    const long m = (long)bs * cs.T + tr;
#pragma unroll
    for (int a = 0; a < CT; ++a) {
      const int n = n0 + 16 * a + 4 * lg;
      const float4 bb = ep.bias ? *reinterpret_cast<const float4*>(ep.bias + n) : make_float4(0.f, 0.f, 0.f, 0.f);
      const float4 rr = ep.res ? *reinterpret_cast<const float4*>(ep.res + m * ep.ld_res + n) : make_float4(0.f, 0.f, 0.f, 0.f);
      const float bv[4] = {bb.x, bb.y, bb.z, bb.w}, rv[4] = {rr.x, rr.y, rr.z, rr.w};
      float o[4];
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        float v = acc[a][t][r];
        if (ep.bias) v = v + bv[r];
        if (ep.res) v = rv[r] + v;
        o[r] = ep.use_elu ? elu<M3X_F32>(v) : v;
      }
      *reinterpret_cast<float4*>(Y + m * ldy + n) = make_float4(o[0], o[1], o[2], o[3]);
    }
  }
}

// ---------------------------------------------------------------------------------------------------------
// Transposed conv overlap-add (:112-130). cols[b * Tin + t, j * C + c] = x[b, t] . W[:, c, j] comes from the GEMM;
// output frame o < Tin * s of seat b is the sum of its contributions (t, j = o - t s, 0 <= j < k) + tail[slot, o, c]
// (o < k - s) + bias[c]; the new tail[slot, i, c] = the contributions to frame Tin * s + i, without bias (the
// reference stores its tail bias-free). Grid (B, ceil(Tin * s / chunk)), chunk >= k - s; 8 channels per thread.
template <int DT>
__device__ __forceinline__ void convt_frame8(const Elt<DT>* cols, long ld_cols, long row0, int o, int c, int Tin,
                                             int C, int k, int s, float (&v)[8]) {
#pragma unroll
  for (int e = 0; e < 8; ++e) v[e] = 0.f;
  for (int t = min(o / s, Tin - 1); t >= 0 && o - t * s < k; --t) {
    const V8<DT> w = ldv<DT>(cols + (row0 + t) * ld_cols + (long)(o - t * s) * C + c);
#pragma unroll
    for (int e = 0; e < 8; ++e) v[e] += E<DT>::to_f(w.v[e]);
  }
}

template <int DT>
__global__ __launch_bounds__(CODEC_THREADS) void convt_overlap_kernel(const Elt<DT>* __restrict__ cols, long ld_cols,
                                                                      Elt<DT>* tail, long ld_tail,
                                                                      const int64_t* __restrict__ slots,
                                                                      const Elt<DT>* __restrict__ bias,
                                                                      Elt<DT>* __restrict__ out, long ld_out, int Tin,
                                                                      int C, int k, int s, int chunk) {
  const int b = blockIdx.x;
  const int nout = Tin * s, ov = k - s;
  const int o0 = blockIdx.y * chunk, o1 = min(nout, o0 + chunk);
  const long row0 = (long)b * Tin;
  Elt<DT>* tl = tail + slots[b] * ld_tail;  // [k - s][C]
  const int cv = C / 8;
  for (int e = threadIdx.x; e < (o1 - o0) * cv; e += CODEC_THREADS) {
    const int o = o0 + e / cv, c = 8 * (e % cv);
    float v[8];
    convt_frame8<DT>(cols, ld_cols, row0, o, c, Tin, C, k, s, v);
    V8<DT> tv = zero_v8<DT>(), bv = zero_v8<DT>(), r;
    if (o < ov) tv = ldv<DT>(tl + (long)o * C + c);
    if (bias) bv = ldv<DT>(bias + c);
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      float y = v[i];
      if (o < ov) y += E<DT>::to_f(tv.v[i]);
      if (bias) y += E<DT>::to_f(bv.v[i]);
      r.v[i] = E<DT>::from_f(y);
    }
    stv<DT>(out + ((long)b * nout + o) * ld_out + c, r);
  }
  if (blockIdx.y) return;
  V8<DT> keep[CODEC_KEEP / 8];  // constant indices: registers, not a private or LDS array
#pragma unroll
  for (int p = 0; p < CODEC_KEEP / 8; ++p) {
    const int e = threadIdx.x + CODEC_THREADS * p;
    if (e < ov * cv) {
      float v[8];
      convt_frame8<DT>(cols, ld_cols, row0, nout + e / cv, 8 * (e % cv), Tin, C, k, s, v);
#pragma unroll
      for (int i = 0; i < 8; ++i) keep[p].v[i] = E<DT>::from_f(v[i]);
    }
  }
  __syncthreads();
#pragma unroll
  for (int p = 0; p < CODEC_KEEP / 8; ++p) {
    const int e = threadIdx.x + CODEC_THREADS * p;
    if (e < ov * cv) stv<DT>(tl + 8 * e, keep[p]);
  }
}

// ---------------------------------------------------------------------------------------------------------
// Decoder transformer attention (:151-184) for T new tokens per seat at positions p = tokens[slot] + t: q and k
// get RoPE (rotate_half; angle p * inv_freq[i] in fp32, cos and sin times rope_scale), k (post-RoPE) and v go to
// the slot's ring entry p % ring with key_pos[slot, p % ring] = p; query p attends the entries with
// p - window < key_pos <= p, softmax at scale 1/sqrt(64). qkv rows [q heads | k heads | v heads] (as many kv heads
// as heads), head_dim 64.
// TM bounds T at compile time, which keeps the unrolled code small.
// One 4-wave workgroup per (seat, head), heads fastest: the 8 heads of a seat, whose rows interleave in the ring, run
// at the same time on the 8 XCDs. Lane (g, d8) of wave w owns dims 8 d8 .. + 7 of ring entries 64 w + g + 8 i (i < 8), of
// the keys and of the values, so every load instruction reads whole rows of 8 lanes and all of them are in flight at
// once, with no branch around them (this call's own entries and entries past the ring are read at a valid place and
// replaced or masked after). A score is 8 products a lane and a sum over the row's 8 lanes (DPP); the lane then holds
// the probability of exactly the value rows it holds, so nothing passes through LDS between softmax and P.V. Each wave
// keeps its own maximum, sum and output over its 64 entries; the four meet in LDS: two barriers in all. One key row a
// thread read whole took 62 us a layer at 224 seats (float32) against 53 now: its loads touched 64 rows of
// 2 KB pitch each, 16 bytes at a time, more lines than the L1 holds. STREAM: the rings of all layers and seats exceed
// the 256 MB memory-side cache, so the rows are read with the non-temporal hint.
// The head-0 workgroup records key_pos; every workgroup knows the positions of the entries this call writes, so none
// depends on another's key_pos write.
constexpr int RA_HD = 64;
constexpr int RA_RING = 256;
constexpr int RA_T = 2;  // tokens per call: Mimi's upsample makes 2 per frame
static_assert(RA_T <= 4, "one wave of the 4-wave workgroup per token");
// K and V bytes of one layer's call from which the rings of a codec's 8 layers pass the 256 MB memory-side cache
constexpr long RA_STREAM_BYTES = 32L << 20;

template <int DT, bool STREAM> __device__ __forceinline__ V8<DT> ld_ring(const Elt<DT>* p) {
  if constexpr (!STREAM) {
    return ldv<DT>(p);
  } else if constexpr (DT == M3X_F32) {
    f32x8 r;
    const u16x8 a = ld16_nt((const uint16_t*)p), c = ld16_nt((const uint16_t*)(p + 4));
    const float4 x = __builtin_bit_cast(float4, a), y = __builtin_bit_cast(float4, c);
    r.v[0] = x.x, r.v[1] = x.y, r.v[2] = x.z, r.v[3] = x.w, r.v[4] = y.x, r.v[5] = y.y, r.v[6] = y.z, r.v[7] = y.w;
    return r;
  } else {
    return ld16_nt(p);
  }
}

template <int DT, int TM, bool STREAM>
__global__ __launch_bounds__(256, STREAM && DT == M3X_F32 ? 3 : 1) void ring_attn_kernel(const Elt<DT>* __restrict__ qkv, long ld_qkv,
                                                        Elt<DT>* kring, Elt<DT>* vring, int64_t* key_pos,
                                                        const int64_t* __restrict__ tokens,
                                                        const int64_t* __restrict__ slots,
                                                        const float* __restrict__ inv_freq, float rope_scale,
                                                        Elt<DT>* __restrict__ out, long ld_out, int T, int H, int ring,
                                                        int window) {
  __shared__ __align__(16) float qs[TM][RA_HD];
  __shared__ float wm[TM][4], wl[TM][4];
  __shared__ int age[RA_RING];  // how many positions an entry lies before token 0 (negative: never visible)
  __shared__ float part[4][TM][RA_HD];
  __shared__ __align__(16) Elt<DT> knew[TM][RA_HD];  // this call's keys (post-RoPE) and values, stored to the
  __shared__ __align__(16) Elt<DT> vnew[TM][RA_HD];  // ring only at the end: reads of them come from here
  const int b = blockIdx.x / H, h = blockIdx.x - b * H;
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), l = tid & 63;
  const long slot = slots[b];
  // wave w < T handles token w: its q, k, v elements do not depend on the position, so they load first
  const int half = RA_HD / 2;
  const int partner = l < half ? l + half : l - half;
  float q_l = 0.f, q_p = 0.f, k_l = 0.f, k_p = 0.f;
  Elt<DT> v_l = 0;
  if (wave < T) {
    const Elt<DT>* r = qkv + ((long)b * T + wave) * ld_qkv;
    q_l = E<DT>::to_f(r[h * RA_HD + l]);
    q_p = E<DT>::to_f(r[h * RA_HD + partner]);
    k_l = E<DT>::to_f(r[(H + h) * RA_HD + l]);
    k_p = E<DT>::to_f(r[(H + h) * RA_HD + partner]);
    v_l = r[(2 * H + h) * RA_HD + l];
  }
  const long p0 = tokens[slot];
  Elt<DT>* kr = kring + slot * (long)ring * H * RA_HD;  // [ring][H][hd]
  Elt<DT>* vr = vring + slot * (long)ring * H * RA_HD;
  int64_t* kp = key_pos + slot * (long)ring;
  const int g = l >> 3, dc = 8 * (l & 7);
  V8<DT> kk[8], vv[8];
  const long kj = kp[min(tid, ring - 1)];
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const int jc = min(64 * wave + g + 8 * i, ring - 1);
    kk[i] = ld_ring<DT, STREAM>(kr + ((long)jc * H + h) * RA_HD + dc);
  }
  auto vload = [&](int i) {
    const int jc = min(64 * wave + g + 8 * i, ring - 1);
    vv[i] = ld_ring<DT, STREAM>(vr + ((long)jc * H + h) * RA_HD + dc);
  };
  // every load at once, one round trip; float32 streaming: a row's values take the registers of its consumed keys,
  // so that three workgroups a CU fit instead of two
  constexpr bool LATE = STREAM && DT == M3X_F32;
  if constexpr (!LATE) {
#pragma unroll
    for (int i = 0; i < 8; ++i) vload(i);
  }
  const int lo = (int)(p0 % ring);  // ring entry of token 0; token t sits at (lo + t) % ring
  if (wave < T) {  // RoPE of token `wave`
    const float f = inv_freq[l < half ? l : l - half];
    const float sgn = l < half ? -1.f : 1.f;
    const float ang = (float)(p0 + wave) * f;
    const float cs = cosf(ang) * rope_scale, sn = sinf(ang) * rope_scale;
    qs[wave][l] = q_l * cs + sgn * q_p * sn;
    knew[wave][l] = E<DT>::from_f(k_l * cs + sgn * k_p * sn);
    vnew[wave][l] = v_l;
  }
  {
    int dd = tid - lo;  // entries this call writes hold p0 + dd, dd < T
    if (dd < 0) dd += ring;
    // an older entry outside (p0 - window, p0) is never visible; window <= ring, so an age fits an int
    age[tid] = tid >= ring ? RA_RING : dd < T ? -dd : kj > p0 - window && kj < p0 ? (int)(p0 - kj) : RA_RING;
  }
  __syncthreads();  // queries, this call's rows and the ages are in LDS
  float q[TM][8];
#pragma unroll
  for (int t = 0; t < TM; ++t) {
    const float4 qa = *reinterpret_cast<const float4*>(&qs[t][dc]);
    const float4 qb = *reinterpret_cast<const float4*>(&qs[t][dc + 4]);
    q[t][0] = qa.x, q[t][1] = qa.y, q[t][2] = qa.z, q[t][3] = qa.w;
    q[t][4] = qb.x, q[t][5] = qb.y, q[t][6] = qb.z, q[t][7] = qb.w;
  }
  float s[TM][8], m[TM];
#pragma unroll
  for (int t = 0; t < TM; ++t) m[t] = -INFINITY;
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const int jj = 64 * wave + g + 8 * i;
    int dd = jj - lo;  // entries this call writes hold p0 + dd, dd < T
    if (dd < 0) dd += ring;
    const bool own = jj < ring && dd < T;
    const bool any_own = __ballot(own) != 0;  // at most T rows of the workgroup
    if (any_own) {
      const V8<DT> kn = *reinterpret_cast<const V8<DT>*>(&knew[own ? dd : 0][dc]);
#pragma unroll
      for (int e = 0; e < 8; ++e) kk[i].v[e] = own ? kn.v[e] : kk[i].v[e];
    }
    const int aj = age[jj];
#pragma unroll
    for (int t = 0; t < TM; ++t) {
      float acc = 0.f;
#pragma unroll
      for (int e = 0; e < 8; ++e) acc = fmaf(q[t][e], E<DT>::to_f(kk[i].v[e]), acc);
      acc = group_sum<8>(acc) * 0.125f;
      s[t][i] = aj + t >= 0 && aj + t < window ? acc : -INFINITY;  // token t: p0 + t - window < position <= p0 + t
      m[t] = fmaxf(m[t], s[t][i]);
    }
    if constexpr (LATE) vload(i);
    if (any_own) {
      const V8<DT> vn = *reinterpret_cast<const V8<DT>*>(&vnew[own ? dd : 0][dc]);
#pragma unroll
      for (int e = 0; e < 8; ++e) vv[i].v[e] = own ? vn.v[e] : vv[i].v[e];
    }
  }
#pragma unroll
  for (int t = 0; t < TM; ++t) {
    if (t >= T) break;
    m[t] = across_max<8>(m[t]);
    float sum = 0.f, o[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) o[e] = 0.f;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const float p = s[t][i] == -INFINITY ? 0.f : expf(s[t][i] - m[t]);
      sum += p;
#pragma unroll
      for (int e = 0; e < 8; ++e) o[e] = fmaf(p, E<DT>::to_f(vv[i].v[e]), o[e]);
    }
    // A row out of the token's sight takes no part, but weight 0 lets an infinity or NaN of an earlier stream on the slot, or
    // of the call's other token, through: where one shows, the sums are taken again without such rows (dropping them in the
    // loop above costs 2 to 4 % of the launch).
    float bad = 0.f;
#pragma unroll
    for (int e = 0; e < 8; ++e) bad = fmaf(0.f, o[e], bad);
    if (__ballot(bad != 0.f)) {
#pragma unroll
      for (int e = 0; e < 8; ++e) o[e] = 0.f;
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const bool seen = s[t][i] != -INFINITY;
        const float p = seen ? expf(s[t][i] - m[t]) : 0.f;
#pragma unroll
        for (int e = 0; e < 8; ++e) o[e] = fmaf(p, seen ? E<DT>::to_f(vv[i].v[e]) : 0.f, o[e]);
      }
    }
    sum = across_sum<8>(sum);
#pragma unroll
    for (int e = 0; e < 8; ++e) o[e] = across_sum<8>(o[e]);
    if (g == 0) {
      float* pt = &part[wave][t][dc];
#pragma unroll
      for (int e = 0; e < 8; ++e) pt[e] = o[e];
    }
    if (l == 0) {
      wm[t][wave] = m[t];
      wl[t][wave] = sum;
    }
  }
  __syncthreads();
  for (int i = tid; i < T * RA_HD; i += 256) {
    const int t = i / RA_HD, d = i % RA_HD;
    const float mx = fmaxf(fmaxf(wm[t][0], wm[t][1]), fmaxf(wm[t][2], wm[t][3]));  // finite: own key
    float sum = 0.f, v = 0.f;
#pragma unroll
    for (int w = 0; w < 4; ++w) {
      const float f = wm[t][w] == -INFINITY ? 0.f : expf(wm[t][w] - mx);
      sum = fmaf(f, wl[t][w], sum);
      v = fmaf(f, part[w][t][d], v);
    }
    out[((long)b * T + t) * ld_out + h * RA_HD + d] = E<DT>::from_f(v / sum);
    // this call's rows into the ring (every wave has read its rows of it)
    const long e = (lo + t) % ring;
    kr[(e * H + h) * RA_HD + d] = knew[t][d];
    vr[(e * H + h) * RA_HD + d] = vnew[t][d];
    if (h == 0 && d == 0) kp[e] = p0 + t;
  }
}

// Seats' token counters advance by T after the transformer (:183-184); the dummy slot's counter returns to 0. One
// thread per seat (the seats' slots other than the dummy are distinct, so no two threads touch one counter).
__global__ void advance_tokens_kernel(int64_t* tokens, const int64_t* __restrict__ slots, int B, int T, int dummy) {
  const int b = blockIdx.x * blockDim.x + threadIdx.x;
  if (b < B) {
    const int64_t s = slots[b];
    if (s != dummy) tokens[s] += T;
  }
  if (b == 0) tokens[dummy] = 0;
}

// ---------------------------------------------------------------------------------------------------------
// Last conv to PCM (decoder.layers[-1], C -> 1 channel, kernel k, causal) in fp32 with fp32 weights:
// pcm[b, t] = bias + sum_j sum_c w[j * C + c] joined[t + j][c], joined = the slot's k - 1 stored frames then x
// (ELU already applied by the producing row op); the state becomes joined's last k - 1 frames.
// Grid (B, ceil(T / chunk)), chunk >= k - 1; one thread per output sample (rows read as 16-byte vectors,
// weights from LDS); k * C <= 4096.
constexpr int FC_W = 4096;
template <int DT>
__global__ __launch_bounds__(CODEC_THREADS) void final_conv_kernel(const Elt<DT>* __restrict__ x, long ld_x,
                                                                   Elt<DT>* state, long ld_state,
                                                                   const int64_t* __restrict__ slots,
                                                                   const float* __restrict__ w, float bias,
                                                                   float* __restrict__ pcm, long ld_pcm, int T, int C,
                                                                   int k, int chunk) {
  __shared__ float ws[FC_W];
  const int b = blockIdx.x;
  const int t0 = blockIdx.y * chunk, t1 = min(T, t0 + chunk);
  const int pad = k - 1;
  const long row0 = (long)b * T;
  Elt<DT>* st = pad ? state + slots[b] * ld_state : nullptr;
  for (int i = threadIdx.x; i < k * C; i += CODEC_THREADS) ws[i] = w[i];
  __syncthreads();
  const int cv = C / 8;
  for (int t = t0 + threadIdx.x; t < t1; t += CODEC_THREADS) {
    float acc = 0.f;
    for (int j = 0; j < k; ++j) {
      const int i = t + j;
      const Elt<DT>* row = i < pad ? st + (long)i * C : x + (row0 + i - pad) * ld_x;
      const float* wj = ws + j * C;
      for (int c8 = 0; c8 < cv; ++c8) {
        const V8<DT> v = ldv<DT>(row + 8 * c8);
#pragma unroll
        for (int e = 0; e < 8; ++e) acc += wj[8 * c8 + e] * E<DT>::to_f(v.v[e]);
      }
    }
    pcm[(long)b * ld_pcm + t] = acc + bias;
  }
  if (!pad || blockIdx.y) return;
  V8<DT> keep[CODEC_KEEP / 8];  // constant indices: registers, not a private or LDS array
#pragma unroll
  for (int p = 0; p < CODEC_KEEP / 8; ++p) {
    const int e = threadIdx.x + CODEC_THREADS * p;
    if (e < pad * cv) keep[p] = joined8<DT>(st, x, ld_x, row0, pad, T + e / cv, 8 * (e % cv), C, 0);
  }
  __syncthreads();
#pragma unroll
  for (int p = 0; p < CODEC_KEEP / 8; ++p) {
    const int e = threadIdx.x + CODEC_THREADS * p;
    if (e < pad * cv) stv<DT>(st + 8 * e, keep[p]);
  }
}

// final_conv_kernel for the codec's shape (C <= 64 channels, k <= 9 taps), FCS_CHUNK samples per workgroup: the
// chunk's input rows and the k - 1 before it (the slot's stored frames for the first chunk) are staged in LDS as
// fp32 with every 16-byte load issued before the first store (clamped indices, no branch around the loads); then
// one thread per sample sums taps j and channels c in the same order as final_conv_kernel, so the two give the same
// bits. One thread per sample reading its rows from memory made every load touch 64 cache lines (180 us for 224
// seats of one frame).
constexpr int FCS_CHUNK = 128, FCS_C = 64, FCS_K = 9, FCS_LD = FCS_C + 4;
template <int DT>
__global__ __launch_bounds__(CODEC_THREADS) void final_conv_staged_kernel(const Elt<DT>* __restrict__ x, long ld_x,
                                                                          Elt<DT>* state, long ld_state,
                                                                          const int64_t* __restrict__ slots,
                                                                          const float* __restrict__ w, float bias,
                                                                          float* __restrict__ pcm, long ld_pcm, int T,
                                                                          int C, int k) {
  __shared__ __align__(16) float ws[FCS_K * FCS_C];
  __shared__ __align__(16) float xs[(FCS_CHUNK + FCS_K - 1) * FCS_LD];
  const int b = blockIdx.x;
  const int t0 = blockIdx.y * FCS_CHUNK, t1 = min(T, t0 + FCS_CHUNK);
  const int pad = k - 1;
  const long row0 = (long)b * T;
  Elt<DT>* st = pad ? state + slots[b] * ld_state : nullptr;
  for (int i = threadIdx.x; i < k * C; i += CODEC_THREADS) ws[i] = w[i];
  const int cv = C / 8;
  const int nvec = (t1 - t0 + pad) * cv;  // staged row r is the joined row t0 + r
  constexpr int VPT = ((FCS_CHUNK + FCS_K - 1) * (FCS_C / 8) + CODEC_THREADS - 1) / CODEC_THREADS;
  V8<DT> v[VPT];
#pragma unroll
  for (int p = 0; p < VPT; ++p) {
    const int e = min((int)threadIdx.x + CODEC_THREADS * p, nvec - 1);
    const int r = e / cv, q = e - (e / cv) * cv;
    const int i = t0 + r;
    v[p] = ldv<DT>(i < pad ? st + (long)i * C + 8 * q : x + (row0 + i - pad) * ld_x + 8 * q);
  }
#pragma unroll
  for (int p = 0; p < VPT; ++p) {
    const int e = min((int)threadIdx.x + CODEC_THREADS * p, nvec - 1);  // repeats store the same values
    const int r = e / cv, q = e - (e / cv) * cv;
    float* d = xs + r * FCS_LD + 8 * q;
    *reinterpret_cast<float4*>(d) =
        make_float4(E<DT>::to_f(v[p].v[0]), E<DT>::to_f(v[p].v[1]), E<DT>::to_f(v[p].v[2]), E<DT>::to_f(v[p].v[3]));
    *reinterpret_cast<float4*>(d + 4) =
        make_float4(E<DT>::to_f(v[p].v[4]), E<DT>::to_f(v[p].v[5]), E<DT>::to_f(v[p].v[6]), E<DT>::to_f(v[p].v[7]));
  }
  __syncthreads();
  for (int t = t0 + threadIdx.x; t < t1; t += CODEC_THREADS) {
    float acc = 0.f;
    for (int j = 0; j < k; ++j) {
      const float* row = xs + (t - t0 + j) * FCS_LD;
      const float* wj = ws + j * C;
      for (int c = 0; c < C; c += 4) {
        const float4 xv = *reinterpret_cast<const float4*>(row + c);
        acc += wj[c] * xv.x;
        acc += wj[c + 1] * xv.y;
        acc += wj[c + 2] * xv.z;
        acc += wj[c + 3] * xv.w;
      }
    }
    pcm[(long)b * ld_pcm + t] = acc + bias;
  }
  if (!pad || blockIdx.y) return;
  // the new history: pad * C / 8 <= 64 vectors, at most one per thread (a register, not a private array)
  const int e = threadIdx.x;
  V8<DT> keep = zero_v8<DT>();
  if (e < pad * cv) keep = joined8<DT>(st, x, ld_x, row0, pad, T + e / cv, 8 * (e % cv), C, 0);
  __syncthreads();
  if (e < pad * cv) stv<DT>(st + 8 * e, keep);
}

// ---------------------------------------------------------------------------------------------------------
// C ABI
// The arguments name the element type ET, which each branch binds to its dtype's storage type.
#define CODEC_LAUNCH(KERNEL, GRID, BLOCK, ...)                                                   \
  do {                                                                                           \
    if (dtype == M3X_BF16) {                                                                     \
      using ET = uint16_t;                                                                        \
      hipLaunchKernelGGL(KERNEL<M3X_BF16>, GRID, BLOCK, 0, (hipStream_t)stream, __VA_ARGS__);    \
    } else if (dtype == M3X_F16) {                                                               \
      using ET = uint16_t;                                                                        \
      hipLaunchKernelGGL(KERNEL<M3X_F16>, GRID, BLOCK, 0, (hipStream_t)stream, __VA_ARGS__);     \
    } else if (dtype == M3X_F32) {                                                               \
      using ET = float;                                                                            \
      hipLaunchKernelGGL(KERNEL<M3X_F32>, GRID, BLOCK, 0, (hipStream_t)stream, __VA_ARGS__);     \
    } else {                                                                                     \
      return M3X_EUNSUPPORTED;                                                                   \
    }                                                                                            \
    M3X_CHECK_LAUNCH();                                                                          \
  } while (0)

M3X_API int m3x_rvq_decode(const int64_t* codes, long ld_codes, const void* tables, void* out, long ld_out, int B,
                           int nq, int n_codes, int dim, int dtype, void* stream) {
  if (B < 0 || nq < 1 || n_codes < 1 || dim < 1 || ld_codes < nq || ld_out < 2L * dim) return M3X_EINVAL;
  if (B == 0) return M3X_OK;
  if (!codes || !tables || !out) return M3X_ENULL;
  CODEC_LAUNCH(rvq_decode_kernel, dim3(B), dim3(256), codes, ld_codes, (const ET*)tables, (ET*)out,
               ld_out, nq, n_codes, dim);
  return M3X_OK;
}

M3X_API int m3x_dwconvt(const void* x, long ld_x, const void* w, void* tail, long ld_tail, const int64_t* slots,
                        void* out, int B, int C, int k, int s, int dtype, void* stream) {
  if (B < 0 || C < 1 || s < 1 || k < s || k > 2 * s || ld_x < C || ld_tail < (long)(k - s) * C) return M3X_EINVAL;
  if (B == 0) return M3X_OK;
  if (!x || !w || !tail || !slots || !out) return M3X_ENULL;
  CODEC_LAUNCH(dwconvt_kernel, dim3(B), dim3(256), (const ET*)x, ld_x, (const ET*)w, (ET*)tail,
               ld_tail, slots, (ET*)out, C, k, s);
  return M3X_OK;
}

M3X_API int m3x_conv_gather(const void* x, long ld_x, void* state, long ld_state, const int64_t* slots, void* cols,
                            long ld_cols, int B, int T, int C, int k, int dil, int use_elu, int chunk, int dtype,
                            void* stream) {
  const int pad = (k - 1) * dil;
  if (B < 0 || T < 1 || C < 8 || C % 8 || k < 1 || dil < 1 || ld_x < C || (cols && ld_cols < (long)k * C) ||
      chunk < max(pad, 1) || ((ld_x | (cols ? ld_cols : 0) | (pad ? ld_state : 0)) & 7))
    return M3X_EINVAL;
  if (!m3x_aligned16(x) || (cols && !m3x_aligned16(cols)) || (pad && !m3x_aligned16(state))) return M3X_EINVAL;
  if (pad && (ld_state < (long)pad * C || pad * C > CODEC_KEEP * CODEC_THREADS)) return M3X_EINVAL;
  if (B == 0) return M3X_OK;
  if (!x || !slots || (pad && !state)) return M3X_ENULL;
  if (!cols && !pad) return M3X_OK;
  CODEC_LAUNCH(conv_gather_kernel, dim3(B, m3x_ceil_div(T, chunk)), dim3(CODEC_THREADS), (const ET*)x, ld_x,
               (ET*)state, ld_state, slots, (ET*)cols, ld_cols, T, C, k, dil, use_elu, chunk);
  return M3X_OK;
}

M3X_API int m3x_rows_op(const void* g, long ld_g, const void* bias, const void* scale, const void* res, long ld_res,
                        void* out, long ld_out, int rows, int C, int use_elu, int dtype, void* stream) {
  if (rows < 0 || C < 8 || C % 8 || ld_g < C || ld_out < C || (res && ld_res < C)) return M3X_EINVAL;
  if ((ld_g | ld_out | (res ? ld_res : 0)) & 7) return M3X_EINVAL;
  if (rows == 0) return M3X_OK;
  if (!g || !out) return M3X_ENULL;
  if (!m3x_aligned16(g) || !m3x_aligned16(out) || (bias && !m3x_aligned16(bias)) ||
      (scale && !m3x_aligned16(scale)) || (res && !m3x_aligned16(res)))
    return M3X_EINVAL;
  CODEC_LAUNCH(rows_op_kernel, dim3(m3x_ceil_div((long)rows * (C / 8), 256)), dim3(256), (const ET*)g, ld_g,
               (const ET*)bias, (const ET*)scale, (const ET*)res, ld_res, (ET*)out, ld_out,
               rows, C, use_elu);
  return M3X_OK;
}

M3X_API int m3x_convt_overlap(const void* cols, long ld_cols, void* tail, long ld_tail, const int64_t* slots,
                              const void* bias, void* out, long ld_out, int B, int Tin, int C, int k, int s, int chunk,
                              int dtype, void* stream) {
  if (B < 0 || Tin < 1 || C < 8 || C % 8 || s < 1 || k <= s || k > 2 * s || ld_cols < (long)k * C || ld_out < C ||
      chunk < k - s || ((ld_cols | ld_tail | ld_out) & 7))
    return M3X_EINVAL;
  if (!m3x_aligned16(cols) || !m3x_aligned16(tail) || !m3x_aligned16(out) || (bias && !m3x_aligned16(bias)))
    return M3X_EINVAL;
  if (ld_tail < (long)(k - s) * C || (k - s) * C > CODEC_KEEP * CODEC_THREADS) return M3X_EINVAL;
  if (B == 0) return M3X_OK;
  if (!cols || !tail || !slots || !out) return M3X_ENULL;
  CODEC_LAUNCH(convt_overlap_kernel, dim3(B, m3x_ceil_div((long)Tin * s, chunk)), dim3(CODEC_THREADS),
               (const ET*)cols, ld_cols, (ET*)tail, ld_tail, slots, (const ET*)bias, (ET*)out,
               ld_out, Tin, C, k, s, chunk);
  return M3X_OK;
}

M3X_API int m3x_ring_attn(const void* qkv, long ld_qkv, void* kring, void* vring, int64_t* key_pos,
                          const int64_t* tokens, const int64_t* slots, const float* inv_freq, float rope_scale,
                          void* out, long ld_out, int B, int T, int H, int head_dim, int ring, int window, int dtype,
                          void* stream) {
  if (B < 0 || T < 1 || T > RA_T || H < 1 || H > 8 || head_dim != RA_HD || ring < 1 || ring > RA_RING ||
      window < 1 || ring < window + T - 1 || ring < T || ld_qkv < 3L * H * RA_HD || ld_out < (long)H * RA_HD || (ld_qkv & 7))
    return M3X_EINVAL;
  if (B == 0) return M3X_OK;
  if (!qkv || !kring || !vring || !key_pos || !tokens || !slots || !inv_freq || !out) return M3X_ENULL;
  if (!m3x_aligned16(qkv) || !m3x_aligned16(kring)) return M3X_EINVAL;
  if (!m3x_aligned16(out) || (ld_out & 7)) return M3X_EINVAL;
  if ((long)B * H > 0x7fffffffL) return M3X_EINVAL;
  const bool stream_rows = (long)B * ring * H * RA_HD * 2 * (dtype == M3X_F32 ? 4 : 2) >= RA_STREAM_BYTES;
#define RA_LAUNCH(DTT, STR)                                                                                       \
  hipLaunchKernelGGL((ring_attn_kernel<DTT, RA_T, STR>), dim3((unsigned)(B * H)), dim3(256), 0, (hipStream_t)stream, \
                     (const Elt<DTT>*)qkv, ld_qkv, (Elt<DTT>*)kring, (Elt<DTT>*)vring, key_pos, tokens, slots,        \
                     inv_freq, rope_scale, (Elt<DTT>*)out, ld_out, T, H, ring, window)
#define RA_DT(DTT)                      \
  do {                                  \
    if (stream_rows) RA_LAUNCH(DTT, true); \
    else RA_LAUNCH(DTT, false);         \
  } while (0)
  if (dtype == M3X_F16) RA_DT(M3X_F16);
  else if (dtype == M3X_BF16) RA_DT(M3X_BF16);
  else if (dtype == M3X_F32) RA_DT(M3X_F32);
  else return M3X_EUNSUPPORTED;
#undef RA_DT
#undef RA_LAUNCH
  M3X_CHECK_LAUNCH();
  return M3X_OK;
}

M3X_API int m3x_advance_tokens(int64_t* tokens, const int64_t* slots, int B, int T, int dummy, void* stream) {
  if (B < 0 || T < 0 || dummy < 0) return M3X_EINVAL;
  if (!tokens || (B && !slots)) return M3X_ENULL;
  hipLaunchKernelGGL(advance_tokens_kernel, dim3(m3x_ceil_div(std::max(B, 1), 256)), dim3(256), 0, (hipStream_t)stream,
                     tokens, slots, B, T, dummy);
  M3X_CHECK_LAUNCH();
  return M3X_OK;
}

M3X_API int m3x_final_conv(const void* x, long ld_x, void* state, long ld_state, const int64_t* slots, const float* w,
                           float bias, float* pcm, long ld_pcm, int B, int T, int C, int k, int chunk, int dtype,
                           void* stream) {
  if (B < 0 || T < 1 || C < 8 || C % 8 || k < 1 || ld_x < C || ld_pcm < T || chunk < max(k - 1, 1) ||
      ((ld_x | (k > 1 ? ld_state : 0)) & 7))
    return M3X_EINVAL;
  if (!m3x_aligned16(x) || (k > 1 && !m3x_aligned16(state))) return M3X_EINVAL;
  if (k > 1 && (ld_state < (long)(k - 1) * C || (k - 1) * C > CODEC_KEEP * CODEC_THREADS)) return M3X_EINVAL;
  if ((long)k * C > FC_W) return M3X_EINVAL;
  if (B == 0) return M3X_OK;
  if (!x || !slots || !w || !pcm || (k > 1 && !state)) return M3X_ENULL;
  if (C <= FCS_C && k <= FCS_K) {  // the codec's shape: rows staged in LDS (chunk is the general path's)
    CODEC_LAUNCH(final_conv_staged_kernel, dim3(B, m3x_ceil_div(T, FCS_CHUNK)), dim3(CODEC_THREADS), (const ET*)x,
                 ld_x, (ET*)state, ld_state, slots, w, bias, pcm, ld_pcm, T, C, k);
    return M3X_OK;
  }
  CODEC_LAUNCH(final_conv_kernel, dim3(B, m3x_ceil_div(T, chunk)), dim3(CODEC_THREADS), (const ET*)x, ld_x,
               (ET*)state, ld_state, slots, w, bias, pcm, ld_pcm, T, C, k, chunk);
  return M3X_OK;
}

M3X_API int m3x_resid_ln(void* h, long ld_h, const void* a, long ld_a, const void* scale, const void* w,
                         const void* b, void* y, long ld_y, float eps, int rows, int n, int dtype, void* stream) {
  if (rows < 0 || n != RLN_N || ld_h < n || ld_a < n || ld_y < n || ((ld_h | ld_a | ld_y) & 7)) return M3X_EINVAL;
  if (rows == 0) return M3X_OK;
  if (!h || !a || !scale || !w || !b || !y) return M3X_ENULL;
  if (!m3x_aligned16(h) || !m3x_aligned16(a) || !m3x_aligned16(scale) || !m3x_aligned16(w) || !m3x_aligned16(b) ||
      !m3x_aligned16(y))
    return M3X_EINVAL;
  CODEC_LAUNCH(resid_ln_kernel, dim3(m3x_ceil_div(rows, 4)), dim3(256), (ET*)h, ld_h, (const ET*)a, ld_a,
               (const ET*)scale, (const ET*)w, (const ET*)b, (ET*)y, ld_y, eps, rows);
  return M3X_OK;
}

M3X_API int m3x_conv_gemm(const void* x, long ldx, const void* w_packed, const void* bias, const void* res,
                          long ld_res, void* y, long ldy, int M, int N, int K, int use_elu, const void* state,
                          long ld_state, const int64_t* slots, int T, int C, int dil, int pre_elu, int dtype,
                          void* stream) {
  // gathered form when C > 0: K = k * C, x rows [M, C], the slot's history of pad = (k - 1) * dil frames
  ConvSrc cs{state, ld_state, slots, T, C, dil, 0, pre_elu};
  const int G = C > 0;
  if (G) {
    if (T < 1 || C % 8 || K % C || M % T || dil < 1 || ldx < C || (ldx & 7)) return M3X_EINVAL;
    cs.pad = (K / C - 1) * dil;
    if (cs.pad && (!state || !slots)) return M3X_ENULL;
    if (cs.pad && (ld_state < (long)cs.pad * C || (ld_state & 7) || !m3x_aligned16(state))) return M3X_EINVAL;
  }
  if (M < 0 || K < 32 || K % 32 || (N != 16 && N != 32 && N != 64 && N != 128) || (!G && ldx < K) || ldy < N || (res && ld_res < N) || ((ldx | ldy | (res ? ld_res : 0)) & 7))
    return M3X_EINVAL;
  if (M == 0) return M3X_OK;
  if (!x || !w_packed || !y) return M3X_ENULL;
  if (!m3x_aligned16(x) || !m3x_aligned16(w_packed) || !m3x_aligned16(y) || (res && !m3x_aligned16(res)) ||
      (bias && (((uintptr_t)bias) & 7)))
    return M3X_EINVAL;
  const int mt = M >= 64 * 1024 ? 2 : 1;  // two row tiles per wave once the grid fills the chip anyway
  // few rows (one seat): the columns split into up to N / 16 groups until 128 workgroups run
  const int gx = m3x_ceil_div(M, 4 * 16 * mt);
  int ny = 1;
  while (ny < N / 16 && (long)gx * ny < 128) ny *= 2;
  const int nt = N / 16 / ny;
  const dim3 grid(gx, ny);
  if (dtype == M3X_F32 && bias && !m3x_aligned16(bias)) return M3X_EINVAL;
  hipStream_t st = (hipStream_t)stream;
  if (dtype == M3X_F32) {
    const F32Epi ep{(const float*)bias, (const float*)res, ld_res, use_elu};
    const float *X = (const float*)x, *W = (const float*)w_packed;
    // conv_x3_kernel: whole channel blocks, 3 taps, 32 or 64 columns a workgroup, at least 70 % of its 128-row blocks'
    // rows live, enough workgroups; reads of x overlapping its own output (y = x in place) are out
    const int rblk = G ? m3x_ceil_div(T, CX_ROWS) : 0, ncol = N == 32 ? 32 : 64;
    if (G && C % 32 == 0 && K == 3 * C && cs.pad <= CX_PAD && N >= 32 && 10L * T >= 7L * rblk * CX_ROWS && y != x &&
        (long)(M / T) * rblk * (N / ncol) >= CX_MIN_BLOCKS && (long)(M / T) * rblk <= 0x7fffffffL) {
      const dim3 gx3((unsigned)((long)(M / T) * rblk), N / ncol);
      if (ncol == 32)
        hipLaunchKernelGGL((conv_x3_kernel<2, 3>), gx3, dim3(256), 0, st, X, ldx, W, (float*)y, ldy, rblk, ep, cs);
      else
        hipLaunchKernelGGL((conv_x3_kernel<4, 3>), gx3, dim3(256), 0, st, X, ldx, W, (float*)y, ldy, rblk, ep, cs);
      M3X_CHECK_LAUNCH();
      return M3X_OK;
    }
    // plain rows (a 1x1 conv, or gathered columns): the projection's kernel with the conv epilogue, from a workgroup a CU:
    // 15360 x 128 x 64 (240) 12.0 against 10.8 us, 19200 (300) 13.4 against 15.0 (in place)
    const int mblk = m3x_ceil_div(M, 64), nblk = N / 64;
    if (!G && N >= 64 && y != x && mblk >= F32X3_MIN_BLOCKS) {
      if (N == 128)
        hipLaunchKernelGGL((linear_f32x3_kernel<2, 2, 4, 2>), dim3((unsigned)xcd_grid(mblk, 1)), dim3(256), 0, st, X, ldx,
                           W, (float*)y, ldy, M, N, K, mblk, 1, ep);
      else
        hipLaunchKernelGGL((linear_f32x3_kernel<2, 2, 2, 2>), dim3((unsigned)xcd_grid(mblk, nblk)), dim3(256), 0, st, X,
                           ldx, W, (float*)y, ldy, M, N, K, mblk, nblk, ep);
      M3X_CHECK_LAUNCH();
      return M3X_OK;
    }
  }
#define CG_CASE(DTT, NTT, MTT)                                                                                   \
  if (dtype == DTT && nt == NTT && mt == MTT) {                                                              \
    using ET = Elt<DTT>;                                                                                         \
    const ET *X = (const ET*)x, *W = (const ET*)w_packed, *Bi = (const ET*)bias, *R = (const ET*)res;                 \
    if (G)                                                                                                       \
      hipLaunchKernelGGL((conv_gemm_kernel<DTT, NTT, MTT, 1>), grid, dim3(256), 0, st, X, ldx, W, Bi, R, ld_res, \
                         (ET*)y, ldy, M, K, use_elu, cs);                                                         \
    else                                                                                                         \
      hipLaunchKernelGGL((conv_gemm_kernel<DTT, NTT, MTT, 0>), grid, dim3(256), 0, st, X, ldx, W, Bi, R, ld_res, \
                         (ET*)y, ldy, M, K, use_elu, cs);                                                         \
    M3X_CHECK_LAUNCH();                                                                                          \
    return M3X_OK;                                                                                               \
  }
  CG_CASE(M3X_F16, 1, 1) CG_CASE(M3X_F16, 2, 1) CG_CASE(M3X_F16, 4, 1) CG_CASE(M3X_F16, 8, 1)
  CG_CASE(M3X_F16, 1, 2) CG_CASE(M3X_F16, 2, 2) CG_CASE(M3X_F16, 4, 2) CG_CASE(M3X_F16, 8, 2)
  CG_CASE(M3X_BF16, 1, 1) CG_CASE(M3X_BF16, 2, 1) CG_CASE(M3X_BF16, 4, 1) CG_CASE(M3X_BF16, 8, 1)
  CG_CASE(M3X_BF16, 1, 2) CG_CASE(M3X_BF16, 2, 2) CG_CASE(M3X_BF16, 4, 2) CG_CASE(M3X_BF16, 8, 2)
  CG_CASE(M3X_F32, 1, 1) CG_CASE(M3X_F32, 2, 1) CG_CASE(M3X_F32, 4, 1) CG_CASE(M3X_F32, 8, 1)
  CG_CASE(M3X_F32, 1, 2) CG_CASE(M3X_F32, 2, 2) CG_CASE(M3X_F32, 4, 2) CG_CASE(M3X_F32, 8, 2)
#undef CG_CASE
  return M3X_EUNSUPPORTED;
}
