// Top-k selection and inverse-CDF draw inside one 256-thread workgroup per row, shared by the samplers of
// sample.hip and the depth frame kernel (depth.hip). The sampling contract is stated at the top of sample.hip.
#pragma once
#include "m3x_norm.h"

namespace {
constexpr int ST = 256;      // threads per row
constexpr int SMAXV = 4096;  // largest vocabulary

__device__ __forceinline__ uint32_t ordkey(float f) {
  uint32_t u = __float_as_uint(f);
  return (u & 0x80000000u) ? ~u : (u | 0x80000000u);
}
__device__ __forceinline__ float ordkey_inv(uint32_t k) {
  return __uint_as_float((k & 0x80000000u) ? (k & 0x7fffffffu) : ~k);
}

// CAP: the most candidates a row can have (its vocabulary size)
template <int CAP>
struct SampleSmemT {
  __align__(16) unsigned long long cand[CAP];
  float w[CAP];
  unsigned int hist[256];
  int nkeep;
  int ncand;  // candidates placed so far
  int code;  // the drawn code, for the waves that build the next level's input
};
using SampleSmem = SampleSmemT<SMAXV>;

// every lane gets the wave's maximum (DPP within rows, permlane swaps across them; max is exact in any order)
__device__ __forceinline__ float wave_max_dpp(float v) {
  v = fmaxf(v, dppf<0xB1>(v));   // quad_perm [1,0,3,2]
  v = fmaxf(v, dppf<0x4E>(v));   // quad_perm [2,3,0,1]
  v = fmaxf(v, dppf<0x141>(v));  // row_half_mirror: the partner quad's maximum
  v = fmaxf(v, dppf<0x140>(v));  // row_mirror: the partner half-row's maximum
  return xor32_max(xor16_max(v));
}

// inclusive prefix sum of an integer over the 64 lanes (integer adds: any order gives the same sums). DPP row
// shifts build the sums within each row of 16, then row broadcasts carry the row totals forward.
__device__ __forceinline__ unsigned int wave_incl_scan(unsigned int x) {
  unsigned int v = x;
  v = v + (unsigned int)__builtin_amdgcn_update_dpp(0, (int)x, 0x111, 0xf, 0xf, true);  // row_shr:1
  v = v + (unsigned int)__builtin_amdgcn_update_dpp(0, (int)x, 0x112, 0xf, 0xf, true);  // row_shr:2
  v = v + (unsigned int)__builtin_amdgcn_update_dpp(0, (int)x, 0x113, 0xf, 0xf, true);  // row_shr:3
  v = v + (unsigned int)__builtin_amdgcn_update_dpp(0, (int)v, 0x114, 0xf, 0xe, false);  // row_shr:4, lanes 4..15
  v = v + (unsigned int)__builtin_amdgcn_update_dpp(0, (int)v, 0x118, 0xf, 0xc, false);  // row_shr:8, lanes 8..15
  v = v + (unsigned int)__builtin_amdgcn_update_dpp(0, (int)v, 0x142, 0xa, 0xf, false);  // row_bcast:15, rows 1, 3
  v = v + (unsigned int)__builtin_amdgcn_update_dpp(0, (int)v, 0x143, 0xc, 0xf, false);  // row_bcast:31, rows 2, 3
  return v;
}

// The first of 256 bins (lane l holds the counts c[0..3] of its 4 bins, in the order they are scanned) at which the
// running count reaches kk, with the count before that bin; every lane of the wave gets the result. (-1, 0) when
// the total stays below kk (or kk is 0).
__device__ __forceinline__ void wave_find_bin(const unsigned int (&c)[4], unsigned int kk, int& idx, unsigned int& before) {
  const int lane = threadIdx.x & 63;
  const unsigned int s = c[0] + c[1] + c[2] + c[3];
  const unsigned int incl = wave_incl_scan(s);
  unsigned int run = incl - s;
  int found = -1;
  unsigned int bef = 0;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    if (found < 0 && kk > 0 && run + c[i] >= kk) {
      found = 4 * lane + i;
      bef = run;
    }
    run += c[i];
  }
  const unsigned long long mk = __ballot(found >= 0);
  const int fl = mk ? __ffsll((long long)mk) - 1 : 0;
  idx = mk ? __builtin_amdgcn_readlane(found, fl) : -1;
  before = mk ? (unsigned int)__builtin_amdgcn_readlane((int)bef, fl) : 0u;
}

// The k-th largest of the valid elements (i < V, not NaN) of a row, counting repeats, by an MSB-first radix select
// over their ordered keys, 8 bits a pass: each pass histograms the next byte of the keys that share the bytes fixed
// so far, and every wave finds the bin where the count from the top reaches the remaining rank. With fewer than k
// valid elements it returns the smallest; with none, NaN. Called by every thread with a block-uniform k, before
// the candidates are placed: the three histograms (used in turn, each cleared two passes ahead, so one barrier a
// pass) live in sm.cand after the coarse histogram of topk_select.
template <int NE, class SM>
__device__ float radix_kth(const float (&x)[NE], int V, int k, SM& sm) {
  static_assert(sizeof(sm.cand) >= 4 * 256 * sizeof(unsigned int), "histograms in sm.cand");
  unsigned int* hb = reinterpret_cast<unsigned int*>(sm.cand) + 256;
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  uint32_t key[NE];
  bool ok[NE];
#pragma unroll
  for (int e = 0; e < NE; ++e) {
    ok[e] = tid + ST * e < V && x[e] == x[e];
    key[e] = ordkey(x[e]);
  }
  hb[tid] = 0;
  hb[256 + tid] = 0;
  __syncthreads();
  uint32_t pre = 0;
  unsigned int kr = (unsigned int)k;
#pragma unroll
  for (int pass = 0; pass < 4; ++pass) {
    const int sh = 24 - 8 * pass;
    const uint32_t hm = pass == 0 ? 0u : ~0u << (sh + 8);
    unsigned int* h = hb + 256 * (pass % 3);
#pragma unroll
    for (int e = 0; e < NE; ++e) {
      const bool in = ok[e] && (key[e] & hm) == pre;
      const uint32_t d = (key[e] >> sh) & 255u;
      // the keys of a row mostly share their top bytes: the lanes holding the wave's first live digit add their
      // count with one atomic, the others one each
      const unsigned long long live = __ballot(in);
      if (live) {
        const int first = __ffsll((long long)live) - 1;
        const uint32_t d0 = (uint32_t)__builtin_amdgcn_readlane((int)d, first);
        const unsigned long long same = __ballot(in && d == d0);
        if (lane == first) atomicAdd(&h[d0], (unsigned int)__popcll(same));
        if (in && d != d0) atomicAdd(&h[d], 1u);
      }
    }
    __syncthreads();
    if (pass < 2) hb[256 * ((pass + 2) % 3) + tid] = 0;  // last read two passes back, next written after a barrier
    // lane l scans bins 255 - 4 l .. 252 - 4 l: descending key order
    unsigned int c[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) c[i] = h[255 - 4 * lane - i];
    int idx;
    unsigned int before;
    if (pass == 0) {
      const unsigned int total = (unsigned int)__builtin_amdgcn_readlane(
          (int)wave_incl_scan(c[0] + c[1] + c[2] + c[3]), 63);
      if (total < kr) kr = total;  // fewer valid elements than k: the smallest of them
    }
    wave_find_bin(c, kr, idx, before);
    if (idx < 0) {  // no valid element (block-uniform)
      __syncthreads();
      return __uint_as_float(0x7fc00000u);
    }
    pre |= (uint32_t)(255 - idx) << sh;
    kr -= before;
  }
  __syncthreads();  // every wave's last scan precedes the candidate stores into sm.cand
  return ordkey_inv(pre);
}

// The k-th largest of 256 values held 4 a lane by every wave, approximately: a value t with at least k of them >= t,
// at most max(k + k / 16, 40) unless values repeat or crowd within the search's reach. lo: a value with count(>= lo) >= k.
// Three thresholds a round (their counts are independent, a round is bound by the latency of one): up to 4-5 rounds. Six
// narrow a row's range to its 4096th part, a step of a bf16 value or less; with repeats at the k-th place more come to
// nothing (224 flat rows of 2048, k = 10: 6.9 us with twelve rounds, 5.1 so). Unrolled, the one-seat depth frame loses 0.4 %.
__device__ __forceinline__ float wave_kth(const float (&c)[4], float lo, float hi, int k) {
  const int enough = max(k + (k >> 4), 40);
#pragma unroll 1
  for (int it = 0; it < 6; ++it) {
    const float m2 = 0.5f * lo + 0.5f * hi;
    const float m1 = 0.5f * lo + 0.5f * m2, m3 = 0.5f * m2 + 0.5f * hi;
    if (!(m2 > lo && m2 < hi)) break;
    int n1 = 0, n2 = 0, n3 = 0;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      n1 += __popcll(__ballot(c[i] >= m1));
      n2 += __popcll(__ballot(c[i] >= m2));
      n3 += __popcll(__ballot(c[i] >= m3));
    }
    // counts fall from lo to hi: the highest threshold that still has k
    int n = 0;
    if (n3 >= k) lo = m3, n = n3;
    else if (n2 >= k) lo = m2, hi = m3, n = n2;
    else if (n1 >= k) lo = m1, hi = m2, n = n1;
    else hi = m1;
    if (n && n <= enough) break;
  }
  return lo;
}

// The candidate marks (bit e: element e) of a row with a large k (more than KFAST): bucket counts of floor(32 * (m - x)).
template <int NE, class SM>
__device__ bool hist_marks(const float (&x)[NE], int V, int k, float m, SM& sm, unsigned int& mark) {
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  unsigned int* h2 = reinterpret_cast<unsigned int*>(sm.cand);  // the coarse histogram (candidates come later)
  __syncthreads();  // every wave has read the threads' maxima
  sm.hist[tid] = 0;
  h2[tid] = 0;
  __syncthreads();
  int bk[NE];
#pragma unroll
  for (int e = 0; e < NE; ++e) {
    bk[e] = 256;
    if (tid + ST * e < V) {
      const float d = (m - x[e]) * 32.0f;
      bk[e] = (d >= 255.0f || d != d) ? 255 : (int)d;
      if (bk[e] < 255) atomicAdd(&sm.hist[bk[e]], 1u);
    }
  }
  __syncthreads();
  // every wave finds b* itself from the histogram (no barrier): lane l holds bins 4 l .. 4 l + 3; bin 255 (8 or
  // more below the max) is not counted
  unsigned int c[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) c[i] = 4 * lane + i < 255 ? sm.hist[4 * lane + i] : 0u;
  int bstar;
  unsigned int before;
  wave_find_bin(c, (unsigned int)k, bstar, before);
  // Fewer than k elements within 8 of the max: a coarse histogram of the rest, 0.5 wide bins from 255/32 below the
  // max (bin 255: 135 or more below, not counted), finds the bin b2 where the count reaches k; the candidates are
  // then the near elements and those in coarse bins <= b2.
  int b2 = 0;
  int cb[NE];
#pragma unroll
  for (int e = 0; e < NE; ++e) cb[e] = 255;
  if (bstar < 0) {
    const unsigned int near =
        (unsigned int)__builtin_amdgcn_readlane((int)wave_incl_scan(c[0] + c[1] + c[2] + c[3]), 63);
#pragma unroll
    for (int e = 0; e < NE; ++e) {
      if (tid + ST * e < V && bk[e] == 255) {
        const float d2 = ((m - x[e]) * 32.0f - 255.0f) * 0.0625f;
        cb[e] = (d2 >= 255.0f || d2 != d2) ? 255 : (int)d2;
        if (cb[e] < 255) atomicAdd(&h2[cb[e]], 1u);
      }
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < 4; ++i) c[i] = 4 * lane + i < 255 ? h2[4 * lane + i] : 0u;
    wave_find_bin(c, (unsigned int)k - near, b2, before);
    __syncthreads();  // every wave's scan of the coarse histogram precedes the candidate stores over it
    if (b2 < 0) return false;
  }
  mark = 0;
#pragma unroll
  for (int e = 0; e < NE; ++e)
    mark |= (tid + ST * e < V && (bstar >= 0 ? bk[e] <= bstar : (bk[e] < 255 || cb[e] <= b2))) ? 1u << e : 0u;
  return true;
}

// After this returns, sm.cand[0 .. sm.nkeep) holds the kept candidates in sampling order and sm.w their weights.
// x[] holds this thread's elements i = tid + 256*e (e < NE, NE * 256 >= V) of the transformed row.
//
// Candidates (any set {x >= t} with t at or below the k-th largest gives the same kept set): for k <= KFAST, t is
// about the k-th largest of the 256 threads' maxima, found by every wave by bisection over the values. At least k
// elements, the maxima themselves, are then >= t, and a random order of the row leaves few others: 55 candidates for
// k = 50 of 2048. It needs no atomics and one barrier, whatever the shape of the row; a histogram of the distances below
// the maximum serialised its atomics on a peaked row, whose bulk falls into a few bins. Rows of 2048 with one code 16
// above the bulk, MI355X: the 224-seat depth frame (30 such samplers) 5.11 -> 4.94 ms, the one-seat frame 2.35 ->
// 2.21 ms. The sampler alone, us, 224 rows, histogram / maxima: peaked k = 10 6.8 / 5.1, 50 8.9 / 5.7, 100 11.6 / 10.0; flat k = 10
// 5.8 / 5.1, 50 6.0 / 5.6, 80 8.8 / 6.6, 100 9.3 / 10.1, 128 10.8 / 12.1 (more than 128 candidates, ranked one a thread). Larger k
// takes the histogram: the maxima would let through several times k candidates (k = 200 of 2048: about 350). More than 256
// candidates (an order that gathers the leaders in a few threads, many repeats), or fewer than k threads with a maximum
// above -inf, take the exact radix select.
// The kernel runs every line of code once or twice a launch, so it is bound by latencies (dependent operations, barriers,
// instruction fetch) and short loops beat unrolled code.
constexpr int KFAST = 128;

template <int NE, class SM>
__device__ void topk_select(const float (&x)[NE], int V, int k, SM& sm) {
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const float NEG = -INFINITY;
  if (tid == 0) {
    sm.nkeep = 0;
    sm.ncand = 0;
  }
  if (tid < 128) sm.cand[tid] = 0ull;  // below every candidate's key
  float lm = NEG;
#pragma unroll
  for (int e = 0; e < NE; ++e)
    if (tid + ST * e < V) lm = fmaxf(lm, x[e]);
  sm.hist[tid] = __float_as_uint(lm);
  __syncthreads();
  float c[4];
  int valid = 0;
  float hi = NEG, lo = INFINITY;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    c[i] = __uint_as_float(sm.hist[4 * lane + i]);
    valid += __popcll(__ballot(c[i] > NEG));
    hi = fmaxf(hi, c[i]);
    lo = fminf(lo, c[i] > NEG ? c[i] : INFINITY);
  }
  hi = wave_max_dpp(hi);
  bool exact = false, all = false;  // exact: t is the k-th largest itself
  float t = NEG;
  unsigned int hmark = 0;
  bool have = false;  // the histogram's marks
  if (k > KFAST) {
    have = hist_marks<NE>(x, V, k, hi, sm, hmark);
    exact = !have;
  } else if (valid >= k) {
    t = wave_kth(c, -wave_max_dpp(-lo), hi, k);
  } else {
    exact = true;
    __syncthreads();  // every wave has read the maxima; sm.cand is free
  }
  int nc;
  for (;;) {
    if (exact) {
      t = radix_kth<NE>(x, V, k, sm);
      all = t != t;  // no valid element
    }
    if (exact || have) {  // histograms lay over the candidates
      if (tid < 128) sm.cand[tid] = 0ull;
      __syncthreads();
    }
    // compaction: every lane marks its candidates; one LDS atomic per wave reserves the wave's places (their order
    // does not matter: the candidates are ranked by key below), and each round stores a lane's lowest remaining mark,
    // in ballot order. Two or three rounds: a lane rarely holds more, and the loop's few lines of code are fetched
    // once where a store per element was fetched NE times.
    unsigned int mark = 0;
    if (!have) {
#pragma unroll
      for (int e = 0; e < NE; ++e) mark |= (tid + ST * e < V && (all || x[e] >= t)) ? 1u << e : 0u;
    } else {
      mark = hmark;
    }
    const unsigned int mine = __popc(mark);
    const unsigned int upto = wave_incl_scan(mine);
    const int total = __builtin_amdgcn_readlane((int)upto, 63);
    int base = 0;
    if (lane == 0 && total > 0) base = (int)atomicAdd((unsigned int*)&sm.ncand, (unsigned int)total);
    int at = __builtin_amdgcn_readfirstlane(base) + (int)(upto - mine);
    while (__ballot(mark != 0)) {
      const int e = __ffs((int)mark) - 1;
      float v = x[0];
#pragma unroll
      for (int q = 1; q < NE; ++q) v = e == q ? x[q] : v;
      if (mark != 0)
        sm.cand[at++] = ((unsigned long long)ordkey(v) << 32) | (unsigned long long)(0xffffffffu - (uint32_t)(tid + ST * e));
      mark &= mark - 1;
    }
    __syncthreads();
    nc = sm.ncand;
    if (have || exact || nc <= ST) break;
    __syncthreads();  // every wave has read the count
    if (tid == 0) sm.ncand = 0;  // ordered before the next compaction by the radix select's barriers
    exact = true;
  }
  int P2 = 2;
  while (P2 < nc) P2 <<= 1;
  if (nc <= 128) {
    // The usual case: rank placement with the count split over the waves. Keys are distinct (the index is part
    // of the key), so candidate l goes to position #{j : key_j > key_l}. A lane takes candidates lane and lane + 64;
    // wave w counts the keys j in [J w, J w + J) (LDS broadcast reads), J = 16 or 32; the partial counts of both
    // (packed in 16 bits each) meet in sm.hist (free by now).
    const unsigned long long key0 = sm.cand[lane];  // 0 past the last candidate, up to 128
    const unsigned long long key1 = sm.cand[64 + lane];
    unsigned int part = 0;
    auto count16 = [&](int j0, bool two) {
      if (j0 >= nc) return;
      ulonglong2 c2[8];
#pragma unroll
      for (int q = 0; q < 8; ++q) c2[q] = *reinterpret_cast<const ulonglong2*>(&sm.cand[j0 + 2 * q]);
#pragma unroll
      for (int q = 0; q < 8; ++q) {
        part += (c2[q].x > key0 ? 1u : 0u) + (c2[q].y > key0 ? 1u : 0u);
        if (two) part += (c2[q].x > key1 ? 0x10000u : 0u) + (c2[q].y > key1 ? 0x10000u : 0u);
      }
    };
    if (nc <= 64) {
      count16(16 * wave, false);
    } else {
      count16(32 * wave, true);
      count16(32 * wave + 16, true);
    }
    sm.hist[tid] = part;
    __syncthreads();
    if (tid < nc) {
      const unsigned int r = sm.hist[lane] + sm.hist[64 + lane] + sm.hist[128 + lane] + sm.hist[192 + lane];
      sm.cand[tid < 64 ? r & 0xffffu : r >> 16] = tid < 64 ? key0 : key1;
    }
    __syncthreads();
  } else if (nc <= ST) {
    // rank placement, one candidate a thread; the reads of key_j are LDS broadcasts
    const unsigned long long key = tid < nc ? sm.cand[tid] : 0ull;
    int rank = 0;
    if ((tid & ~63) < nc) {  // waves holding no candidate skip the count
      for (int j = 0; j < nc; j += 16) {  // sixteen broadcast reads in flight per step (clamped, masked)
        unsigned long long c16[16];
#pragma unroll
        for (int q = 0; q < 16; ++q) c16[q] = sm.cand[min(j + q, nc - 1)];
#pragma unroll
        for (int q = 0; q < 16; ++q) rank += (j + q < nc && c16[q] > key) ? 1 : 0;
      }
    }
    __syncthreads();
    if (tid < nc) sm.cand[rank] = key;
    __syncthreads();
  } else {
  for (int i = nc + tid; i < P2; i += ST) sm.cand[i] = 0ull;
  __syncthreads();
  for (int kk = 2; kk <= P2; kk <<= 1) {
    for (int j = kk >> 1; j > 0; j >>= 1) {
      for (int t2 = tid; t2 < (P2 >> 1); t2 += ST) {
        const int i = ((t2 & ~(j - 1)) << 1) | (t2 & (j - 1));
        const int p = i | j;
        const unsigned long long a = sm.cand[i], b = sm.cand[p];
        const bool desc = (i & kk) == 0;
        if (desc ? (a < b) : (a > b)) {
          sm.cand[i] = b;
          sm.cand[p] = a;
        }
      }
      __syncthreads();
    }
  }
  }
  const int kk = k < nc ? k : nc;
  const float kth = ordkey_inv((uint32_t)(sm.cand[kk - 1] >> 32));
  const float x0 = ordkey_inv((uint32_t)(sm.cand[0] >> 32));
  // the kept set (x >= kth) is a prefix of the sorted order: its last member records the length
  for (int j = tid; j < nc; j += ST) {
    const float xj = ordkey_inv((uint32_t)(sm.cand[j] >> 32));
    if (xj >= kth) {
      sm.w[j] = m3x_expf(xj - x0);
      if (j + 1 == nc || !(ordkey_inv((uint32_t)(sm.cand[j + 1] >> 32)) >= kth)) sm.nkeep = j + 1;
    }
  }
  __syncthreads();
}

__device__ __forceinline__ int cand_index(unsigned long long c) { return (int)(0xffffffffu - (uint32_t)c); }

__device__ __forceinline__ float lanef(float v, int q) {
  return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), q));
}

// Sequential fp32 running sums of 64 values, 4 a lane in lanes 0..15 (w): run = carry + w_0 + ... in order, every sum
// rounded as one running total's. A lane adds its 4 values to the total that the lane before it holds (DPP row_shr:1;
// lane 0 reads +0 and has carry in its first value), 16 times over: lane l is final after l + 1 rounds and repeats the
// same sums from then on. Returns the total in every lane. One lane a value took 63 cross-lane steps and twice the
// time; rows 1..3 of the wave run along on their own values, unused.
__device__ __forceinline__ float wave_seq_scan(float4 w, float carry, float4& run) {
  if ((threadIdx.x & 63) == 0) w.x = carry + w.x;
  run = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll 2
  for (int q = 0; q < 16; ++q) {
    const float in = __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(run.w), 0x111, 0xf, 0xf, true));
    run.x = in + w.x;
    run.y = run.x + w.y;
    run.z = run.y + w.z;
    run.w = run.z + w.w;
  }
  return lanef(run.w, 15);
}

// The weights of positions j0 + 4 l .. + 3 of the kept set (lane l < 16; +0 past n).
template <class SM>
__device__ __forceinline__ float4 weights4(const SM& sm, int j0, int n) {
  const int j = j0 + 4 * (int)(threadIdx.x & 15);
  float4 w;
  w.x = sm.w[min(j, n - 1)];
  w.y = sm.w[min(j + 1, n - 1)];
  w.z = sm.w[min(j + 2, n - 1)];
  w.w = sm.w[min(j + 3, n - 1)];
  if (j >= n) w.x = 0.f;
  if (j + 1 >= n) w.y = 0.f;
  if (j + 2 >= n) w.z = 0.f;
  if (j + 3 >= n) w.w = 0.f;
  return w;
}

// Lane 0..15's first of its four running sums above t, over the wave: the position within the 64, or -1.
__device__ __forceinline__ int first_above(const float4& run, float t) {
  const int sub = run.x > t ? 0 : run.y > t ? 1 : run.z > t ? 2 : 3;
  const unsigned long long hit = __ballot((threadIdx.x & 63) < 16 && run.w > t);  // the sums do not fall
  if (!hit) return -1;
  const int l = __ffsll((long long)hit) - 1;
  return 4 * l + __builtin_amdgcn_readlane(sub, l);
}

// Inverse-CDF pick over cand[0..n) skipping index `skip` (-1: none): the first position whose running sum (the same
// sequential fp32 order as the total S) exceeds u * S, else the last term; -1 when the weights sum to 0. A skipped
// position counts +0, so its running sum is the one before it and is never the first above. Called by one whole wave;
// every lane returns the same index. Rows of more than 64 candidates sum twice. Zeroes the skipped weight in sm.w.
template <class SM>
__device__ int pick(SM& sm, int n, float u, int skip) {
  const int lane = threadIdx.x & 63;
  if (n <= 0) return -1;
  int last = n - 1;
  if (skip >= 0) {
    for (int j0 = 0; j0 < n; j0 += 64) {
      const int j = j0 + lane;
      const bool is = j < n && cand_index(sm.cand[j]) == skip;
      if (is) sm.w[j] = 0.f;
    }
    __builtin_amdgcn_wave_barrier();
    if (cand_index(sm.cand[last]) == skip) --last;
  }
  float4 run;
  float S = wave_seq_scan(weights4(sm, 0, n), 0.f, run);
  for (int j0 = 64; j0 < n; j0 += 64) {
    float4 r;
    S = wave_seq_scan(weights4(sm, j0, n), S, r);
  }
  if (last < 0 || !(S > 0.f)) return -1;
  const float t = u * S;
  int at = first_above(run, t);
  if (at < 0 && n > 64) {
    float c = lanef(run.w, 15);
    for (int j0 = 64; j0 < n && at < 0; j0 += 64) {
      float4 r;
      c = wave_seq_scan(weights4(sm, j0, n), c, r);
      at = first_above(r, t);
      if (at >= 0) at += j0;
    }
  }
  return cand_index(sm.cand[at >= 0 && at <= last ? at : last]);
}

// Top-p cut of the kept set cand[0..n) (maya3/engine.py:669-672: a candidate is dropped when the probability mass
// sorted before it exceeds top_p): position j stays while run_(j-1) / S <= top_p, where run is the sequential fp32
// running sum of the weights in order (wave_seq_scan) and S their total in the same order.
// The kept set stays a prefix of the order. Called by one whole wave; leaves sm.w unchanged; returns the new
// length (>= 1) in every lane.
template <class SM>
__device__ int top_p_keep(const SM& sm, int n, float top_p) {
  float S = 0.f;
  float4 r;
  for (int j0 = 0; j0 < n; j0 += 64) S = wave_seq_scan(weights4(sm, j0, n), S, r);
  float carry = 0.f;
  for (int j0 = 0; j0 < n; j0 += 64) {
    carry = wave_seq_scan(weights4(sm, j0, n), carry, r);
    // the first j with run_j / S > top_p keeps 0 .. j (the quotients do not fall)
    const float4 p = make_float4(r.x / S, r.y / S, r.z / S, r.w / S);
    const int at = first_above(p, top_p);
    if (at >= 0) return min(j0 + at + 1, n);
  }
  return n;
}
}  // namespace
