// Row softmax of attention scores, bit for bit the reference's.
//
// The reference softmaxes each row of scores in place (src/shaders/softmax_rows.wgsl:1-55,
// one invocation per row; dispatched at src/engine/forward.ts:912-926) and checks it against
// softmaxRows (src/reference/cpu.ts:238-264), whose arithmetic is f32 throughout:
//   valid = causal_period ? causal_offset + (row % causal_period) + 1 : row_len
//   M     = Math.max over the row's first `valid` entries (a NaN makes it NaN)
//   e_i   = f32(Math.exp(f32(x_i - M)));  S = f32(S + e_i) left to right from 0
//   out_i = f32(e_i * f32(1 / S)) for i < valid, 0 for the masked rest.
// x_i - M is one f32 subtraction (the reference rounds the f64
// difference of two f32 values to f32, which is the same number); Math.exp rounded to f32 is
// exp_to_f32 (a fast f64 exp, V8's fdlibm method where the f32 rounding is close); 1 / S is an
// f64 division rounded to f32, as JS evaluates it; e_i * inv is one f32 multiplication (the f64
// product of two f32 values is exact, so JS's rounding of it to f32 is the f32 product).
//
// The sequential f32 sum keeps every bit in one of three ways: by one lane per row, as the
// reference adds it (softmax_rows_block_kernel); by chunks whose sums do not depend on the
// running sum (softmax_rows_chunk_kernel); and, for rows too long for registers, by the whole
// wave in steps of 64 (the f32 form of the method in seqsum.h): while the running sum P = m * u
// lies in one binade, with ulp u = 2^(E-23) and integer m < 2^24, fl(P + t) = (m + rint(t / u))
// * u exactly, with an exact half-ulp tie going to the even result (a parity automaton scanned
// over the lanes); so the partial sums are m plus an integer prefix sum, and only a term that
// takes m to 2^24 or beyond (the sum leaves the binade) is added on its own, after which the
// scan resumes. A row of n terms has about log2(n) such events.
//
// Rows of up to 16,384 entries are read once into registers and written once: HBM traffic
// 2 * row_len * 4 bytes, rows at any 4-byte boundary. Longer rows take three passes (max; exp,
// sum and the exps written to `out`; the scaling), as the reference's kernel does.

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <algorithm>
#include <string>

#include "abi_internal.h"
#include "device_math.h"
#include "seqsum.h"
#include "wave_ops.h"

namespace tabby {
namespace {

constexpr int kSmWaves = 4;  // rows per workgroup, one wave each
constexpr int kBlockMinRows = 256;       // rows of up to 512 entries: a lane adds a row from here on
constexpr int kTinyCols = 64;            // one group of one entry per lane
constexpr int kElementCols = 384;        // one entry per lane at a time up to here
constexpr int kBlockMinLongRows = 1024;  // rows of 513-1,024 entries
constexpr int kChunkCols = 16384;        // longest row held in a workgroup's registers
constexpr int kMaxRowThreads = 1024;     // of softmax_rows_chunk_kernel
constexpr int kLaunchRows = (int)(((int64_t)1 << 32) / kMaxRowThreads) - 1;
constexpr double kTwo24 = 16777216.0;
constexpr double kTwo25 = 33554432.0;

typedef float sm_f32x4 __attribute__((ext_vector_type(4)));

// Parity (0/1) of an integer-valued double; values that large only occur at event
// positions, whose parity is never used.
__device__ __forceinline__ uint32_t parity_of(double integral) {
  return (uint32_t)(int64_t)fmin(integral, 1.0e15) & 1u;
}

// P + t_0 + t_1 + ... in f32, one rounding per addition, left to right, over one step of the
// row: lane l holds the step's terms l*V .. l*V + V - 1 in t[]. P is wave-uniform; terms are
// >= 0 and finite (a NaN term makes the sum NaN, as it would sequentially). Returns the sum.
template <int V>
__device__ float seq_sum_f32_step(float P, const float (&t)[V]) {
  const int lane = wave_lane();
  bool nan = false;
#pragma unroll
  for (int j = 0; j < V; ++j) nan |= t[j] != t[j];
  if (P != P || __ballot(nan)) return __builtin_nanf("");
  int start = 0;  // positions of the step below this one are in P already
  while (true) {
    // P = m * 2^sh with m an integer below 2^24 (sh = -149 for zero and subnormal P).
    const int ef = (int)(__float_as_uint(P) >> 23);
    const int sh = (ef == 0 ? 1 : ef) - 150;
    const double m = __builtin_ldexp((double)P, -sh);
    double inc[V], fl[V];
    bool tie[V];
    bool any_tie = false;
#pragma unroll
    for (int j = 0; j < V; ++j) {
      const bool active = lane * V + j >= start;
      const double x = active ? __builtin_ldexp((double)t[j], -sh) : 0.0;  // t / u, exact
      fl[j] = __builtin_floor(x);
      tie[j] = x - fl[j] == 0.5;
      inc[j] = tie[j] ? fl[j] : __builtin_rint(x);
      any_tie |= tie[j];
    }
    if (__ballot(any_tie)) {
      // A tie adds fl or fl + 1, whichever leaves m even: the parity of m before every term,
      // from the maps x -> (x & k) ^ c (a non-tie XORs its increment's parity, a tie resets
      // to 0) composed over the lanes below and this lane's earlier terms.
      uint32_t f[V];
      uint32_t lane_map = kParityId;
#pragma unroll
      for (int j = 0; j < V; ++j) {
        f[j] = tie[j] ? 0u : (1u | (parity_of(inc[j]) << 1));
        lane_map = parity_then(lane_map, f[j]);
      }
      uint32_t p = parity_apply(parity_exclusive_scan(lane_map), parity_of(m));
#pragma unroll
      for (int j = 0; j < V; ++j) {
        if (tie[j]) inc[j] = fl[j] + (double)((p + parity_of(fl[j])) & 1u);
        p = parity_apply(f[j], p);
      }
    }
    // An increment of 2^24 or more is an event whatever its size: capped at 2^25, every
    // prefix below stays an exact integer (64 * V * 2^25 < 2^53).
#pragma unroll
    for (int j = 0; j < V; ++j) inc[j] = fmin(inc[j], kTwo25);
    double c[V];
    c[0] = inc[0];
#pragma unroll
    for (int j = 1; j < V; ++j) c[j] = c[j - 1] + inc[j];
    const double below = wave_inclusive_scan(c[V - 1]) - c[V - 1];
    int first = V;
#pragma unroll
    for (int j = V - 1; j >= 0; --j)
      if (m + (below + c[j]) >= kTwo24) first = j;
    const uint64_t ev = __ballot(first < V);
    if (!ev) return (float)__builtin_ldexp(m + lane_f64(below + c[V - 1], kWaveSize - 1), sh);
    // The first event: every term before it is exact in the integer sum; it is added alone.
    const int L = __ffsll((unsigned long long)ev) - 1;
    const int j = __builtin_amdgcn_readlane(first, L);
    double before = below;
    float tj = t[0];
#pragma unroll
    for (int i = 0; i < V; ++i)
      if (i == j) {
        before = i == 0 ? below : below + c[i > 0 ? i - 1 : 0];
        tj = t[i];
      }
    const float p_before = (float)__builtin_ldexp(m + lane_f64(before, L), sh);
    P = p_before + __uint_as_float((uint32_t)__builtin_amdgcn_readlane((int)__float_as_uint(tj), L));
    start = L * V + j + 1;
    if (start >= kWaveSize * V) return P;
  }
}

// fround(Math.exp(d)), d = x_i - M <= 0 or NaN (exp_to_f32).
__device__ __forceinline__ float exp_f32_of(float d) { return exp_to_f32(d); }

struct RowDims {
  int n_rows;
  int row_len;
  int causal_period;
  int causal_offset;
};

__device__ __forceinline__ int valid_of(const RowDims &d, int row) {
  return d.causal_period != 0 ? d.causal_offset + (row % d.causal_period) + 1 : d.row_len;
}

// Four consecutive floats at any 4-byte boundary (rows of any length need no alignment).
typedef float sm_f32x4u __attribute__((ext_vector_type(4), aligned(4)));

// ---------------------------------------------------------------------------------------
// Rows summed by chunks (softmax_rows_chunk_kernel): thread t of a row's NW waves holds the
// row's entries [t * K, (t + 1) * K), K <= 4 Q, from the load to the store, and the sequential
// sum is made of the chunks' own sequential sums.
//
// Let the running sum be P before a chunk and P' after it. If both lie in one binade
// [B, 2B), with ulp u = B * 2^-23, every addition of the chunk adds an integer number of ulps
// that depends on the term and, for an exact half-ulp tie, on the parity of the running sum;
// so the chunk adds c0 to an even P and c1 to an odd one, whatever P is otherwise. c0 and c1
// come from adding the chunk's terms to B and to B + u in f32, as the reference adds them
// (both stay below 2B, because P' does: B + (P' - P) < 2B); all threads do so at once. Which binade holds P is
// known beforehand from the f64 prefix sums A of the exps: a sequential f32 sum of n
// non-negative terms is within n * 2^-24 of its value, so P >= A0 (1 - g) and P' <= A1 (1 + g)
// with g = (n + 64) * 2^-24 * 1.02 (64: the chunk's own f32 total and the comparisons).
// Chunks for which that does not settle the binade -- the ones where the sum crosses a power
// of two, about log2(n) of them -- are added term by term, in order, by the wave that walks
// the chunks: between two such chunks the c0 sum to an exact f64 (multiples of one u below
// 2^53), so a run of chunks is one addition.
//
// What bounds it: one row per head in a decode step leaves the chip idle, so the call is the
// latency of this chain (loads, max, exps, one scan, the walk). Taking the row in steps of 256
// entries, each with its own scan and a restart per crossing, 14 rows of 1,024, 4,096 and 8,192
// entries took 18.2, 53.1 and 99.2 us per call; this takes 5.9, 8.3 and 10.7 us in the kernel
// (7.7, 7.8 and 10.2 us per call back to back, the first two bound by the host's launches).
// Waves and entries per thread are the fastest for that many entries among 1-16 waves and
// 4-16 entries, on one row per head and on thousands (14 x 1,024 rows of 1,536: 49 us with two
// waves of 16, 59 with four of 8, 93 with eight of 4, and 132 in steps).
// ---------------------------------------------------------------------------------------
template <int NW, int Q>
struct alignas(16) ChunkSmem {
  static constexpr int kThreads = NW * kWaveSize;
  float e[kThreads * 4 * Q];  // the exps of chunks added term by term
  double excl[kThreads];      // sum of the c0 of the wave's chunks before this one
  float c[2][kThreads];       // c0, c1
  double scan_total[NW];
  uint64_t serial[NW], parity[NW];  // chunks added term by term; chunks with c0 != c1
  double wave_total[NW];
  float wave_max[NW];
  float inv;
};

template <int NW, int Q>
__global__ __launch_bounds__(NW == 1 ? kSmWaves * kWaveSize : NW * kWaveSize) void softmax_rows_chunk_kernel(
    const float *x, float *out, RowDims d) {
  constexpr int K = 4 * Q;
  constexpr int kRows = NW == 1 ? kSmWaves : 1;  // rows per workgroup
  constexpr int kThreads = NW * kWaveSize;
  __shared__ ChunkSmem<NW, Q> smem[kRows];
  const int lane = wave_lane();
  const int wave_in_group = __builtin_amdgcn_readfirstlane((int)threadIdx.x / kWaveSize);
  const int row = NW == 1 ? (int)blockIdx.x * kRows + wave_in_group : (int)blockIdx.x;
  if (NW == 1 && row >= d.n_rows) return;  // a whole wave; NW == 1 has no barrier
  ChunkSmem<NW, Q> &sm = smem[NW == 1 ? wave_in_group : 0];
  const int wave = NW == 1 ? 0 : wave_in_group;
  const int t = wave * kWaveSize + lane;
  const int valid = valid_of(d, row);
  const float *src = x + (size_t)row * d.row_len;
  float *dst = out + (size_t)row * d.row_len;
  // Groups of four entries per thread that this row needs: a short causal prefix takes less.
  const int qn = min(Q, (valid + 4 * kThreads - 1) / (4 * kThreads));
  const int first = t * 4 * qn;

  float v[K];
#pragma unroll
  for (int q = 0; q < Q; ++q) {
    const int i = first + 4 * q;
    if (q < qn && i + 4 <= valid) {
      const sm_f32x4u f = *reinterpret_cast<const sm_f32x4u *>(src + i);
#pragma unroll
      for (int j = 0; j < 4; ++j) v[4 * q + j] = f[j];
    } else {
#pragma unroll
      for (int j = 0; j < 4; ++j) v[4 * q + j] = q < qn && i + j < valid ? src[i + j] : -INFINITY;
    }
  }
  // Math.max: the largest valid entry, NaN if any valid entry is NaN.
  float mx = -INFINITY;
  bool nan = false;
#pragma unroll
  for (int k = 0; k < K; ++k) {
    mx = fmaxf(mx, v[k]);
    nan |= v[k] != v[k];
  }
  mx = wave_max(mx);
  if (__ballot(nan)) mx = __builtin_nanf("");
  if constexpr (NW > 1) {
    if (lane == 0) sm.wave_max[wave] = mx;
    __syncthreads();
    const float m = sm.wave_max[lane % NW];
    mx = wave_max(m);
    if (__ballot(m != m)) mx = __builtin_nanf("");
  }

  // The exps; v becomes them. Arguments that need V8's method take it through LDS, so that its
  // code is here once.
  float *mine = sm.e + t * K;
  uint32_t slow = 0u;
  float sum = 0.0f;
#pragma unroll
  for (int q = 0; q < Q; ++q) {
    if (q < qn) {
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int k = 4 * q + j;
        const float a = v[k] - mx;
        bool s;
        const float e = exp_to_f32_fast(a, s);
        const bool in = first + k < valid;
        slow |= in && s ? 1u << k : 0u;
        v[k] = !in ? 0.0f : s ? a : e;
      }
    } else {
#pragma unroll
      for (int j = 0; j < 4; ++j) v[4 * q + j] = 0.0f;
    }
  }
  if (__ballot(slow != 0u)) {
#pragma unroll
    for (int k = 0; k < K; ++k) mine[k] = v[k];
    for (uint32_t b = slow; b != 0u; b &= b - 1u) {
      const int k = __ffs((int)b) - 1;
      mine[k] = exp_to_f32_slow(mine[k]);
    }
#pragma unroll
    for (int k = 0; k < K; ++k) v[k] = mine[k];
  }
#pragma unroll
  for (int k = 0; k < K; ++k) sum += v[k];

  // The f64 prefix sums and what they say about each chunk's binade.
  const double incl = wave_inclusive_scan((double)sum);
  double base = 0.0;
  if constexpr (NW > 1) {
    if (lane == kWaveSize - 1) sm.wave_total[wave] = incl;
    __syncthreads();
    const double totals = wave_inclusive_scan(lane < NW ? sm.wave_total[lane] : 0.0);
    if (wave > 0) base = lane_f64(totals, wave - 1);
  }
  const double g = (double)(valid + 64) * (1.02 * 0x1p-24);
  const float lo = (float)((base + (incl - (double)sum)) * (1.0 - g));
  const float hi = (float)((base + incl) * (1.0 + g));
  const float B = __uint_as_float(__float_as_uint(lo) & 0x7f800000u);
  const bool none = sum == 0.0f;  // zeros change no sum
  bool known = none || (lo >= 0x1p-100f && hi < 2.0f * B);
  // The wave's c0 are summed in f64: exact while they are multiples of one 2^-23 B0 and their
  // total is below 2^28 B0, B0 the wave's smallest known binade (its first).
  const uint64_t settled = __ballot(known && !none);
  if (settled) {
    const int at = __ffsll((unsigned long long)settled) - 1;
    const float b0 = __uint_as_float((uint32_t)__builtin_amdgcn_readlane((int)__float_as_uint(B), at));
    const float end = __uint_as_float((uint32_t)__builtin_amdgcn_readlane((int)__float_as_uint(hi), kWaveSize - 1));
    if (!(end < b0 * 0x1p28f)) known = none;
  }
  const bool use = known && !none;
  float s0 = use ? B : 1.0f;
  const float base0 = s0, base1 = s0 + s0 * 0x1p-23f;
  float s1 = base1;
#pragma unroll
  for (int k = 0; k < K; ++k) {
    s0 = s0 + v[k];
    s1 = s1 + v[k];
  }
  const float c0 = use ? s0 - base0 : 0.0f, c1 = use ? s1 - base1 : 0.0f;
  const uint64_t serial = __ballot(!known), parity = __ballot(c0 != c1);
  const double c_incl = wave_inclusive_scan(c0 == c1 ? (double)c0 : 0.0);
  const double c_excl = c_incl - (c0 == c1 ? (double)c0 : 0.0);
  if (serial) {
    if (!known) {
#pragma unroll
      for (int k = 0; k < K; ++k) mine[k] = v[k];
    }
  }
  if constexpr (NW > 1) {
    sm.excl[t] = c_excl;
    sm.c[0][t] = c0;
    sm.c[1][t] = c1;
    if (lane == 0) {
      sm.serial[wave] = serial;
      sm.parity[wave] = parity;
    }
    if (lane == kWaveSize - 1) sm.scan_total[wave] = c_incl;
    __syncthreads();
  } else {
    wave_lds_sync();
  }

  // The walk, by the row's first wave, all lanes alike.
  float inv = 0.0f;
  if (NW == 1 || wave == 0) {
    float P = 0.0f;
    for (int w = 0; w < NW; ++w) {
      const uint64_t ser = NW == 1 ? serial : sm.serial[w];
      uint64_t stops = ser | (NW == 1 ? parity : sm.parity[w]);
      const double total = NW == 1 ? lane_f64(c_incl, kWaveSize - 1) : sm.scan_total[w];
      double done = 0.0;  // c0 sum already in P
      while (stops) {
        const int j = __builtin_amdgcn_readfirstlane(__ffsll((unsigned long long)stops) - 1);
        stops &= stops - 1;
        const int at = w * kWaveSize + j;
        const double before = NW == 1 ? lane_f64(c_excl, j) : sm.excl[at];
        if (before != done) P = (float)((double)P + (before - done));
        done = before;
        if ((ser >> j) & 1ull) {
          const sm_f32x4 *e4 = reinterpret_cast<const sm_f32x4 *>(sm.e + at * K);
          sm_f32x4 e[Q];
#pragma unroll
          for (int q = 0; q < Q; ++q) e[q] = e4[q];
#pragma unroll
          for (int q = 0; q < Q; ++q) {
            P = P + e[q].x;
            P = P + e[q].y;
            P = P + e[q].z;
            P = P + e[q].w;
          }
        } else {
          const bool odd = (__float_as_uint(P) & 1u) != 0u;
          P = P + (NW == 1 ? __uint_as_float((uint32_t)__builtin_amdgcn_readlane(
                                 (int)__float_as_uint(odd ? c1 : c0), j))
                           : sm.c[odd ? 1 : 0][at]);
        }
      }
      if (total != done) P = (float)((double)P + (total - done));
    }
    inv = (float)(1.0 / (double)P);
    if constexpr (NW > 1) {
      if (lane == 0) sm.inv = inv;
    }
  }
  if constexpr (NW > 1) {
    __syncthreads();
    inv = sm.inv;
  }

#pragma unroll
  for (int q = 0; q < Q; ++q) {
    const int i = first + 4 * q;
    if (q < qn && i < d.row_len) {
      sm_f32x4u o;
#pragma unroll
      for (int j = 0; j < 4; ++j) o[j] = i + j < valid ? v[4 * q + j] * inv : 0.0f;
      if (i + 4 <= d.row_len) {
        *reinterpret_cast<sm_f32x4u *>(dst + i) = o;
      } else {
#pragma unroll
        for (int j = 0; j < 3; ++j)
          if (i + j < d.row_len) dst[i + j] = o[j];
      }
    }
  }
  // The masked entries past the threads' chunks.
  for (int i = 4 * (qn * kThreads + t); i < d.row_len; i += 4 * kThreads) {
    if (i + 4 <= d.row_len) {
      *reinterpret_cast<sm_f32x4u *>(dst + i) = sm_f32x4u{0.0f, 0.0f, 0.0f, 0.0f};
    } else {
      for (int j = i; j < d.row_len; ++j) dst[j] = 0.0f;
    }
  }
}

// Many rows of at most COLS entries: four rows per workgroup of four waves, a wave per row for
// the loads, the row max (DPP) and the exps, which stay in registers and are left in LDS too;
// then lane r of wave 0 adds row r's exps left to right -- the reference's own sequential f32
// sum, one row per lane -- and each wave scales its row from registers and writes it.
// HBM traffic 2 * row_len * 4 bytes per row at most. The sum is a chain of row_len dependent
// adds per lane whose instructions four rows share; the other waves of the CU's workgroups
// load, exponentiate and store meanwhile.
// 14 x 512 causal rows of 512 (22 MB): 11.0 us, 11.8 with the sum reading eight entries ahead,
// element loads and stores and the exps read back from LDS. 14 x 1,024 of 1,024 (88 MB): 27.4
// us, by chunks 33.0, in steps of 256 73. Eight rows per workgroup took 33 us there: fewer
// workgroups of a CU are then in different phases.
//
// VEC: consecutive entries per lane. Four (16-byte loads and stores) take the row in groups of 256,
// whose exps -- what the kernel issues most of -- cost the same however few of them lie in the row;
// one takes it in groups of 64. 28,672 rows of 32, 128, 257 and 384 entries: 14.4, 16.6, 26.0 and
// 26.8 us by fours, 7.9, 12.6, 22.8 and 25.6 by ones (rows of up to 64 in a tile of their own that
// reads eight entries ahead: 9.6 in the tile of 512); of 448: 28.0 against 28.9.
template <int COLS, int VEC>
__global__ __launch_bounds__(kSmWaves *kWaveSize) void softmax_rows_block_kernel(const float *x, float *out,
                                                                                 RowDims d) {
  // Row pitch: four pad words put the four rows the sum reads at once on different banks.
  constexpr int kPitch = COLS + 4;
  constexpr int kGroup = VEC * kWaveSize;
  constexpr int kGroups = COLS / kGroup;
  static_assert(kGroups * VEC <= 32, "a bit per entry of a lane");
  constexpr int kStep = COLS <= kTinyCols ? 8 : 32;  // entries the sum reads ahead of its adds
  __shared__ __align__(16) float tile[kSmWaves * kPitch + kStep];
  __shared__ float inv[kSmWaves];
  const int lane = wave_lane();
  const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x / kWaveSize);
  const int row0 = (int)blockIdx.x * kSmWaves;
  const int rows = min(kSmWaves, d.n_rows - row0);
  const int row = row0 + wave;
  const int valid = wave < rows ? valid_of(d, row) : 0;
  const float *src = x + (size_t)row * d.row_len;
  float *mine = tile + wave * kPitch + VEC * lane;
  float v[kGroups][VEC];
#pragma unroll
  for (int k = 0; k < kGroups; ++k) {
    const int i = k * kGroup + VEC * lane;
    if (VEC == 4 && i + VEC <= valid) {
      const sm_f32x4u f = __builtin_nontemporal_load(reinterpret_cast<const sm_f32x4u *>(src + i));
#pragma unroll
      for (int j = 0; j < VEC; ++j) v[k][j] = f[j];
    } else {
#pragma unroll
      for (int j = 0; j < VEC; ++j) v[k][j] = i + j < valid ? src[i + j] : -INFINITY;
    }
  }
  float mx = -INFINITY;
  bool nan = false;
#pragma unroll
  for (int k = 0; k < kGroups; ++k)
#pragma unroll
    for (int j = 0; j < VEC; ++j) {
      mx = fmaxf(mx, v[k][j]);
      nan |= v[k][j] != v[k][j];
    }
  mx = wave_max(mx);
  if (__ballot(nan)) mx = __builtin_nanf("");
  uint32_t slow = 0u;
#pragma unroll
  for (int k = 0; k < kGroups; ++k) {
    if (k * kGroup < valid) {  // uniform: groups past the row's end or its causal prefix cost nothing
#pragma unroll
      for (int j = 0; j < VEC; ++j) {
        const float a = v[k][j] - mx;
        bool s;
        const float e = exp_to_f32_fast(a, s);
        const bool in = k * kGroup + VEC * lane + j < valid;
        slow |= in && s ? 1u << (VEC * k + j) : 0u;
        v[k][j] = !in ? 0.0f : s ? a : e;
      }
      if constexpr (VEC == 4) {
        *reinterpret_cast<sm_f32x4 *>(mine + k * kGroup) = sm_f32x4{v[k][0], v[k][1], v[k][2], v[k][3]};
      } else {
        mine[k * kGroup] = v[k][0];
      }
    }
  }
  if (__ballot(slow != 0u)) {  // V8's method, once for all entries, through LDS
    for (uint32_t b = slow; b != 0u; b &= b - 1u) {
      const int k = __ffs((int)b) - 1;
      float *at = mine + (k / VEC) * kGroup + k % VEC;
      *at = exp_to_f32_slow(*at);
    }
#pragma unroll
    for (int k = 0; k < kGroups; ++k)
      if (k * kGroup < valid) {
#pragma unroll
        for (int j = 0; j < VEC; ++j) v[k][j] = mine[k * kGroup + j];
      }
  }
  __syncthreads();
  if (wave == 0 && lane < rows) {
    // The row's exps left to right (zeros past its end change nothing); the next kStep are read
    // while these are added.
    const int n = valid_of(d, row0 + lane);
    const sm_f32x4 *t4 = reinterpret_cast<const sm_f32x4 *>(tile + lane * kPitch);
    float sum = 0.0f;
    sm_f32x4 q[kStep / 4];
#pragma unroll
    for (int j = 0; j < kStep / 4; ++j) q[j] = t4[j];
    for (int i = 0; i < n; i += kStep) {
      t4 += kStep / 4;
#pragma unroll
      for (int j = 0; j < kStep / 4; ++j) {
        const sm_f32x4 now = q[j];
        q[j] = t4[j];  // past a full row: the next row's, or the tile's padding; never added
        sum = sum + now.x;
        sum = sum + now.y;
        sum = sum + now.z;
        sum = sum + now.w;
      }
    }
    inv[lane] = (float)(1.0 / (double)sum);
  }
  __syncthreads();
  if (wave >= rows) return;
  const float q = inv[wave];
  float *dst = out + (size_t)row * d.row_len;
#pragma unroll
  for (int k = 0; k < kGroups; ++k) {
    const int i = k * kGroup + VEC * lane;
    if constexpr (VEC == 4) {
      sm_f32x4u o;
#pragma unroll
      for (int j = 0; j < 4; ++j) o[j] = i + j < valid ? v[k][j] * q : 0.0f;
      if (i + 4 <= d.row_len) {
        __builtin_nontemporal_store(o, reinterpret_cast<sm_f32x4u *>(dst + i));
      } else {
#pragma unroll
        for (int j = 0; j < 3; ++j)
          if (i + j < d.row_len) dst[i + j] = o[j];
      }
    } else {
      if (i < d.row_len) __builtin_nontemporal_store(i < valid ? v[k][0] * q : 0.0f, dst + i);
    }
  }
}

// Any row: three passes of one element per lane per step (64 entries), as the reference's
// kernel makes them -- max; exp, sum and e_i written to out; out_i = e_i * inv and the
// masked tail zeroed. In place (out == x) each lane rewrites only entries it has read.
__global__ __launch_bounds__(kSmWaves *kWaveSize) void softmax_rows_stream_kernel(const float *x, float *out,
                                                                                  RowDims d) {
  const int row = (int)blockIdx.x * kSmWaves + (int)threadIdx.x / kWaveSize;
  if (row >= d.n_rows) return;
  const int lane = wave_lane();
  const int valid = valid_of(d, row);
  const float *src = x + (size_t)row * d.row_len;
  float *dst = out + (size_t)row * d.row_len;
  float mx = -INFINITY;
  bool nan = false;
  for (int i = lane; i < valid; i += kWaveSize) {
    const float v = src[i];
    mx = fmaxf(mx, v);
    nan |= v != v;
  }
  mx = wave_max(mx);
  if (__ballot(nan)) mx = __builtin_nanf("");
  float P = 0.0f;
  for (int base = 0; base < valid; base += kWaveSize) {
    const int i = base + lane;
    float e[1];
    e[0] = i < valid ? exp_f32_of(src[i] - mx) : 0.0f;
    if (i < valid) dst[i] = e[0];
    P = seq_sum_f32_step<1>(P, e);
  }
  const float inv = (float)(1.0 / (double)P);
  for (int i = lane; i < d.row_len; i += kWaveSize) dst[i] = i < valid ? dst[i] * inv : 0.0f;
}

template <int NW, int Q>
void launch_chunks(const float *x, float *out, const RowDims &d, hipStream_t s) {
  static_assert(NW * Q * 256 <= kChunkCols, "no wider than the widest rows held in registers");
  static_assert(NW * kWaveSize <= kMaxRowThreads, "kLaunchRows");
  const int per_group = NW == 1 ? kSmWaves : 1;
  hipLaunchKernelGGL((softmax_rows_chunk_kernel<NW, Q>), dim3((unsigned)((d.n_rows + per_group - 1) / per_group)),
                     dim3((unsigned)(NW * per_group * kWaveSize)), 0, s, x, out, d);
}

// One launch (at most kLaunchRows rows).
void launch_rows(const float *x, float *out, const RowDims &d, hipStream_t s) {
  const dim3 grid((unsigned)((d.n_rows + kSmWaves - 1) / kSmWaves)), block(kSmWaves * kWaveSize);
  // Rows of up to kChunkCols entries are held in registers from the load to the store; longer
  // ones take three passes. Enough rows to fill the chip share the instructions of their sums
  // (softmax_rows_block_kernel, four rows per wave's adds; an entry per lane at a time up to
  // kElementCols, four beyond), up to 1,024 entries: 14 x 1,024
  // causal rows of 1,024 took 27.4 us against 33.0 by chunks, but 280 rows of 920 took 9.6 us
  // against 7.1, and 14 x 512 rows of 2,048 took 44.2 us (with room for 2,048) against 41.7.
  if (d.row_len <= 512 && d.n_rows >= kBlockMinRows) {
    if (d.row_len <= kTinyCols) hipLaunchKernelGGL((softmax_rows_block_kernel<kTinyCols, 1>), grid, block, 0, s, x, out, d);
    else if (d.row_len <= kElementCols) hipLaunchKernelGGL((softmax_rows_block_kernel<512, 1>), grid, block, 0, s, x, out, d);
    else hipLaunchKernelGGL((softmax_rows_block_kernel<512, 4>), grid, block, 0, s, x, out, d);
  } else if (d.row_len <= 1024 && d.n_rows >= kBlockMinLongRows) {
    hipLaunchKernelGGL((softmax_rows_block_kernel<1024, 4>), grid, block, 0, s, x, out, d);
  } else if (d.row_len <= 512) {
    launch_chunks<1, 2>(x, out, d, s);
  } else if (d.row_len <= 1024) {
    launch_chunks<4, 1>(x, out, d, s);
  } else if (d.row_len <= 2048) {
    launch_chunks<2, 4>(x, out, d, s);
  } else if (d.row_len <= 4096) {
    launch_chunks<4, 4>(x, out, d, s);
  } else if (d.row_len <= 8192) {
    launch_chunks<8, 4>(x, out, d, s);
  } else if (d.row_len <= kChunkCols) {
    launch_chunks<16, 4>(x, out, d, s);
  } else {
    hipLaunchKernelGGL(softmax_rows_stream_kernel, grid, block, 0, s, x, out, d);
  }
}

__global__ void exp_f32_kernel(const float *x, float *y, int64_t n) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) y[i] = exp_f32_of(x[i]);
}

}  // namespace
}  // namespace tabby

using namespace tabby;

extern "C" int tabby_debug_exp_f32(const float *x_dev, float *y_dev, int64_t n, void *stream) {
  if (!x_dev || !y_dev) return record_failure(TABBY_EINVAL, "null pointer");
  if (n < 1 || n > ((int64_t)1 << 31)) return record_failure(TABBY_EINVAL, "n must be in [1, 2^31]");
  hipLaunchKernelGGL(exp_f32_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, (hipStream_t)stream, x_dev,
                     y_dev, n);
  TABBY_HIP_CHECK(hipGetLastError());
  return TABBY_OK;
}

extern "C" int tabby_softmax_rows_device(const float *x_dev, float *out_dev, int32_t n_rows, int32_t row_len,
                                         int32_t causal_period, int32_t causal_offset, void *stream) {
  if (!x_dev || !out_dev) return record_failure(TABBY_EINVAL, "null pointer");
  if (n_rows < 1 || row_len < 1) return record_failure(TABBY_EINVAL, "n_rows and row_len must be >= 1");
  if (causal_period < 0 || causal_offset < 0)
    return record_failure(TABBY_EINVAL, "causal_period and causal_offset must be >= 0");
  if (causal_period > 0 && (int64_t)causal_offset + causal_period > row_len)
    return record_failure(TABBY_EINVAL, "causal_offset + causal_period (" +
                                            std::to_string((int64_t)causal_offset + causal_period) +
                                            ") exceeds row_len (" + std::to_string(row_len) + ")");
  if ((int64_t)n_rows * row_len > ((int64_t)1 << 40)) return record_failure(TABBY_EINVAL, "tensor too large");
  // In place or disjoint: a partial overlap would let one row's writes reach another's reads.
  const char *xb = (const char *)x_dev, *ob = (const char *)out_dev;
  const size_t bytes = (size_t)n_rows * row_len * sizeof(float);
  if (xb != ob && xb < ob + bytes && ob < xb + bytes)
    return record_failure(TABBY_EINVAL, "out must be x itself or not overlap it");
  const hipStream_t s = (hipStream_t)stream;
  // A launch takes fewer than 2^32 threads (past that its grid wraps, with no error), and a row at most
  // kMaxRowThreads: larger batches go in several, each of whole causal periods, so that every row keeps
  // its place in its own. (causal_period <= row_len, which is below 2^18 for that many rows.)
  const int step = causal_period > 0 && n_rows > kLaunchRows ? kLaunchRows / causal_period * causal_period : kLaunchRows;
  for (int64_t row = 0; row < n_rows; row += step) {
    const RowDims d{(int)std::min<int64_t>(step, n_rows - row), row_len, causal_period, causal_offset};
    launch_rows(x_dev + row * row_len, out_dev + row * row_len, d, s);
  }
  TABBY_HIP_CHECK(hipGetLastError());
  return TABBY_OK;
}
