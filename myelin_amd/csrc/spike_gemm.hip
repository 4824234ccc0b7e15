// fp32 synapse currents of spikes (0/1 inputs) on the int8 MFMA.
//
// An fp32 weight column is written as a 31-bit fixed-point number against
// its own largest magnitude: w = scale * q, |q| <= 2^30, scale a power of
// two, and q as four balanced base-256 digits q = d3 2^24 + d2 2^16 + d1 2^8
// + d0.  Weights down to 2^-6 of their column's largest keep every bit of
// their fp32 value; smaller ones are off by at most 2^-30 of it, so columns
// with more than a few much smaller ones are turned away (weight_digits).
// With 0/1 inputs each digit plane's product is an integer sum without
// rounding; the planes are joined and rounded once per output (twice past
// 2^10 column maxima).  So an output does not depend on the order, the tiles
// or the rows it is computed with, and lies within half an ulp of the digits'
// sum (8192 x 4096 currents of 1024 inputs at 10 % activity: 3.6e-8 of their
// 2-norm from float64, an fp32 GEMM 1.9e-7).
//
// Cost: four int8 planes at twice the bf16 rate against three bf16 planes,
// 2/3 of the matrix time, with one bit per input instead of two bytes.

#include "common.h"

namespace {

typedef int i32x4 __attribute__((ext_vector_type(4)));
typedef int i32x16 __attribute__((ext_vector_type(16)));
typedef float f4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) void lds_void;

constexpr int kPlanes = 4;   // base-256 digits per weight
constexpr int kStage = 128;  // k per LDS stage (bytes of a digit row)
constexpr int kSlack = 6;    // small weights a column may hold beyond their shares (see weight_digits)
constexpr int64_t kMaxK = 508 * 128;  // 128 K 257 < 2^31: two digit sums joined stay in 32 bits

inline int64_t cdiv(int64_t a, int64_t b) { return (a + b - 1) / b; }

// ---------------------------------------------------------------------------
// Operands.
// ---------------------------------------------------------------------------
__device__ __forceinline__ uint16_t to_bf16(float v) { return __builtin_bit_cast(uint16_t, static_cast<__bf16>(v)); }

// flags[0], flags[1] (as cast_spikes sets them) from 64 runs of 64 elements
// spread over x: real-valued inputs, nearly all of whose elements show it, are
// known before any pass over them.  (4,096 elements each on a page of its own
// took 7 to 12 us of address translation.)
__global__ __launch_bounds__(1024) void probe_spikes(const float *x, int64_t n, int *flags) {
  const int64_t step = n / 64 > 64 ? n / 64 : 64;
  float v[4];
#pragma unroll
  for (int u = 0; u < 4; ++u) {
    const int64_t i = (static_cast<int64_t>(threadIdx.x >> 6) * 4 + u) * step + (threadIdx.x & 63);
    v[u] = i < n ? x[i] : 0.0f;
  }
  bool inexact = false, other = false;
#pragma unroll
  for (int u = 0; u < 4; ++u) {
    inexact = inexact || !myelin::bf16_exact(v[u]);
    other = other || !(v[u] == 0.0f || v[u] == 1.0f);
  }
  const int any0 = __syncthreads_or(inexact), any1 = __syncthreads_or(other);
  if (threadIdx.x == 0) {
    flags[0] = any0 != 0;
    flags[1] = any1 != 0;
  }
}

struct CastArgs {
  const float *x;
  uint32_t *words;
  uint16_t *xb;
  int *flags;
  int64_t rows;
  int F, Kw;
};

// x [rows, F] fp32 -> words [Kw / 4][rows][4], bit i of word w of a row
// (stage w / 4) the element 32 w + i, zeros past F, and if xb is given xb
// [rows, F] bf16.  flags[0] is set where a value is not bf16-exact, flags[1] where one
// is neither 0 nor 1; neither is cleared.
// Bound by memory: each lane takes groups of four elements of a row, lane
// after lane, so every load and store instruction of a wave is contiguous;
// eight lanes' four bits are joined to a word by lane exchanges.
template <bool VEC>
__global__ __launch_bounds__(256) void cast_spikes(CastArgs p) {
  if (p.flags[0] != 0 || (p.flags[1] != 0 && p.xb == nullptr)) return;  // uniform: nothing here will be read
  constexpr int U = 4;  // groups per lane
  const uint32_t per = static_cast<uint32_t>(p.Kw) * 8;
  const int64_t total = p.rows * per;
  const int64_t g0 = static_cast<int64_t>(blockIdx.x) * (256 * U) + threadIdx.x;
  const int lane = threadIdx.x & 63;
  float v[U][4];
  int64_t row[U];
  int col[U];
#pragma unroll
  for (int u = 0; u < U; ++u) {
    const int64_t g = g0 + u * 256;
    row[u] = total <= 0x7fffffff ? static_cast<int64_t>(static_cast<uint32_t>(g) / per) : g / per;
    col[u] = static_cast<int>(g - row[u] * per) * 4;
#pragma unroll
    for (int e = 0; e < 4; ++e) v[u][e] = 0.0f;
    if (g < total && col[u] < p.F) {
      const float *src = p.x + row[u] * p.F + col[u];
      if constexpr (VEC) {  // F % 4 == 0 and 16-byte aligned rows
        const f4 t = __builtin_nontemporal_load(reinterpret_cast<const f4 *>(src));
#pragma unroll
        for (int e = 0; e < 4; ++e) v[u][e] = t[e];
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (col[u] + e < p.F) v[u][e] = src[e];
      }
    }
  }
  bool inexact = false, other = false;
#pragma unroll
  for (int u = 0; u < U; ++u) {
    const bool in = g0 + u * 256 < total;  // the same for a word's eight lanes
    uint32_t bits = 0;
    uint16_t h[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const float f = v[u][e];
      inexact = inexact || !myelin::bf16_exact(f);
      other = other || !(f == 0.0f || f == 1.0f);
      bits |= (f != 0.0f ? 1u : 0u) << e;
      h[e] = to_bf16(f);
    }
    bits <<= 4 * (lane & 7);
#pragma unroll
    for (int d = 1; d < 8; d <<= 1) bits |= static_cast<uint32_t>(__shfl_xor(static_cast<int>(bits), d));
    if (in && (lane & 7) == 0) p.words[((col[u] / 128) * p.rows + row[u]) * 4 + (col[u] / 32 & 3)] = bits;
    if (in && p.xb != nullptr && col[u] < p.F) {
      uint16_t *dst = p.xb + row[u] * p.F + col[u];
      if constexpr (VEC) {
        typedef uint16_t h4 __attribute__((ext_vector_type(4)));
        *reinterpret_cast<h4 *>(dst) = h4{h[0], h[1], h[2], h[3]};
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (col[u] + e < p.F) dst[e] = h[e];
      }
    }
  }
  const bool any0 = __ballot(inexact) != 0, any1 = __ballot(other) != 0;
  if (lane == 0) {
    if (any0) p.flags[0] = 1;
    if (any1) p.flags[1] = 1;
  }
}

// The k of byte p (0..15) of 16-byte piece c of a 128-k stage of a digit row:
// piece c is what lanes of half c & 1 multiply in k step c / 2, and their
// input bits are byte-wise masks of one word (see bits_fragment).
__device__ __forceinline__ int piece_k(int c, int p) {
  return 64 * (c >> 2) + 32 * (c & 1) + 8 * (p & 3) + 4 * ((c >> 1) & 1) + (p >> 2);
}

// w [F, N] -> digits [ceil(N / 32)][Kp / 128][4 planes][32 neurons][128] int8
// (zeros past F and N; the 128 k of a stage in the order of piece_k) and
// scale [N].  flags[1] is set where a column holds a non-finite value, its
// largest magnitude is outside [2^-96, 2^128), or its weights span too wide a
// range for one scale (below); nothing is done where it is set already.
//
// The range: a weight below 2^-7 of 2^e (the power of two above its column's
// largest) is rounded, by at most 2^-31 of 2^e.  An fp32 product's own error
// is about 2^-24 of the sum of the magnitudes that spike, so the digits are as
// good where most of those are above 2^-7 of 2^e -- whichever inputs spike,
// and also where the largest weights' inputs are silent.  So of the weights
// in a chunk of a column that the digits round, at most a quarter may be,
// a 16th be below 2^-10 and a 256th below 2^-14 of 2^e (and kSlack more, as
// chance has it: of 128 normal or Laplace weights 3 to 15, 1 to 2 and 0.1).
// One weight 100 times the rest of its column raised the error of its currents
// from 1.2e-7, fp32's, to 7.7e-7 without this, 10^6 times to 6e-3.
// A workgroup writes `chunk` k of 32 neurons: it first finds the columns'
// maxima over all F (re-read from L2 by each of a column's workgroups: one
// launch instead of a reduction and a second pass), then turns tiles of 128
// k around through LDS so that rows are written 16 bytes at a time.
__global__ __launch_bounds__(1024) void weight_digits(const float *__restrict__ w, int8_t *__restrict__ q,
                                                      float *__restrict__ scale, int *__restrict__ flags, int F, int N,
                                                      int Kp, int chunk) {
  __shared__ int skip;  // one answer for the workgroup: others may set the flag meanwhile
  if (threadIdx.x == 0) skip = flags[1];
  __syncthreads();
  if (skip != 0) return;
  __shared__ uint32_t red[32][33];
  __shared__ uint64_t small[32][33];
  __shared__ int tile[32][kStage + 1];
  const int c = threadIdx.x & 31, r = threadIdx.x >> 5;
  const int64_t n = static_cast<int64_t>(blockIdx.x) * 32 + c;
  const bool in = n < N;
  uint32_t mx = 0;
  if (in) {
    // four rows in flight
    int f = r;
    for (; f + 96 < F; f += 128) {
      uint32_t b[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) b[u] = __builtin_bit_cast(uint32_t, w[static_cast<int64_t>(f + 32 * u) * N + n]) & 0x7fffffffu;
#pragma unroll
      for (int u = 0; u < 4; ++u) mx = mx > b[u] ? mx : b[u];
    }
    for (; f < F; f += 32) {
      const uint32_t b = __builtin_bit_cast(uint32_t, w[static_cast<int64_t>(f) * N + n]) & 0x7fffffffu;
      mx = mx > b ? mx : b;
    }
  }
  red[r][c] = mx;
  __syncthreads();
  mx = 0;
#pragma unroll 8
  for (int i = 0; i < 32; ++i) mx = mx > red[i][c] ? mx : red[i][c];
  // every value is below 2^e; a zero column has digits 0 and scale 0
  const int e = static_cast<int>(mx >> 23) - 126;
  const bool bad = mx >= 0x7f800000u || (mx != 0 && e < -96);
  const float up = (mx == 0 || bad) ? 0.0f : __builtin_bit_cast(float, static_cast<uint32_t>(30 - e + 127) << 23);
  if (blockIdx.y == 0 && r == 0 && in) {
    scale[n] = (mx == 0 || bad) ? 0.0f : __builtin_bit_cast(float, static_cast<uint32_t>(e - 30 + 127) << 23);
    if (bad) flags[1] = 1;
  }
  const int k_begin = blockIdx.y * chunk, k_end = k_begin + chunk < Kp ? k_begin + chunk : Kp;
  uint64_t count = 0;  // of the column's weights in this chunk: three sums of 21 bits
  for (int k0 = k_begin; k0 < k_end; k0 += kStage) {
#pragma unroll
    for (int u = 0; u < kStage / 32; ++u) {
      const int f = k0 + r + 32 * u;
      const float v = (in && f < F) ? w[static_cast<int64_t>(f) * N + n] : 0.0f;
      // |w| up is at most 2^30 and a power of two times w: exact but for the
      // integer rounding of magnitudes under 2^23
      const float scaled = v * up, q_f = __builtin_rintf(scaled), mag = __builtin_fabsf(scaled);
      tile[c][r + 32 * u] = static_cast<int>(q_f);
      if (v != 0.0f && (scaled != q_f || q_f == 0.0f)) {
        count += 1;
        if (mag < 1048576.0f) count += uint64_t{1} << 21;
        if (mag < 65536.0f) count += uint64_t{1} << 42;
      }
    }
    __syncthreads();
    // thread -> plane, neuron, piece of 16 k
    const int pl = threadIdx.x >> 8, nn = (threadIdx.x >> 3) & 31, c16 = threadIdx.x & 7;
    uint32_t out[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      uint32_t word = 0;
#pragma unroll
      for (int b = 0; b < 4; ++b) {
        int v = tile[nn][piece_k(c16, 4 * i + b)], d = 0;
        for (int s = 0; s <= pl; ++s) {  // balanced digit pl
          d = static_cast<int8_t>(v & 0xff);
          v = (v - d) >> 8;
        }
        word |= static_cast<uint32_t>(static_cast<uint8_t>(d)) << (8 * b);
      }
      out[i] = word;
    }
    typedef uint32_t u4 __attribute__((ext_vector_type(4)));
    *reinterpret_cast<u4 *>(q + static_cast<int64_t>(blockIdx.x) * 128 * Kp + static_cast<int64_t>(k0) * 128 +
                            (pl * 32 + nn) * kStage + 16 * c16) =
        u4{out[0], out[1], out[2], out[3]};
    __syncthreads();
  }
  small[r][c] = count;
  __syncthreads();
  if (r == 0 && in && up != 0.0f) {
    uint64_t sum = 0;
#pragma unroll 8
    for (int i = 0; i < 32; ++i) sum += small[i][c];
    const int weights = (k_end < F ? k_end : F) - k_begin, mask = (1 << 21) - 1;
    const int rounded = static_cast<int>(sum) & mask, below10 = static_cast<int>(sum >> 21) & mask,
              below14 = static_cast<int>(sum >> 42);
    if (rounded > weights / 4 + kSlack || below10 > weights / 16 + kSlack || below14 > weights / 256 + kSlack) flags[1] = 1;
  }
}

// ---------------------------------------------------------------------------
// C[M, N] = (bits x digits) joined, scaled (+ bias).
//
// The four digit planes of 32 neurons are 128 "virtual" columns that one
// wave owns: its tile is 32 WM rows x 128 virtual columns, WM x 4 blocks of
// 32 x 32 (v_mfma_i32_32x32x32_i8: a lane's fragment is 16 bytes of k, as in
// the bf16 kernels), so an input fragment feeds four MFMAs and the planes of
// an output element end in the same lane and register index: they are joined
// without a second accumulator set.  WGM x WGN waves share a stage of 128 k
// of their rows and virtual columns, staged by direct global -> LDS loads of
// 16 bytes (digit rows unpadded, 16-byte pieces at position c ^ swz(row); a
// row's 128 input bits are one piece).
//
// Measured at 8192 x 4096 x 1024 (MFMA time at peak 55 us), with parts
// switched off: 75 us without loads and stores, 53 without MFMAs and stores,
// and the stores about 30, which added up instead of overlapping.  What
// helped:
// - Two workgroups per CU (256 rows x 32 neurons each, four waves) instead of
//   one of eight waves: one's stores and stage waits under the other's
//   MFMAs, 160 -> 142 us.
// - Inputs as bits, 20 KB a stage and workgroup, widened in registers: a lane
//   of half h takes one word for two k steps, and dword j of its fragment in
//   step s is (word >> (4 s + j)) & 0x01010101, two operations for four k;
//   the digits are stored in that order of k.  With byte inputs the smaller
//   tiles cost more (176 us) than they hid.
// - Operands stored stage by stage, so that a tile's stage is contiguous: at
//   a row pitch of 1,024 bytes a stage's pieces meet a quarter of the L2
//   channels.  142 -> 137 us.
// - No scheduling hints between MFMAs and LDS reads (with them 137, without
//   132 us): the other workgroup fills the waits.
//
// Persistent: each workgroup walks tiles, and the first NS - 1 stages of its
// next tile are loaded during the last stages of this one, before the
// epilogue's stores: K is short here (1024 inputs are eight stages), and the
// vector memory counter retires in order, so loads behind the stores would
// wait for them.
// ---------------------------------------------------------------------------
struct SpikeArgs {
  const uint32_t *x;  // [Kp / 128][x_rows][4] words, M rows of each stage
  const int8_t *q;    // digits
  const float *scale, *bias;
  const int *flags;  // or null: return at once where one of the two is set
  float *C;
  int64_t M, N, ldc, x_rows;
  int Kp;
};

// position of 16-byte piece c of digit row r of a stage: c ^ swz(r).  A
// function of r & 31, so the 32-row blocks of a wave share it, distinct over
// any 8 aligned rows and, with the row's bank half, over any 16: fragment
// reads (32 rows of one piece per half-wave) meet no bank conflict
__device__ __forceinline__ int swz(int r) { return (r ^ ((r >> 3) & 3)) & 7; }

__device__ __forceinline__ int acc_row(int r, int lane) { return 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3); }

// The fragment of k step s (0 or 1) of the two that a word covers.
__device__ __forceinline__ i32x4 bits_fragment(uint32_t word, int s) {
  i32x4 f;
#pragma unroll
  for (int j = 0; j < 4; ++j) f[j] = static_cast<int>((word >> (4 * s + j)) & 0x01010101u);
  return f;
}

template <int WM, int WGM, int WGN, int NS>
__global__ __launch_bounds__(64 * WGM * WGN) __attribute__((amdgpu_waves_per_eu(2))) void spike_gemm(SpikeArgs g) {
  constexpr int NT = 64 * WGM * WGN;
  constexpr int BM = 32 * WM * WGM, BV = 128 * WGN;
  constexpr int TA = BM * 16, TILE = TA + BV * kStage;  // bytes of a stage's bits, of a stage
  constexpr int NPB = BV * 8 / NT;                      // digit pieces per thread
  constexpr int WA = BM / 64;                           // waves that load the bits, one piece a lane
  static_assert(WA <= NT / 64, "one piece of bits per lane at most");
  __shared__ __attribute__((aligned(1024))) char lds[NS * TILE];
  if (g.flags != nullptr && (g.flags[0] | g.flags[1]) != 0) return;  // uniform: no launch beside this one writes them
  const int tid = threadIdx.x, lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6), wm = w / WGN, wn = w % WGN;
  const uint32_t tiles_m = static_cast<uint32_t>((g.M + BM - 1) / BM);
  const uint32_t tiles_n = static_cast<uint32_t>((g.N + 32 * WGN - 1) / (32 * WGN));
  const uint32_t tiles = tiles_m * tiles_n;
  // Workgroup ids go round-robin to the 8 XCDs (each with its own L2): XCD d
  // walks a contiguous run of logical tiles, its workgroups side by side.
  const uint32_t xcds = gridDim.x % 8 == 0 ? 8 : 1;
  const uint32_t xcd = blockIdx.x % xcds, slot = blockIdx.x / xcds, slots = gridDim.x / xcds;
  const uint32_t first = static_cast<uint32_t>(static_cast<uint64_t>(tiles) * xcd / xcds);
  const uint32_t last = static_cast<uint32_t>(static_cast<uint64_t>(tiles) * (xcd + 1) / xcds);
  const int64_t vrows = (g.N + 31) / 32 * 128;  // virtual columns stored
  const int nst = g.Kp / kStage;

  // logical tile -> (row tile, column tile): groups of 8 row tiles walked
  // column by column, so a run shares input rows and digit rows
  auto place = [&](uint32_t t, int64_t &m0, int64_t &n0) {
    const uint32_t per_group = 8 * tiles_n, group = t / per_group, fst = group * 8;
    const uint32_t gs = tiles_m - fst < 8 ? tiles_m - fst : 8, in = t - group * per_group;
    m0 = static_cast<int64_t>(__builtin_amdgcn_readfirstlane(fst + in % gs)) * BM;
    n0 = static_cast<int64_t>(__builtin_amdgcn_readfirstlane(in / gs)) * (32 * WGN);
  };
  auto load16 = [](uint32_t off, const void *base, const char *dst_lds) {
    const uint32_t dst = static_cast<uint32_t>(reinterpret_cast<uintptr_t>((lds_void *)dst_lds));
    uint32_t m0_saved;  // M0 (the LDS base of the load) is the compiler's
    asm volatile(
        "s_mov_b32 %0, m0\n\ts_mov_b32 m0, %3\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2\n\ts_mov_b32 m0, %0"
        : "=&s"(m0_saved)
        : "v"(off), "s"(base), "s"(dst)
        : "memory");
  };

  // load side: pieces of the tile being loaded, as 32-bit offsets from a
  // uniform base; rows past the edge read the last row
  uint32_t oa = 0, ob[NPB];
  const char *ba = nullptr, *bb = nullptr;
  uint32_t lt = first + slot;
  int ls = 0, lbuf = 0, ahead = 0;  // next stage to load, its buffer; stages loaded or in flight, not yet used
  auto point = [&]() {
    int64_t m0, n0;
    place(lt, m0, n0);
    ba = reinterpret_cast<const char *>(g.x) + m0 * 16;
    bb = reinterpret_cast<const char *>(g.q) + n0 * kPlanes * g.Kp;
    const int64_t lim_a = g.M - m0, lim_b = vrows - n0 * kPlanes;
    oa = static_cast<uint32_t>(tid < lim_a ? tid : lim_a - 1) * 16u;
#pragma unroll
    for (int e = 0; e < NPB; ++e) {
      const int idx = e * NT + tid, row = idx >> 3;
      const uint32_t gi = row < lim_b ? static_cast<uint32_t>(row) >> 7 : 0u;
      ob[e] = gi * 128u * static_cast<uint32_t>(g.Kp) + (static_cast<uint32_t>(row) & 127u) * kStage + 16 * ((idx & 7) ^ swz(row));
    }
  };
  auto issue = [&]() {
    if (lt >= last) return;  // uniform
    if (ls == 0) point();
    const char *tile = lds + lbuf * TILE;
    if (w < WA) load16(oa, ba + static_cast<int64_t>(ls) * g.x_rows * 16, tile + w * 1024);
#pragma unroll
    for (int e = 0; e < NPB; ++e) load16(ob[e], bb + ls * 128 * kStage, tile + TA + (e * NT + w * 64) * 16);
    lbuf = lbuf == NS - 1 ? 0 : lbuf + 1;
    ++ahead;
    if (++ls == nst) {
      ls = 0;
      lt += slots;
    }
  };

  // byte offsets in a stage: the lane's word of its row's four (the word of
  // k steps 2, 3 lies 8 bytes on), and its digit fragments (32-row blocks lie
  // 32 rows apart)
  const int fa = (32 * WM * wm + (lane & 31)) * 16 + 4 * (lane >> 5);
  int fb[4];
#pragma unroll
  for (int ks = 0; ks < 4; ++ks) {
    const int c = 2 * ks + (lane >> 5), r = lane & 31;
    fb[ks] = TA + (128 * wn + r) * kStage + ((c ^ swz(r)) << 4);
  }

#pragma unroll
  for (int i = 0; i < NS - 1; ++i) issue();
  int buf = 0, landed = 0;  // the stage's buffer; stages known to have landed
  for (uint32_t t = first + slot; t < last; t += slots) {
    i32x16 acc[WM][kPlanes];
#pragma unroll
    for (int i = 0; i < WM; ++i)
#pragma unroll
      for (int j = 0; j < kPlanes; ++j)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[i][j][r] = 0;
    for (int s = 0; s < nst; ++s) {
      // this stage's loads: all but the NS - 2 later stages' in flight, or
      // all at the end, or none where the epilogue before has waited.  The
      // barrier makes every wave's pieces visible, and retires the LDS reads
      // of the buffer that the loads issued after it overwrite.
      if (landed > 0)
        --landed;
      else if (ahead < NS - 1)
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      else if (w < WA)
        asm volatile("s_waitcnt vmcnt(%0)" ::"n"((NPB + 1) * (NS - 2)) : "memory");
      else
        asm volatile("s_waitcnt vmcnt(%0)" ::"n"(NPB * (NS - 2)) : "memory");
      asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
      const char *cur = lds + buf * TILE;
      uint32_t bits[2][WM];
      i32x4 b[2][kPlanes];
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int i = 0; i < WM; ++i) bits[h][i] = *reinterpret_cast<const uint32_t *>(cur + fa + 512 * i + 8 * h);
      auto rd = [&](int ks, int set) {
#pragma unroll
        for (int j = 0; j < kPlanes; ++j)
          b[set][j] = *reinterpret_cast<const i32x4 *>(cur + fb[ks] + 32 * kStage * j);
      };
      i32x4 a[2][WM];
      auto widen = [&](int ks, int set) {
#pragma unroll
        for (int i = 0; i < WM; ++i) a[set][i] = bits_fragment(bits[ks >> 1][i], ks & 1);
      };
      rd(0, 0);
      --ahead;
      issue();
      widen(0, 0);
#pragma unroll
      for (int ks = 0; ks < 4; ++ks) {
        if (ks + 1 < 4) {
          rd(ks + 1, (ks + 1) & 1);
          widen(ks + 1, (ks + 1) & 1);
        }
#pragma unroll
        for (int i = 0; i < WM; ++i)
#pragma unroll
          for (int j = 0; j < kPlanes; ++j)
            acc[i][j] = __builtin_amdgcn_mfma_i32_32x32x32_i8(a[ks & 1][i], b[ks & 1][j], acc[i][j], 0, 0, 0);
      }
      buf = buf == NS - 1 ? 0 : buf + 1;
    }
    // the next tile's first stages land before this tile's stores are issued
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    landed = ahead;
    int64_t m0, n0;
    place(t, m0, n0);
    const int64_t n = n0 + 32 * wn + (lane & 31);
    if (n < g.N) {
      const float sc = g.scale[n], bi = g.bias != nullptr ? g.bias[n] : 0.0f;
      const int64_t mw = m0 + 32 * WM * wm;
      const bool whole = mw + 32 * WM <= g.M;  // uniform
      // the lane's column and row half, from each row's scalar base
      const uint32_t off = static_cast<uint32_t>((4 * (lane >> 5) * g.ldc + 32 * wn + (lane & 31)) * 4);
#pragma unroll
      for (int i = 0; i < WM; ++i)
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          // the sum is hi 2^16 + lo, both exact in 32 bits; with all but the
          // low 16 bits of lo carried over lo is exact in fp32, and hi while
          // the sum is under 2^10 column maxima
          int lo = (acc[i][1][r] << 8) + acc[i][0][r];
          int hi = (acc[i][3][r] << 8) + acc[i][2][r];
          const int carry = (lo + 0x8000) >> 16;
          hi += carry;
          lo -= carry << 16;
          float v = __builtin_fmaf(static_cast<float>(hi), 65536.0f, static_cast<float>(lo)) * sc;
          if (g.bias != nullptr) v = v + bi;
          const float *base = g.C + (mw + 32 * i + acc_row(r, 0)) * g.ldc + n0;
          if (whole || mw + 32 * i + acc_row(r, lane) < g.M)
            asm volatile("global_store_dword %0, %1, %2" ::"v"(off), "v"(v), "s"(base) : "memory");
        }
    }
  }
}

template <int WM, int WGM, int WGN, int NS>
int launch_spike(const SpikeArgs &g, int per_cu, hipStream_t s) {
  const int64_t tiles = cdiv(g.M, 32 * WM * WGM) * cdiv(g.N, 32 * WGN);
  const int64_t wgs = tiles < 256 * per_cu ? tiles : 256 * per_cu;
  spike_gemm<WM, WGM, WGN, NS><<<dim3(static_cast<unsigned>(wgs)), dim3(64 * WGM * WGN), 0, s>>>(g);
  return myelin::launched("gemm_spikes");
}

}  // namespace

extern "C" int myelin_probe_spikes(const float *x, int64_t n, int *flags, myelin_stream_t stream) {
  if (n < 0) return myelin::invalid("probe_spikes: negative size");
  if (flags == nullptr || (n > 0 && x == nullptr)) return myelin::invalid("probe_spikes: null pointer");
  probe_spikes<<<dim3(1), dim3(1024), 0, myelin::as_hip(stream)>>>(x, n, flags);
  return myelin::launched("probe_spikes");
}

extern "C" int myelin_cast_spikes(const float *x, int32_t *words, uint16_t *xb, int64_t rows, int64_t F, int64_t Kw,
                                  int *flags, myelin_stream_t stream) {
  if (rows < 0 || F < 1) return myelin::invalid("cast_spikes: rows must be >= 0 and F >= 1");
  if (F > kMaxK || Kw % 4 != 0 || Kw * 32 < F || Kw * 32 > kMaxK) return myelin::invalid("cast_spikes: bad row pitch");
  if (rows == 0) return MYELIN_OK;
  if (x == nullptr || words == nullptr || flags == nullptr) return myelin::invalid("cast_spikes: null pointer");
  if (!myelin::aligned(words, 16)) return myelin::invalid("cast_spikes: words must be 16-byte aligned");
  const int64_t blocks = cdiv(rows * Kw * 8, 1024);
  if (blocks > 0x7fffffff) return myelin::invalid("cast_spikes: too many elements");
  const CastArgs a{x, reinterpret_cast<uint32_t *>(words), xb, flags, rows, static_cast<int>(F), static_cast<int>(Kw)};
  const dim3 grid(static_cast<unsigned>(blocks));
  if (F % 4 == 0 && myelin::aligned(x, 16) && (xb == nullptr || myelin::aligned(xb, 8)))
    cast_spikes<true><<<grid, dim3(256), 0, myelin::as_hip(stream)>>>(a);
  else
    cast_spikes<false><<<grid, dim3(256), 0, myelin::as_hip(stream)>>>(a);
  return myelin::launched("cast_spikes");
}

extern "C" int myelin_weight_digits(const float *w, int8_t *digits, float *scale, int64_t F, int64_t N, int64_t Kp,
                                    int *flags, myelin_stream_t stream) {
  if (F < 1 || N < 1) return myelin::invalid("weight_digits: F and N must be positive");
  if (Kp % kStage != 0 || Kp < F || Kp > kMaxK) return myelin::invalid("weight_digits: bad row pitch");
  if (w == nullptr || digits == nullptr || scale == nullptr || flags == nullptr)
    return myelin::invalid("weight_digits: null pointer");
  if (!myelin::aligned(digits, 16)) return myelin::invalid("weight_digits: digits must be 16-byte aligned");
  const int64_t groups = cdiv(N, 32), stages = Kp / kStage;
  if (N > 0x7fffffff || groups > 0x7fffffff) return myelin::invalid("weight_digits: N too large");
  // about 512 workgroups: each of a column's re-reads it once
  int64_t parts = cdiv(512, groups);
  if (parts > stages) parts = stages;
  const int64_t chunk = cdiv(stages, parts) * kStage;
  weight_digits<<<dim3(static_cast<unsigned>(groups), static_cast<unsigned>(cdiv(Kp, chunk))), dim3(1024), 0,
                  myelin::as_hip(stream)>>>(w, digits, scale, flags, static_cast<int>(F), static_cast<int>(N),
                                            static_cast<int>(Kp), static_cast<int>(chunk));
  return myelin::launched("weight_digits");
}

namespace {

int gemm_spikes_impl(const int32_t *words, int64_t x_rows, const int8_t *digits, const float *scale, const float *bias,
                     const int *flags, float *C, int64_t M, int64_t N, int64_t Kp, int64_t ldc, hipStream_t s) {
  if (M < 0 || N < 0) return myelin::invalid("gemm_spikes: negative size");
  if (x_rows < M) return myelin::invalid("gemm_spikes: x_rows < M");
  if (Kp < kStage || Kp % kStage != 0 || Kp > kMaxK) return myelin::invalid("gemm_spikes: bad row pitch");
  if (ldc < N) return myelin::invalid("gemm_spikes: ldc < N");
  if (M == 0 || N == 0) return MYELIN_OK;
  if (words == nullptr || digits == nullptr || scale == nullptr || C == nullptr)
    return myelin::invalid("gemm_spikes: null pointer");
  if (!myelin::aligned(words, 16) || !myelin::aligned(digits, 16))
    return myelin::invalid("gemm_spikes: operands must be 16-byte aligned");
  if (ldc >= (int64_t{1} << 27)) return myelin::invalid("gemm_spikes: rows too long");
  if (cdiv(M, 128) * cdiv(N, 32) > 0x7fffffff) return myelin::invalid("gemm_spikes: output too large");
  const SpikeArgs g{reinterpret_cast<const uint32_t *>(words), digits, scale, bias, flags, C, M, N, ldc, x_rows,
                    static_cast<int>(Kp)};
  // 256 rows x 32 neurons, two workgroups per CU, where that fills the chip;
  // else 128 rows (3200 x 256 x 784, 200 of them: 8.8 us)
  if (cdiv(M, 256) * cdiv(N, 32) >= 512) return launch_spike<2, 4, 1, 3>(g, 2, s);
  return launch_spike<1, 4, 1, 4>(g, 2, s);
}

}  // namespace

extern "C" int myelin_gemm_spikes(const int32_t *words, int64_t x_rows, const int8_t *digits, const float *scale,
                                  const float *bias, float *C, int64_t M, int64_t N, int64_t Kp, int64_t ldc,
                                  myelin_stream_t stream) {
  return gemm_spikes_impl(words, x_rows, digits, scale, bias, nullptr, C, M, N, Kp, ldc, myelin::as_hip(stream));
}

extern "C" int myelin_gemm_spikes_if(const int *flags, const int32_t *words, int64_t x_rows, const int8_t *digits,
                                     const float *scale, const float *bias, float *C, int64_t M, int64_t N, int64_t Kp,
                                     int64_t ldc, myelin_stream_t stream) {
  if (flags == nullptr) return myelin::invalid("gemm_spikes_if: null pointer");
  return gemm_spikes_impl(words, x_rows, digits, scale, bias, flags, C, M, N, Kp, ldc, myelin::as_hip(stream));
}
