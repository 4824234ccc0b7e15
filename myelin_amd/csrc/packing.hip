// Spike bitpacking for gfx950: 32 spikes per int32 word along the last
// dimension, bit i of word w = element 32*w + i (LSB first), padding bits 0.
//
// pack:   elements of 4 and 8 bytes: one lane per element; a wave ballot
//         turns 64 consecutive elements into two words.  Each wave handles
//         64 words (32 ballots) per pass and lane j stores word j, so the
//         word store is one coalesced 256-byte write and every element load
//         is a coalesced wave load.  Elements of 1 and 2 bytes: one lane per
//         word, which reads its 32 elements as whole dwords.
// unpack: one lane per 16 bytes of output.
// counts: popcount with the padding bits of the last word masked.

#include "common.h"

namespace {

using myelin::kWave;

// ---- element predicates: "nonzero" exactly as ATen's (x != 0) ----------
struct F32 {
  using T = float;
  __device__ static bool nz(float v) { return v != 0.0f; }
};
struct F64 {
  using T = double;
  __device__ static bool nz(double v) { return v != 0.0; }
};
struct H16 {  // fp16 and bf16: zero iff all bits but the sign are zero (nonzero_bits)
  using T = uint16_t;
};
struct U8 {
  using T = uint8_t;
};
struct I32 {
  using T = int32_t;
  __device__ static bool nz(int32_t v) { return v != 0; }
};
struct I64 {
  using T = int64_t;
  __device__ static bool nz(int64_t v) { return v != 0; }
};

// words: [rows, W]; total = rows * W.  ALIGNED: n % 32 == 0 so the element
// of (word g, bit i) is simply 32*g + i; else a lane's row and column are
// found by one division and then advanced two words at a time (a 64-bit
// division per word: 15000 rows of 2312 floats 44.6 -> 22.3 us).
template <class E, bool ALIGNED>
__global__ __launch_bounds__(256) void pack_kernel(const typename E::T *__restrict__ src, int32_t *__restrict__ words,
                                                   int64_t total, int64_t W, int64_t n) {
  const int lane = static_cast<int>(threadIdx.x & (kWave - 1));
  const int64_t wave = (static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x) >> 6;
  const int64_t g0 = wave * 64;  // first word of this wave
  if (g0 >= total) return;       // wave-uniform
  const int half = lane >> 5, bit = lane & 31;

  typename E::T v[32];
  if constexpr (ALIGNED) {
#pragma unroll
    for (int i = 0; i < 32; ++i) {
      const int64_t g = g0 + 2 * i + half;
      v[i] = typename E::T(0);
      if (g < total) v[i] = __builtin_nontemporal_load(src + g * 32 + bit);
    }
  } else {
    int64_t r = (g0 + half) / W;
    int64_t col = (g0 + half - r * W) * 32 + bit;
    const typename E::T *p = src + r * n + col;
    const int64_t wide = W * 32, pad = wide - n;
#pragma unroll
    for (int i = 0; i < 32; ++i) {
      v[i] = typename E::T(0);
      if (g0 + 2 * i + half < total && col < n) {
        // (streamed 8-byte loads of unaligned rows measured slower: 30000 x
        // 1000 doubles 56 -> 65 us)
        if constexpr (sizeof(typename E::T) == 8)
          v[i] = *p;
        else
          v[i] = __builtin_nontemporal_load(p);
      }
      // two words on: past the row's last word, `pad` elements fewer per row
      col += 64;
      p += 64;
      if (col >= wide) {
        col -= wide;
        p -= pad;
        if (col >= wide) {  // rows of one word
          col -= wide;
          p -= pad;
        }
      }
    }
  }
  uint32_t mine = 0;
#pragma unroll
  for (int i = 0; i < 32; ++i) {
    const uint64_t b = __ballot(E::nz(v[i]));
    const uint32_t lo = static_cast<uint32_t>(b), hi = static_cast<uint32_t>(b >> 32);
    mine = (lane == 2 * i) ? lo : mine;
    mine = (lane == 2 * i + 1) ? hi : mine;
  }
  if (g0 + lane < total) words[g0 + lane] = static_cast<int32_t>(mine);
}

// The bits of the nonzero elements in a dword of four bytes or of two
// halves (zero but for the sign), the first element in bit 0.
template <int SIZE>
__device__ __forceinline__ uint32_t nonzero_bits(uint32_t d) {
  if constexpr (SIZE == 1) {
    // bit 7 of each byte: some bit of it is set; then the four gathered into
    // the top nibble by one multiplication (no two products share a bit)
    const uint32_t t = ((d & 0x7f7f7f7fu) + 0x7f7f7f7fu) | d;
    return (((t >> 7) & 0x01010101u) * 0x10204080u) >> 28;
  } else {
    const uint32_t t = (d & 0x7fff7fffu) + 0x7fff7fffu;  // bit 15 / 31: magnitude not zero
    return ((t >> 15) & 1u) | ((t >> 30) & 2u);
  }
}

// One lane per word, elements of SIZE (1 or 2) bytes: the lane's 32 elements
// are 8 SIZE dwords.  Rows that start on multiples of G = 16 or 8 bytes are
// read G bytes at a time; others (G = 4) as the whole dwords that hold the
// elements (one more where the row is not dword-aligned), shifted into
// place.  A piece past the last element's is never read.  (Byte elements
// used to take one load instruction per 64 bytes of a wave and a 64-bit
// division per word: 15000 rows of 2312 bytes, G = 8, 44.8 -> 6.4 us (6.1
// TB/s); of 2311, G = 4, 44.6 -> 18.3 us; 8192 bf16, G = 16, 289 -> 111 us
// for 32768 rows.)
template <int SIZE, int G>
__global__ __launch_bounds__(256) void pack_words(const uint8_t *__restrict__ src, int32_t *__restrict__ words,
                                                  int64_t total, int64_t W, int64_t n) {
  typedef uint32_t vec __attribute__((ext_vector_type(G / 4)));
  constexpr int ND = 8 * SIZE, NV = 4 * ND / G + (G == 4 ? 1 : 0);  // dwords of a word, pieces read
  const int64_t g = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (g >= total) return;
  int64_t r;
  if (total <= 0x7fffffff)  // 32-bit division
    r = static_cast<uint32_t>(g) / static_cast<uint32_t>(W);
  else
    r = g / W;
  const int64_t col = (g - r * W) * 32;
  const int64_t left = n - col;  // elements of this word, if under 32
  const uintptr_t first = reinterpret_cast<uintptr_t>(src) + static_cast<uintptr_t>((r * n + col) * SIZE);
  const uintptr_t last = first + static_cast<uintptr_t>((left < 32 ? left : 32) * SIZE - 1);
  const vec *p = reinterpret_cast<const vec *>(first & ~uintptr_t{G - 1});
  const int lim = static_cast<int>(last / G - first / G);  // pieces past the first that hold elements
  vec v[NV];
#pragma unroll
  for (int i = 0; i < NV; ++i) v[i] = p[i < lim ? i : lim];
  uint32_t word = 0;
#pragma unroll
  for (int i = 0; i < ND; ++i) {
    uint32_t d;
    if constexpr (G == 4) {
      const uint32_t sh = static_cast<uint32_t>(first & 3) * 8;
      d = static_cast<uint32_t>(((static_cast<uint64_t>(v[i + 1][0]) << 32) | v[i][0]) >> sh);
    } else {
      d = v[i / (G / 4)][i % (G / 4)];
    }
    word |= nonzero_bits<SIZE>(d) << (4 / SIZE * i);
  }
  if (left < 32) word &= (1u << left) - 1u;
  words[g] = static_cast<int32_t>(word);
}

// The `count` (<= 16) bits from column `col` of a row of words on, reading
// only words that hold some of them.
__device__ __forceinline__ uint32_t row_bits(const int32_t *__restrict__ row, int64_t col, int count) {
  const uint32_t s = static_cast<uint32_t>(col & 31);
  const uint32_t *w = reinterpret_cast<const uint32_t *>(row) + (col >> 5);
  uint32_t b = w[0] >> s;
  if (s + count > 32) b |= w[1] << (32 - s);
  return b & ((1u << count) - 1u);
}

// One lane per 16 bytes (PER elements) of the flat output, one vector store.
// ALIGNED (n % 32 == 0): the elements share a word.  Otherwise a lane finds
// its row by one division, and where its elements run past the row's end
// continues with the next row's; the last elements of an output that is no
// multiple of 16 bytes are stored one by one.  (A division and a store per
// byte took 51.8 us on 15000 rows of 2312 bytes, this 6.7; on aligned rows a
// byte's own stores 106 -> 41 us for 32768 x 8192.)
template <typename S, bool ALIGNED>
__global__ __launch_bounds__(256) void unpack_kernel(const int32_t *__restrict__ words, S *__restrict__ dst,
                                                     int64_t total, int64_t n, int64_t W, S one) {
  constexpr int PER = 16 / sizeof(S);
  const int64_t e = (static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x) * PER;
  if (e >= total) return;
  const int m = total - e < PER ? static_cast<int>(total - e) : PER;  // elements of this lane
  uint32_t bits;
  if constexpr (ALIGNED) {
    bits = static_cast<uint32_t>(words[e >> 5]) >> (e & 31);
  } else {
    int64_t r;
    if (total <= 0x7fffffff && n <= 0x7fffffff)
      r = static_cast<uint32_t>(e) / static_cast<uint32_t>(n);
    else
      r = e / n;
    int64_t col = e - r * n;
    const int32_t *row = words + r * W;
    int got = n - col < m ? static_cast<int>(n - col) : m;
    bits = row_bits(row, col, got);
    while (got < m) {  // the next row, or rows narrower than the lane
      row += W;
      const int take = n < m - got ? static_cast<int>(n) : m - got;
      bits |= row_bits(row, 0, take) << got;
      got += take;
    }
  }
  typedef uint32_t u4 __attribute__((ext_vector_type(4)));
  u4 out;
  if constexpr (sizeof(S) == 1) {
    // bit i of a nibble to byte i
#pragma unroll
    for (int i = 0; i < 4; ++i) out[i] = ((((bits >> (4 * i)) & 0xfu) * 0x00204081u) & 0x01010101u) * one;
  } else if constexpr (sizeof(S) == 2) {
#pragma unroll
    for (int i = 0; i < 4; ++i)
      out[i] = ((bits >> (2 * i)) & 1u) * one + (((bits >> (2 * i + 1)) & 1u) * (static_cast<uint32_t>(one) << 16));
  } else if constexpr (sizeof(S) == 4) {
#pragma unroll
    for (int i = 0; i < 4; ++i) out[i] = ((bits >> i) & 1u) ? one : 0u;
  } else {
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const uint64_t v = ((bits >> i) & 1u) ? one : S(0);
      out[2 * i] = static_cast<uint32_t>(v);
      out[2 * i + 1] = static_cast<uint32_t>(v >> 32);
    }
  }
  if (m == PER) {
    __builtin_nontemporal_store(out, reinterpret_cast<u4 *>(dst + e));
  } else {
    for (int i = 0; i < m; ++i) dst[e + i] = ((bits >> i) & 1u) ? one : S(0);
  }
}

// outputs that do not start on 16 bytes
template <typename S>
__global__ __launch_bounds__(256) void unpack_generic(const int32_t *__restrict__ words, S *__restrict__ dst,
                                                      int64_t total, int64_t n, int64_t W, S one) {
  const int64_t e = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (e >= total) return;
  const int64_t r = e / n;
  const int64_t col = e - r * n;
  const uint32_t w = static_cast<uint32_t>(words[r * W + (col >> 5)]);
  dst[e] = ((w >> (col & 31)) & 1u) ? one : S(0);
}

// ---- counts --------------------------------------------------------------
inline int64_t cdiv64(int64_t a, int64_t b) { return (a + b - 1) / b; }

struct LeadInfo {
  int ndim;
  int64_t shape[8];
  int64_t out_stride[8];  // 0 for reduced dims
};

__device__ __forceinline__ int64_t out_index(int64_t row, const LeadInfo &li) {
  int64_t idx = 0;
  for (int d = li.ndim - 1; d >= 0; --d) {
    const int64_t s = li.shape[d];
    const int64_t q = row / s;
    idx += (row - q * s) * li.out_stride[d];
    row = q;
  }
  return idx;
}

// a finished count as the kernel's output: itself, or the rate count / denom
template <typename OUT>
__device__ __forceinline__ OUT finish(int64_t c, OUT denom) {
  if constexpr (sizeof(OUT) == 8 && OUT(0.5) == OUT(0))
    return c;
  else
    return static_cast<OUT>(c) / denom;
}

__device__ __forceinline__ int64_t wave_sum(int64_t v) {
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1) v += __shfl_xor(v, off);
  return v;
}

// One wave per row.  DIRECT: out[row] = count (every leading dim kept);
// otherwise atomically accumulate into the kept-dims index (out zeroed).
template <bool DIRECT, typename OUT>
__global__ __launch_bounds__(256) void row_counts_wave(const int32_t *__restrict__ words, int64_t rows, int64_t W,
                                                       uint32_t last_mask, LeadInfo li, OUT *__restrict__ out,
                                                       OUT denom) {
  const int lane = static_cast<int>(threadIdx.x & (kWave - 1));
  const int64_t row = (static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x) >> 6;
  if (row >= rows) return;
  const int32_t *rw = words + row * W;
  int64_t c = 0;
  for (int64_t j = lane; j < W; j += kWave) {
    uint32_t w = static_cast<uint32_t>(rw[j]);
    if (j == W - 1) w &= last_mask;
    c += __popc(w);
  }
  c = wave_sum(c);
  if (lane == 0) {
    if constexpr (DIRECT) {
      out[row] = finish<OUT>(c, denom);
    } else {
      atomicAdd(reinterpret_cast<unsigned long long *>(out + out_index(row, li)), static_cast<unsigned long long>(c));
    }
  }
}

// One lane per row, for short rows (W < 16).
template <bool DIRECT, typename OUT>
__global__ __launch_bounds__(256) void row_counts_lane(const int32_t *__restrict__ words, int64_t rows, int64_t W,
                                                       uint32_t last_mask, LeadInfo li, OUT *__restrict__ out,
                                                       OUT denom) {
  const int64_t row = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (row >= rows) return;
  const int32_t *rw = words + row * W;
  int64_t c = 0;
  for (int64_t j = 0; j < W; ++j) {
    uint32_t w = static_cast<uint32_t>(rw[j]);
    if (j == W - 1) w &= last_mask;
    c += __popc(w);
  }
  if constexpr (DIRECT) {
    out[row] = finish<OUT>(c, denom);
  } else {
    atomicAdd(reinterpret_cast<unsigned long long *>(out + out_index(row, li)), static_cast<unsigned long long>(c));
  }
}

// Counts whose kept leading dims form one contiguous block: output o sums
// the rows (a*P + o)*Q + i, a < A, i < Q (k = a*Q + i runs over AQ = A*Q).
// Blocks (o, s) of 16 waves split output o's AQ rows into S slices; wave q
// of a block takes k = q, q + 16, ... of its slice, four rows per pass, and
// wave 0 adds the 16 wave sums.  S == 1 stores the count; S > 1 adds the S
// slice counts atomically (out zeroed; a handful of atomics per output, and
// integer sums are order-independent).
constexpr int kBlkWaves = 16;

template <typename OUT>
__global__ __launch_bounds__(1024) void row_counts_block(const int32_t *__restrict__ words, int64_t W,
                                                         uint32_t last_mask, int64_t P, int64_t Q, int64_t AQ,
                                                         int64_t slice, int atomic, OUT *__restrict__ out, OUT denom) {
  __shared__ int64_t part[kBlkWaves];
  const int lane = static_cast<int>(threadIdx.x & 63), q = static_cast<int>(threadIdx.x >> 6);
  const int64_t o = blockIdx.x;
  const int64_t k_begin = static_cast<int64_t>(blockIdx.y) * slice;
  const int64_t k_end = (k_begin + slice < AQ) ? k_begin + slice : AQ;
  int64_t c = 0;
  for (int64_t k = k_begin + q; k < k_end; k += 4 * kBlkWaves) {
    const int32_t *rw[4];
    bool ok[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int64_t kk = k + u * kBlkWaves;
      ok[u] = kk < k_end;
      const int64_t a = kk / Q, i = kk - a * Q;
      rw[u] = ok[u] ? words + ((a * P + o) * Q + i) * W : words;
    }
    for (int64_t j = lane; j < W; j += kWave) {
      const uint32_t m = (j == W - 1) ? last_mask : 0xffffffffu;
#pragma unroll
      for (int u = 0; u < 4; ++u)
        if (ok[u]) c += __popc(static_cast<uint32_t>(rw[u][j]) & m);
    }
  }
  c = wave_sum(c);
  if (lane == 0) part[q] = c;
  __syncthreads();
  if (threadIdx.x == 0) {
    int64_t t = 0;
#pragma unroll
    for (int i = 0; i < kBlkWaves; ++i) t += part[i];
    if (atomic)
      atomicAdd(reinterpret_cast<unsigned long long *>(out + o), static_cast<unsigned long long>(t));
    else
      out[o] = finish<OUT>(t, denom);
  }
}

__global__ __launch_bounds__(256) void fill_i64(int64_t *__restrict__ p, int64_t n) {
  const int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i < n) p[i] = 0;
}

// Per-neuron counts over R leading rows: words [R, K, W] -> out [K, n].
// Block = 8 waves x 64 word-columns; wave q walks rows r = q, q+8, ...
// inside the block's row range, 16 rows' loads issued before any is used.
// Bit counts are accumulated SWAR-style: acc[j] holds, in its 4 bytes, the
// counts of bits j, j+8, j+16, j+24.  A block spans at most 8 * 255 rows,
// so no byte of a wave's counts passes 255.  The 8 waves' counts are then
// summed through LDS; a block covering all R rows stores, otherwise it
// atomically adds (out zeroed).
constexpr int kKeepWaves = 8;
constexpr int kKeepRows = kKeepWaves * 255;  // rows per block
constexpr int kKeepAhead = 16;               // row loads in flight per lane

__global__ __launch_bounds__(512) void keep_last_counts(const int32_t *__restrict__ words, int64_t R, int64_t KW,
                                                        int64_t W, int64_t n, int64_t *__restrict__ out,
                                                        int atomic) {
  __shared__ uint8_t red[kKeepWaves][32][68];  // [wave][bit][word column], each at most 255
  const int lane = static_cast<int>(threadIdx.x & 63);
  const int q = static_cast<int>(threadIdx.x >> 6);
  const int64_t col = static_cast<int64_t>(blockIdx.x) * 64 + lane;  // (k, w) flattened
  const bool active = col < KW;
  const int64_t r_begin = static_cast<int64_t>(blockIdx.y) * kKeepRows;
  const int64_t r_end = (r_begin + kKeepRows < R) ? r_begin + kKeepRows : R;

  uint32_t acc[8];
#pragma unroll
  for (int j = 0; j < 8; ++j) acc[j] = 0;
  // The loop below is bound by its instructions where few columns leave few
  // waves (25,600 rows of one word).  Four- and eight-byte ones alternate in
  // it, and where it starts on an odd dword it runs faster: 46 against 58 us.
  asm volatile("s_nop 0");
  if (active) {
    const int32_t *p = words + col;
    int64_t r = r_begin + q;
    for (; r + (kKeepAhead - 1) * kKeepWaves < r_end; r += kKeepAhead * kKeepWaves) {
      uint32_t w[kKeepAhead];
#pragma unroll
      for (int u = 0; u < kKeepAhead; ++u) w[u] = static_cast<uint32_t>(p[(r + u * kKeepWaves) * KW]);
#pragma unroll
      for (int u = 0; u < kKeepAhead; ++u)
#pragma unroll
        for (int j = 0; j < 8; ++j) acc[j] += (w[u] >> j) & 0x01010101u;
    }
    for (; r < r_end; r += kKeepWaves) {
      const uint32_t w = static_cast<uint32_t>(p[r * KW]);
#pragma unroll
      for (int j = 0; j < 8; ++j) acc[j] += (w >> j) & 0x01010101u;
    }
  }
#pragma unroll
  for (int j = 0; j < 8; ++j)
#pragma unroll
    for (int y = 0; y < 4; ++y) red[q][8 * y + j][lane] = static_cast<uint8_t>(acc[j] >> (8 * y));
  __syncthreads();
  // the block's 64 words x 32 bits in output order, lanes along the bits:
  // coalesced stores (one wave adding up and each lane storing its own
  // word's 32 counts: 32768 rows of 8192 bits 31.6 -> 25.9 us)
#pragma unroll
  for (int u = 0; u < 2048 / (64 * kKeepWaves); ++u) {
    const int i = u * 64 * kKeepWaves + static_cast<int>(threadIdx.x);
    const int wc = i >> 5, bit = i & 31;
    const int64_t c = static_cast<int64_t>(blockIdx.x) * 64 + wc;
    if (c >= KW) continue;
    int32_t sum = 0;
#pragma unroll
    for (int o = 0; o < kKeepWaves; ++o) sum += red[o][bit][wc];
    const int64_t k = c / W;
    const int64_t j = (c - k * W) * 32 + bit;
    if (j < n) {
      int64_t *dst = out + k * n + j;
      if (atomic)
        atomicAdd(reinterpret_cast<unsigned long long *>(dst), static_cast<unsigned long long>(sum));
      else
        *dst = sum;
    }
  }
}

template <typename OUT>
__global__ __launch_bounds__(256) void rate_kernel(const int64_t *__restrict__ c, OUT *__restrict__ out, int64_t numel,
                                                   OUT denom) {
  const int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i < numel) out[i] = static_cast<OUT>(c[i]) / denom;
}

int64_t blocks(int64_t threads, int per = 256) { return (threads + per - 1) / per; }

template <class E>
int pack_typed(const void *src, int32_t *words, int64_t rows, int64_t n, hipStream_t s) {
  const int64_t W = (n + 31) / 32;
  const int64_t total = rows * W;
  constexpr int size = sizeof(typename E::T);
  if constexpr (size <= 2) {
    const auto *p = static_cast<const uint8_t *>(src);
    const dim3 grid(blocks(total));
    if (n * size % 16 == 0 && myelin::aligned(src, 16))
      pack_words<size, 16><<<grid, dim3(256), 0, s>>>(p, words, total, W, n);
    else if (n * size % 8 == 0 && myelin::aligned(src, 8))
      pack_words<size, 8><<<grid, dim3(256), 0, s>>>(p, words, total, W, n);
    else
      pack_words<size, 4><<<grid, dim3(256), 0, s>>>(p, words, total, W, n);
  } else {
    const int64_t waves = (total + 63) / 64;
    const dim3 grid(blocks(waves * 64));
    const auto *p = static_cast<const typename E::T *>(src);
    if (n % 32 == 0)
      pack_kernel<E, true><<<grid, dim3(256), 0, s>>>(p, words, total, W, n);
    else
      pack_kernel<E, false><<<grid, dim3(256), 0, s>>>(p, words, total, W, n);
  }
  return myelin::launched("pack");
}

template <typename S>
int unpack_typed(const int32_t *words, void *dst, int64_t rows, int64_t n, S one, hipStream_t s) {
  const int64_t W = (n + 31) / 32, total = rows * n;
  S *d = static_cast<S *>(dst);
  if (myelin::aligned(dst, 16)) {
    const dim3 grid(blocks((total + 16 / sizeof(S) - 1) / (16 / sizeof(S))));
    if (n % 32 == 0)
      unpack_kernel<S, true><<<grid, dim3(256), 0, s>>>(words, d, total, n, W, one);
    else
      unpack_kernel<S, false><<<grid, dim3(256), 0, s>>>(words, d, total, n, W, one);
  } else {
    unpack_generic<S><<<dim3(blocks(total)), dim3(256), 0, s>>>(words, d, total, n, W, one);
  }
  return myelin::launched("unpack");
}

}  // namespace

extern "C" int myelin_pack(const void *src, int dtype, int32_t *words, int64_t rows, int64_t n,
                           myelin_stream_t stream) {
  if (rows < 0 || n < 1) return myelin::invalid("pack: rows must be >= 0 and n >= 1");
  if (rows == 0) return MYELIN_OK;
  if (src == nullptr || words == nullptr) return myelin::invalid("pack: null pointer");
  hipStream_t s = myelin::as_hip(stream);
  switch (dtype) {
    case MYELIN_DT_F32: return pack_typed<F32>(src, words, rows, n, s);
    case MYELIN_DT_F64: return pack_typed<F64>(src, words, rows, n, s);
    case MYELIN_DT_F16:
    case MYELIN_DT_BF16: return pack_typed<H16>(src, words, rows, n, s);
    case MYELIN_DT_U8: return pack_typed<U8>(src, words, rows, n, s);
    case MYELIN_DT_I32: return pack_typed<I32>(src, words, rows, n, s);
    case MYELIN_DT_I64: return pack_typed<I64>(src, words, rows, n, s);
    default: return myelin::invalid("pack: unsupported dtype code %d", dtype);
  }
}

extern "C" int myelin_unpack(const int32_t *words, void *dst, int dtype, int64_t rows, int64_t n,
                             myelin_stream_t stream) {
  if (rows < 0 || n < 1) return myelin::invalid("unpack: rows must be >= 0 and n >= 1");
  if (rows == 0) return MYELIN_OK;
  if (words == nullptr || dst == nullptr) return myelin::invalid("unpack: null pointer");
  hipStream_t s = myelin::as_hip(stream);
  switch (dtype) {
    case MYELIN_DT_F32: return unpack_typed<uint32_t>(words, dst, rows, n, 0x3f800000u, s);
    case MYELIN_DT_F64: return unpack_typed<uint64_t>(words, dst, rows, n, 0x3ff0000000000000ull, s);
    case MYELIN_DT_F16: return unpack_typed<uint16_t>(words, dst, rows, n, uint16_t(0x3c00), s);
    case MYELIN_DT_BF16: return unpack_typed<uint16_t>(words, dst, rows, n, uint16_t(0x3f80), s);
    case MYELIN_DT_U8: return unpack_typed<uint8_t>(words, dst, rows, n, uint8_t(1), s);
    case MYELIN_DT_I32: return unpack_typed<uint32_t>(words, dst, rows, n, 1u, s);
    case MYELIN_DT_I64: return unpack_typed<uint64_t>(words, dst, rows, n, 1ull, s);
    default: return myelin::invalid("unpack: unsupported dtype code %d", dtype);
  }
}

namespace {

// Counts (OUT int64) or rates count / denom (float, double) over dims that
// include the last.  `counts` is where counts are summed that several
// workgroups add to (the output itself for OUT int64).
template <typename OUT>
int counts_impl(const int32_t *words, int ndim_lead, const int64_t *lead_shape, uint32_t reduce_mask, int64_t n,
                OUT *out, OUT denom, int64_t *counts, hipStream_t s) {
  constexpr bool RATE = !(sizeof(OUT) == 8 && OUT(0.5) == OUT(0));
  if (ndim_lead < 0 || ndim_lead > 8) return myelin::invalid("packed_counts: 0..8 leading dims supported");
  if (n < 1) return myelin::invalid("packed_counts: n must be >= 1");
  if (out == nullptr || counts == nullptr || (ndim_lead > 0 && lead_shape == nullptr)) return myelin::invalid("packed_counts: null pointer");
  LeadInfo li{};
  li.ndim = ndim_lead;
  int64_t rows = 1, kept = 1;
  for (int d = ndim_lead - 1; d >= 0; --d) {
    if (lead_shape[d] < 0) return myelin::invalid("packed_counts: negative dim");
    li.shape[d] = lead_shape[d];
    rows *= lead_shape[d];
    if (reduce_mask & (1u << d)) {
      li.out_stride[d] = 0;
    } else {
      li.out_stride[d] = kept;
      kept *= lead_shape[d];
    }
  }
  const uint32_t lead_mask = ndim_lead > 0 ? ((1u << ndim_lead) - 1u) : 0u;
  const bool direct = (reduce_mask & lead_mask) == 0;
  // kept leading dims [d0, d1] contiguous (or none kept): out = (row / Q) % P
  int d0 = -1, d1 = -1;
  for (int d = 0; d < ndim_lead; ++d)
    if (!(reduce_mask & (1u << d))) {
      if (d0 < 0) d0 = d;
      d1 = d;
    }
  bool block_ok = !direct;
  int64_t P = 1, Q = 1;
  if (block_ok) {
    for (int d = (d0 < 0 ? ndim_lead : d0); d <= d1; ++d) {
      if (reduce_mask & (1u << d)) block_ok = false;
      P *= lead_shape[d];
    }
    for (int d = (d1 < 0 ? ndim_lead : d1 + 1); d < ndim_lead; ++d) Q *= lead_shape[d];
  }
  // heavy reductions onto few outputs take the block kernel; others scatter
  const int64_t AQ = kept > 0 ? rows / kept : 0;
  block_ok = block_ok && kept <= 65535 && AQ >= 16;
  int64_t S = 1;
  if (block_ok) {
    S = cdiv64(256, kept);
    // up to 320 rows (five passes of a workgroup, 1.5 us each) and 128 KB of
    // words an output, one workgroup sums them sooner than several with a
    // zeroing launch before them (50 outputs of 300 rows of 73 words: 5.2 +
    // 4.7 -> 6 us; but one output of 25,600 rows of one word, 400 passes, 620
    // us against 11, and 32 outputs of 1,000 such rows 27 against 12)
    if (AQ <= 320 && AQ * ((n + 31) / 32) <= 32768) S = 1;
    const int64_t by_rows = cdiv64(AQ, 64);
    if (S > by_rows) S = by_rows;
    if (S > 65535) S = 65535;
    if (S < 1) S = 1;
  }
  // several workgroups add to an output: zeroed counts, and for rates the
  // division after them
  const bool shared = !direct && (!block_ok || S > 1);
  const auto divide = [&]() {
    if constexpr (RATE) {
      if (kept > 0) rate_kernel<OUT><<<dim3(blocks(kept)), dim3(256), 0, s>>>(counts, out, kept, denom);
    }
    return myelin::launched("packed_counts");
  };
  if (shared || rows == 0) {
    if (kept == 0) return MYELIN_OK;
    fill_i64<<<dim3(blocks(kept)), dim3(256), 0, s>>>(counts, kept);
    if (int rc = myelin::launched("packed_counts zero")) return rc;
  }
  if (rows == 0) return divide();
  if (words == nullptr) return myelin::invalid("packed_counts: null words");
  const int64_t W = (n + 31) / 32;
  const int rem = static_cast<int>(n % 32);
  const uint32_t last_mask = rem ? ((1u << rem) - 1u) : 0xffffffffu;
  if (block_ok) {
    const int64_t slice = cdiv64(AQ, S);
    const dim3 grid(static_cast<unsigned>(kept), static_cast<unsigned>(S)), block(1024);
    if (S > 1)
      row_counts_block<int64_t><<<grid, block, 0, s>>>(words, W, last_mask, P, Q, AQ, slice, 1, counts, 1);
    else
      row_counts_block<OUT><<<grid, block, 0, s>>>(words, W, last_mask, P, Q, AQ, slice, 0, out, denom);
  } else if (W >= 16) {
    const dim3 grid(blocks(rows * 64));
    if (direct)
      row_counts_wave<true, OUT><<<grid, dim3(256), 0, s>>>(words, rows, W, last_mask, li, out, denom);
    else
      row_counts_wave<false, int64_t><<<grid, dim3(256), 0, s>>>(words, rows, W, last_mask, li, counts, 1);
  } else {
    const dim3 grid(blocks(rows));
    if (direct)
      row_counts_lane<true, OUT><<<grid, dim3(256), 0, s>>>(words, rows, W, last_mask, li, out, denom);
    else
      row_counts_lane<false, int64_t><<<grid, dim3(256), 0, s>>>(words, rows, W, last_mask, li, counts, 1);
  }
  if (shared) return divide();
  return myelin::launched("packed_counts");
}

}  // namespace

extern "C" int myelin_packed_counts(const int32_t *words, int ndim_lead, const int64_t *lead_shape,
                                    uint32_t reduce_mask, int64_t n, int64_t *out, myelin_stream_t stream) {
  return counts_impl<int64_t>(words, ndim_lead, lead_shape, reduce_mask, n, out, 1, out, myelin::as_hip(stream));
}

extern "C" int myelin_packed_rates(const int32_t *words, int ndim_lead, const int64_t *lead_shape,
                                   uint32_t reduce_mask, int64_t n, int64_t denominator, int64_t *counts, void *out,
                                   int dtype, myelin_stream_t stream) {
  hipStream_t s = myelin::as_hip(stream);
  if (dtype == MYELIN_DT_F32)
    return counts_impl<float>(words, ndim_lead, lead_shape, reduce_mask, n, static_cast<float *>(out),
                              static_cast<float>(denominator), counts, s);
  if (dtype == MYELIN_DT_F64)
    return counts_impl<double>(words, ndim_lead, lead_shape, reduce_mask, n, static_cast<double *>(out),
                               static_cast<double>(denominator), counts, s);
  return myelin::invalid("packed_rates: dtype must be F32 or F64");
}

extern "C" int myelin_packed_counts_keep_last(const int32_t *words, int64_t R, int64_t K, int64_t n, int64_t *out,
                                              myelin_stream_t stream) {
  if (R < 0 || K < 0 || n < 1) return myelin::invalid("packed_counts_keep_last: bad sizes");
  if (out == nullptr) return myelin::invalid("packed_counts_keep_last: null out");
  hipStream_t s = myelin::as_hip(stream);
  const int64_t W = (n + 31) / 32;
  const int64_t KW = K * W;
  const int64_t out_n = K * n;
  if (out_n == 0) return MYELIN_OK;
  const int64_t row_blocks = (R + kKeepRows - 1) / kKeepRows;
  const int atomic = row_blocks > 1 ? 1 : 0;
  if (atomic || R == 0) {
    fill_i64<<<dim3(blocks(out_n)), dim3(256), 0, s>>>(out, out_n);
    if (int rc = myelin::launched("keep_last zero")) return rc;
  }
  if (R == 0) return MYELIN_OK;
  if (words == nullptr) return myelin::invalid("packed_counts_keep_last: null words");
  if (row_blocks > 65535) return myelin::invalid("packed_counts_keep_last: too many rows");
  const dim3 grid((KW + 63) / 64, row_blocks);
  keep_last_counts<<<grid, dim3(64 * kKeepWaves), 0, s>>>(words, R, KW, W, n, out, atomic);
  return myelin::launched("keep_last_counts");
}

extern "C" int myelin_counts_to_rate(const int64_t *counts, void *out, int dtype, int64_t numel, int64_t denominator,
                                     myelin_stream_t stream) {
  if (numel < 0) return myelin::invalid("counts_to_rate: negative numel");
  if (numel == 0) return MYELIN_OK;
  if (counts == nullptr || out == nullptr) return myelin::invalid("counts_to_rate: null pointer");
  hipStream_t s = myelin::as_hip(stream);
  const dim3 grid(blocks(numel));
  if (dtype == MYELIN_DT_F32) {
    rate_kernel<float><<<grid, dim3(256), 0, s>>>(counts, static_cast<float *>(out), numel,
                                                   static_cast<float>(denominator));
  } else if (dtype == MYELIN_DT_F64) {
    rate_kernel<double><<<grid, dim3(256), 0, s>>>(counts, static_cast<double *>(out), numel,
                                                    static_cast<double>(denominator));
  } else {
    return myelin::invalid("counts_to_rate: dtype must be F32 or F64");
  }
  return myelin::launched("counts_to_rate");
}
