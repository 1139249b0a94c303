// ytm_matrix.hip -- clause evaluation for scoring as a product on gfx950's matrix cores.
//
// A clause fires on a patch when every literal it includes is 1 there.  With x_l the patch's
// positive literals (the negated ones their complements) and s_l = [l included] -
// [not-l included], the sum over l of s_l x_l reaches the number of included positive
// literals exactly when the clause fires, and stays below it otherwise (a clause that includes
// a literal and its negation never reaches it).  Without appended negations, or for samples
// whose negated literals are not the complements, the sum runs over all L literals with s_l =
// [l included].  The values 0, 1, -1 are exact in FP4 (E2M1) and the sums are whole numbers
// below 2^24 in f32, so the product on v_mfma_f32_32x32x64_f8f6f4 decides as the bit test
// does, 65536 literal tests an instruction of 32 cycles.
//
// Scoring (calc_class_sums_infer_batch, kernel.cu:319-343) then has three steps: the include
// masks become FP4 fragments (pack_clauses_kernel, kept while the model is unchanged), a
// product gives each sample's firing clauses as a bit row (fire_patches_kernel), and a second
// product, of these bits and the weights' base-256 digits on the int8 matrix cores, gives the
// class sums (votes_kernel).
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <algorithm>

#include "ytm_device.h"
#include "ytm_internal.h"

namespace ytm {

namespace {

typedef int v4i __attribute__((ext_vector_type(4)));
typedef int v8i __attribute__((ext_vector_type(8)));
typedef int v16i __attribute__((ext_vector_type(16)));
typedef float v16f __attribute__((ext_vector_type(16)));

constexpr int kTile = 32;        // rows (patches) and columns (clauses) of one product tile
constexpr int kStep = 64;        // literals of one product instruction
constexpr int kFragBytes = 1024; // one operand of one instruction: 64 lanes x 32 FP4 values
constexpr int kMaxSteps = 9;     // literal steps whose patch operands fit registers
// What no product reaches: the threshold of an empty clause, which does not vote.
constexpr float kNever = 1.0e9f;

// Bits of v (8 of them) as the low bits of 8 nibbles.
__device__ __forceinline__ uint32_t nibbles(uint32_t v) {
  v = (v | (v << 12)) & 0x000F000Fu;
  v = (v | (v << 6)) & 0x03030303u;
  return (v | (v << 3)) & 0x11111111u;
}

// 32 FP4 values, 1.0 (0x2) where the bit of `on` is set, negative (0x8) where `neg` is set too.
__device__ __forceinline__ v4i fp4_of(uint32_t on, uint32_t neg) {
  v4i r;
#pragma unroll
  for (int q = 0; q < 4; ++q)
    r[q] = (int)((nibbles((on >> (8 * q)) & 0xFFu) << 1) | (nibbles((neg >> (8 * q)) & 0xFFu) << 3));
  return r;
}

__device__ __forceinline__ v8i wide(v4i x) { return __builtin_shufflevector(x, x, 0, 1, 2, 3, -1, -1, -1, -1); }

// Word j of the bits [from, from + n) of row m (W words), bit b = bit from + 32 j + b.
__device__ __forceinline__ uint32_t bits_at(const uint32_t* m, int64_t W, int64_t from, int64_t n, int64_t j) {
  const int64_t left = n - 32 * j;
  if (left <= 0) return 0u;
  const int64_t at = from + 32 * j, w = at >> 5;
  const int sh = (int)(at & 31);
  const uint32_t lo = m[w], hi = sh && w + 1 < W ? m[w + 1] : 0u;
  const uint32_t v = sh ? (lo >> sh) | (hi << (32 - sh)) : lo;
  return left >= 32 ? v : v & ((1u << left) - 1u);
}

// Clause operands: frag[tile of 32 clauses][step][lane], lane l holding 32 values (literals
// 64 step + 32 (l / 32) ...) of clause 32 tile + l % 32; zero past the last clause or literal.
__global__ __launch_bounds__(256) void pack_clauses_kernel(const uint32_t* __restrict__ planes, Geom g, int steps,
                                                           int ternary, v4i* __restrict__ frag) {
  const int64_t ct = (g.C + kTile - 1) / kTile;
  const int64_t n = ternary ? g.Lh : g.L;
  for (int64_t idx = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; idx < ct * steps * kWave;
       idx += (int64_t)gridDim.x * blockDim.x) {
    const int l = (int)(idx % kWave);
    const int64_t s = idx / kWave % steps, c = idx / kWave / steps * kTile + (l & 31);
    const int64_t j = 2 * s + (l >> 5);
    uint32_t pos = 0u, neg = 0u;
    if (c < g.C) {
      const uint32_t* m = planes + (c * g.np + g.np - 1) * g.W;
      pos = bits_at(m, g.W, 0, n, j);
      if (ternary) neg = bits_at(m, g.W, g.Lh, g.Lh, j);
    }
    frag[idx] = fp4_of(pos ^ neg, neg & ~pos);
  }
}

// The value a clause's product reaches where it fires, plus the 1 that the products start
// from; a wave per clause.  [32 tiles] floats.
__global__ __launch_bounds__(256) void clause_need_kernel(const uint32_t* __restrict__ planes, Geom g, int ternary,
                                                          float* __restrict__ need) {
  const int lane = lane_id();
  const int64_t n = ternary ? g.Lh : g.L, rows = (g.C + kTile - 1) / kTile * kTile;
  const int64_t nwaves = (int64_t)gridDim.x * blockDim.x / kWave;
  for (int64_t c = (blockIdx.x * (int64_t)blockDim.x + threadIdx.x) / kWave; c < rows; c += nwaves) {
    int pos = 0, all = 0;
    if (c < g.C) {
      const uint32_t* m = planes + (c * g.np + g.np - 1) * g.W;
      for (int64_t j = lane; j < g.W; j += kWave) {
        pos += __popc(bits_at(m, g.W, 0, n, j));
        all |= m[j] != 0u;
      }
    }
    pos = wave_sum_i32(pos);
    const bool empty = !__any(all);
    if (lane == 0) need[c] = empty ? kNever : (float)(pos + 1);
  }
}

// Firing clauses of samples with several patches: bit c % 32 of masks[e][c / 32].
//
// A block takes S samples (or one sample in several rounds) and a range of clause tiles.  Its
// patches are cut into tiles of 32 rows, T per wave, whose FP4 operands are made once from the
// encoded words and stay in registers (a lane's 32 literals are one encoded word of its
// patch); the clause operands stream through two LDS buffers, copied there directly from
// global memory while the buffer before is used, so each is read once per block and used for
// every tile of it.  Only the largest of a clause's sums over its patches matters, so looking
// at a tile is eight three-way maxima; the sums start at 1, which keeps what is compared
// positive, and positive floats order like their bits.  ONE: a wave's tiles are of one sample.
//
// Bound by the matrix cores, and these by power: a loop of this instruction alone takes 17 ns a
// SIMD (32 cycles at 1.9 GHz; bf16 at 2.2 GHz).  28x28 in 10x10 patches (3 steps), 8000
// clauses, 10000 samples: 9.6 ms with literal lists in LDS, 1.64 ms now, 1.49 ms at that rate.
// 32x32x24 in 3x3 patches (5 steps), 20000 clauses, 2000 samples: 6.0 -> 3.6 ms, 3.3 ms.
template <int KS, int T, int WAVES, bool ONE>
__global__ __launch_bounds__(64 * WAVES) void fire_patches_kernel(const uint32_t* __restrict__ X, int64_t N, Geom g,
                                                           const v4i* __restrict__ frag,
                                                           const float* __restrict__ need, int S, int64_t tiles_each,
                                                           int64_t nchunk, int64_t row_words,
                                                           uint32_t* __restrict__ masks) {
  constexpr int CT = KS <= 5 ? 8 : 4;  // clause tiles of one LDS buffer
  constexpr int kBufBytes = CT * KS * kFragBytes + CT * kTile * 4;
  extern __shared__ __attribute__((aligned(16))) unsigned char s_mem[];
  uint32_t* s_fire = (uint32_t*)(s_mem + 2 * kBufBytes);  // [S][tiles_each]
  const int lane = lane_id(), row = lane & 31, half = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x / kWave));
  const int ntile = (int)((g.P + kTile - 1) / kTile);
  const int units = S * (ONE ? (ntile + T - 1) / T * T : ntile);
  const int64_t ctiles = (g.C + kTile - 1) / kTile;
  const int64_t nblk = (N + S - 1) / S * nchunk;
  for (int64_t blk = blockIdx.x; blk < nblk; blk += gridDim.x) {
    const int64_t e0 = blk / nchunk * S, ct0 = blk % nchunk * tiles_each;
    const int nct = (int)(ct0 + tiles_each < ctiles ? tiles_each : ctiles - ct0);
    __syncthreads();  // the previous samples' firing words are written out
    for (int j = threadIdx.x; j < S * (int)tiles_each; j += blockDim.x) s_fire[j] = 0u;
    // Copies the operands and thresholds of clause tiles [at, at + CT) of the range into buffer
    // b; the last buffer's tiles past the range repeat its last one and are not used.
    auto fill = [&](int at, int b) {
      unsigned char* dst = s_mem + b * kBufBytes;
      for (int f = wave; f < CT * KS; f += WAVES) {
        const int t = at + f / KS < nct ? at + f / KS : nct - 1;
        const v4i* src = frag + ((ct0 + t) * KS + f % KS) * kWave + lane;
        __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)src,
                                         (__attribute__((address_space(3))) void*)(dst + f * kFragBytes), 16, 0, 0);
      }
      if (threadIdx.x < CT * kTile) {
        static_assert(CT * kTile <= 64 * WAVES, "a thread copies one threshold");
        const int t = at + (int)threadIdx.x / kTile < nct ? at + (int)threadIdx.x / kTile : nct - 1;
        const float* src = need + (ct0 + t) * kTile + (threadIdx.x & 31);
        __builtin_amdgcn_global_load_lds(
            (const __attribute__((address_space(1))) void*)src,
            (__attribute__((address_space(3))) void*)(dst + CT * KS * kFragBytes + wave * kWave * 4), 4, 0, 0);
      }
    };
    for (int u0 = 0; u0 < units; u0 += WAVES * T) {
      __syncthreads();  // the buffers are no longer read; s_fire is zero
      fill(0, 0);
      v16f ones;  // the start of every sum, held in registers
#pragma unroll
      for (int r = 0; r < 16; ++r) ones[r] = 1.0f;
      asm volatile("" : "+v"(ones));
      v4i a[T][KS];
      int of[T];  // sample of the wave's tile t (of the block's S)
#pragma unroll
      for (int t = 0; t < T; ++t) {
        // tiles past the last, and rows past the last patch or sample, repeat the last one,
        // which changes no clause's largest sum
        int tile;
        if (ONE) {
          const int per = (ntile + T - 1) / T, v = u0 / T + wave;  // waves a sample
          of[t] = v / per < S ? v / per : S - 1;
          tile = v / per < S ? v % per * T + t : ntile;
        } else {
          const int u = u0 + wave * T + t < units ? u0 + wave * T + t : units - 1;
          of[t] = u / ntile;
          tile = u - of[t] * ntile;
        }
        const int64_t e = e0 + of[t] < N ? e0 + of[t] : N - 1;
        const int64_t p = (int64_t)tile * kTile + row;
        const uint32_t* x = X + (e * g.P + (p < g.P ? p : g.P - 1)) * g.W;
#pragma unroll
        for (int k = 0; k < KS; ++k) {
          const int w = 2 * k + half;
          a[t][k] = fp4_of(x[w < g.W ? w : g.W - 1], 0u);  // past the literals the clause operand is 0
        }
      }
      for (int at = 0, b = 0; at < nct; at += CT, b ^= 1) {
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // this wave's copies into buffer b
        __syncthreads();                                  // everyone's; buffer b ^ 1 is no longer read
        if (at + CT < nct) fill(at + CT, b ^ 1);
        const v4i* s_b = (const v4i*)(s_mem + b * kBufBytes);
        const float* s_need = (const float*)(s_mem + b * kBufBytes + CT * KS * kFragBytes);
        const int n = nct - at < CT ? nct - at : CT;
        // lane j: the clauses of tile at + j that fire on the wave's tile t (ONE: on any of them)
        int fire[ONE ? 1 : T];
#pragma unroll
        for (int t = 0; t < (ONE ? 1 : T); ++t) fire[t] = 0;
        // The products of a tile are issued before the one before it is looked at, so that the
        // maxima run beside them.
        v16f d[2];
        int m = 0, want = 0;
        // Looks at the sums of the wave's tile t with clause tile j of the buffer.
        auto look = [&](const v16f& x, int t, int j, int w) {
          m = ONE && t > 0 ? max(m, __float_as_int(x[0])) : __float_as_int(x[0]);
#pragma unroll
          for (int r = 1; r < 16; ++r) m = max(m, __float_as_int(x[r]));
          if (ONE && t + 1 < T) return;
          const unsigned long long hit = __ballot(m == w);
          int& f = fire[ONE ? 0 : t];
          f = lane == j ? (int)((uint32_t)hit | (uint32_t)(hit >> 32)) : f;
        };
#pragma unroll
        for (int r = 0; r < 16; ++r) d[1][r] = 0.0f;
        for (int j0 = 0; j0 < n; j0 += 2) {
#pragma unroll
          for (int q = 0; q < 2; ++q) {
            const int j = j0 + q;  // < CT: the tile past an odd n was copied too, its words are dropped
            v4i bv[KS];
#pragma unroll
            for (int k = 0; k < KS; ++k) bv[k] = s_b[(j * KS + k) * kWave + lane];
            const int before = want;
            want = __float_as_int(s_need[j * kTile + row]);
#pragma unroll
            for (int t = 0; t < T; ++t) {
              const int cur = (q * T + t) & 1;
              if (t == 0) look(d[cur ^ 1], T - 1, j - 1, before);  // while the operands are read
              v16f x = ones;
#pragma unroll
              for (int k = 0; k < KS; ++k)
                x = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(wide(a[t][k]), wide(bv[k]), x, 4, 4, 0, 0, 0, 0);
              d[cur] = x;
              if (t > 0) {
                look(d[cur ^ 1], t - 1, j, want);
                // one product instruction, then a share of the maxima, in turn
#pragma unroll
                for (int k = 0; k < KS; ++k) {
                  __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                  __builtin_amdgcn_sched_group_barrier(0x002, (8 + KS - 1) / KS, 0);
                }
              }
              __builtin_amdgcn_sched_barrier(0);
            }
          }
        }
        look(d[(2 * T - 1) & 1], T - 1, (n - 1) | 1, want);
        // a buffer's firing words together: an LDS atomic waits for the copies in flight
#pragma unroll
        for (int t = 0; t < (ONE ? 1 : T); ++t)
          if (fire[t] && lane < n) atomicOr(&s_fire[of[t] * (int)tiles_each + at + lane], (uint32_t)fire[t]);
      }
    }
    __syncthreads();
    for (int j = threadIdx.x; j < S * nct; j += blockDim.x) {
      const int s = j / nct, w = j - s * nct;
      if (e0 + s < N) masks[(e0 + s) * row_words + ct0 + w] = s_fire[s * (int)tiles_each + w];
    }
  }
}

// Weight operands of votes_kernel: frag[word of 32 clauses][column group][lane], lane l holding
// 16 int8 values (clauses 32 word + 16 (l / 32) ...) of column l % 32: digit col % D of class
// group * (32 / D) + col / D, the weights in signed base-256 digits, least significant first.
__global__ __launch_bounds__(256) void pack_weights_kernel(const float* __restrict__ w, Geom g, int64_t words, int D,
                                                           int groups, v4i* __restrict__ frag) {
  const int per = kTile / D;
  for (int64_t idx = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; idx < words * groups * kWave;
       idx += (int64_t)gridDim.x * blockDim.x) {
    const int l = (int)(idx % kWave), grp = (int)(idx / kWave % groups);
    const int64_t c0 = idx / kWave / groups * kTile + 16 * (l >> 5);
    const int col = l & 31, k = grp * per + col / D, digit = col % D;
    v4i r;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      uint32_t word = 0u;
#pragma unroll
      for (int b = 0; b < 4; ++b) {
        const int64_t c = c0 + 4 * q + b;
        long long v = c < g.C && col / D < per && k < g.K ? (long long)w[c * g.K + k] : 0;
        int d = 0;
        for (int i = 0; i <= digit; ++i) {
          d = (int)(signed char)(v & 255);
          v = (v - d) >> 8;
        }
        word |= (uint32_t)(d & 255) << (8 * b);
      }
      r[q] = (int)word;
    }
    frag[idx] = r;
  }
}

// Class sums of 32 samples from their firing bits: the product of the bits (0 / 1) and the
// weights' digits on v_mfma_i32_32x32x32_i8, 32 clauses an instruction, exact in int32 (a
// digit is at most 128 in magnitude, so 2^24 clauses fit).  The block's waves share the words
// of a row; their sums meet in LDS and the digits are put together in int64, plus the bias,
// rounded once (calc_class_sums_infer_batch, kernel.cu:319-343).  Blocks: x sample tiles, y
// column groups.
constexpr int kVoteWaves = 8;
__global__ __launch_bounds__(64 * kVoteWaves) void votes_kernel(const uint32_t* __restrict__ masks, int64_t row_words,
                                                                int64_t N, const v4i* __restrict__ frag, Geom g, int D,
                                                                int groups, const float* __restrict__ bias,
                                                                float* __restrict__ out) {
  __shared__ int s_sum[kVoteWaves][kTile][kTile];  // [wave][sample][column]
  const int lane = lane_id(), col = lane & 31, half = lane >> 5;
  const int wave = threadIdx.x / kWave;
  const int64_t e0 = (int64_t)blockIdx.x * kTile;
  const int grp = blockIdx.y, per = kTile / D;
  const int64_t e = e0 + col < N ? e0 + col : N - 1;
  const uint32_t* row = masks + e * row_words;
  v16i d;
#pragma unroll
  for (int r = 0; r < 16; ++r) d[r] = 0;
  // four words (one 16-byte read of the row, whose length is a multiple of 4) at a time
  for (int64_t w0 = 4 * wave; w0 < row_words; w0 += 4 * kVoteWaves) {
    const uint4 mw = *(const uint4*)(row + w0);
    const uint32_t m4[4] = {mw.x, mw.y, mw.z, mw.w};
    v4i bv[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) bv[q] = frag[((w0 + q) * groups + grp) * kWave + lane];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const uint32_t m = m4[q] >> (16 * half);
      v4i av;
#pragma unroll
      for (int i = 0; i < 4; ++i) av[i] = (int)((((m >> (4 * i)) & 0xFu) * 0x00204081u) & 0x01010101u);
      d = __builtin_amdgcn_mfma_i32_32x32x32_i8(av, bv[q], d, 0, 0, 0);
    }
  }
#pragma unroll
  for (int r = 0; r < 16; ++r) s_sum[wave][8 * (r >> 2) + 4 * half + (r & 3)][col] = d[r];
  __syncthreads();
  for (int j = threadIdx.x; j < kTile * per; j += blockDim.x) {
    const int s = j / per, kk = j - s * per, k = grp * per + kk;
    if (e0 + s >= N || k >= g.K) continue;
    long long v = (long long)bias[k];
    for (int i = 0; i < D; ++i) {
      long long part = 0;
      for (int wv = 0; wv < kVoteWaves; ++wv) part += s_sum[wv][s][kk * D + i];
      v += part * (1ll << (8 * i));
    }
    out[(e0 + s) * g.K + k] = (float)v;
  }
}

// Clears *ok when some negated literal of an encoded row is not the complement of its
// positive one.  *ok is set before.
__global__ __launch_bounds__(256) void halves_kernel(const uint32_t* __restrict__ X, int64_t rows, Geom g, int* ok) {
  const int64_t hw = (g.Lh + 31) / 32;
  bool bad = false;
  for (int64_t idx = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; idx < rows * hw;
       idx += (int64_t)gridDim.x * blockDim.x) {
    const uint32_t* x = X + idx / hw * g.W;
    const int64_t j = idx % hw;
    const uint32_t valid = g.Lh - 32 * j >= 32 ? 0xFFFFFFFFu : (1u << (g.Lh - 32 * j)) - 1u;
    bad = bad || (bits_at(x, g.W, 0, g.Lh, j) ^ bits_at(x, g.W, g.Lh, g.Lh, j)) != valid;
  }
  if (bad) *ok = 0;
}

int blocks_for(int64_t items, int block) {
  return (int)std::min<int64_t>(std::max<int64_t>((items + block - 1) / block, 1), 65536);
}

int64_t clause_tiles(const Geom& g) { return (g.C + kTile - 1) / kTile; }

template <int KS, int T, int WAVES, bool ONE>
hipError_t launch_fire(const uint32_t* X, int64_t N, const Geom& g, const v4i* frag, const float* need, int cus,
                       int64_t row_words, uint32_t* masks, hipStream_t s) {
  constexpr int CT = KS <= 5 ? 8 : 4;
  const int ntile = (int)((g.P + kTile - 1) / kTile);
  int64_t S = std::max<int64_t>(1, ONE ? WAVES / ((ntile + T - 1) / T) : WAVES * T / ntile);
  S = std::min(S, N);
  // clause ranges: enough blocks for four a CU when the samples alone are few, whole buffers
  // each, and short enough that the firing words stay small beside the buffers
  const int64_t groups = (N + S - 1) / S, tiles = clause_tiles(g);
  const int64_t want = (4 * cus + groups - 1) / groups;
  int64_t each = std::max<int64_t>(CT, ((tiles + want - 1) / want + CT - 1) / CT * CT);
  each = std::min<int64_t>(each, std::max<int64_t>(CT, 8192 / S / CT * CT));
  each = std::min(each, tiles);
  const int64_t nchunk = (tiles + each - 1) / each;
  const size_t lds = 2 * (size_t)(CT * KS * kFragBytes + CT * kTile * 4) + (size_t)(S * each) * 4;
  fire_patches_kernel<KS, T, WAVES, ONE><<<(unsigned)std::min<int64_t>(groups * nchunk, 1 << 22), 64 * WAVES, lds, s>>>(X, N, g, frag, need, (int)S, each, nchunk,
                                                                            row_words, masks);
  return hipGetLastError();
}

// Share of a block's waves and tiles (W waves of T) that a sample of ntile tiles keeps busy.
double tile_use(int ntile, int W, int T, bool one) {
  const int units = one ? (ntile + T - 1) / T * T : ntile, room = W * T;
  if (units <= room) return (double)(room / units * ntile) / room;
  return (double)ntile / ((units + room - 1) / room * room);
}

// The kernel of KS literal steps: HI or LO tiles a wave, and whether a wave's tiles are all of
// one sample, whichever leaves the fewest idle (one sample's tiles share the look at the
// result, about a tenth of the time: preferred unless it wastes more than that; small samples,
// of fewer tiles than a wave takes, share a wave).  Sixteen waves a block, four a SIMD, up to
// three steps: the maxima of some waves then run beside the products of others (28x28 in
// 10x10 patches, 8000 clauses, 10000 samples: 1.64 ms against 1.94 ms with eight); the
// operands of four steps and more need the registers of two waves a SIMD.
template <int KS, int HI, int LO>
hipError_t fire_steps(const uint32_t* X, int64_t N, const Geom& g, const v4i* frag, const float* need, int cus,
                      int64_t row_words, uint32_t* masks, hipStream_t s) {
  constexpr int W = KS <= 3 ? 16 : 8;
  const int ntile = (int)((g.P + kTile - 1) / kTile);
  const double hi = tile_use(ntile, W, HI, true), lo = tile_use(ntile, W, LO, true);
  if (tile_use(ntile, W, HI, false) > 1.1 * std::max(hi, lo))
    return launch_fire<KS, HI, W, false>(X, N, g, frag, need, cus, row_words, masks, s);
  if (lo > hi) return launch_fire<KS, LO, W, true>(X, N, g, frag, need, cus, row_words, masks, s);
  return launch_fire<KS, HI, W, true>(X, N, g, frag, need, cus, row_words, masks, s);
}

}  // namespace

hipError_t launch_halves_check(const uint32_t* X, int64_t N, const Geom& g, int* ok, hipStream_t s) {
  halves_kernel<<<blocks_for(N * g.P * ((g.Lh + 31) / 32), 256), 256, 0, s>>>(X, N * g.P, g, ok);
  return hipGetLastError();
}

MatrixPlan matrix_plan(const Geom& g, bool halves, double w_bound) {
  MatrixPlan p{};
  p.ternary = halves && g.append_negated;
  const int64_t n = p.ternary ? g.Lh : g.L;
  const int64_t steps = (n + kStep - 1) / kStep;
  if (g.P < 2 || steps > kMaxSteps || clause_tiles(g) > (1 << 19)) return p;
  p.steps = (int)steps;
  const int64_t tiles = clause_tiles(g);
  p.row_words = (tiles + 3) / 4 * 4;
  // digits that hold every weight of magnitude up to w_bound
  double top = 127.0;
  for (p.digits = 1; top < w_bound && p.digits < 5; ++p.digits) top = top * 256.0 + 127.0;
  const int per = kTile / p.digits;
  p.groups = (int)((g.K + per - 1) / per);
  auto room = [](size_t n) { return (n + 255) & ~(size_t)255; };
  p.need_at = room((size_t)(tiles * steps) * kFragBytes);
  p.weights_at = p.need_at + room((size_t)tiles * kTile * 4);
  p.bytes = p.weights_at + (size_t)(p.row_words * p.groups) * kFragBytes;
  return p;
}

hipError_t launch_matrix_pack(const uint32_t* planes, const float* w, const Geom& g, const MatrixPlan& p,
                              void* scratch, hipStream_t s) {
  unsigned char* base = (unsigned char*)scratch;
  const int64_t tiles = clause_tiles(g);
  pack_clauses_kernel<<<blocks_for(tiles * p.steps * kWave, 256), 256, 0, s>>>(planes, g, p.steps, p.ternary,
                                                                              (v4i*)base);
  clause_need_kernel<<<blocks_for(tiles * kTile * kWave, 256), 256, 0, s>>>(planes, g, p.ternary,
                                                                           (float*)(base + p.need_at));
  pack_weights_kernel<<<blocks_for(p.row_words * p.groups * kWave, 256), 256, 0, s>>>(
      w, g, p.row_words, p.digits, p.groups, (v4i*)(base + p.weights_at));
  return hipGetLastError();
}

hipError_t launch_matrix_score(const uint32_t* X, int64_t N, const Geom& g, const MatrixPlan& p, const void* scratch,
                               int cus, const float* bias, uint32_t* masks, float* out, hipStream_t s) {
  const unsigned char* base = (const unsigned char*)scratch;
  const v4i* frag = (const v4i*)base;
  const float* need = (const float*)(base + p.need_at);
  hipError_t e = hipSuccess;
  switch (p.steps) {
#define YTM_FIRE(KS, HI, LO)                                                             \
  case KS:                                                                               \
    e = fire_steps<KS, HI, LO>(X, N, g, frag, need, cus, p.row_words, masks, s);         \
    break;
    YTM_FIRE(1, 4, 3)
    YTM_FIRE(2, 4, 3)
    YTM_FIRE(3, 3, 2)
    YTM_FIRE(4, 4, 3)
    YTM_FIRE(5, 4, 3)
    YTM_FIRE(6, 2, 1)
    YTM_FIRE(7, 2, 1)
    YTM_FIRE(8, 2, 1)
    YTM_FIRE(9, 2, 1)
#undef YTM_FIRE
    default:
      return hipErrorInvalidValue;
  }
  if (e != hipSuccess) return e;
  votes_kernel<<<dim3((unsigned)((N + kTile - 1) / kTile), (unsigned)p.groups), 64 * kVoteWaves, 0, s>>>(
      masks, p.row_words, N, (const v4i*)(base + p.weights_at), g, p.digits, p.groups, bias, out);
  return hipGetLastError();
}

}  // namespace ytm
