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
// masks become FP4 fragments (pack_model_kernel, kept while the model is unchanged), a
// product gives each sample's firing clauses as a bit row (fire_patches_kernel, fire_rows_kernel), and a second
// product, of these bits and the weights' base-256 digits on the int8 matrix cores, gives the
// class sums (votes_kernel).
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <algorithm>

#include "ytm_device.h"
#include "ytm_internal.h"

namespace ytm {

namespace {

typedef int v16i __attribute__((ext_vector_type(16)));

constexpr int kTile = 32;        // rows (patches) and columns (clauses) of one product tile
constexpr int kStep = 64;        // literals of one product instruction
constexpr int kFragBytes = 1024; // one operand of one instruction: 64 lanes x 32 FP4 values
constexpr int kMaxSteps = 9;     // literal steps whose patch operands fit registers
// What no product reaches: the threshold of an empty clause, which does not vote.
constexpr float kNever = 1.0e9f;

// Whether word j of the encoded row x's positive literals is the complement of the negated ones.
__device__ __forceinline__ bool complements(const uint32_t* x, const Geom& g, int64_t j) {
  const uint32_t valid = g.Lh - 32 * j >= 32 ? 0xFFFFFFFFu : (1u << (g.Lh - 32 * j)) - 1u;
  return (bits_at(x, g.W, 0, g.Lh, j) ^ bits_at(x, g.W, g.Lh, g.Lh, j)) == valid;
}

// Weight operands wfrag[word of 32 clauses][column group][lane], lane l holding 16 int8 values
// (clauses 32 word + 16 (l / 32) ...) of column l % 32: digit col % D of class group * (32 / D) +
// col / D, the weights in signed base-256 digits, least significant first.  By block `first` of
// `blocks`.
__device__ __forceinline__ void pack_weights(const float* __restrict__ w, const Geom& g, const MatrixPlan& p, v4i* wfrag,
                                             int64_t first, int64_t blocks) {
  const int per = kTile / p.digits;
  for (int64_t idx = first * (int64_t)blockDim.x + threadIdx.x; idx < p.row_words * p.groups * kWave;
       idx += blocks * (int64_t)blockDim.x) {
    const int l = (int)(idx % kWave), grp = (int)(idx / kWave % p.groups);
    const int64_t c0 = idx / kWave / p.groups * kTile + 16 * (l >> 5);
    const int col = l & 31, k = grp * per + col / p.digits, digit = col % p.digits;
    v4i r;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      uint32_t word = 0u;
#pragma unroll
      for (int b = 0; b < 4; ++b) {
        const int64_t c = c0 + 4 * q + b;
        long long v = c < g.C && col / p.digits < per && k < g.K ? (long long)w[c * g.K + k] : 0;
        int d = 0;
        for (int i = 0; i <= digit; ++i) {
          d = (int)(signed char)(v & 255);
          v = (v - d) >> 8;
        }
        word |= (uint32_t)(d & 255) << (8 * b);
      }
      r[q] = (int)word;
    }
    wfrag[idx] = r;
  }
}

// The model's operands, three independent parts of one launch (after every change of the model
// and before its first score: 784 bits, 2000 clauses 15.6 us in a launch each, 9.2 us in one):
//  - clause operands frag[tile of 32 clauses][step][lane], lane l holding 32 values (literals
//    64 step + 32 (l / 32) ...) of clause 32 tile + l % 32; zero past the last clause or literal;
//  - thresholds need[32 tiles]: the value a clause's product reaches where it fires, plus the
//    1 that the products start from; a wave per clause;
//  - weight operands (pack_weights).
// With half_steps, operands and thresholds over the positive literals alone come besides.
__global__ __launch_bounds__(256) void pack_model_kernel(const uint32_t* __restrict__ planes,
                                                         const float* __restrict__ w, Geom g, MatrixPlan p,
                                                         unsigned char* __restrict__ base, int64_t need_blocks,
                                                         int64_t weight_blocks) {
  v4i* frag = (v4i*)base;
  v4i* half = (v4i*)(base + p.half_at);
  float* need = (float*)(base + p.need_at);
  v4i* wfrag = (v4i*)(base + p.weights_at);
  const int64_t ct = (g.C + kTile - 1) / kTile;
  const int64_t n = p.ternary ? g.Lh : g.L;
  if (blockIdx.x < need_blocks) {
    if (blockIdx.x == 0 && threadIdx.x == 0) *(int*)(base + p.flag_at) = 0;
    const int lane = lane_id();
    const int64_t nwaves = need_blocks * blockDim.x / kWave;
    for (int64_t c = (blockIdx.x * (int64_t)blockDim.x + threadIdx.x) / kWave; c < ct * kTile; c += nwaves) {
      int pos = 0, first = 0, all = 0;
      if (c < g.C) {
        const uint32_t* m = planes + (c * g.np + g.np - 1) * g.W;
        for (int64_t j = lane; j < g.W; j += kWave) {
          pos += __popc(bits_at(m, g.W, 0, n, j));
          first += __popc(bits_at(m, g.W, 0, g.Lh, j));
          all |= m[j] != 0u;
        }
      }
      pos = wave_sum_i32(pos);
      first = wave_sum_i32(first);
      const bool empty = !__any(all);
      if (lane == 0) {
        need[c] = empty ? kNever : (float)(pos + 1);
        if (p.half_steps) need[ct * kTile + c] = empty ? kNever : (float)(first + 1);
      }
    }
    return;
  }
  int64_t first = blockIdx.x - need_blocks;
  if (first < weight_blocks) {
    pack_weights(w, g, p, wfrag, first, weight_blocks);
    return;
  }
  first -= weight_blocks;
  const int64_t blocks = gridDim.x - need_blocks - weight_blocks;
  const int each = p.steps + p.half_steps;
  for (int64_t idx = first * (int64_t)blockDim.x + threadIdx.x; idx < ct * each * kWave;
       idx += blocks * (int64_t)blockDim.x) {
    const int l = (int)(idx % kWave);
    const int64_t tile = idx / kWave / each, c = tile * kTile + (l & 31);
    const int st = (int)(idx / kWave % each), s = st < p.steps ? st : st - p.steps;
    const bool ternary = p.ternary || st >= p.steps;
    const int64_t j = 2 * (int64_t)s + (l >> 5);
    uint32_t pos = 0u, neg = 0u;
    if (c < g.C) {
      const uint32_t* m = planes + (c * g.np + g.np - 1) * g.W;
      pos = bits_at(m, g.W, 0, ternary ? g.Lh : g.L, j);
      if (ternary) neg = bits_at(m, g.W, g.Lh, g.Lh, j);
    }
    const v4i v = fp4_column(pos ^ neg, neg & ~pos);
    if (st < p.steps)
      frag[(tile * p.steps + s) * kWave + l] = v;
    else
      half[(tile * p.half_steps + s) * kWave + l] = v;
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
          a[t][k] = fp4_row(x[w < g.W ? w : g.W - 1]);  // past the literals the clause operand is 0
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
                x = fp4_product(a[t][k], bv[k], x);
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

// One patch: the rows of a product tile are samples.

// Sample operands of fire_rows_kernel: frag[tile of 32 samples][step][lane], zero past the last
// sample's words (the rows past the last sample repeat it).  With half_steps, sets *odd when a
// sample's negated literals are not the complements of its positive ones.
__global__ __launch_bounds__(256) void pack_samples_kernel(const uint32_t* __restrict__ X, int64_t N, Geom g,
                                                           int steps, int half_steps, int* odd,
                                                           v4i* __restrict__ frag) {
  const int64_t total = (N + kTile - 1) / kTile * steps * kWave;
  const int64_t hw = half_steps ? (g.Lh + 31) / 32 : 0;
  bool bad = false;
  for (int64_t idx = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; idx < total;
       idx += (int64_t)gridDim.x * blockDim.x) {
    const int l = (int)(idx % kWave);
    const int64_t w = idx / kWave % steps * 2 + (l >> 5), e = idx / kWave / steps * kTile + (l & 31);
    const uint32_t* x = X + (e < N ? e : N - 1) * g.W;
    frag[idx] = fp4_row(w < g.W ? x[w] : 0u);
    if (w < hw) bad = bad || !complements(x, g, w);
  }
  if (bad) *odd = 1;
}

// The firing words of a product tile, from its sums d (a lane: one clause, 16 samples) and the
// lane's threshold: lane i < 32 returns sample i's word, bit j = clause j.
__device__ __forceinline__ uint32_t row_words_of(const v16f& d, float want) {
  const int lane = lane_id();
  const int mine = ((lane >> 3) & 3) << 2 | (lane & 3);  // the register that holds sample `lane`
  uint32_t word = 0u;
#pragma unroll
  for (int r = 0; r < 16; ++r) {
    const unsigned long long hit = __ballot(d[r] == want);
    const uint32_t w = (lane >> 2) & 1 ? (uint32_t)(hit >> 32) : (uint32_t)hit;
    word = mine == r ? w : word;
  }
  return word;
}

// Firing clauses of one-patch samples, bit c % 32 of masks[e][c / 32]: a product of 256 samples
// by 256 clauses per block, each of its 8 waves 128 by 64 (eight tiles whose sums stay in
// registers).  Both operands stream through four LDS buffers of two steps, copied there
// directly from global memory three buffers ahead, which covers the latency of a line that
// another XCD's L2 or the memory holds; six operand reads serve eight product instructions.
// Consecutive blocks go to different XCDs, so the block index is split such that an XCD works
// on neighbouring tiles and finds their operands in its own L2.
// Bound by the matrix cores, behind them by the operands' way through LDS.  20000 literals,
// 10000 clauses, 10000 samples: 3.77 ms with include masks and literal lists, 0.46 ms now, of
// them 0.43 here; the products alone would take 0.27 ms.
constexpr int kRowSteps = 2, kRowBuffers = 4, kBlockTiles = 8;
// Samples not yet looked at (half_steps): *odd says whether the product over the positive
// literals alone, in its own operands, will do; the samples' operands begin alike.
__global__ __launch_bounds__(512) void fire_rows_kernel(const v4i* __restrict__ sfrag, int64_t N, int64_t C,
                                                        const unsigned char* __restrict__ base, MatrixPlan p,
                                                        uint32_t* __restrict__ masks) {
  constexpr int MT = 4, NT = 2;
  constexpr int kBufFrags = 2 * kBlockTiles * kRowSteps;  // samples, then clauses
  extern __shared__ __attribute__((aligned(16))) unsigned char s_mem[];
  const int lane = lane_id();
  const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x / kWave));
  const int64_t mtiles = (N + kTile - 1) / kTile, ctiles = (C + kTile - 1) / kTile;
  const int64_t mb = (mtiles + kBlockTiles - 1) / kBlockTiles, cb = (ctiles + kBlockTiles - 1) / kBlockTiles;
  const int64_t nblk = mb * cb, share = (nblk + 7) / 8;
  const bool half = p.half_steps && *(const int*)(base + p.flag_at) == 0;
  const v4i* cfrag = (const v4i*)(base + (half ? p.half_at : 0));
  const float* need = (const float*)(base + p.need_at) + (half ? ctiles * kTile : 0);
  const int steps = half ? p.half_steps : p.steps, nstage = steps / kRowSteps;
  const int64_t row_words = p.row_words;
  for (int64_t blk = blockIdx.x; blk < 8 * share; blk += gridDim.x) {
    const int64_t idx = blk % 8 * share + blk / 8;  // this XCD's range
    if (idx >= nblk) continue;
    // columns of four sample blocks: their tiles share clause operands
    const int64_t grp = idx / (4 * cb), first = grp * 4, rows = mb - first < 4 ? mb - first : 4;
    const int64_t in = idx - grp * 4 * cb;
    const int64_t m0 = (first + in % rows) * kBlockTiles, c0 = in / rows * kBlockTiles;
    // The wave's copies of stage st: one tile of samples and one of clauses, both steps
    const int64_t mt = m0 + wave < mtiles ? m0 + wave : mtiles - 1, ct = c0 + wave < ctiles ? c0 + wave : ctiles - 1;
    const v4i* sa = sfrag + mt * p.steps * kWave + lane;
    const v4i* sb = cfrag + ct * steps * kWave + lane;
    auto fill = [&](int st) {
      const int at = (st < nstage ? st : nstage - 1) * kRowSteps;  // past the end: copied again, not read
      unsigned char* dst = s_mem + (st & (kRowBuffers - 1)) * kBufFrags * kFragBytes;
#pragma unroll
      for (int k = 0; k < kRowSteps; ++k) {
        __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)(sa + (at + k) * kWave),
                                         (__attribute__((address_space(3))) void*)(dst + (k * kBlockTiles + wave) * kFragBytes),
                                         16, 0, 0);
        __builtin_amdgcn_global_load_lds(
            (const __attribute__((address_space(1))) void*)(sb + (at + k) * kWave),
            (__attribute__((address_space(3))) void*)(dst + ((kRowSteps + k) * kBlockTiles + wave) * kFragBytes), 16, 0, 0);
      }
    };
    __syncthreads();  // the buffers are no longer read
    for (int st = 0; st < kRowBuffers - 1; ++st) fill(st);
    v16f d[MT][NT];
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
      for (int j = 0; j < NT; ++j)
#pragma unroll
        for (int r = 0; r < 16; ++r) d[i][j][r] = 1.0f;
    const int wm = (wave & 1) * MT, wc = (wave >> 1) * NT;
    for (int st = 0; st < nstage; ++st) {
      // this wave's copies of stage st: the 2 * 2 * kRowSteps after them may be in flight
      asm volatile("s_waitcnt vmcnt(8)" ::: "memory");
      static_assert(kRowSteps == 2 && kRowBuffers == 4, "copies in flight");
      __syncthreads();  // everyone's; the buffer of stage st - 1 is no longer read
      fill(st + kRowBuffers - 1);
      const v4i* buf = (const v4i*)(s_mem + (st & (kRowBuffers - 1)) * kBufFrags * kFragBytes) + lane;
      v4i av[kRowSteps][MT], bv[kRowSteps][NT];
#pragma unroll
      for (int k = 0; k < kRowSteps; ++k) {
#pragma unroll
        for (int j = 0; j < NT; ++j) bv[k][j] = buf[((kRowSteps + k) * kBlockTiles + wc + j) * kWave];
#pragma unroll
        for (int i = 0; i < MT; ++i) av[k][i] = buf[(k * kBlockTiles + wm + i) * kWave];
      }
#pragma unroll
      for (int k = 0; k < kRowSteps; ++k)
#pragma unroll
        for (int i = 0; i < MT; ++i)
#pragma unroll
          for (int j = 0; j < NT; ++j)
            d[i][j] = fp4_product(av[k][i], bv[k][j], d[i][j]);
      // the first step's operands, then the second's beside the first's products
      __builtin_amdgcn_sched_group_barrier(0x100, MT + NT, 0);
#pragma unroll
      for (int q = 0; q < MT + NT; ++q) {
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
        __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
      }
      __builtin_amdgcn_sched_group_barrier(0x008, 2 * MT * NT - MT - NT, 0);
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // the copies past the end
#pragma unroll
    for (int j = 0; j < NT; ++j) {
      const int64_t c = c0 + wc + j;
      if (c >= ctiles) continue;
      const float want = need[c * kTile + (lane & 31)];
#pragma unroll
      for (int i = 0; i < MT; ++i) {
        const uint32_t word = row_words_of(d[i][j], want);
        const int64_t e = (m0 + wm + i) * kTile + lane;
        if (lane < kTile && e < N) masks[e * row_words + c] = word;
      }
    }
  }
}

// The same for few samples: a block per product tile, its four waves sharing the steps, the
// operands read straight from global memory (the samples' from their encoded words) and the
// partial sums put together in LDS.
// PACK: the first score of a changed model, up to 32 samples (one tile), over all literals: the
// operands are made from the include masks here and kept, the weights' by the blocks past the
// tiles, so that nothing reads them back and there is a launch less (20000 literals, 10000
// clauses, one sample: 43 us of pack_model_kernel, 27 here and 7 of votes, 68 us with their gaps,
// against 55 so; 784 bits, 2000 clauses: the call 51 -> 47 us).
template <bool PACK>
__global__ __launch_bounds__(256) void fire_few_kernel(const uint32_t* __restrict__ X, int64_t N, Geom g,
                                                       const uint32_t* __restrict__ planes,
                                                       const float* __restrict__ w, unsigned char* __restrict__ base,
                                                       MatrixPlan p, uint32_t* __restrict__ masks) {
  __shared__ float s_d[3][16][kWave];
  __shared__ int s_count[4][kWave];
  const int steps = p.steps;
  const int64_t row_words = p.row_words;
  v4i* cfrag = (v4i*)base;
  float* need = (float*)(base + p.need_at);
  const int lane = lane_id(), wave = threadIdx.x / kWave;
  const int64_t mtiles = (N + kTile - 1) / kTile, ctiles = (g.C + kTile - 1) / kTile;
  const int64_t mt = blockIdx.x % mtiles, ct = blockIdx.x / mtiles;
  if (ct >= ctiles) {
    if (PACK) pack_weights(w, g, p, (v4i*)(base + p.weights_at), blockIdx.x - ctiles, gridDim.x - ctiles);
    return;
  }
  const int64_t e = mt * kTile + (lane & 31) < N ? mt * kTile + (lane & 31) : N - 1;
  const uint32_t* x = X + e * g.W;
  v4i* cf = cfrag + ct * steps * kWave + lane;
  v16f d;
#pragma unroll
  for (int r = 0; r < 16; ++r) d[r] = wave == 0 ? 1.0f : 0.0f;
  const int64_t c = ct * kTile + (lane & 31);
  const uint32_t* m = planes + ((c < g.C ? c : g.C - 1) * g.np + g.np - 1) * g.W;
  int count = 0;  // PACK: the lane's share of its clause's included literals
  float want = PACK ? 0.0f : need[c];
  constexpr int kAhead = 4;  // operands in flight
  for (int s0 = wave; s0 < steps; s0 += 4 * kAhead) {
    uint32_t xw[kAhead];
    v4i bv[kAhead];
#pragma unroll
    for (int q = 0; q < kAhead; ++q) {
      const int st = s0 + 4 * q < steps ? s0 + 4 * q : steps - 1;  // clamped: every load unconditional
      const int64_t w = 2 * st + (lane >> 5);
      xw[q] = x[w < g.W ? w : g.W - 1];  // past the words the clause operand is 0
      if (PACK) {
        const uint32_t on = c < g.C && s0 + 4 * q < steps && w < g.W ? m[w] : 0u;
        count += __popc(on);
        bv[q] = fp4_column(on, 0u);
      } else {
        bv[q] = cf[st * kWave];
      }
    }
#pragma unroll
    for (int q = 0; q < kAhead; ++q)
      if (s0 + 4 * q < steps) {
        d = fp4_product(fp4_row(xw[q]), bv[q], d);
        if (PACK) cf[(s0 + 4 * q) * kWave] = bv[q];
      }
  }
  if (PACK) s_count[wave][lane] = count;
  if (wave > 0)
#pragma unroll
    for (int r = 0; r < 16; ++r) s_d[wave - 1][r][lane] = d[r];
  __syncthreads();
  if (wave > 0) return;
#pragma unroll
  for (int r = 0; r < 16; ++r) d[r] += s_d[0][r][lane] + s_d[1][r][lane] + s_d[2][r][lane];
  if (PACK) {  // the threshold as pack_model_kernel makes it
    int n = 0;
#pragma unroll
    for (int q = 0; q < 4; ++q) n += s_count[q][lane] + s_count[q][lane ^ 32];
    want = n ? (float)(n + 1) : kNever;
    if (lane < kTile) need[c] = want;
  }
  const uint32_t word = row_words_of(d, want);
  if (lane < kTile && mt * kTile + lane < N) masks[(mt * kTile + lane) * row_words + ct] = word;
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
                                                                float* __restrict__ out, int* __restrict__ odd) {
  __shared__ int s_sum[kVoteWaves][kTile][kTile];  // [wave][sample][column]
  if (blockIdx.x == 0 && blockIdx.y == 0 && threadIdx.x == 0) *odd = 0;  // for the next samples
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
    bad = bad || !complements(X + idx / hw * g.W, g, idx % hw);
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

// Bytes of the firing words of N samples, before the samples' operands.
size_t rows_room(const MatrixPlan& p, int64_t N) { return ((size_t)N * p.row_words * 4 + 255) & ~(size_t)255; }

}  // namespace

size_t matrix_rows_bytes(const MatrixPlan& p, int64_t N) {
  return rows_room(p, N) + (size_t)((N + kTile - 1) / kTile * kTile) * p.sample_bytes;
}

hipError_t launch_halves_check(const uint32_t* X, int64_t N, const Geom& g, int* ok, hipStream_t s) {
  halves_kernel<<<blocks_for(N * g.P * ((g.Lh + 31) / 32), 256), 256, 0, s>>>(X, N * g.P, g, ok);
  return hipGetLastError();
}

bool long_rows(const Geom& g, int64_t N) {
  return (N + kTile - 1) / kTile * clause_tiles(g) * ((g.L + kStep - 1) / kStep) > (4 << 20);
}

bool few_rows(const Geom& g, int64_t N) { return (N + kTile - 1) / kTile * clause_tiles(g) <= 2048; }

MatrixPlan matrix_plan(const Geom& g, int halves, double w_bound, int64_t N) {
  MatrixPlan p{};
  const int64_t tiles = clause_tiles(g);
  if (tiles > (1 << 19)) return p;
  p.ternary = halves == 1 && g.append_negated;
  auto steps_of = [](int64_t n) { return (n + kStep - 1) / kStep; };
  const int64_t steps = steps_of(p.ternary ? g.Lh : g.L);
  if (g.P > 1) {
    if (steps > kMaxSteps) return p;
    p.steps = (int)steps;
  } else {
    // Up to 32 clauses of up to 512 literals, the register tiles of samples take less than the
    // operands' passes (100000 samples, 10 clauses of 32 literals: 13 against 31 us; 32 clauses:
    // 21 against 31, of 512: 40 against 37; 64 clauses: 32 and 59 against 33 and 39).
    if (steps > (1 << 16) || (g.W <= 16 && g.C <= 32)) return p;
    auto even = [](int64_t n) { return (int)((n + kRowSteps - 1) / kRowSteps * kRowSteps); };
    p.steps = even(steps);
    p.sample_bytes = (size_t)p.steps * kFragBytes / kTile;
    if (halves < 0 && g.append_negated && !few_rows(g, N)) p.half_steps = even(steps_of(g.Lh));
  }
  p.row_words = (tiles + 3) / 4 * 4;
  // digits that hold every weight of magnitude up to w_bound
  double top = 127.0;
  for (p.digits = 1; top < w_bound && p.digits < 5; ++p.digits) top = top * 256.0 + 127.0;
  const int per = kTile / p.digits;
  p.groups = (int)((g.K + per - 1) / per);
  auto room = [](size_t n) { return (n + 255) & ~(size_t)255; };
  p.half_at = room((size_t)tiles * p.steps * kFragBytes);
  p.need_at = p.half_at + room((size_t)tiles * p.half_steps * kFragBytes);
  p.flag_at = p.need_at + room((size_t)tiles * kTile * 4 * (p.half_steps ? 2 : 1));
  p.weights_at = p.flag_at + 256;
  p.bytes = p.weights_at + (size_t)(p.row_words * p.groups) * kFragBytes;
  return p;
}

hipError_t launch_matrix_score(const uint32_t* planes, const float* w, bool ready, const uint32_t* X, int64_t N,
                               const Geom& g, const MatrixPlan& p, void* scratch, int cus, const float* bias,
                               uint32_t* masks, float* out, hipStream_t s) {
  if (N == 0) return hipSuccess;
  unsigned char* base = (unsigned char*)scratch;
  int* flag = (int*)(base + p.flag_at);
  const v4i* frag = (const v4i*)base;
  const float* need = (const float*)(base + p.need_at);
  hipError_t e = hipSuccess;
  const int64_t mtiles = (N + kTile - 1) / kTile, ctiles = clause_tiles(g);
  const bool few = g.P == 1 && few_rows(g, N), pack_few = few && !ready && mtiles == 1 && !p.half_steps && !p.ternary;
  const int weight_blocks = blocks_for(p.row_words * p.groups * kWave, 256);
  if (!ready && !pack_few) {
    const int need_blocks = blocks_for(ctiles * kTile * kWave, 256);
    pack_model_kernel<<<need_blocks + weight_blocks + blocks_for(ctiles * (p.steps + p.half_steps) * kWave, 256), 256, 0,
                        s>>>(planes, w, g, p, base, need_blocks, weight_blocks);
    e = hipGetLastError();
    if (e != hipSuccess) return e;
  }
  if (pack_few) {
    fire_few_kernel<true><<<(unsigned)ctiles + weight_blocks, 256, 0, s>>>(X, N, g, planes, w, base, p, masks);
    e = hipGetLastError();
  } else if (few) {
    fire_few_kernel<false><<<(unsigned)(mtiles * ctiles), 256, 0, s>>>(X, N, g, planes, w, base, p, masks);
    e = hipGetLastError();
  } else if (g.P == 1) {
    v4i* sfrag = (v4i*)((unsigned char*)masks + rows_room(p, N));
    pack_samples_kernel<<<blocks_for(mtiles * p.steps * kWave, 256), 256, 0, s>>>(X, N, g, p.steps, p.half_steps, flag, sfrag);
    const int64_t blocks = ((mtiles + kBlockTiles - 1) / kBlockTiles) * ((ctiles + kBlockTiles - 1) / kBlockTiles);
    const size_t lds = (size_t)kRowBuffers * 2 * kBlockTiles * kRowSteps * kFragBytes;
    fire_rows_kernel<<<(unsigned)std::min<int64_t>((blocks + 7) / 8 * 8, 1 << 22), 512, lds, s>>>(
        sfrag, N, g.C, base, p, masks);
    e = hipGetLastError();
  } else switch (p.steps) {
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
      masks, p.row_words, N, (const v4i*)(base + p.weights_at), g, p.digits, p.groups, bias, out, flag);
  return hipGetLastError();
}

}  // namespace ytm
