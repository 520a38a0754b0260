// Products of any layout on gfx950 matrix cores: the general path's kernel for
// products large enough to be worth reordering (smaller ones, and every one
// under policy 1, keep k_matmul_general, which sums in the shader's order).
//
// Any op-2 plan (src/alelyon_compute_kit/_kit/kernels/vq4.comp:165-176): A
// packed or dense, either operand stored either way, any sizes, vectors that
// straddle rows. Both operands are decoded into three bf16 terms hi + mid + lo
// (24 bits: each term the rounding of what the previous ones leave, exact for
// values of at least 2^-103) and multiplied as the six products that reach
// 2^-27 of the whole: hi hi, hi mid, mid hi, mid mid, hi lo, lo hi. FP32
// accumulation then rounds 6 times per 16 inner indices, against 32 in the
// shader's loop. FP32 MFMA would need one product but has 1/16 of the rate.
//
// A block owns BM rows x 128 columns and a slice of k, staged 32 inner indices
// at a time through LDS in the MFMA's fragment order, [term][8 indices][row]:
// each thread decodes 8 consecutive indices of a row or column at a time and
// writes 16 bytes per term. The next stage's codes or values are loaded while
// this one is multiplied. Packed operands are split once per block, as books:
//   - rows along k whose length is a multiple of 8: the 8 indices lie in one
//     vector, so a term is a 16-byte copy from the book's plane;
//   - otherwise each index is one 8-byte read of {hi, mid, lo}.
// Dense values are split as they are staged (~6 operations a value).
//
// What bounds it: LDS traffic (the fragments' reads and the books' gathers, about
// 250 KB per 128 x 128 x 32 stage against 1,540 matrix cycles a wave) on large
// products, the loads' latency and the second launch on small ones.
//
// Grids of fewer than kGeneralBlocks blocks cut k into slices. They run side by
// side, their sums go to the workspace and k_sum_slices adds them in slice order;
// or, in batches that fill the chip and where there is no workspace, each block
// walks the slices and adds their sums in the same order in the output. The slices
// are those of the product alone, so neither changes a bit.
#include <hip/hip_runtime.h>

#include <cfloat>
#include <cstdint>

#include "kernels.hpp"

namespace ackvq {
namespace {

typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

constexpr uint32_t kThreads = 256;
constexpr uint32_t kTileN = 128;       // columns of a block
constexpr uint32_t kStageK = 32;       // inner indices per stage
constexpr uint32_t kChunks = kStageK / 8;
constexpr int kTerms = 3;
constexpr uint32_t kGeneralBlocks = 512;
constexpr uint64_t kPartialBytes = uint64_t(8) << 20;  // of one product's slices

// How an operand of R rows (A) or columns (B) lies in memory.
enum Source : int {
  kDenseAlongK = 0,    // float32, index r * k + kk
  kDenseAlongR = 1,    // float32, index kk * R + r
  kPackedAlongK = 2,   // codes of that order
  kPackedAlongR = 3,
};

__device__ __forceinline__ bool finite_f32(float x) { return fabsf(x) <= FLT_MAX; }

template <typename T>
__device__ __forceinline__ const T* item_ptr(const void* base, uint64_t stride, uint32_t item) {
  return reinterpret_cast<const T*>(static_cast<const char*>(base) + stride * item);
}

// Two values as three pairs of bf16 terms, the first value in the low halves.
// hi is the rounding of the value clamped to the largest bf16, so that a
// finite value past it still splits; an infinity or NaN leaves a NaN term.
struct Split2 {
  uint32_t term[kTerms];
};
__device__ __forceinline__ Split2 split2(float a, float b) {
  constexpr float kTop = 3.3895313892515355e38f;  // the largest bf16
  Split2 s;
  float x = fminf(fmaxf(a, -kTop), kTop), y = fminf(fmaxf(b, -kTop), kTop);
  bf16x2 p = {__bf16(x), __bf16(y)};
  s.term[0] = __builtin_bit_cast(uint32_t, p);
  float r = a - __uint_as_float(s.term[0] << 16), t = b - __uint_as_float(s.term[0] & 0xFFFF0000u);
  p = bf16x2{__bf16(r), __bf16(t)};
  s.term[1] = __builtin_bit_cast(uint32_t, p);
  r -= __uint_as_float(s.term[1] << 16);
  t -= __uint_as_float(s.term[1] & 0xFFFF0000u);
  p = bf16x2{__bf16(r), __bf16(t)};
  s.term[2] = __builtin_bit_cast(uint32_t, p);
  return s;
}

// The exponent e of a book's largest finite magnitude, below 2^e.
__device__ __forceinline__ int book_exponent(const float* book, uint32_t entries) {
  float top = 0.0f;
  for (uint32_t i = threadIdx.x % 64; i < entries; i += 64) {
    const float v = fabsf(book[i]);
    top = v <= FLT_MAX ? fmaxf(top, v) : top;
  }
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) top = fmaxf(top, __shfl_xor(top, off));
  int e = 0;
  if (top > 0.0f) (void)frexpf(top, &e);
  return e;
}

// The power of two each book is scaled by: up to 2^-60 where its entries are so
// small that their last terms would be subnormal, and packed A down by 2^8 where the
// products come near FP32's end, which a sum of hi terms may pass by 2^-8 when the
// product does not. Never by a book's largest entry: no code may use it, and those
// that codes do use would lose their last terms.
struct Shifts {
  int a, b;
};
template <bool AD>
__device__ __forceinline__ Shifts book_shifts(const float* a_book, const float* b_book,
                                              uint32_t entries) {
  const int eb = book_exponent(b_book, entries), sb = eb < -60 ? -60 - eb : 0;
  if constexpr (AD) return {0, sb};
  const int ea = book_exponent(a_book, entries);
  return {ea < -60 ? -60 - ea : ea + eb > 100 ? -8 : 0, sb};
}

// A packed operand's book, scaled and split: planes for 16-byte copies along a
// vector, words {hi | mid << 16, lo} for single values.
struct __align__(16) BookTable {
  __bf16 plane[kTerms][16 * 32];
  uint2 word[16 * 32];
};

__device__ __forceinline__ void fill_table(BookTable& t, const float* book, uint32_t entries,
                                           int shift) {
  for (uint32_t i = 2 * threadIdx.x; i < entries; i += 2 * kThreads) {
    const Split2 s = split2(ldexpf(book[i], shift), ldexpf(book[i + 1], shift));
#pragma unroll
    for (int x = 0; x < kTerms; ++x) *reinterpret_cast<uint32_t*>(&t.plane[x][i]) = s.term[x];
    t.word[i] = make_uint2(s.term[0] & 0xFFFFu | s.term[1] << 16, s.term[2] & 0xFFFFu);
    t.word[i + 1] = make_uint2(s.term[0] >> 16 | s.term[1] & 0xFFFF0000u, s.term[2] >> 16);
  }
}

// One operand's staged tile: row r's 8 indices of chunk c are 16 bytes at
// [c][r] of each term; the chunks are two rows apart in banks so that threads
// walking the chunks of a row do not conflict.
template <uint32_t R>
struct __align__(16) Tile {
  uint4 v[kTerms][kChunks][R + 2];
};

// The code of flat index `flat` in its word.
__device__ __forceinline__ uint32_t nibble(uint32_t word, uint32_t flat, uint32_t lg) {
  return __builtin_amdgcn_ubfe(word, flat >> (lg - 2) & 28u, 4);
}

// One thread's loads for one stage: `kTasks` chunks of 8 indices.
template <int SRC, uint32_t R>
struct Loader {
  static constexpr uint32_t kTasks = (R * kChunks + kThreads - 1) / kThreads;
  static constexpr int kRaw = SRC == kPackedAlongK ? 2 : 8;
  uint32_t raw[kTasks][kRaw];

  // task -> (row, chunk): along the memory's fast direction
  static __device__ __forceinline__ uint32_t row(uint32_t id) {
    return SRC == kDenseAlongK || SRC == kPackedAlongK ? id / kChunks : id % R;
  }
  static __device__ __forceinline__ uint32_t chunk(uint32_t id) {
    return SRC == kDenseAlongK || SRC == kPackedAlongK ? id % kChunks : id / R;
  }
  static __device__ __forceinline__ bool idle(uint32_t id) {
    return R * kChunks % kThreads != 0 && id >= R * kChunks;
  }

  // Rows past the operand read its last row; indices past k read index k - 1
  // and are zeroed when they are staged (TAIL: a stage that reaches past the
  // slice). Words are kept as loaded: their codes are taken in stage(), so that
  // nothing waits for the load before the multiplication it overlaps.
  template <bool TAIL>
  __device__ __forceinline__ void load(const void* base, uint32_t r0, uint32_t rows, uint32_t k0,
                                       uint32_t k, uint32_t lg) {
    const uint32_t* words = static_cast<const uint32_t*>(base);
#pragma unroll
    for (uint32_t x = 0; x < kTasks; ++x) {
      const uint32_t id = threadIdx.x + x * kThreads;
      if (idle(id)) continue;
      uint32_t r = r0 + row(id);
      r = r < rows ? r : rows - 1;
      const uint32_t kk = k0 + 8 * chunk(id);
      if constexpr (SRC == kPackedAlongK) {
        const uint32_t flat = r * k + (!TAIL || kk < k ? kk : k - 1);
        const uint32_t last = (rows * k - 1) >> lg;  // the last vector
        const uint32_t v = flat >> lg, w = v < last ? v + 1 : last;
        raw[x][0] = words[v >> 3];
        raw[x][1] = words[w >> 3];
      } else if constexpr (SRC == kPackedAlongR) {
        uint32_t flat = kk * rows + r;
#pragma unroll
        for (uint32_t i = 0; i < 8; ++i, flat += rows)
          raw[x][i] = words[(!TAIL || kk + i < k ? flat : (k - 1) * rows + r) >> (lg + 3)];
      } else {
        // the largest dense operand has 2^28 values
        uint32_t at = SRC == kDenseAlongK ? r * k + kk : kk * rows + r;
        const uint32_t step = SRC == kDenseAlongK ? 1 : rows;
#pragma unroll
        for (uint32_t i = 0; i < 8; ++i, at += step)
          raw[x][i] = words[!TAIL || kk + i < k ? at
                            : SRC == kDenseAlongK ? r * k + k - 1 : (k - 1) * rows + r];
      }
    }
  }

  template <bool TAIL>
  __device__ __forceinline__ void stage(Tile<R>& tile, const BookTable& table, uint32_t r0,
                                        uint32_t rows, uint32_t k0, uint32_t k, uint32_t kend,
                                        uint32_t lg) const {
    const uint32_t mask = (1u << lg) - 1;
#pragma unroll
    for (uint32_t x = 0; x < kTasks; ++x) {
      const uint32_t id = threadIdx.x + x * kThreads;
      if (idle(id)) continue;
      uint32_t r = r0 + row(id);
      r = r < rows ? r : rows - 1;
      const uint32_t kk = k0 + 8 * chunk(id);
      uint4 t[kTerms];
      if (SRC == kPackedAlongK && (k & 7) == 0) {  // one vector: a copy per term
        const uint32_t flat = r * k + kk;
        const uint32_t at = nibble(raw[x][0], flat, lg) << lg | flat & mask;
#pragma unroll
        for (int s = 0; s < kTerms; ++s) {
          t[s] = *reinterpret_cast<const uint4*>(&table.plane[s][at]);
          if (TAIL && kk >= kend) t[s] = make_uint4(0, 0, 0, 0);
        }
      } else {
        uint32_t term[kTerms][4];
        uint32_t flat = SRC == kPackedAlongK ? r * k + kk : kk * rows + r;
        // along k, a chunk's first and second vector
        const uint32_t first = SRC == kPackedAlongK ? nibble(raw[x][0], flat, lg) << lg : 0;
        const uint32_t second =
            SRC == kPackedAlongK ? nibble(raw[x][1], flat + mask + 1, lg) << lg : 0;
        const uint32_t in = flat & mask;
#pragma unroll
        for (uint32_t i = 0; i < 8; i += 2) {
          if constexpr (SRC == kPackedAlongK || SRC == kPackedAlongR) {
            uint2 w[2];
#pragma unroll
            for (uint32_t y = 0; y < 2; ++y) {
              uint32_t at;
              if constexpr (SRC == kPackedAlongK) {
                at = (in + i + y > mask ? second : first) | (in + i + y) & mask;
              } else {
                // a tail index past k reads some entry, zeroed below
                at = nibble(raw[x][i + y], flat, lg) << lg | flat & mask;
                flat += rows;
              }
              w[y] = table.word[at];
              if (TAIL && kk + i + y >= kend) w[y] = make_uint2(0, 0);
            }
            term[0][i / 2] = __builtin_amdgcn_perm(w[1].x, w[0].x, 0x05040100u);
            term[1][i / 2] = __builtin_amdgcn_perm(w[1].x, w[0].x, 0x07060302u);
            term[2][i / 2] = __builtin_amdgcn_perm(w[1].y, w[0].y, 0x05040100u);
          } else {
            const float a = !TAIL || kk + i < kend ? __uint_as_float(raw[x][i]) : 0.0f;
            const float b = !TAIL || kk + i + 1 < kend ? __uint_as_float(raw[x][i + 1]) : 0.0f;
            const Split2 s = split2(a, b);
#pragma unroll
            for (int y = 0; y < kTerms; ++y) term[y][i / 2] = s.term[y];
          }
        }
#pragma unroll
        for (int s = 0; s < kTerms; ++s)
          t[s] = make_uint4(term[s][0], term[s][1], term[s][2], term[s][3]);
      }
#pragma unroll
      for (int s = 0; s < kTerms; ++s) tile.v[s][chunk(id)][row(id)] = t[s];
    }
  }
};

// grid: (ceil(n / 128), ceil(m / BM), instances * slices, or instances where the
// blocks walk the slices: WALK). The block's 4 waves lie 2 x 2 (BM 64
// and 128) or 1 x 4 (BM 32) over the tile.
template <int ASRC, int BSRC, uint32_t BM, bool WALK>
__global__ __launch_bounds__(kThreads, 2) void k_general_mfma(Operands o, uint32_t m, uint32_t n,
                                                              uint32_t k, uint32_t lg,
                                                              uint32_t slices, uint32_t slice_k,
                                                              float* partial) {
  constexpr bool kDenseA = ASRC == kDenseAlongK || ASRC == kDenseAlongR;
  constexpr uint32_t kWaveRows = BM == 32 ? 1 : 2;
  constexpr uint32_t X = BM / kWaveRows / 32, Y = kTileN / (4 / kWaveRows) / 32;
  __shared__ Tile<BM> at;
  __shared__ Tile<kTileN> bt;
  __shared__ BookTable ta, tb;
  const uint32_t lane = threadIdx.x % 64, wave = threadIdx.x / 64;
  const uint32_t i32 = lane % 32, h = lane / 32;
  const uint32_t m0 = blockIdx.y * BM, n0 = blockIdx.x * kTileN;
  const uint32_t wr = wave / (4 / kWaveRows) * (32 * X), wc = wave % (4 / kWaveRows) * (32 * Y);
  const uint32_t entries = 16u << lg;

  const uint32_t each = WALK ? slices : 1;  // slices of a block
  for (uint32_t z = blockIdx.z * each; z < o.count * slices; z += gridDim.z * each) {
    const uint32_t item = z / slices;
    uint32_t slice = z % slices;
    const void* a = item_ptr<char>(o.in[0], o.stride[0], item);
    const float* a_book = item_ptr<float>(o.in[1], o.stride[1], item);
    const void* b = item_ptr<char>(o.in[2], o.stride[2], item);
    const float* b_book = item_ptr<float>(o.in[3], o.stride[3], item);
    uint32_t kbeg = slice * slice_k, kend = k - kbeg < slice_k ? k : kbeg + slice_k;

    // loads run kAhead stages ahead; the 128-row tile has no registers for two
    constexpr uint32_t kAhead = BM == 128 ? 1 : 2;
    Loader<ASRC, BM> la[kAhead];
    Loader<BSRC, kTileN> lb[kAhead];
    auto load = [&](Loader<ASRC, BM>& x, Loader<BSRC, kTileN>& y, uint32_t k0) {
      if (k0 >= kend) return;
      // sizes the compiler cannot see through: it would keep every load's
      // address of the loop in registers, which the accumulators need
      uint32_t ms = m, ns = n;
      asm volatile("" : "+s"(ms), "+s"(ns));
      if (k0 + kStageK <= k) {
        x.template load<false>(a, m0, ms, k0, k, lg);
        y.template load<false>(b, n0, ns, k0, k, lg);
      } else {
        x.template load<true>(a, m0, ms, k0, k, lg);
        y.template load<true>(b, n0, ns, k0, k, lg);
      }
    };
#pragma unroll
    for (uint32_t x = 0; x < kAhead; ++x) load(la[x], lb[x], kbeg + x * kStageK);
    const Shifts shift = book_shifts<kDenseA>(a_book, b_book, entries);
    bool bad = false;
    if (blockIdx.x == 0 && blockIdx.y == 0 && slice == 0)
      for (uint32_t i = threadIdx.x; i < entries; i += kThreads)
        bad |= !finite_f32(b_book[i]) || (!kDenseA && !finite_f32(a_book[i]));
    __syncthreads();  // the previous instance's tables are no longer read
    if constexpr (!kDenseA) fill_table(ta, a_book, entries, shift.a);
    fill_table(tb, b_book, entries, shift.b);
    f32x16 acc[X][Y];
    __syncthreads();

    auto step = [&](Loader<ASRC, BM>& x, Loader<BSRC, kTileN>& y, uint32_t k0) {
      uint32_t ms = m, ns = n;
      asm volatile("" : "+s"(ms), "+s"(ns));
      if (k0 + kStageK <= kend) {
        x.template stage<false>(at, ta, m0, ms, k0, k, kend, lg);
        y.template stage<false>(bt, tb, n0, ns, k0, k, kend, lg);
      } else {
        x.template stage<true>(at, ta, m0, ms, k0, k, kend, lg);
        y.template stage<true>(bt, tb, n0, ns, k0, k, kend, lg);
      }
      __syncthreads();
      load(x, y, k0 + kAhead * kStageK);
#pragma unroll
      for (uint32_t s = 0; s < kChunks; s += 2) {
        bf16x8 fa[X][kTerms], fb[Y][kTerms];
#pragma unroll
        for (int t = 0; t < kTerms; ++t) {
#pragma unroll
          for (uint32_t x = 0; x < X; ++x)
            fa[x][t] = __builtin_bit_cast(bf16x8, at.v[t][s + h][wr + 32 * x + i32]);
#pragma unroll
          for (uint32_t y = 0; y < Y; ++y)
            fb[y][t] = __builtin_bit_cast(bf16x8, bt.v[t][s + h][wc + 32 * y + i32]);
        }
        constexpr int kPairs[6][2] = {{2, 0}, {0, 2}, {1, 1}, {1, 0}, {0, 1}, {0, 0}};
#pragma unroll
        for (int p = 0; p < 6; ++p)
#pragma unroll
          for (uint32_t x = 0; x < X; ++x)
#pragma unroll
            for (uint32_t y = 0; y < Y; ++y)
              acc[x][y] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
                  fa[x][kPairs[p][0]], fb[y][kPairs[p][1]], acc[x][y], 0, 0, 0);
      }
      __syncthreads();
    };
    const bool direct = WALK || slices == 1;
    float* out = direct ? reinterpret_cast<float*>(static_cast<char*>(o.out) + o.stride[4] * item)
                        : partial + uint64_t(z) * m * n;
    const int up = -(shift.a + shift.b);
    for (uint32_t left = each;;) {
#pragma unroll
      for (uint32_t x = 0; x < X; ++x)
#pragma unroll
        for (uint32_t y = 0; y < Y; ++y) acc[x][y] = (f32x16)0.0f;
      for (uint32_t k0 = kbeg; k0 < kend; k0 += kAhead * kStageK)
#pragma unroll
        for (uint32_t x = 0; x < kAhead; ++x)
          if (k0 + x * kStageK < kend) step(la[x], lb[x], k0 + x * kStageK);

      uint32_t rows = m, columns = n;  // as above: not 64 bounds tests kept over the loop
      asm volatile("" : "+s"(rows), "+s"(columns));
      const bool last = direct && (!WALK || left == 1);
#pragma unroll
      for (uint32_t x = 0; x < X; ++x)
#pragma unroll
        for (uint32_t y = 0; y < Y; ++y)
#pragma unroll
          for (uint32_t t = 0; t < 16; ++t) {
            const uint32_t r = m0 + wr + 32 * x + (t % 4) + 4 * h + 8 * (t / 4);
            const uint32_t c = n0 + wc + 32 * y + i32;
            if (r < rows && c < columns) {
              float* at = out + uint64_t(r) * columns + c;
              float v = ldexpf(acc[x][y][t], up);
              if (WALK) v = (slice > 0 ? *at : 0.0f) + v;
              *at = v;
              bad |= last && !finite_f32(v);
            }
          }
      if (!WALK || --left == 0) break;
      ++slice;
      kbeg = kend;
      kend = k - kbeg < slice_k ? k : kbeg + slice_k;
#pragma unroll
      for (uint32_t x = 0; x < kAhead; ++x) load(la[x], lb[x], kbeg + x * kStageK);
    }
    if (__any(bad) && lane == 0) atomicOr(o.status, 1u);
  }
}

// out = the slices' sums, added in slice order. grid: (ceil(m n / 256), instances).
__global__ __launch_bounds__(256) void k_sum_slices(Operands o, uint32_t mn, uint32_t slices,
                                                        const float* partial) {
  const uint32_t i = blockIdx.x * 256 + threadIdx.x;
  const uint32_t at = i < mn ? i : mn - 1;
  for (uint32_t item = blockIdx.y; item < o.count; item += gridDim.y) {
    const float* p = partial + uint64_t(item) * slices * mn + at;
    float sum = 0.0f;
    uint32_t s = 0;
    for (; s + 4 <= slices; s += 4) {
      float v[4];
#pragma unroll
      for (uint32_t x = 0; x < 4; ++x) v[x] = p[uint64_t(s + x) * mn];
#pragma unroll
      for (uint32_t x = 0; x < 4; ++x) sum += v[x];
    }
    for (; s < slices; ++s) sum += p[uint64_t(s) * mn];
    const bool live = i < mn;
    if (live)
      reinterpret_cast<float*>(static_cast<char*>(o.out) + o.stride[4] * item)[i] = sum;
    if (__any(live && !finite_f32(sum)) && threadIdx.x % 64 == 0) atomicOr(o.status, 1u);
  }
}

struct GeneralGrid {
  uint32_t bm, gx, gy, slices, slice_k;
};

// The slices of one product, whatever batch it is in: 128-row blocks where they
// (times their slices) fill the chip, else 64-row ones, 32 for fewer rows. In a
// batch the blocks may be larger, which changes no sum.
GeneralGrid general_grid(uint32_t m, uint32_t n, uint32_t k, uint32_t count) {
  const uint64_t stages = (k + kStageK - 1) / kStageK;
  const uint64_t room = kPartialBytes / (uint64_t(m) * n * 4);
  const uint32_t most = m <= 32 ? 32 : m <= 64 ? 64 : 128;
  GeneralGrid g;
  uint64_t slices = 1;
  g.gx = (n + kTileN - 1) / kTileN;
  for (g.bm = most;; g.bm = 64) {
    g.gy = (m + g.bm - 1) / g.bm;
    const uint64_t blocks = uint64_t(g.gx) * g.gy;
    slices = (kGeneralBlocks + blocks - 1) / blocks;
    if (slices > room) slices = room;
    if (slices > stages / 2) slices = stages / 2;
    if (slices < 1) slices = 1;
    if (g.bm <= 64 || blocks * slices >= kGeneralBlocks / 2) break;
  }
  g.slice_k = uint32_t((stages + slices - 1) / slices) * kStageK;
  g.slices = (k + g.slice_k - 1) / g.slice_k;
  if (g.bm < most && uint64_t(g.gx) * ((m + most - 1) / most) * count >= kGeneralBlocks / 2) {
    g.bm = most;
    g.gy = (m + most - 1) / most;
  }
  return g;
}

template <int ASRC, int BSRC, uint32_t BM>
void run_general_rows(hipStream_t s, const Operands& o, uint32_t m, uint32_t n, uint32_t k,
                      uint32_t lg, const GeneralGrid& g, float* partial) {
  const bool walk = partial == nullptr && g.slices > 1;
  const uint64_t z = uint64_t(o.count) * (walk ? 1 : g.slices);
  const dim3 grid(g.gx, g.gy, z < 65535 ? uint32_t(z) : 65535u);
  if (walk)
    k_general_mfma<ASRC, BSRC, BM, true><<<grid, kThreads, 0, s>>>(o, m, n, k, lg, g.slices,
                                                                   g.slice_k, partial);
  else
    k_general_mfma<ASRC, BSRC, BM, false><<<grid, kThreads, 0, s>>>(o, m, n, k, lg, g.slices,
                                                                    g.slice_k, partial);
}

template <int ASRC, int BSRC>
void run_general(hipStream_t s, const Operands& o, uint32_t m, uint32_t n, uint32_t k, uint32_t lg,
                 const GeneralGrid& g, float* partial) {
  if (g.bm == 32) run_general_rows<ASRC, BSRC, 32>(s, o, m, n, k, lg, g, partial);
  else if (g.bm == 64) run_general_rows<ASRC, BSRC, 64>(s, o, m, n, k, lg, g, partial);
  else run_general_rows<ASRC, BSRC, 128>(s, o, m, n, k, lg, g, partial);
}

template <int ASRC>
void run_general_b(hipStream_t s, const Operands& o, uint32_t m, uint32_t n, uint32_t k,
                   uint32_t lg, uint32_t flags, const GeneralGrid& g, float* partial) {
  if (flags & 2u) run_general<ASRC, kPackedAlongK>(s, o, m, n, k, lg, g, partial);
  else run_general<ASRC, kPackedAlongR>(s, o, m, n, k, lg, g, partial);
}

}  // namespace

void launch_sum_slices(hipStream_t s, const Operands& o, uint32_t mn, uint32_t slices,
                       const float* partial) {
  const dim3 grid((mn + 255) / 256, o.count < 65535 ? o.count : 65535);
  k_sum_slices<<<grid, 256, 0, s>>>(o, mn, slices, partial);
}

size_t general_workspace_bytes(uint32_t m, uint32_t n, uint32_t k, uint32_t count) {
  const GeneralGrid g = general_grid(m, n, k, count);
  const size_t bytes = size_t(m) * n * 4 * count * g.slices;
  const bool walk = g.slices == 1 || uint64_t(g.gx) * g.gy * count >= kGeneralBlocks ||
                    bytes > kBatchPartialBytes;
  return walk ? 0 : bytes;
}

hipError_t launch_general_mfma(hipStream_t s, const Operands& o, uint32_t m, uint32_t n, uint32_t k,
                               uint32_t group, uint32_t flags, bool dense, void* workspace) {
  const GeneralGrid g = general_grid(m, n, k, o.count);
  const uint32_t lg = group == 8 ? 3 : group == 16 ? 4 : 5;
  float* partial =
      general_workspace_bytes(m, n, k, o.count) == 0 ? nullptr : static_cast<float*>(workspace);
  if (dense) {
    if (flags & 1u) run_general_b<kDenseAlongR>(s, o, m, n, k, lg, flags, g, partial);
    else run_general_b<kDenseAlongK>(s, o, m, n, k, lg, flags, g, partial);
  } else {
    if (flags & 1u) run_general_b<kPackedAlongR>(s, o, m, n, k, lg, flags, g, partial);
    else run_general_b<kPackedAlongK>(s, o, m, n, k, lg, flags, g, partial);
  }
  if (partial != nullptr) launch_sum_slices(s, o, m * n, g.slices, partial);
  return hipGetLastError();
}

}  // namespace ackvq
