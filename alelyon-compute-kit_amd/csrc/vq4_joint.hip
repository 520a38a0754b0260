// Packed products with both operands grouped along the output's sides, on
// gfx950 matrix cores: "joint-mfma".
//
// With A stored (k, m) and B stored (k, n) (op 2, flags 1 of
// src/alelyon_compute_kit/_kit/kernels/vq4.comp:165-176 -- the X^T . dY of a
// weight gradient), m and n multiples of the group G, row ig*G + s of A and
// column jg*G + t of B lie in one vector per inner index, so
//   C[ig*G+s][jg*G+t] = sum_e sum_f C_A[e][s] * H[ig][jg][e][f] * C_B[f][t],
//   H[ig][jg][e][f]   = #{kk : a(kk, ig) = e and b(kk, jg) = f}.
// H is a product of two one-hot matrices of 16 m/G and 16 n/G columns over k:
// its operands are exact in 4-bit floats and its sums are whole numbers up to
// 65,536, exact in FP32. Two 16-term FP32 products per output follow, so an
// output carries ~32 roundings whatever k is (the shader's loop has 2 k).
//
// The counts run on v_mfma_f32_16x16x128_f8f6f4 with FP4 operands: one block
// is one (ig, jg) pair, rows e, columns f. A lane's 32 inner indices are 32
// nibbles in four words, which is how the codes already lie once they are
// transposed (k_joint_words), so its one-hot row is each word XOR-ed with the
// lane's code in every nibble and the zero nibbles marked: 2.0 is the nibble
// 0x4, and the products' 4.0 is divided out with the books' scale. An element
// costs 1/8 of 5 integer operations; a bf16 one-hot would cost four times as
// many and half the matrix rate.
//
// The two products with the books take the counts from their registers: on
// v_mfma_f32_16x16x4f32 a result register of one product is an operand
// register of the next (lane l holds rows 4(l/16) + r and column l%16 of a
// result, and inner index l/16 and side l%16 of an operand), so nothing goes
// through LDS or memory, and the last product is taken transposed so that a
// lane ends with four adjacent columns of one row, one 16-byte store.
//
// What bounds it: the two book products (FP32 matrix rate, 32 cycles per 256
// outputs and instruction) and the output's writes; past k ~ 1024 the counts'
// one-hot rows. 4096 x 14336, k = 2048: 71 us at group 32 (235 MB written, 34
// us at this card's fill rate), 131 at 16, 437 at 8, against 5,435 us on the
// general kernel; 4096 x 4096, k = 32 at group 16: 19.4 against 34 us. Errors
// against a float64 product: 1e-7 of its norm at every k measured (8 to 2048);
// the general kernel's grow from 6e-8 to 1.2e-6.
#include <hip/hip_runtime.h>

#include <cfloat>
#include <cstdint>

#include "kernels.hpp"

namespace ackvq {
namespace {

typedef int i32x4 __attribute__((ext_vector_type(4)));
typedef int i32x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

constexpr uint32_t kJointThreads = 256;  // 4 waves, 2 x 2 over the block's pairs
constexpr uint32_t kJointStep = 128;     // inner indices per MFMA
// Up to this k the blocks transpose their own codes: the pre-pass's launch and
// its ~4 us outweigh the repeated reads (4096 x 4096 at group 16: k = 32 19.4
// against 22.3 us, 256 22.5 against 23.8, 512 27.8 against 26.7; 4096 x 14336,
// k = 2048 185 against 131). So they do without a workspace for the transposed
// codes; the counts are whole numbers, so the outputs have the same bits.
constexpr uint32_t kJointGather = 256;
constexpr int kFp4 = 4;                  // the instruction's code for e2m1 operands

__device__ __forceinline__ bool finite_f32(float x) { return fabsf(x) <= FLT_MAX; }

template <typename T>
__device__ __forceinline__ const T* item_ptr(const void* base, uint64_t stride, uint32_t item) {
  return reinterpret_cast<const T*>(static_cast<const char*>(base) + stride * item);
}

__host__ __device__ inline uint32_t padded_k(uint32_t k) {
  return (k + kJointStep - 1) / kJointStep * kJointStep;
}

// The codes of one operand with the inner index along the nibbles of a word:
// out[v * kp / 8 + w] holds vector column v's codes of inner indices 8w ..
// 8w + 7, zero past k. One thread per column and 32 indices; the columns of a
// wave read neighbouring nibbles of each row.
__device__ __forceinline__ void transpose_words(const uint32_t* codes, uint32_t columns, uint32_t k,
                                                uint32_t v, uint32_t w4, uint32_t words,
                                                uint32_t* out) {
  uint32_t word[4] = {0, 0, 0, 0};
#pragma unroll
  for (uint32_t i = 0; i < 32; ++i) {  // rows past k read the last one: no load waits on a branch
    const uint32_t kk = 32 * w4 + i;
    const uint64_t flat = uint64_t(kk < k ? kk : k - 1) * columns + v;
    const uint32_t code = codes[flat >> 3] >> (4 * uint32_t(flat & 7)) & 15u;
    word[i / 8] |= (kk < k ? code : 0u) << (4 * (i % 8));
  }
  *reinterpret_cast<uint4*>(out + uint64_t(v) * words + 4 * w4) =
      make_uint4(word[0], word[1], word[2], word[3]);
}

// grid: (column blocks of 64, kp / 32 / 4, instances); A's columns, then B's.
__global__ __launch_bounds__(256) void k_joint_words(Operands o, uint32_t va, uint32_t vb,
                                                     uint32_t k, uint32_t* workspace) {
  const uint32_t words = padded_k(k) / 8;
  const uint32_t w4 = blockIdx.y * 4 + threadIdx.x / 64;
  const uint32_t v = blockIdx.x * 64 + threadIdx.x % 64;
  if (4 * w4 >= words || v >= va + vb) return;
  for (uint32_t item = blockIdx.z; item < o.count; item += gridDim.z) {
    uint32_t* base = workspace + uint64_t(item) * (va + vb) * words;
    if (v < va)
      transpose_words(item_ptr<uint32_t>(o.in[0], o.stride[0], item), va, k, v, w4, words, base);
    else
      transpose_words(item_ptr<uint32_t>(o.in[2], o.stride[2], item), vb, k, v - va, w4, words,
                      base + uint64_t(va) * words);
  }
}

// A lane's 32 one-hot FP4 values: 2.0 where the nibble equals its code (`same`
// holds the code in every nibble). (x | 8s) - 1s keeps bit 3 of a nibble
// exactly when its low three bits are not all zero, with no borrow between
// nibbles.
__device__ __forceinline__ i32x8 one_hot(i32x4 w, uint32_t same) {
  i32x8 r = {0, 0, 0, 0, 0, 0, 0, 0};
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const uint32_t x = uint32_t(w[i]) ^ same;
    const uint32_t t = (x | 0x88888888u) - 0x11111111u;
    r[i] = int((~(t | x) & 0x88888888u) >> 1);
  }
  return r;
}

// The exponent e of a book's largest finite magnitude, below 2^e. Every wave
// works it out for itself: no barrier delays the block's first loads.
template <int ENTRIES>
__device__ __forceinline__ int book_exponent(const float* book) {
  float top = 0.0f;
#pragma unroll
  for (int i = 0; i < ENTRIES / 64; ++i) {
    const float v = fabsf(book[threadIdx.x % 64 + 64 * i]);
    top = v <= FLT_MAX ? fmaxf(top, v) : top;
  }
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) top = fmaxf(top, __shfl_xor(top, off));
  int e = 0;
  if (top > 0.0f) (void)frexpf(top, &e);
  return e;
}

// The power of two that brings the book's largest magnitude into [2^-61, 2^top):
// almost always 0, seen without a reduction.
template <int ENTRIES>
__device__ __forceinline__ int book_scale(const float* book, int top) {
  bool large = false, usual = false;
#pragma unroll
  for (int i = 0; i < ENTRIES / 64; ++i) {
    const float v = fabsf(book[threadIdx.x % 64 + 64 * i]);
    large |= v >= ldexpf(1.0f, top);
    usual |= v >= 0x1p-61f;
  }
  if (!__any(large) && __any(usual)) return 0;
  const int e = book_exponent<ENTRIES>(book);
  return e > top ? top - e : e < -60 ? -60 - e : 0;
}

// One thread's share of a step's words, gathered from the codes: word `w` (8
// inner indices from 128 step + 8 w) of the block's column `at`, zero past k.
__device__ __forceinline__ uint32_t gather_word(const uint32_t* codes, uint32_t columns, uint32_t v,
                                                uint32_t kk0, uint32_t k) {
  uint32_t word = 0;
#pragma unroll
  for (uint32_t i = 0; i < 8; ++i) {
    const uint32_t kk = kk0 + i;
    const uint64_t flat = uint64_t(kk < k ? kk : k - 1) * columns + v;
    const uint32_t code = codes[flat >> 3] >> (4 * uint32_t(flat & 7)) & 15u;
    word |= (kk < k ? code : 0u) << (4 * i);
  }
  return word;
}

// grid: (ceil(n/G / 2JG), ceil(m/G / 2IG), instances). A wave counts IG x JG
// pairs, four result registers each. GATHER: the block transposes the codes it
// needs itself, step by step through LDS; otherwise k_joint_words has.
template <int G, int IG, int JG, bool GATHER>
__global__ __launch_bounds__(kJointThreads, 2) void k_joint_mfma(Operands o, uint32_t m, uint32_t n,
                                                                 uint32_t k,
                                                                 const uint32_t* workspace) {
  constexpr int kColumns = 2 * (IG + JG);            // code columns of a block
  constexpr int kShare = (kColumns * 16 + kJointThreads - 1) / kJointThreads;
  constexpr int kS = G == 16 ? 1 : 2;  // operand sets of a book: 16-value halves of its rows, or
                                       // (group 8) the row in either half of the sides
  __shared__ __align__(16) uint32_t stage[GATHER ? 2 : 1][GATHER ? kColumns : 1][16];
  const uint32_t va = m / G, vb = n / G;
  const uint32_t kp = padded_k(k), words = kp / 8;
  const uint32_t lane = threadIdx.x % 64, wave = threadIdx.x / 64;
  const uint32_t l16 = lane % 16, q = lane / 16;
  const uint32_t ig0 = (blockIdx.y * 2 + wave / 2) * IG, jg0 = (blockIdx.x * 2 + wave % 2) * JG;
  const uint32_t same = l16 * 0x11111111u;

  for (uint32_t item = blockIdx.z; item < o.count; item += gridDim.z) {
    const float* a_book = item_ptr<float>(o.in[1], o.stride[1], item);
    const float* b_book = item_ptr<float>(o.in[3], o.stride[3], item);
    float* out = reinterpret_cast<float*>(static_cast<char*>(o.out) + o.stride[4] * item);
    // ---- the books as operands (A's times the 1/4 of the counts' unit). Entries
    // that no code uses, or that never meet, add exact zeros, so a book needs a scale
    // only where its counted entries (up to 2^16 times 2^128) would overflow, or where
    // all of it is so small that the sums might be subnormal; scaling by its largest
    // entry otherwise loses or overflows others. Group 8 fills an instruction's 16
    // sides with two vectors: its second operand set holds the book in sides 8 to 15.
    const int sa = book_scale<16 * G>(a_book, 109);
    const int sb = book_scale<16 * G>(b_book, 128);
    const int up = -(sa + sb);
    bool bad = false;
    if (blockIdx.x == 0 && blockIdx.y == 0)
      for (uint32_t i = threadIdx.x; i < 16 * G; i += kJointThreads)
        bad |= !finite_f32(a_book[i]) || !finite_f32(b_book[i]);
    float ca[kS][4], cb[kS][4];
#pragma unroll
    for (int b = 0; b < kS; ++b)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const bool in = G >= 16 || (l16 / 8 == uint32_t(b));
        const uint32_t at = (4 * q + r) * G + (G >= 16 ? 16 * b + l16 : l16 % 8);
        ca[b][r] = in ? ldexpf(a_book[at], sa - 2) : 0.0f;
        cb[b][r] = in ? ldexpf(b_book[at], sb) : 0.0f;
      }

    f32x4 h[IG][JG];
#pragma unroll
    for (int i = 0; i < IG; ++i)
#pragma unroll
      for (int j = 0; j < JG; ++j) h[i][j] = (f32x4)0.0f;
    // indices past k read code 0 on both sides: H[0][0] starts that much lower
    if (lane == 0) {
      const float pad = -4.0f * float(kp - k);
#pragma unroll
      for (int i = 0; i < IG; ++i)
#pragma unroll
        for (int j = 0; j < JG; ++j) h[i][j][0] = pad;
    }

    const uint32_t steps = kp / kJointStep;
    if constexpr (GATHER) {
      const uint32_t* a_codes = item_ptr<uint32_t>(o.in[0], o.stride[0], item);
      const uint32_t* b_codes = item_ptr<uint32_t>(o.in[2], o.stride[2], item);
      const uint32_t ib = blockIdx.y * 2 * IG, jb = blockIdx.x * 2 * JG;
      uint32_t word[kShare];
      auto gather = [&](uint32_t s) {
#pragma unroll
        for (int x = 0; x < kShare; ++x) {
          // neighbouring threads take neighbouring columns of a row
          const uint32_t at = (threadIdx.x + x * kJointThreads) % kColumns;
          const uint32_t w = (threadIdx.x + x * kJointThreads) / kColumns % 16;
          const bool left = at < 2 * IG;
          const uint32_t columns = left ? va : vb;
          const uint32_t v = left ? ib + at : jb + at - 2 * IG;
          word[x] = gather_word(left ? a_codes : b_codes, columns, v < columns ? v : columns - 1,
                                s * kJointStep + 8 * w, k);
        }
      };
      gather(0);
      for (uint32_t s = 0; s < steps; ++s) {
        auto& buf = stage[s % 2];  // the other one may still be read
#pragma unroll
        for (int x = 0; x < kShare; ++x) {
          const uint32_t id = threadIdx.x + x * kJointThreads;
          if (kColumns * 16 % kJointThreads == 0 || id < kColumns * 16)
            buf[id % kColumns][id / kColumns] = word[x];
        }
        __syncthreads();
        if (s + 1 < steps) gather(s + 1);
        i32x8 fa[IG];
#pragma unroll
        for (int i = 0; i < IG; ++i)
          fa[i] = one_hot(*reinterpret_cast<const i32x4*>(&buf[wave / 2 * IG + i][4 * q]), same);
#pragma unroll
        for (int j = 0; j < JG; ++j) {
          const i32x8 fb = one_hot(
              *reinterpret_cast<const i32x4*>(&buf[2 * IG + wave % 2 * JG + j][4 * q]), same);
#pragma unroll
          for (int i = 0; i < IG; ++i)
            h[i][j] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(fa[i], fb, h[i][j], kFp4,
                                                                       kFp4, 0, 0, 0, 0);
        }
      }
      __syncthreads();  // the next instance's first step writes a buffer again
    } else {
      const uint32_t* wa = workspace + uint64_t(item) * (va + vb) * words;
      const uint32_t* wb = wa + uint64_t(va) * words;

      // columns past the matrix count the last one's codes and are not stored
      const i32x4* pa[IG];
      const i32x4* pb[JG];
#pragma unroll
      for (int i = 0; i < IG; ++i) {
        const uint32_t v = ig0 + i < va ? ig0 + i : va - 1;
        pa[i] = reinterpret_cast<const i32x4*>(wa + uint64_t(v) * words) + q;
      }
#pragma unroll
      for (int j = 0; j < JG; ++j) {
        const uint32_t v = jg0 + j < vb ? jg0 + j : vb - 1;
        pb[j] = reinterpret_cast<const i32x4*>(wb + uint64_t(v) * words) + q;
      }
      i32x4 na[IG], nb[JG];
#pragma unroll
      for (int i = 0; i < IG; ++i) na[i] = pa[i][0];
#pragma unroll
      for (int j = 0; j < JG; ++j) nb[j] = pb[j][0];
      for (uint32_t s = 0; s < steps; ++s) {
        const uint32_t next = 4 * (s + 1 < steps ? s + 1 : s);  // the last step reloads itself
        i32x8 fa[IG];
#pragma unroll
        for (int i = 0; i < IG; ++i) {
          fa[i] = one_hot(na[i], same);
          na[i] = pa[i][next];
        }
#pragma unroll
        for (int j = 0; j < JG; ++j) {
          const i32x8 fb = one_hot(nb[j], same);
          nb[j] = pb[j][next];
#pragma unroll
          for (int i = 0; i < IG; ++i)
            h[i][j] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(fa[i], fb, h[i][j], kFp4, kFp4,
                                                                       0, 0, 0, 0);
        }
      }
    }

    float check = 0.0f;  // NaN once an output is not finite
    if constexpr (G == 8) {
      // two vectors of each side per instruction: T and C^T of a 2 x 2 patch
#pragma unroll
      for (int i = 0; i < IG; i += 2)
#pragma unroll
        for (int j = 0; j < JG; j += 2) {
          f32x4 c = (f32x4)0.0f;
#pragma unroll
          for (int y = 0; y < 2; ++y) {
            f32x4 t = (f32x4)0.0f;
#pragma unroll
            for (int x = 0; x < 2; ++x)
#pragma unroll
              for (int r = 0; r < 4; ++r)
                t = __builtin_amdgcn_mfma_f32_16x16x4f32(h[i + x][j + y][r], ca[x][r], t, 0, 0, 0);
#pragma unroll
            for (int r = 0; r < 4; ++r)
              c = __builtin_amdgcn_mfma_f32_16x16x4f32(cb[y][r], t[r], c, 0, 0, 0);
          }
          const uint32_t iv = ig0 + i + l16 / 8, jv = jg0 + j + q / 2;
          if (iv < va && jv < vb) {
#pragma unroll
            for (int r = 0; r < 4; ++r) {
              c[r] = ldexpf(c[r], up);
              check = fmaf(c[r], 0.0f, check);
            }
            *reinterpret_cast<f32x4*>(out + (uint64_t(iv) * 8 + l16 % 8) * n + uint64_t(jv) * 8 +
                                      4 * (q % 2)) = c;
          }
        }
    } else {
#pragma unroll
      for (int i = 0; i < IG; ++i)
#pragma unroll
        for (int j = 0; j < JG; ++j) {
          const bool live = ig0 + i < va && jg0 + j < vb;
#pragma unroll
          for (int sb = 0; sb < kS; ++sb) {
            f32x4 t = (f32x4)0.0f;  // T[f][s] = sum_e H[e][f] C_A[e][s]
#pragma unroll
            for (int r = 0; r < 4; ++r)
              t = __builtin_amdgcn_mfma_f32_16x16x4f32(h[i][j][r], ca[sb][r], t, 0, 0, 0);
#pragma unroll
            for (int tb = 0; tb < kS; ++tb) {
              f32x4 c = (f32x4)0.0f;  // C^T[t][s] = sum_f C_B[f][t] T[f][s]
#pragma unroll
              for (int r = 0; r < 4; ++r)
                c = __builtin_amdgcn_mfma_f32_16x16x4f32(cb[tb][r], t[r], c, 0, 0, 0);
              if (live) {
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                  c[r] = ldexpf(c[r], up);
                  check = fmaf(c[r], 0.0f, check);
                }
                *reinterpret_cast<f32x4*>(out + (uint64_t(ig0 + i) * G + 16 * sb + l16) * n +
                                          uint64_t(jg0 + j) * G + 16 * tb + 4 * q) = c;
              }
            }
          }
        }
    }
    bad |= check != check;
    if (__any(bad) && lane == 0) atomicOr(o.status, 1u);
  }
}

template <int G, int IG, int JG>
void run_joint(hipStream_t s, const Operands& o, uint32_t m, uint32_t n, uint32_t k, uint32_t z,
               const uint32_t* words) {
  const dim3 grid((n / G + 2 * JG - 1) / (2 * JG), (m / G + 2 * IG - 1) / (2 * IG), z);
  if (words == nullptr) k_joint_mfma<G, IG, JG, true><<<grid, kJointThreads, 0, s>>>(o, m, n, k, words);
  else k_joint_mfma<G, IG, JG, false><<<grid, kJointThreads, 0, s>>>(o, m, n, k, words);
}

template <int G>
void choose_joint(hipStream_t s, const Operands& o, uint32_t m, uint32_t n, uint32_t k, uint32_t z,
                  const uint32_t* words) {
  // A wave of 4 x 4 pairs builds half the one-hot rows per pair of a 2 x 2 one,
  // which only wins where 4 x 4 leaves compute units idle (1024 x 1024, k =
  // 2048 at group 16: 12.6 against 18.2 us; 4096 x 4096, k = 512: 34 against
  // 27). 4 x 8 builds fewer still but holds two waves per SIMD against four: it
  // pays at group 8 only, whose counts are four times group 16's (4096 x 14336,
  // k = 2048: 437 against 474 us; k = 512 on 4096 x 4096 even).
  const uint64_t blocks = uint64_t((n / G + 7) / 8) * ((m / G + 7) / 8) * z;
  if (G == 8 && k > 2 * kJointGather && blocks >= 2048) run_joint<G, 4, 8>(s, o, m, n, k, z, words);
  else if (blocks >= 256) run_joint<G, 4, 4>(s, o, m, n, k, z, words);
  else run_joint<G, 2, 2>(s, o, m, n, k, z, words);
}

}  // namespace

bool joint_applies(uint32_t m, uint32_t n, uint32_t k, uint32_t group, uint32_t flags,
                   bool any_size) {
  if (flags != 1 || m % group != 0 || n % group != 0 || m < kJointMinRows) return false;
  if (!any_size && k < (group == 8 ? kJointMinK8 : kJointMinK)) return false;
  return any_size || uint64_t(m) * n * k >= kJointMinMacs;
}

size_t joint_workspace_bytes(uint32_t m, uint32_t n, uint32_t k, uint32_t group, uint32_t count) {
  if (k <= kJointGather) return 0;
  const size_t bytes = size_t(m / group + n / group) * (padded_k(k) / 8) * 4 * count;
  return bytes <= kJointMaxWorkspace ? bytes : 0;
}

hipError_t launch_joint(hipStream_t s, const Operands& o, uint32_t m, uint32_t n, uint32_t k,
                        uint32_t group, void* workspace) {
  const uint32_t z = o.count < 65535 ? o.count : 65535;
  uint32_t* words = joint_workspace_bytes(m, n, k, group, o.count) == 0
                        ? nullptr : static_cast<uint32_t*>(workspace);
  if (words != nullptr) {
    const uint32_t va = m / group, vb = n / group;
    const dim3 pre((va + vb + 63) / 64, (padded_k(k) / 32 + 3) / 4, z);
    k_joint_words<<<pre, 256, 0, s>>>(o, va, vb, k, words);
  }
  if (group == 8) choose_joint<8>(s, o, m, n, k, z, words);
  else if (group == 16) choose_joint<16>(s, o, m, n, k, z, words);
  else choose_joint<32>(s, o, m, n, k, z, words);
  return hipGetLastError();
}

}  // namespace ackvq
