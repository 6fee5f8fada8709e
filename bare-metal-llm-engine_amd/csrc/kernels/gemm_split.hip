// gemm_split.hip -- FP32 GEMM on the bf16 matrix cores.
//
//   C[M x N] = A[M x K] . B, B fp32 or fp16, given [K x N] or (BNK) [N x K].
//
// v_mfma_f32_32x32x16_bf16 runs 16 times the rate of v_mfma_f32_32x32x2_f32.
// Every fp32 value is the exact sum of three bf16 terms (a = a1 + a2 + a3:
// a1 = bf16(a), a2 = bf16(a - a1), a3 = a - a1 - a2, 8 bits each), products of
// two bf16 values are exact in fp32, and the sums accumulate in fp32. Of the
// nine term products six are taken -- (1,1) (1,2) (2,1) (2,2) (1,3) (3,1); the
// three left out are at most 2^-23 of |a b| together. An fp16 B is two terms and
// all six products.
//
// Each call of the instruction rounds its running sum, and not to the nearest
// (with all six products on one sum, A . diag(1..2) came out 0.24 x 2^-24 low on
// average, positive or negative). So the leading products and the five small ones
// (at most 2^-8 of them) have a running sum each, added at the end: a 16-deep
// slice rounds the large sum once, where the FP32 instruction rounds it eight
// times. Error against float64, 2-norms at 4096^3, FP32
// instruction -> this (in brackets all six products on one sum): U[-1, 1] 1.15e-6
// -> 3.8e-7 (1.0e-6), U[0, 1] 8.4e-7 -> 3.0e-7 (5.3e-7), half of A zero 8.1e-7 ->
// 3.2e-7 (9.4e-7), 95% of A zero 2.6e-7 -> 1.0e-7 (4.9e-7). Where one product makes
// the sum (a diagonal factor) its one rounding, 2.49e-8 and 2^-24 at most, becomes
// that and the products left out: 2.53e-8, and 1.85 x 2^-24 at most seen, 3 x 2^-24
// possible.
//
// What the split does not hold is found and done again on v_mfma_f32_32x32x2_f32
// with the unsplit operands, element by element (in the 32 x 32 blocks that hold
// one): sums that are not finite (an infinity, NaN, a sum past the fp32 range), and
// sums next to which values under 2^-110 could matter, whose third remainder may
// have bits below bf16's (a flag is set while such a value is staged; then each
// row's and column's largest magnitudes bound each sum). 4096^3, 630 us, and 900-990
// on the FP32 instruction alone: one NaN 912 us, NaN in every row 1970,
// probabilities down to e^-87 everywhere 830, the same with zero columns beside
// them 834; while one such element had its whole tile done again 2270, 2470, 867
// and 2770.
//
// What bounds it: the matrix cores at the clock the card holds under them
// (4096^3: matrix cores busy 63-72% of the cycles, the clock near 1.75 GHz; chains of
// this instruction on random registers sustain 1594 TFLOP/s, 266 of these six-
// product FLOP), then LDS. 4096^3: 908 -> 629 us (151 -> 218 TFLOP/s) against
// the FP32 instruction; 512 x 4096 x 4096 120 -> 95 us; 509 x 2051 x 1023 (no row
// aligned) 64 -> 29.6 us.
#include "gemm_choice.hpp"
#include "gemm_plan.hpp"
#include "device_sync.hpp"
#include "launch.hpp"

#include <algorithm>
#include <type_traits>
#include <utility>

namespace eng {
namespace {

typedef float floatx16 __attribute__((ext_vector_type(16)));
typedef float floatx4 __attribute__((ext_vector_type(4)));
typedef float floatx2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef _Float16 halfx8 __attribute__((ext_vector_type(8)));
typedef unsigned uintx4 __attribute__((ext_vector_type(4)));
typedef unsigned uintx2 __attribute__((ext_vector_type(2)));
typedef short shortx4 __attribute__((ext_vector_type(4)));

constexpr int BK = kGemmKTile;

// Tile BM x BN by KG groups of WGM x WGN waves; each group takes every KG-th
// K tile with LDS stages of its own, and the groups' sums are added through
// LDS at the end.
template <int BM_, int BN_, int WGM_, int WGN_, int KG_ = 1>
struct SplitCfg {
  static constexpr int BM = BM_;
  static constexpr int BN = BN_;
  static constexpr int WGM = WGM_;
  static constexpr int WGN = WGN_;
  static constexpr int KG = KG_;
  static constexpr int kGroup = 64 * WGM * WGN;  // threads of a group
  static constexpr int kThreads = kGroup * KG;
  static constexpr int WM = BM / WGM;
  static constexpr int WN = BN / WGN;
  static constexpr int MB = WM / 32;
  static constexpr int NB = WN / 32;
  static constexpr int A8 = BM * BK / 8 / kGroup;  // 8-value chunks a thread stages per K tile
  static constexpr int B8 = BN * BK / 8 / kGroup;
  static constexpr int kLds = KG * 2 * 3 * 2 * BK * (BM + BN);
  // workgroups a CU holds: by LDS, and at most two waves per SIMD (256 registers each)
  static constexpr int kPerCuLds = 160 * 1024 / kLds;
  static constexpr int kPerCuWaves = 512 / kThreads;
  static constexpr int kPerCu = kPerCuLds < kPerCuWaves ? kPerCuLds : kPerCuWaves;
  static_assert(A8 * 8 * kGroup == BM * BK && B8 * 8 * kGroup == BN * BK, "staging shape");
  static_assert(KG <= 2 && kPerCu >= 1, "workgroup shape");
};
template <typename C>
using SplitAcc = floatx16[C::MB][C::NB];

// LDS tiles are bf16 planes. Rows along k (A, [N x K] B): 64 bytes, chunk c (8
// values) of row r at c ^ ((r >> 2) & 3). [K x N] B: rows of BN values, chunk
// c of row k at c ^ swz_kn<BN>(k), so the 8 rows x 64 bytes a transposing read
// touches cover the banks twice, the minimum.
__device__ __forceinline__ int swz_rows(int r) { return (r >> 2) & 3; }
template <int BN>
__device__ __forceinline__ int swz_kn(int k) {
  return BN >= 128 ? 4 * (k & 3) : 4 * ((k >> 1) & 1);
}

// f(integral_constant<int, I>{}) for each I.
template <typename F, int... I>
__device__ __forceinline__ void each_index(F&& f, std::integer_sequence<int, I...>) {
  (f(std::integral_constant<int, I>{}), ...);
}

// Eight values as three bf16 planes; flag collects the bits left in the third
// remainder (its low half must be empty for the three terms to hold the value).
__device__ __forceinline__ void split3(const float (&v)[8], uintx4 (&p)[3], unsigned& flag) {
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const floatx2 x = {v[2 * i], v[2 * i + 1]};
    const unsigned p1 = __builtin_bit_cast(unsigned, __builtin_convertvector(x, bf16x2));
    const floatx2 r = {x[0] - __builtin_bit_cast(float, p1 << 16),
                       x[1] - __builtin_bit_cast(float, p1 & 0xffff0000u)};
    const unsigned p2 = __builtin_bit_cast(unsigned, __builtin_convertvector(r, bf16x2));
    const unsigned s0 = __builtin_bit_cast(unsigned, r[0] - __builtin_bit_cast(float, p2 << 16));
    const unsigned s1 =
        __builtin_bit_cast(unsigned, r[1] - __builtin_bit_cast(float, p2 & 0xffff0000u));
#if defined(__HIP_DEVICE_COMPILE__)
    // (in asm: the compiler sinks a plain |= and keeps every remainder live)
    asm("v_or3_b32 %0, %0, %1, %2" : "+v"(flag) : "v"(s0), "v"(s1));
#else
    flag |= s0 | s1;
#endif
    p[0][i] = p1;
    p[1][i] = p2;
    p[2][i] = __builtin_amdgcn_perm(s1, s0, 0x07060302u);
  }
}

// Eight consecutive elements at p as floats. VEC: 16-byte aligned; else only
// element-aligned (global memory takes dword-aligned 16-byte loads).
struct __attribute__((packed, aligned(4))) Float4U {
  float v[4];
};
struct __attribute__((packed, aligned(2))) Half8U {
  _Float16 v[8];
};
template <bool VEC, typename T>
__device__ __forceinline__ void load8(const T* p, float (&v)[8]) {
  if constexpr (std::is_same<T, float>::value) {
    if constexpr (VEC) {
      const floatx4 a = *reinterpret_cast<const floatx4*>(p);
      const floatx4 b = *reinterpret_cast<const floatx4*>(p + 4);
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] = a[e], v[4 + e] = b[e];
    } else {
      const Float4U a = *reinterpret_cast<const Float4U*>(p);
      const Float4U b = *reinterpret_cast<const Float4U*>(p + 4);
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] = a.v[e], v[4 + e] = b.v[e];
    }
  } else {
    if constexpr (VEC) {
      const halfx8 h = *reinterpret_cast<const halfx8*>(p);
#pragma unroll
      for (int e = 0; e < 8; ++e) v[e] = static_cast<float>(h[e]);
    } else {
      const Half8U h = *reinterpret_cast<const Half8U*>(p);
#pragma unroll
      for (int e = 0; e < 8; ++e) v[e] = static_cast<float>(h.v[e]);
    }
  }
}

// The same with halves left as they are, in v[0 .. 3]: nothing waits for the load,
// and it holds four registers until widen8.
template <bool VEC, typename T>
__device__ __forceinline__ void load8_raw(const T* p, float (&v)[8]) {
  if constexpr (std::is_same<T, float>::value) {
    load8<VEC>(p, v);
  } else {
    Half8U h;
    if constexpr (VEC) h = __builtin_bit_cast(Half8U, *reinterpret_cast<const halfx8*>(p));
    else h = *reinterpret_cast<const Half8U*>(p);
    const floatx4 w = __builtin_bit_cast(floatx4, h);
#pragma unroll
    for (int e = 0; e < 4; ++e) v[e] = w[e];
  }
}
template <typename T>
__device__ __forceinline__ void widen8(float (&v)[8]) {
  if constexpr (!std::is_same<T, float>::value) {
    const halfx8 h = __builtin_bit_cast(halfx8, floatx4{v[0], v[1], v[2], v[3]});
#pragma unroll
    for (int e = 0; e < 8; ++e) v[e] = static_cast<float>(h[e]);
  }
}

// The K tiles [kt0, kt1) of the tile at (m0, n0) into acc (zeroed here). With
// two groups only group 0's acc is the sum.
template <typename C, bool BNK, typename BT, Form FORM>
__device__ __forceinline__ void split_tile(const float* __restrict__ A, const BT* __restrict__ B,
                                           int M, int N, int K, int m0, int n0, int kt0, int kt1,
                                           SplitAcc<C>& acc) {
  constexpr int MB = C::MB;
  constexpr int NB = C::NB;
  constexpr int A8 = C::A8;
  constexpr int B8 = C::B8;
  constexpr int T = C::kGroup;
  constexpr int KG = C::KG;
  constexpr int BN = C::BN;
  constexpr int AP = C::BM * BK;  // bf16 values of one A plane tile
  constexpr int BP = C::BN * BK;
  constexpr bool HB = std::is_same<BT, _Float16>::value;
  constexpr int PB = HB ? 2 : 3;  // B planes
  constexpr bool GEN = FORM != ALIGNED;
  __shared__ __attribute__((aligned(1024))) __bf16 As0[KG * 3 * AP];
  __shared__ __attribute__((aligned(1024))) __bf16 As1[KG * 3 * AP];
  __shared__ __attribute__((aligned(1024))) __bf16 Bs0[KG * PB * BP];
  __shared__ __attribute__((aligned(1024))) __bf16 Bs1[KG * PB * BP];
  __shared__ int wave_bad[C::kThreads / 64];

  const int t = threadIdx.x % T;
  const int lane = t & 63;
  const int wg_wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x) >> 6);
  const int group = KG == 1 ? 0 : wg_wave / (T / 64);
  const int wave = wg_wave % (T / 64);
  const int li = lane & 31;
  const int lg = lane >> 5;
  const int wm = wave / C::WGN;
  const int wn = wave % C::WGN;
  constexpr int CPR = BNK ? 4 : BN / 8;  // chunks per B tile row
  auto a_stage = [&](auto st) -> __bf16* {
    if constexpr (decltype(st)::value == 0) return As0 + group * 3 * AP;
    else return As1 + group * 3 * AP;
  };
  auto b_stage = [&](auto st) -> __bf16* {
    if constexpr (decltype(st)::value == 0) return Bs0 + group * PB * BP;
    else return Bs1 + group * PB * BP;
  };

  // Chunk j of thread t: slot q = T j + t; A and [N x K] B: row q / 4, k chunk
  // q % 4; [K x N] B: k row q / CPR, column chunk q % CPR. Rows past the
  // matrix read the last one and columns past it the last chunk: they feed
  // only elements of C that are not stored.
  const float* ap[A8];
  const BT* bp[B8];
#pragma unroll
  for (int j = 0; j < A8; ++j) {
    const int q = T * j + t;
    ap[j] = A + static_cast<long long>(min(m0 + (q >> 2), M - 1)) * K + 8 * (q & 3);
  }
  [[maybe_unused]] int shift[FORM == SHIFT ? B8 : 1];
#pragma unroll
  for (int j = 0; j < B8; ++j) {
    const int q = T * j + t;
    if constexpr (BNK) {
      bp[j] = B + static_cast<long long>(min(n0 + (q >> 2), N - 1)) * K + 8 * (q & 3);
    } else {
      const int c = n0 + 8 * (q % CPR);
      if constexpr (FORM == SHIFT) shift[j] = c < N && c + 8 > N ? c + 8 - N : 0;
      bp[j] = B + static_cast<long long>(q / CPR) * N + min(c, N - 8);
    }
  }

  // Chunks 0 .. A8 - 1 are A's, the rest B's: loaded to raw[ch], then split
  // into the planes.
  constexpr int CH = A8 + B8;
  float raw[CH][8];
  auto load = [&](auto chc, int kt, float(&v)[8]) {
    constexpr int ch = decltype(chc)::value;
    const long long k0 = static_cast<long long>(kt) * BK;
    if constexpr (ch < A8) load8<!GEN>(ap[ch] + k0, v);
    else load8_raw<!GEN>(bp[ch - A8] + (BNK ? k0 : k0 * N), v);
  };
  // The partial K tile, element by element (elements past K are zeros).
  [[maybe_unused]] auto load_partial = [&](auto chc, int kt, float(&v)[8]) {
    constexpr int ch = decltype(chc)::value;
    constexpr bool IS_A = ch < A8;
    constexpr int j = IS_A ? ch : ch - A8;
    int q = T * j + t;
#if defined(__HIP_DEVICE_COMPILE__)
    asm volatile("" : "+v"(q));  // (its addresses are not kept through the pipeline)
#endif
    const int k0 = kt * BK;
    std::conditional_t<IS_A, float, BT> w[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const int k = IS_A || BNK ? k0 + 8 * (q & 3) + e : k0 + q / CPR;
      if constexpr (IS_A)
        w[e] = A[static_cast<long long>(min(m0 + (q >> 2), M - 1)) * K + min(k, K - 1)];
      else if constexpr (BNK)
        w[e] = B[static_cast<long long>(min(n0 + (q >> 2), N - 1)) * K + min(k, K - 1)];
      else
        w[e] = B[static_cast<long long>(min(k, K - 1)) * N + min(n0 + 8 * (q % CPR) + e, N - 1)];
      if (k >= K) w[e] = 0;
    }
    if constexpr (std::is_same<std::decay_t<decltype(w[0])>, float>::value) {
#pragma unroll
      for (int e = 0; e < 8; ++e) v[e] = w[e];
    } else {
      halfx8 h;
#pragma unroll
      for (int e = 0; e < 8; ++e) h[e] = w[e];
      const floatx4 bits = __builtin_bit_cast(floatx4, h);
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] = bits[e];
    }
  };
  unsigned flag = 0;
  // (whole: v as load() leaves it, else as load_partial() does)
  auto put = [&](auto chc, __bf16* as, __bf16* bs, float(&v)[8], auto whole) {
    constexpr int ch = decltype(chc)::value;
    constexpr bool IS_A = ch < A8;
    const int q = T * (IS_A ? ch : ch - A8) + t;
    if constexpr (!IS_A) widen8<BT>(v);
    if constexpr (!IS_A && FORM == SHIFT && decltype(whole)::value) {
#pragma unroll
      for (int b = 4; b > 0; b >>= 1) {
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          const float here = v[e];
          const float there = v[e + b < 8 ? e + b : e];
          v[e] = (shift[ch - A8] & b) ? there : here;
        }
      }
    }
    uintx4 p[3];
    split3(v, p, flag);
    if constexpr (IS_A) {
#pragma unroll
      for (int i = 0; i < 3; ++i)
        *reinterpret_cast<uintx4*>(as + i * AP + (q >> 2) * BK + 8 * ((q & 3) ^ swz_rows(q >> 2))) =
            p[i];
    } else {
      const int off = BNK ? (q >> 2) * BK + 8 * ((q & 3) ^ swz_rows(q >> 2))
                          : (q / CPR) * BN + 8 * ((q % CPR) ^ swz_kn<BN>(q / CPR));
#pragma unroll
      for (int i = 0; i < PB; ++i) *reinterpret_cast<uintx4*>(bs + i * BP + off) = p[i];
    }
  };
  auto each_chunk = [&](auto f) { each_index(f, std::make_integer_sequence<int, CH>{}); };

  struct Slice {
    bf16x8 a[3][MB];
    bf16x8 b[PB][NB];
  };
  auto read_s = [&](const __bf16* as, const __bf16* bs, int sl, Slice& f) {
    const int cq = 2 * sl + lg;  // this lane's chunk: k = 16 sl + 8 lg .. + 7
#pragma unroll
    for (int p = 0; p < 3; ++p) {
#pragma unroll
      for (int mb = 0; mb < MB; ++mb) {
        const int r = wm * C::WM + mb * 32 + li;
        f.a[p][mb] =
            *reinterpret_cast<const bf16x8*>(as + p * AP + r * BK + 8 * (cq ^ swz_rows(r)));
      }
    }
#pragma unroll
    for (int p = 0; p < PB; ++p) {
#pragma unroll
      for (int nb = 0; nb < NB; ++nb) {
        if constexpr (BNK) {
          const int r = wn * C::WN + nb * 32 + li;
          f.b[p][nb] =
              *reinterpret_cast<const bf16x8*>(bs + p * BP + r * BK + 8 * (cq ^ swz_rows(r)));
        } else {
          // Two transposing reads per fragment (ds_read_b64_tr_b16): in each
          // 16-lane group lane l names 8 bytes (row k0 + l / 4, columns cb + 4
          // (l % 4) .. + 3) and receives column cb + l of the 4 rows.
          const int l = lane & 15;
          const int G = lane >> 4;
          const int col = wn * C::WN + nb * 32 + 16 * (G & 1) + 4 * (l & 3);
          uintx4 w;
#pragma unroll
          for (int h = 0; h < 2; ++h) {
            const int k = 16 * sl + 8 * (G >> 1) + 4 * h + (l >> 2);
            const int off = k * (BN * 2) + (((col >> 3) ^ swz_kn<BN>(k)) << 4) + ((col & 7) << 1);
            const uintx2 v = __builtin_bit_cast(
                uintx2, __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                            (__attribute__((address_space(3))) shortx4*)(
                                (__attribute__((address_space(3))) char*)(bs + p * BP) + off)));
            w[2 * h] = v[0];
            w[2 * h + 1] = v[1];
          }
          f.b[p][nb] = __builtin_bit_cast(bf16x8, w);
        }
      }
    }
  };
  SplitAcc<C> small;  // the five small products' sum; acc the leading one's
#pragma unroll
  for (int mb = 0; mb < MB; ++mb)
#pragma unroll
    for (int nb = 0; nb < NB; ++nb)
#pragma unroll
      for (int v = 0; v < 16; ++v) acc[mb][nb][v] = small[mb][nb][v] = 0.0f;
  auto fold = [&] {  // the small sums into the large ones
#pragma unroll
    for (int mb = 0; mb < MB; ++mb)
#pragma unroll
      for (int nb = 0; nb < NB; ++nb)
#pragma unroll
        for (int v = 0; v < 16; ++v) {
          acc[mb][nb][v] += small[mb][nb][v];
          small[mb][nb][v] = 0.0f;
        }
  };
  // MFMAs [lo, hi) of a slice's 6 MB NB, by product, then block.
  constexpr int NM = 6 * MB * NB;
  auto mma = [&](const Slice& f, int lo, int hi) {
    constexpr int P[6][2] = {{2, 0}, {HB ? 2 : 0, HB ? 1 : 2}, {1, 1}, {1, 0}, {0, 1}, {0, 0}};
#pragma unroll
    for (int i = 0; i < 6; ++i) {
#pragma unroll
      for (int mb = 0; mb < MB; ++mb)
#pragma unroll
        for (int nb = 0; nb < NB; ++nb) {
          const int n = (i * MB + mb) * NB + nb;
          if (n >= lo && n < hi) {
            floatx16& sum = i == 5 ? acc[mb][nb] : small[mb][nb];
            sum = __builtin_amdgcn_mfma_f32_32x32x16_bf16(f.a[P[i][0]][mb], f.b[P[i][1]][nb], sum, 0,
                                                          0, 0);
          }
        }
    }
  };

  // One K tile per step from stage st: the first slice is multiplied, the next
  // tile's planes (its values loaded a step ago) written to the other stage
  // meanwhile, the loads of the tile after it issued and the tile's second slice
  // read; one barrier, then the second slice is multiplied and the next tile's
  // first one read. Each slice is read in the last third of the other's MFMAs,
  // when the other's small planes are done with: the second sums fit the registers
  // so (256 x 128 tiles spill outside the loop only; read at the start of the
  // other's MFMAs they spilled 238 inside, 4096^3 1800 us). Past the end the last
  // tile is staged again, never used. The scheduling groups put each chunk's split
  // (about 50 vector instructions) behind its share of the MFMAs, which leave the
  // vector unit free for most of their 32 cycles.
  [[maybe_unused]] constexpr int READS = 3 * MB + PB * NB * (BNK ? 1 : 2);  // fragment reads of a slice
  Slice x, y;
  auto step = [&](auto st, int next_kt) {
    using Next = std::integral_constant<int, 1 - decltype(st)::value>;
    each_chunk([&](auto chc) {
      constexpr int ch = decltype(chc)::value;
      if constexpr (ch == CH - 1) read_s(a_stage(st), b_stage(st), 1, y);
      put(chc, a_stage(Next{}), b_stage(Next{}), raw[ch], std::true_type{});
      load(chc, next_kt, raw[ch]);
      mma(x, ch * NM / CH, (ch + 1) * NM / CH);
#if defined(__HIP_DEVICE_COMPILE__)
      constexpr int n = (ch + 1) * NM / CH - ch * NM / CH;
      constexpr int reads = ch == CH - 1 ? (READS + n - 1) / n : 0;
#pragma unroll
      for (int i = 0; i < n; ++i) {
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);                             // an MFMA
        if constexpr (reads > 0) __builtin_amdgcn_sched_group_barrier(0x100, reads, 0);  // LDS reads
        __builtin_amdgcn_sched_group_barrier(0x002, (52 + n - 1) / n, 0);              // the split
      }
      __builtin_amdgcn_sched_group_barrier(0x200, 3, 0);  // plane writes
      __builtin_amdgcn_sched_group_barrier(0x020, 2, 0);  // the loads
      __builtin_amdgcn_sched_barrier(0);
#endif
    });
    lds_barrier();
    constexpr int H = NM * 2 / 3;
    mma(y, 0, H);
#if defined(__HIP_DEVICE_COMPILE__)
    __builtin_amdgcn_sched_barrier(0);
#endif
    read_s(a_stage(Next{}), b_stage(Next{}), 0, x);
    mma(y, H, NM);
#if defined(__HIP_DEVICE_COMPILE__)
    constexpr int per = NM - H > 1 ? (READS + NM - H - 2) / (NM - H - 1) : READS;
    __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
#pragma unroll
    for (int i = 0; i < (READS + per - 1) / per; ++i) {
      __builtin_amdgcn_sched_group_barrier(0x100, per, 0);
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
    }
    __builtin_amdgcn_sched_group_barrier(0x008, NM, 0);
    __builtin_amdgcn_sched_barrier(0);
#endif
  };
  using I0 = std::integral_constant<int, 0>;
  using I1 = std::integral_constant<int, 1>;
  // n whole K tiles per group in the pipeline (group g: kt0 + g, kt0 + g + KG,
  // ...); the rest -- whole tiles left over, the partial one, and every tile of
  // an N below one chunk -- staged and multiplied one by one.
  const int whole_end = GEN ? (FORM == SHIFT && N < 8 ? 0 : K / BK) : kt1;
  const int n = max(min(kt1, whole_end) - kt0, 0) / KG;
  const int first = kt0 + group;
  const int last = first + (n - 1) * KG;
  auto put_all = [&](auto whole) {
    each_chunk([&](auto c) {
      put(c, a_stage(I0{}), b_stage(I0{}), raw[decltype(c)::value], whole);
    });
  };
  if (n > 0) {
    each_chunk([&](auto c) { load(c, first, raw[decltype(c)::value]); });
    put_all(std::true_type{});
    each_chunk([&](auto c) { load(c, min(first + KG, last), raw[decltype(c)::value]); });
    lds_barrier();
    read_s(a_stage(I0{}), b_stage(I0{}), 0, x);
    int i = 0;
    for (; i + 1 < n; i += 2) {
      step(I0{}, min(first + (i + 2) * KG, last));
      step(I1{}, min(first + (i + 3) * KG, last));
    }
    if (i < n) step(I0{}, last);
    fold();
  }
  // (the small sums are folded at each tile, so that they hold no registers while
  // its elements are loaded: 24 loads in flight, not one by one)
#pragma unroll 1
  for (int k = kt0 + n * KG; k < kt1; k += KG) {
    const int kt = k + group;
    __syncthreads();  // every wave has read the stages
    if (kt < kt1) {
      if (GEN && kt >= whole_end) {
        each_chunk([&](auto c) { load_partial(c, kt, raw[decltype(c)::value]); });
        put_all(std::false_type{});
      } else {
        each_chunk([&](auto c) { load(c, kt, raw[decltype(c)::value]); });
        put_all(std::true_type{});
      }
    }
    __syncthreads();
    if (kt < kt1) {
      read_s(a_stage(I0{}), b_stage(I0{}), 0, x);
      mma(x, 0, NM);
      read_s(a_stage(I0{}), b_stage(I0{}), 1, y);
      mma(y, 0, NM);
      fold();
    }
  }

  // Whether any wave staged a value the three terms do not hold. (After the
  // barrier every wave has also read its stages.)
  const bool wave_any = __ballot((flag & 0xffffu) != 0) != 0;
  if (lane == 0) wave_bad[wg_wave] = wave_any;
  __syncthreads();
  constexpr int W = C::kThreads / 64;
  int any = 0;
#pragma unroll
  for (int w = 0; w < W; ++w) any |= wave_bad[w];
  if constexpr (KG == 2) {
    static_assert(KG * 3 * AP * 2 >= C::BM * C::BN * 4, "the sums fit the A stage");
    float* red = reinterpret_cast<float*>(As0) + wave * (MB * NB * 16 * 64) + lane;
    if (group == 1) {
#pragma unroll
      for (int mb = 0; mb < MB; ++mb)
#pragma unroll
        for (int nb = 0; nb < NB; ++nb)
#pragma unroll
          for (int v = 0; v < 16; ++v) red[((mb * NB + nb) * 16 + v) * 64] = acc[mb][nb][v];
    }
    __syncthreads();
    if (group == 0) {
#pragma unroll
      for (int mb = 0; mb < MB; ++mb)
#pragma unroll
        for (int nb = 0; nb < NB; ++nb)
#pragma unroll
          for (int v = 0; v < 16; ++v) acc[mb][nb][v] += red[((mb * NB + nb) * 16 + v) * 64];
    }
    __syncthreads();  // a following tile may refill the stages
  }
  const int k0 = kt0 * BK;
  const int k1 = min(kt1 * BK, K);
  int li_late = li, lg_late = lg;
#if defined(__HIP_DEVICE_COMPILE__)
  // what follows depends on the lane through these, which keeps its addresses out
  // of the pipeline's registers
  asm volatile("" : "+v"(li_late), "+v"(lg_late));
#endif
  const int lane_late = 32 * lg_late + li_late;
  // The elements to do again, a bit each: sums that are not finite, and sums that
  // values the terms do not hold may be off by too much.
  unsigned again[MB][NB];
#pragma unroll
  for (int mb = 0; mb < MB; ++mb)
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) {
      again[mb][nb] = 0;
#pragma unroll
      for (int v = 0; v < 16; ++v)
        again[mb][nb] |= fabsf(acc[mb][nb][v]) <= 3.4028235e38f ? 0u : 1u << v;
    }
  if (any != 0) {
    // Such a value is under 2^-110 and off by at most 2^-133, so element (r, c) by
    // (k1 - k0) 2^-133 (max |B's column c| if row r of A has one + max |A's row r|
    // if column c of B has one): nothing next to sums of ordinary size (tiny
    // probabilities beside large ones), and nothing at all where the other factor
    // is zero. Largest magnitudes per row and column, negative if the row or
    // column has such a value:
    float* row_most = reinterpret_cast<float*>(As0);
    float* col_most = row_most + C::BM;  // BN, or W x BN partial ones
    static_assert(KG * 3 * AP * 2 >= (C::BM + W * BN) * 4, "the maxima fit the A stage");
    struct Most {
      float m = 0.0f;       // the largest magnitude
      unsigned low = ~0u;   // 2 bits(v) - 2, the least over nonzero v (a zero's wraps)
      __device__ void add(float v) {
        m = fmaxf(m, fabsf(v));
        low = min(low, (__builtin_bit_cast(unsigned, v) << 1) - 2u);
      }
      __device__ float get() const { return low < 2u * 0x08800000u - 2u ? -m : m; }  // 2^-110
    };
    auto both = [](float p, float q) {
      const float n = fmaxf(fabsf(p), fabsf(q));
      return __builtin_signbit(p) || __builtin_signbit(q) ? -n : n;
    };
    // rows along k, four per wave at a time (16 lanes each), 16 loads in flight per
    // lane (past the end the last value again)
    auto rows = [&](const auto* base, int first, int end, int count, float* out) {
      static_assert(C::BM % (4 * W) == 0 && BN % (4 * W) == 0, "whole groups of rows");
      for (int r0 = 4 * wg_wave; r0 < count; r0 += 4 * W) {
        const int r = r0 + (lane_late >> 4);
        const auto* p = base + static_cast<long long>(min(first + r, end)) * K;
        Most m;
        for (int k = k0 + (lane_late & 15); k < k1; k += 16 * 16) {
          float v[16];
#pragma unroll
          for (int u = 0; u < 16; ++u) v[u] = static_cast<float>(p[min(k + 16 * u, k1 - 1)]);
#pragma unroll
          for (int u = 0; u < 16; ++u) m.add(v[u]);
        }
        float x = m.get();
#pragma unroll
        for (int o = 8; o > 0; o >>= 1) x = both(x, __shfl_xor(x, o));
        if ((lane_late & 15) == 0) out[r] = x;
      }
    };
    rows(A, m0, M - 1, C::BM, row_most);
    if constexpr (BNK) {
      rows(B, n0, N - 1, BN, col_most);
    } else {
      Most m[BN / 64];
      for (int k = k0 + 8 * wg_wave; k < k1; k += 8 * W) {
        float v[8][BN / 64];
#pragma unroll
        for (int u = 0; u < 8; ++u)
#pragma unroll
          for (int c = 0; c < BN / 64; ++c)
            v[u][c] = static_cast<float>(B[static_cast<long long>(min(k + u, k1 - 1)) * N +
                                           min(n0 + 64 * c + lane_late, N - 1)]);
#pragma unroll
        for (int u = 0; u < 8; ++u)
#pragma unroll
          for (int c = 0; c < BN / 64; ++c) m[c].add(v[u][c]);
      }
#pragma unroll
      for (int c = 0; c < BN / 64; ++c) col_most[wg_wave * BN + 64 * c + lane_late] = m[c].get();
    }
    __syncthreads();
    if (group == 0) {
      const float terms = static_cast<float>(k1 - k0);
#pragma unroll
      for (int nb = 0; nb < NB; ++nb) {
        const int c = wn * C::WN + nb * 32 + li_late;
        float col = col_most[c];
        if constexpr (!BNK) {
#pragma unroll
          for (int w = 1; w < W; ++w) col = both(col, col_most[w * BN + c]);
        }
#pragma unroll
        for (int mb = 0; mb < MB; ++mb)
#pragma unroll
          for (int v = 0; v < 16; ++v) {
            const float r = row_most[wm * C::WM + mb * 32 + 8 * (v >> 2) + 4 * lg_late + (v & 3)];
            const float off = (__builtin_signbit(r) ? fabsf(col) * 0x1p-66f : 0.0f) +
                              (__builtin_signbit(col) ? fabsf(r) * 0x1p-66f : 0.0f);
            // at most 2^-26 of the sum (both sides times 2^27: 2^-133 is a subnormal)
            again[mb][nb] |= terms * off * 0x1p-40f <= fabsf(acc[mb][nb][v]) * 2.0f ? 0u : 1u << v;
          }
      }
    }
    __syncthreads();  // As0 is refilled by a following tile
  }
  if (group != 0) return;
  // Those elements once more, straight from memory on the FP32 instruction, in the
  // 32 x 32 blocks that hold any: 16 k at a time (lane half lg_late the upper or lower 8
  // of them), the next ones' loads behind the current ones' MFMAs.
  constexpr int U = 8;
  struct Piece {
    float a[U], b[U];
  };
#pragma unroll
  for (int mb = 0; mb < MB; ++mb) {
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) {
      if (__ballot(again[mb][nb] != 0) == 0) continue;
      const float* pa = A + static_cast<long long>(min(m0 + wm * C::WM + mb * 32 + li_late, M - 1)) * K;
      const int n = min(n0 + wn * C::WN + nb * 32 + li_late, N - 1);
      const BT* pb = BNK ? B + static_cast<long long>(n) * K : B + n;
      floatx16 sum;
#pragma unroll
      for (int v = 0; v < 16; ++v) sum[v] = 0.0f;
      auto load_piece = [&](int k, Piece& f) {
        load8<false>(pa + k + U * lg_late, f.a);
        if constexpr (BNK) {
          load8<false>(pb + k + U * lg_late, f.b);
        } else {
#pragma unroll
          for (int u = 0; u < U; ++u)
            f.b[u] = static_cast<float>(pb[static_cast<long long>(k + U * lg_late + u) * N]);
        }
      };
      auto multiply = [&](const Piece& f) {
#pragma unroll
        for (int u = 0; u < U; ++u)
          sum = __builtin_amdgcn_mfma_f32_32x32x2f32(f.a[u], f.b[u], sum, 0, 0, 0);
      };
      Piece f, g;
      int k = k0;
      if (k + 2 * U <= k1) {
        load_piece(k, f);
#pragma unroll 1
        for (; k + 6 * U <= k1; k += 4 * U) {
          load_piece(k + 2 * U, g);
          __builtin_amdgcn_sched_barrier(0);
          multiply(f);
          load_piece(k + 4 * U, f);
          __builtin_amdgcn_sched_barrier(0);
          multiply(g);
        }
        multiply(f);
        k += 2 * U;
      }
#pragma unroll 1
      for (; k < k1; k += 2 * U) {
#pragma unroll
        for (int u = 0; u < U; ++u) {
          const int ku = k + U * lg_late + u;
          const long long kk = min(ku, K - 1);
          const float va = pa[kk];
          const float vb = static_cast<float>(pb[BNK ? kk : kk * N]);
          f.a[u] = ku < k1 ? va : 0.0f;
          f.b[u] = ku < k1 ? vb : 0.0f;
        }
        multiply(f);
      }
#pragma unroll
      for (int v = 0; v < 16; ++v)
        acc[mb][nb][v] = (again[mb][nb] >> v) & 1u ? sum[v] : acc[mb][nb][v];
    }
  }
}

template <typename C>
__device__ __forceinline__ void split_store(const SplitAcc<C>& acc, float* __restrict__ out,
                                            long long ld, int rows_left, int cols_left) {
  if (C::KG > 1 && threadIdx.x >= C::kGroup) return;  // group 0 holds the sum
  int lane = threadIdx.x & 63;
  const int wave = threadIdx.x >> 6;
#if defined(__HIP_DEVICE_COMPILE__)
  // keeps the element offsets out of the tile loop's registers (spilled, each was
  // read back behind the store before: 20 us a tile)
  asm volatile("" : "+s"(ld), "+v"(lane));
#endif
  const int li = lane & 31;
  const int lg = lane >> 5;
  const int wm = wave / C::WGN;
  const int wn = wave % C::WGN;
  const bool whole = rows_left >= C::BM && cols_left >= C::BN;
#pragma unroll
  for (int mb = 0; mb < C::MB; ++mb) {
#pragma unroll
    for (int nb = 0; nb < C::NB; ++nb) {
      const int col = wn * C::WN + nb * 32 + li;
#pragma unroll
      for (int v = 0; v < 16; ++v) {
        const int row = wm * C::WM + mb * 32 + 8 * (v >> 2) + 4 * lg + (v & 3);
        if (whole || (row < rows_left && col < cols_left)) out[row * ld + col] = acc[mb][nb][v];
      }
    }
  }
}

template <typename C, bool BNK, typename BT, Form FORM>
__global__ __launch_bounds__(C::kThreads, C::kPerCu) void gemm_split_kernel(
    const float* __restrict__ A, const BT* __restrict__ B, float* __restrict__ out,
    float* __restrict__ rec, int M, int N, int K, int tiles_m, int tiles_n, SkPlan plan) {
  const int g = blockIdx.x;
  const bool dp = g < plan.dp;
  const long long s = dp ? 0 : g - plan.dp;
  const long long i0 = dp ? 0 : sk_begin(s, plan);
  const long long i1 = dp ? plan.nk : sk_begin(s + 1, plan);
  const int first_tile = dp ? g : plan.dp;
  SplitAcc<C> acc;
  for (long long it = i0; it < i1;) {
    const long long t = it / plan.nk;
    const int ka = static_cast<int>(it - t * plan.nk);
    const long long tend = (t + 1) * plan.nk;
    const int kb = static_cast<int>((i1 < tend ? i1 : tend) - t * plan.nk);
    int tm, tn;
    tile_of(first_tile + static_cast<int>(t), tiles_m, tiles_n, tm, tn);
    const int m0 = tm * C::BM;
    const int n0 = tn * C::BN;
    split_tile<C, BNK, BT, FORM>(A, B, M, N, K, m0, n0, ka, kb, acc);
    if (ka == 0 && kb == plan.nk) {
      split_store<C>(acc, out + static_cast<long long>(m0) * N + n0, N, M - m0, N - n0);
    } else {
      const int slot = it == i0 ? 0 : 1;
      split_store<C>(acc, rec + (s * 2 + slot) * static_cast<long long>(C::BM * C::BN), C::BN, C::BM,
                     C::BN);
    }
    it = t * plan.nk + kb;
  }
}

// False, with nothing launched, if the cut needs records and they cannot be had.
template <typename C, typename BT, bool BNK>
bool run_split(const GemmArgs& a, Form form, const Cut& cut, long long cus, hipStream_t stream) {
  const int M = static_cast<int>(a.M), N = static_cast<int>(a.N), K = static_cast<int>(a.K);
  const int tiles_m = (M + C::BM - 1) / C::BM;
  const int tiles_n = (N + C::BN - 1) / C::BN;
  const long long ntiles = static_cast<long long>(tiles_m) * tiles_n;
  ENG_CHECK(ntiles <= 0x7fffffffLL, "matmul: too many tiles for one launch");
  SkPlan plan;
  plan.nk = (K + BK - 1) / BK;
  const long long tail = cut.split > 0 ? ntiles % cus : 0;
  plan.dp = static_cast<int>(ntiles - tail);
  plan.I = tail * plan.nk;
  plan.nsk = static_cast<int>(tail > 0 ? cut.split : 0);
  const BT* B = static_cast<const BT*>(a.B);
  auto launch = [&](auto f, float* rec) {
    gemm_split_kernel<C, BNK, BT, decltype(f)::value>
        <<<dim3(static_cast<unsigned>(plan.dp + plan.nsk)), C::kThreads, 0, stream>>>(
            a.A, B, a.C, rec, M, N, K, tiles_m, tiles_n, plan);
    ENG_LAUNCH_CHECK();
  };
  auto go = [&](float* rec) {
    if constexpr (std::is_same<BT, float>::value) {
      if (form == ALIGNED) return launch(std::integral_constant<Form, ALIGNED>{}, rec);
    }
    if constexpr (!BNK) {
      if (form == SHIFT) return launch(std::integral_constant<Form, SHIFT>{}, rec);
    }
    launch(std::integral_constant<Form, ANY>{}, rec);
  };
  if (tail == 0) {
    go(nullptr);
    return true;
  }
  StreamScratch records(
      stream, static_cast<std::size_t>(plan.nsk) * 2 * C::BM * C::BN * sizeof(float), 2, true);
  float* rec = static_cast<float*>(records.get());
  if (rec == nullptr) return false;
  go(rec);
  launch_sk_fixup<C::BM, C::BN>(rec, a.C, M, N, tiles_m, tiles_n, static_cast<int>(tail), plan,
                                stream);
  return true;
}

template <typename BT, bool BNK>
bool split_dispatch(const GemmArgs& a, double fp32_us, long long cus, hipStream_t stream,
                    bool may_split = true) {
  const GemmShape shape = gemm_shape(a);
  const SplitChoice c = gemm_split_choice(shape, cus, may_split);
  if (fp32_us <= c.cut.us) return false;
  const Form form = gemm_split_form(shape);
  bool done = false;
  if (c.bm == 256)
    done = run_split<SplitCfg<256, 128, 4, 2>, BT, BNK>(a, form, c.cut, cus, stream);
  else if (c.bn == 128)
    done = run_split<SplitCfg<128, 128, 2, 4>, BT, BNK>(a, form, c.cut, cus, stream);
  else if (c.bm == 128)
    done = run_split<SplitCfg<128, 64, 2, 2, 2>, BT, BNK>(a, form, c.cut, cus, stream);
  else
    done = run_split<SplitCfg<64, 64, 2, 2, 2>, BT, BNK>(a, form, c.cut, cus, stream);
  // Without records (no memory for them, a capturing stream whose arena is too
  // small, a stream or capture that may not share it) the call runs on the best
  // cut that needs none.
  return done || split_dispatch<BT, BNK>(a, fp32_us, cus, stream, false);
}

}  // namespace

bool launch_gemm_split(const GemmArgs& a, double fp32_us, long long cus, hipStream_t stream) {
  if (a.b == Elem::F32)
    return a.b_nk ? split_dispatch<float, true>(a, fp32_us, cus, stream)
                  : split_dispatch<float, false>(a, fp32_us, cus, stream);
  return a.b_nk ? split_dispatch<_Float16, true>(a, fp32_us, cus, stream)
                : split_dispatch<_Float16, false>(a, fp32_us, cus, stream);
}

}  // namespace eng
