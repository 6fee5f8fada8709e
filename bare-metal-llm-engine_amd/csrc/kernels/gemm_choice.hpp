// gemm_choice.hpp -- which kernel a matrix product or few-row linear layer runs
// on: host arithmetic on sizes, alignment and the CU count, without HIP, so that
// the choice can also be computed where there is no GPU.
#pragma once

#include <algorithm>
#include <limits>

namespace eng {

constexpr int kGemmKTile = 32;

struct GemmShape {
  long long M = 0, N = 0, K = 0;
  bool half_b = false;         // B is fp16
  bool b_nk = false;           // B is given [N x K]
  bool a16 = true, b16 = true; // the operand starts on 16 bytes
};

// ---- the FP32 instruction (gemm.hip)

// Direct loads need K % 32 == 0, 16-byte aligned operands and 16-byte
// aligned B rows ([K x N] rows of N elements; [N x K] rows of K), and every
// lane's byte offset from a tile's corner (up to 64 rows of A, 64 rows of an
// [N x K] B or 32 rows of a [K x N] B) must fit the 31 bits of a buffer
// load's offset.
inline bool gemm_direct_ok(const GemmShape& s) {
  constexpr long long kLim = 0x7fffffffLL;
  const long long b_span = s.b_nk ? 64 * s.K : kGemmKTile * s.N;
  return !s.half_b && s.K % kGemmKTile == 0 && s.a16 && s.b16 && (s.b_nk || s.N % 4 == 0) &&
         64 * s.K * 4 <= kLim && b_span * 4 <= kLim;
}

// Estimated time of the 64 x 64 FP32 tiles: per K tile 0.48 us with one
// workgroup on a CU (1024^3: 256 tiles, 17.9 us) and 0.94 us for a pair (512 x
// 4096 x 4096: 512 tiles, 120 us).
inline double gemm_direct_us(const GemmShape& s, long long cus) {
  const long long tiles = ((s.M + 63) / 64) * ((s.N + 63) / 64);
  const double nk = static_cast<double>(s.K / kGemmKTile);
  return tiles <= cus ? 0.48 * nk : 0.94 * nk * static_cast<double>((tiles + 2 * cus - 1) / (2 * cus));
}

// 16-byte loads of A, and of B, in the register-staged kernel.
inline bool gemm_staged_vec_a(const GemmShape& s) { return s.K % 4 == 0 && s.a16; }
inline bool gemm_staged_vec_b(const GemmShape& s) {
  return (s.b_nk ? s.K : s.N) % (s.half_b ? 8 : 4) == 0 && s.b16;
}

// Estimated time of the register-staged kernel: per K tile 0.8 us with one
// workgroup on a CU and 1.05 us for a pair (1000 x 3000 x 200: 17.5 us), more
// with element loads (200 x 3001 x 64: 4.8 us; 509 x 2051 x 1023: 64.6 us).
inline double gemm_staged_us(const GemmShape& s, long long cus) {
  const long long tiles = ((s.M + 63) / 64) * ((s.N + 63) / 64);
  const double nk = static_cast<double>((s.K + kGemmKTile - 1) / kGemmKTile);
  const bool vec = gemm_staged_vec_a(s) && gemm_staged_vec_b(s);
  if (tiles <= cus) return nk * (vec ? 0.8 : !s.half_b ? 1.15 : 1.6);
  return nk * (vec ? 1.05 : 1.9) * static_cast<double>((tiles + 2 * cus - 1) / (2 * cus));
}

inline bool gemm_small_ok(const GemmShape& s) {
  return !s.half_b && !s.b_nk && s.M % 32 == 0 && s.N % 32 == 0 && s.K % 256 == 0 && s.a16;
}

// Estimated time: 0.0065 us per k and round of one 32 x 32 tile per CU (512^3:
// 5.6 us with about 2.5 of launch; 128 x 4096 x 4096: 63.7 us, two rounds).
inline double gemm_small_us(const GemmShape& s, long long cus) {
  const long long tiles = (s.M / 32) * (s.N / 32);
  return 0.0065 * static_cast<double>(s.K) * static_cast<double>((tiles + cus - 1) / cus);
}

enum class Fp32Kernel { Small, Direct, Staged };
struct Fp32Choice {
  Fp32Kernel kernel = Fp32Kernel::Staged;
  double us = 0;
};
inline Fp32Choice gemm_fp32_choice(const GemmShape& s, long long cus, bool may_small = true) {
  const double never = std::numeric_limits<double>::infinity();
  const bool direct = gemm_direct_ok(s);
  const double small = may_small && gemm_small_ok(s) ? gemm_small_us(s, cus) : never;
  const double tiled = direct ? gemm_direct_us(s, cus) : gemm_staged_us(s, cus);
  if (small <= tiled) return {Fp32Kernel::Small, small};
  return {direct ? Fp32Kernel::Direct : Fp32Kernel::Staged, tiled};
}

// ---- the bf16 matrix cores (gemm_split.hip)

// Operand forms. ALIGNED: K % 32 == 0, 16-byte aligned rows, and [K x N] B with N %
// 8 == 0. ANY: any K and element alignment ([K x N] B: N % 8 == 0). SHIFT: [K x N]
// B with any N >= 8: the last column chunk of a row, when it crosses N, is
// read 8 columns before the row's end and shifted into place.
enum Form { ALIGNED, ANY, SHIFT };
inline Form gemm_split_form(const GemmShape& s) {
  if (!s.b_nk && s.N % 8 != 0) return SHIFT;
  if (s.K % kGemmKTile != 0 || !s.a16 || !s.b16 || (s.b_nk ? s.K : s.N) % (s.half_b ? 8 : 4) != 0)
    return ANY;
  return ALIGNED;
}

// How a call is cut: whole rounds of tiles (one per resident workgroup) run one
// per workgroup, and the tiles past them either as one more round or, split by
// K, evenly over up to one workgroup per CU (records and a fix-up pass).
struct Cut {
  double us = 0;        // estimated time
  long long split = 0;  // workgroups sharing the tail tiles (0: not split)
};

// Estimated time of a tiling: `step` is a workgroup's time per K tile on a full
// chip, `fill` what a round costs besides (first loads, stores), `rec` what one
// split workgroup's record adds (written, read back). A split costs the fix-up
// launch and another fill, about 8 us, and 3 more where workgroups cross from
// one tile into the next.
inline Cut cut_of(long long M, long long N, long long nk, long long bm, long long bn, double step,
           double fill, double rec, long long cus, bool may_split) {
  const long long tiles = ((M + bm - 1) / bm) * ((N + bn - 1) / bn);
  const long long tail = tiles % cus;
  const double round = static_cast<double>(nk) * step + fill;
  Cut c;
  c.us = static_cast<double>((tiles + cus - 1) / cus) * round;
  if (may_split && tail != 0 && nk >= 16 && tiles < 2 * cus) {
    // at least 8 K tiles each
    const long long w = std::max<long long>(tail, std::min(cus, tail * nk / 8));
    const double us = static_cast<double>(tiles / cus) * round + fill +
                      static_cast<double>(tail * nk) / static_cast<double>(w) * step + 8.0 +
                      rec * static_cast<double>(w) + (w % tail != 0 ? 3.0 : 0.0);
    if (w > tail && us < c.us) c.us = us, c.split = w;
  }
  return c;
}

// The tiling of the smallest estimated time. Microseconds per K tile and
// workgroup, measured with every CU busy (4096^3, 2048^3 and 512 x 4096 x 4096):
//   256 x 128, 8 waves of 64 x 64                2.46  (4096^3: 629 us, 218 TFLOP/s)
//   128 x 128, 8 waves of 64 x 32                1.39  (2048^3: 91 us, 189 TFLOP/s)
//   128 x 64, two groups of 4 waves of 64 x 32   0.83  (512 x 4096 x 4096: 104 us)
//   64 x 64, two groups of 4 waves of 32 x 32    0.52  (1024^3: 20 us)
// against the FP32 instruction's kernels, which stay ahead where one round of
// their small tiles holds the whole call (1024^3: 17.9 us, 512^3: 5.6).
struct SplitChoice {
  int bm = 0, bn = 0;
  Cut cut;
};
inline SplitChoice gemm_split_choice(const GemmShape& s, long long cus, bool may_split = true) {
  struct Tiling {
    int bm, bn;
    double step, fill, rec;
  };
  constexpr Tiling kTilings[] = {{256, 128, 2.46, 5.0, 0.05},
                                 {128, 128, 1.39, 3.5, 0.02},
                                 {128, 64, 0.83, 3.0, 0.01},
                                 {64, 64, 0.52, 2.0, 0.005}};
  const long long nk = (s.K + kGemmKTile - 1) / kGemmKTile;
  const double part = s.K % kGemmKTile != 0 ? 1.5 : 0.0;  // the partial K tile, by itself
  SplitChoice best;
  // (the kernel counts k in 32 bits, up to 256 past the end)
  if (s.K > 0x7fffffffLL - 1024) {
    best.cut.us = std::numeric_limits<double>::infinity();
    return best;
  }
  for (const Tiling& t : kTilings) {
    const Cut c = cut_of(s.M, s.N, nk, t.bm, t.bn, t.step, t.fill + part, t.rec, cus, may_split);
    if (best.bm == 0 || c.us < best.cut.us) best = {t.bm, t.bn, c};
  }
  return best;
}

// ---- few-row linear layers, fp16 weights [N x K] (few_rows.hip)

constexpr int kFewBlock = 512;  // k of a block

// Estimated microseconds with rt x 16 weight rows per workgroup, at up to 16
// and 17 to 32 activation rows: per block and round, measured at 11008 x 4096
// (rt 3), 4096 x 4096 and 4096 x 11008 (rt 1).
struct Few {
  int rt = 0;
  double us16 = 0, us32 = 0;
};
inline Few few_of(long long N, long long K, long long cus) {
  const double blocks = static_cast<double>((K + kFewBlock - 1) / kFewBlock);
  constexpr double kPer16[3] = {1.35, 1.8, 2.2};
  constexpr double kPer32[3] = {2.6, 3.0, 3.45};
  Few best;
  for (int rt = 1; rt <= 3; ++rt) {
    const double rounds = static_cast<double>(((N + 16 * rt - 1) / (16 * rt) + cus - 1) / cus);
    const Few f{rt, 3.2 + rounds * blocks * kPer16[rt - 1], 3.2 + rounds * blocks * kPer32[rt - 1]};
    if (best.rt == 0 || f.us16 < best.us16) best = f;
  }
  return best;
}

// Where it is estimated ahead of the stream-K few-row kernel (about 8 us plus
// the weights at 5 TB/s up to 16 rows, 9 us plus the weights at 3.3 TB/s up to
// 32) for both row ranges: the choice may not depend on M, whose rows keep
// their bits. Up to one unit of 128 k that kernel splits nothing and needs no
// reduce either (20 x 8256 x 128: 5.7 us against 8.8 here; x 256 9.4 against 7.6).
inline bool few_rows_ahead(long long N, long long K, long long cus) {
  if (K <= 128) return false;
  const Few f = few_of(N, K, cus);
  const double mb = 2e-6 * static_cast<double>(N) * static_cast<double>(K);
  return f.us16 < 8.0 + mb / 5.0 && f.us32 < 9.0 + mb / 3.3;
}

}  // namespace eng
