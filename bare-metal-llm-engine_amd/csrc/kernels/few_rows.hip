// few_rows.hip -- RMSNorm + linear over 5 to 32 activation rows, fp16 weights
// output-major, in one launch: Y[M x N] = s_m (X[m] * gamma) . W^T, W [N x K].
//
// A workgroup of 16 waves owns 16 RT weight rows over the whole of K, so
// nothing is split between workgroups (no records, no second launch). Weights
// come in blocks of 512 k, three stages deep: every load instruction brings a
// whole 1 KiB piece of one row straight into LDS (long runs of a row stream
// faster than the matrix instruction's own 64-byte pieces of 16 rows), and wave
// w multiplies the block's k slice 32 w .. + 31 against all of the rows. A wave
// therefore needs only its own slice of X: it loads it as fp32 straight into the
// operand's lanes, a block or two ahead, and splits it in registers: no X in
// LDS, and one barrier per 512 k. The 16 waves' sums are added through LDS in
// wave order at the end.
//
// The activations enter v_mfma_f32_16x16x32_f16 as three fp16 terms per row
// and 32-deep slice: t = x' 2^e with the slice's largest |t| in [2^14, 2^15), h,
// l, l2 the successive truncations of t to fp16, which add up to t exactly (each
// x' whose bits reach no lower than 2^-39 of the slice's largest); each product
// is exact in fp32, and the slice's sum times 2^-e is added to the running fp32
// sum. A row's arithmetic depends on N, K and the CU count only, so its bits are
// the same in any batch of 5 to 32 rows.
//
// What bounds it: the CU's load path. Each workgroup reads all of X (L2) beside
// its weights, 256 KiB against 384 KiB at 16 x 11008 x 4096: 20.8 us there over
// three weight buffers (26.2 on the stream-K few-row kernel and its reduce), 18.0
// at 5 rows, 30.7 at 32 (36.6), and with cold weights 24.0 (26.7), 22.1 (26.1) and
// 33.8 (36.5); with 16 weight rows per workgroup X outweighs the weights
// (4096 x 11008: 32 against 26.5 us), which is where few_rows_ahead draws
// the line.
#include "device_sync.hpp"
#include "gemm_choice.hpp"
#include "launch.hpp"

#include <algorithm>

namespace eng {
namespace {

typedef float floatx4 __attribute__((ext_vector_type(4)));
typedef _Float16 halfx8 __attribute__((ext_vector_type(8)));
typedef _Float16 halfx2 __attribute__((ext_vector_type(2)));

// Maximum of v over the four lanes j, j + 16, j + 32, j + 48, in all of them.
__device__ __forceinline__ float max4(float v) {
#if defined(__HIP_DEVICE_COMPILE__)
  // each swap leaves this lane's value and its partner's in the two results
  // (copied to scalars: bit-casting the elements in place read one of them twice)
  const unsigned u = __float_as_uint(v);
  const auto a = __builtin_amdgcn_permlane16_swap(u, u, false, false);
  const unsigned a0 = a[0], a1 = a[1];
  v = fmaxf(__uint_as_float(a0), __uint_as_float(a1));
  const unsigned w = __float_as_uint(v);
  const auto b = __builtin_amdgcn_permlane32_swap(w, w, false, false);
  const unsigned b0 = b[0], b1 = b[1];
  v = fmaxf(__uint_as_float(b0), __uint_as_float(b1));
#endif
  return v;
}

// Two values truncated to fp16 (one instruction); r = v minus its fp16 term.
__device__ __forceinline__ halfx2 trunc2(float a, float b) {
  return __builtin_bit_cast(halfx2, __builtin_amdgcn_cvt_pkrtz(a, b));
}

template <int WAVES, int RT, int MB, bool GAIN>
__global__ __launch_bounds__(64 * WAVES, WAVES / 4) void few_rows_nk_kernel(
    const _Float16* __restrict__ W, const float* __restrict__ x, const float* __restrict__ gamma,
    float* __restrict__ y, int M, long long N, int K, float eps) {
  constexpr int BLOCK = 32 * WAVES;     // k of a block

  constexpr int ROWS = 16 * RT;
  constexpr int STAGE = ROWS * BLOCK;   // halves
  constexpr int LOADS = STAGE / 512 / WAVES;  // direct loads per wave and block
  static_assert(LOADS * WAVES * 512 == STAGE, "staging shape");
  __shared__ __attribute__((aligned(1024))) _Float16 W0[STAGE];
  __shared__ __attribute__((aligned(1024))) _Float16 W1[STAGE];
  __shared__ __attribute__((aligned(1024))) _Float16 W2[STAGE];
  __shared__ float ss_part[WAVES][16 * MB];
  __shared__ float row_scale[16 * MB];
  auto stage = [&](auto st) -> _Float16* {
    if constexpr (decltype(st)::value == 0) return W0;
    else if constexpr (decltype(st)::value == 1) return W1;
    else return W2;
  };

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x) >> 6);
  const int j = lane & 15;
  const int s = lane >> 4;
  const long long n0 = static_cast<long long>(blockIdx.x) * ROWS;
  const int blocks = (K + BLOCK - 1) / BLOCK;

  // Load i of a wave fills the 64 chunks (8 values of k) from slot (WAVES i +
  // wave) 64 of the stage; chunk c of row r sits at position c ^ (r % 16) of the
  // row, so the 16 rows of an operand read fall in 16 distinct bank groups.
  // Rows past N read row N - 1, chunks past K chunk 0 of their row.
  constexpr int CPR = BLOCK / 8;  // chunks per row
  const _Float16* wrow[LOADS];
  int wk[LOADS];  // this lane's k within a block
#pragma unroll
  for (int i = 0; i < LOADS; ++i) {
    const int slot = (WAVES * i + wave) * 64 + lane;
    const int r = slot / CPR;
    wrow[i] = W + std::min(n0 + r, N - 1) * K;
    wk[i] = 8 * ((slot % CPR) ^ (r & 15));
  }
  auto fetch = [&](auto st, int b) {
#pragma unroll
    for (int i = 0; i < LOADS; ++i) {
      const int k = b * BLOCK + wk[i];
      dma16(wrow[i] + (k < K ? k : 0), stage(st) + (WAVES * i + wave) * 512);
    }
  };

  // This lane's X: row 16 mb + j at k = BLOCK b + 32 wave + 8 s .. + 7.
  const float* xrow[MB];
#pragma unroll
  for (int mb = 0; mb < MB; ++mb)
    xrow[mb] = x + static_cast<long long>(std::min(16 * mb + j, M - 1)) * K;
  const int xk = 32 * wave + 8 * s;
  struct XSet {
    floatx4 v[MB][2];
    floatx4 g[GAIN ? 2 : 1];
  };
  auto load_x = [&](XSet& X, int b) {
    const int k = b * BLOCK + xk;
    const int ko = k < K ? k : 0;
#pragma unroll
    for (int mb = 0; mb < MB; ++mb) {
      X.v[mb][0] = *reinterpret_cast<const floatx4*>(xrow[mb] + ko);
      X.v[mb][1] = *reinterpret_cast<const floatx4*>(xrow[mb] + ko + 4);
    }
    if constexpr (GAIN) {
      X.g[0] = *reinterpret_cast<const floatx4*>(gamma + ko);
      X.g[1] = *reinterpret_cast<const floatx4*>(gamma + ko + 4);
    }
  };

  floatx4 acc[RT][MB];
#pragma unroll
  for (int r = 0; r < RT; ++r)
#pragma unroll
    for (int mb = 0; mb < MB; ++mb) acc[r][mb] = floatx4{0.0f, 0.0f, 0.0f, 0.0f};
  float ss[MB];
#pragma unroll
  for (int mb = 0; mb < MB; ++mb) ss[mb] = 0.0f;

  // masked: the block may reach past K (lanes there take zeros on both sides)
  auto compute = [&](const XSet& X, const _Float16* ws, int b, auto masked) {
    const bool kok = !decltype(masked)::value || b * BLOCK + xk < K;
    halfx8 w[RT];
#pragma unroll
    for (int r = 0; r < RT; ++r) {
      const halfx8 v = *reinterpret_cast<const halfx8*>(ws + (16 * r + j) * BLOCK +
                                                        8 * ((4 * wave + s) ^ j));
      w[r] = kok ? v : halfx8{};
    }
#pragma unroll
    for (int mb = 0; mb < MB; ++mb) {
      float t[8];
      float amax = 0.0f;
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const float v = kok ? X.v[mb][e >> 2][e & 3] : 0.0f;
        ss[mb] = fmaf(v, v, ss[mb]);
        t[e] = v;
        if constexpr (GAIN) t[e] = v * X.g[e >> 2][e & 3];
        amax = fmaxf(amax, fabsf(t[e]));
      }
      amax = max4(amax);
      // up = 2^(14 - floor(log2 amax)), at most 2^126; down its reciprocal (a
      // zero, infinite or NaN slice keeps an up that makes no new special value)
      const int ex = (__builtin_bit_cast(int, amax) >> 23) & 255;
      const float up = __builtin_bit_cast(float, (ex == 255 ? 127 : min(268 - ex, 253)) << 23);
      const float down = __builtin_bit_cast(float, (ex == 255 ? 127 : 254 - min(268 - ex, 253)) << 23);
      halfx8 h, l, l2;
#pragma unroll
      for (int e = 0; e < 8; e += 2) {
        const float a = t[e] * up;
        const float c = t[e + 1] * up;
        const halfx2 h2 = trunc2(a, c);
        const float ra = a - static_cast<float>(h2[0]);
        const float rc = c - static_cast<float>(h2[1]);
        const halfx2 m2 = trunc2(ra, rc);
        const halfx2 q2 = trunc2(ra - static_cast<float>(m2[0]), rc - static_cast<float>(m2[1]));
        h[e] = h2[0], h[e + 1] = h2[1];
        l[e] = m2[0], l[e + 1] = m2[1];
        l2[e] = q2[0], l2[e + 1] = q2[1];
      }
      const floatx4 zero = floatx4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
      for (int r = 0; r < RT; ++r) {
        const floatx4 ph = __builtin_amdgcn_mfma_f32_16x16x32_f16(w[r], h, zero, 0, 0, 0);
        floatx4 p = __builtin_amdgcn_mfma_f32_16x16x32_f16(w[r], l2, zero, 0, 0, 0);
        p = __builtin_amdgcn_mfma_f32_16x16x32_f16(w[r], l, p, 0, 0, 0);
        p += ph;  // (an fp32 add: the instruction rounds a C operand more coarsely)
#pragma unroll
        for (int v = 0; v < 4; ++v) acc[r][mb][v] = fmaf(p[v], down, acc[r][mb][v]);
      }
    }
  };

  // Block b: its pieces and X have landed and every wave has read block b - 1;
  // X of block b + 1 and then the pieces of block b + 2 are issued (loads
  // complete in order: waiting for X leaves the younger pieces in flight), then
  // block b is computed. Past the last block the loads read block 0 again.
  // Only the loop's steps count X loads among those that may still be in flight:
  // there every set is used by a later step. A set loaded in the last steps may
  // be used by none, and its loads are then not in the compiled code, so those
  // steps allow the pieces alone.
  constexpr int XD = MB == 1 ? 2 : 1;  // blocks X is loaded ahead
  [[maybe_unused]] constexpr int XL = 2 * MB + (GAIN ? 2 : 0);
  XSet x0, x1, x2;
  auto step = [&](auto st, XSet& X, XSet& Y, int b, auto masked) {
    using Prev = std::integral_constant<int, (decltype(st)::value + 2) % 3>;
#if defined(__HIP_DEVICE_COMPILE__)
    constexpr int ahead = decltype(masked)::value ? 0 : (XD - 1) * XL;
    __builtin_amdgcn_s_waitcnt(vmcnt_le(LOADS + ahead));
#endif
    __builtin_amdgcn_sched_barrier(0);
    barrier_no_fence();
    __builtin_amdgcn_sched_barrier(0);
    load_x(Y, b + XD < blocks ? b + XD : 0);
    __builtin_amdgcn_sched_barrier(0);
    fetch(Prev{}, b + 2 < blocks ? b + 2 : 0);
    __builtin_amdgcn_sched_barrier(0);
    compute(X, stage(st), b, masked);
    __builtin_amdgcn_sched_barrier(0);
  };
  using I0 = std::integral_constant<int, 0>;
  using I1 = std::integral_constant<int, 1>;
  using I2 = std::integral_constant<int, 2>;
  using std::false_type;
  using std::true_type;
  const int whole = K / BLOCK;
  int b = 0;
  if constexpr (XD == 2) {
    load_x(x0, 0);
    __builtin_amdgcn_sched_barrier(0);
    fetch(I0{}, 0);
    __builtin_amdgcn_sched_barrier(0);
    load_x(x1, blocks > 1 ? 1 : 0);
    __builtin_amdgcn_sched_barrier(0);
    fetch(I1{}, blocks > 1 ? 1 : 0);
    __builtin_amdgcn_sched_barrier(0);
    for (; b + 2 < whole; b += 3) {
      step(I0{}, x0, x2, b, false_type{});
      step(I1{}, x1, x0, b + 1, false_type{});
      step(I2{}, x2, x1, b + 2, false_type{});
    }
    if (b < blocks) step(I0{}, x0, x2, b, true_type{});
    if (b + 1 < blocks) step(I1{}, x1, x0, b + 1, true_type{});
    if (b + 2 < blocks) step(I2{}, x2, x1, b + 2, true_type{});
  } else {
    fetch(I0{}, 0);
    __builtin_amdgcn_sched_barrier(0);
    load_x(x0, 0);
    __builtin_amdgcn_sched_barrier(0);
    fetch(I1{}, blocks > 1 ? 1 : 0);
    __builtin_amdgcn_sched_barrier(0);
    for (; b + 5 < whole; b += 6) {
      step(I0{}, x0, x1, b, false_type{});
      step(I1{}, x1, x0, b + 1, false_type{});
      step(I2{}, x0, x1, b + 2, false_type{});
      step(I0{}, x1, x0, b + 3, false_type{});
      step(I1{}, x0, x1, b + 4, false_type{});
      step(I2{}, x1, x0, b + 5, false_type{});
    }
    if (b < blocks) step(I0{}, x0, x1, b, true_type{});
    if (b + 1 < blocks) step(I1{}, x1, x0, b + 1, true_type{});
    if (b + 2 < blocks) step(I2{}, x0, x1, b + 2, true_type{});
    if (b + 3 < blocks) step(I0{}, x1, x0, b + 3, true_type{});
    if (b + 4 < blocks) step(I1{}, x0, x1, b + 4, true_type{});
    if (b + 5 < blocks) step(I2{}, x1, x0, b + 5, true_type{});
  }
#if defined(__HIP_DEVICE_COMPILE__)
  __builtin_amdgcn_s_waitcnt(0);
#endif

  // Sums of squares: over the row's four lanes, then the waves.
#pragma unroll
  for (int mb = 0; mb < MB; ++mb) {
    float v = ss[mb];
    v += __shfl_xor(v, 16);
    v += __shfl_xor(v, 32);
    if (s == 0) ss_part[wave][16 * mb + j] = v;
  }
  __syncthreads();
  if (threadIdx.x < 16 * MB) {
    float tot = 0.0f;
#pragma unroll
    for (int w = 0; w < WAVES; ++w) tot += ss_part[w][threadIdx.x];
    row_scale[threadIdx.x] = 1.0f / sqrtf(tot / static_cast<float>(K) + eps);
  }
  // The waves' sums, one m-block at a time (accumulator element v of lane (j, s):
  // weight row 4 s + v, activation row j).
  constexpr int HALF = WAVES * RT * 64 * 16 <= STAGE * 2 ? WAVES : WAVES / 2;  // waves the stage holds
  static_assert(HALF * RT * 64 * 16 <= STAGE * 2, "the sums fit a stage");
  static_assert(HALF == WAVES || HALF * 2 == WAVES, "one or two stages");
  floatx4* red0 = reinterpret_cast<floatx4*>(W0);
  floatx4* red1 = reinterpret_cast<floatx4*>(W1);
#pragma unroll
  for (int mb = 0; mb < MB; ++mb) {
    if (mb > 0) __syncthreads();
    floatx4* mine = (HALF == WAVES || wave < HALF ? red0 + wave * RT * 64 : red1 + (wave - HALF) * RT * 64) + lane;
#pragma unroll
    for (int r = 0; r < RT; ++r) mine[r * 64] = acc[r][mb];
    __syncthreads();
    for (int t = threadIdx.x; t < RT * 256; t += 64 * WAVES) {
      const int i = t & 15;
      const int r = (t >> 4) % RT;
      const int m = (t >> 4) / RT;
      const int at = (r * 64 + m + 16 * (i >> 2)) * 4 + (i & 3);
      float v = 0.0f;
#pragma unroll
      for (int w = 0; w < WAVES; ++w)
        v += (w < HALF ? reinterpret_cast<const float*>(red0) + w * RT * 256
                       : reinterpret_cast<const float*>(red1) + (w - HALF) * RT * 256)[at];
      const long long n = n0 + 16 * r + i;
      const int row = 16 * mb + m;
      if (row < M && n < N) y[static_cast<long long>(row) * N + n] = v * row_scale[row];
    }
  }
}

template <int WAVES, int RT, int MB>
void run(const SkinnyArgs& a, hipStream_t stream) {
  const long long grid = (a.N + 16 * RT - 1) / (16 * RT);
  ENG_CHECK(grid <= 0x7fffffffLL, "linear: grid too large for one launch");
  auto launch = [&](auto gain) {
    few_rows_nk_kernel<WAVES, RT, MB, decltype(gain)::value>
        <<<static_cast<unsigned>(grid), 64 * WAVES, 0, stream>>>(
            static_cast<const _Float16*>(a.W), a.x, a.gamma, a.y, static_cast<int>(a.M), a.N,
            static_cast<int>(a.K), a.eps);
  };
  if (a.gamma != nullptr) launch(std::true_type{});
  else launch(std::false_type{});
  ENG_LAUNCH_CHECK();
}

}  // namespace

bool few_rows_nk_applies(const SkinnyArgs& a) {
  return a.w == Elem::F16 && a.w_nk && a.rms && a.K <= 0x7fffffffLL - kFewBlock &&
         few_rows_ahead(a.N, a.K, device_cu_count());
}

void launch_few_rows_nk(const SkinnyArgs& a, hipStream_t stream) {
  const int rt = few_of(a.N, a.K, device_cu_count()).rt;
  auto go = [&](auto mb) {
    constexpr int MB = decltype(mb)::value;
    if (rt == 3) run<16, 3, MB>(a, stream);
    else if (rt == 2) run<16, 2, MB>(a, stream);
    else run<16, 1, MB>(a, stream);
  };
  if (a.M <= 16) go(std::integral_constant<int, 1>{});
  else go(std::integral_constant<int, 2>{});
}

}  // namespace eng
