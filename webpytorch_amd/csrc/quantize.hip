// Asymmetric min-max group quantizer (GPTQ layout, zero_offset 0), bit-exact with the
// reference's float32 numpy arithmetic: scale = (max - min) / qmax (0 -> 1e-8),
// zero = clip(rint(-min / scale), 0, qmax), code = clip(rint(w / scale) + zero, 0, qmax).
// Division is IEEE round-to-nearest and rint is round-half-even, as numpy's float32 ops.
#include "miq_common.h"

namespace miq {

// The codes' divisor: rint(v / s) for the values of one group. The correctly rounded quotient is
// an IEEE division sequence of about ten instructions; v * (1 / s) is within 2^-22 of it
// relatively (both roundings of the product's factors and the product), so the two round to the
// same integer unless the product lies that close to a half-integer. Only such values (and
// groups whose scale is so small or large that 1 / s is not a normal number) take the division.
struct Divisor {
  float s, r, tol;
  __device__ __forceinline__ explicit Divisor(float scale) : s(scale) {
    const bool normal = scale > 0x1p-100f && scale < 0x1p100f;
    r = 1.f / scale;
    tol = normal ? 0x1p-21f : INFINITY;
  }
  __device__ __forceinline__ float rint_quotient(float v) const {
    const float t = v * r;
    float n = rintf(t);
    // false for NaN, and for every value when tol is infinite (0 * inf is NaN)
    if (!(fabsf(t - n) < 0.5f - fabsf(t) * tol)) n = rintf(v / s);
    return n;
  }
};

// scale, zero point and divisor of one group from its minimum and maximum
template <int QMAX> __device__ __forceinline__ void group_params(float lo, float hi, float* s, float* zf) {
  *s = (hi - lo) / (float)QMAX;
  if (*s == 0.f) *s = 1e-8f;
  *zf = fminf(fmaxf(rintf(-lo / *s), 0.f), (float)QMAX);
}
template <int QMAX> __device__ __forceinline__ uint32_t code(float v, const Divisor& d, float zf) {
  return (uint32_t)fminf(fmaxf(d.rint_quotient(v) + zf, 0.f), (float)QMAX);
}

// W [N][K] (a checkpoint's (out, in) rows), groups of GS = 32, 64 or 128. HBM-bound: each value is
// read once, with 16-byte loads of consecutive k (a thread holds 8 consecutive values of one row,
// GS / 8 consecutive lanes a group, so the group's extrema are DPP moves), and the packed words,
// which the layout wants n-contiguous, are transposed through LDS and stored 256 bytes a wave.
// Workgroup: 64 rows x 256 k, eight passes of 8 rows whose loads are all issued at once (wider
// runs of k leave small layers too few workgroups). Against one thread per (group, column), whose
// loads of a wave were 64 rows apart and which divided every value: K = 4096, N = 14336 fp16,
// 128-value groups 1022 -> 39 us (3.8 TB/s).
constexpr int kRowsN = 64, kRowsK = 256;
template <int BITS, int GS, typename WT>
__global__ __launch_bounds__(256) void quantize_rows_kernel(const WT* __restrict__ W, int K, int N,
                                                            uint32_t* __restrict__ qweight,
                                                            uint32_t* __restrict__ qzeros, float* __restrict__ scales) {
  constexpr int PER = 32 / BITS, QMAX = (1 << BITS) - 1;
  constexpr int LPR = kRowsK / 8;              // lanes of one row
  constexpr int RPP = 256 / LPR, PASSES = kRowsN / RPP;
  constexpr int LPG = GS / 8;                  // lanes of one group
  constexpr int NW = kRowsK / PER, NG = kRowsK / GS, PADN = kRowsN + 1;
  __shared__ uint32_t words[NW * PADN];
  __shared__ float ss[NG * PADN];
  __shared__ uint32_t zs[NG * PADN];
  const int tid = threadIdx.x, c = tid % LPR, rr = tid / LPR;
  const int n0 = blockIdx.x * kRowsN, k0 = blockIdx.y * kRowsK, k = k0 + 8 * c;
  if (k < K) {  // K is whole groups, so a group's lanes are all in or all out
    float v[PASSES][8];
#pragma unroll
    for (int p = 0; p < PASSES; ++p) load8(W + (size_t)min(n0 + p * RPP + rr, N - 1) * K + k, v[p]);
#pragma unroll
    for (int p = 0; p < PASSES; ++p) {
      const int n = p * RPP + rr;
      float lo = v[p][0], hi = lo;
#pragma unroll
      for (int j = 1; j < 8; ++j) {
        lo = fminf(lo, v[p][j]);
        hi = fmaxf(hi, v[p][j]);
      }
      lo = fminf(lo, dpp_move<0xB1>(lo));
      hi = fmaxf(hi, dpp_move<0xB1>(hi));
      lo = fminf(lo, dpp_move<0x4E>(lo));
      hi = fmaxf(hi, dpp_move<0x4E>(hi));
      if constexpr (LPG >= 8) {  // row_half_mirror: the other quad of 8 lanes
        lo = fminf(lo, dpp_move<0x141>(lo));
        hi = fmaxf(hi, dpp_move<0x141>(hi));
      }
      if constexpr (LPG >= 16) {  // row_mirror: the other half of 16 lanes
        lo = fminf(lo, dpp_move<0x140>(lo));
        hi = fmaxf(hi, dpp_move<0x140>(hi));
      }
      float s, zf;
      group_params<QMAX>(lo, hi, &s, &zf);
      const Divisor d(s);
#pragma unroll
      for (int w = 0; w < 8 / PER; ++w) {
        uint32_t word = 0;
#pragma unroll
        for (int j = 0; j < PER; ++j) word |= code<QMAX>(v[p][PER * w + j], d, zf) << (j * BITS);
        words[(c * (8 / PER) + w) * PADN + n] = word;
      }
      if (c % LPG == 0) {
        ss[(c / LPG) * PADN + n] = s;
        zs[(c / LPG) * PADN + n] = (uint32_t)zf;
      }
    }
  }
  __syncthreads();
  const int n = tid % kRowsN, q = tid / kRowsN;  // a wave stores 64 consecutive columns of a row
  const int nw = min(NW, (K - k0) / PER), ng = min(NG, (K - k0) / GS);
  if (n0 + n < N) {
    for (int r = q; r < nw; r += 256 / kRowsN) qweight[(size_t)(k0 / PER + r) * N + n0 + n] = words[r * PADN + n];
    for (int g = q; g < ng; g += 256 / kRowsN) {
      scales[(size_t)(k0 / GS + g) * N + n0 + n] = ss[g * PADN + n];
      if (n % PER == 0) {  // N is whole packed words: the word's other columns exist
        uint32_t word = 0;
#pragma unroll
        for (int j = 0; j < PER; ++j) word |= zs[g * PADN + n + j] << (j * BITS);
        qzeros[(size_t)(k0 / GS + g) * (N / PER) + (n0 + n) / PER] = word;
      }
    }
  }
}

// W [K][N], groups of GS = 32, 64 or 128. A thread holds two adjacent columns of GS / 4 rows of a
// group (one load of 2 values per row, all issued at once); the four threads of a column pair
// meet in LDS for the group's extrema, so every value is read once. Workgroup: 128 columns x one
// group. K = 4096, N = 14336: fp16 108 -> 30 us, fp32 115 -> 48 us (5.6 TB/s).
constexpr int kColsN = 128;
template <int BITS, int GS, typename WT>
__global__ __launch_bounds__(256) void quantize_cols_kernel(const WT* __restrict__ W, int K, int N,
                                                            uint32_t* __restrict__ qweight,
                                                            uint32_t* __restrict__ qzeros, float* __restrict__ scales) {
  constexpr int PER = 32 / BITS, QMAX = (1 << BITS) - 1, R = GS / 4;
  __shared__ float2 lo_s[4][64], hi_s[4][64];
  __shared__ uint32_t zs[kColsN];
  const int lane = threadIdx.x & 63, part = threadIdx.x >> 6, g = blockIdx.y;
  const int n = blockIdx.x * kColsN + 2 * lane;
  const bool ok = n < N;  // N is even
  float a[R], b[R];
  const WT* src = W + ((size_t)g * GS + part * R) * N + min(n, N - 2);
#pragma unroll
  for (int i = 0; i < R; ++i) {
    if constexpr (sizeof(WT) == 2) {
      const uint32_t t = *reinterpret_cast<const uint32_t*>(src + (size_t)i * N);
      a[i] = to_f32(__ushort_as_half((unsigned short)(t & 0xFFFFu)));
      b[i] = to_f32(__ushort_as_half((unsigned short)(t >> 16)));
    } else {
      const float2 t = *reinterpret_cast<const float2*>(src + (size_t)i * N);
      a[i] = t.x;
      b[i] = t.y;
    }
  }
  float2 lo = make_float2(a[0], b[0]), hi = lo;
#pragma unroll
  for (int i = 1; i < R; ++i) {
    lo = make_float2(fminf(lo.x, a[i]), fminf(lo.y, b[i]));
    hi = make_float2(fmaxf(hi.x, a[i]), fmaxf(hi.y, b[i]));
  }
  lo_s[part][lane] = lo;
  hi_s[part][lane] = hi;
  __syncthreads();
#pragma unroll
  for (int p = 0; p < 4; ++p) {
    const float2 l = lo_s[p][lane], h = hi_s[p][lane];
    lo = make_float2(fminf(lo.x, l.x), fminf(lo.y, l.y));
    hi = make_float2(fmaxf(hi.x, h.x), fmaxf(hi.y, h.y));
  }
  float2 s, zf;
  group_params<QMAX>(lo.x, hi.x, &s.x, &zf.x);
  group_params<QMAX>(lo.y, hi.y, &s.y, &zf.y);
  const Divisor dx(s.x), dy(s.y);
  if (ok) {
#pragma unroll
    for (int r = 0; r < R / PER; ++r) {
      uint2 w = make_uint2(0u, 0u);
#pragma unroll
      for (int j = 0; j < PER; ++j) {
        w.x |= code<QMAX>(a[r * PER + j], dx, zf.x) << (j * BITS);
        w.y |= code<QMAX>(b[r * PER + j], dy, zf.y) << (j * BITS);
      }
      *reinterpret_cast<uint2*>(qweight + ((size_t)g * (GS / PER) + part * (R / PER) + r) * N + n) = w;
    }
  }
  if (part == 0) {
    if (ok) *reinterpret_cast<float2*>(scales + (size_t)g * N + n) = s;
    zs[2 * lane] = (uint32_t)zf.x;
    zs[2 * lane + 1] = (uint32_t)zf.y;
  }
  __syncthreads();
  const int cw = threadIdx.x * PER, nz = blockIdx.x * kColsN + cw;  // first column of a zero word
  if (threadIdx.x < kColsN / PER && nz < N) {
    uint32_t word = 0;
#pragma unroll
    for (int j = 0; j < PER; ++j) word |= zs[cw + j] << (j * BITS);
    qzeros[(size_t)g * (N / PER) + nz / PER] = word;
  }
}

// Any group size and alignment: one thread per (group, column). W is [K][N] (from_out_in = 0) or [N][K] (= 1), fp16/fp32.
// Codes are packed per thread (a column's rows are in one thread); zero points are packed
// along N through LDS by the lane that owns the first column of each word.
template <int BITS, typename WT>
__global__ __launch_bounds__(256) void gptq_quantize_kernel(const WT* __restrict__ W, int from_out_in, int K, int N,
                                                            int gs, uint32_t* __restrict__ qweight,
                                                            uint32_t* __restrict__ qzeros, float* __restrict__ scales) {
  constexpr int PER = 32 / BITS;
  constexpr int QMAX = (1 << BITS) - 1;
  __shared__ uint32_t zs[256];
  const int n = blockIdx.x * blockDim.x + threadIdx.x;
  const int g = blockIdx.y;
  uint32_t zp = 0;
  if (n < N) {
    auto at = [&](int k) -> float {
      return to_f32(from_out_in ? W[(size_t)n * K + k] : W[(size_t)k * N + n]);
    };
    const int k0 = g * gs;
    float lo = at(k0), hi = lo;
    for (int k = k0 + 1; k < k0 + gs; ++k) {
      const float v = at(k);
      lo = fminf(lo, v);
      hi = fmaxf(hi, v);
    }
    float s = (hi - lo) / (float)QMAX;
    if (s == 0.f) s = 1e-8f;
    float zf = rintf(-lo / s);
    zf = fminf(fmaxf(zf, 0.f), (float)QMAX);
    zp = (uint32_t)zf;
    scales[(size_t)g * N + n] = s;
    for (int r = k0 / PER; r < (k0 + gs) / PER; ++r) {
      uint32_t word = 0;
#pragma unroll
      for (int j = 0; j < PER; ++j) {
        float c = rintf(at(r * PER + j) / s) + zf;
        c = fminf(fmaxf(c, 0.f), (float)QMAX);
        word |= (uint32_t)c << (j * BITS);
      }
      qweight[(size_t)r * N + n] = word;
    }
  }
  zs[threadIdx.x] = zp;
  __syncthreads();
  if (n < N && (n % PER) == 0) {
    uint32_t word = 0;
#pragma unroll
    for (int j = 0; j < PER; ++j) word |= zs[threadIdx.x + j] << (j * BITS);
    qzeros[(size_t)g * (N / PER) + n / PER] = word;
  }
}

// The single-pass kernel of W's layout, for the group sizes they are built for and buffers
// aligned for their loads and stores (16-byte rows; column pairs); false: not covered.
template <int BITS, typename WT>
static bool quantize_fast(const WT* W, int from_out_in, int K, int N, int gs, uint32_t* qw, uint32_t* qz, float* sc,
                          hipStream_t st) {
  const int ny = (from_out_in ? (K + kRowsK - 1) / kRowsK : K / gs);
  if (ny > 65535) return false;
  if (from_out_in ? !(aligned(W, 16) && K % 8 == 0)
                  : !(aligned(W, 2 * sizeof(WT)) && aligned(qw, 8) && aligned(sc, 8) && N % 2 == 0))
    return false;
  const dim3 g((unsigned)(from_out_in ? (N + kRowsN - 1) / kRowsN : (N + kColsN - 1) / kColsN), (unsigned)ny);
  auto go = [&](auto rows, auto cols) {
    hipLaunchKernelGGL(from_out_in ? rows : cols, g, dim3(256), 0, st, W, K, N, qw, qz, sc);
    return true;
  };
  switch (gs) {
    case 32: return go(quantize_rows_kernel<BITS, 32, WT>, quantize_cols_kernel<BITS, 32, WT>);
    case 64: return go(quantize_rows_kernel<BITS, 64, WT>, quantize_cols_kernel<BITS, 64, WT>);
    case 128: return go(quantize_rows_kernel<BITS, 128, WT>, quantize_cols_kernel<BITS, 128, WT>);
    default: return false;
  }
}

}  // namespace miq

using namespace miq;

extern "C" int miq_gptq_quantize(const void* W, int w_dtype, int from_out_in, int K, int N, int gs, int bits,
                                 int32_t* qweight, int32_t* qzeros, float* scales, void* stream) {
  MIQ_REQUIRE(bits == 4 || bits == 8, MIQ_ERR_UNSUPPORTED, "gptq_quantize: bits=%d", bits);
  const int per = 32 / bits;
  MIQ_REQUIRE(K > 0 && N > 0 && gs > 0 && K % gs == 0 && K % per == 0 && N % per == 0 && gs % per == 0,
              MIQ_ERR_INVALID, "gptq_quantize: dims must divide group/pack size (K=%d N=%d gs=%d)", K, N, gs);
  MIQ_REQUIRE(W && qweight && qzeros && scales, MIQ_ERR_INVALID, "gptq_quantize: null pointer");
  dim3 grid((N + 255) / 256, K / gs);
  hipStream_t st = static_cast<hipStream_t>(stream);
  uint32_t* qw = reinterpret_cast<uint32_t*>(qweight);
  uint32_t* qz = reinterpret_cast<uint32_t*>(qzeros);
#define MIQ_Q(B, T)                                                                                          \
  if (!quantize_fast<B, T>(static_cast<const T*>(W), from_out_in, K, N, gs, qw, qz, scales, st))             \
  hipLaunchKernelGGL((gptq_quantize_kernel<B, T>), grid, dim3(256), 0, st, static_cast<const T*>(W), from_out_in, K, N, \
                     gs, qw, qz, scales)
  if (bits == 4) {
    if (w_dtype == MIQ_F16) { MIQ_Q(4, __half); } else { MIQ_Q(4, float); }
  } else {
    if (w_dtype == MIQ_F16) { MIQ_Q(8, __half); } else { MIQ_Q(8, float); }
  }
#undef MIQ_Q
  return check_launch("gptq_quantize");
}
