// Causal grouped-query attention over the KV cache for the rows of a prompt (or of one token in
// the launch sequence), in fp32 like the reference's numpy path (`webtorch/_core.py:2234-2330`,
// `webtorch/llm.py:1619-1636`): token t sits at position pos0 + t (pos0 read from the device) and
// query head h attends to cache positions 0 .. pos0 + t of kv head h / (NH / NKV).
// scores = (q . k) * scale; p = exp(s - max) / sum; out = sum p v.
#include <math.h>

#include "miq_common.h"

namespace miq {

// Both products run on the fp32 matrix cores (v_mfma_f32_16x16x4_f32: fp32 operands and sums,
// twice the rate of the fp32 VALU without packed instructions), with an online softmax.
//
// A wave takes 16 query rows of one head and the key blocks wave, wave + NW, ... of KB keys, so
// the waves of a workgroup share the rows and split the keys, with no barrier until their
// (maximum, sum, output) meet in LDS. It multiplies transposed: S^T = K Q^T leaves lane
// (c, g) = (lane % 16, lane / 16) with query c's scores of keys 4 g + r (r < 4), and O^T = V^T P^T
// takes exactly those as its B operand in four steps, step r covering keys r, 4 + r, 8 + r,
// 12 + r: no value moves between lanes from the scores to the output, and a query's maximum and
// rescale factor are per-lane scalars. The order of a product's terms is free as long as both
// operands agree, so each lane reads 16 bytes at a time: of a key row, dims 16 j + 4 g ..
// (16 rows x 64 bytes per load); of a value row, dims 64 u + 4 c .. (4 rows x 256 bytes), which
// makes row 4 g + r' of output tile (u, t) dimension 64 u + 16 g + 4 r' + t: a lane ends with 16
// consecutive output dimensions per u.
//
// Blocks that reach past the tile's first position are masked: scores of later keys become -inf.
// Their probabilities are then 0, but 0 times a NaN or infinite value is NaN, so a masked block
// whose values are not all finite is added key by key on the VALU instead, masked keys skipped.
//
// Sums of p v are divided by sum p at the end, so up to LMAX values add up undivided: p is held
// times 2^-14 (exact, and gone with the division), which keeps them within the largest |v|.
//
// Bound: the fp32 matrix cores at long prompts, the round trips to the cache rows (the first
// block's issued before the position is known) at short ones. Against one wave per (head,
// token) with a score row in LDS, from position 0: 14 heads of 64, T = 64 6.1 -> 4.7 us, T = 700 138 -> 22,
// T = 2000 997 -> 92; 28 heads of 128, T = 700 499 -> 58, T = 2000 4264 -> 339 (88 TFLOP/s); one
// row behind 700 positions 37 -> 13 and 71 -> 19; up to 16 rows of heads of 64 lose 0.3-0.7 us there
// (3.2-3.9 -> 4.0-4.2): half of a 32-key block is empty, and skipping it cost longer prompts more.
constexpr int kAttWaves = 4;  // eight were slower from T = 700 on (T = 2000: 92 -> 106 us) and no faster below
constexpr int kAttMaxKeys = 16384;           // LMAX
constexpr float kAttUnit = 1.f / kAttMaxKeys;  // a probability of 1
typedef float f4 __attribute__((ext_vector_type(4)));

// the maximum over the four lanes c, c + 16, c + 32, c + 48
__device__ __forceinline__ float cross_max(float v) {
  const auto a = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  v = fmaxf(__uint_as_float(a[0]), __uint_as_float(a[1]));
  const auto b = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return fmaxf(__uint_as_float(b[0]), __uint_as_float(b[1]));
}
__device__ __forceinline__ float cross_sum(float v) {
  const auto a = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  v = __uint_as_float(a[0]) + __uint_as_float(a[1]);
  const auto b = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return __uint_as_float(b[0]) + __uint_as_float(b[1]);
}

template <int HD>
__global__ __launch_bounds__(64 * kAttWaves, 2) void attention_mma_kernel(
    const float* __restrict__ q, const float* __restrict__ kc, const float* __restrict__ vc,
    const int32_t* __restrict__ state, float* __restrict__ out, int T, int NH, int NKV, int LMAX, float scale) {
  constexpr int NW = kAttWaves;
  constexpr int KB = HD == 64 ? 32 : 16;  // keys per step (registers: K, V and the next K of a block)
  constexpr int NB = KB / 16, NC = HD / 16, NU = HD / 64, QR = 16;
  __shared__ __align__(16) float os[NW][QR][HD + 4];
  __shared__ float ms[NW][QR], ls[NW][QR];
  const int lane = threadIdx.x & 63, wave = uniform(threadIdx.x >> 6), c = lane & 15, g = lane >> 4;
  const int h = blockIdx.x;
  const int t0 = ((int)gridDim.y - 1 - (int)blockIdx.y) * QR;  // the longest tiles first
  const float* K = kc + (size_t)(h / (NH / NKV)) * LMAX * HD;
  const float* V = vc + (size_t)(h / (NH / NKV)) * LMAX * HD;
  const int t = min(t0 + c, T - 1);  // rows past T repeat the last row and are not stored

  f4 kf[NB][NC], kn[NB][NC], vf[NB][4][NU];
  auto load_k = [&](int blk, int end, f4(&kd)[NB][NC]) __attribute__((always_inline)) {
#pragma unroll
    for (int b = 0; b < NB; ++b) {
      const float* r = K + (size_t)min(blk * KB + 16 * b + c, end) * HD + 4 * g;
#pragma unroll
      for (int j = 0; j < NC; ++j) kd[b][j] = *reinterpret_cast<const f4*>(r + 16 * j);
    }
  };
  auto load_v = [&](int blk, int end) __attribute__((always_inline)) {
#pragma unroll
    for (int b = 0; b < NB; ++b)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const float* vr = V + (size_t)min(blk * KB + 16 * b + 4 * g + r, end) * HD + 4 * c;
#pragma unroll
        for (int u = 0; u < NU; ++u) vf[b][r][u] = *reinterpret_cast<const f4*>(vr + 64 * u);
      }
  };
  // the first block's rows before the position is known: rows past the last key are masked
  load_k(wave, LMAX - 1, kf);
  load_v(wave, LMAX - 1);
  f4 qf[NC];
#pragma unroll
  for (int j = 0; j < NC; ++j) qf[j] = *reinterpret_cast<const f4*>(q + ((size_t)t * NH + h) * HD + 16 * j + 4 * g);
  const int pos0 = state[0];
  const int lim = min(pos0 + t, LMAX - 1);                      // this query's last key
  const int first = min(pos0 + t0, LMAX - 1);                   // the tile's smallest last key
  const int S = min(pos0 + min(t0 + QR, T) - 1, LMAX - 1) + 1;  // keys any of its rows attends to
  const int nblk = (S + KB - 1) / KB;
  f4 o[4 * NU];
  float m = -INFINITY, l = 0.f;
#pragma unroll
  for (int u = 0; u < 4 * NU; ++u) o[u] = (f4){0.f, 0.f, 0.f, 0.f};
  for (int blk = wave; blk < nblk; blk += NW) {
    load_k(min(blk + NW, nblk - 1), S - 1, kn);
    f4 s[NB];
#pragma unroll
    for (int b = 0; b < NB; ++b) s[b] = (f4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int j = 0; j < NC; ++j)
#pragma unroll
      for (int e = 0; e < 4; ++e)
#pragma unroll
        for (int b = 0; b < NB; ++b) s[b] = __builtin_amdgcn_mfma_f32_16x16x4f32(kf[b][j][e], qf[j][e], s[b], 0, 0, 0);
    const bool masked = blk * KB + KB - 1 > first;  // wave-uniform
    float mx = -INFINITY;
#pragma unroll
    for (int b = 0; b < NB; ++b)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        float v = s[b][r] * scale;
        if (masked && blk * KB + 16 * b + 4 * g + r > lim) v = -INFINITY;
        s[b][r] = v;
        mx = fmaxf(mx, v);
      }
    const float mn = fmaxf(m, cross_max(mx));
    const float ref = mn == -INFINITY ? 0.f : mn;  // no key yet: every probability is 0
    const float alpha = expf(m - ref);
    m = mn;
    float ps = 0.f;
#pragma unroll
    for (int b = 0; b < NB; ++b)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const float p = expf(s[b][r] - ref) * kAttUnit;
        s[b][r] = p;
        ps += p;
      }
    l = l * alpha + ps;
#pragma unroll
    for (int u = 0; u < 4 * NU; ++u) o[u] *= alpha;
    bool finite = true;
    if (masked) {
      float z = 0.f;
#pragma unroll
      for (int b = 0; b < NB; ++b)
#pragma unroll
        for (int r = 0; r < 4; ++r)
#pragma unroll
          for (int u = 0; u < NU; ++u)
#pragma unroll
            for (int e = 0; e < 4; ++e) z = fmaf(0.f, vf[b][r][u][e], z);  // 0, or NaN
      finite = __ballot(z != z) == 0ull;
    }
    if (finite) {
#pragma unroll
      for (int b = 0; b < NB; ++b)
#pragma unroll
        for (int r = 0; r < 4; ++r)
#pragma unroll
          for (int u = 0; u < NU; ++u)
#pragma unroll
            for (int e = 0; e < 4; ++e)
              o[4 * u + e] = __builtin_amdgcn_mfma_f32_16x16x4f32(vf[b][r][u][e], s[b][r], o[4 * u + e], 0, 0, 0);
    } else {
      const int nk = min(KB, S - blk * KB);
      for (int k = 0; k < nk; ++k) {
        float pk = 0.f;
#pragma unroll
        for (int b = 0; b < NB; ++b)
#pragma unroll
          for (int r = 0; r < 4; ++r)  // key k is score k % 4 of lanes (k / 4) % 4 in group k / 16
            if (b == k / 16 && r == k % 4) pk = __shfl(s[b][r], (k & 12) * 4 + c, 64);
        const float* vr = V + (size_t)(blk * KB + k) * HD + 16 * g;
        if (blk * KB + k <= lim) {
#pragma unroll
          for (int u = 0; u < NU; ++u)
#pragma unroll
            for (int e = 0; e < 4; ++e)
#pragma unroll
              for (int r = 0; r < 4; ++r) o[4 * u + e][r] = fmaf(pk, vr[64 * u + 4 * r + e], o[4 * u + e][r]);
        }
      }
    }
    if (blk + NW >= nblk) break;
#pragma unroll
    for (int b = 0; b < NB; ++b)
#pragma unroll
      for (int j = 0; j < NC; ++j) kf[b][j] = kn[b][j];
    load_v(blk + NW, S - 1);
  }

  // ---- the waves' parts, rescaled to their common maximum ----
  const int nw = min(NW, nblk);  // waves that had keys (wave 0 always)
  if (wave < nw) {
    l = cross_sum(l);
    if (g == 0) {
      ms[wave][c] = m;
      ls[wave][c] = l;
    }
#pragma unroll
    for (int u = 0; u < NU; ++u)
#pragma unroll
      for (int r = 0; r < 4; ++r)
        *reinterpret_cast<f4*>(&os[wave][c][64 * u + 16 * g + 4 * r]) =
            (f4){o[4 * u][r], o[4 * u + 1][r], o[4 * u + 2][r], o[4 * u + 3][r]};
  }
  __syncthreads();
  for (int x = threadIdx.x; x < QR * (HD / 4); x += 64 * NW) {
    const int row = x / (HD / 4), d = 4 * (x % (HD / 4));
    if (t0 + row >= T) continue;
    float mx = ms[0][row];
    for (int w = 1; w < nw; ++w) mx = fmaxf(mx, ms[w][row]);
    const float ref = mx == -INFINITY ? 0.f : mx;
    f4 a = (f4){0.f, 0.f, 0.f, 0.f};
    float sum = 0.f;
    for (int w = 0; w < nw; ++w) {
      const float f = expf(ms[w][row] - ref);
      sum = fmaf(f, ls[w][row], sum);
      const f4 v = *reinterpret_cast<const f4*>(&os[w][row][d]);
#pragma unroll
      for (int e = 0; e < 4; ++e) a[e] = fmaf(f, v[e], a[e]);
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) a[e] = a[e] / sum;
    *reinterpret_cast<f4*>(out + ((size_t)(t0 + row) * NH + h) * HD + d) = a;
  }
}

// Any head dimension: one wave per (head, token), lanes over positions for the scores, lanes over
// the head dimension for the output.
__global__ __launch_bounds__(64) void attention_kernel(const float* __restrict__ q, const float* __restrict__ kc,
                                                       const float* __restrict__ vc, const int32_t* __restrict__ state,
                                                       float* __restrict__ out, int NH, int NKV, int HD, int LMAX,
                                                       float scale) {
  extern __shared__ float sp[];  // [LMAX] scores, then probabilities
  __shared__ float qs[256];
  const int h = blockIdx.x, t = blockIdx.y;
  const int lane = threadIdx.x;
  const int kv = h / (NH / NKV);
  int S = state[0] + t + 1;
  S = S > LMAX ? LMAX : S;
  for (int d = lane; d < HD; d += 64) qs[d] = q[((size_t)t * NH + h) * HD + d];
  __syncthreads();
  const float* K = kc + (size_t)kv * LMAX * HD;
  const float* Vv = vc + (size_t)kv * LMAX * HD;
  float mx = -INFINITY;
  for (int j = lane; j < S; j += 64) {
    const float* kr = K + (size_t)j * HD;
    float a = 0.f;
    for (int d = 0; d < HD; d += 4) {
      const float4 k4 = *reinterpret_cast<const float4*>(kr + d);
      a = fmaf(qs[d], k4.x, a);
      a = fmaf(qs[d + 1], k4.y, a);
      a = fmaf(qs[d + 2], k4.z, a);
      a = fmaf(qs[d + 3], k4.w, a);
    }
    a *= scale;
    sp[j] = a;
    mx = fmaxf(mx, a);
  }
  mx = wave_max(mx);
  float sum = 0.f;
  for (int j = lane; j < S; j += 64) {
    const float e = expf(sp[j] - mx);
    sp[j] = e;
    sum += e;
  }
  sum = wave_sum(sum);
  for (int j = lane; j < S; j += 64) sp[j] = sp[j] / sum;
  __syncthreads();
  for (int d = lane; d < HD; d += 64) {
    float o = 0.f;
    for (int j = 0; j < S; ++j) o = fmaf(sp[j], Vv[(size_t)j * HD + d], o);
    out[((size_t)t * NH + h) * HD + d] = o;
  }
}

}  // namespace miq

using namespace miq;

extern "C" int miq_attention(const float* q, const float* kcache, const float* vcache, const int32_t* state, float* out,
                             int T, int NH, int NKV, int HD, int LMAX, float scale, void* stream) {
  MIQ_REQUIRE(T >= 0 && NH > 0 && NKV > 0 && NH % NKV == 0 && HD > 0 && HD <= 256 && HD % 4 == 0 && LMAX > 0,
              MIQ_ERR_INVALID, "attention: T=%d NH=%d NKV=%d HD=%d LMAX=%d", T, NH, NKV, HD, LMAX);
  if (T == 0) return MIQ_OK;
  MIQ_REQUIRE(LMAX <= kAttMaxKeys, MIQ_ERR_UNSUPPORTED, "attention: LMAX=%d above %d", LMAX, kAttMaxKeys);
  MIQ_REQUIRE(q && kcache && vcache && state && out, MIQ_ERR_INVALID, "attention: null pointer");
  MIQ_REQUIRE(aligned(kcache, 16) && aligned(vcache, 16), MIQ_ERR_ALIGN, "attention: caches must be 16-byte aligned");
  const hipStream_t s = static_cast<hipStream_t>(stream);
  // the matrix-core kernel reads q rows and writes out rows 16 bytes at a time
  const int tiles = (T + 15) / 16;
  if ((HD == 64 || HD == 128) && aligned(q, 16) && aligned(out, 16) && tiles <= 65535) {
    const dim3 g((unsigned)NH, (unsigned)tiles), b(64 * kAttWaves);
    if (HD == 64)
      hipLaunchKernelGGL(attention_mma_kernel<64>, g, b, 0, s, q, kcache, vcache, state, out, T, NH, NKV, LMAX, scale);
    else
      hipLaunchKernelGGL(attention_mma_kernel<128>, g, b, 0, s, q, kcache, vcache, state, out, T, NH, NKV, LMAX, scale);
    return check_launch("attention");
  }
  hipLaunchKernelGGL(attention_kernel, dim3(NH, T), dim3(64), (size_t)LMAX * 4, s, q,
                     kcache, vcache, state, out, NH, NKV, HD, LMAX, scale);
  return check_launch("attention");
}

