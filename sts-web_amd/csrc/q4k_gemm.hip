// q4k_gemm.hip -- Q4_K products for more than one row on the bf16 matrix cores (gfx950).
//
// Y[m][n] = sum_k W[n][k] X[m][k] with W in Q4_K (q4k_matmul with M > 1,
// crates/sts-wasm/src/gguf.rs:810-897, and the depformer's projections,
// depth_engine.rs:953-1360).  f32 results without f32 matrix instructions:
//
//   W = d*sc_j * q - dmin*mn_j per sub-block j of 32 weights, q in 0..15.  A
//   bf16 holds q exactly, and every f32 x is exactly the sum of three bf16
//   values: hi = x truncated to its top 16 bits, mid = (x - hi) truncated
//   likewise, lo = x - hi - mid (24 = 8 + 8 + 8 significand bits, each
//   difference exact).  So three v_mfma_f32_16x16x32_bf16 per sub-block give
//   sum q*x with exact products and f32 accumulation; d*sc_j scales that sum
//   in f32, and dmin*mn_j times the sub-block's sum of x is subtracted by one
//   v_mfma_f32_16x16x4f32 per four sub-blocks.  The weights are never rounded
//   (the f32 weight d*sc*q - dmin*mn of the shader rounds once).
//   Against v_mfma_f32_16x16x4f32 on dequantised weights (one per 4 weights,
//   32 clocks) this takes 48 + 8 matrix clocks instead of 256 per 16x16
//   outputs and 32 weights, and the nibbles become bf16 two at a time
//   (v_cvt_scalef32_pk_bf16_fp8: a byte q is the E4M3 value q * 2^-9).
//
// An output that is not finite is computed again weight by weight in f32
// (row_dot), so infinities, NaN and intermediate overflow come out as the
// plain product has them.
#include <algorithm>
#include <cstdint>

#include "common.hpp"
#include "depformer.hpp"
#include "lane.hpp"
#include "q4k.hpp"

namespace sts {

namespace {

typedef float floatx4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));

constexpr int kGemmBufferWord3 = 0x00020000;  // raw 32-bit buffer, no swizzle
constexpr uint32_t kHalf = 128;               // weights of half a super-block
constexpr uint32_t kSkip = 0x80000000u;       // buffer offset past every resource here

__device__ __forceinline__ u32x4 ld16(const uint8_t* p) {
  return *reinterpret_cast<const u32x4*>(p);
}
__device__ __forceinline__ u32x2 ld8(const uint8_t* p) {
  return *reinterpret_cast<const u32x2*>(p);
}

// Two of the four nibbles (one per byte of w, each 0..15) as bf16: byte q is
// the FP8 E4M3 number q * 2^-9 (subnormal below 8), so the conversion scaled
// by 2^9 gives q exactly.
template <bool HIGH>
__device__ __forceinline__ uint32_t nibbles_bf16(uint32_t w) {
  return __builtin_bit_cast(uint32_t,
                            __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(w, 512.0f, HIGH));
}
// The 8 nibbles of a sub-block's two words (already masked to one per byte).
__device__ __forceinline__ bf16x8 quants_bf16(uint32_t w0, uint32_t w1) {
  return __builtin_bit_cast(bf16x8, u32x4{nibbles_bf16<false>(w0), nibbles_bf16<true>(w0),
                                          nibbles_bf16<false>(w1), nibbles_bf16<true>(w1)});
}

// The upper halves of two registers: bf16(a) | bf16(b) << 16, truncated.
__device__ __forceinline__ uint32_t pack_hi(uint32_t a, uint32_t b) {
  return __builtin_amdgcn_perm(b, a, 0x07060302u);
}

// x = hi + mid + lo, three bf16 operands of eight values.
struct Split3 {
  bf16x8 hi, mid, lo;
};
__device__ __forceinline__ Split3 split3(const float (&x)[8]) {
#pragma clang fp contract(off)
  u32x4 h, m, l;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const uint32_t a = __float_as_uint(x[2 * i]), b = __float_as_uint(x[2 * i + 1]);
    const float ra = x[2 * i] - __uint_as_float(a & 0xFFFF0000u);
    const float rb = x[2 * i + 1] - __uint_as_float(b & 0xFFFF0000u);
    const uint32_t ma = __float_as_uint(ra), mb = __float_as_uint(rb);
    const float la = ra - __uint_as_float(ma & 0xFFFF0000u);
    const float lb = rb - __uint_as_float(mb & 0xFFFF0000u);
    h[i] = pack_hi(a, b);
    m[i] = pack_hi(ma, mb);
    l[i] = pack_hi(__float_as_uint(la), __float_as_uint(lb));
  }
  return {__builtin_bit_cast(bf16x8, h), __builtin_bit_cast(bf16x8, m),
          __builtin_bit_cast(bf16x8, l)};
}

// The products of hi, and those of lo and mid, summed apart and then added.
template <typename F>
__device__ __forceinline__ floatx4 sum8(const Split3& x, F product) {
  const floatx4 zero = {0.f, 0.f, 0.f, 0.f};
  return product(x.hi, zero) + product(x.mid, product(x.lo, zero));
}

__device__ __forceinline__ bool is_finite(float v) {
  return (__float_as_uint(v) & 0x7F800000u) != 0x7F800000u;
}

// sum_k W[n][k] x[k] (* alpha[k]) one weight after the other: what an output
// whose matrix-core sum is not finite takes (x with infinities or NaN, or so
// large that 15 x overflows).  NaN ends the sum.
__device__ __noinline__ float row_dot(const uint8_t* wrow, const float* x, const float* alpha,
                                      uint32_t K) {
#pragma clang fp contract(off)
  float acc = 0.f;
  for (uint32_t k0 = 0; k0 < K && acc == acc; k0 += 32) {
    const uint8_t* blk = wrow + (size_t)(k0 / 256) * kQ4kBlockBytes;
    const u32x4 hd = ld16(blk);
    const uint32_t j = (k0 / 32) & 7u;
    uint32_t sc, mn;
    scale_min(hd.y, hd.z, hd.w, j, sc, mn);
    const float d1 = half_bits_to_float(hd.x) * (float)sc;
    const float m1 = half_bits_to_float(hd.x >> 16) * (float)mn;
    const uint8_t* q = blk + 16 + 32 * (j >> 1);
    for (uint32_t i = 0; i < 32; ++i) {
      const float qv = (float)((q[i] >> (4 * (j & 1u))) & 15u);
      const float xv = alpha ? x[k0 + i] * alpha[k0 + i] : x[k0 + i];
      acc = __builtin_fmaf(__builtin_fmaf(qv, d1, -m1), xv, acc);
    }
  }
  return acc;
}

// q4k_rows_kernel: few rows.  Workgroup = 16 rows of X (the M tile of the
// matrix instructions) x NT tiles of 16 weight rows x all K; its WAVES waves
// share K, wave w taking half super-blocks w, w + WAVES, ... of 128 weights.
// Per half super-block a wave loads its 16 x 128 x values once (lane (r, g):
// row r, eight values of each of the four sub-blocks), splits them into the
// three bf16 operands, and multiplies them with the NT tiles' weights (lane
// (r, g): weight row r, bytes 8g..8g+7 of each 32-byte run, whose low and
// high nibbles are the operands of two sub-blocks).  The next half
// super-block's x and weights are requested as soon as this one's registers
// are free.  The waves' partial tiles meet in LDS at the end and are summed in
// wave order (deterministic), with RMSNorm's 1/rms, SwiGLU and the residual
// applied on the way out.
template <int NT, bool SWIGLU, bool NORM, int WAVES>
__global__ __launch_bounds__(64 * WAVES) void q4k_rows_kernel(const Q4kGemmParams p) {
#pragma clang fp contract(off)
  constexpr int NP = SWIGLU ? NT / 2 : NT;  // output tiles
  __shared__ float part[WAVES][NT][256];
  __shared__ float ssq[WAVES][16];
  __shared__ float s_inv[16];
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r = lane & 15, g = lane >> 4;
  const uint32_t KH = p.K / kHalf;
  const uint32_t z = blockIdx.z, mt = blockIdx.y;
  const uint8_t* W = p.w[z];
  const float* X = p.x + z * p.x_zstride;
  float* Y = p.y + z * p.y_zstride;
  const uint32_t nout = SWIGLU ? p.swiglu_f : p.N;
  const uint32_t row_bytes = p.K / kQ4kBlockWeights * kQ4kBlockBytes;
  const uint32_t t0 = blockIdx.x * NP;  // first output tile

  // Weight tile i and the tile's x rows come in through buffer resources that
  // end with their last row inside the matrix: rows past the end read zeros
  // (their outputs are not stored), and so does a whole load whose offset is
  // kSkip (a step past the last one, without a branch and without traffic).
  __amdgpu_buffer_rsrc_t wrs[NT];
#pragma unroll
  for (int i = 0; i < NT; ++i) {
    const uint32_t first =
        (t0 + (SWIGLU ? i % NP : i)) * 16 + (SWIGLU && i >= NP ? p.swiglu_f : 0u);
    const uint32_t base = min(first, p.N - 1);
    wrs[i] = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<uint8_t*>(W) + (size_t)base * row_bytes, 0,
        (int)(min(16u, p.N - base) * row_bytes), kGemmBufferWord3);
  }
  const uint32_t rows_here = min(16u, p.M - mt * 16);
  const __amdgpu_buffer_rsrc_t xrs = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<float*>(X) + (size_t)mt * 16 * p.ldx, 0,
      (int)(((uint64_t)(rows_here - 1) * p.ldx + p.K) * sizeof(float)), kGemmBufferWord3);
  const __amdgpu_buffer_rsrc_t ars = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<float*>(p.norm_alpha), 0, (int)(p.K * sizeof(float)), kGemmBufferWord3);
  const uint32_t xoff = (uint32_t)((r * p.ldx + 8 * g) * sizeof(float));
  const uint32_t woff = r * row_bytes;

  u32x4 hd[NT];
  u32x2 qa[NT], qb[NT];
  float4 xr[8], al[NORM ? 8 : 1];
  auto load_w = [&](int i, uint32_t hb) {
    const uint32_t o = hb < KH ? woff + (hb >> 1) * kQ4kBlockBytes : kSkip;
    const uint32_t oq = o + 16 + 64 * (hb & 1u) + 8 * g;
    hd[i] = __builtin_amdgcn_raw_buffer_load_b128(wrs[i], o, 0, 0);
    qa[i] = __builtin_amdgcn_raw_buffer_load_b64(wrs[i], oq, 0, 0);
    qb[i] = __builtin_amdgcn_raw_buffer_load_b64(wrs[i], oq + 32, 0, 0);
  };
  auto load_x = [&](uint32_t hb) {
    const uint32_t o = hb < KH ? xoff + hb * kHalf * (uint32_t)sizeof(float) : kSkip;
#pragma unroll
    for (int i = 0; i < 8; ++i)
      xr[i] = __builtin_bit_cast(
          float4, __builtin_amdgcn_raw_buffer_load_b128(
                      xrs, o + (32 * (i >> 1) + 4 * (i & 1)) * (int)sizeof(float), 0, 0));
    if constexpr (NORM) {
      const uint32_t oa = hb < KH ? (hb * kHalf + 8 * g) * (uint32_t)sizeof(float) : kSkip;
#pragma unroll
      for (int i = 0; i < 8; ++i)
        al[i] = __builtin_bit_cast(
            float4, __builtin_amdgcn_raw_buffer_load_b128(
                        ars, oa + (32 * (i >> 1) + 4 * (i & 1)) * (int)sizeof(float), 0, 0));
    }
  };

  floatx4 acc[NT];
#pragma unroll
  for (int i = 0; i < NT; ++i) acc[i] = floatx4{0.f, 0.f, 0.f, 0.f};
  float ss[4] = {0.f, 0.f, 0.f, 0.f};
  const floatx4 zero = {0.f, 0.f, 0.f, 0.f};
  bf16x8 m8;
#pragma unroll
  for (int e = 0; e < 8; ++e) m8[e] = (__bf16)-8.0f;

  // A wave's half super-blocks are all first halves or all second ones.
  static_assert(WAVES % 2 == 0, "half super-blocks alternate between the waves");
  const bool half = wave & 1;
  const uint32_t mask_lo = half ? 0x0F0F0F0Fu : 0x3F3F3F3Fu;
  const uint32_t mask_hi = half ? 0x30303030u : 0u;
  uint32_t hb = wave;
  load_x(hb);
#pragma unroll
  for (int i = 0; i < NT; ++i) load_w(i, hb);
  for (; hb < KH; hb += WAVES) {
    const uint32_t nx = hb + WAVES;
    // Sub-block j of the half super-block: its x operands.
    Split3 xs[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      float x[8] = {xr[2 * j].x,     xr[2 * j].y,     xr[2 * j].z,     xr[2 * j].w,
                    xr[2 * j + 1].x, xr[2 * j + 1].y, xr[2 * j + 1].z, xr[2 * j + 1].w};
      if constexpr (NORM) {
        const float a[8] = {al[2 * j].x,     al[2 * j].y,     al[2 * j].z,     al[2 * j].w,
                            al[2 * j + 1].x, al[2 * j + 1].y, al[2 * j + 1].z, al[2 * j + 1].w};
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          ss[j] = __builtin_fmaf(x[e], x[e], ss[j]);
          x[e] *= a[e];
        }
      }
      xs[j] = split3(x);
    }
    load_x(nx);
    // -8 times the sub-block's sum of x, in both layouts: c8[j] where the
    // tiles' accumulators want it (row 4g + e of every column), and sxg, what
    // lane (r, g) supplies to the min product (row r, sub-block g).  The same
    // products in the same order, so the two agree bit for bit.  The sum of
    // the hi parts is exact but for the widest spreads of x, and mid and lo
    // are added to it by one rounded addition: the matrix instruction
    // truncates what it aligns below its largest term, which here, the mins
    // having one sign, would add up over K (2.9e-7 from 64 bits at K = 4096
    // with one chain of three, 1.7e-7 on the f32 matrix instructions).
    floatx4 c8[4];
    float sxg = 0.f;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      c8[j] = sum8(xs[j], [&](bf16x8 x, floatx4 c) {
        return __builtin_amdgcn_mfma_f32_16x16x32_bf16(x, m8, c, 0, 0, 0);
      });
      const floatx4 t = sum8(xs[j], [&](bf16x8 x, floatx4 c) {
        return __builtin_amdgcn_mfma_f32_16x16x32_bf16(m8, x, c, 0, 0, 0);
      });
      sxg = g == j ? t[0] : sxg;
    }
#pragma unroll
    for (int i = 0; i < NT; ++i) {
      // Scales and mins of the half's four sub-blocks, one per byte (the
      // layout of shader_q4k_matvec.wgsl:85-113).
      const uint32_t sc4 = ((half ? hd[i].w : hd[i].y) & mask_lo) | ((hd[i].y >> 2) & mask_hi);
      const uint32_t mn4 =
          ((half ? hd[i].w >> 4 : hd[i].z) & mask_lo) | ((hd[i].z >> 2) & mask_hi);
      const float d = half_bits_to_float(hd[i].x), dmin = half_bits_to_float(hd[i].x >> 16);
      // dmin*mn/8 - d*sc of sub-block g: what is left of the min after the
      // quants' shift by 8, over -8.
      const float mg = dmin * (float)((mn4 >> (8 * g)) & 0xFFu);
      const float mng = __builtin_fmaf(mg, 0.125f, -(d * (float)((sc4 >> (8 * g)) & 0xFFu)));
      bf16x8 wq[4];
      wq[0] = quants_bf16(qa[i].x & 0x0F0F0F0Fu, qa[i].y & 0x0F0F0F0Fu);
      wq[1] = quants_bf16((qa[i].x >> 4) & 0x0F0F0F0Fu, (qa[i].y >> 4) & 0x0F0F0F0Fu);
      wq[2] = quants_bf16(qb[i].x & 0x0F0F0F0Fu, qb[i].y & 0x0F0F0F0Fu);
      wq[3] = quants_bf16((qb[i].x >> 4) & 0x0F0F0F0Fu, (qb[i].y >> 4) & 0x0F0F0F0Fu);
      load_w(i, nx);
      floatx4 s[4];
#pragma unroll
      for (int j = 0; j < 4; ++j)
        s[j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(xs[j].hi, wq[j], c8[j], 0, 0, 0);
#pragma unroll
      for (int j = 0; j < 4; ++j)
        s[j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(xs[j].mid, wq[j], s[j], 0, 0, 0);
#pragma unroll
      for (int j = 0; j < 4; ++j)
        s[j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(xs[j].lo, wq[j], s[j], 0, 0, 0);
      // This step's share is summed by itself: one rounding at the size of
      // the running total per step.
      floatx4 t = __builtin_amdgcn_mfma_f32_16x16x4f32(sxg, mng, zero, 0, 0, 0);
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const float d1 = d * (float)((sc4 >> (8 * j)) & 0xFFu);
#pragma unroll
        for (int e = 0; e < 4; ++e) t[e] = __builtin_fmaf(s[j][e], d1, t[e]);
      }
      acc[i] += t;
      __builtin_amdgcn_sched_barrier(0);  // one tile's operands at a time in registers
    }
  }

  // Element e of lane (r, g): row 4g + e of the M tile, weight row r.
#pragma unroll
  for (int i = 0; i < NT; ++i)
#pragma unroll
    for (int e = 0; e < 4; ++e) part[wave][i][(4 * g + e) * 16 + r] = acc[i][e];
  if constexpr (NORM) {
    const float q = sum_xor32(sum_xor16((ss[0] + ss[1]) + (ss[2] + ss[3])));
    if (g == 0) ssq[wave][r] = q;
  }
  __syncthreads();
  if constexpr (NORM) {
    // RMSNorm (shader_rmsnorm.wgsl:80-90): alpha went onto x, 1/rms goes
    // onto the row's outputs.
    if (tid < 16) {
      float tot = ssq[0][tid];
#pragma unroll
      for (int w = 1; w < WAVES; ++w) tot += ssq[w][tid];
      s_inv[tid] = 1.0f / sqrtf(tot / (float)p.K + p.norm_eps);
    }
    __syncthreads();
  }
  for (int o = tid; o < NP * 256; o += 64 * WAVES) {
    const int i = o >> 8, c = o & 255;
    const uint32_t mr = (uint32_t)c >> 4, mo = mt * 16 + mr, no = (t0 + i) * 16 + (c & 15);
    if (mo >= p.M || no >= nout) continue;
    float v = part[0][i][c];
#pragma unroll
    for (int w = 1; w < WAVES; ++w) v += part[w][i][c];
    const float* xrow = X + (size_t)mo * p.ldx;
    if (!is_finite(v)) v = row_dot(W + (size_t)no * row_bytes, xrow, p.norm_alpha, p.K);
    const float inv = NORM ? s_inv[mr] : 1.0f;
    v *= inv;
    if constexpr (SWIGLU) {
      float u = part[0][NP + i][c];
#pragma unroll
      for (int w = 1; w < WAVES; ++w) u += part[w][NP + i][c];
      if (!is_finite(u))
        u = row_dot(W + (size_t)(no + p.swiglu_f) * row_bytes, xrow, p.norm_alpha, p.K);
      u *= inv;
      v = v / (1.0f + expf(-v)) * u;
    }
    if (p.res) v += p.res[(size_t)mo * p.ldr + no];
    Y[(size_t)mo * p.ldy + no] = v;
  }
}

constexpr int kRowsWaves = 8;

template <int NT, bool SWIGLU>
int launch_rows(const Q4kGemmParams& p, uint32_t ntiles, uint32_t mtiles, hipStream_t stream) {
  constexpr uint32_t NP = SWIGLU ? NT / 2 : NT;
  const dim3 grid((ntiles + NP - 1) / NP, mtiles, p.Z), block(64 * kRowsWaves);
  if (p.norm_alpha)
    hipLaunchKernelGGL((q4k_rows_kernel<NT, SWIGLU, true, kRowsWaves>), grid, block, 0, stream, p);
  else
    hipLaunchKernelGGL((q4k_rows_kernel<NT, SWIGLU, false, kRowsWaves>), grid, block, 0, stream, p);
  STS_HIP(hipGetLastError());
  return STS_OK;
}

}  // namespace

int launch_q4k_gemm(const Q4kGemmParams& p, hipStream_t stream) {
  // Every check runs before anything is launched.
  if (p.K % kQ4kBlockWeights != 0 || p.K == 0 || p.K > 64 * kQ4kBlockWeights)
    return fail(STS_ERR_INVALID, "GEMM K = %u must be a multiple of 256 in 256..16384", p.K);
  if (p.M == 0 || p.N == 0 || p.Z == 0 || p.Z > (uint32_t)kGemmMaxZ)
    return fail(STS_ERR_INVALID, "GEMM shape M=%u N=%u Z=%u", p.M, p.N, p.Z);
  if ((p.M + 15) / 16 > 65535u) return fail(STS_ERR_INVALID, "M = %u too large", p.M);
  if (p.swiglu_f && (p.swiglu_f * 2 != p.N))
    return fail(STS_ERR_INVALID, "SwiGLU GEMM needs N = 2F (N=%u F=%u)", p.N, p.swiglu_f);
  if (p.ldx % 4 != 0 || p.x_zstride % 4 != 0 || (reinterpret_cast<uintptr_t>(p.x) & 15))
    return fail(STS_ERR_INVALID, "GEMM x rows must be 16-byte aligned");
  // A 16-row tile of x is addressed through one buffer resource (31-bit range).
  if ((uint64_t)p.ldx * 15 * sizeof(float) + (uint64_t)p.K * sizeof(float) > 0x7FFFFFF0ull)
    return fail(STS_ERR_INVALID, "GEMM x row stride %llu too large",
                (unsigned long long)p.ldx);
  for (uint32_t z = 0; z < p.Z; ++z)
    if (!p.w[z] || (reinterpret_cast<uintptr_t>(p.w[z]) & 15))
      return fail(STS_ERR_INVALID, "GEMM weights %u null or not 16-byte aligned", z);
  if (p.K > 16 * kQ4kBlockWeights && (p.Z != 1 || p.swiglu_f || p.norm_alpha))
    return fail(STS_ERR_INVALID, "GEMM with K = %u > 4096 takes no SwiGLU, RMSNorm or Z > 1", p.K);
  const uint32_t mtiles = (p.M + 15) / 16;
  const uint32_t nout = p.swiglu_f ? p.swiglu_f : p.N;
  const uint32_t ntiles = (nout + 15) / 16;
  const uint32_t cus = (uint32_t)device_cu_count();
  // Weight tiles per workgroup: as many as bring the launch to about one
  // workgroup per CU, up to six (eight spill registers).  Every workgroup splits
  // its x rows itself, so fewer and larger workgroups split them less often:
  // two per CU measured 12.7 against 8.1 us (64 rows x [3072, 1024]) and 28.7
  // against 19.2 us (13 x [12288, 4096]); and waves beyond eight leave too few
  // registers (12: 16.9 and 32.0 us).
  const uint64_t tiles = (uint64_t)ntiles * mtiles * p.Z;
  if (p.swiglu_f) {
    if (tiles <= cus) return launch_rows<2, true>(p, ntiles, mtiles, stream);
    if (tiles <= 2 * cus) return launch_rows<4, true>(p, ntiles, mtiles, stream);
    return launch_rows<6, true>(p, ntiles, mtiles, stream);
  }
  if (tiles <= cus) return launch_rows<1, false>(p, ntiles, mtiles, stream);
  if (tiles <= 2 * cus) return launch_rows<2, false>(p, ntiles, mtiles, stream);
  if (tiles <= 3 * cus) return launch_rows<3, false>(p, ntiles, mtiles, stream);
  if (tiles <= 4 * cus) return launch_rows<4, false>(p, ntiles, mtiles, stream);
  return launch_rows<6, false>(p, ntiles, mtiles, stream);
}

}  // namespace sts
