// q4k_gemm.hip -- Q4_K products for more than one row on the f16 matrix cores (gfx950).
//
// Y[m][n] = sum_k W[n][k] X[m][k] with W in Q4_K (q4k_matmul with M > 1,
// crates/sts-wasm/src/gguf.rs:810-897, and the depformer's projections,
// depth_engine.rs:953-1360).  f32 results without f32 matrix instructions:
//
//   W = d*sc_j * (q - z_j) + rest_j per sub-block j of 32 weights, z_j the whole
//   number of quant steps nearest to its min (zero_point).  sc_j * (q - z_j) is a
//   whole number up to 945, exact in f16, and x, scaled by a power of two per row
//   and block, is a sum of f16 values: three of them hold all its 24 bits.  So
//   v_mfma_f32_16x16x32_f16 on x's parts, each with an accumulator of its own,
//   give sum sc*(q - z)*x with exact products and f32 accumulation; d scales that
//   sum in f32, and rest_j times the sub-block's sum of x is added by one
//   v_mfma_f32_16x16x4f32 per four sub-blocks.
//   Against v_mfma_f32_16x16x4f32 on dequantised weights (one per 4 weights,
//   32 clocks) three parts take 48 + 8 matrix clocks instead of 256 per 16x16
//   outputs and 32 weights, and one packed fma forms two weight operands.
//   (The quants as they are and the mins' share taken off afterwards is 3 to 5%
//   faster, but channels of x far above the others at zero weights then leave
//   errors of up to 10% of sum |w x|, where dequantised weights leave none.)
//
// An output that is not finite is computed again weight by weight in f32
// (row_dot), so infinities, NaN and intermediate overflow come out as the
// plain product has them.
#include <algorithm>
#include <cstdint>
#include <type_traits>

#include "common.hpp"
#include "depformer.hpp"
#include "lane.hpp"
#include "q4k.hpp"

namespace sts {

namespace {

typedef float floatx4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));

constexpr int kGemmBufferWord3 = 0x00020000;  // raw 32-bit buffer, no swizzle
constexpr uint32_t kHalf = 128;               // weights of half a super-block
constexpr uint32_t kSkip = 0x80000000u;       // buffer offset past every resource here

__device__ __forceinline__ u32x4 ld16(const uint8_t* p) {
  return *reinterpret_cast<const u32x4*>(p);
}

// The zero point of sub-block g of a weight row: the whole number of quant steps
// nearest to its min, 0..15.  Every weight is then d*sc * (q - z) + rest with
// |rest| at most the weight itself: q = z leaves the rest alone, another q is
// at least half a step away, and where the min lies beyond the quants both terms
// have one sign.  So the two sums a product is made of, over the first terms and
// over the rests, are no larger than a few times sum |w x|, whatever the weights
// and x.  (Sums over quants and mins apart are two large terms under a large x at
// a small weight, whose roundings the difference keeps.)
struct ZeroPoint {
  uint32_t z;
  float rest;  // d*sc*z - dmin*mn, rounded once (the products are exact)
};
__device__ __forceinline__ ZeroPoint zero_point(float d, float dmin, uint32_t sc, uint32_t mn) {
  const float step = d * (float)sc, min = dmin * (float)mn;
  // Any z gives the weights; NaN and infinities clamp.
  const float z = rintf(__builtin_amdgcn_fmed3f(min * __builtin_amdgcn_rcpf(step), 0.f, 15.f));
  return {(uint32_t)z, __builtin_fmaf(step, z, -min)};
}

// A word or'ed over the four 16-lane rows.
__device__ __forceinline__ uint32_t or_rows(uint32_t v) {
  const auto a = __builtin_amdgcn_permlane16_swap(v, v, false, false);
  v = a[0] | a[1];
  const auto b = __builtin_amdgcn_permlane32_swap(v, v, false, false);
  return b[0] | b[1];
}

// Operand scales of two sub-blocks, bytes 2p and 2p + 1 of sc (6-bit scales) and
// z16 (zero points times 16): sc * 2^5 and z * sc * 2^-15.
struct PairScale {
  f16x2 s, zs;
};
__device__ __forceinline__ PairScale pair_scale(uint32_t sc, uint32_t z16, int p) {
  // The half 0x6400 | b is 1024 + b, and the half b of one byte b * 2^-24.
  const f16x2 up = {(_Float16)32.0f, (_Float16)32.0f};
  const f16x2 off = {(_Float16)-32768.0f, (_Float16)-32768.0f};
  const uint32_t b = __builtin_amdgcn_perm(0x64646464u, sc, p ? 0x04030402u : 0x04010400u);
  const uint32_t z = __builtin_amdgcn_perm(0u, z16, p ? 0x0C030C02u : 0x0C010C00u);
  const f16x2 s = __builtin_elementwise_fma(__builtin_bit_cast(f16x2, b), up, off);
  return {s, __builtin_bit_cast(f16x2, z) * s};
}

// Weight operand of one sub-block: the eight values sc * (q - z) * 2^-15, q the
// high nibbles of w's bytes, whole numbers up to 945 and so exact.  The half
// 16 q is the subnormal q * 2^-20, so one fma a pair forms them.
__device__ __forceinline__ f16x8 weights_f16(u32x2 w, _Float16 s, _Float16 zs) {
  const f16x2 ss = {s, s}, tt = {zs, zs};
  u32x4 o;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const uint32_t h = __builtin_amdgcn_perm(0u, (i & 2 ? w.y : w.x) & 0xF0F0F0F0u,
                                             i & 1 ? 0x0C030C02u : 0x0C010C00u);
    o[i] = __builtin_bit_cast(
        uint32_t, __builtin_elementwise_fma(__builtin_bit_cast(f16x2, h), ss, -tt));
  }
  return __builtin_bit_cast(f16x8, o);
}
constexpr float kOperandUp = 0x1p15f;  // takes the operands' 2^-15 off again

// Scales x so that the largest of a row's block lies in [2^14, 2^15): up is
// that power of two and down its inverse, both inside f32's normal range (an
// infinity or NaN passes through unscaled or not and makes the row's outputs
// so, which then take row_dot).
struct BlockScale {
  float up, down;
};
__device__ __forceinline__ BlockScale block_scale(float big) {
  int e = (int)(__float_as_uint(big) >> 23) - 127;
  e = max(-110, min(e, 127));
  return {__uint_as_float((uint32_t)(127 + 14 - e) << 23),
          __uint_as_float((uint32_t)(127 - 14 + e) << 23)};
}

// x = p[0] + 2^-11 p[1] + 2^-22 p[2], f16 operands of eight scaled values: each
// part holds the next 11 bits, scaled up so that it keeps them as a normal
// number.  Exact for values down to 2^-38 of the block's largest; below, off by
// up to 2^-61 of it.
constexpr float kPartUp = 0x1p11f, kPartDown = 0x1p-11f;
struct Split3 {
  f16x8 p[3];
};
__device__ __forceinline__ Split3 split3(const float (&x)[8]) {
#pragma clang fp contract(off)
  u32x4 o[3];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    float a = x[2 * i], b = x[2 * i + 1];
#pragma unroll
    for (int c = 0; c < 3; ++c) {
      const f16x2 h = __builtin_bit_cast(f16x2, __builtin_amdgcn_cvt_pkrtz(a, b));
      o[c][i] = __builtin_bit_cast(uint32_t, h);
      if (c == 2) break;
      a = __builtin_fmaf((float)h.x, -kPartUp, a * kPartUp);  // exact
      b = __builtin_fmaf((float)h.y, -kPartUp, b * kPartUp);
    }
  }
  return {{__builtin_bit_cast(f16x8, o[0]), __builtin_bit_cast(f16x8, o[1]),
           __builtin_bit_cast(f16x8, o[2])}};
}

// The value is computed here: without this the compiler puts off the
// additions of unrolled steps to their end and keeps every step's products in
// registers until then.
__device__ __forceinline__ void pin(floatx4& v) { asm volatile("" : "+v"(v)); }

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
// three f16 operands, and multiplies them with the NT tiles' weights (lane
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
    // Sub-block j's x: the row's largest, its sum, its operands.
    float x[4][8], sx[4], big = 0.f;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const float t[8] = {xr[2 * j].x,     xr[2 * j].y,     xr[2 * j].z,     xr[2 * j].w,
                          xr[2 * j + 1].x, xr[2 * j + 1].y, xr[2 * j + 1].z, xr[2 * j + 1].w};
#pragma unroll
      for (int e = 0; e < 8; ++e) x[j][e] = t[e];
      if constexpr (NORM) {
        const float a[8] = {al[2 * j].x,     al[2 * j].y,     al[2 * j].z,     al[2 * j].w,
                            al[2 * j + 1].x, al[2 * j + 1].y, al[2 * j + 1].z, al[2 * j + 1].w};
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          ss[j] = __builtin_fmaf(x[j][e], x[j][e], ss[j]);
          x[j][e] *= a[e];
        }
      }
#pragma unroll
      for (int e = 0; e < 8; ++e) big = fmaxf(big, fabsf(x[j][e]));
      sx[j] = ((x[j][0] + x[j][1]) + (x[j][2] + x[j][3])) +
              ((x[j][4] + x[j][5]) + (x[j][6] + x[j][7]));
    }
    const BlockScale bs = block_scale(max_xor32(max_xor16(big)));
    Split3 xs[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
#pragma unroll
      for (int e = 0; e < 8; ++e) x[j][e] *= bs.up;
      xs[j] = split3(x[j]);
    }
    load_x(nx);
    // What lane (r, g) supplies to the rests' product: row r's sum of sub-block
    // g, the four lanes' shares added as they are dealt (the swap leaves sum j
    // of one half of the lanes and sum j' of the other in the pair it returns).
    const auto pair = [](auto r) { return __uint_as_float(r[0]) + __uint_as_float(r[1]); };
    const float s02 = pair(__builtin_amdgcn_permlane32_swap(
        __float_as_uint(sx[0]), __float_as_uint(sx[2]), false, false));
    const float s13 = pair(__builtin_amdgcn_permlane32_swap(
        __float_as_uint(sx[1]), __float_as_uint(sx[3]), false, false));
    const float sxg = pair(__builtin_amdgcn_permlane16_swap(
        __float_as_uint(s02), __float_as_uint(s13), false, false));
    // 2^k of row 4g + e, the accumulators' rows: four quarters of it, exactly.
    const floatx4 down = __builtin_amdgcn_mfma_f32_16x16x4f32(0.25f * bs.down, 1.0f, zero, 0, 0, 0);
    // x's own values are out of the registers by here (this instance would spill).
    if constexpr (NT == 4 && NORM) __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int i = 0; i < NT; ++i) {
      // Scales and mins of the half's four sub-blocks, one per byte (the
      // layout of shader_q4k_matvec.wgsl:85-113).
      const uint32_t sc4 = ((half ? hd[i].w : hd[i].y) & mask_lo) | ((hd[i].y >> 2) & mask_hi);
      const uint32_t mn4 =
          ((half ? hd[i].w >> 4 : hd[i].z) & mask_lo) | ((hd[i].z >> 2) & mask_hi);
      const float d = half_bits_to_float(hd[i].x), dmin = half_bits_to_float(hd[i].x >> 16);
      const ZeroPoint zp = zero_point(d, dmin, (sc4 >> (8 * g)) & 0xFFu, (mn4 >> (8 * g)) & 0xFFu);
      const uint32_t z4 = or_rows(zp.z << (8 * g + 4));
      const PairScale s0 = pair_scale(sc4, z4, 0), s1 = pair_scale(sc4, z4, 1);
      f16x8 wq[4];
      wq[0] = weights_f16(u32x2{qa[i].x << 4, qa[i].y << 4}, s0.s.x, s0.zs.x);
      wq[1] = weights_f16(qa[i], s0.s.y, s0.zs.y);
      wq[2] = weights_f16(u32x2{qb[i].x << 4, qb[i].y << 4}, s1.s.x, s1.zs.x);
      wq[3] = weights_f16(qb[i], s1.s.y, s1.zs.y);
      load_w(i, nx);
      // The parts are summed apart and then added, this step's share by itself:
      // one rounding at the size of the running total per step.
      floatx4 t[3] = {zero, zero, zero};
#pragma unroll
      for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int c = 0; c < 3; ++c)
          t[c] = __builtin_amdgcn_mfma_f32_16x16x32_f16(xs[j].p[c], wq[j], t[c], 0, 0, 0);
      const floatx4 m = __builtin_amdgcn_mfma_f32_16x16x4f32(sxg, zp.rest, zero, 0, 0, 0);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const float u = __builtin_fmaf(__builtin_fmaf(t[2][e], kPartDown, t[1][e]), kPartDown, t[0][e]);
        acc[i][e] += __builtin_fmaf(u * (kOperandUp * d), down[e], m[e]);
      }
      pin(acc[i]);  // one tile's operands at a time in registers
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

// One weight of a slot after the other is what a single row of x is worth: no
// 16-row tile to fill.  The 64 weights of slot s of a row (iteration s % 4 of
// super-block s / 4) against the lane's x values.  d*sc, dmin*mn and q*(d*sc)
// are exact in f32, so one fma rounds the weight as the shader does, and a small
// weight stays small under a large x: the quants' and the mins' shares summed
// apart are two large terms there, whose roundings the difference keeps.
__device__ __forceinline__ float slot_dot(u32x4 hd, u32x4 qa, u32x4 qb, uint32_t j,
                                          const float (&x)[64]) {
  const float d = half_bits_to_float(hd.x), dmin = half_bits_to_float(hd.x >> 16);
  uint32_t scl, mnl, sch, mnh;
  scale_min(hd.y, hd.z, hd.w, j, scl, mnl);
  scale_min(hd.y, hd.z, hd.w, j + 1, sch, mnh);
  const float d1 = d * (float)scl, m1 = dmin * (float)mnl;
  const float d2 = d * (float)sch, m2 = dmin * (float)mnh;
  const uint32_t words[8] = {qa.x, qa.y, qa.z, qa.w, qb.x, qb.y, qb.z, qb.w};
  float a[4] = {0.f, 0.f, 0.f, 0.f}, b[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int w = 0; w < 8; ++w) {
    uint32_t lo = words[w] & 0x0F0F0F0Fu;
    uint32_t hi = (words[w] >> 4) & 0x0F0F0F0Fu;
    // Opaque to the optimiser, so each byte below is one v_cvt_f32_ubyte.
    asm("" : "+v"(lo), "+v"(hi));
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const float wl = __builtin_fmaf((float)((lo >> (8 * i)) & 0xFFu), d1, -m1);
      const float wh = __builtin_fmaf((float)((hi >> (8 * i)) & 0xFFu), d2, -m2);
      a[i] = __builtin_fmaf(wl, x[4 * w + i], a[i]);
      b[i] = __builtin_fmaf(wh, x[32 + 4 * w + i], b[i]);
    }
  }
  return ((a[0] + a[1]) + (a[2] + a[3])) + ((b[0] + b[1]) + (b[2] + b[3]));
}

// Decode attention of all heads (dim 64) of one stream over the slots 0..len-1
// of its cache in one wave, slot len-1 being k_new / v_new: head 4k + lane/16
// in registers k, dims 4c..4c+3 with c = lane % 16.  Four slots at a time,
// online softmax, as decode_kernel has it.  Buffer loads past a resource (a
// head or slot that is not there) give zeros.
template <int NK>
struct SlotAttention {
  float4 q[NK], kn[NK], vn[NK], kk[4][NK], vv[4][NK];
  __amdgpu_buffer_rsrc_t krs, vrs;
  uint32_t off[NK];  // of slot 0 of the head in the cache, or kSkip
  int lane;

  static __device__ __forceinline__ float4 ld(__amdgpu_buffer_rsrc_t rs, uint32_t o) {
    return __builtin_bit_cast(float4, __builtin_amdgcn_raw_buffer_load_b128(rs, o, 0, 0));
  }
  __device__ __forceinline__ void load(const DepthAttention& a, uint32_t t0) {
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
      for (int k = 0; k < NK; ++k) {
        const uint32_t o = t0 + j < a.len - 1 && off[k] != kSkip ? off[k] + (t0 + j) * 256 : kSkip;
        kk[j][k] = ld(krs, o);
        vv[j][k] = ld(vrs, o);
      }
  }
  __device__ __forceinline__ void begin(const DepthAttention& a, uint32_t b, uint32_t dim, int l) {
    lane = l;
    const uint32_t row = dim * (uint32_t)sizeof(float), head = a.max_len * 256;
    auto row_of = [&](const float* p) {
      return __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(p) + b * a.q_bstride, 0,
                                               (int)row, kGemmBufferWord3);
    };
    const __amdgpu_buffer_rsrc_t qrs = row_of(a.q), knrs = row_of(a.k_new), vnrs = row_of(a.v_new);
    const int cache = (int)(dim / 64 * head);
    krs = __builtin_amdgcn_make_buffer_rsrc(a.k + b * a.kv_bstride, 0, cache, kGemmBufferWord3);
    vrs = __builtin_amdgcn_make_buffer_rsrc(a.v + b * a.kv_bstride, 0, cache, kGemmBufferWord3);
#pragma unroll
    for (int k = 0; k < NK; ++k) {
      const uint32_t h = 4 * k + lane / 16;
      off[k] = h < dim / 64 ? h * head + (lane & 15) * 16 : kSkip;
      q[k] = ld(qrs, (lane + 64 * k) * 16);
      kn[k] = ld(knrs, (lane + 64 * k) * 16);
      vn[k] = ld(vnrs, (lane + 64 * k) * 16);
    }
    load(a, 0);
  }
  __device__ __forceinline__ void store_new(const DepthAttention& a, uint32_t b) {
#pragma unroll
    for (int k = 0; k < NK; ++k) {
      if (off[k] == kSkip) continue;
      const size_t o = b * a.kv_bstride + off[k] / 4 + (a.len - 1) * 64;
      *reinterpret_cast<float4*>(a.k + o) = kn[k];
      *reinterpret_cast<float4*>(a.v + o) = vn[k];
    }
  }
  __device__ __forceinline__ void finish(const DepthAttention& a, float4 (&out)[NK]) {
    float m[NK], l[NK];
#pragma unroll
    for (int k = 0; k < NK; ++k) {
      m[k] = -3.402823466e+38f;
      l[k] = 0.f;
      out[k] = make_float4(0.f, 0.f, 0.f, 0.f);
      q[k] = make_float4(q[k].x * a.scale_log2, q[k].y * a.scale_log2, q[k].z * a.scale_log2,
                         q[k].w * a.scale_log2);
    }
    for (uint32_t t0 = 0; t0 < a.len; t0 += 4) {
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        if (t0 + j != a.len - 1) continue;
#pragma unroll
        for (int k = 0; k < NK; ++k) {
          kk[j][k] = kn[k];
          vv[j][k] = vn[k];
        }
      }
#pragma unroll
      for (int k = 0; k < NK; ++k) {
        float s[4], mn = m[k];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const float4 t = kk[j][k];
          float d = __builtin_fmaf(q[k].w, t.w, __builtin_fmaf(q[k].z, t.z,
                    __builtin_fmaf(q[k].y, t.y, q[k].x * t.x)));
          d += xchg<0>(d);
          d += xchg<1>(d);
          d += xchg<2>(d);
          d += xchg<3>(d);
          s[j] = t0 + j < a.len ? d : -INFINITY;
          mn = fmaxf(mn, s[j]);
        }
        const float al = __builtin_amdgcn_exp2f(m[k] - mn);
        m[k] = mn;
        l[k] *= al;
        out[k] = make_float4(out[k].x * al, out[k].y * al, out[k].z * al, out[k].w * al);
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const float w = __builtin_amdgcn_exp2f(s[j] - mn);
          l[k] += w;
          out[k].x = __builtin_fmaf(w, vv[j][k].x, out[k].x);
          out[k].y = __builtin_fmaf(w, vv[j][k].y, out[k].y);
          out[k].z = __builtin_fmaf(w, vv[j][k].z, out[k].z);
          out[k].w = __builtin_fmaf(w, vv[j][k].w, out[k].w);
        }
      }
      if (t0 + 4 < a.len) load(a, t0 + 4);
    }
#pragma unroll
    for (int k = 0; k < NK; ++k)
      out[k] = make_float4(out[k].x / l[k], out[k].y / l[k], out[k].z / l[k], out[k].w / l[k]);
  }
};

// q4k_vec_kernel: one or two rows of x (the depformer of one conversation),
// where the products are a few microseconds of latency.  One wave per
// workgroup takes RPW weight rows at once, a slot per lane (64 / RPW lanes a
// row), R times; it stages its row of x in LDS by itself, so no barrier stands
// in its way, and with NORM sums its squares on the way.  1 row, weights from
// the last-level cache: [3072, 1024] with RMSNorm 3.3 us against 5.2 in
// q4k_rows_kernel, [5632, 1024] with SwiGLU 4.1 against 6.3, [1024, 2816] 3.5
// and [1024, 1024] 2.8 against 6.3 for the two, of which an empty launch is 2.5.
// XL: float4 of x per lane, K <= 256 XL.
//
// ATTN: x is the output of one decode step's attention over a few slots, which
// every wave computes for itself from q, k_new, v_new and the cache (XL float4
// a lane: head 4k + lane / 16, 16 lanes a row); the first workgroup of a row
// writes the new slot, which the others take from k_new and v_new.
// [1024, 1024], 16 heads: 4.6 us to four slots, 5.8 to eight, where the two
// launches were 7.0; the second four slots are a second round trip to memory.
struct NoAttention {};
template <int XL, int R, bool NORM, bool SWIGLU, typename A = NoAttention>
__global__ __launch_bounds__(64) void q4k_vec_kernel(const Q4kGemmParams p, const A a) {
#pragma clang fp contract(off)
  constexpr bool ATTN = !std::is_same_v<A, NoAttention>;
  constexpr int RPW = XL <= 4 ? 4 : XL <= 8 ? 2 : 1;
  constexpr int LPR = 64 / RPW;  // lanes of a row
  constexpr int NH = SWIGLU ? 2 : 1;
  __shared__ __align__(16) float xs[XL * 4][68];  // slot, its 64 values (pitch 68)
  __shared__ __align__(16) float xc[ATTN ? XL * 256 : 4];  // for row_dot
  const int lane = threadIdx.x;
  const int s = lane % LPR;
  const uint32_t b = blockIdx.y, z = blockIdx.z;
  const uint8_t* W = p.w[z];
  const float* X = p.x + z * p.x_zstride + (size_t)b * p.ldx;
  const uint32_t nout = SWIGLU ? p.swiglu_f : p.N;
  const size_t row_bytes = (size_t)(p.K / kQ4kBlockWeights) * kQ4kBlockBytes;
  // A lane past the row's last slot reads slot 0 with its d and dmin as zeros.
  const bool has = (uint32_t)s < p.K / 64;
  const uint32_t slot = has ? s : 0u;
  const uint32_t row0 = blockIdx.x * (R * RPW) + lane / LPR;

  // x (and alpha) first, then the weights and the residual.
  const __amdgpu_buffer_rsrc_t xrs = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<float*>(X), 0, (int)(p.K * sizeof(float)), kGemmBufferWord3);
  const __amdgpu_buffer_rsrc_t ars = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<float*>(p.norm_alpha), 0, (int)(p.K * sizeof(float)), kGemmBufferWord3);
  float4 xr[XL], al[NORM ? XL : 1];
  SlotAttention<ATTN ? XL : 1> at;
  if constexpr (ATTN) at.begin(a, b, p.K, lane);
#pragma unroll
  for (int k = 0; k < (ATTN ? 0 : XL); ++k) {
    const uint32_t o = (lane + 64 * k) * 16;  // past K: zeros
    xr[k] = __builtin_bit_cast(float4, __builtin_amdgcn_raw_buffer_load_b128(xrs, o, 0, 0));
    if constexpr (NORM)
      al[k] = __builtin_bit_cast(float4, __builtin_amdgcn_raw_buffer_load_b128(ars, o, 0, 0));
  }
  u32x4 hd[R][NH], qa[R][NH], qb[R][NH];
  float res[R];
#pragma unroll
  for (int j = 0; j < R; ++j) {
    const uint32_t n = min(row0 + j * RPW, nout - 1);
#pragma unroll
    for (int hv = 0; hv < NH; ++hv) {
      const uint8_t* blk = W + (n + (hv ? p.swiglu_f : 0u)) * row_bytes +
                           (size_t)(slot >> 2) * kQ4kBlockBytes;
      hd[j][hv] = ld16(blk);
      hd[j][hv].x = has ? hd[j][hv].x : 0u;
      qa[j][hv] = ld16(blk + 16 + 32 * (slot & 3u));
      qb[j][hv] = ld16(blk + 32 + 32 * (slot & 3u));
    }
    res[j] = p.res ? p.res[(size_t)b * p.ldr + n] : 0.f;
  }
  if constexpr (ATTN) {
    if (blockIdx.x == 0) at.store_new(a, b);
    at.finish(a, xr);
  }
  float ss[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int k = 0; k < XL; ++k) {
    float4 v = xr[k];
    if constexpr (NORM) {
      ss[0] = __builtin_fmaf(v.x, v.x, ss[0]);
      ss[1] = __builtin_fmaf(v.y, v.y, ss[1]);
      ss[2] = __builtin_fmaf(v.z, v.z, ss[2]);
      ss[3] = __builtin_fmaf(v.w, v.w, ss[3]);
      v = make_float4(v.x * al[k].x, v.y * al[k].y, v.z * al[k].z, v.w * al[k].w);
    }
    const int i = lane + 64 * k;
    *reinterpret_cast<float4*>(&xs[i >> 4][4 * (i & 15)]) = v;
    if constexpr (ATTN) *reinterpret_cast<float4*>(&xc[4 * i]) = v;
  }
  __syncthreads();  // one wave: orders its LDS writes before its reads
  float x[64];
#pragma unroll
  for (int j = 0; j < 16; ++j) {
    const float4 t = *reinterpret_cast<const float4*>(&xs[slot][4 * j]);
    x[4 * j] = t.x;
    x[4 * j + 1] = t.y;
    x[4 * j + 2] = t.z;
    x[4 * j + 3] = t.w;
  }
  auto lanes_sum = [&](float v) {
    v += xchg<0>(v);
    v += xchg<1>(v);
    v += xchg<2>(v);
    v += xchg<3>(v);
    if constexpr (LPR >= 32) v = sum_xor16(v);
    if constexpr (LPR >= 64) v = sum_xor32(v);
    return v;
  };
  float inv = 1.f;
  if constexpr (NORM) {
    float q = (ss[0] + ss[1]) + (ss[2] + ss[3]);
    q += xchg<0>(q);
    q += xchg<1>(q);
    q += xchg<2>(q);
    q += xchg<3>(q);
    q = sum_xor32(sum_xor16(q));
    inv = 1.0f / sqrtf(q / (float)p.K + p.norm_eps);
  }
#pragma unroll
  for (int j = 0; j < R; ++j) {
    const uint32_t n = row0 + j * RPW;
    float v[NH];
#pragma unroll
    for (int hv = 0; hv < NH; ++hv)
      v[hv] = lanes_sum(slot_dot(hd[j][hv], qa[j][hv], qb[j][hv], 2 * (slot & 3u), x));
    if (s != 0 || n >= nout) continue;
#pragma unroll
    for (int hv = 0; hv < NH; ++hv) {
      if (!is_finite(v[hv]))
        v[hv] = row_dot(W + (n + (hv ? p.swiglu_f : 0u)) * row_bytes, ATTN ? xc : X,
                        p.norm_alpha, p.K);
      v[hv] *= inv;
    }
    float o = v[0];
    if constexpr (SWIGLU) o = o / (1.0f + expf(-o)) * v[NH - 1];
    if (p.res) o += res[j];
    p.y[z * p.y_zstride + (size_t)b * p.ldy + n] = o;
  }
}

// Many rows.  x as two f16 parts, the first rounded to nearest and the second
// what it leaves: 23 bits of every value down to 2^-28 of the largest in its row
// and super-block.  The f32 sums round at 24 bits of the running total, over
// which this is not seen (x Gaussian, K = 4096: 1.2e-7 from 64 bits, with all 24
// bits on the f32 matrix instructions 1.7e-7).  Super-blocks of 16 rows that
// hold smaller values (beside an outlier) get a third part, whose products only
// they pay for: then 23 bits down to 2^-39.
constexpr int kParts = 2;
constexpr int kTileM = 64, kTileN = 128;

// What split_planes_kernel writes for `rows` rows (a multiple of 64) of K
// columns, in floats: operand units of 64 x 16 bytes per (16-row tile mt,
// sub-block kb, part), entry g*16 + r being row r, columns 8g..8g+7, as lane
// (r, g) of a matrix instruction wants it; the third parts' units in the same
// order, written only where they are used; the sums of x per (mt, kb, row); and
// the scales per (mt, super-block, row), negated where there is a third part.
struct TilePlanes {
  u32x4* units;
  u32x4* third;
  float* sums;
  float* scales;
  static size_t floats(size_t rows, size_t KB) {
    return rows / 16 * KB * (kParts + 1) * 256 + rows * KB + rows * (KB / 8);
  }
  TilePlanes(float* p, size_t rows, size_t KB)
      : units(reinterpret_cast<u32x4*>(p)),
        third(units + rows / 16 * KB * kParts * 64),
        sums(p + rows / 16 * KB * (kParts + 1) * 256),
        scales(sums + rows * KB) {}
};

// Element i of the parts of the scaled value y; returns what they leave, times
// 2^11 (exact).
__device__ __forceinline__ float split_parts(float y, f16x8 (&h)[kParts], int i) {
  static_assert(kParts == 2, "two parts");
  h[0][i] = (_Float16)y;
  const float rest = __builtin_fmaf((float)h[0][i], -kPartUp, y * kPartUp);
  h[1][i] = (_Float16)rest;
  return rest - (float)h[1][i];
}

// One wave per 16-row tile and super-block: lane (r, g) takes row r, columns
// 8g..8g+7 of each of the eight sub-blocks.  Rows past M become zeros.  The
// sums of x are taken in f64 and rounded once.
__global__ __launch_bounds__(256) void split_planes_kernel(const float* __restrict__ x,
                                                              uint64_t ldx, uint32_t M,
                                                              uint32_t SB, const TilePlanes out) {
#pragma clang fp contract(off)
  const int lane = threadIdx.x & 63;
  const int r = lane & 15, g = lane >> 4;
  const uint32_t sb = blockIdx.x * 4 + (threadIdx.x >> 6), mt = blockIdx.y;
  if (sb >= SB) return;
  const uint32_t m = mt * 16 + r;
  const float* row = x + (size_t)(m < M ? m : 0) * ldx + 256 * (size_t)sb + 8 * g;
  float v[8][8];
  float big = 0.f;
  uint32_t least = ~0u;  // twice the bits of the smallest magnitude but zero, less one
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    const float4 a = *reinterpret_cast<const float4*>(row + 32 * j);
    const float4 b = *reinterpret_cast<const float4*>(row + 32 * j + 4);
    const float t[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      v[j][e] = m < M ? t[e] : 0.f;
      big = fmaxf(big, fabsf(v[j][e]));
      least = min(least, 2 * __float_as_uint(v[j][e]) - 1);
    }
  }
  big = max_xor32(max_xor16(big));
  const BlockScale bs = block_scale(big);
  // Of values below 2^-27 of the largest's power of two, two parts can leave more
  // than 2^-23.
  const uint32_t exponent = __float_as_uint(big) >> 23;
  const bool third = __any(least < (exponent > 27 ? exponent - 27 : 0u) << 24);
  if (g == 0) out.scales[((size_t)mt * SB + sb) * 16 + r] = third ? -bs.down : bs.down;
  const size_t kb0 = (size_t)mt * SB * 8 + 8 * sb;
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    u32x4* u = out.units + (kb0 + j) * kParts * 64 + (g * 16 + r);
    double q = 0.0;
#pragma unroll
    for (int i = 0; i < 8; ++i) q += (double)v[j][i];
    f16x8 h[kParts];
#pragma unroll
    for (int i = 0; i < 8; ++i) split_parts(v[j][i] * bs.up, h, i);
#pragma unroll
    for (int c = 0; c < kParts; ++c) u[64 * c] = __builtin_bit_cast(u32x4, h[c]);
    q += __shfl_xor(q, 16, 64);
    q += __shfl_xor(q, 32, 64);
    if (g == 0) out.sums[(kb0 + j) * 16 + r] = (float)q;
  }
  if (!third) return;
  // Rare: x is read again (the compiler not knowing that it is) rather than kept.
  asm volatile("" : "+v"(row));
#pragma nounroll
  for (int j = 0; j < 8; ++j) {
    f16x8 h[kParts], rest;
#pragma unroll
    for (int i = 0; i < 8; ++i)
      rest[i] = (_Float16)(split_parts((m < M ? row[32 * j + i] : 0.f) * bs.up, h, i) * kPartUp);
    out.third[(kb0 + j) * 64 + (g * 16 + r)] = __builtin_bit_cast(u32x4, rest);
  }
}

// q4k_tile_kernel: many rows, the x operands prepared by split_planes_kernel.
// Workgroup = 64 rows x 128 weight rows, four waves of 64 x 32 (4 x 2 tiles of
// 16 x 16), two workgroups a CU, a range of super-blocks of K in steps of 64
// columns (32 quant bytes of every weight row: two sub-blocks).  Operands go to
// LDS through registers, two buffers each: a step's x operands
// one step ahead, a super-block's weight bytes
// (128 x 144) come in two batches during the super-block before.  The
// super-block's products accumulate in the matrix core, each part's apart (only
// the first part's eight additions round at the size of the result); then
// they are scaled by d and the row's scale and added to the total.
struct Q4kTileParams {
  const uint8_t* w;
  const u32x4* units;
  const u32x4* third;
  const float* sums;
  const float* scales;
  const float* x;  // the rows themselves, for outputs that are not finite
  const float* res;
  float* y;
  uint64_t ldx, ldr, ldy, y_split;  // y_split: floats from one K range's y to the next
  uint32_t M, N, K, mtiles, ksplit;  // mtiles: 64-row tiles
};

// Waits for this wave's LDS operations alone, then the workgroup barrier:
// loads into registers stay in flight across it.
__device__ __forceinline__ void lds_barrier() {
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0)
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}

// A weight row's super-block header as lane (r, g) uses it: the eight scales and
// zero points, one per byte, d, and the rests of sub-blocks g and 4 + g.
__device__ __forceinline__ void tile_header(u32x4 h, int g, uint32_t (&sc)[2], uint32_t (&zp)[2],
                                            float& d, float (&rest)[2]) {
  sc[0] = h.y & 0x3F3F3F3Fu;
  sc[1] = (h.w & 0x0F0F0F0Fu) | ((h.y >> 2) & 0x30303030u);
  const uint32_t mn[2] = {h.z & 0x3F3F3F3Fu,
                          ((h.w >> 4) & 0x0F0F0F0Fu) | ((h.z >> 2) & 0x30303030u)};
  d = half_bits_to_float(h.x);
  const float dmin = half_bits_to_float(h.x >> 16);
#pragma unroll
  for (int hf = 0; hf < 2; ++hf) {
    const ZeroPoint z =
        zero_point(d, dmin, (sc[hf] >> (8 * g)) & 0xFFu, (mn[hf] >> (8 * g)) & 0xFFu);
    zp[hf] = or_rows(z.z << (8 * g + 4));
    rest[hf] = z.rest;
  }
}

__global__ __launch_bounds__(256, 2) void q4k_tile_kernel(const Q4kTileParams p) {
#pragma clang fp contract(off)
  __shared__ u32x4 xb[2][4][2][kParts][64];  // buffer, 16-row tile, sub-block, part
  __shared__ u32x4 wb[2][kTileN * 9];        // buffer, weight row's super-block
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r = lane & 15, g = lane >> 4;
  // Workgroups are dealt to the eight XCDs round robin: all row tiles of a
  // weight block run on one XCD, next to each other, and share its L2.
  const uint32_t nblocks = (p.N + kTileN - 1) / kTileN;
  const uint32_t local = blockIdx.x >> 3;
  const uint32_t nz = local / p.mtiles * 8 + (blockIdx.x & 7u), mb = local % p.mtiles;
  if (nz >= nblocks * p.ksplit) return;
  const uint32_t nb = nz % nblocks, z = nz / nblocks;
  const uint32_t KB = p.K / 32, SB = p.K / kQ4kBlockWeights;
  const uint32_t sb0 = z * SB / p.ksplit, sb1 = (z + 1) * SB / p.ksplit;
  const size_t row_bytes = (size_t)SB * kQ4kBlockBytes;

  // x: wave w stages 16-row tile w, contiguous in memory and in LDS.
  constexpr int XU = 2 * kParts;
  // (Buffer resources leave the addresses to scalar registers; none is larger
  // than 4 MiB.)
  auto rsrc = [](const void* base, uint32_t bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), 0, (int)bytes,
                                             kGemmBufferWord3);
  };
  const __amdgpu_buffer_rsrc_t xrs =
      rsrc(p.units + (size_t)(mb * 4 + wave) * KB * kParts * 64, KB * kParts * 1024);
  auto load_x = [&](u32x4 (&d)[XU], uint32_t s) {
#pragma unroll
    for (int u = 0; u < XU; ++u)
      d[u] = __builtin_amdgcn_raw_buffer_load_b128(xrs, lane * 16, (s * XU + u) * 1024, 0);
  };
  auto put_x = [&](int b, const u32x4 (&d)[XU]) {
#pragma unroll
    for (int u = 0; u < XU; ++u) xb[b][wave][u / kParts][u % kParts][lane] = d[u];
  };
  // Weights: 1152 entries of 16 bytes, entry i being bytes 16 (i % 9) .. of
  // weight row i / 9; thread t moves entries t, t + 256, ..., the last half
  // round entry 1151 once more.  Rows past the last read zeros.
  constexpr int WE = kTileN * 9, WU = (WE + 255) / 256;
  uint32_t wsrc[WU], wdst[WU];
  const uint32_t nfirst = nb * kTileN;
#pragma unroll
  for (int k = 0; k < WU; ++k) {
    wdst[k] = min((uint32_t)tid + 256 * k, (uint32_t)WE - 1);
    wsrc[k] = wdst[k] / 9 * (uint32_t)row_bytes + 16 * (wdst[k] % 9);
  }
  const __amdgpu_buffer_rsrc_t wrs =
      rsrc(p.w + (size_t)nfirst * row_bytes, min((uint32_t)kTileN, p.N - nfirst) * (uint32_t)row_bytes);
  // In two batches, entries 0-1 and 2-4 of each thread.
  auto load_w = [&](u32x4 (&d)[3], int batch, uint32_t sb) {
#pragma unroll
    for (int k = 0; k < 2 + batch; ++k)
      d[k] = __builtin_amdgcn_raw_buffer_load_b128(wrs, wsrc[2 * batch + k], sb * kQ4kBlockBytes, 0);
  };
  auto put_w = [&](uint32_t b, const u32x4 (&d)[3], int batch) {
#pragma unroll
    for (int k = 0; k < 2 + batch; ++k) wb[b][wdst[2 * batch + k]] = d[k];
  };
  // Third parts of the four row tiles (at most 2 MiB).
  const __amdgpu_buffer_rsrc_t x3rs = rsrc(p.third + (size_t)mb * 4 * KB * 64, 4 * KB * 1024);
  // Per super-block: row sums for the min product (row r of tile t, sub-block
  // g of each half) and the inverse scales of rows 4g .. 4g+3.
  const __amdgpu_buffer_rsrc_t sxrs = rsrc(p.sums + (size_t)mb * 4 * KB * 16, 4 * KB * 64);
  const __amdgpu_buffer_rsrc_t scrs = rsrc(p.scales + (size_t)mb * 4 * SB * 16, 4 * SB * 64);
  auto load_sx = [&](float (&d)[4][2], uint32_t sb) {
#pragma unroll
    for (int t = 0; t < 4; ++t)
#pragma unroll
      for (int hf = 0; hf < 2; ++hf)
        d[t][hf] = __builtin_bit_cast(
            float, __builtin_amdgcn_raw_buffer_load_b32(sxrs, lane * 4,
                                                        (t * KB + 8 * sb + 4 * hf) * 64, 0));
  };
  auto load_scale = [&](floatx4 (&d)[4], uint32_t sb) {
#pragma unroll
    for (int t = 0; t < 4; ++t)
      d[t] = __builtin_bit_cast(
          floatx4, __builtin_amdgcn_raw_buffer_load_b128(scrs, 16 * g, (t * SB + sb) * 64, 0));
  };
  // Lanes 0..3: a negative value where row tile `lane` has third parts (the
  // others read past the resource: zeros).
  auto load_flags = [&](uint32_t sb) {
    return __builtin_bit_cast(
        float, __builtin_amdgcn_raw_buffer_load_b32(scrs, lane < 4 ? lane * SB * 64 : kSkip,
                                                    sb * 64, 0));
  };

  const floatx4 zero = {0.f, 0.f, 0.f, 0.f};
  floatx4 acc[4][2];
#pragma unroll
  for (int t = 0; t < 4; ++t)
#pragma unroll
    for (int i = 0; i < 2; ++i) acc[t][i] = zero;

  const uint32_t slast = 4 * sb1 - 1;
  u32x4 xr[XU], wr[3];  // the next step's x and the next weights on their way
  float sx[4][2];
  floatx4 xsc[4];
  load_w(wr, 0, sb0);
  load_x(xr, 4 * sb0);
  put_w(0, wr, 0);
  load_w(wr, 1, sb0);
  put_w(0, wr, 1);
  put_x(0, xr);
  float flags = load_flags(sb0);
  lds_barrier();
  for (uint32_t sb = sb0; sb < sb1; ++sb) {
    const uint32_t wcur = (sb - sb0) & 1;
    const u32x4* wt = &wb[wcur][(wave * 32 + r) * 9];
    floatx4 part[4][2], rest[4][2];
    // Scales and zero points, one per byte (sub-blocks 0-3, 4-7), and the rests
    // of sub-blocks g and 4 + g.
    uint32_t sc[2][2], zp[2][2];
    float d[2], mc[2][2];
#pragma unroll
    for (int i = 0; i < 2; ++i) tile_header(wt[16 * 9 * i], g, sc[i], zp[i], d[i], mc[i]);
#pragma unroll
    for (int it = 0; it < 4; ++it) {
      // Step s: its operands are in buffers it & 1.
      const uint32_t s = 4 * sb + it;
      const int b = it & 1;
      load_x(xr, min(s + 1, slast));
      // The third parts' products, of the row tiles that have them, between two
      // steps: the scheduler has no overlap to lose there.
      const uint32_t third = it == 1 ? (uint32_t)__ballot(flags < 0.f) : 0u;
      if (it == 1 && third) {
#pragma nounroll
        for (int k = 0; k < 8; ++k) {
          f16x8 w[2];
#pragma unroll
          for (int i = 0; i < 2; ++i) {
            const u32x2 q = reinterpret_cast<const u32x2*>(wt + 16 * 9 * i + 1 + (k & 6))[g];
            const PairScale ps = pair_scale(sc[i][k >> 2] >> (8 * (k & 3)),
                                            zp[i][k >> 2] >> (8 * (k & 3)), 0);
            const uint32_t sh = k & 1 ? 0u : 4u;
            w[i] = weights_f16(u32x2{q.x << sh, q.y << sh}, ps.s.x, ps.zs.x);
          }
#pragma unroll
          for (int t = 0; t < 4; ++t) {
            if (!(third >> t & 1u)) continue;
            const f16x8 x3 = __builtin_bit_cast(
                f16x8, __builtin_amdgcn_raw_buffer_load_b128(x3rs, lane * 16,
                                                             (t * KB + 8 * sb + k) * 1024, 0));
#pragma unroll
            for (int i = 0; i < 2; ++i) {
              const floatx4 u = __builtin_amdgcn_mfma_f32_16x16x32_f16(x3, w[i], zero, 0, 0, 0);
#pragma unroll
              for (int e = 0; e < 4; ++e)
                rest[t][i][e] = __builtin_fmaf(u[e], kPartDown, rest[t][i][e]);
            }
          }
        }
      }
      if (it == 0) load_w(wr, 0, min(sb + 1, sb1 - 1));
      if (it == 2) load_w(wr, 1, min(sb + 1, sb1 - 1));
      if (it == 2) flags = load_flags(min(sb + 1, sb1 - 1));
      if (it == 3) {
        load_sx(sx, sb);
        load_scale(xsc, sb);
      }
      u32x2 q[2];
#pragma unroll
      for (int i = 0; i < 2; ++i)
        q[i] = reinterpret_cast<const u32x2*>(wt + 16 * 9 * i + 1 + 2 * it)[g];
      // Weight tile i's operands for the step's two sub-blocks.
      f16x8 xs[4][kParts], wq[2][2];
      auto weights = [&](int i) {
        const PairScale ps = pair_scale(sc[i][it >> 1], zp[i][it >> 1], it & 1);
        wq[0][i] = weights_f16(u32x2{q[i].x << 4, q[i].y << 4}, ps.s.x, ps.zs.x);
        wq[1][i] = weights_f16(q[i], ps.s.y, ps.zs.y);
      };
      auto read_x = [&](int t, int j) {
#pragma unroll
        for (int c = 0; c < kParts; ++c)
          xs[t][c] = __builtin_bit_cast(f16x8, xb[b][t][j][c][lane]);
      };
#pragma unroll
      for (int t = 0; t < 4; ++t) read_x(t, 0);
      weights(0);
      weights(1);
#pragma unroll
      for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int t = 0; t < 4; ++t) {
          const bool first = it == 0 && j == 0;
#pragma unroll
          for (int i = 0; i < 2; ++i)
            part[t][i] = __builtin_amdgcn_mfma_f32_16x16x32_f16(
                xs[t][0], wq[j][i], first ? zero : part[t][i], 0, 0, 0);
#pragma unroll
          for (int c = 1; c < kParts; ++c)
#pragma unroll
            for (int i = 0; i < 2; ++i)
              rest[t][i] = __builtin_amdgcn_mfma_f32_16x16x32_f16(
                  xs[t][c], wq[j][i], first && c == 1 ? zero : rest[t][i], 0, 0, 0);
          if (j == 0) read_x(t, 1);  // into the registers just used
          __builtin_amdgcn_sched_barrier(0);
        }
      // The other buffers were last read in step s - 1 (x) and in the
      // super-block before (weights).
      put_x(b ^ 1, xr);
      if (it == 1) put_w(wcur ^ 1, wr, 0);
      if (it == 3) put_w(wcur ^ 1, wr, 1);
      lds_barrier();
    }
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        floatx4 m = __builtin_amdgcn_mfma_f32_16x16x4f32(sx[t][0], mc[i][0], zero, 0, 0, 0);
        m = __builtin_amdgcn_mfma_f32_16x16x4f32(sx[t][1], mc[i][1], m, 0, 0, 0);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const float u = __builtin_fmaf(rest[t][i][e], kPartDown, part[t][i][e]);
          acc[t][i][e] += __builtin_fmaf(u * (kOperandUp * d[i]), fabsf(xsc[t][e]), m[e]);
        }
        pin(acc[t][i]);
      }
  }

  float* y = p.y + z * p.y_split;
#pragma unroll
  for (int t = 0; t < 4; ++t)
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const uint32_t mo = mb * kTileM + 16 * t + 4 * g + e;
      if (mo >= p.M) continue;
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const uint32_t no = nb * kTileN + wave * 32 + 16 * i + r;
        if (no >= p.N) continue;
        float v = acc[t][i][e];
        if (p.ksplit == 1) {
          if (!is_finite(v))
            v = row_dot(p.w + (size_t)no * row_bytes, p.x + (size_t)mo * p.ldx, nullptr, p.K);
          if (p.res) v += p.res[(size_t)mo * p.ldr + no];
        }
        y[(size_t)mo * p.ldy + no] = v;
      }
    }
}

// The K ranges' products added in range order, and the residual.
__global__ __launch_bounds__(256) void q4k_tile_sum_kernel(const Q4kTileParams p,
                                                           const float* __restrict__ part) {
#pragma clang fp contract(off)
  const uint32_t n = blockIdx.x * 256 + threadIdx.x, m = blockIdx.y;
  if (n >= p.N) return;
  const size_t i = (size_t)m * p.N + n;
  float v = part[i];
  for (uint32_t z = 1; z < p.ksplit; ++z) v += part[z * p.y_split + i];
  if (!is_finite(v))
    v = row_dot(p.w + (size_t)n * (p.K / kQ4kBlockWeights * kQ4kBlockBytes),
                p.x + (size_t)m * p.ldx, nullptr, p.K);
  if (p.res) v += p.res[(size_t)m * p.ldr + n];
  p.y[(size_t)m * p.ldy + n] = v;
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

template <int XL, int R>
int launch_vec(const Q4kGemmParams& p, uint32_t nout, hipStream_t stream) {
  constexpr uint32_t rows = R * (XL <= 4 ? 4 : XL <= 8 ? 2 : 1);
  const dim3 grid((nout + rows - 1) / rows, p.M, p.Z), block(64);
  auto kernel = p.swiglu_f ? (p.norm_alpha ? q4k_vec_kernel<XL, R, true, true>
                                           : q4k_vec_kernel<XL, R, false, true>)
                           : (p.norm_alpha ? q4k_vec_kernel<XL, R, true, false>
                                           : q4k_vec_kernel<XL, R, false, false>);
  hipLaunchKernelGGL(kernel, grid, block, 0, stream, p, NoAttention{});
  STS_HIP(hipGetLastError());
  return STS_OK;
}

// Many rows: x split once into scratch memory, then the 64 x 128 tiles, in
// chunks of at most kTileRows rows so that the scratch stays bounded.
// *done stays false where the scratch is not to be had.
constexpr uint32_t kTileRows = 1024;
int launch_tiles(const Q4kGemmParams& p, hipStream_t stream, bool* done) {
  const uint32_t KB = p.K / 32, SB = p.K / kQ4kBlockWeights;
  const uint32_t nblocks = (p.N + kTileN - 1) / kTileN;
  const uint32_t cus = (uint32_t)device_cu_count();
  const uint32_t rows = (std::min(p.M, kTileRows) + kTileM - 1) / kTileM * kTileM;
  // K ranges per output tile: as many as keep the launch within the two
  // workgroups a CU holds, each at least four super-blocks.
  const uint32_t tiles = nblocks * (rows / kTileM);
  const uint32_t ksplit = std::max(1u, std::min(2 * cus / tiles, SB / 4));
  const size_t plane_floats = TilePlanes::floats(rows, KB);
  const size_t y_floats = ksplit > 1 ? (size_t)rows * p.N : 0;
  const Scratch scratch(stream, plane_floats + ksplit * y_floats, 0);  // held to the last launch
  if (!scratch.part) return STS_OK;
  const TilePlanes planes(scratch.part, rows, KB);
  float* part = scratch.part + plane_floats;
  for (uint32_t m0 = 0; m0 < p.M; m0 += kTileRows) {
    Q4kTileParams t;
    t.w = p.w[0];
    t.units = planes.units;
    t.third = planes.third;
    t.sums = planes.sums;
    t.scales = planes.scales;
    t.x = p.x + (size_t)m0 * p.ldx;
    t.res = p.res ? p.res + (size_t)m0 * p.ldr : nullptr;
    t.y = p.y + (size_t)m0 * p.ldy;
    t.ldx = p.ldx;
    t.ldr = p.ldr;
    t.ldy = p.ldy;
    t.y_split = 0;
    t.M = std::min(p.M - m0, kTileRows);
    t.N = p.N;
    t.K = p.K;
    t.mtiles = (t.M + kTileM - 1) / kTileM;
    t.ksplit = ksplit;
    hipLaunchKernelGGL(split_planes_kernel, dim3((SB + 3) / 4, t.mtiles * 4), dim3(256), 0, stream,
                       t.x, t.ldx, t.M, SB, planes);
    STS_HIP(hipGetLastError());
    const uint64_t grid = (uint64_t)((nblocks * ksplit + 7) / 8) * 8 * t.mtiles;
    if (grid > 0x7FFFFFFFull) return fail(STS_ERR_INVALID, "GEMM N = %u too large", p.N);
    Q4kTileParams k = t;
    if (ksplit > 1) {
      k.y = part;
      k.ldy = p.N;
      k.y_split = t.y_split = y_floats;
    }
    hipLaunchKernelGGL(q4k_tile_kernel, dim3((uint32_t)grid), dim3(256), 0, stream, k);
    STS_HIP(hipGetLastError());
    if (ksplit > 1) {
      hipLaunchKernelGGL(q4k_tile_sum_kernel, dim3((p.N + 255) / 256, t.M), dim3(256), 0, stream,
                         t, part);
      STS_HIP(hipGetLastError());
    }
  }
  *done = true;
  return STS_OK;
}

}  // namespace

int launch_q4k_attention(const Q4kGemmParams& p, const DepthAttention& a, hipStream_t stream) {
  if (p.M == 0 || p.M > 2 || p.N == 0 || p.Z != 1 || p.K == 0 || p.K % kQ4kBlockWeights != 0 ||
      p.K > 1024 || p.swiglu_f || p.norm_alpha || a.len == 0 || a.len > a.max_len)
    return fail(STS_ERR_INVALID, "attention and projection M=%u N=%u K=%u len=%u of %u", p.M, p.N,
                p.K, a.len, a.max_len);
  if ((uint64_t)a.max_len * p.K * sizeof(float) > 0x7FFFFFF0ull)
    return fail(STS_ERR_INVALID, "cache of %u slots too large", a.max_len);
  const dim3 grid((p.N + 3) / 4, p.M), block(64);
  hipLaunchKernelGGL((q4k_vec_kernel<4, 1, false, false, DepthAttention>), grid, block, 0, stream,
                     p, a);
  STS_HIP(hipGetLastError());
  return STS_OK;
}

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
  // One or two rows of x, measured against q4k_rows_kernel: 1 x [48000, 1024]
  // 8.2 and 15.1 us, [48000, 4096] 30.6 and 46.5; 2 x [48000, 1024] 13.1 and
  // 14.8, [48000, 2048] 28.0 and 27.7, [4096, 4096] 6.7 and 8.8.  The second row
  // unpacks the weights again, which beyond that costs more than the 16-row
  // tile: 2 x [16384, 3072] 19.8 and 13.2, [48000, 4096] 56.7 and 48.2.
  if (p.K <= 4096 && (p.M == 1 || (p.M == 2 && (p.K <= 2048 || nout * p.Z <= 16 * cus)))) {
    // A wave per few weight rows; where that would be more than eight waves a
    // CU, four times the rows.
    const uint64_t waves = (uint64_t)nout * p.M * p.Z / (p.K <= 1024 ? 4 : p.K <= 2048 ? 2 : 1);
    const bool many = waves > 8ull * cus;
    if (p.K <= 1024) return many ? launch_vec<4, 4>(p, nout, stream) : launch_vec<4, 1>(p, nout, stream);
    if (p.K <= 2048) return many ? launch_vec<8, 4>(p, nout, stream) : launch_vec<8, 1>(p, nout, stream);
    if (p.K <= 3072) return many ? launch_vec<12, 4>(p, nout, stream) : launch_vec<12, 1>(p, nout, stream);
    return many ? launch_vec<16, 4>(p, nout, stream) : launch_vec<16, 1>(p, nout, stream);
  }
  // Weight tiles per workgroup: as many as bring the launch to about one
  // workgroup per CU, up to six (eight spill registers).  Every workgroup splits
  // its x rows itself, so fewer and larger workgroups split them less often:
  // two per CU measured, with x in bf16 parts, 12.7 against 8.1 us (64 rows x
  // [3072, 1024]) and 28.7 against 19.2 us (13 x [12288, 4096]); and waves beyond
  // eight leave too few registers (12: 16.9 and 32.0 us).
  const uint64_t tiles = (uint64_t)ntiles * mtiles * p.Z;
  // The tiles from 33 rows on, where the products outweigh their two extra
  // launches (x split, K ranges summed): 48 rows x [12288, 4096] 37 against
  // 60 us here, 112 x [4096, 4096] 32 against 59, 512 x [22528, 4096] 256
  // against 866, but 80 x [4096, 4096] 31.4 against 32.3, 32 x [12288, 4096]
  // 35 against 32.
  if (p.scratch && p.M > 32 && (uint64_t)mtiles * 16 * p.N * p.K >= 1500000000ull && p.Z == 1 &&
      !p.swiglu_f && !p.norm_alpha) {
    bool done = false;
    if (int rc = launch_tiles(p, stream, &done)) return rc;
    if (done) return STS_OK;
  }
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
