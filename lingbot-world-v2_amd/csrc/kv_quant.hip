// fp8-e4m3fn KV-cache quantiser (gfx950). No reference counterpart: the format is defined
// here. Per (batch, head, block of `block` tokens by absolute index in the buffer):
//   amax  = max |x| over the block's tokens and all head_dim features (fp32)
//   scale = the smallest power of two 2^k >= amax / 448 (k >= -126), or 1 when amax == 0
//   inv   = 1 / scale = 2^-k (exact)
//   code  = round_to_nearest_even_e4m3fn(x * inv)
// Power-of-two scales make a code times its scale exact in bf16: the attention kernel applies
// K's scale as the exponent scale of its fp8 matrix-core product and V's in the exact
// conversion of the codes to bf16, so neither enters the softmax arithmetic.
// HBM-bound: 3 bytes per value, little work on each. One workgroup of 4 waves per (b, h, block):
// 8 lanes cover a token row of 128 values, 32 bytes each, so a row's codes leave as 8 x 16 bytes;
// the block's values stay in registers as they were read (16 bytes x 4 per lane), their largest
// magnitude is found on the packed 16-bit patterns, and the codes come from the packed converter
// v_cvt_scalef32_pk_fp8_bf16 (two values per instruction; for every finite bf16 value, every scale
// exponent that can occur, it gives the code of the integer encoder below). A block with an
// infinity or a NaN, which the packed maximum would misread, takes the integer encoder.
// Measured at 3600 tokens x 40 heads (55 MB, rotating buffers): 12.6 us (4.4 TB/s), 21.5 us with
// the integer encoder on fp32 values for all; 1, 2 and 8 waves per block 13.3, 13.0 and 13.6 us.
// Workgroups are numbered with (b, h) fastest.

#include "common.h"
#include "attn_fwd.h"

namespace lbw {

// fp32 -> OCP e4m3fn code, round to nearest even; |x| >= 480 -> NaN (0x7f), matching
// torch's float8_e4m3fn cast. Written with integer ops so the result does not depend on a
// hardware conversion mode.
__device__ __forceinline__ uint32_t e4m3fn_encode(float x) {
  const uint32_t u = __float_as_uint(x);
  const uint32_t sign = (u >> 24) & 0x80u;
  const uint32_t au = u & 0x7fffffffu;
  if (au >= 0x43f00000u) return sign | 0x7fu;            // >= 480 or NaN
  if (au < 0x3c800000u) {                                // < 2^-6: subnormal, step 2^-9
    const float ax = __uint_as_float(au);
    const uint32_t m = (uint32_t)__float2int_rn(ax * 512.0f);  // exact scale, RNE
    return sign | m;                                     // m == 8 is the min normal
  }
  const uint32_t r = au + 0x7ffffu + ((au >> 20) & 1u);  // RNE on the 20 dropped bits
  const uint32_t code = (r >> 20) - (120u << 3);         // rebias 127 -> 7
  return sign | (code > 0x7fu ? 0x7fu : code);
}

// Four bf16 values (two packed pairs) times 1 / scale -> four codes.
__device__ __forceinline__ uint32_t e4m3fn_pack4(uint32_t w0, uint32_t w1, float scale) {
  typedef short shortx2 __attribute__((ext_vector_type(2)));
  shortx2 r = {0, 0};
  r = __builtin_amdgcn_cvt_scalef32_pk_fp8_bf16(r, __builtin_bit_cast(bf16x2, w0), scale, false);
  r = __builtin_amdgcn_cvt_scalef32_pk_fp8_bf16(r, __builtin_bit_cast(bf16x2, w1), scale, true);
  return __builtin_bit_cast(uint32_t, r);
}

constexpr int KQ_WAVES = 4;                  // waves per workgroup
constexpr int KQ_BLOCK = 64;                 // tokens per scale block
constexpr int KQ_PASSES = KQ_BLOCK / (8 * KQ_WAVES);  // token rows per lane (8 lanes per row)
constexpr uint32_t KQ_INF = 0x7f80u;         // bf16 infinity; larger magnitudes are NaN

// largest value over the workgroup, in every lane
__device__ __forceinline__ uint32_t kq_reduce_max(uint32_t m, uint32_t* red) {
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) {
    const uint32_t y = (uint32_t)__shfl_xor((int)m, o);
    m = y > m ? y : m;
  }
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = m;
  __syncthreads();
#pragma unroll
  for (int w = 0; w < KQ_WAVES; ++w) m = red[w] > m ? red[w] : m;
  return m;
}

__global__ void __launch_bounds__(KQ_WAVES * 64)
kv_quant_fp8_kernel(const KvQuantArgs a) {
  typedef uint16_t u16x2 __attribute__((ext_vector_type(2)));
  __shared__ uint32_t red[2][KQ_WAVES];
  // heads fastest: neighbouring workgroups read and write the same token rows (each row holds
  // every head), which keeps the HBM accesses of concurrent workgroups together
  const uint32_t nbh = (uint32_t)(a.B * a.H);
  const uint32_t bh = blockIdx.x % nbh;
  const int64_t blk = blockIdx.x / nbh;
  const int h = (int)(bh % (uint32_t)a.H);
  const int b = (int)(bh / (uint32_t)a.H);
  const int t = threadIdx.x;
  const int col = 16 * (t & 7);          // first of this lane's 16 values of a row
  const int r0 = t >> 3;
  const int64_t tok0 = blk * KQ_BLOCK;
  const int nrow = (int)(a.L - tok0 < KQ_BLOCK ? a.L - tok0 : KQ_BLOCK);

  u32x4 x[KQ_PASSES][2];
  const uint16_t* src = a.x + a.sb * b + a.sl * tok0 + a.sh * h + col;
#pragma unroll
  for (int i = 0; i < KQ_PASSES; ++i) {
    const int row = r0 + 8 * KQ_WAVES * i;
    x[i][0] = x[i][1] = u32x4{0u, 0u, 0u, 0u};
    if (row < nrow) {
      const u32x4* p = reinterpret_cast<const u32x4*>(src + a.sl * row);
      x[i][0] = p[0];
      x[i][1] = p[1];
    }
  }
  // the largest magnitude, as a bf16 pattern
  u16x2 mm = {0, 0};
#pragma unroll
  for (int i = 0; i < KQ_PASSES; ++i)
#pragma unroll
    for (int j = 0; j < 8; ++j)
      mm = __builtin_elementwise_max(
          mm, __builtin_bit_cast(u16x2, x[i][j >> 2][j & 3] & 0x7fff7fffu));
  uint32_t amax = kq_reduce_max(mm[0] > mm[1] ? mm[0] : mm[1], red[0]);
  const bool finite = amax < KQ_INF;     // of the whole block
  if (!finite) {  // NaNs take no part in the maximum
    uint32_t m = 0;
#pragma unroll
    for (int i = 0; i < KQ_PASSES; ++i)
#pragma unroll
      for (int j = 0; j < 16; ++j) {
        const uint32_t v = (x[i][j >> 3][(j >> 1) & 3] >> (16 * (j & 1))) & 0x7fffu;
        m = v <= KQ_INF && v > m ? v : m;
      }
    amax = kq_reduce_max(m, red[1]);
  }
  // amax = m 2^E, m in [1, 2): amax / 2^k <= 1.75 * 2^8 from k = E - 8 on when m <= 1.75
  // (mantissa field <= 0x600000), else from k = E - 7; a subnormal amax gets k = -126
  int k = 0;
  if (amax > 0) {
    const uint32_t u = amax << 16;
    const int eb = (int)(u >> 23);
    k = eb == 0 ? -126 : eb - 127 - ((u & 0x7fffffu) <= 0x600000u ? 8 : 7);
    k = k < -126 ? -126 : k;
  }
  const float scale = __uint_as_float((uint32_t)(127 + k) << 23);
  if (t == 0) a.scales[(int64_t)bh * a.nblk + blk] = scale;
  uint8_t* dst = a.codes + (((int64_t)b * a.L + tok0) * a.H + h) * a.D + col;
  const int64_t row_b = (int64_t)a.H * a.D;
#pragma unroll
  for (int i = 0; i < KQ_PASSES; ++i) {
    const int row = r0 + 8 * KQ_WAVES * i;
    if (row < nrow) {
      u32x4 o;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const uint32_t w0 = x[i][j >> 1][2 * (j & 1)], w1 = x[i][j >> 1][2 * (j & 1) + 1];
        if (finite) {
          o[j] = e4m3fn_pack4(w0, w1, scale);
        } else {
          const float inv = __uint_as_float((uint32_t)(127 - k) << 23);
          o[j] = e4m3fn_encode(__fmul_rn(bf16_lo(w0), inv)) |
                 e4m3fn_encode(__fmul_rn(bf16_hi(w0), inv)) << 8 |
                 e4m3fn_encode(__fmul_rn(bf16_lo(w1), inv)) << 16 |
                 e4m3fn_encode(__fmul_rn(bf16_hi(w1), inv)) << 24;
        }
      }
      *reinterpret_cast<u32x4*>(dst + row_b * row) = o;
    }
  }
}

hipError_t launch_kv_quant_fp8(const KvQuantArgs& a, hipStream_t stream) {
  const int64_t nwg = (int64_t)a.B * a.H * a.nblk;
  hipLaunchKernelGGL(kv_quant_fp8_kernel, dim3((uint32_t)nwg), dim3(KQ_WAVES * 64), 0, stream, a);
  return hipGetLastError();
}

}  // namespace lbw
