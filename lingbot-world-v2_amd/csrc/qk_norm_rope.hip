// Fused q/k RMSNorm + Wan 3-D RoPE (+ optional V copy into the KV cache slot), gfx950.
//
// Restates kernels/qk_post.py:88-141 (qk_norm_rope) with the sum of squares of
// kernels/qk_post.py:49-73 folded in (one GPU holds the full row, so no all-reduce):
//   y = x + b (fp32); r = 1 / sqrt(sum(y^2) / C + eps); t = bf16(y * r) * gamma (fp32);
//   RoPE on interleaved pairs (fp32, separate multiplies and adds as torch does them), the
//   output scale folded into cos and sin first as kernels/qk_post.py:259-265 does it
//   (cs = cos * s, sn = sin * s in fp32); out = bf16(rot). Rows that are not rotated are
//   out = bf16(t * s).
// RoPE angles follow wan/modules/model_fast.py:878-931: token (fi, hi, wi) of the
// frame-major grid takes pair j's cos/sin from the frame table (j < s0), the height table
// (j < s0 + s1) or the width table. Tokens past f*h*w are not rotated (model_fast.py:972-975).
//
// Two output layouts:
// - rows: q', k' as [L, C] rows (strided), the layout the attention kernel reads;
// - d-major: q', k' as [H, D, L] (token stride 1, a given d stride, head stride D * d stride),
//   the layout of kernels/qk_post.py:228-306 (qk_norm_rope_t). A workgroup of 8 or 16 waves takes 16
//   or 32 consecutive tokens of one tensor, stages each 512-column slice of their outputs in LDS
//   and writes it transposed: 32 or 64 bytes of consecutive tokens per (head, d) line. Tiles are numbered so
//   that each XCD takes a contiguous run of them, and the two 32-byte halves of a 64-byte line are
//   usually written through the same L2.
// With k == NULL only q is processed (kernels/qk_post.py:144-215, 308-402: x_norm_rope and
// x_norm_rope_t3 on one tensor).
//
// HBM-bound, with enough VALU work per byte (unpacking, the bf16 rounding, the rotation) that
// the loads of some waves must overlap the arithmetic of others: one wave holds one tensor's
// token row (lane l holds the 16-byte chunks l, l + 64, ... of the row, NCH of them), which
// keeps it near 120 registers and four waves per SIMD. With the head dim dividing 512 every
// chunk of a lane covers the same 4 rotation pairs, fetched once per row. The per-axis RoPE
// tables and the bias / gamma vectors sit in LDS.

#include "common.h"
#include "attn_fwd.h"

namespace lbw {

constexpr int QK_WAVES = 8;                // waves per workgroup, rows layout
constexpr int QK_MAX_BLOCKS = 512;         // rows layout: two resident per CU, looping over rows
constexpr int QT_TILE = 16, QT_LONG = 32;  // d-major layout: tokens per workgroup, long chunks
constexpr int QT_MAX_NCH = 10;             // d-major: two rows of C <= 5120 fit 128 registers
constexpr int QT_PITCH = 544;              // bf16 per staged token row: the transpose read's four
                                           // rows of two column groups cover the 64 banks once
constexpr int QK_MAX_TABLE = 16384;        // floats of per-axis tables held in LDS (64 KB)
constexpr int LDS_LIMIT = 160 * 1024;
static_assert(QK_MAX_TABLE * 4 + 2 * QT_MAX_NCH * 512 * 2 + 2 * QT_LONG * QT_PITCH * 2 <= LDS_LIMIT,
              "the larger tile fits beside any tables");

int qk_norm_rope_max_table_floats() { return QK_MAX_TABLE; }

// LDS layout: [ntab floats of tables][bq | bk | gq | gk as bf16, C each][d-major staging]
__host__ __device__ inline int qk_table_floats(int ntab) { return (ntab + 3) & ~3; }
__host__ __device__ inline size_t qk_lds_bytes(int ntab, int C) {
  return (size_t)qk_table_floats(ntab) * 4 + (size_t)4 * C * 2;
}
// d-major: [tables][bias, gamma][2 stage buffers of a tile's rows]
static size_t qt_lds_bytes(int ntab, int C, int tile) {
  return (size_t)qk_table_floats(ntab) * 4 + (size_t)2 * C * 2 + (size_t)2 * tile * QT_PITCH * 2;
}

size_t qk_norm_rope_lds_bytes(int ntab, int C, int layout) {
  return layout == QK_LAYOUT_DMAJOR ? qt_lds_bytes(ntab, C, QT_TILE) : qk_lds_bytes(ntab, C);
}
size_t qk_norm_rope_lds_limit() { return LDS_LIMIT; }
int qk_norm_rope_dmajor_max_dim() { return QT_MAX_NCH * 64 * 8; }

// tables and vectors into LDS, several loads in flight per thread (unrolled by 4)
__device__ __forceinline__ void qk_fill_lds(const QkNormRopeArgs& a, float* tab, uint16_t* vec) {
  const int nchunk = a.C / 8;
  const int nt2 = a.ntab / 2;  // cos/sin values come in pairs: 8-byte loads
#pragma unroll 4
  for (int i = threadIdx.x; i < nt2; i += blockDim.x)
    reinterpret_cast<u32x2*>(tab)[i] = reinterpret_cast<const u32x2*>(a.rope)[i];
  const uint16_t* src[4] = {a.bq, a.bk, a.wq, a.wk};
#pragma unroll
  for (int v = 0; v < 4; ++v) {
    if (src[v] != nullptr) {
#pragma unroll 4
      for (int ch = threadIdx.x; ch < nchunk; ch += blockDim.x)
        *reinterpret_cast<u32x4*>(vec + v * a.C + 8 * ch) =
            *reinterpret_cast<const u32x4*>(src[v] + 8 * ch);
    } else {
      for (int ch = threadIdx.x; ch < nchunk; ch += blockDim.x)
        *reinterpret_cast<u32x4*>(vec + v * a.C + 8 * ch) = u32x4{0u, 0u, 0u, 0u};
    }
  }
}

// One tensor's token row held by one wave: its raw chunks, the inverse norm and this lane's
// four rotation pairs with the tensor's output scale folded in.
template <int NCH>
struct QkOne {
  u32x4 x[NCH];
  float r;
  float c[4], sn[4];
  bool rotate;
};

// The operands of one tensor (t = 0: q, t = 1: k).
struct QkTensor {
  const uint16_t* x; int64_t xs;
  uint16_t* o; int64_t os;
  const uint16_t* bias;   // LDS, C bf16
  const uint16_t* gamma;  // LDS, C bf16
  float scale;
};

__device__ __forceinline__ QkTensor qk_tensor(const QkNormRopeArgs& a, const uint16_t* vec, int t) {
  QkTensor u;
  u.x = t ? a.k : a.q;
  u.xs = t ? a.ks : a.qs;
  u.o = t ? a.ko : a.qo;
  u.os = t ? a.kos : a.qos;
  u.bias = vec + t * a.C;
  u.gamma = vec + (2 + t) * a.C;
  u.scale = t ? a.k_scale : a.q_scale;
  return u;
}

// 16 bytes of a row read once: NT, the non-temporal hint (the d-major kernel: its rows stream
// past the caches, 17 % less time at the 14B 720p chunk; the rows kernel, whose outputs the
// attention reads next, measured 7 % slower with it in the layer sequence and keeps plain loads)
template <bool NT>
__device__ __forceinline__ u32x4 qk_load16(const uint16_t* p) {
  if constexpr (NT) return __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(p));
  else return *reinterpret_cast<const u32x4*>(p);
}

// issue the loads of one tensor's row (kept apart from qk_one_norm so that a wave can have the
// loads of several rows in flight)
template <int NCH, bool NT>
__device__ __forceinline__ void qk_one_load(const QkNormRopeArgs& a, const QkTensor& u, int row,
                                            int lane, QkOne<NCH>& s) {
  const int nchunk = a.C / 8;
  const uint16_t* xr = u.x + u.xs * row;
#pragma unroll
  for (int i = 0; i < NCH; ++i) {
    const int ch = lane + 64 * i;
    if (i + 1 < NCH || ch < nchunk)  // only the last chunk can run past the row
      s.x[i] = qk_load16<NT>(xr + 8 * ch);
  }
}

// rotation pairs, sum of squares and inverse norm of a loaded row
template <int NCH>
__device__ __forceinline__ void qk_one_norm(const QkNormRopeArgs& a, const float* tab,
                                            const QkTensor& u, int row, int lane, QkOne<NCH>& s) {
  const int C = a.C;
  const int nchunk = C / 8;
  // ---- this lane's 4 rotation pairs for the row's (frame, row, column)
  const int D = C / a.H;
  const int j0 = ((8 * lane) % D) / 2;  // first rotation pair of every chunk of this lane
  s.rotate = row < a.gf * a.gh * a.gw;
  if (s.rotate) {
    const int base_h = 2 * a.gf * a.s0;
    const int base_w = base_h + 2 * a.gh * a.s1;
    const int wi = row % a.gw;
    const int hi = (row / a.gw) % a.gh;
    const int fi = row / (a.gw * a.gh);
#pragma unroll
    for (int p = 0; p < 4; ++p) {
      const int j = j0 + p;
      int ci, si;
      if (j < a.s0) {
        ci = fi * a.s0 + j;
        si = ci + a.gf * a.s0;
      } else if (j < a.s0 + a.s1) {
        ci = base_h + hi * a.s1 + (j - a.s0);
        si = ci + a.gh * a.s1;
      } else {
        ci = base_w + wi * a.s1 + (j - a.s0 - a.s1);
        si = ci + a.gw * a.s1;
      }
      s.c[p] = __fmul_rn(tab[ci], u.scale);
      s.sn[p] = __fmul_rn(tab[si], u.scale);
    }
  }

  // ---- sum of squares of y = x + b (per lane in chunk order, then across the wave)
  float ss = 0.0f;
#pragma unroll
  for (int i = 0; i < NCH; ++i) {
    const int ch = lane + 64 * i;
    if (i + 1 < NCH || ch < nchunk) {
      const u32x4 b = *reinterpret_cast<const u32x4*>(u.bias + 8 * ch);
#pragma unroll
      for (int w = 0; w < 4; ++w) {
        const float y0 = __fadd_rn(bf16_lo(s.x[i][w]), bf16_lo(b[w]));
        const float y1 = __fadd_rn(bf16_hi(s.x[i][w]), bf16_hi(b[w]));
        ss = __fmaf_rn(y0, y0, ss);
        ss = __fmaf_rn(y1, y1, ss);
      }
    }
  }
  ss = wave_reduce_sum(ss);
  s.r = 1.0f / sqrtf(__fadd_rn(__fmul_rn(ss, a.inv_c), a.eps));

  // recompute y = x + b when finishing (bias re-read from LDS) rather than keeping the fp32
  // values and bias chunks of the first pass alive
#pragma unroll
  for (int i = 0; i < NCH; ++i) asm volatile("" : "+v"(s.x[i]));
  asm volatile("" ::: "memory");
}

// normalise, gamma, rotate (scale folded into c/s) or scale, round: one 8-element chunk
__device__ __forceinline__ u32x4 qk_finish(const u32x4& x, const u32x4& bv, const u32x4& gv,
                                          float r, const float (&c)[4], const float (&sn)[4],
                                          bool rotate, float scale) {
  float t[8];
#pragma unroll
  for (int w = 0; w < 4; ++w) {
    const float y0 = __fadd_rn(bf16_lo(x[w]), bf16_lo(bv[w]));
    const float y1 = __fadd_rn(bf16_hi(x[w]), bf16_hi(bv[w]));
    t[2 * w] = __fmul_rn(round_bf16(__fmul_rn(y0, r)), bf16_lo(gv[w]));
    t[2 * w + 1] = __fmul_rn(round_bf16(__fmul_rn(y1, r)), bf16_hi(gv[w]));
  }
  float o[8];
  if (rotate) {
#pragma unroll
    for (int p = 0; p < 4; ++p) {
      const float re = t[2 * p], im = t[2 * p + 1];
      o[2 * p] = __fsub_rn(__fmul_rn(re, c[p]), __fmul_rn(im, sn[p]));
      o[2 * p + 1] = __fadd_rn(__fmul_rn(re, sn[p]), __fmul_rn(im, c[p]));
    }
  } else if (scale != 1.0f) {
#pragma unroll
    for (int e = 0; e < 8; ++e) o[e] = __fmul_rn(t[e], scale);
  } else {
#pragma unroll
    for (int e = 0; e < 8; ++e) o[e] = t[e];
  }
  u32x4 ov;
#pragma unroll
  for (int w = 0; w < 4; ++w) ov[w] = pack_bf16x2(o[2 * w], o[2 * w + 1]);
  return ov;
}

// copy the chunks i of a V row with i % nsplit == part (the row's waves share the copy)
template <int NCH>
__device__ __forceinline__ void qk_copy_v(const QkNormRopeArgs& a, int row, int lane, int part,
                                          int nsplit) {
  const int nchunk = a.C / 8;
  const uint16_t* vs = a.v + a.vs * row;
  uint16_t* vd = a.vo + a.vos * row;
  u32x4 xv[NCH];
#pragma unroll
  for (int i = 0; i < NCH; ++i) {
    const int ch = lane + 64 * i;
    if (i % nsplit == part && (i + 1 < NCH || ch < nchunk))
      xv[i] = *reinterpret_cast<const u32x4*>(vs + 8 * ch);
  }
#pragma unroll
  for (int i = 0; i < NCH; ++i) {
    const int ch = lane + 64 * i;
    if (i % nsplit == part && (i + 1 < NCH || ch < nchunk))
      *reinterpret_cast<u32x4*>(vd + 8 * ch) = xv[i];
  }
}

// the same for the d-major kernel, with the number of parts known to the compiler and the
// non-temporal hint on both sides (qk_load16). The form above takes more registers than that kernel
// has: the chunks of a row of up to 8 become one array of 32 registers that is merged whole at
// every chunk's branch. It spilled 132 to 772 bytes per lane at 6 to 8 chunks, and with the V copy
// 3600 tokens x 32 heads took 324 us where this form takes 46.
template <int NCH, int NSPLIT>
__device__ __forceinline__ void qk_copy_v_part(const QkNormRopeArgs& a, int row, int lane,
                                               int part) {
  constexpr int N = (NCH + NSPLIT - 1) / NSPLIT;
  const int nchunk = a.C / 8;
  const uint16_t* vs = a.v + a.vs * row;
  uint16_t* vd = a.vo + a.vos * row;
  u32x4 xv[N];
#pragma unroll
  for (int j = 0; j < N; ++j) {
    const int ch = lane + 64 * (NSPLIT * j + part);
    if (NSPLIT * (j + 1) < NCH || ch < nchunk) xv[j] = qk_load16<true>(vs + 8 * ch);
  }
#pragma unroll
  for (int j = 0; j < N; ++j) {
    const int ch = lane + 64 * (NSPLIT * j + part);
    if (NSPLIT * (j + 1) < NCH || ch < nchunk)
      __builtin_nontemporal_store(xv[j], reinterpret_cast<u32x4*>(vd + 8 * ch));
  }
}

// Four rows of one column per lane, from LDS (attn_tiles.h's transpose read).
__device__ __forceinline__ u32x2 qk_read_tr16(int addr) {
  typedef short shortx4 __attribute__((ext_vector_type(4)));
  typedef __attribute__((address_space(3))) shortx4 lds_shortx4;
  return __builtin_bit_cast(u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_shortx4*)(uintptr_t)addr));
}

// ---------------------------------------------------------------- rows layout
// One wave per (row, tensor): with q and k the workgroup's waves pair up, wave 2j taking row
// j's q and wave 2j + 1 its k (and half of its V copy each). A wave holds one tensor's row, so
// the kernel runs four waves per SIMD and one wave's loads overlap another's arithmetic.
template <int NCH>
__global__ void __launch_bounds__(QK_WAVES * 64)
qk_norm_rope_kernel(const QkNormRopeArgs a) {
  extern __shared__ __attribute__((aligned(16))) float smem[];
  const int C = a.C;
  const int nchunk = C / 8;
  float* tab = smem;
  uint16_t* vec = reinterpret_cast<uint16_t*>(smem + qk_table_floats(a.ntab));
  qk_fill_lds(a, tab, vec);
  __syncthreads();

  const int lane = threadIdx.x & 63;
  // (a scalar, so that the row's position, branches and addresses are; 114 registers before, 96)
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int ntens = a.k != nullptr ? 2 : 1;
  const int t = wave % ntens;
  const int rows_per_block = QK_WAVES / ntens;
  const QkTensor u = qk_tensor(a, vec, t);

  for (int row = blockIdx.x * rows_per_block + wave / ntens; row < a.L;
       row += gridDim.x * rows_per_block) {
    QkOne<NCH> s;
    qk_one_load<NCH, false>(a, u, row, lane, s);
    qk_one_norm<NCH>(a, tab, u, row, lane, s);
    uint16_t* o = u.o + u.os * row;
#pragma unroll
    for (int i = 0; i < NCH; ++i) {
      const int ch = lane + 64 * i;
      if (i + 1 < NCH || ch < nchunk)
        *reinterpret_cast<u32x4*>(o + 8 * ch) =
            qk_finish(s.x[i], *reinterpret_cast<const u32x4*>(u.bias + 8 * ch),
                      *reinterpret_cast<const u32x4*>(u.gamma + 8 * ch), s.r, s.c, s.sn,
                      s.rotate, u.scale);
    }
    if (a.v != nullptr) qk_copy_v<NCH>(a, row, lane, t, ntens);
  }
}

// ---------------------------------------------------------------- d-major layout
// One workgroup of W waves per (tile of TILE tokens, tensor), each wave R = TILE / W token
// rows of it, their loads in flight while the vectors and tables fill the LDS. A 512-column slice
// of the results is staged as rows, and each wave then writes CW columns of it: the LDS transpose read
// (ds_read_b64_tr_b16: lane i of a 16-lane group gets four tokens of column i) gives a lane 8 or 16
// tokens of one column, which go back to the wave's own part of the stage and out of it in the
// order of the output, so that neighbouring lanes store neighbouring 16 bytes. The two stage
// buffers need one barrier per slice.
// Bound by the arithmetic (about 15 VALU operations per value, 24 us of the chip for 4680 tokens x
// 40 heads) and the memory in turn: the workgroups of a CU mostly load, compute and store at the
// same time. W = 8 lets two workgroups of any row length share a CU; a workgroup alone on its CU is
// bound by the rate at which a wave issues, and takes W = 16 (launch_nch). No instance may spill
// (128 registers: two rows of 10 chunks take 122), and forming the writer's addresses anew for
// each slice instead of keeping them cost 4-10 % (4680 x 40 72 to 76 us).
template <int NCH, int W, int TILE>
__global__ void __launch_bounds__(W * 64, 4)
qk_norm_rope_dmajor_kernel(const QkNormRopeArgs a) {
  constexpr int R = TILE / W;             // token rows per wave
  constexpr int PPC = TILE / 8;           // 16-byte pieces of a column
  constexpr int CW = 512 / W;             // columns of a slice that one wave writes
  constexpr int NP = CW * PPC / 64;       // pieces per lane and slice
  constexpr int CG = CW / 16;             // 16-column groups of a wave
  extern __shared__ __attribute__((aligned(16))) float smem[];
  const int C = a.C;
  const int nchunk = C / 8;
  const int ntens = a.k != nullptr ? 2 : 1;
  // item numbering: XCD x (= blockIdx % 8) takes items [x * per, (x + 1) * per)
  const int nitem = (a.L + TILE - 1) / TILE * ntens;
  const int per = (nitem + 7) / 8;
  const int item = (int)(blockIdx.x & 7) * per + (int)(blockIdx.x >> 3);
  if (item >= nitem) return;  // whole workgroup, before any barrier
  const int t = item % ntens;
  const int t0 = item / ntens * TILE;
  const int nvalid = min(TILE, a.L - t0);

  // LDS: [tables][bias, gamma of the tensor][2 stage buffers of TILE rows]
  float* tab = smem;
  uint16_t* vec = reinterpret_cast<uint16_t*>(smem + qk_table_floats(a.ntab));
  uint16_t* stage = vec + 2 * C;
  constexpr int SB = TILE * QT_PITCH;     // one stage buffer

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  QkTensor u = qk_tensor(a, vec, t);
  u.bias = vec;
  u.gamma = vec + C;

  // vectors, then the rows, then the tables: the rows' latency covers the others'
  constexpr int NV = (NCH + W - 1) / W;  // 16-byte chunks of a vector per thread
  const uint16_t* src[2] = {t ? a.bk : a.bq, t ? a.wk : a.wq};
  u32x4 xv[2][NV];
#pragma unroll
  for (int v = 0; v < 2; ++v)
#pragma unroll
    for (int i = 0; i < NV; ++i) {
      const int ch = threadIdx.x + W * 64 * i;
      xv[v][i] = u32x4{0u, 0u, 0u, 0u};
      if (src[v] != nullptr && ch < nchunk)
        xv[v][i] = *reinterpret_cast<const u32x4*>(src[v] + 8 * ch);
    }
  QkOne<NCH> s[R];
#pragma unroll
  for (int k = 0; k < R; ++k)
    if (wave + W * k < nvalid)
      qk_one_load<NCH, true>(a, u, t0 + wave + W * k, lane, s[k]);
#pragma unroll
  for (int v = 0; v < 2; ++v)
#pragma unroll
    for (int i = 0; i < NV; ++i) {
      const int ch = threadIdx.x + W * 64 * i;
      if (ch < nchunk) *reinterpret_cast<u32x4*>(vec + v * C + 8 * ch) = xv[v][i];
    }
  const int nt2 = a.ntab / 2;  // cos/sin values come in pairs: 8-byte loads
#pragma unroll 4
  for (int i = threadIdx.x; i < nt2; i += W * 64)
    reinterpret_cast<u32x2*>(tab)[i] = reinterpret_cast<const u32x2*>(a.rope)[i];
  __syncthreads();
#pragma unroll
  for (int k = 0; k < R; ++k)
    if (wave + W * k < nvalid)
      qk_one_norm<NCH>(a, tab, u, t0 + wave + W * k, lane, s[k]);

  // the writing: per slice the wave's CW columns, as 16-byte pieces (8 tokens of a column)
  // numbered column by column, PPC to a column. A lane's transpose reads give it NP pieces of
  // column rcol; piece id goes to chunk ((id / 4) % TILE, id % 4 + 4 (id / (4 TILE))) of the
  // wave's part of the stage and is stored from there by lane id % 64.
  const int i16 = lane & 15, g = lane >> 4;
  const int rcol = 16 * (g % CG) + i16;
  const int rtok = 8 * NP * (g / CG);
  auto lds_at = [](const uint16_t* p) {
    return (int)(uint32_t)(uintptr_t)(__attribute__((address_space(3))) const uint16_t*)p;
  };
  const int rd = lds_at(stage) + 2 * ((rtok + (i16 >> 2)) * QT_PITCH + CW * wave +
                                      16 * (g % CG) + 4 * (i16 & 3));
  auto piece_at = [&](int id) {  // element offset in a stage buffer
    return (id / 4 % TILE) * QT_PITCH + CW * wave + 8 * (id % 4 + 4 * (id / (4 * TILE)));
  };
  uint16_t* const out = t ? a.ko : a.qo;
  const int64_t os = t ? a.kos : a.qos;
  const int ntok = nvalid - 8 * (lane % PPC);  // tokens of this lane's pieces that exist (>= 8: all)
  const int64_t lane_out = (int64_t)(lane / PPC) * os + 8 * (lane % PPC);
  const bool vec_ok = (t ? a.ko_vec : a.qo_vec) != 0;
#pragma unroll
  for (int i = 0; i < NCH; ++i) {
    uint16_t* sb = stage + (i & 1) * SB;
    const int ch = lane + 64 * i;
    if (i + 1 < NCH || ch < nchunk) {
      const u32x4* const bp = reinterpret_cast<const u32x4*>(u.bias + 8 * ch);
      const u32x4* const gp = reinterpret_cast<const u32x4*>(u.gamma + 8 * ch);
      u32x4 bv = *bp, gv = *gp;
#pragma unroll
      for (int k = 0; k < R; ++k) {
        // two rows of more than 8 chunks leave no registers to keep the vectors for the second:
        // read again (36 to 44 bytes of scratch per lane else)
        if (NCH > 8 && k > 0) {
          asm volatile("" ::: "memory");
          bv = *bp;
          gv = *gp;
        }
        if (wave + W * k < nvalid)
          *reinterpret_cast<u32x4*>(sb + (wave + W * k) * QT_PITCH + 8 * lane) =
              qk_finish(s[k].x[i], bv, gv, s[k].r, s[k].c, s[k].sn, s[k].rotate, u.scale);
      }
    }
    __syncthreads();
    const int col0 = 512 * i + CW * wave;  // column e = head * D + d starts at e * d_stride
    if (col0 >= C) continue;
    u32x2 x[2 * NP];
#pragma unroll
    for (int j = 0; j < 2 * NP; ++j)
      x[j] = qk_read_tr16(rd + 2 * ((i & 1) * SB + 4 * j * QT_PITCH));
    wave_lds_fence();
#pragma unroll
    for (int j = 0; j < NP; ++j)
      *reinterpret_cast<u32x4*>(sb + piece_at(rcol * PPC + rtok / 8 + j)) =
          u32x4{x[2 * j][0], x[2 * j][1], x[2 * j + 1][0], x[2 * j + 1][1]};
    wave_lds_fence();
    if (vec_ok) {
#pragma unroll
      for (int j = 0; j < NP; ++j) {
        const int cj = col0 + 64 / PPC * j;  // (wave-uniform) column of lane 0
        const u32x4 v = *reinterpret_cast<const u32x4*>(sb + piece_at(64 * j + lane));
        if (cj + lane / PPC >= C) continue;
        uint16_t* dst = out + cj * os + t0 + lane_out;
        if (ntok >= 8) {
          *reinterpret_cast<u32x4*>(dst) = v;
        } else {
#pragma unroll
          for (int e = 0; e < 7; ++e)
            if (e < ntok) dst[e] = (uint16_t)(v[e >> 1] >> (16 * (e & 1)));
        }
      }
    } else {
      // outputs that 16-byte stores cannot reach: consecutive lanes take consecutive tokens of a column
      for (int e = lane; e < CW * TILE; e += 64) {
        const int col = e / TILE, tok = e % TILE;
        const uint16_t v = sb[piece_at(col * PPC + tok / 8) + tok % 8];
        if (col0 + col < C && tok < nvalid) out[(int64_t)(col0 + col) * os + t0 + tok] = v;
      }
    }
  }
  if (a.v != nullptr) {
#pragma unroll
    for (int k = 0; k < R; ++k)
      if (wave + W * k < nvalid) {
        if (ntens == 2) qk_copy_v_part<NCH, 2>(a, t0 + wave + W * k, lane, t);
        else qk_copy_v_part<NCH, 1>(a, t0 + wave + W * k, lane, 0);
      }
  }
}

template <int NCH, int W, int TILE>
static hipError_t launch_dmajor(const QkNormRopeArgs& a, hipStream_t stream) {
  static hipError_t attr = hipFuncSetAttribute(
      (const void*)qk_norm_rope_dmajor_kernel<NCH, W, TILE>,
      hipFuncAttributeMaxDynamicSharedMemorySize,
      (int)(qt_lds_bytes(QK_MAX_TABLE, 64 * 8 * NCH, TILE) < LDS_LIMIT
                ? qt_lds_bytes(QK_MAX_TABLE, 64 * 8 * NCH, TILE)
                : LDS_LIMIT));
  if (attr != hipSuccess) return attr;
  const int items = (a.L + TILE - 1) / TILE * (a.k != nullptr ? 2 : 1);
  hipLaunchKernelGGL((qk_norm_rope_dmajor_kernel<NCH, W, TILE>), dim3(8 * ((items + 7) / 8)),
                     dim3(W * 64), qt_lds_bytes(a.ntab, a.C, TILE), stream, a);
  return hipGetLastError();
}

template <int NCH>
static hipError_t launch_nch(const QkNormRopeArgs& a, int num_cus, hipStream_t stream) {
  if (a.layout == QK_LAYOUT_DMAJOR) {
    if constexpr (NCH > QT_MAX_NCH) {
      return hipErrorInvalidValue;  // rejected by the host check
    } else {
      // 16 waves of one row or 8 of two. Kernel times, us, W = 8 and W = 16, inputs from HBM:
      // - one workgroup per CU (items or LDS leave no second): 16, a lone one is bound by the rate
      //   at which its waves issue. 1560 tokens x 40 heads, 196 items, 25.9, 23.5.
      // - 3 to 5 chunks: 16, whose 64 registers let two share a CU as well. 3600 x 20 heads 24.4,
      //   23.1; 9360 64.4, 56.5; 4680 x 12 26.9, 25.6 (2 chunks, 4680 x 5: 15.6, 16.3).
      // - above, up to two items per CU: 8, two workgroups side by side where 16 take two rounds.
      //   2560 x 40, 320 items, 34.6, 39.1; 3600, 450, 41.5, 45.8; 3600 x 24 26.8, 32.3.
      // - more items: 8 up to 8 chunks (10800 x 24 85, 92; x 32 108, 110), 16 for longer rows
      //   (4680 x 40 72.2, 64.6; 9360 119, 110; 10800 143, 128).
      // - of these, rows of more than 6 chunks: 16 waves of two rows, tiles of 32 tokens, once a
      //   round of them (39 us at 40 heads) costs less than the 16-token rounds (24 us) it replaces.
      //   A line of the output gets 64 bytes from one workgroup instead of 32 each from two that
      //   drift apart over the rounds. us for 32, 16 and (the form before all of these, one
      //   workgroup of 16 waves per 16 tokens of both tensors): 7200 x 40 80, 99 (83); 8160 88, 105
      //   (97); 10800 119, 128 (122); 14400 157, 178 (164); 7200 x 32 63, 74 (66); not 9360 x 40
      //   119, 116 (116).
      const int items = (a.L + QT_TILE - 1) / QT_TILE * (a.k != nullptr ? 2 : 1);
      const bool pair = 2 * qt_lds_bytes(a.ntab, a.C, QT_TILE) <= LDS_LIMIT;
      if constexpr (NCH > 6) {
        const int items32 = (a.L + QT_LONG - 1) / QT_LONG * (a.k != nullptr ? 2 : 1);
        const int rounds = (items + num_cus - 1) / num_cus;
        const int rounds32 = (items32 + num_cus - 1) / num_cus;
        if (items > 2 * num_cus && 3 * rounds > 5 * rounds32)
          return launch_dmajor<NCH, 16, QT_LONG>(a, stream);
      }
      if constexpr (NCH < 3 || NCH > 5) {
        if (items > num_cus && pair && (NCH < 9 || items <= 2 * num_cus))
          return launch_dmajor<NCH, 8, QT_TILE>(a, stream);
      }
      return launch_dmajor<NCH, 16, QT_TILE>(a, stream);
    }
  }
  static hipError_t attr = hipFuncSetAttribute((const void*)qk_norm_rope_kernel<NCH>,
                                               hipFuncAttributeMaxDynamicSharedMemorySize,
                                               (int)qk_lds_bytes(QK_MAX_TABLE, 64 * 8 * NCH));
  if (attr != hipSuccess) return attr;
  // at most QK_MAX_BLOCKS workgroups, each wave looping over rows so that the LDS fill is
  // amortised
  const int rows_per_block = a.k != nullptr ? QK_WAVES / 2 : QK_WAVES;
  int blocks = (a.L + rows_per_block - 1) / rows_per_block;
  if (blocks > QK_MAX_BLOCKS) blocks = QK_MAX_BLOCKS;
  if (blocks < 1) blocks = 1;
  hipLaunchKernelGGL(qk_norm_rope_kernel<NCH>, dim3(blocks), dim3(QK_WAVES * 64),
                     qk_lds_bytes(a.ntab, a.C), stream, a);
  return hipGetLastError();
}

hipError_t launch_qk_norm_rope(const QkNormRopeArgs& a, int num_cus, hipStream_t stream) {
  const int nch = (a.C / 8 + 63) / 64;
  switch (nch) {
    case 1: return launch_nch<1>(a, num_cus, stream);
    case 2: return launch_nch<2>(a, num_cus, stream);
    case 3: return launch_nch<3>(a, num_cus, stream);
    case 4: return launch_nch<4>(a, num_cus, stream);
    case 5: return launch_nch<5>(a, num_cus, stream);
    case 6: return launch_nch<6>(a, num_cus, stream);
    case 7: return launch_nch<7>(a, num_cus, stream);
    case 8: return launch_nch<8>(a, num_cus, stream);
    case 9: return launch_nch<9>(a, num_cus, stream);
    case 10: return launch_nch<10>(a, num_cus, stream);
    case 11: return launch_nch<11>(a, num_cus, stream);
    case 12: return launch_nch<12>(a, num_cus, stream);
    case 13: return launch_nch<13>(a, num_cus, stream);
    case 14: return launch_nch<14>(a, num_cus, stream);
    case 15: return launch_nch<15>(a, num_cus, stream);
    case 16: return launch_nch<16>(a, num_cus, stream);
    default: return hipErrorInvalidValue;
  }
}

}  // namespace lbw
