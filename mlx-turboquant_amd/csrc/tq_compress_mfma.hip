// MFMA compress for what compress_fast_kernel (fp16, head_dim 128, no sketch)
// does not take: fp16, bf16 and float32 vectors of head_dim 64, 96, 128 and
// 256 at 1-4 bits (integer, or fractional with a split that is a multiple of
// 32), and the QJL sketch of at most 128 projections at head_dim 64 / 96 / 128
// (replaces TurboQuantKVCache._quantize_kv / _quantize_kv_fractional,
// mlx_turboquant/cache.py:232-274, and qjl_quantize of the residual,
// qjl.py:47-67, cache.py:396-427). Other shapes take compress_kernel.
//
// Three float32-class d x d products per vector (rotation; with a sketch the
// reconstruction c R and the projection r S^T) were the bound on the VALU. They
// run on MFMA here with split operands and float32 accumulation:
//  - rotation, fp16 x: x is exact, 256 R = fp16 high part + remainder (2 passes);
//  - rotation, bf16 x: x is exact, R = three bf16 parts (3 passes);
//  - rotation, float32 x: x = three bf16 parts exactly, the six products of
//    order up to 2^-16;
//  - reconstruction: 256 c and 256 R as fp16 high part + remainder (3 passes);
//  - projection: the residual times a power of two, and S, likewise (3 passes).
// (operands in two fp16 parts hold 22 to 24 bits, in three bf16 parts 24). Codes
// differ from float64's only within float32 rounding of a boundary; residual
// norms carry 2e-7 at most.
//
// Work split as in compress_fast_kernel: a persistent workgroup walks tiles of
// 64 vectors, the tile raw in LDS, the next one in flight; wave w owns rotated
// dims [32w, 32w + 32) (D / 32 waves) and keeps its rows of R as MFMA A
// operands in registers for the whole launch (with a sketch its columns of R
// too; S stays in LDS). Row m of output block n2 is dim 32w + 8(m >> 2) + 4 n2 +
// (m & 3), so lane (vector m, g) holds 8 consecutive dims and packs their codes
// in registers. Norms: one thread per (vector, 32-dim block), float64 in the
// library's order. Quantizer: a cell table with at most one boundary per cell.
//
// Measured against compress_kernel (head_dim 128): 64,512 bf16 vectors to 4 / 2
// bits 157 -> 20 us (0.9 TB/s read and written: four tiles per workgroup at
// most, half the time is the set-up of the R operands and the cell table); 65,536
// float32 vectors to 3 bits with 128 projections 359 -> 65 us (one 150 KB
// workgroup per CU: a chain of four phases with barriers on four waves). Spans of
// one token (a decode drain) pay the set-up alone and still win: 8 rows of
// head_dim 64 / 96 / 256 in bf16 11.0 / 8.1 / 20.0 us, from 50.6 / 50.0 / 98.7; with
// 32 projections at head_dim 64 15.3, from 94.

#include <math.h>

#include <algorithm>
#include <atomic>
#include <type_traits>

#include "tq_codec.h"

namespace tq {
namespace {

typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf8 __attribute__((ext_vector_type(8)));
typedef float f4 __attribute__((ext_vector_type(4)));
typedef uint32_t u4 __attribute__((ext_vector_type(4)));
typedef uint32_t u2 __attribute__((ext_vector_type(2)));

constexpr int CT = 64;        // vectors per tile
constexpr float SC = 256.f;   // scale of R and c before an fp16 split
constexpr int TROW = 64;      // bytes per pair-table entry (8 replicas: the sketch's LDS fits one workgroup)

__device__ inline f4 mfma_h(u4 a, u4 b, f4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(half8, a), __builtin_bit_cast(half8, b), c, 0, 0, 0);
}
__device__ inline f4 mfma_b(u4 a, u4 b, f4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf8, a), __builtin_bit_cast(bf8, b), c, 0, 0, 0);
}

// fp16 high part and remainder of 8 values
__device__ inline void split_h(const float (&v)[8], u4& hi, u4& lo) {
  half8 h, l;
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    h[e] = (_Float16)v[e];
    l[e] = (_Float16)(v[e] - (float)h[e]);
  }
  hi = __builtin_bit_cast(u4, h);
  lo = __builtin_bit_cast(u4, l);
}

// v = p[0] + p[1] + p[2], three bf16 parts of 8 values each (truncated: exact)
__device__ inline void split_b(const float (&v)[8], u4 (&p)[3]) {
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    uint32_t a = __float_as_uint(v[2 * j]), b = __float_as_uint(v[2 * j + 1]);
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      p[k][j] = __builtin_amdgcn_perm(b, a, 0x07060302u);  // the high halves
      if (k < 2) {
        a = __float_as_uint(__uint_as_float(a) - __uint_as_float(a & 0xFFFF0000u));
        b = __float_as_uint(__uint_as_float(b) - __uint_as_float(b & 0xFFFF0000u));
      }
    }
  }
}

template <int D, int XT, bool QJ>
struct Lay {
  static constexpr int ES = XT == TQ_F32 ? 4 : 2;
  static constexpr int NT = 2 * D;              // threads
  static constexpr int NB = D / 32;             // waves, 32-dim blocks
  static constexpr int XS = D * ES + 16;        // x tile row
  static constexpr int NBUF = QJ ? 1 : 2;       // x tiles in LDS
  static constexpr int CW = D == 256 ? 128 : 64;  // quantizer cells per unit
  static constexpr int CLO = -CW / 2 - 8, NCELL = 2 * CW + 16;
  static constexpr int x0 = 0;
  static constexpr int nrm = NBUF * CT * XS;    // [64] norms
  static constexpr int scl = nrm + CT * 4;      // [64] scales of the rotated coordinates
  static constexpr int qt = scl + CT * 4;       // [2 codebooks][NCELL] {boundary, base}
  static constexpr int bnd = qt + 2 * NCELL * 8;  // [2][16] boundaries
  static constexpr int flag = bnd + 128;
  static constexpr int dsum = flag + 16;        // [64][NB] float64 block sums (head_dim 96), residual sums (sketch)
  static constexpr int end0 = dsum + (QJ || NB == 3 ? CT * NB * 8 : 0);
  // sketch: codes, residual planes, S planes (128 projections), pair tables, codebook words
  static constexpr int CS = D / 8 + 1;          // dwords per vector of the codes
  static constexpr int RS = 4 * D + 16;         // bytes per vector / projection: high part row, remainder row
  static constexpr int cds = (end0 + 15) / 16 * 16;
  static constexpr int rpl = (cds + CT * CS * 4 + 15) / 16 * 16;
  static constexpr int cwd = rpl + CT * RS;
  static constexpr int spl = cwd + 128;
  static constexpr int end = QJ ? spl : cds;    // S planes and pair tables follow, sized per launch
};

extern "C" __device__ float tq_fmul_legacy(float, float) __asm("llvm.amdgcn.fmul.legacy");

template <int D, int XT, bool QJ>
__global__ __launch_bounds__(2 * D) void compress_mfma_kernel(CompressArgs a, int tiles_per_row, int total) {
  using L = Lay<D, XT, QJ>;
  constexpr int KS = D / 32, NT = L::NT, NB = L::NB, NPL = XT == TQ_F16 ? 2 : 3;
  extern __shared__ __align__(16) uint8_t smem[];
  const int tid = threadIdx.x, lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int m = lane & 15, g = lane >> 4;
  const bool whi = 32 * w < a.split;
  const int nbh = (1 << a.bits_hi) - 1, nbl = (1 << a.bits_lo) - 1;

  // ---- quantizer cells c = round(CW y + CW / 2) of both codebooks; the flag
  // records a cell holding two boundaries (then every code is counted)
  uint32_t* flag = reinterpret_cast<uint32_t*>(smem + L::flag);
  if (tid == 0) *flag = 0u;
  __syncthreads();
  if (tid < 32) {
    const int cb = tid >> 4, k = tid & 15;
    reinterpret_cast<float*>(smem + L::bnd)[tid] = k < (cb ? nbl : nbh) ? (cb ? a.bnd_lo : a.bnd_hi)[k] : 0.f;
  }
  for (int i = tid; i < 2 * L::NCELL; i += NT) {
    const int cb = i / L::NCELL, ci = i % L::NCELL, c = L::CLO + ci;
    const float* bp = cb ? a.bnd_lo : a.bnd_hi;
    const int nb = cb ? nbl : nbh;
    const float eps = 0x1p-20f;  // > the rounding of the cell index near a cell edge, in y units
    const float lo = ci == 0 ? -INFINITY : ((float)c - (L::CW / 2 + 0.5f)) * (1.f / L::CW) - eps;
    const float hi = ci == L::NCELL - 1 ? INFINITY : ((float)c - (L::CW / 2 - 0.5f)) * (1.f / L::CW) + eps;
    uint32_t base = 0, amb = 0;
    float bnd = INFINITY;
    for (int k = 0; k < nb; ++k) {
      const float b = bp[k];
      if (b < lo) ++base;
      else if (b <= hi) { ++amb; bnd = b; }
    }
    float2* q = reinterpret_cast<float2*>(smem + L::qt) + i;
    *q = make_float2(bnd, __uint_as_float(base));
    if (amb > 1) atomicOr(flag, 1u);
  }

  // ---- A operands: rows of R (rotation) and with a sketch columns of R
  u4 ra[2][NPL][KS];
  u4 rt[2][2][QJ ? KS : 1];
#pragma unroll
  for (int n2 = 0; n2 < 2; ++n2) {
    const int j = 32 * w + 8 * (m >> 2) + 4 * n2 + (m & 3);
#pragma unroll
    for (int kb = 0; kb < KS; ++kb) {
      const float* src = a.rot + j * D + 32 * kb + 8 * g;
      float f[8];
#pragma unroll
      for (int e = 0; e < 8; ++e) f[e] = XT == TQ_F16 ? SC * src[e] : src[e];
      if constexpr (XT == TQ_F16) {
        split_h(f, ra[n2][0][kb], ra[n2][1][kb]);
      } else {
        u4 p[3];
        split_b(f, p);
        ra[n2][0][kb] = p[0];
        ra[n2][1][kb] = p[1];
        ra[n2][NPL - 1][kb] = p[2];
      }
      if constexpr (QJ) {
#pragma unroll
        for (int e = 0; e < 8; ++e) f[e] = SC * a.rot[(32 * kb + 8 * g + e) * D + j];
        split_h(f, rt[n2][0][kb], rt[n2][1][kb]);
      }
    }
  }
  const int tab = L::spl + a.qjl_m * L::RS;            // pair tables of the centroids
  const int tab_lo = tab + (1 << (2 * a.bits_hi)) * TROW;
  if constexpr (QJ) {
    uint32_t* cw = reinterpret_cast<uint32_t*>(smem + L::cwd);
    if (tid < 32) {
      const int cb = tid >> 4;
      const float x = SC * (cb ? a.cen_lo : a.cen_hi)[min(tid & 15, cb ? nbl : nbh)];
      const _Float16 h = (_Float16)x, l = (_Float16)(x - (float)h);
      cw[tid] = (uint32_t)__builtin_bit_cast(uint16_t, h) | (uint32_t)__builtin_bit_cast(uint16_t, l) << 16;
    }
    for (int i = tid; i < a.qjl_m * (D / 8); i += NT) {  // S: 8 dims per step
      const int p = i / (D / 8), c8 = i % (D / 8);
      float f[8];
#pragma unroll
      for (int e = 0; e < 8; ++e) f[e] = a.proj[p * D + 8 * c8 + e];
      u4 hi, lo;
      split_h(f, hi, lo);
      *reinterpret_cast<u4*>(smem + L::spl + p * L::RS + 16 * c8) = hi;
      *reinterpret_cast<u4*>(smem + L::spl + p * L::RS + 2 * D + 16 * c8) = lo;
    }
    __syncthreads();
#pragma unroll
    for (int cb = 0; cb < 2; ++cb) {
      const int bits = cb ? a.bits_lo : a.bits_hi, msk = (1 << bits) - 1;
      if (cb && a.split == D) break;
      for (int s = tid; s < (1 << (2 * bits)) * (TROW / 16); s += NT) {
        const int e = s / (TROW / 16);
        const uint32_t x = cw[16 * cb + (e & msk)], y = cw[16 * cb + (e >> bits)];
        const uint32_t hi = __builtin_amdgcn_perm(y, x, 0x05040100u), lo = __builtin_amdgcn_perm(y, x, 0x07060302u);
        *reinterpret_cast<u4*>(smem + (cb ? tab_lo : tab) + 16 * s) = u4{hi, lo, hi, lo};
      }
    }
  }
  __syncthreads();
  const bool table = *flag == 0u;
  constexpr float MAGIC = 12582912.f;  // 1.5 2^23
  const uint32_t qadj = L::qt + (whi ? 0u : L::NCELL * 8u) - 8u * (0x4B400000u + (uint32_t)L::CLO);  // wraps, as the index does

  struct Tile {
    int id, row, nv, src0, dst0;
  };
  auto make_tile = [&](int id) {  // next non-empty tile at or after `id`
    Tile t{id, 0, 0, 0, 0};
    for (; t.id < total; t.id += gridDim.x) {
      t.row = t.id / tiles_per_row;
      const int t0 = (t.id - t.row * tiles_per_row) * CT;
      const int b = t.row / a.span.heads;
      t.nv = min(CT, (a.span.n_tok_b ? a.span.n_tok_b[b] : a.span.n_tok) - t0);
      if (t.nv > 0) {
        t.src0 = (a.span.src_tok0_b ? a.span.src_tok0_b[b] : 0) + t0;
        t.dst0 = (a.span.dst_tok0_b ? a.span.dst_tok0_b[b] : 0) + t0;
        break;
      }
    }
    return t;
  };
  // x tile: 16-byte chunks, NC per thread; vectors past the tile's end re-read
  // its last one (results stored to its place again or not at all)
  constexpr int NC = 2 * L::ES, CPV = D * L::ES / 16;  // chunks per thread, per vector
  auto load_x = [&](u4 (&xr)[NC], const Tile& t) {
    const uint8_t* base = static_cast<const uint8_t*>(a.x) + ((int64_t)t.row * a.x_hs + (int64_t)t.src0 * D) * L::ES;
#pragma unroll
    for (int i = 0; i < NC; ++i) {
      const int c = tid + NT * i;
      xr[i] = *reinterpret_cast<const u4*>(base + min(c / CPV, t.nv - 1) * (D * L::ES) + (c % CPV) * 16);
    }
  };
  auto write_x = [&](const u4 (&xr)[NC], int xo) {
#pragma unroll
    for (int i = 0; i < NC; ++i) {
      const int c = tid + NT * i;
      *reinterpret_cast<u4*>(smem + xo + (c / CPV) * L::XS + (c % CPV) * 16) = xr[i];
    }
  };
  // elements [8 c8, 8 c8 + 8) of vector v of the tile as float32
  auto x8 = [&](int xo, int v, int c8, float (&f)[8]) {
    const uint8_t* p = smem + xo + v * L::XS + c8 * (8 * L::ES);
    const u4 u = *reinterpret_cast<const u4*>(p);
    if constexpr (XT == TQ_F32) {
      const u4 t = *reinterpret_cast<const u4*>(p + 16);
#pragma unroll
      for (int e = 0; e < 8; ++e) f[e] = __uint_as_float(e < 4 ? u[e] : t[e - 4]);
    } else {
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const uint32_t hb = (u[e >> 1] >> (16 * (e & 1))) & 0xFFFFu;
        f[e] = XT == TQ_BF16 ? __uint_as_float(hb << 16) : (float)__builtin_bit_cast(_Float16, (uint16_t)hb);
      }
    }
  };
  float* nrm = reinterpret_cast<float*>(smem + L::nrm);
  float* scl = reinterpret_cast<float*>(smem + L::scl);
  double* dsum = reinterpret_cast<double*>(smem + L::dsum);
  // norm of vector v: scale 1 / max(n, 1e-10) of its coordinates; 0 when the
  // norm overflows float32 (x / inf = 0), -1 marks non-finite inputs (codes 0)
  auto put_norm = [&](int v, double s, const Tile& t) {
    const float n = (float)sqrt(s);
    if (v < t.nv) a.dst.norms[(int64_t)t.row * a.dst.norm_head_stride + t.dst0 + v] = n;
    nrm[v] = n;
    scl[v] = !__builtin_isfinite(s) ? -1.f : 1.f / ((XT == TQ_F16 ? SC : 1.f) * fmaxf(n, 1e-10f));
  };
  auto norms = [&](int xo, const Tile& t) {
    const int v = tid / NB, p = tid % NB;
    double s = 0.0;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      float f[8];
      x8(xo, v, 4 * p + i, f);
#pragma unroll
      for (int e = 0; e < 8; ++e) s = fma((double)f[e], (double)f[e], s);
    }
    if constexpr (NB == 3) {
      dsum[v * 3 + p] = s;
      __syncthreads();
      if (tid < CT) put_norm(tid, (dsum[tid * 3] + dsum[tid * 3 + 1]) + dsum[tid * 3 + 2], t);
    } else {
#pragma unroll
      for (int k = 1; k < NB; k *= 2) s += __shfl_xor(s, k);
      if (p == 0) put_norm(v, s, t);
    }
  };

  // the wave's codes: B dwords at byte 4 B wl of a vector's row, lane g
  // holding bits [8 B g, 8 B g + 8 B) of them
  const int B = whi ? a.bits_hi : a.bits_lo;
  uint8_t* const codes = whi ? a.dst.codes_hi : a.dst.codes_lo;
  const int64_t head_stride = whi ? a.dst.hi_head_stride : a.dst.lo_head_stride;
  const int row_bytes = whi ? a.row_hi : a.row_lo;
  const int wl = whi ? w : w - a.split / 32;
  const float* bnd_l = reinterpret_cast<const float*>(smem + L::bnd) + (whi ? 0 : 16);
  const int nbnd = (1 << B) - 1;
  // dword k = min(g, B - 1) holds bits of lanes la = 4k / B and la + 1 (8 B bits
  // each; a lane past the last dword repeats it); 1-bit codes: all four lanes
  const int dk = min(g, B - 1), la = (4 * dk) / B, off = 32 * dk - 8 * B * la, sh2 = 8 * B - off;
  auto rotate_quantize = [&](auto table_tag, int xo, const Tile& t, int s4) {
    constexpr bool TABLE = decltype(table_tag)::value;
    const int v = 16 * s4 + m;
    f4 z[2], zl[2];
#pragma unroll
    for (int n2 = 0; n2 < 2; ++n2) z[n2] = zl[n2] = f4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int kb = 0; kb < KS; ++kb) {
      if constexpr (XT == TQ_F32) {
        float f[8];
        u4 x[3];
        x8(xo, v, 4 * kb + g, f);
        split_b(f, x);
#pragma unroll
        for (int n2 = 0; n2 < 2; ++n2) {
          z[n2] = mfma_b(ra[n2][0][kb], x[0], z[n2]);
          zl[n2] = mfma_b(ra[n2][1][kb], x[0], zl[n2]);
          zl[n2] = mfma_b(ra[n2][0][kb], x[1], zl[n2]);
          zl[n2] = mfma_b(ra[n2][2][kb], x[0], zl[n2]);
          zl[n2] = mfma_b(ra[n2][1][kb], x[1], zl[n2]);
          zl[n2] = mfma_b(ra[n2][0][kb], x[2], zl[n2]);
        }
      } else {
        const u4 x = *reinterpret_cast<const u4*>(smem + xo + v * L::XS + 64 * kb + 16 * g);
#pragma unroll
        for (int n2 = 0; n2 < 2; ++n2) {
          if constexpr (XT == TQ_F16) {
            z[n2] = mfma_h(ra[n2][0][kb], x, z[n2]);
            zl[n2] = mfma_h(ra[n2][1][kb], x, zl[n2]);
          } else {
            z[n2] = mfma_b(ra[n2][0][kb], x, z[n2]);
            zl[n2] = mfma_b(ra[n2][1][kb], x, zl[n2]);
            zl[n2] = mfma_b(ra[n2][NPL - 1][kb], x, zl[n2]);
          }
        }
      }
    }
    const float sc = scl[v];
    uint32_t V = 0;  // codes of dims 32w + 8g + k at bits B k
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      const float y = tq_fmul_legacy(z[k >> 2][k & 3] + zl[k >> 2][k & 3], sc);  // 0 where sc = 0
      uint32_t c;
      if constexpr (TABLE) {
        // |y| <= 1 up to rounding; z may overflow beside a norm at float32's end
        // and is anything for non-finite inputs (their codes are dropped below):
        // the cells end at 1 + 7 / CW
        const float yc = __builtin_amdgcn_fmed3f(y, -1.05f, 1.05f);
        const uint32_t i = __float_as_uint(fmaf(yc, (float)L::CW, L::CW / 2 + MAGIC));
        const float2 q = *reinterpret_cast<const float2*>(smem + (qadj + 8u * i));
        c = __float_as_uint(q.y) + (y > q.x ? 1u : 0u);
      } else {
        c = 0;
        for (int b = 0; b < nbnd; ++b) c += y > bnd_l[b] ? 1u : 0u;
      }
      V |= c << (B * k);
    }
    if (sc < 0.f) V = 0u;  // non-finite inputs: every coordinate is NaN -> code 0
    if constexpr (QJ) reinterpret_cast<uint32_t*>(smem + L::cds)[v * L::CS + 4 * w + g] = V;
    uint32_t o;  // the wave's dword dk of this vector
    if (B == 1) {
      const uint32_t x = __shfl_xor(V, 16);
      o = g & 1 ? x | V << 8 : V | x << 8;
      const uint32_t y = __shfl_xor(o, 32);
      o = g & 2 ? y | o << 16 : o | y << 16;
    } else {
      const uint32_t Va = __shfl(V, m + 16 * la);
      const uint32_t Vb = __shfl(V, m + 16 * min(la + 1, 3));
      o = (Va >> off) | (sh2 < 32 ? Vb << sh2 : 0u);
    }
    reinterpret_cast<uint32_t*>(codes + (int64_t)t.row * head_stride + (int64_t)(t.dst0 + min(v, t.nv - 1)) * row_bytes +
                                4 * B * wl)[dk] = o;
  };

  // the residual r = x - n (c R) of sub-tile s4: its float64 sum over the
  // wave's dims and its fp16 planes, times 2^10 over the norm's power of two
  auto residual = [&](int xo, int s4) {
    const int v = 16 * s4 + m;
    f4 z[2], zl[2];
#pragma unroll
    for (int n2 = 0; n2 < 2; ++n2) z[n2] = zl[n2] = f4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int s = 0; s < (QJ ? KS : 0); ++s) {
      const uint32_t V = reinterpret_cast<const uint32_t*>(smem + L::cds)[v * L::CS + 4 * s + g];
      const bool hi = 32 * s < a.split;
      const int fb = 2 * (hi ? a.bits_hi : a.bits_lo);
      const uint8_t* tb = smem + (hi ? tab : tab_lo) + 8 * (m & 7);
      u4 bh, bl;
#pragma unroll
      for (int f = 0; f < 4; ++f) {
        const u2 e = *reinterpret_cast<const u2*>(tb + __builtin_amdgcn_ubfe(V, fb * f, fb) * TROW);
        bh[f] = e[0];
        bl[f] = e[1];
      }
#pragma unroll
      for (int n2 = 0; n2 < 2; ++n2) {
        z[n2] = mfma_h(rt[n2][0][s], bh, z[n2]);
        zl[n2] = mfma_h(rt[n2][1][s], bh, zl[n2]);
        zl[n2] = mfma_h(rt[n2][0][s], bl, zl[n2]);
      }
    }
    const float n = nrm[v];
    const int ne = __builtin_isfinite(n) && n > 0.f ? __builtin_amdgcn_frexp_expf(n) : 0;
    float f[8], q[8];
    x8(xo, v, 4 * w + g, f);
    double s = 0.0;
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      const float r = fmaf(-n, (z[k >> 2][k & 3] + zl[k >> 2][k & 3]) * (1.f / (SC * SC)), f[k]);
      s = fma((double)r, (double)r, s);
      q[k] = __builtin_amdgcn_ldexpf(r, 10 - ne);
    }
    u4 hi, lo;
    split_h(q, hi, lo);
    uint8_t* rp = smem + L::rpl + v * L::RS + 64 * w + 16 * g;
    *reinterpret_cast<u4*>(rp) = hi;
    *reinterpret_cast<u4*>(rp + 2 * D) = lo;
    s += __shfl_xor(s, 16);
    s += __shfl_xor(s, 32);
    if (g == 0) dsum[v * NB + w] = s;
  };
  // signs of the 32 projections of block pb on sub-tile s4: lane (vector m, g)
  // gets projections 32 pb + 8g + k
  auto project = [&](const Tile& t, int pb, int s4) {
    const int v = 16 * s4 + m;
    f4 z[2], zl[2];
#pragma unroll
    for (int n2 = 0; n2 < 2; ++n2) z[n2] = zl[n2] = f4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int kb = 0; kb < KS; ++kb) {
      const uint8_t* rp = smem + L::rpl + v * L::RS + 64 * kb + 16 * g;
      const u4 bh = *reinterpret_cast<const u4*>(rp), bl = *reinterpret_cast<const u4*>(rp + 2 * D);
#pragma unroll
      for (int n2 = 0; n2 < 2; ++n2) {
        const uint8_t* sp = smem + L::spl + (32 * pb + 8 * (m >> 2) + 4 * n2 + (m & 3)) * L::RS + 64 * kb + 16 * g;
        const u4 ah = *reinterpret_cast<const u4*>(sp), al = *reinterpret_cast<const u4*>(sp + 2 * D);
        z[n2] = mfma_h(ah, bh, z[n2]);
        zl[n2] = mfma_h(al, bh, zl[n2]);
        zl[n2] = mfma_h(ah, bl, zl[n2]);
      }
    }
    uint32_t bits = 0;
#pragma unroll
    for (int k = 0; k < 8; ++k) bits |= (z[k >> 2][k & 3] + zl[k >> 2][k & 3] >= 0.f ? 1u : 0u) << k;
    if (v < t.nv)
      a.dst.signs[(int64_t)t.row * a.dst.sign_head_stride + (int64_t)(t.dst0 + v) * a.row_sign + 4 * pb + g] =
          (uint8_t)bits;
  };

  auto run_tiles = [&](auto table_tag) {
    Tile cur = make_tile(blockIdx.x);
    if (cur.id >= total) return;
    Tile nxt = make_tile(cur.id + gridDim.x);
    u4 xr[NC];
    {
      u4 x0[NC];
      load_x(x0, cur);
      load_x(xr, nxt.id < total ? nxt : cur);
      write_x(x0, L::x0);
    }
    int xo = L::x0;
    for (;;) {
      __syncthreads();  // x of cur in LDS; every wave is done with the previous tile
      norms(xo, cur);
      const bool more = nxt.id < total;
      const Tile far = more ? make_tile(nxt.id + gridDim.x) : nxt;
      if (!QJ && more) {
        write_x(xr, CT * L::XS - xo);
        load_x(xr, far.id < total ? far : nxt);
      }
      __syncthreads();  // norms and scales of cur
#pragma unroll
      for (int s4 = 0; s4 < 4; ++s4) rotate_quantize(table_tag, xo, cur, s4);
      if constexpr (QJ) {
        __syncthreads();  // codes of cur
#pragma unroll
        for (int s4 = 0; s4 < 4; ++s4) residual(xo, s4);
        __syncthreads();  // residual planes and sums; the x tile is free
        if (more) {
          write_x(xr, xo);
          load_x(xr, far.id < total ? far : nxt);
        }
        if (tid < CT && tid < cur.nv) {
          double s = 0.0;
#pragma unroll
          for (int k = 0; k < NB; ++k) s += dsum[tid * NB + k];
          a.dst.gamma[(int64_t)cur.row * a.dst.gamma_head_stride + cur.dst0 + tid] = (float)sqrt(s);
        }
        for (int i = w; i < a.qjl_m / 8; i += NB) project(cur, i >> 2, i & 3);
      }
      if (!more) break;
      cur = nxt;
      nxt = far;
      if (!QJ) xo = CT * L::XS - xo;
    }
  };
  if (table)
    run_tiles(std::true_type{});
  else
    run_tiles(std::false_type{});
}

template <int D, int XT, bool QJ>
int launch_cm(const CompressArgs& a, hipStream_t s) {
  int lds = Lay<D, XT, QJ>::end;
  if (QJ)
    lds += a.qjl_m * Lay<D, XT, QJ>::RS + (1 << (2 * a.bits_hi)) * TROW +
           (a.split < D ? (1 << (2 * a.bits_lo)) * TROW : 0);
  if (lds > 160 * 1024) return 0;
  int dev = 0, cus = 256;
  if (hipGetDevice(&dev) == hipSuccess &&
      hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess)
    cus = 256;
  // workgroups per CU at the last LDS size asked for (the same on every gfx950
  // device): LDS bytes << 8 | workgroups
  static std::atomic<int64_t> known{-1};
  const int64_t k = known.load(std::memory_order_relaxed);
  int occ = (int)(k & 255);
  if (k < 0 || k >> 8 != lds) {
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&occ, compress_mfma_kernel<D, XT, QJ>, 2 * D, lds) != hipSuccess)
      occ = 1;
    known.store((int64_t)lds << 8 | std::min(occ, 255), std::memory_order_relaxed);
  }
  const int tpr = (a.span.n_tok + CT - 1) / CT;
  const int64_t total = (int64_t)tpr * a.span.rows;
  if (total <= 0 || total >= ((int64_t)1 << 30)) return 0;  // tile ids + 2 grids stay within int
  const int grid = (int)std::min<int64_t>(total, (int64_t)cus * std::max(occ, 1));
  hipLaunchKernelGGL((compress_mfma_kernel<D, XT, QJ>), dim3(grid), dim3(2 * D), lds, s, a, tpr, (int)total);
  return 1;
}

template <int D>
int launch_d(const CompressArgs& a, hipStream_t s) {
  if constexpr (D != 256)
    if (a.proj) {
      if (a.qjl_m > 128) return 0;
      switch (a.x_dtype) {
        case TQ_F16: return launch_cm<D, TQ_F16, true>(a, s);
        case TQ_BF16: return launch_cm<D, TQ_BF16, true>(a, s);
        default: return launch_cm<D, TQ_F32, true>(a, s);
      }
    }
  if (a.proj) return 0;
  switch (a.x_dtype) {
    case TQ_F16: return launch_cm<D, TQ_F16, false>(a, s);
    case TQ_BF16: return launch_cm<D, TQ_BF16, false>(a, s);
    default: return launch_cm<D, TQ_F32, false>(a, s);
  }
}

}  // namespace

int launch_compress_mfma(const CompressArgs& a, hipStream_t s) {
  const int es = a.x_dtype == TQ_F32 ? 4 : 2;
  if ((reinterpret_cast<uintptr_t>(a.x) & 15) || (a.x_hs * es) & 15 || a.split % 32) return 0;
  switch (a.d) {
    case 64: return launch_d<64>(a, s);
    case 96: return launch_d<96>(a, s);
    case 128: return launch_d<128>(a, s);
    case 256: return launch_d<256>(a, s);
  }
  return 0;
}

}  // namespace tq
