// Dequantize on MFMA for gfx950: out = n (c[idx] R) [+ sqrt(pi/2)/d gamma (z S)]
// for head_dim 64, 96, 128 and 256, any width, sketches of at most 128
// projections (replaces metal_dequantize, kernels.py:313-360, and the
// QJL correction, qjl.py:70-94); other shapes take dequant_kernel.
//
// Per output element d multiply-adds against 4 bytes written: the float32
// VALU product was the bound. Here each wave owns 32 output dims and keeps
// its columns of R (and S) as MFMA A operands in registers for the whole
// launch, high part and remainder of 256 R in fp16 (D / 2 registers); the B
// operand is 16 tokens x 32 rotated dims of centroids, looked up from the
// codes in pairs in an LDS table of (high pair, remainder pair) fp16 entries of
// 256 c (16 replicas per entry). Three MFMAs per 32 dims (high x high, high x
// remainder both ways) give the product to the parts' 22 to 24 bits, float32
// accumulation. The
// waves of a workgroup decode the same codes each: 8 lookups of 8 bytes cost
// the LDS reads of the decoded planes, and no barrier is needed in the loop.
// Row m of output block n2 is dim 32 w + 8 (m >> 2) + 4 n2 + (m & 3), so a lane
// ends up with 8 consecutive dims of one token. The next 32 tokens' codes are
// in flight while a tile is computed.
//
// Measured against dequant_kernel: 64,512 vectors of head_dim 128, K4 / V2:
// 106 -> 18.7 us (2.1 TB/s of codes read and floats written; what is left is
// the set-up, strided loads of R's columns, and two short waves of tiles per
// workgroup); 65,536 vectors with 128 projections 213 -> 30 us; 8 rows of one
// token at head_dim 64 / 128 / 256 22.9 / 46.2 / 67.8 -> 4.2 / 4.7 / 9.9 us. Error
// against float64 over every head_dim, width and sketch (165 codecs, 6 inputs
// each): 0.55 of dequant_kernel's (geometric mean), larger for none.

#include <algorithm>
#include <atomic>

#include "tq_codec.h"

namespace tq {
namespace {

typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef float f4 __attribute__((ext_vector_type(4)));
typedef uint32_t u4 __attribute__((ext_vector_type(4)));
typedef uint32_t u2 __attribute__((ext_vector_type(2)));

constexpr float SC = 256.f;   // scale of R, S and c before the fp16 split
constexpr int TROW = 128;     // bytes per table entry (16 replicas)
constexpr int TT = 32;        // tokens per tile

__device__ inline half8 as_h8(u4 v) { return __builtin_bit_cast(half8, v); }
__device__ inline f4 mfma(half8 a, half8 b, f4 c) { return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0); }

// pair table of a 2^bits-entry codebook; codebook word i (fp16 high part |
// remainder << 16 of 256 c_i) in cw[i]
__device__ inline void pair_table(uint8_t* tab, int bits, const uint32_t* cw, int tid, int nt) {
  const uint32_t mask = (1u << bits) - 1u;
  for (int s = tid; s < (1 << (2 * bits)) * (TROW / 16); s += nt) {
    const uint32_t e = s / (TROW / 16);
    const uint32_t a = cw[e & mask], b = cw[e >> bits];
    const uint32_t hi = __builtin_amdgcn_perm(b, a, 0x05040100u), lo = __builtin_amdgcn_perm(b, a, 0x07060302u);
    *reinterpret_cast<u4*>(tab + 16 * s) = u4{hi, lo, hi, lo};
  }
}

// MK: 32-projection words of the sketch held (0: none); projections past
// qjl_m are zero columns
template <int D, int MK>
__global__ __launch_bounds__(2 * D) void dequant_mfma_kernel(DequantArgs a, int tiles_per_row, int total) {
  constexpr int KS = D / 32, NT = 2 * D;
  extern __shared__ __align__(16) uint8_t smem[];
  __shared__ uint32_t cws[2][16];
  const int tid = threadIdx.x, lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r = lane & 15, q4 = lane >> 4;
  const bool frac = a.split < D;
  if (tid < 32) {
    const int lo = tid >> 4, n = 1 << (lo ? a.bits_lo : a.bits_hi);
    const float x = SC * (lo ? a.cen_lo : a.cen_hi)[min(tid & 15, n - 1)];
    const _Float16 h = (_Float16)x, l = (_Float16)(x - (float)h);
    cws[lo][tid & 15] = (uint32_t)__builtin_bit_cast(uint16_t, h) | (uint32_t)__builtin_bit_cast(uint16_t, l) << 16;
  }

  // the lane's 8-dim units of a row (unit 4 s + q4 of step s): a dword of the
  // hi or lo code row, kept inside the row, and the shift of its first code
  const int tab_lo = (1 << (2 * a.bits_hi)) * TROW;
  int uoff[KS], ush[KS], ubits[KS], utab[KS];
  bool ulo[KS];
#pragma unroll
  for (int s = 0; s < KS; ++s) {
    const int j = 8 * (4 * s + q4);
    ulo[s] = frac && j >= a.split;
    ubits[s] = ulo[s] ? a.bits_lo : a.bits_hi;
    const int bit = ubits[s] * (ulo[s] ? j - a.split : j);
    uoff[s] = min(bit >> 3, (ulo[s] ? a.row_lo : a.row_hi) - 4);
    ush[s] = bit - 8 * uoff[s];
    utab[s] = (ulo[s] ? tab_lo : 0) + 8 * r;
  }

  struct Tile {
    int id, row, t0, n, src0, dst0;
  };
  auto make_tile = [&](int id) {
    Tile t{id, 0, 0, 0, 0, 0};
    for (; t.id < total; t.id += gridDim.x) {
      t.row = t.id / tiles_per_row;
      t.t0 = (t.id - t.row * tiles_per_row) * TT;
      const int b = t.row / a.span.heads;
      const int n = a.span.n_tok_b ? a.span.n_tok_b[b] : a.span.n_tok;
      t.n = min(TT, n - t.t0);
      if (t.n > 0) {
        t.src0 = (a.span.src_tok0_b ? a.span.src_tok0_b[b] : 0) + t.t0;
        t.dst0 = (a.span.dst_tok0_b ? a.span.dst_tok0_b[b] : 0) + t.t0;
        break;
      }
    }
    return t;
  };
  struct Codes {
    uint32_t x[2][KS];
    float n[2];
    uint32_t z[2][MK ? MK : 1];
    float g[2];
  };
  // tokens past the tile's end read its last token (not stored)
  auto load = [&](Codes& c, const Tile& t) {
    const uint8_t* hi = a.src.codes_hi + (int64_t)t.row * a.src.hi_head_stride;
    const uint8_t* lo = frac ? a.src.codes_lo + (int64_t)t.row * a.src.lo_head_stride : hi;
    const float* nr = a.src.norms + (int64_t)t.row * a.src.norm_head_stride;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const int64_t tok = t.src0 + min(16 * h + r, t.n - 1);
      const uint8_t* ph = hi + tok * a.row_hi;
      const uint8_t* pl = lo + tok * a.row_lo;
#pragma unroll
      for (int s = 0; s < KS; ++s) __builtin_memcpy(&c.x[h][s], (ulo[s] ? pl : ph) + uoff[s], 4);
      c.n[h] = nr[tok];
      if constexpr (MK > 0) {
        const uint8_t* sg = a.src.signs + (int64_t)t.row * a.src.sign_head_stride + tok * a.row_sign;
#pragma unroll
        for (int s = 0; s < MK; ++s) c.z[h][s] = sg[min(4 * s + q4, a.row_sign - 1)];
        c.g[h] = a.src.gamma[(int64_t)t.row * a.src.gamma_head_stride + tok];
      }
    }
  };
  Tile cur = make_tile(blockIdx.x);
  Codes C;
  if (cur.id < total) load(C, cur);

  // A operands: rows = output dims, k-slots = rotated dims 8 (4 s + q4) + e
  // (projections likewise)
  half8 rh[2][KS], rl[2][KS], sh[2][MK ? MK : 1], sl[2][MK ? MK : 1];
#pragma unroll
  for (int n2 = 0; n2 < 2; ++n2) {
    const int j = 32 * w + 8 * (r >> 2) + 4 * n2 + (r & 3);
#pragma unroll
    for (int s = 0; s < KS; ++s)
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const float v = SC * a.rot[(8 * (4 * s + q4) + e) * D + j];
        const _Float16 h = (_Float16)v;
        rh[n2][s][e] = h;
        rl[n2][s][e] = (_Float16)(v - (float)h);
      }
    if constexpr (MK > 0) {
#pragma unroll
      for (int s = 0; s < MK; ++s)
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          const int p = 8 * (4 * s + q4) + e;
          const float v = p < a.qjl_m ? a.proj[p * D + j] : 0.f;
          const _Float16 h = (_Float16)v;
          sh[n2][s][e] = h;
          sl[n2][s][e] = (_Float16)(SC * (v - (float)h));  // remainders scaled out of the subnormal range
        }
    }
  }
  __syncthreads();
  pair_table(smem, a.bits_hi, cws[0], tid, NT);
  if (frac) pair_table(smem + tab_lo, a.bits_lo, cws[1], tid, NT);
  __syncthreads();

  while (cur.id < total) {
    const Tile nxt = make_tile(cur.id + gridDim.x);
    Codes N = C;
    if (nxt.id < total) load(N, nxt);
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      f4 hh[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}}, xl[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
#pragma unroll
      for (int s = 0; s < KS; ++s) {
        u4 bh, bl;
#pragma unroll
        for (int f = 0; f < 4; ++f) {
          const uint32_t e = __builtin_amdgcn_ubfe(C.x[h][s], ush[s] + 2 * ubits[s] * f, 2 * ubits[s]);
          const u2 t = *reinterpret_cast<const u2*>(smem + e * TROW + utab[s]);
          bh[f] = t[0];
          bl[f] = t[1];
        }
#pragma unroll
        for (int n2 = 0; n2 < 2; ++n2) {
          hh[n2] = mfma(rh[n2][s], as_h8(bh), hh[n2]);
          xl[n2] = mfma(rl[n2][s], as_h8(bh), xl[n2]);
          xl[n2] = mfma(rh[n2][s], as_h8(bl), xl[n2]);
        }
      }
      float o[8];
      // the scale leaves the sum before the norm comes in (2^-16 times a small
      // norm would be subnormal)
#pragma unroll
      for (int i = 0; i < 8; ++i) o[i] = (hh[i >> 2][i & 3] + xl[i >> 2][i & 3]) * (1.f / (SC * SC)) * C.n[h];
      if constexpr (MK > 0) {
        f4 zh[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}}, zl[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
#pragma unroll
        for (int s = 0; s < MK; ++s) {
          // +1 where the bit is set, else -1
          const uint32_t nz = ~C.z[h][s];
          u4 z;
#pragma unroll
          for (int f = 0; f < 4; ++f)
            z[f] = 0x3C003C00u | ((nz << (15 - 2 * f)) & 0x8000u) | ((nz << (30 - 2 * f)) & 0x80000000u);
#pragma unroll
          for (int n2 = 0; n2 < 2; ++n2) {
            zh[n2] = mfma(sh[n2][s], as_h8(z), zh[n2]);
            zl[n2] = mfma(sl[n2][s], as_h8(z), zl[n2]);
          }
        }
        const float cg = 1.2533141373155003f / (float)D * C.g[h];
#pragma unroll
        for (int i = 0; i < 8; ++i) o[i] = fmaf(cg, fmaf(zl[i >> 2][i & 3], 1.f / SC, zh[i >> 2][i & 3]), o[i]);
      }
      if (16 * h + r < cur.n) {
        float* op = a.out + (int64_t)cur.row * a.out_hs + (int64_t)(cur.dst0 + 16 * h + r) * D + 32 * w + 8 * q4;
        *reinterpret_cast<float4*>(op) = make_float4(o[0], o[1], o[2], o[3]);
        *reinterpret_cast<float4*>(op + 4) = make_float4(o[4], o[5], o[6], o[7]);
      }
    }
    C = N;
    cur = nxt;
  }
}

template <int D, int MK>
int launch_dm(const DequantArgs& a, hipStream_t s) {
  // workgroups per CU at the largest table (the same on every gfx950 device)
  static std::atomic<int> known{0};
  const int lds = (1 << (2 * a.bits_hi)) * TROW + (a.split < D ? (1 << (2 * a.bits_lo)) * TROW : 0);
  int occ = known.load(std::memory_order_relaxed);
  if (occ == 0) {
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&occ, dequant_mfma_kernel<D, MK>, 2 * D, 256 * TROW) != hipSuccess)
      occ = 1;
    known.store(occ, std::memory_order_relaxed);
  }
  int dev = 0, cus = 256;
  if (hipGetDevice(&dev) == hipSuccess &&
      hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess)
    cus = 256;
  const int tpr = (a.span.n_tok + TT - 1) / TT;
  const int64_t total = (int64_t)tpr * a.span.rows;
  if (total <= 0 || total >= ((int64_t)1 << 30)) return 0;  // tile ids + 2 grids stay within int
  const int grid = (int)std::min<int64_t>(total, (int64_t)cus * std::max(occ, 1));
  hipLaunchKernelGGL((dequant_mfma_kernel<D, MK>), dim3(grid), dim3(2 * D), lds, s, a, tpr, (int)total);
  return 1;
}

template <int D>
int launch_d(const DequantArgs& a, hipStream_t s) {
  if (!a.apply_qjl) return launch_dm<D, 0>(a, s);
  if (a.qjl_m <= 32) return launch_dm<D, 1>(a, s);
  if (a.qjl_m <= 128) return launch_dm<D, 4>(a, s);
  return 0;
}

}  // namespace

int launch_dequant_mfma(const DequantArgs& a, hipStream_t s) {
  // code rows are read as dwords kept inside the row
  if (a.row_hi < 4 || (a.split < a.d && a.row_lo < 4) || (a.split & 7)) return 0;
  switch (a.d) {
    case 64: return launch_d<64>(a, s);
    case 96: return launch_d<96>(a, s);
    case 128: return launch_d<128>(a, s);
    case 256: return launch_d<256>(a, s);
  }
  return 0;
}

}  // namespace tq
