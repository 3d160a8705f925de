// Decode attention on MFMA for what the K4/V2 / widths / split kernels do not
// take: head_dim 64, 96, 128 and 256, integer widths 2-4 and fractional
// widths on either side, any number of query heads per kv head (groups of at
// most 8), fp16 or bf16 sink / ring tokens, uniform and ragged batches. A
// partials kernel over a fixed grid and a merge kernel.
//
// Grid (ncw + nfw, hkv * gsub, batch), 8 waves. Workgroup c < ncw of a row
// (sequence, head group) takes compressed 32-token blocks (an equal share of
// the sequence's own blocks, wave w blocks w + 8k of it); workgroup ncw + f
// takes 32-token blocks of the uncompressed [sink | ring] list. Each writes one
// partial per query head, [M, L, 0, 0, out[D] / L], in rotated space (c < ncw)
// or original space; the merge weighs them, applies the value codec's R once
// to the rotated sum and adds the other.
//
// Scores are S^T = K q^T on MFMA 16x16x32 f16 (A = 16 tokens x 32 dims). The
// assignment of dims to k-slots is free as long as both operands agree, so
// lane (token r, q4) owns D / 4 contiguous dims of its token: 32 lanes read
// whole code rows, 8 dims per k-step. A pair of codes (2B bits) is looked up
// in an LDS table whose 8-byte entry is (c_hi pair, c_lo pair) in fp16, c_lo =
// c - fp16(c): four lookups fill the high-part and the remainder operand of a
// k-step. The query's fp16 high part and remainder are two columns of B, so
// two MFMAs per step give the whole product but for the operands' own rounding
// (see "Operands" below). For GC = 4 the 16 columns are
// two groups of 8, group t serving 16-token tile t of the block (column c8
// the high part of head c8, c8 < 4, or the remainder of head 7 - c8); for
// GC = 8 column r is part r >> 3 of head r & 7. Columns past the group's
// heads repeat head 0 and are not written.
//
// Output, transposed too: O^T += V^T P^T, A row r = dims (D / 16) r + nb of
// MFMA nb (the value codes of a token's row are one dword, two at D = 256, per
// lane; the two 8-row halves take the two widths of a fractional codec), high
// part and remainder in two MFMAs; P^T = p * n_v as fp16 high part / remainder
// columns, scaled by a power of two per column, and stays in the lane that
// computed the scores.
//
// Tables have 16 replicas per entry (128-byte rows): both sides of every width
// pair fit 80 KB, against 2-way bank conflicts on some lookups.
//
// Operands in two fp16 parts (query, rotated query, R, S, S q, centroids,
// weights) hold 22 to 24 bits where the general kernel's float32 holds 24, and
// low x low products are left out where both sides are in parts. What the sums
// round is more: sixteen MFMA steps here, D float32 steps there. Error against
// float64 over 53 drawn cases (queries N(0, 2), keys of mixed scale) of 3 inputs
// each: 0.54 of the general kernel's (geometric mean; root mean squares 7.0e-7
// and 1.36e-6; 155 of the 159 below it).
//
// Bound: latency, not memory (one layer's codes are 2-9 MB, under 2 us of HBM
// time) and not issue: launch, the set-up's two barriers, the first block's
// round trip, a block's chain of lookups and MFMAs, the combine. Counted: 1,034
// VALU, 150 LDS and 43 MFMA instructions per wave at the first shape below (one
// block a wave), 931 / 103 / 35 at the second (two), 1,323 / 208 / 91 at the third
// (one or none); at four cycles each and two waves per SIMD the VALU takes 3.4,
// 3.1 and 4.4 us of the partials kernel's 12.1, 10.6 and 20.3. Both shrink
// with the work each wave repeats, so the set-up shares it: a thread converts 8
// query elements for all waves, one branch per type around each loop (a branch
// per element took 2.6 us per layer at head_dim 128), bf16 tokens go to bf16
// MFMAs as they are against three bf16 parts of the query and the weights, and
// the accumulators are not rescaled before the first block.
// Measured per layer in a graph of 16 layers, partials + merge against the
// general kernel's three launches (float32 VALU dot products): bf16 K4/V4, 28
// heads on 4, T 16,001: 15.6 us from 101 us (merge 4.1); head_dim 64, bf16
// K4/V2, 2 sequences, 32 heads on 8, T 8,229: 13.0 us from 56 us (merge 3.7);
// head_dim 256, bf16 K4/V3, 8 heads on 2, T 12,000: 26.3 us from 112 us (merge
// 6.5; its rotation reads 256 KB of R per workgroup).
#pragma once

#include <math.h>

#include "tq_common.h"
#include "tq_decode_fast.h"
#include "tq_decode_uniform.h"

namespace tq {
namespace mk {

using uk::as_h8;
using uk::f4;
using uk::fexp2;
using uk::half8;
using uk::mfma;
using uk::row_ror;
using uk::rows_max;
using uk::rows_sum;
using uk::u2;
using uk::u4;

constexpr int MW = MFMA_WAVES;
constexpr int MTH = MW * 64;   // threads
constexpr float M_INIT = uk::M_INIT;
constexpr int TROW = 128;      // bytes per table entry: 16 replicas
// The tables hold CSC times the centroids, and queries are scaled to QLOW <=
// ||q|| <= Q_LIMIT: the fp16 remainders of both stay normal (unscaled, a remainder
// of 0.1 is a multiple of 6e-8) and no element leaves the fp16 range.
constexpr float CSC = 256.f;
constexpr float QLOW = 4096.f;

typedef __bf16 bf8 __attribute__((ext_vector_type(8)));
typedef _Float16 h2 __attribute__((ext_vector_type(2)));
typedef float f2 __attribute__((ext_vector_type(2)));
__device__ inline f4 mfma_b(u4 a, u4 b, f4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf8, a), __builtin_bit_cast(bf8, b), c, 0, 0, 0);
}

// rounded to nearest (one v_cvt_pk_f16_f32): a high part and a remainder hold 24
// bits of a weight without bias; truncated, 22 of them and the sum of weights
// they are divided by too large by 1e-7
__device__ inline h2 to_h2(float a, float b) { return __builtin_convertvector((f2{a, b}), h2); }

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

constexpr int QM = 32;         // projections of the sketch
constexpr int SQS = 2 * QM + 16;
constexpr float SQD = 32.f;    // S q is held over this (fp16 range: |S q| <= ||S_p|| ||q||)
constexpr float SQRT_HALF_PI_M = 1.2533141373155003f;

// N bytes at any address into dwords (the compiler picks the load widths)
template <int N>
__device__ inline void load_bytes(uint32_t (&w)[(N + 3) / 4], const uint8_t* p) {
  w[(N + 3) / 4 - 1] = 0u;
  __builtin_memcpy(&w[0], p, N);
}

// The pair table of one codebook (word i of `cw` lane 16 bk + i: fp16 high
// part | remainder << 16 of centroid i): entry e = (code of dim 2f) | (code
// of dim 2f + 1) << bits.
__device__ inline void build_table(uint8_t* tab, int bk, int bits, uint32_t cw, int tid) {
  const int n16 = (1 << (2 * bits)) * (TROW / 16);  // whole waves (2 bits: 128)
  const uint32_t mask = (1u << bits) - 1u;
  for (int s = tid; s < n16; s += MTH) {
    const uint32_t e = s / (TROW / 16);
    const uint32_t ca = __builtin_amdgcn_ds_bpermute((16 * bk + (e & mask)) * 4, cw);
    const uint32_t cb = __builtin_amdgcn_ds_bpermute((16 * bk + (e >> bits)) * 4, cw);
    const uint32_t hi = __builtin_amdgcn_perm(cb, ca, 0x05040100u), lo = __builtin_amdgcn_perm(cb, ca, 0x07060302u);
    *reinterpret_cast<u4*>(tab + 16 * s) = u4{hi, lo, hi, lo};
  }
}

// Key width kind KK: 2-4 bits, 7 = 3.5 bits (4 / 3), 5 = 2.5 bits (3 / 2),
// the halves split at D / 2.
template <int D, int KK>
struct KGeo {
  static constexpr bool FR = KK > 4;
  static constexpr int NSEG = FR ? 2 : 1;
  static constexpr int SD = D / NSEG;    // dims per segment
  static constexpr int SST = SD / 32;    // k-steps per segment
  static constexpr int KS = D / 32;      // k-steps
  static constexpr int bits(int seg) { return FR ? (seg ? KK / 2 : (KK + 1) / 2) : KK; }
  static constexpr int segb(int seg) { return SD * bits(seg) / 32; }  // bytes per lane and segment
  static constexpr int ndw(int seg) { return (segb(seg) + 3) / 4; }
  static constexpr int NDW = FR ? ndw(0) + ndw(1) : ndw(0);
  static constexpr int tab(int seg) { return seg ? (1 << (2 * bits(0))) * TROW : 0; }  // table offset
  static constexpr int TABS = tab(0) + (1 << (2 * bits(0))) * TROW + (FR ? (1 << (2 * bits(1))) * TROW : 0);
};

// LDS: [key tables | value tables], reused by the combine buffers, then (from
// MfmaArgs::tail) the query operands, the combine headers and the norm staging.
template <int D, int GC, bool QJ>
struct Lds {
  static constexpr int QS = 2 * D + 16;               // bytes per (head, part) of the query operands
  static constexpr int W = D + (QJ ? QM : 0);         // sums per head
  static constexpr int CMS = W + 4;                   // floats per (wave, head) of the combine buffers
  static constexpr int cmb = MW * GC * CMS * 4;
  static constexpr int qsrc = 0;                      // offsets past tail: the query, 2 or 3 parts per head
  static constexpr int qop = qsrc + GC * 3 * QS;      // the rotated query
  static constexpr int qex = qop + GC * 2 * QS;       // 2^qe per head
  static constexpr int sqo = qex + GC * 4;            // S q, high part / remainder rows of 32 (+ 8)
  static constexpr int cml = sqo + (QJ ? GC * 2 * SQS : 0);
  static constexpr int nst = cml + MW * GC * 8;
  static constexpr int end = nst + MW * (QJ ? 512 : 256);
};

template <int D, int KK, bool QJ>
struct Blk {
  uint32_t k[2][KGeo<D, KK>::NDW];
  uint32_t v[8][D == 256 ? 2 : 1];
  float nk, nv;  // of token t0 + (lane & 31)
  uint32_t zk[QJ ? 2 : 1], zv[QJ ? 8 : 1];  // sign bytes: projections 8 q4 .. of token r; 8 (r >> 2) .. of the value tokens
  float gk, gv;
};

// VF: the values' width is fractional (two tables, rows of two widths); QJ: the
// terms of a 32-projection QJL sketch (qjl.py:70-94). Key term: S q is
// computed at the query rotation (S's rows as two more tiles), its fp16 high
// part / remainder columns meet one operand of 16 tokens x 32 signs (+-1, exact)
// per tile: one MFMA. Value term: u = sum_t p_t gamma_t z_t accumulates in two
// more MFMAs (rows = projections) and travels with the partial; the merge
// applies S^T. Per layer: head_dim 64 59.4 -> 16.8 us (13.0 without the sketch),
// head_dim 256 106.7 -> 33.4, bf16 K4/V4 28 heads on 4 104 -> 20.9 (the cases
// above, against the general kernel).
template <int D, int GC, int KK, bool VF, bool QJ>
__global__ __launch_bounds__(MTH) void mfma_decode_kernel(MfmaArgs a) {
  using G_ = KGeo<D, KK>;
  using L_ = Lds<D, GC, QJ>;
  constexpr int U = D / 16;           // dims per MFMA row of the output
  constexpr int NF = U / 2;           // pair fields per row
  constexpr int VW = D == 256 ? 2 : 1;
  constexpr int TS = GC == 4 ? 2 : 1; // tiles sharing the columns
  constexpr int NS = 8 / TS;          // scores per lane per block
  constexpr int PSD = L_::W + 4;
  // the first uncompressed block's keys and values are requested before the
  // query is converted; at D = 256 the registers do not hold both: each is
  // requested where it is used
  constexpr bool EARLY = D < 256;
  // the remainders' score products in accumulators of their own: half as many
  // roundings at the scores' magnitude (a sketch at D >= 128 has no registers
  // for them). Error against float64, relative to the general kernel's, 0.62 ->
  // 0.54 over 53 drawn cases; at most 0.1 us per layer
  constexpr bool SL = !QJ || D < 128;
  extern __shared__ __align__(16) uint8_t smem[];
  uint8_t* tail = smem + a.tail;

  const int c = blockIdx.x, gy = blockIdx.y, b = blockIdx.z;
  const int tid = threadIdx.x, lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r = lane & 15, q4 = lane >> 4;
  const int kvh = gy / a.gsub, row = b * a.hkv + kvh;
  const int head0 = gy * a.g;  // query head of the group's first column: kvh (hq / hkv) + (gy % gsub) g
  const int c8 = r & 7;
  const int tile = TS == 2 ? r >> 3 : 0;
  const bool lo_part = TS == 2 ? c8 >= 4 : r >= 8;
  const int hc = TS == 2 ? (c8 < 4 ? c8 : 7 - c8) : c8;
  const int hd = hc < a.g ? hc : 0;
  const bool writer = !lo_part && c8 < a.g && tile == 0;
  const float partf = lo_part ? 1.f : 0.f;
  const bool packed = c < a.ncw;

  auto clampi = [](int v, int mx) { return min(max(v, 0), mx); };
  const int comp = a.comp_len_b ? clampi(a.comp_len_b[b], a.max_comp) : a.max_comp;
  const int sink = a.sink_len_b ? clampi(a.sink_len_b[b], a.max_sink) : a.max_sink;
  const int res = a.res_len_b ? clampi(a.res_len_b[b], a.max_res) : a.max_res;
  const int nfp = sink + res;
  // blocks [blk0, blk1) of 32 tokens
  const int nblk = ((packed ? comp : nfp) + 31) >> 5;
  const int share = packed ? (nblk + a.ncw - 1) / a.ncw : (nblk + a.nfw - 1) / a.nfw;
  const int blk0 = (packed ? c : c - a.ncw) * share, blk1 = min(blk0 + share, nblk);
  float* part = a.part + ((int64_t)(b * gridDim.y + gy) * gridDim.x + c) * a.g * PSD;
  if (blk0 >= blk1) {  // nothing of this sequence (uniform over the workgroup): empty partials
    if (tid < a.g) *reinterpret_cast<float4*>(part + tid * PSD) = make_float4(M_INIT, 0.f, 0.f, 0.f);
    return;
  }

  // ---- loads of the compressed blocks: tokens past the sequence read its
  // last token (masked); all addresses stay inside the sequence's rows
  const uint8_t* kb0 = a.kc + (int64_t)row * a.k_hs;
  const uint8_t* kb1 = G_::FR ? a.kcl + (int64_t)row * a.kl_hs : nullptr;
  const float* knorm = a.kn + (int64_t)row * a.kn_hs;
  const float* vnorm = a.vn + (int64_t)row * a.vn_hs;
  // the value codes of MFMA row r: dims U r .. of the hi row (r < 8 or an
  // integer width) or of the lo row, read as dwords kept inside the row
  const bool vlo = VF && r >= 8;
  const int vb = VF && vlo ? a.vbl : a.vbh;                  // width of this lane's dims
  const int vrow = (VF ? D / 2 : D) * vb / 8;           // bytes per token
  const uint8_t* vp = a.vc + (int64_t)row * a.v_hs;
  if constexpr (VF) vp = vlo ? a.vcl + (int64_t)row * a.vl_hs : vp;
  int voff[VW], vsh[VW];
#pragma unroll
  for (int i = 0; i < VW; ++i) {
    const int bit = vb * (U * (vlo ? r - 8 : r) + 8 * i);
    voff[i] = min(bit >> 3, vrow - 4);
    vsh[i] = bit - 8 * voff[i];
  }
  auto load_blk = [&](Blk<D, KK, QJ>& B, int blk) {
    const int t0 = blk << 5, last = comp - 1;
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      const uint32_t tt = min(t0 + 16 * t + r, last);
      uint32_t w0[G_::ndw(0)];
      load_bytes<G_::segb(0)>(w0, kb0 + (tt * (uint32_t)(4 * G_::segb(0)) + q4 * G_::segb(0)));
#pragma unroll
      for (int i = 0; i < G_::ndw(0); ++i) B.k[t][i] = w0[i];
      if constexpr (G_::FR) {
        uint32_t w1[G_::ndw(1)];
        load_bytes<G_::segb(1)>(w1, kb1 + (tt * (uint32_t)(4 * G_::segb(1)) + q4 * G_::segb(1)));
#pragma unroll
        for (int i = 0; i < G_::ndw(1); ++i) B.k[t][G_::ndw(0) + i] = w1[i];
      }
    }
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const uint32_t tt = min(t0 + (i < 4 ? 4 * q4 + i : 12 + 4 * q4 + i), last);
#pragma unroll
      for (int j = 0; j < VW; ++j) __builtin_memcpy(&B.v[i][j], vp + (tt * (uint32_t)vrow + voff[j]), 4);
    }
    const int tn = min(t0 + (lane & 31), last);
    B.nk = knorm[tn];
    B.nv = vnorm[tn];
    if constexpr (QJ) {
      const uint8_t* ks = a.ksg + (int64_t)row * a.ksg_hs + q4;
      const uint8_t* vs = a.vsg + (int64_t)row * a.vsg_hs + (r >> 2);
#pragma unroll
      for (int t = 0; t < 2; ++t) B.zk[t] = ks[(uint32_t)min(t0 + 16 * t + r, last) * (QM / 8)];
#pragma unroll
      for (int i = 0; i < 8; ++i)
        B.zv[i] = vs[(uint32_t)min(t0 + (i < 4 ? 4 * q4 + i : 12 + 4 * q4 + i), last) * (QM / 8)];
      B.gk = a.kgam[(int64_t)row * a.kgam_hs + tn];
      B.gv = a.vgam[(int64_t)row * a.vgam_hs + tn];
    }
  };

  // ---- set-up: the query (8 elements per thread, LPH lanes per head) and the
  // codebooks (one centroid per lane: key hi / lo, value hi / lo in the four
  // 16-lane rows), then the first block
  constexpr int LPH = D == 96 ? 16 : D / 8;
  const int qh = tid / LPH, qi = tid % LPH;
  const bool qact = qh < a.g && qi < D / 8;
  u4 qw0 = {0u, 0u, 0u, 0u}, qw1 = {0u, 0u, 0u, 0u};
  if (qact) {
    const int64_t e = ((int64_t)b * a.hq + head0 + qh) * D + 8 * qi;
    if (a.q_dtype == TQ_F32) {
      qw0 = *reinterpret_cast<const u4*>(static_cast<const float*>(a.q) + e);
      qw1 = *reinterpret_cast<const u4*>(static_cast<const float*>(a.q) + e + 4);
    } else {
      qw0 = *reinterpret_cast<const u4*>(static_cast<const uint16_t*>(a.q) + e);
    }
  }
  uint32_t cw = 0;
  Blk<D, KK, QJ> B0, B1;
  // rows 16 jt + r of R (fp16 high part, rls times the remainder) as B operands
  // of the query rotation
  u4 rqh[G_::KS], rql[G_::KS];
  auto load_rot = [&](int jt) {
    const int o = (16 * jt + r) * D + 8 * q4;
#pragma unroll
    for (int kb = 0; kb < G_::KS; ++kb) {
      rqh[kb] = *reinterpret_cast<const u4*>(a.rot16 + o + 32 * kb);
      rql[kb] = *reinterpret_cast<const u4*>(a.rot_lo + o + 32 * kb);
    }
  };
  if (packed) {
    const float* bp = q4 == 0 ? a.kcen_hi : q4 == 1 ? a.kcen_lo : q4 == 2 ? a.vcen_hi : a.vcen_lo;
    const int nb = 1 << (q4 == 0 ? G_::bits(0) : q4 == 1 ? G_::bits(G_::NSEG - 1) : q4 == 2 ? a.vbh : a.vbl);
    const float x = bp[min(r, nb - 1)];
    if (w < U) load_rot(w);
    load_blk(B0, min(blk0 + w, blk1 - 1));
    const _Float16 h = (_Float16)(CSC * x), l = (_Float16)(CSC * x - (float)h);
    cw = (uint32_t)__builtin_bit_cast(uint16_t, h) | (uint32_t)__builtin_bit_cast(uint16_t, l) << 16;
  }
  // uncompressed tokens: keys / values straight from memory
  u4 kr[2][G_::KS];
  uint32_t vr[8][U / 2];
  const int rstart = clampi(a.res_start_b ? a.res_start_b[b] : a.res_start0, max(a.res_cap - 1, 0));
  auto token = [&](int u, const void* sink_p, const void* res_p) {
    u = min(u, nfp - 1);
    int sl = rstart + (u - sink);
    sl = sl >= a.res_cap ? sl - a.res_cap : sl;
    return u < sink ? static_cast<const uint16_t*>(sink_p) + (int64_t)row * a.sink_hs + (int64_t)u * D
                    : static_cast<const uint16_t*>(res_p) + (int64_t)row * a.res_hs + (int64_t)sl * D;
  };
  auto load_k = [&](int t0) {
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      const uint16_t* p = token(t0 + 16 * t + r, a.sink_k, a.res_k) + 8 * q4;
#pragma unroll
      for (int s = 0; s < G_::KS; ++s) kr[t][s] = *reinterpret_cast<const u4*>(p + 32 * s);
    }
  };
  auto load_v = [&](int t0) {
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const uint16_t* p = token(t0 + (i < 4 ? 4 * q4 + i : 12 + 4 * q4 + i), a.sink_v, a.res_v) + U * r;
      __builtin_memcpy(&vr[i][0], __builtin_assume_aligned(p, 4), 2 * U);
    }
  };
  if constexpr (EARLY)
    if (!packed) {
      load_k((blk0 + w) << 5);
      load_v((blk0 + w) << 5);
    }

  // q 2^-qe (query_exponent) in parts: fp16 high part and remainder, or for
  // bf16 uncompressed tokens three bf16 parts
  const bool bfp = !packed && a.bf;
  if (w * 64 < a.g * LPH) {
    float x[8];
    if (a.q_dtype == TQ_F16) {
#pragma unroll
      for (int i = 0; i < 8; ++i) x[i] = (float)as_h8(qw0)[i];
    } else if (a.q_dtype == TQ_BF16) {
#pragma unroll
      for (int i = 0; i < 8; ++i) x[i] = __uint_as_float(i & 1 ? qw0[i >> 1] & 0xFFFF0000u : qw0[i >> 1] << 16);
    } else {
#pragma unroll
      for (int i = 0; i < 8; ++i) x[i] = __uint_as_float(i < 4 ? qw0[i] : qw1[i - 4]);
    }
    float ss = 0.f;
#pragma unroll
    for (int i = 0; i < 8; ++i) ss = fmaf(x[i], x[i], ss);
#pragma unroll
    for (int k = 1; k < LPH; k *= 2) ss += __shfl_xor(ss, k);
    float qn = sqrtf(ss);
    if (__builtin_amdgcn_ballot_w64(qact && !(ss > 1e-30f && ss < 1e30f)) != 0) {
      // (a zero query, or one whose squares leave float32: the norm of q 2^-e)
      float mx = 0.f, s2 = 0.f;
#pragma unroll
      for (int i = 0; i < 8; ++i) mx = fmaxf(mx, fabsf(x[i]));
#pragma unroll
      for (int k = 1; k < LPH; k *= 2) mx = fmaxf(mx, __shfl_xor(mx, k));
      const int e = __builtin_amdgcn_frexp_expf(mx);
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const float y = __builtin_amdgcn_ldexpf(x[i], -e);
        s2 = fmaf(y, y, s2);
      }
#pragma unroll
      for (int k = 1; k < LPH; k *= 2) s2 += __shfl_xor(s2, k);
      qn = fminf(__builtin_amdgcn_ldexpf(sqrtf(s2), e), 3.4e38f);
    }
    const int qe = query_exponent(qn, 1.f, uk::Q_LIMIT, QLOW);
    const float qdown = __builtin_amdgcn_ldexpf(1.f, -qe);
    if (qact) {
      uint8_t* d = tail + L_::qsrc + qh * 3 * L_::QS + 16 * qi;
#pragma unroll
      for (int i = 0; i < 8; ++i) x[i] *= qdown;
      if (bfp) {
        u4 p[3];
        split_b(x, p);
#pragma unroll
        for (int k = 0; k < 3; ++k) *reinterpret_cast<u4*>(d + k * L_::QS) = p[k];
      } else {
        // (the remainder in the scale of R's, whose products it joins)
        half8 hi, lo;
        const float ls = packed ? a.rls : 1.f;
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          hi[i] = (_Float16)x[i];
          lo[i] = (_Float16)((x[i] - (float)hi[i]) * ls);
        }
        *reinterpret_cast<half8*>(d) = hi;
        *reinterpret_cast<half8*>(d + L_::QS) = lo;
      }
      if (qi == 0) *reinterpret_cast<float*>(tail + L_::qex + 4 * qh) = __builtin_amdgcn_ldexpf(1.f, qe);
    }
  }
  if (packed) {
    build_table(smem, 0, G_::bits(0), cw, tid);
    if constexpr (G_::FR) build_table(smem + G_::tab(1), 1, G_::bits(1), cw, tid);
    build_table(smem + G_::TABS, 2, a.vbh, cw, tid);
    if constexpr (VF) build_table(smem + G_::TABS + (1 << (2 * a.vbh)) * TROW, 3, a.vbl, cw, tid);
  }
  __syncthreads();
  const float qe_scale = *reinterpret_cast<const float*>(tail + L_::qex + 4 * hd);
  uint8_t* qop = tail + L_::qop;
  if (packed) {
    // rotated query, D[h][n] = sum_i q[h][i] R[j0 + n][i], written as fp16 high
    // part / remainder rows [head][part][D] (the scores take qscale: a small
    // one here would push the remainders below fp16's normal range)
    const uint8_t* qs = tail + L_::qsrc + min(r, a.g - 1) * 3 * L_::QS + 16 * q4;
    const float lup = 1.f / a.rls;  // a power of two
    for (int jt = w; jt < U; jt += MW) {
      if (jt != w) load_rot(jt);
      f4 dq = {0.f, 0.f, 0.f, 0.f}, dl = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int kb = 0; kb < G_::KS; ++kb) {
        const half8 qhi = *reinterpret_cast<const half8*>(qs + 64 * kb);
        dq = mfma(qhi, as_h8(rqh[kb]), dq);
        dl = mfma(qhi, as_h8(rql[kb]), dl);
        dl = mfma(*reinterpret_cast<const half8*>(qs + L_::QS + 64 * kb), as_h8(rqh[kb]), dl);
      }
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int h = 4 * q4 + i;
        if (h < a.g && h < GC) {
          const float v = fmaf(dl[i], lup, dq[i]);
          const _Float16 hi = (_Float16)v, lo = (_Float16)(v - (float)hi);
          uint8_t* d = qop + (h * 2) * L_::QS + 2 * (16 * jt + r);
          *reinterpret_cast<_Float16*>(d) = hi;
          *reinterpret_cast<_Float16*>(d + L_::QS) = lo;
        }
      }
    }
    if constexpr (QJ) {
      // S (q 2^-qe) / SQD, tiles U and U + 1 of the same waves' sequence
      for (int jt = w; jt < U + QM / 16; jt += MW) {
        if (jt < U) continue;
        const int p = 16 * (jt - U) + r;
        const float* sp = a.proj + p * D + 8 * q4;
        f4 dq = {0.f, 0.f, 0.f, 0.f}, dl = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int kb = 0; kb < G_::KS; ++kb) {
          half8 sh, sl;
#pragma unroll
          for (int e = 0; e < 8; ++e) {
            const float v = sp[32 * kb + e];
            sh[e] = (_Float16)v;
            sl[e] = (_Float16)((v - (float)sh[e]) * a.rls);
          }
          const half8 qhi = *reinterpret_cast<const half8*>(qs + 64 * kb);
          dq = mfma(qhi, sh, dq);
          dl = mfma(qhi, sl, dl);
          dl = mfma(*reinterpret_cast<const half8*>(qs + L_::QS + 64 * kb), sh, dl);
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int h = 4 * q4 + i;
          if (h < a.g && h < GC) {
            const float v = fmaf(dl[i], lup, dq[i]) * (1.f / SQD);
            const _Float16 hi = (_Float16)v, lo = (_Float16)(v - (float)hi);
            uint8_t* d = tail + L_::sqo + h * 2 * SQS + 2 * p;
            *reinterpret_cast<_Float16*>(d) = hi;
            *reinterpret_cast<_Float16*>(d + SQS) = lo;
          }
        }
      }
    }
    __syncthreads();
  }

  // B operands of the scores: step (seg, s) k-slot (q4, e) is dim seg SD +
  // q4 SD / 4 + 8 s + e (uncompressed tokens: 32 s + 8 q4 + e, so that one load
  // covers 64 contiguous bytes of each of 16 rows; the order above would fetch
  // every 128-byte line once per step)
  half8 qb[G_::KS];
  {
    const uint8_t* src = packed ? qop + (hd * 2 + (lo_part ? 1 : 0)) * L_::QS
                                : tail + L_::qsrc + (hd * 3 + (lo_part ? 1 : 0)) * L_::QS;
#pragma unroll
    for (int s = 0; s < G_::KS; ++s) {
      const int d = packed ? s / G_::SST * G_::SD + q4 * (G_::SD / 4) + 8 * (s % G_::SST) : 32 * s + 8 * q4;
      qb[s] = *reinterpret_cast<const half8*>(src + 2 * d);
    }
  }

  // ---- online softmax in base 2, per lane, of column r
  float m_run = M_INIT, l_run = 0.f;
  int vx = 0;         // exponent of the column: acc holds the sums times 2^-vx
  bool vset = false;  // vx set by the wave's first block with a nonzero weight (wave-uniform)
  f4 acc[U];
#pragma unroll
  for (int nb = 0; nb < U; ++nb) acc[nb] = f4{0.f, 0.f, 0.f, 0.f};
  f4 accu[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};  // value term, projections 2 row + n2
  float gv[NS], pu[NS];  // the block's value residual norms, weights times them

  bool any = false;   // the wave has accumulated a block
  uint32_t redo = 0;  // columns whose uncompressed tokens are taken again (wave-uniform)
  // running max and sum over the block's scores s, weights times nv to pv; the
  // accumulators follow a raised max (nothing to follow in the first block)
  auto softmax = [&](const float (&s)[NS], const float (&nv)[NS], float (&pv)[NS]) {
    float bm = s[0];
#pragma unroll
    for (int i = 1; i < NS; ++i) bm = fmaxf(bm, s[i]);
    bm = rows_max(bm);
    if (__builtin_amdgcn_ballot_w64(bm > m_run) != 0) {
      const float mnew = bm > m_run ? bm + uk::RESCALE_MARGIN : m_run;
      if (any) {
        const float corr = fexp2(m_run - mnew);
        l_run *= corr;
#pragma unroll
        for (int nb = 0; nb < U; ++nb) acc[nb] *= corr;
        if constexpr (QJ) accu[0] *= corr, accu[1] *= corr;
      }
      m_run = mnew;
    }
    any = true;
#pragma unroll
    for (int i = 0; i < NS; ++i) {
      const float p = fexp2(s[i] - m_run);
      l_run += p;
      pv[i] = p * nv[i];
      if constexpr (QJ) pu[i] = p * gv[i];
    }
  };
  // the two tiles' k-slots of the P^T operand from the lane's packed pairs
  auto slots = [&](const uint32_t (&d)[NS / 2]) {
    u4 pb;
    if constexpr (TS == 2) {
      pb[0] = tile ? 0u : d[0];
      pb[1] = tile ? 0u : d[1];
      pb[2] = tile ? d[0] : 0u;
      pb[3] = tile ? d[1] : 0u;
    } else {
#pragma unroll
      for (int j = 0; j < 4; ++j) pb[j] = d[j];
    }
    return pb;
  };
  // P^T in fp16 (operand_h): high part or remainder by column, times 2^-vx; vx is
  // set by the wave's first nonzero weight (the accumulators are zero until then)
  auto exponent_h = [&](const float (&pv)[NS]) {
    float pm = 0.f;
#pragma unroll
    for (int i = 0; i < NS; ++i) pm = fmaxf(pm, QJ ? fmaxf(fabsf(pv[i]), fabsf(pu[i])) : fabsf(pv[i]));
    const float pmx = pm * __builtin_amdgcn_ldexpf(1.f, -vx);
    if (__builtin_amdgcn_ballot_w64(pmx > uk::PV_LIMIT || (!vset && pmx > 0.f)) != 0) {
      const float cm = rows_max(pm);  // max of the column (unscaled: 2^-vx times it may pass float32)
      if (!vset) {
        vx = cm > 0.f ? max((int)ceilf(log2f(cm) - log2f(uk::PV_SET)), -126) : 0;
        vset = true;
      } else {
        const int up = min(max((int)ceilf(log2f(cm) - log2f(uk::PV_LIMIT)), vx), 256);
        const float f = __builtin_amdgcn_ldexpf(1.f, vx - up);
#pragma unroll
        for (int nb = 0; nb < U; ++nb) acc[nb] *= f;
        if constexpr (QJ) accu[0] *= f, accu[1] *= f;
        vx = up;
      }
    }
  };
  auto operand_h = [&](const float (&pv)[NS]) {
    const float down = __builtin_amdgcn_ldexpf(1.f, -vx);
    uint32_t d[NS / 2];
#pragma unroll
    for (int j = 0; j < NS / 2; ++j) {
      const float p0 = pv[2 * j] * down, p1 = pv[2 * j + 1] * down;
      const h2 h = to_h2(p0, p1);
      d[j] = __builtin_bit_cast(uint32_t, to_h2(fmaf(-partf, (float)h[0], p0), fmaf(-partf, (float)h[1], p1)));
    }
    return slots(d);
  };
  // the scores of this lane from the two tiles' MFMA results, times `f` per
  // token; masked past `end` tokens
  auto lane_scores = [&](float (&sc)[NS], f4 sA, f4 sB, const float (&f)[NS], int t0, int end) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      if constexpr (TS == 2) {
        const float sv = tile ? sB[i] : sA[i];
        sc[i] = (sv + uk::partner<4>(sv)) * f[i];
      } else {
        sc[i] = (sA[i] + uk::partner<8>(sA[i])) * f[i];
        sc[4 + i] = (sB[i] + uk::partner<8>(sB[i])) * f[4 + i];
      }
    }
    if (t0 + 32 > end) {
#pragma unroll
      for (int i = 0; i < NS; ++i)
        if (t0 + 16 * (tile + (i >> 2)) + 4 * q4 + (i & 3) >= end) sc[i] = -INFINITY;
    }
  };

  if (packed) {
    const uint32_t cp = (uint32_t)r * 8;  // replica of this lane
    const uint32_t cpv = cp + G_::TABS + (vlo ? (1u << (2 * a.vbh)) * TROW : 0u);
    const uint32_t vbw = 2 * vb;  // bits per field
    const float ks = qe_scale * a.qscale * (1.f / CSC);
    float* nst = reinterpret_cast<float*>(tail + L_::nst) + w * (QJ ? 128 : 64);  // [key norms 32][value norms 32][gammas]
    half8 qz;  // S q, k-slot (q4, e) = projection 8 q4 + e
    if constexpr (QJ) qz = *reinterpret_cast<const half8*>(tail + L_::sqo + (hd * 2 + (lo_part ? 1 : 0)) * SQS + 16 * q4);
    auto lut = [&](uint32_t addr) { return *reinterpret_cast<const u2*>(smem + addr); };
    auto compute = [&](const Blk<D, KK, QJ>& B, int blk) {
      const int t0 = blk << 5;
      nst[lane] = lane < 32 ? B.nk : B.nv;
      if constexpr (QJ) nst[64 + lane] = lane < 32 ? B.gk : B.gv;
      float nk[NS], nv[NS], gk[NS];
#pragma unroll
      for (int t = 0; t < 2 / TS; ++t) {
        const float4 k4 = *reinterpret_cast<const float4*>(nst + 16 * (t + tile) + 4 * q4);
        const float4 v4 = *reinterpret_cast<const float4*>(nst + 32 + 16 * (t + tile) + 4 * q4);
        nk[4 * t] = k4.x * ks; nk[4 * t + 1] = k4.y * ks; nk[4 * t + 2] = k4.z * ks; nk[4 * t + 3] = k4.w * ks;
        nv[4 * t] = v4.x; nv[4 * t + 1] = v4.y; nv[4 * t + 2] = v4.z; nv[4 * t + 3] = v4.w;
        if constexpr (QJ) {
          const float4 a4 = *reinterpret_cast<const float4*>(nst + 64 + 16 * (t + tile) + 4 * q4);
          const float4 b4 = *reinterpret_cast<const float4*>(nst + 96 + 16 * (t + tile) + 4 * q4);
          gk[4 * t] = a4.x; gk[4 * t + 1] = a4.y; gk[4 * t + 2] = a4.z; gk[4 * t + 3] = a4.w;
          gv[4 * t] = b4.x; gv[4 * t + 1] = b4.y; gv[4 * t + 2] = b4.z; gv[4 * t + 3] = b4.w;
        }
      }
      f4 sc2[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}}, sl2[2] = {sc2[0], sc2[1]};
#pragma unroll
      for (int s = 0; s < G_::KS; ++s) {
        const int seg = s / G_::SST, bits = G_::bits(seg), o = seg ? G_::ndw(0) : 0;
#pragma unroll
        for (int t = 0; t < 2; ++t) {
          u4 hi, lo;
#pragma unroll
          for (int f = 0; f < 4; ++f) {
            const int bit = bits * (8 * (s % G_::SST) + 2 * f), wd = o + (bit >> 5), sh = bit & 31;
            const uint32_t x = sh + 2 * bits <= 32
                                   ? B.k[t][wd] >> sh
                                   : __builtin_amdgcn_alignbit(B.k[t][wd + 1 < G_::NDW ? wd + 1 : wd], B.k[t][wd], sh);
            const u2 e = lut((((x & ((1u << (2 * bits)) - 1u)) * TROW) | cp) + G_::tab(seg));
            hi[f] = e[0];
            lo[f] = e[1];
          }
          sc2[t] = mfma(as_h8(hi), qb[s], sc2[t]);
          f4& sl = SL ? sl2[t] : sc2[t];
          sl = mfma(as_h8(lo), qb[s], sl);
        }
      }
      if constexpr (SL) sc2[0] += sl2[0], sc2[1] += sl2[1];
      float sc[NS];
      if constexpr (QJ) {
        // key term: + gamma_k sqrt(pi / 2) / D (S q) . z, before the mask
        f4 sz[2];
#pragma unroll
        for (int t = 0; t < 2; ++t) {
          const uint32_t nz = ~B.zk[t];
          u4 z;
#pragma unroll
          for (int f = 0; f < 4; ++f)
            z[f] = 0x3C003C00u | ((nz << (15 - 2 * f)) & 0x8000u) | ((nz << (30 - 2 * f)) & 0x80000000u);
          sz[t] = mfma(as_h8(z), qz, f4{0.f, 0.f, 0.f, 0.f});
        }
        const float zs = qe_scale * a.qscale * (SQD * SQRT_HALF_PI_M / D);
        float fz[NS], sq[NS];
#pragma unroll
        for (int i = 0; i < NS; ++i) fz[i] = gk[i] * zs;
        lane_scores(sq, sz[0], sz[1], fz, t0, comp);
        lane_scores(sc, sc2[0], sc2[1], nk, t0, comp);
#pragma unroll
        for (int i = 0; i < NS; ++i) sc[i] += sq[i];
      } else {
        lane_scores(sc, sc2[0], sc2[1], nk, t0, comp);
      }
      float pv[NS];
      softmax(sc, nv, pv);
      exponent_h(pv);
      const half8 pb = as_h8(operand_h(pv));
      if constexpr (QJ) {
        const half8 ub = as_h8(operand_h(pu));
        u4 z[2];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          // bits 2 (r & 3) + n2 of the pair's sign bytes: clear = -1
          const uint32_t x = ~B.zv[2 * j] >> (2 * (r & 3)), y = ~B.zv[2 * j + 1] >> (2 * (r & 3));
#pragma unroll
          for (int n2 = 0; n2 < 2; ++n2)
            z[n2][j] = 0x3C003C00u | ((x << (15 - n2)) & 0x8000u) | ((y << (31 - n2)) & 0x80000000u);
        }
        accu[0] = mfma(as_h8(z[0]), ub, accu[0]);
        accu[1] = mfma(as_h8(z[1]), ub, accu[1]);
      }
#pragma unroll
      for (int f = 0; f < NF; ++f) {
        // dims U r + 2 f, + 1 of the block's 4 token pairs
        u4 va0, va1, vl0, vl1;
        const uint32_t off = (uint32_t)vsh[f >> 2] + vbw * (f & 3);
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const u2 x = lut(__builtin_amdgcn_ubfe(B.v[2 * j][f >> 2], off, vbw) * TROW + cpv);
          const u2 y = lut(__builtin_amdgcn_ubfe(B.v[2 * j + 1][f >> 2], off, vbw) * TROW + cpv);
          va0[j] = __builtin_amdgcn_perm(y[0], x[0], 0x05040100u);
          va1[j] = __builtin_amdgcn_perm(y[0], x[0], 0x07060302u);
          vl0[j] = __builtin_amdgcn_perm(y[1], x[1], 0x05040100u);
          vl1[j] = __builtin_amdgcn_perm(y[1], x[1], 0x07060302u);
        }
        acc[2 * f] = mfma(as_h8(va0), pb, acc[2 * f]);
        acc[2 * f + 1] = mfma(as_h8(va1), pb, acc[2 * f + 1]);
        acc[2 * f] = mfma(as_h8(vl0), pb, acc[2 * f]);
        acc[2 * f + 1] = mfma(as_h8(vl1), pb, acc[2 * f + 1]);
      }
    };
    // two blocks in flight; blocks past the wave's share re-read its last one
    int blk = blk0 + w;
    if (blk < blk1) {
      for (;;) {
        load_blk(B1, min(blk + MW, blk1 - 1));
        compute(B0, blk);
        blk += MW;
        if (blk >= blk1) break;
        load_blk(B0, min(blk + MW, blk1 - 1));
        compute(B1, blk);
        blk += MW;
        if (blk >= blk1) break;
      }
    }
  } else {
    for (int blk = blk0 + w; blk < blk1; blk += MW) {
      const int t0 = blk << 5;
      if (!EARLY || blk != blk0 + w) {
        load_k(t0);
        if constexpr (EARLY) load_v(t0);
      }
      f4 sc2[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
      float sc[NS], kf[NS], nv[NS], pv[NS];
#pragma unroll
      for (int i = 0; i < NS; ++i) kf[i] = a.qscale * qe_scale, nv[i] = 1.f, gv[i] = 0.f;
      if (a.bf) {
        // bf16 tokens on bf16 MFMAs: the third part of the query (and of the
        // weights) in an operand of its own, in the first part's columns
        const uint8_t* src = tail + L_::qsrc + (hd * 3 + 2) * L_::QS + 16 * q4;
#pragma unroll
        for (int s = 0; s < G_::KS; ++s) {
          const u4 x = *reinterpret_cast<const u4*>(src + 64 * s);
          const u4 q3 = u4{lo_part ? 0u : x[0], lo_part ? 0u : x[1], lo_part ? 0u : x[2], lo_part ? 0u : x[3]};
#pragma unroll
          for (int t = 0; t < 2; ++t) {
            sc2[t] = mfma_b(kr[t][s], __builtin_bit_cast(u4, qb[s]), sc2[t]);
            sc2[t] = mfma_b(kr[t][s], q3, sc2[t]);
          }
        }
      } else {
#pragma unroll
        for (int s = 0; s < G_::KS; ++s)
#pragma unroll
          for (int t = 0; t < 2; ++t) sc2[t] = mfma(as_h8(kr[t][s]), qb[s], sc2[t]);
      }
      if constexpr (!EARLY) load_v(t0);
      lane_scores(sc, sc2[0], sc2[1], kf, t0, nfp);
      softmax(sc, nv, pv);
      u4 pb, p3 = {0u, 0u, 0u, 0u};
      if (a.bf) {
        uint32_t d[NS / 2], d3[NS / 2];
#pragma unroll
        for (int j = 0; j < NS / 2; ++j) {
          uint32_t x[2], y[2];
#pragma unroll
          for (int k = 0; k < 2; ++k) {
            const uint32_t p = __float_as_uint(pv[2 * j + k]);
            const uint32_t p2 = __float_as_uint(__uint_as_float(p) - __uint_as_float(p & 0xFFFF0000u));
            x[k] = lo_part ? p2 : p;
            y[k] = lo_part ? 0u : __float_as_uint(__uint_as_float(p2) - __uint_as_float(p2 & 0xFFFF0000u));
          }
          d[j] = __builtin_amdgcn_perm(x[1], x[0], 0x07060302u);
          d3[j] = __builtin_amdgcn_perm(y[1], y[0], 0x07060302u);
        }
        pb = slots(d);
        p3 = slots(d3);
      } else {
        exponent_h(pv);
        pb = operand_h(pv);
      }
#pragma unroll
      for (int nb = 0; nb < U; ++nb) {
        const uint32_t sel = (nb & 1) ? 0x07060302u : 0x05040100u;
        u4 va;
#pragma unroll
        for (int j = 0; j < 4; ++j) va[j] = __builtin_amdgcn_perm(vr[2 * j + 1][nb >> 1], vr[2 * j][nb >> 1], sel);
        if (a.bf) {
          acc[nb] = mfma_b(va, pb, acc[nb]);
          acc[nb] = mfma_b(va, p3, acc[nb]);
        } else {
          acc[nb] = mfma(as_h8(va), as_h8(pb), acc[nb]);
        }
      }
    }
    // Operands in parts and zero k-slots turn an infinite key or value into NaN
    // where its own products are not (0 times infinity): the columns with a NaN or
    // an infinite sum
    float nn = l_run;
#pragma unroll
    for (int nb = 0; nb < U; ++nb)
#pragma unroll
      for (int i = 0; i < 4; ++i) nn = fmaf(acc[nb][i], 0.f, nn);
    const uint64_t nl = __builtin_amdgcn_ballot_w64(nn != nn);
    redo = (uint32_t)(nl | nl >> 16 | nl >> 32 | nl >> 48) & 0xFFFFu;
  }

  // ---- combine the waves through LDS (the table region); the two fp16 parts
  // of a head meet through `partner`, for GC = 4 the two tiles at their common max
  l_run = rows_sum(l_run);
  if (__builtin_amdgcn_ballot_w64(vx < -64) != 0) {
    // small value norms: part of 2^vx now, so that the factor below stays normal
    const float f = __builtin_amdgcn_ldexpf(1.f, min(vx + 64, 0));
#pragma unroll
    for (int nb = 0; nb < U; ++nb) acc[nb] *= f;
    if constexpr (QJ) accu[0] *= f, accu[1] *= f;
    vx = max(vx, -64);
  }
  float tsc = __builtin_amdgcn_ldexpf(1.f, vx);
  if constexpr (TS == 2) {
    const float m2 = fmaxf(m_run, row_ror<8>(m_run));
    const float t = fexp2(m_run - m2);
    tsc *= t;
    l_run *= t;
    l_run += row_ror<8>(l_run);
    m_run = m2;
  }
  __syncthreads();
  const float tscr = packed ? tsc * (1.f / CSC) : tsc;  // (the tables hold CSC c)
  float* cm = reinterpret_cast<float*>(smem) + (w * GC) * L_::CMS;
  float* cl = reinterpret_cast<float*>(tail + L_::cml);  // [wave][head][M, L]
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    float vr[U];
#pragma unroll
    for (int nb = 0; nb < U; ++nb) {
      float x = (acc[nb][i] + uk::partner<GC>(acc[nb][i])) * tscr;
      if constexpr (TS == 2) x += row_ror<8>(x);
      vr[nb] = x;
    }
    if (writer) {
      float* d = cm + hd * L_::CMS + U * (4 * q4 + i);
#pragma unroll
      for (int nb = 0; nb < U; nb += 2) *reinterpret_cast<float2*>(d + nb) = make_float2(vr[nb], vr[nb + 1]);
    }
    if constexpr (QJ) {
      float u[2];
#pragma unroll
      for (int n2 = 0; n2 < 2; ++n2) {
        u[n2] = (accu[n2][i] + uk::partner<GC>(accu[n2][i])) * tsc;
        if constexpr (TS == 2) u[n2] += row_ror<8>(u[n2]);
      }
      if (writer) *reinterpret_cast<float2*>(cm + hd * L_::CMS + D + 2 * (4 * q4 + i)) = make_float2(u[0], u[1]);
    }
  }
  if (q4 == 0 && writer) *reinterpret_cast<float2*>(cl + (w * GC + hd) * 2) = make_float2(m_run, l_run);
  if (redo != 0) {
    // the heads of those columns again: the wave's tokens one at a time in
    // float32, as in chunk_kernel (never taken with finite tokens and sums)
    constexpr int DL = (D + 63) / 64;
    auto elem = [&](const uint16_t* p) {
      return a.bf ? __uint_as_float((uint32_t)*p << 16) : (float)__builtin_bit_cast(_Float16, *p);
    };
    for (int h = 0; h < a.g; ++h) {
      if ((redo & (TS == 2 ? 0x0101u << h | 0x8080u >> h : 0x0101u << h)) == 0) continue;
      const uint8_t* qs = tail + L_::qsrc + h * 3 * L_::QS;
      const float qf = a.qscale * *reinterpret_cast<const float*>(tail + L_::qex + 4 * h);
      float qv[DL], o[DL], mx = M_INIT, l = 0.f;
#pragma unroll
      for (int j = 0; j < DL; ++j) {
        const int d = lane + 64 * j;
        float x = 0.f;
        for (int k = a.bf ? 2 : 1; k >= 0; --k)
          x += d < D ? elem(reinterpret_cast<const uint16_t*>(qs + k * L_::QS) + d) : 0.f;
        qv[j] = x * qf;
        o[j] = 0.f;
      }
      for (int pass = 0; pass < 2; ++pass)
        for (int blk = blk0 + w; blk < blk1; blk += MW)
          for (int u = blk << 5; u < min((blk + 1) << 5, nfp); ++u) {
            const uint16_t* kp = token(u, a.sink_k, a.res_k) + lane;
            float s = 0.f;
#pragma unroll
            for (int j = 0; j < DL; ++j) s = lane + 64 * j < D ? fmaf(qv[j], elem(kp + 64 * j), s) : s;
            s = uk::wave_sum(s);
            if (pass == 0) {
              mx = fmaxf(mx, s);
              continue;
            }
            const float p = fexp2(s - mx);
            l += p;
            const uint16_t* vp = token(u, a.sink_v, a.res_v) + lane;
#pragma unroll
            for (int j = 0; j < DL; ++j) o[j] = lane + 64 * j < D ? fmaf(p, elem(vp + 64 * j), o[j]) : 0.f;
          }
#pragma unroll
      for (int j = 0; j < DL; ++j)
        if (lane + 64 * j < D) cm[h * L_::CMS + lane + 64 * j] = o[j];
      if (lane == 0) *reinterpret_cast<float2*>(cl + (w * GC + h) * 2) = make_float2(mx, l);
    }
  }
  __syncthreads();
  const float* cms = reinterpret_cast<const float*>(smem);
  for (int e = tid; e < a.g * L_::W; e += MTH) {
    const int h = e / L_::W, j = e % L_::W;
    float M = M_INIT;
#pragma unroll
    for (int ww = 0; ww < MW; ++ww) M = fmaxf(M, cl[(ww * GC + h) * 2]);
    float sr = 0.f, Ls = 0.f;
#pragma unroll
    for (int ww = 0; ww < MW; ++ww) {
      const float2 st = *reinterpret_cast<const float2*>(cl + (ww * GC + h) * 2);
      const float sc = fexp2(st.x - M);
      sr = fmaf(sc, cms[(ww * GC + h) * L_::CMS + j], sr);
      Ls = fmaf(sc, st.y, Ls);
    }
    part[h * PSD + 4 + j] = Ls == 0.f ? 0.f : sr / Ls;
    if (j == 0) *reinterpret_cast<float4*>(part + h * PSD) = make_float4(M, Ls, 0.f, 0.f);
  }
}

// Merge of the np = ncw + nfw partials of a query head: with w_p = 2^(M_p - M)
// L_p / L, out = (sum_{p < ncw} w_p y_p) R + sum_{p >= ncw} w_p x_p (x = R^T y,
// R the value codec's float32 rotation). Grid (hq, batch): a chain of dependent
// round trips, so everything is requested at once: PG groups of D threads hold
// MB partials each (64 of them in one round at D <= 128), every wave reads all
// headers, and thread (4 columns, row block) its D / RB rows of R. A partial
// without a weight (L_p = 0) is skipped; one whose sum is NaN (a NaN or +infinite
// score) is not: the head is then zero, as combine_kernel leaves it, and never
// the attention over the other tokens.
template <int D>
struct MergeGeo {
  static constexpr int PG = D == 256 ? 4 : 8;   // partial groups
  static constexpr int NT = PG * D;             // threads
  static constexpr int MB = D == 256 ? 16 : 8;  // partials per group and round
  static constexpr int CT = D / 4;              // column threads of a row block
  static constexpr int RB = NT / CT;            // row blocks (32; 16 at D = 256)
  static constexpr int RR = D / RB;             // rows per block
};

template <int D, bool QJ>
__global__ __launch_bounds__(MergeGeo<D>::NT) void mfma_merge_kernel(MfmaArgs a, int np) {
  using M_ = MergeGeo<D>;
  constexpr int PSD = D + 4 + (QJ ? QM : 0), MB = M_::MB, PG = M_::PG;
  constexpr int UG = QJ ? M_::NT / QM : 1, SR = QJ ? QM / M_::RB : 1;  // groups of the value term, rows of S per block
  extern __shared__ __align__(16) uint8_t smem[];
  float* wsh = reinterpret_cast<float*>(smem);  // [np rounded up to whole rounds] weights
  __shared__ float ys[PG][D], xs[PG][D], yt[D + (QJ ? QM : 0)], us[UG][QM];
  __shared__ __align__(16) float red[M_::RB][D];
  const int hq = blockIdx.x, b = blockIdx.y;
  const int gy = hq / a.g, h = hq % a.g;
  const int tid = threadIdx.x, lane = tid & 63;
  const int64_t pst = (int64_t)a.g * PSD;
  const float* pp = a.part + (int64_t)(b * a.hkv * a.gsub + gy) * np * pst + h * PSD;
  const int d = tid % D, grp = tid / D;
  float2 hd[4];  // headers lane + 64 k (past 256: the loops below)
#pragma unroll
  for (int k = 0; k < 4; ++k) hd[k] = *reinterpret_cast<const float2*>(pp + min(lane + 64 * k, np - 1) * pst);
  float x[MB];
  auto load = [&](int p0) {
#pragma unroll
    for (int i = 0; i < MB; ++i) x[i] = pp[min(p0 + PG * i + grp, np - 1) * pst + 4 + d];
  };
  load(0);
  const int j4 = 4 * (tid % M_::CT), ib = tid / M_::CT;
  float4 rr[M_::RR];
#pragma unroll
  for (int k = 0; k < M_::RR; ++k) rr[k] = *reinterpret_cast<const float4*>(a.vrot + (M_::RR * ib + k) * D + j4);

  float4 sr[SR];
  if constexpr (QJ) {
#pragma unroll
    for (int k = 0; k < SR; ++k) sr[k] = *reinterpret_cast<const float4*>(a.proj + (SR * ib + k) * D + j4);
  }

  float M = M_INIT;
#pragma unroll
  for (int k = 0; k < 4; ++k) M = hd[k].y != 0.f ? fmaxf(M, hd[k].x) : M;  // (repeats of the last header change nothing)
  for (int p = 256 + lane; p < np; p += 64) {
    const float2 e = *reinterpret_cast<const float2*>(pp + p * pst);
    M = e.y != 0.f ? fmaxf(M, e.x) : M;
  }
  M = uk::wave_max(M);
  float ls = 0.f;
  const int npr = (np + PG * MB - 1) / (PG * MB) * (PG * MB);
  for (int p = lane, k = 0; p < npr; p += 64, ++k) {
    float2 e = k == 0 ? hd[0] : k == 1 ? hd[1] : k == 2 ? hd[2] : hd[3];
    if (k >= 4 && p < np) e = *reinterpret_cast<const float2*>(pp + p * pst);
    const float wp = p < np && e.y != 0.f ? fexp2(e.x - M) * e.y : 0.f;
    if (tid < 64) wsh[p] = wp;
    ls += wp;
  }
  const float Ls = uk::wave_sum(ls);
  const float inv = Ls > 0.f ? 1.f / Ls : 0.f;
  __syncthreads();
  float acc = 0.f, acco = 0.f;
  for (int p0 = 0;;) {
#pragma unroll
    for (int i = 0; i < MB; ++i) {
      const int p = p0 + PG * i + grp;
      const float wp = wsh[p];
      const float v = wp != 0.f ? x[i] : 0.f;  // (empty partials may hold anything)
      acc = fmaf(wp, p < a.ncw ? v : 0.f, acc);  // (the other space's sum may be infinite)
      acco = fmaf(wp, p < a.ncw ? 0.f : v, acco);
    }
    p0 += PG * MB;
    if (p0 >= np) break;
    load(p0);
  }
  ys[grp][d] = acc;
  xs[grp][d] = acco;
  if constexpr (QJ) {
    const int i = tid % QM, q = tid / QM;
    float u = 0.f;
    for (int p = q; p < a.ncw; p += UG) {
      const float wp = wsh[p], x = pp[p * pst + 4 + D + i];
      u = fmaf(wp, wp != 0.f ? x : 0.f, u);
    }
    us[q][i] = u;
  }
  __syncthreads();
  if constexpr (QJ)
    if (tid >= D && tid < D + QM) {
      float u = 0.f;
#pragma unroll
      for (int q = 0; q < UG; ++q) u += us[q][tid - D];
      yt[tid] = u * (SQRT_HALF_PI_M / D);
    }
  if (tid < D) {
    float y = 0.f;
#pragma unroll
    for (int q = 0; q < PG; ++q) y += ys[q][tid];
    yt[tid] = y;
  }
  __syncthreads();
  {
    float4 o = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
    for (int k = 0; k < M_::RR; ++k) {
      const float y = yt[M_::RR * ib + k];
      o.x = fmaf(y, rr[k].x, o.x);
      o.y = fmaf(y, rr[k].y, o.y);
      o.z = fmaf(y, rr[k].z, o.z);
      o.w = fmaf(y, rr[k].w, o.w);
    }
    if constexpr (QJ) {
#pragma unroll
      for (int k = 0; k < SR; ++k) {
        const float u = yt[D + SR * ib + k];
        o.x = fmaf(u, sr[k].x, o.x);
        o.y = fmaf(u, sr[k].y, o.y);
        o.z = fmaf(u, sr[k].z, o.z);
        o.w = fmaf(u, sr[k].w, o.w);
      }
    }
    *reinterpret_cast<float4*>(&red[ib][j4]) = o;
  }
  __syncthreads();
  if (tid < D) {
    float s = 0.f;
#pragma unroll
    for (int k = 0; k < M_::RB; ++k) s += red[k][tid];
#pragma unroll
    for (int q = 0; q < PG; ++q) s += xs[q][tid];
    a.out[((int64_t)b * a.hq + hq) * D + tid] = Ls > 0.f ? s * inv : 0.f;
  }
}

template <int D, int GC, int KK, bool QJ>
static void launch_k(const MfmaArgs& a, hipStream_t s) {
  using G_ = KGeo<D, KK>;
  using L_ = Lds<D, GC, QJ>;
  MfmaArgs x = a;
  const int vt = (1 << (2 * a.vbh)) * TROW + (a.vfrac ? (1 << (2 * a.vbl)) * TROW : 0);
  x.tail = G_::TABS + vt > L_::cmb ? G_::TABS + vt : L_::cmb;
  const int lds = x.tail + L_::end;
  const dim3 grid(a.ncw + a.nfw, a.hkv * a.gsub, a.batch);
  if (a.vfrac)
    hipLaunchKernelGGL((mfma_decode_kernel<D, GC, KK, true, QJ>), grid, dim3(MTH), lds, s, x);
  else
    hipLaunchKernelGGL((mfma_decode_kernel<D, GC, KK, false, QJ>), grid, dim3(MTH), lds, s, x);
}

template <int D, int KK, bool QJ>
static void launch_g(const MfmaArgs& a, hipStream_t s) {
  if (a.g <= 4)
    launch_k<D, 4, KK, QJ>(a, s);
  else
    launch_k<D, 8, KK, QJ>(a, s);
}

// kk: key width kind (KGeo); -1 for one that has no kernel, launch errors are the
// caller's to ask for
template <int D, bool QJ>
int launch_mfma(const MfmaArgs& a, int kk, hipStream_t s) {
  switch (kk) {
    case 2: launch_g<D, 2, QJ>(a, s); break;
    case 3: launch_g<D, 3, QJ>(a, s); break;
    case 4: launch_g<D, 4, QJ>(a, s); break;
    case 5:
      if constexpr (D != 96) launch_g<D, 5, QJ>(a, s);
      break;
    case 7:
      if constexpr (D != 96) launch_g<D, 7, QJ>(a, s);
      break;
    default: return -1;
  }
  const int np = a.ncw + a.nfw;
  constexpr int round = MergeGeo<D>::PG * MergeGeo<D>::MB;
  hipLaunchKernelGGL((mfma_merge_kernel<D, QJ>), dim3(a.hq, a.batch), dim3(MergeGeo<D>::NT),
                     (np + round - 1) / round * round * 4, s, a, np);
  return 0;
}

}  // namespace mk
}  // namespace tq
