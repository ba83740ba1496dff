// units.hip — attention of multi-row segments the prefill kernel has no instance for, and of every
// row of the row layout and f32 pages, on gfx950 matrix cores.
//
// Computes what `attend` computes (crates/engine/model/src/forward.rs:585-807). A unit is up to
// 16 * NB columns (token, query head) of one segment and KV head, flattened token-major as the
// prefill kernel's units are, over the key pages its columns see. A unit's keys are shared by 1 to W
// consecutive waves of one workgroup (the planner packs units into workgroups), whose partials merge
// in LDS; a unit longer than a workgroup's waves should walk runs as key pieces whose partials a
// merge launch combines. So the rows of a short segment (a run of drafted tokens) read each page
// once, not once per row, and wide heads, f32 pages and rows off the tile layout run on the matrix
// cores.
//
// Per step of KT page tiles (32 keys; 16 on f32 pages), operands straight from HBM to registers:
//   S^T[keys x cols] = K . Q^T       16-bit: v_mfma_f32_16x16x32, Q as hi + lo parts of the type
//                                    f32:    v_mfma_f32_16x16x4f32
//   O^T[dims x cols] += V^T . P^T    16-bit: v_mfma_f32_16x16x32_f16, P as f16 hi + lo parts
//                                    f32:    v_mfma_f32_16x16x4f32
// with the same lazy online softmax, precision and q8_0 scheme as the decode work item
// (decode_tile.h); in the row layout Q and P have three parts of the pages' 16-bit type (24 bits, as in
// f32; bf16 there takes P.V in bf16). One step's operands are held; a register is requested again for the
// next step as soon as its products are issued, so every load has a whole step to arrive in (the two-tile
// buffers of the decode item would not leave room for a second column block).
//
// Measured, one step of lmh_attend, against a decode item per row (before; the row layout's and f32
// pages' on the VALU): 24 sequences x 4 rows on 512 .. 4,096 keys (32/8 heads, hd 128, bf16, 190 MB of
// pages): 98.5 -> 42 us, 36.6 of them this kernel (202 MB read at 5.5 TB/s, 5.9 at four times the contexts:
// bound by HBM) and 4.4 the cut units' merge; hd 256 prompts of 600 and 800 tokens, window 1,024: 225 -> 62 us
// (57 before non-finite V of a masked key was kept out: the masked steps wait for V to test it), bound by the
// chain of one wave per SIMD's steps and a second, partly filled round of workgroups (waves resident 62 % of
// the time, issuing VALU 25 % and in the matrix pipe 12 %), two of 2,048: 410 TFLOP/s; hd 80, 32 heads of
// their own K/V, 8 decode rows and a 120-token chunk: 1,038 -> 29 us (23.5 + merge 4.1; 85 MB; decode rows
// alone at 8,000 keys: 5.0 TB/s); f32 prompts of 450 and 390 tokens, hd 64: 102 -> 23 us (four steps a wave:
// the chain from its record to its merge; matrix pipe 21 %). The row layout's loads are ordinary ones: a row's
// lines are touched by several lanes' loads, and as streaming loads they were fetched again for each (8,000
// keys at hd 80: 200 -> 140 us).
//
// An instance of the row layout or of f32 pages takes every width up to its own: lanes past a row's end
// hold zeros (K) or re-read the row's first dims into blocks that are never stored (V).
//
// Row layout and f32 pages hold key rows as they are, so the operands' element order is chosen to
// suit the loads: 16-bit V pairs two dims per lane (a dword per key and 32-dim block: block 2b + p
// holds dims 32b + 2m + p, m = 0..15), f32 K and V four (a float4; f32 K chunk c, product i: k index
// g is dim 16c + 4g + i; V block 4b + j: dims 64b + 4m + j).
#include "decode_tile.h"

#include <algorithm>
#include <atomic>

namespace lmh {
namespace {

using namespace dtile;

constexpr int FT_F16 = 0, FT_BF16 = 1, FT_Q8 = 2, FR_F16 = 3, FR_BF16 = 4, FR_F32 = 5;

// bf16 pair (one uint32) -> f16 pair, exact in the normal f16 range.
__device__ inline uint32_t bf2_h2(uint32_t w) {
  typedef float f2 __attribute__((ext_vector_type(2)));
  typedef _Float16 h2 __attribute__((ext_vector_type(2)));
  const f2 x = {__uint_as_float(w << 16), __uint_as_float(w & 0xffff0000u)};
  return __builtin_bit_cast(uint32_t, __builtin_convertvector(x, h2));
}

typedef float f4u __attribute__((ext_vector_type(4), aligned(4)));   // caller arrays: any float address

template <bool NT>
__device__ inline uint4 load16(const uint8_t* p) {
  if constexpr (NT) return load_stream(p);
  return *(const uint4*)p;
}
template <bool NT>
__device__ inline uint32_t load4(const uint8_t* p) {
  if constexpr (NT) return __builtin_nontemporal_load((const uint32_t*)p);
  return *(const uint32_t*)p;
}

template <int F, int HDP, int HDVP, int NB>
struct Cfg {
  static constexpr bool BF = F == FT_BF16 || F == FR_BF16, Q8 = F == FT_Q8, ROWS = F >= FR_F16, F32 = F == FR_F32;
  static constexpr int KT = F32 ? 1 : 2;                    // page tiles per step
  static constexpr int NC = F32 ? HDP / 16 : HDP / 32;      // Q.K chunks
  static constexpr int NJ = F32 ? HDVP / 64 * 4 : HDVP / 16;  // O^T blocks of 16 dims
  static constexpr int GRP = F32 ? 4 : ROWS ? 2 : 1;        // O^T blocks whose dims interleave
  static constexpr int KR = Q8 ? HDP / 64 : NC;             // 16-byte K registers per tile
  static constexpr int VR = F32 ? HDVP / 64 * 4 : Q8 ? HDVP / 64 : HDVP / 32;   // ... and V
  static constexpr int NKS = Q8 ? (8 * (HDP / 32) + 15) / 16 : 1, NVS = Q8 ? (8 * (HDVP / 32) + 15) / 16 : 1;
  static constexpr int LF = NB * (NJ * 256 + 32);           // floats of a wave's partial in LDS
  // Q in hi + lo parts of the tile layout's type; in three of the row layout's.
  static constexpr int QP = ROWS && !F32 ? 3 : 2;
  // Q's lo parts in LDS where they would spill: two column blocks of 256 dims (Q and O take half of
  // a wave's 512 registers, a step's operands a quarter; a spilled register's reload waits for every
  // page load in flight: 2.4 us per step of 32 keys), or of 96 in the row layout (half the registers)
  static constexpr bool QLDS = !F32 && !Q8 && HDP == (ROWS ? 96 : 256) && NB == 2;
  static constexpr int QF = QLDS ? (QP - 1) * NB * NC * 256 : 0;       // floats of a wave's lo parts
};

// The dims of O^T blocks GRP * gi .. of one column, times `mul`, to the row at `op`.
template <int F>
__device__ inline void store_dims(float* op, int gi, uint32_t grp, uint32_t hdv, const f4* a, float mul) {
  if constexpr (F == FR_F32) {
#pragma unroll
    for (int r = 0; r < 4; r++) {
      const uint32_t d = 64 * gi + 16 * grp + 4 * r;
      if (d < hdv) *(f4u*)(op + d) = f4u{a[0][r] * mul, a[1][r] * mul, a[2][r] * mul, a[3][r] * mul};
    }
  } else if constexpr (F >= FR_F16) {
    const uint32_t d = 32 * gi + 8 * grp;
    if (d < hdv) {
      *(f4u*)(op + d) = f4u{a[0][0] * mul, a[1][0] * mul, a[0][1] * mul, a[1][1] * mul};
      *(f4u*)(op + d + 4) = f4u{a[0][2] * mul, a[1][2] * mul, a[0][3] * mul, a[1][3] * mul};
    }
  } else {
    const f4 o = a[0] * mul;
    *(f4u*)(op + 16 * gi + 4 * grp) = f4u{o[0], o[1], o[2], o[3]};
  }
}

template <int F, int HDP, int HDVP, int NB, bool NT>
__device__ __forceinline__ void unit_wave(const PageGeom& g, const UnitGeom& u, const UnitWave* waves, const float* q,
                                          float* out, float* lds) {
  using C = Cfg<F, HDP, HDVP, NB>;
  constexpr bool BF = C::BF, Q8 = C::Q8, ROWS = C::ROWS, F32 = C::F32;
  constexpr int KT = C::KT, NC = C::NC, NJ = C::NJ, GRP = C::GRP, NCH = HDVP / 32;
  using MT = typename std::conditional<BF, b8, h8>::type;
  const uint32_t lane = threadIdx.x & 63u, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  // the wave's record: one load, a word per lane, broadcast to scalar registers
  const uint32_t W = blockDim.x >> 6, wi = blockIdx.x * W + w;
  const uint32_t word = lane < sizeof(UnitWave) / 4 ? ((const uint32_t*)(waves + wi))[lane] : 0u;
  auto fld = [&](int i) { return (uint32_t)__builtin_amdgcn_readlane((int)word, i); };
  const uint32_t wh = fld(8), wc = fld(9);
  const uint32_t n_share = (wc >> 16) & 0xffu, my_share = (wc >> 8) & 0xffu;   // waves of the unit; 0: idle
  const uint32_t hq = lane & 15u, grp = lane >> 4, G = u.group;
  const uint32_t c_off = wh >> 16, n_col = wc & 0xffu;
  const uint32_t hd = ROWS ? g.hd : (uint32_t)HDP, hdv = ROWS ? g.hdv : (uint32_t)HDVP;
  const uint32_t row0 = fld(1), kvh = wh & 0xffffu, slot = fld(5), stride = wc >> 24;
  // the columns of this lane
  uint32_t ct[NB], ch[NB];
  bool cv[NB];
#pragma unroll
  for (int x = 0; x < NB; x++) {
    const uint32_t c = 16 * x + hq;
    cv[x] = c < n_col;
    ct[x] = cv[x] ? (c + c_off) / G : 0;
    ch[x] = cv[x] ? (c + c_off) - ct[x] * G : 0;
  }
  float m[NB], lsum[NB], pup[NB];
  f4 O[NB][NJ];
  if (n_share != 0) {
    const uint32_t pos0 = fld(2), page0 = fld(3), n_pages = fld(4);
    const uint32_t page_end = page0 + n_pages, n_steps = (n_pages + KT - 1) / KT;
    uint32_t cpos[NB], clo[NB];
#pragma unroll
    for (int x = 0; x < NB; x++) {
      cpos[x] = pos0 + ct[x];
      clo[x] = (u.window > 0 && cpos[x] + 1 > u.window) ? cpos[x] + 1 - u.window : 0;
    }
    const uint32_t pos_last = pos0 + (c_off + n_col - 1) / G;
    const uint32_t lo_max = (u.window > 0 && pos_last + 1 > u.window) ? pos_last + 1 - u.window : 0;

    // ---- page addresses: block ids through scalar loads (the table does not change while the
    // kernel runs), the first step's from the record
    typedef const __attribute__((address_space(4))) int32_t cint;
    cint* tab = (cint*)(uintptr_t)(g.table + (size_t)fld(0) * g.bps);
    const uint32_t bt_mask = (1u << g.bt_shift) - 1u;
    int blk[KT];
    auto ids = [&](uint32_t step) {
#pragma unroll
      for (int kk = 0; kk < KT; kk++) {
        const uint32_t p = min(page0 + step * KT + kk, page_end - 1);
        blk[kk] = tab[(p << 4) >> g.bt_shift];
      }
    };
    blk[0] = (int)fld(6);
    if constexpr (KT > 1) blk[KT - 1] = (int)fld(7);
    // K / V head bases and tile sub-indices of a step's pages
    const uint8_t* kb[KT];
    const uint8_t* vb[KT];
    uint32_t sub[KT];
    auto bases = [&](uint32_t step) {
#pragma unroll
      for (int kk = 0; kk < KT; kk++) {
        const uint32_t p = min(page0 + step * KT + kk, page_end - 1);
        sub[kk] = ((p << 4) & bt_mask) >> 4;
        const uint8_t* b = (const uint8_t*)g.pool + (size_t)(uint32_t)blk[kk] * g.block_bytes;
        kb[kk] = b + g.k_off + (size_t)kvh * g.k_head;
        vb[kk] = b + g.v_off + (size_t)kvh * g.v_head;
      }
    };

    // ---- operand registers of one step; load_k / load_v fetch one 16-byte register of each page tile
    // of the step whose bases are set (so a register is requested again as soon as it has been used,
    // a whole step ahead of its next use)
    uint4 kr[KT][C::KR], vr[KT][C::VR], ks[KT][C::NKS], vs[KT][C::NVS];
    auto load_k = [&](int c) {
#pragma unroll
      for (int kk = 0; kk < KT; kk++) {
        const uint8_t* t = kb[kk] + sub[kk] * g.k_tile;
        if constexpr (!ROWS) {
          kr[kk][c] = load16<NT>(t + c * 1024 + lane * 16);
        } else {   // lane (key hq): 16 bytes of its row, dims past the row's end as zeros
          constexpr uint32_t ES = F32 ? 4 : 2, DL = 16 / ES, DC = 4 * DL;   // bytes, dims per lane and chunk
          const uint32_t d = c * DC + grp * DL;
          const uint4 x = load16<NT>(t + (hq * hd + (d < hd ? d : 0)) * ES);
          kr[kk][c] = d < hd ? x : make_uint4(0, 0, 0, 0);
        }
      }
    };
    auto load_v = [&](int b) {
#pragma unroll
      for (int kk = 0; kk < KT; kk++) {
        const uint8_t* t = vb[kk] + sub[kk] * g.v_tile;
        if constexpr (!ROWS) {
          vr[kk][b] = load16<NT>(t + b * 1024 + lane * 16);
        } else if constexpr (F32) {   // key 4 grp + b % 4, dims 64 (b / 4) + 4hq ..
          const uint32_t d = 64 * (b / 4) + 4 * hq;
          vr[kk][b] = load16<NT>(t + ((4 * grp + (b & 3)) * hdv + (d < hdv ? d : 0)) * 4);
        } else {   // key 4 grp + i in word i, dims 32b + 2hq, + 1
          const uint32_t d = 32 * b + 2 * hq;
          uint32_t x[4];
#pragma unroll
          for (int i = 0; i < 4; i++) x[i] = load4<NT>(t + ((4 * grp + i) * hdv + (d < hdv ? d : 0)) * 2);
          vr[kk][b] = make_uint4(x[0], x[1], x[2], x[3]);
        }
      }
    };
    auto load_ks = [&] {   // q8_0: the scales of keys 4 grp .. + 3, all chunks
#pragma unroll
      for (int kk = 0; kk < KT; kk++)
#pragma unroll
        for (int c = 0; c < C::NKS; c++)
          ks[kk][c] = *(const uint4*)(kb[kk] + g.k_scale + sub[kk] * g.k_tile_s + grp * (8 * (HDP / 32)) + c * 16);
    };
    auto load_vs = [&] {
#pragma unroll
      for (int kk = 0; kk < KT; kk++)
#pragma unroll
        for (int c = 0; c < C::NVS; c++)
          vs[kk][c] = *(const uint4*)(vb[kk] + g.v_scale + sub[kk] * g.v_tile_s + grp * (8 * NCH) + c * 16);
    };
    auto first_loads = [&] {
#pragma unroll
      for (int c = 0; c < C::KR; c++) load_k(c);
      if constexpr (Q8) load_ks();
#pragma unroll
      for (int b = 0; b < C::VR; b++) load_v(b);
      if constexpr (Q8) load_vs();
    };

    bases(0);
    first_loads();
    ids(1);
    // ---- Q of the columns as the B operand of S^T = K Q^T
    // (QP parts: hi + lo of the tile layout's type; three in the row layout, whose Q has all its 24 bits.
    // f16 rows: a column is scaled by a power of two so that its largest element is below 1, and each
    // part is the rest of the one before times 2^11, with scores of its own: 24 bits of every element
    // down to 2^-22 of the largest)
    constexpr int QP = C::QP, QR = C::QLDS ? 1 : QP, QS = F == FR_F16 ? 3 : F == FR_BF16 ? 2 : 1;
    MT qp[QR][NB][F32 ? 1 : NC];
    float* const qlo = lds + w * C::QF + lane * 4;   // QLDS: 16 bytes per lane, lo part, column block and chunk
    auto qlo_at = [&](int p, int x, int c) -> uint4* { return (uint4*)(qlo + (((p - 1) * NB + x) * NC + c) * 256); };
    f4 qf[NB][F32 ? NC : 1];
    float qscale[NB];   // score of a column in the log2 domain per unit of its product
#pragma unroll
    for (int x = 0; x < NB; x++) {
      const float* qrow = q + ((size_t)(row0 + ct[x]) * u.n_head + (size_t)kvh * G + ch[x]) * hd;
      qscale[x] = u.scale_log2;
      if constexpr (F32) {
#pragma unroll
        for (int c = 0; c < NC; c++) {
          const uint32_t d = 16 * c + 4 * grp;
          qf[x][c] = cv[x] && d < hd ? *(const f4u*)(qrow + d) : f4u{0.f, 0.f, 0.f, 0.f};
        }
      } else {
        f4 raw[NC][2];
#pragma unroll
        for (int c = 0; c < NC; c++) {
          const uint32_t d = 32 * c + 8 * grp;
          const bool on = cv[x] && (!ROWS || d < hd);
          raw[c][0] = on ? *(const f4u*)(qrow + d) : f4u{0.f, 0.f, 0.f, 0.f};
          raw[c][1] = on ? *(const f4u*)(qrow + d + 4) : f4u{0.f, 0.f, 0.f, 0.f};
        }
        if constexpr (F == FR_F16) {
          float am = 0.f;
#pragma unroll
          for (int c = 0; c < NC; c++)
#pragma unroll
            for (int i = 0; i < 8; i++) am = fmaxf(am, fabsf(raw[c][i >> 2][i & 3]));
          const int e = __builtin_amdgcn_frexp_expf(xmax_groups(am));
          qscale[x] = ldexpf(u.scale_log2, e);
#pragma unroll
          for (int c = 0; c < NC; c++)
#pragma unroll
            for (int i = 0; i < 8; i++) raw[c][i >> 2][i & 3] = ldexpf(raw[c][i >> 2][i & 3], -e);
        }
#pragma unroll
        for (int c = 0; c < NC; c++) {
          MT part[QP];
#pragma unroll
          for (int i = 0; i < 8; i++) {
            float xv = raw[c][i >> 2][i & 3];
#pragma unroll
            for (int p = 0; p < QP; p++) {
              if constexpr (BF) {
                const uint16_t hb = bf16_rne(xv);
                part[p][i] = __builtin_bit_cast(__bf16, hb);
                xv -= __uint_as_float((uint32_t)hb << 16);
              } else {
                const _Float16 hh = (_Float16)xv;
                part[p][i] = hh;
                xv -= (float)hh;
                if constexpr (QS == 3) xv *= 2048.f;
              }
            }
          }
#pragma unroll
          for (int p = 0; p < QR; p++) qp[p][x][c] = part[p];
          if constexpr (C::QLDS) {
#pragma unroll
            for (int p = 1; p < QP; p++) *qlo_at(p, x, c) = __builtin_bit_cast(uint4, part[p]);
          }
        }
      }
    }

    // pup, `checked`: as decode_item's (q8_0: weight x V scale in f16 range; a product that
    // overflowed leaves O non-finite and the unit runs again with every step's scales checked), but of a
    // column's own keys: the largest scale of the first step in which it sees one. Where the products are
    // in f32's range, 0, and the weights times 2^-8 (of every wave and piece alike): none is over 1, so no
    // weighted V leaves it. (A shift in the exponent would cost its argument the bits it grows by.)
    constexpr bool UNIT_P = F32 || F == FR_BF16;
    // 16-bit rows: O that is not finite makes the unit run again with every step's V tested.
    constexpr bool AGAIN = Q8 || (ROWS && !F32);
    bool checked = false;
    uint32_t bad_blk[NB];   // q8_0: the 32-dim blocks for which a column sees a key of a non-finite V scale
    for (;;) {
      bool unset = true;    // q8_0, uniform: some column has seen no key yet
#pragma unroll
      for (int x = 0; x < NB; x++) {
        pup[x] = Q8 ? INFINITY : UNIT_P ? 0.0f : 7.0f;
        bad_blk[x] = 0;
        m[x] = -INFINITY;
        lsum[x] = 0.f;
#pragma unroll
        for (int j = 0; j < NJ; j++) O[x][j] = f4{0.f, 0.f, 0.f, 0.f};
      }
      if (AGAIN && checked) {
        ids(0);
        bases(0);
        first_loads();
        ids(1);
      }
#pragma clang loop unroll(disable)
      for (uint32_t st = 0; st < n_steps; st++) {
        // the next step's pages (past the last step: its pages again, unused)
        bases(st + 1);
        ids(st + 2);
        if constexpr (C::QLDS) asm volatile("" ::: "memory");   // the lo parts are read again each step
        // ---- scores
        f4 s[NB][KT], s1[NB];   // f32: two chains (half the length, half the rounding)
        // rows: those of Q's first part and of the rest apart (f16: of each part). An infinite K makes the
        // first infinite, as the reference's sum, or NaN, and the rest anything, which is kept finite.
        f4 sp[QS][NB][KT];
#pragma unroll
        for (int x = 0; x < NB; x++) {
          s1[x] = f4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
          for (int kk = 0; kk < KT; kk++) {
            s[x][kk] = f4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int p = 0; p < QS; p++) sp[p][x][kk] = f4{0.f, 0.f, 0.f, 0.f};
          }
        }
#pragma unroll
        for (int c = 0; c < NC; c++) {
#pragma unroll
          for (int kk = 0; kk < KT; kk++) {
            if constexpr (F32) {
              const f4 kc = __builtin_bit_cast(f4, kr[kk][c]);
#pragma unroll
              for (int i = 0; i < 4; i++)
#pragma unroll
                for (int x = 0; x < NB; x++) {
                  if (i & 1) s1[x] = __builtin_amdgcn_mfma_f32_16x16x4f32(kc[i], qf[x][c][i], s1[x], 0, 0, 0);
                  else s[x][0] = __builtin_amdgcn_mfma_f32_16x16x4f32(kc[i], qf[x][c][i], s[x][0], 0, 0, 0);
                }
            } else if constexpr (Q8) {
              const uint32_t* wv = (const uint32_t*)&kr[kk][c >> 1];
              const int o = (c & 1) * 2;
              const h4 lo4 = i8x4_to_h4(wv[o]), hi4 = i8x4_to_h4(wv[o + 1]);
              const h8 kc = h8{lo4[0], lo4[1], lo4[2], lo4[3], hi4[0], hi4[1], hi4[2], hi4[3]};
#pragma unroll
              for (int x = 0; x < NB; x++) {
                f4 t = __builtin_amdgcn_mfma_f32_16x16x32_f16(kc, qp[0][x][c], f4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
                t = __builtin_amdgcn_mfma_f32_16x16x32_f16(kc, qp[1][x][c], t, 0, 0, 0);
#pragma unroll
                for (int r = 0; r < 4; r++) s[x][kk][r] += t[r] * scale_at<NC>(ks[kk], r, c);
              }
            } else {
              const MT kc = __builtin_bit_cast(MT, kr[kk][c]);
#pragma unroll
              for (int p = 0; p < QP; p++)
#pragma unroll
                for (int x = 0; x < NB; x++) {
                  MT qv;
                  if constexpr (C::QLDS) qv = p == 0 ? qp[0][x][c] : __builtin_bit_cast(MT, *qlo_at(p, x, c));
                  else qv = qp[p][x][c];
                  f4& to = QS > 1 ? sp[p < QS ? p : QS - 1][x][kk] : s[x][kk];
                  if constexpr (BF) to = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kc, qv, to, 0, 0, 0);
                  else to = __builtin_amdgcn_mfma_f32_16x16x32_f16(kc, qv, to, 0, 0, 0);
                }
            }
          }
          if constexpr (Q8) {
            if (c & 1) load_k(c >> 1);
          } else {
            load_k(c);
          }
        }
        if constexpr (Q8) load_ks();
        if constexpr (F32) {
#pragma unroll
          for (int x = 0; x < NB; x++) s[x][0] += s1[x];
        }
        if constexpr (QS > 1) {
          constexpr float D = QS == 3 ? 1.f / 2048.f : 1.f;
#pragma unroll
          for (int x = 0; x < NB; x++)
#pragma unroll
            for (int kk = 0; kk < KT; kk++)
#pragma unroll
              for (int r = 0; r < 4; r++) {
                const float s0 = sp[0][x][kk][r], rest = QS == 3 ? fmaf(sp[QS - 1][x][kk][r], D, sp[1][x][kk][r]) : sp[1][x][kk][r];
                s[x][kk][r] = fmaf(__builtin_amdgcn_fmed3f(rest, -1e30f, 1e30f), D, s0);   // (NaN too becomes finite)
              }
        }
        // ---- online softmax (log2 domain), masks on a range's end steps only (uniform)
        const uint32_t key0 = (page0 + st * KT) << 4;
        const bool need_mask = key0 + 16 * KT > pos0 + 1 || key0 < lo_max || page0 + (st + 1) * KT > page_end;
        float p[NB][4 * KT];
#pragma unroll
        for (int x = 0; x < NB; x++) {
#pragma unroll
          for (int kk = 0; kk < KT; kk++)
#pragma unroll
            for (int r = 0; r < 4; r++) p[x][4 * kk + r] = s[x][kk][r] * qscale[x];
          if (need_mask) {
#pragma unroll
            for (int kk = 0; kk < KT; kk++)
#pragma unroll
              for (int r = 0; r < 4; r++) {
                const uint32_t key = key0 + 16 * kk + 4 * grp + r;
                if (key > cpos[x] || key < clo[x] || key >= page_end << 4) p[x][4 * kk + r] = -INFINITY;
              }
          }
          float lm = p[x][0];
#pragma unroll
          for (int i = 1; i < 4 * KT; i++) lm = fmaxf(lm, p[x][i]);
          if (__ballot(lm > m[x] + 8.0f)) {
            const float tm = xmax_groups(lm);
            const float mn = tm > m[x] + 8.0f ? tm : m[x];
            const float alpha = mn == m[x] ? 1.f : (m[x] == -INFINITY ? 0.f : exp2_fast(m[x] - mn));
            lsum[x] *= alpha;
#pragma unroll
            for (int j = 0; j < NJ; j++) O[x][j] *= alpha;
            m[x] = mn;
          }
        }
        // whether column x sees the lane's key i (of page tile i / 4). k0: the lane's first key, from
        // lane_key(), which hides it: a test here is made again, rather than kept since the masks above.
        auto lane_key = [&] {
          uint32_t k0 = key0 + 4 * grp;
          asm volatile("" : "+v"(k0));
          return k0;
        };
        auto sees = [&](int x, int i, uint32_t k0) -> bool {
          const uint32_t key = k0 + 16 * (i >> 2) + (i & 3);
          return key <= cpos[x] && key >= clo[x] && key < page_end << 4;
        };
        if constexpr (Q8) {
          // A scale that is not finite (a value beyond 8.3e6) would make NaN of a weight of 0: on the steps
          // where a column does not see every key, such scales stay out of the products, and the columns
          // that see the key get their NaN at the end.
          auto half_at = [&](int i, int b) -> uint32_t {
            const int at = (i & 3) * NCH + b;
            const uint32_t wv = ((const uint32_t*)vs[i >> 2])[at >> 1];
            return ((at & 1) ? wv >> 16 : wv) & 0x7fffu;
          };
          if (need_mask || checked || unset) {   // uniform: a range's end steps, the first ones, or an overflow
            typedef uint16_t u16x2 __attribute__((ext_vector_type(2)));
            auto largest = [&]() -> uint32_t {
              u16x2 top = 0;
#pragma unroll
              for (int kk = 0; kk < KT; kk++)
#pragma unroll
                for (int i = 0; i < 4 * C::NVS; i++)
                  top = __builtin_elementwise_max(top, __builtin_bit_cast(u16x2, ((const uint32_t*)vs[kk])[i] & 0x7fff7fffu));
              return max(top[0], top[1]);
            };
            uint32_t mx = largest();
            if (__builtin_expect(need_mask && __ballot(mx >= 0x7c00u) != 0, 0)) {
#pragma unroll
              for (int x = 0; x < NB; x++) {
                const uint32_t k0 = lane_key();
                uint32_t hit = 0;
#pragma unroll
                for (int i = 0; i < 4 * KT; i++) {
                  uint32_t of_key = 0;
#pragma unroll
                  for (int b = 0; b < NCH; b++) {
                    uint32_t h = half_at(i, b);
                    asm volatile("" : "+v"(h));   // tested here alone: kept tests would not fit the registers
                    of_key |= h >= 0x7c00u ? 1u << b : 0u;
                  }
                  hit |= sees(x, i, k0) ? of_key : 0u;
                }
                hit |= (uint32_t)__shfl_xor((int)hit, 16);
                hit |= (uint32_t)__shfl_xor((int)hit, 32);
                bad_blk[x] |= hit;
              }
#pragma unroll
              for (int kk = 0; kk < KT; kk++)
#pragma unroll
                for (int i = 0; i < 4 * C::NVS; i++) {
                  uint32_t wv = ((uint32_t*)vs[kk])[i];
                  asm volatile("" : "+v"(wv));
                  wv &= ((wv & 0x7fffu) >= 0x7c00u ? 0u : 0xffffu) | ((wv & 0x7fff0000u) >= 0x7c000000u ? 0u : 0xffff0000u);
                  ((uint32_t*)vs[kk])[i] = wv;
                }
            }
            if (checked || unset) {   // until every column has seen a key, or every step after an overflow
              bool none = false;
#pragma unroll
              for (int x = 0; x < NB; x++) {
                if (need_mask) {
                  const uint32_t k0 = lane_key();
                  mx = 0;
#pragma unroll
                  for (int i = 0; i < 4 * KT; i++) {
                    uint32_t km = 0;
#pragma unroll
                    for (int b = 0; b < NCH; b++) km = max(km, half_at(i, b));
                    mx = max(mx, sees(x, i, k0) ? km : 0u);
                  }
                }
                const float pc = (float)(7 - __builtin_amdgcn_frexp_expf(xmax_groups(h_to_f((uint16_t)mx))));
                none |= m[x] == -INFINITY;
                if (m[x] != -INFINITY && pc < pup[x]) {   // O and lsum are zero on its first step; otherwise an exact rescale
                  const float alpha = exp2_fast(pc - pup[x]);
                  lsum[x] *= alpha;
#pragma unroll
                  for (int j = 0; j < NJ; j++) O[x][j] *= alpha;
                  pup[x] = pc;
                }
              }
              unset = __ballot(none) != 0;
            }
          }
        }
#pragma unroll
        for (int x = 0; x < NB; x++) {
          const float mref = m[x] == -INFINITY ? 0.f : m[x] - pup[x];   // every score is -inf while m is
#pragma unroll
          for (int i = 0; i < 4 * KT; i++) p[x][i] = exp2_fast(p[x][i] - mref) * (UNIT_P ? 0x1p-8f : 1.0f);
#pragma unroll
          for (int kk = 0; kk < KT; kk++)
            lsum[x] += (p[x][4 * kk] + p[x][4 * kk + 1]) + (p[x][4 * kk + 2] + p[x][4 * kk + 3]);
        }
        // A key some columns do not see may hold anything (a later row's value, or what an earlier owner
        // of the page left), and 0 * inf is not 0. Non-finite values of such a step stay out of its
        // products, and reach the columns that see them afterwards. (bf16 tiles: values beyond f16's
        // range too, as their products are taken in f16. q8_0: by its scales, above.) The 16-bit row layout
        // does so on every step of a unit that runs again: inf times the parts of a weight, of either sign,
        // is NaN. (Tested on every step of the first pass: 2,500 tokens of 32/8 heads of 80, bf16, 251 us, so
        // 244; three prompts of 900, 32 heads of 80, f16, 91 and 88.)
        bool bad_v = false;
        auto nonfinite = [](uint32_t v) -> uint32_t {   // mask of the word's non-finite values
          if constexpr (F32) return (v & 0x7f800000u) == 0x7f800000u ? ~0u : 0u;
          constexpr uint32_t E = F == FT_BF16 ? 0x4780u : BF ? 0x7f80u : 0x7c00u;   // the least non-finite magnitude
          return ((v & 0x7fffu) >= E ? 0xffffu : 0u) | ((v & 0x7fff0000u) >= E << 16 ? 0xffff0000u : 0u);
        };
        if constexpr (!Q8) {
          if (need_mask || (AGAIN && checked)) {
            // the largest magnitude (two operations a word: the step waits for it)
            typedef uint16_t u16x2 __attribute__((ext_vector_type(2)));
            typename std::conditional<F32, uint32_t, u16x2>::type top = 0;
#pragma unroll
            for (int b = 0; b < C::VR; b++) {
#pragma unroll
              for (int kk = 0; kk < KT; kk++) {
                const uint32_t* v = (const uint32_t*)&vr[kk][b];
#pragma unroll
                for (int i = 0; i < 4; i++) {
                  if constexpr (F32) top = max(top, v[i] & 0x7fffffffu);
                  else top = __builtin_elementwise_max(top, __builtin_bit_cast(u16x2, v[i] & 0x7fff7fffu));
                }
              }
            }
            bad_v = __ballot(nonfinite(__builtin_bit_cast(uint32_t, top)) != 0) != 0;
            if (__builtin_expect(bad_v, 0)) {
#pragma unroll
              for (int b = 0; b < C::VR; b++) {
#pragma unroll
                for (int kk = 0; kk < KT; kk++) {
                  uint32_t* v = (uint32_t*)&vr[kk][b];
#pragma unroll
                  for (int i = 0; i < 4; i++) {
                    uint32_t t = v[i];
                    asm("" : "+v"(t));   // tested again here, rather than every word's test kept in a register
                    v[i] = t & ~nonfinite(t);
                  }
                }
              }
            }
          }
        }
        // ---- O^T += V^T P^T (the tile layout's V registers requested again as they are used)
        if constexpr (F32) {
#pragma unroll
          for (int b = 0; b < HDVP / 64; b++) {
#pragma unroll
            for (int r = 0; r < 4; r++) {
              const f4 va = __builtin_bit_cast(f4, vr[0][4 * b + r]);
#pragma unroll
              for (int j = 0; j < 4; j++)
#pragma unroll
                for (int x = 0; x < NB; x++)
                  O[x][4 * b + j] = __builtin_amdgcn_mfma_f32_16x16x4f32(va[j], p[x][r], O[x][4 * b + j], 0, 0, 0);
              }
          }
        } else if constexpr (Q8) {
#pragma unroll
          for (int b = 0; b < NCH; b++) {
            h8 ph[NB], pl[NB];
#pragma unroll
            for (int x = 0; x < NB; x++) {
              uint32_t hw[4], lw[4];
#pragma unroll
              for (int i = 0; i < 4; i++) {
                const int kk = i >> 1, e = 2 * (i & 1);
                scaled_split(p[x][4 * kk + e], scale_h<NCH>(vs[kk], e, b), p[x][4 * kk + e + 1],
                             scale_h<NCH>(vs[kk], e + 1, b), hw[i], lw[i]);
              }
              ph[x] = __builtin_bit_cast(h8, make_uint4(hw[0], hw[1], hw[2], hw[3]));
              pl[x] = __builtin_bit_cast(h8, make_uint4(lw[0], lw[1], lw[2], lw[3]));
            }
#pragma unroll
            for (int jj = 0; jj < 2; jj++) {
              const int j = 2 * b + jj;
              const h4 v0 = i8x4_to_h4(((const uint32_t*)&vr[0][j >> 2])[j & 3]);
              const h4 v1 = i8x4_to_h4(((const uint32_t*)&vr[KT - 1][j >> 2])[j & 3]);
              const h8 va = h8{v0[0], v0[1], v0[2], v0[3], v1[0], v1[1], v1[2], v1[3]};
#pragma unroll
              for (int x = 0; x < NB; x++) {
                O[x][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(va, ph[x], O[x][j], 0, 0, 0);
                O[x][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(va, pl[x], O[x][j], 0, 0, 0);
              }
              if constexpr (!ROWS) {
                if ((j & 3) == 3) load_v(j >> 2);
              }
            }
          }
          load_vs();
        } else {
          // P as f16 hi + lo parts on V in f16 (bf16 tiles widened), or in the row layout as three parts of
          // the pages' type on V as it is
          constexpr int PP = ROWS ? 3 : 2;
          using PT = typename std::conditional<F == FR_BF16, b8, h8>::type;
          PT pp[PP][NB];
#pragma unroll
          for (int x = 0; x < NB; x++) {
            uint32_t pw[PP][4];
#pragma unroll
            for (int i = 0; i < 4; i++) {
              if constexpr (F == FR_BF16) {
                typedef float f2 __attribute__((ext_vector_type(2)));
                typedef __bf16 bf2 __attribute__((ext_vector_type(2)));
                f2 r = {p[x][2 * i], p[x][2 * i + 1]};
#pragma unroll
                for (int k = 0; k < PP; k++) {
                  const uint32_t h = __builtin_bit_cast(uint32_t, __builtin_convertvector(r, bf2));
                  pw[k][i] = h;
                  r -= f2{__uint_as_float(h << 16), __uint_as_float(h & 0xffff0000u)};
                }
              } else if constexpr (F == FR_F16) {
                typedef float f2 __attribute__((ext_vector_type(2)));
                typedef _Float16 h2 __attribute__((ext_vector_type(2)));
                f2 r = {p[x][2 * i], p[x][2 * i + 1]};
                float m1 = -1.0f;
                asm("" : "+v"(m1));   // the rest in one fma each, as in split_pair
#pragma unroll
                for (int k = 0; k < PP; k++) {
                  const h2 h = __builtin_convertvector(r, h2);
                  pw[k][i] = __builtin_bit_cast(uint32_t, h);
                  r = f2{__builtin_fmaf((float)h[0], m1, r[0]), __builtin_fmaf((float)h[1], m1, r[1])};
                }
              } else {
                split_pair(p[x][2 * i], p[x][2 * i + 1], pw[0][i], pw[1][i]);
              }
            }
#pragma unroll
            for (int k = 0; k < PP; k++) pp[k][x] = __builtin_bit_cast(PT, make_uint4(pw[k][0], pw[k][1], pw[k][2], pw[k][3]));
          }
#pragma unroll
          for (int j = 0; j < NJ; j++) {
            uint32_t wv[4];
            if constexpr (ROWS) {   // block 2b + par: the low or high halves of the keys' words
              const int b = j >> 1;
              const uint32_t sel = (j & 1) ? 0x07060302u : 0x05040100u;
              const uint4 x0 = vr[0][b], x1 = vr[KT - 1][b];
              wv[0] = __builtin_amdgcn_perm(x0.y, x0.x, sel);
              wv[1] = __builtin_amdgcn_perm(x0.w, x0.z, sel);
              wv[2] = __builtin_amdgcn_perm(x1.y, x1.x, sel);
              wv[3] = __builtin_amdgcn_perm(x1.w, x1.z, sel);
            } else {
              const uint32_t* w0 = (const uint32_t*)&vr[0][j >> 1];
              const uint32_t* w1 = (const uint32_t*)&vr[KT - 1][j >> 1];
              const int o = (j & 1) * 2;
              wv[0] = w0[o];
              wv[1] = w0[o + 1];
              wv[2] = w1[o];
              wv[3] = w1[o + 1];
            }
            if constexpr (F == FT_BF16) {
#pragma unroll
              for (int i = 0; i < 4; i++) wv[i] = bf2_h2(wv[i]);
            }
            const PT va = __builtin_bit_cast(PT, make_uint4(wv[0], wv[1], wv[2], wv[3]));
#pragma unroll
            for (int k = 0; k < PP; k++)
#pragma unroll
              for (int x = 0; x < NB; x++) {
                if constexpr (F == FR_BF16) O[x][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(va, pp[k][x], O[x][j], 0, 0, 0);
                else O[x][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(va, pp[k][x], O[x][j], 0, 0, 0);
              }
            if constexpr (!ROWS) {
              if (j & 1) load_v(j >> 1);
            }
          }
        }
        if constexpr (!Q8) {
          if (__builtin_expect(bad_v, 0)) {
            // how many NaN, +inf and -inf values of a dim a column sees: products of 0 / 1 operands
            ids(st);
            bases(st);
#pragma unroll
            for (int b = 0; b < C::VR; b++) load_v(b);
            const uint32_t k0 = lane_key();
            float see[NB][F32 ? 4 : 1];
            h8 seeh[NB];
#pragma unroll
            for (int x = 0; x < NB; x++)
#pragma unroll
              for (int i = 0; i < 4 * KT; i++) {
                const bool on = sees(x, i, k0);
                if constexpr (F32) see[x][i] = on ? 1.0f : 0.0f;
                else seeh[x][i] = on ? (_Float16)1.0f : (_Float16)0.0f;
              }
            auto kind = [](float v, int k) -> float {   // k: 0 +inf, 1 -inf, 2 NaN
              constexpr float TOP = F == FT_BF16 ? 65536.f : INFINITY;
              return (k == 2 ? v != v : k == 0 ? v >= TOP : v <= -TOP) ? 1.0f : 0.0f;
            };
#pragma unroll
            for (int j = 0; j < NJ; j++) {
              __builtin_amdgcn_sched_barrier(0);   // one block at a time: no registers to spare
#pragma unroll
              for (int k = 0; k < 3; k++) {
                f4 cnt[NB];
#pragma unroll
                for (int x = 0; x < NB; x++) cnt[x] = f4{0.f, 0.f, 0.f, 0.f};
                if constexpr (F32) {
#pragma unroll
                  for (int r = 0; r < 4; r++) {
                    const f4 v = __builtin_bit_cast(f4, vr[0][4 * (j / 4) + r]);
#pragma unroll
                    for (int x = 0; x < NB; x++)
                      cnt[x] = __builtin_amdgcn_mfma_f32_16x16x4f32(kind(v[j & 3], k), see[x][r], cnt[x], 0, 0, 0);
                  }
                } else {
                  h8 a;
#pragma unroll
                  for (int i = 0; i < 8; i++) {
                    // rows: a word per key, its halves two blocks; tiles: a half per key
                    const uint32_t* vw = (const uint32_t*)&vr[i >> 2][j >> 1];
                    const uint32_t w32 = ROWS ? vw[i & 3] : vw[2 * (j & 1) + ((i & 3) >> 1)];
                    const uint16_t w16 = (uint16_t)(((ROWS ? j : i) & 1) ? w32 >> 16 : w32);
                    a[i] = (_Float16)kind(BF ? __uint_as_float((uint32_t)w16 << 16) : h_to_f(w16), k);
                  }
#pragma unroll
                  for (int x = 0; x < NB; x++) cnt[x] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a, seeh[x], cnt[x], 0, 0, 0);
                }
                constexpr uint32_t ADD[3] = {0x7f800000u, 0xff800000u, 0x7fc00000u};
#pragma unroll
                for (int x = 0; x < NB; x++)
#pragma unroll
                  for (int r = 0; r < 4; r++) O[x][j][r] += cnt[x][r] > 0.f ? __uint_as_float(ADD[k]) : 0.f;
              }
            }
            ids(st + 1);
            bases(st + 1);
            ids(st + 2);
            if constexpr (!ROWS && !F32) {   // (K again too: its registers are free in between)
#pragma unroll
              for (int c = 0; c < C::KR; c++) load_k(c);
#pragma unroll
              for (int b = 0; b < C::VR; b++) load_v(b);
            }
          }
          if constexpr (ROWS) {
#pragma unroll
            for (int b = 0; b < C::VR; b++) load_v(b);
          }
        }
      }
      if constexpr (!AGAIN) break;
      if (checked) break;
      bool bad = false;
#pragma unroll
      for (int x = 0; x < NB; x++) {
        float z = 0.f;
#pragma unroll
        for (int j = 0; j < NJ; j++) z += (O[x][j][0] + O[x][j][1]) + (O[x][j][2] + O[x][j][3]);
        bad |= cv[x] && !__builtin_isfinite(z);
      }
      if (!__ballot(bad)) break;
      checked = true;
    }
    if constexpr (Q8) {
#pragma unroll
      for (int x = 0; x < NB; x++) {
        if (!__builtin_expect(__ballot(bad_blk[x] != 0) != 0, 0)) continue;
#pragma unroll
        for (int j = 0; j < NJ; j++)
          if (bad_blk[x] >> (j >> 1) & 1u) O[x][j] = f4{NAN, NAN, NAN, NAN};
      }
    }
#pragma unroll
    for (int x = 0; x < NB; x++) lsum[x] = xsum_groups(lsum[x]);
  }

  // a column's output row, or its partial's (a piece of a longer unit)
  auto row_at = [&](int x) -> float* {
    if (slot == NO_SLOT) return out + ((size_t)(row0 + ct[x]) * u.n_head + (size_t)kvh * G + ch[x]) * hdv;
    return u.part + ((size_t)(slot + ct[x] * stride) * u.ng + ch[x]) * (hdv + 4);
  };
  if (n_share == 1) {
#pragma unroll
    for (int x = 0; x < NB; x++) {
      if (!cv[x]) continue;
      float* op = row_at(x);
      const float mul = slot == NO_SLOT ? 1.0f / lsum[x] : 1.0f;
#pragma unroll
      for (int gi = 0; gi < NJ / GRP; gi++) store_dims<F>(op, gi, grp, hdv, &O[x][gi * GRP], mul);
      if (slot != NO_SLOT && grp == 0) {
        op[hdv] = m[x] - pup[x];   // the reference the weights were taken against
        op[hdv + 1] = lsum[x];
      }
    }
  }
  if (!u.shared) return;   // uniform over the launch: no unit of it is shared between waves
  // ---- a shared unit: each wave's partial in LDS, then wave s of n folds the unit's partials for
  // the O^T block groups s, s + n, .. of all columns (forward.rs:772-806's log-sum-exp merge)
  if constexpr (C::QLDS) __syncthreads();   // the partials take the place of the waves' Q
  if (n_share > 1) {
    float* lw = lds + w * C::LF;
#pragma unroll
    for (int x = 0; x < NB; x++) {
      float* lx = lw + x * (NJ * 256 + 32);
#pragma unroll
      for (int j = 0; j < NJ; j++) *(f4*)(lx + (j * 64 + lane) * 4) = O[x][j];
      if (grp == 0) {
        lx[NJ * 256 + hq] = m[x] - pup[x];
        lx[NJ * 256 + 16 + hq] = lsum[x];
      }
    }
  }
  __syncthreads();   // every wave of the workgroup, with a unit or not
  if (n_share <= 1 || my_share >= n_share || my_share > w || w - my_share + n_share > W) return;
  const float* l0 = lds + (w - my_share) * C::LF;   // the unit's first wave
#pragma unroll
  for (int x = 0; x < NB; x++) {
    const float* lx = l0 + x * (NJ * 256 + 32);
    float M = -INFINITY;
    for (uint32_t k = 0; k < n_share; k++) M = fmaxf(M, lx[k * C::LF + NJ * 256 + hq]);
    float c[UNIT_MAX_WAVES], L = 0.f;
#pragma unroll
    for (int k = 0; k < UNIT_MAX_WAVES; k++) {
      c[k] = 0.f;
      if ((uint32_t)k < n_share) {
        const float ms = lx[k * C::LF + NJ * 256 + hq];
        c[k] = ms == -INFINITY ? 0.f : exp2_fast(ms - M);
        L = fmaf(c[k], lx[k * C::LF + NJ * 256 + 16 + hq], L);
      }
    }
    if (!cv[x]) continue;
    float* op = row_at(x);
    const float mul = slot != NO_SLOT ? 1.0f : L > 0.f ? 1.0f / L : 0.f;
    for (uint32_t gi = my_share; gi < (uint32_t)(NJ / GRP); gi += n_share) {
      f4 acc[GRP];
#pragma unroll
      for (int i = 0; i < GRP; i++) {
        acc[i] = f4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int k = 0; k < UNIT_MAX_WAVES; k++)
          if ((uint32_t)k < n_share) acc[i] += c[k] * *(const f4*)(lx + k * C::LF + ((gi * GRP + i) * 64 + lane) * 4);
      }
      store_dims<F>(op, (int)gi, grp, hdv, acc, mul);
    }
    if (slot != NO_SLOT && my_share == 0 && grp == 0) {
      op[hdv] = M;
      op[hdv + 1] = L;
    }
  }
}

// Waves per SIMD the register allocator must allow: one where Q, O and a step's operands need more than
// half the file, four (two workgroups per CU) where they fit a quarter. (Two instances spill, 8 registers
// to scratch memory each: f16 tiles of hd 256 and f16 rows of 96 dims, both with two column blocks.)
template <int F, int HDP, int HDVP, int NB>
constexpr int unit_wpe() {
  using C = Cfg<F, HDP, HDVP, NB>;
  constexpr int regs = C::KT * 4 * (C::KR + C::VR + (C::Q8 ? C::NKS + C::NVS : 0)) +
                       NB * (C::NC * (C::F32 ? 4 : C::ROWS ? 12 : 8) + C::NJ * 4);
  return regs > 190 ? 1 : NB == 1 && !C::ROWS && regs < 96 ? 4 : 2;
}
template <int F, int HDP, int HDVP, int NB>
constexpr int unit_w() { return unit_wpe<F, HDP, HDVP, NB>() == 1 ? 4 : UNIT_MAX_WAVES; }

template <int F, int HDP, int HDVP, int NB>
__global__ __launch_bounds__((64 * unit_w<F, HDP, HDVP, NB>()))
__attribute__((amdgpu_waves_per_eu(unit_wpe<F, HDP, HDVP, NB>())))
void unit_kernel(PageGeom g, UnitGeom u, const UnitWave* waves, const float* q, float* out, MergeCopy mc) {
  extern __shared__ __attribute__((aligned(16))) float unit_lds[];
  copy_merges(mc, blockIdx.x, gridDim.x);
  unit_wave<F, HDP, HDVP, NB, NB == 1 && !Cfg<F, HDP, HDVP, NB>::ROWS>(g, u, waves, q, out, unit_lds);
}

// f(format, hdp, hdvp) of the instance that takes a geometry; false: none does.
template <typename Fn>
bool with_instance(uint32_t kv_type, uint32_t hd, uint32_t hdv, uint32_t layout, Fn&& f) {
#define LMH_U(FMT, A, B)                                                                             \
  {                                                                                                  \
    f(std::integral_constant<int, FMT>{}, std::integral_constant<int, A>{}, std::integral_constant<int, B>{}); \
    return true;                                                                                     \
  }
  if (kv_type == KV_F32) {
    if (hd % 4 || hdv % 4) return false;
    const uint32_t d = std::max(hd, hdv);
    if (d <= 64) LMH_U(FR_F32, 64, 64)
    if (d <= 128) LMH_U(FR_F32, 128, 128)
    if (d <= 256) LMH_U(FR_F32, 256, 256)
    return false;
  }
  if (layout == LAYOUT_ROWS) {
    if (kv_type == KV_Q8 || hd % 8 || hdv % 8) return false;
    const uint32_t d = std::max(hd, hdv);
#define LMH_UR(A)                                         \
  if (d <= A) {                                           \
    if (kv_type == KV_F16) LMH_U(FR_F16, A, A)            \
    LMH_U(FR_BF16, A, A)                                  \
  }
    LMH_UR(64) LMH_UR(96) LMH_UR(128) LMH_UR(192) LMH_UR(256)
#undef LMH_UR
    return false;
  }
#define LMH_UT(A, B)                                      \
  if (hd == A && hdv == B) {                              \
    if (kv_type == KV_F16) LMH_U(FT_F16, A, B)            \
    if (kv_type == KV_BF16) LMH_U(FT_BF16, A, B)          \
  }
  LMH_UT(32, 32) LMH_UT(64, 64) LMH_UT(96, 96) LMH_UT(128, 128) LMH_UT(192, 192) LMH_UT(256, 256) LMH_UT(192, 128)
#undef LMH_UT
#define LMH_UQ(A) \
  if (kv_type == KV_Q8 && hd == A && hdv == A) LMH_U(FT_Q8, A, A)
  LMH_UQ(64) LMH_UQ(128) LMH_UQ(192) LMH_UQ(256)
#undef LMH_UQ
#undef LMH_U
  return false;
}

// Two column blocks where they fit the register file (past it, q8_0 pages at hd 256 spilled 270
// registers into scratch memory: 5 rows x 6,000 keys 53 us against 28 with one block). In the row layout,
// whose Q and P have three parts, two blocks of 128 dims leave one wave per SIMD: two prompts of 1,500
// tokens, 12/4 heads of 112, f16 99.1 us against 77.3 with one block; bf16, 32/8 heads of 104, 2,500 tokens
// 397 and 312; of 96 dims, with Q's lo parts in LDS, two blocks are faster (two of 300 tokens, 32 heads of
// 80, f16: 30.8 and 33.0).
template <int F, int HDP, int HDVP>
constexpr bool two_blocks() {
  return F == FT_F16 || F == FT_BF16 || (F == FR_F32 ? HDP < 256 : F >= FR_F16 ? HDP < 128 : HDP < 192);
}

}  // namespace

uint32_t unit_waves(uint32_t kv_type, uint32_t hd, uint32_t hdv, uint32_t layout, uint32_t nb) {
  uint32_t w = 0;
  with_instance(kv_type, hd, hdv, layout, [&](auto f, auto a, auto b) {
    constexpr int F = decltype(f)::value, A = decltype(a)::value, B = decltype(b)::value;
    if (nb == 1) w = unit_w<F, A, B, 1>();
    else if (two_blocks<F, A, B>()) w = unit_w<F, A, B, 2>();
  });
  return w;
}

// Asked of the runtime once per kernel and device (a query takes ~10 us, which each new cache's first call
// paid); a query that fails is asked again by the next call.
uint32_t unit_waves_per_cu(int32_t device, uint32_t kv_type, uint32_t hd, uint32_t hdv, uint32_t layout, uint32_t nb) {
  constexpr int DEVICES = 16;   // devices beyond these are asked each time
  uint32_t n = 4;
  auto ask = [&](auto f, auto a, auto b, auto nbt) {   // without LDS, 4-wave workgroups: what the registers allow
    constexpr int F = decltype(f)::value, A = decltype(a)::value, B = decltype(b)::value, NB = decltype(nbt)::value;
    if constexpr (NB == 1 || two_blocks<F, A, B>()) {
      static std::atomic<uint32_t> known[DEVICES];
      const bool keep = device >= 0 && device < DEVICES;
      if (keep && (n = known[device].load(std::memory_order_relaxed)) != 0) return;
      int blocks = 0;
      const bool ok = hipSetDevice(device) == hipSuccess &&
                      hipOccupancyMaxActiveBlocksPerMultiprocessor(&blocks, unit_kernel<F, A, B, NB>, 256, 0) == hipSuccess && blocks > 0;
      n = ok ? 4 * (uint32_t)blocks : 4;
      if (ok && keep) known[device].store(n, std::memory_order_relaxed);
    }
  };
  with_instance(kv_type, hd, hdv, layout, [&](auto f, auto a, auto b) {
    if (nb == 1) ask(f, a, b, std::integral_constant<int, 1>{});
    else ask(f, a, b, std::integral_constant<int, 2>{});
  });
  return n;
}

hipError_t launch_units(const PageGeom& g, const UnitGeom& u, uint32_t nb, uint32_t w, const UnitWave* waves, uint32_t n_wg,
                        const float* q, float* out, const MergeCopy& mc, hipStream_t s, const LaunchEv& ev) {
  if (n_wg == 0) return hipSuccess;
  hipError_t e = hipErrorInvalidValue;
  auto go = [&](auto f, auto a, auto b, auto nbt) {
    constexpr int F = decltype(f)::value, A = decltype(a)::value, B = decltype(b)::value, NB = decltype(nbt)::value;
    if constexpr (NB == 1 || two_blocks<F, A, B>()) {
      if (w == 0 || w > (uint32_t)unit_w<F, A, B, NB>()) return;
      const uint32_t lds = w * 4 * std::max(Cfg<F, A, B, NB>::QF, u.shared ? Cfg<F, A, B, NB>::LF : 0);
      LMH_LAUNCH(ev, (unit_kernel<F, A, B, NB>), dim3(n_wg), dim3(64 * w), lds, s, g, u, waves, q, out, mc);
      e = hipGetLastError();
    }
  };
  with_instance(g.kv_type, g.hd, g.hdv, g.layout, [&](auto f, auto a, auto b) {
    if (nb == 1) go(f, a, b, std::integral_constant<int, 1>{});
    else if (nb == 2) go(f, a, b, std::integral_constant<int, 2>{});
  });
  return e;
}

}  // namespace lmh
