// cx_gemm.hip — multi-row k-quant contraction on int8 MFMA (gfx950):
// dst[a][r] = fused dot of weight row r with activation row a, for m
// activation rows at once (ops::matmul_auto with m > 1, src/ops.rs:1056-1093;
// BASELINE config 4 and prefill-shaped calls).
//
// Q4_K and Q5_K, whose 32-value sub-blocks are exactly the K = 32 of
// v_mfma_i32_16x16x32_i8: one MFMA gives the exact integer sums E_j of one
// sub-block for a 16 (weight rows) x 16 (activation rows) tile. Each lane
// applies the scalar kernel's f32 term to its four results,
//   term_j = xe_j * (d*sc_j * E_j - dmin*mn_j * xs_j),
// and the terms of one output are added sub-block after sub-block from 0
// (src/kernels/scalar.rs:132-217), so every output equals the per-row dot bit
// for bit and a row of a batch equals the row alone (src/ops.rs:1364-1393).
// The reference's own m >= 24 path (src/ops.rs:607-829) adds in another order
// within 1e-4 of the maximum (src/ops.rs:1518-1561); keeping the per-row
// order makes a batched prefill bit-identical to token-by-token.
//
// The per-sub-block f32 term (6 VALU operations per output and sub-block in
// k_gemm, 5 in k_gemm_w) is most of this path's work, not the MFMA: a 16x16x32
// MFMA is followed by 24 or 20 VALU instructions per lane.
//
// MFMA lane layout (checked on the device): A 16x32 — lane l holds row
// l%16, k = 8(l/16)..+8 as 8 bytes; B 32x16 — lane l holds column l%16,
// same k range; C 16x16 — lane l element i is row 4(l/16)+i, column l%16.
// Activations are the A operand and weights the B operand, so a lane's four
// results share one weight row (l%16): the lane decodes that row's d, dmin
// and 6-bit scales itself, from one 16-byte read of the block header, and
// reads xe, xs of its four activation rows as float4s.
//
// k_gemm's workgroup: 4 or 8 waves over a TW x MT tile (TW = 16 RW weight rows, MT =
// 16 AW WA activation rows); the waves split rows (RW), activation tiles (AW)
// and, when a tile is too small to give every wave its own rows, the eight
// sub-blocks of each super-block (KS). With KS > 1 the waves write their
// terms to LDS and each thread adds the terms of its outputs in sub-block
// order. The k loop walks super-blocks through an S-stage ring of
// direct-to-LDS loads: a stage is the tile's weight bytes of one super-block,
// the MT activation rows' 256 bytes, and their xe and xs. Every wave issues
// D loads per stage, so the wait for a stage is a fixed vmcnt; loads beyond
// the stage's bytes reload a valid address into the stage's tail.

#include "cx_act.h"
#include "cx_internal.h"

namespace {

typedef int v4i __attribute__((ext_vector_type(4)));

// The B operand (weights): positions 8g..8g+7 of sub-block j of a block in
// LDS as 8 i8 values. load() reads the raw bytes, operand() unpacks them.
template <int T> struct GQ;
template <> struct GQ<CX_Q4_K> {
  static constexpr int BPB = 144;
  struct Raw {
    uint2 q;  // qs bytes 32(j/2) + 8g .. +8 (low nibbles: even j, high: odd j)
  };
  __device__ static Raw load(const uint8_t* blk, int j, int g) {
    return Raw{*reinterpret_cast<const uint2*>(blk + 16 + 32 * (j >> 1) + 8 * g)};
  }
  __device__ static long operand(const Raw& r, int j) {
    const uint32_t sh = 4 * (j & 1);
    const uint32_t lo = (r.q.x >> sh) & 0x0F0F0F0Fu, hi = (r.q.y >> sh) & 0x0F0F0F0Fu;
    return (long)(((uint64_t)hi << 32) | lo);
  }
};
template <> struct GQ<CX_Q5_K> {
  static constexpr int BPB = 176;
  struct Raw {
    uint2 q;  // qs bytes 32(j/2) + 8g .. +8
    uint2 h;  // qh bytes 8g .. +8: bit j is the fifth bit of sub-block j
  };
  __device__ static Raw load(const uint8_t* blk, int j, int g) {
    return Raw{*reinterpret_cast<const uint2*>(blk + 48 + 32 * (j >> 1) + 8 * g),
               *reinterpret_cast<const uint2*>(blk + 16 + 8 * g)};
  }
  __device__ static long operand(const Raw& r, int j) {
    const uint32_t sh = 4 * (j & 1);
    const uint32_t lo = ((r.q.x >> sh) & 0x0F0F0F0Fu) | (((r.h.x >> j) & 0x01010101u) << 4);
    const uint32_t hi = ((r.q.y >> sh) & 0x0F0F0F0Fu) | (((r.h.y >> j) & 0x01010101u) << 4);
    return (long)(((uint64_t)hi << 32) | lo);
  }
};

// quant::escala_y_minimo (src/quant.rs:108-117) of sub-block j from the 12
// scale bytes q[0..12) held as the words y (q0..q3), z (q4..q7), w (q8..q11)
__device__ inline void scale_min(uint32_t y, uint32_t z, uint32_t w, int j, uint32_t& sc,
                                 uint32_t& mn) {
  if (j < 4) {
    const int s = 8 * j;
    sc = (y >> s) & 63;
    mn = (z >> s) & 63;
  } else {
    const int s = 8 * (j - 4);
    sc = ((w >> s) & 0xF) | (((y >> (s + 6)) & 3) << 4);
    mn = ((w >> (s + 4)) & 0xF) | (((z >> (s + 6)) & 3) << 4);
  }
}

template <bool B>
struct Bool {
  static constexpr bool value = B;
};

struct GemmParams {
  const uint8_t* w;     // n rows x row_bytes, GGUF raw
  const int8_t* xq;     // m_pad rows x k (rows >= m are zero)
  const float* xexs;    // per sub-block J: xe of the m_pad rows, then their xs
  float* dst;           // m x n
  uint32_t n, k, m, m_pad, nb, row_bytes, row_tiles, act_tiles;
  const float* lhs;     // m x k f32: the quantizer's input (not read by the kernels)
  uint8_t* scratch;     // where xq and xexs are carved (not read by the kernels)
  // with nseg > 1 the n rows are nseg matrices of one type and
  // width, rows [sr[i], sr[i + 1]) matrix i with weights sw[i] and its own
  // output sd[i] (m x (sr[i + 1] - sr[i])); every sr[i] is a multiple of
  // the tile's rows, so a tile lies in one matrix
  uint32_t nseg, sr[CX_GEMM_SEGS + 1];
  const uint8_t* sw[CX_GEMM_SEGS];
  float* sd[CX_GEMM_SEGS];
  // per matrix (index 0 without segments): a bias added to
  // every output row (dst = acc + bias[r]), and with accum the output added
  // to what dst holds (dst = dst + (acc [+ bias])), f32 adds as written
  const float* sbias[CX_GEMM_SEGS];
  uint32_t accum;
};

template <int T, int RW, int AW, int WA, int KS, int NSB>
struct Shape {
  static constexpr int NW = RW * AW * KS;  // waves
  static_assert(NW == 4 || NW == 8, "4 or 8 waves");
  static constexpr int BPB = GQ<T>::BPB;
  static constexpr int TW = 16 * RW, MT = 16 * AW * WA;
  static constexpr int NU = 8 * NSB;  // sub-blocks per stage
  static constexpr int NJ = NU / KS;  // sub-blocks per wave per stage
  static_assert(NU % KS == 0 && (NJ >= 8 ? NJ % 8 == 0 : 8 % NJ == 0), "even split");
  static constexpr int NBW = NJ >= 8 ? NJ / 8 : 1;  // blocks a wave touches per stage
  static constexpr int RB = NSB * BPB;              // LDS bytes per weight row
  // LDS bytes per activation row: 68 mod 64 words, so the 8-byte A operand
  // reads of 16 rows x 2 lane groups (one half-wave pass) hit 64 distinct banks
  static constexpr int XS = NSB * 256 + 16;
  static constexpr int WB = TW * RB, XB = MT * XS, EB = NU * MT * 8;
  static constexpr int WCH = WB / 16, XCH = XB / 16, ECH = EB / 16;
  static constexpr int SLOT = NW * 1024;  // bytes of one load of every wave
  static constexpr int STAGE = (WB + XB + EB + SLOT - 1) / SLOT * SLOT;
  static constexpr int D = STAGE / SLOT;  // loads per wave per stage
  static constexpr int TERMS = KS > 1 ? 2 * NU * TW * MT * 4 : 0;
  static constexpr size_t lds(int S) { return (size_t)S * STAGE + TERMS; }
};

// wait until at most `ahead` stages (D loads each) of this wave are in flight
template <int D, int N>
__device__ inline void wait_stages(int ahead) {
  if constexpr (N == 0) {
    cx_wait_vm<0>();
  } else {
    if (ahead >= N)
      cx_wait_vm<N * D>();
    else
      wait_stages<D, N - 1>(ahead);
  }
}

template <int T, int RW, int AW, int WA, int KS, int NSB, int S>
__global__ __launch_bounds__(64 * RW * AW * KS) void k_gemm(GemmParams P) {
  using SH = Shape<T, RW, AW, WA, KS, NSB>;
  constexpr int BPB = SH::BPB, TW = SH::TW, MT = SH::MT, NU = SH::NU, NJ = SH::NJ;
  constexpr int D = SH::D, NW = SH::NW, RB = SH::RB, XS = SH::XS;
  static_assert(S >= 2 && (S - 2) * D <= 63, "stage waits must fit vmcnt");
  extern __shared__ __align__(16) uint8_t lds[];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);  // wave-uniform
  const int g = lane >> 4, c16 = lane & 15;
  const int ks = wave % KS, aw = (wave / KS) % AW, rw = wave / (KS * AW);

  // blockIdx -> (row tile, activation tile): the activation tiles of one row
  // tile share blockIdx % 8, i.e. one XCD and its L2, which then holds the
  // row tile's weights for all of them
  const uint32_t b = blockIdx.x, A = P.act_tiles;
  const uint32_t rt = b / (8 * A) * 8 + b % 8, at = b / 8 % A;
  if (rt >= P.row_tiles) return;  // whole workgroup, before any load or barrier
  const uint32_t a0 = at * MT;
  // the tile's matrix: its weights W, rows N, output DST; r0 its first row there
  const uint8_t* W = P.w;
  float* DST = P.dst;
  const float* BIAS = P.sbias[0];
  uint32_t N = P.n, r0 = rt * TW;
  if (P.nseg > 1) {
    uint32_t i = 0;
    while (i + 1 < P.nseg && r0 >= P.sr[i + 1]) i++;
    W = P.sw[i];
    DST = P.sd[i];
    BIAS = P.sbias[i];
    N = P.sr[i + 1] - P.sr[i];
    r0 -= P.sr[i];
  }
  auto put = [&](uint32_t a, uint32_t r, float v) {  // output (a, r) of the tile's matrix
    float* d = DST + (size_t)a * N + r;
    if (BIAS) v = v + BIAS[r];
    if (P.accum) v = *d + v;
    *d = v;
  };

  // this lane's load sources: slot s carries chunk NW*64 s + 64 wave + lane
  // of a stage, i.e. LDS bytes [16 c, 16 c + 16) of the stage; the chunk
  // belongs to super-block bis[s] of the stage (a stage past the last
  // super-block loads a valid dummy address instead)
  const uint8_t* src[D];
  uint32_t inc[D];
  uint32_t bis[D];
#pragma unroll
  for (int s = 0; s < D; s++) {
    const uint32_t c = NW * 64 * s + 64 * wave + lane;
    src[s] = W;
    inc[s] = 0;
    bis[s] = 0;
    if (c < (uint32_t)SH::WCH) {
      const uint32_t r = c / (RB / 16), part = c % (RB / 16);
      const uint32_t row = r0 + r < N ? r0 + r : N - 1;  // past the end: a valid row
      src[s] = W + (size_t)row * P.row_bytes + 16 * part;
      inc[s] = RB;
      bis[s] = part / (BPB / 16);
    } else if (c < (uint32_t)(SH::WCH + SH::XCH)) {
      const uint32_t cc = c - SH::WCH, a = cc / (XS / 16);
      uint32_t part = cc % (XS / 16);
      if (part == 16 * NSB) part = 0;  // the row's pad chunk
      src[s] = reinterpret_cast<const uint8_t*>(P.xq) + (size_t)(a0 + a) * P.k + 16 * part;
      inc[s] = 256 * NSB;
      bis[s] = part / 16;
    } else if (c < (uint32_t)(SH::WCH + SH::XCH + SH::ECH)) {
      // sub-block u of the stage: MT xe, then MT xs
      const uint32_t cc = c - SH::WCH - SH::XCH, u = cc / (MT / 2);
      const uint32_t h = cc % (MT / 2) / (MT / 4), part = cc % (MT / 4);
      src[s] = reinterpret_cast<const uint8_t*>(P.xexs + (size_t)(2 * u + h) * P.m_pad + a0) +
               16 * part;
      inc[s] = NU * 2 * P.m_pad * 4;
      bis[s] = u / 8;
    }
  }
  const uint32_t nb = P.nb, nst = (nb + NSB - 1) / NSB;
  auto issue = [&](uint32_t sb) {
    uint8_t* base = lds + (sb % S) * SH::STAGE + 1024 * wave;
#pragma unroll
    for (int s = 0; s < D; s++) {
      const uint8_t* p = sb * NSB + bis[s] < nb ? src[s] + (size_t)sb * inc[s] : W;
      cx_dma16_async(p, base + SH::SLOT * s);
    }
  };

  float* terms = reinterpret_cast<float*>(lds + S * SH::STAGE);  // [2][NU][TW][MT]
  constexpr int NQ = TW * MT;  // outputs of the tile
  constexpr int PP = KS > 1 ? (NQ + 64 * NW - 1) / (64 * NW) : 1;  // outputs chained per thread
  float acc[WA][4];
  float cacc[PP];
#pragma unroll
  for (int t = 0; t < WA; t++)
#pragma unroll
    for (int i = 0; i < 4; i++) acc[t][i] = 0.0f;
#pragma unroll
  for (int i = 0; i < PP; i++) cacc[i] = 0.0f;
  // thread `tid` adds, sub-block by sub-block, the terms of outputs
  // q = tid + 64 NW i (weight row q / MT, activation row q % MT) over the
  // first `nu` sub-blocks of a stage
  auto chain = [&](const float* tb, uint32_t nu) {
#pragma unroll
    for (int i = 0; i < PP; i++) {
      const int q = tid + 64 * NW * i;
      if (NQ % (64 * NW) == 0 || q < NQ) {
        float v[NU];  // every load first (all in the buffer), then the adds in order
#pragma unroll
        for (int u = 0; u < NU; u++) v[u] = tb[u * NQ + q];
#pragma unroll
        for (int u = 0; u < NU; u++)
          if ((uint32_t)u < nu) cacc[i] += v[u];
      }
    }
  };
  auto valid_sub = [&](uint32_t sb) { return 8 * (nb - sb * NSB < NSB ? nb - sb * NSB : NSB); };

  for (uint32_t st = 0; st < (uint32_t)(S - 1) && st < nst; st++) issue(st);
  for (uint32_t sb = 0; sb < nst; sb++) {
    const uint32_t last = sb + S - 2 < nst - 1 ? sb + S - 2 : nst - 1;
    wait_stages<D, S - 2>((int)(last - sb));
    cx_wait_lds();  // this wave's reads of the previous stage are done
    cx_barrier();   // stage sb is in LDS for every wave; slot (sb - 1) % S is free
    if (sb + S - 1 < nst) issue(sb + S - 1);
    const uint8_t* cur = lds + (sb % S) * SH::STAGE;
    const uint8_t* X = cur + SH::WB;
    const float* E = reinterpret_cast<const float*>(cur + SH::WB + SH::XB);
    float* tb = terms + (sb & 1) * (NU * NQ);
    const int ub = ks * NJ;  // this wave's first sub-block of the stage
#pragma unroll
    for (int bb = 0; bb < SH::NBW; bb++) {
      const int bi = (ub >> 3) + bb;  // super-block of the stage
      if (sb * NSB + bi >= nb) break;
      // this lane's weight row: d, dmin and the 12 scale bytes in one read
      const uint8_t* wrow = cur + (16 * rw + c16) * RB + bi * BPB;
      const uint4 hd = *reinterpret_cast<const uint4*>(wrow);
      constexpr int NJB = NJ < 8 ? NJ : 8;  // sub-blocks of this block for this wave
      // every operand of the block first when few (one round of LDS latency),
      // else per sub-block
      constexpr bool BATCH = NJB * WA <= 8;
      typename GQ<T>::Raw wr[BATCH ? NJB : 1];
      long axb[BATCH ? NJB : 1][WA];
      float4 xeb[BATCH ? NJB : 1][WA], xsb[BATCH ? NJB : 1][WA];
      auto fetch = [&](int slot, int u, int j) {
        wr[slot] = GQ<T>::load(wrow, j, g);
#pragma unroll
        for (int t = 0; t < WA; t++) {
          const int ab = 16 * (aw * WA + t);  // first activation row of the MFMA tile
          axb[slot][t] = *reinterpret_cast<const long*>(X + (ab + c16) * XS + 32 * u + 8 * g);
          xeb[slot][t] = *reinterpret_cast<const float4*>(E + u * 2 * MT + ab + 4 * g);
          xsb[slot][t] = *reinterpret_cast<const float4*>(E + u * 2 * MT + MT + ab + 4 * g);
        }
      };
      if constexpr (BATCH) {
#pragma unroll
        for (int jj = 0; jj < NJB; jj++) fetch(jj, ub + 8 * bb + jj, (ub + 8 * bb + jj) & 7);
      }
      const float d = cx_h2f(hd.x & 0xFFFFu), dmin = cx_h2f(hd.x >> 16);
#pragma unroll
      for (int jj = 0; jj < NJB; jj++) {
        const int u = ub + 8 * bb + jj, j = u & 7, sl = BATCH ? jj : 0;
        if constexpr (!BATCH) fetch(0, u, j);
        uint32_t sc, mn;
        scale_min(hd.y, hd.z, hd.w, j, sc, mn);
        const float ds = d * (float)sc, dm = dmin * (float)mn;
        const long bw = GQ<T>::operand(wr[sl], j);
#pragma unroll
        for (int t = 0; t < WA; t++) {
          const int ab = 16 * (aw * WA + t);
          v4i e = {0, 0, 0, 0};
          e = __builtin_amdgcn_mfma_i32_16x16x32_i8(axb[sl][t], bw, e, 0, 0, 0);
          const float4 xe = xeb[sl][t], xs = xsb[sl][t];
          const float xev[4] = {xe.x, xe.y, xe.z, xe.w}, xsv[4] = {xs.x, xs.y, xs.z, xs.w};
          float tv[4];
#pragma unroll
          for (int i = 0; i < 4; i++) tv[i] = xev[i] * (ds * (float)e[i] - dm * xsv[i]);
          if constexpr (KS == 1) {
#pragma unroll
            for (int i = 0; i < 4; i++) acc[t][i] += tv[i];
          } else {
            *reinterpret_cast<float4*>(tb + (u * TW + 16 * rw + c16) * MT + ab + 4 * g) =
                make_float4(tv[0], tv[1], tv[2], tv[3]);
          }
        }
      }
    }
    if constexpr (KS > 1) {
      if (sb > 0) chain(terms + ((sb - 1) & 1) * (NU * NQ), valid_sub(sb - 1));
    }
  }

  if constexpr (KS > 1) {
    cx_wait_lds();
    cx_barrier();
    chain(terms + ((nst - 1) & 1) * (NU * NQ), valid_sub(nst - 1));
#pragma unroll
    for (int i = 0; i < PP; i++) {
      const int q = tid + 64 * NW * i;
      const uint32_t a = a0 + q % MT, r = r0 + q / MT;
      if (q < NQ && a < P.m && r < N) put(a, r, cacc[i]);
    }
  } else {
    // lane: weight row r, activation rows 4g .. 4g+3 of each MFMA tile
    const uint32_t r = r0 + 16 * rw + c16;
    if (r < N) {
#pragma unroll
      for (int t = 0; t < WA; t++)
#pragma unroll
        for (int i = 0; i < 4; i++) {
          const uint32_t a = a0 + 16 * (aw * WA + t) + 4 * g + i;
          if (a < P.m) put(a, r, acc[t][i]);
        }
    }
  }
}

// ------------------------------------------------ Q4_K/Q5_K, many rows
// The same products and terms with the weights in registers. A workgroup of 4
// waves takes 64 weight rows x 16 WA activation rows, wave w the 16 rows from
// 16 w: no two waves share a weight byte, so each lane loads its share straight
// into registers, a super-block ahead; only the activation rows and their xe, xs
// pass through LDS for the workgroup (double-buffered direct-to-LDS loads, one
// super-block a stage, one barrier).
//
// Lane layout as k_gemm: lane l holds weight row l % 16 and the results of
// activation rows 4 (l / 16) .. + 4 of each tile. The four lanes of a row decode
// two sub-blocks' scales each, once a super-block, and pass them around by
// ds_bpermute (two reads a sub-block): every lane decoding all eight cost ~12
// operations a sub-block, half of them (bit-field extract, convert) at half rate.
//
// In LDS an activation row is its 256 bytes in 16-byte chunks, chunk c at c ^
// (row % 16): the 16 rows that a read takes at once fall on all banks.
//
// E as f32 costs no conversion: the MFMA starts from the bits of E_BASE = 1.5 *
// 2^23, so its result read as f32 is E_BASE + E exactly (|E| < 2^22), and
// fma(ds, E_BASE + E, -ds * E_BASE) is ds * E rounded once, the reference's
// product: ds = d * sc has at most 17 significant bits, so -ds * E_BASE is exact.
// Where a d of the wave is not finite the product is formed the plain way. (A
// zero may come out with the other sign; it is added to a sum that starts at
// +0.0, which no zero changes.)
//
// What bounds it, by counters (11008 x 2048, m = 512, 74 us at 2.24 GHz): 35.4 M
// VALU instructions, 34.6 k a SIMD, of which the terms are 27.5 k. At the 2.5 to 3.1
// clocks an instruction that two to three waves a SIMD reach they are 39 to 48 us. Of
// the waves' time 32% waits to issue and 24% for loads, LDS and the barrier of every
// super-block, and the 1376 workgroups are 1.8 rounds of 768. 2048 x 11008: 39.0 M
// instructions in 88 us, 512 workgroups, two waves a SIMD.
// Measured beside it and dropped: weights as the A operand with the scales in an
// LDS table (no better), 12 and 16 waves a workgroup (slower: the barrier), scales
// by DPP or in SGPRs (conversions and scalar loads cost what they save).
constexpr float E_BASE = 12582912.0f;
constexpr int E_BASE_BITS = 0x4B400000;

// one lane's share of a super-block of its weight row: the header, the nibbles
// of its k group in the four sub-block pairs, and (Q5_K) its fifth bits
template <int T> struct WRegs {
  uint4 hd;
  uint2 q[4], h;
  __device__ void load(const uint8_t* blk, int G) {
    hd = *reinterpret_cast<const uint4*>(blk);
    if constexpr (T == CX_Q5_K) h = *reinterpret_cast<const uint2*>(blk + 16 + 8 * G);
#pragma unroll
    for (int p = 0; p < 4; p++)
      q[p] = *reinterpret_cast<const uint2*>(blk + GQ<T>::BPB - 128 + 32 * p + 8 * G);
  }
  // every word has arrived here (the compiler's waits for them go before this)
  __device__ void arrived() {
    asm volatile("" : "+v"(hd.x), "+v"(hd.y), "+v"(hd.z), "+v"(hd.w));
    pin();
  }
  __device__ void pin() {
    asm volatile("" : "+v"(q[0].x), "+v"(q[0].y), "+v"(q[1].x), "+v"(q[1].y), "+v"(q[2].x),
                 "+v"(q[2].y), "+v"(q[3].x), "+v"(q[3].y));
    if constexpr (T == CX_Q5_K) asm volatile("" : "+v"(h.x), "+v"(h.y));
  }
  __device__ long operand(int j) const {
    uint32_t lo = (q[j >> 1].x >> (4 * (j & 1))) & 0x0F0F0F0Fu;
    uint32_t hi = (q[j >> 1].y >> (4 * (j & 1))) & 0x0F0F0F0Fu;
    if constexpr (T == CX_Q5_K) {
      lo |= ((h.x >> j) & 0x01010101u) << 4;
      hi |= ((h.y >> j) & 0x01010101u) << 4;
    }
    return (long)(((uint64_t)hi << 32) | lo);
  }
};

template <int NW, int WA> struct WShape {
  static constexpr int TW = 16 * NW, MT = 16 * WA;
  static constexpr int LX = 4 * WA, LE = WA;     // 1 KiB loads a stage: activation rows; xe, xs
  static constexpr int STAGE = (LX + LE) * 1024;  // bytes
  static constexpr size_t lds = 2 * STAGE;
};

// the sums of one lane: weight row wr, activation rows 4 G .. + 3 of each tile from a0
template <int WA>
__device__ inline void store_rows(const GemmParams& P, const float (&acc)[WA][4], float* dst,
                                  const float* bias, uint32_t n, uint32_t wr, uint32_t a0, int G) {
  if (wr >= n) return;
  const float bv = bias ? bias[wr] : 0.0f;
#pragma unroll
  for (int t = 0; t < WA; t++)
#pragma unroll
    for (int i = 0; i < 4; i++) {
      const uint32_t a = a0 + 16 * t + 4 * G + i;
      if (a >= P.m) continue;
      float* o = dst + (size_t)a * n + wr;
      float v = acc[t][i];
      if (bias) v = v + bv;
      if (P.accum) v = *o + v;
      *o = v;
    }
}

template <int T, int NW, int WA, int OCC>
__global__ __launch_bounds__(64 * NW, OCC) void k_gemm_w(GemmParams P) {
  static_assert(NW % 4 == 0, "a wave's loads are rows of one remainder mod 16");
  using SH = WShape<NW, WA>;
  constexpr int TW = SH::TW, MT = SH::MT, LX = SH::LX, LE = SH::LE;
  extern __shared__ __align__(16) uint8_t lds[];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int col = lane % 16, G = lane / 16;
  // blockIdx -> (row tile, activation tile), as k_gemm
  const uint32_t b = blockIdx.x, A = P.act_tiles;
  const uint32_t rt = b / (8 * A) * 8 + b % 8, at = b / 8 % A;
  if (rt >= P.row_tiles) return;  // whole workgroup, before any load or barrier
  const uint32_t a0 = at * MT;
  const uint8_t* W = P.w;
  float* DST = P.dst;
  const float* BIAS = P.sbias[0];
  uint32_t N = P.n, r0 = rt * TW;
  // (constant indices: a struct argument indexed by a variable goes to scratch)
#pragma unroll
  for (uint32_t i = 0; i < CX_GEMM_SEGS; i++)
    if (i < P.nseg && rt * TW >= P.sr[i]) {
      W = P.sw[i];
      DST = P.sd[i];
      BIAS = P.sbias[i];
      N = P.sr[i + 1] - P.sr[i];
      r0 = rt * TW - P.sr[i];
    }
  r0 += 16 * wave;  // the wave's first row
  const uint32_t wr = r0 + col;  // this lane's weight row (past the end: a valid row)
  const uint8_t* wrow = W + (size_t)(wr < N ? wr : N - 1) * P.row_bytes;
  // Load l of a stage (l = wave, wave + NW, ...) fills its chunks 64 l + lane: for
  // l < LX the activation rows 4 l .. + 4 (a wave's l agree mod 4, so the lanes'
  // offsets are the same in each and the row a uniform base), then xe and xs, of
  // which a wave has one load at most.
  const uint32_t xoff = (lane / 16) * P.k + 16 * ((lane % 16) ^ ((4 * wave + lane / 16) % 16));
  const uint32_t el = (wave + NW - LX % NW) % NW, ec = 64 * el + lane;
  const uint32_t eoff =  // sub-block ec / (MT / 2): MT xe, then MT xs
      (2 * (ec / (MT / 2)) + ec % (MT / 2) / (MT / 4)) * P.m_pad * 4 + 16 * (ec % (MT / 4));
  const int8_t* xbase = P.xq + (size_t)a0 * P.k;
  const float* ebase = P.xexs + a0;
  auto issue = [&](uint32_t sb) {
    uint8_t* l = lds + (sb & 1) * SH::STAGE;
#pragma unroll
    for (int u = 0; u < (LX + NW - 1) / NW; u++) {
      const int i = wave + NW * u;
      if (i < LX) cx_dma16_async_s(xbase + (size_t)(4 * i) * P.k + 256 * sb, xoff, l + 1024 * i);
    }
    if (el < (uint32_t)LE)
      cx_dma16_async_s(ebase + (size_t)sb * 16 * P.m_pad, eoff, l + 1024 * (LX + el));
  };
  float acc[WA][4];
#pragma unroll
  for (int t = 0; t < WA; t++)
#pragma unroll
    for (int i = 0; i < 4; i++) acc[t][i] = 0.0f;
  const uint32_t nb = P.nb;
  WRegs<T> wn;
  wn.load(wrow, G);
  issue(0);
#pragma unroll 1
  for (uint32_t sb = 0; sb < nb; sb++) {
    cx_wait_vm<0>();  // this wave's part of stage sb, and its weights
    cx_wait_lds();
    cx_barrier();     // every wave's part; stage sb - 1 is read
    WRegs<T> w = wn;
    // before the next loads are issued: a wait that the compiler placed later
    // would count the direct-to-LDS loads, which it does not know of, as done
    w.arrived();
    if (sb + 1 < nb) issue(sb + 1);
    wn.load(wrow + (size_t)(sb + 1 < nb ? sb + 1 : sb) * GQ<T>::BPB, G);
    const uint8_t* X = lds + (sb & 1) * SH::STAGE;
    const float* E = reinterpret_cast<const float*>(X + 256 * MT) + 4 * G;
    // sub-blocks 2G and 2G + 1 of this lane's row: for G < 2 the 6-bit fields
    // themselves, else 4 bits of the third scale word and 2 of the others
    const bool wild = __any((w.hd.x & 0x7C00u) == 0x7C00u);
    float ds2[2], dm2[2];
    {
      const float d = cx_h2f(w.hd.x & 0xFFFFu), dmin = cx_h2f(w.hd.x >> 16);
      const uint32_t sh = 16 * (G & 1);
      const uint32_t y = w.hd.y >> sh, z = w.hd.z >> sh, v = w.hd.w >> sh;
#pragma unroll
      for (int u = 0; u < 2; u++) {
        const uint32_t yb = (y >> (8 * u)) & 0xFFu, zb = (z >> (8 * u)) & 0xFFu,
                       vb = (v >> (8 * u)) & 0xFFu;
        const uint32_t sc = G < 2 ? yb & 63u : (vb & 15u) | ((yb >> 6) << 4);
        const uint32_t mn = G < 2 ? zb & 63u : (vb >> 4) | ((zb >> 6) << 4);
        ds2[u] = d * (float)sc;
        dm2[u] = dmin * (float)mn;
      }
    }
    auto block = [&](auto fin) {
      constexpr bool FIN = decltype(fin)::value;
      // the activation operand: row 16 t + col, chunk (2 j + G / 2) ^ col. (ax is
      // made opaque so that the eight addresses are formed where they are used,
      // one operation each, and not kept in eight registers.)
      uint32_t ax = 256 * col + 16 * ((G / 2) ^ col) + 8 * (G & 1);
      asm volatile("" : "+v"(ax));
      auto act = [&](int j, int t) {
        return *reinterpret_cast<const long*>(X + (ax ^ (32 * j)) + 4096 * t);
      };
      auto from = [&](int j, const float (&v)[2]) {  // this row's value for sub-block j
        return __int_as_float(
            __builtin_amdgcn_ds_bpermute(4 * col + 64 * (j / 2), __float_as_int(v[j & 1])));
      };
      v4i base;
#pragma unroll
      for (int i = 0; i < 4; i++) base[i] = FIN ? E_BASE_BITS : 0;
      v4i e[WA];
      float dsj[2], dmj[2];
      dsj[0] = from(0, ds2);
      dmj[0] = from(0, dm2);
      // xe, xs of a tile's four activation rows, the next tile's read under this
      // one's terms
      float4 xeb[2], xsb[2];
      auto scales = [&](int j, int t, int buf) {
        const float* p = E + 2 * MT * j + 16 * t;
        xeb[buf] = *reinterpret_cast<const float4*>(p);
        xsb[buf] = *reinterpret_cast<const float4*>(p + MT);
      };
      scales(0, 0, 0);
      {
        const long bw = w.operand(0);
#pragma unroll
        for (int t = 0; t < WA; t++)
          e[t] = __builtin_amdgcn_mfma_i32_16x16x32_i8(act(0, t), bw, base, 0, 0, 0);
      }
#pragma unroll
      for (int j = 0; j < 8; j++) {
        w.pin();  // (left alone, the compiler unpacks all eight sub-blocks first)
        const float ds = dsj[j & 1], dm = dmj[j & 1], nds = -(ds * E_BASE);
        long bw = 0;
        if (j + 1 < 8) {
          dsj[(j + 1) & 1] = from(j + 1, ds2);
          dmj[(j + 1) & 1] = from(j + 1, dm2);
          bw = w.operand(j + 1);
        }
#pragma unroll
        for (int t = 0; t < WA; t++) {
          const int st = j * WA + t, buf = st & 1;
          long xa = 0;
          if (j + 1 < 8) xa = act(j + 1, t);
          if (st + 1 < 8 * WA) scales((st + 1) / WA, (st + 1) % WA, buf ^ 1);
          __builtin_amdgcn_sched_barrier(0);
          const float4 xe = xeb[buf], xs = xsb[buf];
          const float xev[4] = {xe.x, xe.y, xe.z, xe.w}, xsv[4] = {xs.x, xs.y, xs.z, xs.w};
          // the four terms side by side (left alone, the compiler forms one after
          // the other, each operation waiting for the one before)
          float se[4], dx[4];
#pragma unroll
          for (int i = 0; i < 4; i++)
            se[i] = FIN ? fmaf(ds, __int_as_float(e[t][i]), nds) : ds * (float)e[t][i];
#pragma unroll
          for (int i = 0; i < 4; i++) dx[i] = dm * xsv[i];
          __builtin_amdgcn_sched_barrier(0);
#pragma unroll
          for (int i = 0; i < 4; i++) se[i] = se[i] - dx[i];
          __builtin_amdgcn_sched_barrier(0);
#pragma unroll
          for (int i = 0; i < 4; i++) se[i] = xev[i] * se[i];
          __builtin_amdgcn_sched_barrier(0);
#pragma unroll
          for (int i = 0; i < 4; i++) acc[t][i] += se[i];
          // the next sub-block's sums run under the other tiles' terms
          if (j + 1 < 8) e[t] = __builtin_amdgcn_mfma_i32_16x16x32_i8(xa, bw, base, 0, 0, 0);
          __builtin_amdgcn_sched_barrier(0);
        }
      }
    };
    if (wild)
      block(Bool<false>{});
    else
      block(Bool<true>{});
  }
  store_rows<WA>(P, acc, DST, BIAS, N, wr, a0, G);
}

// ---------------------------- the other formats (Q2_K, Q3_K, Q6_K, Q8_0, Q5_0)
// The same layout and pipeline as k_gemm_w for the formats whose blocks sit at any
// even offset of a row (84, 110 and 210 bytes of 256 values; 34 and 22 of 32):
// XQ<T> holds one lane's share of a stage of 256 values of its weight row.
//
// A 32-value group is one v_mfma_i32_16x16x32_i8 for the 32-value formats (the
// reference's buffer path, ops::matmul_i8_directo, src/ops.rs:310-414; its m >= 24
// blocked path adds in another order, src/ops.rs:726). The others have two 16-value
// sub-blocks in it: lanes of groups 0 and 1 hold the first, 2 and 3 the second, and
// two MFMAs, each with the other half's weight bytes zero, give the two sums.
//
// The offsets that Q6_K (32), Q3_K (4) and Q5_0 (16) take off a value are taken off
// its byte: the MFMA then sums E' = E - 32 xs itself, the exact integer that the
// per-row kernel's (float)E - 32.0f * xs is, and the term is (xe * scale) * E' as
// there. The MFMA starts from the bits of E_BASE, so that E' as f32 is one
// subtraction at full rate, not a conversion at half (|E'| < 2^22: exact).
//
// With few rows the round trip of a stage bounds it: Q6_K 2048 x 11008, m = 77, is
// 160 workgroups, one wave a SIMD, and 43 stages of 1.8 us (77.7 us), 11 clocks an
// instruction; by m = 8 nothing is shorter.
typedef uint32_t u32_at2 __attribute__((aligned(2)));  // a word at any even address
__device__ inline uint32_t at2(const uint8_t* p) { return *reinterpret_cast<const u32_at2*>(p); }
__device__ inline uint2 at2x2(const uint8_t* p) {
  struct __attribute__((packed, aligned(2))) Pair {
    uint32_t x, y;
  };
  const Pair v = *reinterpret_cast<const Pair*>(p);
  return make_uint2(v.x, v.y);
}
__device__ inline void pin(uint2& v) { asm volatile("" : "+v"(v.x), "+v"(v.y)); }
__device__ inline uint2 both(uint2 v, uint32_t sh, uint32_t mask) {
  return make_uint2((v.x >> sh) & mask, (v.y >> sh) & mask);
}
// every byte less `off`, as i8 (bytes <= 127 - (128 - off) before)
__device__ inline uint2 less(uint2 v, uint32_t off) {
  const uint32_t a = 0x01010101u * (128 - off);
  return make_uint2((v.x + a) ^ 0x80808080u, (v.y + a) ^ 0x80808080u);
}

// Members: load(), this lane's words of the stage at p, of which `left` blocks are
// in the row (words of a block past them are left as they are, no term uses them: a
// row of 32 to 400 values waited for eight blocks' loads, and for the last stage's
// twice. Q5_0 4864 x 96, m = 64, 14.3 -> 11.0 us, x 288 19.3 -> 14.5; Q8_0 4864 x
// 896, m = 512, 31.0 -> 29.5); pin(); scales(), the factors of
// this lane's sub-blocks PL G .. + PL (MIN: and their minima); operand(), its bytes
// 8 G .. + 8 of the stage's 32-value group gg.
template <int T> struct XQ;

// Q2_K, 84 B: scales(16: low nibble scale, high nibble min) qs(64) d dmin;
// value (qs[32(gg/4) + i] >> 2(gg%4)) & 3 (src/kernels/q2k.rs:41-69)
template <> struct XQ<CX_Q2_K> {
  static constexpr int BPB = 84, SUB = 16, NB = 1, PL = 4;
  static constexpr bool MIN = true;
  uint2 q[2];
  uint32_t sc, d;
  __device__ void load(const uint8_t* p, int G, uint32_t) {
    q[0] = at2x2(p + 16 + 8 * G);
    q[1] = at2x2(p + 48 + 8 * G);
    sc = at2(p + 4 * G);
    d = at2(p + 80);
  }
  __device__ void pin() { ::pin(q[0]), ::pin(q[1]); }
  __device__ void arrived() {
    asm volatile("" : "+v"(sc), "+v"(d));
    pin();
  }
  __device__ void scales(int, float (&s)[PL], float (&m)[PL]) const {
    const float df = cx_h2f(d & 0xFFFFu), dm = cx_h2f(d >> 16);
#pragma unroll
    for (int i = 0; i < PL; i++) {
      s[i] = df * (float)((sc >> (8 * i)) & 15u);
      m[i] = dm * (float)((sc >> (8 * i + 4)) & 15u);
    }
  }
  __device__ uint2 operand(int gg, int) const { return both(q[gg / 4], 2 * (gg % 4), 0x03030303u); }
};

// Q3_K, 110 B: hmask(32) qs(64) scales(12) d; value (q + 4) =
// ((qs[32(gg/4) + i] >> 2(gg%4)) & 3) | ((hmask[i] >> gg) & 1) << 2
// (src/kernels/scalar.rs:236-275), scales as quant::escalas_q3k (src/quant.rs:87-106)
template <> struct XQ<CX_Q3_K> {
  static constexpr int BPB = 110, SUB = 16, NB = 1, PL = 4;
  static constexpr bool MIN = false;
  uint2 q[2], h;
  uint32_t s0, s1, s2, d;
  __device__ void load(const uint8_t* p, int G, uint32_t) {
    h = at2x2(p + 8 * G);
    q[0] = at2x2(p + 32 + 8 * G);
    q[1] = at2x2(p + 64 + 8 * G);
    s0 = at2(p + 96);
    s1 = at2(p + 100);
    s2 = at2(p + 104);
    d = *reinterpret_cast<const uint16_t*>(p + 108);
  }
  __device__ void pin() { ::pin(q[0]), ::pin(q[1]), ::pin(h); }
  __device__ void arrived() {
    asm volatile("" : "+v"(s0), "+v"(s1), "+v"(s2), "+v"(d));
    pin();
  }
  __device__ void scales(int G, float (&s)[PL], float (&)[PL]) const {
    const uint32_t low = ((G & 1 ? s1 : s0) >> (G & 2 ? 4 : 0)) & 0x0F0F0F0Fu;
    const uint32_t w = low | (((s2 >> (2 * G)) & 0x03030303u) << 4);
    const float df = cx_h2f(d);
#pragma unroll
    for (int i = 0; i < PL; i++) s[i] = df * ((float)((w >> (8 * i)) & 63u) - 32.0f);
  }
  __device__ uint2 operand(int gg, int) const {
    const uint2 a = both(q[gg / 4], 2 * (gg % 4), 0x03030303u), b = both(h, gg, 0x01010101u);
    return less(make_uint2(a.x | (b.x << 2), a.y | (b.y << 2)), 4);
  }
};

// Q6_K, 210 B: ql(128) qh(64) scales(16, i8) d. Group gg: half = gg/4, gi = gg%4;
// value = nibble | ((qh[32 half + i] >> 2gi) & 3) << 4, the nibble low (gi < 2) or
// high of ql[64 half + 32 (gi%2) + i] (src/kernels/scalar.rs:294-324)
template <> struct XQ<CX_Q6_K> {
  static constexpr int BPB = 210, SUB = 16, NB = 1, PL = 4;
  static constexpr bool MIN = false;
  uint2 q[4], h[2];
  uint32_t sc, d;
  __device__ void load(const uint8_t* p, int G, uint32_t) {
#pragma unroll
    for (int i = 0; i < 4; i++) q[i] = at2x2(p + 32 * i + 8 * G);
    h[0] = at2x2(p + 128 + 8 * G);
    h[1] = at2x2(p + 160 + 8 * G);
    sc = at2(p + 192 + 4 * G);
    d = *reinterpret_cast<const uint16_t*>(p + 208);
  }
  __device__ void pin() {
    ::pin(q[0]), ::pin(q[1]), ::pin(q[2]), ::pin(q[3]), ::pin(h[0]), ::pin(h[1]);
  }
  __device__ void arrived() {
    asm volatile("" : "+v"(sc), "+v"(d));
    pin();
  }
  __device__ void scales(int, float (&s)[PL], float (&)[PL]) const {
    const float df = cx_h2f(d);
#pragma unroll
    for (int i = 0; i < PL; i++) s[i] = df * (float)(int8_t)(uint8_t)(sc >> (8 * i));
  }
  __device__ uint2 operand(int gg, int) const {
    const int half = gg / 4, gi = gg % 4;
    const uint2 a = both(q[2 * half + gi % 2], gi < 2 ? 0 : 4, 0x0F0F0F0Fu);
    const uint2 b = both(h[half], 2 * gi, 0x03030303u);
    return less(make_uint2(a.x | (b.x << 4), a.y | (b.y << 4)), 32);
  }
};

// Q8_0, 34 B: d, 32 signed bytes
template <> struct XQ<CX_Q8_0> {
  static constexpr int BPB = 34, SUB = 32, NB = 8, PL = 2;
  static constexpr bool MIN = false;
  uint2 q[8];
  uint32_t d[2];
  __device__ void load(const uint8_t* p, int G, uint32_t left) {
#pragma unroll
    for (uint32_t i = 0; i < 8; i++)
      if (i < left) q[i] = at2x2(p + i * BPB + 2 + 8 * G);
#pragma unroll
    for (uint32_t i = 0; i < 2; i++)
      d[i] = *reinterpret_cast<const uint16_t*>(p + min(2 * G + i, left - 1) * BPB);
  }
  __device__ void pin() {
#pragma unroll
    for (int i = 0; i < 8; i++) ::pin(q[i]);
  }
  __device__ void arrived() {
    asm volatile("" : "+v"(d[0]), "+v"(d[1]));
    pin();
  }
  __device__ void scales(int, float (&s)[PL], float (&)[PL]) const {
    s[0] = cx_h2f(d[0]);
    s[1] = cx_h2f(d[1]);
  }
  __device__ uint2 operand(int gg, int) const { return q[gg]; }
};

// Q5_0, 22 B: d, the fifth bits of the 32 values, their nibbles: value i < 16 is
// the low nibble of byte i, value 16 + i the high one
template <> struct XQ<CX_Q5_0> {
  static constexpr int BPB = 22, SUB = 32, NB = 8, PL = 2;
  static constexpr bool MIN = false;
  uint2 q[8];
  uint32_t h[8], d[2];
  __device__ void load(const uint8_t* p, int G, uint32_t left) {
#pragma unroll
    for (uint32_t i = 0; i < 8; i++) {
      if (i < left) {
        const uint8_t* b = p + i * BPB;
        q[i] = at2x2(b + 6 + 8 * (G & 1));
        h[i] = b[2 + G];
      }
    }
#pragma unroll
    for (uint32_t i = 0; i < 2; i++)
      d[i] = *reinterpret_cast<const uint16_t*>(p + min(2 * G + i, left - 1) * BPB);
  }
  __device__ void pin() {
#pragma unroll
    for (int i = 0; i < 8; i++) {
      ::pin(q[i]);
      asm volatile("" : "+v"(h[i]));
    }
  }
  __device__ void arrived() {
    asm volatile("" : "+v"(d[0]), "+v"(d[1]));
    pin();
  }
  __device__ void scales(int, float (&s)[PL], float (&)[PL]) const {
    s[0] = cx_h2f(d[0]);
    s[1] = cx_h2f(d[1]);
  }
  // bit i of a nibble to bit 4 of byte i
  __device__ static uint32_t spread4(uint32_t t) {
    return ((t & 1u) << 4) | ((t & 2u) << 11) | ((t & 4u) << 18) | ((t & 8u) << 25);
  }
  __device__ uint2 operand(int gg, int G) const {
    const uint2 a = both(q[gg], G < 2 ? 0 : 4, 0x0F0F0F0Fu);
    return less(make_uint2(a.x | spread4(h[gg] & 15u), a.y | spread4(h[gg] >> 4)), 16);
  }
};

template <int T, int WA> struct XShape {
  static constexpr int TW = 64, MT = 16 * WA;
  static constexpr int NS = 256 / XQ<T>::SUB;      // sub-blocks a stage
  static constexpr int PARTS = XQ<T>::MIN ? 2 : 1;  // xe, with minima xs too
  static constexpr int ROW = PARTS * MT / 4;        // 16-byte chunks of a sub-block's xe (, xs)
  // 1 KiB loads a stage: the activation rows; their xe (, xs)
  static constexpr int LX = 4 * WA, LE = (NS * ROW + 63) / 64;
  static constexpr int STAGE = (LX + LE) * 1024;
  static constexpr size_t lds = 2 * STAGE;
};

template <int T, int WA, int OCC>
__global__ __launch_bounds__(256, OCC) void k_gemm_x(GemmParams P) {
  using Q = XQ<T>;
  using SH = XShape<T, WA>;
  constexpr int TW = SH::TW, MT = SH::MT, LX = SH::LX, LE = SH::LE, NS = SH::NS, NH = 32 / Q::SUB;
  extern __shared__ __align__(16) uint8_t lds[];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int col = lane % 16, G = lane / 16;
  // blockIdx -> (row tile, activation tile), as k_gemm
  const uint32_t b = blockIdx.x, A = P.act_tiles;
  const uint32_t rt = b / (8 * A) * 8 + b % 8, at = b / 8 % A;
  if (rt >= P.row_tiles) return;  // whole workgroup, before any load or barrier
  const uint32_t a0 = at * MT;
  const uint8_t* W = P.w;
  float* DST = P.dst;
  const float* BIAS = P.sbias[0];
  uint32_t N = P.n, r0 = rt * TW;
#pragma unroll
  for (uint32_t i = 0; i < CX_GEMM_SEGS; i++)
    if (i < P.nseg && rt * TW >= P.sr[i]) {
      W = P.sw[i];
      DST = P.sd[i];
      BIAS = P.sbias[i];
      N = P.sr[i + 1] - P.sr[i];
      r0 = rt * TW - P.sr[i];
    }
  r0 += 16 * wave;
  const uint32_t wr = r0 + col;  // this lane's weight row (past the end: a valid row)
  const uint8_t* wrow = W + (size_t)(wr < N ? wr : N - 1) * P.row_bytes;
  // the loads of a stage as k_gemm_w's; in the row's last stage a chunk past k, and
  // past the last sub-block, reads the stage's first one again (no term uses it)
  const uint32_t xr = (lane / 16) * P.k, xc = 16 * ((lane % 16) ^ ((4 * wave + lane / 16) % 16));
  const int8_t* xbase = P.xq + (size_t)a0 * P.k;
  const float* ebase = P.xexs + a0;
  const uint32_t nst = (P.nb + Q::NB - 1) / Q::NB;
  auto issue = [&](uint32_t sb) {
    uint8_t* l = lds + (sb & 1) * SH::STAGE;
    const uint32_t left = P.k - 256 * sb;  // values
    const uint32_t xoff = xr + (Q::NB == 1 || xc < left ? xc : 0u);
#pragma unroll
    for (int u = 0; u < LX / 4; u++) {
      const int i = wave + 4 * u;
      cx_dma16_async_s(xbase + (size_t)(4 * i) * P.k + 256 * sb, xoff, l + 1024 * i);
    }
#pragma unroll
    for (int u = 0; u < (LE + 3) / 4; u++) {
      const int i = wave + 4 * u;
      if (i < LE) {
        const uint32_t c = 64 * i + lane;  // chunk: sub-block c / ROW
        uint32_t s = c / SH::ROW;
        if (s >= (uint32_t)NS || (Q::NB > 1 && Q::SUB * s >= left)) s = 0;
        const uint32_t eoff =
            (2 * s + c % SH::ROW / (MT / 4)) * P.m_pad * 4 + 16 * (c % (MT / 4));
        cx_dma16_async_s(ebase + (size_t)sb * (2 * NS) * P.m_pad, eoff, l + 1024 * (LX + i));
      }
    }
  };
  float acc[WA][4];
#pragma unroll
  for (int t = 0; t < WA; t++)
#pragma unroll
    for (int i = 0; i < 4; i++) acc[t][i] = 0.0f;
  Q wn{};  // (words that a short row never loads)
  wn.load(wrow, G, P.nb);
  issue(0);
  const uint32_t half = G < 2 ? ~0u : 0u;  // (16-value sub-blocks)
#pragma unroll 1
  for (uint32_t sb = 0; sb < nst; sb++) {
    cx_wait_vm<0>();  // this wave's part of stage sb, and its weights
    cx_wait_lds();
    cx_barrier();     // every wave's part; stage sb - 1 is read
    Q w = wn;
    w.arrived();  // before the next loads are issued, as in k_gemm_w
    if (sb + 1 < nst) {
      issue(sb + 1);
      wn.load(wrow + (size_t)(sb + 1) * (Q::NB * Q::BPB), G, P.nb - (sb + 1) * Q::NB);
    }
    const uint8_t* X = lds + (sb & 1) * SH::STAGE;
    const float* E = reinterpret_cast<const float*>(X + 256 * MT) + 4 * G;
    const uint32_t ng = Q::NB == 1 ? 8 : P.nb - sb * Q::NB;  // 32-value groups (more than 8: 8)
    float sv[Q::PL], mv[Q::PL];
    w.scales(G, sv, mv);
    uint32_t ax = 256 * col + 16 * ((G / 2) ^ col) + 8 * (G & 1);
    asm volatile("" : "+v"(ax));
    auto act = [&](int gg, int t) {
      return *reinterpret_cast<const long*>(X + (ax ^ (32 * gg)) + 4096 * t);
    };
    auto from = [&](int j, const float (&v)[Q::PL]) {  // this row's value for sub-block j
      return __int_as_float(__builtin_amdgcn_ds_bpermute(4 * col + 64 * (j / Q::PL),
                                                         __float_as_int(v[j % Q::PL])));
    };
    // the weight operands of group gg: one, or one per sub-block
    auto operands = [&](int gg, long (&o)[NH]) {
      const uint2 v = w.operand(gg, G);
      if constexpr (NH == 1) {
        o[0] = (long)(((uint64_t)v.y << 32) | v.x);
      } else {
        o[0] = (long)(((uint64_t)(v.y & half) << 32) | (v.x & half));
        o[1] = (long)(((uint64_t)(v.y & ~half) << 32) | (v.x & ~half));
      }
    };
    v4i base;
#pragma unroll
    for (int i = 0; i < 4; i++) base[i] = E_BASE_BITS;
    v4i e[WA][NH];
    float dsj[2][NH], dmj[2][NH];
    auto factors = [&](int gg) {
#pragma unroll
      for (int h = 0; h < NH; h++) {
        dsj[gg & 1][h] = from(NH * gg + h, sv);
        if constexpr (Q::MIN) dmj[gg & 1][h] = from(NH * gg + h, mv);
      }
    };
    // xe (, xs) of a tile's four activation rows, the next tile's read under this
    // one's terms
    float4 xeb[2], xsb[2];
    auto scales = [&](int st) {  // st = (gg * WA + t) * NH + h
      const int h = st % NH, t = st / NH % WA, gg = st / NH / WA;
      const float* p = E + SH::PARTS * MT * (NH * gg + h) + 16 * t;
      xeb[st & 1] = *reinterpret_cast<const float4*>(p);
      if constexpr (Q::MIN) xsb[st & 1] = *reinterpret_cast<const float4*>(p + MT);
    };
    factors(0);
    scales(0);
    {
      long bw[NH];
      operands(0, bw);
#pragma unroll
      for (int t = 0; t < WA; t++)
#pragma unroll
        for (int h = 0; h < NH; h++)
          e[t][h] = __builtin_amdgcn_mfma_i32_16x16x32_i8(act(0, t), bw[h], base, 0, 0, 0);
    }
#pragma unroll
    for (int gg = 0; gg < 8; gg++) {
      if (Q::NB > 1 && (uint32_t)gg >= ng) break;
      w.pin();
      long bw[NH];
      if (gg + 1 < 8) {
        factors(gg + 1);
        operands(gg + 1, bw);
      }
#pragma unroll
      for (int t = 0; t < WA; t++) {
        long xa = 0;
        if (gg + 1 < 8) xa = act(gg + 1, t);
#pragma unroll
        for (int h = 0; h < NH; h++) {
          const int st = (gg * WA + t) * NH + h;
          if (st + 1 < 8 * WA * NH) scales(st + 1);
          __builtin_amdgcn_sched_barrier(0);
          const float ds = dsj[gg & 1][h];
          const float4 xe = xeb[st & 1];
          const float xev[4] = {xe.x, xe.y, xe.z, xe.w};
          float se[4], tx[4];
#pragma unroll
          for (int i = 0; i < 4; i++) se[i] = __int_as_float(e[t][h][i]) - E_BASE;
          if constexpr (Q::MIN) {  // xe * (d * sc * E - dmin * mn * xs)
            const float dm = dmj[gg & 1][h];
            const float4 xs = xsb[st & 1];
            const float xsv[4] = {xs.x, xs.y, xs.z, xs.w};
#pragma unroll
            for (int i = 0; i < 4; i++) tx[i] = dm * xsv[i];
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int i = 0; i < 4; i++) se[i] = ds * se[i];
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int i = 0; i < 4; i++) se[i] = se[i] - tx[i];
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int i = 0; i < 4; i++) se[i] = xev[i] * se[i];
          } else {  // (xe * scale) * E'
#pragma unroll
            for (int i = 0; i < 4; i++) tx[i] = xev[i] * ds;
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int i = 0; i < 4; i++) se[i] = tx[i] * se[i];
          }
          __builtin_amdgcn_sched_barrier(0);
#pragma unroll
          for (int i = 0; i < 4; i++) acc[t][i] += se[i];
          if (gg + 1 < 8)
            e[t][h] = __builtin_amdgcn_mfma_i32_16x16x32_i8(xa, bw[h], base, 0, 0, 0);
          __builtin_amdgcn_sched_barrier(0);
        }
      }
      if (Q::NB > 1) {  // (a branch follows: the adds stay on this side of it)
#pragma unroll
        for (int t = 0; t < WA; t++)
          asm volatile("" : "+v"(acc[t][0]), "+v"(acc[t][1]), "+v"(acc[t][2]), "+v"(acc[t][3]));
      }
    }
  }
  store_rows<WA>(P, acc, DST, BIAS, N, wr, a0, G);
}

// ops::cuantizar_i8_en (src/ops.rs:178-198) of m rows into the layout above:
// xq rows [m, m_pad) and their xe, xs are zero
template <int SUB>
__global__ __launch_bounds__(256) void k_quantize_gemm(const float* x, uint32_t m, uint32_t k,
                                                       uint32_t m_pad, int8_t* xq, float* xexs) {
  const size_t i = 8 * (blockIdx.x * 256ull + threadIdx.x);
  if (i >= (size_t)m_pad * k) return;
  const uint32_t a = (uint32_t)(i / k), col = (uint32_t)(i % k);
  float v[8] = {0, 0, 0, 0, 0, 0, 0, 0};
  if (a < m) cx_load8(x + i, v);
  uint32_t lo, hi;
  float d;
  int32_t s;
  cx_quant8_vals<SUB>(v, lo, hi, d, s);
  *reinterpret_cast<uint2*>(xq + i) = make_uint2(lo, hi);
  if ((col & (SUB - 1)) == 0) {
    float* e = xexs + (size_t)(col / SUB) * 2 * m_pad + a;
    e[0] = d;
    e[m_pad] = (float)s;
  }
}

// The prefill's row ops straight into that layout, for the contraction that
// reads them: rmsnorm (k_norm_rows' arithmetic: the reference's factor by
// cx_rms_scale, then (float)(x * scale) * w; src/kernels/scalar.rs:36-54),
// one workgroup a row; and silu(g) * u (src/forward.rs:483-487); each
// value is what the row kernel writes, then quantized as k_quantize_gemm
// quantizes it. Rows [m, m_pad) are zero.
template <int SUB, bool WG>
__global__ __launch_bounds__(256) void k_norm_quant_gemm(const float* x, const float* w,
                                                         uint32_t m, uint32_t k, float eps,
                                                         uint32_t m_pad, int8_t* xq, float* xexs) {
  __shared__ double red[9];
  __shared__ int flag;
  const int tid = threadIdx.x;
  const uint32_t a = blockIdx.x;
  const float* xr = x + (size_t)a * k;
  double scale = 0.0;
  if (a < m) scale = cx_rms_scale<WG>(xr, k, eps, red, &flag);  // the same for the whole workgroup
  for (uint32_t i = 8 * tid; i < k; i += 2048) {  // whole quads of lanes (k % 32 == 0)
    float v[8] = {0, 0, 0, 0, 0, 0, 0, 0};
    if (a < m) {
      float nw[8];
      cx_load8(xr + i, v);
      cx_load8(w + i, nw);
#pragma unroll
      for (int j = 0; j < 8; j++) v[j] = (float)((double)v[j] * scale) * nw[j];
    }
    uint32_t lo, hi;
    float d;
    int32_t s;
    cx_quant8_vals<SUB>(v, lo, hi, d, s);
    *reinterpret_cast<uint2*>(xq + (size_t)a * k + i) = make_uint2(lo, hi);
    if ((i & (SUB - 1)) == 0) {
      float* e = xexs + (size_t)(i / SUB) * 2 * m_pad + a;
      e[0] = d;
      e[m_pad] = (float)s;
    }
  }
}

template <int SUB>
__global__ __launch_bounds__(256) void k_swiglu_quant_gemm(const float* g, const float* u,
                                                           uint32_t m, uint32_t k, uint32_t m_pad,
                                                           int8_t* xq, float* xexs) {
  const size_t i = 8 * (blockIdx.x * 256ull + threadIdx.x);
  if (i >= (size_t)m_pad * k) return;
  const uint32_t a = (uint32_t)(i / k), col = (uint32_t)(i % k);
  float v[8] = {0, 0, 0, 0, 0, 0, 0, 0};
  if (a < m) {
    float b[8];
    cx_load8(g + i, v);
    cx_load8(u + i, b);
#pragma unroll
    for (int j = 0; j < 8; j++) v[j] = cx_swiglu(v[j], b[j]);
  }
  uint32_t lo, hi;
  float d;
  int32_t s;
  cx_quant8_vals<SUB>(v, lo, hi, d, s);
  *reinterpret_cast<uint2*>(xq + i) = make_uint2(lo, hi);
  if ((col & (SUB - 1)) == 0) {
    float* e = xexs + (size_t)(col / SUB) * 2 * m_pad + a;
    e[0] = d;
    e[m_pad] = (float)s;
  }
}

struct Config {
  int tw, mt, threads;
  size_t lds;
};

typedef void (*gemm_kernel)(GemmParams);

template <int T, int RW, int AW, int WA, int KS, int NSB, int S>
Config make_config(gemm_kernel* k) {
  using SH = Shape<T, RW, AW, WA, KS, NSB>;
  static_assert(SH::lds(S) <= 160 * 1024, "LDS of one CU");
  *k = k_gemm<T, RW, AW, WA, KS, NSB, S>;
  return Config{SH::TW, SH::MT, 64 * SH::NW, SH::lds(S)};
}

template <int T, int NW, int WA, int OCC>
Config make_config_w(gemm_kernel* k) {
  using SH = WShape<NW, WA>;
  *k = k_gemm_w<T, NW, WA, OCC>;
  return Config{SH::TW, SH::MT, 64 * NW, SH::lds};
}

// The tile shapes: weight rows x activation rows, waves, super-blocks per
// stage, ring stages: 0 to 5 are k_gemm, 6 to 8 k_gemm_w.
template <int T>
Config config(int id, gemm_kernel* k) {
  switch (id) {
    case 0: return make_config<T, 1, 1, 1, 8, 4, 2>(k);  // 16 x 16, 8 waves split k
    case 1: return make_config<T, 1, 1, 1, 8, 2, 3>(k);  // 16 x 16, 8 waves split k
    case 2: return make_config<T, 4, 1, 1, 1, 2, 3>(k);  // 64 x 16
    case 3: return make_config<T, 4, 2, 1, 1, 2, 2>(k);  // 64 x 32, 8 waves
    case 4: return make_config<T, 2, 2, 1, 1, 2, 2>(k);  // 32 x 32
    case 5: return make_config<T, 4, 2, 2, 1, 1, 3>(k);  // 64 x 64, 8 waves
    case 6: return make_config_w<T, 4, 1, 4>(k);         // 64 x 16
    case 7: return make_config_w<T, 4, 2, 4>(k);         // 64 x 32
    default: return make_config_w<T, 4, 4, 3>(k);        // 64 x 64
  }
}

// Weights in registers (k_gemm_w) where its tiles give the chip enough
// workgroups, the larger tile first. Whole calls (the quantization with it), us,
// Q4_K, beside the best of k_gemm's tiles:
//   64 x 64: 11008 x 2048 m = 512 73, 103, m = 256 45, 59; 4096 x 4096 m = 512 58, 75.
//     Not for m <= 32, half of it padding: 151936 x 2048 m = 32 103, in 64 x 32 74
//   64 x 32: 11008 x 2048 m = 128 31, 36; 4096 x 4096 m = 256 39, 42; 2048 x 11008
//     m = 512 88, 96 (its 512 workgroups; at m = 256 76, 66: k_gemm)
//   64 x 16: no better than k_gemm's 64 x 16 and 64 x 32, and no worse than by 10%:
//     4096 x 4096 m = 64 26.5, 26.3, m = 128 29.9, 30.2; 4096 x 14336 (Q5_K) m = 64
//     78, 71; 2048 x 11008 m = 128 57, 54, 1847 x 2048 m = 389 33, 26: k_gemm. Not
//     past two rounds of workgroups: 9000 x 4096 m = 64 40 (Q5_K 47), in 64 x 32 37
//     (40), 16500 x 2048 m = 32 25.6 (29.1), 23.2 (24.6); nor, for m <= 32, past one:
//     11008 x 2048 m = 32 19.6 (Q5_K 22.2), in k_gemm's 64 x 32 19.6 (20.8)
// Otherwise, with m <= 16 rows of many weights, 64 x 16 of k_gemm (11008 x 2048 17.9;
// 16 x 16 20.8), and for few weight rows (n < 4096: 2048 x 11008 and the q/o/k/v
// shapes) the largest k_gemm tile (64 x 64, 64 x 32, then 32 x 32) that gives at
// least 5/8 of the CUs a workgroup; below that, 16 x 16 tiles that split k over the
// waves (four super-blocks a stage up to a workgroup per CU, two past it): 2048 x
// 11008 m = 256 66 us in 64 x 32 tiles, 90 in 64 x 64, 2048 x 2048 20.4, 24.7, 256 x
// 2048 13.4 in 16 x 16, 24.8. Within 5% of the best tile there but for m = 389 of
// 2048 x 11008 (94; 64 x 32 of k_gemm_w 85).
// Where n >= 4096 the line at 16 rows costs, most where k is long: 4096 x 4096, m <=
// 16, 26 us where 16 x 16 tiles over a split k take 15.6, 4096 x 14336 65 and 29 (m =
// 17 to 32 69 and 48), 8192 x 2048 17.9 and 15.0; 22016 x 2048 27 and 19.7 (k_gemm_w's
// 64 x 16).
int choose(uint32_t n, uint32_t m) {
  auto tiles = [&](uint32_t tw, uint32_t mt) { return (n + tw - 1) / tw * ((m + mt - 1) / mt); };
  const bool few = n < 4096;
  if (m > 16) {
    if (m > 32 && tiles(64, 64) >= (few ? 768u : 440u)) return 8;
    if (tiles(64, 32) >= (few ? 512u : 300u)) return 7;
    const uint32_t t16 = tiles(64, 16);
    if (!few && t16 >= (m <= 32 ? 513u : 528u)) return 7;
    if (!few && t16 >= 128) return m <= 32 && t16 >= 264 ? 3 : 6;
  } else if (!few) {
    return 2;
  }
  constexpr uint32_t ENOUGH = 256 * 5 / 8;  // workgroups, on 256 CUs
  if (tiles(64, 64) >= ENOUGH) return 5;
  if (tiles(64, 32) >= ENOUGH) return 3;
  if (tiles(32, 32) >= ENOUGH) return 4;
  return tiles(16, 16) <= 256 ? 0 : 1;
}

// xq and xexs of m_pad quantized rows in scratch
inline int8_t* scratch_xq(uint8_t* scratch) { return reinterpret_cast<int8_t*>(scratch); }
inline float* scratch_xexs(uint8_t* scratch, size_t m_pad, size_t k) {
  return reinterpret_cast<float*>(scratch + (m_pad * k + 255) / 256 * 256);
}

int quantize(const float* lhs, uint32_t m, uint32_t k, uint32_t m_pad, int sub, uint8_t* scratch,
             hipStream_t s) {
  const size_t qgrid = ((size_t)m_pad * k / 8 + 255) / 256;
  CX_REQUIRE(qgrid < (1ull << 31), "gemm: %zu activation values is too many", (size_t)m_pad * k);
  if (sub == 16)
    hipLaunchKernelGGL(k_quantize_gemm<16>, dim3((unsigned)qgrid), dim3(256), 0, s, lhs, m, k,
                       m_pad, scratch_xq(scratch), scratch_xexs(scratch, m_pad, k));
  else
    hipLaunchKernelGGL(k_quantize_gemm<32>, dim3((unsigned)qgrid), dim3(256), 0, s, lhs, m, k,
                       m_pad, scratch_xq(scratch), scratch_xexs(scratch, m_pad, k));
  CX_HIP(hipGetLastError());
  return CX_OK;
}

// every tile height (16, 32 or 64 rows) divides 64
inline uint32_t pad64(size_t m) { return (uint32_t)((m + 63) / 64 * 64); }

// the formats of k_gemm_x
bool direct_type(int type) { return cx_is_block32(type) || cx_sub(type) == 16; }

template <int T, int WA, int OCC>
Config make_config_x(gemm_kernel* k) {
  using SH = XShape<T, WA>;
  *k = k_gemm_x<T, WA, OCC>;
  return Config{SH::TW, SH::MT, 256, SH::lds};
}

// The largest tile whose workgroups still keep the chip busy; whole calls, us, with
// 16, 32, 64 activation rows a workgroup (the 32-value formats' term is shorter):
//   Q6_K 4096 x 14336 m = 512 437, 285, 253, m = 256 237, 169, 203; 11008 x 2048
//   m = 128 52, 41, 45, m = 17 26, 26, 36; 2048 x 11008 m = 256 128, 112, 164,
//   m = 128 88, 111, 163
//   Q8_0 4864 x 896 m = 512 44, 31, 29, m = 128 21.5, 19.5, 19.7; 2048 x 2048
//   m = 512 61, 39, 32, m = 256 37, 27, 31; 896 x 4864 m = 512 60, 48, 60
//   Q5_0 4864 x 896 m = 512 64, 41, 35, m = 128 28, 24, 23; 2048 x 2048 m = 512 89,
//   53, 39
// Q6_K, Q8_0 and Q5_0 are within 5% of their best tile over these widths and m = 17
// to 512. Q2_K and Q3_K keep 16 rows longer, which this rule does not know:
//   Q2_K 4096 x 14336 m = 77 105, 139, 236, 2048 x 11008 m = 256 90, 113, 185 (both
//   take 32: 1.36 and 1.28 of the best); Q3_K 95, 120, 188 and 89, 102, 150
template <int T>
Config config_x(uint32_t n, uint32_t m, gemm_kernel* k) {
  auto tiles = [&](uint32_t mt) { return (n + 63) / 64 * ((m + mt - 1) / mt); };
  if (tiles(64) >= (XQ<T>::SUB == 32 ? 256u : 440u)) return make_config_x<T, 4, 3>(k);
  if (tiles(32) >= 160u) return make_config_x<T, 2, 4>(k);
  return make_config_x<T, 1, 4>(k);
}
Config config_x(int type, uint32_t n, uint32_t m, gemm_kernel* k) {
  switch (type) {
    case CX_Q8_0: return config_x<CX_Q8_0>(n, m, k);
    case CX_Q5_0: return config_x<CX_Q5_0>(n, m, k);
    case CX_Q2_K: return config_x<CX_Q2_K>(n, m, k);
    case CX_Q3_K: return config_x<CX_Q3_K>(n, m, k);
    default: return config_x<CX_Q6_K>(n, m, k);
  }
}

// the tile of n weight rows of a type x m activation rows
Config config_of(int type, uint32_t n, uint32_t m, gemm_kernel* k) {
  if (type == CX_Q4_K) return config<CX_Q4_K>(choose(n, m), k);
  if (type == CX_Q5_K) return config<CX_Q5_K>(choose(n, m), k);
  return config_x(type, n, m, k);
}

// the contraction over rows quantized with a row count m_pad that is a
// multiple of the chosen tile's height
int contract(int type, GemmParams& P, hipStream_t s) {
  gemm_kernel k = nullptr;
  const Config c = config_of(type, P.n, P.m, &k);
  CX_REQUIRE(P.m_pad % c.mt == 0 && P.m_pad >= P.m, "gemm: %u padded rows for tiles of %d",
             P.m_pad, c.mt);
  P.xq = scratch_xq(P.scratch);
  P.xexs = scratch_xexs(P.scratch, P.m_pad, P.k);
  P.row_tiles = (P.n + c.tw - 1) / c.tw;
  P.act_tiles = (P.m + c.mt - 1) / c.mt;
  const size_t grid = (size_t)(P.row_tiles + 7) / 8 * 8 * P.act_tiles;
  CX_REQUIRE(grid < (1ull << 31), "gemm: %u x %u is too large", P.n, P.m);
  hipLaunchKernelGGL(k, dim3((unsigned)grid), dim3(c.threads), c.lds, s, P);
  CX_HIP(hipGetLastError());
  return CX_OK;
}
}  // namespace

bool cx_gemm_supported(int type) { return cx_has_gemv(type); }

size_t cx_gemm_scratch_bytes(size_t m, size_t k) {  // xe and xs for sub-blocks of 16
  const size_t m_pad = (m + 63) / 64 * 64;
  return (m_pad * k + 255) / 256 * 256 + m_pad * (k / 16) * 8;
}

int cx_launch_gemm(int type, const uint8_t* w, size_t n, size_t k, const float* lhs, size_t m,
                   float* dst, void* scratch, hipStream_t s) {
  CX_REQUIRE(cx_gemm_supported(type), "gemm: type %d has no MFMA path", type);
  CX_REQUIRE(w && lhs && dst && scratch, "gemm: null pointer");
  const size_t vpb = (size_t)cx_vpb(type);
  CX_REQUIRE(k % vpb == 0 && k > 0, "gemm: k=%zu is not a multiple of %zu", k, vpb);
  CX_REQUIRE(n < (1u << 31) && m < (1u << 24) && k < (1u << 24), "gemm: shape too large");
  CX_REQUIRE(((uintptr_t)w & (direct_type(type) ? 1 : 15)) == 0 && ((uintptr_t)lhs & 15) == 0 &&
                 ((uintptr_t)scratch & 255) == 0,
             "gemm: weights (Q4_K/Q5_K 16-byte, others 2-byte) and activations (16-byte) misaligned");
  if (!n || !m) return CX_OK;
  GemmParams P{};
  P.lhs = lhs;
  P.scratch = reinterpret_cast<uint8_t*>(scratch);
  P.w = w;
  P.dst = dst;
  P.n = (uint32_t)n;
  P.k = (uint32_t)k;
  P.m = (uint32_t)m;
  P.nb = (uint32_t)(k / vpb);
  P.row_bytes = P.nb * cx_bpb(type);
  // activation rows padded to the tile height (zero rows quantize to zero)
  gemm_kernel kern = nullptr;
  const uint32_t mt = (uint32_t)config_of(type, P.n, P.m, &kern).mt;
  P.m_pad = (P.m + mt - 1) / mt * mt;
  const int rc = quantize(lhs, P.m, P.k, P.m_pad, cx_sub(type), P.scratch, s);
  return rc ? rc : contract(type, P, s);
}

int cx_gemm_quantize(const float* lhs, size_t m, size_t k, int sub, void* scratch, hipStream_t s) {
  CX_REQUIRE(lhs && scratch, "gemm: null pointer");
  CX_REQUIRE(sub == 16 || sub == 32, "gemm: sub-blocks of 16 or 32, not %d", sub);
  CX_REQUIRE(k % 32 == 0 && k > 0 && k < (1u << 24) && m < (1u << 24), "gemm: %zu x %zu", m, k);
  CX_REQUIRE(((uintptr_t)lhs & 15) == 0 && ((uintptr_t)scratch & 255) == 0,
             "gemm: activations must be 16-byte and scratch 256-byte aligned");
  if (!m) return CX_OK;
  return quantize(lhs, (uint32_t)m, (uint32_t)k, pad64(m), sub, reinterpret_cast<uint8_t*>(scratch),
                  s);
}

int cx_gemm_norm_quantize(const float* x, const float* w, size_t m, size_t k, float eps, int sub,
                          void* scratch, hipStream_t s) {
  CX_REQUIRE(x && w && scratch, "gemm: null pointer");
  CX_REQUIRE(sub == 16 || sub == 32, "gemm: sub-blocks of 16 or 32, not %d", sub);
  CX_REQUIRE(k % 32 == 0 && k > 0 && k < (1u << 24) && m < (1u << 24), "gemm: %zu x %zu", m, k);
  CX_REQUIRE(((uintptr_t)x & 15) == 0 && ((uintptr_t)w & 15) == 0 &&
                 ((uintptr_t)scratch & 255) == 0,
             "gemm: rows and weights must be 16-byte and scratch 256-byte aligned");
  if (!m) return CX_OK;
  const uint32_t mp = pad64(m);
  uint8_t* sc = reinterpret_cast<uint8_t*>(scratch);
  const bool wg = cx_rms_wg(k);
  const auto norm = sub == 16 ? (wg ? k_norm_quant_gemm<16, true> : k_norm_quant_gemm<16, false>)
                              : (wg ? k_norm_quant_gemm<32, true> : k_norm_quant_gemm<32, false>);
  hipLaunchKernelGGL(norm, dim3(mp), dim3(256), 0, s, x, w, (uint32_t)m, (uint32_t)k, eps, mp,
                     scratch_xq(sc), scratch_xexs(sc, mp, k));
  CX_HIP(hipGetLastError());
  return CX_OK;
}

int cx_gemm_swiglu_quantize(const float* g, const float* u, size_t m, size_t k, int sub,
                            void* scratch, hipStream_t s) {
  CX_REQUIRE(g && u && scratch, "gemm: null pointer");
  CX_REQUIRE(sub == 16 || sub == 32, "gemm: sub-blocks of 16 or 32, not %d", sub);
  CX_REQUIRE(k % 32 == 0 && k > 0 && k < (1u << 24) && m < (1u << 24), "gemm: %zu x %zu", m, k);
  CX_REQUIRE(((uintptr_t)g & 15) == 0 && ((uintptr_t)u & 15) == 0 &&
                 ((uintptr_t)scratch & 255) == 0,
             "gemm: rows must be 16-byte and scratch 256-byte aligned");
  if (!m) return CX_OK;
  const uint32_t mp = pad64(m);
  uint8_t* sc = reinterpret_cast<uint8_t*>(scratch);
  const size_t grid = ((size_t)mp * k / 8 + 255) / 256;
  CX_REQUIRE(grid < (1ull << 31), "gemm: %zu activation values is too many", (size_t)mp * k);
  if (sub == 16)
    hipLaunchKernelGGL(k_swiglu_quant_gemm<16>, dim3((unsigned)grid), dim3(256), 0, s, g, u,
                       (uint32_t)m, (uint32_t)k, mp, scratch_xq(sc), scratch_xexs(sc, mp, k));
  else
    hipLaunchKernelGGL(k_swiglu_quant_gemm<32>, dim3((unsigned)grid), dim3(256), 0, s, g, u,
                       (uint32_t)m, (uint32_t)k, mp, scratch_xq(sc), scratch_xexs(sc, mp, k));
  CX_HIP(hipGetLastError());
  return CX_OK;
}

int cx_gemm_apply(int type, const uint8_t* w, size_t n, size_t k, size_t m, float* dst,
                  const void* scratch, hipStream_t s) {
  CX_REQUIRE(cx_gemm_supported(type), "gemm: type %d has no MFMA path", type);
  CX_REQUIRE(w && dst && scratch, "gemm: null pointer");
  const size_t vpb = (size_t)cx_vpb(type);
  CX_REQUIRE(k % vpb == 0 && k > 0, "gemm: k=%zu is not a multiple of %zu", k, vpb);
  CX_REQUIRE(n < (1u << 31) && m < (1u << 24) && k < (1u << 24), "gemm: shape too large");
  CX_REQUIRE(((uintptr_t)w & (direct_type(type) ? 1 : 15)) == 0 && ((uintptr_t)scratch & 255) == 0,
             "gemm: weights (Q4_K/Q5_K 16-byte, others 2-byte) or scratch (256-byte) misaligned");
  if (!n || !m) return CX_OK;
  GemmParams P{};
  P.scratch = const_cast<uint8_t*>(reinterpret_cast<const uint8_t*>(scratch));
  P.w = w;
  P.dst = dst;
  P.n = (uint32_t)n;
  P.k = (uint32_t)k;
  P.m = (uint32_t)m;
  P.m_pad = pad64(m);
  P.nb = (uint32_t)(k / vpb);
  P.row_bytes = P.nb * cx_bpb(type);
  return contract(type, P, s);
}

bool cx_gemm_multi_fits(int type, const uint32_t* n, uint32_t count, size_t m) {
  if (!n || count < 1 || count > CX_GEMM_SEGS || !m || m >= (1u << 24) ||
      !cx_gemm_supported(type))
    return false;
  uint32_t total = 0;
  for (uint32_t i = 0; i < count; i++) total += n[i];
  if (!total) return false;
  gemm_kernel kern = nullptr;
  const Config c = config_of(type, total, (uint32_t)m, &kern);
  for (uint32_t i = 0; count > 1 && i < count; i++)
    if (n[i] % c.tw != 0) return false;  // a tile would straddle two matrices
  return true;
}

int cx_gemm_apply_multi(int type, const uint8_t* const* w, const uint32_t* n, uint32_t count,
                        size_t k, size_t m, float* const* dst, const float* const* bias, int accum,
                        const void* scratch, hipStream_t s) {
  CX_REQUIRE(w && dst && cx_gemm_multi_fits(type, n, count, m),
             "gemm: %u matrices of type %d over %zu rows do not fit one launch", count, type, m);
  const size_t vpb = (size_t)cx_vpb(type);
  CX_REQUIRE(k % vpb == 0 && k > 0 && k < (1u << 24), "gemm: k=%zu", k);
  CX_REQUIRE(((uintptr_t)scratch & 255) == 0, "gemm: scratch misaligned");
  GemmParams P{};
  P.scratch = const_cast<uint8_t*>(reinterpret_cast<const uint8_t*>(scratch));
  P.nseg = count;
  for (uint32_t i = 0; i < count; i++) {
    CX_REQUIRE(w[i] && dst[i] && ((uintptr_t)w[i] & (direct_type(type) ? 1 : 15)) == 0,
               "gemm: matrix %u: null or misaligned (Q4_K/Q5_K 16-byte, others 2-byte) pointer", i);
    P.sw[i] = w[i];
    P.sd[i] = dst[i];
    P.sbias[i] = bias ? bias[i] : nullptr;
    P.sr[i + 1] = P.sr[i] + n[i];
  }
  P.accum = accum ? 1u : 0u;
  P.w = w[0];
  P.dst = dst[0];
  P.n = P.sr[count];
  P.k = (uint32_t)k;
  P.m = (uint32_t)m;
  P.m_pad = pad64(m);
  P.nb = (uint32_t)(k / vpb);
  P.row_bytes = P.nb * cx_bpb(type);
  return contract(type, P, s);
}
