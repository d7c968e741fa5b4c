// cx_attn_many.hip — order-exact causal GQA attention of many query tokens
// (ops::atencion, src/ops.rs:1258-1325: the batched prefill and the general
// operator), gfx950.
//
// The reference's arithmetic and order, bit for bit (as cx_attn.hip): the
// sequential head_dim-term dot times 1/sqrt(hd); the exact maximum; e = exp(s -
// max) (glibc's expf); the sum of e in position order from 0; p = e * (1/sum),
// or 1/total everywhere when the maximum is not finite; out[d] = p * v[d] added
// in position order from 0. Every product and every add is one f32 operation,
// so a multiply and an add a term is the floor.
//
// The query heads of one KV group share its K and V, so the rows of the work
// are (token, head of the group) pairs: row r of group g is token r / per, head
// g * per + r % per, R = tokens * per rows a group. Scores and exps lie
// position-major, sc[(g * total + p) * rp + r] with rp = R rounded up to 64.
//
// k_mq_scores  q.k as a register-tiled product: a lane holds TI rows x TJ
//   positions, its operands 16 bytes (4 dims) at a time from LDS.
// k_mq_softmax 64 rows a workgroup, lane = row: waves 1-15 form a stage's exps
//   (in place, and in LDS), wave 0 adds the stage before in position order.
// k_mq_pv      p.v the same way: a lane holds RM rows x 4 dims.
//
// Why register tiles from LDS (f32 multiply + add, clocks an instruction and
// SIMD with two or more waves; one wave alone issues every ~4.6): both operands
// in VGPRs 2.4. The broadcasts that would spare the LDS reads cost more: a DPP
// row_newbcast operand ~7.7 for the multiply, readlane + SGPR 4.0; SGPR operands
// 2.4-2.6, but their scalar loads miss the scalar cache on every K or V row and
// cover only one batch (scores 1063 us at 512 tokens x 8192 positions, 32/8
// heads, of a 508 us floor). An f32 outer-product MFMA gives the same rounded
// products but takes the VALU's own multiplier time (64 clocks per 2048) and
// does not run beside it.
#include "cx_ops.h"
#include "cx_act.h"

namespace {

constexpr uint32_t MQ_R = 64;  // rows a softmax workgroup; rows are padded to it
constexpr uint32_t MQ_C = 64;  // positions a chunk of the maxima

__device__ inline uint32_t rp_of(uint32_t R) { return (R + MQ_R - 1) / MQ_R * MQ_R; }

// ------------------------------------------------------------------ scores
// A workgroup of 4 waves takes 16 TI rows x 16 TJ positions, a wave 8 TI x 8 TJ:
// lane (ty, tx) = (lane / 8, lane % 8) the TI rows from TI ty and the TJ
// positions from TJ tx. 16 dims a stage, double-buffered direct-to-LDS loads. In
// LDS four tile rows share 256 bytes (all banks): row r's 16-byte chunk c sits
// at slot (4 (r % 4) + c) ^ (r / T % 8), so the eight rows (T apart) that a wave
// reads at once fall on different banks.
// cm[(g * nck + chunk) * rp + r]: the maximum of the chunk's scores that row r
// sees (fmaxf: a NaN is passed over).
// slot -> tile row and chunk (T = 4 or 8 rows a lane)
template <int T>
__device__ inline void tile_at(uint32_t slot, uint32_t& r, uint32_t& c) {
  const uint32_t x = (slot & 15) ^ ((slot / 16 * 4 / T) & 7);
  r = slot / 16 * 4 + x / 4;
  c = x % 4;
}
template <int HD, int TI, int TJ>
__global__ __launch_bounds__(256, TI * TJ > 16 ? 4 : 6) void k_mq_scores(const float* __restrict__ q,
                                                  const float* __restrict__ kc, uint32_t heads,
                                                  uint32_t kvh, uint32_t tokens, uint32_t pos,
                                                  float scale, float* __restrict__ sc,
                                                  float* __restrict__ cm, uint32_t nck) {
  constexpr uint32_t QR = 16 * TI, KP = 16 * TJ;     // the tile
  constexpr uint32_t LQ = QR * 4 / 256, LK = KP * 4 / 256;  // 1 KiB loads a wave and stage
  constexpr uint32_t NS = HD / 16;
  __shared__ float4 lq[2][QR * 4], lk[2][KP * 4];
  const uint32_t per = heads / kvh, R = tokens * per, total = pos + tokens, rp = rp_of(R);
  const uint32_t g = blockIdx.z, r0 = blockIdx.x * QR, p0 = blockIdx.y * KP, kvd = kvh * HD;
  if (p0 > pos + (min(r0 + QR, R) - 1) / per) return;  // no row of the tile sees it
  const uint32_t tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const uint32_t ty = lane >> 3, tx = lane & 7, wr = (w >> 1) * 8 * TI, wp = (w & 1) * 8 * TJ;
  // this lane's sources: LDS slot 64 (4 u + w) + lane of the tile; rows and
  // positions past the end repeat the last (their scores are not used)
  const float4 *sq[LQ], *sk[LK];
#pragma unroll
  for (uint32_t u = 0; u < LQ; u++) {
    uint32_t r, c;
    tile_at<TI>(64 * (4 * u + w) + lane, r, c);
    r = min(r0 + r, R - 1);
    const uint32_t tk = r / per;
    sq[u] = reinterpret_cast<const float4*>(
                q + ((size_t)tk * heads + g * per + (r - tk * per)) * HD) + c;
  }
#pragma unroll
  for (uint32_t u = 0; u < LK; u++) {
    uint32_t r, c;
    tile_at<TJ>(64 * (4 * u + w) + lane, r, c);
    sk[u] = reinterpret_cast<const float4*>(kc + (size_t)min(p0 + r, total - 1) * kvd + g * HD) + c;
  }
  auto issue = [&](uint32_t s) {
#pragma unroll
    for (uint32_t u = 0; u < LQ; u++) cx_dma16_async(sq[u] + 4 * s, &lq[s & 1][64 * (4 * u + w)]);
#pragma unroll
    for (uint32_t u = 0; u < LK; u++) cx_dma16_async(sk[u] + 4 * s, &lk[s & 1][64 * (4 * u + w)]);
  };
  float acc[TI][TJ];
#pragma unroll
  for (int i = 0; i < TI; i++)
#pragma unroll
    for (int j = 0; j < TJ; j++) acc[i][j] = 0.0f;
  issue(0);
#pragma unroll 1
  for (uint32_t s = 0; s < NS; s++) {
    cx_wait_vm<0>();  // this wave's part of stage s has landed
    cx_wait_lds();
    cx_barrier();     // every wave's; stage s - 1 is read
    if (s + 1 < NS) issue(s + 1);
    const float4* a = &lq[s & 1][(wr + TI * ty) / 4 * 16];
    const float4* b = &lk[s & 1][(wp + TJ * tx) / 4 * 16];
#pragma unroll 1
    for (uint32_t c = 0; c < 4; c++) {
      float4 x[TI];
#pragma unroll
      for (int i = 0; i < TI; i++) x[i] = a[(i >> 2) * 16 + ((((i & 3) << 2) | c) ^ ty)];
      auto rd = [&](int j) { return b[(j >> 2) * 16 + ((((j & 3) << 2) | c) ^ tx)]; };
      float4 yn = rd(0);
#pragma unroll
      for (int j = 0; j < TJ; j++) {
        const float4 y = yn;
        if (j + 1 < TJ) yn = rd(j + 1);  // under this one's arithmetic
#pragma unroll
        for (int i = 0; i < TI; i++) acc[i][j] += x[i].x * y.x;
#pragma unroll
        for (int i = 0; i < TI; i++) acc[i][j] += x[i].y * y.y;
#pragma unroll
        for (int i = 0; i < TI; i++) acc[i][j] += x[i].z * y.z;
#pragma unroll
        for (int i = 0; i < TI; i++) acc[i][j] += x[i].w * y.w;
      }
    }
  }
  // scores position-major (a lane's TI rows together), and each row's maximum
  const uint32_t rb = r0 + wr + TI * ty, pb = p0 + wp + TJ * tx;
  float mx[TI];
#pragma unroll
  for (int i = 0; i < TI; i++) mx[i] = -INFINITY;
#pragma unroll
  for (int j = 0; j < TJ; j++) {
    const uint32_t p = pb + j;
#pragma unroll
    for (int i = 0; i < TI; i++) {
      acc[i][j] = acc[i][j] * scale;
      if (p <= pos + (rb + i) / per) mx[i] = fmaxf(mx[i], acc[i][j]);
    }
    if (p < total && rb < rp) {
      float* o = sc + ((size_t)g * total + p) * rp + rb;
#pragma unroll
      for (int i = 0; i < TI; i += 4)
        *reinterpret_cast<float4*>(o + i) =
            make_float4(acc[i][j], acc[i + 1][j], acc[i + 2][j], acc[i + 3][j]);
    }
  }
#pragma unroll
  for (int i = 0; i < TI; i++) {
    mx[i] = fmaxf(mx[i], __uint_as_float(cx_dpp<CX_DPP_XOR1>(__float_as_uint(mx[i]))));
    mx[i] = fmaxf(mx[i], __uint_as_float(cx_dpp<CX_DPP_XOR2>(__float_as_uint(mx[i]))));
    mx[i] = fmaxf(mx[i], __uint_as_float(cx_dpp<CX_DPP_HALF_MIRROR>(__float_as_uint(mx[i]))));
  }
  if constexpr (8 * TJ == MQ_C) {  // a wave's positions are one chunk
    if (tx == 0 && rb < rp && (p0 + wp) / MQ_C < nck) {
      float* o = cm + ((size_t)g * nck + (p0 + wp) / MQ_C) * rp + rb;
#pragma unroll
      for (int i = 0; i < TI; i++) o[i] = mx[i];
    }
  } else {  // two waves' are: through LDS
    static_assert(16 * TJ == MQ_C, "the workgroup's positions are one chunk");
    float* m = reinterpret_cast<float*>(lq);
    __syncthreads();
    if (tx == 0)
#pragma unroll
      for (int i = 0; i < TI; i++) m[(w & 1) * QR + wr + TI * ty + i] = mx[i];
    __syncthreads();
    if (tid < QR && r0 + tid < rp)
      cm[((size_t)g * nck + p0 / MQ_C) * rp + r0 + tid] = fmaxf(m[tid], m[QR + tid]);
  }
}

// ----------------------------------------------------------------- softmax
constexpr uint32_t SM_W = 15;          // waves that form exps
constexpr uint32_t SM_E = 8;           // positions a wave and stage
constexpr uint32_t SM_P = SM_W * SM_E;  // positions a stage
// grid: (row tiles, KV groups); 16 waves. e replaces the scores; inv[g * rp + r]
// = 1 / sum (1, with e = 1/total, when the maximum is not finite)
__global__ __launch_bounds__(1024) void k_mq_softmax(float* __restrict__ sc,
                                                    const float* __restrict__ cm, uint32_t nck,
                                                    uint32_t R, uint32_t per, uint32_t pos,
                                                    uint32_t total, float* inv) {
  __shared__ float e[2][SM_P][MQ_R];
  __shared__ uint64_t etab[32];
  const uint32_t tid = threadIdx.x, t = tid & 63;
  const uint32_t w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const uint32_t rp = rp_of(R), g = blockIdx.y, tile = gridDim.x - 1 - blockIdx.x;
  const uint32_t col = tile * MQ_R + t, last = min(tile * MQ_R + MQ_R, R) - 1;
  const uint32_t tmax = pos + last / per + 1, ns = (tmax + SM_P - 1) / SM_P;
  const uint32_t n = pos + min(col, R - 1) / per + 1;  // positions this lane's row sees
  if (tid < 32) {
    const uint64_t tab[32] = CX_EXP2_TAB;
    uint64_t v = tab[0];
#pragma unroll
    for (int i = 1; i < 32; i++) v = tid == (uint32_t)i ? tab[i] : v;
    etab[tid] = v;
  }
  // the row's maximum over its chunks, a share of them by each wave
  float mx = -INFINITY;
  for (uint32_t c = w; c < (tmax + MQ_C - 1) / MQ_C; c += 16) mx = fmaxf(mx, cm[((size_t)g * nck + c) * rp + col]);
  e[0][w][t] = mx;
  __syncthreads();
#pragma unroll
  for (int i = 0; i < 16; i++) mx = fmaxf(mx, e[0][i][t]);
  const bool fin = isfinite(mx);
  __syncthreads();
  if (w == 0) {
    float tot = 0.0f;
    for (uint32_t s = 0; s <= ns; s++) {
      if (s >= 1) {  // stage s - 1, while the others write s into the other half
        const float* p = &e[(s - 1) & 1][0][t];
        float v[2][SM_P / 5];  // five batches of 24, one ahead
        constexpr int NBT = SM_P / 5;
#pragma unroll
        for (int i = 0; i < NBT; i++) v[0][i] = p[i * MQ_R];
#pragma unroll
        for (int b = 0; b < 5; b++) {
          if (b + 1 < 5) {
#pragma unroll
            for (int i = 0; i < NBT; i++) v[(b + 1) & 1][i] = p[((b + 1) * NBT + i) * MQ_R];
          }
#pragma unroll
          for (int i = 0; i < NBT; i++) tot += v[b & 1][i];
        }
      }
      __syncthreads();  // stage s is in LDS
    }
    inv[(size_t)g * rp + col] = fin ? 1.0f / tot : 1.0f;
    return;
  }
  const float pu = 1.0f / (float)n;
  float* x0 = sc + (size_t)g * total * rp + col;
  float nxt[SM_E];
  auto load = [&](uint32_t s) {
#pragma unroll
    for (uint32_t i = 0; i < SM_E; i++) {
      const uint32_t p = s * SM_P + (w - 1) * SM_E + i;
      nxt[i] = 0.0f;
      if (p < tmax) nxt[i] = x0[(size_t)p * rp];
    }
  };
  load(0);
  for (uint32_t s = 0; s <= ns; s++) {
    if (s < ns) {
      float cur[SM_E];
#pragma unroll
      for (uint32_t i = 0; i < SM_E; i++) cur[i] = nxt[i];
      if (s + 1 < ns) load(s + 1);
#pragma unroll
      for (uint32_t i = 0; i < SM_E; i++) {
        const uint32_t p = s * SM_P + (w - 1) * SM_E + i;
        const float y = p >= n ? 0.0f : fin ? cx_expf_tab(cur[i] - mx, etab) : pu;
        e[s & 1][(w - 1) * SM_E + i][t] = y;
        if (p < tmax) x0[(size_t)p * rp] = y;
      }
    }
    __syncthreads();
  }
}

// --------------------------------------------------------------------- P·V
// A lane holds RM rows x 4 dims, a wave 256 / HD such groups of rows x all dims;
// a workgroup of 4 waves takes ROWS rows. V and e stream through an LDS ring of
// NST stages of PV_P positions (direct-to-LDS loads, issued NST - 1 stages
// ahead: with few rows a CU runs one wave a SIMD, and a stage's arithmetic is
// shorter than a load). Each wave turns the e it loaded itself into p = e * inv,
// in place, at the end of the stage before.
constexpr uint32_t PV_P = 32;
template <int HD, int RM, int NST>
__global__ __launch_bounds__(256) void k_mq_pv(const float* __restrict__ vc,
                                              const float* __restrict__ sc,
                                              const float* __restrict__ inv, uint32_t heads,
                                              uint32_t kvh, uint32_t tokens, uint32_t pos,
                                              float* __restrict__ out) {
  constexpr uint32_t DL = HD / 4;           // lanes over the dims
  constexpr uint32_t ROWS = 256 / DL * RM;  // rows a workgroup
  constexpr uint32_t SV = PV_P * DL, SE = PV_P * ROWS;  // a stage: float4s of V, floats of e
  constexpr uint32_t LV = SV / 256;                     // V loads a wave and stage
  constexpr uint32_t W = SE >= 1024 ? 4 : 1;            // floats a lane and load of e
  constexpr uint32_t LE = SE / (256 * W);               // e loads a wave and stage
  constexpr uint32_t L = LV + LE;
  static_assert(LV >= 1 && LE >= 1 && ROWS % W == 0 && (NST - 1) * L <= 63, "a stage's loads");
  extern __shared__ __align__(16) uint8_t lds[];
  float4* lv = reinterpret_cast<float4*>(lds);         // [NST][PV_P][DL]
  float* lp = reinterpret_cast<float*>(lv + NST * SV);  // [NST][PV_P][ROWS]
  const uint32_t per = heads / kvh, R = tokens * per, total = pos + tokens, rp = rp_of(R);
  const uint32_t g = blockIdx.y, kvd = kvh * HD, tile = gridDim.x - 1 - blockIdx.x;
  const uint32_t r0 = tile * ROWS, tid = threadIdx.x, lane = tid & 63;
  const uint32_t w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const uint32_t dl = tid % DL, rg = tid / DL * RM;  // this lane's dims and first row
  const uint32_t lo = pos + r0 / per + 1;            // every row of the tile sees the first lo
  const uint32_t hi = pos + (min(r0 + ROWS, R) - 1) / per + 1, ns = (hi + PV_P - 1) / PV_P;
  // load u of this wave: V float4s 64 (4 u + w) + lane of the stage, e floats
  // W (64 (4 u + w) + lane); positions past the last repeat it, never used
  const float* vb = vc + g * HD;
  const float* eb = sc + (size_t)g * total * rp + r0;
  auto issue = [&](uint32_t s) {
    const uint32_t slot = s % NST;
#pragma unroll
    for (uint32_t u = 0; u < LV; u++) {
      const uint32_t f = 64 * (4 * u + w) + lane, p = min(s * PV_P + f / DL, total - 1);
      cx_dma16_async(vb + (size_t)p * kvd + 4 * (f % DL), lv + slot * SV + 64 * (4 * u + w));
    }
#pragma unroll
    for (uint32_t u = 0; u < LE; u++) {
      const uint32_t f = W * (64 * (4 * u + w) + lane), p = min(s * PV_P + f / ROWS, total - 1);
      const float* e = eb + (size_t)p * rp + f % ROWS;
      float* d = lp + slot * SE + W * 64 * (4 * u + w);
      if constexpr (W == 4) cx_dma16_async(e, d);
      else cx_dma4_async(e, d);
    }
  };
  float iv[LE][W];
#pragma unroll
  for (uint32_t u = 0; u < LE; u++)
#pragma unroll
    for (uint32_t i = 0; i < W; i++)
      iv[u][i] = inv[(size_t)g * rp + r0 + W * (64 * (4 * u + w) + lane) % ROWS + i];
  auto scale = [&](uint32_t s) {  // what this wave loaded of stage s, landed
#pragma unroll
    for (uint32_t u = 0; u < LE; u++) {
      float* d = lp + s % NST * SE + W * (64 * (4 * u + w) + lane);
      if constexpr (W == 4) {
        const float4 e = *reinterpret_cast<const float4*>(d);
        *reinterpret_cast<float4*>(d) =
            make_float4(e.x * iv[u][0], e.y * iv[u][1], e.z * iv[u][2], e.w * iv[u][3]);
      } else {
        *d = *d * iv[u][0];
      }
    }
  };
  float4 acc[RM];
  uint32_t n[RM];
#pragma unroll
  for (int i = 0; i < RM; i++) {
    acc[i] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    n[i] = pos + min(r0 + rg + i, R - 1) / per + 1;
  }
#pragma unroll
  for (int s = 0; s < NST - 1; s++) issue(s);
  cx_wait_vm<(NST - 2) * L>();
  scale(0);
#pragma unroll 1
  for (uint32_t s = 0; s < ns; s++) {
    cx_wait_lds();
    cx_barrier();  // stage s is in LDS from every wave, stage s - 1 is read
    issue(s + NST - 1);
    const float4* v = lv + s % NST * SV + dl;
    const float* p = lp + s % NST * SE + rg;
    if (s * PV_P + PV_P <= lo) {
      // four positions at a time, the next four's reads under their arithmetic
      float4 x[2][4];
      float y[2][4][RM];
      auto rd = [&](int b, uint32_t j) {
#pragma unroll
        for (int k = 0; k < 4; k++) {
          x[b][k] = v[(j + k) * DL];
#pragma unroll
          for (int i = 0; i < RM; i++) y[b][k][i] = p[(j + k) * ROWS + i];
        }
      };
      rd(0, 0);
#pragma unroll
      for (int b = 0; b < (int)PV_P / 4; b++) {
        if (b + 1 < (int)PV_P / 4) rd((b + 1) & 1, 4 * (b + 1));
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int k = 0; k < 4; k++) {
          const float4 z = x[b & 1][k];
#pragma unroll
          for (int i = 0; i < RM; i++) {
            const float w = y[b & 1][k][i];
            float4 m = make_float4(w * z.x, w * z.y, w * z.z, w * z.w);
            // (four products, then their adds: an add right behind its multiply waits for it)
            asm volatile("" : "+v"(m.x), "+v"(m.y), "+v"(m.z), "+v"(m.w));
            acc[i].x += m.x;
            acc[i].y += m.y;
            acc[i].z += m.z;
            acc[i].w += m.w;
          }
        }
        __builtin_amdgcn_sched_barrier(0);
      }
    } else {
      // positions that some rows do not see: an add only where the row does
      // (V there may hold anything)
      const uint32_t je = min(PV_P, hi - s * PV_P);
      for (uint32_t j = 0; j < je; j++) {
        const float4 x = v[j * DL];
#pragma unroll
        for (int i = 0; i < RM; i++) {
          const float y = p[j * ROWS + i];
          const bool see = s * PV_P + j < n[i];
          const float4 z = make_float4(acc[i].x + y * x.x, acc[i].y + y * x.y, acc[i].z + y * x.z,
                                       acc[i].w + y * x.w);
          acc[i].x = see ? z.x : acc[i].x;
          acc[i].y = see ? z.y : acc[i].y;
          acc[i].z = see ? z.z : acc[i].z;
          acc[i].w = see ? z.w : acc[i].w;
        }
      }
    }
    cx_wait_vm<(NST - 2) * L>();
    scale(s + 1);
  }
  cx_wait_vm<0>();  // the loads of stages past the last
#pragma unroll
  for (int i = 0; i < RM; i++) {
    const uint32_t r = r0 + rg + i, tk = r / per;
    if (r < R)
      reinterpret_cast<float4*>(out + ((size_t)tk * heads + g * per + (r - tk * per)) * HD)[dl] =
          acc[i];
  }
}

template <int HD, int T>
void launch_scores(const cx_attn_many_args& a, uint32_t R, uint32_t total, uint32_t nck,
                   float scale, hipStream_t s) {
  constexpr uint32_t W = 16 * T;
  hipLaunchKernelGGL((k_mq_scores<HD, T, T>), dim3((R + W - 1) / W, (total + W - 1) / W, a.kvh),
                     dim3(256), 0, s, a.q, a.k, a.heads, a.kvh, a.tokens, a.pos, scale, a.sc, a.cm,
                     nck);
}
template <int HD, int RM>
void launch_pv(const cx_attn_many_args& a, uint32_t R, hipStream_t s) {
  constexpr uint32_t ROWS = 1024 / HD * RM;
  constexpr int NST = RM == 4 ? 3 : 4;  // two workgroups a CU either way
  hipLaunchKernelGGL((k_mq_pv<HD, RM, NST>), dim3((R + ROWS - 1) / ROWS, a.kvh), dim3(256),
                     NST * PV_P * (HD + ROWS) * sizeof(float), s, a.v, a.sc, a.inv, a.heads, a.kvh,
                     a.tokens, a.pos, a.out);
}

template <int HD>
int launch(const cx_attn_many_args& a, hipStream_t s) {
  const uint32_t per = a.heads / a.kvh, R = a.tokens * per, total = a.pos + a.tokens;
  const uint32_t nt = (R + MQ_R - 1) / MQ_R, nck = (total + MQ_C - 1) / MQ_C;
  const float scale = 1.0f / sqrtf((float)HD);
  CX_REQUIRE(nck <= 65535 && a.kvh <= 65535, "attention: %u positions", total);
  // 128 x 128 score tiles where they give the chip four workgroups a CU (8B
  // shape, 512 tokens at 4096 positions: 374 us against 400 in 64 x 64 tiles),
  // else 64 x 64 (16/2 heads, 256 tokens at 512: 21 us against 45)
  if ((size_t)((R + 127) / 128) * ((total + 127) / 128) * a.kvh >= 1024)
    launch_scores<HD, 8>(a, R, total, nck, scale, s);
  else
    launch_scores<HD, 4>(a, R, total, nck, scale, s);
  CX_HIP(hipGetLastError());
  hipLaunchKernelGGL(k_mq_softmax, dim3(nt, a.kvh), dim3(1024), 0, s, a.sc, a.cm, nck, R, per,
                     a.pos, total, a.inv);
  CX_HIP(hipGetLastError());
  // P.V rows a lane: the outputs are what there is to spread over the CUs, so
  // the more rows, the more of them a lane. Measured (4, 2, 1 rows a lane): 8B
  // shape, 512 tokens at 8192 positions 981, 1483 and 2459 us; 16/2 heads x 128,
  // 512 tokens at 512 57, 47 and 63, 256 tokens 55, 39.6 and 42; 14/2 x 64, 512
  // tokens at 512 47, 30 and 24
  const size_t wg1 = (size_t)((R + 1024 / HD - 1) / (1024 / HD)) * a.kvh;  // workgroups of 1 a lane
  if (wg1 / 4 >= 512)
    launch_pv<HD, 4>(a, R, s);
  else if (wg1 / 2 >= 256)
    launch_pv<HD, 2>(a, R, s);
  else
    launch_pv<HD, 1>(a, R, s);
  CX_HIP(hipGetLastError());
  return CX_OK;
}

}  // namespace

// Few tokens leave these kernels a handful of waves, and a P.V chain of ~45 ns a
// position then decides; the kernels of a few tokens (4 a workgroup up to 4096
// cached positions, one a grid slice above) give every chain a wave. Prefill of
// T tokens, 4 layers, these against those (us): 3B shape after 60 positions
// T = 128 770, 745, T = 256 1081, 1124; after 7000 T = 64 2177, 1878, T = 128
// 2462, 3290; 8B shape after 60 T = 64 1287, 1249, T = 128 2125, 2145, after 7000
// T = 32 2527, 3201; 0.5B shape after 60 T = 256 1233, 1233, after 7000 T = 128
// 2558, 2232, T = 256 2880, 3664. The product of tokens and width does not decide
// alone: the line gives up the 8B shape's T = 32 after 7000 positions, whose product
// is that of the 3B shape's T = 64, which the other kernels serve better.
bool cx_attn_many_suits_prefill(size_t tokens, size_t total, size_t heads, size_t hd) {
  return (hd == 64 || hd == 128) &&
         tokens * heads * hd >= (total < 1024 ? 320 * 1024 : 176 * 1024);
}

// Against the general kernel (a workgroup a head and token), us: 16/2 heads x
// 128, 512 positions, 16 tokens 54, 57, 64 tokens 57, 137, 256 tokens 72, 613; 64
// positions, 64 tokens 29, 18; 3000 positions, one token 180, 414.
bool cx_attn_many_suits_general(size_t tokens, size_t total, size_t heads, size_t hd) {
  return (hd == 64 || hd == 128) && (total >= 1024 || tokens * heads * total >= 300000);
}

cx_attn_many_floats cx_attn_many_scratch(size_t tokens, size_t total, size_t heads, size_t kvh) {
  const size_t rows = (tokens * (heads / kvh) + MQ_R - 1) / MQ_R * MQ_R * kvh;
  return {rows * total, rows * ((total + MQ_C - 1) / MQ_C), rows};
}

// 256 MB: 256 tokens at 32 heads and 8000 positions, so that only the largest
// calls take several slabs. 64 tokens are whole tiles of rows whatever the heads
// a group; where they alone are more (128 heads, 8192 positions), as few as fill
// one 64-row tile a group.
size_t cx_attn_many_slab(size_t tokens, size_t total, size_t heads, size_t kvh) {
  constexpr size_t budget = 256ull << 20;
  auto bytes = [&](size_t t) {
    const cx_attn_many_floats f = cx_attn_many_scratch(t, total, heads, kvh);
    return (f.sc + f.cm + f.inv) * 4;
  };
  if (bytes(tokens) <= budget) return tokens;
  size_t slab = 64;
  if (bytes(64) <= budget)
    slab = budget / bytes(64) * 64;
  else
    while (bytes(slab) > budget && slab * (heads / kvh) > MQ_R) slab /= 2;
  return slab < tokens ? slab : tokens;
}

int cx_launch_attn_many(const cx_attn_many_args& a, hipStream_t s) {
  CX_REQUIRE(a.hd == 64 || a.hd == 128, "attention: head_dim %u (64 or 128 supported)", a.hd);
  CX_REQUIRE(a.kvh && a.heads % a.kvh == 0, "attention: %u heads / %u groups", a.heads, a.kvh);
  CX_REQUIRE(a.tokens && a.sc && a.cm && a.inv, "attention: many query tokens need their scratch");
  CX_REQUIRE((((uintptr_t)a.q | (uintptr_t)a.k | (uintptr_t)a.v | (uintptr_t)a.out) & 15) == 0,
             "attention: rows must be 16-byte aligned");
  CX_REQUIRE((size_t)a.tokens * a.heads < (1u << 31) && (size_t)a.pos + a.tokens < (1u << 31),
             "attention: %u query tokens", a.tokens);
  return a.hd == 64 ? launch<64>(a, s) : launch<128>(a, s);
}
