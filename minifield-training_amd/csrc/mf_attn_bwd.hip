// Backward of the segment-masked flash forward on gfx950.
//
// Three deterministic launches (no atomics, fixed reduction order):
//   1. delta:  D[b,h,t] = sum_d dO * O   (fp32), one thread per (b, t, h);
//              the workspace keeps -D and lse2 = lse * log2(e) per row.
//   2. dq:     per 128-query tile (like the forward): recompute
//              S^T = K Q^T and dP^T = V dO^T over the tile's non-empty key
//              stages, P^T = exp2(c S^T - lse2), dS^T = P^T (dP^T - D), and
//              dQ^T += K^T dS^T, with dS^T fed from its accumulator
//              registers as the B operand and K^T read from the natural K
//              tile in LDS by transposing reads.
//   3. dkdv:   per 128-key tile and KV head: K and V stay in registers;
//              for every non-empty query stage and every query head of the
//              GQA group, S = Q K^T and dP = dO V^T (accumulator column =
//              key), then dV^T += dO^T P and dK^T += Q^T dS with dO^T and
//              Q^T read transposed from the Q / dO tiles.  The group's heads
//              are summed in registers, which is the transpose of the
//              reference's jnp.repeat of K/V (kernels/attention.py:19-22).
// The fp32 kernels split the same work finer (32 rows and one head per
// workgroup, the other side over its waves) and use v_mfma_f32_32x32x2_f32.
// Rows with no valid key have lse = +inf, so their P is exactly 0 and they
// contribute nothing; their dq is written as 0.
#include "mf_common.h"
#include "mf_f32.h"
#include "mf_lds.h"

namespace mf {

struct BwdArgs {
  const void* q;
  const void* k;
  const void* v;
  const void* out;
  const void* dout;
  const float* lse;
  float* ndelta;  // workspace: -D per row, [B, Hq, T]
  float* lse2;    // workspace: lse * log2(e) per row, [B, Hq, T]
  void* dq;
  void* dk;
  void* dv;
  const int* qid;
  const int* kid;
  const int* qcnt;
  const int* qlist;
  const int* kcnt;
  const int* klist;
  const int* qorder;
  const int* korder;
  int T, S, Hq, Hkv, G, hchunks;
  int nq, nk, tq_pad, tk_pad;
  int causal;
  int fuse_delta;  // dq computes D = rowsum(dO * O) itself and writes -D and lse2
  float scale, scale_log2;
  FastDiv div_nh, div_hchunks, div_nq, div_hkv, div_nk, div_g, div_hq;  // Hkv * hchunks, hchunks, nq, Hkv, nk, G, Hq
  FastDiv div_qsub, div_ksub;  // row blocks per query and key tile (fp32 units)
};

constexpr int kStep = 64;

// ---------------------------------------------------------------------------
// 1. delta
// ---------------------------------------------------------------------------
template <bool F32>
__global__ __launch_bounds__(256) void bwd_delta_kernel(BwdArgs a, int B) {
  const size_t idx = (size_t)blockIdx.x * blockDim.x + threadIdx.x;  // (b, t, h)
  const size_t total = (size_t)B * a.T * a.Hq;
  if (idx >= total) return;
  const int h = idx % a.Hq;
  const size_t bt = idx / a.Hq;
  const int t = bt % a.T;
  const int b = bt / a.T;
  float acc = 0.f;
  if constexpr (!F32) {
    const bf16* o = reinterpret_cast<const bf16*>(a.out) + idx * kD;
    const bf16* g = reinterpret_cast<const bf16*>(a.dout) + idx * kD;
#pragma unroll
    for (int c8 = 0; c8 < 8; ++c8) {
      const bf16x8 x = ld_bf16x8(o + c8 * 8);
      const bf16x8 y = ld_bf16x8(g + c8 * 8);
#pragma unroll
      for (int e = 0; e < 8; ++e) acc = fmaf((float)x[e], (float)y[e], acc);
    }
  } else {
    const float* o = reinterpret_cast<const float*>(a.out) + idx * kD;
    const float* g = reinterpret_cast<const float*>(a.dout) + idx * kD;
#pragma unroll
    for (int c4 = 0; c4 < 8; ++c4) {  // dims d and 32 + d in turn, as dq adds them
      const f32x4 x0 = *reinterpret_cast<const f32x4*>(o + c4 * 4);
      const f32x4 x1 = *reinterpret_cast<const f32x4*>(o + 32 + c4 * 4);
      const f32x4 y0 = *reinterpret_cast<const f32x4*>(g + c4 * 4);
      const f32x4 y1 = *reinterpret_cast<const f32x4*>(g + 32 + c4 * 4);
#pragma unroll
      for (int e = 0; e < 4; ++e) acc = fmaf(x1[e], y1[e], fmaf(x0[e], y0[e], acc));
    }
  }
  const size_t li = ((size_t)b * a.Hq + h) * a.T + t;
  a.ndelta[li] = -acc;
  a.lse2[li] = a.lse[li] * kLog2e;
}

// ---------------------------------------------------------------------------
// 2. dq, fp32: one workgroup per (32-query block, query head), its four waves
// on every fourth 32-key block of the tile's list, their dQ added through LDS
// in wave order (the fp32 forward's split, for the same reason: the kernel is
// bound by the chain of 64-cycle MFMAs a wave has to run, 96 per block).
// Measured (same box, us per launch, before -> after): 2 x 256 tokens, 4/2
// heads, segments 1-64: 59.9 + 6.7 -> 13.1; 2 x 1499, 16/8 heads, causal, mean
// segment 512: 144 + 8.0 -> 38.8 (the second term is the separate D pass).
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2)))
void bwd_dq_f32_kernel(BwdArgs a) {
  __shared__ F32Tile kt[4], vt[4], qt;  // the waves' K and V blocks; the queries
  const int lane = threadIdx.x & 63;
  const int wave = uniform(threadIdx.x >> 6);
  const int half = lane >> 5, col = lane & 31;
  F32Unit w;
  if (!f32_unit(a.qorder, a.div_hq, a.div_hkv, a.div_qsub, a.div_nq, a.T, a.G, w)) return;
  const int b = w.b, q0 = w.row0;
  const int qpos = q0 + col;
  const int qrow = min(qpos, a.T - 1);
  const int myqid = a.qid[(size_t)b * a.tq_pad + qpos];
  const int u = uniform(myqid);
  const bool quni = __all(myqid == u);
  const bool qactive = qpos < a.T && myqid != 0;

  constexpr size_t kRow = kD * sizeof(float);
  const size_t q_off = ((size_t)b * a.T * a.Hq + w.head) * kRow;
  const uint32_t q_stride = (uint32_t)(a.Hq * kRow);
  f32x4 kx[8], vx[8];  // rows in flight
  f32x4 gf[8];         // the lane's dO operand, through the wave's V tile
  f32_load(reinterpret_cast<const char*>(a.dout) + q_off, q_stride, q0, a.T - 1, lane, vx);
  if (wave == 0)
    f32_load(reinterpret_cast<const char*>(a.q) + q_off, q_stride, q0, a.T - 1, lane, kx);
  f32_store(vt[wave], lane, vx);
  if (wave == 0) f32_store(qt, lane, kx);
  if (a.fuse_delta)
    f32_load(reinterpret_cast<const char*>(a.out) + q_off, q_stride, q0, a.T - 1, lane, kx);
  wave_lds_fence();
#pragma unroll
  for (int j = 0; j < 8; ++j) gf[j] = vt[wave].row4(lane, j);
  const size_t li = ((size_t)b * a.Hq + w.head) * a.T + qrow;
  float nd;  // -D
  if (a.fuse_delta) {
    f32_store(kt[wave], lane, kx);  // O
    wave_lds_fence();
    // D in the order in which the MFMA steps add dP's products (dims d and 32 + d
    // in turn), from zero as dP: where P is near 1 the two cancel, and so then do
    // their rounding errors (dq of one-token segments, whose gradient is zero,
    // was off by 1e-6 with D in another order or dP started from -D, 1e-7 so)
    float part = 0.f;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const f32x4 o0 = kt[wave].row4(col, j), o1 = kt[wave].row4(col + 32, j);
      const f32x4 g0 = vt[wave].row4(col, j), g1 = vt[wave].row4(col + 32, j);
#pragma unroll
      for (int e = 0; e < 4; ++e) part = fmaf(o1[e], g1[e], fmaf(o0[e], g0[e], part));
    }
    nd = -part;
  } else {
    nd = a.ndelta[li];
  }
  const float lse2 = qactive ? a.lse[li] * kLog2e : kPosInf;
  nd = qactive ? nd : 0.f;
  if (a.fuse_delta && wave == 0 && half == 0 && qpos < a.T) {
    a.ndelta[li] = nd;
    a.lse2[li] = lse2;
  }

  f32x16 dqacc[2] = {zero16(), zero16()};
  const float c = a.scale_log2;
  const int* list = a.qlist + ((size_t)b * a.nq + w.tile) * 2 * a.nk;
  const int nb = 2 * ld_const(a.qcnt, b * a.nq + w.tile);  // 32-key blocks
  const int* kid_row = a.kid + (size_t)b * a.tk_pad;
  const char* kg = reinterpret_cast<const char*>(a.k) + ((size_t)b * a.S * a.Hkv + w.kvh) * kRow;
  const char* vg = reinterpret_cast<const char*>(a.v) + ((size_t)b * a.S * a.Hkv + w.kvh) * kRow;
  const uint32_t kv_stride = (uint32_t)(a.Hkv * kRow);

  int kidl = 0, entry = 0, k0 = 0;
  // (as in the forward: stages ascend, so a block past the queries ends it)
  auto fetch = [&](int i) {
    if (i >= nb) return false;
    entry = ld_const(list, i >> 1);
    k0 = (entry >> 2) * kStep + (i & 1) * 32;
    if (a.causal && k0 > q0 + 31) return false;
    kidl = kid_row[k0 + col];
    f32_load(kg, kv_stride, k0, a.S - 1, lane, kx);
    f32_load(vg, kv_stride, k0, a.S - 1, lane, vx);
    return true;
  };
  int i = wave;
  bool more = fetch(i);
  __syncthreads();
  while (more) {
    const int kb = k0;
    bool run = true, mask_ids = false, diag = false;
    if ((entry & 3) == 1) {
      diag = a.causal && kb + 31 > q0;
      mask_ids = true;
      if (quni) {
        const uint64_t same = __ballot(kidl == u);
        run = u != 0 && same != 0;
        mask_ids = same != ~0ull;
      }
    }
    i += 4;
    if (!run) {
      more = fetch(i);
      continue;
    }
    wave_lds_fence();
    f32_store(kt[wave], lane, kx, a.S - kb);
    f32_store(vt[wave], lane, vx, a.S - kb);
    wave_lds_fence();
    more = fetch(i);
    f32x16 s = zero16(), dp = zero16();
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const f32x4 kr = kt[wave].row4(lane, j), qr = qt.row4(lane, j);
      const f32x4 vr = vt[wave].row4(lane, j);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        s = mfma32x32x2(kr[e], qr[e], s);
        dp = mfma32x32x2(vr[e], gf[j][e], dp);
      }
    }
    if (mask_ids) {
#pragma unroll
      for (int g4 = 0; g4 < 4; ++g4) {
        const int4 kids = *reinterpret_cast<const int4*>(&kid_row[kb + 8 * g4 + 4 * half]);
        const int kv[4] = {kids.x, kids.y, kids.z, kids.w};
#pragma unroll
        for (int e = 0; e < 4; ++e) s[g4 * 4 + e] = kv[e] == myqid ? s[g4 * 4 + e] : kNegInf;
      }
    }
    if (diag) {
#pragma unroll
      for (int r = 0; r < 16; ++r) s[r] = kb + acc_row(r, lane) <= qpos ? s[r] : kNegInf;
    }
#pragma unroll
    for (int r = 0; r < 16; ++r) s[r] = fast_exp2(fmaf(s[r], c, -lse2)) * (dp[r] + nd);
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      dqacc[0] = mfma32x32x2(kt[wave].col(lane, 0, r), s[r], dqacc[0]);
      dqacc[1] = mfma32x32x2(kt[wave].col(lane, 1, r), s[r], dqacc[1]);
    }
  }

  wave_lds_fence();
  f32_put(kt[wave], lane, dqacc);
  __syncthreads();
  const int eq = threadIdx.x >> 3, d0 = 8 * (threadIdx.x & 7);
  if (q0 + eq >= a.T) return;
  const bool keep = a.qid[(size_t)b * a.tq_pad + q0 + eq] != 0;
  float* dst = reinterpret_cast<float*>(reinterpret_cast<char*>(a.dq) + q_off +
                                        (size_t)(q0 + eq) * q_stride) + d0;
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    f32x4 o = f32_sum(kt, eq, d0 + 4 * h);
#pragma unroll
    for (int e = 0; e < 4; ++e) o[e] = keep ? o[e] * a.scale : 0.f;
    *reinterpret_cast<f32x4*>(dst + 4 * h) = o;
  }
}

// ---------------------------------------------------------------------------
// 3. dk, dv, fp32: one workgroup per (32-key block, KV head), its eight waves
// on every eighth (32-query block, head of the group) pair, their dK and dV
// added through LDS in wave order.  Eight waves, not
// four: the longest tile's chain of iterations ends the launch.  Measured (as
// above): 73.6 -> 17.4; 215 -> 46.4 (with the rows read from memory in operand
// order: 59.4 with eight waves, 71.4 with four).
// ---------------------------------------------------------------------------
constexpr int kKvWaves = 8;
constexpr int kKvDims = 32 * kD / (64 * kKvWaves);  // outputs per thread

__global__ __launch_bounds__(64 * kKvWaves) __attribute__((amdgpu_waves_per_eu(2)))
void bwd_dkdv_f32_kernel(BwdArgs a) {
  __shared__ F32Tile qt[kKvWaves], gt[kKvWaves];  // the waves' Q and dO blocks
  __shared__ F32Tile kt, vt;
  __shared__ float rows[kKvWaves][2][32];        // per wave: lse2 and -D of the block's queries
  const int lane = threadIdx.x & 63;
  const int wave = uniform(threadIdx.x >> 6);
  const int half = lane >> 5, col = lane & 31;
  F32Unit w;
  if (!f32_unit(a.korder, a.div_hkv, a.div_hkv, a.div_ksub, a.div_nk, a.S, 1, w)) return;
  const int b = w.b, k0 = w.row0, kvh = w.kvh;
  const int kpos = k0 + col;
  const int mykid = a.kid[(size_t)b * a.tk_pad + kpos];
  const int u = uniform(mykid);
  const bool kuni = __all(mykid == u);
  constexpr size_t kRow = kD * sizeof(float);
  const size_t kv_off = ((size_t)b * a.S * a.Hkv + kvh) * kRow;
  const uint32_t kv_stride = (uint32_t)(a.Hkv * kRow);
  if (wave < 2) {
    f32x4 x[8];
    f32_load(reinterpret_cast<const char*>(wave ? a.v : a.k) + kv_off, kv_stride, k0, a.S - 1,
             lane, x);
    f32_store(wave ? vt : kt, lane, x);
  }
  __syncthreads();

  f32x16 dkacc[2] = {zero16(), zero16()}, dvacc[2] = {zero16(), zero16()};
  const float c = a.scale_log2;
  const int* list = a.klist + ((size_t)b * a.nk + w.tile) * 2 * a.nq;
  const int niters = 2 * ld_const(a.kcnt, b * a.nk + w.tile) * a.G;  // (32-query block, head) pairs
  const int* qid_row = a.qid + (size_t)b * a.tq_pad;
  const uint32_t q_stride = (uint32_t)(a.Hq * kRow);
  const char* qg = reinterpret_cast<const char*>(a.q) + (size_t)b * a.T * q_stride;
  const char* gg = reinterpret_cast<const char*>(a.dout) + (size_t)b * a.T * q_stride;

  f32x4 qx[8], gx[8];
  int qidl = 0, entry = 0, q0 = 0, head = 0;
  float rowl = 0.f;  // lse2 (lanes of half 0) or -D (half 1) of row q0 + col
  // the next pair at or after `it` (in steps of kKvWaves) that is not wholly before
  // the keys, and its rows; -1 past the list
  auto fetch = [&](int it) {
    for (; it < niters; it += kKvWaves) {
      const int blk = uniform(fast_div(it, a.div_g));
      entry = ld_const(list, blk >> 1);
      q0 = (entry >> 2) * kStep + (blk & 1) * 32;
      head = kvh * a.G + (it - blk * a.G);
      if (q0 < a.T && !(a.causal && k0 > q0 + 31)) break;
    }
    if (it >= niters) return -1;
    qidl = qid_row[q0 + col];
    f32_load(qg + head * kRow, q_stride, q0, a.T - 1, lane, qx);
    f32_load(gg + head * kRow, q_stride, q0, a.T - 1, lane, gx);
    // (a row past the end: D = 0 and an infinite lse, so P = 0)
    const size_t row = ((size_t)b * a.Hq + head) * a.T;
    const bool in = q0 + col < a.T;
    const uint32_t at = 4u * (uint32_t)min(q0 + col, a.T - 1);
    const float l2 = *reinterpret_cast<const float*>(reinterpret_cast<const char*>(a.lse2 + row) + at);
    const float nd = *reinterpret_cast<const float*>(reinterpret_cast<const char*>(a.ndelta + row) + at);
    rowl = half ? (in ? nd : 0.f) : (in ? l2 : kPosInf);
    return it;
  };
  int it = fetch(wave);
  while (it >= 0) {
    const int qb = q0;
    bool run = true, mask_ids = false, diag = false;
    if ((entry & 3) == 1) {
      diag = a.causal && k0 + 31 > qb;
      mask_ids = true;
      if (kuni) {
        const uint64_t same = __ballot(qidl == u);
        run = u != 0 && same != 0;
        mask_ids = same != ~0ull;
      }
    }
    if (!run) {
      it = fetch(it + kKvWaves);
      continue;
    }
    wave_lds_fence();
    rows[wave][half][col] = rowl;
    f32_store(qt[wave], lane, qx, a.T - qb);
    f32_store(gt[wave], lane, gx, a.T - qb);
    wave_lds_fence();
    it = fetch(it + kKvWaves);
    f32x16 s = zero16(), dp = zero16();
    auto row4 = [&](int which, int g4) {
      return *reinterpret_cast<const f32x4*>(&rows[wave][which][8 * g4 + 4 * half]);
    };
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const f32x4 kr = kt.row4(lane, j), qr = qt[wave].row4(lane, j);
      const f32x4 vr = vt.row4(lane, j), gr = gt[wave].row4(lane, j);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        s = mfma32x32x2(qr[e], kr[e], s);
        dp = mfma32x32x2(gr[e], vr[e], dp);
      }
    }
    if (mask_ids) {
#pragma unroll
      for (int g4 = 0; g4 < 4; ++g4) {
        const int4 ids = *reinterpret_cast<const int4*>(&qid_row[qb + 8 * g4 + 4 * half]);
        const int iv[4] = {ids.x, ids.y, ids.z, ids.w};
#pragma unroll
        for (int e = 0; e < 4; ++e) s[g4 * 4 + e] = iv[e] == mykid ? s[g4 * 4 + e] : kNegInf;
      }
    }
    if (diag) {
#pragma unroll
      for (int r = 0; r < 16; ++r) s[r] = kpos <= qb + acc_row(r, lane) ? s[r] : kNegInf;
    }
#pragma unroll
    for (int g4 = 0; g4 < 4; ++g4) {
      const f32x4 l4 = row4(0, g4), d4 = row4(1, g4);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int r = g4 * 4 + e;
        s[r] = fast_exp2(fmaf(s[r], c, -l4[e]));
        dp[r] = (dp[r] + d4[e]) * s[r];
      }
    }
#pragma unroll
    for (int r = 0; r < 16; ++r)
#pragma unroll
      for (int db = 0; db < 2; ++db) {
        dvacc[db] = mfma32x32x2(gt[wave].col(lane, db, r), s[r], dvacc[db]);
        dkacc[db] = mfma32x32x2(qt[wave].col(lane, db, r), dp[r], dkacc[db]);
      }
  }

  const int etid = 64 * wave + fresh_lane_id();  // (not kept across the loop)
  const int ek = etid / (2 * kKvWaves), d0 = kKvDims * (etid % (2 * kKvWaves));
  const bool in = k0 + ek < a.S;
  const bool keep = a.kid[(size_t)b * a.tk_pad + k0 + ek] != 0;
  const size_t off = kv_off + (size_t)(k0 + ek) * kv_stride + d0 * sizeof(float);
  auto store = [&](void* dst, const F32Tile (&t)[kKvWaves], float mul) {
    if (!in) return;
#pragma unroll
    for (int h = 0; h < kKvDims / 4; ++h) {
      f32x4 o = f32_sum(t, ek, d0 + 4 * h);
#pragma unroll
      for (int e = 0; e < 4; ++e) o[e] = keep ? o[e] * mul : 0.f;
      *reinterpret_cast<f32x4*>(reinterpret_cast<char*>(dst) + off + 16 * h) = o;
    }
  };
  wave_lds_fence();
  f32_put(qt[wave], etid & 63, dkacc);
  f32_put(gt[wave], etid & 63, dvacc);
  __syncthreads();
  store(a.dk, qt, a.scale);
  store(a.dv, gt, 1.f);
}

// ---------------------------------------------------------------------------
// bf16 dq: the structure of the bf16 forward (one head per wave, 4*HPW
// waves, K/V tiles DMA'd into a two-slot LDS ring).
// dQ^T += K^T dS^T takes its K^T operand from the K tile through
// transposing LDS reads.
// ---------------------------------------------------------------------------
template <int HPW, int SLOT>  // SLOT: 64-key stages per ring slot
__global__ __launch_bounds__(256 * HPW) __attribute__((amdgpu_waves_per_eu(HPW < SLOT ? 2 : HPW + 2)))
void bwd_dq_bf16_kernel(BwdArgs a) {
  constexpr int W = 4 * HPW;
  __shared__ __attribute__((aligned(16))) char slotA[SLOT * kStageBytes], slotB[SLOT * kStageBytes];
  const int lane = threadIdx.x & 63;
  const int wave = uniform(threadIdx.x >> 6);
  const int half = lane >> 5;
  // 1-D grid: (query-tile item in launch order, kvh, head chunk), heads fastest
  const int nh = a.Hkv * a.hchunks;
  const int slot = uniform(fast_div(blockIdx.x, a.div_nh));
  const int hr = uniform(blockIdx.x - slot * nh);
  const int kvh = uniform(fast_div(hr, a.div_hchunks));
  const int hc = uniform(hr - kvh * a.hchunks);
  const int item = ld_const(a.qorder, slot);  // (row, query tile), longest first
  const int b = uniform(fast_div(item, a.div_nq));
  const int qt = uniform(item - b * a.nq);
  const int head = kvh * a.G + hc * HPW + (wave >> 2);
  const int qpos = qt * kTile + (wave & 3) * 32 + (lane & 31);
  const int myqid = a.qid[(size_t)b * a.tq_pad + qpos];
  const bool qvalid = qpos < a.T;
  const bool qactive = qvalid && myqid != 0;

  bf16x8 qf[4], gf[4];  // query and output-gradient fragments (loaded below)
  float lse2 = 0.f, dlt = 0.f;
  uint64_t ndlt2 = 0;  // (-D, -D) of the lane's row, the start of each dP^T block
  f32x16 dqacc[2] = {zero16(), zero16()};
  const float c = a.scale_log2;

  const int count = ld_const(a.qcnt, b * a.nq + qt);
  const int* list = a.qlist + ((size_t)b * a.nq + qt) * 2 * a.nk;
  const int nsteps = count;  // one 64-key stage per list entry
  const int tr_row = tr_row_of(lane);
  const int tr_col = tr_col_of(lane);
  const int* kid_row = a.kid + (size_t)b * a.tk_pad;
  const uint32_t row_stride = (uint32_t)a.Hkv * kD * sizeof(bf16);
  const char* kg = reinterpret_cast<const char*>(a.k) + ((size_t)b * a.S * a.Hkv + kvh) * kD * sizeof(bf16);
  const char* vg = reinterpret_cast<const char*>(a.v) + ((size_t)b * a.S * a.Hkv + kvh) * kD * sizeof(bf16);

  // (the precomputed-offset form of kv_dma measured 2-5% slower here while
  // its offsets made dq spill; without spills, at 128 VGPRs, it measures
  // within 0.6%)
  auto issue = [&](int entry, char* stage) {
    kv_dma<W>(kg, vg, row_stride, a.S, kid_row, (entry >> 2) * kKvStep, wave, stage);
  };

  // Sub-block classification inside PARTIAL tiles, as in the forward: a
  // wave's 32 queries against one 32-key block are skipped when no pair can
  // be valid and run without id masks when every id matches.
  const int q0 = qt * kTile + (wave & 3) * 32;
  const int u = uniform(myqid);
  const bool quni = __all(myqid == u);

  auto block = [&](const char* kt, const char* vt, const int* kids_lds, int kb, int kb2,
                   bool mask_ids, bool diag) {
    f32x16 s = zero16();
    f32x16 dp;
    {
      // dP^T starts from -D (per lane: one query row), so the MFMA chain
      // yields dP - D and the 16 subtractions per block go: eight 64-bit
      // moves of the lane's (-D, -D) pair, in asm because the compiler either
      // hoists a sixteen-register splat out of the loop (spilling at 128
      // VGPRs) or emits sixteen 32-bit moves.  s_nop 1 gives the two wait
      // states between a VALU write and an MFMA reading it as SrcC.  The
      // registers written are the block's dP accumulators, which no MFMA in
      // flight reads as SrcC (the previous block's dP chain finished before
      // its probabilities were formed).
      uint64_t p0, p1, p2, p3, p4, p5, p6, p7;
      asm volatile(
          "v_mov_b64 %0, %8\n\tv_mov_b64 %1, %8\n\tv_mov_b64 %2, %8\n\tv_mov_b64 %3, %8\n\t"
          "v_mov_b64 %4, %8\n\tv_mov_b64 %5, %8\n\tv_mov_b64 %6, %8\n\tv_mov_b64 %7, %8\n\t"
          "s_nop 1"
          : "=&v"(p0), "=&v"(p1), "=&v"(p2), "=&v"(p3), "=&v"(p4), "=&v"(p5), "=&v"(p6),
            "=&v"(p7)
          : "v"(ndlt2));
      typedef uint64_t u64x8 __attribute__((ext_vector_type(8)));
      dp = __builtin_bit_cast(f32x16, (u64x8){p0, p1, p2, p3, p4, p5, p6, p7});
    }
    const int krow = kb2 * 32 + (lane & 31);
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) {
      s = mfma32x32x16(tile_chunk(kt, krow, 2 * ks + half), qf[ks], s);
      dp = mfma32x32x16(tile_chunk(vt, krow, 2 * ks + half), gf[ks], dp);
    }
    if (mask_ids) {
#pragma unroll
      for (int g4 = 0; g4 < 4; ++g4) {
        const int4 kids = *reinterpret_cast<const int4*>(&kids_lds[kb2 * 32 + 8 * g4 + 4 * half]);
        const int kv[4] = {kids.x, kids.y, kids.z, kids.w};
#pragma unroll
        for (int i = 0; i < 4; ++i) s[g4 * 4 + i] = kv[i] == myqid ? s[g4 * 4 + i] : kNegInf;
      }
    }
    if (diag) {
#pragma unroll
      for (int r = 0; r < 16; ++r)
        s[r] = kb + kb2 * 32 + acc_row(r, lane) <= qpos ? s[r] : kNegInf;
    }
#pragma unroll
    for (int r = 0; r < 16; ++r) s[r] = fast_exp2(fmaf(s[r], c, -lse2)) * dp[r];
    const bf16x8 ds0 = pack8(s, 0), ds1 = pack8(s, 8);
#pragma unroll
    for (int db = 0; db < 2; ++db) {
      const bf16x8 k0 = tile_tr_operand(kt, kb2 * 32 + tr_row, db * 32 + tr_col);
      const bf16x8 k1 = tile_tr_operand(kt, kb2 * 32 + 16 + tr_row, db * 32 + tr_col);
      dqacc[db] = mfma32x32x16(k0, ds0, dqacc[db]);
      dqacc[db] = mfma32x32x16(k1, ds1, dqacc[db]);
    }
  };

  auto compute = [&](int entry, const char* stage) {
    const int kb = (entry >> 2) * kKvStep;
    const bool partial = (entry & 3) == 1;
    const char* kt = stage;
    const char* vt = stage + kTileBytes;
    const int* kids_lds = reinterpret_cast<const int*>(stage + 2 * kTileBytes);
#pragma unroll
    for (int kb2 = 0; kb2 < 2; ++kb2) {
      bool run = true, mask_ids = false, diag = false;
      if (partial) {
        const int k0 = kb + kb2 * 32;
        const bool above = a.causal && k0 > q0 + 31;
        diag = a.causal && k0 + 31 > q0;
        if (quni) {
          const uint64_t m = __ballot(kids_lds[kb2 * 32 + (lane & 31)] == u);
          run = !above && u != 0 && m != 0;
          mask_ids = m != ~0ull;
        } else {
          run = !above;
          mask_ids = true;
        }
      }
      if (run) block(kt, vt, kids_lds, kb, kb2, mask_ids, diag);
    }
  };

  // Ring of two slots (as in the forward): slot i+1's DMAs are issued right
  // after the barrier that opens slot i; whole pairs of slots, with the
  // computes past the end skipped.
  auto issue_slot = [&](int i, int e0, int e1, char* slot) {
    if (SLOT * i < nsteps) issue(e0, slot);
    if (SLOT == 2 && 2 * i + 1 < nsteps) issue(e1, slot + kStageBytes);
  };
  const int nslots = SLOT == 2 ? (nsteps + 1) >> 1 : nsteps;
  // Both slots and the query-side rows (q, dO, lse, O for D) are in flight
  // together before the first wait; after that slot i+1's DMAs are issued
  // when slot i opens.  The list entries a pair of slots needs (steps
  // 2i .. 2i+5) arrive in one scalar load of eight; the read may run up to 7
  // entries past the list's end, into the plan's next section (query lists
  // are followed by the key-tile counts), and entries at or past nsteps are
  // never used.
  {
    const i32x8u e = ld_const8(list, 0);
    issue_slot(0, e[0], e[1], slotA);
    issue_slot(1, e[SLOT], e[SLOT + 1], slotB);
  }
  {
    const size_t row = (((size_t)b * a.T + min(qpos, a.T - 1)) * a.Hq + head) * kD + 8 * half;
    const bf16* qs = reinterpret_cast<const bf16*>(a.q) + row;
    const bf16* gs = reinterpret_cast<const bf16*>(a.dout) + row;
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) {
      qf[ks] = ld_bf16x8(qs + ks * 16);
      gf[ks] = ld_bf16x8(gs + ks * 16);
    }
  }
  const size_t li = ((size_t)b * a.Hq + head) * a.T + min(qpos, a.T - 1);
  const float lse_raw = a.lse[li];
  float dlt_raw;
  if (a.fuse_delta) {
    // D = rowsum(dO * O): this lane holds half of the row's 64 dims
    const bf16* os = reinterpret_cast<const bf16*>(a.out) +
                     (((size_t)b * a.T + min(qpos, a.T - 1)) * a.Hq + head) * kD + 8 * half;
    float part = 0.f;
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) {
      const u32x4 ow = ld_u32x4(os + ks * 16);
      const u32x4 gw = __builtin_bit_cast(u32x4, gf[ks]);
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        // through scalars: __builtin_bit_cast of a vector element reads
        // element 0 whatever the index (clang 22)
        const uint32_t oj = ow[j], gj = gw[j];
        part = __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2, oj),
                                               __builtin_bit_cast(bf16x2, gj), part, false);
      }
    }
    dlt_raw = halves_sum(part);
  } else {
    dlt_raw = -a.ndelta[li];
  }
  drain_memory();
  lse2 = qactive ? lse_raw * kLog2e : kPosInf;
  dlt = qactive ? dlt_raw : 0.f;
  {
    const uint32_t nd = __builtin_bit_cast(uint32_t, -dlt);
    ndlt2 = ((uint64_t)nd << 32) | nd;
  }
  // (a slot past the end is skipped whole, as in the forward)
  for (int i = 0; i < nslots; i += 2) {
    const i32x8u e = ld_const8(list, SLOT * i);
    wait_vmcnt<0>();
    barrier();
    if (i > 0) issue_slot(i + 1, e[SLOT], e[SLOT + 1], slotB);
    compute(e[0], slotA);
    if (SLOT == 2 && 2 * i + 1 < nsteps) compute(e[1], slotA + kStageBytes);
    if (i + 1 < nslots) {
      wait_vmcnt<0>();
      barrier();
      issue_slot(i + 2, e[2 * SLOT], e[2 * SLOT + 1], slotA);
      compute(e[SLOT], slotB);
      if (SLOT == 2 && 2 * i + 3 < nsteps) compute(e[3], slotB + kStageBytes);
    }
  }
  wait_vmcnt<0>();

  // the lane's query position and half again from a fresh lane id
  // (cheaper than keeping them across the loop)
  const int elane = fresh_lane_id();
  const int ehalf = elane >> 5;
  const int eqpos = qt * kTile + (wave & 3) * 32 + (elane & 31);
  if (eqpos >= a.T) return;
  // -D and lse * log2(e) for the dk/dv kernel, stored after the loop rather
  // than before it (a store in flight would hold up the first stage's wait).
  // The values the loop used: an inactive row's are 0 and +inf, which dk/dv
  // never combines with a non-zero probability.
  if (a.fuse_delta && ehalf == 0) {
    const size_t lj = ((size_t)b * a.Hq + head) * a.T + eqpos;
    a.ndelta[lj] = -dlt;
    a.lse2[lj] = lse2;
  }
  store_bf16_rows(reinterpret_cast<bf16*>(a.dq) + (((size_t)b * a.T + eqpos) * a.Hq + head) * kD,
                  dqacc, a.scale, qactive, ehalf);
}

// ---------------------------------------------------------------------------
// bf16 dk/dv: 4 waves per workgroup for one 128-key tile of one KV head; each
// wave owns 32 keys (K, V as B operands in registers) and walks the GQA
// group's query heads in turn, summing their dK/dV in the same accumulators.
// Q, dO, lse, D and the query ids are DMA'd into a three-stage LDS ring of
// 64-query stages, two steps ahead of use; dV^T += dO^T P and dK^T += Q^T dS
// read their transposed operands from the Q / dO tiles.  Each 32-query block
// runs its scores, VALU and accumulation before the next block starts: that
// keeps the kernel within 168 VGPRs and 51 KB of LDS, i.e. three workgroups
// (12 waves) per CU, which measured 10% faster at C2 and C3 than two
// workgroups with both blocks' scores issued first and the two-slot ring of
// the forward.
// ---------------------------------------------------------------------------
struct QDma {
  static constexpr int W = 4;
  static constexpr int kTiles = 2;                           // Q, dO
  static constexpr int kGroupsPerWave = kTiles * 8 / W;      // 8-row groups
  static constexpr int kWordArrays = 3;                      // lse, D, ids
  // stage layout: tiles [Q, dO], then lse[64], D[64], ids[64]
  static constexpr int kLseOff = kTiles * kTileBytes;
  static constexpr int kDltOff = kLseOff + 256;
  static constexpr int kIdOff = kDltOff + 256;
  static constexpr int kStageBytes = kIdOff + 256;
};

__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(3)))
void bwd_dkdv_bf16_kernel(BwdArgs a) {
  using Q = QDma;
  constexpr int W = Q::W;
  __shared__ __attribute__((aligned(16))) char stage0[Q::kStageBytes], stage1[Q::kStageBytes],
      stage2[Q::kStageBytes];
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = uniform(tid >> 6);
  const int half = lane >> 5;
  // 1-D grid: (key-tile item in launch order, kvh), heads fastest
  const int slot = uniform(fast_div(blockIdx.x, a.div_hkv));
  const int kvh = uniform(blockIdx.x - slot * a.Hkv);
  const int item = ld_const(a.korder, slot);  // (row, key tile), longest first
  const int b = uniform(fast_div(item, a.div_nk));
  const int kt = uniform(item - b * a.nk);
  const int kpos = kt * kTile + (wave & 3) * 32 + (lane & 31);
  const int mykid = a.kid[(size_t)b * a.tk_pad + kpos];

  bf16x8 kf[4], vf[4];
  {
    const size_t row = (((size_t)b * a.S + min(kpos, a.S - 1)) * a.Hkv + kvh) * kD + 8 * half;
    const bf16* ks = reinterpret_cast<const bf16*>(a.k) + row;
    const bf16* vs = reinterpret_cast<const bf16*>(a.v) + row;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      kf[i] = ld_bf16x8(ks + i * 16);
      vf[i] = ld_bf16x8(vs + i * 16);
    }
  }
  drain_memory();
  f32x16 dkacc[2] = {zero16(), zero16()}, dvacc[2] = {zero16(), zero16()};

  const int count = ld_const(a.kcnt, b * a.nk + kt);
  const int* list = a.klist + ((size_t)b * a.nk + kt) * 2 * a.nq;
  const int hps = a.G;             // heads of the group, walked in turn
  const int niters = count * hps;  // (64-query stage, head) iterations
  const float c = a.scale_log2;
  const uint32_t qrow_stride = (uint32_t)a.Hq * kD * sizeof(bf16);

  const char* const qbase = reinterpret_cast<const char*>(a.q);
  const char* const gbase = reinterpret_cast<const char*>(a.dout);
  // DMA of iteration `it` (query rows qb .. qb+63 of one head) into a stage.
  auto issue = [&](int it, char* stage) {
    it = min(it, niters - 1);
    const int si = fast_div(it, a.div_g);  // hps == G
    const int entry = ld_const(list, si);
    const int hj = it - si * hps;
    const int qb = (entry >> 2) * kKvStep;
    // the word arrays first, so the short step wait covers them
    if (wave < Q::kWordArrays) {
      // rows past T re-read row T-1 (finite values); their ids are 0, so
      // every pair they form is masked or belongs to a zeroed inactive key
      const size_t row = ((size_t)b * a.Hq + kvh * a.G + hj) * a.T;
      const void* sbase = wave == 2 ? (const void*)(a.qid + (size_t)b * a.tq_pad + qb)
                          : (wave & 1) ? (const void*)(a.ndelta + row)
                                       : (const void*)(a.lse2 + row);
      const uint32_t voff = 4u * (wave == 2 ? lane : min(qb + lane, a.T - 1));
      char* dst = wave == 2 ? stage + Q::kIdOff
                  : (wave & 1) ? stage + Q::kDltOff
                               : stage + Q::kLseOff;
      dma_word64(sbase, voff, dst);
    }
#pragma unroll
    for (int j = 0; j < Q::kGroupsPerWave; ++j) {
      // 8-row group wave + W j: its tile (W j) / 8 is a compile-time
      // constant, so the Q / dO choice is a register select rather than a
      // reload of the argument
      const int tile = (W * j) >> 3, r0 = 8 * ((wave + W * j) & 7);
      const int h = kvh * a.G + hj;
      const char* base = ((tile & 1) ? gbase : qbase) + ((size_t)b * a.T * a.Hq + h) * kD * sizeof(bf16);
      dma_rows8(base, qrow_stride, qb, r0, a.T - 1, stage + tile * kTileBytes);
    }
  };

  // Sub-block classification inside PARTIAL tiles (mirror of the forward's,
  // with the roles of queries and keys swapped): the wave's 32 keys against
  // one 32-query block are skipped when no pair can be valid and run without
  // id masks when every id matches.
  const int k0 = kt * kTile + (wave & 3) * 32;
  const int uk = uniform(mykid);
  const bool kuni = __all(mykid == uk);

  // One 32-query block in three parts: S = Q K^T and dP - D = dO V^T - D
  // (MFMA, the accumulator starting from the stage's -D), P and dS (VALU),
  // dV^T += dO^T P and dK^T += Q^T dS (MFMA).
  auto scores = [&](const char* qt, const char* gt, const float* ndlt_l, int qb2, f32x16& s,
                    f32x16& dp) {
    s = zero16();
#pragma unroll
    for (int g4 = 0; g4 < 4; ++g4) {
      const float4 d4 = *reinterpret_cast<const float4*>(&ndlt_l[qb2 * 32 + 8 * g4 + 4 * half]);
      dp[g4 * 4 + 0] = d4.x;
      dp[g4 * 4 + 1] = d4.y;
      dp[g4 * 4 + 2] = d4.z;
      dp[g4 * 4 + 3] = d4.w;
    }
    const int qrow = qb2 * 32 + (lane & 31);
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) {
      s = mfma32x32x16(tile_chunk(qt, qrow, 2 * ks + half), kf[ks], s);
      dp = mfma32x32x16(tile_chunk(gt, qrow, 2 * ks + half), vf[ks], dp);
    }
  };
  auto probs = [&](f32x16& s, f32x16& dp, const float* lse_l, const int* qid_l, int qb, int qb2,
                   bool mask_ids, bool diag,
                   bf16x8 (&pf)[2], bf16x8 (&sf)[2]) {
    if (mask_ids) {
#pragma unroll
      for (int g4 = 0; g4 < 4; ++g4) {
        const int4 ids = *reinterpret_cast<const int4*>(&qid_l[qb2 * 32 + 8 * g4 + 4 * half]);
        const int iv[4] = {ids.x, ids.y, ids.z, ids.w};
#pragma unroll
        for (int i = 0; i < 4; ++i) s[g4 * 4 + i] = iv[i] == mykid ? s[g4 * 4 + i] : kNegInf;
      }
    }
    if (diag) {
#pragma unroll
      for (int r = 0; r < 16; ++r)
        s[r] = kpos <= qb + qb2 * 32 + acc_row(r, lane) ? s[r] : kNegInf;
    }
#pragma unroll
    for (int g4 = 0; g4 < 4; ++g4) {
      const float4 l4 = *reinterpret_cast<const float4*>(&lse_l[qb2 * 32 + 8 * g4 + 4 * half]);
      const float lv[4] = {l4.x, l4.y, l4.z, l4.w};
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int r = g4 * 4 + i;
        // lse_l holds lse * log2(e); masked scores are -inf and inactive
        // rows have lse = +inf: p = 0
        const float p = fast_exp2(fmaf(s[r], c, -lv[i]));
        s[r] = p;
        dp[r] *= p;
      }
    }
    pf[0] = pack8(s, 0);
    pf[1] = pack8(s, 8);
    sf[0] = pack8(dp, 0);
    sf[1] = pack8(dp, 8);
  };
  auto accumulate = [&](const char* qt, const char* gt, int qb2, const bf16x8 (&pf)[2],
                        const bf16x8 (&sf)[2]) {
    const int r0 = qb2 * 32 + tr_row_of(lane);
    const int cb = tr_col_of(lane);
#pragma unroll
    for (int db = 0; db < 2; ++db) {
      const bf16x8 g0 = tile_tr_operand(gt, r0, db * 32 + cb);
      const bf16x8 g1 = tile_tr_operand(gt, r0 + 16, db * 32 + cb);
      dvacc[db] = mfma32x32x16(g0, pf[0], dvacc[db]);
      dvacc[db] = mfma32x32x16(g1, pf[1], dvacc[db]);
      const bf16x8 q0 = tile_tr_operand(qt, r0, db * 32 + cb);
      const bf16x8 q1 = tile_tr_operand(qt, r0 + 16, db * 32 + cb);
      dkacc[db] = mfma32x32x16(q0, sf[0], dkacc[db]);
      dkacc[db] = mfma32x32x16(q1, sf[1], dkacc[db]);
    }
  };

  auto compute = [&](int it, const char* stage) {
    const int entry = ld_const(list, fast_div(it, a.div_g));
    const int qb = (entry >> 2) * kKvStep;
    const bool partial = (entry & 3) == 1;
    const char* qt = stage;
    const char* gt = stage + kTileBytes;
    const float* lse_l = reinterpret_cast<const float*>(stage + Q::kLseOff);
    const float* ndlt_l = reinterpret_cast<const float*>(stage + Q::kDltOff);
    const int* qid_l = reinterpret_cast<const int*>(stage + Q::kIdOff);
    bool run[2] = {true, true}, mask_ids[2] = {false, false}, diag[2] = {false, false};
    if (partial) {
#pragma unroll
      for (int qb2 = 0; qb2 < 2; ++qb2) {
        const int q0 = qb + qb2 * 32;
        const bool above = a.causal && k0 > q0 + 31;
        diag[qb2] = a.causal && k0 + 31 > q0;
        if (kuni) {
          const uint64_t m = __ballot(qid_l[qb2 * 32 + (lane & 31)] == uk);
          run[qb2] = !above && uk != 0 && m != 0;
          mask_ids[qb2] = m != ~0ull;
        } else {
          run[qb2] = !above;
          mask_ids[qb2] = true;
        }
      }
    }
    f32x16 s0, dp0, s1, dp1;
    bf16x8 pf[2], sf[2];
    if (run[0]) {
      scores(qt, gt, ndlt_l, 0, s0, dp0);
      probs(s0, dp0, lse_l, qid_l, qb, 0, mask_ids[0], diag[0], pf, sf);
      accumulate(qt, gt, 0, pf, sf);
    }
    if (run[1]) {
      scores(qt, gt, ndlt_l, 1, s1, dp1);
      probs(s1, dp1, lse_l, qid_l, qb, 1, mask_ids[1], diag[1], pf, sf);
      accumulate(qt, gt, 1, pf, sf);
    }
  };

  // Whole groups of three steps; the computes past the end are skipped
  // rather than leaving the loop mid-group (a mid-group exit gives the
  // accumulators three exit paths, resolved with 64-register copies).  Waves
  // below kWordArrays issue one more DMA per step than the others; the step
  // wait uses the tile count, which for them also covers the oldest DMA of
  // the stage issued one step earlier.  (Skipping the steps past the end
  // whole -- their waits, barriers and clamped re-issues of the last stage --
  // measured 1.7-2.2% slower at C2 and within 1% at C3 and C5.)
  constexpr int G = Q::kGroupsPerWave;
  if (niters > 0) {
    issue(0, stage0);
    issue(1, stage1);
  }
  for (int it = 0; it < niters; it += 3) {
    wait_vmcnt<G>();
    barrier();
    issue(it + 2, stage2);
    compute(it, stage0);
    wait_vmcnt<G>();
    barrier();
    issue(it + 3, stage0);
    if (it + 1 < niters) compute(it + 1, stage1);
    wait_vmcnt<G>();
    barrier();
    issue(it + 4, stage1);
    if (it + 2 < niters) compute(it + 2, stage2);
  }
  wait_vmcnt<0>();

  // the lane's row and half from a fresh lane id, as in dq, and its row offset
  // apart from the wave's scalar one (a 64-bit offset per lane spilled three
  // registers across the loop)
  const int elane = fresh_lane_id();
  const bool kactive = mykid != 0;
  const int krow = kt * kTile + (wave & 3) * 32;
  if ((elane & 31) < a.S - krow) {
    const size_t off = (((size_t)b * a.S + krow) * a.Hkv + kvh) * kD;
    const uint32_t lane_off = (elane & 31) * a.Hkv * kD;
    store_bf16_rows(reinterpret_cast<bf16*>(a.dk) + off + lane_off, dkacc, a.scale, kactive,
                    elane >> 5);
    store_bf16_rows(reinterpret_cast<bf16*>(a.dv) + off + lane_off, dvacc, 1.f, kactive,
                    elane >> 5);
  }
}

hipError_t launch_attn_bwd(const void* q, const void* k, const void* v, const void* out,
                           const void* dout, const float* lse, bool f32, int batch, int T, int S,
                           int Hq, int Hkv, int mode, float scale, const void* plan, void* dq,
                           void* dk, void* dv, float* workspace, int phases, hipStream_t stream) {
  BwdArgs a;
  const PlanLayout lay = plan_layout(batch, T, S);
  const char* p = reinterpret_cast<const char*>(plan);
  a.q = q;
  a.k = k;
  a.v = v;
  a.out = out;
  a.dout = dout;
  a.lse = lse;
  a.ndelta = workspace;
  a.lse2 = workspace + (size_t)batch * Hq * T;
  a.dq = dq;
  a.dk = dk;
  a.dv = dv;
  a.qid = reinterpret_cast<const int*>(p + lay.qid);
  a.kid = reinterpret_cast<const int*>(p + lay.kid);
  a.qcnt = reinterpret_cast<const int*>(p + lay.qcnt);
  a.qlist = reinterpret_cast<const int*>(p + lay.qlist);
  a.kcnt = reinterpret_cast<const int*>(p + lay.kcnt);
  a.klist = reinterpret_cast<const int*>(p + lay.klist);
  a.qorder = reinterpret_cast<const int*>(p + lay.qorder);
  a.korder = reinterpret_cast<const int*>(p + lay.korder);
  a.T = T;
  a.S = S;
  a.Hq = Hq;
  a.Hkv = Hkv;
  a.G = Hq / Hkv;
  // dq: two heads per workgroup where the group splits into pairs, one for odd
  // groups (one_stage_slots has their slots).  Small even calls keep two heads:
  // one measured 24 us against 20.5 at 1 x 8192 of short segments and -6 to
  // +5% at others.
  const int hpw = (a.G % 2 == 0) ? 2 : 1;
  a.hchunks = a.G / hpw;
  a.nq = lay.nq;
  a.nk = lay.nk;
  a.tq_pad = lay.tq_pad;
  a.tk_pad = lay.tk_pad;
  a.causal = mode == 0;
  a.scale = scale;
  a.scale_log2 = scale * kLog2e;
  a.div_nh = make_fastdiv(a.Hkv * a.hchunks);
  a.div_hchunks = make_fastdiv(a.hchunks);
  a.div_nq = make_fastdiv(a.nq);
  a.div_hkv = make_fastdiv(a.Hkv);
  a.div_nk = make_fastdiv(a.nk);
  a.div_g = make_fastdiv(a.G);
  a.div_hq = make_fastdiv(Hq);
  a.div_qsub = make_fastdiv(f32_blocks(T));
  a.div_ksub = make_fastdiv(f32_blocks(S));
  const size_t rows = (size_t)batch * T * Hq;
  const unsigned dgrid = (unsigned)((rows + 255) / 256);
  // with both the delta and the dq phase the dq kernel, which holds the dO
  // rows of its queries in registers anyway, also loads O and writes D; the
  // separate delta pass (a full read of O and dO) is skipped
  a.fuse_delta = (phases & 3) == 3;
  if ((phases & 1) && !a.fuse_delta) {
    if (f32)
      hipLaunchKernelGGL((bwd_delta_kernel<true>), dim3(dgrid), dim3(256), 0, stream, a, batch);
    else
      hipLaunchKernelGGL((bwd_delta_kernel<false>), dim3(dgrid), dim3(256), 0, stream, a, batch);
  }
  const dim3 qgrid(Hkv * a.hchunks * batch * lay.nq);
  if (!(phases & 2)) {
  } else if (f32) {
    f32_launch(a.qorder, (size_t)batch * lay.nq, (size_t)f32_blocks(T) * Hq, 256,
               [&](const int* order, unsigned blocks) {
                 a.qorder = order;
                 hipLaunchKernelGGL(bwd_dq_f32_kernel, dim3(blocks), dim3(256), 0, stream, a);
               });
  } else {
    if (hpw == 2)
      hipLaunchKernelGGL((bwd_dq_bf16_kernel<2, 2>), qgrid, dim3(512), 0, stream, a);
    else if (one_stage_slots(mode, a.nq, qgrid.x))
      hipLaunchKernelGGL((bwd_dq_bf16_kernel<1, 1>), qgrid, dim3(256), 0, stream, a);
    else
      hipLaunchKernelGGL((bwd_dq_bf16_kernel<1, 2>), qgrid, dim3(256), 0, stream, a);
  }
  const dim3 kgrid(Hkv * batch * lay.nk);
  if (phases & 4) {
    // 4-wave workgroups, one head at a time: measured 11-32% faster at
    // C2/C3/C5 than 8-wave workgroups whose halves took different heads and
    // summed through LDS, because the workgroups of a CU share no barriers.
    if (f32)
      f32_launch(a.korder, (size_t)batch * lay.nk, (size_t)f32_blocks(S) * Hkv, 64 * kKvWaves,
                 [&](const int* order, unsigned blocks) {
                   a.korder = order;
                   hipLaunchKernelGGL(bwd_dkdv_f32_kernel, dim3(blocks), dim3(64 * kKvWaves), 0,
                                      stream, a);
                 });
    else
      hipLaunchKernelGGL(bwd_dkdv_bf16_kernel, kgrid, dim3(256), 0, stream, a);
  }
  return hipGetLastError();
}

}  // namespace mf
