// Flash-style forward for segment-masked GQA attention on gfx950.
//
// Two kernels: the bf16 one (further below; the benchmarked path) and an
// fp32 one.  Both walk the compacted list of non-empty 64-key stages of a
// 128-query tile (from the block map).
//
// Scores are formed transposed, S^T = K Q^T, so an accumulator column is one
// query: the row max and row sum are in-lane reductions plus one
// v_permlane32_swap, and the exponentiated block is already in the register
// layout of the B operand of O^T += V^T P^T.  PARTIAL stages compare the
// canonical ids (and causality) per element; FULL stages skip the compare.
// Online softmax in base 2 with the logit scale folded into one FMA.
#include "mf_common.h"
#include "mf_f32.h"
#include "mf_lds.h"

namespace mf {

struct FwdArgs {
  const void* q;
  const void* k;
  const void* v;
  void* out;
  float* lse;
  const int* qid;
  const int* kid;
  const int* qcnt;
  const int* qlist;
  const int* qorder;
  int T, S, Hq, Hkv, G, hchunks;
  int nq, nk, tq_pad, tk_pad;
  int causal;
  float scale, scale_log2;
  FastDiv div_nh, div_hchunks, div_nq;  // Hkv * hchunks, hchunks, nq
  FastDiv div_hq, div_hkv, div_qsub;    // Hq, Hkv, row blocks per tile (fp32 units)
  // query prologue fused into the bf16 kernel's query loads (ROPE instances)
  const void* q_gain;           // [64], tensor dtype
  const int32_t* positions;     // [B, T] or null (0 .. T-1 on every row)
  const uint32_t* rope_table;   // [B * T][32] (bf16 cos | bf16 sin << 16)
  float eps;
  float freq[kD / 2];
};

constexpr int kStepK = 64;          // keys per inner step

// ---------------------------------------------------------------------------
// fp32 forward: one workgroup per (32-query block, query head); its four
// waves take every fourth 32-key block of the tile's work list and merge
// their softmax states through LDS at the end (fixed wave order).
//
// Bound: v_mfma_f32_32x32x2_f32, 64 cycles each and 64 of them per 32x32
// block, one dependent chain per wave.  A 128-query x 2-head workgroup (the
// bf16 kernel's shape) leaves the chip idle at the sizes fp32 is used at and
// makes each wave walk the whole list twice over; splitting queries, heads
// and keys gives 16 times the workgroups with a chain an eighth as long, and
// skips the 32x32 blocks no pair of which is valid.  Measured (same box, us
// per launch, before -> after): 2 x 256 tokens, 4/2 heads, segments 1-64:
// 42.5 -> 10.5; 2 x 1499, 16/8 heads, causal, mean segment 512: 105 -> 29.7.
// Each wave stages its own K and V blocks (its keys are nobody else's), the
// next block's rows in flight while it works on this one's.
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2)))
void attn_fwd_f32_kernel(FwdArgs a) {
  __shared__ F32Tile kt[4], vt[4], qt;  // the waves' K and V blocks; the queries
  __shared__ float lm[4][32], ll[4][32];
  const int lane = threadIdx.x & 63;
  const int wave = uniform(threadIdx.x >> 6);
  const int half = lane >> 5, col = lane & 31;
  F32Unit w;
  if (!f32_unit(a.qorder, a.div_hq, a.div_hkv, a.div_qsub, a.div_nq, a.T, a.G, w)) return;
  const int b = w.b, q0 = w.row0, kvh = w.kvh, head = w.head;
  const int qpos = q0 + col;
  const int myqid = a.qid[(size_t)b * a.tq_pad + qpos];
  const int u = uniform(myqid);
  const bool quni = __all(myqid == u);

  constexpr size_t kRow = kD * sizeof(float);
  if (wave == 0) {
    f32x4 x[8];
    f32_load(reinterpret_cast<const char*>(a.q) + ((size_t)b * a.T * a.Hq + head) * kRow,
             (uint32_t)(a.Hq * kRow), q0, a.T - 1, lane, x);
    f32_store(qt, lane, x);
  }

  f32x16 oacc[2] = {zero16(), zero16()};
  float m = kNegInf, l = 0.f;
  const float c = a.scale_log2;
  const int* list = a.qlist + ((size_t)b * a.nq + w.tile) * 2 * a.nk;
  const int nb = 2 * ld_const(a.qcnt, b * a.nq + w.tile);  // 32-key blocks
  const int* kid_row = a.kid + (size_t)b * a.tk_pad;
  const char* kg = reinterpret_cast<const char*>(a.k) + ((size_t)b * a.S * a.Hkv + kvh) * kRow;
  const char* vg = reinterpret_cast<const char*>(a.v) + ((size_t)b * a.S * a.Hkv + kvh) * kRow;
  const uint32_t kv_stride = (uint32_t)(a.Hkv * kRow);

  f32x4 kx[8], vx[8];
  int kidl = 0, entry = 0, k0 = 0;
  // block i's rows; false past the list or, when causal, past the
  // queries (stages ascend, so every later block is past them too)
  auto fetch = [&](int i) {
    if (i >= nb) return false;
    entry = ld_const(list, i >> 1);
    k0 = (entry >> 2) * kStepK + (i & 1) * 32;
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
    f32x16 s = zero16();
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const f32x4 kr = kt[wave].row4(lane, j), qr = qt.row4(lane, j);
#pragma unroll
      for (int e = 0; e < 4; ++e) s = mfma32x32x2(kr[e], qr[e], s);
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
    float mx = s[0];
#pragma unroll
    for (int r = 1; r < 16; ++r) mx = fmaxf(mx, s[r]);
    mx = halves_max(mx);
    if (__any(mx > m)) {
      const float mnew = fmaxf(m, mx);
      const float alpha = mnew == kNegInf ? 1.f : fast_exp2((m - mnew) * c);
      m = mnew;
      l *= alpha;
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        oacc[0][r] *= alpha;
        oacc[1][r] *= alpha;
      }
    }
    const float mc = m == kNegInf ? 0.f : m * c;
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      s[r] = fast_exp2(fmaf(s[r], c, -mc));
      l += s[r];
    }
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      oacc[0] = mfma32x32x2(vt[wave].col(lane, 0, r), s[r], oacc[0]);
      oacc[1] = mfma32x32x2(vt[wave].col(lane, 1, r), s[r], oacc[1]);
    }
  }

  // merge the waves' (max, sum, O): thread = (query, 8 dims)
  l = halves_sum(l);
  if (half == 0) {
    lm[wave][col] = m;
    ll[wave][col] = l;
  }
  wave_lds_fence();
  f32_put(kt[wave], lane, oacc);
  __syncthreads();
  const int eq = threadIdx.x >> 3, d0 = 8 * (threadIdx.x & 7);
  const int eqpos = q0 + eq;
  if (eqpos >= a.T) return;
  float M = lm[0][eq];
#pragma unroll
  for (int x = 1; x < 4; ++x) M = fmaxf(M, lm[x][eq]);
  float wt[4], lt = 0.f;
#pragma unroll
  for (int x = 0; x < 4; ++x) {
    wt[x] = M == kNegInf ? 0.f : fast_exp2((lm[x][eq] - M) * c);
    lt = fmaf(wt[x], ll[x][eq], lt);
  }
  const bool has = a.qid[(size_t)b * a.tq_pad + eqpos] != 0 && lt > 0.f;
  const float inv = has ? 1.f / lt : 0.f;
  if ((threadIdx.x & 7) == 0)
    a.lse[((size_t)b * a.Hq + head) * a.T + eqpos] = has ? fmaf(M, a.scale, __logf(lt)) : kPosInf;
  float* dst = reinterpret_cast<float*>(a.out) + (((size_t)b * a.T + eqpos) * a.Hq + head) * kD + d0;
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    f32x4 o = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int x = 0; x < 4; ++x) o += f32_at(kt[x], eq, d0 + 4 * h) * wt[x];
#pragma unroll
    for (int e = 0; e < 4; ++e) o[e] = has ? o[e] * inv : 0.f;
    *reinterpret_cast<f32x4*>(dst + 4 * h) = o;
  }
}

// ---------------------------------------------------------------------------
// bf16 forward: one head per wave, 4*HPW waves per workgroup.
//
// Wave w serves head hc*HPW + w/4 of the KV group and queries
// [qt*128 + 32 (w%4), +32).  All waves of the workgroup share each 64-key
// step's K and V tiles (the GQA sharing).  The tiles are DMA'd from HBM into a
// two-slot LDS ring of 128-key slots, one slot ahead of use (no staging
// registers); K feeds the S^T = K Q^T MFMAs directly and V^T is read with
// transposing LDS reads.  Rescaling of the output accumulator is lazy: the
// running max used for the exponentials only moves when the true max exceeds
// it by more than 8 in log2 units, so P <= 2^8 and the final division by the
// row sum is unchanged.  Row sums are v_dot2 of the bf16 probabilities with
// (1, 1), a full-rate VALU op that halves the adds.
//
// A workgroup serves HPW heads, four waves each.  Two heads share every K/V
// stage and win where the chip is full.  One head with ring slots of one
// stage (33 KB of LDS, so four workgroups fit a CU, as two two-head ones do)
// is the finer unit; a wave's arithmetic, and so every output bit, is the
// same.  heads_per_block and one_stage_slots have the rules and what they
// measure.
// ---------------------------------------------------------------------------
// The query half of the attention prologue on the query fragments a lane
// holds (dims 16 ks + 8 half .. +7 of one query row, ks = 0..3; the other
// half of the row is in lane ^ 32): RMS normalisation with the per-dimension
// gain, then the rotary embedding, with the arithmetic and the bf16 rounding
// points of qk_norm_rope_kernel step for step, so the fragments equal that
// kernel's output bit for bit.  Its sum of squares adds the fma-chain sums
// of the eight 8-dim chunks as ((c0 + c1) + (c2 + c3)) + ((c7 + c6) + (c5 +
// c4)) (its 8-lane DPP butterfly); here chunk 2 ks + half is this lane's and
// chunk 2 ks + (1 - half) comes from lane ^ 32.  The rotation partner of
// dims 16 ks + .. (ks < 2) is the same lane's fragment ks + 2.  cos and sin
// come from the token's row of the table rope_table_kernel fills.
__device__ __forceinline__ void rope_query(const FwdArgs& a, int b, int qpos, int half,
                                           bf16x8 (&qf)[4]) {
  const int t = min(qpos, a.T - 1);
  // angle pairs of this lane's dims: angles 8 half + i (fragments 0, 2) and
  // 16 + 8 half + i (fragments 1, 3), i < 8
  uint32_t cs[2][8];
  const uint32_t* row = a.rope_table + ((size_t)b * a.T + t) * (kD / 2) + 8 * half;
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    const u32x4 lo = *reinterpret_cast<const u32x4*>(row + 16 * j);
    const u32x4 hi = *reinterpret_cast<const u32x4*>(row + 16 * j + 4);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const uint32_t l = lo[i], h = hi[i];  // through scalars (vector element reads)
      cs[j][i] = l;
      cs[j][4 + i] = h;
    }
  }
  bf16x8 w[4];  // gains of this lane's dims
#pragma unroll
  for (int ks = 0; ks < 4; ++ks)
    w[ks] = ld_bf16x8(reinterpret_cast<const bf16*>(a.q_gain) + 16 * ks + 8 * half);
  // chunk sums: mine[ks] is chunk 2 ks + half, theirs[ks] chunk 2 ks + 1 - half
  float mine[4], theirs[4];
#pragma unroll
  for (int ks = 0; ks < 4; ++ks) {
    float ss = 0.f;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const float x = (float)qf[ks][i];
      ss = fmaf(x, x, ss);
    }
    mine[ks] = ss;
    theirs[ks] = __shfl_xor(ss, 32);
  }
  float c[8];
#pragma unroll
  for (int ks = 0; ks < 4; ++ks) {
    c[2 * ks] = half ? theirs[ks] : mine[ks];
    c[2 * ks + 1] = half ? mine[ks] : theirs[ks];
  }
  const float total = ((c[0] + c[1]) + (c[2] + c[3])) + ((c[7] + c[6]) + (c[5] + c[4]));
  const float inv = rsqrtf(total * (1.f / kD) + a.eps);
  // n = bf16(bf16(x * inv) * gain), kept as bf16 pairs
  uint32_t n[4][4];
#pragma unroll
  for (int ks = 0; ks < 4; ++ks)
#pragma unroll
    for (int i = 0; i < 8; i += 2) {
      const uint32_t y = round_bf16_pair((float)qf[ks][i] * inv, (float)qf[ks][i + 1] * inv);
      n[ks][i / 2] = round_bf16_pair(bf16_lo(y) * (float)w[ks][i], bf16_hi(y) * (float)w[ks][i + 1]);
    }
  auto nval = [&](int ks, int i) { return (i & 1) ? bf16_hi(n[ks][i / 2]) : bf16_lo(n[ks][i / 2]); };
  const bf16x2 ones = __builtin_bit_cast(bf16x2, 0x3F803F80u);
#pragma unroll
  for (int ks = 0; ks < 4; ++ks) {
    const int j = ks & 1;  // angle block of fragment ks
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      // rotate_half: dims < 32 take -n[d + 32], dims >= 32 take n[d - 32]
      const float r = ks < 2 ? -nval(ks + 2, i) : nval(ks - 2, i);
      const float cv = bf16_lo(cs[j][i]), sv = bf16_hi(cs[j][i]);
      const uint32_t pq = round_bf16_pair(nval(ks, i) * cv, r * sv);
      qf[ks][i] = (bf16)__builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2, pq), ones, 0.f,
                                                        false);
    }
  }
}

template <int HPW, int SLOT, bool ROPE>  // SLOT: 64-key stages per ring slot
__global__ __launch_bounds__(256 * HPW) __attribute__((amdgpu_waves_per_eu(HPW < SLOT ? 2 : 4)))
void attn_fwd_bf16_kernel(FwdArgs a) {
  constexpr int W = 4 * HPW;
  __shared__ __attribute__((aligned(16))) char slotA[SLOT * kStageBytes], slotB[SLOT * kStageBytes];
  const int lane = threadIdx.x & 63;
  // scalar wave index: keeps the DMA destinations scalar expressions of the
  // stage arrays, so the compiler sees which stage each DMA writes
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

  bf16x8 qf[4];
  {
    const bf16* src = reinterpret_cast<const bf16*>(a.q) +
                      (((size_t)b * a.T + min(qpos, a.T - 1)) * a.Hq + head) * kD + 8 * half;
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) qf[ks] = ld_bf16x8(src + ks * 16);
  }
  if constexpr (ROPE) rope_query(a, b, qpos, half, qf);
  drain_memory();

  f32x16 oacc[2] = {zero16(), zero16()};
  // Exponentials are taken of x = s*c - shift (base 2).  shift is the running
  // max in log2 units once a valid key was seen (0 before); it only moves
  // when a new max exceeds it by more than `lag` (8 once set, -inf before).
  float shift = 0.f, lag = kNegInf;
  float l0 = 0.f, l1 = 0.f;  // row-sum partials
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

  const KvLanes<W> kv_lane = kv_lanes<W>(row_stride, wave);
  auto issue = [&](int entry, char* stage) {
    kv_dma<W>(kg, vg, row_stride, a.S, kid_row, (entry >> 2) * kStepK, wave, stage, kv_lane);
  };

  // Sub-block classification inside PARTIAL tiles.  A wave's 32 queries
  // against one 32-key block are skipped when no pair can be valid, run
  // without masks when every pair is valid, and masked otherwise (ids only,
  // causal only, or both).  When the wave's query ids are not all equal
  // every block of a PARTIAL tile is masked.
  const int q0 = qt * kTile + (wave & 3) * 32;
  const int u = uniform(myqid);
  const bool quni = __all(myqid == u);

  auto scores = [&](const char* kt, int kb2) {
    f32x16 s = zero16();
    const int krow = kb2 * 32 + (lane & 31);
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) s = mfma32x32x16(tile_chunk(kt, krow, 2 * ks + half), qf[ks], s);
    return s;
  };

  // masks of one block; returns the row max of its raw scores (both halves)
  auto mask_block = [&](f32x16& s, const int* kids_lds, int kb, int kb2, bool mask_ids, bool diag) {
    if (mask_ids) {
#pragma unroll
      for (int g4 = 0; g4 < 4; ++g4) {
        const int kk0 = kb2 * 32 + 8 * g4 + 4 * half;
        const int4 kids = *reinterpret_cast<const int4*>(&kids_lds[kk0]);
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
    float mx = fmaxf(s[0], s[1]);
#pragma unroll
    for (int r = 2; r < 16; r += 2) mx = fmaxf(fmaxf(mx, s[r]), s[r + 1]);
    return mx;
  };
  // probabilities 2^(s c - shift), row sums and O += P V of one block
  auto finish_pv = [&](f32x16& s, const char* vt, int kb2) {
#pragma unroll
    for (int r = 0; r < 16; ++r) s[r] = fast_exp2(fmaf(s[r], c, -shift));
    const bf16x8 p0 = pack8(s, 0), p1 = pack8(s, 8);
    // row sum of the bf16 probabilities that P V uses: one v_dot2 with
    // (1, 1) per pair (copied through scalars: __builtin_bit_cast of a
    // vector element reads element 0 whatever the index, clang 22)
    {
      const u32x4 w0 = __builtin_bit_cast(u32x4, p0), w1 = __builtin_bit_cast(u32x4, p1);
      const bf16x2 ones = __builtin_bit_cast(bf16x2, 0x3F803F80u);
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const uint32_t a0 = w0[j], a1 = w1[j];
        l0 = __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2, a0), ones, l0, false);
        l1 = __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2, a1), ones, l1, false);
      }
    }
#pragma unroll
    for (int db = 0; db < 2; ++db) {
      const bf16x8 v0 = tile_tr_operand(vt, kb2 * 32 + tr_row, db * 32 + tr_col);
      const bf16x8 v1 = tile_tr_operand(vt, kb2 * 32 + 16 + tr_row, db * 32 + tr_col);
      oacc[db] = mfma32x32x16(v0, p0, oacc[db]);
      oacc[db] = mfma32x32x16(v1, p1, oacc[db]);
    }
  };

  // One step = two 32-key blocks.  Both score blocks are issued before any
  // softmax work, so the second block's MFMAs run under the first block's
  // masks and max; both blocks share one shift decision; the first block's
  // P V then runs under the second block's exponentials.
  auto compute = [&](int step, int entry, const char* stage) {
    const int kb = (entry >> 2) * kStepK;
    const bool partial = (entry & 3) == 1;
    const char* kt = stage;
    const char* vt = stage + kTileBytes;
    const int* kids_lds = reinterpret_cast<const int*>(stage + 2 * kTileBytes);
    bool run[2] = {true, true}, mask_ids[2] = {false, false}, diag[2] = {false, false};
    if (partial) {
#pragma unroll
      for (int kb2 = 0; kb2 < 2; ++kb2) {
        const int k0 = kb + kb2 * 32;
        const bool above = a.causal && k0 > q0 + 31;
        diag[kb2] = a.causal && k0 + 31 > q0;
        if (quni) {
          const uint64_t m = __ballot(kids_lds[kb2 * 32 + (lane & 31)] == u);
          run[kb2] = !above && u != 0 && m != 0;
          mask_ids[kb2] = m != ~0ull;
        } else {
          run[kb2] = !above;
          mask_ids[kb2] = true;
        }
      }
    }
    f32x16 s0, s1;
    if (run[0]) s0 = scores(kt, 0);
    if (run[1]) s1 = scores(kt, 1);
    // One shift decision for the step's two blocks, taken on the raw scores
    // before either block's probabilities exist: c > 0 and the rounding of
    // an FMA is monotone, so fma(max s, c, -shift) is exactly the max of the
    // shifted scores.  A growing lane moves its shift to the new max: d > 0
    // and finite, so alpha = 2^-d is finite (a lane with no valid key yet has
    // l = 0, O = 0).  At a tile's first step every lane has l = 0 and O = 0,
    // so the rescale is skipped there.
    float mx = kNegInf;
    if (run[0]) mx = mask_block(s0, kids_lds, kb, 0, mask_ids[0], diag[0]);
    if (run[1]) mx = fmaxf(mx, mask_block(s1, kids_lds, kb, 1, mask_ids[1], diag[1]));
    mx = fmaf(halves_max(mx), c, -shift);
    const bool grow = mx > lag;
    if (__any(grow)) {
      const float d = grow ? mx : 0.f;
      shift += d;
      lag = grow ? 8.f : lag;
      if (step > 0) {
        const float alpha = fast_exp2(-d);
        l0 *= alpha;
        l1 *= alpha;
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          oacc[0][r] *= alpha;
          oacc[1][r] *= alpha;
        }
      }
    }
    if (run[0]) finish_pv(s0, vt, 0);
    if (run[1]) finish_pv(s1, vt, 1);
  };

  // Ring of two slots: the DMAs of slot i+1 are issued right after the barrier
  // that opens slot i, so they have the compute of slot i to land, and one
  // barrier serves a slot.
  auto issue_slot = [&](int i, int e0, int e1, char* slot) {
    if (SLOT * i < nsteps) issue(e0, slot);
    if (SLOT == 2 && 2 * i + 1 < nsteps) issue(e1, slot + kStageBytes);
  };
  const int nslots = SLOT == 2 ? (nsteps + 1) >> 1 : nsteps;
  // The list entries a pair of slots needs (the pair's and the next slot's)
  // arrive in one scalar load of eight, issued before the pair's first wait.
  // The read may run up to 7 entries past the list's end, into the plan's next
  // section (query lists are followed by the key-tile counts); entries at or
  // past nsteps are never used.
  {
    const i32x8u e = ld_const8(list, 0);
    issue_slot(0, e[0], e[1], slotA);
  }
  // Whole pairs of slots; a slot past the end is skipped whole (its wait,
  // barrier and computes; nslots is uniform over the workgroup) rather than
  // leaving the loop mid-pair (a mid-pair exit gives the accumulators two
  // exit paths, resolved with register copies).
  for (int i = 0; i < nslots; i += 2) {
    const i32x8u e = ld_const8(list, SLOT * i);
    wait_vmcnt<0>();
    barrier();
    issue_slot(i + 1, e[SLOT], e[SLOT + 1], slotB);
    compute(SLOT * i, e[0], slotA);
    if (SLOT == 2 && 2 * i + 1 < nsteps) compute(2 * i + 1, e[1], slotA + kStageBytes);
    if (i + 1 < nslots) {
      wait_vmcnt<0>();
      barrier();
      issue_slot(i + 2, e[2 * SLOT], e[2 * SLOT + 1], slotA);
      compute(SLOT * i + SLOT, e[SLOT], slotB);
      if (SLOT == 2 && 2 * i + 3 < nsteps) compute(2 * i + 3, e[3], slotB + kStageBytes);
    }
  }
  wait_vmcnt<0>();  // no DMA may still target this workgroup's LDS at exit

  // the lane's query position and half again from the lane id: recomputing
  // them is cheaper than keeping them (the compiler would spill them) across
  // the loop
  const int elane = fresh_lane_id();
  const int ehalf = elane >> 5;
  const int eqpos = qt * kTile + (wave & 3) * 32 + (elane & 31);
  const bool eqvalid = eqpos < a.T;
  const bool qactive = eqvalid && myqid != 0;
  const float lt = halves_sum(l0 + l1);
  const bool has = qactive && lt > 0.f;
  const float inv = has ? 1.f / lt : 0.f;
  if (eqvalid) {
    // natural-log LSE: shift / log2(e) + ln(l)
    if (ehalf == 0)
      a.lse[((size_t)b * a.Hq + head) * a.T + eqpos] = has ? fmaf(shift, kLn2, __logf(lt)) : kPosInf;
    store_bf16_rows(reinterpret_cast<bf16*>(a.out) +
                        (((size_t)b * a.T + eqpos) * a.Hq + head) * kD,
                    oacc, inv, has, ehalf);
  }
}

// Heads per workgroup of the bf16 forward, even groups (odd ones take one, see
// one_stage_slots): two share every K/V stage; one is the finer unit, and with
// slots of one stage four fit a CU.  What decides is the heads the fullest CU
// gets, ceil(w / 256) of w tile-heads against 2 ceil(w / 512).  They differ up to
// 256 and from 513 to 768, where one head wins.  Where they are equal, one head
// still wins if the tiles' lists differ in length, and loses up to 8 % if they do
// not: it is taken for causal rows of several tiles up to 512, and up to 1024 for
// several rows of at least eight (one row alone keeps the order its own tiles
// come in), where it loses at most 4 % on short segments.  Bidirectional calls
// there, whose lists are equal when a row is one segment, and rows of one tile
// keep two.  us with two heads and with one:
//   1 x 2048 causal, segments 128-1024, 16/8  (w = 256)     26.9 -> 22.1
//   1 x 2048 bidirectional, one segment, 16/8 (256)         41.7 -> 34.2
//   1 x 4096 causal, one segment, 16/8        (512)         77.1 -> 65.9
//   1 x 4096 causal, segments 16-128, 16/8    (512)         11.6 -> 10.7
//   1 x 4096 bidirectional, one segment, 16/8 (512)         82.0 -> 86.2 (two)
//   1 x 4096 bidirectional, 64-1024, 16/8     (512)         48.4 -> 40.4 (two)
//   32 x 128, one segment, 16/8               (512)          8.1 -> 8.3  (two)
//   1 x 5003 causal, one segment, 16/8        (640)          122 -> 102
//   1 x 6000 bidirectional, one segment, 16/8 (752)          219 -> 197
//   6 x 1000 causal, segments 16-128, 16/8    (768)         16.3 -> 14.1
//   48 x 128 causal, one segment, 16/8        (768)         11.7 -> 12.3 (two)
//   1 x 7168 causal, one segment, 16/8        (896)          148 -> 156  (two)
//   1 x 7168 causal, segments 64-1024, 16/8   (896)         34.4 -> 29.7 (two)
//   2 x 3400 causal, one segment, 16/8        (864)         94.6 -> 83.0
//   4 x 2048 causal, one segment, 16/8        (1024)        55.3 -> 50.1
//   4 x 2048 causal, segments 16-128, 16/8    (1024)        16.9 -> 17.7
//   8 x 512 causal, segments 16-512, 32/8     (1024)        20.6 -> 21.6 (two)
//   1 x 4096 bidirectional, one segment, 32/8 (1024)         147 -> 157  (two)
//   4 x 8192, mean segment 512, 16/8          (4096)          98 -> 106  (two)
static int heads_per_block(int G, int mode, int batch, int nq, long long tile_heads) {
  if (G % 2 || tile_heads <= 256) return 1;
  if (nq == 1 || tile_heads > 4 * 256) return 2;
  if (tile_heads > 3 * 256) return mode == 0 && batch > 1 && nq >= 8 ? 1 : 2;
  return mode == 0 || tile_heads > 2 * 256 ? 1 : 2;
}

// Arguments of one forward launch: operands, the plan's sections, shapes and
// the workgroup shape (heads per workgroup).
static FwdArgs fwd_args(const void* q, const void* k, const void* v, int batch, int T, int S,
                        int Hq, int Hkv, int mode, float scale, const void* plan, void* out,
                        float* lse, int* hpw) {
  FwdArgs a = {};
  const PlanLayout lay = plan_layout(batch, T, S);
  const char* p = reinterpret_cast<const char*>(plan);
  a.q = q;
  a.k = k;
  a.v = v;
  a.out = out;
  a.lse = lse;
  a.qid = reinterpret_cast<const int*>(p + lay.qid);
  a.kid = reinterpret_cast<const int*>(p + lay.kid);
  a.qcnt = reinterpret_cast<const int*>(p + lay.qcnt);
  a.qlist = reinterpret_cast<const int*>(p + lay.qlist);
  a.qorder = reinterpret_cast<const int*>(p + lay.qorder);
  a.T = T;
  a.S = S;
  a.Hq = Hq;
  a.Hkv = Hkv;
  a.G = Hq / Hkv;
  *hpw = heads_per_block(a.G, mode, batch, lay.nq, (long long)batch * lay.nq * Hq);
  a.hchunks = a.G / *hpw;
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
  a.div_hq = make_fastdiv(Hq);
  a.div_hkv = make_fastdiv(Hkv);
  a.div_qsub = make_fastdiv(f32_blocks(T));
  return a;
}

template <bool ROPE>
static void launch_fwd_bf16(const FwdArgs& a, int hpw, int mode, dim3 grid, hipStream_t stream) {
  if (hpw == 2)
    hipLaunchKernelGGL((attn_fwd_bf16_kernel<2, 2, ROPE>), grid, dim3(512), 0, stream, a);
  else if (a.G % 2 == 0 || one_stage_slots(mode, a.nq, grid.x))
    hipLaunchKernelGGL((attn_fwd_bf16_kernel<1, 1, ROPE>), grid, dim3(256), 0, stream, a);
  else
    hipLaunchKernelGGL((attn_fwd_bf16_kernel<1, 2, ROPE>), grid, dim3(256), 0, stream, a);
}

hipError_t launch_attn_fwd(const void* q, const void* k, const void* v, bool f32, int batch,
                           int T, int S, int Hq, int Hkv, int mode, float scale,
                           const void* plan, void* out, float* lse, hipStream_t stream) {
  int hpw;
  FwdArgs a = fwd_args(q, k, v, batch, T, S, Hq, Hkv, mode, scale, plan, out, lse, &hpw);
  const dim3 grid(Hkv * a.hchunks * batch * a.nq);
  if (f32) {
    f32_launch(a.qorder, (size_t)batch * a.nq, (size_t)f32_blocks(T) * Hq, 256,
               [&](const int* order, unsigned blocks) {
                 a.qorder = order;
                 hipLaunchKernelGGL(attn_fwd_f32_kernel, dim3(blocks), dim3(256), 0, stream, a);
               });
  } else {
    launch_fwd_bf16<false>(a, hpw, mode, grid, stream);
  }
  return hipGetLastError();
}

// cos and sin of each token's 32 angles f32(position) * freq[i], rounded to
// bf16 and packed (cos in the low half): the values qk_norm_rope_kernel
// computes for the token (the same position, the same sincosf of the same
// single-precision product) and rounds before use.
__global__ __launch_bounds__(256) void rope_table_kernel(FwdArgs a, uint32_t* table, size_t n) {
  const size_t idx = (size_t)blockIdx.x * 256 + threadIdx.x;
  if (idx >= n * (kD / 2)) return;
  const size_t tok = idx / (kD / 2);
  const int i = (int)(idx % (kD / 2));
  const float pos = (float)(a.positions ? a.positions[tok] : (int)(tok % a.T));
  float f = a.freq[0];
#pragma unroll
  for (int j = 1; j < kD / 2; ++j) f = i == j ? a.freq[j] : f;  // no per-lane argument indexing
  float sv, cv;
  sincosf(pos * f, &sv, &cv);
  table[idx] = round_bf16_pair(cv, sv);
}

size_t rope_table_bytes(int B, int T) { return sizeof(uint32_t) * (kD / 2) * (size_t)B * T; }

hipError_t launch_attn_fwd_rope_q(const void* q_raw, const void* k, const void* v,
                                  const void* q_gain, const int32_t* positions, int batch, int T,
                                  int S, int Hq, int Hkv, int mode, float scale, float eps,
                                  float theta, const void* plan, void* table, void* out,
                                  float* lse, hipStream_t stream) {
  int hpw;
  FwdArgs a = fwd_args(q_raw, k, v, batch, T, S, Hq, Hkv, mode, scale, plan, out, lse, &hpw);
  a.q_gain = q_gain;
  a.positions = positions;
  a.rope_table = reinterpret_cast<const uint32_t*>(table);
  a.eps = eps;
  // theta ** (-arange(0, D, 2) / D) in single precision (rotary.py:33-35), as
  // the prologue's launcher computes them
  for (int i = 0; i < kD / 2; ++i) a.freq[i] = powf(theta, -((float)(2 * i) / (float)kD));
  const size_t tokens = (size_t)batch * T;
  hipLaunchKernelGGL(rope_table_kernel, dim3((unsigned)((tokens * (kD / 2) + 255) / 256)),
                     dim3(256), 0, stream, a, reinterpret_cast<uint32_t*>(table), tokens);
  const dim3 grid(Hkv * a.hchunks * batch * a.nq);
  launch_fwd_bf16<true>(a, hpw, mode, grid, stream);
  return hipGetLastError();
}

}  // namespace mf
