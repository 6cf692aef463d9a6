// VSA fine block-sparse attention over a CSR block selection (gfx950, bf16 MFMA 32x32x16).
//
// Tokens are [BH, L, 128] bf16 rows, L = NB * 64 in 64-token blocks. Every kernel is instantiated for the logical
// head dim DH = 128 and DH = 64: at DH = 64 (columns 64..127 zero by contract) it stages only the first 128 bytes
// of each row, runs half the QK^T k-steps and half the 32-column output blocks, and writes zeros past column 64
// (C2 shape at D = 64: forward 2.21 -> 1.76 ms, forward + backward 10.2 -> 7.6 ms). blk_cnt[NB] gives each block's valid
// tokens (valid-first). Query block i of head bh attends to the kv blocks row_ptr / col_idx list for row
// (bh, i), with key columns >= blk_cnt[kv] masked; query rows >= blk_cnt[i] and rows with an empty list get
// O = 0 and lse = -inf. lse is the natural-log row sum. Semantics: reference csrc/vsa/generic/attn_fwd.cu:16-24,
// tests/vsa_reference.py:90-107.
//
// Forward: one workgroup per (query block, head), 4 waves = 2 row groups of 32 queries x 2 key halves of each
// 64-key chunk. Every chunk is staged once in LDS (double-buffered direct global->LDS loads, swizzled 256-byte
// rows) and each wave runs its own online softmax over its 32-key halves (S^T = K Q^T so that exp(S^T) is directly
// the B operand of O^T += V^T P^T); the two key-half states of a row group are merged once at the end through
// LDS. The running max is only moved when a row's new maximum exceeds it by more than 8 (log2 units), which
// keeps the O rescale off the common path without changing the result beyond rounding.
// Task mode (split-KV, reference attn_fwd.cu:216-237): the grid walks (row, beg, end, slot) tasks; slot >= 0
// writes an fp32 normalized partial O and its log2 lse to part_o / part_lse, slot < 0 the final O / lse.
#include "../../include/vsa_hip.h"
#include "common.h"
#include "elem.h"
#include "queues.h"

namespace es {

namespace {

constexpr float LN2 = 0.6931471805599453f;
constexpr float RESCALE_SLACK = 8.0f;

struct VsaFwdArgs {
  const e16_t *q, *k, *v;
  e16_t* out;
  float* lse;
  const int *row_ptr, *col_idx, *blk_cnt;
  const int4* tasks;
  const int* info;  // device task count (task mode)
  float *part_o, *part_lse;
  int* queues;  // the eight row-block queue counters of this launch (queues.h)
  int L, NB, BH, per_xcd, fixed;
  int ld;       // columns of a stored row
  float scale;  // log2(e) / sqrt(D)
};

// (K / V are staged with the inline-assembly transfer dma16. With the compiler-visible buffer-to-LDS builtin the
// compiler cannot tell the next chunk's buffer from this one's and waits for the next chunk's transfers before
// this chunk's V^T reads.)
template <bool TASKS, int DH>
__global__ __launch_bounds__(256, 2) void vsa_fwd_kernel(VsaFwdArgs a) {
  constexpr int NKS = DH / 16, NDB = DH / 32;  // MFMA k-steps of QK^T, 32-column blocks of O (D = 64: the first half)
  __shared__ __attribute__((aligned(16))) char kv_s[2][2][BK * 256];

  int qb, bh, beg, end, slot = -1;
  if (TASKS) {
    if ((int)blockIdx.x >= sload(a.info)) return;
    const int4 tk = a.tasks[blockIdx.x];
    bh = tk.x / a.NB;
    qb = tk.x - bh * a.NB;
    beg = tk.y;
    end = tk.z;
    slot = tk.w;
  } else {
    // XCD-aware, run-time balanced order of (query block, head) (queues.h)
    if (!balanced_item(a.queues, a.fixed, a.per_xcd, a.BH, a.NB, bh, qb)) return;
    const int* rp = a.row_ptr + (size_t)bh * (a.NB + 1) + qb;
    beg = sload(rp);
    end = sload(rp + 1);
  }
  beg = __builtin_amdgcn_readfirstlane(beg);
  end = __builtin_amdgcn_readfirstlane(end);
  const int nc = end - beg;

  const int tid = threadIdx.x, l = tid & 63, hi = l >> 5, lq = l & 31;
  const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int rg = wv & 1, kh = wv >> 1;
  const int qrow = 32 * rg + lq;  // row inside the query block
  const int qcnt = sload(a.blk_cnt + qb);
  const bool qvalid = qrow < qcnt;
  const size_t head = (size_t)bh * a.L;

  const int ld = DH == HD ? HD : a.ld;  // columns of a stored row
  const unsigned head_bytes = (unsigned)((size_t)a.L * ld * 2);
  const srd_t rk = make_srd(a.k + head * ld, head_bytes);
  const srd_t rv = make_srd(a.v + head * ld, head_bytes);
  // this lane's four load rows R = 16 wv + 4 i + l / 16 of a chunk and its swizzled 16-byte chunk in them
  unsigned ld_off[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int P = (wv * 4 + i) * 64 + l, R = P >> 4, g = (P & 15) ^ swz(R);
    ld_off[i] = g < DH / 8 ? (unsigned)(R * ld * 2) + (unsigned)(g * 16) : 0x80000000u;
  }
  auto issue = [&](int b, int sb) {
    const unsigned soff = (unsigned)(b * BK * ld * 2);
    char* kd = kv_s[sb][0] + wv * 4096;
    char* vd = kv_s[sb][1] + wv * 4096;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      dma16(rk, kd + i * 1024, ld_off[i], soff);
      dma16(rv, vd + i * 1024, ld_off[i], soff);
    }
  };

  ev8 qreg[8];
  {
    const e16_t* qp = a.q + (head + (size_t)qb * BK + qrow) * ld;
#pragma unroll
    for (int ks = 0; ks < NKS; ++ks) qreg[ks] = *reinterpret_cast<const ev8*>(qp + 16 * ks + 8 * hi);
  }
  int koff[8];
#pragma unroll
  for (int ks = 0; ks < 8; ++ks) koff[ks] = kh * 8192 + tile_off(lq, 2 * ks + hi);
  int voff[2][4];
  {
    const int g1 = (l >> 4) & 1, sub = (l & 1) * 8, rowA = 4 * hi + ((l & 15) >> 2);
#pragma unroll
    for (int db = 0; db < 4; ++db) {
      voff[0][db] = tile_off(rowA, 4 * db + 2 * g1 + ((l & 3) >> 1)) + sub;
      voff[1][db] = tile_off(rowA + 8, 4 * db + 2 * g1 + ((l & 3) >> 1)) + sub;
    }
  }

  f32x16 o[4];
#pragma unroll
  for (int db = 0; db < 4; ++db) o[db] = f32x16{};
  float lsum = 0.0f, mref = -INFINITY;
  const float scale = a.scale;

  int bcur = nc > 0 ? sload(a.col_idx + beg) : 0;
  int ccur = nc > 0 ? sload(a.blk_cnt + bcur) : 0;
  int bnext = nc > 1 ? sload(a.col_idx + beg + 1) : 0;
  if (nc > 0) issue(bcur, 0);
  wait_vmem();
  __syncthreads();

  for (int j = 0; j < nc; ++j) {
    const int sb = j & 1;
    int cnext = 0, bnn = 0;
    if (j + 1 < nc) {
      issue(bnext, sb ^ 1);
      cnext = sload(a.blk_cnt + bnext);
      if (j + 2 < nc) bnn = sload(a.col_idx + beg + j + 2);
    }
    const char* kb = kv_s[sb][0];
    const char* vb = kv_s[sb][1] + kh * 8192;
    f32x16 s = {};
#pragma unroll
    for (int ks = 0; ks < NKS; ++ks) s = emfma(elds16(kb, koff[ks]), qreg[ks], s);
    // the maximum is taken on the raw products (scale > 0: max(s) * scale is the maximum of the scaled logits, the
    // rounding being monotone), and the scaling is folded into the multiply-add in front of each exponential
    if (ccur < BK) {  // key columns past the block's valid tokens
#pragma unroll
      for (int r = 0; r < 16; ++r)
        if (32 * kh + 8 * (r / 4) + 4 * hi + (r % 4) >= ccur) s[r] = -INFINITY;
    }
    float mx = s[0];
#pragma unroll
    for (int r = 1; r < 16; ++r) mx = fmaxf(mx, s[r]);
    mx = max_xor32(mx) * scale;
    if (__builtin_amdgcn_ballot_w64(mx > mref + RESCALE_SLACK) != 0) {
      const float mnew = fmaxf(mref, mx);
      const float alpha = mref == -INFINITY ? 0.0f : exp2f_fast(mref - mnew);
      lsum *= alpha;
#pragma unroll
      for (int db = 0; db < 4; ++db)
#pragma unroll
        for (int r = 0; r < 16; ++r) o[db][r] *= alpha;
      mref = mnew;
    }
    const float msub = mref == -INFINITY ? 0.0f : mref;
    float p[16];
#pragma unroll
    for (int r = 0; r < 16; ++r) p[r] = exp2f_fast(fmaf(s[r], scale, -msub));
    const ev8 pa = epack8(&p[0]), pb = epack8(&p[8]);
    lsum += esum8(pb, esum8(pa, 0.0f));
#pragma unroll
    for (int db = 0; db < NDB; ++db) {
      o[db] = emfma(ecat_tr(lds_read_tr(vb, voff[0][db]), lds_read_tr(vb, voff[1][db])), pa, o[db]);
      o[db] = emfma(ecat_tr(lds_read_tr(vb + 4096, voff[0][db]), lds_read_tr(vb + 4096, voff[1][db])), pb, o[db]);
    }
    wait_vmem();
    __syncthreads();
    bcur = bnext;
    ccur = cnext;
    bnext = bnn;
  }

  // merge the two key halves of each row group: kh = 1 waves hand (m, l, O) to the kh = 0 waves through LDS
  float* xo = reinterpret_cast<float*>(&kv_s[0][0][0]) + rg * (64 * 64);        // [64 regs][64 lanes]
  float* xm = reinterpret_cast<float*>(&kv_s[1][0][0]) + rg * 128;              // [m | l][64 lanes]
  const float ltot = sum_xor32(lsum);
  if (kh == 1) {
#pragma unroll
    for (int db = 0; db < NDB; ++db)
#pragma unroll
      for (int r = 0; r < 16; ++r) xo[(db * 16 + r) * 64 + l] = o[db][r];
    xm[l] = mref;
    xm[64 + l] = ltot;
  }
  __syncthreads();
  if (kh == 1) return;
  const float m1 = xm[l], l1 = xm[64 + l];
  const float M = fmaxf(mref, m1);
  const float a0 = mref == -INFINITY ? 0.0f : exp2f_fast(mref - M);
  const float a1 = m1 == -INFINITY ? 0.0f : exp2f_fast(m1 - M);
  const float lt = a0 * ltot + a1 * l1;
  const bool live = qvalid && lt > 0.0f;
  const float inv = live ? 1.0f / lt : 0.0f;
  const size_t tok = head + (size_t)qb * BK + qrow;
  const float lse2 = live ? M + log2f(lt) : -INFINITY;
  if (!TASKS || slot < 0) {
    e16_t* orow = a.out + tok * ld;
#pragma unroll
    for (int db = 0; db < 4; ++db)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        if (DH < HD && 32 * db >= ld) break;
        ushort4 v4;
        v4 = ushort4{0, 0, 0, 0};
        if (db < NDB) {
          v4.x = f2e((a0 * o[db][4 * i + 0] + a1 * xo[(db * 16 + 4 * i + 0) * 64 + l]) * inv);
          v4.y = f2e((a0 * o[db][4 * i + 1] + a1 * xo[(db * 16 + 4 * i + 1) * 64 + l]) * inv);
          v4.z = f2e((a0 * o[db][4 * i + 2] + a1 * xo[(db * 16 + 4 * i + 2) * 64 + l]) * inv);
          v4.w = f2e((a0 * o[db][4 * i + 3] + a1 * xo[(db * 16 + 4 * i + 3) * 64 + l]) * inv);
        }
        *reinterpret_cast<ushort4*>(orow + 32 * db + 8 * i + 4 * hi) = v4;
      }
    if (hi == 0) a.lse[tok] = live ? lse2 * LN2 : -INFINITY;
  } else {
    float* prow = a.part_o + ((size_t)slot * BK + qrow) * ld;
#pragma unroll
    for (int db = 0; db < 4; ++db)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        if (DH < HD && 32 * db >= ld) break;
        float4 v4 = make_float4(0.f, 0.f, 0.f, 0.f);
        if (db < NDB) {
          v4.x = (a0 * o[db][4 * i + 0] + a1 * xo[(db * 16 + 4 * i + 0) * 64 + l]) * inv;
          v4.y = (a0 * o[db][4 * i + 1] + a1 * xo[(db * 16 + 4 * i + 1) * 64 + l]) * inv;
          v4.z = (a0 * o[db][4 * i + 2] + a1 * xo[(db * 16 + 4 * i + 2) * 64 + l]) * inv;
          v4.w = (a0 * o[db][4 * i + 3] + a1 * xo[(db * 16 + 4 * i + 3) * 64 + l]) * inv;
        }
        *reinterpret_cast<float4*>(prow + 32 * db + 8 * i + 4 * hi) = v4;
      }
    if (hi == 0) a.part_lse[(size_t)slot * BK + qrow] = lse2;
  }
}


// ------------------------------------------------------------------------------------------------ backward
// Per selected pair (query block i, kv block j), with P = exp(S / sqrt(D) - lse) and dS = P (dP - delta) / sqrt(D)
// (reference csrc/vsa/generic/attn_bwd.cu:1-34; rows with lse = -inf and key columns >= blk_cnt get P = 0):
//   KV owner (dK, dV; k2q lists): one workgroup per (kv block, head), 4 waves = 2 key halves x 2 query halves of
//     each staged query block. S = Q K^T and dP = dO V^T come out with keys on lanes, so P and dS are directly the
//     B operands of dV^T += dO^T P and dK^T += Q^T dS (dO^T / Q^T through transposed LDS reads). K and V stay in
//     registers; Q, dO, lse and delta of each listed query block stream through LDS. 4 products per pair.
//   Q owner (dQ; q2k lists): the forward's layout. S^T = K Q^T, dP^T = V dO^T, dQ^T += K^T dS^T with K^T through
//     transposed LDS reads. 3 products per pair; dQ is deterministic (no atomics).
// The two partial accumulators of a workgroup (query halves, or key halves) are summed once at the end in LDS.
struct VsaBwdArgs {
  const e16_t *q, *k, *v, *dout;
  const float *lse, *delta;
  const int *row_ptr, *col_idx, *blk_cnt;
  const int4* tasks;
  const int* info;
  const float *add_a, *add_b;  // per-block gradients distributed as add / cnt (KV owner: dK, dV; Q owner: dQ)
  int add_nb;
  e16_t *out_a, *out_b;       // bf16 outputs
  float *out_a32, *out_b32;    // fp32 outputs (KV owner) / accumulator dq_acc += dQ (Q owner)
  float *part_a, *part_b;      // split partials [slot, 64, D]
  int* queues;                 // the eight row-block queue counters of this launch (queues.h)
  int L, NB, BH, per_xcd, fixed;
  int ld;                      // columns of a stored row
  float scale_log2, scale;
};

// decode the workgroup's (owner block, head, list range, slot); false = nothing to do
template <bool TASKS>
__device__ __forceinline__ bool owner_of(const VsaBwdArgs& a, int& blk, int& bh, int& beg, int& end, int& slot) {
  slot = -1;
  if (TASKS) {
    if ((int)blockIdx.x >= sload(a.info)) return false;
    const int4 tk = a.tasks[blockIdx.x];
    bh = tk.x / a.NB;
    blk = tk.x - bh * a.NB;
    beg = tk.y;
    end = tk.z;
    slot = tk.w;
  } else {
    if (!balanced_item(a.queues, a.fixed, a.per_xcd, a.BH, a.NB, bh, blk)) return false;
    const int* rp = a.row_ptr + (size_t)bh * (a.NB + 1) + blk;
    beg = sload(rp);
    end = sload(rp + 1);
  }
  beg = __builtin_amdgcn_readfirstlane(beg);
  end = __builtin_amdgcn_readfirstlane(end);
  return true;
}

// lse (natural) -> log2 domain, +inf for rows that must get P = 0
__device__ __forceinline__ float lse_to_log2(float lse) { return lse == -INFINITY ? INFINITY : lse * LOG2E; }

// The KV-owner backward: one 256-thread workgroup per (kv block, head), two per CU. Wave (key half, query half) owns a
// 32 x 32 tile of every staged query block and runs all four products on it: S = Q K^T and P, dV += P^T dO, dP = dO V^T
// and dS, dK += dS^T Q, with K and V of its keys in registers; 32 matrix instructions per wave and chunk and one
// barrier. The two query halves' sums are added once at the end. Both accumulator sets and both operand rows need 192 of
// the 256 registers that two waves per SIMD leave; what else is loop-invariant (LDS and transfer offsets) is therefore
// rebuilt from one register each by XOR, and lse and delta go to LDS without passing through registers. (At D = 128 thirteen
// registers, sixteen in the task form, still spill: 52 bytes of scratch a lane, outside the chunk loop.) What bounds it
// is each wave's chain of products and exponentials per chunk, as in the forward. Against a dV wave and a dK wave per
// key half that handed P over through LDS with a second barrier: 4256 -> 3625 us at 480 blocks, 24 heads, top 60
// (666 -> 800 TFLOP/s; 3690 to 3730 on other cards), 604 -> 540 at 240 blocks, 12 heads, top 24; at D = 64, 3187 -> 2400.
template <bool TASKS, int DH>
__global__ __launch_bounds__(256, 2) void vsa_bwd_kv_kernel(VsaBwdArgs a) {
  constexpr int NKS = DH / 16, NDB = DH / 32;
  __shared__ __attribute__((aligned(16))) char qd_s[2][2][BK * 256];  // [buffer][Q | dO]
  __shared__ __attribute__((aligned(16))) float st_s[2][2][BK];       // [buffer][lse2 (+inf: P = 0) | delta]
  __shared__ float lse_s[BK];                                         // the next block's lse as stored
  int kb, bh, beg, end, slot;
  if (!owner_of<TASKS>(a, kb, bh, beg, end, slot)) return;
  const int nc = end - beg;
  const int tid = threadIdx.x, l = tid & 63, hi = l >> 5, lq = l & 31;
  const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int qh = wv >> 1, kh = wv & 1;
  const int key = 32 * kh + lq;
  const int kcnt = sload(a.blk_cnt + kb);
  const bool kvalid = key < kcnt;
  const size_t head = (size_t)bh * a.L;

  const int ld = DH == HD ? HD : a.ld;  // columns of a stored row
  const unsigned head_bytes = (unsigned)((size_t)a.L * ld * 2);
  const srd_t rq = make_srd(a.q + head * ld, head_bytes);
  const srd_t rd = make_srd(a.dout + head * ld, head_bytes);
  // transfer r of a wave moves rows 16 wv + 4 r + l / 16: this lane's source offset is ld_off ^ 16 r plus 4 r rows
  unsigned ld_off;
  {
    const int g = (l & 15) ^ ((l >> 4) << 2);
    ld_off = g < DH / 8 ? (unsigned)((wv * 16 + (l >> 4)) * ld * 2) + (unsigned)(g * 16) : 0x80000000u;
  }
  ev8 kreg[8], vreg[8];  // this lane's key row
  {
    const size_t off = (head + (size_t)kb * BK + key) * ld + 8 * hi;
#pragma unroll
    for (int ks = 0; ks < NKS; ++ks) {
      kreg[ks] = *reinterpret_cast<const ev8*>(a.k + off + 16 * ks);
      vreg[ks] = *reinterpret_cast<const ev8*>(a.v + off + 16 * ks);
    }
  }
  // stage query block i: Q and dO (16 rows of each per wave), and, wave 0, its 64 delta and raw lse values, which
  // `stats` turns into what the exponent subtracts once the transfers have landed
  const srd_t rl = make_srd(a.lse + head, (unsigned)a.L * 4u);
  const srd_t re = make_srd(a.delta + head, (unsigned)a.L * 4u);
  auto issue = [&](int i, int sb) {
    const unsigned soff = (unsigned)(i * BK * ld * 2);
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      dma16(rq, qd_s[sb][0] + wv * 4096 + r * 1024, ld_off ^ (16u * r), soff + (unsigned)(8 * r * ld));
      dma16(rd, qd_s[sb][1] + wv * 4096 + r * 1024, ld_off ^ (16u * r), soff + (unsigned)(8 * r * ld));
    }
    if (wv == 0) {
      dma4(rl, lse_s, 4u * l, (unsigned)i * (BK * 4));
      dma4(re, st_s[sb][1], 4u * l, (unsigned)i * (BK * 4));
    }
  };
  auto stats = [&](int sb) {  // wave 0, after dma_wait()
    st_s[sb][0][l] = lse_to_log2(lse_s[l]);
  };
  // LDS offsets of this wave's query half: row reads of k-step ks at aoff ^ 32 ks, transposed reads of channel block
  // db at toff ^ 64 db (exact: the swizzle is an XOR of the 16-byte chunk), so two registers hold what would be
  // sixteen; the chunk loop fits its two accumulator sets and both operand rows in 256 registers that way
  int aoff = qh * 8192 + tile_off(lq, hi);
  int toff0, toff1;
  {
    const int g1 = (l >> 4) & 1, sub = (l & 1) * 8, rowA = 4 * hi + ((l & 15) >> 2);
    toff0 = qh * 8192 + tile_off(rowA, 2 * g1 + ((l & 3) >> 1)) + sub;
    toff1 = qh * 8192 + tile_off(rowA + 8, 2 * g1 + ((l & 3) >> 1)) + sub;
  }
  f32x16 acc_v[4], acc_k[4];  // this lane's key: dV and dK over this query half
#pragma unroll
  for (int db = 0; db < 4; ++db) acc_v[db] = acc_k[db] = f32x16{};

  int inext = nc > 1 ? sload(a.col_idx + beg + 1) : 0;
  if (nc > 0) {
    issue(sload(a.col_idx + beg), 0);
    dma_wait();
    if (wv == 0) stats(0);
  }
  dma_wait();
  __syncthreads();
  // masked key columns: every row's lse2 becomes +inf for this lane, so P = 2^(s - inf) = 0 without a branch
  const float kmask = kvalid ? 0.0f : INFINITY;
  for (int j = 0; j < nc; ++j) {
    const int sb = j & 1;
    int inn = 0;
    if (j + 1 < nc) {
      issue(inext, sb ^ 1);
      if (j + 2 < nc) inn = sload(a.col_idx + beg + j + 2);
    }
    asm volatile("" : "+v"(aoff), "+v"(toff0), "+v"(toff1), "+v"(ld_off));  // (keeps the offsets from being hoisted)
    const char* qt = qd_s[sb][0];
    const char* dt = qd_s[sb][1];
    auto product = [&](const char* xt, const ev8& xa, const ev8& xb, f32x16 (&acc)[4]) {  // acc += xt^T [xa | xb]
#pragma unroll
      for (int db = 0; db < NDB; ++db) {
        const int t0 = toff0 ^ (64 * db), t1 = toff1 ^ (64 * db);
        acc[db] = emfma(ecat_tr(lds_read_tr(xt, t0), lds_read_tr(xt, t1)), xa, acc[db]);
        acc[db] = emfma(ecat_tr(lds_read_tr(xt + 4096, t0), lds_read_tr(xt + 4096, t1)), xb, acc[db]);
      }
    };
    f32x16 s = {}, dp = {};
#pragma unroll
    for (int ks = 0; ks < NKS; ++ks) s = emfma(elds16(qt, aoff ^ (32 * ks)), kreg[ks], s);
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      const f32x4 l4 = *reinterpret_cast<const f32x4*>(&st_s[sb][0][32 * qh + 8 * g + 4 * hi]);
#pragma unroll
      for (int e = 0; e < 4; ++e) s[4 * g + e] = exp2f_fast(fmaf(s[4 * g + e], a.scale_log2, -(l4[e] + kmask)));
    }
    {
      float p[16];
#pragma unroll
      for (int r = 0; r < 16; ++r) p[r] = s[r];
      product(dt, epack8(&p[0]), epack8(&p[8]), acc_v);
    }
    __builtin_amdgcn_sched_barrier(0);  // (dP after dV: raised above it, its operands do not fit the registers)
#pragma unroll
    for (int ks = 0; ks < NKS; ++ks) dp = emfma(elds16(dt, aoff ^ (32 * ks)), vreg[ks], dp);
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      const f32x4 d4 = *reinterpret_cast<const f32x4*>(&st_s[sb][1][32 * qh + 8 * g + 4 * hi]);
#pragma unroll
      for (int e = 0; e < 4; ++e) s[4 * g + e] = s[4 * g + e] * (dp[4 * g + e] - d4[e]) * a.scale;
    }
    {
      float ds[16];
#pragma unroll
      for (int r = 0; r < 16; ++r) ds[r] = s[r];
      product(qt, epack8(&ds[0]), epack8(&ds[8]), acc_k);
    }
    dma_wait();
    if (j + 1 < nc && wv == 0) stats(sb ^ 1);
    __syncthreads();
    inext = inn;
  }

  // the second query half hands its sums over through the staging buffers: [key half][dV | dK][register][lane]
  float* xch = reinterpret_cast<float*>(&qd_s[0][0][0]) + kh * (128 * 64);
  if (qh == 1) {
#pragma unroll
    for (int db = 0; db < NDB; ++db)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        xch[(db * 16 + r) * 64 + l] = acc_v[db][r];
        xch[(64 + db * 16 + r) * 64 + l] = acc_k[db][r];
      }
  }
  __syncthreads();
  if (qh == 1) return;
#pragma unroll
  for (int db = 0; db < NDB; ++db)
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      acc_v[db][r] += xch[(db * 16 + r) * 64 + l];
      acc_k[db][r] += xch[(64 + db * 16 + r) * 64 + l];
    }
  const size_t tok = head + (size_t)kb * BK + key;
  // valid keys: dK and dV + add / cnt; padding keys: 0; split chunks: fp32 partials without the add
  const float inv = kvalid ? 1.0f / (float)kcnt : 0.0f;
  const float keep = kvalid ? 1.0f : 0.0f;
  auto store = [&](const f32x16 (&acc)[4], const float* add, float* part, float* out32, e16_t* out16) {
    const float* adp = add + ((size_t)bh * a.add_nb + kb) * ld;
#pragma unroll
    for (int db = 0; db < 4; ++db)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        if (DH < HD && 32 * db >= ld) break;
        const int c = 32 * db + 8 * i + 4 * hi;
        f32x4 x4 = {};
        if (db < NDB)  // (columns past D: zero)
          x4 = f32x4{acc[db][4 * i], acc[db][4 * i + 1], acc[db][4 * i + 2], acc[db][4 * i + 3]};
        if (TASKS && slot >= 0) {
          *reinterpret_cast<f32x4*>(part + ((size_t)slot * BK + key) * ld + c) = x4;
          continue;
        }
        x4 *= keep;
        if (add != nullptr) x4 += *reinterpret_cast<const f32x4*>(adp + c) * inv;
        if (out32 != nullptr) {
          *reinterpret_cast<f32x4*>(out32 + tok * ld + c) = x4;
        } else {
          ushort4 o4;
          o4.x = f2e(x4[0]); o4.y = f2e(x4[1]); o4.z = f2e(x4[2]); o4.w = f2e(x4[3]);
          *reinterpret_cast<ushort4*>(out16 + tok * ld + c) = o4;
        }
      }
  };
  store(acc_k, a.add_a, a.part_a, a.out_a32, a.out_a);
  store(acc_v, a.add_b, a.part_b, a.out_b32, a.out_b);
}


template <bool TASKS, int DH>
__global__ __launch_bounds__(256, 2) void vsa_bwd_q_kernel(VsaBwdArgs a) {
  constexpr int NKS = DH / 16, NDB = DH / 32;
  __shared__ __attribute__((aligned(16))) char kv_s[2][2][BK * 256];
  int qb, bh, beg, end, slot;
  if (!owner_of<TASKS>(a, qb, bh, beg, end, slot)) return;
  const int nc = end - beg;
  const int tid = threadIdx.x, l = tid & 63, hi = l >> 5, lq = l & 31;
  const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int rg = wv & 1, kh = wv >> 1;
  const int qrow = 32 * rg + lq;
  const int qcnt = sload(a.blk_cnt + qb);
  const bool qvalid = qrow < qcnt;
  const size_t head = (size_t)bh * a.L;
  const size_t tok = head + (size_t)qb * BK + qrow;

  const int ld = DH == HD ? HD : a.ld;  // columns of a stored row
  ev8 qreg[8], dreg[8];
#pragma unroll
  for (int ks = 0; ks < NKS; ++ks) {
    qreg[ks] = *reinterpret_cast<const ev8*>(a.q + tok * ld + 16 * ks + 8 * hi);
    dreg[ks] = *reinterpret_cast<const ev8*>(a.dout + tok * ld + 16 * ks + 8 * hi);
  }
  const float ls = qvalid ? lse_to_log2(a.lse[tok]) : INFINITY;
  const float dl = a.delta[tok];

  const unsigned head_bytes = (unsigned)((size_t)a.L * ld * 2);
  const srd_t rk = make_srd(a.k + head * ld, head_bytes);
  const srd_t rv = make_srd(a.v + head * ld, head_bytes);
  unsigned ld_off[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int P = (wv * 4 + i) * 64 + l, R = P >> 4, g = (P & 15) ^ swz(R);
    ld_off[i] = g < DH / 8 ? (unsigned)(R * ld * 2) + (unsigned)(g * 16) : 0x80000000u;
  }
  auto issue = [&](int b, int sb) {
    const unsigned soff = (unsigned)(b * BK * ld * 2);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      dma16(rk, kv_s[sb][0] + wv * 4096 + i * 1024, ld_off[i], soff);
      dma16(rv, kv_s[sb][1] + wv * 4096 + i * 1024, ld_off[i], soff);
    }
  };
  int koff[8];
#pragma unroll
  for (int ks = 0; ks < 8; ++ks) koff[ks] = kh * 8192 + tile_off(lq, 2 * ks + hi);
  int toff[2][4];
  {
    const int g1 = (l >> 4) & 1, sub = (l & 1) * 8, rowA = 4 * hi + ((l & 15) >> 2);
#pragma unroll
    for (int db = 0; db < 4; ++db) {
      toff[0][db] = kh * 8192 + tile_off(rowA, 4 * db + 2 * g1 + ((l & 3) >> 1)) + sub;
      toff[1][db] = kh * 8192 + tile_off(rowA + 8, 4 * db + 2 * g1 + ((l & 3) >> 1)) + sub;
    }
  }
  f32x16 dq[4];
#pragma unroll
  for (int db = 0; db < 4; ++db) dq[db] = f32x16{};

  int bcur = nc > 0 ? sload(a.col_idx + beg) : 0;
  int ccur = nc > 0 ? sload(a.blk_cnt + bcur) : 0;
  int bnext = nc > 1 ? sload(a.col_idx + beg + 1) : 0;
  if (nc > 0) issue(bcur, 0);
  dma_wait();
  __syncthreads();
  for (int j = 0; j < nc; ++j) {
    const int sb = j & 1;
    int cnext = 0, bnn = 0;
    if (j + 1 < nc) {
      issue(bnext, sb ^ 1);
      cnext = sload(a.blk_cnt + bnext);
      if (j + 2 < nc) bnn = sload(a.col_idx + beg + j + 2);
    }
    const char* kt = kv_s[sb][0];
    const char* vt = kv_s[sb][1];
    f32x16 s = {}, dp = {};
#pragma unroll
    for (int ks = 0; ks < NKS; ++ks) s = emfma(elds16(kt, koff[ks]), qreg[ks], s);
#pragma unroll
    for (int ks = 0; ks < NKS; ++ks) dp = emfma(elds16(vt, koff[ks]), dreg[ks], dp);
    float ds[16];
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const float kill = 32 * kh + 8 * (r / 4) + 4 * hi + (r % 4) < ccur ? 0.0f : INFINITY;
      const float p = exp2f_fast(fmaf(s[r], a.scale_log2, -(ls + kill)));
      ds[r] = p * (dp[r] - dl) * a.scale;
    }
    const ev8 sa = epack8(&ds[0]), sb8 = epack8(&ds[8]);
#pragma unroll
    for (int db = 0; db < NDB; ++db) {
      dq[db] = emfma(ecat_tr(lds_read_tr(kt, toff[0][db]), lds_read_tr(kt, toff[1][db])), sa, dq[db]);
      dq[db] = emfma(ecat_tr(lds_read_tr(kt + 4096, toff[0][db]), lds_read_tr(kt + 4096, toff[1][db])), sb8, dq[db]);
    }
    dma_wait();
    __syncthreads();
    bcur = bnext;
    ccur = cnext;
    bnext = bnn;
  }

  float* xq = reinterpret_cast<float*>(&kv_s[0][0][0]) + rg * (64 * 64);
  if (kh == 1) {
#pragma unroll
    for (int db = 0; db < NDB; ++db)
#pragma unroll
      for (int r = 0; r < 16; ++r) xq[(db * 16 + r) * 64 + l] = dq[db][r];
  }
  __syncthreads();
  if (kh == 1) return;
#pragma unroll
  for (int db = 0; db < NDB; ++db)
#pragma unroll
    for (int r = 0; r < 16; ++r) dq[db][r] += xq[(db * 16 + r) * 64 + l];
#pragma unroll
  for (int db = NDB; db < 4; ++db) dq[db] = f32x16{};  // columns past D: zero
  if (TASKS && slot >= 0) {
    float* pq = a.part_a + ((size_t)slot * BK + qrow) * ld;
#pragma unroll
    for (int db = 0; db < 4; ++db)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        if (DH < HD && 32 * db >= ld) break;
        *reinterpret_cast<float4*>(pq + 32 * db + 8 * i + 4 * hi) =
            make_float4(dq[db][4 * i], dq[db][4 * i + 1], dq[db][4 * i + 2], dq[db][4 * i + 3]);
      }
    return;
  }
  const float inv = qvalid ? 1.0f / (float)qcnt : 0.0f;
  const float keep = qvalid ? 1.0f : 0.0f;
  const float* adq = a.add_a + ((size_t)bh * a.add_nb + qb) * ld;
#pragma unroll
  for (int db = 0; db < 4; ++db)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      if (DH < HD && 32 * db >= ld) break;
      const int c = 32 * db + 8 * i + 4 * hi;
      f32x4 x;
#pragma unroll
      for (int e = 0; e < 4; ++e) x[e] = dq[db][4 * i + e] * keep;
      if (a.out_a32 != nullptr) {  // dq_acc += dQ (padding rows keep their value)
        f32x4* dst = reinterpret_cast<f32x4*>(a.out_a32 + tok * ld + c);
        *dst = *dst + x;
      } else {
        if (a.add_a != nullptr) x += *reinterpret_cast<const f32x4*>(adq + c) * inv;
        ushort4 q4;
        q4.x = f2e(x[0]); q4.y = f2e(x[1]); q4.z = f2e(x[2]); q4.w = f2e(x[3]);
        *reinterpret_cast<ushort4*>(a.out_a + tok * ld + c) = q4;
      }
    }
}

}  // namespace

}  // namespace es

using namespace es;

static int vsa_check_qkv(const void* q, const void* k, const void* v, int BH, int L, int D) {
  ES_REQUIRE(q && k && v, ES_ERR_INVALID, "VSA: null q / k / v");
  ES_REQUIRE(BH > 0 && L > 0 && L % BK == 0, ES_ERR_INVALID, "VSA: tokens must be [BH, L = NB * 64, D]");
  HeadDim h;
  VSA_REQUIRE_DIM(D, h);
  ES_REQUIRE((size_t)L * HD * 2 < (1ull << 31), ES_ERR_UNSUPPORTED, "VSA: one head's tokens exceed 2 GiB");
  return ES_OK;
}

static VsaFwdArgs fwd_args(const void* q, const void* k, const void* v, const int* blk_cnt, int BH, int L, int D) {
  VsaFwdArgs a = {};
  a.q = (const e16_t*)q;
  a.k = (const e16_t*)k;
  a.v = (const e16_t*)v;
  a.blk_cnt = blk_cnt;
  a.L = L;
  a.NB = L / BK;
  a.BH = BH;
  HeadDim h;
  head_dim(D, h);
  a.ld = h.ld;
  a.scale = LOG2E / sqrtf((float)h.d);
  return a;
}

extern "C" int ES_VSA_API(vsa_attn_fwd)(const void* q, const void* k, const void* v, const int* row_ptr, const int* col_idx,
                            const int* blk_cnt, void* out, float* lse, int BH, int L, int D, hipStream_t stream) {
  if (int st = vsa_check_qkv(q, k, v, BH, L, D)) return st;
  ES_REQUIRE(row_ptr && blk_cnt && out && lse, ES_ERR_INVALID, "VSA: null tensor pointer");
  VsaFwdArgs a = fwd_args(q, k, v, blk_cnt, BH, L, D);
  a.row_ptr = row_ptr;
  a.col_idx = col_idx;
  a.out = (e16_t*)out;
  a.lse = lse;
  a.per_xcd = (a.NB + 7) / 8;
  ES_REQUIRE(8LL * BH * a.per_xcd < (1LL << 30), ES_ERR_UNSUPPORTED, "VSA: grid too large");
  Queues qs;
  ES_REQUIRE(balanced_launch(BH, a.per_xcd, stream, qs), ES_ERR_LAUNCH, "VSA: row-block queues unavailable");
  a.queues = qs.counters;
  a.fixed = qs.fixed;
  if ((D & 0xffff) == 64) hipLaunchKernelGGL((vsa_fwd_kernel<false, 64>), dim3((unsigned)qs.grid), dim3(256), 0, stream, a);
  else hipLaunchKernelGGL((vsa_fwd_kernel<false, 128>), dim3((unsigned)qs.grid), dim3(256), 0, stream, a);
  return check_launch("vsa_attn_fwd");
}

extern "C" int ES_VSA_API(vsa_attn_fwd_tasks)(const void* q, const void* k, const void* v, const int* col_idx,
                                  const int* blk_cnt, const int* tasks, const int* info, int max_tasks, void* out,
                                  float* lse, float* part_o, float* part_lse, int BH, int L, int D,
                                  hipStream_t stream) {
  if (int st = vsa_check_qkv(q, k, v, BH, L, D)) return st;
  // part_o / part_lse may be null when the plan has no split slots (no task then writes a partial)
  ES_REQUIRE(blk_cnt && tasks && info && out && lse, ES_ERR_INVALID, "VSA: null tensor pointer");
  ES_REQUIRE(max_tasks >= 0, ES_ERR_INVALID, "VSA: negative task capacity");
  if (max_tasks == 0) return ES_OK;
  VsaFwdArgs a = fwd_args(q, k, v, blk_cnt, BH, L, D);
  a.col_idx = col_idx;
  a.tasks = (const int4*)tasks;
  a.info = info;
  a.out = (e16_t*)out;
  a.lse = lse;
  a.part_o = part_o;
  a.part_lse = part_lse;
  if ((D & 0xffff) == 64) hipLaunchKernelGGL((vsa_fwd_kernel<true, 64>), dim3((unsigned)max_tasks), dim3(256), 0, stream, a);
  else hipLaunchKernelGGL((vsa_fwd_kernel<true, 128>), dim3((unsigned)max_tasks), dim3(256), 0, stream, a);
  return check_launch("vsa_attn_fwd_tasks");
}


static VsaBwdArgs bwd_args(const void* q, const void* k, const void* v, const void* dout, const float* lse,
                           const float* delta, const int* blk_cnt, int BH, int L, int D) {
  VsaBwdArgs a = {};
  a.q = (const e16_t*)q;
  a.k = (const e16_t*)k;
  a.v = (const e16_t*)v;
  a.dout = (const e16_t*)dout;
  a.lse = lse;
  a.delta = delta;
  a.blk_cnt = blk_cnt;
  a.L = L;
  a.NB = L / BK;
  a.BH = BH;
  a.per_xcd = (a.NB + 7) / 8;
  HeadDim h;
  head_dim(D, h);
  a.ld = h.ld;
  a.scale = 1.0f / sqrtf((float)h.d);
  a.scale_log2 = LOG2E / sqrtf((float)h.d);
  return a;
}

extern "C" int ES_VSA_API(vsa_attn_bwd_kv)(const void* q, const void* k, const void* v, const void* dout, const float* lse,
                               const float* delta, const int* k2q_ptr, const int* k2q_idx, const int* blk_cnt,
                               const float* add_dk, const float* add_dv, int add_nb, void* dk, void* dv,
                               int out_fp32, int BH, int L, int D, hipStream_t stream) {
  if (int st = vsa_check_qkv(q, k, v, BH, L, D)) return st;
  ES_REQUIRE(dout && lse && delta && k2q_ptr && blk_cnt && dk && dv, ES_ERR_INVALID, "VSA: null tensor pointer");
  ES_REQUIRE((add_dk == nullptr && add_dv == nullptr) || add_nb >= L / BK, ES_ERR_INVALID,
             "VSA: per-block gradient has fewer rows than blocks");
  VsaBwdArgs a = bwd_args(q, k, v, dout, lse, delta, blk_cnt, BH, L, D);
  a.row_ptr = k2q_ptr;
  a.col_idx = k2q_idx;
  a.add_a = add_dk;
  a.add_b = add_dv;
  a.add_nb = add_nb;
  if (out_fp32) {
    a.out_a32 = (float*)dk;
    a.out_b32 = (float*)dv;
  } else {
    a.out_a = (e16_t*)dk;
    a.out_b = (e16_t*)dv;
  }
  ES_REQUIRE(8LL * BH * a.per_xcd < (1LL << 30), ES_ERR_UNSUPPORTED, "VSA: grid too large");
  Queues qs;
  ES_REQUIRE(balanced_launch(BH, a.per_xcd, stream, qs), ES_ERR_LAUNCH, "VSA: row-block queues unavailable");
  a.queues = qs.counters;
  a.fixed = qs.fixed;
  if ((D & 0xffff) == 64) hipLaunchKernelGGL((vsa_bwd_kv_kernel<false, 64>), dim3((unsigned)qs.grid), dim3(256), 0, stream, a);
  else hipLaunchKernelGGL((vsa_bwd_kv_kernel<false, 128>), dim3((unsigned)qs.grid), dim3(256), 0, stream, a);
  return check_launch("vsa_attn_bwd_kv");
}

extern "C" int ES_VSA_API(vsa_attn_bwd_kv_tasks)(const void* q, const void* k, const void* v, const void* dout, const float* lse,
                                     const float* delta, const int* k2q_idx, const int* blk_cnt, const int* tasks,
                                     const int* info, int max_tasks, const float* add_dk, const float* add_dv,
                                     int add_nb, void* dk, void* dv, float* part_dk, float* part_dv, int BH, int L,
                                     int D, hipStream_t stream) {
  if (int st = vsa_check_qkv(q, k, v, BH, L, D)) return st;
  ES_REQUIRE(dout && lse && delta && blk_cnt && tasks && info && dk && dv, ES_ERR_INVALID, "VSA: null tensor pointer");
  ES_REQUIRE(max_tasks >= 0, ES_ERR_INVALID, "VSA: negative task capacity");
  if (max_tasks == 0) return ES_OK;
  VsaBwdArgs a = bwd_args(q, k, v, dout, lse, delta, blk_cnt, BH, L, D);
  a.col_idx = k2q_idx;
  a.tasks = (const int4*)tasks;
  a.info = info;
  a.add_a = add_dk;
  a.add_b = add_dv;
  a.add_nb = add_nb;
  a.out_a = (e16_t*)dk;
  a.out_b = (e16_t*)dv;
  a.part_a = part_dk;
  a.part_b = part_dv;
  if ((D & 0xffff) == 64) hipLaunchKernelGGL((vsa_bwd_kv_kernel<true, 64>), dim3((unsigned)max_tasks), dim3(256), 0, stream, a);
  else hipLaunchKernelGGL((vsa_bwd_kv_kernel<true, 128>), dim3((unsigned)max_tasks), dim3(256), 0, stream, a);
  return check_launch("vsa_attn_bwd_kv_tasks");
}

extern "C" int ES_VSA_API(vsa_attn_bwd_q)(const void* q, const void* k, const void* v, const void* dout, const float* lse,
                              const float* delta, const int* q2k_ptr, const int* q2k_idx, const int* blk_cnt,
                              const float* add_dq, int add_nb, void* dq, float* dq_acc, int BH, int L, int D,
                              hipStream_t stream) {
  if (int st = vsa_check_qkv(q, k, v, BH, L, D)) return st;
  ES_REQUIRE(dout && lse && delta && q2k_ptr && blk_cnt && (dq || dq_acc), ES_ERR_INVALID, "VSA: null tensor pointer");
  ES_REQUIRE(add_dq == nullptr || add_nb >= L / BK, ES_ERR_INVALID, "VSA: per-block gradient has fewer rows than blocks");
  VsaBwdArgs a = bwd_args(q, k, v, dout, lse, delta, blk_cnt, BH, L, D);
  a.row_ptr = q2k_ptr;
  a.col_idx = q2k_idx;
  a.add_a = add_dq;
  a.add_nb = add_nb;
  a.out_a = (e16_t*)dq;
  a.out_a32 = dq_acc;
  ES_REQUIRE(8LL * BH * a.per_xcd < (1LL << 30), ES_ERR_UNSUPPORTED, "VSA: grid too large");
  Queues qs;
  ES_REQUIRE(balanced_launch(BH, a.per_xcd, stream, qs), ES_ERR_LAUNCH, "VSA: row-block queues unavailable");
  a.queues = qs.counters;
  a.fixed = qs.fixed;
  if ((D & 0xffff) == 64) hipLaunchKernelGGL((vsa_bwd_q_kernel<false, 64>), dim3((unsigned)qs.grid), dim3(256), 0, stream, a);
  else hipLaunchKernelGGL((vsa_bwd_q_kernel<false, 128>), dim3((unsigned)qs.grid), dim3(256), 0, stream, a);
  return check_launch("vsa_attn_bwd_q");
}

extern "C" int ES_VSA_API(vsa_attn_bwd_q_tasks)(const void* q, const void* k, const void* v, const void* dout, const float* lse,
                                    const float* delta, const int* q2k_idx, const int* blk_cnt, const int* tasks,
                                    const int* info, int max_tasks, const float* add_dq, int add_nb, void* dq,
                                    float* part_dq, int BH, int L, int D, hipStream_t stream) {
  if (int st = vsa_check_qkv(q, k, v, BH, L, D)) return st;
  ES_REQUIRE(dout && lse && delta && blk_cnt && tasks && info && dq, ES_ERR_INVALID, "VSA: null tensor pointer");
  ES_REQUIRE(max_tasks >= 0, ES_ERR_INVALID, "VSA: negative task capacity");
  if (max_tasks == 0) return ES_OK;
  VsaBwdArgs a = bwd_args(q, k, v, dout, lse, delta, blk_cnt, BH, L, D);
  a.col_idx = q2k_idx;
  a.tasks = (const int4*)tasks;
  a.info = info;
  a.add_a = add_dq;
  a.add_nb = add_nb;
  a.out_a = (e16_t*)dq;
  a.part_a = part_dq;
  if ((D & 0xffff) == 64) hipLaunchKernelGGL((vsa_bwd_q_kernel<true, 64>), dim3((unsigned)max_tasks), dim3(256), 0, stream, a);
  else hipLaunchKernelGGL((vsa_bwd_q_kernel<true, 128>), dim3((unsigned)max_tasks), dim3(256), 0, stream, a);
  return check_launch("vsa_attn_bwd_q_tasks");
}
