// VSA2 split-KV scheduling: the device-side task plan over a CSR list and the two merges (gfx950).
//
// Plan (reference csrc/vsa/split.cu:1-19, vsa2_kernels.h:48-74; contract of the pure-Python planner in
// tests/test_vsa2_split.py:60-87). For the NR = BH * NB rows of a CSR list (q2k for the forward and the Q-owner
// backward, k2q for the KV-owner backward):
//   thr    = max(chunk + 1, min_len, ceil(tail_frac * W / resident)) and, with rel_mean > 0, per (b, h)
//            max(thr, ceil(rel_mean * nnz_bh / NB)); W = all edges of the list
//   cnt_r  = n_r >= thr ? ceil(n_r / chunk) : 0; E = #rows with n_r >= thr
//   split  = E <= budget && cnt_r > 0 && (inclusive scan of cnt up to r) <= max_slots
//   tasks  : split rows first, chunk j of row r = [beg + j n / c, beg + (j + 1) n / c) with slot = (exclusive scan
//            of cnt) + j; then one direct task (slot -1) per other row, in row order
//   merges : one {r, first slot, c, 0} per split row; info = {tasks, split rows, split slots, NR, E, E <= budget,
//            thr without the per-(b, h) term, W}
// One workgroup of 1024 threads plans the whole list: each thread owns a contiguous run of rows, and two workgroup
// scans give every thread its slot, task and merge bases. Nothing is read back to the host. What bounds it is one
// CU's instructions and the latency of a thread's list pointers: a row costs no division (its head and the head's
// threshold move along) and PLAN_ROWS rows' pointers are loaded together (with a division, a double-precision
// threshold and a wait per row: 67 us for 9 456 rows, 53 now, most of it the task stores of one CU).
//
// Merges (one workgroup per split row, in chunk order: deterministic):
//   forward : o = sum_i 2^(lse_i - M) o_i / sum_i 2^(lse_i - M), lse = (M + log2 sum) ln 2 (reference
//             split.cu:117-155); padded query rows get o = 0, lse = -inf when mask_rows
//   sum     : out = valid ? sum_i part_i + add[blk] / cnt : 0 (reference split.cu:157-200)
#include "../../include/vsa_hip.h"
#include "common.h"
#include "elem.h"

#include <cmath>

namespace es {

namespace {

constexpr int PLAN_THREADS = 1024;
constexpr int PLAN_ROWS = 8;  // rows of a thread whose list pointers are loaded together

struct PlanArgs {
  const int* ptr;
  int BH, NB, chunk, max_slots, min_len, resident, budget;
  double rel_mean, tail_frac;
  int4* tasks;
  int4* merges;
  int* info;
};

// exclusive scan of x over the 1024 threads (16 waves); returns the prefix, total in *tot
__device__ long long plan_scan(long long x, long long* red, long long* tot) {
  const int l = threadIdx.x & 63, wv = threadIdx.x >> 6;
  long long inc = x;
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) {
    const long long y = __shfl_up(inc, d, 64);
    if (l >= d) inc += y;
  }
  __syncthreads();
  if (l == 63) red[wv] = inc;
  __syncthreads();
  long long before = 0, all = 0;
  for (int i = 0; i < PLAN_THREADS / 64; ++i) {
    before += i < wv ? red[i] : 0;
    all += red[i];
  }
  *tot = all;
  return before + inc - x;
}

__global__ __launch_bounds__(PLAN_THREADS) void plan_kernel(PlanArgs a) {
  __shared__ long long red[PLAN_THREADS / 64];
  const int NR = a.BH * a.NB;
  const int per = (NR + PLAN_THREADS - 1) / PLAN_THREADS;
  const int r0 = min(NR, (int)threadIdx.x * per), r1 = min(NR, r0 + per);
  const long long W = (long long)a.ptr[(size_t)a.BH * (a.NB + 1) - 1] - a.ptr[0];
  int gthr = max(a.chunk + 1, a.min_len);
  if (a.tail_frac > 0.0) gthr = max(gthr, (int)ceil(a.tail_frac * (double)W / (double)a.resident));
  auto head_thr = [&](int bh) {
    if (!(a.rel_mean > 0.0) || bh >= a.BH) return gthr;
    const int* hp = a.ptr + (size_t)bh * (a.NB + 1);
    return max(gthr, (int)ceil(a.rel_mean * (double)(hp[a.NB] - hp[0]) / (double)a.NB));
  };
  const int bh0 = r0 / a.NB, i0 = r0 - bh0 * a.NB, thr0 = head_thr(bh0);
  // f(row, list begin, list length, chunks) for this thread's rows in order; row r of head bh starts at ptr[r + bh]
  auto each_row = [&](auto&& f) {
    int bl = bh0, il = i0, bh = bh0, i = i0, thr = thr0;
    for (int rb = r0; rb < r1; rb += PLAN_ROWS) {
      int beg[PLAN_ROWS], end[PLAN_ROWS];
#pragma unroll
      for (int k = 0; k < PLAN_ROWS; ++k) {
        const size_t at = rb + k < r1 ? (size_t)(rb + k) + bl : 0;
        beg[k] = a.ptr[at];
        end[k] = a.ptr[at + 1];
        if (++il == a.NB) {
          il = 0;
          ++bl;
        }
      }
#pragma unroll
      for (int k = 0; k < PLAN_ROWS; ++k) asm volatile("" : "+v"(beg[k]), "+v"(end[k]));  // (loads not sunk to uses)
#pragma unroll
      for (int k = 0; k < PLAN_ROWS; ++k) {
        if (rb + k >= r1) break;
        const int n = end[k] - beg[k];
        f(rb + k, beg[k], n, n >= thr ? (n + a.chunk - 1) / a.chunk : 0);
        if (++i == a.NB) {
          i = 0;
          thr = head_thr(++bh);
        }
      }
    }
  };
  // Two counts share a 64-bit scan (each is below 2^32: at most the edges plus the rows of an int32 CSR)
  auto pair = [](unsigned lo, unsigned up) { return (long long)(((unsigned long long)up << 32) | lo); };
  auto lo32 = [](long long x) { return (long long)(unsigned)x; };
  auto up32 = [](long long x) { return (long long)(unsigned)((unsigned long long)x >> 32); };
  // 1: chunk counts and eligible rows
  unsigned cnt_mine = 0, elig_mine = 0;
  each_row([&](int, int, int, int c) {
    cnt_mine += (unsigned)c;
    elig_mine += c > 0;
  });
  long long tot;
  const long long cnt_before = lo32(plan_scan(pair(cnt_mine, elig_mine), red, &tot));
  const long long E = up32(tot);
  const bool ok = E <= (long long)a.budget;
  // 2: split rows and their chunks before this thread (every other row is direct)
  unsigned split_mine = 0, chunks_mine = 0;
  long long incl = cnt_before;
  each_row([&](int, int, int, int c) {
    incl += c;
    const bool split = ok && c > 0 && incl <= a.max_slots;
    split_mine += split;
    chunks_mine += split ? (unsigned)c : 0u;
  });
  const long long split_before = lo32(plan_scan(pair(split_mine, chunks_mine), red, &tot));
  const long long nsplit = lo32(tot), t_split = up32(tot), ndirect = NR - nsplit, direct_before = r0 - split_before;
  // 3: write
  long long ms = split_before, dt = direct_before;
  incl = cnt_before;
  each_row([&](int r, int beg, int n, int c) {
    const long long slot0 = incl;
    incl += c;
    if (ok && c > 0 && incl <= a.max_slots) {
      // j n / c, in 32 bits where j n fits them
      auto cut = [&](int j) {
        return n < 65536 ? (int)((unsigned)j * (unsigned)n / (unsigned)c) : (int)((long long)j * n / c);
      };
      for (int j = 0; j < c; ++j)
        a.tasks[slot0 + j] = make_int4(r, beg + cut(j), beg + cut(j + 1), (int)(slot0 + j));
      a.merges[ms++] = make_int4(r, (int)slot0, c, 0);
    } else {
      a.tasks[t_split + dt++] = make_int4(r, beg, beg + n, -1);
    }
  });
  if (threadIdx.x == 0) {
    a.info[0] = (int)(t_split + ndirect);
    a.info[1] = (int)nsplit;
    a.info[2] = (int)t_split;
    a.info[3] = NR;
    a.info[4] = (int)E;
    a.info[5] = ok ? 1 : 0;
    a.info[6] = gthr;
    a.info[7] = (int)W;
  }
}

// Merges: grid (max_merges, 4), 16 rows of a split row block per workgroup, thread -> (row, 8 columns). The partials of
// a row are summed in chunk order, MERGE_AHEAD of them loaded together (a thread of 32 columns with one partial in
// flight waited for each in turn: 128 rows of 19 partials, forward 45 us, sum 34; 27, 3.4 TB/s, and 24 now).
constexpr int MERGE_AHEAD = 8;

__device__ __forceinline__ uint4 pack8e(const f32x4& x0, const f32x4& x1) {
  uint4 u;
  u.x = (unsigned)f2e(x0[0]) | ((unsigned)f2e(x0[1]) << 16);
  u.y = (unsigned)f2e(x0[2]) | ((unsigned)f2e(x0[3]) << 16);
  u.z = (unsigned)f2e(x1[0]) | ((unsigned)f2e(x1[1]) << 16);
  u.w = (unsigned)f2e(x1[2]) | ((unsigned)f2e(x1[3]) << 16);
  return u;
}

__global__ __launch_bounds__(256) void merge_fwd_kernel(const float* __restrict__ part_o,
                                                        const float* __restrict__ part_lse,
                                                        const int4* __restrict__ merges, const int* __restrict__ info,
                                                        const int* __restrict__ blk_cnt, e16_t* __restrict__ o,
                                                        float* __restrict__ lse, int L, int NB, int ld, int mask_rows) {
  if ((int)blockIdx.x >= info[1]) return;
  const int4 mg = merges[blockIdx.x];
  const int bh = mg.x / NB, qb = mg.x - bh * NB, slot0 = mg.y, c = mg.z;
  const int row = blockIdx.y * 16 + (threadIdx.x >> 4), c0 = (threadIdx.x & 15) * 8;
  if (c0 >= ld) return;  // (rows of ld columns)
  const size_t tok = (size_t)bh * L + (size_t)qb * BK + row;
  f32x4 acc[2] = {f32x4{}, f32x4{}};
  float out_lse = -INFINITY;
  if (row < blk_cnt[qb] || !mask_rows) {
    const float* pl = part_lse + (size_t)slot0 * BK + row;
    float mx = -INFINITY;
#pragma unroll 8
    for (int j = 0; j < c; ++j) mx = fmaxf(mx, pl[(size_t)j * BK]);
    if (mx != -INFINITY) {
      float sum = 0.0f;
      for (int j0 = 0; j0 < c; j0 += MERGE_AHEAD) {
        f32x4 x[MERGE_AHEAD][2];
        float w[MERGE_AHEAD];
#pragma unroll
        for (int k = 0; k < MERGE_AHEAD; ++k) {
          const int j = min(j0 + k, c - 1);
          const f32x4* src = reinterpret_cast<const f32x4*>(part_o + ((size_t)(slot0 + j) * BK + row) * ld + c0);
          x[k][0] = src[0];
          x[k][1] = src[1];
          w[k] = pl[(size_t)j * BK];
        }
#pragma unroll
        for (int k = 0; k < MERGE_AHEAD; ++k) asm volatile("" : "+v"(x[k][0]), "+v"(x[k][1]), "+v"(w[k]));  // (not sunk)
#pragma unroll
        for (int k = 0; k < MERGE_AHEAD; ++k) {
          if (j0 + k >= c) break;
          const float wk = exp2f(w[k] - mx);
          sum += wk;
          acc[0] += wk * x[k][0];
          acc[1] += wk * x[k][1];
        }
      }
      const float inv = 1.0f / sum;
      acc[0] *= inv;
      acc[1] *= inv;
      out_lse = (mx + log2f(sum)) * 0.6931471805599453f;
    }
  }
  *reinterpret_cast<uint4*>(o + tok * ld + c0) = pack8e(acc[0], acc[1]);
  if (c0 == 0) lse[tok] = out_lse;
}

__global__ __launch_bounds__(256) void merge_sum_kernel(const float* __restrict__ part, const int4* __restrict__ merges,
                                                        const int* __restrict__ info, const float* __restrict__ add,
                                                        int add_nb, const int* __restrict__ blk_cnt,
                                                        e16_t* __restrict__ out, float* __restrict__ out_f32, int L,
                                                        int NB, int ld) {
  if ((int)blockIdx.x >= info[1]) return;
  const int4 mg = merges[blockIdx.x];
  const int bh = mg.x / NB, blk = mg.x - bh * NB, slot0 = mg.y, c = mg.z;
  const int row = blockIdx.y * 16 + (threadIdx.x >> 4), c0 = (threadIdx.x & 15) * 8;
  if (c0 >= ld) return;  // (rows of ld columns)
  const size_t tok = (size_t)bh * L + (size_t)blk * BK + row;
  const int cnt = blk_cnt[blk];
  f32x4 acc[2] = {f32x4{}, f32x4{}};
  if (row < cnt) {
    for (int j0 = 0; j0 < c; j0 += MERGE_AHEAD) {
      f32x4 x[MERGE_AHEAD][2];
#pragma unroll
      for (int k = 0; k < MERGE_AHEAD; ++k) {
        const int j = min(j0 + k, c - 1);
        const f32x4* src = reinterpret_cast<const f32x4*>(part + ((size_t)(slot0 + j) * BK + row) * ld + c0);
        x[k][0] = src[0];
        x[k][1] = src[1];
      }
#pragma unroll
      for (int k = 0; k < MERGE_AHEAD; ++k) asm volatile("" : "+v"(x[k][0]), "+v"(x[k][1]));  // (not sunk to their uses)
#pragma unroll
      for (int k = 0; k < MERGE_AHEAD; ++k) {
        if (j0 + k >= c) break;
        acc[0] += x[k][0];
        acc[1] += x[k][1];
      }
    }
    if (add != nullptr) {
      const float inv = 1.0f / (float)cnt;
      const f32x4* ad = reinterpret_cast<const f32x4*>(add + ((size_t)bh * add_nb + blk) * ld + c0);
      acc[0] += ad[0] * inv;
      acc[1] += ad[1] * inv;
    }
  }
  if (out_f32 != nullptr) {
    f32x4* dst = reinterpret_cast<f32x4*>(out_f32 + tok * ld + c0);
    dst[0] = acc[0];
    dst[1] = acc[1];
  } else {
    *reinterpret_cast<uint4*>(out + tok * ld + c0) = pack8e(acc[0], acc[1]);
  }
}

}  // namespace

}  // namespace es

using namespace es;

#ifndef ES_ELEM_F16  // no token tensors: built once
extern "C" int vsa_split_plan(const int* ptr, int BH, int NB, int chunk, int max_slots, int min_len, double rel_mean,
                              double tail_frac, int resident, int budget, int* tasks, int* merges, int* info,
                              hipStream_t stream) {
  ES_REQUIRE(ptr && tasks && merges && info, ES_ERR_INVALID, "VSA2: null tensor pointer");
  ES_REQUIRE(BH >= 1 && NB >= 1, ES_ERR_INVALID, "ptr must be [B, H, NB+1]");
  ES_REQUIRE(chunk >= 1 && chunk <= (1 << 30), ES_ERR_INVALID, "split chunk must be in [1, 2^30]");
  ES_REQUIRE(max_slots >= 0 && max_slots < (1 << 30), ES_ERR_INVALID, "bad max_slots");
  ES_REQUIRE(rel_mean >= 0.0 && tail_frac >= 0.0 && resident >= 1, ES_ERR_INVALID, "bad split policy");
  PlanArgs a = {};
  a.ptr = ptr;
  a.BH = BH;
  a.NB = NB;
  a.chunk = chunk;
  a.max_slots = max_slots;
  a.min_len = min_len;
  a.resident = resident;
  a.budget = budget < 0 ? 0x7fffffff : budget;
  a.rel_mean = rel_mean;
  a.tail_frac = tail_frac;
  a.tasks = (int4*)tasks;
  a.merges = (int4*)merges;
  a.info = info;
  hipLaunchKernelGGL(plan_kernel, dim3(1), dim3(PLAN_THREADS), 0, stream, a);
  return check_launch("vsa_split_plan");
}
#endif

extern "C" int ES_VSA_API(vsa_split_merge_fwd)(const float* part_o, const float* part_lse, const int* merges, const int* info,
                                   int max_merges, const int* blk_cnt, void* o, float* lse, int BH, int L, int D,
                                   int mask_rows, hipStream_t stream) {
  HeadDim h;
  VSA_REQUIRE_DIM(D, h);
  ES_REQUIRE(BH >= 1 && L > 0 && L % BK == 0, ES_ERR_INVALID, "o must be [B,H,L,D]");
  if (max_merges <= 0) return ES_OK;
  ES_REQUIRE(part_o && part_lse && merges && info && blk_cnt && o && lse, ES_ERR_INVALID, "VSA2: null tensor pointer");
  hipLaunchKernelGGL(merge_fwd_kernel, dim3(max_merges, 4), dim3(256), 0, stream, part_o, part_lse, (const int4*)merges,
                     info, blk_cnt, (e16_t*)o, lse, L, L / BK, h.ld, mask_rows);
  return check_launch("vsa_split_merge_fwd");
}

extern "C" int ES_VSA_API(vsa_split_merge_sum)(const float* part, const int* merges, const int* info, int max_merges,
                                   const float* add, int add_nb, const int* blk_cnt, void* out, float* out_f32, int BH,
                                   int L, int D, hipStream_t stream) {
  HeadDim h;
  VSA_REQUIRE_DIM(D, h);
  ES_REQUIRE(BH >= 1 && L > 0 && L % BK == 0, ES_ERR_INVALID, "out must be [B,H,L,D]");
  if (max_merges <= 0) return ES_OK;
  ES_REQUIRE(part && merges && info && blk_cnt && (out || out_f32), ES_ERR_INVALID, "VSA2: null tensor pointer");
  hipLaunchKernelGGL(merge_sum_kernel, dim3(max_merges, 4), dim3(256), 0, stream, part, (const int4*)merges, info, add,
                     add_nb, blk_cnt, (e16_t*)out, out_f32, L, L / BK, h.ld);
  return check_launch("vsa_split_merge_sum");
}
