// VSA / VSA2 elementwise passes: pooling, gate fusion (forward / backward) and the coarse-unpool finalize.
//
// Token tensors are [BH, L, D] bf16 with L = NB * 64 in block-major order; blk_cnt [NB] holds the valid tokens of
// each 64-token block (valid-first: rows >= blk_cnt of a block are padding). D = 128. Pooled tensors are
// [BH, rows_pad, D] with rows_pad a multiple of 64; their padding rows are written as zeros.
//
// Every kernel here moves each token row once and is HBM-bound. A 16-lane DPP row of a wave covers one 256-byte
// token row with 16-byte accesses, so row reductions stay inside one DPP row.
//
//   pool_kernel      reference csrc/vsa/router/pool.cu:16-51 (router group means of R tokens, whole-block means)
//   fuse_fwd_kernel  reference csrc/vsa/fuse.cu:3 (O = O_f + act(gate) * O_c[blk] on valid rows, 0 elsewhere)
//   fuse_bwd_kernel  reference csrc/vsa/fuse.cu:4-8 (dO_f, delta_f, dO_c, delta_c, dgate)
//   finalize_kernel  reference csrc/vsa/fuse.cu:9 (dX = acc + add[blk] / cnt on valid rows, 0 elsewhere)
#include "../../include/vsa_hip.h"
#include "common.h"
#include "elem.h"

namespace es {

namespace {

__device__ __forceinline__ void unpack8(const uint4& u, float* x) {
  const unsigned w[4] = {u.x, u.y, u.z, u.w};
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    x[2 * i] = e2f((e16_t)(w[i] & 0xffffu));
    x[2 * i + 1] = e2f((e16_t)(w[i] >> 16));
  }
}

__device__ __forceinline__ void ld8(const e16_t* p, float* x) { unpack8(*reinterpret_cast<const uint4*>(p), x); }

__device__ __forceinline__ void st8(e16_t* p, const float* x) {
  uint4 u;
  u.x = (unsigned)f2e(x[0]) | ((unsigned)f2e(x[1]) << 16);
  u.y = (unsigned)f2e(x[2]) | ((unsigned)f2e(x[3]) << 16);
  u.z = (unsigned)f2e(x[4]) | ((unsigned)f2e(x[5]) << 16);
  u.w = (unsigned)f2e(x[6]) | ((unsigned)f2e(x[7]) << 16);
  *reinterpret_cast<uint4*>(p) = u;
}

// gate activations: 0 = tanh, 1 = identity; the derivative is written in terms of a = act(g)
__device__ __forceinline__ float gact(float g, int act) { return act == 0 ? tanhf(g) : g; }
__device__ __forceinline__ float gdact(float a, int act) { return act == 0 ? 1.f - a * a : 1.f; }


struct PoolArgs {
  const e16_t* src[3];  // q, k, v
  e16_t* grp[3];        // qr, kr, vr (any may be null)
  e16_t* blk[3];        // qc, kc, vc
  const int* blk_cnt;
  int NB, L, R, Lr_pad, NBc_pad;
  int ld;  // columns of a stored row
};

constexpr int POOL_BLOCKS = 4;  // 64-token blocks per workgroup

// grid (cdiv(ceil64(NB), 4), BH), 192 threads: 48 per block = 3 tensors x 16 chunks of 8 columns. Each column sums its
// group's rows in order, then the group sums in order, so the float result is that of a sequential loop. The rows are
// read sixteen at a time, all in flight before the first is added (one row after the other, the sums waited for each
// load in turn: 24 us for three 4096-token, 2-head tensors against 8 now, 36 against 24 for 240 blocks and 12 heads). The
// pooled tensors' padding rows are written as zeros here, so callers need not clear them first.
template <int R>
__global__ __launch_bounds__(192) void pool_kernel(PoolArgs a) {
  constexpr int G = BK / R, BATCH = 16;
  const int sub = threadIdx.x / 48, t = threadIdx.x % 48;
  const int blk = blockIdx.x * POOL_BLOCKS + sub;
  const int which = t / 16, c8 = (t % 16) * 8;
  const int ld = a.ld;
  if (a.src[which] == nullptr || c8 >= ld) return;  // a null source: that tensor is not pooled
  const size_t bh = blockIdx.y;
  e16_t* grp = a.grp[which];
  if (blk >= a.NB) {
    const uint4 z = {0u, 0u, 0u, 0u};
    if (blk < a.NBc_pad) *reinterpret_cast<uint4*>(a.blk[which] + (bh * a.NBc_pad + blk) * ld + c8) = z;
    if (grp != nullptr)
      for (int r = blk * G; r < min((blk + 1) * G, a.Lr_pad); ++r)
        *reinterpret_cast<uint4*>(grp + (bh * a.Lr_pad + r) * ld + c8) = z;
    return;
  }
  const int n = a.blk_cnt[blk];
  const e16_t* src = a.src[which] + (bh * a.L + (size_t)blk * BK) * ld + c8;
  float tot[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
  float s[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
#pragma unroll 1
  for (int r0 = 0; r0 < BK; r0 += BATCH) {
    uint4 u[BATCH];
#pragma unroll
    for (int i = 0; i < BATCH; ++i)
      u[i] = r0 + i < n ? *reinterpret_cast<const uint4*>(src + (size_t)(r0 + i) * ld) : uint4{0u, 0u, 0u, 0u};
#pragma unroll
    for (int i = 0; i < BATCH; ++i) {
      float x[8];
      unpack8(u[i], x);
#pragma unroll
      for (int e = 0; e < 8; ++e) s[e] += x[e];  // (a row past n adds +0 to a sum that is never -0)
      if ((r0 + i + 1) % R == 0) {
        const int g = (r0 + i) / R;
        if (grp != nullptr) {
          const int in = min(max(n - g * R, 0), R);
          const float inv = in > 0 ? 1.f / (float)in : 0.f;
          float m[8];
#pragma unroll
          for (int e = 0; e < 8; ++e) m[e] = mul_rn(s[e], inv);
          st8(grp + (bh * a.Lr_pad + (size_t)blk * G + g) * ld + c8, m);
        }
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          tot[e] += s[e];
          s[e] = 0.f;
        }
      }
    }
  }
  const float inv = 1.f / (float)n;
#pragma unroll
  for (int e = 0; e < 8; ++e) tot[e] = mul_rn(tot[e], inv);
  st8(a.blk[which] + (bh * a.NBc_pad + blk) * ld + c8, tot);
}

static void launch_pool(const PoolArgs& a, int BH, hipStream_t stream) {
  const dim3 grid((a.NBc_pad + POOL_BLOCKS - 1) / POOL_BLOCKS, BH);
  switch (a.R) {
    case 4: hipLaunchKernelGGL(pool_kernel<4>, grid, dim3(192), 0, stream, a); break;
    case 8: hipLaunchKernelGGL(pool_kernel<8>, grid, dim3(192), 0, stream, a); break;
    case 16: hipLaunchKernelGGL(pool_kernel<16>, grid, dim3(192), 0, stream, a); break;
    case 32: hipLaunchKernelGGL(pool_kernel<32>, grid, dim3(192), 0, stream, a); break;
    default: hipLaunchKernelGGL(pool_kernel<64>, grid, dim3(192), 0, stream, a); break;
  }
}

struct FuseArgs {
  const e16_t *dout, *of, *oc, *gate;
  e16_t *o, *dout_f, *dout_c, *dgate;
  float *delta_f, *delta_c;
  const int* blk_cnt;
  int NB, L, NBc_pad, gate_mode, gate_act;
  int ld;  // columns of a stored row
};

// Both fusion kernels: one workgroup per 64-token block (grid (blocks, BH), 256 threads), thread -> (row slot
// s = thread / 16, column chunk c8 = 8 * (thread % 16)), which walks rows s, s + 16, s + 32, s + 48 with all four rows'
// loads in flight. (One wave per block walked sixteen rows a lane, and the backward's row sums went through LDS
// shuffles. 264 blocks, 12 heads, elementwise gate: forward 40 -> 28 us, 3.6 TB/s, backward 55 -> 40 us, 3.9 TB/s; 64
// blocks, two heads: 10 -> 4.5 and 16 -> 6 us.)
__global__ __launch_bounds__(256) void fuse_fwd_kernel(FuseArgs a) {
  const int blk = blockIdx.x, s = threadIdx.x >> 4, c8 = (threadIdx.x & 15) * 8, ld = a.ld;
  if (c8 >= ld) return;
  const size_t bh = blockIdx.y;
  const int n = a.blk_cnt[blk];
  float c[8];
  ld8(a.oc + (bh * a.NBc_pad + blk) * ld + c8, c);
  const size_t tok0 = bh * a.L + (size_t)blk * BK;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int r = s + 16 * i;
    const size_t tok = tok0 + r;
    float x[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    if (r < n) {
      ld8(a.of + tok * ld + c8, x);
      if (a.gate_mode == 1) {
        const float g = gact(e2f(a.gate[tok]), a.gate_act);
#pragma unroll
        for (int e = 0; e < 8; ++e) x[e] += g * c[e];
      } else if (a.gate_mode == 2) {
        float g[8];
        ld8(a.gate + tok * ld + c8, g);
#pragma unroll
        for (int e = 0; e < 8; ++e) x[e] += gact(g[e], a.gate_act) * c[e];
      } else {
#pragma unroll
        for (int e = 0; e < 8; ++e) x[e] += c[e];
      }
    }
    st8(a.o + tok * ld + c8, x);
  }
}

__global__ __launch_bounds__(256) void fuse_bwd_kernel(FuseArgs a) {
  __shared__ __attribute__((aligned(16))) float dc_s[16][HD];  // [row slot][column]: sums over the slot's rows
  const int blk = blockIdx.x, s = threadIdx.x >> 4, c8 = (threadIdx.x & 15) * 8, ld = a.ld;
  const bool col = c8 < ld;  // (lanes past a stored row hold zeros and store nothing)
  const size_t bh = blockIdx.y;
  const size_t crow = (bh * a.NBc_pad + blk) * ld;
  if (blk >= a.NB) {  // padding rows of the coarse tensors
    if (s == 0 && col) *reinterpret_cast<uint4*>(a.dout_c + crow + c8) = uint4{0u, 0u, 0u, 0u};
    if (threadIdx.x == 0) a.delta_c[bh * a.NBc_pad + blk] = 0.f;
    return;
  }
  const int n = a.blk_cnt[blk];
  float c[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f}, dc[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
  if (col) ld8(a.oc + crow + c8, c);
  const size_t tok0 = bh * a.L + (size_t)blk * BK;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int r = s + 16 * i;
    const size_t tok = tok0 + r;
    const bool valid = r < n;
    float d[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f}, f[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    if (valid && col) {
      ld8(a.dout + tok * ld + c8, d);
      ld8(a.of + tok * ld + c8, f);
    }
    if (a.dout_f != nullptr && col) st8(a.dout_f + tok * ld + c8, d);
    float dot_f = 0.f, dot_c = 0.f;
#pragma unroll
    for (int e = 0; e < 8; ++e) dot_f += d[e] * f[e];
    if (a.gate_mode == 1) {
      const float g = valid ? gact(e2f(a.gate[tok]), a.gate_act) : 0.f;
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        dot_c += d[e] * c[e];
        dc[e] += g * d[e];
      }
      dot_c *= gdact(g, a.gate_act);
    } else if (a.gate_mode == 2) {
      float g[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f}, dg[8];
      if (valid && col) ld8(a.gate + tok * ld + c8, g);
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const float ge = valid ? gact(g[e], a.gate_act) : 0.f;
        dg[e] = valid ? gdact(ge, a.gate_act) * d[e] * c[e] : 0.f;
        dc[e] += ge * d[e];
      }
      if (col) st8(a.dgate + tok * ld + c8, dg);
    } else {
#pragma unroll
      for (int e = 0; e < 8; ++e) dc[e] += d[e];
    }
    dot_f = row16_sum(dot_f);
    if (a.gate_mode == 1) dot_c = row16_sum(dot_c);
    if ((threadIdx.x & 15) == 15) {
      a.delta_f[tok] = valid ? dot_f : 0.f;
      if (a.gate_mode == 1) a.dgate[tok] = f2e(valid ? dot_c : 0.f);
    }
  }
  // dO_c = the sixteen row slots' column sums (fixed order), rounded; delta_c = <dO_c (rounded), O_c>
#pragma unroll
  for (int e = 0; e < 8; e += 4)
    *reinterpret_cast<f32x4*>(&dc_s[s][c8 + e]) = f32x4{dc[e], dc[e + 1], dc[e + 2], dc[e + 3]};
  __syncthreads();
  if (s != 0) return;
#pragma unroll
  for (int g = 1; g < 16; ++g)
#pragma unroll
    for (int e = 0; e < 8; ++e) dc[e] += dc_s[g][c8 + e];
  float part = 0.f;
  if (col) {
    st8(a.dout_c + crow + c8, dc);
#pragma unroll
    for (int e = 0; e < 8; ++e) part += e2f(f2e(dc[e])) * c[e];
  }
  part = row16_sum(part);
  if (threadIdx.x == 15) a.delta_c[bh * a.NBc_pad + blk] = part;
}

// grid (cdiv(NB, 4), BH), 256 threads: one wave per 64-token block; acc fp32 [BH, L, D] (optional), add fp32
// [BH, add_nb, D] (optional)
__global__ __launch_bounds__(256) void finalize_kernel(const float* __restrict__ acc, const float* __restrict__ add,
                                                       e16_t* __restrict__ out, const int* __restrict__ blk_cnt,
                                                       int NB, int L, int add_nb, int ld) {
  const int blk = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (blk >= NB) return;
  const int l = threadIdx.x & 63, s = l >> 4, c8 = (l & 15) * 8;
  if (c8 >= ld) return;
  const size_t bh = blockIdx.y;
  const int n = blk_cnt[blk];
  float ad[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
  if (add != nullptr) {
    const float inv = 1.f / (float)n;
    const float4* p = reinterpret_cast<const float4*>(add + (bh * add_nb + blk) * ld + c8);
    const float4 u = p[0], w = p[1];
    ad[0] = u.x * inv; ad[1] = u.y * inv; ad[2] = u.z * inv; ad[3] = u.w * inv;
    ad[4] = w.x * inv; ad[5] = w.y * inv; ad[6] = w.z * inv; ad[7] = w.w * inv;
  }
  const size_t tok0 = bh * L + (size_t)blk * BK;
#pragma unroll 4
  for (int r = s; r < BK; r += 4) {
    const size_t tok = tok0 + r;
    float x[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    if (r < n) {
      if (acc != nullptr) {
        const float4* p = reinterpret_cast<const float4*>(acc + tok * ld + c8);
        const float4 u = p[0], w = p[1];
        x[0] = u.x; x[1] = u.y; x[2] = u.z; x[3] = u.w; x[4] = w.x; x[5] = w.y; x[6] = w.z; x[7] = w.w;
      }
#pragma unroll
      for (int e = 0; e < 8; ++e) x[e] += ad[e];
    }
    st8(out + tok * ld + c8, x);
  }
}

// log2 of the valid tokens of every representative group (RM per block) and of every block; -inf when empty
__global__ void rep_counts_kernel(const int* __restrict__ blk_cnt, float* __restrict__ lc_mid,
                                  float* __restrict__ lc_tail, int NB, int RM) {
  const int e = blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= NB * RM) return;
  const int blk = e / RM, g = e - blk * RM, gs = BK / RM;
  const int cnt = blk_cnt[blk];
  const int n = min(max(cnt - g * gs, 0), gs);
  lc_mid[e] = n > 0 ? log2f((float)n) : -INFINITY;
  if (g == 0) lc_tail[blk] = cnt > 0 ? log2f((float)cnt) : -INFINITY;
}

}  // namespace

}  // namespace es

using namespace es;

static int check_tokens(int BH, int L, int D, HeadDim& h) {
  ES_REQUIRE(BH > 0 && BH <= 65535 && L > 0 && L % BK == 0, ES_ERR_INVALID,
             "VSA: tokens must be [BH <= 65535, L = NB * 64, D]");
  VSA_REQUIRE_DIM(D, h);
  return ES_OK;
}

extern "C" int ES_VSA_API(vsa_pool)(const void* q, const void* k, const void* v, const int* blk_cnt, void* qr, void* kr, void* vr,
                        void* qc, void* kc, void* vc, int BH, int L, int D, int R, hipStream_t stream) {
  HeadDim h;
  if (int st = check_tokens(BH, L, D, h)) return st;
  ES_REQUIRE(q && k && v && blk_cnt && qc && kc && vc, ES_ERR_INVALID, "VSA: null tensor pointer");
  ES_REQUIRE(R == 4 || R == 8 || R == 16 || R == 32, ES_ERR_INVALID, "VSA2: router pool size R must be 4, 8, 16 or 32");
  const int NB = L / BK, G = BK / R;
  PoolArgs a{{(const e16_t*)q, (const e16_t*)k, (const e16_t*)v},
             {(e16_t*)qr, (e16_t*)kr, (e16_t*)vr},
             {(e16_t*)qc, (e16_t*)kc, (e16_t*)vc},
             blk_cnt, NB, L, R, (NB * G + 63) / 64 * 64, (NB + 63) / 64 * 64, h.ld};
  launch_pool(a, BH, stream);
  return check_launch("vsa_pool");
}

extern "C" int ES_VSA_API(vsa_fuse_fwd)(const void* of, const void* oc, const void* gate, void* o, const int* blk_cnt, int BH,
                            int L, int D, int NBc_pad, int gate_mode, int gate_act, hipStream_t stream) {
  HeadDim h;
  if (int st = check_tokens(BH, L, D, h)) return st;
  ES_REQUIRE(of && oc && o && blk_cnt && (gate_mode == 0 || gate), ES_ERR_INVALID, "VSA: null tensor pointer");
  ES_REQUIRE(gate_mode >= 0 && gate_mode <= 2 && (gate_act == 0 || gate_act == 1), ES_ERR_INVALID,
             "VSA: gate_mode must be 0 (none), 1 (per token) or 2 (elementwise), gate_act 0 (tanh) or 1 (identity)");
  const int NB = L / BK;
  ES_REQUIRE(NBc_pad >= NB, ES_ERR_INVALID, "VSA: coarse output has fewer rows than blocks");
  FuseArgs a{nullptr, (const e16_t*)of, (const e16_t*)oc, (const e16_t*)gate, (e16_t*)o, nullptr, nullptr, nullptr,
             nullptr, nullptr, blk_cnt, NB, L, NBc_pad, gate_mode, gate_act, h.ld};
  hipLaunchKernelGGL(fuse_fwd_kernel, dim3(NB, BH), dim3(256), 0, stream, a);
  return check_launch("vsa_fuse_fwd");
}

extern "C" int ES_VSA_API(vsa_fuse_bwd)(const void* dout, const void* of, const void* oc, const void* gate, void* dout_f,
                            float* delta_f, void* dout_c, float* delta_c, void* dgate, const int* blk_cnt, int BH,
                            int L, int D, int NBc_pad, int gate_mode, int gate_act, hipStream_t stream) {
  HeadDim h;
  if (int st = check_tokens(BH, L, D, h)) return st;
  ES_REQUIRE(dout && of && oc && delta_f && dout_c && delta_c && blk_cnt, ES_ERR_INVALID, "VSA: null tensor pointer");
  ES_REQUIRE(gate_mode >= 0 && gate_mode <= 2 && (gate_act == 0 || gate_act == 1), ES_ERR_INVALID,
             "VSA: gate_mode must be 0 (none), 1 (per token) or 2 (elementwise), gate_act 0 (tanh) or 1 (identity)");
  ES_REQUIRE(gate_mode == 0 || (gate && dgate), ES_ERR_INVALID, "VSA: a gated fusion needs gate and dgate");
  const int NB = L / BK;
  ES_REQUIRE(NBc_pad >= NB, ES_ERR_INVALID, "VSA: coarse output has fewer rows than blocks");
  FuseArgs a{(const e16_t*)dout, (const e16_t*)of, (const e16_t*)oc, (const e16_t*)gate, nullptr, (e16_t*)dout_f,
             (e16_t*)dout_c, (e16_t*)dgate, delta_f, delta_c, blk_cnt, NB, L, NBc_pad, gate_mode, gate_act, h.ld};
  hipLaunchKernelGGL(fuse_bwd_kernel, dim3(NBc_pad, BH), dim3(256), 0, stream, a);
  return check_launch("vsa_fuse_bwd");
}

extern "C" int ES_VSA_API(vsa_finalize)(const float* acc, const float* add, int add_nb, void* out, const int* blk_cnt, int BH,
                            int L, int D, hipStream_t stream) {
  HeadDim h;
  if (int st = check_tokens(BH, L, D, h)) return st;
  ES_REQUIRE(out && blk_cnt, ES_ERR_INVALID, "VSA: null tensor pointer");
  const int NB = L / BK;
  ES_REQUIRE(add == nullptr || add_nb >= NB, ES_ERR_INVALID, "VSA: finalize add has fewer rows than blocks");
  hipLaunchKernelGGL(finalize_kernel, dim3((NB + 3) / 4, BH), dim3(256), 0, stream, acc, add, (e16_t*)out, blk_cnt,
                     NB, L, add_nb, h.ld);
  return check_launch("vsa_finalize");
}

extern "C" int ES_VSA_API(vsa_rep_build)(const void* k, const void* v, const int* blk_cnt, void* k_mid, void* v_mid,
                             float* lc_mid, void* k_tail, void* v_tail, float* lc_tail, int BH, int L, int D, int RM,
                             hipStream_t stream) {
  HeadDim h;
  if (int st = check_tokens(BH, L, D, h)) return st;
  ES_REQUIRE(D == h.d, ES_ERR_UNSUPPORTED, "VSA2-rep: rows must be stored with 128 columns");
  ES_REQUIRE(k && v && blk_cnt && k_mid && v_mid && lc_mid && k_tail && v_tail && lc_tail, ES_ERR_INVALID,
             "VSA2-rep: null tensor pointer");
  ES_REQUIRE(RM == 1 || RM == 2 || RM == 4 || RM == 8 || RM == 16, ES_ERR_INVALID,
             "RepTiers.mid_reps must be one of (1, 2, 4, 8, 16)");
  const int NB = L / BK, R = BK / RM;
  // the mid table is the pooled groups of R = 64 / RM tokens, the tail table the block means
  PoolArgs a{{nullptr, (const e16_t*)k, (const e16_t*)v},
             {nullptr, (e16_t*)k_mid, (e16_t*)v_mid},
             {nullptr, (e16_t*)k_tail, (e16_t*)v_tail},
             blk_cnt, NB, L, R, (NB * RM + 63) / 64 * 64, (NB + 63) / 64 * 64, HD};
  launch_pool(a, BH, stream);
  hipLaunchKernelGGL(rep_counts_kernel, dim3((NB * RM + 255) / 256), dim3(256), 0, stream, blk_cnt, lc_mid, lc_tail,
                     NB, RM);
  return check_launch("vsa_rep_build");
}
