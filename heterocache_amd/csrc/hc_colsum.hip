// Column sums of a whole prompt's attention on gfx950 MFMA:
//
//   out[b, h, t] = sum_i softmax_t(scale * q[b, h, i] . k[b, h, t]),  i, t < L
//
// the heavy-hitter scores of H2OKVCluster.update_kv (heterocache/
// kv_cluster.py:434-447: softmax over all keys, no mask, summed over every
// query position).  Two passes of one kernel with the roles swapped:
//
//   pass 1: columns = queries, streamed rows = keys  -> log-sum-exp per query
//   pass 2: columns = keys, streamed rows = queries  -> sum of exp2(s - lse)
//
// Structure: a wave keeps the operands of NC blocks of 16 columns in
// registers and walks the streamed rows 64 at a time; the rows are staged
// through double-buffered LDS by the four waves of a workgroup (LDS-DMA
// loads, the KV store's tile layout, so an MFMA operand is one 16-byte read
// and feeds NC matrix instructions).  The 16 x 16 blocks of S are reduced in
// the accumulators; nothing of size L x L leaves the registers.
//
// What bounds it: per 16 x 16 block 64 matrix cycles, and 4 elements a lane
// of fma + v_exp (a quarter of the VALU rate) + add, which the other waves of
// the SIMD (four resident at 124 and 126 registers) run beside the matrix
// instructions, and under load the chip's power.  At 32 heads x 8190 tokens
// the matrix pipe is busy half of the cycles, waves wait for dependencies half
// of theirs, LDS is active in 12 and 16 % without conflicts, and a pass takes
// 0.54-0.67 ms with the clock.  (So an order with one block's exponentials
// between the next block's matrix instructions, three waves a SIMD, measured
// no faster: 1.11 ms against 1.07.)
// Pass 1 takes no maximum in its loop: the row reference m is the maximum of
// the first rows, and an iteration's sums are only redone against a new
// maximum when they pass kCsLazy (the sums are needed anyway; one compare
// replaces 16 maxima a lane and the cross-lane fold).  The terms and sums stay
// float32 and no counted exponent passes log2(kCsLazy), so a sum is as exact
// as one against the true maximum.  Against 32 calls of the window scorer, 256
// query rows each (two launches and a merge per call, keys re-read by each):
// 2.63 -> 1.02 ms at 32 heads x 8190 tokens float16 (208 -> 540 TFLOP/s,
// counting the product once; it is formed twice), 0.70 -> 0.18 ms at 3000,
// 0.097 -> 0.026 ms at 400.
#include <algorithm>
#include <cfloat>
#include <cmath>

#include "hc_common.h"
#include "hc_internal.h"

namespace hc {
namespace {

constexpr int kCsWaves = 4;
constexpr int kCsThreads = kCsWaves * 64;
constexpr int kCsRows = 64;       // streamed rows per iteration
constexpr int kCsLseIts = 16;     // iterations whose log-sum-exps are staged together (pass 2)
constexpr int kCsLseRows = kCsLseIts * kCsRows;
constexpr float kCsLazy = 128.f;  // pass 1: largest sum of a lane's terms of an iteration before m moves

struct CsArgs {
  const void* x;  // columns
  const void* y;  // streamed rows
  int64_t x_sb, x_sh, x_st, y_sb, y_sh, y_st;  // element strides: batch, head, token
  int H, L, njobs, nxb, nsplit, its;  // column blocks, splits of the streamed rows, iterations per split
  float scale2;
  float* ml;   // [job][split][L][2]: (m, l) of pass 1
  float* out;  // pass 2: [job][split][L]
};

// Column blocks of 16 a wave holds (64 registers of operands either way).
template <typename T>
constexpr int cs_nc() {
  return sizeof(T) == 4 ? 2 : 4;
}
template <typename T>
constexpr int cs_block() {
  return kCsWaves * 16 * cs_nc<T>();
}
template <typename T>
constexpr size_t cs_lds_bytes() {
  return (size_t)2 * kCsRows * HC_HEAD_DIM * sizeof(T) + (size_t)2 * kCsLseRows * sizeof(float);
}

template <typename T, int PASS>
__global__ __launch_bounds__(kCsThreads, sizeof(T) == 4 ? 2 : 4) void column_sum_kernel(const CsArgs a) {
  typedef typename Elem<T>::vec8 vec8;
  constexpr int NC = cs_nc<T>();
  constexpr int kUnits = (int)sizeof(T) / 2;  // 16-byte units per 8-element chunk
  constexpr int kSet = kCsRows * HC_HEAD_DIM;  // elements of one staged set
  extern __shared__ __attribute__((aligned(16))) unsigned char cs_lds[];
  T* const lds = reinterpret_cast<T*>(cs_lds);
  float* const s_lse = reinterpret_cast<float*>(cs_lds + (size_t)2 * kSet * sizeof(T));

  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int g4 = lane >> 4, n16 = lane & 15;
  // Jobs vary fastest: with a multiple of 8 jobs all blocks of a job run on
  // one XCD, whose L2 then holds the rows they stream together.
  const int job = blockIdx.x % a.njobs;
  const int rest = blockIdx.x / a.njobs;
  const int split = rest % a.nsplit, xb = rest / a.nsplit;
  const int b = job / a.H, h = job % a.H;
  const T* const xp = reinterpret_cast<const T*>(a.x) + b * a.x_sb + h * a.x_sh;
  const T* const yp = reinterpret_cast<const T*>(a.y) + b * a.y_sb + h * a.y_sh;
  const int nit_all = (a.L + kCsRows - 1) / kCsRows;
  const int it0 = split * a.its, it1 = min(it0 + a.its, nit_all);
  const int x0 = xb * cs_block<T>() + wave * 16 * NC;

  // Columns past L repeat the last one; their results are not stored.
  vec8 xop[NC][4];
#pragma unroll
  for (int c = 0; c < NC; ++c) {
    const T* p = xp + (int64_t)min(x0 + 16 * c + n16, a.L - 1) * a.x_st + 8 * g4;
#pragma unroll
    for (int s = 0; s < 4; ++s) xop[c][s] = load8(p + 32 * s);
  }

  // Staging: unit w = r * 256 + tid of 16 bytes lands at LDS byte 16 w; it is
  // (half w % kUnits of) chunk w / kUnits of the tile layout.  A load is a
  // uniform base plus a 32-bit offset (the host bounds 64 token strides below
  // 2^31 bytes).  Rows past L repeat the last one and are masked.
  const uint32_t y_stb = (uint32_t)(a.y_st * (int64_t)sizeof(T));
  auto stage = [&](int buf, int it) {
    char* sk = reinterpret_cast<char*>(lds + buf * kSet);
    const char* yit = reinterpret_cast<const char*>(yp) + (int64_t)it * kCsRows * a.y_st * (int64_t)sizeof(T);
    const int last = a.L - 1 - it * kCsRows;
#pragma unroll
    for (int r = 0; r < 4 * kUnits; ++r) {
      const int w = r * kCsThreads + tid;
      const int u = w / kUnits, half = w % kUnits;
      const int v = u & 511, t = (u >> 9) * HC_TILE + (v >> 8) * 16 + (v & 15);
      const int d = 32 * ((v >> 6) & 3) + 8 * ((v >> 4) & 3) + half * 4;
      lds_dma16(yit + (uint32_t)min(t, last) * y_stb + (uint32_t)(d * (int)sizeof(T)),
                sk + 16 * (r * kCsThreads + wave * 64));
    }
  };
  // Log-sum-exps of the next kCsLseRows streamed rows (+inf past L: those
  // rows add exp2(-inf) = 0), folded from pass 1's splits.
  auto stage_lse = [&](int blk) {
    float* s = s_lse + (blk & 1) * kCsLseRows;
    for (int i = tid; i < kCsLseRows; i += kCsThreads) {
      const int y = (it0 + blk * kCsLseIts) * kCsRows + i;
      float v = INFINITY;
      if (y < a.L) {
        const float* p = a.ml + ((int64_t)job * a.nsplit * a.L + y) * 2;
        float m = p[0], l = p[1];
        for (int sp = 1; sp < a.nsplit; ++sp) {
          const float m2 = p[(int64_t)sp * a.L * 2], l2 = p[(int64_t)sp * a.L * 2 + 1];
          const float mn = fmaxf(m, m2);
          l = l * fast_exp2(m - mn) + l2 * fast_exp2(m2 - mn);
          m = mn;
        }
        v = m + __log2f(l);
      }
      s[i] = v;
    }
  };

  float m[NC], sum[NC], sum8[NC];
#pragma unroll
  for (int c = 0; c < NC; ++c) {
    m[c] = -FLT_MAX;
    sum[c] = 0.f;
    sum8[c] = 0.f;
  }

  if (it0 < it1) stage(0, it0);
  for (int it = it0; it < it1; ++it) {
    const int n = it - it0, cur = n & 1;
    if constexpr (PASS == 2) {
      // Written to the other half of s_lse than the one waves behind the
      // last barrier may still read.
      if ((n % kCsLseIts) == 0) stage_lse(n / kCsLseIts);
    }
    wait_lds_dma();
    __syncthreads();  // set `it` is whole, and every wave is done with the other one
    if (it + 1 < it1) stage(cur ^ 1, it + 1);
    const T* sk = lds + cur * kSet;
    const int left = a.L - it * kCsRows;  // valid rows of this set, if below kCsRows
    // Rows 16 tb + 4 g4 + r of the set against the wave's columns.
    auto products = [&](int tb, f32x4 (&acc)[NC]) {
      const T* kt = sk + (tb >> 1) * HC_TILE_ELEMS + (tb & 1) * 4 * 64 * 8;
#pragma unroll
      for (int c = 0; c < NC; ++c) acc[c] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int s = 0; s < 4; ++s) {
        const vec8 ka = load8(kt + (s * 64 + lane) * 8);
#pragma unroll
        for (int c = 0; c < NC; ++c) acc[c] = mma_16x16x32(ka, xop[c][s], acc[c]);
      }
    };
    if constexpr (PASS == 1) {
      auto mask = [&](int tb, f32x4 (&acc)[NC]) {
#pragma unroll
        for (int r = 0; r < 4; ++r)
          if (16 * tb + 4 * g4 + r >= left) {
#pragma unroll
            for (int c = 0; c < NC; ++c) acc[c][r] = -INFINITY;
          }
      };
      float ps[NC];
#pragma unroll
      for (int c = 0; c < NC; ++c) ps[c] = 0.f;
      // A set that reaches past L takes the masked form below at once.
      bool redo = left < kCsRows;
      if (!redo) {
#pragma unroll
        for (int tb = 0; tb < 4; ++tb) {
          f32x4 acc[NC];
          products(tb, acc);
#pragma unroll
          for (int c = 0; c < NC; ++c) {
            float p[4];
#pragma unroll
            for (int r = 0; r < 4; ++r) p[r] = fast_exp2(fmaf(acc[c][r], a.scale2, -m[c]));
            ps[c] += (p[0] + p[1]) + (p[2] + p[3]);
          }
        }
        float worst = ps[0];
#pragma unroll
        for (int c = 1; c < NC; ++c) worst += ps[c];
        redo = __any(!(worst <= kCsLazy));  // no sum is negative; a NaN fails the comparison
      }
      if (redo) {
        float mx[NC];
#pragma unroll
        for (int c = 0; c < NC; ++c) mx[c] = -FLT_MAX;
#pragma unroll 1
        for (int tb = 0; tb < 4; ++tb) {
          f32x4 acc[NC];
          products(tb, acc);
          mask(tb, acc);
#pragma unroll
          for (int c = 0; c < NC; ++c)
#pragma unroll
            for (int r = 0; r < 4; ++r) mx[c] = fmaxf(mx[c], acc[c][r] * a.scale2);
        }
#pragma unroll
        for (int c = 0; c < NC; ++c) {
          const float mn = fmaxf(m[c], rows4_max(mx[c]));
          const float alpha = fast_exp2(m[c] - mn);
          sum[c] *= alpha;
          sum8[c] *= alpha;
          m[c] = mn;
          ps[c] = 0.f;
        }
#pragma unroll 1
        for (int tb = 0; tb < 4; ++tb) {
          f32x4 acc[NC];
          products(tb, acc);
          mask(tb, acc);
#pragma unroll
          for (int c = 0; c < NC; ++c)
#pragma unroll
            for (int r = 0; r < 4; ++r) ps[c] += fast_exp2(fmaf(acc[c][r], a.scale2, -m[c]));
        }
      }
#pragma unroll
      for (int c = 0; c < NC; ++c) sum8[c] += ps[c];
    } else {
      const float* ls = s_lse + ((n / kCsLseIts) & 1) * kCsLseRows + (n % kCsLseIts) * kCsRows + 4 * g4;
      float ps[NC];
#pragma unroll
      for (int c = 0; c < NC; ++c) ps[c] = 0.f;
#pragma unroll
      for (int tb = 0; tb < 4; ++tb) {
        f32x4 acc[NC];
        products(tb, acc);
        const f32x4 e = *reinterpret_cast<const f32x4*>(ls + 16 * tb);
#pragma unroll
        for (int c = 0; c < NC; ++c) {
          float p[4];
#pragma unroll
          for (int r = 0; r < 4; ++r) p[r] = fast_exp2(fmaf(acc[c][r], a.scale2, -e[r]));
          ps[c] += (p[0] + p[1]) + (p[2] + p[3]);
        }
      }
#pragma unroll
      for (int c = 0; c < NC; ++c) sum8[c] += ps[c];
    }
    // Sums of eight iterations first: a run of L / 64 additions onto one
    // growing sum would round more than the terms do.
    if ((n & 7) == 7) {
#pragma unroll
      for (int c = 0; c < NC; ++c) {
        sum[c] += sum8[c];
        sum8[c] = 0.f;
      }
    }
  }
#pragma unroll
  for (int c = 0; c < NC; ++c) {
    const float v = rows4_sum(sum[c] + sum8[c]);
    const int x = x0 + 16 * c + n16;
    if (g4 != 0 || x >= a.L) continue;
    const int64_t o = ((int64_t)job * a.nsplit + split) * a.L + x;
    if constexpr (PASS == 1) {
      a.ml[2 * o] = m[c];
      a.ml[2 * o + 1] = v;
    } else {
      a.out[o] = v;
    }
  }
}

// out[job][t] = sum over the splits, in their order.
__global__ __launch_bounds__(256) void column_sum_merge_kernel(const float* __restrict__ part, int nsplit, int L,
                                                               float* __restrict__ out) {
  const int t = blockIdx.x * 256 + threadIdx.x, job = blockIdx.y;
  if (t >= L) return;
  const float* p = part + (int64_t)job * nsplit * L + t;
  float v = 0.f;
#pragma unroll 4
  for (int s = 0; s < nsplit; ++s) v += p[(int64_t)s * L];
  out[(int64_t)job * L + t] = v;
}

// Splits of the streamed rows: the count that gives the busiest CU the least
// work, in iterations, with kCsSetup for a workgroup's start (its column
// operands, the first set, the first maximum) and kCsMerge for the fold of
// the splits.  With every workgroup resident a CU's matrix cores are shared
// by its workgroups, so only their number matters.  Measured (float16, 32
// heads, us): 400 tokens 34 with one split, 25 with three; 1500 tokens 73 /
// 67 / 79 with three / four / six; 4100 tokens 335 / 330 / 363 with two /
// four / eight; 8192 tokens 1018 / 1026 / 1045 with one / two / four, and on
// 28 heads 947 / 861 / 905 / 946 with one / two / three / five.
constexpr int kCsCus = 256;
constexpr int kCsMinIts = 2;  // iterations a split keeps
constexpr int kCsMaxSplits = 64;
constexpr float kCsSetup = 1.5f, kCsMerge = 2.f;
template <typename T>
int cs_splits(int64_t njobs, int L) {
  const int64_t blocks = njobs * ((L + cs_block<T>() - 1) / cs_block<T>());
  const int nit = (L + kCsRows - 1) / kCsRows;
  int best = 1;
  double best_cost = 0.;
  for (int n = 1; n <= kCsMaxSplits && (n == 1 || nit / n >= kCsMinIts); ++n) {
    const int its = (nit + n - 1) / n;
    if ((nit + its - 1) / its != n) continue;  // the last split would be empty
    const double cost = (double)((blocks * n + kCsCus - 1) / kCsCus) * (its + kCsSetup) + (n > 1 ? kCsMerge : 0.f);
    if (n == 1 || cost < best_cost) best = n, best_cost = cost;
  }
  return best;
}

int cs_splits_dtype(int dtype, int64_t njobs, int L) {
  return dtype == HC_DTYPE_F32 ? cs_splits<float>(njobs, L) : cs_splits<__bf16>(njobs, L);
}

template <typename T>
int launch_column_sums(CsArgs a, const void* q, const int64_t* qs, const void* k, const int64_t* ks, float* part,
                       float* out, hipStream_t s) {
  a.nxb = (a.L + cs_block<T>() - 1) / cs_block<T>();
  const int64_t grid = (int64_t)a.njobs * a.nxb * a.nsplit;
  if (grid > 0x7fffffffLL) return set_error(HC_ERR_INVALID, "hc_attn_column_sums: grid too large");
  const size_t lds = cs_lds_bytes<T>();
  auto f1 = column_sum_kernel<T, 1>;
  auto f2 = column_sum_kernel<T, 2>;
  for (const void* f : {reinterpret_cast<const void*>(f1), reinterpret_cast<const void*>(f2)}) {
    const hipError_t e = hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    if (e != hipSuccess) return set_error(HC_ERR_HIP, "hc_attn_column_sums: %s", hipGetErrorString(e));
  }
  a.x = q, a.x_sb = qs[0], a.x_sh = qs[1], a.x_st = qs[2];
  a.y = k, a.y_sb = ks[0], a.y_sh = ks[1], a.y_st = ks[2];
  hipLaunchKernelGGL(f1, dim3((unsigned)grid), dim3(kCsThreads), lds, s, a);
  int rc = check_launch("hc_attn_column_sums(pass 1)");
  if (rc) return rc;
  std::swap(a.x, a.y);
  std::swap(a.x_sb, a.y_sb);
  std::swap(a.x_sh, a.y_sh);
  std::swap(a.x_st, a.y_st);
  a.out = a.nsplit > 1 ? part : out;
  hipLaunchKernelGGL(f2, dim3((unsigned)grid), dim3(kCsThreads), lds, s, a);
  if ((rc = check_launch("hc_attn_column_sums(pass 2)"))) return rc;
  if (a.nsplit > 1) {
    hipLaunchKernelGGL(column_sum_merge_kernel, dim3((a.L + 255) / 256, a.njobs), dim3(256), 0, s, part, a.nsplit, a.L,
                       out);
    rc = check_launch("hc_attn_column_sums(merge)");
  }
  return rc;
}

}  // namespace
}  // namespace hc

using namespace hc;

extern "C" size_t hc_attn_column_sums_workspace(int dtype, int batch, int heads, int seq_len) {
  if (batch <= 0 || heads <= 0 || seq_len <= 0) return 0;
  const int64_t njobs = (int64_t)batch * heads;
  const int64_t ns = cs_splits_dtype(dtype, njobs, seq_len);
  return (size_t)(njobs * ns * seq_len) * (ns > 1 ? 3 : 2) * sizeof(float);
}

extern "C" int hc_attn_column_sums(int dtype, const void* q, const int64_t* q_strides, const void* k,
                                   const int64_t* k_strides, int batch, int heads, int seq_len, float scale, float* out,
                                   void* workspace, size_t workspace_bytes, void* stream) {
  clear_error();
  const int esz = dtype == HC_DTYPE_F32 ? 4 : (dtype == HC_DTYPE_BF16 || dtype == HC_DTYPE_F16) ? 2 : 0;
  if (esz == 0) return set_error(HC_ERR_INVALID, "hc_attn_column_sums: unknown dtype %d", dtype);
  if (batch < 0 || heads < 0 || seq_len < 0 || (int64_t)batch * heads > 65535)
    return set_error(HC_ERR_INVALID, "hc_attn_column_sums: batch=%d heads=%d seq_len=%d", batch, heads, seq_len);
  if (batch == 0 || heads == 0 || seq_len == 0) return HC_OK;
  if (!q || !k || !q_strides || !k_strides || !out || !workspace)
    return set_error(HC_ERR_INVALID, "hc_attn_column_sums: null pointer argument");
  if (((uintptr_t)q | (uintptr_t)k | (uintptr_t)workspace) & 15)
    return set_error(HC_ERR_INVALID, "hc_attn_column_sums: buffers must be 16-byte aligned");
  for (int j = 0; j < 3; ++j)
    if (q_strides[j] < 0 || (q_strides[j] * esz) % 16 || k_strides[j] < 0 || (k_strides[j] * esz) % 16)
      return set_error(HC_ERR_INVALID, "hc_attn_column_sums: strides must be non-negative 16-byte multiples");
  if ((int64_t)kCsRows * std::max(q_strides[2], k_strides[2]) * esz >= (int64_t)1 << 31)
    return set_error(HC_ERR_INVALID, "hc_attn_column_sums: token strides too large");
  if (!std::isfinite(scale) || !(scale > 0.f))
    return set_error(HC_ERR_INVALID, "hc_attn_column_sums: scale must be finite and positive");
  if (workspace_bytes < hc_attn_column_sums_workspace(dtype, batch, heads, seq_len))
    return set_error(HC_ERR_INVALID, "hc_attn_column_sums: workspace too small");
  CsArgs a = {};
  a.H = heads;
  a.L = seq_len;
  a.njobs = batch * heads;
  a.nsplit = cs_splits_dtype(dtype, a.njobs, seq_len);
  const int nit = (seq_len + kCsRows - 1) / kCsRows;
  a.its = (nit + a.nsplit - 1) / a.nsplit;
  a.scale2 = scale * 1.4426950408889634f;
  a.ml = reinterpret_cast<float*>(workspace);
  float* part = a.ml + (int64_t)a.njobs * a.nsplit * seq_len * 2;
  hipStream_t s = (hipStream_t)stream;
  switch (dtype) {
    case HC_DTYPE_BF16: return launch_column_sums<__bf16>(a, q, q_strides, k, k_strides, part, out, s);
    case HC_DTYPE_F16: return launch_column_sums<_Float16>(a, q, q_strides, k, k_strides, part, out, s);
    default: return launch_column_sums<float>(a, q, q_strides, k, k_strides, part, out, s);
  }
}
