// fp32-mode triangle attention for gfx950: LayerNorm, the q | k | v | g and triangle
// bias projections and the attention's operands in one pass over x, then the
// split-bf16 attention (pair_bias.hip).  Upstream's fp32 forward is
// TriangleAttention with autocast off (reference triangle.py:38-52).
//
// What bounds it: HBM.  The projection reads 512 B and writes 2.1 KB per pair
// (q and g fp32, K and V^T as bf16 high / low parts).  As separate passes (LayerNorm
// to a split operand, library GEMM to fp32 rows, a bias permute, the K / V split)
// the same step moved 7 KB per pair: 751 us at n = 576, this kernel 178 (4.8
// TB/s).
// Products are split bf16 (xh wh + xl wh + xh wl, about 2^-16 relative), as the
// library GEMM's were.
#include "bmx_common.h"

using namespace bmx;

namespace {

constexpr int kH = 4, kD = 32;
constexpr int kTP = 64;            // pairs per tile
constexpr int kWaves = 16;         // wave w: head w % 4 of q, k, v or g (w / 4)
constexpr int kKRow = kD + 8;      // staged K row of one pair (bf16)
constexpr int kVRow = kTP + 8;     // staged V^T row of one head dim (bf16)

__device__ __forceinline__ f32x4 mfma16(bf16x8 a, bf16x8 b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}

// Key slot inside a 32-key block: the attention's P operand order (x3_slot of pair_bias.hip).
__device__ __forceinline__ int key_slot(int key) { return ((key & 15) >> 2) * 8 + (key >> 4) * 4 + (key & 3); }

struct ProjArgs {
  const float *x, *mask, *ln_w, *ln_b;
  const bf16* w;         // packed split weight [q; k; v; g], 512 x 128
  const float* b;        // [512 + 4]
  const bf16* w_bias;    // triangle bias rows, [high, low][16][128], rows 4..15 zero
  float eps, inf;
  int n, nkp, i0, rows;  // frame rows i0 .. i0 + rows - 1
  float* qg;             // [rows][n][q 128 | g 128]; null: triangle bias only
  bf16 *kh, *kl, *vth, *vtl;  // [rows][4][nkp][32], [rows][4][32][nkp]
  float* mterm;          // [rows][nkp]
  float* tri_bias;       // [4][n][n]; null: not written
};

// Persistent and weight-stationary: 16 waves keep 32 output rows each (8 k steps,
// high and low: 64 VGPRs), one block per CU, the next tile's rows prefetched into
// registers.  (8 waves of 64 rows spilled at 256 VGPRs, and a scratch reload
// waits for every prefetch and store before it: 347 us against 178.)  q, k, g come as D[output][pair] (4 consecutive
// channels per lane), v as D[pair][dim] (4 consecutive keys).  q and g leave as
// 16-byte stores, K and V^T through an LDS stage stored in the next iteration
// before the next prefetch (vmcnt counts stores in issue order).
template <bool starting>
__global__ __launch_bounds__(64 * kWaves) void triattn_fp32_proj_kernel(ProjArgs a) {
  __shared__ __attribute__((aligned(16))) bf16 xh[kTP * kLdsRow], xl[kTP * kLdsRow];
  __shared__ __attribute__((aligned(16))) bf16 sk[2][kH * kTP * kKRow];
  __shared__ __attribute__((aligned(16))) bf16 sv[2][kH * kD * kVRow];
  __shared__ __attribute__((aligned(16))) bf16 wb[2 * 16 * kLdsRow];
  __shared__ __attribute__((aligned(16))) float sb[4 * kC + kH];
  __shared__ __attribute__((aligned(16))) float sln[2 * kC];  // LayerNorm weight, bias
  const int t = threadIdx.x, l = lane_id(), w = __builtin_amdgcn_readfirstlane(t >> 6);
  const int hw = t >> 5, hl = t & 31, kind = w >> 2, h = w & 3;  // 0 q, 1 k, 2 v, 3 g
  const int n = a.n, nkp = a.nkp;
  const bool project = a.qg != nullptr;
  const int tiles_x = nkp / kTP, total = a.rows * tiles_x;

  bf16x8 wh[8], wl[8];
#pragma unroll
  for (int ks = 0; ks < 8; ++ks) {
    const bf16* src = a.w + ((int64_t)w * 8 + ks) * 1024 + 8 * l;
    wh[ks] = gload8(src);
    wl[ks] = gload8(src + 512);
  }
  for (int e = t; e < 2 * 16 * 16; e += 64 * kWaves)  // 16-byte chunks of the triangle-bias rows
    *(bf16x8*)(wb + (e >> 4) * kLdsRow + 8 * (e & 15)) = gload8(a.w_bias + 8 * e);

  for (int e = t; e < 4 * kC + kH; e += 64 * kWaves) sb[e] = a.b[e];
  if (t < kC) sln[t] = a.ln_w[t], sln[kC + t] = a.ln_b ? a.ln_b[t] : 0.f;
  __syncthreads();
  const float bv = a.b[2 * kC + 32 * h + (l & 31)];

  constexpr int kRowsPer = kTP / (2 * kWaves);
  f32x4 px[kRowsPer];
  float mpre = 1.f;
  auto fetch = [&](int tile) {
    const int i = a.i0 + tile / tiles_x, j0 = (tile % tiles_x) * kTP;
    const int jc = min(j0 + (t & (kTP - 1)), n - 1);
    if (a.mask) mpre = starting ? a.mask[(int64_t)i * n + jc] : a.mask[(int64_t)jc * n + i];
#pragma unroll
    for (int u = 0; u < kRowsPer; ++u) {  // keys past n re-read the last one and are zeroed after the LayerNorm
      const int j = min(j0 + hw + 2 * kWaves * u, n - 1);
      px[u] = load4(a.x + (starting ? (int64_t)i * n + j : (int64_t)j * n + i) * kC + 4 * hl);
    }
  };
  // Coordinates opaque to the compiler, so that it recomputes addresses per
  // tile instead of keeping all of them in registers (which spilled weights).
  auto opaque = [](int v) {
    asm volatile("" : "+v"(v));
    return v;
  };
  auto store_stage = [&](int tile) {
    const int r = tile / tiles_x, j0 = (tile % tiles_x) * kTP, t = opaque(threadIdx.x);
#pragma unroll
    for (int part = 0; part < 2; ++part) {
      bf16 *dk = part ? a.kl : a.kh, *dv = part ? a.vtl : a.vth;
#pragma unroll
      for (int u = 0; u < kH * kTP * kD / 8 / (64 * kWaves); ++u) {
        const int c = t + 64 * kWaves * u;
        const int hk = c >> 8, p = (c >> 2) & (kTP - 1), ck = c & 3;
        *(bf16x8*)(dk + (((int64_t)r * kH + hk) * nkp + j0 + p) * kD + 8 * ck) =
            *(const bf16x8*)(sk[part] + (hk * kTP + p) * kKRow + 8 * ck);
        const int hd = c >> 3, cv = c & 7;  // head * 32 + dim
        *(bf16x8*)(dv + ((int64_t)r * kH * kD + hd) * nkp + j0 + 8 * cv) =
            *(const bf16x8*)(sv[part] + hd * kVRow + 8 * cv);
        __builtin_amdgcn_sched_barrier(0);  // a chunk of each at a time: all of them at once spill weights
      }
    }
  };

  int tile = blockIdx.x, prev = -1;
  if (tile < total) fetch(tile);
  for (; tile < total; tile += gridDim.x) {
    const int r = tile / tiles_x, i = a.i0 + r, j0 = (tile % tiles_x) * kTP;
    bool keep[kRowsPer];
#pragma unroll
    for (int u = 0; u < kRowsPer; ++u) keep[u] = j0 + hw + 2 * kWaves * u < n;
    const int lane4 = 4 * opaque(hl);
    const LnAffine aff{*(const f32x4*)(sln + lane4), *(const f32x4*)(sln + kC + lane4)};
    ln128_half_rows(px, keep, aff, a.eps);
#pragma unroll
    for (int u = 0; u < kRowsPer; ++u) {
      bf16x4 hi, lo;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        hi[e] = (bf16)px[u][e];
        lo[e] = (bf16)(px[u][e] - (float)hi[e]);
      }
      const int at = (hw + 2 * kWaves * u) * kLdsRow + 4 * hl;
      *(bf16x4*)(xh + at) = hi;
      *(bf16x4*)(xl + at) = lo;
    }
    if (project && t < kTP)
      a.mterm[(int64_t)r * nkp + j0 + t] = j0 + t < n ? (1.f - mpre) * -a.inf : -INFINITY;
    if (project && prev >= 0) store_stage(prev);
    __syncthreads();  // x tiles written; the stage has been read
    if (tile + (int)gridDim.x < total) fetch(tile + gridDim.x);

    if (project) {
#pragma unroll
      for (int nt = 0; nt < kTP / 32; ++nt) {
        const int l = opaque(lane_id());
        f32x16 acc = zero16();
        if (kind == 2) {  // wave-uniform
#pragma unroll
          for (int ks = 0; ks < 8; ++ks) {
            const bf16x8 fh = frag(xh, kLdsRow, nt * 32, ks), fl = frag(xl, kLdsRow, nt * 32, ks);
            acc = mfma32(fh, wh[ks], acc);
            acc = mfma32(fl, wh[ks], acc);
            acc = mfma32(fh, wl[ks], acc);
            if (ks % 2) __builtin_amdgcn_sched_barrier(0);  // four fragments read ahead at most
          }
          // D[pair][dim]: lane -> dim l % 32, registers 4c .. 4c+3 -> keys 32 nt + 8 c + 4 (l / 32) + 0..3
#pragma unroll
          for (int c = 0; c < 4; ++c) {
            bf16x4 hi, lo;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
              const int key = nt * 32 + 8 * c + 4 * (l >> 5) + e;
              const float y = j0 + key < n ? acc[4 * c + e] + bv : 0.f;
              hi[e] = (bf16)y;
              lo[e] = (bf16)(y - (float)hi[e]);
            }
            const int at = (h * kD + (l & 31)) * kVRow + nt * 32 + key_slot(8 * c + 4 * (l >> 5));
            *(bf16x4*)(sv[0] + at) = hi;
            *(bf16x4*)(sv[1] + at) = lo;
          }
        } else {
#pragma unroll
          for (int ks = 0; ks < 8; ++ks) {
            const bf16x8 fh = frag(xh, kLdsRow, nt * 32, ks), fl = frag(xl, kLdsRow, nt * 32, ks);
            acc = mfma32(wh[ks], fh, acc);
            acc = mfma32(wh[ks], fl, acc);
            acc = mfma32(wl[ks], fh, acc);
            if (ks % 2) __builtin_amdgcn_sched_barrier(0);
          }
          // D[output][pair]: lane -> pair 32 nt + l % 32, registers 4c .. 4c+3 -> channel 8 c + 4 (l / 32) + 0..3
          const int p = nt * 32 + (l & 31), j = j0 + p;
#pragma unroll
          for (int c = 0; c < 4; ++c) {
            const int d = 8 * c + 4 * (l >> 5);
            f32x4 y = {acc[4 * c], acc[4 * c + 1], acc[4 * c + 2], acc[4 * c + 3]};
            y += *(const f32x4*)(sb + kind * kC + 32 * h + d);
            if (kind == 1) {
              bf16x4 hi, lo;
#pragma unroll
              for (int e = 0; e < 4; ++e) {
                const float v = j < n ? y[e] : 0.f;
                hi[e] = (bf16)v;
                lo[e] = (bf16)(v - (float)hi[e]);
              }
              const int at = (h * kTP + p) * kKRow + d;
              *(bf16x4*)(sk[0] + at) = hi;
              *(bf16x4*)(sk[1] + at) = lo;
            } else if (j < n) {
              store4(a.qg + ((int64_t)r * n + j) * 2 * kC + (kind == 3 ? kC : 0) + 32 * h + d, y);
            }
          }
        }
      }
    }
    if (a.tri_bias && w < 4) {
      // Triangle bias of pairs j0 + 16 w .. + 15 on 16x16x32: D[head][pair], lanes of group 0 hold heads 0..3.
      const int g = l >> 4, lq = l & 15;
      f32x4 ab = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int ks = 0; ks < 4; ++ks) {
        const int ox = (16 * w + lq) * kLdsRow + 32 * ks + 8 * g, ow = lq * kLdsRow + 32 * ks + 8 * g;
        const bf16x8 fh = *(const bf16x8*)(xh + ox), fl = *(const bf16x8*)(xl + ox);
        const bf16x8 bh = *(const bf16x8*)(wb + ow), bl = *(const bf16x8*)(wb + 16 * kLdsRow + ow);
        ab = mfma16(bh, fh, ab);
        ab = mfma16(bh, fl, ab);
        ab = mfma16(bl, fh, ab);
      }
      const int j = j0 + 16 * w + lq;
      if (g == 0 && j < n) {
#pragma unroll
        for (int e = 0; e < kH; ++e) a.tri_bias[((int64_t)e * n + i) * n + j] = ab[e] + sb[4 * kC + e];
      }
    }
    __syncthreads();  // the stage is written; the x tiles have been read
    prev = tile;
  }
  if (project && prev >= 0) store_stage(prev);
}

struct Workspace {
  int64_t qg, kv[4], mterm, total;
};
Workspace make_workspace(int64_t n, int64_t rows) {
  const int64_t nkp = (n + kTP - 1) / kTP * kTP;
  Workspace w;
  int64_t at = 0;
  auto take = [&](int64_t bytes) {
    const int64_t here = at;
    at += (bytes + 255) / 256 * 256;
    return here;
  };
  w.qg = take(rows * n * 2 * kC * 4);
  for (int i = 0; i < 4; ++i) w.kv[i] = take(rows * kC * nkp * 2);
  w.mterm = take(rows * nkp * 4);
  w.total = at;
  return w;
}

}  // namespace

extern "C" {

size_t bmx_triattn_fp32_workspace_bytes(int64_t n, int64_t rows) {
  if (n <= 0 || rows <= 0) return 0;
  return (size_t)make_workspace(n, rows).total;
}

int bmx_triattn_fp32_fwd(const float* x, const float* mask, int64_t n, int starting, int64_t row0, int64_t rows,
                         float inf, const float* ln_w, const float* ln_b, float eps, const void* w_qkvg,
                         const float* b_qkvg, const void* w_bias, float* tri_bias, int stages, float* out,
                         void* workspace, size_t workspace_bytes, hipStream_t stream) {
  const char* fn = "bmx_triattn_fp32_fwd";
  BMX_REQUIRE(n >= 0 && n <= 32768, "bmx_triattn_fp32_fwd: n must be in [0, 32768] (got %lld)", (long long)n);
  BMX_REQUIRE(row0 >= 0 && rows >= 0 && row0 + rows <= n, "bmx_triattn_fp32_fwd: rows must lie inside [0, n)");
  BMX_REQUIRE(stages >= 1 && stages <= 3 && (stages != 3 || rows == n),
              "bmx_triattn_fp32_fwd: stages must be 1 (triangle bias), 2 (attention) or, for all rows, 3");
  BMX_REQUIRE(eps > 0.f && inf > 0.f, "bmx_triattn_fp32_fwd: eps and inf must be positive");
  if (n == 0 || rows == 0) return BMX_OK;
  BMX_REQUIRE(x && ln_w && w_qkvg && b_qkvg && w_bias && tri_bias, "bmx_triattn_fp32_fwd: null pointer");
  BMX_REQUIRE(((uintptr_t)x | (uintptr_t)ln_w | (uintptr_t)ln_b | (uintptr_t)w_qkvg | (uintptr_t)b_qkvg |
               (uintptr_t)w_bias) % 16 == 0,
              "bmx_triattn_fp32_fwd: x and parameters must be 16-byte aligned");
  const Workspace ws = make_workspace(n, rows);
  if (stages & 2) {
    BMX_REQUIRE(out && workspace, "bmx_triattn_fp32_fwd: null pointer");
    BMX_REQUIRE((uintptr_t)out % 16 == 0 && (uintptr_t)workspace % 256 == 0 && workspace_bytes >= (size_t)ws.total,
                "bmx_triattn_fp32_fwd: out must be 16-byte aligned, workspace 256-byte and hold %lld bytes",
                (long long)ws.total);
  }
  char* base = (char*)workspace;
  ProjArgs a{};
  a.x = x, a.mask = mask, a.ln_w = ln_w, a.ln_b = ln_b;
  a.w = (const bf16*)w_qkvg, a.b = b_qkvg, a.w_bias = (const bf16*)w_bias;
  a.eps = eps, a.inf = inf;
  a.n = (int)n, a.nkp = (int)((n + kTP - 1) / kTP * kTP), a.i0 = (int)row0, a.rows = (int)rows;
  a.tri_bias = stages & 1 ? tri_bias : nullptr;
  if (stages & 2) {
    a.qg = (float*)(base + ws.qg);
    a.kh = (bf16*)(base + ws.kv[0]), a.kl = (bf16*)(base + ws.kv[1]);
    a.vth = (bf16*)(base + ws.kv[2]), a.vtl = (bf16*)(base + ws.kv[3]);
    a.mterm = (float*)(base + ws.mterm);
  }
  const int total = a.rows * (a.nkp / kTP);
  const int grid = total < device_cu_count() ? total : device_cu_count();
  if (starting)
    triattn_fp32_proj_kernel<true><<<grid, 64 * kWaves, 0, stream>>>(a);
  else
    triattn_fp32_proj_kernel<false><<<grid, 64 * kWaves, 0, stream>>>(a);
  if (int rc = check_launch(fn)) return rc;
  if (!(stages & 2)) return BMX_OK;
  return seq_attention_x3_presplit(fn, a.qg, a.qg + kC, 2 * kC, n * 2 * kC, rows, n, kH, kD, tri_bias, rows, a.kh, a.kl,
                                   a.vth, a.vtl, a.mterm, out, stream);
}

}  // extern "C"
