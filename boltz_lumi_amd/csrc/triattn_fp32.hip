// fp32-mode triangle attention for gfx950: LayerNorm, the q | k | v | g and triangle
// bias projections and the attention's operands in one pass over x, then the
// split-bf16 attention.  Upstream's fp32 forward is TriangleAttention with
// autocast off (reference triangle.py:38-52).
//
// What bounds the projection: HBM, and next the matrix cores.  The projection reads 512 B and writes 2.1 KB
// per pair (q and g fp32, K and V^T as bf16 high / low parts).  As separate passes (LayerNorm
// to a split operand, library GEMM to fp32 rows, a bias permute, the K / V split)
// the same step moved 7 KB per pair: 751 us at n = 576, this kernel 199 (4.3
// TB/s; 174 with three products).
// Products are split bf16, all four of them in the projections (xl wl + xh wh + xl wh + xh wl), three in the
// attention (about 2^-16 relative).  The fourth pays for the attention's offsets: whole numbers, so the largest
// probability of a row is no longer exactly 1 and has a split error too.  Against 64 bits, mean of n = 17 .. 576:
// 7.3e-6 with the separate passes, 7.7e-6 with three products here, 6.6e-6 with four (at every size below the
// separate passes; four for v and g alone are not).
#include "bmx_common.h"

using namespace bmx;

namespace {

constexpr int kH = 4, kD = 32;
constexpr int kTP = 64;            // pairs per tile
constexpr int kWaves = 16;         // wave w: head w % 4 of q, k, v or g (w / 4)
constexpr int kKRow = kD + 8;      // staged K row of one pair (bf16)
constexpr int kVRow = kTP + 8;     // staged V^T row of one head dim (bf16)
constexpr float kLog2e = 1.44269504088896340736f;
typedef unsigned u32x4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ f32x4 mfma16(bf16x8 a, bf16x8 b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}

// K and V^T of one (row, head): a record of four 2 KB tiles per 32-key block, K
// high, K low ([key][dim]), V^T high, V^T low ([dim][key slot]), each 32 rows of
// four 16-byte chunks, chunk c of row r at position c ^ chunk_swizzle(r): one LDS DMA
// copies 1 KB of it as it lies, and the attention's reads (lane l: row l % 16,
// chunk l / 16) meet no bank twice.
constexpr int kTile = 2048, kRecord = 4 * kTile;
__device__ __forceinline__ int tile_at(int row, int chunk) { return row * 64 + ((chunk ^ chunk_swizzle(row)) << 4); }

// Key slot inside a 32-key block: the attention's P operand order (slot 8 gi + e holds key 4 gi + e, or
// 16 + 4 gi + e - 4 from e = 4 on).
__device__ __forceinline__ int key_slot(int key) { return ((key & 15) >> 2) * 8 + (key >> 4) * 4 + (key & 3); }

struct ProjArgs {
  const float *x, *mask, *ln_w, *ln_b;
  const bf16* w;         // packed split weight [q; k; v; g], 512 x 128
  const float* b;        // [512 + 4]
  const bf16* w_bias;    // triangle bias rows, [high, low][16][128], rows 4..15 zero
  float eps, inf;
  int n, nkp, i0, rows;  // frame rows i0 .. i0 + rows - 1
  float* qg;             // [rows][n][q 128 | g 128]; null: triangle bias only
  char* kv;              // [rows][4][nkp / 32] records
  float* mterm;          // [rows][nkp]: (1 - mask) * -inf in log2 units, -infinity past n
  int* mflag;            // [rows][nkp / 64]: 1 if some term of the tile is not zero, 2 if all are
  float* tri_bias;       // [4][n][nkp], log2 units, zero past n; null: not written
};

// Persistent and weight-stationary: 16 waves keep 32 output rows each (8 k steps,
// high and low: 64 VGPRs), one block per CU, the next tile's rows prefetched into
// registers.  (8 waves of 64 rows spilled at 256 VGPRs, and a scratch reload
// waits for every prefetch and store before it: twice the time.)  q, k, g come as D[output][pair] (4 consecutive
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
#pragma unroll
      for (int u = 0; u < kH * kTP * kD / 8 / (64 * kWaves); ++u) {
        const int c = t + 64 * kWaves * u;
        char* rec = a.kv + ((int64_t)r * kH * nkp + j0) / 32 * kRecord + part * kTile;
        const int hk = c >> 8, p = (c >> 2) & (kTP - 1), ck = c & 3;
        *(bf16x8*)(rec + ((int64_t)hk * nkp + p) / 32 * kRecord + tile_at(p & 31, ck)) =
            *(const bf16x8*)(sk[part] + (hk * kTP + p) * kKRow + 8 * ck);
        const int d = (c >> 2) & 31, blk = hk * (nkp / 32) + ((c >> 7) & 1);
        *(bf16x8*)(rec + (int64_t)blk * kRecord + 2 * kTile + tile_at(d, ck)) =
            *(const bf16x8*)(sv[part] + (hk * kD + d) * kVRow + 32 * ((c >> 7) & 1) + 8 * ck);
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
    if (project && t < kTP) {  // wave 0
      float term = (1.f - mpre) * -a.inf * kLog2e;
      term = j0 + t >= n ? -INFINITY : term < -3e38f ? -3e38f : term;
      a.mterm[(int64_t)r * nkp + j0 + t] = term;
      const bool any = __any(!(term == 0.f)), all = __all(!(term == 0.f));
      if (t == 0) a.mflag[(int64_t)r * tiles_x + j0 / kTP] = any + all;
    }
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
            acc = mfma32(fl, wl[ks], acc);
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
            acc = mfma32(wl[ks], fl, acc);
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
        ab = mfma16(bl, fl, ab);
        ab = mfma16(bh, fh, ab);
        ab = mfma16(bh, fl, ab);
        ab = mfma16(bl, fh, ab);
      }
      const int j = j0 + 16 * w + lq;
      if (g == 0) {
#pragma unroll
        for (int e = 0; e < kH; ++e)
          a.tri_bias[((int64_t)e * n + i) * nkp + j] = j < n ? (ab[e] + sb[4 * kC + e]) * kLog2e : 0.f;
      }
    }
    __syncthreads();  // the stage is written; the x tiles have been read
    prev = tile;
  }
  if (project && prev >= 0) store_stage(prev);
}

// ------------------------------------------------------------------ attention
// A block serves 128 queries of one head (16 per wave) in kG = 2 frame rows,
// which share the triangle bias; it walks the keys in 32-key stages: LDS DMA
// copies the two rows' K / V^T records (16 KB), the bias in operand order (16 KB:
// each lane reads back the 16 bytes that it copied, so the copy is an
// asynchronous register load) and the mask terms into one of two buffers (65
// KB; two blocks of 8 waves share a CU at <= 128 VGPRs).  v_mfma_f32_16x16x32_bf16
// (lane l, gi = l / 16, c = l % 16: A holds A[c][8 gi .. + 7], B holds B[8 gi .. + 7][c], D
// register r holds D[4 gi + r][c]); per stage, row and wave:
//   S^T[key][q] = bias + mask + K Q^T   2 key tiles, 3 products each, the bias as C
//   O^T[d][q] += V^T P^T                2 dim tiles, 3 products each.
// Scores are in log2 units (q times log2(e) / sqrt(32) in fp32 before its split).
//
// What bounds it: VALU issue (the exponential, the split of P), next the matrix
// cores and LDS reads.  The general split-bf16 attention kernel (pair_bias.hip),
// with the bias and the mask terms loaded per row and stage, four more VALU
// operations a score and a running max, took 890 us at n = 576, this one 473
// (0.6 PF/s over the three products).
constexpr int kG = 2, kCoreWaves = 8, kCoreQ = 16 * kCoreWaves, kCoreThreads = 64 * kCoreWaves;
constexpr int kOffBias = kG * kRecord, kOffTerm = kOffBias + kCoreWaves * 2048, kStageBytes = kOffTerm + kG * 32 * 4;

struct CoreArgs {
  const float* qg;    // [rows][n][q 128 | g 128]
  const char* kv;     // records
  const float* mterm;
  const int* mflag;
  const float* bias;  // [4][n][nkp]
  float* out;         // [rows][n][128]
  int n, nkp, rows;
};

// LDS DMA of 64 lanes x 16 (4) bytes to lds_addr + 16 (4) * lane.  It reads M0, and one wait state must
// lie between M0's write and the read (s_nop 0): the compiler does not see into the asm.
__device__ __forceinline__ void lds_dma16(const void* src, unsigned lds_addr) {
  asm volatile("s_nop 0\n\tglobal_load_lds_dwordx4 %0, off" ::"v"(src), "{m0}"(lds_addr) : "memory");
}
__device__ __forceinline__ void lds_dma4(const void* src, unsigned lds_addr) {
  asm volatile("s_nop 0\n\tglobal_load_lds_dword %0, off" ::"v"(src), "{m0}"(lds_addr) : "memory");
}
__device__ __forceinline__ void wait_vm0() { __builtin_amdgcn_s_waitcnt(0x0F70); }  // vmcnt(0)

// Four probabilities as bf16 high and low parts, two to a register.
__device__ __forceinline__ void split4(const float* p, unsigned* hi, unsigned* lo) {
#pragma unroll
  for (int e = 0; e < 2; ++e) {
    const f32x2 v = {p[2 * e], p[2 * e + 1]};
    const unsigned h = __builtin_bit_cast(unsigned, __builtin_convertvector(v, bf16x2));
    const f32x2 r = {v[0] - __uint_as_float(h << 16), v[1] - __uint_as_float(h & 0xffff0000u)};
    hi[e] = h;
    lo[e] = __builtin_bit_cast(unsigned, __builtin_convertvector(r, bf16x2));
  }
}

__device__ __forceinline__ float query_max(float v) {  // over the four lanes of a query
  v = fmaxf(v, __shfl_xor(v, 16, kWave));
  return fmaxf(v, __shfl_xor(v, 32, kWave));
}

// SPEC: one offset for both rows and all keys, the first stage's maximum, so that
// it costs one subtraction per bias value and no maximum afterwards; false
// (nothing written) if a row sum leaves [2^-60, 2^101) or an output is not finite,
// i.e. if a later score lies far above, or a row far below, or the first keys are
// closed.  Else the running maximum of each row.  Offsets are whole numbers: a power of two changes no rounding of P's parts.
template <bool SPEC>
__device__ __forceinline__ bool core_rows(const CoreArgs& a, int i0, int h, int q0, int mask_k0, char* lds) {
  const int l = lane_id(), gi = l >> 4, c = l & 15, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int n = a.n, nkp = a.nkp, nk = (n + 31) / 32 * 32;
  const int qc = min(q0 + c, n - 1);   // queries past the end re-read the last one and are not stored
  const bool active = q0 < n;          // wave-uniform
  const unsigned lds0 = (unsigned)(uintptr_t)(__attribute__((address_space(3))) void*)lds;

  bf16x8 qh[kG], ql[kG];
  const char* kv_src[kG];
#pragma unroll
  for (int r = 0; r < kG; ++r) {
    const int64_t i = min(i0 + r, a.rows - 1);  // a row past the end repeats the last one
    const float* q = a.qg + (i * n + qc) * 2 * kC + h * kD + 8 * gi;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const float v = q[e] * (0.17677669529663687f * kLog2e);
      qh[r][e] = (bf16)v;
      ql[r][e] = (bf16)(v - (float)qh[r][e]);
    }
    kv_src[r] = a.kv + (i * kH + h) * (nkp / 32) * kRecord + w * 1024 + 16 * l;
  }
  const float* b_src = a.bias + ((int64_t)h * n + qc) * nkp + 4 * gi;
  const float* t_src = a.mterm + (int64_t)min(i0 + (l >> 5), a.rows - 1) * nkp + (l & 31);
  auto dma_stage = [&](int buf, int k0) {
    const unsigned dst = lds0 + buf * kStageBytes;
#pragma unroll
    for (int r = 0; r < kG; ++r)
      lds_dma16(kv_src[r] + k0 / 32 * kRecord, __builtin_amdgcn_readfirstlane(dst + r * kRecord + w * 1024));
#pragma unroll
    for (int t = 0; t < 2; ++t)
      lds_dma16(b_src + k0 + 16 * t, __builtin_amdgcn_readfirstlane(dst + kOffBias + w * 2048 + t * 1024));
    if (w == 0) lds_dma4(t_src + k0, __builtin_amdgcn_readfirstlane(dst + kOffTerm));
  };

  f32x4 o[kG][2];
  float m[kG], ls[kG];
#pragma unroll
  for (int r = 0; r < kG; ++r) {
    o[r][0] = o[r][1] = f32x4{0.f, 0.f, 0.f, 0.f};
    m[r] = SPEC ? 0.f : -3.4e38f;
    ls[r] = 0.f;
  }
  const int rd = tile_at(c, gi);
  bool ok = true;
  wait_vm0();  // q: a later wait for it would wait for the DMA in flight too
  dma_stage(0, 0);
  wait_vm0();
  __syncthreads();
  for (int k0 = 0; k0 < nk; k0 += 32) {
    const int cur = (k0 >> 5) & 1;
    if (k0 + 32 < nk) dma_stage(cur ^ 1, k0 + 32);
    if (active) {
      const char* sb = lds + cur * kStageBytes;
      f32x4 b4[2], s[kG][2];
#pragma unroll
      for (int t = 0; t < 2; ++t) {
        b4[t] = *(const f32x4*)(sb + kOffBias + w * 2048 + t * 1024 + 16 * l);
        if (SPEC) b4[t] = b4[t] - m[0];
      }
#pragma unroll
      for (int r = 0; r < kG; ++r)
#pragma unroll
        for (int t = 0; t < 2; ++t) s[r][t] = b4[t];
#pragma unroll
      for (int r = 0; r < kG; ++r)
#pragma unroll
        for (int t = 0; t < 2; ++t) {
          const bf16x8 kh = *(const bf16x8*)(sb + r * kRecord + 1024 * t + rd);
          const bf16x8 kl = *(const bf16x8*)(sb + r * kRecord + kTile + 1024 * t + rd);
          s[r][t] = mfma16(kh, qh[r], s[r][t]);
          s[r][t] = mfma16(kh, ql[r], s[r][t]);
          s[r][t] = mfma16(kl, qh[r], s[r][t]);
        }
      // After the products: -1e9 as their C would be rounded inside the MFMA, to other values for
      // other products, where every key of a closed row must come out alike.
      if (k0 >= mask_k0) {  // wave-uniform
#pragma unroll
        for (int r = 0; r < kG; ++r)
#pragma unroll
          for (int t = 0; t < 2; ++t) s[r][t] += *(const f32x4*)(sb + kOffTerm + (r * 32 + 16 * t + 4 * gi) * 4);
      }
      auto row_max = [&](int r) {
        const f32x4 v = s[r][0], u = s[r][1];
        return fmaxf(fmaxf(fmaxf(v[0], v[1]), fmaxf(v[2], v[3])), fmaxf(fmaxf(u[0], u[1]), fmaxf(u[2], u[3])));
      };
      if (SPEC) {
        if (k0 == 0) {
          m[0] = ceilf(query_max(fmaxf(row_max(0), row_max(1))));
          ok = m[0] > -1e6f;  // as C of the products it must keep their digits
#pragma unroll
          for (int r = 0; r < kG; ++r)
#pragma unroll
            for (int t = 0; t < 2; ++t) s[r][t] = s[r][t] - m[0];
        }
      } else {
#pragma unroll
        for (int r = 0; r < kG; ++r) {
          const float mn = fmaxf(m[r], ceilf(query_max(row_max(r))));
          const float alpha = __builtin_amdgcn_exp2f(m[r] - mn);
          m[r] = mn;
          ls[r] *= alpha;
          o[r][0] *= alpha;
          o[r][1] *= alpha;
#pragma unroll
          for (int t = 0; t < 2; ++t) s[r][t] = s[r][t] - mn;
        }
      }
#pragma unroll
      for (int r = 0; r < kG; ++r) {
        u32x4 ph, pl;
        float p[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) p[e] = __builtin_amdgcn_exp2f(s[r][e >> 2][e & 3]);
        ls[r] += ((p[0] + p[1]) + (p[2] + p[3])) + ((p[4] + p[5]) + (p[6] + p[7]));
        unsigned hi[4], lo[4];
        split4(p, hi, lo);
        split4(p + 4, hi + 2, lo + 2);
#pragma unroll
        for (int e = 0; e < 4; ++e) ph[e] = hi[e], pl[e] = lo[e];
        const bf16x8 bh = __builtin_bit_cast(bf16x8, ph), bl = __builtin_bit_cast(bf16x8, pl);
#pragma unroll
        for (int dt = 0; dt < 2; ++dt) {
          const bf16x8 vh = *(const bf16x8*)(sb + r * kRecord + 2 * kTile + 1024 * dt + rd);
          const bf16x8 vl = *(const bf16x8*)(sb + r * kRecord + 3 * kTile + 1024 * dt + rd);
          o[r][dt] = mfma16(vh, bh, o[r][dt]);
          o[r][dt] = mfma16(vh, bl, o[r][dt]);
          o[r][dt] = mfma16(vl, bh, o[r][dt]);
        }
      }
    }
    wait_vm0();  // this wave's DMAs of the next stage
    __syncthreads();
  }
#pragma unroll
  for (int r = 0; r < kG; ++r) {
    ls[r] += __shfl_xor(ls[r], 16, kWave);
    ls[r] += __shfl_xor(ls[r], 32, kWave);
  }
  if (SPEC) {
#pragma unroll
    for (int r = 0; r < kG; ++r) {
      const unsigned ex = (__float_as_uint(ls[r]) >> 23) & 0xff;
      ok &= ex >= 127 - 60 && ex <= 127 + 100;
#pragma unroll
      for (int e = 0; e < 8; ++e) ok &= (__float_as_uint(o[r][e >> 2][e & 3]) & 0x7f800000u) != 0x7f800000u;
    }
    if (__syncthreads_or(active && !ok)) return false;
  }
  const int j = q0 + c;
#pragma unroll
  for (int r = 0; r < kG; ++r) {
    if (i0 + r < a.rows && j < n) {
      const int64_t row = (int64_t)(i0 + r) * n + j;
      const float inv = 1.f / ls[r];
#pragma unroll
      for (int dt = 0; dt < 2; ++dt) {
        const int d = h * kD + 16 * dt + 4 * gi;
        const f32x4 gv = load4(a.qg + row * 2 * kC + kC + d);
        f32x4 y;
#pragma unroll
        for (int e = 0; e < 4; ++e) y[e] = sigmoid_f(gv[e]) * (o[r][dt][e] * inv);
        store4(a.out + row * kC + d, y);
      }
    }
  }
  return true;
}

// Block L runs on XCD L % 8; each XCD takes a contiguous run of the items in the
// order (head, group of 8 query tiles, row pair, query tile), so that the blocks in
// flight on it (64) share both their rows' K / V^T and their queries' bias in its L2.
__global__ __launch_bounds__(kCoreThreads) __attribute__((amdgpu_waves_per_eu(4))) void triattn_fp32_core_kernel(
    CoreArgs a) {
  __shared__ __attribute__((aligned(16))) char lds[2 * kStageBytes];
  const int qtiles = (a.n + kCoreQ - 1) / kCoreQ, pairs = (a.rows + kG - 1) / kG, per_head = pairs * qtiles;
  const int item = (blockIdx.x & 7) * (gridDim.x >> 3) + (blockIdx.x >> 3);
  if (item >= kH * per_head) return;  // the padding of the last XCD's run (whole block)
  const int h = item / per_head, in_head = item % per_head, group = in_head / (8 * pairs);
  const int width = min(8, qtiles - 8 * group), in_group = in_head - 8 * pairs * group;
  const int i0 = in_group / width * kG, q0 = (8 * group + in_group % width) * kCoreQ + 16 * (threadIdx.x >> 6);

  // The first 64-key tile with a mask term in either row (every wave reads the same flags), and whether
  // one of them starts with a tile of closed keys: its first maximum says nothing of the others.
  const int tiles = a.nkp / kTP;
  int first = tiles;
  bool closed = false;
#pragma unroll
  for (int r = 0; r < kG; ++r) {
    const int* f = a.mflag + (int64_t)min(i0 + r, a.rows - 1) * tiles;
    closed |= f[0] == 2;
    for (int e = lane_id(); e < tiles; e += kWave)
      if (f[e]) first = min(first, e);
  }
#pragma unroll
  for (int d = 32; d >= 1; d >>= 1) first = min(first, __shfl_xor(first, d, kWave));
  const int mask_k0 = __builtin_amdgcn_readfirstlane(first) * kTP;
  const int qw = __builtin_amdgcn_readfirstlane(q0);
  if (closed || !core_rows<true>(a, i0, h, qw, mask_k0, lds)) core_rows<false>(a, i0, h, qw, mask_k0, lds);
}

// ------------------------------------------------------------------ output linear
// out = o W^T + b over rows of 128, fp32 MFMA (32x32x2).  Weight-stationary: wave w
// keeps outputs 32 (w % 4) .. + 31 (64 VGPRs) and takes rows 32 (w / 4) .. + 31 of a
// 64-row tile; the next tile comes by LDS DMA, 16-byte chunk c of row r at position
// c ^ (r % 32).  Lane l holds chunk 2 j + l / 32 of its row for k step j, so MFMA e of a step
// multiplies k = 8 j + e and 8 j + 4 + e; D[output][row] leaves as 16-byte stores.
// What bounds it: the fp32 matrix cores (75 us of them at n = 576; 129 us).  The library GEMM took
// 162-179 us.  out may be o: a block has read a tile when it writes it, and nobody else reads it.
constexpr int kLinRows = 64, kLinWaves = 8, kLinTile = kLinRows * kC * 4;

__global__ __launch_bounds__(64 * kLinWaves) __attribute__((amdgpu_waves_per_eu(4))) void linear128_f32_kernel(
    const float* o, int64_t rows, const float* __restrict__ w_o, const float* __restrict__ b_o, float* out) {
  __shared__ __attribute__((aligned(16))) char lds[2 * kLinTile];
  __shared__ __attribute__((aligned(16))) float sbias[kC];
  const int l = lane_id(), hh = l >> 5, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int c0 = 32 * (w & 3), r0 = 32 * (w >> 2), row = r0 + (l & 31);
  const unsigned lds0 = (unsigned)(uintptr_t)(__attribute__((address_space(3))) void*)lds;
  f32x4 wf[16];
#pragma unroll
  for (int j = 0; j < 16; ++j) wf[j] = load4(w_o + (c0 + (l & 31)) * kC + 8 * j + 4 * hh);
  if (threadIdx.x < kC) sbias[threadIdx.x] = b_o[threadIdx.x];
  auto dma_tile = [&](int buf, int64_t tile) {
#pragma unroll
    for (int u = 0; u < kLinTile / 1024 / kLinWaves; ++u) {
      const int piece = w + kLinWaves * u, r = 2 * piece + hh;  // 1 KB: two rows
      const int64_t at = tile * kLinRows + r < rows ? tile * kLinRows + r : rows - 1;  // not stored past the end
      lds_dma16(o + at * kC + 4 * ((l & 31) ^ (r & 31)),
                __builtin_amdgcn_readfirstlane(lds0 + buf * kLinTile + 1024 * piece));
    }
  };
  const int64_t tiles = (rows + kLinRows - 1) / kLinRows;
  int64_t tile = blockIdx.x;
  int cur = 0;
  wait_vm0();
  dma_tile(0, tile);  // the grid is at most tiles
  wait_vm0();
  __syncthreads();
  for (; tile < tiles; tile += gridDim.x, cur ^= 1) {
    if (tile + gridDim.x < tiles) dma_tile(cur ^ 1, tile + gridDim.x);
    const char* sb = lds + cur * kLinTile + row * kC * 4;
    int first = (hh ^ (row & 31)) << 4;
    asm volatile("" : "+v"(first));  // the reads' 16 addresses again per tile: kept, they spill weights
    f32x16 acc;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const f32x4 b4 = *(const f32x4*)(sbias + c0 + 8 * q + 4 * hh);
#pragma unroll
      for (int e = 0; e < 4; ++e) acc[4 * q + e] = b4[e];
    }
#pragma unroll
    for (int j = 0; j < 16; ++j) {
      const f32x4 x = *(const f32x4*)(sb + (first ^ (32 * j)));
#pragma unroll
      for (int e = 0; e < 4; ++e) acc = __builtin_amdgcn_mfma_f32_32x32x2f32(wf[j][e], x[e], acc, 0, 0, 0);
    }
    const int64_t at = tile * kLinRows + row;
    if (at < rows) {
#pragma unroll
      for (int q = 0; q < 4; ++q)
        store4(out + at * kC + c0 + 8 * q + 4 * hh, f32x4{acc[4 * q], acc[4 * q + 1], acc[4 * q + 2], acc[4 * q + 3]});
    }
    wait_vm0();
    __syncthreads();
  }
}

struct Workspace {
  int64_t qg, kv, mterm, mflag, total;
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
  w.kv = take(rows * kH * (nkp / 32) * kRecord);
  w.mterm = take(rows * nkp * 4);
  w.mflag = take(rows * (nkp / kTP) * 4);
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
               (uintptr_t)w_bias | (uintptr_t)tri_bias) % 16 == 0,
              "bmx_triattn_fp32_fwd: x, tri_bias and parameters must be 16-byte aligned");
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
    a.kv = base + ws.kv;
    a.mterm = (float*)(base + ws.mterm);
    a.mflag = (int*)(base + ws.mflag);
  }
  const int total = a.rows * (a.nkp / kTP);
  const int grid = total < device_cu_count() ? total : device_cu_count();
  if (starting)
    triattn_fp32_proj_kernel<true><<<grid, 64 * kWaves, 0, stream>>>(a);
  else
    triattn_fp32_proj_kernel<false><<<grid, 64 * kWaves, 0, stream>>>(a);
  if (int rc = check_launch(fn)) return rc;
  if (!(stages & 2)) return BMX_OK;
  const CoreArgs c{a.qg, a.kv, a.mterm, a.mflag, tri_bias, out, a.n, a.nkp, a.rows};
  const int64_t items = (int64_t)kH * ((a.rows + kG - 1) / kG) * ((a.n + kCoreQ - 1) / kCoreQ);
  triattn_fp32_core_kernel<<<(unsigned)((items + 7) / 8 * 8), kCoreThreads, 0, stream>>>(c);
  return check_launch(fn);
}

int bmx_linear128_f32_fwd(const float* x, int64_t rows, const float* w, const float* b, float* out,
                          hipStream_t stream) {
  BMX_REQUIRE(rows >= 0, "bmx_linear128_f32_fwd: rows must be >= 0 (got %lld)", (long long)rows);
  if (rows == 0) return BMX_OK;
  BMX_REQUIRE(x && w && b && out, "bmx_linear128_f32_fwd: null pointer");
  BMX_REQUIRE(((uintptr_t)x | (uintptr_t)w | (uintptr_t)b | (uintptr_t)out) % 16 == 0,
              "bmx_linear128_f32_fwd: pointers must be 16-byte aligned");
  const int64_t tiles = (rows + kLinRows - 1) / kLinRows, most = 2 * device_cu_count();
  linear128_f32_kernel<<<(unsigned)(tiles < most ? tiles : most), 64 * kLinWaves, 0, stream>>>(x, rows, w, b, out);
  return check_launch("bmx_linear128_f32_fwd");
}

}  // extern "C"
