// The Pairformer sequence stack (fp32, autocast off): pre_norm_s, AttentionPairBias
// and the 384 -> 1536 -> 384 transition, each with its residual add, as five
// launches on fp32 MFMA linears:
//   LayerNorm + q | k | v | g,  attention,  proj_o + s,  LayerNorm + fc1 | fc2 + SwiGLU,  fc3 + s.
//
// What bounds it: at a trunk's token counts (tens to some thousands of rows) each
// linear is a few microseconds of matrix work behind launches and load latency.
// Through torch the stack was ten launches (two LayerNorms, four GEMMs, a copy
// for the out-of-place residual, silu, mul, attention).  Here a 32 x 32 or 32 x
// 64 tile is a block, its waves split K (v_mfma_f32_32x32x2f32, fp32 products and
// sums), and every operand a wave streams lies packed in MFMA order
// (f32_packed_index): read as rows, a fragment load touches 32 cache lines and
// the texture pipe, not the matrix cores, sets the time (fc1 | fc2 at 1134 rows 69
// us against 54, at 117 17.5 against 13.5).  The rows a LayerNorm stands in
// front of are normalised by each block into LDS in that order; activations
// and residuals are the epilogue.  The whole stack, before (torch, bound by the
// host up to some 1200 rows) and after: 117 tokens 199 -> 49 us, 312 198 -> 64,
// 1024 197 -> 141, 1280 195 -> 181; its kernels alone 64 -> 48 us at 117 tokens,
// 223 -> 210 at 1134.  From about 1536 rows on the library's larger tiles win
// (pairformer.py draws the line).
#include "bmx_common.h"

using namespace bmx;

namespace {

constexpr int kMaxLn = 512;  // widest row normalised in LDS

struct LinearF32 {
  const float* x;  // LN: [m][k] rows, else the packed operand
  const float *ln_w, *ln_b;
  float eps;
  const float* w;     // packed weight rows (swiglu: tiles of fc1 and of fc2 in turn)
  const float* bias;  // first n_bias outputs (null: none)
  const float* res;   // residual rows at ldo (null: none), may alias out
  float* out;         // rows at ldo; swiglu: packed operand of m x n
  int64_t ldo;
  int m, n, k, n_bias;
  int tiles_m, tiles_n;
};

__device__ __forceinline__ f32x16 mfma32f(float a, float b, f32x16 c) {
  return __builtin_amdgcn_mfma_f32_32x32x2f32(a, b, c, 0, 0, 0);
}

// TJ output tiles of 32 columns per block, W waves splitting K in steps of 8.
// SWIGLU (TJ = 2): the two tiles are the same 32 columns of fc1 and of fc2 and
// the result is silu(first) * second.
template <int TJ, int W, bool LN, bool SWIGLU>
__global__ __launch_bounds__(64 * W) void linear_f32_kernel(LinearF32 a) {
  constexpr int TN = 32 * TJ, kRow = TN + 4, kBatch = 6;
  static_assert(!SWIGLU || TJ == 2, "one tile of each half");
  constexpr int kRed = W * 32 * kRow, kX = LN ? 32 * kMaxLn : 0;
  __shared__ __attribute__((aligned(16))) float smem[kRed > kX ? kRed : kX];
  const int t = threadIdx.x, l = lane_id(), wv = __builtin_amdgcn_readfirstlane(t >> 6);
  // Blocks go round-robin over the 8 XCDs; each XCD takes a contiguous run of
  // tiles, x row tiles first, so its L2 holds few weight tiles at a time.
  const int tiles = a.tiles_m * a.tiles_n, per_xcd = (tiles + 7) / 8;
  const int tile = (blockIdx.x & 7) * per_xcd + (blockIdx.x >> 3);
  if (tile >= tiles) return;  // whole block
  const int tm = tile % a.tiles_m, tn = tile / a.tiles_m;
  const int steps = a.k / 8, s0 = steps * wv / W, s1 = steps * (wv + 1) / W, nt = a.n / 32 * (SWIGLU ? 2 : 1);
  const int64_t tstride = (int64_t)steps * 256;  // one packed 32-row tile
  const float* pw[TJ];
#pragma unroll
  for (int j = 0; j < TJ; ++j) pw[j] = a.w + min(TJ * tn + j, nt - 1) * tstride + 4 * l;  // past the end: not stored
  const float* px = LN ? nullptr : a.x + tm * tstride + 4 * l;

  f32x4 x[kBatch], w[kBatch][TJ];
  auto load = [&](int st) {
#pragma unroll
    for (int u = 0; u < kBatch; ++u) {
      const int o = 256 * min(st + u, s1 - 1);  // past the end: the last step again, unused
#pragma unroll
      for (int j = 0; j < TJ; ++j) w[u][j] = load4(pw[j] + o);
      if constexpr (!LN) x[u] = load4(px + o);
    }
  };
  load(s0);
  if constexpr (LN) {
    // Rows to LDS in packed order, normalised: 2 W threads per row, each its
    // float4 chunks p, p + 2 W, ...  The lane slot is XORed with the step so that
    // a row's chunks, one step apart, do not meet in the same banks.
    constexpr int kPer = 2 * W, kChunks = kMaxLn / 4 / kPer;
    const int r = t / kPer, p = t % kPer, chunks = a.k / 4;
    const float* xr = a.x + (int64_t)min(tm * 32 + r, a.m - 1) * a.k;
    f32x4 v[kChunks];
    float s = 0.f;
#pragma unroll
    for (int u = 0; u < kChunks; ++u) {
      const int c = p + kPer * u;
      v[u] = load4(xr + 4 * min(c, chunks - 1));
      if (c < chunks) s += (v[u][0] + v[u][1]) + (v[u][2] + v[u][3]);
    }
#pragma unroll
    for (int d = kPer / 2; d >= 1; d >>= 1) s += __shfl_xor(s, d, kWave);
    const float mu = s / a.k;
    float q = 0.f;
#pragma unroll
    for (int u = 0; u < kChunks; ++u) {
      v[u] -= mu;
      if (p + kPer * u < chunks) q += (v[u][0] * v[u][0] + v[u][1] * v[u][1]) + (v[u][2] * v[u][2] + v[u][3] * v[u][3]);
    }
#pragma unroll
    for (int d = kPer / 2; d >= 1; d >>= 1) q += __shfl_xor(q, d, kWave);
    const float inv = rsqrtf(q / a.k + a.eps);
#pragma unroll
    for (int u = 0; u < kChunks; ++u) {
      const int c = p + kPer * u;
      if (c < chunks)
        *(f32x4*)(smem + ((c >> 1) * 64 + (r ^ ((c >> 1) & 31)) + 32 * (c & 1)) * 4) =
            v[u] * inv * load4(a.ln_w + 4 * c) + load4(a.ln_b + 4 * c);
    }
    __syncthreads();
  }
  f32x16 acc[TJ];
#pragma unroll
  for (int j = 0; j < TJ; ++j) acc[j] = zero16();
  for (int st = s0; st < s1; st += kBatch) {
    if (st != s0) load(st);
    if constexpr (LN) {
#pragma unroll
      for (int u = 0; u < kBatch; ++u) {
        const int o = min(st + u, s1 - 1);
        x[u] = *(const f32x4*)(smem + (o * 64 + (l ^ (o & 31))) * 4);
      }
    }
#pragma unroll
    for (int u = 0; u < kBatch; ++u) {
      if (st + u < s1) {  // wave-uniform
#pragma unroll
        for (int e = 0; e < 4; ++e)
#pragma unroll
          for (int j = 0; j < TJ; ++j) acc[j] = mfma32f(w[u][j][e], x[u][e], acc[j]);
      }
    }
  }
  if constexpr (LN) __syncthreads();  // the rows have been read
  float(*red)[32 * kRow] = (float(*)[32 * kRow])smem;
  // D[n][m]: lane -> row l % 32, registers 4q .. 4q+3 -> n = 32 j + 8 q + 4 (l / 32) + 0..3
#pragma unroll
  for (int j = 0; j < TJ; ++j)
#pragma unroll
    for (int q = 0; q < 4; ++q)
      *(f32x4*)(&red[wv][(l & 31) * kRow + 32 * j + 8 * q + 4 * (l >> 5)]) =
          f32x4{acc[j][4 * q], acc[j][4 * q + 1], acc[j][4 * q + 2], acc[j][4 * q + 3]};
  __syncthreads();
  auto sum = [&](int r, int c) {
    f32x4 v = *(const f32x4*)(&red[0][r * kRow + c]);
#pragma unroll
    for (int p = 1; p < W; ++p) v += *(const f32x4*)(&red[p][r * kRow + c]);
    return v;
  };
  constexpr int kCols = SWIGLU ? 32 : TN;
  for (int e = t; e < 32 * kCols / 4; e += 64 * W) {
    const int r = e / (kCols / 4), c = 4 * (e % (kCols / 4)), m = tm * 32 + r, n = tn * kCols + c;
    if (m >= a.m || n >= a.n) continue;
    f32x4 v = sum(r, c);
    if constexpr (SWIGLU) {
      const f32x4 g = sum(r, 32 + c);
#pragma unroll
      for (int i = 0; i < 4; ++i) v[i] = v[i] / (1.f + expf(-v[i])) * g[i];  // __expf: an error of |v| ulp
    }
    if (a.bias && n < a.n_bias) v += load4(a.bias + n);
    if (a.res) v += load4(a.res + (int64_t)m * a.ldo + n);
    store4(SWIGLU ? a.out + f32_packed_index(m, n, a.n >> 3) : a.out + (int64_t)m * a.ldo + n, v);
  }
}

template <bool LN, bool SWIGLU>
int launch_linear(const char* name, LinearF32 a, hipStream_t stream) {
  a.tiles_m = (a.m + 31) / 32;
  const int nt = a.n / 32;
  const int64_t tiles = (int64_t)a.tiles_m * nt;
  // Two column tiles per block (one read of x for both) once that leaves more
  // than a block per CU: q | k | v | g at 600 rows 20.3 us against 24.9, at 1134
  // 32.0 against 37.5; at 312 rows (480 tiles) one tile each, 13.2 us.
  const bool wide = SWIGLU || tiles > 700;
  a.tiles_n = !SWIGLU && wide ? (nt + 1) / 2 : nt;
  const dim3 grid((unsigned)(8 * (((int64_t)a.tiles_m * a.tiles_n + 7) / 8)));
  if (SWIGLU || wide) {
    linear_f32_kernel<2, 4, LN, SWIGLU><<<grid, 256, 0, stream>>>(a);
    return check_launch(name);
  }
  if constexpr (!LN) {  // normalised rows are at most kMaxLn wide
    if (a.k >= 1024) {
      linear_f32_kernel<1, 8, LN, false><<<grid, 512, 0, stream>>>(a);
      return check_launch(name);
    }
  }
  linear_f32_kernel<1, 4, LN, false><<<grid, 256, 0, stream>>>(a);
  return check_launch(name);
}

// fp32 weight rows to packed operand tiles: 32-row tile t of w goes to packed
// tile tile0 + t * tile_stride.  One wave per (32-row tile, 8-column step).
__global__ __launch_bounds__(64) void f32_pack_kernel(const float* __restrict__ w, int64_t ldw, int steps,
                                                      int64_t tile0, int64_t tile_stride, float* __restrict__ out) {
  const int l = threadIdx.x;
  const f32x4 v = load4(w + ((int64_t)blockIdx.y * 32 + (l & 31)) * ldw + 8 * blockIdx.x + 4 * (l >> 5));
  store4(out + ((tile0 + blockIdx.y * tile_stride) * steps + blockIdx.x) * 256 + 4 * l, v);
}

}  // namespace

extern "C" {

int bmx_f32_pack(const float* w, int64_t rows, int64_t k, int64_t ldw, int64_t tile0, int64_t tile_stride, float* out,
                 hipStream_t stream) {
  BMX_REQUIRE(rows >= 0 && rows % 32 == 0 && k > 0 && k % 8 == 0 && ldw >= k && ldw % 4 == 0,
              "bmx_f32_pack: rows must be a multiple of 32, k a positive multiple of 8, ldw >= k a multiple of 4");
  BMX_REQUIRE(rows / 32 <= 65535 && k / 8 <= (1 << 30) && tile0 >= 0 && tile_stride >= 1,
              "bmx_f32_pack: at most 65535 tiles of 32 rows, tile0 >= 0, tile_stride >= 1");
  if (rows == 0) return BMX_OK;
  BMX_REQUIRE(w && out, "bmx_f32_pack: null pointer");
  BMX_REQUIRE((uintptr_t)w % 16 == 0 && (uintptr_t)out % 16 == 0, "bmx_f32_pack: w and out must be 16-byte aligned");
  f32_pack_kernel<<<dim3((unsigned)(k / 8), (unsigned)(rows / 32)), 64, 0, stream>>>(w, ldw, (int)(k / 8), tile0,
                                                                                   tile_stride, out);
  return check_launch("bmx_f32_pack");
}

size_t bmx_sequence_stack_workspace_bytes(int64_t rows, int64_t d, int64_t hidden) {
  if (rows <= 0 || d <= 0 || hidden <= 0) return 0;
  const int64_t rp = (rows + 31) / 32 * 32;  // packed operands hold whole 32-row tiles
  return (size_t)(rows * 4 * d + rp * (d + hidden)) * sizeof(float);
}

int bmx_sequence_stack_fwd(const float* s, int64_t batch, int64_t n, int heads, int head_dim, int64_t hidden,
                           const void* const* params, float eps_attn, float eps_trans, const float* bias,
                           const float* mask, int64_t smask, float inf, float* out, void* workspace,
                           size_t workspace_bytes, hipStream_t stream) {
  const char* fn = "bmx_sequence_stack_fwd";
  const int64_t d = (int64_t)heads * head_dim, m = batch * n;
  BMX_REQUIRE(batch >= 0 && batch <= 65535 && n >= 0 && n <= (1 << 20) && m <= (1 << 20),
              "bmx_sequence_stack_fwd: need 0 <= batch <= 65535, 0 <= batch * n <= 2^20");
  BMX_REQUIRE(head_dim == 24 || head_dim == 32 || head_dim == 48,
              "bmx_sequence_stack_fwd: head_dim must be 24, 32 or 48 (got %d)", head_dim);
  BMX_REQUIRE(heads >= 1 && heads <= 64 && d % 32 == 0 && d <= kMaxLn && hidden > 0 && hidden % 32 == 0 &&
                  hidden <= (1 << 16),
              "bmx_sequence_stack_fwd: heads * head_dim (at most %d) and hidden must be multiples of 32", kMaxLn);
  BMX_REQUIRE(eps_attn > 0.f && eps_trans > 0.f && inf > 0.f && smask >= 0,
              "bmx_sequence_stack_fwd: eps and inf must be positive, smask >= 0");
  if (m == 0) return BMX_OK;
  BMX_REQUIRE(s && params && bias && mask && out && workspace, "bmx_sequence_stack_fwd: null pointer");
  for (int i = 0; i < 9; ++i) {
    BMX_REQUIRE(params[i] || i == 3, "bmx_sequence_stack_fwd: null parameter %d", i);  // proj_q's bias may be null
    BMX_REQUIRE((uintptr_t)params[i] % 16 == 0, "bmx_sequence_stack_fwd: parameter %d must be 16-byte aligned", i);
  }
  BMX_REQUIRE(((uintptr_t)s | (uintptr_t)out | (uintptr_t)workspace) % 16 == 0,
              "bmx_sequence_stack_fwd: s, out and workspace must be 16-byte aligned");
  BMX_REQUIRE(workspace_bytes >= bmx_sequence_stack_workspace_bytes(m, d, hidden),
              "bmx_sequence_stack_fwd: workspace too small (%zu < %zu bytes)", workspace_bytes,
              bmx_sequence_stack_workspace_bytes(m, d, hidden));
  const float* const* p = (const float* const*)params;
  const int64_t mp = (m + 31) / 32 * 32;
  float *proj = (float*)workspace, *o = proj + 4 * m * d, *hid = o + mp * d;
  LinearF32 a{};
  a.m = (int)m;
  a.x = s, a.k = (int)d;
  a.ln_w = p[0], a.ln_b = p[1], a.eps = eps_attn;
  a.w = p[2], a.n = (int)(4 * d), a.bias = p[3], a.n_bias = (int)d;
  a.out = proj, a.ldo = 4 * d;
  if (int rc = launch_linear<true, false>(fn, a, stream)) return rc;
  if (int rc = sequence_attention_packed(proj, batch, n, heads, head_dim, bias, mask, smask, inf, o, stream)) return rc;
  a = LinearF32{};
  a.m = (int)m;
  a.x = o, a.k = (int)d;
  a.w = p[4], a.n = (int)d;
  a.res = s, a.out = out, a.ldo = d;
  if (int rc = launch_linear<false, false>(fn, a, stream)) return rc;
  a = LinearF32{};
  a.m = (int)m;
  a.x = out, a.k = (int)d;
  a.ln_w = p[5], a.ln_b = p[6], a.eps = eps_trans;
  a.w = p[7], a.n = (int)hidden;
  a.out = hid;
  if (int rc = launch_linear<true, true>(fn, a, stream)) return rc;
  a = LinearF32{};
  a.m = (int)m;
  a.x = hid, a.k = (int)hidden;
  a.w = p[8], a.n = (int)d;
  a.res = out, a.out = out, a.ldo = d;
  return launch_linear<false, false>(fn, a, stream);
}

}  // extern "C"
