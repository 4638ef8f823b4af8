// Near-fp32 linears on bf16 MFMA for few rows, and the score model's token
// transformer built from them.
//
// out[m][n] = sum_k x[m][k] w[n][k] + b[n] with both operands split into bf16
// high and low parts (x = xh + xl, w = wh + wl) and the products xh wh + xl wh +
// xh wl accumulated in fp32: the split-bf16 form of the fp32 linears
// (split_operand.hip; about 2^-16 relative per product).
//
// What bounds it: with few rows (one sample of a small target: 117 tokens, or
// up to 1024 rows) a linear is one pass over its weights and a chain of
// latencies, not matrix work.  A library GEMM takes 15-24 us for any of them
// (few tiles, one after another along K); here every 32 x 32 or 32 x 64 tile
// is a block of its own, its four waves split K, and both operands lie packed
// in MFMA operand order (x3_packed_index), so that a fragment is one
// contiguous 1 KB load straight to registers, with no LDS stage and no barrier
// before the waves' sums meet.  Measured (weights in the Infinity Cache; library
// split-bf16 GEMM in brackets): 117 x 768 x 768 4.1 us (21), 117 x 3072 x 768
// 5.3 (21), 117 x 768 x 1536 5.8 (24), 512 x 3072 x 768 11.8 (21), 1024 x 768 x
// 768 7.5 (21), 1024 x 3072 x 768 21 (22), 2048 x 3072 x 768 48 (34): the line
// to the library GEMM lies at 1024 rows (kMaxRows).  Whole stacks of 24 layers on
// either side of it, one call here and per-layer calls in brackets (bound by the
// host, 11 launches a layer): 117 rows 1.6 ms (7.2), 512 3.1 (6.9), 1024 5.1
// (6.5 .. 7.0), 5 x 204 4.5 (7.2); 1025 rows by per-layer calls 6.5.
#include "bmx_common.h"

using namespace bmx;

namespace {

constexpr int64_t kMaxRows = 1024;

struct LinearArgs {
  const bf16* x;   // packed operand of m x k
  const bf16* x2;  // packed operand of the output tiles from tile_split on
  const bf16* w;   // packed weight rows, n x k (swiglu: tiles x, gate, b in turn)
  const float* bias;
  float* out;
  bf16* op;  // swiglu: packed operand of m x inner
  int64_t ldo;
  int m, n, ksteps;  // ksteps = k / 16
  int tiles_m, tiles_n, tile_split;
};

constexpr int kW = 4;  // waves of a block, each a quarter of the k steps

// One 32 x (32 TJ) tile per block.  SWIGLU (TJ = 3): the three column tiles are
// 32 outputs each of the swish gate's value and gate halves and of a_to_b, and
// the result is the packed operand of silu(gate) * value * b.
template <int TJ, bool SWIGLU>
__global__ __launch_bounds__(64 * kW) void linear_x3_kernel(LinearArgs a) {
  constexpr int TN = 32 * TJ, kRow = TN + 4;
  constexpr int kBatch = TJ == 1 ? 6 : TJ == 2 ? 3 : 2;
  static_assert(!SWIGLU || TJ == 3, "value, gate and b tiles");
  __shared__ __attribute__((aligned(16))) float red[kW][32 * kRow];
  const int l = lane_id(), wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  // Blocks go round-robin over the 8 XCDs; each XCD takes a contiguous run of
  // tiles, x row tiles first, so its L2 holds few weight tiles at a time.
  const int tiles = a.tiles_m * a.tiles_n, per_xcd = (tiles + 7) / 8;
  const int tile = (blockIdx.x & 7) * per_xcd + (blockIdx.x >> 3);
  if (tile >= tiles) return;  // whole block
  const int tm = tile % a.tiles_m, tn = tile / a.tiles_m;
  const int64_t tstride = (int64_t)a.ksteps * 1024;  // elements of one packed 32-row tile
  const int nt = a.n / 32;
  const bf16* px = (tn * TJ < a.tile_split ? a.x : a.x2) + tm * tstride + 8 * l;
  const bf16* pw[TJ];
#pragma unroll
  for (int j = 0; j < TJ; ++j) pw[j] = a.w + min(tn * TJ + j, nt - 1) * tstride + 8 * l;
  f32x16 acc[TJ];
#pragma unroll
  for (int j = 0; j < TJ; ++j) acc[j] = zero16();
  const int k0 = a.ksteps * wv / kW, k1 = a.ksteps * (wv + 1) / kW;
  // The loads of kBatch k steps are requested together: a pass over all
  // layers' weights finds them in HBM, and a quarter of K = 768 (12 steps) then
  // waits twice for them. 32-wide tiles at 117 rows, mean of a layer's four:
  // 11.3 us with the compiler's three steps of one wave in flight, 9.4 with 6, 9.3
  // with 12 (and half the blocks per CU).  Wide tiles have the blocks to hide
  // it: 3 steps, 2 with the SwiGLU (500 rows: 17.6 us against 20.0 with 4).
  for (int ks = k0; ks < k1; ks += kBatch) {
    bf16x8 xh[kBatch], xl[kBatch], wh[kBatch][TJ], wl[kBatch][TJ];
#pragma unroll
    for (int b = 0; b < kBatch; ++b) {
      const int64_t o = (int64_t)min(ks + b, k1 - 1) * 1024;  // past the end: the last step again, unused
#pragma unroll
      for (int j = 0; j < TJ; ++j) wh[b][j] = gload8(pw[j] + o), wl[b][j] = gload8(pw[j] + o + 512);
      xh[b] = gload8(px + o), xl[b] = gload8(px + o + 512);
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int b = 0; b < kBatch; ++b) {
      if (ks + b < k1) {  // wave-uniform
#pragma unroll
        for (int j = 0; j < TJ; ++j) {
          acc[j] = mfma32(wh[b][j], xh[b], acc[j]);
          acc[j] = mfma32(wh[b][j], xl[b], acc[j]);
          acc[j] = mfma32(wl[b][j], xh[b], acc[j]);
        }
      }
    }
  }
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
    for (int p = 1; p < kW; ++p) v += *(const f32x4*)(&red[p][r * kRow + c]);
    return v;
  };
  if constexpr (SWIGLU) {
    const int r = threadIdx.x / 8, c = 4 * (threadIdx.x % 8), m = tm * 32 + r, col = tn * 32 + c;
    f32x4 x = sum(r, c), g = sum(r, 32 + c), b = sum(r, 64 + c);
    if (m < a.m) {
      const int inner = a.n / 3;
      if (a.bias) {
        x += load4(a.bias + col);
        g += load4(a.bias + inner + col);
        b += load4(a.bias + 2 * inner + col);
      }
      f32x4 y;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const float act = g[e] / (1.f + __expf(-g[e]));
        const float prod = act * x[e];
        y[e] = prod * b[e];
      }
      x3_packed_store4(a.op, m, col, inner >> 4, y);
    }
  } else {
#pragma unroll
    for (int u = 0; u < TJ; ++u) {
      const int e = threadIdx.x + 64 * kW * u, r = e / (TN / 4), c = 4 * (e % (TN / 4));
      const int m = tm * 32 + r, n = tn * TN + c;
      f32x4 v = sum(r, c);
      if (m < a.m && n < a.n) {
        if (a.bias) v += load4(a.bias + n);
        store4(a.out + (int64_t)m * a.ldo + n, v);
      }
    }
  }
}

int launch_linear(const char* name, LinearArgs a, hipStream_t stream) {
  a.tiles_m = (a.m + 31) / 32;
  const int nt = a.n / 32;
  // 32-wide tiles while that is at most three blocks per CU, 64-wide ones (one
  // read of the x tile for two weight tiles) above: 117 x 768: 4.1 us against
  // 4.9, 1024 x 768: 7.5 against 8.5, 512 x 3072: 12.7 against 11.8, 1024 x 3072:
  // 24 against 21.
  const bool wide = (int64_t)a.tiles_m * nt > 3 * device_cu_count();
  a.tiles_n = a.op ? nt / 3 : wide ? (nt + 1) / 2 : nt;
  if (!a.x2) a.x2 = a.x, a.tile_split = nt;
  const dim3 grid(8 * ((a.tiles_m * a.tiles_n + 7) / 8)), block(64 * kW);
  if (a.op)
    linear_x3_kernel<3, true><<<grid, block, 0, stream>>>(a);
  else if (wide)
    linear_x3_kernel<2, false><<<grid, block, 0, stream>>>(a);
  else
    linear_x3_kernel<1, false><<<grid, block, 0, stream>>>(a);
  return check_launch(name);
}

// Weight rows (times col_scale per column, if given) to packed operand tiles:
// 32 rows tile t of w goes to packed tile tile0 + t * tile_stride.  One wave per
// (32-row tile, 16-column step): lane (row l % 32, 8 columns).
__global__ __launch_bounds__(64) void x3_pack_kernel(const float* __restrict__ w, int64_t ldw, int ksteps,
                                                     const float* __restrict__ col_scale, int64_t tile0,
                                                     int64_t tile_stride, bf16* __restrict__ out) {
  const int l = threadIdx.x, ks = blockIdx.x, c0 = 16 * ks + 8 * (l >> 5);
  const float* row = w + ((int64_t)blockIdx.y * 32 + (l & 31)) * ldw + c0;
  bf16x8 hi, lo;
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    const float v = col_scale ? row[e] * col_scale[c0 + e] : row[e];
    hi[e] = (bf16)v;
    lo[e] = (bf16)(v - (float)hi[e]);
  }
  bf16* dst = out + ((tile0 + blockIdx.y * tile_stride) * ksteps + ks) * 1024 + 8 * l;
  *(bf16x8*)dst = hi;
  *(bf16x8*)(dst + 512) = lo;
}

inline int64_t align256(int64_t v) { return (v + 255) / 256 * 256; }

// Workspace of a token stack: byte offsets of its parts.
struct StackWorkspace {
  int64_t xn, xs, op, up, cond[2], proj, y, attn, total;
};
StackWorkspace stack_workspace(int64_t batch, int64_t n, int heads, int head_dim, int64_t inner) {
  const int64_t d = (int64_t)heads * head_dim, m = batch * n, mp = (m + 31) / 32 * 32;
  StackWorkspace w;
  int64_t at = 0;
  auto take = [&](int64_t bytes) {
    const int64_t here = at;
    at += align256(bytes);
    return here;
  };
  w.xn = take(mp * d * 4);  // packed: 2 x bf16
  w.xs = take(mp * d * 4);
  w.op = take(mp * d * 4);
  w.up = take(mp * inner * 4);
  w.cond[0] = take(m * 6 * d * 4);
  w.cond[1] = take(m * 6 * d * 4);
  w.proj = take(m * 4 * d * 4);
  w.y = take(m * d * 4);
  w.attn = take((int64_t)token_attention_workspace(batch, n, heads, head_dim));
  w.total = at;
  return w;
}

}  // namespace

extern "C" {

int bmx_gated_residual(const float* a, const float* gate, int64_t ld_gate, const float* c, float* out, int64_t rows,
                       int64_t cols, hipStream_t stream);

int bmx_x3_pack(const float* w, int64_t rows, int64_t k, int64_t ldw, const float* col_scale, int64_t tile0,
                int64_t tile_stride, void* out, hipStream_t stream) {
  BMX_REQUIRE(rows >= 0 && rows % 32 == 0 && k > 0 && k % 16 == 0 && ldw >= k,
              "bmx_x3_pack: rows must be a multiple of 32, k a positive multiple of 16, ldw >= k");
  BMX_REQUIRE(rows / 32 <= 65535 && k / 16 <= (1 << 30) && tile0 >= 0 && tile_stride >= 1,
              "bmx_x3_pack: at most 65535 tiles of 32 rows, tile0 >= 0, tile_stride >= 1");
  if (rows == 0) return BMX_OK;
  BMX_REQUIRE(w && out, "bmx_x3_pack: null pointer");
  BMX_REQUIRE((uintptr_t)out % 16 == 0, "bmx_x3_pack: out must be 16-byte aligned");
  x3_pack_kernel<<<dim3((unsigned)(k / 16), (unsigned)(rows / 32)), 64, 0, stream>>>(w, ldw, (int)(k / 16), col_scale,
                                                                                     tile0, tile_stride, (bf16*)out);
  return check_launch("bmx_x3_pack");
}

size_t bmx_token_stack_workspace_bytes(int64_t batch, int64_t n, int heads, int head_dim, int64_t inner) {
  if (batch <= 0 || n <= 0 || heads <= 0 || head_dim <= 0 || inner <= 0) return 0;
  return (size_t)stack_workspace(batch, n, heads, head_dim, inner).total;
}

int bmx_token_stack_fwd(const float* a, const float* s, int64_t batch, int64_t n, int heads, int head_dim,
                        int64_t inner, int layers, const void* const* params, float eps_s, const float* eps,
                        const float* mask, int64_t smask, int64_t sbias, int64_t bias_div, float inf, float* out,
                        void* workspace, size_t workspace_bytes, hipStream_t stream) {
  const char* fn = "bmx_token_stack_fwd";
  BMX_REQUIRE(batch >= 0 && n >= 0 && batch <= kMaxRows && n <= kMaxRows && batch * n <= kMaxRows,
              "bmx_token_stack_fwd: batch * n must be in [0, %lld]", (long long)kMaxRows);
  BMX_REQUIRE(head_dim == 24 || head_dim == 32 || head_dim == 48,
              "bmx_token_stack_fwd: head_dim must be 24, 32 or 48 (got %d)", head_dim);
  BMX_REQUIRE(heads >= 1 && heads <= 64, "bmx_token_stack_fwd: heads must be in [1, 64] (got %d)", heads);
  const int64_t d = (int64_t)heads * head_dim, m = batch * n;
  BMX_REQUIRE(d % 32 == 0 && d <= 1024 && inner > 0 && inner % 32 == 0 && inner <= (1 << 20),
              "bmx_token_stack_fwd: need heads * head_dim a multiple of 32, at most 1024, inner a multiple of 32");
  BMX_REQUIRE(layers >= 0 && bias_div >= 1 && smask >= 0 && sbias >= 0 && inf > 0.f && eps_s > 0.f,
              "bmx_token_stack_fwd: need layers >= 0, bias_div >= 1, strides >= 0, inf and eps positive");
  if (m == 0 || layers == 0) return BMX_OK;
  BMX_REQUIRE(a && s && params && eps && mask && out && workspace, "bmx_token_stack_fwd: null pointer");
  for (int i = 0; i < 11 * layers; ++i)  // the five biases may be null
    BMX_REQUIRE(params[i] || (i % 11 < 10 && i % 11 % 2 == 1), "bmx_token_stack_fwd: null parameter %d of layer %d",
                i % 11, i / 11);
  for (int i = 0; i < 11 * layers; ++i)
    BMX_REQUIRE((uintptr_t)params[i] % 16 == 0 || i % 11 == 10,
                "bmx_token_stack_fwd: parameter %d of layer %d must be 16-byte aligned", i % 11, i / 11);
  for (int i = 0; i < 2 * layers; ++i) BMX_REQUIRE(eps[i] > 0.f, "bmx_token_stack_fwd: eps must be positive");
  BMX_REQUIRE(((uintptr_t)a | (uintptr_t)s | (uintptr_t)out) % 16 == 0,
              "bmx_token_stack_fwd: a, s and out must be 16-byte aligned");
  const StackWorkspace ws = stack_workspace(batch, n, heads, head_dim, inner);
  BMX_REQUIRE(workspace_bytes >= (size_t)ws.total && (uintptr_t)workspace % 256 == 0,
              "bmx_token_stack_fwd: workspace must be 256-byte aligned and hold %lld bytes", (long long)ws.total);
  char* base = (char*)workspace;
  bf16 *xn = (bf16*)(base + ws.xn), *xs = (bf16*)(base + ws.xs), *op = (bf16*)(base + ws.op),
       *up = (bf16*)(base + ws.up);
  float *proj = (float*)(base + ws.proj), *y = (float*)(base + ws.y);
  const int di = (int)d, mi = (int)m;
  const int64_t ldc = 6 * d;
  auto linear = [&](const bf16* x, const void* w, const void* b, int64_t nn, int64_t k, float* o, bf16* o_op) {
    LinearArgs p{};
    p.x = x;
    p.w = (const bf16*)w;
    p.bias = (const float*)b;
    p.out = o;
    p.op = o_op;
    p.ldo = nn;
    p.m = mi;
    p.n = (int)nn;
    p.ksteps = (int)(k / 16);
    return launch_linear(fn, p, stream);
  };
  // [attention scale | shift | transition scale | shift] of LayerNorm(s), [attention | transition gate] of s
  auto conditioning = [&](int i) {
    LinearArgs p{};
    p.x = xn;
    p.x2 = xs;
    p.tile_split = (int)(4 * d / 32);
    p.w = (const bf16*)params[11 * i];
    p.bias = (const float*)params[11 * i + 1];
    p.out = (float*)(base + ws.cond[i & 1]);
    p.ldo = ldc;
    p.m = mi;
    p.n = (int)ldc;
    p.ksteps = (int)(d / 16);
    return launch_linear(fn, p, stream);
  };
  int rc = split_packed(s, m, di, xs, stream);
  if (!rc) rc = layernorm_packed(s, m, di, eps_s, xn, stream);
  if (!rc) rc = conditioning(0);
  if (!rc) {
    const float* c = (const float*)(base + ws.cond[0]);
    rc = adaln_packed(a, c, c + d, ldc, m, di, eps[0], op, stream);
  }
  for (int i = 0; i < layers && !rc; ++i) {
    const void* const* p = params + 11 * i;
    const float* c = (const float*)(base + ws.cond[i & 1]);
    rc = linear(op, p[2], p[3], 4 * d, d, proj, nullptr);
    if (!rc)
      rc = token_attention_packed(proj, batch, n, heads, head_dim, (const float*)p[10], sbias, bias_div, mask, smask,
                                  inf, op, base + ws.attn, stream);
    if (!rc) rc = linear(op, p[4], p[5], d, d, y, nullptr);
    if (!rc)
      rc = gated_residual_adaln_packed(y, c + 4 * d, ldc, i ? out : a, out, c + 2 * d, c + 3 * d, ldc, m, di,
                                       eps[2 * i + 1], op, stream);
    if (!rc) rc = linear(op, p[6], p[7], 3 * inner, d, nullptr, up);
    if (!rc) rc = linear(up, p[8], p[9], d, inner, y, nullptr);
    if (rc) break;
    if (i + 1 < layers) {
      rc = conditioning(i + 1);
      const float* cn = (const float*)(base + ws.cond[(i + 1) & 1]);
      if (!rc)
        rc = gated_residual_adaln_packed(y, c + 5 * d, ldc, out, out, cn, cn + d, ldc, m, di, eps[2 * i + 2], op,
                                         stream);
    } else {
      rc = bmx_gated_residual(y, c + 5 * d, ldc, out, out, m, d, stream);
    }
  }
  return rc;
}

}  // extern "C"
