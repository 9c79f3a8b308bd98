// Tiled bf16-MFMA GEMM for fp32 activations, and what the VAE decoder builds on it:
//   * conv3x3 (pad 1) of an NHWC image, with the 2x nearest upsample of the input and the residual add
//     fused (the "conv3" loader of app/gpu/gemm.js:56-80, dispatched by ops.conv3x3 / conv3x3Into,
//     app/gpu/ops.js:95-109): by rows, on spatial tiles, or as an implicit GEMM;
//   * the Wan channel norm y = x / max(||x||, 1e-12) * sqrt(C) * gamma (+ SiLU) of
//     app/gpu/kernels.js:62-89 (mode 1), in the shader's reduction order;
//   * attention for head dims other than 128: 384 (the VAE's single head) fused, others on the
//     reference's chunked path (app/gpu/ops.js:177-207): scores for a chunk of query rows, a row
//     softmax (optionally causal), then P.V.
//
// The GEMM: C[m][n] = alpha * sum_k A[m][k] B[n][k] (* rs[m]) (+ bias[n]) (act), stored or added
// to C.  One workgroup = 4 waves = a 128 x 128 output tile, each wave 64 x 64 (2 x 2 tiles of
// v_mfma_f32_32x32x16_bf16); k-tiles of 32 are converted to bf16 while they move from global
// memory into a double-buffered LDS image (one barrier per k-tile, the next tile's global loads
// issued before the current tile's MFMAs).  fp32 operands are rounded to bf16, or, with SPLIT,
// written as two bf16 terms x = hi + lo (lo = bf16(x - hi), exact difference): the products
// hi.hi + lo.hi (+ hi.lo for an fp32 B) then carry about 16 significant bits of each operand, an
// fp32-level result (relative error ~1e-5 over long sums) from the bf16 matrix cores.  bf16
// weights (the VAE's checkpoint format) are exact and never split.
#include <algorithm>
#include <cmath>

#include "common.h"
#include "internal.h"

namespace anima {

constexpr int TG_BM = 128, TG_BN = 128, TG_BK = 32;
constexpr int TG_ROW = TG_BK + 8;  // LDS row stride in bf16 (80 B): conflict-free fragment reads

enum { TG_A_ROWS = 0, TG_A_CONV = 1 };
enum { TG_B_W16 = 0, TG_B_F32 = 1 };

struct TGemmArgs {
  // A: a[z*a_bs + m*lda + k], or (conv) the im2col of the NHWC image a[z*a_bs + ((b*Hin + y)*Win + x)*cin + c]
  const float* a;
  int64_t lda, a_bs;
  int cin, H, W, up;  // conv: output H x W per image; the input is H x W, or H/2 x W/2 with up
  // B: b[z*b_bs + n*ldb + k], bf16 or fp32
  const void* b;
  int64_t ldb, b_bs;
  float* c;
  int64_t ldc, c_bs;
  const float* bias;  // [N] or null
  const float* rs;    // per-row scale rs[z*rs_bs + m] or null
  int64_t rs_bs;
  float alpha;
  int act, resid;
  int M, N, K;
};

// The output pixel of a conv A row, decomposed once per thread: image base pointer and (oy, ox).
struct ConvRow {
  const float* img;  // first element of this row's image
  int oy, ox;
};

__device__ __forceinline__ ConvRow conv_row(const TGemmArgs& p, const float* a, int m) {
  ConvRow r;
  const int hw = p.H * p.W;
  const int img = m / hw, q = m - img * hw;
  r.oy = q / p.W;
  r.ox = q - r.oy * p.W;
  const int Hin = p.up ? p.H >> 1 : p.H, Win = p.up ? p.W >> 1 : p.W;
  r.img = a + (int64_t)img * Hin * Win * p.cin;
  return r;
}

// 16 consecutive k of A row m starting at k (k % 16 == 0), fp32; zeros outside the matrix / image.
template <int AM>
__device__ __forceinline__ void tg_load_a(const TGemmArgs& p, const float* a, const ConvRow& cr, int m, int k,
                                          float (&v)[16]) {
  bool ok = m < p.M && k < p.K;
  const float* src = nullptr;
  if (ok) {
    if constexpr (AM == TG_A_ROWS) {
      src = a + (int64_t)m * p.lda + k;
    } else {
      const int tap = k / p.cin, ci = k - tap * p.cin;  // cin is uniform: a scalar division
      const int ty = tap / 3, tx = tap - 3 * ty;
      const int iy = cr.oy + ty - 1, ix = cr.ox + tx - 1;
      ok = iy >= 0 && ix >= 0 && iy < p.H && ix < p.W;
      const int Win = p.up ? p.W >> 1 : p.W;
      const int sy = p.up ? iy >> 1 : iy, sx = p.up ? ix >> 1 : ix;
      src = cr.img + ((int64_t)sy * Win + sx) * p.cin + ci;
    }
  }
  if (ok && (AM == TG_A_CONV || k + 16 <= p.K)) {  // conv: cin % 16 == 0, a run never crosses a tap
#pragma unroll
    for (int j = 0; j < 4; j++) {
      const float4 t = *(const float4*)(src + 4 * j);
      v[4 * j] = t.x; v[4 * j + 1] = t.y; v[4 * j + 2] = t.z; v[4 * j + 3] = t.w;
    }
  } else if (ok) {  // rows: the last, partial k-run
#pragma unroll
    for (int j = 0; j < 16; j++) v[j] = k + j < p.K ? src[j] : 0.0f;
  } else {
#pragma unroll
    for (int j = 0; j < 16; j++) v[j] = 0.0f;
  }
}

__device__ __forceinline__ void tg_split(const float (&v)[16], bf16x8 (&hi)[2], bf16x8 (&lo)[2], bool split) {
#pragma unroll
  for (int j = 0; j < 16; j++) {
    const bf16 h = to_bf16(v[j]);
    hi[j >> 3][j & 7] = h;
    if (split) lo[j >> 3][j & 7] = to_bf16(v[j] - (float)h);
  }
}

template <int AM, int BMODE, bool SPLIT>
__global__ __launch_bounds__(256) void tgemm_kernel(TGemmArgs p) {
  constexpr int NA = SPLIT ? 2 : 1;
  constexpr int NB = (SPLIT && BMODE == TG_B_F32) ? 2 : 1;
  __shared__ __attribute__((aligned(16))) bf16 sa[2][NA][TG_BM * TG_ROW];
  __shared__ __attribute__((aligned(16))) bf16 sb[2][NB][TG_BN * TG_ROW];
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, lq = lane & 31, hf = lane >> 5;
  const int z = blockIdx.z;
  const int m0 = blockIdx.x * TG_BM, n0 = blockIdx.y * TG_BN;
  const float* a = p.a + (int64_t)z * p.a_bs;
  const char* bb = (const char*)p.b + (int64_t)z * p.b_bs * (BMODE == TG_B_W16 ? 2 : 4);
  // loader role: row t/2 of the A and B tiles, k-half t%2 (16 k)
  const int lr = tid >> 1, lk = 16 * (tid & 1);
  const int am = m0 + lr, bn = n0 + lr;
  const bool bok = bn < p.N;

  ConvRow cr{};
  if constexpr (AM == TG_A_CONV) {
    if (am < p.M) cr = conv_row(p, a, am);
  }
  float av[16];
  uint4 bw[2];   // bf16 B: 16 values
  float bv[16];  // fp32 B
  auto load = [&](int k0) {
    tg_load_a<AM>(p, a, cr, am, k0 + lk, av);
    const int k = k0 + lk;
    if constexpr (BMODE == TG_B_W16) {
      const uint16_t* src = (const uint16_t*)bb + (int64_t)bn * p.ldb + k;
      if (bok && k + 16 <= p.K) {
        bw[0] = *(const uint4*)src;
        bw[1] = *(const uint4*)(src + 8);
      } else {
        uint16_t t[16];
#pragma unroll
        for (int j = 0; j < 16; j++) t[j] = bok && k + j < p.K ? src[j] : (uint16_t)0;
        uint32_t u[8];
#pragma unroll
        for (int j = 0; j < 8; j++) u[j] = (uint32_t)t[2 * j] | ((uint32_t)t[2 * j + 1] << 16);
        bw[0] = make_uint4(u[0], u[1], u[2], u[3]);
        bw[1] = make_uint4(u[4], u[5], u[6], u[7]);
      }
    } else {
      const float* src = (const float*)bb + (int64_t)bn * p.ldb + k;
      if (bok && k + 16 <= p.K) {
#pragma unroll
        for (int j = 0; j < 4; j++) {
          const float4 t = *(const float4*)(src + 4 * j);
          bv[4 * j] = t.x; bv[4 * j + 1] = t.y; bv[4 * j + 2] = t.z; bv[4 * j + 3] = t.w;
        }
      } else {
#pragma unroll
        for (int j = 0; j < 16; j++) bv[j] = bok && k + j < p.K ? src[j] : 0.0f;
      }
    }
  };
  auto store = [&](int st) {
    bf16x8 hi[2], lo[2];
    tg_split(av, hi, lo, SPLIT);
    *(bf16x8*)(&sa[st][0][lr * TG_ROW + lk]) = hi[0];
    *(bf16x8*)(&sa[st][0][lr * TG_ROW + lk + 8]) = hi[1];
    if constexpr (SPLIT) {
      *(bf16x8*)(&sa[st][NA - 1][lr * TG_ROW + lk]) = lo[0];
      *(bf16x8*)(&sa[st][NA - 1][lr * TG_ROW + lk + 8]) = lo[1];
    }
    if constexpr (BMODE == TG_B_W16) {
      *(uint4*)(&sb[st][0][lr * TG_ROW + lk]) = bw[0];
      *(uint4*)(&sb[st][0][lr * TG_ROW + lk + 8]) = bw[1];
    } else {
      bf16x8 bh[2], bl[2];
      tg_split(bv, bh, bl, NB == 2);
      *(bf16x8*)(&sb[st][0][lr * TG_ROW + lk]) = bh[0];
      *(bf16x8*)(&sb[st][0][lr * TG_ROW + lk + 8]) = bh[1];
      if constexpr (NB == 2) {
        *(bf16x8*)(&sb[st][NB - 1][lr * TG_ROW + lk]) = bl[0];
        *(bf16x8*)(&sb[st][NB - 1][lr * TG_ROW + lk + 8]) = bl[1];
      }
    }
  };

  const int wm = wave >> 1, wn = wave & 1;
  f32x16 acc[2][2];
#pragma unroll
  for (int i = 0; i < 2; i++)
#pragma unroll
    for (int j = 0; j < 2; j++) acc[i][j] = f32x16{};

  const int nkt = (p.K + TG_BK - 1) / TG_BK;
  load(0);
  store(0);
  __syncthreads();
  for (int kt = 0; kt < nkt; kt++) {
    const int st = kt & 1;
    if (kt + 1 < nkt) load((kt + 1) * TG_BK);
#pragma unroll
    for (int ks = 0; ks < 2; ks++) {
      bf16x8 fa[2][NA], fb[2][NB];
#pragma unroll
      for (int i = 0; i < 2; i++) {
        const int r = (64 * wm + 32 * i + lq) * TG_ROW + 16 * ks + 8 * hf;
#pragma unroll
        for (int s = 0; s < NA; s++) fa[i][s] = *(const bf16x8*)(&sa[st][s][r]);
      }
#pragma unroll
      for (int j = 0; j < 2; j++) {
        const int r = (64 * wn + 32 * j + lq) * TG_ROW + 16 * ks + 8 * hf;
#pragma unroll
        for (int s = 0; s < NB; s++) fb[j][s] = *(const bf16x8*)(&sb[st][s][r]);
      }
#pragma unroll
      for (int i = 0; i < 2; i++)
#pragma unroll
        for (int j = 0; j < 2; j++) {
          acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fa[i][0], fb[j][0], acc[i][j], 0, 0, 0);
          if constexpr (SPLIT) {
            acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fa[i][1], fb[j][0], acc[i][j], 0, 0, 0);
            if constexpr (NB == 2) acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fa[i][0], fb[j][1], acc[i][j], 0, 0, 0);
          }
        }
    }
    if (kt + 1 < nkt) store(st ^ 1);
    __syncthreads();
  }

  // epilogue: register r of tile (i, j) holds row 8(r/4) + 4hf + r%4 and column lq of the tile
  float* cz = p.c + (int64_t)z * p.c_bs;
  const float* rs = p.rs ? p.rs + (int64_t)z * p.rs_bs : nullptr;
#pragma unroll
  for (int j = 0; j < 2; j++) {
    const int n = n0 + 64 * wn + 32 * j + lq;
    if (n >= p.N) continue;
    const float bias = p.bias ? p.bias[n] : 0.0f;
#pragma unroll
    for (int i = 0; i < 2; i++)
#pragma unroll
      for (int r = 0; r < 16; r++) {
        const int m = m0 + 64 * wm + 32 * i + 8 * (r >> 2) + 4 * hf + (r & 3);
        if (m >= p.M) continue;
        float v = acc[i][j][r] * p.alpha;
        if (rs) v = v * rs[m];
        v = v + bias;
        if (p.act == ANIMA_ACT_SILU) v = silu_f(v);
        else if (p.act == ANIMA_ACT_GELU) v = gelu_erf(v);
        float* dst = cz + (int64_t)m * p.ldc + n;
        *dst = p.resid ? *dst + v : v;
      }
  }
}

// Launches tgemm_kernel over a batch of `batch` independent products (blockIdx.z).
static int tgemm_launch(anima_ctx* c, const TGemmArgs& p, int amode, int bmode, bool split, int batch, const char* name,
                        double flops) {
  if (p.M <= 0 || p.N <= 0 || p.K <= 0 || batch <= 0) return ANIMA_OK;
  const int64_t gn = (p.N + TG_BN - 1) / TG_BN;
  if (gn > 65535 || batch > 65535) return fail(c, ANIMA_E_ARG, "%s: N=%d, batch %d beyond the grid", name, p.N, batch);
  dim3 grid((p.M + TG_BM - 1) / TG_BM, (unsigned)gn, batch);
  Launch L(c, name, flops, 0.0);
#define TG(A, B, S) hipLaunchKernelGGL((tgemm_kernel<A, B, S>), grid, dim3(256), 0, c->stream, p)
  if (amode == TG_A_CONV) {
    if (split) TG(TG_A_CONV, TG_B_W16, true);
    else TG(TG_A_CONV, TG_B_W16, false);
  } else if (bmode == TG_B_W16) {
    if (split) TG(TG_A_ROWS, TG_B_W16, true);
    else TG(TG_A_ROWS, TG_B_W16, false);
  } else {
    if (split) TG(TG_A_ROWS, TG_B_F32, true);
    else TG(TG_A_ROWS, TG_B_F32, false);
  }
#undef TG
  return L.end();
}

// ---- conv3x3 on spatial tiles (the 3-channel head, more than 384 channels, and sizes of more than 192 where it is
// shorter than conv3x3_rows_kernel below): a workgroup (8 waves) computes a 16 x 32 block of output pixels
// for BN = 96 output channels (or one 32-wide column tile when cout <= 32: the 3-channel head).  Per step of 32 input channels the input halo it needs (18 x 34 pixels in
// output coordinates, sampled through the 2x nearest upsample when up; zero outside the image) and
// the 9 x 96 x 32 weights are copied once into LDS, so every input value is read from memory once
// per step instead of once per tap (the row-tiled implicit GEMM reads each pixel nine times).  The
// next step's halo and weights are loaded into registers before this step's MFMAs.  With NW waves,
// wave w owns MT = 16 / NW output rows from MT w (32-pixel MFMA row tiles) x three 32-channel
// column tiles (NW = 8: 4 waves ran the fp32 convs 10-15% slower and the bf16 ones 2% faster); for tap
// (ty, tx) the A row of output pixel (r, c) is halo pixel (r + ty, c + tx).  LDS rows are 64 bytes
// (32 channels) with the 16-byte unit u of row q stored at slot u ^ ((q / 4) % 4), so the fragment
// reads of 16 consecutive rows fall in distinct bank groups.  Products and sums are those of
// tgemm_kernel (activation rounded to bf16, or split hi + lo with SPLIT; bf16 weights exact); only
// the order of the k-terms differs (input-channel chunk outer, tap inner).
constexpr int CT_TH = 16, CT_TW = 32, CT_HH = CT_TH + 2, CT_HW = CT_TW + 2, CT_HP = CT_HH * CT_HW;
constexpr int CT_CC = 32, CT_NW = 8;
constexpr int CT_HU = CT_HP * 4;          // 16-byte units of one halo plane (8 channels each)

__device__ __forceinline__ int ct_off(int row, int u) { return row * 64 + ((u ^ ((row >> 2) & 3)) << 4); }

template <bool SPLIT, int NW, int BN>
__global__ __launch_bounds__(64 * NW) void conv3x3_tile_kernel(TGemmArgs p) {
  constexpr int NA = SPLIT ? 2 : 1;
  constexpr int NJ = BN / 32;              // 32-channel MFMA column tiles per wave
  constexpr int CT_WU = 9 * BN * 4;        // 16-byte units of the step's weights
  constexpr int NT = 64 * NW, MT = CT_TH / NW;  // threads; output rows (32-pixel MFMA tiles) per wave
  constexpr int CT_HJ = (CT_HU + NT - 1) / NT, CT_WJ = (CT_WU + NT - 1) / NT;
  __shared__ __attribute__((aligned(16))) char lds[NA * CT_HP * 64 + 9 * BN * 64];
  char* const wl = lds + NA * CT_HP * 64;
  const int t = threadIdx.x, wave = t >> 6, lane = t & 63, lq = lane & 31, hf = lane >> 5;
  const int tx_n = p.W / CT_TW, ty_n = p.H / CT_TH;
  const int tile = blockIdx.x, img = tile / (tx_n * ty_n), trem = tile - img * tx_n * ty_n;
  const int oy0 = (trem / tx_n) * CT_TH, ox0 = (trem % tx_n) * CT_TW;
  const int n0 = blockIdx.y * BN;
  const int Hin = p.up ? p.H >> 1 : p.H, Win = p.up ? p.W >> 1 : p.W;
  const float* imgp = p.a + (int64_t)img * Hin * Win * p.cin;
  const uint16_t* W = (const uint16_t*)p.b;

  // staged loads of one step (input channels c0 .. c0 + 31); addresses past the image or the
  // unit count are clamped to valid memory and their units stored as zeros / skipped
  float4 hv[CT_HJ][2];
  uint4 wv[CT_WJ];
  unsigned hok = 0;
  auto stage = [&](int c0) {
    hok = 0;
#pragma unroll
    for (int j = 0; j < CT_HJ; j++) {
      const int U = t + NT * j, px = min(U, CT_HU - 1) >> 2, u = U & 3;
      const int hy = px / CT_HW, hx = px - hy * CT_HW;
      const int y = oy0 - 1 + hy, x = ox0 - 1 + hx;
      const bool ok = U < CT_HU && y >= 0 && x >= 0 && y < p.H && x < p.W;
      const int sy = ok ? (p.up ? y >> 1 : y) : 0, sx = ok ? (p.up ? x >> 1 : x) : 0;
      const float* src = imgp + ((int64_t)sy * Win + sx) * p.cin + c0 + 8 * u;
      hv[j][0] = *(const float4*)src;
      hv[j][1] = *(const float4*)(src + 4);
      hok |= (ok ? 1u : 0u) << j;
    }
#pragma unroll
    for (int j = 0; j < CT_WJ; j++) {
      const int V = min(t + NT * j, CT_WU - 1), tap = V / (BN * 4), rem = V - tap * BN * 4;
      const int n = min(n0 + (rem >> 2), p.N - 1), u = rem & 3;  // channels past cout: never stored
      wv[j] = *(const uint4*)(W + (int64_t)n * p.ldb + tap * p.cin + c0 + 8 * u);
    }
  };
  auto publish = [&]() {
#pragma unroll
    for (int j = 0; j < CT_HJ; j++) {
      const int U = t + NT * j;
      if (U >= CT_HU) break;
      const int px = U >> 2, u = U & 3;
      const bool ok = (hok >> j) & 1;
      const float v[8] = {hv[j][0].x, hv[j][0].y, hv[j][0].z, hv[j][0].w, hv[j][1].x, hv[j][1].y, hv[j][1].z, hv[j][1].w};
      bf16x8 hi, lo;
#pragma unroll
      for (int e = 0; e < 8; e++) {
        const float f = ok ? v[e] : 0.0f;
        hi[e] = to_bf16(f);
        if (SPLIT) lo[e] = to_bf16(f - (float)hi[e]);
      }
      *(bf16x8*)(lds + ct_off(px, u)) = hi;
      if constexpr (SPLIT) *(bf16x8*)(lds + CT_HP * 64 + ct_off(px, u)) = lo;
    }
#pragma unroll
    for (int j = 0; j < CT_WJ; j++) {
      const int V = t + NT * j;
      if (V >= CT_WU) break;
      const int tap = V / (BN * 4), rem = V - tap * BN * 4;
      *(uint4*)(wl + ct_off(tap * BN + (rem >> 2), rem & 3)) = wv[j];
    }
  };

  f32x16 acc[MT][NJ];
#pragma unroll
  for (int i = 0; i < MT; i++)
#pragma unroll
    for (int j = 0; j < NJ; j++) acc[i][j] = f32x16{};

  stage(0);
  for (int c0 = 0; c0 < p.cin; c0 += CT_CC) {
    if (c0 > 0) __syncthreads();  // every wave is done with the previous step's tiles
    publish();
    __syncthreads();
    stage(min(c0 + CT_CC, p.cin - CT_CC));  // the next step's loads fly during these MFMAs
#pragma unroll
    for (int tap = 0; tap < 9; tap++) {
      const int ty = tap / 3, tx = tap - 3 * ty;
#pragma unroll
      for (int s = 0; s < 2; s++) {
        const int u = 2 * s + hf;
        bf16x8 fa[MT][NA], fb[NJ];
#pragma unroll
        for (int i = 0; i < MT; i++) {
          const int px = (MT * wave + i + ty) * CT_HW + lq + tx;
#pragma unroll
          for (int a = 0; a < NA; a++) fa[i][a] = *(const bf16x8*)(lds + a * CT_HP * 64 + ct_off(px, u));
        }
#pragma unroll
        for (int j = 0; j < NJ; j++) fb[j] = *(const bf16x8*)(wl + ct_off(tap * BN + 32 * j + lq, u));
#pragma unroll
        for (int i = 0; i < MT; i++)
#pragma unroll
          for (int j = 0; j < NJ; j++) {
            acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fa[i][0], fb[j], acc[i][j], 0, 0, 0);
            if constexpr (SPLIT) acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fa[i][1], fb[j], acc[i][j], 0, 0, 0);
          }
      }
    }
  }

  // epilogue: register r of tile (i, j) holds pixel 8(r/4) + 4hf + r%4 of output row oy0 + 2w + i
  // and channel n0 + 32j + lq
#pragma unroll
  for (int j = 0; j < NJ; j++) {
    const int n = n0 + 32 * j + lq;
    if (n >= p.N) continue;
    const float bias = p.bias ? p.bias[n] : 0.0f;
#pragma unroll
    for (int i = 0; i < MT; i++) {
      const int y = oy0 + MT * wave + i;
      float* orow = p.c + (((int64_t)img * p.H + y) * p.W + ox0) * p.ldc + n;
#pragma unroll
      for (int r = 0; r < 16; r++) {
        const int x = 8 * (r >> 2) + 4 * hf + (r & 3);
        float v = acc[i][j][r] * p.alpha;
        v = v + bias;
        float* dst = orow + (int64_t)x * p.ldc;
        *dst = p.resid ? *dst + v : v;
      }
    }
  }
}

// ---- conv3x3 by rows: a wave owns 16 output channels x 32 input columns (30 of them with outputs, two
// halo) and walks the input rows of a strip.  Each input pixel's nine products with the taps,
// P[ty][tx] = W[ty][tx] . x(y, x), go to the accumulators of the outputs they belong to; the columns'
// shifts are taken on the finished sums (a neighbouring column is a neighbouring lane: DPP), so the
// pixels need no halo in LDS and no barrier.  They are read AHEAD 32-channel steps ahead, four
// consecutive lanes taking 64 contiguous bytes (loads in the operand layout, where consecutive lanes
// are different pixels, return one lane per cycle and ran at a third of the matrix rate), split, and
// put into the operand layout through 4 KiB of LDS of the wave's own.  The weights of the workgroup's
// BN channels stay in LDS (in fragment order) for its whole run; their reads take half the LDS rate.
// 16 channels and not 32: nine 32 x 32 accumulators leave no second wave per SIMD.
//
// Plain: input row y adds P[0] to output row y + 1, P[1] to row y and P[2] to row y - 1, which is then
// complete: out(x) = A[0](x - 1) + A[1](x) + A[2](x + 1) over its three column accumulators.
//
// UP (2x nearest upsample of the input): output pixel (2y + i, 2x + j) reads upsampled row
// 2y + i + ty - 1, input row y - 1 for (i, ty) = (0, 0), y + 1 for (1, 2) and y otherwise (columns
// alike): the 36 products of an input pixel's four outputs are sums of only nine distinct ones, a
// quarter of the matrix work of convolving at the output's resolution (same products):
//   S[ty][even] = P[ty][0](x - 1) + P[ty][1](x) + P[ty][2](x),  S[ty][odd] = P[ty][0](x) + P[ty][1](x)
//   + P[ty][2](x + 1);  row 2y = S[0](y - 1) + S[1](y) + S[2](y),  row 2y + 1 = S[0](y) + S[1](y) + S[2](y + 1).
// Measured against the spatial tiles below (fp32 / bf16, with the channel norms around them): residual
// block 96 channels 1024 x 1024 1560 -> 1238 / 1303 -> 1074 us, 384 channels 32 x 32 275 -> 97 / 190 ->
// 73; with the upsampling 192 channels 320 x 448 1120 -> 679 / 814 -> 507, 384 channels 256 x 256
// 1498 -> 1277 / 971 -> 817 (an upsampling conv of 192 channels at 512 x 512 alone 707 -> 301, a plain
// one 484 -> 472: about 30% of the matrix rate in both).
constexpr int CR_COLS = 30, CR_LDS = 110592, CR_WLDS = 4096;  // weights; a wave's pixels
constexpr int CR_MAXK = CR_LDS / (9 * 2);  // input channels times BN


__device__ __forceinline__ f32x4 cr_load(__amdgpu_buffer_rsrc_t r, unsigned voff, int soff) {
  const auto v = __builtin_amdgcn_raw_buffer_load_b128(r, voff, soff, 0);
  return __builtin_bit_cast(f32x4, v);
}
// The whole offset in the vector register: with a scalar register as the offset, the compiler lets the
// next vector instruction overwrite the data of a 16-byte store (no hazard on older chips), and first
// components of outputs came out wrong here.
__device__ __forceinline__ void cr_store(__amdgpu_buffer_rsrc_t r, unsigned voff, f32x4 v) {
  typedef unsigned u32x4 __attribute__((ext_vector_type(4)));
  __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, v), r, voff, 0, 0);
}

// v of the column to the left / right; tiles a (columns 0 - 15) and b (16 - 31) in lanes 0 - 15 of a row
__device__ __forceinline__ float cr_dpp(float old, float v, bool right) {
  const int o = __builtin_bit_cast(int, old), s = __builtin_bit_cast(int, v);
  return __builtin_bit_cast(float, right ? __builtin_amdgcn_update_dpp(o, s, 0x101, 0xf, 0xf, false)    // row_shl:1
                                         : __builtin_amdgcn_update_dpp(o, s, 0x111, 0xf, 0xf, false));  // row_shr:1
}
__device__ __forceinline__ float cr_ror(float v, bool right) {
  const int s = __builtin_bit_cast(int, v);
  return __builtin_bit_cast(float, right ? __builtin_amdgcn_mov_dpp(s, 0x12f, 0xf, 0xf, false)    // row_ror:15
                                         : __builtin_amdgcn_mov_dpp(s, 0x121, 0xf, 0xf, false));  // row_ror:1
}

typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
typedef float f32x2_t __attribute__((ext_vector_type(2)));
// eight channels as bf16 hi (+ lo = the rounding's rest), two at a time (packed conversions)
template <bool SPLIT>
__device__ __forceinline__ void cr_split(const f32x4 (&v)[2], bf16x8& hi, bf16x8& lo) {
#pragma unroll
  for (int e = 0; e < 8; e += 2) {
    const f32x2_t f = {v[e >> 2][e & 3], v[e >> 2][(e & 3) + 1]};
    const bf16x2_t h = __builtin_convertvector(f, bf16x2_t);
    hi[e] = h[0];
    hi[e + 1] = h[1];
    if constexpr (SPLIT) {
      const bf16x2_t l = __builtin_convertvector(f - __builtin_convertvector(h, f32x2_t), bf16x2_t);
      lo[e] = l[0];
      lo[e + 1] = l[1];
    }
  }
}
// orders this wave's LDS accesses for the compiler (the hardware keeps a wave's LDS order)
__device__ __forceinline__ void cr_order() { asm volatile("" ::: "memory"); }

template <bool UP, bool SPLIT, int BN, int AHEAD>
__global__ __launch_bounds__(512, 2) void conv3x3_rows_kernel(TGemmArgs p, int R, int ncol, int nstrip, int ncg, int ntask) {
  __shared__ __attribute__((aligned(16))) char lds[CR_LDS + 8 * CR_WLDS];
  constexpr int NG = BN / 16, TPW = 8 / NG;  // channel groups; tasks per workgroup
  const int t = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(t >> 6), lane = t & 63, l16 = lane & 15, lg = lane >> 4;
  // an XCD takes all channel blocks of a task one after the other: they read the same pixels
  const int j8 = blockIdx.x >> 3, cg = j8 % ncg, tg = (blockIdx.x & 7) + 8 * (j8 / ncg);
  if (tg * TPW >= ntask) return;
  const int n0 = cg * BN, cin = p.cin, nst = cin / 32;
  const uint16_t* W = (const uint16_t*)p.b;
  // weights in fragment order: [32-channel step][tap][channel group][lane: channel lane % 16, k = input
  // channels 4 (lane / 16) .. + 3 of each half of the step].  (Pixels are then 64 contiguous bytes per
  // load instruction; eight channels in a row per lane would take twice the segments.)
#pragma unroll 4
  for (int u = t; u < nst * 9 * NG * 64; u += 512) {
    const int ln = u & 63, f = u >> 6, g = f % NG, tap = (f / NG) % 9, st = f / (9 * NG);
    const int n = min(n0 + 16 * g + (ln & 15), p.N - 1);  // channels past cout: never stored
    const uint16_t* src = W + (int64_t)n * p.ldb + tap * cin + 32 * st + 4 * (ln >> 4);
    const uint2 a = *(const uint2*)src, b = *(const uint2*)(src + 16);
    *(uint4*)(lds + 16 * u) = make_uint4(a.x, a.y, b.x, b.y);
  }
  __syncthreads();
  const int task = tg * TPW + wave / NG, g = wave % NG;
  if (task >= ntask) return;
  const int Hin = UP ? p.H >> 1 : p.H, Win = UP ? p.W >> 1 : p.W;
  const int img = task / (ncol * nstrip), rem = task - img * ncol * nstrip;
  const int strip = rem / ncol, x0 = (rem - strip * ncol) * CR_COLS;
  const int y0 = strip * R, y1 = min(y0 + R, Hin);
  const __amdgpu_buffer_rsrc_t rx = __builtin_amdgcn_make_buffer_rsrc(
      (void*)(p.a + (int64_t)img * Hin * Win * cin), (short)0, Hin * Win * cin * 4, 0x00020000);
  const __amdgpu_buffer_rsrc_t ro = __builtin_amdgcn_make_buffer_rsrc(
      (void*)(p.c + (int64_t)img * p.H * p.W * p.ldc), (short)0, p.H * p.W * (int)p.ldc * 4, 0x00020000);
  const int n = n0 + 16 * g + 4 * lg;  // this lane's four channels
  // this lane's pixel of each tile, as read (pixel lane / 4, channels 4 (lane % 4) .. + 3 of each half of
  // the step) and as multiplied and written: columns outside the image read zeros past the resource,
  // halo lanes' loads of the output read zeros and their stores are dropped (unsigned: with a row's offset
  // added, below 2^31 - 2^16, those lanes' offsets pass 2^31 but not 2^32)
  unsigned xo[2], oo[2];
#pragma unroll
  for (int i = 0; i < 2; i++) {
    const int xr = x0 - 1 + 16 * i + (lane >> 2), lx = 16 * i + l16, x = x0 - 1 + lx;
    xo[i] = xr >= 0 && xr < Win ? (xr * cin + 4 * (lane & 3)) * 4 : 0x7ffffff0u;
    oo[i] = lx >= 1 && lx <= CR_COLS && x < Win && n < p.N ? ((UP ? 2 * x : x) * (int)p.ldc + n) * 4 : 0x7fff0000u;
  }
  f32x4 raw[AHEAD][2][2];  // slot d: the next step d, d + AHEAD, ... of a row (nst % AHEAD == 0)
  auto load = [&](int y, int st, f32x4 (&v)[2][2]) __attribute__((always_inline)) {
    const int so = (min(max(y, 0), Hin - 1) * Win * cin + 32 * st) * 4;
#pragma unroll
    for (int i = 0; i < 2; i++) {
      v[i][0] = cr_load(rx, xo[i], so);
      v[i][1] = cr_load(rx, xo[i], so + 64);
    }
  };
  const char* wl = lds + (g * 64 + lane) * 16;
  // pixel a, channel group b of a tile at slot 4 a + (b ^ (a / 4)): both sides' accesses are conflict-free
  char* const px = lds + CR_LDS + wave * CR_WLDS;
  char* const pw = px + 16 * (4 * (lane >> 2) + ((lane & 3) ^ (lane >> 4)));
  const char* const pr = px + 16 * (4 * l16 + (lg ^ (l16 >> 2)));
  f32x4 bias = {};
  if (p.bias && n < p.N)
#pragma unroll
    for (int r = 0; r < 4; r++) bias[r] = p.bias[n + r];
  const unsigned row_bytes = p.W * (int)p.ldc * 4;  // of the output

  // UP: the row's products P, and the previous row's S[0] and S[0] + S[1] ([tile][even, odd]).
  // Plain: P[3 ty + tx] are the column accumulators of output row y + 1 - ty.
  f32x4 P[9][2], c0[2][2] = {}, c01[2][2] = {};
#pragma unroll
  for (int k = 0; k < 9; k++) P[k][0] = P[k][1] = f32x4{};
#pragma unroll
  for (int d = 0; d < AHEAD; d++) load(y0 - 1, d, raw[d]);
  for (int y = y0 - 1; y <= y1; y++) {
    f32x4 res[2] = {};
    if (!UP && p.resid && y > y0)
#pragma unroll
      for (int i = 0; i < 2; i++) res[i] = cr_load(ro, oo[i] + (y - 1) * row_bytes, 0);
    if (y >= 0 && y < Hin) {
      for (int st = 0; st < nst; st += AHEAD)
#pragma unroll
        for (int d = 0; d < AHEAD; d++) {
          bf16x8 hi[2], lo[2];
#pragma unroll
          for (int i = 0; i < 2; i++) {
            cr_split<SPLIT>(raw[d][i], hi[i], lo[i]);
            *(bf16x8*)(pw + 1024 * i) = hi[i];
            if constexpr (SPLIT) *(bf16x8*)(pw + 2048 + 1024 * i) = lo[i];
          }
          cr_order();
#pragma unroll
          for (int i = 0; i < 2; i++) {
            hi[i] = *(const bf16x8*)(pr + 1024 * i);
            if constexpr (SPLIT) lo[i] = *(const bf16x8*)(pr + 2048 + 1024 * i);
          }
          cr_order();
          if (st + d + AHEAD < nst) load(y, st + d + AHEAD, raw[d]);
          else load(y + 1, d, raw[d]);
          const char* ws = wl + (st + d) * (9 * NG * 1024);
          // three taps at a time, so that a product and the next one on its accumulator are six apart
#pragma unroll
          for (int ty = 0; ty < 3; ty++) {
            bf16x8 w[3];
#pragma unroll
            for (int tx = 0; tx < 3; tx++) w[tx] = *(const bf16x8*)(ws + (3 * ty + tx) * (NG * 1024));
#pragma unroll
            for (int q = 0; q < 6; q++)
              P[3 * ty + q / 2][q & 1] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[q / 2], hi[q & 1], P[3 * ty + q / 2][q & 1], 0, 0, 0);
            if constexpr (SPLIT)
#pragma unroll
              for (int q = 0; q < 6; q++)
                P[3 * ty + q / 2][q & 1] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[q / 2], lo[q & 1], P[3 * ty + q / 2][q & 1], 0, 0, 0);
          }
        }
    } else {
#pragma unroll
      for (int d = 0; d < AHEAD; d++) load(y + 1, d, raw[d]);
    }
    if constexpr (!UP) {
      if (y > y0) {  // output row y - 1
        f32x4 o[2];
#pragma unroll
        for (int r = 0; r < 4; r++) {
          const float a0 = P[6][0][r], a1 = P[6][1][r], b0 = P[8][0][r], b1 = P[8][1][r];
          o[0][r] = (cr_dpp(0.0f, a0, false) + P[7][0][r]) + cr_dpp(cr_ror(b1, true), b0, true);
          o[1][r] = (cr_dpp(cr_ror(a0, false), a1, false) + P[7][1][r]) + cr_dpp(0.0f, b1, true);
        }
#pragma unroll
        for (int i = 0; i < 2; i++) cr_store(ro, oo[i] + (y - 1) * row_bytes, res[i] + (o[i] + bias));
      }
#pragma unroll
      for (int k = 8; k >= 3; k--) P[k][0] = P[k - 3][0], P[k][1] = P[k - 3][1];
#pragma unroll
      for (int k = 0; k < 3; k++) P[k][0] = P[k][1] = f32x4{};
    } else {
      // S of one kernel row: [tile][even, odd].  Rows 2, 1, 0 in turn, so that each row's products are
      // dead before the next row's sums are formed.
      const auto sums = [&](int ty, f32x4 (&S)[2][2]) __attribute__((always_inline)) {
#pragma unroll
        for (int r = 0; r < 4; r++) {
          const float l0 = P[3 * ty][0][r], l1 = P[3 * ty][1][r], r0 = P[3 * ty + 2][0][r], r1 = P[3 * ty + 2][1][r];
          const float m0 = P[3 * ty + 1][0][r], m1 = P[3 * ty + 1][1][r];
          const float left0 = cr_dpp(0.0f, l0, false), left1 = cr_dpp(cr_ror(l0, false), l1, false);
          const float right0 = cr_dpp(cr_ror(r1, true), r0, true), right1 = cr_dpp(0.0f, r1, true);
          S[0][0][r] = left0 + (m0 + r0);
          S[0][1][r] = (l0 + m0) + right0;
          S[1][0][r] = left1 + (m1 + r1);
          S[1][1][r] = (l1 + m1) + right1;
        }
      };
      const auto put = [&](int i, int e, int row, f32x4 v) __attribute__((always_inline)) {
        const unsigned vo = oo[i] + row * row_bytes + e * (int)p.ldc * 4;
        v = v + bias;
        if (p.resid) v = cr_load(ro, vo, 0) + v;
        cr_store(ro, vo, v);
      };
      f32x4 S2[2][2], S1[2][2];
      sums(2, S2);
      if (y > y0)  // the odd row of y - 1
#pragma unroll
        for (int i = 0; i < 2; i++)
#pragma unroll
          for (int e = 0; e < 2; e++) put(i, e, 2 * y - 1, c01[i][e] + S2[i][e]);
      __builtin_amdgcn_sched_barrier(0);
      sums(1, S1);
      if (y >= y0 && y < y1)
#pragma unroll
        for (int i = 0; i < 2; i++)
#pragma unroll
          for (int e = 0; e < 2; e++) put(i, e, 2 * y, c0[i][e] + (S1[i][e] + S2[i][e]));
      __builtin_amdgcn_sched_barrier(0);
      sums(0, c0);
#pragma unroll
      for (int i = 0; i < 2; i++)
#pragma unroll
        for (int e = 0; e < 2; e++) c01[i][e] = c0[i][e] + S1[i][e];
#pragma unroll
      for (int k = 0; k < 9; k++) P[k][0] = P[k][1] = f32x4{};
    }
  }
}

static bool al16(const void* p) { return ((uintptr_t)p & 15) == 0; }

// Rows per strip of conv3x3_rows_kernel: an XCD's workgroups run in rounds of one per CU, and each
// takes R + 2 rows' products; R with the smallest cost, rounds * (R + 2).
struct ConvStrip {
  int R;
  int64_t cost;
};
static ConvStrip conv3x3_rows_strip(int num_cus, int64_t cols, int Hin, int ncg, int tpw) {
  const int64_t cus = num_cus >= 8 ? num_cus / 8 : 1;
  ConvStrip best{1, -1};
  for (int r = 1; r <= 256 && r <= Hin; r++) {
    const int64_t ntg = (cols * ((Hin + r - 1) / r) + tpw - 1) / tpw, wgs = (ntg + 7) / 8 * ncg, cost = (wgs + cus - 1) / cus * (r + 2);
    if (best.cost < 0 || cost <= best.cost) best = {r, cost};
  }
  return best;
}

// Whether the conv by rows (bn output channels per workgroup) is the shorter kernel.  It nearly always is; by measured
// time per 32 input channels (us, fp32 / bf16 precision) it is not
//   * on spatial tiles' sizes with more than 192 input channels, where half of its waves hold the same pixels: rows
//     0.97 / 0.49 per unit of cost; tiles 11 + 4 / 7.6 + 2.8 times the share of the CUs in use, per round
//     (384 channels fp32 256 x 256 426 us and 376, 256 x 128 253 and 180, 128 x 128 130 and 152);
//   * on images of up to 8 columns, where most of a wave's 32 are empty: the implicit GEMM's 128 x 128 tiles
//     (4096 x 1 pixels, 384 channels fp32 512 us and 124).
static bool conv3x3_rows_shorter(int num_cus, const anima_conv_desc* d, bool split, int bn, int64_t cost) {
  const float k = (float)(d->cin / 32), cus = (float)num_cus;
  if (d->cout % 96 == 0 && d->H % CT_TH == 0 && d->W % CT_TW == 0) {
    if (d->up || bn != 16) return true;
    const int64_t n = (int64_t)d->B * (d->H / CT_TH) * (d->W / CT_TW) * (d->cout / 96), q = n / num_cus, rest = n % num_cus;
    const float a = split ? 11.0f : 7.6f, b = split ? 4.0f : 2.8f;
    return (split ? 0.97f : 0.49f) * (float)cost <= (float)q * (a + b) + (rest ? a + b * (float)rest / cus : 0.0f);
  }
  if ((d->up ? d->W / 2 : d->W) > 8) return true;
  const int64_t n = (((int64_t)d->B * d->H * d->W + TG_BM - 1) / TG_BM) * ((d->cout + TG_BN - 1) / TG_BN), slots = (int64_t)num_cus * (split ? 2 : 4);
  const int64_t q = n / slots, rest = n % slots;
  const float gemm = (split ? 16.0f : 18.0f) * (float)q + (rest ? (split ? 8.8f : 7.0f) + (split ? 2.0f : 2.5f) * (float)rest / cus : 0.0f);
  const float row = bn == 32 ? (d->up ? (split ? 1.2f : 0.85f) : (split ? 0.97f : 0.63f)) : (d->up ? (split ? 0.87f : 0.61f) : (split ? 0.85f : 0.53f));
  return 0.85f * (3.0f + row * (float)cost * k) <= 10.0f + gemm * k;
}

int conv3x3_launch(anima_ctx* c, const anima_conv_desc* d) {
  if (!d) return fail(c, ANIMA_E_ARG, "anima_conv3x3: null descriptor");
  if (!d->x || !d->w || !d->out) return fail(c, ANIMA_E_ARG, "anima_conv3x3: null x / w / out");
  if (d->B < 1 || d->H < 1 || d->W < 1 || d->cin < 1 || d->cout < 1)
    return fail(c, ANIMA_E_ARG, "anima_conv3x3: B=%d H=%d W=%d cin=%d cout=%d", d->B, d->H, d->W, d->cin, d->cout);
  if (d->cin % 16) return fail(c, ANIMA_E_UNSUPPORTED, "anima_conv3x3: cin=%d (this build needs cin %% 16 == 0)", d->cin);
  if (d->up && (d->H % 2 || d->W % 2)) return fail(c, ANIMA_E_ARG, "anima_conv3x3: up needs an even output size (H=%d W=%d)", d->H, d->W);
  if (d->precision != ANIMA_PREC_BF16 && d->precision != ANIMA_PREC_FP32)
    return fail(c, ANIMA_E_ARG, "anima_conv3x3: unknown precision %d", d->precision);
  if (!al16(d->x) || !al16(d->w)) return fail(c, ANIMA_E_ARG, "anima_conv3x3: x and w must be 16-byte aligned");
  const int64_t M = (int64_t)d->B * d->H * d->W;
  if (M > 0x7fffffffLL - TG_BM) return fail(c, ANIMA_E_ARG, "anima_conv3x3: %lld output pixels", (long long)M);
  TGemmArgs p{};
  p.a = d->x;
  p.cin = d->cin;
  p.H = d->H;
  p.W = d->W;
  p.up = d->up ? 1 : 0;
  p.b = d->w;
  p.ldb = 9LL * d->cin;
  p.c = d->out;
  p.ldc = d->cout;
  p.bias = d->bias;
  p.alpha = 1.0f;
  p.act = ANIMA_ACT_NONE;
  p.resid = d->resid ? 1 : 0;
  p.M = (int)M;
  p.N = d->cout;
  p.K = 9 * d->cin;
  const bool split = d->precision == ANIMA_PREC_FP32;
  // conv by rows: weights of 32 (or 16) output channels in LDS, 16-byte stores of four channels, 32-bit
  // offsets into an image
  const int Hin = d->up ? d->H / 2 : d->H, Win = d->up ? d->W / 2 : d->W;
  const int64_t in_bytes = (int64_t)Hin * Win * d->cin * 4, out_bytes = (int64_t)d->H * d->W * d->cout * 4;
  if (d->cin % 32 == 0 && d->cin * 16 <= CR_MAXK && d->cout % 4 == 0 && d->cout <= 4096 && al16(d->out) &&
      in_bytes < (1LL << 31) - 65536 && out_bytes < (1LL << 31) - 65536) {
    const int bn = d->cin * 32 <= CR_MAXK && d->cout > 16 ? 32 : 16, tpw = 8 / (bn / 16);
    const int ncol = (Win + CR_COLS - 1) / CR_COLS, ncg = (d->cout + bn - 1) / bn;
    const auto [R, cost] = conv3x3_rows_strip(c->num_cus, (int64_t)d->B * ncol, Hin, ncg, tpw);
    const int nstrip = (Hin + R - 1) / R;
    const int64_t ntask = (int64_t)d->B * ncol * nstrip, ntg = (ntask + tpw - 1) / tpw, blocks = (ntg + 7) / 8 * 8 * ncg;
    if (ntask <= 0x7ffffff && blocks <= 0x7fffffff && conv3x3_rows_shorter(c->num_cus, d, split, bn, cost)) {
      const dim3 grid((unsigned)blocks);
      // (an upsampling conv takes its products at the input's resolution)
      Launch L(c, d->up ? "conv3x3.up.rows" : "conv3x3.rows", 2.0 * d->B * Hin * Win * d->cout * 9.0 * d->cin, 0.0);
#define CRA(U, S, BN, A) hipLaunchKernelGGL((conv3x3_rows_kernel<U, S, BN, A>), grid, dim3(512), 0, c->stream, p, R, ncol, nstrip, ncg, (int)ntask)
#define CRB(U, S, BN)                     \
  {                                       \
    if (d->cin % 96 == 0) CRA(U, S, BN, 3); \
    else CRA(U, S, BN, 1);                \
  }
#define CRU(S, BN)              \
  {                             \
    if (d->up) CRB(true, S, BN) \
    else CRB(false, S, BN)      \
  }
      if (bn == 32) {
        if (split) CRU(true, 32)
        else CRU(false, 32)
      } else {
        if (split) CRU(true, 16)
        else CRU(false, 16)
      }
#undef CRU
#undef CRB
#undef CRA
      return L.end();
    }
  }
  const int bn = d->cout % 96 == 0 ? 96 : d->cout <= 32 ? 32 : 0;  // 96-channel tiles, or one 32-wide tile
  if (bn && d->cin % CT_CC == 0 && d->H % CT_TH == 0 && d->W % CT_TW == 0 &&
      (int64_t)d->B * (d->H / CT_TH) * (d->W / CT_TW) <= 0x7fffffff && (d->cout + bn - 1) / bn <= 65535) {
    // spatial tiles with the input halo in LDS
    const dim3 grid((unsigned)((int64_t)d->B * (d->H / CT_TH) * (d->W / CT_TW)), (unsigned)((d->cout + bn - 1) / bn));
    Launch L(c, d->up ? "conv3x3.up.tile" : "conv3x3.tile", 2.0 * M * d->cout * 9.0 * d->cin, 0.0);
#define CTL(S, BN) hipLaunchKernelGGL((conv3x3_tile_kernel<S, CT_NW, BN>), grid, dim3(64 * CT_NW), 0, c->stream, p)
    if (bn == 96) {
      if (split) CTL(true, 96);
      else CTL(false, 96);
    } else {
      if (split) CTL(true, 32);
      else CTL(false, 32);
    }
#undef CTL
    return L.end();
  }
  return tgemm_launch(c, p, TG_A_CONV, TG_B_W16, split, 1, d->up ? "conv3x3.up" : "conv3x3",
                      2.0 * M * d->cout * 9.0 * d->cin);
}

// ---- channel norm: one wave per row; lane t sums x[c]^2 over c = t, t + 64, ... in order, then the
// 32 .. 1 tree of the shader's shared-memory reduction (kernels.js:78-79).
__global__ __launch_bounds__(256) void channel_norm_kernel(const float* X, const float* G, float* Y, int64_t rows, int cols,
                                                           int silu) {
  const int lane = threadIdx.x & 63;
  const int64_t row = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (row >= rows) return;
  const float* x = X + row * cols;
  float ss = 0.0f;
  for (int c = lane; c < cols; c += 64) ss += x[c] * x[c];
  ss = tree_sum_down(ss, 64);
  const float r = sqrtf((float)cols) / fmaxf(sqrtf(__shfl(ss, 0)), 1e-12f);
  float* y = Y + row * cols;
  for (int c = lane; c < cols; c += 64) {
    float v = x[c] * r * G[c];
    if (silu) v = silu_f(v);
    y[c] = v;
  }
}

// The same per-row arithmetic for rows of at most 64 NV channels, CN_RPW rows per wave with every
// load of the wave issued first: one row per wave kept too few bytes in flight (a row of 96
// channels is 384 bytes) and left the pass at a third of the HBM rate.  Channels past cols read as
// zero, which adds nothing to a lane's sum (0 + x^2 and x^2 + 0 are exact).
constexpr int CN_RPW = 8;
template <int NV>
__global__ __launch_bounds__(256) void channel_norm_rows_kernel(const float* X, const float* G, float* Y, int64_t rows,
                                                                int cols, int silu) {
  const int lane = threadIdx.x & 63;
  const int64_t row0 = ((int64_t)blockIdx.x * 4 + (threadIdx.x >> 6)) * CN_RPW;
  float xv[CN_RPW][NV], g[NV];
#pragma unroll
  for (int v = 0; v < NV; v++) {
    const int c = lane + 64 * v;
    g[v] = c < cols ? G[c] : 0.0f;
  }
#pragma unroll
  for (int r = 0; r < CN_RPW; r++)
#pragma unroll
    for (int v = 0; v < NV; v++) {
      const int c = lane + 64 * v;
      xv[r][v] = row0 + r < rows && c < cols ? X[(row0 + r) * cols + c] : 0.0f;
    }
#pragma unroll
  for (int r = 0; r < CN_RPW; r++) {
    if (row0 + r >= rows) break;  // uniform across the wave
    float ss = 0.0f;
#pragma unroll
    for (int v = 0; v < NV; v++) ss += xv[r][v] * xv[r][v];
    ss = tree_sum_down(ss, 64);
    const float rn = sqrtf((float)cols) / fmaxf(sqrtf(__shfl(ss, 0)), 1e-12f);
    float* y = Y + (row0 + r) * cols;
#pragma unroll
    for (int v = 0; v < NV; v++) {
      const int c = lane + 64 * v;
      float o = xv[r][v] * rn * g[v];
      if (silu) o = silu_f(o);
      if (c < cols) y[c] = o;
    }
  }
}

int channel_norm_launch(anima_ctx* c, const float* x, const float* gamma, float* y, int64_t rows, int cols, int silu) {
  if (!x || !gamma || !y) return fail(c, ANIMA_E_ARG, "anima_channel_norm: null pointer");
  if (rows < 0 || cols < 1) return fail(c, ANIMA_E_ARG, "anima_channel_norm: rows=%lld cols=%d", (long long)rows, cols);
  if (rows == 0) return ANIMA_OK;
  Launch lc(c, "vae.channel_norm", 0.0, (double)rows * cols * 8);
  const unsigned gr = (unsigned)((rows + 4 * CN_RPW - 1) / (4 * CN_RPW));
  const int sl = silu ? 1 : 0;
  if (cols <= 128) hipLaunchKernelGGL(channel_norm_rows_kernel<2>, dim3(gr), dim3(256), 0, c->stream, x, gamma, y, rows, cols, sl);
  else if (cols <= 192) hipLaunchKernelGGL(channel_norm_rows_kernel<3>, dim3(gr), dim3(256), 0, c->stream, x, gamma, y, rows, cols, sl);
  else if (cols <= 384) hipLaunchKernelGGL(channel_norm_rows_kernel<6>, dim3(gr), dim3(256), 0, c->stream, x, gamma, y, rows, cols, sl);
  else
    hipLaunchKernelGGL(channel_norm_kernel, dim3((unsigned)((rows + 3) / 4)), dim3(256), 0, c->stream, x, gamma, y, rows,
                       cols, sl);
  return lc.end();
}

// ---- the decoder's output image (app/models/vae.js:104-112): RGBA bytes of [n][3] values,
// channel = round((clamp(v, -1, 1) + 1) / 2 * 255) in double precision with JS Math.round
// (nearest, ties toward +inf; t - floor(t) is exact in double), NaN -> 0 as the reference's
// Uint8ClampedArray store makes it, alpha 255.
__global__ __launch_bounds__(256) void rgba_kernel(const float* x, int64_t n, uint8_t* out) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= n) return;
  uchar4 o;
  unsigned char c[3];
#pragma unroll
  for (int j = 0; j < 3; j++) {
    const float xv = x[3 * i + j];
    const double v = (fmin(1.0, fmax(-1.0, (double)xv)) + 1.0) / 2.0;
    const double t = v * 255.0;
    double r = floor(t);
    if (t - r >= 0.5) r += 1.0;
    c[j] = xv != xv ? 0 : (unsigned char)r;
  }
  o.x = c[0];
  o.y = c[1];
  o.z = c[2];
  o.w = 255;
  ((uchar4*)out)[i] = o;
}

int to_rgba_launch(anima_ctx* c, const float* x, int64_t n, uint8_t* out) {
  if (!x || !out || n < 0) return fail(c, ANIMA_E_ARG, "anima_to_rgba: bad arguments");
  if (((uintptr_t)out & 3) != 0) return fail(c, ANIMA_E_ARG, "anima_to_rgba: out must be 4-byte aligned");
  if (n == 0) return ANIMA_OK;
  Launch l(c, "vae.to_rgba", 0.0, (double)n * 16);
  hipLaunchKernelGGL(rgba_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, c->stream, x, n, out);
  return l.end();
}

// ---- attention on the chunked path (head dims other than 64 / 128)

// In place on row r of S (row stride ld), columns [0, cols): e = exp(s * scale - m), m the maximum of
// s * scale over the row's first `lim` columns, 0 past them; rl[r] = 1 / sum of e (the P.V
// product's row scale).  lim = valid, or with the causal mask (app/gpu/kernels.js:49,
// limit = min(cols, row + 1)) min(valid, q + 1) for the row's query index q = row0 + r.  One
// workgroup per row.
__global__ __launch_bounds__(256) void chunk_softmax_kernel(float* S, int64_t ld, float* rl, int cols, int valid,
                                                            float scale, int row0, int causal) {
  __shared__ float red[4];
  float* s = S + (int64_t)blockIdx.x * ld;
  const int t = threadIdx.x, wave = t >> 6, lane = t & 63;
  const int lim = causal ? min(valid, row0 + (int)blockIdx.x + 1) : valid;
  float mx = -INFINITY;
  for (int c = t; c < lim; c += 256) mx = fmaxf(mx, s[c] * scale);
  mx = wave_max(mx);
  if (lane == 0) red[wave] = mx;
  __syncthreads();
  mx = fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
  __syncthreads();
  float sum = 0.0f;
  for (int c = t; c < cols; c += 256) {
    const float e = c < lim ? expf(s[c] * scale - mx) : 0.0f;
    s[c] = e;
    sum += e;
  }
  sum = wave_sum(sum);
  if (lane == 0) red[wave] = sum;
  __syncthreads();
  if (t == 0) rl[blockIdx.x] = 1.0f / ((red[0] + red[1]) + (red[2] + red[3]));
}

// The same row softmax with the row held in registers (NPT values per thread, columns t + 256 i):
// one read and one write of the score row instead of two reads and a write; the maximum, the
// exponentials and the sums are taken in the same order as chunk_softmax_kernel (bit-identical).
template <int NPT>
__global__ __launch_bounds__(256) void chunk_softmax_reg_kernel(float* S, int64_t ld, float* rl, int cols, int valid,
                                                                float scale, int row0, int causal) {
  __shared__ float red[4];
  float* s = S + (int64_t)blockIdx.x * ld;
  const int t = threadIdx.x, wave = t >> 6, lane = t & 63;
  const int lim = causal ? min(valid, row0 + (int)blockIdx.x + 1) : valid;
  float v[NPT];
#pragma unroll
  for (int i = 0; i < NPT; i++) {
    const int c = t + 256 * i;
    v[i] = c < cols ? s[c] : 0.0f;
  }
  float mx = -INFINITY;
#pragma unroll
  for (int i = 0; i < NPT; i++)
    if (t + 256 * i < lim) mx = fmaxf(mx, v[i] * scale);
  mx = wave_max(mx);
  if (lane == 0) red[wave] = mx;
  __syncthreads();
  mx = fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
  __syncthreads();
  float sum = 0.0f;
#pragma unroll
  for (int i = 0; i < NPT; i++) {
    const int c = t + 256 * i;
    if (c < cols) {
      const float e = c < lim ? expf(v[i] * scale - mx) : 0.0f;
      s[c] = e;
      sum += e;
    }
  }
  sum = wave_sum(sum);
  if (lane == 0) red[wave] = sum;
  __syncthreads();
  if (t == 0) rl[blockIdx.x] = 1.0f / ((red[0] + red[1]) + (red[2] + red[3]));
}

// dst[d * ldd + j] = src[j * ld + d] for j < L, d < D (V -> V^T for the P.V product's B operand).
__global__ __launch_bounds__(256) void transpose_kernel(const float* src, int64_t ld, int L, int D, float* dst, int64_t ldd) {
  __shared__ float tile[32][33];
  const int j0 = blockIdx.x * 32, d0 = blockIdx.y * 32;
  const int tx = threadIdx.x & 31, ty = threadIdx.x >> 5;
  for (int r = ty; r < 32; r += 8) {
    const int j = j0 + r, d = d0 + tx;
    tile[r][tx] = j < L && d < D ? src[(int64_t)j * ld + d] : 0.0f;
  }
  __syncthreads();
  for (int r = ty; r < 32; r += 8) {
    const int d = d0 + r, j = j0 + tx;
    if (d < D && j < L) dst[(int64_t)d * ldd + j] = tile[tx][r];
  }
}

// Checks of the chunked path: plain attention (no fused norm / RoPE, no prepared K/V; causal mask
// allowed) with 16-byte aligned rows, D % 4 == 0.
int attention_chunked_check(anima_ctx* c, const anima_attn_desc* d) {
  if (d->D < 4 || d->D % 4 || d->D > 4096)
    return fail(c, ANIMA_E_UNSUPPORTED, "anima_attention: head dim %d (the chunked path takes D %% 4 == 0, D <= 4096)", d->D);
  if (d->q_norm || d->k_norm || d->rope_cs || d->kv_prep)
    return fail(c, ANIMA_E_UNSUPPORTED, "anima_attention: head dim %d takes no fused norm / RoPE or prepared K/V", d->D);
  if (d->precision != ANIMA_PREC_BF16 && d->precision != ANIMA_PREC_FP32)
    return fail(c, ANIMA_E_ARG, "anima_attention: unknown precision %d", d->precision);
  const int group = d->group <= 0 ? 1 : d->group;
  if (d->B < 1 || d->Lq < 1 || d->Lk < 1 || d->H < 1 || d->H % group)
    return fail(c, ANIMA_E_ARG, "anima_attention: B=%d Lq=%d Lk=%d H=%d group=%d", d->B, d->Lq, d->Lk, d->H, group);
  if (!d->q || !d->k || !d->v || !d->o) return fail(c, ANIMA_E_ARG, "anima_attention: null q/k/v/o");
  const int64_t lds[4] = {d->ldq, d->ldk, d->ldv, d->ldo}, offs[4] = {d->q_off, d->k_off, d->v_off, d->o_off},
                bss[4] = {d->q_bstride, d->k_bstride, d->v_bstride, d->o_bstride};
  const int heads[4] = {d->H, d->H / group, d->H / group, d->H};
  const char* nm[4] = {"q", "k", "v", "o"};
  for (int i = 0; i < 4; i++) {
    if (lds[i] % 4 || offs[i] % 4 || bss[i] % 4 || lds[i] < 0 || offs[i] < 0 || bss[i] < 0)
      return fail(c, ANIMA_E_ARG, "anima_attention: %s ld/off/bstride must be non-negative multiples of 4", nm[i]);
    if (lds[i] < offs[i] + (int64_t)heads[i] * d->D)
      return fail(c, ANIMA_E_ARG, "anima_attention: %s rows of %lld elements cannot hold off %lld + %d heads x %d", nm[i],
                  (long long)lds[i], (long long)offs[i], heads[i], d->D);
  }
  if (!al16(d->q) || !al16(d->k) || !al16(d->v) || !al16(d->o))
    return fail(c, ANIMA_E_ARG, "anima_attention: q/k/v/o must be 16-byte aligned");
  return ANIMA_OK;
}

// Key ranges of the chunked P.V product: 1 unless its grid has fewer than 1024 tiles; then up to
// 8 ranges of at least 1024 keys, each a multiple of the 32-key k-tile (so a range never reads past
// the valid keys).
static int pv_splits(int rows, int D, int valid) {
  const int64_t tiles = (int64_t)((rows + TG_BM - 1) / TG_BM) * ((D + TG_BN - 1) / TG_BN);
  int ks = 1;
  while (ks < 8 && tiles * ks < 1024 && valid % (2 * ks * TG_BK) == 0 && valid / (2 * ks) >= 1024) ks *= 2;
  return ks;
}

// o[m][d] = (sum over the key ranges of part[z][m][d]) * rl[m]
__global__ __launch_bounds__(256) void pv_sum_kernel(const float* part, int ks, int rows, int D, const float* rl, float* o,
                                                     int64_t ldo) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  const int64_t n = (int64_t)rows * D;
  if (i >= n) return;
  float acc = part[i];
  for (int z = 1; z < ks; z++) acc = acc + part[(int64_t)z * n + i];
  const int64_t m = i / D;
  o[m * ldo + (i - m * D)] = acc * rl[m];
}

// ---- attention of 384-dim heads (the VAE decoder's single head over all latent positions), fused
//
// The chunked path writes the score matrix (1 GiB at 128 x 128 latents), reads and rewrites it for the
// softmax and reads it again; here scores live in registers.  Bound by the matrix cores (with SPLIT
// three bf16 products per score and per output, as on the chunked path: hi.hi + lo.hi + hi.lo).  A
// pass first writes K and V as bf16 planes in MFMA fragment order, per block of 32 keys: K as
// [16-dim step][plane][lane][8 dims], V^T as [32-dim tile][16-key step][plane][lane][8 keys], 1 KiB
// per fragment, so that the main loop's copies and LDS reads are linear.  A workgroup is 128 queries,
// 8 waves: waves w and w + 4 share 32 queries and split the 384 dims (queries, and outputs, of 192 dims
// take 96 registers each with SPLIT; all 384 in one wave per SIMD spilled and overlapped nothing).
// Each takes half of the score products; the halves are exchanged through LDS.  A block's weights are
// formed beside the next block's score products.  K and V go through one LDS slot each, copied one
// phase ahead.  Scores are computed transposed (a lane holds one query's keys), so a row's softmax
// needs one lane exchange, and its weights are the next product's operand as they stand (V^T's keys
// are stored in that order: 0-3, 8-11, 4-7, 12-15 of each 16).  Queries too few for the CUs split the
// keys, partial outputs (unnormalized, with the row's maximum and sum) combined afterwards.
// Against the chunked path: 128 x 128 latents fp32 2645 -> 1075 us (this kernel 1055, 1173 TFLOP/s of the three
// products; a large library product reaches 1250), bf16 2000 -> 490; 64 x 64 193 -> 117 / 159 -> 76; 32 x 32 115 -> 60
// / 87 -> 44.
constexpr int FA_D = 384, FA_KB = 32, FA_Q = 128, FA_NS = FA_D / 16, FA_NT = FA_D / 32, FA_MAXB = 64;

struct FaArgs {
  const float *q, *k, *v;
  float* o;
  int64_t ldq, ldk, ldv, ldo, qbs, kbs, vbs, obs;  // rows, batch strides (offsets applied)
  char* kv;       // prepared blocks [B][Hkv][nkb][K, V]
  float* part;    // partial outputs [item][split][128][384], then (maximum, sum) [item][split][128][2]
  float* ml;
  int64_t kv_head;  // bytes of one (batch, kv head) of kv
  int Lq, H, group, nkb, nqt, splits, per;  // per: key blocks per split
  float c;          // scale * log2(e)
  int valid[FA_MAXB];
};

// bf16 hi (and the rest lo) of 8 values
template <bool SPLIT>
__device__ __forceinline__ void fa_split(const float (&v)[8], bf16x8& hi, bf16x8& lo) {
  cr_split<SPLIT>({f32x4{v[0], v[1], v[2], v[3]}, f32x4{v[4], v[5], v[6], v[7]}}, hi, lo);
}

// One block of 32 keys of one kv head: K and V rows to fragments (keys past the valid ones as zeros).
template <bool SPLIT>
__global__ __launch_bounds__(256) void attn384_prep_kernel(FaArgs a) {
  constexpr int NP = SPLIT ? 2 : 1;
  __shared__ float vs[FA_KB][FA_D + 1];
  const int t = threadIdx.x, kb = blockIdx.x, hk = blockIdx.y, b = blockIdx.z, k0 = kb * FA_KB;
  const int nv = min(FA_KB, a.valid[b] - k0);  // may be <= 0: a block of zeros
  const float* K = a.k + (int64_t)b * a.kbs + (int64_t)hk * FA_D;
  const float* V = a.v + (int64_t)b * a.vbs + (int64_t)hk * FA_D;
  char* out = a.kv + ((int64_t)b * gridDim.y + hk) * a.kv_head + (int64_t)kb * (2 * FA_NS * NP * 1024);
  for (int u = t; u < FA_KB * FA_D / 4; u += 256) {
    const int r = u / (FA_D / 4), d = 4 * (u % (FA_D / 4));
    const f32x4 x = r < nv ? *(const f32x4*)(V + (int64_t)(k0 + r) * a.ldv + d) : f32x4{};
#pragma unroll
    for (int e = 0; e < 4; e++) vs[r][d + e] = x[e];
  }
  for (int u = t; u < FA_KB * FA_D / 8; u += 256) {
    const int r = u / (FA_D / 8), pc = u % (FA_D / 8);  // row, piece of 8 dims: step pc / 2, half pc % 2
    f32x4 x[2] = {};
    if (r < nv) {
      const float* src = K + (int64_t)(k0 + r) * a.ldk + 8 * pc;
      x[0] = *(const f32x4*)src;
      x[1] = *(const f32x4*)(src + 4);
    }
    bf16x8 hi, lo;
    cr_split<SPLIT>(x, hi, lo);
    char* dst = out + (pc >> 1) * (NP * 1024) + (r + 32 * (pc & 1)) * 16;
    *(bf16x8*)dst = hi;
    if constexpr (SPLIT) *(bf16x8*)(dst + 1024) = lo;
  }
  __syncthreads();
  out += FA_NS * NP * 1024;
  for (int u = t; u < FA_NT * 2 * 64; u += 256) {
    const int ln = u & 63, f = u >> 6, tile = f >> 1, s2 = f & 1, d = 32 * tile + (ln & 31), hf = ln >> 5;
    float x[8];
#pragma unroll
    for (int j = 0; j < 8; j++) x[j] = vs[16 * s2 + 4 * hf + (j & 3) + 8 * (j >> 2)][d];
    bf16x8 hi, lo;
    fa_split<SPLIT>(x, hi, lo);
    char* dst = out + f * (NP * 1024) + ln * 16;
    *(bf16x8*)dst = hi;
    if constexpr (SPLIT) *(bf16x8*)(dst + 1024) = lo;
  }
}

typedef __attribute__((address_space(3))) void fa_lds_t;
__device__ __forceinline__ void fa_copy(__amdgpu_buffer_rsrc_t r, char* dst, int voff, int soff) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (fa_lds_t*)dst, 16, voff, soff, 0, 0);
}
// this wave's copies have landed and its LDS accesses are done; then every wave's
__device__ __forceinline__ void fa_wait_barrier() {
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_waitcnt(7 << 4);  // vmcnt(0), lgkmcnt(0)
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}

template <bool SPLIT>
__global__ __launch_bounds__(512, 2) void attn384_kernel(FaArgs a, int nitem) {
  constexpr int NP = SPLIT ? 2 : 1, TB = FA_NS * NP * 1024, CPW = TB / 8192;  // bytes of a K (V) block; copies per wave
  constexpr int HS = FA_NS / 2, HT = FA_NT / 2;                              // 16-dim steps, 32-dim tiles of a wave
  __shared__ __attribute__((aligned(1024))) char smem[2 * TB + 2 * 8 * 4096];
  const int t = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(t >> 6), lane = t & 63, lq = lane & 31, hf = lane >> 5;
  const int u = wave >> 2;  // dims 192 u .. + 191 of the queries of wave % 4
  // items [batch, head][split][query tile]: an XCD's contiguous range shares K / V streams in its L2
  const int it = xcd_remap(blockIdx.x, nitem);
  const int bh = it / (a.splits * a.nqt), rem = it - bh * a.splits * a.nqt, sp = rem / a.nqt, qt = rem - sp * a.nqt;
  const int b = bh / a.H, h = bh - b * a.H;
  const int valid = a.valid[b], nkb = (valid + FA_KB - 1) / FA_KB;
  const int kb0 = sp * a.per, nb = min(a.per, nkb - kb0);  // may be <= 0 for a shorter batch element
  const int row = qt * FA_Q + 32 * (wave & 3) + lq;

  f32x16 O[HT];
#pragma unroll
  for (int i = 0; i < HT; i++) O[i] = f32x16{};
  // mf: m, or 0 while no score was finite: weights of zero then (as they are beside the finite scores of other blocks)
  float m = -INFINITY, mf = 0.0f, l = 0.0f;

  if (nb > 0) {
    const char* src = a.kv + ((int64_t)b * (a.H / a.group) + h / a.group) * a.kv_head + (int64_t)kb0 * (2 * TB);
    const __amdgpu_buffer_rsrc_t rk = __builtin_amdgcn_make_buffer_rsrc((void*)src, (short)0, 2 * nb * TB, 0x00020000);
    // K blocks go through the first slot, V blocks through the second; block 2 j (+ 1) of the stream
    auto issue = [&](int blk) __attribute__((always_inline)) {
      char* dst = smem + (blk & 1) * TB + wave * (CPW * 1024);
#pragma unroll
      for (int c = 0; c < CPW; c++) fa_copy(rk, dst + c * 1024, (wave * CPW + c) * 1024 + lane * 16, blk * TB);
    };
    issue(0);
    bf16x8 qh[HS], ql[SPLIT ? HS : 1];
    {
      const float* Q = a.q + (int64_t)b * a.qbs + (int64_t)min(row, a.Lq - 1) * a.ldq + (int64_t)h * FA_D + 192 * u + 8 * hf;
#pragma unroll
      for (int s = 0; s < HS; s++) {
        const f32x4 x[2] = {*(const f32x4*)(Q + 16 * s), *(const f32x4*)(Q + 16 * s + 4)};
        bf16x8 lo;
        cr_split<SPLIT>(x, qh[s], lo);
        if constexpr (SPLIT) ql[s] = lo;
      }
    }
    const char* const kp = smem + u * (HS * NP * 1024) + lane * 16;
    const char* const vp = smem + TB + u * (2 * HT * NP * 1024) + lane * 16;
    // this wave's partial scores and its partner's, [quad][lane], of even and odd blocks
    char* const xo = smem + 2 * TB + wave * 4096 + lane * 16;
    const char* const xi = smem + 2 * TB + (wave ^ 4) * 4096 + lane * 16;
    auto scores = [&](f32x16& S) __attribute__((always_inline)) {
#pragma unroll
      for (int s = 0; s < HS; s++) {
        const bf16x8 kh = *(const bf16x8*)(kp + s * (NP * 1024));
        S = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kh, qh[s], S, 0, 0, 0);
        if constexpr (SPLIT) {
          const bf16x8 kl = *(const bf16x8*)(kp + s * (NP * 1024) + 1024);
          S = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kh, ql[s], S, 0, 0, 0);
          S = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kl, qh[s], S, 0, 0, 0);
        }
      }
    };
    auto give = [&](const f32x16& S, int j) __attribute__((always_inline)) {
#pragma unroll
      for (int q = 0; q < 4; q++)
        *(f32x4*)(xo + (j & 1) * 32768 + q * 1024) = f32x4{S[4 * q], S[4 * q + 1], S[4 * q + 2], S[4 * q + 3]};
    };
    fa_wait_barrier();
    f32x16 S = {};
    scores(S);
    give(S, 0);
    fa_wait_barrier();
    if (nb > 1) issue(2);
    for (int j = 0; j < nb; j++) {
      fa_wait_barrier();  // K j + 1 and the scores of j are there; V j - 1 has been read
      issue(2 * j + 1);
      // scores times c, keys past the valid ones out; register r is key 8 (r / 4) + 4 hf + r % 4
      float y[16];
      const int left = valid - (kb0 + j) * FA_KB;
#pragma unroll
      for (int q = 0; q < 4; q++) {
        const f32x4 x = *(const f32x4*)(xi + (j & 1) * 32768 + q * 1024);
#pragma unroll
        for (int e = 0; e < 4; e++) y[4 * q + e] = (S[4 * q + e] + x[e]) * a.c;
      }
      if (left < FA_KB)
#pragma unroll
        for (int r = 0; r < 16; r++) y[r] = 8 * (r >> 2) + 4 * hf + (r & 3) < left ? y[r] : -INFINITY;
      float mx = y[0];
#pragma unroll
      for (int r = 1; r < 16; r++) mx = fmaxf(mx, y[r]);
      mx = fmaxf(mx, __shfl_xor(mx, 32));
      if (__any(mx > m)) {  // (rare once the first blocks are done)
        const float mn = fmaxf(m, mx), al = mx > m ? __builtin_amdgcn_exp2f(m - mn) : 1.0f;  // (m may be -inf still)
        m = mn;
        mf = mn == -INFINITY ? 0.0f : mn;
        l = l * al;
#pragma unroll
        for (int i = 0; i < HT; i++) O[i] = O[i] * al;
      }
      // the next block's scores beside this block's weights (after the last block: of the last again, unused)
      S = f32x16{};
      scores(S);
      bf16x8 ph[2], pl[2];
#pragma unroll
      for (int s2 = 0; s2 < 2; s2++) {
        float e[8];
#pragma unroll
        for (int r = 0; r < 8; r++) {
          e[r] = __builtin_amdgcn_exp2f(y[8 * s2 + r] - mf);
          l += e[r];
        }
        fa_split<SPLIT>(e, ph[s2], pl[s2]);
      }
      give(S, j + 1);
      fa_wait_barrier();  // V j is there; K j + 1 has been read
      if (j + 2 < nb) issue(2 * j + 4);
#pragma unroll
      for (int f = 0; f < 2 * HT; f++) {  // tile f / 2, keys 16 (f % 2) .. + 15
        const bf16x8 vh = *(const bf16x8*)(vp + f * NP * 1024);
        f32x16& o = O[f >> 1];
        o = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vh, ph[f & 1], o, 0, 0, 0);
        if constexpr (SPLIT) {
          const bf16x8 vl = *(const bf16x8*)(vp + f * NP * 1024 + 1024);
          o = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vh, pl[f & 1], o, 0, 0, 0);
          o = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vl, ph[f & 1], o, 0, 0, 0);
        }
      }
    }
  }
  l = l + __shfl_xor(l, 32);
  float* dst;
  float f = 1.0f;
  if (a.splits == 1) {
    if (row >= a.Lq) return;
    dst = a.o + (int64_t)b * a.obs + (int64_t)row * a.ldo + (int64_t)h * FA_D;
    f = 1.0f / l;
  } else {
    const int64_t pr = ((int64_t)bh * a.splits + sp) * a.nqt * FA_Q + row;
    dst = a.part + pr * FA_D;
    if (hf == 0 && u == 0) {
      a.ml[2 * pr] = m;
      a.ml[2 * pr + 1] = l;
    }
  }
#pragma unroll
  for (int i = 0; i < HT; i++)
#pragma unroll
    for (int q = 0; q < 4; q++) {
      const f32x4 v = {O[i][4 * q] * f, O[i][4 * q + 1] * f, O[i][4 * q + 2] * f, O[i][4 * q + 3] * f};
      *(f32x4*)(dst + 192 * u + 32 * i + 8 * q + 4 * hf) = v;
    }
}

// out = sum_z 2^(m_z - M) O_z / sum_z 2^(m_z - M) l_z, M = max m_z: 96 threads (4 dims each) per row.
__global__ __launch_bounds__(192) void attn384_combine_kernel(FaArgs a) {
  const int row = blockIdx.x * 2 + threadIdx.x / 96, d = 4 * (threadIdx.x % 96), bh = blockIdx.y;
  if (row >= a.Lq) return;
  const int64_t st = (int64_t)a.nqt * FA_Q, pr = (int64_t)bh * a.splits * st + row;
  float M = -INFINITY;
  for (int z = 0; z < a.splits; z++) M = fmaxf(M, a.ml[2 * (pr + z * st)]);
  f32x4 acc = {};
  float l = 0.0f;
  for (int z = 0; z < a.splits; z++) {
    const float lz = a.ml[2 * (pr + z * st) + 1];
    if (lz == 0.0f) continue;  // a split past this batch element's keys
    const float w = __builtin_amdgcn_exp2f(a.ml[2 * (pr + z * st)] - M);
    acc = acc + *(const f32x4*)(a.part + (pr + z * st) * FA_D + d) * w;
    l = l + lz * w;
  }
  const int b = bh / a.H, h = bh - b * a.H;
  *(f32x4*)(a.o + (int64_t)b * a.obs + (int64_t)row * a.ldo + (int64_t)h * FA_D + d) = acc * (1.0f / l);
}

// 384-dim heads without a causal mask, where the operands and partial outputs stay below 1 GiB of
// workspace (the chunked path's own bound on scores): returns 1 if launched, 0 if not taken, or an error.
static int attention384_launch(anima_ctx* c, const anima_attn_desc* d, const int* kv_len) {
  if (d->D != FA_D || d->causal || d->B > FA_MAXB) return 0;
  const int group = d->group <= 0 ? 1 : d->group, Hk = d->H / group;
  const bool split = d->precision == ANIMA_PREC_FP32;
  FaArgs a{};
  int vmax = 0;
  for (int b = 0; b < d->B; b++) {
    if (kv_len[b] < 1) return 0;
    a.valid[b] = kv_len[b];
    vmax = std::max(vmax, kv_len[b]);
  }
  a.nkb = (vmax + FA_KB - 1) / FA_KB;
  a.nqt = (d->Lq + FA_Q - 1) / FA_Q;
  const int64_t bh = (int64_t)d->B * d->H, wgs = bh * a.nqt;
  // key splits: rounds of one workgroup per CU times its key blocks (and about three blocks' time of
  // prologue and stores, and each split's share of the combining pass), splits of at least 4 blocks
  int64_t best = -1;
  for (int s = 1; s <= 16 && (s == 1 || a.nkb / s >= 4); s++) {
    const int64_t cost = (wgs * s + c->num_cus - 1) / c->num_cus * ((a.nkb + s - 1) / s + 3) + (s > 1 ? s : 0);
    if (best < 0 || cost < best) {
      best = cost;
      a.splits = s;
    }
  }
  a.per = (a.nkb + a.splits - 1) / a.splits;
  a.splits = (a.nkb + a.per - 1) / a.per;
  const int64_t tb = (int64_t)FA_NS * (split ? 2 : 1) * 1024, rows = a.splits > 1 ? bh * a.splits * a.nqt * FA_Q : 0;
  a.kv_head = 2 * tb * a.nkb;
  const int64_t kv_bytes = a.kv_head * d->B * Hk, bytes = kv_bytes + rows * (FA_D + 2) * 4;
  if (a.kv_head >= (1LL << 31) || bytes > (1LL << 30) || wgs * a.splits > 0x7fffffff || bh > 65535 || Hk > 65535) return 0;
  void* ws = nullptr;
  int rc = workspace(c, (size_t)bytes, &ws);
  if (rc == ANIMA_E_OOM) {
    (void)hipGetLastError();
    return 0;  // (the chunked path asks for its own amount)
  }
  if (rc) return rc;
  a.q = d->q + d->q_off;
  a.k = d->k + d->k_off;
  a.v = d->v + d->v_off;
  a.o = d->o + d->o_off;
  a.ldq = d->ldq, a.ldk = d->ldk, a.ldv = d->ldv, a.ldo = d->ldo;
  a.qbs = d->q_bstride, a.kbs = d->k_bstride, a.vbs = d->v_bstride, a.obs = d->o_bstride;
  a.kv = (char*)ws;
  a.part = (float*)((char*)ws + kv_bytes);
  a.ml = a.part + rows * FA_D;
  a.Lq = d->Lq;
  a.H = d->H;
  a.group = group;
  a.c = (d->scale != 0.0f ? d->scale : 1.0f / sqrtf((float)FA_D)) * 1.4426950408889634f;
  {
    Launch L(c, "attn.384.prep", 0.0, 8.0 * d->B * Hk * vmax * FA_D * 2);
    const dim3 grid(a.nkb, Hk, d->B);
    if (split) hipLaunchKernelGGL(attn384_prep_kernel<true>, grid, dim3(256), 0, c->stream, a);
    else hipLaunchKernelGGL(attn384_prep_kernel<false>, grid, dim3(256), 0, c->stream, a);
    if ((rc = L.end())) return rc;
  }
  {
    Launch L(c, "attn.384", 4.0 * bh * d->Lq * (double)vmax * FA_D, 0.0);
    const int n = (int)(wgs * a.splits);
    if (split) hipLaunchKernelGGL(attn384_kernel<true>, dim3(n), dim3(512), 0, c->stream, a, n);
    else hipLaunchKernelGGL(attn384_kernel<false>, dim3(n), dim3(512), 0, c->stream, a, n);
    if ((rc = L.end())) return rc;
  }
  if (a.splits > 1) {
    Launch L(c, "attn.384.combine", 0.0, 4.0 * rows * FA_D);
    hipLaunchKernelGGL(attn384_combine_kernel, dim3((d->Lq + 1) / 2, (unsigned)bh), dim3(192), 0, c->stream, a);
    if ((rc = L.end())) return rc;
  }
  return 1;
}

int attention_chunked_launch(anima_ctx* c, const anima_attn_desc* d, const int* kv_len) {
  const int group = d->group <= 0 ? 1 : d->group;
  const int D = d->D, Lq = d->Lq, Lk = d->Lk;
  const float scale = d->scale != 0.0f ? d->scale : 1.0f / sqrtf((float)D);
  const bool split = d->precision == ANIMA_PREC_FP32;
  if (const int r384 = attention384_launch(c, d, kv_len)) return r384 < 0 ? r384 : ANIMA_OK;
  // score rows per chunk: at most 1 GiB of scores (one chunk for the VAE's 16384 tokens at 1024x1024;
  // the device has 288 GB), a multiple of the 128-row tile
  int64_t rows = std::max<int64_t>(TG_BM, ((int64_t)(1 << 30) / 4 / Lk) / TG_BM * TG_BM);
  rows = std::min<int64_t>(rows, ((int64_t)Lq + TG_BM - 1) / TG_BM * TG_BM);
  const int64_t ldk4 = ((int64_t)Lk + 3) / 4 * 4;  // row stride of the scores and of V^T (16-byte rows)
  const size_t s_bytes = (size_t)rows * ldk4 * 4, l_bytes = ((size_t)rows * 4 + 255) / 256 * 256,
               vt_bytes = ((size_t)D * ldk4 * 4 + 255) / 256 * 256;
  int max_ks = 1;
  for (int b = 0; b < d->B; b++) max_ks = std::max(max_ks, pv_splits((int)rows, D, kv_len[b]));
  const size_t p_bytes = max_ks > 1 ? (size_t)max_ks * rows * D * 4 : 0;
  void* ws = nullptr;
  int rc = workspace(c, s_bytes + l_bytes + vt_bytes + p_bytes, &ws);
  if (rc) return rc;
  float* S = (float*)ws;
  float* L = (float*)((char*)ws + s_bytes);
  float* VT = (float*)((char*)ws + s_bytes + l_bytes);
  float* P = (float*)((char*)ws + s_bytes + l_bytes + vt_bytes);
  for (int b = 0; b < d->B; b++) {
    const int valid = kv_len[b];
    for (int h = 0; h < d->H; h++) {
      const int hk = h / group;
      if (h % group == 0) {  // V^T of this kv head
        const float* v = d->v + (int64_t)b * d->v_bstride + d->v_off + (int64_t)hk * D;
        Launch lt(c, "attn.chunk.transpose_v", 0.0, 8.0 * Lk * D);
        hipLaunchKernelGGL(transpose_kernel, dim3((Lk + 31) / 32, (D + 31) / 32), dim3(256), 0, c->stream, v, d->ldv, Lk, D,
                           VT, ldk4);
        if ((rc = lt.end())) return rc;
      }
      for (int r0 = 0; r0 < Lq; r0 += (int)rows) {
        const int nr = (int)std::min<int64_t>(rows, Lq - r0);
        TGemmArgs qk{};
        qk.a = d->q + (int64_t)b * d->q_bstride + (int64_t)r0 * d->ldq + d->q_off + (int64_t)h * D;
        qk.lda = d->ldq;
        qk.b = d->k + (int64_t)b * d->k_bstride + d->k_off + (int64_t)hk * D;
        qk.ldb = d->ldk;
        qk.c = S;
        qk.ldc = ldk4;
        qk.alpha = 1.0f;
        qk.M = nr;
        qk.N = Lk;
        qk.K = D;
        if ((rc = tgemm_launch(c, qk, TG_A_ROWS, TG_B_F32, split, 1, "attn.chunk.qk", 2.0 * nr * Lk * D))) return rc;
        {
          Launch ls(c, "attn.chunk.softmax", 0.0, 8.0 * nr * Lk);
          const int cz = d->causal ? 1 : 0;
          if (Lk <= 256 * 16)
            hipLaunchKernelGGL(chunk_softmax_reg_kernel<16>, dim3(nr), dim3(256), 0, c->stream, S, ldk4, L, Lk, valid, scale, r0, cz);
          else if (Lk <= 256 * 32)
            hipLaunchKernelGGL(chunk_softmax_reg_kernel<32>, dim3(nr), dim3(256), 0, c->stream, S, ldk4, L, Lk, valid, scale, r0, cz);
          else if (Lk <= 256 * 64)
            hipLaunchKernelGGL(chunk_softmax_reg_kernel<64>, dim3(nr), dim3(256), 0, c->stream, S, ldk4, L, Lk, valid, scale, r0, cz);
          else
            hipLaunchKernelGGL(chunk_softmax_kernel, dim3(nr), dim3(256), 0, c->stream, S, ldk4, L, Lk, valid, scale, r0, cz);
          if ((rc = ls.end())) return rc;
        }
        TGemmArgs pv{};
        pv.a = S;
        pv.lda = ldk4;
        pv.b = VT;
        pv.ldb = ldk4;
        pv.alpha = 1.0f;
        pv.M = nr;
        pv.N = D;
        float* o = d->o + (int64_t)b * d->o_bstride + (int64_t)r0 * d->ldo + d->o_off + (int64_t)h * D;
        // A grid of few tiles over a long key range (the VAE's 16384 keys x 384 dims: 384 tiles)
        // splits the keys into ks ranges, products into ks partial outputs, summed and scaled by
        // 1 / rowsum afterwards
        const int ks = pv_splits(nr, D, valid);
        if (ks > 1) {
          pv.c = P;
          pv.ldc = D;
          pv.c_bs = (int64_t)nr * D;
          pv.a_bs = valid / ks;
          pv.b_bs = valid / ks;
          pv.K = valid / ks;
          if ((rc = tgemm_launch(c, pv, TG_A_ROWS, TG_B_F32, split, ks, "attn.chunk.pv", 2.0 * nr * valid * D))) return rc;
          Launch lsum(c, "attn.chunk.pv_sum", 0.0, 4.0 * nr * D * (ks + 1));
          const int64_t n = (int64_t)nr * D;
          hipLaunchKernelGGL(pv_sum_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, c->stream, P, ks, nr, D, L, o,
                             d->ldo);
          if ((rc = lsum.end())) return rc;
        } else {
          pv.c = o;
          pv.ldc = d->ldo;
          pv.rs = L;
          pv.K = valid;  // columns past the valid keys hold zero weights
          if ((rc = tgemm_launch(c, pv, TG_A_ROWS, TG_B_F32, split, 1, "attn.chunk.pv", 2.0 * nr * valid * D))) return rc;
        }
      }
    }
  }
  return ANIMA_OK;
}

}  // namespace anima
