// Direct-convolution potential (leniax/core.py:105-146 get_potential): the depthwise
// cross-correlation of the wrap-padded state with small real kernels, as
// jax.lax.conv_general_dilated(..., 'VALID', feature_group_count=C) computes it, with the
// padding of leniax/helpers.py:465-481 (before = size // 2 on every axis).
//
//   U[b][k][y][x] = sum_{i<kh, j<kw} A[b][cin k][(y + i - ph) mod H][(x + j - pw) mod W] * kern[k][i][j]
//
// One workgroup computes a TH x TW tile of one (world, kernel) output: the input tile and its
// halo are staged in LDS (wrap indexing), each thread keeps a 1 x 4 strip of outputs and slides
// a 4-wide register window along each kernel row, so that one LDS read feeds 4 FMAs; the kernel
// taps are uniform (scalar loads).  Any world size; kernels up to 64 x 64.
#include <algorithm>
#include <type_traits>

#include "lx_internal.h"

namespace {

constexpr int TH = 16, TW = 64, MAXK = 64;

// LDS tile row length: the output tile, the kernel's halo and one spare column (the window's
// last shift reads it), rounded up to a multiple of 4 so that rows start 16-byte aligned
__host__ __device__ inline int tile_cols(int kw) { return (TW + kw + 3) & ~3; }

// Stage rows [y0 - qh, y0 - qh + trows) x columns [x0 - qw, x0 - qw + tcols) of an H x W
// image, wrapped, into tile[trows][stride]: each thread keeps one column (one modulo per thread,
// not per element) and walks rows nsplit apart.  tcols <= 256.  Returns whether this thread met a
// value that is not finite.
LX_DEV bool not_finite(float v) { return !(fabsf(v) <= 3.402823466e38f); }

LX_DEV bool stage_tile(float* tile, const float* img, int H, int W, int y0, int x0, int qh, int qw, int trows,
                       int tcols, int stride) {
  const int nsplit = 256 / tcols;
  const int t = threadIdx.x;
  bool odd = false;
  if (t < nsplit * tcols) {
    const int c = t % tcols, r0 = t / tcols;
    int gx = (x0 + c - qw) % W;
    gx += gx < 0 ? W : 0;
    int gy = (y0 + r0 - qh) % H;
    gy += gy < 0 ? H : 0;
    // 8 rows per round: the loads are all issued before the first LDS write waits on them.
    // The row advances by nsplit, i.e. by step = nsplit mod H < H, so one conditional
    // subtraction keeps gy in [0, H) for any world height.
    const int step = nsplit % H;
    for (int rb = r0; rb < trows; rb += 8 * nsplit) {
      float v[8];
      int rows[8];
#pragma unroll
      for (int u = 0; u < 8; ++u) {
        rows[u] = rb + u * nsplit;
        v[u] = rows[u] < trows ? img[int64_t(gy) * W + gx] : 0.f;
        gy += step;
        gy -= gy >= H ? H : 0;
      }
#pragma unroll
      for (int u = 0; u < 8; ++u)
        if (rows[u] < trows) {
          tile[rows[u] * stride + c] = v[u];
          odd |= not_finite(v[u]);
        }
    }
  }
  return odd;
}

// acc[e] += sum_{j < kw} k_j row[e + j], e < 4, j in increasing order (k_j = kr[j], or kr[kw-1-j]
// when FLIP): taps in blocks of 4 against an 8-wide window read 16 bytes at a time (16 FMAs per
// two LDS reads, no register shifts), the remaining taps one at a time.
template <bool FLIP>
LX_DEV void row_taps(const float* row, const float* kr, int kw, float (&acc)[4]) {
  float4 lo = *reinterpret_cast<const float4*>(row);
  int j = 0;
  for (; j + 4 <= kw; j += 4) {
    const float4 hi = *reinterpret_cast<const float4*>(row + j + 4);
    const float w[8] = {lo.x, lo.y, lo.z, lo.w, hi.x, hi.y, hi.z, hi.w};
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      const float kv = FLIP ? kr[kw - 1 - (j + t)] : kr[j + t];
#pragma unroll
      for (int e = 0; e < 4; ++e) acc[e] = fmaf(kv, w[e + t], acc[e]);
    }
    lo = hi;
  }
  float w0 = lo.x, w1 = lo.y, w2 = lo.z, w3 = lo.w;
  for (; j < kw; ++j) {
    const float kv = FLIP ? kr[kw - 1 - j] : kr[j];
    acc[0] = fmaf(kv, w0, acc[0]);
    acc[1] = fmaf(kv, w1, acc[1]);
    acc[2] = fmaf(kv, w2, acc[2]);
    acc[3] = fmaf(kv, w3, acc[3]);
    w0 = w1; w1 = w2; w2 = w3; w3 = row[j + 4];
  }
}

struct DirectArgs {
  const float* A;
  const float* kern;
  float* U;
  int H, W, C, K, kh, kw, ph, pw;
  int cin[LX_MAX_K];
};

__global__ __launch_bounds__(256) void direct_kernel(DirectArgs a) {
  extern __shared__ __align__(16) float tile[];  // (TH + kh - 1) rows x tile_cols(kw) columns
  const int tcols = tile_cols(a.kw);
  const int trows = TH + a.kh - 1;
  const int x0 = blockIdx.x * TW, y0 = blockIdx.y * TH;
  const int64_t bk = blockIdx.z;
  const int64_t b = bk / a.K;
  const int k = int(bk - b * a.K);
  const float* A = a.A + (b * a.C + a.cin[k]) * int64_t(a.H) * a.W;
  stage_tile(tile, A, a.H, a.W, y0, x0, a.ph, a.pw, trows, tcols, tcols);
  __syncthreads();
  const int ty = threadIdx.x / (TW / 4), tx4 = (threadIdx.x % (TW / 4)) * 4;
  const float* kk = a.kern + int64_t(k) * a.kh * a.kw;
  float acc[4] = {0.f, 0.f, 0.f, 0.f};
  for (int i = 0; i < a.kh; ++i) row_taps<false>(tile + (ty + i) * tcols + tx4, kk + i * a.kw, a.kw, acc);
  const int y = y0 + ty;
  if (y < a.H) {
    float* out = a.U + (bk * a.H + y) * int64_t(a.W) + x0 + tx4;
#pragma unroll
    for (int e = 0; e < 4; ++e)
      if (x0 + tx4 + e < a.W) out[e] = acc[e];
  }
}

// Reverse of the direct potential, state side: dA[b][c] = sum over kernels k fed by c of the
// correlation of dU[b][k] with the flipped kernel, wrap-padded with kh - 1 - ph before (grid:
// tiles x B * C).  The tile of each kernel's dU is staged in LDS in turn.
__global__ __launch_bounds__(256) void direct_adj_kernel(DirectArgs a, const float* dU, float* dA) {
  extern __shared__ __align__(16) float tile[];
  const int tcols = tile_cols(a.kw);
  const int trows = TH + a.kh - 1;
  const int x0 = blockIdx.x * TW, y0 = blockIdx.y * TH;
  const int64_t bc = blockIdx.z;
  const int64_t b = bc / a.C;
  const int c = int(bc - b * a.C);
  const int qh = a.kh - 1 - a.ph, qw = a.kw - 1 - a.pw;
  const int ty = threadIdx.x / (TW / 4), tx4 = (threadIdx.x % (TW / 4)) * 4;
  float acc[4] = {0.f, 0.f, 0.f, 0.f};
  for (int k = 0; k < a.K; ++k) {
    if (a.cin[k] != c) continue;
    const float* G = dU + (b * a.K + k) * int64_t(a.H) * a.W;
    __syncthreads();  // the previous kernel's tile is consumed
    stage_tile(tile, G, a.H, a.W, y0, x0, qh, qw, trows, tcols, tcols);
    __syncthreads();
    const float* kk = a.kern + int64_t(k) * a.kh * a.kw;
    for (int i = 0; i < a.kh; ++i)  // flipped rows and columns
      row_taps<true>(tile + (ty + i) * tcols + tx4, kk + (a.kh - 1 - i) * a.kw, a.kw, acc);
  }
  const int y = y0 + ty;
  if (y < a.H) {
    float* out = dA + (bc * a.H + y) * int64_t(a.W) + x0 + tx4;
#pragma unroll
    for (int e = 0; e < 4; ++e)
      if (x0 + tx4 + e < a.W) out[e] = acc[e];
  }
}

// Reverse of the direct potential, kernel side: dK[k][i][j] = sum over worlds and cells of
// dU[b][k][y][x] A[b][cin k][(y + i - ph) mod H][(x + j - pw) mod W] (grid: kh * kw x K; one block
// per tap, so the sum needs no atomics and is deterministic).
__global__ __launch_bounds__(256) void direct_kgrad_kernel(DirectArgs a, int64_t B, const float* dU, float* dK) {
  const int tap = blockIdx.x;
  const int i = tap / a.kw, j = tap - i * a.kw;
  const int k = blockIdx.y;
  const int64_t n = int64_t(a.H) * a.W;
  float acc = 0.f;
  for (int64_t b = 0; b < B; ++b) {
    const float* G = dU + (b * a.K + k) * n;
    const float* A = a.A + (b * a.C + a.cin[k]) * n;
    for (int64_t p = threadIdx.x; p < n; p += 256) {
      const int y = int(p / a.W), x = int(p - int64_t(y) * a.W);
      int gy = (y + i - a.ph) % a.H;
      gy += gy < 0 ? a.H : 0;
      int gx = (x + j - a.pw) % a.W;
      gx += gx < 0 ? a.W : 0;
      acc = fmaf(G[p], A[int64_t(gy) * a.W + gx], acc);
    }
  }
  __shared__ float red[4];
  const float s = wave_sum(acc);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = s;
  __syncthreads();
  if (threadIdx.x == 0) dK[(int64_t(k) * a.kh + i) * a.kw + j] = red[0] + red[1] + red[2] + red[3];
}

// The kernel side on the matrix cores, for callers with a workspace.  With i = 4 ib + n and
// j = 4 jb + m, dK[i][j] = sum over cells of dU[y][x - m] A[y + 4 ib + n - ph][x + 4 jb - pw] (both
// images are periodic, so the sum over x may start at any shift): for each cell (y, x) a 4 x 4 outer
// product per (ib, jb), which is one v_mfma_f32_4x4x1 for 16 (ib, jb) pairs.  Lane 4 s + n of a set
// holds its pair's n-th row of A, four cells per 16-byte LDS read; the dU operand is the same for
// every pair, so one register holds 16 cells' (lane 4 p + m: dU[y][x + p - m]) and the instruction
// broadcasts block p of it.  A block takes tiles of kGY x kGX cells in turn (waves take rows), adds
// its waves' sums in order and stores one row of partial sums; direct_kgrad_sum_kernel adds the rows
// in a fixed order, so the gradient is deterministic.  In the matrix form every LDS value feeds 4
// multiply-adds of its lane and the pass is bound by LDS reads and MFMA issue (the one-block-per-tap
// kernel above re-reads both images for every tap with a division and two remainders per product).
// A row stride of 16 mod 64 floats puts the four rows n of a read in different banks.
// Measured, 128 worlds of 128^2 with a 25 x 25 kernel: 3457 -> 59 + 5 us (2.6 GFLOP of taps: 41 TFLOP/s),
// error against 64 bits 1.6e-6 -> 4.7e-7 (shorter chains of additions).
constexpr int kGY = 16, kGX = 64, kGridRows = 1024, kGSets = 4;
typedef float f4v __attribute__((ext_vector_type(4)));

__host__ __device__ inline int kgrad_stride(int kw) {  // >= kGX + 4 ceil(kw / 4), 16 mod 64
  const int need = kGX + ((kw + 3) & ~3);
  return ((need - 16 + 63) / 64) * 64 + 16;
}
__host__ __device__ inline int kgrad_rows(int kh) { return kGY - 1 + ((kh + 3) & ~3); }
constexpr int kGDU = kGX + 4;  // dU tile row: 3 columns before, one spare

// NS: sets of 16 (ib, jb) pairs per block; blockIdx.y = k * groups + group of NS sets
template <int NS>
__global__ __launch_bounds__(256) void direct_kgrad_mfma_kernel(DirectArgs a, int64_t B, const float* dU, float* part,
                                                                int groups, int tx, int64_t ntiles) {
  extern __shared__ __align__(16) float lds[];
  const int S = kgrad_stride(a.kw), R = kgrad_rows(a.kh);
  float* tA = lds;          // [R][S]
  float* tG = lds + R * S;  // [kGY][kGDU]
  const int k = blockIdx.y / groups, set0 = (blockIdx.y - k * groups) * NS;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int nj = (a.kw + 3) / 4, nb = nj * ((a.kh + 3) / 4);
  int off[NS];  // the lane's first A value of each set (pairs past the last read pair 0, unused)
#pragma unroll
  for (int s = 0; s < NS; ++s) {
    int blk = (set0 + s) * 16 + (lane >> 2);
    if (blk >= nb) blk = 0;
    const int ib = blk / nj, jb = blk - ib * nj;
    off[s] = (4 * ib + (lane & 3)) * S + 4 * jb;
  }
  f4v acc[NS];
#pragma unroll
  for (int s = 0; s < NS; ++s) acc[s] = f4v{0.f, 0.f, 0.f, 0.f};
  const int64_t n = int64_t(a.H) * a.W;
  const int ty = (a.H + kGY - 1) / kGY;
  for (int64_t tile = blockIdx.x; tile < ntiles; tile += gridDim.x) {
    const int64_t b = tile / (int64_t(tx) * ty);
    const int rem = int(tile - b * tx * ty);
    const int y0 = (rem / tx) * kGY, x0 = (rem % tx) * kGX;
    __syncthreads();  // the previous tile is consumed
    const bool odd = stage_tile(tA, a.A + (b * a.C + a.cin[k]) * n, a.H, a.W, y0, x0, a.ph, a.pw, R,
                                kGX + 4 * nj, S);
    stage_tile(tG, dU + (b * a.K + k) * n, a.H, a.W, y0, x0, 0, 3, kGY, kGDU, kGDU);
    const bool slow = __syncthreads_or(odd);
    const int rows = min(kGY, a.H - y0), cols = min(kGX, a.W - x0);
    if (!slow) {
      for (int r = wave; r < rows; r += 4) {
        for (int xg = 0; xg < cols; xg += 16) {
          const int p = lane >> 2;
          // cells past the image's last column count nothing
          const float g = xg + p < cols ? tG[r * kGDU + xg + p - (lane & 3) + 3] : 0.f;
          const float* row = tA + r * S + xg;
          auto quad = [&](auto q_c) {
            constexpr int Q = decltype(q_c)::value;
            float4 v[NS];
#pragma unroll
            for (int s = 0; s < NS; ++s) v[s] = *reinterpret_cast<const float4*>(row + off[s] + 4 * Q);
#pragma unroll
            for (int s = 0; s < NS; ++s) acc[s] = __builtin_amdgcn_mfma_f32_4x4x1f32(g, v[s].x, acc[s], 4, 4 * Q, 0);
#pragma unroll
            for (int s = 0; s < NS; ++s)
              acc[s] = __builtin_amdgcn_mfma_f32_4x4x1f32(g, v[s].y, acc[s], 4, 4 * Q + 1, 0);
#pragma unroll
            for (int s = 0; s < NS; ++s)
              acc[s] = __builtin_amdgcn_mfma_f32_4x4x1f32(g, v[s].z, acc[s], 4, 4 * Q + 2, 0);
#pragma unroll
            for (int s = 0; s < NS; ++s)
              acc[s] = __builtin_amdgcn_mfma_f32_4x4x1f32(g, v[s].w, acc[s], 4, 4 * Q + 3, 0);
          };
          quad(std::integral_constant<int, 0>{});
          quad(std::integral_constant<int, 1>{});
          quad(std::integral_constant<int, 2>{});
          quad(std::integral_constant<int, 3>{});
        }
      }
    } else {
      // a state that is not finite: product by product, so that none is taken with the zero of a
      // cell past the last column
      for (int r = wave; r < rows; r += 4)
        for (int x = 0; x < cols; ++x)
#pragma unroll
          for (int s = 0; s < NS; ++s) {
            const float v = tA[r * S + x + off[s]];
#pragma unroll
            for (int m = 0; m < 4; ++m) acc[s][m] = fmaf(tG[r * kGDU + x - m + 3], v, acc[s][m]);
          }
    }
  }
  // the waves' sums in order, then the block's row of partial sums
  __syncthreads();
  float* red = lds;  // [4][NS][64][4] floats
#pragma unroll
  for (int s = 0; s < NS; ++s)
    *reinterpret_cast<f4v*>(red + ((wave * NS + s) * 64 + lane) * 4) = acc[s];
  __syncthreads();
  float* dst = part + (int64_t(blockIdx.x) * a.K + k) * a.kh * a.kw;
  for (int e = threadIdx.x; e < NS * 256; e += 256) {
    const int s = e >> 8, l = (e >> 2) & 63, m = e & 3;
    const int blk = (set0 + s) * 16 + (l >> 2);
    const int ib = blk / nj, jb = blk - ib * nj;
    const int i = 4 * ib + (l & 3), j = 4 * jb + m;
    if (blk < nb && i < a.kh && j < a.kw) {
      float v = 0.f;
#pragma unroll
      for (int w = 0; w < 4; ++w) v += red[(w * NS * 64) * 4 + e];
      dst[i * a.kw + j] = v;
    }
  }
}

// dK[tap] = sum of the partial rows: 32 taps per block, 32 threads per tap take every 32nd row (8 loads
// in flight), then their sums are added in order
__global__ __launch_bounds__(1024) void direct_kgrad_sum_kernel(const float* part, int rows, int taps, float* dK) {
  __shared__ float red[32][32];
  const int t = threadIdx.x & 31, sl = threadIdx.x >> 5;
  const int tap = blockIdx.x * 32 + t;
  float acc = 0.f;
  if (tap < taps) {
#pragma unroll 8
    for (int r = sl; r < rows; r += 32) acc += part[int64_t(r) * taps + tap];
  }
  red[sl][t] = acc;
  __syncthreads();
  if (sl == 0 && tap < taps) {
#pragma unroll
    for (int i = 1; i < 32; ++i) acc += red[i][t];
    dK[tap] = acc;
  }
}

int kgrad_tiles_x(int W) { return (W + kGX - 1) / kGX; }
int64_t kgrad_tiles(const lx_rule* r, int64_t B) {
  return B * kgrad_tiles_x(r->dims[1]) * ((r->dims[0] + kGY - 1) / kGY);
}
// blocks of NS = kgrad_ns(sets) sets per kernel and rows of partial sums: enough blocks to fill 256 CUs
// a few times over, no more than tiles; at most kGridRows x 16 kGSets taps x 16 B of partial sums
int kgrad_sets(int kh, int kw) { return (((kh + 3) / 4) * ((kw + 3) / 4) + 15) / 16; }
int kgrad_ns(int sets) { return sets < 3 ? sets : kGSets; }
int64_t kgrad_part_rows(const lx_rule* r, int64_t B, int kh, int kw) {
  const int sets = kgrad_sets(kh, kw), per = r->K * ((sets + kgrad_ns(sets) - 1) / kgrad_ns(sets));
  return std::min<int64_t>(kgrad_tiles(r, B), (kGridRows + per - 1) / per);
}

DirectArgs direct_args(const lx_rule* rule, const float* A, const float* kern, int kh, int kw) {
  DirectArgs a;
  a.A = A; a.kern = kern; a.U = nullptr;
  a.H = rule->dims[0]; a.W = rule->dims[1]; a.C = rule->C; a.K = rule->K;
  a.kh = kh; a.kw = kw; a.ph = kh / 2; a.pw = kw / 2;
  for (int k = 0; k < LX_MAX_K; ++k) a.cin[k] = k < rule->K ? rule->cin[k] : 0;
  return a;
}

}  // namespace

namespace {

// the reverse of the direct potential; work: lx_potential_direct_adjoint_size bytes, or NULL (the
// kernel side then takes one block per tap)
int direct_adjoint(const char* fn, const lx_rule* rule, const float* state_d, int64_t B, const float* kern_d,
                   int32_t kh, int32_t kw, const float* dpot_d, float* dstate_d, float* dkern_d, float* work,
                   hipStream_t st) {
  int rc = lx_check_rule(rule);
  if (rc) return rc;
  if (rule->ndim != 2) return lx_fail(LX_ENOTSUP, "%s: 2-D worlds only", fn);
  if (kh < 1 || kw < 1 || kh > MAXK || kw > MAXK) return lx_fail(LX_ENOTSUP, "kernel %dx%d (1..%d)", kh, kw, MAXK);
  if (B < 0) return lx_fail(LX_EINVAL, "B < 0");
  if (B == 0) return LX_OK;
  if (!kern_d || !dpot_d || (!dstate_d && !dkern_d) || (dkern_d && !state_d)) return lx_fail(LX_EINVAL, "NULL pointer");
  if (B * rule->C > 65535) return lx_fail(LX_ENOTSUP, "%s: B * C > 65535", fn);
  const DirectArgs a = direct_args(rule, state_d, kern_d, kh, kw);
  if (dstate_d) {
    const size_t lds = size_t(TH + kh - 1) * size_t(tile_cols(kw)) * sizeof(float);
    const dim3 grid(unsigned((a.W + TW - 1) / TW), unsigned((a.H + TH - 1) / TH), unsigned(B * rule->C));
    hipLaunchKernelGGL(direct_adj_kernel, grid, dim3(256), lds, st, a, dpot_d, dstate_d);
  }
  if (dkern_d && work) {
    const int64_t rows = kgrad_part_rows(rule, B, kh, kw);
    const int sets = kgrad_sets(kh, kw);
    auto go = [&](auto ns_c) {
      constexpr int NS = decltype(ns_c)::value;
      const int groups = (sets + NS - 1) / NS;
      const size_t tiles = size_t(kgrad_rows(kh)) * kgrad_stride(kw) + size_t(kGY) * kGDU;
      const size_t lds = std::max(tiles, size_t(4) * NS * 256) * sizeof(float);
      hipLaunchKernelGGL((direct_kgrad_mfma_kernel<NS>), dim3(unsigned(rows), unsigned(rule->K * groups)), dim3(256),
                         lds, st, a, B, dpot_d, work, groups, kgrad_tiles_x(a.W), kgrad_tiles(rule, B));
    };
    switch (kgrad_ns(sets)) {
      case 1: go(std::integral_constant<int, 1>{}); break;
      case 2: go(std::integral_constant<int, 2>{}); break;
      default: go(std::integral_constant<int, kGSets>{}); break;
    }
    const int taps = rule->K * kh * kw;
    hipLaunchKernelGGL(direct_kgrad_sum_kernel, dim3(unsigned((taps + 31) / 32)), dim3(1024), 0, st, work, int(rows),
                       taps, dkern_d);
  } else if (dkern_d) {
    hipLaunchKernelGGL(direct_kgrad_kernel, dim3(unsigned(kh * kw), unsigned(rule->K)), dim3(256), 0, st, a, B,
                       dpot_d, dkern_d);
  }
  hipError_t e = hipGetLastError();
  return e == hipSuccess ? LX_OK : lx_fail(LX_EDEVICE, "direct adjoint launch: %s", hipGetErrorString(e));
}

}  // namespace

extern "C" int lx_potential_direct_adjoint(const lx_rule* rule, const float* state_d, int64_t B,
                                           const float* kern_d, int32_t kh, int32_t kw, const float* dpot_d,
                                           float* dstate_d, float* dkern_d, void* stream) {
  return direct_adjoint("lx_potential_direct_adjoint", rule, state_d, B, kern_d, kh, kw, dpot_d, dstate_d, dkern_d,
                        nullptr, (hipStream_t)stream);
}

extern "C" int lx_potential_direct_adjoint_size(const lx_rule* rule, int64_t B, int32_t kh, int32_t kw,
                                                size_t* bytes) {
  int rc = lx_check_rule(rule);
  if (rc) return rc;
  if (rule->ndim != 2) return lx_fail(LX_ENOTSUP, "lx_potential_direct_adjoint_size: 2-D worlds only");
  if (kh < 1 || kw < 1 || kh > MAXK || kw > MAXK) return lx_fail(LX_ENOTSUP, "kernel %dx%d (1..%d)", kh, kw, MAXK);
  if (B < 0 || !bytes) return lx_fail(LX_EINVAL, "B < 0 or NULL pointer");
  *bytes = size_t(kgrad_part_rows(rule, B, kh, kw)) * rule->K * kh * kw * sizeof(float);
  return LX_OK;
}

extern "C" int lx_potential_direct_adjoint_work(const lx_rule* rule, const float* state_d, int64_t B,
                                                const float* kern_d, int32_t kh, int32_t kw, const float* dpot_d,
                                                float* dstate_d, float* dkern_d, void* work_d, void* stream) {
  if (B > 0 && dkern_d && !work_d) return lx_fail(LX_EINVAL, "lx_potential_direct_adjoint_work: NULL workspace");
  return direct_adjoint("lx_potential_direct_adjoint_work", rule, state_d, B, kern_d, kh, kw, dpot_d, dstate_d,
                        dkern_d, static_cast<float*>(work_d), (hipStream_t)stream);
}

extern "C" int lx_potential_direct(const lx_rule* rule, const float* state_d, int64_t B, const float* kern_d,
                                   int32_t kh, int32_t kw, float* potential_d, void* stream) {
  int rc = lx_check_rule(rule);
  if (rc) return rc;
  if (rule->ndim != 2) return lx_fail(LX_ENOTSUP, "lx_potential_direct: 2-D worlds only");
  if (kh < 1 || kw < 1 || kh > MAXK || kw > MAXK) return lx_fail(LX_ENOTSUP, "kernel %dx%d (1..%d)", kh, kw, MAXK);
  if (B < 0) return lx_fail(LX_EINVAL, "B < 0");
  if (B == 0) return LX_OK;
  if (!state_d || !kern_d || !potential_d) return lx_fail(LX_EINVAL, "NULL pointer");
  if (B * rule->K > 65535) return lx_fail(LX_ENOTSUP, "lx_potential_direct: B * K > 65535");
  DirectArgs a = direct_args(rule, state_d, kern_d, kh, kw);
  a.U = potential_d;
  const size_t lds = size_t(TH + kh - 1) * size_t(tile_cols(kw)) * sizeof(float);
  const dim3 grid(unsigned((a.W + TW - 1) / TW), unsigned((a.H + TH - 1) / TH), unsigned(B * rule->K));
  hipLaunchKernelGGL(direct_kernel, grid, dim3(256), lds, (hipStream_t)stream, a);
  hipError_t e = hipGetLastError();
  return e == hipSuccess ? LX_OK : lx_fail(LX_EDEVICE, "direct potential launch: %s", hipGetErrorString(e));
}
