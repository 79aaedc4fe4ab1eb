// Prefill-path kernels (a chunk of n tokens) for gfx950: row LayerNorm, a
// vector-unit projection GEMM for formats the matrix cores do not take, the
// fused in-projection epilogue, SiLU-gate and the parallel residual.
// Follows prefill.go:33-115 step for step.
#include <algorithm>
#include <initializer_list>

#include "epilogue.h"

namespace {

__global__ __launch_bounds__(256) void layer_norm_rows_kernel(const float *x, const float *w, const float *b,
                                                               double eps, int d, float *out, uint16_t *oh,
                                                               uint16_t *ol, int ldo) {
  extern __shared__ __align__(16) float lds[];
  double *red = reinterpret_cast<double *>(lds + ((d + 3) & ~3));
  const int64_t row = blockIdx.x;
  for (int i = threadIdx.x; i < d; i += blockDim.x) lds[i] = x[row * d + i];
  __syncthreads();
  layer_norm_lds(lds, d, w, b, eps, red);
  for (int i = threadIdx.x; i < d; i += blockDim.x) {
    if (out) out[row * d + i] = lds[i];
    if (oh) store_bf16_split(oh, ol, row * ldo + i, lds[i]);
  }
}

// out[n][N] = x[n][K] * W[N][K]^T, fp32 SIMT tiles of 64 tokens x 64 rows,
// each thread a 4 x 4 micro-tile; weights dequantized into LDS. As mulBatch
// does (matmul.go:55-95), products accumulate in float32 within 512-column
// blocks and the block partials in float64.
constexpr int kTM = 64, kTN = 64, kTK = 32, kBlockCols = 512;

__global__ __launch_bounds__(256) void gemm_simt_kernel(MatDesc w, const float *__restrict__ x, int n,
                                                         float *__restrict__ out) {
  __shared__ float xs[kTK][kTM + 4];
  __shared__ float ws[kTK][kTN + 4];
  const int m0 = blockIdx.y * kTM, n0 = blockIdx.x * kTN;
  const int K = w.cols, N = w.rows;
  const int tx = threadIdx.x % 16, ty = threadIdx.x / 16;
  float acc[4][4] = {};
  double total[4][4] = {};
  for (int k0 = 0; k0 < K; k0 += kTK) {
    for (int e = threadIdx.x; e < kTM * kTK; e += 256) {
      const int r = e / kTK, c = e % kTK;
      const int tok = m0 + r, col = k0 + c;
      xs[c][r] = (tok < n && col < K) ? x[(int64_t)tok * K + col] : 0.f;
      const int row = n0 + r;
      ws[c][r] = (row < N && col < K) ? mat_value(w, row, col) : 0.f;
    }
    __syncthreads();
#pragma unroll 8
    for (int c = 0; c < kTK; c++) {
      float a[4], b[4];
#pragma unroll
      for (int i = 0; i < 4; i++) {
        a[i] = xs[c][ty * 4 + i];
        b[i] = ws[c][tx * 4 + i];
      }
#pragma unroll
      for (int i = 0; i < 4; i++)
#pragma unroll
        for (int jj = 0; jj < 4; jj++) acc[i][jj] = fmaf(a[i], b[jj], acc[i][jj]);
    }
    __syncthreads();
    if ((k0 + kTK) % kBlockCols == 0 || k0 + kTK >= K) {
#pragma unroll
      for (int i = 0; i < 4; i++)
#pragma unroll
        for (int jj = 0; jj < 4; jj++) {
          total[i][jj] += (double)acc[i][jj];
          acc[i][jj] = 0.f;
        }
    }
  }
#pragma unroll
  for (int i = 0; i < 4; i++) {
    const int tok = m0 + ty * 4 + i;
    if (tok >= n) continue;
#pragma unroll
    for (int jj = 0; jj < 4; jj++) {
      const int row = n0 + tx * 4 + jj;
      if (row < N) out[(int64_t)tok * N + row] = (float)total[i][jj];
    }
  }
}

// One block per token: the fused in-projection epilogue (RoPE on q and k,
// storeKV at the token's absolute position, SiLU-gate), as prefill.go:60-96
// applies it row by row. With mh, the SiLU-gate outputs (the units from
// mu0 on) also go out as the down projection's bf16 operand planes, and to
// m only when m is given.
// With rows, token j sits at position rows[2j] and its K and V go to slot
// rows[2j + 1] of the cache kv (a branch cache: the slot of the branch's
// suffix entry).
// One epilogue's block (token blockIdx.x, block by of its gy on the grid's
// second dimension).
__device__ __forceinline__ void in_epilogue_body(const StableDims &s, const KVDev &kv, const float *y, int ldy,
                                                 const float *rope, const int *pos0, int units, float *q, float *m,
                                                 uint16_t *mh, uint16_t *ml, const int *rows, int ys, int ldm, int by,
                                                 int gy) {
  const int j = blockIdx.x;
  const int pos = rows ? rows[2 * j] : *pos0 + j;
  const int slot = rows ? rows[2 * j + 1] : pos;
  const float *yj = y + (int64_t)j * ldy;
  const float *rope_row = rope + (int64_t)pos * s.rot;
  const int mu0 = (s.win_q + 2 * s.win_kv) / 2;
  float *qj = q + (int64_t)j * s.heads * s.hd, *mj = m ? m + (int64_t)j * s.inter : nullptr;
  const int64_t split = (int64_t)gridDim.x * ldy;
  // block by takes every gy-th group of blockDim.x units; a thread
  // loads kBatch of its units before it stores any, and the next kBatch
  // before it stores those (the stores could alias y as far as the
  // compiler knows, so loads placed after them would each wait a memory
  // round trip).
  constexpr int kBatch = 4;
  const int stride = gy * blockDim.x;
  auto load = [&](int u0, float2 (&v)[kBatch]) {
#pragma unroll
    for (int b = 0; b < kBatch; b++) {
      const int u = u0 + b * stride;
      v[b] = u < units ? *reinterpret_cast<const float2 *>(yj + 2 * u) : make_float2(0.f, 0.f);
      for (int s2 = 1; s2 < ys; s2++) {
        if (u >= units) break;
        const float2 t = *reinterpret_cast<const float2 *>(yj + s2 * split + 2 * u);
        v[b].x = __fadd_rn(v[b].x, t.x);
        v[b].y = __fadd_rn(v[b].y, t.y);
      }
    }
  };
  float2 v[kBatch], nv[kBatch];
  int u0 = by * blockDim.x + threadIdx.x;
  if (u0 < units) load(u0, v);
  for (; u0 < units; u0 += kBatch * stride) {
    const int un = u0 + kBatch * stride;
    if (un < units) load(un, nv);
#pragma unroll
    for (int b = 0; b < kBatch; b++) {
      const int u = u0 + b * stride;
      if (u >= units) break;
      if (mh && u >= mu0) {
        const float g = s.silu ? silu_gate_llama(v[b].x, v[b].y) : silu_gate(v[b].x, v[b].y);
        if (mj) mj[u - mu0] = g;
        store_bf16_split(mh, ml, (int64_t)j * ldm + (u - mu0), g);
      } else {
        in_pair_epilogue(s, kv, rope_row, slot, u, v[b].x, v[b].y, qj, mj);
      }
    }
#pragma unroll
    for (int b = 0; b < kBatch; b++) v[b] = nv[b];
  }
}

__global__ void in_epilogue_kernel(StableDims s, KVDev kv, const float *y, int ldy, const float *rope,
                                   const int *pos0, int units, float *q, float *m, uint16_t *mh, uint16_t *ml,
                                   const int *rows, int ys, int ldm) {
  in_epilogue_body(s, kv, y, ldy, rope, pos0, units, q, m, mh, ml, rows, ys, ldm, blockIdx.y, gridDim.y);
}

struct InEpiArgs {
  StableDims s;
  const float *y;
  int ldy, units, ys, gy;
  float *m;
};
// Two epilogues of the same tokens in one launch (the second's blocks after
// the first's on the grid's second dimension): the branch step's q/k/v and
// gate/up products, each with its own dims, partials and split count.
__global__ void in_epilogue_pair_kernel(InEpiArgs a, InEpiArgs b, KVDev kv, const float *rope, float *q,
                                        const int *rows) {
  if ((int)blockIdx.y < a.gy)
    in_epilogue_body(a.s, kv, a.y, a.ldy, rope, nullptr, a.units, q, a.m, nullptr, nullptr, rows, a.ys, a.s.inter,
                     blockIdx.y, a.gy);
  else
    in_epilogue_body(b.s, kv, b.y, b.ldy, rope, nullptr, b.units, q, b.m, nullptr, nullptr, rows, b.ys, b.s.inter,
                     (int)blockIdx.y - a.gy, b.gy);
}

// sum = ((v[0] + v[1]) + v[2]) + ... over s partials n apart, eight
// loads in flight before their adds (the same order as one at a time).
__device__ __forceinline__ float sum_partials(const float *v, int s, int64_t n, int64_t i) {
  constexpr int B = 8;
  float acc = v[i];
  for (int s0 = 1; s0 < s; s0 += B) {
    float t[B];
#pragma unroll
    for (int k = 0; k < B; k++) t[k] = s0 + k < s ? v[(s0 + k) * n + i] : 0.f;
#pragma unroll
    for (int k = 0; k < B; k++)
      if (s0 + k < s) acc = __fadd_rn(acc, t[k]);
  }
  return acc;
}

// The residual of a chunk's row (residual_kernel's arithmetic) and the
// next layer's LayerNorm of it (layer_norm_rows_kernel's): one block per
// row stages the new row in LDS while it stores it, so the row is read
// once for both. Two elements per thread at a time, their loads issued
// before their stores.
__global__ __launch_bounds__(256) void residual_norm_rows_kernel(float *x, const float *p, int sp, const float *dd,
                                                                 int sd, int64_t n, int d, const float *w,
                                                                 const float *b, double eps, float *out, uint16_t *oh,
                                                                 uint16_t *ol, int ldo) {
  extern __shared__ __align__(16) float lds[];
  double *red = reinterpret_cast<double *>(lds + ((d + 3) & ~3));
  const int64_t row = blockIdx.x;
  constexpr int E = 2;
  for (int i0 = threadIdx.x; i0 < d; i0 += E * blockDim.x) {
    float v[E];
#pragma unroll
    for (int e = 0; e < E; e++) {
      const int i = i0 + e * blockDim.x;
      if (i < d) {
        const int64_t k = row * d + i;
        v[e] = __fadd_rn(__fadd_rn(x[k], sum_partials(p, sp, n, k)), sum_partials(dd, sd, n, k));
      }
    }
#pragma unroll
    for (int e = 0; e < E; e++) {
      const int i = i0 + e * blockDim.x;
      if (i < d) {
        x[row * d + i] = v[e];
        lds[i] = v[e];
      }
    }
  }
  __syncthreads();
  layer_norm_lds(lds, d, w, b, eps, red);
  for (int i = threadIdx.x; i < d; i += blockDim.x) {
    if (out) out[row * d + i] = lds[i];
    if (oh) store_bf16_split(oh, ol, row * ldo + i, lds[i]);
  }
}

// The same two for rows of up to 4096 values, a multiple of 4, held in
// registers (4 float4 a thread): every load of the row, its weights and up to
// four partials is in flight at once, where the loops above wait for one
// round trip per 256 values (19 rows of 2560: 9.5 us; 700 rows with their
// residual 23 us, against 4.9 and 15 here). The new row may leave as fp16
// planes too (launch_split_f16's, zeros up to fp.ld).
constexpr int kNormG = 4;
template <bool RESID>
__global__ __launch_bounds__(256) void norm_rows_kernel(float *x, const float *p, int sp, const float *dd, int sd,
                                                        int64_t n, int d, const float *w, const float *b, double eps,
                                                        float *out, uint16_t *oh, uint16_t *ol, int ldo,
                                                        Fp16Planes fp) {
  __shared__ double red[4];
  __shared__ int most[4], votes[4];
  const int64_t row = blockIdx.x;
  const int tid = threadIdx.x;
  auto at = [&](int g) { return 4 * (tid + 256 * g); };
  // past the row: the last group's values, replaced by zeros
  auto load = [&](const float *s, float4 (&v)[kNormG]) {
#pragma unroll
    for (int g = 0; g < kNormG; g++) v[g] = *reinterpret_cast<const float4 *>(s + min(at(g), d - 4));
  };
  float4 v[kNormG], wv[kNormG], bv[kNormG];
  load(x + row * d, v);
  load(w, wv);
  load(b, bv);
  if constexpr (RESID) {
    // sums of the partials in order of the split, four splits' loads at once
    auto sum = [&](const float *s, int ks, float4 (&a)[kNormG]) {
      load(s + row * d, a);
      for (int s0 = 1; s0 < ks; s0 += 4) {
        float4 t[4][kNormG];
#pragma unroll
        for (int k = 0; k < 4; k++) load(s + min(s0 + k, ks - 1) * n + row * d, t[k]);
#pragma unroll
        for (int k = 0; k < 4; k++) {
          if (s0 + k >= ks) break;
#pragma unroll
          for (int g = 0; g < kNormG; g++)
            a[g] = make_float4(__fadd_rn(a[g].x, t[k][g].x), __fadd_rn(a[g].y, t[k][g].y),
                               __fadd_rn(a[g].z, t[k][g].z), __fadd_rn(a[g].w, t[k][g].w));
        }
      }
    };
    float4 a[kNormG];
    auto add = [&]() {
#pragma unroll
      for (int g = 0; g < kNormG; g++)
        v[g] = make_float4(__fadd_rn(v[g].x, a[g].x), __fadd_rn(v[g].y, a[g].y), __fadd_rn(v[g].z, a[g].z),
                           __fadd_rn(v[g].w, a[g].w));
    };
    sum(p, sp, a);
    add();
    sum(dd, sd, a);
    add();
  }
#pragma unroll
  for (int g = 0; g < kNormG; g++) {
    if (at(g) >= d) v[g] = make_float4(0.f, 0.f, 0.f, 0.f);
    else if (RESID) *reinterpret_cast<float4 *>(x + row * d + at(g)) = v[g];
  }
  // LayerNorm (layer_norm_lds's arithmetic: float64 two-pass moments, float32
  // affine with separately rounded steps)
  double s = 0;
#pragma unroll
  for (int g = 0; g < kNormG; g++) s += ((double)v[g].x + (double)v[g].y) + ((double)v[g].z + (double)v[g].w);
  const double mean = block_sum_d(s, red) / (double)d;
  s = 0;
#pragma unroll
  for (int g = 0; g < kNormG; g++) {
    if (at(g) >= d) continue;
    const double e[4] = {v[g].x - mean, v[g].y - mean, v[g].z - mean, v[g].w - mean};
    s += (e[0] * e[0] + e[1] * e[1]) + (e[2] * e[2] + e[3] * e[3]);
  }
  const double var = block_sum_d(s, red);
  const float inv = (float)(1.0 / sqrt(var / (double)d + eps)), fm = (float)mean;
  auto affine = [&](float t, float wi, float bi) {
    return __fadd_rn(__fmul_rn(__fmul_rn(__fsub_rn(t, fm), inv), wi), bi);
  };
  int mag = 0;
#pragma unroll
  for (int g = 0; g < kNormG; g++) {
    const int i = at(g);
    if (i < d) {
      v[g] = make_float4(affine(v[g].x, wv[g].x, bv[g].x), affine(v[g].y, wv[g].y, bv[g].y),
                         affine(v[g].z, wv[g].z, bv[g].z), affine(v[g].w, wv[g].w, bv[g].w));
      if (out) *reinterpret_cast<float4 *>(out + row * d + i) = v[g];
    }
    const float f[4] = {v[g].x, v[g].y, v[g].z, v[g].w};
    if (oh && i < d) {
      uint32_t hb[4], lb[4];  // store_bf16_split's values
#pragma unroll
      for (int e = 0; e < 4; e++) {
        const __bf16 h = (__bf16)f[e];
        hb[e] = __builtin_bit_cast(uint16_t, h);
        lb[e] = __builtin_bit_cast(uint16_t, (__bf16)(f[e] - (float)h));
      }
      *reinterpret_cast<uint2 *>(oh + row * ldo + i) = make_uint2(hb[0] | hb[1] << 16, hb[2] | hb[3] << 16);
      *reinterpret_cast<uint2 *>(ol + row * ldo + i) = make_uint2(lb[0] | lb[1] << 16, lb[2] | lb[3] << 16);
    }
#pragma unroll
    for (int e = 0; e < 4; e++) mag = max(mag, fp16_magnitude(f[e]));
  }
  if (!fp.hi) return;  // uniform
  for (int o = 32; o > 0; o >>= 1) mag = max(mag, __shfl_xor(mag, o));
  if ((tid & 63) == 0) most[tid >> 6] = mag;
  __syncthreads();
  mag = max(max(most[0], most[1]), max(most[2], most[3]));
  float down;
  const float up = fp16_scale(mag, down);
  bool suspect = false;
#pragma unroll
  for (int g = 0; g < kNormG; g++) {
    if (at(g) >= fp.ld) continue;
    uint2 hi, lo;
    fp16_split4(v[g], up, hi, lo);
    suspect |= fp16_suspect(v[g], mag);
    *reinterpret_cast<uint2 *>(fp.hi + row * fp.ld + at(g)) = hi;
    *reinterpret_cast<uint2 *>(fp.lo + row * fp.ld + at(g)) = lo;
  }
  const bool wave_suspect = __any(suspect);
  if ((tid & 63) == 0) votes[tid >> 6] = wave_suspect;
  __syncthreads();
  bool marked = false;
  if (votes[0] | votes[1] | votes[2] | votes[3]) {  // uniform
    int vote = 0;
#pragma unroll
    for (int g = 0; g < kNormG; g++)  // (zeros past the row)
      vote += (fp16_vote(v[g].x, mag) + fp16_vote(v[g].y, mag)) + (fp16_vote(v[g].z, mag) + fp16_vote(v[g].w, mag));
    for (int o = 32; o > 0; o >>= 1) vote += __shfl_xor(vote, o);
    __syncthreads();
    if ((tid & 63) == 0) votes[tid >> 6] = vote;
    __syncthreads();
    marked = (votes[0] + votes[1]) + (votes[2] + votes[3]) > 0;
  }
  if (tid == 0) fp.unscale[row] = marked ? -down : down;
  if (!marked) return;
#pragma unroll
  for (int g = 0; g < kNormG; g++)
    if (at(g) < d) *reinterpret_cast<float4 *>(fp.rows + row * d + at(g)) = v[g];
}

__global__ void residual_kernel(float *x, const float *p, int sp, const float *d, int sd, int64_t n) {
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
    const float o = sum_partials(p, sp, n, i), m = sum_partials(d, sd, n, i);
    x[i] = __fadd_rn(__fadd_rn(x[i], o), m);
  }
}

// out[i] = ((p[0][i] + p[1][i]) + p[2][i]) + ... over sp partials n apart.
__global__ void sum_splits_kernel(float *out, const float *p, int sp, int64_t n) {
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
    out[i] = sum_partials(p, sp, n, i);
  }
}

__global__ void copy_kernel(const float *src, float *dst, int n) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) dst[i] = src[i];
}

struct RowPairs {
  int src[kRowPairs], dst[kRowPairs];
};
// Row src[i] of x -> row dst[i] of out (d values each), one block per row.
__global__ void gather_rows_kernel(const float *x, float *out, int d, RowPairs p) {
  const float *s = x + (int64_t)p.src[blockIdx.x] * d;
  float *o = out + (int64_t)p.dst[blockIdx.x] * d;
  for (int i = threadIdx.x; i < d; i += blockDim.x) o[i] = s[i];
}

// n 32-bit words, 16 bytes per store where both ends allow it: a wide copy
// (a host-mapped destination then takes full PCIe writes).
__global__ void copy_words_kernel(const uint32_t *src, uint32_t *dst, int n) {
  const int i4 = (blockIdx.x * blockDim.x + threadIdx.x);
  const int n4 = n / 4;
  if (i4 < n4) reinterpret_cast<uint4 *>(dst)[i4] = reinterpret_cast<const uint4 *>(src)[i4];
  const int t = n4 * 4 + i4;
  if (i4 < n - n4 * 4) dst[t] = src[t];
}

int elementwise_grid(int64_t n) { return (int)std::min<int64_t>((n + 255) / 256, 4096); }

}  // namespace

bool norm_rows_planes_ok(int d) { return d % 4 == 0 && d <= 1024 * kNormG; }

namespace {
// Rows that norm_rows_kernel takes: every pointer on 16 bytes.
bool norm_rows_ok(int d, std::initializer_list<const void *> ptrs) {
  uintptr_t bits = 0;
  for (const void *q : ptrs) bits |= reinterpret_cast<uintptr_t>(q);
  return norm_rows_planes_ok(d) && !(bits & 15);
}
bool fp16_planes_ok(const Fp16Planes &f, int d) {
  return f.lo && f.unscale && f.rows && !(reinterpret_cast<uintptr_t>(f.rows) & 15) && f.ld >= d && f.ld % 4 == 0 && f.ld <= 1024 * kNormG;
}
}  // namespace

hipError_t launch_residual_norm_rows(float *x, const float *p, int sp, const float *dd, int sd, int n, int d,
                                     const float *w, const float *b, double eps, float *out, uint16_t *oh,
                                     uint16_t *ol, hipStream_t st, Fp16Planes fp) {
  if (sp < 1 || sd < 1 || !oh != !ol || (!out && !oh && !fp.hi)) return hipErrorInvalidValue;
  if (norm_rows_ok(d, {x, p, dd, w, b, out, oh, ol}) && (!fp.hi || fp16_planes_ok(fp, d))) {
    hipLaunchKernelGGL(norm_rows_kernel<true>, dim3(n), dim3(256), 0, st, x, p, sp, dd, sd, (int64_t)n * d, d, w, b,
                       eps, out, oh, ol, d, fp);
    return hipGetLastError();
  }
  if (fp.hi) return hipErrorInvalidValue;
  const size_t lds = (size_t)((d + 3) & ~3) * 4 + 8 * sizeof(double);
  hipLaunchKernelGGL(residual_norm_rows_kernel, dim3(n), dim3(256), lds, st, x, p, sp, dd, sd, (int64_t)n * d, d, w, b,
                     eps, out, oh, ol, d);
  return hipGetLastError();
}

hipError_t launch_layer_norm_rows(const float *x, const float *w, const float *b, double eps, int n, int d,
                                  float *out, hipStream_t st, uint16_t *oh, uint16_t *ol, int ldo, Fp16Planes fp) {
  if (!oh != !ol || (ldo && ldo < d)) return hipErrorInvalidValue;
  if (norm_rows_ok(d, {x, w, b, out, oh, ol}) && ldo % 4 == 0 && (!fp.hi || fp16_planes_ok(fp, d))) {
    hipLaunchKernelGGL(norm_rows_kernel<false>, dim3(n), dim3(256), 0, st, const_cast<float *>(x), nullptr, 0, nullptr,
                       0, 0, d, w, b, eps, out, oh, ol, ldo ? ldo : d, fp);
    return hipGetLastError();
  }
  if (fp.hi) return hipErrorInvalidValue;
  const size_t lds = (size_t)((d + 3) & ~3) * 4 + 8 * sizeof(double);
  hipLaunchKernelGGL(layer_norm_rows_kernel, dim3(n), dim3(256), lds, st, x, w, b, eps, d, out, oh, ol,
                     ldo ? ldo : d);
  return hipGetLastError();
}

hipError_t launch_gemm(const MatDesc &w, const float *x, int n, float *out, hipStream_t st) {
  dim3 grid((w.rows + kTN - 1) / kTN, (n + kTM - 1) / kTM);
  hipLaunchKernelGGL(gemm_simt_kernel, grid, dim3(256), 0, st, w, x, n, out);
  return hipGetLastError();
}

hipError_t launch_in_epilogue(const StableDims &s, const KVDev &kv, const float *y, int ldy, const float *rope,
                              const int *pos0, int n, float *q, float *m, hipStream_t st, uint16_t *mh,
                              uint16_t *ml, const int *rows, int ys, int ldm) {
  if (ldy % 2 || !mh != !ml || (!m && !mh) || s.win_q % 2 || (!rows && !pos0) || ys < 1 || (ldm && ldm < s.inter))
    return hipErrorInvalidValue;
  const int units = (s.win_q + 2 * s.win_kv + 2 * s.inter) / 2;
  // each token's units over several blocks (about 8192 blocks for a chunk)
  const int per_token = std::max(1, std::min((units + 255) / 256, 8192 / std::max(1, n)));
  hipLaunchKernelGGL(in_epilogue_kernel, dim3(n, per_token), dim3(256), 0, st, s, kv, y, ldy, rope, pos0, units, q,
                     m, mh, ml, rows, ys, ldm ? ldm : s.inter);
  return hipGetLastError();
}

hipError_t launch_in_epilogue_pair(const StableDims &sa, const float *ya, int ldya, int ysa, const StableDims &sb,
                                   const float *yb, int ldyb, int ysb, const KVDev &kv, const float *rope,
                                   const int *rows, int n, float *q, float *m, hipStream_t st) {
  const StableDims *ss[2] = {&sa, &sb};
  const int ld[2] = {ldya, ldyb}, ys[2] = {ysa, ysb};
  InEpiArgs g[2];
  if (!rows || n < 1 || !ya || !yb) return hipErrorInvalidValue;
  for (int i = 0; i < 2; i++) {
    const StableDims &s = *ss[i];
    if (ld[i] % 2 || s.win_q % 2 || ys[i] < 1 || (s.inter && !m)) return hipErrorInvalidValue;
    const int units = (s.win_q + 2 * s.win_kv + 2 * s.inter) / 2;
    const int gy = std::max(1, std::min((units + 255) / 256, 8192 / n));
    g[i] = InEpiArgs{s, i ? yb : ya, ld[i], units, ys[i], gy, m};
  }
  hipLaunchKernelGGL(in_epilogue_pair_kernel, dim3(n, g[0].gy + g[1].gy), dim3(256), 0, st, g[0], g[1], kv, rope, q,
                     rows);
  return hipGetLastError();
}

hipError_t launch_residual(float *x, const float *p, int sp, const float *d, int sd, int64_t n, hipStream_t st) {
  if (sp < 1 || sd < 1) return hipErrorInvalidValue;
  hipLaunchKernelGGL(residual_kernel, dim3(elementwise_grid(n)), dim3(256), 0, st, x, p, sp, d, sd, n);
  return hipGetLastError();
}

hipError_t launch_sum_splits(float *out, const float *p, int sp, int64_t n, hipStream_t st) {
  if (sp < 1 || n < 1) return hipErrorInvalidValue;
  hipLaunchKernelGGL(sum_splits_kernel, dim3(elementwise_grid(n)), dim3(256), 0, st, out, p, sp, n);
  return hipGetLastError();
}

hipError_t launch_copy_words(const void *src, void *dst, int n, hipStream_t st) {
  if ((reinterpret_cast<uintptr_t>(src) | reinterpret_cast<uintptr_t>(dst)) & 15) return hipErrorInvalidValue;
  const int threads = 256, blocks = std::max(1, (n / 4 + threads - 1) / threads);
  hipLaunchKernelGGL(copy_words_kernel, dim3(blocks), dim3(threads), 0, st, reinterpret_cast<const uint32_t *>(src),
                     reinterpret_cast<uint32_t *>(dst), n);
  return hipGetLastError();
}

hipError_t launch_gather_rows(const float *x, float *out, int d, const int *src, const int *dst, int n, hipStream_t st) {
  for (int i0 = 0; i0 < n; i0 += kRowPairs) {
    RowPairs p{};
    const int c = std::min(n - i0, kRowPairs);
    std::copy(src + i0, src + i0 + c, p.src);
    std::copy(dst + i0, dst + i0 + c, p.dst);
    hipLaunchKernelGGL(gather_rows_kernel, dim3(c), dim3(1024), 0, st, x, out, d, p);
  }
  return hipGetLastError();
}

hipError_t launch_copy_row(const float *src, float *dst, int n, hipStream_t st) {
  hipLaunchKernelGGL(copy_kernel, dim3((n + 255) / 256), dim3(256), 0, st, src, dst, n);
  return hipGetLastError();
}
