// Products of many rows with F16, F32 and 5/6-bit weights on the gfx950
// matrix cores, no further from float64 than fp32 products with float64 totals
// of 512 columns: Y[M][N] = X[M][K] * W^T with v_mfma_f32_32x32x16_f16.
//
// What bounds it: the matrix cores, at two (F16) or three products per
// multiply-add. The vector-unit GEMM runs at about 2 TFLOP/s here, and the
// few-row kernel (kq_rows.hip) over 32-row slices reads and decodes the
// matrix once per slice.
//
// Operands: X comes as fp16 hi + lo planes of rows scaled by a power of two
// (Fp16Planes: 22 bits of a value down to 2^-16 of its row's largest; a row
// that the planes do not serve is marked, and its outputs come from its fp32
// values). F16 weights are used as stored. Other formats are decoded once per
// block to the fp32 values of mat_value, scaled by the row's power of two
// (Matrix::rscale, from the row's largest value) and split into fp16 hi + lo
// planes, which hold them as X's do (a matrix that they do not serve is marked
// at its upload and does not come here); the products are hi hi + lo hi + hi
// lo. A K step of 32 columns is summed on the matrix cores from zero and added
// to the fp32 totals, so a total rounds once per step (kExactRun columns at
// most).
//
// Tile: 128 * WM rows x 256 columns per block of eight waves (two per SIMD:
// one's decoding runs beside the other's matrix products), a wave 32 * WM x
// 128. X planes land in one of two LDS stages by buffer_load ... lds; the
// weights are loaded as stored into registers two steps ahead, and decoded
// into one of two LDS buffers of fp16 planes while the step before runs.
#include <algorithm>

#include "gemm_wide.h"
#include "plain_rows.h"

using namespace tinyoai_gemm;

namespace {

typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));

constexpr int kThreads = 512, kBN = 256;
constexpr uint32_t kNone = 0x80000000u, kPast = 0x40000000u;
constexpr int kPlane = kBN * 64;  // bytes of one weight plane of a step

// One block per row: x (fp32) -> its fp16 planes (Fp16Planes), zeros past k.
__global__ __launch_bounds__(256) void split_f16_kernel(const float *x, int64_t ldx, int k, uint16_t *hi, uint16_t *lo,
                                                        int ldo, float *unscale) {
  const int64_t row = blockIdx.x;
  uint16_t *h = hi + row * ldo, *l = lo + row * ldo;
  const __amdgpu_buffer_rsrc_t r = plane_rsrc(reinterpret_cast<const uint8_t *>(x + row * ldx), (int64_t)k * 4);
  constexpr int U = 8;  // float4 per thread held at once: rows of up to 8192 values are read once
  float4 v[U];
  auto load = [&](int i0) {
#pragma unroll
    for (int u = 0; u < U; u++) {
      const int i = i0 + 4 * ((int)threadIdx.x + 256 * u);
      const u32x4 w = __builtin_amdgcn_raw_buffer_load_b128(r, i < k ? i * 4 : (int)kNone, 0, 0);  // zeros past k
      v[u] = make_float4(__uint_as_float(w.x), __uint_as_float(w.y), __uint_as_float(w.z), __uint_as_float(w.w));
    }
  };
  __shared__ int wave_most[4], wave_vote[4];
  int most = 0, vote = 0;
  bool suspect = false;
  for (int i0 = 0; i0 < k; i0 += U * 1024) {
    load(i0);
#pragma unroll
    for (int u = 0; u < U; u++)
      most = max(max(most, max(fp16_magnitude(v[u].x), fp16_magnitude(v[u].y))),
                 max(fp16_magnitude(v[u].z), fp16_magnitude(v[u].w)));
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) most = max(most, __shfl_xor(most, o));
  if ((threadIdx.x & 63) == 0) wave_most[threadIdx.x >> 6] = most;
  __syncthreads();
  most = max(max(wave_most[0], wave_most[1]), max(wave_most[2], wave_most[3]));
  float inverse;
  const float s = fp16_scale(most, inverse);
  for (int i0 = 0; i0 < ldo; i0 += U * 1024) {
    if (k > U * 1024) load(i0);
#pragma unroll
    for (int u = 0; u < U; u++) {
      const int i = i0 + 4 * ((int)threadIdx.x + 256 * u);
      if (i >= ldo) break;
      uint2 a, b;
      fp16_split4(v[u], s, a, b);
      suspect |= fp16_suspect(v[u], most);
      *reinterpret_cast<uint2 *>(h + i) = a;
      *reinterpret_cast<uint2 *>(l + i) = b;
    }
  }
  const bool wave_suspect = __any(suspect);
  if ((threadIdx.x & 63) == 0) wave_vote[threadIdx.x >> 6] = wave_suspect;
  __syncthreads();
  bool marked = false;
  if (wave_vote[0] | wave_vote[1] | wave_vote[2] | wave_vote[3]) {
    for (int i0 = 0; i0 < k; i0 += U * 1024) {
      load(i0);
#pragma unroll
      for (int u = 0; u < U; u++)
        vote += (fp16_vote(v[u].x, most) + fp16_vote(v[u].y, most)) + (fp16_vote(v[u].z, most) + fp16_vote(v[u].w, most));
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) vote += __shfl_xor(vote, o);
    __syncthreads();
    if ((threadIdx.x & 63) == 0) wave_vote[threadIdx.x >> 6] = vote;
    __syncthreads();
    marked = (wave_vote[0] + wave_vote[1]) + (wave_vote[2] + wave_vote[3]) > 0;
  }
  if (threadIdx.x == 0) unscale[row] = marked ? -inverse : inverse;
}

template <int WF>
constexpr int planes_of() { return WF == FMT_F16 ? 1 : 2; }
template <int WM>
constexpr size_t lds_bytes() { return 2 * (size_t)(2 * 128 * WM * 64) + 2 * (size_t)2 * kPlane; }

struct ExactArgs {
  ExactProduct p[2];
  int nprod, M;
};

// One thread's weights of a step as stored: row tid / 2, values 8 h .. + 7
// and 16 + 8 h .. + 7 (h = tid % 2) of its 32.
template <int WF>
struct Stored {
  uint4 v[WF == FMT_F32 ? 4 : 2];  // 5/6-bit: v[0].x, .y the quant bytes; v[1] the block header
  uint2 h;
};
// Loads per step (the same for every thread and step).
template <int WF>
constexpr int loads_of() {
  return WF == FMT_F32 ? 4 : WF == FMT_F16 || WF == FMT_Q4_K ? 2 : WF == FMT_Q6_K ? 4 : 3;
}

template <int WF, int WM>
__device__ __forceinline__ void exact_body(const ExactArgs &g, const ExactProduct &P, int t, uint8_t *lds8) {
  constexpr int BM = 128 * WM, NW = 4, WP = planes_of<WF>();
  constexpr int kAPlane = BM * 64, kSlot = 2 * kAPlane, kB0 = 2 * kSlot;
  uint16_t *lds16 = reinterpret_cast<uint16_t *>(lds8);
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, wm = wave & 3, wn = wave >> 2;
  const int K = P.w.cols, N = P.w.rows, nk = (K + kWK - 1) / kWK;
  const int MT = (g.M + BM - 1) / BM, NT = (N + kBN - 1) / kBN, tiles = MT * NT;
  const int split = t / tiles, tt = t - split * tiles, nt = tt / MT, mt = tt - nt * MT;
  const int m0 = mt * BM, n0 = nt * kBN;
  const int k_lo = (int)((int64_t)nk * split / P.ksplit), k_hi = (int)((int64_t)nk * (split + 1) / P.ksplit);

  // ---- X: wave w loads rows (w + 8 i) * 16 .. + 15 of each plane
  const __amdgpu_buffer_rsrc_t rxh = plane_rsrc(reinterpret_cast<const uint8_t *>(P.xh), (int64_t)g.M * P.lda * 2);
  const __amdgpu_buffer_rsrc_t rxl = plane_rsrc(reinterpret_cast<const uint8_t *>(P.xl), (int64_t)g.M * P.lda * 2);
  uint32_t aoff[WM];
#pragma unroll
  for (int i = 0; i < WM; i++) {
    const int row = (wave + 8 * i) * 16 + (lane >> 2), lc = (lane & 3) ^ ((row >> 2) & 3);
    aoff[i] = m0 + row < g.M ? (uint32_t)(((m0 + row) * P.lda + lc * 8) * 2) : kNone;
  }
  const uint32_t lds_base = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) void *)lds8;
  const uint32_t wave_u = __builtin_amdgcn_readfirstlane(wave);
  auto issue_x = [&](int kb, int slot) {
    const uint32_t ka = kb < k_hi ? (uint32_t)(kb * kWK * 2) : kPast, sb = lds_base + slot * kSlot + wave_u * 1024;
#pragma unroll
    for (int i = 0; i < WM; i++) {
      lds_dma16(rxh, aoff[i] + ka, sb + i * 8192);
      lds_dma16(rxl, aoff[i] + ka, sb + kAPlane + i * 8192);
    }
  };

  // ---- weights
  const int row = tid >> 1, h = tid & 1, n = n0 + row;
  const __amdgpu_buffer_rsrc_t rv = plane_rsrc(P.w.vals, (int64_t)N * P.w.vstride);
  const __amdgpu_buffer_rsrc_t rm = plane_rsrc(P.w.meta, (int64_t)N * P.w.mstride);
  const __amdgpu_buffer_rsrc_t rh = plane_rsrc(P.w.hbits, (int64_t)N * P.w.hstride);
  const uint32_t vrow = (uint32_t)n * (uint32_t)P.w.vstride, mrow = (uint32_t)n * (uint32_t)P.w.mstride,
                 hrow = (uint32_t)n * (uint32_t)P.w.hstride;
  float rs = 1.f;  // the row's scale
  if constexpr (WF != FMT_F16) rs = P.w.rscale[min(n, N - 1)];
  auto load_w = [&](Stored<WF> &s, int kb) {
    const bool in = n < N && kb < k_hi;
    auto b128 = [](__amdgpu_buffer_rsrc_t r, uint32_t off) {
      const u32x4 v = __builtin_amdgcn_raw_buffer_load_b128(r, (int)off, 0, 0);
      return make_uint4(v.x, v.y, v.z, v.w);
    };
    if constexpr (WF == FMT_F32) {
#pragma unroll
      for (int i = 0; i < 4; i++) {  // values 16 (i / 2) + 8 h + 4 (i % 2) ..; rows zero-padded to whole chunks
        const int k = kb * kWK + 16 * (i >> 1) + 8 * h + 4 * (i & 1);
        s.v[i] = b128(rv, in && k < K ? vrow + k * 4 : kNone);
      }
    } else if constexpr (WF == FMT_F16) {
#pragma unroll
      for (int i = 0; i < 2; i++) {
        const int k = kb * kWK + 16 * i + 8 * h;
        s.v[i] = b128(rv, in && k < K ? vrow + k * 2 : kNone);
      }
    } else {
      const u32x2 q = __builtin_amdgcn_raw_buffer_load_b64(rv, in ? (int)(vrow + kb * 16 + 8 * h) : (int)kNone, 0, 0);
      s.v[0].x = q.x;
      s.v[0].y = q.y;
      if constexpr (WF == FMT_Q4_K || WF == FMT_Q5_K) s.v[1] = b128(rm, in ? mrow + (kb >> 3) * 16 : kNone);
      if constexpr (WF == FMT_Q5_1)
        s.v[1].x = __builtin_amdgcn_raw_buffer_load_b32(rm, in ? (int)(mrow + kb * 4) : (int)kNone, 0, 0);
      if constexpr (WF == FMT_Q5_1 || WF == FMT_Q5_K)
        s.h.x = __builtin_amdgcn_raw_buffer_load_b32(rh, in ? (int)(hrow + kb * 4) : (int)kNone, 0, 0);
      if constexpr (WF == FMT_Q6_K) {
        const u32x2 hb = __builtin_amdgcn_raw_buffer_load_b64(rh, in ? (int)(hrow + kb * 8) : (int)kNone, 0, 0);
        s.h = make_uint2(hb.x, hb.y);
        const uint32_t mo = in ? mrow + (kb >> 3) * 32 : kNone;
        s.v[1].x = __builtin_amdgcn_raw_buffer_load_b16(rm, (int)(in ? mo + 2 * (kb & 7) : kNone), 0, 0);
        s.v[1].y = __builtin_amdgcn_raw_buffer_load_b16(rm, (int)(in ? mo + 16 : kNone), 0, 0);
      }
    }
  };
  // Two values -> their dwords in the hi and lo planes.
  auto split2 = [](float a, float b, uint32_t &hi, uint32_t &lo) {
    const f16x2 t = __builtin_convertvector((f32x2){a, b}, f16x2);
    const f16x2 r = __builtin_convertvector((f32x2){a - (float)t.x, b - (float)t.y}, f16x2);
    hi = __builtin_bit_cast(uint32_t, t);
    lo = __builtin_bit_cast(uint32_t, r);
  };
  // The weights of step kb into plane buffer bb (fp16 rows of 64 bytes, swz).
  auto decode = [&](const Stored<WF> &s, int kb, int bb) {
    uint16_t *wb = lds16 + (kB0 + bb * 2 * kPlane) / 2;
    auto put = [&](int c, const uint32_t (&hi)[4], const uint32_t (&lo)[4]) {
      *reinterpret_cast<uint4 *>(wb + swz(row, c)) = make_uint4(hi[0], hi[1], hi[2], hi[3]);
      *reinterpret_cast<uint4 *>(wb + kPlane / 2 + swz(row, c)) = make_uint4(lo[0], lo[1], lo[2], lo[3]);
    };
    if constexpr (WF == FMT_F16) {
#pragma unroll
      for (int i = 0; i < 2; i++) *reinterpret_cast<uint4 *>(wb + swz(row, 2 * i + h)) = s.v[i];
    } else if constexpr (WF == FMT_F32) {
#pragma unroll
      for (int i = 0; i < 2; i++) {
        uint32_t hi[4], lo[4];
#pragma unroll
        for (int j = 0; j < 2; j++) {
          const uint4 v = s.v[2 * i + j];
          split2(__uint_as_float(v.x) * rs, __uint_as_float(v.y) * rs, hi[2 * j], lo[2 * j]);
          split2(__uint_as_float(v.z) * rs, __uint_as_float(v.w) * rs, hi[2 * j + 1], lo[2 * j + 1]);
        }
        put(2 * i + h, hi, lo);
      }
    } else {
      // The block's constants times the row's scale (a power of two: the
      // values below are mat_value's times it, every rounding the same).
      KConst k{};
      if constexpr (WF == FMT_Q6_K) {
        const float d = hw_half((uint16_t)s.v[1].y);
        k.a = d * (float)(int8_t)s.v[1].x;
        k.a2 = d * (float)(int8_t)(s.v[1].x >> 8);
      } else {
        k = kquant_const<WF>(s.v[1], 0, kb);
      }
      k.a *= rs;
      k.a2 *= rs;
      k.b *= rs;
      const uint32_t q[2] = {s.v[0].x, s.v[0].y};
#pragma unroll
      for (int i = 0; i < 2; i++) {  // values 16 i + 8 h + e
        const uint32_t hb = WF == FMT_Q6_K ? (i ? s.h.y : s.h.x) >> (16 * h) : s.h.x >> (16 * i + 8 * h);
        float v[8];
#pragma unroll
        for (int e = 0; e < 8; e++) {
          int x = (q[e >> 2] >> (8 * (e & 3) + 4 * i)) & 15;
          if constexpr (WF == FMT_Q5_1 || WF == FMT_Q5_K) x |= ((hb >> e) & 1) << 4;
          if constexpr (WF == FMT_Q6_K) x |= ((hb >> (2 * e)) & 3) << 4;
          v[e] = kquant_value<WF>(k, x, 16 * i + e);
        }
        uint32_t hi[4], lo[4];
#pragma unroll
        for (int j = 0; j < 4; j++) split2(v[2 * j], v[2 * j + 1], hi[j], lo[j]);
        put(2 * i + h, hi, lo);
      }
    }
  };

  f32x16 acc[WM][NW];
#pragma unroll
  for (int f = 0; f < WM; f++)
#pragma unroll
    for (int j = 0; j < NW; j++)
#pragma unroll
      for (int v = 0; v < 16; v++) acc[f][j][v] = 0.f;
  const int arow = wm * 32 * WM + (lane & 31), brow = wn * 128 + (lane & 31);
  auto frag = [&](const uint16_t *base, int r, int s) {
    return *reinterpret_cast<const f16x8 *>(base + swz(r, 2 * (lane >> 5) + s));
  };
  const f32x16 zero = {};
  auto compute = [&](int slot, int bb) {
    const uint16_t *st = lds16 + slot * (kSlot / 2);
    const uint16_t *wb = lds16 + (kB0 + bb * 2 * kPlane) / 2;
    f16x8 af[2][WM][2];
#pragma unroll
    for (int s = 0; s < 2; s++)
#pragma unroll
      for (int f = 0; f < WM; f++)
#pragma unroll
        for (int p = 0; p < 2; p++) af[s][f][p] = frag(st + p * (kAPlane / 2), arow + f * 32, s);
#pragma unroll
    for (int j = 0; j < NW; j++) {
      f32x16 t[WM];
      f16x8 bf[2][WP];
#pragma unroll
      for (int s = 0; s < 2; s++)
#pragma unroll
        for (int p = 0; p < WP; p++) bf[s][p] = frag(wb + p * (kPlane / 2), brow + j * 32, s);
      // the small products first
#pragma unroll
      for (int s = 0; s < 2; s++)
#pragma unroll
        for (int f = 0; f < WM; f++) t[f] = __builtin_amdgcn_mfma_f32_32x32x16_f16(af[s][f][1], bf[s][0], s ? t[f] : zero, 0, 0, 0);
      if constexpr (WP == 2) {
#pragma unroll
        for (int s = 0; s < 2; s++)
#pragma unroll
          for (int f = 0; f < WM; f++) t[f] = __builtin_amdgcn_mfma_f32_32x32x16_f16(af[s][f][0], bf[s][1], t[f], 0, 0, 0);
      }
#pragma unroll
      for (int s = 0; s < 2; s++)
#pragma unroll
        for (int f = 0; f < WM; f++) t[f] = __builtin_amdgcn_mfma_f32_32x32x16_f16(af[s][f][0], bf[s][0], t[f], 0, 0, 0);
#pragma unroll
      for (int f = 0; f < WM; f++)
#pragma unroll
        for (int v = 0; v < 16; v++) acc[f][j][v] = __fadd_rn(acc[f][j][v], t[f][v]);
      // the totals are formed here, not at their next use: the products die
#pragma unroll
      for (int f = 0; f < WM; f++) asm volatile("" : "+v"(acc[f][j]));
    }
  };

  // Step kb: X of kb and the weights of kb + 1 have landed (those of kb + 2
  // may be in flight); after the barrier X of kb + 1 goes to the other
  // stage (free: every wave is past step kb - 1), the weights of kb + 1 are
  // decoded and their registers refilled with kb + 3.
  constexpr int kLoads = loads_of<WF>();
  Stored<WF> s0, s1;
  issue_x(k_lo, 0);
  load_w(s0, k_lo);
  load_w(s1, k_lo + 1);
  wait_vmcnt<kLoads>();
  decode(s0, k_lo, 0);
  load_w(s0, k_lo + 2);
  auto step = [&](int kb, int par, Stored<WF> &s) {  // par: kb - k_lo mod 2; s: the weights of kb + 1
    wait_vmcnt<kLoads>();
    __syncthreads();
    issue_x(kb + 1, par ^ 1);
    decode(s, kb + 1, par ^ 1);  // past k_hi: zeros, never read
    load_w(s, kb + 3);
    // with 256 rows the decoding's registers must be free before the products'
    if constexpr (WM == 2) __builtin_amdgcn_sched_barrier(0);
    compute(par, par);
  };
  int kb = k_lo;
#pragma unroll 1
  for (; kb + 2 <= k_hi; kb += 2) {
    step(kb, 0, s1);
    step(kb + 1, 1, s0);
  }
  if (kb < k_hi) step(kb, 0, s1);
  wait_vmcnt<0>();  // no load may land in LDS after the block ends

  // D fragment: lane holds column lane % 32 of rows (v / 4) * 8 + (lane / 32) * 4 + v % 4.
  float *y = P.y + (int64_t)split * P.split_stride;
  bool marked = false;
  // Both factors as one exponent: a total of 1e36 times X's factor alone may
  // pass the range before the weights' brings it back.
  int ew[NW];
#pragma unroll
  for (int j = 0; j < NW; j++) {
    ew[j] = 0;
    if constexpr (WF != FMT_F16) ew[j] = 127 - (int)(__float_as_uint(P.w.rscale[min(n0 + brow + j * 32, N - 1)]) >> 23);
  }
#pragma unroll
  for (int f = 0; f < WM; f++)
#pragma unroll
    for (int v = 0; v < 16; v++) {
      const int m = m0 + wm * 32 * WM + f * 32 + (v >> 2) * 8 + (lane >> 5) * 4 + (v & 3);
      if (m >= g.M) continue;
      const int u = __float_as_int(P.unscale[m]), ex = (u >> 23) - 127;
      marked |= u < 0;
      if (u < 0) continue;
#pragma unroll
      for (int j = 0; j < NW; j++) {
        const int c = n0 + brow + j * 32;
        if (c < N) y[(int64_t)m * P.ldy + c] = __builtin_ldexpf(acc[f][j][v], ex + ew[j]);
      }
    }
  if (!__any(marked)) return;
  const int mw = m0 + wm * 32 * WM, c0 = n0 + wn * 128;
  const uint64_t rows = __ballot(lane < 32 * WM && mw + lane < g.M && P.unscale[min(mw + lane, g.M - 1)] < 0.f);
  plain_rows<WF>(P.w, P.x, P.ldx, rows, mw, c0, min(c0 + 128, N), k_lo * kWK, min(K, k_hi * kWK), y, P.ldy);
}

template <int WM>
int tiles_of(const ExactArgs &g, int i) {
  const ExactProduct &p = g.p[i];
  return ((g.M + 128 * WM - 1) / (128 * WM)) * ((p.w.rows + kBN - 1) / kBN) * p.ksplit;
}
// The launch's tiles in runs over the 8 XCDs (blocks go to them round-robin):
// XCD x takes tiles [x * per, (x + 1) * per) of both products together, so one
// XCD's blocks share weight tiles and none holds more than its share. (A run
// per product gave seven XCDs 33 blocks for 32 CUs where the whole launch had
// 252: 472 us instead of 280 for 700 rows of 21504 x 2560.)
__device__ __forceinline__ int tile_of(int per) { return ((int)blockIdx.x & 7) * per + ((int)blockIdx.x >> 3); }

template <int WF, int WM>
__global__ __launch_bounds__(kThreads) void gemm_exact_kernel(ExactArgs g, int tiles, int per) {
  extern __shared__ __align__(16) uint8_t exact_lds[];
  const int t = tile_of(per);
  if (t < tiles) exact_body<WF, WM>(g, g.p[0], t, exact_lds);
}
// Two products of the same rows (their own planes, formats and splits), the
// second's tiles after the first's.
template <int WFA, int WFB, int WM>
__global__ __launch_bounds__(kThreads) void gemm_exact_pair_kernel(ExactArgs g, int tiles0, int tiles, int per) {
  extern __shared__ __align__(16) uint8_t exact_lds[];
  const int t = tile_of(per);
  if (t < tiles0)
    exact_body<WFA, WM>(g, g.p[0], t, exact_lds);
  else if (t < tiles)
    exact_body<WFB, WM>(g, g.p[1], t - tiles0, exact_lds);
}

template <int WF, int WM>
hipError_t exact_launch(const ExactArgs &g, hipStream_t st) {
  constexpr size_t lds = lds_bytes<WM>();
  static const hipError_t attr = hipFuncSetAttribute(reinterpret_cast<const void *>(&gemm_exact_kernel<WF, WM>),
                                                     hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
  if (attr != hipSuccess) return attr;
  const int tiles = tiles_of<WM>(g, 0), per = (tiles + 7) / 8;
  hipLaunchKernelGGL((gemm_exact_kernel<WF, WM>), dim3(8 * per), dim3(kThreads), lds, st, g, tiles, per);
  return hipGetLastError();
}
template <int WFA, int WFB, int WM>
hipError_t exact_pair_launch(const ExactArgs &g, hipStream_t st) {
  constexpr size_t lds = lds_bytes<WM>();
  static const hipError_t attr = hipFuncSetAttribute(reinterpret_cast<const void *>(&gemm_exact_pair_kernel<WFA, WFB, WM>),
                                                     hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
  if (attr != hipSuccess) return attr;
  const int t0 = tiles_of<WM>(g, 0), tiles = t0 + tiles_of<WM>(g, 1), per = (tiles + 7) / 8;
  hipLaunchKernelGGL((gemm_exact_pair_kernel<WFA, WFB, WM>), dim3(8 * per), dim3(kThreads), lds, st, g, t0, tiles, per);
  return hipGetLastError();
}

template <int WM>
hipError_t exact_dispatch(const ExactArgs &g, hipStream_t st) {
  if (g.nprod == 2) {
    const int a = g.p[0].w.fmt, b = g.p[1].w.fmt;
    if (a == FMT_Q6_K && b == FMT_Q4_K) return exact_pair_launch<FMT_Q6_K, FMT_Q4_K, WM>(g, st);
    if (a == FMT_Q4_K && b == FMT_Q6_K) return exact_pair_launch<FMT_Q4_K, FMT_Q6_K, WM>(g, st);
    if (a == FMT_Q5_K && b == FMT_Q5_K) return exact_pair_launch<FMT_Q5_K, FMT_Q5_K, WM>(g, st);
    if (a == FMT_F16 && b == FMT_F16) return exact_pair_launch<FMT_F16, FMT_F16, WM>(g, st);
    return hipErrorInvalidValue;
  }
  switch (g.p[0].w.fmt) {
    case FMT_F16: return exact_launch<FMT_F16, WM>(g, st);
    case FMT_F32: return exact_launch<FMT_F32, WM>(g, st);
    case FMT_Q4_K: return exact_launch<FMT_Q4_K, WM>(g, st);
    case FMT_Q5_K: return exact_launch<FMT_Q5_K, WM>(g, st);
    case FMT_Q6_K: return exact_launch<FMT_Q6_K, WM>(g, st);
    case FMT_Q5_1: return exact_launch<FMT_Q5_1, WM>(g, st);
    default: return hipErrorInvalidValue;
  }
}

}  // namespace

hipError_t launch_split_f16(const float *x, int64_t ldx, int k, int rows, uint16_t *hi, uint16_t *lo, int ldo,
                            float *unscale, hipStream_t st) {
  if (rows < 1 || k < 1 || ldo < k || ldo % 4 || ldx < k) return hipErrorInvalidValue;
  hipLaunchKernelGGL(split_f16_kernel, dim3(rows), dim3(256), 0, st, x, ldx, k, hi, lo, ldo, unscale);
  return hipGetLastError();
}

// Planes of less than 1 GiB: the kernel's offsets are 32 bits, with kPast
// (2^30) added to those past a range, and must stay past every plane.
bool gemm_exact_supported(const Matrix &w, int M, int max_splits) {
  constexpr int64_t kGiB = int64_t(1) << 30;
  const bool fmt = w.fmt == FMT_F16 || ((w.fmt == FMT_F32 || is_kquant(w.fmt)) && w.rscale);
  return fmt && !w.special && M >= 2 && gemm_exact_min_splits(w) <= max_splits && w.cols >= 2 * kWK && w.vstride % 16 == 0 &&
         (reinterpret_cast<uintptr_t>(w.vals) & 15) == 0 && (int64_t)w.rows * w.vstride < kGiB &&
         (int64_t)w.rows * w.mstride < kGiB && (int64_t)M * gemm_exact_ld(w) * 2 < kGiB;
}

// (each pair is two more kernels to compile: there are those that the K-quant
// mix, F16 and Q5_K models form; others, a whole model of Q4_K or Q6_K among
// them, run as two launches, and what a pair would give there is not measured)
bool gemm_exact_pair_supported(int a, int b) {
  return (a == FMT_Q6_K && b == FMT_Q4_K) || (a == FMT_Q4_K && b == FMT_Q6_K) || (a == b && (a == FMT_Q5_K || a == FMT_F16));
}

ExactPlan gemm_exact_plan(int M, const MatDesc &a, const MatDesc *b, int max_splits) {
  ExactPlan best;
  double cost = 1e30;
  for (int f = 2; f >= 1; f--) {
    const int64_t mt = (M + 128 * f - 1) / (128 * f), ta = mt * ((a.rows + kBN - 1) / kBN),
                  tb = b ? mt * ((b->rows + kBN - 1) / kBN) : 0;
    const int ka = (a.cols + kWK - 1) / kWK, kb = b ? (b->cols + kWK - 1) / kWK : 0;
    // blocks of at most `steps` K steps each, whichever product they work for
    for (int steps = 8; steps <= std::min(std::max({ka, kb, 8}), kExactRun / kWK); steps++) {
      const int sa = std::min((ka + steps - 1) / steps, max_splits);
      const int sb = b ? std::min((kb + steps - 1) / steps, max_splits) : 0;
      const int longest = std::max((ka + sa - 1) / sa, b ? (kb + sb - 1) / sb : 0);
      const double rounds = (double)((ta * sa + tb * sb + 255) / 256);
      // a step's time, a block's start and end in steps, and the partial
      // outputs (written and read) over the steps of the chip
      const double step = f == 2 ? 3.4 : 2.3;
      const double c = rounds * (longest + 6) * step + 8e-6 / 5 * M * ((sa - 1.0) * a.rows + (b ? (sb - 1.0) * b->rows : 0));
      if (c < cost) cost = c, best = ExactPlan{f == 2, sa, sb};
    }
  }
  return best;
}

hipError_t launch_gemm_exact(const ExactProduct *p, int nprod, int M, bool tall, hipStream_t st) {
  if (nprod < 1 || nprod > 2) return hipErrorInvalidValue;
  ExactArgs g{};
  g.nprod = nprod;
  g.M = M;
  for (int i = 0; i < nprod; i++) {
    const ExactProduct &q = p[i];
    if (!gemm_exact_supported(q.w, M, q.ksplit) || !q.x || q.ldx < q.w.cols || !q.xh || !q.xl || !q.unscale || !q.y || q.lda < gemm_exact_ld(q.w) ||
        q.lda % 8 || ((reinterpret_cast<uintptr_t>(q.xh) | reinterpret_cast<uintptr_t>(q.xl)) & 15) || q.ksplit < 1 ||
        q.ksplit > (q.w.cols + kWK - 1) / kWK || (q.ksplit > 1 && q.split_stride < (int64_t)M * q.ldy))
      return hipErrorInvalidValue;
    g.p[i] = q;
  }
  return tall ? exact_dispatch<2>(g, st) : exact_dispatch<1>(g, st);
}
