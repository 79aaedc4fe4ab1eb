// Products of a few activation rows (2 to 64) with an F16, BF16 or Q8_0
// matrix on the gfx950 matrix cores: Y[M][N] = X[M][K] * W^T.
//
// What bounds it: the matrix is read once from HBM, so the weight stream
// should never wait. A wave owns one tile of 32 matrix rows and streams it in
// batches of 128 bytes a row, up to four batches in flight in registers, each
// load instruction covering 8 rows' whole 128 bytes; a batch then goes
// through a buffer of the wave's own in LDS into the fragment layout of
// v_mfma_f32_32x32x16. (Loads in the fragment layout itself, a row per lane,
// keep the address unit busy for 64 cycles an instruction, one cache access
// per lane: 33 us for the 21504 x 2560 Q8_0 product of 19 rows.) X is what
// the eight waves of a block share: a segment of its columns sits in LDS as
// two 16-bit planes, formed by the block from the fp32 rows, so no launch
// prepares operands and there is no barrier inside a segment. The 128-row
// tiles (gemm.hip) do 128 / M of their work for padding at these sizes and
// keep one K step of loads in flight.
//
// Operands: F16 and Q8_0 weights take X as fp16 hi + lo planes of the row
// scaled by a power of two (its largest value in the segment lands in
// [2^14, 2^15), so nothing overflows, and hi + lo carry 22 bits of a value
// down to 2^-16 of the largest, 16 down to 2^-22). A row with 256 columns that
// this does not serve is marked, and its outputs come from its fp32 values
// (plain_rows): where most of the groups of four values that are not all zero
// lie below 2^-16 of the segment's largest (Q8_0: 2^-22, since two bf16 planes
// would carry 16 bits of every value). Q8_0 quants are exact in fp16, each
// quant block's product is formed unscaled and added as acc += d * block. BF16
// weights take bf16 hi + lo planes (16 bits, as the wide tiles). Each
// segment's sums (F16: every 1024 columns') are unscaled and added to fp32
// totals.
//
// K ranges (splits) write partial outputs, split s at y + s * split_stride,
// which the consumer sums in order.
#include <algorithm>
#include <type_traits>

#include "kernels.h"
#include "plain_rows.h"

namespace {

typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

constexpr int kT = 512, kWaves = 8, kTile = 32, kBlockRows = kWaves * kTile;
constexpr int kItem = 256;                  // columns of one row a wave stages at once
constexpr int kItems = 8;                   // staging items per wave and segment (64 KB of planes)
constexpr uint32_t kNone = 0x80000000u;     // past every operand: the buffer load reads zeros

struct FewArgs {
  FewProduct p[2];
  int nprod, M;
  int seg;  // columns per segment, a multiple of kItem with M * seg / kItem <= kWaves * kItems
};

// A batch is 128 bytes of each of the wave's 32 rows: 64 columns (F16,
// BF16) or 128 (Q8_0, four quant blocks).
__host__ __device__ constexpr int batch_cols(int fmt) { return fmt == FMT_Q8_0 ? 128 : 64; }
constexpr int kBatchBytes = 32 * 128, kScaleBytes = 32 * 8;  // a wave's batch in LDS, then (Q8_0) its scales
constexpr int kWaveBytes = 2 * (kBatchBytes + kScaleBytes);  // two of them
// Batches in flight per wave; a segment holds whole rounds of them.
constexpr int few_stages(int fmt, int mt) { return fmt == FMT_Q8_0 && mt > 1 ? 2 : 4; }

// A lane's part of a batch: 16-byte chunk lane % 8 of rows 8 i + lane / 8;
// Q8_0: scales 2 (lane % 2), + 1 of row lane / 2.
struct Raw {
  uint4 v[4];
  uint32_t d;
};

template <int WF>
__device__ __forceinline__ f32x16 mfma(uint4 a, uint4 b, f32x16 c) {
  if constexpr (WF == FMT_BF16)
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0,
                                                   0, 0);
  else
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), c, 0, 0,
                                                  0);
}

// 8 quants (two dwords) -> fp16, exact: the byte q + 128 below 0x64 is the
// fp16 number 1024 + q + 128, whose distance to 1152 is a small integer.
__device__ __forceinline__ uint4 q8_to_f16(uint32_t lo, uint32_t hi) {
  auto two = [](uint32_t v, uint32_t sel) {
    const f16x2 m = __builtin_bit_cast(f16x2, __builtin_amdgcn_perm(0x64646464u, v, sel));
    return __builtin_bit_cast(uint32_t, m - f16x2{(_Float16)1152.f, (_Float16)1152.f});
  };
  const uint32_t a = lo ^ 0x80808080u, b = hi ^ 0x80808080u;
  return make_uint4(two(a, 0x04010400u), two(a, 0x04030402u), two(b, 0x04010400u), two(b, 0x04030402u));
}

// The largest of the wave's 64 values.
__device__ __forceinline__ uint32_t wave_max(uint32_t v) {
  auto step = [&](auto ctrl) {
    v = max(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, decltype(ctrl)::value, 0xf, 0xf, false));
  };
  step(std::integral_constant<int, 0xb1>{});   // quad_perm [1, 0, 3, 2]
  step(std::integral_constant<int, 0x4e>{});   // quad_perm [2, 3, 0, 1]
  step(std::integral_constant<int, 0x141>{});  // row_half_mirror
  step(std::integral_constant<int, 0x128>{});  // row_ror 8
  const uint32_t a = __builtin_amdgcn_readlane(v, 0), b = __builtin_amdgcn_readlane(v, 16);
  const uint32_t c = __builtin_amdgcn_readlane(v, 32), d = __builtin_amdgcn_readlane(v, 48);
  return max(max(a, b), max(c, d));
}

// Block-wide layout: LDS row r of the planes starts at r * pitch; each group
// of 128 columns takes 512 bytes, hi then lo, its 16-byte chunk c at
// position c ^ (r & 15), so the 16 rows that one cycle of a fragment read
// covers hit distinct banks.
template <int WF, int MT>
__global__ __launch_bounds__(kT) __attribute__((amdgpu_waves_per_eu(2, 2))) void few_rows_kernel(FewArgs g) {
  extern __shared__ __align__(16) uint8_t lds[];
  __shared__ uint32_t item_max[kWaves * kItems];
  __shared__ uint32_t marks[2];  // rows to take from their fp32 values
  __shared__ __align__(16) float unscale[MT * 32];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  int b = blockIdx.x, pi = 0;
  const int nb0 = g.p[0].ks * ((g.p[0].w.rows + kBlockRows - 1) / kBlockRows);
  if (b >= nb0) {
    b -= nb0;
    pi = 1;
  }
  const FewProduct &P = g.p[pi];
  constexpr bool Q8 = WF == FMT_Q8_0;
  constexpr int kStep = batch_cols(WF), kStages = few_stages(WF, MT), kUnits = kStep / 32;
  constexpr int kVal = Q8 ? 1 : 2;  // bytes of a value
  const int N = P.w.rows, K = P.w.cols, M = g.M, nk = (K + kStep - 1) / kStep;
  const int nblk = (N + kBlockRows - 1) / kBlockRows, split = b / nblk;
  const int n0 = (b - split * nblk) * kBlockRows + wave * kTile, n = n0 + (lane & 31), h = lane >> 5;
  const int kb_lo = (int)((int64_t)nk * split / P.ks), kb_hi = (int)((int64_t)nk * (split + 1) / P.ks);

  const __amdgpu_buffer_rsrc_t rw = plane_rsrc(P.w.vals, (int64_t)N * P.w.vstride);
  const __amdgpu_buffer_rsrc_t rm = plane_rsrc(P.w.meta, (int64_t)N * P.w.mstride);
  const int lrow = n0 + (lane >> 3), lcol = (lane & 7) * (16 / kVal);  // this lane's chunk of load 0
  const uint32_t wbase = (uint32_t)lrow * (uint32_t)P.w.vstride + (lane & 7) * 16, wstep = 8 * (uint32_t)P.w.vstride;
  const uint32_t mbase = (uint32_t)(n0 + (lane >> 1)) * (uint32_t)P.w.mstride + (lane & 1) * 4;
  auto issue = [&](Raw &r, int kb) {
    // rows are zero-padded to whole chunks; past K the next section may follow
    const bool in = kb < kb_hi && kb * kStep + lcol < K;
#pragma unroll
    for (int i = 0; i < 4; i++) {
      const u32x4 v = __builtin_amdgcn_raw_buffer_load_b128(
          rw, in && lrow + 8 * i < N ? (int)(wbase + i * wstep + kb * 128) : (int)kNone, 0, 0);
      r.v[i] = make_uint4(v.x, v.y, v.z, v.w);
    }
    if constexpr (Q8) {
      const bool ok = kb < kb_hi && n0 + (lane >> 1) < N && kb * kStep + (lane & 1) * 64 < K;
      r.d = __builtin_amdgcn_raw_buffer_load_b32(rm, ok ? (int)(mbase + kb * 8) : (int)kNone, 0, 0);
    }
  };

  // The wave's two batch buffers: chunk c of row r at position
  // c ^ ((r >> 1) & 7) of its 128 bytes, so 16 rows' reads of a chunk hit
  // distinct banks.
  uint8_t *wbuf = lds + (size_t)M * g.seg * 4 + wave * kWaveBytes;
  const int srow = lane >> 3;
  const uint32_t sput = (uint32_t)srow * 128 + (((lane & 7) ^ ((srow >> 1) & 7)) << 4);
  auto put = [&](const Raw &r, int buf) {
    uint8_t *p = wbuf + buf * (kBatchBytes + kScaleBytes);
#pragma unroll
    for (int i = 0; i < 4; i++)  // row srow + 8 i: the swizzle's bit 2 flips with i's bit 0
      *reinterpret_cast<uint4 *>(p + ((sput ^ ((i & 1) << 6)) + i * 1024)) = r.v[i];
    if constexpr (Q8) *reinterpret_cast<uint32_t *>(p + kBatchBytes + lane * 4) = r.d;
  };
  const uint32_t wrow = (lane & 31) * 128, wx = (((lane & 31) >> 1) & 7) ^ h;

  const uint32_t pitch = (uint32_t)g.seg * 4;
  uint32_t xrow[MT], xor_[MT];
#pragma unroll
  for (int mt = 0; mt < MT; mt++) {
    const int r = min(mt * 32 + (lane & 31), M - 1);  // rows past M repeat the last one, never stored
    xrow[mt] = (uint32_t)r * pitch;
    xor_[mt] = (Q8 ? 2 * h : h) ^ (r & 15);
  }
  f32x16 acc[MT], tot[MT];
#pragma unroll
  for (int mt = 0; mt < MT; mt++)
#pragma unroll
    for (int v = 0; v < 16; v++) acc[mt][v] = tot[mt][v] = 0.f;
  const f32x16 zero = {};
  // The fragments of a unit of 32 columns (unit u of batch kb of the
  // segment, in the wave's buffer buf): X's two planes, the weights, and for
  // Q8_0 the unit's block scale. They are read one unit ahead of the
  // products (a read placed before its product would leave the wave waiting
  // for LDS most of the time), which the scheduling barriers keep in place.
  struct Frags {
    uint4 x[2][2][MT];  // [16-column step][plane][row tile]
    uint4 w[Q8 ? 1 : 2];
    uint32_t d;
  };
  auto read = [&](Frags &f, int kb, int u, int buf) {
    const int c0 = kb * (kStep / 8) + 4 * u;  // the unit's first 8-column chunk
    const uint32_t grp = (uint32_t)(c0 >> 4) * 512;
    const uint8_t *p = wbuf + buf * (kBatchBytes + kScaleBytes);
    // (the empty asm keeps every unit's addresses from being formed ahead and
    // held in registers)
    uint32_t wo = wx;
    asm volatile("" : "+v"(wo));
#pragma unroll
    for (int mt = 0; mt < MT; mt++) asm volatile("" : "+v"(xor_[mt]));
#pragma unroll
    for (int s = 0; s < 2; s++)
#pragma unroll
      for (int mt = 0; mt < MT; mt++) {
        const uint8_t *q = lds + xrow[mt] + grp + ((xor_[mt] ^ ((c0 & 12) | (Q8 ? s : 2 * s))) << 4);
        f.x[s][0][mt] = *reinterpret_cast<const uint4 *>(q);
        f.x[s][1][mt] = *reinterpret_cast<const uint4 *>(q + 256);
      }
    if constexpr (Q8) {  // lane half h holds values 16 h .. 16 h + 15 of the block
      f.w[0] = *reinterpret_cast<const uint4 *>(p + wrow + ((wo ^ (2 * u)) << 4));
      f.d = *reinterpret_cast<const uint16_t *>(p + kBatchBytes + (lane & 31) * 8 + 2 * u);
    } else {
#pragma unroll
      for (int s = 0; s < 2; s++) f.w[s] = *reinterpret_cast<const uint4 *>(p + wrow + ((wo ^ (4 * u + 2 * s)) << 4));
    }
  };
  auto compute = [&](const Frags &f) {
    if constexpr (Q8) {
      const uint4 b[2] = {q8_to_f16(f.w[0].x, f.w[0].y), q8_to_f16(f.w[0].z, f.w[0].w)};
      const float d = hw_half((uint16_t)f.d);
      f32x16 t[MT];
#pragma unroll
      for (int s = 0; s < 2; s++)
#pragma unroll
        for (int p = 0; p < 2; p++)
#pragma unroll
          for (int mt = 0; mt < MT; mt++) t[mt] = mfma<WF>(f.x[s][p][mt], b[s], s || p ? t[mt] : zero);
#pragma unroll
      for (int mt = 0; mt < MT; mt++)
#pragma unroll
        for (int v = 0; v < 16; v++) acc[mt][v] = fmaf(d, t[mt][v], acc[mt][v]);
      // the sums are formed here, not at their next use: the products die
#pragma unroll
      for (int mt = 0; mt < MT; mt++) asm volatile("" : "+v"(acc[mt]));
    } else {
#pragma unroll
      for (int s = 0; s < 2; s++)
#pragma unroll
        for (int p = 0; p < 2; p++)
#pragma unroll
          for (int mt = 0; mt < MT; mt++) acc[mt] = mfma<WF>(f.x[s][p][mt], f.w[s], acc[mt]);
    }
  };

  // The sums so far, unscaled, to the totals.
  auto fold = [&]() {
#pragma unroll
    for (int mt = 0; mt < MT; mt++)
#pragma unroll
      for (int r = 0; r < 4; r++) {
        float4 u = make_float4(1.f, 1.f, 1.f, 1.f);
        if constexpr (WF != FMT_BF16) u = *reinterpret_cast<const float4 *>(&unscale[mt * 32 + r * 8 + h * 4]);
        const float us[4] = {u.x, u.y, u.z, u.w};
#pragma unroll
        for (int e = 0; e < 4; e++) {
          tot[mt][r * 4 + e] = fmaf(acc[mt][r * 4 + e], us[e], tot[mt][r * 4 + e]);
          acc[mt][r * 4 + e] = 0.f;
        }
      }
  };

  const __amdgpu_buffer_rsrc_t rx =
      plane_rsrc(reinterpret_cast<const uint8_t *>(P.x), ((int64_t)(M - 1) * P.ldx + K) * 4);
  const int ipr = g.seg / kItem, items = M * ipr, segb = g.seg / kStep, k_end = min(K, kb_hi * kStep);
  Raw ring[kStages];
#pragma unroll
  for (int j = 0; j < kStages; j++) issue(ring[j], kb_lo + j);
  bool first = true;
  constexpr uint32_t kSmall = (Q8 ? 22u : 16u) << 23;  // 2^22, 2^16 in the bits of a ratio
  if (WF != FMT_BF16 && tid < 2) marks[tid] = 0;
#pragma unroll 1
  for (int kb0 = kb_lo; kb0 < kb_hi; kb0 += segb) {
    // X columns [kStep kb0, + seg) of every row -> planes in LDS (zeros past
    // the range). Item it: 256 columns of row it / ipr. (X's loads ahead of
    // the first batches': the same times.)
    float4 xv[kItems];
#pragma unroll
    for (int j = 0; j < kItems; j++) {
      const int it = wave + kWaves * j, row = it / ipr, k = kb0 * kStep + (it - row * ipr) * kItem + lane * 4;
      const u32x4 v = __builtin_amdgcn_raw_buffer_load_b128(
          rx, it < items && k < k_end ? (int)(((uint32_t)row * (uint32_t)P.ldx + k) * 4) : (int)kNone, 0, 0);
      xv[j].x = __uint_as_float(v.x);
      xv[j].y = k + 1 < k_end ? __uint_as_float(v.y) : 0.f;
      xv[j].z = k + 2 < k_end ? __uint_as_float(v.z) : 0.f;
      xv[j].w = k + 3 < k_end ? __uint_as_float(v.w) : 0.f;
    }
    __syncthreads();  // every wave is past the previous segment's planes
    if constexpr (WF != FMT_BF16) {
      // the largest finite magnitude of each item, as ordered bits
      auto mag = [](float f) {
        const uint32_t u = __float_as_uint(f) & 0x7fffffffu;
        return u < 0x7f800000u ? u : 0u;
      };
#pragma unroll
      for (int j = 0; j < kItems; j++) {
        const uint32_t m =
            wave_max(max(max(mag(xv[j].x), mag(xv[j].y)), max(mag(xv[j].z), mag(xv[j].w))));
        if (lane == 0) item_max[wave + kWaves * j] = m;
      }
      __syncthreads();
    }
    uint32_t l4 = lane * 4;
    if constexpr (MT > 1) asm volatile("" : "+v"(l4));  // (addresses held from segment to segment were spilled)
    uint32_t small = 0;
#pragma unroll
    for (int j = 0; j < kItems; j++) {
      const int it = wave + kWaves * j;
      if (it >= items) break;
      const int row = it / ipr, q = it - row * ipr;
      float s = 1.f;
      if constexpr (WF != FMT_BF16) {
        // 2^(14 - e) of the row's largest value (in [2^e, 2^(e+1))): an exact
        // scaling, its inverse a normal number too.
        const uint32_t m = wave_max(lane < ipr ? item_max[row * ipr + lane] : 0u);
        const int e = min(max((int)(m >> 23) - 127, -112), 127);
        s = __uint_as_float((uint32_t)(127 + 14 - e) << 23);
        if (q == 0 && lane == 0) unscale[row] = __uint_as_float((uint32_t)(127 - 14 + e) << 23);
        // a lane's group of four below kSmall of the largest, but not zero
        // (0 - 1 is the largest number)
        const float a = fmaxf(fmaxf(fabsf(xv[j].x), fabsf(xv[j].y)), fmaxf(fabsf(xv[j].z), fabsf(xv[j].w)));
        small += __float_as_uint(a) - 1 < max(m, kSmall + 1) - kSmall - 1;
      }
      const float f[4] = {xv[j].x * s, xv[j].y * s, xv[j].z * s, xv[j].w * s};
      uint32_t hi[4], lo[4];
#pragma unroll
      for (int e = 0; e < 4; e++) {
        if constexpr (WF == FMT_BF16) {
          const __bf16 a = (__bf16)f[e];
          hi[e] = __builtin_bit_cast(uint16_t, a);
          lo[e] = __builtin_bit_cast(uint16_t, (__bf16)(f[e] - (float)a));
        } else {
          const _Float16 a = (_Float16)f[e];
          hi[e] = __builtin_bit_cast(uint16_t, a);
          // an infinity or NaN stays in the hi plane alone
          lo[e] = (hi[e] & 0x7c00u) == 0x7c00u ? 0u : __builtin_bit_cast(uint16_t, (_Float16)(f[e] - (float)a));
        }
      }
      const uint32_t c = ((uint32_t)(q * kItem) + l4) >> 3;  // the 16-byte chunk of the row's segment
      uint8_t *d = lds + row * pitch + (c >> 4) * 512 + (((c & 15) ^ (row & 15)) << 4) + (lane & 1) * 8;
      *reinterpret_cast<uint2 *>(d) = make_uint2(hi[0] | hi[1] << 16, hi[2] | hi[3] << 16);
      *reinterpret_cast<uint2 *>(d + 256) = make_uint2(lo[0] | lo[1] << 16, lo[2] | lo[3] << 16);
    }
    if constexpr (WF != FMT_BF16) {
      // Only where some lane's group is that small (hardly ever) they are
      // counted by item, the values read again: kept until here they would
      // cost registers.
      if (__builtin_expect(__any(small), 0)) {
#pragma unroll 1
        for (int it = wave; it < items; it += kWaves) {
          const int row = it / ipr, k = kb0 * kStep + (it - row * ipr) * kItem + lane * 4;
          const int most = (int)wave_max(lane < ipr ? item_max[row * ipr + lane] : 0u);
          const u32x4 v = __builtin_amdgcn_raw_buffer_load_b128(
              rx, k < k_end ? (int)(((uint32_t)row * (uint32_t)P.ldx + k) * 4) : (int)kNone, 0, 0);
          auto mag = [&](uint32_t u, int e) { return k + e < k_end ? (int)(u & 0x7fffffffu) : 0; };
          const int a = max(max(mag(v.x, 0), mag(v.y, 1)), max(mag(v.z, 2), mag(v.w, 3)));
          const uint64_t some = __ballot(a > 0), less = __ballot(a > 0 && a < most - (int)kSmall);
          if (lane == 0 && 2 * __popcll(less) > __popcll(some)) atomicOr(&marks[row >> 5], 1u << (row & 31));
        }
      }
    }
    __syncthreads();
    // The segment's batches in rounds of kStages. Batch kb + 1 goes to LDS, and its registers to
    // batch kb + 1 + kStages, while batch kb is computed.
    if (first) {
      put(ring[0], 0);
      issue(ring[0], kb_lo + kStages);
      first = false;
    }
    const int nb = min(segb, kb_hi - kb0);
    Frags f[2];
    read(f[0], 0, 0, 0);
#pragma unroll 1
    for (int kb = 0; kb < nb; kb += kStages) {
#pragma unroll
      for (int j = 0; j < kStages; j++) {
        // past the range: the rest of the round would multiply zeros (512 x 64
        // Q8_0 of 2 rows 11.0 us with it, 7.9 without; 6912 x 2560 of 16 18.1,
        // 17.2)
        if (j > 0 && kb + j >= nb) break;
        put(ring[(j + 1) % kStages], (j + 1) & 1);
        issue(ring[(j + 1) % kStages], kb0 + kb + j + 1 + kStages);
#pragma unroll
        for (int u = 0; u < kUnits; u++) {
          const bool last = u + 1 == kUnits;
          read(f[(u + 1) & 1], last ? min(kb + j + 1, segb - 1) : kb + j, last ? 0 : u + 1, last ? (j + 1) & 1 : j & 1);
          __builtin_amdgcn_sched_barrier(0);
          compute(f[u & 1]);
        }
      }
      // F16: every 1024 columns (the chain of products on the matrix cores,
      // of 4096 columns, erred by 6.0e-7; so 3.1e-7)
      if constexpr (WF == FMT_F16 && MT == 1)
        if ((kb + kStages) * kStep % 1024 == 0 && kb + kStages < nb) fold();
    }
    fold();
  }
  // D fragment: lane holds column lane % 32 of rows (v / 4) * 8 + (lane / 32) * 4 + v % 4.
  float *y = P.y + (int64_t)split * P.split_stride;
#pragma unroll
  for (int mt = 0; mt < MT; mt++)
#pragma unroll
    for (int v = 0; v < 16; v++) {
      const int m = mt * 32 + (v >> 2) * 8 + h * 4 + (v & 3);
      if (m < M && n < N) y[(int64_t)m * P.ldy + n] = tot[mt][v];
    }
  if constexpr (WF != FMT_BF16) {
    // (the marks were made before the barrier that ended the last staging)
    const uint64_t rows = (uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)marks[1]) << 32 |
                          (uint32_t)__builtin_amdgcn_readfirstlane((int)marks[0]);
    if (__builtin_expect(!rows, 1)) return;
    wait_vmcnt<0>();  // the stores above, which the marked rows' outputs replace
    asm volatile("" ::: "memory");
    // The arguments are read again: kept in registers through the loops above
    // they would not fit beside what those need.
    const FewArgs *args = reinterpret_cast<const FewArgs *>((const void *)__builtin_amdgcn_kernarg_segment_ptr());
    asm volatile("" : "+s"(args));
    int bq = blockIdx.x;
    asm volatile("" : "+s"(bq));
    const int first_blocks = args->p[0].ks * ((args->p[0].w.rows + kBlockRows - 1) / kBlockRows);
    const FewProduct &Q = args->p[bq >= first_blocks];
    if (bq >= first_blocks) bq -= first_blocks;
    const int rb = (Q.w.rows + kBlockRows - 1) / kBlockRows, sq = bq / rb, nkq = (Q.w.cols + kStep - 1) / kStep;
    const int c0 = (bq - sq * rb) * kBlockRows + wave * kTile;
    plain_rows<WF>(Q.w, Q.x, Q.ldx, rows, 0, c0, min(c0 + kTile, Q.w.rows), (int)((int64_t)nkq * sq / Q.ks) * kStep,
                   min(Q.w.cols, (int)((int64_t)nkq * (sq + 1) / Q.ks) * kStep), Q.y + (int64_t)sq * Q.split_stride, Q.ldy);
  }
}

template <int WF>
hipError_t few_rows_launch(const FewArgs &g, int blocks, hipStream_t st) {
  const size_t bytes = (size_t)g.M * g.seg * 4 + kWaves * kWaveBytes;
  constexpr int kMax = kWaves * (kItems * kItem * 4 + kWaveBytes);
  static const hipError_t attr1 = hipFuncSetAttribute(reinterpret_cast<const void *>(&few_rows_kernel<WF, 1>),
                                                      hipFuncAttributeMaxDynamicSharedMemorySize, kMax);
  static const hipError_t attr2 = hipFuncSetAttribute(reinterpret_cast<const void *>(&few_rows_kernel<WF, 2>),
                                                      hipFuncAttributeMaxDynamicSharedMemorySize, kMax);
  if (attr1 != hipSuccess || attr2 != hipSuccess) return attr1 != hipSuccess ? attr1 : attr2;
  if (g.M <= 32)
    hipLaunchKernelGGL((few_rows_kernel<WF, 1>), dim3(blocks), dim3(kT), bytes, st, g);
  else
    hipLaunchKernelGGL((few_rows_kernel<WF, 2>), dim3(blocks), dim3(kT), bytes, st, g);
  return hipGetLastError();
}

double value_bytes(int fmt) { return fmt == FMT_Q8_0 ? 34.0 / 32 : 2.0; }
int row_blocks(const MatDesc &w) { return (w.rows + kBlockRows - 1) / kBlockRows; }

// Microseconds of a launch of `blocks` blocks whose longest covers `kb`
// batches, and of the partial outputs (written and read): about 20 KB of
// matrix per CU and microsecond, 3 us before a block's stream is going.
double launch_cost(int blocks, int kb, int fmt, double partial_bytes) {
  const double batch = kBlockRows * batch_cols(fmt) * value_bytes(fmt) / 20e3;
  return ((blocks + 255) / 256) * (kb * batch + 3.0) + partial_bytes / 5e6;
}

}  // namespace

bool few_rows_supported(const Matrix &w, int M, int64_t ldx) {
  if (M < 2 || M > kFewRowsMax || w.cols < 1 || w.vstride % 16 || (reinterpret_cast<uintptr_t>(w.vals) & 15) ||
      (int64_t)w.rows * w.vstride > 0x7fffffff || (int64_t)M * ldx * 4 > 0x7fffffff)
    return false;
  if (w.fmt == FMT_Q8_0)
    return w.cols % 64 == 0 && (reinterpret_cast<uintptr_t>(w.meta) & 3) == 0 && w.mstride % 4 == 0;
  return w.fmt == FMT_BF16 ? w.cols % 32 == 0 : w.fmt == FMT_F16 && !w.special;
}

int few_rows_splits(const MatDesc &w, int M, int max_splits) {
  const int step = batch_cols(w.fmt), nk = (w.cols + step - 1) / step, tb = row_blocks(w);
  int best = 1;
  double cost = 1e30;
  for (int s = 1; s <= std::min(max_splits, nk); s++) {
    const double c = launch_cost(tb * s, (nk + s - 1) / s, w.fmt, s > 1 ? 8.0 * s * M * w.rows : 0);
    if (c < cost) cost = c, best = s;
  }
  return best;
}

void few_rows_pair_splits(const MatDesc &a, const MatDesc &b, int M, int max_splits, int *sa, int *sb) {
  const int step = batch_cols(a.fmt), ka = (a.cols + step - 1) / step, kb = (b.cols + step - 1) / step;
  double cost = 1e30;
  // every block about `per` batches long, whichever product it works for
  for (int per = 1; per <= std::max(ka, kb); per++) {
    const int s = std::min((ka + per - 1) / per, max_splits), t = std::min((kb + per - 1) / per, max_splits);
    const int longest = std::max((ka + s - 1) / s, (kb + t - 1) / t);
    const double c = launch_cost(row_blocks(a) * s + row_blocks(b) * t, longest, a.fmt,
                                 8.0 * M * ((double)s * a.rows + (double)t * b.rows));
    if (c < cost) cost = c, *sa = s, *sb = t;
  }
}

hipError_t launch_few_rows(const FewProduct *p, int nprod, int M, hipStream_t st) {
  if (nprod < 1 || nprod > 2) return hipErrorInvalidValue;
  FewArgs g{};
  g.nprod = nprod;
  g.M = M;
  int blocks = 0, longest = 0;
  for (int i = 0; i < nprod; i++) {
    const FewProduct &q = p[i];
    const int step = batch_cols(q.w.fmt), nk = (q.w.cols + step - 1) / step;
    if (!few_rows_supported(q.w, M, q.ldx) || q.w.fmt != p[0].w.fmt || q.ldx < q.w.cols || !q.x || !q.y || q.ks < 1 ||
        q.ks > nk || (reinterpret_cast<uintptr_t>(q.x) & 3) || (q.ks > 1 && q.split_stride < (int64_t)M * q.ldy))
      return hipErrorInvalidValue;
    g.p[i] = q;
    blocks += q.ks * row_blocks(q.w);
    longest = std::max(longest, (nk + q.ks - 1) / q.ks * step);
  }
  // Segments as long as the staging items allow, no longer than a block's
  // K range.
  const int round = few_stages(p[0].w.fmt, M > 32 ? 2 : 1) * batch_cols(p[0].w.fmt), most = kWaves * kItems / M * kItem;
  g.seg = std::min(std::max(1, most / round), (longest + round - 1) / round) * round;
  switch (p[0].w.fmt) {
    case FMT_Q8_0: return few_rows_launch<FMT_Q8_0>(g, blocks, st);
    case FMT_BF16: return few_rows_launch<FMT_BF16>(g, blocks, st);
    case FMT_F16: return few_rows_launch<FMT_F16>(g, blocks, st);
    default: return hipErrorInvalidValue;
  }
}
