// The decoder block's products for ticks of few rows (gfx950): y = x W^T for up to 16 rows.
//
// Reference: the projections of GroupedQueryAttention and FeedForward (layers.py:13-27,
// :131-164) with the steps around them (layers.py:30-40, :202-232). A tick of a few decode
// rows reads every weight once for a handful of multiply-adds each, so the product is a
// stream of W from HBM; the row steps ride on it:
//   NORM      x is RMSNormed on its way in (statistics per workgroup, from L2);
//   residual  out = residual + round(y);
//   SwiGLU    W holds gate rows, then up rows: out = silu(round(gate)) * round(up).
// Every value rounds to the element type where the separate steps round it.
//
// A workgroup owns 16 columns of y (SwiGLU: 16 gate and the 16 up columns they multiply)
// and all rows; its waves split K and merge through LDS in wave order. A wave reads W and x
// in whole lines (64 k elements of eight rows per instruction), a few batches ahead in
// registers, and turns them into the MFMA operand layout through its own part of LDS. (Loads
// straight into that layout touch 16 lines per 16 lanes and streamed W at 2 TB/s.)
//
// A layer of hidden 2560, 32/8 heads of 128 and ffn 9728 at 8 rows, W from HBM: the four
// products 11.6 + 7.7 + 28.1 + 15.0 = 62 us (2.7 / 2.7 / 3.5 / 3.3 TB/s of W; about 3.5 us of
// each is launch, first load and merge). As library products with the norms, adds and SwiGLU
// of block_ops.hip between them: 102 us at 8 rows, 102 at 16 (here 71), 77-82 at 17-32, where
// a second row tile brings this kernel to 88-94: hence up to 16 rows.

#include "hx_common.h"

namespace {

constexpr int kSkRows = 16;                   // rows of x at most: one MFMA tile
constexpr int kSkBatch = 64;                  // k elements per batch: one 128-byte line of a row
constexpr int kSkTileBytes = 16 * 2 * kSkBatch;  // 16 rows of a batch: 2 KiB

enum : int { kEpiPlain = 0, kEpiResidual = 1, kEpiSwiglu = 2 };

struct SkinnyArgs {
  const uint16_t* x;
  const uint16_t* w;
  int64_t x_row, w_row;
  int32_t rows, cols, k;   // cols: of the output
  const float* norm_w;
  float eps;
  const uint16_t* res;
  int64_t res_row;
  uint16_t* out;
  int64_t out_row;
};

// Batches of one wave's 16-row tile: lane l of load j takes 16 bytes of row 8 j + (l >> 3),
// so an instruction reads eight whole lines, and stores them at 1024 j + 16 l. The 16-byte
// pieces of a row are permuted on the way (piece p of LDS row r is piece p ^ ((r >> 1) & 7)
// of the line): a fragment read's 16 rows, one piece each, then hit all 64 banks once.
__device__ __forceinline__ int sk_piece(int row, int p) { return p ^ ((row >> 1) & 7); }

// D: batches in flight per wave.
template <typename T, bool NORM, int EPI, int WAVES, int D>
__global__ __launch_bounds__(64 * WAVES) void skinny_gemm_kernel(SkinnyArgs a) {
  typedef hx::Elem<T> E;
  constexpr int NV = EPI == kEpiSwiglu ? 2 : 1;  // W tiles: the output's 16 columns, or gate and up
  constexpr int kWaveBytes = (NV + 1) * kSkTileBytes;
  // Each wave's batch, then the waves' sums.
  __shared__ __attribute__((aligned(16))) uint8_t smem[WAVES * kWaveBytes];
  static_assert(NV * 1024 <= kWaveBytes, "the sums fit the batches' space");
  __shared__ float s_r[kSkRows];
  const int tid = hx::tid_x(), lane = tid & 63, lr = lane & 15, lg = lane >> 4;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int n0 = hx::wg_x() * 16;
  const int batches = a.k / kSkBatch;
  const int b_begin = (int)((int64_t)batches * w / WAVES), b_end = (int)((int64_t)batches * (w + 1) / WAVES);

  // The statistics' reads of x go first: loads complete in order, and W comes from HBM. A
  // wave sums rows w, w + WAVES, ...; the first kStat x 512 elements of each are held here.
  constexpr int kStat = 5, kStatRows = kSkRows / WAVES > 0 ? kSkRows / WAVES : 1;
  uint4 st[NORM ? kStatRows : 1][kStat];
  if constexpr (NORM) {
#pragma unroll
    for (int i = 0; i < kStatRows; ++i)
#pragma unroll
      for (int c = 0; c < kStat; ++c) {
        const int row = w + i * WAVES, at = 64 * c + lane;
        st[i][c] = hx::zero4();
        if (row < a.rows && at < a.k / 8)
          st[i][c] = *reinterpret_cast<const uint4*>(a.x + (int64_t)row * a.x_row + 8 * at);
      }
  }

  const uint16_t* wp[NV][2];
  const uint16_t* xp[2];
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    const int row = 8 * j + (lane >> 3), c = 8 * sk_piece(row, lane & 7);
#pragma unroll
    for (int v = 0; v < NV; ++v) wp[v][j] = a.w + (int64_t)(n0 + v * a.cols + row) * a.w_row + c;
    xp[j] = a.x + (int64_t)min(row, a.rows - 1) * a.x_row + c;
  }
  const bool high = a.rows > 8;  // rows past the last feed unused sums only
  uint4 wb[D][NV][2], xb[D][2];
  auto load_w = [&](int i, int b) __attribute__((always_inline)) {
#pragma unroll
    for (int v = 0; v < NV; ++v)
#pragma unroll
      for (int j = 0; j < 2; ++j) wb[i][v][j] = hx::ld16_stream(wp[v][j] + (int64_t)b * kSkBatch);
  };
  auto load_x = [&](int i, int b) __attribute__((always_inline)) {
    xb[i][0] = *reinterpret_cast<const uint4*>(xp[0] + (int64_t)b * kSkBatch);
    if (high) xb[i][1] = *reinterpret_cast<const uint4*>(xp[1] + (int64_t)b * kSkBatch);
  };
#pragma unroll
  for (int i = 0; i < D; ++i) {
    xb[i][0] = xb[i][1] = hx::zero4();
    if (b_begin + i < b_end) {
      load_x(i, b_begin + i);
      load_w(i, b_begin + i);
    }
  }

  float r = 1.f;
  if constexpr (NORM) {
    // mean(x^2) of each row: squares rounded to fp32, then summed.
#pragma unroll
    for (int i = 0; i < kStatRows; ++i) {
      const int row = w + i * WAVES;
      float ss = 0.f;
      auto add = [&](uint4 u) {
        const uint32_t wd[4] = {u.x, u.y, u.z, u.w};
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const float e0 = E::lo(wd[q]), e1 = E::hi(wd[q]);
          ss = __fadd_rn(ss, __fmul_rn(e0, e0));
          ss = __fadd_rn(ss, __fmul_rn(e1, e1));
        }
      };
#pragma unroll
      for (int c = 0; c < kStat; ++c) add(st[i][c]);
      if (row >= a.rows) continue;  // wave-uniform
      for (int at = 64 * kStat + lane; at < a.k / 8; at += 64)
        add(*reinterpret_cast<const uint4*>(a.x + (int64_t)row * a.x_row + 8 * at));
      ss = hx::wave_sum_xor(ss, 1, 32);
      if (lane == 0) s_r[row] = rsqrtf(__fadd_rn(__fdiv_rn(ss, (float)a.k), a.eps));
    }
    __syncthreads();
    r = s_r[min(lr, a.rows - 1)];
  }

  hx::f32x4_t acc[NV];
#pragma unroll
  for (int v = 0; v < NV; ++v) acc[v] = hx::f32x4_t{0.f, 0.f, 0.f, 0.f};

  // Lanes read what other lanes of the wave stored. One wave's LDS accesses complete in order,
  // so its stage needs no barrier; the wavefront fences (no instruction) hold the compiler to
  // the order of stores, reads and the next batch's stores.
  uint8_t* const stage = smem + w * kWaveBytes;
  auto consume = [&](int i, int b) __attribute__((always_inline)) {
#pragma unroll
    for (int j = 0; j < 2; ++j) {
#pragma unroll
      for (int v = 0; v < NV; ++v)
        *reinterpret_cast<uint4*>(stage + v * kSkTileBytes + 1024 * j + 16 * lane) = wb[i][v][j];
      *reinterpret_cast<uint4*>(stage + NV * kSkTileBytes + 1024 * j + 16 * lane) = xb[i][j];
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    if (b + D < b_end) {  // wave-uniform
      load_x(i, b + D);
      load_w(i, b + D);
    }
#pragma unroll
    for (int s = 0; s < kSkBatch / 32; ++s) {
      const int at = 128 * lr + 16 * sk_piece(lr, 4 * s + lg);
      uint4 xv = *reinterpret_cast<const uint4*>(stage + NV * kSkTileBytes + at);
      if constexpr (NORM) {
        const float* p = a.norm_w + (int64_t)b * kSkBatch + 32 * s + 8 * lg;
        const float4 lo = *reinterpret_cast<const float4*>(p), hi = *reinterpret_cast<const float4*>(p + 4);
        const float nw[8] = {lo.x, lo.y, lo.z, lo.w, hi.x, hi.y, hi.z, hi.w};
        const uint32_t wd[4] = {xv.x, xv.y, xv.z, xv.w};
        uint32_t o[4];
#pragma unroll
        for (int q = 0; q < 4; ++q)
          o[q] = hx::pack2_round<T>(__fmul_rn(__fmul_rn(E::lo(wd[q]), r), nw[2 * q]),
                                    __fmul_rn(__fmul_rn(E::hi(wd[q]), r), nw[2 * q + 1]));
        xv = make_uint4(o[0], o[1], o[2], o[3]);
      }
#pragma unroll
      for (int v = 0; v < NV; ++v) {
        const uint4 wf = *reinterpret_cast<const uint4*>(stage + v * kSkTileBytes + at);
        acc[v] = E::mfma16x16x32(hx::as_v8<T>(wf), hx::as_v8<T>(xv), acc[v]);
      }
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  };
  for (int b = b_begin; b < b_end; b += D) {
#pragma unroll
    for (int i = 0; i < D; ++i)
      if (b + i < b_end) consume(i, b + i);
  }

  float (*const red)[NV][256] = reinterpret_cast<float (*)[NV][256]>(smem);
  __syncthreads();  // every wave is done with its batches
  // Lane holds columns 4 lg .. +3 of row lr.
#pragma unroll
  for (int v = 0; v < NV; ++v)
    *reinterpret_cast<float4*>(&red[w][v][16 * lr + 4 * lg]) = make_float4(acc[v][0], acc[v][1], acc[v][2], acc[v][3]);
  __syncthreads();
  // A thread finishes a column pair: the waves' sums in wave order.
  if (tid >= 128) return;
  const int e = 2 * tid, row = e >> 4, n = n0 + (e & 15);
  if (row >= a.rows) return;
  float2 y[NV];
#pragma unroll
  for (int v = 0; v < NV; ++v) {
    y[v] = make_float2(0.f, 0.f);
#pragma unroll
    for (int ww = 0; ww < WAVES; ++ww) {
      const float2 q = *reinterpret_cast<const float2*>(&red[ww][v][e]);
      y[v].x += q.x;
      y[v].y += q.y;
    }
  }
  uint32_t o = hx::pack2_round<T>(y[0].x, y[0].y);
  if constexpr (EPI == kEpiSwiglu) o = hx::swiglu2<T>(o, hx::pack2_round<T>(y[NV - 1].x, y[NV - 1].y));
  if constexpr (EPI == kEpiResidual)
    o = hx::add2<T>(*reinterpret_cast<const uint32_t*>(a.res + (int64_t)row * a.res_row + n), o);
  *reinterpret_cast<uint32_t*>(a.out + (int64_t)row * a.out_row + n) = o;
}

// Waves that split K, and batches in flight: the most that pay. At 8 rows (us, qkv / o /
// gate_up / down): 8 waves and 2 batches 11.6 / 7.7 / 28.1 / 15.0, 3 batches 14.6 / 7.6 / 29.4
// / 14.8 (with the norm's registers they cost occupancy); 4 waves 13.5-13.6 / 8.2-8.8 /
// 28.4-28.9 / 17.0-18.6; 16 waves 13.6-14.0 / 7.5-7.8 / 31.9-32.8 / 15.3.
constexpr int kSkWaves = 8;

template <typename T, bool NORM, int EPI>
void launch_one(const SkinnyArgs& a, hipStream_t s) {
  hipLaunchKernelGGL((skinny_gemm_kernel<T, NORM, EPI, kSkWaves, NORM ? 2 : 3>), dim3((unsigned)(a.cols / 16)),
                     dim3(64 * kSkWaves), 0, s, a);
}

template <typename T>
void launch_epi(const SkinnyArgs& a, bool swiglu, hipStream_t s) {
  const bool norm = a.norm_w != nullptr;
  if (swiglu && norm) launch_one<T, true, kEpiSwiglu>(a, s);
  else if (swiglu) launch_one<T, false, kEpiSwiglu>(a, s);
  else if (a.res != nullptr && norm) launch_one<T, true, kEpiResidual>(a, s);
  else if (a.res != nullptr) launch_one<T, false, kEpiResidual>(a, s);
  else if (norm) launch_one<T, true, kEpiPlain>(a, s);
  else launch_one<T, false, kEpiPlain>(a, s);
}

}  // namespace

extern "C" int hx_skinny_gemm(const void* x, int64_t x_row_stride, int64_t rows, const void* weight,
                              int64_t weight_row_stride, int32_t cols, int32_t k, int32_t dtype,
                              const float* norm_weight, float eps, const void* residual, int64_t residual_row_stride,
                              int32_t swiglu, void* out, int64_t out_row_stride, void* stream) {
  if (dtype != HX_DTYPE_BF16 && dtype != HX_DTYPE_FP16) return HX_E_UNSUPPORTED;
  if (rows < 0 || cols < 1 || k < 1 || (norm_weight != nullptr && !(eps >= 0.f))) return HX_E_INVALID_ARG;
  if (rows > kSkRows || cols % 16 || k % kSkBatch) return HX_E_UNSUPPORTED;
  if (rows == 0) return HX_OK;
  if (!x || !weight || !out || (swiglu && residual)) return HX_E_INVALID_ARG;
  const uintptr_t ptrs = reinterpret_cast<uintptr_t>(x) | reinterpret_cast<uintptr_t>(weight) |
                         reinterpret_cast<uintptr_t>(norm_weight);
  if ((ptrs & 15) || x_row_stride % 8 || weight_row_stride % 8 || x_row_stride < k || weight_row_stride < k)
    return HX_E_INVALID_ARG;
  if (((reinterpret_cast<uintptr_t>(out) | reinterpret_cast<uintptr_t>(residual)) & 3) || out_row_stride % 2 ||
      out_row_stride < cols || (residual != nullptr && (residual_row_stride % 2 || residual_row_stride < cols)))
    return HX_E_INVALID_ARG;
  SkinnyArgs a;
  a.x = static_cast<const uint16_t*>(x);
  a.w = static_cast<const uint16_t*>(weight);
  a.x_row = x_row_stride;
  a.w_row = weight_row_stride;
  a.rows = (int32_t)rows;
  a.cols = cols;
  a.k = k;
  a.norm_w = norm_weight;
  a.eps = eps;
  a.res = static_cast<const uint16_t*>(residual);
  a.res_row = residual_row_stride;
  a.out = static_cast<uint16_t*>(out);
  a.out_row = out_row_stride;
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  if (dtype == HX_DTYPE_BF16) launch_epi<__bf16>(a, swiglu != 0, s);
  else launch_epi<_Float16>(a, swiglu != 0, s);
  return hx::status_from_hip(hipGetLastError());
}
