// Dense D x D rotation y = x @ R (or x @ R^T) for gfx950.
//
// Replaces the fp32 matmuls of oscar_ascend/backend.py:371 (q @ R_k) and :382
// (out_rot @ R_v^T).  Few rows (decode steps): rotate_kernel.  A workgroup of four waves computes a 32 x 32 output tile with
// v_mfma_f32_32x32x16_bf16 over a three-term split of both operands
// (x_hi R_hi + x_lo R_hi + x_hi R_lo, hi = bf16(v), lo = bf16(v - hi)), which keeps
// the product error below 2^-16 of |x||R| with fp32 accumulation; each wave takes
// a quarter of the contraction, the four partial tiles are summed in LDS and the
// result is rounded once to the output dtype.
//
// The input dtype, the output dtype and the transpose flag are template
// parameters, so the operand loads of all K-steps are plain vector loads with no
// branch between them, issued together ahead of the MFMAs.
#include "common.h"

namespace oscar {

namespace {

typedef __bf16 __attribute__((ext_vector_type(2))) bf16x2;
typedef float __attribute__((ext_vector_type(2))) f32x2;

// hi/lo bf16 split of 8 floats into two MFMA operands
__device__ __forceinline__ void split8(const float* v, bf16x8& hi, bf16x8& lo) {
  u32x4 h, l;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const f32x2 a = {v[2 * i], v[2 * i + 1]};
    const bf16x2 hb = __builtin_convertvector(a, bf16x2);
    const f32x2 hv = __builtin_convertvector(hb, f32x2);
    h[i] = __builtin_bit_cast(unsigned, hb);
    l[i] = __builtin_bit_cast(unsigned, __builtin_convertvector(a - hv, bf16x2));
  }
  hi = __builtin_bit_cast(bf16x8, h);
  lo = __builtin_bit_cast(bf16x8, l);
}

template <int D, int XT, int OT, bool TR>
__global__ __launch_bounds__(256) void rotate_kernel(oscar_rotate_args_v1 a) {
  constexpr int KS = D / 16 / 4;  // K-steps per wave
  const int lane = threadIdx.x & 63, m = lane & 31, g = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int64_t row0 = (int64_t)blockIdx.x * 32;
  const int col0 = blockIdx.y * 32;
  const int64_t row = row0 + m;
  const bool row_ok = row < a.rows;
  const int64_t xrow = (row_ok ? row : row0) * a.x_stride_row;  // row0 < rows always
  const int col = col0 + m;
  // all operand loads of this wave's K range first
  float xv[KS][8], rv[KS][8];
#pragma unroll
  for (int s = 0; s < KS; ++s) {
    const int kk = (wave * KS + s) * 16 + 8 * g;
    load8<XT>(a.x, xrow + kk, xv[s]);
    // B[k][n]: R[k][col], or R^T[k][col] = R[col][k] (contiguous in k)
    if constexpr (TR) {
      load8<OSCAR_F32>(a.r, (int64_t)col * D + kk, rv[s]);
    } else {
#pragma unroll
      for (int e = 0; e < 8; ++e) rv[s][e] = a.r[(int64_t)(kk + e) * D + col];
    }
  }
  f32x16 acc = {};
#pragma unroll
  for (int s = 0; s < KS; ++s) {
    if (!row_ok) {
#pragma unroll
      for (int e = 0; e < 8; ++e) xv[s][e] = 0.f;
    }
    bf16x8 xh, xl, rh, rl;
    split8(xv[s], xh, xl);
    split8(rv[s], rh, rl);
    acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(xh, rh, acc, 0, 0, 0);
    acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(xl, rh, acc, 0, 0, 0);
    acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(xh, rl, acc, 0, 0, 0);
  }
  // sum of the four wave tiles (register order), then the store
  __shared__ f32x4 part[3][4][64];
  if (wave > 0) {
#pragma unroll
    for (int q = 0; q < 4; ++q)
      part[wave - 1][q][lane] = f32x4{acc[4 * q], acc[4 * q + 1], acc[4 * q + 2], acc[4 * q + 3]};
  }
  __syncthreads();
  if (wave != 0) return;
#pragma unroll
  for (int w = 0; w < 3; ++w)
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const f32x4 v = part[w][q][lane];
#pragma unroll
      for (int j = 0; j < 4; ++j) acc[4 * q + j] += v[j];
    }
  // D[i][j]: lane = j + 32*((i/4)%2), register = (i%4) + 4*(i/8); here i = row, j = col
#pragma unroll
  for (int r = 0; r < 16; ++r) {
    const int i = 8 * (r >> 2) + 4 * g + (r & 3);
    const int64_t orow = row0 + i;
    if (orow < a.rows) store_elem(a.out, OT, orow * a.out_stride_row + col, acc[r]);
  }
}

// Many rows: a workgroup of eight waves keeps all of R and walks over tiles of 32 (D = 256)
// or 64 (D = 128) rows.  Wave w holds the hi and lo operands of one 32-column block of R for
// the whole contraction in registers (128 at D = 256, loaded once), the tile's rows are split
// into hi and lo planes in LDS once for all waves, and the next tile's rows are in flight
// beside the products.  rotate_kernel reads a row tile once per column block and R once per
// 32 x 32 outputs: 55536 x 256 fp32 rows to bf16 101 us there, 28 us here (85 MB, 17 us at
// the rate of a large copy; 48 MFMAs per wave and tile, 1.4 us).
constexpr int kBigThreads = 512;
constexpr int64_t kBigGrid = 256;  // one workgroup per compute unit
// rotate_rows_kernel from this many bytes of x on: its workgroups first take all of R, which
// is most of its time for few rows.  Measured (us, tiled kernel against this one): 2400 fp32
// rows of 256 8.5 / 8.6, 6400 16.7 / 9.1; 3200 bf16 rows of 256 6.8 / 7.6, 6400 9.6 / 8.0;
// 3200 fp32 rows of 128 4.9 / 6.0, 6400 6.7 / 6.1; bf16 6400 4.9 / 5.4, 12800 6.6 / 5.8.
constexpr int64_t kBigBytes = 5 << 19;
template <int D, int XT, int OT, bool TR>
__global__ __launch_bounds__(kBigThreads, 2) void rotate_rows_kernel(oscar_rotate_args_v1 a) {
  constexpr int KS = D / 16;              // K-steps
  constexpr int CB = D / 32;              // column blocks
  constexpr int ROWS = 32 * (8 / CB);     // rows of a tile
  constexpr int CPR = D / 8;              // 8-element parts of a row
  constexpr int NP = ROWS * CPR / kBigThreads;
  constexpr bool LO = XT != OSCAR_BF16;   // bf16 rows are their own hi plane
  const int tid = threadIdx.x, lane = tid & 63, m = lane & 31, g = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int col = (wave % CB) * 32 + m, r0 = (wave / CB) * 32;
  // rows padded by 16 bytes: the row-per-lane operand reads cover all banks
  __shared__ __attribute__((aligned(16))) uint16_t s_x[2][LO ? 2 : 1][ROWS][D + 8];
  float xv[NP][8];
  auto fetch = [&](int64_t tile) {
#pragma unroll
    for (int i = 0; i < NP; ++i) {
      const int part = i * kBigThreads + tid;
      int64_t row = tile * ROWS + part / CPR;
      row = row < a.rows ? row : a.rows - 1;  // computed, never stored
      load8<XT>(a.x, row * a.x_stride_row + 8 * (part % CPR), xv[i]);
    }
  };
  auto stash = [&](int buf) {
#pragma unroll
    for (int i = 0; i < NP; ++i) {
      const int part = i * kBigThreads + tid;
      bf16x8 h, l;
      split8(xv[i], h, l);
      *(bf16x8*)&s_x[buf][0][part / CPR][8 * (part % CPR)] = h;
      if constexpr (LO) *(bf16x8*)&s_x[buf][1][part / CPR][8 * (part % CPR)] = l;
    }
  };
  const int64_t tiles = (a.rows + ROWS - 1) / ROWS;
  int64_t tile = blockIdx.x;  // < tiles (host)
  fetch(tile);
  bf16x8 rh[KS], rl[KS];
  if constexpr (TR) {
    // B[k][n] = R[n][k]: the wave's 32 rows of R in parts of 64 columns, read along the rows
    // (256 bytes each) and handed over through LDS; a lane's own 32 bytes of 32 rows would
    // touch 64 lines a load (11.3 us for one row tile, 7.6 us this way)
    constexpr int KP = 64;
    __shared__ __attribute__((aligned(16))) float s_r[8][32][KP + 4];
    f32x4 rr[8];
    auto rfetch = [&](int k0) {
#pragma unroll
      for (int i = 0; i < 8; ++i)
        rr[i] = *(const f32x4*)(a.r + (int64_t)((wave % CB) * 32 + 4 * i + (lane >> 4)) * D + k0 + 4 * (lane & 15));
    };
    rfetch(0);
#pragma unroll
    for (int k0 = 0; k0 < D; k0 += KP) {
#pragma unroll
      for (int i = 0; i < 8; ++i) *(f32x4*)&s_r[wave][4 * i + (lane >> 4)][4 * (lane & 15)] = rr[i];
      if (k0 + KP < D) rfetch(k0 + KP);
      wait_lds();  // the wave's own rows: no barrier
      __builtin_amdgcn_wave_barrier();
#pragma unroll
      for (int s = 0; s < KP / 16; ++s) {
        float rv[8];
        load8<OSCAR_F32>(&s_r[wave][m][0], 16 * s + 8 * g, rv);
        split8(rv, rh[k0 / 16 + s], rl[k0 / 16 + s]);
      }
      __builtin_amdgcn_wave_barrier();
    }
  } else {
#pragma unroll
    for (int s = 0; s < KS; ++s) {
      const int kk = s * 16 + 8 * g;
      float rv[8];
#pragma unroll
      for (int e = 0; e < 8; ++e) rv[e] = a.r[(int64_t)(kk + e) * D + col];
      split8(rv, rh[s], rl[s]);
    }
  }
  stash(0);
  __syncthreads();
  for (int buf = 0; tile < tiles; tile += gridDim.x, buf ^= 1) {
    const bool more = tile + gridDim.x < tiles;
    if (more) fetch(tile + gridDim.x);
    // the leading products and the corrections apart: half the rounding of one chain
    f32x16 acc = {}, cor = {};
#pragma unroll
    for (int s = 0; s < KS; ++s) {
      const bf16x8 xh = *(const bf16x8*)&s_x[buf][0][r0 + m][16 * s + 8 * g];
      acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(xh, rh[s], acc, 0, 0, 0);
      cor = __builtin_amdgcn_mfma_f32_32x32x16_bf16(xh, rl[s], cor, 0, 0, 0);
      if constexpr (LO) {
        const bf16x8 xl = *(const bf16x8*)&s_x[buf][1][r0 + m][16 * s + 8 * g];
        cor = __builtin_amdgcn_mfma_f32_32x32x16_bf16(xl, rh[s], cor, 0, 0, 0);
      }
    }
    // D[i][j]: lane = j + 32*((i/4)%2), register = (i%4) + 4*(i/8); here i = row, j = col
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const int64_t row = tile * ROWS + r0 + 8 * (r >> 2) + 4 * g + (r & 3);
      if (row < a.rows) store_elem(a.out, OT, row * a.out_stride_row + col, acc[r] + cor[r]);
    }
    if (more) stash(buf ^ 1);
    __syncthreads();
  }
}

template <int D, int XT, int OT>
void launch_tr(const oscar_rotate_args_v1& a, hipStream_t s) {
  if (a.rows * D * (XT == OSCAR_F32 ? 4 : 2) >= kBigBytes) {
    const int64_t rows = 32 * (8 / (D / 32)), tiles = (a.rows + rows - 1) / rows;
    const dim3 grid((unsigned)(tiles < kBigGrid ? tiles : kBigGrid));
    if (a.transpose) hipLaunchKernelGGL((rotate_rows_kernel<D, XT, OT, true>), grid, dim3(kBigThreads), 0, s, a);
    else hipLaunchKernelGGL((rotate_rows_kernel<D, XT, OT, false>), grid, dim3(kBigThreads), 0, s, a);
    return;
  }
  const dim3 grid((unsigned)((a.rows + 31) / 32), (unsigned)(D / 32));
  if (a.transpose) hipLaunchKernelGGL((rotate_kernel<D, XT, OT, true>), grid, dim3(256), 0, s, a);
  else hipLaunchKernelGGL((rotate_kernel<D, XT, OT, false>), grid, dim3(256), 0, s, a);
}

template <int D, int XT>
void launch_out(const oscar_rotate_args_v1& a, hipStream_t s) {
  if (a.out_dtype == OSCAR_BF16) launch_tr<D, XT, OSCAR_BF16>(a, s);
  else if (a.out_dtype == OSCAR_F16) launch_tr<D, XT, OSCAR_F16>(a, s);
  else launch_tr<D, XT, OSCAR_F32>(a, s);
}

template <int D>
void launch_in(const oscar_rotate_args_v1& a, hipStream_t s) {
  if (a.x_dtype == OSCAR_BF16) launch_out<D, OSCAR_BF16>(a, s);
  else if (a.x_dtype == OSCAR_F16) launch_out<D, OSCAR_F16>(a, s);
  else launch_out<D, OSCAR_F32>(a, s);
}

}  // namespace

}  // namespace oscar

using namespace oscar;

extern "C" int oscar_rotate_v1(const oscar_rotate_args_v1* args, void* stream) {
  if (!args) return fail(-22, "oscar_rotate_v1: null args");
  const oscar_rotate_args_v1& a = *args;
  if (a.rows == 0) return 0;
  if (a.rows < 0 || !a.x || !a.r || !a.out) return fail(-22, "oscar_rotate_v1: invalid arguments");
  if (a.head_dim != 128 && a.head_dim != 256)
    return fail(-22, "oscar_rotate_v1: head_dim %lld unsupported (128/256)", (long long)a.head_dim);
  if (a.x_stride_row < a.head_dim || a.out_stride_row < a.head_dim)
    return fail(-22, "oscar_rotate_v1: row strides smaller than head_dim");
  if ((a.x_dtype != OSCAR_F32 && a.x_dtype != OSCAR_F16 && a.x_dtype != OSCAR_BF16) ||
      (a.out_dtype != OSCAR_F32 && a.out_dtype != OSCAR_F16 && a.out_dtype != OSCAR_BF16))
    return fail(-22, "oscar_rotate_v1: unsupported dtype");
  // rows are read as 16-byte vectors (8 elements of bf16/fp16, 2 x 4 of fp32)
  const int esz = a.x_dtype == OSCAR_F32 ? 4 : 2;
  if ((((uintptr_t)a.x) & 15) || ((a.x_stride_row * esz) & 15) || (((uintptr_t)a.r) & 15))
    return fail(-22, "oscar_rotate_v1: x rows and R must be 16-byte aligned");
  if (a.rows > (int64_t)1 << 36) return fail(-22, "oscar_rotate_v1: too many rows");
  hipStream_t s = (hipStream_t)stream;
  if (a.head_dim == 256) launch_in<256>(a, s);
  else launch_in<128>(a, s);
  OSCAR_CHECK_LAUNCH("rotate_kernel");
  return 0;
}
