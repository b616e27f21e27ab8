// The MoE layer's shared expert in the reference's 8-bit affine form, for the staged and batched paths (the one-row
// fused step computes the same rows inside its launch, moe_fused.hip): reference kernels/fn_moe.metal:40-46 (shared
// gate / up rows in the router dispatch) and :264-290 (shared down rows on rr(silu(g) u)), with the row dot of
// kernels/ne_common.h:58-88. Each row's arithmetic is q8_chunk / q8_wave_sum (moe_device.h), the same in every path.
//
//   moe_q8_gu  wave per gate / up row (its weights held in registers), looping over a block of kQ8Rows input rows:
//              q8gu[t][row] = rr(row . x_t) (gate rows 0 .. inter-1, up rows inter .. 2 inter-1)
//   moe_q8_dn  workgroup of 4 waves: h[t] = rr(silu(g_t) u_t) for its block of input rows into LDS, then 4 down rows
//              per wave: q8o[t][row] = rr(row . h_t)
#include <hip/hip_runtime.h>

#include <algorithm>
#include <type_traits>

#include "exl3_device.h"
#include "kernels.h"
#include "moe_device.h"

namespace ijah {

namespace {

constexpr int kQ8Rows = 8;          // input rows per workgroup (x / h reads per loaded weight row)
constexpr int kQ8MaxInter = 1024;   // h of kQ8Rows rows in LDS
constexpr int kQ8DnRows = 4;        // down rows per wave
constexpr int kQ8FewRows = 32;      // above: the matrix-core form

template <int NCH>
__global__ __launch_bounds__(256) void moe_q8_gu(MoeArgs a) {
  const int lane = threadIdx.x & 63, row = blockIdx.x * 4 + (int)(threadIdx.x >> 6);
  if (row >= 2 * a.inter) return;
  const Q8Off o = q8_offsets(a.hid, a.inter);
  const int proj = row >= a.inter ? 1 : 0, rr = row - proj * a.inter;
  Q8Row<NCH> w;
  q8_load<NCH>(a.q8 + o.w[proj] + (uint64_t)rr * a.hid,
               (const uint32_t *)(a.q8 + o.sb[proj]) + (uint64_t)rr * (a.hid / kQ8Group), a.hid, w);
  const int t1 = min(a.R, (int)(blockIdx.y + 1) * kQ8Rows);
  for (int t = blockIdx.y * kQ8Rows; t < t1; t++) {
    const float v = q8_dot<NCH>(w, a.x + (uint64_t)t * a.hid, a.hid);
    if (lane == 0) a.q8gu[(uint64_t)t * 2 * a.inter + row] = moe_rr(v, a.refr);
  }
}

template <int NCH>
__global__ __launch_bounds__(256) void moe_q8_dn(MoeArgs a) {
  __shared__ __attribute__((aligned(16))) float h[kQ8Rows * kQ8MaxInter];
  const int lane = threadIdx.x & 63, wave = (int)(threadIdx.x >> 6);
  const int t0 = blockIdx.y * kQ8Rows, nt = min(a.R - t0, kQ8Rows);
  for (int i = threadIdx.x; i < nt * a.inter; i += blockDim.x) {
    const int t = i / a.inter, j = i - t * a.inter;
    const float *gu = a.q8gu + (uint64_t)(t0 + t) * 2 * a.inter;
    h[t * a.inter + j] = q8_act(gu[j], gu[a.inter + j], a.refr);
  }
  __syncthreads();
  const Q8Off o = q8_offsets(a.hid, a.inter);
  for (int k = 0; k < kQ8DnRows; k++) {
    const int row = (blockIdx.x * 4 + wave) * kQ8DnRows + k;
    if (row >= a.hid) break;
    Q8Row<NCH> w;
    q8_load<NCH>(a.q8 + o.w[2] + (uint64_t)row * a.inter,
                 (const uint32_t *)(a.q8 + o.sb[2]) + (uint64_t)row * (a.inter / kQ8Group), a.inter, w);
    for (int t = 0; t < nt; t++) {
      const float v = q8_dot<NCH>(w, h + t * a.inter, a.inter);
      if (lane == 0) a.q8o[(uint64_t)(t0 + t) * a.hid + row] = moe_rr(v, a.refr);
    }
  }
}

// ---------------------------------------------------------------------------------------------------- many rows
// R > 32 (prefill): the same rows on the matrix cores. The weight bytes are held a second time as bf16 (exact: a
// byte has at most 8 significant bits), x is split into bf16 hi + lo (16 significant bits reach the products), and
// v_mfma_f32_32x32x16_bf16 sums each group of 128 inputs from zero; per group acc = fmaf(s, P, acc) and
// acc = fmaf(b, sum of x over the group, acc). Rows agree with the one-row arithmetic within f32 rounding (the
// many-row path's bar).
// A workgroup's tile is BT rows x BT outputs, 2 x 2 waves. One group (128 inputs) is staged in LDS at a time, x already
// split (once for the column waves) and the group's row sums with it, while the next group's loads are in flight; a
// group whose lo parts are all zero (inputs that are bf16 values: the model's rounded activations, and h under
// rounding) leaves their products, exact zeros, out. Against waves that load and split their own fragments a k step at
// a time: 300 rows of 2560 -> 1280 and 640 -> 2560, 114 and 27 -> 49 and 15 us; the whole layer 596 -> 508 us, 4000 rows
// at 2048 x 512 1009 -> 886 us. At few rows what is left is the staging's serial VALU work on one wave per SIMD.
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
constexpr int kMmPitch = kQ8Group + 8;  // LDS row pitch in bf16: 16-byte reads of 8 consecutive rows free of conflicts
template <int BT>
constexpr size_t mm_lds() { return (size_t)3 * BT * kMmPitch * 2 + BT * 4 + 8; }

// y[t][o] = rr(row o . x[t]) for t < R, o < nout (a multiple of BT): x f32 rows ldx apart, weights bf16 [nout][in],
// group words [nout][in / 128]
template <int BT>
__global__ __launch_bounds__(256, BT == 64 ? 2 : 1) void moe_q8_mm(const float *x, int ldx, int R, const uint16_t *wbf,
                                                                   const uint32_t *sb, int in, float *y, int ldy,
                                                                   int refr) {
  constexpr int S = BT / 64;  // 32 x 32 tiles per wave and side
  extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
  __bf16 *xh = (__bf16 *)lds, *xl = xh + BT * kMmPitch, *wl = xl + BT * kMmPitch;
  float *sxl = (float *)(wl + BT * kMmPitch);
  int *lowf = (int *)(sxl + BT);  // [2], by the group's parity: some lo part is not zero
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, m = lane & 31, h = lane >> 5;
  const int t0 = blockIdx.x * BT, o0 = blockIdx.y * BT, rw = (wave >> 1) * (BT / 2), cw = (wave & 1) * (BT / 2);
  const int ng = in / kQ8Group;
  // staging: thread t takes inputs 4 (t % 32) .. + 3 of rows t / 32 + 8 i, and 16 bytes of weight rows t / 16 + 16 i
  // 64-tiles keep two groups' loads in flight (their products are too short to cover one), 128-tiles one
  constexpr int D = BT == 64 ? 2 : 1;
  f32x4 xr[D][BT / 8];
  u32x4 wr[D][BT / 16];
  uint32_t sw[D][S];
  auto load = [&](int d, int g) {
#pragma unroll
    for (int i = 0; i < BT / 8; i++)
      xr[d][i] = *(const f32x4 *)(x + (uint64_t)min(t0 + (tid >> 5) + 8 * i, R - 1) * ldx + g * kQ8Group + 4 * (tid & 31));
#pragma unroll
    for (int i = 0; i < BT / 16; i++)
      wr[d][i] = *(const u32x4 *)(wbf + (uint64_t)(o0 + (tid >> 4) + 16 * i) * in + g * kQ8Group + 8 * (tid & 15));
#pragma unroll
    for (int c = 0; c < S; c++) sw[d][c] = sb[(uint64_t)(o0 + cw + 32 * c + m) * ng + g];
  };
  f32x16 tot[S][S];
#pragma unroll
  for (int r = 0; r < S; r++)
#pragma unroll
    for (int c = 0; c < S; c++)
#pragma unroll
      for (int i = 0; i < 16; i++) tot[r][c][i] = 0.f;
  auto group = [&](int d, int g) {
    uint32_t low = 0;  // the lo parts' bits
#pragma unroll
    for (int i = 0; i < BT / 8; i++) {
      const float v[4] = {xr[d][i].x, xr[d][i].y, xr[d][i].z, xr[d][i].w};
      bf16x4 hi, lo;
#pragma unroll
      for (int e = 0; e < 4; e++) {
        hi[e] = (__bf16)v[e];
        lo[e] = (__bf16)(v[e] - (float)hi[e]);
      }
      const uint2 lb = __builtin_bit_cast(uint2, lo);
      low |= lb.x | lb.y;
      const int row = (tid >> 5) + 8 * i;
      *(bf16x4 *)(xh + row * kMmPitch + 4 * (tid & 31)) = hi;
      *(bf16x4 *)(xl + row * kMmPitch + 4 * (tid & 31)) = lo;
      float sx = (v[0] + v[1]) + (v[2] + v[3]);  // the row's sum over the group, on its 32 threads
      sx += xor_lane<1>(sx, lane);
      sx += xor_lane<2>(sx, lane);
      sx += xor_lane<4>(sx, lane);
      sx += xor_lane<8>(sx, lane);
      sx += xor_lane<16>(sx, lane);
      if ((tid & 31) == 0) sxl[row] = sx;
    }
#pragma unroll
    for (int i = 0; i < BT / 16; i++) *(u32x4 *)(wl + ((tid >> 4) + 16 * i) * kMmPitch + 8 * (tid & 15)) = wr[d][i];
    if (__any(low != 0) && lane == 0) lowf[g & 1] = 1;
    __syncthreads();
    const int any = __builtin_amdgcn_readfirstlane(lowf[g & 1]);
    if (tid == 0) lowf[(g + 1) & 1] = 0;  // the next group's, written past the barrier below
    uint32_t word[S];
#pragma unroll
    for (int c = 0; c < S; c++) word[c] = sw[d][c];
    if (g + D < ng) load(d, g + D);
    f32x16 P[S][S];
#pragma unroll
    for (int r = 0; r < S; r++)
#pragma unroll
      for (int c = 0; c < S; c++)
#pragma unroll
        for (int i = 0; i < 16; i++) P[r][c][i] = 0.f;
    auto products = [&](auto with_lo) {
#pragma unroll
      for (int st = 0; st < kQ8Group / 16; st++) {
        bf16x8 b[S];
#pragma unroll
        for (int c = 0; c < S; c++) b[c] = *(const bf16x8 *)(wl + (cw + 32 * c + m) * kMmPitch + 16 * st + 8 * h);
#pragma unroll
        for (int part = 0; part < (decltype(with_lo)::value ? 2 : 1); part++) {
          bf16x8 a[S];
#pragma unroll
          for (int r = 0; r < S; r++)
            a[r] = *(const bf16x8 *)((part ? xl : xh) + (rw + 32 * r + m) * kMmPitch + 16 * st + 8 * h);
#pragma unroll
          for (int r = 0; r < S; r++)
#pragma unroll
            for (int c = 0; c < S; c++) P[r][c] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[r], b[c], P[r][c], 0, 0, 0);
        }
      }
    };
    if (any)
      products(std::true_type{});
    else
      products(std::false_type{});
    // lane: column cw + 32 c + m, rows rw + 32 r + 8 (i / 4) + 4 h + i % 4
#pragma unroll
    for (int r = 0; r < S; r++)
#pragma unroll
      for (int j = 0; j < 4; j++) {
        const float4 s4 = *(const float4 *)(sxl + rw + 32 * r + 8 * j + 4 * h);
        const float sx[4] = {s4.x, s4.y, s4.z, s4.w};
#pragma unroll
        for (int c = 0; c < S; c++)
#pragma unroll
          for (int e = 0; e < 4; e++) {
            const float t = __builtin_fmaf(bf16_f32(word[c] & 0xFFFFu), P[r][c][4 * j + e], tot[r][c][4 * j + e]);
            tot[r][c][4 * j + e] = __builtin_fmaf(bf16_f32(word[c] >> 16), sx[e], t);
          }
      }
    __syncthreads();  // the group's LDS is read
  };
  if (tid == 0) lowf[0] = 0;
  __syncthreads();
#pragma unroll
  for (int d = 0; d < D; d++)
    if (d < ng) load(d, d);
  for (int g = 0; g < ng; g += D) {
#pragma unroll
    for (int d = 0; d < D; d++)
      if (g + d < ng) group(d, g + d);
  }
#pragma unroll
  for (int r = 0; r < S; r++)
#pragma unroll
    for (int c = 0; c < S; c++)
#pragma unroll
      for (int i = 0; i < 16; i++) {
        const int t = t0 + rw + 32 * r + 8 * (i / 4) + 4 * h + i % 4;
        if (t < R) y[(uint64_t)t * ldy + o0 + cw + 32 * c + m] = moe_rr(tot[r][c][i], refr);
      }
}
// 128 x 128 tiles where they still give every CU a workgroup, else 64 x 64
void launch_mm(const float *x, int ldx, int R, const uint16_t *wbf, const uint32_t *sb, int in, int nout, float *y,
               int ldy, int refr, hipStream_t s) {
  if ((R + 127) / 128 * (nout / 128) >= 256)
    hipLaunchKernelGGL(moe_q8_mm<128>, dim3((R + 127) / 128, nout / 128), dim3(256), mm_lds<128>(), s, x, ldx, R, wbf, sb,
                       in, y, ldy, refr);
  else
    hipLaunchKernelGGL(moe_q8_mm<64>, dim3((R + 63) / 64, nout / 64), dim3(256), mm_lds<64>(), s, x, ldx, R, wbf, sb, in,
                       y, ldy, refr);
}
// h = rr(silu(g) u) in place of g: q8gu[t][j] for j < inter (the down GEMM's input rows, 2 inter apart)
__global__ __launch_bounds__(256) void moe_q8_act(float *gu, int R, int inter, int refr) {
  const uint64_t i = blockIdx.x * 256ull + threadIdx.x;
  if (i >= (uint64_t)R * inter) return;
  const uint64_t t = i / inter, j = i % inter;
  float *row = gu + t * 2 * inter;
  row[j] = q8_act(row[j], row[inter + j], refr);
}
// the weight bytes as bf16 values (exact), once at set-up
__global__ void q8_to_bf16(const uint8_t *w, uint16_t *o, uint64_t n) {
  for (uint64_t i = blockIdx.x * 256ull + threadIdx.x; i < n; i += (uint64_t)gridDim.x * 256)
    o[i] = (uint16_t)(__float_as_uint((float)w[i]) >> 16);
}

template <int NCH>
void launch_gu(const MoeArgs &a, hipStream_t s) {
  hipLaunchKernelGGL(moe_q8_gu<NCH>, dim3((2 * a.inter + 3) / 4, (a.R + kQ8Rows - 1) / kQ8Rows), dim3(256), 0, s, a);
}
template <int NCH>
void launch_dn(const MoeArgs &a, hipStream_t s) {
  hipLaunchKernelGGL(moe_q8_dn<NCH>, dim3((a.hid + 4 * kQ8DnRows - 1) / (4 * kQ8DnRows), (a.R + kQ8Rows - 1) / kQ8Rows),
                     dim3(256), 0, s, a);
}

}  // namespace

// the dynamic LDS limits, once at device set-up
void init_q8_attrs() {
  IJ_HIP(hipFuncSetAttribute((const void *)&moe_q8_mm<64>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)mm_lds<64>()));
  IJ_HIP(hipFuncSetAttribute((const void *)&moe_q8_mm<128>, hipFuncAttributeMaxDynamicSharedMemorySize,
                             (int)mm_lds<128>()));
}

bool moe_q8_supported(int hid, int inter) {
  return hid % kQ8Group == 0 && inter % kQ8Group == 0 && hid <= 8192 && inter <= kQ8MaxInter && inter % 64 == 0;
}

void launch_q8_bf16(const uint8_t *q8, uint16_t *bf, int hid, int inter, hipStream_t s) {
  const uint64_t n = 3ull * hid * inter;
  hipLaunchKernelGGL(q8_to_bf16, dim3((unsigned)std::min<uint64_t>(4096, (n + 255) / 256)), dim3(256), 0, s, q8, bf, n);
}

void launch_moe_q8(const MoeArgs &a, hipStream_t s) {
  IJ_CHECK(a.q8 && a.q8gu && a.q8o, "8-bit shared expert: no block or scratch");
  IJ_CHECK(moe_q8_supported(a.hid, a.inter), "8-bit shared expert: %d x %d not supported", a.hid, a.inter);
  if (a.R > kQ8FewRows && a.q8bf) {  // many rows: the matrix cores
    const Q8Off o = q8_offsets(a.hid, a.inter);
    const uint32_t *sb = (const uint32_t *)(a.q8 + o.sb[0]);
    launch_mm(a.x, a.hid, a.R, a.q8bf, sb, a.hid, 2 * a.inter, a.q8gu, 2 * a.inter, a.refr, s);
    hipLaunchKernelGGL(moe_q8_act, dim3((unsigned)(((uint64_t)a.R * a.inter + 255) / 256)), dim3(256), 0, s, a.q8gu,
                       a.R, a.inter, a.refr);
    launch_mm(a.q8gu, 2 * a.inter, a.R, a.q8bf + 2ull * a.inter * a.hid, (const uint32_t *)(a.q8 + o.sb[2]), a.inter,
              a.hid, a.q8o, a.hid, a.refr, s);
    return;
  }
  const int ng = (a.hid + 1023) / 1024;
  if (ng <= 2)
    launch_gu<2>(a, s);
  else if (ng <= 4)
    launch_gu<4>(a, s);
  else
    launch_gu<8>(a, s);
  launch_dn<1>(a, s);  // inter <= 1024: one chunk per lane
}

}  // namespace ijah
