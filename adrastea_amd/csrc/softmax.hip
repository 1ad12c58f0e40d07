// Row-wise softmax with temperature over a contiguous [heads, h, w] fp16 tensor
// (adrastea_kernels/cpp/normalize.cu:147-220; host call adrastea_models/src/kernels.rs:892-915,
// in place between QK^T and P.V at llama.rs:551, clip.rs:385, whisper.rs:432):
//   v_i   = float(in_i) / temp
//   out_i = fp16( expf(v_i - max_j v_j) / sum_j expf(v_j - max_j v_j) )
// The operation is bound by reading and writing the tensor once each.  Rows of up to 4096
// elements are held in registers by one wavefront (one pass over memory, shuffle reductions):
// 16-byte accesses of the row's own elements where the rows are 16-byte aligned, of the aligned
// pieces a row touches where they start at any even address (a row length that is no multiple of
// 8); longer rows take a three-pass kernel with one workgroup per row.
#include "adr_common.hpp"

namespace adr {

namespace {

// e^x for x <= 0 (and NaN, and -inf -> 0) as the hardware's 2^t of t = x * log2 e.  The rounding
// of the product and of the constant put t off by at most 7.3e-8 |t|, the exp2 unit adds one ulp:
// a relative error below 1.4e-6 wherever the result can still be seen in fp16 (|t| < 25), 0.3 %
// of one fp16 step.  Carrying the product in two floats brings that to 2 ulp of expf but costs six
// more VALU instructions per element, and this kernel is bound by them as much as by memory
// (106 us against 95 us on 65536 rows of 2048).
__device__ __forceinline__ float exp_neg(float x) {
  return __builtin_amdgcn_exp2f(x * 1.44269502162933349609375f);
}

__device__ __forceinline__ float wave_max(float v) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) v = fmaxf(v, __shfl_xor(v, off, 64));
  return v;
}
__device__ __forceinline__ float wave_sum(float v) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
  return v;
}

// NV 16-byte vectors per lane: rows of w <= 512 * NV elements, w % 8 == 0, 16-byte aligned rows.
template <int NV>
__global__ __launch_bounds__(256) void softmax_rows_reg_kernel(half_t* out, const half_t* in,
                                                               int64_t rows, int w, float temp) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int64_t row = (int64_t)blockIdx.x * 4 + wave;
  if (row >= rows) return;
  const half_t* src = in + row * w;
  half_t* dst = out + row * w;
  float v[NV][8];
  float mx = -INFINITY;
  const bool unit_temp = temp == 1.0f;
#pragma unroll
  for (int i = 0; i < NV; i++) {
    const int c = (i * 64 + lane) * 8;
    if (c < w) {
      const half8_t x = *(const half8_t*)(src + c);
#pragma unroll
      for (int e = 0; e < 8; e++) {
        v[i][e] = unit_temp ? (float)x[e] : (float)x[e] / temp;  // x / 1 == x: skip the division
        mx = fmaxf(mx, v[i][e]);
      }
    } else {
#pragma unroll
      for (int e = 0; e < 8; e++) v[i][e] = -INFINITY;
    }
  }
  mx = wave_max(mx);
  float sum = 0.0f;
#pragma unroll
  for (int i = 0; i < NV; i++) {
    const int c = (i * 64 + lane) * 8;
    if (c < w) {
#pragma unroll
      for (int e = 0; e < 8; e++) {
        v[i][e] = exp_neg(v[i][e] - mx);
        sum += v[i][e];
      }
    }
  }
  sum = wave_sum(sum);
  // v / sum for 32+ values per lane: one reciprocal per row and a product per value (within
  // 1.5 ulp of the quotient, before the narrowing to fp16 takes 13 bits off)
  const float rs = 1.0f / sum;
#pragma unroll
  for (int i = 0; i < NV; i++) {
    const int c = (i * 64 + lane) * 8;
    if (c < w) {
      half8_t r;
#pragma unroll
      for (int e = 0; e < 8; e++) {
        r[e] = (half_t)(v[i][e] * rs);
      }
      // streaming store: the probabilities are consumed by a later launch
      __builtin_nontemporal_store(r, (half8_t*)(dst + c));
    }
  }
}

// The same for rows that start at any even address and hold any number of elements: a sequence
// length that is no multiple of 8 (Whisper's 1500 positions, CLIP's 77 and 257, any odd prompt
// length).  Bound by memory once its requests are whole: chunks are the 16-byte pieces of the address
// space the row touches, not of the row, so every load is one aligned 16-byte access -- the first
// and the last chunk of a row bring elements of the rows beside it, which are replaced by -inf -- and
// so is every store where `out` lies as `in` does (in place always); a row's end pieces go out as
// the dwords and halves that are its own.  Chunks counted from the row's first element had to be
// shifted into place, a second request per chunk: 48000 rows of 1500 80 -> 64 us = 4.5 TB/s, 30000 of
// them 52.7 -> 42.5, 32016 of 2001 65.8 -> 52.5, 24008 of 3001 76.4 -> 59.7, 32760 of 4095 119.5 -> 103,
// 12240 of 1530 22.7 -> 19.1; 16352 of 2044 29.7 either way.  (Cached stores
// instead of streaming ones, and a contiguous piece of the tensor for each die, change nothing.)
// NV: chunks per lane; every row of the tensor touches at most 64 NV chunks (see the launch).
template <int NV>
__global__ __launch_bounds__(256) void softmax_rows_anyrow_kernel(half_t* out, const half_t* in,
                                                                  int64_t rows, int w, float temp) {
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int64_t row = (int64_t)blockIdx.x * 4 + wave;
  if (row >= rows) return;
  const half_t* src = in + row * w;
  half_t* dst = out + row * w;
  const uintptr_t base = (uintptr_t)src & ~(uintptr_t)15;
  const int lead = (int)((uintptr_t)src & 15) >> 1;  // elements of the first chunk before the row
  const int chunks = (lead + w + 7) >> 3;
  const bool same = (((uintptr_t)dst ^ (uintptr_t)src) & 15) == 0;
  half8_t x[NV];
  // (the tensor's own first and last row alone can have chunks that reach outside of it: those rows
  // are read element by element)
  if (base >= (uintptr_t)in && base + 16 * (uintptr_t)chunks <= (uintptr_t)(in + rows * w)) {
#pragma unroll
    for (int i = 0; i < NV; i++)
      x[i] = *(const ADR_GLOBAL_AS half8_t*)(base + 16 * (uintptr_t)min(i * 64 + lane, chunks - 1));
  } else {
#pragma unroll
    for (int i = 0; i < NV; i++)
#pragma unroll
      for (int e = 0; e < 8; e++)
        x[i][e] = src[min(max((i * 64 + lane) * 8 - lead + e, 0), w - 1)];
  }
  float v[NV][8];
  float mx = -INFINITY;
  const bool unit_temp = temp == 1.0f;
#pragma unroll
  for (int i = 0; i < NV; i++) {
    const int c = (i * 64 + lane) * 8 - lead;  // the chunk's first element, as counted from the row's
#pragma unroll
    for (int e = 0; e < 8; e++) v[i][e] = unit_temp ? (float)x[i][e] : (float)x[i][e] / temp;
    if (i == 0 || (i + 1) * 64 >= chunks) {  // (whole chunks for all lanes in between)
#pragma unroll
      for (int e = 0; e < 8; e++) v[i][e] = (unsigned)(c + e) < (unsigned)w ? v[i][e] : -INFINITY;
    }
#pragma unroll
    for (int e = 0; e < 8; e++) mx = fmaxf(mx, v[i][e]);
  }
  mx = wave_max(mx);
  float sum = 0.0f;
#pragma unroll
  for (int i = 0; i < NV; i++)
#pragma unroll
    for (int e = 0; e < 8; e++) {
      v[i][e] = exp_neg(v[i][e] - mx);  // (-inf - mx: 0 for the elements beside the row)
      sum += v[i][e];
    }
  sum = wave_sum(sum);
  const float rs = 1.0f / sum;
#pragma unroll
  for (int i = 0; i < NV; i++) {
    const int c = (i * 64 + lane) * 8 - lead;
    half8_t r;
#pragma unroll
    for (int e = 0; e < 8; e++) r[e] = (half_t)(v[i][e] * rs);
    if (c >= 0 && c + 8 <= w) {
      if (same) __builtin_nontemporal_store(r, (half8_t*)(dst + c));
      else store8_any(dst + c, r);
    } else if (c < w) {
#pragma unroll
      for (int e = 0; e < 8; e += 2) {
        const bool first = (unsigned)(c + e) < (unsigned)w, second = (unsigned)(c + e + 1) < (unsigned)w;
        if (first && second && same) *(half2_t*)(dst + c + e) = half2_t{r[e], r[e + 1]};
        else {
          if (first) dst[c + e] = r[e];
          if (second) dst[c + e + 1] = r[e + 1];
        }
      }
    }
  }
}

// The same on chunks counted from the row's first element, moved with load8_any / store8_any.  Up to 1024
// elements, one or two chunks per lane, the second request is cheaper than the masks of the pieces at
// both ends (544714 rows of 77 218 us against 238, 163202 of 257 69.2 against 75.6, 125955 of 333 54.9 against
// 59.7; 436 of 601 3.7 against 3.9, 69788 of them 57.6 either way; at 1100 238 rows take 4.6 against 4.0 and
// 38130 58 against 45).  So it is for the lengths just short of 2048 whose aligned pieces are one more
// per lane, unless the tensor is large (4098 rows of 2047 11.5 against 12.6, 8196 17.8 against 19.5, 20490
// 42.5 against 40.1).
template <int NV>
__global__ __launch_bounds__(256) void softmax_rows_shifted_kernel(half_t* out, const half_t* in,
                                                                  int64_t rows, int w, float temp) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int64_t row = (int64_t)blockIdx.x * 4 + wave;
  if (row >= rows) return;
  const half_t* src = in + row * w;
  half_t* dst = out + row * w;
  const uintptr_t end = (uintptr_t)(in + rows * w);  // one past the tensor's last element
  const uintptr_t last = ((end + 3) & ~(uintptr_t)3) - 4;
  float v[NV][8];
  float mx = -INFINITY;
  const bool unit_temp = temp == 1.0f;
#pragma unroll
  for (int i = 0; i < NV; i++) {
    const int c = (i * 64 + lane) * 8;
    // (chunks past the row read the row's first chunk again: no load under a lane mask)
    const half8_t x = load8_any(src + (c < w ? c : 0), last);
#pragma unroll
    for (int e = 0; e < 8; e++) {
      const float t = unit_temp ? (float)x[e] : (float)x[e] / temp;
      v[i][e] = c + e < w ? t : -INFINITY;
      mx = fmaxf(mx, v[i][e]);
    }
  }
  mx = wave_max(mx);
  float sum = 0.0f;
#pragma unroll
  for (int i = 0; i < NV; i++)
#pragma unroll
    for (int e = 0; e < 8; e++) {
      v[i][e] = exp_neg(v[i][e] - mx);  // (-inf - mx: 0 for the elements past the row)
      sum += v[i][e];
    }
  sum = wave_sum(sum);
  const float rs = 1.0f / sum;
#pragma unroll
  for (int i = 0; i < NV; i++) {
    const int c = (i * 64 + lane) * 8;
    half8_t r;
#pragma unroll
    for (int e = 0; e < 8; e++) r[e] = (half_t)(v[i][e] * rs);
    if (c + 8 <= w) {
      store8_any(dst + c, r);
    } else if (c < w) {
#pragma unroll
      for (int e = 0; e < 8; e++)
        if (c + e < w) dst[c + e] = r[e];
    }
  }
}

// Any width and alignment: one workgroup per row, three passes over the row.
__global__ __launch_bounds__(256) void softmax_rows_general_kernel(half_t* out, const half_t* in,
                                                                   int w, float temp) {
  __shared__ float red[4];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int64_t row = blockIdx.x;
  const half_t* src = in + row * w;
  half_t* dst = out + row * w;
  float mx = -INFINITY;
  for (int i = tid; i < w; i += 256) mx = fmaxf(mx, (float)src[i] / temp);
  mx = wave_max(mx);
  if (lane == 0) red[wave] = mx;
  __syncthreads();
  mx = fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
  __syncthreads();
  float sum = 0.0f;
  for (int i = tid; i < w; i += 256) sum += expf((float)src[i] / temp - mx);
  sum = wave_sum(sum);
  if (lane == 0) red[wave] = sum;
  __syncthreads();
  sum = (red[0] + red[1]) + (red[2] + red[3]);
  // in place: an element is read and then written by the same thread
  for (int i = tid; i < w; i += 256) dst[i] = (half_t)(expf((float)src[i] / temp - mx) / sum);
}

}  // namespace

hipError_t launch_softmax_rows(hipStream_t stream, half_t* out, const half_t* in, int64_t rows,
                               int w, float temp) {
  const bool vec = w % 8 == 0 && w <= 4096 && ((uintptr_t)out % 16) == 0 && ((uintptr_t)in % 16) == 0;
  if (vec) {
    const int64_t blocks = (rows + 3) / 4;
    if (blocks > 0x7fffffffLL) return hipErrorInvalidConfiguration;
    const dim3 grid((unsigned)blocks), block(256);
    if (w <= 512)
      hipLaunchKernelGGL(softmax_rows_reg_kernel<1>, grid, block, 0, stream, out, in, rows, w, temp);
    else if (w <= 1024)
      hipLaunchKernelGGL(softmax_rows_reg_kernel<2>, grid, block, 0, stream, out, in, rows, w, temp);
    else if (w <= 2048)
      hipLaunchKernelGGL(softmax_rows_reg_kernel<4>, grid, block, 0, stream, out, in, rows, w, temp);
    else
      hipLaunchKernelGGL(softmax_rows_reg_kernel<8>, grid, block, 0, stream, out, in, rows, w, temp);
  } else if (w <= 4096) {
    const int64_t blocks = (rows + 3) / 4;
    if (blocks > 0x7fffffffLL) return hipErrorInvalidConfiguration;
    const dim3 grid((unsigned)blocks), block(256);
    // Chunks per lane as the row that starts worst needs them: rows start at `in` plus multiples of w,
    // so their first chunks hold as many elements of other rows as `in` does modulo the largest power
    // of two in w (or 8), and at most that much short of a chunk more.
    const int g = w % 2 ? 1 : w % 4 ? 2 : w % 8 ? 4 : 8;
    const int lead = 8 - g + (int)(((uintptr_t)in & 15) >> 1) % g;
    const int per_lane = ((lead + w + 7) / 8 + 63) / 64;
    if (w <= 512)
      hipLaunchKernelGGL(softmax_rows_shifted_kernel<1>, grid, block, 0, stream, out, in, rows, w, temp);
    else if (w <= 1024)
      hipLaunchKernelGGL(softmax_rows_shifted_kernel<2>, grid, block, 0, stream, out, in, rows, w, temp);
    else if (per_lane == 5 && w < 2048 && rows <= 12288)
      hipLaunchKernelGGL(softmax_rows_shifted_kernel<4>, grid, block, 0, stream, out, in, rows, w, temp);
    else switch (per_lane) {
      case 3: hipLaunchKernelGGL(softmax_rows_anyrow_kernel<3>, grid, block, 0, stream, out, in, rows, w, temp); break;
      case 4: hipLaunchKernelGGL(softmax_rows_anyrow_kernel<4>, grid, block, 0, stream, out, in, rows, w, temp); break;
      case 5: hipLaunchKernelGGL(softmax_rows_anyrow_kernel<5>, grid, block, 0, stream, out, in, rows, w, temp); break;
      case 6: hipLaunchKernelGGL(softmax_rows_anyrow_kernel<6>, grid, block, 0, stream, out, in, rows, w, temp); break;
      case 7: hipLaunchKernelGGL(softmax_rows_anyrow_kernel<7>, grid, block, 0, stream, out, in, rows, w, temp); break;
      case 8: hipLaunchKernelGGL(softmax_rows_anyrow_kernel<8>, grid, block, 0, stream, out, in, rows, w, temp); break;
      default: hipLaunchKernelGGL(softmax_rows_anyrow_kernel<9>, grid, block, 0, stream, out, in, rows, w, temp); break;
    }
  } else {
    if (rows > 0x7fffffffLL) return hipErrorInvalidConfiguration;
    hipLaunchKernelGGL(softmax_rows_general_kernel, dim3((unsigned)rows), dim3(256), 0, stream, out,
                       in, w, temp);
  }
  return hipGetLastError();
}

}  // namespace adr
