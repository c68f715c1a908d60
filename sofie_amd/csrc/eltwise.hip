// HBM-bound elementwise operators: QuantizeLinear / DequantizeLinear, the stand-alone activations,
// broadcast Add, GlobalAveragePool.  Each thread moves 16 bytes of the widest operand per step and
// the grid strides over the tensor, so the launches stay coalesced for any length.
#include "common.hpp"
#include <cfloat>
#include <type_traits>

namespace sofie_hip {

static inline unsigned grid_for(size_t work_items, unsigned block = 256, unsigned max_blocks = 256 * 32)
{
   size_t b = (work_items + block - 1) / block;
   if (b < 1)
      b = 1;
   if (b > max_blocks)
      b = max_blocks;
   return (unsigned)b;
}

// Divisor31 of common.hpp for indices of any size.
struct Divisor64 {
   unsigned long long d;
   explicit Divisor64(long long extent) : d((unsigned long long)extent) {}
   typedef unsigned long long index;
   __device__ __forceinline__ index over(index n) const { return n / d; }
};

typedef float f32x4 __attribute__((ext_vector_type(4)));

// q = sat8(rne(x / scale)), fp32 division (ONNX QuantizeLinear, zero point 0)
// A load per thread: the divisions of four values take a wave that is alone on its SIMD as long as the trip to memory, and sixteen of them, with four loads in flight,
// three times as long.  us with sixteen -> four, launches of a captured loop: over data in the caches 16 K values 2.74 -> 2.27, 1 M 2.97 -> 2.58, 3 M 4.08 -> 3.77, 50 M 38.4 -> 35.9; over
// data that is not (600 MB in turn) 2.37 -> 1.85, 3.66 -> 3.19, 5.56 -> 5.36, 47.3 -> 46.1 (past 8 M values a thread takes several, one after the other).  Behind the other kernels of a
// network, traced: 16 K 2.7 -> 2.2, 1 M 4.1 .. 4.8 and 4.5 .. 4.8, 3 M 5.2 -> 5.1: what bounds the larger ones there is the trip.
__global__ __launch_bounds__(256) void quantize_linear_kernel(int8_t *__restrict__ dst, const float *__restrict__ src,
                                                               size_t n, float scale, int vec)
{
   const size_t stride = (size_t)gridDim.x * blockDim.x;
   size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x;
   if (vec) {
      const size_t n4 = n / 4;
      for (size_t k = i; k < n4; k += stride) {
         const float4 v = ((const float4 *)src)[k];
         const int q0 = quantize_rne_sat8(__fdiv_rn(v.x, scale));
         const int q1 = quantize_rne_sat8(__fdiv_rn(v.y, scale));
         const int q2 = quantize_rne_sat8(__fdiv_rn(v.z, scale));
         const int q3 = quantize_rne_sat8(__fdiv_rn(v.w, scale));
         ((uint32_t *)dst)[k] = (uint32_t)(q0 & 0xff) | ((uint32_t)(q1 & 0xff) << 8) | ((uint32_t)(q2 & 0xff) << 16) | ((uint32_t)(q3 & 0xff) << 24);
      }
      i += n4 * 4;
      if (i < n)
         dst[i] = (int8_t)quantize_rne_sat8(__fdiv_rn(src[i], scale));
   } else {
      for (; i < n; i += stride)
         dst[i] = (int8_t)quantize_rne_sat8(__fdiv_rn(src[i], scale));
   }
}

template <typename T>
__global__ __launch_bounds__(256) void dequantize_linear_kernel(float *__restrict__ dst, const T *__restrict__ src, size_t n,
                                                                 float scale)
{
   const size_t stride = (size_t)gridDim.x * blockDim.x;
   for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < n; i += stride)
      dst[i] = mul_nofma((float)src[i], scale);
}

__global__ __launch_bounds__(256) void unary_f32_kernel(float *dst, const float *src, size_t n, PostChain chain, int vec)
{
   const size_t stride = (size_t)gridDim.x * blockDim.x;
   size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x;
   if (vec) {
      const size_t n4 = n / 4;
      for (; i < n4; i += stride) {
         float4 v = ((const float4 *)src)[i];
         v.x = apply_chain(v.x, chain);
         v.y = apply_chain(v.y, chain);
         v.z = apply_chain(v.z, chain);
         v.w = apply_chain(v.w, chain);
         ((float4 *)dst)[i] = v;
      }
      i = n4 * 4 + (blockIdx.x * (size_t)blockDim.x + threadIdx.x);
      if (i < n)
         dst[i] = apply_chain(src[i], chain);
   } else {
      for (; i < n; i += stride)
         dst[i] = apply_chain(src[i], chain);
   }
}

// the sum of a window that begins at (i, j, k) by the elements it counts
__device__ __forceinline__ float pool_average(float sum, const sofie_pool3d_desc &d, int i, int j, int k)
{
   int nsum = d.k[0] * d.k[1] * d.k[2];
   if (d.dynamic_divisor) {
      const int start[3] = {i, j, k};
      nsum = 1;
#pragma unroll
      for (int a = 0; a < 3; ++a) {
         const int hi = d.count_include_pad ? d.in[a] + d.pad_end[a] : d.in[a];
         const int lo = d.count_include_pad ? start[a] : (start[a] > 0 ? start[a] : 0);
         nsum *= (start[a] + d.k[a] < hi ? start[a] + d.k[a] : hi) - lo;
      }
   }
   return __fdiv_rn(sum, (float)nsum);
}

// One output element per thread (grid-stride); neighbouring lanes take neighbouring outputs of the fastest axis, so the
// window rows they read overlap and lie next to each other in memory.  Three spatial axes, slowest first (a 2-D pooling has a
// first axis of extent 1): the window is visited axis 0, then 1, then 2, one fp32 addition at a time -- the order of the
// reference's generated loops, so an average has the bits of the reference's scalar loop.
// KH, KW > 0: a flat window of that size.  All its elements are loaded before the first is used (a loop over a clipped window waits
// for memory once per element); positions outside the image read its nearest element and count as -inf or +0, which change neither
// a maximum nor a sum that began at +0.  Bound by the lines that the strided rows touch in the vector L1.
template <typename DIV, int KH, int KW>
__global__ __launch_bounds__(256) void pool_f32_kernel(float *__restrict__ Y, const float *__restrict__ X, sofie_pool3d_desc d, size_t total, DIV out0, DIV out1,
                                                       DIV out2)
{
   typedef typename DIV::index index;
   const size_t stride = (size_t)gridDim.x * blockDim.x;
   const size_t s0 = (size_t)d.in[1] * (size_t)d.in[2], s1 = (size_t)d.in[2];
   for (size_t idx = blockIdx.x * (size_t)blockDim.x + threadIdx.x; idx < total; idx += stride) {
      const index row = out2.over((index)idx), slice = out1.over(row), plane = out0.over(slice);
      const int o2 = (int)((index)idx - row * out2.d), o1 = (int)(row - slice * out1.d), o0 = (int)(slice - plane * out0.d);
      const int i = o0 * d.stride[0] - d.pad_begin[0], j = o1 * d.stride[1] - d.pad_begin[1], k = o2 * d.stride[2] - d.pad_begin[2];
      const float *x = X + (size_t)plane * (size_t)d.in[0] * s0;
      float value = d.mode == SOFIE_POOL_MAX ? -INFINITY : 0.0f;
      if constexpr (KH > 0) {
         float v[KH][KW];
#pragma unroll
         for (int m = 0; m < KH; ++m) {
            const int at = j + m < 0 ? 0 : j + m < d.in[1] ? j + m : d.in[1] - 1;
            const float *r = x + (size_t)at * s1;
#pragma unroll
            for (int p = 0; p < KW; ++p)
               v[m][p] = r[k + p < 0 ? 0 : k + p < d.in[2] ? k + p : d.in[2] - 1];
         }
#pragma unroll
         for (int m = 0; m < KH; ++m)
#pragma unroll
            for (int p = 0; p < KW; ++p) {
               const bool inside = (unsigned)(j + m) < (unsigned)d.in[1] && (unsigned)(k + p) < (unsigned)d.in[2];
               if (d.mode == SOFIE_POOL_MAX) {
                  const float xv = inside ? v[m][p] : -INFINITY;
                  if (xv > value)
                     value = xv;
               } else {
                  value += inside ? v[m][p] : 0.0f;
               }
            }
      } else {
         const int l0 = i < 0 ? 0 : i, l1 = i + d.k[0] < d.in[0] ? i + d.k[0] : d.in[0];
         const int m0 = j < 0 ? 0 : j, m1 = j + d.k[1] < d.in[1] ? j + d.k[1] : d.in[1];
         const int p0 = k < 0 ? 0 : k, p1 = k + d.k[2] < d.in[2] ? k + d.k[2] : d.in[2];
         for (int l = l0; l < l1; ++l)
            for (int m = m0; m < m1; ++m)
               for (int p = p0; p < p1; ++p) {
                  const float xv = x[(size_t)l * s0 + (size_t)m * s1 + p];
                  if (d.mode == SOFIE_POOL_MAX) {
                     if (xv > value)
                        value = xv;
                  } else {
                     value += xv;
                  }
               }
      }
      if (d.mode == SOFIE_POOL_AVERAGE)
         value = pool_average(value, d, i, j, k);
      Y[idx] = value;
   }
}

// A flat 3 x 3 window with strides of two, at most one column of padding before a row.  Three loads per window row touch every line three times; here a lane
// loads a pair, its middle and right column, and takes the left one from the lane before it (the first lane of a wave or of a row loads it), and a thread has two
// outputs, one below the other, which share a row.  The order of the general kernel's sums and comparisons.  us before -> after: 2048 planes of 64 x 64 12.0 ->
// 8.5 (42 MB), 16384 of them 107 -> 60 (5.6 TB/s), 300 of 95 x 95 5.5 -> 4.5, 64 of 64 x 64 3.1 either way (a launch).
template <typename DIV>
__global__ __launch_bounds__(256) void pool_f32_3x3_step2_kernel(float *__restrict__ Y, const float *__restrict__ X, sofie_pool3d_desc d, size_t total, DIV rows, DIV columns)
{
   typedef typename DIV::index index;
   typedef float pair __attribute__((ext_vector_type(2), aligned(4)));
   const size_t stride = (size_t)gridDim.x * blockDim.x;
   const int H = d.in[1], W = d.in[2];
   for (size_t idx = blockIdx.x * (size_t)blockDim.x + threadIdx.x; idx < total; idx += stride) {
      const index row = columns.over((index)idx), plane = rows.over(row);
      const int o2 = (int)((index)idx - row * columns.d), o1 = (int)(row - plane * rows.d) * 2;
      const int j = o1 * 2 - d.pad_begin[1], k = o2 * 2 - d.pad_begin[2];
      const float *x = X + (size_t)plane * H * W;
      const int at = k + 1 < W - 1 ? k + 1 : W - 2;
      const bool loads_left = k >= 0 && (o2 == 0 || (threadIdx.x & 63) == 0);
      pair p[5];
      float left[5] = {0.0f, 0.0f, 0.0f, 0.0f, 0.0f};
      const float *line[5];
#pragma unroll
      for (int m = 0; m < 5; ++m) {
         const int r = j + m < 0 ? 0 : j + m < H ? j + m : H - 1;
         line[m] = x + (size_t)r * W;
         p[m] = *(const pair *)(line[m] + at);
      }
      if (loads_left) {
#pragma unroll
         for (int m = 0; m < 5; ++m)
            left[m] = line[m][k < W ? k : W - 1];
      }
      const float outside = d.mode == SOFIE_POOL_MAX ? -INFINITY : 0.0f;
      float v[5][3];
#pragma unroll
      for (int m = 0; m < 5; ++m) {
         const float middle = p[m].x, right = p[m].y; // (a bit cast of a vector's element takes the first one)
         const float before = __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, right), 0x138, 0xf, 0xf, false)); // wave_shr:1
         const bool inside = (unsigned)(j + m) < (unsigned)H;
         v[m][0] = inside && (unsigned)k < (unsigned)W ? (loads_left ? left[m] : before) : outside;
         v[m][1] = inside && k + 1 < W ? (at == k + 1 ? middle : right) : outside;
         v[m][2] = inside && k + 2 < W ? right : outside;
      }
      float *y = Y + ((size_t)plane * d.out[1] + o1) * d.out[2] + o2;
#pragma unroll
      for (int q = 0; q < 2; ++q) {
         float value = outside;
#pragma unroll
         for (int m = 0; m < 3; ++m)
#pragma unroll
            for (int c = 0; c < 3; ++c) {
               const float xv = v[2 * q + m][c];
               value = d.mode == SOFIE_POOL_MAX ? (xv > value ? xv : value) : value + xv;
            }
         if (d.mode == SOFIE_POOL_AVERAGE)
            value = pool_average(value, d, 0, j + 2 * q, k);
         if (o1 + q < d.out[1])
            y[(size_t)q * d.out[2]] = value;
      }
   }
}

struct AddShape {
   int rank;
   long long y[6], sa[6], sb[6]; // output dims, element strides of A and B (0 where broadcast)
};

struct TransposeShape {
   int rank;
   long long y[6], sx[6]; // output dims and, per OUTPUT axis, the element stride of the input axis it reads
};

// Axes that lie one behind the other in the input as in the output are one axis, axes of extent 1 none (the swap of two inner axes
// of a four-dimensional tensor keeps four, a permutation that moves nothing keeps one).
static TransposeShape fold_axes(const TransposeShape &in)
{
   TransposeShape out{};
   for (int k = 0; k < in.rank; ++k) {
      if (in.y[k] == 1)
         continue;
      if (out.rank > 0 && out.sx[out.rank - 1] == in.y[k] * in.sx[k]) {
         out.y[out.rank - 1] *= in.y[k];
         out.sx[out.rank - 1] = in.sx[k];
      } else {
         out.y[out.rank] = in.y[k];
         out.sx[out.rank++] = in.sx[k];
      }
   }
   if (out.rank == 0) {
      out.rank = 1;
      out.y[0] = out.sx[0] = 1;
   }
   return out;
}

// One element T (a float, or four that are neighbours on both sides) per thread and step: writes are coalesced, reads are strided by
// the permutation.  `sx` counts elements of T.  Heads of an attention block apart (2048 x 384): 5.3 -> 5.2 us, together again 5.8 -> 3.1 us.
template <typename DIV>
struct GatherAxes {
   int rank;
   DIV y[6]; // the slowest axis is never divided by
   long long sx[6];
};
template <typename T, typename DIV>
__global__ __launch_bounds__(256) void transpose_f32_kernel(T *__restrict__ Y, const T *__restrict__ X, size_t n, GatherAxes<DIV> sh)
{
   typedef typename DIV::index index;
   const size_t stride = (size_t)gridDim.x * blockDim.x;
   for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < n; i += stride) {
      index rest = (index)i;
      long long ix = 0;
#pragma unroll
      for (int d = 5; d > 0; --d)
         if (d < sh.rank) {
            const index q = sh.y[d].over(rest);
            ix += (long long)(rest - q * sh.y[d].d) * sh.sx[d];
            rest = q;
         }
      Y[i] = X[ix + (long long)rest * sh.sx[0]];
   }
}

static int launch_transpose(sofie_hip_ctx *ctx, float *Y, const float *X, size_t n, const TransposeShape &any)
{
   TransposeShape sh = fold_axes(any);
   // four floats at a time where the fastest axis is contiguous and every address a multiple of 16 bytes
   bool vec = sh.sx[sh.rank - 1] == 1 && sh.y[sh.rank - 1] % 4 == 0 && (((uintptr_t)X | (uintptr_t)Y) & 15) == 0;
   for (int k = 0; k + 1 < sh.rank; ++k)
      vec = vec && sh.sx[k] % 4 == 0;
   if (vec) {
      n /= 4;
      sh.y[sh.rank - 1] /= 4;
      for (int k = 0; k + 1 < sh.rank; ++k)
         sh.sx[k] /= 4;
   }
   auto go = [&](auto div) {
      typedef decltype(div) DIV;
      GatherAxes<DIV> g{sh.rank, {div, div, div, div, div, div}, {}};
      for (int k = 0; k < sh.rank; ++k) {
         g.y[k] = DIV(sh.y[k]);
         g.sx[k] = sh.sx[k];
      }
      if (vec)
         launch_kernel((transpose_f32_kernel<f32x4, DIV>), dim3(grid_for(n)), dim3(256), 0, ctx->stream, (f32x4 *)Y, (const f32x4 *)X, n, g);
      else
         launch_kernel((transpose_f32_kernel<float, DIV>), dim3(grid_for(n)), dim3(256), 0, ctx->stream, Y, X, n, g);
   };
   if (n < (1ull << 31))
      go(Divisor31(1));
   else
      go(Divisor64(1));
   return launch_status("transpose_f32_kernel");
}

__global__ __launch_bounds__(256) void copy_rows_kernel(uint32_t *__restrict__ dst, size_t dst_pitch, const uint32_t *__restrict__ src, size_t src_pitch,
                                                         size_t rows, size_t row_words)
{
   const size_t n = rows * row_words, stride = (size_t)gridDim.x * blockDim.x;
   for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < n; i += stride) {
      const size_t r = i / row_words, c = i - r * row_words;
      dst[r * dst_pitch + c] = src[r * src_pitch + c];
   }
}

__device__ __forceinline__ float binary_op(float a, float b, int op, float param)
{
   switch (op) {
   case SOFIE_BINARY_SUB: return a - b;
   case SOFIE_BINARY_MUL: return mul_nofma(a, b);
   case SOFIE_BINARY_DIV: return __fdiv_rn(a, b);
   case SOFIE_BINARY_POW: return powf(a, b);
   case SOFIE_BINARY_MAX: return a < b ? b : a;
   case SOFIE_BINARY_MIN: return b < a ? b : a;
   case SOFIE_BINARY_ADD_DIV: return __fdiv_rn(a + b, param);
   default: return a + b;
   }
}

__global__ __launch_bounds__(256) void binary_f32_kernel(float *__restrict__ Y, const float *__restrict__ A, const float *__restrict__ B, size_t n,
                                                          AddShape sh, int op, float param)
{
   const size_t stride = (size_t)gridDim.x * blockDim.x;
   for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < n; i += stride) {
      size_t rest = i;
      long long ia = 0, ib = 0;
      for (int d = sh.rank - 1; d >= 0; --d) {
         long long idx = (long long)(rest % (size_t)sh.y[d]);
         rest /= (size_t)sh.y[d];
         ia += idx * sh.sa[d];
         ib += idx * sh.sb[d];
      }
      Y[i] = binary_op(A[ia], B[ib], op, param);
   }
}

__global__ __launch_bounds__(256) void add_f32_kernel(float *__restrict__ Y, const float *__restrict__ A,
                                                       const float *__restrict__ B, size_t n, AddShape sh)
{
   const size_t stride = (size_t)gridDim.x * blockDim.x;
   for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < n; i += stride) {
      size_t rest = i;
      long long ia = 0, ib = 0;
      for (int d = sh.rank - 1; d >= 0; --d) {
         long long idx = (long long)(rest % (size_t)sh.y[d]);
         rest /= (size_t)sh.y[d];
         ia += idx * sh.sa[d];
         ib += idx * sh.sb[d];
      }
      Y[i] = A[ia] + B[ib];
   }
}

// One wave per (n,c) plane: lanes stride over the plane, then a wave reduction.
template <typename T, typename ACC>
__global__ __launch_bounds__(256) void gap_kernel(float *__restrict__ Y, const T *__restrict__ X, int NC, int HW, float mul, int vec)
{
   const int plane = blockIdx.x * 4 + (threadIdx.x >> 6);
   const int lane = threadIdx.x & 63;
   if (plane >= NC)
      return;
   const T *p = X + (size_t)plane * HW;
   ACC s = 0;
   if (sizeof(T) == 4 && vec) {
      // four 16-byte loads in flight: 4096 planes of 1024 floats 6.9 -> 5.3 us
      const int n4 = HW / 4;
      f32x4 part = {0.f, 0.f, 0.f, 0.f};
      for (int i = lane; i < n4; i += 256) {
         f32x4 v[4];
#pragma unroll
         for (int u = 0; u < 4; ++u)
            v[u] = ((const f32x4 *)p)[i + 64 * u < n4 ? i + 64 * u : i];
         __builtin_amdgcn_sched_barrier(0); // the compiler would take the loads one after the other
#pragma unroll
         for (int u = 0; u < 4; ++u)
#pragma unroll
            for (int e = 0; e < 4; ++e)
               part[e] += i + 64 * u < n4 ? v[u][e] : 0.0f;
      }
      s = (ACC)((part[0] + part[1]) + (part[2] + part[3]));
   } else {
      for (int i = lane; i < HW; i += 64)
         s += (ACC)p[i];
   }
   if constexpr (sizeof(T) == 4) {
      s = (ACC)sum_over_lanes((float)s);
   } else {
#pragma unroll
      for (int off = 32; off > 0; off >>= 1)
         s += __shfl_xor(s, off, 64);
   }
   // fp32 input: sum / HW as the reference's pooling loop ends with `value /= float(nsum)`
   // (core/inc/SOFIE/operators/ROperator_Pool.hxx:362-368); int8 input: (float(sum) * scale) / HW
   if (lane == 0)
      Y[plane] = __fdiv_rn(mul_nofma((float)s, mul), (float)HW);
}

// NHWC int8 input, any channel count: one workgroup per image; thread c (strided) sums channel c over the
// pixels, so consecutive lanes read consecutive bytes.
__global__ __launch_bounds__(256) void gap_i8_nhwc_kernel(float *__restrict__ Y, const int8_t *__restrict__ X, int C, int HW,
                                                           float scale)
{
   const int8_t *p = X + (size_t)blockIdx.x * HW * C;
   for (int c = threadIdx.x; c < C; c += blockDim.x) {
      int s = 0;
      for (int i = 0; i < HW; ++i)
         s += (int)p[(size_t)i * C + c];
      Y[(size_t)blockIdx.x * C + c] = __fdiv_rn(mul_nofma((float)s, scale), (float)HW);
   }
}

// A contiguous line of at most G * NV vectors of VEC floats, held in the registers of G neighbouring lanes (G a power of two: short
// lines share a wave): it is read once, and the passes over it are arithmetic.  Vector j of a lane is vector lane + G j of the line.
template <int VEC, int NV>
struct LineRegisters {
   float v[NV][VEC];
   int lane, G, vectors; // vectors in the line
   __device__ __forceinline__ bool has(int j) const { return lane + G * j < vectors; }
   __device__ __forceinline__ void load(const float *line, float outside)
   {
#pragma unroll
      for (int j = 0; j < NV; ++j) {
         if constexpr (VEC == 4) {
            f32x4 q = {outside, outside, outside, outside};
            if (has(j))
               q = ((const f32x4 *)line)[lane + G * j];
#pragma unroll
            for (int e = 0; e < 4; ++e)
               v[j][e] = q[e];
         } else {
            v[j][0] = has(j) ? line[lane + G * j] : outside;
         }
      }
   }
   __device__ __forceinline__ void store(float *line) const
   {
#pragma unroll
      for (int j = 0; j < NV; ++j)
         if (has(j)) {
            if constexpr (VEC == 4)
               ((f32x4 *)line)[lane + G * j] = f32x4{v[j][0], v[j][1], v[j][2], v[j][3]};
            else
               line[lane + G * j] = v[j][0];
         }
   }
   __device__ __forceinline__ float sum_over_lanes(float s) const
   {
      return sofie_hip::sum_over_lanes(s, G);
   }
};

// Launches `line.template operator()<VEC, NV>(G, blocks)` for `lines` lines of `len` floats if they fit the registers.
template <class F>
static bool with_line_registers(long long lines, int len, bool aligned, F &&line)
{
   const bool vec = aligned && len % 4 == 0;
   const int vectors = vec ? len / 4 : len;
   int G = 1;
   while (G < 64 && G < vectors)
      G *= 2;
   const int need = (vectors + G - 1) / G;
   const long long waves = (lines + 64 / G - 1) / (64 / G), all = (waves + 3) / 4, blocks = all < 256 * 64 ? all : 256 * 64;
   if (vec) {
      if (need <= 1)
         line(std::integral_constant<int, 4>{}, std::integral_constant<int, 1>{}, G, (unsigned)blocks);
      else if (need <= 2)
         line(std::integral_constant<int, 4>{}, std::integral_constant<int, 2>{}, G, (unsigned)blocks);
      else if (need <= 4)
         line(std::integral_constant<int, 4>{}, std::integral_constant<int, 4>{}, G, (unsigned)blocks);
      else
         return false;
   } else {
      if (need <= 1)
         line(std::integral_constant<int, 1>{}, std::integral_constant<int, 1>{}, G, (unsigned)blocks);
      else if (need <= 4)
         line(std::integral_constant<int, 1>{}, std::integral_constant<int, 4>{}, G, (unsigned)blocks);
      else if (need <= 16)
         line(std::integral_constant<int, 1>{}, std::integral_constant<int, 16>{}, G, (unsigned)blocks);
      else
         return false;
   }
   return true;
}

// Softmax over contiguous lines (inner == 1) that fit the registers of a group of lanes; one read, one exponential per element.
// 12288 lines of 128: 8.0 -> 5.0 us.
template <int VEC, int NV>
__global__ __launch_bounds__(256) void softmax_lines_f32_kernel(float *__restrict__ Y, const float *__restrict__ X, long long lines, int A, int G, int log_softmax)
{
   const int in_wave = threadIdx.x & 63, per_wave = 64 / G;
   LineRegisters<VEC, NV> x;
   x.lane = in_wave & (G - 1);
   x.G = G;
   x.vectors = A / VEC;
   const long long wave = (long long)blockIdx.x * 4 + (threadIdx.x >> 6), nwaves = (long long)gridDim.x * 4;
   for (long long first = wave * per_wave; first < lines; first += nwaves * per_wave) {
      const long long line = first + in_wave / G;
      const bool live = line < lines;
      const long long at = (live ? line : lines - 1) * A;
      x.load(X + at, -INFINITY);
      float vmax = -INFINITY;
#pragma unroll
      for (int j = 0; j < NV; ++j)
#pragma unroll
         for (int e = 0; e < VEC; ++e)
            vmax = x.v[j][e] > vmax ? x.v[j][e] : vmax;
      vmax = over_lanes(vmax, G, [](float a, float b) { return b > a ? b : a; });
      float sum = 0.0f;
#pragma unroll
      for (int j = 0; j < NV; ++j)
#pragma unroll
         for (int e = 0; e < VEC; ++e) {
            const float centred = x.v[j][e] - vmax, ex = expf(centred);
            sum += x.has(j) ? ex : 0.0f;
            x.v[j][e] = log_softmax ? centred : ex;
         }
      sum = x.sum_over_lanes(sum);
      const float log_sum = log_softmax ? logf(sum) : 0.0f, inv_sum = 1.0f / sum;
#pragma unroll
      for (int j = 0; j < NV; ++j)
#pragma unroll
         for (int e = 0; e < VEC; ++e)
            x.v[j][e] = log_softmax ? x.v[j][e] - log_sum : mul_nofma(x.v[j][e], inv_sum);
      if (live)
         x.store(Y + at);
   }
}

// Any other softmax over the middle dimension of [outer, A, inner]: one wave per (outer, inner) line, lanes stride over the axis
// (consecutive lanes read consecutive elements when inner == 1), three passes over a line that stays in cache.
__global__ __launch_bounds__(256) void softmax_f32_kernel(float *__restrict__ Y, const float *__restrict__ X, long long lines, int A, long long inner,
                                                          int log_softmax)
{
   const int lane = threadIdx.x & 63;
   const long long wave = (long long)blockIdx.x * 4 + (threadIdx.x >> 6), nwaves = (long long)gridDim.x * 4;
   for (long long line = wave; line < lines; line += nwaves) {
      const long long o = line / inner, in = line - o * inner;
      const float *x = X + o * A * inner + in;
      float *y = Y + o * A * inner + in;
      float vmax = -INFINITY;
      for (int i = lane; i < A; i += 64) {
         const float v = x[i * inner];
         vmax = v > vmax ? v : vmax;
      }
      vmax = over_lanes(vmax, 64, [](float a, float b) { return b > a ? b : a; });
      float sum = 0.0f;
      for (int i = lane; i < A; i += 64)
         sum += expf(x[i * inner] - vmax);
      sum = sum_over_lanes(sum);
      if (log_softmax) {
         const float log_sum = logf(sum);
         for (int i = lane; i < A; i += 64)
            y[i * inner] = x[i * inner] - vmax - log_sum;
      } else if (inner == 1) {
         const float inv_sum = 1.0f / sum;
         for (int i = lane; i < A; i += 64)
            y[i] = mul_nofma(expf(x[i] - vmax), inv_sum);
      } else {
         for (int i = lane; i < A; i += 64)
            y[i * inner] = __fdiv_rn(expf(x[i * inner] - vmax), sum);
      }
   }
}

__device__ __forceinline__ float reduce_start(int op)
{
   return op == SOFIE_REDUCE_PROD ? 1.0f : op == SOFIE_REDUCE_MAX ? -FLT_MAX : op == SOFIE_REDUCE_MIN ? FLT_MAX : 0.0f;
}
__device__ __forceinline__ float reduce_step(float y, float x, int op)
{
   switch (op) {
   case SOFIE_REDUCE_SUM_SQUARE:
   case SOFIE_REDUCE_L2: return y + mul_nofma(x, x);
   case SOFIE_REDUCE_PROD: return mul_nofma(y, x);
   case SOFIE_REDUCE_MAX: return y < x ? x : y;
   case SOFIE_REDUCE_MIN: return x < y ? x : y;
   default: return y + x;
   }
}
// folds two partial results (the tree form): partial sums of squares add, everything else combines as a step does
__device__ __forceinline__ float reduce_merge(float a, float b, int op)
{
   return (op == SOFIE_REDUCE_SUM_SQUARE || op == SOFIE_REDUCE_L2) ? a + b : reduce_step(a, b, op);
}
__device__ __forceinline__ float reduce_finish(float y, int A, int op)
{
   return op == SOFIE_REDUCE_MEAN ? __fdiv_rn(y, (float)A) : op == SOFIE_REDUCE_L2 ? sqrtf(y) : y;
}

// One output per thread, the reduced elements in increasing order: the reference's loop (neighbouring threads read neighbouring `inner`).
__global__ __launch_bounds__(256) void reduce_f32_kernel(float *__restrict__ Y, const float *__restrict__ X, size_t outputs, int A, long long inner, int op)
{
   const size_t stride = (size_t)gridDim.x * blockDim.x;
   for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < outputs; i += stride) {
      const size_t o = i / (size_t)inner, in = i - o * (size_t)inner;
      const float *x = X + o * (size_t)A * (size_t)inner + in;
      float y = reduce_start(op);
      for (int a = 0; a < A; ++a)
         y = reduce_step(y, x[(size_t)a * (size_t)inner], op);
      Y[i] = reduce_finish(y, A, op);
   }
}

// Long contiguous lines: one wave per line, lanes stride over it, then a shuffle tree.
__global__ __launch_bounds__(256) void reduce_lines_f32_kernel(float *__restrict__ Y, const float *__restrict__ X, long long lines, int A, int op)
{
   const int lane = threadIdx.x & 63;
   const long long wave = (long long)blockIdx.x * 4 + (threadIdx.x >> 6), nwaves = (long long)gridDim.x * 4;
   for (long long line = wave; line < lines; line += nwaves) {
      const float *x = X + line * A;
      float y = reduce_start(op);
      for (int a = lane; a < A; a += 64)
         y = reduce_step(y, x[a], op);
      y = over_lanes(y, 64, [&](float a, float b) { return reduce_merge(a, b, op); });
      if (lane == 0)
         Y[line] = reduce_finish(y, A, op);
   }
}

// LayerNormalization of rows that fit the registers of a group of lanes: mean, then the centred sum of squares, then the output,
// from one read.  2048 rows of 384: 7.8 -> 4.1 us.
template <int VEC, int NV>
__global__ __launch_bounds__(256) void layernorm_lines_f32_kernel(float *__restrict__ Y, const float *__restrict__ X, const float *__restrict__ scale,
                                                                  const float *__restrict__ bias, long long rows, int L, int G, float epsilon,
                                                                  float *__restrict__ mean_out, float *__restrict__ inv_std_out)
{
   const int in_wave = threadIdx.x & 63, per_wave = 64 / G;
   LineRegisters<VEC, NV> x, s, b;
   x.lane = s.lane = b.lane = in_wave & (G - 1);
   x.G = s.G = b.G = G;
   x.vectors = s.vectors = b.vectors = L / VEC;
   const long long wave = (long long)blockIdx.x * 4 + (threadIdx.x >> 6), nwaves = (long long)gridDim.x * 4;
   for (long long first = wave * per_wave; first < rows; first += nwaves * per_wave) {
      const long long row = first + in_wave / G;
      const bool live = row < rows;
      const long long at = (live ? row : rows - 1) * L;
      x.load(X + at, 0.0f);
      s.load(scale, 0.0f); // after the first row from the cache
      if (bias)
         b.load(bias, 0.0f);
      float mean = 0.0f;
#pragma unroll
      for (int j = 0; j < NV; ++j)
#pragma unroll
         for (int e = 0; e < VEC; ++e)
            mean += x.v[j][e];
      mean = __fdiv_rn(x.sum_over_lanes(mean), (float)L);
      float sum = 0.0f;
#pragma unroll
      for (int j = 0; j < NV; ++j)
#pragma unroll
         for (int e = 0; e < VEC; ++e) {
            x.v[j][e] -= mean;
            sum += x.has(j) ? mul_nofma(x.v[j][e], x.v[j][e]) : 0.0f;
         }
      sum = x.sum_over_lanes(sum);
      const float inv_std = __fdiv_rn(1.0f, sqrtf(__fdiv_rn(sum, (float)L) + epsilon));
      if (live && x.lane == 0) {
         if (mean_out)
            mean_out[row] = mean;
         if (inv_std_out)
            inv_std_out[row] = inv_std;
      }
#pragma unroll
      for (int j = 0; j < NV; ++j)
#pragma unroll
         for (int e = 0; e < VEC; ++e) {
            float v = mul_nofma(mul_nofma(s.v[j][e], inv_std), x.v[j][e]);
            if (bias)
               v += b.v[j][e];
            x.v[j][e] = v;
         }
      if (live)
         x.store(Y + at);
   }
}

// Longer rows: one wave per row of L elements, lanes stride over the row.
__global__ __launch_bounds__(256) void layernorm_f32_kernel(float *__restrict__ Y, const float *__restrict__ X, const float *__restrict__ scale,
                                                            const float *__restrict__ bias, long long rows, int L, float epsilon,
                                                            float *__restrict__ mean_out, float *__restrict__ inv_std_out)
{
   const int lane = threadIdx.x & 63;
   const long long wave = (long long)blockIdx.x * 4 + (threadIdx.x >> 6), nwaves = (long long)gridDim.x * 4;
   for (long long row = wave; row < rows; row += nwaves) {
      const float *x = X + row * L;
      float *y = Y + row * L;
      float mean = 0.0f;
      for (int j = lane; j < L; j += 64)
         mean += x[j];
      mean = sum_over_lanes(mean);
      mean = __fdiv_rn(mean, (float)L);
      float sum = 0.0f;
      for (int j = lane; j < L; j += 64) {
         const float tmp = x[j] - mean;
         sum += mul_nofma(tmp, tmp);
      }
      sum = sum_over_lanes(sum);
      const float inv_std = __fdiv_rn(1.0f, sqrtf(__fdiv_rn(sum, (float)L) + epsilon));
      if (lane == 0) {
         if (mean_out)
            mean_out[row] = mean;
         if (inv_std_out)
            inv_std_out[row] = inv_std;
      }
      for (int j = lane; j < L; j += 64) {
         float v = mul_nofma(mul_nofma(scale[j], inv_std), x[j] - mean);
         if (bias)
            v += bias[j];
         y[j] = v;
      }
   }
}

// The last step of an average whose integer plane sums already exist (a convolution added them up in its store).
__global__ __launch_bounds__(256) void plane_sums_to_average_kernel(float *__restrict__ Y, const int32_t *__restrict__ sums, int NC, int HW,
                                                                    float scale)
{
   const int i = blockIdx.x * blockDim.x + threadIdx.x;
   if (i < NC)
      Y[i] = __fdiv_rn(mul_nofma((float)sums[i], scale), (float)HW);
}

// The same, and the sums are cleared behind the read: a buffer that starts out zero is zero again for the next convolution.
__global__ __launch_bounds__(256) void plane_sums_take_average_kernel(float *__restrict__ Y, int32_t *__restrict__ sums, int NC, int HW, float scale)
{
   const int i = blockIdx.x * blockDim.x + threadIdx.x;
   if (i < NC) {
      Y[i] = __fdiv_rn(mul_nofma((float)sums[i], scale), (float)HW);
      sums[i] = 0;
   }
}

// NHWC int8 input with C a multiple of 16 (and 16-byte aligned): one workgroup per (image, block of 16 << chunks_log2 channels).
// A thread owns 16 consecutive channels and every (512 >> chunks_log2)-th pixel, reads 16 bytes per pixel, and the
// per-thread int32 sums are added up (integer sums: exact in any order) across a wave's lanes in registers, and over the eight waves through LDS.  us, with all of it through
// LDS -> now: 5 images of 28 x 28 x 64 3.60 -> 2.79, one of 8 x 8 x 256 2.81 -> 1.97, 100 of 50 x 50 x 32 3.79 -> 3.03, 256 of 64 x 64 x 256 (read from memory) 38.5 -> 38.2.
constexpr int GAP_THREADS = 512;
__global__ __launch_bounds__(GAP_THREADS) void gap_i8_nhwc_vec_kernel(float *__restrict__ Y, const int8_t *__restrict__ X, int C, int HW,
                                                               float scale, int chunks_log2)
{
   __shared__ int part[GAP_THREADS / 64][256];
   const int img = blockIdx.x, c_first = blockIdx.y << (4 + chunks_log2);
   const int groups = GAP_THREADS >> chunks_log2;
   const int chunk = threadIdx.x & ((1 << chunks_log2) - 1), group = threadIdx.x >> chunks_log2;
   int s[16];
#pragma unroll
   for (int k = 0; k < 16; ++k)
      s[k] = 0;
   if (c_first + chunk * 16 < C) {
      const int8_t *p = X + (size_t)img * HW * C + c_first + chunk * 16;
      typedef int int4v __attribute__((ext_vector_type(4)));
      // eight pixels per round: eight independent 16-byte loads in flight per lane, in the last round too
      for (int i = group; i < HW; i += 8 * groups) {
         int4v v[8];
#pragma unroll
         for (int u = 0; u < 8; ++u)
            v[u] = *(const int4v *)(p + (size_t)(i + u * groups < HW ? i + u * groups : i) * C);
         __builtin_amdgcn_sched_barrier(0); // the compiler would take the loads one after the other
#pragma unroll
         for (int u = 0; u < 8; ++u)
            if (i + u * groups < HW) {
#pragma unroll
               for (int d = 0; d < 4; ++d)
#pragma unroll
                  for (int b = 0; b < 4; ++b)
                     s[4 * d + b] = __builtin_amdgcn_sdot4(v[u][d], 1 << (8 * b), s[4 * d + b], false); // adds byte b
            }
      }
   }
   // Over the pixels of a wave: halves of the wave, then of either half, keep the sums of half of the channels each; lanes of a row of 16 that differ in their pixels alone
   // add up in place.  Lane l then holds channels l / 16 * 4 .. + 3 of its 16.
#pragma unroll
   for (int k = 0; k < 8; ++k) {
      const auto both = __builtin_amdgcn_permlane32_swap((unsigned)s[k], (unsigned)s[k + 8], false, false);
      s[k] = (int)((unsigned)both[0] + (unsigned)both[1]);
   }
#pragma unroll
   for (int k = 0; k < 4; ++k) {
      const auto both = __builtin_amdgcn_permlane16_swap((unsigned)s[k], (unsigned)s[k + 4], false, false);
      s[k] = (int)((unsigned)both[0] + (unsigned)both[1]);
   }
   auto fold = [&](auto control) {
#pragma unroll
      for (int k = 0; k < 4; ++k)
         s[k] += __builtin_amdgcn_update_dpp(0, s[k], decltype(control)::value, 0xf, 0xf, false);
   };
   if (chunks_log2 < 4)
      fold(std::integral_constant<int, 0x128>{}); // row_ror:8
   if (chunks_log2 < 3)
      fold(std::integral_constant<int, 0x124>{}); // row_ror:4, the same as lane ^ 4 now
   if (chunks_log2 < 2)
      fold(std::integral_constant<int, 0x122>{});
   if (chunks_log2 < 1)
      fold(std::integral_constant<int, 0x121>{});
   const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
   if ((lane & 15) >> chunks_log2 == 0) {
#pragma unroll
      for (int k = 0; k < 4; ++k)
         part[wave][chunk * 16 + (lane >> 4) * 4 + k] = s[k];
   }
   __syncthreads();
   const int of = threadIdx.x;
   if (of < 16 << chunks_log2 && c_first + of < C) {
      int tot = 0;
#pragma unroll
      for (int w = 0; w < GAP_THREADS / 64; ++w)
         tot += part[w][of];
      Y[(size_t)img * C + c_first + of] = __fdiv_rn(mul_nofma((float)tot, scale), (float)HW);
   }
}

// Y = (X - mean[c]) * fused_scale[c] + bias[c] (+ relu); element i belongs to channel (i / spatial) % C.  T: a float, or four of one
// plane; the extents count elements of T.  Four of them are in flight per lane, a workgroup's width apart.  64 x 64 planes of 32x32: 10.0 -> 6.6 us.
template <typename T, typename DIV>
__global__ __launch_bounds__(256) void batchnorm_f32_kernel(T *__restrict__ Y, const T *__restrict__ X, const float *__restrict__ fused,
                                                             const float *__restrict__ mean, const float *__restrict__ bias, size_t n, DIV channels, DIV spatial,
                                                             int relu)
{
   typedef typename DIV::index index;
   constexpr int VEC = sizeof(T) / sizeof(float);
   const size_t stride = (size_t)gridDim.x * blockDim.x * 4;
   for (size_t base = blockIdx.x * (size_t)blockDim.x * 4 + threadIdx.x; base < n; base += stride) {
      T x[4];
      float f[4], m[4], b[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) {
         const size_t at = base + (size_t)u * blockDim.x < n ? base + (size_t)u * blockDim.x : n - 1;
         x[u] = X[at];
         const index plane = spatial.over((index)at), c = plane - channels.over(plane) * channels.d;
         f[u] = fused[c], m[u] = mean[c], b[u] = bias[c];
      }
      __builtin_amdgcn_sched_barrier(0); // the compiler would take the loads one after the other
#pragma unroll
      for (int u = 0; u < 4; ++u) {
         auto one = [&](float v) {
            v = __fmul_rn(v - m[u], f[u]) + b[u];
            return relu && !(v > 0.0f) ? 0.0f : v;
         };
         if constexpr (VEC == 4) {
#pragma unroll
            for (int e = 0; e < 4; ++e)
               x[u][e] = one(x[u][e]);
         } else {
            x[u] = one(x[u]);
         }
         if (base + (size_t)u * blockDim.x < n)
            Y[base + (size_t)u * blockDim.x] = x[u];
      }
   }
}

} // namespace sofie_hip

using namespace sofie_hip;

extern "C" {

int sofie_hip_quantize_linear(sofie_hip_ctx *ctx, int8_t *dst, const float *src, size_t n, float scale)
{
   SOFIE_HIP_REQUIRE(ctx != nullptr, "sofie_hip_quantize_linear: ctx is NULL");
   if (n == 0)
      return SOFIE_HIP_OK;
   SOFIE_HIP_REQUIRE(dst && src, "sofie_hip_quantize_linear: NULL pointer");
   SOFIE_HIP_REQUIRE(scale > 0.0f, "sofie_hip_quantize_linear: scale must be positive");
   const int vec = (((uintptr_t)src & 15) == 0) && (((uintptr_t)dst & 3) == 0);
   launch_kernel(quantize_linear_kernel, dim3(grid_for(vec ? (n + 3) / 4 : n)), dim3(256), 0, ctx->stream, dst, src, n, scale, vec);
   return launch_status("quantize_linear_kernel");
}

int sofie_hip_dequantize_linear_i8(sofie_hip_ctx *ctx, float *dst, const int8_t *src, size_t n, float scale)
{
   SOFIE_HIP_REQUIRE(ctx != nullptr, "sofie_hip_dequantize_linear_i8: ctx is NULL");
   if (n == 0)
      return SOFIE_HIP_OK;
   SOFIE_HIP_REQUIRE(dst && src, "sofie_hip_dequantize_linear_i8: NULL pointer");
   launch_kernel(dequantize_linear_kernel<int8_t>, dim3(grid_for(n)), dim3(256), 0, ctx->stream, dst, src, n, scale);
   return launch_status("dequantize_linear_kernel");
}

int sofie_hip_dequantize_linear_i32(sofie_hip_ctx *ctx, float *dst, const int32_t *src, size_t n, float scale)
{
   SOFIE_HIP_REQUIRE(ctx != nullptr, "sofie_hip_dequantize_linear_i32: ctx is NULL");
   if (n == 0)
      return SOFIE_HIP_OK;
   SOFIE_HIP_REQUIRE(dst && src, "sofie_hip_dequantize_linear_i32: NULL pointer");
   launch_kernel(dequantize_linear_kernel<int32_t>, dim3(grid_for(n)), dim3(256), 0, ctx->stream, dst, src, n, scale);
   return launch_status("dequantize_linear_kernel");
}

static int launch_unary_chain(sofie_hip_ctx *ctx, float *dst, const float *src, size_t n, const PostChain &chain)
{
   const int vec = (((uintptr_t)src & 15) == 0) && (((uintptr_t)dst & 15) == 0);
   launch_kernel(unary_f32_kernel, dim3(grid_for(vec ? (n + 3) / 4 : n)), dim3(256), 0, ctx->stream, dst, src, n, chain, vec);
   return launch_status("unary_f32_kernel");
}

int sofie_hip_unary_f32(sofie_hip_ctx *ctx, float *dst, const float *src, size_t n, int32_t act, float act_alpha)
{
   SOFIE_HIP_REQUIRE(ctx != nullptr, "sofie_hip_unary_f32: ctx is NULL");
   PostChain chain;
   int bad = 0;
   SOFIE_HIP_REQUIRE(make_post_chain(chain, act, act_alpha, nullptr, bad), "sofie_hip_unary_f32: unknown activation %d", act);
   if (n == 0)
      return SOFIE_HIP_OK;
   SOFIE_HIP_REQUIRE(dst && src, "sofie_hip_unary_f32: NULL pointer");
   return launch_unary_chain(ctx, dst, src, n, chain);
}

int sofie_hip_unary_chain_f32(sofie_hip_ctx *ctx, float *dst, const float *src, size_t n, const sofie_post_ops *ops)
{
   SOFIE_HIP_REQUIRE(ctx != nullptr && ops != nullptr, "sofie_hip_unary_chain_f32: NULL argument");
   PostChain chain;
   int bad = 0;
   SOFIE_HIP_REQUIRE(make_post_chain(chain, SOFIE_ACT_NONE, 0.0f, ops, bad),
                     "sofie_hip_unary_chain_f32: unknown operator %d (or more than %d operators)", bad, SOFIE_MAX_POST_OPS);
   if (n == 0)
      return SOFIE_HIP_OK;
   SOFIE_HIP_REQUIRE(dst && src, "sofie_hip_unary_chain_f32: NULL pointer");
   return launch_unary_chain(ctx, dst, src, n, chain);
}

int sofie_hip_add_f32(sofie_hip_ctx *ctx, const sofie_add_desc *d)
{
   return sofie_hip_binary_f32(ctx, d, SOFIE_BINARY_ADD, 0.0f);
}

int sofie_hip_binary_f32(sofie_hip_ctx *ctx, const sofie_add_desc *d, int32_t op, float param)
{
   SOFIE_HIP_REQUIRE(ctx && d, "sofie_hip_add_f32: NULL argument");
   SOFIE_HIP_REQUIRE(op >= SOFIE_BINARY_ADD && op <= SOFIE_BINARY_LAST, "sofie_hip_binary_f32: unknown operator %d", op);
   SOFIE_HIP_REQUIRE(d->rank >= 0 && d->rank <= 6, "sofie_hip_add_f32: rank %d not in [0,6]", d->rank);
   AddShape sh;
   sh.rank = d->rank;
   size_t n = 1;
   long long stride_a = 1, stride_b = 1;
   for (int i = d->rank - 1; i >= 0; --i) {
      SOFIE_HIP_REQUIRE(d->y_shape[i] >= 0, "sofie_hip_add_f32: negative dimension");
      SOFIE_HIP_REQUIRE((d->a_shape[i] == d->y_shape[i] || d->a_shape[i] == 1) &&
                           (d->b_shape[i] == d->y_shape[i] || d->b_shape[i] == 1),
                        "sofie_hip_add_f32: operand dimension %d cannot be broadcast to the output", i);
      sh.y[i] = d->y_shape[i];
      sh.sa[i] = (d->a_shape[i] == 1 && d->y_shape[i] != 1) ? 0 : stride_a;
      sh.sb[i] = (d->b_shape[i] == 1 && d->y_shape[i] != 1) ? 0 : stride_b;
      stride_a *= d->a_shape[i];
      stride_b *= d->b_shape[i];
      n *= (size_t)d->y_shape[i];
   }
   if (n == 0)
      return SOFIE_HIP_OK;
   SOFIE_HIP_REQUIRE(d->A && d->B && d->Y, "sofie_hip_add_f32: NULL pointer");
   if (op == SOFIE_BINARY_ADD) {
      launch_kernel(add_f32_kernel, dim3(grid_for(n)), dim3(256), 0, ctx->stream, d->Y, d->A, d->B, n, sh);
      return launch_status("add_f32_kernel");
   }
   launch_kernel(binary_f32_kernel, dim3(grid_for(n)), dim3(256), 0, ctx->stream, d->Y, d->A, d->B, n, sh, op, param);
   return launch_status("binary_f32_kernel");
}

int sofie_hip_batchnorm_f32(sofie_hip_ctx *ctx, float *Y, const float *X, const float *fused_scale, const float *mean,
                            const float *bias, int32_t N, int32_t C, int32_t spatial, int32_t relu)
{
   SOFIE_HIP_REQUIRE(ctx != nullptr, "sofie_hip_batchnorm_f32: ctx is NULL");
   SOFIE_HIP_REQUIRE(N >= 0 && C > 0 && spatial > 0, "sofie_hip_batchnorm_f32: bad shape");
   if (N == 0)
      return SOFIE_HIP_OK;
   SOFIE_HIP_REQUIRE(Y && X && fused_scale && mean && bias, "sofie_hip_batchnorm_f32: NULL pointer");
   const size_t n = (size_t)N * (size_t)C * (size_t)spatial;
   const bool vec = spatial % 4 == 0 && (((uintptr_t)X | (uintptr_t)Y) & 15) == 0;
   auto go = [&](auto div) {
      typedef decltype(div) DIV;
      if (vec)
         launch_kernel((batchnorm_f32_kernel<f32x4, DIV>), dim3(grid_for((n / 4 + 3) / 4)), dim3(256), 0, ctx->stream, (f32x4 *)Y, (const f32x4 *)X,
                            fused_scale, mean, bias, n / 4, DIV(C), DIV(spatial / 4), relu);
      else
         launch_kernel((batchnorm_f32_kernel<float, DIV>), dim3(grid_for((n + 3) / 4)), dim3(256), 0, ctx->stream, Y, X, fused_scale, mean, bias, n, DIV(C),
                            DIV(spatial), relu);
   };
   if (n < (1ull << 31))
      go(Divisor31(1));
   else
      go(Divisor64(1));
   return launch_status("batchnorm_f32_kernel");
}

int sofie_hip_pool3d_f32(sofie_hip_ctx *ctx, const sofie_pool3d_desc *d, float *Y, const float *X)
{
   SOFIE_HIP_REQUIRE(ctx && d, "sofie_hip_pool3d_f32: NULL argument");
   SOFIE_HIP_REQUIRE(d->planes >= 0, "sofie_hip_pool3d_f32: bad shape");
   SOFIE_HIP_REQUIRE(d->mode == SOFIE_POOL_MAX || d->mode == SOFIE_POOL_AVERAGE, "sofie_hip_pool3d_f32: unknown mode %d", d->mode);
   long long total = d->planes, in_total = d->planes;
   for (int a = 0; a < 3; ++a) {
      SOFIE_HIP_REQUIRE(d->in[a] > 0 && d->out[a] > 0 && d->k[a] > 0, "sofie_hip_pool3d_f32: bad shape");
      SOFIE_HIP_REQUIRE(d->stride[a] > 0, "sofie_hip_pool3d_f32: bad stride");
      SOFIE_HIP_REQUIRE(d->pad_begin[a] >= 0 && d->pad_end[a] >= 0, "sofie_hip_pool3d_f32: negative padding");
      // every window start must lie where the reference's loops put it: the last one begins inside the padded volume
      SOFIE_HIP_REQUIRE((long long)(d->out[a] - 1) * d->stride[a] - d->pad_begin[a] < d->in[a] + d->pad_end[a],
                        "sofie_hip_pool3d_f32: the output extent %d of axis %d does not fit the padded input", d->out[a], a);
      total *= d->out[a];
      in_total *= d->in[a];
      SOFIE_HIP_REQUIRE(total < (1LL << 40) && in_total < (1LL << 40), "sofie_hip_pool3d_f32: tensor too large");
   }
   if (total == 0)
      return SOFIE_HIP_OK;
   SOFIE_HIP_REQUIRE(Y && X, "sofie_hip_pool3d_f32: NULL pointer");
   auto window = [&](auto div) {
      typedef decltype(div) DIV;
      const DIV o0(d->out[0]), o1(d->out[1]), o2(d->out[2]);
      auto go = [&](auto kernel) { launch_kernel(kernel, dim3(grid_for((size_t)total)), dim3(256), 0, ctx->stream, Y, X, *d, (size_t)total, o0, o1, o2); };
      // the flat windows in common use; the first axis has to be one of a single, unpadded slice
      const bool flat = d->in[0] == 1 && d->out[0] == 1 && d->k[0] == 1 && d->pad_begin[0] == 0;
      if (flat && d->k[1] == 3 && d->k[2] == 3)
         go(pool_f32_kernel<DIV, 3, 3>);
      else if (flat && d->k[1] == 2 && d->k[2] == 2)
         go(pool_f32_kernel<DIV, 2, 2>);
      else
         go(pool_f32_kernel<DIV, 0, 0>);
   };
   // windows and strides of the pair kernel; one more column of padding and its pairs would begin before a row.  Fewer outputs than fill the chip take a
   // launch's time either way.
   const bool step2 = d->in[0] == 1 && d->out[0] == 1 && d->k[0] == 1 && d->pad_begin[0] == 0 && d->k[1] == 3 && d->k[2] == 3 && d->stride[1] == 2 &&
                      d->stride[2] == 2 && d->pad_begin[2] <= 1 && d->in[2] >= 2;
   if (step2 && total < (1LL << 31)) {
      const long long rows = (d->out[1] + 1) / 2, pairs = (long long)d->planes * rows * d->out[2];
      launch_kernel((pool_f32_3x3_step2_kernel<Divisor31>), dim3(grid_for((size_t)pairs)), dim3(256), 0, ctx->stream, Y, X, *d, (size_t)pairs, Divisor31(rows),
                    Divisor31(d->out[2]));
   } else if (total < (1LL << 31)) {
      window(Divisor31(1));
   } else {
      window(Divisor64(1));
   }
   return launch_status("pool_f32_kernel");
}

int sofie_hip_pool_f32(sofie_hip_ctx *ctx, const sofie_pool_desc *d, float *Y, const float *X)
{
   SOFIE_HIP_REQUIRE(ctx && d, "sofie_hip_pool_f32: NULL argument");
   SOFIE_HIP_REQUIRE(d->planes >= 0 && d->H > 0 && d->W > 0 && d->OH > 0 && d->OW > 0 && d->kh > 0 && d->kw > 0, "sofie_hip_pool_f32: bad shape");
   SOFIE_HIP_REQUIRE(d->stride_h > 0 && d->stride_w > 0, "sofie_hip_pool_f32: bad stride");
   SOFIE_HIP_REQUIRE(d->pad_h0 >= 0 && d->pad_w0 >= 0 && d->pad_h1 >= 0 && d->pad_w1 >= 0, "sofie_hip_pool_f32: negative padding");
   SOFIE_HIP_REQUIRE(d->mode == SOFIE_POOL_MAX || d->mode == SOFIE_POOL_AVERAGE, "sofie_hip_pool_f32: unknown mode %d", d->mode);
   // every window start must lie where the reference's loops put it: the last one begins inside the padded image
   SOFIE_HIP_REQUIRE((long long)(d->OH - 1) * d->stride_h - d->pad_h0 < d->H + d->pad_h1 &&
                        (long long)(d->OW - 1) * d->stride_w - d->pad_w0 < d->W + d->pad_w1,
                     "sofie_hip_pool_f32: the output shape %dx%d does not fit the padded input", d->OH, d->OW);
   // a volume of depth one
   sofie_pool3d_desc v{};
   v.planes = d->planes;
   v.in[0] = 1, v.in[1] = d->H, v.in[2] = d->W;
   v.out[0] = 1, v.out[1] = d->OH, v.out[2] = d->OW;
   v.k[0] = 1, v.k[1] = d->kh, v.k[2] = d->kw;
   v.pad_begin[0] = 0, v.pad_begin[1] = d->pad_h0, v.pad_begin[2] = d->pad_w0;
   v.pad_end[0] = 0, v.pad_end[1] = d->pad_h1, v.pad_end[2] = d->pad_w1;
   v.stride[0] = 1, v.stride[1] = d->stride_h, v.stride[2] = d->stride_w;
   v.mode = d->mode, v.count_include_pad = d->count_include_pad, v.dynamic_divisor = d->dynamic_divisor;
   return sofie_hip_pool3d_f32(ctx, &v, Y, X);
}

int sofie_hip_global_avg_pool_f32(sofie_hip_ctx *ctx, float *Y, const float *X, int32_t NC, int32_t HW)
{
   SOFIE_HIP_REQUIRE(ctx != nullptr, "sofie_hip_global_avg_pool_f32: ctx is NULL");
   SOFIE_HIP_REQUIRE(NC >= 0 && HW > 0, "sofie_hip_global_avg_pool_f32: bad shape");
   if (NC == 0)
      return SOFIE_HIP_OK;
   SOFIE_HIP_REQUIRE(Y && X, "sofie_hip_global_avg_pool_f32: NULL pointer");
   launch_kernel((gap_kernel<float, float>), dim3((NC + 3) / 4), dim3(256), 0, ctx->stream, Y, X, NC, HW, 1.0f,
                      (int)(HW % 4 == 0 && ((uintptr_t)X & 15) == 0));
   return launch_status("gap_kernel");
}

int sofie_hip_global_avg_pool_i8(sofie_hip_ctx *ctx, float *Y, const int8_t *X, int32_t N, int32_t C, int32_t HW,
                                 int32_t x_layout, float scale)
{
   SOFIE_HIP_REQUIRE(ctx != nullptr, "sofie_hip_global_avg_pool_i8: ctx is NULL");
   SOFIE_HIP_REQUIRE(N >= 0 && C > 0 && HW > 0, "sofie_hip_global_avg_pool_i8: bad shape");
   SOFIE_HIP_REQUIRE(x_layout == SOFIE_LAYOUT_NCHW || x_layout == SOFIE_LAYOUT_NHWC, "sofie_hip_global_avg_pool_i8: unknown layout");
   SOFIE_HIP_REQUIRE((long long)N * C < (1LL << 31), "sofie_hip_global_avg_pool_i8: too many planes");
   if (N == 0)
      return SOFIE_HIP_OK;
   SOFIE_HIP_REQUIRE(Y && X, "sofie_hip_global_avg_pool_i8: NULL pointer");
   if (x_layout == SOFIE_LAYOUT_NHWC) {
      if (C % 16 == 0 && (((uintptr_t)X & 15) == 0) && C / 16 <= 65535) {
         // a few images: fewer channels per workgroup, until there is one for each CU
         int chunks_log2 = 4;
         auto blocks = [&] { return (C + (16 << chunks_log2) - 1) / (16 << chunks_log2); };
         while (chunks_log2 > 0 && (long long)N * blocks() < 256)
            --chunks_log2;
         launch_kernel(gap_i8_nhwc_vec_kernel, dim3((unsigned)N, (unsigned)blocks()), dim3(GAP_THREADS), 0, ctx->stream, Y, X, C, HW, scale, chunks_log2);
         return launch_status("gap_i8_nhwc_vec_kernel");
      }
      launch_kernel(gap_i8_nhwc_kernel, dim3((unsigned)N), dim3(256), 0, ctx->stream, Y, X, C, HW, scale);
      return launch_status("gap_i8_nhwc_kernel");
   }
   const int NC = N * C;
   launch_kernel((gap_kernel<int8_t, int>), dim3((NC + 3) / 4), dim3(256), 0, ctx->stream, Y, X, NC, HW, scale, 0);
   return launch_status("gap_kernel");
}

int sofie_hip_transpose_f32(sofie_hip_ctx *ctx, float *Y, const float *X, int32_t rank, const int64_t *shape, const int32_t *perm)
{
   SOFIE_HIP_REQUIRE(ctx && shape && perm, "sofie_hip_transpose_f32: NULL argument");
   SOFIE_HIP_REQUIRE(rank >= 1 && rank <= 6, "sofie_hip_transpose_f32: rank %d not in [1,6]", rank);
   long long in_stride[6];
   size_t n = 1;
   unsigned seen = 0;
   for (int d = rank - 1; d >= 0; --d) {
      SOFIE_HIP_REQUIRE(shape[d] >= 0 && shape[d] < (1LL << 40), "sofie_hip_transpose_f32: bad dimension");
      in_stride[d] = (long long)n;
      n *= (size_t)shape[d];
      SOFIE_HIP_REQUIRE(n < (1ULL << 40), "sofie_hip_transpose_f32: tensor too large");
   }
   TransposeShape sh;
   sh.rank = rank;
   for (int k = 0; k < rank; ++k) {
      SOFIE_HIP_REQUIRE(perm[k] >= 0 && perm[k] < rank && !(seen & (1u << perm[k])), "sofie_hip_transpose_f32: perm is not a permutation of 0..%d", rank - 1);
      seen |= 1u << perm[k];
      sh.y[k] = shape[perm[k]];
      sh.sx[k] = in_stride[perm[k]];
   }
   if (n == 0)
      return SOFIE_HIP_OK;
   SOFIE_HIP_REQUIRE(Y && X, "sofie_hip_transpose_f32: NULL pointer");
   return launch_transpose(ctx, Y, X, n, sh);
}

int sofie_hip_strided_gather_f32(sofie_hip_ctx *ctx, float *Y, const float *X, int32_t rank, const int64_t *out_shape, const int64_t *in_strides,
                                 int64_t in_offset, int64_t in_elements)
{
   SOFIE_HIP_REQUIRE(ctx && out_shape && in_strides, "sofie_hip_strided_gather_f32: NULL argument");
   SOFIE_HIP_REQUIRE(rank >= 1 && rank <= 6, "sofie_hip_strided_gather_f32: rank %d not in [1,6]", rank);
   SOFIE_HIP_REQUIRE(in_elements >= 0 && in_elements < (1LL << 40) && in_offset >= 0, "sofie_hip_strided_gather_f32: bad input size or offset");
   TransposeShape sh;
   sh.rank = rank;
   size_t n = 1;
   long long lo = in_offset, hi = in_offset; // the smallest and the largest input index the output reads
   for (int k = 0; k < rank; ++k) {
      SOFIE_HIP_REQUIRE(out_shape[k] >= 0 && out_shape[k] < (1LL << 40), "sofie_hip_strided_gather_f32: bad dimension");
      SOFIE_HIP_REQUIRE(in_strides[k] > -(1LL << 40) && in_strides[k] < (1LL << 40), "sofie_hip_strided_gather_f32: bad stride");
      n *= (size_t)out_shape[k];
      SOFIE_HIP_REQUIRE(n < (1ULL << 40), "sofie_hip_strided_gather_f32: tensor too large");
      sh.y[k] = out_shape[k];
      sh.sx[k] = in_strides[k];
   }
   if (n == 0)
      return SOFIE_HIP_OK;
   for (int k = 0; k < rank; ++k) {
      const double span = (double)(out_shape[k] - 1) * (double)in_strides[k];
      SOFIE_HIP_REQUIRE(span > -1.0e15 && span < 1.0e15, "sofie_hip_strided_gather_f32: axis %d reaches outside the input", k);
      (in_strides[k] < 0 ? lo : hi) += (long long)(out_shape[k] - 1) * in_strides[k];
   }
   SOFIE_HIP_REQUIRE(lo >= 0 && hi < in_elements, "sofie_hip_strided_gather_f32: reads elements %lld..%lld of an input of %lld", lo, hi, (long long)in_elements);
   SOFIE_HIP_REQUIRE(Y && X, "sofie_hip_strided_gather_f32: NULL pointer");
   return launch_transpose(ctx, Y, X + in_offset, n, sh);
}

int sofie_hip_copy_rows(sofie_hip_ctx *ctx, void *dst, size_t dst_pitch_bytes, const void *src, size_t src_pitch_bytes, size_t rows, size_t row_bytes)
{
   SOFIE_HIP_REQUIRE(ctx != nullptr, "sofie_hip_copy_rows: ctx is NULL");
   SOFIE_HIP_REQUIRE(row_bytes % 4 == 0 && dst_pitch_bytes % 4 == 0 && src_pitch_bytes % 4 == 0, "sofie_hip_copy_rows: sizes must be multiples of 4 bytes");
   SOFIE_HIP_REQUIRE(dst_pitch_bytes >= row_bytes && src_pitch_bytes >= row_bytes, "sofie_hip_copy_rows: a pitch is smaller than the row");
   SOFIE_HIP_REQUIRE(rows < (1ULL << 40) && row_bytes < (1ULL << 40) && (double)rows * (double)row_bytes < 1.0e13, "sofie_hip_copy_rows: too large");
   if (rows == 0 || row_bytes == 0)
      return SOFIE_HIP_OK;
   SOFIE_HIP_REQUIRE(dst && src && (((uintptr_t)dst | (uintptr_t)src) & 3) == 0, "sofie_hip_copy_rows: NULL or misaligned pointer");
   launch_kernel(copy_rows_kernel, dim3(grid_for(rows * (row_bytes / 4))), dim3(256), 0, ctx->stream, (uint32_t *)dst, dst_pitch_bytes / 4,
                      (const uint32_t *)src, src_pitch_bytes / 4, rows, row_bytes / 4);
   return launch_status("copy_rows_kernel");
}

int sofie_hip_softmax_f32(sofie_hip_ctx *ctx, float *Y, const float *X, int64_t outer, int32_t axis_len, int64_t inner, int32_t log_softmax)
{
   SOFIE_HIP_REQUIRE(ctx != nullptr, "sofie_hip_softmax_f32: ctx is NULL");
   SOFIE_HIP_REQUIRE(outer >= 0 && axis_len > 0 && inner > 0, "sofie_hip_softmax_f32: bad shape");
   SOFIE_HIP_REQUIRE(outer < (1LL << 40) && inner < (1LL << 40) && (double)outer * axis_len * (double)inner < 1.0e12, "sofie_hip_softmax_f32: tensor too large");
   const long long lines = (long long)outer * inner;
   if (lines == 0)
      return SOFIE_HIP_OK;
   SOFIE_HIP_REQUIRE(Y && X, "sofie_hip_softmax_f32: NULL pointer");
   if (inner == 1 && with_line_registers(lines, axis_len, (((uintptr_t)X | (uintptr_t)Y) & 15) == 0, [&](auto vec, auto nv, int G, unsigned blocks) {
          launch_kernel((softmax_lines_f32_kernel<decltype(vec)::value, decltype(nv)::value>), dim3(blocks), dim3(256), 0, ctx->stream, Y, X, lines, axis_len, G,
                             log_softmax);
       }))
      return launch_status("softmax_lines_f32_kernel");
   const long long blocks = (lines + 3) / 4;
   launch_kernel(softmax_f32_kernel, dim3((unsigned)(blocks < 256 * 64 ? blocks : 256 * 64)), dim3(256), 0, ctx->stream, Y, X, lines, axis_len,
                      (long long)inner, log_softmax);
   return launch_status("softmax_f32_kernel");
}

int sofie_hip_reduce_f32(sofie_hip_ctx *ctx, float *Y, const float *X, int64_t outer, int32_t A, int64_t inner, int32_t op)
{
   SOFIE_HIP_REQUIRE(ctx != nullptr, "sofie_hip_reduce_f32: ctx is NULL");
   SOFIE_HIP_REQUIRE(op >= SOFIE_REDUCE_SUM && op <= SOFIE_REDUCE_MIN, "sofie_hip_reduce_f32: unknown operator %d", op);
   SOFIE_HIP_REQUIRE(outer >= 0 && A > 0 && inner > 0 && outer < (1LL << 40) && inner < (1LL << 40) && (double)outer * A * (double)inner < 1.0e12,
                     "sofie_hip_reduce_f32: bad shape");
   const long long outputs = (long long)outer * inner;
   if (outputs == 0)
      return SOFIE_HIP_OK;
   SOFIE_HIP_REQUIRE(Y && X, "sofie_hip_reduce_f32: NULL pointer");
   if (inner == 1 && A >= 64 && outputs < 16384) {
      launch_kernel(reduce_lines_f32_kernel, dim3((unsigned)((outputs + 3) / 4)), dim3(256), 0, ctx->stream, Y, X, outputs, A, op);
      return launch_status("reduce_lines_f32_kernel");
   }
   launch_kernel(reduce_f32_kernel, dim3(grid_for((size_t)outputs)), dim3(256), 0, ctx->stream, Y, X, (size_t)outputs, A, (long long)inner, op);
   return launch_status("reduce_f32_kernel");
}

int sofie_hip_layernorm_f32(sofie_hip_ctx *ctx, float *Y, const float *X, const float *scale, const float *bias, int64_t rows, int32_t L, float epsilon,
                            float *mean_out, float *inv_std_out)
{
   SOFIE_HIP_REQUIRE(ctx != nullptr, "sofie_hip_layernorm_f32: ctx is NULL");
   SOFIE_HIP_REQUIRE(rows >= 0 && L > 0 && rows < (1LL << 40) && (double)rows * L < 1.0e12, "sofie_hip_layernorm_f32: bad shape");
   SOFIE_HIP_REQUIRE(epsilon >= 0.0f, "sofie_hip_layernorm_f32: epsilon is negative");
   if (rows == 0)
      return SOFIE_HIP_OK;
   SOFIE_HIP_REQUIRE(Y && X && scale, "sofie_hip_layernorm_f32: NULL pointer");
   const uintptr_t addresses = (uintptr_t)X | (uintptr_t)Y | (uintptr_t)scale | (uintptr_t)bias;
   if (with_line_registers(rows, L, (addresses & 15) == 0, [&](auto vec, auto nv, int G, unsigned blocks) {
          launch_kernel((layernorm_lines_f32_kernel<decltype(vec)::value, decltype(nv)::value>), dim3(blocks), dim3(256), 0, ctx->stream, Y, X, scale, bias,
                             (long long)rows, L, G, epsilon, mean_out, inv_std_out);
       }))
      return launch_status("layernorm_lines_f32_kernel");
   const long long blocks = (rows + 3) / 4;
   launch_kernel(layernorm_f32_kernel, dim3((unsigned)(blocks < 256 * 64 ? blocks : 256 * 64)), dim3(256), 0, ctx->stream, Y, X, scale, bias, (long long)rows, L,
                      epsilon, mean_out, inv_std_out);
   return launch_status("layernorm_f32_kernel");
}

int sofie_hip_plane_sums_to_average(sofie_hip_ctx *ctx, float *Y, const int32_t *sums, int32_t NC, int32_t HW, float scale)
{
   SOFIE_HIP_REQUIRE(ctx != nullptr, "sofie_hip_plane_sums_to_average: ctx is NULL");
   SOFIE_HIP_REQUIRE(NC >= 0 && HW > 0, "sofie_hip_plane_sums_to_average: bad shape");
   if (NC == 0)
      return SOFIE_HIP_OK;
   SOFIE_HIP_REQUIRE(Y && sums, "sofie_hip_plane_sums_to_average: NULL pointer");
   launch_kernel(plane_sums_to_average_kernel, dim3((NC + 255) / 256), dim3(256), 0, ctx->stream, Y, sums, NC, HW, scale);
   return launch_status("plane_sums_to_average_kernel");
}

int sofie_hip_plane_sums_take_average(sofie_hip_ctx *ctx, float *Y, int32_t *sums, int32_t NC, int32_t HW, float scale)
{
   SOFIE_HIP_REQUIRE(ctx != nullptr, "sofie_hip_plane_sums_take_average: ctx is NULL");
   SOFIE_HIP_REQUIRE(NC >= 0 && HW > 0, "sofie_hip_plane_sums_take_average: bad shape");
   if (NC == 0)
      return SOFIE_HIP_OK;
   SOFIE_HIP_REQUIRE(Y && sums, "sofie_hip_plane_sums_take_average: NULL pointer");
   launch_kernel(plane_sums_take_average_kernel, dim3((NC + 255) / 256), dim3(256), 0, ctx->stream, Y, sums, NC, HW, scale);
   return launch_status("plane_sums_take_average_kernel");
}

} // extern "C"
