// fp32 products on the matrix cores (v_mfma_f32_32x32x2_f32, v_mfma_f32_16x16x4_f32: full fp32 multiply-adds at twice the rate of the unpacked vector
// instructions), for Gemm / MatMul and for convolutions as implicit GEMM.  Three kernels:
//   f32_tile_kernel          a workgroup of four or eight waves owns a BM x BN tile; slabs of k go straight from memory into a ring in LDS
//   f32_direct_kernel        small products: a workgroup owns one small tile and its waves split the reduction; every fragment is
//                            loaded from memory into the registers the MFMA reads, with many loads in flight and no LDS in the loop
//   f32_direct_ring_kernel   the same where both operands have 16-byte rows along k: whole lines through a ring in LDS per wave
//
// Both feed an MFMA the n side as first operand and the m side as second, so a lane ends up with 4 consecutive columns n of one
// row m.  Four MFMAs take four consecutive k from every lane: which k a lane supplies to which MFMA only has to agree between the
// operands, and this order lets an operand that is contiguous in k be read as one 16-byte word per lane.
#pragma once
#include "mfma8_common.hpp"
#include "mfma8_direct.hpp"

namespace sofie_hip {

typedef float v4f __attribute__((ext_vector_type(4)));

// What loads of positions outside an operand read.
static __device__ __attribute__((aligned(256))) float f32_zero_page[64] = {};

__device__ __forceinline__ v4f mfma_f32_step(const v4f &n_side, const v4f &m_side, v4f acc)
{
#pragma unroll
   for (int j = 0; j < 4; ++j)
      acc = __builtin_amdgcn_mfma_f32_16x16x4f32(n_side[j], m_side[j], acc, 0, 0, 0);
   return acc;
}

// a value that is the same in all lanes, in scalar registers
__device__ __forceinline__ long long uniform(long long v)
{
   const unsigned lo = __builtin_amdgcn_readfirstlane((int)v), hi = __builtin_amdgcn_readfirstlane((int)(v >> 32));
   return (long long)(((unsigned long long)hi << 32) | lo);
}

// Loads into LDS go through a buffer descriptor: its base is scalar and may move, so is a second offset; a lane adds an offset of 31
// bits, and F32_OUTSIDE, which lies behind the buffer's end, reads as zero.  Vector instructions take their turn on the multipliers of the fp32
// matrix cores (two waves per SIMD, eight additions per MFMA of 64 cycles: 3.0 cycles each, 64-bit ones 5.2; one wave alone: 6), so
// what a loop spends on addresses is lost to it: two 64-bit additions and an address in LDS per load took a tenth of it.
constexpr long long F32_BUFFER_BYTES = 0x7fffff00;
constexpr int F32_OUTSIDE = -1;
template <int FLOATS>
__device__ __forceinline__ void f32_buffer_load(lds_void_t *to, const void *base, int offset, int scalar_offset = 0)
{
   const __amdgpu_buffer_rsrc_t buffer = __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(base), 0, (int)F32_BUFFER_BYTES, 0x00020000);
   if constexpr (FLOATS == 4)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(buffer, to, 16, offset, scalar_offset, 0, 0);
   else
      __builtin_amdgcn_raw_ptr_buffer_load_lds(buffer, to, 4, offset, scalar_offset, 0, 0);
}

// ---- operands ---------------------------------------------------------------------------------------------------------------
// An operand is a matrix of `rows` (m or n) by K.  KC: contiguous in k (a row's k neighbours lie side by side); otherwise
// contiguous along the rows.  VEC: floats per load; 4 needs 16-byte aligned pieces (the host checks that the address, the
// pitch and the extent along the contiguous direction are multiples of 16 bytes).
template <bool KC_, int VEC_>
struct F32Matrix {
   static constexpr int kLeastRows = 16; // of a tile of the tile kernel
   static constexpr bool KC = KC_;
   static constexpr int VEC = VEC_;
   const float *p;
   long long ld;
   int rows, K;
   __device__ __forceinline__ void shift(long long elements) { p += elements; }
   __device__ __forceinline__ void select_group(int) {}
   // whether the slabs of any tile lie within a buffer of their own (rows of up to four million floats)
   bool in_buffers() const { return (KC ? (rows < 128 ? rows : 128) : 32) * ld * 4 + 1024 <= F32_BUFFER_BYTES; }

   // A slab is loaded through a buffer whose base, in scalar registers, walks along k; what a lane keeps per load instruction of a
   // slab is its distance from there (32 bits: the host checks that they do).
   template <int LD>
   struct walk_state {
      const char *base; // first row of the tile, first k of the slab to be asked for next
      long long step;
      unsigned k0; // up to a slab past K
   };
   template <int LD, class F>
   __device__ __forceinline__ void walk_start(walk_state<LD> &w, int r0, int, int slab, F &&) const
   {
      w.base = (const char *)uniform((long long)(KC ? p + (long long)r0 * ld : p + r0));
      w.step = (KC ? (long long)slab : slab * ld) * 4;
      w.k0 = 0;
   }
   template <int LD>
   __device__ __forceinline__ void walk_on(walk_state<LD> &w, int slab) const
   {
      w.base += w.step;
      w.k0 += slab;
   }
   template <int LD>
   struct lane_state {
      int at[LD];
   };
   template <int LD>
   __device__ __forceinline__ void init(lane_state<LD> &st, int i, int r0, int row, int kk) const
   {
      // rows past the edge re-read the last piece (their results are not stored)
      const int last = (KC || VEC == 1 ? rows - 1 : rows - VEC) - r0, r = row < last ? row : last;
      st.at[i] = (int)(KC ? (long long)r * ld + kk : (long long)kk * ld + r) * 4;
   }
   // load i of the slab (kk: the lane's k within the slab; WHOLE: no k of the slab lies past K)
   template <bool WHOLE, int LD>
   __device__ __forceinline__ void load(lds_void_t *to, const lane_state<LD> &st, const walk_state<LD> &w, int i, int kk) const
   {
      f32_buffer_load<VEC>(to, w.base, WHOLE || w.k0 + (unsigned)kk < (unsigned)K ? st.at[i] : F32_OUTSIDE);
   }

   // direct fetch of row `row`, k..k+3
   struct row_state {
      const float *at;
   };
   __device__ __forceinline__ row_state row_of(int row) const
   {
      const int r = row < rows ? row : rows - 1;
      return row_state{KC ? p + (long long)r * ld : p + r};
   }
   // WHOLE: k..k+3 lie before K.  Otherwise `left` of them do, none if it is negative.  Floats past K are read as the first k of the row, and dropped: no branch stands between
   // the loads.  (For the one load of four that start on 16 bytes a branch is the shorter way: 2.46 us with that, 2.34 with the branch for 16 x 16 x 4 .. 8.)
   template <bool WHOLE>
   __device__ __forceinline__ v4f fetch(const row_state &st, int k, int left) const
   {
      typedef float v4f_by_floats __attribute__((ext_vector_type(4), aligned(4)));
      if constexpr (KC && (VEC == 4 || WHOLE)) {
         v4f v = {0.f, 0.f, 0.f, 0.f};
         if (WHOLE || left > 0)
            v = *(const v4f_by_floats *)(st.at + k);
         return v;
      } else {
         v4f v;
         const float *at = st.at + (KC ? (long long)k : (long long)k * ld);
#pragma unroll
         for (int j = 0; j < 4; ++j) {
            const float *from = at + (KC ? (long long)j : j * ld);
            v[j] = *(WHOLE || j < left ? from : st.at);
         }
#pragma unroll
         for (int j = 0; j < 4; ++j)
            v[j] = WHOLE || j < left ? v[j] : 0.f;
         return v;
      }
   }
};

// The column matrix of a convolution, gathered from the NCHW input as it is asked for: row m = (image, output position), column
// k = (channel, kernel position), zero outside the image -- the index arithmetic of the reference's Im2col / Im2col_3d
// (core/src/utils/SOFIE_common_helpers.cxx:47-139).  Neighbouring rows are neighbouring output positions of one image row, so a
// load instruction (64 rows, one k) reads (almost) consecutive floats; what depends on k alone is scalar arithmetic.
struct F32ConvShape {
   int C, D, H, W, kd, kh, kw, OD, OH, OW; // input channels (all groups); a 2-D convolution has D = kd = OD = 1
   int pad_d, pad_h, pad_w, stride_d, stride_h, stride_w, dil_d, dil_h, dil_w;
   int Cg;                                 // channels per group
   int positions;                          // kd * kh * kw
   unsigned long long ow_mul, oh_mul, od_mul; // ceil(2^64 / extent), 0 for an extent of 1: m / extent == umul64hi(m, mul) for 32-bit m
   Divisor31 by_kw{1}, by_kh{1}, by_kd{1}, by_positions{1};
};
// MASKED (at most 31 kernel positions, extents that fit a buffer): a lane keeps its row's place and one bit per kernel position that
// lies outside the image; the walk along k, from slab to slab, is scalar.  Three vector instructions per 64 elements.
template <bool MASKED>
struct F32ConvRows {
   static constexpr int kLeastRows = 64; // a load instruction covers one k: what depends on k is scalar
   static constexpr bool KC = false;
   static constexpr int VEC = 1;
   const float *X;
   F32ConvShape s;
   int rows, K;
   long long image, channel; // elements per image and per channel
   bool in_buffers() const { return true; }
   __device__ __forceinline__ void shift(long long) {}
   __device__ __forceinline__ void select_group(int g) { X += (long long)g * s.Cg * channel; }

   struct position {
      int image, d, h, w; // of an output
   };
   __device__ __forceinline__ position position_of(int row) const
   {
      auto quotient = [](int n, unsigned long long mul) { return mul ? (int)__umul64hi((unsigned long long)(unsigned)n, mul) : n; };
      const int m = row < rows ? row : rows - 1;
      const int t = quotient(m, s.ow_mul), u = quotient(t, s.oh_mul), image = quotient(u, s.od_mul);
      return position{image, u - image * s.OD, t - u * s.OH, m - t * s.OW};
   }
   struct row_state {
      const float *at; // element of channel 0 at (id0, ih0, iw0): dereferenced only inside the image
      int id0, ih0, iw0;
   };
   __device__ __forceinline__ row_state row_of(int row) const
   {
      const position o = position_of(row);
      row_state r;
      r.id0 = o.d * s.stride_d - s.pad_d;
      r.ih0 = o.h * s.stride_h - s.pad_h;
      r.iw0 = o.w * s.stride_w - s.pad_w;
      r.at = X + (long long)o.image * image + ((long long)r.id0 * s.H + r.ih0) * s.W + r.iw0;
      return r;
   }
   static __device__ __forceinline__ int divide(unsigned k, const Divisor31 &by) { return (int)by.over(k); }
   // address of column k of a row, or of a zero
   __device__ __forceinline__ const float *element(const row_state &r, unsigned k) const
   {
      const int t = divide(k, s.by_kw), kx = (int)k - t * s.kw;
      const int u = divide(t, s.by_kh), ky = t - u * s.kh;
      const int ci = divide(u, s.by_kd), kz = u - ci * s.kd;
      const int dz = kz * s.dil_d, dy = ky * s.dil_h, dx = kx * s.dil_w;
      const bool inside = k < (unsigned)K && (unsigned)(r.id0 + dz) < (unsigned)s.D && (unsigned)(r.ih0 + dy) < (unsigned)s.H && (unsigned)(r.iw0 + dx) < (unsigned)s.W;
      const float *p = r.at + ((long long)ci * channel + ((long long)dz * s.H + dy) * s.W + dx);
      return inside ? p : f32_zero_page;
   }
   // a lane keeps the same row through all load instructions of a slab (tiles of 64 rows or more, an even number of waves)
   template <int LD>
   struct lane_state {
      row_state r;
      int at;           // MASKED: where the window of this row begins in the padded image, from the tile's base, in bytes
      unsigned outside; // MASKED: bit t: kernel position t of this row lies outside the image; bit 31 is set
   };
   template <int LD>
   __device__ __forceinline__ void init(lane_state<LD> &st, int i, int r0, int row, int) const
   {
      if (i != 0)
         return;
      st.r = row_of(r0 + row);
      if constexpr (MASKED) {
         unsigned columns = 0, lines = 0, inside = 0;
         for (int kx = 0; kx < s.kw; ++kx)
            columns |= ((unsigned)(st.r.iw0 + kx * s.dil_w) < (unsigned)s.W ? 1u : 0u) << kx;
         for (int ky = 0; ky < s.kh; ++ky)
            lines |= ((unsigned)(st.r.ih0 + ky * s.dil_h) < (unsigned)s.H ? columns : 0u) << (ky * s.kw);
         for (int kz = 0; kz < s.kd; ++kz)
            inside |= ((unsigned)(st.r.id0 + kz * s.dil_d) < (unsigned)s.D ? lines : 0u) << (kz * s.kh * s.kw);
         st.outside = ~inside;
         st.at = (int)((const char *)st.r.at - base_of(r0));
      }
   }
   // the padded image of the first row of a tile: no window of the tile begins before it
   __device__ __forceinline__ const char *base_of(int r0) const
   {
      const long long pad = ((long long)s.pad_d * s.H + s.pad_h) * s.W + s.pad_w;
      return (const char *)(X + (long long)position_of(r0).image * image - pad);
   }
   // For MASKED, scalars: of load i of the slab to be asked for its first k in that slab, its kernel position and the offset of its channel.
   template <int LD>
   struct walk_state {
      const char *base;
      unsigned k0;
      int first[LD], position[LD], channel[LD];
      int step_channels, step_rest; // a slab's worth of k in channels (as an offset) and kernel positions
      int table;                    // lane t: offset of kernel position t
   };
   template <int LD, class F>
   __device__ __forceinline__ void walk_start(walk_state<LD> &w, int r0, int lane, int slab, F &&first_k) const
   {
      w.k0 = 0;
      if constexpr (MASKED) {
         w.base = (const char *)uniform((long long)base_of(r0));
         const int t = divide(lane, s.by_kw), kx = lane - t * s.kw, kz = divide(t, s.by_kh), ky = t - kz * s.kh;
         w.table = ((kz * s.dil_d * s.H + ky * s.dil_h) * s.W + kx * s.dil_w) * 4; // lanes past the last position are not asked
         const int channels = divide(slab, s.by_positions);
         w.step_channels = channels * (int)channel * 4;
         w.step_rest = slab - channels * s.positions;
#pragma unroll
         for (int i = 0; i < LD; ++i) {
            w.first[i] = first_k(i);
            const int ci = divide(w.first[i], s.by_positions);
            w.position[i] = w.first[i] - ci * s.positions;
            w.channel[i] = ci * (int)channel * 4;
         }
      }
   }
   template <int LD>
   __device__ __forceinline__ void walk_on(walk_state<LD> &w, int slab) const // by the slab of walk_start
   {
      w.k0 += slab;
      if constexpr (MASKED) {
#pragma unroll
         for (int i = 0; i < LD; ++i) {
            const int position = w.position[i] + w.step_rest;
            const bool over = position >= s.positions;
            w.position[i] = position - (over ? s.positions : 0);
            w.channel[i] += w.step_channels + (over ? (int)channel * 4 : 0);
         }
      }
   }
   template <bool WHOLE, int LD>
   __device__ __forceinline__ void load(lds_void_t *to, const lane_state<LD> &st, const walk_state<LD> &w, int i, int kk) const
   {
      if constexpr (MASKED) {
         const bool any = WHOLE || w.k0 + (unsigned)w.first[i] < (unsigned)K;
         const int position = any ? w.position[i] : 31;
         const int offset = any ? w.channel[i] + __builtin_amdgcn_readlane(w.table, w.position[i]) : 0;
         const int outside = __builtin_amdgcn_sbfe(st.outside, position, 1); // all ones, or none
         f32_buffer_load<1>(to, w.base, st.at | outside, offset);
      } else {
         const float *at = element(st.r, w.k0 + (unsigned)__builtin_amdgcn_readfirstlane(kk));
         __builtin_amdgcn_global_load_lds((global_void_t *)at, to, 4, 0, 0);
      }
   }
   template <bool>
   __device__ __forceinline__ v4f fetch(const row_state &st, int k, int) const
   {
      v4f v;
#pragma unroll
      for (int j = 0; j < 4; ++j)
         v[j] = *element(st, (unsigned)k + j);
      return v;
   }
};

// ---- stores -----------------------------------------------------------------------------------------------------------------
struct F32Epilogue {
   float alpha, beta;
   const float *C;
   int bias_mode;
   long long ldc;
   PostChain chain; // the activation, then the caller's chain of one-to-one operators
   const float *R;  // tensor of Y's shape added before the activation, or nullptr
   long long ldr;
};

// one activation and no further link: the cases worth a straight path (a chain of count 0 is a chain of "none")
__device__ __forceinline__ float f32_activate(float v, const PostChain &chain)
{
   if (chain.count == 0)
      return v;
   if (chain.count == 1 && chain.op0 == SOFIE_ACT_RELU)
      return v > 0.0f ? v : 0.0f;
   return apply_chain(v, chain);
}

// f32_activate of C values, the choice made once: with a choice per value (of the activation, of the bias, of the residual) the store of a 64 x 64 tile took 1 us
// longer.  With the bias asked for before the products, us before -> after: 2048 x 1536 x 384 with no activation 28.9 -> 27.3, relu 28.3 -> 26.7, gelu 30.2 -> 27.4,
// sigmoid 29.5 -> 25.9; 2000 x 512 x 1024 19.6 -> 18.8, 19.9 -> 19.0, 21.5 -> 19.8, 21.4 -> 19.6; 300 x 1000 x 500 7.9 -> 7.7 .. 9.0 -> 8.3.
template <int C, class V>
__device__ __forceinline__ void f32_activate_all(V &v, const PostChain &chain)
{
   auto each = [&](auto act) {
#pragma unroll
      for (int i = 0; i < C; ++i)
         v[i] = apply_activation(v[i], decltype(act)::value, chain.a0);
   };
   if (chain.count == 0)
      return;
   if (chain.count == 1) {
      switch (chain.op0) {
      case SOFIE_ACT_RELU: return each(std::integral_constant<int, SOFIE_ACT_RELU>{});
      case SOFIE_ACT_LEAKYRELU: return each(std::integral_constant<int, SOFIE_ACT_LEAKYRELU>{});
      case SOFIE_ACT_SIGMOID: return each(std::integral_constant<int, SOFIE_ACT_SIGMOID>{});
      case SOFIE_ACT_TANH: return each(std::integral_constant<int, SOFIE_ACT_TANH>{});
      case SOFIE_ACT_GELU: return each(std::integral_constant<int, SOFIE_ACT_GELU>{});
      default: break;
      }
   }
#pragma unroll
   for (int i = 0; i < C; ++i)
      v[i] = apply_chain(v[i], chain);
}

// everything before the activation
__device__ __forceinline__ float f32_linear(const F32Epilogue &ep, float acc, int m, int n)
{
   float v = ep.alpha * acc;
   switch (ep.bias_mode) {
   case SOFIE_BIAS_ROW: v += ep.C[n]; break;
   case SOFIE_BIAS_COL: v += ep.C[m]; break;
   case SOFIE_BIAS_SCALAR: v += ep.C[0]; break;
   case SOFIE_BIAS_FULL: v += ep.beta * ep.C[m * ep.ldc + n]; break;
   default: break;
   }
   if (ep.R)
      v += ep.R[m * ep.ldr + n];
   return v;
}
__device__ __forceinline__ float f32_epilogue(const F32Epilogue &ep, float acc, int m, int n)
{
   return f32_activate(f32_linear(ep, acc, m, n), ep.chain);
}
// The same in two parts: what is added to the element (m, n), asked for before the products it is there when they are done, and the rest.
struct F32Added {
   float bias, residual;
};
__device__ __forceinline__ F32Added f32_look_up(const F32Epilogue &ep, int m, int n)
{
   F32Added a = {0.0f, 0.0f};
   switch (ep.bias_mode) {
   case SOFIE_BIAS_ROW: a.bias = ep.C[n]; break;
   case SOFIE_BIAS_COL: a.bias = ep.C[m]; break;
   case SOFIE_BIAS_SCALAR: a.bias = ep.C[0]; break;
   case SOFIE_BIAS_FULL: a.bias = ep.C[m * ep.ldc + n]; break;
   default: break;
   }
   if (ep.R)
      a.residual = ep.R[m * ep.ldr + n];
   return a;
}
__device__ __forceinline__ float f32_finish(const F32Epilogue &ep, float acc, const F32Added &a)
{
   float v = ep.alpha * acc;
   if (ep.bias_mode == SOFIE_BIAS_FULL)
      v += ep.beta * a.bias;
   else if (ep.bias_mode >= SOFIE_BIAS_ROW && ep.bias_mode <= SOFIE_BIAS_SCALAR)
      v += a.bias;
   if (ep.R)
      v += a.residual;
   return f32_activate(v, ep.chain);
}

// Row-major results of a product.
struct F32RowStore {
   static constexpr bool kAlongRows = false; // neighbouring lanes store neighbouring columns
   float *Y;
   long long ldy;
   F32Epilogue ep;
   int vec; // rows may be written 16 bytes at a time
   long long strideC, strideY;
   __device__ __forceinline__ void select_batch(int b)
   {
      Y += b * strideY;
      if (ep.C)
         ep.C += b * strideC;
      if (ep.R)
         ep.R += b * strideY;
   }
   typedef F32Added added;
   __device__ __forceinline__ added look_up(int m, int n) const { return f32_look_up(ep, m, n); }
   __device__ __forceinline__ void put(float acc, int m, int n, const added &a) const { Y[m * ldy + n] = f32_finish(ep, acc, a); }
   // the bias of columns n..n+3, where each has its own: asked for before the products it is there when they are done
   __device__ __forceinline__ v4f ahead(int n, int N) const
   {
      v4f c = {0.0f, 0.0f, 0.0f, 0.0f};
      if (ep.bias_mode == SOFIE_BIAS_ROW && n + 4 <= N) {
#pragma unroll
         for (int e = 0; e < 4; ++e)
            c[e] = ep.C[n + e];
      }
      return c;
   }
   // columns n..n+3 of row m (those before N); bias: what ahead() gave for them
   __device__ __forceinline__ void put4(v4f a, int m, int n, int N, v4f bias) const
   {
      float *y = Y + m * ldy + n;
      if (n + 4 <= N) { // f32_epilogue of four at a time: each choice once
         v4f v;
#pragma unroll
         for (int e = 0; e < 4; ++e)
            v[e] = ep.alpha * a[e];
         auto add = [&](const float *from, int step) {
#pragma unroll
            for (int e = 0; e < 4; ++e)
               v[e] += from[e * step];
         };
         switch (ep.bias_mode) {
         case SOFIE_BIAS_ROW: v += bias; break;
         case SOFIE_BIAS_COL: add(ep.C + m, 0); break;
         case SOFIE_BIAS_SCALAR: add(ep.C, 0); break;
         case SOFIE_BIAS_FULL: {
            const float *c = ep.C + m * ep.ldc + n;
#pragma unroll
            for (int e = 0; e < 4; ++e)
               v[e] += ep.beta * c[e];
            break;
         }
         default: break;
         }
         if (ep.R)
            add(ep.R + m * ep.ldr + n, 1);
         f32_activate_all<4>(v, ep.chain);
         if (vec) {
            *(v4f *)y = v;
         } else {
#pragma unroll
            for (int e = 0; e < 4; ++e)
               y[e] = v[e];
         }
      } else {
#pragma unroll
         for (int e = 0; e < 4; ++e)
            if (n + e < N)
               y[e] = f32_epilogue(ep, a[e], m, n + e);
      }
   }
};

// NCHW results of a convolution: row m = (image, position), column n = output channel of the group.
struct F32ConvStore {
   static constexpr bool kAlongRows = true; // neighbouring lanes store neighbouring positions of one channel
   float *Y;
   const float *bias;
   const float *R; // tensor of Y's shape added before the activation, or nullptr
   PostChain chain;
   int Cout, Cout_g, positions, first;
   __device__ __forceinline__ void select_batch(int g) { first = g * Cout_g; }
   struct row_state {
      size_t at;
   };
   __device__ __forceinline__ row_state row_of(int m) const
   {
      const int img = m / positions;
      return row_state{(size_t)img * Cout * positions + (m - img * positions)};
   }
   // C columns of one row; those from N on are left out
   template <int C>
   __device__ __forceinline__ void put_columns(float (&v)[C], const row_state &r, const int (&n)[C], int N) const
   {
      size_t at[C];
#pragma unroll
      for (int i = 0; i < C; ++i) {
         const int co = first + (n[i] < N ? n[i] : N - 1);
         at[i] = r.at + (size_t)co * positions;
      }
      if (bias) {
#pragma unroll
         for (int i = 0; i < C; ++i)
            v[i] += bias[first + (n[i] < N ? n[i] : N - 1)];
      }
      if (R) {
#pragma unroll
         for (int i = 0; i < C; ++i)
            v[i] += R[at[i]];
      }
      f32_activate_all<C>(v, chain);
#pragma unroll
      for (int i = 0; i < C; ++i)
         if (n[i] < N)
            Y[at[i]] = v[i];
   }
   struct added {};
   __device__ __forceinline__ added look_up(int, int) const { return added{}; }
   __device__ __forceinline__ void put(float v, int m, int n, const added &) const
   {
      float one[1] = {v};
      const int col[1] = {n};
      put_columns<1>(one, row_of(m), col, n + 1);
   }
};

// ---- the tile kernel ----------------------------------------------------------------------------------------------------------
// Its fragments are those of v_mfma_f32_32x32x2_f32: a step is 8 k, lane (lk = lane / 32, c = lane % 32) supplies k = 4 lk + j of row
// c to MFMA j, and ends up with columns 8 g + 4 lk + e (g, e = 0..3) of row c.

// Position of (row r, k) of an operand's slab of BK k in LDS, in floats.  Contiguous in k: rows of BK floats whose 16-byte chunks
// are permuted by the row, free of bank conflicts for the fragment read (32 rows, chunks lk = 0, 1).  Contiguous along the
// rows: BK lines of R floats; the two k of a fragment read lie four lines apart, and a gap of 32 floats behind every fourth line
// puts them in different banks (R >= 64: a load instruction never crosses such a gap).
template <int BK>
__device__ __forceinline__ int f32_row_swizzle(int r)
{
   return BK == 16 ? (r >> 2) & 3 : (r >> 1) & 7;
}
template <bool KC, int R>
__device__ __forceinline__ int f32_gap(int k)
{
   return !KC && R >= 64 ? (k >> 2) * 32 : 0;
}
template <bool KC, int R, int BK>
constexpr int f32_slab_floats()
{
   return R * BK + (!KC && R >= 64 ? BK / 4 * 32 : 0);
}

template <class SRC, int R, int BK, int NW>
struct F32Slab {
   static constexpr int VEC = SRC::VEC;
   static constexpr int TOTAL = R * BK / (64 * VEC);  // wave-wide load instructions per slab
   static constexpr int LD = (TOTAL + NW - 1) / NW;   // per wave; where they do not divide, some waves repeat a load
   static constexpr bool KC = SRC::KC;
   static constexpr int FLOATS = f32_slab_floats<SRC::KC, R, BK>();
   typename SRC::template lane_state<LD> st;
   typename SRC::template walk_state<LD> walk;

   // (row, k) of the slab that load i of this wave brings to this lane's place in LDS
   static __device__ __forceinline__ void place(int i, int wave, int lane, int &row, int &kk)
   {
      const int f = (((i * NW + wave) % TOTAL) * 64 + lane) * VEC;
      if (SRC::KC) {
         row = f / BK;
         const int pos = f % BK;
         kk = (((pos >> 2) ^ f32_row_swizzle<BK>(row)) << 2) + (pos & 3);
      } else {
         kk = f / R;
         row = f % R;
      }
   }
   __device__ __forceinline__ void init(const SRC &src, int r0, int wave, int lane)
   {
#pragma unroll
      for (int i = 0; i < LD; ++i) {
         int row, kk;
         place(i, wave, lane, row, kk);
         src.template init<LD>(st, i, r0, row, kk);
      }
      src.template walk_start<LD>(walk, r0, lane, BK, [&](int i) { return ((i * NW + wave) % TOTAL) * 64 * VEC / R; });
   }
   // asks for the next slab; the slabs are asked for one after the other
   template <bool WHOLE>
   __device__ __forceinline__ void issue(const SRC &src, float *lds, int wave, int lane)
   {
      static_for<LD>([&](auto ic) {
         constexpr int i = decltype(ic)::value;
         int row, kk;
         place(i, wave, lane, row, kk);
         const int f = ((i * NW + wave) % TOTAL) * 64 * VEC;
         src.template load<WHOLE, LD>((lds_void_t *)(lds + f + f32_gap<SRC::KC, R>(f / R)), st, walk, i, kk);
      });
      src.walk_on(walk, BK);
   }
   // fragment of k = 8 g .. 8 g + 7 of the 32 rows from r on
   static __device__ __forceinline__ v4f fragment(const float *lds, int r, int g, int lane)
   {
      const int lk = lane >> 5, row = r + (lane & 31);
      if (SRC::KC)
         return *(const v4f *)(lds + row * BK + (((2 * g + lk) ^ f32_row_swizzle<BK>(row)) << 2));
      v4f v;
#pragma unroll
      for (int j = 0; j < 4; ++j)
         v[j] = lds[(8 * g + 4 * lk + j) * R + f32_gap<SRC::KC, R>(8 * g + 4 * lk) + row];
      return v;
   }
};

template <int TM, int TN, bool ALONG_ROWS>
constexpr int f32_store_floats()
{
   return ALONG_ROWS ? TN * (TM + 4) : TM * (TN + 4);
}
// LDS of a tile kernel with a ring of `stages` slabs
template <int BM, int BN, int BK, int WAVES_M, int WAVES_N, int WAVES_K, bool KCA, bool KCB, bool ALONG_ROWS>
constexpr size_t f32_tile_lds_bytes(int stages)
{
   const size_t ring = (size_t)stages * (f32_slab_floats<KCA, BM, BK>() + f32_slab_floats<KCB, BN, BK>()) * 4;
   const size_t store = (size_t)WAVES_M * WAVES_N * WAVES_K * f32_store_floats<BM / WAVES_M, BN / WAVES_N, ALONG_ROWS>() * 4;
   return ring > store ? ring : store;
}

// Ring of STAGES slabs, one barrier per slab.  An fp32 MFMA is slow against what it reads (a 32 x 32 wave tile: 8 KB from LDS per
// 1024 cycles), so neither LDS nor L2 bounds the loop; the matrix cores do where there are enough tiles, and the last, partly
// filled round of tiles where there are not.  WAVES_K waves share a wave tile: each takes its part of the k of every slab,
// which puts all four SIMDs of a CU to work on tiles smaller than four blocks of 32 x 32.
template <class ASRC, class BSRC, class STORE, int BM, int BN, int BK, int WAVES_M, int WAVES_N, int WAVES_K, int STAGES>
__global__ __launch_bounds__(WAVES_M *WAVES_N *WAVES_K * 64, 2) void f32_tile_kernel(ASRC A, BSRC B, STORE out, int M, int N, int K, TileOrder order, int first_tile, long long strideA, long long strideB)
{
   constexpr int NW = WAVES_M * WAVES_N * WAVES_K;
   constexpr int TM = BM / WAVES_M, TN = BN / WAVES_N, MT = TM / 32, NT = TN / 32;
   constexpr int GS = BK / 8 / WAVES_K; // steps of 8 k per slab and wave
   static_assert(TM % 32 == 0 && TN % 32 == 0 && GS >= 1 && GS * WAVES_K * 8 == BK, "wave tile of 32 x 32 blocks");
   typedef F32Slab<ASRC, BM, BK, NW> SA;
   typedef F32Slab<BSRC, BN, BK, NW> SB;
   constexpr int LPT = SA::LD + SB::LD;
   constexpr int STAGE = SA::FLOATS + SB::FLOATS;
   static_assert((STAGES - 1) * LPT < 64, "vmcnt counts fewer than 64 loads");
   extern __shared__ __attribute__((aligned(16))) float f32_lds[];

   int tm, tn, z;
   order.place(first_tile + blockIdx.x, tm, tn, z);
   A.shift(z * strideA);
   B.shift(z * strideB);
   A.select_group(z);
   out.select_batch(z);
   const int m0 = tm * BM, n0 = tn * BN;
   const int lane = threadIdx.x & 63;
   const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
   const int wk = wave % WAVES_K, wm = wave / WAVES_K / WAVES_N, wn = wave / WAVES_K % WAVES_N;

   SA sa;
   SB sb;
   sa.init(A, m0, wave, lane);
   sb.init(B, n0, wave, lane);
   v16f acc[MT][NT];
#pragma unroll
   for (int i = 0; i < MT; ++i)
#pragma unroll
      for (int j = 0; j < NT; ++j)
#pragma unroll
         for (int e = 0; e < 16; ++e)
            acc[i][j][e] = 0.0f;

   constexpr int LPR = TN / 4, RPP = 64 / LPR; // of the store of rows: lanes per row, rows per pass
   const int n_store = n0 + wn * TN + (lane % LPR) * 4;
   v4f bias = {0.0f, 0.0f, 0.0f, 0.0f};
   const int KT = (int)(((unsigned)K + BK - 1) / BK);
   // asks for the next slab, number kt
   auto issue = [&](int kt, int stage, auto whole) {
      float *s = f32_lds + stage * STAGE;
      auto both = [&](auto all) {
         sa.template issue<decltype(all)::value>(A, s, wave, lane);
         sb.template issue<decltype(all)::value>(B, s + SA::FLOATS, wave, lane);
      };
      if (decltype(whole)::value || kt < K / BK)
         both(std::true_type{});
      else
         both(std::false_type{});
   };
   // until at most `slabs` of the slabs asked for last are still on their way (counts past STAGES - 2 wait for that many)
   auto wait_slabs = [&](int slabs) {
      if (slabs >= STAGES - 2)
         wait_vmcnt<(STAGES - 2) * LPT>();
      else if (STAGES > 3 && slabs == 1)
         wait_vmcnt<LPT>();
      else
         wait_vmcnt<0>();
   };
   static_assert(STAGES == 3 || STAGES == 4, "the cases of wait_slabs");
   constexpr std::false_type any{};
   v4f fa[2][GS][MT], fb[2][GS][NT];
   auto read = [&](int stage, v4f(&a)[GS][MT], v4f(&b)[GS][NT]) {
      const float *cA = f32_lds + stage * STAGE, *cB = cA + SA::FLOATS;
#pragma unroll
      for (int g = 0; g < GS; ++g) {
#pragma unroll
         for (int i = 0; i < MT; ++i)
            a[g][i] = SA::fragment(cA, wm * TM + i * 32, wk * GS + g, lane);
#pragma unroll
         for (int j = 0; j < NT; ++j)
            b[g][j] = SB::fragment(cB, wn * TN + j * 32, wk * GS + g, lane);
      }
   };
   if (KT > 0) { // an empty reduction reads nothing
#pragma unroll
      for (int s = 0; s < STAGES; ++s)
         if (s < KT)
            issue(s, s, any);
   }
   // behind the first slabs, whose loads are what a small product waits for (the counts below then wait for a few loads more than they need to)
   if constexpr (!STORE::kAlongRows)
      bias = out.ahead(n_store, N);
   if (KT > 0) {
      if (KT >= STAGES)
         wait_vmcnt<(STAGES - 1) * LPT>();
      else
         wait_slabs(KT - 1);
      __builtin_amdgcn_s_barrier();
      read(0, fa[0], fb[0]);
   }
   // Slab kt: its fragments are in registers.  Behind the barrier slab kt + 1 has landed for every wave and slab kt has been read by
   // every wave: the next fragments are asked for and slab kt + STAGES takes the place of slab kt.  The barrier sits between
   // two halves of the MFMAs, and what is issued behind it is dealt out among those of the second half: a wave that runs alone
   // on its SIMD keeps the matrix core busy.
   // Which place of the ring a step reads is known where the code is written, so every address in LDS is a lane's constant plus an
   // immediate (what computing them took of the multipliers: see F32Matrix).
   auto step = [&](int kt, auto number, auto whole) {
      constexpr int cur = decltype(number)::value % 2, stage = decltype(number)::value % STAGES, next = (stage + 1) % STAGES;
      constexpr bool WHOLE = decltype(whole)::value;
      constexpr int QS = GS * 4, HALF = QS / 2;
      auto multiply = [&](auto from, auto to) {
         static_for<decltype(to)::value - decltype(from)::value>([&](auto qc) {
            constexpr int q = decltype(from)::value + decltype(qc)::value;
#pragma unroll
            for (int i = 0; i < MT; ++i)
#pragma unroll
               for (int j = 0; j < NT; ++j)
                  acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(fb[cur][q / 4][j][q % 4], fa[cur][q / 4][i][q % 4], acc[i][j], 0, 0, 0);
         });
      };
      multiply(std::integral_constant<int, 0>{}, std::integral_constant<int, HALF>{});
      __builtin_amdgcn_sched_barrier(0);
      if constexpr (WHOLE)
         wait_vmcnt<(STAGES - 2) * LPT>();
      else
         wait_slabs(KT - 2 - kt);
      __builtin_amdgcn_s_waitcnt(0xc07f); // lgkmcnt(0): all of this wave's fragments of slab kt are in registers
      __builtin_amdgcn_s_barrier();
      __builtin_amdgcn_sched_barrier(0);
      if (WHOLE || kt + 1 < KT)
         read(next, fa[cur ^ 1], fb[cur ^ 1]);
      if (WHOLE || kt + STAGES < KT)
         issue(kt + STAGES, stage, whole);
      multiply(std::integral_constant<int, HALF>{}, std::integral_constant<int, QS>{});
      constexpr int GROUPS = (QS - HALF) * MT * NT;
      constexpr int READS = GS * ((SA::KC ? MT : 2 * MT) + (SB::KC ? NT : 2 * NT)); // pairs of dwords go into one instruction
#pragma unroll
      for (int g = 0; g < GROUPS; ++g) {
         __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
         __builtin_amdgcn_sched_group_barrier(0x100, (READS + GROUPS - 1) / GROUPS, 0);
         __builtin_amdgcn_sched_group_barrier(0x020, (LPT + GROUPS - 1) / GROUPS, 0);
      }
      __builtin_amdgcn_sched_barrier(0);
   };
   constexpr int ROUND = STAGES % 2 ? 2 * STAGES : STAGES; // steps until ring and register sets are where they were
   int kt = 0;
   // as long as what is asked for is a whole slab, no load looks at its k (the comparison and the selection of an address per load
   // cost 5 - 8 % of the loop)
   for (; kt + ROUND - 1 + STAGES < K / BK; kt += ROUND)
      static_for<ROUND>([&](auto u) { step(kt + decltype(u)::value, u, std::true_type{}); });
   for (; kt < KT; kt += ROUND)
      static_for<ROUND>([&](auto u) {
         if (kt + decltype(u)::value < KT)
            step(kt + decltype(u)::value, u, any);
      });

   // The tile store reuses the ring, one region per wave: the wave's tile is laid out as the result is (rows of columns, or columns
   // of rows), and read back in one rolled loop, so that a wave instruction stores whole lines and the code of the
   // activations exists once.  Waves that share a tile add their parts up as they read, each for its share of the lines.
   wait_vmcnt<0>();
   __syncthreads();
   const int lk = lane >> 5, c = lane & 31;
   constexpr int REGION = f32_store_floats<TM, TN, STORE::kAlongRows>();
   float *mine = f32_lds + wave * REGION, *first = f32_lds + (wave - wk) * REGION;
#pragma unroll
   for (int i = 0; i < MT; ++i)
#pragma unroll
      for (int j = 0; j < NT; ++j)
#pragma unroll
         for (int g = 0; g < 4; ++g) {
            if constexpr (!STORE::kAlongRows)
               *(v4f *)(mine + (i * 32 + c) * (TN + 4) + j * 32 + g * 8 + lk * 4) =
                  v4f{acc[i][j][4 * g], acc[i][j][4 * g + 1], acc[i][j][4 * g + 2], acc[i][j][4 * g + 3]};
            else
#pragma unroll
               for (int e = 0; e < 4; ++e)
                  mine[(j * 32 + g * 8 + lk * 4 + e) * (TM + 4) + i * 32 + c] = acc[i][j][4 * g + e];
         }
   if constexpr (WAVES_K > 1)
      __syncthreads();
   else
      __builtin_amdgcn_wave_barrier();
   if constexpr (!STORE::kAlongRows) {
#pragma unroll 1
      for (int r = wk * RPP + lane / LPR; r < TM; r += RPP * WAVES_K) {
         const int m = m0 + wm * TM + r;
         const float *at = first + r * (TN + 4) + (lane % LPR) * 4;
         v4f v = *(const v4f *)at;
#pragma unroll
         for (int w = 1; w < WAVES_K; ++w)
            v += *(const v4f *)(at + w * REGION);
         if (m < M && n_store < N)
            out.put4(v, m, n_store, N, bias);
      }
   } else {
      constexpr int CPP = TM >= 64 ? 1 : 64 / TM; // columns per pass
      static_assert(TM <= 64, "a column of the wave tile is at most one lane per row");
      const int m = m0 + wm * TM + lane % TM;
      const auto where = out.row_of(m < M ? m : M - 1);
      // four columns at a time: their biases (and residuals) are on their way together
      constexpr int STEP = CPP * WAVES_K, C = TN / STEP >= 4 ? 4 : TN / STEP;
      static_assert(TN % (STEP * C) == 0, "columns divide over the passes");
#pragma unroll 1
      for (int r = wk * CPP + lane / TM; r < TN; r += STEP * C) {
         float v[C];
         int n[C];
#pragma unroll
         for (int i = 0; i < C; ++i) {
            n[i] = n0 + wn * TN + r + i * STEP;
            const float *at = first + (r + i * STEP) * (TM + 4) + lane % TM;
            v[i] = *at;
#pragma unroll
            for (int w = 1; w < WAVES_K; ++w)
               v[i] += at[w * REGION];
         }
         if (m < M)
            out.template put_columns<C>(v, where, n, N);
      }
   }
}

// ---- the direct kernel --------------------------------------------------------------------------------------------------------
// The partial tiles of W waves meet in LDS and are stored, an element by a thread.
template <int MB, int NB, int W, class STORE>
struct F32DirectStore {
   static constexpr int TM = MB * 16, TN = NB * 16;
   static_assert(TM * TN <= W * 64, "an element by a thread");
   int r, q; // neighbouring threads store neighbouring elements of the direction that is contiguous in the result
   bool live;
   typename STORE::added added = {};
   __device__ __forceinline__ F32DirectStore(int m0, int n0, int M, int N)
   {
      const int e = threadIdx.x;
      r = STORE::kAlongRows ? e % TM : e / TN, q = STORE::kAlongRows ? e / TM : e % TN;
      live = e < TM * TN && m0 + r < M && n0 + q < N;
   }
   // what is added to the element, behind the first loads of the operands
   __device__ __forceinline__ void ask(const STORE &out, int m0, int n0)
   {
      if (live)
         added = out.look_up(m0 + r, n0 + q);
   }
   __device__ __forceinline__ void store(const STORE &out, const v4f (&acc)[MB][NB], float (*part)[TM][TN + 4], int m0, int n0, int wave, int lane) const
   {
      const int lk = lane >> 4, c = lane & 15;
#pragma unroll
      for (int i = 0; i < MB; ++i)
#pragma unroll
         for (int j = 0; j < NB; ++j)
            *(v4f *)&part[wave][i * 16 + c][j * 16 + lk * 4] = acc[i][j];
      __syncthreads();
      if (live) {
         float v = part[0][r][q];
#pragma unroll
         for (int w = 1; w < W; ++w)
            v += part[w][r][q];
         out.put(v, m0 + r, n0 + q, added);
      }
   }
};

// W waves split the reduction of one (16 MB) x (16 NB) tile in steps of 16 k (v_mfma_f32_16x16x4_f32: lane (lk = lane / 16, c = lane
// % 16) supplies k = 4 lk + j of row c to MFMA j); the partial tiles meet in LDS.  What such a product
// costs is one trip to memory for its operands: every wave has UNROLL steps of loads in flight at once.  No step but the last looks at its k, and no branch stands
// between loads of single floats: with one around each, a wave alone on its SIMD took as long for them as for the trip.  us, before -> after, with the bias asked for behind the first
// loads: 64 x 10 x 64 3.09 -> 2.57, 256 x 10 x 256 4.2 -> 3.05, 16 x 10 x 333 4.4 -> 2.95, 100 x 33 x 77 3.7 -> 2.95, 200 x 17 x 50 3.5 -> 2.75, 1 x 1000 x 2048 5.9 -> 5.6.
template <class ASRC, class BSRC, class STORE, int MB, int NB, int W, int UNROLL>
__global__ __launch_bounds__(W * 64) void f32_direct_kernel(ASRC A, BSRC B, STORE out, int M, int N, int K, TileOrder order, int first_tile, long long strideA,
                                                            long long strideB)
{
   constexpr int TM = MB * 16, TN = NB * 16, PITCH = TN + 4;
   __shared__ __attribute__((aligned(16))) float part[W][TM][PITCH];
   int tm, tn, z;
   order.place(first_tile + blockIdx.x, tm, tn, z);
   A.shift(z * strideA);
   B.shift(z * strideB);
   A.select_group(z);
   out.select_batch(z);
   const int m0 = tm * TM, n0 = tn * TN;
   const int lane = threadIdx.x & 63;
   const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
   const int lk = lane >> 4, c = lane & 15;
   typename ASRC::row_state ra[MB];
   typename BSRC::row_state rb[NB];
#pragma unroll
   for (int i = 0; i < MB; ++i)
      ra[i] = A.row_of(m0 + i * 16 + c);
#pragma unroll
   for (int j = 0; j < NB; ++j)
      rb[j] = B.row_of(n0 + j * 16 + c);
   v4f acc[MB][NB];
#pragma unroll
   for (int i = 0; i < MB; ++i)
#pragma unroll
      for (int j = 0; j < NB; ++j)
         acc[i][j] = v4f{0.f, 0.f, 0.f, 0.f};
   F32DirectStore<MB, NB, W, STORE> store(m0, n0, M, N);
   const int KS = (int)(((unsigned)K + 15) / 16);
   for (int s0 = wave; s0 < KS; s0 += W * UNROLL) {
      v4f fa[UNROLL][MB], fb[UNROLL][NB];
#pragma unroll
      for (int u = 0; u < UNROLL; ++u) {
         const unsigned first = (unsigned)(s0 + u * W) * 16; // of steps past the end it may leave 31 bits
         auto load = [&](auto whole) {
            constexpr bool WHOLE = decltype(whole)::value;
            const int k = (int)(first + lk * 4), left = (int)((unsigned)K - first) - lk * 4;
#pragma unroll
            for (int i = 0; i < MB; ++i)
               fa[u][i] = A.template fetch<WHOLE>(ra[i], k, left);
#pragma unroll
            for (int j = 0; j < NB; ++j)
               fb[u][j] = B.template fetch<WHOLE>(rb[j], k, left);
         };
         if (first + 16 <= (unsigned)K) {
            load(std::true_type{});
         } else if (first < (unsigned)K) {
            load(std::false_type{});
         } else {
#pragma unroll
            for (int i = 0; i < MB; ++i)
               fa[u][i] = v4f{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int j = 0; j < NB; ++j)
               fb[u][j] = v4f{0.f, 0.f, 0.f, 0.f};
         }
      }
      if (s0 == wave)
         store.ask(out, m0, n0);
#pragma unroll
      for (int u = 0; u < UNROLL; ++u)
#pragma unroll
         for (int i = 0; i < MB; ++i)
#pragma unroll
            for (int j = 0; j < NB; ++j)
               acc[i][j] = mfma_f32_step(fb[u][j], fa[u][i], acc[i][j]);
   }
   if (wave >= KS)
      store.ask(out, m0, n0);
   store.store(out, acc, part, m0, n0, wave, lane);
}

// The same through LDS, where both operands are contiguous in k and their rows start on 16 bytes (see direct_ring_sums): 64 x 128 x 784 takes 4.1 us instead of
// 4.9, 16 x 1024 x 1024 4.4 instead of 6.3, 1 x 1000 x 2048 6.0 instead of 7.3.  Lane (lk, c) holds k = 8 lk .. 8 lk + 7 of 32 of row c of either operand, and
// MFMA j takes the j-th of them; the two halves are summed apart, so that a partial sum is as short as it is above.
struct DirectF32 {
   typedef float acc_t __attribute__((ext_vector_type(8)));
   static __device__ __forceinline__ acc_t mma(const v4i (&n_side)[2], const v4i (&m_side)[2], acc_t acc)
   {
      const v4f first = mfma_f32_step(__builtin_bit_cast(v4f, n_side[0]), __builtin_bit_cast(v4f, m_side[0]), __builtin_shufflevector(acc, acc, 0, 1, 2, 3));
      const v4f second = mfma_f32_step(__builtin_bit_cast(v4f, n_side[1]), __builtin_bit_cast(v4f, m_side[1]), __builtin_shufflevector(acc, acc, 4, 5, 6, 7));
      return __builtin_shufflevector(first, second, 0, 1, 2, 3, 4, 5, 6, 7);
   }
};
template <class STORE, int MB, int NB, int W>
__global__ __launch_bounds__(W * 64) void f32_direct_ring_kernel(RowMajorRows A, RowMajorRows B, STORE out, int M, int N, int K, TileOrder order, int first_tile, long long strideA,
                                                                 long long strideB, int depth)
{
   extern __shared__ __attribute__((aligned(16))) int8_t smem[];
   int tm, tn, z;
   order.place(first_tile + blockIdx.x, tm, tn, z);
   A.base += z * strideA;
   B.base += z * strideB;
   out.select_batch(z);
   const int m0 = tm * MB * 16, n0 = tn * NB * 16;
   const int lane = threadIdx.x & 63;
   const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
   DirectF32::acc_t both[MB][NB];
   direct_ring_sums<DirectF32, MB, NB, W>(both, A, B, M, N, K, m0, n0, smem, depth, wave, lane);
   v4f acc[MB][NB];
#pragma unroll
   for (int i = 0; i < MB; ++i)
#pragma unroll
      for (int j = 0; j < NB; ++j)
         acc[i][j] = __builtin_shufflevector(both[i][j], both[i][j], 0, 1, 2, 3) + __builtin_shufflevector(both[i][j], both[i][j], 4, 5, 6, 7);
   F32DirectStore<MB, NB, W, STORE> store(m0, n0, M, N);
   store.ask(out, m0, n0);
   __syncthreads();
   store.store(out, acc, (float(*)[MB * 16][NB * 16 + 4])smem, m0, n0, wave, lane);
}

// ---- launches -----------------------------------------------------------------------------------------------------------------
template <class ASRC, class BSRC, class STORE, int BM, int BN, int BK, int WAVES_M, int WAVES_N, int WAVES_K, int STAGES>
static int launch_f32_tile(hipStream_t stream, const ASRC &A, const BSRC &B, const STORE &out, int M, int N, int K, int batch, long long strideA, long long strideB)
{
   const int tiles_m = (M + BM - 1) / BM, tiles_n = (N + BN - 1) / BN;
   const long long nwg = (long long)tiles_m * tiles_n;
   if (nwg > 0x7fffffffLL)
      return fail(SOFIE_HIP_ERR_INVALID, "fp32 product: too many tiles");
   // a reduction of fewer slabs than the ring holds takes only their places: more workgroups share a CU (first convolution of a
   // 64-image network, one slab: 40 -> 32 us)
   const int slabs = K > BK * (STAGES - 1) ? STAGES : K > BK ? (K + BK - 1) / BK : 1;
   const size_t smem = f32_tile_lds_bytes<BM, BN, BK, WAVES_M, WAVES_N, WAVES_K, ASRC::KC, BSRC::KC, STORE::kAlongRows>(slabs);
   constexpr size_t most = f32_tile_lds_bytes<BM, BN, BK, WAVES_M, WAVES_N, WAVES_K, ASRC::KC, BSRC::KC, STORE::kAlongRows>(STAGES);
   static_assert(most <= 160 * 1024, "LDS of a CU");
   auto kern = f32_tile_kernel<ASRC, BSRC, STORE, BM, BN, BK, WAVES_M, WAVES_N, WAVES_K, STAGES>;
   static bool configured[64] = {};
   if (int st = configure_lds_once(kern, most, configured))
      return st;
   constexpr int NTHREADS = WAVES_M * WAVES_N * WAVES_K * 64;
   const TileOrder order(tiles_m, tiles_n, 4, batch);
   in_launches(order.workgroups(batch), NTHREADS, [&](int first, unsigned count) {
      launch_kernel(kern, dim3(count, 1, order.depth(batch)), dim3(NTHREADS), smem, stream, A, B, out, M, N, K, order, first, strideA, strideB);
   });
   return launch_status("f32_tile_kernel");
}

template <class ASRC, class BSRC, class STORE, int MB, int NB, int W, int UNROLL>
static int launch_f32_direct(hipStream_t stream, const ASRC &A, const BSRC &B, const STORE &out, int M, int N, int K, int batch, long long strideA, long long strideB)
{
   const int tiles_m = (M + MB * 16 - 1) / (MB * 16), tiles_n = (N + NB * 16 - 1) / (NB * 16);
   const long long nwg = (long long)tiles_m * tiles_n;
   if (nwg > 0x7fffffffLL)
      return fail(SOFIE_HIP_ERR_INVALID, "fp32 product: too many tiles");
   const TileOrder order(tiles_m, tiles_n, 4, batch);
   if constexpr (ASRC::KC && BSRC::KC && ASRC::VEC == 4 && BSRC::VEC == 4) {
      typedef DirectRing<MB, NB, W> Ring;
      // A single step has nothing to pipeline: 64 x 640 x 32 2.83 us, 2.89 through the ring, 130 x 1500 x 32 9 % longer.  Few rows that do not start on lines take two
      // lines a step, which the registers' finer steps hide up to K = 512: 4 x 97 x 436 3.84 us, 4.10 through the ring.
      const bool by_lines = K > 32 && (M > 8 || K <= 128 || K >= 512 || (A.ld % 32 == 0 && B.ld % 32 == 0));
      if (by_lines && Ring::takes(A.p, B.p, A.ld * 4, B.ld * 4, K * 4LL)) {
         const Ring ring(nwg * batch, K * 4);
         auto kern = f32_direct_ring_kernel<STORE, MB, NB, W>;
         static bool configured[64] = {};
         if (int st = configure_lds_once(kern, 128 * 1024, configured))
            return st;
         const RowMajorRows a{(const int8_t *)A.p, (int)(A.ld * 4)}, b{(const int8_t *)B.p, (int)(B.ld * 4)};
         in_launches(order.workgroups(batch), W * 64, [&](int first, unsigned count) {
            launch_kernel(kern, dim3(count, 1, order.depth(batch)), dim3(W * 64), ring.bytes, stream, a, b, out, M, N, K * 4, order, first, strideA * 4,
                          strideB * 4, ring.depth);
         });
         return launch_status("f32_direct_ring_kernel");
      }
   }
   in_launches(order.workgroups(batch), W * 64, [&](int first, unsigned count) {
      launch_kernel((f32_direct_kernel<ASRC, BSRC, STORE, MB, NB, W, UNROLL>), dim3(count, 1, order.depth(batch)), dim3(W * 64), 0, stream, A, B, out, M, N, K, order,
                    first, strideA, strideB);
   });
   return launch_status("f32_direct_kernel");
}

} // namespace sofie_hip
