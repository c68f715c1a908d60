// fp32 3 x 3 convolution (stride 1, no dilation, two spatial axes) of up to four input channels per group: the first layer of an image network.
//
// A result takes 9 to 36 products and is written once: the layer is bound by its stores (3 -> 32 channels on 64 images of 64 x 64: 33.6 MB) and by the instructions
// around the MFMAs.  With a tile of 128 pixels a workgroup of f32_conv3x3.hpp spent 300 vector instructions a wave on places, weights and addresses beside 18 MFMAs, four
// channels wide.  Here the reduction is the layer's own 9 C, in the order the weights have in memory, padded to a multiple of four (v_mfma_f32_16x16x4_f32: seven MFMAs for
// three channels, 32 cycles each), and a workgroup takes `span` consecutive pixels of an image: weights and the distances of a lane's products in the patch are worked out
// once, and 32 pixels more cost two quotients, the reads of their fragments and the stores.  us, tiles of 128 pixels -> here: 64 images of 64 x 64, 3 -> 32 channels 14.6 ->
// 12.1, 8 of 96 x 96, 3 -> 48 10.8 -> 10.0, 30 of 47 x 47, 3 -> 9 5.9 -> 4.6, 1 of 20 x 20, 3 -> 16 3.6 -> 2.9 (not for
// many small images: f32_conv3x3_few_preferred).  Of the first, 7.1 are left without MFMAs and stores, 8.9 with the stores, 11.9 with the MFMAs: all its workgroups start together, and wait for the same things.
#pragma once
#include "f32_conv3x3.hpp"
#include <cmath>

namespace sofie_hip {

// Floats of LDS a workgroup may take for its patch: four workgroups a CU.
constexpr int F32_CONV3X3_FEW_PATCH = 10 * 1024;

// Positions of the patch of any `span` pixels of an image, padded to whole load instructions.
inline long long f32_conv3x3_few_patch(int OH, int OW, int span)
{
   const long long plane = (long long)OH * OW, most = span < plane ? span : plane;
   const long long rows = most % OW == 0 && span % OW == 0 ? most / OW : (most - 2 + OW) / OW + 1;
   return (((rows < OH ? rows : OH) + 2) * (OW + 2LL) + 63) / 64 * 64;
}

// STEPS: MFMAs of four k, of a block of 16 channels; NB: blocks of 16 channels.  A wave takes 32 pixels at a time, two blocks of 16 that share the weights.
template <int STEPS, int NB, bool PLAIN>
__global__ __launch_bounds__(256, 4) void f32_conv3x3_few_kernel(F32Conv3x3 a, F32ConvStore out, TileOrder order, Divisor31 by_chunks, int span, int plane, int first)
{
   extern __shared__ __attribute__((aligned(16))) float few_lds[]; // [channel][plane]
   const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lk = lane >> 4, c = lane & 15;
   int id, tn, z;
   order.place(first + blockIdx.x, id, tn, z);
   a.X += z * a.group;
   a.W += (long long)z * a.N * a.K;
   out.select_batch(z);
   auto quotient = [](int n, const Divisor31 &by) { return (int)by.over((unsigned)n); };
   // image by image, pixels side by side: the workgroups of an XCD share the rows between their patches, and the patch of a tile's channels
   const int image = quotient(id, by_chunks), p0 = (id - image * (int)by_chunks.d) * span, n0 = tn * NB * 16;
   const int count = out.positions - p0 < span ? out.positions - p0 : span;
   const int VW = a.OW + 2, row0 = quotient(p0, a.by_ow), rows = quotient(p0 + count - 1, a.by_ow) - row0 + 3;

   // weights: lane (lk, c) supplies k = 4 j + lk of channel c of a block to MFMA j
   const char *weights = (const char *)uniform((long long)(a.W + (long long)n0 * a.K));
   float w[NB][STEPS];
#pragma unroll
   for (int b = 0; b < NB; ++b) {
      const int at = n0 + b * 16 + c < a.N ? ((b * 16 + c) * a.K + lk) * 4 : F32_OUTSIDE;
#pragma unroll
      for (int j = 0; j < STEPS; ++j) // (an immediate behind F32_OUTSIDE stays outside)
         w[b][j] = f32_bounded_read(weights, j < STEPS - 1 || 4 * j + lk < a.K ? (at == F32_OUTSIDE ? (int)0x80000000 : at) + 16 * j : (int)0x80000000, (int)F32_BUFFER_BYTES);
   }
   // the patch: rows row0 .. of the padded image, OW + 2 columns, channel by channel
   const char *base = (const char *)uniform((long long)(a.X + image * a.image));
   const int plane_bytes = a.H * a.Wd * 4;
   for (int q = wave; q * 64 < rows * VW; q += 4) {
      const int f = q * 64 + lane, vr = quotient(f, a.by_vw), ix = f - vr * VW - a.pad_w, iy = row0 + vr - a.pad_h;
      const int at = vr < rows && (unsigned)ix < (unsigned)a.Wd && (unsigned)iy < (unsigned)a.H ? (iy * a.Wd + ix) * 4 : F32_OUTSIDE;
#pragma unroll
      for (int ch = 0; ch < 4; ++ch)
         if (ch * 9 < STEPS * 4 && ch < a.C)
            f32_buffer_load<1>((lds_void_t *)(few_lds + ch * plane + q * 64), base, at, ch * plane_bytes);
   }
   float bias[NB][4];
   int from[STEPS]; // where this lane's k lie in the patch, a choice of four scalars; any place for those past the last
#pragma unroll
   for (int j = 0; j < STEPS; ++j) {
      int at[4];
#pragma unroll
      for (int q = 0; q < 4; ++q) {
         const int k = 4 * j + q;
         at[q] = k < STEPS / 2 * 9 ? k / 9 * plane + k % 9 / 3 * VW + k % 3 : 0;
      }
      from[j] = lk == 0 ? at[0] : at[1];
      from[j] = lk == 2 ? at[2] : from[j];
      from[j] = lk == 3 ? at[3] : from[j];
   }
   // results: a lane holds channels 4 lk .. 4 lk + 3 of a block, of one pixel
   const long long origin = ((long long)image * out.Cout + out.first + n0) * out.positions;
   float *Y = (float *)uniform((long long)(out.Y + origin));
   const float *R = out.R ? (const float *)uniform((long long)(out.R + origin)) : nullptr;
   const float *B = out.bias ? (const float *)uniform((long long)(out.bias + out.first + n0)) : nullptr;
#pragma unroll
   for (int b = 0; b < NB; ++b)
#pragma unroll
      for (int e = 0; e < 4; ++e)
         bias[b][e] = B ? f32_bounded_read(B, (b * 16 + lk * 4 + e) * 4, (a.N - n0) * 4) : 0.0f;
   wait_vmcnt<0>();
   __syncthreads();

   const int channel_bytes = out.positions * 4, patch0 = row0 * VW;
   for (int i0 = wave * 32; i0 < count; i0 += 128) {
      float x[2][STEPS];
      int lane_at[2];
#pragma unroll
      for (int s = 0; s < 2; ++s) {
         const int i = i0 + s * 16 + c, pixel = p0 + (i < count ? i : count - 1), row = quotient(pixel, a.by_ow);
         const float *at = few_lds + pixel + 2 * row - patch0; // (row - row0) VW + pixel - row OW
#pragma unroll
         for (int j = 0; j < STEPS; ++j)
            x[s][j] = at[from[j]];
         if (4 * STEPS - 4 + lk >= a.K) // no value of the layer: one that is not finite would not vanish beside the weight of zero
            x[s][STEPS - 1] = 0.0f;
         lane_at[s] = i < count ? (pixel + lk * 4 * out.positions) * 4 : F32_OUTSIDE;
      }
      v4f acc[2][NB];
#pragma unroll
      for (int s = 0; s < 2; ++s)
#pragma unroll
         for (int b = 0; b < NB; ++b)
            acc[s][b] = v4f{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
      for (int j = 0; j < STEPS; ++j)
#pragma unroll
         for (int b = 0; b < NB; ++b)
#pragma unroll
            for (int s = 0; s < 2; ++s)
               acc[s][b] = __builtin_amdgcn_mfma_f32_16x16x4f32(w[b][j], x[s][j], acc[s][b], 0, 0, 0);
      // what(s, b, e, where), the place of element e of block b as a lane's offset and a scalar; channels past the last lie behind the buffer
      auto each = [&](auto &&what) {
         auto all = [&](auto whole) {
            int N = a.N - n0; // compared here: kept from one place to the next, the comparisons fill the scalar registers
            forget(N);
#pragma unroll
            for (int b = 0; b < NB; ++b)
#pragma unroll
               for (int e = 0; e < 4; ++e)
#pragma unroll
                  for (int s = 0; s < 2; ++s)
                     what(s, b, e, decltype(whole)::value || b * 16 + lk * 4 + e < N ? lane_at[s] : F32_OUTSIDE, (b * 16 + e) * channel_bytes);
         };
         if (n0 + NB * 16 <= a.N)
            all(std::true_type{});
         else
            all(std::false_type{});
      };
#pragma unroll
      for (int s = 0; s < 2; ++s)
#pragma unroll
         for (int b = 0; b < NB; ++b)
#pragma unroll
            for (int e = 0; e < 4; ++e)
               acc[s][b][e] += bias[b][e];
      if (R) {
         float r[2][NB][4];
         each([&](int s, int b, int e, int at, int scalar) { r[s][b][e] = f32_buffer_read(R, at, scalar); });
#pragma unroll
         for (int s = 0; s < 2; ++s)
#pragma unroll
            for (int b = 0; b < NB; ++b)
#pragma unroll
               for (int e = 0; e < 4; ++e)
                  acc[s][b][e] += r[s][b][e];
      }
      if constexpr (PLAIN) {
         if (out.chain.count)
#pragma unroll
            for (int s = 0; s < 2; ++s)
#pragma unroll
               for (int b = 0; b < NB; ++b)
#pragma unroll
                  for (int e = 0; e < 4; ++e)
                     asm("v_max_f32 %0, 0, %0" : "+v"(acc[s][b][e])); // v > 0 ? v : 0, NaN and -0 among them
      } else {
         // one copy of the activations' code for four elements
#pragma unroll 1
         for (int g = 0; g < 2 * NB; ++g) {
            v4f four = acc[0][0];
#pragma unroll
            for (int q = 1; q < 2 * NB; ++q)
               four = g == q ? acc[q / NB][q % NB] : four;
            f32_activate_all<4>(four, out.chain);
#pragma unroll
            for (int q = 0; q < 2 * NB; ++q)
               acc[q / NB][q % NB] = g == q ? four : acc[q / NB][q % NB];
         }
      }
      each([&](int s, int b, int e, int at, int scalar) { f32_buffer_store(acc[s][b][e], Y, at, scalar); });
   }
}

// Whether the kernel takes a layer: channels, workgroups of one launch, results and inputs of an image within a buffer, a patch within its LDS.
inline bool f32_conv3x3_few_takes(const F32Conv3x3 &a, const F32ConvStore &out)
{
   const long long bytes = F32_BUFFER_BYTES - (1 << 20);
   return a.C <= 4 && (long long)a.images * ((out.positions + 127) / 128) * ((a.N + 15) / 16) <= 0x7fffffffLL && 80LL * out.positions * 4 < bytes && 4LL * a.H * a.Wd * 4 < bytes && f32_conv3x3_few_patch(a.OH, a.OW, 128) * a.C <= F32_CONV3X3_FEW_PATCH;
}

// How a layer is split: pixels and blocks of channels of a workgroup, floats of a channel of its patch.
struct F32Conv3x3FewSplit {
   int span, chunks, nb, tiles_n, plane;
   long long total; // workgroups of a group
   F32Conv3x3FewSplit(const F32Conv3x3 &a, const F32ConvStore &out, int group)
   {
      // Channels of a tile: as many blocks of 16 as there are, or as few tiles as hold four each.  Pixels: as many as leave two workgroups for each CU, us with 128 / 256 / 512 / 1024:
      // 64 images of 64 x 64, 3 -> 32 channels 16.2 / 13.5 / 12.6 / 13.8, 16 of 28 x 28, 1 -> 32 3.2 / 3.9 / 5.3 / 7.2, 64 of 96 x 96, 3 -> 16 18.9 / 15.0 / 14.5 / 15.6.
      const int blocks = (a.N + 15) / 16;
      tiles_n = (blocks + 3) / 4;
      span = 512;
      auto workgroups = [&] { return (long long)a.images * ((out.positions + span - 1) / span) * tiles_n; };
      while (span > 128 && (workgroups() * group < 512 || f32_conv3x3_few_patch(a.OH, a.OW, span) * a.C > F32_CONV3X3_FEW_PATCH))
         span /= 2;
      while (tiles_n < blocks && workgroups() * group < 256)
         ++tiles_n;
      nb = (blocks + tiles_n - 1) / tiles_n;
      tiles_n = (blocks + nb - 1) / nb;
      chunks = (out.positions + span - 1) / span;
      span = ((out.positions + chunks - 1) / chunks + 31) / 32 * 32; // as much for each
      plane = (int)f32_conv3x3_few_patch(a.OH, a.OW, span);
      total = workgroups();
   }
};

// Whether the kernel is faster than tiles of 128 pixels, four channels wide, that run through images (f32_conv3x3.hpp; `patch`: their positions).  A workgroup here stays within an
// image, so that one of 9 pixels is a workgroup of 128 places for each, and the four-channel kernel with four blocks spills: us, those tiles / here, 65536 images of 3 x 3, 4 -> 64 channels 60 / 614,
// 16384 of 5 x 5, 3 -> 32 23 / 67, 124 of 14 x 14, 4 -> 48 6.0 / 7.5, 21 of 63 x 63, 4 -> 159 21.9 / 30.3, but 6311 of 8 x 8, 3 -> 2 17.2 / 13.2, and 64 of 64 x 64, 3 -> 32 14.6 /
// 12.1.  Costs, us: a launch, the trip to memory, a CU's workgroups by their patches and MFMAs, the layer's bytes; a launch and a CU's tiles.  Fitted for the choice to 1161 layers
// of 1 to 65536 images of 3 to 115 columns, up to 160 channels out, up to 256 groups: 0.2 % above the faster on average, 15 % the most (always here: 9.4 %, 5.7 times; always there: 50 %).
inline bool f32_conv3x3_few_preferred(const F32Conv3x3 &a, const F32ConvStore &out, const F32Conv3x3FewSplit &split, int group, long long patch)
{
   const int steps = (9 * a.C + 3) / 4;
   const double cus = 256.0, workgroups = std::ceil((double)split.total * group / cus), tiles = std::ceil((double)((a.M + 127LL) / 128) * ((a.N + 31LL) / 32) * group / cus);
   const double trip = 0.106 * split.nb * steps, bytes = 4.0 * a.images * group * (a.C + a.N) * out.positions;
   const double each = 0.036 + 0.000189 * split.plane * a.C + (split.span + 127) / 128 * split.nb * (0.0306 * steps + 0.126) * (a.C < 4 ? 1.0 : split.nb < 4 ? 1.13 : 1.82);
   const double here = 2.89 + std::sqrt(trip * trip + workgroups * each * workgroups * each + bytes / 6.8e6 * (bytes / 6.8e6));
   return here <= 3.47 + tiles * (1.07 + 0.000244 * patch);
}

static int launch_f32_conv3x3_few(hipStream_t stream, const F32Conv3x3 &a, const F32ConvStore &out, const F32Conv3x3FewSplit &split, int group)
{
   const size_t smem = (size_t)split.plane * a.C * 4;
   auto with = [&](auto steps, auto nbc, auto plain) {
      auto kern = f32_conv3x3_few_kernel<decltype(steps)::value, decltype(nbc)::value, decltype(plain)::value>;
      const TileOrder order((int)(split.total / split.tiles_n), split.tiles_n, 0, group);
      in_launches(order.workgroups(group), 256, [&](int first, unsigned count) {
         launch_kernel(kern, dim3(count, 1, order.depth(group)), dim3(256), smem, stream, a, out, order, Divisor31(split.chunks), split.span, split.plane, first);
      });
      return launch_status("f32_conv3x3_few_kernel");
   };
   auto blocks_of = [&](auto steps, auto plain) {
      switch (split.nb) {
      case 1: return with(steps, std::integral_constant<int, 1>{}, plain);
      case 2: return with(steps, std::integral_constant<int, 2>{}, plain);
      case 3: return with(steps, std::integral_constant<int, 3>{}, plain);
      default: return with(steps, std::integral_constant<int, 4>{}, plain);
      }
   };
   auto go = [&](auto plain) {
      switch (a.C) {
      case 1: return blocks_of(std::integral_constant<int, 3>{}, plain);
      case 2: return blocks_of(std::integral_constant<int, 5>{}, plain);
      case 3: return blocks_of(std::integral_constant<int, 7>{}, plain);
      default: return blocks_of(std::integral_constant<int, 9>{}, plain);
      }
   };
   return conv3x3_plain(out.chain) ? go(std::true_type{}) : go(std::false_type{});
}

} // namespace sofie_hip
