// fp32 3 x 3 convolution (stride 1, no dilation, two spatial axes) with the input patch of a tile in LDS.
//
// The implicit product of f32_mfma.hpp gathers every element of the column matrix, nine times the input: a load instruction of 64
// floats touches three or four lines, and a slab of 32 k of a 64 x 64 tile took 0.60 us where its MFMAs take 0.43.  Here a tile is BM consecutive output pixels
// (through rows and images) and BN output channels; what it reads of a channel is one run of rows, loaded once, and the nine kernel
// positions read it from LDS at offsets that are known where the code is written.  64 images, us before -> after: 32 -> 64 channels at
// 32 x 32 36.7 -> 26.8, 64 -> 64 57.2 -> 43.8 (110 TFLOP/s of the matrix cores' 157; on another card 44.7, with a residual 45.3), 3 -> 32 at
// 64 x 64 24.2 -> 17.0 (14.9 with the stores below); one image, 48 -> 96 at 40 x 40 12.8 -> 8.4.  (Up to four channels: a slab of four, or f32_conv3x3_few.hpp.)  On 64 -> 64 the matrix cores work in 0.72 of the cycles and no bank conflicts are
// counted; what is left is a patch that is loaded once per 32 output channels and one MFMA per value read from LDS.
//
// The images are taken as one column of OH + 2 rows each, padding included (row r of image i is row i (OH + 2) + r), and OW + 2 columns:
// the patch of a tile is the rows from its first pixel's to two below its last pixel's.
#pragma once
#include "f32_mfma.hpp"
#include <algorithm>

namespace sofie_hip {

struct F32Conv3x3 {
   const float *X, *W; // NCHW; [Cout][C][3][3]
   int images, C, H, Wd, OH, OW, pad_h, pad_w; // C: channels per group
   long long image, group;                     // elements per image and per group of channels
   int M, N, K;                                // output pixels, output channels per group, 9 C
   int chunks;                                 // of 64 positions that a patch fills
   int near;                                   // the results of a tile's images lie within a buffer
   Divisor31 by_ow, by_oh, by_vw, by_vh;       // by OW, OH, OW + 2, OH + 2
};

// The largest patch that is taken: square images of up to 115 columns at every tile but the largest, and wider ones up to 168 whose columns a
// tile divides.  No image wider than 96 was timed when the line was drawn (a tile across two of those: 686 places); beyond it the gathering
// kernels run.  It is not a limit of LDS: 904 places, for any image of 224 columns, would be 80 KB for two slabs, twice on a CU.
constexpr int F32_CONV3X3_PATCH = 704;

// Positions of the patch of any tile of `bm` pixels: rows it touches, two more, and two per image that it runs into.
inline long long f32_conv3x3_patch(int OH, int OW, int bm)
{
   const long long plane = (long long)OH * OW;
   const long long rows = bm % OW == 0 ? bm / OW : (bm - 2 + OW) / OW + 1;
   const long long images = plane % bm == 0 ? 0 : (bm - 2 + plane) / plane;
   return (rows + 2 + 2 * images) * (OW + 2);
}

// A float of a buffer of which `base` is the (scalar) start; F32_OUTSIDE reads as zero.
__device__ __forceinline__ float f32_buffer_read(const void *base, int offset, int scalar_offset)
{
   const __amdgpu_buffer_rsrc_t buffer = __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(base), 0, (int)F32_BUFFER_BYTES, 0x00020000);
   return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(buffer, offset, scalar_offset, 0));
}
// A float of a buffer of `bytes`, zero from its end on.  No scalar offset: the check against the end leaves it out.
__device__ __forceinline__ float f32_bounded_read(const void *base, int offset, int bytes)
{
   const __amdgpu_buffer_rsrc_t buffer = __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(base), 0, bytes, 0x00020000);
   return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(buffer, offset, 0, 0));
}
__device__ __forceinline__ void f32_buffer_store(float v, const void *base, int offset, int scalar_offset)
{
   const __amdgpu_buffer_rsrc_t buffer = __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(base), 0, (int)F32_BUFFER_BYTES, 0x00020000);
   __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned, v), buffer, offset, scalar_offset, 0);
}

// A scalar that the compiler takes for a new one: what is worked out from it is worked out again.  Kept from one place to the next (bounds of a slab's loads, a
// mask each) it fills the scalar registers, and a spilled one costs a vector instruction where it is written and one where it is read.
__device__ __forceinline__ void forget(int &v) { asm volatile("" : "+s"(v)); }

// Activations that take no call.  Kernels apart for those that do, whose calls keep registers free: they spill 17 - 70 scalars where most of the plain ones spill fewer.
inline bool conv3x3_plain(const PostChain &chain) { return chain.count == 0 || (chain.count == 1 && chain.op0 == SOFIE_ACT_RELU); }

// The results that a lane holds of a block: E of the 16 channels first + 4 lk + e / 4 * 8 + e % 4, from element e0 (a multiple of 4) on, of one pixel.  32 neighbouring
// lanes hold 32 neighbouring pixels of a channel: whole lines, loaded and stored straight from the registers.  Addresses are an offset per lane, one for all
// channels, and a scalar per channel.  A tile of few input channels is bound by the instructions around its MFMAs: with an address, a bound and a branch per
// channel, places of the patch worked out by every wave and more scalars spilled, 3 -> 32 channels had 18 MFMAs a wave among 573 vector and 357 scalar instructions, now
// 303 and 298.  64 images of 64 x 64, us before -> after, for all of these together: 3 -> 32 channels 19.3 -> 14.9; 40 of 90 x 90, 3 -> 12 23.2 -> 16.7; 1 of 64 x 64
// 5.5 -> 4.0.  Still spilled, in plain kernels: 6 scalars with few channels, 20 - 32 at 128 pixels, up to 66 where waves share a tile (none at 256 places with wide
// weights).
template <int E>
struct Conv3x3Block {
   float *Y;         // result of channel `first`, pixel 0 of the tile's first image (scalar)
   const float *R;   // the same of the residual, or nullptr
   const float *B;   // bias of channel `first`, or nullptr
   long long at;     // of this lane's pixel from Y, in floats, channel first + 4 lk
   int positions, N; // N: channels from `first` on
   int lk, e0;
   bool live, near; // the pixel is one of the layer's; the tile's results lie within a buffer
   __device__ __forceinline__ Conv3x3Block(const F32ConvStore &out, int image0, int image, int pixel, int first, int N, int lk, int e0, bool live, bool near)
      : positions(out.positions), N(N - first), lk(lk), e0(e0), live(live), near(near)
   {
      const long long from = (long long)image0 * out.Cout * out.positions + (long long)(out.first + first) * out.positions;
      Y = (float *)uniform((long long)(out.Y + from));
      R = out.R ? (const float *)uniform((long long)(out.R + from)) : nullptr;
      B = out.bias ? (const float *)uniform((long long)(out.bias + out.first + first)) : nullptr;
      at = (long long)(image - image0) * out.Cout * out.positions + pixel + (long long)lk * 4 * out.positions;
   }
   __device__ __forceinline__ int channel(int e) const { return e0 * 2 + e / 4 * 8 + e % 4; } // that lane half 0 holds
   // what(e, byte offset of this lane, F32_OUTSIDE where there is no result, and of the channel) for every element
   template <typename F>
   __device__ __forceinline__ void for_each(F &&what) const
   {
      const int lane = live ? (int)at * 4 : F32_OUTSIDE;
      if (N >= 32) {
#pragma unroll
         for (int e = 0; e < E; ++e)
            what(e, lane, channel(e) * positions * 4);
      } else {
#pragma unroll
         for (int g = 0; g < E; g += 4)
            if (channel(g) < N) {
#pragma unroll
               for (int e = g; e < g + 4; ++e)
                  what(e, channel(e) + lk * 4 < N ? lane : F32_OUTSIDE, channel(e) * positions * 4);
            }
      }
   }
   __device__ __forceinline__ void load(float (&bias)[E], float (&residual)[E]) const
   {
#pragma unroll
      for (int e = 0; e < E; ++e)
         bias[e] = residual[e] = 0.0f;
      if (B) {
#pragma unroll
         for (int e = 0; e < E; ++e)
            bias[e] = f32_bounded_read(B, lk * 16 + channel(e) * 4, N * 4);
      }
      if (R) {
         if (near) {
            for_each([&](int e, int lane, int scalar) { residual[e] = f32_buffer_read(R, lane, scalar); });
         } else if (live) {
#pragma unroll
            for (int e = 0; e < E; ++e)
               if (channel(e) + lk * 4 < N)
                  residual[e] = R[at + (long long)channel(e) * positions];
         }
      }
   }
   template <bool PLAIN>
   __device__ __forceinline__ void store(float (&v)[E], const PostChain &chain) const
   {
      if constexpr (PLAIN) {
         if (chain.count) {
#pragma unroll
            for (int e = 0; e < E; ++e)
               v[e] = v[e] > 0.0f ? v[e] : 0.0f;
         }
      } else if (chain.count != 0) {
         // one copy of the activations' code for four elements
#pragma unroll 1
         for (int g = 0; g < E; g += 4) {
            float four[4];
#pragma unroll
            for (int e = 0; e < E; ++e)
               four[e % 4] = e < 4 || g == e / 4 * 4 ? v[e] : four[e % 4];
            f32_activate_all<4>(four, chain);
#pragma unroll
            for (int e = 0; e < E; ++e)
               v[e] = g == e / 4 * 4 ? four[e % 4] : v[e];
         }
      }
      if (near) {
         Conv3x3Block again = *this;
         forget(again.positions); // the channels' offsets are worked out here: kept from the residual's loads they are spilled
         again.for_each([&](int e, int lane, int scalar) { f32_buffer_store(v[e], Y, lane, scalar); });
      } else if (live) {
#pragma unroll
         for (int e = 0; e < E; ++e)
            if (channel(e) + lk * 4 < N)
               Y[at + (long long)channel(e) * positions] = v[e];
      }
   }
};

// CS channels per slab; lane half lk multiplies the channels from lk * CS / 2 on, kernel position by kernel position.
template <int BM, int BN, int CS, int PLANE, int WVEC>
struct F32Conv3x3Shape {
   static constexpr int HALF = CS / 2 * 9;                      // k per lane half and slab
   static constexpr int PITCH = CS == 8 ? 76 : 38;              // of a weight row in LDS: the rows of a fragment start in different banks
   static constexpr int READ = CS == 8 ? 4 : 2;                 // floats of a weight row that a lane reads at once
   static constexpr int PATCH = CS * PLANE + 32;                // the second half of the channels starts 32 banks on
   static constexpr int WEIGHTS = (BN * PITCH + 64 * WVEC - 1) / (64 * WVEC) * 64 * WVEC;
   static constexpr int STAGE = (PATCH + WEIGHTS + 3) / 4 * 4;
   static constexpr int CHUNKS = PLANE / 64;                    // load instructions per channel
   static constexpr int WLOADS = WEIGHTS / (64 * WVEC);         // load instructions per slab of weights
   static_assert(PLANE % 64 == 0 && (WVEC == 1 || PITCH % 4 == 0), "whole load instructions");
};

// Two slabs in LDS, the next on its way while one is multiplied (2304 cycles of MFMAs for 32 x 32 wave tiles), and several workgroups per CU
// that cover each other's trips to memory and barriers.  WAVES_K waves share a wave tile, each multiplying every WAVES_K-th step of
// a slab: where there are few tiles, smaller ones keep as many matrix cores busy.
template <int BM, int BN, int WAVES_M, int WAVES_N, int WAVES_K, int CS, int PLANE, int WVEC, bool PLAIN>
__global__ __launch_bounds__(256, 2) void f32_conv3x3_kernel(F32Conv3x3 a, F32ConvStore out, TileOrder order, int first_tile, int places_at)
{
   typedef F32Conv3x3Shape<BM, BN, CS, PLANE, WVEC> S;
   constexpr int TM = BM / WAVES_M, TN = BN / WAVES_N, MT = TM / 32, NT = TN / 32;
   // Waves that share a tile wait for their loads: bounds worked out again before each slab's cost more than their spills (2 images of 25 x 25, 128 -> 66 channels
   // 16.8 us against 15.9).  With a tile each they are what a slab's issue waits for.
   constexpr bool FORGET = WAVES_K == 1;
   constexpr int OWN = 16 / WAVES_K; // of a block's 16 elements per lane, those this wave finishes
   static_assert(WAVES_M * WAVES_N * WAVES_K == 4 && TM % 32 == 0 && TN % 32 == 0, "four waves of 32 x 32 blocks");
   extern __shared__ __attribute__((aligned(16))) float f32_lds[];
   const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
   const int wk = wave % WAVES_K, wm = wave / WAVES_K / WAVES_N, wn = wave / WAVES_K % WAVES_N, lk = lane >> 5, c = lane & 31;
   const int wave_id = wave;
   int tm, tn, z;
   order.place(first_tile + blockIdx.x, tm, tn, z);
   a.X += z * a.group;
   a.W += (long long)z * a.N * a.K;
   out.select_batch(z);
   const int m0 = tm * BM, n0 = tn * BN;
   const int VW = a.OW + 2, VH = a.OH + 2;
   auto quotient = [](int n, const Divisor31 &by) { return (int)by.over((unsigned)n); };

   // where the patch begins
   const int line0 = quotient(m0, a.by_ow), image0 = quotient(line0, a.by_oh);
   const int row0 = line0 - image0 * a.OH; // of image0, padding row 0 first
   const char *base = (const char *)uniform((long long)(a.X + image0 * a.image));
   const int plane_bytes = a.H * a.Wd * 4;
   // bytes from `base` of the patch's positions, of channel 0: the waves load a channel each, all its positions, and work out a part of them
   int *const places = (int *)f32_lds + places_at;
#pragma unroll
   for (int q0 = 0; q0 < S::CHUNKS; q0 += 4) {
      const int q = q0 + wave;
      if (q < a.chunks) {
         const int f = q * 64 + lane, vr = quotient(f, a.by_vw), ix = f - vr * VW - a.pad_w;
         const int on = row0 + vr, image = quotient(on, a.by_vh), iy = on - image * VH - a.pad_h;
         const bool inside = (unsigned)ix < (unsigned)a.Wd && (unsigned)iy < (unsigned)a.H && image0 + image < a.images;
         places[f] = inside ? (int)((image * a.image + (long long)iy * a.Wd + ix) * 4) : F32_OUTSIDE;
      }
   }
   // the weights of this tile: rows past N and the gaps between rows read as zero
   constexpr int LDW = (S::WLOADS + 3) / 4;
   const char *weights = (const char *)uniform((long long)(a.W + (long long)n0 * a.K));
   int weight_at[LDW];
   auto weight_place = [&](int i, int &row, int &k) {
      const int f = ((i * 4 + wave) * 64 + lane) * WVEC;
      row = f / S::PITCH;
      k = f - row * S::PITCH;
   };
#pragma unroll
   for (int i = 0; i < LDW; ++i) {
      int row, k;
      weight_place(i, row, k);
      weight_at[i] = n0 + row < a.N && k < 2 * S::HALF ? (row * a.K + k) * 4 : F32_OUTSIDE;
   }

   const int slabs = CS == 4 ? 1 : (a.C + CS - 1) / CS; // slabs of 4 channels are for layers that have no more
   auto issue_weights = [&](int s, int stage) {
      float *lds = f32_lds + stage * S::STAGE;
      const bool whole = (s + 1) * CS <= a.C;
      int wave = wave_id;
      if constexpr (FORGET)
         forget(wave);
#pragma unroll
      for (int i = 0; i < LDW; ++i) {
         if (i * 4 + wave < S::WLOADS) {
            int at = weight_at[i];
            if (!whole) { // k past the last channel are the next row's
               int row, k;
               weight_place(i, row, k);
               at = s * CS * 9 + k < a.K ? at : F32_OUTSIDE;
            }
            f32_buffer_load<WVEC>((lds_void_t *)(lds + S::PATCH + (i * 4 + wave) * 64 * WVEC), weights + (long long)s * CS * 9 * 4, at);
         }
      }
   };
   issue_weights(0, 0);
   __builtin_amdgcn_s_waitcnt(0xc07f); // lgkmcnt(0)
   __builtin_amdgcn_s_barrier();
   __builtin_amdgcn_sched_barrier(0);
   int patch_at[S::CHUNKS];
#pragma unroll
   for (int q = 0; q < S::CHUNKS; ++q)
      patch_at[q] = q < a.chunks ? places[q * 64 + lane] : F32_OUTSIDE;
   auto issue_patch = [&](int s, int stage) {
      float *lds = f32_lds + stage * S::STAGE;
      int wave = wave_id, chunks = a.chunks;
      if constexpr (FORGET)
         forget(wave), forget(chunks);
      // channels wave, wave + 4
#pragma unroll
      for (int h = 0; h < CS; h += 4) {
         const int ch = h + wave;
         const bool there = s * CS + ch < a.C;
         float *to = lds + ch * PLANE + (ch >= CS / 2 ? 32 : 0);
         const int offset = there ? (s * CS + ch) * plane_bytes : 0;
#pragma unroll
         for (int q = 0; q < S::CHUNKS; ++q)
            if (q < chunks)
               f32_buffer_load<1>((lds_void_t *)(to + q * 64), base, there ? patch_at[q] : F32_OUTSIDE, offset);
      }
   };
   issue_patch(0, 0);

   // this lane's pixels in the patch, one address per kernel row, and its weights
   int pixel[MT][3];
   // Bias and residual are on their way with the first slab's loads (behind the loop they were four trips to memory in a row) and wait in
   // registers: as the start of the sums they would be rounded with every product (bias of 100, 64 channels: 4.2e-7 of the result against 2.4e-8).
   v16f acc[MT][NT];
   float bias[MT][NT][OWN], residual[MT][NT][OWN]; // of the elements that this wave finishes
   int image_of[MT], pixel_of[MT];
   auto block = [&](int i, int j) {
      return Conv3x3Block<OWN>(out, image0, image_of[i], pixel_of[i], n0 + wn * TN + j * 32, a.N, lk, wk * OWN, m0 + wm * TM + i * 32 + c < a.M, a.near);
   };
#pragma unroll
   for (int i = 0; i < MT; ++i) {
      const int m = m0 + wm * TM + i * 32 + c, mm = m < a.M ? m : a.M - 1;
      const int line = quotient(mm, a.by_ow), image = quotient(line, a.by_oh);
      const int vr = (image - image0) * VH + line - image * a.OH - row0;
      image_of[i] = image, pixel_of[i] = mm - image * out.positions;
#pragma unroll
      for (int ky = 0; ky < 3; ++ky)
         pixel[i][ky] = (vr + ky) * VW + mm - line * a.OW + lk * (CS / 2 * PLANE + 32);
#pragma unroll
      for (int j = 0; j < NT; ++j) {
         block(i, j).load(bias[i][j], residual[i][j]);
#pragma unroll
         for (int e = 0; e < 16; ++e)
            acc[i][j][e] = 0.0f;
      }
   }
   const int weight = S::PATCH + (wn * TN + c) * S::PITCH + lk * S::HALF;

   // READ k at a time; the fragments of the next ones are read while these are multiplied
   typedef float part __attribute__((ext_vector_type(S::READ)));
   part w[2][NT];
   float x[2][MT][S::READ];
   auto multiply = [&](auto stage) {
      const float *lds = f32_lds + decltype(stage)::value * S::STAGE;
      constexpr int STEPS = S::HALF / S::READ;
      auto read = [&](auto number, auto set) {
         constexpr int to = decltype(set)::value, g = decltype(number)::value * S::READ;
#pragma unroll
         for (int j = 0; j < NT; ++j)
            w[to][j] = *(const part *)(lds + weight + j * 32 * S::PITCH + g);
#pragma unroll
         for (int i = 0; i < MT; ++i)
#pragma unroll
            for (int u = 0; u < S::READ; ++u)
               x[to][i][u] = lds[pixel[i][(g + u) % 9 / 3] + (g + u) / 9 * PLANE + (g + u) % 3];
      };
      // the steps of wave p of those that share a tile
      auto steps_of = [&](auto pc) {
         constexpr int p = decltype(pc)::value, COUNT = (STEPS - p + WAVES_K - 1) / WAVES_K;
         read(std::integral_constant<int, p>{}, std::integral_constant<int, 0>{});
         static_for<COUNT>([&](auto gc) {
            constexpr int g = decltype(gc)::value, set = g % 2;
            __builtin_amdgcn_sched_barrier(0);
            if constexpr (g + 1 < COUNT)
               read(std::integral_constant<int, p + (g + 1) * WAVES_K>{}, std::integral_constant<int, set ^ 1>{});
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int u = 0; u < S::READ; ++u)
#pragma unroll
               for (int i = 0; i < MT; ++i)
#pragma unroll
                  for (int j = 0; j < NT; ++j)
                     acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(w[set][j][u], x[set][i][u], acc[i][j], 0, 0, 0);
         });
      };
      static_for<WAVES_K>([&](auto pc) {
         if (WAVES_K == 1 || wk == decltype(pc)::value)
            steps_of(pc);
      });
   };

   auto turn = [&](int s, auto stage) {
      wait_vmcnt<0>();
      __builtin_amdgcn_s_barrier(); // slab s has landed for every wave, and every wave has read slab s - 1
      __builtin_amdgcn_sched_barrier(0);
      if (s + 1 < slabs)
         issue_patch(s + 1, decltype(stage)::value ^ 1), issue_weights(s + 1, decltype(stage)::value ^ 1);
      __builtin_amdgcn_sched_barrier(0);
      multiply(stage);
      __builtin_amdgcn_s_waitcnt(0xc07f); // lgkmcnt(0)
      __builtin_amdgcn_sched_barrier(0);
   };
   for (int s = 0; s < slabs; s += 2) {
      turn(s, std::integral_constant<int, 0>{});
      if (s + 1 < slabs)
         turn(s + 1, std::integral_constant<int, 1>{});
   }

   // Waves that share a tile: each leaves the elements it does not finish in LDS and adds up the others' parts of its own.
   static_assert(WAVES_K == 1 || (MT == 1 && NT == 1), "one block per wave where waves share it");
   if constexpr (WAVES_K > 1) {
      __syncthreads();
      float *parts = f32_lds + (wave - wk) * 1024;
#pragma unroll
      for (int e = 0; e < 16; ++e)
         parts[wk * 1024 + e * 64 + lane] = acc[0][0][e];
      __syncthreads();
      static_for<WAVES_K>([&](auto pc) {
         constexpr int p = decltype(pc)::value;
         if (wk == p) {
#pragma unroll
            for (int e = p * OWN; e < (p + 1) * OWN; ++e)
#pragma unroll
               for (int o = 0; o < WAVES_K; ++o)
                  if (o != p)
                     acc[0][0][e] += parts[o * 1024 + e * 64 + lane];
         }
      });
   }
   static_for<WAVES_K>([&](auto pc) {
      constexpr int p = decltype(pc)::value;
      if (WAVES_K == 1 || wk == p) {
#pragma unroll
         for (int i = 0; i < MT; ++i)
#pragma unroll
            for (int j = 0; j < NT; ++j) {
               float v[OWN];
#pragma unroll
               for (int o = 0; o < OWN; ++o)
                  v[o] = (acc[i][j][p * OWN + o] + bias[i][j][o]) + residual[i][j][o];
               block(i, j).template store<PLAIN>(v, out.chain);
            }
      }
   });
}

template <int BM, int BN, int WAVES_M, int WAVES_N, int WAVES_K, int CS, int PLANE, int WVEC>
static int launch_f32_conv3x3_as(hipStream_t stream, const F32Conv3x3 &a, const F32ConvStore &out, int group)
{
   const int tiles_m = (a.M + BM - 1) / BM, tiles_n = (a.N + BN - 1) / BN;
   if ((long long)tiles_m * tiles_n > 0x7fffffffLL)
      return fail(SOFIE_HIP_ERR_INVALID, "fp32 convolution: too many tiles");
   constexpr size_t stage = sizeof(float) * F32Conv3x3Shape<BM, BN, CS, PLANE, WVEC>::STAGE, parts = WAVES_K > 1 ? 4 * 1024 * sizeof(float) : 0;
   const size_t slabs = std::max(stage * (a.C > CS ? 2 : 1), parts), smem = slabs + PLANE * sizeof(int);
   auto go = [&](auto plain) {
      auto kern = f32_conv3x3_kernel<BM, BN, WAVES_M, WAVES_N, WAVES_K, CS, PLANE, WVEC, decltype(plain)::value>;
      static bool configured[64] = {};
      if (int st = configure_lds_once(kern, std::max(stage * 2, parts) + PLANE * sizeof(int), configured))
         return st;
      const TileOrder order(tiles_m, tiles_n, 4, group);
      in_launches(order.workgroups(group), 256, [&](int first, unsigned count) {
         launch_kernel(kern, dim3(count, 1, order.depth(group)), dim3(256), smem, stream, a, out, order, first, (int)(slabs / sizeof(int)));
      });
      return launch_status("f32_conv3x3_kernel");
   };
   return conv3x3_plain(out.chain) ? go(std::true_type{}) : go(std::false_type{});
}

} // namespace sofie_hip
