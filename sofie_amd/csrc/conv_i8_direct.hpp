// int8 convolution of a small layer over NHWC input (channels per group a multiple of 8): the direct kernel of mfma8_direct.hpp with the rows of A cut from the image on their way
// into the registers.  A workgroup owns one small tile of output pixels and channels, its waves split the reduction, and what a layer costs is one trip to memory and the
// instructions around it: the general loop (mfma8_staged.hpp) takes a slab of 128 bytes of k after the other through LDS, four waves on 64 x 64 tiles of which a few small images make
// 60 for 256 CUs.
#pragma once
#include "mfma8_staged.hpp"

namespace sofie_hip {

// Row m is an output pixel, k = tap * Cg + channel; a chunk of 16 bytes is 16 / PIECE pieces that each lie inside one tap.
template <int PIECE_>
struct DirectConvRows {
   static constexpr int PIECE = PIECE_;
   const int8_t *X; // first channel of the group
   int rows, H, W, C, stride_h, stride_w, pad_h0, pad_w0, dil_h, dil_w, K;
   Divisor31 by_plane, by_ow, by_cg, by_kw; // output pixels of an image and of a row, channels, kernel columns
   struct place {
      int off, ih0, iw0; // of channel 0 at (ih0, iw0), in bytes from X: may be negative
   };
   __device__ __forceinline__ place place_of(int row) const
   {
      const int m = row < rows ? row : rows - 1, n = (int)by_plane.over((unsigned)m), rem = m - n * (int)by_plane.d, oh = (int)by_ow.over((unsigned)rem), ow = rem - oh * (int)by_ow.d;
      place p;
      p.ih0 = oh * stride_h - pad_h0;
      p.iw0 = ow * stride_w - pad_w0;
      p.off = ((n * H + p.ih0) * W + p.iw0) * C;
      return p;
   }
   typedef int piece_t __attribute__((ext_vector_type(PIECE / 4), aligned(PIECE)));
   union chunk_t {
      v4i v;
      piece_t p[16 / PIECE];
   };
   // the chunk at k of MB rows, zero outside the image and from K on
   template <int MB>
   __device__ __forceinline__ void fetch(const place (&at)[MB], int k, v4i (&out)[MB]) const
   {
      chunk_t c[MB];
#pragma unroll
      for (int q = 0; q < 16 / PIECE; ++q) {
         const int kk = k + q * PIECE, tap = (int)by_cg.over((unsigned)kk), ci = kk - tap * (int)by_cg.d, ky = (int)by_kw.over((unsigned)tap), kx = tap - ky * (int)by_kw.d;
         const int dy = ky * dil_h, dx = kx * dil_w, off = (dy * W + dx) * C + ci;
#pragma unroll
         for (int i = 0; i < MB; ++i) {
            const bool inside = kk < K && (unsigned)(at[i].ih0 + dy) < (unsigned)H && (unsigned)(at[i].iw0 + dx) < (unsigned)W;
            c[i].p[q] = *(const piece_t *)(inside ? X + (ptrdiff_t)(at[i].off + off) : (const int8_t *)conv_zero_page);
         }
      }
#pragma unroll
      for (int i = 0; i < MB; ++i)
         out[i] = c[i].v;
   }
};

// Two steps of 128 bytes of k a wave are on their way at once; Kp: bytes of a row of weights (a multiple of 16, from K on zero).
template <int PIECE, int MB, int NB, int W, class EPI>
__global__ __launch_bounds__(W * 64) void conv_i8_direct_kernel(DirectConvRows<PIECE> A, const int8_t *Wp, int Kp, int M, int N, EPI ep, TileOrder order, int first_tile)
{
   constexpr int STEP = 128, TM = MB * 16, TN = NB * 16, UNROLL = 2;
   typedef DirectI8 MMA;
   __shared__ __attribute__((aligned(16))) int part[W][TM][TN + 4];
   int tm, tn;
   order.place(first_tile + blockIdx.x, tm, tn);
   const int m0 = tm * TM, n0 = tn * TN;
   const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lk = lane >> 4, c = lane & 15;
   typename DirectConvRows<PIECE>::place at[MB];
   const int8_t *rb[NB]; // rows past the edge re-read the last one
#pragma unroll
   for (int i = 0; i < MB; ++i)
      at[i] = A.place_of(m0 + i * 16 + c);
#pragma unroll
   for (int j = 0; j < NB; ++j)
      rb[j] = Wp + (size_t)(n0 + j * 16 + c < N ? n0 + j * 16 + c : N - 1) * (size_t)Kp;
   MMA::acc_t acc[MB][NB];
#pragma unroll
   for (int i = 0; i < MB; ++i)
#pragma unroll
      for (int j = 0; j < NB; ++j)
         acc[i][j] = MMA::acc_t{0, 0, 0, 0};
   DirectStore<MMA, MB, NB, W, EPI> store(m0, n0, M, N);
   const int steps = (A.K + STEP - 1) / STEP;
   for (int s0 = wave; s0 < steps; s0 += W * UNROLL) {
      v4i fa[UNROLL][2][MB], fb[UNROLL][2][NB];
#pragma unroll
      for (int u = 0; u < UNROLL; ++u) {
         if (s0 + u * W < steps) {
            const int k = (s0 + u * W) * STEP + lk * 32;
#pragma unroll
            for (int h = 0; h < 2; ++h) {
#pragma unroll
               for (int j = 0; j < NB; ++j)
                  fb[u][h][j] = *(const v4i_unaligned *)(k + 16 * h < Kp ? rb[j] + k + 16 * h : (const int8_t *)conv_zero_page);
               A.template fetch<MB>(at, k + 16 * h, fa[u][h]);
            }
         }
      }
      if (s0 == wave)
         store.ask(ep);
#pragma unroll
      for (int u = 0; u < UNROLL; ++u)
         if (s0 + u * W < steps) {
#pragma unroll
            for (int i = 0; i < MB; ++i)
#pragma unroll
               for (int j = 0; j < NB; ++j) {
                  const v4i n_side[2] = {fb[u][0][j], fb[u][1][j]}, m_side[2] = {fa[u][0][i], fa[u][1][i]};
                  acc[i][j] = MMA::mma(n_side, m_side, acc[i][j]);
               }
         }
   }
   if (wave >= steps)
      store.ask(ep);
   store.store(ep, acc, part, wave, lane);
}

template <int PIECE, int MB, int NB, int W, class EPI>
static int launch_conv_i8_direct(const LaunchCfg &lc, const DirectConvRows<PIECE> &A, const int8_t *Wp, int M, int N, int Kp, const EPI &ep)
{
   const int tiles_m = (M + MB * 16 - 1) / (MB * 16), tiles_n = (N + NB * 16 - 1) / (NB * 16);
   const long long nwg = (long long)tiles_m * tiles_n;
   if (nwg > 0x7fffffffLL)
      return fail(SOFIE_HIP_ERR_INVALID, "int8 convolution: too many tiles");
   const TileOrder order(tiles_m, tiles_n, lc.swizzle);
   in_launches(nwg, W * 64, [&](int first, unsigned count) {
      launch_kernel((conv_i8_direct_kernel<PIECE, MB, NB, W, EPI>), dim3(count), dim3(W * 64), 0, lc.stream, A, Wp, Kp, M, N, ep, order, first);
   });
   return launch_status("conv_i8_direct_kernel");
}

} // namespace sofie_hip
