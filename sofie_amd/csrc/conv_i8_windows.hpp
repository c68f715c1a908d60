// int8 convolution over FEW input channels of an NCHW image, any image and output size: the general form of
// conv_i8_few_channels_kernel, which stores whole 64-channel rows of 64-pixel groups.  Same reduction order, (channel, ky) pairs of
// four kx positions each, same windows; here a window is cut from an unaligned 8-byte load, a wave takes 16 pixels at a time
// (so that a handful of small images still spreads over the chip), the last pixels may be missing, and the results go out
// straight from the accumulators: a lane holds 4 consecutive channels of one pixel, the four lanes of a pixel 16 of them.
#pragma once
#include "conv_i8_few_channels.hpp"
#include "mfma8_direct.hpp"

namespace sofie_hip {

// NT: blocks of 16 output channels.
template <class EPI, int NT>
__global__ __launch_bounds__(256) void conv_i8_windows_kernel(FewChannelConv g, int stride_w, const int8_t *__restrict__ Wp, int Kp, EPI ep, int M, int N, int ngroups, int kh_mul, Divisor31 by_plane, Divisor31 by_ow)
{
   typedef uint64_t u64_unaligned __attribute__((aligned(1)));
   __shared__ v4i wfrag[NT * 16 * 4]; // [column][quarter of the reduction]: 16 bytes each
   const int t = threadIdx.x, lane = t & 63;
   const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
   const int c = lane & 15, lk = lane >> 4;
   const int npairs = g.Cg * g.kh;

   auto channel_of = [&](int pair) { return pair * kh_mul >> 8; }; // pair / kh for the 16 pairs there may be
   // ---- weights, re-ordered from k = (ky * kw + kx) * Cg + channel: sixteen bytes of a thread on their way at once, those that are none read as the first and dropped
   for (int e = t; e < NT * 16 * 4; e += 256) {
      const int col = e >> 2, q = e & 3;
      uint8_t v[4][4];
#pragma unroll
      for (int p = 0; p < 4; ++p) {
         const int pair = q * 4 + p, ch = channel_of(pair), ky = pair - ch * g.kh;
#pragma unroll
         for (int kx = 0; kx < 4; ++kx)
            v[p][kx] = (uint8_t)Wp[pair < npairs && kx < g.kw && col < N ? (size_t)col * Kp + (ky * g.kw + kx) * g.Cg + ch : 0];
      }
      __builtin_amdgcn_sched_barrier(0);
      uint32_t w[4] = {0, 0, 0, 0};
#pragma unroll
      for (int p = 0; p < 4; ++p)
#pragma unroll
         for (int kx = 0; kx < 4; ++kx)
            w[p] |= q * 4 + p < npairs && kx < g.kw && col < N ? (uint32_t)v[p][kx] << (8 * kx) : 0u;
      wfrag[e] = v4i{(int)w[0], (int)w[1], (int)w[2], (int)w[3]};
   }
   // ---- the lane's four pairs: plane and row offset, and the row distance (a pair past the end never lies inside the image)
   int pair_off[4], pair_dy[4];
#pragma unroll
   for (int q = 0; q < 4; ++q) {
      const int pair = lk * 4 + q, ch = channel_of(pair), ky = pair - ch * g.kh;
      pair_off[q] = (ch * g.H + ky * g.dil_h) * g.W;
      pair_dy[q] = pair < npairs ? ky * g.dil_h : -(1 << 30); // above any image (rows of 8 bytes or more: at most 2^28 of them)
   }
   typename EPI::template col_params<4> prm[NT];
#pragma unroll
   for (int j = 0; j < NT; ++j)
      ep.template load_params<4>(j * 16 + lk * 4 < N ? j * 16 + lk * 4 : N - 1, prm[j]);
   __syncthreads();
   v4i fb[NT];
#pragma unroll
   for (int j = 0; j < NT; ++j)
      fb[j] = wfrag[(j * 16 + c) * 4 + lk];

   // the windows of a group are requested one group ahead
   uint64_t chunk[4];
   bool ok[4];
   int shift;
   auto request = [&](int grp) {
      const int m = grp * 16 + c < M ? grp * 16 + c : M - 1;
      const int img = (int)by_plane.over((unsigned)m), r = m - img * (int)by_plane.d, oh = (int)by_ow.over((unsigned)r), ow = r - oh * g.OW;
      const int ih0 = oh * g.stride_h - g.pad_h0, iw0 = ow * stride_w - g.pad_w0;
      // the 8 bytes lie inside the row; `shift` moves the window down (positive) or up
      const int cs = iw0 < 0 ? 0 : iw0 > g.W - 8 ? g.W - 8 : iw0;
      shift = 8 * (iw0 - cs);
      const int8_t *row = g.X + (long long)img * g.img_stride + (ih0 * g.W + cs);
#pragma unroll
      for (int q = 0; q < 4; ++q) {
         ok[q] = (unsigned)(ih0 + pair_dy[q]) < (unsigned)g.H;
         chunk[q] = *(const u64_unaligned *)(ok[q] ? row + pair_off[q] : g.X);
      }
   };
   const int stride = gridDim.x * 4;
   int grp = blockIdx.x * 4 + wave;
   if (grp < ngroups)
      request(grp);
   for (; grp < ngroups; grp += stride) {
      v4i fa;
#pragma unroll
      for (int q = 0; q < 4; ++q) {
         // a window that lies wholly beside the row is all zeros (shifts of 64 and more)
         const uint64_t moved = shift >= 64 || shift <= -64 ? 0 : shift >= 0 ? chunk[q] >> shift : chunk[q] << -shift;
         fa[q] = ok[q] ? (int)(uint32_t)moved : 0;
      }
      if (grp + stride < ngroups)
         request(grp + stride);
      v4i acc[NT];
#pragma unroll
      for (int j = 0; j < NT; ++j)
         acc[j] = __builtin_amdgcn_mfma_i32_16x16x64_i8(fb[j], fa, v4i{0, 0, 0, 0}, 0, 0, 0);
      const int m = grp * 16 + c;
      if (m < M)
         ep.dispatch([&](auto mode) {
#pragma unroll
            for (int j = 0; j < NT; ++j)
               if (j * 16 + lk * 4 < N)
                  store_four_columns<decltype(mode)::value>(ep, prm[j], acc[j], m, j * 16 + lk * 4, N);
         });
   }
}

inline bool conv_i8_windows_applies(const FewChannelConv &g, int N)
{
   return g.kw <= 4 && g.Cg * g.kh <= 16 && g.W >= 8 && N <= 64;
}

template <class EPI>
static int launch_conv_i8_windows(const LaunchCfg &lc, const FewChannelConv &g, int stride_w, const int8_t *Wp, int M, int N, int Kp, const EPI &ep)
{
   const int ngroups = (M + 15) / 16;
   // up to 16 waves per CU, each with its next group of windows on the way
   int grid = (ngroups + 3) / 4;
   if (grid > 1024)
      grid = 1024;
   auto go = [&](auto nt) {
      constexpr int NT = decltype(nt)::value;
      launch_kernel((conv_i8_windows_kernel<EPI, NT>), dim3((unsigned)grid), dim3(256), 0, lc.stream, g, stride_w, Wp, Kp, ep, M, N, ngroups,
                    (255 + g.kh) / g.kh, Divisor31((long long)g.OH * g.OW), Divisor31(g.OW));
      return launch_status("conv_i8_windows_kernel");
   };
   return N <= 16 ? go(std::integral_constant<int, 1>{}) : N <= 32 ? go(std::integral_constant<int, 2>{}) : go(std::integral_constant<int, 4>{});
}

} // namespace sofie_hip
