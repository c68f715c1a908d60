// The convolution over few input channels as a GEMM of one slab: every lane gathers the bytes of its own row (output pixel), the
// tile is multiplied from LDS (swizzled layout of lds_chunk_offset, 32x32 MFMA tiles) and stored.  The packed weights' rows are
// the MFMA's first operand and the pixels its second, so that a lane ends up holding 4 consecutive output channels of one pixel.
// Also here: what every launcher of the matrix-core kernels shares.
#pragma once
#include "mfma8_common.hpp"

namespace sofie_hip {

// KP: the padded reduction length.  OCC: waves per SIMD the register allocation leaves room for.
template <class MMA, int BM, int BN, int BK, int WAVES_M, int WAVES_N, class EPI, int KP, int OCC>
__global__ __launch_bounds__(WAVES_M *WAVES_N * 64, OCC) void mfma8_gather_kernel(GatherConvRowsT<KP> A, RowMajorRows Bt, int M, int N, EPI ep, TileOrder order)
{
   constexpr int NTHREADS = WAVES_M * WAVES_N * 64;
   constexpr int CPR = BK / 16;
   constexpr int TM = BM / WAVES_M, TN = BN / WAVES_N; // wave tile
   constexpr int MT = TM / 32, NT = TN / 32;           // 32x32 MFMA tiles per wave
   constexpr int B_LD = BN * CPR / NTHREADS;
   static_assert(BN * CPR % NTHREADS == 0, "tile must divide over the threads");
   static_assert(TM % 32 == 0 && TN % 32 == 0, "wave tile must be a multiple of 32x32");
   static_assert(BM == NTHREADS && BK == 64 && KP <= BK, "one row per thread of one 64-byte slab");
   typedef typename MMA::acc_t acc_t;
   typedef typename MMA::frag_t frag_t;

   extern __shared__ __attribute__((aligned(16))) int8_t smem[];
   int8_t *sA = smem;           // [BM*BK]
   int8_t *sB = smem + BM * BK; // [BN*BK]

   int tm, tn;
   order.place(blockIdx.x, tm, tn);
   const int m0 = tm * BM, n0 = tn * BN;
   const int t = threadIdx.x;
   const int lane = t & 63, wave = t >> 6;
   const int wm = wave / WAVES_N, wn = wave % WAVES_N;

   acc_t acc[MT][NT];
#pragma unroll
   for (int i = 0; i < MT; ++i)
#pragma unroll
      for (int j = 0; j < NT; ++j)
#pragma unroll
         for (int v = 0; v < 16; ++v)
            acc[i][j][v] = 0;

   const auto ref = A.ref_of(m0 + t, M);
   unsigned w[16];
#pragma unroll
   for (int i = 0; i < 16; ++i)
      w[i] = 0;
   // every load is issued unconditionally (a tap outside the image reads the first byte of the tensor instead and is
   // masked afterwards), so that the loads of a row are in flight together instead of one memory round trip per tap
   unsigned v[KP];
   unsigned ok_lo = 0, ok_hi = 0; // bit k: tap k lies inside the image
#pragma unroll
   for (int k = 0; k < KP; ++k) {
      const int ih = ref.ih0 + A.dy[k], iw = ref.iw0 + A.dx[k];
      const bool in = k < A.K && (unsigned)ih < (unsigned)A.H && (unsigned)iw < (unsigned)A.W; // k >= K: padding of the reduction
      if (k < 32)
         ok_lo |= in ? (1u << (k & 31)) : 0u;
      else
         ok_hi |= in ? (1u << (k & 31)) : 0u;
      const int8_t *p = in ? ref.origin + A.koff[k] : A.X;
      v[k] = (unsigned char)*p;
   }
#pragma unroll
   for (int k = 0; k < KP; ++k) {
      const unsigned bit = ((k < 32 ? ok_lo : ok_hi) >> (k & 31)) & 1u;
      w[k / 4] |= (bit ? v[k] : 0u) << (8 * (k % 4));
   }
#pragma unroll
   for (int c = 0; c < 4; ++c)
      *(v4i *)(sA + lds_chunk_offset<BK>(t, c)) = v4i{(int)w[4 * c], (int)w[4 * c + 1], (int)w[4 * c + 2], (int)w[4 * c + 3]};
#pragma unroll
   for (int i = 0; i < B_LD; ++i) {
      const int id = t + i * NTHREADS, row = id / CPR, k = id % CPR * 16;
      const int8_t *p = Bt.row(n0 + row < N ? n0 + row : N - 1) + k;
      *(v4i *)(sB + lds_chunk_offset<BK>(row, id % CPR)) = k < KP ? *(const v4i *)p : v4i{0, 0, 0, 0};
   }
   __syncthreads();

   const int lr = lane & 31, lk = lane >> 5;
#pragma unroll
   for (int ks = 0; ks < BK / MMA::KSTEP; ++ks) {
      frag_t fa[MT], fb[NT];
#pragma unroll
      for (int j = 0; j < NT; ++j)
#pragma unroll
         for (int c = 0; c < MMA::CHUNKS; ++c)
            fb[j].c[c] = *(const v4i *)(sB + lds_chunk_offset<BK>(wn * TN + j * 32 + lr, (ks * 2 + lk) * MMA::CHUNKS + c));
#pragma unroll
      for (int i = 0; i < MT; ++i)
#pragma unroll
         for (int c = 0; c < MMA::CHUNKS; ++c)
            fa[i].c[c] = *(const v4i *)(sA + lds_chunk_offset<BK>(wm * TM + i * 32 + lr, (ks * 2 + lk) * MMA::CHUNKS + c));
#pragma unroll
      for (int i = 0; i < MT; ++i)
#pragma unroll
         for (int j = 0; j < NT; ++j)
            acc[i][j] = MMA::mma(fb[j], fa[i], acc[i][j]);
   }

   __syncthreads(); // the slab is dead: the tile store reuses LDS, one region per wave
   char *wsm = (char *)smem + wave * tile_store_lds_bytes(TN);
   ep.dispatch([&](auto mode) {
      tile_store_via_lds<decltype(mode)::value, MT, NT>(ep, acc, m0 + wm * TM, n0 + wn * TN, M, N, lane, wsm);
   });
}

// One attribute call per kernel and device (it is far slower than a launch).
template <class KERN>
static int configure_lds_once(KERN kern, size_t smem, bool (&configured)[64])
{
   int dev = 0;
   SOFIE_HIP_CHECK(hipGetDevice(&dev));
   if (dev < 0 || dev >= 64 || !configured[dev]) {
      SOFIE_HIP_CHECK(hipFuncSetAttribute((const void *)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)smem));
      if (dev >= 0 && dev < 64)
         configured[dev] = true;
   }
   return SOFIE_HIP_OK;
}

// Tile choice: the largest one that still gives every one of the 256 CUs a workgroup.
inline int pick_tile(int M, int N, int force_tile)
{
   if (force_tile == 256 || force_tile == 128 || force_tile == 64)
      return force_tile;
   // any other request (the convolution's extra tile shapes) leaves the plain product to the heuristic
   auto tiles = [&](int bm, int bn) { return (long long)((M + bm - 1) / bm) * ((N + bn - 1) / bn); };
   // a tile wider than the matrix would spend its matrix-core time on columns that do not exist
   if (N > 128 && tiles(256, 256) >= 256)
      return 256;
   if (N > 64 && tiles(128, 128) >= 192)
      return 128;
   return 64;
}

// Convolution over few input channels as ONE launch: 256 x 64 tiles (one output pixel per thread in the gather), a single
// 64-byte slab.  Wp is the packed weight [N][Kp], Kp = the reduction length rounded up to 16, at most 64.
template <class EPI, int KP>
static int launch_mfma8_gather_kp(const LaunchCfg &lc, const GatherConvRows &a, const int8_t *Wp, int M, int N, const EPI &ep)
{
   constexpr int BM = 256, BN = 64, BK = 64;
   const int tiles_m = (M + BM - 1) / BM, tiles_n = (N + BN - 1) / BN;
   const long long nwg = (long long)tiles_m * tiles_n;
   if (nwg > 0x7fffffffLL)
      return fail(SOFIE_HIP_ERR_INVALID, "conv: too many tiles");
   constexpr size_t slab = (size_t)(BM + BN) * BK, store = 4 * (size_t)tile_store_lds_bytes(BN);
   constexpr size_t smem = slab > store ? slab : store;
   // three waves per SIMD (at most 170 registers; the kernel needs 168): each workgroup is one chain of memory round trips
   // (gather, weights, store), so the time goes down with the number of workgroups a CU holds (first layer of the benchmark CNN:
   // 74 us with two, 59 us with three; four would spill)
   auto kern = mfma8_gather_kernel<MfmaI8, BM, BN, BK, 4, 1, EPI, KP, 3>;
   static bool configured[64] = {};
   if (int st = configure_lds_once(kern, smem, configured))
      return st;
   GatherConvRowsT<KP> src;
   static_cast<GatherConvRows &>(src) = a;
   launch_kernel(kern, dim3((unsigned)nwg), dim3(256), smem, lc.stream, src, RowMajorRows{Wp, KP}, M, N, ep, TileOrder(tiles_m, tiles_n, 0));
   return launch_status("mfma8_gather_kernel");
}

// Convolution over few input channels as ONE launch: 256 x 64 tiles (one output pixel per thread in the gather), a single
// 64-byte slab.  Wp is the packed weight [N][Kp], Kp = the reduction length rounded up to 16, at most 64.
template <class EPI>
static int launch_mfma8_gather(const LaunchCfg &lc, const GatherConvRows &a, const int8_t *Wp, int M, int N, int Kp, const EPI &ep)
{
   if (a.K > Kp)
      return fail(SOFIE_HIP_ERR_INVALID, "conv: the gathered form needs a reduction of at most 64 bytes");
   switch (Kp) {
   case 16: return launch_mfma8_gather_kp<EPI, 16>(lc, a, Wp, M, N, ep);
   case 32: return launch_mfma8_gather_kp<EPI, 32>(lc, a, Wp, M, N, ep);
   case 48: return launch_mfma8_gather_kp<EPI, 48>(lc, a, Wp, M, N, ep);
   case 64: return launch_mfma8_gather_kp<EPI, 64>(lc, a, Wp, M, N, ep);
   default: return fail(SOFIE_HIP_ERR_INVALID, "conv: the gathered form needs a reduction of at most 64 bytes");
   }
}

} // namespace sofie_hip
