// int8 / FP8 products of few rows (or few tiles): no LDS on the way in.  A workgroup owns one small tile of Y and its W waves
// split the reduction; every fragment is loaded from memory into the registers the MFMA reads, UNROLL steps of 128 bytes of k
// ahead, and the partial tiles meet in LDS.  What such a product costs is the trip to memory for its operands, and one workgroup
// has its whole share of them (tens of KB) on the way at once; the ring kernels wait for a few KB at a time.  A tile has as few
// as 16 rows, where theirs have 64.  Rows may start at any byte: a chunk is one unaligned 16-byte load.
#pragma once
#include "mfma8_gemm_dma.hpp"

namespace sofie_hip {

typedef int v4i_unaligned __attribute__((ext_vector_type(4), aligned(1)));

// The 16 bytes of a row from k on, zero from K on.  Never reads outside the row's K bytes.
__device__ __forceinline__ v4i load_chunk_tail(const int8_t *row, int k, int K)
{
   if (k <= K - 16)
      return *(const v4i_unaligned *)(row + k);
   union {
      v4i v;
      unsigned long long q[2];
      int8_t b[16];
   } u;
   u.v = v4i{0, 0, 0, 0};
   if (k >= K)
      return u.v;
   if (K >= 16) {
      // the last 16 bytes of the row, shifted down to where k lies
      u.v = *(const v4i_unaligned *)(row + K - 16);
      const int drop = (k - K + 16) * 8; // bits; 8 .. 120
      if (drop >= 64) {
         u.q[0] = u.q[1] >> (drop - 64);
         u.q[1] = 0;
      } else {
         u.q[0] = (u.q[0] >> drop) | (u.q[1] << (64 - drop));
         u.q[1] >>= drop;
      }
      return u.v;
   }
#pragma unroll
   for (int i = 0; i < 16; ++i)
      if (k + i < K)
         u.b[i] = row[k + i];
   return u.v;
}

// Columns n..n+3 of row m from four accumulators, as a 4-element store where the row allows it.
template <int MODE, class EPI, class ACC>
__device__ __forceinline__ void store_four_columns(const EPI &ep, const typename EPI::template col_params<4> &prm, const ACC &v, int m, int n, int N)
{
   constexpr int ESZ = EPI::template out_bytes<MODE>();
   uint32_t w4[4];
   ep.template pack4<MODE, 4>(prm, 0, v[0], v[1], v[2], v[3], w4);
   if (ep.rows_vectorizable() && n + 4 <= N) {
      char *y = ep.out_base() + ep.out_index(m, n) * ESZ;
      if constexpr (ESZ == 1)
         *(uint32_t *)y = w4[0];
      else if constexpr (ESZ == 2)
         *(uint2 *)y = make_uint2(w4[0], w4[1]);
      else
         *(uint4 *)y = make_uint4(w4[0], w4[1], w4[2], w4[3]);
   } else {
#pragma unroll
      for (int i = 0; i < 4; ++i)
         if (n + i < N) {
            char *y = ep.out_base() + ep.out_index(m, n + i) * ESZ;
            if constexpr (ESZ == 1)
               *y = (char)(w4[0] >> (8 * i));
            else if constexpr (ESZ == 2)
               *(uint16_t *)y = (uint16_t)(w4[i / 2] >> (16 * (i % 2)));
            else
               *(uint32_t *)y = w4[i];
         }
   }
}

// One step of 128 bytes of k on a 16 x 16 block: lane (lk = lane / 16, c = lane % 16) holds bytes 32 lk .. 32 lk + 31 of row c of either
// operand.  The n side goes first, so that a lane ends up with 4 consecutive columns of one row.
struct DirectI8 {
   typedef v4i acc_t;
   typedef int elem_t;
   static __device__ __forceinline__ acc_t mma(const v4i (&n_side)[2], const v4i (&m_side)[2], acc_t c)
   {
      c = __builtin_amdgcn_mfma_i32_16x16x64_i8(n_side[0], m_side[0], c, 0, 0, 0);
      return __builtin_amdgcn_mfma_i32_16x16x64_i8(n_side[1], m_side[1], c, 0, 0, 0);
   }
};
typedef float v4f32 __attribute__((ext_vector_type(4)));
struct DirectF8 {
   typedef v4f32 acc_t;
   typedef float elem_t;
   static __device__ __forceinline__ acc_t mma(const v4i (&n_side)[2], const v4i (&m_side)[2], acc_t c)
   {
      const v8i a = {n_side[0][0], n_side[0][1], n_side[0][2], n_side[0][3], n_side[1][0], n_side[1][1], n_side[1][2], n_side[1][3]};
      const v8i b = {m_side[0][0], m_side[0][1], m_side[0][2], m_side[0][3], m_side[1][0], m_side[1][1], m_side[1][2], m_side[1][3]};
      return __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(a, b, c, 0, 0, 0, 0, 0, 0);
   }
};

template <class MMA, int MB, int NB, int W, int UNROLL, class EPI>
__global__ __launch_bounds__(W * 64) void mfma8_direct_kernel(RowMajorRows A, RowMajorRows Bt, int M, int N, int K, EPI ep, int tiles_m, int tiles_n, int sw,
                                                              int first_tile)
{
   constexpr int STEP = 128, TM = MB * 16, TN = NB * 16, PITCH = TN + 4;
   typedef typename MMA::acc_t acc_t;
   typedef typename MMA::elem_t elem_t;
   __shared__ __attribute__((aligned(16))) elem_t part[W][TM][PITCH];
   int tm, tn;
   tile_of_block(first_tile + blockIdx.x, tiles_m * tiles_n, tiles_m, tiles_n, sw, tm, tn);
   const int m0 = tm * TM, n0 = tn * TN;
   const int lane = threadIdx.x & 63;
   const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
   const int lk = lane >> 4, c = lane & 15;
   const int8_t *ra[MB], *rb[NB]; // rows past the edge re-read the last one (their results are not stored)
#pragma unroll
   for (int i = 0; i < MB; ++i)
      ra[i] = A.row(m0 + i * 16 + c < M ? m0 + i * 16 + c : M - 1);
#pragma unroll
   for (int j = 0; j < NB; ++j)
      rb[j] = Bt.row(n0 + j * 16 + c < N ? n0 + j * 16 + c : N - 1);
   acc_t acc[MB][NB];
#pragma unroll
   for (int i = 0; i < MB; ++i)
#pragma unroll
      for (int j = 0; j < NB; ++j)
         acc[i][j] = acc_t{0, 0, 0, 0};

   const int whole = K / STEP; // steps without a chunk past K
   for (int s0 = wave; s0 < whole; s0 += W * UNROLL) {
      v4i fa[UNROLL][MB][2], fb[UNROLL][NB][2];
#pragma unroll
      for (int u = 0; u < UNROLL; ++u) {
         const int s = s0 + u * W;
         if (s < whole) {
            const int k = s * STEP + lk * 32;
#pragma unroll
            for (int j = 0; j < NB; ++j)
#pragma unroll
               for (int h = 0; h < 2; ++h)
                  fb[u][j][h] = *(const v4i_unaligned *)(rb[j] + k + 16 * h);
#pragma unroll
            for (int i = 0; i < MB; ++i)
#pragma unroll
               for (int h = 0; h < 2; ++h)
                  fa[u][i][h] = *(const v4i_unaligned *)(ra[i] + k + 16 * h);
         }
      }
#pragma unroll
      for (int u = 0; u < UNROLL; ++u)
         if (s0 + u * W < whole) {
#pragma unroll
            for (int i = 0; i < MB; ++i)
#pragma unroll
               for (int j = 0; j < NB; ++j)
                  acc[i][j] = MMA::mma(fb[u][j], fa[u][i], acc[i][j]);
         }
   }
   if (K % STEP != 0 && wave == whole % W) { // the wave whose turn it is
      const int k = whole * STEP + lk * 32;
      v4i fa[MB][2], fb[NB][2];
#pragma unroll
      for (int h = 0; h < 2; ++h) {
#pragma unroll
         for (int j = 0; j < NB; ++j)
            fb[j][h] = load_chunk_tail(rb[j], k + 16 * h, K);
#pragma unroll
         for (int i = 0; i < MB; ++i)
            fa[i][h] = load_chunk_tail(ra[i], k + 16 * h, K);
      }
#pragma unroll
      for (int i = 0; i < MB; ++i)
#pragma unroll
         for (int j = 0; j < NB; ++j)
            acc[i][j] = MMA::mma(fb[j], fa[i], acc[i][j]);
   }

#pragma unroll
   for (int i = 0; i < MB; ++i)
#pragma unroll
      for (int j = 0; j < NB; ++j)
         *(acc_t *)&part[wave][i * 16 + c][j * 16 + lk * 4] = acc[i][j];
   __syncthreads();
   ep.dispatch([&](auto mode) {
      constexpr int MODE = decltype(mode)::value;
#pragma unroll 1
      for (int e = threadIdx.x; e < TM * TN / 4; e += W * 64) {
         const int r = e / (TN / 4), q = e % (TN / 4) * 4;
         acc_t v = *(const acc_t *)&part[0][r][q];
#pragma unroll
         for (int w = 1; w < W; ++w)
            v += *(const acc_t *)&part[w][r][q];
         const int m = m0 + r, n = n0 + q;
         if (m >= M || n >= N)
            continue;
         typename EPI::template col_params<4> prm;
         ep.template load_params<4>(n, prm);
         store_four_columns<MODE>(ep, prm, v, m, n, N);
      }
   });
}

template <class MMA, int MB, int NB, int W, int UNROLL, class EPI>
static int launch_mfma8_direct(const LaunchCfg &lc, const int8_t *A, const int8_t *Bt, int M, int N, int K, int lda, int ldb, const EPI &ep)
{
   const int tiles_m = (M + MB * 16 - 1) / (MB * 16), tiles_n = (N + NB * 16 - 1) / (NB * 16);
   const long long nwg = (long long)tiles_m * tiles_n;
   if (nwg > 0x7fffffffLL)
      return fail(SOFIE_HIP_ERR_INVALID, "gemm: too many tiles");
   in_launches(nwg, W * 64, [&](int first, unsigned count) {
      launch_kernel((mfma8_direct_kernel<MMA, MB, NB, W, UNROLL, EPI>), dim3(count), dim3(W * 64), 0, lc.stream, RowMajorRows{A, lda}, RowMajorRows{Bt, ldb}, M, N, K, ep,
                    tiles_m, tiles_n, lc.swizzle, first);
   });
   return launch_status("mfma8_direct_kernel");
}

} // namespace sofie_hip
