// int8 / FP8 products of few rows (or few tiles): no LDS on the way in.  A workgroup owns one small tile of Y and its W waves
// split the reduction; every fragment is loaded from memory into the registers the MFMA reads, UNROLL steps of 128 bytes of k
// ahead, and the partial tiles meet in LDS.  What such a product costs is the trip to memory for its operands, and one workgroup
// has its whole share of them (tens of KB) on the way at once; the ring kernels wait for a few KB at a time.  A tile has as few
// as 16 rows, where theirs have 64.  Rows may start at any byte: those that start on no word are read as the words they lie in.
#pragma once
#include "mfma8_gemm_dma.hpp"
#include <algorithm>

namespace sofie_hip {

typedef int v4i_unaligned __attribute__((ext_vector_type(4), aligned(1)));

// 16 bytes from any address as words: those they lie in, five of them (four where the address is a multiple of four, so that every word that is read has at least one of the
// bytes).  One load of 16 bytes at an address that is no multiple of four takes the vector L1 three times as long as at one that is.
struct AnyChunk {
   typedef int words_t __attribute__((ext_vector_type(4), aligned(4)));
   v4i v;
   unsigned behind, shift;
   __device__ __forceinline__ void load(const int8_t *p)
   {
      shift = (unsigned)(uintptr_t)p & 3u;
      const int8_t *word = p - shift;
      v = *(const words_t *)word;
      behind = *(const unsigned *)(word + (shift ? 16 : 12));
   }
   static __device__ __forceinline__ v4i aligned(v4i v, unsigned behind, unsigned shift)
   {
      v4i out;
#pragma unroll
      for (int i = 0; i < 4; ++i)
         out[i] = (int)__builtin_amdgcn_alignbyte(i < 3 ? (unsigned)v[i + 1 < 4 ? i + 1 : 3] : behind, (unsigned)v[i], shift);
      return out;
   }
   __device__ __forceinline__ v4i bytes() const { return aligned(v, behind, shift); }
};

inline bool rows_of_words(const int8_t *base, int ld) { return ((uintptr_t)base & 3) == 0 && (ld & 3) == 0; }

// The chunk at k of a row of K >= 16 bytes as a load inside the row: where it crosses K, the last 16 bytes of the row instead,
// which cut_chunk moves down to k, zeros behind them.
__device__ __forceinline__ const int8_t *chunk_in_row(const int8_t *row, int k, int K) { return row + (k <= K - 16 ? k : K - 16); }
__device__ __forceinline__ v4i cut_chunk(v4i v, int k, int K)
{
   union {
      v4i v;
      unsigned long long q[2];
   } u;
   u.v = v;
   const int drop = (k - K + 16) * 8; // bits that lie before k
   if (drop > 0) {
      const unsigned long long hi = drop >= 128 ? 0 : u.q[1];
      u.q[0] = drop >= 64 ? hi >> (drop & 63) : (u.q[0] >> drop) | (u.q[1] << (64 - drop));
      u.q[1] = drop >= 64 ? 0 : u.q[1] >> drop;
   }
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

// 16 bytes per lane into LDS, from a buffer that starts at `base`; an offset past its end (-1) reads as zero.
constexpr int DIRECT_BUFFER_BYTES = 0x7fffff00;
__device__ __forceinline__ void direct_buffer_load(lds_void_t *to, const void *base, int offset)
{
   const __amdgpu_buffer_rsrc_t buffer = __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(base), 0, DIRECT_BUFFER_BYTES, 0x00020000);
   __builtin_amdgcn_raw_ptr_buffer_load_lds(buffer, to, 16, offset, 0, 0, 0);
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

// The partial tiles of W waves meet in LDS and are stored, four columns of a row by a thread.
template <class MMA, int MB, int NB, int W, class EPI>
struct DirectStore {
   static constexpr int TM = MB * 16, TN = NB * 16;
   static_assert(TM * TN / 4 <= W * 64, "four elements by a thread");
   int m0, n0, M, N, r, q;
   bool live;
   typename EPI::template col_params<4> prm;
   __device__ __forceinline__ DirectStore(int m0, int n0, int M, int N) : m0(m0), n0(n0), M(M), N(N)
   {
      r = (int)threadIdx.x / (TN / 4), q = (int)threadIdx.x % (TN / 4) * 4;
      live = r < TM && m0 + r < M && n0 + q < N;
   }
   // the columns' parameters
   __device__ __forceinline__ void ask(const EPI &ep)
   {
      if (live)
         ep.template load_params<4>(n0 + q, prm);
   }
   __device__ __forceinline__ void store(const EPI &ep, const typename MMA::acc_t (&acc)[MB][NB], typename MMA::elem_t (*part)[TM][TN + 4], int wave, int lane) const
   {
      typedef typename MMA::acc_t acc_t;
      const int lk = lane >> 4, c = lane & 15;
#pragma unroll
      for (int i = 0; i < MB; ++i)
#pragma unroll
         for (int j = 0; j < NB; ++j)
            *(acc_t *)&part[wave][i * 16 + c][j * 16 + lk * 4] = acc[i][j];
      __syncthreads();
      if (!live)
         return;
      acc_t v = *(const acc_t *)&part[0][r][q];
#pragma unroll
      for (int w = 1; w < W; ++w)
         v += *(const acc_t *)&part[w][r][q];
      ep.dispatch([&](auto mode) { store_four_columns<decltype(mode)::value>(ep, prm, v, m0 + r, n0 + q, N); });
   }
};

// What a lane reads of a row in a step: 32 bytes, as nine words of any row (BYTES) or two chunks of one that starts on four bytes.  The vector L1 bounds this kernel where rows start
// at any byte: as two unaligned chunks 7 bytes a clock reached a CU, as words 15 - 26; 16 x 193 x 395 3.45 us before, 2.85 now, 2 x 900 x 4001 9.3 and 5.1, 16 x 4096 x 4093 12.9 and
// 6.7, 50 x 1500 x 767 7.6 and 4.1.
template <bool BYTES>
struct DirectLane {
   v4i v[2];
   unsigned behind;
   __device__ __forceinline__ void load(const int8_t *row, int k)
   {
      if constexpr (BYTES) {
         const unsigned shift = (unsigned)(uintptr_t)row & 3u;
         const int8_t *word = row - shift + k;
         v[0] = *(const AnyChunk::words_t *)word;
         v[1] = *(const AnyChunk::words_t *)(word + 16);
         behind = *(const unsigned *)(word + (shift ? 32 : 28));
      } else {
         v[0] = *(const v4i_unaligned *)(row + k);
         v[1] = *(const v4i_unaligned *)(row + k + 16);
      }
   }
   __device__ __forceinline__ void finish(const int8_t *row)
   {
      if constexpr (BYTES) {
         const unsigned shift = (unsigned)(uintptr_t)row & 3u;
         v[0] = AnyChunk::aligned(v[0], (unsigned)v[1][0], shift);
         v[1] = AnyChunk::aligned(v[1], behind, shift);
      }
   }
};

// The step that K cuts off.
template <bool BYTES>
struct DirectLast {
   std::conditional_t<BYTES, AnyChunk, v4i> c[2];
   v4i v[2];
   __device__ __forceinline__ void load(const int8_t *row, int k, int K)
   {
#pragma unroll
      for (int h = 0; h < 2; ++h) {
         const int8_t *p = chunk_in_row(row, k + 16 * h, K);
         if constexpr (BYTES)
            c[h].load(p);
         else
            c[h] = *(const v4i_unaligned *)p;
      }
   }
   __device__ __forceinline__ void finish(int k, int K)
   {
#pragma unroll
      for (int h = 0; h < 2; ++h) {
         if constexpr (BYTES)
            v[h] = cut_chunk(c[h].bytes(), k + 16 * h, K);
         else
            v[h] = cut_chunk(c[h], k + 16 * h, K);
      }
   }
   // rows of fewer than 16 bytes
   __device__ __forceinline__ void load_short(const int8_t *row, int k, int K)
   {
      union {
         v4i v[2];
         int8_t b[32];
      } u;
      u.v[0] = u.v[1] = v4i{0, 0, 0, 0};
#pragma unroll
      for (int i = 0; i < 15; ++i)
         if (k + i < K)
            u.b[i] = row[k + i];
      v[0] = u.v[0], v[1] = u.v[1];
   }
};

template <class MMA, int MB, int NB, int W, int UNROLL, bool BYTES, class EPI>
__global__ __launch_bounds__(W * 64) void mfma8_direct_kernel(RowMajorRows A, RowMajorRows Bt, int M, int N, int K, EPI ep, TileOrder order, int first_tile)
{
   constexpr int STEP = 128, TM = MB * 16, TN = NB * 16, PITCH = TN + 4;
   typedef typename MMA::acc_t acc_t;
   typedef typename MMA::elem_t elem_t;
   __shared__ __attribute__((aligned(16))) elem_t part[W][TM][PITCH];
   int tm, tn;
   order.place(first_tile + blockIdx.x, tm, tn);
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
   // the step that K cuts off: asked for ahead of the others by the wave whose turn it is
   const bool last = K % STEP != 0 && wave == whole % W;
   const int last_k = whole * STEP + lk * 32;
   DirectLast<BYTES> la[MB], lb[NB];
   if (last) {
      if (K >= 16) {
#pragma unroll
         for (int j = 0; j < NB; ++j)
            lb[j].load(rb[j], last_k, K);
#pragma unroll
         for (int i = 0; i < MB; ++i)
            la[i].load(ra[i], last_k, K);
      } else {
#pragma unroll
         for (int j = 0; j < NB; ++j)
            lb[j].load_short(rb[j], last_k, K);
#pragma unroll
         for (int i = 0; i < MB; ++i)
            la[i].load_short(ra[i], last_k, K);
      }
   }
   for (int s0 = wave; s0 < whole; s0 += W * UNROLL) {
      DirectLane<BYTES> fa[UNROLL][MB], fb[UNROLL][NB];
#pragma unroll
      for (int u = 0; u < UNROLL; ++u) {
         const int s = s0 + u * W;
         if (s < whole) {
            const int k = s * STEP + lk * 32;
#pragma unroll
            for (int j = 0; j < NB; ++j)
               fb[u][j].load(rb[j], k);
#pragma unroll
            for (int i = 0; i < MB; ++i)
               fa[u][i].load(ra[i], k);
         }
      }
#pragma unroll
      for (int u = 0; u < UNROLL; ++u)
         if (s0 + u * W < whole) {
#pragma unroll
            for (int j = 0; j < NB; ++j)
               fb[u][j].finish(rb[j]);
#pragma unroll
            for (int i = 0; i < MB; ++i)
               fa[u][i].finish(ra[i]);
#pragma unroll
            for (int i = 0; i < MB; ++i)
#pragma unroll
               for (int j = 0; j < NB; ++j)
                  acc[i][j] = MMA::mma(fb[u][j].v, fa[u][i].v, acc[i][j]);
         }
   }
   if (last) {
      if (K >= 16) {
#pragma unroll
         for (int j = 0; j < NB; ++j)
            lb[j].finish(last_k, K);
#pragma unroll
         for (int i = 0; i < MB; ++i)
            la[i].finish(last_k, K);
      }
#pragma unroll
      for (int i = 0; i < MB; ++i)
#pragma unroll
         for (int j = 0; j < NB; ++j)
            acc[i][j] = MMA::mma(lb[j].v, la[i].v, acc[i][j]);
   }

   DirectStore<MMA, MB, NB, W, EPI> store(m0, n0, M, N);
   store.ask(ep);
   store.store(ep, acc, part, wave, lane);
}

// The same with the operands going through LDS, for rows that start on 16 bytes.  A vector L1 takes four cycles per line that a load instruction touches: fragments
// in the layout of the MFMA come from 16 rows, 64 bytes of a line each, at 16 B/clk, which bounds the kernel above (its 16 rows of 4096 bytes and as
// many of B: 128 KB, 3.5 us of 6.8).  Loaded line by line, 128 bytes of eight rows per instruction, straight into LDS, they come at twice that.  A wave's steps
// pass through a ring of its own of `depth` places: no barrier in the loop.
// (Pitches and K are in bytes: the fp32 products use it too.)
template <class MMA, int MB, int NB, int W>
__device__ __forceinline__ void direct_ring_sums(typename MMA::acc_t (&acc)[MB][NB], const RowMajorRows &A, const RowMajorRows &Bt, int M, int N, int K, int m0, int n0,
                                                 int8_t *smem, int depth, int wave, int lane)
{
   constexpr int STEP = 128, LA = MB * 2, LB = NB * 2, LOADS = LA + LB, PLACE = (MB + NB) * 16 * STEP;
   const int lk = lane >> 4, c = lane & 15;
   // load i brings rows 8 i .. 8 i + 7 of the tile's B, then A, in the order of lds_chunk_offset; rows past the edge re-read the last one
   int at[LOADS], chunk[LOADS];
#pragma unroll
   for (int i = 0; i < LOADS; ++i) {
      const int row = i * 8 + lane / 8, r = i < LB ? row : row - NB * 16, last = i < LB ? N - 1 - n0 : M - 1 - m0;
      chunk[i] = ((lane & 7) ^ (row >> 1 & 7)) * 16;
      at[i] = (r < last ? r : last) * (i < LB ? Bt.ld : A.ld) + chunk[i];
   }
   int8_t *const mine = smem + wave * depth * PLACE;
   const int8_t *const base_a = A.row(m0), *const base_b = Bt.row(n0);
   const int steps = (int)(((unsigned)K + STEP - 1) / STEP), own = wave < steps ? (steps - wave + W - 1) / W : 0;
   auto issue = [&](int i, int place) {
      const int k = (wave + i * W) * STEP;
#pragma unroll
      for (int l = 0; l < LOADS; ++l) {
         direct_buffer_load((lds_void_t *)(mine + place * PLACE + l * 1024), (l < LB ? base_b : base_a) + k, chunk[l] < K - k ? at[l] : -1);
      }
   };
#pragma unroll
   for (int i = 0; i < MB; ++i)
#pragma unroll
      for (int j = 0; j < NB; ++j)
         acc[i][j] = typename MMA::acc_t{0};
   for (int i = 0; i < depth && i < own; ++i)
      issue(i, i);
   int place = 0;
#pragma unroll 1
   for (int i = 0; i < own; ++i) {
      const int ahead = own - 1 - i < depth - 1 ? own - 1 - i : depth - 1; // steps that may still be on their way
      if (ahead >= 3)
         wait_vmcnt<3 * LOADS>();
      else if (ahead == 2)
         wait_vmcnt<2 * LOADS>();
      else if (ahead == 1)
         wait_vmcnt<LOADS>();
      else
         wait_vmcnt<0>();
      __builtin_amdgcn_sched_barrier(0);
      v4i fa[MB][2], fb[NB][2];
      const int8_t *const from = mine + place * PLACE;
#pragma unroll
      for (int h = 0; h < 2; ++h) {
#pragma unroll
         for (int j = 0; j < NB; ++j)
            fb[j][h] = *(const v4i *)(from + lds_chunk_offset<STEP>(j * 16 + c, lk * 2 + h));
#pragma unroll
         for (int m = 0; m < MB; ++m)
            fa[m][h] = *(const v4i *)(from + lds_chunk_offset<STEP>((NB + m) * 16 + c, lk * 2 + h));
      }
      __builtin_amdgcn_s_waitcnt(0xc07f); // lgkmcnt(0): the place may be filled again
      __builtin_amdgcn_sched_barrier(0);
      if (i + depth < own)
         issue(i + depth, place);
      place = place + 1 == depth ? 0 : place + 1;
#pragma unroll
      for (int m = 0; m < MB; ++m)
#pragma unroll
         for (int j = 0; j < NB; ++j)
            acc[m][j] = MMA::mma(fb[j], fa[m], acc[m][j]);
   }
}

template <class MMA, int MB, int NB, int W, class EPI>
__global__ __launch_bounds__(W * 64) void mfma8_direct_ring_kernel(RowMajorRows A, RowMajorRows Bt, int M, int N, int K, EPI ep, TileOrder order, int first_tile, int depth)
{
   extern __shared__ __attribute__((aligned(16))) int8_t smem[];
   int tm, tn;
   order.place(first_tile + blockIdx.x, tm, tn);
   const int m0 = tm * MB * 16, n0 = tn * NB * 16;
   const int lane = threadIdx.x & 63;
   const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
   typename MMA::acc_t acc[MB][NB];
   direct_ring_sums<MMA, MB, NB, W>(acc, A, Bt, M, N, K, m0, n0, smem, depth, wave, lane);
   DirectStore<MMA, MB, NB, W, EPI> store(m0, n0, M, N);
   store.ask(ep);
   __syncthreads();
   store.store(ep, acc, (typename MMA::elem_t(*)[MB * 16][NB * 16 + 4])smem, wave, lane);
}

// The ring of a launch: places per wave (as many as fit and are used; half of them where a CU has several tiles), and bytes of LDS, in which the partial tiles
// meet too.  K in bytes.
template <int MB, int NB, int W>
struct DirectRing {
   static constexpr int PLACE = (MB + NB) * 16 * 128, MOST = 128 * 1024 / (W * PLACE);
   static constexpr size_t PART = (size_t)W * MB * 16 * (NB * 16 + 4) * 4;
   int depth;
   size_t bytes;
   DirectRing(long long workgroups, int K)
   {
      const int steps = (int)(((unsigned)K + 127) / 128);
      depth = std::max(1, std::min(workgroups > 256 ? MOST / 2 : MOST, (steps + W - 1) / W));
      bytes = std::max((size_t)std::min(steps, W) * depth * PLACE, PART);
   }
   // rows on 16 bytes, and a tile's rows within a buffer
   static bool takes(const void *A, const void *Bt, long long lda, long long ldb, long long K)
   {
      return ((uintptr_t)A & 15) == 0 && ((uintptr_t)Bt & 15) == 0 && lda % 16 == 0 && ldb % 16 == 0 && K % 16 == 0 && K > 0 && K <= 0x7fffffff &&
             (MB > NB ? MB : NB) * 16 * (lda > ldb ? lda : ldb) + 256 < DIRECT_BUFFER_BYTES;
   }
};

// Whether an int8 / FP8 product of 16-byte rows in tiles of b x b comes line by line.  A wave with a single step has nothing to pipeline, and the trip through LDS is
// what the ring adds: K = 128 in 16 x 16 tiles 2.49 us, 2.62 through the ring, in 32 x 32 tiles 2.85 and 3.08; K = 256 2.60 and 2.63, 3.02 and 3.09.  With more than
// two tiles of 32 x 32 a CU, lines count again (500 x 1500 x 256 5.3 us, 4.4).  Up to four rows are as many lines less for the registers: 1 x 1000 x 640 2.81 us and
// 2.97, even at K = 896.  A last step that is not whole is loaded chunk by chunk into the registers, which costs more than the ring (16 rows of 112 bytes 2.7, 2.5).
inline bool mfma8_direct_by_lines(int b, int M, int N, int K)
{
   if (K % 128 != 0)
      return true;
   if (K <= 256)
      return b > 16 && (long long)((M + b - 1) / b) * ((N + b - 1) / b) > 512;
   return !(b == 16 && M <= 4 && K <= 768);
}

template <class MMA, int MB, int NB, int W, int UNROLL, class EPI>
static int launch_mfma8_direct(const LaunchCfg &lc, const int8_t *A, const int8_t *Bt, int M, int N, int K, int lda, int ldb, const EPI &ep)
{
   const int tiles_m = (M + MB * 16 - 1) / (MB * 16), tiles_n = (N + NB * 16 - 1) / (NB * 16);
   const long long nwg = (long long)tiles_m * tiles_n;
   if (nwg > 0x7fffffffLL)
      return fail(SOFIE_HIP_ERR_INVALID, "gemm: too many tiles");
   const TileOrder order(tiles_m, tiles_n, lc.swizzle);
   typedef DirectRing<MB, NB, W> Ring;
   if (mfma8_direct_by_lines(MB * 16, M, N, K) && Ring::takes(A, Bt, lda, ldb, K)) {
      const Ring ring(nwg, K);
      auto kern = mfma8_direct_ring_kernel<MMA, MB, NB, W, EPI>;
      static bool configured[64] = {};
      if (int st = configure_lds_once(kern, 128 * 1024, configured))
         return st;
      in_launches(nwg, W * 64, [&](int first, unsigned count) {
         launch_kernel(kern, dim3(count), dim3(W * 64), ring.bytes, lc.stream, RowMajorRows{A, lda}, RowMajorRows{Bt, ldb}, M, N, K, ep, order, first,
                       ring.depth);
      });
      return launch_status("mfma8_direct_ring_kernel");
   }
   const bool bytes = !rows_of_words(A, lda) || !rows_of_words(Bt, ldb);
   in_launches(nwg, W * 64, [&](int first, unsigned count) {
      launch_kernel(bytes ? mfma8_direct_kernel<MMA, MB, NB, W, UNROLL, true, EPI> : mfma8_direct_kernel<MMA, MB, NB, W, UNROLL, false, EPI>, dim3(count), dim3(W * 64), 0, lc.stream, RowMajorRows{A, lda}, RowMajorRows{Bt, ldb}, M, N, K, ep,
                    order, first);
   });
   return launch_status("mfma8_direct_kernel");
}

} // namespace sofie_hip
