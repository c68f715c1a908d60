// General tile loop of the int8 and the FP8 GEMM: any K, any alignment, B stored either way.  The pipelined kernels load straight
// into LDS, which takes rows that start on 16 bytes and a K of whole slabs; here the slabs go through registers, so that a chunk
// may start at any byte, the last chunk of a row is cut off at K, and a B given as
// [K,N] is transposed on its way into LDS, four bytes by four, instead of by a launch of its own.
//
// A workgroup owns a BM x BN tile of Y and walks K in slabs of BK bytes, DEPTH slabs of loads ahead in registers, two slabs of LDS in
// the swizzled layout of lds_chunk_offset, one barrier per slab.  The Bt rows are the MFMA's first operand, so that a lane ends up
// with 4 consecutive columns of one row.
#pragma once
#include "mfma8_direct.hpp"

namespace sofie_hip {

// An operand of `rows` rows that are contiguous in k.
struct StagedRows {
   static constexpr bool kTransposed = false;
   static constexpr int kWaves = 2; // a SIMD at least
   const int8_t *base;
   int ld, rows;
};
// The same with rows that start at any byte, fewer than 2^24 bytes apart: read as words, which the vector L1 takes faster than chunks that start on none (us, chunks -> words: 1537 x
// 1000 x 777 9.7 -> 8.7, 777 x 1555 x 1999 16.3 -> 14.6, 384 x 2976 x 3501 20.4 -> 17.3).  Not for tiles of 128 x 128, which have no registers left for it beside four waves a SIMD: 4001 x 4001
// x 1001 57 as chunks, 61 as words by two waves; nor for columns, whose short pieces would be two loads each: 777 x 1555 x 1999 16.0 and 18.3.
struct StagedAnyRows : StagedRows {
   static constexpr int kWaves = 4;
   static bool takes(int ld) { return ld < 1 << 24; } // offsets inside a slab in 32 bits
};
// An operand stored [K][rows]: contiguous along the rows.
struct StagedColumns {
   static constexpr bool kTransposed = true;
   const int8_t *base;
   int ld, rows;
};

// A convolution input that is never laid out as a matrix: row m is the output pixel (image, oh, ow), k = tap * Cg + channel, read from the
// NHWC activation tensor in pieces of PIECE bytes that lie inside one tap (PIECE divides the channels per group).  For layers whose
// channels are no power of two of 64 or more (ConvRows serves those): 16, 24, 32, 48 ...
template <int PIECE_>
struct StagedConvRows {
   static constexpr bool kTransposed = false;
   static constexpr int kWaves = 2;
   static constexpr int PIECE = PIECE_;
   const int8_t *X; // first channel of the group
   int rows, H, W, C, OH, OW, stride_h, stride_w, pad_h0, pad_w0, dil_h, dil_w, kw, Cg, K;
   unsigned cg_mul, kw_mul; // ceil(2^31 / extent): k / extent == umulhi(2 k, mul) while k * extent < 2^31 (checked on the host)
   unsigned long long ohw_mul, ow_mul; // see ConvRows
};

// A slab of R rows x BK bytes on its way from memory to LDS: what one of NTHREADS threads carries.
template <class SRC, int R, int BK, int NTHREADS>
struct StagedSlab {
   struct places {}; // what a thread works out once about its rows
   static __device__ __forceinline__ void find(const SRC &, int, int, places &) {}
   static constexpr int CPR = BK / 16;
   static constexpr int LD = R * CPR / NTHREADS; // 16-byte chunks per thread: chunk t + i * NTHREADS of the slab, row by row
   static_assert(R * CPR % NTHREADS == 0, "the slab divides over the threads");
   v4i v[LD];
   static __device__ __forceinline__ const int8_t *row_of(const SRC &s, int r0, int i, int t)
   {
      const int r = r0 + (t + i * NTHREADS) / CPR;
      return s.base + (size_t)(r < s.rows ? r : s.rows - 1) * (size_t)s.ld; // rows past the edge re-read the last one
   }
   static __device__ __forceinline__ int k_of(int k0, int i, int t) { return k0 + (t + i * NTHREADS) % CPR * 16; }
   // a slab that lies before K
   __device__ __forceinline__ void load(const SRC &s, const places &, int r0, int k0, int, int t)
   {
#pragma unroll
      for (int i = 0; i < LD; ++i)
         v[i] = *(const v4i_unaligned *)(row_of(s, r0, i, t) + k_of(k0, i, t));
   }
   // the slab that K cuts off: fetched as whole chunks of the row, cut later
   __device__ __forceinline__ void load_last(const SRC &s, const places &, int r0, int k0, int K, int t)
   {
#pragma unroll
      for (int i = 0; i < LD; ++i)
         v[i] = *(const v4i_unaligned *)chunk_in_row(row_of(s, r0, i, t), k_of(k0, i, t), K);
   }
   __device__ __forceinline__ void finish_last(int k0, int K, int t)
   {
#pragma unroll
      for (int i = 0; i < LD; ++i)
         v[i] = cut_chunk(v[i], k_of(k0, i, t), K);
   }
   __device__ __forceinline__ void store(int8_t *lds, int t) const
   {
#pragma unroll
      for (int i = 0; i < LD; ++i) {
         const int id = t + i * NTHREADS;
         *(v4i *)(lds + lds_chunk_offset<BK>(id / CPR, id % CPR)) = v[i];
      }
   }
};

template <int R, int BK, int NTHREADS>
struct StagedSlab<StagedAnyRows, R, BK, NTHREADS> {
   typedef StagedAnyRows SRC;
   typedef StagedSlab<StagedRows, R, BK, NTHREADS> Words;
   static constexpr int CPR = Words::CPR, LD = Words::LD;
   static_assert(CPR == 8, "half a row of lanes to a row of the slab");
   // from the word that the tile starts in: a chunk's first word and the word behind the slab's row (the one its last byte lies in, where the row starts on a word)
   struct places {
      unsigned at[LD], behind[LD], shift[LD];
   };
   AnyChunk c[LD];
   static __device__ __forceinline__ const int8_t *tile_of(const SRC &s, int r0) { return s.base + (size_t)r0 * (size_t)s.ld; }
   static __device__ __forceinline__ void find(const SRC &s, int r0, int t, places &p)
   {
#pragma unroll
      for (int i = 0; i < LD; ++i) {
         const int r = (t + i * NTHREADS) / CPR;
         const unsigned from = ((unsigned)(uintptr_t)tile_of(s, r0) & 3u) + (unsigned)(r0 + r < s.rows ? r : s.rows - 1 - r0) * (unsigned)s.ld;
         p.at[i] = (from & ~3u) + (unsigned)(t % CPR * 16);
         p.behind[i] = (from + BK - 1) & ~3u;
         p.shift[i] = from & 3u;
      }
   }
   __device__ __forceinline__ void load(const SRC &s, const places &p, int r0, int k0, int, int)
   {
      const int8_t *tile = tile_of(s, r0);
      tile += k0 - (int)((unsigned)(uintptr_t)tile & 3u);
#pragma unroll
      for (int i = 0; i < LD; ++i) {
         c[i].v = *(const AnyChunk::words_t *)(tile + p.at[i]);
         c[i].behind = *(const unsigned *)(tile + p.behind[i]);
         c[i].shift = p.shift[i];
      }
   }
   __device__ __forceinline__ void load_last(const SRC &s, const places &, int r0, int k0, int K, int t)
   {
#pragma unroll
      for (int i = 0; i < LD; ++i)
         c[i].load(chunk_in_row(Words::row_of(s, r0, i, t), Words::k_of(k0, i, t), K));
   }
   __device__ __forceinline__ void finish_last(int k0, int K, int t)
   {
#pragma unroll
      for (int i = 0; i < LD; ++i) {
         c[i].v = cut_chunk(c[i].bytes(), Words::k_of(k0, i, t), K);
         c[i].shift = 0;
      }
   }
   __device__ __forceinline__ void store(int8_t *lds, int t) const
   {
#pragma unroll
      for (int i = 0; i < LD; ++i) {
         const int id = t + i * NTHREADS;
         const unsigned next = (unsigned)__builtin_amdgcn_mov_dpp(c[i].v[0], 0x101, 0xf, 0xf, true); // row_shl:1
         *(v4i *)(lds + lds_chunk_offset<BK>(id / CPR, id % CPR)) = AnyChunk::aligned(c[i].v, id % CPR == CPR - 1 ? c[i].behind : next, c[i].shift);
      }
   }
};

template <int PIECE, int R, int BK, int NTHREADS>
struct StagedSlab<StagedConvRows<PIECE>, R, BK, NTHREADS> {
   typedef StagedConvRows<PIECE> SRC;
   static constexpr int CPR = BK / 16, LD = R * CPR / NTHREADS;
   static_assert(R * CPR % NTHREADS == 0 && NTHREADS % CPR == 0, "the slab divides over the threads");
   typedef int piece_t __attribute__((ext_vector_type(PIECE / 4), aligned(PIECE)));
   union chunk_t {
      v4i v;
      piece_t p[16 / PIECE];
   };
   struct places {
      int off[LD], ih0[LD], iw0[LD]; // of channel 0 at (ih0, iw0), in bytes from X: may be negative
   };
   v4i v[LD];
   static __device__ __forceinline__ void find(const SRC &s, int r0, int t, places &at)
   {
#pragma unroll
      for (int i = 0; i < LD; ++i) {
         const int r = r0 + (t + i * NTHREADS) / CPR, m = r < s.rows ? r : s.rows - 1;
         const int ohw = s.OH * s.OW;
         const int n = s.ohw_mul ? (int)__umul64hi((unsigned long long)(unsigned)m, s.ohw_mul) : m, rem = m - n * ohw;
         const int oh = s.ow_mul ? (int)__umul64hi((unsigned long long)(unsigned)rem, s.ow_mul) : rem, ow = rem - oh * s.OW;
         at.ih0[i] = oh * s.stride_h - s.pad_h0;
         at.iw0[i] = ow * s.stride_w - s.pad_w0;
         at.off[i] = ((n * s.H + at.ih0[i]) * s.W + at.iw0[i]) * s.C;
      }
   }
   __device__ __forceinline__ void load(const SRC &s, const places &at, int, int k0, int, int t)
   {
      // the chunk's place in the slab is the same in every load of a thread
#pragma unroll
      for (int q = 0; q < 16 / PIECE; ++q) {
         const int k = k0 + t % CPR * 16 + q * PIECE;
         const int tap = (int)__umulhi((unsigned)k * 2u, s.cg_mul), ci = k - tap * s.Cg;
         const int ky = (int)__umulhi((unsigned)tap * 2u, s.kw_mul), kx = tap - ky * s.kw;
         const int dy = ky * s.dil_h, dx = kx * s.dil_w, off = (dy * s.W + dx) * s.C + ci;
#pragma unroll
         for (int i = 0; i < LD; ++i) {
            const bool inside = k < s.K && (unsigned)(at.ih0[i] + dy) < (unsigned)s.H && (unsigned)(at.iw0[i] + dx) < (unsigned)s.W;
            chunk_t c;
            c.v = v[i];
            c.p[q] = *(const piece_t *)(inside ? s.X + (ptrdiff_t)(at.off[i] + off) : (const int8_t *)conv_zero_page);
            v[i] = c.v;
         }
      }
   }
   __device__ __forceinline__ void load_last(const SRC &s, const places &at, int r0, int k0, int K, int t) { load(s, at, r0, k0, K, t); }
   __device__ __forceinline__ void finish_last(int, int, int) {}
   __device__ __forceinline__ void store(int8_t *lds, int t) const
   {
#pragma unroll
      for (int i = 0; i < LD; ++i) {
         const int id = t + i * NTHREADS;
         *(v4i *)(lds + lds_chunk_offset<BK>(id / CPR, id % CPR)) = v[i];
      }
   }
};

// four bytes each of the k neighbours r0..r3 -> four k bytes of each of four rows
__device__ __forceinline__ void transpose_4x4_bytes(unsigned r0, unsigned r1, unsigned r2, unsigned r3, unsigned (&out)[4])
{
   const unsigned a = __builtin_amdgcn_perm(r1, r0, 0x05010400u), b = __builtin_amdgcn_perm(r1, r0, 0x07030602u);
   const unsigned c = __builtin_amdgcn_perm(r3, r2, 0x05010400u), d = __builtin_amdgcn_perm(r3, r2, 0x07030602u);
   out[0] = __builtin_amdgcn_perm(c, a, 0x05040100u);
   out[1] = __builtin_amdgcn_perm(c, a, 0x07060302u);
   out[2] = __builtin_amdgcn_perm(d, b, 0x05040100u);
   out[3] = __builtin_amdgcn_perm(d, b, 0x07060302u);
}

template <int R, int BK, int NTHREADS>
struct StagedSlab<StagedColumns, R, BK, NTHREADS> {
   // a thread carries blocks of 4 k of PR rows, eight or, where there are threads enough, four: four pieces of as many bytes, one per k
   static constexpr int PR = R / 8 * (BK / 4) >= NTHREADS ? 8 : 4;
   static constexpr int RB = R / PR; // blocks along the rows
   static constexpr int LD = RB * (BK / 4) / NTHREADS;
   static_assert(RB * (BK / 4) % NTHREADS == 0, "the slab divides over the threads");
   typedef std::conditional_t<PR == 8, unsigned long long, unsigned> piece_t;
   typedef piece_t piece_unaligned_t __attribute__((aligned(1)));
   piece_t v[LD][4];
   struct places {};
   static __device__ __forceinline__ void find(const StagedColumns &, int, int, places &) {}
   static __device__ __forceinline__ unsigned word(piece_t v, int q) { return (unsigned)((unsigned long long)v >> (32 * q)); }
   static __device__ __forceinline__ int row_of(int i, int t) { return (t + i * NTHREADS) % RB * PR; }
   static __device__ __forceinline__ int k_of(int i, int t) { return (t + i * NTHREADS) / RB * 4; }
   // pieces past the last column are fetched from the last columns (align_edge moves them), k past K from the last k (finish_last)
   __device__ __forceinline__ void load_last(const StagedColumns &s, const places &, int r0, int k0, int K, int t)
   {
#pragma unroll
      for (int i = 0; i < LD; ++i) {
         const int r = r0 + row_of(i, t), k = k0 + k_of(i, t);
#pragma unroll
         for (int j = 0; j < 4; ++j)
            v[i][j] = *(const piece_unaligned_t *)(s.base + (size_t)(k + j < K ? k + j : K - 1) * (size_t)s.ld + (r + PR <= s.rows ? r : s.rows - PR));
      }
   }
   __device__ __forceinline__ void load(const StagedColumns &s, const places &, int r0, int k0, int K, int t)
   {
#pragma unroll
      for (int i = 0; i < LD; ++i) {
         const int r = r0 + row_of(i, t);
         const int8_t *p = s.base + (size_t)(k0 + k_of(i, t)) * (size_t)s.ld + (r + PR <= s.rows ? r : s.rows - PR);
#pragma unroll
         for (int j = 0; j < 4; ++j)
            v[i][j] = *(const piece_unaligned_t *)(p + (size_t)j * (size_t)s.ld);
      }
   }
   __device__ __forceinline__ void finish_last(int k0, int K, int t)
   {
#pragma unroll
      for (int i = 0; i < LD; ++i)
#pragma unroll
         for (int j = 0; j < 4; ++j)
            if (k0 + k_of(i, t) + j >= K)
               v[i][j] = 0;
   }
   __device__ __forceinline__ void align_edge(const StagedColumns &s, int r0, int t)
   {
#pragma unroll
      for (int i = 0; i < LD; ++i) {
         const int drop = (r0 + row_of(i, t) + PR - s.rows) * 8; // bits that lie before the piece's first row
#pragma unroll
         for (int j = 0; j < 4; ++j)
            v[i][j] = drop <= 0 ? v[i][j] : drop >= 8 * PR ? 0 : v[i][j] >> drop;
      }
   }
   __device__ __forceinline__ void store(int8_t *lds, int t) const
   {
#pragma unroll
      for (int i = 0; i < LD; ++i) {
         const int r = row_of(i, t), k = k_of(i, t);
#pragma unroll
         for (int q = 0; q < PR / 4; ++q) {
            unsigned w[4];
            transpose_4x4_bytes(word(v[i][0], q), word(v[i][1], q), word(v[i][2], q), word(v[i][3], q), w);
#pragma unroll
            for (int e = 0; e < 4; ++e)
               *(unsigned *)(lds + lds_chunk_offset<BK>(r + 4 * q + e, k / 16) + k % 16) = w[e];
         }
      }
   }
};

template <class MMA, int BM, int BN, int BK, int WAVES_M, int WAVES_N, int DEPTH, class ASRC, class BSRC, class EPI>
__global__ __launch_bounds__(WAVES_M *WAVES_N * 64, ASRC::kWaves) void mfma8_staged_kernel(ASRC A, BSRC B, int M, int N, int K, EPI ep, TileOrder order)
{
   constexpr int NTHREADS = WAVES_M * WAVES_N * 64;
   constexpr int TM = BM / WAVES_M, TN = BN / WAVES_N, MT = TM / 32, NT = TN / 32;
   constexpr int STAGE = (BM + BN) * BK;
   static_assert(TM % 32 == 0 && TN % 32 == 0 && BK % MMA::KSTEP == 0, "wave tile of 32 x 32 blocks, slab of whole steps");
   static_assert(DEPTH % 2 == 0, "the LDS slot of a slab follows from its place in the unrolled group");
   typedef typename MMA::acc_t acc_t;
   typedef typename MMA::frag_t frag_t;
   extern __shared__ __attribute__((aligned(16))) int8_t smem[];

   int tm, tn;
   order.place(blockIdx.x, tm, tn);
   const int m0 = tm * BM, n0 = tn * BN;
   const int t = threadIdx.x, lane = t & 63;
   const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
   const int wm = wave / WAVES_N, wn = wave % WAVES_N;
   const int lr = lane & 31, lk = lane >> 5;

   acc_t acc[MT][NT];
#pragma unroll
   for (int i = 0; i < MT; ++i)
#pragma unroll
      for (int j = 0; j < NT; ++j)
#pragma unroll
         for (int v = 0; v < 16; ++v)
            acc[i][j][v] = 0;

   typedef StagedSlab<ASRC, BM, BK, NTHREADS> SA;
   typedef StagedSlab<BSRC, BN, BK, NTHREADS> SB;
   const int whole = K / BK; // slabs that lie before K
   const bool at_edge = BSRC::kTransposed && n0 + BN > N;
   auto multiply = [&](const int8_t *cA, const int8_t *cB) {
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
      __builtin_amdgcn_s_barrier();
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
#pragma unroll
      for (int ks = 0; ks < BK / MMA::KSTEP; ++ks) {
         frag_t fa[MT], fb[NT];
#pragma unroll
         for (int j = 0; j < NT; ++j)
#pragma unroll
            for (int c = 0; c < MMA::CHUNKS; ++c)
               fb[j].c[c] = *(const v4i *)(cB + lds_chunk_offset<BK>(wn * TN + j * 32 + lr, (ks * 2 + lk) * MMA::CHUNKS + c));
#pragma unroll
         for (int i = 0; i < MT; ++i)
#pragma unroll
            for (int c = 0; c < MMA::CHUNKS; ++c)
               fa[i].c[c] = *(const v4i *)(cA + lds_chunk_offset<BK>(wm * TM + i * 32 + lr, (ks * 2 + lk) * MMA::CHUNKS + c));
#pragma unroll
         for (int i = 0; i < MT; ++i)
#pragma unroll
            for (int j = 0; j < NT; ++j)
               acc[i][j] = MMA::mma(fb[j], fa[i], acc[i][j]);
      }
   };
   // The slab that K cuts off comes first (the order of the slabs does not matter), its chunks fetched ahead of the others.
   typename SA::places pa;
   typename SB::places pb;
   SA::find(A, m0, t, pa);
   SB::find(B, n0, t, pb);
   SA last_a;
   SB last_b;
   if (whole * BK < K) {
      last_a.load_last(A, pa, m0, whole * BK, K, t);
      last_b.load_last(B, pb, n0, whole * BK, K, t);
   }
   SA sa[DEPTH];
   SB sb[DEPTH];
   // a slab past the end is asked for as the last one again: no branch stands between a load and the wait for it
   auto load = [&](int kt, auto dc) {
      constexpr int d = decltype(dc)::value;
      const int k0 = (kt < whole ? kt : whole - 1) * BK;
      sa[d].load(A, pa, m0, k0, K, t);
      sb[d].load(B, pb, n0, k0, K, t);
   };
   if (whole > 0)
      static_for<DEPTH>([&](auto dc) { load(decltype(dc)::value, dc); });
   if (whole * BK < K) {
      last_a.finish_last(whole * BK, K, t);
      if constexpr (BSRC::kTransposed)
         last_b.align_edge(B, n0, t);
      last_b.finish_last(whole * BK, K, t);
      last_a.store(smem + STAGE, t);
      last_b.store(smem + STAGE + BM * BK, t);
      multiply(smem + STAGE, smem + STAGE + BM * BK);
   }
   auto step = [&](int kt, auto dc, auto more) {
      constexpr int d = decltype(dc)::value;
      int8_t *cA = smem + (d & 1) * STAGE, *cB = cA + BM * BK;
      // this slot was read two slabs ago: the barrier of the slab in between has seen every wave done with it
      sa[d].store(cA, t);
      if constexpr (BSRC::kTransposed)
         if (at_edge)
            sb[d].align_edge(B, n0, t);
      sb[d].store(cB, t);
      if constexpr (decltype(more)::value)
         load(kt + DEPTH, dc);
      multiply(cA, cB);
   };
   int kt = 0;
   for (; kt + DEPTH < whole; kt += DEPTH)
      static_for<DEPTH>([&](auto dc) { step(kt + decltype(dc)::value, dc, std::true_type{}); });
   static_for<DEPTH>([&](auto dc) {
      if (kt + decltype(dc)::value < whole)
         step(kt + decltype(dc)::value, dc, std::false_type{});
   });

   __syncthreads(); // the slabs are dead: the tile store reuses LDS, one region per wave
   char *wsm = (char *)smem + wave * tile_store_lds_bytes(TN);
   ep.dispatch([&](auto mode) {
      tile_store_via_lds<decltype(mode)::value, MT, NT>(ep, acc, m0 + wm * TM, n0 + wn * TN, M, N, lane, wsm);
   });
}

template <class MMA, int BM, int BN, int BK, int WAVES_M, int WAVES_N, int DEPTH, class ASRC, class BSRC, class EPI>
static int launch_mfma8_staged(const LaunchCfg &lc, const ASRC &A, const BSRC &B, int M, int N, int K, const EPI &ep)
{
   const int tiles_m = (M + BM - 1) / BM, tiles_n = (N + BN - 1) / BN;
   const long long nwg = (long long)tiles_m * tiles_n;
   if (nwg > 0x7fffffffLL)
      return fail(SOFIE_HIP_ERR_INVALID, "gemm: too many tiles");
   constexpr size_t slabs = 2 * (size_t)(BM + BN) * BK, store = (size_t)WAVES_M * WAVES_N * tile_store_lds_bytes(BN / WAVES_N);
   constexpr size_t smem = slabs > store ? slabs : store;
   auto kern = mfma8_staged_kernel<MMA, BM, BN, BK, WAVES_M, WAVES_N, DEPTH, ASRC, BSRC, EPI>;
   static bool configured[64] = {};
   if (int st = configure_lds_once(kern, smem, configured))
      return st;
   launch_kernel(kern, dim3((unsigned)nwg), dim3(WAVES_M * WAVES_N * 64), smem, lc.stream, A, B, M, N, K, ep, TileOrder(tiles_m, tiles_n, lc.swizzle));
   return launch_status("mfma8_staged_kernel");
}

} // namespace sofie_hip
