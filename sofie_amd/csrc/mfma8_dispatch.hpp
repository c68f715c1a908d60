// Kernel choice for the int8 / FP8 GEMM and the int8 convolution: which tile, which pipelined kernel, or the general one.
#pragma once
#include "conv_i8_resident.hpp"
#include "conv_i8_direct.hpp"
#include "mfma8_staged.hpp"
#include <algorithm>
#include <cmath>

namespace sofie_hip {

// ---- estimates ------------------------------------------------------------------------------------------------------------
// Below the sizes that fill the matrix cores, all of these kernels are bound by the bytes a CU takes in (33 - 58 KB/us through
// registers, by what the loads' alignment costs, 67 - 75 KB/us straight into LDS) and by what a tile costs besides (start, store).
inline double mfma8_rounds(int M, int N, int bm, int bn)
{
   const double rounds = (double)((M + bm - 1) / bm) * ((N + bn - 1) / bn) / 256.0; // tiles per CU; a CU works on a few at a time
   return rounds <= 1.0 ? 1.0 : 0.5 * (rounds + std::ceil(rounds));
}
inline double mfma8_time(int M, int N, int K, int bm, int bn, double fixed_us, double tile_us, double bytes_per_us)
{
   return fixed_us + mfma8_rounds(M, N, bm, bn) * (tile_us + (double)(bm + bn) * K / bytes_per_us);
}
// `lines`: rows start on 16 bytes, so that the direct kernel loads line by line through its ring where that pays: 120 KB/us a CU for the first 2048 of a row, which
// are asked for at once, and as much behind them while few CUs are at work, 20 TB/s from L2 over all of them (us, estimated / measured: 16 x 4096 x 4096
// 4.4 / 4.2, 600 x 320 x 6144 6.7 / 6.4, 108 x 4096 x 8192 16.0 / 14.4); whole steps of a short K through registers at the rates below.  Fitted, int8 and FP8, to 1900
// products of 1 .. 800 rows by 32 .. 4096 columns, K = 32 .. 8192, with what the 64 x 64 tiles took: the choice is 0.05 % above the fastest on average, 7 % the most.
// `words`: rows start on four bytes; others are read as the words they lie in (33 KB/us a CU of the rows there are).  Fitted to 482 and 524 products.
inline double mfma8_direct_time(int M, int N, int K, int b, bool words, bool lines)
{
   if (!lines) {
      if (words)
         return b == 16 ? mfma8_time(M, N, K, 16, 16, 2.75, 0.43, 54e3) : mfma8_time(M, N, K, 32, 32, 2.85, 1.0, 51e3);
      const double bytes = (double)(std::min(M, b) + std::min(N, b)) * K;
      return b == 16 ? 2.24 + mfma8_rounds(M, N, 16, 16) * (0.64 + bytes / 32.7e3) : 1.17 + mfma8_rounds(M, N, 32, 32) * (2.06 + bytes / 33.6e3);
   }
   if (!mfma8_direct_by_lines(b, M, N, K))
      return b == 16 ? mfma8_time(M, N, K, 16, 16, 2.5, 0.3, 41e3) : mfma8_time(M, N, K, 32, 32, 2.5, 0.45, 80e3);
   const double tiles = (double)((M + b - 1) / b) * ((N + b - 1) / b), ahead = std::min(K, 2048);
   return 2.5 + mfma8_rounds(M, N, b, b) * ((b == 16 ? 0.5 : 0.62) + 2.0 * b * (ahead / 120e3 + (K - ahead) / std::min(120e3, 20e6 / std::min(tiles, 256.0))));
}
// The general loop: tiles of 64 x 64, 128 x 64 and 128 x 128 (0, 1, 2).  By what it reads: rows that start on four bytes, rows that start anywhere, rows against a B that is
// transposed on its way (its k start anywhere, only they start on four bytes, both do), a convolution's pixels.  Each fitted to 201 .. 1000 products of 1 .. 8192 rows and columns (int8 and FP8; 124 layers): the choice among the tiles is 0.4 - 1.3 % above the
// fastest on average.  Between 64 x 64, of which a CU has one or two, and 128 x 128, of which the chip has too few, the tile in the middle: us, the better of those two -> 128 x 64,
// 1537 x 1000 x 777 with B transposed 10.8 -> 9.7, 1000 x 2000 x 500 8.9 -> 7.7, 2048^3 22.6 -> 19.4, 384 x 2976 x 3500 23.8 -> 19.5.  (A convolution's
// rows are worked out by each thread for its chunks: equal at best there.)
enum Mfma8Source { MFMA8_WORD_ROWS, MFMA8_ROWS, MFMA8_COLUMNS, MFMA8_WORD_COLUMNS, MFMA8_WORD_ROWS_COLUMNS, MFMA8_PIXELS };
inline Mfma8Source mfma8_source(bool a_words, bool b_words, bool columns)
{
   if (columns)
      return !b_words ? MFMA8_COLUMNS : a_words ? MFMA8_WORD_ROWS_COLUMNS : MFMA8_WORD_COLUMNS;
   return a_words && b_words ? MFMA8_WORD_ROWS : MFMA8_ROWS;
}
inline double mfma8_general_time(int M, int N, int K, Mfma8Source source, int *tile = nullptr)
{
   static constexpr struct {
      double fixed, tile, rate;
   } COSTS[6][3] = {{{3.0, 1.1, 58e3}, {1.6, 2.95, 58e3}, {1.5, 4.9, 52e3}},
                    {{3.1, 1.25, 47.6e3}, {1.5, 3.1, 51e3}, {1.5, 5.6, 42e3}},
                    {{3.5, 1.13, 32e3}, {1.9, 3.0, 37e3}, {0.0, 6.7, 33e3}},
                    {{3.65, 1.03, 36e3}, {2.1, 2.68, 43.8e3}, {0.5, 6.4, 33e3}},
                    {{3.36, 1.04, 37e3}, {1.9, 2.7, 49.8e3}, {0.3, 6.25, 38e3}},
                    {{3.3, 0.95, 139e3}, {1e9, 0.0, 1.0}, {8.6, 3.6, 41e3}}};
   double least = 1e30;
   for (int t = 0; t < 3; ++t) {
      const auto &c = COSTS[source][t];
      const double time = mfma8_time(M, N, K, t ? 128 : 64, t == 2 ? 128 : 64, c.fixed, c.tile, c.rate);
      if (time < least) {
         least = time;
         if (tile)
            *tile = t;
      }
   }
   return least;
}
inline double mfma8_ring_time(int M, int N, int K, int tile)
{
   return tile >= 128 ? mfma8_time(M, N, K, 128, 128, 3.5, 3.4, 67e3) : mfma8_time(M, N, K, 64, 64, 2.9, 0.6, 75e3);
}

// The general loop (any alignment, a convolution's input or plain rows, B either way).
template <class MMA, class ASRC, class BSRC, class EPI>
static int launch_mfma8_general(const LaunchCfg &lc, const ASRC &A, const BSRC &B, int M, int N, int K, const EPI &ep)
{
   constexpr bool PIXELS = !std::is_same_v<ASRC, StagedRows>;
   Mfma8Source source = MFMA8_PIXELS;
   bool by_words = false; // whether rows that start on no word are read as words
   if constexpr (!PIXELS) {
      const bool a = rows_of_words(A.base, A.ld), b = rows_of_words(B.base, B.ld);
      source = mfma8_source(a, b, BSRC::kTransposed);
      by_words = BSRC::kTransposed ? !a && StagedAnyRows::takes(A.ld) : !(a && b) && StagedAnyRows::takes(A.ld) && StagedAnyRows::takes(B.ld);
   }
   int tile = 0;
   mfma8_general_time(M, N, K, source, &tile);
   if (lc.tile)
      tile = lc.tile == 64 ? 0 : lc.tile == 164 ? PIXELS ? tile : 1 : lc.tile >= 128 ? 2 : tile;
   if (tile == 2)
      return launch_mfma8_staged<MMA, 128, 128, 128, 4, 2, 2, ASRC, BSRC, EPI>(lc, A, B, M, N, K, ep);
   auto smaller = [&](const auto &a, const auto &b) {
      typedef std::decay_t<decltype(a)> AT;
      typedef std::decay_t<decltype(b)> BT;
      if constexpr (!PIXELS) {
         if (tile == 1)
            return launch_mfma8_staged<MMA, 128, 64, 128, 4, 2, 2, AT, BT, EPI>(lc, a, b, M, N, K, ep);
      }
      return launch_mfma8_staged<MMA, 64, 64, 128, 2, 2, 2, AT, BT, EPI>(lc, a, b, M, N, K, ep);
   };
   if constexpr (!PIXELS) {
      if (by_words) {
         if constexpr (BSRC::kTransposed)
            return smaller(StagedAnyRows{A}, B);
         else
            return smaller(StagedAnyRows{A}, StagedAnyRows{B});
      }
   }
   return smaller(A, B);
}

// Chooses between the direct kernel (few rows or tiles, short rows), the pipelined kernels (aligned operands, K a multiple of 64) and the general one.
// `variant` selects a tuning alternative of the pipelined kernel (0 = default); -1 forces the general kernel.
template <class MMA, class EPI>
static int launch_mfma8_best(const LaunchCfg &lc, const int8_t *A, const int8_t *Bt, int M, int N, int K, int lda, int ldb,
                             const EPI &ep)
{
   const int force_tile = lc.tile, variant = lc.variant;
   typedef std::conditional_t<(MMA::KSTEP * 2 <= 64), DirectI8, DirectF8> Direct;
   const bool aligned = (lda % 16 == 0) && (ldb % 16 == 0) && (((uintptr_t)A & 15) == 0) && (((uintptr_t)Bt & 15) == 0);
   const bool ring = variant >= 0 && aligned && K >= 64 && K % 64 == 0 && (MMA::KSTEP * 2 <= 64 || K % 128 == 0);
   const bool lines = aligned && K % 16 == 0, words = rows_of_words(A, lda) && rows_of_words(Bt, ldb);
   const double t16 = mfma8_direct_time(M, N, K, 16, words, lines), t32 = mfma8_direct_time(M, N, K, 32, words, lines);
   const double others = ring ? mfma8_ring_time(M, N, K, pick_tile(M, N, 0)) : mfma8_general_time(M, N, K, mfma8_source(words, words, false));
   if (force_tile == 16 || K < 16 || (!force_tile && variant == 0 && t16 <= t32 && t16 < others))
      return launch_mfma8_direct<Direct, 1, 1, 8, 4, EPI>(lc, A, Bt, M, N, K, lda, ldb, ep);
   if (force_tile == 32 || (!force_tile && variant == 0 && t32 < others))
      return launch_mfma8_direct<Direct, 2, 2, 8, 2, EPI>(lc, A, Bt, M, N, K, lda, ldb, ep);
   if (!ring || force_tile == 164)
      return launch_mfma8_general<MMA, StagedRows, StagedRows, EPI>(lc, StagedRows{A, lda, M}, StagedRows{Bt, ldb, N}, M, N, K, ep);
   const int tile = pick_tile(M, N, force_tile);
   const bool k128 = (K % 128 == 0);
   if constexpr (MMA::KSTEP * 2 <= 64) {
      // Large products that divide into whole 256 x 256 tiles: the persistent kernel (512 asks for it by force)
      if ((force_tile == 512 || (!force_tile && variant == 0 && tile == 256)) && mfma8_persist_applies(A, Bt, M, N, K, lda, ldb, ep.elements_per_16_bytes()) &&
          ep.stores_plain_rows())
         return launch_mfma8_persist<MfmaI8x16, EPI>(lc, A, Bt, M, N, K, lda, ldb, ep);
      // Short reductions over many tiles: the 256 x 128 tile with a ring of three slabs fits twice on a CU, and one
      // workgroup's prologue and store overlap the other's K loop (8192 x 4096 x 512: 829 -> 1019 TOP/s, 8192 x 1024 x 1024:
      // 1003 -> 1091; no gain from K = 2048 on).  258 asks for it by force.
      const long long tiles_256x128 = (long long)((M + 255) / 256) * ((N + 127) / 128);
      if (force_tile == 258 || (!force_tile && variant == 0 && K <= 1024 && N >= 128 && tiles_256x128 >= 512))
         return launch_mfma8_dma_src<MMA, 256, 128, 64, 2, 2, 3, EPI, RowMajorRows, 2>(lc, RowMajorRows{A, lda}, Bt, M, N, K, ldb, ep);
   }
   if constexpr (MMA::KSTEP * 2 > 64) {
      // two K-steps per slab are the minimum: a 64-byte K-step needs 128-byte slabs, which `ring` has made sure of
      if ((force_tile == 512 || (!force_tile && variant == 0 && tile == 256)) && mfma8_persist_applies(A, Bt, M, N, K, lda, ldb, ep.elements_per_16_bytes()) &&
          ep.stores_plain_rows())
         return launch_mfma8_persist<MMA, EPI>(lc, A, Bt, M, N, K, lda, ldb, ep);
      switch (tile) {
      case 256:
         if (variant == 1)
            return launch_mfma8_dma<MMA, 256, 128, 128, 2, 2, 3, EPI>(lc, A, Bt, M, N, K, lda, ldb, ep);
         return launch_mfma8_pair<MMA, 256, 256, 64, 2, 2, 5, EPI>(lc, A, Bt, M, N, K, lda, ldb, ep);
      case 128: return launch_mfma8_dma<MMA, 128, 128, 128, 2, 2, 3, EPI>(lc, A, Bt, M, N, K, lda, ldb, ep);
      case 64: return launch_mfma8_dma<MMA, 64, 64, 128, 2, 2, 4, EPI>(lc, A, Bt, M, N, K, lda, ldb, ep);
      default: return fail(SOFIE_HIP_ERR_INVALID, "gemm: unknown tile %d", tile);
      }
   } else {
      switch (tile) {
      case 256:
         if (variant == 1 || !k128)
            return launch_mfma8_dma<MMA, 256, 256, 64, 2, 2, 4, EPI>(lc, A, Bt, M, N, K, lda, ldb, ep);
         return launch_mfma8_pair<MMA, 256, 256, 64, 2, 2, 5, EPI>(lc, A, Bt, M, N, K, lda, ldb, ep);
      case 128:
         if (variant == 1 || !k128)
            return launch_mfma8_dma<MMA, 128, 128, 64, 2, 2, 4, EPI>(lc, A, Bt, M, N, K, lda, ldb, ep);
         return launch_mfma8_dma<MMA, 128, 128, 128, 2, 2, 3, EPI>(lc, A, Bt, M, N, K, lda, ldb, ep);
      case 64:
         if (variant == 1 || !k128)
            return launch_mfma8_dma<MMA, 64, 64, 64, 2, 2, 4, EPI>(lc, A, Bt, M, N, K, lda, ldb, ep);
         return launch_mfma8_dma<MMA, 64, 64, 128, 2, 2, 4, EPI>(lc, A, Bt, M, N, K, lda, ldb, ep);
      default: return fail(SOFIE_HIP_ERR_INVALID, "gemm: unknown tile %d", tile);
      }
   }
}

// Whether a product whose B is stored [K,N] is better off with the general loop, which transposes B on its way into LDS, than
// with a launch that re-lays B out and the kernels above: that launch takes 3.6 us and 3.6 TB/s for the bytes it moves.  Fitted to 445 products; us, in the loop / re-laid out: 1537 x
// 1000 x 777 9.7 / 13.2, 2048^3 19.4 / 22.6, 100 x 4000 x 4000 17.9 / 23.6, 5113 x 3917 x 1376 93.8 / 74.0, 2432 x 1125 x 3968 37.4 / 31.0.
static bool mfma8_columns_preferred(const LaunchCfg &lc, const int8_t *A, int lda, const int8_t *B, int ldb, int M, int N, int K, bool aligned_behind)
{
   if (K < 16 || N < 16 || lc.tile == 16 || lc.tile == 32)
      return false;
   if (lc.tile == 164)
      return true;
   const bool lines = aligned_behind && K % 16 == 0, a_words = rows_of_words(A, lda), words_behind = a_words && K % 4 == 0;
   double behind = std::min(std::min(mfma8_direct_time(M, N, K, 16, words_behind, lines), mfma8_direct_time(M, N, K, 32, words_behind, lines)),
                            mfma8_general_time(M, N, K, mfma8_source(words_behind, words_behind, false)));
   if (aligned_behind && K >= 64 && K % 64 == 0)
      behind = std::min(behind, mfma8_ring_time(M, N, K, pick_tile(M, N, 0)));
   return lc.tile == 0 && lc.variant <= 0 && mfma8_general_time(M, N, K, mfma8_source(a_words, rows_of_words(B, ldb), true)) < 3.6 + (double)K * N / 1.8e6 + behind;
}

} // namespace sofie_hip

namespace sofie_hip {

// Convolution as one implicit GEMM: A is read through ConvRows (BK = 64 must divide the channels per group),
// Wp is the packed weight [N][K] with K = taps * Cg.
template <class EPI>
static int launch_mfma8_conv(const LaunchCfg &lc, const ConvRows &a, int Cg, const int8_t *Wp, int M, int N, int K, const EPI &ep)
{
   // requests for kernels of other layers, or that have turned this one down: no request here
   const int force_tile = lc.tile == 17 || lc.tile == 33 || lc.tile == 27 || lc.tile == 164 ? 0 : lc.tile;
   auto tiles = [&](int bm, int bn) { return (long long)((M + bm - 1) / bm) * ((N + bn - 1) / bn); };
   const bool pairs = (Cg % 128 == 0);
   int tile = force_tile;
   if (!tile)
      // Short reductions (a 3x3 convolution over 64 or 128 channels) spend as long in a tile's prologue and store as in its
      // K loop.  258 = the 256 x 128 tile with a ring of three slabs (72 KB) and 229 registers per lane: two workgroups
      // share a CU and one's prologue and store overlap the other's MFMAs (measured on 1M rows: K = 576, N = 128
      // 157 -> 134 us, K = 1152, N = 256 479 -> 355 us; K = 2304 is better off with the 256 x 256 tile, 760 vs 807 us).
      // 128 x 128 tiles also fit twice.  257 = the 256 x 128 tile with a ring of five, by request only.
      tile = (N > 128 && K > 1536 && tiles(256, 256) >= 256) ? 256
             : (N >= 128 && tiles(256, 128) >= 512)          ? 258
             : (N > 64 && tiles(128, 128) >= 192)            ? 128
                                                             : 64;
   // A small 3 x 3 layer (64 channels in, 128 out): weights resident in LDS, each tile's pixels fetched once with their halo.
   // 576 asks for it by force (and any other forced tile keeps it away).
   if ((force_tile == 576 || (!force_tile && lc.variant == 0 && tiles(256, 128) >= 256)) && conv_i8_resident_applies(a, Cg, Wp, M, N, K) &&
       ep.stores_plain_rows())
      return launch_conv_i8_resident<EPI>(lc, a, Wp, M, ep);
   // Whole 256 x 256 tiles, at least one per CU, and a store the register path handles (NHWC rows, or the plane sums of
   // planes that hold whole wave tiles): the persistent kernel.  512 asks for it by force.
   if ((force_tile == 512 || (!force_tile && lc.variant == 0 && tiles(256, 256) >= 256)) &&
       mfma8_persist_conv_applies(a, Wp, M, N, K, ep.elements_per_16_bytes(), !ep.stores_plain_rows()) &&
       (ep.stores_plain_rows() || ep.sums_rows_of_whole_wave_tiles(128)))
      return launch_mfma8_persist_src<MfmaI8x16, EPI, PersistConvRows>(lc, persist_conv_rows(a), Wp, M, N, K, K, ep);
   if (tile == 512 || tile == 576)
      tile = 256;
   switch (tile) {
   case 256:
      if (pairs)
         return launch_mfma8_pair_src<MfmaI8, 256, 256, 64, 2, 2, 5, EPI, ConvRows>(lc, a, Wp, M, N, K, K, ep);
      return launch_mfma8_dma_src<MfmaI8, 256, 256, 64, 2, 2, 4, EPI, ConvRows>(lc, a, Wp, M, N, K, K, ep);
   case 257:
      if (pairs)
         return launch_mfma8_pair_src<MfmaI8, 256, 128, 64, 2, 2, 5, EPI, ConvRows>(lc, a, Wp, M, N, K, K, ep);
      return launch_mfma8_dma_src<MfmaI8, 256, 128, 64, 2, 2, 4, EPI, ConvRows>(lc, a, Wp, M, N, K, K, ep);
   case 258: return launch_mfma8_dma_src<MfmaI8, 256, 128, 64, 2, 2, 3, EPI, ConvRows, 2>(lc, a, Wp, M, N, K, K, ep);
   case 128: return launch_mfma8_dma_src<MfmaI8, 128, 128, 64, 2, 2, 4, EPI, ConvRows>(lc, a, Wp, M, N, K, K, ep);
   case 64: return launch_mfma8_dma_src<MfmaI8, 64, 64, 64, 2, 2, 4, EPI, ConvRows>(lc, a, Wp, M, N, K, K, ep);
   default: return fail(SOFIE_HIP_ERR_INVALID, "conv: unknown tile %d", force_tile);
   }
}

} // namespace sofie_hip
