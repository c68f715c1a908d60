// Which tile of which product a workgroup takes, and the divisions by run-time values that this needs.  Plain arithmetic: a check on the CPU compiles it too.
#pragma once
#include <algorithm>

#if defined(__HIPCC__)
#define SOFIE_ORDER_FN __host__ __device__ __forceinline__
#else
#define SOFIE_ORDER_FN inline
#endif

namespace sofie_hip {

// Index arithmetic by an extent that the launch knows: a multiplication while every index fits 31 bits (a 64-bit division by a
// run-time value is some hundred instructions per element, several times what the memory traffic of most kernels leaves room for).
struct Divisor31 {
   // with s = ceil(log2 d) and mul = ceil(2^(31 + s) / d), mul d - 2^(31 + s) < 2^s: below 2^31 the error of n mul / 2^(31 + s) is
   // smaller than 1 / d, and mul < 2^32
   unsigned d, mul, shift;
   explicit Divisor31(long long extent) : d((unsigned)extent), shift(0)
   {
      while ((1ull << shift) < d)
         ++shift;
      mul = (unsigned)(((1ull << (31 + shift)) + d - 1) / d);
   }
   typedef unsigned index;
   SOFIE_ORDER_FN index over(index n) const
   {
#if defined(__HIP_DEVICE_COMPILE__)
      return __umulhi(2 * n, mul) >> shift;
#else
      return (index)((unsigned long long)(2 * n) * mul >> 32) >> shift;
#endif
   }
};

// Tiles in bands of `mode & 0xff` rows, column by column inside a band, and workgroups regrouped so that the eight XCDs, which take them in turn, each have a run of them (not
// with `mode & 0x100`).  The tiles are known to the host, which works out the divisors: four divisions by run-time values are 400 cycles that a small product waits for before its
// first load.  What is left is the trip to the scalar cache for the fields, and a branch around some of them makes it two: 0.05 us of a small product's 2.5.  So a single column of tiles has no way of
// its own (one without the divisions made products of several columns 1.2 % slower, int8 and FP8 0.5 %).  The products of a batch are laid side by side in the same
// list, so that those of one product meet in one XCD's L2: 96 products of 128 x 128 x 64 read 18 MB through eight L2s, whose operands are 6.
struct TileOrder {
   int tiles_m, tiles_n, band, last; // last: rows of the last band
   int per, rem;                     // workgroups of an XCD, XCDs with one more; per < 0: no regrouping
   int tiles;                        // of a product of a batch; 0: the products are the grid's z
   Divisor31 by_width, by_band, by_last, by_tiles;
   TileOrder(int tiles_m, int tiles_n, int mode, int batch = 1)
      : tiles_m(tiles_m), tiles_n(tiles_n), band(std::max(1, std::min(mode & 0xff, tiles_m))), last(tiles_m % band ? tiles_m % band : band), by_width((long long)band * tiles_n),
        by_band(band), by_last(last), by_tiles(1)
   {
      const long long one = (long long)tiles_m * tiles_n, all = one * batch;
      tiles = batch > 1 && all <= 0x7fffffffLL ? (int)one : 0;
      if (tiles)
         by_tiles = Divisor31(tiles);
      per = mode & 0x100 ? -1 : (int)((tiles ? all : one) / 8);
      rem = (int)((tiles ? all : one) % 8);
   }
   long long workgroups(int batch) const { return (long long)tiles_m * tiles_n * (tiles ? batch : 1); } // of the grid's x
   unsigned depth(int batch) const { return tiles ? 1u : (unsigned)batch; }                            // its z
   // BATCHES: for the fp32 kernels, without a branch (above): 3 % of a small product of a batch.  The int8 and FP8 kernels, which have no batches, take 1 % longer without it.
   template <bool BATCHES>
   SOFIE_ORDER_FN void place_of(int bid, int z, int &tm, int &tn, int &product) const
   {
      int id = bid;
      if (per >= 0) {
         const int xcd = bid & 7;
         id = xcd * per + (xcd < rem ? xcd : rem) + (bid >> 3);
      }
      product = z;
      if (BATCHES) {
         const int listed = (int)by_tiles.over((unsigned)id);
         product = tiles ? listed : z;
         id -= listed * tiles;
      } else if (tiles) {
         product = (int)by_tiles.over((unsigned)id);
         id -= product * tiles;
      }
      const int group = (int)by_width.over((unsigned)id), first = group * band, in = id - group * band * tiles_n;
      const bool whole = first + band <= tiles_m;
      tn = whole ? (int)by_band.over((unsigned)in) : (int)by_last.over((unsigned)in);
      tm = first + in - tn * (whole ? band : last);
   }
#if defined(__HIPCC__)
   __device__ __forceinline__ void place(int bid, int &tm, int &tn, int &product) const { place_of<true>(bid, blockIdx.z, tm, tn, product); }
   __device__ __forceinline__ void place(int bid, int &tm, int &tn) const
   {
      int product;
      place_of<false>(bid, 0, tm, tn, product);
   }
#endif
};

} // namespace sofie_hip
