// TileOrder of sofie_amd/csrc/tile_order.hpp against the order in plain divisions: every workgroup of lists that can be walked, and workgroups spread over those of up to 2^31 - 1 tiles
// (a launch that is not the first one's among them).  Prints the workgroups compared and those that differ.
#include "tile_order.hpp"
#include <cstdio>
#include <cstdlib>
#include <vector>
using sofie_hip::TileOrder;

struct Place {
   long long tm, tn, product;
};
static Place plain(long long bid, long long z, long long tiles_m, long long tiles_n, int mode, bool listed, long long batch)
{
   const long long one = tiles_m * tiles_n, all = listed ? one * batch : one;
   long long id = bid;
   if (!(mode & 0x100))
      id = bid % 8 * (all / 8) + (bid % 8 < all % 8 ? bid % 8 : all % 8) + bid / 8;
   const long long product = listed ? id / one : z, rows = mode & 0xff ? mode & 0xff : 1;
   id %= one;
   const long long first = id / (rows * tiles_n) * rows, here = tiles_m - first < rows ? tiles_m - first : rows, in = id % (rows * tiles_n);
   return Place{first + in % here, in / here, product};
}

int main()
{
   long long compared = 0, bad = 0;
   auto check = [&](const TileOrder &o, long long bid, int z, long long tiles_m, long long tiles_n, int mode, long long batch) {
      int tm = -1, tn = -1, product = -1;
      o.place_of<true>((int)bid, z, tm, tn, product);
      const Place p = plain(bid, z, tiles_m, tiles_n, mode, o.tiles != 0, batch);
      ++compared;
      int tm2 = -1, tn2 = -1, product2 = -1;
      o.place_of<false>((int)bid, z, tm2, tn2, product2);
      if (tm2 != tm || tn2 != tn || product2 != product)
         ++bad;
      if (tm != p.tm || tn != p.tn || product != p.product)
         ++bad;
      return Place{tm, tn, product};
   };
   const int modes[] = {0, 1, 3, 4, 255, 0x100, 0x104};
   for (int mode : modes)
      for (int tiles_m = 1; tiles_m <= 40; ++tiles_m)
         for (int tiles_n = 1; tiles_n <= 11; ++tiles_n)
            for (int batch : {1, 2, 7, 8, 33}) {
               const TileOrder o(tiles_m, tiles_n, mode, batch);
               std::vector<char> seen((size_t)tiles_m * tiles_n * batch);
               for (long long bid = 0; bid < o.workgroups(batch); ++bid)
                  for (int z = 0; z < (int)o.depth(batch); ++z) {
                     const Place p = check(o, bid, z, tiles_m, tiles_n, mode, batch);
                     if (p.tm < 0 || p.tm >= tiles_m || p.tn < 0 || p.tn >= tiles_n || p.product < 0 || p.product >= batch)
                        ++bad;
                     else if (seen[(p.product * tiles_m + p.tm) * tiles_n + p.tn]++)
                        ++bad;
                  }
            }
   // long lists: one product of many tiles, a batch in the list, and a batch that does not fit it and is the grid's z
   const long long longest[][3] = {{0x7fffffff, 1, 1}, {1, 0x7fffffff, 1}, {46340, 46340, 1}, {3, 715827882, 1}, {33554432, 63, 1}, {1000, 1000, 2147}, {7, 5, 61356675}, {1, 1, 0x7fffffff},
                                   {8388607, 255, 1}, {100000, 3, 65535}, {46341, 46340, 1}, {5, 3, 0x7fffffff}, {46340, 46339, 2}};
   unsigned long long state = 12345;
   for (int mode : modes)
      for (auto &l : longest) {
         if (l[0] * l[1] > 0x7fffffffLL)
            continue; // refused before a launch
         const TileOrder o((int)l[0], (int)l[1], mode, (int)l[2]);
         const long long n = o.workgroups((int)l[2]), depth = o.depth((int)l[2]);
         if (n > 0x7fffffffLL || (o.tiles == 0) != (l[2] == 1 || l[0] * l[1] * l[2] > 0x7fffffffLL))
            ++bad;
         for (int i = 0; i < 200000; ++i) {
            state = state * 6364136223846793005ull + 1442695040888963407ull;
            const long long bid = i < 100 ? i % n : i < 200 ? (n - 1 - (i - 100) % n) : (long long)((state >> 20) % (unsigned long long)n);
            check(o, bid, (int)((state >> 33) % (unsigned long long)depth), l[0], l[1], mode, l[2]);
         }
      }
   printf("%lld %lld\n", compared, bad);
   return bad != 0;
}
