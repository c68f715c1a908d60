// fp32 Gemm / MatMul and fp32 convolution (implicit GEMM) with the bias + activation epilogue fused into the store: the entry
// points and the choice among the kernels of f32_mfma.hpp, and the kernel that runs a chain of small products in one launch.
#include "f32_conv3x3_few.hpp"
#include "f32_conv3x3_split.hpp"
#include <algorithm>
#include <cmath>

namespace sofie_hip {

// ---- a chain of small products in one launch -----------------------------------------------------------------
// Layer l+1 reads what layer l wrote (an MLP at small batch): per layer launches cost more than the arithmetic, so one
// workgroup takes RB rows through every layer, the rows of activations staying in LDS between layers (each layer's
// output is also written to its Y, as separate launches would).  The weights stream from L2 once per workgroup:
//   transB (W stored [N][K], the ONNX export of a Linear layer): groups of lanes take an output each, 16 bytes of its row a lane, then the partial sums are folded across the
//     lanes (2 rows through 304-16-32-193 7.5 -> 6.1 us, 60 through 160-16-16-176 7.0 -> 5.9, 64 through 784-128-64-10, one launch, 9.7 -> 9.3; rows of W that do not start
//     on 16 bytes: a wave takes 4 outputs at a time, 256 bytes of each);
//   else (W stored [K][N]): a thread owns output n and walks k (lanes read consecutive n of one weight row); up to 512 outputs, whose threads alone
//     would leave the others idle, k is dealt out over groups of threads, and their sums are added up through LDS (39 rows through
//     256-137-1800-17: 28.6 -> 19.9 us, most of it by taking the first layer into the chain, whose waves were one in eight before; 4 rows through
//     128-112-32-9 9.3 -> 8.1).
struct ChainLayerArgs {
   const float *B;
   long long ldb;
   int transB, N, K;
   float *Y;
   long long ldy;
   F32Epilogue ep;
};
struct ChainArgs {
   int count, M;
   const float *A;
   long long lda;
   ChainLayerArgs layer[SOFIE_MAX_GEMM_CHAIN];
};

// 16 waves per workgroup: what a layer costs is the round trips to L2 for its weights, and the waves' loads overlap
constexpr int CHAIN_THREADS = 1024;

// A thread's column of W (its floats `ldb` apart) times RB rows in LDS, for k0 <= k < k1, sixteen loads in flight.
template <int RB>
__device__ __forceinline__ void chain_walk(float (&acc)[RB], const float *column, long long ldb, const float *in, int width, int k0, int k1)
{
   int k = k0;
   const float *w = column + k * ldb;
   auto some = [&](auto count) {
      constexpr int U = decltype(count)::value;
      for (; k + U <= k1; k += U) {
         float v[U];
#pragma unroll
         for (int u = 0; u < U; ++u) {
            v[u] = *w;
            w += ldb;
         }
         if constexpr (U > 1)
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
         for (int u = 0; u < U; ++u)
#pragma unroll
            for (int r = 0; r < RB; ++r)
               acc[r] = fmaf(v[u], in[r * width + k + u], acc[r]);
      }
   };
   some(std::integral_constant<int, 16>{});
   some(std::integral_constant<int, 4>{});
   some(std::integral_constant<int, 1>{});
}

// The sums of J * 64 / G outputs from n0 on, rows of W on 16 bytes: G lanes an output (as many as its row has 16-byte pieces, up to 64), so that a wave's load brings 64 / G rows, and
// two pieces of J outputs are on their way in every lane.  Lane j of group s of G lanes ends up with output n0 + j 64 / G + s.
// behind() is called once, with the first of them on their way.
template <int RB, int G, int J, class F>
__device__ __forceinline__ void chain_rows(float (&sums)[RB], const ChainLayerArgs &L, int n0, const float *in, int width, int lane, F &&behind)
{
   constexpr int P = 64 / G;
   const int N = L.N, pieces = L.K / 4, sub = lane / G, l = lane % G;
   const v4f *w[J]; // rows of W past N are read as row N - 1 and their sums dropped
#pragma unroll
   for (int j = 0; j < J; ++j)
      w[j] = (const v4f *)(L.B + (long long)(n0 + j * P + sub < N ? n0 + j * P + sub : N - 1) * L.ldb);
   float acc[J][RB];
#pragma unroll
   for (int j = 0; j < J; ++j)
#pragma unroll
      for (int r = 0; r < RB; ++r)
         acc[j][r] = 0.0f;
   constexpr int U = G < 64 ? 1 : 2; // rows of fewer than 64 pieces are read at once
#pragma unroll 1
   for (int k = l; k - l < pieces; k += U * G) {
      v4f v[U][J];
#pragma unroll
      for (int u = 0; u < U; ++u)
         if (k - l + u * G < pieces) // for some lane
#pragma unroll
            for (int j = 0; j < J; ++j)
               v[u][j] = w[j][k + u * G < pieces ? k + u * G : 0];
      if (k == l)
         behind();
#pragma unroll
      for (int u = 0; u < U; ++u)
         if (k + u * G < pieces) {
#pragma unroll
            for (int r = 0; r < RB; ++r) {
               const v4f x = *(const v4f *)(in + r * width + 4 * (k + u * G));
#pragma unroll
               for (int j = 0; j < J; ++j)
#pragma unroll
                  for (int e = 0; e < 4; ++e)
                     acc[j][r] = fmaf(v[u][j][e], x[e], acc[j][r]);
            }
         }
   }
#pragma unroll
   for (int r = 0; r < RB; ++r) {
      sums[r] = 0.0f;
#pragma unroll
      for (int j = 0; j < J; ++j) {
         const float sum = sum_over_lanes(acc[j][r], G);
         sums[r] = l == j ? sum : sums[r];
      }
   }
}

// Rows of W that chain_rows reads.
__host__ __device__ __forceinline__ bool chain_layer_by_rows(const ChainLayerArgs &L) { return L.transB && L.K % 4 == 0 && L.ldb % 4 == 0 && ((uintptr_t)L.B & 15) == 0; }

// ROWS: some layer goes through chain_rows.  Its code costs the others' registers (92 - 112 vector registers and up to 29 scalars spilled, 64 - 92 and up to two without): layers
// with W stored [K][N] in the kernel with it / without, M x K-..-N, 40 x 256-128-128-1123-11 15.7 / 15.0 us, 3 x 4-128-5 5.10 / 4.98.
template <int RB, bool ROWS>
__global__ __launch_bounds__(CHAIN_THREADS) void gemm_chain_f32_kernel(ChainArgs a, int width)
{
   // two buffers of RB rows x width, RB sums per thread; chain_rows reads 16 bytes at a time: width is a multiple of four
   extern __shared__ __attribute__((aligned(16))) float chain_lds[];
   const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
   const int m0 = blockIdx.x * RB;
   const int rows = (a.M - m0) < RB ? (a.M - m0) : RB;
   float *in = chain_lds, *out = chain_lds + RB * width;
   // rows beyond the matrix are kept at zero so that the loops below need no row test
   if (rows < RB) {
      for (int i = t; i < 2 * RB * width; i += CHAIN_THREADS)
         chain_lds[i] = 0.0f;
      __syncthreads();
   }
   const int K0 = a.layer[0].K;
   for (int r = 0; r < rows; ++r)
      for (int k = t; k < K0; k += CHAIN_THREADS)
         in[r * width + k] = a.A[(long long)(m0 + r) * a.lda + k];
   __syncthreads();
   for (int l = 0; l < a.count; ++l) {
      const ChainLayerArgs &L = a.layer[l];
      const int N = L.N, K = L.K;
      const float *__restrict__ B = L.B;
      if (ROWS && chain_layer_by_rows(L)) {
         // four outputs a wave, sixteen where one pass would not do and rows are short enough for as many loads
         const int g_log2 = K <= 64 ? 4 : K <= 128 ? 5 : 6, j_log2 = N > 64 ? 2 : g_log2 - 4, per_wave = 64 >> g_log2 << j_log2;
         for (int n0 = wave * per_wave; n0 < N; n0 += CHAIN_THREADS / 64 * per_wave) {
            const int l = lane & ((1 << g_log2) - 1), n = n0 + (l << (6 - g_log2)) + (lane >> g_log2);
            const bool mine = l >> j_log2 == 0 && n < N;
            F32Added added[RB];
            auto ask = [&]() {
#pragma unroll
               for (int r = 0; r < RB; ++r)
                  added[r] = mine && r < rows ? f32_look_up(L.ep, m0 + r, n) : F32Added{0.0f, 0.0f};
            };
            float sums[RB];
            if (g_log2 == 6)
               chain_rows<RB, 64, 4>(sums, L, n0, in, width, lane, ask);
            else if (g_log2 == 5 && j_log2 == 2)
               chain_rows<RB, 32, 4>(sums, L, n0, in, width, lane, ask);
            else if (g_log2 == 5)
               chain_rows<RB, 32, 2>(sums, L, n0, in, width, lane, ask);
            else if (j_log2 == 2)
               chain_rows<RB, 16, 4>(sums, L, n0, in, width, lane, ask);
            else
               chain_rows<RB, 16, 1>(sums, L, n0, in, width, lane, ask);
#pragma unroll
            for (int r = 0; r < RB; ++r)
               if (mine && r < rows) {
                  const float v = f32_finish(L.ep, sums[r], added[r]);
                  out[r * width + n] = v;
                  L.Y[(long long)(m0 + r) * L.ldy + n] = v;
               }
         }
      } else if (L.transB) {
         for (int n0 = wave * 4; n0 < N; n0 += CHAIN_THREADS / 16) {
            float acc[4][RB];
#pragma unroll
            for (int j = 0; j < 4; ++j)
#pragma unroll
               for (int r = 0; r < RB; ++r)
                  acc[j][r] = 0.0f;
            // rows of W past N are read as row N-1 and their sums dropped
            const float *w0 = B + (long long)(n0 + 0 < N ? n0 + 0 : N - 1) * L.ldb;
            const float *w1 = B + (long long)(n0 + 1 < N ? n0 + 1 : N - 1) * L.ldb;
            const float *w2 = B + (long long)(n0 + 2 < N ? n0 + 2 : N - 1) * L.ldb;
            const float *w3 = B + (long long)(n0 + 3 < N ? n0 + 3 : N - 1) * L.ldb;
            // (issuing the loads of eight guarded k-positions at once instead, with no remainder loop, measured slower)
#pragma unroll 8
            for (int k = lane; k < K; k += 64) {
               const float w[4] = {w0[k], w1[k], w2[k], w3[k]};
#pragma unroll
               for (int r = 0; r < RB; ++r) {
                  const float x = in[r * width + k];
#pragma unroll
                  for (int j = 0; j < 4; ++j)
                     acc[j][r] = fmaf(w[j], x, acc[j][r]);
               }
            }
#pragma unroll
            for (int j = 0; j < 4; ++j)
#pragma unroll
               for (int r = 0; r < RB; ++r)
                  acc[j][r] = sum_over_lanes(acc[j][r]);
            // every lane now holds the 4 x RB sums: lane j finishes output n0 + j
            const int n = n0 + lane;
            if (lane < 4 && n < N) {
#pragma unroll
               for (int r = 0; r < RB; ++r) {
                  if (r < rows) {
                     const float s = lane == 0 ? acc[0][r] : lane == 1 ? acc[1][r] : lane == 2 ? acc[2][r] : acc[3][r];
                     const float v = f32_epilogue(L.ep, s, m0 + r, n);
                     out[r * width + n] = v;
                     L.Y[(long long)(m0 + r) * L.ldy + n] = v;
                  }
               }
            }
         }
      } else if (N <= CHAIN_THREADS / 2) {
         const int shift = N <= 64 ? 6 : N <= 128 ? 7 : N <= 256 ? 8 : 9, span = 1 << shift, parts = CHAIN_THREADS >> shift;
         const int n = t & (span - 1), part = t >> shift, per = (K + parts - 1) / parts, k1 = (part + 1) * per < K ? (part + 1) * per : K;
         float acc[RB];
#pragma unroll
         for (int r = 0; r < RB; ++r)
            acc[r] = 0.0f;
         chain_walk<RB>(acc, B + (n < N ? n : N - 1), L.ldb, in, width, part * per, k1); // columns past N are the last one's, and their sums dropped
         float *sums = chain_lds + 2 * RB * width;
#pragma unroll
         for (int r = 0; r < RB; ++r)
            sums[r * CHAIN_THREADS + t] = acc[r];
         __syncthreads();
#pragma unroll
         for (int r = 0; r < RB; ++r) {
            // row r is finished by the threads of group r % parts
            if (part == r % parts && r < rows && n < N) {
               float s = sums[r * CHAIN_THREADS + n];
               for (int p = 1; p < parts; ++p)
                  s += sums[r * CHAIN_THREADS + (p << shift) + n];
               const float v = f32_epilogue(L.ep, s, m0 + r, n);
               out[r * width + n] = v;
               L.Y[(long long)(m0 + r) * L.ldy + n] = v;
            }
         }
      } else {
         for (int n = t; n < N; n += CHAIN_THREADS) {
            float acc[RB];
#pragma unroll
            for (int r = 0; r < RB; ++r)
               acc[r] = 0.0f;
            chain_walk<RB>(acc, B + n, L.ldb, in, width, 0, K);
#pragma unroll
            for (int r = 0; r < RB; ++r) {
               if (r < rows) {
                  const float v = f32_epilogue(L.ep, acc[r], m0 + r, n);
                  out[r * width + n] = v;
                  L.Y[(long long)(m0 + r) * L.ldy + n] = v;
               }
            }
         }
      }
      __syncthreads();
      float *tmp = in;
      in = out;
      out = tmp;
   }
}

} // namespace sofie_hip

namespace sofie_hip {

// The kernel for a product of M x N x K, `batch` times: the one whose time, estimated from what each was measured to do, is the
// shortest.  A CU multiplies a 32 x 32 block by 32 k in 0.107 us at best.  A tile kernel takes a launch, `alone` per slab of 32 k where its tiles wait for their
// loads, and `slab` and `tile` in as many rounds as the tiles need over 256 CUs; operands that come float by float (ragged) take longer.  The direct
// kernel takes a launch, `alone` per 128 k (16 of each wave) and `row` for every sixteenth of its 16 rows or, where there are many tiles, `slab` per 16 k and 256
// tiles, and `tile` per 256 tiles; where both operands come line by line through its ring, 78 KB/us a CU and 0.48 us for the first 256 tiles, 73 and 0.49 a tile where
// there are more.  Fitted to 1220 products of each kind of 16-byte loads, and to 1384 that come float by float, 1 .. 4096 rows, K = 8 .. 2048; on 1500 other products on average 0.15 %
// (float by float), 0.2 % (float by float along k), 0.13 % and 0.11 % (16 bytes, along k) above the best kernel's time, 18 % the most.  (With the costs of a direct kernel that branched
// around its loads, those float by float were 7.8 and 9.5 % above, 90 % the most: 291 x 6 x 1532 11.2 us, now 5.9; 2 x 4 x 1991 11.6, now 6.3.  The two larger tiles' costs are fitted to
// 2700 products of either float by float kind, half of them batches of up to 128: on 1000 others each 0.12 and 0.19 % above the best, batches 0.54 and 0.41 %, 31 % the most; fitted to
// single products alone they had batches 1.3 % above, 2.1 times the most: 63 products of 693 x 163 x 19 47 us on tiles of 128, now 24 on 64.  Launches take 0.4 us more or less from one
// card to another; these are of the shorter kind, as the chain's costs below are.)
enum F32Tile { F32_CONV3X3_FEW = 3004, F32_CONV3X3_32 = 3032, F32_CONV3X3_64 = 3064, F32_CONV3X3_128 = 3128, F32_CONV3X3_SPLIT_128 = 4128, F32_CONV3X3_SPLIT_256 = 4256, F32_DIRECT = 16, F32_TILE_32 = 32, F32_TILE_64x32 = 62, F32_TILE_64 = 64, F32_TILE_128x32 = 126, F32_TILE_128 = 128 };
// Pixels of a tile of the 3 x 3 convolution kernels; 0 for any other kernel.
static int conv3x3_pixels(int tile)
{
   switch (tile) {
   case F32_CONV3X3_32: return 32;
   case F32_CONV3X3_64: return 64;
   case F32_CONV3X3_128:
   case F32_CONV3X3_SPLIT_128: return 128;
   case F32_CONV3X3_SPLIT_256: return 256;
   default: return 0;
   }
}
enum F32Loads { F32_LOADS_RAGGED, F32_LOADS_RAGGED_LINES, F32_LOADS_WIDE, F32_LOADS_LINES }; // float by float, 16 bytes; lines: along k of both operands
static F32Loads f32_loads(bool wide, bool lines) { return wide ? lines ? F32_LOADS_LINES : F32_LOADS_WIDE : lines ? F32_LOADS_RAGGED_LINES : F32_LOADS_RAGGED; }
static int pick_f32_tile(int M, int N, int K, int batch, F32Loads loads, double *time_us = nullptr)
{
   struct Cost {
      double launch, alone, slab, tile, row;
   };
   struct Costs {
      Cost direct, tile32, tile64x32, tile64, tile128;
   };
   static constexpr Costs COSTS[] = { // by F32Loads
      {{2.75, 0.23, 0.063, 0.40, 0.092}, {3.12, 0.15, 0.152, 0.52}, {3.44, 0.32, 0.325, 0.94}, {3.54, 0.59, 0.566, 1.44}, {5.13, 0.05, 2.48, 4.64}},
      {{2.75, 0.26, 0.066, 0.41, 0.080}, {3.11, 0.14, 0.144, 0.55}, {3.36, 0.25, 0.313, 0.99}, {3.62, 0.195, 0.504, 1.37}, {5.88, 2.25, 2.12, 3.49}},
      {{3.09, 0.31, 0.068, 0.38, 0.038}, {3.06, 0.09, 0.134, 0.53}, {3.64, 0.14, 0.262, 0.78}, {3.14, 0.34, 0.504, 1.53}, {5.94, 0.03, 2.01, 3.56}},
      {{}, {2.78, 0.10, 0.125, 0.49}, {3.45, 0.18, 0.251, 0.66}, {2.68, 0.48, 0.478, 1.47}, {5.36, 0.03, 1.80, 3.55}}};
   auto tiles = [&](int bm, int bn) { return std::ceil((double)M / bm) * std::ceil((double)N / bn) * batch; };
   const double slabs = std::ceil(K / 32.0), steps = std::ceil(K / 16.0), each = tiles(16, 16) / 256.0;
   const Costs &costs = COSTS[loads];
   int best = F32_DIRECT;
   double least;
   if (loads == F32_LOADS_LINES) {
      const double rounds = each <= 1.0 ? 1.0 : 0.5 * (each + std::ceil(each));
      least = 2.36 + rounds * (each <= 1.0 ? 0.48 + 128.0 * K / 78e3 : 0.49 + 128.0 * K / 73e3);
   } else {
      const Cost &c = costs.direct;
      least = c.launch + std::max((c.alone + c.row * std::min(M, 16) / 16.0) * std::ceil(steps / 8.0), c.slab * each * steps) + c.tile * each;
   }
   auto offer = [&](int tile, int bm, int bn, const Cost &c) {
      const double t = c.launch + std::max(slabs * c.alone, std::ceil(tiles(bm, bn) / 256.0) * (slabs * c.slab + c.tile));
      if (t < least)
         least = t, best = tile;
   };
   offer(F32_TILE_32, 32, 32, costs.tile32);
   offer(F32_TILE_64x32, 64, 32, costs.tile64x32);
   offer(F32_TILE_64, 64, 64, costs.tile64);
   offer(F32_TILE_128, 128, 128, costs.tile128);
   if (time_us)
      *time_us = least;
   return best;
}
// The same for a convolution, whose slabs wait for their gather: a load instruction brings 64 floats from three or four lines, and a
// vector L1 takes four cycles per line.  A slab of 32 k takes 0.42 us (64 x 32 tiles), 0.60 (64 x 64: as many image elements for twice
// the products) and 0.92 (128 x 32).  The direct kernel decomposes every k by itself: for few tiles only.
static int pick_f32_conv_tile(int M, int N, int K, int group)
{
   auto tiles = [&](int bm, int bn) { return std::ceil((double)M / bm) * std::ceil((double)N / bn) * group; };
   const double slabs = std::ceil(K / 32.0);
   auto tiled = [&](int bm, int bn, double launch, double slab, double tile) { return launch + std::ceil(tiles(bm, bn) / 256.0) * (slabs * slab + tile); };
   int best = F32_DIRECT;
   double least = 5.3 + tiles(16, 16) / 256.0 * (0.9 + 0.17 * std::ceil(K / 16.0));
   auto offer = [&](int tile, double t) {
      if (t < least)
         least = t, best = tile;
   };
   offer(F32_TILE_64x32, tiled(64, 32, 6.5, 0.42, 1.15));
   offer(F32_TILE_64, tiled(64, 64, 6.5, 0.60, 2.4));
   offer(F32_TILE_128x32, tiled(128, 32, 6.0, 0.92, 1.5));
   return best;
}

template <class ASRC, class BSRC, class STORE>
static int launch_f32_product(sofie_hip_ctx *ctx, const ASRC &A, const BSRC &B, const STORE &out, int M, int N, int K, int batch, long long strideA, long long strideB)
{
   hipStream_t s = ctx->stream;
   int tile = ctx->opt.f32_tile;
   if (ctx->opt.f32_skinny == 1 || K == 0 || !A.in_buffers() || !B.in_buffers())
      tile = F32_DIRECT;
   else if (ctx->opt.f32_skinny == 0 && !tile)
      tile = F32_TILE_64;
   constexpr bool CONV = ASRC::kLeastRows == 64;
   if (!tile)
      tile = CONV ? pick_f32_conv_tile(M, N, K, batch) : pick_f32_tile(M, N, K, batch, f32_loads(ASRC::VEC == 4 && BSRC::VEC == 4, ASRC::KC && BSRC::KC));
   if (conv3x3_pixels(tile) || tile == F32_CONV3X3_FEW || (CONV ? tile == F32_TILE_32 || tile == F32_TILE_128 : tile == F32_TILE_128x32))
      tile = F32_TILE_64; // a request for a tile that the other kind of product has
   if constexpr (CONV) {
      switch (tile) {
      case F32_TILE_64x32: return launch_f32_tile<ASRC, BSRC, STORE, 64, 32, 32, 2, 1, 2, 4>(s, A, B, out, M, N, K, batch, strideA, strideB);
      case F32_TILE_128x32: return launch_f32_tile<ASRC, BSRC, STORE, 128, 32, 16, 4, 1, 1, 4>(s, A, B, out, M, N, K, batch, strideA, strideB);
      }
   } else {
      switch (tile) {
      case F32_TILE_32: return launch_f32_tile<ASRC, BSRC, STORE, 32, 32, 32, 1, 1, 4, 4>(s, A, B, out, M, N, K, batch, strideA, strideB);
      case F32_TILE_64x32: return launch_f32_tile<ASRC, BSRC, STORE, 64, 32, 32, 2, 1, 2, 4>(s, A, B, out, M, N, K, batch, strideA, strideB);
      case F32_TILE_128: return launch_f32_tile<ASRC, BSRC, STORE, 128, 128, 16, 2, 2, 1, 4>(s, A, B, out, M, N, K, batch, strideA, strideB);
      }
   }
   switch (tile) {
   case F32_DIRECT: return launch_f32_direct<ASRC, BSRC, STORE, 1, 1, 8, 4>(s, A, B, out, M, N, K, batch, strideA, strideB);
   case F32_TILE_64: return launch_f32_tile<ASRC, BSRC, STORE, 64, 64, 32, 2, 2, 2, 4>(s, A, B, out, M, N, K, batch, strideA, strideB);
   default: return fail(SOFIE_HIP_ERR_INVALID, "fp32 product: unknown tile %d", tile);
   }
}

// The kernel of f32_conv3x3.hpp for a convolution it takes (*taken tells): faster than the gathering kernels at every size measured, if only
// by the launch where a few tiles of one slab are all there is.
static int launch_f32_conv3x3(sofie_hip_ctx *ctx, const float *X, const F32ConvShape &s, const float *W, const F32ConvStore &out, int images, int M, int group, bool *taken)
{
   const int K = s.Cg * 9, N = out.Cout_g, force = ctx->opt.f32_tile;
   *taken = false;
   if (s.kd != 1 || s.D != 1 || s.kh != 3 || s.kw != 3 || s.stride_h != 1 || s.stride_w != 1 || s.dil_h != 1 || s.dil_w != 1 || ctx->opt.f32_skinny >= 0)
      return SOFIE_HIP_OK;
   // the images a patch touches, from the first one's base, within a buffer; channels within its scalar offset
   const long long plane = (long long)s.H * s.W, most = F32_CONV3X3_PATCH / ((long long)(s.OW + 2) * (s.OH + 2)) + 2;
   if ((most * s.C + s.Cg) * plane * 4 >= F32_BUFFER_BYTES || 128LL * K * 4 >= F32_BUFFER_BYTES)
      return SOFIE_HIP_OK;
   const bool vec = ((uintptr_t)W & 15) == 0 && K % 4 == 0;
   F32Conv3x3 a{X, W, images, s.Cg, s.H, s.W, s.OH, s.OW, s.pad_h, s.pad_w, plane * s.C, plane * s.Cg, M, N, K, 0, 0, Divisor31(s.OW), Divisor31(s.OH),
                Divisor31(s.OW + 2LL), Divisor31(s.OH + 2LL)};
   int tile = force;
   if ((!tile || tile == F32_CONV3X3_FEW) && f32_conv3x3_few_takes(a, out)) {
      const F32Conv3x3FewSplit split(a, out, group);
      const long long patch = f32_conv3x3_patch(s.OH, s.OW, 128);
      if (tile || patch > F32_CONV3X3_PATCH || f32_conv3x3_few_preferred(a, out, split, group, patch)) {
         *taken = true;
         return launch_f32_conv3x3_few(ctx->stream, a, out, split, group);
      }
   }
   if (!tile && s.Cg <= 4) {
      tile = F32_CONV3X3_128; // slabs of four channels; half of any other kernel's slab would be zeros
   } else if (!tile) {
      // us: a launch; a slab (8 channels, 16 of the split kernel) of a CU whose tiles wait for their loads, and of one with several tiles at work; a tile.  The
      // second set is for weights that come float by float.  Fitted to 156 layers (the split kernel's to 230 others) from 1 image of 6 x 6 to 64 of 64 x 64, 5 to 130
      // channels; holds to a sixth, and costs 0.4 % of the best of these kernels on average over the 260 layers, 14 % the most, 10 % but for that one.
      double least = 1e30;
      struct Cost {
         double launch, alone, slab, each;
      };
      auto offer = [&](int which, int channels, long long room, Cost wide, Cost narrow) {
         const int bm = conv3x3_pixels(which);
         const Cost cost = vec ? wide : narrow;
         const double tiles = (double)((M + bm - 1) / bm) * ((N + 31) / 32) * group / 256.0, slabs = (s.Cg + channels - 1) / channels;
         // (two workgroups of the split kernel share a CU, and one's odd tile runs beside the other's)
         const double rounds = channels == 8 || tiles <= 1.0 ? std::ceil(tiles) : 0.5 * (tiles + std::ceil(tiles));
         const double t = cost.launch + std::max(slabs * cost.alone, rounds * (slabs * cost.slab + cost.each));
         if (f32_conv3x3_patch(s.OH, s.OW, bm) <= room && t < least)
            least = t, tile = which;
      };
      offer(F32_CONV3X3_32, 8, F32_CONV3X3_PATCH, {3.21, 0.82, 0.49, 0.40}, {3.56, 1.09, 0.58, 0.68});
      offer(F32_CONV3X3_64, 8, F32_CONV3X3_PATCH, {3.10, 1.09, 0.69, 0.72}, {3.67, 1.35, 0.84, 0.68});
      offer(F32_CONV3X3_128, 8, F32_CONV3X3_PATCH, {3.32, 1.59, 1.26, 0.84}, {3.75, 1.89, 1.47, 0.63});
      offer(F32_CONV3X3_SPLIT_128, 16, F32_CONV3X3_SPLIT_PATCH, {3.95, 3.25, 2.20, 1.06}, {5.12, 3.65, 2.82, 0.65});
      offer(F32_CONV3X3_SPLIT_256, 16, F32_CONV3X3_SPLIT_PATCH, {5.17, 4.60, 3.75, 0.65}, {6.95, 4.60, 4.19, 0.30});
   }
   const int pixels = conv3x3_pixels(tile);
   if (!pixels)
      return SOFIE_HIP_OK; // another kernel, or a request for one that there is not: launch_f32_product's
   const bool split = tile == F32_CONV3X3_SPLIT_128 || tile == F32_CONV3X3_SPLIT_256;
   const long long patch = f32_conv3x3_patch(s.OH, s.OW, pixels);
   if (patch > (split ? F32_CONV3X3_SPLIT_PATCH : F32_CONV3X3_PATCH))
      return SOFIE_HIP_OK;
   // the images that 256 pixels touch, all their channels
   const int near = (255 / ((long long)s.OH * s.OW) + 2) * (long long)out.Cout * out.positions * 4 < F32_BUFFER_BYTES - (1 << 20);
   a.chunks = (int)(patch + 63) / 64;
   a.near = near;
   *taken = true;
   hipStream_t st = ctx->stream;
   if (split) {
      // (a patch of 256 pixels has 324 places and more)
      auto go = [&](auto wide) {
         constexpr int V = decltype(wide)::value;
         if (tile == F32_CONV3X3_SPLIT_256)
            return launch_f32_conv3x3_split_as<256, F32_CONV3X3_SPLIT_PATCH, V>(st, a, out, group);
         return patch <= 256 ? launch_f32_conv3x3_split_as<128, 256, V>(st, a, out, group) : launch_f32_conv3x3_split_as<128, F32_CONV3X3_SPLIT_PATCH, V>(st, a, out, group);
      };
      return vec ? go(std::integral_constant<int, 4>{}) : go(std::integral_constant<int, 1>{});
   }
   auto go = [&](auto room, auto wide) {
      constexpr int P = decltype(room)::value, V = decltype(wide)::value;
      if (s.Cg <= 4 && tile == F32_CONV3X3_128)
         return launch_f32_conv3x3_as<128, 32, 4, 1, 1, 4, P, 1>(st, a, out, group);
      switch (tile) {
      case F32_CONV3X3_32: return launch_f32_conv3x3_as<32, 32, 1, 1, 4, 8, P, V>(st, a, out, group);
      case F32_CONV3X3_64: return launch_f32_conv3x3_as<64, 32, 2, 1, 2, 8, P, V>(st, a, out, group);
      default: return launch_f32_conv3x3_as<128, 32, 4, 1, 1, 8, P, V>(st, a, out, group);
      }
   };
   auto with = [&](auto room) { return vec ? go(room, std::integral_constant<int, 4>{}) : go(room, std::integral_constant<int, 1>{}); };
   // the places a channel has in LDS: the fewer, the more workgroups share a CU (with 128 pixels, images of up to 17, 54 and 98 columns, and
   // those that such a tile divides: 32, 64, 80, 112, 128 ...)
   return patch <= 256 ? with(std::integral_constant<int, 256>{}) : patch <= 448 ? with(std::integral_constant<int, 448>{}) : with(std::integral_constant<int, F32_CONV3X3_PATCH>{});
}

// A convolution of `group` groups as products of M = images x positions rows and Cout / group columns.
template <bool MASKED>
static int launch_f32_conv_rows(sofie_hip_ctx *ctx, const F32ConvRows<MASKED> &A, const float *W, const F32ConvStore &out, int M, int group)
{
   const int K = A.K, N = out.Cout_g;
   const long long strideB = (long long)N * K;
   if (((uintptr_t)W & 15) == 0 && K % 4 == 0)
      return launch_f32_product(ctx, A, F32Matrix<true, 4>{W, K, N, K}, out, M, N, K, group, 0, strideB);
   return launch_f32_product(ctx, A, F32Matrix<true, 1>{W, K, N, K}, out, M, N, K, group, 0, strideB);
}
static int launch_f32_conv(sofie_hip_ctx *ctx, const float *X, F32ConvShape s, const float *W, const F32ConvStore &out, long long M, int group, const char *who)
{
   const int taps = s.kd * s.kh * s.kw, K = s.Cg * taps;
   s.by_kw = Divisor31(s.kw), s.by_kh = Divisor31(s.kh), s.by_kd = Divisor31(s.kd), s.by_positions = Divisor31(taps);
   SOFIE_HIP_REQUIRE(group <= 65535, "%s: too many groups for one launch", who);
   SOFIE_HIP_REQUIRE(M <= MOST_ROWS && out.Cout_g <= MOST_ROWS, "%s: too many output pixels or channels", who);
   auto rows = [&](auto A) {
      A.X = X;
      A.s = s;
      A.rows = (int)M;
      A.K = K;
      A.channel = (long long)s.D * s.H * s.W;
      A.image = A.channel * s.C;
      return launch_f32_conv_rows(ctx, A, W, out, (int)M, group);
   };
   s.positions = taps;
   auto reciprocal64 = [](unsigned d) -> unsigned long long { return d <= 1 ? 0ull : (~0ull / d) + 1; };
   s.ow_mul = reciprocal64(s.OW), s.oh_mul = reciprocal64(s.OH), s.od_mul = reciprocal64(s.OD);
   bool taken = false;
   if (int st = launch_f32_conv3x3(ctx, X, s, W, out, (int)(M / ((long long)s.OD * s.OH * s.OW)), (int)M, group, &taken); st || taken)
      return st;
   // one bit per kernel position; the images that the 128 rows of a tile touch within a buffer, and the channels within its scalar offset
   const long long plane = (long long)s.D * s.H * s.W, window = ((long long)s.kd * s.dil_d * s.H + (long long)s.kh * s.dil_h) * s.W + (long long)s.kw * s.dil_w;
   const long long images = 127 / ((long long)s.OD * s.OH * s.OW) + 2;
   const long long padded = ((long long)s.pad_d * s.H + s.pad_h) * s.W + s.pad_w + ((long long)s.D * s.H + s.H) * s.W; // strides step inside it
   if (taps <= 31 && (images * s.C * plane + 2 * padded) * 4 < F32_BUFFER_BYTES && (s.Cg * plane + window) * 4 < (1LL << 32) &&
       (s.Cg + 64) * plane * 4 < (1LL << 32))
      return rows(F32ConvRows<true>{});
   return rows(F32ConvRows<false>{});
}

// `count` layers in one launch of the chain kernel, if their shapes, strides and memory allow it (*launched tells).
static int launch_f32_chain(sofie_hip_ctx *ctx, const sofie_gemm_f32_desc *layers, int32_t count, bool *launched)
{
   *launched = false;
   const int M = layers[0].M;
   bool fused = count >= 2 && M >= 1 && M <= MOST_ROWS;
   int width = layers[0].K;
   ChainArgs a;
   a.count = count;
   a.M = M;
   a.A = layers[0].A;
   a.lda = layers[0].lda ? layers[0].lda : layers[0].K;
   for (int l = 0; l < count && fused; ++l) {
      const sofie_gemm_f32_desc &d = layers[l];
      const long long ldb = d.ldb ? d.ldb : (d.transB ? d.K : d.N), ldy = d.ldy ? d.ldy : d.N;
      fused = d.M == M && d.N >= 1 && d.N <= 8192 && d.K >= 1 && d.K <= 8192 && !d.transA && d.batch == 1 && d.A && d.B && d.Y && ldb >= (d.transB ? d.K : d.N) && ldy >= d.N &&
              d.bias_mode >= SOFIE_BIAS_NONE && d.bias_mode <= SOFIE_BIAS_FULL && (d.bias_mode == SOFIE_BIAS_NONE || d.C != nullptr) &&
              (l == 0 ? a.lda >= d.K : (d.K == layers[l - 1].N && (d.lda ? d.lda : d.K) == (layers[l - 1].ldy ? layers[l - 1].ldy : layers[l - 1].N)));
      if (!fused)
         break;
      ChainLayerArgs &L = a.layer[l];
      L.B = d.B;
      L.ldb = ldb;
      L.transB = d.transB ? 1 : 0;
      L.N = d.N;
      L.K = d.K;
      L.Y = d.Y;
      L.ldy = ldy;
      int bad = 0;
      fused = make_post_chain(L.ep.chain, d.act, d.act_alpha, d.post, bad);
      L.ep.alpha = d.alpha;
      L.ep.beta = d.beta;
      L.ep.C = d.bias_mode == SOFIE_BIAS_NONE ? nullptr : d.C;
      L.ep.bias_mode = d.bias_mode;
      L.ep.ldc = d.N;
      L.ep.R = d.residual;
      L.ep.ldr = ldy;
      width = d.N > width ? d.N : width;
   }
   // In one launch a workgroup takes ITS rows through every layer, independently of the other workgroups.  Two tensors of the
   // chain may therefore share memory only row for row (same address, same pitch, same width: the ping-pong of equal layers,
   // where a row is rewritten by the workgroup that owns it); any other overlap of what a layer writes with what a layer
   // reads or writes would let one workgroup's rows land on another's.  Callers that planned the layers' tensors by
   // per-layer lifetimes get the layer-by-layer form then.
   if (fused) {
      struct Range {
         const char *lo, *hi;
         long long pitch, width;
      };
      auto range = [](const void *p, long long bytes, long long pitch, long long w) {
         return Range{(const char *)p, (const char *)p + (bytes > 0 ? bytes : 0), pitch, w};
      };
      auto overlap = [](const Range &x, const Range &y) { return x.lo < y.hi && y.lo < x.hi; };
      auto same_rows = [](const Range &x, const Range &y) { return x.lo == y.lo && x.pitch == y.pitch && x.width == y.width; };
      Range reads[2 * SOFIE_MAX_GEMM_CHAIN], writes[SOFIE_MAX_GEMM_CHAIN];
      int nr = 0;
      const Range input = range(layers[0].A, ((long long)(M - 1) * a.lda + layers[0].K) * 4, a.lda, layers[0].K);
      for (int l = 0; l < count; ++l) {
         const sofie_gemm_f32_desc &d = layers[l];
         const long long ldy = d.ldy ? d.ldy : d.N, ybytes = ((long long)(M - 1) * ldy + d.N) * 4;
         writes[l] = range(d.Y, ybytes, ldy, d.N);
         if (d.bias_mode != SOFIE_BIAS_NONE)
            reads[nr++] = range(d.C, 4LL * (d.bias_mode == SOFIE_BIAS_ROW ? d.N : d.bias_mode == SOFIE_BIAS_COL ? M : d.bias_mode == SOFIE_BIAS_FULL ? (long long)M * d.N : 1), 0, 0);
         if (d.residual)
            reads[nr++] = range(d.residual, ybytes, 0, 0);
      }
      for (int l = 0; l < count && fused; ++l) {
         if (overlap(writes[l], input) && !same_rows(writes[l], input))
            fused = false;
         for (int m = 0; m < l && fused; ++m)
            if (overlap(writes[l], writes[m]) && !same_rows(writes[l], writes[m]))
               fused = false;
         for (int r = 0; r < nr && fused; ++r)
            if (overlap(writes[l], reads[r]))
               fused = false;
      }
   }
   const int RB = M <= 64 ? 1 : M <= 128 ? 2 : 4;
   width = (width + 3) / 4 * 4;
   if (fused && (long long)RB * width <= 8192) {
      const size_t lds = ((size_t)2 * RB * width + RB * CHAIN_THREADS) * sizeof(float);
      const dim3 grid((unsigned)((M + RB - 1) / RB));
      bool any = false;
      for (int l = 0; l < count; ++l)
         any = any || chain_layer_by_rows(a.layer[l]);
      auto launch = [&](auto rows, auto by_rows) -> int {
         auto kern = gemm_chain_f32_kernel<decltype(rows)::value, decltype(by_rows)::value>;
         static bool configured[64] = {};
         if (int st = configure_lds_once(kern, (2 * 8192 + decltype(rows)::value * CHAIN_THREADS) * sizeof(float), configured))
            return st;
         launch_kernel(kern, grid, dim3(CHAIN_THREADS), lds, ctx->stream, a, width);
         return SOFIE_HIP_OK;
      };
      auto with = [&](auto by_rows) {
         return RB == 1 ? launch(std::integral_constant<int, 1>{}, by_rows) : RB == 2 ? launch(std::integral_constant<int, 2>{}, by_rows) : launch(std::integral_constant<int, 4>{}, by_rows);
      };
      if (int st = any ? with(std::true_type{}) : with(std::false_type{}))
         return st;
      *launched = true;
      return launch_status("gemm_chain_f32_kernel");
   }
   return SOFIE_HIP_OK;
}

} // namespace sofie_hip

using namespace sofie_hip;

extern "C" {

int sofie_hip_gemm_f32(sofie_hip_ctx *ctx, const sofie_gemm_f32_desc *d)
{
   SOFIE_HIP_REQUIRE(ctx && d, "sofie_hip_gemm_f32: NULL argument");
   SOFIE_HIP_REQUIRE(d->M >= 0 && d->N >= 0 && d->K >= 0, "sofie_hip_gemm_f32: negative dimension");
   SOFIE_HIP_REQUIRE(d->batch >= 1, "sofie_hip_gemm_f32: batch must be >= 1");
   SOFIE_HIP_REQUIRE(d->bias_mode >= SOFIE_BIAS_NONE && d->bias_mode <= SOFIE_BIAS_FULL, "sofie_hip_gemm_f32: unknown bias mode %d", d->bias_mode);
   F32Epilogue ep;
   int bad = 0;
   SOFIE_HIP_REQUIRE(make_post_chain(ep.chain, d->act, d->act_alpha, d->post, bad),
                     "sofie_hip_gemm_f32: unknown activation or post operator %d (or more than %d post operators)", bad, SOFIE_MAX_POST_OPS);
   if (d->M == 0 || d->N == 0)
      return SOFIE_HIP_OK;
   SOFIE_HIP_REQUIRE(d->Y != nullptr, "sofie_hip_gemm_f32: Y is NULL");
   SOFIE_HIP_REQUIRE(d->K == 0 || (d->A && d->B), "sofie_hip_gemm_f32: A or B is NULL");
   SOFIE_HIP_REQUIRE(d->bias_mode == SOFIE_BIAS_NONE || d->C != nullptr, "sofie_hip_gemm_f32: bias mode set but C is NULL");
   const int M = d->M, N = d->N, K = d->K;
   const long long lda = d->lda ? d->lda : (d->transA ? M : K);
   const long long ldb = d->ldb ? d->ldb : (d->transB ? K : N);
   const long long ldy = d->ldy ? d->ldy : N;
   SOFIE_HIP_REQUIRE(lda >= (d->transA ? M : K) && ldb >= (d->transB ? K : N) && ldy >= N,
                     "sofie_hip_gemm_f32: leading dimension too small");
   SOFIE_HIP_REQUIRE(M <= MOST_ROWS && N <= MOST_ROWS, "sofie_hip_gemm_f32: M or N too long");
   ep.alpha = d->alpha;
   ep.beta = d->beta;
   ep.C = d->bias_mode == SOFIE_BIAS_NONE ? nullptr : d->C;
   ep.bias_mode = d->bias_mode;
   ep.ldc = N;
   ep.R = d->residual;
   ep.ldr = ldy;
   SOFIE_HIP_REQUIRE(d->batch <= 65535, "sofie_hip_gemm_f32: batch too large for one launch");
   auto in_vectors = [](const void *p, long long a, long long b, long long c) { return ((uintptr_t)p & 15) == 0 && a % 4 == 0 && b % 4 == 0 && c % 4 == 0; };
   F32RowStore out;
   out.Y = d->Y;
   out.ldy = ldy;
   out.ep = ep;
   out.vec = in_vectors(d->Y, ldy, d->strideY, 0);
   out.strideC = d->strideC;
   out.strideY = d->strideY;
   // 16-byte loads where both operands allow them: address, pitch, and the extent along the contiguous direction
   const bool vec = in_vectors(d->A, lda, d->strideA, d->transA ? M : K) && in_vectors(d->B, ldb, d->strideB, d->transB ? K : N);
   auto with_b = [&](const auto &A) {
      auto go = [&](const auto &B) {
         return launch_f32_product(ctx, A, B, out, M, N, K, d->batch, d->strideA, d->strideB);
      };
      constexpr int VEC = std::remove_reference_t<decltype(A)>::VEC;
      return d->transB ? go(F32Matrix<true, VEC>{d->B, ldb, N, K}) : go(F32Matrix<false, VEC>{d->B, ldb, N, K});
   };
   if (vec)
      return d->transA ? with_b(F32Matrix<false, 4>{d->A, lda, M, K}) : with_b(F32Matrix<true, 4>{d->A, lda, M, K});
   return d->transA ? with_b(F32Matrix<false, 1>{d->A, lda, M, K}) : with_b(F32Matrix<true, 1>{d->A, lda, M, K});
}

int sofie_hip_gemm_chain_f32(sofie_hip_ctx *ctx, const sofie_gemm_f32_desc *layers, int32_t count)
{
   SOFIE_HIP_REQUIRE(ctx && layers, "sofie_hip_gemm_chain_f32: NULL argument");
   SOFIE_HIP_REQUIRE(count >= 1 && count <= SOFIE_MAX_GEMM_CHAIN, "sofie_hip_gemm_chain_f32: %d layers (1..%d allowed)", count, SOFIE_MAX_GEMM_CHAIN);
   for (int l = 1; l < count; ++l)
      SOFIE_HIP_REQUIRE(layers[l].A == layers[l - 1].Y && layers[l].A != nullptr, "sofie_hip_gemm_chain_f32: layer %d does not read the output of layer %d", l, l - 1);
   // Which layers share a launch.  A launch of its own spreads a layer over the chip and costs 2.5 us or more; in the chain kernel a workgroup does its rows' share alone: a pass over
   // the outputs that its waves take at once (W stored [N][K]) or a walk along k (W stored [K][N]) at a time.  So large layers run one by one, and small ones behind them share a
   // launch.  Costs by the rows of a workgroup, one, two or four (M <= 64, <= 128, <= 256).  Of 4000 networks of two to four layers, all layers together or each by itself, the choice is 0.1 %
   // above the better of the two on average where W is stored [N][K] (0.2, 0.7 and 1.0 % with factors of 1, 1.27 and 1.7 for the rows, 36 % the most: 183 x 128-112-94-48-3 16.7 us together,
   // 12.3 apart) and 0.5, 0.7 and 1.8 % where it is [K][N] (25 % the most: more than 128 rows are taken together too seldom).
   const int M = layers[0].M;
   int first = count; // first layer of the shared launch
   if (ctx->opt.f32_chain == 1) {
      first = 0;
   } else if (ctx->opt.f32_chain < 0 && M >= 1 && M <= 256) {
      auto loads = [&](int l) {
         const auto &d = layers[l];
         return f32_loads((d.transA ? d.M : d.K) % 4 == 0 && (d.transB ? d.K : d.N) % 4 == 0, d.transB && !d.transA);
      };
      auto apart = [](double t) { return std::max(1.02 * t - 0.27, 2.5); }; // behind another layer
      struct Costs {
         double launch, layer, pass, k;                  // W stored [N][K]
         double columns_launch, columns_pass, columns_k; // W stored [K][N]
      };
      static constexpr Costs COSTS[] = {{1.76, 0.44, 0.81, 0.0013, 1.76, 1.55, 0.025}, {1.56, 0.15, 1.76, 0.0014, 1.76, 1.97, 0.0318}, {2.30, 0.23, 2.80, 0.0020, 1.76, 2.64, 0.0425}};
      const Costs &cost = COSTS[M <= 64 ? 0 : M <= 128 ? 1 : 2];
      double before = 0.0, least = 0.0;
      for (int l = 0; l < count; ++l) {
         double t = 0.0;
         pick_f32_tile(M, layers[l].N, layers[l].K, 1, loads(l), &t);
         least += apart(t);
      }
      for (int s = 0; s + 2 <= count; ++s) {
         double together = 0.0, t = 0.0;
         for (int l = s; l < count; ++l) {
            const double K = layers[l].K, N = layers[l].N;
            const bool wide = layers[l].K % 4 == 0 && layers[l].ldb % 4 == 0; // chain_rows
            const double outputs = !layers[l].transB ? 1024.0 : !wide || N <= 64 ? 64.0 : K <= 64 ? 256.0 : K <= 128 ? 128.0 : 64.0, passes = std::ceil(N / outputs);
            const double groups = N <= 64 ? 16.0 : N <= 128 ? 8.0 : N <= 256 ? 4.0 : N <= 512 ? 2.0 : 1.0; // that deal out k
            // (rows of W that are no whole 16-byte pieces: a little less a pass, more for its k)
            together += layers[l].transB ? cost.layer + passes * (wide ? cost.pass + cost.k * K : 0.96 * cost.pass + 1.8 * cost.k * K) : passes * (cost.columns_pass + cost.columns_k * K / groups);
         }
         together += before + (layers[count - 1].transB ? cost.launch : cost.columns_launch);
         if (together < least)
            least = together, first = s;
         pick_f32_tile(M, layers[s].N, layers[s].K, 1, loads(s), &t);
         before += apart(t);
      }
   }
   for (int l = 0; l < count; ++l) {
      if (l == first) {
         bool launched = false;
         const int st = launch_f32_chain(ctx, layers + first, count - first, &launched);
         if (st || launched)
            return st;
      }
      // (and every malformed descriptor, which the single product reports)
      if (int st = sofie_hip_gemm_f32(ctx, &layers[l]))
         return st;
   }
   return SOFIE_HIP_OK;
}

int sofie_hip_conv_f32(sofie_hip_ctx *ctx, const sofie_conv_desc *d, const float *X, const float *W, const float *bias,
                       int32_t act, float act_alpha, float *Y, const sofie_post_ops *post, const float *residual)
{
   SOFIE_HIP_REQUIRE(ctx && d, "sofie_hip_conv_f32: NULL argument");
   SOFIE_HIP_REQUIRE(d->N >= 0 && d->C > 0 && d->H > 0 && d->W > 0 && d->Cout > 0 && d->kh > 0 && d->kw > 0,
                     "sofie_hip_conv_f32: bad shape");
   SOFIE_HIP_REQUIRE(d->group > 0 && d->C % d->group == 0 && d->Cout % d->group == 0,
                     "sofie_hip_conv_f32: group %d does not divide the channels", d->group);
   SOFIE_HIP_REQUIRE(d->stride_h > 0 && d->stride_w > 0 && d->dil_h > 0 && d->dil_w > 0, "sofie_hip_conv_f32: bad stride or dilation");
   SOFIE_HIP_REQUIRE(d->pad_h0 >= 0 && d->pad_w0 >= 0 && d->pad_h1 >= 0 && d->pad_w1 >= 0, "sofie_hip_conv_f32: negative padding");
   const int eff_kh = d->dil_h * (d->kh - 1) + 1, eff_kw = d->dil_w * (d->kw - 1) + 1;
   SOFIE_HIP_REQUIRE(d->H + d->pad_h0 + d->pad_h1 >= eff_kh && d->W + d->pad_w0 + d->pad_w1 >= eff_kw,
                     "sofie_hip_conv_f32: kernel larger than the padded image");
   const int OH = (d->H + d->pad_h0 + d->pad_h1 - eff_kh) / d->stride_h + 1;
   const int OW = (d->W + d->pad_w0 + d->pad_w1 - eff_kw) / d->stride_w + 1;
   SOFIE_HIP_REQUIRE(OH == d->OH && OW == d->OW, "sofie_hip_conv_f32: output shape %dx%d does not match the descriptor's %dx%d", OH, OW,
                     d->OH, d->OW);
   PostChain chain;
   int bad = 0;
   SOFIE_HIP_REQUIRE(make_post_chain(chain, act, act_alpha, post, bad),
                     "sofie_hip_conv_f32: unknown activation or post operator %d (or more than %d post operators)", bad, SOFIE_MAX_POST_OPS);
   if (d->N == 0)
      return SOFIE_HIP_OK;
   SOFIE_HIP_REQUIRE(X && W && Y, "sofie_hip_conv_f32: NULL pointer");
   const long long M = (long long)d->N * OH * OW;
   SOFIE_HIP_REQUIRE(M < (1LL << 31), "sofie_hip_conv_f32: too many output pixels");
   SOFIE_HIP_REQUIRE((long long)(d->C / d->group) * d->kh * d->kw < (1LL << 31), "sofie_hip_conv_f32: reduction too long");
   const F32ConvShape s{d->C, 1, d->H, d->W, 1, d->kh, d->kw, 1, OH, OW, 0, d->pad_h0, d->pad_w0, 1, d->stride_h, d->stride_w, 1, d->dil_h, d->dil_w,
                        d->C / d->group, 0, 0, 0, 0};
   const F32ConvStore out{Y, bias, residual, chain, d->Cout, d->Cout / d->group, OH * OW, 0};
   return launch_f32_conv(ctx, X, s, W, out, M, d->group, "sofie_hip_conv_f32");
}

int sofie_hip_conv3d_f32(sofie_hip_ctx *ctx, const sofie_conv3d_desc *d, const float *X, const float *W, const float *bias,
                         int32_t act, float act_alpha, float *Y, const sofie_post_ops *post, const float *residual)
{
   SOFIE_HIP_REQUIRE(ctx && d, "sofie_hip_conv3d_f32: NULL argument");
   SOFIE_HIP_REQUIRE(d->N >= 0 && d->C > 0 && d->D > 0 && d->H > 0 && d->W > 0 && d->Cout > 0 && d->kd > 0 && d->kh > 0 && d->kw > 0,
                     "sofie_hip_conv3d_f32: bad shape");
   SOFIE_HIP_REQUIRE(d->group > 0 && d->C % d->group == 0 && d->Cout % d->group == 0,
                     "sofie_hip_conv3d_f32: group %d does not divide the channels", d->group);
   const int in[3] = {d->D, d->H, d->W}, kern[3] = {d->kd, d->kh, d->kw}, want[3] = {d->OD, d->OH, d->OW};
   int outd[3];
   for (int a = 0; a < 3; ++a) {
      SOFIE_HIP_REQUIRE(d->stride[a] > 0 && d->dil[a] > 0, "sofie_hip_conv3d_f32: bad stride or dilation");
      SOFIE_HIP_REQUIRE(d->pad[a] >= 0 && d->pad[a + 3] >= 0, "sofie_hip_conv3d_f32: negative padding");
      const int eff = d->dil[a] * (kern[a] - 1) + 1;
      SOFIE_HIP_REQUIRE(in[a] + d->pad[a] + d->pad[a + 3] >= eff, "sofie_hip_conv3d_f32: kernel larger than the padded volume");
      outd[a] = (in[a] + d->pad[a] + d->pad[a + 3] - eff) / d->stride[a] + 1;
      SOFIE_HIP_REQUIRE(outd[a] == want[a], "sofie_hip_conv3d_f32: output extent %d of axis %d does not match the descriptor's %d", outd[a], a, want[a]);
   }
   PostChain chain;
   int bad = 0;
   SOFIE_HIP_REQUIRE(make_post_chain(chain, act, act_alpha, post, bad),
                     "sofie_hip_conv3d_f32: unknown activation or post operator %d (or more than %d post operators)", bad, SOFIE_MAX_POST_OPS);
   if (d->N == 0)
      return SOFIE_HIP_OK;
   SOFIE_HIP_REQUIRE(X && W && Y, "sofie_hip_conv3d_f32: NULL pointer");
   const long long plane = (long long)outd[0] * outd[1] * outd[2], M = (long long)d->N * plane;
   SOFIE_HIP_REQUIRE(M < (1LL << 31) && (long long)d->C * d->D * d->H * d->W < (1LL << 31), "sofie_hip_conv3d_f32: too many output or input elements");
   const long long Kg64 = (long long)(d->C / d->group) * d->kd * d->kh * d->kw;
   SOFIE_HIP_REQUIRE(Kg64 < (1LL << 31), "sofie_hip_conv3d_f32: reduction too long");
   const F32ConvShape s{d->C, d->D, d->H, d->W, d->kd, d->kh, d->kw, outd[0], outd[1], outd[2], d->pad[0], d->pad[1], d->pad[2],
                        d->stride[0], d->stride[1], d->stride[2], d->dil[0], d->dil[1], d->dil[2], d->C / d->group, 0, 0, 0, 0};
   const F32ConvStore out{Y, bias, residual, chain, d->Cout, d->Cout / d->group, (int)plane, 0};
   return launch_f32_conv(ctx, X, s, W, out, M, d->group, "sofie_hip_conv3d_f32");
}

} // extern "C"
