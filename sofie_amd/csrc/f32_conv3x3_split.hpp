// fp32 3 x 3 convolution (stride 1, no dilation, two spatial axes) on the bf16 matrix cores.
//
// Every fp32 value from 2^-110 on is the sum of three bf16 values, x = h + m + l (h = bf16(x), m = bf16(x - h), l = x - h - m; |m| <= 2^-8 |x|, |l| <= 2^-17 |x|;
// Henry, Tang, Heinecke, "Leveraging the bfloat16 Artificial Intelligence Datatype For Higher-Precision Computations", ARITH 2019), and a product of two such sums is taken as eight terms:
//   a b = ah bh + (ah bm + am bh) + (ah bl + am bm + al bh) + (am bl + al bm),       left out: al bl <= 2^-34 a b.
// (Without the last two, each up to 2^-25 of the product, a sum with one product that counts would be known to 2^-23 only, where fp32 gives 2^-24.)
// bf16 products are exact in the fp32 accumulators, and v_mfma_f32_32x32x16_bf16 multiplies 16 k in 32 cycles where v_mfma_f32_32x32x2_f32 needs
// 512: the eight terms cost half of the fp32 instructions.  The leading products and the other terms are summed apart: an accumulator of leading products is
// rounded once per 16 k and instruction, by up to 1.6 2^-24 of the magnitudes in it (measured; 1.9 per 2 k for the fp32 instruction).
//
// What the pieces cost is vector instructions (5.5 per value) and LDS (6 bytes written per value, at 79 B/clk): a 3 x 3 convolution uses every value of its
// input patch nine times, which pays for both.  (A plain product of 64 x 64 tiles uses a value twice per wave: 20 - 27 us where fp32 takes 20 - 32.)
// 64 images of 32 x 32, us, the fp32 kernel's best tile -> this one: 32 -> 64 channels 26.1 -> 22.8, 64 -> 64 43.4 -> 37.0 (with a residual 47.0 -> 37.7); 128 -> 128
// at 16 x 16 45.2 -> 40.2; 48 images of 37 x 37, 32 -> 96 44.3 -> 42.9.  With six terms 20.6, 31.0 (32.3), 35.7, 39.4.  Error of 64 -> 64 against 64 bits: 2.4e-7 to
// 3.4e-7 -> 1.0e-7 of the result.
//
// Exceptions: bf16 has the exponents of fp32, and the matrix cores keep subnormal numbers, so pieces hold every multiple of 2^-133.  Three things do not fit:
// a value within 2^-8 of the largest rounds to an infinity, the remainders of an infinity are NaN, and the last bits of a value below 2^-110 are lost.  The first two
// end in a sum that is not finite; the last shows where a value is split, as a subnormal third piece.  A wave whose sums are not finite, and a workgroup that met
// such a piece, compute their sums again with fp32 instructions straight from memory.  (The matrix cores' treatment of subnormals was measured: subnormal
// operands, products and sums of v_mfma_f32_32x32x16_bf16 come out exact.)  Telling costs an instruction per value: 64 -> 64 at 32 x 32 takes 1.3 us longer.  Summing
// again, in every tile of 64 images of 32 x 32, has its price: 32 -> 64 channels 22.8 -> 59 us, 64 -> 64 37 -> 109, 128 -> 128 at 16 x 16 40 -> 180.  It takes two channels at a
// time with their loads in flight; eight k at a time with their index arithmetic were 132 for the second.
#pragma once
#include "f32_conv3x3.hpp"

namespace sofie_hip {

typedef __bf16 v2bf __attribute__((ext_vector_type(2)));
typedef __bf16 v8bf __attribute__((ext_vector_type(8)));
typedef float v2f __attribute__((ext_vector_type(2)));
typedef unsigned v4u __attribute__((ext_vector_type(4)));

// The next piece of eight values, and what is left of them.  (v_dot2_f32_bf16 takes a remainder in one instruction instead of two, but not beside the
// matrix cores: an MFMA and four of them take 58 cycles, an MFMA and four subtractions 34.)
template <int P>
__device__ __forceinline__ v4u f32_next_piece(float (&x)[8])
{
   v4u words;
#pragma unroll
   for (int e = 0; e < 4; ++e) {
      const unsigned both = __builtin_bit_cast(unsigned, __builtin_convertvector((v2f{x[2 * e], x[2 * e + 1]}), v2bf));
      words[e] = both;
      if constexpr (P < 2) {
         x[2 * e] -= __builtin_bit_cast(float, both << 16);
         x[2 * e + 1] -= __builtin_bit_cast(float, both & 0xffff0000u);
      }
   }
   return words;
}

// The largest patch that is taken: with it two workgroups fit a CU (81 KB each); one alone takes 1.9 times as long (32 images, 64 -> 128 at 56 x 56: 206 us
// against the fp32 kernel's 165).
constexpr int F32_CONV3X3_SPLIT_PATCH = 360;

// LDS of a workgroup.  A slab is 16 channels.  Pieces lie in columns of 16 bytes, eight channels each: of a patch, [piece][half of the channels][position]; of the
// weights, [piece][kernel position][half][output channel], columns 16 bytes apart beside their 32 rows (the 18 columns of a row, which are written
// side by side, start in different banks).  The weights come as they are in memory, a row of 144 floats per output channel, and are split from there.
template <int PLANE, int WVEC>
struct F32Conv3x3SplitShape {
   static constexpr int CS = 16, BN = 32;
   static constexpr int PITCH = CS * 9;                                                    // of a row of weights, in floats
   static constexpr int WLOADS = (BN * PITCH + 64 * WVEC - 1) / (64 * WVEC);               // load instructions per slab of weights
   static constexpr int HALF = PLANE * 16, PATCH = 2 * HALF;                               // bytes of a piece of a patch
   static constexpr int COLUMN = BN * 16 + 16, WEIGHTS = 18 * COLUMN;                      // bytes of a piece of the weights
   static constexpr int RAW_AT = 3 * (PATCH + WEIGHTS), BYTES = RAW_AT + WLOADS * 64 * WVEC * 4;
};

// Four waves, each with BM / 4 pixels and 32 output channels.  One slab lies in LDS in pieces, the next one as raw weights and, in registers, as raw patch; two
// workgroups per CU, one of which splits while the other multiplies.  (One workgroup whose other four waves split for it, through two slabs of pieces, is no
// faster: 36 us, bound by LDS.)  8 - 14 scalars are spilled, 48 - 70 in the kernels of activations with calls; 256 pixels with narrow weights fill the 256 vector registers.
template <int BM, int PLANE, int WVEC, bool PLAIN>
__global__ __launch_bounds__(256, 2) void f32_conv3x3_split_kernel(F32Conv3x3 a, F32ConvStore out, TileOrder order, int first_tile)
{
   typedef F32Conv3x3SplitShape<PLANE, WVEC> S;
   constexpr int CS = S::CS, BN = S::BN, TM = BM / 4, MT = TM / 32;
   static_assert(TM % 32 == 0 && PLANE % 8 == 0, "wave tiles of 32 x 32 blocks");
   extern __shared__ __attribute__((aligned(16))) char split_lds[];
   const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lk = lane >> 5, c = lane & 31;
   const int wave_id = wave;
   int tm, tn, z;
   order.place(first_tile + blockIdx.x, tm, tn, z);
   a.X += z * a.group;
   a.W += (long long)z * a.N * a.K;
   out.select_batch(z);
   const int m0 = tm * BM, n0 = tn * BN;
   const int VW = a.OW + 2, VH = a.OH + 2;
   auto quotient = [](int n, const Divisor31 &by) { return (int)by.over((unsigned)n); };

   // where the patch begins; a wave splits every other 64 positions of one half of a slab's channels
   const int line0 = quotient(m0, a.by_ow), image0 = quotient(line0, a.by_oh);
   const int row0 = line0 - image0 * a.OH; // of image0, padding row 0 first
   const char *base = (const char *)uniform((long long)(a.X + image0 * a.image));
   const int plane_bytes = a.H * a.Wd * 4;
   constexpr int CHUNKS = (PLANE + 127) / 128; // of 64 positions per wave
   const int half = wave & 1;
   int patch_at[CHUNKS]; // bytes from `base`, of channel 0
   auto position = [&](int q) { return (2 * q + (wave >> 1)) * 64 + lane; };
#pragma unroll
   for (int q = 0; q < CHUNKS; ++q) {
      const int f = position(q), vr = quotient(f, a.by_vw), ix = f - vr * VW - a.pad_w;
      const int on = row0 + vr, image = quotient(on, a.by_vh), iy = on - image * VH - a.pad_h;
      const bool inside = (unsigned)ix < (unsigned)a.Wd && (unsigned)iy < (unsigned)a.H && image0 + image < a.images;
      patch_at[q] = inside ? (int)((image * a.image + (long long)iy * a.Wd + ix) * 4) : F32_OUTSIDE;
   }
   // the weights of this tile: rows past N and the gaps between rows read as zero
   constexpr int LDW = (S::WLOADS + 3) / 4;
   const char *weights = (const char *)uniform((long long)(a.W + (long long)n0 * a.K));
   auto weight_place = [&](int i, int &row, int &k) {
      const int f = ((i * 4 + wave) * 64 + lane) * WVEC;
      row = f / S::PITCH;
      k = f - row * S::PITCH;
   };
   // eight weights that a thread splits: an output channel, half the channels of a slab, a kernel position
   constexpr int TASKS = BN * 18, PER = (TASKS + 255) / 256;
   int from[PER], to[PER];
#pragma unroll
   for (int t = 0; t < PER; ++t) {
      const int f = t * 256 + threadIdx.x, n = f / 18, r = f - n * 18, h = r / 9, pos = r - h * 9;
      from[t] = S::RAW_AT + (n * S::PITCH + h * 72 + pos) * 4;
      to[t] = 3 * S::PATCH + (pos * 2 + h) * S::COLUMN + n * 16;
   }

   const int slabs = (a.C + CS - 1) / CS;
   float raw[CHUNKS][8];
   auto issue = [&](int s) {
      int wave = wave_id, C = a.C, K = a.K, N = a.N;
      forget(wave), forget(C), forget(K), forget(N);
      const int first = s * CS + (wave & 1) * 8;
#pragma unroll
      for (int q = 0; q < CHUNKS; ++q)
#pragma unroll
         for (int e = 0; e < 8; ++e) {
            const bool there = first + e < C;
            raw[q][e] = f32_buffer_read(base, there ? patch_at[q] : F32_OUTSIDE, there ? (first + e) * plane_bytes : 0);
         }
#pragma unroll
      for (int i = 0; i < LDW; ++i) {
         if (i * 4 + wave < S::WLOADS) {
            int row, k;
            weight_place(i, row, k);
            // k past the last channel are the next row's
            const int at = n0 + row < N && s * CS * 9 + k < K ? (row * K + k) * 4 : F32_OUTSIDE;
            f32_buffer_load<WVEC>((lds_void_t *)(split_lds + S::RAW_AT + (i * 4 + wave) * 64 * WVEC * 4), weights + (long long)s * CS * 9 * 4, at);
         }
      }
   };
   bool small = false; // a remainder was met that the third piece may not hold
   auto split = [&]() {
      auto pieces = [&](float (&x)[8], char *at, int step) {
         *(v4u *)at = f32_next_piece<0>(x);
         *(v4u *)(at + step) = f32_next_piece<1>(x);
#pragma unroll
         for (int e = 0; e < 8; ++e)
            small |= __builtin_amdgcn_classf(x[e], 0x90); // a subnormal number of either sign
         *(v4u *)(at + 2 * step) = f32_next_piece<2>(x);
      };
#pragma unroll
      for (int t = 0; t < PER; ++t) {
         if ((t + 1) * 256 <= TASKS || t * 256 + (int)threadIdx.x < TASKS) {
            float x[8];
#pragma unroll
            for (int e = 0; e < 8; ++e)
               x[e] = *(const float *)(split_lds + from[t] + e * 36);
            pieces(x, split_lds + to[t], S::WEIGHTS);
         }
      }
#pragma unroll
      for (int q = 0; q < CHUNKS; ++q)
         if (position(q) < PLANE)
            pieces(raw[q], split_lds + half * S::HALF + position(q) * 16, S::PATCH);
   };

   // this lane's pixels in the patch, one address per kernel row, and its weights
   int pixel[MT][3];
#pragma unroll
   for (int i = 0; i < MT; ++i) {
      const int m = m0 + wave * TM + i * 32 + c, mm = m < a.M ? m : a.M - 1;
      const int line = quotient(mm, a.by_ow), image = quotient(line, a.by_oh);
      const int vr = (image - image0) * VH + line - image * a.OH - row0;
#pragma unroll
      for (int ky = 0; ky < 3; ++ky)
         pixel[i][ky] = ((vr + ky) * VW + mm - line * a.OW) * 16 + lk * S::HALF;
   }
   const int weight = 3 * S::PATCH + lk * S::COLUMN + c * 16;

   v16f acc[MT], low[MT];
   auto clear = [](v16f(&sums)[MT]) {
#pragma unroll
      for (int i = 0; i < MT; ++i)
#pragma unroll
         for (int e = 0; e < 16; ++e)
            sums[i][e] = 0.0f;
   };
   clear(acc);
   clear(low);
   // kernel position by kernel position; the fragments of the next one are read while these are multiplied
   v8bf w[2][3], x[2][MT][3];
   auto multiply = [&]() {
      auto read = [&](auto number) {
         constexpr int t = decltype(number)::value, set = t % 2;
#pragma unroll
         for (int p = 0; p < 3; ++p) {
            w[set][p] = *(const v8bf *)(split_lds + weight + p * S::WEIGHTS + t * 2 * S::COLUMN);
#pragma unroll
            for (int i = 0; i < MT; ++i)
               x[set][i][p] = *(const v8bf *)(split_lds + pixel[i][t / 3] + p * S::PATCH + t % 3 * 16);
         }
      };
      read(std::integral_constant<int, 0>{});
      static_for<9>([&](auto tc) {
         constexpr int t = decltype(tc)::value, set = t % 2;
         __builtin_amdgcn_sched_barrier(0);
         if constexpr (t < 8)
            read(std::integral_constant<int, t + 1>{});
         __builtin_amdgcn_sched_barrier(0);
         constexpr int TERM[8][2] = {{0, 0}, {2, 1}, {1, 2}, {2, 0}, {0, 2}, {1, 1}, {1, 0}, {0, 1}};
         static_for<8>([&](auto qc) {
            constexpr int q = decltype(qc)::value;
            auto &sums = q == 0 ? acc : low;
#pragma unroll
            for (int i = 0; i < MT; ++i)
               sums[i] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(w[set][TERM[q][1]], x[set][i][TERM[q][0]], sums[i], 0, 0, 0);
         });
      });
   };
   auto meet = []() {
      __builtin_amdgcn_sched_barrier(0);
      __builtin_amdgcn_s_waitcnt(0xc07f); // lgkmcnt(0)
      __builtin_amdgcn_s_barrier();
      __builtin_amdgcn_sched_barrier(0);
   };

   issue(0);
#pragma unroll 1
   for (int s = 0; s < slabs; ++s) {
      wait_vmcnt<0>();
      meet(); // the raw weights have landed for every wave, and every wave has read the pieces of slab s - 1
      split();
      meet();
      if (s + 1 < slabs)
         issue(s + 1);
      __builtin_amdgcn_sched_barrier(0);
      multiply();
   }

   float finite = 0.0f;
#pragma unroll
   for (int i = 0; i < MT; ++i)
#pragma unroll
      for (int e = 0; e < 16; ++e) {
         acc[i][e] += low[i][e];
         finite = __builtin_fmaf(acc[i][e], 0.0f, finite);
      }
   // the raw weights of the last slab have been split by every wave: their place takes a word per wave
   int *const cut = (int *)(split_lds + S::RAW_AT);
   const bool mine = __builtin_amdgcn_ballot_w64(small) != 0;
   if (lane == 0)
      cut[wave] = mine;
   meet();
   const bool any = __builtin_amdgcn_readfirstlane(cut[0] | cut[1] | cut[2] | cut[3]) != 0;
   if (any || __builtin_amdgcn_ballot_w64(finite != 0.0f) != 0) {
      clear(acc);
      int at[MT][9]; // bytes from `base` of this lane's pixels at the nine positions, of channel lk
#pragma unroll
      for (int i = 0; i < MT; ++i) {
         const int m = m0 + wave * TM + i * 32 + c, mm = m < a.M ? m : a.M - 1;
         const int line = quotient(mm, a.by_ow), image = quotient(line, a.by_oh);
#pragma unroll
         for (int t = 0; t < 9; ++t) {
            const int iy = line - image * a.OH + t / 3 - a.pad_h, ix = mm - line * a.OW + t % 3 - a.pad_w;
            const bool inside = (unsigned)iy < (unsigned)a.H && (unsigned)ix < (unsigned)a.Wd;
            at[i][t] = inside ? (int)(((image - image0) * a.image + (long long)iy * a.Wd + ix) * 4) + lk * plane_bytes : F32_OUTSIDE;
         }
      }
      const int row = n0 + c < a.N ? (c * a.K + lk * 9) * 4 : F32_OUTSIDE;
#pragma unroll 1
      for (int ch = 0; ch < a.C; ch += 2) { // lane half lk multiplies channel ch + lk
         const bool there = ch + lk < a.C;
         float u[9], v[MT][9];
#pragma unroll
         for (int t = 0; t < 9; ++t) {
            u[t] = f32_buffer_read(weights, there && row != F32_OUTSIDE ? row + t * 4 : F32_OUTSIDE, ch * 36);
#pragma unroll
            for (int i = 0; i < MT; ++i)
               v[i][t] = f32_buffer_read(base, there ? at[i][t] : F32_OUTSIDE, ch * plane_bytes);
         }
         __builtin_amdgcn_sched_barrier(0);
#pragma unroll
         for (int t = 0; t < 9; ++t)
#pragma unroll
            for (int i = 0; i < MT; ++i)
               acc[i] = __builtin_amdgcn_mfma_f32_32x32x2f32(u[t], v[i][t], acc[i], 0, 0, 0);
      }
   }

#pragma unroll
   for (int i = 0; i < MT; ++i) {
      const int m = m0 + wave * TM + i * 32 + c, mm = m < a.M ? m : a.M - 1, image = quotient(quotient(mm, a.by_ow), a.by_oh);
      const Conv3x3Block<16> block(out, image0, image, mm - image * out.positions, n0, a.N, lk, 0, m < a.M, a.near);
      float bias[16], residual[16], v[16];
      block.load(bias, residual);
#pragma unroll
      for (int e = 0; e < 16; ++e)
         v[e] = (acc[i][e] + bias[e]) + residual[e];
      block.store<PLAIN>(v, out.chain);
   }
}

template <int BM, int PLANE, int WVEC>
static int launch_f32_conv3x3_split_as(hipStream_t stream, const F32Conv3x3 &a, const F32ConvStore &out, int group)
{
   constexpr int BN = F32Conv3x3SplitShape<PLANE, WVEC>::BN;
   const int tiles_m = (a.M + BM - 1) / BM, tiles_n = (a.N + BN - 1) / BN;
   if ((long long)tiles_m * tiles_n > 0x7fffffffLL)
      return fail(SOFIE_HIP_ERR_INVALID, "fp32 convolution: too many tiles");
   constexpr size_t smem = F32Conv3x3SplitShape<PLANE, WVEC>::BYTES;
   static_assert(smem <= 160 * 1024, "LDS of a CU");
   auto go = [&](auto plain) {
      auto kern = f32_conv3x3_split_kernel<BM, PLANE, WVEC, decltype(plain)::value>;
      static bool configured[64] = {};
      if (int st = configure_lds_once(kern, smem, configured))
         return st;
      const TileOrder order(tiles_m, tiles_n, 4, group);
      in_launches(order.workgroups(group), 256, [&](int first, unsigned count) {
         launch_kernel(kern, dim3(count, 1, order.depth(group)), dim3(256), smem, stream, a, out, order, first);
      });
      return launch_status("f32_conv3x3_split_kernel");
   };
   return conv3x3_plain(out.chain) ? go(std::true_type{}) : go(std::false_type{});
}

} // namespace sofie_hip
