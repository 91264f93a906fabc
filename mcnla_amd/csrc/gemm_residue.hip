// FP64 products C = A B by residues on the INT8 matrix cores (gfx950).
//
// FP64 MFMA peaks at 78.6 TFLOP/s, INT8 MFMA at 64 times that, so an FP64 product of long rows is
// cheaper as kMods exact INT8 products (the residue form of error-free matrix multiplication:
// K. Ozaki, Y. Uchino, T. Imamura, "Ozaki Scheme II", 2025; the arithmetic below is the Chinese
// remainder theorem):
//   1. scale: row i of A by 2^ea_i and column j of B by 2^eb_j, powers of two such that
//      ||a_i|| 2^ea_i and ||b_j|| 2^eb_j stay below 2^58.2 and every entry below 2^53, and round
//      to integers a', b' (the only rounding of the operands: at most 2^-57.2 of the row's norm
//      per entry);
//   2. take the residues of a', b' modulo kMods pairwise coprime p <= 256 (symmetric, one byte
//      each), and multiply modulus by modulus on v_mfma_i32_16x16x64_i8: exact for K ranges up to
//      2^17 (|r| <= 128, products below 2^14);
//   3. |sum a'b'| <= ||a'|| ||b'|| < P/2, P the product of the moduli (2^117.5), so the residues
//      of the sum determine it: the reconstruction below is exact to 2^-70 of ||a'|| ||b'||, and
//      one rounding to FP64 follows.
// The result differs from the exact product by the rounding of the operands and does not depend on
// how rows or K are cut into panels, ranges and tiles.  Measured against 128-bit sums on Gaussian
// operands, in units of sqrt(K): 3.3e-16 where the FP64 MFMA kernels have 3.4e-15 (K = 10000),
// 2.7e-16 against 1.5e-15 (K = 2503), 1.5e-16 against 7e-16 (K = 700); symmetric (squares on the
// diagonal) 6.9e-15 against 8.6e-14 (K = 100000).
//
// The error is bounded by the two rows' norms -- at most 1.7 units of 2^-53 ||a_i|| ||b_j||
// measured on any data, where sums in FP64 had 54 to 2200 -- and not entry by entry by |A||B|: an
// entry 2^-j below its row's largest keeps about 53 - j bits.  Where the large entries of two rows
// lie at different places that is less than FP64 sums give.  In units of 2^-53 |A||B|, residues
// against FP64 sums: Gaussian rows 0.8 / 54, Y = A Omega of the matrices in perf/cases.py 0.8-2 /
// 130-500, but A'A for columns with lognormal(3) entries 3.8e3 / 104, Cauchy 1.5e4 / 170, a lone
// 1e8 in each column 4e8 / 2e3.  What a solve computes from such an A'A multiplies it by dense
// matrices, which rounds by norms in any arithmetic: sigma of these three matrices (40000 x 1200,
// Gram-of-A route) are 8e-15, 9e-15 and 1.6e-14 from 64 bits, on the FP64 tiles 1.2e-14, 1.1e-14 and
// 2.6e-14.
//
// Time (FP64 kernels -> this): 100000 x 2048 x 10000 57.3 -> 33.2 ms (123 TFLOP/s of FP64 work),
// 30011 x 840 x 2503 3.39 -> 2.0 ms, 2048^2 x 100000 (symmetric) 6.7 -> 4.4 ms.
//
// Rows with a non-finite entry, or whose norm leaves [2^-400, 2^400], have no such scale: the
// scale kernels raise a device flag, at which everything after them ends at once, and the caller's
// FP64 product, launched behind it and gated on the flag, makes the result.
#include <algorithm>
#include <cmath>

#include "common.hpp"
#include "kernels.hpp"

namespace mcnla {

namespace {

typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
typedef int i32x4 __attribute__((ext_vector_type(4)));
typedef unsigned __int128 u128;

constexpr int kMods = 15;
// Pairwise coprime; the largest odd one is 251, which keeps a quotient that is off by 2/p (the
// rounding of x * (1/p) for |x| = 2^53) inside a signed byte: |r| <= p/2 + 2 <= 127.5.
struct Moduli {
  int p[kMods] = {256, 251, 249, 247, 245, 241, 239, 233, 229, 227, 223, 211, 199, 197, 193};
  constexpr int operator[](int i) const { return p[i]; }
};
constexpr Moduli kP;

constexpr u128 modulus_product() {
  u128 P = 1;
  for (int i = 0; i < kMods; ++i) P *= static_cast<u128>(kP[i]);
  return P;
}
// s_i = (P / p_i) ((P / p_i)^-1 mod p_i): s_i = 1 mod p_i and 0 modulo the others, so a sum with
// residues r_i is sum r_i s_i mod P.
constexpr u128 crt_weight(int i) {
  const u128 M = modulus_product() / static_cast<u128>(kP[i]);
  const int m = static_cast<int>(M % static_cast<u128>(kP[i]));
  int w = 1;
  while ((m * w) % kP[i] != 1) ++w;
  return M * static_cast<u128>(w);
}
// The weights and P in two parts: multiples of 2^82, and the rest rounded to FP64.  |r_i| <= 2^7, so
// the sum of the high parts is an integer multiple of 2^82 below 2^129: exact in FP64.  (The
// residues of at most kMaxRanges ranges are added first, as integers below 2^12.)
constexpr int kGrid = 82;
constexpr int kMaxRanges = 32;
constexpr double hi_part(u128 v) {
  return static_cast<double>(static_cast<uint64_t>(v >> kGrid)) * 0x1.0p82;
}
constexpr double lo_part(u128 v) {
  const u128 r = v & ((static_cast<u128>(1) << kGrid) - 1);
  return static_cast<double>(static_cast<uint64_t>(r >> 41)) * 0x1.0p41 +
         static_cast<double>(static_cast<uint64_t>(r & ((static_cast<u128>(1) << 41) - 1)));
}
struct CrtTable {
  double hi[kMods] = {}, lo[kMods] = {};
  double P_hi = 0.0, P_lo = 0.0, P_inv = 0.0;
  constexpr CrtTable() {
    for (int i = 0; i < kMods; ++i) {
      hi[i] = hi_part(crt_weight(i));
      lo[i] = lo_part(crt_weight(i));
    }
    P_hi = hi_part(modulus_product());
    P_lo = lo_part(modulus_product());
    P_inv = 1.0 / P_hi;
  }
};
constexpr CrtTable kCrt;
static_assert(modulus_product() >> 117 == 1, "P lies in [2^117, 2^118)");

// Operands are packed into blocks of 256 rows x 64 k bytes (16 KiB): [modulus][row tile][k block]
// [256][64].  The 16-byte chunk c of row r sits at chunk position c ^ ((r / 4) % 4), so that a
// linear copy into LDS gives fragment reads on distinct banks (the layout of the 16-bit sketch's
// blocks).
constexpr int kBR = 256;
constexpr int kBK = 64;
constexpr int kBlk = kBR * kBK;  // bytes
constexpr int kUnroll = 10;      // steps per loop body: 5 ring slots x 2 fragment buffers

__host__ __device__ constexpr int blk_off(int r, int chunk) {
  return r * kBK + 16 * (chunk ^ ((r >> 2) & 3));
}

// K steps, padded with zero blocks to the GEMM loop's unrolling.
int64_t k_steps(int64_t k) { return ceil_div(ceil_div(k, kBK), kUnroll) * kUnroll; }

// ---- scales -----------------------------------------------------------------------------------
// Row maxima and sums of squares over K ranges, in a fixed order.  Operand element (r, k) at
// src[r + k ld] (R_CONTIG) or src[r ld + k].
template <typename TS>
__global__ __launch_bounds__(256) void norm_rcontig_kernel(const TS* __restrict__ src, int64_t ld,
                                                           int64_t rows, int64_t K, int64_t kchunk,
                                                           double2* __restrict__ part) {
  const int64_t r = blockIdx.x * 256ll + threadIdx.x;
  if (r >= rows) return;
  const int64_t k0 = blockIdx.y * kchunk;
  const int64_t k1 = k0 + kchunk < K ? k0 + kchunk : K;
  double mx = 0.0, ss = 0.0;
  int64_t k = k0;
  for (; k + 8 <= k1; k += 8) {
    double v[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) v[i] = static_cast<double>(src[r + (k + i) * ld]);
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      mx = fmax(mx, fabs(v[i]));
      ss = fma(v[i], v[i], ss);
    }
  }
  for (; k < k1; ++k) {
    const double v = static_cast<double>(src[r + k * ld]);
    mx = fmax(mx, fabs(v));
    ss = fma(v, v, ss);
  }
  part[blockIdx.y * rows + r] = make_double2(mx, ss);
}

// Row-major operand: one wave per row.
template <typename TS>
__global__ __launch_bounds__(256) void norm_kcontig_kernel(const TS* __restrict__ src, int64_t ld,
                                                           int64_t rows, int64_t K,
                                                           double2* __restrict__ part) {
  const int64_t r = blockIdx.x * 4ll + threadIdx.x / kWave;
  const int lane = threadIdx.x % kWave;
  if (r >= rows) return;
  const TS* row = src + r * ld;
  double mx = 0.0, ss = 0.0;
#pragma unroll 4
  for (int64_t k = lane; k < K; k += kWave) {
    const double v = static_cast<double>(row[k]);
    mx = fmax(mx, fabs(v));
    ss = fma(v, v, ss);
  }
  for (int off = 32; off > 0; off >>= 1) {
    mx = fmax(mx, __shfl_xor(mx, off, kWave));
    ss += __shfl_xor(ss, off, kWave);
  }
  if (lane == 0) {
    part[r] = make_double2(mx, ss);
  }
}

__global__ void clear_flag_kernel(int* flag) { *flag = 0; }

// The exponent of each row from its partials: the largest e with ||a|| 2^e < 2^58.2 and
// max |a| 2^e < 2^53 (a zero row: 0).  A sum of squares that is NaN (a NaN or infinite entry), or
// out of [2^-800, 2^800], raises the flag.
__global__ __launch_bounds__(256) void exponent_kernel(const double2* __restrict__ part,
                                                       int64_t chunks, int64_t rows,
                                                       int* __restrict__ e, int* __restrict__ flag) {
  // 32 rows per workgroup; 8 threads per row sum every eighth partial, then one adds the 8 sums
  __shared__ double2 t[8][32];
  const int row = threadIdx.x % 32, sub = threadIdx.x / 32;
  const int64_t r = blockIdx.x * 32ll + row;
  double mx = 0.0, ss = 0.0;
  if (r < rows) {
#pragma unroll 4
    for (int64_t c = sub; c < chunks; c += 8) {
      const double2 v = part[c * rows + r];
      mx = fmax(mx, v.x);
      ss += v.y;
    }
  }
  t[sub][row] = make_double2(mx, ss);
  __syncthreads();
  if (sub != 0 || r >= rows) return;
  for (int c = 1; c < 8; ++c) {
    mx = fmax(mx, t[c][row].x);
    ss += t[c][row].y;
  }
  int ex = 0;
  if (!(ss <= 0x1.0p800) || (ss < 0x1.0p-800 && (ss > 0.0 || mx > 0.0))) {
    atomicOr(flag, 1);
  } else if (ss > 0.0) {
    int em = 0;
    (void)frexp(mx, &em);  // mx < 2^em
    // the largest e with ss 4^e < 2^116.39 (2^116.53 = P/2; the rounding of ss and of the entries
    // stays within the difference)
    int es = 0;
    const double f = frexp(ss, &es);                       // ss = f 2^es, f in [0.5, 1)
    const int room = 116 - es + ((es & 1) && f < 0.65);    // 0.65 < 2^-0.61
    ex = room >> 1;                                        // floor
    ex = ex < 53 - em ? ex : 53 - em;
  }
  e[r] = ex;
}

// ---- packing ----------------------------------------------------------------------------------
// Residues of rows [0, rows) and k in [k0, k0 + K) of an operand as int8 blocks.  A wave packs 16
// rows of one 64-k block: lane L takes row L % 16 and the 16 k of chunk L / 16, so that a load
// instruction reads whole 128-byte pieces of an R_CONTIG source and every store instruction
// writes 1 KiB of one block.  Per entry and modulus: q = round(x / p) by adding 1.5 * 2^52, then
// r = x - p q, whose low byte is read off the sum r + 1.5 * 2^52 (four FP64 VALU instructions,
// full rate on this chip; three byte permutes pack four residues).
// Memory-bound: 8 (or 4) bytes read and 15 written per entry.
template <typename TS, bool R_CONTIG>
__global__ __launch_bounds__(256) void pack_residues_kernel(
    const TS* __restrict__ src, int64_t ld, int64_t rows, int64_t K, int64_t steps, int64_t tiles,
    const int* __restrict__ exps, const int* __restrict__ flag, uint8_t* __restrict__ dst) {
  if (*flag != 0) return;
  const int lane = threadIdx.x % kWave, wave = threadIdx.x / kWave;
  const int64_t kt = R_CONTIG ? blockIdx.y : blockIdx.x;
  const int64_t strip = (R_CONTIG ? blockIdx.x : blockIdx.y) * 4ll + wave;  // 16 rows
  const int64_t tile = strip / 16;
  const int rt = static_cast<int>(strip % 16) * 16 + lane % 16;  // row in the tile
  const int chunk = lane / 16;
  const int64_t r = tile * kBR + rt, k = kt * kBK + chunk * 16;
  double x[16];
#pragma unroll
  for (int i = 0; i < 16; ++i) x[i] = 0.0;
  if (r < rows && k < K) {
    const TS* s = R_CONTIG ? src + r + k * ld : src + r * ld + k;
    const int64_t step = R_CONTIG ? ld : 1;
    const int e = exps[r];
    if (k + 16 <= K) {
#pragma unroll
      for (int i = 0; i < 16; ++i) x[i] = static_cast<double>(s[i * step]);
    } else {
#pragma unroll
      for (int i = 0; i < 16; ++i)
        if (k + i < K) x[i] = static_cast<double>(s[i * step]);
    }
#pragma unroll
    for (int i = 0; i < 16; ++i) x[i] = rint(ldexp(x[i], e));
  }
  constexpr double kMagic = 0x1.8p52;
  uint8_t* out = dst + (tile * steps + kt) * kBlk + blk_off(rt, chunk);
  const int64_t plane = tiles * steps * kBlk;
#pragma unroll
  for (int m = 0; m < kMods; ++m) {
    const double p = static_cast<double>(kP[m]), ip = 1.0 / static_cast<double>(kP[m]);
    u32x4 w;
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      uint32_t b[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const double v = x[4 * g + i];
        const double q = fma(v, ip, kMagic) - kMagic;
        const double res = fma(-q, p, v) + kMagic;
        b[i] = static_cast<uint32_t>(__builtin_bit_cast(uint64_t, res));
      }
      // the low bytes of b[0..3]
      const uint32_t lo = __builtin_amdgcn_perm(b[1], b[0], 0x0c0c0400u);
      const uint32_t hi = __builtin_amdgcn_perm(b[3], b[2], 0x0c0c0400u);
      w[g] = __builtin_amdgcn_perm(hi, lo, 0x05040100u);
    }
    *reinterpret_cast<u32x4*>(out + m * plane) = w;
  }
}

// ---- the INT8 products ------------------------------------------------------------------------
typedef __attribute__((address_space(3))) void lds_void;

// vmcnt <= VM and lgkmcnt == 0
template <int VM>
__device__ __forceinline__ void wait_vmcnt_lgkm0() {
  __builtin_amdgcn_s_waitcnt((VM & 0xF) | (0x7 << 4) | (((VM >> 4) & 3) << 14));
}
template <int VM>
__device__ __forceinline__ void wait_vmcnt() {
  __builtin_amdgcn_s_waitcnt((VM & 0xF) | (0x7 << 4) | (0xF << 8) | (((VM >> 4) & 3) << 14));
}

// acc += a b with the accumulator tied to the destination (256 live accumulators: an untied
// destination makes the register allocator copy them).  Inline asm is outside the compiler's
// hazard tracking: consecutive MFMAs on one accumulator are 64 instructions apart, and s_nops
// cover the first MFMA after the zeroing and the reads after the last one.
__device__ __forceinline__ void mfma_i8(i32x4& acc, const u32x4& a, const u32x4& b) {
  asm volatile("v_mfma_i32_16x16x64_i8 %0, %1, %2, %0" : "+a"(acc) : "v"(a), "v"(b));
}

// R[range][modulus][i][j] = (sum over the range's k of A_i B_j mod p) as int8 (accumulate: added
// to what R holds, modulo p), for tiles of 256 x 256 outputs: the structure of the 16-bit sketch kernel (4 waves of 128 x 128, blocks
// streamed by global_load_lds through a five-slot ring, fragments of step k + 1 read and the
// stage four ahead issued between the MFMA rows of step k) on twice the k per byte.  The rows of
// the MFMA result are output columns, so a lane holds 4 consecutive columns and stores them as
// one word.  Grid: ((range * kMods + modulus) * tiles + tile); sym: lower-triangle tiles only.
// Bound by the INT8 matrix cores and the L2-to-LDS path together: matrix pipe 60 % busy in the sketch
// and 51 % in the Gram at 100000 x 10000, Nl = 2048 (one wave per SIMD and a barrier per 64 k leave
// the rest), waves waiting 20 and 28 % of their cycles, 0.2 % on LDS, 39 and 18 % of the L2 requests
// missing (3.8 TB/s).  With all operands zero the same launches take 19 % less: that much is the
// clock under load.
__global__ __launch_bounds__(256) void residue_gemm_kernel(
    const uint8_t* __restrict__ Ab, const uint8_t* __restrict__ Bb, int64_t tiles_m,
    int64_t tiles_n, int64_t steps, int64_t kper, bool accumulate, bool sym, int64_t ldr,
    int64_t plane, const int* __restrict__ flag, int8_t* __restrict__ R) {
  constexpr int L = 8;  // DMA instructions per wave and stage (4 per operand)
  const int no_scale = *flag;  // looked at once the first stages are on their way
  __shared__ __attribute__((aligned(16))) uint8_t S0[2 * kBlk], S1[2 * kBlk], S2[2 * kBlk],
      S3[2 * kBlk], S4[2 * kBlk];
  const int64_t ntiles = sym ? tiles_m * (tiles_m + 1) / 2 : tiles_m * tiles_n;
  // the tiles of one modulus are dealt to the XCDs in contiguous runs where that divides evenly,
  // so that the chip works on one modulus' blocks at a time and an XCD's tiles share rows
  int64_t group, tile;
  if (ntiles % kXcds == 0) {
    group = blockIdx.x / ntiles;
    tile = xcd_swizzle(blockIdx.x % ntiles, ntiles);
  } else {
    const int64_t logical = xcd_swizzle(blockIdx.x, gridDim.x);
    group = logical / ntiles;
    tile = logical % ntiles;
  }
  const int mod = static_cast<int>(group % kMods);
  const int range = static_cast<int>(group / kMods);
  int tm, tn;
  if (sym) {
    const int t = static_cast<int>(tile);
    tm = static_cast<int>((sqrtf(8.f * static_cast<float>(t) + 1.f) - 1.f) * 0.5f);
    while (tm * (tm + 1) / 2 > t) --tm;
    while ((tm + 1) * (tm + 2) / 2 <= t) ++tm;
    tm = __builtin_amdgcn_readfirstlane(tm);  // uniform, but from vector arithmetic
    tn = t - tm * (tm + 1) / 2;
  } else {
    tm = static_cast<int>(tile / tiles_n);
    tn = static_cast<int>(tile % tiles_n);
  }
  const int lane = threadIdx.x % kWave, wave = threadIdx.x / kWave;
  const int wm0 = (wave / 2) * 128, wn0 = (wave % 2) * 128;
  const int kg = lane / 16;
  const int64_t kbeg = range * kper;
  const int64_t kend = kbeg + kper < steps ? kbeg + kper : steps;
  const uint8_t* abase = Ab + (mod * tiles_m + tm) * steps * kBlk;
  const uint8_t* bbase = Bb + (mod * tiles_n + tn) * steps * kBlk;
  auto dma = [&](const uint8_t* ak, const uint8_t* bk, uint8_t* sd, int i) {
    const int off = ((i >> 1) * 4 + wave) * 1024;  // 1 KiB per wave instruction
    if (i & 1)
      __builtin_amdgcn_global_load_lds(bk + off + lane * 16, (lds_void*)&sd[kBlk + off], 16, 0, 0);
    else
      __builtin_amdgcn_global_load_lds(ak + off + lane * 16, (lds_void*)&sd[off], 16, 0, 0);
  };
  auto issue = [&](int64_t kt, uint8_t* sd) {
#pragma unroll
    for (int i = 0; i < L; ++i) dma(abase + kt * kBlk, bbase + kt * kBlk, sd, i);
  };
  i32x4 acc[8][8];  // [column tile][row tile]
#pragma unroll
  for (int i = 0; i < 8; ++i)
#pragma unroll
    for (int j = 0; j < 8; ++j) acc[i][j] = i32x4{0, 0, 0, 0};
  u32x4 fa0[8], fb0[8], fa1[8], fb1[8];
  auto frags = [&](const uint8_t* ss, u32x4* af, u32x4* bf) {
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      af[i] = *reinterpret_cast<const u32x4*>(&ss[blk_off(wm0 + i * 16 + lane % 16, kg)]);
      bf[i] = *reinterpret_cast<const u32x4*>(&ss[kBlk + blk_off(wn0 + i * 16 + lane % 16, kg)]);
    }
  };
  // Step kt: stage kt + 1 has landed in every wave after the wait and the barrier (two stages may
  // still be in flight); the stage issued here, kt + 4 (clamped to the last block), overwrites
  // the slot whose fragments every wave read in step kt - 2.
  auto step = [&](int64_t kt, const u32x4* caf, const u32x4* cbf, const uint8_t* snext,
                  u32x4* naf, u32x4* nbf, uint8_t* sn) {
    asm volatile("" ::: "memory");
    wait_vmcnt_lgkm0<2 * L>();
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    const int64_t kn = kt + 4 < kend ? kt + 4 : kend - 1;
    const uint8_t *ak = abase + kn * kBlk, *bk = bbase + kn * kBlk;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
#pragma unroll
      for (int j = 0; j < 8; ++j) mfma_i8(acc[i][j], cbf[i], caf[j]);
      asm volatile("" ::: "memory");
      dma(ak, bk, sn, i);
      naf[i] = *reinterpret_cast<const u32x4*>(&snext[blk_off(wm0 + i * 16 + lane % 16, kg)]);
      nbf[i] =
          *reinterpret_cast<const u32x4*>(&snext[kBlk + blk_off(wn0 + i * 16 + lane % 16, kg)]);
      asm volatile("" ::: "memory");
    }
  };
  issue(kbeg, S0);
  issue(kbeg + 1, S1);
  issue(kbeg + 2, S2);
  issue(kbeg + 3, S3);
  asm volatile("" ::: "memory");
  if (no_scale != 0) {
    wait_vmcnt<0>();
    return;
  }
  wait_vmcnt<3 * L>();  // stage 0 landed in every wave
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
  frags(S0, fa0, fb0);
  asm volatile("s_nop 7");  // zeroed accumulators before their first MFMA read
  for (int64_t kt = kbeg; kt < kend; kt += kUnroll) {  // kbeg % 10 == 0: stage s in slot s % 5
    step(kt, fa0, fb0, S1, fa1, fb1, S4);
    step(kt + 1, fa1, fb1, S2, fa0, fb0, S0);
    step(kt + 2, fa0, fb0, S3, fa1, fb1, S1);
    step(kt + 3, fa1, fb1, S4, fa0, fb0, S2);
    step(kt + 4, fa0, fb0, S0, fa1, fb1, S3);
    step(kt + 5, fa1, fb1, S1, fa0, fb0, S4);
    step(kt + 6, fa0, fb0, S2, fa1, fb1, S0);
    step(kt + 7, fa1, fb1, S3, fa0, fb0, S1);
    step(kt + 8, fa0, fb0, S4, fa1, fb1, S2);
    step(kt + 9, fa1, fb1, S0, fa0, fb0, S3);
  }
  asm volatile("s_nop 7\n s_nop 7\n s_nop 7\n s_nop 7");  // last MFMAs drain before VALU reads
  wait_vmcnt<0>();  // no DMA may still target LDS when the workgroup ends
  // sums of at most 2^31 in magnitude: reduce modulo p (exact in FP64; a sum of 2^31, which wraps,
  // occurs for p = 256 only) and store 4 columns per word
  const double p = static_cast<double>(kP[mod]), ip = 1.0 / p;
  int8_t* Rp = R + (static_cast<int64_t>(range) * kMods + mod) * plane;
  constexpr double kMagic = 0x1.8p52;
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    const int64_t gi = tm * kBR + wm0 + j * 16 + lane % 16;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const int64_t gj = tn * kBR + wn0 + i * 16 + 4 * (lane / 16);
      uint32_t* dst = reinterpret_cast<uint32_t*>(Rp + gi * ldr + gj);
      const uint32_t old = accumulate ? *dst : 0u;
      uint32_t b[4];
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const double v = static_cast<double>(acc[i][j][r]) +
                         static_cast<double>(static_cast<int8_t>(old >> (8 * r)));
        const double q = fma(v, ip, kMagic) - kMagic;
        b[r] = static_cast<uint32_t>(__builtin_bit_cast(uint64_t, fma(-q, p, v) + kMagic));
      }
      const uint32_t lo = __builtin_amdgcn_perm(b[1], b[0], 0x0c0c0400u);
      const uint32_t hi = __builtin_amdgcn_perm(b[3], b[2], 0x0c0c0400u);
      *dst = __builtin_amdgcn_perm(hi, lo, 0x05040100u);
    }
  }
}

// ---- reconstruction ---------------------------------------------------------------------------
// The sums of 4 consecutive columns from their residues: R points at modulus 0 of range 0.  The
// ranges' residues are added and reduced before the weights are applied, so that what the FP64
// arithmetic sees is the residue of the whole sum in [-p/2, p/2], however K was cut (the GEMM
// leaves that residue for one range; the two-part sums below are rounded, and would differ in
// their last bits for other representatives).
__device__ __forceinline__ void reconstruct4(const int8_t* __restrict__ R, int64_t plane,
                                             int ranges, double* out) {
  int r[kMods][4];
#pragma unroll
  for (int m = 0; m < kMods; ++m) {
    const uint32_t w = *reinterpret_cast<const uint32_t*>(R + m * plane);
#pragma unroll
    for (int i = 0; i < 4; ++i) r[m][i] = static_cast<int8_t>(w >> (8 * i));
  }
  if (ranges > 1) {
    for (int g = 1; g < ranges; ++g) {
      const int8_t* Rg = R + g * kMods * plane;
      uint32_t w[kMods];
#pragma unroll
      for (int m = 0; m < kMods; ++m) w[m] = *reinterpret_cast<const uint32_t*>(Rg + m * plane);
#pragma unroll
      for (int m = 0; m < kMods; ++m)
#pragma unroll
        for (int i = 0; i < 4; ++i) r[m][i] += static_cast<int8_t>(w[m] >> (8 * i));
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      r[0][i] = static_cast<int8_t>(r[0][i]);  // p = 256: -128, never 128, as the GEMM stores it
#pragma unroll
      for (int m = 1; m < kMods; ++m) {  // odd p: no ties, and |sum| / p < 2^5 is far from one
        const float s = static_cast<float>(r[m][i]);
        r[m][i] -= kP[m] * static_cast<int>(rintf(s * (1.0f / static_cast<float>(kP[m]))));
      }
    }
  }
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    double c1 = 0.0, c2 = 0.0;
#pragma unroll
    for (int m = 0; m < kMods; ++m) {
      const double x = static_cast<double>(r[m][i]);
      c1 = fma(x, kCrt.hi[m], c1);
      c2 = fma(x, kCrt.lo[m], c2);
    }
    const double q = rint(c1 * kCrt.P_inv);
    out[i] = fma(-q, kCrt.P_hi, c1) + fma(-q, kCrt.P_lo, c2);
  }
}

// C (rows x N, row-major) from the residue planes (leading dimension ldr).  A thread makes 4
// columns of one row: 15 words read, 4 FP64 written.
__global__ __launch_bounds__(256) void reconstruct_kernel(const int8_t* __restrict__ R, int64_t ldr,
                                                          int64_t plane, int ranges, int64_t rows,
                                                          int64_t N, const int* __restrict__ ea,
                                                          const int* __restrict__ eb,
                                                          const int* __restrict__ flag,
                                                          double* __restrict__ C, int64_t ldc) {
  if (*flag != 0) return;
  const int64_t quads = ceil_div(N, 4), total = rows * quads;
  for (int64_t t = blockIdx.x * 256ll + threadIdx.x; t < total; t += gridDim.x * 256ll) {
    const int64_t i = t / quads, j = (t % quads) * 4;
    double v[4];
    reconstruct4(R + i * ldr + j, plane, ranges, v);
    const int e = ea[i];
#pragma unroll
    for (int c = 0; c < 4; ++c)
      if (j + c < N) C[i * ldc + j + c] = ldexp(v[c], -(e + eb[j + c]));
  }
}

// The symmetric case: 64 x 64 tiles of the lower triangle, each written with its mirror image
// (through LDS, so that both go out in whole rows).
__global__ __launch_bounds__(256) void reconstruct_sym_kernel(const int8_t* __restrict__ R,
                                                              int64_t ldr, int64_t plane,
                                                              int ranges, int64_t N,
                                                              const int* __restrict__ e,
                                                              const int* __restrict__ flag,
                                                              double* __restrict__ C,
                                                              int64_t ldc) {
  __shared__ double t[64][65];
  if (*flag != 0) return;
  const int64_t x = blockIdx.x;
  int64_t ti = static_cast<int64_t>((sqrt(8.0 * static_cast<double>(x) + 1.0) - 1.0) / 2.0);
  while (ti * (ti + 1) / 2 > x) --ti;
  while ((ti + 1) * (ti + 2) / 2 <= x) ++ti;
  const int64_t tj = x - ti * (ti + 1) / 2;
  for (int u = threadIdx.x; u < 64 * 16; u += 256) {
    const int r = u / 16, c = (u % 16) * 4;
    const int64_t i = ti * 64 + r, j = tj * 64 + c;
    if (i < N) {  // columns past N read padding of the planes and are not written
      double v[4];
      reconstruct4(R + i * ldr + j, plane, ranges, v);
#pragma unroll
      for (int q = 0; q < 4; ++q)
        t[r][c + q] = j + q < N ? ldexp(v[q], -(e[i] + e[j + q])) : 0.0;
    }
  }
  __syncthreads();
  for (int u = threadIdx.x; u < 64 * 64; u += 256) {
    const int r = u / 64, c = u % 64;
    const int64_t i = ti * 64 + r, j = tj * 64 + c;
    if (i < N && j < N) C[i * ldc + j] = t[r][c];
    const int64_t i2 = tj * 64 + r, j2 = ti * 64 + c;
    if (ti != tj && i2 < N && j2 < N) C[i2 * ldc + j2] = t[c][r];
  }
}

// ---- host side --------------------------------------------------------------------------------
struct Operand {
  const void* p;
  int64_t ld;
  bool f32, rcontig;
  const void* at(int64_t r, int64_t k) const {
    const int64_t o = rcontig ? r + k * ld : r * ld + k;
    return f32 ? static_cast<const void*>(static_cast<const float*>(p) + o)
               : static_cast<const void*>(static_cast<const double*>(p) + o);
  }
};

// K ranges of the norm pass over an R_CONTIG operand: enough workgroups to fill the device, each
// with at least 64 k; and the most (range, row) pairs for any number of rows up to `rows`.
int64_t norm_chunks(const Operand& o, int64_t rows, int64_t K) {
  if (!o.rcontig) return 1;
  const int64_t blocks = ceil_div(rows, 256);
  return std::max<int64_t>(1, std::min<int64_t>(ceil_div(4096, blocks), ceil_div(K, 64)));
}

size_t norm_pairs(const Operand& o, int64_t rows, int64_t K) {
  if (!o.rcontig) return rows;
  return static_cast<size_t>(std::min<int64_t>(ceil_div(K, 64) * rows, (int64_t{1} << 20) + rows));
}

template <typename TS>
void launch_norms(const Operand& o, const void* src, int64_t rows, int64_t K, double2* part,
                  int64_t chunks, hipStream_t st) {
  if (o.rcontig) {
    const int64_t kc = ceil_div(K, chunks);
    hipLaunchKernelGGL(norm_rcontig_kernel<TS>,
                       dim3(static_cast<unsigned>(ceil_div(rows, 256)),
                            static_cast<unsigned>(ceil_div(K, kc))),
                       dim3(256), 0, st, static_cast<const TS*>(src), o.ld, rows, K, kc, part);
  } else {
    hipLaunchKernelGGL(norm_kcontig_kernel<TS>, dim3(static_cast<unsigned>(ceil_div(rows, 4))),
                       dim3(256), 0, st, static_cast<const TS*>(src), o.ld, rows, K, part);
  }
  MCNLA_LAUNCHED();
}

void scales(const Operand& o, int64_t r0, int64_t rows, int64_t K, double2* part, int* e, int* flag,
            hipStream_t st) {
  int64_t chunks = norm_chunks(o, rows, K);
  chunks = ceil_div(K, ceil_div(K, chunks));
  const void* src = o.at(r0, 0);
  if (o.f32)
    launch_norms<float>(o, src, rows, K, part, chunks, st);
  else
    launch_norms<double>(o, src, rows, K, part, chunks, st);
  hipLaunchKernelGGL(exponent_kernel, dim3(static_cast<unsigned>(ceil_div(rows, 32))), dim3(256),
                     0, st, part, chunks, rows, e, flag);
  MCNLA_LAUNCHED();
}

template <typename TS>
void launch_pack(const Operand& o, const void* src, int64_t rows, int64_t K, int64_t steps,
                 int64_t tiles, const int* e, const int* flag, uint8_t* dst, hipStream_t st) {
  const unsigned strips = static_cast<unsigned>(tiles * (kBR / 64));
  const TS* s = static_cast<const TS*>(src);
  if (o.rcontig)
    hipLaunchKernelGGL((pack_residues_kernel<TS, true>),
                       dim3(strips, static_cast<unsigned>(steps)), dim3(256), 0, st, s, o.ld, rows,
                       K, steps, tiles, e, flag, dst);
  else
    hipLaunchKernelGGL((pack_residues_kernel<TS, false>),
                       dim3(static_cast<unsigned>(steps), strips), dim3(256), 0, st, s, o.ld, rows,
                       K, steps, tiles, e, flag, dst);
  MCNLA_LAUNCHED();
}

void pack(const Operand& o, int64_t r0, int64_t rows, int64_t k0, int64_t K, int64_t steps,
          int64_t tiles, const int* e, const int* flag, uint8_t* dst, hipStream_t st) {
  const void* src = o.at(r0, k0);
  if (o.f32)
    launch_pack<float>(o, src, rows, K, steps, tiles, e, flag, dst, st);
  else
    launch_pack<double>(o, src, rows, K, steps, tiles, e, flag, dst, st);
}

constexpr int64_t kMaxK = 1 << 17;  // |sum| <= 2^14 K < 2^31 (2^31 = 0 mod 256)

size_t align256(size_t v) { return (v + 255) / 256 * 256; }

// How a product is cut into panels: M panels of `rows` with the whole K (general), or K panels
// (symmetric), each multiplied in `ranges` K ranges of kper steps.  The norms' partials lie where the
// first product's residues go: the exponents are made before it.
struct Plan {
  int64_t rows = 0, kpanel = 0, panels = 0, steps = 0, ranges = 0, kper = 0;
  size_t off_part = 0, off_ea = 0, off_eb = 0, off_b = 0, off_a = 0, off_r = 0, bytes = 0;
  double cost = 0.0;  // GEMM time in steps of a workgroup (kStepUs each)
};

// Measured on MI355X (K = 10000, 1 to 32 row tiles of 8 column tiles): a workgroup costs its steps
// plus about 11 of start and epilogue, 0.83 us a step; a partial round of the CUs costs between
// its share and a whole round (the matrix cores are power-limited when all run: 2.3 POPS, 0.79 us
// a step on a half-empty device); a panel costs about 20 steps of launches and of a device that
// drains.
constexpr int64_t kStart = 11, kPanel = 20;
constexpr double kStepUs = 0.83;
double grid_cost(int64_t cus, int64_t blocks, int64_t per) {
  const double rounds = static_cast<double>(blocks) / static_cast<double>(cus);
  const double whole = static_cast<double>(ceil_div(blocks, cus));
  return (0.6 * whole + 0.4 * (rounds < 1.0 ? 1.0 : rounds)) * static_cast<double>(per + kStart);
}

// Cuts `steps` into `ranges` ranges (in whole loop bodies) for `tiles` output tiles; false when a
// range would hold more than 2^17 k.
bool set_ranges(Plan& p, int64_t cus, int64_t tiles, int64_t ranges) {
  const int64_t units = p.steps / kUnroll;
  p.kper = ceil_div(units, ranges) * kUnroll;
  p.ranges = ceil_div(p.steps, p.kper);
  p.cost = grid_cost(cus, tiles * kMods * p.ranges, p.kper);
  return ranges <= units && p.kper * kBK <= kMaxK;
}

Plan plan_general(const ResidueArgs& a, int64_t cus, int64_t tm, int64_t ranges) {
  Plan p;
  const Operand A{a.A, a.lda, a.a_f32, a.a_mcontig}, B{a.B, a.ldb, false, a.b_ncontig};
  const int64_t tn = ceil_div(a.N, kBR);
  p.rows = tm * kBR;
  p.panels = ceil_div(a.M, p.rows);
  p.steps = k_steps(a.K);
  if (!set_ranges(p, cus, tm * tn, ranges)) return Plan{};
  const int64_t last = ceil_div(a.M, kBR) - (p.panels - 1) * tm;  // tile rows of the last panel
  p.cost = (p.panels - 1) * p.cost + kPanel * p.panels +
           grid_cost(cus, last * tn * kMods * p.ranges, p.kper);
  size_t o = 0;
  p.off_ea = o;
  o += align256(4 * a.M);
  p.off_eb = o;
  o += align256(4 * a.N);
  p.off_b = o;
  o += static_cast<size_t>(kMods) * tn * p.steps * kBlk;
  p.off_a = o;
  o += static_cast<size_t>(kMods) * tm * p.steps * kBlk;
  p.off_r = p.off_part = o;
  o += std::max(align256(16 * std::max(norm_pairs(A, a.M, a.K), norm_pairs(B, a.N, a.K))),
                static_cast<size_t>(p.ranges) * kMods * p.rows * tn * kBR);
  p.bytes = o;
  return p;
}

Plan plan_sym(const ResidueArgs& a, int64_t cus, int64_t panels, int64_t ranges) {
  Plan p;
  const Operand A{a.A, a.lda, a.a_f32, a.a_mcontig};
  const int64_t tm = ceil_div(a.M, kBR);
  p.rows = tm * kBR;
  p.kpanel = ceil_div(ceil_div(a.K, panels), kBK * kUnroll) * kBK * kUnroll;
  p.panels = ceil_div(a.K, p.kpanel);
  p.steps = p.kpanel / kBK;
  if (!set_ranges(p, cus, tm * (tm + 1) / 2, ranges)) return Plan{};
  p.cost = p.panels * (p.cost + kPanel);
  size_t o = 0;
  p.off_ea = o;
  o += align256(4 * a.M);
  p.off_a = o;
  o += static_cast<size_t>(kMods) * tm * p.steps * kBlk;
  p.off_r = p.off_part = o;
  o += std::max(align256(16 * norm_pairs(A, a.M, a.K)),
                static_cast<size_t>(p.ranges) * kMods * p.rows * p.rows);
  p.bytes = o;
  return p;
}

// The cheapest plan within `limit` bytes; bytes 0: none.  (A few dozen candidates: this runs on
// the host in every product.)
Plan plan_for(const ResidueArgs& a, size_t limit) {
  Plan best;
  if (a.M < 1 || a.N < 1 || a.K < 1) return best;
  const int64_t cus = compute_units(), tm = ceil_div(a.M, kBR), tn = ceil_div(a.N, kBR);
  auto consider = [&](int64_t i, int64_t tiles, int64_t steps) {
    // ranges: as few as 2^17 k each allow, more while the grid is short
    int64_t r = std::max<int64_t>(1, ceil_div(steps * kBK, kMaxK));
    for (; r <= kMaxRanges; ++r) {
      const Plan p = a.sym ? plan_sym(a, cus, i, r) : plan_general(a, cus, i, r);
      // a larger workspace has to be worth it
      if (p.bytes != 0 && p.bytes <= limit &&
          (best.bytes == 0 || p.cost < best.cost * (p.bytes > best.bytes ? 0.99 : 1.0)))
        best = p;
      if (p.bytes != 0 && tiles * kMods * r > 8 * cus) break;
    }
  };
  if (a.sym) {
    for (int64_t panels = 1; panels <= 64; panels += ceil_div(panels, 4))
      consider(panels, tm * (tm + 1) / 2, ceil_div(ceil_div(a.K, panels), kBK));
  } else {
    for (int64_t rows = 1; rows <= std::min<int64_t>(tm, 40); rows += ceil_div(rows, 8))
      consider(rows, rows * tn, k_steps(a.K));
    if (tm <= 40) consider(tm, tm * tn, k_steps(a.K));
  }
  return best;
}

}  // namespace

size_t residue_bytes(const ResidueArgs& a, size_t limit, double* cost) {
  const Plan p = plan_for(a, limit);
  if (cost) *cost = p.cost;
  return p.bytes;
}

// Both sides measured on MI355X.  The FP64 kernels: the register-fed tiles in whole rounds of the
// CUs, 64 x 64 at 44 TFLOP/s or 32 x 32 at 38, or 256 x 128 DMA tiles (M-contiguous FP64 A of even
// sizes) at 0.237 us per k and round, the rows past whole rounds with K split in up to 4.  The
// residue product: its INT8 grid, the norm, pack and reconstruction passes at 5 TB/s and 30 us of
// launches.  Examples (FP64 / residue): 100000 x 2048 x 10000 57.3 / 33.1 ms,
// 30011 x 840 x 2503 2.9 / 1.95 ms, 10000 x 800 x 4000 1.1 / 1.03 ms, but 40000 x 800 x 1000
// 1.26 / 1.58 ms and 10000 x 400 x 1000 0.2 / 0.28 ms (start-up, padding and epilogue of 20-step
// workgroups).  Symmetric, where the DMA side also writes and sums its split-K partials (`limit`
// is their size): 2048^2 x 100000 6.62 / 4.37 ms, 1000^2 x 10000 265 / 205 us; 640^2 x 10000
// (125 / 130 us), 512^2 x 10000 and 1000^2 x 3000 are even.
bool residue_pays(const ResidueArgs& a, size_t limit) {
  const double M = static_cast<double>(a.M), N = static_cast<double>(a.N),
               K = static_cast<double>(a.K);
  if (a.K < 256 || a.M < 128 || a.N < 16) return false;
  const int64_t cus = compute_units();
  double fp64;
  if (a.sym) {
    const int64_t tm = ceil_div(a.M, 256), t64 = ceil_div(a.M, 64);
    fp64 = std::min(static_cast<double>(tm * (tm + 1)) * K * 0.237 / static_cast<double>(cus) +
                        2 * static_cast<double>(limit) / 4.5e6,
                    static_cast<double>(t64 * (t64 + 1)) * 4096 * K / 44e6 + 15.0);
  } else {
    fp64 = HUGE_VAL;
    for (int wg = 1; wg <= 2; ++wg) {
      const int64_t t = ceil_div(a.M, 32 * wg) * ceil_div(a.N, 32 * wg);
      fp64 = std::min(fp64, static_cast<double>(ceil_div(t, cus)) *
                                (static_cast<double>(cus * 2048 * wg * wg) * K /
                                     (wg == 1 ? 38e6 : 44e6) + 4.0));
    }
  }
  if (!a.sym && a.a_mcontig && !a.a_f32 && a.b_ncontig && a.N >= 128 && a.M % 2 == 0 &&
      a.N % 2 == 0) {
    // the DMA tiles; by the shape alone, so that a problem takes one path wherever its operands lie
    const int64_t tiles = ceil_div(a.M, 256) * ceil_div(a.N, 128), full = tiles / cus;
    const int64_t rest = tiles - full * cus;
    double last = rest ? 1.0 : 0.0;
    if (full > 0 && rest > 0 && 2 * rest <= cus)
      last = 1.0 / static_cast<double>(std::min<int64_t>(cus / rest, 4));
    fp64 = std::min(fp64, (static_cast<double>(full) + last) * K * 0.237);
  }
  if (fp64 < 60.0) return false;
  const Plan p = plan_for(a, limit);
  if (p.bytes == 0) return false;
  const double padk = static_cast<double>(p.steps * (a.sym ? p.panels : 1) * kBK) / K;
  double traffic = M * K * (2 * (a.a_f32 ? 4.0 : 8.0) + kMods * padk);
  if (a.sym)
    traffic += N * N * (8 + 0.5 * kMods * static_cast<double>(p.ranges));
  else
    traffic += N * K * (16 + kMods * padk) + M * N * (8 + kMods * static_cast<double>(p.ranges));
  return p.cost * kStepUs + traffic / 5e6 + 40.0 < 0.95 * (fp64 + 10.0);
}

void gemm_residue(const ResidueArgs& a, void* ws, size_t ws_bytes, int* flag, hipStream_t st) {
  const Plan p = plan_for(a, ws_bytes);
  MCNLA_REQUIRE(p.bytes != 0 && p.bytes <= ws_bytes, MCNLA_ERR_INVALID,
                "residue product workspace too small");
  char* w = static_cast<char*>(ws);
  double2* part = reinterpret_cast<double2*>(w + p.off_part);
  int* ea = reinterpret_cast<int*>(w + p.off_ea);
  uint8_t* pa = reinterpret_cast<uint8_t*>(w + p.off_a);
  int8_t* R = reinterpret_cast<int8_t*>(w + p.off_r);
  const Operand A{a.A, a.lda, a.a_f32, a.a_mcontig};
  hipLaunchKernelGGL(clear_flag_kernel, dim3(1), dim3(1), 0, st, flag);
  MCNLA_LAUNCHED();
  auto gemm = [&](const uint8_t* pb, int64_t tm, int64_t tn, bool accumulate, int64_t ldr,
                  int64_t plane) {
    const int64_t tiles = a.sym ? tm * (tm + 1) / 2 : tm * tn;
    const int64_t blocks = tiles * kMods * p.ranges;
    MCNLA_REQUIRE(blocks < (1LL << 31), MCNLA_ERR_INVALID, "GEMM grid too large");
    hipLaunchKernelGGL(residue_gemm_kernel, dim3(static_cast<unsigned>(blocks)), dim3(256), 0, st,
                       pa, pb, tm, tn, p.steps, p.kper, accumulate, a.sym, ldr, plane, flag, R);
    MCNLA_LAUNCHED();
  };
  if (a.sym) {
    const int64_t tm = p.rows / kBR;
    scales(A, 0, a.M, a.K, part, ea, flag, st);
    const int64_t plane = p.rows * p.rows;
    for (int64_t q = 0; q < p.panels; ++q) {
      const int64_t k0 = q * p.kpanel, kn = std::min(p.kpanel, a.K - k0);
      pack(A, 0, a.M, k0, kn, p.steps, tm, ea, flag, pa, st);
      gemm(pa, tm, tm, q > 0, p.rows, plane);
    }
    const int64_t T = ceil_div(a.M, 64);
    hipLaunchKernelGGL(reconstruct_sym_kernel, dim3(static_cast<unsigned>(T * (T + 1) / 2)),
                       dim3(256), 0, st, R, p.rows, plane, static_cast<int>(p.ranges),
                       a.M, ea, flag, a.C, a.ldc);
    MCNLA_LAUNCHED();
    return;
  }
  const Operand B{a.B, a.ldb, false, a.b_ncontig};
  int* eb = reinterpret_cast<int*>(w + p.off_eb);
  uint8_t* pb = reinterpret_cast<uint8_t*>(w + p.off_b);
  const int64_t tn = ceil_div(a.N, kBR);
  scales(B, 0, a.N, a.K, part, eb, flag, st);
  scales(A, 0, a.M, a.K, part, ea, flag, st);
  pack(B, 0, a.N, 0, a.K, p.steps, tn, eb, flag, pb, st);
  for (int64_t r0 = 0; r0 < a.M; r0 += p.rows) {
    const int64_t rows = std::min(p.rows, a.M - r0), tm = ceil_div(rows, kBR);
    pack(A, r0, rows, 0, a.K, p.steps, tm, ea + r0, flag, pa, st);
    const int64_t ldr = tn * kBR, plane = tm * kBR * ldr;
    gemm(pb, tm, tn, false, ldr, plane);
    const int64_t quads = rows * ceil_div(a.N, 4);
    const int64_t blocks = std::min<int64_t>(ceil_div(quads, 256), 16384);
    hipLaunchKernelGGL(reconstruct_kernel, dim3(static_cast<unsigned>(blocks)), dim3(256), 0, st,
                       R, ldr, plane, static_cast<int>(p.ranges), rows, a.N, ea + r0, eb, flag,
                       a.C + r0 * a.ldc, a.ldc);
    MCNLA_LAUNCHED();
  }
}

}  // namespace mcnla
