// The dequant GEMM of the prefill linears (gfx950): bf16 / fp16 activations x a tiled 4- or 8-bit weight.
// Included by the translation units that instantiate it per weight format.
#pragma once

#include <type_traits>

#include "sqx_common.h"

namespace sqx {

typedef unsigned u32x2_t __attribute__((__vector_size__(2 * sizeof(unsigned))));

constexpr int kGemmGroupM = 4;  // tile rows per group in the walk over output tiles

// Output tile (tm, tn) of workgroup `bid`.
__device__ inline void mx_tile_of(int bid, int tiles_m, int tiles_n, int& tm, int& tn) {
  const int total = tiles_m * tiles_n;
  int lin = bid;
  if ((total & 7) == 0) lin = (bid & 7) * (total >> 3) + (bid >> 3);  // XCD b % 8 gets a contiguous range
  const int per_group = kGemmGroupM * tiles_n;
  const int g = lin / per_group;
  const int first_m = g * kGemmGroupM;
  const int gm = min(tiles_m - first_m, kGemmGroupM);
  const int r = lin - g * per_group;
  tm = first_m + r % gm;
  tn = r / gm;
}

// y[m, n] = sum_k x[m, k] W[n, k] (+ bias[n]) for x [M, K] row-major and W in the tiled layout of
// sqx_int4.hip (group INT4, symmetric or asymmetric), sqx_fp4.hip (MXFP4 / NVFP4), sqx_int8.hip or
// sqx_fp8.hip: the prefill form of w4a16_linear (int4_group.py:148-164), awq_linear (awq.py:184-192),
// the config-4 FP4-weight linear, the int8 weight-only linear and fp8_linear (fp8_weights.py:211-262).
// Each weight is decoded to the activation dtype in registers: INT4 as the fp32 (q - z) * s rounded to
// nearest even, exactly as the reference's dequantize(...).to(x.dtype) produces it; FP4 as
// e2m1 * scale (exact; NVFP4's global scale multiplies the fp32 result); int8 and E4M3 codes as their
// values (exact in bf16 and fp16), with the per-output-channel scale cs[n] (and for FP8 the
// per-token scale rs[m]) on the fp32 sum.
//
// Tiling. A workgroup owns a TMR x TNC output tile. Its waves form a 2 x TNC/64 grid of 64-column parts
// (TMR/2 rows each, TMR/32 x 4 tiles of v_mfma_f32_16x16x32 with the weight as the first operand, so a
// lane's four accumulators are four consecutive output columns of one row), times KG k-groups: with
// KG = 2 the second half of the waves takes the second 32 columns of every stage and the two halves'
// sums are added through LDS at the end, which gives a 128 x 128 tile two waves per SIMD without a
// second workgroup's partials. A stage covers 64 k: the activation rows (128 bytes each, 16-byte chunks
// XOR-swizzled by row so the operand reads of 8 consecutive rows hit distinct banks), the weight bytes
// of the TNC/16 row tiles for those 64 columns, and their scales; NS stages form a ring filled by
// buffer -> LDS copies NS - 1 stages ahead. Every wave decodes its own 4 weight tiles per 32-k MFMA step
// (the decode is shared by the wave's row tiles).
namespace dqg {
constexpr int kBK = 64;
constexpr int kEpiPitch = 136;  // LDS bytes per row of a wave's (TMR / 2) x 64 16-bit output tile
}  // namespace dqg

// Weight formats of the dequant GEMM.
enum : int { kDqInt4 = 0, kDqMx = 1, kDqNv = 2, kDqI8 = 3, kDqF8 = 4 };

template <int FMT, bool ASYM, bool PBF16, int GROUP, int TMR, int TNC, int KG, int NS>
struct DqW {
  static constexpr bool B8 = FMT == kDqI8 || FMT == kDqF8;  // 8-bit codes: 64-column blocks, no group parameters
  static constexpr int WT = TNC / 16;                        // weight row tiles of an output tile
  static constexpr int NWG = 2 * (TNC / 64);                 // waves of a k-group: two along m, TNC / 64 along n
  static constexpr int NW = NWG * KG;
  static constexpr int TPW = WT / NW;                        // weight row tiles a wave copies (1 or 2)
  // parameter bytes per stage and tile: INT4 scales (and zero-points) of the stage's groups;
  // MXFP4 32 E8M0 bytes (lanes 32h..32h+31 of the 64-byte block), NVFP4 64 E4M3 bytes
  // asymmetric bf16 INT4 parameters are (scale, zero) pairs in one dword (sqx_int4_tile)
  static constexpr bool PAIR = ASYM && PBF16;
  static constexpr bool ZSEP = ASYM && !PBF16;  // zero-points in a buffer of their own
  static constexpr int PB = (PBF16 && !PAIR) ? 2 : 4;
  static_assert(TPW == 1 || TPW == 2, "one or two weight row tiles per wave");
  // weight copies per wave per stage: 1 KiB per 8-bit tile; two dwords a lane per INT4 tile; FP4's 512 bytes
  // a tile as one 16-byte copy for two tiles or two 4-byte copies for one
  static constexpr int kWInstr = FMT == kDqInt4 ? 2 * TPW : B8 ? TPW : 3 - TPW;
  static constexpr int NGS = GROUP >= 64 ? 1 : 64 / GROUP;  // INT4 groups per stage
  static constexpr int NP = B8 ? 0 : FMT == kDqMx ? WT / 8 : FMT == kDqNv ? WT / 4 : (ZSEP ? 2 : 1) * NGS * WT * 16 * PB / 256;
  static constexpr int kPInstr = (NP + NW - 1) / NW;  // parameter copies per wave per stage (0, 1 or 2)
  static_assert(kPInstr <= 2, "one offset per copy in a 2-vector");
  // LDS bytes: activations | weights | parameters of one stage; the epilogue reuses the stages
  static constexpr int kXBytes = TMR * dqg::kBK * 2;
  static constexpr int kWTile = B8 ? 1024 : 512;  // a weight row tile's bytes of one stage
  static constexpr int kWBytes = WT * kWTile;
  static constexpr int kPBytes = kPInstr * NW * 256;  // every wave issues kPInstr copies; those past NP write zeros
  static constexpr int kStage = kXBytes + kWBytes + kPBytes;
  static constexpr int kEpi = NWG * (TMR / 2) * dqg::kEpiPitch;
  static constexpr int kRed = KG == 2 ? NW * (TMR / 64) * 4 * 1024 : 0;  // each wave hands over half its tiles
  static constexpr int kLds = std::max(std::max(kEpi, kRed), NS * kStage);
  static_assert(kLds <= 160 * 1024, "one workgroup's LDS");
};

template <class A, int FMT, bool ASYM, bool PBF16, int GROUP, int YKIND, int TMR, int TNC, int KG, int NS>
__global__ __launch_bounds__(2 * TNC * KG, 2) void dq_gemm_kernel(const uint16_t* __restrict__ x, const uint8_t* __restrict__ wt,
                                                     const void* __restrict__ st, const void* __restrict__ zt,
                                                     const float* __restrict__ s_global, const float* __restrict__ rs,
                                                     void* __restrict__ y, const uint16_t* __restrict__ bias, int m, int n, int K, int KB,
                                                     int tiles_m, int tiles_n, int vec16, int splits,
                                                     float* __restrict__ ws) {
  using P = DqW<FMT, ASYM, PBF16, GROUP, TMR, TNC, KG, NS>;
  static_assert((TMR == 256 || TMR == 128) && (TNC == 256 || TNC == 128), "256 or 128 output rows and columns");
  constexpr int group = GROUP;
  extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
  constexpr int NW = P::NW;
  constexpr int RPW = TMR / NW;   // activation rows a wave copies
  constexpr int kXI = RPW / 8;    // activation copies per wave per stage (8 rows each)
  constexpr int MT = TMR / 32;    // 16-row MFMA tiles of a wave (it owns TMR / 2 rows)
  constexpr int kPerStage = kXI + P::kWInstr + P::kPInstr;  // buffer -> LDS copies per wave per stage
  static_assert(kPerStage * (NS - 2) < 64, "vmcnt is 6 bits");
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  int tm, tn;
  // split-K: workgroup b computes split b % splits of tile b / splits (stages s0 .. s0+S-1)
  const int tile = blockIdx.x / splits, split = blockIdx.x - tile * splits;
  mx_tile_of(tile, tiles_m, tiles_n, tm, tn);
  const int S_all = P::B8 ? KB : 2 * KB;  // stages of 64 columns (4-bit weights are padded to 128-column blocks)
  const int Sp = (S_all + splits - 1) / splits;
  const int s0 = split * Sp;
  const int S = min(S_all, s0 + Sp) - s0;
  const int wT = (n + 15) >> 4;
  const int w_t0 = tn * P::WT;
  const int Gp = KB * (128 / (FMT == kDqInt4 ? GROUP : 128));  // INT4 groups per row (padded)

  const rsrc_t xr = make_rsrc(x, (uint32_t)((uint64_t)m * (uint64_t)K * 2u));
  const rsrc_t wr = make_rsrc(wt, (uint32_t)wT * (uint32_t)KB * 1024u);
  uint32_t pbytes;
  if (P::B8) pbytes = 0u;
  else if (FMT == kDqInt4) pbytes = (uint32_t)wT * (uint32_t)Gp * 16u * P::PB;
  else pbytes = (uint32_t)wT * (uint32_t)KB * (FMT == kDqMx ? 64u : 128u);
  const rsrc_t sr = make_rsrc(st, pbytes);
  const rsrc_t zr = make_rsrc(ASYM ? zt : st, pbytes);
  constexpr int np = P::NP;

  // ---- copies. Per-lane offsets are fixed for the whole walk; a stage's position rides in the scalar
  // offset. Offsets of rows past the last one lie past the buffer resource (zeros, no memory traffic;
  // 2 GiB: an operand's bytes and a stage's offset are both below it).
  constexpr uint32_t kNone = 0x80000000u;
  // a vector, not an array: hipcc drops the host stub of a kernel whose lambda indexes a captured array
  // in the builtin
  u32x4_t xoff = u32x4_t{kNone, kNone, kNone, kNone};
  static_assert(kXI <= 4, "one offset per copy in a 4-vector");
#pragma unroll
  for (int j = 0; j < kXI; ++j) {
    const int r = RPW * wave + 8 * j + (lane >> 3);
    const int R = tm * TMR + r;
    if (R < m) xoff[j] = ((uint32_t)R * (uint32_t)K + 8u * (uint32_t)((lane & 7) ^ (r & 7))) * 2u;
  }
  const uint32_t wrow = (uint32_t)KB * 1024u;  // bytes of one weight row tile
  // FP4 with two tiles per wave: tile 2w from lanes 0-31, tile 2w + 1 from lanes 32-63, 512 bytes each
  const uint32_t wvo = (P::B8 || FMT == kDqInt4) ? (uint32_t)lane * 16u
                       : P::TPW == 1 ? (uint32_t)min(w_t0 + wave, wT - 1) * wrow + (uint32_t)lane * 4u
                                     : (uint32_t)min(w_t0 + 2 * wave + (lane >> 5), wT - 1) * wrow + (uint32_t)(lane & 31) * 16u;
  // parameter copies: index kPInstr wave + j; those past np read nothing
  u32x2_t poff = u32x2_t{kNone, kNone};
  if constexpr (!P::B8) {
#pragma unroll
    for (int j = 0; j < P::kPInstr; ++j) {
      const int pr = P::kPInstr * wave + j;
      if (pr >= np) continue;
      if (FMT == kDqInt4) {
        // layout in LDS: [scales | zeros][group gi][tile f][row] of PB bytes; 256 bytes per copy
        constexpr int TPI = 256 / (16 * P::PB);  // tiles per copy
        const int per_kind = np / (P::ZSEP ? 2 : 1);
        const int q = pr - (P::ZSEP && pr >= per_kind ? per_kind : 0);
        const int gi = q / (P::WT / TPI);
        const int f = TPI * (q % (P::WT / TPI)) + lane / (64 / TPI);
        const int t = min(w_t0 + f, wT - 1);
        poff[j] = ((uint32_t)t * (uint32_t)Gp + (uint32_t)gi) * 16u * P::PB + (uint32_t)(lane % (64 / TPI)) * 4u;
      } else if (FMT == kDqMx) {
        const int t = min(w_t0 + 8 * pr + (lane >> 3), wT - 1);
        poff[j] = (uint32_t)t * (uint32_t)KB * 64u + (uint32_t)(lane & 7) * 4u;
      } else {
        const int t = min(w_t0 + 4 * pr + (lane >> 4), wT - 1);
        poff[j] = (uint32_t)t * (uint32_t)KB * 128u + (uint32_t)(lane & 15) * 4u;
      }
    }
  }
  // activations of stage s into ring slot `slot`; `full`: all 64 columns are below K
  auto issue_x = [&](int s, int slot, auto full) {
    uint8_t* base = smem + slot * P::kStage;
    // activations: wave w copies rows RPW*w .. RPW*w + RPW-1 (8 rows of 8 chunks per instruction)
    if constexpr (decltype(full)::value) {
#pragma unroll
      for (int j = 0; j < kXI; ++j)
        __builtin_amdgcn_raw_ptr_buffer_load_lds(xr, (lds_void*)(base + (RPW * wave + 8 * j) * 128), 16, xoff[j], 128 * s, 0, 0);
    } else {  // possibly the partial last stage: columns at or beyond K copy zeros
#pragma unroll
      for (int j = 0; j < kXI; ++j) {
        const int r = RPW * wave + 8 * j + (lane >> 3);
        const uint32_t off = 64 * s + 8 * ((lane & 7) ^ (r & 7)) < K ? xoff[j] : kNone;
        __builtin_amdgcn_raw_ptr_buffer_load_lds(xr, (lds_void*)(base + (RPW * wave + 8 * j) * 128), 16, off, 128 * s, 0, 0);
      }
    }
  };
  // weights and parameters of stage s
  auto issue_w = [&](int s, int slot) {
    uint8_t* base = smem + slot * P::kStage;
    const uint32_t kb = (uint32_t)(P::B8 ? s : s >> 1), h = (uint32_t)(s & 1);
    uint8_t* wbase = base + P::kXBytes;
    if constexpr (FMT == kDqInt4 || P::B8) {
#pragma unroll
      for (int j = 0; j < P::TPW; ++j) {
        const int f = P::TPW * wave + j;
        const uint32_t so = (uint32_t)min(w_t0 + f, wT - 1) * wrow + kb * 1024u;
        if constexpr (P::B8) {  // the tile's whole 1 KiB block (16 rows x 64 columns)
          __builtin_amdgcn_raw_ptr_buffer_load_lds(wr, (lds_void*)(wbase + f * 1024), 16, wvo, so, 0, 0);
        } else {  // dwords 2h and 2h+1 of every lane's 16 bytes, 256 bytes per copy
          __builtin_amdgcn_raw_ptr_buffer_load_lds(wr, (lds_void*)(wbase + f * 512), 4, wvo, so + 8u * h, 0, 0);
          __builtin_amdgcn_raw_ptr_buffer_load_lds(wr, (lds_void*)(wbase + f * 512 + 256), 4, wvo, so + 8u * h + 4u, 0, 0);
        }
      }
    } else {  // bytes 512h .. 512h+511 of the tiles' blocks
      const uint32_t so = kb * 1024u + 512u * h;
      if constexpr (P::TPW == 2) {
        __builtin_amdgcn_raw_ptr_buffer_load_lds(wr, (lds_void*)(wbase + wave * 1024), 16, wvo, so, 0, 0);
      } else {
        __builtin_amdgcn_raw_ptr_buffer_load_lds(wr, (lds_void*)(wbase + wave * 512), 4, wvo, so, 0, 0);
        __builtin_amdgcn_raw_ptr_buffer_load_lds(wr, (lds_void*)(wbase + wave * 512 + 256), 4, wvo, so + 256u, 0, 0);
      }
    }
    if constexpr (!P::B8) {
      uint8_t* pbase = base + P::kXBytes + P::kWBytes;
#pragma unroll
      for (int j = 0; j < P::kPInstr; ++j) {
        const int pi = P::kPInstr * wave + j;
        const bool zsrc = FMT == kDqInt4 && P::ZSEP && pi >= np / 2;
        uint32_t so;
        if (FMT == kDqInt4) so = (uint32_t)((64 * s) / group) * 16u * P::PB;
        else if (FMT == kDqMx) so = kb * 64u + 32u * h;
        else so = kb * 128u + 64u * h;
        __builtin_amdgcn_raw_ptr_buffer_load_lds(zsrc ? zr : sr, (lds_void*)(pbase + pi * 256), 4, poff[j], so, 0, 0);
      }
    }
  };

  f32x4_t acc[MT][4];
#pragma unroll
  for (int i = 0; i < MT; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[i][j] = f32x4_t{0.f, 0.f, 0.f, 0.f};

  const int kg = KG == 2 ? wave / P::NWG : 0;  // k-group
  const int wg = wave % P::NWG;
  const int wm = wg / (P::NWG / 2), wn = wg % (P::NWG / 2);
  const int nl = lane & 15, jg = lane >> 4;
  // p0: the scale's fp32 bits, or for bf16 INT4 parameters bf16 scale | bf16 zero-point << 16;
  // p1: fp32 zero-points (asymmetric INT4 with fp32 parameters only)
  constexpr int kP0 = P::B8 ? 1 : 4;
  constexpr int kP1 = (FMT == kDqInt4 && ASYM && !PBF16) ? 4 : 1;
  constexpr int kWD = P::B8 ? 2 : 1;  // code dwords per column tile and MFMA step
  struct Raw {
    uint32_t wd[4 * kWD];  // weight codes of the 4 column tiles
    uint32_t p0[kP0], p1[kP1];
  };
  // weight codes and parameters of column tile nt, MFMA step q (32 columns) of the stage at `base`
  auto read_w = [&](const uint8_t* base, int q, int nt, Raw& o) {
    const uint8_t* wb = base + P::kXBytes;
    const uint8_t* pb = base + P::kXBytes + P::kWBytes;
    const int f = wn * 4 + nt;
    if (P::B8) {
      // columns 32q + 8jg .. +7 of row nl: half of lane (nl, 2q + jg / 2)'s 16 bytes
      const u32x2_t v = *reinterpret_cast<const u32x2_t*>(wb + f * 1024 + (16 * (2 * q + (jg >> 1)) + nl) * 16 + 8 * (jg & 1));
      o.wd[(nt * kWD) % (4 * kWD)] = v[0];
      o.wd[(nt * kWD + 1) % (4 * kWD)] = v[1];
    } else if (FMT == kDqInt4) {
      o.wd[nt] = *reinterpret_cast<const uint32_t*>(wb + f * 512 + q * 256 + lane * 4);
      const int gi = GROUP >= 64 ? 0 : q;
      constexpr int zoff = P::NGS * P::WT * 16 * P::PB;
      const int po = ((gi * P::WT + f) * 16 + nl) * P::PB;
      if (P::PAIR) {
        o.p0[nt % kP0] = *reinterpret_cast<const uint32_t*>(pb + po);  // bf16 scale | bf16 zero << 16
      } else if (PBF16) {
        o.p0[nt % kP0] = *reinterpret_cast<const uint16_t*>(pb + po);
      } else {
        o.p0[nt % kP0] = *reinterpret_cast<const uint32_t*>(pb + po);
        if (ASYM) o.p1[nt % kP1] = *reinterpret_cast<const uint32_t*>(pb + zoff + po);
      }
    } else {
      const int ll = 16 * q + nl;  // lane of the 128-column block within the stage's half
      o.wd[nt] = *reinterpret_cast<const uint32_t*>(wb + f * 512 + ll * 16 + jg * 4);
      if (FMT == kDqMx) {
        o.p0[nt % kP0] = pb[f * 32 + ll];
      } else {
        o.p0[nt % kP0] = pb[f * 64 + 2 * ll + (jg >> 1)];
      }
    }
  };
  auto read_x = [&](const uint8_t* base, int q, u32x4_t (&xo)[MT]) {  // activation operands of the wave's row tiles
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) {
      const int r = wm * (TMR / 2) + 16 * mt + nl;
      const int sl = (4 * q + jg) ^ (nl & 7);
      xo[mt] = *reinterpret_cast<const u32x4_t*>(base + r * 128 + sl * 16);
    }
  };
  // Decode of column tile nt's weight operand (8 consecutive k of row nl, in the activation dtype) in four
  // parts of one dword each, to be spread between MFMAs: a wave issues a VALU instruction about every
  // 5.6 cycles, 8.7 beside another wave's MFMAs (16 cycles each; both measured), so a tile decoded in one
  // go leaves the matrix unit idle. `t` carries what the parts of a tile share.
  struct Tmp {
    uint32_t d0, d1;
    float f[4];
    float sc, c;
  };
  auto decode_part = [&](const Raw& o, int nt, int part, Tmp& t, u32x4_t& out) {
    if constexpr (P::B8) {
      if (part == 0) {
        t.d0 = o.wd[(nt * kWD) % (4 * kWD)], t.d1 = o.wd[(nt * kWD + 1) % (4 * kWD)];
        if constexpr (FMT == kDqI8) t.d0 ^= 0x80808080u, t.d1 ^= 0x80808080u;  // stored q + 128 -> two's complement bytes
      }
      const uint32_t d = part < 2 ? t.d0 : t.d1;
      if constexpr (FMT == kDqF8) out[part] = (part & 1) ? A::template fp8_pair<true>(d) : A::template fp8_pair<false>(d);
      else out[part] = (part & 1) ? A::pack_exact(sbyte_f32<2>(d), sbyte_f32<3>(d)) : A::pack_exact(sbyte_f32<0>(d), sbyte_f32<1>(d));
    } else if constexpr (FMT == kDqMx) {
      if (part == 0) t.sc = __builtin_bit_cast(float, o.p0[nt % kP0] << 23);  // the E8M0 byte as 2**(e - 127)
      out[part] = A::fp4_pair_scaled(o.wd[nt], t.sc, part);
    } else if constexpr (FMT == kDqNv) {
      if (part == 0) t.sc = e4m3_value(o.p0[nt % kP0]);
      const f32x2_t f = A::fp4_pair_f32(o.wd[nt], part);
      out[part] = A::pack_exact(f[0] * t.sc, f[1] * t.sc);
    } else {
      // INT4: element e in nibble e/2 (even e) or 4 + e/2 (odd e). A code u = 0..15 read as an E4M3 byte is
      // u * 2**-9 (subnormal below 8, exponent 2**-6 from 8 on), so one scaled conversion gives two codes as
      // exact fp32; then fp32 (u - z) * s rounded to nearest even. Part order: dwords 0, 2, 1, 3.
      const uint32_t d = o.wd[nt];
      if (part == 0) {
        t.sc = PBF16 ? bf16_bits_to_f32((uint16_t)(o.p0[nt % kP0] & 0xffffu)) : __builtin_bit_cast(float, o.p0[nt % kP0]);
        if (!ASYM || PBF16) {
          // z * s is exact (z = 8, or z <= 15 and s has at most 8 significant bits), so the fma rounds
          // the exact (u - z) * s once
          const float zf = ASYM ? bf16_bits_to_f32((uint16_t)(o.p0[nt % kP0] >> 16)) : 8.0f;
          t.c = -zf * t.sc;
        } else {
          t.c = __builtin_bit_cast(float, o.p1[nt % kP1]);
        }
      }
      if ((part & 1) == 0) {
        const uint32_t v = (part == 0 ? d : d >> 4) & 0x0F0F0F0Fu;
        const f32x2_t lo = __builtin_amdgcn_cvt_scalef32_pk_f32_fp8(v, 512.0f, false);
        const f32x2_t hi = __builtin_amdgcn_cvt_scalef32_pk_f32_fp8(v, 512.0f, true);
        t.f[0] = lo[0], t.f[1] = hi[0], t.f[2] = lo[1], t.f[3] = hi[1];
      }
      const float u0 = t.f[2 * (part & 1)], u1 = t.f[2 * (part & 1) + 1];
      float w0, w1;
      if (!ASYM || PBF16) w0 = fmaf(u0, t.sc, t.c), w1 = fmaf(u1, t.sc, t.c);
      else w0 = (u0 - t.c) * t.sc, w1 = (u1 - t.c) * t.sc;
      out[(part >> 1) + 2 * (part & 1)] = A::pack_rne(w0, w1);
    }
  };

  // Pipeline: two wave groups in antiphase. Every SIMD holds one wave of each group (waves w and w + NW/2).
  // A step (SUB x 32 columns, index i, Q steps a stage) is a load phase (copies, LDS reads of step i's
  // activations and step i + 1's weights) and an MFMA phase (step i's MFMAs with step i + 1's decode between
  // them); a barrier ends each phase, and the second group runs one phase behind the first, so on every
  // SIMD one wave's MFMAs and decode cover the other's LDS reads. (With all waves in the same phase the
  // LDS reads and the MFMAs add up: 256 x 256 x 64 int8 took 1.50 us a stage on an otherwise idle chip
  // against 0.85 us of MFMAs.)
  //
  // Phase numbers: the first group loads in step i in phase 2i, the second in phase 2i + 1. Stage s's last
  // step is e = Q (s + 1) - 1; its last reads (activations) finish within load phase e, phase 2e + 1 at the
  // latest, so after that phase's barrier the slot is free: the copies of stage s + NS go into it at the
  // load phases e + 1 = Q (s + 1) and on. The first reads of stage s + 1 (weights) are the first group's
  // in phase 2e; every wave waits for its own copies of it in load phase e - 1, which ends with the
  // barrier of phase 2e - 1 at the latest.
  using Full = std::true_type;
  using Part = std::false_type;
  // 256 rows: 32 columns a step (the registers hold no more); 128 x 256: the whole stage, half the barriers for
  // the same MFMAs; 128 x 128: each k-group its 32 columns of the stage
  constexpr int SUB = KG == 1 && TMR == 128 ? 2 : 1;
  constexpr int Q = 2 / (KG * SUB);
  // copies that may stay in flight at that wait: the stages after s + 1; with two steps a stage, the weights of
  // stage s + NS - 1 are not yet issued then
  constexpr int kFlight = kPerStage * (NS - 3) + (Q == 2 ? kXI : 0);
  static_assert(NS >= 3, "ring too short");
  const int grp = __builtin_amdgcn_readfirstlane(wave / (NW / 2));
#pragma unroll
  for (int s = 0; s < NS - 1; ++s)
    if (s < S) issue_x(s0 + s, s, Part{}), issue_w(s0 + s, s);
  // stage 0 (and for Q = 1 stage 1, whose weights are read in step 0) has landed
  if (S >= NS - 1) wait_vmcnt<kPerStage * (Q == 2 ? NS - 2 : NS - 3)>();
  else wait_vmcnt<0>();
  __builtin_amdgcn_s_barrier();
  // stages of this split whose columns are all below K: 4-bit weights are padded to 128 columns, so at K % 128 of 1..63
  // the last two stages are not, and the next row's activations must not enter them (0 * Inf is NaN)
  const int Sf = min(S, K / 64 - s0);
  int s = 0, cur = 0;                            // cur: slot of stage s
  auto wrap = [](int v) { return v >= NS ? v - NS : v; };
  auto phase_end = [&]() {
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
  };
  Raw w[SUB];
  u32x4_t xo[SUB][MT], b0[SUB][4], b1[SUB][4];
  // one step: weights `b`, decoded before; reads and decodes those of the next step (slot nslot, its q nq)
  auto step = [&](auto steady, int q, const u32x4_t (&b)[SUB][4], u32x4_t (&bn)[SUB][4], int nslot, int nq, bool more) {
    // the copies of stage s + NS - 1, spread over the stage's load phases (a copy takes about 50 cycles to issue)
    const int cs = s0 + s + NS - 1, cslot = wrap(cur + NS - 1);
    if constexpr (decltype(steady)::value) {
      if (q == 0) issue_x(cs, cslot, Full{});
      if (q == Q - 1) issue_w(cs, cslot);
    } else if (s + NS - 1 < S) {
      if (q == 0) issue_x(cs, cslot, Part{});
      if (q == Q - 1) issue_w(cs, cslot);
    }
#pragma unroll
    for (int u = 0; u < SUB; ++u) read_x(smem + cur * P::kStage, KG == 2 ? kg : q + u, xo[u]);
    if (decltype(steady)::value || more) {
#pragma unroll
      for (int u = 0; u < SUB; ++u)
#pragma unroll
        for (int nt = 0; nt < 4; ++nt) read_w(smem + nslot * P::kStage, nq + u, nt, w[u]);
    }
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0): this wave's LDS reads are done
    if (Q == 1 || q == 0) {
      if constexpr (decltype(steady)::value) wait_vmcnt<kFlight>();
      else wait_vmcnt<0>();
    }
    phase_end();
    __builtin_amdgcn_s_setprio(1);
    Tmp t;
#pragma unroll
    for (int u = 0; u < SUB; ++u)
#pragma unroll
      for (int nt = 0; nt < 4; ++nt)
#pragma unroll
        for (int p = 0; p < 4; ++p) {
#pragma unroll
          for (int mt = p * MT / 4; mt < (p + 1) * MT / 4; ++mt) acc[mt][nt] = A::mfma(b[u][nt], xo[u][mt], acc[mt][nt]);
          decode_part(w[u], nt, p, t, bn[u][nt]);  // (after the last step: of stale codes, unused)
          __builtin_amdgcn_sched_barrier(0);
        }
    __builtin_amdgcn_s_setprio(0);
    phase_end();
  };
  auto advance = [&]() { cur = wrap(cur + 1), ++s; };
  {
    Tmp t;
#pragma unroll
    for (int u = 0; u < SUB; ++u) {
#pragma unroll
      for (int nt = 0; nt < 4; ++nt) read_w(smem, (KG == 2 ? kg : 0) + u, nt, w[u]);
#pragma unroll
      for (int nt = 0; nt < 4; ++nt)
#pragma unroll
        for (int p = 0; p < 4; ++p) decode_part(w[u], nt, p, t, b0[u][nt]);
    }
  }
  if (grp == 1) phase_end();
  if constexpr (Q == 2) {
    while (s + NS - 1 < Sf) {
      step(Full{}, 0, b0, b1, cur, 1, true);
      step(Full{}, 1, b1, b0, wrap(cur + 1), 0, true);
      advance();
    }
    while (s < S) {
      step(Part{}, 0, b0, b1, cur, 1, true);
      step(Part{}, 1, b1, b0, wrap(cur + 1), 0, s + 1 < S);
      advance();
    }
  } else {
    while (s + NS < Sf) {
      step(Full{}, 0, b0, b1, wrap(cur + 1), kg, true);
      advance();
      step(Full{}, 0, b1, b0, wrap(cur + 1), kg, true);
      advance();
    }
    while (s < S) {
      step(Part{}, 0, b0, b1, wrap(cur + 1), kg, s + 1 < S);
      advance();
#pragma unroll
      for (int u = 0; u < SUB; ++u)
#pragma unroll
        for (int nt = 0; nt < 4; ++nt) b0[u][nt] = b1[u][nt];
    }
  }
  if (grp == 0) phase_end();

  // epilogue: acc[mt][nt][i] is y[m0 + 16mt + (l & 15)][n0 + 16nt + 4(l >> 4) + i]
  // KG = 2: the wave of k-group g keeps row tiles g MT/2 .. +MT/2 and takes its partner's sums of them
  // (first group's + second group's), so both waves finish half of the 64 columns' rows.
  constexpr int ME = MT / KG;  // row tiles this wave finishes
  if constexpr (KG == 2) {
    f32x4_t* red = reinterpret_cast<f32x4_t*>(smem);  // [wave][ME * 4][64]
    __syncthreads();  // every wave is done reading the stages
#pragma unroll
    for (int i = 0; i < ME; ++i)
#pragma unroll
      for (int nt = 0; nt < 4; ++nt)
        red[((wave * ME + i) * 4 + nt) * 64 + lane] = kg == 0 ? acc[ME + i][nt] : acc[i][nt];
    __syncthreads();
    const int other = wave ^ P::NWG;
#pragma unroll
    for (int i = 0; i < ME; ++i)
#pragma unroll
      for (int nt = 0; nt < 4; ++nt) {
        const f32x4_t p = red[((other * ME + i) * 4 + nt) * 64 + lane];
        const f32x4_t own = kg == 0 ? acc[i][nt] : acc[ME + i][nt];
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[i][nt][j] = own[j] + p[j];
      }
  }
  const int m0 = tm * TMR + wm * (TMR / 2) + kg * 16 * ME;
  const int n0 = tn * TNC + wn * 64;
  if (splits > 1) {
    // raw fp32 partial sums of this split; dq_reduce_kernel adds the splits in order
    float* part = ws + (int64_t)split * m * n;
#pragma unroll
    for (int nt = 0; nt < 4; ++nt) {
      const int col = n0 + 16 * nt + 4 * jg;
      if (col >= n) continue;
#pragma unroll
      for (int mt = 0; mt < ME; ++mt) {
        const int row = m0 + 16 * mt + nl;
        if (row >= m) continue;
        float* dst = part + (int64_t)row * n + col;
        if ((n & 3) == 0) {
          *reinterpret_cast<f32x4_t*>(dst) = acc[mt][nt];
        } else {
#pragma unroll
          for (int j = 0; j < 4; ++j)
            if (col + j < n) dst[j] = acc[mt][nt][j];
        }
      }
    }
    return;
  }
  const float gs = FMT == kDqNv ? *s_global : 1.0f;
  // per-row factor of row m0 + 16mt + nl (FP8's per-token scale)
  float rsv[FMT == kDqF8 ? ME : 1];
  if (FMT == kDqF8) {
#pragma unroll
    for (int mt = 0; mt < ME; ++mt) rsv[mt % (FMT == kDqF8 ? ME : 1)] = rs[min(m0 + 16 * mt + nl, m - 1)];
  }
  // the finished fp32 value of accumulator j of tile (mt, nt), before the bias
  auto finish = [&](int mt, int nt, int j, float csv) -> float {
    const float v = acc[mt][nt][j];
    if (FMT == kDqF8) return v * rsv[mt % (FMT == kDqF8 ? ME : 1)] * csv;
    return v * (FMT == kDqI8 ? csv : gs);
  };
  auto col_params = [&](int col, float (&csv)[4], float (&badd)[4]) {
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int c = min(col + j, n - 1);
      csv[j] = P::B8 ? s_global[c] : 1.0f;
      badd[j] = bias ? (YKIND == 1 ? f16_bits_to_f32(bias[c]) : bf16_bits_to_f32(bias[c])) : 0.0f;
    }
  };
  if (YKIND != 2) {
    // 16-bit y: each wave converts its tile into its own LDS area, then stores whole rows of 64 columns:
    // 16 bytes a lane when every row start is 16-byte aligned (vec16), else one element a lane
    __syncthreads();  // every wave is done reading the stages (or its partner's sums)
    uint8_t* ep = smem + wave * (16 * ME) * dqg::kEpiPitch;
#pragma unroll
    for (int nt = 0; nt < 4; ++nt) {
      const int cl = 16 * nt + 4 * jg;
      float csv[4], badd[4];
      col_params(n0 + cl, csv, badd);
#pragma unroll
      for (int mt = 0; mt < ME; ++mt) {
        const int rl = 16 * mt + nl;
        float v[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) v[j] = finish(mt, nt, j, csv[j]) + badd[j];
        const uint32_t lo = YKIND == 0 ? ActBF16::pack_rne(v[0], v[1]) : ActF16::pack_rne(v[0], v[1]);
        const uint32_t hi = YKIND == 0 ? ActBF16::pack_rne(v[2], v[3]) : ActF16::pack_rne(v[2], v[3]);
        *reinterpret_cast<u32x2_t*>(ep + rl * dqg::kEpiPitch + cl * 2) = u32x2_t{lo, hi};
      }
    }
    // Each wave reads back only what it wrote (LDS accesses of one wave execute in order).
    __builtin_amdgcn_wave_barrier();
    if (vec16) {
      const int cc = (lane & 7) * 8;
#pragma unroll 4
      for (int p = 0; p < 2 * ME; ++p) {
        const int rl = 8 * p + (lane >> 3);
        const int row = m0 + rl, col = n0 + cc;
        const u32x4_t v = *reinterpret_cast<const u32x4_t*>(ep + rl * dqg::kEpiPitch + cc * 2);
        if (row >= m || col >= n) continue;
        uint16_t* dst = static_cast<uint16_t*>(y) + (int64_t)row * n + col;
        __builtin_nontemporal_store(v, reinterpret_cast<u32x4_t*>(dst));
      }
    } else {
      const int col = n0 + lane;
      const int rows = min(16 * ME, m - m0);
      if (col < n) {
        uint16_t* dst = static_cast<uint16_t*>(y) + (int64_t)m0 * n + col;
#pragma unroll 4
        for (int rl = 0; rl < rows; ++rl)
          dst[(int64_t)rl * n] = *reinterpret_cast<const uint16_t*>(ep + rl * dqg::kEpiPitch + lane * 2);
      }
    }
    return;
  }
#pragma unroll
  for (int nt = 0; nt < 4; ++nt) {
    const int col = n0 + 16 * nt + 4 * jg;
    if (col >= n) continue;
    float csv[4], badd[4];
    col_params(col, csv, badd);
#pragma unroll
    for (int mt = 0; mt < ME; ++mt) {
      const int row = m0 + 16 * mt + nl;
      if (row >= m) continue;
      float* dst = static_cast<float*>(y) + (int64_t)row * n + col;
      f32x4_t v;
#pragma unroll
      for (int j = 0; j < 4; ++j) v[j] = finish(mt, nt, j, csv[j]);
      if (vec16) {
        *reinterpret_cast<f32x4_t*>(dst) = v;
      } else {
#pragma unroll
        for (int j = 0; j < 4; ++j)
          if (col + j < n) dst[j] = v[j];
      }
    }
  }
}

// y[i] = (sum over splits, in order, of the fp32 partials) * scale (+ bias[i % n]), rounded to y's dtype. The
// scale is s_global (NVFP4), cs[n] (int8: rs null) or rs[m] * cs[n] (FP8). Four outputs per thread where the
// rows keep 16-byte alignment (n % 4 == 0: a quad never straddles two rows).
template <int YKIND>
__global__ __launch_bounds__(256) void dq_reduce_kernel(const float* __restrict__ ws, int splits, int64_t mn, int n,
                                                        const float* __restrict__ s_global,
                                                        const float* __restrict__ rs, const float* __restrict__ cs,
                                                        const uint16_t* __restrict__ bias, void* __restrict__ y,
                                                        int vec) {
  const int64_t i = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) * (vec ? 4 : 1);
  if (i >= mn) return;
  const int cnt = vec ? 4 : 1;
  float v[4] = {0.0f, 0.0f, 0.0f, 0.0f};
  if (vec) {
#pragma unroll 4
    for (int s = 0; s < splits; ++s) {
      const f32x4_t p = *reinterpret_cast<const f32x4_t*>(ws + (int64_t)s * mn + i);
#pragma unroll
      for (int j = 0; j < 4; ++j) v[j] += p[j];
    }
  } else {
    for (int s = 0; s < splits; ++s) v[0] += ws[(int64_t)s * mn + i];
  }
  const uint32_t row = (uint32_t)(i / n);
  const int c0 = (int)(i - (int64_t)row * n);
  const float gs = s_global ? *s_global : 1.0f;
  const float r = rs ? rs[row] : 1.0f;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    if (j >= cnt) break;
    if (s_global) v[j] *= gs;
    if (rs) v[j] *= r;
    if (cs) v[j] *= cs[c0 + j];
    if (bias) v[j] += YKIND == 1 ? f16_bits_to_f32(bias[c0 + j]) : bf16_bits_to_f32(bias[c0 + j]);
  }
  if (YKIND == 2) {
    float* dst = static_cast<float*>(y) + i;
    if (vec) *reinterpret_cast<f32x4_t*>(dst) = f32x4_t{v[0], v[1], v[2], v[3]};
    else *dst = v[0];
  } else {
    uint16_t* dst = static_cast<uint16_t*>(y) + i;
    if (vec) {
      const uint32_t lo = YKIND == 0 ? ActBF16::pack_rne(v[0], v[1]) : ActF16::pack_rne(v[0], v[1]);
      const uint32_t hi = YKIND == 0 ? ActBF16::pack_rne(v[2], v[3]) : ActF16::pack_rne(v[2], v[3]);
      *reinterpret_cast<u32x2_t*>(dst) = u32x2_t{lo, hi};
    } else {
      *dst = YKIND == 0 ? f32_to_bf16_bits(v[0]) : f32_to_f16_bits(v[0]);
    }
  }
}

// Output tile and K splits of a launch: splits > 1 leave fp32 partials [splits][m][n] in a workspace.
struct DqPlan {
  int tm, tn, splits;
};
// The plan for an m-row product with `stages` 64-column k-stages (sqx_gemm.hip).
DqPlan dq_plan(int64_t m, int64_t rows, int64_t stages, int fmt);
inline int64_t dq_workspace_bytes(const DqPlan& p, int64_t m, int64_t rows) {
  return p.splits > 1 ? (int64_t)p.splits * m * rows * 4 : 0;
}

// Launch the dequant GEMM. scale: NVFP4's global scale (one value) or the 8-bit formats' per-row scales [n];
// rs: FP8's per-token scales [m]. Without a workspace large enough for the plan's splits: one pass per tile.
template <class A, int FMT, bool ASYM, bool PBF16, int GROUP, int YK>
hipError_t launch_dq(const uint16_t* x, const uint8_t* wt, const void* st, const void* zt, const float* scale,
                     const float* rs, void* y, const uint16_t* bias, int m, int n, int K, int KB, float* ws,
                     int64_t ws_bytes, hipStream_t s) {
  constexpr bool B8 = FMT == kDqI8 || FMT == kDqF8;
  const DqPlan plan = dq_plan(m, n, B8 ? KB : 2 * KB, FMT);
  const int tiles_m = (m + plan.tm - 1) / plan.tm, tiles_n = (n + plan.tn - 1) / plan.tn;
  int splits = plan.splits;
  if (splits > 1 && (ws == nullptr || ws_bytes < (int64_t)splits * m * n * 4 || reinterpret_cast<uintptr_t>(ws) % 16))
    splits = 1;
  const int vec16 = YK == 2 ? (n % 4 == 0) && (reinterpret_cast<uintptr_t>(y) % 16 == 0)
                            : (n % 8 == 0) && (reinterpret_cast<uintptr_t>(y) % 16 == 0);
  auto go = [&](auto kern, int lds, int threads) -> hipError_t {
    const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kern),
                                             hipFuncAttributeMaxDynamicSharedMemorySize, lds);
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(kern, dim3((unsigned)(tiles_m * tiles_n * splits)), dim3((unsigned)threads), (size_t)lds, s, x, wt,
                       st, zt, scale, rs, y, bias, m, n, K, KB, tiles_m, tiles_n, vec16, splits, ws);
    return hipSuccess;
  };
  hipError_t e;
#define SQX_DQ_TILE(TM_, TN_, KG_, NS_)                                      \
  e = go(dq_gemm_kernel<A, FMT, ASYM, PBF16, GROUP, YK, TM_, TN_, KG_, NS_>, \
         DqW<FMT, ASYM, PBF16, GROUP, TM_, TN_, KG_, NS_>::kLds, 2 * TN_ * KG_)
  if (plan.tm == 256) SQX_DQ_TILE(256, 256, 1, 3);
  else if (plan.tn == 256) SQX_DQ_TILE(128, 256, 1, 5);
  else SQX_DQ_TILE(128, 128, 2, 6);
#undef SQX_DQ_TILE
  if (e != hipSuccess) return e;
  if (splits > 1) {
    const int64_t mn = (int64_t)m * n;
    const int vec = n % 4 == 0 && reinterpret_cast<uintptr_t>(y) % (YK == 2 ? 16 : 8) == 0;
    hipLaunchKernelGGL(dq_reduce_kernel<YK>, dim3((unsigned)ceil_div(mn, vec ? 1024 : 256)), dim3(256), 0, s, ws, splits,
                       mn, n, FMT == kDqNv ? scale : nullptr, FMT == kDqF8 ? rs : nullptr, B8 ? scale : nullptr, bias, y,
                       vec);
  }
  return hipGetLastError();
}

}  // namespace sqx
