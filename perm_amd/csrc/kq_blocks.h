// Block-level bodies of the k-quant encoder and decoder (bit-exact with
// coldpress/kquant.py), shared by the single-tensor kernels of kq_codec.hip and
// the many-tensor kernels of the EF driver.
//
// Encoder mapping: one lane per sub-block. A wave64 holds S = 64/G superblocks
// (G = 16 lanes per superblock for the 16-wide sub-blocks, 8 for the 32-wide
// ones of Q4_K and Q5_K). Sub-block fits run in-lane on registers; superblock-level
// steps (maxima, super-scale fits, the 256-wide sum of squares) run across the
// G lanes of the superblock with xor-butterfly reductions that reproduce
// numpy's pairwise order. What leaves (KqOut) is the container bytes, the scale fields
// alone (the EF commits, whose code bytes the repack writes), or the decoded weights
// (the PERM objective, which needs no bytes).
#pragma once
#include <hip/hip_runtime.h>

#include "cp_device.h"
#include "cp_host.h"
#include "kq_fit.h"

namespace cp {

constexpr int kWavesPerBlock = 4;

template <int TT>
struct Kq;
template <>
struct Kq<CP_Q2_K> {
  static constexpr int G = 16, SUBW = 16, BP = 84;
};
template <>
struct Kq<CP_Q3_K> {
  static constexpr int G = 16, SUBW = 16, BP = 110;
};
template <>
struct Kq<CP_Q4_K> {
  static constexpr int G = 8, SUBW = 32, BP = 144;
};
template <>
struct Kq<CP_Q5_K> {
  static constexpr int G = 8, SUBW = 32, BP = 176;
};
template <>
struct Kq<CP_Q6_K> {
  static constexpr int G = 16, SUBW = 16, BP = 210;
};

// Per-superblock fields staged in LDS before packing.
//  Q2_K: a[k] = scale byte (sc & 0xF) | (min & 0xF) << 4
//  Q3_K: a[k] = 6-bit scale 0..63
//  Q4_K, Q5_K: a[0..7] = 6-bit scales, a[8..15] = 6-bit mins
//  Q6_K: a[k] = int8 scale
struct alignas(4) SbFields {
  uint8_t a[16];
  uint16_t d, dmin;
};

// What an encode leaves in memory.
enum class KqOut { kBytes, kFields, kRecon };

// numpy's pairwise sum of a superblock's 256 values staged in LDS, computed by
// the G lanes of the superblock: split 128 + 128, each half with 8 sequential
// accumulators over stride 8, then the 8-way tree (kquant.py:381, :453, :537).
template <int G>
__device__ __forceinline__ float sum256_lds(const float* a, int g) {
  if constexpr (G == 16) {
    const float* p = a + (g >> 3) * 128 + (g & 7);
    float r = p[0];
#pragma unroll
    for (int m = 1; m < 16; ++m) r = r + p[8 * m];
    r = tree8(r);
    return 0.0f + (r + dpp<kDppRor8>(r));
  } else {
    float r0 = a[g], r1 = a[128 + g];
#pragma unroll
    for (int m = 1; m < 16; ++m) {
      r0 = r0 + a[g + 8 * m];
      r1 = r1 + a[128 + g + 8 * m];
    }
    return 0.0f + (tree8(r0) + tree8(r1));
  }
}

// Items 0 .. C - 1 of each of a wave's S superblocks, handed to its lanes: f(superblock, item).
template <int S, int C, class F>
__device__ __forceinline__ void wave_items(int lane, const F& f) {
  static_assert((C & (C - 1)) == 0, "power of two per superblock");
#pragma unroll
  for (int i0 = 0; i0 < S * C; i0 += 64) {
    const int i = i0 + lane;
    if (S * C - i0 >= 64 || i < S * C) f(i / C, i % C);
  }
}

// The packed superblocks of a wave (ggml block layouts; kquant.py:407-413, :474-485,
// :565-571, :664-677): its S superblocks of BP bytes at dst, four bytes per item from four
// codes at a time (the codes of a superblock are consecutive LDS bytes, so one LDS word holds
// the codes of four output bytes). Packed byte by byte, each byte chosen among the fields by
// its offset, this was a fifth of the Q6_K encode's instructions (divergent branches and one
// LDS byte read per code). Superblocks from nvalid on are left out. CODES false: the scale
// fields alone.
template <int TT, bool CODES>
__device__ __forceinline__ void pack_wave(const uint8_t* codes, const SbFields* f, int lane,
                                          int nvalid, uint8_t* dst) {
  constexpr int S = 64 / Kq<TT>::G, BP = Kq<TT>::BP;
  constexpr uint32_t M1 = 0x01010101u, M3 = 0x03030303u, MF = 0x0F0F0F0Fu;
  const auto c = [&](int s, int k) { return *reinterpret_cast<const uint32_t*>(codes + s * 256 + k); };
  const auto a = [&](int s, int w) { return *reinterpret_cast<const uint32_t*>(f[s].a + 4 * w); };
  const auto put = [&](int s, int off, uint32_t v) {  // four bytes at a 2- or 4-byte boundary
    if (s >= nvalid) return;
    uint8_t* p = dst + s * BP + off;
    if constexpr (BP % 4 == 0) {
      *reinterpret_cast<uint32_t*>(p) = v;
    } else {
      reinterpret_cast<uint16_t*>(p)[0] = (uint16_t)v;
      reinterpret_cast<uint16_t*>(p)[1] = (uint16_t)(v >> 16);
    }
  };
  const auto put_d = [&](int off) {  // the lone fp16 d of the types without mins
    if (lane < S && lane < nvalid) *reinterpret_cast<uint16_t*>(dst + lane * BP + off) = f[lane].d;
  };
  if constexpr (TT == CP_Q2_K) {
    if constexpr (CODES)
      wave_items<S, 16>(lane, [&](int s, int j) {
        const int k = (j >> 3) * 128 + 4 * (j & 7);
        put(s, 16 + 4 * j, c(s, k) | c(s, k + 32) << 2 | c(s, k + 64) << 4 | c(s, k + 96) << 6);
      });
    wave_items<S, 4>(lane, [&](int s, int j) { put(s, 4 * j, a(s, j)); });
    wave_items<S, 1>(lane, [&](int s, int) { put(s, 80, (uint32_t)f[s].d | (uint32_t)f[s].dmin << 16); });
  } else if constexpr (TT == CP_Q3_K) {
    if constexpr (CODES) {
      wave_items<S, 8>(lane, [&](int s, int j) {
        uint32_t v = 0;
#pragma unroll
        for (int q = 0; q < 8; ++q) v |= ((c(s, 32 * q + 4 * j) >> 2) & M1) << q;
        put(s, 4 * j, v);
      });
      wave_items<S, 16>(lane, [&](int s, int j) {
        const int k = (j >> 3) * 128 + 4 * (j & 7);
        put(s, 32 + 4 * j, (c(s, k) & M3) | (c(s, k + 32) & M3) << 2 | (c(s, k + 64) & M3) << 4 |
                               (c(s, k + 96) & M3) << 6);
      });
    }
    wave_items<S, 4>(lane, [&](int s, int j) {
      const uint32_t w0 = a(s, 0), w1 = a(s, 1), w2 = a(s, 2), w3 = a(s, 3);
      if (j == 0) put(s, 96, (w0 & MF) | (w2 & MF) << 4);
      if (j == 1) put(s, 100, (w1 & MF) | (w3 & MF) << 4);
      if (j == 2)
        put(s, 104, ((w0 >> 4) & M3) | ((w1 >> 4) & M3) << 2 | ((w2 >> 4) & M3) << 4 | ((w3 >> 4) & M3) << 6);
    });
    put_d(108);
  } else if constexpr (TT == CP_Q4_K || TT == CP_Q5_K) {
    constexpr int body = TT == CP_Q5_K ? 48 : 16;
    if constexpr (CODES) {
      if constexpr (TT == CP_Q5_K)  // qh: bit q of byte j is code (32q + j) >= 16
        wave_items<S, 8>(lane, [&](int s, int j) {
          uint32_t v = 0;
#pragma unroll
          for (int q = 0; q < 8; ++q) v |= ((c(s, 32 * q + 4 * j) >> 4) & M1) << q;
          put(s, 16 + 4 * j, v);
        });
      wave_items<S, 32>(lane, [&](int s, int j) {
        const int k = (j >> 3) * 64 + 4 * (j & 7);
        put(s, body + 4 * j, (c(s, k) & MF) | (c(s, k + 32) & MF) << 4);
      });
    }
    wave_items<S, 4>(lane, [&](int s, int j) {
      const uint32_t s0 = a(s, 0), s1 = a(s, 1), m0 = a(s, 2), m1 = a(s, 3);
      put(s, 4 * j, j == 0   ? (uint32_t)f[s].d | (uint32_t)f[s].dmin << 16
                    : j == 1 ? s0 | ((s1 >> 4) & M3) << 6
                    : j == 2 ? m0 | ((m1 >> 4) & M3) << 6
                             : (s1 & MF) | (m1 & MF) << 4);
    });
  } else {  // Q6_K
    if constexpr (CODES) {
      wave_items<S, 32>(lane, [&](int s, int j) {
        const int k = (j >> 4) * 128 + 4 * (j & 15);
        put(s, 4 * j, (c(s, k) & MF) | (c(s, k + 64) & MF) << 4);
      });
      wave_items<S, 16>(lane, [&](int s, int j) {
        const int k = (j >> 3) * 128 + 4 * (j & 7);
        put(s, 128 + 4 * j, ((c(s, k) >> 4) & M3) | ((c(s, k + 32) >> 4) & M3) << 2 |
                                ((c(s, k + 64) >> 4) & M3) << 4 | ((c(s, k + 96) >> 4) & M3) << 6);
      });
    }
    wave_items<S, 4>(lane, [&](int s, int j) { put(s, 192 + 4 * j, a(s, j)); });
    put_d(208);
  }
}

// LDS writes of this wave's lanes before its later LDS reads (the LDS serves one wave's
// accesses in order; this keeps the compiler from moving them).
__device__ __forceinline__ void wave_lds_fence() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Encode the superblocks of block ``blk`` (kWavesPerBlock waves of S
// superblocks each) of one [NB superblocks] tensor; nsb superblocks per row.
// OUT: kBytes and kFields write container bytes to ``out``; kRecon writes the decoded
// float32 weights to ``recon`` and no bytes.
template <int TT, bool IMAT, KqOut OUT = KqOut::kBytes>
__device__ __forceinline__ void kq_encode_block(const float* __restrict__ x,
                                                const float* __restrict__ qw, int64_t NB,
                                                int64_t nsb, uint8_t* __restrict__ out,
                                                int64_t blk, float* __restrict__ recon = nullptr) {
  constexpr int G = Kq<TT>::G, SUBW = Kq<TT>::SUBW, BP = Kq<TT>::BP, S = 64 / G;
  // one buffer per wave: the squares of the weighted path, then the packed bytes or the
  // decoded weights on their way out
  constexpr bool kSquares = IMAT && TT != CP_Q6_K;
  constexpr int kOutBytes = OUT == KqOut::kBytes ? (S * BP + 15) / 16 * 16
                            : OUT == KqOut::kRecon ? S * 256 * 4 : 16;
  constexpr int kBufBytes = kSquares && S * 256 * 4 > kOutBytes ? S * 256 * 4 : kOutBytes;
  __shared__ __align__(16) uint8_t s_buf[kWavesPerBlock][kBufBytes];
  __shared__ __align__(16) uint8_t s_codes[OUT == KqOut::kBytes ? kWavesPerBlock : 1]
                                          [OUT == KqOut::kBytes ? S * 256 : 16];
  __shared__ SbFields s_f[kWavesPerBlock][S];
  // the make_qp_quants problems of the weighted affine types: two per superblock
  constexpr bool kQp = IMAT && (TT == CP_Q2_K || TT == CP_Q4_K || TT == CP_Q5_K);
  __shared__ QpStage<G, kQp ? 2 * kWavesPerBlock * S : 2> s_qp;

  const int wv = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int g = lane % G, sl = lane / G;
  const int64_t sb0 = (blk * kWavesPerBlock + wv) * S;
  const int64_t sb = sb0 + sl;
  const bool valid = sb < NB;
  const int64_t sbr = valid ? sb : 0;  // tail lanes compute on superblock 0, write nothing

  float xv[SUBW];
  {
    const float4* p = reinterpret_cast<const float4*>(x + sbr * 256 + g * SUBW);
#pragma unroll
    for (int i = 0; i < SUBW / 4; ++i) {
      float4 v = p[i];
      xv[4 * i] = v.x;
      xv[4 * i + 1] = v.y;
      xv[4 * i + 2] = v.z;
      xv[4 * i + 3] = v.w;
    }
  }

  // importance weights qw * sqrt(k*sum(x^2)/256 + x^2)  (kquant.py:380-383, :453-455, :537-539)
  float wt[SUBW];
  if constexpr (kSquares) {
    float* sq = reinterpret_cast<float*>(s_buf[wv]) + sl * 256;
#pragma unroll
    for (int i = 0; i < SUBW; ++i) sq[g * SUBW + i] = xv[i] * xv[i];
    __syncthreads();
    float sx2 = sum256_lds<G>(sq, g);
    float var = (TT == CP_Q2_K ? sx2 : 2.0f * sx2) / 256.0f;
    const float4* q = reinterpret_cast<const float4*>(qw + (sbr % nsb) * 256 + g * SUBW);
#pragma unroll
    for (int i = 0; i < SUBW / 4; ++i) {
      float4 v = q[i];
      wt[4 * i] = v.x * sqrtf(var + xv[4 * i] * xv[4 * i]);
      wt[4 * i + 1] = v.y * sqrtf(var + xv[4 * i + 1] * xv[4 * i + 1]);
      wt[4 * i + 2] = v.z * sqrtf(var + xv[4 * i + 2] * xv[4 * i + 2]);
      wt[4 * i + 3] = v.w * sqrtf(var + xv[4 * i + 3] * xv[4 * i + 3]);
    }
  } else if constexpr (IMAT) {  // Q6_K: the importance vector is the weight itself
    const float4* q = reinterpret_cast<const float4*>(qw + (sbr % nsb) * 256 + g * SUBW);
#pragma unroll
    for (int i = 0; i < SUBW / 4; ++i) {
      float4 v = q[i];
      wt[4 * i] = v.x;
      wt[4 * i + 1] = v.y;
      wt[4 * i + 2] = v.z;
      wt[4 * i + 3] = v.w;
    }
  }

  int L[SUBW];
  float rdl = 0.0f, rml = 0.0f;  // the decoders' sub-block step and offset (kRecon)
  SbFields& F = s_f[wv][sl];

  if constexpr (TT == CP_Q2_K) {
    float scale, mn;
    int sc_i, mn_i;
    float d, dmin;
    AffineFit fit;
    if constexpr (IMAT) {
      fit = fit_affine<16>(xv, wt, kQkxQ2Imat, false, true);
      float sw = psum<16>(wt);
      gfit_nonneg_pair<16>(fit.scale, fit.min, sw, 15, g, wv * S + sl, s_qp, &d, &sc_i, &dmin, &mn_i);
    } else {
#pragma unroll
      for (int i = 0; i < 16; ++i) wt[i] = fabsf(xv[i]);
      fit = fit_affine<16>(xv, wt, kQkxQ2Ref, true, false);
      scale = fit.scale;
      mn = fit.min;
      float smax = gmax<16>(scale), mmax = gmax<16>(mn);
      bool ps = smax > 0.0f, pm = mmax > 0.0f;
      float is = ps ? 15.0f / smax : 0.0f, im = pm ? 15.0f / mmax : 0.0f;
      sc_i = ps ? rint_magic(is * scale) : 0;
      mn_i = pm ? rint_magic(im * mn) : 0;
      d = ps ? smax / 15.0f : 0.0f;
      dmin = pm ? mmax / 15.0f : 0.0f;
    }
    uint16_t d16 = half_bits(d), m16 = half_bits(dmin);
    float dl = half_value(d16) * (float)sc_i, ml = half_value(m16) * (float)mn_i;
    if constexpr (OUT != KqOut::kFields) {
      if (dl != 0.0f) {
#pragma unroll
        for (int i = 0; i < 16; ++i) L[i] = clampi(rint_magic((xv[i] + ml) / dl), 0, 3);
      } else {
        affine_final_codes<16>(xv, fit, 3, L);  // the search's codes stay where dl == 0
      }
    }
    if constexpr (OUT == KqOut::kRecon) {
      rdl = half_value(d16) * (float)(sc_i & 0xF);
      rml = half_value(m16) * (float)(mn_i & 0xF);
    }
    F.a[g] = (uint8_t)((sc_i & 0xF) | (mn_i & 0xF) << 4);
    if (g == 0) {
      F.d = d16;
      F.dmin = m16;
    }
  } else if constexpr (TT == CP_Q3_K) {
    int Ls;
    float d;
    SignedFit fit;
    if constexpr (IMAT) {
      fit = fit_signed<16>(xv, wt, kQxQ3);
      float sw = psum<16>(wt);
      d = gfit_signed<16>(fit.scale, sw, 32, g, &Ls);
    } else {
      float scale = fit_signed_descent16(xv, 4, L);
      float amax;
      float smax = gfirst_absmax<16>(scale, g, &amax);
      bool nz = smax != 0.0f;
      float is = nz ? -32.0f / smax : 0.0f;
      Ls = nz ? clampi(rint_magic(is * scale), -32, 31) + 32 : 0;
      d = nz ? 1.0f / is : 0.0f;
      d = (nz && isfinite(d)) ? d : 0.0f;
    }
    uint16_t d16 = half_bits(d);
    float dsub = half_value(d16) * (float)(Ls - 32);
    if constexpr (OUT != KqOut::kFields) {
      if constexpr (IMAT) {
        if (dsub != 0.0f)
          signed_requant<16>(xv, fit, dsub, 4, L);
        else
          signed_final_codes<16>(xv, fit, 4, L);  // the search's codes stay where dsub == 0
      } else if (dsub != 0.0f) {
#pragma unroll
        for (int i = 0; i < 16; ++i) L[i] = clampi(rint_magic(xv[i] / dsub), -4, 3) + 4;
      }
    }
    if constexpr (OUT == KqOut::kRecon) rdl = half_value(d16) * (float)((Ls & 63) - 32);
    F.a[g] = (uint8_t)Ls;
    if (g == 0) F.d = d16;
  } else if constexpr (TT == CP_Q4_K || TT == CP_Q5_K) {
    // Q5_K is Q4_K with 32 levels and its own reference-path search (kquant.py:508-593)
    constexpr int TOP = TT == CP_Q5_K ? 31 : 15;
    float scale, mn, d, dmin;
    int Ls, Lm;
    AffineFit fit;
    if constexpr (IMAT) {
      if constexpr (TT == CP_Q5_K)
        fit = fit_affine<32>(xv, wt, kQkxQ5Imat, false, true);
      else
        fit = fit_affine<32>(xv, wt, kQkxQ4Imat, false, true);
      float sw = psum<32>(wt);
      gfit_nonneg_pair<8>(fit.scale, fit.min, sw, 63, g, wv * S + sl, s_qp, &d, &Ls, &dmin, &Lm);
      if constexpr (TT == CP_Q5_K) {
        Ls = Ls < 63 ? Ls : 63;
        Lm = Lm < 63 ? Lm : 63;
      }
    } else {
      float sq[32];
#pragma unroll
      for (int i = 0; i < 32; ++i) sq[i] = xv[i] * xv[i];
      float av = sqrtf(psum<32>(sq) / 32.0f);
#pragma unroll
      for (int i = 0; i < 32; ++i) wt[i] = av + fabsf(xv[i]);
      if constexpr (TT == CP_Q5_K)
        fit = fit_affine<32>(xv, wt, kQkxQ5Ref, false, false);
      else
        fit = fit_affine<32>(xv, wt, kQkxQ4Ref, false, false);
      scale = fit.scale;
      mn = fit.min;
      float smax = gmax<8>(scale), mmax = gmax<8>(mn);
      float is = smax > 0.0f ? 63.0f / smax : 0.0f;
      float im = mmax > 0.0f ? 63.0f / mmax : 0.0f;
      // int -> uint8 narrowing wraps before the cap at 63 (kquant.py:530-532)
      Ls = (int)(uint8_t)rint_magic(is * scale);
      Lm = (int)(uint8_t)rint_magic(im * mn);
      Ls = Ls < 63 ? Ls : 63;
      Lm = Lm < 63 ? Lm : 63;
      d = smax / 63.0f;
      dmin = mmax / 63.0f;
    }
    uint16_t d16 = half_bits(d), m16 = half_bits(dmin);
    float dl = half_value(d16) * (float)Ls, ml = half_value(m16) * (float)Lm;
    if constexpr (OUT != KqOut::kFields) {
      if (dl != 0.0f) {
#pragma unroll
        for (int i = 0; i < 32; ++i) L[i] = clampi(rint_magic((xv[i] + ml) / dl), 0, TOP);
      } else {
        affine_final_codes<32>(xv, fit, TOP, L);  // the search's codes stay where dl == 0
      }
    }
    if constexpr (OUT == KqOut::kRecon) {
      rdl = half_value(d16) * (float)(Ls & 63);
      rml = half_value(m16) * (float)(Lm & 63);
    }
    F.a[g] = (uint8_t)Ls;
    F.a[8 + g] = (uint8_t)Lm;
    if (g == 0) {
      F.d = d16;
      F.dmin = m16;
    }
  } else {  // Q6_K
    if constexpr (!IMAT) {
#pragma unroll
      for (int i = 0; i < 16; ++i) wt[i] = xv[i] * xv[i];
    }
    const SignedFit fit = fit_signed<16>(xv, wt, kQxQ6);
    float amax;
    float smax = gfirst_absmax<16>(fit.scale, g, &amax);
    bool dead = amax < 1e-15f;
    float is = -128.0f / (dead ? 1.0f : smax);
    float d = 1.0f / is;
    int q = rint_magic(is * fit.scale);
    int8_t sc = (int8_t)(q < 127 ? q : 127);
    uint16_t d16 = half_bits(dead ? 0.0f : d);
    float dsub = half_value(d16) * (float)sc;
    if constexpr (OUT != KqOut::kFields) {
      if (dsub != 0.0f && !dead)
        signed_requant<16>(xv, fit, dsub, 32, L);
      else
        signed_final_codes<16>(xv, fit, 32, L);  // the search's codes stay where dsub == 0
    }
    if (dead) {
#pragma unroll
      for (int i = 0; i < 16; ++i) L[i] = 0;
      sc = 0;
    }
    if constexpr (OUT == KqOut::kRecon) rdl = half_value(d16) * (float)sc;
    F.a[g] = (uint8_t)sc;
    if (g == 0) F.d = d16;
  }

  const int nvalid = sb0 >= NB ? 0 : (int)((NB - sb0) < S ? (NB - sb0) : S);
  // what follows exchanges data between the lanes of one wave only
  if constexpr (OUT == KqOut::kRecon) {
    // y = (d*sc)*q - (dmin*m), the decoders' expression; each store writes 1 KB
    constexpr int kOff = TT == CP_Q3_K ? 4 : TT == CP_Q6_K ? 32 : 0;
    constexpr bool kMin = TT == CP_Q2_K || TT == CP_Q4_K || TT == CP_Q5_K;
    float* o = reinterpret_cast<float*>(s_buf[wv]);
    wave_lds_fence();
#pragma unroll
    for (int i = 0; i < SUBW; i += 4) {
      float r[4];
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const float v = rdl * (float)(L[i + k] - kOff);
        r[k] = kMin ? v - rml : v;
      }
      *reinterpret_cast<float4*>(o + lane * SUBW + i) = make_float4(r[0], r[1], r[2], r[3]);
    }
    wave_lds_fence();
    float4* y = reinterpret_cast<float4*>(recon + sb0 * 256);
#pragma unroll
    for (int i = 0; i < S; ++i)
      if (i < nvalid) y[64 * i + lane] = reinterpret_cast<const float4*>(o)[64 * i + lane];
  } else if constexpr (OUT == KqOut::kFields) {
    wave_lds_fence();
    pack_wave<TT, false>(nullptr, s_f[wv], lane, nvalid, out + sb0 * BP);
  } else {
    uint8_t* c = &s_codes[wv][sl * 256 + g * SUBW];
#pragma unroll
    for (int i = 0; i < SUBW; i += 4) {
      uint32_t v = (uint32_t)(L[i] & 0xFF) | (uint32_t)(L[i + 1] & 0xFF) << 8 |
                   (uint32_t)(L[i + 2] & 0xFF) << 16 | (uint32_t)(L[i + 3] & 0xFF) << 24;
      *reinterpret_cast<uint32_t*>(c + i) = v;
    }
    wave_lds_fence();
    uint8_t* pk = s_buf[wv];
    pack_wave<TT, true>(s_codes[wv], s_f[wv], lane, S, pk);
    wave_lds_fence();
    // the wave's contiguous bytes leave as coalesced dword stores
    const int bytes = nvalid * BP;
    uint8_t* dst = out + sb0 * BP;
    for (int dw = lane; dw < bytes / 4; dw += 64)
      reinterpret_cast<uint32_t*>(dst)[dw] = reinterpret_cast<const uint32_t*>(pk)[dw];
    if ((bytes & 3) && lane == 0)
      reinterpret_cast<uint16_t*>(dst)[bytes / 2 - 1] = reinterpret_cast<const uint16_t*>(pk)[bytes / 2 - 1];
  }
}

// ---------------------------------------------------------------- decoders
// One thread per 16 consecutive weights of a superblock (16 threads per
// superblock); y = (d*sc)*q - (dmin*m) in float32 (kquant.py:416-427, :489-503,
// :596-627, :681-701).
// The 16 weights k * 16 .. k * 16 + 15 of the superblock at b (global or LDS bytes).
template <int TT>
__device__ __forceinline__ void kq_decode16(const uint8_t* __restrict__ b, int k, float (&out)[16]) {
  if constexpr (TT == CP_Q2_K) {
    float d = half_value(b[80] | b[81] << 8), dm = half_value(b[82] | b[83] << 8);
    float dl = d * (float)(b[k] & 0xF), ml = dm * (float)(b[k] >> 4);
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      int e = 16 * k + i, h = e >> 7, gq = (e >> 5) & 3, l = e & 31;
      int q = (b[16 + h * 32 + l] >> (2 * gq)) & 3;
      out[i] = dl * (float)q - ml;
    }
  } else if constexpr (TT == CP_Q3_K) {
    float d = half_value(b[108] | b[109] << 8);
    const uint8_t* sc = b + 96;
    int lo = (k < 8) ? (sc[k] & 0xF) : (sc[k - 8] >> 4);
    int hi = (sc[8 + (k & 3)] >> (2 * (k >> 2))) & 3;
    float dl = d * (float)((lo | hi << 4) - 32);
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      int e = 16 * k + i, h = e >> 7, gq = (e >> 5) & 3, l = e & 31;
      int q = (b[32 + h * 32 + l] >> (2 * gq)) & 3;
      int hb = (b[e & 31] >> (e >> 5)) & 1;
      out[i] = dl * (float)(q - (hb ? 0 : 4));
    }
  } else if constexpr (TT == CP_Q4_K || TT == CP_Q5_K) {
    constexpr int body = TT == CP_Q5_K ? 48 : 16;
    float d = half_value(b[0] | b[1] << 8), dm = half_value(b[2] | b[3] << 8);
    const uint8_t* sc = b + 4;
    int j = k >> 1, s, m;
    if (j < 4) {
      s = sc[j] & 63;
      m = sc[j + 4] & 63;
    } else {
      s = (sc[j + 4] & 0xF) | (sc[j - 4] >> 6) << 4;
      m = (sc[j + 4] >> 4) | (sc[j] >> 6) << 4;
    }
    float dl = d * (float)s, ml = dm * (float)m;
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      int e = 16 * k + i, c = e >> 6, r = e & 63;
      int q = (r < 32) ? (b[body + c * 32 + r] & 0xF) : (b[body + c * 32 + r - 32] >> 4);
      if constexpr (TT == CP_Q5_K) q |= ((b[16 + (r & 31)] >> (2 * c + (r >> 5))) & 1) << 4;
      out[i] = dl * (float)q - ml;
    }
  } else {  // Q6_K
    float d = half_value(b[208] | b[209] << 8);
    float dl = d * (float)(int8_t)b[192 + k];
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      int e = 16 * k + i, h = e >> 7, gq = (e >> 5) & 3, l = e & 31;
      int qlb = b[h * 64 + (gq & 1) * 32 + l];
      int low = (gq < 2) ? (qlb & 0xF) : (qlb >> 4);
      int high = (b[128 + h * 32 + l] >> (2 * gq)) & 3;
      out[i] = dl * (float)((low | high << 4) - 32);
    }
  }
}

// Decode 16 weights of one superblock: global thread t covers superblock t / 16.
template <int TT>
__device__ __forceinline__ void kq_decode_thread(const uint8_t* __restrict__ raw, int64_t NB,
                                                 float* __restrict__ y, int64_t t) {
  constexpr int BP = Kq<TT>::BP;
  const int64_t sb = t >> 4;
  if (sb >= NB) return;
  const int k = (int)(t & 15);
  float out[16];
  kq_decode16<TT>(raw + sb * BP, k, out);
  float4* o = reinterpret_cast<float4*>(y + sb * 256 + 16 * k);
#pragma unroll
  for (int i = 0; i < 4; ++i) o[i] = make_float4(out[4 * i], out[4 * i + 1], out[4 * i + 2], out[4 * i + 3]);
}

// Decode of whole rows by workgroups of 4 waves, each wave 4 superblocks (1024 weights):
// the wave's container bytes arrive with dword loads (byte loads when the buffer is not
// 4-byte aligned) into LDS, every lane decodes 16 weights from there (lane = superblock
// (l / 16), 16-weight group (l % 16)), and the weights leave through LDS so that each
// store instruction writes 1 KB of consecutive floats. Waves past the end stage and store
// nothing but take part in both barriers.
constexpr int kDecSb = 4;  // superblocks per wave

template <int TT>
struct KqDecodeLds {
  static constexpr int kBytes = (kDecSb * Kq<TT>::BP + 15) / 16 * 16;
  uint8_t bytes[4][kBytes];
  float out[4][kDecSb * 256];
};

template <int TT>
__device__ __forceinline__ void kq_decode_block(const uint8_t* __restrict__ raw, int64_t NB,
                                                float* __restrict__ y, int64_t block, KqDecodeLds<TT>& L) {
  constexpr int BP = Kq<TT>::BP;
  const int w = threadIdx.x >> 6, l = threadIdx.x & 63;
  const int64_t sb0 = (block * 4 + w) * kDecSb;
  const int nsb = sb0 >= NB ? 0 : (int)(NB - sb0 < kDecSb ? NB - sb0 : kDecSb);
  const int nbytes = nsb * BP;
  const uint8_t* src = raw + sb0 * BP;
  uint8_t* dst = L.bytes[w];
  if ((((uintptr_t)src) & 3) == 0) {
    const int nd = nbytes >> 2;
    for (int i = l; i < nd; i += 64)
      reinterpret_cast<uint32_t*>(dst)[i] = reinterpret_cast<const uint32_t*>(src)[i];
    for (int i = 4 * nd + l; i < nbytes; i += 64) dst[i] = src[i];
  } else {
    for (int i = l; i < nbytes; i += 64) dst[i] = src[i];
  }
  __syncthreads();
  const int s = l >> 4, k = l & 15;
  if (s < nsb) {
    float out[16];
    kq_decode16<TT>(dst + s * BP, k, out);
    float4* o = reinterpret_cast<float4*>(&L.out[w][s * 256 + 16 * k]);
#pragma unroll
    for (int i = 0; i < 4; ++i) o[i] = make_float4(out[4 * i], out[4 * i + 1], out[4 * i + 2], out[4 * i + 3]);
  }
  __syncthreads();
  const int nw = nsb * 256;
  float* yo = y + sb0 * 256;
#pragma unroll
  for (int i = 0; i < kDecSb; ++i) {
    const int idx = 256 * i + 4 * l;
    if (idx < nw) *reinterpret_cast<float4*>(yo + idx) = *reinterpret_cast<const float4*>(&L.out[w][idx]);
  }
}

// ---------------------------------------------------------------- Q8_0
// Blocks of 32 weights: d = max|x|/127 (fp16), codes int8 = round-half-away(x/d)
// (kquant.py:706-727). A wave covers 256 consecutive weights (8 blocks) with one
// float4 per lane; the 8 lanes of a block reduce max|x| with xor shuffles (max is
// exact in any order). The wave's 8*34 = 272 output bytes are assembled in LDS
// and leave as 68 dword stores.
constexpr int kQ8Bytes = 34;

// numpy's float32 -> int8 cast of sign(v)*floor(|v|+0.5) on x86: truncation to
// int32 (0x80000000 for NaN, inf and |v| >= 2^31), then the low byte. Finite
// scales keep |v| <= 127; a scale whose reciprocal overflows (max|x| < 3.7e-37)
// sends v to +-inf or NaN, and the reference then stores code 0.
__device__ __forceinline__ uint32_t q8_code(float x, float inv) {
  const float v = x * inv;
  const float a = floorf(fabsf(v) + 0.5f);
  int q = a < 2147483648.0f ? (int)a : 0;
  q = v < 0.0f ? -q : q;
  return (uint32_t)q & 0xFFu;
}

// Encode the 8 * kWavesPerBlock blocks of workgroup ``wg`` (nblk blocks in all).
// Every thread of the workgroup must call this (it holds a barrier).
__device__ __forceinline__ void q8_encode_block(const float* __restrict__ x, int64_t nblk,
                                                uint8_t* __restrict__ out, int64_t wg) {
  __shared__ uint32_t s_out[kWavesPerBlock][68];
  const int wv = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int64_t chunk = wg * kWavesPerBlock + wv;  // 8 blocks per chunk
  const int64_t blk = chunk * 8 + (lane >> 3);
  float4 v = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
  if (blk < nblk) v = reinterpret_cast<const float4*>(x)[chunk * 64 + lane];
  float amax = fmaxf(fmaxf(fabsf(v.x), fabsf(v.y)), fmaxf(fabsf(v.z), fabsf(v.w)));
  amax = fmaxf(amax, __shfl_xor(amax, 1));
  amax = fmaxf(amax, __shfl_xor(amax, 2));
  amax = fmaxf(amax, __shfl_xor(amax, 4));
  const float d = amax / 127.0f;
  const float inv = d != 0.0f ? 1.0f / d : 0.0f;
  const uint32_t codes = q8_code(v.x, inv) | q8_code(v.y, inv) << 8 | q8_code(v.z, inv) << 16 |
                         q8_code(v.w, inv) << 24;
  uint16_t* so = reinterpret_cast<uint16_t*>(s_out[wv]);
  const int h = (lane >> 3) * (kQ8Bytes / 2) + 1 + 2 * (lane & 7);  // in halfwords
  so[h] = (uint16_t)codes;
  so[h + 1] = (uint16_t)(codes >> 16);
  if ((lane & 7) == 0) so[h - 1] = half_bits(d);
  __syncthreads();
  if (chunk * 8 >= nblk) return;
  const int64_t nvalid = nblk - chunk * 8 < 8 ? nblk - chunk * 8 : 8;
  const int bytes = (int)nvalid * kQ8Bytes;
  uint8_t* dst = out + chunk * 8 * kQ8Bytes;
  for (int dw = lane; dw < bytes / 4; dw += 64) reinterpret_cast<uint32_t*>(dst)[dw] = s_out[wv][dw];
  if ((bytes & 3) && lane == 0)
    reinterpret_cast<uint16_t*>(dst)[bytes / 2 - 1] = so[bytes / 2 - 1];
}

// Decode 4 consecutive weights (global thread t): y = d * code in float32.
__device__ __forceinline__ void q8_decode_thread(const uint8_t* __restrict__ raw, int64_t nblk,
                                                 float* __restrict__ y, int64_t t) {
  const int64_t blk = t >> 3;
  if (blk >= nblk) return;
  const uint16_t* b = reinterpret_cast<const uint16_t*>(raw + blk * kQ8Bytes);
  const int j = (int)(t & 7);
  const float d = half_value(b[0]);
  const uint32_t c = (uint32_t)b[1 + 2 * j] | (uint32_t)b[2 + 2 * j] << 16;
  reinterpret_cast<float4*>(y)[t] =
      make_float4(d * (float)(int8_t)(c & 0xFF), d * (float)(int8_t)((c >> 8) & 0xFF),
                  d * (float)(int8_t)((c >> 16) & 0xFF), d * (float)(int8_t)(c >> 24));
}

}  // namespace cp
