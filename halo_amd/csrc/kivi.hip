// KIVI-style 2/4/8-bit cold-chunk format: quantize and dequantize kernels
// (gfx950, wave64).  Byte/integer work bound by HBM; nothing here is a GEMM.
//
// Arithmetic: baselines/kivi_cache.py:44-78 with every operation rounded to
// the storage dtype as torch evaluates a chain of fp16/bf16 tensor ops:
//   scale = dtype(dtype(max(dtype(x_max - x_min), dtype(1e-8))) / qmax)
//   zero  = x_min
//   code  = clamp(rint(dtype(dtype(x - zero) / scale)), 0, qmax), NaN -> 0
//   x'    = dtype(fp32(fp32(code) * fp32(scale)) + fp32(zero))
// (built with -ffp-contract=off: no fused multiply-add anywhere).
// K is grouped per channel over 32 consecutive tokens, V per token over 32
// consecutive channels (the reference groups along the last axis only,
// kivi_cache.py:56; K per-channel applies the same per-element arithmetic
// along the token axis).
//
// Block layout (one block = 32 tokens of one (b, h_kv); byte offsets):
//   [0, C)            K codes, token-major rows of D*bits/8 bytes (code
//                     positions within a row below)
//   [C, C+2D)         K scale, D elements of the dtype (per channel)
//   [C+2D, C+4D)      K zero
//   [C+4D, 2C+4D)     V codes, channel-major rows of 32*bits/8 bytes, one
//                     code per token slot
//   [2C+4D, 2C+6D)    V scale, D/32 groups x 32 token slots (group-major)
//   [2C+6D, 2C+8D)    V zero
// with C = 32*D*bits/8.  D=128, bits=2: 3072 bytes per block.  The V side
// is transposed, and its 32 tokens are stored in slot order: slot 8g + j
// holds token 4g + j (j < 4) or 16 + 4g + j - 4 (j >= 4), the tokens one
// lane group g of a 16x16x32 MFMA holds in its score accumulator (rows
// 4g..4g+3 of both 16-token halves).  So the P.V operand of one lane is 8
// slots = 16 contiguous bits of one channel, its scales (or zeros) are 16
// contiguous bytes of one group, and its p values are its own scores.
// Code positions within a row: 4- and 8-bit codes, element e at bit e*bits
// (8-bit: one byte per code); 2-bit
// codes, each 16-bit word holds 8 elements, the even ones (2j) at bits 2j
// of its low byte and the odd ones (2j+1) at bits 8+2j of its high byte, so
// that w | w << 8 holds elements 2j and 2j+1 at bits 2j and 16+2j: one mask
// places a pair in the two fp16 halves of a register.

#include "common.hpp"

namespace halo {

constexpr int kKiviG = 32;

// token held by V slot s of a block, and the slot of token t
__host__ __device__ constexpr int kivi_vtok(int s) { return (s & 4 ? 16 : 0) + 4 * (s >> 3) + (s & 3); }
__host__ __device__ constexpr int kivi_vslot(int t) { return 8 * ((t >> 2) & 3) + 4 * (t >> 4) + (t & 3); }
static_assert(kivi_vslot(kivi_vtok(13)) == 13 && kivi_vtok(kivi_vslot(21)) == 21, "V slot order");

// element (within its row) of the code at bits [c*BITS, (c+1)*BITS) of byte q
// of the row, and the bit position of element e (its inverse)
template <int BITS>
__host__ __device__ constexpr int kivi_elem(int q, int c) {
  return BITS == 2 ? (q & ~1) * 4 + 2 * c + (q & 1) : q * (8 / BITS) + c;
}
template <int BITS>
__host__ __device__ constexpr int kivi_bit(int e) {
  return BITS == 2 ? 16 * (e >> 3) + 2 * ((e & 7) >> 1) + 8 * (e & 1) : e * BITS;
}
static_assert(kivi_bit<2>(kivi_elem<2>(5, 3)) == 5 * 8 + 3 * 2 && kivi_bit<2>(kivi_elem<2>(6, 1)) == 6 * 8 + 2 &&
                  kivi_bit<4>(kivi_elem<4>(3, 1)) == 3 * 8 + 4,
              "code positions");

__host__ __device__ constexpr int kivi_code_bytes(int D, int bits) { return kKiviG * D * bits / 8; }
__host__ __device__ constexpr int kivi_block_bytes(int D, int bits) { return 2 * kivi_code_bytes(D, bits) + 8 * D; }

template <int DT>
__device__ __forceinline__ float round_dt(float x) {
  if constexpr (DT == HALO_BF16) return __uint_as_float((uint32_t)f32_to_bf16_rne(x) << 16);
  return f16_bits_to_f32(f32_to_f16_rne(x));
}
template <int DT>
__device__ __forceinline__ uint16_t bits_dt(float x) {
  if constexpr (DT == HALO_BF16) return f32_to_bf16_rne(x);
  return f32_to_f16_rne(x);
}
template <int DT>
__device__ __forceinline__ float from_bits(uint16_t h) {
  if constexpr (DT == HALO_BF16) return __uint_as_float((uint32_t)h << 16);
  return f16_bits_to_f32(h);
}

// scale/zero of one group from its (dtype-exact) min and max
template <int DT, int BITS>
__device__ __forceinline__ void kivi_params(float mn, float mx, float& scale, float& zero) {
  constexpr float qmax = (float)((1 << BITS) - 1);
  const float eps = round_dt<DT>(1e-8f);
  float rng = round_dt<DT>(opaque(mx - mn));
  rng = round_dt<DT>(fmaxf(rng, eps));
  scale = round_dt<DT>(opaque(rng / qmax));
  zero = mn;
}
template <int DT, int BITS>
__device__ __forceinline__ uint32_t kivi_code(float x, float scale, float zero) {
  constexpr float qmax = (float)((1 << BITS) - 1);
  const float diff = round_dt<DT>(opaque(x - zero));
  float ratio = round_dt<DT>(opaque(diff / scale));
  if (ratio != ratio) ratio = 0.f;
  const float c = fminf(fmaxf(rintf(ratio), 0.f), qmax);
  return (uint32_t)c;
}

struct KiviQuantParams {
  const void* k;
  int64_t ksb, ksh, kst;
  const void* v;
  int64_t vsb, vsh, vst;
  int H_kv, n_blk;
  uint8_t* blocks;
  int64_t bsb, bsh;  // bytes
  int vec16;         // K and V rows 16-byte aligned: tiles loaded with 16-byte loads
};

// Keeps an fp32 value from being folded into the conversion behind it.
__device__ __forceinline__ float pin(float x) {
  asm("" : "+v"(x));
  return x;
}

// Two values rounded to the dtype; bf16 in one v_cvt_pk_bf16_f32.
template <int DT>
__device__ __forceinline__ void round_pair(float& a, float& b) {
  if constexpr (DT == HALO_BF16) {
    typedef __attribute__((ext_vector_type(2))) __bf16 b2;
    const b2 v = {(__bf16)a, (__bf16)b};
    const uint32_t w = __builtin_bit_cast(uint32_t, v);
    a = bf16_lo(w);
    b = bf16_hi(w);
  } else {
    a = (float)(_Float16)pin(a);
    b = (float)(_Float16)pin(b);
  }
}

// Codes of x without a division: with inv = 1/scale correctly rounded, d =
// dtype(x - zero) >= 0, q = d * inv, r = fma(-q, scale, d), the quotient q' =
// fma(r, inv, q) equals the correctly rounded d / scale whenever d is 0 or in
// [2^-63, 2^63] and scale is in [2^-63, 2^63] -- checked exhaustively for every
// pair of fp16 and bf16 values.  Scales of [2^-60, 2^50] are taken here, so that
// d <= 2^8 * scale * (1 + 2^-7) stays in range above, and below 2^-63 both the
// quotient and q' are under 1/4: code 0.  A zero scale (an fp16 group whose
// range rounds to 0 in qmax parts) goes with inv = 2^100: d = 0 gives 0 (as the
// NaN of 0 / 0 does) and any other d infinity in fp16, as d / 0 does.
__device__ __forceinline__ bool kivi_scale_ok(float scale) {
  return (scale >= 0x1p-60f && scale <= 0x1p50f) || scale == 0.f;
}
__device__ __forceinline__ float4 kivi_code_params(float scale, float zero) {
  return make_float4(scale, scale == 0.f ? 0x1p100f : 1.0f / scale, zero, 0.f);
}
// codes of two elements, as floats; p = (scale, inv, zero, -) of each
template <int DT, int BITS>
__device__ __forceinline__ void kivi_code_pair(float& a, float& b, const float4& pa, const float4& pb) {
  constexpr float qmax = (float)((1 << BITS) - 1);
  a -= pa.z;
  b -= pb.z;
  round_pair<DT>(a, b);
  const float qa = pin(a * pa.y), qb = pin(b * pb.y);
  a = __builtin_fmaf(__builtin_fmaf(-qa, pa.x, a), pa.y, qa);
  b = __builtin_fmaf(__builtin_fmaf(-qb, pb.x, b), pb.y, qb);
  round_pair<DT>(a, b);
  // clamp in one operation; of a NaN it is the smallest of the others, 0
  a = __builtin_amdgcn_fmed3f(rintf(a), 0.f, qmax);
  b = __builtin_amdgcn_fmed3f(rintf(b), 0.f, qmax);
}
// min(a, x, y) and max(a, x, y), NaN dropped, in one operation each.  With the
// IEEE bit of the mode register set, as a kernel begins, a signalling NaN (a bf16
// element can be one: its conversion is a shift) comes back as a quiet one and
// takes `a` with it; drop_all_nan clears the bit.  Quieting every element
// instead costs an operation each.
__device__ __forceinline__ void drop_all_nan() {
  constexpr int kMode = 1, kIeeeBit = 9;  // hwreg(HW_REG_MODE, 9, 1)
  __builtin_amdgcn_s_setreg(kMode | kIeeeBit << 6, 0);
}
__device__ __forceinline__ float kmin3(float a, float x, float y) {
  float r;
  asm("v_min3_f32 %0, %1, %2, %3" : "=v"(r) : "v"(a), "v"(x), "v"(y));
  return r;
}
__device__ __forceinline__ float kmax3(float a, float x, float y) {
  float r;
  asm("v_max3_f32 %0, %1, %2, %3" : "=v"(r) : "v"(a), "v"(x), "v"(y));
  return r;
}

// Codes of one block from its staged tiles.  An 8-element run is 8 * BITS bits,
// collected as BITS/2 fp32 sums of code * 2^position (16 bits each: exact).
template <int DT, int D, int BITS, bool FAST>
__device__ __forceinline__ void kivi_store_codes(const uint16_t* s_k, const uint16_t* s_v, const float4* s_kp,
                                                 const float4* s_vp, uint8_t* out) {
  constexpr int G = kKiviG, NG = D / G, RS = D + 8, C = kivi_code_bytes(D, BITS);
  constexpr int NW = BITS / 2;  // 16-bit words of an 8-element run
  const int tid = threadIdx.x;
  auto codes = [](float& a, float& b, const float4& pa, const float4& pb) {
    if constexpr (FAST) {
      kivi_code_pair<DT, BITS>(a, b, pa, pb);
    } else {
      a = (float)kivi_code<DT, BITS>(a, pa.x, pa.z);
      b = (float)kivi_code<DT, BITS>(b, pb.x, pb.z);
    }
  };
  auto put_words = [](uint8_t* dst, const float (&sum)[NW]) {  // BITS bytes
    if constexpr (BITS == 2) {
      *reinterpret_cast<uint16_t*>(dst) = (uint16_t)(uint32_t)sum[0];
    } else if constexpr (BITS == 4) {
      *reinterpret_cast<uint32_t*>(dst) = (uint32_t)sum[0] | (uint32_t)sum[1] << 16;
    } else {
      *reinterpret_cast<uint2*>(dst) = make_uint2((uint32_t)sum[0] | (uint32_t)sum[1] << 16,
                                                  (uint32_t)sum[2] | (uint32_t)sum[3] << 16);
    }
  };
  // K: 32 rows x D elements; thread = (8 channels, TT tokens), so that the
  // parameters of its channels, the larger part of the LDS reads, are read once.
  // At D = 64 the V codes below occupy half of the threads, so the other half
  // takes the K codes (32768 tokens x 8 heads of f16 in 4 / 8 bits: 27.5 / 28.5 us
  // with all threads on K first, 26.4 / 27.1 so, 26.2 / 27.0 with the V
  // parameters on threads of their own as well).
  constexpr int KT = D == 64 ? 128 : 256;  // threads on the K codes
  if (KT == 256 || tid < KT) {
    constexpr int TT = 4 * D / KT;
    const int oct = tid % (D / 8), t0 = (tid / (D / 8)) * TT;
    float sum[TT][NW] = {};
    uint4 r[TT];
#pragma unroll
    for (int t = 0; t < TT; ++t) r[t] = *reinterpret_cast<const uint4*>(&s_k[(t0 + t) * RS + 8 * oct]);
#pragma unroll
    for (int i = 0; i < 8; i += 2) {
      const float4 pa = s_kp[9 * oct + i], pb = s_kp[9 * oct + i + 1];
#pragma unroll
      for (int t = 0; t < TT; ++t) {
        const uint32_t w = i == 0 ? r[t].x : i == 2 ? r[t].y : i == 4 ? r[t].z : r[t].w;
        float a = from_bits<DT>((uint16_t)w), c = from_bits<DT>((uint16_t)(w >> 16));
        codes(a, c, pa, pb);
        const int b0 = kivi_bit<BITS>(i), b1 = kivi_bit<BITS>(i + 1);
        sum[t][b0 >> 4] = __builtin_fmaf(a, (float)(1 << (b0 & 15)), sum[t][b0 >> 4]);
        sum[t][b1 >> 4] = __builtin_fmaf(c, (float)(1 << (b1 & 15)), sum[t][b1 >> 4]);
      }
    }
#pragma unroll
    for (int t = 0; t < TT; ++t) put_words(out + (t0 + t) * (D * BITS / 8) + oct * BITS, sum[t]);
  }
  // V: D rows (channels) x 32 slots; thread = (two channels, 8 consecutive slots)
  constexpr int VRB = G * BITS / 8;          // V code bytes per channel row
  for (int u = tid - (256 - KT); u < 2 * D; u += 256) {
    if (KT < 256 && u < 0) break;
    const int d = 2 * (u >> 2), o = u & 3;
    const int g = d / G;
    float sum[2][NW] = {};
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const int t = (i & 4 ? 16 : 0) + 4 * o + (i & 3);  // kivi_vtok(8 * o + i)
      const float4 pv = s_vp[t * NG + g];
      const uint32_t w = *reinterpret_cast<const uint32_t*>(&s_v[t * RS + d]);
      float a = from_bits<DT>((uint16_t)w), c = from_bits<DT>((uint16_t)(w >> 16));
      codes(a, c, pv, pv);
      const int bit = kivi_bit<BITS>(i);
      sum[0][bit >> 4] = __builtin_fmaf(a, (float)(1 << (bit & 15)), sum[0][bit >> 4]);
      sum[1][bit >> 4] = __builtin_fmaf(c, (float)(1 << (bit & 15)), sum[1][bit >> 4]);
    }
    put_words(out + C + 4 * D + d * VRB + o * BITS, sum[0]);
    put_words(out + C + 4 * D + (d + 1) * VRB + o * BITS, sum[1]);
  }
}

// One workgroup per block, 256 threads.  The 32 x D K and V tiles are staged
// in LDS in their storage dtype (16-byte loads; rows padded by 16 bytes so
// column and row-run reads spread over the banks); 512/D threads reduce each
// pair of K channels and two each V (token, 32-channel group) to its min / max;
// then each thread codes 8 channels of D/64 output rows (K, token-major) and
// two channels x 8 slots (V, channel-major in slot order), at D = 64 one of the
// two with as much work, and stores packed bytes.  An element costs about 14 VALU operations (bf16 rounding in hardware
// two at a time, no per-element range branch, codes packed by fp32
// multiply-adds of up to 16 bits), where rounding by hand and a checked quotient
// took 23 in fp16 and more than twice that in bf16.  32768 tokens x 8 heads x 128
// bf16 in 2 bits: 102.9 us before, 45.7 now (3.4 TB/s), bound by the phases
// behind its barriers.  Workgroups that walk several blocks with the next
// block's loads in flight took 69: the barriers wait for those loads.
template <int DT, int D, int BITS>
__global__ void __launch_bounds__(256) kivi_quantize_kernel(KiviQuantParams P) {
  constexpr int G = kKiviG;
  constexpr int C = kivi_code_bytes(D, BITS);
  constexpr int NG = D / G;                  // V groups per token
  constexpr int RS = D + 8;                  // LDS row stride (elements)
  constexpr int KP = D + D / 8;              // padded params (one float4 per channel, a pad per 8)
  __shared__ __align__(16) uint16_t s_k[G * RS], s_v[G * RS];
  constexpr int NP = 512 / D, PT = G / NP;   // partial K ranges per channel, of PT tokens: a pair per thread
  __shared__ __align__(8) float s_kmn[NP][D], s_kmx[NP][D];
  __shared__ float s_vmn[2][G * NG], s_vmx[2][G * NG];
  __shared__ __align__(16) float4 s_kp[KP];  // kivi_code_params per channel
  __shared__ __align__(16) float4 s_vp[G * NG];
  drop_all_nan();
  const int tid = threadIdx.x;
  const int j = blockIdx.x % P.n_blk;
  const int bh = blockIdx.x / P.n_blk;
  const int h = bh % P.H_kv, b = bh / P.H_kv;
  const uint16_t* kb = reinterpret_cast<const uint16_t*>(P.k) + (int64_t)b * P.ksb + (int64_t)h * P.ksh +
                       (int64_t)j * G * P.kst;
  const uint16_t* vb = reinterpret_cast<const uint16_t*>(P.v) + (int64_t)b * P.vsb + (int64_t)h * P.vsh +
                       (int64_t)j * G * P.vst;
  if (P.vec16) {
    constexpr int PR = D / 8;  // 16-byte pieces per row
    uint4 kk[G * PR / 256], vv[G * PR / 256];
#pragma unroll
    for (int i = 0; i < G * PR / 256; ++i) {
      const int e = tid + 256 * i, t = e / PR, c = e % PR;
      kk[i] = *reinterpret_cast<const uint4*>(kb + (int64_t)t * P.kst + 8 * c);
      vv[i] = *reinterpret_cast<const uint4*>(vb + (int64_t)t * P.vst + 8 * c);
    }
#pragma unroll
    for (int i = 0; i < G * PR / 256; ++i) {
      const int e = tid + 256 * i, t = e / PR, c = e % PR;
      *reinterpret_cast<uint4*>(&s_k[t * RS + 8 * c]) = kk[i];
      *reinterpret_cast<uint4*>(&s_v[t * RS + 8 * c]) = vv[i];
    }
  } else {
    for (int e = tid; e < G * D; e += 256) {
      const int t = e / D, d = e % D;
      s_k[t * RS + d] = kb[(int64_t)t * P.kst + d];
      s_v[t * RS + d] = vb[(int64_t)t * P.vst + d];
    }
  }
  __syncthreads();
  // min / max: K per (two channels, PT of the tokens), V per (token, group, half of the channels)
  {
    const int d = 2 * (tid % (D / 2)), qt = tid / (D / 2);
    uint32_t w[PT];
#pragma unroll
    for (int t = 0; t < PT; ++t) w[t] = *reinterpret_cast<const uint32_t*>(&s_k[(PT * qt + t) * RS + d]);
    float mn[2], mx[2];
#pragma unroll
    for (int c = 0; c < 2; ++c) {
      float x[PT];
#pragma unroll
      for (int t = 0; t < PT; ++t) x[t] = from_bits<DT>((uint16_t)(c ? w[t] >> 16 : w[t]));
      mn[c] = fminf(x[0], x[1]);
      mx[c] = fmaxf(x[0], x[1]);
#pragma unroll
      for (int t = 2; t < PT; t += 2) {
        mn[c] = kmin3(mn[c], x[t], x[t + 1]);
        mx[c] = kmax3(mx[c], x[t], x[t + 1]);
      }
    }
    *reinterpret_cast<float2*>(&s_kmn[qt][d]) = make_float2(mn[0], mn[1]);
    *reinterpret_cast<float2*>(&s_kmx[qt][d]) = make_float2(mx[0], mx[1]);
  }
  for (int i = tid; i < 2 * G * NG; i += 256) {
    const int tg = i >> 1, hf = i & 1;
    const int t = tg / NG, g = tg % NG;
    const uint4* row = reinterpret_cast<const uint4*>(&s_v[t * RS + g * G + 16 * hf]);
    const uint4 r0 = row[0], r1 = row[1];
    const uint32_t w[8] = {r0.x, r0.y, r0.z, r0.w, r1.x, r1.y, r1.z, r1.w};
    float mn = from_bits<DT>((uint16_t)w[0]), mx = mn;
#pragma unroll
    for (int c = 0; c < 8; ++c) {
      const float lo = from_bits<DT>((uint16_t)w[c]), hi = from_bits<DT>((uint16_t)(w[c] >> 16));
      mn = kmin3(mn, lo, hi);
      mx = kmax3(mx, lo, hi);
    }
    s_vmn[hf][tg] = mn;
    s_vmx[hf][tg] = mx;
  }
  __syncthreads();
  uint8_t* out = P.blocks + (int64_t)b * P.bsb + (int64_t)h * P.bsh + (int64_t)j * kivi_block_bytes(D, BITS);
  uint16_t* meta_k = reinterpret_cast<uint16_t*>(out + C);
  uint16_t* meta_v = reinterpret_cast<uint16_t*>(out + 2 * C + 4 * D);
  bool ok = true;
  for (int d = tid; d < D; d += 256) {
    float sc, z;
    float mn = s_kmn[0][d], mx = s_kmx[0][d];
#pragma unroll
    for (int p = 1; p < NP; ++p) {
      mn = fminf(mn, s_kmn[p][d]);
      mx = fmaxf(mx, s_kmx[p][d]);
    }
    kivi_params<DT, BITS>(mn, mx, sc, z);
    s_kp[d + d / 8] = kivi_code_params(sc, z);
    ok = ok && kivi_scale_ok(sc);
    meta_k[d] = bits_dt<DT>(sc);
    meta_k[D + d] = bits_dt<DT>(z);
  }
  for (int tg = tid - D % 256; tg < G * NG; tg += 256) {  // on the threads behind K's
    if (tg < 0) break;
    float sc, z;
    kivi_params<DT, BITS>(fminf(s_vmn[0][tg], s_vmn[1][tg]), fmaxf(s_vmx[0][tg], s_vmx[1][tg]), sc, z);
    s_vp[tg] = kivi_code_params(sc, z);
    ok = ok && kivi_scale_ok(sc);
    const int t = tg / NG, g = tg % NG;
    meta_v[g * G + kivi_vslot(t)] = bits_dt<DT>(sc);            // group-major, slot order
    meta_v[G * NG + g * G + kivi_vslot(t)] = bits_dt<DT>(z);
  }
  // every group's scale in range: no division; else all of the block divides
  if (__syncthreads_and(ok)) kivi_store_codes<DT, D, BITS, true>(s_k, s_v, s_kp, s_vp, out);
  else kivi_store_codes<DT, D, BITS, false>(s_k, s_v, s_kp, s_vp, out);
}

struct KiviDequantParams {
  const uint8_t* blocks;
  int64_t bsb, bsh;
  int H_kv, n_blk;
  void* k;
  int64_t ksb, ksh, kst;
  void* v;
  int64_t vsb, vsh, vst;
};

// One thread per (block, K or V, 8-channel piece c, lane group o): it turns the
// codes of 8 channels x 8 tokens (K: tokens o + 4i; V: slots 8o..8o+7, whose
// codes are one BITS-byte word a channel) with the scales and zeros of its piece
// held in registers, and stores 16 bytes a token, so that a wave stores whole
// rows.  K and V take the two halves of a workgroup.  32768 tokens x 8 heads x
// 128 bf16 in 2 bits: 51.2 us with a thread per element (byte and 2-byte loads,
// 2-byte stores), 28.2 here (5.7 TB/s).
template <int DT, int D, int BITS>
__global__ void __launch_bounds__(256) kivi_dequant_piece_kernel(KiviDequantParams P, int n) {
  constexpr int G = kKiviG;
  constexpr int C = kivi_code_bytes(D, BITS);
  constexpr int NG = D / G;
  constexpr int PR = D / 8;               // pieces per row
  constexpr int NB = 128 / (4 * PR);      // blocks per workgroup
  constexpr uint32_t MASK = (1u << BITS) - 1;
  const bool is_v = threadIdx.x >= 128;
  const int x = threadIdx.x & 127;
  const int c = x % PR, o = (x / PR) & 3;
  const int blk = blockIdx.x * NB + x / (4 * PR);
  if (blk >= n) return;
  const int j = blk % P.n_blk;
  const int bh = blk / P.n_blk;
  const int h = bh % P.H_kv, b = bh / P.H_kv;
  const uint8_t* src = P.blocks + (int64_t)b * P.bsb + (int64_t)h * P.bsh + (int64_t)j * kivi_block_bytes(D, BITS);
  // the 8 codes of word i: two 32-bit halves for 8-bit codes, one below
  uint32_t code[8][BITS == 8 ? 2 : 1];
  const uint8_t* cb = src + (is_v ? C + 4 * D + 8 * c * (G * BITS / 8) + o * BITS : o * (D * BITS / 8) + c * BITS);
  const int step = is_v ? G * BITS / 8 : 4 * (D * BITS / 8);
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    if constexpr (BITS == 2) {
      code[i][0] = *reinterpret_cast<const uint16_t*>(cb + i * step);
    } else if constexpr (BITS == 4) {
      code[i][0] = *reinterpret_cast<const uint32_t*>(cb + i * step);
    } else {
      const uint2 w = *reinterpret_cast<const uint2*>(cb + i * step);
      code[i][0] = w.x;
      code[i][1] = w.y;
    }
  }
  const uint8_t* meta = src + (is_v ? 2 * C + 4 * D + (c / 4) * 2 * G + 16 * o : C + 16 * c);
  float sc[8], z[8];  // K: of the channels, V: of the slots
  unpack16<DT>(*reinterpret_cast<const uint4*>(meta), sc);
  unpack16<DT>(*reinterpret_cast<const uint4*>(meta + (is_v ? 2 * G * NG : 2 * D)), z);
  auto at = [&](int w, int e) {  // code e of word w
    const int bit = kivi_bit<BITS>(e);
    return (float)((code[w][BITS == 8 ? bit >> 5 : 0] >> (bit & 31)) & MASK);
  };
  auto put = [&](uint16_t* base, int64_t row, const float* f) {
    uint32_t w[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      if constexpr (DT == HALO_BF16) {
        typedef __attribute__((ext_vector_type(2))) __bf16 b2;
        const b2 v = {(__bf16)f[2 * e], (__bf16)f[2 * e + 1]};
        w[e] = __builtin_bit_cast(uint32_t, v);
      } else {
        w[e] = (uint32_t)f32_to_f16_rne(pin(f[2 * e])) | (uint32_t)f32_to_f16_rne(pin(f[2 * e + 1])) << 16;
      }
    }
    *reinterpret_cast<uint4*>(base + row + 8 * c) = make_uint4(w[0], w[1], w[2], w[3]);
  };
  if (!is_v) {
    uint16_t* ko = reinterpret_cast<uint16_t*>(P.k) + (int64_t)b * P.ksb + (int64_t)h * P.ksh + (int64_t)j * G * P.kst;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      float f[8];
#pragma unroll
      for (int e = 0; e < 8; ++e) f[e] = pin(at(i, e) * sc[e]) + z[e];
      put(ko, (int64_t)(o + 4 * i) * P.kst, f);
    }
  } else {
    uint16_t* vo = reinterpret_cast<uint16_t*>(P.v) + (int64_t)b * P.vsb + (int64_t)h * P.vsh + (int64_t)j * G * P.vst;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      float f[8];
#pragma unroll
      for (int e = 0; e < 8; ++e) f[e] = pin(at(e, i) * sc[i]) + z[i];
      put(vo, (int64_t)((i & 4 ? 16 : 0) + 4 * o + (i & 3)) * P.vst, f);
    }
  }
}

// Any alignment of blocks and rows: one thread per element.
template <int DT, int D, int BITS>
__global__ void __launch_bounds__(256) kivi_dequant_kernel(KiviDequantParams P) {
  constexpr int G = kKiviG;
  constexpr int C = kivi_code_bytes(D, BITS);
  constexpr int NG = D / G;
  constexpr uint32_t MASK = (1u << BITS) - 1;
  const int tid = threadIdx.x;
  const int j = blockIdx.x % P.n_blk;
  const int bh = blockIdx.x / P.n_blk;
  const int h = bh % P.H_kv, b = bh / P.H_kv;
  const uint8_t* blk = P.blocks + (int64_t)b * P.bsb + (int64_t)h * P.bsh + (int64_t)j * kivi_block_bytes(D, BITS);
  const uint16_t* meta_k = reinterpret_cast<const uint16_t*>(blk + C);
  const uint16_t* meta_v = reinterpret_cast<const uint16_t*>(blk + 2 * C + 4 * D);
  uint16_t* ko = reinterpret_cast<uint16_t*>(P.k) + (int64_t)b * P.ksb + (int64_t)h * P.ksh + (int64_t)j * G * P.kst;
  uint16_t* vo = reinterpret_cast<uint16_t*>(P.v) + (int64_t)b * P.vsb + (int64_t)h * P.vsh + (int64_t)j * G * P.vst;
  for (int e = tid; e < G * D; e += 256) {
    const int t = e / D, d = e % D;
    const int bit = kivi_bit<BITS>(d);
    const uint32_t ck = (blk[t * (D * BITS / 8) + bit / 8] >> (bit % 8)) & MASK;
    const int ts = kivi_vslot(t);
    const int tbit = kivi_bit<BITS>(ts);
    const uint32_t cv = (blk[C + 4 * D + d * (G * BITS / 8) + tbit / 8] >> (tbit % 8)) & MASK;
    const float sk = from_bits<DT>(meta_k[d]), zk = from_bits<DT>(meta_k[D + d]);
    const float sv = from_bits<DT>(meta_v[(d / G) * G + ts]), zv = from_bits<DT>(meta_v[G * NG + (d / G) * G + ts]);
    // both fp32 results are materialised so the conversion rounds the fp32
    // sum (no mixed-precision fused add-and-convert)
    ko[(int64_t)t * P.kst + d] = bits_dt<DT>(opaque(opaque((float)ck * sk) + zk));
    vo[(int64_t)t * P.vst + d] = bits_dt<DT>(opaque(opaque((float)cv * sv) + zv));
  }
}

}  // namespace halo

using namespace halo;

extern "C" size_t halo_kivi_block_bytes(int D, int bits) {
  if ((bits != 2 && bits != 4 && bits != 8) || D <= 0 || D % kKiviG) return 0;
  return (size_t)kivi_block_bytes(D, bits);
}

namespace {

template <int DT, int D>
int quant_bits(const KiviQuantParams& p, int bits, int n, hipStream_t st) {
  if (bits == 2) hipLaunchKernelGGL((kivi_quantize_kernel<DT, D, 2>), dim3(n), dim3(256), 0, st, p);
  else if (bits == 4) hipLaunchKernelGGL((kivi_quantize_kernel<DT, D, 4>), dim3(n), dim3(256), 0, st, p);
  else hipLaunchKernelGGL((kivi_quantize_kernel<DT, D, 8>), dim3(n), dim3(256), 0, st, p);
  HALO_CHECK_HIP(hipGetLastError());
  return HALO_OK;
}
template <int DT, int D, int BITS>
int dequant_run(const KiviDequantParams& p, int n, hipStream_t st) {
  auto a16 = [](const void* q, int64_t sb, int64_t sh, int64_t s) {
    return (reinterpret_cast<uintptr_t>(q) & 15) == 0 && sb % 16 == 0 && sh % 16 == 0 && s % 16 == 0;
  };
  // 16-byte loads and stores where blocks and rows allow them
  if (a16(p.blocks, p.bsb, p.bsh, 0) && a16(p.k, 2 * p.ksb, 2 * p.ksh, 2 * p.kst) &&
      a16(p.v, 2 * p.vsb, 2 * p.vsh, 2 * p.vst)) {
    constexpr int NB = 256 / D;
    hipLaunchKernelGGL((kivi_dequant_piece_kernel<DT, D, BITS>), dim3((n + NB - 1) / NB), dim3(256), 0, st, p, n);
  } else {
    hipLaunchKernelGGL((kivi_dequant_kernel<DT, D, BITS>), dim3(n), dim3(256), 0, st, p);
  }
  HALO_CHECK_HIP(hipGetLastError());
  return HALO_OK;
}
template <int DT, int D>
int dequant_bits(const KiviDequantParams& p, int bits, int n, hipStream_t st) {
  if (bits == 2) return dequant_run<DT, D, 2>(p, n, st);
  if (bits == 4) return dequant_run<DT, D, 4>(p, n, st);
  return dequant_run<DT, D, 8>(p, n, st);
}

}  // namespace

extern "C" int halo_kivi_quantize(const void* k, int64_t k_stride_b, int64_t k_stride_h, int64_t k_stride_t,
                                  const void* v, int64_t v_stride_b, int64_t v_stride_h, int64_t v_stride_t,
                                  int dtype, int B, int H_kv, int T, int D, int bits,
                                  void* blocks, int64_t blk_stride_b, int64_t blk_stride_h, void* stream) {
  HALO_CHECK_ARG(k && v && blocks, "null pointer");
  HALO_CHECK_ARG(dtype == HALO_F16 || dtype == HALO_BF16, "KIVI storage dtype must be fp16 or bf16");
  HALO_CHECK_ARG(bits == 2 || bits == 4 || bits == 8, "bits must be 2, 4 or 8");
  HALO_CHECK_ARG(D == 64 || D == 128 || D == 256, "head_dim must be 64, 128 or 256");
  HALO_CHECK_ARG(B >= 0 && H_kv > 0 && T >= 0 && T % kKiviG == 0, "T must be a multiple of the group size 32");
  const int n_blk = T / kKiviG;
  const int64_t n = (int64_t)B * H_kv * n_blk;
  if (n == 0) return HALO_OK;
  HALO_CHECK_ARG(n < (1ll << 31), "too many blocks");
  auto a16 = [](const void* p, int64_t stride_elems) {
    return (reinterpret_cast<uintptr_t>(p) & 15) == 0 && (stride_elems * 2) % 16 == 0;
  };
  const int vec16 = a16(k, k_stride_t) && a16(v, v_stride_t) && (k_stride_b * 2) % 16 == 0 &&
                    (k_stride_h * 2) % 16 == 0 && (v_stride_b * 2) % 16 == 0 && (v_stride_h * 2) % 16 == 0;
  HALO_CHECK_ARG((reinterpret_cast<uintptr_t>(blocks) & 15) == 0 && blk_stride_b % 16 == 0 && blk_stride_h % 16 == 0,
                 "block buffer must be 16-byte aligned");
  KiviQuantParams p{k, k_stride_b, k_stride_h, k_stride_t, v, v_stride_b, v_stride_h, v_stride_t,
                    H_kv, n_blk, reinterpret_cast<uint8_t*>(blocks), blk_stride_b, blk_stride_h, vec16};
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  if (dtype == HALO_F16) {
    if (D == 64) return quant_bits<HALO_F16, 64>(p, bits, (int)n, st);
    if (D == 128) return quant_bits<HALO_F16, 128>(p, bits, (int)n, st);
    return quant_bits<HALO_F16, 256>(p, bits, (int)n, st);
  }
  if (D == 64) return quant_bits<HALO_BF16, 64>(p, bits, (int)n, st);
  if (D == 128) return quant_bits<HALO_BF16, 128>(p, bits, (int)n, st);
  return quant_bits<HALO_BF16, 256>(p, bits, (int)n, st);
}

extern "C" int halo_kivi_dequantize(const void* blocks, int64_t blk_stride_b, int64_t blk_stride_h,
                                    int dtype, int B, int H_kv, int n_blocks, int D, int bits,
                                    void* k, int64_t k_stride_b, int64_t k_stride_h, int64_t k_stride_t,
                                    void* v, int64_t v_stride_b, int64_t v_stride_h, int64_t v_stride_t,
                                    void* stream) {
  HALO_CHECK_ARG(k && v && blocks, "null pointer");
  HALO_CHECK_ARG(dtype == HALO_F16 || dtype == HALO_BF16, "KIVI storage dtype must be fp16 or bf16");
  HALO_CHECK_ARG(bits == 2 || bits == 4 || bits == 8, "bits must be 2, 4 or 8");
  HALO_CHECK_ARG(D == 64 || D == 128 || D == 256, "head_dim must be 64, 128 or 256");
  HALO_CHECK_ARG(B >= 0 && H_kv > 0 && n_blocks >= 0, "bad sizes");
  const int64_t n = (int64_t)B * H_kv * n_blocks;
  if (n == 0) return HALO_OK;
  HALO_CHECK_ARG(n < (1ll << 31), "too many blocks");
  KiviDequantParams p{reinterpret_cast<const uint8_t*>(blocks), blk_stride_b, blk_stride_h, H_kv, n_blocks,
                      k, k_stride_b, k_stride_h, k_stride_t, v, v_stride_b, v_stride_h, v_stride_t};
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  if (dtype == HALO_F16) {
    if (D == 64) return dequant_bits<HALO_F16, 64>(p, bits, (int)n, st);
    if (D == 128) return dequant_bits<HALO_F16, 128>(p, bits, (int)n, st);
    return dequant_bits<HALO_F16, 256>(p, bits, (int)n, st);
  }
  if (D == 64) return dequant_bits<HALO_BF16, 64>(p, bits, (int)n, st);
  if (D == 128) return dequant_bits<HALO_BF16, 128>(p, bits, (int)n, st);
  return dequant_bits<HALO_BF16, 256>(p, bits, (int)n, st);
}
