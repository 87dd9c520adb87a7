// Chunked causal prefill attention on CDNA4 bf16/fp16 MFMA (gfx950, wave64).
//
// Reference semantics: HALOCacheChunked._chunk_attention + _lse_merge
// (halo/kv_cache_chunked.py:194-276) walked over the chunk list, i.e. for
// every query row the softmax over all attended key rows of all chunks, with
// the causal rule chunk_start + t <= q_start + i (halo/triton_chunked.py:
// 114-119).  The per-chunk partials of the reference merge associatively by
// log-sum-exp, so one online-softmax pass over the whole chunk list gives the
// same (out, lse).
//
// Work split: the query rows of one KV head's group are flattened position-
// major, row r = (position r / rep, head r % rep), and one workgroup (8 waves)
// takes 256 consecutive flattened rows, so every K/V tile staged in LDS serves
// all query heads of the group.  Each wave owns 32 rows = the 32 columns of
// v_mfma_f32_32x32x16; a lane owns one query row, so the running max and sum
// are per-lane scalars.
//   scores  S^T[key][q]  = sum_d K[key][d] Q[q][d]          (A = K tile, B = Q^T)
//   output  O^T[d][q]   += sum_key V^T[d][key] P^T[key][q]   (A = V^T, B = P^T)
// S^T's accumulator gives lane (q, half h) the keys 8i + 4h + j of a 32-key
// block; the PV step over 16 keys takes, per lane half, the keys
// {4h + j, 8 + 4h + j} of a 16-key run, so P^T is packed from the score
// registers without any cross-lane move, and V^T is read with
// ds_read_b64_tr_b16 in the same key order.  The output's MFMA row m of
// d-block db is d = (m / 16) * D/2 + 16 db + m % 16, which spreads one
// transposed read over the whole 256-byte bank window (with the row swizzles
// below, every LDS read of the loop is bank-conflict free).
//
// Pipeline: K tiles are staged two tiles ahead and V tiles one ahead
// (LDS-DMA, each lane choosing the global piece that lands in its slot, which
// lays out the swizzles), so one barrier per 64-key tile suffices, and the
// score MFMAs of tile t+1 are issued in the same basic block as the softmax of
// tile t, which lets the matrix core and the VALU overlap within a wave.
// Workgroups of one KV group run on one XCD (they share its L2), the ones with
// the longest causal extent first.
//
// Calls whose rows give fewer workgroups than CUs, or a last round of few,
// leave the chip idle (512 rows x 32/8 heads: 64 of 256; the time is that of
// one workgroup's walk over all keys).  There the walk is cut into n_split runs
// of key tiles, one workgroup each, and prefill_merge_kernel folds the fp32
// partials (halo_prefill_splits holds the rule).  Per call, kernels only, bf16:
//   512 rows over 8192 + 512 keys, 32/8 x 128:    238.6 us -> 90.4 us (4 splits)
//   64 rows over 8192 + 64 keys, 32/8 x 128:      214.7 us -> 33.5 us (22)
//   2 x 137 rows over 3000 + 137, 16/4 x 64, f16:  66.7 us -> 24.0 us (10)
//   2304 rows over 32768 + 2304, 32/8 x 128 (288 workgroups): 1898 us -> 1273 (6)
// The partials cost 2 x 4 bytes of traffic and 4 of workspace per output
// element and split, which is what ends the cutting: the first in the rule's
// model, the second by kPfMaxPartials.

#include <type_traits>

#include "common.hpp"

namespace halo {

namespace {

typedef __attribute__((ext_vector_type(16))) float pf32x16;

template <int DT>
struct PMfma;
template <>
struct PMfma<HALO_BF16> {
  typedef __attribute__((ext_vector_type(8))) __bf16 v8;
  __device__ static __forceinline__ pf32x16 run(const uint4& a, const uint4& b, pf32x16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(v8, a), __builtin_bit_cast(v8, b), c, 0, 0, 0);
  }
  __device__ static __forceinline__ uint32_t pack(float a, float b) {
    typedef __attribute__((ext_vector_type(2))) __bf16 b2;
    const b2 v = {(__bf16)a, (__bf16)b};  // round to nearest even
    return __builtin_bit_cast(uint32_t, v);
  }
};
template <>
struct PMfma<HALO_F16> {
  typedef __attribute__((ext_vector_type(8))) _Float16 v8;
  __device__ static __forceinline__ pf32x16 run(const uint4& a, const uint4& b, pf32x16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(v8, a), __builtin_bit_cast(v8, b), c, 0, 0, 0);
  }
  __device__ static __forceinline__ uint32_t pack(float a, float b) {
    typedef __attribute__((ext_vector_type(2))) _Float16 h2;
    const h2 v = {(_Float16)a, (_Float16)b};  // round to nearest even
    return __builtin_bit_cast(uint32_t, v);
  }
};

__device__ __forceinline__ __amdgpu_buffer_rsrc_t prsrc(const char* base, int64_t bytes) {
  const int nrec = bytes <= 0 ? 0 : (bytes > 0x7fffffffLL ? 0x7fffffff : (int)bytes);
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<char*>(base), 0, nrec, 0x00020000);
}

template <typename T>
__device__ __forceinline__ T uni(T v) {
  return __builtin_amdgcn_readfirstlane(v);
}
__device__ __forceinline__ int64_t uni64(int64_t v) {
  const uint64_t u = (uint64_t)v;
  return (int64_t)(((uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)(u >> 32)) << 32) |
                   (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)u));
}
__device__ __forceinline__ const char* uniptr(const void* p) {
  return reinterpret_cast<const char*>((uintptr_t)uni64((int64_t)(uintptr_t)p));
}

// value of lane l ^ 32 next to the own value: {lanes 0-31 of v, lanes 32-63 of v}
__device__ __forceinline__ float half_max(float v) {
  const auto s = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return fmaxf(__uint_as_float(s[0]), __uint_as_float(s[1]));
}
__device__ __forceinline__ float half_sum(float v) {
  const auto s = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return __uint_as_float(s[0]) + __uint_as_float(s[1]);
}

// ds_read_b64_tr_b16: within each 16-lane group, lane i receives element i%4
// of the 8-byte reads of lanes 4e + i/4 (e = 0..3).
typedef short pv4i16_t __attribute__((ext_vector_type(4)));
__device__ __forceinline__ uint2 pf_tr16(const char* p) {
  const pv4i16_t r = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
      (__attribute__((address_space(3))) pv4i16_t*)(__attribute__((address_space(3))) char*)(p));
  return __builtin_bit_cast(uint2, r);
}

}  // namespace

struct PrefillParams {
  const void* q;
  int64_t q_stride_b, q_stride_h, q_stride_t;
  int B, H, H_kv, rep, T_q, n_wg, n_units;
  const int64_t* q_start;  // [B] global position of query row 0
  const halo_chunk_desc* descs;
  int n_desc;
  float scale2;
  void* out;
  int64_t o_stride_b, o_stride_h, o_stride_t;
  int out_dtype, out_vec4;
  float* lse;  // (B, H, T_q) contiguous, or null
  // split walk (n_split > 1): the partials of (split, unit, wave), see PfPart
  int n_split;
  float4* part_o;
  float2* part_ml;
};

constexpr int kPfNW = 8;             // waves per workgroup
constexpr int kPfRows = kPfNW * 32;  // flattened query rows per workgroup
constexpr int kPfBK = 64;            // key rows per LDS tile
// Slack (log2 units) by which a tile's max may exceed the running max before
// the running max moves: probabilities stay below 2^8 and the accumulators are
// rescaled only when the max really moves; out = o / l and lse = m + log2(l)
// use the same m, so the result does not depend on when m moved.
constexpr float kPfLazyMax = 8.0f;

// 16-byte piece swizzles of a staged row (RB = row bytes).  K: the 16 rows of
// one b128 read pass land on distinct banks.  V: the 4 rows x 2 d-halves of
// one transposed read pass land on distinct 32-byte bank windows.
template <int RB>
__device__ __forceinline__ int pf_kswz(int r) {
  return RB == 256 ? (r & 15) : ((r >> 1) & 7);
}
template <int RB>
__device__ __forceinline__ int pf_vswz(int r) {
  return RB == 256 ? 2 * (r & 3) : 2 * ((r >> 1) & 1);
}

// One chunk tile of the walk, all fields wave-uniform.
struct PfTile {
  const char* kb;  // K rows of this (batch, KV head), row 0 of the chunk
  const char* vb;
  int64_t kst, vst;  // row strides in bytes
  int64_t cstart;
  int ci, kt, rows, causal;
  bool valid;
};

// Workgroup order shared by the attention and the merge launch: XCD-aware
// (blockIdx % 8), a contiguous run of (KV group, split, workgroup) per XCD, so
// the workgroups that read the same K/V rows share an L2; within a group the
// workgroups with the most keys start first.
struct PfUnit {
  int unit, split, grp, wg;
};
__device__ __forceinline__ PfUnit pf_unit(const PrefillParams& P, int blk) {
  const int n = P.n_units * P.n_split;
  int u = blk;
  if ((n & 7) == 0) u = (blk & 7) * (n >> 3) + (blk >> 3);
  PfUnit r;
  const int per = P.n_wg * P.n_split;
  r.grp = u / per;
  const int x = u - r.grp * per;
  r.split = x / P.n_wg;
  r.wg = P.n_wg - 1 - (x - r.split * P.n_wg);
  r.unit = r.grp * P.n_wg + r.wg;
  return r;
}

// Partial of one wave of a split unit, in the wave's own register order so
// that every store and load is 1 KiB of consecutive bytes: piece x = 4 db + i
// of lane l is the float4 at ((split * n_units + unit) * waves + wave) * PIECES
// * 64 + x * 64 + l, its (m, l) pair at (...) * 32 + row.
template <int NW>
__device__ __forceinline__ int64_t pf_part(const PrefillParams& P, int split, int unit, int wave) {
  return ((int64_t)split * P.n_units + unit) * NW + wave;
}

// Where split `split` of n_split starts in the walk of batch row `b` (keys up
// to `qmax`), and how many tiles it takes: lane l reads descriptor c0 + l, so
// the whole table costs one memory round trip per 64 chunks and not one per
// chunk.  Every lane returns the same values.
__device__ __forceinline__ void pf_split_range(const halo_chunk_desc* descs, int n_desc, int b, int64_t qmax, int tile,
                                               int split, int n_split, int& chunk, int& kt, int& n) {
  const int lane = threadIdx.x & 63;
  auto scan = [&](int c0, int& mine) {  // inclusive prefix of the tile counts of chunks [c0, c0 + 64)
    mine = 0;
    if (c0 + lane < n_desc) {
      const halo_chunk_desc* d = descs + c0 + lane;
      if (d->batch < 0 || d->batch == b) {
        int64_t rows = d->T_c;
        if (d->flags & HALO_CHUNK_CAUSAL) rows = min<int64_t>(rows, qmax - d->chunk_start + 1);
        if (rows > 0) mine = (int)((rows + tile - 1) / tile);
      }
    }
    int x = mine;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
      const int y = __shfl_up(x, off, 64);
      if (lane >= off) x += y;
    }
    return x;
  };
  int total = 0, mine;
  for (int c0 = 0; c0 < n_desc; c0 += 64) total += __shfl(scan(c0, mine), 63, 64);
  const int t0 = uni((int)((int64_t)total * split / n_split));
  n = uni((int)((int64_t)total * (split + 1) / n_split)) - t0;
  chunk = n_desc;
  kt = 0;
  int base = 0;
  for (int c0 = 0; n > 0 && c0 < n_desc; c0 += 64) {
    const int x = base + scan(c0, mine);
    const uint64_t past = __ballot(x > t0);
    if (past != 0) {
      const int at = __builtin_ctzll(past);
      chunk = uni(c0 + at);
      kt = uni((t0 - (__shfl(x, at, 64) - __shfl(mine, at, 64))) * tile);
      return;
    }
    base = __shfl(x, 63, 64);
  }
}

// First channel of the four that piece x = 4 db + i of lane half hh holds.
// 16-bit kernel: MFMA row m of d-block db is channel (m / 16) D/2 + 16 db + m % 16.
template <int D>
struct PfRowsTr {
  __device__ static __forceinline__ int first(int x, int hh) {
    const int db = x >> 2, m = 8 * (x & 3) + 4 * hh;
    return (m >> 4) * (D / 2) + 16 * db + (m & 15);
  }
};
// fp32 kernel: row m of block db is channel m D/32 + db; piece x = i D/32 + g
// holds channels 4 g .. 4 g + 3 of the 4 D/32 consecutive ones of rows 8 i + 4 hh + {0..3}.
template <int D>
struct PfRowsF32 {
  __device__ static __forceinline__ int first(int x, int hh) {
    constexpr int DB = D / 32;
    return (8 * (x / DB) + 4 * hh) * DB + 4 * (x % DB);
  }
};

__device__ __forceinline__ void pf_store4(const PrefillParams& P, int64_t at, const float* v4) {
  if (P.out_vec4) {
    store_elem4(P.out, at, P.out_dtype, v4);
  } else {
#pragma unroll
    for (int j = 0; j < 4; ++j) store_elem(P.out, at + j, P.out_dtype, v4[j]);
  }
}

// The first chunk at or after `from` with rows for this (batch row, KV head) and keys up to `qmax`.
template <int ESZ>
__device__ __forceinline__ void pf_open_chunk(const PrefillParams& P, int b, int h_kv, int64_t qmax, int from,
                                              PfTile& t) {
  t.valid = false;
  for (int c = uni(from); c < P.n_desc; ++c) {
    const halo_chunk_desc* dp = P.descs + c;
    const int batch = uni(dp->batch);
    if (batch >= 0 && batch != b) continue;
    const int causal = uni(dp->flags) & HALO_CHUNK_CAUSAL;
    const int64_t cstart = uni64(dp->chunk_start);
    int rows = uni(dp->T_c);
    if (causal) rows = (int)max<int64_t>(0, min<int64_t>(rows, qmax - cstart + 1));
    if (rows <= 0) continue;
    const int64_t ksb = uni64(dp->k_stride_b), ksh = uni64(dp->k_stride_h);
    const int64_t vsb = uni64(dp->v_stride_b), vsh = uni64(dp->v_stride_h);
    t.kb = uniptr(dp->k) + ((batch < 0 ? (int64_t)b * ksb : 0) + (int64_t)h_kv * ksh) * ESZ;
    t.vb = uniptr(dp->v) + ((batch < 0 ? (int64_t)b * vsb : 0) + (int64_t)h_kv * vsh) * ESZ;
    t.kst = uni64(dp->k_stride_t) * ESZ;
    t.vst = uni64(dp->v_stride_t) * ESZ;
    t.cstart = cstart;
    t.rows = rows;
    t.kt = 0;
    t.causal = causal;
    t.ci = c;
    t.valid = true;
    return;
  }
}

template <int DT, int D, bool SPLIT>
__global__ void __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(2, 2))) prefill_attn_kernel(PrefillParams P) {
  constexpr int KS = D / 16;               // d-steps of the score MFMA
  constexpr int DB = D / 32;               // d-blocks of the output MFMA
  constexpr int RB = D * 2;                // row bytes
  constexpr int SL = RB / 16;              // 16-byte pieces per row
  constexpr int TB = kPfBK * RB;           // one K or V tile in LDS
  constexpr int RPI = 1024 / RB;           // rows per 1 KiB LDS-DMA instruction
  constexpr int BPW = TB / 1024 / kPfNW;   // 1 KiB DMA blocks per wave per tile
  static_assert(BPW >= 1 && TB % (1024 * kPfNW) == 0, "prefill tile shape");
  // K stages 0/1 and V stages 0/1 as four LDS objects: the stage a step
  // reads is a compile-time constant in each of the two unrolled steps, so
  // the compiler can tell the tiles being filled by LDS-DMA from the ones
  // being read and does not wait for the fills before every read
  __shared__ __attribute__((aligned(16))) char sK0[TB], sK1[TB], sV0[TB], sV1[TB];

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = uni(tid >> 6);
  const int qc = lane & 31, hh = lane >> 5;

  const PfUnit un = pf_unit(P, blockIdx.x);
  const int grp = un.grp, wg = un.wg;
  const int b = grp / P.H_kv, h_kv = grp % P.H_kv;
  const int RG = P.T_q * P.rep;  // flattened rows of the group
  const int wrow0 = wg * kPfRows;
  const int64_t qs = P.q_start[b];
  const int64_t wg_qmax = qs + (min(wrow0 + kPfRows, RG) - 1) / P.rep;
  const int64_t wave_qmin = qs + min(wrow0 + wave * 32, RG - 1) / P.rep;

  // this lane's query row
  const int r_lane = wrow0 + wave * 32 + qc;
  const bool row_ok = r_lane < RG;
  const int r_eff = row_ok ? r_lane : RG - 1;
  const int pos = r_eff / P.rep;
  const int h = h_kv * P.rep + (r_eff - pos * P.rep);
  const int64_t qpos = qs + pos;

  // Q^T as B operands: lane (q, half) holds d = 16 s + 8 half .. +8
  uint4 qb[KS];
  {
    const char* qrow = reinterpret_cast<const char*>(P.q) +
                       ((int64_t)b * P.q_stride_b + (int64_t)h * P.q_stride_h + (int64_t)pos * P.q_stride_t) * 2;
#pragma unroll
    for (int s = 0; s < KS; ++s) qb[s] = *reinterpret_cast<const uint4*>(qrow + (s * 16 + hh * 8) * 2);
  }

  // ---- the (chunk, 64-row tile) walk
  auto open_chunk = [&](int from, PfTile& t) { pf_open_chunk<2>(P, b, h_kv, wg_qmax, from, t); };
  int left = 0;  // tiles from the furthest cursor to the end of this split, itself included
  auto next_tile = [&](PfTile& t) {
    if (!t.valid) return;
    if constexpr (SPLIT) {
      if (--left <= 0) {
        t.valid = false;
        return;
      }
    }
    t.kt += kPfBK;
    if (t.kt >= t.rows) open_chunk(t.ci + 1, t);
  };
  // LDS-DMA of one tile's K (or V) rows [kt, kt+64) into `st`: each 1 KiB
  // instruction of a wave fills RPI consecutive rows, lane l the 16-byte slot
  // l % SL of row l / SL, reading the global piece that belongs there.  Rows
  // past the chunk read as zeros (buffer range check).
  auto issue = [&](const char* base, int64_t rst, int kt, int rows, char* st, bool is_v) {
    const __amdgpu_buffer_rsrc_t rs = prsrc(base + (int64_t)kt * rst, (int64_t)(rows - kt) * rst);
#pragma unroll
    for (int j = 0; j < BPW; ++j) {
      const int blk = wave * BPW + j;
      const int r = blk * RPI + lane / SL, slot = lane % SL;
      const int piece = slot ^ (is_v ? pf_vswz<RB>(r) : pf_kswz<RB>(r));
      const int off = (int)(r * rst) + (piece << 4);
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (__attribute__((address_space(3))) void*)(st + blk * 1024), 16,
                                               off, 0, 0, 0);
    }
  };

  // LDS operand reads.  K (A of the score MFMA): step i = (d-step i/2, key
  // block i%2).  V^T (A of the PV MFMA): step i = (key step i/DB, d-block
  // i%DB), two transposed reads.
  auto kread = [&](const char* sk, int i) -> uint4 {
    const int kr = (i & 1) * 32 + qc;
    return *reinterpret_cast<const uint4*>(sk + kr * RB + (((2 * (i >> 1) + hh) ^ pf_kswz<RB>(kr)) << 4));
  };
  const int vG = lane >> 4, vei = (lane & 15) >> 2, vai = lane & 3;
  auto vread = [&](const char* sv, int i) -> uint4 {
    const int t = i / DB, db = i % DB;
    const int rlo = 16 * t + 4 * (vG >> 1) + vei, rhi = rlo + 8;
    const int byte = ((vG & 1) * (D / 2) + 16 * db + 4 * vai) * 2;
    const int pc = byte >> 4, wi = byte & 15;
    const uint2 a0 = pf_tr16(sv + rlo * RB + ((pc ^ pf_vswz<RB>(rlo)) << 4) + wi);
    const uint2 a1 = pf_tr16(sv + rhi * RB + ((pc ^ pf_vswz<RB>(rhi)) << 4) + wi);
    return make_uint4(a0.x, a0.y, a1.x, a1.y);
  };
  constexpr int NKS = 2 * KS;  // score MFMAs per tile
  constexpr int NPV = 4 * DB;  // PV MFMAs per tile
  constexpr int RING = 4;      // operand reads in flight ahead of their MFMA
  // scores of one staged K tile (prologue only; the loop interleaves them)
  auto scores = [&](const char* sk, pf32x16* S) {
#pragma unroll
    for (int i = 0; i < NKS; ++i) S[i & 1] = PMfma<DT>::run(kread(sk, i), qb[i >> 1], i < 2 ? pf32x16{} : S[i & 1]);
  };

  pf32x16 o[DB];
#pragma unroll
  for (int db = 0; db < DB; ++db) o[db] = pf32x16{};
  float m_run = -INFINITY, l_run = 0.f;

  PfTile c0, c1, c2;
  if constexpr (SPLIT) {
    int chunk, kt;
    pf_split_range(P.descs, P.n_desc, b, wg_qmax, kPfBK, un.split, P.n_split, chunk, kt, left);
    open_chunk(chunk, c0);
    c0.kt = kt;
  } else {
    open_chunk(0, c0);
  }
  c1 = c0;
  next_tile(c1);
  c2 = c1;
  next_tile(c2);
  if (c0.valid) {
    issue(c0.kb, c0.kst, c0.kt, c0.rows, sK0, false);
    issue(c0.vb, c0.vst, c0.kt, c0.rows, sV0, true);
  }
  if (c1.valid) issue(c1.kb, c1.kst, c1.kt, c1.rows, sK1, false);
  __builtin_amdgcn_s_waitcnt(0);
  __syncthreads();

  // Masks tile `c`'s scores: keys at or past `lim` (tile-relative) for this
  // lane are the chunk end, and for a causal chunk the lane's own position.
  auto mask_tile = [&](const PfTile& c, pf32x16* S) {
    const bool masked = c.kt + kPfBK > c.rows || (c.causal && c.cstart + c.kt + kPfBK - 1 > wave_qmin);
    if (masked) {
      int lim = min(c.rows - c.kt, kPfBK);
      if (c.causal) {
        const int64_t dq = qpos - (c.cstart + c.kt) + 1;  // keys this lane may see
        lim = dq < (int64_t)lim ? (int)max<int64_t>(dq, -1) : lim;
      }
      lim -= 4 * hh;
#pragma unroll
      for (int kb = 0; kb < 2; ++kb)
#pragma unroll
        for (int e = 0; e < 16; ++e)
          S[kb][e] = (kb * 32 + 8 * (e >> 2) + (e & 3)) < lim ? S[kb][e] : -INFINITY;
    }
  };
  // The running max takes tile S's max into account (it moves only when the
  // tile's max exceeds it by the slack); returns whether it moved.
  float ms = 0.f;  // exponent offset of the current tile: m_run, or 0 while m_run is -inf
  auto tile_max = [](const pf32x16* S) -> float {
    float bm = -INFINITY;
#pragma unroll
    for (int kb = 0; kb < 2; ++kb)
#pragma unroll
      for (int e = 0; e < 16; ++e) bm = fmaxf(bm, S[kb][e]);
    return bm;
  };
  auto take_max = [&](float bm, float& m_old) -> bool {
    bm = half_max(bm);
    const float bms = bm * P.scale2;  // scores scale after the max (scale > 0)
    m_old = m_run;
    const float m_new = (bms > m_old + kPfLazyMax) ? bms : m_old;
    m_run = m_new;
    ms = (m_new == -INFINITY) ? 0.f : m_new;
    return m_new != m_old;
  };

  pf32x16 S[2];
  if (c0.valid) {
    scores(sK0, S);
    mask_tile(c0, S);
    float m_old;
    take_max(tile_max(S), m_old);  // o and l are still zero: nothing to rescale
  }
  __syncthreads();  // K stage 0 is refilled below

  // One 64-key tile t (its scores S masked, the running max already updated
  // for it): stage K(t+2) and V(t+1); block 1 = score MFMAs of tile t+1 with
  // the exponentials of tile t between them; mask tile t+1 if it crosses a
  // chunk end or the diagonal (rare); block 2 = O += V(t) P(t) with tile
  // t+1's max between the MFMAs; rescale O and l if the max moved (rare).
  // The loop alternates the roles of the two score arrays instead of copying.
  auto step = [&](auto stage_c, pf32x16* S, pf32x16* Sn) {
    constexpr int stage = decltype(stage_c)::value;
    char* const kcur = stage ? sK1 : sK0;  // K(t), scored; receives K(t+2)
    char* const knxt = stage ? sK0 : sK1;  // K(t+1); stale past the last tile, never used then
    char* const vcur = stage ? sV1 : sV0;  // V(t)
    char* const vnxt = stage ? sV0 : sV1;  // receives V(t+1)
    if (c2.valid) issue(c2.kb, c2.kst, c2.kt, c2.rows, kcur, false);
    if (c1.valid) issue(c1.vb, c1.vst, c1.kt, c1.rows, vnxt, true);

    // Both blocks are issued in source order (a scheduling barrier after
    // each MFMA step): every MFMA's operand was read RING steps earlier, and
    // the VALU work is spread evenly between the MFMAs.
    uint4 kr[RING], vr[RING];
#pragma unroll
    for (int i = 0; i < RING; ++i) kr[i] = kread(knxt, i);
    // P^T operands: key step 2 kb + u holds keys 16u + {4h + j, 8 + 4h + j} of block kb
    constexpr int EPM = 32 / NKS;  // exponentials per score MFMA
    uint4 pb[4];
    float p[8];
    float psum = 0.f;
#pragma unroll
    for (int i = 0; i < NKS; ++i) {
      Sn[i & 1] = PMfma<DT>::run(kr[i % RING], qb[i >> 1], i < 2 ? pf32x16{} : Sn[i & 1]);
      if (i + RING < NKS) kr[i % RING] = kread(knxt, i + RING);
      const int st = (i * EPM) >> 3, kb = st >> 1, u = st & 1;
#pragma unroll
      for (int x = 0; x < EPM; ++x) {
        const int e = (i * EPM + x) & 7;
        p[e] = __builtin_amdgcn_exp2f(__builtin_fmaf(S[kb][8 * u + e], P.scale2, -ms));
        psum += p[e];
      }
      // keeps the row sum's additions next to their exponentials (sunk
      // below the block they form one serial chain with the matrix pipe idle)
      asm volatile("" : "+v"(psum));
      if (((i + 1) * EPM & 7) == 0) {
        pb[st] = make_uint4(PMfma<DT>::pack(p[0], p[1]), PMfma<DT>::pack(p[2], p[3]), PMfma<DT>::pack(p[4], p[5]),
                            PMfma<DT>::pack(p[6], p[7]));
        // keeps the exponentials here (they would otherwise sink to block 2)
        asm volatile("" : "+v"(pb[st].x), "+v"(pb[st].y), "+v"(pb[st].z), "+v"(pb[st].w));
      }
      __builtin_amdgcn_sched_barrier(0);
    }
    l_run += psum;
    if (c1.valid) mask_tile(c1, Sn);

    // block 2: O += V(t) P(t), with tile t+1's max between the MFMAs
    constexpr int MPM = 32 / NPV;  // score elements folded into the max per PV MFMA
    float bm = -INFINITY;
#pragma unroll
    for (int i = 0; i < RING; ++i) vr[i] = vread(vcur, i);
#pragma unroll
    for (int i = 0; i < NPV; ++i) {
      o[i % DB] = PMfma<DT>::run(vr[i % RING], pb[i / DB], o[i % DB]);
      if (i + RING < NPV) vr[i % RING] = vread(vcur, i + RING);
#pragma unroll
      for (int x = 0; x < MPM; ++x) {
        const int e = i * MPM + x;
        bm = fmaxf(bm, Sn[e >> 4][e & 15]);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
    // past the last tile the scores came from a stale (or never filled)
    // stage: no max to take from them
    if (!c1.valid) bm = -INFINITY;
    float m_old;
    const bool moved = take_max(bm, m_old);
    if (__builtin_amdgcn_read_exec() & __ballot(moved)) {
      const float alpha = __builtin_amdgcn_exp2f(m_old - m_run);
      l_run *= alpha;
#pragma unroll
      for (int db = 0; db < DB; ++db) o[db] *= alpha;
    }
    __builtin_amdgcn_s_waitcnt(0);  // this wave's loads of K(t+2) and V(t+1) have landed
    __syncthreads();                // every wave's have; tile t's stages are free
    c0 = c1;
    c1 = c2;
    next_tile(c2);
  };
  pf32x16 S2[2];
  while (c0.valid) {
    step(std::integral_constant<int, 0>(), S, S2);
    if (!c0.valid) break;
    step(std::integral_constant<int, 1>(), S2, S);
  }

  // normalise and store: lane holds O^T[d][q] for MFMA rows m = 8i + 4h + j
  const float lt = half_sum(l_run);
  if constexpr (SPLIT) {
    const int64_t pw = pf_part<kPfNW>(P, un.split, un.unit, wave);
    float4* po = P.part_o + pw * (DB * 4 * 64) + lane;
#pragma unroll
    for (int db = 0; db < DB; ++db)
#pragma unroll
      for (int i = 0; i < 4; ++i)
        po[(db * 4 + i) * 64] = make_float4(o[db][4 * i], o[db][4 * i + 1], o[db][4 * i + 2], o[db][4 * i + 3]);
    if (hh == 0) P.part_ml[pw * 32 + qc] = make_float2(m_run, lt);
    return;
  }
  if (row_ok) {
    const float inv = lt > 0.f ? 1.f / lt : 0.f;
    const int64_t ob = (int64_t)b * P.o_stride_b + (int64_t)h * P.o_stride_h + (int64_t)pos * P.o_stride_t;
#pragma unroll
    for (int db = 0; db < DB; ++db)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        float v4[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) v4[j] = o[db][4 * i + j] * inv;
        pf_store4(P, ob + PfRowsTr<D>::first(4 * db + i, hh), v4);
      }
    if (P.lse != nullptr && hh == 0)
      P.lse[((int64_t)b * P.H + h) * P.T_q + pos] = lt > 0.f ? (m_run + log2f(lt)) * kLn2 : -INFINITY;
  }
}

// ---------------------------------------------------------------------------
// fp32 queries and chunks: the same walk on v_mfma_f32_32x32x2 (fp32 products
// and sums; error against 64 bits 3.3e-7, the VALU form had 3.3e-7).  Bound by the fp32 matrix
// rate (148 TFLOP/s reached by a large product); the row-per-query form this
// replaces read K/V once per query row and was planned on the host row by row.
// 512 rows over 1536 prior + 512 keys, 16/4 heads x 64: kernels 1318 us -> 59 us
// (attention 56 and 8-way merge 5 by themselves, 64 TFLOP/s), the call 7.2-8.0
// ms -> 70 us.
//
// One workgroup of 4 waves takes 128 flattened rows, a wave 32 of them (the
// columns); 32-key tiles (one MFMA block of keys: 64 cycles x (D/2 + D/2)
// MFMAs per tile leave the next tile's LDS-DMA time to land) are double
// buffered, one barrier per tile.  Step s of the score product multiplies
// channel s (lane half 0) and D/2 + s (half 1), so a lane reads its key row in
// 16-byte pieces; S^T's accumulator holds keys 8i + 4h + j, which are the two
// keys of step (i, j) of the output product, so the probabilities are that
// product's operand as they stand.  Output row m of block db is channel
// m D/32 + db: one read per key step gives a lane its operand of every block.
// ---------------------------------------------------------------------------
constexpr int kPf32NW = 4;
constexpr int kPf32Rows = kPf32NW * 32;
constexpr int kPf32BK = 32;

template <int D, bool SPLIT>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2)))
prefill_attn_f32_kernel(PrefillParams P) {
  constexpr int DB = D / 32;
  constexpr int RB = D * 4;                       // row bytes
  constexpr int SL = RB / 16;                     // 16-byte pieces per row
  constexpr int TB = kPf32BK * RB;                // one K or V tile in LDS
  constexpr int RPI = 1024 / RB;                  // rows per 1 KiB LDS-DMA instruction
  constexpr int BPW = TB / 1024 / kPf32NW;        // 1 KiB DMA blocks per wave per tile
  static_assert(BPW >= 1 && TB % (1024 * kPf32NW) == 0, "prefill tile shape");
  __shared__ __attribute__((aligned(16))) char sK0[TB], sK1[TB], sV0[TB], sV1[TB];

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = uni(tid >> 6);
  const int qc = lane & 31, hh = lane >> 5;
  const PfUnit un = pf_unit(P, blockIdx.x);
  const int b = un.grp / P.H_kv, h_kv = un.grp % P.H_kv;
  const int RG = P.T_q * P.rep;
  const int wrow0 = un.wg * kPf32Rows;
  const int64_t qs = P.q_start[b];
  const int64_t wg_qmax = qs + (min(wrow0 + kPf32Rows, RG) - 1) / P.rep;
  const int64_t wave_qmin = qs + min(wrow0 + wave * 32, RG - 1) / P.rep;
  const bool active = wrow0 + wave * 32 < RG;  // a wave past the rows only stages tiles

  const int r_lane = wrow0 + wave * 32 + qc;
  const bool row_ok = r_lane < RG;
  const int r_eff = row_ok ? r_lane : RG - 1;
  const int pos = r_eff / P.rep;
  const int h = h_kv * P.rep + (r_eff - pos * P.rep);
  const int64_t qpos = qs + pos;

  float qf[D / 2];  // channels hh D/2 + s
  {
    const float4* qrow = reinterpret_cast<const float4*>(
        reinterpret_cast<const float*>(P.q) + (int64_t)b * P.q_stride_b + (int64_t)h * P.q_stride_h +
        (int64_t)pos * P.q_stride_t + hh * (D / 2));
#pragma unroll
    for (int s = 0; s < D / 8; ++s) {
      const float4 x = qrow[s];
      qf[4 * s] = x.x;
      qf[4 * s + 1] = x.y;
      qf[4 * s + 2] = x.z;
      qf[4 * s + 3] = x.w;
    }
  }

  int left = 0;
  auto open_chunk = [&](int from, PfTile& t) { pf_open_chunk<4>(P, b, h_kv, wg_qmax, from, t); };
  auto next_tile = [&](PfTile& t) {
    if (!t.valid) return;
    if constexpr (SPLIT) {
      if (--left <= 0) {
        t.valid = false;
        return;
      }
    }
    t.kt += kPf32BK;
    if (t.kt >= t.rows) open_chunk(t.ci + 1, t);
  };
  // K pieces are swizzled (piece ^ row % 16: the 16 rows of a b128 read pass
  // land on distinct banks), V rows are read whole.  Rows past the chunk read
  // as zeros (buffer range check).
  auto issue = [&](const char* base, int64_t rst, int kt, int rows, char* st, bool is_v) {
    const __amdgpu_buffer_rsrc_t rs = prsrc(base + (int64_t)kt * rst, (int64_t)(rows - kt) * rst);
#pragma unroll
    for (int j = 0; j < BPW; ++j) {
      const int blk = wave * BPW + j;
      const int r = blk * RPI + lane / SL, slot = lane % SL;
      const int piece = is_v ? slot : slot ^ (r & 15);
      const int off = (int)(r * rst) + (piece << 4);
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (__attribute__((address_space(3))) void*)(st + blk * 1024), 16,
                                               off, 0, 0, 0);
    }
  };

  pf32x16 o[DB];
#pragma unroll
  for (int db = 0; db < DB; ++db) o[db] = pf32x16{};
  float m_run = -INFINITY, l_run = 0.f;

  PfTile c0, c1;
  if constexpr (SPLIT) {
    int chunk, kt;
    pf_split_range(P.descs, P.n_desc, b, wg_qmax, kPf32BK, un.split, P.n_split, chunk, kt, left);
    open_chunk(chunk, c0);
    c0.kt = kt;
  } else {
    open_chunk(0, c0);
  }
  c1 = c0;
  next_tile(c1);
  if (c0.valid) {
    issue(c0.kb, c0.kst, c0.kt, c0.rows, sK0, false);
    issue(c0.vb, c0.vst, c0.kt, c0.rows, sV0, true);
  }
  __builtin_amdgcn_s_waitcnt(0);
  __syncthreads();

  auto step = [&](auto stage_c) {
    constexpr int stage = decltype(stage_c)::value;
    const char* const sk = stage ? sK1 : sK0;
    const char* const sv = stage ? sV1 : sV0;
    if (c1.valid) {  // the other stage was last read before the barrier that ended the previous tile
      issue(c1.kb, c1.kst, c1.kt, c1.rows, stage ? sK0 : sK1, false);
      issue(c1.vb, c1.vst, c1.kt, c1.rows, stage ? sV0 : sV1, true);
    }
    if (active) {
      pf32x16 S = pf32x16{};
      // operand reads two steps (8 MFMAs, 512 cycles) ahead, in source order:
      // left alone the compiler reads a whole tile ahead and spills at D = 128
      int swz = (hh * (D / 8)) ^ (qc & 15);  // D / 8 is 8 or 16 and s below it: (hh D/8 + s) ^ x = s ^ swz
      asm volatile("" : "+v"(swz));          // one xor per read: the hoisted addresses would take D / 8 registers
      auto kread = [&](int s) { return *reinterpret_cast<const float4*>(sk + qc * RB + ((s ^ swz) << 4)); };
      float4 kk[2] = {kread(0), kread(1)};
#pragma unroll
      for (int s = 0; s < D / 8; ++s) {
        const float4 x = kk[s & 1];
        if (s + 2 < D / 8) kk[s & 1] = kread(s + 2);
        S = __builtin_amdgcn_mfma_f32_32x32x2f32(x.x, qf[4 * s], S, 0, 0, 0);
        S = __builtin_amdgcn_mfma_f32_32x32x2f32(x.y, qf[4 * s + 1], S, 0, 0, 0);
        S = __builtin_amdgcn_mfma_f32_32x32x2f32(x.z, qf[4 * s + 2], S, 0, 0, 0);
        S = __builtin_amdgcn_mfma_f32_32x32x2f32(x.w, qf[4 * s + 3], S, 0, 0, 0);
        __builtin_amdgcn_sched_barrier(0);
      }
      // tile-relative number of keys this lane's row sees
      int lim = min(c0.rows - c0.kt, kPf32BK);
      const bool diag = c0.causal && c0.cstart + c0.kt + kPf32BK - 1 > wave_qmin;
      if (diag) {
        const int64_t dq = qpos - (c0.cstart + c0.kt) + 1;
        lim = dq < (int64_t)lim ? (int)max<int64_t>(dq, 0) : lim;
      }
      if (diag || c0.kt + kPf32BK > c0.rows) {
        // the sign of the scale decides which infinity weighs nothing
        const float none = P.scale2 >= 0.f ? -INFINITY : INFINITY;
#pragma unroll
        for (int e = 0; e < 16; ++e) S[e] = 8 * (e >> 2) + (e & 3) + 4 * hh < lim ? S[e] : none;
      }
      float bm = -INFINITY;
#pragma unroll
      for (int e = 0; e < 16; ++e) bm = fmaxf(bm, S[e] * P.scale2);
      bm = half_max(bm);
      const float m_old = m_run;
      m_run = bm > m_old + kPfLazyMax ? bm : m_old;
      const float ms = m_run == -INFINITY ? 0.f : m_run;
      if (__ballot(m_run != m_old)) {
        const float alpha = m_run != m_old ? __builtin_amdgcn_exp2f(m_old - m_run) : 1.f;
        l_run *= alpha;
#pragma unroll
        for (int db = 0; db < DB; ++db) o[db] *= alpha;
      }
      float p[16];
      float ps[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        p[e] = __builtin_amdgcn_exp2f(__builtin_fmaf(S[e], P.scale2, -ms));
        ps[e & 3] += p[e];
      }
      l_run += (ps[0] + ps[1]) + (ps[2] + ps[3]);
      // A row in front of the diagonal has weight 0 for the keys behind it,
      // but 0 x inf is not 0: in a diagonal tile, values that are not finite
      // are kept out of the product and reach the rows that see them only.
      bool odd = false;
      if (diag) {
        bool bad = false;
        for (int x = lane; x < TB / 16; x += 64) {
          const float4 y = *reinterpret_cast<const float4*>(sv + x * 16);
          bad |= (y.x * 0.f + y.y * 0.f) + (y.z * 0.f + y.w * 0.f) != 0.f;  // inf x 0 and NaN x 0 are NaN
        }
        odd = __ballot(bad) != 0;
      }
      // A tile's products are summed by themselves and then added to O: with O
      // as the accumulator of every product its rounding error was 1.2 x the
      // row-by-row form's, with one addition per tile it is below it.
      constexpr int GB = DB == 2 ? 2 : 1;  // blocks at a time: more would spill at D = 128
      typedef __attribute__((ext_vector_type(GB))) float vrow;
      constexpr int VR = 8 / GB;  // rows read ahead: 8 MFMAs
#pragma unroll
      for (int b0 = 0; b0 < DB; b0 += GB) {
        auto vread = [&](int e) {
          return *reinterpret_cast<const vrow*>(sv + (8 * (e >> 2) + 4 * hh + (e & 3)) * RB + (qc * DB + b0) * 4);
        };
        vrow vv[VR];
#pragma unroll
        for (int e = 0; e < VR; ++e) vv[e] = vread(e);
        pf32x16 t[GB];
#pragma unroll
        for (int g = 0; g < GB; ++g) t[g] = pf32x16{};
#pragma unroll
        for (int e = 0; e < 16; ++e) {
          const vrow v = vv[e % VR];
          if (e + VR < 16) vv[e % VR] = vread(e + VR);
#pragma unroll
          for (int g = 0; g < GB; ++g) {
            const float x = odd && !(fabsf(v[g]) < INFINITY) ? 0.f : v[g];
            t[g] = __builtin_amdgcn_mfma_f32_32x32x2f32(x, p[e], t[g], 0, 0, 0);
          }
          __builtin_amdgcn_sched_barrier(0);
        }
#pragma unroll
        for (int g = 0; g < GB; ++g) o[b0 + g] += t[g];
      }
      if (odd) {
        // how many of +inf (or NaN), then of -inf (or NaN), each row sees in each channel
#pragma unroll
        for (int x = 0; x < 2 * DB; ++x) {
          const float inf = x & 1 ? -INFINITY : INFINITY;
          pf32x16 n = pf32x16{};
#pragma unroll
          for (int e = 0; e < 16; ++e) {
            const float v = *reinterpret_cast<const float*>(sv + (8 * (e >> 2) + 4 * hh + (e & 3)) * RB +
                                                            (qc * DB + (x >> 1)) * 4);
            const float sees = 8 * (e >> 2) + (e & 3) + 4 * hh < lim ? 1.f : 0.f;
            n = __builtin_amdgcn_mfma_f32_32x32x2f32(v == inf || v != v ? 1.f : 0.f, sees, n, 0, 0, 0);
            __builtin_amdgcn_sched_barrier(0);
          }
#pragma unroll
          for (int e = 0; e < 16; ++e) o[x >> 1][e] += n[e] > 0.f ? inf : 0.f;
        }
      }
    }
    __builtin_amdgcn_s_waitcnt(0);  // this wave's loads of the next tile have landed
    __syncthreads();                // every wave's have; this tile's stage is free
    c0 = c1;
    next_tile(c1);
  };
  while (c0.valid) {
    step(std::integral_constant<int, 0>());
    if (!c0.valid) break;
    step(std::integral_constant<int, 1>());
  }

  if (!active) return;
  // rows m = 8i + 4h + {0..3} are 4 DB consecutive channels: DB float4s
  const float lt = half_sum(l_run);
  float4 piece[4 * DB];
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int g = 0; g < DB; ++g) {
      float x[4];
#pragma unroll
      for (int y = 0; y < 4; ++y) {
        const int c = 4 * g + y;  // channel within the run: (j, db) = (c / DB, c % DB)
        x[y] = o[c % DB][4 * i + c / DB];
      }
      piece[i * DB + g] = make_float4(x[0], x[1], x[2], x[3]);
    }
  if constexpr (SPLIT) {
    const int64_t pw = pf_part<kPf32NW>(P, un.split, un.unit, wave);
    float4* po = P.part_o + pw * (DB * 4 * 64) + lane;
#pragma unroll
    for (int x = 0; x < 4 * DB; ++x) po[x * 64] = piece[x];
    if (hh == 0) P.part_ml[pw * 32 + qc] = make_float2(m_run, lt);
    return;
  }
  if (row_ok) {
    const float inv = lt > 0.f ? 1.f / lt : 0.f;
    const int64_t ob = (int64_t)b * P.o_stride_b + (int64_t)h * P.o_stride_h + (int64_t)pos * P.o_stride_t;
#pragma unroll
    for (int x = 0; x < 4 * DB; ++x) {
      const float v4[4] = {piece[x].x * inv, piece[x].y * inv, piece[x].z * inv, piece[x].w * inv};
      pf_store4(P, ob + PfRowsF32<D>::first(x, hh), v4);
    }
    if (P.lse != nullptr && hh == 0)
      P.lse[((int64_t)b * P.H + h) * P.T_q + pos] = lt > 0.f ? (m_run + log2f(lt)) * kLn2 : -INFINITY;
  }
}

// Merge of the n_split partials of every flattened query row: one wave per
// (unit, wave, 4 pieces), reading the partials in the order they were stored.
// With M the largest of the row's running maxima, out = sum_s 2^(m_s - M) o_s /
// sum_s 2^(m_s - M) l_s; a split without visible keys has m = -inf and weight 0.
// NW waves per workgroup of the attention launch, PM the placement of its output rows.
template <int D, int NW, class PM>
__global__ void __launch_bounds__(256) prefill_merge_kernel(PrefillParams P) {
  constexpr int PIECES = D / 8;  // float4 pieces of a lane
  constexpr int PPW = 4;         // of which a wave of this launch merges
  const int lane = threadIdx.x & 63;
  const int job = uni((int)(blockIdx.x * 4 + (threadIdx.x >> 6)));
  const int x0 = (job % (PIECES / PPW)) * PPW;
  const int wave = (job / (PIECES / PPW)) % NW;
  const int unit = job / (PIECES / PPW) / NW;
  if (unit >= P.n_units) return;
  const int grp = unit / P.n_wg, wg = unit - grp * P.n_wg;
  const int b = grp / P.H_kv, h_kv = grp % P.H_kv;
  const int qc = lane & 31, hh = lane >> 5;
  const int r = (wg * NW + wave) * 32 + qc;
  if (r >= P.T_q * P.rep) return;
  const int pos = r / P.rep;
  const int h = h_kv * P.rep + (r - pos * P.rep);

  float m = -INFINITY, l = 0.f;
  float4 acc[PPW];
#pragma unroll
  for (int x = 0; x < PPW; ++x) acc[x] = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll 4
  for (int s = 0; s < P.n_split; ++s) {
    const int64_t pw = pf_part<NW>(P, s, unit, wave);
    const float2 ml = P.part_ml[pw * 32 + qc];
    float4 v[PPW];
#pragma unroll
    for (int x = 0; x < PPW; ++x) v[x] = P.part_o[pw * (PIECES * 64) + (x0 + x) * 64 + lane];
    const float mn = fmaxf(m, ml.x);
    const float ms = mn == -INFINITY ? 0.f : mn;
    const float wo = __builtin_amdgcn_exp2f(m - ms), wn = __builtin_amdgcn_exp2f(ml.x - ms);
    m = mn;
    l = l * wo + ml.y * wn;
#pragma unroll
    for (int x = 0; x < PPW; ++x) {
      acc[x].x = __builtin_fmaf(v[x].x, wn, acc[x].x * wo);
      acc[x].y = __builtin_fmaf(v[x].y, wn, acc[x].y * wo);
      acc[x].z = __builtin_fmaf(v[x].z, wn, acc[x].z * wo);
      acc[x].w = __builtin_fmaf(v[x].w, wn, acc[x].w * wo);
    }
  }
  const float inv = l > 0.f ? 1.f / l : 0.f;
  const int64_t ob = (int64_t)b * P.o_stride_b + (int64_t)h * P.o_stride_h + (int64_t)pos * P.o_stride_t;
#pragma unroll
  for (int x = 0; x < PPW; ++x) {
    const int d = PM::first(x0 + x, hh);
    const float v4[4] = {acc[x].x * inv, acc[x].y * inv, acc[x].z * inv, acc[x].w * inv};
    pf_store4(P, ob + d, v4);
  }
  if (P.lse != nullptr && hh == 0 && x0 == 0)
    P.lse[((int64_t)b * P.H + h) * P.T_q + pos] = l > 0.f ? (m + log2f(l)) * kLn2 : -INFINITY;
}

}  // namespace halo

using namespace halo;

namespace {

int64_t prefill_units(int dtype, int B, int H, int H_kv, int T_q, int64_t* n_wg) {
  const int64_t rows = (int64_t)T_q * (H / H_kv);
  const int per = dtype == HALO_F32 ? kPf32Rows : kPfRows;
  *n_wg = (rows + per - 1) / per;
  return (int64_t)B * H_kv * *n_wg;
}

constexpr int kPfMaxSplit = 32;
// Partials of the splits that are chosen here.  A call without splits takes no
// workspace, so one that fits beside a large cache should not need much: 219 MiB
// give the 288 workgroups of 2304 rows over 32768 keys their 6 splits, and more
// workgroups need fewer (520 of 4100 rows: 2991 us unsplit, 2538 with the 3 that
// fit, 2411 with 6 in 396 MiB; 1056 of 8392 rows over 65536: 10.65 ms unsplit,
// which is all that fits, 9.29 with 5 in 670 MiB).
constexpr int64_t kPfMaxPartials = 256ll << 20;

// bytes of one wave's partial: 32 rows x D fp32 and 32 (m, l) pairs
int64_t prefill_part_bytes(int D) { return 32ll * D * 4 + 32 * 8; }

}  // namespace

// The number of key splits by a cost model of one call, in us: `rounds` of one
// 8-wave workgroup per CU, each `mean` tiles at the measured time of a 64-key
// tile (1.75 us at D = 128, 1.2 us at D = 64, every CU busy) plus prologue and
// epilogue, or the longest workgroup alone; a split call adds the merge launch
// and the partials written and read at 4 TB/s.  Against sweeps of 1 to 32
// splits over 28 shapes (8 to 8392 rows, 0 to 131072 prior keys, 64 to 2080
// units) the model's choice was the fastest or within 5 % of it, but for one
// (256 rows over 2048 keys 37.5 us for 35.6 us); the partials have to fit
// kPfMaxPartials.  fp32: 32-key tiles, 3.1 and 5.5 us with one 4-wave workgroup
// on a CU, 4.4 and 9.2 us each with two; fastest or within 3 % over 6 shapes
// (512 to 4100 rows, 2048 and 8192 keys).
extern "C" int halo_prefill_splits(int dtype, int B, int H, int H_kv, int T_q, int D, int64_t keys, int64_t causal_keys) {
  if (B <= 0 || H <= 0 || H_kv <= 0 || H % H_kv != 0 || T_q <= 0 || D <= 0 || keys <= 0) return 1;
  int64_t n_wg;
  const int64_t units = prefill_units(dtype, B, H, H_kv, T_q, &n_wg);
  const bool f32 = dtype == HALO_F32;
  const int bk = f32 ? kPf32BK : kPfBK, nw = f32 ? kPf32NW : kPfNW;
  const double fixed_us = 4.0;
  const double longest = (double)(keys + bk - 1) / bk;
  const int64_t tri = causal_keys < T_q ? causal_keys : T_q;
  const double mean = longest - 0.5 * (double)tri / bk;
  const int64_t part = units * nw * prefill_part_bytes(D);
  double best = 0;
  int best_s = 1;
  for (int s = 1; s <= kPfMaxSplit && s <= (int)longest && (s == 1 || s * part <= kPfMaxPartials); ++s) {
    const bool pairs = f32 && units * s > 256;  // fp32: two 4-wave workgroups per CU
    const int slots = pairs ? 512 : 256;
    const double tile_us = f32 ? (pairs ? (D == 128 ? 9.2 : 4.4) : (D == 128 ? 5.5 : 3.1)) : (D == 128 ? 1.75 : 1.2);
    const double rounds = (double)((units * s + slots - 1) / slots);
    const double chip = rounds * (mean / s * tile_us + fixed_us);
    const double one = std::ceil(longest / s) * tile_us + fixed_us;
    double us = chip > one ? chip : one;
    if (s > 1) us += 5.0 + (double)s * (double)part * 2.0 / 4.0e6;
    if (s == 1 || us < best) {
      best = us;
      best_s = s;
    }
  }
  return best_s;
}

extern "C" size_t halo_prefill_workspace_size(int dtype, int B, int H, int H_kv, int T_q, int D, int n_split) {
  if (B <= 0 || H <= 0 || H_kv <= 0 || H % H_kv != 0 || T_q <= 0 || D <= 0 || n_split <= 1) return 0;
  int64_t n_wg;
  const int64_t units = prefill_units(dtype, B, H, H_kv, T_q, &n_wg);
  const int nw = dtype == HALO_F32 ? kPf32NW : kPfNW;
  return (size_t)n_split * (size_t)units * nw * (size_t)prefill_part_bytes(D);
}

extern "C" int halo_prefill_attn_split(const void* q, int64_t q_stride_b, int64_t q_stride_h, int64_t q_stride_t,
                                       int dtype, int B, int H, int H_kv, int T_q, int D, const int64_t* q_start,
                                       const halo_chunk_desc* descs, int n_desc, float scale,
                                       void* out, int64_t out_stride_b, int64_t out_stride_h, int64_t out_stride_t,
                                       int out_dtype, float* lse, int n_split, void* workspace,
                                       size_t workspace_bytes, void* stream) {
  HALO_CHECK_ARG(q && q_start && descs && out, "null pointer argument");
  HALO_CHECK_ARG(dtype == HALO_BF16 || dtype == HALO_F16 || dtype == HALO_F32, "dtype must be bf16, f16 or f32");
  HALO_CHECK_ARG(out_dtype == HALO_F32 || out_dtype == HALO_BF16 || out_dtype == HALO_F16, "bad out_dtype");
  HALO_CHECK_ARG(B > 0 && H > 0 && H_kv > 0 && H % H_kv == 0 && T_q >= 0, "need H % H_kv == 0 and positive sizes");
  HALO_CHECK_ARG(D == 64 || D == 128, "head_dim must be 64 or 128");
  HALO_CHECK_ARG(n_desc >= 0, "bad chunk count");
  const int64_t esz = elem_size(dtype);
  HALO_CHECK_ARG(reinterpret_cast<uintptr_t>(q) % 16 == 0 && (q_stride_t * esz) % 16 == 0 &&
                     (q_stride_h * esz) % 16 == 0 && (q_stride_b * esz) % 16 == 0,
                 "q rows must be 16-byte aligned");
  HALO_CHECK_ARG(n_split >= 1 && n_split <= kPfMaxSplit, "n_split must be in [1, 32]");
  if (T_q == 0) return HALO_OK;
  const size_t ws_need = halo_prefill_workspace_size(dtype, B, H, H_kv, T_q, D, n_split);
  HALO_CHECK_ARG(ws_need == 0 || (workspace != nullptr && workspace_bytes >= ws_need &&
                                  reinterpret_cast<uintptr_t>(workspace) % 16 == 0),
                 "workspace missing, too small or not 16-byte aligned");
  PrefillParams p;
  p.q = q;
  p.q_stride_b = q_stride_b;
  p.q_stride_h = q_stride_h;
  p.q_stride_t = q_stride_t;
  p.B = B;
  p.H = H;
  p.H_kv = H_kv;
  p.rep = H / H_kv;
  p.T_q = T_q;
  const int64_t rows = (int64_t)T_q * p.rep;
  int64_t n_wg;
  const int64_t units = prefill_units(dtype, B, H, H_kv, T_q, &n_wg);
  const int nw = dtype == HALO_F32 ? kPf32NW : kPfNW;
  p.n_wg = (int)n_wg;
  HALO_CHECK_ARG(rows < (1ll << 31) && units * n_split < (1ll << 31) &&
                     (n_split == 1 || units * nw * (D / 32) < (1ll << 31)),
                 "too many query rows");
  p.n_split = n_split;
  p.part_o = reinterpret_cast<float4*>(workspace);
  p.part_ml = reinterpret_cast<float2*>(p.part_o + (n_split > 1 ? units * nw * n_split * (D / 8) * 64 : 0));
  p.n_units = (int)units;
  p.q_start = q_start;
  p.descs = descs;
  p.n_desc = n_desc;
  p.scale2 = (float)((double)scale * 1.4426950408889634);
  // a masked score is an infinity times the scale: a zero scale would make it NaN.
  // The smallest subnormal, 2^-149, leaves scores below 2^125 at 2^0 and the fp32
  // maximum within 3.3e-7 of it
  if (dtype == HALO_F32 && p.scale2 == 0.f) p.scale2 = 0x1p-149f;
  p.out = out;
  p.o_stride_b = out_stride_b;
  p.o_stride_h = out_stride_h;
  p.o_stride_t = out_stride_t;
  p.out_dtype = out_dtype;
  // 4-element stores need every row start aligned to 4 elements' bytes
  const int64_t ea = out_dtype == HALO_F32 ? 16 : 8;
  const int64_t es = elem_size(out_dtype);
  p.out_vec4 = reinterpret_cast<uintptr_t>(out) % ea == 0 && (out_stride_b * es) % ea == 0 &&
               (out_stride_h * es) % ea == 0 && (out_stride_t * es) % ea == 0;
  p.lse = lse;
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  const dim3 grid((unsigned)(units * n_split)), block(nw * 64);
  if (dtype == HALO_F32) {
    if (n_split > 1) {
      if (D == 128) hipLaunchKernelGGL((prefill_attn_f32_kernel<128, true>), grid, block, 0, st, p);
      else hipLaunchKernelGGL((prefill_attn_f32_kernel<64, true>), grid, block, 0, st, p);
    } else {
      if (D == 128) hipLaunchKernelGGL((prefill_attn_f32_kernel<128, false>), grid, block, 0, st, p);
      else hipLaunchKernelGGL((prefill_attn_f32_kernel<64, false>), grid, block, 0, st, p);
    }
  }
#define HALO_PREFILL(DTV, DV)                                                                        \
  do {                                                                                               \
    if (n_split > 1) hipLaunchKernelGGL((prefill_attn_kernel<DTV, DV, true>), grid, block, 0, st, p); \
    else hipLaunchKernelGGL((prefill_attn_kernel<DTV, DV, false>), grid, block, 0, st, p);           \
  } while (0)
  else if (dtype == HALO_BF16) {
    if (D == 128) HALO_PREFILL(HALO_BF16, 128);
    else HALO_PREFILL(HALO_BF16, 64);
  } else {
    if (D == 128) HALO_PREFILL(HALO_F16, 128);
    else HALO_PREFILL(HALO_F16, 64);
  }
#undef HALO_PREFILL
  if (n_split > 1) {
    const int64_t jobs = units * nw * (D / 8 / 4);
    const dim3 mgrid((unsigned)((jobs + 3) / 4));
#define HALO_MERGE(DV)                                                                                             \
  do {                                                                                                             \
    if (dtype == HALO_F32)                                                                                         \
      hipLaunchKernelGGL((prefill_merge_kernel<DV, kPf32NW, PfRowsF32<DV>>), mgrid, dim3(256), 0, st, p);          \
    else                                                                                                           \
      hipLaunchKernelGGL((prefill_merge_kernel<DV, kPfNW, PfRowsTr<DV>>), mgrid, dim3(256), 0, st, p);             \
  } while (0)
    if (D == 128) HALO_MERGE(128);
    else HALO_MERGE(64);
#undef HALO_MERGE
  }
  HALO_CHECK_HIP(hipGetLastError());
  return HALO_OK;
}

extern "C" int halo_prefill_attn(const void* q, int64_t q_stride_b, int64_t q_stride_h, int64_t q_stride_t,
                                 int dtype, int B, int H, int H_kv, int T_q, int D, const int64_t* q_start,
                                 const halo_chunk_desc* descs, int n_desc, float scale,
                                 void* out, int64_t out_stride_b, int64_t out_stride_h, int64_t out_stride_t,
                                 int out_dtype, float* lse, void* stream) {
  HALO_CHECK_ARG(dtype == HALO_BF16 || dtype == HALO_F16, "prefill runs on bf16/fp16 MFMA: dtype must be bf16 or f16");
  return halo_prefill_attn_split(q, q_stride_b, q_stride_h, q_stride_t, dtype, B, H, H_kv, T_q, D, q_start, descs,
                                 n_desc, scale, out, out_stride_b, out_stride_h, out_stride_t, out_dtype, lse, 1,
                                 nullptr, 0, stream);
}
