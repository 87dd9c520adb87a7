// Quest bounding-box page scoring (gfx950, wave64): per-page channel-wise
// key minima and maxima, Quest's per-page upper bound
// sum_d max(q_d * kmin_d, q_d * kmax_d) and a deterministic top-k.  All of
// it is HBM/L2-bound reduction work; none of it is shaped into a GEMM.
//
// Reference semantics:
//   page min / max   baselines/quest_path_d.py:125-150 (amin / amax over the
//                    page's rows, kept in the key dtype: exact)
//   GQA mean query   baselines/quest_path_d.py:166-172 (mean over the rep
//                    query heads, kept in the query dtype)
//   bound            baselines/quest_path_d.py:173-178 (fp32 products,
//                    elementwise maximum, sum over the channels)
//   page score       baselines/quest_path_d.py:196 (max over b, h_kv, t_q)
//   top-K            baselines/quest_path_d.py:197-203 (descending score
//                    order; ties by lower page index, NaN bounds rank as -inf)

#include "common.hpp"

#include <algorithm>

namespace halo {

// torch.amin / amax / maximum propagate NaN; fminf / fmaxf would drop it.
__device__ __forceinline__ float nan_min(float a, float x) { return (x < a || x != x) ? x : a; }
__device__ __forceinline__ float nan_max(float a, float x) { return (x > a || x != x) ? x : a; }

// ---------------------------------------------------------------------------
// Page minima / maxima: one workgroup per (b, h, page).  Thread t owns the
// 16-byte piece t % SL of rows t/SL, t/SL + RG, ... (RG = 256/SL row groups),
// so the loads are whole coalesced rows; the RG partial results meet through
// LDS.  min / max are exact in any order, so the stored elements are the
// key elements themselves.
// ---------------------------------------------------------------------------
template <int DT>
__global__ void __launch_bounds__(256) page_minmax_kernel(const void* k, int64_t ksb, int64_t ksh, int64_t kst,
                                                          int H_kv, int D, int64_t row0, int page, int n_pages,
                                                          void* kmin, void* kmax, int64_t msb, int64_t msh,
                                                          int64_t msp) {
  constexpr int ESZ = DT == HALO_F32 ? 4 : 2;
  constexpr int EPC = 16 / ESZ;
  __shared__ float s_mn[256 * 8];
  __shared__ float s_mx[256 * 8];
  const int j = blockIdx.x % n_pages;
  const int bh = blockIdx.x / n_pages;
  const int h = bh % H_kv, b = bh / H_kv;
  const int SL = D / EPC;
  const int RG = 256 / SL;
  const int tid = threadIdx.x;
  const int col = tid % SL, rg = tid / SL;
  float mn[EPC], mx[EPC];
#pragma unroll
  for (int e = 0; e < EPC; ++e) {
    mn[e] = INFINITY;
    mx[e] = -INFINITY;
  }
  if (rg < RG) {
    const char* base = reinterpret_cast<const char*>(k) +
                       ((int64_t)b * ksb + (int64_t)h * ksh + (row0 + (int64_t)j * page) * kst) * ESZ + col * 16;
#pragma unroll 4
    for (int t = rg; t < page; t += RG) {
      const uint4 v = *reinterpret_cast<const uint4*>(base + (int64_t)t * kst * ESZ);
      const uint32_t w[4] = {v.x, v.y, v.z, v.w};
      float f[EPC];
      if constexpr (DT == HALO_F32) {
#pragma unroll
        for (int e = 0; e < 4; ++e) f[e] = __uint_as_float(w[e]);
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          if constexpr (DT == HALO_BF16) {
            f[2 * e] = bf16_lo(w[e]);
            f[2 * e + 1] = bf16_hi(w[e]);
          } else {
            f[2 * e] = f16_bits_to_f32((uint16_t)(w[e] & 0xffffu));
            f[2 * e + 1] = f16_bits_to_f32((uint16_t)(w[e] >> 16));
          }
        }
      }
#pragma unroll
      for (int e = 0; e < EPC; ++e) {
        mn[e] = nan_min(mn[e], f[e]);
        mx[e] = nan_max(mx[e], f[e]);
      }
    }
  }
#pragma unroll
  for (int e = 0; e < EPC; ++e) {
    s_mn[tid * 8 + e] = mn[e];
    s_mx[tid * 8 + e] = mx[e];
  }
  __syncthreads();
  const int64_t o = (int64_t)b * msb + (int64_t)h * msh + (int64_t)j * msp;
  for (int d = tid; d < D; d += 256) {
    const int c = d / EPC, e = d % EPC;
    float a = INFINITY, z = -INFINITY;
    for (int g = 0; g < RG; ++g) {
      a = nan_min(a, s_mn[(g * SL + c) * 8 + e]);
      z = nan_max(z, s_mx[(g * SL + c) * 8 + e]);
    }
    // a stored element of the key dtype converts back exactly
    store_elem(kmin, o + d, DT, a);
    store_elem(kmax, o + d, DT, z);
  }
}

// min / max of three numbers in one operation (NaN is dropped, and of zeros of
// both signs either may be kept).
__device__ __forceinline__ float min3(float a, float x, float y) {
  float r;
  asm("v_min3_f32 %0, %1, %2, %3" : "=v"(r) : "v"(a), "v"(x), "v"(y));
  return r;
}
__device__ __forceinline__ float max3(float a, float x, float y) {
  float r;
  asm("v_max3_f32 %0, %1, %2, %3" : "=v"(r) : "v"(a), "v"(x), "v"(y));
  return r;
}

// The same for pages of at most 2*RG rows: one thread per 16-byte column piece
// of a page reads all its rows.  Such a page gives the kernel above one or two
// loads a thread in front of a barrier and an LDS pass over RG partials, so it
// was bound by latency and not by HBM: 31.5 us for 32768 rows of 8 heads x 128
// bf16 in 16-row pages (2.1 TB/s), 13.9 here.  Compares that keep NaN cost
// seven operations an element and bound it in turn, so rows are folded two at a
// time without that; a piece that met a NaN, or ends at a zero (of two signs),
// is read again and folded in the other kernel's order.
template <int DT>
__global__ void __launch_bounds__(256) page_minmax_col_kernel(const void* k, int64_t ksb, int64_t ksh, int64_t kst,
                                                              int H_kv, int D, int64_t row0, int page, int n_pages,
                                                              int64_t total, void* kmin, void* kmax, int64_t msb,
                                                              int64_t msh, int64_t msp, int vec) {
  constexpr int ESZ = DT == HALO_F32 ? 4 : 2;
  constexpr int EPC = 16 / ESZ;
  constexpr int U = 8;  // rows in flight
  const int64_t gid = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (gid >= total) return;
  const int SL = D / EPC;
  const int RG = 256 / SL;
  const int col = (int)(gid % SL);
  const int pg = (int)(gid / SL);
  const int j = pg % n_pages, bh = pg / n_pages;
  const int h = bh % H_kv, b = bh / H_kv;
  const char* base = reinterpret_cast<const char*>(k) +
                     ((int64_t)b * ksb + (int64_t)h * ksh + (row0 + (int64_t)j * page) * kst) * ESZ + col * 16;
  float mn[EPC], mx[EPC];
#pragma unroll
  for (int e = 0; e < EPC; ++e) {
    mn[e] = INFINITY;
    mx[e] = -INFINITY;
  }
  bool again = false;
  for (int t0 = 0; t0 < page; t0 += U) {
    uint4 v[U];
#pragma unroll
    for (int u = 0; u < U; ++u)  // a row past the page repeats its last one: no effect on min or max
      v[u] = *reinterpret_cast<const uint4*>(base + (int64_t)min(t0 + u, page - 1) * kst * ESZ);
#pragma unroll
    for (int u = 0; u < U; u += 2) {
      float x[EPC], y[EPC];
      unpack16<DT>(v[u], x);
      unpack16<DT>(v[u + 1], y);
#pragma unroll
      for (int e = 0; e < EPC; ++e) {
        mn[e] = min3(mn[e], x[e], y[e]);
        mx[e] = max3(mx[e], x[e], y[e]);
        again |= __builtin_isunordered(x[e], y[e]);
      }
    }
  }
#pragma unroll
  for (int e = 0; e < EPC; ++e) again |= mn[e] == 0.f || mx[e] == 0.f;
  if (again) {
    // NaN has to stay, and of zeros the first in row-group order
#pragma unroll
    for (int e = 0; e < EPC; ++e) {
      mn[e] = INFINITY;
      mx[e] = -INFINITY;
    }
    for (int g = 0; g < min(page, RG); ++g)
      for (int t = g; t < page; t += RG) {
        float x[EPC];
        unpack16<DT>(*reinterpret_cast<const uint4*>(base + (int64_t)t * kst * ESZ), x);
#pragma unroll
        for (int e = 0; e < EPC; ++e) {
          mn[e] = nan_min(mn[e], x[e]);
          mx[e] = nan_max(mx[e], x[e]);
        }
      }
  }
  const int64_t o = (int64_t)b * msb + (int64_t)h * msh + (int64_t)j * msp + col * EPC;
  store_piece<DT>(kmin, o, vec != 0, mn);  // a stored element of the key dtype converts back exactly
  store_piece<DT>(kmax, o, vec != 0, mx);
}

// ---------------------------------------------------------------------------
// Bound scores.  A selection covers batch row `sel` (per_row) or every row
// (the reference's max over the batch).  Its rows are the (b, h_kv, t_q)
// triples.  A page's bound is summed by G = D/16 lanes, lane c over slice c,
// so that a wave reads whole rows of 64/G2 pages in 16-byte pieces (one lane
// per page read 256 bytes apart and left 192 of 256 CUs idle at 2048 pages x
// 8 heads: 13.3 us, 8.0 here).  The waves of a workgroup take runs of its
// rows, which keep the page pieces of one (b, h) in registers over t_q, and
// meet in LDS; the max is folded on an order-preserving encoding of the float,
// exact in any order.  With row_split > 1 workgroups share a page's rows and
// merge with atomics, else they store.
// ---------------------------------------------------------------------------
struct QuestParams {
  const void* q;
  int64_t qsb, qsh, qst;
  int B, H, H_kv, T_q, D, rep;
  float inv_rep;  // fp32(1/rep): torch's mean factor
  const void* kmin;
  const void* kmax;
  int64_t msb, msh, msp;
  int P, per_row, rows_sel, row_split, page_tiles, qvec;
  float* dots;       // optional (B, H_kv, T_q, P) fp32
  uint32_t* keys;    // (n_sel, P) encoded page scores
};

constexpr int kQuestMaxD = 256;
constexpr int kQuestMaxPages = 8192;
constexpr uint32_t kKeyNegInf = 0x007fffffu;  // key(-inf); NaN is never encoded: it is ranked as -inf

__global__ void __launch_bounds__(256) quest_init_kernel(uint32_t* keys, int n) {
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i < n) keys[i] = kKeyNegInf;
}

template <int DT, int G2, int IT>
__global__ void __launch_bounds__(IT == 1 ? 1024 : 256) quest_score_kernel(QuestParams P) {
  constexpr int PPW = 64 / G2;  // pages of one pass of a wave, IT passes
  constexpr int esz = DT == HALO_F32 ? 4 : 2;
  constexpr int ep = 16 / esz;
  __shared__ uint32_t s_best[IT == 1 ? 16 : 4][PPW * IT];
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int pt = blockIdx.x % P.page_tiles;
  const int rs = (blockIdx.x / P.page_tiles) % P.row_split;
  const int sel = blockIdx.x / (P.page_tiles * P.row_split);
  const int G = P.D / 16;
  const int c = lane % G2, pw = lane / G2;
  const int p0 = pt * PPW * IT + pw;  // pages p0 + it*PPW
  uint32_t best[IT];
#pragma unroll
  for (int it = 0; it < IT; ++it) best[it] = kKeyNegInf;
  // this wave's rows, in (b, h, t) order: the pages are read again only where (b, h) changes
  const int nw = blockDim.x >> 6;
  const int per = (P.rows_sel + nw * P.row_split - 1) / (nw * P.row_split);
  const int lo_r = min((rs * nw + w) * per, P.rows_sel), hi_r = min(lo_r + per, P.rows_sel);
  uint4 vn[IT][16 / ep], vx[IT][16 / ep];
  int held = -1;
  for (int r = lo_r; r < hi_r; ++r) {
    const int t = r % P.T_q, bh = r / P.T_q;
    const int h = bh % P.H_kv;
    const int b = P.per_row ? sel : bh / P.H_kv;
    if (bh != held) {
      held = bh;
#pragma unroll
      for (int it = 0; it < IT; ++it) {
        // lanes without a slice or page read slice 0 of the last page and drop it
        const int p = min(p0 + it * PPW, P.P - 1), cc = c < G ? c : 0;
        const int64_t mo = ((int64_t)b * P.msb + (int64_t)h * P.msh + (int64_t)p * P.msp) * esz;
#pragma unroll
        for (int pp = 0; pp < 16 / ep; ++pp) {
          vn[it][pp] = *reinterpret_cast<const uint4*>(reinterpret_cast<const char*>(P.kmin) + mo + (cc + pp * G) * 16);
          vx[it][pp] = *reinterpret_cast<const uint4*>(reinterpret_cast<const char*>(P.kmax) + mo + (cc + pp * G) * 16);
        }
      }
    }
    float qg[16];
    gqa_mean_slice<DT>(P.q, (int64_t)b * P.qsb + (int64_t)t * P.qst, P.qsh, h, P.rep, P.inv_rep, c < G ? c : 0, G,
                       P.qvec != 0, qg);
#pragma unroll
    for (int it = 0; it < IT; ++it) {
      // slice c: elements ep*(c + pp*G) + e in (pp, e) order, products and sums rounded separately
      float a = 0.f;
#pragma unroll
      for (int pp = 0; pp < 16 / ep; ++pp) {
        float fn[ep], fx[ep];
        unpack16<DT>(vn[it][pp], fn);
        unpack16<DT>(vx[it][pp], fx);
#pragma unroll
        for (int e = 0; e < ep; ++e) {
          const float qd = qg[pp * ep + e];
          const float lo = __fmul_rn(qd, fn[e]), hi = __fmul_rn(qd, fx[e]);
          a = __fadd_rn(a, (lo > hi || lo != lo) ? lo : hi);
        }
      }
      const float dot = slice_tree<G2>(a, c, G);
      const int p = p0 + it * PPW;
      if (c == 0 && p < P.P) {
        if (P.dots) P.dots[(((int64_t)b * P.H_kv + h) * P.T_q + t) * P.P + p] = dot;
        if (dot == dot) best[it] = max(best[it], float_key(dot));
      }
    }
  }
  if (c == 0) {
#pragma unroll
    for (int it = 0; it < IT; ++it) s_best[w][it * PPW + pw] = best[it];
  }
  __syncthreads();
  const int i = threadIdx.x;
  const int p = pt * PPW * IT + i;
  if (i < PPW * IT && p < P.P) {
    uint32_t m = s_best[0][i];
    for (int x = 1; x < nw; ++x) m = max(m, s_best[x][i]);
    uint32_t* dst = P.keys + (int64_t)sel * P.P + p;
    if (P.row_split > 1) atomicMax(dst, m);
    else *dst = m;
  }
}

// Top-k of one selection: page i's rank is the number of pages with a
// larger score or an equal score and a lower index; ranks below k are
// written in rank order (descending score, as torch.topk returns them).
// A workgroup ranks 64 pages, one per lane, and its 16 waves count over the
// 64-key blocks in turn, one key per lane handed round by v_readlane.  One
// workgroup per selection took 153 us for 2048 pages on one CU, 6.2 here.
constexpr int kRankWaves = 16;
__global__ void __launch_bounds__(64 * kRankWaves) quest_rank_kernel(const uint32_t* __restrict__ keys, int P, int k,
                                                                     int tiles, int32_t* __restrict__ idx_out,
                                                                     float* __restrict__ score_out) {
  __shared__ int s_rank[kRankWaves][64];
  const int sel = blockIdx.x / tiles, tile = blockIdx.x % tiles;
  const uint32_t* kk = keys + (int64_t)sel * P;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int i = tile * 64 + lane;
  const uint32_t ki = i < P ? kk[i] : 0u;  // 0 is below every key of a page
  int rank = 0;
  for (int jt = w; jt < tiles; jt += kRankWaves) {
    const int jl = jt * 64 + lane;
    const int kj = (int)(jl < P ? kk[jl] : 0u);
    // a page ahead of this one wins ties, one behind it has to be above: no
    // key is above key(+inf), so ki + 1 does not wrap
    if (jt == tile) {
#pragma unroll
      for (int j = 0; j < 64; ++j)
        rank += (uint32_t)__builtin_amdgcn_readlane(kj, j) >= ki + (j < lane ? 0u : 1u) ? 1 : 0;
    } else {
      const uint32_t thr = ki + (jt > tile ? 1u : 0u);
#pragma unroll
      for (int j = 0; j < 64; ++j) rank += (uint32_t)__builtin_amdgcn_readlane(kj, j) >= thr ? 1 : 0;
    }
  }
  s_rank[w][lane] = rank;
  __syncthreads();
  if (threadIdx.x < 64 && i < P) {
    int r = 0;
#pragma unroll
    for (int x = 0; x < kRankWaves; ++x) r += s_rank[x][lane];
    if (r < k) idx_out[(int64_t)sel * k + r] = i;
    if (score_out) score_out[(int64_t)sel * P + i] = key_float(ki);
  }
}

}  // namespace halo

using namespace halo;

extern "C" int halo_page_minmax(const void* k, int64_t k_stride_b, int64_t k_stride_h, int64_t k_stride_t,
                                int dtype, int B, int H_kv, int D, int64_t row0, int page, int n_pages,
                                void* kmin, void* kmax, int64_t km_stride_b, int64_t km_stride_h,
                                int64_t km_stride_p, void* stream) {
  HALO_CHECK_ARG(k && kmin && kmax, "null pointer");
  HALO_CHECK_ARG(dtype == HALO_F32 || dtype == HALO_BF16 || dtype == HALO_F16, "bad dtype");
  HALO_CHECK_ARG(B > 0 && H_kv > 0 && D > 0 && page > 0 && n_pages >= 0 && row0 >= 0, "bad sizes");
  if (n_pages == 0) return HALO_OK;
  HALO_CHECK_ARG(D % (dtype == HALO_F32 ? 4 : 8) == 0 && D <= 256 * (dtype == HALO_F32 ? 4 : 8),
                 "head dim must fill whole 16-byte pieces");
  HALO_CHECK_ARG(reinterpret_cast<uintptr_t>(k) % 16 == 0 && (k_stride_t * elem_size(dtype)) % 16 == 0 &&
                 (k_stride_h * elem_size(dtype)) % 16 == 0 && (k_stride_b * elem_size(dtype)) % 16 == 0,
                 "key rows must be 16-byte aligned");
  const int64_t blocks = (int64_t)B * H_kv * n_pages;
  HALO_CHECK_ARG(blocks <= 0x7fffffffLL, "too many pages for one launch");
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  const int es = elem_size(dtype);
  const int SL = D / (16 / es), RG = 256 / SL;
  // Whole pages per thread for pages of up to 16 rows, and of up to 32 where
  // that still gives 64K threads; 256 threads a page otherwise.  8 heads x 128
  // bf16, here / 256 threads a page: 16-row pages of 8192 rows 5.2 / 9.4 us, of
  // 32768 rows 13.8 / 29.5; 32-row pages of 8192 rows (32K threads) 7.5 / 6.6,
  // of 32768 rows 12.9 / 19.7; 64-row pages of 32768 rows x 64 13.6 / 11.2.
  const int64_t total = blocks * SL;
  const bool col = page <= 2 * RG && (page <= 16 || (page <= 32 && total >= 65536));
  const int vec = reinterpret_cast<uintptr_t>(kmin) % 16 == 0 && reinterpret_cast<uintptr_t>(kmax) % 16 == 0 &&
                  (km_stride_b * es) % 16 == 0 && (km_stride_h * es) % 16 == 0 && (km_stride_p * es) % 16 == 0;
#define HALO_MINMAX(DTV)                                                                                  \
  do {                                                                                                    \
    if (col)                                                                                              \
      hipLaunchKernelGGL(page_minmax_col_kernel<DTV>, dim3((unsigned)((total + 255) / 256)), dim3(256), 0, st, k, \
                         k_stride_b, k_stride_h, k_stride_t, H_kv, D, row0, page, n_pages, total, kmin, kmax, \
                         km_stride_b, km_stride_h, km_stride_p, vec);                                     \
    else                                                                                                  \
      hipLaunchKernelGGL(page_minmax_kernel<DTV>, dim3((unsigned)blocks), dim3(256), 0, st, k, k_stride_b, \
                         k_stride_h, k_stride_t, H_kv, D, row0, page, n_pages, kmin, kmax, km_stride_b,   \
                         km_stride_h, km_stride_p);                                                       \
  } while (0)
  if (dtype == HALO_F32) HALO_MINMAX(HALO_F32);
  else if (dtype == HALO_BF16) HALO_MINMAX(HALO_BF16);
  else HALO_MINMAX(HALO_F16);
#undef HALO_MINMAX
  HALO_CHECK_HIP(hipGetLastError());
  return HALO_OK;
}

extern "C" int halo_quest_score_topk(const void* q, int64_t q_stride_b, int64_t q_stride_h, int64_t q_stride_t,
                                     int dtype, int B, int H, int H_kv, int T_q, int D, const void* kmin,
                                     const void* kmax, int64_t km_stride_b, int64_t km_stride_h,
                                     int64_t km_stride_p, int P, int k, int per_row, uint32_t* workspace,
                                     float* dots_out, float* score_out, int32_t* idx_out, void* stream) {
  HALO_CHECK_ARG(q && kmin && kmax && workspace, "null pointer");
  HALO_CHECK_ARG(dtype == HALO_F32 || dtype == HALO_BF16 || dtype == HALO_F16, "bad dtype");
  HALO_CHECK_ARG(B > 0 && H > 0 && H_kv > 0 && H % H_kv == 0 && T_q > 0, "bad head sizes");
  HALO_CHECK_ARG(D % 16 == 0 && D > 0 && D <= kQuestMaxD, "head dim must be a multiple of 16, at most 256");
  HALO_CHECK_ARG(P > 0 && P <= kQuestMaxPages, "page count must be in [1, 8192]");
  HALO_CHECK_ARG(k >= 0 && k <= P, "k must be in [0, P]");
  HALO_CHECK_ARG(k == 0 || idx_out != nullptr, "idx_out is required when k > 0");
  const int es = elem_size(dtype);
  HALO_CHECK_ARG(reinterpret_cast<uintptr_t>(kmin) % 16 == 0 && reinterpret_cast<uintptr_t>(kmax) % 16 == 0 &&
                 (km_stride_p * es) % 16 == 0 && (km_stride_h * es) % 16 == 0 && (km_stride_b * es) % 16 == 0,
                 "kmin/kmax rows must be 16-byte aligned");
  const int n_sel = per_row ? B : 1;
  const int64_t rows_sel = (int64_t)(per_row ? 1 : B) * H_kv * T_q;
  const int G = D / 16;
  const int G2 = G <= 1 ? 1 : G <= 2 ? 2 : G <= 4 ? 4 : G <= 8 ? 8 : 16;
  // Few rows: one pass of pages a workgroup and all rows in it, so that no
  // merge (and no fill of the keys, a launch) is needed: 4 waves, or 16 from 9
  // rows on.  Many rows: the query mean of a row costs more than its products
  // with one page, so a wave takes 4 passes of pages to a mean and the rows
  // are split, at least 2 a wave, up to about 2048 workgroups.  Score and rank
  // at 2048 pages x 8 heads, here / one row a wave and one page a lane (with
  // its 153 us rank): t_q 1 13 / 165 us, 4 17 / 166, 64 78 / 246, 512 516 / 670.
  const bool many = rows_sel > 64;
  const int waves = !many && rows_sel > 8 ? 16 : 4;
  const int64_t tile_pages = (64 / G2) * (many ? 4 : 1);
  const int64_t page_tiles = (P + tile_pages - 1) / tile_pages;
  int64_t row_split = 1;
  if (many)
    row_split = std::min<int64_t>((rows_sel + 7) / 8, (2048 + n_sel * page_tiles - 1) / (n_sel * page_tiles));
  const int64_t blocks = (int64_t)n_sel * row_split * page_tiles;
  HALO_CHECK_ARG(rows_sel <= 0x7fffffffLL && blocks <= 0x7fffffffLL, "too many (row, page) tiles for one launch");
  QuestParams p;
  p.q = q;
  p.qsb = q_stride_b;
  p.qsh = q_stride_h;
  p.qst = q_stride_t;
  p.B = B;
  p.H = H;
  p.H_kv = H_kv;
  p.T_q = T_q;
  p.D = D;
  p.rep = H / H_kv;
  p.inv_rep = (float)(1.0 / (double)p.rep);
  p.kmin = kmin;
  p.kmax = kmax;
  p.msb = km_stride_b;
  p.msh = km_stride_h;
  p.msp = km_stride_p;
  p.P = P;
  p.per_row = per_row;
  p.rows_sel = (int)rows_sel;
  p.row_split = (int)row_split;
  p.page_tiles = (int)page_tiles;
  p.qvec = reinterpret_cast<uintptr_t>(q) % 16 == 0 && (q_stride_b * es) % 16 == 0 && (q_stride_h * es) % 16 == 0 &&
           (q_stride_t * es) % 16 == 0;
  p.dots = dots_out;
  p.keys = workspace;
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  const int n_keys = n_sel * P;
  if (row_split > 1)
    hipLaunchKernelGGL(quest_init_kernel, dim3((n_keys + 255) / 256), dim3(256), 0, st, workspace, n_keys);
#define HALO_QUEST_G(DTV, G2V)                                                                              \
  do {                                                                                                      \
    if (many)                                                                                               \
      hipLaunchKernelGGL((quest_score_kernel<DTV, G2V, 4>), dim3((unsigned)blocks), dim3(256), 0, st, p);   \
    else                                                                                                    \
      hipLaunchKernelGGL((quest_score_kernel<DTV, G2V, 1>), dim3((unsigned)blocks), dim3(64 * waves), 0, st, p); \
  } while (0)
#define HALO_QUEST(DTV)                       \
  do {                                        \
    if (G2 == 1) HALO_QUEST_G(DTV, 1);        \
    else if (G2 == 2) HALO_QUEST_G(DTV, 2);   \
    else if (G2 == 4) HALO_QUEST_G(DTV, 4);   \
    else if (G2 == 8) HALO_QUEST_G(DTV, 8);   \
    else HALO_QUEST_G(DTV, 16);               \
  } while (0)
  if (dtype == HALO_F32) HALO_QUEST(HALO_F32);
  else if (dtype == HALO_BF16) HALO_QUEST(HALO_BF16);
  else HALO_QUEST(HALO_F16);
#undef HALO_QUEST
#undef HALO_QUEST_G
  const int rank_tiles = (P + 63) / 64;
  hipLaunchKernelGGL(quest_rank_kernel, dim3((unsigned)(n_sel * rank_tiles)), dim3(64 * kRankWaves), 0, st, workspace, P,
                     k, rank_tiles, idx_out, score_out);
  HALO_CHECK_HIP(hipGetLastError());
  return HALO_OK;
}
