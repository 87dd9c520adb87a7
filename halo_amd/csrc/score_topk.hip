// Chunk-relevance scoring: page-mean keys, q.Kbar scores and a
// deterministic top-k that writes the selected chunks into a device chunk
// table (gfx950, wave64).  All of it is HBM/L2-bound reduction work; none of
// it is shaped into a GEMM.
//
// Reference semantics:
//   page means        baselines/scorer_ablations.py:209-216
//   GQA mean query    baselines/scorer_ablations.py:223-232 (kept in q dtype)
//   score             baselines/scorer_ablations.py:233-237 (max over rows, heads)
//   top-k             baselines/scorer_ablations.py:265-266 with the build's
//                     tie rule (score desc, chunk index asc), indices sorted
//   budget            baselines/scorer_ablations.py:133-139 (host side)

#include "common.hpp"

namespace halo {

// fp16 means of two sums, each product rounded once, to fp16 (written out: left
// to the compiler a product and its conversion are one or two roundings; the
// wait state is the one between two writes of halves of a register).
__device__ __forceinline__ uint32_t mean_f16(float lo, float hi, float inv) {
  uint32_t r;
  asm("v_fma_mixlo_f16 %0, %1, %3, 0\n\ts_nop 0\n\tv_fma_mixhi_f16 %0, %2, %3, 0"
      : "=&v"(r)
      : "v"(lo), "v"(hi), "v"(inv));
  return r;
}

// ---------------------------------------------------------------------------
// Page means: kmean[b,h,j,d] = dtype(sum_t K[b,h,row0+j*page+t,d] / page).
// One workgroup per (b, h, page).  Thread t owns the 16-byte piece
// t % SL of rows t/SL, t/SL + RG, ... (RG = 256/SL row groups), so loads are
// whole coalesced rows and independent; the RG fp32 partial sums are then
// added in row-group order through LDS and rounded once to the key dtype.
// ---------------------------------------------------------------------------
// U rows of a thread are in flight at a time: 8, 32 for 16-bit pages of at least 32
// rows a thread, whose few workgroups are each bound by their own round trips
// (one page of 1024 rows x 8 heads x 128 bf16, eight workgroups: 12.3 -> 5.7 us;
// 256 rows 4.8 -> 3.0), or 0: left to the compiler (fp32, whose 1024 rows took 6.5
// us so and 6.9-7.5 in batches).
template <int DT, int U>
__global__ void __launch_bounds__(256) chunk_means_kernel(const void* k, int64_t ksb, int64_t ksh, int64_t kst,
                                                          int H_kv, int D, int64_t row0, int page, int n_pages,
                                                          void* km, int64_t msb, int64_t msh, int64_t msp) {
  constexpr int ESZ = DT == HALO_F32 ? 4 : 2;
  constexpr int EPC = 16 / ESZ;
  __shared__ float s_part[256 * 8];
  const int j = blockIdx.x % n_pages;
  const int bh = blockIdx.x / n_pages;
  const int h = bh % H_kv, b = bh / H_kv;
  const int SL = D / EPC;
  const int RG = 256 / SL;
  const int tid = threadIdx.x;
  const int col = tid % SL, rg = tid / SL;
  float acc[EPC];
#pragma unroll
  for (int e = 0; e < EPC; ++e) acc[e] = 0.f;
  if (rg < RG) {
    const char* base = reinterpret_cast<const char*>(k) +
                       ((int64_t)b * ksb + (int64_t)h * ksh + (row0 + (int64_t)j * page) * kst) * ESZ + col * 16;
    auto add = [&](const uint4& v) {
      float x[EPC];
      unpack16<DT>(v, x);
#pragma unroll
      for (int e = 0; e < EPC; ++e) acc[e] += x[e];
    };
    int t = rg;
    for (; U > 0 && t + (U - 1) * RG < page; t += U * RG) {
      uint4 v[U > 0 ? U : 1];
#pragma unroll
      for (int u = 0; u < U; ++u) v[u] = *reinterpret_cast<const uint4*>(base + (int64_t)(t + u * RG) * kst * ESZ);
#pragma unroll
      for (int u = 0; u < U; ++u) add(v[u]);
    }
    if constexpr (U > 0) {
#pragma unroll 8
      for (; t < page; t += RG) add(*reinterpret_cast<const uint4*>(base + (int64_t)t * kst * ESZ));
    } else {
#pragma unroll 8
      for (int r = rg; r < page; r += RG) {
        const uint4 v = *reinterpret_cast<const uint4*>(base + (int64_t)r * kst * ESZ);
        const uint32_t w[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
        for (int e = 0; e < 4; ++e) acc[e] += __uint_as_float(w[e]);
      }
    }
  }
#pragma unroll
  for (int e = 0; e < EPC; ++e) s_part[tid * 8 + e] = acc[e];
  __syncthreads();
  const float inv = 1.0f / (float)page;
  for (int d = tid; d < D; d += 256) {
    const int c = d / EPC, e = d % EPC;
    float sum = 0.f;
    for (int g = 0; g < RG; ++g) sum += s_part[(g * SL + c) * 8 + e];
    const int64_t o = (int64_t)b * msb + (int64_t)h * msh + (int64_t)j * msp + d;
    if constexpr (DT == HALO_F16) reinterpret_cast<uint16_t*>(km)[o] = (uint16_t)mean_f16(sum, 0.f, inv);
    else store_elem(km, o, DT, sum * inv);
  }
}

// The same for pages of at most RG rows, one to a row group: one thread per
// 16-byte column piece of a page adds all its rows in row-group order, so the
// means are the other kernel's bit for bit.  Such a page gives the kernel above
// one load a thread in front of a barrier and an LDS pass: 8.4 us for 8192 rows
// of 8 heads x 128 bf16 in 16-row pages, 5.4 here.
template <int DT>
__global__ void __launch_bounds__(256) chunk_means_col_kernel(const void* k, int64_t ksb, int64_t ksh, int64_t kst,
                                                              int H_kv, int D, int64_t row0, int page, int n_pages,
                                                              int64_t total, void* km, int64_t msb, int64_t msh,
                                                              int64_t msp, int vec) {
  constexpr int ESZ = DT == HALO_F32 ? 4 : 2;
  constexpr int EPC = 16 / ESZ;
  constexpr int U = 8;  // rows in flight
  const int64_t gid = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (gid >= total) return;
  const int SL = D / EPC;
  const int col = (int)(gid % SL);
  const int pg = (int)(gid / SL);
  const int j = pg % n_pages, bh = pg / n_pages;
  const int h = bh % H_kv, b = bh / H_kv;
  const char* base = reinterpret_cast<const char*>(k) +
                     ((int64_t)b * ksb + (int64_t)h * ksh + (row0 + (int64_t)j * page) * kst) * ESZ + col * 16;
  float sum[EPC];
#pragma unroll
  for (int e = 0; e < EPC; ++e) sum[e] = 0.f;
  for (int t0 = 0; t0 < page; t0 += U) {
    uint4 v[U];
#pragma unroll
    for (int u = 0; u < U; ++u)  // a row past the page is loaded as its last one and not used
      v[u] = *reinterpret_cast<const uint4*>(base + (int64_t)min(t0 + u, page - 1) * kst * ESZ);
#pragma unroll
    for (int u = 0; u < U; ++u) {
      float f[EPC];
      unpack16<DT>(v[u], f);
      // adding +0 leaves a sum that began at +0 as it is
#pragma unroll
      for (int e = 0; e < EPC; ++e) sum[e] += t0 + u < page ? f[e] : 0.f;
    }
  }
  const float inv = 1.0f / (float)page;
  const int64_t o = (int64_t)b * msb + (int64_t)h * msh + (int64_t)j * msp + col * EPC;
  if constexpr (DT == HALO_F16) {
    uint32_t w[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) w[e] = mean_f16(sum[2 * e], sum[2 * e + 1], inv);
    uint16_t* dst = reinterpret_cast<uint16_t*>(km) + o;
    if (vec) {
      *reinterpret_cast<uint4*>(dst) = make_uint4(w[0], w[1], w[2], w[3]);
    } else {
#pragma unroll
      for (int e = 0; e < 8; ++e) dst[e] = (uint16_t)(w[e >> 1] >> (16 * (e & 1)));
    }
  } else {
#pragma unroll
    for (int e = 0; e < EPC; ++e) sum[e] *= inv;
    store_piece<DT>(km, o, vec != 0, sum);
  }
}

// ---------------------------------------------------------------------------
// Score + top-k.  One workgroup per selection.  Selection s covers batch row
// s (per_row) or every row (per_row == 0, the reference's amax over batch).
// ---------------------------------------------------------------------------
struct ScoreParams {
  const void* q;
  int64_t qsb, qsh;
  int dtype;
  int B, H, H_kv, D, rep;
  float inv_rep;  // fp32(1/rep), rounded on the host: torch's mean factor
  const void* km;
  int64_t msb, msh, msp;
  const int32_t* elig;
  int64_t elig_stride;
  const int32_t* n_elig_per_sel;
  int n_elig;
  int k;
  int per_row;
  int32_t* idx_out;
  float* score_out;
  const halo_chunk_desc* catalog;
  int64_t catalog_stride;
  halo_chunk_desc* table;
  int64_t table_stride;
  int table_slot0;
  // page score = alpha*minmax(attn) + beta*recency + gamma*sink when
  // normalize != 0 (baselines/scorer_ablations.py:238-263); raw attn otherwise.
  int normalize;
  float alpha, beta, gamma;
  int refresh, sink_pages, P_total;
  // HBM staging (residency == NULL: off): a chosen chunk whose residency
  // entry names a slot is written to the table with that slot's addresses
  // and strides; res_out[sel * k + j] gets the entry used (-1: in place).
  const int32_t* residency;
  const halo_chunk_desc* slot_catalog;
  int n_slots;
  int32_t* res_out;
  int qvec;    // q rows are 16-byte aligned (score_pages_kernel)
  float* raw;  // (n_sel, n_elig) raw scores between score_pages_kernel and the selection
};

constexpr int kMaxElig = 1024;
constexpr int kMaxQg = 8192;    // floats of GQA-mean query rows held in LDS
constexpr int kMaxDots = 4096;  // (page, row, head) dot products per batch

// a ranks before b: larger score, then lower chunk index (NaN scores are
// stored as -inf before ranking).
__device__ __forceinline__ bool beats(float sa, int ea, float sb, int eb) {
  return sa > sb || (sa == sb && ea < eb);
}

// Wave-wide selection of the kk largest of n <= 64*NX scores (lower position
// first among equals, zeros of both signs equal): s_sel[i] = number of selected
// positions before i, or -1.  The kk-th largest key is built bit by bit from
// ballot counts (taken as int: `ties` goes below 0 once the equals are taken).
template <int NX>
__device__ __forceinline__ void select_ascending(const float* s_score, int n, int kk, int lane, int* s_sel) {
  uint32_t key[NX];
#pragma unroll
  for (int x = 0; x < NX; ++x) {
    const int i = 64 * x + lane;
    key[x] = i < n ? float_key(s_score[i] + 0.f) : 0u;  // 0 is below the key of every score
  }
  uint32_t thr = 0;
  for (int bit = 31; bit >= 0; --bit) {
    const uint32_t trial = thr | (1u << bit);
    int cnt = 0;
#pragma unroll
    for (int x = 0; x < NX; ++x) cnt += (int)__popcll(__ballot(key[x] >= trial));
    if (cnt >= kk) thr = trial;
    if (cnt == kk) break;
  }
  int ties = kk, pos0 = 0;
#pragma unroll
  for (int x = 0; x < NX; ++x) ties -= (int)__popcll(__ballot(key[x] > thr));
  const uint64_t below = (1ull << lane) - 1;
#pragma unroll
  for (int x = 0; x < NX; ++x) {
    const uint64_t eq = __ballot(key[x] == thr);
    const bool take = key[x] > thr || (key[x] == thr && (int)__popcll(eq & below) < ties);
    const uint64_t m = __ballot(take);
    if (64 * x + lane < n) s_sel[64 * x + lane] = take ? pos0 + (int)__popcll(m & below) : -1;
    pos0 += (int)__popcll(m);
    ties -= (int)__popcll(eq);
  }
}

// Raw scores of many pages, spread over the GPU: raw[sel, i] = max over
// (row, head) of qg . kbar, in the slice order of score_topk_kernel.  G = D/16
// lanes per page, lane c on slice c, so a wave reads whole rows of 64/G2 pages;
// the four waves of a workgroup take the (row, head) pairs in turn and meet in
// LDS.  A launch bound by latency: one round trip for q and the page means.  With
// the selection below, 512 pages x 8 heads x 128 took 67.5 us in one workgroup,
// 6.1 + 8.4 here.
template <int DT, int G2>
__global__ void __launch_bounds__(256) score_pages_kernel(ScoreParams P, int tiles) {
  constexpr int PPW = 64 / G2;  // pages per wave
  constexpr int esz = DT == HALO_F32 ? 4 : 2;
  constexpr int ep = 16 / esz;
  __shared__ float s_best[4][PPW];
  const int sel = blockIdx.x / tiles, tile = blockIdx.x % tiles;
  const int w = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int b0 = P.per_row ? sel : 0;
  const int nrh = (P.per_row ? 1 : P.B) * P.H_kv;
  const int n = P.n_elig_per_sel ? min(P.n_elig_per_sel[sel], P.n_elig) : P.n_elig;
  const int G = P.D / 16;
  const int c = lane % G2, pw = lane / G2;
  const int i = tile * PPW + pw;
  const int chunk = i < n ? P.elig[(int64_t)sel * P.elig_stride + i] : 0;
  float best = -INFINITY;
  for (int rh = w; rh < nrh; rh += 4) {
    const int r = rh / P.H_kv, h = rh % P.H_kv;
    float a = 0.f;
    if (c < G && i < n) {
      const char* row = reinterpret_cast<const char*>(P.km) +
                        ((int64_t)(b0 + r) * P.msb + (int64_t)h * P.msh + (int64_t)chunk * P.msp) * esz;
      uint4 v[16 / ep];
#pragma unroll
      for (int p = 0; p < 16 / ep; ++p) v[p] = *reinterpret_cast<const uint4*>(row + (c + p * G) * 16);
      float qg[16];
      gqa_mean_slice<DT>(P.q, (int64_t)(b0 + r) * P.qsb, P.qsh, h, P.rep, P.inv_rep, c, G, P.qvec != 0, qg);
#pragma unroll
      for (int p = 0; p < 16 / ep; ++p) {
        float f[ep];
        unpack16<DT>(v[p], f);
#pragma unroll
        for (int e = 0; e < ep; ++e) a = __fadd_rn(a, __fmul_rn(qg[p * ep + e], f[e]));
      }
    }
    best = fmaxf(best, slice_tree<G2>(a, c, G));
  }
  if (c == 0) s_best[w][pw] = best;
  __syncthreads();
  const int t = threadIdx.x;
  if (t < PPW && tile * PPW + t < n)
    P.raw[(int64_t)sel * P.n_elig + tile * PPW + t] =
        fmaxf(fmaxf(s_best[0][t], s_best[1][t]), fmaxf(s_best[2][t], s_best[3][t]));
}

// DC: the head dim when known at compile time (64, 128, 256: the dot-product
// loops unroll and every load of a triple is issued before the first use),
// 0 for any other multiple of 16 (runtime loops), -1: P.raw holds the raw
// scores (score_pages_kernel) and only the combination and the top-k remain.
template <int DT, int DC>
__global__ void __launch_bounds__(512) score_topk_kernel(ScoreParams P) {
  constexpr bool kGiven = DC < 0;
  __shared__ float s_qg[kGiven ? 1 : kMaxQg];
  __shared__ __align__(16) float s_score[kMaxElig];
  __shared__ __align__(16) int s_chunk[kMaxElig];
  __shared__ __align__(16) int s_sel[kMaxElig];
  __shared__ float s_dot[kGiven ? 1 : kMaxDots];
  const int sel = blockIdx.x;
  const int tid = threadIdx.x;
  const int nthr = blockDim.x;
  const int b0 = P.per_row ? sel : 0;
  const int nrows = P.per_row ? 1 : P.B;
  const int n = P.n_elig_per_sel ? min(P.n_elig_per_sel[sel], P.n_elig) : P.n_elig;
  const int kk = min(P.k, n);
  const int32_t* elig = P.elig + (int64_t)sel * P.elig_stride;

  for (int i = tid; i < n; i += nthr) s_chunk[i] = elig[i];
  if constexpr (kGiven) {
    for (int i = tid; i < n; i += nthr) {
      const float v = P.raw[(int64_t)sel * P.n_elig + i];
      s_score[i] = v != v ? -INFINITY : v;
    }
    __syncthreads();
  } else {
  // GQA mean of the query heads of each KV head, rounded to the q dtype
  // (torch's .mean keeps the dtype); rep == 1 uses q as is.
  const int Dq = DC ? DC : P.D;
  const int QG = nrows * P.H_kv * Dq;
  for (int i = tid; i < QG; i += nthr) {
    const int d = i % Dq;
    const int h = (i / Dq) % P.H_kv;
    const int r = i / (Dq * P.H_kv);
    const int64_t qb = (int64_t)(b0 + r) * P.qsb;
    float v;
    if (P.rep == 1) {
      v = load_elem(P.q, qb + (int64_t)h * P.qsh + d, DT);
    } else {
      // the rep loads are independent: issue them in batches of 4, then add in head order
      float acc = 0.f;
      for (int j0 = 0; j0 < P.rep; j0 += 4) {
        float x[4];
#pragma unroll
        for (int j = 0; j < 4; ++j)
          x[j] = j0 + j < P.rep ? load_elem(P.q, qb + (int64_t)(h * P.rep + j0 + j) * P.qsh + d, DT) : 0.f;
#pragma unroll
        for (int j = 0; j < 4; ++j)
          if (j0 + j < P.rep) acc += x[j];
      }
      acc = opaque(acc * P.inv_rep);  // fp32 product, then one rounding to the q dtype
      v = DT == HALO_F32 ? acc
          : (DT == HALO_BF16 ? __uint_as_float((uint32_t)f32_to_bf16_rne(acc) << 16)
                             : f16_bits_to_f32(f32_to_f16_rne(acc)));
    }
    s_qg[i] = v;
  }
  __syncthreads();

  // score[i] = max over (row, h) of sum_d qg * kbar.  One thread per
  // (page, row, head) triple computes the whole dot product from 16-byte
  // loads that are all independent (one memory round trip per batch of
  // triples), products and sums rounded separately (no fused multiply-add),
  // summed in the scorer's slice order (below); the max over (row, h) is
  // folded in order.
  const int nrh = nrows * P.H_kv;
  const int triples = n * nrh;
  constexpr int esz = DT == HALO_F32 ? 4 : 2;
  constexpr int ep = 16 / esz;
  for (int i = tid; i < n; i += nthr) s_score[i] = -INFINITY;
  for (int t0 = 0; t0 < triples; t0 += kMaxDots) {
    const int nt = min(kMaxDots, triples - t0);
    for (int t = tid; t < nt; t += nthr) {
      const int tt = t0 + t;
      const int i = tt / nrh, rh = tt % nrh;
      const int r = rh / P.H_kv, h = rh % P.H_kv;
      const int64_t mb = (int64_t)(b0 + r) * P.msb + (int64_t)h * P.msh + (int64_t)s_chunk[i] * P.msp;
      const char* row = reinterpret_cast<const char*>(P.km) + mb * esz;
      const float* qg = s_qg + (r * P.H_kv + h) * Dq;
      // D is cut into G = D/16 slices; slice c holds elements
      // ep*(c + p*G) + e (p < 16/ep, e < ep), summed in (p, e) order; the G
      // slice sums are added as a balanced pairwise tree in slice order.  This
      // is the order of the fused selection in decode_attn.hip, whose slices
      // sit in G lanes and meet in an xor butterfly.
      constexpr int GC = DC / 16;  // compile-time slice count (0: runtime)
      const int G = DC ? GC : P.D / 16;
      float part[16];
      // compile-time D: every piece of the row is loaded before the first use
      uint4 rowv[DC ? (DC / 16) * (16 / ep) : 1];
      if constexpr (DC != 0) {
#pragma unroll
        for (int x = 0; x < GC * (16 / ep); ++x) rowv[x] = *reinterpret_cast<const uint4*>(row + x * 16);
      }
#pragma unroll
      for (int c = 0; c < (DC ? GC : 16); ++c) {
        if (!DC && c >= G) break;
        float a = 0.f;
#pragma unroll
        for (int p = 0; p < 16 / ep; ++p) {
          const uint4 v = DC ? rowv[(c + p * G) % (DC ? GC * (16 / ep) : 1)]
                             : *reinterpret_cast<const uint4*>(row + (c + p * G) * 16);
          float f[8];
          if constexpr (DT == HALO_F32) {
            f[0] = __uint_as_float(v.x); f[1] = __uint_as_float(v.y);
            f[2] = __uint_as_float(v.z); f[3] = __uint_as_float(v.w);
          } else if constexpr (DT == HALO_BF16) {
            f[0] = bf16_lo(v.x); f[1] = bf16_hi(v.x); f[2] = bf16_lo(v.y); f[3] = bf16_hi(v.y);
            f[4] = bf16_lo(v.z); f[5] = bf16_hi(v.z); f[6] = bf16_lo(v.w); f[7] = bf16_hi(v.w);
          } else {
            const uint32_t w[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
            for (int e = 0; e < 4; ++e) {
              f[2 * e] = f16_bits_to_f32((uint16_t)(w[e] & 0xffffu));
              f[2 * e + 1] = f16_bits_to_f32((uint16_t)(w[e] >> 16));
            }
          }
#pragma unroll
          for (int e = 0; e < ep; ++e) a = __fadd_rn(a, __fmul_rn(qg[ep * (c + p * G) + e], f[e]));
        }
        part[c] = a;
      }
      for (int w = 1; w < G; w <<= 1)
        for (int c = 0; c + w < G; c += 2 * w) part[c] = __fadd_rn(part[c], part[c + w]);
      const float acc = part[0];
      s_dot[t] = acc;
    }
    __syncthreads();
    for (int i = tid; i < n; i += nthr) {
      const int lo = max(i * nrh, t0) - t0, hi = min((i + 1) * nrh, t0 + nt) - t0;
      float best = s_score[i];
      for (int t = lo; t < hi; ++t) best = fmaxf(best, s_dot[t]);
      s_score[i] = best;
    }
    __syncthreads();
  }
  for (int i = tid; i < n; i += nthr) s_score[i] = (s_score[i] != s_score[i]) ? -INFINITY : s_score[i];
  __syncthreads();
  }  // !kGiven

  if (P.normalize) {
    // min and max over the eligible pages; x - min grows with x, so the
    // largest (attn - min) is (max - min).  Recency over all P_total pages:
    // exp(-(P-1-p)/refresh), / (sum + 1e-12), / (max + 1e-12).  The partial
    // sums of the 512 threads are added as a halving tree (t and t + 256, then
    // t + 128, ...), whose last six levels are a wave's shuffles.
    __shared__ float s_mn[8], s_mx[8], s_red[512];
    const int lane = tid & 63;
    float mn = INFINITY, mx = -INFINITY;
    for (int i = tid; i < n; i += nthr) {
      mn = fminf(mn, s_score[i]);
      mx = fmaxf(mx, s_score[i]);
    }
    mn = -wave_max(-mn);
    mx = wave_max(mx);
    const float dec = (float)max(P.refresh, 1);
    float rs = 0.f;
    for (int j = tid; j < P.P_total; j += nthr) rs += expf(-((float)(P.P_total - 1) - (float)j) / dec);
    s_red[tid] = rs;
    if (lane == 0) {
      s_mn[tid >> 6] = mn;
      s_mx[tid >> 6] = mx;
    }
    __syncthreads();
#pragma unroll
    for (int w = 0; w < 8; ++w) {
      mn = fminf(mn, s_mn[w]);
      mx = fmaxf(mx, s_mx[w]);
    }
    mx -= mn;
    float t4[4];
#pragma unroll
    for (int x = 0; x < 4; ++x) t4[x] = s_red[lane + 64 * x] + s_red[lane + 64 * x + 256];
    const float rtot = wave_sum((t4[0] + t4[2]) + (t4[1] + t4[3]));
    const float rsum = rtot + 1e-12f;
    // the largest recency term is the last page's exp(0) = 1
    const float rmax = 1.0f / rsum + 1e-12f;
    for (int i = tid; i < n; i += nthr) {
      float a = s_score[i] - mn;
      if (mx > 0.f) a = a / mx;
      const int pg = s_chunk[i];
      const float rec = (expf(-((float)(P.P_total - 1) - (float)pg) / dec) / rsum) / rmax;
      const float sink = pg < P.sink_pages ? 1.f : 0.f;
      float v = __fadd_rn(__fadd_rn(__fmul_rn(P.alpha, a), __fmul_rn(P.beta, rec)), __fmul_rn(P.gamma, sink));
      s_score[i] = (v != v) ? -INFINITY : v;
    }
    __syncthreads();
  }

  // Selected chunks in ascending order.  An ascending eligible list (a page
  // range, as the scorers pass it) is selected by wave 0 in registers; any
  // other order is ranked by comparing every pair (512 pages with their
  // scoring: 11.8 us, 38 in any other order).
  bool up = true;
  for (int i = tid; i < n; i += nthr) up = up && (i == 0 || s_chunk[i - 1] < s_chunk[i]);
  const bool asc = __syncthreads_and(up);
  const int n16 = (n + 15) & ~15;
  if (asc) {
    if (tid < 64) {
      if (n <= 64) select_ascending<1>(s_score, n, kk, tid, s_sel);
      else if (n <= 128) select_ascending<2>(s_score, n, kk, tid, s_sel);
      else if (n <= 256) select_ascending<4>(s_score, n, kk, tid, s_sel);
      else if (n <= 512) select_ascending<8>(s_score, n, kk, tid, s_sel);
      else select_ascending<16>(s_score, n, kk, tid, s_sel);
    }
  } else {
    // rank by (score desc, chunk asc); selected = rank < kk.  Candidates are
    // read four at a time (16-byte LDS reads, several in flight); entries past
    // n are padding that never outranks (-inf, index past every chunk).
    for (int i = n + tid; i < n16; i += nthr) {
      s_score[i] = -INFINITY;
      s_chunk[i] = 0x7fffffff;
      s_sel[i] = 0;
    }
    __syncthreads();
    for (int i = tid; i < n; i += nthr) {
      const float si = s_score[i];
      const int ei = s_chunk[i];
      int rank = 0;
      for (int j = 0; j < n16; j += 16) {
        float4 sv[4];
        int4 ev[4];
#pragma unroll
        for (int x = 0; x < 4; ++x) {
          sv[x] = *reinterpret_cast<const float4*>(&s_score[j + 4 * x]);
          ev[x] = *reinterpret_cast<const int4*>(&s_chunk[j + 4 * x]);
        }
#pragma unroll
        for (int x = 0; x < 4; ++x)
          rank += (beats(sv[x].x, ev[x].x, si, ei) ? 1 : 0) + (beats(sv[x].y, ev[x].y, si, ei) ? 1 : 0) +
                  (beats(sv[x].z, ev[x].z, si, ei) ? 1 : 0) + (beats(sv[x].w, ev[x].w, si, ei) ? 1 : 0);
      }
      s_sel[i] = rank < kk;
    }
  }
  __syncthreads();
  // Output slot = number of selected chunks with a smaller index.
  for (int i = tid; i < n; i += nthr) {
    if (P.score_out) P.score_out[(int64_t)sel * P.n_elig + i] = s_score[i];
    if (asc ? s_sel[i] < 0 : !s_sel[i]) continue;
    const int ei = s_chunk[i];
    int pos = asc ? s_sel[i] : 0;
    for (int j = asc ? n16 : 0; j < n16; j += 16) {
      int4 sv[4], ev[4];
#pragma unroll
      for (int x = 0; x < 4; ++x) {
        sv[x] = *reinterpret_cast<const int4*>(&s_sel[j + 4 * x]);
        ev[x] = *reinterpret_cast<const int4*>(&s_chunk[j + 4 * x]);
      }
#pragma unroll
      for (int x = 0; x < 4; ++x)
        pos += (sv[x].x && ev[x].x < ei) + (sv[x].y && ev[x].y < ei) + (sv[x].z && ev[x].z < ei) +
               (sv[x].w && ev[x].w < ei);
    }
    if (P.idx_out) P.idx_out[(int64_t)sel * P.k + pos] = ei;
    int rs = -1;
    if (P.residency != nullptr) {
      const int r = P.residency[(int64_t)sel * P.catalog_stride + ei];
      rs = (r >= 0 && r < P.n_slots) ? r : -1;
    }
    if (P.res_out) P.res_out[(int64_t)sel * P.k + pos] = rs;
    if (P.table) {
      halo_chunk_desc d = P.catalog[(int64_t)sel * P.catalog_stride + ei];
      if (rs >= 0) {  // rows, start, flags and batch stay the chunk's own
        const halo_chunk_desc& sd = P.slot_catalog[(int64_t)sel * P.n_slots + rs];
        d.k = sd.k;
        d.v = sd.v;
        d.k_stride_b = sd.k_stride_b;
        d.k_stride_h = sd.k_stride_h;
        d.k_stride_t = sd.k_stride_t;
        d.v_stride_b = sd.v_stride_b;
        d.v_stride_h = sd.v_stride_h;
        d.v_stride_t = sd.v_stride_t;
      }
      P.table[(int64_t)sel * P.table_stride + P.table_slot0 + pos] = d;
    }
  }
  // Unfilled slots: index -1 and an empty descriptor (T_c = 0, never read).
  for (int j = kk + tid; j < P.k; j += nthr) {
    if (P.idx_out) P.idx_out[(int64_t)sel * P.k + j] = -1;
    if (P.res_out) P.res_out[(int64_t)sel * P.k + j] = -1;
    if (P.table) {
      halo_chunk_desc e = {};
      e.k = nullptr;
      e.v = nullptr;
      e.T_c = 0;
      e.batch = P.per_row ? sel : -1;
      P.table[(int64_t)sel * P.table_stride + P.table_slot0 + j] = e;
    }
  }
}

}  // namespace halo

using namespace halo;

extern "C" int halo_chunk_means(const void* k, int64_t k_stride_b, int64_t k_stride_h, int64_t k_stride_t,
                                int dtype, int B, int H_kv, int D, int64_t row0, int page, int n_pages,
                                void* kmean, int64_t km_stride_b, int64_t km_stride_h, int64_t km_stride_p,
                                void* stream) {
  HALO_CHECK_ARG(k && kmean, "null pointer");
  HALO_CHECK_ARG(dtype == HALO_F32 || dtype == HALO_BF16 || dtype == HALO_F16, "bad dtype");
  HALO_CHECK_ARG(B > 0 && H_kv > 0 && D > 0 && page > 0 && n_pages >= 0 && row0 >= 0, "bad sizes");
  if (n_pages == 0) return HALO_OK;
  HALO_CHECK_ARG(D % (dtype == HALO_F32 ? 4 : 8) == 0 && D <= 256 * (dtype == HALO_F32 ? 4 : 8),
                 "head dim must fill whole 16-byte pieces");
  HALO_CHECK_ARG(reinterpret_cast<uintptr_t>(k) % 16 == 0 && (k_stride_t * elem_size(dtype)) % 16 == 0 &&
                 (k_stride_h * elem_size(dtype)) % 16 == 0 && (k_stride_b * elem_size(dtype)) % 16 == 0,
                 "key rows must be 16-byte aligned");
  const int64_t blocks = (int64_t)B * H_kv * n_pages;
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  const int es = elem_size(dtype);
  const int SL = D / (16 / es), RG = 256 / SL;
  // Whole pages per thread for pages of up to 16 rows, and longer ones that give
  // 64K threads, while a row group holds one row; 256 threads a page otherwise.
  // bf16, here / 256 threads a page: 16-row pages of 8 heads x 128, 8192 rows 4.0 /
  // 6.9 us, 32768 rows 15.0 / 20.4; 32-row pages of 8 heads x 64, 8192 rows (16K
  // threads) 4.4 / 4.4, 32768 rows 5.4 / 10.7.
  const int64_t total = blocks * SL;
  const bool col = page <= RG && (page <= 16 || total >= 65536);
  const int vec = reinterpret_cast<uintptr_t>(kmean) % 16 == 0 && (km_stride_b * es) % 16 == 0 &&
                  (km_stride_h * es) % 16 == 0 && (km_stride_p * es) % 16 == 0;
#define HALO_MEANS(DTV)                                                                                  \
  do {                                                                                                   \
    if (col)                                                                                             \
      hipLaunchKernelGGL(chunk_means_col_kernel<DTV>, dim3((unsigned)((total + 255) / 256)), dim3(256), 0, st, k, \
                         k_stride_b, k_stride_h, k_stride_t, H_kv, D, row0, page, n_pages, total, kmean, \
                         km_stride_b, km_stride_h, km_stride_p, vec);                                    \
    else if (DTV != HALO_F32 && page >= 32 * RG)                                                         \
      hipLaunchKernelGGL((chunk_means_kernel<DTV, DTV == HALO_F32 ? 0 : 32>), dim3((unsigned)blocks), dim3(256), 0, \
                         st, k, k_stride_b, k_stride_h, k_stride_t, H_kv, D, row0, page, n_pages, kmean, \
                         km_stride_b, km_stride_h, km_stride_p);                                         \
    else                                                                                                 \
      hipLaunchKernelGGL((chunk_means_kernel<DTV, DTV == HALO_F32 ? 0 : 8>), dim3((unsigned)blocks), dim3(256), 0, \
                         st, k, k_stride_b, k_stride_h, k_stride_t, H_kv, D, row0, page, n_pages, kmean, \
                         km_stride_b, km_stride_h, km_stride_p);                                         \
  } while (0)
  if (dtype == HALO_F32) HALO_MEANS(HALO_F32);
  else if (dtype == HALO_BF16) HALO_MEANS(HALO_BF16);
  else HALO_MEANS(HALO_F16);
#undef HALO_MEANS
  HALO_CHECK_HIP(hipGetLastError());
  return HALO_OK;
}

static int score_topk_impl(const void* q, int64_t q_stride_b, int64_t q_stride_h, int dtype,
                                     int B, int H, int H_kv, int D,
                                     const void* kmean, int64_t km_stride_b, int64_t km_stride_h,
                                     int64_t km_stride_p,
                                     const int32_t* eligible, int64_t elig_stride,
                                     const int32_t* n_elig_per_sel, int n_elig, int k, int per_row,
                                     int32_t* idx_out, float* score_out,
                                     const halo_chunk_desc* catalog, int64_t catalog_stride,
                                     halo_chunk_desc* table, int64_t table_stride, int table_slot0,
                                     int normalize, float alpha, float beta, float gamma,
                                     int refresh, int sink_pages, int P_total,
                                     const int32_t* residency, const halo_chunk_desc* slot_catalog, int n_slots,
                                     int32_t* res_out, float* workspace, void* stream) {
  HALO_CHECK_ARG(q && kmean && eligible, "null pointer");
  HALO_CHECK_ARG(residency == nullptr || (slot_catalog != nullptr && n_slots >= 1 && table != nullptr),
                 "staging needs slot_catalog, n_slots >= 1 and a table");
  HALO_CHECK_ARG(dtype == HALO_F32 || dtype == HALO_BF16 || dtype == HALO_F16, "bad dtype");
  HALO_CHECK_ARG(B > 0 && H > 0 && H_kv > 0 && H % H_kv == 0 && D > 0, "bad head sizes");
  HALO_CHECK_ARG(n_elig >= 0 && n_elig <= kMaxElig, "n_elig must be in [0, 1024]");
  HALO_CHECK_ARG(D % 16 == 0 && D <= 256, "head dim must be a multiple of 16, at most 256");
  HALO_CHECK_ARG(reinterpret_cast<uintptr_t>(kmean) % 16 == 0 &&
                 (km_stride_p * (dtype == HALO_F32 ? 4 : 2)) % 16 == 0 &&
                 (km_stride_h * (dtype == HALO_F32 ? 4 : 2)) % 16 == 0 &&
                 (km_stride_b * (dtype == HALO_F32 ? 4 : 2)) % 16 == 0,
                 "kmean rows must be 16-byte aligned");
  HALO_CHECK_ARG(k >= 0, "k must be >= 0");
  HALO_CHECK_ARG(table == nullptr || catalog != nullptr, "table needs a catalog");
  const int nrows = per_row ? 1 : B;
  HALO_CHECK_ARG((int64_t)nrows * H_kv * D <= kMaxQg, "B*H_kv*D too large for one selection");
  ScoreParams p;
  p.q = q;
  p.qsb = q_stride_b;
  p.qsh = q_stride_h;
  p.dtype = dtype;
  p.B = B;
  p.H = H;
  p.H_kv = H_kv;
  p.D = D;
  p.rep = H / H_kv;
  p.inv_rep = (float)(1.0 / (double)p.rep);
  p.km = kmean;
  p.msb = km_stride_b;
  p.msh = km_stride_h;
  p.msp = km_stride_p;
  p.elig = eligible;
  p.elig_stride = elig_stride;
  p.n_elig_per_sel = n_elig_per_sel;
  p.n_elig = n_elig;
  p.k = k;
  p.per_row = per_row;
  p.idx_out = idx_out;
  p.score_out = score_out;
  p.catalog = catalog;
  p.catalog_stride = catalog_stride;
  p.table = table;
  p.table_stride = table_stride;
  p.table_slot0 = table_slot0;
  p.normalize = normalize;
  p.alpha = alpha;
  p.beta = beta;
  p.gamma = gamma;
  p.refresh = refresh;
  p.sink_pages = sink_pages;
  p.P_total = P_total;
  p.residency = residency;
  p.slot_catalog = slot_catalog;
  p.n_slots = n_slots;
  p.res_out = res_out;
  HALO_CHECK_ARG(!normalize || P_total > 0, "P_total must be positive when normalising");
  const int n_sel = per_row ? B : 1;
  const int es = elem_size(dtype);
  p.qvec = reinterpret_cast<uintptr_t>(q) % 16 == 0 && (q_stride_b * es) % 16 == 0 && (q_stride_h * es) % 16 == 0;
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  // Scores on their own grid, held by the workspace until the selection reads
  // them, where one CU would walk the means for longer than a launch costs.
  // Own grid / one workgroup, at 8 heads x 128 bf16: 16 pages 8.3 / 8.4 us, 32
  // 8.9 / 9.1, 64 8.8 / 10.8, 512 11.8 / 38; at 4 heads x 64: 64 pages 7.3 / 6.6,
  // 128 7.6 / 7.8, 512 9.9 / 15.3.
  p.raw = workspace;
  if (workspace != nullptr && (int64_t)n_elig * nrows * H_kv * D >= 32768) {
    const int G = D / 16;
    const int G2 = G <= 1 ? 1 : G <= 2 ? 2 : G <= 4 ? 4 : G <= 8 ? 8 : 16;
    const int tiles = (n_elig + 64 / G2 - 1) / (64 / G2);
    const dim3 grid((unsigned)(n_sel * tiles));
#define HALO_PAGES(DTV)                                                                                        \
  do {                                                                                                         \
    if (G2 == 1) hipLaunchKernelGGL((score_pages_kernel<DTV, 1>), grid, dim3(256), 0, st, p, tiles);           \
    else if (G2 == 2) hipLaunchKernelGGL((score_pages_kernel<DTV, 2>), grid, dim3(256), 0, st, p, tiles);      \
    else if (G2 == 4) hipLaunchKernelGGL((score_pages_kernel<DTV, 4>), grid, dim3(256), 0, st, p, tiles);      \
    else if (G2 == 8) hipLaunchKernelGGL((score_pages_kernel<DTV, 8>), grid, dim3(256), 0, st, p, tiles);      \
    else hipLaunchKernelGGL((score_pages_kernel<DTV, 16>), grid, dim3(256), 0, st, p, tiles);                  \
    hipLaunchKernelGGL((score_topk_kernel<DTV, -1>), dim3(n_sel), dim3(512), 0, st, p);                        \
  } while (0)
    if (dtype == HALO_F32) HALO_PAGES(HALO_F32);
    else if (dtype == HALO_BF16) HALO_PAGES(HALO_BF16);
    else HALO_PAGES(HALO_F16);
#undef HALO_PAGES
    HALO_CHECK_HIP(hipGetLastError());
    return HALO_OK;
  }
#define HALO_SCORE(DTV)                                                                                    \
  do {                                                                                                     \
    if (D == 64) hipLaunchKernelGGL((score_topk_kernel<DTV, 64>), dim3(n_sel), dim3(512), 0, st, p);       \
    else if (D == 128) hipLaunchKernelGGL((score_topk_kernel<DTV, 128>), dim3(n_sel), dim3(512), 0, st, p); \
    else if (D == 256) hipLaunchKernelGGL((score_topk_kernel<DTV, 256>), dim3(n_sel), dim3(512), 0, st, p); \
    else hipLaunchKernelGGL((score_topk_kernel<DTV, 0>), dim3(n_sel), dim3(512), 0, st, p);                \
  } while (0)
  if (dtype == HALO_F32) HALO_SCORE(HALO_F32);
  else if (dtype == HALO_BF16) HALO_SCORE(HALO_BF16);
  else HALO_SCORE(HALO_F16);
#undef HALO_SCORE
  HALO_CHECK_HIP(hipGetLastError());
  return HALO_OK;
}

extern "C" int halo_chunk_score_topk(const void* q, int64_t q_stride_b, int64_t q_stride_h, int dtype,
                                     int B, int H, int H_kv, int D,
                                     const void* kmean, int64_t km_stride_b, int64_t km_stride_h,
                                     int64_t km_stride_p,
                                     const int32_t* eligible, int64_t elig_stride,
                                     const int32_t* n_elig_per_sel, int n_elig, int k, int per_row,
                                     int32_t* idx_out, float* score_out,
                                     const halo_chunk_desc* catalog, int64_t catalog_stride,
                                     halo_chunk_desc* table, int64_t table_stride, int table_slot0,
                                     int normalize, float alpha, float beta, float gamma,
                                     int refresh, int sink_pages, int P_total,
                                     void* stream) {
  return score_topk_impl(q, q_stride_b, q_stride_h, dtype, B, H, H_kv, D, kmean, km_stride_b, km_stride_h,
                         km_stride_p, eligible, elig_stride, n_elig_per_sel, n_elig, k, per_row, idx_out, score_out,
                         catalog, catalog_stride, table, table_stride, table_slot0, normalize, alpha, beta, gamma,
                         refresh, sink_pages, P_total, nullptr, nullptr, 0, nullptr, nullptr, stream);
}

extern "C" int halo_chunk_score_topk_staged(const void* q, int64_t q_stride_b, int64_t q_stride_h, int dtype,
                                            int B, int H, int H_kv, int D,
                                            const void* kmean, int64_t km_stride_b, int64_t km_stride_h,
                                            int64_t km_stride_p,
                                            const int32_t* eligible, int64_t elig_stride,
                                            const int32_t* n_elig_per_sel, int n_elig, int k, int per_row,
                                            int32_t* idx_out, float* score_out,
                                            const halo_chunk_desc* catalog, int64_t catalog_stride,
                                            halo_chunk_desc* table, int64_t table_stride, int table_slot0,
                                            const int32_t* residency, const halo_chunk_desc* slot_catalog,
                                            int n_slots, int32_t* res_out, void* stream) {
  HALO_CHECK_ARG(residency != nullptr, "residency is NULL: use halo_chunk_score_topk");
  return score_topk_impl(q, q_stride_b, q_stride_h, dtype, B, H, H_kv, D, kmean, km_stride_b, km_stride_h,
                         km_stride_p, eligible, elig_stride, n_elig_per_sel, n_elig, k, per_row, idx_out, score_out,
                         catalog, catalog_stride, table, table_stride, table_slot0, 0, 1.f, 0.f, 0.f, 64, 0, 1,
                         residency, slot_catalog, n_slots, res_out, nullptr, stream);
}

extern "C" int halo_chunk_score_topk_ws(const void* q, int64_t q_stride_b, int64_t q_stride_h, int dtype,
                                        int B, int H, int H_kv, int D,
                                        const void* kmean, int64_t km_stride_b, int64_t km_stride_h,
                                        int64_t km_stride_p,
                                        const int32_t* eligible, int64_t elig_stride,
                                        const int32_t* n_elig_per_sel, int n_elig, int k, int per_row,
                                        int32_t* idx_out, float* score_out,
                                        const halo_chunk_desc* catalog, int64_t catalog_stride,
                                        halo_chunk_desc* table, int64_t table_stride, int table_slot0,
                                        int normalize, float alpha, float beta, float gamma,
                                        int refresh, int sink_pages, int P_total,
                                        const int32_t* residency, const halo_chunk_desc* slot_catalog,
                                        int n_slots, int32_t* res_out, float* workspace, void* stream) {
  HALO_CHECK_ARG(residency == nullptr || !normalize, "the staged selection uses raw scores");
  return score_topk_impl(q, q_stride_b, q_stride_h, dtype, B, H, H_kv, D, kmean, km_stride_b, km_stride_h,
                         km_stride_p, eligible, elig_stride, n_elig_per_sel, n_elig, k, per_row, idx_out, score_out,
                         catalog, catalog_stride, table, table_stride, table_slot0, normalize, alpha, beta, gamma,
                         refresh, sink_pages, P_total, residency, slot_catalog, n_slots, res_out, workspace, stream);
}
