// llmk_device.h — what the sampling kernels share on the device: geometry and
// workspace, wave and workgroup helpers, history tables, logit loads, the
// sorted-list semantics, the exact sequential sums in binades and the sorts.
// Included by llmk_sampler.hip, which holds the kernels.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "llmk_numerics.h"
#include "llmk_sampler.h"

namespace llmk {


// Explicit address spaces: LDS (3) and global (1).  Pointers that pass
// through structs or function parameters would otherwise become generic
// (flat) pointers, whose loads wait on both the vector-memory and the LDS
// counters.
#define LDS __attribute__((address_space(3)))
#define GLB __attribute__((address_space(1)))
template <class T>
__device__ __forceinline__ GLB T* G(T* p) { return (GLB T*)p; }
template <class T>
__device__ __forceinline__ const GLB T* G(const T* p) { return (const GLB T*)p; }

typedef float f2v __attribute__((ext_vector_type(2)));
typedef float f4v __attribute__((ext_vector_type(4)));
typedef uint32_t u2v __attribute__((ext_vector_type(2)));
typedef uint32_t u4v __attribute__((ext_vector_type(4)));

constexpr uint32_t TILE = 1024;      // canonical vocabulary tile
constexpr int WAVE = 64;
constexpr int NW = 16;               // waves per workgroup
constexpr int NT = NW * WAVE;        // 1024 threads
constexpr uint32_t NBINS = 4096;     // fine histogram bins: key >> 20
constexpr uint32_t BIN_SHIFT = 20;
constexpr uint32_t CBIN_SHIFT = 26;  // coarse bins: key >> 26 (64 bins)
constexpr uint32_t U_MAX = 8192;     // distinct history tokens per segment
constexpr uint32_t CAND_CAP = 8192;  // candidate entries per workgroup
constexpr uint32_t SORT_CAP = 4096;  // candidates sorted in finalize
constexpr uint32_t KMAX = 1024;      // largest top-k served by the fast path
constexpr uint32_t KCAND_NOK = 1024; // candidate target when top-k is off
constexpr uint32_t MAX_TILES = 1024; // max_vocab <= 2^20
constexpr uint32_t CHUNK_TILES = 16;  // tiles per history chunk (segments are whole chunks)
constexpr uint32_t MAX_CHUNKS = MAX_TILES / CHUNK_TILES;
constexpr uint32_t MAX_SLOTS = MAX_TILES + MAX_CHUNKS;  // partials per row: tiles, then chunks
constexpr uint32_t LCAP = 1024;       // candidates a single-segment row keeps in LDS
constexpr uint32_t MAX_SEG = 64;     // segments per row
constexpr uint32_t MAX_WGS = 4096;   // candidate-buffer pool entries
constexpr uint32_t SLOW_SLOTS = 512;  // most global scratch slots of the slow path
constexpr uint32_t SLOW_BINS = 2048; // slow path: bins of the processed logits
constexpr uint32_t EMPTY = 0xffffffffu;
constexpr float NEG_INF = -__builtin_huge_valf();
constexpr float LOG2E_F = 0x1.715476p+0f;  // the slow path's bins of (l - L)/T, in octaves
// The exact S of rows that fail the band check, on many workgroups (phase 1)
constexpr uint32_t XS_JOBS = 8;                        // rows per call
constexpr uint32_t XS_W = 16 * TILE;                   // a window: 16 segments of a tile
constexpr uint32_t XS_SAVE = 2 * MAX_SLOTS + 2 * LCAP;  // LDS partials + candidates
constexpr uint32_t XS_JOB_WORDS = 32;
constexpr uint32_t XS_PRE = 2 + XS_JOBS;                // xs_ctl: window 0's (sum, tag) per job
constexpr uint32_t XS_CTL_WORDS = XS_PRE + 2 * XS_JOBS;

// Words a workgroup passes from one phase to the next past the dynamic
// shared memory, which each phase lays out afresh (static LDS).
__shared__ uint32_t g_bcast[4];

enum : uint32_t { MODE_INVALID = 0, MODE_GREEDY = 1, MODE_SAMPLE = 2 };
enum : uint32_t { FLAG_OVERFLOW = 1u, FLAG_HIST_OVERFLOW = 2u, FLAG_NAN = 4u };

struct Args {
  const void* logits;
  int32_t dtype;
  float sc_m1, sc_cap;  // softcap: 1/cap and cap in the logits' dtype (DT & SOFTCAP)
  uint32_t B, V;
  uint64_t stride;
  const float *T, *top_p, *min_p, *rp, *pp, *fp;
  const int32_t* top_k;
  const uint32_t *hoff, *htok, *mask;
  const uint32_t* hlen;  // optional: row b's history is htok[hoff[b] .. hoff[b] + hlen[b])
  const uint32_t* hcnt;  // optional: occurrences of each htok entry (the count-table form)
  uint32_t mask_words;
  const float* u;
  uint32_t *out_tok, *out_ids, *out_cnt;
  float* out_probs;
  uint32_t out_cap;
  uint32_t G, tps, ntiles, nchunks;
  // single-segment rows: LDS word offsets of the kept partials (MAX_SLOTS
  // f2v) and candidates (LCAP u2v), past both the stream and finalize layouts
  uint32_t lds_part, lds_cand;
  uint32_t xcd_map;  // 1: the segments of a row share an XCD
  // apply_top_p: per row, the last kept entry's index, the kept count and
  // the m and S its probabilities used; top_p clamped to [0, 1], NaN read as 1
  // (the mask form's no-op, not an invalid row)
  u4v* cut;
  uint32_t tp_clamp;
  // 0: the sampling launch; 1: the launch after it that sums the reference's
  // S, window by window on many workgroups, for the rows whose band check
  // failed (up to xs_cap rows per call; the sampling launch does the rest
  // itself)
  uint32_t phase, xs_cap;
  uint32_t xs_lds;  // phase 1's dynamic LDS in words
  // the call's parity: its jobs are counted in xs_ctl[epoch & 1], and its
  // sampling launch clears the other count for the next call
  uint32_t epoch;
  // phase 1's bounded waits (for the sums of earlier windows, for window
  // 0's own walk): at most this many polls (XS_SPIN; a test sets 0 to take
  // the paths where a wait runs out)
  uint32_t xs_spin;
};

struct Ws {
  uint32_t* row_arrive;  // [max_batch]
  f2v* tile_part;        // [max_batch][MAX_SLOTS]: max, sum (or first argmax) per slot
  u4v* seg_meta;         // [pool]: count, beta, flags, -
  u2v* cand;             // [pool][CAND_CAP]: value bits, index
  uint32_t* slow_lock;   // [slow_slots]
  uint64_t* slow_keys;   // [slow_slots][3][max_vocab]
  float* slow_p;         // [slow_slots][max_vocab]
  uint32_t* slow_idx;    // [slow_slots][max_vocab]
  uint32_t* status;      // [1]
  u4v* cut;              // [max_batch]: apply_top_p's cut per row
  uint32_t* mtok;        // [max_batch]: apply_top_p's (unused) draws
  float* zu;             // [max_batch]: zeros, its uniforms
  // the exact S of deferred rows (phase 1): jobs posted, workgroups done and
  // per job its arrival count; the jobs; per job and window its sum and that
  // sum's flag; per job and segment its pairs and terms; per job the
  // single-segment row's LDS partials and candidates
  uint32_t* xs_ctl;      // [XS_CTL_WORDS]: job counts of even / odd calls, arrivals,
                         // window 0's (sum, tag) per job
  uint32_t* xs_job;      // [XS_JOBS][XS_JOB_WORDS]
  float* xs_wsum;        // [XS_JOBS][xs_maxw]
  uint32_t* xs_wflag;    // [XS_JOBS][xs_maxw]: the tag of the call it was summed in
  uint32_t* xs_meta;     // [XS_JOBS][xs_maxw * 16][8]
  float* xs_terms;       // [XS_JOBS][xs_maxw * 16][TILE]
  uint32_t* xs_runs;     // [XS_JOBS][xs_maxw * 16][XS_RUNW]
  uint32_t* xs_save;     // [XS_JOBS][XS_SAVE]
  uint32_t xs_maxw;
  uint32_t max_vocab;
  uint32_t slow_slots;   // min(max_batch, SLOW_SLOTS): rows b, b + slow_slots, ... share one
};

struct RowP {
  float T, top_p, min_p, rp, pp, fp;
  int32_t K;
  uint32_t mode;
  uint32_t Kc;  // candidate target; 0 = candidate path impossible
};

__device__ __forceinline__ bool finitef(float x) { return __builtin_isfinite(x); }

// Defaults of absent per-row arrays (SampleParams, llm-core/src/types.rs:
// 186-195), read in place of the array: every load is then unconditional.
__constant__ float kOneF = 1.0f;
__constant__ uint32_t kZeroU = 0u;
template <class T>
__device__ __forceinline__ const T* row_or(const T* p, uint32_t b, const void* dflt) {
  return p ? p + b : (const T*)dflt;
}

// The row's parameters, uniform, history extent and uniform as loaded: all
// requested together, before anything branches on one of them, so that they
// cost one round trip.
struct RowIn {
  float T, top_p, min_p, rp, pp, fp, u;
  int32_t K;
  uint32_t h0, hn, hl;
};
__device__ __forceinline__ RowIn load_row(const Args& a, uint32_t b) {
  RowIn r;
  r.T = *G(row_or(a.T, b, &kOneF));
  r.top_p = *G(row_or(a.top_p, b, &kOneF));
  r.min_p = *G((const float*)row_or(a.min_p, b, &kZeroU));
  r.rp = *G(row_or(a.rp, b, &kOneF));
  r.pp = *G((const float*)row_or(a.pp, b, &kZeroU));
  r.fp = *G((const float*)row_or(a.fp, b, &kZeroU));
  r.K = *G((const int32_t*)row_or(a.top_k, b, &kZeroU));
  r.u = *G(a.u + b);
  r.h0 = *G(row_or(a.hoff, b, &kZeroU));
  r.hn = *G(row_or(a.hoff, b + 1, &kZeroU));
  r.hl = *G(row_or(a.hlen, b, &kZeroU));
  return r;
}

__device__ __forceinline__ RowP row_params(const Args& a, const RowIn& in) {
  RowP r;
  r.T = in.T;
  r.top_p = in.top_p;
  if (a.tp_clamp) r.top_p = r.top_p < 0.0f ? 0.0f : (r.top_p < 1.0f ? r.top_p : 1.0f);
  r.min_p = in.min_p;
  r.rp = in.rp;
  r.pp = in.pp;
  r.fp = in.fp;
  r.K = in.K;
  const bool bad = !finitef(r.T) || r.K < 0 || !finitef(r.top_p) ||
                   !finitef(r.min_p) || !(r.min_p >= 0.0f) || !finitef(r.rp) ||
                   !finitef(r.pp) || !finitef(r.fp);
  r.mode = bad ? MODE_INVALID : (r.T <= 1e-5f ? MODE_GREEDY : MODE_SAMPLE);
  const bool topk_on = r.K > 0 && (uint32_t)r.K < a.V;
  // top-k rows gather one candidate past the K-th (the band check compares
  // the two)
  r.Kc = topk_on ? ((uint32_t)r.K <= KMAX ? (uint32_t)r.K + 1u : 0u) : KCAND_NOK;
  return r;
}

// ---------------------------------------------------------------------------
// Wave64 helpers on DPP (row_shr within 16-lane rows, row_bcast across rows)
// ---------------------------------------------------------------------------
template <int CTRL, int RM, bool BC>
__device__ __forceinline__ float dppf(float old, float src) {
  return __int_as_float(__builtin_amdgcn_update_dpp(
      __float_as_int(old), __float_as_int(src), CTRL, RM, 0xf, BC));
}
template <int CTRL, int RM, bool BC>
__device__ __forceinline__ uint32_t dppu(uint32_t old, uint32_t src) {
  return (uint32_t)__builtin_amdgcn_update_dpp((int)old, (int)src, CTRL, RM, 0xf, BC);
}
__device__ __forceinline__ uint32_t umax_(uint32_t a, uint32_t b) { return a > b ? a : b; }
__device__ __forceinline__ float bcast63f(float x) {
  return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(x), 63));
}
__device__ __forceinline__ uint32_t bcast63u(uint32_t x) {
  return (uint32_t)__builtin_amdgcn_readlane((int)x, 63);
}

// Sum of lanes 0..63 as a balanced binary tree over contiguous lanes
// ((x0+x1)+(x2+x3))+...; the root forms in lane 63 and is broadcast.
__device__ __forceinline__ float wave_tree_sum(float x) {
  x = x + dppf<0x111, 0xf, true>(0.0f, x);
  x = x + dppf<0x112, 0xf, true>(0.0f, x);
  x = x + dppf<0x114, 0xf, true>(0.0f, x);
  x = x + dppf<0x118, 0xf, true>(0.0f, x);
  x = x + dppf<0x142, 0xa, false>(0.0f, x);
  x = x + dppf<0x143, 0xc, false>(0.0f, x);
  return bcast63f(x);
}
// Maximum over the lanes of x (never NaN): on order-preserving keys, whose
// maximum needs no NaN handling, so each step is one v_max_u32 with DPP;
// lanes outside a row read 0, the smallest key.
__device__ __forceinline__ float wave_max(float x) {
  const uint32_t b = __float_as_uint(x);
  uint32_t k = b ^ ((uint32_t)((int32_t)b >> 31) | 0x80000000u);
  k = umax_(k, dppu<0x111, 0xf, true>(0u, k));
  k = umax_(k, dppu<0x112, 0xf, true>(0u, k));
  k = umax_(k, dppu<0x114, 0xf, true>(0u, k));
  k = umax_(k, dppu<0x118, 0xf, true>(0u, k));
  k = umax_(k, dppu<0x142, 0xa, true>(0u, k));
  k = umax_(k, dppu<0x143, 0xc, true>(0u, k));
  const uint32_t r = bcast63u(k);
  return __uint_as_float((r & 0x80000000u) ? (r & 0x7fffffffu) : ~r);
}
__device__ __forceinline__ uint32_t umin(uint32_t a, uint32_t b) { return a < b ? a : b; }
__device__ __forceinline__ uint32_t wave_min_u32(uint32_t x) {
  x = umin(x, dppu<0x111, 0xf, false>(x, x));
  x = umin(x, dppu<0x112, 0xf, false>(x, x));
  x = umin(x, dppu<0x114, 0xf, false>(x, x));
  x = umin(x, dppu<0x118, 0xf, false>(x, x));
  x = umin(x, dppu<0x142, 0xa, false>(x, x));
  x = umin(x, dppu<0x143, 0xc, false>(x, x));
  return bcast63u(x);
}
__device__ __forceinline__ uint32_t umax(uint32_t a, uint32_t b) { return a > b ? a : b; }
__device__ __forceinline__ uint32_t wave_max_u32(uint32_t x) {
  x = umax(x, dppu<0x111, 0xf, true>(0u, x));
  x = umax(x, dppu<0x112, 0xf, true>(0u, x));
  x = umax(x, dppu<0x114, 0xf, true>(0u, x));
  x = umax(x, dppu<0x118, 0xf, true>(0u, x));
  x = umax(x, dppu<0x142, 0xa, true>(0u, x));
  x = umax(x, dppu<0x143, 0xc, true>(0u, x));
  return bcast63u(x);
}
// Inclusive prefix sum over lanes.
__device__ __forceinline__ uint32_t wave_incl_scan(uint32_t x) {
  x += dppu<0x111, 0xf, true>(0u, x);
  x += dppu<0x112, 0xf, true>(0u, x);
  x += dppu<0x114, 0xf, true>(0u, x);
  x += dppu<0x118, 0xf, true>(0u, x);
  x += dppu<0x142, 0xa, false>(0u, x);
  x += dppu<0x143, 0xc, false>(0u, x);
  return x;
}
__device__ __forceinline__ uint32_t lanes_below(uint64_t m) {
  return __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32),
                                   __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u));
}

// Block-wide exclusive scan of one value per thread (NT threads).
__device__ __forceinline__ uint32_t block_excl_scan(uint32_t x, LDS uint32_t* red, uint32_t& total) {
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const uint32_t incl = wave_incl_scan(x);
  if (lane == 63) red[wv] = incl;
  __syncthreads();
  uint32_t off = 0, tot = 0;
#pragma unroll
  for (int i = 0; i < NW; ++i) {
    const uint32_t c = red[i];
    off += (i < wv) ? c : 0u;
    tot += c;
  }
  __syncthreads();
  total = tot;
  return off + incl - x;
}
__device__ __forceinline__ float block_max(float x, LDS float* red) {
  x = wave_max(x);
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  if (lane == 0) red[wv] = x;
  __syncthreads();
  float r = red[0];
#pragma unroll
  for (int i = 1; i < NW; ++i) r = fmaxf(r, red[i]);
  __syncthreads();
  return r;
}
__device__ __forceinline__ uint32_t block_min_u32(uint32_t x, LDS uint32_t* red) {
  x = wave_min_u32(x);
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  if (lane == 0) red[wv] = x;
  __syncthreads();
  uint32_t r = red[0];
#pragma unroll
  for (int i = 1; i < NW; ++i) r = umin(r, red[i]);
  __syncthreads();
  return r;
}

// Wait until this wave's global stores have reached L2 (vmcnt(0)).
__device__ __forceinline__ void wait_stores() { __builtin_amdgcn_s_waitcnt(0x0f70); }

// ---------------------------------------------------------------------------
// History: bitmap over a vocabulary range, popcount prefix, penalised values
// ---------------------------------------------------------------------------
// Penalties on one logit of a history token (sampler.rs:139-143, then the
// presence/frequency formula of llm-tests/tests/mlc_parity.rs:1083).
__device__ __forceinline__ float penalize(float x, const RowP& P,
                                          uint32_t count) {
  if (P.rp != 1.0f) x = (x > 0.0f) ? x / P.rp : x * P.rp;
  if (P.pp != 0.0f || P.fp != 0.0f) {
    const float cf = (float)count * P.fp;
    x = x - (P.pp + cf);
  }
  return x;
}

// A 16-bit logit (bf16 or f16 bits) as f32, exactly.
template <int DT>
__device__ __forceinline__ float cvt16(uint32_t h) {
  if ((DT & 3) == LLMK_BF16) return __uint_as_float(h << 16);
  return (float)__builtin_bit_cast(_Float16, (uint16_t)h);
}

// Template flag on the dtype: the logits are the lm_head output before
// final_logit_softcapping, capped as they are read.  1/cap and cap (in the
// logits' dtype) sit in LDS, written before the kernel's first barrier.
constexpr int SOFTCAP = 4;
__shared__ float g_softcap[2];
// f32 -> the logits' dtype, round to nearest even (NaN stays NaN)
template <int DT>
__device__ __forceinline__ float round_dt(float x) {
  if ((DT & 3) == LLMK_BF16) {
    uint32_t u = __float_as_uint(x);
    if ((u & 0x7fffffffu) > 0x7f800000u) return __uint_as_float((u | 0x00400000u) & 0xffff0000u);
    u += 0x7fffu + ((u >> 16) & 1u);
    return __uint_as_float(u & 0xffff0000u);
  }
  if ((DT & 3) == LLMK_F16) return (float)(_Float16)x;
  return x;
}
// final_logit_softcapping as candle evaluates it on the logits tensor
// (candle.rs:1803-1807): (x / cap).tanh() * cap, where dividing or
// multiplying a tensor by a scalar is its affine map x * m + 0 (m = 1/cap or
// cap, as the dtype) and tanh is glibc's tanhf; in a 16-bit dtype every
// operation rounds to it.
template <int DT>
__device__ __forceinline__ float softcap(float x) {
  if (!(DT & SOFTCAP)) return x;
  float y = round_dt<DT>(x * g_softcap[0]);
  y = round_dt<DT>(y + 0.0f);
  float t = round_dt<DT>(tanh_ref(y));
  t = round_dt<DT>(t * g_softcap[1]);
  return round_dt<DT>(t + 0.0f);
}
template <int DT>
__device__ __forceinline__ void softcap_init(const Args& a) {
  if (DT & SOFTCAP)
    if (threadIdx.x < 2) g_softcap[threadIdx.x] = threadIdx.x ? a.sc_cap : a.sc_m1;
}

template <int DT>
__device__ __forceinline__ float load_logit(const void* row, uint32_t e) {
  if ((DT & 3) == LLMK_F32) return softcap<DT>(G((const float*)row)[e]);
  return softcap<DT>(cvt16<DT>(G((const uint16_t*)row)[e]));
}

struct Hist {
  LDS uint32_t* bitmap;  // nwords
  LDS uint16_t* pre;     // nwords: distinct history tokens in words before
  LDS float* pen;        // U_MAX: penalised logit by rank (counts while building)
  LDS uint32_t* tokr;    // U_MAX: token of each rank
  uint32_t lo;
  __device__ __forceinline__ uint32_t rank(uint32_t t) const {
    const uint32_t o = t - lo, w = o >> 5;
    return pre[w] + __popc(bitmap[w] & ((1u << (o & 31)) - 1u));
  }
};

__host__ __device__ inline size_t hist_lds_words(uint32_t nwords) {
  return (size_t)((nwords + 3) & ~3u) + (size_t)(((nwords + 1) / 2 + 3) & ~3u) + 2 * U_MAX;
}
__device__ __forceinline__ void hist_carve(Hist& h, LDS uint32_t* base, uint32_t nwords) {
  h.bitmap = base;
  h.pre = (LDS uint16_t*)(base + ((nwords + 3) & ~3u));
  h.pen = (LDS float*)(base + ((nwords + 3) & ~3u) + (((nwords + 1) / 2 + 3) & ~3u));
  h.tokr = (LDS uint32_t*)(h.pen + U_MAX);
}

// Ranks of the segment's history tokens once its bitmap is complete, built
// by the first nw waves, which call sync() together twice (the second time
// at the end).  Thread i of them owns a contiguous run of bitmap words: the
// run's popcount, an exclusive scan over the threads, then pre[w] = history
// tokens in the words before w and tokr[r] = the token of rank r (tokens in
// increasing order).  Tokens of rank >= U_MAX are cleared from the bitmap
// and the overflow flag is raised: they are then ordinary, unpenalised
// tokens.  Returns the number of ranks (<= U_MAX).  wtot: nw words.
template <class Sync>
__device__ __forceinline__ uint32_t build_ranks(const Hist& h, uint32_t nwords,
                                                LDS uint32_t* wtot, LDS uint32_t* flags,
                                                uint32_t nw, Sync& sync) {
  const uint32_t tid = threadIdx.x, lane = tid & 63u, wv = tid >> 6;
  const uint32_t per = (nwords + 64u * nw - 1u) / (64u * nw);
  const uint32_t w0 = tid * per < nwords ? tid * per : nwords;
  const uint32_t w1 = w0 + per < nwords ? w0 + per : nwords;
  // runs of up to 8 words are read at once (taken branches cost a lone
  // wave more than the reads)
  uint32_t c = 0;
  for (uint32_t b0 = w0; b0 < w1; b0 += 8) {
    uint32_t x[8];
#pragma unroll
    for (uint32_t q = 0; q < 8; ++q) x[q] = b0 + q < w1 ? h.bitmap[b0 + q] : 0u;
#pragma unroll
    for (uint32_t q = 0; q < 8; ++q) c += (uint32_t)__popc(x[q]);
  }
  const uint32_t incl = wave_incl_scan(c);
  if (lane == 63) wtot[wv] = incl;
  sync();
  uint32_t r = incl - c, total = 0;
  for (uint32_t i = 0; i < nw; ++i) {
    const uint32_t t = wtot[i];
    r += i < wv ? t : 0u;
    total += t;
  }
  for (uint32_t b0 = w0; b0 < w1; b0 += 8) {
    uint32_t x[8];
#pragma unroll
    for (uint32_t q = 0; q < 8; ++q) x[q] = b0 + q < w1 ? h.bitmap[b0 + q] : 0u;
#pragma unroll
    for (uint32_t q = 0; q < 8; ++q) {
      const uint32_t wi = b0 + q;
      uint32_t bits = x[q];
      const uint32_t cw = (uint32_t)__popc(bits);
      if (wi < w1) h.pre[wi] = (uint16_t)(r < U_MAX ? r : U_MAX);
      if (wi < w1 && r + cw > U_MAX) {  // keep the first U_MAX - r tokens of the word
        const uint32_t keep = r < U_MAX ? U_MAX - r : 0u;
        uint32_t kept = 0, rest = bits;
        for (uint32_t k = 0; k < keep; ++k) {
          kept |= rest & (0u - rest);
          rest &= rest - 1u;
        }
        bits = kept;
        h.bitmap[wi] = kept;
      }
      // two tokens per step
      while (bits) {
        const uint32_t b1 = (uint32_t)__builtin_ctz(bits);
        bits &= bits - 1u;
        h.tokr[r++] = h.lo + 32u * wi + b1;
        if (bits) {
          const uint32_t b2 = (uint32_t)__builtin_ctz(bits);
          bits &= bits - 1u;
          h.tokr[r++] = h.lo + 32u * wi + b2;
        }
      }
    }
  }
  if (total > U_MAX && tid == 0) __atomic_fetch_or(flags, FLAG_HIST_OVERFLOW, __ATOMIC_RELAXED);
  sync();
  return total < U_MAX ? total : U_MAX;
}

// pre[w] = history tokens in the bitmap words before w, built by the first nw
// waves from contiguous runs of words (a popcount per run, an exclusive scan
// over the threads), which call sync() together twice.  Returns the number
// of tokens, which the caller knows to be at most U_MAX.  wtot: nw words.
template <class Sync>
__device__ __forceinline__ uint32_t build_pre(const Hist& h, uint32_t nwords,
                                              LDS uint32_t* wtot, uint32_t nw, Sync& sync) {
  const uint32_t tid = threadIdx.x, lane = tid & 63u, wv = tid >> 6;
  const uint32_t per = (nwords + 64u * nw - 1u) / (64u * nw);
  const uint32_t w0 = tid * per < nwords ? tid * per : nwords;
  const uint32_t w1 = w0 + per < nwords ? w0 + per : nwords;
  uint32_t c = 0;
  for (uint32_t b0 = w0; b0 < w1; b0 += 8) {
    uint32_t x[8];
#pragma unroll
    for (uint32_t q = 0; q < 8; ++q) x[q] = b0 + q < w1 ? h.bitmap[b0 + q] : 0u;
#pragma unroll
    for (uint32_t q = 0; q < 8; ++q) c += (uint32_t)__popc(x[q]);
  }
  const uint32_t incl = wave_incl_scan(c);
  if (lane == 63) wtot[wv] = incl;
  sync();
  uint32_t r = incl - c, total = 0;
  for (uint32_t i = 0; i < nw; ++i) {
    const uint32_t t = wtot[i];
    r += i < wv ? t : 0u;
    total += t;
  }
  for (uint32_t b0 = w0; b0 < w1; b0 += 8) {
    uint32_t x[8];
#pragma unroll
    for (uint32_t q = 0; q < 8; ++q) x[q] = b0 + q < w1 ? h.bitmap[b0 + q] : 0u;
#pragma unroll
    for (uint32_t q = 0; q < 8; ++q) {
      if (b0 + q < w1) h.pre[b0 + q] = (uint16_t)r;
      r += (uint32_t)__popc(x[q]);
    }
  }
  sync();
  return total;
}

// A barrier among waves 0 .. n-1 while the others run on: an arrival count
// in LDS that the waiting waves poll.  Every one of the n waves makes every
// call, and none of them waits on the other waves in between, so each wait
// ends.
struct GroupSync {
  LDS uint32_t* ctr;
  uint32_t n, gen;
  __device__ __forceinline__ void operator()() {
    ++gen;
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
    if ((threadIdx.x & 63u) == 0) __atomic_fetch_add(ctr, 1u, __ATOMIC_RELAXED);
    while (__atomic_load_n(ctr, __ATOMIC_RELAXED) < n * gen) __builtin_amdgcn_s_sleep(1);
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
  }
};
struct BarrierSync {
  __device__ __forceinline__ void operator()() { __syncthreads(); }
};

// Builds the history tables for tokens in [lo, hi) of row b.  All threads.
// Global round trips: the row's history (held in registers, HTPT tokens per
// thread per pass) and one gather of the logits of the distinct tokens.
// Occurrences of history entry i: its count in the count-table form (read
// as at least 1: a listed token is in the history), else 1 per entry.
__device__ __forceinline__ uint32_t hist_weight(const Args& a, uint32_t i) {
  return a.hcnt ? umax(G(a.hcnt)[i], 1u) : 1u;
}

constexpr int HTPT = 8;
template <int DT>
__device__ __forceinline__ void build_history(const Args& a, const RowP& P, uint32_t b,
                              const void* row, uint32_t lo, uint32_t hi,
                              uint32_t nwords, Hist& h, LDS uint32_t* red,
                              LDS uint32_t* flags) {
  const uint32_t tid = threadIdx.x;
  const bool need_pen = P.rp != 1.0f || P.pp != 0.0f || P.fp != 0.0f;
  const bool have = need_pen && a.hoff;
  const uint32_t h0 = have ? G(a.hoff)[b] : 0u;
  const uint32_t h1 = have ? (a.hlen ? h0 + G(a.hlen)[b] : G(a.hoff)[b + 1]) : 0u;
  uint32_t tk[HTPT];
#pragma unroll
  for (int q = 0; q < HTPT; ++q) {
    const uint32_t i = h0 + q * NT + tid;
    tk[q] = (i < h1) ? G(a.htok)[i] : EMPTY;
  }
  for (uint32_t i = tid; i < nwords; i += NT) h.bitmap[i] = 0;
  __syncthreads();
  if (!have) {  // uniform; the tables stay empty
    for (uint32_t i = tid; i < nwords; i += NT) h.pre[i] = 0;
    __syncthreads();
    return;
  }
  const bool need_cnt = P.fp != 0.0f;
  const bool one_pass = h1 - h0 <= (uint32_t)(HTPT * NT);
  for (uint32_t c0 = h0; c0 < h1; c0 += HTPT * NT) {
#pragma unroll
    for (int q = 0; q < HTPT; ++q) {
      uint32_t t = tk[q];
      if (c0 != h0) {
        const uint32_t i = c0 + q * NT + tid;
        t = (i < h1) ? G(a.htok)[i] : EMPTY;
      }
      if (t >= lo && t < hi) __atomic_fetch_or(&h.bitmap[(t - lo) >> 5], 1u << (t & 31), __ATOMIC_RELAXED);
    }
  }
  __syncthreads();
  // exclusive popcount prefix over the words, each thread a contiguous run;
  // the token of every rank is recorded
  const uint32_t wpt = (nwords + NT - 1) / NT;
  const uint32_t w0 = tid * wpt, w1 = (w0 + wpt < nwords) ? w0 + wpt : nwords;
  uint32_t local = 0;
  for (uint32_t wi = w0; wi < w1; ++wi) local += __popc(h.bitmap[wi]);
  uint32_t U;
  uint32_t run = block_excl_scan(local, red, U);
  for (uint32_t wi = w0; wi < w1; ++wi) {
    h.pre[wi] = (uint16_t)(run < 0xffffu ? run : 0xffffu);
    uint32_t bits = h.bitmap[wi];
    while (bits) {
      const uint32_t bit = __builtin_ctz(bits);
      bits &= bits - 1;
      if (run < U_MAX) h.tokr[run] = lo + 32 * wi + bit;
      ++run;
    }
  }
  if (U > U_MAX && tid == 0) __atomic_fetch_or(flags, FLAG_HIST_OVERFLOW, __ATOMIC_RELAXED);
  const uint32_t Uc = U < U_MAX ? U : U_MAX;
  LDS uint32_t* cnt = (LDS uint32_t*)h.pen;
  if (need_cnt) {
    for (uint32_t i = tid; i < Uc; i += NT) cnt[i] = 0;
    __syncthreads();
    for (uint32_t c0 = h0; c0 < h1; c0 += HTPT * NT) {
#pragma unroll
      for (int q = 0; q < HTPT; ++q) {
        uint32_t t = tk[q];
        const uint32_t i = c0 + q * NT + tid;
        if (!one_pass) t = (i < h1) ? G(a.htok)[i] : EMPTY;
        if (t >= lo && t < hi) {
          const uint32_t r = h.rank(t);
          if (r < U_MAX) __atomic_fetch_add(&cnt[r], hist_weight(a, i), __ATOMIC_RELAXED);
        }
      }
    }
  }
  __syncthreads();
  // penalised logit of every distinct history token: loads first, then math
  for (uint32_t r0 = 0; r0 < Uc; r0 += HTPT * NT) {
    float x[HTPT];
#pragma unroll
    for (int q = 0; q < HTPT; ++q) {
      const uint32_t r = r0 + q * NT + tid;
      x[q] = (r < Uc) ? load_logit<DT>(row, h.tokr[r]) : 0.0f;
    }
#pragma unroll
    for (int q = 0; q < HTPT; ++q) {
      const uint32_t r = r0 + q * NT + tid;
      if (r < Uc) h.pen[r] = penalize(x[q], P, need_cnt ? cnt[r] : 1u);
    }
  }
  __syncthreads();
}

// ---------------------------------------------------------------------------
// Candidate-threshold histogram
// ---------------------------------------------------------------------------
// Largest fine bin beta such that at least Kc counted elements have bin >=
// beta (0 if fewer are counted).  Counts are lower bounds of the true counts,
// so beta never exceeds the bin of the true Kc-th largest logit.
__device__ __forceinline__ uint32_t compute_beta(LDS const uint32_t* hc, LDS const uint32_t* hf,
                                 uint32_t Kc, int lane) {
  const uint32_t c = hc[63 - lane];
  const uint32_t incl = wave_incl_scan(c);
  const uint64_t m = __ballot(incl >= Kc);
  if (m == 0) return 0;
  const int l = __ffsll((unsigned long long)m) - 1;
  const uint32_t cb = 63u - (uint32_t)l;
  const uint32_t before = __shfl(incl - c, l);
  const uint32_t need = Kc - before;
  const uint32_t f = hf[cb * 64 + 63 - lane];
  const uint32_t fincl = wave_incl_scan(f);
  const uint64_t m2 = __ballot(fincl >= need);
  if (m2 == 0) return 0;
  const int l2 = __ffsll((unsigned long long)m2) - 1;
  return cb * 64u + 63u - (uint32_t)l2;
}

// Smallest float whose key lies in bin `beta` (all finite values for the
// bins below that of -FLT_MAX, which hold only NaN and -inf keys).  For
// finite v: v >= theta_of(beta) exactly when bin(v) >= beta, except that
// -0.0 also passes at beta = bin(+0.0), which only adds a candidate.
__device__ __forceinline__ float theta_of(uint32_t beta) {
  return beta <= 8u ? -3.402823466e+38f : funkey(beta << BIN_SHIFT);
}

// ---------------------------------------------------------------------------
// Geometry
// ---------------------------------------------------------------------------
__device__ __forceinline__ void wg_to_row_seg(const Args& a, uint32_t i,
                                              uint32_t& b, uint32_t& g) {
  if (a.xcd_map) {
    const uint32_t x = i & 7u, j = i >> 3;
    b = x + 8u * (j / a.G);
    g = j % a.G;
  } else {
    b = i / a.G;
    g = i % a.G;
  }
}
__device__ __forceinline__ uint32_t row_seg_to_wg(const Args& a, uint32_t b,
                                                  uint32_t g) {
  if (a.xcd_map) return 8u * (a.G * (b >> 3) + g) + (b & 7u);
  return b * a.G + g;
}

// ---------------------------------------------------------------------------
// Tile loads
// ---------------------------------------------------------------------------

struct Raw {
  uint32_t d[16];  // fp32 bits (bf16: 8 dwords of pairs)
  uint32_t mw[4];  // allow-mask words of the lane's 4 runs
};

// The vocabulary index of the lane's value j of the tile at tb: an f32 tile
// is four runs of 256 tokens, the lane holding 4 consecutive tokens of each
// (one 16-byte load per run); a 16-bit tile two runs of 512, the lane holding
// 8 consecutive tokens of each (again one 16-byte load per run).
template <int DT>
__device__ __forceinline__ uint32_t tile_pos(uint32_t tb, int lane, int j) {
  if ((DT & 3) == LLMK_F32)
    return tb + 256u * (uint32_t)(j >> 2) + 4u * (uint32_t)lane + (uint32_t)(j & 3);
  return tb + 512u * (uint32_t)(j >> 3) + 8u * (uint32_t)lane + (uint32_t)(j & 7);
}

// Lane `lane` owns the tile positions tile_pos gives.
template <int DT>
__device__ __forceinline__ void load_tile(const Args& a, const void* row,
                                          const uint32_t* mrow, const Hist& h,
                                          uint32_t t, int lane, Raw& raw) {
  const uint32_t tb = t * TILE;
  (void)h;
  if (tb + TILE <= a.V) {
    if ((DT & 3) == LLMK_F32) {
      const GLB f4v* p = (const GLB f4v*)G((const float*)row + tb) + lane;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const f4v x = __builtin_nontemporal_load(p + 64 * r);
        raw.d[4 * r + 0] = __float_as_uint(x.x);
        raw.d[4 * r + 1] = __float_as_uint(x.y);
        raw.d[4 * r + 2] = __float_as_uint(x.z);
        raw.d[4 * r + 3] = __float_as_uint(x.w);
      }
    } else {
      // two 16-byte loads: tokens 512h + 8 lane .. 512h + 8 lane + 7
      const GLB u4v* p = (const GLB u4v*)G((const uint16_t*)row + tb) + lane;
#pragma unroll
      for (int hh = 0; hh < 2; ++hh) {
        const u4v x = __builtin_nontemporal_load(p + 64 * hh);
        raw.d[4 * hh + 0] = x.x;
        raw.d[4 * hh + 1] = x.y;
        raw.d[4 * hh + 2] = x.z;
        raw.d[4 * hh + 3] = x.w;
      }
    }
  } else {
#pragma unroll
    for (int j = 0; j < 16; ++j) {
      const uint32_t e = tile_pos<DT>(tb, lane, j);
      if ((DT & 3) == LLMK_F32) {
        raw.d[j] = e < a.V ? G((const uint32_t*)row)[e] : 0xff800000u;  // -inf past V
      } else {
        // the raw 16-bit value, -inf past V
        const uint32_t hv = e < a.V ? (uint32_t)G((const uint16_t*)row)[e]
                                    : ((DT & 3) == LLMK_BF16 ? 0xff80u : 0xfc00u);
        if ((j & 1) == 0) raw.d[j >> 1] = hv;
        else raw.d[j >> 1] |= hv << 16;
      }
    }
  }
  if (mrow) {
    if ((DT & 3) == LLMK_F32) {
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const uint32_t wi = (tb >> 5) + 8u * r + ((uint32_t)lane >> 3);
        raw.mw[r] = (wi < a.mask_words) ? G(mrow)[wi] : 0u;
      }
    } else {
#pragma unroll
      for (int hh = 0; hh < 2; ++hh) {
        const uint32_t wi = (tb >> 5) + 16u * hh + ((uint32_t)lane >> 2);
        raw.mw[hh] = (wi < a.mask_words) ? G(mrow)[wi] : 0u;
      }
    }
  }
}

template <int DT>
__device__ __forceinline__ void unpack(const Raw& raw, float v[16]) {
  if ((DT & 3) == LLMK_F32) {
#pragma unroll
    for (int j = 0; j < 16; ++j) v[j] = __uint_as_float(raw.d[j]);
  } else {
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      if ((DT & 3) == LLMK_BF16) {
        v[4 * r + 0] = __uint_as_float(raw.d[2 * r] << 16);
        v[4 * r + 1] = __uint_as_float(raw.d[2 * r] & 0xffff0000u);
        v[4 * r + 2] = __uint_as_float(raw.d[2 * r + 1] << 16);
        v[4 * r + 3] = __uint_as_float(raw.d[2 * r + 1] & 0xffff0000u);
      } else {
        v[4 * r + 0] = cvt16<DT>(raw.d[2 * r] & 0xffffu);
        v[4 * r + 1] = cvt16<DT>(raw.d[2 * r] >> 16);
        v[4 * r + 2] = cvt16<DT>(raw.d[2 * r + 1] & 0xffffu);
        v[4 * r + 3] = cvt16<DT>(raw.d[2 * r + 1] >> 16);
      }
    }
  }
  if (DT & SOFTCAP) {
#pragma unroll
    for (int j = 0; j < 16; ++j) v[j] = softcap<DT>(v[j]);
  }
}

// ---------------------------------------------------------------------------
// Probabilities and the sequential semantics
// ---------------------------------------------------------------------------
// p of a (penalised, masked) logit v given the temperature, x_max = m and
// the normaliser S: sampler.rs:53-70, with glibc's expf (exp_ref).  S is
// the reference's sequential sum, or 1 on a row that top-k renormalises
// (where S cancels: p is then e itself).
__device__ __forceinline__ float prob_of(float v, float T, float m, float S) {
  const float x = (T != 1.0f) ? v / T : v;
  const float e = (x == NEG_INF) ? 0.0f : exp_ref(x - m);
  return (S > 0.0f) ? e / S : e;
}

__device__ __forceinline__ uint64_t pkey(float p, uint32_t idx) {
  return ((uint64_t)(~__float_as_uint(p)) << 32) | idx;
}

// Synchronisation policies: a whole workgroup (barriers) or one wave (LDS
// traffic of a single wave completes in order; waiting for it suffices).
// excl_scan(keep): this thread's position among the keeping threads of the
// policy (in id order) and their total.
struct BlockSync {
  static constexpr uint32_t N = NT;
  __device__ static __forceinline__ uint32_t id() { return threadIdx.x; }
  __device__ static __forceinline__ void sync() { __syncthreads(); }
  __device__ static __forceinline__ uint32_t excl_scan(bool keep, LDS uint32_t* red,
                                                       uint32_t& total) {
    return block_excl_scan(keep ? 1u : 0u, red, total);
  }
};
struct WaveSync {
  static constexpr uint32_t N = WAVE;
  __device__ static __forceinline__ uint32_t id() { return threadIdx.x & 63u; }
  __device__ static __forceinline__ void sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0): this wave's LDS ops done
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  }
  __device__ static __forceinline__ uint32_t excl_scan(bool keep, LDS uint32_t*,
                                                       uint32_t& total) {
    const uint64_t mk = __ballot(keep);
    total = (uint32_t)__popcll(mk);
    return lanes_below(mk);
  }
};

// A list sorted by (p desc, idx asc) holding the probabilities as first
// computed; renormalisations (sampler.rs:84-87, :104-109) are recorded as a
// chain of divisors and applied on every read, fl(fl(p/s1)/s2), exactly as
// the reference's in-place divisions, so the list itself is never rewritten.
struct Chain {
  float d0, d1, d2;
  int n;
  __device__ __forceinline__ float apply(float x) const {
    if (n > 0) x = x / d0;
    if (n > 1) x = x / d1;
    if (n > 2) x = x / d2;
    return x;
  }
  __device__ __forceinline__ void push(float s) {
    if (n == 0) d0 = s;
    else if (n == 1) d1 = s;
    else d2 = s;
    ++n;
  }
};
// p and idx are generic pointers (LDS or global memory): one type, so the
// semantics below are compiled once.
struct List {
  const float* p;
  const uint32_t* idx;
  Chain c;
  float* wp;  // p, writable (an LDS list): renormalisations rewrite it
  __device__ float raw(uint32_t i) const { return p[i]; }
  __device__ float get(uint32_t i) const { return c.apply(p[i]); }
  __device__ uint32_t id(uint32_t i) const { return idx[i]; }
};
template <class T>
__device__ __forceinline__ const T* flat(LDS const T* x) {
  return (const T*)x;
}
template <class T>
__device__ __forceinline__ const T* flat(const GLB T* x) {
  return (const T*)x;
}

__device__ __forceinline__ float rl(float x, uint32_t j) {
  return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(x), (int)j));
}

// Increments of the running sum, in units of the binade's quantum, from an
// even (a0) and from an odd (a1) running sum.
struct Par {
  uint32_t a0, a1;
};
// f, then g
__device__ __forceinline__ Par par_then(Par f, Par g) {
  return Par{f.a0 + ((f.a0 & 1u) ? g.a1 : g.a0), f.a1 + ((f.a1 & 1u) ? g.a0 : g.a1)};
}

// The sequential f32 running sums ((p_0 + p_1) + p_2) + ... of list[0..n),
// exactly, computed by wave 0 a window of 512 entries at a time (8
// consecutive entries per lane).  While the running sum c lies in the binade
// [2^e, 2^(e+1)) (e >= -126 also covers the subnormals), c is a multiple of
// q = 2^(e-23), c/q < 2^24, and fl(c + p) is c + q*r with r the nearest
// integer to p/q, a tie going to the even sum: r depends on p alone except
// for a tie, where it depends on the parity of c/q.  So every entry is a
// pair of integer increments (from an even, from an odd sum), and a wave scan
// of the pairs gives every running sum of the binade exactly.  The first
// addition whose result would reach 2^(e+1) is done as one f32 addition and
// the scan resumes after it (a sum of probabilities crosses a few tens of
// binades at most).  Every thread calls it.
// mode 0: sum of all n.  mode 1: stop at the first j with cum >= thr.
// mode 2: stop at the first j with thr <= cum (the draw's `r <= cumulative`).
// Returns the stop index (n if none) and the running sum including it (the
// total if none).  sh: 2 words; z: 128 words.
// Every lane forms its own prefix: lane l of c0 receives ((p_0 + p_1) + ...)
// + p_l and lane l of c1 the prefix through entry 64 + l -- the same f32
// additions in the same order as one sequential sum.  z holds 64 zeros before
// each half of the entries; lane l reads z[1 + l + t] at step t = 0..63, so it
// adds 63 - l zeros (+0.0 + +0.0 stays +0.0) and then p_0..p_l.  All 64 reads
// are issued before the adds and there is no branch: two operations per step.
// Lanes at or past m hold junk.
__device__ __forceinline__ float prefix_half(LDS const float* zb, float c) {
  float x[64];
#pragma unroll
  for (uint32_t t = 0; t < 64u; ++t) x[t] = zb[t];
#pragma unroll
  for (uint32_t t = 0; t < 64u; ++t) c = c + x[t];
  return c;
}
// prefix_half with sixteen reads in flight at a time (fewer registers)
__device__ __forceinline__ float prefix_half16(LDS const float* zb, float c) {
#pragma unroll
  for (uint32_t t0 = 0; t0 < 64u; t0 += 16u) {
    float x[16];
#pragma unroll
    for (uint32_t t = 0; t < 16u; ++t) x[t] = zb[t0 + t];
#pragma unroll
    for (uint32_t t = 0; t < 16u; ++t) c = c + x[t];
  }
  return c;
}
// Exclusive scan of the pairs over the wave (DPP row shifts and row
// broadcasts; shifted-in lanes read (0, 0), the identity).
template <int CTRL, int RM, bool BC>
__device__ __forceinline__ Par dpp_par(Par x) {
  return Par{dppu<CTRL, RM, BC>(0u, x.a0), dppu<CTRL, RM, BC>(0u, x.a1)};
}
__device__ __forceinline__ Par wave_par_excl(Par x) {
  x = par_then(dpp_par<0x111, 0xf, true>(x), x);
  x = par_then(dpp_par<0x112, 0xf, true>(x), x);
  x = par_then(dpp_par<0x114, 0xf, true>(x), x);
  x = par_then(dpp_par<0x118, 0xf, true>(x), x);
  x = par_then(dpp_par<0x142, 0xa, false>(x), x);
  x = par_then(dpp_par<0x143, 0xc, false>(x), x);
  return dpp_par<0x138, 0xf, true>(x);  // wave_shr:1
}
template <int Q>
__device__ __forceinline__ float pickf(const float (&x)[Q], uint32_t k) {
  float r = x[0];
#pragma unroll
  for (int q = 1; q < Q; ++q) r = (k == (uint32_t)q) ? x[q] : r;
  return r;
}
template <class L>
__device__ __forceinline__ uint32_t seq_scan(const L& list, uint32_t n, int mode, float thr,
                                             float& cum_out, LDS uint32_t* sh, LDS float* z) {
  if (threadIdx.x < WAVE) {
    constexpr uint32_t Q = 8, W = Q * WAVE;
    constexpr uint32_t TOP = 1u << 24;
    const uint32_t lane = threadIdx.x, l0 = Q * lane;
    const bool stops = mode != 0;
    uint32_t stop = n;
    float c = 0.0f;
    uint32_t j0 = 0;
    if (n > 0 && stops && thr <= 0.0f) {  // the first running sum already meets it
      stop = 0;
      c = 0.0f + list.get(0);
    } else if (n > 0) {
      // the first 256 entries, where the sum crosses binades often, 64 at a
      // time: every lane forms its own running sum (prefix_half16 from c:
      // 63 - lane zeros, which leave c as it is, then p_base .. p_base+lane,
      // the same f32 additions in the same order)
      const uint32_t hn = umin(n, 4u * WAVE);
      while (j0 < hn) {
        const uint32_t h = umin(hn - j0, (uint32_t)WAVE);
        z[lane] = 0.0f;
        z[WAVE + lane] = lane < h ? list.get(j0 + lane) : 0.0f;
        WaveSync::sync();
        const float cl = prefix_half16(z + 1 + lane, c);
        WaveSync::sync();
        const uint64_t hit = stops ? __ballot(lane < h && cl >= thr) : 0ull;
        if (hit) {
          const uint32_t js = (uint32_t)__ffsll((unsigned long long)hit) - 1;
          stop = j0 + js;
          c = rl(cl, js);
          break;
        }
        c = rl(cl, h - 1);
        j0 += h;
      }
    }
    // the raw entries of the window at jj (the divisor chain is applied when
    // it is scanned); the next window's are requested before a window is
    // scanned, so that a list in global memory is not waited for window by
    // window
    float pr[Q];
    auto fetch = [&](uint32_t jj) __attribute__((always_inline)) {
#pragma unroll
      for (uint32_t q = 0; q < Q; ++q) pr[q] = jj + l0 + q < n ? list.raw(jj + l0 + q) : 0.0f;
    };
    if (j0 < n && stop == n) fetch(j0);
    for (uint32_t j = j0; j < n && stop == n; j += W) {
      const uint32_t lim = umin(n - j, W);
      float p[Q];
#pragma unroll
      for (uint32_t q = 0; q < Q; ++q) p[q] = (l0 + q < lim) ? list.c.apply(pr[q]) : 0.0f;
      if (j + W < n) fetch(j + W);
      uint32_t s = 0;  // window entries before s are summed
      while (s < lim) {
        if (c == 0.0f) {
          // 0 + p is exact: the first nonzero entry starts the sum (zeros
          // leave it 0, below thr > 0)
          uint32_t fz = EMPTY;
#pragma unroll
          for (int q = (int)Q - 1; q >= 0; --q)
            if (l0 + q >= s && l0 + q < lim && p[q] != 0.0f) fz = l0 + q;
          fz = wave_min_u32(fz);
          if (fz == EMPTY) {
            s = lim;
            break;
          }
          c = 0.0f + rl(pickf(p, fz % Q), fz / Q);
          s = fz + 1;
          if (stops && c >= thr) {
            stop = j + fz;
            break;
          }
          continue;
        }
        const uint32_t cb = __float_as_uint(c);
        const int e = (int)umax((cb >> 23) & 255u, 1u) - 127;
        const uint32_t C = (uint32_t)__builtin_ldexpf(c, 23 - e);
        uint32_t r[Q], tie = 0;  // increments; ties: the value from an even sum differs
#pragma unroll
        for (uint32_t q = 0; q < Q; ++q) {
          const float x = __builtin_ldexpf(p[q], 23 - e);  // exact, < 2^24
          const float k = __builtin_floorf(x);
          const float fr = x - k;
          const uint32_t ki = (uint32_t)k;
          const bool live = l0 + q >= s && l0 + q < lim;
          r[q] = !live ? 0u : (fr > 0.5f ? ki + 1u : ki);
          if (live && fr == 0.5f) tie |= 1u << q;
        }
        // this lane's increments from an even and from an odd sum (a tie
        // adds k or k + 1, whichever makes the sum even)
        uint32_t s0 = 0, s1 = 1;
#pragma unroll
        for (uint32_t q = 0; q < Q; ++q) {
          const uint32_t t = (tie >> q) & 1u;
          s0 += r[q] + (t & ((s0 ^ r[q]) & 1u));
          s1 += r[q] + (t & ((s1 ^ r[q]) & 1u));
        }
        const Par ex = wave_par_excl(Par{s0, s1 - 1u});
        uint32_t cur = C + ((C & 1u) ? ex.a1 : ex.a0);
        // the lane's first event (crossing or stop) with the sum before (a
        // crossing) or at (a stop) it, and the sum at the window's last entry
        uint32_t ev = EMPTY, evv = 0, endv = 0, evx = 0;
#pragma unroll
        for (uint32_t q = 0; q < Q; ++q) {
          const uint32_t t = (tie >> q) & 1u;
          const uint32_t nx = cur + r[q] + (t & ((cur ^ r[q]) & 1u));
          if (ev == EMPTY && l0 + q >= s && l0 + q < lim) {
            if (nx >= TOP) {
              ev = l0 + q;
              evx = 1;
              evv = cur;
            } else if (stops && __builtin_ldexpf((float)nx, e - 23) >= thr) {
              ev = l0 + q;
              evv = nx;
            }
          }
          if (l0 + q == lim - 1) endv = nx;
          cur = nx;
        }
        const uint32_t evm = wave_min_u32(ev);
        if (evm == EMPTY) {
          const uint32_t v = (uint32_t)__builtin_amdgcn_readlane((int)endv, (int)((lim - 1) / Q));
          c = __builtin_ldexpf((float)v, e - 23);
          s = lim;
          break;
        }
        const int ol = (int)(evm / Q);
        const float v =
            __builtin_ldexpf((float)(uint32_t)__builtin_amdgcn_readlane((int)evv, ol), e - 23);
        if (!__builtin_amdgcn_readlane((int)evx, ol)) {
          stop = j + evm;
          c = v;
          break;
        }
        // the addition that leaves the binade, as one f32 addition
        c = v + rl(pickf(p, evm % Q), (uint32_t)ol);
        s = evm + 1;
        if (stops && c >= thr) {
          stop = j + evm;
          break;
        }
      }
    }
    if (lane == 0) {
      sh[0] = stop;
      sh[1] = __float_as_uint(c);
    }
  }
  __syncthreads();
  const uint32_t stop = sh[0];
  cum_out = __uint_as_float(sh[1]);
  __syncthreads();
  return stop;
}

// The renormalisation p /= s of the first len entries (sampler.rs:84-87,
// :104-109): rewritten in place for a writable list (every thread calls
// it), else recorded in the divisor chain.
__device__ __forceinline__ void div_all(List& list, float s, uint32_t len) {
  if (!(s > 0.0f)) return;
  if (list.wp) {
    for (uint32_t i = threadIdx.x; i < len; i += NT) list.wp[i] = list.wp[i] / s;
    __syncthreads();
  } else {
    list.c.push(s);
  }
}

// First i < n with list[i] < thr (strict) or <= thr, n if none; the list is
// sorted descending, so the predicate is monotone: one probe per thread
// finds the block of n/NT entries holding the first hit, then the block is
// searched.  n <= NT * NT.  sh: 1 word.
__device__ __forceinline__ uint32_t first_below(const List& list, uint32_t n, float thr,
                                                bool strict,
                                LDS uint32_t* sh) {
  const uint32_t tid = threadIdx.x;
  auto hit = [&](uint32_t i) {
    const float v = list.get(i);
    return strict ? v < thr : v <= thr;
  };
  const uint32_t step = (n + NT - 1) / NT;
  if (tid == 0) sh[0] = EMPTY;
  __syncthreads();
  const uint32_t lo = tid * step;
  if (lo < n && hit(umin(lo + step, n) - 1)) __atomic_fetch_min(&sh[0], tid, __ATOMIC_RELAXED);
  __syncthreads();
  const uint32_t kb = sh[0];
  __syncthreads();
  if (kb == EMPTY) return n;
  if (tid == 0) sh[0] = EMPTY;
  __syncthreads();
  const uint32_t b0 = kb * step;
  if (tid < step && b0 + tid < n && hit(b0 + tid))
    __atomic_fetch_min(&sh[0], b0 + tid, __ATOMIC_RELAXED);
  __syncthreads();
  const uint32_t r = sh[0];
  __syncthreads();
  return r;
}

// Lists at least this long are scanned by the whole workgroup
// (block_list_scan), shorter ones by wave 0 (seq_scan); only the slow path's
// lists get that long (the candidate path keeps at most SORT_CAP).
constexpr uint32_t BLOCK_SCAN_MIN = 4096;
__device__ __attribute__((noinline)) u2v block_list_scan(List list, uint32_t n, int mode,
                                                        float thr, LDS uint32_t* sc);

// min-p / top-k / top-p / draw (sampler.rs:77-124 + min-p) over a sorted list
// of full_len entries whose first E are exact; every entry past E has
// p <= ptail.  Every thread of the workgroup.  Returns false if an entry
// beyond E would be needed.  The four steps share one running-sum call.
template <bool LONG>
__device__ __forceinline__ bool run_semantics(const RowP& P, float u, uint32_t E,
                                              uint32_t full_len, float ptail, List& list,
                                              LDS uint32_t* sh, LDS float* z,
                                              uint32_t& tok_out, uint32_t& len_out) {
  uint32_t len = full_len;
  bool trunc = E < full_len;
  for (int step = 0; step < 4; ++step) {
    uint32_t n;
    int mode = 0;
    float thr = 0.0f;
    if (step == 0) {
      // ---- min-p (extension): keep p >= min_p * p_max, renormalise if it cuts
      if (!(P.min_p > 0.0f)) continue;
      if (E == 0) return false;
      const float t = P.min_p * list.get(0);
      const uint32_t lim = E < len ? E : len;
      uint32_t cut = first_below(list, lim, t, true, sh);
      if (cut == lim) cut = EMPTY;
      // every entry past E is below the threshold: the cut is at E
      if (cut == EMPTY && trunc && ptail < t) cut = E;
      if (cut == EMPTY) {
        if (trunc) return false;
        continue;
      }
      if (cut >= len) continue;
      len = cut;
      trunc = false;
      n = len;
    } else if (step == 1) {
      // ---- top-k, sampler.rs:80-89
      if (!(P.K > 0 && (uint32_t)P.K < len)) continue;
      if ((uint32_t)P.K > E) return false;
      len = (uint32_t)P.K;
      trunc = false;
      n = len;
    } else {
      // ---- top-p, sampler.rs:92-110; the draw, sampler.rs:113-124
      if (step == 2 && !(P.top_p < 1.0f)) continue;
      n = (trunc && E < len) ? E : len;
      mode = step == 2 ? 1 : 2;
      thr = step == 2 ? P.top_p : u;
    }
    float s;
    uint32_t j;
    if (LONG && n >= BLOCK_SCAN_MIN) {
      const u2v r = block_list_scan(list, n, mode, thr, (LDS uint32_t*)z);
      j = r.x;
      s = __uint_as_float(r.y);
    } else {
      j = seq_scan(list, n, mode, thr, s, sh, z);
    }
    if (step == 3) {
      uint32_t tok;
      if (j < n) tok = list.id(j);
      else {
        if (trunc) return false;
        tok = len > 0 ? list.id(len - 1) : 0u;
      }
      tok_out = tok;
      len_out = len;
      return true;
    }
    if (step == 2) {
      if (j == n && trunc) return false;
      // the renormalisation sum over the kept prefix is the same sequential
      // sum as the cumulative at the cut
      len = (j < n) ? j + 1 : len;
      trunc = false;
    }
    div_all(list, s, len);
  }
  return false;
}

__device__ __forceinline__ void write_outputs(const Args& a, uint32_t b, uint32_t tok,
                                              uint32_t len, const List& list, float m,
                                              float S) {
  if (threadIdx.x == 0) {
    G(a.out_tok)[b] = tok;
    if (a.out_cnt) G(a.out_cnt)[b] = len;
    if (a.cut)
      G(a.cut)[b] = u4v{(len > 0 && len < a.V) ? list.id(len - 1) : 0u, len,
                        __float_as_uint(m), __float_as_uint(S)};
  }
  if (a.out_cap) {
    const uint32_t n = len < a.out_cap ? len : a.out_cap;
    for (uint32_t j = threadIdx.x; j < n; j += NT) {
      if (a.out_ids) G(a.out_ids)[(uint64_t)b * a.out_cap + j] = list.id(j);
      if (a.out_probs) G(a.out_probs)[(uint64_t)b * a.out_cap + j] = list.get(j);
    }
  }
}

// ---------------------------------------------------------------------------
// min-p / top-k / top-p / draw for a sorted list of at most 128 entries held
// in registers of one wave: lane j holds entries j (p0, i0) and 64 + j (p1,
// i1).  The same sequential f32 sums and divisions as run_semantics, in the
// same order; the running sums are wave-uniform, each step reading one entry
// with v_readlane.  Returns false if an entry beyond E = n would be needed.
// ---------------------------------------------------------------------------
// z: 256 LDS words owned by the calling wave; 1 <= m <= 128.
__device__ __forceinline__ void prefix_regs(float p0, float p1, uint32_t m, int lane,
                                            LDS float* z, float& c0, float& c1) {
  z[lane] = 0.0f;
  z[64 + lane] = p0;
  z[128 + lane] = 0.0f;
  z[192 + lane] = p1;
  WaveSync::sync();
  c0 = prefix_half(z + 1 + lane, 0.0f);
  c1 = 0.0f;
  if (m > 64u) c1 = prefix_half(z + 129 + lane, rl(c0, 63));
  WaveSync::sync();  // z is rewritten by the next call
}
// ((p_0 + p_1) + ...) + p_{m-1}
__device__ __forceinline__ float seq_sum_regs(float p0, float p1, uint32_t m, int lane,
                                              LDS float* z) {
  if (m == 0) return 0.0f;
  float c0, c1;
  prefix_regs(p0, p1, m, lane, z, c0, c1);
  return m <= 64 ? rl(c0, m - 1) : rl(c1, m - 65);
}
// First j < m whose running sum meets the condition (mode 1: cum >= thr,
// mode 2: thr <= cum), m if none; cum_out: the running sum there (or the
// total).
__device__ __forceinline__ uint32_t seq_find_regs(float p0, float p1, uint32_t m, int mode,
                                                  float thr, int lane, LDS float* z,
                                                  float& cum_out) {
  if (m == 0) {
    cum_out = 0.0f;
    return 0;
  }
  float c0, c1;
  prefix_regs(p0, p1, m, lane, z, c0, c1);
  auto meets = [&](float x) { return mode == 1 ? x >= thr : thr <= x; };
  const uint64_t m0 = __ballot((uint32_t)lane < m && meets(c0));
  const uint64_t m1 = __ballot((uint32_t)lane + 64 < m && meets(c1));
  uint32_t j = m;
  if (m0) j = (uint32_t)__ffsll((unsigned long long)m0) - 1;
  else if (m1) j = 64u + (uint32_t)__ffsll((unsigned long long)m1) - 1;
  const uint32_t jc = j < m ? j : m - 1;
  cum_out = jc < 64 ? rl(c0, jc) : rl(c1, jc - 64);
  return j;
}

// Index of kept entry len - 1 of a register list of n (wave-uniform), 0 when
// it is not held (len 0, or every entry kept).
__device__ __forceinline__ uint32_t cut_id(uint32_t len, uint32_t n, uint32_t i0, uint32_t i1) {
  const uint32_t lc = (len > 0 && len <= n) ? len - 1 : 0u;
  const uint32_t v = lc < 64 ? (uint32_t)__builtin_amdgcn_readlane((int)i0, (int)lc)
                             : (uint32_t)__builtin_amdgcn_readlane((int)i1, (int)(lc - 64));
  return (len > 0 && len <= n) ? v : 0u;
}

// ---------------------------------------------------------------------------
// The rounding band of S = 1 on rows that top-k renormalises
// ---------------------------------------------------------------------------
// Such a row is sampled with S = 1 (p = e): the reference divides by its
// sequential sum S first (sampler.rs:66-71) and by a renormalising sum before
// any later step reads a probability (min-p's cut, then top-k, :83-88), so S
// cancels in exact arithmetic.  band_certain_wave proves from the sorted e
// alone that every decision (min-p cut, top-k set and order, top-p cut at
// :97, the draw at :118) is the reference's for any S it can hold; a row it
// cannot prove is sampled again with the reference's own S.  The bound: p
// known to relative R (2^-24 for fl(e / S)); a sequential sum rounds each
// partial sum by at most half an ulp of it (u times the value while the
// scale is S's, the binade's half ulp once normalised); a renormalisation
// divides by a sum known to relative sigma and rounds once more:
// R' = (R + sigma + u)(1 + 2^-10), the factor covering second-order terms.
// A decision is certain when its exact value (sums of the e in double)
// lies outside its bound; order is certain unless two entries within 2^-20
// relative have their indices inverted (fl(e_a/S) == fl(e_b/S) ties go by
// index); entries below 2^-100 (p could be subnormal) are never certain.
// The doubles are summed in one fixed order, which the CPU oracle follows:
// a wave's DPP scan within 64 entries (row_shr 1, 2, 4, 8 within rows of 16,
// then row_bcast 15 and 31), then the chunk's carry.  One wave; acc(j) =
// (e bits, index) of entry j < E; entries past E are <= ptail.
constexpr double BAND_U = 0x1p-24;
constexpr double BAND_F = 1.0 + 0x1p-10;
constexpr double BAND_SL = 0x1p-36;
constexpr double BAND_CLOSE = 1.0 + 0x1p-20;
// half an ulp of a float of magnitude x in (0, 2): 2^(floor(log2 x) - 24)
__device__ __forceinline__ double band_hu(double x) {
  if (!(x > 0.0)) return 0.0;
  const uint64_t ex = ((uint64_t)__double_as_longlong(x) >> 52) & 0x7ffu;
  return __longlong_as_double((long long)((ex - 24u) << 52));
}
template <int CTRL, int RM, bool BC>
__device__ __forceinline__ double dppd(double x) {
  const uint64_t b = (uint64_t)__double_as_longlong(x);
  const uint32_t lo = dppu<CTRL, RM, BC>(0u, (uint32_t)b);
  const uint32_t hi = dppu<CTRL, RM, BC>(0u, (uint32_t)(b >> 32));
  return __longlong_as_double((long long)(((uint64_t)hi << 32) | lo));
}
// inclusive prefix over the wave (lanes outside a step's reach add +0)
__device__ __forceinline__ double wave_prefix_d(double x) {
  x = x + dppd<0x111, 0xf, true>(x);
  x = x + dppd<0x112, 0xf, true>(x);
  x = x + dppd<0x114, 0xf, true>(x);
  x = x + dppd<0x118, 0xf, true>(x);
  x = x + dppd<0x142, 0xa, false>(x);
  x = x + dppd<0x143, 0xc, false>(x);
  return x;
}
__device__ __forceinline__ double readlane_d(double x, int l) {
  const uint64_t b = (uint64_t)__double_as_longlong(x);
  const uint32_t lo = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)b, l);
  const uint32_t hi = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(b >> 32), l);
  return __longlong_as_double((long long)(((uint64_t)hi << 32) | lo));
}
template <class ACC>
struct BandList {
  ACC acc;
  uint32_t E;
  __device__ __forceinline__ double e(uint32_t j) const {
    return j < E ? (double)__uint_as_float(acc(j).x) : 0.0;
  }
  // P_{n-1} (prefix of e over [0, n)) and sum_{1 <= j < n} P_j
  __device__ __forceinline__ void sums(uint32_t n, int lane, double& ptot, double& qtot) const {
    double cp = 0.0, cq = 0.0;
    for (uint32_t c0 = 0; c0 < n; c0 += WAVE) {
      const uint32_t j = c0 + (uint32_t)lane;
      const double Pj = wave_prefix_d(j < n ? e(j) : 0.0) + cp;
      const double Qj = wave_prefix_d((j < n && j >= 1) ? Pj : 0.0) + cq;
      if (c0 + WAVE >= n) {
        ptot = readlane_d(Pj, (int)((n - 1) & 63u));
        qtot = readlane_d(Qj, (int)((n - 1) & 63u));
      } else {
        cp = readlane_d(Pj, 63);
        cq = readlane_d(Qj, 63);
      }
    }
  }
  // The first j < n whose cumulative may reach thr (C_j + B_j >= thr), n if
  // none; certain: the reference's cumulative surely reaches it there and
  // not before.  C_j = P_j (1 / tot), B_j = R C_j + sum_{1<=i<=j} hu(C_i (1 +
  // R) F) + SL C_j.  bj, pj: B_j and P_j there (at n - 1 when none).
  __device__ __forceinline__ uint32_t find(uint32_t n, double tot, double R, double thr,
                                           int lane, bool& certain, double& bj,
                                           double& pj) const {
    const double rt = 1.0 / tot;
    double cp = 0.0, ch = 0.0;
    for (uint32_t c0 = 0; c0 < n; c0 += WAVE) {
      const uint32_t j = c0 + (uint32_t)lane;
      const double Pj = wave_prefix_d(j < n ? e(j) : 0.0) + cp;
      const double C = Pj * rt;
      const double hj = (j < n && j >= 1) ? band_hu(C * (1.0 + R) * BAND_F) : 0.0;
      const double Hj = wave_prefix_d(hj) + ch;
      const double b = R * C + Hj + BAND_SL * C;
      const uint64_t hit = __ballot(j < n && C + b >= thr);
      if (hit) {
        const int l = __ffsll((unsigned long long)hit) - 1;
        certain = __builtin_amdgcn_readlane((int)(C - b >= thr), l) != 0;
        bj = readlane_d(b, l);
        pj = readlane_d(Pj, l);
        return c0 + (uint32_t)l;
      }
      if (c0 + WAVE >= n) {
        bj = readlane_d(b, (int)((n - 1) & 63u));
        pj = readlane_d(Pj, (int)((n - 1) & 63u));
      } else {
        cp = readlane_d(Pj, 63);
        ch = readlane_d(Hj, 63);
      }
    }
    certain = true;
    return n;
  }
};
// sorted (p desc, idx asc) keys
struct KeyAcc {
  LDS const uint64_t* k;
  __device__ __forceinline__ u2v operator()(uint32_t j) const {
    const uint64_t x = k[j];
    return u2v{~(uint32_t)(x >> 32), (uint32_t)x};
  }
};
// sorted p and index arrays (LDS or global)
template <class PF, class PI>
struct ArrAcc {
  PF p;
  PI i;
  __device__ __forceinline__ u2v operator()(uint32_t j) const {
    return u2v{__float_as_uint(p[j]), i[j]};
  }
};
template <class ACC>
__device__ __noinline__ bool band_certain_wave(ACC acc, uint32_t E, uint32_t full,
                                               float ptail, float min_p, int32_t K,
                                               float top_p, float u) {
  const int lane = (int)(threadIdx.x & 63u);
  const BandList<ACC> L{acc, E};
  uint32_t len = full;
  double R = BAND_U;
  bool normalised = false;
  // entries whose p = e / S could be subnormal
  const uint32_t lim = (K > 0 && (uint32_t)K + 1u < E) ? (uint32_t)K + 1u : E;
  for (uint32_t c0 = 0; c0 < lim; c0 += WAVE) {
    const uint32_t j = c0 + (uint32_t)lane;
    const float x = j < lim ? __uint_as_float(acc(j).x) : 0.0f;
    if (__ballot(x > 0.0f && x < 0x1p-100f)) return false;
  }
  double ptot = 0.0, qtot = 0.0;
  auto renormalise = [&](uint32_t n) {
    L.sums(n, lane, ptot, qtot);
    const double sg = R + BAND_U * (1.0 + R) * BAND_F * (qtot / ptot);
    R = (R + sg + BAND_U) * BAND_F;
    normalised = true;
  };
  // min-p: kept iff fl(e/S) >= fl(min_p fl(1/S)) (e_0 = 1, the maximum);
  // certain outside min_p (1 -+ 2^-21)
  if (min_p > 0.0f) {
    if (min_p < 0x1p-100f || E == 0) return false;
    const double hi = (double)min_p * (1.0 + 0x1p-21);
    const double lo = (double)min_p * (1.0 - 0x1p-21);
    const uint32_t n = E < len ? E : len;
    uint32_t cut = EMPTY;
    for (uint32_t c0 = 0; c0 < n; c0 += WAVE) {
      const uint32_t j = c0 + (uint32_t)lane;
      const uint64_t hit = __ballot(j < n && L.e(j) < hi);
      if (hit) {
        cut = c0 + (uint32_t)(__ffsll((unsigned long long)hit) - 1);
        break;
      }
    }
    if (cut != EMPTY) {
      if (L.e(cut) >= lo) return false;
    } else if (E < len) {
      if ((double)ptail >= lo) return false;
      cut = E;
    }
    if (cut != EMPTY && cut < len) {
      len = cut;
      if (len == 0) return false;
      renormalise(len);
      if (!(ptot > 0.0)) return false;
    }
  }
  // top-k: the first K in (p desc, idx asc) order; no pair whose order could
  // change, across the boundary included (an unknown entry K close to the
  // last kept one could be either side of it)
  uint32_t np;
  if (K > 0 && (uint32_t)K < len) {
    if ((uint32_t)K > E) return false;
    if ((uint32_t)K == E && L.e(K - 1) < (double)ptail * BAND_CLOSE) return false;
    np = (uint32_t)K < E ? (uint32_t)K + 1u : (uint32_t)K;
  } else {
    np = E < len ? E : len;
  }
  for (uint32_t c0 = 0; c0 + 1 < np; c0 += WAVE) {
    const uint32_t j = c0 + (uint32_t)lane;
    bool bad = false;
    if (j + 1 < np) {
      const u2v x0 = acc(j), x1 = acc(j + 1);
      bad = (double)__uint_as_float(x0.x) < (double)__uint_as_float(x1.x) * BAND_CLOSE &&
            x0.y > x1.y;
    }
    if (__ballot(bad)) return false;
  }
  if (K > 0 && (uint32_t)K < len) {
    len = (uint32_t)K;
    renormalise(len);
    if (!(ptot > 0.0)) return false;
  }
  if (!normalised || len > E) return false;
  // top-p: the first cumulative >= top_p, then the renormalisation by that
  // same cumulative
  if (top_p < 1.0f) {
    bool cert;
    double b, pc;
    const uint32_t j = L.find(len, ptot, R, (double)top_p, lane, cert, b, pc);
    if (!cert) return false;
    const double sp = b / (pc * (1.0 / ptot));
    R = (R + sp + BAND_U) * BAND_F;
    len = j < len ? j + 1 : len;
    ptot = pc;
  }
  // the draw: the first cumulative >= u, else the last
  bool cert;
  double b, pc;
  (void)L.find(len, ptot, R, (double)u, lane, cert, b, pc);
  return cert;
}

__device__ __forceinline__ bool semantics_regs(const RowP& P, float u, uint32_t n,
                                               uint32_t full_len, float ptail, float& p0,
                                               float& p1,
                                               uint32_t i0, uint32_t i1, int lane,
                                               LDS float* z, uint32_t& tok_out,
                                               uint32_t& len_out) {
  const uint32_t E = n;
  uint32_t len = full_len;
  bool trunc = E < full_len;
  auto divide = [&](float s) {
    if (s > 0.0f) {
      p0 = p0 / s;
      p1 = p1 / s;
    }
  };
  // ---- min-p (extension): keep p >= min_p * p_max, renormalise if it cuts
  if (P.min_p > 0.0f) {
    if (E == 0) return false;
    const float thr = P.min_p * rl(p0, 0);
    const uint32_t lim = E < len ? E : len;
    const uint64_t c0 = __ballot((uint32_t)lane < lim && p0 < thr);
    const uint64_t c1 = __ballot((uint32_t)lane + 64 < lim && p1 < thr);
    uint32_t cut = EMPTY;
    if (c0) cut = (uint32_t)__ffsll((unsigned long long)c0) - 1;
    else if (c1) cut = 64u + (uint32_t)__ffsll((unsigned long long)c1) - 1;
    // every entry past E is below the threshold: the cut is at E
    if (cut == EMPTY && trunc && ptail < thr) cut = E;
    if (cut == EMPTY) {
      if (trunc) return false;
    } else if (cut < len) {
      len = cut;
      trunc = false;
      divide(seq_sum_regs(p0, p1, len, lane, z));
    }
  }
  // ---- top-k, sampler.rs:80-89
  if (P.K > 0 && (uint32_t)P.K < len) {
    if ((uint32_t)P.K > E) return false;
    len = (uint32_t)P.K;
    trunc = false;
    divide(seq_sum_regs(p0, p1, len, lane, z));
  }
  // ---- top-p, sampler.rs:92-110
  if (P.top_p < 1.0f) {
    const uint32_t lim = (trunc && E < len) ? E : len;
    float s;
    const uint32_t j = seq_find_regs(p0, p1, lim, 1, P.top_p, lane, z, s);
    if (j == lim && trunc) return false;
    len = (j < lim) ? j + 1 : len;
    trunc = false;
    divide(s);
  }
  // ---- draw, sampler.rs:113-124
  const uint32_t lim = (trunc && E < len) ? E : len;
  float s;
  const uint32_t j = seq_find_regs(p0, p1, lim, 2, u, lane, z, s);
  uint32_t tok;
  if (j < lim) tok = j < 64 ? (uint32_t)__builtin_amdgcn_readlane((int)i0, (int)j)
                            : (uint32_t)__builtin_amdgcn_readlane((int)i1, (int)(j - 64));
  else {
    if (trunc) return false;
    const uint32_t l1 = len - 1;
    tok = len == 0 ? 0u
                   : (l1 < 64 ? (uint32_t)__builtin_amdgcn_readlane((int)i0, (int)l1)
                              : (uint32_t)__builtin_amdgcn_readlane((int)i1, (int)(l1 - 64)));
  }
  tok_out = tok;
  len_out = len;
  return true;
}

// ---------------------------------------------------------------------------
// Shared-memory layouts (in 32-bit words)
// ---------------------------------------------------------------------------
enum : uint32_t {
  M_BETA = 0, M_CCOUNT = 1, M_FLAGS = 2, M_LAST = 3, M_NEXT = 4,
  M_GSYNC = 5,  // arrivals of the token waves' group barrier
  M_NMISC = 16
};

__host__ __device__ inline size_t stream_lds_words(uint32_t tps) {
  return 64 + M_NMISC + NBINS + 64 + hist_lds_words(tps * 32) + NW;
}
__host__ __device__ inline size_t finalize_lds_words() {
  // slots (2 x MAX_SLOTS) + keys + sorted keys (2 x SORT_CAP u64) + p + idx
  // + scratch + segment table + reductions + block sums
  return 2 * MAX_SLOTS + 4 * SORT_CAP + 2 * SORT_CAP + 128 + MAX_SEG + 16 + 64 + 2 * MAX_SLOTS / 64;
}
__host__ __device__ inline size_t slow_lds_words(uint32_t V) {
  return 128 + 256 + NW * 256 + SLOW_BINS + hist_lds_words((V + 31) / 32);
}

// ---------------------------------------------------------------------------
// The reference's softmax normaliser, exactly (sampler.rs:56-66)
// ---------------------------------------------------------------------------
// Sixteen consecutive logits of a row from e0 (a multiple of 16), as f32;
// positions past V read -inf.
template <int DT>
__device__ __forceinline__ void load16(const void* row, uint32_t e0, uint32_t V, float x[16]) {
  if (e0 + 16 <= V) {
    if ((DT & 3) == LLMK_F32) {
      const GLB f4v* r = (const GLB f4v*)((const GLB float*)row + e0);
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const f4v a = r[k];
        x[4 * k + 0] = a.x;
        x[4 * k + 1] = a.y;
        x[4 * k + 2] = a.z;
        x[4 * k + 3] = a.w;
      }
    } else {
      const GLB u2v* r = (const GLB u2v*)((const GLB uint16_t*)row + e0);
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const u2v a = r[k];
        x[4 * k + 0] = cvt16<DT>(a.x & 0xffffu);
        x[4 * k + 1] = cvt16<DT>(a.x >> 16);
        x[4 * k + 2] = cvt16<DT>(a.y & 0xffffu);
        x[4 * k + 3] = cvt16<DT>(a.y >> 16);
      }
    }
    if (DT & SOFTCAP) {
#pragma unroll
      for (int q = 0; q < 16; ++q) x[q] = softcap<DT>(x[q]);
    }
  } else {
#pragma unroll
    for (int q = 0; q < 16; ++q) x[q] = e0 + q < V ? load_logit<DT>(row, e0 + q) : NEG_INF;
  }
}

// The smallest of the lanes' keys (~0 = none), whose high words (entry
// indices) differ between lanes that hold one: the minimum high word over
// the wave, then its lane's key.  One LDS atomic per wave then suffices
// (after a crossing every later entry of the window also reports one).
__device__ __forceinline__ uint64_t wave_min_key(uint64_t k) {
  const uint32_t hi = wave_min_u32((uint32_t)(k >> 32));
  const uint64_t owner = __ballot(k != ~0ull && (uint32_t)(k >> 32) == hi);
  if (!owner) return ~0ull;
  const int l = __ffsll((unsigned long long)owner) - 1;
  const uint32_t lo = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)k, l);
  return ((uint64_t)hi << 32) | lo;
}

// Inclusive scan of the pairs over the wave (shifted-in lanes read the
// identity (0, 0)).
__device__ __forceinline__ Par wave_par_incl(Par x) {
  x = par_then(dpp_par<0x111, 0xf, true>(x), x);
  x = par_then(dpp_par<0x112, 0xf, true>(x), x);
  x = par_then(dpp_par<0x114, 0xf, true>(x), x);
  x = par_then(dpp_par<0x118, 0xf, true>(x), x);
  x = par_then(dpp_par<0x142, 0xa, false>(x), x);
  x = par_then(dpp_par<0x143, 0xc, false>(x), x);
  return x;
}

// The sequential f32 sum c = ((c + e_0) + e_1) + ... of one window's
// entries (all >= 0), continued from c and returned, exactly, by the whole
// workgroup.  Thread t holds entries 16t .. 16t+nq-1 (nq 16, or 4 for a wave
// whose window part was compacted; wave-uniform), so entry j = 16t + q of
// the window comes before entry j' exactly when j < j'.  The running-sum
// argument of seq_scan over the block: while c lies in the binade of quantum
// q = 2^(eb-23), each entry adds the integer r = p/q rounded to nearest (a
// tie to the even sum), a pair of increments (from an even, from an odd sum)
// per entry; the pairs of a thread compose in order, the workgroup scans
// them (waves by DPP, then the sixteen wave totals), and the first entry
// whose sum would reach 2^(eb+1) is added as one f32 addition, after which
// the scan resumes.  Entries p/q >= 2^25 are clamped (they cross at once);
// every sum before the first crossing stays below 2^24 + 2^25, so no count
// wraps where it is read.  A zero c takes the first nonzero entry as it is
// (0 + p = p).  A wave whose entries all lie before the resume point adds
// the identity.  Each round's first event goes through one of three LDS
// slots in turn (round it uses slot it % 3 and clears slot (it + 1) % 3,
// read two rounds ago), so a round needs two barriers; `it` carries the
// rotation from call to call, and the slots start cleared
// (exact_normaliser).  sc: 6 + NW*2 words; uniform barriers only.
//
// block_seq_scan<true> also stops at the first entry whose running sum
// reaches thr (stop_at: its index in the window, EMPTY if none) and returns
// that sum: a stop is an event like a crossing, the first event in index
// order taken, and a crossing's sum is compared with thr after its addition.
template <bool STOPS>
__device__ __forceinline__ float block_seq_scan(const float (&e)[16], uint32_t nq, float c,
                                                uint32_t& it, LDS uint32_t* sc, float thr,
                                                uint32_t& stop_at, uint32_t s_start = 0) {
  constexpr uint32_t Q = 16, TOP = 1u << 24;
  stop_at = EMPTY;
  const uint32_t tid = threadIdx.x, lane = tid & 63u, wv = tid >> 6;
  LDS uint64_t* ev = (LDS uint64_t*)sc;  // [3]: first event (index << 32 | new sum bits)
  LDS uint32_t* wt = sc + 6;             // [NW][2]: wave totals
  uint32_t s = s_start;                  // entries before s are summed (into c)
  for (;; ++it) {
    LDS uint64_t* slot = ev + it % 3u;
    if (tid == 0) ev[(it + 1) % 3u] = ~0ull;
    // every entry of this wave lies before s
    const bool wave_done = Q * (64u * wv + 63u) + Q - 1u < s;
    if (c == 0.0f) {
      uint64_t best = ~0ull;
      if (!wave_done) {
#pragma unroll
        for (int q = (int)Q - 1; q >= 0; --q) {
          const uint32_t j = Q * tid + (uint32_t)q;
          if ((uint32_t)q < nq && j >= s && e[q] != 0.0f)
            best = ((uint64_t)j << 32) | __float_as_uint(e[q]);
        }
      }
      best = wave_min_key(best);
      if (lane == 0 && best != ~0ull) __atomic_fetch_min(slot, best, __ATOMIC_RELAXED);
      __syncthreads();
      const uint64_t r = *slot;
      if (r == ~0ull) {  // every remaining entry is 0
        ++it;
        return 0.0f;
      }
      c = __uint_as_float((uint32_t)r);
      s = (uint32_t)(r >> 32) + 1u;
      if (STOPS && c >= thr) {
        stop_at = s - 1u;
        ++it;
        return c;
      }
      if (s >= NT * Q) {
        ++it;
        return c;
      }
      continue;
    }
    const uint32_t cb = __float_as_uint(c);
    const int eb = (int)umax((cb >> 23) & 255u, 1u) - 127;
    const uint32_t C = (uint32_t)__builtin_ldexpf(c, 23 - eb);
    uint32_t r[Q], tie = 0;
    Par own{0u, 0u};
    if (!wave_done) {
#pragma unroll
      for (uint32_t q = 0; q < Q; ++q) {
        r[q] = 0u;
        if (q < nq) {
          const float x = __builtin_fminf(__builtin_ldexpf(e[q], 23 - eb), 0x1p25f);  // exact below the clamp
          const float k = __builtin_floorf(x);
          const float fr = x - k;
          const uint32_t ki = (uint32_t)k;
          const bool live = Q * tid + q >= s;
          r[q] = !live ? 0u : (fr > 0.5f ? ki + 1u : ki);
          if (live && fr == 0.5f) tie |= 1u << q;
        }
      }
      uint32_t s0 = 0, s1 = 1;
#pragma unroll
      for (uint32_t q = 0; q < Q; ++q) {
        if (q < nq) {
          const uint32_t t = (tie >> q) & 1u;
          s0 += r[q] + (t & ((s0 ^ r[q]) & 1u));
          s1 += r[q] + (t & ((s1 ^ r[q]) & 1u));
        }
      }
      own = Par{s0, s1 - 1u};
    }
    const Par inc = wave_par_incl(own);
    if (lane == 63) {
      wt[2 * wv] = inc.a0;
      wt[2 * wv + 1] = inc.a1;
    }
    Par ex = dpp_par<0x138, 0xf, true>(inc);  // wave_shr:1, lane 0 reads (0, 0)
    __syncthreads();
    Par pre{0u, 0u}, tot{0u, 0u};
#pragma unroll
    for (uint32_t i = 0; i < NW; ++i) {
      const Par wtot{wt[2 * i], wt[2 * i + 1]};
      if (i < wv) pre = par_then(pre, wtot);
      tot = par_then(tot, wtot);
    }
    uint64_t cand = ~0ull;
    if (!wave_done) {
      ex = par_then(pre, ex);
      uint32_t cur = C + ((C & 1u) ? ex.a1 : ex.a0);
#pragma unroll
      for (uint32_t q = 0; q < Q; ++q) {
        if (q < nq) {
          const uint32_t t = (tie >> q) & 1u;
          const uint32_t nx = cur + r[q] + (t & ((cur ^ r[q]) & 1u));
          if (cand == ~0ull && Q * tid + q >= s) {
            if (nx >= TOP) {
              // the addition that leaves the binade, as one f32 addition
              const float before = __builtin_ldexpf((float)cur, eb - 23);
              cand = ((uint64_t)(Q * tid + q) << 32) | __float_as_uint(before + e[q]);
            } else if (STOPS) {
              const float cv = __builtin_ldexpf((float)nx, eb - 23);  // exact
              if (cv >= thr) cand = ((uint64_t)(Q * tid + q) << 32) | __float_as_uint(cv);
            }
          }
          cur = nx;
        }
      }
    }
    cand = wave_min_key(cand);
    if (lane == 0 && cand != ~0ull) __atomic_fetch_min(slot, cand, __ATOMIC_RELAXED);
    __syncthreads();
    const uint64_t res = *slot;
    if (res == ~0ull) {
      ++it;
      return __builtin_ldexpf((float)(C + ((C & 1u) ? tot.a1 : tot.a0)), eb - 23);
    }
    c = __uint_as_float((uint32_t)res);
    s = (uint32_t)(res >> 32) + 1u;
    if (STOPS && c >= thr) {
      stop_at = s - 1u;
      ++it;
      return c;
    }
    if (s >= NT * Q) {
      ++it;
      return c;
    }
  }
}
__device__ __forceinline__ float block_seq_sum(const float (&e)[16], uint32_t nq, float c,
                                               uint32_t& it, LDS uint32_t* sc) {
  uint32_t st;
  return block_seq_scan<false>(e, nq, c, it, sc, 0.0f, st);
}

// seq_scan's running sums of list[0..n) (mode 0: the total; 1 and 2: the
// first j whose running sum reaches thr) by the whole workgroup, for long
// lists (the slow path's nuclei): windows of NT*16 entries, thread t holding
// entries 16t .. 16t+15 of a window, each window through block_seq_scan.
// Returns (the stop index, n if none; the running sum there, the total if
// none).  sc: 6 + NW*2 words.  A call of its own, its registers apart from
// the kernel's.
__device__ __attribute__((noinline)) u2v block_list_scan(List list, uint32_t n, int mode,
                                                        float thr, LDS uint32_t* sc) {
  constexpr uint32_t Q = 16;
  const uint32_t tid = threadIdx.x;
  const bool stops = mode != 0;
  if (n > 0 && stops && thr <= 0.0f) return u2v{0u, __float_as_uint(0.0f + list.get(0))};
  if (tid < 3) ((LDS uint64_t*)sc)[tid] = ~0ull;  // the event slots start cleared
  __syncthreads();
  uint32_t it = 0, stop = n;
  float c = 0.0f;
  for (uint32_t w0 = 0; w0 < n; w0 += NT * Q) {
    float e[Q];
#pragma unroll
    for (uint32_t q = 0; q < Q; ++q) {
      const uint32_t i = w0 + Q * tid + q;
      e[q] = i < n ? list.get(i) : 0.0f;
    }
    uint32_t st;
    c = stops ? block_seq_scan<true>(e, Q, c, it, sc, thr, st)
              : block_seq_scan<false>(e, Q, c, it, sc, 0.0f, st);
    if (st != EMPTY) {
      stop = w0 + st;
      break;
    }
  }
  __syncthreads();  // the caller may reuse sc
  return u2v{stop, __float_as_uint(c)};
}

// ---------------------------------------------------------------------------
// Sequential f32 sums in binades
// ---------------------------------------------------------------------------
// While a running sum c >= 0 stays in the binade [2^eb, 2^(eb+1)) (below
// 2^-125 the quantum is 2^-149 throughout) it is an integer C of quanta
// q = 2^(eb-23), C < 2^24, and adding a term p adds round(p / q) quanta, a
// tie going to the even sum: the increment of a run of terms depends on C
// only through its parity, so a run is a pair of increments (from an even,
// from an odd C), and runs compose in order.  An increment that would take C
// to 2^24 or beyond leaves the binade; it saturates at XS_SAT, and the run is
// then taken apart.
constexpr uint32_t XS_SAT = 1u << 24;
__device__ __forceinline__ Par sat_then(Par f, Par g) {
  const uint32_t a0 = f.a0 + ((f.a0 & 1u) ? g.a1 : g.a0);
  const uint32_t a1 = f.a1 + ((f.a1 & 1u) ? g.a0 : g.a1);
  return Par{umin(a0, XS_SAT), umin(a1, XS_SAT)};
}
__device__ __forceinline__ Par wave_par_incl_sat(Par x) {
  x = sat_then(dpp_par<0x111, 0xf, true>(x), x);
  x = sat_then(dpp_par<0x112, 0xf, true>(x), x);
  x = sat_then(dpp_par<0x114, 0xf, true>(x), x);
  x = sat_then(dpp_par<0x118, 0xf, true>(x), x);
  x = sat_then(dpp_par<0x142, 0xa, false>(x), x);
  x = sat_then(dpp_par<0x143, 0xc, false>(x), x);
  return x;
}
// binade exponent of a positive normal or subnormal float (subnormals: -126)
__device__ __forceinline__ int binade_of(float c) {
  return (int)umax((__float_as_uint(c) >> 23) & 255u, 1u) - 127;
}
// floor(log2 x) of a positive normal double
__device__ __forceinline__ int binade_d(double x) {
  return (int)(((uint64_t)__double_as_longlong(x) >> 52) & 0x7ffu) - 1023;
}
// The pair of a lane's Q consecutive terms (>= 0) in the binade of exponent eb.
template <int Q>
__device__ __forceinline__ Par lane_pair(const float (&e)[Q], int eb) {
  uint32_t s0 = 0, s1 = 1;
#pragma unroll
  for (int q = 0; q < Q; ++q) {
    const float x = __builtin_fminf(__builtin_ldexpf(e[q], 23 - eb), 0x1p25f);
    const float k = __builtin_floorf(x);
    const float fr = x - k;
    const uint32_t ki = (uint32_t)k;
    const uint32_t r = fr > 0.5f ? ki + 1u : ki;
    const uint32_t t = fr == 0.5f ? 1u : 0u;
    s0 += r + (t & ((s0 ^ r) & 1u));
    s1 += r + (t & ((s1 ^ r) & 1u));
  }
  return Par{umin(s0, XS_SAT), umin(s1 - 1u, XS_SAT)};
}

// c + the terms of lanes pos .. nl - 1 of a wave in order, exactly (lane l
// holding terms Q l .. Q l + Q - 1, zeros past the count), by rounds: a lane
// at a time while c is 0 (from 0 the sum leaves its binade at almost every
// term); then the lanes' pairs in c's binade, a wave scan; the lanes before
// the first one where c leaves the binade are added by their pairs, that
// lane's terms one f32 addition each, and the scan resumes after it.  Every
// lane returns the sum.
// c + lane j's Q terms in order, one f32 addition each, added by lane j
// itself (a chain of register additions; read lane by lane into scalar
// registers the same chain is several times slower); j wave-uniform, every
// lane returns the sum.
template <int Q>
__device__ __forceinline__ float lane_chain(float c, const float (&p)[Q], uint32_t j) {
  float x = c;
  if ((threadIdx.x & 63u) == j) {
#pragma unroll
    for (int q = 0; q < Q; ++q) x = x + p[q];
  }
  return rl(x, j);
}
template <int Q>
__device__ __forceinline__ float wave_sum_rounds(float c, const float (&p)[Q], uint32_t nl,
                                                 uint32_t pos) {
  const uint32_t lane = threadIdx.x & 63u;
  while (pos < nl) {
    if (c == 0.0f) {
      c = lane_chain<Q>(c, p, pos);  // zeros past n add nothing
      ++pos;
      continue;
    }
    const int eb = binade_of(c);
    const uint32_t C = (uint32_t)__builtin_ldexpf(c, 23 - eb);
    Par x = Par{0u, 0u};
    if (lane >= pos) x = lane_pair<Q>(p, eb);
    const Par in = wave_par_incl_sat(x);
    const uint32_t inc = (C & 1u) ? in.a1 : in.a0;
    const uint64_t cross = __ballot(lane >= pos && lane < nl && C + inc >= XS_SAT);
    if (cross == 0ull) {
      c = __builtin_ldexpf((float)(C + (uint32_t)__builtin_amdgcn_readlane((int)inc, 63)), eb - 23);
      break;
    }
    const uint32_t l = (uint32_t)__builtin_ctzll(cross);
    const uint32_t Cb = l > pos ? C + (uint32_t)__builtin_amdgcn_readlane((int)inc, (int)l - 1) : C;
    c = lane_chain<Q>(__builtin_ldexpf((float)Cb, eb - 23), p, l);
    pos = l + 1;
  }
  return c;
}

// The runs of a wave's terms (lane l holding terms Q l .. Q l + Q - 1, zeros
// from lane nl on) for a running sum that enters them anywhere in [clo, chi].
// Each lane bounds the running sums over its terms from those bounds and the
// exact prefix of the lanes' sums: the sequential f32 sum of k positive terms
// from c is within k u (1.001) of the exact one (u = 2^-24 per addition; plus
// 2^-150 per addition below 2^-126), and a lane's own f32 sum within Q u of
// its terms'.  A lane whose bounds share one binade forms its pair there;
// consecutive such lanes of one binade form a run, and a segmented wave scan
// gives each lane its run's pair so far.  RunLane.k: the lane's binade + 512
// (0: no run, the lane is summed one addition a term), bit 16 set where a
// run (or such a lane) starts.
struct RunLane {
  uint32_t a0, a1, k;
};
template <int Q>
__device__ __forceinline__ RunLane seg_runs(const float (&p)[Q], uint32_t nl, double clo,
                                            double chi) {
  const uint32_t lane = threadIdx.x & 63u;
  float ls = 0.0f;
#pragma unroll
  for (int q = 0; q < Q; ++q) ls += p[q];
  const double lsd = (double)ls;
  const double pre = wave_prefix_d(lsd) - lsd;
  const double d = (double)(Q * (lane + 2u) + 4u) * 0x1p-24 * 1.02 + 0x1p-45;
  const double ab = (double)(Q * (lane + 1u)) * 0x1p-150;
  const double lo = (clo + pre) * (1.0 - d) - ab, hi = (chi + pre + lsd) * (1.0 + d) + ab;
  const int eb = binade_d(lo);
  const bool ok = lane < nl && lo >= 0x1p-126 && hi < 0x1p120 && binade_d(hi) == eb;
  const uint32_t key = ok ? (uint32_t)(eb + 512) : 0u;
  const uint32_t prev =
      (uint32_t)__builtin_amdgcn_ds_bpermute((int)(((lane + 63u) & 63u) * 4u), (int)key);
  const bool head = !ok || lane == 0 || prev != key;
  const uint64_t heads = __ballot(head);
  // each lane's run start, then the pairs scanned within runs
  const uint32_t rs = 63u - (uint32_t)__builtin_clzll(heads & ((2ull << lane) - 1ull));
  Par x = lane_pair<Q>(p, ok ? eb : 0);
  Par y = sat_then(dpp_par<0x111, 0xf, true>(x), x);
  x = rs + 1u <= lane ? y : x;
  y = sat_then(dpp_par<0x112, 0xf, true>(x), x);
  x = rs + 2u <= lane ? y : x;
  y = sat_then(dpp_par<0x114, 0xf, true>(x), x);
  x = rs + 4u <= lane ? y : x;
  y = sat_then(dpp_par<0x118, 0xf, true>(x), x);
  x = rs + 8u <= lane ? y : x;
  y = sat_then(dpp_par<0x142, 0xa, false>(x), x);
  x = rs + 1u <= (lane & ~15u) ? y : x;
  y = sat_then(dpp_par<0x143, 0xc, false>(x), x);
  x = rs <= 31u ? y : x;
  return RunLane{x.a0, x.a1, key | (head ? 0x10000u : 0u)};
}
// c + the terms of lanes 0 .. nl - 1 in order, exactly, c inside the bounds
// r was formed for: a run at once (its sum provably stays in its binade),
// every other lane (a binade crossing, or c = 0) one f32 addition a term.
// Where the sum is not where the bounds say (it cannot be; the check keeps
// the result exact whatever), the rest goes by rounds (wave_sum_rounds).
// Every lane returns the sum.
template <int Q>
__device__ __forceinline__ float runs_walk(float c, const float (&p)[Q], uint32_t nl, RunLane r) {
  const uint64_t heads = __ballot((r.k >> 16) & 1u);
  const uint64_t bad = __ballot((r.k & 0xffffu) == 0u);
  uint32_t pos = 0;
  while (pos < nl) {
    if ((bad >> pos) & 1ull) {
      c = lane_chain<Q>(c, p, pos);
      ++pos;
      continue;
    }
    const uint64_t after = heads & ~((2ull << pos) - 1ull);
    const uint32_t end = after ? (uint32_t)__builtin_ctzll(after) : 64u;
    const uint32_t last = (end < nl ? end : nl) - 1u;
    const int ebr = (int)((uint32_t)__builtin_amdgcn_readlane((int)r.k, (int)pos) & 0xffffu) - 512;
    if (!(c >= 0x1p-126f) || binade_of(c) != ebr) break;
    const uint32_t C = (uint32_t)__builtin_ldexpf(c, 23 - ebr);
    const uint32_t inc = (C & 1u) ? (uint32_t)__builtin_amdgcn_readlane((int)r.a1, (int)last)
                                  : (uint32_t)__builtin_amdgcn_readlane((int)r.a0, (int)last);
    if (C + inc >= XS_SAT) break;
    c = __builtin_ldexpf((float)(C + inc), ebr - 23);
    pos = last + 1u;
  }
  return pos < nl ? wave_sum_rounds<Q>(c, p, nl, pos) : c;
}
// c + the first n of a wave's terms in order, exactly, by their runs from c.
template <int Q>
__device__ __forceinline__ float wave_sum_q(float c, const float (&p)[Q], uint32_t n) {
  const uint32_t nl = (n + Q - 1) / Q;  // lanes holding terms
  if (nl == 0) return c;
  return runs_walk<Q>(c, p, nl, seg_runs<Q>(p, nl, (double)c, (double)c));
}

// A wave-uniform 64-bit value, or LDS pointer, in scalar registers.
__device__ __forceinline__ uint64_t sgpr_u64(uint64_t x) {
  const uint32_t lo = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)x);
  const uint32_t hi = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)(x >> 32));
  return ((uint64_t)hi << 32) | lo;
}
template <class T>
__device__ __forceinline__ LDS T* sgpr_lds(LDS T* p) {
  const uint32_t a = (uint32_t)(uintptr_t)p;
  return (LDS T*)(uintptr_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)a);
}


// Stable LSD radix sort of the keys src[0..npos) (pkey: the inverted bits of a
// probability in (0, 1], then the index) by probability, by the whole
// workgroup; the last pass writes the sorted probabilities and indices to pl
// and il itself (a pass of its own to unpack them cost the widest nuclei 5 %:
// 64 bf16 rows of 151936 with mixed parameters 1.18 -> 1.25 times the rate of
// the four-pass sort).  A probability's bits are at most
// 0x3f800000, so the inverted ones differ in their low 30 bits alone: three
// passes of 10 bits.  Each pass is a chain of rounds of 8192 keys (loads, the
// waves' ranks, two barriers, scattered stores) on one workgroup, so passes
// are what it costs: three, and one read of the keys for the histograms of
// all three, in place of four passes of 8 bits that each read the keys twice
// (64 bf16 rows of 151936 with mixed parameters 689 -> 586 us, 8 f16 rows of
// 32000 without top-k or top-p 345 -> 307 us a call).  A round
// ranks at most 8192 keys, so the waves' counts are 16 bits wide and their
// 1024 digits take no more room than the history's token table, which
// nothing reads any more.  Inlined: as a call of its own it measured C5
// 1.5 us slower (the stream kernel's code moves).
// wc: NW * 1024 counts, hist: 3 * 1024 words, base: 1024 words, red: 16.
constexpr uint32_t RS_BITS = 10, RS_DIGITS = 1u << RS_BITS;
static_assert(RS_DIGITS == NT, "a thread a digit");
static_assert(NW * RS_DIGITS / 2 <= U_MAX, "the counts fit the token table");
static_assert(3 * RS_DIGITS <= NW * 256 && RS_DIGITS <= SLOW_BINS, "the slow path's tables");
__device__ __forceinline__ void radix_sort_keys(GLB uint64_t* src, GLB uint64_t* dst,
                                                uint32_t npos, LDS uint16_t* wc,
                                                LDS uint32_t* hist, LDS uint32_t* base,
                                                LDS uint32_t* red, GLB float* pl,
                                                GLB uint32_t* il) {
  const uint32_t tid = threadIdx.x, lane = tid & 63u;
  const uint32_t wv = (uint32_t)__builtin_amdgcn_readfirstlane((int)(tid >> 6));
  src = (GLB uint64_t*)sgpr_u64((uint64_t)src);
  dst = (GLB uint64_t*)sgpr_u64((uint64_t)dst);
  pl = (GLB float*)sgpr_u64((uint64_t)pl);
  il = (GLB uint32_t*)sgpr_u64((uint64_t)il);
  npos = (uint32_t)__builtin_amdgcn_readfirstlane((int)npos);
  constexpr int RE = 8;
  constexpr uint32_t DM = RS_DIGITS - 1u;
  LDS uint16_t* mine = wc + wv * RS_DIGITS;  // this wave's counts
  // cleared two at a time: a type of its own, since a plain 32-bit store may
  // by the aliasing rules move past the 16-bit reads
  typedef uint32_t __attribute__((may_alias)) CountPair;
  LDS CountPair* pairs = (LDS CountPair*)mine;
  for (uint32_t j = lane; j < RS_DIGITS / 2; j += WAVE) pairs[j] = 0;
  for (uint32_t j = tid; j < 3 * RS_DIGITS; j += NT) hist[j] = 0;
  __syncthreads();
  // the digit histograms of all passes, RE keys per thread loaded at once.
  // Lane 0 adds for every lane of its wave that holds its key (the valid lanes
  // are a prefix of the wave): adds to one address take their turns, which in
  // a row of equal logits is 64 a wave (64 such f32 rows of 128256 without
  // top-k or top-p: 1086 us a call with every lane's own add, 791 so; rows of
  // spread logits, where lane 0 seldom has company, stay within 1 %).
  for (uint32_t b0 = 0; b0 < npos; b0 += RE * NT) {
    uint32_t kk[RE];
#pragma unroll
    for (int q = 0; q < RE; ++q) {
      const uint32_t i = b0 + q * NT + tid;
      kk[q] = i < npos ? (uint32_t)(src[i] >> 32) : 0u;
    }
#pragma unroll
    for (int q = 0; q < RE; ++q) {
      const bool valid = b0 + q * NT + tid < npos;
      const uint32_t k0 = (uint32_t)__builtin_amdgcn_readfirstlane((int)kk[q]);
      const bool as0 = kk[q] == k0;
      const uint64_t alike = __ballot(valid && as0);
      const uint32_t n = lane == 0 ? (uint32_t)__popcll(alike) : 1u;
      if (valid && (lane == 0 || !as0)) {
#pragma unroll
        for (uint32_t ps = 0; ps < 3; ++ps)
          __atomic_fetch_add(&hist[ps * RS_DIGITS + ((kk[q] >> (RS_BITS * ps)) & DM)], n,
                             __ATOMIC_RELAXED);
      }
    }
  }
  __syncthreads();
  for (uint32_t ps = 0; ps < 3; ++ps) {
    const uint32_t sh_bits = 32u + RS_BITS * ps;
    // thread t: where digit t's keys begin
    uint32_t at;
    {
      const uint32_t c = hist[ps * RS_DIGITS + tid];
      const uint32_t incl = wave_incl_scan(c);
      if (lane == 63) red[wv] = incl;
      __syncthreads();
      at = incl - c;
      for (uint32_t q = 0; q < wv; ++q) at += red[q];
    }
    // stable scatter, RE * NT keys per round: wave w ranks its own run of
    // RE * 64 consecutive keys slot after slot (equal digits found by
    // ballots, counted on in the wave's counts), then one prefix per digit
    // across the waves (written over the counts) places every key; each wave
    // reads only its own counts when it scatters and clears them after, so
    // two barriers per round
    for (uint32_t b0 = 0; b0 < npos; b0 += RE * NT) {
      const uint32_t wb = b0 + wv * (RE * WAVE);
      uint64_t ky[RE];
      uint32_t pw[RE];
#pragma unroll
      for (int q = 0; q < RE; ++q) {
        const uint32_t i = wb + q * WAVE + lane;
        ky[q] = i < npos ? src[i] : 0ull;
      }
#pragma unroll
      for (int q = 0; q < RE; ++q) {
        const bool valid = wb + q * WAVE + lane < npos;
        const uint32_t d = (uint32_t)(ky[q] >> sh_bits) & DM;
        uint64_t peers = __ballot(valid);
        pw[q] = 0;
        if (peers == 0) continue;  // wave-uniform: this slot is past the keys
        // the lanes holding this lane's digit: all valid lanes when the wave
        // holds one digit, else matched bit by bit
        const uint32_t d0 = (uint32_t)__builtin_amdgcn_readfirstlane((int)d);
        if (__ballot(valid && d != d0) != 0) {
#pragma unroll
          for (uint32_t bit = 0; bit < RS_BITS; ++bit) {
            const uint64_t bb = __ballot(((d >> bit) & 1u) != 0);
            peers &= ((d >> bit) & 1u) ? bb : ~bb;
          }
        }
        const uint32_t rank = lanes_below(peers);
        const uint32_t n = valid ? (uint32_t)mine[d] : 0u;
        pw[q] = n + rank;
        WaveSync::sync();  // every lane has read the count before it moves on
        if (valid && rank == 0) mine[d] = (uint16_t)(n + (uint32_t)__popcll(peers));
        WaveSync::sync();  // the next slot reads the new counts
      }
      __syncthreads();
      {
        // thread t: digit t's sixteen counts read at once, then their prefix
        uint32_t c[NW];
#pragma unroll
        for (int w2 = 0; w2 < NW; ++w2) c[w2] = wc[w2 * RS_DIGITS + tid];
        uint32_t acc = 0;
#pragma unroll
        for (int w2 = 0; w2 < NW; ++w2) {
          wc[w2 * RS_DIGITS + tid] = (uint16_t)acc;
          acc += c[w2];
        }
        base[tid] = at;
        at += acc;
      }
      __syncthreads();
#pragma unroll
      for (int q = 0; q < RE; ++q) {
        if (wb + q * WAVE + lane < npos) {
          const uint32_t d = (uint32_t)(ky[q] >> sh_bits) & DM;
          const uint32_t o = base[d] + mine[d] + pw[q];
          if (ps < 2) {
            dst[o] = ky[q];
          } else {
            pl[o] = __uint_as_float(~(uint32_t)(ky[q] >> 32));
            il[o] = (uint32_t)ky[q];
          }
        }
      }
      WaveSync::sync();  // this wave's reads of its counts are done
#pragma unroll
      for (uint32_t j = 0; j < RS_DIGITS / 2; j += WAVE) pairs[j + lane] = 0;
      WaveSync::sync();  // the next round's slots read counts other lanes cleared
    }
    wait_stores();
    __syncthreads();
    if (tid == 0) __threadfence();
    __syncthreads();
    GLB uint64_t* tmp = src;
    src = dst;
    dst = tmp;
  }
}

enum : uint32_t {
  F_DONE = 0, F_S = 1, F_M = 2, F_TOTAL = 3, F_LAM = 4, F_PLIM = 5, F_L = 6, F_GREEDY = 7,
  F_SCR = 8,
  F_BAND = 120  // band_certain_wave's verdict (wave 1 beside wave 0's semantics)
};
// LDS layout of the finalize (words): slots, candidate lists, keys, tables
struct FinLds {
  LDS float* tl;        // MAX_SLOTS: slot maxima
  LDS float* ts;        // MAX_SLOTS: slot sums (or first argmax)
  LDS uint64_t* keys;   // SORT_CAP
  LDS uint64_t* skeys;  // SORT_CAP (sorted)
  LDS float* pp;        // SORT_CAP
  LDS uint32_t* pidx;   // SORT_CAP
  LDS uint32_t* fm;     // 128
  LDS uint32_t* soff;   // MAX_SEG + 16
  LDS uint32_t* red;    // 64
};
__device__ __forceinline__ FinLds fin_carve(LDS uint32_t* smem) {
  FinLds f;
  f.tl = (LDS float*)smem;
  f.ts = f.tl + MAX_SLOTS;
  f.keys = (LDS uint64_t*)(smem + 2 * MAX_SLOTS);
  f.skeys = f.keys + SORT_CAP;
  f.pp = (LDS float*)(f.skeys + SORT_CAP);
  f.pidx = (LDS uint32_t*)(f.pp + SORT_CAP);
  f.fm = f.pidx + SORT_CAP;
  f.soff = f.fm + 128;
  f.red = f.soff + MAX_SEG + 16;
  return f;
}

// Ascending sort of keys[0..n) into skeys[0..n) (keys distinct), by the
// whole workgroup.
//   n <= 256: a rank sort split over the threads (key i against one of
//     NT / npad segments in thread g * npad + i; the partial ranks meet in
//     LDS), three barriers;
//   n <= NT: one key per thread: NT bins over the range of the keys' top
//     words, the keys moved to bin order, then each key's rank among its bin
//     (a key or two, more only for equal probabilities);
//   larger n: a bitonic sort.
// The ranks, bins and moved keys use pp / pidx, free until the sorted keys
// are unpacked.
template <class SY>
__device__ __forceinline__ void sort_keys(const FinLds& f, uint32_t n) {
  if (n <= 256) {
    uint32_t npad = WAVE;
    while (npad < n) npad <<= 1;
    const uint32_t ns = SY::N / npad;
    const uint32_t seg = (n + ns - 1) / ns;
    const uint32_t i = SY::id() % npad, g = SY::id() / npad;
    LDS uint32_t* rk = (LDS uint32_t*)f.pp;
    if (SY::id() < n) rk[SY::id()] = 0;
    SY::sync();
    const uint32_t j0 = g * seg, j1 = umin(j0 + seg, n);
    if (i < n && j0 < j1) {
      const uint64_t k = f.keys[i];
      uint32_t r = 0;
      for (uint32_t j = j0; j < j1; ++j) r += (f.keys[j] < k) ? 1u : 0u;
      if (r) __atomic_fetch_add(&rk[i], r, __ATOMIC_RELAXED);
    }
    SY::sync();
    if (SY::id() < n) f.skeys[rk[SY::id()]] = f.keys[SY::id()];
    SY::sync();
    return;
  }
  if (n <= SY::N) {
    const uint32_t id = SY::id();
    LDS uint64_t* tmp = (LDS uint64_t*)f.pp;  // n keys in bin order
    LDS uint32_t* bo = (LDS uint32_t*)f.pp + 2 * SY::N;  // NT bin offsets
    LDS uint32_t* bq = bo + SY::N;                       // NT cursors
    const uint64_t k = id < n ? f.keys[id] : ~0ull;
    const uint32_t hi = (uint32_t)(k >> 32);
    const uint32_t hmin = block_min_u32(id < n ? hi : EMPTY, f.red);
    const uint32_t hmax = ~block_min_u32(id < n ? ~hi : EMPTY, f.red);
    uint32_t sh = 0;
    while (((hmax - hmin) >> sh) >= SY::N) ++sh;
    const uint32_t bi = (hi - hmin) >> sh;
    bo[id] = 0;
    SY::sync();
    if (id < n) __atomic_fetch_add(&bo[bi], 1u, __ATOMIC_RELAXED);
    SY::sync();
    {
      uint32_t tot;
      const uint32_t ex = block_excl_scan(bo[id], f.red, tot);
      bo[id] = ex;
      bq[id] = ex;
    }
    SY::sync();
    if (id < n) tmp[__atomic_fetch_add(&bq[bi], 1u, __ATOMIC_RELAXED)] = k;
    SY::sync();
    if (id < n) {
      const uint32_t o = bo[bi], oe = bi + 1 < SY::N ? bo[bi + 1] : n;
      uint32_t r = o;
      for (uint32_t j = o; j < oe; ++j) r += tmp[j] < k ? 1u : 0u;
      f.skeys[r] = k;
    }
    SY::sync();
    return;
  }
  uint32_t npad = 1;
  while (npad < n) npad <<= 1;
  for (uint32_t i = SY::id(); i < npad; i += SY::N) f.skeys[i] = i < n ? f.keys[i] : ~0ull;
  SY::sync();
  for (uint32_t k = 2; k <= npad; k <<= 1)
    for (uint32_t j = k >> 1; j > 0; j >>= 1) {
      for (uint32_t i = SY::id(); i < npad / 2; i += SY::N) {
        const uint32_t lo = ((i & ~(j - 1)) << 1) | (i & (j - 1));
        const uint32_t hi = lo | j;
        const uint64_t x = f.skeys[lo], y = f.skeys[hi];
        const bool up = (lo & k) == 0;
        if ((x > y) == up) {
          f.skeys[lo] = y;
          f.skeys[hi] = x;
        }
      }
      SY::sync();
    }
}

}  // namespace llmk
