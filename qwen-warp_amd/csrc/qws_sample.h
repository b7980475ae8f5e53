// The record format of the sampling kernels and k_resolve, shared by qws_sample.hip (k_scan, the sampling rows'
// k_resolve) and qws_verify.hip (the verify rows' k_resolve, instantiated there so that each kernel family keeps its
// own code object).  The overview of both kernels is at the top of qws_sample.hip.
#pragma once
#include <math.h>
#include <stdlib.h>

#include <atomic>
#include <mutex>

#include "qws_rows.h"

namespace qws {

constexpr int NT1S = 512, NT1L = 1024;        // k_scan workgroups: 3 per CU; one per CU when the grid fits one round
constexpr int NXCD = 8;                      // accelerator complex dies (XCDs), each with its own L2
// (row, block) items of k_scan per XCD: an equal share of the grid; with fewer rows than XCDs, a whole row (G items,
// one workgroup per CU of the XCD), so that each row's blocks and its k_resolve workgroup share one L2
__host__ __device__ inline int scan_chunk(int B, int G) { return B < NXCD && G <= 32 ? G : (B * G + NXCD - 1) / NXCD; }
inline unsigned scan_grid(int B, int G) { return (unsigned)(NXCD * scan_chunk(B, G)); }
constexpr int NT2 = 512, NWV2 = NT2 / 64;    // k_resolve workgroup
// k_resolve's grid: workgroup i takes row (i mod 8) * ceil(B / 8) + i / 8, the row k_scan ran on workgroup i's XCD
inline unsigned resolve_grid(int B) { return (unsigned)(NXCD * ((B + NXCD - 1) / NXCD)); }
constexpr int CAP = 1024;                    // elements a block may list
// The listed window of a block with more than CAP elements above its own cuts' deepest bin.
// top-p: a flat block's own boundary is close to the row's: MARGIN_FLAT fine bins on either side.  A peaked block (its top
// CTOP elements carry a quarter of its mass) lists one range of as many bins as the list holds, ending MARGIN_NEAR bins or
// BELOW elements below its boundary, whichever is nearer, or from its top when that fits: the row's boundary tends to lie
// above a block's own, since the outliers of other blocks add mass at the top, but where the bins are dense it is close.
// min-p: from the top when the cut expected in the row (from the spread of the block's G best) fits the list, else the bins
// ending at the block's own cut; with top-p too, the top-p window instead of the latter.
// Chosen on a CPU model over rows of 31 blocks: N(0, s) logits (s 0.5-6), N(0, 2.5) with 32 tokens 8 higher, Laplace,
// exponential, Gumbel, t(4), uniform and Zipf ones and a 1% mixture, T 0.7-1.3, top-p 0.3-0.999, min-p 0.001-0.1 and
// both.  Rescans of eight blocks per row, summed: 263 (265 with BELOW = CAP / 4); 340 with the range ending 31 bins below
// the boundary whatever they hold and the top under every min-p; 368 with two ranges, the top 256 elements and up to 100
// bins around the boundary.  On the GPU, 640 calls of such rows take 0.842 of the time with two ranges (k_resolve's rescans
// and small sets included).  The rows that still miss are those whose other blocks' outliers move the cut past 1,024 elements.
constexpr int MARGIN_FLAT = 6, MARGIN_NEAR = 31, BELOW = 3 * CAP / 8;
constexpr int CTOP = 256;
constexpr int MAXG = 64;                     // blocks per row (V <= 524,288)
constexpr int NR = NBIN;                     // row bins with a nonzero weight (row-relative, 0 = the top)
constexpr unsigned long long M40 = (1ull << 40) - 1;

// ---------------------------------------------------------------------------------------------- block record
enum : int { RF_CAND = 1, RF_SAMP = 2 };  // has a candidate; has bins (top-list records write no flags: listed_top)
// Bins of a block are top-down: rel = (c * 64 + 63) - fine bin, so rel 0..63 is the power of two 2^c of the block's
// best and rel >> 6 = e counts powers of two below it.  Elements with rel >= NBIN weigh nothing in any row.
struct Rec {
  uint32_t max_key, max_idx;     // best candidate's okey (KEY_NEGINF: none); its lowest index on greedy rows, 0 on sampled ones
  int c, flags;                  // power of two of the best; RF_*
  int nbw;                       // bins written: rel 0 .. nbw - 1 (every bin a cut of any row can fall in)
  int w0, w1;                    // listed bins: rel in [w0, w1] (none when w0 > w1)
  int n_list, n_patch;           // listed elements; processed touched tokens recorded (-1: more than TCAP)
  uint32_t pad[7];
  uint32_t ecnt[NEXP];           // candidates of power of two e = rel >> 6
  unsigned long long emu[NEXP];  // their summed mantissas (< 2^37)
};
constexpr size_t HDR_BYTES = 512;
static_assert(sizeof(Rec) <= HDR_BYTES && offsetof(Rec, ecnt) == 64 && offsetof(Rec, emu) % 8 == 0, "record header");
// then the bin words: mantissa sum (bits 0..36) | count (37..50) | list offset (51..61) | listed (62), then the
// listed elements comp(key, index), bucketed by bin, then the patches {local index, processed value}
constexpr size_t BIN_OFF = HDR_BYTES;
constexpr size_t EL_OFF = BIN_OFF + (size_t)NBIN * 8;
constexpr size_t PATCH_OFF = EL_OFF + (size_t)CAP * 8;
constexpr size_t REC_BYTES = PATCH_OFF + (size_t)TCAP * 8;
static_assert(CAP <= 2048 && BLK < (1 << 14), "bin word fields");
__device__ inline char* rec_of(char* ws, int G, int row, int g) { return ws + ((size_t)row * G + g) * REC_BYTES; }
constexpr unsigned long long BW_MU = (1ull << 37) - 1;
__device__ inline uint32_t bw_cnt(unsigned long long w) { return (uint32_t)(w >> 37) & 0x3FFFu; }
__device__ inline unsigned long long bw_mu(unsigned long long w) { return w & BW_MU; }
__device__ inline uint32_t bw_off(unsigned long long w) { return (uint32_t)(w >> 51) & 0x7FFu; }
__device__ inline bool bw_listed(unsigned long long w) { return (w >> 62) & 1ull; }

// ---- top-list records: rows whose top_k is at most TOPK_MAX.  Their kept set lies inside the row's top_k best
// candidates, so a block records its own best ones (at least top_k of them, or all it has; at most TOPN, unordered) and
// nothing else: no histogram, no window, no patches.  They fit the record's first 512 bytes, which the resolver reads in
// its first round of loads: a key and the token's index inside the block, 6 bytes each, in the header's place of the
// per-power sums.  Measured (k_scan / k_resolve, rocprofv3): 32 bf16 rows, top-k 50, 300 biases 22.0 / 8.9 -> 15.0 / 8.7 us;
// 80 bf16 verify rows, top-k 50, 46.6 / 22.2 -> 31.0 / 12.7 us; one fp32 row, top-k 20, 10.4 / 14.0 -> 8.4 / 8.0 us.
// Larger K keeps the general records: its candidates no longer fit one wave, and the bound's overshoot grows with K.
constexpr int TOPK_MAX = 64;                                  // the kept set fits one wave
// A bound is accepted once at most TOP_SLACK keys more than top_k reach it: the resolver's bisection without slack (top_k 64
// and at most 64 keys) ran through most of the 64 bits, 40 bf16 rows 17.0 -> 13.5 us.  A block's list keeps to 64 threads:
// with 72 it exceeds TOPN more often and is cut by a second bisection (40 rows, N(0, 3) 20.6 -> 22.0 us, tied values 24 -> 52).
constexpr int TOP_SLACK = 8;
constexpr int TOPN = (int)(HDR_BYTES - 64) / 6;               // 74
constexpr int TOP_KEYS = 64, TOP_IDS = TOP_KEYS + TOPN * 4;   // byte offsets of u32 okey[TOPN] and u16 local[TOPN]
static_assert(TOP_IDS + TOPN * 2 <= (int)HDR_BYTES && TOPN >= TOPK_MAX, "top list inside the header");
// Test flags that ask for rescans, staged draws or separate passes keep the general records.
__device__ inline bool listed_top(const qws_row& R) {
  return R.top_k > 0 && R.top_k <= TOPK_MAX && R.temperature > 0.0f && kscale(R.temperature) < INFINITY &&
         !(R.test_flags & (QWS_TF_RESCAN | QWS_TF_STAGED_DRAW | QWS_TF_SPLIT_SELECT));
}

// A key that at least `need` of a wave's N keys per lane reach (key(j): the calling lane's j-th), and few more: a
// bisection between lo (keys below it, as the 0 of an empty place, never count) and the largest key, which stops at the
// first bound that at most `enough` keys reach.  *n = the keys at or above the returned bound: fewer than `need` only
// when fewer exist; more than `enough` only when the keys equal to the bound are tied (fewer than `need` above it).
template <int N, typename T, typename F>
__device__ __forceinline__ T top_bound(F key, T lo, int need, int enough, int* n) {
  auto count = [&](T b) {
    int c = 0;
#pragma unroll
    for (int j = 0; j < N; j++) c += __popcll(__ballot(key(j) >= b));
    return c;
  };
  T lm = key(0);
#pragma unroll
  for (int j = 1; j < N; j++) lm = key(j) > lm ? key(j) : lm;
  T h, bot;  // past the largest key, and the smallest of the lanes' largest (64 keys or more lie at or above it)
  if constexpr (sizeof(T) == 8) {
    h = wave_max_u64(lm) + 1;
    bot = wave_min_u64(lm);
  } else {
    h = wave_max_u32(lm) + 1;
    bot = ~wave_max_u32(~lm);
  }
  if (need <= 64 && bot > lo) lo = bot;
  int c = count(lo);
  while (c > enough && h - lo > 1) {  // uniform
    const T mid = lo + (h - lo) / 2;
    const int cm = count(mid);
    if (cm >= need) {
      lo = mid;
      c = cm;
    } else {
      h = mid;
    }
  }
  *n = c;
  return lo;
}

// ---------------------------------------------------------------------------------------------- k_resolve
// One workgroup per row.  Global loads come in few parallel rounds (the headers; the fine bins of one power of two of
// every block; one bin's listed elements; the block of the draw); everything else runs from LDS.
constexpr int NBK = 256;         // buckets of a round of the in-bin selection
constexpr int XG = 3072;         // elements of one bin held in LDS (a larger bin is streamed from its sources)
static_assert(MAXG * HDR_BYTES <= (size_t)MAXG * FB * 8, "the headers are staged in the fine-bin region");
static_assert(BLK / NT2 == 16, "a thread's 16 staged tokens start at word 17 t");

struct BI {                      // a block as the resolver uses it
  uint32_t max_key;
  int c, nbw, n_patch;
  int dn;                        // N - c (row powers of two above the block's top one); -1: nothing of it weighs in the row
  int gcnt, goff, gsrc, gofs;    // the bin being gathered: the block's count, list offset, source (0 none, 1 list, 2 rescan),
                                 // first slot in the gathered list
  int w0, w1;                    // the block's listed bins (its record header's window)
  int n_list, wcnt;              // its listed elements; its candidates inside the row's weight window
};

struct RS {                      // row state (LDS)
  int G, N, row_top;
  int fpow;                      // row power of two whose fine bins are staged (-1: none)
  int gbin, gn, gl, gstaged;     // the gathered bin: row bin, elements, listed ones, held in LDS
  int gres;                      // blocks of the gathered bin rescanned (their window missed it)
  unsigned long long gfast;      // bit g: block g is rescanned from its raw logits and patches (rescan_fast)
  unsigned long long gslow;      // bit g: block g is rescanned through the staged block (more processed tokens than patches)
  float xlo, xhi;                // the gathered bin's value interval (bin_edges), when gfast is not 0
  int rescans;                   // blocks rescanned because their window missed a bin
  float K;
  unsigned long long best;
  uint32_t Rc[NEXP];             // the row's candidates per power of two (row power e: 2^(N - e))
  unsigned long long Rm[NEXP];   // their summed mantissas (< 2^42)
  uint32_t fcnt[FB];             // the staged power's fine bins over the row: counts, mantissa sums
  unsigned long long fmu[FB];
  uint32_t pcnt[NWV2][FB];       // stage_power's per-wave partial sums
  unsigned long long pmu[NWV2][FB];
  int si[8];
  unsigned long long su[8];
  unsigned long long kmin, kmax;
  unsigned long long gmin, gmax;  // comp range of the gathered bin (held in LDS)
  unsigned long long wmn[NWV2], wmx[NWV2];  // per-wave comp ranges of a bin gathered by select_listed
  uint32_t bcnt[NBK];
  unsigned long long bsum[NBK];
  unsigned long long Klo[MAXG], Khi[MAXG];  // kept mass per block (row units)
  uint64_t xs[64], xv[64];
  uint32_t fbc[NBK];             // topp_cut_fast's buckets (zeroed at the start of k_resolve, used once per row)
  unsigned long long fbs[NBK];
  int fxn;                       // its crossing bucket's elements
  uint64_t fxs[64], fxv[64];
};

struct RL {                      // k_resolve LDS views
  BI* bi;
  RS* st;
  float2* ts;
  uint32_t* big;                 // [BIGW]: a staged block
  unsigned long long* fb;        // [MAXG][FB]: the staged power's bin words per block (first: the staged headers)
  unsigned long long* emu;       // [MAXG][NEXP]: the blocks' per-power mantissa sums
  uint64_t* ec;                  // [XG] gathered elements: comp
  uint32_t* em;                  //                          mantissa
  int* nt;
  u128* red;
};

__device__ inline u128 ld128(unsigned long long lo, unsigned long long hi) { return ((u128)hi << 64) | lo; }
// row weight of one mantissa in row bin r (< 2^59)
__device__ inline uint64_t rw1(uint32_t mu, int r) { return (uint64_t)mu << (D_EXP - (r >> 6)); }
__device__ inline const QWS_G uint64_t* els_of(char* ws, int G, int row, int g) { return gmem((const uint64_t*)(rec_of(ws, G, row, g) + EL_OFF)); }
__device__ inline const QWS_G unsigned long long* bins_of(char* ws, int G, int row, int g) {
  return gmem((const unsigned long long*)(rec_of(ws, G, row, g) + BIN_OFF));
}
// The smallest sh with (range >> sh) < NBK: the bucket width of a selection round over a comp range
__device__ inline int bucket_shift(uint64_t range) {
  const int bits = range ? 64 - __clzll((long long)range) : 0;
  return max(bits - 8, 0);
}

// Sum / min / max of one value per thread over the workgroup, via one atomic per wave (st.su[7] / kmin / kmax); the
// caller reads the result after the barrier these end with.
__device__ inline void block_add_u64(RS& st, unsigned long long v) {
  if (threadIdx.x == 0) st.su[7] = 0ull;
  bar();
  v = wave_sum<unsigned long long>(v);
  if (lane_id() == 0 && v) atomicAdd(&st.su[7], v);
  bar();
}
__device__ inline void block_range_u64(RS& st, unsigned long long mn, unsigned long long mx) {
  if (threadIdx.x == 0) {
    st.kmin = ~0ull;
    st.kmax = 0ull;
  }
  bar();
  mn = wave_min_u64(mn);
  mx = wave_max_u64(mx);
  if (lane_id() == 0) {
    atomicMin(&st.kmin, mn);
    atomicMax(&st.kmax, mx);
  }
  bar();
}

// Staged block layout: token l at word l + l / 16, so that a thread reading its 16 consecutive tokens (word 17 t + k)
// and the other lanes of its wave hit distinct LDS banks.
constexpr int BIGW = BLK + BLK / 16;
__device__ inline int big_at(int l) { return l + (l >> 4); }

// k_resolve's LDS.  The rarer parts of a row (a min-p or top-k cut inside a bin, a top-p cut that the fast form does not
// take, dense probabilities) are out-of-line functions that get it by one LDS pointer: inlined, with the selections'
// several copies, the kernel was 76,000 instructions (ten times the instruction cache), and every launch fetches its
// path anew.
#define QWS_L __attribute__((address_space(3)))
struct ResolveLds {
  __attribute__((aligned(16))) unsigned long long fb[MAXG * FB];
  unsigned long long emu[MAXG * NEXP];
  uint64_t ec[XG];
  uint32_t em[XG];
  __attribute__((aligned(16))) uint32_t big[BIGW];
  __attribute__((aligned(16))) float2 ts[1024];
  __attribute__((aligned(16))) u128 red[NWV2 + 1];
  RS st;
  BI bi[MAXG];
  qws_batch B;                   // the call's arguments and the row, for the out-of-line parts
  qws_row R;
  int nt;
};
__device__ __forceinline__ RL rl_of(ResolveLds& S) { return RL{S.bi, &S.st, S.ts, S.big, S.fb, S.emu, S.ec, S.em, &S.nt, S.red}; }
__device__ __forceinline__ char* uniform_ptr(char* p) { return (char*)readlane<uint64_t>((uint64_t)p, 0); }

// A block's raw values as the stager loads them: the logits (thread layout of Blk), the mask words and the patches.
template <int DT>
struct Staged {
  using BL = Blk<DT, NT2>;
  float x[BL::EPT];
  uint32_t mw[BL::S];
  uint2 pv[TCAP / NT2];
  int lo, hi;  // the block's tokens
};
// Issues the loads of block g (recorded patches: n_patch >= 0) into S without waiting for them.
template <int DT>
__device__ __forceinline__ void stage_issue(const RL& L, const qws_batch& B, const qws_row& R, char* ws, int row, int g, Staged<DT>& S) {
  using BL = Blk<DT, NT2>;
  const int lo = g * BLK, hi = min(B.V, lo + BLK);
  const int np = L.bi[g].n_patch;
  const QWS_G unsigned long long* PT = gmem((const unsigned long long*)(rec_of(ws, L.st->G, row, g) + PATCH_OFF));
#pragma unroll
  for (int k = 0; k < TCAP / NT2; k++) {
    const int p = (int)threadIdx.x + k * NT2;
    const unsigned long long w = p < np ? PT[p] : 0xFFFFFFFFull;  // {local index, value bits}; local ~0: none
    S.pv[k] = make_uint2((uint32_t)w, (uint32_t)(w >> 32));
  }
  BL::load_raw(B, row, lo, hi, S.x);
  BL::mask_words(B, R, lo, hi, S.mw);
  S.lo = lo;
  S.hi = hi;
}
// Block g from S into L.big in token order: NaN -> -inf, the mask, then the patches.  All threads; ends with a barrier.
template <int DT>
__device__ __forceinline__ void stage_store(const RL& L, const qws_row& R, int g, Staged<DT>& S) {
  using BL = Blk<DT, NT2>;
  float* xs = (float*)L.big;
  BL::fixnan(S.x);
  BL::apply_mask(R, S.lo, S.hi, S.mw, S.x);
#pragma unroll
  for (int e = 0; e < BL::EPT; e++) xs[big_at(BL::local(e))] = S.x[e];
  if (L.bi[g].n_patch > 0) {
    bar();
#pragma unroll
    for (int k = 0; k < TCAP / NT2; k++)
      if (S.pv[k].x != 0xFFFFFFFFu) xs[big_at((int)S.pv[k].x)] = __uint_as_float(S.pv[k].y);
  }
  bar();
}

// Block g of the row, processed, into L.big in token order (tokens past V read -inf).  With the block's patches
// recorded by k_scan the raw logits get the mask and the patches (the patches load together with the logits);
// otherwise the processors are rebuilt from the row's lists.  B and R are the workgroup's LDS copies.  All threads, after a
// barrier that follows the last reads of L.big; ends with a barrier.
template <int DT>
__device__ __forceinline__ void stage_block_body(const RL& L, const qws_batch& B, const qws_row& R, char* ws, int row, int g) {
  using BL = Blk<DT, NT2>;
  const int lo = g * BLK, hi = min(B.V, lo + BLK);
  if (R.proc_on && L.bi[g].n_patch < 0) {
    float x[BL::EPT];
    float* xs = (float*)L.big;
    load_processed<DT, NT2>(B, R, row, lo, hi, L.big, x, nullptr, L.nt);
    bar();
#pragma unroll
    for (int e = 0; e < BL::EPT; e++) xs[big_at(BL::local(e))] = x[e];
    bar();
    return;
  }
  Staged<DT> S;
  stage_issue<DT>(L, B, R, ws, row, g, S);
  stage_store<DT>(L, R, g, S);
}
// The out-of-line copy for the rare rescans (the draw stages its block inline: a call would spill the caller's
// registers to scratch around it).
template <int DT>
__device__ __noinline__ void stage_block(QWS_L ResolveLds* s, char* ws, int row, int g) {
  ResolveLds& S = *(ResolveLds*)s;
  stage_block_body<DT>(rl_of(S), S.B, S.R, uniform_ptr(ws), __builtin_amdgcn_readfirstlane(row), __builtin_amdgcn_readfirstlane(g));
}

// The fine bins of row power p of every block into L.fb and summed over the row into st.fcnt / st.fmu.  Bins a block
// did not write lie below its deepest possible cut and read as empty.  Thread t loads fine bin t % 64 of blocks t / 64,
// t / 64 + 8, ... and sums them in registers; each wave's sums go to its row of st.part, and every wave then adds the
// eight rows up and writes the same totals (so no barrier is needed before a wave reads them).  All threads; when it
// stages, it begins with a barrier (the previous power's staged bins and sums may still be read) and has one more.
__device__ __forceinline__ void stage_power(const RL& L, char* ws, int row, int p) {
  RS& st = *L.st;
  const int G = st.G;
  if (st.fpow == p) return;  // uniform: every wave writes st.fpow itself, after the same barriers
  constexpr int NB = (MAXG * FB) / NT2;  // blocks per thread
  const int f = (int)threadIdx.x & 63, g0 = (int)threadIdx.x >> 6;
  unsigned long long w[NB];  // every load issued before the barrier
#pragma unroll
  for (int k = 0; k < NB; k++) {
    const int g = g0 + k * (NT2 / 64);
    w[k] = 0;
    if (g < G) {
      const BI& b = L.bi[g];
      const int pb = p - b.dn, rel = pb * FB + f;
      if (b.dn >= 0 && pb >= 0 && pb < NEXP && rel < b.nbw) w[k] = bins_of(ws, G, row, g)[rel];
    }
  }
  bar();
  uint32_t cn = 0;
  unsigned long long mu = 0;
#pragma unroll
  for (int k = 0; k < NB; k++) {
    const int g = g0 + k * (NT2 / 64);
    if (g < G) L.fb[g * FB + f] = w[k];
    cn += bw_cnt(w[k]);
    mu += bw_mu(w[k]);
  }
  st.pcnt[g0][f] = cn;
  st.pmu[g0][f] = mu;
  bar();
  cn = 0;
  mu = 0;
#pragma unroll
  for (int v = 0; v < NWV2; v++) {
    cn += st.pcnt[v][f];
    mu += st.pmu[v][f];
  }
  st.fcnt[f] = cn;  // every wave writes the same totals
  st.fmu[f] = mu;
  st.fpow = p;
}

// The first row power of two whose inclusive cumulative count reaches tgt (NEXP: none) -> *p, the count before it ->
// *before.  Every wave computes it from st.Rc (final after the per-power sums): no barrier.
__device__ __forceinline__ void pow_cross_cnt(const RL& L, unsigned long long tgt, int* p, unsigned long long* before) {
  const RS& st = *L.st;
  const int lane = lane_id();
  const unsigned long long v = lane < NEXP ? st.Rc[lane] : 0ull;
  const unsigned long long inc = wave_scan_incl<unsigned long long>(v);
  const int q = first_lane(lane < NEXP && inc >= tgt);
  const unsigned long long bf = readlane<unsigned long long>(inc - v, q < 64 ? q : 0);
  *p = q < NEXP ? q : NEXP;
  *before = q < NEXP ? bf : 0ull;
}
// The first row power whose inclusive cumulative mass (row units) reaches tgt (NEXP: none) -> *p, the mass before it
// -> *before.  Every wave, from st.Rm: no barrier.
__device__ __forceinline__ void pow_cross_mass(const RL& L, u128 tgt, int* p, u128* before) {
  const RS& st = *L.st;
  const int lane = lane_id();
  const u128 v = lane < NEXP ? shl128(st.Rm[lane], D_EXP - lane) : (u128)0;
  const u128 inc = wave_scan_incl_u128(v);
  const int q = first_lane(lane < NEXP && inc >= tgt);
  *before = readlane<u128>(inc - v, q < 64 ? q : 0);
  *p = q < NEXP ? q : NEXP;
}
// Over the staged power's fine bins: the first whose base + inclusive cumulative count (by_mass: mass in row units)
// reaches tgt -> returned (64: none), the cumulative value before it -> *before.  Every wave, from st.fcnt / st.fmu
// (final after stage_power): no barrier.
__device__ __forceinline__ int fine_cross(const RL& L, bool by_mass, u128 base, u128 tgt, u128* before) {
  const RS& st = *L.st;
  const int lane = lane_id();
  const u128 v = by_mass ? shl128(st.fmu[lane], D_EXP - st.fpow) : (u128)st.fcnt[lane];
  const u128 inc = wave_scan_incl_u128(v) + base;
  const int f = first_lane(inc >= tgt);
  *before = readlane<u128>(inc - v, f < 64 ? f : 0);
  return f;
}
// Mass (row units) and count of the row's candidates in bins above row bin r (r >= NR: every bin; else r's power's
// fine bins are staged).  Every wave, from st.Rm / st.Rc and the staged sums; ends with a barrier (the stage that
// follows may rewrite row state, such as the gathered bin's, that the stage before it read).
__device__ __forceinline__ void before_bin(const RL& L, int r, u128* mass, unsigned long long* count) {
  const RS& st = *L.st;
  const int lane = lane_id(), p = r >> 6;
  u128 m = lane < NEXP && lane < p ? shl128(st.Rm[lane], D_EXP - lane) : (u128)0;
  unsigned long long n = lane < NEXP && lane < p ? st.Rc[lane] : 0ull;
  if (r < NR && lane < (r & 63)) {
    m += shl128(st.fmu[lane], D_EXP - p);
    n += st.fcnt[lane];
  }
  *mass = wave_sum_u128(m);
  *count = wave_sum<unsigned long long>(n);
  bar();
}

// The smallest value x, in the order -inf < ... < -0 < +0 < ... < +inf, with tval(x, K) >= tc (tval is monotone in
// x, so tval(x, K) >= tc  <=>  x >= that value  <=>  okey(x) >= its okey).  From tc / K in a few steps of one value;
// false if more than 64 steps would be needed (the caller then selects by count).
__device__ inline bool first_x_t(float tc, float K, float* out) {
  if (tval(-INFINITY, K) >= tc) {
    *out = -INFINITY;
    return true;
  }
  auto step = [](float v, int d) {  // the next value below (d = -1) or above (d = 1), -0 and +0 distinct
    const uint32_t u = __float_as_uint(v);
    return okey_val(((u & 0x80000000u) ? ~u : (u | 0x80000000u)) + (uint32_t)d);
  };
  float x = tc / K;
  if (!(x == x) || fabsf(x) == INFINITY) return false;
  int n = 0;
  while (tval(x, K) >= tc && n < 64) {
    x = step(x, -1);
    n++;
  }
  while (!(tval(x, K) >= tc) && n < 128) {
    x = step(x, 1);
    n++;
  }
  if (n >= 64 || !(tval(x, K) >= tc) || tval(step(x, -1), K) >= tc) return false;
  *out = x;
  return true;
}

// block of flat gathered-list index i (blocks' gofs ascending, list sources only)
__device__ inline int gblock_at(const RL& L, int G, int i) {
  int a = 0, b = G - 1;
  while (a < b) {
    const int m = (a + b + 1) >> 1;
    if (L.bi[m].gofs <= i)
      a = m;
    else
      b = m - 1;
  }
  return a;
}
__device__ inline uint32_t mu_of_comp(uint64_t c, float K, const float2* ts) { return weigh(tval(okey_val(comp_key(c)), K), ts).mu; }

// The values x of the bin with floor(tval(x, K)) >> 4 == qb: xlo <= x < xhi exactly (tval is monotone in x; NaN and -inf lie
// outside).  False where the edges are no exact floats or lie at the clamps of t, or first_x_t gives up.
__device__ inline bool bin_edges(int qb, float K, float* xlo, float* xhi) {
  if (qb <= -(1 << 19) || qb >= (1 << 19)) return false;  // |t| < 2^23 + 16: multiples of 16 are exact
  return first_x_t((float)(16 * qb), K, xlo) && first_x_t((float)(16 * qb + 16), K, xhi) && *xlo > -INFINITY;
}

// Calls fn(comp, mu) for every candidate of row bin rb (gathered: from LDS; else from the blocks' lists and rescans).
// All threads; ends with a barrier.
template <int DT, typename F>
__device__ __forceinline__ void for_bin(ResolveLds& S, char* ws, int row, F fn) {
  using BL = Blk<DT, NT2>;
  const RL L = rl_of(S);
  const RS& st = *L.st;
  const int tid = threadIdx.x;
  if (st.gstaged) {
    for (int i = tid; i < st.gn; i += NT2) fn(L.ec[i], L.em[i]);
    bar();
    return;
  }
  const int G = st.G, rb = st.gbin;
  for (int i = tid; i < st.gl; i += NT2) {
    const int g = gblock_at(L, G, i);
    const BI& b = L.bi[g];
    const uint64_t c = els_of(ws, G, row, g)[b.goff + (i - b.gofs)];
    fn(c, mu_of_comp(c, st.K, L.ts));
  }
  for (int g = 0; g < (st.gres ? G : 0); g++) {
    if (L.bi[g].gsrc != 2) continue;
    stage_block<DT>((QWS_L ResolveLds*)&S, ws, row, g);
    const float* xs = (const float*)L.big;
    const int t0 = tid * BL::EPT;
#pragma unroll
    for (int k = 0; k < BL::EPT; k++) {
      const float v = xs[big_at(t0) + k];
      const W w = weigh(tval(v, st.K), L.ts);
      if (v != -INFINITY && st.row_top - w.bin() == rb) fn(comp(okey(v), (uint32_t)(g * BLK + t0 + k)), w.mu);
    }
    bar();
  }
  bar();
}

// The blocks of st.gfast rescanned for the elements of row bin rb, into the gathered list: their raw logits, streamed through
// registers RD blocks deep, each value tested against the bin's interval (bin_edges).  A wave counts its hits in a block,
// takes their slots with one atomic and writes their comps; the mantissas follow for all of them at the end, one per
// thread.  Masked and processed tokens are marked in a bitmap per block (in L.big) that takes raw values out, and the
// patches' values are tested themselves.  (Through the staged block, one at a time, a block costs ~5 us.)
// Bound by what one CU loads (~16 bytes per cycle: 31 fp32 blocks 26 us) and the tests beside it.  Out of line: the rare
// path's registers would spill the resolver's other paths; few of them and little code (15 KB), since it saves its callers'
// and every call fetches it anew.  32 rows, k_resolve: one block missed 29.0 -> 26.1 us, 31 missed 68.8 -> 59.1, 31 missed for
// each of two cuts 171.7 -> 112.7, against batches of eight blocks held in registers whose every element was placed through
// an LDS atomic of its own (62 KB of code, 300 bytes of frame); RD 2 and 4 within 0.9 us of 3.
// All threads; ends with a barrier that hands L.big over: a block staged next clears it before a barrier of its own
// (load_processed), and a wave still testing the last bitmaps would take masked and processed tokens' raw values.
template <int DT>
__device__ __noinline__ void rescan_fast(QWS_L ResolveLds* s, char* ws_, int row_, int rb_) {
  using BL = Blk<DT, NT2>;
  ResolveLds& S = *(ResolveLds*)s;
  const RL L = rl_of(S);
  const qws_batch& B = S.B;
  const qws_row& R = S.R;
  RS& st = *L.st;
  char* const ws = uniform_ptr(ws_);
  const int row = __builtin_amdgcn_readfirstlane(row_);
  const int G = __builtin_amdgcn_readfirstlane(st.G), V = __builtin_amdgcn_readfirstlane(B.V), tid = threadIdx.x, lane = lane_id();
  constexpr int RD = 3, BW32 = BLK / 32, GRP = 32;
  static_assert(GRP * BW32 + GRP <= BIGW && MAXG <= 2 * GRP, "bitmaps of a group of blocks and their numbers");
  uint32_t* const bm = L.big;
  int* const gl = (int*)(L.big + GRP * BW32);  // the group's blocks
  const float xlo = st.xlo, xhi = st.xhi;
  auto hit = [&](float v) { return v >= xlo && v < xhi; };
  unsigned long long fm = readlane<unsigned long long>(st.gfast, 0);  // in scalar registers: the loops branch on it
  const bool marks = R.mask_mode != 0 || __ballot(lane < G && ((fm >> lane) & 1ull) && L.bi[lane].n_patch > 0) != 0ull;  // uniform
  while (fm) {  // uniform; a group of at most GRP blocks, the lowest first
    unsigned long long gm = fm;
    if (__popcll(gm) > GRP) gm &= 0xFFFFFFFFull;  // MAXG <= 64: each half holds at most GRP
    fm &= ~gm;
    const unsigned long long gm0 = gm;
    if (marks) {
      const int nb = __popcll(gm);
      bar();  // the bitmaps of the group before are read no more
      if (tid < 64 && ((gm >> lane) & 1ull)) gl[__popcll(gm & ((1ull << lane) - 1ull))] = lane;
      bar();
      const uint32_t flip = R.mask_mode == QWS_MASK_ALLOWED ? 0xFFFFFFFFu : 0u;
      const unsigned* const mrow = B.masks + (R.mask_mode ? (size_t)R.mask_row * (size_t)B.mask_words : 0);
#pragma unroll 4
      for (int i = tid; i < nb * BW32; i += NT2) {
        const int w = gl[i / BW32] * BW32 + i % BW32;
        bm[i] = R.mask_mode && w * 32 < V ? gmem(mrow)[w] ^ flip : 0u;
      }
      bar();
      for (int j = wave_id(); j < nb; j += NWV2) {  // a wave per block's patches
        const int g = gl[j], np = L.bi[g].n_patch;
        const QWS_G unsigned long long* PT = gmem((const unsigned long long*)(rec_of(ws, G, row, g) + PATCH_OFF));
        for (int i0 = lane; i0 < np; i0 += 256) {
          unsigned long long pv[4];
#pragma unroll
          for (int k = 0; k < 4; k++) pv[k] = i0 + 64 * k < np ? PT[i0 + 64 * k] : 0xFFFFFFFFull;  // {local index, value}; local ~0: none
#pragma unroll
          for (int k = 0; k < 4; k++) {
            const uint32_t l = (uint32_t)pv[k];
            if (l == 0xFFFFFFFFu) continue;
            atomicOr(&bm[j * BW32 + (l >> 5)], 1u << (l & 31));
            const float v = __uint_as_float((uint32_t)(pv[k] >> 32));
            if (hit(v)) {
              const int p = L.bi[g].gofs + atomicAdd(&L.bi[g].goff, 1);
              if (p < XG) L.ec[p] = comp(okey(v), (uint32_t)g * BLK + l);  // always: the bin words count these elements
            }
          }
        }
      }
      bar();
    }
    typename BL::Raw raw[RD];
    float xr[RD][BL::EPT];  // bf16 blocks stay packed in raw
    int gq[RD];
    auto next = [&](int d) {  // the next block's loads issued
      gq[d] = gm ? __ffsll((long long)gm) - 1 : -1;
      gm &= gm - 1ull;
      if (gq[d] >= 0) BL::load_bits(B, row, gq[d] * BLK, min(V, gq[d] * BLK + BLK), raw[d], xr[d]);  // uniform; -inf past V
    };
#pragma unroll
    for (int d = 0; d < RD; d++) next(d);
    while (gq[0] >= 0) {  // uniform
#pragma unroll
      for (int d = 0; d < RD; d++) {
        const int g = gq[d];
        if (g < 0) break;  // uniform
        float x[BL::EPT];
        if constexpr (DT == QWS_DTYPE_F32) {
#pragma unroll
          for (int e = 0; e < BL::EPT; e++) x[e] = xr[d][e];
        } else {
          BL::unpack(raw[d], x);
        }
        uint32_t hm = 0;  // bit e: element e lies in the bin
#pragma unroll
        for (int e = 0; e < BL::EPT; e++) hm |= hit(x[e]) ? 1u << e : 0u;
        if (marks) {
          const uint32_t* const bg = bm + __popcll(gm0 & ((1ull << g) - 1ull)) * BW32;
#pragma unroll
          for (int t = 0; t < BL::S; t++) {  // a stripe's VEC tokens share a bitmap word
            const int l = BL::local(t * BL::VEC);
            hm &= ~(((bg[l >> 5] >> (l & 31)) & ((1u << BL::VEC) - 1u)) << (t * BL::VEC));
          }
        }
        const int c = __popc(hm), inc = wave_scan_incl<int>(c), tot = readlane<int>(inc, 63);
        if (tot) {  // uniform in the wave
          int base = 0;
          if (lane == 63) base = atomicAdd(&L.bi[g].goff, tot);
          int p = L.bi[g].gofs + readlane<int>(base, 63) + inc - c;
#pragma unroll
          for (int e = 0; e < BL::EPT; e++) {
            if ((hm >> e) & 1u) {
              if (p < XG) L.ec[p] = comp(okey(x[e]), (uint32_t)(g * BLK + BL::local(e)));  // always, as above
              p++;
            }
          }
        }
        next(d);
      }
    }
  }
  bar();  // every comp is there (and the bitmaps in L.big are read no more)
  const int i1 = min(st.si[7], XG);  // the rescanned blocks' slots: behind the listed ones
  unsigned long long mn = ~0ull, mx = 0ull;
  for (int i = st.gl + tid; i < i1; i += NT2) {
    const uint64_t c = L.ec[i];
    L.em[i] = mu_of_comp(c, st.K, L.ts);
    mn = c < mn ? c : mn;
    mx = c > mx ? c : mx;
  }
  mn = wave_min_u64(mn);
  mx = wave_max_u64(mx);
  if (lane == 0) {
    atomicMin(&st.gmin, mn);
    atomicMax(&st.gmax, mx);
  }
  bar();  // st.si[7] is read no more
}

// Gathers row bin rb (its power's fine bins staged): each block's elements come from its list when its window held
// the bin, else from a rescan of the block.  The bin is held in LDS when it has at most XG elements.  All threads.
template <int DT>
__device__ __forceinline__ void gather(ResolveLds& S, char* ws, int row, int rb) {
  const RL L = rl_of(S);
  const qws_row& R = S.R;
  RS& st = *L.st;
  const int G = st.G, tid = threadIdx.x;
  if (st.gbin == rb) return;  // uniform: st.gbin is written only after the barrier below, which every wave passes after this test
  if (tid < 64) {
    // slots of the staged bin: the listed blocks' elements first (block order), then those of the blocks rescanned
    // from their raw logits (block order, each at a slot range fixed by its bin count), then the other rescans
    const int g = tid;
    uint32_t cn = 0, ln = 0, fr = 0;
    int nres = 0;
    if (g < G) {
      BI& b = L.bi[g];
      const unsigned long long w = L.fb[g * FB + (rb & 63)];
      cn = bw_cnt(w);
      b.gcnt = (int)cn;
      b.goff = (int)bw_off(w);
      b.gsrc = cn == 0 ? 0 : ((bw_listed(w) && !(R.test_flags & QWS_TF_RESCAN)) ? 1 : 2);
      ln = b.gsrc == 1 ? cn : 0u;
      fr = b.gsrc == 2 && b.n_patch >= 0 ? cn : 0u;
      nres = b.gsrc == 2 ? 1 : 0;
    }
    if (__ballot(fr != 0) != 0ull) {  // uniform in the wave
      float xlo = 0.0f, xhi = 0.0f;
      if (!bin_edges(st.row_top - rb, st.K, &xlo, &xhi)) fr = 0;  // through the staged block
      if (tid == 0) {
        st.xlo = xlo;
        st.xhi = xhi;
      }
    }
    const uint32_t linc = wave_scan_incl<uint32_t>(ln), finc = wave_scan_incl<uint32_t>(fr);
    const uint32_t tot = wave_sum<uint32_t>(cn), nl = readlane<uint32_t>(linc, 63);
    const bool staged = tot <= (uint32_t)XG;
    const unsigned long long fast = staged ? __ballot(fr != 0) : 0ull, slow = __ballot(nres != 0) & ~fast;
    if (g < G) {
      // unstaged, gofs stays the listed prefix (ascending over the blocks, as for_bin's block search needs)
      L.bi[g].gofs = fr && staged ? (int)(nl + finc - fr) : (int)(linc - ln);
      if (fr && staged) L.bi[g].goff = 0;  // the rescan's slot cursor (a rescanned block has no list offset)
    }
    const int nr = wave_sum<int>(nres);
    if (tid == 0) {
      st.gl = (int)nl;
      st.gn = (int)tot;
      st.gstaged = 0;
      st.gres = nr;
      st.gfast = fast;
      st.gslow = slow;
      st.gmin = ~0ull;  // the staged bin's comp range, reduced by one atomic per wave at the end
      st.gmax = 0ull;
      st.si[7] = (int)(nl + readlane<uint32_t>(finc, 63));  // the first slot of the other rescans
      st.rescans += nr;
    }
  }
  bar();
  if (tid == 0) st.gbin = rb;  // read again only after this function's last barrier
  if (st.gn <= XG) {
    const int nl = st.gl;
    // eight threads per block (G <= 64), each loading every eighth element of its block's list range, U loads in
    // flight (a block's first 64 elements in one round); the comp range of the bin is reduced on the way (the
    // selection's first range)
    constexpr int U = 8;
    unsigned long long mn = ~0ull, mx = 0ull;
    {
      const int g = tid >> 3, j = tid & 7;
      if (g < G && L.bi[g].gsrc == 1) {
        const BI& b = L.bi[g];
        const QWS_G uint64_t* src = els_of(ws, G, row, g) + b.goff;
        for (int i0 = j; i0 < b.gcnt; i0 += 8 * U) {
          uint64_t cv[U];
#pragma unroll
          for (int k = 0; k < U; k++) cv[k] = i0 + 8 * k < b.gcnt ? src[i0 + 8 * k] : 0ull;
#pragma unroll
          for (int k = 0; k < U; k++) {
            const int i = i0 + 8 * k;
            if (i < b.gcnt) {
              L.ec[b.gofs + i] = cv[k];
              L.em[b.gofs + i] = mu_of_comp(cv[k], st.K, L.ts);
              mn = cv[k] < mn ? cv[k] : mn;
              mx = cv[k] > mx ? cv[k] : mx;
            }
          }
        }
      }
    }
    bar();
    using BL = Blk<DT, NT2>;
    if (st.gfast) rescan_fast<DT>((QWS_L ResolveLds*)&S, ws, row, rb);  // uniform
    for (unsigned long long sm = st.gslow; sm; sm &= sm - 1ull) {  // uniform: read after the barrier
      const int g = __ffsll((long long)sm) - 1;
      if (tid == 0) L.bi[g].gofs = st.si[7];  // the block's elements follow (their order within the block is free)
      stage_block<DT>((QWS_L ResolveLds*)&S, ws, row, g);
      const float* xs = (const float*)L.big;
      const int t0 = tid * BL::EPT;
#pragma unroll
      for (int k = 0; k < BL::EPT; k++) {
        const float v = xs[big_at(t0) + k];
        const W w = weigh(tval(v, st.K), L.ts);
        if (v != -INFINITY && st.row_top - w.bin() == rb) {
          const int p = atomicAdd(&st.si[7], 1);
          const uint64_t c = comp(okey(v), (uint32_t)(g * BLK + t0 + k));
          mn = c < mn ? c : mn;
          mx = c > mx ? c : mx;
          if (p < XG) {  // always: the bin words count these elements
            L.ec[p] = c;
            L.em[p] = w.mu;
          }
        }
      }
      bar();
    }
    mn = wave_min_u64(mn);
    mx = wave_max_u64(mx);
    if (lane_id() == 0) {
      atomicMin(&st.gmin, mn);
      atomicMax(&st.gmax, mx);
    }
    if (tid == 0) st.gstaged = 1;
  }
  bar();
}

// The selection: in comp-descending order over the gathered bin, the first element whose inclusive prefix of value
// (1 per element, or its mantissa) reaches target (>= 1): its comp -> st.su[4] and that prefix -> st.su[5] (both
// left as they were when the target exceeds the bin's total).  Radix refinement on the whole comp (value key, then
// index): each round buckets the elements of the current comp range into NBK equal ranges, finds the bucket where the
// prefix crosses the target and narrows the range to it; at most a wave of elements left are ranked directly.
//
// select_rounds: the rounds from the comp range [kmin, kmax] with value base before it.  All threads, after a barrier
// that follows the last reads of the buckets.
template <int DT>
__device__ __forceinline__ void select_rounds(ResolveLds& S, char* ws, int row, bool by_mass, uint64_t target,
                                              uint64_t kmin, uint64_t kmax, uint64_t base) {
  RS& st = S.st;
  const int tid = threadIdx.x;
  for (int round = 0; round < 16; round++) {
    const int sh = bucket_shift(kmax - kmin);
    for (int i = tid; i < NBK; i += NT2) {
      st.bcnt[i] = 0;
      st.bsum[i] = 0;
    }
    bar();
    for_bin<DT>(S, ws, row, [&](uint64_t c, uint32_t mu) {
      if (c >= kmin && c <= kmax) {
        const int b = NBK - 1 - (int)((c - kmin) >> sh);  // bucket 0 = the largest comps
        atomicAdd(&st.bcnt[b], 1u);
        atomicAdd(&st.bsum[b], by_mass ? (unsigned long long)mu : 1ull);
      }
    });
    if (wave_id() == 0) {  // the bucket where base + the prefix of the bucket values crosses the target
      const int lane = lane_id();
      uint64_t v[NBK / 64], loc = 0;
#pragma unroll
      for (int k = 0; k < NBK / 64; k++) {
        v[k] = st.bsum[lane * (NBK / 64) + k];
        loc += v[k];
      }
      const uint64_t incl = wave_scan_incl<uint64_t>(loc);
      uint64_t run = base + incl - loc, before = 0;
      int hit = -1;
#pragma unroll
      for (int k = 0; k < NBK / 64; k++) {
        if (hit < 0 && run + v[k] >= target) {
          hit = lane * (NBK / 64) + k;
          before = run;
        }
        run += v[k];
      }
      const int l = first_lane(hit >= 0);
      if (lane == (l < 64 ? l : 0)) {
        st.si[4] = l < 64 ? hit : -1;
        st.su[6] = before;
        st.si[5] = l < 64 ? (int)st.bcnt[hit] : 0;
      }
    }
    bar();
    const int hb = st.si[4];
    if (hb < 0) return;  // the target exceeds the total
    base = st.su[6];
    const int nb = st.si[5];
    const uint64_t bl = kmin + ((uint64_t)(NBK - 1 - hb) << sh);
    const uint64_t span = (1ull << sh) - 1;
    const uint64_t bh = kmax - bl <= span ? kmax : bl + span;
    if (nb <= 64) {  // at most a wave of elements left: wave 0 ranks them directly
      if (tid == 0) st.si[3] = 0;
      bar();
      for_bin<DT>(S, ws, row, [&](uint64_t c, uint32_t mu) {
        if (c >= bl && c <= bh) {
          const int p = atomicAdd(&st.si[3], 1);
          if (p < 64) {  // always: the bucket held nb <= 64 of them
            st.xs[p] = c;
            st.xv[p] = by_mass ? (uint64_t)mu : 1ull;
          }
        }
      });
      if (wave_id() == 0) {
        const int lane = lane_id();
        const uint64_t c = lane < nb ? st.xs[lane] : 0ull;
        const uint64_t v = lane < nb ? st.xv[lane] : 0ull;
        uint64_t above = 0;  // value of the elements with a larger comp
        for (int j = 0; j < nb; j++) {
          const uint64_t cj = readlane<uint64_t>(c, j), vj = readlane<uint64_t>(v, j);
          above += cj > c ? vj : 0ull;
        }
        const bool hit = lane < nb && base + above < target && base + above + v >= target;
        const int l = first_lane(hit);
        if (lane == (l < 64 ? l : 0) && l < 64) {
          st.su[4] = c;
          st.su[5] = base + above + v;
        }
      }
      bar();
      return;
    }
    kmin = bl;
    kmax = bh;
  }
}
// select_in_bin: the selection over the gathered bin (gather called first).  All threads.
template <int DT>
__device__ __forceinline__ void select_in_bin(ResolveLds& S, char* ws, int row, bool by_mass, uint64_t target) {
  RS& st = S.st;
  if (!st.gstaged) {
    unsigned long long mn = ~0ull, mx = 0ull;
    for_bin<DT>(S, ws, row, [&](uint64_t c, uint32_t) {
      mn = c < mn ? c : mn;
      mx = c > mx ? c : mx;
    });
    block_range_u64(st, mn, mx);
  } else {
    bar();
  }
  const uint64_t kmin = st.gstaged ? st.gmin : st.kmin, kmax = st.gstaged ? st.gmax : st.kmax;
  if (kmin > kmax) return;
  select_rounds<DT>(S, ws, row, by_mass, target, kmin, kmax, 0ull);
}

// The gather and selection of row bin rb together, for a bin whose elements all lie in their blocks' lists and fit
// in LDS (the dense cut bin of a flat row): every wave finds each element's block from the per-block counts held in
// its lanes, so the element loads need no barrier before them; the first bucket round runs over the elements held in
// registers; every wave finds the crossing bucket and ranks its elements itself.  Three barriers where gather and
// select_in_bin take about ten; the same result, and the same gathered-bin state left in LDS.  The crossing
// element's comp -> *cut, its inclusive prefix -> *incl (~0 and 0 when the target exceeds the bin's total).  Returns
// false, having changed nothing, when the bin does not qualify (a block's elements not listed, more than XG
// elements, rescans or separate passes asked for by the test flags, or the bin gathered already).  A barrier must
// separate the previous selection's last reads of its buckets from this call.  All threads.
constexpr int XS = XG / NT2;  // elements per thread
static_assert(XG % NT2 == 0 && MAXG <= 64, "select_listed layout");
template <int DT>
__device__ __forceinline__ bool select_listed(ResolveLds& S, char* ws, int row, int rb, bool by_mass, uint64_t target,
                                              uint64_t* cut, uint64_t* incl) {
  const RL L = rl_of(S);
  const qws_row& R = S.R;
  RS& st = *L.st;
  const int G = st.G, tid = threadIdx.x, lane = lane_id();
  if (st.gbin == rb || (R.test_flags & (QWS_TF_RESCAN | QWS_TF_SPLIT_SELECT))) return false;  // uniform: st.gbin is written after the first barrier below
  uint32_t cn = 0, off = 0;  // lane g: block g's count in the bin and its list offset
  bool unlisted = false;
  if (lane < G) {
    const unsigned long long w = L.fb[lane * FB + (rb & 63)];
    cn = bw_cnt(w);
    off = bw_off(w);
    unlisted = cn != 0 && !bw_listed(w);
  }
  const uint32_t inc = wave_scan_incl<uint32_t>(cn), tot = readlane<uint32_t>(inc, 63), exc = inc - cn;
  if (__ballot(unlisted) != 0ull || tot == 0u || tot > (uint32_t)XG) return false;  // uniform: the same words in every wave
  if (tid < 64) {  // the gathered-bin state gather leaves: block g's elements at LDS slots [exc, inc)
    if (lane < G) {
      BI& b = L.bi[lane];
      b.gcnt = (int)cn;
      b.goff = (int)off;
      b.gsrc = cn ? 1 : 0;
      b.gofs = (int)exc;
    }
    if (lane == 0) {
      st.gl = st.gn = (int)tot;
      st.gstaged = 1;
      st.gres = 0;
      st.gfast = st.gslow = 0ull;
      st.si[3] = 0;
    }
  }
  for (int i = tid; i < NBK; i += NT2) {
    st.bcnt[i] = 0u;
    st.bsum[i] = 0ull;
  }
  // element i = tid + k NT2 of the bin (blocks in order, each block's in list order): its block by a binary search
  // over the lanes' inclusive counts; every load issued before any is used (a slot past the end reloads the last)
  uint64_t ce[XS];
  uint32_t me[XS];
#pragma unroll
  for (int k = 0; k < XS; k++) {
    if (k * NT2 >= (int)tot) break;  // uniform
    const int i = min(tid + k * NT2, (int)tot - 1);
    int g = 0;
#pragma unroll
    for (int s = 32; s > 0; s >>= 1) g += __shfl((int)inc, g + s - 1) <= i ? s : 0;
    const int e = __shfl((int)exc, g), o = __shfl((int)off, g);
    ce[k] = els_of(ws, G, row, g)[o + (i - e)];
  }
  unsigned long long mn = ~0ull, mx = 0ull;
#pragma unroll
  for (int k = 0; k < XS; k++) {
    if (k * NT2 >= (int)tot) break;  // uniform
    const int i = tid + k * NT2;
    me[k] = mu_of_comp(ce[k], st.K, L.ts);
    if (i < (int)tot) {
      L.ec[i] = ce[k];
      L.em[i] = me[k];
      mn = ce[k] < mn ? ce[k] : mn;
      mx = ce[k] > mx ? ce[k] : mx;
    }
  }
  mn = wave_min_u64(mn);
  mx = wave_max_u64(mx);
  if (lane == 0) {
    st.wmn[wave_id()] = mn;
    st.wmx[wave_id()] = mx;
  }
  bar();
  if (tid == 0) st.gbin = rb;
  uint64_t kmin = st.wmn[0], kmax = st.wmx[0];
#pragma unroll
  for (int w = 1; w < NWV2; w++) {
    kmin = st.wmn[w] < kmin ? st.wmn[w] : kmin;
    kmax = st.wmx[w] > kmax ? st.wmx[w] : kmax;
  }
  if (tid == 0) {  // the bin's range, as gather leaves it
    st.gmin = kmin;
    st.gmax = kmax;
  }
  const int sh = bucket_shift(kmax - kmin);
#pragma unroll
  for (int k = 0; k < XS; k++) {
    if (k * NT2 >= (int)tot) break;  // uniform
    if (tid + k * NT2 < (int)tot) {
      const int b = NBK - 1 - (int)((ce[k] - kmin) >> sh);  // bucket 0 = the largest comps
      atomicAdd(&st.bcnt[b], 1u);
      atomicAdd(&st.bsum[b], by_mass ? (unsigned long long)me[k] : 1ull);
    }
  }
  bar();
  // every wave: the bucket where the prefix of the bucket values crosses the target
  uint64_t base;
  int hb, nb;
  {
    uint64_t v[NBK / 64], loc = 0;
#pragma unroll
    for (int k = 0; k < NBK / 64; k++) {
      v[k] = st.bsum[lane * (NBK / 64) + k];
      loc += v[k];
    }
    const uint64_t inc2 = wave_scan_incl<uint64_t>(loc);
    uint64_t run = inc2 - loc, before = 0;
    int hit = -1;
#pragma unroll
    for (int k = 0; k < NBK / 64; k++) {
      if (hit < 0 && run + v[k] >= target) {
        hit = lane * (NBK / 64) + k;
        before = run;
      }
      run += v[k];
    }
    const int l = first_lane(hit >= 0);
    if (l >= 64) {  // the target exceeds the bin's total
      *cut = ~0ull;
      *incl = 0ull;
      return true;
    }
    hb = readlane<int>(hit, l);
    base = readlane<uint64_t>(before, l);
    nb = (int)st.bcnt[hb];
  }
  const uint64_t bl = kmin + ((uint64_t)(NBK - 1 - hb) << sh);
  const uint64_t span = (1ull << sh) - 1;
  const uint64_t bh = kmax - bl <= span ? kmax : bl + span;
  if (nb > 64) {  // more rounds, over the elements in LDS
    bar();
    select_rounds<DT>(S, ws, row, by_mass, target, bl, bh, base);
    *cut = st.su[4];
    *incl = st.su[5];
    return true;
  }
#pragma unroll
  for (int k = 0; k < XS; k++) {
    if (k * NT2 >= (int)tot) break;  // uniform
    if (tid + k * NT2 < (int)tot && ce[k] >= bl && ce[k] <= bh) {
      const int p = atomicAdd(&st.si[3], 1);
      if (p < 64) {  // always: the bucket holds nb <= 64 of them
        st.xs[p] = ce[k];
        st.xv[p] = by_mass ? (uint64_t)me[k] : 1ull;
      }
    }
  }
  bar();
  // every wave: the bucket's elements ranked directly
  const uint64_t c = lane < nb ? st.xs[lane] : 0ull;
  const uint64_t v = lane < nb ? st.xv[lane] : 0ull;
  uint64_t above = 0;  // value of the elements with a larger comp
  for (int j = 0; j < nb; j++) {  // uniform
    const uint64_t cj = readlane<uint64_t>(c, j), vj = readlane<uint64_t>(v, j);
    above += cj > c ? vj : 0ull;
  }
  const int l = first_lane(lane < nb && base + above < target && base + above + v >= target);
  *cut = l < 64 ? readlane<uint64_t>(c, l) : ~0ull;
  *incl = l < 64 ? base + readlane<uint64_t>(above + v, l) : 0ull;
  return true;
}

// The top-p cut inside row bin rb together with every block's kept mass, for a bin whose elements every block holding
// some has listed (at most 8 FPT per block): the common case of a flat row's dense cut bin.  Eight threads per block
// each load up to FPT of the block's listed elements of rb into registers and weigh them; the elements are bucketed by
// their value key over the key range the bin's t interval [16 qb, 16 qb + 16) spans (clamped at its ends, so the
// buckets stay in comp order without a reduction of the actual range); every wave finds the bucket where the prefix
// of the mantissas (comp-descending) crosses target, and ranks that bucket's elements (at most 64) itself.  Then the
// same eight threads of each block sum its kept mass in row units -- its powers above the cut's, its fine bins above
// rb and its elements of rb from the cut on -- into st.Klo / st.Khi.  Three barriers where select_listed and the
// separate kept-mass pass take about seven.  The crossing element's comp -> *cut, its inclusive mantissa prefix ->
// *incl.  Returns false, having changed nothing the other paths read, when the bin does not qualify (a block's
// elements not listed or more than 8 FPT of them, the bin gathered already, test flags asking for other paths) or
// its crossing bucket holds more than 64 elements.  rb's power must be the staged one, and the fast-cut state
// (st.fbc, st.fbs, st.fxn) as k_resolve's start leaves it.  All threads; ends with a barrier.
constexpr int FPT = 8;
static_assert(MAXG * 8 <= NT2, "eight threads per block");
__device__ __forceinline__ bool topp_cut_fast(const RL& L, const qws_row& R, char* ws, int row, int rb, uint64_t target, uint64_t* cut,
                                              uint64_t* incl) {
  RS& st = *L.st;
  const int G = st.G, tid = threadIdx.x, lane = lane_id();
  if (st.gbin == rb || (R.test_flags & (QWS_TF_RESCAN | QWS_TF_SPLIT_SELECT))) return false;  // uniform
  {
    bool bad = false;
    if (lane < G) {
      const unsigned long long w = L.fb[lane * FB + (rb & 63)];
      const uint32_t cn = bw_cnt(w);
      bad = cn != 0 && (!bw_listed(w) || cn > 8u * FPT);
    }
    if (__ballot(bad) != 0ull) return false;  // uniform: the same words in every wave
  }
  const int g = tid >> 3, j = tid & 7;
  const bool own = g < G;
  uint32_t cn = 0, off = 0;
  if (own) {
    const unsigned long long w = L.fb[g * FB + (rb & 63)];
    cn = bw_cnt(w);
    off = bw_off(w);
  }
  // the block's elements j, j + 8, ...: every load issued before any is used
  uint64_t ce[FPT];
  uint32_t me[FPT];
  {
    const QWS_G uint64_t* src = els_of(ws, G, row, own ? g : 0) + off;
#pragma unroll
    for (int k = 0; k < FPT; k++) ce[k] = j + 8 * k < (int)cn ? src[j + 8 * k] : 0ull;
  }
  // each block's kept mass above the cut bin in row units, while the loads are in flight: its powers above the cut's
  // (u128) and its fine bins above rb (mantissas, < 2^40 for eight of them), summed over the block's eight lanes
  const int pc = rb >> 6, fsh = D_EXP - pc;
  u128 km = 0;
  uint64_t mbin = 0;
  if (own && L.bi[g].dn >= 0) {
    const int dn = L.bi[g].dn;
    for (int er = dn + j; er < pc; er += 8) km += shl128(L.emu[g * NEXP + er - dn], D_EXP - er);
    for (int f = j; f < (rb & 63); f += 8) mbin += bw_mu(L.fb[g * FB + f]);
  }
#pragma unroll
  for (int x = 1; x < 8; x <<= 1) {  // sums over the block's eight lanes (xor partners stay inside the group)
    uint32_t w[6] = {(uint32_t)km, (uint32_t)(km >> 32), (uint32_t)(km >> 64), (uint32_t)(km >> 96), (uint32_t)mbin, (uint32_t)(mbin >> 32)};
#pragma unroll
    for (int i = 0; i < 6; i++) w[i] = (uint32_t)__shfl_xor((int)w[i], x);
    km += ((u128)w[3] << 96) | ((u128)w[2] << 64) | ((u128)w[1] << 32) | (u128)w[0];
    mbin += ((uint64_t)w[5] << 32) | w[4];
  }
  // bucket range: the keys of the bin's t interval (x = t / K is increasing in t for K > 0)
  const float K = st.K;
  const int qb = st.row_top - rb;
  const uint32_t klo = okey((float)(16 * qb) / K), khi = okey((float)(16 * qb + 16) / K);
  const uint32_t span = khi > klo ? khi - klo : 0u;
  const int bsh = max((span ? 32 - __clz((int)span) : 0) - 8, 0);
#pragma unroll
  for (int k = 0; k < FPT; k++) {
    if (j + 8 * k >= (int)cn) continue;
    me[k] = mu_of_comp(ce[k], K, L.ts);
    const uint32_t key = comp_key(ce[k]);
    const uint32_t d = key > klo ? (key - klo) >> bsh : 0u;
    const int b = NBK - 1 - (int)min(d, (uint32_t)(NBK - 1));  // bucket 0 = the largest keys
    atomicAdd(&st.fbc[b], 1u);
    atomicAdd(&st.fbs[b], (unsigned long long)me[k]);
  }
  bar();
  // every wave: the bucket where the prefix of the bucket sums crosses the target
  uint64_t base;
  int hb, nb;
  {
    uint64_t v[NBK / 64], loc = 0;
#pragma unroll
    for (int k = 0; k < NBK / 64; k++) {
      v[k] = st.fbs[lane * (NBK / 64) + k];
      loc += v[k];
    }
    const uint64_t inc2 = wave_scan_incl<uint64_t>(loc);
    uint64_t run = inc2 - loc, before = 0;
    int hit = -1;
#pragma unroll
    for (int k = 0; k < NBK / 64; k++) {
      if (hit < 0 && run + v[k] >= target) {
        hit = lane * (NBK / 64) + k;
        before = run;
      }
      run += v[k];
    }
    const int l = first_lane(hit >= 0);
    if (l >= 64) return false;  // uniform: the target exceeds the bin (not reached: the bin was found by this target)
    hb = readlane<int>(hit, l);
    base = readlane<uint64_t>(before, l);
    nb = (int)st.fbc[hb];
  }
  if (nb > 64) return false;  // uniform
  {
#pragma unroll
    for (int k = 0; k < FPT; k++) {
      if (j + 8 * k >= (int)cn) continue;
      const uint32_t key = comp_key(ce[k]);
      const uint32_t d = key > klo ? (key - klo) >> bsh : 0u;
      if (NBK - 1 - (int)min(d, (uint32_t)(NBK - 1)) == hb) {
        const int p = atomicAdd(&st.fxn, 1);
        if (p < 64) {  // always: the bucket holds nb <= 64 of them
          st.fxs[p] = ce[k];
          st.fxv[p] = me[k];
        }
      }
    }
  }
  bar();
  // every wave: the bucket's elements ranked directly
  uint64_t cC, pref;
  {
    const uint64_t c = lane < nb ? st.fxs[lane] : 0ull;
    const uint64_t v = lane < nb ? st.fxv[lane] : 0ull;
    uint64_t above = 0;  // value of the elements with a larger comp
    for (int i = 0; i < nb; i++) {  // uniform
      const uint64_t ci = readlane<uint64_t>(c, i), vi = readlane<uint64_t>(v, i);
      above += ci > c ? vi : 0ull;
    }
    const int l = first_lane(lane < nb && base + above < target && base + above + v >= target);
    if (l >= 64) return false;  // uniform (not reached: the bucket holds the crossing)
    cC = readlane<uint64_t>(c, l);
    pref = base + readlane<uint64_t>(above + v, l);
  }
  // each block's kept elements of rb (mantissas), summed over its eight lanes, complete its kept mass
  uint64_t mown = 0;
#pragma unroll
  for (int k = 0; k < FPT; k++)
    if (j + 8 * k < (int)cn && ce[k] >= cC) mown += me[k];
#pragma unroll
  for (int x = 1; x < 8; x <<= 1) {
    const uint32_t lo = (uint32_t)__shfl_xor((int)(uint32_t)mown, x), hi = (uint32_t)__shfl_xor((int)(uint32_t)(mown >> 32), x);
    mown += ((uint64_t)hi << 32) | lo;
  }
  km += shl128(mbin + mown, fsh);
  if (own && j == 0) {
    st.Klo[g] = (unsigned long long)km;
    st.Khi[g] = (unsigned long long)(km >> 64);
  }
  bar();
  *cut = cC;
  *incl = pref;
  return true;
}

// The draw inside block g when its kept set lies whole in its list (every bin down to the cut listed, n <= 64 listed
// elements there): the token whose interval of the kept weights (index order) holds the local target tl, from lane i
// holding listed element i.  One wave; the same token as draw_in_block.
__device__ __forceinline__ int draw_listed(const RL& L, char* ws, int row, int g, int n, int cR, uint64_t cC, u128 tl) {
  const RS& st = *L.st;
  const int lane = lane_id();
  uint64_t w = 0;
  uint32_t idx = 0xFFFFFFFFu;
  if (lane < n) {
    const uint64_t c = els_of(ws, st.G, row, g)[lane];
    const float t = tval(okey_val(comp_key(c)), st.K);
    const int r = st.row_top - (tfloor(t) >> 4);
    if (r < cR || (r == cR && r < NR && c >= cC)) w = rw1(weigh(t, L.ts).mu, r);  // cR == NR: no cut
    idx = comp_idx(c);
  }
  u128 below = 0;  // kept weight of the listed elements before this one in index order
  for (int j = 0; j < n; j++) {  // uniform
    const uint32_t ij = readlane<uint32_t>(idx, j);
    const uint64_t wj = readlane<uint64_t>(w, j);
    below += ij < idx ? (u128)wj : (u128)0;
  }
  const int l = first_lane(w != 0 && below <= tl && tl < below + w);
  return l < 64 ? (int)readlane<uint32_t>(idx, l) : -1;
}

// Kept weight (row units) of one staged token: 0 outside the cut.  NINF: -inf excluded by value, needed when the row's
// best lies within the window's depth of the lower clamp (-inf shares t = -2^30 with the clamped finite values)
// t = tval(v, K) and e its table entry (read beforehand, so that no branch separates the loop's LDS reads)
template <bool NINF>
__device__ __forceinline__ uint64_t kept_weight(float v, float t, float2 e, int row_top, int cR, uint64_t cC, uint32_t idx) {
  const W ww = weigh_e(t, e);
  const int r = row_top - ww.bin();
  bool keep = r < cR;
  if (r == cR) keep = r < NR && comp(okey(v), idx) >= cC;  // cR == NR: no cut
  if constexpr (NINF) keep = keep && v != -INFINITY;
  const uint64_t wk = (uint64_t)ww.mu << (D_EXP - min(r >> 6, D_EXP));  // r >= 0: no token lies above the row's best
  return keep ? wk : 0ull;
}

// The token whose interval of the kept weights of block g (index order) holds the local target tl.  All threads.
template <int DT>
__device__ __forceinline__ int draw_in_block(const RL& L, const qws_batch& B, const qws_row& R, char* ws, int row, int g, int cR, uint64_t cC, u128 tl) {
  using BL = Blk<DT, NT2>;
  constexpr int EPT = BL::EPT;
  RS& st = *L.st;
  const int lo = g * BLK;
  const float* xs = (const float*)L.big;
  if (threadIdx.x == 0) st.si[2] = -1;
  stage_block_body<DT>(L, B, R, ws, row, g);  // the processed block in L.big, token order
  const int t0 = (int)threadIdx.x * EPT;
  const float K = st.K;
  const int row_top = st.row_top;
  // the thread's values, then their table entries, each in one round of LDS reads
  float xv[EPT], tv[EPT];
  float2 te[EPT];
#pragma unroll
  for (int k = 0; k < EPT; k++) xv[k] = xs[big_at(t0) + k];
#pragma unroll
  for (int k = 0; k < EPT; k++) {
    tv[k] = tval(xv[k], K);
    te[k] = L.ts[tab_index(tv[k])];
  }
  uint64_t w[EPT];
  uint64_t loc = 0;  // EPT weights < 2^59 each: the thread's sum fits 64 bits
  if (row_top + (1 << 26) < NR) {  // uniform: -inf's bin (t = -2^30) lies inside the window
#pragma unroll
    for (int k = 0; k < EPT; k++) w[k] = kept_weight<true>(xv[k], tv[k], te[k], row_top, cR, cC, (uint32_t)(lo + t0 + k));
  } else {
#pragma unroll
    for (int k = 0; k < EPT; k++) w[k] = kept_weight<false>(xv[k], tv[k], te[k], row_top, cR, cC, (uint32_t)(lo + t0 + k));
  }
#pragma unroll
  for (int k = 0; k < EPT; k++) loc += w[k];
  u128 tot;
  const u128 incl = block_scan_incl_u128<NWV2>((u128)loc, L.red, &tot);
  const u128 c0 = incl - loc;
  if (c0 <= tl && tl < incl) {
    const uint64_t t = (uint64_t)(tl - c0);  // < loc
    uint64_t run = 0;
#pragma unroll
    for (int k = 0; k < EPT; k++) {
      if (w[k] && run <= t && t < run + w[k]) st.si[2] = lo + t0 + k;
      run += w[k];
    }
  }
  bar();
  return st.si[2];
}

// The step of a row that drew `tok`, on the device (qws_batch.advance): the token added to the row's state slot as
// qws_state_note adds one token (its block's entry counted, saturating, or appended), then the row's ngen and
// position incremented in the row array.  When tok lies in block g_pre, n_pre / e_pre are that block's entry count
// and this thread's first entry (entry threadIdx.x), loaded ahead.  All threads (tok and the row uniform); ends with
// the row written.
__device__ __forceinline__ void advance_row(const qws_batch& B, const qws_row& R, int row, int tok, int* s_hit, int g_pre, int n_pre, uint32_t e_pre) {
  if (tok < 0) return;
  const int slot = row_state(B, R);
  if (slot >= 0) {
    const int g = tok / BLK;
    const uint32_t local = (uint32_t)(tok - g * BLK);
    uint32_t* cnt = state_counts(B.state_mem, B.V, slot);
    uint32_t* ent = state_entries(B.state_mem, B.V, slot, g);
    const bool pre = g == g_pre;
    const int n0 = min(pre ? n_pre : (int)cnt[g], BLK);
    if (threadIdx.x == 0) *s_hit = -1;
    bar();
    for (int j = (int)threadIdx.x; j < n0; j += NT2)
      if (((pre && j < NT2 ? e_pre : ent[j]) & SE_LOCAL) == local) *s_hit = j;  // distinct tokens: one writer at most
    bar();
    if (threadIdx.x == 0) {
      const int j = *s_hit;
      if (j >= 0) {
        const uint32_t e = ent[j];
        ent[j] = (e & ((1u << SE_CNT_SHIFT) - 1u)) | (min((e >> SE_CNT_SHIFT) + 1u, SE_CNT_MAX) << SE_CNT_SHIFT);
      } else {
        const uint32_t p = atomicAdd(&cnt[g], 1u);
        if (p < (uint32_t)BLK) ent[p] = local | (1u << SE_CNT_SHIFT);
      }
    }
  }
  if (threadIdx.x == 0) {
    qws_row* rw = const_cast<qws_row*>(B.rows) + row;
    rw->ngen = R.ngen + 1;
    rw->position = R.position + 1u;
  }
}

// ---------------------------------------------------------------------------------------------- top-list rows
// A row of top-list records (listed_top): its top_k best candidates from the blocks' lists, then min-p, top-p and the
// draw over them by one wave, one candidate per lane in rank order.  The same definition as the general path: a
// candidate below the row's weight window weighs nothing and still counts for top-k; min-p, top-k and top-p each keep a
// prefix of the rank order, so their order does not matter to the kept set.
// Selection: a bound from the threads' largest entries that at least top_k entries reach (top_bound; the entries are
// distinct, so it ends), the entries at or above it gathered (about top_k + a few) and ranked by counting.  Latency
// bound (one workgroup per row): one round of global loads, then LDS round trips; every loop over LDS entries has a
// fixed length, so that its reads go out together.
// hdrs: the blocks' records' first 512 bytes; ts: the exp2 table; buf: TOP_BUF bytes.  All threads, uniform arguments;
// returns the row's token (-1: none) once its outputs are written.  Out of line: inlined into k_resolve it slowed the
// general rows by its place in the code (C4 resolve 20.5 -> 22.4 us).
struct TopRow {
  int row, V, G, K, B;
  uint32_t u_draw;
  float temperature, top_p, min_p;
  double log2_min_p;
  unsigned long long thr_lo, thr_hi;       // finish_small: the top-p threshold (row units), 0 = from top_p over the candidates
  int* out_tokens;
  int* out_info;
  float* out_probs;
  RowRes* rres;
};
constexpr int TOP_NL1 = 128;               // entries ranked at once
constexpr int TOP_EPL = (TOPN + 7) / 8;    // entries per thread at most (G > 32: eight threads per block)
struct TopBuf {
  uint64_t mxs[NT2];                       // the threads' largest entries, later the reduced list
  uint64_t lst[64 * TOP_EPL];              // entries at or above the bound (zeros past them, to TOP_NL1)
  uint32_t rk[4][TOP_NL1];                 // partial ranks
  uint64_t srt[64];                        // the top_k best in rank order
  uint64_t w[64];                          // their kept weights (row units)
  uint64_t part[NWV2][64];                 // partial sums of the kept weights before a candidate in index order
  uint64_t bound;
  int cnt, tok;
  int cnt2;                                // entries of the reduced list (its own word: late waves may still read cnt)
};
static_assert(TOP_NL1 <= NT2 / 4 && TOP_NL1 <= 64 * TOP_EPL && sizeof(TopBuf) <= BIGW * 4, "LDS of resolve_top");
// Inclusive prefix over lanes of row weights (< 2^59 each: a row of 16 lanes sums to less than 2^63)
__device__ inline u128 wave_scan_weights(uint64_t v) {
  v = row16_scan_incl<uint64_t>(v);
  const uint64_t r0 = readlane<uint64_t>(v, 15), r1 = readlane<uint64_t>(v, 31), r2 = readlane<uint64_t>(v, 47);
  const int row = lane_id() >> 4;
  const u128 b1 = r0, b2 = b1 + r1, b3 = b2 + r2;
  return (u128)v + (row == 0 ? (u128)0 : row == 1 ? b1 : row == 2 ? b2 : b3);
}
// The row's token from n <= TOP_NL1 distinct candidates (src, zeros past them to TOP_NL1), among which are its best
// min(top_k, 64) and, with a threshold given, every one down to its crossing: ranked by counting, then one per lane in
// rank order weighed, cut by top-k, min-p and top-p, and drawn from in index order.  All threads; ends with a barrier.
template <bool VER>
__device__ __forceinline__ int finish_ranked(const TopRow& A, int n, const uint64_t* src, const float2* ts, TopBuf& L) {
  const int tid = threadIdx.x, lane = lane_id(), wave = __builtin_amdgcn_readfirstlane(wave_id());
  const int K = A.K;
  {  // ranks by counting: thread (i, p) counts the larger ones of entries [32 p, 32 p + 32)
    const int i = tid & (TOP_NL1 - 1), p = tid / TOP_NL1;
    const uint64_t ci = src[i];
    uint32_t r = 0;
    if (TOP_NL1 / 4 * p < n) {  // uniform in the wave
#pragma unroll
      for (int j = 0; j < TOP_NL1 / 4; j++) r += src[TOP_NL1 / 4 * p + j] > ci ? 1u : 0u;
    }
    L.rk[p][i] = r;
    bar();
    if (tid < n) {  // n <= TOP_NL1: p = 0
      const uint32_t rank = L.rk[0][tid] + L.rk[1][tid] + L.rk[2][tid] + L.rk[3][tid];
      if (rank < (uint32_t)K) L.srt[rank] = ci;
    }
    bar();
  }
  // every wave: the row's candidates (top-k applied), one per lane in rank order, weighed and cut by min-p and top-p
  const int m0 = min(n, K);
  const uint64_t cc = lane < m0 ? L.srt[lane] : 0ull;
  const uint32_t idx = comp_idx(cc);
  const float Ks = kscale(A.temperature);
  const float t = tval(okey_val(comp_key(cc)), Ks);
  const float tmax = readlane<float>(t, 0);
  const int row_top = (tfloor(tmax) >> 10) * FB + (FB - 1);
  const W ww = weigh(lane < m0 ? t : 0.0f, ts);
  const int r = row_top - (tfloor(t) >> 4);
  bool keep = lane < m0 && r < NR;
  if (A.min_p > 0.0f) keep = keep && t >= (float)((double)(tmax / 1024.0f) + A.log2_min_p) * 1024.0f;
  uint64_t w = keep ? rw1(ww.mu, r) : 0ull;
  const u128 incl = wave_scan_weights(w);
  u128 S2 = readlane<u128>(incl, 63);
  int m = __popcll(__ballot(w != 0));  // weighted candidates: lanes 0 .. m - 1
  {
    u128 thr = ld128(A.thr_lo, A.thr_hi);
    if (thr == 0 && A.top_p < 1.0f) thr = mul_shr_ceil(S2, (uint64_t)floor((double)A.top_p * 4294967296.0), 32);
    if (thr > 0) {
      m = min(first_lane(w != 0 && thr <= incl), 63) + 1;  // thr <= S2: one lane crosses
      S2 = readlane<u128>(incl, m - 1);
      w = lane < m ? w : 0ull;
    }
  }
  // the draw in index order: wave p sums, for each candidate, the kept weights of candidates [8 p, 8 p + 8) with a lower
  // index (below 2^62), wave 0 adds the eight sums up
  if (wave * 8 < m) {  // uniform in the wave
    uint64_t b = 0;
#pragma unroll
    for (int j = 0; j < 8; j++) {
      const uint32_t ij = readlane<uint32_t>(idx, wave * 8 + j);
      const uint64_t wj = readlane<uint64_t>(w, wave * 8 + j);
      b += ij < idx ? wj : 0ull;
    }
    L.part[wave][lane] = b;
  }
  bar();
  if (wave == 0) {
    const u128 tt = mul_shr_floor(S2, A.u_draw, 24);
    u128 below = 0;
#pragma unroll
    for (int p = 0; p < NWV2; p++)
      if (p * 8 < m) below += L.part[p][lane];
    const int l = first_lane(w != 0 && below <= tt && tt < below + w);
    const int tok = l < 64 ? (int)readlane<uint32_t>(idx, l) : (n == 0 ? 0 : -1);  // no candidate: token 0, as a greedy row's
    if (A.out_probs && lane < m) {  // k_scan has written zeros
      const double S2d = (double)(uint64_t)(S2 >> 64) * 18446744073709551616.0 + (double)(uint64_t)S2;
      A.out_probs[(size_t)A.row * A.V + idx] = (float)((double)w / S2d);
    }
    if (VER && lane < m) {
      KeptSet& ks = kept_sets(A.rres, A.B)[A.row];
      ks.w[lane] = w;
      ks.idx[lane] = idx;
    }
    const int rl = readlane<int>(r, max(m - 1, 0));
    const uint64_t cl = readlane<uint64_t>(cc, max(m - 1, 0));
    if (lane == 0) {
      A.out_tokens[A.row] = tok;
      if (A.out_info) A.out_info[A.row] = n == 0 ? 2 : tok < 0 ? -1 : 0;
      if (VER) {
        RowRes o = {};
        o.kind = n == 0 ? RR_EMPTY : tok < 0 ? RR_FAIL : RR_SAMPLED;
        o.tok = tok;
        if (n != 0) {
          o.s_lo = (unsigned long long)S2;
          o.s_hi = (unsigned long long)(S2 >> 64);
          o.cC = cl;  // the kept set: the rank prefix down to its last member
          o.cR = rl;
          o.row_top = row_top;
          o.K = Ks;
          o.n_kept = m;
        }
        A.rres[A.row] = o;
      }
      L.tok = tok;
    }
  }
  bar();
  return __builtin_amdgcn_readfirstlane(L.tok);
}
template <bool VER>
__device__ __forceinline__ int resolve_top_body(const TopRow& A, const char* hdrs, const float2* ts, TopBuf& L) {
  const int tid = threadIdx.x, lane = lane_id(), wave = __builtin_amdgcn_readfirstlane(wave_id());
  const int K = A.K, G = A.G;
  // 2^sh threads per block: every thread holds a few entries, spread over as many threads as there are
  const int sh = G <= 8 ? 6 : G <= 16 ? 5 : G <= 32 ? 4 : 3, g = tid >> sh, j0 = tid & ((1 << sh) - 1);
  uint64_t c[TOP_EPL], mx = 0;
  {
    const char* h = hdrs + (size_t)min(g, G - 1) * HDR_BYTES;
    const int n = g < G ? min(((const Rec*)h)->n_list, TOPN) : 0;
#pragma unroll
    for (int k = 0; k < TOP_EPL; k++) {
      c[k] = 0;
      if ((k << sh) >= TOPN) continue;  // uniform
      const int i = j0 + (k << sh);
      if (i < n) c[k] = comp(((const uint32_t*)(h + TOP_KEYS))[i], (uint32_t)(g * BLK + ((const uint16_t*)(h + TOP_IDS))[i]));
      mx = c[k] > mx ? c[k] : mx;
    }
  }
  L.mxs[tid] = mx;
  if (tid < TOP_NL1) L.lst[tid] = 0ull;
  if (tid == 0) L.cnt = 0;
  bar();
  if (wave == 0) {
    uint64_t m[NT2 / 64];
    int cn;
#pragma unroll
    for (int j = 0; j < NT2 / 64; j++) m[j] = L.mxs[j * 64 + lane];
    const uint64_t b = top_bound<NT2 / 64, uint64_t>([&](int j) { return m[j]; }, 1ull, K, G <= 32 ? K + TOP_SLACK : min(K + TOP_SLACK, 64), &cn);
    if (lane == 0) L.bound = b;
  }
  bar();
  {
    // at most 64 threads hold entries at or above it, or 72 of at most five each (16 threads or more per block)
    static_assert((TOPK_MAX + TOP_SLACK) * ((TOPN + 15) / 16) <= 64 * TOP_EPL, "entries at or above the bound");
    const uint64_t b = L.bound;
#pragma unroll
    for (int k = 0; k < TOP_EPL; k++)
      if (c[k] >= b) L.lst[atomicAdd(&L.cnt, 1)] = c[k];
  }
  bar();
  int n = __builtin_amdgcn_readfirstlane(L.cnt);
  const uint64_t* src = L.lst;
  if (n > TOP_NL1) {  // uniform: the best candidates crowd into few threads' entries
    if (wave == 0) {
      auto m = [&](int j) { return j * 64 + lane < n ? L.lst[j * 64 + lane] : 0ull; };
      int cn, base = 0;
      const uint64_t b = top_bound<TOP_EPL, uint64_t>(m, 1ull, K, TOP_NL1, &cn);
      for (int j = 0; j < TOP_EPL; j++) {
        const uint64_t e = m(j);
        const unsigned long long bal = __ballot(e >= b);
        if (e >= b) L.mxs[base + __popcll(bal & ((1ull << lane) - 1ull))] = e;
        base += __popcll(bal);
      }
      for (int i = base + lane; i < TOP_NL1; i += 64) L.mxs[i] = 0ull;
      if (lane == 0) L.cnt2 = base;
    }
    bar();
    n = __builtin_amdgcn_readfirstlane(L.cnt2);
    src = L.mxs;
  }
  return finish_ranked<VER>(A, n, src, ts, L);
}
// The calls pass the row's arguments through LDS (an out-of-line function's arguments would arrive in vector registers)
__device__ __forceinline__ TopRow top_row(QWS_L const TopRow* a) {
  TopRow A;
  A.row = __builtin_amdgcn_readfirstlane(a->row);
  A.V = __builtin_amdgcn_readfirstlane(a->V);
  A.G = __builtin_amdgcn_readfirstlane(a->G);
  A.K = __builtin_amdgcn_readfirstlane(a->K);
  A.B = __builtin_amdgcn_readfirstlane(a->B);
  A.u_draw = a->u_draw;
  A.temperature = a->temperature;
  A.top_p = a->top_p;
  A.min_p = a->min_p;
  A.log2_min_p = a->log2_min_p;
  A.thr_lo = a->thr_lo;
  A.thr_hi = a->thr_hi;
  A.out_tokens = a->out_tokens;
  A.out_info = a->out_info;
  A.out_probs = a->out_probs;
  A.rres = a->rres;
  return A;
}
template <bool VER>
__device__ __noinline__ int resolve_top(QWS_L const TopRow* a, QWS_L const char* hdrs, QWS_L const float2* ts, QWS_L char* buf) {
  return resolve_top_body<VER>(top_row(a), (const char*)hdrs, (const float2*)ts, *(TopBuf*)(char*)buf);
}
// finish_ranked over the n candidates in the buffer's list
template <bool VER>
__device__ __noinline__ int finish_small(QWS_L const TopRow* a, int n, QWS_L const float2* ts, QWS_L char* buf) {
  TopBuf& L = *(TopBuf*)(char*)buf;
  return finish_ranked<VER>(top_row(a), __builtin_amdgcn_readfirstlane(n), L.lst, (const float2*)ts, L);
}

// ---------------------------------------------------------------------------------------------- out-of-line parts of a row
// (each uniform arguments, all threads; results in the row state after a barrier)
// The min-p cut inside row bin rc (its power staged): the cut's comp -> st.su[4], the bin's kept candidates -> st.su[5]
template <int DT>
__device__ __noinline__ void minp_cut(QWS_L ResolveLds* s, char* ws_, int row_, int rc_, float tcut) {
  ResolveLds& S = *(ResolveLds*)s;
  char* const ws = uniform_ptr(ws_);
  const int row = __builtin_amdgcn_readfirstlane(row_), rc = __builtin_amdgcn_readfirstlane(rc_);
  RS& st = S.st;
  const float K = st.K;
  gather<DT>(S, ws, row, rc);
  unsigned long long v = 0;  // kept: t >= tcut, a prefix of the bin in comp order
  for_bin<DT>(S, ws, row, [&](uint64_t c, uint32_t) { v += tval(okey_val(comp_key(c)), K) >= tcut ? 1ull : 0ull; });
  block_add_u64(st, v);
  const unsigned long long nk = st.su[7];
  uint64_t cC;
  float xc;
  if (nk == 0) {
    cC = ~0ull;
  } else if (nk == (unsigned long long)st.gn) {
    cC = 0;
  } else if (first_x_t(tcut, K, &xc)) {  // the kept prefix from the threshold's value: no selection
    cC = (uint64_t)okey(xc) << 32;
  } else {
    select_in_bin<DT>(S, ws, row, false, nk);
    cC = st.su[4];
  }
  bar();
  if (threadIdx.x == 0) {
    st.su[4] = cC;
    st.su[5] = nk;
  }
  bar();
}
// The cut by count (by_mass = 0) or mantissa sum inside row bin rb: its comp -> st.su[4], its inclusive prefix -> st.su[5]
template <int DT>
__device__ __noinline__ void rank_cut(QWS_L ResolveLds* s, char* ws_, int row_, int rb_, int by_mass_, uint64_t target_) {
  ResolveLds& S = *(ResolveLds*)s;
  char* const ws = uniform_ptr(ws_);
  const int row = __builtin_amdgcn_readfirstlane(row_), rb = __builtin_amdgcn_readfirstlane(rb_);
  const bool by_mass = __builtin_amdgcn_readfirstlane(by_mass_) != 0;
  const uint64_t target = readlane<uint64_t>(target_, 0);
  RS& st = S.st;
  uint64_t c = ~0ull, pref = 0;
  if (!select_listed<DT>(S, ws, row, rb, by_mass, target, &c, &pref)) {
    gather<DT>(S, ws, row, rb);
    select_in_bin<DT>(S, ws, row, by_mass, target);
    c = st.su[4];
    pref = st.su[5];
  }
  bar();
  if (threadIdx.x == 0) {
    st.su[4] = c;
    st.su[5] = pref;
  }
  bar();
}
// The mantissa sum of the gathered bin's candidates with comp >= cmin -> st.su[7]
template <int DT>
__device__ __noinline__ void bin_mass(QWS_L ResolveLds* s, char* ws, int row, uint64_t cmin) {
  ResolveLds& S = *(ResolveLds*)s;
  unsigned long long v = 0;
  for_bin<DT>(S, uniform_ptr(ws), __builtin_amdgcn_readfirstlane(row), [&](uint64_t c, uint32_t mu) { v += c >= cmin ? (unsigned long long)mu : 0ull; });
  block_add_u64(S.st, v);
}
// Adds the gathered bin's kept candidates (comp >= cC) to the blocks' kept masses
template <int DT>
__device__ __noinline__ void kept_unstaged(QWS_L ResolveLds* s, char* ws, int row, uint64_t cC, int sh_) {
  ResolveLds& S = *(ResolveLds*)s;
  const int sh = __builtin_amdgcn_readfirstlane(sh_);
  for_bin<DT>(S, uniform_ptr(ws), __builtin_amdgcn_readfirstlane(row), [&](uint64_t c, uint32_t mu) {
    if (c >= cC) {
      const int g = (int)(comp_idx(c) / BLK);
      atomic_add_u128(&S.st.Klo[g], &S.st.Khi[g], (u128)mu << sh);
    }
  });
}
// Dense probabilities of the kept set, by rescans of every block (k_scan has written zeros)
template <int DT>
__device__ __noinline__ void dense_probs(QWS_L ResolveLds* s, char* ws_, int row_, unsigned long long s2lo, unsigned long long s2hi, int cR_, uint64_t cC_) {
  using BL = Blk<DT, NT2>;
  ResolveLds& S = *(ResolveLds*)s;
  char* const ws = uniform_ptr(ws_);
  const int row = __builtin_amdgcn_readfirstlane(row_), cR = __builtin_amdgcn_readfirstlane(cR_);
  const uint64_t cC = readlane<uint64_t>(cC_, 0);
  const double S2d = (double)s2hi * 18446744073709551616.0 + (double)s2lo;
  const int G = __builtin_amdgcn_readfirstlane(S.st.G), V = S.B.V, row_top = S.st.row_top;
  const float K = S.st.K;
  float* out = S.B.out_probs + (size_t)row * V;
  for (int g = 0; g < G; g++) {
    if (__builtin_amdgcn_readfirstlane(S.bi[g].dn) < 0) continue;
    stage_block<DT>(s, ws, row, g);
    const float* xs = (const float*)S.big;
    const int t0 = (int)threadIdx.x * BL::EPT;
#pragma unroll
    for (int k = 0; k < BL::EPT; k++) {
      const float v = xs[big_at(t0) + k];
      if (v == -INFINITY) continue;
      const W w = weigh(tval(v, K), S.ts);
      const int r = row_top - w.bin();
      const uint32_t idx = (uint32_t)(g * BLK + t0 + k);
      if (r < NR && (r < cR || (r == cR && comp(okey(v), idx) >= cC))) out[idx] = (float)((double)rw1(w.mu, r) / S2d);
    }
    bar();
  }
}

// VER: the rows of a verify call (rres != nullptr)
template <int DT, bool VER>
__global__ void __launch_bounds__(NT2) k_resolve(qws_batch B, int G, char* ws, RowRes* rres) {
  __shared__ __attribute__((aligned(16))) ResolveLds S;
  QWS_L ResolveLds* const SL = (QWS_L ResolveLds*)&S;
  const RL L = rl_of(S);
  auto& s_fb = S.fb;
  auto& s_emu = S.emu;
  auto& s_bi = S.bi;
  RS& st = S.st;
  // Workgroup i runs on XCD i % 8 (round-robin dispatch): it takes a row whose blocks k_scan ran on that XCD (rows
  // [x * RB, (x + 1) * RB) there, RB = ceil(B / 8)), so the row's records are read back through the L2 that wrote them.
  const int RB = (B.B + NXCD - 1) / NXCD;
  const int row = (int)(blockIdx.x % NXCD) * RB + (int)(blockIdx.x / NXCD), tid = threadIdx.x;
  if (row >= B.B) return;  // whole workgroups, before any barrier
  // ---- round 1: every block header and the exp2 table into LDS (the headers in the fine-bin region).  All loads,
  // the row's parameters included, are issued before any is waited for.
  constexpr int HW = (int)(HDR_BYTES / 16), HPT = MAXG * HW / NT2;  // header words per thread
  static_assert(MAXG * HW % NT2 == 0 && 512 <= NT2, "round 1 layout");
  vu4 hv[HPT];
#pragma unroll
  for (int k = 0; k < HPT; k++) {
    const int i = tid + k * NT2;
    if (i < G * HW) hv[k] = gmem((const vu4*)rec_of(ws, G, row, i / HW))[i % HW];
  }
  vu4 tv;
  if (tid < 512) tv = gmem((const vu4*)EXP2_TS)[tid];
  const qws_row R = B.rows[row];
  if (tid == 0) {
    S.B = B;
    S.R = R;
  }
  const qws_batch& BB = S.B;
  const qws_row& RR = S.R;
  const uint32_t u_draw = draw_u24(R.seed, R.position, R.stream, R.row_key, R.draw_word);  // the draw's Philox word
  if (tid < 512) ((vu4*)S.ts)[tid] = tv;
#pragma unroll
  for (int k = 0; k < HPT; k++) {
    const int i = tid + k * NT2;
    if (i < G * HW) ((vu4*)s_fb)[i] = hv[k];
  }
  if (tid < NEXP) {
    st.Rc[tid] = 0u;
    st.Rm[tid] = 0ull;
  }
  for (int i = tid; i < NBK; i += NT2) {
    st.fbc[i] = 0u;
    st.fbs[i] = 0ull;
  }
  if (tid == 0) {
    st.G = G;
    st.fpow = -1;
    st.gbin = -1;
    st.rescans = 0;
    st.fxn = 0;
  }
  bar();
  __shared__ TopRow s_top;
  if (listed_top(R)) {  // uniform
    if (tid == 0) s_top = TopRow{row, B.V, G, R.top_k, B.B, u_draw, R.temperature, R.top_p, R.min_p, R.log2_min_p, 0, 0, B.out_tokens, B.out_info, B.out_probs, rres};
    bar();
    const int tk = resolve_top<VER>((QWS_L const TopRow*)&s_top, (QWS_L const char*)s_fb, (QWS_L const float2*)S.ts, (QWS_L char*)S.big);
    if (!VER && B.advance) advance_row(B, R, row, tk, &S.nt, -1, 0, 0u);
    return;
  }
  auto hdr = [&](int g) -> const Rec& { return *(const Rec*)((const char*)s_fb + (size_t)g * HDR_BYTES); };
  if (tid < 64) {  // the row's best: one wave max over the blocks (G <= 64: lane g reads block g)
    uint64_t v = 0;
    if (tid < G) {
      const Rec& H = hdr(tid);
      BI b;
      b.max_key = H.max_key;
      b.c = H.c;
      b.nbw = H.nbw;
      b.n_patch = (H.flags & RF_CAND) ? H.n_patch : -1;
      b.dn = -1;
      b.gcnt = b.goff = b.gsrc = b.gofs = 0;
      b.w0 = H.w0;
      b.w1 = H.w1;
      b.n_list = H.n_list;
      b.wcnt = 0;
      s_bi[tid] = b;
      if (H.flags & RF_CAND) v = comp(H.max_key, H.max_idx);
    }
    const uint64_t m = wave_max_u64(v);
    if (tid == 0) st.best = m;
  }
  bar();
  const uint64_t best = st.best;
  const float K = kscale(R.temperature);
  if (best == 0 || !(R.temperature > 0.0f) || !(K < INFINITY)) {  // no candidate, or a greedy row
    if (tid == 0) {
      B.out_tokens[row] = best == 0 ? 0 : (int)comp_idx(best);
      if (B.out_probs && best != 0) B.out_probs[(size_t)row * B.V + comp_idx(best)] = 1.0f;  // the point mass
      if (B.out_info) B.out_info[row] = 2;
      if (VER) {
        RowRes o = {};
        o.kind = best == 0 ? RR_EMPTY : RR_GREEDY;
        o.tok = B.out_tokens[row];
        rres[row] = o;
      }
    }
    // a row without a candidate emits token 0 (its greedy token) and takes the step with it, as qws_finish_rows does
    if (!VER && B.advance) advance_row(B, R, row, best == 0 ? 0 : (int)comp_idx(best), &S.nt, -1, 0, 0u);
    return;
  }
  const float tmax = tval(okey_val(comp_key(best)), K);
  const int N = tfloor(tmax) >> 10;
  const int row_top = N * FB + (FB - 1);
  if (tid == 0) {
    st.K = K;
    st.N = N;
    st.row_top = row_top;
  }
  // ---- the row's per-power sums: block power e is row power e + (N - c) (consecutive threads read consecutive powers
  // of one staged header: no bank conflicts; the sums by LDS atomics)
  for (int i = tid; i < G * NEXP; i += NT2) {
    const int g = i / NEXP, e = i - g * NEXP;
    const Rec& H = hdr(g);
    const bool samp = (H.flags & RF_SAMP) && N - H.c <= D_EXP;
    const unsigned long long mu = samp ? H.emu[e] : 0ull;
    s_emu[i] = mu;
    if (e == 0) s_bi[g].dn = samp ? N - H.c : -1;
    const int er = e + N - H.c;
    if (samp && er <= D_EXP && H.ecnt[e]) {
      atomicAdd(&st.Rc[er], H.ecnt[e]);
      atomicAdd(&st.Rm[er], mu);
      atomicAdd(&s_bi[g].wcnt, (int)H.ecnt[e]);
    }
  }
  bar();
  // ---- the cuts: min-p, then top-k, then top-p; kept = row bin r < cR, or r == cR and comp >= cC (cR = NR: none)
  int cR = NR;
  uint64_t cC = 0;
  u128 mb = 0;                    // mass (row units) of the bins above the cut
  unsigned long long kept_n = 0;  // candidates kept so far
  before_bin(L, NR, &mb, &kept_n);
  // candidates below the row's window (weight 0) still count for top-k: the window's count is a lower bound, and a
  // K at or beyond it keeps every weighted candidate
  // ---- at most 64 candidates down to row bin rb (NR: all that weigh something; else rb's power is the staged one), all in
  // their blocks' lists (each block's bins from its best down to rb's listed): they are taken from the lists and the row
  // is finished over them, with no selection inside a bin, no other power staged, no kept masses per block and no block
  // of the draw.  thr: the top-p threshold when the row's mass is known (0: min-p, then top-p over the candidates'
  // own mass).  Test flags that ask for rescans or staged draws keep the general path.
  auto small = [&](int rb, u128 thr) -> bool {
    if (R.test_flags & (QWS_TF_RESCAN | QWS_TF_STAGED_DRAW | QWS_TF_SPLIT_SELECT)) return false;
    const int lane = lane_id();
    int cnt = 0;
    bool ok = true;
    if (lane < G && s_bi[lane].dn >= 0) {
      const BI& b = s_bi[lane];
      if (rb >= NR) {
        cnt = b.wcnt;
        ok = cnt == 0 || (b.w0 == 0 && cnt <= b.n_list);
      } else {
        const int cb = rb - FB * b.dn;  // the bin among the block's own
        const int r0 = b.c * FB + (FB - 1) - (tfloor(tval(okey_val(b.max_key), K)) >> 4);  // its best's
        if (cb >= r0) {
          if (cb < b.nbw) {
            const unsigned long long wd = s_fb[lane * FB + (rb & 63)];
            ok = b.w0 == 0 && bw_listed(wd);
            cnt = (int)(bw_off(wd) + bw_cnt(wd));
          } else {  // past its last occupied bin (with a top-k cut the bins may end earlier)
            ok = b.w0 == 0 && b.w1 >= b.nbw - 1 && R.top_k <= 0;
            cnt = b.n_list;
          }
        }
      }
    }
    const int inc = wave_scan_incl<int>(cnt), tot = readlane<int>(inc, 63), exc = inc - cnt;
    if (__ballot(!ok) != 0ull || tot > 64 || tot == 0) return false;  // uniform: the same words in every wave
    TopBuf& T = *(TopBuf*)S.big;
    if (wave_id() == 0) {
      // list entry `lane` of the concatenation: its block by a binary search over the inclusive counts
      int g = 0;
      for (int sft = 32; sft > 0; sft >>= 1) g += __shfl(inc, g + sft - 1) <= lane ? sft : 0;
      const int e0 = __shfl(exc, min(g, 63));
      T.lst[lane] = lane < tot ? els_of(ws, G, row, g)[lane - e0] : 0ull;
      if (lane == 0)
        s_top = TopRow{row, B.V, G, 64, B.B, u_draw, R.temperature, R.top_p, thr == 0 ? R.min_p : 0.0f, R.log2_min_p, (unsigned long long)thr,
                       (unsigned long long)(thr >> 64), B.out_tokens, B.out_info, B.out_probs, rres};
    } else if (wave_id() == 1) {
      T.lst[64 + lane] = 0ull;
    }
    bar();
    const int tk = finish_small<VER>((QWS_L const TopRow*)&s_top, tot, (QWS_L const float2*)S.ts, (QWS_L char*)S.big);
    if (tid == 0 && B.out_info && tk >= 0 && st.rescans) B.out_info[row] = 1;
    if (!VER && B.advance) advance_row(B, R, row, tk, &S.nt, -1, 0, 0u);
    return true;
  };
  if (R.min_p > 0.0f) {
    const float tcut = (float)((double)(tmax / 1024.0f) + R.log2_min_p) * 1024.0f;
    const int rc = row_top - (tfloor(tcut) >> 4);
    bool need = rc < NR;
    if (need) {
      stage_power(L, ws, row, rc >> 6);
      if (small(rc, 0)) return;  // uniform
    }
    if (need && R.top_k > 0) {  // uniform: top_k candidates in the bins above the min-p cut's: the top-k cut decides
      const int lane = lane_id();
      const uint32_t above = wave_sum<uint32_t>((lane < (rc >> 6) ? st.Rc[lane] : 0u) + (lane < (rc & 63) ? st.fcnt[lane] : 0u));
      need = above < (uint32_t)R.top_k;
    }
    if (need) {
      minp_cut<DT>(SL, ws, row, rc, tcut);
      cR = rc;
      cC = st.su[4];
      const unsigned long long nk = st.su[5];
      before_bin(L, rc, &mb, &kept_n);
      kept_n += nk;
    }
  }
  // With top-k beside min-p a block writes its bins only down to the shallower of its own min-p cut and its own K-th
  // candidate, so the count above the row's min-p cut is exact when it is below K and at least K otherwise: the cut
  // runs when K <= kept_n (at kept_n == K it keeps the same set)
  if (R.top_k > 0 && (unsigned long long)R.top_k <= kept_n) {
    int pk;
    unsigned long long before_p;
    pow_cross_cnt(L, (unsigned long long)R.top_k, &pk, &before_p);
    stage_power(L, ws, row, pk);
    u128 before_f;
    const int bk = pk * FB + fine_cross(L, false, (u128)before_p, (u128)(unsigned long long)R.top_k, &before_f);
    const unsigned long long need = (unsigned long long)R.top_k - (unsigned long long)before_f;
    cR = bk;
    if (st.fcnt[bk & 63] == need) {  // the whole bin is kept (cC = 0): no gather
      cC = 0;
    } else {
      rank_cut<DT>(SL, ws, row, bk, 0, need);
      cC = st.su[4];
    }
  }
  if (cR == NR && kept_n <= 64 && small(NR, 0)) return;  // uniform: no cut so far (a few strongly biased tokens, say)
  u128 S2;
  int tok = -1;
  int a_g = -1, a_n = 0;  // advance: the drawn block and its state entries, loaded before the draw
  uint32_t a_e = 0u;
  {
    bool kept_done = false;  // the kept mass of every block computed with the cut (topp_cut_fast)
    // cC = 0: every element of bin cR is kept, and the bin's words give its mass (the staged power is cR's)
    u128 Sm = mb;  // the row's mass (after min-p and top-k)
    if (cR < NR) {
      unsigned long long cnt_unused;
      before_bin(L, cR, &mb, &cnt_unused);
      if (cC != 0) bin_mass<DT>(SL, ws, row, cC);
      Sm = mb + shl128(cC == 0 ? st.fmu[cR & 63] : st.su[7], D_EXP - (cR >> 6));
    }
    if (R.top_p < 1.0f) {
      const uint64_t TP = (uint64_t)floor((double)R.top_p * 4294967296.0);
      const u128 thr = mul_shr_ceil(Sm, TP, 32);
      if (thr > 0) {
        int pp;
        u128 before_p, before_f;
        pow_cross_mass(L, thr, &pp, &before_p);
        stage_power(L, ws, row, pp);
        const int bp = pp * FB + fine_cross(L, true, before_p, thr, &before_f);
        if (small(bp, thr)) return;  // uniform
        const int sh = D_EXP - pp;
        cR = bp;
        mb = before_f;
        if (st.fcnt[bp & 63] == 1) {  // the crossing bin holds one element: the cut, the whole bin kept (no gather)
          cC = 0;
          Sm = mb + ((u128)st.fmu[bp & 63] << sh);
        } else {
          // the crossing in mantissa units of the bin's power: sum of mu * 2^sh >= thr - before  <=>  sum of mu >= ceil(...)
          const u128 need = thr - before_f;
          const uint64_t tmu = (uint64_t)((need + (((u128)1 << sh) - 1)) >> sh);
          uint64_t pref;  // the selection's inclusive mantissa sum at the cut
          if (topp_cut_fast(L, RR, ws, row, bp, tmu, &cC, &pref)) {
            kept_done = true;
          } else {
            rank_cut<DT>(SL, ws, row, bp, 1, tmu);
            cC = st.su[4];
            pref = st.su[5];
          }
          Sm = mb + ((u128)pref << sh);
        }
      }
    }
    S2 = Sm;
    // a verify row ends at S2: the verify kernels draw from p for the one row of a sequence that needs it
    if constexpr (!VER) {
      // ---- kept mass per block: its powers above the cut's, its fine bins above the cut's bin and its kept elements there
      // (sixteen threads per block; topp_cut_fast has computed them already)
      for (int g0 = 0; g0 < (kept_done ? 0 : G); g0 += NT2 / 16) {  // uniform
        const int g = g0 + (tid >> 4), j = tid & 15;
        u128 k = 0;
        if (g < G && s_bi[g].dn >= 0) {
          const BI& b = s_bi[g];
          const int pc = cR < NR ? (cR >> 6) : NEXP;
          for (int er = b.dn + j; er < pc; er += 16) k += shl128(s_emu[g * NEXP + er - b.dn], D_EXP - er);
          if (cR < NR) {
            const int sh = D_EXP - pc;
            for (int f = j; f < (cR & 63) + (cC == 0 ? 1 : 0); f += 16) k += shl128(bw_mu(s_fb[g * FB + f]), sh);
            if (cC != 0 && st.gstaged) {  // a partial cut: the gathered bin is cR's
              for (int i = b.gofs + j; i < b.gofs + (b.gsrc ? b.gcnt : 0); i += 16)
                if (L.ec[i] >= cC) k += (u128)L.em[i] << sh;
            }
          }
        }
        k = row16_scan_incl<u128>(k);  // a block's sixteen threads are one DPP row: its last lane holds the total
        if (g < G && j == 15) {
          st.Klo[g] = (unsigned long long)k;
          st.Khi[g] = (unsigned long long)(k >> 64);
        }
      }
      if (!kept_done) bar();
      // a bin too large for LDS: its kept elements by block from the sources
      if (!kept_done && cR < NR && cC != 0 && !st.gstaged) kept_unstaged<DT>(SL, ws, row, cC, D_EXP - (cR >> 6));
      // ---- the draw: the block by its kept mass (index order), then the token inside it
      const u128 tt = mul_shr_floor(S2, u_draw, 24);
      int gs;   // every wave picks it from the final kept masses (no barrier)
      u128 tl;  // the target inside that block
      {
        const int lane = lane_id();
        const u128 k = lane < G ? ld128(st.Klo[lane], st.Khi[lane]) : (u128)0;
        const u128 incl = wave_scan_incl_u128(k);
        const int l = first_lane(k != 0 && tt < incl);
        gs = l < 64 ? l : -1;
        tl = l < 64 ? tt - readlane<u128>(incl - k, l) : (u128)0;
      }
      // advance: the drawn block's state entries loaded now, so that noting the token waits for nothing after the draw
      const int aslot = (!VER && B.advance) ? row_state(B, R) : -1;
      if (aslot >= 0 && gs >= 0) {  // uniform; entry tid lies inside the block's BLK entry words
        a_g = gs;
        a_n = (int)gmem(state_counts(B.state_mem, B.V, aslot))[gs];  // global loads: no LDS wait of the draw waits for them
        a_e = gmem(state_entries(B.state_mem, B.V, aslot, gs))[tid];
      }
      // the drawn block's kept set whole in its list (its bins listed from the top without a gap down to the cut's, at most
      // a wave of elements there): drawn from those by wave 0; else the block is staged and weighed
      int nlist = 65;
      if (gs >= 0 && s_bi[gs].w0 == 0 && !(R.test_flags & QWS_TF_STAGED_DRAW)) {  // uniform
        const BI& b = s_bi[gs];
        if (cR == NR) {
          // no cut: the block's candidates inside the weight window, a top-down prefix of its bins as the (gap-free) list
          // is, lie whole in the list iff they are no more than the list holds
          if (b.wcnt <= b.n_list) nlist = b.n_list;
        } else if (st.fpow == (cR >> 6)) {  // the cut's power is the staged one
          const int cb = cR - FB * b.dn;    // the cut's bin among the block's own
          if (cb >= 0 && cb <= b.w1) {  // bins 0 .. cb all listed
            const unsigned long long wd = s_fb[gs * FB + (cR & 63)];
            if (bw_listed(wd)) nlist = (int)(bw_off(wd) + bw_cnt(wd));
          }
        }
      }
      if (nlist <= 64) {
        if (wave_id() == 0) tok = draw_listed(L, ws, row, gs, nlist, cR, cC, tl);
      } else if (gs >= 0) {
        tok = draw_in_block<DT>(L, BB, RR, ws, row, gs, cR, cC, tl);
      }
    }
  }
  if (B.out_probs) dense_probs<DT>(SL, ws, row, (unsigned long long)S2, (unsigned long long)(S2 >> 64), cR, cC);  // uniform
  if (tid == 0) {
    B.out_tokens[row] = tok;
    if (B.out_info) B.out_info[row] = tok < 0 && !VER ? -1 : (st.rescans ? 1 : 0);
    if (VER) {
      RowRes o;
      o.s_lo = (unsigned long long)S2;
      o.s_hi = (unsigned long long)(S2 >> 64);
      o.cC = cC;
      o.cR = cR;
      o.row_top = row_top;
      o.K = K;
      o.kind = RR_SAMPLED;  // tok = -1: not drawn here
      o.tok = tok;
      o.n_kept = 0;
      rres[row] = o;
    }
  }
  if (!VER && B.advance) {  // uniform
    __shared__ int s_tok;
    if (tid == 0) s_tok = tok;  // thread 0 holds the row's token (a listed draw leaves it in wave 0 only)
    bar();
    advance_row(B, R, row, s_tok, &S.nt, a_g, a_n, a_e);
  }
}

}  // namespace qws
