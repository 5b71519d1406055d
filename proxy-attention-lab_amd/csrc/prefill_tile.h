// Paged causal attention for query tiles (prefill and the prefill rows of the
// fused mixed batch) on gfx950 MFMA.
//
// Reference behaviour: kernels/paged_attention/prefill/paged_attention_prefill.h.metal
// -- a prompt token attends to the cached history and to prompt tokens at or
// before it (:147-234, :251-360), scores scaled by 1/sqrt(HD) after the dot
// product (:178, :302), output rows (token, head) (:379-381).  In the fused
// op every key is read from pages: row r of sequence s sees keys
// [0, min(len[s], q_offset[r])), which is exactly the causal mask when the
// new tokens were written to the pages first.
//
// Design (MI355X):
//  * One workgroup (4 wavefronts, one per SIMD) has a CU to itself and owns a
//    tile of RG * 128 "M-rows": consecutive query tokens of one sequence times
//    the (up to 16) query heads sharing a kv head, so one K/V tile in LDS
//    serves the whole GQA group.  A wavefront holds RG groups of 32 rows and the
//    whole register file of its SIMD, so with RG = 2 an operand read from LDS
//    feeds two MFMAs: with one (two wavefronts of 32 rows per SIMD), the LDS
//    reads, the copies and the per-step work cost as much as the products.
//    RG = 1 keeps the same code for problems of few tiles, whose time is one
//    tile's latency (the choice is in prefill_choose_tiles).
//  * O and the running PV accumulators live in registers above the compiler's
//    reach (PAL_ACC_KERNEL), named by the MFMA instructions directly: as
//    ordinary values they were copied and spilled around every step.
//  * Per 32-key step the K and V tiles reach LDS by direct-to-LDS copies
//    (global_load_lds_dwordx4, no registers), kLeadK and kLeadV steps ahead,
//    into four LDS buffers each, with counted waits and one barrier per step.
//    Page ids come from an LDS copy of the tile's page-table slice.  Steps of
//    dense prompt keys are copied the same way from the prompt rows (V rows
//    untransposed, read back with transposing LDS reads); fp8 pages (window
//    mode) as fp8 bytes, converted in the operand reads.  Steps across the
//    history / prompt boundary or with invalid page ids take a synchronous
//    register path.
//  * Each wavefront computes S^T = K * Q^T with v_mfma_f32_32x32x16 (A = K
//    from LDS, B = Q^T held in registers) and O^T += V^T * P^T with the same
//    instruction.  In the transposed products a lane owns one M-row, so the
//    softmax max needs one cross-half exchange (v_permlane32_swap) and the
//    probabilities go into the PV MFMA without leaving the lane.  The sum of
//    the rounded probabilities comes from two MFMAs with ones per step (v_dot2
//    holds the matrix pipe for 16 cycles each) or from vector adds.  K is stored in the QK operand's row
//    order and V rows are swizzled, so every operand read is one conflict-free
//    16-byte LDS access.
//  * Steps are software-pipelined inside a wavefront: the QK MFMAs of step
//    st+1 are issued among the exponentials of step st, the row max of step
//    st+1 and the step's copies among the PV MFMAs.  Over ragged chunks a
//    step of 128 dims takes 2,090 cycles of a wavefront with RG = 2, masked
//    steps, tile set-up and waits included, 1,024 of them MFMA.
//  * Online softmax in log2 units, scale and max folded into one fma per score,
//    with a lazy rescale: the running max is only moved when a score exceeds
//    it by more than 2^8, so O is rescaled rarely.
//  * Causal skipping: the key loop stops at the tile's largest limit, and key
//    steps below every row's limit skip the mask arithmetic.
//  * The output leaves through LDS as whole rows of 16-byte stores.
//  * Measured (bf16, 32 query heads on 8 kv heads, head dim 128), against 32
//    rows per wavefront and two workgroups per CU: 16 sequences of 1,280 rows
//    on 1,024 cached 670 -> 570 us (0.98 PFLOP/s over the keys seen); one prompt
//    of 777 rows 29.6 -> 19.2 us (RG 1).  Under this load the card's clock falls
//    to about 1.9 GHz.
//  * Two ways to name the work, both without a planning pass: the reference
//    prefill's uniform prompt (S sequences x P prompt rows; tiles are pure
//    arithmetic; keys [0, hist[s]) come from pages and keys hist[s] + i from
//    the dense prompt K/V rows s*P + i, as prefill.h.metal:147-234 reads
//    them), or windows of consecutive query rows (the fused op), each run of
//    rows of one sequence in a window being a tile.
//
// This header holds the device code of a tile (prefill_tile) so that both the
// prefill kernel (prefill.hip) and the fused mixed-batch kernel (decode.hip)
// compile it (and prefill_half_tile.h the tiles that share a CU, for the calls
// that those serve faster); a translation unit includes it after defining its debug-check
// flag word (PAL_DEBUG_FLAGS_DEFINE).
#pragma once

#include <type_traits>

#include "pal_device.h"
#include "pid_window.h"

namespace pal {
namespace {


constexpr int kPfWaves = 4;
constexpr int kPfThreads = kPfWaves * kWave;
// M-rows (token, head) of a workgroup whose wavefronts hold rg groups of 32 each
constexpr int m_rows(int rg) { return kPfWaves * 32 * rg; }
static_assert(kPidChunk % kPfThreads == 0, "a page-id chunk is a whole number of loads per thread");
constexpr float kLazyRescale = 8.f;    // log2 headroom before the running max moves
constexpr float kNoMax = 0x1p126f;     // minus the running max of a row that has seen no score above -inf

// A step moves 4*HD items of 16 bytes of K and as many of V.
template <int HD>
struct StepGeo {
  static constexpr int kItems = 4 * HD;
  static constexpr int kLoads = (kItems + kPfThreads - 1) / kPfThreads;  // per thread, per K (or V)
};

// Item <-> (page, offset) maps.  LDS holds each step's items in item order,
// so one direct-to-LDS load per wavefront fills 1 KiB of consecutive slots
// (lane l -> slot base + l).  With TPP 16 the items are page-major (2*HD per
// page), which also makes each load instruction read a single page.
//   K item i: stripe c, slot t of the step holds key kperm(t):  page offset (c*TPP + kperm(t) % TPP) * 8
//   V item i: row d, 8-key group g' = g ^ swz(d) of the row:     page offset d*TPP + 8 g'
// K keys are stored in the QK operand's row order (kperm, an involution
// swapping bits 2 and 3 of the key index), so the operand reads are
// contiguous; the V groups are swizzled by row so that the PV operand reads
// (one 16-byte chunk per lane and row) spread over all banks.
__device__ __forceinline__ int kperm(int m) { return (m & ~12) | ((m & 4) << 1) | ((m & 8) >> 1); }
// fp8 steps: QK operand row m holds key 16 b2 + 8 b4 + 4 b3 + (m & 3) (b_i:
// bit i of m), so that the scores a lane holds after the QK product are
// the 16 consecutive keys 16 h .. 16 h + 15 (h: its lane half) in register
// order, and one 16-byte V item (16 keys of one row) feeds both PV k-steps.
__device__ __forceinline__ int kperm_f8(int m) {
  return ((m & 4) << 2) | ((m & 16) >> 1) | ((m & 8) >> 1) | (m & 3);
}

template <int HD, int TPP>
struct ItemMap {
  static __device__ __forceinline__ int k_page_half(int i) { return TPP == 16 ? i / (2 * HD) : 0; }
  // K item i: stripe c and the key (within the step) it carries
  static __device__ __forceinline__ void k_item(int i, int& c, int& key) {
    if (TPP == 16) {
      const int rem = i % (2 * HD);
      c = rem / 16;
      key = (i / (2 * HD)) * 16 + kperm(rem % 16);
    } else {
      c = i / 32;
      key = kperm(i % 32);
    }
  }
  static __device__ __forceinline__ int k_offset(int i) {  // element offset inside the (page, kv head) block
    int c, key;
    k_item(i, c, key);
    return (c * TPP + key % TPP) * 8;
  }
  // Conflict-free for 8-lane groups over 32 banks and 16-lane groups over 64
  // banks: within any 8 (and any 16) consecutive rows the 16-byte chunk each
  // lane reads lands on a distinct bank group.
  static __device__ __forceinline__ int v_swz(int d) {
    return TPP == 16 ? ((d >> 2) ^ (d >> 3)) & 1 : ((d >> 1) ^ (d >> 3)) & 3;
  }
  // V item i: row d and the group g stored in its slot (key offset in the step)
  static __device__ __forceinline__ void v_item(int i, int& d, int& key) {
    if (TPP == 16) {
      const int rem = i % (2 * HD);
      d = rem / 2;
      key = (i / (2 * HD)) * 16 + 8 * ((rem % 2) ^ v_swz(d));
    } else {
      d = i / 4;
      key = 8 * ((i % 4) ^ v_swz(d));
    }
  }
  // LDS slot of K operand row m (key kperm(m) of the step), stripe c
  static __device__ __forceinline__ int k_slot(int m, int c) {
    return TPP == 16 ? (m / 16) * (2 * HD) + c * 16 + m % 16 : c * 32 + m;
  }
  // LDS slot holding V row d, keys kg .. kg+7 of the step (kg multiple of 8)
  static __device__ __forceinline__ int v_slot(int d, int kg) {
    return TPP == 16 ? (kg / 16) * (2 * HD) + d * 2 + (((kg / 8) % 2) ^ v_swz(d)) : d * 4 + ((kg / 8) ^ v_swz(d));
  }
  // v_slot(d + 32 n, kg) - v_slot(d, kg): v_swz depends on bits 1..3 of d only
  static constexpr int kVRowTile = TPP == 16 ? 64 : 128;
};

// Untransposed V rows (dense prompt steps), read back with transposing reads:
// each 16-lane group reads 32 bytes of each of 4 consecutive keys, the other
// group of its half-wavefront the next 32 bytes.  16-byte chunk c of key k is
// stored at chunk c ^ vd_swz(k), which puts a 16-lane group on distinct banks in
// a 32-bank pass and a half-wavefront on distinct banks in a 64-bank pass (HD
// 96 rows are not swizzled).
template <int HD>
__device__ __forceinline__ int vd_swz(int key) {
  const int r = key & 3;
  return HD % 128 == 0 ? 4 * r + 2 * (r >> 1) : (HD == 64 ? 2 * r : (HD == 32 ? 2 * (r >> 1) : 0));
}
// The PV operand of k-step ks and row tile n from such rows.  Lane 4r + c of a
// 16-lane group points at keys kg + 4t + r, dims d0 + 4c .. +3 (d0 = 32 n + (col
// & 16)); the transposing read hands lane j dim d0 + j = col + 32 n of those 4 keys.
template <int HD>
__device__ __forceinline__ u32x4 read_dense_v(const uint16_t* rows, int ks, int n, int col, int half) {
  const int l16 = static_cast<int>(threadIdx.x) & 15;
  const int key = 16 * ks + 8 * half + (l16 >> 2);
  const int d = 32 * n + (col & 16) + 4 * (l16 & 3);
  const uint16_t* vr = rows + key * HD + (((d >> 3) ^ vd_swz<HD>(key)) << 3) + (d & 7);
  const u32x2 lo = lds_read_tr16(vr);           // keys kg .. kg+3
  const u32x2 hi = lds_read_tr16(vr + 4 * HD);  // keys kg+4 .. kg+7 (vd_swz(key + 4) = vd_swz(key))
  return u32x4{lo[0], lo[1], hi[0], hi[1]};
}

// Next-item claims of the window mode.  Items 8 apart (workgroups of one XCD:
// the same few kv heads) form a queue with a counter of its own; a workgroup
// claims from the queue of its XCD and, when that is empty, from the others in
// turn.  Of the workspace only the claim word is zero when a call starts, so the
// first workgroup of the call to claim (it sets kClaimsTaken) clears the
// counters and then sets kClaimsReady; one that comes while it does so waits for
// that bit.  The wait ends: the clearing thread is running and waits for
// nothing.  The merge kernel clears the claim word.
constexpr int kQueues = 8;
struct Claim {
  uint32_t queue;   // queue asked
  uint32_t got;     // thread 0: the counter's value (in flight until read)
  bool wanted;      // are there items that are not taken by place?
  bool asked;
  bool ready;       // thread 0: the counters have been seen ready
  __device__ __forceinline__ uint32_t take(const PrefillParams& p, uint32_t q) {
    return atomicAdd(p.claim + kTileClaims + q, 1u);
  }
  __device__ __forceinline__ void ask(const PrefillParams& p) {
    if (threadIdx.x == 0) {
      if (!ready) make_ready(p);
      ready = true;
      got = take(p, queue);
    }
    asked = true;
  }
  __device__ __forceinline__ void make_ready(const PrefillParams& p) {
    uint32_t word = __hip_atomic_fetch_or(p.claim, kClaimsTaken, __ATOMIC_ACQUIRE, __HIP_MEMORY_SCOPE_AGENT);
    if (!(word & kClaimsTaken)) {
      for (int q = 0; q < kQueues; ++q)
        __hip_atomic_exchange(p.claim + kTileClaims + q, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      __hip_atomic_fetch_or(p.claim, kClaimsReady, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_AGENT);
      return;
    }
    while (!(word & kClaimsReady)) {
      __builtin_amdgcn_s_sleep(1);
      word = __hip_atomic_load(p.claim, __ATOMIC_ACQUIRE, __HIP_MEMORY_SCOPE_AGENT);
    }
  }
};

// One query tile: rows [row0, row0 + nrows) of sequence s (nrows <= tokens
// per tile), query heads h0 .. h0+15 of kv head kvh.  PROMPT: the
// uniform-prompt mode (keys below the history length from pages, the rest
// from the dense prompt rows of sequence s); otherwise every key from pages.
template <int DT, int HD, int TPP, bool PROMPT, bool KV8, int RG>
__device__ __forceinline__ void prefill_tile(const PrefillParams& p, int row0, int nrows, int64_t s, int kvh, int h0,
                                             uint16_t* k_lds_base, uint16_t* v_lds_base, uint16_t* junk_lds,
                                             uint32_t* pid_lds, int* lim_lds, float* scl_lds, const int32_t* off_lds,
                                             Claim* claim) {
  static_assert(!PROMPT || !KV8, "prompts over fp8 pages run on half tiles (prefill_choose_tiles)");
  static_assert(HD % 32 == 0, "prefill needs head_dim % 32 == 0");
  constexpr int kMRows = m_rows(RG);
  constexpr int KS = HD / 16;  // QK k-steps of 16
  constexpr int DT32 = HD / 32;  // O^T row tiles of 32 dims
  constexpr int NI = StepGeo<HD>::kItems;
  constexpr int NL = StepGeo<HD>::kLoads;
  constexpr int NCH = KS * RG;  // MFMAs (and chunks) of each product per step
  using IM = ItemMap<HD, TPP>;
  // fp8 pools in window mode: steps are copied as fp8 bytes (16-byte items:
  // 16 dims of one key for K, 16 keys of one row for V; 2 HD items each, in
  // item order) and converted in the operand reads, each lane reading whole
  // items: a K item gives the 8 dims of two QK k-steps, a V item the 8 keys
  // of both PV k-steps (the keys of an fp8 step are in kperm_f8 order, the
  // query operand permuted to match).  A copy instruction must stay in one
  // page: with TPP 16 that needs HD % 64 == 0 (every fp8 pool's head dim).
  constexpr bool F8 = KV8;
  constexpr int NI8 = 2 * HD;
  constexpr int NL8 = (NI8 + kPfThreads - 1) / kPfThreads;
  constexpr int NC = F8 ? NL8 : NL;  // copies per thread per step of K, and as many of V
  static_assert(2 * NC <= NCH, "a step's copies fit in its PV chunks");
  float* ks_lds = scl_lds;                   // fp8: K scale of page-table entry e in slot e % 1024
  float* vs_lds = scl_lds + 2 * kPidChunk;   // and V scale
  auto k_lds = [&](int j) { return k_lds_base + (j & (kNBuf - 1)) * NI * 8; };  // step j's buffer
  auto v_lds = [&](int j) { return v_lds_base + (j & (kNBuf - 1)) * NI * 8; };

  // tile coordinates are workgroup-uniform: keep them in scalar registers
  row0 = __builtin_amdgcn_readfirstlane(row0);
  nrows = __builtin_amdgcn_readfirstlane(nrows);
  s = static_cast<int64_t>(__builtin_amdgcn_readfirstlane(static_cast<uint32_t>(s)));
  const int hg = min(16, p.group - h0);  // heads of this chunk
  const int qt = kMRows / p.hg_max;      // tokens per tile (hg_max = min(group, 16))
  constexpr bool prompt_mode = PROMPT;
  const bool seq_ok = s < p.num_seqs;  // a row naming no sequence attends to nothing
  if (!seq_ok) s = 0;
  const int tid = threadIdx.x;
  const int lane = lane_id();
  const int w = wave_id();
  const int col = lane & 31;  // this lane's M-row within a row group
  const int half = lane >> 5;

  const int64_t max_tokens = p.page_table_width * TPP;
  int64_t hist = 0;  // prompt mode: keys below hist come from pages
  int64_t slen;
  if (prompt_mode) {
    hist = p.seq_lens[s];
    PAL_DEBUG_FLAG(hist > max_tokens, kDebugLength);
    hist = hist < 0 ? 0 : (hist > max_tokens ? max_tokens : hist);
    slen = hist + p.prompt_len;
  } else {
    slen = seq_ok ? p.seq_lens[s] : 0;
    PAL_DEBUG_FLAG(slen > max_tokens, kDebugLength);
    slen = slen < 0 ? 0 : (slen > max_tokens ? max_tokens : slen);
  }

  // Loads that need nothing but the tile's coordinates go out first, so
  // their latency overlaps the row-limit round trip: the query operand and
  // the first kPidChunk page-table entries of the row (staged into LDS once
  // the limits say how many the tile reads; entries past the sequence's
  // pages are never used).
  constexpr int kLim = kMRows;  // lim_lds: per token; then 4 maxima and 4 minima, and the invalid-page flag
  constexpr int kBad = kLim + 2 * kPfWaves;  // word set when a staged page id is out of range
  const bool live_tok = tid < nrows && tid < qt;
  int64_t tok_off = 0;
  if (live_tok) tok_off = prompt_mode ? hist + (row0 + tid - s * p.prompt_len) + 1 : off_lds[tid];
  const uint32_t* pt = p.page_table + s * p.page_table_width;
  constexpr int kPidPre = kPidChunk / kPfThreads;  // entries of chunk 0 per thread
  uint32_t pid_pre[kPidPre];
#pragma unroll
  for (int j = 0; j < kPidPre; ++j) {
    const int e = tid + j * kPfThreads;
    pid_pre[j] = e < p.page_table_width ? pt[e] : 0u;
  }
  int m_row[RG], my_t[RG], my_h[RG];
  bool row_ok[RG];
  // Q^T operand: lane holds Q[M-row col of the group][16kk + 8 half .. +7] for all k-steps.
  // (An M-row past the tile takes row 0's query; its result is not written.)
  u32x4 qv[RG][KS];
#pragma unroll
  for (int r = 0; r < RG; ++r) {
    m_row[r] = (w * RG + r) * 32 + col;
    my_t[r] = static_cast<int>((static_cast<uint32_t>(m_row[r]) * p.hg_magic) >> 16);
    my_h[r] = m_row[r] - my_t[r] * p.hg_max;
    row_ok[r] = my_t[r] < nrows && my_t[r] < qt && my_h[r] < hg;
    const int64_t qrow = static_cast<int64_t>(row0 + (row_ok[r] ? my_t[r] : 0)) * p.num_q_heads + kvh * p.group + h0 +
                         (row_ok[r] ? my_h[r] : 0);
    if constexpr (F8) {
      // fp8 steps read 16 dims of stripe 2j + half per K item: k-step 2j + e
      // of this lane half takes dims 16 (2j + half) + 8e .. +7
      const uint16_t* qp = p.q + qrow * HD + 16 * half;
#pragma unroll
      for (int kk = 0; kk < KS; ++kk)
        qv[r][kk] = *reinterpret_cast<const u32x4*>(qp + 32 * (kk / 2) + 8 * (kk % 2));
    } else {
      const uint16_t* qp = p.q + qrow * HD + 8 * half;
#pragma unroll
      for (int kk = 0; kk < KS; ++kk) qv[r][kk] = *reinterpret_cast<const u32x4*>(qp + 16 * kk);
    }
  }

  // Key limits of the tile's tokens, and their largest and smallest per
  // wavefront (reduced across lanes by DPP: LDS atomics on one word serialise
  // over the lanes)
  __syncthreads();  // the previous tile is done with every LDS array
  {
    int lim = 0;
    if (live_tok) {
      const int64_t off = tok_off < 0 ? 0 : tok_off;
      lim = static_cast<int>(off < slen ? off : slen);
    }
    if (tid < kMRows) lim_lds[tid] = lim;
    const int mx = wave_max(lim);
    const int mn = -wave_max(live_tok ? -lim : -(1 << 30));
    if (lane == 0) {
      lim_lds[kLim + w] = mx;
      lim_lds[kLim + kPfWaves + w] = mn;
    }
    if (tid == 0) lim_lds[kBad] = 0;
  }
  // fp8: the scales of those page-table entries, behind the page ids
  float ks_pre[kPidPre], vs_pre[kPidPre];
#pragma unroll
  for (int j = 0; j < kPidPre; ++j) {
    ks_pre[j] = 0.f;
    vs_pre[j] = 0.f;
    if constexpr (F8) {
      const int e = tid + j * kPfThreads;
      if (e < p.page_table_width && pid_pre[j] < p.num_pages) {
        const int64_t si = static_cast<int64_t>(pid_pre[j]) * p.num_kv_heads + kvh;
        ks_pre[j] = p.k_scales[si];
        vs_pre[j] = p.v_scales[si];
      }
    }
  }
  __syncthreads();
  int max_lim = 0, min_lim = 1 << 30;
#pragma unroll
  for (int i = 0; i < kPfWaves; ++i) {
    max_lim = max(max_lim, lim_lds[kLim + i]);
    min_lim = min(min_lim, lim_lds[kLim + kPfWaves + i]);
  }
  max_lim = __builtin_amdgcn_readfirstlane(max_lim);
  min_lim = __builtin_amdgcn_readfirstlane(min_lim);
  int my_lim[RG];
#pragma unroll
  for (int r = 0; r < RG; ++r) my_lim[r] = row_ok[r] ? lim_lds[my_t[r]] : 0;

  const int64_t head_block = static_cast<int64_t>(HD) * TPP;
  const int64_t page_stride = head_block * p.num_kv_heads;
  const int64_t page_stride8 = page_stride;            // fp8 pools: bytes per page (one byte per element)
  const int64_t kv_head_off8 = kvh * head_block;       // and of a kv head's block
  const int64_t dense_row0 = s * p.prompt_len - hist;  // dense row of key token tok: dense_row0 + tok
  const int64_t dense_stride = static_cast<int64_t>(p.num_kv_heads) * HD;
  const int64_t kv_head_off = kvh * head_block;
  const int nsteps = (max_lim + kKeys - 1) / kKeys;
  // page-table entries the tile reads: keys below max_lim, and in prompt mode
  // only those below the history (the rest are dense) -- never past the width
  const int paged_keys = prompt_mode ? min(max_lim, static_cast<int>(hist)) : max_lim;
  const int n_pid = (paged_keys + TPP - 1) / TPP;

  // Page ids live in LDS (two chunks of 512 entries, entry e in slot e % 1024):
  // reading them is an LDS broadcast, so the only vector-memory traffic in the
  // step loop is the K/V copies, whose count the waits below rely on.
  // fp8: the (page, kv head) scales of entry e, beside its page id (0 for an
  // invalid id: such a step takes the register path, which reads none)
  auto stage_scales = [&](int e, uint32_t pg) {
    if constexpr (F8) {
      const bool ok = pg < p.num_pages;
      const int64_t si = static_cast<int64_t>(ok ? pg : 0) * p.num_kv_heads + kvh;
      ks_lds[pid_slot(e)] = ok ? p.k_scales[si] : 0.f;
      vs_lds[pid_slot(e)] = ok ? p.v_scales[si] : 0.f;
    }
  };
  auto stage_pids = [&](int chunk) {  // synchronous; callers hold a barrier after it
    for (int e = chunk * kPidChunk + tid; e < min((chunk + 1) * kPidChunk, n_pid); e += kPfThreads) {
      const uint32_t pg = pt[e];
      pid_lds[pid_slot(e)] = pg;
      if (pg >= p.num_pages) lim_lds[kBad] = 1;
      stage_scales(e, pg);
    }
  };

  // Fast step: its first key below the tile's largest limit (the last step
  // may end past it), in valid pages (and, in prompt mode, all 32 keys below
  // the history, or all of them prompt keys): one direct-to-LDS copy per
  // item, no registers, nothing to wait for here.  Every wavefront issues exactly
  // NC copies of K and NC of V (items past the step go to a junk slot), so the
  // wait counts are the same on every wavefront.
  // Slow step (invalid pages, history / prompt boundary): register loads,
  // masked, then LDS stores -- synchronous, and it drains the copies in
  // flight, which keeps the counted waits safe.
  // pg0 / pg1: the pages of the step's first and (TPP 16) second 16 keys.
  constexpr bool kAllItems = (F8 ? NI8 : NI) % kPfThreads == 0;  // no wavefront has a padding copy
  __builtin_assume(w >= 0 && w < kPfWaves);
  // The copies take a page's (a prompt row's) stride as 32 bits; longer ones go
  // the slow path.
  const bool long_pages = page_stride * (KV8 ? 1 : 2) > 0xFFFFFFFFll;
  const bool long_rows = PROMPT && dense_stride * 2 > 0xFFFFFFFFll;
  // page ids >= 2^32 - 1 cannot occur with fewer pages; such an id takes the slow path
  const uint32_t np32 =
      long_pages ? 0u : (p.num_pages > 0xFFFFFFFFll ? 0xFFFFFFFFu : static_cast<uint32_t>(p.num_pages));
  // fp8 items.  K item i: page half ph (TPP 16), stripe c (dims 16c ..
  // 16c+15), key of the step; V item i: page half ph (TPP 16) or 16-key half
  // of the page row (TPP 32), row d.  Item i is LDS slot i.
  auto k8_item = [](int i, int& ph, int& c, int& key) {
    if (TPP == 16) {  // page-major; page 1's keys at positions XOR 12, so a 16-lane operand read spans all banks
      ph = i / HD;
      c = (i % HD) / 16;
      key = 16 * ph + ((i % 16) ^ (ph ? 12 : 0));
    } else {  // operand row order: slot 32 c + m holds key kperm_f8(m)
      ph = 0;
      c = i / 32;
      key = kperm_f8(i % 32);
    }
  };
  auto v8_item = [](int i, int& ph, int& d, int& kb) {  // kb: the item's first key in the step
    ph = TPP == 16 ? i / HD : 0;
    d = i % HD;
    kb = 16 * (i / HD);
  };
  const uint8_t* k8_pool = reinterpret_cast<const uint8_t*>(p.k_pool) + kv_head_off8;
  const uint8_t* v8_pool = reinterpret_cast<const uint8_t*>(p.v_pool) + kv_head_off8;
  // This lane's source address of copy q in page 0 of the pool: a copy of
  // page pg reads page_bytes * pg further (one v_mad_u64_u32).
  const uint32_t page_bytes = static_cast<uint32_t>(page_stride * (KV8 ? 1 : 2));
  auto item_of = [&](int q) { return tid + q * kPfThreads; };
  auto wave_item = [&](int q) { return w * kWave + q * kPfThreads; };  // first item of this wavefront's load
  auto live_copy = [&](int q) { return kAllItems || wave_item(q) < (F8 ? NI8 : NI); };
  auto k_src = [&](int q) {
    const int i = live_copy(q) ? item_of(q) : lane;
    if constexpr (F8) {
      int ph, c, key;
      k8_item(i, ph, c, key);
      return reinterpret_cast<uint64_t>(k8_pool) + static_cast<uint32_t>((c * TPP + key % TPP) * 16);
    } else {
      return reinterpret_cast<uint64_t>(p.k_pool + kv_head_off) + 2u * static_cast<uint32_t>(IM::k_offset(i));
    }
  };
  auto v_src = [&](int q) {
    const int i = live_copy(q) ? item_of(q) : lane;
    if constexpr (F8) {
      int ph, d, kb;
      v8_item(i, ph, d, kb);
      return reinterpret_cast<uint64_t>(v8_pool) + static_cast<uint32_t>(d * TPP + kb % TPP);
    } else {
      int d, key;
      IM::v_item(i, d, key);
      return reinterpret_cast<uint64_t>(p.v_pool + kv_head_off) + 2u * static_cast<uint32_t>(d * TPP + key % TPP);
    }
  };
  uint64_t ksrc[NC], vsrc[NC];
#pragma unroll
  for (int q = 0; q < NC; ++q) {
    ksrc[q] = k_src(q);
    vsrc[q] = v_src(q);
  }
  // the page half (TPP 16) a wavefront's load q reads: one page per instruction
  auto copy_half = [&](int q) { return F8 ? (TPP == 16 ? wave_item(q) / HD : 0) : IM::k_page_half(wave_item(q)); };
  auto copy_k = [&](int q, int j, uint32_t pg0, uint32_t pg1) {
    const bool ok = live_copy(q);
    const uint32_t pg = ok && copy_half(q) ? pg1 : pg0;
    copy_row_to_lds16(ksrc[q], pg, page_bytes, lds_addr(ok ? k_lds(j) + wave_item(q) * 8 : junk_lds));
  };
  auto copy_v = [&](int q, int j, uint32_t pg0, uint32_t pg1) {
    const bool ok = live_copy(q);
    const uint32_t pg = ok && copy_half(q) ? pg1 : pg0;
    copy_row_to_lds16(vsrc[q], pg, page_bytes, lds_addr(ok ? v_lds(j) + wave_item(q) * 8 : junk_lds));
  };
  // step j takes the fast path
  // (the tile's last step may end past max_lim: its copies then read keys
  // no row sees, from valid pages, and fix_tail clears their V entries)
  auto is_fast = [&](int j, uint32_t pg0, uint32_t pg1) {
    const int k0 = j * kKeys;
    return k0 < max_lim && pg0 < np32 && pg1 < np32 && (!prompt_mode || k0 + kKeys <= hist);
  };
  // Prompt mode: a step whose 32 keys are all prompt keys below the tile's
  // largest limit copies them from the dense prompt rows (16-bit in every
  // pool dtype): K into its operand layout, V rows untransposed (V items of
  // the row layout are 16 contiguous bytes of one key; the PV operand reads
  // of such a step transpose).
  auto is_dense = [&](int j) {
    const int k0 = j * kKeys;
    return PROMPT && !long_rows && k0 >= hist && k0 < max_lim;
  };
  // the dense row of the step's key `key` (keys past max_lim repeat the last one's row)
  auto dense_row = [&](int j, int key) {
    return static_cast<uint32_t>(static_cast<int>(dense_row0) + min(j * kKeys + key, max_lim - 1));
  };
  const uint32_t dense_bytes = static_cast<uint32_t>(dense_stride * 2);
  auto copy_dense_k = [&](int q, int j) {  // K in its operand layout, as from pages
    const bool ok = live_copy(q);
    int c = 0, key = 0;
    if (ok) IM::k_item(item_of(q), c, key);
    const uint64_t src = reinterpret_cast<uint64_t>(p.k_dense + kvh * HD + c * 8);
    copy_row_to_lds16(src, dense_row(j, key), dense_bytes, lds_addr(ok ? k_lds(j) + wave_item(q) * 8 : junk_lds));
  };
  auto copy_dense_v = [&](int q, int j) {  // raw rows: slot i = (key, 8-dim chunk c ^ vd_swz(key))
    const bool ok = live_copy(q);
    const int i = item_of(q);
    const int key = ok ? i / (HD / 8) : 0, c = ok ? (i % (HD / 8)) ^ vd_swz<HD>(key) : 0;
    const uint64_t src = reinterpret_cast<uint64_t>(p.v_dense + kvh * HD + c * 8);
    copy_row_to_lds16(src, dense_row(j, key), dense_bytes, lds_addr(ok ? v_lds(j) + wave_item(q) * 8 : junk_lds));
  };

  // The K (V) part of a step on the register path.
  auto slow_k = [&](int j, uint32_t pg0, uint32_t pg1) {
    const int k0 = j * kKeys;
    uint16_t* kb = k_lds(j);
    if constexpr (F8) {  // a page id out of range: the same items, zero for invalid pages
#pragma unroll
      for (int jj = 0; jj < NL8; ++jj) {
        const int i = item_of(jj);
        if (i >= NI8) continue;
        int ph, c, key;
        k8_item(i, ph, c, key);
        const uint32_t pg = ph ? pg1 : pg0;
        PAL_DEBUG_FLAG(pg >= p.num_pages && k0 + key < max_lim, kDebugPageId);
        u32x4 val = {0u, 0u, 0u, 0u};
        if (pg < p.num_pages && k0 + key < max_lim)
          val = *reinterpret_cast<const u32x4*>(k8_pool + static_cast<int64_t>(pg) * page_stride8 +
                                                (c * TPP + key % TPP) * 16);
        *reinterpret_cast<u32x4*>(kb + i * 8) = val;
      }
    } else {
#pragma unroll
      for (int jj = 0; jj < NL; ++jj) {
        const int i = item_of(jj);
        if (i >= NI) continue;
        int kj, c;
        IM::k_item(i, c, kj);
        const int tok = k0 + kj;
        const uint32_t pg = IM::k_page_half(i) ? pg1 : pg0;
        const bool pg_ok = pg < p.num_pages;
        PAL_DEBUG_FLAG(!pg_ok && k0 + (IM::k_page_half(i) ? 16 : 0) < paged_keys, kDebugPageId);
        u32x4 val = {0u, 0u, 0u, 0u};
        if (!prompt_mode || tok < hist) {
          if (pg_ok && tok < max_lim)
            val = *reinterpret_cast<const u32x4*>(p.k_pool + static_cast<int64_t>(pg) * page_stride + kv_head_off +
                                                  IM::k_offset(i));
        } else if (tok < max_lim) {
          val = *reinterpret_cast<const u32x4*>(p.k_dense + (dense_row0 + tok) * dense_stride + kvh * HD + c * 8);
        }
        *reinterpret_cast<u32x4*>(kb + i * 8) = val;
      }
    }
    __builtin_amdgcn_s_waitcnt(vmcnt_only(0));
  };
  auto slow_v = [&](int j, uint32_t pg0, uint32_t pg1) {
    const int k0 = j * kKeys;
    uint16_t* vb = v_lds(j);
    if constexpr (F8) {  // zero for invalid pages, keys past max_lim cleared
#pragma unroll
      for (int jj = 0; jj < NL8; ++jj) {
        const int i = item_of(jj);
        if (i >= NI8) continue;
        int ph, d, kb;
        v8_item(i, ph, d, kb);
        const uint32_t pg = ph ? pg1 : pg0;
        u32x4 val = {0u, 0u, 0u, 0u};
        const int valid = max_lim - (k0 + kb);
        if (pg < p.num_pages && valid > 0) {
          val = *reinterpret_cast<const u32x4*>(v8_pool + static_cast<int64_t>(pg) * page_stride8 + d * TPP + kb % TPP);
#pragma unroll
          for (int e = 0; e < 4; ++e)
#pragma unroll
            for (int bb = 0; bb < 4; ++bb)
              if (4 * e + bb >= valid) val[e] &= ~(0xFFu << (8 * bb));
        }
        *reinterpret_cast<u32x4*>(vb + i * 8) = val;
      }
    } else {
#pragma unroll
      for (int jj = 0; jj < NL; ++jj) {
        const int i = item_of(jj);
        if (i >= NI) continue;
        // row d, keys key .. key+7 of the step (they share a page)
        int d, key;
        IM::v_item(i, d, key);
        const int tok = k0 + key;
        const uint32_t pg = IM::k_page_half(i) ? pg1 : pg0;
        const bool pg_ok = pg < p.num_pages;
        const uint16_t* vrow = p.v_pool + static_cast<int64_t>(pg) * page_stride + kv_head_off + d * TPP + key % TPP;
        u32x4 val = {0u, 0u, 0u, 0u};
        if (!prompt_mode || tok + 8 <= hist) {
          if (pg_ok && tok < max_lim) val = *reinterpret_cast<const u32x4*>(vrow);
        } else if (tok < max_lim) {
          // some of the 8 keys are prompt tokens (dense, strided by row)
          uint32_t e16[8];
#pragma unroll
          for (int e = 0; e < 8; ++e) {
            const int t2 = tok + e;
            const bool pgd = t2 < hist;
            uint16_t x = 0;
            if (t2 < max_lim && (!pgd || pg_ok))
              x = pgd ? vrow[e] : p.v_dense[(dense_row0 + t2) * dense_stride + kvh * HD + d];
            e16[e] = x;
          }
          val = {e16[0] | (e16[1] << 16), e16[2] | (e16[3] << 16), e16[4] | (e16[5] << 16), e16[6] | (e16[7] << 16)};
        }
        // keys past the largest limit may hold anything (NaN bits included)
        const int valid = max_lim - tok;
        if (valid < 8) {
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const uint32_t keep = (2 * e < valid ? 0x0000FFFFu : 0u) | (2 * e + 1 < valid ? 0xFFFF0000u : 0u);
            val[e] &= keep;
          }
        }
        *reinterpret_cast<u32x4*>(vb + i * 8) = val;
      }
    }
    __builtin_amdgcn_s_waitcnt(vmcnt_only(0));
  };
  auto issue_k = [&](int j, uint32_t pg0, uint32_t pg1) {
    if (is_dense(j)) {
#pragma unroll
      for (int q = 0; q < NC; ++q) copy_dense_k(q, j);
    } else if (is_fast(j, pg0, pg1)) {
#pragma unroll
      for (int q = 0; q < NC; ++q) copy_k(q, j, pg0, pg1);
    } else {
      slow_k(j, pg0, pg1);
    }
  };
  auto issue_v = [&](int j, uint32_t pg0, uint32_t pg1) {
    if (is_dense(j)) {
#pragma unroll
      for (int q = 0; q < NC; ++q) copy_dense_v(q, j);
    } else if (is_fast(j, pg0, pg1)) {
#pragma unroll
      for (int q = 0; q < NC; ++q) copy_v(q, j, pg0, pg1);
    } else {
      slow_v(j, pg0, pg1);
    }
  };
  // The tile's last step j, when it ends past max_lim and was copied: the
  // keys no row sees hold whatever the pages (or, in prompt mode, the row of
  // the last key) held, and a masked probability of 0 times a NaN there
  // would still be NaN, so their V entries are cleared.  Each thread clears
  // the items it copied itself, once its copies have landed and before the
  // barrier preceding the step's V reads (a slow step's entries are zero
  // already).
  auto fix_tail = [&](int j) {
    __builtin_amdgcn_s_waitcnt(vmcnt_only(0));
    compiler_fence();
    const int valid0 = max_lim - j * kKeys;  // valid keys of the step, 1 .. 31
    uint16_t* vb = v_lds(j);
    if constexpr (F8) {  // fp8 items: 16 key bytes of one row
#pragma unroll
      for (int jj = 0; jj < NL8; ++jj) {
        const int i = item_of(jj);
        if (i >= NI8) continue;
        int ph, d, kb;
        v8_item(i, ph, d, kb);
        const int valid = valid0 - kb;
        if (valid < 16) {
          u32x4* slot = reinterpret_cast<u32x4*>(vb + i * 8);
          u32x4 val = *slot;
#pragma unroll
          for (int e = 0; e < 4; ++e)
#pragma unroll
            for (int bb = 0; bb < 4; ++bb)
              if (4 * e + bb >= valid) val[e] &= ~(0xFFu << (8 * bb));
          *slot = val;
        }
      }
      return;
    }
    const bool dense = is_dense(j);
#pragma unroll
    for (int jj = 0; jj < NL; ++jj) {
      const int i = item_of(jj);
      if (i >= NI) continue;
      u32x4* slot = reinterpret_cast<u32x4*>(vb + i * 8);
      if (dense) {  // raw rows: slot i holds 8 dims of key i / (HD / 8)
        if (i / (HD / 8) >= valid0) *slot = u32x4{0u, 0u, 0u, 0u};
      } else {  // operand layout: 8 keys key .. key+7 of row d
        int d, key;
        IM::v_item(i, d, key);
        const int valid = valid0 - key;
        if (valid < 8) {
          u32x4 val = *slot;
#pragma unroll
          for (int e = 0; e < 4; ++e)
            val[e] &= (2 * e < valid ? 0x0000FFFFu : 0u) | (2 * e + 1 < valid ? 0xFFFF0000u : 0u);
          *slot = val;
        }
      }
    }
  };
  const bool tail_partial = max_lim % kKeys != 0;  // the last step ends past max_lim
  // fp8: the scales of step j's first and (TPP 16) second page (LDS
  // broadcast); 0 for a page past the tile's last staged entry (the tail
  // step's keys past max_lim: their V bytes are cleared, and 0 x a stale
  // scale could be NaN)
  auto read_scales = [&](const float* arr, int j, float& s0, float& s1) {
    const int e = j * (kKeys / TPP);  // (even with TPP 16)
    const float a0 = arr[pid_slot(e)], a1 = arr[pid_slot(e + (TPP == 16))];
    s0 = e < n_pid ? a0 : 0.f;
    s1 = TPP == 16 ? (e + 1 < n_pid ? a1 : 0.f) : s0;
  };
  // the page ids of step j (an LDS broadcast read; TPP 32: one page)
  auto read_pids = [&](int j) {
    const int e = pid_slot(j * (kKeys / TPP));
    u32x2 v;
    if (TPP == 16) {
      v = *reinterpret_cast<const u32x2*>(pid_lds + e);  // e is even: 8-byte aligned
    } else {
      v.x = pid_lds[e];
      v.y = v.x;
    }
    return v;
  };

  // minus the running max of this lane's M-row (log2 units).  kNoMax, until the
  // row's first score above -inf: with it the exponent of -inf is -inf, and that
  // of any other score so far past the headroom that the max moves to it.
  float mb[RG];
  // exp-sum: of the probabilities as rounded for the PV product, by MFMA (kMmaSum:
  // the whole row's, in every lane) or by unpacking and adding; over fp8 pages of
  // the probabilities before the V scale (both: this lane's share).  Adds where the
  // steps are longest and the matrix pipe is the busier one: two row groups at
  // head dim 128, 16 x 1,024 prompt rows on 1,024 cached 436 -> 425 us; at head dim 64
  // 275 -> 304, one row group 67 -> 71.
  constexpr bool kMmaSum = !F8 && !(RG == 2 && HD >= 128);
  float l_run[RG];
  // kMmaSum: the last step's, not yet in l_run, of M-rows 0 .. 15 and 16 .. 31 of the group
  float step_lo[RG], step_hi[RG];
  // O^T of row group r, row tile n (dims 32 n ..): accumulator r * DT32 + n
  static_assert(RG * DT32 <= 8, "eight accumulators");
  acc_reserve();
  auto acc_zero = [&] { static_for<RG * DT32 * 16>([](auto x) { acc_put<decltype(x)::value>(0.f); }); };
#pragma unroll
  for (int r = 0; r < RG; ++r) {
    mb[r] = 0.f;
    l_run[r] = step_lo[r] = step_hi[r] = 0.f;
  }

  // Key order inside a 32-key step.  The QK product's A operand takes key
  // kperm(m) as its row m (bits 2 and 3 of m swapped); then the 8 scores a
  // lane feeds into each PV k-step are 8 consecutive keys, and the V^T operand
  // is one 16-byte LDS read per lane.  LDS already holds K in this row order.

  // S^T[key][M-row] = sum_d K[key][d] Q[M-row][d]: k-step kk's K operand.
  // fp8: lane: key kperm_f8(col), all 16 dims of stripe 2j + half: k-steps 2j
  // and 2j + 1 (read raw into k16, converted by the k-step's chunk).
  auto read_k = [&](int j, int kk) {
    const int c = 2 * kk + half;  // stripe of dims 16kk + 8 half .. +7
    return *reinterpret_cast<const u32x4*>(k_lds(j) + IM::k_slot(col, c) * 8);
  };
  auto read_k8 = [&](int j, int kj) {
    const int key = kperm_f8(col);
    const int c = 2 * kj + half;
    const int slot = TPP == 16 ? (key / 16) * HD + c * 16 + ((key % 16) ^ (key >= 16 ? 12 : 0)) : c * 32 + col;
    return *reinterpret_cast<const u32x4*>(reinterpret_cast<const uint8_t*>(k_lds(j)) + slot * 16);
  };
  // V^T operand bases: k-step kk takes keys 16kk + 8 half .. +7; row tile n
  // (dims 32n + col) sits kVRowTile slots further
  const int v_base[2] = {IM::v_slot(col, 8 * half), IM::v_slot(col, 16 + 8 * half)};
  // Score register x of a step holds key k0 + 16 (x/8) + 8 half + 4 ((x/4)%2) +
  // x%4 of M-row col (fp8 steps: key k0 + 16 half + x).  The exponent is one
  // fma: s * scale_log2 - m * scale_log2.  The rounding of m * scale_log2 is
  // common to a step's keys and cancels in the normalisation while that
  // product stays below ~2^14 (log2 units; trained models' logits are far
  // below); it grows with the product and overflows exp2 past ~2^31.  An exact
  // (s - m) * scale_log2 costs one more VALU instruction per score.
  // keys of step j's half-step that M-row r sees: register x is visible while
  // its key's place in the lane's order is below
  auto seen = [&](int r, int j) { return my_lim[r] - j * kKeys - (F8 ? 16 : 8) * half; };
  auto place = [](int x) { return F8 ? x : 16 * (x >> 3) + 4 * ((x >> 2) & 1) + (x & 3); };
  // fp8: the K scale of each key's page rides on the score scale (the lane's
  // keys are one page half)
  auto score_scale = [&](int j) {
    if constexpr (F8) {
      float s0, s1;
      read_scales(ks_lds, j, s0, s1);
      return p.scale_log2 * (half ? s1 : s0);
    } else {
      return p.scale_log2;
    }
  };

  // Pipeline (iteration st; step st's exponents e are in registers, and the K
  // operands of step st+1).
  //  Memory: iteration st issues the copies of K step st+5 and V step st+3, in
  //  that order.  At its top it waits for those issued three iterations ago or
  //  earlier (K step st+2, V step st) and passes the barrier.  K step st+2 is
  //  read in this iteration's second half, so buffers hold K steps st+2 ..
  //  st+5 and V steps st .. st+3; the copies overwrite K step st+1 and V step
  //  st-1, which every wavefront finished reading before the barrier.
  //  Compute, first half: the QK MFMAs of step st+1 beside the exponentials
  //  of step st and the V operand reads; second half: the PV MFMAs of step st
  //  beside the exp-sum of step st, the exponents and row max of step st+1 and
  //  the K operand reads of step st+2.
  if (nsteps > 0) {
#pragma unroll
    for (int j = 0; j < kPidPre; ++j) {  // chunk 0, loaded above
      const int e = tid + j * kPfThreads;
      if (e < n_pid) {
        pid_lds[e] = pid_pre[j];
        if (pid_pre[j] >= p.num_pages) lim_lds[kBad] = 1;
        if constexpr (F8) {
          ks_lds[e] = ks_pre[j];
          vs_lds[e] = vs_pre[j];
        }
      }
    }
    if (n_pid > kPidChunk) stage_pids(1);
  }
  // The query loads are waited for here, on every path: the compiler would
  // otherwise wait for them (and so for the copies, which it does not see)
  // inside the step loops.
#pragma unroll
  for (int r = 0; r < RG; ++r)
#pragma unroll
    for (int kk = 0; kk < KS; ++kk) asm volatile("" : "+v"(qv[r][kk]));
  __syncthreads();
  auto barrier = [&] {
    __builtin_amdgcn_s_waitcnt(kLgkmZero);
    __builtin_amdgcn_s_barrier();
    compiler_fence();
  };
  // all copies but those of the last two iterations landed (fewer were
  // issued near the tile's end: the V copies only, or none)
  auto wait_top = [&](int st) {
    compiler_fence();
    if (st + kLeadK - 1 < nsteps)
      __builtin_amdgcn_s_waitcnt(vmcnt_only(4 * NC));
    else if (st + kLeadV - 1 < nsteps)
      __builtin_amdgcn_s_waitcnt(vmcnt_only(2 * NC));
    else
      __builtin_amdgcn_s_waitcnt(vmcnt_only(0));
    barrier();
  };
  f32x16 e_cur[RG];
  // Step j's largest score (log2 units) of M-row r that the row sees, and its
  // exponents with the running max as it is now.  Both come from the raw scores:
  // an exponent is rounded once, in its fma, however far the max moves.
  auto step_max = [&](int r, int j, bool masked, const f32x16& s, float sc) {
    float bm = -INFINITY;
#pragma unroll
    for (int x = 0; x < 16; ++x)
      if (!masked || place(x) < seen(r, j)) bm = fmaxf(bm, s[x] * sc);
    return max_xor32(bm);
  };
  auto exponents = [&](int r, int j, bool masked, const f32x16& s, float sc) {
#pragma unroll
    for (int x = 0; x < 16; ++x) {
      const float v = fmaf(s[x], sc, mb[r]);
      e_cur[r][x] = !masked || place(x) < seen(r, j) ? v : -INFINITY;
    }
  };
  u32x4 ka[F8 ? KS / 2 : KS];  // K operands of the next QK product (fp8: raw items of two k-steps)
  auto k_operand = [&](int kk) {
    if constexpr (F8) {  // exact in 16 bits; the K scale goes on the scores
      const u32x4 v = ka[kk / 2];
      return fp8x8_exact<DT>(kk % 2 ? u32x2{v.z, v.w} : u32x2{v.x, v.y});
    } else {
      return ka[kk];
    }
  };
  auto read_k_all = [&](int j) {
#pragma unroll
    for (int kk = 0; kk < (F8 ? KS / 2 : KS); ++kk) ka[kk] = F8 ? read_k8(j, kk) : read_k(j, kk);
  };
  // whole steps in pages that the copies can read
  const int paged_full = !long_pages ? paged_keys / kKeys : 0;
  if (nsteps > 0) {
    auto pids = [&](int j, uint32_t& a, uint32_t& b) {
      const u32x2 v = read_pids(j);
      a = __builtin_amdgcn_readfirstlane(v.x);
      b = TPP == 16 ? __builtin_amdgcn_readfirstlane(v.y) : a;
    };
    // K 0, K 1, V 0, K 2, V 1, K 3, V 2
    if (paged_full >= 4 && __builtin_amdgcn_readfirstlane(lim_lds[kBad]) == 0) {
      u32x2 pg[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) pg[j] = read_pids(j);
#pragma unroll
      for (int t = 0; t < 7; ++t) {
        const bool is_k = t == 0 || (t & 1);
        const int j = is_k ? (t + 1) / 2 : t / 2 - 1;
#pragma unroll
        for (int q = 0; q < NC; ++q) {
          if (is_k)
            copy_k(q, j, pg[j].x, pg[j].y);
          else
            copy_v(q, j, pg[j].x, pg[j].y);
        }
      }
    } else {
#pragma unroll 1
      for (int t = 0; t < 7; ++t) {
        const bool is_k = t == 0 || (t & 1);
        const int j = is_k ? (t + 1) / 2 : t / 2 - 1;
        if (j >= nsteps) continue;
        uint32_t pa, pb;
        pids(j, pa, pb);
        if (is_k)
          issue_k(j, pa, pb);
        else
          issue_v(j, pa, pb);
      }
    }
    acc_zero();
    compiler_fence();
    if (nsteps >= 4)
      __builtin_amdgcn_s_waitcnt(vmcnt_only(5 * NC));  // K steps 0 and 1
    else
      __builtin_amdgcn_s_waitcnt(vmcnt_only(0));
    if (nsteps == 1 && tail_partial) fix_tail(0);
    barrier();
    read_k_all(0);
    f32x16 s0[RG];
#pragma unroll
    for (int r = 0; r < RG; ++r)
#pragma unroll
      for (int x = 0; x < 16; ++x) s0[r][x] = 0.f;
#pragma unroll
    for (int kk = 0; kk < KS; ++kk) {
      const u32x4 kop = k_operand(kk);
#pragma unroll
      for (int r = 0; r < RG; ++r) s0[r] = Dt<DT>::mma32x32x16(kop, qv[r][kk], s0[r]);
    }
    read_k_all(1);
    barrier();  // every wavefront has read K step 0: its buffer takes step 4
    if (nsteps > 4) {
      uint32_t pa, pb;
      pids(4, pa, pb);
      issue_k(4, pa, pb);
    }
    const float sc = score_scale(0);
#pragma unroll
    for (int r = 0; r < RG; ++r) {
      const float bm = step_max(r, 0, min_lim < kKeys, s0[r], sc);
      mb[r] = bm == -INFINITY ? kNoMax : -bm;
      exponents(r, 0, min_lim < kKeys, s0[r], sc);
    }
  }
  auto take_sums = [&] {  // the last step's exp-sums into the running ones
    if constexpr (kMmaSum) {
#pragma unroll
      for (int r = 0; r < RG; ++r) {
        l_run[r] += (lane & 16) ? step_hi[r] : step_lo[r];
        step_lo[r] = step_hi[r] = 0.f;
      }
    }
  };
  // One iteration.  kFast: step st+1 needs no mask and the iteration's copies
  // are plain (pages known to be valid, or whole dense steps): no test of a
  // page id and no branch in the body.  Otherwise scores are masked and each
  // copy's route is looked up.  kLast: the tile's last step (nothing follows).
  // vdense: step st's V rows were copied untransposed (a dense prompt step);
  // each combination is its own loop body, so the operand reads carry no
  // per-chunk branch.
  enum { kFast, kAny, kLast };
  auto step = [&](auto mode_c, auto dense_v, int st) {
    constexpr int kMode = decltype(mode_c)::value;
    constexpr bool vdense = decltype(dense_v)::value;
    if constexpr (kMode == kFast) {
      compiler_fence();
      __builtin_amdgcn_s_waitcnt(vmcnt_only(4 * NC));
      barrier();
    } else {
      wait_top(st);
    }
    take_sums();
    const int jk = st + kLeadK, jv = st + kLeadV;
    const u32x2 pgk = read_pids(jk), pgv = read_pids(jv);  // used in the second half (in bounds whether or not the steps exist)
    if (kMode == kAny && st + 2 == nsteps && tail_partial) fix_tail(st + 1);
    // The rest is written in issue order, chunk by chunk, with scheduling
    // fences between chunks (the compiler would otherwise keep two operand
    // reads in flight, wait before every MFMA and bunch the vector work).
    sched_fence();
    float vs0 = 1.f, vs1 = 1.f;  // fp8: V scales of step st's pages
    if constexpr (F8) read_scales(vs_lds, st, vs0, vs1);
    const float svs = half ? vs1 : vs0;  // the lane's keys 16 half .. +15: page half (TPP 32: vs1 == vs0)
    f32x16 s_next[RG];
#pragma unroll
    for (int r = 0; r < RG; ++r)
#pragma unroll
      for (int x = 0; x < 16; ++x) s_next[r][x] = 0.f;
    u32x4 va[KS];  // PV operand m: k-step m / DT32, row tile m % DT32 (KS == 2 * DT32)
    u32x4 v16[F8 ? DT32 : 1];  // fp8: row tile t's item (16 keys of one row), both PV k-steps
    u32x4 pp[RG][2];  // packed probabilities of the lane's scores, 8 per PV k-step
    // probability pair q (row group q / 8): exponentials, and one chunk later
    // (past their latency) the conversion
    auto pair_exp = [&](int q) {
      const int r = q / 8, i = q % 8;
      e_cur[r][2 * i] = __builtin_amdgcn_exp2f(e_cur[r][2 * i]);
      e_cur[r][2 * i + 1] = __builtin_amdgcn_exp2f(e_cur[r][2 * i + 1]);
    };
    auto pair_pack = [&](int q) {
      const int r = q / 8, i = q % 8;
      const float p0 = e_cur[r][2 * i], p1 = e_cur[r][2 * i + 1];
      if constexpr (F8)  // P times its key's page V scale (the exp-sum stays unscaled)
        pp[r][i / 4][i % 4] = Dt<DT>::pack2(p0 * svs, p1 * svs);
      else
        pp[r][i / 4][i % 4] = Dt<DT>::pack2(p0, p1);
      // Held here: code motion would otherwise sink the conversion to the PV
      // MFMA that reads it, which (as inline assembly) must stand two
      // instructions or more behind it.
      if (i % 4 == 3) asm volatile("" : "+v"(pp[r][i / 4]));
    };
    auto pair_sum = [&](int q) {
      if constexpr (kMmaSum) return;
      const int r = q / 8, i = q % 8;
      const uint32_t w = pp[r][i / 4][i % 4];
      l_run[r] += F8 ? e_cur[r][2 * i] : Dt<DT>::lo(w);
      l_run[r] += F8 ? e_cur[r][2 * i + 1] : Dt<DT>::hi(w);
    };
    constexpr int kPairs = 8 * RG;
    // row group 0's share of the exp-sum goes beside the QK MFMAs, row group
    // 1's beside the first PV MFMAs (its exponents are replaced last)
    constexpr int kSumA = RG == 2 ? 8 : kPairs;
    u32x4 kop;
#pragma unroll
    for (int c = 0; c < NCH; ++c) {
      const int kk = c / RG;
      if constexpr (kMode != kLast) {
        if (c % RG == 0) kop = k_operand(kk);
        s_next[c % RG] = Dt<DT>::mma32x32x16(kop, qv[c % RG][kk], s_next[c % RG]);
      }
      if (c % RG == 0) {
        if constexpr (vdense) {
          va[kk] = read_dense_v<HD>(v_lds(st), kk / DT32, kk % DT32, col, half);
        } else if constexpr (F8) {
          // chunk t < DT32 reads row tile t's item (half, d = col + 32 t): keys
          // 16 half .. +7 for k-step 0 (operand t), +8 .. +15 for k-step 1
          // (operand t + DT32).  Exact in 16 bits; the V scale is on P.
          if (kk < DT32)
            v16[kk] = *reinterpret_cast<const u32x4*>(reinterpret_cast<const uint8_t*>(v_lds(st)) +
                                                      (half * HD + col + 32 * kk) * 16);
          // each half is converted in a later chunk than its read (the LDS
          // read has landed) and consumed there, so the conversions are not
          // sunk to the PV MFMAs
          if (kk >= 1 && kk <= DT32) {
            va[kk - 1] = fp8x8_exact<DT>(u32x2{v16[kk - 1].x, v16[kk - 1].y});
            asm volatile("" ::"v"(va[kk - 1]));
          }
          if (kk >= DT32) {
            va[kk] = fp8x8_exact<DT>(u32x2{v16[kk - DT32].z, v16[kk - DT32].w});
            asm volatile("" ::"v"(va[kk]));
          }
        } else {
          va[kk] = *reinterpret_cast<const u32x4*>(v_lds(st) + (v_base[kk / DT32] + (kk % DT32) * IM::kVRowTile) * 8);
        }
      }
#pragma unroll
      for (int q = c * kPairs / NCH; q < (c + 1) * kPairs / NCH; ++q) pair_exp(q);
      if (c > 0) {
#pragma unroll
        for (int q = (c - 1) * kPairs / NCH; q < c * kPairs / NCH; ++q) {
          pair_pack(q);
          if (q < kSumA) pair_sum(q);
        }
      }
      sched_fence();
    }
    // O^T[d][M-row] += sum_key V[key][d] P[M-row][key]; k-step kk takes
    // registers 8kk .. 8kk+7 = keys 16kk + 8 half .. +7.
    float bm[RG];
#pragma unroll
    for (int r = 0; r < RG; ++r) bm[r] = -INFINITY;
    // The iteration's copies go out one per PV chunk, K then V, so the
    // wavefront's MFMAs run while an issue waits for the memory pipeline
    // (steps that cannot be copied take the synchronous path below).
    bool kdn = false, vdn = false, kfast = false, vfast = false;
    uint32_t kp0 = 0, kp1 = 0, vp0 = 0, vp1 = 0;
    if (kMode == kAny && jv < nsteps) {
      kp0 = __builtin_amdgcn_readfirstlane(pgk.x);
      kp1 = TPP == 16 ? __builtin_amdgcn_readfirstlane(pgk.y) : kp0;
      vp0 = __builtin_amdgcn_readfirstlane(pgv.x);
      vp1 = TPP == 16 ? __builtin_amdgcn_readfirstlane(pgv.y) : vp0;
      kdn = jk < nsteps && (vdense || is_dense(jk));  // steps after a dense one are dense
      vdn = jv < nsteps && (vdense || is_dense(jv));
      kfast = jk < nsteps && (kdn || is_fast(jk, kp0, kp1));
      vfast = jv < nsteps && (vdn || is_fast(jv, vp0, vp1));
    }
    int vis[RG];
#pragma unroll
    for (int r = 0; r < RG; ++r) vis[r] = seen(r, st + 1);
    const float sc = kMode == kLast ? 0.f : score_scale(st + 1);
    constexpr int kFirst = NCH >= 8 ? 2 : 1;  // the chunks before it cover the last QK MFMAs
#pragma unroll
    for (int c = 0; c < NCH; ++c) {
      const int m = c / RG, r = c % RG;
      if constexpr (kMode == kFast) {
        if (c < NC) {
          if constexpr (vdense) copy_dense_k(c, jk); else copy_k(c, jk, pgk.x, pgk.y);
        } else if (c < 2 * NC) {
          if constexpr (vdense) copy_dense_v(c - NC, jv); else copy_v(c - NC, jv, pgv.x, pgv.y);
        }
      } else if constexpr (kMode == kAny) {
        if (c < NC) {
          if (kfast) {
            if (kdn) copy_dense_k(c, jk); else copy_k(c, jk, kp0, kp1);
          }
        } else if (c < 2 * NC) {
          if (vfast) {
            if (vdn) copy_dense_v(c - NC, jv); else copy_v(c - NC, jv, vp0, vp1);
          }
        }
      }
      acc_mma_at<DT, !F8>(r * DT32 + m % DT32, va[m], pp[r][m / DT32]);
      if (c == 0) {
#pragma unroll
        for (int q = (NCH - 1) * kPairs / NCH; q < kPairs; ++q) {
          pair_pack(q);
          if (q < kSumA) pair_sum(q);
        }
      }
      if constexpr (RG == 2) {  // before chunk kFirst + (NCH - kFirst) / 2
#pragma unroll
        for (int q = c * 8 / (NCH / 2); q < (c + 1) * 8 / (NCH / 2); ++q)
          if (q < 8) pair_sum(8 + q);
      }
      if constexpr (kMode != kLast) {
        // (all in the first chunks, so they have landed by the next barrier)
        if (c < (F8 ? KS / 2 : KS)) ka[c] = F8 ? read_k8(st + 2, c) : read_k(st + 2, c);
        if (c >= kFirst) {
          constexpr int kTot = 16 * RG, kN = NCH - kFirst;
#pragma unroll
          for (int x = (c - kFirst) * kTot / kN; x < (c - kFirst + 1) * kTot / kN; ++x) {
            const int rr = x / 16, xx = x % 16;
            float v = fmaf(s_next[rr][xx], sc, mb[rr]);
            if (kMode == kAny) v = place(xx) < vis[rr] ? v : -INFINITY;
            e_cur[rr][xx] = v;
            bm[rr] = fmaxf(bm[rr], v);
          }
        }
      }
      sched_fence();
    }
    if constexpr (kMmaSum) {
      // The step's exp-sums, the probabilities' registers being free now: the
      // 16-lane groups of the two k-steps are exchanged so that one operand holds
      // all of M-rows 0 .. 15 and the other of 16 .. 31, each four k-groups of a
      // column of its own.  (Without the exchange a column would hold two rows,
      // kept apart by zeros, and a NaN in one would reach the other.)
#pragma unroll
      for (int r = 0; r < RG; ++r) {
        u32x4 lo = pp[r][0], hi = pp[r][1];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const auto t = __builtin_amdgcn_permlane16_swap(lo[i], hi[i], false, false);
          lo[i] = t[0];
          hi[i] = t[1];
        }
        constexpr u32x4 ones = {Dt<DT>::kOnes, Dt<DT>::kOnes, Dt<DT>::kOnes, Dt<DT>::kOnes};
        const f32x4 none = {0.f, 0.f, 0.f, 0.f};
        step_lo[r] = Dt<DT>::mma16x16x32(ones, lo, none)[0];
        step_hi[r] = Dt<DT>::mma16x16x32(ones, hi, none)[0];
      }
    }
    if constexpr (kMode == kLast) {
      acc_settle();
    } else {
      // the running max of a row moves only when a score passes it by more
      // than the headroom (rescaling the row's O and exp-sum)
      float big = bm[0];
#pragma unroll
      for (int r = 1; r < RG; ++r) big = fmaxf(big, bm[r]);
      if (__ballot(big > kLazyRescale)) {
        acc_settle();
        float scale[RG];
#pragma unroll
        for (int r = 0; r < RG; ++r) {
          const bool moves = max_xor32(bm[r]) > kLazyRescale;
          // (a row that moves has a score above -inf)
          const float m_new = moves ? -step_max(r, st + 1, kMode == kAny, s_next[r], sc) : mb[r];
          scale[r] = __builtin_amdgcn_exp2f(m_new - mb[r]);
          mb[r] = m_new;
          exponents(r, st + 1, kMode == kAny, s_next[r], sc);
        }
        take_sums();
#pragma unroll
        for (int r = 0; r < RG; ++r) l_run[r] *= scale[r];
        static_for<RG * DT32 * 16>([&](auto x) {
          constexpr int X = decltype(x)::value;
          acc_put<X>(acc_get<X>() * scale[X / (DT32 * 16)]);
        });
        acc_settle();
      }
      if constexpr (kMode == kAny) {
        if (const int chunk = pid_chunk_to_stage(st, TPP, n_pid)) stage_pids(chunk);
        if (jv < nsteps) {
          if (jk < nsteps && !kfast) slow_k(jk, kp0, kp1);
          if (!vfast) slow_v(jv, vp0, vp1);
        }
      }
    }
  };
  using Fast = std::integral_constant<int, kFast>;
  using Any = std::integral_constant<int, kAny>;
  using Last = std::integral_constant<int, kLast>;
  constexpr std::true_type yes{};
  constexpr std::false_type no{};
  // Iterations [0, n_main) need no mask in their next step (every row sees all
  // its keys).  In prompt mode steps from fd = ceil(hist / 32) on are dense
  // (the one across the boundary, if any, is not).  The fast body runs where
  // the K and V steps it copies are whole steps of one kind: pages, up to the
  // next iteration that stages a page-id chunk (an Any iteration), or dense
  // rows.
  const int n_main = min(nsteps - 1, min_lim / kKeys - 1);
  const int fd = PROMPT && !long_rows ? min(nsteps, static_cast<int>((hist + kKeys - 1) / kKeys)) : nsteps;
  int st = 0;
  int staged_at = -2;  // the iteration that staged page ids last (its flag is read two iterations later)
  while (st < min(nsteps - 1, fd)) {
    const int chunk_st = pid_next_staging(st, TPP);
    const int fast_end = min(min(n_main, paged_full - kLeadK), chunk_st);
    if (st < fast_end && st >= staged_at + 2 && __builtin_amdgcn_readfirstlane(lim_lds[kBad]) == 0) {
      for (; st < fast_end; ++st) step(Fast{}, no, st);
    } else {
      if (st == chunk_st) staged_at = st;
      step(Any{}, no, st);
      ++st;
    }
  }
  if constexpr (PROMPT) {
    const int fast_end = min(n_main, max_lim / kKeys - kLeadK);
    for (; st < fast_end; ++st) step(Fast{}, yes, st);
    for (; st < nsteps - 1; ++st) step(Any{}, yes, st);
  }
  if (nsteps > 0) {
    if (PROMPT && st >= fd)
      step(Last{}, yes, st);
    else
      step(Last{}, no, st);
  }

  if (claim && claim->wanted) claim->ask(p);  // the workgroup's next item, on its way while this tile is written
  // ---- normalise and write: lane holds O[M-row col][32n + 8(x/4) + 4 half + x%4].
  // A store straight from the accumulators would write 16 bytes of each of 32
  // rows per instruction; the rows go through the step buffers instead (a
  // region per row group, 16-byte chunk c of row i at chunk c ^ i, so that both
  // sides spread over the banks) and out as whole rows, 16 bytes per lane,
  // non-temporally (nothing here reads them again).
  take_sums();
  if (nsteps == 0) {
    acc_zero();
    acc_settle();
  }
  __syncthreads();  // every wavefront has read the last step
  constexpr int kCh = HD / 8;  // 16-byte chunks of a row
  auto place_chunk = [](int row, int c) { return (kCh & (kCh - 1)) == 0 ? c ^ (row & (kCh - 1)) : (c + row) % kCh; };
  static_for<RG>([&](auto rc) {
    constexpr int r = decltype(rc)::value;
    uint16_t* region = k_lds_base + (w * RG + r) * 32 * HD;  // K buffers, then V buffers: 8 regions of 32 rows
    float l;
    if constexpr (kMmaSum) l = l_run[r];
    else l = sum_xor32(l_run[r]);
    const float inv = l > 0.f ? 1.f / l : 0.f;
    static_for<DT32 * 4>([&](auto qc) {
      constexpr int c = decltype(qc)::value, n = c / 4, q4 = c % 4;
      constexpr int x = (r * DT32 + n) * 16 + 4 * q4;
      const u32x2 pk = {Dt<DT>::pack2(acc_get<x>() * inv, acc_get<x + 1>() * inv),
                        Dt<DT>::pack2(acc_get<x + 2>() * inv, acc_get<x + 3>() * inv)};
      *reinterpret_cast<u32x2*>(region + col * HD + place_chunk(col, c) * 8 + 4 * half) = pk;
    });
  });
  uint16_t* out_tile = p.out + (static_cast<int64_t>(row0) * p.num_q_heads + kvh * p.group + h0) * HD;
  compiler_fence();
  __builtin_amdgcn_s_waitcnt(kLgkmZero);  // a wavefront reads only what it wrote
  compiler_fence();
#pragma unroll
  for (int r = 0; r < RG; ++r) {
    const uint16_t* region = k_lds_base + (w * RG + r) * 32 * HD;
#pragma unroll
    for (int it = 0; it < kCh / 2; ++it) {
      const int i = it * kWave + lane;
      const int row = i / kCh, c = i % kCh;
      const int m = (w * RG + r) * 32 + row;
      const int t = static_cast<int>((static_cast<uint32_t>(m) * p.hg_magic) >> 16);
      const int h = m - t * p.hg_max;
      const u32x4 val = *reinterpret_cast<const u32x4*>(region + row * HD + place_chunk(row, c) * 8);
      if (t < nrows && t < qt && h < hg)
        __builtin_nontemporal_store(
            val, reinterpret_cast<u32x4_align8*>(out_tile + (static_cast<int64_t>(t) * p.num_q_heads + h) * HD + c * 8));
    }
  }
}

// LDS of a prefill workgroup: four K and four V step buffers, the target of
// padding copies, two chunks of page ids, the tokens' key limits (with their
// largest and smallest per wavefront) and the runs of a window.
template <int HD, bool KV8, int RG>
struct PrefillLds {
  __attribute__((aligned(16))) uint16_t k[kNBuf * StepGeo<HD>::kItems * 8];
  __attribute__((aligned(16))) uint16_t v[kNBuf * StepGeo<HD>::kItems * 8];
  __attribute__((aligned(16))) uint16_t junk[kWave * 8];
  uint32_t pid[2 * kPidChunk];
  float scl[KV8 ? 4 * kPidChunk : 1];  // fp8 pools: K then V scale of each staged page id
  int lim[m_rows(RG) + 2 * kPfWaves + 1];
  uint32_t seq[m_rows(RG)];               // window: the rows' sequences and key limits
  int32_t off[m_rows(RG)];
  uint64_t start[m_rows(RG) / kWave];     // window: rows that start a run, rows alone in their run
  uint64_t lone[m_rows(RG) / kWave];
  uint32_t next[2];                       // the claimed item (or none left), the queue it came from
};

// Window mode: one row of an item's window per thread (its sequence, those of
// the rows beside it, its key limit).
struct RowMap {
  uint32_t cur, prev, next;
  int32_t off;
};
template <int RG>
__device__ __forceinline__ RowMap load_row_map(const PrefillParams& p, unsigned item) {
  RowMap m{0u, 0u, 0u, 0};
  const unsigned G = static_cast<unsigned>(p.num_kv_heads) * p.head_chunks;
  const int unit = static_cast<int>(item / G);
  const int qt = m_rows(RG) / p.hg_max;
  const int64_t r = static_cast<int64_t>(p.num_units - 1 - unit) * qt + threadIdx.x;
  if (unit < p.num_units && static_cast<int>(threadIdx.x) < qt && r < p.num_rows) {
    m.cur = p.q2seq[r];
    m.prev = r > 0 ? p.q2seq[r - 1] : 0u;
    m.next = r + 1 < p.num_rows ? p.q2seq[r + 1] : 0u;
    m.off = p.q_offset[r];
  }
  return m;
}

// Work item `item` of the prefill: head group g = item % G (G = kv heads x
// head chunks) and work unit item / G, so that items 8 apart -- workgroups of
// one XCD -- take the same few kv heads and a kv head's K/V stay in few L2s.
//  * prompt mode: unit = (sequence, tile), the last tile of a sequence first
//    (it has the most keys);
//  * window mode (fused op): unit = window of `tokens per tile` rows, the
//    last window first (rows of a sequence usually come in position order,
//    so its later windows see more keys); every run of rows of one sequence
//    inside the window that is not a lone decode row (served by the decode
//    workers) is computed as a tile.
template <int DT, int HD, int TPP, bool KV8, int RG, bool kPromptMode>
__device__ __forceinline__ void prefill_item(const PrefillParams& p, unsigned item, Claim& claim,
                                             PrefillLds<HD, KV8, RG>& L) {
  const int G = p.num_kv_heads * p.head_chunks;
  const int g = static_cast<int>(item % static_cast<unsigned>(G));
  const int unit = static_cast<int>(item / static_cast<unsigned>(G));
  const int kvh = g / p.head_chunks;
  const int h0 = (g % p.head_chunks) * 16;
  const int qt = m_rows(RG) / p.hg_max;
  if constexpr (kPromptMode) {
    const int tps = (p.prompt_len + qt - 1) / qt;
    const int s = unit / tps;
    const int j = tps - 1 - (unit - s * tps);
    const int row0 = s * p.prompt_len + j * qt;
    prefill_tile<DT, HD, TPP, true, KV8, RG>(p, row0, min(qt, p.prompt_len - j * qt), s, kvh, h0, L.k, L.v, L.junk, L.pid,
                                             L.lim, L.scl, nullptr, nullptr);
  } else {
    const int w0 = (p.num_units - 1 - unit) * qt;
    const int n = static_cast<int>(min(static_cast<int64_t>(qt), p.num_rows - w0));
    constexpr int kMasks = m_rows(RG) / kWave;
    const RowMap rm = load_row_map<RG>(p, item);
    __syncthreads();  // the previous item is done with the run masks
    if (wave_id() < kMasks) {  // a wavefront per 64 rows of the window
      const int i = wave_id() * kWave + lane_id();
      const bool in = i < n;
      const bool head = in && (w0 + i == 0 || rm.prev != rm.cur);  // starts a run of its sequence's rows
      const bool tail = in && (w0 + i + 1 == p.num_rows || rm.next != rm.cur);
      L.seq[i] = rm.cur;
      L.off[i] = rm.off;
      const uint64_t st = __ballot(in && (i == 0 || head));
      const uint64_t lo = __ballot(head && tail);
      if (lane_id() == 0) {
        L.start[wave_id()] = st;
        L.lone[wave_id()] = lo;
      }
    }
    __syncthreads();
    auto uniform64 = [](uint64_t v) {
      return (static_cast<uint64_t>(__builtin_amdgcn_readfirstlane(static_cast<uint32_t>(v >> 32))) << 32) |
             static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(static_cast<uint32_t>(v)));
    };
    int cur = 0;
    while (cur < n) {
      // the next run's start, from the masks' bits past cur
      int end = n;
      const int from = cur + 1;
      for (int i = from / kWave; i < kMasks; ++i) {
        uint64_t m = uniform64(L.start[i]);
        if (i == from / kWave) m &= ~0ull << (from % kWave);
        if (m) {
          end = min(n, i * kWave + __builtin_ctzll(m));
          break;
        }
      }
      const bool lone = (uniform64(L.lone[cur / kWave]) >> (cur % kWave)) & 1;
      if (!lone)
        prefill_tile<DT, HD, TPP, false, KV8, RG>(p, w0 + cur, end - cur, L.seq[cur], kvh, h0, L.k, L.v, L.junk, L.pid,
                                                  L.lim, L.scl, L.off + cur, end == n ? &claim : nullptr);
      cur = end;
    }
  }
}

// The prefill's items on a resident grid, one workgroup per CU: a workgroup
// that starts on a CU pays several us before its first load (tiles take 30 to 60).
//  * Window mode: items are claimed, the first by place (workgroup b starts on
//    item b).  Lengths differ by item, and a static share left CUs idle for up
//    to a fifth of the time (16 sequences of 512 to 2,048 rows on 0 to 2,048
//    cached keys).
//  * Prompt mode (no workspace to hold counters): workgroup b of nb takes items
//    b, nb + b', 2 nb + b, ... (b' = the mirrored place among the workgroups of
//    b's XCD, so that a pass over ever shorter items evens out the previous one).
template <int DT, int HD, int TPP, bool KV8, int RG, bool kPromptMode>
__device__ __forceinline__ void prefill_items(const PrefillParams& p, unsigned b, unsigned nb,
                                              PrefillLds<HD, KV8, RG>& L) {
  const unsigned items = static_cast<unsigned>(p.num_units) * p.num_kv_heads * p.head_chunks;
  Claim claim{b % kQueues, 0u, items > nb, false, false};
  if constexpr (kPromptMode) {
    const unsigned mirrored = nb % 8 == 0 ? nb - 8 - (b & ~7u) + (b & 7u) : b;
    for (unsigned pass = 0; pass * nb < items; ++pass) {
      const unsigned item = pass * nb + ((pass & 1) ? mirrored : b);
      if (item < items) prefill_item<DT, HD, TPP, KV8, RG, true>(p, item, claim, L);
    }
  } else {
    // queue q: items q, q + 8, ...; its first ceil((nb - q) / 8) are taken by place
    auto item_of = [&](uint32_t q, uint32_t n) { return q + kQueues * (n + (nb + kQueues - 1 - q) / kQueues); };
    unsigned item = b;
    while (item < items) {
      claim.asked = false;
      prefill_item<DT, HD, TPP, KV8, RG, false>(p, item, claim, L);
      if (!claim.wanted) return;
      if (!claim.asked) claim.ask(p);
      if (threadIdx.x == 0) {
        uint32_t q = claim.queue;
        unsigned next = item_of(q, claim.got);
        for (int k = 1; k < kQueues && next >= items; ++k) {  // that queue is empty: the next one with an item
          q = (q + 1) % kQueues;
          next = item_of(q, claim.take(p, q));
        }
        L.next[0] = next;
        L.next[1] = q;
      }
      __syncthreads();
      item = __builtin_amdgcn_readfirstlane(L.next[0]);
      claim.queue = __builtin_amdgcn_readfirstlane(L.next[1]);
    }
  }
}

}  // namespace
}  // namespace pal
