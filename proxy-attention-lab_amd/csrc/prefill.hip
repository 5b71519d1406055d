// Paged causal attention for query tiles on gfx950 MFMA: the prefill kernel
// (the reference's uniform-prompt signature) and the prefill half of the
// fused mixed batch.  The tile code and its design notes are in
// prefill_tile.h and prefill_half_tile.h.
//
// Reference behaviour: kernels/paged_attention/prefill/paged_attention_prefill.h.metal
// (history + causal prompt keys :147-234, :251-360; scores scaled after the
// dot product :178, :302; output rows (token, head) :379-381).
#include "pal_device.h"

namespace pal {

// flag word of this translation unit's debug checks (see pal_device.h)
PAL_DEBUG_FLAGS_DEFINE(prefill_debug_flags)

}  // namespace pal

#include "prefill_half_tile.h"  // half tiles (and prefill_tile.h)

namespace pal {

namespace {

// The prompts that whole tiles of rg row groups serve (measured in
// prefill_choose_tiles; tpp 0: a run-time page size).
constexpr bool wide_prompts(int hd, int tpp, bool kv8, int rg) {
  return hd <= 128 && tpp != 0 && !kv8 && (rg == 1 || hd < 128 || tpp == 16);
}

// One resident workgroup per CU, one wavefront per SIMD (the work mapping is
// in prefill_items).
template <int DT, int HD, int TPP, bool KV8, int RG, bool kPromptMode>
__global__ __launch_bounds__(kPfThreads) PAL_ACC_KERNEL void prefill_tile_kernel(const PrefillParams p) {
  __shared__ PrefillLds<HD, KV8, RG> lds;
  prefill_items<DT, HD, TPP, KV8, RG, kPromptMode>(p, blockIdx.x, gridDim.x, lds);
}

// Half tiles, a workgroup each: up to head dim 128 within half of the register
// file, two workgroups per CU, so that a tile's prologue, its register-path
// steps and its epilogue run beside another tile's products.
template <int DT, int HD, int TPP, bool KV8, bool kPromptMode>
__global__ __launch_bounds__(kPfThreads) __attribute__((amdgpu_waves_per_eu(HD <= 128 ? 2 : 1, HD <= 128 ? 2 : 1)))
void prefill_half_kernel(const PrefillParams p) {
  __shared__ HalfTileLds<HD, KV8> lds;
  half_tile_block<DT, HD, TPP, KV8, kPromptMode>(p, blockIdx.x, lds);
}

hipError_t device_cus(int* cus) {
  int dev = 0;
  const hipError_t err = hipGetDevice(&dev);
  return err != hipSuccess ? err : hipDeviceGetAttribute(cus, hipDeviceAttributeMultiprocessorCount, dev);
}

template <int DT, int HD, int TPP, bool KV8>
hipError_t launch_prefill_t(const PrefillParams& p, hipStream_t stream) {
  const int64_t items = static_cast<int64_t>(p.num_units) * p.num_kv_heads * p.head_chunks;
  const dim3 threads(kPfThreads);
  if (p.row_groups == 0) {
    const dim3 grid(static_cast<unsigned>(items));
    if (p.prompt_len > 0) {
      hipLaunchKernelGGL((prefill_half_kernel<DT, HD, TPP, KV8, true>), grid, threads, 0, stream, p);
      return hipGetLastError();
    }
    if constexpr (HD > 128 && TPP != 0 && !KV8) {
      hipLaunchKernelGGL((prefill_half_kernel<DT, HD, TPP, KV8, false>), grid, threads, 0, stream, p);
      return hipGetLastError();
    }
    return hipErrorInvalidValue;
  }
  int cus = 0;
  const hipError_t err = device_cus(&cus);
  if (err != hipSuccess) return err;
  const dim3 grid(static_cast<unsigned>(items < cus ? items : cus));
  if (p.prompt_len > 0) {
    if constexpr (wide_prompts(HD, TPP, KV8, 2)) {
      if (p.row_groups == 2) {
        hipLaunchKernelGGL((prefill_tile_kernel<DT, HD, TPP, KV8, 2, true>), grid, threads, 0, stream, p);
        return hipGetLastError();
      }
    }
    if constexpr (wide_prompts(HD, TPP, KV8, 1)) {
      if (p.row_groups == 1) {
        hipLaunchKernelGGL((prefill_tile_kernel<DT, HD, TPP, KV8, 1, true>), grid, threads, 0, stream, p);
        return hipGetLastError();
      }
    }
    return hipErrorInvalidValue;
  }
  // windows: the head dims that the fused kernels do not take (launch_fused)
  if constexpr (HD > 128 && TPP != 0) {
    hipLaunchKernelGGL((prefill_tile_kernel<DT, HD, TPP, KV8, 1, false>), grid, threads, 0, stream, p);
    return hipGetLastError();
  }
  return hipErrorInvalidValue;
}

// Page sizes 16 and 32 have their own kernels; other multiples of 8 (16-bit
// pools, uniform-prompt mode) run the kernel built for a run-time page size.
template <int DT, int HD, bool KV8>
hipError_t prefill_tpp(const PrefillParams& p, int tpp, hipStream_t stream) {
  switch (tpp) {
    case 16: return launch_prefill_t<DT, HD, 16, KV8>(p, stream);
    case 32: return launch_prefill_t<DT, HD, 32, KV8>(p, stream);
    default:
      if constexpr (!KV8) {
        if (tpp > 0 && tpp % 8 == 0 && p.prompt_len > 0) return launch_prefill_t<DT, HD, 0, false>(p, stream);
      }
      return hipErrorInvalidValue;
  }
}

template <int DT>
hipError_t prefill_hd(const PrefillParams& p, int hd, int tpp, hipStream_t stream) {
  if (p.k_scales) {  // fp8 pools: head dims of whole 16-dim stripes
    switch (hd) {
      case 64: return prefill_tpp<DT, 64, true>(p, tpp, stream);
      case 128: return prefill_tpp<DT, 128, true>(p, tpp, stream);
      case 256: return prefill_tpp<DT, 256, true>(p, tpp, stream);
      default: return hipErrorInvalidValue;
    }
  }
  switch (hd) {
    case 32: return prefill_tpp<DT, 32, false>(p, tpp, stream);
    case 64: return prefill_tpp<DT, 64, false>(p, tpp, stream);
    case 96: return prefill_tpp<DT, 96, false>(p, tpp, stream);
    case 128: return prefill_tpp<DT, 128, false>(p, tpp, stream);
    case 256: return prefill_tpp<DT, 256, false>(p, tpp, stream);
    default: return hipErrorInvalidValue;
  }
}

}  // namespace

int prefill_tokens_per_tile(int group) { return m_rows(1) / (group < 16 ? group : 16); }

// Half tiles (0), or tiles that have a CU to themselves, of one row group or two?
//
// The latter run one per CU, in rounds over the CUs.  A tile of two row groups
// holds twice the rows and takes 1.65 times as long (16 sequences of 1,280
// rows on 1,024 cached, bf16, head dim 128: 0.62 ms in 10 rounds against 0.73
// ms in 20; one prompt of 768 rows, one round either way: 27.7 against 19.9 us).
// Head dims above 128 have one: their accumulators fill the registers.
//
// Prompts, half -> whole tiles (us; 32 query heads on 8 kv heads, head dim 128,
// 16-token pages unless named):
//  * one round of one group: whole.  1 x 1,024 37 -> 25, 8 x 128 on 4,000 cached 128
//    -> 79.  Several rounds of one group: half, whose second workgroup per CU runs
//    beside a tile's prologue (32 kv heads, 64 x 64 on 50 cached: 1.36 times the
//    time; 16 heads on 2 of dim 64, 16 x 333 on 100 and 128 x 33 on 200 1.12 and 1.05).
//  * two groups, head dims up to 64: whole.  16 x 1,024: head dim 64 0.73, 32 0.72 of
//    the time; the worst of 30 shapes 0.97.
//  * two groups above: these kernels spill a little outside of the step loops,
//    and a static share of tiles that are not alike costs more than the tiles
//    gain.  Whole where tiles are full and a round is whole sequences or a
//    sequence whole rounds (16 x 1,024 234 -> 196), there is one sequence (group 7,
//    1 x 4,096 140 -> 120), or the page table has room for as many cached tokens
//    as new ones, which make the tiles alike (group 7, 32 x 128 on 2,000 168 -> 141);
//    else half (16 x 333 on 100 82 -> 86; group 7, 4 x 2,048 1.19, 32 x 512 1.06
//    times the time).  At head dim 128 over 32-token pages, with twice the spills,
//    half (0.91 to 1.34 times, 1.08 on average).
//  * fp8 pages and run-time page sizes, whose history goes through registers (1.04
//    to 1.57 times), and head dim 256, whose prompt kernels spilled 190 registers
//    (1.01 to 1.66 times): half.
// Windows (head dims up to 128: called for the whole tiles alone): whole, except
// for 16-bit pools above head dim 128, whose tiles pay for 100 spilled registers
// at their start and end.  There half where their keys are shared by several
// heads and contexts are at most 256 tokens, or tiles are many and contexts at
// most 512 tokens or most runs of rows smaller than a window (32 query heads on 8:
// 64 x 64 97 -> 111, 4 x 256 35 -> 38, 64 x 16 on 2,000 218 -> 242; but 16 x 64 on 1,000
// 70 -> 63, 1 x 512 43 -> 35; 8 on 8, 32 x 128 46 -> 43; 16 on 2, 64 x 16 on 2,000 102 ->
// 75; fp8, 64 x 64 97 -> 82).
hipError_t prefill_choose_tiles(PrefillParams& p, int head_dim) {
  int cus = 0;
  const hipError_t err = device_cus(&cus);
  if (err != hipSuccess) return err;
  const int64_t qt = 2 * prefill_tokens_per_tile(p.group);
  const int64_t seq_units_2 = (p.prompt_len + qt - 1) / qt;
  const int64_t units_2 = p.prompt_len > 0 ? p.num_seqs * seq_units_2 : (p.num_rows + qt - 1) / qt;
  const int64_t heads = static_cast<int64_t>(p.num_kv_heads) * p.head_chunks;
  const int64_t tiles_1 = p.num_units * heads;
  const int64_t rounds_1 = (tiles_1 + cus - 1) / cus, rounds_2 = (units_2 * heads + cus - 1) / cus;
  p.row_groups = head_dim <= 128 && 3 * rounds_1 >= 5 * rounds_2 ? 2 : 1;
  if (p.prompt_len > 0) {
    const int64_t seq_tiles = seq_units_2 * heads;
    const bool alike = 4 * p.prompt_len >= 3 * seq_units_2 * qt &&
                       (cus % seq_tiles == 0 || seq_tiles % cus == 0 || p.num_seqs == 1 ||
                        p.page_table_width * p.tokens_per_page >= p.prompt_len);
    if (!wide_prompts(head_dim, p.tokens_per_page == 16 || p.tokens_per_page == 32 ? p.tokens_per_page : 0,
                      p.k_scales != nullptr, p.row_groups) ||
        (p.row_groups == 1 ? rounds_1 > 1 : head_dim > 64 && !alike))
      p.row_groups = 0;
  } else if (head_dim > 128 && !p.k_scales && p.group > 1) {
    const int64_t keys = p.page_table_width * p.tokens_per_page;  // the longest context has no more
    const bool small_runs = 2 * p.num_rows < qt * p.num_seqs;
    if (keys <= 256 || (2 * tiles_1 > cus && (keys <= 512 || small_runs))) p.row_groups = 0;
  }
  if (p.row_groups == 2) p.num_units = static_cast<int>(units_2);
  return hipSuccess;
}

hipError_t launch_prefill(const PrefillParams& params, int dtype, int head_dim, int tokens_per_page,
                          hipStream_t stream) {
  if (params.num_units <= 0) return hipSuccess;
  PrefillParams p = params;
  const hipError_t err = prefill_choose_tiles(p, head_dim);
  if (err != hipSuccess) return err;
  if (dtype == kBF16) return prefill_hd<kBF16>(p, head_dim, tokens_per_page, stream);
  return prefill_hd<kF16>(p, head_dim, tokens_per_page, stream);
}

}  // namespace pal
