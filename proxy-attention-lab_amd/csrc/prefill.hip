// Paged causal attention for query tiles on gfx950 MFMA: the prefill kernel
// (the reference's uniform-prompt signature) and the prefill half of the
// fused mixed batch.  The tile code and its design notes are in
// prefill_tile.h.
//
// Reference behaviour: kernels/paged_attention/prefill/paged_attention_prefill.h.metal
// (history + causal prompt keys :147-234, :251-360; scores scaled after the
// dot product :178, :302; output rows (token, head) :379-381).
#include "pal_device.h"

namespace pal {

// flag word of this translation unit's debug checks (see pal_device.h)
PAL_DEBUG_FLAGS_DEFINE(prefill_debug_flags)

}  // namespace pal

#include "prefill_tile.h"

namespace pal {

namespace {

// One resident workgroup per CU, one wavefront per SIMD (the work mapping is
// in prefill_items).
template <int DT, int HD, int TPP, bool KV8, int RG, bool kPromptMode>
__global__ __launch_bounds__(kPfThreads) PAL_ACC_KERNEL void prefill_tile_kernel(const PrefillParams p) {
  __shared__ PrefillLds<HD, KV8, RG> lds;
  prefill_items<DT, HD, TPP, KV8, RG, kPromptMode>(p, blockIdx.x, gridDim.x, lds);
}

hipError_t device_cus(int* cus) {
  int dev = 0;
  const hipError_t err = hipGetDevice(&dev);
  return err != hipSuccess ? err : hipDeviceGetAttribute(cus, hipDeviceAttributeMultiprocessorCount, dev);
}

template <int DT, int HD, int TPP, bool KV8>
hipError_t launch_prefill_t(const PrefillParams& p, hipStream_t stream) {
  const int64_t items = static_cast<int64_t>(p.num_units) * p.num_kv_heads * p.head_chunks;
  int cus = 0;
  const hipError_t err = device_cus(&cus);
  if (err != hipSuccess) return err;
  const dim3 grid(static_cast<unsigned>(items < cus ? items : cus));
  if (p.prompt_len > 0) {
    if constexpr (HD <= 128) {
      if (p.row_groups == 2) {
        hipLaunchKernelGGL((prefill_tile_kernel<DT, HD, TPP, KV8, 2, true>), grid, dim3(kPfThreads), 0, stream, p);
        return hipGetLastError();
      }
    }
    hipLaunchKernelGGL((prefill_tile_kernel<DT, HD, TPP, KV8, 1, true>), grid, dim3(kPfThreads), 0, stream, p);
    return hipGetLastError();
  }
  // windows: the head dims that the fused kernels do not take (launch_fused)
  if constexpr (HD > 128 && TPP != 0) {
    hipLaunchKernelGGL((prefill_tile_kernel<DT, HD, TPP, KV8, 1, false>), grid, dim3(kPfThreads), 0, stream, p);
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

// Tiles run one per CU, in rounds over the CUs.  A tile of two row groups
// holds twice the rows and takes 1.65 times as long (16 sequences of 1,280
// rows on 1,024 cached, bf16, head dim 128: 0.62 ms in 10 rounds against 0.73
// ms in 20; one prompt of 768 rows, one round either way: 27.7 against 19.9 us).
// Head dims above 128 have one: their accumulators fill the registers.
hipError_t prefill_choose_tiles(PrefillParams& p, int head_dim) {
  p.row_groups = 1;
  if (head_dim > 128) return hipSuccess;
  int cus = 0;
  const hipError_t err = device_cus(&cus);
  if (err != hipSuccess) return err;
  const int64_t qt = 2 * prefill_tokens_per_tile(p.group);
  const int64_t units_2 = p.prompt_len > 0 ? p.num_seqs * ((p.prompt_len + qt - 1) / qt) : (p.num_rows + qt - 1) / qt;
  const int64_t heads = static_cast<int64_t>(p.num_kv_heads) * p.head_chunks;
  const int64_t rounds_1 = (p.num_units * heads + cus - 1) / cus, rounds_2 = (units_2 * heads + cus - 1) / cus;
  if (3 * rounds_1 < 5 * rounds_2) return hipSuccess;
  p.row_groups = 2;
  p.num_units = static_cast<int>(units_2);
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
