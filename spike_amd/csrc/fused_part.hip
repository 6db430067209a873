// fused_part.hip -- one part of the persistent kernels' instances (SPK_FUSED_PART 0..5: the
// synapse kind PART / 2 with one label (even) or several (odd); 6: the compact forms).
#include "fused.hpp"
#include "fused_table.hpp"

#ifndef SPK_FUSED_PART
#error "SPK_FUSED_PART selects the instances of this translation unit"
#endif

namespace spk {

template <int KIND, bool L1>
FusedKernels instances() {
  FusedKernels k;
  k.run = (const void*)k_fused<KIND, L1, kRulesOff>;
  k.run_plastic = (const void*)k_fused<KIND, L1, kRulesDense>;
  k.run_events = (const void*)k_fused<KIND, L1, kRulesEvents>;
  k.run_delayed = (const void*)k_fused<KIND, L1, kRulesDelayed>;
  k.batch = (const void*)k_fused_batch<KIND, L1, kRulesOff, kFusedBlock>;
  k.batch_small = (const void*)k_fused_batch<KIND, L1, kRulesOff, kBatchSmallBlock>;
  return k;
}

#if SPK_FUSED_PART == 0
FusedKernels fused_kernels_k0l1() { return instances<0, true>(); }
#elif SPK_FUSED_PART == 1
FusedKernels fused_kernels_k0ln() { return instances<0, false>(); }
#elif SPK_FUSED_PART == 2
FusedKernels fused_kernels_k1l1() { return instances<1, true>(); }
#elif SPK_FUSED_PART == 3
FusedKernels fused_kernels_k1ln() { return instances<1, false>(); }
#elif SPK_FUSED_PART == 4
FusedKernels fused_kernels_k2l1() { return instances<2, true>(); }
#elif SPK_FUSED_PART == 5
FusedKernels fused_kernels_k2ln() { return instances<2, false>(); }
#else
const void* fused_kernel_lds_table() { return (const void*)k_fused<0, true, kRulesOff, kDeliverLdsTable>; }
const void* fused_kernel_compact() { return (const void*)k_fused<0, true, kRulesOff, kDeliverCompact>; }
const void* batch_kernel_compact(bool small, bool tables) {
  if (small) return (const void*)k_fused_batch<0, true, kRulesOff, kBatchSmallBlock, kDeliverCompact>;   // (no tables)
  return tables ? (const void*)k_fused_batch<0, true, kRulesOff, kFusedBlock, kDeliverCompactAny>
                : (const void*)k_fused_batch<0, true, kRulesOff, kFusedBlock, kDeliverCompact>;
}
#endif

}  // namespace spk
