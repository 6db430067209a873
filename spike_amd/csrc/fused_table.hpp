// fused_table.hpp -- the instances of the persistent kernels by what a network needs.  They
// are compiled in several translation units (fused_part.hip, one part per synapse kind and
// label class, one for the compact forms), which the build runs side by side.
#pragma once

namespace spk {

struct FusedKernels {
  const void* run;            // k_fused, no plasticity
  const void* run_plastic;    // k_fused with plasticity, every rule per synapse
  const void* run_events;     // k_fused with one spike-driven weight-dependent rule
  const void* run_delayed;    // k_fused with one spike-driven Vogels, Evans or Custom rule
  const void* batch;          // k_fused_batch of kFusedBlock threads
  const void* batch_small;    // k_fused_batch of kBatchSmallBlock threads
};

// Instances of every delivery form, by synapse kind (0..2) and single label or not.
FusedKernels fused_kernels_k0l1();
FusedKernels fused_kernels_k0ln();
FusedKernels fused_kernels_k1l1();
FusedKernels fused_kernels_k1ln();
FusedKernels fused_kernels_k2l1();
FusedKernels fused_kernels_k2ln();
inline FusedKernels fused_kernels(int kind, bool l1) {
  if (kind == 0) return l1 ? fused_kernels_k0l1() : fused_kernels_k0ln();
  if (kind == 1) return l1 ? fused_kernels_k1l1() : fused_kernels_k1ln();
  return l1 ? fused_kernels_k2l1() : fused_kernels_k2ln();
}

// Instances that hold one compact delivery form (voltage synapses, one label).
const void* fused_kernel_lds_table();
const void* fused_kernel_compact();
const void* batch_kernel_compact(bool small, bool tables);

}  // namespace spk
