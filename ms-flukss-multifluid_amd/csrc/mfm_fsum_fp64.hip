// FP64 (parity) build of the face-sum kernels,
// -ffp-contract=off as mfm_kernels_fp64.hip: every product and sum rounds
// as in the reference.
#include "mfm_kernels.inc"
#include "mfm_fsum.inc"

namespace mfm {
template hipError_t launch_face_sums<double>(const Consts&, const Consts*, const DevPatch*,
                                            const StageLists&, const StepArgs&, hipStream_t,
                                            KernelTimer*);
}  // namespace mfm
