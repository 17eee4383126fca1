// Register-resident PCG kernels for any stateSize up to 32, double reference-recurrence
// instances (the kernel is in pcg_reg_impl.h).
#include "pcg_reg_impl.h"

namespace gbdpcg {

namespace {
template <int NT, int SET>
const void *ap() {
  return reinterpret_cast<const void *>(&pcg_any_kernel<double, NT, false, SET>);
}
}  // namespace

const void *any_ref_kernel_ptr_f64(int nt, int set) {
  if (nt == 64) return set == kAnyTiny ? ap<64, kAnyTiny>() : nullptr;
  if (nt == 512) return set == kAnyAll ? ap<512, kAnyAll>() : set == kAnyLong ? ap<512, kAnyLong>() : nullptr;
  if (nt != 256) return nullptr;
  switch (set) {
    case kAnyNarrow: return ap<256, kAnyNarrow>();
    case kAnyWide: return ap<256, kAnyWide>();
    case kAnyRows: return ap<256, kAnyRows>();
    default: return nullptr;
  }
}

}  // namespace gbdpcg
