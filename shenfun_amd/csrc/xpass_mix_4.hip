#include "xpass_mix.h"

namespace sfa {

int xpass_mix_4(const XMixArgs& a, int64_t nb, hipStream_t s) { return xpass_mix_run<4>(a, nb, s); }

}  // namespace sfa
