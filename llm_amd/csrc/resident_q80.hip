// The many-token product with resident activations for one weight type.
#include "resident.h"

namespace llmhip {
template int resident_launch_qt<LLMHIP_Q8_0>(const GemvArgs&, const ResArgs&, const ResPlan&, int, int, hipStream_t);
template int resident_ready_qt<LLMHIP_Q8_0>();
}  // namespace llmhip
