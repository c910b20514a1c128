// Instantiates the NTT pass shapes beyond the planner's static choice for
// u64 words, lazy reduction with headroom (2^33 <= q < 2^60).
#include "ntt_kernels.hpp"

namespace cbw {
namespace ntt_detail {
void register_alt_u64_headroom() { add_alt_u64<kHeadroom>(); }
}  // namespace ntt_detail
}  // namespace cbw
