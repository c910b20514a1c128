// Instantiates the NTT pass kernels for u64 words, lazy reduction with headroom
// (2^33 <= q < 2^60), one-pass 2^13- and 2^14-point rows among them.
#include "ntt_kernels.hpp"

namespace cbw {
namespace ntt_detail {
void register_u64_headroom() {
    register_all<std::uint64_t, kHeadroom>();
    add_long_rows<std::uint64_t, kHeadroom>();
}
}  // namespace ntt_detail
}  // namespace cbw
