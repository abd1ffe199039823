// Host-and-device arithmetic of the attention launches' plans (no HIP types).
#pragma once

#include <cstdint>

namespace hyperion::hip {

// First of `blocks` key blocks that split `split` of `splits` takes (split = splits: the end):
// blocks * split / splits, without the product, which passes 2^32 at 2^29 keys in 256 splits.
constexpr uint32_t split_first_block(uint32_t blocks, uint32_t split, uint32_t splits) {
    return blocks / splits * split + blocks % splits * split / splits;
}

}  // namespace hyperion::hip
