// Which positions a decode step's kernels take: the rules of torch's indexing, in plain C++ so that the host
// can check them too. The kernels end the launch at an index outside its tensor, as torch's own index kernel
// does on the device: nothing is read or written there, and the caller's process learns of it.
#pragma once

#include <cstdint>

#if defined(__HIPCC__)
#define SKV_HOST_DEVICE __host__ __device__
#else
#define SKV_HOST_DEVICE
#endif

namespace starkv {

// Index i into `size` entries: a negative one counts from the end. False outside them.
SKV_HOST_DEVICE inline bool wrap_index(int64_t& i, int64_t size) {
    if (i < 0) i += size;
    return i >= 0 && i < size;
}

// Position pos as (entry `block` of a block-table row of `width`, offset `in` into the block), both by
// floor division. False for a block outside the row.
SKV_HOST_DEVICE inline bool split_position(int64_t pos, int64_t block_size, int64_t width, int64_t& block, int64_t& in) {
    block = pos / block_size;
    in = pos % block_size;
    if (in < 0) {
        in += block_size;
        --block;
    }
    return wrap_index(block, width);
}

}  // namespace starkv
