// The token a frame's decision key stands for, in the joint scan and the
// decoders.  A key is {order-preserving score bits, 0xffff - id, duration and
// tag}; a NaN score makes no key.  constexpr, so that it is the same function
// on the host and on the device.
#pragma once

#include <cstdint>

namespace pk {

// `low` is the key's lower word (0xffff - id in its upper half).  An empty key
// (every token score of the frame NaN: an infinite encoder feature against
// weights of 0 gives that) is token 0, what pk_joint_gemv decides for such a
// frame; read as an id it would be 65535, past the embedding and the table.
constexpr int key_token(uint32_t low) { return (low >> 16) == 0 ? 0 : (int)(0xffffu - (low >> 16)); }

}  // namespace pk
