// Vector types of the fp32 MFMA kernels and the XCD count of gfx950: workgroup i of a 1-D
// grid is dispatched to XCD i % 8 and every XCD has its own L2, so the kernels give all
// tiles of one utterance (or of a part or a run of them) ids that land on one XCD (place_block in
// simple_logprobs.hip, find_tile in simple_normalizer.hip).
#pragma once

#include "common.hip.h"

namespace frnnt {
namespace dgemm {

constexpr int kXcds = 8;

typedef float floatx16 __attribute__((ext_vector_type(16)));  // a 32 x 32 MFMA accumulator
typedef float floatx4 __attribute__((ext_vector_type(4)));

}  // namespace dgemm
}  // namespace frnnt
