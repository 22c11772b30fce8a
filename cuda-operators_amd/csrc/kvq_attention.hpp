// kvq_attention.hpp -- what the dense-attention kernels share.
#pragma once

#include <limits.h>
#include <math.h>

#include "kvq_device.hpp"
#include "kvq_internal.hpp"

namespace kvq {

typedef float f32x4 __attribute__((ext_vector_type(4)));

}  // namespace kvq
