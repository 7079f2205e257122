// 3x3 convolutions at stride 1 taken directly on the FP16 MFMA (conv3.hip)
// where that is faster than Winograd's four launches.  Strides in elements.
#pragma once

#include <hip/hip_runtime.h>
#include <stddef.h>
#include <stdint.h>

#include "winograd.h"

namespace sdhip {

// Whether the convolution `a` (F(4x4)'s arguments) has a shape taken directly,
// whether it is (its output not over its inputs), its work buffer -- the
// weights once over -- and its launches.
bool conv3_shape(const WinogradArgs &a);
bool conv3_taken(const WinogradArgs &a);
size_t conv3_work_size(const WinogradArgs &a);
sdhip_status conv3(const WinogradArgs &a, void *work, hipStream_t stream);

}  // namespace sdhip
