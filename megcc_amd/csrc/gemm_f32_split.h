// f32 products of many output tiles on the bf16 matrix instructions (gemm_f32_split.hip).
#pragma once
#include "gevm_f32.h"
#include "megcc_gfx950.h"

namespace mg {

bool gemm_f32_split_supported(const GevmArgs& v);
TinyNNStatus gemm_f32_split_launch(const GevmArgs& v, int ta, int tb);

}  // namespace mg
