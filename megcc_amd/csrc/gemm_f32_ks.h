// f32 products of few output tiles (gemm_f32_ks.hip).
#pragma once
#include "conv_geom.h"
#include "gevm_f32.h"
#include "megcc_gfx950.h"

namespace mg {

// estimated cycles of the busiest CU
double gemm_f32_ks_cycles(const GevmArgs& v);
bool gemm_f32_ks_supported(const GevmArgs& v);
TinyNNStatus gemm_f32_ks_launch(const GevmArgs& v, int ta, int tb);
bool conv_f32_ks_supported(const ConvGeom& g);
TinyNNStatus conv_f32_ks_launch(const ConvGeom& g, const void* src, const void* flt, const void* bias, void* dst);

}  // namespace mg
