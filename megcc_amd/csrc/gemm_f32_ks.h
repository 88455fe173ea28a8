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

// 64 x 64 ... 256 tiles on the bf16 instructions, slices of K in the workspace where it has room for them (gemm_f32_ks_split.hip);
// false: not where this product is faster
bool gemm_f32_ks_split(const GevmArgs& v, int ta, int tb, const Workspace* ws, TinyNNStatus* status);
struct KpPlan {
    int kg, slices;  // groups of waves that share a stage of K; slices of K
    bool swap;       // the staged rows are B's (with four groups both operands have 64 rows: never)
};
// ... by that plan, whatever the choice would be; a workspace for the slices where there are several
TinyNNStatus gemm_f32_ks_split_launch(const GevmArgs& v, int ta, int tb, const KpPlan& p, const Workspace* ws);
// C = the sum of partial[slices][M][N], in order (gemm_f32.hip)
void gemm_f32_add_slices(const float* partial, int slices, int M, int N, float* C, long ldc);

// f32 convolutions of many pixels: a wave has its pixels for the whole of K (conv_f32_wide.hip)
bool conv_f32_wide_supported(const ConvGeom& g);
TinyNNStatus conv_f32_wide_launch(const ConvGeom& g, const void* src, const void* flt, const void* bias, void* dst);

}  // namespace mg
