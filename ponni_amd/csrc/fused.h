// FUSED path: per-plan generated kernels compiled with hipRTC (fused.cpp).
#pragma once

#include <string>
#include <vector>

#include "plan.h"

namespace ponni_hip {

// Packed parameter blocks up to this size are staged in LDS by the kernel.
constexpr int64_t kFusedLdsParamBytes = 64 * 1024;
// LDS of one workgroup on gfx950.
constexpr int kFusedLdsBytes = 160 * 1024;
// CUs of an MI355X: workgroups i, i + kChipCus, ... of a launch share one.
constexpr int kChipCus = 256;

struct FusedConfig {
  int lds_bytes = 0;          // 0: parameters stream from L2
  int vec_bytes = 0;          // LDS copy of the per-feature vectors (0: none)
  int waves = 4;              // waves per workgroup
  int waves_per_simd = 2;     // occupancy the kernel is compiled for
  bool params_in_registers = false;  // parameters loaded once per wave, kept in VGPRs
  bool saved_in_lds = false;         // Save_State slots kept in LDS, not registers
  // 16-bit plans: every A fragment stays in LDS.  In: where that is possible
  // (the kernels that forward passes run; kernel sources handed out keep the
  // staged form); out: that it is.
  bool resident = false;
  bool by_wave = false;  // persistent kernels: tiles go to waves, not to workgroups
  bool persistent_loop = false;      // staged 16-bit plans: one workgroup per CU loops over tiles
  int columns_per_block = 128;
  int lds_total = 0;                 // bytes of LDS the kernel declares
  // The small-batch kernel (fused_split.h): a workgroup's waves share one
  // tile of columns and split each contraction's output tiles.
  bool split = false;
  bool any_rows = false;     // 16-bit: input rows at any alignment through LDS
  bool rows_in_lds = false;  // input rows go through LDS a tile ahead
  bool io32 = false;  // a 16-bit plan's kernel on fp32 input and output rows
  int split_waves = 8, split_nt = 1, split_wps = 2;
  std::string suffix() const { return std::string(io32 ? "_io32" : "") + (split ? "_split" : any_rows ? "_any" : ""); }
};

// Widest state a FUSED kernel of this dtype keeps on chip.
int fused_max_width(int dtype);
bool fused_supports(ponni_plan_s const& p);
// Can the NARROW plan run as a generated kernel (narrow_jit.h)?
bool narrow_jit_supports(ponni_plan_s const& p);
std::string fused_kernel_name(ponni_plan_s const& p);
std::string fused_source(ponni_plan_s const& p, FusedConfig& cfg);
// Compile (or fetch from cache) the plan's main kernel, a 16-bit plan's with
// resident fragments if asked and possible; needs no device.  The first call
// settles the kernel's occupancy (ponni_plan_s::fused_wps, resident_wps).
int fused_compile(ponni_plan_s& p, bool resident, std::string& key, std::vector<char>& code, std::string& error);
// Compile if needed one of the plan's kernels (ponni_plan_s::kernels) and load
// it on the current device; the main one first.
int fused_prepare(ponni_plan_s& p, bool io32, FusedForm form, std::string& error);
// The form of the plan's kernel that a call runs on once it is loaded (the
// main one takes any call).
FusedForm fused_wanted_form(ponni_plan_s const& p, void const* x, int64_t ld_in, int64_t batch, bool io32);
// The form that such a call runs on (rows that start on multiples of
// row_alignment bytes), compiling what that depends on; needs no device.
int fused_call_form(ponni_plan_s& p, int64_t batch, int row_alignment, bool io32, FusedForm& form, std::string& error);
hipError_t fused_launch(ponni_plan_s const& p, LaunchArgs const& a, bool io32, hipStream_t stream);

}  // namespace ponni_hip
