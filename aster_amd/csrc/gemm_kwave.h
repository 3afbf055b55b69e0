// K split over the waves of a workgroup (gemm_kwave_kernel.hpp): which shape a problem takes, its launch
// and its description.
#pragma once
#include "astergemm_internal.h"

namespace astergemm {

struct KwaveForm {
  int shape = -1;  // -1: the problem stays with the other kernels
  int per = 0;     // weight rows of a workgroup
  int ranges = 1;  // K ranges
  bool k8 = false; // weights (MXFP4: and both scale planes) in the order of ASTERGEMM_OPERAND_DIRECT_B_K8
  explicit operator bool() const { return shape >= 0; }
};

// M <= 64, as part of the decode kernels' launchers (`dt` operands, `cus` = compute units, 0 = no device;
// at most `max_ranges` K ranges, what the launcher states as its workspace).
KwaveForm kwave_decode_form(int dt, int64_t M, int64_t N, int64_t K, int cus, int max_ranges);
// M <= 64 on rows the kernels with resident activations do not take, without dynamic LDS past the default
// limit (the launcher it is part of sets no function attribute).
KwaveForm kwave_small_decode_form(int dt, int64_t M, int64_t N, int64_t K, int cus);

// 64 < M <= 512 against at most about a round of panels, as part of the launchers of 128 x 128 tiles.
KwaveForm kwave_prompt_form(int dt, int64_t M, int64_t N, int64_t K, int cus);
// M <= 512 on pre-shuffled weights (*rows: the operand rows of a workgroup), as part of the launchers of 128 x 256
// tiles that load them straight into MFMA operands.
KwaveForm kwave_k8_form(int dt, int64_t M, int64_t N, int cus, int* rows);
// Any M and N: the smallest tile that leaves at most one workgroup per CU, else (and without a device) 64 x 64.
KwaveForm kwave_tile_form(int64_t M, int64_t N, int cus);
// Small products that AUTO takes the tile form for, where it takes the general tile kernels otherwise.
bool kwave_small_product(int dt, int64_t M, int64_t N, int64_t K, int cus);
// What the variants of these kernels run, by AUTO or by name: the tile form for small products (split: never),
// else the decode form where there is one, else the prompt form, else the tile form.
KwaveForm kwave_variant_form(bool split, int dt, int64_t M, int64_t N, int64_t K, int cus);

int kwave_launch(int dt, int out, const GemmArgs& a, const KwaveForm& f, hipStream_t s);
// The one-time step of every shape of `dt` on the current device (see lds_attr_once).
int kwave_ready(int dt, bool k8 = false);
void kwave_describe(int dt, const KwaveForm& f, int64_t M, int64_t N, int cus, LaunchForm* o);
bool kwave_decode_describe(const astergemm_config& c, int cus, int max_ranges, LaunchForm* o);
bool kwave_prompt_describe(const astergemm_config& c, int cus, LaunchForm* o);
bool kwave_small_decode_describe(const astergemm_config& c, int cus, LaunchForm* o);

}  // namespace astergemm
