// pf_gemm8.hpp — the large-tile prefill GEMM kernels (pf_gemm8.hip), launched by launch_pf_gemm.
#pragma once

#include "prefill.hpp"

namespace fllm {

// a GEMM kernel, its LDS bytes, its tile (bm tokens x bn weight rows), its threads, and the time of one
// 256-element block of a full wave of its workgroups
typedef void (*PfGemmKernel)(const PfGemm);
struct PfKernel {
    PfGemmKernel k;
    size_t lds;
    int bm, bn, threads;
    double block_us;
};
// a launch's form: the type its tile-interleaved segments share, PF_FORM_MIX when they differ, or
// PF_FORM_ROWS + the type of GGUF rows (rows of whole 256-element blocks)
enum { PF_FORM_ROWS = 100, PF_FORM_MIX = 1000 };
// bm 64 or 128 (x 256 weight rows); .k null for a form without one
PfKernel pf_gemm8_kernel(int form, int bm);

}  // namespace fllm
