// Entry of the library for its own registration module, beside the public C ABI.
#pragma once
#include "flash_hypercons.h"

// fh_hc_mix (grad null; out = Y, aux = exp(H) or null) and fh_hc_mix_backward
// (out = dX, aux = dE or null) over rows in whole dwords at any dword, where the
// public entries take whole 16-byte vectors only.
extern "C" FH_API int fh_hc_mix_dwords(const void* h, const int64_t h_strides[3], int h_neg, const void* x,
                                       const int64_t x_strides[3], const void* grad, const int64_t* grad_strides,
                                       void* dh, void* out, float* aux, int dtype, int64_t batch, int n, int64_t cols,
                                       hipStream_t stream);
