// Image-size transforms as matrix products (lengths without a register transform).
#pragma once

#include "oi_internal.h"

namespace oi {

// Cosines and sines of a length's forward (order x folded sample) and inverse
// (folded position x order) sums; null: the length has a register transform.
struct DftTable {
  const float* fcos = nullptr;
  const float* fsin = nullptr;
  const float* icos = nullptr;
  const float* isin = nullptr;
  int frows = 0, fpitch = 0;
  int irows = 0, ipitch = 0, iodd = 0;   // iodd: where the odd orders start
};

struct FpArgs;

// A table for orders up to amax: its size, and its values from tw[m] =
// exp(-2 pi i m / n) (exact copies or halves, built on the stream).
size_t dft_table_bytes(int n, int amax);
int dft_table_build(const float2* tw, int n, int amax, float* mem, DftTable& t, hipStream_t st);

// The stage is the faster as a product (the general transforms take the others).
bool dft_rows_ok(const FpArgs& a);
bool dft_cols_ok(const FpArgs& a);
bool dft_ucols_ok(const FpArgs& a);

// The launches of the register-transform kernels of the same stage.
int dft_rows(const FpArgs& a, hipStream_t st);
int dft_cols(const FpArgs& a, hipStream_t st);
int dft_ucols(const FpArgs& a, hipStream_t st);
int dft_urows(const FpArgs& a, hipStream_t st);   // the image only

}  // namespace oi
