// Definitions of MixKernels<R>, instantiated once per precision.
#pragma once

#include <hip/hip_ext.h>

#include "sgpe_mixed.h"

namespace sgpe {

#define SGPE_MIX_LAUNCH(K, ...)                                               \
  do {                                                                        \
    if (e0)                                                                   \
      hipExtLaunchKernelGGL(K, g, b, (uint32_t)l, s, e0, e1, 0, __VA_ARGS__); \
    else                                                                      \
      hipLaunchKernelGGL(K, g, b, l, s, __VA_ARGS__);                         \
  } while (0)

template <typename R>
void MixKernels<R>::col(dim3 g, dim3 b, size_t l, hipStream_t s, hipEvent_t e0, hipEvent_t e1, const InstDev* i,
                        RunDev* r, const MixFft& f, const void* tw, int w, unsigned div_w, int mode, int dp, int dc) {
  SGPE_MIX_LAUNCH((mix_col_pass_kernel<R>), i, r, f, (const typename Cx<R>::T*)tw, w, div_w, mode, dp, dc);
}

template <typename R>
void MixKernels<R>::row(dim3 g, dim3 b, size_t l, hipStream_t s, hipEvent_t e0, hipEvent_t e1, const InstDev* i,
                        RunDev* r, const MixFft& f, const void* tw, int rows, unsigned div_n, int dur, int first,
                        int col_w, bool general) {
  const typename Cx<R>::T* t = (const typename Cx<R>::T*)tw;
  if (general)
    SGPE_MIX_LAUNCH((mix_row_pass_kernel<R, true>), i, r, f, t, rows, div_n, dur, first, col_w);
  else
    SGPE_MIX_LAUNCH((mix_row_pass_kernel<R, false>), i, r, f, t, rows, div_n, dur, first, col_w);
}

template <typename R>
void MixKernels<R>::fft(dim3 g, dim3 b, size_t l, hipStream_t s, FftPair io, const MixFft& f, const void* tw, int nx,
                        int batch, unsigned div_batch, bool rows, bool inv, double scale) {
  const hipEvent_t e0 = nullptr, e1 = nullptr;
  const typename Cx<R>::T* t = (const typename Cx<R>::T*)tw;
  if (rows && inv)
    SGPE_MIX_LAUNCH((mix_fft_kernel<R, true, true>), io, f, t, nx, batch, div_batch, scale);
  else if (rows)
    SGPE_MIX_LAUNCH((mix_fft_kernel<R, true, false>), io, f, t, nx, batch, div_batch, scale);
  else if (inv)
    SGPE_MIX_LAUNCH((mix_fft_kernel<R, false, true>), io, f, t, nx, batch, div_batch, scale);
  else
    SGPE_MIX_LAUNCH((mix_fft_kernel<R, false, false>), io, f, t, nx, batch, div_batch, scale);
}

template <typename R> const void* MixKernels<R>::kernel(int which) {
  switch (which) {
    case MIX_COL: return (const void*)&mix_col_pass_kernel<R>;
    case MIX_ROW: return (const void*)&mix_row_pass_kernel<R, false>;
    case MIX_ROW_GENERAL: return (const void*)&mix_row_pass_kernel<R, true>;
    case MIX_FFT_COLS: return (const void*)&mix_fft_kernel<R, false, false>;
    case MIX_FFT_COLS_INV: return (const void*)&mix_fft_kernel<R, false, true>;
    case MIX_FFT_ROWS: return (const void*)&mix_fft_kernel<R, true, false>;
    default: return (const void*)&mix_fft_kernel<R, true, true>;
  }
}

}  // namespace sgpe
