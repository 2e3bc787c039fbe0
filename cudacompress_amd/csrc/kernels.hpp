// Internal launch interface of the gfx950 kernels (namespace cca).  Every launcher checks its
// arguments on the host before launching and throws cca::Error on failure.
#pragma once

#include "common.hpp"
#include "profile.hpp"

namespace cca {

// ---- DWT (src/cudaCompress/util/DWTFloat.cu, DWTInt.cu) -------------------------------------
// one 9/7 analysis level in FP64 (no reference counterpart; measures the FP32 transform's error)
void dwt97_forward_f64(double* dst, double* buf, const double* src, int sx, int sy, int sz, int row, int slice,
                       hipStream_t st);
void dwt97_forward(float* dst, float* buf2, float* buf1, const float* src, int sx, int sy, int sz, int srcCh,
                   int dRow, int dSlice, int sRow, int sSlice, hipStream_t st);
void dwt97_inverse(float* dst, float* buf2, float* buf1, const float* src, int sx, int sy, int sz, int dstCh,
                   int dRow, int dSlice, int sRow, int sSlice, hipStream_t st);
void dwt97_inverse_from_symbols(float* dst, float* buf2, float* buf1, const float* lowpass,
                                const void* const* dd_highpass, int symbolSize, float step, int sx, int sy, int sz,
                                int dstCh, int dRow, int dSlice, int lpRow, int lpSlice, hipStream_t st);
void dwt97_forward_from_byte(float* dst, float* buf2, float* buf1, const uint8_t* src, int sx, int sy, int sz,
                             int srcCh, int dRow, int dSlice, int sRow, int sSlice, hipStream_t st);
void dwt97_inverse_to_byte(uint8_t* dst, float* buf2, float* buf1, const float* src, int sx, int sy, int sz, int dstCh,
                           int dRow, int dSlice, int sRow, int sSlice, hipStream_t st);
void dwt97_inverse_from_symbols_to_byte(uint8_t* dst, float* buf2, float* buf1, const float* lowpass,
                                        const void* const* dd_highpass, float step, int sx, int sy, int sz, int dstCh,
                                        int dRow, int dSlice, int lpRow, int lpSlice, hipStream_t st);
void dwt97_forward_lowpass_only_from_byte(float* dst, float* buf, const uint8_t* src, int sx, int sy, int srcCh,
                                          int dRow, int sRow, hipStream_t st);
void dwt53_forward(int16_t* dst, int16_t* buf, const int16_t* src, int sx, int sy, int sz, int dRow, int dSlice,
                   int sRow, int sSlice, hipStream_t st);
void dwt53_forward_lowpass_only(int16_t* dst, int16_t* buf, const int16_t* src, int sx, int sy, int dRow, int sRow,
                                hipStream_t st);
void dwt53_inverse(int16_t* dst, int16_t* buf, const int16_t* src, int sx, int sy, int sz, int dRow, int dSlice,
                   int sRow, int sSlice, hipStream_t st);

// ---- quantization (src/cudaCompress/util/Quantize.cu) ---------------------------------------
void symbolize(uint16_t* sym, const int16_t* data, uint32_t sx, uint32_t sy, uint32_t sz, uint32_t row,
               uint32_t slice, hipStream_t st);
void unsymbolize(int16_t* data, const uint16_t* sym, uint32_t sx, uint32_t sy, uint32_t sz, uint32_t row,
                 uint32_t slice, hipStream_t st);
void quantize_to_symbols(void* sym, int symSize, float* data, bool roundtrip, uint32_t sx, uint32_t sy, uint32_t sz,
                         float step, uint32_t row, uint32_t slice, int qtype, hipStream_t st);
void unquantize_from_symbols(float* data, const void* sym, int symSize, uint32_t sx, uint32_t sy, uint32_t sz,
                             float step, uint32_t row, uint32_t slice, int qtype, hipStream_t st);
void quantize_to_short(int16_t* q, const float* data, uint32_t sx, uint32_t sy, uint32_t sz, float step,
                       uint32_t row, uint32_t slice, int qtype, hipStream_t st);
void unquantize_from_short(float* data, const int16_t* q, uint32_t sx, uint32_t sy, uint32_t sz, float step,
                           uint32_t row, uint32_t slice, int qtype, hipStream_t st);
void max_abs(const float* data, uint32_t n, float* out, hipStream_t st);

// ---- image path and bit planes (src/cudaCompress/util/Quantize.cu, YCoCg.cu, Bits.cu) ---------
void float_to_byte_2d(uint8_t* out, uint32_t channelCount, uint32_t channel, const float* data, uint32_t sx,
                      uint32_t sy, uint32_t row, hipStream_t st);
void byte_to_float_2d(float* data, const uint8_t* in, uint32_t channelCount, uint32_t channel, uint32_t sx,
                      uint32_t sy, uint32_t row, hipStream_t st);
void quantize_difference_2d(uint16_t* sym, float* data, float step, const uint8_t* ref, uint32_t channelCount,
                            uint32_t channel, uint32_t sx, uint32_t sy, uint32_t row, int qtype, bool roundtrip,
                            hipStream_t st);
void unquantize_difference_2d(float* data, const uint16_t* sym, float step, const uint8_t* ref, uint32_t channelCount,
                              uint32_t channel, uint32_t sx, uint32_t sy, uint32_t row, int qtype, hipStream_t st);
// One level's coefficients (lx x ly x lz from data, row and slice pitches; lz 1: 2D) as symbols: the
// highpass octants (quadrants) b = bx + 2 by (+ 4 bz) >= 1 to dense bands hp + (b - 1) band_stride, the
// lowpass one to low_sym as symbols, or to low as values, or (both null) nowhere; and back (with both
// null the lowpass octant of data stays as it is).
void symbolize_level(uint16_t* hp, uint64_t band_stride, uint16_t* low_sym, int16_t* low, const int16_t* data,
                     uint32_t lx, uint32_t ly, uint32_t lz, uint32_t row, uint64_t slice, hipStream_t st);
void unsymbolize_level(int16_t* data, const uint16_t* hp, uint64_t band_stride, const uint16_t* low_sym,
                       const int16_t* low, uint32_t lx, uint32_t ly, uint32_t lz, uint32_t row, uint64_t slice,
                       hipStream_t st);
void convert_ycocg(uint8_t* out, const uint8_t* in, uint32_t pixels, int channels, bool to_ycocg, hipStream_t st);
void lsb_get(const int16_t* data, uint32_t* bits, uint32_t n, hipStream_t st);
void lsb_remove(int16_t* data, uint32_t* bits, uint32_t n, int16_t shift, hipStream_t st);
void lsb_append(int16_t* data, const uint32_t* bits, uint32_t n, int16_t shift, hipStream_t st);
void shift_elems(int16_t* data, uint32_t n, int16_t shift, hipStream_t st);

}  // namespace cca
