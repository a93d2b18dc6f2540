// The row-major side of a strip (32 rows x 512 bytes) whose rows start at any element and end anywhere, moved in aligned 16-byte
// chunks: a row of the strip covers up to 33 of them.  Loading keeps the chunks as they are in a row-major LDS image with a
// 33-chunk pitch and shifts when the image is read (five dwords and a funnel shift per chunk); storing shifts when it makes the
// aligned chunks.  Element accesses remain where a chunk crosses the end of the buffer (loads) or of a row (stores).
#pragma once
#include <type_traits>

#include "ttm_common.h"

constexpr int kRaggedPitch = 33;                        // chunks of an image row
constexpr int kRaggedImage = 32 * kRaggedPitch + 1;     // one more: the shift reads a dword ahead

template <int ELEM>
using ragged_elem = typename std::conditional<ELEM == 4, uint32_t, typename std::conditional<ELEM == 2, uint16_t, uint8_t>::type>::type;

// Strip `id` of a [rows, cols] matrix cut into `strips` per row of tiles.
struct RaggedStrip {
  int sx, ty, ct, yt;    // strip in the row, row of tiles; tile columns and rows of the matrix
  int nrows, nbytes;     // real rows; real bytes of a row segment
  int tiles;             // tiles of the strip (16 / ELEM of them, fewer at the end of a row)
  int64_t stride;        // bytes of a row
};
// Neighbouring strips share the lines at their common edge: consecutive ones go to one XCD (workgroups are dealt to the eight
// XCDs in turn), whose L2 then puts the two parts of a line together.
template <int ELEM>
__device__ __forceinline__ RaggedStrip ragged_strip(int rows, int cols, int strips) {
  const int n8 = gridDim.x >> 3, id = (int)blockIdx.x < n8 * 8 ? ((int)blockIdx.x & 7) * n8 + ((int)blockIdx.x >> 3) : (int)blockIdx.x;
  RaggedStrip s;
  s.sx = id % strips; s.ty = id / strips; s.ct = (cols + 31) >> 5; s.yt = (rows + 31) >> 5;
  s.nrows = min(32, rows - s.ty * 32);
  s.nbytes = min(512, (cols - s.sx * (512 / ELEM)) * ELEM);
  s.tiles = min(16 / ELEM, s.ct - s.sx * (16 / ELEM));
  s.stride = (int64_t)cols * ELEM;
  return s;
}

// 16 bytes of the image from byte `off` on
__device__ __forceinline__ u32x4 lds_unaligned16(const uint8_t *image, int off) {
  const uint32_t *w = (const uint32_t *)image + (off >> 2);
  const int sh = (off & 3) * 8;
  const uint32_t d0 = w[0], d1 = w[1], d2 = w[2], d3 = w[3], d4 = w[4];
  return u32x4{__builtin_amdgcn_alignbit(d1, d0, sh), __builtin_amdgcn_alignbit(d2, d1, sh), __builtin_amdgcn_alignbit(d3, d2, sh),
               __builtin_amdgcn_alignbit(d4, d3, sh)};
}

// chunk slot idx: row and number of the aligned chunk in the row; slots 1024 .. 1055 are the rows' 33rd chunks
__device__ __forceinline__ int ragged_row(int idx) { return idx < 1024 ? idx >> 5 : idx - 1024; }
__device__ __forceinline__ int ragged_chunk(int idx) { return idx < 1024 ? idx & 31 : 32; }

// The aligned chunks that cover the strip, whose first element is at address rm, into the image; [lo, hi) is the buffer.
template <int ELEM>
__device__ __forceinline__ void ragged_load(u32x4 *image, const RaggedStrip &s, uintptr_t rm, uintptr_t lo, uintptr_t hi) {
  typedef ragged_elem<ELEM> T;
  u32x4 v[5];
#pragma unroll
  for (int i = 0; i < 5; ++i) {
    const int idx = i * 256 + (int)threadIdx.x, r = ragged_row(idx);
    if (idx >= 1056 || r >= s.nrows) continue;
    const uintptr_t a = rm + r * s.stride, c = (a & ~(uintptr_t)15) + ragged_chunk(idx) * 16;
    if (c >= a + s.nbytes) continue;
    if (c >= lo && c + 16 <= hi) {
      v[i] = __builtin_nontemporal_load((const u32x4 *)c);
    } else {
      T e[16 / ELEM];
#pragma unroll
      for (int k = 0; k < 16 / ELEM; ++k) e[k] = c + k * ELEM >= lo && c + k * ELEM < hi ? *(const T *)(c + k * ELEM) : T(0);
      v[i] = *(const u32x4 *)e;
    }
  }
#pragma unroll
  for (int i = 0; i < 5; ++i) {
    const int idx = i * 256 + (int)threadIdx.x;
    if (idx < 1056) image[ragged_row(idx) * kRaggedPitch + ragged_chunk(idx)] = v[i];
  }
}
// 16 bytes of the strip's row r from byte column `at` on, zeros outside the matrix
__device__ __forceinline__ u32x4 ragged_read(const u32x4 *image, const RaggedStrip &s, uintptr_t rm, int r, int at) {
  u32x4 o = lds_unaligned16((const uint8_t *)image, r * kRaggedPitch * 16 + (int)((rm + r * s.stride) & 15) + at);
  const int n = r < s.nrows ? s.nbytes - at : 0;   // real bytes of the chunk
  if (n < 16) {
#pragma unroll
    for (int k = 0; k < 4; ++k) o[k] = n >= 4 * k + 4 ? o[k] : n <= 4 * k ? 0u : o[k] & ((1u << (8 * (n - 4 * k))) - 1u);
  }
  return o;
}

// A strip stores the aligned chunks that begin in it: the last one of a row reaches into the next strip, whose first 16 bytes of
// every row (a face row or a part of one) are the image's 33rd chunk.
__device__ __forceinline__ int ragged_left(const RaggedStrip &s) { return (int)min(s.stride - (int64_t)s.sx * 512, (int64_t)1024); }   // bytes of a row from the strip on
template <int ELEM>
__device__ __forceinline__ void ragged_store(const u32x4 *image, const RaggedStrip &s, uintptr_t rm) {
  typedef ragged_elem<ELEM> T;
  const uint8_t *bytes = (const uint8_t *)image;
  const int left = ragged_left(s);
#pragma unroll
  for (int i = 0; i < 5; ++i) {
    const int idx = i * 256 + (int)threadIdx.x, r = ragged_row(idx);
    if (idx >= 1056 || r >= s.nrows || (i == 4 && s.sx > 0)) continue;   // i = 4: the piece in front of the first whole chunk of a row
    const uintptr_t a = rm + r * s.stride;
    const int head = (int)(-a & 15), at = i == 4 ? head - 16 : head + ragged_chunk(idx) * 16;   // byte column of the chunk in the strip
    if (at >= s.nbytes) continue;
    if (at >= 0 && at + 16 <= left) {
      *(u32x4 *)(a + at) = lds_unaligned16(bytes, r * kRaggedPitch * 16 + at);
    } else {   // the ends of a row
#pragma unroll
      for (int k = 0; k < 16 / ELEM; ++k)
        if (at + k * ELEM >= 0 && at + k * ELEM < left) *(T *)(a + at + k * ELEM) = *(const T *)(bytes + r * kRaggedPitch * 16 + at + k * ELEM);
    }
  }
}
