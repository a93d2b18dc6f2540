// bfp8_b / bfp4_b block-float pack and unpack.
//
// Format (per 32x32 tile, faces in order (0,0) (0,1) (1,0) (1,1), 16 rows x 16 columns each):
//   bytes [0,64)   one shared exponent per 16-element face row: the largest biased fp32 exponent
//   bfp8_b         1024 mantissa bytes, sign<<7 | 7-bit magnitude
//   bfp4_b         512 mantissa bytes, two elements per byte, even column in the low nibble,
//                  nibble = sign<<3 | 3-bit magnitude
// Encode: hidden bit added, shifted right by (shared - own exponent), rounded to nearest even to
// the kept width, saturated; a magnitude of 0 drops the sign.  Decode: mag * 2^(E-127-(W-1)).
//
// Work split: a lane owns one 16-byte chunk of the plain side (4 fp32 or 8 bf16 elements of one
// face row), so a face row is a quad (fp32) or a pair (bf16) of adjacent lanes and the shared
// exponent is a max-reduction with DPP quad_perm moves.  A 256-lane workgroup owns 1024 chunks:
// on a row-major plain side that is a strip of 32 rows x 512 bytes which is read / written in
// fully contiguous 512-byte row segments and permuted through a padded LDS image, exactly like
// the tilize kernel; the packed side of a strip is one contiguous run of tiles.
// Row-major shapes whose rows are not a multiple of 512 bytes, or that need zero padding, are moved chunk by chunk at any
// address without LDS, large ones and those of host memory by strips that start anywhere; tile-ordered tensors that are no whole number of strips take a generic kernel with one face row quad
// per lane group and bounds-checked scalar accesses.
#include <type_traits>

#include "ttm_common.h"
#include "ttm_ragged.h"

// ------------------------------------------------------------------------------------ element math
// W = magnitude bits (7 or 3).  Returns the magnitude only; signs are merged per chunk.
template <int W>
__device__ __forceinline__ uint32_t bfp_mag(uint32_t bits, uint32_t E) {
  constexpr int DROP = 24 - W;
  uint32_t a = bits & 0x7FFFFFFFu;
  uint32_t e = a >> 23;
  uint32_t shift = min(E - e, 31u);
  uint32_t m = (a & 0x7FFFFFu) | (min(a, 1u) << 23);  // hidden bit unless the value is +-0
  m >>= shift;
  m += ((1u << (DROP - 1)) - 1) + ((m >> DROP) & 1u);  // round to nearest, ties to even
  return min(m >> DROP, (1u << W) - 1);
}

template <int W>
__device__ __forceinline__ uint32_t bfp_encode(uint32_t bits, uint32_t E) {
  uint32_t k = bfp_mag<W>(bits, E);
  return k ? (k | ((bits >> 31) << W)) : 0u;
}

template <int W>
__device__ __forceinline__ float bfp_decode(uint32_t mag, uint32_t signbit_at31, int E) {
  // mag * 2^(E - 127 - (W-1)), exact (subnormal results included); the sign is dropped at 0
  float v = ldexpf((float)mag, E - 127 - (W - 1));
  return mag ? __uint_as_float(__float_as_uint(v) | (signbit_at31 & 0x80000000u)) : 0.0f;
}

template <int LANES>
__device__ __forceinline__ uint32_t group_max(uint32_t v) {
  uint32_t o = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0xB1, 0xF, 0xF, true);  // quad_perm [1,0,3,2]
  v = max(v, o);
  if (LANES == 4) {
    o = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x4E, 0xF, 0xF, true);  // quad_perm [2,3,0,1]
    v = max(v, o);
  }
  return v;
}

// Encode one chunk of EPT elements (bit patterns of fp32 values) of a face row.
// out[] receives EPT*(W+1)/32 packed words (bfp8: EPT/4 words, bfp4: EPT/8 words, or a half word).
template <int W, int EPT>
__device__ __forceinline__ uint32_t encode_chunk(const uint32_t (&bits)[EPT], uint32_t (&out)[2]) {
  uint32_t E = 0;
#pragma unroll
  for (int i = 0; i < EPT; ++i) E = max(E, (bits[i] >> 23) & 0xFFu);
  E = group_max<16 / EPT>(E);
  out[0] = out[1] = 0;
  if (W == 7) {
#pragma unroll
    for (int w = 0; w < EPT / 4; ++w) {
      uint32_t k0 = bfp_mag<7>(bits[4 * w + 0], E), k1 = bfp_mag<7>(bits[4 * w + 1], E);
      uint32_t k2 = bfp_mag<7>(bits[4 * w + 2], E), k3 = bfp_mag<7>(bits[4 * w + 3], E);
      uint32_t mags = k0 | (k1 << 8) | (k2 << 16) | (k3 << 24);
      uint32_t nz = (mags + 0x7F7F7F7Fu) & 0x80808080u;  // 0x80 in every byte whose magnitude is non-zero
      uint32_t top = __builtin_amdgcn_perm(bits[4 * w + 1], bits[4 * w + 0], 0x0C0C0703u) |
                     __builtin_amdgcn_perm(bits[4 * w + 3], bits[4 * w + 2], 0x07030C0Cu);  // the four sign bytes
      out[w] = mags | (top & nz);
    }
  } else {
    uint32_t word = 0;
#pragma unroll
    for (int i = 0; i < EPT; ++i) word |= bfp_encode<3>(bits[i], E) << (4 * i);
    out[0] = word;
  }
  return E;
}

// The same for eight bf16 values, two per operation in 16-bit halves: the 8 significant bits stand at bit 7 of a half, so an
// alignment shift up to 7 loses nothing, and from 8 on both kept widths round to 0 whatever is lost.  Against the fp32 form, which
// bounded the bf16 packs: [8192, 8192] bfp8_b 41.2 -> 37.0 us, bfp4_b 42.8 -> 35.5.
typedef uint16_t u16x2 __attribute__((ext_vector_type(2)));
template <int W>
__device__ __forceinline__ uint32_t encode_bf16_chunk(const u32x4 &v, uint32_t (&out)[2]) {
  u16x2 a[4], top = {0, 0};
  uint32_t mags[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const uint32_t x = v[i] & 0x7FFF7FFFu;
    a[i] = *(const u16x2 *)&x;
    top = __builtin_elementwise_max(top, a[i]);
  }
  const uint32_t E = group_max<2>((uint32_t)(top.x > top.y ? top.x : top.y) >> 7);
  const u16x2 Ev = {(uint16_t)E, (uint16_t)E}, one = {1, 1};
  constexpr uint16_t DROP = 15 - W;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    u16x2 m = ((a[i] << 7) & (u16x2){0x3F80, 0x3F80}) | (__builtin_elementwise_min(a[i], one) << 14);   // hidden bit unless the value is +-0
    m >>= __builtin_elementwise_min((u16x2)(Ev - (a[i] >> 7)), (u16x2){15, 15});
    m += ((m >> DROP) & one) + (uint16_t)((1 << (DROP - 1)) - 1);   // round to nearest, ties to even
    m = __builtin_elementwise_min((u16x2)(m >> DROP), (u16x2){(1 << W) - 1, (1 << W) - 1});
    if (W == 3) {
      const uint32_t x = v[i];
      m |= (*(const u16x2 *)&x >> 12) & (__builtin_elementwise_min(m, one) << 3);
    }
    mags[i] = *(const uint32_t *)&m;
  }
  if (W == 7) {
#pragma unroll
    for (int w = 0; w < 2; ++w) {
      const uint32_t k = __builtin_amdgcn_perm(mags[2 * w + 1], mags[2 * w], 0x06040200u);
      const uint32_t sign = __builtin_amdgcn_perm(v[2 * w + 1], v[2 * w], 0x07050301u);
      out[w] = k | (sign & (k + 0x7F7F7F7Fu) & 0x80808080u);   // 0x80 in every byte whose magnitude is non-zero
    }
  } else {
#pragma unroll
    for (int i = 0; i < 4; ++i) mags[i] |= mags[i] >> 12;   // low byte: even column low, odd column high
    out[0] = __builtin_amdgcn_perm(mags[1], mags[0], 0x0C0C0400u) | __builtin_amdgcn_perm(mags[3], mags[2], 0x04000C0Cu);
    out[1] = 0;
  }
  return E;
}

// One chunk of the plain side
template <int W, int ELEM>
__device__ __forceinline__ uint32_t encode_plain(const u32x4 &v, uint32_t (&out)[2]) {
  if constexpr (ELEM == 2) {
    return encode_bf16_chunk<W>(v, out);
  } else {
    const uint32_t bits[4] = {v.x, v.y, v.z, v.w};
    return encode_chunk<W, 4>(bits, out);
  }
}

// Decode EPT elements from packed words into one 16-byte chunk of the plain side.
template <int W, bool BF16, int EPT>
__device__ __forceinline__ u32x4 decode_chunk(const uint32_t (&in)[2], int E) {
  float f[EPT];
  if (W == 7) {
#pragma unroll
    for (int i = 0; i < EPT; ++i) {
      uint32_t word = in[i / 4];
      int b = i & 3;
      f[i] = bfp_decode<7>((word >> (8 * b)) & 0x7Fu, word << (24 - 8 * b), E);
    }
  } else {
#pragma unroll
    for (int i = 0; i < EPT; ++i) f[i] = bfp_decode<3>((in[0] >> (4 * i)) & 0x7u, in[0] << (28 - 4 * i), E);
  }
  u32x4 v;
  if (BF16) {  // exact: a decoded value has at most 7 significant bits
#pragma unroll
    for (int i = 0; i < 4; ++i) v[i] = (__float_as_uint(f[2 * i]) >> 16) | (__float_as_uint(f[2 * i + 1]) & 0xFFFF0000u);
  } else {
#pragma unroll
    for (int i = 0; i < 4; ++i) v[i] = __float_as_uint(f[i]);
  }
  return v;
}

// ------------------------------------------------------------------------------------ strip kernels
// ELEM = bytes per plain element (4: fp32, 2: bf16).  A tile is CPT = 64*ELEM chunks; a face row is
// ELEM chunks.  The workgroup handles 1024 chunks = 16/ELEM tiles.
// Packing bfp8_b from row-major fp32 gains from four workgroups per CU (8192 x 8192: 53.2 -> 50.9 us); every other
// combination is fastest without a cap.
template <int W, int ELEM, bool ROWMAJOR, bool PACK>
__global__ __launch_bounds__(256) TTM_MAX_WAVES((PACK && ROWMAJOR && W == 7 && ELEM == 4) ? 4 : 8) void ttm_bfp_strip_k(const void *__restrict__ src_, void *__restrict__ dst_,
                                                       int64_t xt, int64_t strips_per_row) {
  constexpr int EPT = 16 / ELEM;
  constexpr int CPT = 64 * ELEM;
  constexpr int TILE_BYTES = 64 + (W == 7 ? 1024 : 512);
  constexpr int CHUNK_OUT = EPT * (W + 1) / 8;  // packed bytes per chunk: 4, 8 (bfp8) or 2, 4 (bfp4)
  constexpr int PITCH = 33;
  __shared__ u32x4 lds[ROWMAJOR ? 32 * PITCH : 1];
  // PACK to bfp4_b: the workgroup's 16 / ELEM packed tiles are contiguous in the output; they are assembled here (exponent
  // bytes and 2- or 4-byte mantissa pieces per lane) and leave as 16-byte stores (8192 x 8192 fp32: 51 -> 46 us; bfp8_b with
  // its 4- and 8-byte pieces is faster storing them directly: 53 against 55 us)
  constexpr int PK_BYTES = (16 / ELEM) * TILE_BYTES;
  constexpr bool VIA_LDS = PACK && W == 3;
  __shared__ __attribute__((aligned(16))) uint8_t pk[VIA_LDS ? PK_BYTES : 16];
  const int tid = threadIdx.x;
  const int64_t strip = blockIdx.x;
  const int64_t tyb = ROWMAJOR ? strip / strips_per_row : 0;
  const int64_t sx = ROWMAJOR ? strip % strips_per_row : 0;
  const int64_t row_chunks = xt * 2 * ELEM;
  // first tile of this workgroup on the packed / tile-ordered side
  const int64_t tile0 = ROWMAJOR ? (tyb * xt + sx * (16 / ELEM)) : strip * (16 / ELEM);
  const u32x4 *plain_in = (const u32x4 *)src_;
  u32x4 *plain_out = (u32x4 *)dst_;
  const uint8_t *packed_in = (const uint8_t *)src_;
  uint8_t *packed_out = (uint8_t *)dst_;
  const int64_t rm_base = tyb * 32 * row_chunks + sx * 32;

  u32x4 v[4];
  if (PACK) {
    if (ROWMAJOR) {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        int r = i * 8 + (tid >> 5), j = tid & 31;
        v[i] = __builtin_nontemporal_load(&plain_in[rm_base + r * row_chunks + j]);
      }
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        int r = i * 8 + (tid >> 5), j = tid & 31;
        lds[r * PITCH + j] = v[i];
      }
      __syncthreads();
    } else {
#pragma unroll
      for (int i = 0; i < 4; ++i) v[i] = __builtin_nontemporal_load(&plain_in[tile0 * CPT + i * 256 + tid]);
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      int oc = i * 256 + tid;
      int tl = oc / CPT, w = oc % CPT;
      int face = w / (16 * ELEM), dy = (w / ELEM) % 16, q = w % ELEM;
      if (ROWMAJOR) {
        int r = (face >> 1) * 16 + dy, j = tl * 2 * ELEM + (face & 1) * ELEM + q;
        v[i] = lds[r * PITCH + j];
      }
      uint32_t out[2];
      const uint32_t E = encode_plain<W, ELEM>(v[i], out);
      if constexpr (VIA_LDS) {
        uint8_t *tile = pk + tl * TILE_BYTES;
        if (q == 0) tile[face * 16 + dy] = (uint8_t)E;
        uint8_t *m = tile + 64 + w * CHUNK_OUT;
        if (CHUNK_OUT == 4) *(uint32_t *)m = out[0];
        else *(uint16_t *)m = (uint16_t)out[0];
      } else {
        uint8_t *tile = packed_out + (tile0 + tl) * TILE_BYTES;
        if (q == 0) tile[face * 16 + dy] = (uint8_t)E;
        uint8_t *m = tile + 64 + w * CHUNK_OUT;
        if (CHUNK_OUT == 8) {
          u32x2 o = {out[0], out[1]};
          __builtin_nontemporal_store(o, (u32x2 *)m);
        } else {
          __builtin_nontemporal_store(out[0], (uint32_t *)m);
        }
      }
    }
    if constexpr (VIA_LDS) {
      __syncthreads();
      u32x4 *dst16 = (u32x4 *)(packed_out + tile0 * TILE_BYTES);   // tile sizes are multiples of 16 bytes
      for (int c = tid; c < PK_BYTES / 16; c += 256) __builtin_nontemporal_store(((const u32x4 *)pk)[c], &dst16[c]);
    }
  } else {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      int oc = i * 256 + tid;
      int tl = oc / CPT, w = oc % CPT;
      int face = w / (16 * ELEM), dy = (w / ELEM) % 16;
      const uint8_t *tile = packed_in + (tile0 + tl) * TILE_BYTES;
      int E = tile[face * 16 + dy];
      const uint8_t *m = tile + 64 + w * CHUNK_OUT;
      uint32_t in[2] = {0, 0};
      if (CHUNK_OUT == 8) {
        u32x2 t = __builtin_nontemporal_load((const u32x2 *)m);
        in[0] = t.x; in[1] = t.y;
      } else if (CHUNK_OUT == 4) {
        in[0] = __builtin_nontemporal_load((const uint32_t *)m);
      } else {
        in[0] = __builtin_nontemporal_load((const uint16_t *)m);
      }
      v[i] = decode_chunk<W, ELEM == 2, EPT>(in, E);
    }
    if (ROWMAJOR) {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        int oc = i * 256 + tid;
        int tl = oc / CPT, w = oc % CPT;
        int face = w / (16 * ELEM), dy = (w / ELEM) % 16, q = w % ELEM;
        int r = (face >> 1) * 16 + dy, j = tl * 2 * ELEM + (face & 1) * ELEM + q;
        lds[r * PITCH + j] = v[i];
      }
      __syncthreads();
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        int r = i * 8 + (tid >> 5), j = tid & 31;
        __builtin_nontemporal_store(lds[r * PITCH + j], &plain_out[rm_base + r * row_chunks + j]);
      }
    } else {
#pragma unroll
      for (int i = 0; i < 4; ++i) __builtin_nontemporal_store(v[i], &plain_out[tile0 * CPT + i * 256 + tid]);
    }
  }
}

// ------------------------------------------------------------------------------------ ragged shapes
// A lane owns a chunk, a wavefront 8 rows x 8 chunks (narrower tensors: more rows): 128 bytes of a row, which starts at any element
// (16-byte accesses at its own alignment; the chunk that crosses the end of a row takes elements), against 8 face rows of packed
// mantissas, the whole or half of a 128-byte line.  U chunks per lane: two for packing beyond 16 MiB, whose loads are the larger
// side, else one.  HBM-bound; bf16 packs also by the encoding.  Neighbouring
// workgroups go to one XCD (25.3 / 18.4 -> 19.0 / 18.1 us for the first figure below).  Against strips through LDS with funnel shifts
// and, below 2304 tiles, a workgroup per tile with element accesses, pack / unpack: [4096, 8190] bf16 bfp8_b 25.2 / 24.5 -> 19.0 / 18.1
// us (5.7 TB/s), [3, 1966, 1888] fp32 bfp4_b 13.4 / 16.8 -> 12.9 / 12.2, [2, 700, 1500] bf16 bfp8_b 6.0 / 5.8 -> 3.5 / 3.5,
// [1024, 1056] fp32 4.2 / 4.6 -> 2.9 / 3.1.
template <int W, int ELEM, int U, bool PACK>
__global__ __launch_bounds__(256) void ttm_bfp_direct_k(const uint8_t *__restrict__ src, uint8_t *__restrict__ dst, int rows, int cols, int lw, int wc,
                                                        uint32_t xu, uint32_t matrices, uint32_t first, uint32_t groups) {
  typedef typename std::conditional<ELEM == 4, uint32_t, uint16_t>::type T;
  constexpr int EPT = 16 / ELEM, TILE_BYTES = 64 + (W == 7 ? 1024 : 512), CHUNK_OUT = EPT * (W + 1) / 8;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int ct = (cols + 31) >> 5, yt = (rows + 31) >> 5;
  const uint32_t bid = first + xcd_order(groups), by = bid / xu;
  const int chunk = (int)((((bid - by * xu) << wc) + (wave & ((1 << wc) - 1))) << lw) + (lane & ((1 << lw) - 1));
  const uint32_t row0 = ((by << (2 - wc)) + (wave >> wc)) * (64 >> lw) * U + (lane >> lw);   // of the rows of all matrices, padded ones for pack
  const uint32_t per = PACK ? yt * 32 : rows;
  const int n = (int)((uint32_t)cols - (uint32_t)chunk * EPT);   // elements of the row from this chunk on; a lane past a row of almost 2^31 elements goes beyond int
  if (PACK ? chunk >= ct * 2 * ELEM : n <= 0) return;      // a face row is ELEM chunks: its lanes stay or go together
  const int tc = chunk / (2 * ELEM), f = chunk / ELEM & 1, q = chunk % ELEM;
  u32x4 v[U];
  uint32_t in[U][2];
  int E[U];
  int64_t tile[U], rm[U];
  int fr[U];   // face row of the tile
#pragma unroll
  for (int u = 0; u < U; ++u) {
    const uint32_t g = row0 + u * (64 >> lw), b = matrices > 1 ? g / per : 0, r = g - b * per;
    tile[u] = g < per * (uint64_t)matrices ? (((int64_t)b * yt + (r >> 5)) * ct + tc) * TILE_BYTES : -1;
    fr[u] = (r >> 4 & 1) * 32 + f * 16 + (r & 15);
    rm[u] = (int)r < rows ? ((int64_t)b * rows + r) * cols + chunk * EPT : -1;
    if (PACK) {
      v[u] = u32x4{0, 0, 0, 0};
      if (tile[u] >= 0 && rm[u] >= 0 && n >= EPT) v[u] = *(const chunk_any *)((const T *)src + rm[u]);
    } else if (tile[u] >= 0) {
      const uint8_t *t = src + tile[u], *m = t + 64 + (fr[u] * ELEM + q) * CHUNK_OUT;
      E[u] = t[fr[u]];
      if (CHUNK_OUT == 8) { const u32x2 w = *(const u32x2 *)m; in[u][0] = w.x; in[u][1] = w.y; }
      else if (CHUNK_OUT == 4) in[u][0] = *(const uint32_t *)m;
      else in[u][0] = *(const uint16_t *)m;
    }
  }
  if (PACK && n > 0 && n < EPT) {   // the end of a row
#pragma unroll
    for (int u = 0; u < U; ++u) {
      if (tile[u] < 0 || rm[u] < 0) continue;
      T e[EPT];
#pragma unroll
      for (int j = 0; j < EPT; ++j) e[j] = j < n ? ((const T *)src)[rm[u] + j] : T(0);
      v[u] = *(const u32x4 *)e;
    }
  }
#pragma unroll
  for (int u = 0; u < U; ++u) {
    if (PACK) {
      uint32_t out[2];
      const uint32_t Eu = encode_plain<W, ELEM>(v[u], out);
      if (tile[u] < 0) continue;
      uint8_t *t = dst + tile[u], *m = t + 64 + (fr[u] * ELEM + q) * CHUNK_OUT;
      if (q == 0) t[fr[u]] = (uint8_t)Eu;
      if (CHUNK_OUT == 8) __builtin_nontemporal_store(u32x2{out[0], out[1]}, (u32x2 *)m);
      else if (CHUNK_OUT == 4 && W == 7) __builtin_nontemporal_store(out[0], (uint32_t *)m);
      else if (CHUNK_OUT == 4) *(uint32_t *)m = out[0];
      else *(uint16_t *)m = (uint16_t)out[0];
    } else {
      if (tile[u] < 0) continue;
      const u32x4 o = decode_chunk<W, ELEM == 2, EPT>(in[u], E[u]);
      T *p = (T *)dst + rm[u];
      if (n >= EPT) {
        *(chunk_any *)p = o;
      } else {
        T e[EPT];
        *(u32x4 *)e = o;
#pragma unroll
        for (int j = 0; j < EPT; ++j)
          if (j < n) p[j] = e[j];
      }
    }
  }
}

// ------------------------------------------------------------------------------------ ragged shapes, large
// Where the two sides no longer meet in the last-level cache, or one is host memory: the row-major side in strips of 32 rows x 512 bytes
// that start and end anywhere, moved in shifted aligned chunks (ttm_ragged.h), the packed side as in the strip kernel.  HBM-bound.
template <int W, int ELEM, bool PACK>
__global__ __launch_bounds__(256) void ttm_bfp_ragged_k(const uint8_t *__restrict__ src, uint8_t *__restrict__ dst, int rows, int cols, int strips) {
  constexpr int EPT = 16 / ELEM, CPT = 64 * ELEM, TPS = 16 / ELEM;   // elements per chunk, chunks per tile, tiles per strip
  constexpr int TILE_BYTES = 64 + (W == 7 ? 1024 : 512), CHUNK_OUT = EPT * (W + 1) / 8;
  constexpr bool VIA_LDS = PACK && W == 3;   // bfp4_b leaves as whole 16-byte chunks, as in the strip kernel
  __shared__ u32x4 image[kRaggedImage];
  __shared__ __attribute__((aligned(16))) uint8_t pk[VIA_LDS ? TPS * TILE_BYTES : 16];
  const int tid = threadIdx.x;
  const RaggedStrip st = ragged_strip<ELEM>(rows, cols, strips);
  const int64_t b = blockIdx.y;
  const int64_t tile_off = ((b * st.yt + st.ty) * st.ct + st.sx * TPS) * (int64_t)TILE_BYTES;
  const uintptr_t rm = (uintptr_t)(PACK ? src : dst) + (b * rows + st.ty * 32) * st.stride + st.sx * 512;
  if (PACK) {
    ragged_load<ELEM>(image, st, rm, (uintptr_t)src, (uintptr_t)src + (int64_t)gridDim.y * rows * st.stride);
    __syncthreads();
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int oc = i * 256 + tid, tl = oc / CPT, w = oc % CPT;
      if (tl >= st.tiles) continue;   // wavefront-uniform: a tile is a whole number of wavefronts
      const int face = w / (16 * ELEM), dy = (w / ELEM) % 16, q = w % ELEM;
      uint32_t out[2];
      const uint32_t E = encode_plain<W, ELEM>(ragged_read(image, st, rm, (face >> 1) * 16 + dy, (tl * 2 * ELEM + (face & 1) * ELEM + q) * 16), out);
      uint8_t *tile = (VIA_LDS ? pk : dst + tile_off) + tl * TILE_BYTES, *m = tile + 64 + w * CHUNK_OUT;
      if (q == 0) tile[face * 16 + dy] = (uint8_t)E;
      if (CHUNK_OUT == 8) __builtin_nontemporal_store(u32x2{out[0], out[1]}, (u32x2 *)m);
      else if (CHUNK_OUT == 2) *(uint16_t *)m = (uint16_t)out[0];
      else if (VIA_LDS) *(uint32_t *)m = out[0];
      else __builtin_nontemporal_store(out[0], (uint32_t *)m);
    }
    if constexpr (VIA_LDS) {
      __syncthreads();
      for (int c = tid; c < st.tiles * (TILE_BYTES / 16); c += 256) __builtin_nontemporal_store(((const u32x4 *)pk)[c], (u32x4 *)(dst + tile_off) + c);
    }
  } else {
    const bool more = ragged_left(st) > 512;
    u32x4 v[5];
#pragma unroll
    for (int i = 0; i < 5; ++i) {
      // i = 4: row tid of the next tile's column 0
      const int tl = i < 4 ? (i * 256 + tid) / CPT : TPS, w = i < 4 ? (i * 256 + tid) % CPT : (tid >> 4) * (32 * ELEM) + (tid & 15) * ELEM;
      if (!(i < 4 ? tl < st.tiles : tid < 32 && more)) continue;
      const uint8_t *tile = src + tile_off + tl * TILE_BYTES, *m = tile + 64 + w * CHUNK_OUT;
      const int E = tile[w / ELEM];   // face rows in order
      uint32_t in[2] = {0, 0};
      if (CHUNK_OUT == 8) {
        const u32x2 t = __builtin_nontemporal_load((const u32x2 *)m);
        in[0] = t.x; in[1] = t.y;
      } else if (CHUNK_OUT == 4) {
        in[0] = __builtin_nontemporal_load((const uint32_t *)m);
      } else {
        in[0] = __builtin_nontemporal_load((const uint16_t *)m);
      }
      v[i] = decode_chunk<W, ELEM == 2, EPT>(in, E);
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int oc = i * 256 + tid, tl = oc / CPT, w = oc % CPT;
      const int face = w / (16 * ELEM), dy = (w / ELEM) % 16, q = w % ELEM;
      if (tl < st.tiles) image[((face >> 1) * 16 + dy) * kRaggedPitch + tl * 2 * ELEM + (face & 1) * ELEM + q] = v[i];
    }
    if (tid < 32 && more) image[tid * kRaggedPitch + 32] = v[4];
    __syncthreads();
    ragged_store<ELEM>(image, st, rm);
  }
}

// ------------------------------------------------------------------------------------ generic kernels
// One lane per 4 elements of a face row; grid = (tile columns, tile rows, batch).
template <int W, bool BF16, bool PACK>
__global__ __launch_bounds__(256) void ttm_bfp_generic_k(const void *__restrict__ src_, void *__restrict__ dst_,
                                                         int64_t rows, int64_t cols, int rowmajor) {
  constexpr int TILE_BYTES = 64 + (W == 7 ? 1024 : 512);
  const int64_t xt = gridDim.x, yt = gridDim.y;
  const int64_t tx = blockIdx.x, ty = blockIdx.y, b = blockIdx.z;
  const int64_t tile_idx = (b * yt + ty) * xt + tx;
  const int w = threadIdx.x;
  const int face = w >> 6, dy = (w >> 2) & 15, q = w & 3;
  const int64_t r = ty * 32 + (face >> 1) * 16 + dy;
  const int64_t c = tx * 32 + (face & 1) * 16 + q * 4;
  const int64_t off = rowmajor ? (b * rows + r) * cols + c : tile_idx * 1024 + w * 4;
  uint8_t *tile = (uint8_t *)(PACK ? dst_ : const_cast<void *>(src_)) + tile_idx * TILE_BYTES;
  if (PACK) {
    uint32_t bits[4], out[2];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      bool in = !rowmajor || (r < rows && (c + i) < cols);
      if (BF16) bits[i] = in ? ((uint32_t)((const uint16_t *)src_)[off + i] << 16) : 0u;
      else bits[i] = in ? ((const uint32_t *)src_)[off + i] : 0u;
    }
    uint32_t E = encode_chunk<W, 4>(bits, out);
    if (q == 0) tile[face * 16 + dy] = (uint8_t)E;
    if (W == 7) ((uint32_t *)(tile + 64))[w] = out[0];
    else ((uint16_t *)(tile + 64))[w] = (uint16_t)out[0];
  } else {
    int E = tile[face * 16 + dy];
    uint32_t in[2] = {0, 0};
    if (W == 7) in[0] = ((const uint32_t *)(tile + 64))[w];
    else in[0] = ((const uint16_t *)(tile + 64))[w];
    u32x4 v = decode_chunk<W, false, 4>(in, E);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      bool inb = !rowmajor || (r < rows && (c + i) < cols);
      if (inb) {
        if (BF16) ((uint16_t *)dst_)[off + i] = (uint16_t)(v[i] >> 16);
        else ((uint32_t *)dst_)[off + i] = v[i];
      }
    }
  }
}

TTM_EXPORT int64_t ttm_bfp_tile_bytes(int fmt) { return fmt == TTM_BFP8B ? 1088 : (fmt == TTM_BFP4B ? 576 : -1); }

// Page-locked host memory or not: 0.1 us.  A pointer that HIP does not know counts as device memory.
static bool on_host(const void *p) {
  hipPointerAttribute_t a;
  if (hipPointerGetAttributes(&a, p) == hipSuccess) return a.type == hipMemoryTypeHost;
  (void)hipGetLastError();
  return false;
}

template <bool PACK>
static int run_bfp(const void *src, void *dst, int fmt, int dtype, int layout, int64_t batch, int64_t rows,
                   int64_t cols, void *stream, const char *who) {
  TTM_REQUIRE(fmt == TTM_BFP8B || fmt == TTM_BFP4B, "%s: fmt must be BFP_BFloat8 (4) or BFP_BFloat4 (6), got %d",
              who, fmt);
  TTM_REQUIRE(dtype == TTM_F32 || dtype == TTM_BF16, "%s: plain dtype must be Float32 or BFloat16, got %d", who,
              dtype);
  TTM_REQUIRE(layout == TTM_ROW_MAJOR || layout == TTM_TILE, "%s: bad layout %d", who, layout);
  TTM_REQUIRE(batch >= 0 && rows >= 0 && cols >= 0, "%s: negative dimension", who);
  if (batch == 0 || rows == 0 || cols == 0) return TTM_OK;
  TTM_REQUIRE(src && dst, "%s: null pointer", who);
  const int64_t pr = ttm_round_up32(rows), pc = ttm_round_up32(cols);
  const int64_t yt = pr / 32, xt = pc / 32;
  const int64_t ntiles = batch * yt * xt;
  const bool rm = layout == TTM_ROW_MAJOR;
  const bool bf16 = dtype == TTM_BF16;
  const int elem = bf16 ? 2 : 4;
  const bool aligned = ((uintptr_t)src & 15) == 0 && ((uintptr_t)dst & 15) == 0;
  const bool padded = rm && (rows != pr || cols != pc);
  hipStream_t s = (hipStream_t)stream;
  const int tiles_per_wg = 16 / elem;
  const int variant = ttm_option(PACK ? "pack_variant" : "unpack_variant");   // 0 by the rules below, 1 generic, 2 chunk by chunk, 3 strips of any size
  bool strip = aligned && !padded && (variant == 0 || variant == 3);
  int64_t strips_per_row = 0, blocks = 0;
  if (strip) {
    if (rm) {
      strip = (cols * elem) % 512 == 0;
      strips_per_row = cols * elem / 512;
      blocks = batch * yt * strips_per_row;
    } else {
      strip = ntiles % tiles_per_wg == 0;
      blocks = ntiles / tiles_per_wg;
    }
  }
  if (strip) {
    TTM_REQUIRE(blocks < (1ll << 31), "%s: tensor too large", who);
    dim3 grid((unsigned)blocks), block(256);
#define STRIP(Wv, EL, RM) \
  hipLaunchKernelGGL((ttm_bfp_strip_k<Wv, EL, RM, PACK>), grid, block, 0, s, src, dst, xt, strips_per_row)
#define STRIP_RM(Wv, EL)        \
  do {                          \
    if (rm) STRIP(Wv, EL, true); \
    else STRIP(Wv, EL, false);  \
  } while (0)
    if (fmt == TTM_BFP8B) { if (bf16) STRIP_RM(7, 2); else STRIP_RM(7, 4); }
    else { if (bf16) STRIP_RM(3, 2); else STRIP_RM(3, 4); }
#undef STRIP_RM
#undef STRIP
    TTM_LAUNCH_CHECK();
    return TTM_OK;
  }
  const bool plain = rm && variant != 1 && ((uintptr_t)(PACK ? dst : src) & 15) == 0 && (uintptr_t)(PACK ? src : dst) % elem == 0 &&
                     yt <= 65535 && batch <= 65535;
  // Strips from where the two sides are too large for the last-level cache: unpacking, whose stores make partial lines, above 160 MiB
  // of fp32 or 80 MiB of bf16 (bfp8_b, us, chunk by chunk / strips: [8192, 8191] fp32 85 / 71, [2, 4096, 4000] fp32 30 / 39; [3, 4096,
  // 8190] bf16 72 / 58, [3, 4096, 4000] bf16 30 to 36 / 32, [4096, 8190] bf16 18 / 24),
  // packing fp32 above 96 MiB ([3, 4096, 4000] 48 / 44, [2, 4096, 4000] 34 / 31, [3, 4000, 8001] 88 / 86; [4096, 4000] 16.1 / 17.4),
  // packing bf16 never ([3, 4096, 8190] 59 / 68).
  // To and from page-locked host memory, where every piece of a line is an access of its own, strips from 2304 tiles packed, 1536 unpacked
  // on (us, chunk by chunk / strips: pack [1500, 2001] fp32 bfp8_b from the host 261 / 244, to it 82 / 74, [4096, 4000] bf16 752 / 678,
  // 435 / 371; unpack from the host [2, 700, 1500] bf16 bfp8_b 66 / 57, [2000, 3001] bfp4_b 89 / 84).  Chunk by chunk is the better one for
  // bfp4_b packed to the host (190 / 205), unpacked from it to fp32 (193 / 206) and for unpacking to it (165 / 168).
  const int64_t strips = ttm_cdiv(pc * elem, 512);
  const bool large = !(PACK && bf16) && batch * pr * pc * elem > ((int64_t)(PACK ? 96 : bf16 ? 80 : 160) << 20);
  const auto host_side = [&] {
    if (ntiles < (PACK ? 2304 : 1536)) return false;
    if (PACK) return on_host(src) || (fmt == TTM_BFP8B && on_host(dst));
    return (fmt == TTM_BFP8B || bf16) && on_host(src);
  };
  if (plain && pr * pc < ((int64_t)1 << 31) &&
      (variant == 3 || (variant == 0 && rows >= 24 && cols * elem * 4 >= strips * 512 * 3 && (large || host_side())))) {
    const dim3 grid((unsigned)(strips * yt), (unsigned)batch);
#define RAGGED(Wv, EL) \
  hipLaunchKernelGGL((ttm_bfp_ragged_k<Wv, EL, PACK>), grid, dim3(256), 0, s, (const uint8_t *)src, (uint8_t *)dst, (int)rows, (int)cols, (int)strips)
    if (fmt == TTM_BFP8B) { if (bf16) RAGGED(7, 2); else RAGGED(7, 4); }
    else { if (bf16) RAGGED(3, 2); else RAGGED(3, 4); }
#undef RAGGED
    TTM_LAUNCH_CHECK();
    return TTM_OK;
  }
  // Chunk by chunk: rows of any width and start.  Matrices that are mostly padding are packed a tile per workgroup: few rows ([1000, 3, 100]
  // fp32 bfp4_b 6.2 us by chunks, 4.8), and fp32 of up to half a tile's columns ([64, 5093, 4] bfp8_b 11.9 by chunks, 9.2, [64, 5093, 16] 10.9
  // and 9.5, out of cache 11.6 and 11.0; [64, 5093, 25] 13.6 and 13.7; bf16 [64, 5093, 4] 9.1 and 9.9).
  const int64_t across = ttm_cdiv((PACK ? pc : cols) * elem, 16), rows_all = batch * (PACK ? pr : rows);   // chunks of a row; rows of all matrices
  const int lw = across > 4 ? 3 : 2, u = PACK && batch * rows * cols * elem > ((int64_t)16 << 20) ? 2 : 1;
  const int wc = ttm_wavefronts_across(across, lw);
  const int64_t xu = ttm_cdiv(across, 1 << (lw + wc)), groups = ttm_cdiv(rows_all, ((64 >> lw) * u) << (2 - wc));
  if (plain && (!PACK || (rows >= 24 && (bf16 || cols > 16)) || variant == 2) && pc < INT32_MAX && rows_all < INT32_MAX && groups * xu < INT32_MAX) {
#define DIRECT(Wv, EL, U)                                                                                                                       \
  ttm_launches(groups * xu, [&](uint32_t first, dim3 grid) {                                                                                    \
    hipLaunchKernelGGL((ttm_bfp_direct_k<Wv, EL, U, PACK>), grid, dim3(256), 0, s, (const uint8_t *)src, (uint8_t *)dst, (int)rows, (int)cols,  \
                       lw, wc, (uint32_t)xu, (uint32_t)batch, first, grid.x);                                                                   \
  })
#define DIRECT_U(Wv, EL)            \
  do {                              \
    if constexpr (PACK) {           \
      if (u == 2) DIRECT(Wv, EL, 2); \
      else DIRECT(Wv, EL, 1);       \
    } else DIRECT(Wv, EL, 1);       \
  } while (0)
    if (fmt == TTM_BFP8B) { if (bf16) DIRECT_U(7, 2); else DIRECT_U(7, 4); }
    else { if (bf16) DIRECT_U(3, 2); else DIRECT_U(3, 4); }
#undef DIRECT_U
#undef DIRECT
  } else {
    TTM_REQUIRE(yt <= 65535 && batch <= 65535, "%s: more than 65535 tile rows or batches on the generic path", who);
    TTM_REQUIRE(((uintptr_t)(PACK ? dst : src) & 3) == 0, "%s: packed buffer must be 4-byte aligned", who);
    dim3 grid((unsigned)xt, (unsigned)yt, (unsigned)batch), block(256);
#define GEN(Wv, B16) \
  hipLaunchKernelGGL((ttm_bfp_generic_k<Wv, B16, PACK>), grid, block, 0, s, src, dst, rows, cols, (int)rm)
    if (fmt == TTM_BFP8B) { if (bf16) GEN(7, true); else GEN(7, false); }
    else { if (bf16) GEN(3, true); else GEN(3, false); }
#undef GEN
  }
  TTM_LAUNCH_CHECK();
  return TTM_OK;
}

TTM_EXPORT int ttm_bfp_pack(const void *src, int src_dtype, int src_layout, void *dst, int fmt, int64_t batch,
                            int64_t rows, int64_t cols, void *stream) {
  TTM_EXTENTS(bfp_pack, src, src_dtype, src_layout, dst, fmt, batch, rows, cols);
  return run_bfp<true>(src, dst, fmt, src_dtype, src_layout, batch, rows, cols, stream, "ttm_bfp_pack");
}

TTM_EXPORT int ttm_bfp_unpack(const void *src, int fmt, void *dst, int dst_dtype, int dst_layout, int64_t batch,
                              int64_t rows, int64_t cols, void *stream) {
  TTM_EXTENTS(bfp_unpack, src, fmt, dst, dst_dtype, dst_layout, batch, rows, cols);
  return run_bfp<false>(src, dst, fmt, dst_dtype, dst_layout, batch, rows, cols, stream, "ttm_bfp_unpack");
}
