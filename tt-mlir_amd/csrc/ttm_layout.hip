// Tilize / untilize for Tenstorrent's 32x32 tile layout with 16x16 faces, plus the plain copy
// kernel used as the measured HBM ceiling.  All kernels move 16 bytes per lane per access.
//
// Formulations of each direction (the rule with its measurements stands at run_layout):
//   direct: one lane per 16-byte chunk of the tiled side, whose row-major half may start at any element (the part takes 16-byte
//           accesses at any address).  No LDS, no barrier; every shape.
//   strips: a workgroup owns a strip of 32 rows x 512 bytes (16/elem tiles).  Global reads and writes are both contiguous (512 B
//           per row segment on the row-major side, 16 KiB on the tiled side); the face permutation happens between a padded LDS
//           image and registers.  Tensors that pass through the last-level cache.
// ttm_set_option("tilize_variant" / "untilize_variant"): 0 by the rule, 1 direct, 2 strips of any size where a strip kernel takes the shape.
#include "ttm_common.h"
#include "ttm_ragged.h"

typedef u32x4 chunk_t;  // 16 bytes

// ------------------------------------------------------------------------------------ copy
// five workgroups of 16 KiB per CU: 256 MiB 84.4 -> 82.7 us, 64 MiB 25.6 -> 24.1 us against no cap
__global__ __launch_bounds__(256) TTM_MAX_WAVES(5) void ttm_copy_kernel_k(const chunk_t *__restrict__ src,
                                                         chunk_t *__restrict__ dst, size_t nchunks) {
  size_t base = (size_t)blockIdx.x * (256 * 4) + threadIdx.x;
  chunk_t v[4];
#pragma unroll
  for (int u = 0; u < 4; ++u) {
    size_t i = base + u * 256;
    if (i < nchunks) v[u] = __builtin_nontemporal_load(&src[i]);
  }
#pragma unroll
  for (int u = 0; u < 4; ++u) {
    size_t i = base + u * 256;
    if (i < nchunks) __builtin_nontemporal_store(v[u], &dst[i]);
  }
}

TTM_EXPORT int ttm_copy_kernel(const void *src, void *dst, size_t bytes, void *stream) {
  TTM_EXTENTS(copy_kernel, src, dst, bytes);
  if (bytes == 0) return TTM_OK;
  TTM_REQUIRE(src && dst, "ttm_copy_kernel: null pointer");
  TTM_REQUIRE(bytes % 16 == 0 && ((uintptr_t)src & 15) == 0 && ((uintptr_t)dst & 15) == 0,
              "ttm_copy_kernel: size and pointers must be multiples of 16 bytes");
  size_t n = bytes / 16;
  size_t blocks = (n + 1023) / 1024;
  TTM_REQUIRE(blocks < (1ull << 31), "ttm_copy_kernel: too large");
  hipLaunchKernelGGL(ttm_copy_kernel_k, dim3((unsigned)blocks), dim3(256), 0, (hipStream_t)stream,
                     (const chunk_t *)src, (chunk_t *)dst, n);
  TTM_LAUNCH_CHECK();
  return TTM_OK;
}

// ------------------------------------------------------------------------------------ direct
// A wavefront's access covers 8 / ELEM rows x 8 ELEM chunks (more rows of narrower tensors, fewer and longer ones of small tensors):
// 8 / ELEM face rows of 16 ELEM bytes are one 128-byte line of the tiled side, and a row's 8 ELEM chunks are 128 ELEM contiguous bytes
// of the row-major side, which starts and ends at any element: 16-byte accesses at their own alignment (a lane whose chunk crosses the
// end of a row takes elements), so nothing outside the tensor is read and nothing is shifted or exchanged.  U accesses per lane.  What
// bounds it is bytes in flight against the number of workgroups: two loads per lane are best for tilize from 192 KiB to 32 MiB, one beyond
// and for untilize (a store needs no more).  Below, a lane's second load is no shorter than the launch (kernel alone, two / one: [49, 8]
// bytes 2.7 / 2.2 us, [2, 19, 444] bf16 2.8 / 2.35, from page-locked memory [256, 264] bytes 6.5 / 5.2, but [256, 512] bf16 7.9 / 8.2).
// Tilize streams its stores past the caches, untilize does not (partial lines at the ends of rows meet in L2).  Against strips of 32
// rows x 512 bytes through LDS with funnel shifts for odd rows: [3, 1000, 3001] bf16 tilize / untilize 9.0 / 10.6 -> 7.0 / 6.9 us,
// [4000, 7001] fp32 42.0 / 37.2 -> 39.4 / 35.6, [2, 1266, 771] bf16 4.2 / 5.5 -> 3.1 / 3.2, [7, 33, 9000] fp32 7.7 / 6.2 -> 4.4 / 4.4,
// [65536, 64] bf16 5.3 / 6.2 -> 3.1 / 3.6, [70000, 3, 100] bf16 590 / 528 -> 89 / 20.
template <int ELEM>
using layout_elem = typename std::conditional<ELEM == 4, uint32_t, typename std::conditional<ELEM == 2, uint16_t, uint8_t>::type>::type;

template <int ELEM, int U, bool TILIZE>
__global__ __launch_bounds__(256) void ttm_tile_direct_k(const uint8_t *__restrict__ src, uint8_t *__restrict__ dst, int rows, int cols, int lw, int wc,
                                                         uint32_t xu, uint32_t matrices, uint32_t first, uint32_t groups) {
  typedef layout_elem<ELEM> T;
  constexpr int V = 16 / ELEM;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int ct = (cols + 31) >> 5, yt = (rows + 31) >> 5;
  // a wavefront's accesses are 1 << lw chunks wide, a workgroup 1 << wc wavefronts; its other wavefronts lie below
  const uint32_t bid = first + xcd_order(groups), by = bid / xu;
  const int chunk = (int)((((bid - by * xu) << wc) + (wave & ((1 << wc) - 1))) << lw) + (lane & ((1 << lw) - 1));
  const uint32_t row0 = ((by << (2 - wc)) + (wave >> wc)) * (64 >> lw) * U + (lane >> lw);   // of the rows of all matrices, padded ones for tilize
  const uint32_t per = TILIZE ? yt * 32 : rows;
  const int n = (int)((uint32_t)cols - (uint32_t)chunk * V);   // elements of the row from this chunk on; a lane past a row of almost 2^31 elements goes beyond int
  if (TILIZE ? chunk >= ct * 2 * ELEM : n <= 0) return;
  const int tc = chunk / (2 * ELEM), in = (chunk / ELEM & 1) * (16 * ELEM) + chunk % ELEM;   // tile column, face column and chunk of a face row
  chunk_t v[U];
  int64_t tiled[U], rm[U];   // chunk of the tiled side, element of the other; rm < 0: padding
#pragma unroll
  for (int u = 0; u < U; ++u) {
    const uint32_t g = row0 + u * (64 >> lw), b = matrices > 1 ? g / per : 0, r = g - b * per;
    tiled[u] = g < per * (uint64_t)matrices ? (((int64_t)b * yt + (r >> 5)) * ct + tc) * (64 * ELEM) + (r >> 4 & 1) * (32 * ELEM) + (r & 15) * ELEM + in : -1;
    rm[u] = (int)r < rows ? ((int64_t)b * rows + r) * cols + chunk * V : -1;
    if (TILIZE) {
      v[u] = chunk_t{0, 0, 0, 0};
      if (tiled[u] >= 0 && rm[u] >= 0 && n >= V) v[u] = *(const chunk_any *)((const T *)src + rm[u]);
    } else if (tiled[u] >= 0) {
      v[u] = ((const chunk_t *)src)[tiled[u]];
    }
  }
  if (TILIZE && n > 0 && n < V) {   // the end of a row
#pragma unroll
    for (int u = 0; u < U; ++u) {
      if (tiled[u] < 0 || rm[u] < 0) continue;
      T e[V];
#pragma unroll
      for (int j = 0; j < V; ++j) e[j] = j < n ? ((const T *)src)[rm[u] + j] : T(0);
      v[u] = *(const chunk_t *)e;
    }
  }
#pragma unroll
  for (int u = 0; u < U; ++u) {
    if (tiled[u] < 0) continue;
    if (TILIZE) {
      __builtin_nontemporal_store(v[u], (chunk_t *)dst + tiled[u]);
    } else {
      T *p = (T *)dst + rm[u];
      if (n >= V) {
        *(chunk_any *)p = v[u];
      } else {
        T e[V];
        *(chunk_t *)e = v[u];
#pragma unroll
        for (int j = 0; j < V; ++j)
          if (j < n) p[j] = e[j];
      }
    }
  }
}

// ------------------------------------------------------------------------------------ LDS staged
// Strip = 32 rows x 32 chunks (512 B).  LDS image is row-major with a 33-chunk pitch.
// Three (tilize) / four (untilize) workgroups per CU: 8192 x 8192 fp32 84.0 -> 80 / 81 us, the same 3 - 5 % for bf16 and for
// [16384, 4096], [2048, 14336], [65536, 2048].
template <int ELEM, bool TILIZE>
__global__ __launch_bounds__(256) TTM_MAX_WAVES(TILIZE ? 3 : 4) void ttm_tile_strip_k(const chunk_t *__restrict__ src,
                                                        chunk_t *__restrict__ dst, int64_t xt,
                                                        int64_t strips_per_row) {
  constexpr int CPT = 64 * ELEM;
  constexpr int PITCH = 33;
  __shared__ chunk_t lds[32 * PITCH];
  const int tid = threadIdx.x;
  const int64_t strip = blockIdx.x;                 // over (batch*yt) x strips_per_row
  const int64_t tyb = strip / strips_per_row;       // tile-row index over batch
  const int64_t sx = strip % strips_per_row;
  const int64_t row_chunks = xt * 2 * ELEM;
  const chunk_t *rm_base = (TILIZE ? src : dst) + tyb * 32 * row_chunks + sx * 32;  // unused const-ness below
  const int64_t tiled_base = (tyb * xt + sx * (16 / ELEM)) * CPT;

  chunk_t v[4];
  if (TILIZE) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      int r = i * 8 + (tid >> 5), j = tid & 31;
      v[i] = __builtin_nontemporal_load(&rm_base[r * row_chunks + j]);
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      int r = i * 8 + (tid >> 5), j = tid & 31;
      lds[r * PITCH + j] = v[i];
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      int oc = i * 256 + tid;
      int tl = oc / CPT, w = oc % CPT;
      int face = w / (16 * ELEM), dy = (w / ELEM) % 16, q = w % ELEM;
      int r = (face >> 1) * 16 + dy, j = tl * 2 * ELEM + (face & 1) * ELEM + q;
      __builtin_nontemporal_store(lds[r * PITCH + j], &dst[tiled_base + oc]);
    }
  } else {
#pragma unroll
    for (int i = 0; i < 4; ++i) v[i] = __builtin_nontemporal_load(&src[tiled_base + i * 256 + tid]);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      int oc = i * 256 + tid;
      int tl = oc / CPT, w = oc % CPT;
      int face = w / (16 * ELEM), dy = (w / ELEM) % 16, q = w % ELEM;
      int r = (face >> 1) * 16 + dy, j = tl * 2 * ELEM + (face & 1) * ELEM + q;
      lds[r * PITCH + j] = v[i];
    }
    __syncthreads();
    chunk_t *out = dst + tyb * 32 * row_chunks + sx * 32;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      int r = i * 8 + (tid >> 5), j = tid & 31;
      __builtin_nontemporal_store(lds[r * PITCH + j], &out[r * row_chunks + j]);
    }
  }
}

// ------------------------------------------------------------------------------------ scalar: tile-order sides at any address
template <typename T, bool TILIZE>
__global__ __launch_bounds__(256) void ttm_tile_scalar_k(const T *__restrict__ src, T *__restrict__ dst,
                                                         int64_t batch, int64_t rows, int64_t cols,
                                                         int64_t pr, int64_t pc) {
  int64_t n = batch * pr * pc;
  int64_t ct = pc / 32;
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (int64_t)gridDim.x * 256) {
    // i enumerates the tiled side
    int64_t b = i / (pr * pc), w = i % (pr * pc);
    int64_t tile = w / 1024;
    int e = (int)(w % 1024);
    int face = e >> 8, dy = (e >> 4) & 15, dx = e & 15;
    int64_t r = (tile / ct) * 32 + (face >> 1) * 16 + dy, c = (tile % ct) * 32 + (face & 1) * 16 + dx;
    bool in = r < rows && c < cols;
    if (TILIZE) dst[i] = in ? src[(b * rows + r) * cols + c] : T(0);
    else if (in) dst[(b * rows + r) * cols + c] = src[i];
  }
}

// ------------------------------------------------------------------------------------ untilize of ragged shapes, large
// Rows or columns that are not multiples of 32, or a row-major side that starts anywhere.  The strip kernel's plan (32 rows x 512
// bytes per workgroup) with the row-major side stored in shifted chunks (ttm_ragged.h).  HBM-bound as the strip kernel is.  The
// padding is skipped.  grid (strips x tile rows, matrices).
template <int ELEM>
__global__ __launch_bounds__(256) void ttm_untilize_ragged_k(const uint8_t *__restrict__ src, uint8_t *__restrict__ dst, int rows, int cols,
                                                             int strips, int64_t matrices) {
  constexpr int CPT = 64 * ELEM;   // chunks per tile
  __shared__ u32x4 image[kRaggedImage];
  const int tid = threadIdx.x;
  const RaggedStrip st = ragged_strip<ELEM>(rows, cols, strips);
  for (int64_t b = blockIdx.y; b < matrices; b += gridDim.y) {
    const int64_t tile_off = ((b * st.yt + st.ty) * st.ct + st.sx * (16 / ELEM)) * (int64_t)(CPT * 16);
    const uintptr_t rm = (uintptr_t)dst + (b * rows + st.ty * 32) * st.stride + st.sx * 512;
    const bool more = ragged_left(st) > 512;
    u32x4 v[5];
#pragma unroll
    for (int i = 0; i < 5; ++i) {
      const int oc = i < 4 ? i * 256 + tid : 16 / ELEM * CPT + (tid >> 4) * (32 * ELEM) + (tid & 15) * ELEM;   // i = 4: row tid of the next tile's column 0
      if (i < 4 ? oc / CPT < st.tiles : tid < 32 && more) v[i] = __builtin_nontemporal_load((const u32x4 *)(src + tile_off) + oc);
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
    if (matrices > gridDim.y) __syncthreads();
  }
}

// The kernel of a shape, by `bytes`, one side with its padding.  Times in us, tilize / untilize, of the same tensors over and over | of
// tensors that left the 256 MB last-level cache in between:
//   whole strips: direct up to 64 MiB, where neither form wins everywhere: [4096, 4096] bf16 direct 10.6 / 11.0 | 14.1 / 14.3, strips
//     11.8 / 11.2 | 12.5 / 12.4, right behind the kernel that wrote the input 10.5 / 11.2 and 10.9 / 10.7; into page-locked host memory
//     direct is the faster one ([2048, 4096] bf16 310, strips 355).  Strips beyond: [6144, 8192] bf16 30.7 / 32.4 | 31.5 / 32.4, direct
//     24.1 / 24.2 | 34.8 / 36.9, [8192, 8192] fp32 79.8 / 82.6 | 79.6 / 82.5, direct 61.3 / 91.2 | 87.9 / 91.3, [12288, 8192] fp32
//     120 / 123, direct 133 / 139.
//   other shapes: tilize direct.  Untilize direct up to 160 MiB ([4096, 8160] fp32 37.7 | 52.8, shifted strips 43.2 | 53.3; [10240, 8160]
//     bf16 53.7 | 59.7, 56.2 | 61.2), shifted strips where a strip is mostly real rows and columns beyond ([8192, 8191] fp32 69.2 | 96.0,
//     direct 91.1 | 91.6, [2, 8192, 8191] bf16 72.4 | 97.0, 90.9 | 91.2).
template <bool TILIZE>
static int run_layout(const void *src, void *dst, int64_t batch, int64_t rows, int64_t cols, int elem,
                      void *stream, const char *who) {
  TTM_REQUIRE(batch >= 0 && rows >= 0 && cols >= 0, "%s: negative dimension", who);
  TTM_REQUIRE(elem == 1 || elem == 2 || elem == 4, "%s: elem_bytes must be 1, 2 or 4 (got %d)", who, elem);
  if (batch == 0 || rows == 0 || cols == 0) return TTM_OK;
  TTM_REQUIRE(src && dst, "%s: null pointer", who);
  TTM_REQUIRE(src != dst, "%s: in-place conversion is not supported", who);
  hipStream_t s = (hipStream_t)stream;
  const int64_t pr = ttm_round_up32(rows), pc = ttm_round_up32(cols), bytes = batch * pr * pc * elem;
  const bool aligned = rows == pr && cols == pc && ((uintptr_t)src & 15) == 0 && ((uintptr_t)dst & 15) == 0;
  // whole 16-byte chunks on the tile-order side, whole elements on the other
  const bool plain = pr < INT32_MAX && pc < INT32_MAX && ((uintptr_t)(TILIZE ? dst : src) & 15) == 0 && (uintptr_t)(TILIZE ? src : dst) % elem == 0;
  const bool whole = aligned && cols * elem % 512 == 0;   // strips, all of them
  const int variant = ttm_option(TILIZE ? "tilize_variant" : "untilize_variant");
  const bool large = variant == 2 || (variant == 0 && bytes > ((int64_t)(whole ? 64 : 160) << 20));
  const int64_t strips = ttm_cdiv(pc * elem, 512);
  if (large && whole) {
    const int64_t blocks = batch * (pr / 32) * strips;
    TTM_REQUIRE(blocks < (1ll << 31), "%s: tensor too large", who);
#define STRIP(E) \
  hipLaunchKernelGGL((ttm_tile_strip_k<E, TILIZE>), dim3((unsigned)blocks), dim3(256), 0, s, \
                     (const chunk_t *)src, (chunk_t *)dst, pc / 32, strips)
    if (elem == 4) STRIP(4);
    else if (elem == 2) STRIP(2);
    else STRIP(1);
#undef STRIP
    TTM_LAUNCH_CHECK();
    return TTM_OK;
  }
  if constexpr (!TILIZE) {
    if (large && plain && pr * pc < ((int64_t)1 << 31) && (variant == 2 || (rows >= 24 && cols * elem * 4 >= strips * 512 * 3))) {
      const dim3 grid((unsigned)(strips * (pr / 32)), (unsigned)(batch > 65535 ? 65535 : batch));
#define RAGGED(E) \
  hipLaunchKernelGGL((ttm_untilize_ragged_k<E>), grid, dim3(256), 0, s, (const uint8_t *)src, (uint8_t *)dst, (int)rows, (int)cols, (int)strips, batch)
      if (elem == 4) RAGGED(4);
      else if (elem == 2) RAGGED(2);
      else RAGGED(1);
#undef RAGGED
      TTM_LAUNCH_CHECK();
      return TTM_OK;
    }
  }
  const int u = TILIZE && bytes > 192 << 10 && bytes <= ((int64_t)32 << 20) ? 2 : 1;   // accesses per lane
  const int64_t across = ttm_cdiv((TILIZE ? pc : cols) * elem, 16);   // chunks of a row
  // Chunks of a row that a wavefront's access covers: whole lines of the tiled side, and for tilize up to 4 MiB at least 512 bytes, as these are
  // mostly uploads whose rows a kernel reads from page-locked memory, while on the device the launch hides the partial lines of the
  // tiled side (3.6 us either way).  512 against 256 bytes there: a program of [256, 512] x [512, 256] bf16 70.1 -> 68.7 us, [250, 520] x
  // [520, 264] 71.4 -> 70.9; tilize alone [700, 264] bf16 10.2 -> 9.4, [500, 712] 17.1 -> 16.0, [512, 1024] of one byte 15.0 -> 12.9,
  // [1024, 1024] bf16 42.9 -> 42.8; 1024 bytes are no better ([256, 512] fp32 12.8 -> 13.9).
  const int widest = TILIZE && bytes <= ((int64_t)4 << 20) && elem < 4 ? 32 : 8 * elem;
  int lw = 0;
  while ((1 << lw) < widest && (1 << lw) < across) ++lw;
  const int wc = ttm_wavefronts_across(across, lw);
  const int64_t xu = ttm_cdiv(across, 1 << (lw + wc)), rows_all = batch * (TILIZE ? pr : rows), groups = ttm_cdiv(rows_all, ((64 >> lw) * u) << (2 - wc));
  if (plain && rows_all < INT32_MAX && groups * xu < INT32_MAX) {
#define DIRECT(E, U)                                                                                                                            \
  ttm_launches(groups * xu, [&](uint32_t first, dim3 grid) {                                                                                    \
    hipLaunchKernelGGL((ttm_tile_direct_k<E, U, TILIZE>), grid, dim3(256), 0, s, (const uint8_t *)src, (uint8_t *)dst, (int)rows, (int)cols, lw, wc, \
                       (uint32_t)xu, (uint32_t)batch, first, grid.x);                                                                           \
  })
#define DIRECT_U(E)                                       \
  do {                                                    \
    if constexpr (TILIZE) {                               \
      if (u == 2) DIRECT(E, 2);                           \
      else DIRECT(E, 1);                                  \
    } else DIRECT(E, 1);                                  \
  } while (0)
    if (elem == 4) DIRECT_U(4);
    else if (elem == 2) DIRECT_U(2);
    else DIRECT_U(1);
#undef DIRECT_U
#undef DIRECT
    TTM_LAUNCH_CHECK();
    return TTM_OK;
  }
  int64_t n = batch * pr * pc;
  unsigned blocks = (unsigned)(ttm_cdiv(n, 256) > 1048576 ? 1048576 : ttm_cdiv(n, 256));
#define SCALAR(T) \
  hipLaunchKernelGGL((ttm_tile_scalar_k<T, TILIZE>), dim3(blocks), dim3(256), 0, s, (const T *)src, (T *)dst, \
                     batch, rows, cols, pr, pc)
  if (elem == 4) SCALAR(uint32_t);
  else if (elem == 2) SCALAR(uint16_t);
  else SCALAR(uint8_t);
#undef SCALAR
  TTM_LAUNCH_CHECK();
  return TTM_OK;
}

TTM_EXPORT int ttm_tilize(const void *src, void *dst, int64_t batch, int64_t rows, int64_t cols,
                          int elem_bytes, void *stream) {
  TTM_EXTENTS(tilize, src, dst, batch, rows, cols, elem_bytes);
  return run_layout<true>(src, dst, batch, rows, cols, elem_bytes, stream, "ttm_tilize");
}

// ---- several small tensors in one launch
// A lane per 16-byte chunk of the tiled side (of a copy's bytes), chunks numbered along the rows, so that a wavefront reads 1 KiB of a row.  Bound
// by the way to the host and back: five inputs of a decode step (256 KiB and four of a few bytes) in launches of their own 18 us one behind
// the other, of which the large one 7.9; in one launch the small ones come along.
struct TilizeGroup {
  struct Item {
    const uint8_t *src;
    uint8_t *dst;
    uint32_t rows, cols, elem, groups;   // workgroups of this and the items before it
  } item[TTM_GROUP_MAX];
};
template <typename T>
__device__ __forceinline__ void tilize_chunk(const TilizeGroup::Item &t, uint32_t i) {
  constexpr uint32_t EPT = 16 / sizeof(T);
  const uint32_t ct = (t.cols + 31) >> 5, across = ct * (32 / EPT), r = i / across, c = (i - r * across) * EPT;
  if (r >= ((t.rows + 31) & ~31u)) return;
  const T *src = (const T *)t.src + (uint64_t)r * t.cols + c;
  union { T e[EPT]; u32x4 v; } x;
  x.v = u32x4{0, 0, 0, 0};
  if (r < t.rows) {
    if (c + EPT <= t.cols && ((uintptr_t)src & 15) == 0) {
      x.v = *(const u32x4 *)src;
    } else {
#pragma unroll
      for (uint32_t k = 0; k < EPT; ++k) x.e[k] = c + k < t.cols ? src[k] : (T)0;
    }
  }
  const uint64_t tile = (uint64_t)(r >> 5) * ct + (c >> 5);
  *(u32x4 *)((T *)t.dst + tile * 1024 + (((r >> 4) & 1) * 2 + ((c >> 4) & 1)) * 256 + (r & 15) * 16 + (c & 15)) = x.v;
}
__global__ __launch_bounds__(256) void ttm_tilize_group_k(TilizeGroup p) {
  uint32_t first = 0;
  int i = 0;
  while (blockIdx.x >= p.item[i].groups) first = p.item[i++].groups;   // uniform; the last item's is the size of the grid
  const TilizeGroup::Item t = p.item[i];
  const uint32_t chunk = (blockIdx.x - first) * 256 + threadIdx.x;
  if (t.elem == 0) {
    if (chunk < t.cols / 16) ((u32x4 *)t.dst)[chunk] = ((const u32x4 *)t.src)[chunk];
  } else if (t.elem == 1) {
    tilize_chunk<uint8_t>(t, chunk);
  } else if (t.elem == 2) {
    tilize_chunk<uint16_t>(t, chunk);
  } else {
    tilize_chunk<uint32_t>(t, chunk);
  }
}
TTM_EXPORT int ttm_tilize_group(const ttm_tilize_item *items, int n, void *stream) {
  TTM_REQUIRE(n >= 0 && n <= TTM_GROUP_MAX, "ttm_tilize_group: 0 to %d tensors (got %d)", TTM_GROUP_MAX, n);
  TTM_REQUIRE(items || n == 0, "ttm_tilize_group: null pointer");
  TilizeGroup p = {};
  int64_t groups = 0;
  int used = 0;
  for (int i = 0; i < n; ++i) {
    const ttm_tilize_item &t = items[i];
    TTM_REQUIRE(t.elem_bytes == 0 || t.elem_bytes == 1 || t.elem_bytes == 2 || t.elem_bytes == 4, "ttm_tilize_group: unsupported element size %d", t.elem_bytes);
    TTM_REQUIRE(t.rows >= 0 && t.cols >= 0, "ttm_tilize_group: negative dimension");
    if (t.rows == 0 || t.cols == 0) continue;
    TTM_REQUIRE(t.src && t.dst, "ttm_tilize_group: null pointer");
    TTM_REQUIRE(((uintptr_t)t.dst & 15) == 0, "ttm_tilize_group: the destination must be 16-byte aligned");
    TTM_REQUIRE(t.rows < (1 << 24) && t.cols < (1 << 30), "ttm_tilize_group: tensor %d is too large", i);
    int64_t chunks;
    if (t.elem_bytes == 0) {
      TTM_REQUIRE(t.rows == 1 && t.cols % 16 == 0 && ((uintptr_t)t.src & 15) == 0, "ttm_tilize_group: a copy takes multiples of 16 bytes");
      TTM_EXTENTS(copy_kernel, t.src, t.dst, (size_t)t.cols);
      chunks = t.cols / 16;
    } else {
      TTM_REQUIRE(((uintptr_t)t.src & (uintptr_t)(t.elem_bytes - 1)) == 0, "ttm_tilize_group: the source is not aligned to its elements");
      TTM_EXTENTS(tilize, t.src, t.dst, 1, t.rows, t.cols, t.elem_bytes);
      chunks = ttm_round_up32(t.rows) * ttm_round_up32(t.cols) * t.elem_bytes / 16;
    }
    TTM_REQUIRE(chunks < (1ll << 31), "ttm_tilize_group: tensor %d is too large", i);   // the kernel counts them in 32 bits
    groups += ttm_cdiv(chunks, 256);
    TTM_REQUIRE(groups < (1ll << 31), "ttm_tilize_group: too large");
    p.item[used++] = {(const uint8_t *)t.src, (uint8_t *)t.dst, (uint32_t)t.rows, (uint32_t)t.cols, (uint32_t)t.elem_bytes, (uint32_t)groups};
  }
  if (groups == 0) return TTM_OK;
  hipLaunchKernelGGL(ttm_tilize_group_k, dim3((unsigned)groups), dim3(256), 0, (hipStream_t)stream, p);
  TTM_LAUNCH_CHECK();
  return TTM_OK;
}

TTM_EXPORT int ttm_untilize(const void *src, void *dst, int64_t batch, int64_t rows, int64_t cols,
                            int elem_bytes, void *stream) {
  TTM_EXTENTS(untilize, src, dst, batch, rows, cols, elem_bytes);
  return run_layout<false>(src, dst, batch, rows, cols, elem_bytes, stream, "ttm_untilize");
}
