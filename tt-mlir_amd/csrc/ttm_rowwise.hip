// Row-wise bandwidth kernels on tile-ordered tensors: RMSNorm, softmax and reductions over the
// last dimension.  A workgroup owns RPB = 32 or 8 rows of one tile row (32 logical rows x all columns,
// one contiguous run of tiles in memory); 8 rows per workgroup are used when whole tile rows would
// leave most CUs without work.  Thread (r = tid % RPB, j = tid / RPB) walks the chunks of row r with
// stride 256 / RPB; the lanes of a step read whole face rows, so global accesses are contiguous runs
// of at least 256 bytes.  Partial results of the lanes of a row meet in LDS.  Math is fp32; columns beyond
// the logical width are masked with the operation's identity, rows beyond the logical height are
// written as zeros.
#include "ttm_common.h"
#include "ttm_math.h"

enum { RW_RMSNORM = 0, RW_SOFTMAX = 1, RW_SUM = 2, RW_MEAN = 3, RW_MAX = 4, RW_MIN = 5 };

struct RowArgs {
  const void *x;
  void *out;
  const void *w, *b;   // rmsnorm weight / bias (same dtype as x) or null
  int64_t rows;        // logical extent of the last two dims
  int cols;
  int rt, ct;          // tiles per batch entry
  float eps;
  uint8_t w_tiled, b_tiled;
  uint8_t stream;      // band kernel: the input is read past the caches
  // ttm_rowwise_row_k<.., PRE = true>: x is not read but made on the way in from the fp32 partial sums of a split-K
  // projection of one row tile, x = bf16(bf16(sum over slices) + residual), and also stored to sum_out
  int slices;
  const float *partial;
  int64_t per;         // floats per slice
  const void *residual;
  void *sum_out;
};

template <int ELEM>
struct ChunkPos {  // chunk q of row r inside a tile row
  int64_t off;     // element offset from the start of the tile row
  int c0;          // logical column of the chunk's first element
};
template <int ELEM>
__device__ __forceinline__ ChunkPos<ELEM> chunk_pos(int r, int q) {
  constexpr int EPC = 16 / ELEM;
  int tile = q / (2 * ELEM), fx = (q % (2 * ELEM)) / ELEM, part = q % ELEM;
  ChunkPos<ELEM> p;
  p.off = (int64_t)tile * 1024 + ((r >> 4) * 2 + fx) * 256 + (r & 15) * 16 + part * EPC;
  p.c0 = tile * 32 + fx * 16 + part * EPC;
  return p;
}

template <int ELEM>
__device__ __forceinline__ void unpack_vals(u32x4 v, float (&f)[16 / ELEM]) {
  if (ELEM == 2) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      f[2 * i] = __uint_as_float(v[i] << 16);
      f[2 * i + 1] = __uint_as_float(v[i] & 0xFFFF0000u);
    }
  } else {
#pragma unroll
    for (int i = 0; i < 4; ++i) f[i] = __uint_as_float(v[i]);
  }
}
template <int ELEM>
__device__ __forceinline__ void load_vals(const void *base, int64_t off, float (&f)[16 / ELEM]) {
  u32x4 v = *(const u32x4 *)((const uint8_t *)base + off * ELEM);
  if (ELEM == 2) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      f[2 * i] = __uint_as_float(v[i] << 16);
      f[2 * i + 1] = __uint_as_float(v[i] & 0xFFFF0000u);
    }
  } else {
#pragma unroll
    for (int i = 0; i < 4; ++i) f[i] = __uint_as_float(v[i]);
  }
}
template <int ELEM>
__device__ __forceinline__ void store_vals(void *base, int64_t off, const float (&f)[16 / ELEM]) {
  u32x4 v;
  if (ELEM == 2) {
#pragma unroll
    for (int i = 0; i < 4; ++i) v[i] = ttm_pack_bf16x2(f[2 * i], f[2 * i + 1]);
  } else {
#pragma unroll
    for (int i = 0; i < 4; ++i) v[i] = __float_as_uint(f[i]);
  }
  *(u32x4 *)((uint8_t *)base + off * ELEM) = v;
}

// weight / bias vector element c: tiled [1, C] tensor (row 0 of a 32-row tile) or plain [C]
template <int ELEM>
__device__ __forceinline__ void load_vec(const void *v, int tiled, int c0, float (&f)[16 / ELEM]) {
  int64_t off = tiled ? (int64_t)(c0 >> 5) * 1024 + ((c0 >> 4) & 1) * 256 + (c0 & 15) : c0;
  load_vals<ELEM>(v, off, f);
}

template <int MODE, int ELEM, int RPB>
__global__ __launch_bounds__(256) void ttm_rowwise_k(RowArgs p) {
  constexpr int EPC = 16 / ELEM;
  constexpr int J = 256 / RPB;                           // lanes per row
  __shared__ float part[J][RPB];
  __shared__ float part2[J][RPB];
  const int tid = threadIdx.x, j = tid / RPB;
  const int r = (int)(blockIdx.x % (32 / RPB)) * RPB + tid % RPB;   // row inside the tile row
  const int rl = tid % RPB;
  const int64_t trow = blockIdx.x / (32 / RPB);          // tile row over all batch entries
  const int64_t row = (trow % p.rt) * 32 + r;            // logical row inside the batch entry
  const bool row_ok = row < p.rows;
  const int nq = p.ct * 2 * ELEM;                        // chunks per row
  const uint8_t *x = (const uint8_t *)p.x + trow * p.ct * 1024 * ELEM;
  const int cols = p.cols;

  constexpr bool IS_MAX = MODE == RW_SOFTMAX || MODE == RW_MAX;
  float acc = IS_MAX ? -INFINITY : (MODE == RW_MIN ? INFINITY : 0.0f);
  #pragma unroll 4
  for (int q = j; q < nq; q += J) {
    ChunkPos<ELEM> cp = chunk_pos<ELEM>(r, q);
    float f[EPC];
    load_vals<ELEM>(x, cp.off, f);
#pragma unroll
    for (int i = 0; i < EPC; ++i) {
      bool ok = cp.c0 + i < cols;
      if (MODE == RW_RMSNORM) acc += ok ? f[i] * f[i] : 0.0f;
      else if (IS_MAX) acc = ok ? ttm_max(acc, f[i]) : acc;
      else if (MODE == RW_MIN) acc = ok ? ttm_min(acc, f[i]) : acc;
      else acc += ok ? f[i] : 0.0f;
    }
  }
  part[j][rl] = acc;
  __syncthreads();
  float stat = part[0][rl];
#pragma unroll
  for (int k = 1; k < J; ++k) {
    float o = part[k][rl];
    stat = IS_MAX ? ttm_max(stat, o) : (MODE == RW_MIN ? ttm_min(stat, o) : stat + o);
  }

  if (MODE == RW_SUM || MODE == RW_MEAN || MODE == RW_MAX || MODE == RW_MIN) {
    // output [.., rows, 1] in tile order: one column tile per tile row; zero padded
    if (MODE == RW_MEAN) stat = stat / (float)cols;
    uint8_t *o = (uint8_t *)p.out + trow * 1024 * ELEM;
    // the lanes clear the block's rows of the tile (both faces), then column 0 is written
    for (int e = tid; e < RPB * 2 * (16 * ELEM / 16); e += 256) {
      const int rr = (int)(blockIdx.x % (32 / RPB)) * RPB + e / (2 * ELEM), fx = (e / ELEM) & 1, part_i = e % ELEM;
      ((u32x4 *)o)[(((rr >> 4) * 2 + fx) * 256 + (rr & 15) * 16) * ELEM / 16 + part_i] = u32x4{0, 0, 0, 0};
    }
    __syncthreads();
    if (j == 0 && row_ok) {
      int64_t off = ((r >> 4) * 2) * 256 + (r & 15) * 16;
      if (ELEM == 2) ((uint16_t *)o)[off] = ttm_f32_to_bf16(stat);
      else ((float *)o)[off] = stat;
    }
    return;
  }

  uint8_t *o = (uint8_t *)p.out + trow * p.ct * 1024 * ELEM;
  if (MODE == RW_RMSNORM) {
    const float rs = 1.0f / sqrtf(stat / (float)cols + p.eps);
    #pragma unroll 4
  for (int q = j; q < nq; q += J) {
      ChunkPos<ELEM> cp = chunk_pos<ELEM>(r, q);
      float f[EPC], w[EPC], b[EPC];
      load_vals<ELEM>(x, cp.off, f);
      if (p.w) load_vec<ELEM>(p.w, p.w_tiled, cp.c0, w);
      if (p.b) load_vec<ELEM>(p.b, p.b_tiled, cp.c0, b);
#pragma unroll
      for (int i = 0; i < EPC; ++i) {
        float v = f[i] * rs;
        if (p.w) v *= w[i];
        if (p.b) v += b[i];
        f[i] = (row_ok && cp.c0 + i < cols) ? v : 0.0f;
      }
      store_vals<ELEM>(o, cp.off, f);
    }
  } else {  // softmax: second pass for the sum of exponentials, third pass writes
    const float mx = stat;
    float sum = 0.0f;
    #pragma unroll 4
  for (int q = j; q < nq; q += J) {
      ChunkPos<ELEM> cp = chunk_pos<ELEM>(r, q);
      float f[EPC];
      load_vals<ELEM>(x, cp.off, f);
#pragma unroll
      for (int i = 0; i < EPC; ++i) sum += cp.c0 + i < cols ? expf(f[i] - mx) : 0.0f;
    }
    part2[j][rl] = sum;
    __syncthreads();
    float tot = 0.0f;
#pragma unroll
    for (int k = 0; k < J; ++k) tot += part2[k][rl];
    const float inv = 1.0f / tot;
    #pragma unroll 4
  for (int q = j; q < nq; q += J) {
      ChunkPos<ELEM> cp = chunk_pos<ELEM>(r, q);
      float f[EPC];
      load_vals<ELEM>(x, cp.off, f);
#pragma unroll
      for (int i = 0; i < EPC; ++i) f[i] = (row_ok && cp.c0 + i < cols) ? expf(f[i] - mx) * inv : 0.0f;
      store_vals<ELEM>(o, cp.off, f);
    }
  }
}

// RMSNorm / softmax for rows of up to 16 chunks per lane (4096 bf16 or 2048 fp32 columns): 8 rows per workgroup,
// 32 lanes per row.  The row slice of a lane is read from global memory once and parked in LDS (64 KiB per
// workgroup, each lane reads back only what it wrote, so no barrier is involved) for the output pass.  The loops
// are kept rolled (8 loads in flight per lane): fully unrolled, the once-executed code ran at instruction-fetch speed.
template <int MODE, int ELEM>
__global__ __launch_bounds__(256) void ttm_rowwise_resident_k(RowArgs p) {
  constexpr int EPC = 16 / ELEM, RPB = 8, J = 32, NQ = 16;
  __shared__ u32x4 park[NQ * 256];
  __shared__ float part[J][RPB];
  __shared__ float part2[J][RPB];
  const int tid = threadIdx.x, j = tid / RPB, rl = tid % RPB;
  const int r = (int)(blockIdx.x % 4) * RPB + rl;
  const int trow = (int)(blockIdx.x / 4);
  const int row = (trow % p.rt) * 32 + r;
  const bool row_ok = row < p.rows;
  const int nq = p.ct * 2 * ELEM;
  const uint8_t *x = (const uint8_t *)p.x + (int64_t)trow * p.ct * 1024 * ELEM;
  uint8_t *o = (uint8_t *)p.out + (int64_t)trow * p.ct * 1024 * ELEM;
  const int cols = p.cols;
  const int nk = (nq - j + J - 1) / J;   // chunks of this lane
  float acc = MODE == RW_SOFTMAX ? -INFINITY : 0.0f;
#pragma unroll 8
  for (int k = 0; k < nk; ++k) {
    const ChunkPos<ELEM> cp = chunk_pos<ELEM>(r, j + k * J);
    const u32x4 v = *(const u32x4 *)(x + cp.off * ELEM);
    park[k * 256 + tid] = v;
    float f[EPC];
    unpack_vals<ELEM>(v, f);
#pragma unroll
    for (int i = 0; i < EPC; ++i) {
      const bool ok = cp.c0 + i < cols;
      if (MODE == RW_RMSNORM) acc += ok ? f[i] * f[i] : 0.0f;
      else acc = ok ? ttm_max(acc, f[i]) : acc;
    }
  }
  part[j][rl] = acc;
  __syncthreads();
  float stat = part[0][rl];
#pragma unroll
  for (int k = 1; k < J; ++k) stat = MODE == RW_SOFTMAX ? ttm_max(stat, part[k][rl]) : stat + part[k][rl];
  float mul = 0.0f;
  if (MODE == RW_RMSNORM) mul = 1.0f / sqrtf(stat / (float)cols + p.eps);
  else {
    float sum = 0.0f;
#pragma unroll 4
    for (int k = 0; k < nk; ++k) {
      const int c0 = chunk_pos<ELEM>(r, j + k * J).c0;
      float f[EPC];
      unpack_vals<ELEM>(park[k * 256 + tid], f);
#pragma unroll
      for (int i = 0; i < EPC; ++i) sum += c0 + i < cols ? expf(f[i] - stat) : 0.0f;
    }
    part2[j][rl] = sum;
    __syncthreads();
    float tot = 0.0f;
#pragma unroll
    for (int k = 0; k < J; ++k) tot += part2[k][rl];
    mul = 1.0f / tot;
  }
#pragma unroll 4
  for (int k = 0; k < nk; ++k) {
    const ChunkPos<ELEM> cp = chunk_pos<ELEM>(r, j + k * J);
    float f[EPC], w[EPC], b[EPC];
    unpack_vals<ELEM>(park[k * 256 + tid], f);
    if (MODE == RW_RMSNORM) {
      if (p.w) load_vec<ELEM>(p.w, p.w_tiled, cp.c0, w);
      if (p.b) load_vec<ELEM>(p.b, p.b_tiled, cp.c0, b);
    }
#pragma unroll
    for (int i = 0; i < EPC; ++i) {
      float v;
      if (MODE == RW_RMSNORM) {
        v = f[i] * mul;
        if (p.w) v *= w[i];
        if (p.b) v += b[i];
      } else {
        v = expf(f[i] - stat) * mul;
      }
      f[i] = (row_ok && cp.c0 + i < cols) ? v : 0.0f;
    }
    store_vals<ELEM>(o, cp.off, f);
  }
}

// RMSNorm / softmax with one row per workgroup of NT = 256, 512 or 1024 lanes, NK = 2 chunks per lane (at most 16384 bf16 or
// 8192 fp32 columns).  Wide rows on more lanes instead of more chunks per lane: [238, 5184] fp32 RMSNorm 7.6 -> 4.4 us, softmax 8.0 -> 5.2.
// The row stays in registers between the reduction and the output pass, weights are fetched while the reduction is in
// flight, and a workgroup issues all its loads at once: a [32, 4096] input is 32 short workgroups instead of 4 long ones.
// Consecutive rows of a face share 128-byte lines, so the row -> workgroup map gives every XCD (workgroup id mod 8)
// a contiguous range of rows and its L2 sees each line of that range whole.
template <int MODE, int ELEM, bool PRE, int NT>
__global__ __launch_bounds__(NT) void ttm_rowwise_row_k(RowArgs p, int total_rows) {
  constexpr int EPC = 16 / ELEM, NW = NT / 64, NK = 2;
  __shared__ float red[NW], red2[NW];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int per_xcd = total_rows / 8;                    // total_rows is a multiple of 32
  const int lrow = (int)(blockIdx.x % 8) * per_xcd + (int)(blockIdx.x / 8);
  const int r = lrow & 31, trow = lrow >> 5;
  const int row = (trow % p.rt) * 32 + r;
  const bool row_ok = row < p.rows;
  const int nq = p.ct * 2 * ELEM, cols = p.cols;
  const uint8_t *x = (const uint8_t *)p.x + (int64_t)trow * p.ct * 1024 * ELEM;
  uint8_t *o = (uint8_t *)p.out + (int64_t)trow * p.ct * 1024 * ELEM;
  u32x4 v[NK];
#pragma unroll
  for (int k = 0; k < NK; ++k) {
    const int q = tid + k * NT;
    v[k] = u32x4{0, 0, 0, 0};
    if constexpr (PRE) {   // bf16 rows made from partial sums: the projection's rounding, then the residual add's
      static_assert(!PRE || ELEM == 2, "partial sums finish as bf16");
      if (q < nq) {
        const int64_t off = chunk_pos<ELEM>(r, q).off;
        if (row_ok) {
          f32x4 s0 = *(const f32x4 *)(p.partial + off), s1 = *(const f32x4 *)(p.partial + off + 4);
          for (int sl = 1; sl < p.slices; ++sl) {
            s0 += *(const f32x4 *)(p.partial + sl * p.per + off);
            s1 += *(const f32x4 *)(p.partial + sl * p.per + off + 4);
          }
          const u32x4 y = {ttm_pack_bf16x2(s0.x, s0.y), ttm_pack_bf16x2(s0.z, s0.w), ttm_pack_bf16x2(s1.x, s1.y), ttm_pack_bf16x2(s1.z, s1.w)};
          const u32x4 t = *(const u32x4 *)((const uint8_t *)p.residual + off * 2);
#pragma unroll
          for (int i = 0; i < 4; ++i)
            v[k][i] = ttm_pack_bf16x2(__uint_as_float(y[i] << 16) + __uint_as_float(t[i] << 16),
                                      __uint_as_float(y[i] & 0xFFFF0000u) + __uint_as_float(t[i] & 0xFFFF0000u));
        }
        *(u32x4 *)((uint8_t *)p.sum_out + off * 2) = v[k];
      }
    } else if (q < nq && row_ok) v[k] = *(const u32x4 *)(x + chunk_pos<ELEM>(r, q).off * ELEM);
  }
  u32x4 wraw[NK], braw[NK];   // weight / bias chunks, still packed
  if (MODE == RW_RMSNORM) {
#pragma unroll
    for (int k = 0; k < NK; ++k) {
      const int q = tid + k * NT;
      if (q < nq) {
        const int c0 = chunk_pos<ELEM>(r, q).c0;
        const int64_t tiled = (int64_t)(c0 >> 5) * 1024 + ((c0 >> 4) & 1) * 256 + (c0 & 15);
        if (p.w) wraw[k] = *(const u32x4 *)((const uint8_t *)p.w + (p.w_tiled ? tiled : c0) * ELEM);
        if (p.b) braw[k] = *(const u32x4 *)((const uint8_t *)p.b + (p.b_tiled ? tiled : c0) * ELEM);
      }
    }
  }
  float acc = MODE == RW_SOFTMAX ? -INFINITY : 0.0f;
#pragma unroll
  for (int k = 0; k < NK; ++k) {
    const int q = tid + k * NT;
    if (q < nq) {
      const int c0 = chunk_pos<ELEM>(r, q).c0;
      float f[EPC];
      unpack_vals<ELEM>(v[k], f);
#pragma unroll
      for (int i = 0; i < EPC; ++i) {
        const bool ok = c0 + i < cols;
        if (MODE == RW_RMSNORM) acc += ok ? f[i] * f[i] : 0.0f;
        else acc = ok ? ttm_max(acc, f[i]) : acc;
      }
    }
  }
#pragma unroll
  for (int s = 32; s > 0; s >>= 1) acc = MODE == RW_SOFTMAX ? ttm_max(acc, __shfl_xor(acc, s)) : acc + __shfl_xor(acc, s);
  // chains of four wavefronts, added in pairs: sixteen one behind the other doubled the error of a sum
  auto total = [&](const float (&r)[NW], bool is_max) __attribute__((always_inline)) {
    const auto op = [&](float a, float b) { return is_max ? ttm_max(a, b) : a + b; };
    float q[NW / 4];
#pragma unroll
    for (int i = 0; i < NW / 4; ++i) q[i] = op(op(op(r[4 * i], r[4 * i + 1]), r[4 * i + 2]), r[4 * i + 3]);
#pragma unroll
    for (int s = NW / 8; s > 0; s >>= 1)
#pragma unroll
      for (int i = 0; i < s; ++i) q[i] = op(q[i], q[i + s]);
    return q[0];
  };
  if (lane == 0) red[wave] = acc;
  __syncthreads();
  const float stat = total(red, MODE == RW_SOFTMAX);
  float mul;
  if (MODE == RW_RMSNORM) {
    mul = 1.0f / sqrtf(stat / (float)cols + p.eps);
  } else {
    float sum = 0.0f;
#pragma unroll
    for (int k = 0; k < NK; ++k) {
      const int q = tid + k * NT;
      if (q < nq) {
        const int c0 = chunk_pos<ELEM>(r, q).c0;
        float f[EPC];
        unpack_vals<ELEM>(v[k], f);
#pragma unroll
        for (int i = 0; i < EPC; ++i) sum += c0 + i < cols ? expf(f[i] - stat) : 0.0f;
      }
    }
#pragma unroll
    for (int s = 32; s > 0; s >>= 1) sum += __shfl_xor(sum, s);
    if (lane == 0) red2[wave] = sum;
    __syncthreads();
    mul = 1.0f / total(red2, false);
  }
#pragma unroll
  for (int k = 0; k < NK; ++k) {
    const int q = tid + k * NT;
    if (q < nq) {
      const ChunkPos<ELEM> cp = chunk_pos<ELEM>(r, q);
      float f[EPC], w[EPC], b[EPC];
      unpack_vals<ELEM>(v[k], f);
      if (MODE == RW_RMSNORM) {
        if (p.w) unpack_vals<ELEM>(wraw[k], w);
        if (p.b) unpack_vals<ELEM>(braw[k], b);
      }
#pragma unroll
      for (int i = 0; i < EPC; ++i) {
        float y;
        if (MODE == RW_RMSNORM) {
          y = f[i] * mul;
          if (p.w) y *= w[i];
          if (p.b) y += b[i];
        } else {
          y = expf(f[i] - stat) * mul;
        }
        f[i] = (row_ok && cp.c0 + i < cols) ? y : 0.0f;
      }
      store_vals<ELEM>(o, cp.off, f);
    }
  }
}

// All six modes with four consecutive rows per workgroup, for large row counts.  Four rows of a face are one run of whole
// 128-byte lines (128 bytes of bf16, 256 of fp32) in every tile, so a workgroup reads and writes nothing but whole lines
// that no other workgroup touches; consecutive lanes take consecutive 16-byte chunks of those runs.  A lane keeps its NK
// chunks (the same row in each: 256 is a multiple of the chunks per run) in registers from the single read to the write,
// and every load of the workgroup is in flight before the first use: 4 KiB x NK per workgroup, which is what keeps HBM
// busy when each workgroup lives only a few microseconds.  Row statistics: shuffles over the lanes of a wavefront that
// hold the same row, then four values per row through LDS.
#ifndef TTM_BAND_EXP
#define TTM_BAND_EXP expf
#endif
// Workgroups per CU of 256-lane bands of 16 KiB, measured at 65536 rows: reductions 4 (44 -> 40 us for 1024 fp32 columns), fp32 softmax
// 4 (94 -> 88 us); everything else runs best without a cap.
template <int MODE, int ELEM, int NK, int NT>
constexpr int band_max_waves() {
  return NT == 256 && NK == 4 && (MODE >= RW_SUM || (MODE == RW_SOFTMAX && ELEM == 4)) ? 4 : 8;
}
// NT lanes, up to eight chunks each: bands wider than a few chunks per 256 lanes take 512 or 1024 lanes instead of more chunks per
// lane, whose unrolled code is executed once and mostly waits for its own instructions.  In turn over three tensors (us, sixteen or
// eight chunks per lane before, now): RMSNorm [2048, 4096] bf16 9.1 -> 7.5, [843, 5952] fp32 29.3 -> 8.7, [2048, 8192] bf16 17.4 -> 14.1;
// softmax [2048, 4096] bf16 11.0 -> 9.3, [843, 5952] fp32 18.5 -> 11.6; sum [560, 8000] bf16 14.1 -> 3.6, [2048, 8192] fp32 13.3 -> 11.7.
template <int MODE, int ELEM, int NK, int NT>
__global__ __launch_bounds__(NT) TTM_MAX_WAVES((band_max_waves<MODE, ELEM, NK, NT>())) void ttm_rowwise_band_k(RowArgs p) {
  constexpr int EPC = 16 / ELEM, RUN = 4 * ELEM;         // chunks per run of four face rows
  constexpr bool IS_MAX = MODE == RW_SOFTMAX || MODE == RW_MAX;
  constexpr bool REDUCE = MODE == RW_SUM || MODE == RW_MEAN || MODE == RW_MAX || MODE == RW_MIN;
  constexpr int NW = NT / 64;
  __shared__ float red[NW][4], red2[NW][4];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int g4 = (int)(blockIdx.x & 7);                  // group of four rows inside the tile row
  const int64_t trow = blockIdx.x >> 3;                  // tile row over all batch entries
  const int rl = (tid % RUN) / ELEM, part = tid % ELEM;
  const int r = g4 * 4 + rl;
  const int64_t row = (trow % p.rt) * 32 + r;
  const bool row_ok = row < p.rows;
  const int nruns = p.ct * 2, cols = p.cols;        // runs per band: one per (tile, face column)
  const uint8_t *x = (const uint8_t *)p.x + trow * p.ct * 1024 * ELEM;
  // chunk k of this lane: run tid / RUN + k * (NT / RUN)
  auto run_of = [&](int k) { return tid / RUN + k * (NT / RUN); };
  auto off_of = [&](int run) { return (int64_t)(run >> 1) * 1024 + ((r >> 4) * 2 + (run & 1)) * 256 + (r & 15) * 16 + part * EPC; };
  auto col_of = [&](int run) { return (run >> 1) * 32 + (run & 1) * 16 + part * EPC; };
  u32x4 v[NK];
  // unconditional (a run past the end repeats the last one and is masked where it is used): a branch around a load
  // makes the compiler wait for each load before it issues the next
  auto at = [&](int k) { return (const u32x4 *)(x + off_of(min(run_of(k), nruns - 1)) * ELEM); };
  if (REDUCE || p.stream) {   // uniform; the empty asm keeps the compiler from merging the two forms of a load
    asm volatile("");
#pragma unroll
    for (int k = 0; k < NK; ++k) v[k] = __builtin_nontemporal_load(at(k));
    asm volatile("");
  } else {
#pragma unroll
    for (int k = 0; k < NK; ++k) v[k] = *at(k);
  }
  // RMSNorm: the weight and bias chunks of this lane's columns, beside the input where the registers allow it ([2048, 4096] fp32 11.2 us,
  // 14.2 at the use), else four chunks at a time where they are used (they come from the L2: every row shares them; [2048, 4096] bf16 7.4
  // us, 7.8 up front)
  constexpr bool WB_EARLY = MODE == RW_RMSNORM && NK * NT <= (ELEM == 4 ? 4096 : 1024);
  auto vec_load = [&](const void *vec, int tiled, int k) {
    const int c0 = min(col_of(run_of(k)), (cols - 1) / EPC * EPC);   // the padding of the last tile has no weight: a valid chunk again
    return *(const u32x4 *)((const uint8_t *)vec + (tiled ? (int64_t)(c0 >> 5) * 1024 + ((c0 >> 4) & 1) * 256 + (c0 & 15) : (int64_t)c0) * ELEM);
  };
  u32x4 wraw[WB_EARLY ? NK : 1], braw[WB_EARLY ? NK : 1];
  if constexpr (WB_EARLY) {
    if (p.w) {   // uniform
#pragma unroll
      for (int k = 0; k < NK; ++k) wraw[k] = vec_load(p.w, p.w_tiled, k);
    }
    if (p.b) {
#pragma unroll
      for (int k = 0; k < NK; ++k) braw[k] = vec_load(p.b, p.b_tiled, k);
    }
  }
  // the lanes of a wavefront that share a row differ in the chunk-part bits (below ELEM) and the run bits (RUN and up)
  auto wave_combine = [&](float a, bool is_max, bool is_min) {
#pragma unroll
    for (int sft = 1; sft < 64; sft <<= 1) {
      if (sft >= ELEM && sft < RUN) continue;            // the row bits
      const float o = __shfl_xor(a, sft);
      a = is_max ? ttm_max(a, o) : (is_min ? ttm_min(a, o) : a + o);
    }
    return a;
  };
  // the wavefronts' results in pairs, four of them at a time (all sixteen at once cost registers: fp32 RMSNorm [1534, 3072] 7.5 -> 9.4 us)
  auto total = [&](const float (&part)[NW][4], bool is_max, bool is_min) __attribute__((always_inline)) {
    const auto op = [&](float a, float b) { return is_max ? ttm_max(a, b) : is_min ? ttm_min(a, b) : a + b; };
    const auto four = [&](int w) { return op(op(part[w][rl], part[w + 1][rl]), op(part[w + 2][rl], part[w + 3][rl])); };
    float sum = four(0);
    if constexpr (NW >= 8) {
      sum = op(sum, four(4));
      __builtin_amdgcn_sched_barrier(0);
    }
    if constexpr (NW == 16) sum = op(sum, op(four(8), four(12)));
    return sum;
  };
  float acc = IS_MAX ? -INFINITY : (MODE == RW_MIN ? INFINITY : 0.0f);
#pragma unroll
  for (int k = 0; k < NK; ++k) {
    const int run = run_of(k);
    const int c0 = col_of(run);
    const int lim = run < nruns ? cols : 0;
    float f[EPC];
    unpack_vals<ELEM>(v[k], f);
#pragma unroll
    for (int i = 0; i < EPC; ++i) {
      const bool ok = c0 + i < lim;
      if (MODE == RW_RMSNORM) acc += ok ? f[i] * f[i] : 0.0f;
      else if (IS_MAX) acc = ok ? ttm_max(acc, f[i]) : acc;
      else if (MODE == RW_MIN) acc = ok ? ttm_min(acc, f[i]) : acc;
      else acc += ok ? f[i] : 0.0f;
    }
  }
  acc = wave_combine(acc, IS_MAX, MODE == RW_MIN);
  if ((lane & ~(RUN - ELEM)) == 0) red[wave][rl] = acc;  // one lane per row and wavefront
  __syncthreads();
  float stat = total(red, IS_MAX, MODE == RW_MIN);
  if constexpr (REDUCE) {
    // output [.., rows, 1] in tile order: one column tile per tile row; this workgroup owns its four rows of it, both faces
    if (MODE == RW_MEAN) stat = stat / (float)cols;
    if (tid < 2 * RUN) {
      const int fx = tid / RUN;
      u32x4 z = u32x4{0, 0, 0, 0};
      if (fx == 0 && part == 0 && row_ok) z.x = ELEM == 2 ? (uint32_t)ttm_f32_to_bf16(stat) : __float_as_uint(stat);
      uint8_t *o = (uint8_t *)p.out + trow * 1024 * ELEM;
      *(u32x4 *)(o + (int64_t)(((r >> 4) * 2 + fx) * 256 + (r & 15) * 16 + part * EPC) * ELEM) = z;
    }
    return;
  } else {
    uint8_t *o = (uint8_t *)p.out + trow * p.ct * 1024 * ELEM;
    float mul;
    float e[MODE == RW_SOFTMAX ? NK : 1][EPC];
    if constexpr (MODE == RW_RMSNORM) {
      mul = 1.0f / sqrtf(stat / (float)cols + p.eps);
    } else {
      float sum = 0.0f;
#pragma unroll
      for (int k = 0; k < NK; ++k) {
        const int run = run_of(k);
        const int c0 = col_of(run);
        float f[EPC];
        unpack_vals<ELEM>(v[k], f);
#pragma unroll
        for (int i = 0; i < EPC; ++i) {
          e[k][i] = (run < nruns && c0 + i < cols) ? TTM_BAND_EXP(f[i] - stat) : 0.0f;
          sum += e[k][i];
        }
      }
      sum = wave_combine(sum, false, false);
      if ((lane & ~(RUN - ELEM)) == 0) red2[wave][rl] = sum;
      __syncthreads();
      mul = 1.0f / total(red2, false, false);
    }
    u32x4 wlate[4], blate[4];
#pragma unroll
    for (int k = 0; k < NK; ++k) {
      if constexpr (MODE == RW_RMSNORM && !WB_EARLY) {
        if (k % 4 == 0) {
          __builtin_amdgcn_sched_barrier(0);   // the loads of one batch only: the scheduler would hoist all of them
          if (p.w) {
#pragma unroll
            for (int u = 0; u < 4; ++u) wlate[u] = vec_load(p.w, p.w_tiled, min(k + u, NK - 1));
          }
          if (p.b) {
#pragma unroll
            for (int u = 0; u < 4; ++u) blate[u] = vec_load(p.b, p.b_tiled, min(k + u, NK - 1));
          }
          __builtin_amdgcn_sched_barrier(0);
        }
      }
      const int run = run_of(k);
      if (run < nruns) {
        const int c0 = col_of(run);
        float f[EPC];
        if constexpr (MODE == RW_RMSNORM) {
          float w[EPC], b[EPC];
          unpack_vals<ELEM>(v[k], f);
          if (p.w) unpack_vals<ELEM>(WB_EARLY ? wraw[WB_EARLY ? k : 0] : wlate[k % 4], w);
          if (p.b) unpack_vals<ELEM>(WB_EARLY ? braw[WB_EARLY ? k : 0] : blate[k % 4], b);
#pragma unroll
          for (int i = 0; i < EPC; ++i) {
            float y = f[i] * mul;
            if (p.w) y *= w[i];
            if (p.b) y += b[i];
            f[i] = (row_ok && c0 + i < cols) ? y : 0.0f;
          }
        } else {
#pragma unroll
          for (int i = 0; i < EPC; ++i) f[i] = row_ok ? e[k][i] * mul : 0.0f;
        }
        u32x4 ov;
        if (ELEM == 2) {
#pragma unroll
          for (int i = 0; i < 4; ++i) ov[i] = ttm_pack_bf16x2(f[2 * i], f[2 * i + 1]);
        } else {
#pragma unroll
          for (int i = 0; i < 4; ++i) ov[i] = __float_as_uint(f[i]);
        }
        __builtin_nontemporal_store(ov, (u32x4 *)(o + off_of(run) * ELEM));
      }
    }
  }
}

// ------------------------------------------------------------------------------------------------ few, very wide rows
// A vocabulary-sized row for a handful of tokens: too few tile rows to fill the device with one workgroup each.  grid
// (slices, tile rows): a workgroup takes a range of column tiles of one tile row (all 32 rows of it).  Lane t holds the
// same 16-byte chunk position in every tile it visits, hence one row; the eight lanes that share a row are combined
// through LDS.  Step one leaves per (row, slice) the statistics - (max, sum of exp relative to it) for softmax, the sum of
// squares for RMSNorm, the partial result for the reductions; step two forms each row's total from all slices and, for
// softmax and RMSNorm, reads the slice again and writes the output.  stats: [tile row][32][slices][2] floats.
template <int ELEM>
struct WideLane {
  static constexpr int EPC = 16 / ELEM, CPT = 1024 / EPC, TPI = 256 / CPT;   // chunks per tile, tiles per step of a workgroup
  int e, r, col_in, sub;
  __device__ __forceinline__ WideLane(int tid) {
    const int c = tid % CPT;
    sub = tid / CPT;
    e = c * EPC;
    const int face = e >> 8;
    r = (face >> 1) * 16 + ((e >> 4) & 15);
    col_in = (face & 1) * 16 + (e & 15);
  }
  // LDS slot of the i-th of the eight lanes that hold row rr
  static __device__ __forceinline__ int partner(int rr, int i) {
    const int q = i % ELEM, f1 = (i / ELEM) & 1, sb = i / (2 * ELEM);
    return sb * CPT + ((rr >> 4) * 2 + f1) * (16 * ELEM) + (rr & 15) * ELEM + q;
  }
};

template <int MODE, int ELEM>
__global__ __launch_bounds__(256) void ttm_rowwise_wide_stats_k(RowArgs p, float *__restrict__ stats, int slices, int tiles_per_slice) {
  using L = WideLane<ELEM>;
  constexpr int EPC = L::EPC;
  constexpr bool IS_MAX = MODE == RW_SOFTMAX || MODE == RW_MAX;
  __shared__ float sa[256], sb[256];
  const int tid = threadIdx.x, slice = blockIdx.x, cols = p.cols;
  const int64_t trow = blockIdx.y;
  const L ln(tid);
  const uint8_t *x = (const uint8_t *)p.x + trow * p.ct * 1024 * ELEM;
  const int t0 = slice * tiles_per_slice, t1 = min(p.ct, t0 + tiles_per_slice);
  float a = IS_MAX ? -INFINITY : (MODE == RW_MIN ? INFINITY : 0.0f), l = 0.0f;
  constexpr int UN = 4;   // loads in flight per lane: unconditional, clamped to the slice (a branch around a load serialises them)
  for (int tb = t0 + ln.sub; tb < t1; tb += UN * L::TPI) {
    u32x4 raw[UN];
#pragma unroll
    for (int u = 0; u < UN; ++u) raw[u] = __builtin_nontemporal_load((const u32x4 *)(x + ((int64_t)min(tb + u * L::TPI, t1 - 1) * 1024 + ln.e) * ELEM));
#pragma unroll
    for (int u = 0; u < UN; ++u) {
    const int t = tb + u * L::TPI;
    if (t >= t1) break;
    float f[EPC];
    unpack_vals<ELEM>(raw[u], f);
    const int c0 = t * 32 + ln.col_in;
    if (MODE == RW_SOFTMAX) {
      float cm = -INFINITY;
#pragma unroll
      for (int i = 0; i < EPC; ++i) cm = c0 + i < cols ? ttm_max(cm, f[i]) : cm;
      if (cm > a || cm != cm) { l *= expf(a - cm); a = cm; }   // a = -inf at first: l is 0 and stays 0; a NaN maximum stays and makes l NaN
      if (a != -INFINITY) {
#pragma unroll
        for (int i = 0; i < EPC; ++i) l += c0 + i < cols ? expf(f[i] - a) : 0.0f;
      }
    } else {
#pragma unroll
      for (int i = 0; i < EPC; ++i) {
        const bool ok = c0 + i < cols;
        if (MODE == RW_RMSNORM) a += ok ? f[i] * f[i] : 0.0f;
        else if (MODE == RW_MAX) a = ok ? ttm_max(a, f[i]) : a;
        else if (MODE == RW_MIN) a = ok ? ttm_min(a, f[i]) : a;
        else a += ok ? f[i] : 0.0f;
      }
    }
    }
  }
  sa[tid] = a; sb[tid] = l;
  __syncthreads();
  if (tid < 32) {
    float A = IS_MAX ? -INFINITY : (MODE == RW_MIN ? INFINITY : 0.0f), Lsum = 0.0f;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const float v = sa[L::partner(tid, i)];
      A = IS_MAX ? ttm_max(A, v) : (MODE == RW_MIN ? ttm_min(A, v) : A + v);
    }
    if (MODE == RW_SOFTMAX) {
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const int k = L::partner(tid, i);
        Lsum += sa[k] == -INFINITY ? 0.0f : sb[k] * expf(sa[k] - A);
      }
    }
    float *o = stats + ((trow * 32 + tid) * slices + slice) * 2;
    o[0] = A; o[1] = Lsum;
  }
}

// row totals from the slices, by the whole workgroup: lane (row = tid % 32, part = tid / 32) folds every eighth slice of its
// row, the eight parts of a row meet in LDS.  Softmax folds (max, sum relative to that max) pairs.
template <int MODE>
__device__ __forceinline__ void wide_fold(float &A, float &Ls, float v, float w) {
  if (MODE == RW_SOFTMAX) {
    if (v > A) { Ls = Ls * expf(A - v) + w; A = v; }   // A = -inf: Ls is 0 and exp gives 0
    else if (v != -INFINITY) Ls += w * expf(v - A);
  } else if (MODE == RW_MAX) A = ttm_max(A, v);
  else if (MODE == RW_MIN) A = ttm_min(A, v);
  else A += v;
}
template <int MODE>
__device__ __forceinline__ void wide_totals(const float *st, int slices, float *ga, float *gb, float *ta, float *tb) {
  constexpr bool IS_MAX = MODE == RW_SOFTMAX || MODE == RW_MAX;
  const int tid = threadIdx.x, rr = tid & 31, part = tid >> 5;
  float A = IS_MAX ? -INFINITY : (MODE == RW_MIN ? INFINITY : 0.0f), Ls = 0.0f;
  for (int s = part; s < slices; s += 8) wide_fold<MODE>(A, Ls, st[((int64_t)rr * slices + s) * 2], st[((int64_t)rr * slices + s) * 2 + 1]);
  ta[tid] = A; tb[tid] = Ls;
  __syncthreads();
  if (tid < 32) {
    for (int k = 1; k < 8; ++k) wide_fold<MODE>(A, Ls, ta[tid + 32 * k], tb[tid + 32 * k]);
    ga[tid] = A; gb[tid] = Ls;
  }
  __syncthreads();
}

template <int MODE, int ELEM>   // softmax or RMSNorm
__global__ __launch_bounds__(256) void ttm_rowwise_wide_apply_k(RowArgs p, const float *__restrict__ stats, int slices, int tiles_per_slice) {
  using L = WideLane<ELEM>;
  constexpr int EPC = L::EPC;
  __shared__ float ga[32], gb[32], ta[256], tb[256];
  const int tid = threadIdx.x, slice = blockIdx.x, cols = p.cols;
  const int64_t trow = blockIdx.y;
  wide_totals<MODE>(stats + trow * 32 * slices * 2, slices, ga, gb, ta, tb);
  const L ln(tid);
  const bool row_ok = (trow % p.rt) * 32 + ln.r < p.rows;
  const float A = ga[ln.r];
  const float mul = MODE == RW_RMSNORM ? 1.0f / sqrtf(A / (float)cols + p.eps) : 1.0f / gb[ln.r];
  const uint8_t *x = (const uint8_t *)p.x + trow * p.ct * 1024 * ELEM;
  uint8_t *o = (uint8_t *)p.out + trow * p.ct * 1024 * ELEM;
  const int t0 = slice * tiles_per_slice, t1 = min(p.ct, t0 + tiles_per_slice);
  constexpr int UN = 4;
  for (int tb = t0 + ln.sub; tb < t1; tb += UN * L::TPI) {
    u32x4 raw[UN];
#pragma unroll
    for (int u = 0; u < UN; ++u) raw[u] = __builtin_nontemporal_load((const u32x4 *)(x + ((int64_t)min(tb + u * L::TPI, t1 - 1) * 1024 + ln.e) * ELEM));
#pragma unroll
    for (int u = 0; u < UN; ++u) {
    const int t = tb + u * L::TPI;
    if (t >= t1) break;
    const int64_t off = (int64_t)t * 1024 + ln.e;
    float f[EPC];
    unpack_vals<ELEM>(raw[u], f);
    const int c0 = t * 32 + ln.col_in;
    if (MODE == RW_RMSNORM) {
      float w[EPC], b[EPC];
      const int cc = min(c0, ((cols + EPC - 1) / EPC - 1) * EPC);   // the padding of the last tile has no weight: reread a valid chunk
      if (p.w) load_vec<ELEM>(p.w, p.w_tiled, cc, w);
      if (p.b) load_vec<ELEM>(p.b, p.b_tiled, cc, b);
#pragma unroll
      for (int i = 0; i < EPC; ++i) {
        float y = f[i] * mul;
        if (p.w) y *= w[i];
        if (p.b) y += b[i];
        f[i] = (row_ok && c0 + i < cols) ? y : 0.0f;
      }
    } else {
#pragma unroll
      for (int i = 0; i < EPC; ++i) f[i] = (row_ok && c0 + i < cols) ? expf(f[i] - A) * mul : 0.0f;
    }
    store_vals<ELEM>(o, off, f);
    }
  }
}

template <int MODE, int ELEM>   // reductions: the [.., rows, 1] output tile of every tile row
__global__ __launch_bounds__(256) void ttm_rowwise_wide_finish_k(RowArgs p, const float *__restrict__ stats, int slices) {
  using L = WideLane<ELEM>;
  __shared__ float ga[32], gb[32], ta[256], tb[256];
  const int tid = threadIdx.x;
  const int64_t trow = blockIdx.x;
  wide_totals<MODE>(stats + trow * 32 * slices * 2, slices, ga, gb, ta, tb);
  if (tid < L::CPT) {
    const L ln(tid);
    u32x4 z = {0, 0, 0, 0};
    const float total = MODE == RW_MEAN ? ga[ln.r] / (float)p.cols : ga[ln.r];
    if (ln.col_in == 0 && (trow % p.rt) * 32 + ln.r < p.rows) z.x = ELEM == 2 ? (uint32_t)ttm_f32_to_bf16(total) : __float_as_uint(total);
    *(u32x4 *)((uint8_t *)p.out + (trow * 1024 + ln.e) * ELEM) = z;
  }
}

template <int MODE>
static int launch_rowwise(const RowArgs &p, int dtype, int64_t trows, hipStream_t s) {
  TTM_REQUIRE(trows < (1ll << 29), "row-wise kernel: tensor too large");
  {
    const int elem = dtype == TTM_BF16 ? 2 : 4, variant = ttm_option("rowwise_variant");
    const int64_t bands = trows * 8;
    const int nk = (int)ttm_cdiv((int64_t)p.ct * 2 * 4 * elem, 256);   // chunks per lane of a 256-lane workgroup
    // Four rows per workgroup, whole lines, the band in registers: rows of up to 32 chunks per 256 lanes (16384 bf16 or 8192 fp32
    // columns).  RMSNorm and softmax take it from one workgroup per CU upwards, wide rows from half of that (fp32 [500, 4096] 4.9 us, one
    // row per workgroup 5.3; fewer rows are faster that way: [238, 5184] 4.4, as bands 7.5); reductions, whose other kernel gives a lane
    // of 32 per row, always ([238, 5184] bf16 6.8 -> 3.5 us), but for the rows that ttm_rowwise_wide_* spreads over the device.
    // rowwise_variant: 2 forces it, 1 and 3 exclude it.
    bool band = nk <= 32 && bands < (1ll << 31) && variant != 1 && variant != 3;
    if constexpr (MODE == RW_RMSNORM || MODE == RW_SOFTMAX) band = band && (variant == 2 || bands >= 256 || (nk > 8 && bands >= 128));
    else band = band && (variant == 2 || p.ct < 256 || bands >= 64);
    if (band) {
      const dim3 grid((unsigned)bands);
      RowArgs q = p;
      // Plain loads find what the producer left in the last-level cache (RMSNorm [8192, 4096] bf16 30.9 -> 23.1 us); an input of which little
      // can be there is read past it, and that of a reduction always, whose short workgroups the choice itself delays (sum over twelve tensors, us: plain /
      // past the caches, bf16 [8192, 2048] 7.6 / 7.1, [2048, 8192] 7.7 / 7.2, fp32 [4096, 2048] 7.4 / 6.9, [500, 8000] 4.9 / 5.5, [8192, 8192] 47.6 / 42.7)
      q.stream = (int64_t)p.ct * 1024 * elem * trows > 100000000;
      // LDS that only limits how many bands are on the way in a CU: 32 KiB each, three for reductions (65536 fp32 rows of 2048 86 -> 82 us, of bf16 4096
      // 82.3 -> 81.3; narrower ones are faster without: bf16 3000 60.7, 64.1), two for fp32 softmax past the caches (192 -> 188; 8192 rows 20.9, 21.7)
      size_t lds = 0;
      if (nk == 8 && MODE != RW_RMSNORM && MODE != RW_SOFTMAX) lds = 50 << 10;
      if (nk == 8 && MODE == RW_SOFTMAX && elem == 4 && q.stream) {
        lds = 72 << 10;
        const hipError_t e = hipFuncSetAttribute((const void *)ttm_rowwise_band_k<MODE, 4, 4, 512>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
        if (e != hipSuccess) return ttm_set_error(TTM_ERR_HIP, "hipFuncSetAttribute(LDS %zu): %s", lds, hipGetErrorString(e));
      }
#define TTM_BAND(N, T) \
      do { if (dtype == TTM_BF16) hipLaunchKernelGGL((ttm_rowwise_band_k<MODE, 2, N, T>), grid, dim3(T), lds, s, q); \
           else hipLaunchKernelGGL((ttm_rowwise_band_k<MODE, 4, N, T>), grid, dim3(T), lds, s, q); } while (0)
      // lanes by width: measured per mode at 500 to 8192 rows.  RMSNorm of 3 and 4 chunks: [6738, 1920] bf16 10.4 us, 11.4 with 256 lanes
      // (softmax 11.5 / 11.1); 9 to 16 chunks: softmax [4000, 6000] bf16 26.8 with 512 lanes, 31.3 with 1024 (843 rows 9.5 / 8.4, RMSNorm
      // 26.5 / 23.1)
      if (nk <= 1) TTM_BAND(1, 256);
      else if (nk <= 2) TTM_BAND(2, 256);
      else if (nk <= 4) { if (MODE == RW_RMSNORM) TTM_BAND(2, 512); else TTM_BAND(4, 256); }
      else if (nk <= 8) TTM_BAND(4, 512);
      else if (nk <= 16) { if (MODE == RW_SOFTMAX && bands >= 256) TTM_BAND(8, 512); else TTM_BAND(4, 1024); }
      else TTM_BAND(8, 1024);
#undef TTM_BAND
      TTM_LAUNCH_CHECK();
      return TTM_OK;
    }
  }
  // few tile rows of very wide rows: slices of at least eight column tiles, enough of them for about 512 workgroups
  const bool row_kernel_fits = (MODE == RW_RMSNORM || MODE == RW_SOFTMAX) && p.ct * 2 * (dtype == TTM_BF16 ? 2 : 4) <= 8 * 256;
  if (p.ct >= 256 && !row_kernel_fits && trows * 2 <= 256 && ttm_option("rowwise_variant") == 0) {
    int slices = (int)(512 / trows);
    if (slices > p.ct / 8) slices = p.ct / 8;
    if (slices > 256) slices = 256;
    if (slices < 1) slices = 1;
    const int tps = (int)ttm_cdiv(p.ct, slices);
    slices = (int)ttm_cdiv(p.ct, tps);
    void *ws = nullptr;
    if (int rc = ttm_stream_workspace(s, (size_t)(trows * 32 * slices * 2) * sizeof(float), &ws)) return rc;
    const dim3 grid((unsigned)slices, (unsigned)trows);
    if (trows <= 65535) {
      if (dtype == TTM_BF16) hipLaunchKernelGGL((ttm_rowwise_wide_stats_k<MODE, 2>), grid, dim3(256), 0, s, p, (float *)ws, slices, tps);
      else hipLaunchKernelGGL((ttm_rowwise_wide_stats_k<MODE, 4>), grid, dim3(256), 0, s, p, (float *)ws, slices, tps);
      TTM_LAUNCH_CHECK();
      if constexpr (MODE == RW_RMSNORM || MODE == RW_SOFTMAX) {
        if (dtype == TTM_BF16) hipLaunchKernelGGL((ttm_rowwise_wide_apply_k<MODE, 2>), grid, dim3(256), 0, s, p, (const float *)ws, slices, tps);
        else hipLaunchKernelGGL((ttm_rowwise_wide_apply_k<MODE, 4>), grid, dim3(256), 0, s, p, (const float *)ws, slices, tps);
      } else {
        if (dtype == TTM_BF16) hipLaunchKernelGGL((ttm_rowwise_wide_finish_k<MODE, 2>), dim3((unsigned)trows), dim3(256), 0, s, p, (const float *)ws, slices);
        else hipLaunchKernelGGL((ttm_rowwise_wide_finish_k<MODE, 4>), dim3((unsigned)trows), dim3(256), 0, s, p, (const float *)ws, slices);
      }
      TTM_LAUNCH_CHECK();
      return TTM_OK;
    }
  }
  if constexpr (MODE == RW_RMSNORM || MODE == RW_SOFTMAX) {
    const int elem = dtype == TTM_BF16 ? 2 : 4;
    if (p.ct * 2 * elem <= 8 * 256 && trows * 32 < (1 << 24) && ttm_option("rowwise_variant") != 1) {   // one row per workgroup
      const int total = (int)(trows * 32), nq = p.ct * 2 * elem;
      const dim3 grid((unsigned)total);
#define TTM_ROW_LAUNCH(T) \
      do { if (dtype == TTM_BF16) hipLaunchKernelGGL((ttm_rowwise_row_k<MODE, 2, false, T>), grid, dim3(T), 0, s, p, total); \
           else hipLaunchKernelGGL((ttm_rowwise_row_k<MODE, 4, false, T>), grid, dim3(T), 0, s, p, total); } while (0)
      if (nq <= 512) TTM_ROW_LAUNCH(256);
      else if (nq <= 1024) TTM_ROW_LAUNCH(512);
      else TTM_ROW_LAUNCH(1024);
#undef TTM_ROW_LAUNCH
      TTM_LAUNCH_CHECK();
      return TTM_OK;
    }
    if (p.ct * 2 * elem <= 16 * 32) {   // a lane's share of the row fits in registers
      if (dtype == TTM_BF16) hipLaunchKernelGGL((ttm_rowwise_resident_k<MODE, 2>), dim3((unsigned)trows * 4), dim3(256), 0, s, p);
      else hipLaunchKernelGGL((ttm_rowwise_resident_k<MODE, 4>), dim3((unsigned)trows * 4), dim3(256), 0, s, p);
      TTM_LAUNCH_CHECK();
      return TTM_OK;
    }
  }
  if (trows >= 1024) {   // enough tile rows to fill the device with one workgroup each
    if (dtype == TTM_BF16) hipLaunchKernelGGL((ttm_rowwise_k<MODE, 2, 32>), dim3((unsigned)trows), dim3(256), 0, s, p);
    else hipLaunchKernelGGL((ttm_rowwise_k<MODE, 4, 32>), dim3((unsigned)trows), dim3(256), 0, s, p);
  } else {
    if (dtype == TTM_BF16) hipLaunchKernelGGL((ttm_rowwise_k<MODE, 2, 8>), dim3((unsigned)trows * 4), dim3(256), 0, s, p);
    else hipLaunchKernelGGL((ttm_rowwise_k<MODE, 4, 8>), dim3((unsigned)trows * 4), dim3(256), 0, s, p);
  }
  TTM_LAUNCH_CHECK();
  return TTM_OK;
}

static int fill_args(RowArgs &p, const void *x, void *out, int dtype, int64_t batch, int64_t rows, int64_t cols,
                     const char *who) {
  TTM_REQUIRE(dtype == TTM_BF16 || dtype == TTM_F32, "%s: dtype must be BFloat16 or Float32 (got %d)", who, dtype);
  TTM_REQUIRE(batch >= 0 && rows >= 0 && cols >= 0, "%s: negative dimension", who);
  TTM_REQUIRE(x && out, "%s: null pointer", who);
  TTM_REQUIRE(((uintptr_t)x & 15) == 0 && ((uintptr_t)out & 15) == 0, "%s: pointers must be 16-byte aligned", who);
  p.x = x; p.out = out; p.w = p.b = nullptr; p.w_tiled = p.b_tiled = 0;
  p.rows = rows; p.cols = (int)cols;
  p.rt = (int)ttm_cdiv(rows, 32); p.ct = (int)ttm_cdiv(cols, 32);
  p.eps = 0.0f; p.stream = 0;
  p.partial = nullptr; p.slices = 0; p.per = 0; p.residual = nullptr; p.sum_out = nullptr;
  return TTM_OK;
}

// RMSNorm of x = bf16(bf16(sum of the partial sums) + residual) for one row tile ([rows <= 32, cols] bf16 tiles), x
// stored to sum_out on the way: what ttm_linear_reduce_k with an add tail followed by ttm_rms_norm computes, with the
// kernel ttm_rms_norm itself uses at this size, so the two agree bit for bit.
bool ttm_rowwise_partials_supported(int64_t rows, int64_t cols) {
  const int v = ttm_option("rowwise_variant");
  return rows >= 1 && rows <= 32 && cols >= 1 && ttm_cdiv(cols, 32) * 4 <= 8 * 256 && (v == 0 || v == 3);
}
int ttm_rowwise_rmsnorm_from_partials(const float *partial, int slices, int64_t per, const void *residual, void *sum_out,
                                      const void *weight, int weight_layout, const void *bias, int bias_layout, void *out,
                                      int64_t rows, int64_t cols, float eps, hipStream_t s) {
  TTM_REQUIRE(ttm_rowwise_partials_supported(rows, cols), "rms_norm from partial sums: at most 32 rows and 16384 columns");
  RowArgs p;
  if (int rc = fill_args(p, residual, out, TTM_BF16, 1, rows, cols, "ttm_linear_add_rms_norm")) return rc;
  TTM_REQUIRE(partial && sum_out && slices >= 1, "rms_norm from partial sums: null pointer");
  TTM_REQUIRE((((uintptr_t)weight | (uintptr_t)bias | (uintptr_t)sum_out) & 15) == 0, "ttm_linear_add_rms_norm: operands must be 16-byte aligned");
  p.w = weight; p.b = bias; p.w_tiled = weight_layout == TTM_TILE; p.b_tiled = bias_layout == TTM_TILE; p.eps = eps;
  p.partial = partial; p.slices = slices; p.per = per; p.residual = residual; p.sum_out = sum_out;
  const int nq = p.ct * 4;
  const dim3 grid(32);
  if (nq <= 512) hipLaunchKernelGGL((ttm_rowwise_row_k<RW_RMSNORM, 2, true, 256>), grid, dim3(256), 0, s, p, 32);
  else if (nq <= 1024) hipLaunchKernelGGL((ttm_rowwise_row_k<RW_RMSNORM, 2, true, 512>), grid, dim3(512), 0, s, p, 32);
  else hipLaunchKernelGGL((ttm_rowwise_row_k<RW_RMSNORM, 2, true, 1024>), grid, dim3(1024), 0, s, p, 32);
  TTM_LAUNCH_CHECK();
  return TTM_OK;
}

TTM_EXPORT int ttm_rms_norm(const void *x, const void *weight, int weight_layout, const void *bias, int bias_layout,
                            void *out, int dtype, int64_t batch, int64_t rows, int64_t cols, float eps, void *stream) {
  TTM_EXTENTS(rms_norm, x, weight, weight_layout, bias, bias_layout, out, dtype, batch, rows, cols);
  if (batch == 0 || rows == 0 || cols == 0) return TTM_OK;
  RowArgs p;
  int rc = fill_args(p, x, out, dtype, batch, rows, cols, "ttm_rms_norm");
  if (rc) return rc;
  TTM_REQUIRE((((uintptr_t)weight | (uintptr_t)bias) & 15) == 0, "ttm_rms_norm: weight/bias must be 16-byte aligned");
  p.w = weight; p.b = bias; p.w_tiled = weight_layout == TTM_TILE; p.b_tiled = bias_layout == TTM_TILE; p.eps = eps;
  return launch_rowwise<RW_RMSNORM>(p, dtype, batch * p.rt, (hipStream_t)stream);
}

TTM_EXPORT int ttm_softmax_lastdim(const void *x, void *out, int dtype, int64_t batch, int64_t rows, int64_t cols,
                                   void *stream) {
  TTM_EXTENTS(softmax, x, out, dtype, batch, rows, cols);
  if (batch == 0 || rows == 0 || cols == 0) return TTM_OK;
  RowArgs p;
  int rc = fill_args(p, x, out, dtype, batch, rows, cols, "ttm_softmax_lastdim");
  if (rc) return rc;
  return launch_rowwise<RW_SOFTMAX>(p, dtype, batch * p.rt, (hipStream_t)stream);
}

TTM_EXPORT int ttm_reduce_lastdim(int op, const void *x, void *out, int dtype, int64_t batch, int64_t rows, int64_t cols,
                                  void *stream) {
  TTM_EXTENTS(reduce, x, out, dtype, batch, rows, cols);
  TTM_REQUIRE(op >= 0 && op <= 3, "ttm_reduce_lastdim: op must be Sum(0), Mean(1), Max(2) or Min(3), got %d", op);
  if (batch == 0 || rows == 0 || cols == 0) return TTM_OK;
  RowArgs p;
  int rc = fill_args(p, x, out, dtype, batch, rows, cols, "ttm_reduce_lastdim");
  if (rc) return rc;
  hipStream_t s = (hipStream_t)stream;
  switch (op) {
  case 0: return launch_rowwise<RW_SUM>(p, dtype, batch * p.rt, s);
  case 1: return launch_rowwise<RW_MEAN>(p, dtype, batch * p.rt, s);
  case 2: return launch_rowwise<RW_MAX>(p, dtype, batch * p.rt, s);
  default: return launch_rowwise<RW_MIN>(p, dtype, batch * p.rt, s);
  }
}
