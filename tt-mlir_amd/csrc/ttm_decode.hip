// Decode-path transformer kernels: rotary embedding, KV-cache update / fill, single-token attention over a KV cache.
// All tensors are TILE layout (32 x 32 tiles of four 16 x 16 faces); every kernel here is bound by HBM bandwidth.
#include <mutex>

#include "ttm_common.h"

namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4v __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));

// 8 consecutive elements <-> 8 floats
__device__ __forceinline__ void load8(const uint16_t *p, float *v) {
  const u32x4 r = *(const u32x4 *)p;
  const uint32_t w[4] = {r.x, r.y, r.z, r.w};
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    v[2 * j] = __uint_as_float(w[j] << 16);
    v[2 * j + 1] = __uint_as_float(w[j] & 0xFFFF0000u);
  }
}
__device__ __forceinline__ void load8(const float *p, float *v) {
  const f32x4 a = *(const f32x4 *)p, b = *(const f32x4 *)(p + 4);
  v[0] = a.x; v[1] = a.y; v[2] = a.z; v[3] = a.w; v[4] = b.x; v[5] = b.y; v[6] = b.z; v[7] = b.w;
}
__device__ __forceinline__ void store8(uint16_t *p, const float *v) {
  u32x4 r;
  r.x = ttm_pack_bf16x2(v[0], v[1]);
  r.y = ttm_pack_bf16x2(v[2], v[3]);
  r.z = ttm_pack_bf16x2(v[4], v[5]);
  r.w = ttm_pack_bf16x2(v[6], v[7]);
  *(u32x4 *)p = r;
}
__device__ __forceinline__ void store8(float *p, const float *v) {
  *(f32x4 *)p = f32x4{v[0], v[1], v[2], v[3]};
  *(f32x4 *)(p + 4) = f32x4{v[4], v[5], v[6], v[7]};
}

// ------------------------------------------------------------------------------------------------ rotary embedding
// out[b, s, d] = x[b, s, d] * cos[r, d] + rot(x)[b, s, d] * sin[r, d],  rot(x)[d] = d < D/2 ? -x[d + D/2] : x[d - D/2],
// r = token_index when given, else s.  One thread per 8 consecutive columns of a face row: the partner columns
// d +- D/2 are 8 consecutive elements of another face row because D/2 is a multiple of 16.
// src_cols > 0: x is not laid out like `out` but is the [batch, rows * cols] matrix a projection leaves (row b holds
// the `rows` heads of user b side by side); the head split [batch, rows * cols] -> [batch, rows, cols] happens on the
// way in and the padding rows of `out` are written as zeros.
template <typename T>
__global__ __launch_bounds__(256) void ttm_rotary_k(const T *__restrict__ x, const T *__restrict__ cosc,
                                                    const T *__restrict__ sinc, T *__restrict__ out, int64_t rows_pad,
                                                    int64_t cols, int64_t per_batch, int64_t total8, int64_t token_index,
                                                    int64_t rows, int64_t src_cols) {
  int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= total8) return;
  const int64_t ct = cols >> 5, half = cols >> 1;
  const int64_t e = i * 8, b = e / per_batch, o = e % per_batch;
  // o -> (row, col) of the tiled [rows_pad, cols] matrix
  const int64_t tile = o >> 10;
  const int in = (int)(o & 1023), face = in >> 8, fr = (in >> 4) & 15, fc = in & 15;
  const int64_t r = (tile / ct) * 32 + (face >> 1) * 16 + fr, c = (tile % ct) * 32 + (face & 1) * 16 + fc;
  const int64_t cr = token_index >= 0 ? token_index : r;
  const int64_t pc = c < half ? c + half : c - half;
  const float sign = c < half ? -1.0f : 1.0f;
  const T *xp = x + b * per_batch;
  const int64_t co = ttm_tiled_offset(cr, c, ct);
  float xv[8], pv[8], cv[8], sv[8], ov[8];
  if (src_cols > 0) {
    if (r >= rows) {
#pragma unroll
      for (int j = 0; j < 8; ++j) ov[j] = 0.0f;
      store8(out + b * per_batch + o, ov);
      return;
    }
    load8(x + ttm_tiled_offset(b, r * cols + c, src_cols >> 5), xv);
    load8(x + ttm_tiled_offset(b, r * cols + pc, src_cols >> 5), pv);
  } else {
    load8(xp + o, xv);
    load8(xp + ttm_tiled_offset(r, pc, ct), pv);
  }
  load8(cosc + co, cv);
  load8(sinc + co, sv);
#pragma unroll
  for (int j = 0; j < 8; ++j) ov[j] = ttm_rotary_value(xv[j], pv[j], cv[j], sv[j], sign);
  store8(out + b * per_batch + o, ov);
}

// ------------------------------------------------------------------------------------------------ cache update / fill
// cache[batch_offset + b, h, *index, :] = input[0, h, b, :]; one thread per 8 elements (never straddles a face row)
template <typename T>
__global__ __launch_bounds__(256) void ttm_update_cache_k(T *__restrict__ cache, const T *__restrict__ input,
                                                          const int32_t *__restrict__ index, int64_t heads, int64_t seq_pad,
                                                          int64_t max_seq, int64_t dim, int64_t in_users, int64_t in_users_pad,
                                                          int64_t batch_offset, int64_t total8) {
  int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= total8) return;
  const int64_t pos = index[0];
  if (pos < 0 || pos >= max_seq) return;          // out of range positions write nothing
  const int64_t d8 = dim >> 3;
  const int64_t c = (i % d8) * 8, b = (i / d8) % in_users, h = i / (d8 * in_users);
  const int64_t ct = dim >> 5;
  const T *src = input + h * in_users_pad * dim + ttm_tiled_offset(b, c, ct);
  T *dst = cache + ((batch_offset + b) * heads + h) * seq_pad * dim + ttm_tiled_offset(pos, c, ct);
  *(u32x4 *)dst = *(const u32x4 *)src;
  if (sizeof(T) == 4) *(u32x4 *)(dst + 4) = *(const u32x4 *)(src + 4);
}

// cache[batch_offset, h, 0:seq_tiles*32, :] = input[0, h, :, :] tile by tile (the padding rows of the last tile come along)
__global__ __launch_bounds__(256) void ttm_fill_cache_k(u32x4 *__restrict__ cache, const u32x4 *__restrict__ input,
                                                        int64_t head_stride_cache16, int64_t head_stride_in16, int64_t base16,
                                                        int64_t total16) {
  int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= total16) return;
  const int64_t h = i / head_stride_in16, o = i % head_stride_in16;
  cache[base16 + h * head_stride_cache16 + o] = input[i];
}

// Paged cache writes.  The cache is [blocks, heads, block_size, dim]; a user's positions live in the blocks its row of
// the page table names.  Without a page table the cache is [users, heads, max_seq, dim] (block_size = max_seq) and user
// u owns entry u (entry 0 for all users when the cache is shared).  Positions, page numbers and block numbers outside
// their ranges write nothing.
//
// update: cache[block(u, pos_u), h, pos_u % block_size, :] = input[0, u, h, :] with pos_u = index[u]; one thread per 8 elements
template <typename T>
__global__ __launch_bounds__(256) void ttm_paged_update_cache_k(T *__restrict__ cache, const T *__restrict__ input,
                                                                const int32_t *__restrict__ index, const int32_t *__restrict__ table,
                                                                int64_t blocks, int64_t heads, int64_t block_size, int64_t dim,
                                                                int64_t users, int64_t pages, int shared, int64_t total8) {
  int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= total8) return;
  const int64_t d8 = dim >> 3, ct = dim >> 5;
  const int64_t c = (i % d8) * 8, h = (i / d8) % heads, u = i / (d8 * heads);
  const int64_t pos = index[u];
  if (pos < 0) return;
  int64_t blk, off;
  if (table) {
    const int64_t page = pos / block_size;
    if (page >= pages) return;
    blk = table[u * pages + page];
    off = pos % block_size;
  } else {
    if (pos >= block_size) return;
    blk = shared ? 0 : u;
    off = pos;
  }
  if (blk < 0 || blk >= blocks) return;
  const int64_t heads_pad = ttm_round_up32(heads), bs_pad = ttm_round_up32(block_size);
  const T *src = input + u * heads_pad * dim + ttm_tiled_offset(h, c, ct);
  T *dst = cache + (blk * heads + h) * bs_pad * dim + ttm_tiled_offset(off, c, ct);
  *(u32x4 *)dst = *(const u32x4 *)src;
  if (sizeof(T) == 4) *(u32x4 *)(dst + 4) = *(const u32x4 *)(src + 4);
}

// fill: cache[table[row(b), s / block_size], h, s % block_size, :] = input[b, h, s, :] for s < seq, where row(b) is
// batch_idx[b] when given and b otherwise; one thread per 8 elements
template <typename T>
__global__ __launch_bounds__(256) void ttm_paged_fill_cache_k(T *__restrict__ cache, const T *__restrict__ input,
                                                              const int32_t *__restrict__ table, const int32_t *__restrict__ batch_idx,
                                                              int64_t blocks, int64_t heads, int64_t block_size, int64_t dim,
                                                              int64_t seq, int64_t table_rows, int64_t pages, int64_t total8) {
  int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= total8) return;
  const int64_t d8 = dim >> 3, ct = dim >> 5;
  const int64_t c = (i % d8) * 8, s = (i / d8) % seq, h = (i / (d8 * seq)) % heads, b = i / (d8 * seq * heads);
  const int64_t row = batch_idx ? batch_idx[b] : b;
  const int64_t page = s / block_size;
  if (row < 0 || row >= table_rows || page >= pages) return;
  const int64_t blk = table[row * pages + page];
  if (blk < 0 || blk >= blocks) return;
  const int64_t seq_pad = ttm_round_up32(seq), bs_pad = ttm_round_up32(block_size);
  const T *src = input + (b * heads + h) * seq_pad * dim + ttm_tiled_offset(s, c, ct);
  T *dst = cache + (blk * heads + h) * bs_pad * dim + ttm_tiled_offset(s % block_size, c, ct);
  *(u32x4 *)dst = *(const u32x4 *)src;
  if (sizeof(T) == 4) *(u32x4 *)(dst + 4) = *(const u32x4 *)(src + 4);
}

// gather: out[b, h, s, :] = cache[table[b, s / block_size], h, s % block_size, :] for s < pages * block_size, the inverse
// of the paged fill; positions whose page is outside the cache read as zeros; one thread per 8 elements
template <typename T>
__global__ __launch_bounds__(256) void ttm_paged_gather_k(const T *__restrict__ cache, const int32_t *__restrict__ table, T *__restrict__ out,
                                                          int64_t blocks, int64_t heads, int64_t block_size, int64_t dim, int64_t pages,
                                                          int64_t total8) {
  int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= total8) return;
  const int64_t d8 = dim >> 3, ct = dim >> 5, seq = pages * block_size;
  const int64_t c = (i % d8) * 8, s = (i / d8) % seq, h = (i / (d8 * seq)) % heads, b = i / (d8 * seq * heads);
  const int64_t blk = table[b * pages + s / block_size];
  T *dst = out + (b * heads + h) * seq * dim + ttm_tiled_offset(s, c, ct);
  u32x4 lo = {0, 0, 0, 0}, hi = {0, 0, 0, 0};
  if (blk >= 0 && blk < blocks) {
    const T *src = cache + (blk * heads + h) * block_size * dim + ttm_tiled_offset(s % block_size, c, ct);
    lo = *(const u32x4 *)src;
    if (sizeof(T) == 4) hi = *(const u32x4 *)(src + 4);
  }
  *(u32x4 *)dst = lo;
  if (sizeof(T) == 4) *(u32x4 *)(dst + 4) = hi;
}

// additive mask of a prefill chunk: query row i stands at absolute position *start + i and sees the keys up to it;
// mask[i, j] = 0 where j <= *start + i, -inf elsewhere.  bf16 tiles [rows_pad, cols_pad]; the offset is read from device
// memory, so the launch can be recorded into a graph and replayed for the next chunk
__global__ __launch_bounds__(256) void ttm_chunk_mask_k(uint16_t *__restrict__ mask, const int32_t *__restrict__ start, int64_t rows_pad,
                                                        int64_t cols_pad, int64_t total8) {
  int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= total8) return;
  const int64_t c8 = cols_pad >> 3, r = i / c8, c = (i % c8) * 8;
  const int64_t limit = (int64_t)start[0] + r;
  uint32_t w[4];
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const uint32_t lo = c + 2 * k <= limit ? 0u : 0xFF80u, hi = c + 2 * k + 1 <= limit ? 0u : 0xFF80u;
    w[k] = lo | (hi << 16);
  }
  *(u32x4 *)(mask + ttm_tiled_offset(r, c, cols_pad >> 5)) = u32x4{w[0], w[1], w[2], w[3]};
}

// rotary embedding with a transformation matrix: out = x * cos + (x T) * sin, where T is a 32 x 32 matrix applied to
// every 32-column tile of a row (for the matrix Llama uses this rotates the interleaved pairs (x[2i], x[2i+1])).
// x / out [batch, rows, cols] tiles; cos / sin [cs_batch, cs_rows, cols] tiles, row r of batch entry b reads cos row
// (r if cs_rows > 1 else 0) of entry (b % cs_batch if cs_batch > 1 else 0).  One thread per element; T sits in LDS.
__global__ __launch_bounds__(256) void ttm_rotary_llama_k(const uint16_t *__restrict__ x, const uint16_t *__restrict__ cosc,
                                                          const uint16_t *__restrict__ sinc, const uint16_t *__restrict__ tmat,
                                                          uint16_t *__restrict__ out, int64_t rows, int64_t rows_pad, int64_t cols,
                                                          int64_t cs_batch, int64_t cs_rows, int64_t cs_rows_pad, int64_t total) {
  __shared__ float T[32][33];
  for (int e = threadIdx.x; e < 1024; e += 256) T[e >> 5][e & 31] = ttm_bf16_to_f32(tmat[ttm_tiled_offset(e >> 5, e & 31, 1)]);
  __syncthreads();
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= total) return;
  const int64_t c = i % cols, r = (i / cols) % rows_pad, b = i / (cols * rows_pad), ct = cols >> 5;
  const int64_t off = b * rows_pad * cols + ttm_tiled_offset(r, c, ct);
  if (r >= rows) { out[off] = 0; return; }   // tile padding stays zero
  const int64_t cb = cs_batch > 1 ? b % cs_batch : 0, cr = cs_rows > 1 ? r : 0;
  const int64_t coff = cb * cs_rows_pad * cols + ttm_tiled_offset(cr, c, ct);
  const uint16_t *xr = x + b * rows_pad * cols;
  float rot = 0.0f;
  const int64_t c0 = c & ~(int64_t)31;
#pragma unroll 8
  for (int j = 0; j < 32; ++j) rot += ttm_bf16_to_f32(xr[ttm_tiled_offset(r, c0 + j, ct)]) * T[j][c & 31];
  // fp32 throughout, one rounding at the end (the convention of the CPU path: compute in f32, cast back)
  out[off] = ttm_f32_to_bf16(ttm_bf16_to_f32(x[off]) * ttm_bf16_to_f32(cosc[coff]) + rot * ttm_bf16_to_f32(sinc[coff]));
}

// ------------------------------------------------------------------------------------------------ attention, one query token
// q [1, B, H, D], k / v [B, Hkv, S, D] (or pages [blocks, Hkv, block, D] behind a page table), out [1, B, H, D], bf16 tiles.
// HBM-bound: K and V up to the users' positions are read once.  A workgroup owns the G = H / Hkv query heads of one kv head and a
// range of 32-key tiles; its wavefronts take the tiles in turn, each with a running maximum, sum and output of its own:
//   scores = K Q^T with v_mfma_f32_16x16x32_bf16 (keys are the rows, heads the columns: a lane holds four consecutive keys of one
//   head), softmax numerators against the running maximum, rounded to bf16 and exchanged through 16 G dwords of LDS, then P V on
//   the vector ALU with v_dot2_f32_bf16: a lane owns two adjacent columns for all keys of the tile, so nothing is summed across lanes.
// The next tile's K is requested when the scores are made, its V behind the products, so a wavefront has 16 KiB (D = 128) on the
// way at any time and no wavefront waits for another before the end, where the partial results meet in LDS.
//
// Two forms.  Direct: grid (Hkv, B), 16 wavefronts for up to four heads of 32, 64 or 128 columns, else eight; the whole context of a
// user and the output in one launch.  Shares, four wavefronts: the visible tiles of all users of a kv head form one line (user after
// user), workgroup j of grid (shares, Hkv) streams its j-th equal part whatever the users' context lengths are; (max, sum,
// unnormalised output) of a piece go to slot j + user of the kv head (along the line either j or the user advances from one piece
// to the next, so the sum numbers the pieces) and ttm_sdpa_decode_combine_k merges a user's slots (merging in the last workgroup to
// arrive was measured: the device-scope fences it needs double the kernel time).
struct DecodeArgs {
  const uint16_t *q, *k, *v, *mask;
  const int32_t *cur_pos, *page_table;
  float *part;        // [Hkv][shares + B][G][D + 2]
  uint16_t *out;
  int B, H, Hkv, G, S, D, shares, block, pages_per_user, mask_heads, is_causal;
  int blocks;         // number of blocks in a paged cache: page-table entries outside [0, blocks) are masked
  int concat_heads;   // out is [B, H * D] (row b holds user b's heads side by side) instead of [B, H, D]
  int Gt, g0;         // query heads per kv head in the tensors, and the first of them this launch serves (it serves G of them)
  int mask_b;         // 1: one mask per user, 0: one mask shared by all
  int window;         // >= 0: only the last `window` keys up to the decode position are visible
  const uint16_t *sink;   // [H, 32] in tiles, column 0: one more logit per head (times scale) with a zero value row; or null
  float scale;
  __device__ __forceinline__ const DecodeArgs &full() const { return *this; }
};
// The same without mask and sink, in the 112 bytes that launch quickly (ttm_common.h)
struct DecodeLean {
  const uint16_t *q, *k, *v;
  const int32_t *cur_pos, *page_table;
  float *part;
  uint16_t *out;
  int B, Hkv, S, shares, block, pages_per_user, blocks, Gt, g0, window;
  float scale;
  uint16_t D;
  uint8_t G, flags;
  explicit DecodeLean(const DecodeArgs &a)
      : q(a.q), k(a.k), v(a.v), cur_pos(a.cur_pos), page_table(a.page_table), part(a.part), out(a.out), B(a.B), Hkv(a.Hkv), S(a.S), shares(a.shares),
        block(a.block), pages_per_user(a.pages_per_user), blocks(a.blocks), Gt(a.Gt), g0(a.g0), window(a.window), scale(a.scale), D((uint16_t)a.D),
        G((uint8_t)a.G), flags((uint8_t)((a.is_causal ? 1 : 0) | (a.concat_heads ? 2 : 0))) {}
  __device__ __forceinline__ DecodeArgs full() const {
    DecodeArgs p = {};
    p.q = q; p.k = k; p.v = v; p.cur_pos = cur_pos; p.page_table = page_table; p.part = part; p.out = out;
    p.B = B; p.H = Hkv * Gt; p.Hkv = Hkv; p.G = G; p.S = S; p.D = D; p.shares = shares; p.block = block; p.pages_per_user = pages_per_user;
    p.is_causal = flags & 1; p.blocks = blocks; p.concat_heads = flags >> 1; p.Gt = Gt; p.g0 = g0; p.window = window; p.scale = scale;
    return p;
  }
};
static_assert(sizeof(DecodeLean) <= 112, "the size up to which a launch is quick");

constexpr int kMaxG = 8;
// K is read by streaming (nontemporal) loads: each line once per launch, by one instruction.  STREAM = false when several launches
// share one cache (more than kMaxG query heads per kv head), where the later launches profit from what the first one left.  V's
// loads are plain ones: a lane takes a dword of every row, so a line is fetched by four instructions and has to stay until the last.
template <bool STREAM, typename T>
__device__ __forceinline__ T kv_load(const T *p) {
  if constexpr (STREAM) return __builtin_nontemporal_load(p);
  else return *p;
}
constexpr int kDecodeBlocks = 512;   // workgroups of the shares form: two of four wavefronts per CU

// the visible keys of user b: [lo, valid); tiles in front of lo's are not read at all
__device__ __forceinline__ void visible_keys(const DecodeArgs &p, int b, int &lo, int &valid) {
  valid = p.S;
  int pos = p.S - 1;
  if (p.cur_pos) {
    pos = p.cur_pos[b];
    if (p.is_causal) valid = min(max(pos + 1, 0), p.S);
  }
  lo = p.window >= 0 && pos + 1 > p.window ? pos + 1 - p.window : 0;
}
__device__ __forceinline__ int visible_tiles(const DecodeArgs &p, int b) {
  int lo, valid;
  visible_keys(p, b, lo, valid);
  return max(((valid + 31) >> 5) - (lo >> 5), 0);
}
// inclusive sum over the lanes of a wavefront, DPP moves only
__device__ __forceinline__ int wave_scan(int v) {
  v += __builtin_amdgcn_update_dpp(0, v, 0x111, 0xF, 0xF, false);   // row_shr 1, 2, 4, 8
  v += __builtin_amdgcn_update_dpp(0, v, 0x112, 0xF, 0xF, false);
  v += __builtin_amdgcn_update_dpp(0, v, 0x114, 0xF, 0xF, false);
  v += __builtin_amdgcn_update_dpp(0, v, 0x118, 0xF, 0xF, false);
  v += __builtin_amdgcn_update_dpp(0, v, 0x142, 0xA, 0xF, false);   // row_bcast 15 into rows 1 and 3, row_bcast 31 into rows 2 and 3
  v += __builtin_amdgcn_update_dpp(0, v, 0x143, 0xC, 0xF, false);
  return v;
}
// tiles of the users in front of user b0 + lane (exclusive sum) for the chunk of 64 users that holds user b, and all users' tiles
__device__ __forceinline__ void line_of(const DecodeArgs &p, int b, int lane, int &before, int &mine, int &total) {
  total = before = mine = 0;
  for (int b0 = 0; b0 < p.B; b0 += 64) {
    const int own = b0 + lane < p.B ? visible_tiles(p, b0 + lane) : 0, sum = wave_scan(own);
    if (b >= b0 && b < b0 + 64) {
      mine = __builtin_amdgcn_readlane(own, b - b0);
      before = total + __builtin_amdgcn_readlane(sum, b - b0) - mine;
    }
    total += __builtin_amdgcn_readlane(sum, 63);
  }
}
// first tile of share j (the host keeps tiles x shares below 2^31)
__device__ __forceinline__ int share_begin(int total, int shares, int j) { return (int)((uint32_t)(total * j) / (uint32_t)shares); }

__device__ __forceinline__ int64_t kv_tile_row(const DecodeArgs &p, int b, int hk, int key_tile, bool &ok) {
  // first element of the row of tiles holding keys [32 key_tile, 32 key_tile + 32) of (b, hk).  A page-table entry outside the
  // cache's blocks (an unused slot, -1) gives ok = false and the address of block 0: the caller treats those keys as masked
  const int64_t row_elems = (int64_t)32 * p.D;
  ok = true;
  if (p.page_table) {
    const int tiles_per_block = p.block >> 5;
    int page = p.page_table[(int64_t)b * p.pages_per_user + key_tile / tiles_per_block];
    ok = page >= 0 && page < p.blocks;
    page = ok ? page : 0;
    return (((int64_t)page * p.Hkv + hk) * tiles_per_block + key_tile % tiles_per_block) * row_elems;
  }
  return (((int64_t)b * p.Hkv + hk) * (p.S >> 5) + key_tile) * row_elems;
}

// the output of head h of user b, column c; padding columns do not exist (D is a multiple of 32)
__device__ __forceinline__ void store_head(const DecodeArgs &p, int b, int h, int c, float v) {
  const uint16_t val = ttm_f32_to_bf16(v);
  if (p.concat_heads) p.out[ttm_tiled_offset(b, h * p.D + c, (p.H * p.D) >> 5)] = val;
  else p.out[(int64_t)b * ttm_round_up32(p.H) * p.D + ttm_tiled_offset(h, c, p.D >> 5)] = val;
}
// zeros in the padding rows of the output, by the workgroup(s) of the last user / last kv head
__device__ __forceinline__ void store_padding(const DecodeArgs &p, int b, int hk, int tid, int threads) {
  const int G = p.G, D = p.D;
  if (p.concat_heads) {   // padding rows below the last user, this kv head's columns
    if (b == p.B - 1) {
      const int pad = (int)ttm_round_up32(p.B) - p.B;
      for (int i = tid; i < pad * G * D; i += threads)
        p.out[ttm_tiled_offset(p.B + i / (G * D), (hk * p.Gt + p.g0) * D + i % (G * D), (p.H * D) >> 5)] = 0;
    }
  } else if (hk == p.Hkv - 1 && p.g0 + G == p.Gt) {   // padding rows of the last head tile
    const int pad = (int)ttm_round_up32(p.H) - p.H;
    for (int i = tid; i < pad * D; i += threads)
      p.out[(int64_t)b * ttm_round_up32(p.H) * D + ttm_tiled_offset(p.H + i / D, i % D, D >> 5)] = 0;
  }
}

// GM: most query heads, DM: most column tiles (1, 2, 4, 8), NW: wavefronts
template <bool STREAM, int GM, int DM, bool EXACT, int NW, bool DIRECT, class ARGS>
__global__ __launch_bounds__(NW * 64, NW == 16 ? 4 : 2) void ttm_sdpa_decode_k(ARGS args) {
  const DecodeArgs p = args.full();
  constexpr int KS = DM >= 4 ? 1 : 4 / DM;   // lanes of a column pair that share the tile's keys
  constexpr int NP = DM > 4 ? 2 : 1;         // column pairs of a lane
  constexpr int KEYS = 32 / KS;              // keys of a tile a lane multiplies
  __shared__ uint32_t pbuf[NW][GM][16];      // softmax numerators of a tile: pairs of adjacent keys
  __shared__ float om[NW][GM][2];            // max, sum
  extern __shared__ float oo[];              // [NW][G][D] outputs
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int G = p.G, D = EXACT ? 32 * DM : p.D, DT = D >> 5;
  const int hk = DIRECT ? blockIdx.x : blockIdx.y;
  int t0 = 0, t1 = 0, b = 0, first = 0;   // the share's tiles on the line, the user it begins in and that user's first tile
  if (DIRECT) {
    b = blockIdx.y;
    t1 = visible_tiles(p, b);
  } else {
    int unused, total;
    line_of(p, 0, lane, unused, unused, total);
    t0 = share_begin(total, p.shares, blockIdx.x);
    t1 = share_begin(total, p.shares, blockIdx.x + 1);
    if (t0 >= t1) return;
    for (int b0 = 0; b0 < p.B; b0 += 64) {
      const int own = b0 + lane < p.B ? visible_tiles(p, b0 + lane) : 0;
      const int n = wave_scan(own);
      const uint64_t past = __ballot(first + n > t0);   // users that end behind t0
      if (past) {
        const int l = __ffsll((unsigned long long)past) - 1;
        b = b0 + l;
        first += __builtin_amdgcn_readlane(n - own, l);
        break;
      }
      first += __builtin_amdgcn_readlane(n, 63);
    }
    b = __builtin_amdgcn_readfirstlane(b);
    first = __builtin_amdgcn_readfirstlane(first);
  }
  // lane roles: score phase (head hq, keys 4 kq .. + 3 of 16), product phase (column pairs cp + 64 i, keys KEYS ks .. of 32)
  const int hq = lane & 15, kq = lane >> 4, dq = kq * 8;
  const int cp = DM == 1 ? lane & 15 : DM == 2 ? lane & 31 : lane, ks = DM == 1 ? lane >> 4 : DM == 2 ? lane >> 5 : 0;
  const int k_off = (dq >> 4) * 256 + hq * 16 + (dq & 15);   // inside a tile; + 512 for keys 16 .. 31 (A operand row = lane % 16)
  int v_off[NP];
#pragma unroll
  for (int n = 0; n < NP; ++n) {
    const int c = 2 * min(cp + 64 * n, 16 * DT - 1);
    v_off[n] = (c >> 5) * 1024 + ((c >> 4) & 1) * 256 + (c & 15) + ks * (KEYS == 8 ? 0 : 512);
    if (KEYS == 8) v_off[n] += (ks >> 1) * 512 + (ks & 1) * 128;
  }
  // (the line's last user ends the loop: t1 is at most the total)
  for (int next; first < t1 || DIRECT; ++b, first = next) {   // workgroup-uniform
  next = DIRECT ? t1 : first + visible_tiles(p, b);
  if (!DIRECT && next == first) continue;
  int lo, valid;
  visible_keys(p, b, lo, valid);
  const int tb = (lo >> 5) - first;                 // tile on the line + tb = tile of the user's cache
  const int ta = max(t0, first), tz = min(t1, next);
  // query fragments: lane supplies head lane % 16, columns 32 c + 8 (lane / 16) .. + 7
  bf16x8 qf[DM];
  const uint16_t *qb = p.q + (int64_t)b * ttm_round_up32(p.H) * D;
#pragma unroll
  for (int c = 0; c < DM; ++c) {
    u32x4 z = {0, 0, 0, 0};
    if (c < DT && hq < G) z = *(const u32x4 *)(qb + ttm_tiled_offset(hk * p.Gt + p.g0 + hq, 32 * c + dq, DT));
    qf[c] = *(bf16x8 *)&z;
  }
  float m = -INFINITY, l = 0.0f, o[GM][NP][2];
#pragma unroll
  for (int g = 0; g < GM; ++g)
#pragma unroll
    for (int n = 0; n < NP; ++n) o[g][n][0] = o[g][n][1] = 0.0f;
  u32x4 kf[2][DM];
  uint32_t vf[NP][KEYS];
  bool kok = true, vok = true;
  int64_t krow = 0, vrow = 0;
  auto load_k = [&](int t) __attribute__((always_inline)) {
    krow = kv_tile_row(p, b, hk, t + tb, kok);
    const uint16_t *kt = p.k + krow + k_off;
#pragma unroll
    for (int u = 0; u < 2; ++u)
#pragma unroll
      for (int c = 0; c < DM; ++c)
        if (c < DT) kf[u][c] = kv_load<STREAM>((const u32x4 *)(kt + c * 1024 + u * 512));
  };
  auto load_v = [&]() __attribute__((always_inline)) {   // of the tile whose K was requested last
    vrow = krow;
    vok = kok;
    const uint16_t *vt = p.v + vrow;
#pragma unroll
    for (int n = 0; n < NP; ++n)
#pragma unroll
      for (int r = 0; r < KEYS; ++r)   // four rows share a line
        vf[n][r] = *(const uint32_t *)(vt + v_off[n] + (r >> 4) * 512 + (r & 15) * 16);
  };
  int t = ta + wave;
  if (t < tz) { load_k(t); load_v(); }
  for (; t < tz; t += NW) {
    const int kb = (t + tb) * 32;   // first key
    f32x4 s[2];
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      s[u] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
      for (int c = 0; c < DM; ++c)
        if (c < DT) s[u] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(*(bf16x8 *)&kf[u][c], qf[c], s[u], 0, 0, 0);
    }
    const bool ok = kok;
    // pins the products in front of the loads that overwrite their operands (left to itself the compiler copies the 64 registers
    // and multiplies behind the next tile's requests)
    asm volatile("" : "+v"(s[0]), "+v"(s[1]));
    if (t + NW < tz) load_k(t + NW);   // wavefront-uniform
    const bool inner = ok && kb >= lo && kb + 32 <= valid;   // wavefront-uniform: every key of the tile is visible
    float tm = -INFINITY;
#pragma unroll
    for (int u = 0; u < 2; ++u)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int key = kb + u * 16 + kq * 4 + i;
        float x = s[u][i];
        if (p.mask && hq < G) {
          const int mh = p.mask_heads == 1 ? 0 : hk * p.Gt + p.g0 + hq;
          x += ttm_bf16_to_f32(p.mask[(int64_t)b * p.mask_b * ttm_round_up32(p.mask_heads) * p.S + ttm_tiled_offset(mh, key, p.S >> 5)]);
        }
        x *= p.scale;
        s[u][i] = inner || (ok && key >= lo && key < valid) ? x : -INFINITY;
        tm = fmaxf(tm, s[u][i]);
      }
    tm = fmaxf(tm, __shfl_xor(tm, 16));
    tm = fmaxf(tm, __shfl_xor(tm, 32));
    const float mn = fmaxf(m, tm);
    const float alpha = m == mn ? 1.0f : __expf(m - mn);      // (-inf, -inf) -> 1, (-inf, finite) -> 0
    l *= alpha;
    m = mn;
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      uint32_t pair[2];
#pragma unroll
      for (int e = 0; e < 2; ++e) {
        const float x = s[u][2 * e], y = s[u][2 * e + 1];
        pair[e] = ttm_pack_bf16x2(x == -INFINITY ? 0.0f : __expf(x - mn), y == -INFINITY ? 0.0f : __expf(y - mn));
        l += __uint_as_float(pair[e] << 16) + __uint_as_float(pair[e] & 0xFFFF0000u);   // numerator and denominator see the same rounding
      }
      if (hq < GM) *(u32x2 *)&pbuf[wave][hq][u * 8 + kq * 2] = u32x2{pair[0], pair[1]};
    }
    if (__any(alpha != 1.0f && hq < GM)) {
#pragma unroll
      for (int g = 0; g < GM; ++g) {
        const float ag = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(alpha), g));
#pragma unroll
        for (int n = 0; n < NP; ++n) { o[g][n][0] *= ag; o[g][n][1] *= ag; }
      }
    }
    // LDS traffic of one wavefront is processed in order; the fence only pins the compiler's order
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
    if (!inner) {   // rows outside the visible keys may hold anything, NaN included
#pragma unroll
      for (int r = 0; r < KEYS; ++r) {
        const int key = kb + ks * KEYS + r;
        const bool in = ok && key >= lo && key < valid;
#pragma unroll
        for (int n = 0; n < NP; ++n) vf[n][r] = in ? vf[n][r] : 0u;
      }
    }
#pragma unroll
    for (int j = 0; j < KEYS / 2; j += 4) {
      uint32_t vp[NP][4][2];   // (key 2 j, key 2 j + 1) of either column
#pragma unroll
      for (int n = 0; n < NP; ++n)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          vp[n][e][0] = __builtin_amdgcn_perm(vf[n][2 * (j + e) + 1], vf[n][2 * (j + e)], 0x05040100u);
          vp[n][e][1] = __builtin_amdgcn_perm(vf[n][2 * (j + e) + 1], vf[n][2 * (j + e)], 0x07060302u);
        }
#pragma unroll
      for (int g = 0; g < GM; ++g) {
        const u32x4 pg = *(const u32x4 *)&pbuf[wave][g][ks * (KEYS / 2) + j];
#pragma unroll
        for (int e = 0; e < 4; ++e)
#pragma unroll
          for (int n = 0; n < NP; ++n) {
            const uint32_t pe = pg[e];
            o[g][n][0] = __builtin_amdgcn_fdot2_f32_bf16(*(bf16x2 *)&vp[n][e][0], *(const bf16x2 *)&pe, o[g][n][0], false);
            o[g][n][1] = __builtin_amdgcn_fdot2_f32_bf16(*(bf16x2 *)&vp[n][e][1], *(const bf16x2 *)&pe, o[g][n][1], false);
          }
      }
      __builtin_amdgcn_sched_barrier(0);   // eight keys at a time: all numerators and pairs at once do not fit the registers
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
#pragma unroll
    for (int g = 0; g < GM; ++g)
#pragma unroll
      for (int n = 0; n < NP; ++n) asm volatile("" : "+v"(o[g][n][0]), "+v"(o[g][n][1]));
    if (t + NW < tz) load_v();
  }
  // the wavefronts' results meet in LDS
  l += __shfl_xor(l, 16);
  l += __shfl_xor(l, 32);
  if (kq == 0 && hq < GM) { om[wave][hq][0] = m; om[wave][hq][1] = l; }
#pragma unroll
  for (int g = 0; g < GM; ++g) {
    if (g < G) {
#pragma unroll
      for (int n = 0; n < NP; ++n) {
        float x = o[g][n][0], y = o[g][n][1];
        if (KS >= 2) { x += __shfl_xor(x, 32); y += __shfl_xor(y, 32); }
        if (KS == 4) { x += __shfl_xor(x, 16); y += __shfl_xor(y, 16); }
        if (ks == 0 && cp + 64 * n < 16 * DT) {
          oo[(wave * G + g) * D + 2 * (cp + 64 * n)] = x;
          oo[(wave * G + g) * D + 2 * (cp + 64 * n) + 1] = y;
        }
      }
    }
  }
  __syncthreads();
  float *slot = DIRECT ? nullptr : p.part + ((size_t)hk * (p.shares + p.B) + blockIdx.x + b) * G * (D + 2);
  for (int i = tid; i < G * D; i += NW * 64) {
    const int g = i / D, c = i - g * D, h = hk * p.Gt + p.g0 + g;
    const float sinkv = DIRECT && p.sink ? ttm_bf16_to_f32(p.sink[ttm_tiled_offset(h, 0, 1)]) * p.scale : -INFINITY;
    float M = sinkv;
#pragma unroll
    for (int w = 0; w < NW; ++w) M = fmaxf(M, om[w][g][0]);
    float num = 0.0f, den = 0.0f;
#pragma unroll
    for (int w = 0; w < NW; ++w) {
      const float e = om[w][g][0] == -INFINITY ? 0.0f : __expf(om[w][g][0] - M);
      num += oo[(w * G + g) * D + c] * e;
      den += om[w][g][1] * e;
    }
    if (DIRECT) {
      if (p.sink) den += __expf(sinkv - M);
      store_head(p, b, h, c, den > 0.0f ? num / den : 0.0f);
    } else {
      slot[g * (D + 2) + c] = num;
      if (c == 0) { slot[g * (D + 2) + D] = M; slot[g * (D + 2) + D + 1] = den; }
    }
  }
  if (DIRECT) {
    store_padding(p, b, hk, tid, NW * 64);
    return;
  }
  __syncthreads();   // the next user's piece reuses the arrays
  }  // users of this share
}

// merges a user's slots: out = sum_s o_s exp(m_s - M) / sum_s l_s exp(m_s - M).  grid (B * Hkv, G), 256 lanes: a workgroup per head,
// 256 / D lanes of it share a column and take every (256 / D)-th slot.  Bound by the memory round trips that follow each other (a few
// hundred KiB in all), so there are two: the users' positions, then a lane's maxima and sums together with its first eight
// numerators, which do not wait for the weights.  5 users x 4 heads of 4 kv heads, 1300 keys on average (about 20 slots each):
// both launches 27.4 us with a workgroup per 256 outputs, one head after the other and numerators behind the weights -> 13.9 us.
template <class ARGS>
__global__ __launch_bounds__(256) void ttm_sdpa_decode_combine_k(ARGS args) {
  const DecodeArgs p = args.full();
  __shared__ float wgt[kDecodeBlocks];   // a user's slots lie in at most that many shares
  __shared__ float red[256];
  __shared__ float tops[4], sums[4];
  constexpr int kAhead = 8;
  const int bh = blockIdx.x, g = blockIdx.y, tid = threadIdx.x;
  const int b = bh / p.Hkv, hk = bh % p.Hkv;
  const int G = p.G, D = p.D, h = hk * p.Gt + p.g0 + g;
  // the user's tiles on the line and the shares that hold them
  int before, total, mine;
  line_of(p, b, tid & 63, before, mine, total);
  // share of tile t: the last one that begins at or before it
  auto share_of = [&](int t) { return (int)(((uint32_t)((t + 1) * p.shares) - 1u) / (uint32_t)total); };
  const int j0 = mine ? share_of(before) : 0, S = mine ? share_of(before + mine - 1) - j0 + 1 : 0;
  const bool gaps = total < p.shares;   // fewer tiles than shares: some of them are empty and left their slots as they were
  auto filled = [&](int s) { return s < S && !(gaps && share_begin(total, p.shares, j0 + s) == share_begin(total, p.shares, j0 + s + 1)); };
  const float *base = p.part + (((size_t)hk * (p.shares + p.B) + j0 + b) * G + g) * (D + 2);   // piece s: + s * sstride
  const size_t sstride = (size_t)G * (D + 2);
  const int nsub = 256 / D, c = tid % D, sub = tid / D;
  const float sinkv = p.sink ? ttm_bf16_to_f32(p.sink[ttm_tiled_offset(h, 0, 1)]) * p.scale : -INFINITY;
  float ms[kDecodeBlocks / 256], ls[kDecodeBlocks / 256], ahead[kAhead];
#pragma unroll
  for (int i = 0; i < kDecodeBlocks / 256; ++i) {
    const bool in = filled(tid + 256 * i);
    ms[i] = in ? base[(tid + 256 * i) * sstride + D] : -INFINITY;
    ls[i] = in ? base[(tid + 256 * i) * sstride + D + 1] : 0.0f;
  }
#pragma unroll
  for (int k = 0; k < kAhead; ++k) {
    const int s = sub + nsub * k;
    ahead[k] = sub < nsub && filled(s) ? base[s * sstride + c] : 0.0f;
  }
  float M = sinkv;
#pragma unroll
  for (int i = 0; i < kDecodeBlocks / 256; ++i) M = fmaxf(M, ms[i]);
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) M = fmaxf(M, __shfl_xor(M, o));
  if ((tid & 63) == 0) tops[tid >> 6] = M;
  __syncthreads();
  M = fmaxf(fmaxf(tops[0], tops[1]), fmaxf(tops[2], tops[3]));
  float den = 0.0f, num = 0.0f;
#pragma unroll
  for (int i = 0; i < kDecodeBlocks / 256; ++i) {
    const float w = ms[i] == -INFINITY ? 0.0f : __expf(ms[i] - M);
    wgt[tid + 256 * i] = w;
    den += ls[i] * w;
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) den += __shfl_xor(den, o);
  if ((tid & 63) == 0) sums[tid >> 6] = den;
  __syncthreads();
  if (sub < nsub) {
#pragma unroll
    for (int k = 0; k < kAhead; ++k)
      if (sub + nsub * k < S) num += ahead[k] * wgt[sub + nsub * k];
    if (gaps) {
      for (int s = sub + nsub * kAhead; s < S; s += nsub)
        if (wgt[s] != 0.0f) num += base[s * sstride + c] * wgt[s];
    } else {
#pragma unroll 8
      for (int s = sub + nsub * kAhead; s < S; s += nsub) num += base[s * sstride + c] * wgt[s];
    }
  }
  red[tid] = num;
  __syncthreads();
  den = (sums[0] + sums[1]) + (sums[2] + sums[3]) + (p.sink ? __expf(sinkv - M) : 0.0f);
  if (sub == 0) {
    for (int u = 1; u < nsub; ++u) num += red[tid + u * D];
    store_head(p, b, h, c, den > 0.0f ? num / den : 0.0f);
  }
  if (g == 0) store_padding(p, b, hk, tid, 256);   // the padding belongs to the first head's workgroup
}

}  // namespace

static int rotary_entry(const void *x, const void *cos_cache, const void *sin_cache, void *out, int dtype, int64_t batch, int64_t rows,
                        int64_t cols, int64_t cache_rows, int64_t token_index, bool split, void *stream) {
  TTM_REQUIRE(x && cos_cache && sin_cache && out, "ttm_rotary_embedding: null pointer");
  TTM_REQUIRE(!split || token_index >= 0, "ttm_rotary_embedding_split_heads: rows are heads here, so the position must come from token_index");
  TTM_REQUIRE(dtype == TTM_BF16 || dtype == TTM_F32, "ttm_rotary_embedding: dtype must be BFloat16 or Float32");
  TTM_REQUIRE(batch >= 0 && rows > 0 && cols > 0 && cols % 32 == 0, "ttm_rotary_embedding: head dim must be a positive multiple of 32");
  if (token_index >= 0)
    TTM_REQUIRE(token_index < cache_rows, "ttm_rotary_embedding: token_index %lld outside the %lld cached positions",
                (long long)token_index, (long long)cache_rows);
  else
    TTM_REQUIRE(cache_rows >= rows, "ttm_rotary_embedding: cos / sin caches hold %lld positions, input has %lld",
                (long long)cache_rows, (long long)rows);
  if (batch == 0) return TTM_OK;
  const int64_t rows_pad = ttm_round_up32(rows), per_batch = rows_pad * cols, total8 = batch * per_batch / 8;
  const int64_t src_cols = split ? rows * cols : 0;
  const dim3 grid((unsigned)ttm_cdiv(total8, 256));
  if (dtype == TTM_BF16)
    hipLaunchKernelGGL(ttm_rotary_k<uint16_t>, grid, dim3(256), 0, (hipStream_t)stream, (const uint16_t *)x,
                       (const uint16_t *)cos_cache, (const uint16_t *)sin_cache, (uint16_t *)out, rows_pad, cols, per_batch,
                       total8, token_index, rows, src_cols);
  else
    hipLaunchKernelGGL(ttm_rotary_k<float>, grid, dim3(256), 0, (hipStream_t)stream, (const float *)x, (const float *)cos_cache,
                       (const float *)sin_cache, (float *)out, rows_pad, cols, per_batch, total8, token_index, rows, src_cols);
  TTM_LAUNCH_CHECK();
  return TTM_OK;
}

TTM_EXPORT int ttm_rotary_embedding(const void *x, const void *cos_cache, const void *sin_cache, void *out, int dtype,
                                    int64_t batch, int64_t rows, int64_t cols, int64_t cache_rows, int64_t token_index,
                                    void *stream) {
  TTM_EXTENTS(rotary_embedding, x, cos_cache, sin_cache, out, dtype, batch, rows, cols, cache_rows);
  return rotary_entry(x, cos_cache, sin_cache, out, dtype, batch, rows, cols, cache_rows, token_index, false, stream);
}

TTM_EXPORT int ttm_rotary_embedding_split_heads(const void *x, const void *cos_cache, const void *sin_cache, void *out, int dtype,
                                                int64_t batch, int64_t heads, int64_t head_dim, int64_t cache_rows,
                                                int64_t token_index, void *stream) {
  TTM_EXTENTS(rotary_embedding_split_heads, x, cos_cache, sin_cache, out, dtype, batch, heads, head_dim, cache_rows);
  return rotary_entry(x, cos_cache, sin_cache, out, dtype, batch, heads, head_dim, cache_rows, token_index, true, stream);
}

TTM_EXPORT int ttm_update_cache(void *cache, const void *input, const int32_t *update_index, int dtype, int64_t users,
                                int64_t heads, int64_t max_seq, int64_t head_dim, int64_t input_users, int64_t batch_offset,
                                void *stream) {
  TTM_EXTENTS(update_cache, cache, input, update_index, dtype, users, heads, max_seq, head_dim, input_users);
  TTM_REQUIRE(cache && input && update_index, "ttm_update_cache: null pointer");
  TTM_REQUIRE(dtype == TTM_BF16 || dtype == TTM_F32, "ttm_update_cache: dtype must be BFloat16 or Float32");
  TTM_REQUIRE(head_dim > 0 && head_dim % 32 == 0, "ttm_update_cache: head dim must be a positive multiple of 32");
  TTM_REQUIRE(batch_offset >= 0 && input_users >= 0 && batch_offset + input_users <= users,
              "ttm_update_cache: users [%lld, %lld) outside the cache's %lld", (long long)batch_offset,
              (long long)(batch_offset + input_users), (long long)users);
  const int64_t total8 = heads * input_users * (head_dim / 8);
  if (total8 == 0) return TTM_OK;
  const dim3 grid((unsigned)ttm_cdiv(total8, 256));
  const int64_t seq_pad = ttm_round_up32(max_seq), in_pad = ttm_round_up32(input_users);
  if (dtype == TTM_BF16)
    hipLaunchKernelGGL(ttm_update_cache_k<uint16_t>, grid, dim3(256), 0, (hipStream_t)stream, (uint16_t *)cache,
                       (const uint16_t *)input, update_index, heads, seq_pad, max_seq, head_dim, input_users, in_pad, batch_offset,
                       total8);
  else
    hipLaunchKernelGGL(ttm_update_cache_k<float>, grid, dim3(256), 0, (hipStream_t)stream, (float *)cache, (const float *)input,
                       update_index, heads, seq_pad, max_seq, head_dim, input_users, in_pad, batch_offset, total8);
  TTM_LAUNCH_CHECK();
  return TTM_OK;
}

TTM_EXPORT int ttm_fill_cache(void *cache, const void *input, int dtype, int64_t users, int64_t heads, int64_t max_seq,
                              int64_t head_dim, int64_t seq, int64_t batch_offset, void *stream) {
  TTM_EXTENTS(fill_cache, cache, input, dtype, users, heads, max_seq, head_dim, seq);
  TTM_REQUIRE(cache && input, "ttm_fill_cache: null pointer");
  const int eb = ttm_dtype_bytes(dtype);
  TTM_REQUIRE(eb == 2 || eb == 4, "ttm_fill_cache: element size must be 2 or 4 bytes");
  TTM_REQUIRE(head_dim > 0 && head_dim % 32 == 0, "ttm_fill_cache: head dim must be a positive multiple of 32");
  TTM_REQUIRE(batch_offset >= 0 && batch_offset < users, "ttm_fill_cache: batch offset %lld outside the cache's %lld users",
              (long long)batch_offset, (long long)users);
  TTM_REQUIRE(seq >= 0 && seq <= max_seq, "ttm_fill_cache: %lld positions do not fit a cache of %lld", (long long)seq, (long long)max_seq);
  const int64_t in16 = ttm_round_up32(seq) * head_dim * eb / 16, cache16 = ttm_round_up32(max_seq) * head_dim * eb / 16;
  const int64_t total16 = heads * in16;
  if (total16 == 0) return TTM_OK;
  hipLaunchKernelGGL(ttm_fill_cache_k, dim3((unsigned)ttm_cdiv(total16, 256)), dim3(256), 0, (hipStream_t)stream, (u32x4 *)cache,
                     (const u32x4 *)input, cache16, in16, batch_offset * heads * cache16, total16);
  TTM_LAUNCH_CHECK();
  return TTM_OK;
}

TTM_EXPORT int ttm_paged_update_cache(void *cache, const void *input, const int32_t *update_index, const int32_t *page_table,
                                      int dtype, int64_t blocks, int64_t heads, int64_t block_size, int64_t head_dim, int64_t users,
                                      int64_t pages_per_user, int share_cache, void *stream) {
  TTM_EXTENTS(paged_update_cache, cache, input, update_index, page_table, dtype, blocks, heads, block_size, head_dim, users, pages_per_user);
  TTM_REQUIRE(cache && input && update_index, "ttm_paged_update_cache: null pointer");
  TTM_REQUIRE(dtype == TTM_BF16 || dtype == TTM_F32, "ttm_paged_update_cache: dtype must be BFloat16 or Float32");
  TTM_REQUIRE(head_dim > 0 && head_dim % 32 == 0, "ttm_paged_update_cache: head dim must be a positive multiple of 32");
  TTM_REQUIRE(blocks > 0 && heads > 0 && block_size > 0 && users >= 0, "ttm_paged_update_cache: bad extents");
  TTM_REQUIRE(!page_table || pages_per_user > 0, "ttm_paged_update_cache: a page table needs pages_per_user > 0");
  TTM_REQUIRE(page_table || share_cache || users <= blocks, "ttm_paged_update_cache: %lld users do not fit a cache of %lld entries",
              (long long)users, (long long)blocks);
  const int64_t total8 = users * heads * (head_dim / 8);
  if (total8 == 0) return TTM_OK;
  const dim3 grid((unsigned)ttm_cdiv(total8, 256));
  if (dtype == TTM_BF16)
    hipLaunchKernelGGL(ttm_paged_update_cache_k<uint16_t>, grid, dim3(256), 0, (hipStream_t)stream, (uint16_t *)cache,
                       (const uint16_t *)input, update_index, page_table, blocks, heads, block_size, head_dim, users, pages_per_user,
                       share_cache, total8);
  else
    hipLaunchKernelGGL(ttm_paged_update_cache_k<float>, grid, dim3(256), 0, (hipStream_t)stream, (float *)cache, (const float *)input,
                       update_index, page_table, blocks, heads, block_size, head_dim, users, pages_per_user, share_cache, total8);
  TTM_LAUNCH_CHECK();
  return TTM_OK;
}

TTM_EXPORT int ttm_paged_fill_cache(void *cache, const void *input, const int32_t *page_table, const int32_t *batch_idx, int dtype,
                                    int64_t blocks, int64_t heads, int64_t block_size, int64_t head_dim, int64_t in_batch, int64_t seq,
                                    int64_t table_rows, int64_t pages_per_user, void *stream) {
  TTM_EXTENTS(paged_fill_cache, cache, input, page_table, batch_idx, dtype, blocks, heads, block_size, head_dim, in_batch, seq, table_rows, pages_per_user);
  TTM_REQUIRE(cache && input && page_table, "ttm_paged_fill_cache: null pointer");
  TTM_REQUIRE(dtype == TTM_BF16 || dtype == TTM_F32, "ttm_paged_fill_cache: dtype must be BFloat16 or Float32");
  TTM_REQUIRE(head_dim > 0 && head_dim % 32 == 0, "ttm_paged_fill_cache: head dim must be a positive multiple of 32");
  TTM_REQUIRE(blocks > 0 && heads > 0 && block_size > 0 && in_batch >= 0 && seq >= 0 && table_rows > 0 && pages_per_user > 0,
              "ttm_paged_fill_cache: bad extents");
  const int64_t total8 = in_batch * heads * seq * (head_dim / 8);
  if (total8 == 0) return TTM_OK;
  const dim3 grid((unsigned)ttm_cdiv(total8, 256));
  if (dtype == TTM_BF16)
    hipLaunchKernelGGL(ttm_paged_fill_cache_k<uint16_t>, grid, dim3(256), 0, (hipStream_t)stream, (uint16_t *)cache,
                       (const uint16_t *)input, page_table, batch_idx, blocks, heads, block_size, head_dim, seq, table_rows,
                       pages_per_user, total8);
  else
    hipLaunchKernelGGL(ttm_paged_fill_cache_k<float>, grid, dim3(256), 0, (hipStream_t)stream, (float *)cache, (const float *)input,
                       page_table, batch_idx, blocks, heads, block_size, head_dim, seq, table_rows, pages_per_user, total8);
  TTM_LAUNCH_CHECK();
  return TTM_OK;
}

// ---- scratch of ttm_sdpa_decode_static: the per-slice (max, sum, output) slots live in a device array of the library's
// own instead of the stream's workspace, so that entry point never allocates.  Every GPU holds its own copy of the array at
// its own address until the process ends; in host code the array's name is only a handle for hipGetSymbolAddress, the
// kernels get the address that call returned for the current device.
constexpr size_t kDecodeScratchBytes = (size_t)8 << 20;
static __device__ __align__(256) float scratch[kDecodeScratchBytes / sizeof(float)];

constexpr int kMaxDevices = 64;
static std::mutex g_scratch_mu;
static float *g_scratch_ptr[kMaxDevices];   // per device, set on the first call with that device current

static int decode_scratch_ptr(void **ptr) {
  int dev = 0;
  TTM_HIP(hipGetDevice(&dev));
  TTM_REQUIRE(dev >= 0 && dev < kMaxDevices, "ttm_sdpa_decode_static: device ordinal %d beyond %d", dev, kMaxDevices);
  std::lock_guard<std::mutex> g(g_scratch_mu);
  if (!g_scratch_ptr[dev]) {
    float *d = nullptr;
    TTM_HIP(hipGetSymbolAddress((void **)&d, HIP_SYMBOL(scratch)));
    TTM_REQUIRE(d != nullptr, "ttm_sdpa_decode_static: hipGetSymbolAddress returned a null address");
    g_scratch_ptr[dev] = d;
  }
  *ptr = g_scratch_ptr[dev];
  return TTM_OK;
}

template <bool STREAM, int GM, int DM, bool EXACT, int NW, bool DIRECT>
static void launch_decode(const DecodeArgs &p, dim3 grid, hipStream_t s) {
  const size_t lds = (size_t)NW * p.G * p.D * sizeof(float);   // at most 32 KiB
  if (p.mask || p.sink) hipLaunchKernelGGL((ttm_sdpa_decode_k<STREAM, GM, DM, EXACT, NW, DIRECT, DecodeArgs>), grid, dim3(NW * 64), lds, s, p);
  else hipLaunchKernelGGL((ttm_sdpa_decode_k<STREAM, GM, DM, EXACT, NW, DIRECT, DecodeLean>), grid, dim3(NW * 64), lds, s, DecodeLean(p));
}
// The head dims 32, 64, 128 and 256 have kernels of their own; others, and heads in several launches, the next larger one's loops
// with a bound.  Up to four heads (and 128 columns) the direct form holds its state in 128 registers and takes 16 wavefronts.
template <bool DIRECT>
static void launch_decode(const DecodeArgs &p, dim3 grid, hipStream_t s) {
  constexpr int NW = DIRECT ? 8 : 4, NWS = DIRECT ? 16 : 4;
  const bool few = p.G <= 4 && p.Gt <= kMaxG, once = p.Gt <= kMaxG;
  switch (p.D) {
  case 32: return few ? launch_decode<true, 4, 1, true, NWS, DIRECT>(p, grid, s) : once ? launch_decode<true, 8, 1, true, NW, DIRECT>(p, grid, s) : launch_decode<false, 8, 1, true, NW, DIRECT>(p, grid, s);
  case 64: return few ? launch_decode<true, 4, 2, true, NWS, DIRECT>(p, grid, s) : once ? launch_decode<true, 8, 2, true, NW, DIRECT>(p, grid, s) : launch_decode<false, 8, 2, true, NW, DIRECT>(p, grid, s);
  case 128: return few ? launch_decode<true, 4, 4, true, NWS, DIRECT>(p, grid, s) : once ? launch_decode<true, 8, 4, true, NW, DIRECT>(p, grid, s) : launch_decode<false, 8, 4, true, NW, DIRECT>(p, grid, s);
  case 256:
    if constexpr (DIRECT) return once ? launch_decode<true, 4, 8, true, NW, DIRECT>(p, grid, s) : launch_decode<false, 4, 8, true, NW, DIRECT>(p, grid, s);   // at most 1024 outputs
    else return few ? launch_decode<true, 4, 8, true, NW, DIRECT>(p, grid, s) : once ? launch_decode<true, 8, 8, true, NW, DIRECT>(p, grid, s) : launch_decode<false, 8, 8, true, NW, DIRECT>(p, grid, s);
  default: return p.D < 128 ? launch_decode<false, 8, 4, false, NW, DIRECT>(p, grid, s) : launch_decode<false, 8, 8, false, NW, DIRECT>(p, grid, s);
  }
}

static int sdpa_decode_entry(const void *q, const void *k, const void *v, const int32_t *cur_pos, const void *mask, int mask_heads,
                             const int32_t *page_table, int64_t pages_per_user, int64_t page_block, int64_t page_blocks, void *out, int dtype, int64_t batch,
                             int64_t heads, int64_t kv_heads, int64_t seq, int64_t head_dim, int is_causal, float scale, int concat_heads,
                             int64_t window, const void *sink, int64_t mask_batch, bool static_scratch, void *stream) {
  TTM_REQUIRE(q && k && v && out, "ttm_sdpa_decode: null pointer");
  TTM_REQUIRE(dtype == TTM_BF16, "ttm_sdpa_decode: tensors must be BFloat16");
  TTM_REQUIRE(batch > 0 && heads > 0 && kv_heads > 0 && heads % kv_heads == 0, "ttm_sdpa_decode: heads must be a multiple of kv heads");
  // a launch serves up to kMaxG query heads per kv head; more (multi-query attention) take several launches over the same cache
  const int64_t Gt = heads / kv_heads, G = Gt < kMaxG ? Gt : kMaxG;
  TTM_REQUIRE(head_dim % 32 == 0 && head_dim >= 32 && head_dim <= 256, "ttm_sdpa_decode: head dim must be a multiple of 32 up to 256");
  TTM_REQUIRE(seq > 0 && seq % 32 == 0, "ttm_sdpa_decode: cache length must be a positive multiple of 32");
  TTM_REQUIRE(!mask || mask_heads == 1 || mask_heads == heads, "ttm_sdpa_decode: mask must have 1 or %lld head rows", (long long)heads);
  if (page_table) {
    TTM_REQUIRE(page_block > 0 && page_block % 32 == 0 && pages_per_user * page_block == seq,
                "ttm_sdpa_decode: page table of %lld blocks x %lld positions does not cover %lld positions",
                (long long)pages_per_user, (long long)page_block, (long long)seq);
    TTM_REQUIRE(page_blocks > 0 && page_blocks <= INT32_MAX, "ttm_sdpa_decode: a page table needs the number of blocks in the cache (got %lld)",
                (long long)page_blocks);
  }
  hipStream_t s = (hipStream_t)stream;
  // Direct form where the users alone fill the device or their caches are short; shares for few users with long caches.  Measured
  // (D = 128, 8 kv heads of 4 query heads, contexts of a quarter of the cache to all of it; direct / shares, us): 1 user x 512 positions
  // 7.4 / 9.9, 1 x 1024 10.7 / 10.2, 1 x 2048 12.1 / 10.4, 1 x 4096 30.2 / 11.5, 8 x 1024 14.8 / 15.2, 8 x 2048 24.3 / 18.8, 16 x 2048
  // 26.4 / 26.0, 16 x 4096 43.8 / 35.9, 32 x 1024 19.7 / 26.2, 32 x 2048 32.9 / 37.2; D = 64: 5 x 2048 12.2 / 13.6, 5 x 4096 21.6 / 15.6,
  // 16 x 2048 15.4 / 18.1, 16 x 4096 26.5 / 25.5.  A tile of 32 columns takes about as long as one of 64, so narrower heads count as 64:
  // D = 32, 16 kv heads of 5 query heads: 1 x 4096 15.3 / 11.0, 2 x 2048 12.0 / 13.7, 2 x 4096 18.0 / 14.1, 8 x 4096 25.4 / 24.1 (under a
  // window they see few tiles: 4 x 2080, 8 kv heads of 12, window 100 9.6 / 20.9).
  const int form = ttm_option("sdpa_decode_form");   // 0 by this rule, 1 direct, 2 shares
  // (the results of the wavefronts fit in 32 KiB of LDS)
  bool direct = G * head_dim <= 1024 && (form ? form == 1 : seq * (window < 0 ? std::max<int64_t>(64, head_dim) : head_dim) <= 2048 * std::max<int64_t>(64, batch * kv_heads));
  const int64_t all = batch * (seq / 32);          // tiles of a kv head when every cache is full
  int64_t shares = ttm_cdiv(kDecodeBlocks, kv_heads);
  if (shares > all / 4) shares = all / 4 > 0 ? all / 4 : 1;   // a tile for every wavefront
  if (shares > INT32_MAX / (all + 1)) shares = INT32_MAX / (all + 1);
  TTM_REQUIRE(all < INT32_MAX, "ttm_sdpa_decode: caches of %lld x %lld positions are too long", (long long)batch, (long long)seq);
  DecodeArgs p;
  p.q = (const uint16_t *)q; p.k = (const uint16_t *)k; p.v = (const uint16_t *)v; p.mask = (const uint16_t *)mask;
  p.cur_pos = cur_pos; p.page_table = page_table; p.out = (uint16_t *)out;
  p.B = (int)batch; p.H = (int)heads; p.Hkv = (int)kv_heads; p.G = (int)G; p.S = (int)seq; p.D = (int)head_dim;
  p.shares = (int)shares; p.block = (int)page_block; p.pages_per_user = (int)pages_per_user;
  p.blocks = (int)page_blocks;
  p.mask_heads = mask_heads; p.is_causal = is_causal; p.concat_heads = concat_heads;
  p.scale = scale > 0.0f ? scale : 1.0f / sqrtf((float)head_dim);
  p.Gt = (int)Gt;
  p.window = window < 0 ? -1 : (int)(window < seq ? window : seq);
  p.sink = (const uint16_t *)sink;
  TTM_REQUIRE(!mask || mask_batch == 1 || mask_batch == batch, "ttm_sdpa_decode: mask batch must be 1 or %lld", (long long)batch);
  p.mask_b = mask_batch == 1 ? 0 : 1;
  const size_t slot_bytes = (size_t)(kv_heads * G * (head_dim + 2)) * sizeof(float);   // of one share or user, all kv heads
  size_t part_bytes = direct ? 0 : slot_bytes * (size_t)(shares + batch);
  int64_t per_launch = kMaxG;
  void *ws = nullptr;
  if (static_scratch) {
    TTM_REQUIRE(slot_bytes * (size_t)batch <= kDecodeScratchBytes,
                "ttm_sdpa_decode_static: one partial result per user and head of this call takes %zu bytes, the static scratch holds %zu "
                "(batch * kv_heads * heads-per-kv-head * (head_dim + 2) floats): use ttm_sdpa_decode_windowed",
                slot_bytes * (size_t)batch, (size_t)kDecodeScratchBytes);
    if (part_bytes > kDecodeScratchBytes) {
      // More than some 500 users x kv heads (a share and a user take a slot each): the direct form needs no slots, and that many
      // workgroups fill the device; above 1024 outputs per kv head in several launches of fewer heads
      direct = true;
      part_bytes = 0;
      per_launch = std::min<int64_t>(kMaxG, 1024 / head_dim);
    }
    if (int rc = decode_scratch_ptr(&ws)) return rc;
  } else if (part_bytes) {
    if (int rc = ttm_stream_workspace(s, part_bytes, &ws)) return rc;
  }
  p.part = (float *)ws;
  for (int64_t g0 = 0; g0 < Gt; g0 += per_launch) {   // the launches of one call follow each other on the stream and share the workspace
    p.g0 = (int)g0;
    p.G = (int)(Gt - g0 < per_launch ? Gt - g0 : per_launch);
    if (direct) {
      launch_decode<true>(p, dim3((unsigned)kv_heads, (unsigned)batch), s);
      TTM_LAUNCH_CHECK();
      continue;
    }
    launch_decode<false>(p, dim3((unsigned)shares, (unsigned)kv_heads), s);
    TTM_LAUNCH_CHECK();
    const dim3 heads_of_users((unsigned)(batch * kv_heads), (unsigned)p.G);
    if (p.mask || p.sink) hipLaunchKernelGGL(ttm_sdpa_decode_combine_k<DecodeArgs>, heads_of_users, dim3(256), 0, s, p);
    else hipLaunchKernelGGL(ttm_sdpa_decode_combine_k<DecodeLean>, heads_of_users, dim3(256), 0, s, DecodeLean(p));
    TTM_LAUNCH_CHECK();
  }
  return TTM_OK;
}

TTM_EXPORT int ttm_sdpa_decode(const void *q, const void *k, const void *v, const int32_t *cur_pos, const void *mask,
                               int mask_heads, const int32_t *page_table, int64_t pages_per_user, int64_t page_block, int64_t page_blocks,
                               void *out, int dtype, int64_t batch, int64_t heads, int64_t kv_heads, int64_t seq, int64_t head_dim,
                               int is_causal, float scale, void *stream) {
  TTM_EXTENTS(sdpa_decode, q, k, v, cur_pos, mask, mask_heads, batch, page_table, pages_per_user, page_block, page_blocks, out, dtype, batch, heads, kv_heads, seq, head_dim, 0, nullptr);
  return sdpa_decode_entry(q, k, v, cur_pos, mask, mask_heads, page_table, pages_per_user, page_block, page_blocks, out, dtype, batch, heads, kv_heads,
                           seq, head_dim, is_causal, scale, 0, -1, nullptr, batch, false, stream);
}

TTM_EXPORT int ttm_sdpa_decode_concat_heads(const void *q, const void *k, const void *v, const int32_t *cur_pos, const void *mask,
                                            int mask_heads, const int32_t *page_table, int64_t pages_per_user, int64_t page_block,
                                            int64_t page_blocks, void *out, int dtype, int64_t batch, int64_t heads, int64_t kv_heads,
                                            int64_t seq, int64_t head_dim, int is_causal, float scale, void *stream) {
  TTM_EXTENTS(sdpa_decode, q, k, v, cur_pos, mask, mask_heads, batch, page_table, pages_per_user, page_block, page_blocks, out, dtype, batch, heads, kv_heads, seq, head_dim, 1, nullptr);
  return sdpa_decode_entry(q, k, v, cur_pos, mask, mask_heads, page_table, pages_per_user, page_block, page_blocks, out, dtype, batch, heads, kv_heads,
                           seq, head_dim, is_causal, scale, 1, -1, nullptr, batch, false, stream);
}

TTM_EXPORT int ttm_sdpa_decode_windowed(const void *q, const void *k, const void *v, const int32_t *cur_pos, const void *mask,
                                        int mask_heads, int64_t mask_batch, const int32_t *page_table, int64_t pages_per_user,
                                        int64_t page_block, int64_t page_blocks, void *out, int dtype, int64_t batch, int64_t heads, int64_t kv_heads,
                                        int64_t seq, int64_t head_dim, int is_causal, float scale, int concat_heads, int64_t sliding_window,
                                        const void *attention_sink, void *stream) {
  TTM_EXTENTS(sdpa_decode, q, k, v, cur_pos, mask, mask_heads, mask_batch, page_table, pages_per_user, page_block, page_blocks, out, dtype, batch, heads, kv_heads, seq, head_dim, concat_heads, attention_sink);
  return sdpa_decode_entry(q, k, v, cur_pos, mask, mask_heads, page_table, pages_per_user, page_block, page_blocks, out, dtype, batch, heads, kv_heads,
                           seq, head_dim, is_causal, scale, concat_heads != 0, sliding_window, attention_sink, mask_batch, false, stream);
}

// ttm_sdpa_decode_windowed for callers that cannot allocate: the slots come from the library's static device array.
TTM_EXPORT int ttm_sdpa_decode_static(const void *q, const void *k, const void *v, const int32_t *cur_pos, const void *mask,
                                      int mask_heads, int64_t mask_batch, const int32_t *page_table, int64_t pages_per_user,
                                      int64_t page_block, int64_t page_blocks, void *out, int dtype, int64_t batch, int64_t heads, int64_t kv_heads,
                                      int64_t seq, int64_t head_dim, int is_causal, float scale, int concat_heads, int64_t sliding_window,
                                      const void *attention_sink, void *stream) {
  TTM_EXTENTS(sdpa_decode, q, k, v, cur_pos, mask, mask_heads, mask_batch, page_table, pages_per_user, page_block, page_blocks, out, dtype, batch, heads, kv_heads, seq, head_dim, concat_heads, attention_sink);
  return sdpa_decode_entry(q, k, v, cur_pos, mask, mask_heads, page_table, pages_per_user, page_block, page_blocks, out, dtype, batch, heads, kv_heads,
                           seq, head_dim, is_causal, scale, concat_heads != 0, sliding_window, attention_sink, mask_batch, true, stream);
}

TTM_EXPORT int ttm_paged_gather(const void *cache, const int32_t *page_table, void *out, int dtype, int64_t blocks, int64_t heads,
                                int64_t block_size, int64_t head_dim, int64_t users, int64_t pages_per_user, void *stream) {
  TTM_EXTENTS(paged_gather, cache, page_table, out, dtype, blocks, heads, block_size, head_dim, users, pages_per_user);
  TTM_REQUIRE(cache && page_table && out, "ttm_paged_gather: null pointer");
  TTM_REQUIRE(dtype == TTM_BF16 || dtype == TTM_F32, "ttm_paged_gather: dtype must be BFloat16 or Float32");
  TTM_REQUIRE(head_dim > 0 && head_dim % 32 == 0, "ttm_paged_gather: head dim must be a positive multiple of 32");
  TTM_REQUIRE(block_size > 0 && block_size % 32 == 0, "ttm_paged_gather: block size must be a positive multiple of 32");
  TTM_REQUIRE(blocks > 0 && heads > 0 && users >= 0 && pages_per_user > 0, "ttm_paged_gather: bad extents");
  const int64_t total8 = users * heads * pages_per_user * block_size * (head_dim / 8);
  if (total8 == 0) return TTM_OK;
  const dim3 grid((unsigned)ttm_cdiv(total8, 256));
  if (dtype == TTM_BF16)
    hipLaunchKernelGGL(ttm_paged_gather_k<uint16_t>, grid, dim3(256), 0, (hipStream_t)stream, (const uint16_t *)cache, page_table,
                       (uint16_t *)out, blocks, heads, block_size, head_dim, pages_per_user, total8);
  else
    hipLaunchKernelGGL(ttm_paged_gather_k<float>, grid, dim3(256), 0, (hipStream_t)stream, (const float *)cache, page_table, (float *)out,
                       blocks, heads, block_size, head_dim, pages_per_user, total8);
  TTM_LAUNCH_CHECK();
  return TTM_OK;
}

TTM_EXPORT int ttm_chunk_causal_mask(void *mask, const int32_t *chunk_start, int64_t rows, int64_t cols, void *stream) {
  TTM_EXTENTS(chunk_causal_mask, mask, chunk_start, rows, cols);
  TTM_REQUIRE(mask && chunk_start, "ttm_chunk_causal_mask: null pointer");
  TTM_REQUIRE(rows > 0 && cols > 0, "ttm_chunk_causal_mask: bad extents");
  const int64_t rp = ttm_round_up32(rows), cp = ttm_round_up32(cols), total8 = rp * cp / 8;
  hipLaunchKernelGGL(ttm_chunk_mask_k, dim3((unsigned)ttm_cdiv(total8, 256)), dim3(256), 0, (hipStream_t)stream, (uint16_t *)mask,
                     chunk_start, rp, cp, total8);
  TTM_LAUNCH_CHECK();
  return TTM_OK;
}

TTM_EXPORT int ttm_rotary_embedding_llama(const void *x, const void *cos_cache, const void *sin_cache, const void *trans_mat, void *out,
                                          int dtype, int64_t batch, int64_t rows, int64_t cols, int64_t cs_batch, int64_t cs_rows,
                                          void *stream) {
  TTM_EXTENTS(rotary_embedding_llama, x, cos_cache, sin_cache, trans_mat, out, dtype, batch, rows, cols, cs_batch, cs_rows);
  TTM_REQUIRE(x && cos_cache && sin_cache && trans_mat && out, "ttm_rotary_embedding_llama: null pointer");
  TTM_REQUIRE(dtype == TTM_BF16, "ttm_rotary_embedding_llama: tensors must be BFloat16");
  TTM_REQUIRE(batch >= 0 && rows > 0 && cols > 0 && cols % 32 == 0 && cols <= 256,
              "ttm_rotary_embedding_llama: head dim must be a multiple of 32 up to 256");
  TTM_REQUIRE(cs_batch >= 1 && (cs_rows == 1 || cs_rows == rows), "ttm_rotary_embedding_llama: cos / sin must have 1 or %lld rows",
              (long long)rows);
  const int64_t rp = ttm_round_up32(rows), total = batch * rp * cols;
  if (total == 0) return TTM_OK;
  hipLaunchKernelGGL(ttm_rotary_llama_k, dim3((unsigned)ttm_cdiv(total, 256)), dim3(256), 0, (hipStream_t)stream, (const uint16_t *)x,
                     (const uint16_t *)cos_cache, (const uint16_t *)sin_cache, (const uint16_t *)trans_mat, (uint16_t *)out, rows, rp, cols,
                     cs_batch, cs_rows, ttm_round_up32(cs_rows), total);
  TTM_LAUNCH_CHECK();
  return TTM_OK;
}
