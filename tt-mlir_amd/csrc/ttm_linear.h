// What the kernels of ttm_linear.hip and ttm_linear_mid.hip share: launch arguments, epilogue pieces, operand helpers.
#pragma once
#include <type_traits>

#include "ttm_common.h"
#include "ttm_math.h"

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

enum { WF_BFP8 = 0, WF_BFP4 = 1, WF_BF16_KN = 2, WF_BF16_NK = 3 };

struct LinearArgs {
  const uint8_t *A;     // bf16, tile order, [Mt*32, Kt*32]
  const uint8_t *W;     // weights, format WF_*
  const uint16_t *bias; // bf16 or null
  uint8_t *C;           // bf16, tile order, [Mt*32, Nt*32]
  int Mt, Nt, Kt;       // extents in tiles
  int act, bias_tiled;
  int64_t a_batch, w_batch, c_batch;  // byte strides between batch entries (w_batch 0 = shared weights)
  int m_blocks, n_blocks;
  int ntw;                            // block-float main kernel: column tiles per wavefront (block width / 2)
  int nt_split, n_blocks1, ntw2;      // two-part grid: blocks [0, n_blocks1) cover column tiles [0, nt_split) at width ntw,
                                      // the rest cover [nt_split, Nt) at width ntw2; nt_split = 0: one part
  int k_slice;                        // k-tiles per grid.y slice (split-K); Kt when the reduction is not split
  int slices;                         // of K (grid.y) in a launch that leaves partial sums
  float *partial;                     // split-K: fp32 partial sums [slices][Mt * Nt * 1024] in output tile order
  int img_zero_step;                  // two-pass launch: W points at the dequantised images, this step index holds zeros
  // group launch (group_n >= 2): several weight matrices [K, N_i] applied to the same activations, each with its own
  // output; W / C / Nt above describe the virtual concatenation (Nt = sum of the members' column tiles) and are not
  // dereferenced.  Each member may have its own activation; no bias, tail or batch in a group.
  int group_n;
  const uint8_t *gW[4];
  uint8_t *gC[4];
  int gNt[4];
  int gAct[4];                        // per-member activation
  int glu;                            // gated pair (decode kernel only): C = gC[0] = act0(A gW[0]) x act1(A gW[1]), both [K, gNt[0] * 32]
  int tail;                           // 0 none, 1 add, 2 multiply: element-wise tail with a tensor laid out like the output
  int64_t tail_delta;                 // byte distance from an output element to its tail operand
  int plan_batch;                     // host side only: batch entries the launch plan counts (a pair of matrices plans as one alone)
  const struct QkvFinishArgs *qkv;    // host side only: the decode launch leaves partial sums and ttm_qkv_finish_k ends it
  const struct NormFinishArgs *norm;  // host side only: ... and the RMSNorm kernel ends it (residual add, then the norm)
  __device__ __forceinline__ const LinearArgs &full() const { return *this; }
};

// The same for a launch that is neither a group nor a gated pair, in the 112 bytes that launch quickly (ttm_common.h)
struct LinearPlain {
  const uint8_t *A, *W;
  const uint16_t *bias;
  uint8_t *C;
  int Mt, Nt, Kt;
  uint8_t act, bias_tiled, tail;
  int n_blocks, k_slice, slices;
  int64_t a_batch, w_batch, c_batch;
  float *partial;
  int64_t tail_delta;
  explicit LinearPlain(const LinearArgs &a)
      : A(a.A), W(a.W), bias(a.bias), C(a.C), Mt(a.Mt), Nt(a.Nt), Kt(a.Kt), act((uint8_t)a.act), bias_tiled((uint8_t)a.bias_tiled), tail((uint8_t)a.tail),
        n_blocks(a.n_blocks), k_slice(a.k_slice), slices(a.slices), a_batch(a.a_batch), w_batch(a.w_batch), c_batch(a.c_batch), partial(a.partial),
        tail_delta(a.tail_delta) {}
  __device__ __forceinline__ LinearArgs full() const {
    LinearArgs p = {};
    p.A = A; p.W = W; p.bias = bias; p.C = C; p.Mt = Mt; p.Nt = Nt; p.Kt = Kt; p.act = act; p.bias_tiled = bias_tiled; p.tail = tail;
    p.n_blocks = n_blocks; p.k_slice = k_slice; p.slices = slices; p.a_batch = a_batch; p.w_batch = w_batch; p.c_batch = c_batch;
    p.partial = partial; p.tail_delta = tail_delta;
    return p;
  }
};
static_assert(sizeof(LinearPlain) <= 112, "the size up to which a launch is quick");

// x1 = residual + projection (stored to sum_out), then out = rms_norm(x1): the operands of the second launch
struct NormFinishArgs {
  const void *residual, *weight, *bias;
  int weight_layout, bias_layout;
  void *sum_out, *out;
  int64_t rows, cols;
  float eps;
};

// What follows the Q, K and V projections of a decode step (one token per user): head split, rotary embedding of q and k
// at the cos / sin row `cos_row`, q to its own tensor, k and v into the cache row of position *index.
struct QkvFinishArgs {
  const float *partial;               // [slices][per] fp32 in tile order over the concatenation q | k | v (one row tile)
  int slices;
  int64_t per;
  int users, heads, heads_pad, kv_heads, dim;
  const uint16_t *cosc, *sinc;        // [.., dim] bf16 tiles
  int64_t cos_row;
  uint16_t *q_out;                    // [1, users, heads, dim] bf16 tiles
  uint16_t *k_cache, *v_cache;        // [cache users, kv_heads, max_seq, dim] bf16 tiles
  int64_t max_seq, seq_pad, batch_offset;
  const int32_t *index;               // device memory: the position all users write
};

// The member of a group launch that owns column unit `u`, where a unit is `unit_tiles` column tiles and every member's
// units are numbered one after another (a member's last unit may be partial).  Constant indices only: the arrays stay in
// scalar registers.
struct GroupMember {
  const uint8_t *W;
  uint8_t *C;
  int Nt, local, tile_base, act;   // column tiles, unit index inside the member, first column tile in the concatenation
};
__device__ __forceinline__ GroupMember group_member(const LinearArgs &p, int u, int unit_tiles) {
  GroupMember m = {p.gW[0], p.gC[0], p.gNt[0], u, 0, p.gAct[0]};
  int start = 0, tiles = 0;
  bool found = false;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    if (j < p.group_n) {
      const int n = (p.gNt[j] + unit_tiles - 1) / unit_tiles;
      if (!found && (u < start + n || j == p.group_n - 1)) {
        found = true;
        m.W = p.gW[j]; m.C = p.gC[j]; m.Nt = p.gNt[j]; m.local = u - start; m.tile_base = tiles; m.act = p.gAct[j];
      }
      start += n; tiles += p.gNt[j];
    }
  }
  return m;
}

template <int ACT>
__device__ __forceinline__ float apply_act(float x) {
  if (ACT == TTM_ACT_GELU) return ttm_gelu_fast(x);
  if (ACT == TTM_ACT_SILU) return ttm_silu(x);
  if (ACT == TTM_ACT_SIGMOID) return ttm_sigmoid(x);
  if (ACT == TTM_ACT_RELU) return ttm_max(x, 0.0f);   // keeps NaN, as arith.maximumf does
  return x;
}

typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
typedef float f32x2_t __attribute__((ext_vector_type(2)));
// two floats -> packed bf16 pair, round to nearest even (v_cvt_pk_bf16_f32)
__device__ __forceinline__ uint32_t pack_bf16(float a, float b) {
  f32x2_t v = {a, b};
  bf16x2_t h = __builtin_convertvector(v, bf16x2_t);
  return *(uint32_t *)&h;
}

// Four consecutive bias values of column tile nt, from column n_in of the tile on
__device__ __forceinline__ u32x2 bias_quad(const LinearArgs &p, int nt, int n_in) {
  return *(const u32x2 *)(p.bias_tiled ? p.bias + (int64_t)nt * 1024 + (n_in >> 4) * 256 + (n_in & 15) : p.bias + nt * 32 + n_in);
}
// Bias and tail operands are loaded for many outputs in front of the first of them: requested one by one behind the store before (which
// they might alias as far as the compiler knows), every quad waited for a memory round trip of its own.
// Four consecutive outputs -> bf16, optionally followed by the element-wise tail with the quad `r`.  The result is rounded to bf16
// before the tail and again after it, exactly as a separate binary op on the stored result would do.
__device__ __forceinline__ u32x2 finish_quad(int tail, u32x2 r, const float (&v)[4]) {
  u32x2 o = {pack_bf16(v[0], v[1]), pack_bf16(v[2], v[3])};
  if (tail != 0) {   // uniform
    const float y[4] = {__uint_as_float(o.x << 16), __uint_as_float(o.x & 0xFFFF0000u), __uint_as_float(o.y << 16),
                        __uint_as_float(o.y & 0xFFFF0000u)};
    const float t[4] = {__uint_as_float(r.x << 16), __uint_as_float(r.x & 0xFFFF0000u), __uint_as_float(r.y << 16),
                        __uint_as_float(r.y & 0xFFFF0000u)};
    float z[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) z[i] = tail == 1 ? y[i] + t[i] : y[i] * t[i];
    o = u32x2{pack_bf16(z[0], z[1]), pack_bf16(z[2], z[3])};
  }
  return o;
}

// LDS image of an operand block: [row][8 chunks of 8 k], chunk slot XOR-swizzled by the row so that every
// group of 8 consecutive lanes hits 8 distinct 16-byte slots in all three access patterns: fragment
// reads (8 consecutive rows), activation copies (4 rows x 2 chunks) and dequantised weight writes
// (rows 8 apart x 2 chunks).
__device__ __forceinline__ int lds_swz(int row) { return (((row << 1) & 6) | ((row >> 2) & 1)) ^ (((row >> 3) & 3) << 1); }
__device__ __forceinline__ int lds_chunk(int row, int kc) { return row * 8 + (kc ^ lds_swz(row)); }
// The images of the two-pass route (written by the image pass, read by the second pass as 16 rows x four chunks per
// ds_read_b128 for v_mfma_f32_16x16x32_bf16) swizzle the slot by the low three row bits instead: under that read the
// swizzle above puts pairs of lanes on one bank group (51 against 32 cycles per instruction with eight wavefronts reading),
// this one none.
__device__ __forceinline__ int lds_swz16(int row) { return row & 7; }
__device__ __forceinline__ int lds_chunk16(int row, int kc) { return row * 8 + (kc ^ lds_swz16(row)); }

// high halves of two floats -> packed bf16 pair (lo = a, hi = b); exact for dequantised weights
__device__ __forceinline__ uint32_t pack_hi(float a, float b) {
  return __builtin_amdgcn_perm(__float_as_uint(b), __float_as_uint(a), 0x07060302u);
}

// The activation of N values at once: the branches of a switch per value took longer than summing the wavefronts' shares of it
template <int N>
__device__ __forceinline__ void linear_act_rt(int act, float (&v)[N]) {
  auto all = [&](auto a) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < N; ++i) v[i] = apply_act<decltype(a)::value>(v[i]);
  };
  if (act == TTM_ACT_NONE) return;   // uniform
  switch (act) {
  case TTM_ACT_GELU: all(std::integral_constant<int, TTM_ACT_GELU>{}); break;
  case TTM_ACT_SILU: all(std::integral_constant<int, TTM_ACT_SILU>{}); break;
  case TTM_ACT_SIGMOID: all(std::integral_constant<int, TTM_ACT_SIGMOID>{}); break;
  case TTM_ACT_RELU: all(std::integral_constant<int, TTM_ACT_RELU>{}); break;
  }
}
// act0(a) x act1(b) of a gated pair, the factors rounded to bf16 as the two projections alone would store them
__device__ __forceinline__ u32x2 glu_quad(const float *a, const float *b) {
  const u32x2 g = {pack_bf16(a[0], a[1]), pack_bf16(a[2], a[3])}, u = {pack_bf16(b[0], b[1]), pack_bf16(b[2], b[3])};
  const float z[4] = {__uint_as_float(g.x << 16) * __uint_as_float(u.x << 16), __uint_as_float(g.x & 0xFFFF0000u) * __uint_as_float(u.x & 0xFFFF0000u),
                      __uint_as_float(g.y << 16) * __uint_as_float(u.y << 16), __uint_as_float(g.y & 0xFFFF0000u) * __uint_as_float(u.y & 0xFFFF0000u)};
  return u32x2{pack_bf16(z[0], z[1]), pack_bf16(z[2], z[3])};
}
typedef float f32x4v __attribute__((ext_vector_type(4)));

// 4 x 4 transpose of dwords within every quad of lanes: lane q ends up with dword q of the rows that lanes 0..3 hold
__device__ __forceinline__ void quad_transpose(uint32_t *v, int lane) {
  const bool odd = (lane & 1) != 0, hi = (lane & 2) != 0;
#pragma unroll
  for (int a = 0; a < 4; a += 2) {   // lanes 2 j and 2 j + 1 exchange (v[a + 1] of the even, v[a] of the odd)
    const uint32_t ta = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v[a], 0xB1, 0xF, 0xF, true);
    const uint32_t tb = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v[a + 1], 0xB1, 0xF, 0xF, true);
    v[a + 1] = odd ? v[a + 1] : ta;
    v[a] = odd ? tb : v[a];
  }
#pragma unroll
  for (int a = 0; a < 2; ++a) {      // lanes j and j + 2 exchange (v[a + 2] of the lower, v[a] of the upper)
    const uint32_t ta = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v[a], 0x4E, 0xF, 0xF, true);
    const uint32_t tb = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v[a + 2], 0x4E, 0xF, 0xF, true);
    v[a + 2] = hi ? v[a + 2] : ta;
    v[a] = hi ? tb : v[a];
  }
}


// ---- bfp4_b operands of the kernels that keep weights in registers (decode and mid-size): a lane's 8 (k) x 4 (n) block
// Load: the four lanes of a quad need 8 k rows x 8 bytes, one 64-byte half of a face; each fetches two whole rows with one 16-byte load (eight
// 2-byte words took 8 loads and 128 line look-ups per tile pair) and the quad transposes: pk[i] = the lane's four nibbles of the rows 2 i and 2 i + 1.
__device__ __forceinline__ void bfp4_rows(const u32x4 &x, int lane, uint32_t (&pk)[4]) {
  pk[0] = __builtin_amdgcn_perm(x.z, x.x, 0x05040100u); pk[1] = __builtin_amdgcn_perm(x.z, x.x, 0x07060302u);
  pk[2] = __builtin_amdgcn_perm(x.w, x.y, 0x05040100u); pk[3] = __builtin_amdgcn_perm(x.w, x.y, 0x07060302u);
  quad_transpose(pk, lane);
}
// (257 - E) << 7 of the rows 2 i and 2 i + 1 in the halves of a word
__device__ __forceinline__ uint32_t bfp4_exponent_pair(const u32x2 &ex, int i) {
  return (0x01010101u - __builtin_amdgcn_perm(0u, i < 2 ? ex.x : ex.y, (i & 1) ? 0x0c030c02u : 0x0c010c00u)) << 7;
}
__device__ __forceinline__ void bfp4_exponents(const u32x2 &ex, uint32_t (&sub)[4]) {
#pragma unroll
  for (int i = 0; i < 4; ++i) sub[i] = bfp4_exponent_pair(ex, i);
}
// The columns n and n + 2 (n = 0, 1) as bf16 pairs along k.  A magnitude of 1 .. 7 has four fractions and three exponents: v_perm looks the
// two bytes of 0x7F80 + (its bf16 less that of 1) up for four elements at once, 0 for a magnitude of 0; less (257 - E) << 7, saturating at zero, that
// is the bf16 of magnitude x 2^(E - 129).  From exponent 2 down the value may be a subnormal bf16, of which the subtraction loses the leading one: it comes
// out at most 2^-127 too small (half the smallest normal number; flushing those exponents, as two conversions to float did, is off by up to 7 x 2^-127).
// Exponent 255 stands over rows with an infinity (magnitude 4, infinite again) or a NaN (5 .. 7: NaN).  100 vector instructions for a block, where the
// conversions took 205 and the two-term operand 100 with twice the matrix instructions.  To flush them to zero took 3.5 % of the time
// over 200 shapes, exact values behind a branch 5.5 %, and up to 40 % where ragged outputs take the branch for their padding.
__device__ __forceinline__ void bfp4_pair(uint32_t pk, uint32_t sub, int n, uint32_t &w0, uint32_t &w2) {
  typedef unsigned short u16x2 __attribute__((ext_vector_type(2)));
  const uint32_t sel = (n ? pk >> 4 : pk) & 0x07070707u;
  const uint32_t lo = __builtin_amdgcn_perm(0xE0C0A080u, 0x40008000u, sel), hi = __builtin_amdgcn_perm(0x80808080u, 0x80807F00u, sel);
  const uint32_t a = __builtin_amdgcn_perm(hi, lo, 0x06020400u), b = __builtin_amdgcn_perm(hi, lo, 0x07030501u);
  const u16x2 x = __builtin_elementwise_sub_sat(*(const u16x2 *)&a, *(const u16x2 *)&sub), y = __builtin_elementwise_sub_sat(*(const u16x2 *)&b, *(const u16x2 *)&sub);
  w0 = *(const uint32_t *)&x | (n ? (pk & 0x00800080u) << 8 : (pk & 0x00080008u) << 12);
  w2 = *(const uint32_t *)&y | (n ? pk & 0x80008000u : (pk & 0x08000800u) << 4);
}
__device__ __forceinline__ void bfp4_columns(const uint32_t (&pk)[4], const uint32_t (&sub)[4], int n, u32x4 &w0, u32x4 &w2) {
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    uint32_t a, b;
    bfp4_pair(pk[i], sub[i], n, a, b);
    w0[i] = a;
    w2[i] = b;
  }
}

static inline int device_cu_count() {
  static int cus = 0;
  if (cus == 0) {
    int dev = 0, n = 0;
    if (hipGetDevice(&dev) == hipSuccess && hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) == hipSuccess && n > 0) cus = n;
    else cus = 256;
  }
  return cus;
}

// column units of `unit_tiles` tiles in a launch: a group numbers its members' units one after another
static inline int column_units(const LinearArgs &p, int unit_tiles) {
  if (p.group_n <= 1) return (p.Nt + unit_tiles - 1) / unit_tiles;
  int n = 0;
  for (int j = 0; j < p.group_n; ++j) n += (p.gNt[j] + unit_tiles - 1) / unit_tiles;
  return n;
}


// Split-K partial sums -> output (ttm_linear.hip): grid ((per / 4 + 255) / 256, 1, batch) of 256 lanes, per = Mt * Nt * 1024
void ttm_linear_launch_reduce(const LinearArgs &p, int64_t batch, hipStream_t s);

// The mid-size kernel (ttm_linear_mid.hip).  Launch plan: row tiles per workgroup, shares of K in a workgroup (wavefronts), slices
// of K over grid.y, modelled time.
struct MidPlan {
  int mt = 0, wk = 8, slices = 1;
  double us = 0;
};
MidPlan ttm_linear_plan_mid(const LinearArgs &p, int wf, bool glu, int max_slices = 16);
int ttm_linear_launch_mid(const LinearArgs &a, int wf, const MidPlan &plan, int64_t batch, bool glu, hipStream_t s);
