// Dense contraction at row counts between decode and prefill, and small products (see ttm_linear.hip for the operands).
#include <algorithm>

#include "ttm_linear.h"

// =============================================================================================
// Mid-size kernel: row counts between the decode kernel's and those that fill the device with 256-row blocks, and any product too
// small for them.  A workgroup owns 32 MT rows x 64 columns; its 4 or 8 wavefronts are shares of K (every fourth or eighth k-tile; the
// gated form: 2 matrices x 4 shares), summed through LDS at the end.  No operand passes through LDS on the way in: weights go from global
// memory to registers and become the MFMA operand there as in the decode kernel (byte j of eight row words feeds MFMA j, whose
// row r stands for column 4 r + j), activation fragments are 16-byte loads of whole face-row halves.  That leaves no barrier in the loop and nothing to fill before it: a launch costs 3 us + its k-tiles, where
// the LDS-direct kernels' blocks cost 12 k-steps (20 us) before and after theirs - what bounded every product below some
// 10 GFLOP.  Bounds inside the loop, per 32 k of a wavefront: about 670 cycles of vector issue for the conversion of bfp8_b (bfp4_b: 400, bf16
// weights: 64), 128 MT of the matrix core, 32 + 32 MT of L1; MT = 2 balances them for short launches, MT = 4 halves the weight
// traffic and conversions where the row count fills it.  Vector issue and products mostly add up (512 rows x 14336 x 4096: 74k and 57k of 150k
// cycles per SIMD with bfp4_b, 99k and 57k of 169k with bfp8_b; interleaving one column's products with the next one's conversion gave nothing).
// bfp4_b by table look-up: 74.9 -> 63.4 us there, 113 rows x 5515 x 5253 28.8 -> 21.2, 259 x 576 x 8256 12.5 -> 10.7.
// =============================================================================================
template <int WF, int MT, int WK, bool TT, bool GLU, class ARGS>
__global__ __launch_bounds__((GLU ? 2 : 1) * WK * 64) void ttm_linear_mid_k(ARGS args) {
  const LinearArgs p = args.full();
  constexpr int WN = GLU ? 2 : 1;    // column pairs of the workgroup
  constexpr int THREADS = WN * WK * 64, D = 2;
  __shared__ f32x4v part[WN * WK * 512];   // partial sums of one row tile: per wavefront 8 x 64 float4 = 8 KiB
  constexpr bool BFP = WF == WF_BFP8 || WF == WF_BFP4;
  constexpr uint32_t TB = WF == WF_BFP8 ? 1088u : WF == WF_BFP4 ? 576u : 2048u;
  constexpr uint32_t FACE = WF == WF_BFP8 ? 256u : WF == WF_BFP4 ? 128u : 512u, ROW = FACE / 16;
  constexpr int RW = WF == WF_BFP8 ? 8 : WF == WF_BFP4 ? 4 : 16;   // dwords of weights per lane, k-tile and column pair
  static_assert(!TT || BFP, "block-float weights");
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), wn = GLU ? wave / WK : 0, wk = wave & (WK - 1);
  // row blocks of one column unit are neighbours on one XCD: its L2 serves the weights to all but the first of them
  const int mblocks = (p.Mt + MT - 1) / MT;
  const int slot = (int)blockIdx.x >> 3, mt0 = slot % mblocks * MT;
  int cg = slot / mblocks * 8 + ((int)blockIdx.x & 7);
  if (cg >= p.n_blocks) return;
  int Nt = p.Nt, tile_base = 0, act = p.act;
  const uint8_t *A = p.A + (int64_t)blockIdx.z * p.a_batch;
  const uint8_t *W = p.W + (int64_t)blockIdx.z * p.w_batch;
  uint8_t *C = p.C + (int64_t)blockIdx.z * p.c_batch;
  if constexpr (GLU) {
    C = p.gC[0]; Nt = p.gNt[0];
  } else if (p.group_n > 1) {   // workgroup-uniform
    const GroupMember m = group_member(p, cg, 2);
    W = m.W; C = m.C; Nt = m.Nt; cg = m.local; tile_base = m.tile_base; act = m.act;
  }
  const int q16 = lane & 15, kg = lane >> 4;   // weight operand row and 8-k group of this lane
  const int fc = (q16 >> 2) & 1, quad = q16 & 3, fr = kg >> 1, half = kg & 1;
  if (GLU) W = wn ? p.gW[1] : p.gW[0];
  const uint32_t nt_l = (uint32_t)min(2 * cg + (q16 >> 3), Nt - 1);
  // bfp8_b: two whole 16-byte rows of the quad's 128-byte line; bfp4_b: two whole 8-byte rows of its 64; bf16 [K, N]: eight 8-byte words;
  // bf16 [N, K]: the 8 k of each of the four columns
  const uint32_t offW = WF == WF_BF16_NK ? (uint32_t)(fc * 1024 + quad * 128 + fr * 512 + half * 16)
                                         : nt_l * TB + (BFP ? 64u : 0u) + (fr * 2 + fc) * FACE + half * (FACE / 2) + quad * (BFP ? 16 : ROW / 4);
  const uint32_t offE = nt_l * TB + (fr * 2 + fc) * 16 + half * 8;
  const uint32_t offA = fr * 512 + q16 * 32 + half * 16;
  int64_t rowA[MT];
#pragma unroll
  for (int r = 0; r < MT; ++r) rowA[r] = (int64_t)min(mt0 + r, p.Mt - 1) * p.Kt * 2048;

  // accs: the sums over the S terms; bfp4_b, whose operand is one term: of the activations times zero (see launch_mid)
  f32x4v acc[2 * MT][4], accs[TT ? 2 * MT : 1][WF == WF_BFP4 ? 1 : 4];
#pragma unroll
  for (int h = 0; h < 2 * MT; ++h)
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      acc[h][j] = f32x4v{0.f, 0.f, 0.f, 0.f};
      if (TT && (j == 0 || WF != WF_BFP4)) accs[h][j] = f32x4v{0.f, 0.f, 0.f, 0.f};
    }
  uint32_t rows[D][RW];
  u32x2 ex[D];
  bool live[D];
  u32x4 af[D][2 * MT];
  const int kbase = p.partial ? (int)blockIdx.y * p.k_slice : 0;
  const int kend = p.partial ? min(kbase + p.k_slice, p.Kt) : p.Kt;
  const int nchunks = (kend - kbase + WK - 1) / WK;
  auto load_slot = [&](int s, int c) __attribute__((always_inline)) {
    const int kt = kbase + wk + WK * c, ktc = min(kt, kend - 1);
    live[s] = kt < kend;
    uint32_t *rw = rows[s];
    if constexpr (WF == WF_BF16_NK) {
      const uint8_t *Wk = W + ((int64_t)nt_l * p.Kt + ktc) * TB + offW;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const u32x4 x = *(const u32x4 *)(Wk + j * 32);
        rw[4 * j] = x.x; rw[4 * j + 1] = x.y; rw[4 * j + 2] = x.z; rw[4 * j + 3] = x.w;
      }
    } else {
      const uint8_t *Wt = W + (int64_t)ktc * Nt * TB, *Wk = Wt + offW;
      if constexpr (WF == WF_BFP8) {
        const u32x4 x = *(const u32x4 *)Wk, y = *(const u32x4 *)(Wk + 64);
        rw[0] = x.x; rw[1] = x.y; rw[2] = x.z; rw[3] = x.w;
        rw[4] = y.x; rw[5] = y.y; rw[6] = y.z; rw[7] = y.w;
      } else if constexpr (WF == WF_BFP4) {
        const u32x4 x = *(const u32x4 *)Wk;
        rw[0] = x.x; rw[1] = x.y; rw[2] = x.z; rw[3] = x.w;
      } else {
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          const u32x2 x = *(const u32x2 *)(Wk + i * ROW);
          rw[2 * i] = x.x; rw[2 * i + 1] = x.y;
        }
      }
      if constexpr (BFP) ex[s] = *(const u32x2 *)(Wt + offE);
    }
#pragma unroll
    for (int h = 0; h < 2 * MT; ++h) af[s][h] = *(const u32x4 *)(A + rowA[h >> 1] + (int64_t)ktc * 2048 + offA + (h & 1) * 1024);
  };
  auto process = [&](int s) __attribute__((always_inline)) {
    if (!live[s]) return;   // wavefront-uniform: a k-tile past the end contributes nothing
    uint32_t *rw = rows[s];
    if constexpr (WF == WF_BFP4) {
      uint32_t pk[4], sub[4];
      bfp4_rows(u32x4{rw[0], rw[1], rw[2], rw[3]}, lane, pk);
      bfp4_exponents(ex[s], sub);
#pragma unroll
      for (int n = 0; n < 2; ++n) {
        u32x4 w[2];
        bfp4_columns(pk, sub, n, w[0], w[1]);
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
          for (int h = 0; h < 2 * MT; ++h)
            acc[h][n + 2 * j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(*(bf16x8 *)&w[j], *(bf16x8 *)&af[s][h], acc[h][n + 2 * j], 0, 0, 0);
        if constexpr (MT > 2) __builtin_amdgcn_sched_barrier(0);   // two columns' operands at a time: more of them do not fit the registers
      }
      if constexpr (TT) {
        const u32x4 none = {0, 0, 0, 0};
#pragma unroll
        for (int h = 0; h < 2 * MT; ++h) accs[h][0] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(*(const bf16x8 *)&none, *(bf16x8 *)&af[s][h], accs[h][0], 0, 0, 0);
      }
      return;
    }
    if constexpr (TT && WF == WF_BFP8) {
      quad_transpose(rw, lane); quad_transpose(rw + 4, lane);
      // (E + 1) << 7 for the rows 2 ip and 2 ip + 1, in the two halves of a word; E is capped so that the field stays 8 bits
      uint32_t epk[4];
#pragma unroll
      for (int ip = 0; ip < 4; ++ip) {
        uint32_t e2 = __builtin_amdgcn_perm(0u, ip < 2 ? ex[s].x : ex[s].y, (ip & 1) ? 0x0c030c02u : 0x0c010c00u);
        typedef unsigned short u16x2 __attribute__((ext_vector_type(2)));
        const u16x2 capped = __builtin_elementwise_min(*(const u16x2 *)&e2, u16x2{0xFD, 0xFD});
        e2 = *(const uint32_t *)&capped;
        epk[ip] = (e2 + 0x00010001u) << 7;
      }
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        u32x4 wv, ws;
#pragma unroll
        for (int ip = 0; ip < 4; ++ip) {
          const uint32_t q = __builtin_amdgcn_perm(rw[2 * ip + 1], rw[2 * ip], 0x0c040c00u + 0x00010001u * j);
          ws[ip] = ((q & 0x00800080u) << 8) | epk[ip];
          wv[ip] = (q & 0x007F007Fu) | ws[ip];
        }
#pragma unroll
        for (int h = 0; h < 2 * MT; ++h) {
          acc[h][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(*(bf16x8 *)&wv, *(bf16x8 *)&af[s][h], acc[h][j], 0, 0, 0);
          accs[h][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(*(bf16x8 *)&ws, *(bf16x8 *)&af[s][h], accs[h][j], 0, 0, 0);
        }
      }
      return;
    }
    float scale[8], nscale[8];
    uint32_t t[8];
    if constexpr (WF == WF_BFP8) {
      quad_transpose(rw, lane); quad_transpose(rw + 4, lane);
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        uint32_t E = ((i < 4 ? ex[s].x : ex[s].y) >> (8 * (i & 3))) & 0xFFu;
        // value = magnitude x 2^(E - 127 - 6); smaller exponents flush to zero
        E = max(E, 6u);
        scale[i] = __uint_as_float((E - 6u) << 23);
        nscale[i] = -128.0f * scale[i];
        const uint32_t d = rw[i], sg = d & 0x80808080u, sb = sg >> 7;
        t[i] = (d ^ 0x80808080u ^ (sg - sb)) + sb;
      }
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      u32x4 w;
      if constexpr (WF == WF_BFP8) {
        float f[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) f[i] = fmaf((float)((t[i] >> (8 * j)) & 0xFFu), scale[i], nscale[i]);
        w = u32x4{pack_hi(f[0], f[1]), pack_hi(f[2], f[3]), pack_hi(f[4], f[5]), pack_hi(f[6], f[7])};
      } else if constexpr (WF == WF_BF16_KN) {
        const uint32_t sel = (j & 1) ? 0x07060302u : 0x05040100u;
#pragma unroll
        for (int i = 0; i < 4; ++i) w[i] = __builtin_amdgcn_perm(rw[4 * i + 2 + (j >> 1)], rw[4 * i + (j >> 1)], sel);
      } else {
        w = u32x4{rw[4 * j], rw[4 * j + 1], rw[4 * j + 2], rw[4 * j + 3]};
      }
#pragma unroll
      for (int h = 0; h < 2 * MT; ++h)
        acc[h][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(*(bf16x8 *)&w, *(bf16x8 *)&af[s][h], acc[h][j], 0, 0, 0);
      if constexpr (MT > 2) __builtin_amdgcn_sched_barrier(0);   // one column's operand at a time: more of them do not fit the registers
    }
  };
#pragma unroll
  for (int s = 0; s < D; ++s) {
    load_slot(s, s);
    __builtin_amdgcn_sched_barrier(0);
  }
  for (int c0 = 0; c0 < nchunks; c0 += D) {
#pragma unroll
    for (int s = 0; s < D; ++s) {
      process(s);
      __builtin_amdgcn_sched_barrier(0);   // keep the loads in slot order, D - 1 slots ahead of their use
      load_slot(s, c0 + s + D);
      __builtin_amdgcn_sched_barrier(0);
    }
  }

  if constexpr (TT) {
#pragma unroll
    for (int h = 0; h < 2 * MT; ++h)
#pragma unroll
      for (int j = 0; j < 4; ++j) acc[h][j] -= accs[h][WF == WF_BFP4 ? 0 : j];
  }
  // one row tile at a time: the wavefronts' sums -> LDS as float4 (four consecutive n of one m), then the threads finish the 512
  // slots, (h, i, lane) = (t >> 8, (t >> 6) & 3, t & 63)
  static_assert(THREADS == 256 || THREADS == 512, "element() counts four wavefronts per pass");
  constexpr int T = 512 / THREADS;
  const int n_in = 16 * (kg & 1) + 4 * (wave & 3), nt = 2 * cg + (kg >> 1), ntc = min(nt, Nt - 1);
  const u32x2 bias = !GLU && p.bias && !p.partial ? bias_quad(p, ntc, n_in) : u32x2{0, 0};
  const float bv[4] = {__uint_as_float(bias.x << 16), __uint_as_float(bias.x & 0xFFFF0000u), __uint_as_float(bias.y << 16), __uint_as_float(bias.y & 0xFFFF0000u)};
  auto element = [&](int t) __attribute__((always_inline)) { return (((wave + 4 * t) >> 2) * 2 + (n_in >> 4)) * 256 + q16 * 16 + (n_in & 15); };
#pragma unroll
  for (int r = 0; r < MT; ++r) {
    if (mt0 + r >= p.Mt) break;      // workgroup-uniform
    u32x2 tail[T];
#pragma unroll
    for (int t = 0; t < T; ++t)
      tail[t] = !GLU && p.tail && !p.partial ? *(const u32x2 *)(C + (((int64_t)(mt0 + r) * Nt + ntc) * 1024 + element(t)) * 2 + p.tail_delta) : u32x2{0, 0};
    if (r > 0) __syncthreads();
#pragma unroll
    for (int hh = 0; hh < 2; ++hh)
#pragma unroll
      for (int ii = 0; ii < 4; ++ii)
        part[(wave * 8 + hh * 4 + ii) * 64 + lane] = f32x4v{acc[2 * r + hh][0][ii], acc[2 * r + hh][1][ii], acc[2 * r + hh][2][ii], acc[2 * r + hh][3][ii]};
    __syncthreads();
#pragma unroll
    for (int t = 0; t < T; ++t) {
      const int in = element(t), slot = t * THREADS + tid;
      if (nt >= Nt) continue;
      f32x4v sums[WN];
#pragma unroll
      for (int q = 0; q < WN; ++q) {
        sums[q] = part[q * WK * 512 + slot];
#pragma unroll
        for (int w = 1; w < WK; ++w) sums[q] += part[(q * WK + w) * 512 + slot];
      }
      uint8_t *c = C + (((int64_t)(mt0 + r) * Nt + nt) * 1024 + in) * 2;
      float v[4] = {sums[0][0], sums[0][1], sums[0][2], sums[0][3]};
      if constexpr (GLU) {
        float v1[4] = {sums[WN - 1][0], sums[WN - 1][1], sums[WN - 1][2], sums[WN - 1][3]};
        linear_act_rt(p.gAct[0], v);
        linear_act_rt(p.gAct[1], v1);
        *(u32x2 *)c = glu_quad(v, v1);
      } else if (p.partial) {   // bias, activation and rounding happen in ttm_linear_reduce_k
        *(f32x4v *)(p.partial + (((int64_t)blockIdx.z * p.slices + blockIdx.y) * p.Mt + mt0 + r) * p.Nt * 1024 + (int64_t)(tile_base + nt) * 1024 + in) = sums[0];
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] += bv[e];
        linear_act_rt(act, v);
        *(u32x2 *)c = finish_quad(p.tail, tail[t], v);
      }
    }
  }
}

// ---- the mid-size kernel's launch plan
static int mid_units(const LinearArgs &p, bool glu) { return glu ? (p.gNt[0] + 1) / 2 : column_units(p, 2); }

// The model was fitted to 2700 random shapes (33 .. 2048 rows, weights of 512 .. 8192 x 512 .. 14336, all formats) under every plan, two terms of it to
// 1000 more: 5 % rms (bf16 8 %) for the plan it picks, which is 0.3 % slower than the best one on average, 2 % at the 95th percentile (one without figures of their
// own for the formats and wavefront counts 2 - 3 %, 15 %: 113 rows x 5515 x 5253 bfp4_b 21.2 / 18.4 us, 64 x 4096 x 14336
// bfp8_b 19.8 / 17.8).  us = 3.0 for launch, first loads and the last wavefronts; per round of workgroups the k-tiles that
// the wavefronts of a SIMD take and the sums through LDS; for a split K the reduction's launch and its traffic.
MidPlan ttm_linear_plan_mid(const LinearArgs &p, int wf, bool glu, int max_slices) {
  // option linear_mid: 0 by the model, 1 never, 1000 * shares + 100 * row tiles + slices pins a plan
  const int force = ttm_option("linear_mid");
  MidPlan best;
  best.us = 1e30;
  const int cus = device_cu_count(), units = mid_units(p, glu);
  // a lane's place in a k row of weights is a 32-bit offset
  if (wf != WF_BF16_NK && (int64_t)(glu ? p.gNt[0] : p.Nt) * 2048 >= (int64_t)1 << 32) return best;
  const int f = wf == WF_BFP8 ? 0 : wf == WF_BFP4 ? 1 : 2;
  // row tiles, shares of K; us of the sums of a round; how whole a last round counts (two or three of the smaller workgroups share a CU), and every
  // round behind the first; us per k-tile of a wavefront of bfp8_b / bfp4_b / bf16 weights (wavefronts of a SIMD share it, so they add up)
  static const struct { int mt, wk; double sums, whole, further, chunk[3], drift; } kPlain[] = {{2, 4, 1.57, 0.75, 0.87, {0.440, 0.356, 0.466}, 0.75e-4},
                                                                                                {1, 8, 0.64, 0.87, 1.00, {0.297, 0.242, 0.345}, 0.0},
                                                                                                {2, 8, 2.15, 0.89, 1.25, {0.355, 0.285, 0.391}, 2.30e-4},
                                                                                                {4, 8, 4.74, 0.84, 1.17, {0.491, 0.414, 0.565}, 0.95e-4}};
  // the gated form: eight wavefronts, four shares of K of either matrix (36 shapes)
  static const struct { int mt, wk; double sums, chunk; } kGated[] = {{2, 4, 2.1, 0.44}, {4, 4, 4.0, 0.57}};
  static const double kAlone[3] = {1.08, 1.0, 0.80};   // of a k-tile where a SIMD has one wavefront
  // us per slice of K beside the reduction's launch and traffic: with bf16 weights alone (1085 shapes of 1 .. 2048 rows: the plan picked is 0.36 % slower
  // than the best one, without the term 0.69 %, [36, 2432] x [2432, 3424] 11.6 us in four slices, 9.8 in one)
  static const double kSlice[3] = {0.0, 0.0, 0.3};
  // Every column unit passes all activations by; beyond 1024 rows the workgroups of a unit drift apart along K and out of their XCD's L2 the further, the more
  // there are: kPlain's last figure (of the workgroups of 64 rows on half a CU per round) per row tile beyond 32 and MB of activations, times this.
  // Over 834 shapes of 1000 .. 2048 rows the modelled time of the plan picked is 5 % rms off (6 / 9 / 6 % without, bfp8_b / bfp4_b / bf16) and the plan
  // 0.13 % slower than the best one (0.31 %): 1900 rows x 3000 x 3400 bfp4_b 84 us with 64 rows, modelled at 62 before; 1952 x 3872 x 3298 111, 77 before.
  static const double kDrift[3] = {1.0, 2.0, 0.9};
  const auto consider = [&](int mt, int wk, double sums, double whole, double further, double chunk, double drift) {
    const int blocks = (units + 7) / 8 * 8 * ((p.Mt + mt - 1) / mt) * p.plan_batch;   // a column unit's row blocks run on one XCD
    for (int slices = 1; slices <= (glu ? 1 : max_slices); slices *= 2) {
      if (force >= 1000) {
        if (force / 1000 != wk || force % 1000 / 100 != mt || force % 100 != slices) continue;
      } else if ((mt > 1 && mt >= 2 * p.Mt) || (slices > 1 && p.Kt < 2 * wk * slices)) {
        continue;
      }
      const int kt = (p.Kt + slices - 1) / slices, chunks = (kt + wk - 1) / wk, rounds = (blocks * slices + cus - 1) / cus;
      if (force < 1000 && rounds > 8) continue;   // beyond what was measured; larger blocks amortise their ends better
      const double r = rounds > 1 ? 1 + further * (whole * rounds + (1 - whole) * blocks * slices / cus - 1) : 1.0;
      double us;
      if (glu) us = 3.3 + r * 2 * chunks * chunk + r * sums;
      else us = 3.0 + r * (wk / 4) * chunks * chunk * (wk == 4 && rounds == 1 ? kAlone[f] : 1.0) + (wk == 8 ? r : 0.5 + 0.5 * r) * sums;
      us *= 1 + drift * (wk == 4 ? (double)blocks * slices / cus : 1.0) * std::max(0, p.Mt - 32) * p.Mt * p.Kt * 2048e-6;
      if (slices > 1) us += 2.65 + kSlice[f] * slices + (slices + 0.5) * (double)p.Mt * p.Nt * p.plan_batch * 4096.0 / 3.8e6;
      if (us < best.us) { best.us = us; best.mt = mt; best.wk = wk; best.slices = slices; }
    }
  };
  if (glu) {
    for (const auto &k : kGated) consider(k.mt, k.wk, k.sums, 1.0, 1.0, k.chunk, 0.0);
  } else {
    for (const auto &k : kPlain) consider(k.mt, k.wk, k.sums, k.whole, k.further, k.chunk[f], kDrift[f] * k.drift);
  }
  return best;
}

template <int WF, int MT, int WK, bool TT>
static void launch_mid_mt(const LinearArgs &p, dim3 grid, hipStream_t s) {
  if (p.group_n > 1) hipLaunchKernelGGL((ttm_linear_mid_k<WF, MT, WK, TT && (WF == WF_BFP8 || WF == WF_BFP4), false, LinearArgs>), grid, dim3(WK * 64), 0, s, p);
  else hipLaunchKernelGGL((ttm_linear_mid_k<WF, MT, WK, TT && (WF == WF_BFP8 || WF == WF_BFP4), false, LinearPlain>), grid, dim3(WK * 64), 0, s, LinearPlain(p));
}
template <int WF>
static int launch_mid(const LinearArgs &a, const MidPlan &plan, int64_t batch, bool glu, hipStream_t s) {
  LinearArgs p = a;
  int slices = plan.slices;
  p.partial = nullptr;
  p.k_slice = p.Kt;
  const int64_t per = (int64_t)p.Mt * p.Nt * 1024;
  if (slices > 1) {   // a pinned split of a short K may come down to fewer slices, or to one
    p.k_slice = (p.Kt + slices - 1) / slices;
    slices = (p.Kt + p.k_slice - 1) / p.k_slice;
  }
  if (slices > 1) {
    void *ws = nullptr;
    if (int rc = ttm_stream_workspace(s, (size_t)(per * slices * batch) * sizeof(float), &ws)) return rc;
    p.partial = (float *)ws;
  }
  p.slices = slices;
  p.n_blocks = mid_units(a, glu);
  const dim3 grid((unsigned)((p.n_blocks + 7) / 8 * 8 * ((p.Mt + plan.mt - 1) / plan.mt)), (unsigned)slices, (unsigned)batch);
  if (glu) {
    if constexpr (WF == WF_BFP8) {
      if (plan.mt == 2) hipLaunchKernelGGL((ttm_linear_mid_k<WF_BFP8, 2, 4, false, true, LinearArgs>), grid, dim3(512), 0, s, p);
      else hipLaunchKernelGGL((ttm_linear_mid_k<WF_BFP8, 4, 4, false, true, LinearArgs>), grid, dim3(512), 0, s, p);
      return 0;
    }
    return ttm_set_error(TTM_ERR_INVALID, "ttm_linear_glu: the mid-size kernel's gated form takes bfp8_b weights");
  }
  switch (plan.wk * 10 + plan.mt) {
  case 81:
    // The two-term operand of bfp8_b (1.m and 1.0 products, subtracted at the end) saves conversion work, but an infinite activation leaves
    // inf - inf: only up to 64 rows, where the decode kernel multiplies the same way.  bfp4_b has one term and adds the activations times zero there,
    // so that such a row is NaN in every column whatever the format.
    if (a.Mt <= 2) launch_mid_mt<WF, 1, 8, true>(p, grid, s);
    else launch_mid_mt<WF, 1, 8, false>(p, grid, s);
    break;
  case 82: launch_mid_mt<WF, 2, 8, false>(p, grid, s); break;
  case 84: launch_mid_mt<WF, 4, 8, false>(p, grid, s); break;
  default: launch_mid_mt<WF, 2, 4, false>(p, grid, s);   // 42: ttm_linear_plan_mid has no others
  }
  if (slices > 1)
    ttm_linear_launch_reduce(p, batch, s);
  return 0;
}


int ttm_linear_launch_mid(const LinearArgs &a, int wf, const MidPlan &best, int64_t batch, bool glu, hipStream_t s) {
  MidPlan plan = best;
  // A recording stream cannot allocate the slices' partial sums: unless an earlier call left room for them, the best plan without
  // (the kernels this one took over from ran such products unsplit, so they could always be recorded)
  if (plan.slices > 1 && ttm_option("linear_mid") < 1000 &&
      !ttm_stream_workspace_ready(s, (size_t)((int64_t)a.Mt * a.Nt * 1024 * plan.slices * batch) * sizeof(float)))
    plan = ttm_linear_plan_mid(a, wf, glu, 1);
  if (plan.mt == 0)
    return ttm_set_error(TTM_ERR_INVALID, "ttm_linear: no such plan of the mid-size kernel%s (linear_mid = %d)", glu ? "'s gated form" : "", ttm_option("linear_mid"));
  switch (wf) {
  case WF_BFP8: return launch_mid<WF_BFP8>(a, plan, batch, glu, s);
  case WF_BFP4: return launch_mid<WF_BFP4>(a, plan, batch, glu, s);
  case WF_BF16_KN: return launch_mid<WF_BF16_KN>(a, plan, batch, glu, s);
  default: return launch_mid<WF_BF16_NK>(a, plan, batch, glu, s);
  }
}
