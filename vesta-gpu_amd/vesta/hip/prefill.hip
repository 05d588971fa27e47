// Multi-token prefill for the GPT-2 program on gfx950: the P prompt positions
// of all B rows go through each layer together (M = B * P rows), so the
// projections are matrix products on the matrix cores instead of P decode
// steps. With P = 1 the same launches are one step of the layered decode
// engine. Appended to the prelude (hip/prelude.h, VBLOCK 256) and compiled at
// run time by hipRTC.
//
// Row m of every activation buffer is position p = m % P of batch row
// b = m / P, at sequence position t0 + p, t0 read from the device (the
// model's position counter, advanced by P at the end). The residual and the
// queries are fp32 [M, width]; what a product reads is in fragment order
// (below). The key/value cache is the decode kernel's [B, L, tmax, H, 64]
// fp16. Positions at or past tmax write no cache row and attend to rows
// 0 .. tmax - 1 only.
//
// Arithmetic follows the program's statements (fp16 weights, fp32 math, the
// cache rounded to fp16 before attention reads it); products run on
// v_mfma_f32_16x16x32_f16 with every activation split into two fp16 halves
// (hi + lo / 2048: 22 significant bits at any magnitude), each half's products
// accumulated in fp32 on its own and combined at the end. The attention's
// contractions run there too, its queries and softmax weights in three planes
// (pf_split24), so that they keep fp32's 24 bits.

#define PF_E 64                 // head width

// ---------------------------------------------------------------- fragment order
// Every product reads both operands in the
// order the matrix cores take them (v_mfma_f32_16x16x32_f16: lane l = 16 q + r
// holds row r, fold positions 8 q .. 8 q + 7 of a 16 x 32 operand tile), so
// that each operand load of a wave is one contiguous kilobyte:
//   weights      Wf[n-tile][k-step][lane][8]         n = 16 n-tile + r
//   activations  Af[plane][m-tile][k-step][lane][8]  m = 16 m-tile + r
// with k = 32 k-step + 8 q + e; plane 0 holds the nearest fp16 (hi), plane 1
// the remainder scaled by 2^11 (vh_split8s). MT m-tiles, KT k-steps; rows
// past the last real one are never written and only reach discarded outputs.
// A producer of an activation row stores eight values k8 .. k8 + 7 (k8 a
// multiple of 8) of row m at once; `bad` is raised for a value beyond the
// fp16 range.
__device__ __forceinline__ void pf_frag_put8(vh_half* __restrict__ F, int MT, int KT, int m, int k8, const float* v,
                                             bool& bad) {
  bad |= vh_beyond_half8(v);
  vh_u32x4 hi, lo;
  vh_split8s(v, hi, lo);
  const size_t at = (((size_t)(m >> 4) * KT + (k8 >> 5)) * 64 + ((k8 >> 3) & 3) * 16 + (m & 15)) * 8;
  *(vh_u32x4*)(F + at) = hi;
  *(vh_u32x4*)(F + (size_t)MT * KT * 512 + at) = lo;
}

// The same for four values k4 .. k4 + 3 (k4 a multiple of 4; 8-byte stores):
// what a lane holds of a product's output tile taken with the weights as the
// row operand (four consecutive outputs of one activation row).
__device__ __forceinline__ void pf_frag_put4(vh_half* __restrict__ F, int MT, int KT, int m, int k4, const float* v,
                                             bool& bad) {
  typedef _Float16 h4 __attribute__((ext_vector_type(4)));
  h4 hi, lo;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    bad |= !(__builtin_fabsf(v[j]) <= VH_HALF_MAX);
    hi[j] = (_Float16)v[j];
    lo[j] = (_Float16)((v[j] - (float)hi[j]) * VH_LO_SCALE);
  }
  const size_t at = (((size_t)(m >> 4) * KT + (k4 >> 5)) * 64 + ((k4 >> 3) & 3) * 16 + (m & 15)) * 8 + (k4 & 7);
  *(vh_u32x2*)(F + at) = __builtin_bit_cast(vh_u32x2, hi);
  *(vh_u32x2*)(F + (size_t)MT * KT * 512 + at) = __builtin_bit_cast(vh_u32x2, lo);
}

// Eight floats of at most 1 in magnitude as three fp16 planes v = hi + (lo +
// tail) / 2^11, each plane what is left, cut off (not rounded) after 11 bits:
// all 24 bits of a value down to 2^-12, smaller ones to 2^-35. The conversions
// take two values an instruction.
__device__ __forceinline__ void pf_split24(const float* v, vh_u32x4& hi, vh_u32x4& lo, vh_u32x4& tail) {
  typedef __fp16 h2 __attribute__((ext_vector_type(2)));
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const h2 h = __builtin_amdgcn_cvt_pkrtz(v[2 * j], v[2 * j + 1]);
    const float r0 = fmaf((float)h[0], -VH_LO_SCALE, v[2 * j] * VH_LO_SCALE);
    const float r1 = fmaf((float)h[1], -VH_LO_SCALE, v[2 * j + 1] * VH_LO_SCALE);
    const h2 l = __builtin_amdgcn_cvt_pkrtz(r0, r1);
    const h2 t = __builtin_amdgcn_cvt_pkrtz(r0 - (float)l[0], r1 - (float)l[1]);
    hi[j] = __builtin_bit_cast(unsigned, h);
    lo[j] = __builtin_bit_cast(unsigned, l);
    tail[j] = __builtin_bit_cast(unsigned, t);
  }
}

// ---------------------------------------------------------------- products
// C = A W over K (A [M, K] and W [N, K] in fragment order; W row n holds
// output n's weights), then the epilogue of `mode`:
//   0  out[m, n] = C + bias[n]                       (plain; bias optional)
//   1  out[m, n] = (out[m, n] + C) + bias[n]          (residual add, in place)
//   2  F[m, n] = gelu_tanh(C + bias[n])               (feed-forward widening, in fragment order)
//   3  qkv: n < D -> out[m, n] (queries); D <= n < 2D -> key cache;
//      2D <= n -> value cache, at this row's sequence position (fp16)
// Up to 64 rows the products are pf_mgemm* (waves split the fold), beyond
// pf_pgemm* (output tiles).
// gelu_tanh(u) = 0.5 u (1 + tanh(y)), y = 0.7978845608028654 (u + 0.044715 u^3),
// evaluated as u / (1 + exp(-2 y)) (0.5 (1 + tanh y) is the logistic function
// of 2 y): one exponential and one division instead of tanh; in fp32 its
// error against the exact function is that of the tanh form (5e-7 absolute
// over |u| <= 12 for either).
__device__ __forceinline__ float pf_gelu(float u) {
  const float y = 0.7978845608028654f * (u + 0.044715f * u * u * u);
  return u / (1.0f + __expf(-2.0f * y));
}

// The epilogue of one output value c = C[m, n] (modes 1 and 3).
__device__ __forceinline__ void pf_epi(int mode, int m, int n, float c, const vh_half* __restrict__ bias, int N,
                                       float* __restrict__ out, int ldo, vh_half* __restrict__ kc,
                                       vh_half* __restrict__ vc, int P, const int* __restrict__ tp, int layer,
                                       int L, int tmax) {
  const float bn = bias ? h2f(bias[n]) : 0.0f;
  if (mode == 1) {
    float* o = out + (size_t)m * ldo + n;
    *o = (*o + c) + bn;
  } else {
    const int D = N / 3;
    const float val = c + bn;
    if (n < D) {
      out[(size_t)m * ldo + n] = val;
    } else {
      const int b = m / P, pos = *tp + m % P;
      if (pos >= 0 && pos < tmax) {
        const size_t at = ((size_t)(b * L + layer) * tmax + pos) * D + (n % D);
        (n < 2 * D ? kc : vc)[at] = f2h(val);
      }
    }
  }
}

// Products of more than 64 rows. A block makes an output tile of 16 TM WM rows
// x 16 TN WN columns; its WM x WN waves hold TM x TN tiles of 16 x 16 each, hi
// and lo halves in separate accumulators (the weights are the instruction's
// row operand, so a lane ends with four consecutive outputs of one activation
// row: 16-byte residual / query stores, 8-byte fragment-order stores). The
// fold goes through LDS in double-buffered stages. Fragment order makes every
// global load one contiguous kilobyte and every LDS access conflict-free
// without padding, and the halves are made once, by the activation's producer.
// What bounds them: the matrix cores twice per product (hi and lo) at the
// clock that load leaves; at 24576 x 2304 x 768 the 128 x 256 tile takes 174
// us (500 TFLOP/s of the product, 1000 of the matrix cores; hipBLASLt's fp16
// product of the same operation count 171 us), where 64 x 64 tiles that
// converted fp32 activations in every block took 380. With few tiles a CU it
// is the tile's fixed part (first loads, epilogue: 4-8 us).
// `ks` > 1 splits the fold over blocks: part p of tile t stores its sums in
// ws[p][m][n] for pf_reduce_ln, pf_reduce or pf_reduce_frag.
//
// Tiles go to the 8 XCDs (blockIdx % 8) in contiguous runs, within a run in
// groups of 4 row tiles, so that the blocks resident on one XCD share their
// operands in its L2.
struct PfTile {
  int part, mt0, nt0;
};
template <int BM, int BN>
__device__ __forceinline__ bool pf_tile(PfTile& tl, int MT, int NT, int ks) {
  constexpr int GM = 4;
  const int ntn = (NT + BN - 1) / BN, ntm = (MT + BM - 1) / BM, T = ntn * ntm * ks;
  const int per = (T + 7) / 8, id = (int)(blockIdx.x & 7) * per + (int)(blockIdx.x >> 3);
  if ((int)(blockIdx.x >> 3) >= per || id >= T) return false;      // grid: 8 * ceil(T / 8) blocks
  const int tile = id % (ntn * ntm), g = tile / (GM * ntn), gm = min(GM, ntm - g * GM), in = tile - g * GM * ntn;
  tl.part = id / (ntn * ntm);
  tl.mt0 = (g * GM + in % gm) * BM;
  tl.nt0 = (in / gm) * BN;
  return true;
}

// A wave's TM x TN output tiles (from row tile mt0, column tile nt0) through
// the epilogue of `mode`, or into ws[part] with a split fold. Lane 16 q + r
// holds row r, columns 4 q .. + 3 of each tile. All operands of a row of tiles
// are loaded before any is used, and what differs by tile alone is scalar:
// with a load, a wait and per-lane divisions for each tile the epilogue of the
// 128 x 256 tile took about 8 us, a third of a 768-deep product (24576 x 2304
// x 768 192 -> 174 us, 8192 x 4800 x 1600 237 -> 229).
template <int TM, int TN>
__device__ __forceinline__ void pf_pgemm_out(
    const vh_f32x4 (&ah)[TM][TN], const vh_f32x4 (&al)[TM][TN], int mt0, int nt0, int part, int ks, int MT,
    const vh_half* __restrict__ bias, int M, int N, int mode, float* __restrict__ out, int ldo,
    vh_half* __restrict__ kc, vh_half* __restrict__ vc, int P, const int* __restrict__ tp, int layer, int L, int tmax,
    float* __restrict__ ws, vh_half* __restrict__ F, unsigned* __restrict__ err) {
  const int lane = threadIdx.x & 63, r = lane & 15, q = lane >> 4;
  const int m0 = 16 * mt0 + r, n0 = 16 * nt0 + 4 * q;              // this lane's row of row tile 0, column of column tile 0
  auto value = [&](int a, int b) {
    return vh_f32x4{vh_hilo(ah[a][b][0], al[a][b][0]), vh_hilo(ah[a][b][1], al[a][b][1]),
                    vh_hilo(ah[a][b][2], al[a][b][2]), vh_hilo(ah[a][b][3], al[a][b][3])};
  };
  if (ks > 1) {
    float* w = ws + ((size_t)part * M + m0) * N + n0;
#pragma unroll
    for (int a = 0; a < TM; ++a) {
      if (m0 + 16 * a >= M) continue;
#pragma unroll
      for (int b = 0; b < TN; ++b)
        if (n0 + 16 * b < N) *(vh_f32x4*)(w + (size_t)(16 * a) * N + 16 * b) = value(a, b);
    }
    return;
  }
  if (mode == 0) {                                                 // N of any size (the output head)
#pragma unroll
    for (int a = 0; a < TM; ++a)
#pragma unroll
      for (int b = 0; b < TN; ++b) {
        const vh_f32x4 v = value(a, b);
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const int m = m0 + 16 * a, n = n0 + 16 * b + j;
          if (m < M && n < N) out[(size_t)m * ldo + n] = bias ? v[j] + h2f(bias[n]) : v[j];
        }
      }
    return;
  }
  float bn[TN][4];
#pragma unroll
  for (int b = 0; b < TN; ++b) unpack4(ld8(bias + min(n0 + 16 * b, N - 4)), bn[b]);
  if (mode == 1) {
    float* o = out + (size_t)m0 * ldo + n0;
#pragma unroll
    for (int a = 0; a < TM; ++a) {
      if (m0 + 16 * a >= M) continue;
      vh_f32x4 z[TN];
#pragma unroll
      for (int b = 0; b < TN; ++b)
        z[b] = n0 + 16 * b < N ? *(const vh_f32x4*)(o + (size_t)(16 * a) * ldo + 16 * b) : vh_f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
      for (int b = 0; b < TN; ++b) {
        const vh_f32x4 v = value(a, b);
        if (n0 + 16 * b < N)
          *(vh_f32x4*)(o + (size_t)(16 * a) * ldo + 16 * b) =
              vh_f32x4{(z[b][0] + v[0]) + bn[b][0], (z[b][1] + v[1]) + bn[b][1], (z[b][2] + v[2]) + bn[b][2],
                       (z[b][3] + v[3]) + bn[b][3]};
      }
    }
    return;
  }
  if (mode == 2) {
    // fragment order: the lane's eight bytes of tile (mt0 + a, nt0 + b) are at a place of its own in half a fragment
    bool bad = false;
    const size_t at = (((q >> 1) * 16 + r) * 8) + (q & 1) * 4, plane = (size_t)MT * (N / 32) * 512;
#pragma unroll
    for (int a = 0; a < TM; ++a) {
      if (m0 + 16 * a >= M) continue;
#pragma unroll
      for (int b = 0; b < TN; ++b) {
        if (n0 + 16 * b >= N) continue;
        const vh_f32x4 v = value(a, b);
        typedef _Float16 h4 __attribute__((ext_vector_type(4)));
        h4 hi, lo;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const float g = pf_gelu(v[j] + bn[b][j]);
          bad |= !(__builtin_fabsf(g) <= VH_HALF_MAX);
          hi[j] = (_Float16)g;
          lo[j] = (_Float16)((g - (float)hi[j]) * VH_LO_SCALE);
        }
        vh_half* f = F + ((size_t)(mt0 + a) * (N / 32) + ((nt0 + b) >> 1)) * 512 + ((nt0 + b) & 1) * 256 + at;
        *(vh_u32x2*)f = __builtin_bit_cast(vh_u32x2, hi);
        *(vh_u32x2*)(f + plane) = __builtin_bit_cast(vh_u32x2, lo);
      }
    }
    if (bad) stc_u(err, VH_ERR_RANGE);
    return;
  }
  // qkv: a 16-column tile is all queries, keys or values (D is a multiple of 64)
  const int D = N / 3, t0 = *tp;
#pragma unroll
  for (int a = 0; a < TM; ++a) {
    const int m = m0 + 16 * a, bi = m / P, pos = t0 + m - bi * P;
    if (m >= M) continue;
    const bool cached = pos >= 0 && pos < tmax;
    const size_t row = ((size_t)(bi * L + layer) * tmax + pos) * D + 4 * q;
#pragma unroll
    for (int b = 0; b < TN; ++b) {
      const int nt = 16 * (nt0 + b);                               // uniform
      if (nt >= N) continue;
      vh_f32x4 v = value(a, b);
#pragma unroll
      for (int j = 0; j < 4; ++j) v[j] += bn[b][j];
      if (nt < D) {
        *(vh_f32x4*)(out + (size_t)m * ldo + nt + 4 * q) = v;
      } else if (cached) {
        vh_half* c = (nt < 2 * D ? kc + (nt - D) : vc + (nt - 2 * D)) + row;
        *(vh_u32x2*)c = vh_u32x2{f2h(v[0]) | ((unsigned)f2h(v[1]) << 16), f2h(v[2]) | ((unsigned)f2h(v[3]) << 16)};
      }
    }
  }
}

// Ring: two stages of S k-steps of 32 in flight in registers before they go to
// LDS; with WDIR the weight fragments skip LDS and go from the caches straight
// into each wave's registers one stage ahead (the WM waves that share them
// meet in the CU's L1). With ANEW the hi halves' sums start anew with each turn
// of the loop (two stages) and are added in fp32: a fold in one running sum is up
// to 1.7 times further from 64 bits than in parts of 256, which is what few rows
// get from the waves and the blocks that split their folds (pf_pgemm32, 128
// rows, in one sum / anew every 128: 1024 deep 2.10e-7 / 1.08e-7). It costs 0-1%
// (1024 x 2304 x 768 17.9 -> 18.0 us); sums twice as long, behind a condition,
// 2%.
template <int TM, int TN, int WM, int WN, int S, bool WDIR, bool ANEW>
__device__ __forceinline__ void pf_pgemm_ring(
    const vh_u32x4* __restrict__ Af, const vh_u32x4* __restrict__ Wf, int MT, int KT, int NT, int ks,
    const vh_half* __restrict__ bias, int M, int N, int mode, float* __restrict__ out, int ldo,
    vh_half* __restrict__ kc, vh_half* __restrict__ vc, int P, const int* __restrict__ tp, int layer, int L, int tmax,
    float* __restrict__ ws, vh_half* __restrict__ F, unsigned* __restrict__ err) {
  constexpr int NW = WM * WN, BM = TM * WM, BN = TN * WN;
  constexpr int FA = 2 * BM * S, FR = FA + (WDIR ? 0 : BN * S);     // fragments (1 KB) of a stage: A, all
  constexpr int PER = FR / NW;
  static_assert(FR % NW == 0, "whole fragments per wave");
  __shared__ __attribute__((aligned(16))) vh_u32x4 lds[2][FR * 64];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int wm = wave / WN, wn = wave % WN;
  PfTile tl;
  if (!pf_tile<BM, BN>(tl, MT, NT, ks)) return;
  const int part = tl.part, mt0 = tl.mt0, nt0 = tl.nt0;
  const int nst = KT / S, c0 = part * nst / ks, ns = (part + 1) * nst / ks - c0;     // this part's stages
  // tiles past the last one read the last one; their sums are not stored
  const vh_u32x4* src[PER];
#pragma unroll
  for (int i = 0; i < PER; ++i) {
    const int f = wave * PER + i;
    if (f < FA) {
      const int s = f % S, t = (f / S) % BM, p = f / (S * BM);
      src[i] = Af + ((size_t)(p * MT + min(mt0 + t, MT - 1)) * KT + c0 * S + s) * 64 + lane;
    } else {
      const int e = f - FA, s = e % S, t = e / S;
      src[i] = Wf + ((size_t)min(nt0 + t, NT - 1) * KT + c0 * S + s) * 64 + lane;
    }
  }
  vh_f32x4 ah[TM][TN], al[TM][TN], sum[TM][TN];
#pragma unroll
  for (int a = 0; a < TM; ++a)
#pragma unroll
    for (int b = 0; b < TN; ++b) ah[a][b] = al[a][b] = sum[a][b] = vh_f32x4{0.0f, 0.0f, 0.0f, 0.0f};
  vh_u32x4 st[2][PER];
  auto gload = [&](vh_u32x4 (&d)[PER], int c) {
#pragma unroll
    for (int i = 0; i < PER; ++i) d[i] = src[i][(size_t)c * S * 64];
  };
  auto put = [&](const vh_u32x4 (&d)[PER], int buf) {
#pragma unroll
    for (int i = 0; i < PER; ++i) lds[buf][(wave * PER + i) * 64 + lane] = d[i];
  };
  const vh_u32x4* wp[TN];
  vh_u32x4 wd[S][TN];
  gload(st[0], 0);
  if constexpr (WDIR) {
#pragma unroll
    for (int b = 0; b < TN; ++b) {
      wp[b] = Wf + ((size_t)min(nt0 + wn * TN + b, NT - 1) * KT + c0 * S) * 64 + lane;
#pragma unroll
      for (int s = 0; s < S; ++s) wd[s][b] = wp[b][s * 64];
    }
  }
  put(st[0], 0);
#pragma unroll
  for (int u = 1; u <= 2; ++u)
    if (u < ns) gload(st[u % 2], u);
  vh_lds_sync();
  for (int cc = 0; cc < ns; cc += 2) {
    if constexpr (ANEW)
#pragma unroll
      for (int a = 0; a < TM; ++a)
#pragma unroll
        for (int b = 0; b < TN; ++b) ah[a][b] = vh_f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const int c = cc + u;
      if (c >= ns) break;
      const vh_u32x4* sh = lds[u & 1];
#pragma unroll
      for (int s = 0; s < S; ++s) {
        vh_u32x4 w[TN], x[2][TM];
#pragma unroll
        for (int b = 0; b < TN; ++b) {
          if constexpr (WDIR)
            w[b] = wd[s][b];
          else
            w[b] = sh[(FA + (wn * TN + b) * S + s) * 64 + lane];
        }
#pragma unroll
        for (int p = 0; p < 2; ++p)
#pragma unroll
          for (int a = 0; a < TM; ++a) x[p][a] = sh[((p * BM + wm * TM + a) * S + s) * 64 + lane];
#pragma unroll
        for (int a = 0; a < TM; ++a)
#pragma unroll
          for (int b = 0; b < TN; ++b) {
            ah[a][b] = vh_mfma(w[b], x[0][a], ah[a][b]);
            al[a][b] = vh_mfma(w[b], x[1][a], al[a][b]);
          }
        if constexpr (WDIR)
          if (c + 1 < ns)
#pragma unroll
            for (int b = 0; b < TN; ++b) wd[s][b] = wp[b][(size_t)((c + 1) * S + s) * 64];
      }
      if (c + 1 < ns) {       // the buffer written here was last read before the previous barrier
        put(st[u ^ 1], u ^ 1);
        if (c + 3 < ns) gload(st[u ^ 1], c + 3);
      }
      vh_lds_sync();
    }
    if constexpr (ANEW)
#pragma unroll
      for (int a = 0; a < TM; ++a)
#pragma unroll
        for (int b = 0; b < TN; ++b)
          sum[a][b] = vh_f32x4{sum[a][b][0] + ah[a][b][0], sum[a][b][1] + ah[a][b][1], sum[a][b][2] + ah[a][b][2],
                               sum[a][b][3] + ah[a][b][3]};
  }
  pf_pgemm_out<TM, TN>(ANEW ? sum : ah, al, mt0 + wm * TM, nt0 + wn * TN, part, ks, MT, bias, M, N, mode, out, ldo, kc,
                       vc, P, tp, layer, L, tmax, ws, F, err);
}

// Pipe: one k-step a stage; while a stage's products run, the next stage's
// fragments go from LDS into a second register set, the stage after that from
// registers into LDS and the one after from the caches into registers, so no
// wave waits for LDS between its products.
// The block barrier of the loop is in builtins the compiler counts waits by: it
// then knows that the fragments read before it have arrived, and does not
// wait for the next ones at the first product that uses the former.
__device__ __forceinline__ void pf_pipe_sync() {
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_waitcnt(0xc07f);          // lgkmcnt(0): this wave's LDS reads and writes are done
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}
template <int TM, int TN, int WM, int WN>
__device__ __forceinline__ void pf_pgemm_pipe(
    const vh_u32x4* __restrict__ Af, const vh_u32x4* __restrict__ Wf, int MT, int KT, int NT, int ks,
    const vh_half* __restrict__ bias, int M, int N, int mode, float* __restrict__ out, int ldo,
    vh_half* __restrict__ kc, vh_half* __restrict__ vc, int P, const int* __restrict__ tp, int layer, int L, int tmax,
    float* __restrict__ ws, vh_half* __restrict__ F, unsigned* __restrict__ err) {
  constexpr int NW = WM * WN, BM = TM * WM, BN = TN * WN;
  constexpr int FA = 2 * BM, FR = FA + BN;           // fragments (1 KB) of a stage: A, all
  constexpr int PER = FR / NW;
  static_assert(FR % NW == 0 && TM % 2 == 0, "whole fragments per wave");
  __shared__ __attribute__((aligned(16))) vh_u32x4 lds[2][FR * 64];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int wm = wave / WN, wn = wave % WN;
  PfTile tl;
  if (!pf_tile<BM, BN>(tl, MT, NT, ks)) return;
  const int part = tl.part, mt0 = tl.mt0, nt0 = tl.nt0;
  const int c0 = part * KT / ks, ns = (part + 1) * KT / ks - c0;
  const vh_u32x4* src[PER];
#pragma unroll
  for (int i = 0; i < PER; ++i) {
    const int f = wave * PER + i;
    if (f < FA) {
      const int t = f % BM, p = f / BM;
      src[i] = Af + ((size_t)(p * MT + min(mt0 + t, MT - 1)) * KT + c0) * 64 + lane;
    } else {
      src[i] = Wf + ((size_t)min(nt0 + f - FA, NT - 1) * KT + c0) * 64 + lane;
    }
  }
  vh_f32x4 ah[TM][TN], al[TM][TN];
#pragma unroll
  for (int a = 0; a < TM; ++a)
#pragma unroll
    for (int b = 0; b < TN; ++b) ah[a][b] = al[a][b] = vh_f32x4{0.0f, 0.0f, 0.0f, 0.0f};
  vh_u32x4 st[PER], w[2][TN], x[2][2][TM];
  auto gload = [&](int c) {
#pragma unroll
    for (int i = 0; i < PER; ++i) st[i] = src[i][(size_t)c * 64];
  };
  auto put = [&](int buf) {
#pragma unroll
    for (int i = 0; i < PER; ++i) lds[buf][(wave * PER + i) * 64 + lane] = st[i];
  };
  auto frags = [&](vh_u32x4 (&wf)[TN], vh_u32x4 (&xf)[2][TM], int buf) {
#pragma unroll
    for (int b = 0; b < TN; ++b) wf[b] = lds[buf][(FA + wn * TN + b) * 64 + lane];
#pragma unroll
    for (int a = 0; a < TM; ++a)
#pragma unroll
      for (int p = 0; p < 2; ++p) xf[p][a] = lds[buf][(p * BM + wm * TM + a) * 64 + lane];
  };
  auto mma = [&](const vh_u32x4 (&wf)[TN], const vh_u32x4 (&xf)[2][TM], int a0, int a1) {
#pragma unroll
    for (int a = 0; a < TM; ++a) {
      if (a < a0 || a >= a1) continue;
#pragma unroll
      for (int b = 0; b < TN; ++b) {
        ah[a][b] = vh_mfma(wf[b], xf[0][a], ah[a][b]);
        al[a][b] = vh_mfma(wf[b], xf[1][a], al[a][b]);
      }
    }
  };
  gload(0);
  put(0);
  if (1 < ns) gload(1);
  pf_pipe_sync();
  frags(w[0], x[0], 0);
  if (1 < ns) put(1);
  if (2 < ns) gload(2);
  pf_pipe_sync();
  for (int cc = 0; cc < ns; cc += 2) {
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const int c = cc + u;
      if (c >= ns) break;
      if (c + 1 < ns) frags(w[u ^ 1], x[u ^ 1], u ^ 1);
      __builtin_amdgcn_sched_barrier(0);
      mma(w[u], x[u], 0, TM / 2);
      __builtin_amdgcn_sched_barrier(0);
      if (c + 2 < ns) {       // buffer u: its last reads were before the previous barrier
        put(u);
        if (c + 3 < ns) gload(c + 3);
      }
      __builtin_amdgcn_sched_barrier(0);
      mma(w[u], x[u], TM / 2, TM);
      __builtin_amdgcn_sched_barrier(0);
      pf_pipe_sync();
    }
  }
  pf_pgemm_out<TM, TN>(ah, al, mt0 + wm * TM, nt0 + wn * TN, part, ks, MT, bias, M, N, mode, out, ldo, kc, vc, P, tp,
                       layer, L, tmax, ws, F, err);
}

#define PF_PGEMM(name, threads, waves, ...)                                                                         \
  extern "C" __global__ __launch_bounds__(threads, waves) void name(                                                \
      const vh_u32x4* __restrict__ Af, const vh_u32x4* __restrict__ Wf, int MT, int KT, int NT, int ks,             \
      const vh_half* __restrict__ bias, int M, int N, int mode, float* __restrict__ out, int ldo,                   \
      vh_half* __restrict__ kc, vh_half* __restrict__ vc, int P, const int* __restrict__ tp, int layer, int L,      \
      int tmax, float* __restrict__ ws, vh_half* __restrict__ F, unsigned* __restrict__ err) {                      \
    __VA_ARGS__(Af, Wf, MT, KT, NT, ks, bias, M, N, mode, out, ldo, kc, vc, P, tp, layer, L, tmax, ws, F, err);     \
  }
PF_PGEMM(pf_pgemm128, 512, 2, pf_pgemm_pipe<4, 4, 2, 4>)              // 128 x 256
PF_PGEMM(pf_pgemm64, 512, 4, pf_pgemm_pipe<2, 2, 2, 4>)               // 64 x 128, eight waves
PF_PGEMM(pf_pgemm64w, 256, 2, pf_pgemm_ring<2, 4, 2, 2, 1, true, false>)  // 64 x 128, four waves
PF_PGEMM(pf_pgemm32, 256, 2, pf_pgemm_ring<1, 2, 2, 2, 2, false, true>)   // 32 x 64
PF_PGEMM(pf_pgemm32o, 256, 2, pf_pgemm_ring<1, 2, 2, 2, 2, false, false>) // 32 x 64, one sum a part

// The parts of a split product added in part order, then the epilogue. One
// thread per output value.
extern "C" __global__ __launch_bounds__(256) void pf_reduce(
    const float* __restrict__ ws, int ksplit, const vh_half* __restrict__ bias, int M, int N, int mode,
    float* __restrict__ out, int ldo, vh_half* __restrict__ kc, vh_half* __restrict__ vc, int P,
    const int* __restrict__ tp, int layer, int L, int tmax) {
  const size_t e = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= (size_t)M * N) return;
  const int m = (int)(e / N), n = (int)(e % N);
  float c = ws[e];
  for (int k = 1; k < ksplit; ++k) c += ws[(size_t)k * M * N + e];
  pf_epi(mode, m, n, c, bias, N, out, ldo, kc, vc, P, tp, layer, L, tmax);
}

// ---------------------------------------------------------------- layer norm
// F[i] = (X[r] - mean) / sqrt(var + 1e-5) * w + b for r = row0 + i * rstride
// (biased variance; mean and variance as sums of x / D and (x - mean)^2 / D,
// as gpt2.vst Q2 writes them): one block per output row, D <= 8 * 256,
// thread t holding the row's eight consecutive values 8t .. 8t + 7 (16-byte
// loads, so a wave's load is a whole kilobyte of the row), summed per thread,
// then over the block. The row goes to F in fragment order (MT m-tiles: the
// thread writes its own piece). (Thread t on values
// t, t + 256, .., one 4-byte load each, measured slower: XL B=64 decode 4.06
// against 3.41 ms per step with the reduction below written that way.)
__device__ __forceinline__ void pf_ld8f(const float* p, float* v) {
  const vh_f32x4 a = *(const vh_f32x4*)p, b = *(const vh_f32x4*)(p + 4);
  v[0] = a[0]; v[1] = a[1]; v[2] = a[2]; v[3] = a[3]; v[4] = b[0]; v[5] = b[1]; v[6] = b[2]; v[7] = b[3];
}
__device__ __forceinline__ void pf_norm8_out(const float* v, const float* wv, const float* bv, bool in, int D, int i,
                                             vh_half* __restrict__ F, int MT, unsigned* __restrict__ err,
                                             float* red) {
  const float fd = (float)D;
  float s = 0.0f;
  if (in)
#pragma unroll
    for (int j = 0; j < 8; ++j) s += v[j] / fd;
  const float mean = block_red_sum(s, red);
  float q = 0.0f;
  if (in)
#pragma unroll
    for (int j = 0; j < 8; ++j) q += (v[j] - mean) * (v[j] - mean) / fd;
  vh_lds_sync();
  const float sd = sqrtf(block_red_sum(q, red) + 0.00001f);
  if (!in) return;
  float y[8];
#pragma unroll
  for (int j = 0; j < 8; ++j) y[j] = (v[j] - mean) / sd * wv[j] + bv[j];
  bool bad = false;
  pf_frag_put8(F, MT, D / 32, i, 8 * threadIdx.x, y, bad);
  if (bad) stc_u(err, VH_ERR_RANGE);
}

extern "C" __global__ __launch_bounds__(256) void pf_ln(const float* __restrict__ X, int row0, int rstride,
                                                         const vh_half* __restrict__ w, const vh_half* __restrict__ b,
                                                         int D, vh_half* __restrict__ F, int MT,
                                                         unsigned* __restrict__ err) {
  __shared__ float red[VNWAVE];
  const int k8 = 8 * threadIdx.x;
  const bool in = k8 < D;
  float v[8] = {}, wv[8] = {}, bv[8] = {};
  if (in) {
    pf_ld8f(X + (size_t)(row0 + (size_t)blockIdx.x * rstride) * D + k8, v);
    unpack8(ld16(w + k8), wv);
    unpack8(ld16(b + k8), bv);
  }
  pf_norm8_out(v, wv, bv, in, D, blockIdx.x, F, MT, err, red);
}

// The embedding Z[m] = wte[tok[m]] + wpe[t0 + p] (gpt2.vst Q1; ids and
// positions clamped into their tables) and the first layer's LayerNorm of it
// (pf_ln) in one launch: one block per row, the row kept in registers between
// the two.
extern "C" __global__ __launch_bounds__(256) void pf_embed_ln(const int* __restrict__ tok, int P,
                                                               const int* __restrict__ tp,
                                                               const vh_half* __restrict__ wte,
                                                               const vh_half* __restrict__ wpe, float* __restrict__ Z,
                                                               int D, int V, int npos, const vh_half* __restrict__ w,
                                                               const vh_half* __restrict__ b, vh_half* __restrict__ F,
                                                               int MT, unsigned* __restrict__ err) {
  __shared__ float red[VNWAVE];
  const int m = blockIdx.x, k8 = 8 * threadIdx.x;
  const bool in = k8 < D;
  int x = tok[m];
  x = x < 0 ? 0 : (x >= V ? V - 1 : x);
  int pos = *tp + (P == 1 ? 0 : m % P);
  pos = pos < 0 ? 0 : (pos >= npos ? npos - 1 : pos);
  float v[8] = {}, wv[8] = {}, bv[8] = {};
  if (in) {
    float a[8], c[8];
    unpack8(ld16(wte + (size_t)x * D + k8), a);
    unpack8(ld16(wpe + (size_t)pos * D + k8), c);
    unpack8(ld16(w + k8), wv);
    unpack8(ld16(b + k8), bv);
#pragma unroll
    for (int j = 0; j < 8; ++j) v[j] = a[j] + c[j];
    float* z = Z + (size_t)m * D + k8;
    *(vh_f32x4*)z = vh_f32x4{v[0], v[1], v[2], v[3]};
    *(vh_f32x4*)(z + 4) = vh_f32x4{v[4], v[5], v[6], v[7]};
  }
  pf_norm8_out(v, wv, bv, in, D, m, F, MT, err, red);
}

// A split residual product's parts added in part order (pf_reduce, mode 1:
// Z[m, n] = (Z[m, n] + C) + bias[n]) and the LayerNorm that reads Z next (as
// pf_ln), in one launch: one block per row, the row kept in
// registers between the two.
extern "C" __global__ __launch_bounds__(256) void pf_reduce_ln(
    const float* __restrict__ ws, int ksplit, const vh_half* __restrict__ bias, int M, int D,
    float* __restrict__ Z, const vh_half* __restrict__ w, const vh_half* __restrict__ b, vh_half* __restrict__ F,
    int MT, unsigned* __restrict__ err) {
  __shared__ float red[VNWAVE];
  const int m = blockIdx.x, k8 = 8 * threadIdx.x;
  const bool in = k8 < D;
  float v[8] = {}, zr[8] = {}, bn[8] = {}, wv[8] = {}, bv[8] = {};
  if (in) {
    pf_ld8f(ws + (size_t)m * D + k8, v);
    pf_ld8f(Z + (size_t)m * D + k8, zr);
    if (bias) unpack8(ld16(bias + k8), bn);
    unpack8(ld16(w + k8), wv);
    unpack8(ld16(b + k8), bv);
    for (int k0 = 1; k0 < ksplit; k0 += 4) {      // four parts' loads in flight, added in part order
      float p[4][8];
#pragma unroll
      for (int u = 0; u < 4; ++u)
        if (k0 + u < ksplit) pf_ld8f(ws + ((size_t)(k0 + u) * M + m) * D + k8, p[u]);
#pragma unroll
      for (int u = 0; u < 4; ++u)
        if (k0 + u < ksplit)
#pragma unroll
          for (int j = 0; j < 8; ++j) v[j] += p[u][j];
    }
#pragma unroll
    for (int j = 0; j < 8; ++j) v[j] = (zr[j] + v[j]) + bn[j];
    float* zp = Z + (size_t)m * D + k8;
    *(vh_f32x4*)zp = vh_f32x4{v[0], v[1], v[2], v[3]};
    *(vh_f32x4*)(zp + 4) = vh_f32x4{v[4], v[5], v[6], v[7]};
  }
  pf_norm8_out(v, wv, bv, in, D, m, F, MT, err, red);
}

// pf_ln of rows 0 .. M - 1 for many rows: a block per 16 rows, lane 16 q + r of
// wave w holding row r's values 8 (16 i + 4 w + q) .. + 7, i < NP (D <= 128 NP),
// so that a wave stores a whole fragment, one contiguous kilobyte, where a
// block per row stores 16 bytes of each 256 and eight XCDs write each line.
// Sums pairwise over a lane's eight values (pf_sum8), then over its pieces;
// divided by D there, where a rounding is a sixteenth of one of the whole mean;
// then over the lanes of a row and pairwise over the waves: 0.77-1.01 times
// pf_ln's distance from 64 bits at a mean of 30 deviations (one running sum
// divided at the end 1.5), 0.99-1.01 at none. pf_sum8 scales its terms by 2^-11
// (D <= 2048), where pf_ln divides each by D: exact, and a row overflows here if
// it does there (a variance beyond fp32 leaves the biases in both).
// Bound by the bytes where there are blocks enough: 24576 rows of 768 65.8 ->
// 25.6 us (5.9 TB/s), 8192 of 1600 46.6 -> 20.8; 2048 of 768 8.7 -> 7.7; at 999
// rows 6.3 against 7.3 and below, the block per row is faster.
__device__ __forceinline__ float pf_sum8(const float* v) {         // their sum, times 2^-11
  constexpr float c = 1.0f / 2048.0f;
  return (fmaf(v[0], c, v[1] * c) + fmaf(v[2], c, v[3] * c)) + (fmaf(v[4], c, v[5] * c) + fmaf(v[6], c, v[7] * c));
}
template <int NP>
__device__ __forceinline__ void pf_lnm_body(const float* __restrict__ X, int M, int D, const vh_half* __restrict__ w,
                                            const vh_half* __restrict__ b, vh_half* __restrict__ F, int MT,
                                            unsigned* __restrict__ err) {
  __shared__ float red[2][VNWAVE][16];
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, r = lane & 15;
  const int m = 16 * blockIdx.x + r, pc0 = 4 * wave + (lane >> 4), np = D / 8;
  const bool live = m < M;
  const float* x = X + (size_t)(live ? m : M - 1) * D;
  float v[NP][8];
#pragma unroll
  for (int i = 0; i < NP; ++i)
    if (pc0 + 16 * i < np) pf_ld8f(x + 8 * (pc0 + 16 * i), v[i]);
  float s = 0.0f;
#pragma unroll
  for (int i = 0; i < NP; ++i)
    if (pc0 + 16 * i < np) s += pf_sum8(v[i]);
  const float d2 = (float)D / 2048.0f;
  auto row_sum = [&](float p, float (*part)[16]) {                 // the lanes' sums p over the row, / D
    p /= d2;
    p += __shfl_xor(p, 16, 64);
    p += __shfl_xor(p, 32, 64);
    if (lane < 16) part[wave][r] = p;
    vh_lds_sync();
    static_assert(VNWAVE == 4, "pairwise over the waves");
    return (part[0][r] + part[1][r]) + (part[2][r] + part[3][r]);
  };
  const float mean = row_sum(s, red[0]);
  s = 0.0f;
#pragma unroll
  for (int i = 0; i < NP; ++i)
    if (pc0 + 16 * i < np) {
      float u[8];
#pragma unroll
      for (int j = 0; j < 8; ++j) u[j] = (v[i][j] - mean) * (v[i][j] - mean);
      s += pf_sum8(u);
    }
  float sd = sqrtf(row_sum(s, red[1]) + 0.00001f), rs = 1.0f / sd;
  if (!live) return;
  if (sd == INFINITY) sd = 1.0f, rs = 0.0f;                        // x / inf by vh_divr's two products
  bool bad = false;
#pragma unroll
  for (int i = 0; i < NP; ++i) {
    const int k8 = 8 * (pc0 + 16 * i);
    if (k8 >= D) continue;
    float y[8], wv[8], bv[8];
    unpack8(ld16(w + k8), wv);
    unpack8(ld16(b + k8), bv);
#pragma unroll
    for (int j = 0; j < 8; ++j) y[j] = vh_divr(v[i][j] - mean, sd, rs) * wv[j] + bv[j];
    pf_frag_put8(F, MT, D / 32, m, k8, y, bad);
  }
  if (bad) stc_u(err, VH_ERR_RANGE);
}
#define PF_LNM(name, NP)                                                                                            \
  extern "C" __global__ __launch_bounds__(256, 2) void name(const float* __restrict__ X, int M, int D,              \
                                                            const vh_half* __restrict__ w,                          \
                                                            const vh_half* __restrict__ b, vh_half* __restrict__ F, \
                                                            int MT, unsigned* __restrict__ err) {                   \
    pf_lnm_body<NP>(X, M, D, w, b, F, MT, err);                                                                     \
  }
PF_LNM(pf_lnm8, 8)
PF_LNM(pf_lnm16, 16)

// ---------------------------------------------------------------- products of few rows
// C = A W over K for M <= 16 MT rows, both operands in fragment order (above):
// the weights streamed from memory straight into the matrix cores' registers,
// the activations read as they are (hi and lo planes, each multiplied into
// its own accumulator and combined at the end). A block is PF_MW waves on the
// same MN n-tiles of 16 columns, MN = 1 up to 32 rows and 2 at 64 rows (with
// MN = 2 throughout, same box: GPT-2 small at 32 rows 0.585 -> 0.601 ms per
// step, medium at 16 rows 0.969 -> 1.058, XL at 64 rows even; with MN = 1 at
// 64 rows XL 3.02 -> 3.79, the activation rows re-read by twice the blocks);
// block vb takes n-tiles MN (vb / ks) .. + MN and fold part vb % ks of ks,
// and its waves split that part's k-steps into PF_MW consecutive runs. A
// wave with at most PF_WFIRST k-steps issues all its
// weight fragments at once, then the activation fragments one k-step ahead
// of the one it multiplies (XL B=64 decode 3.35 -> 3.10 ms per step against
// both one k-step ahead; activations two ahead 3.15); a longer run keeps the
// next k-step's weights and activations in flight. The waves' partial tiles
// are added in LDS in wave order. Then either the part is stored (ks > 1:
// ws[part][m][n], added by pf_reduce / pf_reduce_ln / pf_reduce_frag), or the
// epilogue of `mode` is applied: 1 and 3 as pf_epi;
// 2 (GELU) writes the result in fragment order into F, as the activation of
// the next product (N / 32 k-steps).
#define PF_MW 8
#define PF_WFIRST 8     // k-steps of a wave up to which all its weight fragments are loaded first

// pf_epi for eight consecutive columns n .. n + 7 of row m (at sequence
// position pos), modes 1 (residual) and 3 (qkv: queries, or eight values of a key /
// value cache row as one 16-byte store); the same arithmetic per value.
__device__ __forceinline__ void pf_epi8(int mode, int m, int n, float* v, const float* bn, const float* z, int pos,
                                        int N, float* __restrict__ out, int ldo, vh_half* __restrict__ kc,
                                        vh_half* __restrict__ vc, int P, int layer, int L, int tmax) {
  if (mode == 1) {
    float* o = out + (size_t)m * ldo + n;
#pragma unroll
    for (int j = 0; j < 8; ++j) v[j] = (z[j] + v[j]) + bn[j];
    *(vh_f32x4*)o = vh_f32x4{v[0], v[1], v[2], v[3]};
    *(vh_f32x4*)(o + 4) = vh_f32x4{v[4], v[5], v[6], v[7]};
    return;
  }
#pragma unroll
  for (int j = 0; j < 8; ++j) v[j] = v[j] + bn[j];
  const int D = N / 3;
  if (n < D) {
    float* o = out + (size_t)m * ldo + n;
    *(vh_f32x4*)o = vh_f32x4{v[0], v[1], v[2], v[3]};
    *(vh_f32x4*)(o + 4) = vh_f32x4{v[4], v[5], v[6], v[7]};
    return;
  }
  if (pos < 0 || pos >= tmax) return;
  unsigned short h[8];
#pragma unroll
  for (int j = 0; j < 8; ++j) h[j] = f2h(v[j]);
  const size_t at = ((size_t)((P == 1 ? m : m / P) * L + layer) * tmax + pos) * D + (n % D);
  *(vh_u32x4*)((n < 2 * D ? kc : vc) + at) =
      vh_u32x4{h[0] | ((unsigned)h[1] << 16), h[2] | ((unsigned)h[3] << 16), h[4] | ((unsigned)h[5] << 16),
               h[6] | ((unsigned)h[7] << 16)};
}
template <int MT, int MN, bool WNT>
__device__ __forceinline__ void pf_mgemm_body(
    int vb, const vh_u32x4* __restrict__ Af, const vh_u32x4* __restrict__ Wf, int KT, int NT, int ks,
    const vh_half* __restrict__ bias, int M, int N, int mode, float* __restrict__ out, int ldo,
    vh_half* __restrict__ kc, vh_half* __restrict__ vc, int P, const int* __restrict__ tp, int layer, int L, int tmax,
    float* __restrict__ ws, vh_half* __restrict__ F, unsigned* __restrict__ err) {
  __shared__ __attribute__((aligned(16))) vh_f32x4 red[PF_MW][MN * MT * 64];
  __shared__ __attribute__((aligned(16))) float tile[16 * MT][16 * MN + 4];
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int part = vb % ks, nt0 = (vb / ks) * MN;
  const int ka = part * KT / ks, kb = (part + 1) * KT / ks;
  const int k0 = ka + (kb - ka) * wave / PF_MW, k1 = ka + (kb - ka) * (wave + 1) / PF_MW;
  vh_f32x4 acc[MN][MT], acl[MN][MT];
#pragma unroll
  for (int t = 0; t < MN; ++t)
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) acc[t][mt] = acl[t][mt] = vh_f32x4{0.0f, 0.0f, 0.0f, 0.0f};
  const size_t plane = (size_t)MT * KT * 64;
  // the epilogue's operands of this thread's item (a thread has at most one:
  // 16 MT x 2 MN <= PF_MW x 64), loaded before the products so that their
  // latency is not added at the end: the bias, the residual row piece, the
  // sequence position of the cache rows
  const int ei = threadIdx.x, em = ei / (2 * MN), ec8 = 8 * (ei % (2 * MN)), en = 16 * nt0 + ec8;
  const bool eok = ks == 1 && ei < 16 * MT * 2 * MN && em < M && en < N;
  float eb[8] = {}, ez[8] = {};
  int epos = 0;
  // the GELU product adds the bias and applies GELU where the waves' sums are
  // added (every thread has at most one item there: MN MT 64 <= PF_MW 64),
  // so that all threads share that work; this thread's item's column bias:
  const bool gelu_red = ks == 1 && mode == 2;
  const int rn = 16 * (nt0 + (threadIdx.x >> 6) / MT) + (threadIdx.x & 15);
  const float rb = gelu_red && bias != nullptr && threadIdx.x < MN * MT * 64 && rn < N ? h2f(bias[rn]) : 0.0f;
  if (eok) {
    if (bias && mode != 2) unpack8(ld16(bias + en), eb);
    if (mode == 1) pf_ld8f(out + (size_t)em * ldo + en, ez);
    if (mode == 3) epos = *tp + (P == 1 ? 0 : em % P);
  }
  // weight fragments: nontemporal (WNT) where the model's weights cannot stay
  // in the memory-side cache between steps (the host picks the kernel)
  auto wld = [&](size_t i) {
    if constexpr (WNT)
      return __builtin_nontemporal_load(Wf + i);
    else
      return Wf[i];
  };
  vh_u32x4 wa[MN], aa[2][MT], wb[MN], ab[2][MT];
  auto load = [&](vh_u32x4 (&w)[MN], vh_u32x4 (&a)[2][MT], int k) {
    const bool in = k < k1;
#pragma unroll
    for (int t = 0; t < MN; ++t)
      w[t] = in && nt0 + t < NT ? wld(((size_t)(nt0 + t) * KT + k) * 64 + lane) : vh_u32x4{0u, 0u, 0u, 0u};
#pragma unroll
    for (int p = 0; p < 2; ++p)
#pragma unroll
      for (int mt = 0; mt < MT; ++mt)
        a[p][mt] = in ? Af[p * plane + ((size_t)mt * KT + k) * 64 + lane] : vh_u32x4{0u, 0u, 0u, 0u};
  };
  auto mma = [&](const vh_u32x4 (&w)[MN], const vh_u32x4 (&a)[2][MT]) {
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
      for (int t = 0; t < MN; ++t) {
        acc[t][mt] = vh_mfma(a[0][mt], w[t], acc[t][mt]);
        acl[t][mt] = vh_mfma(a[1][mt], w[t], acl[t][mt]);
      }
  };
  // up to 8 rows: the hi halves of rows 0-7 and the lo halves in one operand
  // tile (its rows 0-7 and 8-15), so one product and one activation fragment a
  // k-step; all of a wave's loads are issued at once, the activations (from L2)
  // before the weights, which the products then wait for one by one (XL at one
  // row: 7.9 -> 6.9 us a product, 2.08 -> 1.90 ms per step)
  const bool packed = MT == 1 && M <= 8;
  if (packed) {
    const vh_u32x4* Ap = Af + ((lane & 8) ? plane : 0) + (lane & 0x37);
    for (int kb8 = k0; kb8 < k1; kb8 += PF_WFIRST) {
      vh_u32x4 a8[PF_WFIRST], w8[PF_WFIRST][MN];
#pragma unroll
      for (int j = 0; j < PF_WFIRST; ++j) a8[j] = kb8 + j < k1 ? Ap[(size_t)(kb8 + j) * 64] : vh_u32x4{0u, 0u, 0u, 0u};
#pragma unroll
      for (int j = 0; j < PF_WFIRST; ++j)
#pragma unroll
        for (int t = 0; t < MN; ++t)
          w8[j][t] = kb8 + j < k1 && nt0 + t < NT ? wld(((size_t)(nt0 + t) * KT + kb8 + j) * 64 + lane)
                                                  : vh_u32x4{0u, 0u, 0u, 0u};
#pragma unroll
      for (int j = 0; j < PF_WFIRST; ++j)
        if (kb8 + j < k1)
#pragma unroll
          for (int t = 0; t < MN; ++t) acc[t][0] = vh_mfma(a8[j], w8[j][t], acc[t][0]);
    }
#pragma unroll
    for (int t = 0; t < MN; ++t)
#pragma unroll
      for (int v = 0; v < 4; ++v) acl[t][0][v] = __shfl_xor(acc[t][0][v], 32, 64);     // rows 8 .. 15: the lo sums
  } else if (k1 - k0 <= PF_WFIRST) {
    // all of the wave's weight fragments first (so they are in flight at once),
    // then the activation fragments one k-step ahead
    vh_u32x4 wall[PF_WFIRST][MN];
#pragma unroll
    for (int j = 0; j < PF_WFIRST; ++j)
#pragma unroll
      for (int t = 0; t < MN; ++t)
        wall[j][t] = k0 + j < k1 && nt0 + t < NT ? wld(((size_t)(nt0 + t) * KT + k0 + j) * 64 + lane)
                                                 : vh_u32x4{0u, 0u, 0u, 0u};
    auto loada = [&](vh_u32x4 (&a)[2][MT], int k) {
      const bool in = k < k1;
#pragma unroll
      for (int p = 0; p < 2; ++p)
#pragma unroll
        for (int mt = 0; mt < MT; ++mt)
          a[p][mt] = in ? Af[p * plane + ((size_t)mt * KT + k) * 64 + lane] : vh_u32x4{0u, 0u, 0u, 0u};
    };
    loada(aa, k0);
#pragma unroll
    for (int j = 0; j < PF_WFIRST; j += 2) {
      if (k0 + j < k1) {
        loada(ab, k0 + j + 1);
        mma(wall[j], aa);
      }
      if (k0 + j + 1 < k1) {
        loada(aa, k0 + j + 2);
        mma(wall[j + 1], ab);
      }
    }
  } else {
    load(wa, aa, k0);
    for (int k = k0; k < k1; k += 2) {
      load(wb, ab, k + 1);
      mma(wa, aa);
      if (k + 1 >= k1) break;
      load(wa, aa, k + 2);
      mma(wb, ab);
    }
  }
#pragma unroll
  for (int t = 0; t < MN; ++t)
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) {
      const vh_f32x4 h = acc[t][mt], l = acl[t][mt];
      red[wave][(t * MT + mt) * 64 + lane] =
          vh_f32x4{vh_hilo(h[0], l[0]), vh_hilo(h[1], l[1]), vh_hilo(h[2], l[2]), vh_hilo(h[3], l[3])};
    }
  __syncthreads();
  for (int i = threadIdx.x; i < MN * MT * 64; i += PF_MW * 64) {
    vh_f32x4 s = red[0][i];
#pragma unroll
    for (int w = 1; w < PF_MW; ++w) {
      const vh_f32x4 o = red[w][i];
      s = vh_f32x4{s[0] + o[0], s[1] + o[1], s[2] + o[2], s[3] + o[3]};
    }
    const int l = i & 63, tm = i >> 6, mt = tm % MT, t = tm / MT;
    if (gelu_red)
#pragma unroll
      for (int v = 0; v < 4; ++v) s[v] = pf_gelu(s[v] + rb);
#pragma unroll
    for (int v = 0; v < 4; ++v) tile[16 * mt + 4 * (l >> 4) + v][16 * t + (l & 15)] = s[v];
  }
  __syncthreads();
  const int n0 = 16 * nt0;
  if (ks == 1 && mode == 2) {
    bool bad = false;
    for (int e = threadIdx.x; e < 16 * MT * 2 * MN; e += PF_MW * 64) {
      const int m = e / (2 * MN), c8 = 8 * (e % (2 * MN));
      if (m >= M || n0 + c8 >= N) continue;
      float v[8];
#pragma unroll
      for (int j = 0; j < 8; ++j) v[j] = tile[m][c8 + j];     // bias and GELU applied above
      pf_frag_put8(F, MT, N / 32, m, n0 + c8, v, bad);
    }
    if (bad) stc_u(err, VH_ERR_RANGE);
    return;
  }
  for (int e = threadIdx.x; e < 16 * MT * 2 * MN; e += PF_MW * 64) {   // eight consecutive columns per thread, 16-byte stores
    const int m = e / (2 * MN), c8 = 8 * (e % (2 * MN)), n = n0 + c8;
    if (m >= M || n >= N) continue;
    float v[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) v[j] = tile[m][c8 + j];
    if (ks > 1) {
      float* p = ws + ((size_t)part * M + m) * N + n;
      *(vh_f32x4*)p = vh_f32x4{v[0], v[1], v[2], v[3]};
      *(vh_f32x4*)(p + 4) = vh_f32x4{v[4], v[5], v[6], v[7]};
    } else {
      pf_epi8(mode, m, n, v, eb, ez, epos, N, out, ldo, kc, vc, P, layer, L, tmax);     // (e is this thread's item)
    }
  }
}

#define PF_MGEMM(name, MT, MN, WNT)                                                                                     \
  extern "C" __global__ __launch_bounds__(PF_MW * 64) void name(                                                  \
      const vh_u32x4* __restrict__ Af, const vh_u32x4* __restrict__ Wf, int KT, int NT, int ks,                    \
      const vh_half* __restrict__ bias, int M, int N, int mode, float* __restrict__ out, int ldo,                 \
      vh_half* __restrict__ kc, vh_half* __restrict__ vc, int P, const int* __restrict__ tp, int layer, int L,      \
      int tmax, float* __restrict__ ws, vh_half* __restrict__ F, unsigned* __restrict__ err) {                              \
    pf_mgemm_body<MT, MN, WNT>(blockIdx.x, Af, Wf, KT, NT, ks, bias, M, N, mode, out, ldo, kc, vc, P, tp, layer, L, \
                               tmax, ws, F, err);                                                                 \
  }
PF_MGEMM(pf_mgemm1, 1, 1, false)
PF_MGEMM(pf_mgemm2, 2, 1, false)
PF_MGEMM(pf_mgemm4, 4, 2, false)
PF_MGEMM(pf_mgemm1n, 1, 1, true)
PF_MGEMM(pf_mgemm2n, 2, 1, true)
PF_MGEMM(pf_mgemm4n, 4, 2, true)

// The output head (a plain product with many columns: out[m, n] = C, no
// bias): block b's wave w makes n-tiles 2 (PF_MW b + w) and the next one
// over the whole fold, weights and activations one k-step ahead. The block's
// waves read the same activation fragments at about the same time, so they
// come from the CU's L1 after the first wave: the activations cross from L2
// once per block, not once per pair of n-tiles as in pf_mgemm*. The sums go
// straight from the accumulators to out (lane l: rows 4 (l / 16) .. +4 of
// column l % 16).
template <int MT>
__device__ __forceinline__ void pf_mhead_body(const vh_u32x4* __restrict__ Af, const vh_u32x4* __restrict__ Wf, int KT,
                                              int NT, int M, int N, float* __restrict__ out, int ldo) {
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int nt0 = 2 * (PF_MW * (int)blockIdx.x + wave);
  if (nt0 >= NT) return;
  vh_f32x4 acc[2][MT], acl[2][MT];
#pragma unroll
  for (int t = 0; t < 2; ++t)
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) acc[t][mt] = acl[t][mt] = vh_f32x4{0.0f, 0.0f, 0.0f, 0.0f};
  const size_t plane = (size_t)MT * KT * 64;
  vh_u32x4 wa[2], aa[2][MT], wb[2], ab[2][MT];
  auto load = [&](vh_u32x4 (&w)[2], vh_u32x4 (&a)[2][MT], int k) {
    const bool in = k < KT;
#pragma unroll
    for (int t = 0; t < 2; ++t)
      w[t] = in && nt0 + t < NT ? Wf[((size_t)(nt0 + t) * KT + k) * 64 + lane] : vh_u32x4{0u, 0u, 0u, 0u};
#pragma unroll
    for (int p = 0; p < 2; ++p)
#pragma unroll
      for (int mt = 0; mt < MT; ++mt)
        a[p][mt] = in ? Af[p * plane + ((size_t)mt * KT + k) * 64 + lane] : vh_u32x4{0u, 0u, 0u, 0u};
  };
  auto mma = [&](const vh_u32x4 (&w)[2], const vh_u32x4 (&a)[2][MT]) {
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
      for (int t = 0; t < 2; ++t) {
        acc[t][mt] = vh_mfma(a[0][mt], w[t], acc[t][mt]);
        acl[t][mt] = vh_mfma(a[1][mt], w[t], acl[t][mt]);
      }
  };
  load(wa, aa, 0);
  for (int k = 0; k < KT; k += 2) {
    load(wb, ab, k + 1);
    mma(wa, aa);
    if (k + 1 >= KT) break;
    load(wa, aa, k + 2);
    mma(wb, ab);
  }
#pragma unroll
  for (int t = 0; t < 2; ++t) {
    const int n = 16 * (nt0 + t) + (lane & 15);
    if (nt0 + t >= NT || n >= N) continue;
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const int m = 16 * mt + 4 * (lane >> 4) + v;
        if (m < M) out[(size_t)m * ldo + n] = vh_hilo(acc[t][mt][v], acl[t][mt][v]);
      }
  }
}
#define PF_MHEAD(name, MT)                                                                                         \
  extern "C" __global__ __launch_bounds__(PF_MW * 64) void name(const vh_u32x4* __restrict__ Af,                 \
                                                                const vh_u32x4* __restrict__ Wf, int KT, int NT,  \
                                                                int M, int N, float* __restrict__ out, int ldo) {  \
    pf_mhead_body<MT>(Af, Wf, KT, NT, M, N, out, ldo);                                                           \
  }
PF_MHEAD(pf_mhead1, 1)
PF_MHEAD(pf_mhead2, 2)
PF_MHEAD(pf_mhead4, 4)

// The parts of a split GELU product (ws[part][m][n], part order) with the
// bias and GELU, written in fragment order into F like pf_mgemm's mode 2: one
// thread per eight consecutive columns of a row.
extern "C" __global__ __launch_bounds__(256) void pf_reduce_frag(const float* __restrict__ ws, int ksplit,
                                                                  const vh_half* __restrict__ bias, int M, int N,
                                                                  vh_half* __restrict__ F, int MT,
                                                                  unsigned* __restrict__ err) {
  const int e = blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= M * (N / 8)) return;
  const int m = e / (N / 8), n8 = 8 * (e % (N / 8));
  float v[8];
  const float* p = ws + (size_t)m * N + n8;
  pf_ld8f(p, v);
  for (int k = 1; k < ksplit; ++k) {
    float q[8];
    pf_ld8f(p + (size_t)k * M * N, q);
#pragma unroll
    for (int j = 0; j < 8; ++j) v[j] += q[j];
  }
#pragma unroll
  for (int j = 0; j < 8; ++j) v[j] = pf_gelu(v[j] + h2f(bias[n8 + j]));
  bool bad = false;
  pf_frag_put8(F, MT, N / 32, m, n8, v, bad);
  if (bad) stc_u(err, VH_ERR_RANGE);
}

// ---------------------------------------------------------------- attention
// Prefill attention on the matrix cores: a block of four waves makes 64 queries
// of one (batch row, head), 16 to a wave, over the cache positions up to its
// last query's in tiles of 64, with a running maximum, sum and weighted
// values (gpt2.vst Q5-Q7: dot over e, divided by 8; max-subtracted softmax;
// weighted values), read from the fp16 cache the qkv product just wrote.
// Scores are K Q^T (K tile rows x 16 queries) and outputs V^T P^T (64 dims x
// 16 queries), so that a lane holds values of one query (lane % 16) in both,
// and the weights of a tile feed the second product from the registers the
// first left them in: the instruction's fold position 8q + e of lane group q
// stands for cache position 4q + e (e < 4) and 16 + 4q + e - 4 of a tile's 32,
// and V is staged in that order. Queries (scaled by a power of two per query,
// so that any fp32 magnitude splits) and softmax weights go in as three fp16
// planes (pf_split24: 24 bits), the two lower ones in one accumulator. The two
// halves of a score's dims, and each tile's weighted values and weights, are
// summed on their own and added in fp32 after, so that no sum is a chain over
// all positions. Errors against 64 bits, relative (2-norm), fp32 throughout with
// a wave per (query row, head) / halves of 22 bits in running accumulators / this:
// GPT-2 small 1 x 37 7.5e-8 / 7.8e-8 / 7.3e-8, 2 x 768 1.03e-7 / 1.15e-7 / 8.7e-8,
// 1 x 200 after 700 positions 1.93e-7 / 2.26e-7 / 1.2e-7, medium 3 x 333 after 100
// 1.33e-7 / 1.50e-7 / 1.08e-7.
// A score whose hi part is not finite (the cache may hold an infinity) is made
// again in fp32: 0 * inf of a plane that is 0 where the query is not would make
// an infinity a NaN.
// What bounds it: vector work on the scores (exponentials, maxima, splits;
// about twice the matrix-core time); few queries: the chain of tiles, 1.6 us
// each. GPT-2 small, 32 x 768: 144 us a layer alone and 153 in a pass, against
// 1198 with a wave per (query row, head), which read every cache row once per
// query; 8 x 128 6.8 against 19.7; medium 3 x 333 after 100 positions 16.5 alone
// and 18 in a pass against 59. The third plane and the sums by tile are 6-15% of
// that (32 x 768 140 -> 161 on one box, 8 x 128 7.1 -> 7.5), the check for scores
// that are not finite -5 to 5% (8 x 128 7.2 -> 6.8, XL 64 x 128 37.2 -> 39.0).
// F receives the head's output, row m, in fragment order.

// A wave's lanes hand each other values through LDS, whose operations a wave
// executes in order: this keeps the compiler to that order too (it emits
// nothing).
__device__ __forceinline__ void pf_wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

// One query over at most 64 positions by one wave, in fp32 throughout: eight
// lanes per position for the dots (the partial dots added across them), a
// lane per position for the weights, eight lanes of 8 dims for each residue of
// the positions mod 8 in the weighted values. `ws`: 64 floats of LDS.
__device__ __forceinline__ void pf_attn_short(const float* __restrict__ qp, const vh_half* __restrict__ kb,
                                              const vh_half* __restrict__ vb, int D, int pos, float* ws, int lane,
                                              float* o) {
  const int g = lane >> 3, c8 = lane & 7;
  float qv[8];
  pf_ld8f(qp + 8 * c8, qv);
  float mx = -INFINITY;
  pf_wave_sync();                                                  // the query before is read
  for (int s = g; s <= pos; s += 8) {
    float kv[8], acc = 0.0f;
    unpack8(ld16(kb + (size_t)s * D + 8 * c8), kv);
#pragma unroll
    for (int j = 0; j < 8; ++j) acc = fmaf(qv[j], kv[j], acc);
    acc += __shfl_xor(acc, 1, 64);
    acc += __shfl_xor(acc, 2, 64);
    acc += __shfl_xor(acc, 4, 64);
    const float sc = acc * 0.125f;                                 // / 8, exact
    if (c8 == 0) ws[s] = sc;
    mx = fmaxf(mx, sc);
  }
  mx = wave_red_max(mx);
  pf_wave_sync();
  const float ex = lane <= pos ? expf(ws[lane] - mx) : 0.0f;
  const float sum = wave_red_sum(ex);
  ws[lane] = ex / sum;
  pf_wave_sync();
#pragma unroll
  for (int j = 0; j < 8; ++j) o[j] = 0.0f;
  for (int s = g; s <= pos; s += 8) {
    float v[8];
    unpack8(ld16(vb + (size_t)s * D + 8 * c8), v);
    const float w = ws[s];
#pragma unroll
    for (int j = 0; j < 8; ++j) o[j] = fmaf(w, v[j], o[j]);
  }
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    o[j] += __shfl_xor(o[j], 8, 64);
    o[j] += __shfl_xor(o[j], 16, 64);
    o[j] += __shfl_xor(o[j], 32, 64);
  }
}

// With SPLIT a block makes 16 queries: its waves take every fourth tile of
// positions each, staged for themselves, and combine at the end: where few
// queries would leave waves or most of the chip idle over a long cache
// (GPT-2 small, 3 tokens after 900 positions: 25.1 -> 11.1 us a launch). A
// prompt of at most PF_SHORT tokens that sees at most 64 positions goes a
// query at a time instead (pf_attn_short; no slower: one tile has no parts to
// split).
#define PF_SHORT 8
template <bool SPLIT>
__device__ __forceinline__ void pf_attn_body(const float* __restrict__ Q, const vh_half* __restrict__ kc,
                                             const vh_half* __restrict__ vc, int B, int P, const int* __restrict__ tp,
                                             int layer, int L, int tmax, int H, vh_half* __restrict__ F, int MT,
                                             unsigned* __restrict__ err) {
  constexpr int QT = SPLIT ? 16 : 64, NB = SPLIT ? 4 : 2;          // queries of a block; staged tiles
  constexpr int NK = SPLIT ? 8 : 2, NV = SPLIT ? 4 : 1;            // a lane's pieces of a staged tile
  __shared__ __attribute__((aligned(16))) vh_u32x4 lk[NB][512];    // [position tile][k-step of dims][lane]
  __shared__ __attribute__((aligned(16))) vh_u32x4 lv[NB][512];    // [dim tile][k-step of positions][lane]
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
  const int r = lane & 15, q = lane >> 4;
  const int nq = (P + QT - 1) / QT, T = B * H * nq;
  // contiguous runs of blocks per XCD (blockIdx % 8): a (row, head)'s blocks
  // share its cache rows in one L2; within it the longest first
  const int per = (T + 7) / 8, id = (int)(blockIdx.x & 7) * per + (int)(blockIdx.x >> 3);
  if ((int)(blockIdx.x >> 3) >= per || id >= T) return;            // grid: 8 * ceil(T / 8) blocks
  const int p0 = (nq - 1 - id % nq) * QT, h = id / nq % H, b = id / nq / H;
  const int D = H * PF_E, t0 = *tp;
  const size_t base = (size_t)(b * L + layer) * tmax * D + (size_t)h * PF_E;
  const int w0 = SPLIT ? p0 : p0 + 16 * wave;                      // the wave's first query
  const int pq = w0 + r;                                           // this lane's query
  const bool live = pq < P;
  const int lim = min(t0 + min(pq, P - 1), tmax - 1);              // its last position
  const int last = min(t0 + min(p0 + QT, P) - 1, tmax - 1);     // the block's
  const int wlast = min(t0 + min(w0 + 15, P - 1), tmax - 1);       // the wave's, and its first query's
  const int wfirst = min(t0 + min(w0, P - 1), tmax - 1);
  const bool wlive = w0 < P;
  const int nt = last < 0 ? 0 : last / 64 + 1;
  if (SPLIT && P <= PF_SHORT && last < 64) {
    bool bad = false;
    for (int p = wave; p < P; p += 4) {
      float o[8];
      pf_attn_short(Q + ((size_t)b * P + p) * D + h * PF_E, kc + base, vc + base, D, min(t0 + p, tmax - 1),
                    (float*)lk[wave], lane, o);
      if (lane < 8) pf_frag_put8(F, MT, D / 32, b * P + p, h * PF_E + 8 * lane, o, bad);
    }
    if (bad) stc_u(err, VH_ERR_RANGE);
    return;
  }
  // the query, scaled to below 1 by 2^-e, in its three planes: dims 32 s + 8 q .. + 7
  vh_u32x4 qh[2], ql[2], qt[2];
  float k2;                                                        // 2^e / 8 log2(e): scores in powers of 2
  {
    const float* qp = Q + ((size_t)b * P + min(pq, P - 1)) * D + h * PF_E + 8 * q;
    float v[2][8];
    float mx = 0.0f;
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      const vh_f32x4 a = *(const vh_f32x4*)(qp + 32 * s), c = *(const vh_f32x4*)(qp + 32 * s + 4);
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        v[s][j] = a[j];
        v[s][4 + j] = c[j];
      }
#pragma unroll
      for (int j = 0; j < 8; ++j) mx = fmaxf(mx, __builtin_fabsf(v[s][j]));
    }
    mx = fmaxf(mx, __shfl_xor(mx, 16, 64));
    mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
    int e = 0;
    if (mx > 0.0f && mx < INFINITY) e = max(__builtin_amdgcn_frexp_expf(mx), -100);
#pragma unroll
    for (int s = 0; s < 2; ++s) {
#pragma unroll
      for (int j = 0; j < 8; ++j) v[s][j] = __builtin_ldexpf(v[s][j], -e);
      pf_split24(v[s], qh[s], ql[s], qt[s]);
    }
    k2 = __builtin_ldexpf(0.125f * 1.44269504088896341f, e);
  }
  // staging: keys as they are, row 16 i + r of the tile in 16-byte pieces
  // c = 4 j + q; values of positions 4 va .. + 3, dims 4 vd .. + 3, transposed
  // in registers. A tile is staged by the block, or with SPLIT by each wave.
  // Positions past the last are read as the last (their weights are 0).
  const int sl0 = SPLIT ? 0 : wave, vd = tid & 15;
  vh_u32x4 kr[NK];
  vh_u32x2 vr[NV][4];
  auto gload = [&](int t) {
#pragma unroll
    for (int n = 0; n < NK; ++n) {
      const int kp = min(64 * t + 16 * (sl0 + n / 2) + r, last);
      kr[n] = ld16(kc + base + (size_t)kp * D + 8 * (4 * (n & 1) + q));
    }
#pragma unroll
    for (int n = 0; n < NV; ++n)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int vp = min(64 * t + 4 * (4 * (sl0 + n) + q) + i, last);
        vr[n][i] = ld8(vc + base + (size_t)vp * D + 4 * vd);
      }
  };
  auto put = [&](int buf) {
#pragma unroll
    for (int n = 0; n < NK; ++n) lk[buf][(2 * (sl0 + n / 2) + (n & 1)) * 64 + lane] = kr[n];
    // dims 4 vd + j: dim tile vd / 4, row 4 (vd % 4) + j of it; positions
    // 4 va ..: k-step va / 8, half (va % 8) / 4 of lane group va % 4's eight
#pragma unroll
    for (int n = 0; n < NV; ++n) {
      const int va = 4 * (sl0 + n) + q;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const unsigned sel = j & 1 ? 0x07060302u : 0x05040100u;
        const vh_u32x2 w = {__builtin_amdgcn_perm(vr[n][1][j >> 1], vr[n][0][j >> 1], sel),
                            __builtin_amdgcn_perm(vr[n][3][j >> 1], vr[n][2][j >> 1], sel)};
        const int piece = (vd / 4 * 2 + va / 8) * 64 + (va & 3) * 16 + 4 * (vd & 3) + j;
        *((vh_u32x2*)&lv[buf][piece] + ((va & 7) >> 2)) = w;
      }
    }
  };
  float o[4][4] = {};                    // weighted values: dim tile, dim of it
  float m2 = -INFINITY, sum = 0.0f;      // largest score in powers of 2; the sum of this lane's positions
  if constexpr (SPLIT) {
    if (wave < nt) gload(wave);
  } else if (nt > 0) {
    gload(0);
    put(0);
    if (nt > 1) gload(1);
  }
  for (int t = SPLIT ? wave : 0; t < nt; t += SPLIT ? 4 : 1) {
    if constexpr (SPLIT) {
      pf_wave_sync();                      // the wave's own tile: the one before is read
      put(wave);
      pf_wave_sync();
      if (t + 4 < nt) gload(t + 4);
    } else {
      vh_lds_sync();
      if (t + 1 < nt) {                    // the other buffer: read before the previous barrier
        put((t + 1) & 1);
        if (t + 2 < nt) gload(t + 2);
      }
      if (!wlive || 64 * t > wlast) continue;
    }
    const int buf = SPLIT ? wave : t & 1;
    const vh_u32x4 *K = lk[buf], *V = lv[buf];
    float s[4][4], fin = 0.0f;                                     // fin: a NaN if any hi part is not finite
    vh_f32x4 sh[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      vh_f32x4 h[2] = {}, sl = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
      for (int k = 0; k < 2; ++k) {
        const vh_u32x4 kf = K[(2 * i + k) * 64 + lane];
        h[k] = vh_mfma(kf, qh[k], h[k]);
        sl = vh_mfma(kf, ql[k], sl);
        sl = vh_mfma(kf, qt[k], sl);
      }
      sh[i] = vh_f32x4{h[0][0] + h[1][0], h[0][1] + h[1][1], h[0][2] + h[1][2], h[0][3] + h[1][3]};
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        s[i][j] = vh_hilo(sh[i][j], sl[j]);
        fin = fmaf(sh[i][j], 0.0f, fin);
      }
    }
    if (__any(fin != fin)) {
      const float* qp = Q + ((size_t)b * P + min(pq, P - 1)) * D + h * PF_E;
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          float acc = 0.0f;
#pragma nounroll
          for (int c = 0; c < 8; ++c) {
            float kv[8];
            unpack8(K[(2 * i + (c >> 2)) * 64 + 16 * (c & 3) + 4 * q + j], kv);
#pragma unroll
            for (int d = 0; d < 8; ++d) acc = fmaf(qp[8 * c + d], kv[d], acc);
          }
          if (!(__builtin_fabsf(sh[i][j]) < INFINITY)) s[i][j] = acc;
        }
    }
    if (64 * t + 63 > wfirst) {                                    // a tile that some query sees in part
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) s[i][j] = 64 * t + 16 * i + 4 * q + j <= lim ? s[i][j] : -INFINITY;
    }
    float bm = s[0][0];
#pragma unroll
    for (int n = 1; n < 16; ++n) bm = fmaxf(bm, s[n >> 2][n & 3]);
    bm = fmaxf(bm, __shfl_xor(bm, 16, 64));
    bm = fmaxf(bm, __shfl_xor(bm, 32, 64));
    const float n2 = fmaxf(m2, bm * k2);
    const float ref = n2 == -INFINITY ? 0.0f : n2;                 // no score above -inf yet: all weights 0
    const float c = __builtin_amdgcn_exp2f(m2 - ref);              // 0 while m2 is -inf
    m2 = n2;
    vh_u32x4 ph[2], pl[2], pt[2];
    float ts[2];
#pragma unroll
    for (int k = 0; k < 2; ++k) {
      float w[8];
#pragma unroll
      for (int j = 0; j < 8; ++j) w[j] = __builtin_amdgcn_exp2f(fmaf(s[2 * k + (j >> 2)][j & 3], k2, -ref));
      ts[k] = ((w[0] + w[1]) + (w[2] + w[3])) + ((w[4] + w[5]) + (w[6] + w[7]));
      pf_split24(w, ph[k], pl[k], pt[k]);
    }
    sum = fmaf(sum, c, ts[0] + ts[1]);
#pragma unroll
    for (int d = 0; d < 4; ++d) {
      vh_f32x4 th = {0.0f, 0.0f, 0.0f, 0.0f}, tl = th;
#pragma unroll
      for (int k = 0; k < 2; ++k) {
        const vh_u32x4 vf = V[(2 * d + k) * 64 + lane];
        th = vh_mfma(vf, ph[k], th);
        tl = vh_mfma(vf, pl[k], tl);
        tl = vh_mfma(vf, pt[k], tl);
      }
#pragma unroll
      for (int j = 0; j < 4; ++j) o[d][j] = fmaf(o[d][j], c, vh_hilo(th[j], tl[j]));
    }
  }
  sum += __shfl_xor(sum, 16, 64);
  sum += __shfl_xor(sum, 32, 64);
  if constexpr (SPLIT) {
    // each wave's maximum, sum and output rescaled to the common maximum and
    // added in wave order; wave w then writes dim tile w
    float *om = (float*)lk[0], *ow = (float*)lv[0];                // [wave][maximum, sum][16], [wave][dim tile][j][lane]
    __syncthreads();
    if (q == 0) {
      om[wave * 32 + r] = m2;
      om[wave * 32 + 16 + r] = sum;
    }
#pragma unroll
    for (int d = 0; d < 4; ++d)
#pragma unroll
      for (int j = 0; j < 4; ++j) ow[((wave * 4 + d) * 4 + j) * 64 + lane] = o[d][j];
    __syncthreads();
    float m = om[r];
#pragma unroll
    for (int w = 1; w < 4; ++w) m = fmaxf(m, om[w * 32 + r]);
    sum = 0.0f;
    float v[4] = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int w = 0; w < 4; ++w) {
      const float wm = om[w * 32 + r], f = wm == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(wm - m);   // no score: 0
      sum = fmaf(om[w * 32 + 16 + r], f, sum);
#pragma unroll
      for (int j = 0; j < 4; ++j) v[j] = fmaf(ow[((w * 4 + wave) * 4 + j) * 64 + lane], f, v[j]);
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) o[0][j] = v[j];
  }
  if (!live) return;
  bool bad = false;
#pragma unroll
  for (int d = 0; d < (SPLIT ? 1 : 4); ++d) {
#pragma unroll
    for (int j = 0; j < 4; ++j) o[d][j] = lim < 0 ? 0.0f : o[d][j] / sum;
    pf_frag_put4(F, MT, D / 32, b * P + pq, h * PF_E + 16 * (SPLIT ? wave : d) + 4 * q, o[d], bad);
  }
  if (bad) stc_u(err, VH_ERR_RANGE);
}
#define PF_ATTN(name, split)                                                                                        \
  extern "C" __global__ __launch_bounds__(256, 2) void name(                                                        \
      const float* __restrict__ Q, const vh_half* __restrict__ kc, const vh_half* __restrict__ vc, int B, int P,    \
      const int* __restrict__ tp, int layer, int L, int tmax, int H, vh_half* __restrict__ F, int MT,               \
      unsigned* __restrict__ err) {                                                                                 \
    pf_attn_body<split>(Q, kc, vc, B, P, tp, layer, L, tmax, H, F, MT, err);                                        \
  }
PF_ATTN(pf_attn, false)
PF_ATTN(pf_attn16, true)

// One position per row (a decode step): one block per (row m, head h), every
// thread of the block on the positions 0 .. t0, so that a step's cache rows
// are read with a block's worth of loads in flight instead of a wave's. Each
// score is read by eight lanes, one 16-byte piece of the position's key row
// each (so a wave's load covers eight whole rows), the eight partial dots
// added across the lanes, / 8; the max-subtracted softmax (block-wide maximum
// and sum); the weighted values with wave w, lane 8a + b on positions
// s = 8w + a (mod 32), dims 8b..8b+7, the four waves' partial outputs added
// in order through LDS. (Keys read a row per lane, eight 16-byte loads of it,
// measured slower: XL B=64 decode 4.32 against 4.06 ms per step.) The cache
// rows are loaded nontemporal here and in pf_attn1s: a step reads each once,
// and with the default policy they displaced the products' weights from the
// caches (same box: GPT-2 small at 32 rows 0.586 -> 0.550 ms per step, the
// attention launch 19.3 -> 17.8 us; XL at 64 rows 3.023 -> 3.000).
extern "C" __global__ __launch_bounds__(256) void pf_attn1(const float* __restrict__ Q, const vh_half* __restrict__ kc,
                                                            const vh_half* __restrict__ vc,
                                                            const int* __restrict__ tp, int layer, int L, int tmax,
                                                            int H, vh_half* __restrict__ F, int MT,
                                                            unsigned* __restrict__ err) {
  __shared__ float qs[PF_E];
  __shared__ float ws[PF_TMAX];
  __shared__ float red[VNWAVE];
  __shared__ float part[VNWAVE][PF_E];
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  const int m = blockIdx.x / H, h = blockIdx.x % H;      // grid: rows * H blocks exactly
  const int D = H * PF_E;
  const size_t base = (size_t)(m * L + layer) * tmax * D + (size_t)h * PF_E;
  // scores: eight lanes per position (lane 8g + b holds dims 8b .. 8b + 7, one
  // 16-byte load), positions g, g + 32, .. of the block's 32 lane groups, four
  // in flight per lane; the eight partial dots added across the group. The
  // query and the first batch (positions below 128, clamped into the cache) are
  // loaded before the position is read, so that their round trips overlap;
  // the batch's positions beyond the step's are loaded but not used.
  const int g = tid >> 3, b8 = tid & 7;
  float qv[8];
  {
    const float* qp = Q + (size_t)m * D + h * PF_E + 8 * b8;
    const vh_f32x4 q0 = *(const vh_f32x4*)qp, q1 = *(const vh_f32x4*)(qp + 4);
    qv[0] = q0[0]; qv[1] = q0[1]; qv[2] = q0[2]; qv[3] = q0[3];
    qv[4] = q1[0]; qv[5] = q1[1]; qv[6] = q1[2]; qv[7] = q1[3];
  }
  vh_u32x4 kr[4];
#pragma unroll
  for (int u = 0; u < 4; ++u) {
    const int s = g + 32 * u < tmax ? g + 32 * u : tmax - 1;     // clamped: loads without a branch
    kr[u] = ld16_nt(kc + base + (size_t)s * D + 8 * b8);
  }
  __builtin_amdgcn_sched_barrier(0);    // the loads above issued before the position is waited for
  const int at = *tp;
  const int pos = at < tmax ? at : tmax - 1;
  float mx = -INFINITY;
  int s0 = g;
  do {                                  // the first batch even where g > pos (then none of it is used)
    if (s0 != g) {
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const int s = s0 + 32 * u;
        kr[u] = s <= pos ? ld16_nt(kc + base + (size_t)s * D + 8 * b8) : vh_u32x4{0u, 0u, 0u, 0u};
      }
    }
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      float kv[8];
      unpack8(kr[u], kv);
      float acc = 0.0f;
#pragma unroll
      for (int j = 0; j < 8; ++j) acc = fmaf(qv[j], kv[j], acc);
      acc += __shfl_xor(acc, 1, 64);
      acc += __shfl_xor(acc, 2, 64);
      acc += __shfl_xor(acc, 4, 64);
      const int s = s0 + 32 * u;
      if (s <= pos) {
        const float sc = acc * 0.125f;      // / 8, exact
        if (b8 == 0) ws[s] = sc;
        mx = fmaxf(mx, sc);
      }
    }
    s0 += 32 * 4;
  } while (s0 <= pos);
  __syncthreads();                      // ws written by the groups' first lanes, read by all below
  mx = wave_red_max(mx);
  if (lane == 0) red[wave] = mx;
  __syncthreads();
  mx = red[0];
#pragma unroll
  for (int w = 1; w < VNWAVE; ++w) mx = fmaxf(mx, red[w]);
  __syncthreads();                      // red is reused for the sum
  float sum = 0.0f;
  for (int s = tid; s <= pos; s += VBLOCK) {
    const float ex = expf(ws[s] - mx);
    ws[s] = ex;
    sum += ex;
  }
  sum = wave_red_sum(sum);
  if (lane == 0) red[wave] = sum;
  __syncthreads();
  sum = red[0];
#pragma unroll
  for (int w = 1; w < VNWAVE; ++w) sum += red[w];
  for (int s = tid; s <= pos; s += VBLOCK) ws[s] = ws[s] / sum;
  __syncthreads();
  const int a = lane >> 3, b = lane & 7;
  float o[8] = {0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f};
  for (int s0 = 8 * wave; s0 <= pos; s0 += 32 * 4) {
    vh_u32x4 vr[4];
    float wv[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int s = s0 + 32 * u + a;
      const bool in = s <= pos;
      vr[u] = in ? ld16_nt(vc + base + (size_t)s * D + 8 * b) : vh_u32x4{0u, 0u, 0u, 0u};
      wv[u] = in ? ws[s] : 0.0f;
    }
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      float v[8];
      unpack8(vr[u], v);
#pragma unroll
      for (int j = 0; j < 8; ++j) o[j] = fmaf(wv[u], v[j], o[j]);
    }
  }
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    o[j] += __shfl_xor(o[j], 8, 64);
    o[j] += __shfl_xor(o[j], 16, 64);
    o[j] += __shfl_xor(o[j], 32, 64);
  }
  if (a == 0) {
#pragma unroll
    for (int j = 0; j < 8; ++j) part[wave][8 * b + j] = o[j];
  }
  __syncthreads();
  if (tid < PF_E) {
    float r = part[0][tid];
#pragma unroll
    for (int w = 1; w < VNWAVE; ++w) r += part[w][tid];
    qs[tid] = r;
  }
  __syncthreads();
  bool bad = false;         // the head's 64 outputs in fragment order, eight per thread
  if (tid < PF_E / 8) pf_frag_put8(F, MT, D / 32, m, h * PF_E + 8 * tid, qs + 8 * tid, bad);
  if (bad) stc_u(err, VH_ERR_RANGE);
}

// pf_attn1 in one pass over the cache (a running softmax): lane group g
// (eight lanes, one 16-byte piece of a row each) takes positions g, g + 32, ..
// and loads each position's key and value pieces together, four positions a
// batch. Per batch the group's running maximum m becomes max(m, its scores),
// its sum l and weighted values (eight dims per lane) are rescaled by
// exp(m_old - m) and the batch's exp(score - m) added. The 32 groups are then
// combined in group order, each rescaled by exp(m_g - max_g m_g): the output is
// the sum of the weighted values over the sum of the l's. One round trip to
// the cache per batch instead of one for the keys and one for the values:
// faster where there are few (row, head) blocks (GPT-2 small, 32 rows, 1024
// positions: 0.666 -> 0.637 ms per step), not with many (XL, 64 rows x 25
// heads: 3.110 -> 3.128), so the decode pass takes it up to
// ATTN_ONE_PASS_BLOCKS blocks. The first batch (positions below 128, clamped into
// the cache) is loaded before the position is read, so that its round trip
// overlaps that read and the query's; its positions beyond the step's are
// loaded but not used.
extern "C" __global__ __launch_bounds__(256) void pf_attn1s(const float* __restrict__ Q, const vh_half* __restrict__ kc,
                                                             const vh_half* __restrict__ vc,
                                                             const int* __restrict__ tp, int layer, int L, int tmax,
                                                             int H, vh_half* __restrict__ F, int MT,
                                                             unsigned* __restrict__ err) {
  __shared__ float qs[PF_E];
  __shared__ float gm[32], gl[32], gf[32];
  __shared__ float part[32][PF_E];
  const int tid = threadIdx.x;
  const int m = blockIdx.x / H, h = blockIdx.x % H;      // grid: rows * H blocks exactly
  const int D = H * PF_E;
  const size_t base = (size_t)(m * L + layer) * tmax * D + (size_t)h * PF_E;
  const int g = tid >> 3, b8 = tid & 7;
  float qv[8];
  {
    const float* qp = Q + (size_t)m * D + h * PF_E + 8 * b8;
    const vh_f32x4 q0 = *(const vh_f32x4*)qp, q1 = *(const vh_f32x4*)(qp + 4);
    qv[0] = q0[0]; qv[1] = q0[1]; qv[2] = q0[2]; qv[3] = q0[3];
    qv[4] = q1[0]; qv[5] = q1[1]; qv[6] = q1[2]; qv[7] = q1[3];
  }
  vh_u32x4 kr[4], vr[4];
#pragma unroll
  for (int u = 0; u < 4; ++u) {
    const int s = g + 32 * u < tmax ? g + 32 * u : tmax - 1;     // clamped: loads without a branch
    const size_t at8 = base + (size_t)s * D + 8 * b8;
    kr[u] = ld16_nt(kc + at8);
    vr[u] = ld16_nt(vc + at8);
  }
  __builtin_amdgcn_sched_barrier(0);    // the loads above issued before the position is waited for
  const int at = *tp;
  const int pos = at < tmax ? at : tmax - 1;
  float mx = -INFINITY, sm = 0.0f, o[8] = {0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f};
  int s0 = g;
  do {                                      // the first batch even where g > pos (then none of it is used)
    if (s0 != g) {
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const int s = s0 + 32 * u;
        const size_t at8 = base + (size_t)s * D + 8 * b8;
        kr[u] = s <= pos ? ld16_nt(kc + at8) : vh_u32x4{0u, 0u, 0u, 0u};
        vr[u] = s <= pos ? ld16_nt(vc + at8) : vh_u32x4{0u, 0u, 0u, 0u};
      }
    }
    float sc[4];
    float bm = mx;
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      float kv[8];
      unpack8(kr[u], kv);
      float acc = 0.0f;
#pragma unroll
      for (int j = 0; j < 8; ++j) acc = fmaf(qv[j], kv[j], acc);
      acc += __shfl_xor(acc, 1, 64);
      acc += __shfl_xor(acc, 2, 64);
      acc += __shfl_xor(acc, 4, 64);
      sc[u] = acc * 0.125f;                 // / 8, exact
      if (s0 + 32 * u <= pos) bm = fmaxf(bm, sc[u]);
    }
    const float c = bm == -INFINITY ? 0.0f : expf(mx - bm);   // 0 while mx is -inf, or no position yet
    sm *= c;
#pragma unroll
    for (int j = 0; j < 8; ++j) o[j] *= c;
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      if (s0 + 32 * u > pos) continue;
      const float p = expf(sc[u] - bm);
      float v[8];
      unpack8(vr[u], v);
      sm += p;
#pragma unroll
      for (int j = 0; j < 8; ++j) o[j] = fmaf(p, v[j], o[j]);
    }
    mx = bm;
    s0 += 32 * 4;
  } while (s0 <= pos);
  if (b8 == 0) {
    gm[g] = mx;
    gl[g] = sm;
  }
#pragma unroll
  for (int j = 0; j < 8; ++j) part[g][8 * b8 + j] = o[j];
  __syncthreads();
  if (tid < 32) {             // each group's scale (0 for a group with no position)
    float M = gm[0];
    for (int k = 1; k < 32; ++k) M = fmaxf(M, gm[k]);
    gf[tid] = gm[tid] == -INFINITY ? 0.0f : expf(gm[tid] - M);
  }
  __syncthreads();
  if (tid < PF_E) {
    float l = 0.0f, r = 0.0f;
    for (int k = 0; k < 32; ++k) {
      l = fmaf(gl[k], gf[k], l);
      r = fmaf(part[k][tid], gf[k], r);
    }
    r = r / l;
    qs[tid] = r;
  }
  __syncthreads();
  bool bad = false;         // the head's 64 outputs in fragment order, eight per thread
  if (tid < PF_E / 8) pf_frag_put8(F, MT, D / 32, m, h * PF_E + 8 * tid, qs + 8 * tid, bad);
  if (bad) stc_u(err, VH_ERR_RANGE);
}

// ---------------------------------------------------------------- argmax
// Per row of logits [B, V]: the largest value, a tie to the lowest id
// (gpt2.vst Q10), in two launches so that a row is read by S blocks at once.
// pf_argmax_part: block b * S + s takes chunk s of row b and writes its pair
// (value, id) to pv / pi. pf_argmax: one block per row combines the S pairs
// (the rule picks the same pair in any order), writes the token into x (the
// next step's input) and, as a float, into `next`; block 0 advances the
// position counter by P.
extern "C" __global__ __launch_bounds__(256) void pf_argmax_part(const float* __restrict__ logit, int V, int S,
                                                                  float* __restrict__ pv, int* __restrict__ pi) {
  __shared__ float rv[VNWAVE];
  __shared__ int ri[VNWAVE];
  const int b = blockIdx.x / S, s = blockIdx.x % S;
  const int chunk = (V + S - 1) / S;
  const int n0 = s * chunk, n1 = min(V, n0 + chunk);
  const float* lg = logit + (size_t)b * V;
  float best = -INFINITY;
  int id = V;
#pragma unroll 4
  for (int n = n0 + (int)threadIdx.x; n < n1; n += VBLOCK) argmax_pair(best, id, lg[n], n);
  block_argmax(best, id, rv, ri);
  if (threadIdx.x == 0) {
    pv[blockIdx.x] = best;
    pi[blockIdx.x] = id;
  }
}

extern "C" __global__ __launch_bounds__(256) void pf_argmax(const float* __restrict__ pv, const int* __restrict__ pi,
                                                             int S, int* __restrict__ x, float* __restrict__ next,
                                                             int* __restrict__ tp, int P) {
  __shared__ float rv[VNWAVE];
  __shared__ int ri[VNWAVE];
  float best = -INFINITY;
  int id = 0x7fffffff;
  for (int k = threadIdx.x; k < S; k += VBLOCK) argmax_pair(best, id, pv[blockIdx.x * S + k], pi[blockIdx.x * S + k]);
  block_argmax(best, id, rv, ri);
  if (threadIdx.x == 0) {
    x[blockIdx.x] = id;
    next[blockIdx.x] = (float)id;
    if (blockIdx.x == 0) *tp += P;     // the last kernel of a pass: advance the position
  }
}
