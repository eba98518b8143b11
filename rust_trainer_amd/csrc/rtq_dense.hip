// rtq_dense.hip — products of the trainer-native weights (FrozenWeight::{F32, Q8_0},
// src/frozen.rs:33-187: f32 [N][K], or f32 scales per 32 elements and int8 codes) with f32
// activations.  Included by rtq_kernels.hip (one code object).
//
//   rtq_dense_fwd32 / 64[_q8]:  y[t][n]  = sum_k x[t][k] W[n][k] (+ bias[n]) (+ s sum_j h[t][j] B[n][j])
//   rtq_dense_bwd32 / 64[_q8]:  part[z][t][k] = sum over the rows n of split z of dy[t][n] W[n][k]
//     (rtq_bwd_finish sums the splits in order), or dx itself when there is one split and no adapter.
//
// An f32 value is exactly the sum of three bf16 values (each the truncation of what is left: mid is below
// 2^-7 of the value's leading bit, lo below 2^-15), so a product is eight bf16 MFMAs (all pairs of planes but
// lo lo, below 2^-30 of the product, a fraction of an f32 rounding) at 16 times the f32 MFMA's rate.  Without
// mid lo and lo mid a product lost up to 2^-21, always in its own sign: a sum of one or a few large terms was
// off by up to 3.5e-7 where f32 products leave 6e-8.
// hi hi and the corrections accumulate apart.  The forward of codes needs three: a code is one exact
// bf16 value, and a 32-element step is one scale's block, whose sum is scaled once (f32 FMA).  Its hi part and
// the rest meet in an f32 add: the MFMA's own sum of the two is not rounded to nearest (a product of one term
// was off by up to 2.4 2^-24 instead of 2 2^-24).
// bf16 keeps f32's exponent range, so no operand is scaled.  But the bf16 MFMA takes a denormal operand or
// product as zero: below about 2^-110 a value loses its lo plane, and products below 2^-100 their corrections
// (1e-34 times 0.02 was off by up to 3000 2^-24).  What is lost is below 2^-126 a term, so an output of 2^-80
// or more does not notice, and a smaller one is summed again on the f32 MFMA.  (An output below the least
// normal value can come out as 0.)  An infinite or NaN operand turns the split
// sums into NaN, and an unscaled sum of codes can overflow where the scaled one does not: an output that is
// not finite is summed again too.  1024 x 1024, 512 tokens, all outputs summed again: 82 us a forward product
// against 20, 108 against 18 for TQ8_0.
//
// Workgroup: four waves, 64 weight-side outputs x 16 TT tokens (TT = 4: wave (w % 2, w / 2) takes 32 x
// 32; TT = 2: wave w takes 16 x 32).  Per 32-element step the operands go global -> registers (D - 1
// steps ahead) -> planes in LDS, double buffered, one barrier per step.  The loads put a row's 128 bytes
// in consecutive lanes: the L1 looks up one line per cycle, and lanes of one load that each touch a row
// of their own (the order the fragments want) held the forward at 0.9 lookups per cycle: 273 us against
// 230 at 4096 x 4096, 1024 tokens, and 212 without the bank conflicts below.  A fragment (16 rows x 32 elements of one plane) is 64 16-byte
// slots, row r of k-group g at (r ^ g) + 16 g, a transposed weight tile's fragments lie one slot further
// apart, and the eight rows of a wave's load are 4 apart (two sets): reads and writes then spread
// over the banks (a 16-byte access serves lanes 0-3, 12-15, 20-23, 24-27 together, an 8-byte one a half-wave;
// conflicts are 0.1% of the forward's cycles and 6% of the backward's).
// Measured, TQ8_0 2048 x 1024, 300 tokens, forward + backward with a rank-8 adapter, whole call: 313 us
// on the f32 MFMA GEMM with one launch per adapter product, 61 here (six products: 59; 4096 x 4096, 1024 tokens,
// backward 327 against 300); against float64 8.5e-7 there, 2.6e-7 here.  Bound by the wait of each step (one
// barrier, LDS and MFMA latency) at small grids, by MFMA and LDS at large ones.
#define DENSE_D 4
constexpr int kDenseFrag = 64;  // 16-byte slots of a fragment
__device__ __forceinline__ int dense_slot(int r, int g) { return (r ^ g) + 16 * g; }

template <bool BWD, bool Q8>
struct DenseSlotW {
  f4 v[2];      // f32: fwd rows tid / 4.. (see below), bwd rows n, n + 1
  u2v q;        // codes
  float sc[2];  // bwd: the rows' scales; fwd: sc[0] of row tid (tid < 64)
};

// three bf16 planes of the pair (a, b), each one word: a in the low half
__device__ __forceinline__ void split3(float a, float b, uint32_t& h, uint32_t& m, uint32_t& l) {
  const uint32_t ua = __float_as_uint(a), ub = __float_as_uint(b);
  h = __builtin_amdgcn_perm(ub, ua, 0x07060302u);
  const float ra = a - __uint_as_float(ua & 0xffff0000u), rb = b - __uint_as_float(ub & 0xffff0000u);
  const uint32_t va = __float_as_uint(ra), vb = __float_as_uint(rb);
  m = __builtin_amdgcn_perm(vb, va, 0x07060302u);
  const float sa = ra - __uint_as_float(va & 0xffff0000u), sb = rb - __uint_as_float(vb & 0xffff0000u);
  l = __builtin_amdgcn_perm(__float_as_uint(sb), __float_as_uint(sa), 0x07060302u);
}

__device__ __forceinline__ bool dense_again(float v) {
  const float m = fabsf(v);
  return !(m < INFINITY) || (m > 0.0f && m < 0x1p-80f);
}

template <bool BWD, bool Q8, int TT>
__device__ __forceinline__ void dense_tile(const DenseGemmArgs& a) {
  constexpr int D = DENSE_D, WC = TT == 4 ? 2 : 1, WT = 2;  // a wave's weight-side and token tiles
  constexpr bool CODES = Q8 && !BWD;                        // weight operand: exact codes, one plane
  constexpr int PW = CODES ? 1 : 3, NX = TT / 2;            // float4 of x per thread and step
  constexpr int WS = PW * kDenseFrag + (BWD ? 1 : 0);       // slots of a weight tile
  const int O = BWD ? a.K : a.N, C = BWD ? a.N : a.K;       // outputs per token, contraction length
  const int ncb = (O + 63) / 64, ntb = (a.T + 16 * TT - 1) / (16 * TT), nmain = ncb * ntb * a.nsplit;
  if ((int)blockIdx.x >= (nmain + 7) / 8 * 8) {
    if (BWD) dx_lora_sums(a, blockIdx.x - (nmain + 7) / 8 * 8, gridDim.x - (nmain + 7) / 8 * 8);
    return;  // uniform, before any barrier
  }
  // XCD blockIdx % 8 takes a run of units, token tiles fastest: the workgroups of a weight tile share its L2
  const int xcd = blockIdx.x & 7, per = nmain >> 3, rem = nmain & 7, in = blockIdx.x >> 3;
  if (in >= per + (xcd < rem ? 1 : 0)) return;
  const int u = xcd * per + min(xcd, rem) + in;
  const int tb = u % ntb, cb = u / ntb % ncb, z = u / (ntb * ncb);
  const int t0 = tb * 16 * TT, o0 = cb * 64;
  const int c0 = BWD ? z * a.n_per_split : 0, c1 = BWD ? min(C, c0 + a.n_per_split) : C;
  const int nsteps = (c1 - c0 + 31) / 32;

  __shared__ u4v lds[2][TT * 3 * kDenseFrag + 4 * WS];
  __shared__ float sD[2][64];
  const int tid = threadIdx.x, lane = tid & 63, li = lane & 15, g = lane >> 4;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wc = TT == 4 ? (w & 1) * 2 : w, wt = TT == 4 ? (w >> 1) * 2 : 0;
  f4 acc[WT][WC], low[WT][WC];
#pragma unroll
  for (int i = 0; i < WT; i++)
#pragma unroll
    for (int j = 0; j < WC; j++) acc[i][j] = low[i][j] = f4{0.0f, 0.0f, 0.0f, 0.0f};

  const __amdgpu_buffer_rsrc_t rx = make_rsrc(a.x, (uint32_t)a.T * C * 4u);
  const __amdgpu_buffer_rsrc_t rw = Q8 ? make_rsrc(a.qs, (uint32_t)a.N * a.K) : make_rsrc(a.w, (uint32_t)a.N * a.K * 4u);
  const __amdgpu_buffer_rsrc_t rs = make_rsrc(a.sc, Q8 ? (uint32_t)a.N * (a.K / 32) * 4u : 0u);
  const bool xvec = !BWD || (C & 3) == 0;
  // x loader: row xr (+ 32), elements 4 q4 .. + 3 of the step
  const int xr = 16 * (w >> 1) + 2 * (w & 1) + 4 * ((lane >> 3) & 3) + (lane >> 5), q4 = lane & 7;
  uint32_t xo[NX];
#pragma unroll
  for (int m = 0; m < NX; m++) xo[m] = ((uint32_t)min(t0 + xr + 32 * m, a.T) * C + 4 * q4) * 4u;  // row T: past the end, zeros
  // weight loader.  fwd f32: as x, rows o0 + xr (+ 32); fwd codes: row o0 + cr, 8 codes from 8 c8;
  // bwd: rows n = 8 w + 2 g, n + 1 of the step, columns o0 + 4 li .. + 3
  const int cr = 16 * w + 4 * ((lane >> 2) & 3) + (lane >> 4), c8 = lane & 3, nb = 8 * w + 2 * g, kb = o0 + 4 * li;
  auto issue = [&](f4 (&X)[NX], DenseSlotW<BWD, Q8>& W, int step) {
    const int c = c0 + 32 * min(step, max(nsteps - 1, 0));  // clamped: always a real step
#pragma unroll
    for (int m = 0; m < NX; m++) {
      if (xvec) {
        X[m] = __builtin_bit_cast(f4, __builtin_amdgcn_raw_buffer_load_b128(rx, xo[m], (uint32_t)c * 4u, 0));
      } else {
#pragma unroll
        for (int e = 0; e < 4; e++)
          X[m][e] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rx, xo[m] + 4u * e, (uint32_t)c * 4u, 0));
      }
    }
    if constexpr (CODES) {
      const uint32_t o = (uint32_t)min(o0 + cr, a.N) * a.K + 8 * c8;
      W.q = __builtin_bit_cast(u2v, __builtin_amdgcn_raw_buffer_load_b64(rw, o, (uint32_t)c, 0));
      // every wave loads the 64 scales (no branch around a load), the first one stores them
      W.sc[0] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rs, (uint32_t)min(o0 + lane, a.N) * (a.K / 32) * 4u, (uint32_t)(c >> 5) * 4u, 0));
    } else if constexpr (!BWD) {
#pragma unroll
      for (int m = 0; m < 2; m++)
        W.v[m] = __builtin_bit_cast(f4, __builtin_amdgcn_raw_buffer_load_b128(
                                            rw, ((uint32_t)min(o0 + xr + 32 * m, a.N) * a.K + 4 * q4) * 4u, (uint32_t)c * 4u, 0));
    } else {
      const int kc = min(kb, a.K - 4);  // columns past K are computed and not stored
#pragma unroll
      for (int r = 0; r < 2; r++) {
        const uint32_t n = (uint32_t)min(c + nb + r, a.N);  // row N: past the end, zeros
        if constexpr (Q8) {
          W.q[r] = __builtin_amdgcn_raw_buffer_load_b32(rw, n * a.K + kc, 0, 0);
          W.sc[r] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rs, (n * (a.K / 32) + (kc >> 5)) * 4u, 0, 0));
        } else {
          W.v[r] = __builtin_bit_cast(f4, __builtin_amdgcn_raw_buffer_load_b128(rw, (n * a.K + kc) * 4u, 0, 0));
        }
      }
    }
  };
  // planes of four consecutive elements of row r -> slot (r % 16, k-group q4 / 2), half q4 % 2
  auto put4 = [&](u4v* base, int ts, int r, f4 v) {
    uint32_t h0, m0, l0, h1, m1, l1;
    split3(v[0], v[1], h0, m0, l0);
    split3(v[2], v[3], h1, m1, l1);
    u2v* p = reinterpret_cast<u2v*>(base + (r >> 4) * ts + dense_slot(r & 15, q4 >> 1)) + (q4 & 1);
    p[0] = u2v{h0, h1};
    p[2 * kDenseFrag] = u2v{m0, m1};
    p[4 * kDenseFrag] = u2v{l0, l1};
  };
  auto stage = [&](const f4 (&X)[NX], const DenseSlotW<BWD, Q8>& W, int buf, int step) {
    u4v* SX = lds[buf];
    u4v* SW = lds[buf] + TT * 3 * kDenseFrag;
    const int c = c0 + 32 * min(step, max(nsteps - 1, 0));
#pragma unroll
    for (int m = 0; m < NX; m++) {
      f4 v = X[m];
      if (BWD && c + 32 > a.N) {  // elements past N hold the next row's
#pragma unroll
        for (int e = 0; e < 4; e++)
          if (c + 4 * q4 + e >= a.N) v[e] = 0.0f;
      }
      put4(SX, 3 * kDenseFrag, xr + 32 * m, v);
    }
    if constexpr (CODES) {
      u4v o;
#pragma unroll
      for (int p = 0; p < 4; p++) {
        const uint32_t q = W.q[p >> 1] >> (16 * (p & 1));
        const float x0 = (float)(int)(int8_t)(q & 0xff), x1 = (float)(int)(int8_t)((q >> 8) & 0xff);
        o[p] = __builtin_amdgcn_perm(__float_as_uint(x1), __float_as_uint(x0), 0x07060302u);  // |code| <= 128: exact
      }
      SW[(cr >> 4) * WS + dense_slot(cr & 15, c8)] = o;
      if (tid < 64) sD[buf][tid] = W.sc[0];
    } else if constexpr (!BWD) {
#pragma unroll
      for (int m = 0; m < 2; m++) put4(SW, WS, xr + 32 * m, W.v[m]);
    } else {
      // column 4 li + e: tile li / 4, row 4 (li % 4) + e of k-group w, word g
      uint32_t* p = reinterpret_cast<uint32_t*>(SW + (li >> 2) * WS + 4 * (li & 3) + 16 * w) + g;
#pragma unroll
      for (int e = 0; e < 4; e++) {
        float x0, x1;
        if constexpr (Q8) {
          x0 = W.sc[0] * (float)(int)(int8_t)((W.q.x >> (8 * e)) & 0xff);
          x1 = W.sc[1] * (float)(int)(int8_t)((W.q.y >> (8 * e)) & 0xff);
        } else {
          x0 = W.v[0][e];
          x1 = W.v[1][e];
        }
        uint32_t h, m, l;
        split3(x0, x1, h, m, l);
        const int se = 4 * (e ^ w);  // dense_slot(4 (li % 4) + e, w)
        p[se] = h;
        p[se + 4 * kDenseFrag] = m;
        p[se + 8 * kDenseFrag] = l;
      }
    }
  };
  struct Frags {
    bf8 x[WT][3], w[WC][PW];
    f4 d[WC];
  };
  auto load_frags = [&](int buf, Frags& F) {
    const int sl = dense_slot(li, g);
#pragma unroll
    for (int i = 0; i < WT; i++)
#pragma unroll
      for (int p = 0; p < 3; p++) F.x[i][p] = __builtin_bit_cast(bf8, lds[buf][((wt + i) * 3 + p) * kDenseFrag + sl]);
#pragma unroll
    for (int j = 0; j < WC; j++) {
#pragma unroll
      for (int p = 0; p < PW; p++) F.w[j][p] = __builtin_bit_cast(bf8, lds[buf][TT * 3 * kDenseFrag + (wc + j) * WS + p * kDenseFrag + sl]);
      if constexpr (CODES) F.d[j] = *reinterpret_cast<const f4*>(&sD[buf][16 * (wc + j) + 4 * g]);
    }
  };
  auto compute = [&](const Frags& F) {
    if constexpr (CODES) {
      f4 b[WT][WC], hi[WT][WC];
#pragma unroll
      for (int p = 2; p >= 1; p--)
#pragma unroll
        for (int j = 0; j < WC; j++)
#pragma unroll
          for (int i = 0; i < WT; i++) b[i][j] = mfma_bf16(F.w[j][0], F.x[i][p], p == 2 ? f4{0.0f, 0.0f, 0.0f, 0.0f} : b[i][j]);
#pragma unroll
      for (int j = 0; j < WC; j++)
#pragma unroll
        for (int i = 0; i < WT; i++) hi[i][j] = mfma_bf16(F.w[j][0], F.x[i][0], f4{0.0f, 0.0f, 0.0f, 0.0f});
#pragma unroll
      for (int j = 0; j < WC; j++)
#pragma unroll
        for (int i = 0; i < WT; i++)
#pragma unroll
          for (int e = 0; e < 4; e++) acc[i][j][e] = fmaf(F.d[j][e], hi[i][j][e] + b[i][j][e], acc[i][j][e]);
    } else {
      constexpr int PA[7] = {2, 1, 2, 0, 1, 1, 0}, PB[7] = {1, 2, 0, 2, 1, 0, 1};
#pragma unroll
      for (int p = 0; p < 7; p++)
#pragma unroll
        for (int j = 0; j < WC; j++)
#pragma unroll
          for (int i = 0; i < WT; i++) low[i][j] = mfma_bf16(F.w[j][PA[p]], F.x[i][PB[p]], low[i][j]);
#pragma unroll
      for (int j = 0; j < WC; j++)
#pragma unroll
        for (int i = 0; i < WT; i++) acc[i][j] = mfma_bf16(F.w[j][0], F.x[i][0], acc[i][j]);
    }
  };
  f4 X[D][NX];
  DenseSlotW<BWD, Q8> W[D];
#pragma unroll
  for (int s = 0; s < D - 1; s++) issue(X[s], W[s], s);
  stage(X[0], W[0], 0, 0);
  // step s: buffer s & 1 is staged by every wave, the other one is free (its readers passed this barrier);
  // its fragments are read, step s + 1 is staged while they arrive, then its MFMAs run.  full: a step of a
  // complete group of D (no guards; staging past the last step only writes the unused buffer)
  auto step_body = [&](int v, int s, bool full) {
    issue(X[(v + D - 1) % D], W[(v + D - 1) % D], s + D - 1);
    __builtin_amdgcn_sched_barrier(0);
    __syncthreads();
    Frags F;
    if (full || s < nsteps) load_frags(s & 1, F);
    if (full || s + 1 < nsteps) stage(X[(v + 1) % D], W[(v + 1) % D], (s + 1) & 1, s + 1);
    if (full || s < nsteps) compute(F);
    __builtin_amdgcn_sched_barrier(0);
  };
  const int nfull = nsteps / D * D;
  for (int s0 = 0; s0 < nfull; s0 += D) {
#pragma unroll
    for (int v = 0; v < D; v++) step_body(v, s0 + v, true);
  }
  if (nfull < nsteps) {
#pragma unroll
    for (int v = 0; v < D; v++) step_body(v, nfull + v, false);
  }
  bool again = false;
#pragma unroll
  for (int i = 0; i < WT; i++)
#pragma unroll
    for (int j = 0; j < WC; j++) {
      acc[i][j] += low[i][j];
#pragma unroll
      for (int e = 0; e < 4; e++) again |= dense_again(acc[i][j][e]);
    }
  // A wave with such an output sums its tiles once more on the f32 MFMA (the operands straight from memory; a step
  // of 16 elements, k-group g taking 4 g .. + 3) and takes those outputs.  One lane per output took some
  // hundred times as long where a whole activation is NaN
  if (__ballot(again) != 0) {
    f4 full[WT][WC];
#pragma unroll
    for (int i = 0; i < WT; i++)
#pragma unroll
      for (int j = 0; j < WC; j++) full[i][j] = f4{0.0f, 0.0f, 0.0f, 0.0f};
    for (int c = c0; c < c1; c += 16) {
      f4 xv[WT], wv[WC];
#pragma unroll
      for (int i = 0; i < WT; i++)
#pragma unroll
        for (int e = 0; e < 4; e++) {
          const uint32_t o = ((uint32_t)min(t0 + 16 * (wt + i) + li, a.T) * C + 4 * g + e) * 4u;
          const float v = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rx, o, (uint32_t)c * 4u, 0));
          xv[i][e] = c + 4 * g + e < C ? v : 0.0f;  // elements past C hold the next row's
        }
#pragma unroll
      for (int j = 0; j < WC; j++)
#pragma unroll
        for (int e = 0; e < 4; e++) {
          const int o = o0 + 16 * (wc + j) + li, ce = c + 4 * g + e;
          const uint32_t n = min(BWD ? ce : o, a.N), k = BWD ? min(o, a.K - 1) : ce;  // row N: past the end, zeros
          if constexpr (Q8) {
            const int q = (int8_t)__builtin_amdgcn_raw_buffer_load_b8(rw, n * a.K + k, 0, 0);
            wv[j][e] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rs, (n * (a.K / 32) + (k >> 5)) * 4u, 0, 0)) * (float)q;
          } else {
            wv[j][e] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rw, (n * a.K + k) * 4u, 0, 0));
          }
        }
#pragma unroll
      for (int e = 0; e < 4; e++)
#pragma unroll
        for (int i = 0; i < WT; i++)
#pragma unroll
          for (int j = 0; j < WC; j++) full[i][j] = mfma_f32(wv[j][e], xv[i][e], full[i][j]);
    }
#pragma unroll
    for (int i = 0; i < WT; i++)
#pragma unroll
      for (int j = 0; j < WC; j++)
#pragma unroll
        for (int e = 0; e < 4; e++) acc[i][j][e] = dense_again(acc[i][j][e]) ? full[i][j][e] : acc[i][j][e];
  }

  // the adapter's part, 32 ranks at a time: forward s h B^T, h summed from its slice partials; backward
  // (the first split) g A, g likewise
  f4 lacc[WT][WC];
#pragma unroll
  for (int i = 0; i < WT; i++)
#pragma unroll
    for (int j = 0; j < WC; j++) lacc[i][j] = f4{0.0f, 0.0f, 0.0f, 0.0f};
  const bool lora = BWD ? a.gp != nullptr && z == 0 : a.hp != nullptr;
  if (lora) {
    constexpr int LR = 33, NR = 64 + 16 * TT;
    static_assert(NR * LR * 4 <= sizeof(lds), "LoRA operands fit the operand buffers");
    float* sh = reinterpret_cast<float*>(&lds[0][0]);  // [16 TT][LR]
    float* sb = sh + 16 * TT * LR;                     // [64][LR]
    for (int j0 = 0; j0 < a.r; j0 += 32) {
      __syncthreads();
      for (int e = tid; e < NR * 32; e += 256) {  // consecutive threads: ranks (forward), rows (backward)
        const int row = BWD ? e % NR : e >> 5, jl = BWD ? e / NR : e & 31, j = j0 + jl, o = o0 + row - 16 * TT;
        float v = 0.0f;
        if (j < a.r) {
          if (row >= 16 * TT) {
            if (o < O) v = a.lb[BWD ? (int64_t)j * O + o : (int64_t)o * a.r + j];
          } else if (t0 + row < a.T) {
            const int64_t i = (int64_t)(t0 + row) * a.r + j;
            v = BWD ? sum_slices(a.gp, i, a.ngq, (int64_t)a.T * a.r) : sum_partials(a.hp, i, a.nhp);
          }
        }
        sh[row * LR + jl] = v;
      }
      __syncthreads();
      for (int k = 0; k < 32 && j0 + k < a.r; k += 4) {
        float bv[WC], hv[WT];
#pragma unroll
        for (int j = 0; j < WC; j++) bv[j] = sb[(16 * (wc + j) + li) * LR + k + g];
#pragma unroll
        for (int i = 0; i < WT; i++) hv[i] = sh[(16 * (wt + i) + li) * LR + k + g];
#pragma unroll
        for (int i = 0; i < WT; i++)
#pragma unroll
          for (int j = 0; j < WC; j++) lacc[i][j] = mfma_f32(bv[j], hv[i], lacc[i][j]);
      }
    }
  }
  // lane (token li, g): outputs 4g .. 4g + 3 of the tile
  float* out = a.out + (BWD ? (int64_t)z * a.T * O : 0);
#pragma unroll
  for (int i = 0; i < WT; i++) {
    const int t = t0 + 16 * (wt + i) + li;
    if (t >= a.T) continue;
#pragma unroll
    for (int j = 0; j < WC; j++) {
      const int o = o0 + 16 * (wc + j) + 4 * g;
      float* p = out + (int64_t)t * O + o;
      f4 v = acc[i][j];
#pragma unroll
      for (int e = 0; e < 4; e++) {
        if (!BWD && a.bias) v[e] += a.bias[min(o + e, O - 1)];
        if (lora) v[e] += a.s * lacc[i][j][e];
        if (BWD && a.accumulate && o + e < O) v[e] = p[e] + v[e];
      }
      if ((O & 3) == 0 && o < O) {
        *reinterpret_cast<f4*>(p) = v;
      } else {
#pragma unroll
        for (int e = 0; e < 4; e++)
          if (o + e < O) p[e] = v[e];
      }
    }
  }
}

extern "C" __global__ __launch_bounds__(256) void rtq_dense_fwd32(DenseGemmArgs a) { dense_tile<false, false, 2>(a); }
extern "C" __global__ __launch_bounds__(256) void rtq_dense_fwd32_q8(DenseGemmArgs a) { dense_tile<false, true, 2>(a); }
extern "C" __global__ __launch_bounds__(256) void rtq_dense_fwd64(DenseGemmArgs a) { dense_tile<false, false, 4>(a); }
extern "C" __global__ __launch_bounds__(256) void rtq_dense_fwd64_q8(DenseGemmArgs a) { dense_tile<false, true, 4>(a); }
extern "C" __global__ __launch_bounds__(256) void rtq_dense_bwd32(DenseGemmArgs a) { dense_tile<true, false, 2>(a); }
extern "C" __global__ __launch_bounds__(256) void rtq_dense_bwd32_q8(DenseGemmArgs a) { dense_tile<true, true, 2>(a); }
extern "C" __global__ __launch_bounds__(256) void rtq_dense_bwd64(DenseGemmArgs a) { dense_tile<true, false, 4>(a); }
extern "C" __global__ __launch_bounds__(256) void rtq_dense_bwd64_q8(DenseGemmArgs a) { dense_tile<true, true, 4>(a); }
