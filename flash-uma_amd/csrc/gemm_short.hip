// The SO(2) convolution pair (model.py:150-154) of a block on few edges: every contraction of
// conv1 + gate + conv2, or of their input gradients, in three launches.
//
// With few edges the tiled kernels of gemm.hip and cgemm.hip are bound by one workgroup's
// latency, not by the chip: 29 atoms give 7 to 42 workgroups on 256 CUs, each walking its K loop
// chunk by chunk (one 16-wide chunk of loads in flight, a split, two LDS trips and a barrier:
// 0.84 us a chunk).  Here
//  * a workgroup owns a 32 x 64 output tile (32 x 32 complex values), so that few rows still give
//    many workgroups, and its 4 waves split K between them: wave w takes chunks w nk / 4 ..
//    (w + 1) nk / 4 - 1 of the same tile.  No wave waits for another inside the loop: each loads
//    its fragments of A (fp32, 8 consecutive k of a row per lane, the MFMA operand layout) and of
//    the pre-split weight (fu_linear_weight_split, fu_complex_weight_split) straight into
//    registers, the next segment's in flight.  At most 168 VGPRs: three workgroups per CU;
//  * a row's power-of-two scale is the exact one of its first nonzero segment, with one bit of
//    headroom, lowered (and the accumulators with it) when a later segment would overflow: no pass
//    over the row beforehand.  The window rule of split_f16.h is applied per segment, to runs of 4
//    elements, against the weight's precomputed flags; a segment that fails it runs the products of
//    pass 2.  Small runs elsewhere in the row do not reach a segment's verdict, so a weight's own runs
//    below the window always do (bit 0 of its flags);
//  * the four partial tiles are summed once, in LDS, in wave order (bitwise reproducible), and the
//    epilogues are those of the tiled kernels;
//  * the column tiles of a row tile go to one XCD (its L2 then reads those rows of A once).
// The independent contractions of one stage share a launch (conv1 m = 1 and 2; conv2 m = 0, 1, 2;
// the three conv1 input gradients), so a pair takes three launches forward and three backward.
//
// Measured, us for forward / backward (captured launches; tiled kernels -> this), C = 128, lmax 2:
// 859 edges 171 / 161 -> 40 / 40, 3,000 edges 168 / 160 -> 80 / 81, 6,000 edges 174 / 180 -> 141 /
// 141, 12,000 edges 211 / 248 -> 270 / 279.  Past the small sizes the operand traffic through the
// L2s bounds it (270 KB per edge at a 32 x 64 tile, 11 TB/s): 8 waves of K / 8 (one workgroup per
// CU) took 50 / 51 and 124 / 137 us at 859 and 3,000 edges, 64 x 64 tiles 45 / 45 and 98 / 95, and
// tiles dealt over all XCDs 41 / 39 and 90 / 86.
#include "split_f16.h"

namespace fu {
namespace sg {

constexpr int NW = 4;           // waves per workgroup: the K split
constexpr int TR = 32;          // tile rows
constexpr int ES = 64 + 8;      // floats per row of a wave's partial tile: 4 ES = 32 mod 64 banks
constexpr int RSEG = 2;         // chunks per segment of the real products

// One contraction of a launch: Y = A W^T on 64 n_tiles real columns, or the complex
// product on 32 n_tiles columns of [real | imaginary].
struct Prob {
  const float* A;       // real rows, or the real parts
  const float* Ai;      // imaginary parts (complex)
  int64_t lda;
  const uint4* W;       // fp16 fragments of the pre-split weight
  const float* cinv;    // its columns' unscale factors
  const int* flags;     // real: the summary word; complex: one word per column
  int32_t nk;           // 16-wide K chunks
  int32_t n_tiles;      // column tiles
  int32_t first;        // first workgroup of this contraction
  int32_t cplx;
  const float* bias;    // real, or null
  float* Y;             // output, or its real parts
  float* Yi;
  int64_t ldy;
  float* Z;             // gated copy (MODE 1), or the gate sums (MODE 2, complex)
  float* Zi;
  int64_t ldz;
  const float* G;       // gate-paired conv1 m = 0 output Y0 (gate source)
  int64_t ldg;
  const float* F;       // MODE 2, complex: forward pre-activation; real: gate sums of m = 1
  const float* Fi;      // MODE 2, complex: its imaginary parts; real: gate sums of m = 2
  int64_t ldf;
  int64_t ldfi;
  int32_t s_off;        // gate column offset (complex)
};

struct Group {
  Prob p[3];
  int32_t count;
  int64_t M;
  int32_t C;
  int32_t L;
};

__device__ __forceinline__ float4 zero4() { return make_float4(0.f, 0.f, 0.f, 0.f); }
__device__ __forceinline__ float4 sigmoid4(const float4& v) {
  return make_float4(sigmoidf_(v.x), sigmoidf_(v.y), sigmoidf_(v.z), sigmoidf_(v.w));
}

// Running power-of-two scale of a lane's row (lane r and r ^ 32 hold the same row).  The first
// nonzero segment sets it so that the segment's largest magnitude lies in [2^13, 2^14); a later
// segment that would overflow lowers it, and the accumulators of that row with it.
struct RowScale {
  int e = 0;
  bool set = false;
  // returns the factor the row's accumulators take (1 unless the scale was lowered)
  __device__ __forceinline__ float update(float R) {
    R = fmaxf(R, __shfl_xor(R, 32));
    const int en = f16_exp_row(R) - 1;
    const bool lower = set && !(R * pow2i(e) < 60000.0f);
    const int d = lower ? (en - e < -126 ? -126 : en - e) : 0;
    if (R > 0.0f && (!set || lower)) {
      e = en < -126 ? -126 : en;
      set = true;
    }
    return pow2i(d);
  }
};

// Factors of a lane's 16 accumulator rows (8 (r / 4) + 4 fh + r % 4); lane `row` holds its row's.
__device__ __forceinline__ void row_factors(float v, int fh, float (&rs)[16]) {
#pragma unroll
  for (int r = 0; r < 16; ++r) rs[r] = __shfl(v, 8 * (r >> 2) + 4 * fh + (r & 3));
}
__device__ __forceinline__ floatx16 zero16() {
  floatx16 z;
#pragma unroll
  for (int r = 0; r < 16; ++r) z[r] = 0.0f;
  return z;
}
// split2h with the lo pieces times a power of two (1, or 2^11: pass 2 of split_f16.h)
__device__ __forceinline__ void split2h_by(const float4& a, const float4& b, float up, uint4& H, uint4& L) {
  const float x[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
#pragma unroll
  for (int t = 0; t < 4; ++t) {
    const float2v v = {x[2 * t], x[2 * t + 1]};
    const f16x2 h = __builtin_convertvector(v, f16x2);
    const float2v r = (v - __builtin_convertvector(h, float2v)) * up;
    (&H.x)[t] = __builtin_bit_cast(unsigned, h);
    (&L.x)[t] = __builtin_bit_cast(unsigned, __builtin_convertvector(r, f16x2));
  }
}
__device__ __forceinline__ f16x8 frag(const uint4& v) { return __builtin_bit_cast(f16x8, v); }
__device__ __forceinline__ int wave_id() { return __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)); }

// This wave's partial 32 x (32 NB) tile of a real contraction, unscaled, into red (rows of STR
// floats), the K range split over W waves.
template <int W, int NB, int STR>
__device__ __forceinline__ void real_part(const Prob& p, int64_t row0, int n_tile, int64_t M, float* red) {
  constexpr int S = RSEG;
  const int lane = threadIdx.x & 63, wave = wave_id();
  const int fr = lane & 31, fh = lane >> 5;
  const int c0 = wave * p.nk / W, c1 = (wave + 1) * p.nk / W;
  const int64_t row = row0 + fr < M ? row0 + fr : M - 1;   // a row past M: nothing of it is stored
  const float* pa = p.A + row * p.lda + 8 * fh;
  const uint4* wb = p.W + (int64_t)(NB * n_tile) * p.nk * 192 + lane;
  const int64_t wj = (int64_t)p.nk * 192;
  const int wbits = p.flags[0];
  const int last = c1 > c0 ? c1 - 1 : 0;
  // chunk k0 + s of a segment, the last one repeated past the wave's range (not multiplied)
  auto chunk = [&](int k0, int s) { return k0 + s < c1 ? k0 + s : last; };
  float4 raw[S][2];
  uint4 bh[S][NB], bl[S][NB];   // hi, lo fragments of the 32-column blocks
  auto load_a = [&](int k0) {
#pragma unroll
    for (int s = 0; s < S; ++s) {
      raw[s][0] = ld4(pa + 16 * chunk(k0, s));
      raw[s][1] = ld4(pa + 16 * chunk(k0, s) + 4);
    }
  };
  auto load_b = [&](int k0) {
#pragma unroll
    for (int s = 0; s < S; ++s)
#pragma unroll
      for (int j = 0; j < NB; ++j) {
        bh[s][j] = wb[j * wj + (int64_t)chunk(k0, s) * 192];
        bl[s][j] = wb[j * wj + (int64_t)chunk(k0, s) * 192 + 64];
      }
  };
  floatx16 acc[NB];
#pragma unroll
  for (int j = 0; j < NB; ++j) acc[j] = zero16();
  RowScale sc;
  load_a(c0);
  load_b(c0);
  for (int k0 = c0; k0 < c1; k0 += S) {
    float m[S], R = 0.0f;
#pragma unroll
    for (int s = 0; s < S; ++s) {
      m[s] = amax8(raw[s][0], raw[s][1]);
      R = fmaxf(R, m[s]);
    }
    const float fac = sc.update(R), f = pow2i(sc.e);
    if (__any(fac != 1.0f)) {
      float rs[16];
      row_factors(fac, fh, rs);
#pragma unroll
      for (int j = 0; j < NB; ++j)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[j][r] *= rs[r];
    }
    // The window rule of split_f16.h (a weight with a piece below its window always takes pass 2).
    // Pass 2: the residual planes hold 2^11 times the residuals, whose products are added to
    // accumulators scaled up by as much (exact), and scaled down again before hi * hi.
    bool two = (wbits & 1) != 0;
    if (wbits & 2) {
      bool low = false;
#pragma unroll
      for (int s = 0; s < S; ++s)
#pragma unroll
        for (int h = 0; h < 2; ++h) low = low || f16_lossy(amax4(raw[s][h]) * f);
      two = two || __any(low);
    }
    if (two) {
#pragma unroll
      for (int j = 0; j < NB; ++j) {
        acc[j] *= F16_LO_UP;
#pragma unroll
        for (int s = 0; s < S; ++s) bl[s][j] = wb[j * wj + (int64_t)chunk(k0, s) * 192 + 128];
      }
    }
    uint4 ah[S], al[S];
    const float up = two ? F16_LO_UP : 1.0f;
#pragma unroll
    for (int s = 0; s < S; ++s) split2h_by(scale4(raw[s][0], f), scale4(raw[s][1], f), up, ah[s], al[s]);
    if (k0 + S < c1) load_a(k0 + S);
#pragma unroll
    for (int s = 0; s < S; ++s)
      if (k0 + s < c1) {
#pragma unroll
        for (int q = 0; q < 2; ++q)
#pragma unroll
          for (int j = 0; j < NB; ++j)
            acc[j] = mfma_f16(frag(q == 0 ? al[s] : ah[s]), frag(q == 1 ? bl[s][j] : bh[s][j]), acc[j]);
      }
    if (two) {
#pragma unroll
      for (int j = 0; j < NB; ++j) acc[j] *= F16_LO_DOWN;
    }
#pragma unroll
    for (int s = 0; s < S; ++s)
      if (k0 + s < c1) {
#pragma unroll
        for (int j = 0; j < NB; ++j) acc[j] = mfma_f16(frag(ah[s]), frag(bh[s][j]), acc[j]);
      }
    if (k0 + S < c1) load_b(k0 + S);
  }
  float* ws = red + wave * TR * STR;
  float rs[16];
  row_factors(pow2i(-sc.e), fh, rs);
#pragma unroll
  for (int j = 0; j < NB; ++j) {
    const float cs = p.cinv[32 * NB * n_tile + 32 * j + fr];
#pragma unroll
    for (int r = 0; r < 16; ++r) ws[(8 * (r >> 2) + 4 * fh + (r & 3)) * STR + 32 * j + fr] = acc[j][r] * rs[r] * cs;
  }
}

// This wave's partial 32 x (32 | 32) tile of a complex contraction (three products, out_r =
// T1 - T2, out_i = T3 - T1 - T2; cgemm.hip), unscaled, into red: one chunk at a time, the next
// chunk's operands in flight.
__device__ __forceinline__ void complex_part(const Prob& p, int64_t row0, int n_tile, int64_t M, float* red) {
  const int lane = threadIdx.x & 63, wave = wave_id();
  const int fr = lane & 31, fh = lane >> 5;
  const int c0 = wave * p.nk / NW, c1 = (wave + 1) * p.nk / NW;
  const int64_t row = row0 + fr < M ? row0 + fr : M - 1;
  const float *pr = p.A + row * p.lda + 8 * fh, *pi = p.Ai + row * p.lda + 8 * fh;
  const uint4* wb = p.W + (int64_t)n_tile * p.nk * 576 + lane;
  const int cf = p.flags[32 * n_tile + fr];
  const bool lowW = __any(cf & 1) != 0, roughW = __any(cf & 2) != 0;
  float4 xr[2], xi[2];
  uint4 b[3][2];   // P, Q, S: hi, lo
  auto load_a = [&](int kc) {
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      xr[h] = ld4(pr + 16 * kc + 4 * h);
      xi[h] = ld4(pi + 16 * kc + 4 * h);
    }
  };
  auto load_b = [&](int kc, int op) {
    b[op][0] = wb[(int64_t)kc * 576 + 128 * op];
    b[op][1] = wb[(int64_t)kc * 576 + 128 * op + 64];
  };
  floatx16 T[3] = {zero16(), zero16(), zero16()};
  RowScale sc;
  if (c0 < c1) {
    load_a(c0);
#pragma unroll
    for (int op = 0; op < 3; ++op) load_b(c0, op);
  }
  for (int kc = c0; kc < c1; ++kc) {
    const float mr = amax8(xr[0], xr[1]), mi = amax8(xi[0], xi[1]);
    const float fac = sc.update(fmaxf(fmaxf(mr, mi), amax8(xr[0] + xi[0], xr[1] + xi[1]))), f = pow2i(sc.e);
    if (__any(fac != 1.0f)) {
      float rs[16];
      row_factors(fac, fh, rs);
#pragma unroll
      for (int op = 0; op < 3; ++op)
#pragma unroll
        for (int r = 0; r < 16; ++r) T[op][r] *= rs[r];
    }
    // pieces of 4 of a_r and of a_i, as in the tiled kernel: a run of 4 below the window next to
    // normal elements counts
    bool two = lowW;
    if (roughW) {
      bool low = false;
#pragma unroll
      for (int h = 0; h < 2; ++h) low = low || f16_lossy(amax4(xr[h]) * f) || f16_lossy(amax4(xi[h]) * f);
      two = two || __any(low);
    }
    if (two) {   // pass 2 of split_f16.h, as in real_part
#pragma unroll
      for (int op = 0; op < 3; ++op) {
        T[op] *= F16_LO_UP;
        b[op][1] = wb[(int64_t)kc * 576 + 384 + 64 * op];
      }
    }
    uint4 h[3], l[3];   // a_r, a_i, a_r + a_i
    const float up = two ? F16_LO_UP : 1.0f;
    split2h_by(scale4(xr[0], f), scale4(xr[1], f), up, h[0], l[0]);
    split2h_by(scale4(xi[0], f), scale4(xi[1], f), up, h[1], l[1]);
    split2h_by(scale4(xr[0] + xi[0], f), scale4(xr[1] + xi[1], f), up, h[2], l[2]);
    const int kn = kc + 1 < c1 ? kc + 1 : kc;
    load_a(kn);
#pragma unroll
    for (int q = 0; q < 2; ++q)
#pragma unroll
      for (int op = 0; op < 3; ++op) T[op] = mfma_f16(frag(q == 0 ? l[op] : h[op]), frag(b[op][q]), T[op]);
    if (two) {
#pragma unroll
      for (int op = 0; op < 3; ++op) T[op] *= F16_LO_DOWN;
    }
#pragma unroll
    for (int op = 0; op < 3; ++op) {
      T[op] = mfma_f16(frag(h[op]), frag(b[op][0]), T[op]);
      load_b(kn, op);
    }
  }
  float* ws = red + wave * TR * ES;
  const float cs = p.cinv[32 * n_tile + fr];
  float rs[16];
  row_factors(pow2i(-sc.e), fh, rs);
#pragma unroll
  for (int r = 0; r < 16; ++r) {
    float* o = ws + (8 * (r >> 2) + 4 * fh + (r & 3)) * ES + fr;
    const float f = rs[r] * cs;
    o[0] = (T[0][r] - T[1][r]) * f;
    o[32] = (T[2][r] - T[0][r] - T[1][r]) * f;
  }
}

// Sum of the waves' partial values at (row, c .. c + 3), in wave order.
template <int W = NW, int STR = ES>
__device__ __forceinline__ float4 sum_parts(const float* red, int row, int c) {
  float4 v = ld4(red + row * STR + c);
#pragma unroll
  for (int w = 1; w < W; ++w) v = v + ld4(red + (w * TR + row) * STR + c);
  return v;
}

// The tile of a contraction's workgroup blk.  Workgroups are dealt round-robin over the 8 XCDs, so
// every column tile of a row tile goes to one XCD, whose L2 then fetches those rows of A once;
// row tiles are padded to a multiple of 8 (false: nothing to do).
__device__ __forceinline__ bool tile_of(const Prob& p, const Group& g, int blk, int64_t& row0, int& n_tile) {
  const int q = blk >> 3;
  n_tile = q % p.n_tiles;
  row0 = (int64_t)(q / p.n_tiles * 8 + (blk & 7)) * TR;
  return row0 < g.M;
}

// Epilogues on a summed tile, as in gemm.hip (MODE 0, 1, 2) and cgemm.hip.
template <int MODE>
__device__ __forceinline__ void real_tile(const Prob& p, const Group& g, int blk, float* red) {
  int64_t row0;
  int n_tile;
  if (!tile_of(p, g, blk, row0, n_tile)) return;
  const int col0 = 64 * n_tile;
  const int C = g.C, n1 = C / 32, L = g.L;
  real_part<NW, 2, ES>(p, row0, n_tile, g.M, red);
  // MODE 1: a thread takes (row, 4 + 4 columns of the gate pair); otherwise (row, 4 columns)
  constexpr int Q = MODE == 1 ? 8 : 16, IT = TR * Q / (64 * NW);
  const int c = (threadIdx.x % Q) * 4;
  const int kb = col0 / C, ch = col0 + c - kb * C;   // MODE 2: degree block and channel
  const int gate_col = 64 * ((kb - 1) * n1 + (ch >> 5)) + (ch & 31);
  // the epilogue's global operands, loaded while the other waves finish
  float4 gp[IT], y[IT], q[IT];
#pragma unroll
  for (int it = 0; it < IT; ++it) {
    gp[it] = y[it] = q[it] = zero4();
    const int64_t row = row0 + threadIdx.x / Q + it * (64 * NW / Q);
    const int64_t rc = row < g.M ? row : g.M - 1;
    if constexpr (MODE == 2) {
      const float* y0 = p.G + rc * p.ldg;
      if (kb == 0) {
        y[it] = ld4(y0 + 2 * L * C + ch);
      } else {
        gp[it] = ld4(y0 + gate_col);
        y[it] = ld4(y0 + gate_col + 32);
        q[it] = ld4(p.F + rc * p.ldf + (kb - 1) * C + ch);
        if (kb >= 2) q[it] = q[it] + ld4(p.Fi + rc * p.ldfi + (kb - 2) * C + ch);
      }
    } else if (p.bias) {
      gp[it] = ld4(p.bias + col0 + c);
      if constexpr (MODE == 1) y[it] = ld4(p.bias + col0 + 32 + c);
    }
  }
  __syncthreads();
#pragma unroll
  for (int it = 0; it < IT; ++it) {
    const int r = threadIdx.x / Q + it * (64 * NW / Q);
    const int64_t row = row0 + r;
    if (row >= g.M) continue;
    if constexpr (MODE == 0) {
      float4 v = sum_parts(red, r, c);
      if (p.bias) v = v + gp[it];
      st4(p.Y + row * p.ldy + col0 + c, v);
    } else if constexpr (MODE == 1) {
      const float4 a = sum_parts(red, r, c) + gp[it], v = sum_parts(red, r, 32 + c) + y[it];
      st4(p.Y + row * p.ldy + col0 + c, a);
      st4(p.Y + row * p.ldy + col0 + 32 + c, v);
      if (n_tile < L * n1) {
        const int kind = n_tile / n1;
        st4(p.Z + row * p.ldz + (1 + kind) * C + 32 * (n_tile - kind * n1) + c, v * sigmoid4(a));
      } else {
        float* z = p.Z + row * p.ldz + col0 - 2 * L * C + c;
        st4(z, a * sigmoid4(a));
        st4(z + 32, v * sigmoid4(v));
      }
    } else {
      const float4 v = sum_parts(red, r, c);
      float* out = p.Y + row * p.ldy;
      if (kb == 0) {
        float4 o;
#pragma unroll
        for (int t = 0; t < 4; ++t) {
          const float yt = (&y[it].x)[t], sl = sigmoidf_(yt);
          (&o.x)[t] = (&v.x)[t] * (sl + yt * (sl * (1.0f - sl)));
        }
        st4(out + 2 * L * C + ch, o);
      } else {
        float4 og, ov;
#pragma unroll
        for (int t = 0; t < 4; ++t) {
          const float st = sigmoidf_((&gp[it].x)[t]), gt = (&v.x)[t];
          (&ov.x)[t] = gt * st;
          (&og.x)[t] = (st * (1.0f - st)) * (gt * (&y[it].x)[t] + (&q[it].x)[t]);
        }
        st4(out + gate_col, og);
        st4(out + gate_col + 32, ov);
      }
    }
  }
}

template <int MODE>
__device__ __forceinline__ void complex_tile(const Prob& p, const Group& g, int blk, float* red) {
  int64_t row0;
  int n_tile;
  if (!tile_of(p, g, blk, row0, n_tile)) return;
  complex_part(p, row0, n_tile, g.M, red);
  constexpr int IT = TR * 8 / (64 * NW), RS = 64 * NW / 8;
  const int c = (threadIdx.x & 7) * 4, gc = 32 * n_tile + c;
  float4 gp[IT], fre[IT], fim[IT];
  if constexpr (MODE != 0) {
    const int t = p.s_off + gc, l1 = t / g.C, ch = t - l1 * g.C;
    const int gate_col = 64 * (l1 * (g.C >> 5) + (ch >> 5)) + (ch & 31);
#pragma unroll
    for (int it = 0; it < IT; ++it) {
      const int64_t row = row0 + (threadIdx.x >> 3) + it * RS;
      const int64_t rc = row < g.M ? row : g.M - 1;
      gp[it] = ld4(p.G + rc * p.ldg + gate_col);
      if constexpr (MODE == 2) {
        fre[it] = ld4(p.F + rc * p.ldf + gc);
        fim[it] = ld4(p.Fi + rc * p.ldf + gc);
      }
    }
  }
  __syncthreads();
#pragma unroll
  for (int it = 0; it < IT; ++it) {
    const int r = (int)(threadIdx.x >> 3) + it * RS;
    const int64_t row = row0 + r;
    if (row >= g.M) continue;
    const float4 yr = sum_parts(red, r, c), yi = sum_parts(red, r, 32 + c);
    if constexpr (MODE == 2) {
      const float4 s = sigmoid4(gp[it]);
      st4(p.Y + row * p.ldy + gc, yr * s);
      st4(p.Yi + row * p.ldy + gc, yi * s);
      st4(p.Z + row * p.ldz + gc, yr * fre[it] + yi * fim[it]);
    } else {
      st4(p.Y + row * p.ldy + gc, yr);
      st4(p.Yi + row * p.ldy + gc, yi);
      if constexpr (MODE == 1) {
        const float4 s = sigmoid4(gp[it]);
        st4(p.Z + row * p.ldz + gc, yr * s);
        st4(p.Zi + row * p.ldz + gc, yi * s);
      }
    }
  }
}

// KIND 0: real contractions, 1: complex, 2: both in one launch.
template <int MODE, int KIND>
__global__ __launch_bounds__(64 * NW, 3) void short_kernel(const Group g) {
  __shared__ __attribute__((aligned(16))) float red[NW * TR * ES];
  int b = (int)blockIdx.x, k = 0;
  if (g.count > 1 && b >= g.p[1].first) k = 1;
  if (g.count > 2 && b >= g.p[2].first) k = 2;
  const Prob& p = k == 0 ? g.p[0] : k == 1 ? g.p[1] : g.p[2];
  b -= p.first;
  if constexpr (KIND == 0) {
    real_tile<MODE>(p, g, b, red);
  } else if constexpr (KIND == 1) {
    complex_tile<MODE>(p, g, b, red);
  } else {
    if (p.cplx) complex_tile<MODE>(p, g, b, red);
    else real_tile<MODE>(p, g, b, red);
  }
}

// A radial output layer's input gradient with the LayerNorm-SiLU backward of its group in the
// epilogue (MODE 5 of gemm.hip: the product is the output gradient, the LayerNorm input x is read),
// on few rows: a workgroup owns 32 whole 128-column rows and 8 waves split K (1,536 at lmax 2, C =
// 128), whose 96 chunks a workgroup of the tiled kernel walks one by one however few rows there
// are: 870 rows 61 -> 19 us, 9,000 rows 77 -> 40 (alone).  Bound by each workgroup's read of the
// whole weight (786 KB at 64 bytes a cycle, 6 us) and its start and end.
constexpr int LW = 8, LES = 128 + 8;
struct LnBwd {
  const float* x;
  int64_t ldx;
  const float* gamma;
  const float* beta;
  const float* mean;
  const float* rstd;
  int32_t G;   // row stride of mean and rstd
};
__global__ __launch_bounds__(64 * LW, 2) void short_ln_bwd_kernel(const Prob p, const LnBwd ln, int64_t M) {
  __shared__ __attribute__((aligned(16))) float red[LW * TR * LES];
  const int64_t row0 = (int64_t)blockIdx.x * TR;
  real_part<LW, 4, LES>(p, row0, 0, M, red);
  constexpr int IT = TR * 32 / (64 * LW), RS = 2 * LW;   // rows at a time: 32 lanes each
  const int c = (threadIdx.x & 31) * 4;
  const float4 gm = ld4(ln.gamma + c), bt = ld4(ln.beta + c);
  float4 x[IT];
  float mu[IT], rs[IT];
#pragma unroll
  for (int it = 0; it < IT; ++it) {
    const int64_t row = row0 + (threadIdx.x >> 5) + it * RS;
    const int64_t rc = row < M ? row : M - 1;
    x[it] = ld4(ln.x + rc * ln.ldx + c);
    mu[it] = ln.mean[rc * ln.G];
    rs[it] = ln.rstd[rc * ln.G];
  }
  __syncthreads();
#pragma unroll
  for (int it = 0; it < IT; ++it) {
    const int r = (int)(threadIdx.x >> 5) + it * RS;
    const float4 go = sum_parts<LW, LES>(red, r, c);
    float xh[4], gx[4], s1 = 0.0f, s2 = 0.0f;
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      xh[t] = ((&x[it].x)[t] - mu[it]) * rs[it];
      const float y = xh[t] * (&gm.x)[t] + (&bt.x)[t], sg = sigmoidf_(y);
      gx[t] = (&go.x)[t] * (sg + y * sg * (1.0f - sg)) * (&gm.x)[t];
      s1 += gx[t];
      s2 += gx[t] * xh[t];
    }
    s1 = group_sum<32>(s1);
    s2 = group_sum<32>(s2);
    if (row0 + r < M) {
      float4 o;
#pragma unroll
      for (int t = 0; t < 4; ++t) (&o.x)[t] = rs[it] * (gx[t] - (s1 + xh[t] * s2) / 128.0f);
      st4(p.Y + (row0 + r) * p.ldy + c, o);
    }
  }
}

template <int MODE, int KIND>
static void launch(Group& g, int count, hipStream_t st) {
  const int m_tiles = (int)((g.M + TR - 1) / TR + 7) / 8 * 8;
  int total = 0;
  for (int k = 0; k < count; ++k) {
    g.p[k].first = total;
    total += m_tiles * g.p[k].n_tiles;
  }
  g.count = count;
  const dim3 grid((unsigned)total), block(64 * NW);
  hipLaunchKernelGGL((short_kernel<MODE, KIND>), grid, block, 0, st, g);
}

// Fragments, column factors and flags of a pre-split real weight (N, K) / complex (Nc, Kc).
static void real_weight(Prob& p, const void* W2, int32_t N, int32_t K) {
  p.W = static_cast<const uint4*>(W2);
  p.cinv = reinterpret_cast<const float*>(p.W + resident_frag_vectors(N, K));
  p.flags = reinterpret_cast<const int*>(p.cinv + resident_cols(N)) + resident_cols(N);
  p.nk = K / 16;
  p.n_tiles = N / 64;
  p.cplx = 0;
}
static void complex_weight(Prob& p, const void* W3, int32_t Nc, int32_t Kc) {
  const int64_t planes = (int64_t)(Nc / 32) * (Kc / 16) * 9 * 64;   // bf16 planes, then the fp16 ones
  p.W = static_cast<const uint4*>(W3) + planes;
  p.cinv = reinterpret_cast<const float*>(p.W + planes);
  p.flags = reinterpret_cast<const int*>(p.cinv + Nc);
  p.nk = Kc / 16;
  p.n_tiles = Nc / 32;
  p.cplx = 1;
}

// Shared checks; 1 when there is nothing to do.
static int pair_check(const char* who, int64_t E, int32_t C, int32_t L, const void* const* ptrs, int n) {
  if (E < 0 || E > (1 << 24)) return set_error(FU_ERR_SHAPE, "%s: E=%lld outside [0, 2^24]", who, (long long)E);
  if (C <= 0 || C % 64 != 0 || C > 256) return set_error(FU_ERR_UNSUPPORTED, "%s: C=%d must be 64, 128, 192 or 256", who, C);
  if (L < 2 || L > 4) return set_error(FU_ERR_UNSUPPORTED, "%s: lmax=%d unsupported (2, 3 or 4)", who, L);
  if (matmul_mode() != FU_MATMUL_SPLIT_F16)
    return set_error(FU_ERR_UNSUPPORTED, "%s: only in the split-fp16 matrix-core mode", who);
  if (E == 0) return 1;
  for (int k = 0; k < n; ++k) {
    if (!ptrs[k]) return set_error(FU_ERR_NULL, "%s: NULL argument", who);
    if (!aligned16(ptrs[k])) return set_error(FU_ERR_ALIGN, "%s: arrays must be 16-byte aligned", who);
  }
  return FU_OK;
}

}  // namespace sg

// fu_linear_dgrad_ln_silu_bwd on few rows (operands checked by the caller).
void launch_short_ln_bwd(const float* A, int64_t lda, const void* W2, float* g_x, int64_t ldgx, int64_t M, int32_t K,
                         const float* x, int64_t ldx, const float* gamma, const float* beta, const float* mean,
                         const float* rstd, int32_t G, hipStream_t st) {
  sg::Prob p{};
  sg::real_weight(p, W2, 128, K);
  p.A = A;
  p.lda = lda;
  p.Y = g_x;
  p.ldy = ldgx;
  hipLaunchKernelGGL(sg::short_ln_bwd_kernel, dim3(cdiv(M, sg::TR)), dim3(64 * sg::LW), 0, st, p,
                     sg::LnBwd{x, ldx, gamma, beta, mean, rstd, G}, M);
}

}  // namespace fu

using namespace fu;

extern "C" int fu_linear_short(const float* A, int64_t lda, const void* W2, const float* bias, float* Y, int64_t ldy,
                               int64_t M, int32_t N, int32_t K, void* stream) {
  using namespace fu::sg;
  const char* who = "fu_linear_short";
  if (M < 0 || M > (1 << 24) || N <= 0 || N % 64 != 0 || K < 16 || K % 16 != 0 || lda < K || ldy < N)
    return set_error(FU_ERR_SHAPE, "%s: M=%lld N=%d K=%d (0 <= M <= 2^24, N %% 64 == 0, K %% 16 == 0)", who,
                     (long long)M, N, K);
  if (M == 0) return FU_OK;
  if (!A || !W2 || !Y) return set_error(FU_ERR_NULL, "%s: NULL argument", who);
  if (!aligned16(A) || !aligned16(W2) || !aligned16(Y) || (bias && !aligned16(bias)) || lda % 4 != 0 || ldy % 4 != 0)
    return set_error(FU_ERR_ALIGN, "%s: A, W2, bias and Y must be 16-byte aligned, lda and ldy multiples of 4", who);
  Group g{};
  g.M = M;
  g.C = 64;   // unused by the plain epilogue
  g.L = 2;
  real_weight(g.p[0], W2, N, K);
  g.p[0].A = A;
  g.p[0].lda = lda;
  g.p[0].bias = bias;
  g.p[0].Y = Y;
  g.p[0].ldy = ldy;
  launch<0, 0>(g, 1, as_stream(stream));
  return check_launch(who);
}

extern "C" int fu_so2_pair_fwd(const float* X0, const float* X1, const float* X2, const void* W0, const float* b0,
                               const void* W1, const void* W2, const void* V0, const float* c0, const void* V1,
                               const void* V2, float* Y0, float* Y1, float* Y2, float* Z0, float* Z1, float* Z2,
                               float* O0, float* O1, float* O2, int64_t E, int32_t C, int32_t lmax, void* stream) {
  using namespace fu::sg;
  const char* who = "fu_so2_pair_fwd";
  const void* ptrs[] = {X0, X1, X2, W0, b0, W1, W2, V0, c0, V1, V2, Y0, Y1, Y2, Z0, Z1, Z2, O0, O1, O2};
  const int st = pair_check(who, E, C, lmax, ptrs, 20);
  if (st != FU_OK) return st > 0 ? FU_OK : st;
  const int L = lmax, n0 = (L + 1) * C, nm[3] = {0, L * C, (L - 1) * C};
  const float* X[3] = {X0, X1, X2};
  float *Y[3] = {Y0, Y1, Y2}, *Z[3] = {Z0, Z1, Z2}, *O[3] = {O0, O1, O2};
  const void *W[3] = {W0, W1, W2}, *V[3] = {V0, V1, V2};
  hipStream_t s = as_stream(stream);
  Group g{};
  g.M = E;
  g.C = C;
  g.L = L;
  // conv1 m = 0 with its gates
  real_weight(g.p[0], W0, (2 * L + 1) * C, 2 * n0);
  g.p[0].A = X0;
  g.p[0].lda = 2 * n0;
  g.p[0].bias = b0;
  g.p[0].Y = Y0;
  g.p[0].ldy = (2 * L + 1) * C;
  g.p[0].Z = Z0;
  g.p[0].ldz = n0;
  launch<1, 0>(g, 1, s);
  // conv1 m = 1, 2, gated by the columns of Y0
  for (int m = 1; m < 3; ++m) {
    Prob& p = g.p[m - 1] = Prob{};
    const int n = nm[m];
    complex_weight(p, W[m], n, 2 * n);
    p.A = X[m];
    p.Ai = X[m] + 2 * n;
    p.lda = 4 * n;
    p.Y = Y[m];
    p.Yi = Y[m] + n;
    p.ldy = p.ldz = 2 * n;
    p.Z = Z[m];
    p.Zi = Z[m] + n;
    p.G = Y0;
    p.ldg = (2 * L + 1) * C;
    p.s_off = (m - 1) * C;
  }
  launch<1, 1>(g, 2, s);
  // conv2, all three orders
  g.p[0] = Prob{};
  real_weight(g.p[0], V0, n0, n0);
  g.p[0].A = Z0;
  g.p[0].lda = g.p[0].ldy = n0;
  g.p[0].bias = c0;
  g.p[0].Y = O0;
  for (int m = 1; m < 3; ++m) {
    Prob& p = g.p[m] = Prob{};
    const int n = nm[m];
    complex_weight(p, V[m], n, n);
    p.A = Z[m];
    p.Ai = Z[m] + n;
    p.lda = p.ldy = 2 * n;
    p.Y = O[m];
    p.Yi = O[m] + n;
  }
  launch<0, 2>(g, 3, s);
  return check_launch(who);
}

extern "C" int fu_so2_pair_bwd(const float* G0, const float* G1, const float* G2, const float* Y0, const float* Y1,
                               const float* Y2, const void* W0t, const void* W1t, const void* W2t, const void* V0t,
                               const void* V1t, const void* V2t, float* gY0, float* gY1, float* gY2, float* P1,
                               float* P2, float* gX0, float* gX1, float* gX2, int64_t E, int32_t C, int32_t lmax,
                               void* stream) {
  using namespace fu::sg;
  const char* who = "fu_so2_pair_bwd";
  const void* ptrs[] = {G0, G1, G2, Y0, Y1, Y2, W0t, W1t, W2t, V0t, V1t, V2t, gY0, gY1, gY2, P1, P2, gX0, gX1, gX2};
  const int st = pair_check(who, E, C, lmax, ptrs, 20);
  if (st != FU_OK) return st > 0 ? FU_OK : st;
  const int L = lmax, n0 = (L + 1) * C, nm[3] = {0, L * C, (L - 1) * C}, ny0 = (2 * L + 1) * C;
  const float *G[3] = {G0, G1, G2}, *Y[3] = {Y0, Y1, Y2};
  float *gY[3] = {gY0, gY1, gY2}, *gX[3] = {gX0, gX1, gX2}, *P[3] = {nullptr, P1, P2};
  const void *W[3] = {W0t, W1t, W2t}, *V[3] = {V0t, V1t, V2t};
  hipStream_t s = as_stream(stream);
  Group g{};
  g.M = E;
  g.C = C;
  g.L = L;
  // conv2 m = 1, 2 input gradients with the gate backward: g_Y and the gate sums
  for (int m = 1; m < 3; ++m) {
    Prob& p = g.p[m - 1];
    const int n = nm[m];
    complex_weight(p, V[m], n, n);
    p.A = G[m];
    p.Ai = G[m] + n;
    p.lda = p.ldy = p.ldf = 2 * n;
    p.Y = gY[m];
    p.Yi = gY[m] + n;
    p.Z = P[m];
    p.ldz = n;
    p.G = Y0;
    p.ldg = ny0;
    p.F = Y[m];
    p.Fi = Y[m] + n;
    p.s_off = (m - 1) * C;
  }
  launch<2, 1>(g, 2, s);
  // conv2 m = 0: the gate-paired g_Y_m0 with the gate gradients
  g.p[0] = Prob{};
  real_weight(g.p[0], V0t, n0, n0);
  g.p[0].A = G0;
  g.p[0].lda = n0;
  g.p[0].Y = gY0;
  g.p[0].ldy = g.p[0].ldg = ny0;
  g.p[0].G = Y0;
  g.p[0].F = P1;
  g.p[0].ldf = nm[1];
  g.p[0].Fi = P2;
  g.p[0].ldfi = nm[2];
  launch<2, 0>(g, 1, s);
  // conv1 input gradients, all three orders
  g.p[0] = Prob{};
  real_weight(g.p[0], W0t, 2 * n0, ny0);
  g.p[0].A = gY0;
  g.p[0].lda = ny0;
  g.p[0].Y = gX0;
  g.p[0].ldy = 2 * n0;
  for (int m = 1; m < 3; ++m) {
    Prob& p = g.p[m] = Prob{};
    const int n = nm[m];
    complex_weight(p, W[m], 2 * n, n);
    p.A = gY[m];
    p.Ai = gY[m] + n;
    p.lda = 2 * n;
    p.Y = gX[m];
    p.Yi = gX[m] + 2 * n;
    p.ldy = 4 * n;
  }
  launch<0, 2>(g, 3, s);
  return check_launch(who);
}
