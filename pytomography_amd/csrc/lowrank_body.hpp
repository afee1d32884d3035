// lowrank_body.hpp -- wave bodies of the projector that blurs a few combined
// images instead of every plane (lowrank.hpp), float32 with a PSF.  Everything
// here runs per wave of 64 lanes; LDS holds a wave's bilinear taps, the sums over
// images of a forward block and the projection tiles of a backward block.
//
// Measured for 15 angles at 128^3 with attenuation, plane by plane / combined:
// forward 106 us / 58 (samples to images) + 26 (blur), back projection 111 + 29 /
// 21 (blur) + 61 (field) + 29 (the same gather).  Float32 matrix products run at
// the vector rate here; the gain is the images' number, 29 instead of 180 planes.
//
// Matrix instructions: v_mfma_f32_16x16x4_f32, D[16][16] += A[16][4] B[4][16],
// float32 inputs and accumulation.  Lane l holds A[l % 16][l / 16],
// B[l / 16][l % 16] and D[4 (l / 16) + r][l % 16], r = 0..3.
#pragma once

#include <type_traits>

#include "lowrank_launch.hpp"

namespace spect {

#ifndef SPECT_CPU_MFMA
typedef float lr_f4 __attribute__((ext_vector_type(4)));
__device__ __forceinline__ lr_f4 lr_mfma(float a, float b, lr_f4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ lr_f4 lr_load4_stream(const float *p, uint32_t byte) {
  return __builtin_nontemporal_load(reinterpret_cast<const lr_f4 *>(reinterpret_cast<const char *>(p) + byte));
}
__device__ __forceinline__ float lr_load1_stream(const float *p, uint32_t byte) {
  return __builtin_nontemporal_load(reinterpret_cast<const float *>(reinterpret_cast<const char *>(p) + byte));
}
// no instruction is scheduled across
__device__ __forceinline__ void lr_fence() { __builtin_amdgcn_sched_barrier(0); }
// LDS written by a lane is read by the wave's other lanes
__device__ __forceinline__ void lr_wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}
#endif

// Bilinear taps of one plane and column: byte offsets and weights.
struct alignas(16) LrTap {
  uint32_t o[4];
  float w[4];
};

__device__ __forceinline__ lr_f4 lr_load4(const float *p) { return *reinterpret_cast<const lr_f4 *>(p); }
// 32-bit byte offsets: the base stays in scalar registers (the object and one
// angle of the field are below 4 GiB, checked when the plan is made)
__device__ __forceinline__ lr_f4 lr_load4(const float *p, uint32_t byte) {
  return *reinterpret_cast<const lr_f4 *>(reinterpret_cast<const char *>(p) + byte);
}
__device__ __forceinline__ float lr_load1(const float *p, uint32_t byte) {
  return *reinterpret_cast<const float *>(reinterpret_cast<const char *>(p) + byte);
}
// Attenuation factors, read once per call: past the caches (kLrStream) or not.
template <int ATT> __device__ __forceinline__ lr_f4 lr_factor4(const float *p, uint32_t byte) {
  if constexpr (ATT == kLrStream) return lr_load4_stream(p, byte);
  else return lr_load4(p, byte);
}
template <int ATT> __device__ __forceinline__ float lr_factor1(const float *p, uint32_t byte) {
  if constexpr (ATT == kLrStream) return lr_load1_stream(p, byte);
  else return lr_load1(p, byte);
}
__device__ __forceinline__ lr_f4 lr_zero4() {
  lr_f4 z;
  z[0] = z[1] = z[2] = z[3] = 0.0f;
  return z;
}

// Planes [i_lo, i_hi] of rotated-frame column xn whose samples can lie in the
// footprint square (Geo::lo, Geo::hi): the intersection of two intervals of
// yn, widened by half a pixel of the square and one plane, so a superset of
// what in_footprint finds (i_hi < i_lo: none).  Solving for the interval
// replaces a per-column table: the tiles' ranges (32 columns wide) hold a
// third more planes than the columns use at 128^3.
__device__ __forceinline__ void lr_column_planes(const Geo<float> &g, float2 cs, float xn, int &i_lo, int &i_hi) {
  const float lo = (g.lo - 0.5f) / g.half - 1.0f, hi = (g.hi + 0.5f) / g.half - 1.0f;
  float a = -1.0f, b = 1.0f;
  bool none = false;
  // col: lo < c xn - s yn < hi;  row: lo < s xn + c yn < hi
  auto cut = [&](float k, float off) {
    float l = lo - off, h = hi - off;  // l < k yn < h
    if (fabsf(k) < 1e-4f) {            // moves by less than a pixel over all planes
      if (l > 1e-4f || h < -1e-4f) none = true;
      return;
    }
    const float p = l / k, q = h / k;
    a = fmaxf(a, fminf(p, q));
    b = fminf(b, fmaxf(p, q));
  };
  cut(-cs.y, cs.x * xn);
  cut(cs.x, cs.y * xn);
  i_lo = 1;
  i_hi = 0;
  if (none || b < a) return;
  i_lo = max(0, (int)floorf((a + 1.0f) * g.half) - 1);
  i_hi = min(g.P - 1, (int)ceilf((b + 1.0f) * g.half) + 1);
}

// 16-plane units [u0, u1) of segment seg of the angle's radius.
__device__ __forceinline__ void lr_segment(const LrTables &lr, int rix, int seg, int &u0, int &u1) {
  const int32_t *s = lr.seg_unit + (size_t)rix * (lr.nseg + 1) + seg;
  u0 = ld_uniform(s);
  u1 = ld_uniform(s + 1);
}

// ---------------------------------------------------------------------------
// Forward, first pass: the images G_r(j, z) = sum_i c[i][r] a(i,j,z) f_rot(i,j,z)
// of two neighbouring columns j, 32 z, and one segment's planes
// (Nz not a multiple of 4: one column, 64 z).
//
// A wave takes four planes at a time: lane l samples plane 4 q + l / 16 of column
// j0 + (l % 16) / 8 at z = 4 (l % 8) .. + 3, so each of the four taps and the
// attenuation factor is one 16-byte load, a 128-byte line per plane and column
// (scalar: z = l % 16 + 16 e).  The four values are the B operands of four
// products whose A operand holds the 16 image weights of the four planes -- the
// columns of B are any 16 samples of a plane -- so the sums over planes are left to
// the matrix instructions, and nothing is written until the planes are done.
// Taking the taps through LDS (one lane computes them for the eight along z)
// leaves about 40 of 120 vector instructions per four planes.
//
// What bounds it is the traffic between the L2s and memory, about 5 TB/s.  The
// factors are read once (lr_factor_mode); the object is read four
// times a voxel and should come from the L2.  With 32 z per wave and the launch
// giving each XCD one 32-z slab of the object at a time (2 MB of the 8 MB at
// 128^3), it does: 64 z per wave read it from memory once per angle and column
// strip (252 MB in all for 15 angles, 130 MB of them factors).
template <int ATT, bool VEC>
__device__ __forceinline__ void lr_gather_body(const LrGatherJob &J, int al, int seg, int jg, int zg, int lane,
                                               LrTap *lds) {
  constexpr int CW = VEC ? kLrGatherCols : 1, ZL = 16 / CW;  // columns of a wave, lanes along z
  const Geo<float> &g = J.g;
  const int ang = ld_uniform(J.angle_idx + al);
  if ((unsigned)ang >= (unsigned)g.A) return;
  const int rix = ld_uniform(J.radius_index + ang);
  const int n_jext = g.je1 - g.je0;
  const float2 cs = ld_uniform(J.trig + ang);
  int u0, u1;
  lr_segment(J.lr, rix, seg, u0, u1);
  // quads of the segment's planes that the wave's columns visit
  int q0 = 4 * u0, q1 = 4 * u1;
  {
    int i_lo = g.P, i_hi = -1;
#pragma unroll
    for (int c = 0; c < CW; ++c) {
      int lo, hi;
      lr_column_planes(g, cs, ld_uniform(J.lin + g.je0 + min(jg * CW + c, n_jext - 1)), lo, hi);
      if (lo <= hi) {
        i_lo = min(i_lo, lo);
        i_hi = max(i_hi, hi);
      }
    }
    q0 = max(q0, i_lo >> 2);
    q1 = min(q1, (i_hi >> 2) + 1);  // i_hi = -1: no quads
  }
  const int kg = lane >> 4, m = lane & 15;
  const int jx = jg * CW + m / ZL, jc = min(jx, n_jext - 1);
  const uint32_t sz = 4u * (uint32_t)g.Nz, sr = sz * (uint32_t)g.N;  // bytes per column, per row
  constexpr int NE = VEC ? 1 : 4;                                     // loads per sample
  // lanes past Nz sample z = 0 instead: their sums are set to zero at the end
  uint32_t zo[NE];
#pragma unroll
  for (int e = 0; e < NE; ++e) {
    const int z = VEC ? (zg * ZL + m % ZL) * 4 : zg * 64 + 16 * e + m;
    zo[e] = 4u * (uint32_t)(z < g.Nz ? z : 0);
  }
  const float *cf = J.lr.cf + (size_t)rix * J.lr.quads * 64 + lane;
  const float *af = ATT ? J.attf + (size_t)ang * g.P * n_jext * g.Nz : nullptr;
  const uint32_t ap = (uint32_t)n_jext * sz, ac = (uint32_t)jc * sz;  // bytes per plane, to the column
  lr_f4 acc[4];
#pragma unroll
  for (int e = 0; e < 4; ++e) acc[e] = lr_zero4();
  float vmin = 0.0f;

  // The bilinear taps of QB quads, one plane and column per lane, into the
  // wave's own LDS (each is used by the ZL lanes along z): offsets and weights
  // as taps4().
  constexpr int QB = 8;
  auto taps = [&](int q) {
    if (4 * QB * CW < 64 && lane >= 4 * QB * CW) return;
    const int col = lane % CW, i = 4 * q + lane / CW;  // entry lane = 4 CW * quad + CW * plane + column
    const float yn = J.lin[min(i, g.P - 1)], xn = J.lin[g.je0 + min(jg * CW + col, n_jext - 1)];
    float ix, iy;
    rot_coord<float>(cs.x, cs.y, xn, yn, g.half, ix, iy);
    const Src<float> s = make_src<float>(ix, iy, g.pad);
    const float ex = 1.0f - s.tx, ny = 1.0f - s.ty;
    const bool r0 = (unsigned)s.r0 < (unsigned)g.N, r1 = (unsigned)(s.r0 + 1) < (unsigned)g.N;
    const bool c0 = (unsigned)s.c0 < (unsigned)g.N, c1 = (unsigned)(s.c0 + 1) < (unsigned)g.N;
    const uint32_t rr0 = (uint32_t)min(max(s.r0, 0), g.N - 1), rr1 = (uint32_t)min(max(s.r0 + 1, 0), g.N - 1);
    const uint32_t cc0 = (uint32_t)min(max(s.c0, 0), g.N - 1), cc1 = (uint32_t)min(max(s.c0 + 1, 0), g.N - 1);
    // row and column products of 24-bit factors (rows of an object below 4 GiB
    // are below 2^24 bytes for every N the plan accepts)
    const uint32_t b0 = __umul24(rr0, sr), b1 = __umul24(rr1, sr);
    const uint32_t d0 = __umul24(cc0, sz), d1 = __umul24(cc1, sz);
    LrTap t;
    t.w[0] = (r0 && c0) ? ny * ex : 0.0f;
    t.w[1] = (r0 && c1) ? ny * s.tx : 0.0f;
    t.w[2] = (r1 && c0) ? s.ty * ex : 0.0f;
    t.w[3] = (r1 && c1) ? s.ty * s.tx : 0.0f;
    t.o[0] = b0 + d0;
    t.o[1] = b0 + d1;
    t.o[2] = b1 + d0;
    t.o[3] = b1 + d1;
    lds[lane] = t;
  };

  // The factors and weights of a block of QB quads; each step's are requested
  // when the same step of the block before is done.
  constexpr int U = 2, STEPS = QB / U;  // quads per step, steps per block
  struct Ahead {
    float c[U];
    lr_f4 a[U];
  } ring[STEPS];
  auto ahead = [&](int q, Ahead &t) {
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int qc = min(q + u, q1 - 1);
      t.c[u] = cf[(size_t)qc * 64];
      if constexpr (ATT) {  // weights of planes past P are zero
        const uint32_t ao = __umul24((uint32_t)min(4 * qc + kg, g.P - 1), ap) + ac;
        if constexpr (VEC) t.a[u] = lr_factor4<ATT>(af, ao + zo[0]);
        else
#pragma unroll
          for (int e = 0; e < 4; ++e) t.a[u][e] = lr_factor1<ATT>(af, ao + zo[e]);
      }
    }
  };
  // quads q, q + 1 of the block of taps from qb on
  auto step = [&](int qb, int q, const Ahead &cur) {
    LrTap t[U];
    lr_f4 v[U][4];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      t[u] = lds[4 * CW * (min(q + u, q1 - 1) - qb) + CW * kg + m / ZL];
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        if constexpr (VEC) v[u][k] = lr_load4(J.f, t[u].o[k] + zo[0]);
        else
#pragma unroll
          for (int e = 0; e < 4; ++e) v[u][k][e] = lr_load1(J.f, t[u].o[k] + zo[e]);
      }
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const float c = q + u < q1 ? cur.c[u] : 0.0f;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        // interp()'s order of the four taps
        float x = v[u][0][e] * t[u].w[0];
        x = x + v[u][1][e] * t[u].w[1];
        x = x + v[u][2][e] * t[u].w[2];
        x = x + v[u][3][e] * t[u].w[3];
        if constexpr (ATT) x = x * cur.a[u][e];
        vmin = fminf(vmin, x);
        acc[e] = lr_mfma(c, x, acc[e]);
      }
    }
  };
  if (q0 < q1) {
#pragma unroll
    for (int k = 0; k < STEPS; ++k) ahead(min(q0 + k * U, q1 - 1), ring[k]);
  }
  for (int qb = q0; qb < q1; qb += QB) {
    lr_wave_sync();  // the taps of the block before have been read
    taps(qb);
    lr_wave_sync();
#pragma unroll
    for (int k = 0; k < STEPS; ++k) {
      const int q = qb + k * U;
      if (q >= q1) break;
      step(qb, q, ring[k]);
      if (q + QB < q1) ahead(q + QB, ring[k]);
    }
  }
  // rows 4 kg + r of the segment's images; z past Nz (up to NzP) holds zeros
  const int rows = ld_uniform(J.lr.seg_rows + (size_t)rix * J.lr.nseg + seg);
  const size_t image = lr_image_floats(g, J.NzP);
  float *G = J.G + ((size_t)al * J.lr.nseg + seg) * kLrRowsDev * image;
  if (jx < n_jext) {
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      if (4 * kg + r >= rows) continue;
      float *dst = G + (size_t)(4 * kg + r) * image;
      if constexpr (VEC) {
        const int z = (zg * ZL + m % ZL) * 4;
        lr_f4 o;
#pragma unroll
        for (int e = 0; e < 4; ++e) o[e] = z < g.Nz ? acc[e][r] : 0.0f;
        if (z < J.NzP) *reinterpret_cast<lr_f4 *>(dst + lr_image_at(g, J.NzP, jx, z)) = o;
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const int z = zg * 64 + 16 * e + m;
          if (z < J.NzP) dst[lr_image_at(g, J.NzP, jx, z)] = z < g.Nz ? acc[e][r] : 0.0f;
        }
      }
    }
  }
  // whether any sample was negative (see the blur)
  const bool neg = __ballot(vmin < 0.0f) != 0;
  if (lane == 0)
    J.neg[(((size_t)al * J.lr.nseg + seg) * J.zgroups + zg) * J.cgroups + jg] = neg ? 1 : 0;
}

// ---------------------------------------------------------------------------
// The separable blur of one image by matrix products with the Toeplitz
// matrices of its node's taps, 16 x 16 tiles, for one tile of 16 z and NT
// tiles of 16 output rows:
//   X[j][z'] = sum_z G[j][z] Tz[z][z'],   out[j'][z'] += sum_j Ty[j'][j] X[j][z'].
// The K index of a product is summed over, so its order is free: the z product
// takes z = 16 c + 4 (l / 16) + e in step e (one 16-byte load per lane and tile
// of G), and the y product takes j = 16 J + 4 (l / 16) + r in step r -- which is
// the row that lane already holds in register r of X, so X passes from the
// result of the first product into the second without leaving its registers.
// Both operands then hold tap 16 D + 4 (l / 16) + e - l % 16 + H for tiles D
// apart.  ND: tiles to either side that the half width reaches (H <= 16: 1).
template <int ND> struct LrToeplitz {
  float z[2 * ND + 1][4], y[2 * ND + 1][4];
};

// The taps are stored with zeros around them (lr_tap_stride), stride floats for
// z, then for y.
template <int ND>
__device__ __forceinline__ void lr_toeplitz(const float *taps, int stride, int lane, LrToeplitz<ND> &t) {
  const float *c = taps + (stride / 2 + 4 * (lane >> 4) - (lane & 15));
#pragma unroll
  for (int d = -ND; d <= ND; ++d)
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      t.z[d + ND][e] = c[16 * d + e];
      t.y[d + ND][e] = c[stride + 16 * d + e];
    }
}

// z tiles zt + d outside [0, ztiles) get a zero operand, so that the loads of
// the image may be clamped to it.
template <int ND>
__device__ __forceinline__ void lr_toeplitz_edges(int zt, int ztiles, LrToeplitz<ND> &t) {
#pragma unroll
  for (int d = -ND; d <= ND; ++d) {
    const bool in = zt + d >= 0 && zt + d < ztiles;
#pragma unroll
    for (int e = 0; e < 4; ++e) t.z[d + ND][e] = in ? t.z[d + ND][e] : 0.0f;
  }
}

// The products of one row J of tiles (a[d + ND]: its tiles at z tile zt + d): X,
// then its share in the output rows within reach.  Rows [row_lo, row_hi) (in
// rows of tile 0) are inside the image, any others count as zero.
template <int NT, int ND>
__device__ __forceinline__ void lr_blur_row(const LrToeplitz<ND> &t, int J, int row_lo, int row_hi, int lane,
                                            const lr_f4 (&a)[2 * ND + 1], lr_f4 (&acc)[NT]) {
  if (16 * J + 16 <= row_lo || 16 * J >= row_hi) return;  // wave-uniform
  lr_f4 x = lr_zero4(), x1 = lr_zero4();                  // two chains of products
#pragma unroll
  for (int d = 0; d < 2 * ND + 1; ++d)
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      if (e & 1) x1 = lr_mfma(a[d][e], t.z[d][e], x1);
      else x = lr_mfma(a[d][e], t.z[d][e], x);
    }
  const int row = 16 * J + 4 * (lane >> 4);
#pragma unroll
  for (int r = 0; r < 4; ++r) x[r] = row + r >= row_lo && row + r < row_hi ? x[r] + x1[r] : 0.0f;
#pragma unroll
  for (int r = 0; r < 4; ++r)
#pragma unroll
    for (int d = -ND; d <= ND; ++d) {
      const int o = J - d;
      if (o >= 0 && o < NT) acc[o] = lr_mfma(t.y[d + ND][r], x[r], acc[o]);  // compile-time choice
    }
}

// Adds the blur of one image to acc.  fetch(J, a) requests the tiles of row J;
// they arrive AHEAD rows early, and the block's other waves cover the rest of
// the wait: few enough registers for four waves per SIMD beat holding all the
// tiles of two images with two (26 against 30 us for 15 angles at 128^3, 174
// against 202 for 120; back projection 21 against 45).
template <int NT, int ND, int AHEAD, typename Fetch>
__device__ __forceinline__ void lr_blur_image(const LrToeplitz<ND> &t, int row_lo, int row_hi, int lane, Fetch fetch,
                                              lr_f4 (&acc)[NT]) {
  lr_f4 a[AHEAD + 1][2 * ND + 1];
#pragma unroll
  for (int k = 0; k < AHEAD; ++k) fetch(k - ND, a[k]);
#pragma unroll
  for (int k = 0; k < NT + 2 * ND; ++k) {
    if (k + AHEAD < NT + 2 * ND) fetch(k + AHEAD - ND, a[(k + AHEAD) % (AHEAD + 1)]);
    lr_fence();
    lr_blur_row<NT, ND>(t, k - ND, row_lo, row_hi, lane, a[k % (AHEAD + 1)], acc);
  }
}

// Forward, second pass: projection rows [16 NT jr, + 16 NT) x z tile zt of one
// angle.  Wave w of the block blurs images w, w + nw, ...; the waves' sums are
// added in LDS in wave order, and the Poisson ratio is formed as in
// reduce_body.
//
// The weights c[i][r] have both signs, so where no blurred plane reaches, the
// sum of the images is rounding noise of either sign instead of an exact zero.
// A ray sum of samples none of which was negative is not negative: when no
// wave of the angle's first pass saw a negative sample, negative sums are set
// to zero (taps are non-negative; a PSF with negative taps does not run here).
template <int NT, int ND>
__device__ __forceinline__ void lr_blur_forward_body(const LrBlurJob &J, int al, int zt, int jr, int wave, int nw,
                                                     int lane, float *smem) {
  const Geo<float> &g = J.g;
  const int ang = ld_uniform(J.angle_idx + al);
  if ((unsigned)ang >= (unsigned)g.A) return;
  const int rix = ld_uniform(J.radius_index + ang);
  const int n_jext = g.je1 - g.je0, nout = g.jo1 - g.jo0;
  const int kg = lane >> 4, m = lane & 15, ztiles = J.NzP / 16, stride = 2 * (16 * ND + 15) + 1;
  const int count = ld_uniform(J.lr.count + rix);
  const int row0 = g.jo0 - g.je0 + 16 * NT * jr;  // extended column of output row 0
  const uint32_t lane_off = 4u * (uint32_t)(m * 16 + 4 * kg);
  const size_t image = lr_image_floats(g, J.NzP);
  lr_f4 acc[NT];
#pragma unroll
  for (int o = 0; o < NT; ++o) acc[o] = lr_zero4();
  for (int r = wave; r < count; r += nw) {
    const int4 img = ld_uniform_struct(J.lr.img + (size_t)rix * J.lr.nimg + r);
    const float *taps = J.lr.taps + ((size_t)rix * J.lr.nimg + r) * 2 * stride;
    const float *G = J.G + ((size_t)(al * J.lr.nseg + img.x) * kLrRowsDev + img.y) * image;
    auto run = [&](auto nd) {
      constexpr int D = decltype(nd)::value;
      LrToeplitz<D> t;
      lr_toeplitz<D>(taps, stride, lane, t);
      // columns outside the extended range hold anything, and tiles past the
      // image are those of the next (padded after the last): they only reach
      // rows of X that are set to zero
      auto fetch = [&](int row, lr_f4 (&a)[2 * D + 1]) {
#pragma unroll
        for (int d = -D; d <= D; ++d) {
          const int c = min(max(zt + d, 0), ztiles - 1);
          a[d + D] = lr_load4(G + (size_t)((NT * jr + row + kLrLead) * ztiles + c) * 256, lane_off);
        }
      };
      lr_toeplitz_edges<D>(zt, ztiles, t);
      lr_blur_image<NT, D, (D > 1 ? 1 : 2)>(t, -row0, n_jext - row0, lane, fetch, acc);
    };
    if constexpr (ND > 1) {
      if (img.z <= 16) {  // this image's taps end within one tile
        run(std::integral_constant<int, 1>{});
        continue;
      }
    }
    run(std::integral_constant<int, ND>{});
  }
  // any negative sample of the angle
  const int tid = wave * 64 + lane;
  int neg = 0;
  const int nflags = J.lr.nseg * J.zgroups * J.cgroups;
  for (int q = tid; q < nflags; q += nw * 64) neg |= J.neg[(size_t)al * nflags + q];
  neg = __syncthreads_or(neg);
#pragma unroll
  for (int o = 0; o < NT; ++o)
#pragma unroll
    for (int r = 0; r < 4; ++r) smem[((wave * NT + o) * 4 + r) * 64 + lane] = acc[o][r];
  __syncthreads();
  for (int q = tid; q < NT * 256; q += nw * 64) {
    float v = smem[q];
    for (int w = 1; w < nw; ++w) v += smem[w * NT * 256 + q];
    const int l = q & 63, jx = 16 * (NT * jr + (q >> 8)) + 4 * (l >> 4) + ((q >> 6) & 3), z = 16 * zt + (l & 15);
    if (jx >= nout || z >= g.Nz) continue;
    if (!neg && v < 0.0f) v = 0.0f;  // keeps NaN
    const size_t idx = ((size_t)al * nout + jx) * g.Nz + z;
    if (J.proj) J.proj[idx] = v;
    if (J.gm) {
      float p = v;
      if (J.s) p = p + J.s[idx];
      if (J.pred) J.pred[idx] = p;
      J.ratio[idx] = J.gm[idx] / (p + J.delta);
    }
  }
}

// ---------------------------------------------------------------------------
// Back projection, first pass: Q_r = k_(node r) * p for images wave, wave + nw,
// ... of one angle, tile rows [NT jr, + NT) of the images, z tile zt.  The block
// takes its tiles of p to LDS once ([row][z][lane], the products' A operands),
// which leaves registers for four waves per SIMD.
template <int NT, int ND, bool VEC>
__device__ __forceinline__ void lr_blur_backward_body(const LrBackJob &J, int al, int zt, int jr, int wave, int nw,
                                                      int lane, lr_f4 *smem) {
  const Geo<float> &g = J.g;
  const int ang = ld_uniform(J.angle_idx + al);
  if ((unsigned)ang >= (unsigned)g.A) return;
  const int rix = ld_uniform(J.radius_index + ang);
  const int count = ld_uniform(J.lr.count + rix);
  const int nout = g.jo1 - g.jo0;
  const int kg = lane >> 4, m = lane & 15, ztiles = J.NzP / 16, stride = 2 * (16 * ND + 15) + 1;
  const int tile0 = lr_first_tile(g) + NT * jr, ntiles = lr_row_tiles(nout);
  const int row0 = 16 * (tile0 - kLrLead);  // detector column of output row 0
  const float *p = J.proj + (size_t)al * nout * g.Nz;
  float pmin = 0.0f;
  constexpr int W = 2 * ND + 1, R = NT + 2 * ND;
  for (int q = wave; q < R * W; q += nw) {
    const int k = q / W, d = q - k * W;
    const int j = row0 + 16 * (k - ND) + m, z = 16 * (zt + d - ND) + 4 * kg;
    const float *src = p + (uint32_t)(min(max(j, 0), nout - 1) * g.Nz);
    lr_f4 v;
    if constexpr (VEC) {
      v = lr_load4(src + min(max(z, 0), g.Nz - 4));
    } else {
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] = src[min(max(z + e, 0), g.Nz - 1)];
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      v[e] = (unsigned)j < (unsigned)nout && (unsigned)(z + e) < (unsigned)g.Nz ? v[e] : 0.0f;
      pmin = fminf(pmin, v[e]);
    }
    smem[q * 64 + lane] = v;
  }
  const int neg = __syncthreads_or(pmin < 0.0f);
  if (wave == 0 && lane == 0) J.neg[((size_t)al * J.jranges + jr) * ztiles + zt] = neg ? 1 : 0;
  for (int r = wave; r < count; r += nw) {
    const int4 img = ld_uniform_struct(J.lr.img + (size_t)rix * J.lr.nimg + r);
    const float *taps = J.lr.taps + ((size_t)rix * J.lr.nimg + r) * 2 * stride;
    lr_f4 acc[NT];
#pragma unroll
    for (int o = 0; o < NT; ++o) acc[o] = lr_zero4();
    auto run = [&](auto nd) {
      constexpr int D = decltype(nd)::value;
      LrToeplitz<D> t;
      lr_toeplitz<D>(taps, stride, lane, t);
      auto fetch = [&](int row, lr_f4 (&a)[2 * D + 1]) {
#pragma unroll
        for (int d = -D; d <= D; ++d) a[d + D] = smem[((row + ND) * W + d + ND) * 64 + lane];
      };
      lr_blur_image<NT, D, 1>(t, -row0, nout - row0, lane, fetch, acc);
    };
    if (ND > 1 && img.z <= 16) run(std::integral_constant<int, 1>{});  // its taps end within one tile
    else run(std::integral_constant<int, ND>{});
    float *Q = J.Q + ((size_t)(al * J.lr.nseg + img.x) * kLrRowsDev + img.y) * lr_image_floats(g, J.NzP);
    // whole tiles; those of columns outside the extended range are not read
#pragma unroll
    for (int o = 0; o < NT; ++o) {
      if (tile0 + o >= ntiles) continue;
      float *dst = Q + (size_t)((tile0 + o) * ztiles + zt) * 256;
#pragma unroll
      for (int k = 0; k < 4; ++k) dst[(uint32_t)((4 * kg + k) * 16 + m)] = acc[o][k];
    }
  }
}

// ---------------------------------------------------------------------------
// Back projection, second pass: W(i,j,z) = a(i,j,z) sum_r c[i][r] Q_r(j,z) of
// one column j, 64 z and one segment's planes: per unit of 16 planes a product
// of the unit's weights (A) with the column's images (B, held for all units).
// The images of a column are read once, the factors and W stream through.
// With a non-negative projection W is not negative (as in the forward).
template <int ATT, bool VEC>
__device__ __forceinline__ void lr_field_body(const LrBackJob &J, int al, int seg, int jx, int zb, int lane) {
  const Geo<float> &g = J.g;
  const int ang = ld_uniform(J.angle_idx + al);
  if ((unsigned)ang >= (unsigned)g.A) return;
  const int rix = ld_uniform(J.radius_index + ang);
  int u0, u1;
  lr_segment(J.lr, rix, seg, u0, u1);
  const float2 cs = ld_uniform(J.trig + ang);
  const float xn = ld_uniform(J.lin + g.je0 + jx);
  int i_lo, i_hi;
  lr_column_planes(g, cs, xn, i_lo, i_hi);
  u0 = max(u0, i_lo >> 4);
  u1 = min(u1, (i_hi >> 4) + 1);
  if (u0 >= u1) return;
  const int kg = lane >> 4, m = lane & 15;
  const int n_jext = g.je1 - g.je0;
  const int rows = ld_uniform(J.lr.seg_rows + (size_t)rix * J.lr.nseg + seg);
  int neg = 0;
  const int nflags = J.jranges * (J.NzP / 16);
  for (int q = lane; q < nflags; q += 64) neg |= J.neg[(size_t)al * nflags + q];
  const float floor_w = __ballot(neg != 0) != 0 ? -__builtin_inff() : 0.0f;
  // B operands: step s holds image row 4 s + kg at this lane's z values
  const size_t image = lr_image_floats(g, J.NzP);
  const float *Q = J.Q + (size_t)(al * J.lr.nseg + seg) * kLrRowsDev * image;
  lr_f4 b[4];
#pragma unroll
  for (int s = 0; s < 4; ++s) {
    const bool ok = 4 * s + kg < rows;
    const float *src = Q + (size_t)(ok ? 4 * s + kg : 0) * image;
    if constexpr (VEC) {
      const int z = zb * 64 + 4 * m;
      const lr_f4 u = lr_load4(src + lr_image_at(g, J.NzP, jx, z < J.NzP ? z : 0));
#pragma unroll
      for (int e = 0; e < 4; ++e) b[s][e] = ok ? u[e] : 0.0f;
    } else {
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int z = zb * 64 + 16 * e + m;
        const float u = src[lr_image_at(g, J.NzP, jx, z < J.NzP ? z : 0)];
        b[s][e] = ok ? u : 0.0f;
      }
    }
  }
  const float *cb = J.lr.cb + (size_t)rix * (J.lr.quads / 4) * 256 + lane;
  const uint32_t pb = (uint32_t)n_jext * 4u * (uint32_t)g.Nz;  // bytes per plane
  const size_t column = (size_t)jx * g.Nz, frame = (size_t)g.P * n_jext * g.Nz;
  const float *af = ATT ? J.attf + (size_t)ang * frame + column : nullptr;
  float *W = J.W + (size_t)al * frame + column;
  for (int u = u0; u < u1; ++u) {
    lr_f4 a[4];  // factors of planes 16 u + 4 kg + r
    bool pok[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int i = 16 * u + 4 * kg + r;
      pok[r] = i >= i_lo && i <= i_hi;
      if constexpr (ATT) {
        const uint32_t ao = __umul24((uint32_t)(pok[r] ? i : i_lo), pb);
        if constexpr (VEC) {
          const int z = zb * 64 + 4 * m;
          a[r] = lr_factor4<ATT>(af, ao + 4u * (uint32_t)(z < g.Nz ? z : 0));
        } else {
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const int z = zb * 64 + 16 * e + m;
            a[r][e] = lr_factor1<ATT>(af, ao + 4u * (uint32_t)(z < g.Nz ? z : 0));
          }
        }
      }
    }
    lr_f4 d[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) d[e] = lr_zero4();
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      const float c = cb[(size_t)u * 256 + s * 64];
      if (4 * s < rows) {  // wave-uniform
#pragma unroll
        for (int e = 0; e < 4; ++e) d[e] = lr_mfma(c, b[s][e], d[e]);
      }
    }
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      if (!pok[r]) continue;
      const int i = 16 * u + 4 * kg + r;
      lr_f4 w;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        w[e] = d[e][r] < floor_w ? floor_w : d[e][r];  // keeps NaN
        if constexpr (ATT) w[e] = w[e] * a[r][e];
      }
      float *dst = reinterpret_cast<float *>(reinterpret_cast<char *>(W) + __umul24((uint32_t)i, pb));
      if constexpr (VEC) {
        const int z = zb * 64 + 4 * m;
        if (z < g.Nz) *reinterpret_cast<lr_f4 *>(dst + z) = w;
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const int z = zb * 64 + 16 * e + m;
          if (z < g.Nz) dst[z] = w[e];
        }
      }
    }
  }
}

}  // namespace spect
