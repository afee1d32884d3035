// sensitivity.hip -- the field of a back projection of ones, in float64.
//
// A plane's PSF is separable, so the blur of a constant projection is the outer
// product of two profiles: W(i,j,z) = a(i,j,z) u_i(j) v_i(z), u_i and v_i the
// sums of the taps that fall on the detector.  No plane is blurred: what is left
// is the attenuation march and the store of W, 8 bytes a sample.  8 angles at
// 128^3 with the suffix table: 61 us, against 451 us for blurring a projection
// of ones.
#include <type_traits>

#include "launch.hpp"

namespace spect {
namespace {

// Entries of a plane's profiles: u, then v, each padded to whole 16-byte words.
__host__ __device__ inline int even(int x) { return (x + 1) & ~1; }
__host__ __device__ inline int profile_len(int n_jext, int Nz) { return even(n_jext) + even(Nz); }

// One block per (angle, plane): u over the extended columns, then v over z.
__global__ __launch_bounds__(256) void ones_profiles_kernel(Geo<double> g, Tables<double> tb, const int32_t *angle_idx,
                                                            double *prof) {
  const int al = blockIdx.y, i = blockIdx.x;
  const int ang = ld_uniform(angle_idx + al);
  if ((unsigned)ang >= (unsigned)g.A) return;
  const int K = 2 * g.H + 1, n_jext = g.je1 - g.je0, nout = g.jo1 - g.jo0;
  const int rix = ld_uniform(tb.radius_index + ang);
  const size_t row = ((size_t)rix * g.P + i) * K;
  const int he = g.H > 0 ? ld_uniform(tb.tier + (size_t)rix * g.P + i) : 0;
  double *dst = prof + ((size_t)al * g.P + i) * profile_len(n_jext, g.Nz);
  for (int q = threadIdx.x; q < n_jext + g.Nz; q += blockDim.x) {
    const bool col = q < n_jext;
    const int at = col ? q + g.je0 - g.jo0 : q - n_jext, end = col ? nout : g.Nz;
    double s = 0.0;
    if (g.H == 0) {
      s = at >= 0 && at < end ? 1.0 : 0.0;
    } else {
      const double *w = (col ? tb.taps_r : tb.taps_z) + row + g.H;
      for (int t = max(-he, -at); t <= min(he, end - 1 - at); ++t) s += w[t];
    }
    dst[col ? q : even(n_jext) + q - n_jext] = s;
  }
}

// A wave takes one column and 64 ZV z of one chunk of planes, z along the lanes.
// MODE 0: no attenuation, 1: factors of the field, 2: march from the chunk's
// row of the suffix table.
template <int MODE, int ZV>
__global__ __launch_bounds__(256) void ones_field_kernel(Geo<double> g, Tables<double> tb, const double *prof,
                                                         const double *mu, const double *att, int att_global,
                                                         const double *attf, const int32_t *angle_idx, double *W,
                                                         int zblocks) {
  const int n_jext = g.je1 - g.je0, len = profile_len(n_jext, g.Nz), Nz = g.Nz;
  const int v = blockIdx.x * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int jx = v / zblocks, c = blockIdx.y, al = blockIdx.z;
  if (jx >= n_jext) return;
  const int z = ((v - jx * zblocks) * 64 + (threadIdx.x & 63)) * ZV;
  const int ang = ld_uniform(angle_idx + al);
  if ((unsigned)ang >= (unsigned)g.A) return;
  const auto cs = ld_uniform(tb.trig + ang);
  const double lin = ld_uniform(tb.lin + g.je0 + jx);
  const bool mine = z < Nz;  // Nz is a multiple of ZV
  double S[ZV];
#pragma unroll
  for (int m = 0; m < ZV; ++m) S[m] = 0.0;
  if constexpr (MODE == 2) {
    if (mine) load_run<double, ZV>(att + (((size_t)(att_global ? ang : al) * g.C + c) * n_jext + jx) * Nz, z, Nz, S);
  }
  const int i_lo = c * g.L, i_hi = min(g.P, i_lo + g.L);
  for (int i = i_hi - 1; i >= i_lo; --i) {
    double ix, iy;
    rot_coord<double>(cs.x, cs.y, lin, ld_uniform(tb.lin + i), g.half, ix, iy);
    if (!in_footprint<double>(ix, iy, g)) continue;  // wave-uniform; the gather does not read it
    if (!mine) continue;
    const double *u = prof + ((size_t)al * g.P + i) * len;
    const size_t at = (((size_t)(MODE == 1 ? ang : al) * g.P + i) * n_jext + jx) * Nz;
    double w[ZV], x[ZV];
    load_run<double, ZV>(u + even(n_jext), z, Nz, w);
    if constexpr (MODE == 1) load_run<double, ZV>(attf + at, z, Nz, x);
    if constexpr (MODE == 2) {
      const Taps4<double> t = taps4<double>(make_src<double>(ix, iy, g.pad), g.N, Nz);
      gather_run<double, ZV>(mu, t, z, Nz, x);
    }
    const double uj = u[jx];
#pragma unroll
    for (int m = 0; m < ZV; ++m) {
      w[m] = uj * w[m];
      if constexpr (MODE == 1) w[m] = w[m] * x[m];
      if constexpr (MODE == 2) {
        const double xm = x[m] * g.dx;
        S[m] += xm;
        w[m] = w[m] * att_factor<double>(S[m], xm);
      }
    }
    double *dst = W + (((size_t)al * g.P + i) * n_jext + jx) * Nz + z;
    if constexpr (ZV == 2) *reinterpret_cast<double2 *>(dst) = make_double2(w[0], w[1]);
    else dst[0] = w[0];
  }
}

}  // namespace

size_t ones_profile_bytes(int n, int P, int n_jext, int Nz) {
  return ((size_t)n * P * profile_len(n_jext, Nz) * sizeof(double) + 255) & ~size_t(255);
}

hipError_t launch_ones_field(const Geo<double> &g, const Tables<double> &tb, const double *mu, const double *att,
                             bool att_global, const double *attf, const int32_t *angle_idx, int n, double *W,
                             double *prof, hipStream_t st) {
  const int n_jext = g.je1 - g.je0;
  if (n > 65535 || g.C > 65535) return hipErrorInvalidConfiguration;
  ones_profiles_kernel<<<dim3(g.P, n), 256, 0, st>>>(g, tb, angle_idx, prof);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  // 16-byte accesses; gather_run and load_run use them from Nz % 4 == 0
  const int zv = g.Nz % 4 == 0 ? 2 : 1, zblocks = (g.Nz + 64 * zv - 1) / (64 * zv);
  auto pick = [&](auto mode) {
    constexpr int M = decltype(mode)::value;
    return zv == 2 ? ones_field_kernel<M, 2> : ones_field_kernel<M, 1>;
  };
  auto kern = attf ? pick(std::integral_constant<int, 1>{})
              : mu ? pick(std::integral_constant<int, 2>{})
                   : pick(std::integral_constant<int, 0>{});
  kern<<<dim3((n_jext * zblocks + 3) / 4, g.C, n), 256, 0, st>>>(g, tb, prof, mu, att, att_global ? 1 : 0, attf,
                                                                 angle_idx, W, zblocks);
  return hipGetLastError();
}

}  // namespace spect
