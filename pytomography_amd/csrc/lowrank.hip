// lowrank.hip -- kernels of the projector on combined images (lowrank_body.hpp).
#include "lowrank_body.hpp"

namespace spect {
namespace {

// Adjacent groups of columns per block (their taps share cache lines).
constexpr int kGatherWaves = 4;
__host__ __device__ inline bool zgroups_inside(int Nz) { return Nz % 32 != 0; }

// The blocks of one XCD run through one contiguous part of
// [z group][angle][segment][columns], or, where a z group of the factors does
// not end at a cache line (Nz no multiple of 32), of [angle][segment][columns]
// [z group]: the groups that share lines run together.
template <int ATT, bool VEC>
__global__ __launch_bounds__(kGatherWaves * 64) void lr_gather_kernel(LrGatherJob J, int jgroups, int items) {
  __shared__ LrTap lds[kGatherWaves][64];
  const int b = xcd_piece(blockIdx.x, gridDim.x);
  if (b >= items) return;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), nseg = J.lr.nseg;
  const int r = b / jgroups, q = r / nseg;
  int jg = (b - r * jgroups) * kGatherWaves + wave, zg = q / J.n;
  if (zgroups_inside(J.g.Nz)) {
    zg = jg % J.zgroups;
    jg = jg / J.zgroups;
  }
  if (jg >= J.cgroups) return;
  lr_gather_body<ATT, VEC>(J, q % J.n, r - q * nseg, jg, zg, threadIdx.x & 63, lds[wave]);
}

// Waves of a block of the blurs: four per SIMD, their sums (4 KB each) in 64 KB
// of LDS.
constexpr int kBlurWaves = 15;

// The blocks of one XCD run through one contiguous part of [angle][row range]
// [z tile]: neighbouring z tiles read the same tiles of G.
template <int NT, int ND>
__global__ __launch_bounds__(kBlurWaves * 64) void lr_blur_forward_kernel(LrBlurJob J, int ranges, int items) {
  extern __shared__ __align__(16) unsigned char smem[];
  const int b = xcd_piece(blockIdx.x, gridDim.x), ztiles = J.NzP / 16;
  if (b >= items) return;
  const int zt = b % ztiles, r = b / ztiles;
  lr_blur_forward_body<NT, ND>(J, r / ranges, zt, r % ranges, __builtin_amdgcn_readfirstlane(threadIdx.x >> 6),
                                  blockDim.x >> 6, threadIdx.x & 63, reinterpret_cast<float *>(smem));
}

template <int NT, int ND, bool VEC>
__global__ __launch_bounds__(kBlurWaves * 64) void lr_blur_backward_kernel(LrBackJob J, int items) {
  __shared__ lr_f4 smem[(NT + 2 * ND) * (2 * ND + 1) * 64];
  const int b = xcd_piece(blockIdx.x, gridDim.x), ztiles = J.NzP / 16;
  if (b >= items) return;
  const int zt = b % ztiles, r = b / ztiles;
  lr_blur_backward_body<NT, ND, VEC>(J, r / J.jranges, zt, r % J.jranges,
                                     __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), blockDim.x >> 6,
                                     threadIdx.x & 63, smem);
}

// [angle][segment][column][z block], the waves of a block along the last two:
// they read and write consecutive memory.
template <int ATT, bool VEC>
__global__ __launch_bounds__(256) void lr_field_kernel(LrBackJob J, int jgroups, int items) {
  const int b = xcd_piece(blockIdx.x, gridDim.x);
  if (b >= items) return;
  const int r = b / jgroups, al = r / J.lr.nseg;
  const int w = (b - r * jgroups) * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int jx = w / J.zblocks;
  if (jx >= J.g.je1 - J.g.je0) return;
  lr_field_body<ATT, VEC>(J, al, r - al * J.lr.nseg, jx, w - jx * J.zblocks, threadIdx.x & 63);
}

int xcd_grid(long long items) { return (int)((items + kXcds - 1) / kXcds * kXcds); }

}  // namespace

hipError_t launch_lr_forward(const Geo<float> &g, const Tables<float> &tb, const LrTables &lr, const float *f,
                             const float *attf, const int32_t *angle_idx, int n, float *proj,
                             const float *gm, const float *s, float *pred, float *ratio, float delta,
                             unsigned char *scratch, size_t scratch_bytes, hipStream_t st) {
  if (scratch_bytes < lr_forward_bytes(lr, g, n)) return hipErrorInvalidValue;
  const int NzP = lr_nzp(g.Nz);
  float *G = reinterpret_cast<float *>(scratch);
  int32_t *neg = reinterpret_cast<int32_t *>(scratch + lr_forward_image_bytes(lr, g, n));
  const int zgroups = lr_gather_zgroups(g), cgroups = lr_gather_cgroups(g);
  const LrGatherJob J{g, tb.trig, tb.lin, tb.radius_index, lr, f, attf, angle_idx,
                      n, NzP,     zgroups, cgroups,        G,  neg};
  const bool inside = zgroups_inside(g.Nz);
  const int jgroups = (cgroups * (inside ? zgroups : 1) + kGatherWaves - 1) / kGatherWaves;
  const long long items = (long long)jgroups * lr.nseg * n * (inside ? 1 : zgroups);
  if (items > 0x7ffffff0) return hipErrorInvalidConfiguration;
  const bool vec = g.Nz % 4 == 0;
  auto pick = [&](auto att) {
    constexpr int ATT = decltype(att)::value;
    return vec ? lr_gather_kernel<ATT, true> : lr_gather_kernel<ATT, false>;
  };
  const int mode = lr_factor_mode(g, attf);
  auto kern = mode == kLrStream   ? pick(std::integral_constant<int, kLrStream>{})
              : mode == kLrCached ? pick(std::integral_constant<int, kLrCached>{})
                                  : pick(std::integral_constant<int, 0>{});
  kern<<<xcd_grid(items), kGatherWaves * 64, 0, st>>>(J, jgroups, (int)items);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  const LrBlurJob B{g,  tb.radius_index, lr, angle_idx, n, NzP, zgroups, cgroups, G, neg, proj, gm, s,
                    pred, ratio, delta};
  // Row tiles per block: the halo of a range is two tiles, so long ranges do
  // less work (30 products per output tile with four, 36 with two, 48 with one);
  // short ones when the blocks would not cover the CUs.
  const int nout = g.jo1 - g.jo0, ztiles = NzP / 16;
  auto ranges = [&](int nt) { return (nout + 16 * nt - 1) / (16 * nt); };
  auto launch = [&](auto nt_c, auto nd) {
    constexpr int NT = decltype(nt_c)::value, ND = decltype(nd)::value;
    const int rounds = (lr.nimg + kBlurWaves - 1) / kBlurWaves;
    const int nw = (lr.nimg + rounds - 1) / rounds, items = n * ranges(NT) * ztiles;
    lr_blur_forward_kernel<NT, ND><<<xcd_grid(items), nw * 64, (size_t)nw * NT * 256 * sizeof(float), st>>>(
        B, ranges(NT), items);
  };
  using I1 = std::integral_constant<int, 1>;
  using I2 = std::integral_constant<int, 2>;
  using I4 = std::integral_constant<int, 4>;
  auto with_nd = [&](auto nd) {
    if (n * ranges(2) * ztiles < 256) launch(I1{}, nd);
    else if (n * ranges(4) * ztiles < 224) launch(I2{}, nd);
    else launch(I4{}, nd);
  };
  if (g.H <= 16) with_nd(I1{});
  else with_nd(I2{});
  return hipGetLastError();
}

hipError_t launch_lr_field(const Geo<float> &g, const Tables<float> &tb, const LrTables &lr, const float *proj,
                           const float *attf, const int32_t *angle_idx, int n, float *W, unsigned char *scratch,
                           size_t scratch_bytes, hipStream_t st) {
  if (scratch_bytes < lr_backward_bytes(lr, g, n)) return hipErrorInvalidValue;
  const int n_jext = g.je1 - g.je0, NzP = lr_nzp(g.Nz), zblocks = lr_zblocks(g.Nz);
  const int jranges = lr_back_ranges(g, n);
  float *Q = reinterpret_cast<float *>(scratch);
  int32_t *neg = reinterpret_cast<int32_t *>(scratch + lr_backward_image_bytes(lr, g, n));
  const LrBackJob J{g, tb.trig, tb.lin, tb.radius_index, lr, proj, attf, angle_idx, n, NzP, zblocks,
                    jranges, Q, neg, W};
  const bool vec = g.Nz % 4 == 0;
  {
    const int items = n * jranges * (NzP / 16), rounds = (lr.nimg + kBlurWaves - 1) / kBlurWaves;
    const int nw = (lr.nimg + rounds - 1) / rounds;
    auto pick = [&](auto nt) {
      constexpr int NT = decltype(nt)::value;
      return g.H <= 16 ? (vec ? lr_blur_backward_kernel<NT, 1, true> : lr_blur_backward_kernel<NT, 1, false>)
                       : (vec ? lr_blur_backward_kernel<NT, 2, true> : lr_blur_backward_kernel<NT, 2, false>);
    };
    auto blur = lr_back_tiles(g, n) == kLrBackTiles ? pick(std::integral_constant<int, kLrBackTiles>{})
                                                    : pick(std::integral_constant<int, kLrBackTilesFew>{});
    blur<<<xcd_grid(items), nw * 64, 0, st>>>(J, items);
  }
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  const int jgroups = (n_jext * zblocks + 3) / 4;
  const long long items = (long long)jgroups * lr.nseg * n;
  if (items > 0x7ffffff0) return hipErrorInvalidConfiguration;
  auto pick = [&](auto att) {
    constexpr int ATT = decltype(att)::value;
    return vec ? lr_field_kernel<ATT, true> : lr_field_kernel<ATT, false>;
  };
  const int mode = lr_factor_mode(g, attf);
  auto kern = mode == kLrStream   ? pick(std::integral_constant<int, kLrStream>{})
              : mode == kLrCached ? pick(std::integral_constant<int, kLrCached>{})
                                  : pick(std::integral_constant<int, 0>{});
  kern<<<xcd_grid(items), 256, 0, st>>>(J, jgroups, (int)items);
  return hipGetLastError();
}

}  // namespace spect
