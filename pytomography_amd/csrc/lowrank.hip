// lowrank.hip -- kernels of the projector on combined images (lowrank_body.hpp),
// of one call or of a batch of calls.
#include "lowrank_body.hpp"

namespace spect {
namespace {

// Adjacent groups of columns per block (their taps share cache lines).
constexpr int kGatherWaves = 4;
__host__ __device__ inline bool zgroups_inside(int Nz) { return Nz % 32 != 0; }
__host__ __device__ inline int gather_jgroups(const LrGatherJob &J) {
  return (J.cgroups * (zgroups_inside(J.g.Nz) ? J.zgroups : 1) + kGatherWaves - 1) / kGatherWaves;
}
__host__ __device__ inline int field_jgroups(const LrBackJob &J) {
  return ((J.g.je1 - J.g.je0) * J.zblocks + 3) / 4;
}
__host__ __device__ inline int xcd_grid(int items) { return (items + kXcds - 1) / kXcds * kXcds; }

// The blocks of each pass; a launch (or a call's part of one) holds xcd_grid of
// them, a multiple of the XCDs.
__host__ __device__ inline long long gather_items(const LrGatherJob &J) {
  return (long long)gather_jgroups(J) * J.lr.nseg * J.n * (zgroups_inside(J.g.Nz) ? 1 : J.zgroups);
}
__host__ __device__ inline int blur_ranges(const Geo<float> &g, int nt) {
  return (g.jo1 - g.jo0 + 16 * nt - 1) / (16 * nt);
}
__host__ __device__ inline long long blur_items(const LrBlurJob &J, int nt) {
  return (long long)J.n * blur_ranges(J.g, nt) * (J.NzP / 16);
}
__host__ __device__ inline long long back_items(const LrBackJob &J) {
  return (long long)J.n * J.jranges * (J.NzP / 16);
}
__host__ __device__ inline long long field_items(const LrBackJob &J) {
  return (long long)field_jgroups(J) * J.lr.nseg * J.n;
}

// The blocks of one XCD run through one contiguous part of
// [z group][angle][segment][columns], or, where a z group of the factors does
// not end at a cache line (Nz no multiple of 32), of [angle][segment][columns]
// [z group]: the groups that share lines run together.
template <int ATT, bool VEC>
__device__ __forceinline__ void gather_block(const LrGatherJob &J, int block, LrTap (*lds)[64]) {
  const int items = (int)gather_items(J), b = xcd_piece(block, xcd_grid(items));
  if (b >= items) return;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), nseg = J.lr.nseg, jgroups = gather_jgroups(J);
  const int r = b / jgroups, q = r / nseg;
  int jg = (b - r * jgroups) * kGatherWaves + wave, zg = q / J.n;
  if (zgroups_inside(J.g.Nz)) {
    zg = jg % J.zgroups;
    jg = jg / J.zgroups;
  }
  if (jg >= J.cgroups) return;
  lr_gather_body<ATT, VEC>(J, q % J.n, r - q * nseg, jg, zg, threadIdx.x & 63, lds[wave]);
}

// The blocks of one XCD run through one contiguous part of [angle][row range]
// [z tile]: neighbouring z tiles read the same tiles of G.
template <int NT, int ND>
__device__ __forceinline__ void blur_block(const LrBlurJob &J, int block, unsigned char *smem) {
  const int items = (int)blur_items(J, NT), b = xcd_piece(block, xcd_grid(items)), ztiles = J.NzP / 16;
  if (b >= items) return;
  const int ranges = blur_ranges(J.g, NT), zt = b % ztiles, r = b / ztiles;
  lr_blur_forward_body<NT, ND>(J, r / ranges, zt, r % ranges, __builtin_amdgcn_readfirstlane(threadIdx.x >> 6),
                               blockDim.x >> 6, threadIdx.x & 63, reinterpret_cast<float *>(smem));
}

template <int NT, int ND, bool VEC>
__device__ __forceinline__ void back_block(const LrBackJob &J, int block, lr_f4 *smem) {
  const int items = (int)back_items(J), b = xcd_piece(block, xcd_grid(items)), ztiles = J.NzP / 16;
  if (b >= items) return;
  const int zt = b % ztiles, r = b / ztiles;
  lr_blur_backward_body<NT, ND, VEC>(J, r / J.jranges, zt, r % J.jranges,
                                     __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), blockDim.x >> 6,
                                     threadIdx.x & 63, smem);
}

// [angle][segment][column][z block], the waves of a block along the last two:
// they read and write consecutive memory.
template <int ATT, bool VEC>
__device__ __forceinline__ void field_block(const LrBackJob &J, int block) {
  const int items = (int)field_items(J), b = xcd_piece(block, xcd_grid(items)), jgroups = field_jgroups(J);
  if (b >= items) return;
  const int r = b / jgroups, al = r / J.lr.nseg;
  const int w = (b - r * jgroups) * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int jx = w / J.zblocks;
  if (jx >= J.g.je1 - J.g.je0) return;
  lr_field_body<ATT, VEC>(J, al, r - al * J.lr.nseg, jx, w - jx * J.zblocks, threadIdx.x & 63);
}

// Waves of a block of the blurs: four per SIMD, their sums (4 KB each) in 64 KB
// of LDS.
constexpr int kBlurWaves = 15;
inline int blur_waves(int nimg) {
  const int rounds = (nimg + kBlurWaves - 1) / kBlurWaves;
  return (nimg + rounds - 1) / rounds;
}
inline size_t blur_smem(int waves, int nt) { return (size_t)waves * nt * 256 * sizeof(float); }

template <int ATT, bool VEC>
__global__ __launch_bounds__(kGatherWaves * 64) void lr_gather_kernel(LrGatherJob J) {
  __shared__ LrTap lds[kGatherWaves][64];
  gather_block<ATT, VEC>(J, blockIdx.x, lds);
}
template <int NT, int ND>
__global__ __launch_bounds__(kBlurWaves * 64) void lr_blur_forward_kernel(LrBlurJob J) {
  extern __shared__ __align__(16) unsigned char smem[];
  blur_block<NT, ND>(J, blockIdx.x, smem);
}
template <int NT, int ND, bool VEC>
__global__ __launch_bounds__(kBlurWaves * 64) void lr_blur_backward_kernel(LrBackJob J) {
  __shared__ lr_f4 smem[(NT + 2 * ND) * (2 * ND + 1) * 64];
  back_block<NT, ND, VEC>(J, blockIdx.x, smem);
}
// Eight waves per SIMD cover its stream of factors and W best (58 against 61 us
// with the six that the compiler's registers allow, 15 angles at 128^3).
template <int ATT, bool VEC>
__global__ __launch_bounds__(256, 8) void lr_field_kernel(LrBackJob J) {
  field_block<ATT, VEC>(J, blockIdx.x);
}

// The same blocks of the call that owns a block.
template <typename Job>
__device__ __forceinline__ Job own_job(const Job *jobs, const int *starts, int njobs, int &block) {
  const int j = find_job(starts, njobs, blockIdx.x);
  block = blockIdx.x - ld_uniform(starts + j);
  return ld_uniform_struct(jobs + j);
}
template <int ATT, bool VEC>
__global__ __launch_bounds__(kGatherWaves * 64) void lr_gather_batch_kernel(const LrGatherJob *jobs, const int *starts,
                                                                          int njobs) {
  __shared__ LrTap lds[kGatherWaves][64];
  int block;
  const LrGatherJob J = own_job(jobs, starts, njobs, block);
  gather_block<ATT, VEC>(J, block, lds);
}
template <int NT, int ND>
__global__ __launch_bounds__(kBlurWaves * 64) void lr_blur_forward_batch_kernel(const LrBlurJob *jobs,
                                                                              const int *starts, int njobs) {
  extern __shared__ __align__(16) unsigned char smem[];
  int block;
  const LrBlurJob J = own_job(jobs, starts, njobs, block);
  blur_block<NT, ND>(J, block, smem);
}
template <int NT, int ND, bool VEC>
__global__ __launch_bounds__(kBlurWaves * 64) void lr_blur_backward_batch_kernel(const LrBackJob *jobs,
                                                                               const int *starts, int njobs) {
  __shared__ lr_f4 smem[(NT + 2 * ND) * (2 * ND + 1) * 64];
  int block;
  const LrBackJob J = own_job(jobs, starts, njobs, block);
  back_block<NT, ND, VEC>(J, block, smem);
}
template <int ATT, bool VEC>
__global__ __launch_bounds__(256, 8) void lr_field_batch_kernel(const LrBackJob *jobs, const int *starts, int njobs) {
  int block;
  const LrBackJob J = own_job(jobs, starts, njobs, block);
  field_block<ATT, VEC>(J, block);
}

// Row tiles of a forward wave: the halo of a range is two tiles, so long ranges
// do less work (30 products per output tile with four, 36 with two, 48 with
// one); short ones when the blocks would not cover the CUs.
int forward_tiles(long long blocks2, long long blocks4) { return blocks2 < 256 ? 1 : blocks4 < 224 ? 2 : kLrRowTiles; }
int backward_tiles(long long blocks) { return blocks >= 192 ? kLrBackTiles : kLrBackTilesFew; }

// run(std::integral_constant)... of the variant that the sizes ask for.
template <typename F> void with_att(int mode, F run) {
  if (mode == kLrStream) run(std::integral_constant<int, kLrStream>{});
  else if (mode == kLrCached) run(std::integral_constant<int, kLrCached>{});
  else run(std::integral_constant<int, 0>{});
}
template <typename F> void with_vec(int Nz, F run) {
  if (Nz % 4 == 0) run(std::true_type{});
  else run(std::false_type{});
}
template <typename F> void with_width(int H, F run) {
  if (H <= 16) run(std::integral_constant<int, 1>{});
  else run(std::integral_constant<int, 2>{});
}
template <typename F> void with_row_tiles(int nt, F run) {
  if (nt == 1) run(std::integral_constant<int, 1>{});
  else if (nt == 2) run(std::integral_constant<int, 2>{});
  else run(std::integral_constant<int, kLrRowTiles>{});
}
template <typename F> void with_back_tiles(int nt, F run) {
  if (nt == kLrBackTiles) run(std::integral_constant<int, kLrBackTiles>{});
  else run(std::integral_constant<int, kLrBackTilesFew>{});
}
constexpr long long kMaxItems = 0x7ffffff0;

}  // namespace

LrGatherJob lr_gather_job(const Geo<float> &g, const Tables<float> &tb, const LrTables &lr, const float *f,
                          const float *attf, const int32_t *angle_idx, int n, unsigned char *scratch) {
  return LrGatherJob{g, tb.trig, tb.lin, tb.radius_index, lr, f, attf, angle_idx, n, lr_nzp(g.Nz),
                     lr_gather_zgroups(g), lr_gather_cgroups(g), reinterpret_cast<float *>(scratch),
                     reinterpret_cast<int32_t *>(scratch + lr_forward_image_bytes(lr, g, n))};
}

LrBlurJob lr_blur_job(const LrGatherJob &J, float *proj, const float *gm, const float *s, float *pred, float *ratio,
                      float delta) {
  return LrBlurJob{J.g, J.radius_index, J.lr, J.angle_idx, J.n, J.NzP, J.zgroups, J.cgroups, J.G, J.neg,
                   proj, gm, s, pred, ratio, delta};
}

LrBackJob lr_back_job(const Geo<float> &g, const Tables<float> &tb, const LrTables &lr, const float *proj,
                      const float *attf, const int32_t *angle_idx, int n, float *W, unsigned char *scratch) {
  return LrBackJob{g, tb.trig, tb.lin, tb.radius_index, lr, proj, attf, angle_idx, n, lr_nzp(g.Nz),
                   lr_zblocks(g.Nz), lr_back_ranges(g, kLrBackTilesFew), reinterpret_cast<float *>(scratch),
                   reinterpret_cast<int32_t *>(scratch + lr_backward_image_bytes(lr, g, n)), W};
}

hipError_t launch_lr_forward(const LrGatherJob &J, const LrBlurJob &B, size_t scratch_bytes, hipStream_t st) {
  if (scratch_bytes < lr_forward_bytes(J.lr, J.g, J.n)) return hipErrorInvalidValue;
  const int nt = forward_tiles(blur_items(B, 2), blur_items(B, 4)), waves = blur_waves(J.lr.nimg);
  if (gather_items(J) > kMaxItems || blur_items(B, nt) > kMaxItems) return hipErrorInvalidConfiguration;
  with_att(lr_factor_mode(J.g, J.attf), [&](auto att) {
    with_vec(J.g.Nz, [&](auto vec) {
      lr_gather_kernel<decltype(att)::value, decltype(vec)::value>
          <<<xcd_grid((int)gather_items(J)), kGatherWaves * 64, 0, st>>>(J);
    });
  });
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  with_row_tiles(nt, [&](auto t) {
    with_width(J.g.H, [&](auto nd) {
      lr_blur_forward_kernel<decltype(t)::value, decltype(nd)::value>
          <<<xcd_grid((int)blur_items(B, nt)), waves * 64, blur_smem(waves, nt), st>>>(B);
    });
  });
  return hipGetLastError();
}

hipError_t launch_lr_field(LrBackJob J, size_t scratch_bytes, hipStream_t st) {
  if (scratch_bytes < lr_backward_bytes(J.lr, J.g, J.n)) return hipErrorInvalidValue;
  J.jranges = lr_back_ranges(J.g, kLrBackTiles);
  const int nt = backward_tiles(back_items(J)), waves = blur_waves(J.lr.nimg);
  J.jranges = lr_back_ranges(J.g, nt);
  if (back_items(J) > kMaxItems || field_items(J) > kMaxItems) return hipErrorInvalidConfiguration;
  with_vec(J.g.Nz, [&](auto vec) {
    with_back_tiles(nt, [&](auto t) {
      with_width(J.g.H, [&](auto nd) {
        lr_blur_backward_kernel<decltype(t)::value, decltype(nd)::value, decltype(vec)::value>
            <<<xcd_grid((int)back_items(J)), waves * 64, 0, st>>>(J);
      });
    });
  });
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  with_att(lr_factor_mode(J.g, J.attf), [&](auto att) {
    with_vec(J.g.Nz, [&](auto vec) {
      lr_field_kernel<decltype(att)::value, decltype(vec)::value><<<xcd_grid((int)field_items(J)), 256, 0, st>>>(J);
    });
  });
  return hipGetLastError();
}

bool lr_batch_finish(LrBatch &b) {
  long long two = 0, four = 0, back = 0, samples = 0;
  size_t field = 0;
  int nimg = 0;
  for (size_t i = 0; i < b.gather.size(); ++i) {
    const Geo<float> &g = b.gather[i].g;
    two += blur_items(b.blur[i], 2);
    four += blur_items(b.blur[i], 4);
    b.back[i].jranges = lr_back_ranges(g, kLrBackTiles);
    back += back_items(b.back[i]);
    samples += lr_back_samples(g, b.back[i].n);
    nimg = std::max(nimg, b.gather[i].lr.nimg);
    field += (size_t)g.A * g.P * (g.je1 - g.je0) * g.Nz * sizeof(float);
  }
  b.row_tiles = forward_tiles(two, four);
  b.back_tiles = backward_tiles(back);
  b.back_pays = samples >= kLrBackSamples;
  b.waves = blur_waves(nimg);
  b.H = b.gather[0].g.H;
  b.Nz = b.gather[0].g.Nz;
  b.factor_mode = lr_factor_mode(b.Nz, b.gather[0].attf, field);
  long long tot[4] = {0, 0, 0, 0};
  for (auto &s : b.starts) s.clear();
  for (size_t i = 0; i < b.gather.size(); ++i) {
    b.back[i].jranges = lr_back_ranges(b.gather[i].g, b.back_tiles);
    const long long items[4] = {gather_items(b.gather[i]), blur_items(b.blur[i], b.row_tiles), back_items(b.back[i]),
                                field_items(b.back[i])};
    for (int q = 0; q < 4; ++q) {
      b.starts[q].push_back((int)tot[q]);
      tot[q] += (items[q] + kXcds - 1) / kXcds * kXcds;
      if (tot[q] > kMaxItems) return false;
    }
  }
  for (int q = 0; q < 4; ++q) b.blocks[q] = (int)tot[q];
  return true;
}

hipError_t launch_lr_batch_forward(const LrBatch &b, const LrGatherJob *gather, const LrBlurJob *blur,
                                   const int *gather_starts, const int *blur_starts, hipStream_t st) {
  const int njobs = (int)b.gather.size();
  with_att(b.factor_mode, [&](auto att) {
    with_vec(b.Nz, [&](auto vec) {
      lr_gather_batch_kernel<decltype(att)::value, decltype(vec)::value>
          <<<b.blocks[0], kGatherWaves * 64, 0, st>>>(gather, gather_starts, njobs);
    });
  });
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  with_row_tiles(b.row_tiles, [&](auto t) {
    with_width(b.H, [&](auto nd) {
      lr_blur_forward_batch_kernel<decltype(t)::value, decltype(nd)::value>
          <<<b.blocks[1], b.waves * 64, blur_smem(b.waves, b.row_tiles), st>>>(blur, blur_starts, njobs);
    });
  });
  return hipGetLastError();
}

hipError_t launch_lr_batch_field(const LrBatch &b, const LrBackJob *back, const int *blur_starts,
                                 const int *field_starts, hipStream_t st) {
  const int njobs = (int)b.back.size();
  with_vec(b.Nz, [&](auto vec) {
    with_back_tiles(b.back_tiles, [&](auto t) {
      with_width(b.H, [&](auto nd) {
        lr_blur_backward_batch_kernel<decltype(t)::value, decltype(nd)::value, decltype(vec)::value>
            <<<b.blocks[2], b.waves * 64, 0, st>>>(back, blur_starts, njobs);
      });
    });
  });
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  with_att(b.factor_mode, [&](auto att) {
    with_vec(b.Nz, [&](auto vec) {
      lr_field_batch_kernel<decltype(att)::value, decltype(vec)::value>
          <<<b.blocks[3], 256, 0, st>>>(back, field_starts, njobs);
    });
  });
  return hipGetLastError();
}

}  // namespace spect
