// lowrank_launch.hpp -- job descriptors and launchers of the projector on
// combined images (lowrank_body.hpp, lowrank.hip).
#pragma once

#include <vector>

#include "common.hpp"

namespace spect {

constexpr int kLrRowsDev = 16;  // image rows of a segment in G and Q (kLrRows)

// Device tables of the images of every radius (lowrank.hpp).
struct LrTables {
  int nseg;    // segments per radius (short ones padded with empty segments)
  int nimg;    // most images of a radius
  int quads;   // groups of four planes, a multiple of four
  const int32_t *seg_unit;  // [n_radii][nseg + 1] 16-plane units
  const int32_t *seg_rows;  // [n_radii][nseg] image rows in use
  const int32_t *count;     // [n_radii] images
  const int4 *img;          // [n_radii][nimg] (segment, row, half width, 0)
  const float *taps;        // [n_radii][nimg][2][2 (16 ND + 15) + 1] node taps, z then y
  // plane weights in the lane order of the products' A operand:
  const float *cf;  // [n_radii][quads][64]: plane 4 q + l / 16, image row l % 16
  const float *cb;  // [n_radii][quads / 4][4][64]: plane 16 u + l % 16, row 4 s + l / 16
};

struct LrGatherJob {
  Geo<float> g;
  const float2 *trig;
  const float *lin;
  const int32_t *radius_index;
  LrTables lr;
  const float *f;
  const float *attf;  // attenuation factors [A][P][je1-je0][Nz], or null
  const int32_t *angle_idx;
  int n, NzP, zgroups, cgroups;
  float *G;       // [n][nseg][16] images (lr_image_floats)
  int32_t *neg;   // [n][nseg][zgroups][cgroups]: a sample was negative
};

struct LrBlurJob {
  Geo<float> g;
  const int32_t *radius_index;
  LrTables lr;
  const int32_t *angle_idx;
  int n, NzP, zgroups, cgroups;
  const float *G;
  const int32_t *neg;
  float *proj;
  const float *gm, *s;
  float *pred, *ratio;
  float delta;
};

struct LrBackJob {
  Geo<float> g;
  const float2 *trig;
  const float *lin;
  const int32_t *radius_index;
  LrTables lr;
  const float *proj;
  const float *attf;
  const int32_t *angle_idx;
  int n, NzP, zblocks, jranges;
  float *Q;      // [n][nseg][16] images (lr_image_floats)
  int32_t *neg;  // [n][jranges][NzP / 16]: a projection value was negative
  float *W;      // [n][P][je1-je0][Nz]
};

// Output row tiles per wave of the blurs: at most kLrRowTiles forward,
// kLrBackTiles backward, fewer when the blocks would not cover the chip.
constexpr int kLrRowTiles = 4, kLrBackTiles = 5, kLrBackTilesFew = 2;

inline int lr_nzp(int Nz) { return (Nz + 15) / 16 * 16; }
inline int lr_zblocks(int Nz) { return (Nz + 63) / 64; }
// Whether an n-angle back projection is faster on combined images: three launches
// instead of two, so not with few detector samples.  Plane by plane / combined,
// with attenuation: 64^3 x 4 angles 27.3 / 27.5 us, x 8 35.4 / 33.3, x 16
// 46.6 / 39.7; 80^3 x 4 31.1 / 34.9, x 8 42.9 / 39.2; 128^3 x 2 33.3 / 38.3,
// x 4 49.6 / 43.9, x 16 144 / 108.  (The forward's two launches replace two:
// 64^3 x 2 27.8 / 19.4, 128^3 x 16 105 / 85.)  The line lies between 128^3 x 2
// (39936 samples of the extended detector) and 64^3 x 8 (43008).
constexpr long long kLrBackSamples = 41000;
inline long long lr_back_samples(const Geo<float> &g, int n) { return (long long)n * (g.je1 - g.je0) * g.Nz; }
inline bool lr_back_pays(const Geo<float> &g, int n) { return lr_back_samples(g, n) >= kLrBackSamples; }

// Columns and z of a wave in the first forward pass (lr_gather_body).
constexpr int kLrGatherCols = 2;
inline int lr_gather_cgroups(const Geo<float> &g) {
  const int cw = g.Nz % 4 == 0 ? kLrGatherCols : 1;
  return (g.je1 - g.je0 + cw - 1) / cw;
}
inline int lr_gather_zgroups(const Geo<float> &g) {
  const int z = g.Nz % 4 == 0 ? 64 / kLrGatherCols : 64;
  return (g.Nz + z - 1) / z;
}

// How the passes over planes read the attenuation factors: kLrStream past the
// caches, which leaves those to the object and the images, kLrCached where that
// costs more: waves that share cache lines (z pieces that do not end at one), or
// a field of all angles that stays in the 256 MB last-level cache between calls.
// OSEM, cached / streamed: 128^3 x 120 angles 1743 / 1638 us, 192^3 x 180 8283 /
// 8099, 100^2 x 47 655 / 731, 64^3 x 60 518 / 528.
constexpr int kLrCached = 1, kLrStream = 2;
inline int lr_factor_mode(int Nz, const float *attf, size_t field_bytes) {
  if (!attf) return 0;
  return Nz % 32 != 0 || field_bytes <= (size_t)256 << 20 ? kLrCached : kLrStream;
}
inline int lr_factor_mode(const Geo<float> &g, const float *attf) {
  return lr_factor_mode(g.Nz, attf, (size_t)g.A * g.P * (g.je1 - g.je0) * g.Nz * sizeof(float));
}

// An image is stored in tiles of 16 columns j x 16 z, the blurs' unit, each
// 1 KB contiguous (a tile of rows of z would use half of every cache line it
// touches).  Rows of tiles: the detector columns start a tile, so that the
// forward's tiles are aligned with its outputs; the extended columns before
// them end the kLrLead tiles before.
constexpr int kLrLead = 2;
__host__ __device__ inline int lr_row_tiles(int nout) { return (nout + 15) / 16 + 2 * kLrLead; }
__host__ __device__ inline size_t lr_image_floats(const Geo<float> &g, int NzP) {
  return (size_t)lr_row_tiles(g.jo1 - g.jo0) * 16 * NzP;
}
// Offset of extended column jx (0 = je0), z.
__host__ __device__ inline uint32_t lr_image_at(const Geo<float> &g, int NzP, int jx, int z) {
  const uint32_t j = (uint32_t)(jx + g.je0 - g.jo0 + 16 * kLrLead);
  return ((j >> 4) * (uint32_t)(NzP >> 4) + ((uint32_t)z >> 4)) * 256u + (j & 15u) * 16u + ((uint32_t)z & 15u);
}
// First tile row that holds an extended column, and tile rows from it to the last.
__host__ __device__ inline int lr_first_tile(const Geo<float> &g) { return kLrLead - (g.jo0 - g.je0 + 15) / 16; }
inline int lr_back_rows(const Geo<float> &g) { return (g.jo0 - g.je0 + 15) / 16 + (g.je1 - g.jo0 + 15) / 16; }
inline int lr_back_ranges(const Geo<float> &g, int nt) { return (lr_back_rows(g) + nt - 1) / nt; }
// Row tiles after the last image that the forward's blur may read (and ignore).
constexpr int kLrPadTiles = kLrRowTiles;

// Bytes of the images and flags of an n-angle call.
inline size_t lr_align(size_t b) { return (b + 255) & ~size_t(255); }
inline size_t lr_image_bytes(const LrTables &lr, const Geo<float> &g, int n) {
  return lr_align((size_t)n * lr.nseg * kLrRowsDev * lr_image_floats(g, lr_nzp(g.Nz)) * sizeof(float));
}
inline size_t lr_pad_bytes(const Geo<float> &g) { return (size_t)kLrPadTiles * 16 * lr_nzp(g.Nz) * sizeof(float); }
inline size_t lr_forward_image_bytes(const LrTables &lr, const Geo<float> &g, int n) {
  return lr_image_bytes(lr, g, n) + lr_pad_bytes(g);
}
inline size_t lr_forward_bytes(const LrTables &lr, const Geo<float> &g, int n) {
  return lr_forward_image_bytes(lr, g, n) +
         lr_align((size_t)n * lr.nseg * lr_gather_zgroups(g) * lr_gather_cgroups(g) * sizeof(int32_t));
}
inline size_t lr_backward_image_bytes(const LrTables &lr, const Geo<float> &g, int n) {
  return lr_image_bytes(lr, g, n);
}
// (flags for the most ranges, so that a launch may choose its tiles)
inline size_t lr_backward_bytes(const LrTables &lr, const Geo<float> &g, int n) {
  return lr_backward_image_bytes(lr, g, n) +
         lr_align((size_t)n * lr_back_ranges(g, kLrBackTilesFew) * (lr_nzp(g.Nz) / 16) * sizeof(int32_t));
}

// The descriptors of one call.  scratch: lr_forward_bytes / lr_backward_bytes.
LrGatherJob lr_gather_job(const Geo<float> &g, const Tables<float> &tb, const LrTables &lr, const float *f,
                          const float *attf, const int32_t *angle_idx, int n, unsigned char *scratch);
LrBlurJob lr_blur_job(const LrGatherJob &J, float *proj, const float *gm, const float *s, float *pred, float *ratio,
                      float delta);
// W[n][P][je1-je0][Nz], every entry that the gathers read
LrBackJob lr_back_job(const Geo<float> &g, const Tables<float> &tb, const LrTables &lr, const float *proj,
                      const float *attf, const int32_t *angle_idx, int n, float *W, unsigned char *scratch);

// Scratch smaller than that is refused.
hipError_t launch_lr_forward(const LrGatherJob &J, const LrBlurJob &B, size_t scratch_bytes, hipStream_t st);
hipError_t launch_lr_field(LrBackJob J, size_t scratch_bytes, hipStream_t st);

// The four passes of several calls with one Nz and one class of half widths
// (H <= 16 or not), all with attenuation factors or all without, in one launch
// each.
// back_pays: whether the launch's samples make the back projection on images
// the faster one (lr_back_pays, of all calls together).
struct LrBatch {
  std::vector<LrGatherJob> gather;
  std::vector<LrBlurJob> blur;
  std::vector<LrBackJob> back;
  std::vector<int> starts[4];  // first block of each call: gather, blur, back blur, field
  int blocks[4];
  int row_tiles, back_tiles, waves, factor_mode, H, Nz;
  bool back_pays;
};
// Fills everything that follows from gather, blur and back.
bool lr_batch_finish(LrBatch &b);
// Descriptors and starts in device memory.
hipError_t launch_lr_batch_forward(const LrBatch &b, const LrGatherJob *gather, const LrBlurJob *blur,
                                   const int *gather_starts, const int *blur_starts, hipStream_t st);
hipError_t launch_lr_batch_field(const LrBatch &b, const LrBackJob *back, const int *blur_starts,
                                 const int *field_starts, hipStream_t st);

}  // namespace spect
