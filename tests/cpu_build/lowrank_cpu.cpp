// CPU build of the projector on combined images: the wave bodies of
// pytomography_amd/csrc/lowrank_body.hpp, one wave of 64 std::threads per
// block, with the 16x16x4 matrix product emulated in the documented lane
// layout.  Images, W and LDS start as NaN, so a read of an entry that no lane
// wrote shows in the output.
//
//   lowrank_cpu <dir> <row tiles>  (problem files as in cpu_runtime.hpp, plus f.bin
//       float32 [N][N][Nz] and p.bin float32 [n_sel][N][Nz]); writes
//       <dir>/proj.bin (forward of f) and <dir>/bp.bin (reference back
//       projection of p) and prints "segments .. images .. uncovered ..":
//       columns' planes that in_footprint finds and lr_column_planes does not.
#include "cpu_attenuation.hpp"

struct int4 {
  int x, y, z, w;
};
inline unsigned __umul24(unsigned a, unsigned b) {
  if ((a >> 24) || (b >> 24)) std::abort();
  return a * b;
}

#define SPECT_CPU_MFMA
typedef float lr_f4 __attribute__((vector_size(16)));
static float g_mfma_a[1024], g_mfma_b[1024];
inline lr_f4 lr_mfma(float a, float b, lr_f4 c) {
  const unsigned l = threadIdx.x & 63u, w = threadIdx.x & ~63u;
  g_mfma_a[w + l] = a;
  g_mfma_b[w + l] = b;
  cpu_block_barrier->arrive_and_wait();
  for (int r = 0; r < 4; ++r)
    for (int k = 0; k < 4; ++k) c[r] += g_mfma_a[w + 16 * k + 4 * (l >> 4) + r] * g_mfma_b[w + 16 * k + (l & 15)];
  cpu_block_barrier->arrive_and_wait();
  return c;
}
inline lr_f4 lr_load4_stream(const float *p, uint32_t byte) {
  return *reinterpret_cast<const lr_f4 *>(reinterpret_cast<const char *>(p) + byte);
}
inline float lr_load1_stream(const float *p, uint32_t byte) {
  return *reinterpret_cast<const float *>(reinterpret_cast<const char *>(p) + byte);
}

inline void lr_fence() {}
inline void lr_wave_sync() { cpu_block_barrier->arrive_and_wait(); }

#include "lowrank.hpp"
#include "lowrank_body.hpp"
#include "backward_body.hpp"

using namespace spect;

int main(int argc, char **argv) {
  if (argc != 3) return 2;
  const std::string dir = argv[1];
  const cpu_build::Problem p = cpu_build::load_problem(dir);
  const Geo<float> &g = p.g;
  const int n = p.n, row_tiles = std::atoi(argv[2]), n_jext = g.je1 - g.je0, NzP = lr_nzp(g.Nz), zb = lr_zblocks(g.Nz);
  const auto f = cpu_build::read_file<float>(dir + "/f.bin", (size_t)g.N * g.N * g.Nz);
  const auto pr = cpu_build::read_file<float>(dir + "/p.bin", (size_t)n * g.N * g.Nz);
  const cpu_build::Attenuation att = cpu_build::build_attenuation(p);
  LrHostTables t;
  if (!lowrank_tables<float>(p.taps_r.data(), p.taps_z.data(), p.n_radii, g.P, g.H, t)) return 3;
  const LrTables lr{t.nseg, t.nimg, t.quads, t.seg_unit.data(), t.seg_rows.data(), t.count.data(),
                    reinterpret_cast<const int4 *>(t.img.data()), t.taps.data(), t.cf.data(), t.cb.data()};
  size_t uncovered = 0;
  for (int al = 0; al < n; ++al)
    for (int jx = 0; jx < n_jext; ++jx) {
      int lo, hi;
      lr_column_planes(g, p.trig[p.sel[al]], p.lin[g.je0 + jx], lo, hi);
      for (int i = 0; i < g.P; ++i) {
        float ix, iy;
        rot_coord<float>(p.trig[p.sel[al]].x, p.trig[p.sel[al]].y, p.lin[g.je0 + jx], p.lin[i], g.half, ix, iy);
        if (in_footprint<float>(ix, iy, g) && (i < lo || i > hi)) ++uncovered;
      }
    }
  const float nan = std::numeric_limits<float>::quiet_NaN();
  const int parts = lr.nseg;
  // exact sizes (not rounded up to whole cache lines), so that an access past
  // the end is one the sanitizer sees
  std::vector<float> Gpad((size_t)n * parts * kLrRowsDev * lr_image_floats(g, NzP) + lr_pad_bytes(g) / sizeof(float), nan), proj((size_t)n * g.N * g.Nz, nan);
  float *G = Gpad.data();
  const int zgroups = lr_gather_zgroups(g), cgroups = lr_gather_cgroups(g);
  std::vector<int32_t> neg((size_t)n * parts * zgroups * cgroups, 0);
  const bool vec = g.Nz % 4 == 0;
  std::vector<unsigned char> smem((size_t)kLrRowTiles * 256 * sizeof(float));
  const LrGatherJob J{g, p.trig.data(), p.lin.data(), p.ridx.data(), lr, f.data(), att.attf, p.sel.data(), n,
                      NzP, zgroups, cgroups, G, neg.data()};
  auto lane = [] { return (int)(threadIdx.x & 63u); };
  static LrTap lds[64];
  cpu_build::run_grid(n * parts, cgroups, zgroups, 64, smem, [&](int b, int jg, int z, unsigned char *) {
    if (att.attf) vec ? lr_gather_body<kLrCached, true>(J, b / parts, b % parts, jg, z, lane(), lds)
                      : lr_gather_body<kLrStream, false>(J, b / parts, b % parts, jg, z, lane(), lds);
    else vec ? lr_gather_body<0, true>(J, b / parts, b % parts, jg, z, lane(), lds)
             : lr_gather_body<0, false>(J, b / parts, b % parts, jg, z, lane(), lds);
  });
  const LrBlurJob B{g, p.ridx.data(), lr, p.sel.data(), n, NzP, zgroups, cgroups, G, neg.data(), proj.data(),
                    nullptr, nullptr, nullptr, nullptr, 0.0f};
  auto blur = [&](auto nt, auto nd) {
    constexpr int NT = decltype(nt)::value;
    cpu_build::run_grid(n, NzP / 16, (g.N + 16 * NT - 1) / (16 * NT), 64, smem, [&](int al, int zt, int r, unsigned char *s) {
      lr_blur_forward_body<NT, decltype(nd)::value>(B, al, zt, r, 0, 1, lane(), reinterpret_cast<float *>(s));
    });
  };
  using I1 = std::integral_constant<int, 1>;
  using I2 = std::integral_constant<int, 2>;
  using I4 = std::integral_constant<int, 4>;
  auto with_nd = [&](auto nd) {
    if (row_tiles == 1) blur(I1{}, nd);
    else if (row_tiles == 2) blur(I2{}, nd);
    else blur(I4{}, nd);
  };
  if (g.H <= 16) with_nd(I1{});
  else with_nd(I2{});
  cpu_build::write_file(dir + "/proj.bin", proj);

  const int back_tiles = row_tiles == 4 ? kLrBackTiles : kLrBackTilesFew;
  const int jranges = (lr_back_rows(g) + back_tiles - 1) / back_tiles;
  std::vector<float> Q((size_t)n * lr.nseg * kLrRowsDev * lr_image_floats(g, NzP), nan), W((size_t)n * g.P * n_jext * g.Nz, nan);
  std::vector<int32_t> bneg((size_t)n * jranges * (NzP / 16), 0);
  const LrBackJob K{g, p.trig.data(), p.lin.data(), p.ridx.data(), lr, pr.data(), att.attf, p.sel.data(), n,
                    NzP, zb, jranges, Q.data(), bneg.data(), W.data()};
  auto back = [&](auto nt, auto nd) {
    constexpr int NT = decltype(nt)::value, ND = decltype(nd)::value;
    std::vector<unsigned char> tiles((NT + 2 * ND) * (2 * ND + 1) * 64 * sizeof(lr_f4));
    cpu_build::run_grid(n, jranges, NzP / 16, 64, tiles, [&](int al, int jr, int zt, unsigned char *s) {
      lr_f4 *t = reinterpret_cast<lr_f4 *>(s);
      vec ? lr_blur_backward_body<NT, ND, true>(K, al, zt, jr, 0, 1, lane(), t)
          : lr_blur_backward_body<NT, ND, false>(K, al, zt, jr, 0, 1, lane(), t);
    });
  };
  auto back_nd = [&](auto nd) {
    if (back_tiles == kLrBackTiles) back(std::integral_constant<int, kLrBackTiles>{}, nd);
    else back(std::integral_constant<int, kLrBackTilesFew>{}, nd);
  };
  if (g.H <= 16) back_nd(I1{});
  else back_nd(I2{});
  cpu_build::run_grid(n * parts, n_jext, zb, 64, smem, [&](int b, int jx, int z, unsigned char *) {
    if (att.attf) vec ? lr_field_body<kLrCached, true>(K, b / parts, b % parts, jx, z, lane())
                      : lr_field_body<kLrStream, false>(K, b / parts, b % parts, jx, z, lane());
    else vec ? lr_field_body<0, true>(K, b / parts, b % parts, jx, z, lane())
             : lr_field_body<0, false>(K, b / parts, b % parts, jx, z, lane());
  });
  std::vector<float> out((size_t)g.N * g.N * g.Nz, nan);
  GatherJob<float> GJ{};
  GJ.g = g;
  GJ.tb = p.tables();
  GJ.W = W.data();
  GJ.angle_idx = p.sel.data();
  GJ.n = n;
  GJ.out_mode = SPECT_OUT_STORE;
  GJ.out = out.data();
  constexpr int ZV = gather_zv<float>();
  const size_t lanes = (size_t)g.N * g.N * ((g.Nz + ZV - 1) / ZV);
  for (size_t q = 0; q < lanes; ++q) gather_body<float, ZV, 0>(GJ, q);
  cpu_build::write_file(dir + "/bp.bin", out);
  std::printf("segments %d images %d uncovered %zu\n", lr.nseg, lr.nimg, uncovered);
  return 0;
}
