// Rules of the launches that need no device: which form of a kernel a call's sizes
// take.  Host code without HIP, so that tests check them by themselves.
#pragma once
#include <cmath>
#include <cstdint>

namespace fdk {
namespace rules {

// Forms of the row filter: the in-place kernel, filter_wide_kernel with 32-bit offsets
// in a view, and with every point outside its row left out before the store.
enum FilterForm { kFilterInPlace = 0, kFilterWide = 1, kFilterWideFar = 2 };

// filter_wide_kernel (N = 2^7 .. 2^14) stores a thread's point u of a transposed FP32
// view at byte 4 (u nrows + row) mod 2^32 and lets the view's resource drop the points
// outside the row, u = 1 - N/16 .. -1 and nu .. nu + N/16 - 2.  They fall outside the
// view up to (nu + N/16) nrows = 2^30; past that (views much shorter than N of a million
// rows) some would wrap into it.  The resource itself spans less than 2 GiB.  Row-major
// stores have a resource a row, 16-bit stores 64-bit addresses, so they have no such limit.
inline FilterForm filter_form(int nu, int nrows, int nviews, int log_n, bool transposed_f32) {
  if (log_n < 7 || log_n > 14) return kFilterInPlace;
  if ((int64_t)(nrows + 64) * nviews >= (int64_t)1 << 29) return kFilterInPlace;  // the kernel's ints
  if (transposed_f32 && ((int64_t)nu * nrows * 4 >= (int64_t)1 << 31 ||
                         (int64_t)(nu + (1 << log_n) / 16) * nrows * 4 > (int64_t)1 << 32))
    return kFilterWideFar;
  return kFilterWide;
}

// Columns of a wave's strip in bp_wave_kernel's LDS: the v extent of a run of 64 zpt
// voxels at dvz pixels a voxel, with room for floor rounding and the 4-column alignment
// of its start, then the two-column zero slot.  A column is `sides` floats; the strips of
// a block's waves follow each other, so theirs are a multiple of 4 floats, which keeps
// the 16-byte stores of every wave aligned.  0: no such strip.
inline int wave_strip_columns(double dvz, int zpt, int sides) {
  const double span = dvz * (64 * zpt - 1);
  const double quads = (std::ceil(span) + 9) / 4 + 1;
  return quads < 1e6 ? 4 * (int)quads + (sides == 2 ? 2 : 4) : 0;
}

// A run of bp_wave_kernel: voxels per lane (0: no strip fits), its strip's columns, and
// the vector instructions per view of a slab's runs.
struct WaveRun {
  int zpt, columns;
  double cost;
};

// Voxels per lane: of the values whose strips fit, the one with the least vector
// instructions per view for a column of zext voxels.  A run of 64 zpt voxels costs about
// fixed + staged quad slots + taps, and 95 once a launch.  Forced values (1 / 2 / 4 / 8)
// agree, a pass of 32 FP32 views of n^2 into n^3: 1024, pair 30.7 / 15.9 / 10.9 / 9.9 ms;
// 512, pair 3.84 / 2.00 / 1.26 / 1.77 ms; 256, pair 470 / 243 / 268 / 431 us; 256, one slab
// 536 / 286 / 181 / 281 us.
inline WaveRun wave_run(double dvz, int zext, int sides, int nproj, int forced) {
  constexpr int kZpt[4] = {8, 4, 2, 1}, kSlots[4] = {3, 2, 1, 1};
  WaveRun best{0, 0, 0.0};
  for (int k = 0; k < 4; ++k) {
    const int z = kZpt[k], columns = wave_strip_columns(dvz, z, sides);
    if (columns <= 0 || (columns - 2) / 4 > 64 * kSlots[k] || 16LL * columns * sides > 60 * 1024) continue;
    const int runs = (zext + 64 * z - 1) / (64 * z);
    const double cost = runs * (25 + 10 * sides * kSlots[k] + z * (sides == 2 ? 9 : 7) + 95.0 / nproj);
    if (forced ? z == forced : (!best.zpt || cost < best.cost)) best = {z, columns, cost};
  }
  return best;
}

// Whether runs of single slabs beat the block-strip and gather kernels.  Those take
// about 35 instructions a view and 64 voxels, in groups of 256.  Where a voxel step covers
// two samples and more, only strips of one voxel a lane fit: 256^3 from 4 FP32 views of
// 513^2 67.5 us by the gather kernel, 126 by runs, from 32 459 and 545, 512^3 from 32 of
// 1025^2 3.80 and 4.59 ms.  Single views: 256^3 pair from one of 257^2 41.8 and 47.6 us,
// 512^3 pair 345 and 321, 300^3 64.5 and 54.5, 128^3 pair 11.1 and 13.1.  `least`: by how
// much, where the runs need their views copied first (160^3 pair from 4 views of 321^2
// 48 us, 59 with a copy).
inline bool wave_run_pays(const WaveRun& r, int zext, int nproj, double least = 1.0) {
  if (!r.zpt || (nproj == 1 && zext <= 64)) return false;
  return r.cost * least <= 35.0 * 4 * ((zext + 255) / 256);
}

// Whether 16-bit views with odd rows are worth copying to rows of a multiple of 4
// samples, so that bp_wave_kernel takes them: columns of zext voxels in `slabs` slabs,
// `nproj` views of `view` samples.  Per view and slab the gather kernel takes about
// 0.5 us + 0.18 ns a wave more than nothing, the wave-strip kernel half of the latter;
// the copy, its event and launch cost 14 us, and 4 bytes a sample at about 1 TB/s.  FP16
// cubes of n^3 from views of (n + 1)^2, gather against copy, us: 48, pair, 32 views 68 / 28;
// 96, pair, 4 views 20.3 / 22.4, 8 views 36.8 / 27.9; 160, one slab, 3 views 21.6 / 24.7;
// 256, pair, 4 views 134 / 85; 512, 32 views 3950 / 1650.  One view never pays (256: 31 / 41).
inline bool pitched_copy_pays(double columns, int zext, int slabs, int nproj, double view) {
  const double waves = columns * ((zext + 511) / 512);
  const double save = (double)nproj * slabs * (0.5e-6 + 0.09e-9 * waves);
  return nproj > 1 && save > 14e-6 + view * nproj * 4 / 1e12;
}

// Which march of the forward projector is the faster: fp_kernel through the volume
// itself or fp_zfast_kernel through its padded copy.
struct March {
  int nu, nv;               // detector, pitch dv, the volume's mid plane on row cv
  double cv, dv, mag;       // magnification of the volume's centre
  int nx, ny, nz;
  double vx, vy, vz, step;  // mm
  int views;
  double sum_sin, max_sin;  // of |sin angle| over the views
};

// fp_zfast_kernel's waves are 64 rows of a column, and cost what 64 rays do however many
// of them are on the detector and meet the volume: 0.95 ps a lane and sample, at least
// 0.15 us a sample of a ray (its samples are a chain), plus 16 us and 12 bytes a voxel at
// 2.8 TB/s for the copy.  A copy above what the scratch list keeps is mapped for the call:
// 17 to 56 ms a GB where the caller waits between calls.  fp_kernel's waves are 64 columns
// of a row: 0.7 ps a lane and sample where rays run along y to 7.4 where they run along x,
// its chain 0.13 to 0.39 us a sample, more in rows over 256 voxels.  The constants give
// fp_kernel where it measured faster, at 400 sizes, to 5 % or 2 us.  Measured, 256^3 at
// half-voxel steps, fp_kernel / fp_zfast_kernel: 24 views of 256 x 64 round the scan 1216 /
// 260 us, 60 of 256 x 16 686 / 524, 360 of 256 x 8 1902 / 2400, 360 of 256 x 1 268 / 2400,
// 2 of 256 x 200 near 0 degrees 124 / 152; 80^3 at whole steps, 4 views 19.4 / 29.6.
inline bool zfast_pays(const March& m, double copy_bytes, double kept_bytes) {
  const double across = std::sqrt(m.nx * m.vx * m.nx * m.vx + m.ny * m.vy * m.ny * m.vy);
  const double samples = 0.6 * across / m.step;  // a ray's, about
  const double shadow = 0.6 * m.nz * m.vz * m.mag / m.dv + 1;  // half the volume's height in rows
  const double r0 = std::fmax(0.0, m.cv + 0.5 - shadow), r1 = std::fmin((double)m.nv, m.cv + 0.5 + shadow);
  if (!(r1 - r0 >= 16)) return false;
  const double waves = (std::ceil(r1 / 64) - std::floor(r0 / 64)) * m.nu;
  const double rays = (r1 - r0) * 64 * std::ceil(m.nu / 64.0);
  const double direct = std::fmax(
      samples * rays * (0.7e-12 * m.views + 6.7e-12 * m.sum_sin),
      samples * (0.13e-6 + 0.26e-6 * std::fmax(1.0, m.nx / 256.0) * std::fmin(1.0, 1.3 * m.max_sin)));
  const double copy = 16e-6 + copy_bytes * 1.5 / 2.8e12 + (copy_bytes > kept_bytes ? copy_bytes * 60e-12 : 0.0);
  const double zfast = copy + samples * std::fmax(0.15e-6, 64 * 0.95e-12 * waves * m.views);
  return direct > 1.05 * zfast;
}

// How the RTK-form backprojector runs matrices without a z term: voxels of a column a lane
// takes (0: rtk_kernel, a voxel a lane), and whether the views' rows are paired first.
struct RtkForm {
  int per_lane;
  bool pairs;
};

// pu, pv: detector samples a voxel step covers along u and v, at most, at the volume's
// centre.  Microseconds a voxel a lane / two / two or eight with pairs, 32 views unless said:
//  * below 8192 waves of single voxels the chip is not filled: 64^3 16.4 / 17.3 / 27;
//  * dense views leave neighbouring lanes nothing to share: 160^3, pu = pv 5.6, 254 / 292 /
//    607, 320^3 with 3.7 1668 / 1738 / 2540, with 2.8 1346 / 1231 / 1520; with 8 views the
//    line lies higher (3.7: 54 / 43 / 60, 5.6: 56.5 / 58.6 / 107);
//  * pairs lose first, along u: 256^3 with pu 3.7, pv 0.9 606 / 491 / 510, the other way
//    round 613 / 549 / 345.  They cost 9 us and 12 bytes a sample at 2.8 TB/s, and save 0.4
//    ps an update: 96^3 45.1 / 47.4 / 43.9, 128^3 76 / 65 / 48, 512 x 512 x 2 24 / 18 / 29;
//  * eight a lane where that leaves 4096 waves: 128^3 paired two 55, eight 48; 96^3 44, 40.
//    Without pairs only for a view or two, where the volume's own traffic is all: 256^3
//    from one view 42 / 32, eight 27; from 32 of 480^2 160^3 two 151, eight 165.
inline RtkForm rtk_form(int nx, int ny, int nz, int nproj, int W, int H, double pu, double pv) {
  const double rows = (double)((nx + 63) / 64) * ny;
  const bool fill = rows * ((nz + 7) / 8) >= 4096;
  if (rows * nz < 8192 || !(pu * pv >= 0)) return {0, false};
  if (nproj <= 2 && fill && nz >= 8) return {8, false};
  if (pu * pv >= (nproj >= 16 ? 12.0 : 20.0)) return {0, false};
  const double updates = (double)nx * ny * nz * nproj, samples = (double)W * H * nproj;
  if (pu >= 2.4 || updates * 0.4e-12 < 9e-6 + samples * 12.0 / 2.8e12) return {2, false};
  return {fill ? 8 : 2, true};
}

}  // namespace rules
}  // namespace fdk
