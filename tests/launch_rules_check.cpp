// The launch rules of csrc/launch_rules.hpp behind C entry points, for the tests.
#include "launch_rules.hpp"

extern "C" int check_filter_form(int nu, int nrows, int nviews, int log_n, int transposed_f32) {
  return fdk::rules::filter_form(nu, nrows, nviews, log_n, transposed_f32 != 0);
}

extern "C" int check_wave_strip_columns(double dvz, int zpt, int sides) {
  return fdk::rules::wave_strip_columns(dvz, zpt, sides);
}

extern "C" int check_pitched_copy_pays(double columns, int zext, int slabs, int nproj, double view) {
  return fdk::rules::pitched_copy_pays(columns, zext, slabs, nproj, view);
}

extern "C" int check_zfast_pays(int nu, int nv, double cv, double dv, int nx, int nz, double voxel, double step,
                                int views, double sum_sin, double max_sin) {
  const fdk::rules::March m{nu, nv, cv, dv, 1.5, nx, nx, nz, voxel, voxel, voxel, step, views, sum_sin, max_sin};
  return fdk::rules::zfast_pays(m, 8.0 * (nx + 4) * (nx + 4) * (nz + 4), 512.0 * 1024 * 1024);
}

// voxels a lane, negative with pairs
extern "C" int check_rtk_form(int nx, int ny, int nz, int nproj, int W, int H, double pu, double pv) {
  const fdk::rules::RtkForm f = fdk::rules::rtk_form(nx, ny, nz, nproj, W, H, pu, pv);
  return f.pairs ? -f.per_lane : f.per_lane;
}

extern "C" int check_wave_run(double dvz, int zext, int sides, int nproj, int* columns) {
  const fdk::rules::WaveRun r = fdk::rules::wave_run(dvz, zext, sides, nproj, 0);
  *columns = r.columns;
  return fdk::rules::wave_run_pays(r, zext, nproj) ? r.zpt : -r.zpt;
}
