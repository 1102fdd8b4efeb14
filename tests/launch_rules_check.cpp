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
