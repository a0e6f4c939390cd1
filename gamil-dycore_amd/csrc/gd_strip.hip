// gd_strip.hip -- the coefficient rows of the strip tiles (gd_strip.hpp).
#include <hip/hip_runtime.h>

#include <vector>

#include "gd_strip.hpp"
#include "gd_device.hpp"
#include "gd_launch.hpp"

namespace gd {

namespace {

template <typename CT>
void fill_rows(const std::vector<RowCoef> &rc, std::vector<unsigned char> &out) {
  out.assign(rc.size() * sizeof(StripRow<CT>), 0);
  StripRow<CT> *t = (StripRow<CT> *)out.data();
  for (size_t j = 0; j < rc.size(); ++j) {
    const RowCoef &r = rc[j];
    StripRow<CT> b{};
    b.f = (CT)r.f;
    b.c = (CT)r.c;
    b.c1 = (CT)r.c1;
    b.c2 = (CT)r.c2;
    b.hc = (CT)r.hcos;
    b.fdlon = (CT)r.fdlon;
    b.r_fdlon = (CT)1 / b.fdlon;
    b.hdlat = (CT)r.hdlat;
    b.r_hdlat = r.hdlat != 0.0 ? (CT)1 / b.hdlat : (CT)0;
    b.kul = (CT)r.k_uadv_lon;
    b.kut = (CT)r.k_uadv_lat;
    b.kvl = (CT)r.k_vadv_lon;
    b.kvt = (CT)r.k_vadv_lat;
    b.hcos = r.hcos;
    b.fcos = r.fcos;
    b.fdlon_d = r.fdlon;
    b.r_fdlon_d = 1.0 / r.fdlon;
    b.fdlat_d = r.fdlat;
    b.r_fdlat_d = 1.0 / r.fdlat;
    t[j] = b;
  }
}

}  // namespace

void strip_rows_fill(const std::vector<RowCoef> &rc, int prec, std::vector<unsigned char> &out) {
  if (prec == 0)
    fill_rows<double>(rc, out);
  else
    fill_rows<float>(rc, out);
}

}  // namespace gd
