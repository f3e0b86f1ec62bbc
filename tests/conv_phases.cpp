// csrc/conv_geometry.h for a test on the CPU.
#include "conv_geometry.h"

// geometry: N C H W D KH KW OH OW pad_h pad_w stride_h stride_w dil_h dil_w.  out: phases, dkh dkw ch cw, columns, least,
// then eleven words a phase.
extern "C" void phases(const int* geometry, long long image_bytes, int parts, int* out) {
  const int* v = geometry;
  const conv::Geometry g{v[0], v[1], v[2], v[3], v[4], v[5], v[6], v[7], v[8], v[9], v[10], v[11], v[12], v[13], v[14]};
  const conv::PhasePlan p = conv::plan_phases(g, image_bytes, parts);
  for (int word : {p.phases, p.by.dkh, p.by.dkw, p.by.ch, p.by.cw, p.columns, p.least}) *out++ = word;
  for (int f = 0; f < p.phases; ++f) {
    const conv::PhaseOfDx& q = p.phase[f];
    for (int word : {q.first, q.rows, q.cols, q.y, q.x, q.kh, q.kw, q.nkh, q.nkw, q.oy, q.ox}) *out++ = word;
  }
}
