// The intensity of a pixel as a quadratic form in the E rotation (laboratory
// frame), shared by the fused executors' per-pixel kernels.
#pragma once

#include <hip/hip_runtime.h>

#include "kernels.hpp"

namespace cyr {

// With E(theta) = c e1 + s e2 the polarization is p = c u + s v, u = Q (F0, F1, F2),
// v = Q (F1, F3, F4), so I(theta) = c^2 |M u|^2 + s^2 |M v|^2 + 2 c s Re<M u, M v>.
// quad[pixel] = (|Mu|^2, |Mv|^2, Re<Mu, Mv>), interpolated between the bins.  T: the forms'
// precision (fields S).
template <typename T, typename S, int NG>
__device__ inline void quad_form_write(const Mat3<T> &Q, const cx<S> (&F)[NG][kEbFields], const double (&md)[NG][6],
                                       T w1, T *o) {
  T qa[NG], qb[NG], qm[NG];
#pragma unroll
  for (int q = 0; q < NG; q++) {
    cx<T> u[3], v[3], mu[3], mv[3];
    const cx<T> ue[3] = {cx_as<T, S>(F[q][0]), cx_as<T, S>(F[q][1]), cx_as<T, S>(F[q][2])};
    const cx<T> ve[3] = {ue[1], cx_as<T, S>(F[q][3]), cx_as<T, S>(F[q][4])};
#pragma unroll
    for (int i = 0; i < 3; i++) {
      u[i] = mk<T>(Q.m[3 * i] * ue[0].x + Q.m[3 * i + 1] * ue[1].x + Q.m[3 * i + 2] * ue[2].x,
                   Q.m[3 * i] * ue[0].y + Q.m[3 * i + 1] * ue[1].y + Q.m[3 * i + 2] * ue[2].y);
      v[i] = mk<T>(Q.m[3 * i] * ve[0].x + Q.m[3 * i + 1] * ve[1].x + Q.m[3 * i + 2] * ve[2].x,
                   Q.m[3 * i] * ve[0].y + Q.m[3 * i + 1] * ve[1].y + Q.m[3 * i + 2] * ve[2].y);
    }
    const T m0 = (T)md[q][0], m1 = (T)md[q][1], m2 = (T)md[q][2], m3 = (T)md[q][3], m4 = (T)md[q][4],
            m5 = (T)md[q][5];
    const T mm[3][3] = {{m0, m1, m2}, {m1, m3, m4}, {m2, m4, m5}};
#pragma unroll
    for (int i = 0; i < 3; i++) {
      mu[i] = mk<T>(mm[i][0] * u[0].x + mm[i][1] * u[1].x + mm[i][2] * u[2].x,
                    mm[i][0] * u[0].y + mm[i][1] * u[1].y + mm[i][2] * u[2].y);
      mv[i] = mk<T>(mm[i][0] * v[0].x + mm[i][1] * v[1].x + mm[i][2] * v[2].x,
                    mm[i][0] * v[0].y + mm[i][1] * v[1].y + mm[i][2] * v[2].y);
    }
    qa[q] = mu[0].x * mu[0].x + mu[0].y * mu[0].y + mu[1].x * mu[1].x + mu[1].y * mu[1].y + mu[2].x * mu[2].x +
            mu[2].y * mu[2].y;
    qb[q] = mv[0].x * mv[0].x + mv[0].y * mv[0].y + mv[1].x * mv[1].x + mv[1].y * mv[1].y + mv[2].x * mv[2].x +
            mv[2].y * mv[2].y;
    qm[q] = mu[0].x * mv[0].x + mu[0].y * mv[0].y + mu[1].x * mv[1].x + mu[1].y * mv[1].y + mu[2].x * mv[2].x +
            mu[2].y * mv[2].y;
  }
  if constexpr (NG == 2) {
    o[0] = (1 - w1) * qa[0] + w1 * qa[1];
    o[1] = (1 - w1) * qb[0] + w1 * qb[1];
    o[2] = (1 - w1) * qm[0] + w1 * qm[1];
  } else {
    o[0] = qa[0];
    o[1] = qb[0];
    o[2] = qm[0];
  }
}

}  // namespace cyr
