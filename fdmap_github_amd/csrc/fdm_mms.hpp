// fdm_mms.hpp -- the manufactured solution on the device.
#pragma once

#include <hip/hip_runtime.h>

namespace fdm {

// mms_sin (mms.f90:52-234) on the device; same expression order as the
// reference.  field: 0 vx,1 vy,2 sxx,3 sxy,4 syy,5 szz, 6..11 sources.
__device__ inline double mms_sin(double x, double y, double t, int side, int field) {
  const double G = 32.0, cs = 3.0, cp = 5.0;
  double rho = G / (cs * cs);
  double lambda = rho * (cp * cp) - 2.0 * G;
  double Zs = rho * cs;
  double pi = 4.0 * atan(1.0);
  double kx = 2.0 * pi, ky = 2.0 * pi, mv = 2.0;
  double w = (4.0 / 0.46) * pi;
  double ft = cos(w * t);
  double ft_t = -w * sin(w * t);
  double mf = 0.1, kf = 1.0 * pi;
  double ftpp = mf * kf * cos(kf * x);
  double ftpp_x = -mf * (kf * kf) * sin(kf * x);
  double nx = ftpp / sqrt(1.0 + ftpp * ftpp);
  double ny = -1.0 / sqrt(1.0 + ftpp * ftpp);
  double mx = ny, my = -nx;
  double q = 1.0 + ftpp * ftpp;
  double q3 = q * q * q;
  double nx_x = ftpp_x / sqrt(q3);
  double ny_x = ftpp * ftpp_x / sqrt(q3);
  double mx_x = ny_x, my_x = -nx_x;
  double nx_y = 0.0, ny_y = 0.0;
  double mx_y = ny_y, my_y = -nx_y;
  double sd = (double)side;
  double amp = 2.0 * 12.6 / Zs;
  double ckx = cos(kx * x), sky = sin(ky * y), cky = cos(ky * y), skx = sin(kx * x);
  double vx = mv * (3.0 - 2.0 * sd) * amp * ckx * cky * ft;
  double vx_t = mv * (3.0 - 2.0 * sd) * amp * ckx * cky * ft_t;
  double vx_x = -mv * (3.0 - 2.0 * sd) * kx * amp * skx * cky * ft;
  double vx_y = -mv * (3.0 - 2.0 * sd) * ky * amp * ckx * sky * ft;
  double vy = amp * ckx * cky * ft;
  double vy_t = amp * ckx * cky * ft_t;
  double vy_x = -kx * amp * skx * cky * ft;
  double vy_y = -ky * amp * ckx * sky * ft;
  double syy = -63.0 * ckx * cky * ft - 126.0;
  double syy_t = -63.0 * ckx * cky * ft_t;
  double syy_x = kx * 63.0 * skx * cky * ft;
  double syy_y = ky * 63.0 * ckx * sky * ft;
  double sxy = 0.6 * 126.0 * ckx * cky * ft;
  double sxy_t = 0.6 * 126.0 * ckx * cky * ft_t;
  double sxy_x = -kx * 0.6 * 126.0 * skx * cky * ft;
  double sxy_y = -ky * 0.6 * 126.0 * ckx * sky * ft;
  double sxx = (2.0 * sd - 3.0) * 0.6 * 1260.0 * ckx * cky * ft;
  double sxx_t = (2.0 * sd - 3.0) * 0.6 * 1260.0 * ckx * cky * ft_t;
  double sxx_x = -(2.0 * sd - 3.0) * kx * 0.6 * 1260.0 * skx * cky * ft;
  double sxx_y = -(2.0 * sd - 3.0) * ky * 0.6 * 1260.0 * ckx * sky * ft;
  switch (field) {
    case 5:
      return 0.0;
    case 0:
      return ny * vx - my * vy;
    case 1:
      return mx * vy - nx * vx;
    case 2:
      return syy * (my * my) + sxx * (ny * ny) - 2.0 * sxy * my * ny;
    case 4:
      return syy * (mx * mx) + sxx * (nx * nx) - 2.0 * sxy * mx * nx;
    case 3:
      return -syy * my * mx - sxx * ny * nx + sxy * (ny * mx + nx * my);
    case 6: {
      double vxt = ny * vx_t - my * vy_t;
      double sxxx = syy_x * (my * my) + sxx_x * (ny * ny) - 2.0 * sxy_x * my * ny +
                    2.0 * syy * my * my_x + 2.0 * sxx * ny * ny_x -
                    2.0 * sxy * (my_x * ny + my * ny_x);
      double sxyy = -syy_y * my * mx - sxx_y * ny * nx + sxy_y * (ny * mx + nx * my) -
                    syy * (my_y * mx + my * mx_y) - sxx * (ny_y * nx + ny * nx_y) +
                    sxy * (ny_y * mx + ny * mx_y + nx_y * my + nx * my_y);
      return vxt - (1.0 / rho) * (sxxx + sxyy);
    }
    case 7: {
      double vyt = mx * vy_t - nx * vx_t;
      double sxyx = -syy_x * my * mx - sxx_x * ny * nx + sxy_x * (ny * mx + nx * my) -
                    syy * (my_x * mx + my * mx_x) - sxx * (ny_x * nx + ny * nx_x) +
                    sxy * (ny_x * mx + ny * mx_x + nx_x * my + nx * my_x);
      double syyy = syy_y * (mx * mx) + sxx_y * (nx * nx) - 2.0 * sxy_y * mx * nx +
                    2.0 * syy * mx * mx_y + 2.0 * sxx * nx * nx_y -
                    2.0 * sxy * (mx_y * nx + mx * nx_y);
      return vyt - (1.0 / rho) * (sxyx + syyy);
    }
    case 8: {
      double sxxt = syy_t * (my * my) + sxx_t * (ny * ny) - 2.0 * sxy_t * my * ny;
      double vxx = ny_x * vx - my_x * vy + ny * vx_x - my * vy_x;
      double vyy = mx_y * vy - nx_y * vx + mx * vy_y - nx * vx_y;
      return sxxt - (lambda + 2.0 * G) * vxx - lambda * vyy;
    }
    case 10: {
      double vxx = ny_x * vx - my_x * vy + ny * vx_x - my * vy_x;
      double vyy = mx_y * vy - nx_y * vx + mx * vy_y - nx * vx_y;
      double syyt = syy_t * (mx * mx) + sxx_t * (nx * nx) - 2.0 * sxy_t * mx * nx;
      return syyt - lambda * vxx - (lambda + 2.0 * G) * vyy;
    }
    case 9: {
      double vxy = ny_y * vx - my_y * vy + ny * vx_y - my * vy_y;
      double vyx = mx_x * vy - nx_x * vx + mx * vy_x - nx * vx_x;
      double sxyt = -syy_t * my * mx - sxx_t * ny * nx + sxy_t * (ny * mx + nx * my);
      return sxyt - G * (vyx + vxy);
    }
    case 11: {
      double szzt = 0.0;
      double vxx = ny_x * vx - my_x * vy + ny * vx_x - my * vy_x;
      double vyy = mx_y * vy - nx_y * vx + mx * vy_y - nx * vx_y;
      return szzt - lambda * vxx - lambda * vyy;
    }
    default:
      return 0.0;
  }
}

}  // namespace fdm
