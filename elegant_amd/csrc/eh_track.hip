/*
 * eh_track.hip - gfx950 tracking kernel: one particle per lane, FP64.
 *
 * Each lane loads its particle's (x, x', y, y', s, delta) into registers,
 * runs a contiguous run of element-program records for one or many passes,
 * and writes the coordinates back once.  A particle that is lost stops, with
 * its row frozen exactly as the reference leaves a lost row (s = loss
 * position, delta = Po(1+delta)) and its pass and element/stage recorded;
 * the host reproduces the reference's row order from those records.
 *
 * Arithmetic follows the reference routines' operation order with no FP
 * contraction (built with -ffp-contract=off); transcendentals come from
 * emath.h so the CPU checker can reproduce every bit.
 */
#include <hip/hip_runtime.h>

#include <stdio.h>
#include <string.h>

#include "../../include/elegant_hip.h"
#include "eh_consts.h"
#include "eh_device.h"
#include "eh_aperture.h"
#include "eh_program.h"
#include "emath.h"
#include "ehd_internal.h"

#pragma clang fp contract(off)

#define DEV static __device__ __forceinline__

DEV double sq(double v) { return v * v; }

/* Element records and positions are read-only while a kernel runs and every
 * lane of a wave reads the same ones: in the constant address space a uniform
 * address is a scalar load instead of a vector load and wait. */
#define EH_CONST const __attribute__((address_space(4)))
typedef EH_CONST eh_op eh_opc;
typedef EH_CONST double eh_zc;

DEV double opc(EH_CONST double *p) { return *p; }

/* What a common path reads of a record, in scalar registers: the header, read
 * an element ahead, and the element's hot values.  The empty asm makes one
 * group of loads and one wait of them: left to itself the compiler loads each
 * field where it is first used, and a wave alone on its SIMD waits for every
 * one (37 % of its cycles on the FODO ring). */
typedef int hdr_t __attribute__((ext_vector_type(4)));
#define HD_OP(h) ((h).x)
#define HD_FLAGS(h) ((h).y)
#define HD_NSLICES(h) ((h).z)
#define HD_BODY(h) ((h).w)

DEV hdr_t load_hdr(eh_opc *op) { return *(EH_CONST hdr_t *)op; }

struct bounds_t {
  double chk_x, chk_y, in_x, in_y;
};
struct mult_t {
  bounds_t b;
  double dsh[4], kick[3], dx, dy;
};
struct bendc_t { /* the substeps of a bend */
  bounds_t b;
  double rho0, rhoa, rrho0, rrhoa, dshr[4], ds[3], zlim;
};
struct bend_t { /* around them */
  double dxi, dyi, dzi, ct, st, tane1, te1, po, dxf, dyf, dzf, tane2, te2;
};

DEV bounds_t load_bounds(eh_opc &op) {
  bounds_t b = {op.hot[EH_H_CHKX], op.hot[EH_H_CHKY], op.hot[EH_H_INBX], op.hot[EH_H_INBY]};
  return b;
}

DEV mult_t load_mult(eh_opc &op, hdr_t next) {
  mult_t m;
  m.b = load_bounds(op);
  for (int k = 0; k < 4; k++)
    m.dsh[k] = op.hot[EH_H_DSH + k];
  for (int k = 0; k < 3; k++)
    m.kick[k] = op.hot[EH_H_KICK + k];
  m.dx = op.hot[EH_H_DXA];
  m.dy = op.hot[EH_H_DYA];
  asm volatile(""
               : "+s"(m.b.chk_x), "+s"(m.b.chk_y), "+s"(m.b.in_x), "+s"(m.b.in_y), "+s"(m.dsh[0]), "+s"(m.dsh[1]),
                 "+s"(m.dsh[2]), "+s"(m.dsh[3]), "+s"(m.kick[0]), "+s"(m.kick[1]), "+s"(m.kick[2]), "+s"(m.dx),
                 "+s"(m.dy)
               : "s"(next));
  return m;
}

DEV bendc_t load_bendc(eh_opc &op, hdr_t next) {
  bendc_t m;
  m.b = load_bounds(op);
  m.rho0 = op.hot[EH_H_RHO0];
  m.rhoa = op.hot[EH_H_RHOA];
  m.rrho0 = op.hot[EH_H_RRHO0];
  m.rrhoa = op.hot[EH_H_RRHOA];
  for (int k = 0; k < 4; k++)
    m.dshr[k] = op.hot[EH_H_BDSHR + k];
  for (int k = 0; k < 3; k++)
    m.ds[k] = op.hot[EH_H_BDS + k];
  m.zlim = op.hot[EH_H_ZLIM];
  asm volatile("" ::"s"(next));
  return m;
}

DEV bend_t load_bend(eh_opc &op) {
  bend_t b = {op.bend[EH_B_DXI], op.bend[EH_B_DYI], op.bend[EH_B_DZI],   op.bend[EH_B_CT],   op.bend[EH_B_ST],
              op.bend[EH_B_TANE1], op.bend[EH_B_TE1], op.bend[EH_B_PO],  op.bend[EH_B_DXF],  op.bend[EH_B_DYF],
              op.bend[EH_B_DZF], op.bend[EH_B_TANE2], op.bend[EH_B_TE2]};
  return b;
}

struct particle {
  double x, xp, y, yp, s, dp;
};

/* true on every active lane: a scalar test, so the rarely taken side of a
 * branch costs one uniform jump instead of a divergent if/else */
#define ALL_LANES(c) (__builtin_amdgcn_ballot_w64(!(c)) == 0)

DEV int imin3(int a, int b, int c) {
  int m = a < b ? a : b;
  return m < c ? m : c;
}

/* ---- frozen rows of lost particles ---- */

/* limit_amplitudes loss (limit_amplitudes.c:232-268): extrapolate along the
 * preceding drift if asked, then s = z + dz, delta = Po(1 + delta) */
DEV void aperture_loss(particle &p, double xmax, double ymax, int is_out, bool extrap, double z, double Po) {
  double dz = 0;
  if (is_out && !(is_out & 4) && extrap) {
    double dzx = -1.7976931348623157e308, dzy = -1.7976931348623157e308;
    if ((is_out & 1) && p.xp != 0)
      dzx = (p.x - (p.xp > 0 ? 1 : -1) * xmax) / p.xp;
    if ((is_out & 2) && p.yp != 0)
      dzy = (p.y - (p.yp > 0 ? 1 : -1) * ymax) / p.yp;
    if (dzx > dzy)
      dz = -dzx;
    else
      dz = -dzy;
    if (dz == -1.7976931348623157e308)
      dz = 0;
  }
  p.x += dz * p.xp;
  p.y += dz * p.yp;
  p.s = z + dz;
  p.dp = Po * (1 + p.dp);
}

/* the two checks that follow every element (do_tracking.c:2459-2477, 2628-2637).
 * Returns 0 if the particle survives, else stage + 1 with the row frozen.
 * A shaped MAXAMP (ap_code != 0) takes elimit_amplitudes or the open-sided
 * limit_amplitudes instead of the rectangle. */
DEV int post_element_checks(particle &p, eh_opc &op, eh_zc *z) {
  if (op.flags & EH_F_ALONE)
    return 0;
  if ((op.flags & EH_F_AP) && op.ap_code) {
    if (ap_maxamp_shaped(p.x, p.xp, p.y, p.yp, p.s, p.dp, op.ap_xmax, op.ap_ymax, op.ap_code,
                         (op.flags & EH_F_EXTRAP) != 0, opc(&z[1]), op.Po))
      return EH_STAGE_MAXAMP + 1;
  } else if (op.flags & EH_F_AP) {
    double xmax = op.ap_xmax, ymax = op.ap_ymax;
    int is_out = 0;
    if (xmax > 0 && __builtin_fabs(p.x) > xmax)
      is_out += 1;
    if (ymax > 0 && __builtin_fabs(p.y) > ymax)
      is_out += 2;
    if (__builtin_isinf(p.x) || __builtin_isinf(p.y) || __builtin_isnan(p.x) || __builtin_isnan(p.y))
      is_out += 4;
    if (is_out) {
      aperture_loss(p, xmax, ymax, is_out, (op.flags & EH_F_EXTRAP) != 0, opc(&z[1]), op.Po);
      return EH_STAGE_MAXAMP + 1;
    }
  }
  {
    const double big = 1.7976931348623157e308;
    int is_out = 0;
    if (__builtin_fabs(p.x) > big)
      is_out += 1;
    if (__builtin_fabs(p.y) > big)
      is_out += 2;
    if (__builtin_isinf(p.x) || __builtin_isinf(p.y) || __builtin_isnan(p.x) || __builtin_isnan(p.y))
      is_out += 4;
    if (is_out) {
      aperture_loss(p, big, big, is_out, false, opc(&z[1]), op.Po);
      return EH_STAGE_NAN + 1;
    }
  }
  return 0;
}

/* ---- drifts ---- */

/* The drift's matrix applied as the sparse order-2 loop of matrix.c:389-429
 * does it: for each output i (5..0), sum = C[i], then for each input j
 * (5..0) with coord[j] != 0 (NaN counts as nonzero), sum1 = R[i][j] plus
 * T[i][j][k] coord[k] for k = j..0, and sum += sum1 coord[j].  For the drift
 * (R = 1 + L at (0,1) and (2,3), T[4][1][1] = T[4][3][3] = L/2, C[4] = L)
 * every zero entry still multiplies a coordinate, so an infinite or NaN
 * coordinate turns others into NaN, and zero sums take the sign the loop
 * gives them.  drift2_exact is that loop term for term; drift2 is the same
 * result in a few operations for rows where the zero terms cannot matter. */
DEV double drift_R(int i, int j, double L) {
  return i == j ? 1.0 : (((i == 0 && j == 1) || (i == 2 && j == 3)) ? L : 0.0);
}

DEV void drift2_exact(particle &p, double L, double hL) {
  const double v[6] = {p.x, p.xp, p.y, p.yp, p.s, p.dp};
  double out[6];
#pragma unroll
  for (int i = 5; i >= 0; i--) {
    double sum = i == 4 ? L : 0.0;
#pragma unroll
    for (int j = 5; j >= 0; j--) {
      if (v[j] != 0 || v[j] != v[j]) {
        double sum1 = drift_R(i, j, L);
#pragma unroll
        for (int k = j; k >= 0; k--)
          sum1 += ((i == 4 && ((j == 1 && k == 1) || (j == 3 && k == 3))) ? hL : 0.0) * v[k];
        sum += sum1 * v[j];
      }
    }
    out[i] = sum;
  }
  p.x = out[0];
  p.xp = out[1];
  p.y = out[2];
  p.yp = out[3];
  p.s = out[4];
  p.dp = out[5];
}

/* drift2 equals drift2_exact when every coordinate is finite, |x'| and |y'|
 * are 0 or within [2^-300, 2^300] and the element's 2^-300 <= |L| <= 2^300
 * (EH_F_DFAST): then each zero term is a +0 that leaves a sum unchanged
 * (the sums start at +0 or L), no product of a nonzero slope rounds to zero,
 * and a zero x', y' or delta comes out as +0 (the loop skips it and keeps
 * sum = C[i] = +0). */
DEV bool drift2_ok(const particle &p) {
  const double fin = (__builtin_fabs(p.x) + __builtin_fabs(p.y)) + (__builtin_fabs(p.s) + __builtin_fabs(p.dp));
  return fin <= 0x1.0p+1000 && __builtin_fabs(p.xp) + __builtin_fabs(p.yp) <= 0x1.0p+300 &&
         imin3(__builtin_amdgcn_frexp_exp(p.xp), __builtin_amdgcn_frexp_exp(p.yp), 0) >= -299;
}

DEV void drift2(particle &p, double L, double hL) {
  double s = L;
  if (p.s != 0)
    s = s + p.s;
  if (p.yp != 0)
    s = s + (hL * p.yp) * p.yp;
  if (p.xp != 0)
    s = s + (hL * p.xp) * p.xp;
  double y = (p.yp != 0) ? L * p.yp : 0.0;
  if (p.y != 0)
    y = y + p.y;
  double x = (p.xp != 0) ? L * p.xp : 0.0;
  if (p.x != 0)
    x = x + p.x;
  p.x = x;
  p.y = y;
  p.s = s;
  p.xp = p.xp + 0.0;
  p.yp = p.yp + 0.0;
  p.dp = p.dp + 0.0;
}

/* order-1 matrix branch (matrix.c:430-455): sum = C[i] + R[i][j] ini[j] over
 * j = 5..0 for every output, zeros included */
DEV void drift1(particle &p, double L) {
  const double x0 = p.x, xp0 = p.xp, y0 = p.y, yp0 = p.yp, s0 = p.s, dp0 = p.dp;
  p.dp = 0.0 + 1.0 * dp0 + 0.0 * s0 + 0.0 * yp0 + 0.0 * y0 + 0.0 * xp0 + 0.0 * x0;
  p.s = L + 0.0 * dp0 + 1.0 * s0 + 0.0 * yp0 + 0.0 * y0 + 0.0 * xp0 + 0.0 * x0;
  p.yp = 0.0 + 0.0 * dp0 + 0.0 * s0 + 1.0 * yp0 + 0.0 * y0 + 0.0 * xp0 + 0.0 * x0;
  p.y = 0.0 + 0.0 * dp0 + 0.0 * s0 + L * yp0 + 1.0 * y0 + 0.0 * xp0 + 0.0 * x0;
  p.xp = 0.0 + 0.0 * dp0 + 0.0 * s0 + 0.0 * yp0 + 0.0 * y0 + 1.0 * xp0 + 0.0 * x0;
  p.x = 0.0 + 0.0 * dp0 + 0.0 * s0 + 0.0 * yp0 + 0.0 * y0 + L * xp0 + 1.0 * x0;
}

/* track_particles with a first-order matrix (matrix.c:430-458): each
 * coordinate is C[i] plus R[i][j] x[j] added from j = 5 down to 0 */
DEV void matrix1(particle &p, EH_CONST double *m) {
  const double x[6] = {p.x, p.xp, p.y, p.yp, p.s, p.dp};
  double o[6];
#pragma unroll
  for (int i = 0; i < 6; i++) {
    double sum = m[EH_D_M1_C + i];
#pragma unroll
    for (int j = 5; j >= 0; j--)
      sum += m[EH_D_M1_R + 6 * i + j] * x[j];
    o[i] = sum;
  }
  p.x = o[0];
  p.xp = o[1];
  p.y = o[2];
  p.yp = o[3];
  p.s = o[4];
  p.dp = o[5];
}

DEV void exact_drift(particle &p, double L) {
  p.x += p.xp * L;
  p.y += p.yp * L;
  p.s += L * em_sqrt(1 + sq(p.xp) + sq(p.yp));
}

/* ---- misalignment (malign_mat.c:172-182, tilt_matrices.c:156-188) ---- */

DEV void offset(particle &p, double dx, double dy, double dz) {
  /* without DZ the path term is dz times a finite root: dz itself */
  if (dz == 0 && ALL_LANES(__builtin_fabs(p.xp) + __builtin_fabs(p.yp) <= 0x1.0p+500))
    p.s += dz;
  else
    p.s += dz * em_sqrt(1 + sq(p.xp) + sq(p.yp));
  p.x = p.x - dx + dz * p.xp;
  p.y = p.y - dy + dz * p.yp;
}

DEV void rotate(particle &p, double c, double s) {
  double x = p.x, xp = p.xp, y = p.y, yp = p.yp;
  p.x = x * c + y * s;
  p.y = -x * s + y * c;
  p.xp = xp * c + yp * s;
  p.yp = -xp * s + yp * c;
}

/* ---- multipoles ---- */


/* checkMultAperture (multipole.c:1786-1833) */
DEV bool in_aperture(double x, double y, eh_opc &op) {
  if (!(op.flags & EH_F_INAP))
    return true;
  if (op.flags & EH_F_INTILT) {
    double x0 = x, y0 = y;
    x = x0 * op.in_cs0 + y0 * op.in_cs1;
    y = -x0 * op.in_cs1 + y0 * op.in_cs0;
  }
  if (op.in_code)
    return ap_inside_shaped(x, y, op.in_xmax, op.in_ymax, op.in_code);
  return !((op.in_xmax > 0 && __builtin_fabs(x) > op.in_xmax) || (op.in_ymax > 0 && __builtin_fabs(y) > op.in_ymax));
}

/* surely inside it (bounds from eh_op_finish): two compares without
 * a branch for the common paths, whose lanes outside take the general code.
 * ANY: of an ellipse the circle, with a margin for the roundings here and in
 * the general test */
template <bool ANY> DEV bool in_bounds(double x, double y, const bounds_t &b, int flags, eh_opc &op) {
  if (flags & EH_F_INTILT) {
    double x0 = x, y0 = y;
    x = x0 * op.in_cs0 + y0 * op.in_cs1;
    y = -x0 * op.in_cs1 + y0 * op.in_cs0;
  }
  if (ANY && (flags & EH_F_INELL)) {
    const double u = x * op.bend[EH_B_INRX], v = y * op.bend[EH_B_INRY];
    return u * u + v * v <= 1 - 0x1.0p-45;
  }
  return (__builtin_fabs(x) <= b.in_x) & (__builtin_fabs(y) <= b.in_y);
}

/* 1 + delta and its reciprocal for the IEEE quotients of emath.h, fixed for
 * the whole element */
struct opd_recip {
  double v, r;
  int ok;
};

DEV opd_recip make_opd(double dp) {
  opd_recip o;
  o.v = 1 + dp;
  o.r = em_recip(o.v);
  o.ok = em_recip_ok(o.v);
  return o;
}

/* convertMomentaToSlopes (multipole.h:266-281) */
DEV bool momenta_to_slopes(double &xp, double &yp, double qx, double qy, double dp, bool expand,
                           const opd_recip &o) {
  if (expand) {
    xp = em_div(qx, o.v, o.r, o.ok);
    yp = em_div(qy, o.v, o.r, o.ok);
    return true;
  }
  double denom = sq(1 + dp) - sq(qx) - sq(qy);
  if (denom <= 0)
    return false;
  denom = em_sqrt(denom);
  const double r = em_recip(denom);
  const int ok = em_recip_ok(denom);
  xp = em_div(qx, denom, r, ok);
  yp = em_div(qy, denom, r, ok);
  return true;
}

/* sum_Fx, sum_Fy of apply_canonical_multipole_kicks (multipole.h:208-241)
 * for order n, written out: coefficients (-1)^floor(i/2)/(i!(n-i)!) are
 * 1,1 | 1/2,1,-1/2 | 1/6,1/2,-1/2,-1/6, and products with 1 or sums with 0
 * in the reference loop are exact. */
DEV void multipole_fields(int order, double x, double y, double &Fx, double &Fy) {
  if (order == 1) {
    Fx = y;
    Fy = x;
  } else if (order == 2) {
    Fx = x * y;
    Fy = 0.5 * (x * x) + -0.5 * (y * y);
  } else if (order == 3) {
    double x2 = x * x, y2 = y * y;
    Fx = (0.5 * x2) * y + (-1.0 / 6.0) * (y2 * y);
    Fy = (1.0 / 6.0) * (x2 * x) + (-0.5 * x) * y2;
  } else { /* order 0 */
    Fx = 0;
    Fy = 1;
  }
}

DEV void apply_kick(double &qx, double &qy, int order, int skew, double KnL, double x, double y) {
  double Fx, Fy;
  multipole_fields(order, x, y, Fx, Fy);
  if (skew) {
    double t = Fx;
    Fx = -Fy;
    Fy = t;
  }
  qx -= KnL * Fy;
  qy += KnL * Fx;
}

/* The slices of integrate_kick_multipole_ordn (multipole.c:1122-1410), with
 * op.nsub drift substeps per slice (per-substep coefficients are scalar
 * loads of the element record).
 * Returns 0, or the loss kind: 1 aperture (x, y hold the loss point),
 * 2 slopes (the row is left as received). */
DEV int multipole_body(double &x, double &xp, double &y, double &yp, double &s, double &qx, double &qy,
                       double &dzLoss, const double dp, const bool expand, const opd_recip &o, eh_opc &op) {
  const int nsub = op.nsub;
  const int flags = op.flags;
  const double dxa = op.d[EH_D_DX], dya = op.d[EH_D_DY];
  const bool has_drift = op.d[EH_D_DRIFT] != 0;
  const int nko = op.nkick_orders;
  for (int ik = 0; ik < op.nslices; ik++) {
    if (!in_aperture(x + dxa, y + dya, op))
      return 1;
    for (int step = 0; step < nsub; step++) {
      if (has_drift) {
        const double dsh = opc(&op.d[EH_D_DSH + step]);
        x += xp * dsh;
        y += yp * dsh;
        if (expand)
          s += dsh * (1 + (sq(xp) + sq(yp)) / 2);
        else
          s += dsh * em_sqrt(1 + sq(xp) + sq(yp));
        dzLoss += dsh;
      }
      if (step == nsub - 1)
        break; /* kickFrac[last] == 0 */
      if (nko > 0)
        apply_kick(qx, qy, op.order0, op.skew0, opc(&op.d[EH_D_KICK + step]), x, y);
      if (nko > 1)
        apply_kick(qx, qy, op.order1, op.skew1, opc(&op.d[EH_D_KICK + 8 + step]), x, y);
      if (nko > 2)
        apply_kick(qx, qy, op.order2, op.skew2, opc(&op.d[EH_D_KICK + 16 + step]), x, y);
      if (flags & EH_F_XKICK)
        apply_kick(qx, qy, 0, 0, opc(&op.d[EH_D_XK + step]), x, y);
      if (flags & EH_F_YKICK)
        apply_kick(qx, qy, 0, 1, opc(&op.d[EH_D_YK + step]), x, y);
      if (!momenta_to_slopes(xp, yp, qx, qy, dp, expand, o))
        return 2;
      if (has_drift) {
        /* rad_coef = 0, isr_coef < 0: the q/(1+dp)*(1+dp) round trip (multipole.c:1321-1351) */
        qx = em_div(qx, o.v, o.r, o.ok);
        qy = em_div(qy, o.v, o.r, o.ok);
        qx *= (1 + dp);
        qy *= (1 + dp);
        if (!momenta_to_slopes(xp, yp, qx, qy, dp, expand, o))
          return 2;
      }
    }
  }
  return 0;
}

/* The whole integrator - entry, slices, exit - on its common path
 * (EXPAND_HAMILTONIAN=0), with no per-lane branches: unscaled square roots and
 * quotients by positive divisors (emath.h), no loss.  Returns false for a
 * lane where that may not hold; the caller then recomputes the lane from the
 * row it received with the general code.
 *
 * One v_rsq_f64 per kick, and none per drift: den = sqrt(opd^2 - q^2) and its
 * reciprocal r come from one iteration, and with slopes q/den the drift's
 * root of t = 1 + x'^2 + y'^2 is opd r and half its reciprocal den/(2 opd), both
 * to within 3 u (u = 2^-52).  Two residual corrections g + (t - g^2) h round
 * it.  Both estimates are taken 4 u low: then the first correction gives the
 * root rounded, less a relative 2^-97 before rounding, so a root just below
 * a midpoint of two doubles (t = 1 + (2k + 1) u for small slopes) goes down as
 * it must, and the second one keeps it.  A root just above the midpoint g + u/2
 * has t = (g + u/2)^2 + (m - 1/4) u^2 with m even as t is a double, and comes
 * out wrong only for m <= 10: nine doubles below 4, the least of them 1.1525,
 * which the bound on the slopes (t < 1.137) leaves out.
 * The slopes at the exit are those after the last kick, as the momenta have
 * not changed since.  A slice of four substeps of a quadrupole takes 182 VALU
 * instructions, 3 of them transcendental (276 with 16 before).  FODO ring, 10^4
 * particles, 64 turns: 84.1 -> 54.9 ms (36.4 with what came after it).
 *
 * What makes every step valid:
 *  - the entry and exit limits of the integrator and the aperture at every
 *    slice hold (a NaN in the row or the momenta reaches one of them);
 *  - opd in [2^-64, 2^64], the received slopes are 0 or >= 2^-600;
 *  - opd^2 - qx^2 - qy^2 >= 0.88 opd^2 at every conversion to slopes, tested
 *    after the round trip, which moves it by a few ulps: no slope loss on
 *    either side of it, the roots in range, t < 1.137;
 *  - after the kicks qx and qy are 0 or >= 2^-700 in magnitude (binary
 *    exponent >= -699), so every dividend is 0 or within [2^-900, 2^900].
 * Arithmetic is otherwise the general code's, operation for operation. */
template <int ORD, bool ELL>
DEV bool multipole_fast(const particle &p, double &x, double &xp, double &y, double &yp, double &s,
                        const opd_recip &o, const hdr_t H, const mult_t &m, eh_opc &op) {
  const int nsub = ORD ? 4 : op.nsub;
  const int flags = HD_FLAGS(H);
  const double dxa = m.dx, dya = m.dy;
  const bool has_drift = ORD > 0 || op.d[EH_D_DRIFT] != 0;
  const double opd = o.v, o2 = sq(opd), hr = (0.5 - 0x1.0p-51) * o.r;
  x = p.x;
  y = p.y;
  xp = p.xp;
  yp = p.yp;
  s = 0;
  /* & instead of &&: no lane skips the rest of a test that all lanes pass */
  bool good = (opd >= 0x1.0p-64) & (opd <= 0x1.0p+64) & (__builtin_fabs(x) <= EH_COORD_LIMIT) &
              (__builtin_fabs(y) <= EH_COORD_LIMIT) & (__builtin_fabs(xp) <= EH_SLOPE_LIMIT) &
              (__builtin_fabs(yp) <= EH_SLOPE_LIMIT) &
              (imin3(__builtin_amdgcn_frexp_exp(xp), __builtin_amdgcn_frexp_exp(yp), 0) >= -599);
  double r, den = em_sqrt_recip_mid(1 + sq(xp) + sq(yp), &r);
  double qx = em_div_pos(opd * xp, den, r), qy = em_div_pos(opd * yp, den, r);
  double den2 = o2 - sq(qx) - sq(qy), dmin = den2;
  den = em_sqrt_recip_mid(den2, &r);
  xp = em_div_pos(qx, den, r);
  yp = em_div_pos(qy, den, r);
  int emin = 0;
  for (int ik = 0; ik < HD_NSLICES(H); ik++) {
    good &= in_bounds<ELL>(x + dxa, y + dya, m.b, flags, op);
#pragma unroll
    for (int step = 0; step < nsub; step++) {
      if (has_drift) {
        const double dsh = ORD ? m.dsh[step & 3] : opc(&op.d[EH_D_DSH + step]);
        x += xp * dsh;
        y += yp * dsh;
        const double t = 1 + sq(xp) + sq(yp), h = den * hr;
        double g = __builtin_fma(opd, r, -0x1.0p-50);
        g = __builtin_fma(__builtin_fma(-g, g, t), h, g);
        g = __builtin_fma(__builtin_fma(-g, g, t), h, g);
        s += dsh * g;
      }
      if (step == nsub - 1)
        break; /* kickFrac[last] == 0 */
      if (ORD > 0) {
        apply_kick(qx, qy, ORD, 0, m.kick[step % 3], x, y);
      } else {
        const int nko = op.nkick_orders;
        if (nko > 0)
          apply_kick(qx, qy, op.order0, op.skew0, opc(&op.d[EH_D_KICK + step]), x, y);
        if (nko > 1)
          apply_kick(qx, qy, op.order1, op.skew1, opc(&op.d[EH_D_KICK + 8 + step]), x, y);
        if (nko > 2)
          apply_kick(qx, qy, op.order2, op.skew2, opc(&op.d[EH_D_KICK + 16 + step]), x, y);
        if (flags & EH_F_XKICK)
          apply_kick(qx, qy, 0, 0, opc(&op.d[EH_D_XK + step]), x, y);
        if (flags & EH_F_YKICK)
          apply_kick(qx, qy, 0, 1, opc(&op.d[EH_D_YK + step]), x, y);
      }
      emin = imin3(emin, __builtin_amdgcn_frexp_exp(qx), __builtin_amdgcn_frexp_exp(qy));
      if (has_drift) {
        /* rad_coef = 0, isr_coef < 0: the q/(1+dp)*(1+dp) round trip (multipole.c:1321-1351) */
        qx = em_div_pos(qx, opd, o.r) * opd;
        qy = em_div_pos(qy, opd, o.r) * opd;
      }
      den2 = o2 - sq(qx) - sq(qy);
      dmin = __builtin_fmin(dmin, den2);
      den = em_sqrt_recip_mid(den2, &r);
      xp = em_div_pos(qx, den, r);
      yp = em_div_pos(qy, den, r);
    }
  }
  return good & (emin >= -699) & (dmin >= 0.88 * o2) & in_bounds<ELL>(x + dxa, y + dya, m.b, flags, op) &
         (__builtin_fabs(x) <= EH_COORD_LIMIT) & (__builtin_fabs(y) <= EH_COORD_LIMIT) &
         (__builtin_fabs(xp) <= EH_SLOPE_LIMIT) & (__builtin_fabs(yp) <= EH_SLOPE_LIMIT);
}

/* the integrator's entry (multipole.c:1176-1205): limits, slopes to
 * momenta and back.  Returns 0, or 2 for a slope loss (dzLoss set). */
DEV int multipole_entry(const particle &p, double &xp, double &yp, double &qx, double &qy, double &dzLoss,
                        const bool expand, const opd_recip &o, eh_opc &op) {
  const double dp = p.dp;
  xp = p.xp;
  yp = p.yp;
  if (__builtin_isnan(p.x) || __builtin_isnan(xp) || __builtin_isnan(p.y) || __builtin_isnan(yp) ||
      __builtin_fabs(p.x) > EH_COORD_LIMIT || __builtin_fabs(p.y) > EH_COORD_LIMIT ||
      __builtin_fabs(xp) > EH_SLOPE_LIMIT || __builtin_fabs(yp) > EH_SLOPE_LIMIT) {
    dzLoss = op.d[EH_D_TOTLEN];
    return 2;
  }
  if (expand) {
    qx = (1 + dp) * xp;
    qy = (1 + dp) * yp;
  } else {
    double denom = em_sqrt(1 + sq(xp) + sq(yp));
    qx = (1 + dp) * xp / denom;
    qy = (1 + dp) * yp / denom;
  }
  if (!momenta_to_slopes(xp, yp, qx, qy, dp, expand, o)) {
    dzLoss = op.d[EH_D_TOTLEN];
    return 2;
  }
  return 0;
}

/* the integrator of integrate_kick_multipole_ordn (multipole.c:1122-1410) on
 * one particle by the general code.  Returns 0, or the loss kind with the
 * row frozen. */
DEV int multipole_general(particle &p, const bool expand, const opd_recip &o, eh_opc &op, eh_zc *z) {
  const double dp = p.dp;
  double x = p.x, xp = 0, y = p.y, yp = 0, s = 0, qx = 0, qy = 0, dzLoss = 0;
  const double dxa = op.d[EH_D_DX], dya = op.d[EH_D_DY];
  /* 1: aperture (x, y written), 2: slopes (nothing written), 3: final limits */
  int lost = multipole_entry(p, xp, yp, qx, qy, dzLoss, expand, o, op);
  if (!lost)
    lost = multipole_body(x, xp, y, yp, s, qx, qy, dzLoss, dp, expand, o, op);
  if (!lost) {
    if (!in_aperture(x + dxa, y + dya, op))
      lost = 1;
    else if (!momenta_to_slopes(xp, yp, qx, qy, dp, expand, o))
      lost = 2;
    else {
      p.x = x;
      p.xp = xp;
      p.y = y;
      p.yp = yp;
      p.s += s;
      p.dp = dp;
      if (__builtin_isnan(x) || __builtin_isnan(xp) || __builtin_isnan(y) || __builtin_isnan(yp) ||
          __builtin_fabs(x) > EH_COORD_LIMIT || __builtin_fabs(y) > EH_COORD_LIMIT ||
          __builtin_fabs(xp) > EH_SLOPE_LIMIT || __builtin_fabs(yp) > EH_SLOPE_LIMIT)
        lost = 3;
    }
  }
  if (lost) {
    if (lost == 1) {
      p.x = x;
      p.y = y;
    }
    /* lost == 2: row as received; lost == 3: row fully written */
    p.s = opc(&z[0]) + dzLoss;
    p.dp = op.Po * (1 + p.dp);
  }
  return lost;
}

/* entry and exit of multipole_tracking2: misalignment, roll and the exact
 * drifts of KQUAD LEFFECTIVE around the body (multipole.c:1028-1030), the
 * exit ones applied to lost rows too (multipole.c:1098-1104) */
DEV void multipole_in(particle &p, eh_opc &op) {
  const int flags = op.flags;
  if (flags & EH_F_OFFSET)
    offset(p, op.d[EH_D_DX], op.d[EH_D_DY], op.d[EH_D_DZ]);
  if (flags & EH_F_ROTATE)
    rotate(p, op.d[EH_D_COS_IN], op.d[EH_D_SIN_IN]);
  if (flags & EH_F_LEND)
    exact_drift(p, op.d[EH_D_LEND]);
}

DEV void multipole_out(particle &p, eh_opc &op) {
  const int flags = op.flags;
  if (flags & EH_F_LEND)
    exact_drift(p, op.d[EH_D_LEND]);
  if (flags & EH_F_ROTATE)
    rotate(p, op.d[EH_D_COS_OUT], op.d[EH_D_SIN_OUT]);
  if (flags & EH_F_OFFSET)
    offset(p, -op.d[EH_D_DX], -op.d[EH_D_DY], -op.d[EH_D_DZ]);
}

/* multipole_tracking2 per particle by the general code.  Returns 0 if
 * alive, EH_STAGE_ELEMENT + 1 if lost (row frozen). */
DEV int track_multipole(particle &p, eh_opc &op, eh_zc *z) {
  multipole_in(p, op);
  const opd_recip o = make_opd(p.dp);
  const int lost = multipole_general(p, (op.flags & EH_F_EXPAND) != 0, o, op, z);
  multipole_out(p, op);
  return lost ? EH_STAGE_ELEMENT + 1 : 0;
}

/* the same on the common path; false: p is not to be used */
template <bool ELL> DEV bool track_multipole_fast(particle &p, const hdr_t H, const mult_t &m, eh_opc &op) {
  const int flags = HD_FLAGS(H);
  if (flags & EH_F_EXPAND)
    return false;
  if (flags & (EH_F_OFFSET | EH_F_ROTATE | EH_F_LEND))
    multipole_in(p, op);
  opd_recip o;
  o.v = 1 + p.dp;
  o.r = em_recip(o.v);
  /* the common thick element with one normal multipole and no steering gets
   * a body specialised to its order: the kick is straight-line code */
  const int body = HD_BODY(H);
  double x, xp, y, yp, s;
  bool done;
  if (body == 1)
    done = multipole_fast<1, ELL>(p, x, xp, y, yp, s, o, H, m, op);
  else if (body == 2)
    done = multipole_fast<2, ELL>(p, x, xp, y, yp, s, o, H, m, op);
  else if (body == 3)
    done = multipole_fast<3, ELL>(p, x, xp, y, yp, s, o, H, m, op);
  else
    done = multipole_fast<0, ELL>(p, x, xp, y, yp, s, o, H, m, op);
  p.x = x;
  p.xp = xp;
  p.y = y;
  p.yp = yp;
  p.s += s;
  if (flags & (EH_F_OFFSET | EH_F_ROTATE | EH_F_LEND))
    multipole_out(p, op);
  return done;
}

/* ---- CSBEND ---- */

/* The slices of integrate_csbend_ordn (csbend.c:1434-1693) for a pure
 * dipole (Fx = 0, Fy = 1, csbend.c:106-110), op.nsub drift substeps per
 * slice; per-substep coefficients are scalar loads of the element record.  Returns true if the particle is lost; X, QX, Y, QY, dist
 * and dz_lost then hold their values at the loss, as the reference leaves
 * them. */
/* computeCSBENDFields (csbend.c:100-141), normal multipoles: the
 * coefficients in the order eh_bend_field_flatten lays them out, each term
 * (F x^i) y^j with the powers of y built by repeated multiplication as the
 * reference's table of powers is */
DEV void bend_fields(eh_opc &op, double x, double y, double &Fx, double &Fy) {
  const int n1 = op.nfield;
  double sumFx = 0, sumFy = 0, xt = 1;
  int k = 0;
  for (int i = 0; i < n1; i++) {
    double p = y; /* y^1 */
    for (int j = 1; j < n1 - i; j += 2) {
      sumFx += opc(&op.d[EH_D_FIELD + k]) * xt * p;
      k++;
      p *= y;
      p *= y;
    }
    p = 1.0; /* y^0 */
    for (int j = 0; j < n1 - i; j += 2) {
      sumFy += opc(&op.d[EH_D_FIELD + k]) * xt * p;
      k++;
      p *= y;
      p *= y;
    }
    xt *= x;
  }
  Fx = sumFx;
  Fy = sumFy;
}

DEV bool csbend_body(double &X, double &QX, double &Y, double &QY, const double DP, double &dist, double &dz_lost,
                     eh_opc &op) {
  const double rho0 = op.d[EH_D_RHO0], rhoa = op.d[EH_D_RHOA], rsgn = op.d[EH_D_RHOA_SGN];
  const double opd = 1 + DP;
  const int nsub = op.nsub;
  /* reciprocals shared by the divisions below (IEEE quotients, emath.h);
   * those of rho0 and rho_actual are rounded on the host */
  const double r_opd = em_recip(opd);
  const int ok_opd = em_recip_ok(opd);
  const int ok_rho = (op.flags & EH_F_RCP) != 0;
  for (int i = 0; i < op.nslices; i++) {
    if (!in_aperture(X, Y, op))
      return true;
    for (int j = 0; j < nsub; j++) {
      double f = sq(opd) - sq(QY);
      if (f <= 0)
        return true;
      f = em_sqrt(f);
      const double r_f = em_recip(f);
      const int ok_f = em_recip_ok(f);
      double sin_phi = em_div(QX, f, r_f, ok_f);
      if (__builtin_fabs(sin_phi) > 1)
        return true;
      double phi = em_asin(sin_phi);
      double sine, cosi;
      em_sincos(opc(&op.d[EH_D_BDSHR + j]) + phi, &sine, &cosi);
      if (cosi == 0)
        return true;
      const double r_c = em_recip(cosi);
      const int ok_c = em_recip_ok(cosi);
      double tang = em_div(sine, cosi, r_c, ok_c);
      double cos_phi = em_cos(phi);
      QX = f * sine;
      double factor = em_div((rho0 + X) * cos_phi, f, r_f, ok_f) * (tang - sin_phi / cos_phi);
      Y += QY * factor;
      dist += factor * opd;
      dz_lost += opc(&op.d[EH_D_BDSH + j]);
      f = em_div(cos_phi, cosi, r_c, ok_c);
      X = rho0 * (f - 1) + f * X;
      if (j == nsub - 1)
        break; /* kickFrac[last] == 0 */
      double ds = opc(&op.d[EH_D_BDS + j]);
      double g = 1 + em_div(X, rho0, opc(&op.d[EH_D_RRHO0]), ok_rho);
      if (op.flags & EH_F_FIELD) {
        double Fx, Fy;
        bend_fields(op, X, Y, Fx, Fy);
        QX += em_div(-ds * g * Fy, rhoa, opc(&op.d[EH_D_RRHOA]), ok_rho);
        QY += em_div(ds * g * Fx, rhoa, opc(&op.d[EH_D_RRHOA]), ok_rho);
      } else {
        QX += em_div(-ds * g * 1.0, rhoa, opc(&op.d[EH_D_RRHOA]), ok_rho);
        /* Fx = 0: ds*g*0.0 is +-0 or NaN, and dividing it by rho_actual only
         * sets its sign, which the multiplication by sign(rho_actual) does */
        QY += ds * g * 0.0 * rsgn;
      }
      QX = em_div(QX, opd, r_opd, ok_opd);
      QY = em_div(QY, opd, r_opd, ok_opd);
      QX *= opd;
      QY *= opd;
    }
  }
  return false;
}


/* csbend_body on its common path, with no per-lane branches: every substep
 * takes the narrow bands of asin/sin/cos (z < 2^-10, emath.h *_small), the
 * unscaled quotients by positive divisors (em_div_pos) and the unscaled
 * square root, and no loss occurs.  Returns false for a lane where any of
 * that may not hold; the caller then discards the lane's results and runs
 * csbend_body from the saved state.
 *
 * A pure dipole leaves QY alone but for the round trip q -> (q/opd) opd after
 * each kick, and the trip's result q1 is a fixed point of it: when the grid
 * of q/opd is the finer of the two, q1/opd lies within half its step of the
 * quotient taken, whose product is within half a step of q1; when it is the
 * coarser one, q1/opd rounds back to the first quotient.  That is tested
 * once (q2 == q1), not relied on.  So sqrt(opd^2 - QY^2) and its reciprocal
 * take two values in the whole element, one before the first kick and one
 * after it, and both are computed before the loop: per substep that saves
 * the square root, a reciprocal, the trip and their range checks.  Together
 * with the secant's series in place of two v_rcp_f64 and the checks below, a
 * slice of four substeps takes 329 VALU and 36 scalar instructions, where it
 * took 495 (16 of them transcendental, at four times the issue cycles) and
 * 107.  10 turns of 10^6 particles of the storage ring with upload and
 * download: 360 -> 288 ms (203 with what came after it).
 *
 * What makes every step valid:
 *  - at the entry X, QX, QY are 0 or within [2^-700, 2^600] in magnitude
 *    (QY not -0, whose sign the first kick could change), opd^2 - QY^2 >=
 *    2^-128, opd in [2^-64, 2^64]; the host has checked radii, substep
 *    angles c (2^-20 <= |c| < 2^-5) and kick lengths (EH_F_FAST);
 *  - phi^2 < zlim at every substep (a running maximum), where zlim keeps
 *    |phi| and |c + phi| below 2^-5 (in the WIDE instance, for substep
 *    angles of 2^-6 and more, both squares are watched).  |phi| >= |sin phi|
 *    as the series' terms have one sign, so that rules out |sin phi| > 1 and
 *    cos = 0, and cos phi / cos(c + phi) lies within 1 % of 1 (and is not
 *    1 / (1 - 2^-53), as c is far above 2^-26);
 *  - the dividends stay 0 or >= 2^-718: c + phi is 0 or at least an ulp of
 *    2^-20, hence QX = f sin(c + phi) is 0 or >= 2^-140 after a drift, and
 *    after a kick 0 or an ulp of such terms; X = rho0 (f - 1) + f X is its
 *    old value when f = 1 and otherwise has a term of at least 2^-117;
 *  - |X| + |QX| <= 2^600 at the start of every slice and at the end: X
 *    changes by at most 1 % and rho0 2^-6 in a substep, a kick that makes QX
 *    large fails the bound on phi at the next substep, and a NaN stays in X;
 *  - the aperture holds at every slice; dz_lost only matters for a loss.
 * Arithmetic is otherwise csbend_body's, operation for operation.
 *
 * ANY: substep angles below 2^-20 too (EH_F_SMALL; correctors modelled as
 * bends), and ellipses beyond their box.  A cosine may be 1 - 2^-53 at any
 * substep then, so the cosines' reciprocals are em_recip's, and a running
 * minimum keeps the exponents of c + phi and of QX after a kick at -600 or
 * more, or the values 0. */
template <int NSUB, bool WIDE, bool ANY>
DEV bool csbend_body_fast(double &X, double &QX, double &Y, double &QY, const double opd, const double r_opd,
                          double &dist, const hdr_t H, const bendc_t &m, eh_opc &op) {
  const double rho0 = m.rho0, rhoa = m.rhoa;
  const int nsub = NSUB ? NSUB : op.nsub;
  bool good = (opd >= 0x1.0p-64) & (opd <= 0x1.0p+64) & (em_bits(QY) != 0x8000000000000000ULL) &
              ((__builtin_fabs(X) + __builtin_fabs(QX)) + __builtin_fabs(QY) <= 0x1.0p+600) &
              (imin3(__builtin_amdgcn_frexp_exp(X), __builtin_amdgcn_frexp_exp(QX), __builtin_amdgcn_frexp_exp(QY)) >=
               -699);
  const double q1 = em_div_pos(QY, opd, r_opd) * opd;
  good &= em_div_pos(q1, opd, r_opd) * opd == q1;
  const double fin = sq(opd) - sq(QY), fin1 = sq(opd) - sq(q1);
  good &= __builtin_fmin(fin, fin1) >= 0x1.0p-128;
  double r_f, r_f1;
  double f = em_sqrt_recip_mid(fin, &r_f);
  const double f1 = em_sqrt_recip_mid(fin1, &r_f1);
  /* sin_phi = 2^-26 exactly over cos_phi = 1 - 2^-53 (em_recip_cos_small): a
   * slope of sqrt(machine epsilon) at the entry, a usual finite-difference step */
  if (!ANY)
    good &= __builtin_fabs(QX) != 0x1.0p-26 * f;
  double acc = 0, zmax = 0;
  int emin = 0;
  const em_small_k K = em_small_coefs();
  for (int i = 0; i < HD_NSLICES(H); i++) {
    good &= in_bounds<ANY>(X, Y, m.b, HD_FLAGS(H), op);
    acc += __builtin_fabs(X) + __builtin_fabs(QX);
#pragma unroll
    for (int j = 0; j < nsub; j++) {
      double sin_phi = em_div_pos(QX, f, r_f);
      double phi = em_asin_small_c(sin_phi, sin_phi * sin_phi, &K);
      const double ang = (NSUB ? m.dshr[j & 3] : opc(&op.d[EH_D_BDSHR + j])) + phi;
      const double za = ang * ang, zp = phi * phi;
      zmax = __builtin_fmax(zmax, zp);
      if (WIDE)
        zmax = __builtin_fmax(zmax, za);
      if (ANY)
        emin = imin3(emin, __builtin_amdgcn_frexp_exp(ang), 0);
      double sine = em_sin_small_c(ang, za, &K), cosi = em_cos_small_c(za, &K);
      const double r_c = ANY ? em_recip(cosi) : em_recip_cos_small(cosi, za, &K);
      double tang = em_div_pos(sine, cosi, r_c);
      double cos_phi = em_cos_small_c(zp, &K);
      const double r_p = ANY ? em_recip(cos_phi) : em_recip_cos_small(cos_phi, zp, &K);
      QX = f * sine;
      double factor = em_div_pos((rho0 + X) * cos_phi, f, r_f) * (tang - em_div_pos(sin_phi, cos_phi, r_p));
      Y += QY * factor;
      dist += factor * opd;
      const double fc = em_div_pos(cos_phi, cosi, r_c);
      X = rho0 * (fc - 1) + fc * X;
      if (j == nsub - 1)
        break; /* kickFrac[last] == 0 */
      double ds = NSUB ? m.ds[j % 3] : opc(&op.d[EH_D_BDS + j]);
      double g = 1 + em_div_pos(X, rho0, m.rrho0);
      /* (-ds) g 1.0 = -(ds g): the general code's bits, one product fewer */
      QX += em_div_pos(-(ds * g), rhoa, m.rrhoa);
      if (ANY)
        emin = imin3(emin, __builtin_amdgcn_frexp_exp(QX), 0);
      QX = em_div_pos(QX, opd, r_opd);
      QX *= opd;
      QY = q1;
      f = f1;
      r_f = r_f1;
    }
  }
  acc += __builtin_fabs(X) + __builtin_fabs(QX);
  return good & (acc <= 0x1.0p+600) & (zmax < (WIDE ? EM_SMALL_Z : m.zlim)) & (emin >= -600);
}

/* The slices of a combined-function bend with expansion order 4 (K1 and K2),
 * four substeps a slice: csbend_body with FIELD, without branches.  Bound by
 * the latency of the general code's 15 coefficient loads per kick, each used
 * as it arrives; here they are loaded once per element, and the powers of x
 * and y are shared by the terms they appear in (the same products: y^k is
 * built from y^(k-1) in every sum of bend_fields).  Fx and Fy are summed in
 * its order.  A bend of 16 slices over 20011 rows: 378 -> 287 us with the
 * transfers.
 *
 * Against the dipole's conditions above: QY moves with the kicks, so f is
 * taken anew after each (a running minimum keeps it >= 2^-64), the kicks'
 * dividends and the momenta after them are 0 or >= 2^-700 by their running
 * minimum exponent, and acc bounds the dividends from above and catches a NaN
 * of either plane (in Y it reaches QX through Fy). */
DEV void field5(const double *F, double x, double y, double &Fx, double &Fy) {
  const double y2 = y * y, y3 = y2 * y, y4 = y3 * y, x2 = x * x, x3 = x2 * x, x4 = x3 * x;
  Fx = 0.0 + F[0] * y;
  Fx += F[1] * y3;
  Fy = 0.0 + F[2];
  Fy += F[3] * y2;
  Fy += F[4] * y4;
  Fx += F[5] * x * y;
  Fx += F[6] * x * y3;
  Fy += F[7] * x;
  Fy += F[8] * x * y2;
  Fx += F[9] * x2 * y;
  Fy += F[10] * x2;
  Fy += F[11] * x2 * y2;
  Fx += F[12] * x3 * y;
  Fy += F[13] * x3;
  Fy += F[14] * x4;
}

DEV bool csbend_field_fast(double &X, double &QX, double &Y, double &QY, const double opd, const double r_opd,
                           double &dist, const hdr_t H, const bendc_t &m, eh_opc &op) {
  const double rho0 = m.rho0, rhoa = m.rhoa;
  double F[15];
  for (int k = 0; k < 15; k++)
    F[k] = op.d[EH_D_FIELD + k];
  bool good = (opd >= 0x1.0p-64) & (opd <= 0x1.0p+64) &
              ((__builtin_fabs(X) + __builtin_fabs(QX)) + __builtin_fabs(QY) <= 0x1.0p+600) &
              (imin3(__builtin_amdgcn_frexp_exp(X), __builtin_amdgcn_frexp_exp(QX), __builtin_amdgcn_frexp_exp(QY)) >=
               -699);
  const double o2 = sq(opd);
  double f2 = o2 - sq(QY), fmin2 = f2, r_f, f = em_sqrt_recip_mid(f2, &r_f);
  good &= __builtin_fabs(QX) != 0x1.0p-26 * f; /* as for the dipole */
  double acc = 0, zmax = 0;
  int emin = 0;
  const em_small_k K = em_small_coefs();
  for (int i = 0; i < HD_NSLICES(H); i++) {
    good &= in_bounds<false>(X, Y, m.b, HD_FLAGS(H), op);
    acc += __builtin_fabs(X) + __builtin_fabs(QX);
#pragma unroll
    for (int j = 0; j < 4; j++) {
      double sin_phi = em_div_pos(QX, f, r_f);
      double phi = em_asin_small_c(sin_phi, sin_phi * sin_phi, &K);
      const double ang = m.dshr[j] + phi;
      const double za = ang * ang, zp = phi * phi;
      zmax = __builtin_fmax(zmax, __builtin_fmax(zp, za));
      double sine = em_sin_small_c(ang, za, &K), cosi = em_cos_small_c(za, &K);
      const double r_c = em_recip_cos_small(cosi, za, &K);
      double tang = em_div_pos(sine, cosi, r_c);
      double cos_phi = em_cos_small_c(zp, &K);
      QX = f * sine;
      double factor = em_div_pos((rho0 + X) * cos_phi, f, r_f) *
                      (tang - em_div_pos(sin_phi, cos_phi, em_recip_cos_small(cos_phi, zp, &K)));
      Y += QY * factor;
      dist += factor * opd;
      const double fc = em_div_pos(cos_phi, cosi, r_c);
      X = rho0 * (fc - 1) + fc * X;
      if (j == 3)
        break; /* kickFrac[last] == 0 */
      double Fx, Fy;
      field5(F, X, Y, Fx, Fy);
      /* (-ds g) Fy = -(ds g Fy) */
      const double dg = m.ds[j] * (1 + em_div_pos(X, rho0, m.rrho0)), kx = -(dg * Fy), ky = dg * Fx;
      QX += em_div_pos(kx, rhoa, m.rrhoa);
      QY += em_div_pos(ky, rhoa, m.rrhoa);
      acc += __builtin_fabs(kx) + __builtin_fabs(ky);
      emin = imin3(emin, __builtin_amdgcn_frexp_exp(kx), __builtin_amdgcn_frexp_exp(ky));
      emin = imin3(emin, __builtin_amdgcn_frexp_exp(QX), __builtin_amdgcn_frexp_exp(QY));
      QX = em_div_pos(QX, opd, r_opd);
      QY = em_div_pos(QY, opd, r_opd);
      QX *= opd;
      QY *= opd;
      f2 = o2 - sq(QY);
      fmin2 = __builtin_fmin(fmin2, f2);
      f = em_sqrt_recip_mid(f2, &r_f);
    }
  }
  acc += __builtin_fabs(X) + __builtin_fabs(QX) + __builtin_fabs(QY);
  return good & (acc <= 0x1.0p+600) & (emin >= -699) & (fmin2 >= 0x1.0p-128) & (zmax < EM_SMALL_Z);
}

DEV int track_csbend(particle &p, eh_opc &op, eh_zc *z) {
  const int flags = op.flags;
  const double ct = op.d[EH_D_CT], st = op.d[EH_D_ST];
  const double rho0 = op.d[EH_D_RHO0], rhoa = op.d[EH_D_RHOA];
  double x, xp, y, yp, s, dp, dp0;
  /* entry: misalignment then rotation by the total tilt (csbend.c:1120-1131) */
  p.s += op.d[EH_D_DZI] * em_sqrt(1 + sq(p.xp) + sq(p.yp));
  p.x = p.x + op.d[EH_D_DXI] + op.d[EH_D_DZI] * p.xp;
  p.y = p.y + op.d[EH_D_DYI] + op.d[EH_D_DZI] * p.yp;
  x = p.x * ct + p.y * st;
  y = -p.x * st + p.y * ct;
  xp = p.xp * ct + p.yp * st;
  yp = -p.xp * st + p.yp * ct;
  s = p.s;
  dp = dp0 = p.dp;
  if (flags & EH_F_EDGE1) {
    double rho = (1 + dp) * rhoa;
    double delta_xp = op.d[EH_D_TANE1] / rho * x;
    if ((flags & EH_F_KLIM1) && __builtin_fabs(delta_xp) > op.d[EH_D_KLIM1])
      delta_xp = (delta_xp > 0 ? 1 : -1) * op.d[EH_D_KLIM1];
    xp += delta_xp;
    double te = em_tan(op.d[EH_D_E1] - op.d[EH_D_PSI1] / (1 + dp));
    yp -= te / rho * y;
  }
  /* canonical (csbend.c:1411-1419) */
  double X = x, QX, Y = y, QY, S = 0, DP = dp;
  {
    double f = (1 + DP) / em_sqrt(1 + sq(xp) + sq(yp));
    QX = xp * f;
    QY = yp * f;
  }
  /* integrate_csbend_ordn (csbend.c:1434-1693) */
  double dist = 0, dz_lost = 0;
  bool lost = csbend_body(X, QX, Y, QY, DP, dist, dz_lost, op);
  if (!lost) {
    dz_lost = op.d[EH_D_NS];
    if (!in_aperture(X, Y, op))
      lost = true;
    else
      S += dist;
  }
  {
    /* convertFromDipoleCanonicalCoordinates (csbend.c:1421-1429) */
    double f = 1 / em_sqrt(sq(1 + DP) - sq(QX) - sq(QY));
    QX *= f;
    QY *= f;
  }
  if (lost) {
    /* memcpy(Qf) + convertFromCSBendCoords (csbend.c:1237-1239, 4502-4524) */
    p.x = X * ct - Y * st;
    p.y = X * st + Y * ct;
    p.xp = QX * ct - QY * st;
    p.yp = QX * st + QY * ct;
    p.s = opc(&z[0]) + dz_lost;
    p.dp = op.Po * (1 + DP);
    return EH_STAGE_ELEMENT + 1;
  }
  /* velocity rescaling of s (csbend.c:1280-1292) */
  {
    double p0 = op.Po * (1 + dp0);
    double beta0 = p0 / em_sqrt(sq(p0) + 1);
    double p1 = op.Po * (1 + DP);
    double beta1 = p1 / em_sqrt(sq(p1) + 1);
    s = beta1 * s / beta0 + S;
  }
  x = X;
  xp = QX;
  y = Y;
  yp = QY;
  dp = DP;
  if (flags & EH_F_EDGE2) {
    double rho = (1 + dp) * rhoa;
    double delta_xp = op.d[EH_D_TANE2] / rho * x;
    if ((flags & EH_F_KLIM2) && __builtin_fabs(delta_xp) > op.d[EH_D_KLIM2])
      delta_xp = (delta_xp > 0 ? 1 : -1) * op.d[EH_D_KLIM2];
    xp += delta_xp;
    double te = em_tan(op.d[EH_D_E2] - op.d[EH_D_PSI2] / (1 + dp));
    yp -= te / rho * y;
  }
  /* the error tilt's exit offsets, zero without one (csbend.c:1359-1364) */
  double o0 = 0.0, o1 = 0.0, o2 = 0.0, o3 = 0.0, o4 = 0.0;
  if (flags & EH_F_ETILT) {
    o0 = opc(&op.d[EH_D_ET]);
    o1 = opc(&op.d[EH_D_ET + 1]);
    o2 = opc(&op.d[EH_D_ET + 2]);
    o3 = opc(&op.d[EH_D_ET + 3]);
    o4 = opc(&op.d[EH_D_ET + 4]);
  }
  p.x = x * ct - y * st + o0;
  p.y = x * st + y * ct + o2;
  p.xp = xp * ct - yp * st + o1;
  p.yp = xp * st + yp * ct + o3;
  p.s = s + o4;
  p.dp = dp;
  p.x += op.d[EH_D_DXF] + op.d[EH_D_DZF] * p.xp;
  p.y += op.d[EH_D_DYF] + op.d[EH_D_DZF] * p.yp;
  p.s += op.d[EH_D_DZF] * em_sqrt(1 + sq(p.xp) + sq(p.yp));
  return 0;
}

/* tan of a fringe field's edge angle, which depends on the particle */
static __device__ __attribute__((noinline)) double edge_tan(double a) { return em_tan(a); }

/* track_through_csbend on the common path: the general code's operations
 * with the unscaled quotients and roots; false: p is not to be used.  Beside
 * csbend_body_fast's conditions the slopes, the path and the momentum are
 * moderate, and the host has checked the edges (EH_F_FAST).  1 + delta, the
 * edges' radius and the velocity are the same at both ends (nothing changes
 * delta here), so each has one reciprocal. */
enum bend_kind { DIPOLE, FIELD_BEND, ANY_DIPOLE };
template <bend_kind KIND> DEV bool track_csbend_fast(particle &p, const hdr_t H, hdr_t next, eh_opc &op) {
  const int flags = HD_FLAGS(H);
  if (!(flags & (KIND == ANY_DIPOLE ? EH_F_SMALL | EH_F_FAST : EH_F_FAST)) ||
      (KIND != FIELD_BEND && (flags & EH_F_FIELD)))
    return false;
  const bendc_t m = load_bendc(op, next);
  const bend_t B = load_bend(op);
  const double rhoa = m.rhoa, dzi = B.dzi, dzf = B.dzf;
  const double dp = p.dp, opd = 1 + dp, r_opd = em_recip(opd);
  bool good = (__builtin_fabs(p.xp) + __builtin_fabs(p.yp) <= 0x1.0p+60) & (__builtin_fabs(p.s) <= 0x1.0p+500) &
              (__builtin_amdgcn_frexp_exp(p.s) >= -500);
  p.s += dzi != 0 ? dzi * em_sqrt_mid(1 + sq(p.xp) + sq(p.yp)) : dzi;
  p.x = p.x + B.dxi + dzi * p.xp;
  p.y = p.y + B.dyi + dzi * p.yp;
  double x = p.x * B.ct + p.y * B.st;
  double y = -p.x * B.st + p.y * B.ct;
  double xp = p.xp * B.ct + p.yp * B.st;
  double yp = -p.xp * B.st + p.yp * B.ct;
  double rho = 1.0, r_rho = 1.0;
  if (flags & (EH_F_EDGE1 | EH_F_EDGE2)) {
    rho = opd * rhoa;
    r_rho = em_recip(rho);
    good &= (rho >= 0x1.0p-64) & (rho <= 0x1.0p+64);
  }
  if (flags & EH_F_EDGE1) {
    double delta_xp = em_div_pos(B.tane1, rho, r_rho) * x;
    if ((flags & EH_F_KLIM1) && __builtin_fabs(delta_xp) > op.d[EH_D_KLIM1])
      delta_xp = (delta_xp > 0 ? 1 : -1) * op.d[EH_D_KLIM1];
    xp += delta_xp;
    double te = B.te1;
    if (flags & EH_F_PSI1)
      te = edge_tan(op.d[EH_D_E1] - em_div_pos(op.d[EH_D_PSI1], opd, r_opd));
    yp -= em_div_pos(te, rho, r_rho) * y;
  }
  double X = x, Y = y, dist = 0, r, g = em_sqrt_recip_mid(1 + sq(xp) + sq(yp), &r);
  const double f = em_div_pos(opd, g, r);
  double QX = xp * f, QY = yp * f;
  good &= __builtin_fabs(xp) + __builtin_fabs(yp) <= 0x1.0p+60;
  /* the 4th-order integrator's four substeps of a slice unrolled (NSUB = 4):
   * the scheduler overlaps neighbouring substeps */
  if (KIND == FIELD_BEND)
    good &= csbend_field_fast(X, QX, Y, QY, opd, r_opd, dist, H, m, op);
  else if (KIND == ANY_DIPOLE && op.nsub == 4 && !(flags & EH_F_WIDE))
    good &= csbend_body_fast<4, false, true>(X, QX, Y, QY, opd, r_opd, dist, H, m, op);
  else if (KIND == ANY_DIPOLE)
    good &= csbend_body_fast<0, true, true>(X, QX, Y, QY, opd, r_opd, dist, H, m, op);
  else if (op.nsub == 4 && !(flags & EH_F_WIDE))
    good &= csbend_body_fast<4, false, false>(X, QX, Y, QY, opd, r_opd, dist, H, m, op);
  else
    good &= csbend_body_fast<0, true, false>(X, QX, Y, QY, opd, r_opd, dist, H, m, op);
  good &= in_bounds<KIND == ANY_DIPOLE>(X, Y, m.b, flags, op);
  {
    const double den2 = sq(opd) - sq(QX) - sq(QY);
    good &= den2 >= 0x1.0p-128;
    g = em_sqrt_recip_mid(den2, &r);
    const double q = em_div_pos(1.0, g, r);
    QX *= q;
    QY *= q;
  }
  /* velocity rescaling of s: beta1 = beta0 */
  const double p0 = B.po * opd;
  good &= (p0 >= 0x1.0p-60) & (p0 <= 0x1.0p+60);
  g = em_sqrt_recip_mid(sq(p0) + 1, &r);
  const double beta0 = em_div_pos(p0, g, r);
  const double s = em_div_pos(beta0 * p.s, beta0, em_recip(beta0)) + dist;
  x = X;
  xp = QX;
  y = Y;
  yp = QY;
  if (flags & EH_F_EDGE2) {
    double delta_xp = em_div_pos(B.tane2, rho, r_rho) * x;
    if ((flags & EH_F_KLIM2) && __builtin_fabs(delta_xp) > op.d[EH_D_KLIM2])
      delta_xp = (delta_xp > 0 ? 1 : -1) * op.d[EH_D_KLIM2];
    xp += delta_xp;
    double te = B.te2;
    if (flags & EH_F_PSI2)
      te = edge_tan(op.d[EH_D_E2] - em_div_pos(op.d[EH_D_PSI2], opd, r_opd));
    yp -= em_div_pos(te, rho, r_rho) * y;
  }
  double o0 = 0.0, o1 = 0.0, o2 = 0.0, o3 = 0.0, o4 = 0.0;
  if (flags & EH_F_ETILT) {
    o0 = op.d[EH_D_ET];
    o1 = op.d[EH_D_ET + 1];
    o2 = op.d[EH_D_ET + 2];
    o3 = op.d[EH_D_ET + 3];
    o4 = op.d[EH_D_ET + 4];
  }
  const double ct = B.ct, st = B.st;
  p.x = x * ct - y * st + o0;
  p.y = x * st + y * ct + o2;
  p.xp = xp * ct - yp * st + o1;
  p.yp = xp * st + yp * ct + o3;
  p.s = s + o4;
  p.x += B.dxf + dzf * p.xp;
  p.y += B.dyf + dzf * p.yp;
  good &= __builtin_fabs(p.xp) + __builtin_fabs(p.yp) <= 0x1.0p+60;
  p.s += dzf != 0 ? dzf * em_sqrt_mid(1 + sq(p.xp) + sq(p.yp)) : dzf;
  return good;
}

/* ---- RFCA ---- */

/* add_to_particle_energy (simple_rfca.c:987-1007) */
DEV void add_energy(particle &p, double tof, double Po, double dgamma) {
  double P = Po * (1 + p.dp);
  double gamma = em_sqrt(P * P + 1);
  double gamma1 = gamma + dgamma;
  if (gamma1 <= 1)
    gamma1 = 1 + 1e-7;
  double P1 = em_sqrt(gamma1 * gamma1 - 1);
  p.dp = (P1 - Po) / Po;
  p.s = tof * EH_C_MKS * P1 / gamma1;
  double Pz = P / em_sqrt(1 + sq(p.xp) + sq(p.yp));
  double Pz1 = em_sqrt(Pz * Pz + gamma1 * gamma1 - gamma * gamma);
  double ratio = Pz / Pz1;
  p.xp *= ratio;
  p.yp *= ratio;
}

/* trackRfCavityWithWakes for one particle, forward tracking, no wakes
 * (simple_rfca.c:557-984) followed by removeInvalidParticles (:975) */
DEV int track_rfca(particle &p, eh_opc &op, eh_zc *z) {
  const double Po = op.Po;
  const double volt = op.d[EH_D_VOLT], omega = op.d[EH_D_OMEGA], phase = op.d[EH_D_PHASE];
  const double length = op.d[EH_D_LENGTH], dtLight = op.d[EH_D_DTLIGHT];
  const int nKicks = op.nkicks_rf;
  /* CHANGE_T (simple_rfca.c:488-497): whole RF periods in the arrival time
   * of the beam's first row, which the host supplies, or of the particle
   * itself when every particle is its own beam */
  double timeOffset = op.d[EH_D_TOFF];
  if (op.flags & EH_F_CHT_SELF) {
    const double To = op.d[EH_D_TO];
    double P = Po * (1 + p.dp);
    double beta_i = P / em_sqrt(sq(P) + 1);
    double t = p.s / (EH_C_MKS * beta_i);
    timeOffset = t > (0.9 * To) ? (double)(int64_t)(t / To + 0.5) * To : 0.0;
  }
  const bool change_t = (op.flags & EH_F_CHANGE_T) && timeOffset != 0;
  p.x -= op.d[EH_D_RFDX];
  p.y -= op.d[EH_D_RFDY];
  if (!(op.flags & EH_F_MATRIX)) {
    double inverseF = 0;
    for (int ik = 0; ik < nKicks; ik++) {
      if (p.dp != -1) {
        double dc4 = length ? length / 2 * em_sqrt(1 + sq(p.xp) + sq(p.yp)) : 0;
        double P = Po * (1 + p.dp);
        double gamma = em_sqrt(sq(P) + 1);
        double beta_i = P / gamma;
        double t = (p.s + dc4) / (EH_C_MKS * beta_i) - timeOffset;
        if (ik == 0 && change_t)
          p.s = t * EH_C_MKS * beta_i - dc4;
        double phi = omega * (t - 0 - ik * dtLight) + phase;
        double dgamma = volt * em_sin(phi) * 1;
        if (length) {
          if ((op.flags & EH_F_END1FOCUS) && ik == 0) {
            inverseF = dgamma / (2 * gamma * length);
            p.xp -= p.x * inverseF;
            p.yp -= p.y * inverseF;
          }
          p.x += p.xp * length / 2;
          p.y += p.yp * length / 2;
          p.s += length / 2 * em_sqrt(1 + sq(p.xp) + sq(p.yp));
        }
        add_energy(p, t, Po, dgamma);
        double gamma1 = gamma + dgamma;
        if (gamma1 <= 1)
          p.dp = -1;
        else
          inverseF = -dgamma / (2 * gamma1 * length);
      }
      if (length) {
        p.x += p.xp * length / 2;
        p.y += p.yp * length / 2;
        p.s += length / 2 * em_sqrt(1 + sq(p.xp) + sq(p.yp));
        if ((op.flags & EH_F_END2FOCUS) && ik == nKicks - 1) {
          p.xp -= p.x * inverseF;
          p.yp -= p.y * inverseF;
        }
      }
    }
  } else {
    for (int ik = 0; ik < nKicks; ik++) {
      double P = Po * (1 + p.dp);
      double gamma = em_sqrt(sq(P) + 1);
      double beta_i = P / gamma;
      double ds1 = length / 2 * em_sqrt(1 + sq(p.xp) + sq(p.yp));
      double t = (p.s + ds1) / (EH_C_MKS * beta_i) - timeOffset;
      if (change_t)
        p.s = t * EH_C_MKS * beta_i - ds1;
      double sin_phase = em_sin(omega * (t - 0 - ik * dtLight) + phase);
      double dgamma = volt * 1 * sin_phase;
      if ((op.flags & EH_F_END1FOCUS) && length && ik == 0) {
        double inverseF = dgamma / (2 * gamma * length);
        p.xp -= p.x * inverseF;
        p.yp -= p.y * inverseF;
      }
      double dP = em_sqrt(sq(gamma + dgamma) - 1) - P;
      double R22 = 1 / (1 + dP / P), R12, R11 = 1, R21 = 0;
      if (__builtin_fabs(dP / P) > 1e-14)
        R12 = length * (P / dP * em_log(1 + dP / P));
      else
        R12 = length;
      p.s += ds1;
      double xx = p.x, xxp = p.xp;
      p.x = xx * R11 + xxp * R12;
      p.xp = xx * R21 + xxp * R22;
      xx = p.y;
      xxp = p.yp;
      p.y = xx * R11 + xxp * R12;
      p.yp = xx * R21 + xxp * R22;
      p.s += length / 2 * em_sqrt(1 + sq(p.xp) + sq(p.yp));
      p.dp = (P + dP - Po) / Po;
      if ((gamma += dgamma) <= 1)
        p.dp = -1;
      if ((op.flags & EH_F_END2FOCUS) && length && ik == nKicks - 1) {
        double inverseF = -dgamma / (2 * gamma * length);
        p.xp -= p.x * inverseF;
        p.yp -= p.y * inverseF;
      }
      p.s = (P + dP) / gamma * p.s / beta_i;
    }
  }
  p.x += op.d[EH_D_RFDX];
  p.y += op.d[EH_D_RFDY];
  /* removeInvalidParticles (limit_amplitudes.c:274-320) */
  if (__builtin_isnan(p.x) || __builtin_isnan(p.xp) || __builtin_isnan(p.y) || __builtin_isnan(p.yp) ||
      __builtin_isnan(p.s) || __builtin_isnan(p.dp) || p.dp <= -1) {
    p.s = opc(&z[1]);
    p.dp = Po * (1 + p.dp);
    return EH_STAGE_ELEMENT + 1;
  }
  return 0;
}

/* offset_beam (do_tracking.c:3243-3306) for one particle, on pass ON_PASS
 * or, with -1, every pass (do_tracking.c:1818-1822) */
DEV void track_malign(particle &p, eh_opc &op, int64_t pass) {
  const int32_t on_pass = op.nkicks_rf;
  if (!(on_pass == -1 || on_pass == pass))
    return;
  const double dz = op.d[EH_D_MA_DZ];
  const double dt = op.d[EH_D_MA_DT], ddp = op.d[EH_D_MA_DP], de = op.d[EH_D_MA_DE];
  const double Po = op.Po;
  double ds = dz ? dz * em_sqrt(1 + sq(p.xp) + sq(p.yp)) : 0;
  p.x += op.d[EH_D_MA_DX] + dz * p.xp;
  p.xp += op.d[EH_D_MA_DXP];
  p.y += op.d[EH_D_MA_DY] + dz * p.yp;
  p.yp += op.d[EH_D_MA_DYP];
  p.s += ds;
  if (dt || ddp || de) {
    double pc = Po * (1 + p.dp);
    double gamma = em_sqrt(1 + pc * pc);
    double beta = pc / gamma;
    const double t = p.s / (beta * EH_C_MKS) + dt;
    if (ddp) {
      p.dp += ddp;
      pc = Po * (1 + p.dp);
      beta = pc / em_sqrt(1 + pc * pc);
    }
    if (de) {
      gamma += de * gamma;
      pc = em_sqrt(gamma * gamma - 1);
      beta = pc / gamma;
      p.dp = (pc - Po) / Po;
    }
    p.s = t * beta * EH_C_MKS;
  }
}

/* rectangular_collimator (limit_amplitudes.c:32-185), the entrance check:
 * lost outside the half-widths (an open side may spare it) or with a
 * non-finite x or y, INVERT swapping the verdict; the loss at the
 * element's start */
DEV int track_rcol_in(particle &p, eh_opc &op, eh_zc *z) {
  const double xsize = op.d[EH_D_RC_XMAX], ysize = op.d[EH_D_RC_YMAX];
  const double dx = p.x - op.d[EH_D_RC_DX], dy = p.y - op.d[EH_D_RC_DY];
  const int open = op.order1;
  bool lost = false;
  if ((xsize > 0 && __builtin_fabs(dx) > xsize) || (ysize > 0 && __builtin_fabs(dy) > ysize))
    lost = open ? ap_open_lost(open, dx, dy, xsize, ysize) : true;
  else if (__builtin_isinf(p.x) || __builtin_isinf(p.y) || __builtin_isnan(p.x) || __builtin_isnan(p.y))
    lost = true;
  if (op.order0)
    lost = !lost;
  if (lost) {
    p.s = opc(&z[0]);
    p.dp = op.Po * (1 + p.dp);
    return EH_STAGE_ELEMENT + 1;
  }
  return 0;
}

/* the collimator's drift and exit check: a particle outside at the exit
 * is lost where its straight orbit met the jaw (no open side), a
 * non-finite exit position at the exit; survivors take the drift */
DEV int track_rcol_body(particle &p, eh_opc &op, eh_zc *z) {
  const double length = op.d[EH_D_RC_LEN];
  const double xsize = op.d[EH_D_RC_XMAX], ysize = op.d[EH_D_RC_YMAX];
  const double xc = op.d[EH_D_RC_DX], yc = op.d[EH_D_RC_DY];
  const int open = op.order1;
  const double x1 = p.x + length * p.xp, y1 = p.y + length * p.yp;
  const double dx = x1 - xc, dy = y1 - yc;
  const double z0 = opc(&z[0]);
  int is_out = 0;
  if (xsize > 0 && __builtin_fabs(dx) > xsize)
    is_out += 1 * (open ? (ap_open_lost(open, dx, 0, xsize, ysize) ? 1 : 0) : 1);
  if (ysize > 0 && __builtin_fabs(dy) > ysize)
    is_out += 2 * (open ? (ap_open_lost(open, 0, dy, xsize, ysize) ? 1 : 0) : 1);
  if (__builtin_isinf(x1) || __builtin_isinf(y1) || __builtin_isnan(x1) || __builtin_isnan(y1))
    is_out += 4;
  if (is_out & 4) {
    p.s = z0 + length;
    p.x = x1;
    p.y = y1;
    p.dp = op.Po * (1 + p.dp);
    return EH_STAGE_ELEMENT + 1;
  }
  if ((is_out && !op.order0) || (!is_out && op.order0)) {
    if (!open) {
      double zx = 1.7976931348623157e308, zy = 1.7976931348623157e308;
      if ((is_out & 1) && p.xp != 0)
        zx = ((p.xp > 0 ? 1 : -1) * xsize - (p.x - xc)) / p.xp;
      if ((is_out & 2) && p.yp != 0)
        zy = ((p.yp > 0 ? 1 : -1) * ysize - (p.y - yc)) / p.yp;
      const double zz = zx < zy ? zx : zy;
      p.x += p.xp * zz;
      p.y += p.yp * zz;
      p.s = z0 + zz;
    }
    p.dp = op.Po * (1 + p.dp);
    return EH_STAGE_ELEMENT + 1;
  }
  p.s += length * em_sqrt(1 + sq(p.xp) + sq(p.yp));
  p.x = x1;
  p.y = y1;
  return 0;
}

/* The general code, out of line: it decides for the lanes that a common path
 * hands on, and for element kinds met once a turn or less.  Inlined, its
 * polynomials and branches took the registers of the common paths (11,500
 * instructions with scalar values spilled to vector lanes around every
 * element; 4,600 now).  FODO ring, 10^4 particles, 64 turns: 54.9 -> 44.9 ms;
 * storage ring, 10^6, 10 turns: 258 -> 242 ms. */
struct step_out {
  particle p;
  int lost;
};
#define SLOW static __device__ __attribute__((noinline)) step_out

/* a pointer that every lane holds alike, back in scalar registers */
template <class T> DEV T *uniform(T *p) {
  const uint64_t u = (uint64_t)p;
  return (T *)(((uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)(u >> 32)) << 32) |
               (uint32_t)__builtin_amdgcn_readfirstlane((int)u));
}

/* the common path for lanes beyond an ellipse's box but inside the ellipse
 * (eh_op_finish), part of slow_multipole: called from it, it cost the kernels
 * scalar registers that they keep across (FODO ring of 10^4 particles 37.2 ms,
 * 36.4 so).  lost < 0: not taken, the row as it came */
DEV step_out slow_multipole_ell(particle p, eh_opc *op) {
  step_out o;
  eh_opc &u = *uniform(op);
  const hdr_t H = load_hdr(&u);
  o.p = p;
  o.lost = 0;
  if (!track_multipole_fast<true>(o.p, H, load_mult(u, H), u)) {
    o.p = p;
    o.lost = -1;
  }
  return o;
}

SLOW slow_multipole(particle p, eh_opc *op, eh_zc *z) {
  step_out o;
  eh_opc &u = *uniform(op);
  if (u.flags & EH_F_INELL) {
    o = slow_multipole_ell(p, &u);
    if (!o.lost)
      return o;
    p = o.p;
  }
  o.lost = track_multipole(p, u, uniform(z));
  o.p = p;
  return o;
}

/* the common path of small bends, and of lanes beyond an ellipse's box, out of
 * line behind the general code's entry, so that the others keep their code and
 * registers (as a branch of run_op it took the FODO ring of 10^4 particles from
 * 37 to 44 ms).  A ring of 20 correctors of 1e-6 rad, 10^4 particles, 10 turns:
 * 1.86 ms, 4.65 by the general code.  lost < 0: not taken, the row as it came */
SLOW slow_csbend_any(particle p, eh_opc *op) {
  step_out o;
  eh_opc &u = *uniform(op);
  const hdr_t H = load_hdr(&u);
  o.p = p;
  o.lost = 0;
  if (!track_csbend_fast<ANY_DIPOLE>(o.p, H, H, u)) {
    o.p = p;
    o.lost = -1;
  }
  return o;
}

SLOW slow_csbend(particle p, eh_opc *op, eh_zc *z) {
  step_out o;
  eh_opc &u = *uniform(op);
  if (u.flags & (EH_F_SMALL | EH_F_INELL)) {
    o = slow_csbend_any(p, &u);
    if (!o.lost)
      return o;
    p = o.p;
  }
  o.lost = track_csbend(p, u, uniform(z));
  o.p = p;
  return o;
}

/* the same with the common path of combined-function bends, out of line with
 * its registers.  Only the tracking kernel takes it: in the batch kernel the
 * values kept across the call spill (27 VGPRs with two particles per lane),
 * and an aperture study without such bends took 96 ms where it takes 83 */
SLOW slow_csbend_field(particle p, eh_opc *op, eh_zc *z) {
  step_out o;
  eh_opc &u = *uniform(op);
  const hdr_t H = load_hdr(&u);
  o.p = p;
  o.lost = 0;
  if ((HD_FLAGS(H) & EH_F_FIELD) && track_csbend_fast<FIELD_BEND>(o.p, H, H, u))
    return o;
  if (HD_FLAGS(H) & (EH_F_SMALL | EH_F_INELL)) {
    o = slow_csbend_any(p, &u);
    if (!o.lost)
      return o;
    p = o.p;
  }
  o.lost = track_csbend(p, u, uniform(z));
  o.p = p;
  return o;
}

SLOW slow_rfca(particle p, eh_opc *op, eh_zc *z) {
  step_out o;
  o.lost = track_rfca(p, *uniform(op), uniform(z));
  o.p = p;
  return o;
}

/* the rare kinds: MALIGN, RCOL */
SLOW slow_other(particle p, eh_opc *op, eh_zc *z, int64_t pass) {
  step_out o;
  eh_opc &u = *uniform(op);
  eh_zc *zu = uniform(z);
  o.lost = 0;
  if (u.op == EH_OP_MALIGN)
    track_malign(p, u, pass);
  else
    o.lost = u.op == EH_OP_RCOL_IN ? track_rcol_in(p, u, zu) : track_rcol_body(p, u, zu);
  o.p = p;
  return o;
}

SLOW slow_drift2(particle p, double L, double hL) {
  step_out o;
  drift2_exact(p, L, hL);
  o.lost = 0;
  o.p = p;
  return o;
}

SLOW slow_checks(particle p, eh_opc *op, eh_zc *z) {
  step_out o;
  o.lost = post_element_checks(p, *uniform(op), uniform(z));
  o.p = p;
  return o;
}

/* One element on one particle.  z points at the element's (z_start, z_end),
 * which only the loss paths read: in the element record itself, or in the
 * position table of a program whose repeated cells share one record. */
template <bool FIELD> DEV int run_op(particle &p, const hdr_t H, hdr_t next, eh_opc &op, eh_zc *z, int64_t pass) {
  const int code = HD_OP(H);
  step_out o;
  o.lost = 0;
  /* elements before the recirculation point act on pass 0 only */
  if ((HD_FLAGS(H) & EH_F_FIRSTPASS) && pass != 0)
    return 0;
  if (code == EH_OP_MULT) {
    particle q = p;
    const mult_t m = load_mult(op, next);
    const bool done = track_multipole_fast<false>(q, H, m, op);
    if (ALL_LANES(done))
      p = q;
    else if (done)
      p = q;
    else {
      o = slow_multipole(p, &op, z);
      p = o.p;
    }
  } else if (code == EH_OP_DRIFT2) {
    double L = op.hot[EH_H_L], hL = op.hot[EH_H_L + 1];
    asm volatile("" : "+s"(L), "+s"(hL) : "s"(next));
    if ((HD_FLAGS(H) & EH_F_DFAST) && ALL_LANES(drift2_ok(p)))
      drift2(p, L, hL);
    else
      p = slow_drift2(p, L, hL).p;
  } else if (code == EH_OP_CSBEND) {
    particle q = p;
    const bool done = track_csbend_fast<DIPOLE>(q, H, next, op);
    if (ALL_LANES(done))
      p = q;
    else if (done)
      p = q;
    else {
      o = FIELD ? slow_csbend_field(p, &op, z) : slow_csbend(p, &op, z);
      p = o.p;
    }
  } else {
    switch (code) {
    case EH_OP_DRIFT1:
      drift1(p, op.d[0]);
      break;
    case EH_OP_EXACT_DRIFT:
      exact_drift(p, op.d[0]);
      break;
    case EH_OP_MATRIX1:
      matrix1(p, op.d);
      break;
    case EH_OP_RFCA:
      o = slow_rfca(p, &op, z);
      p = o.p;
      break;
    case EH_OP_MALIGN:
    case EH_OP_RCOL_IN:
    case EH_OP_RCOL_BODY:
      o = slow_other(p, &op, z, pass);
      p = o.p;
      break;
    case EH_OP_RFCA_DRIFT:
      /* VOLT=0: a drift when the cavity has length, else nothing (simple_rfca.c:389-402) */
      if (op.d[EH_D_RFLEN_TOTAL] != 0) {
        p.x += p.xp * op.d[EH_D_RFLEN_TOTAL];
        p.y += p.yp * op.d[EH_D_RFLEN_TOTAL];
        p.s += op.d[EH_D_RFLEN_TOTAL] * em_sqrt(1 + sq(p.xp) + sq(p.yp));
      }
      break;
    default:
      break;
    }
  }
  if (o.lost)
    return o.lost;
  /* inside these bounds none of the checks after the element can fire */
  const bool inside = (__builtin_fabs(p.x) <= op.hot[EH_H_CHKX]) & (__builtin_fabs(p.y) <= op.hot[EH_H_CHKY]);
  if (!ALL_LANES(inside) && !inside) {
    o = slow_checks(p, &op, z);
    p = o.p;
  }
  return o.lost;
}

/* Four waves per SIMD (up to 128 VGPRs).  The bound reaches the general code's
 * functions only if every kernel that calls them states it: the batch kernel
 * does too (without it they took 148 VGPRs, three waves).
 * The beamline of nflat elements arrives as runs (eh_run): a body of
 * records executed reps times in a row, so a ring of identical cells keeps
 * one cell's records hot in the scalar cache instead of streaming every
 * element's record through it each pass.  Loss codes and op_first/op_last
 * count positions in the flat beamline; zpos holds (z_start, z_end) for
 * each of them. */
__global__ void __launch_bounds__(256, 4) eh_track_kernel(eh_state st, const eh_op *__restrict__ ops,
                                                       const eh_run *__restrict__ runs, int32_t nruns,
                                                       const double *__restrict__ zpos, int64_t pass0,
                                                       int32_t npasses, int32_t op_first, int32_t op_last,
                                                       int32_t nflat) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= st.n)
    return;
  if (st.loss_pass[i] >= 0)
    return;
  particle p;
  p.x = st.x[i];
  p.xp = st.xp[i];
  p.y = st.y[i];
  p.yp = st.yp[i];
  p.s = st.s[i];
  p.dp = st.dp[i];
  eh_opc *cops = (eh_opc *)ops;
  eh_zc *zs = (eh_zc *)zpos;
  EH_CONST eh_run *cruns = (EH_CONST eh_run *)runs;
  /* the loops are the same for all lanes; a lost lane sits out (its mask would
   * otherwise be kept at every loop level) */
  int lost = 0, lost_op = 0, lost_pass = 0;
  for (int32_t ip = 0; ip < npasses; ip++) {
    /* element positions [ob, oe) of the flat beamline in this pass */
    const int32_t ob = (ip == 0) ? op_first : 0;
    const int32_t oe = (ip == npasses - 1) ? op_last : nflat;
    if (ALL_LANES(lost))
      break;
    for (int32_t r = 0; r < nruns; r++) {
      const int32_t fs = cruns[r].flat, len = cruns[r].len, first = cruns[r].first;
      const int32_t fe = fs + len * cruns[r].reps;
      if (fe <= ob)
        continue;
      if (fs >= oe)
        break;
      int32_t f = fs > ob ? fs : ob;
      const int32_t f1 = fe < oe ? fe : oe;
      eh_opc *op0 = cops + first, *op1 = op0 + len, *op = op0 + (f - fs) % len;
      hdr_t h = load_hdr(op);
      for (; f < f1; f++) {
        eh_opc *nxt = op + 1 == op1 ? op0 : op + 1;
        hdr_t hn = load_hdr(nxt);
        if (!lost) {
          lost = run_op<true>(p, h, hn, *op, zs + 2 * f, pass0 + ip);
          if (lost) {
            lost_op = f;
            lost_pass = ip;
          }
        }
        op = nxt;
        h = hn;
      }
    }
  }
  st.x[i] = p.x;
  st.xp[i] = p.xp;
  st.y[i] = p.y;
  st.yp[i] = p.yp;
  st.s[i] = p.s;
  st.dp[i] = p.dp;
  if (lost) {
    st.loss_pass[i] = (int32_t)(pass0 + lost_pass);
    st.loss_code[i] = 4 * lost_op + (lost - 1);
  }
}

/* Persistent batch kernel: each workgroup pulls chunks (a variant and a run
 * of its particles) from a queue until it is empty; every lane tracks PPL
 * particles of the chunk through the variant's program.  The chunk queue is
 * ordered by variant so that workgroups resident at the same time share a few
 * programs in L2. */
template <int PPL>
__global__ void __launch_bounds__(256, 4) eh_batch_kernel(eh_state st, const eh_op *__restrict__ ops,
                                                       const eh_vdesc *__restrict__ vars,
                                                       const eh_chunk *__restrict__ chunks,
                                                       const int32_t *__restrict__ nchunks_p,
                                                       const int32_t *__restrict__ perm, int64_t pass0,
                                                       int32_t npasses, unsigned int *queue) {
  __shared__ int s_chunk;
  const int32_t nchunks = *nchunks_p; /* device-resident: a queue rebuilt on the device sets it */
  for (;;) {
    if (threadIdx.x == 0)
      s_chunk = (int)atomicAdd(queue, 1u);
    __syncthreads();
    const int c = s_chunk;
    __syncthreads();
    if (c >= nchunks)
      return;
    const eh_chunk ch = chunks[c];
    const eh_vdesc vd = vars[ch.variant];
    eh_opc *vops = (eh_opc *)ops + vd.op_offset;
    const int32_t nops = vd.nops;
    particle p[PPL];
    int lost[PPL], lost_op[PPL];
    int64_t lost_pass[PPL], idx[PPL];
    bool live[PPL];
    for (int k = 0; k < PPL; k++) {
      const int64_t local = threadIdx.x + (int64_t)k * blockDim.x;
      const bool in = local < ch.count;
      idx[k] = perm ? (in ? (int64_t)perm[ch.first + local] : 0) : ch.first + local;
      live[k] = in && st.loss_pass[idx[k]] < 0;
      lost[k] = 0;
      lost_op[k] = 0;
      lost_pass[k] = 0;
      if (live[k]) {
        p[k].x = st.x[idx[k]];
        p[k].xp = st.xp[idx[k]];
        p[k].y = st.y[idx[k]];
        p[k].yp = st.yp[idx[k]];
        p[k].s = st.s[idx[k]];
        p[k].dp = st.dp[idx[k]];
      }
    }
    for (int32_t ip = 0; ip < npasses; ip++) {
      bool any = false;
      for (int k = 0; k < PPL; k++)
        any |= live[k];
      if (!any)
        break;
      hdr_t h = load_hdr(vops);
      for (int32_t io = 0; io < nops; io++) {
        eh_opc &op = vops[io];
        const hdr_t hcur = h;
        h = load_hdr(vops + (io + 1 < nops ? io + 1 : 0));
        for (int k = 0; k < PPL; k++) {
          if (!live[k])
            continue;
          int l = run_op<false>(p[k], hcur, h, op, &op.z_start, pass0 + ip);
          if (l) {
            live[k] = false;
            lost[k] = l;
            lost_op[k] = io;
            lost_pass[k] = pass0 + ip;
          }
        }
      }
    }
    for (int k = 0; k < PPL; k++) {
      const int64_t local = threadIdx.x + (int64_t)k * blockDim.x;
      if (local >= ch.count)
        continue;
      if (live[k] || lost[k]) {
        const int64_t i = idx[k];
        st.x[i] = p[k].x;
        st.xp[i] = p[k].xp;
        st.y[i] = p[k].y;
        st.yp[i] = p[k].yp;
        st.s[i] = p[k].s;
        st.dp[i] = p[k].dp;
        if (lost[k]) {
          st.loss_pass[i] = (int32_t)lost_pass[k];
          st.loss_code[i] = 4 * lost_op[k] + (lost[k] - 1);
        }
      }
    }
  }
}

__global__ void eh_queue_reset(unsigned int *queue) { *queue = 0u; }

/* ---- rows <-> columns ----
 * One thread a row: both sides are streamed once (128 B a row, about 30 us for
 * 10^6 rows), against 6 ms for the copies to and from the host around them,
 * so nothing is staged through LDS. */

/* columns from rows; the loss records start here, and with cull rows with a
 * NaN or infinite x or y are lost before the first element */
__global__ void __launch_bounds__(256) rows_in(const double *__restrict__ rows, int64_t first, int64_t m, int32_t w,
                                               int32_t cull, double Po, eh_state st, double *ids) {
  const int64_t j = (int64_t)blockIdx.x * 256 + threadIdx.x, i = first + j;
  if (j >= m)
    return;
  const double *r = rows + j * w;
  double v[7];
#pragma unroll
  for (int k = 0; k < 7; k++)
    v[k] = r[k];
  const bool bad = cull && (__builtin_isinf(v[0]) || __builtin_isinf(v[2]) || __builtin_isnan(v[0]) ||
                            __builtin_isnan(v[2]));
  if (bad) {
    /* limit_amplitudes(DBL_MAX) at z = 0: s = 0, delta = Po(1+delta) */
    v[4] = 0.0;
    v[5] = Po * (1 + v[5]);
  }
  st.x[i] = v[0];
  st.xp[i] = v[1];
  st.y[i] = v[2];
  st.yp[i] = v[3];
  st.s[i] = v[4];
  st.dp[i] = v[5];
  ids[i] = v[6];
  st.loss_pass[i] = bad ? 0 : -1;
  st.loss_code[i] = bad ? -1 : 0;
}

/* columns 0..5 back into the rows, the loss records behind the last row */
__global__ void __launch_bounds__(256) rows_back(double *rows, int32_t w, eh_state st) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= st.n)
    return;
  double *r = rows + i * w;
  int32_t *rec = (int32_t *)(rows + st.n * w);
  r[0] = st.x[i];
  r[1] = st.xp[i];
  r[2] = st.y[i];
  r[3] = st.yp[i];
  r[4] = st.s[i];
  r[5] = st.dp[i];
  rec[i] = st.loss_pass[i];
  rec[st.n + i] = st.loss_code[i];
}

/* m rows of 8 columns in the given order (NULL: from slot first on), column 7
 * = pass of loss */
__global__ void __launch_bounds__(256) rows_out(double *__restrict__ out, eh_state st, const double *__restrict__ ids,
                                                int64_t first, int64_t m, const int32_t *__restrict__ order) {
  const int64_t j = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (j >= m)
    return;
  const int64_t i = order ? order[j] : first + j;
  double *r = out + 8 * j;
  r[0] = st.x[i];
  r[1] = st.xp[i];
  r[2] = st.y[i];
  r[3] = st.yp[i];
  r[4] = st.s[i];
  r[5] = st.dp[i];
  r[6] = ids[i];
  r[7] = st.loss_pass[i] >= 0 ? (double)st.loss_pass[i] : -1.0;
}

/* whole rows in the given order */
__global__ void __launch_bounds__(256) rows_gather(const double *__restrict__ in, double *__restrict__ out, int64_t n,
                                                   int32_t w, const int32_t *__restrict__ order) {
  const int64_t e = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (e >= n * w)
    return;
  out[e] = in[(int64_t)order[e / w] * w + e % w];
}

__global__ void __launch_bounds__(256) fiducial_times(eh_state st, int64_t first, int64_t m, double Po, double ahead,
                                                      double *t) {
  const int64_t j = (int64_t)blockIdx.x * 256 + threadIdx.x, i = first + j;
  if (j >= m)
    return;
  const double p = Po * (1 + st.dp[i]);
  const double beta = p / __builtin_sqrt(p * p + 1);
  t[j] = (st.s[i] + ahead) / (EH_C_MKS * beta);
}

/* out[0] += passes completed from pass0 on, out[1] += particles alive.  One
 * pair of atomics per workgroup: with a pair per wave, all on one line, 10^6
 * records took 102 us */
__global__ void __launch_bounds__(256) effort_sum(const int32_t *__restrict__ lp, int64_t n, int64_t pass0, int64_t end,
                                                  unsigned long long *out) {
  __shared__ unsigned long long we[4], wa[4];
  unsigned long long e = 0, a = 0;
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (int64_t)gridDim.x * 256) {
    const int64_t l = lp[i];
    if (l < 0) {
      e += (unsigned long long)(end - pass0);
      a++;
    } else if (l >= pass0)
      e += (unsigned long long)(l - pass0);
  }
  for (int off = 32; off > 0; off >>= 1) {
    e += __shfl_xor(e, off);
    a += __shfl_xor(a, off);
  }
  if ((threadIdx.x & 63) == 0) {
    we[threadIdx.x >> 6] = e;
    wa[threadIdx.x >> 6] = a;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    atomicAdd(&out[0], we[0] + we[1] + we[2] + we[3]);
    atomicAdd(&out[1], wa[0] + wa[1] + wa[2] + wa[3]);
  }
}

__global__ void clear_counters(unsigned long long *c) {
  if (threadIdx.x < 2)
    c[threadIdx.x] = 0;
}

/* ------------------------------------------------------------ host side */

extern "C" {

static int hip_fail(ehd_dev *d, hipError_t e, const char *what) {
  if (d)
    snprintf(d->msg, sizeof(d->msg), "%s: %s", what, hipGetErrorString(e));
  return EH_ERR_HIP;
}

#define HIPCHK(d, call)                                                                                                \
  do {                                                                                                                 \
    hipError_t e_ = (call);                                                                                            \
    if (e_ != hipSuccess)                                                                                              \
      return hip_fail((d), e_, #call);                                                                                 \
  } while (0)

int ehd_create(int device, ehd_dev **out, char *msg, int msglen) {
  int count = 0;
  hipError_t e = hipGetDeviceCount(&count);
  if (e != hipSuccess || count <= 0) {
    if (msg && msglen > 0)
      snprintf(msg, msglen, "no HIP device available (%s)", hipGetErrorString(e));
    return EH_ERR_NODEVICE;
  }
  if (device < 0 || device >= count) {
    if (msg && msglen > 0)
      snprintf(msg, msglen, "device %d out of range (%d devices)", device, count);
    return EH_ERR_INVALID;
  }
  ehd_dev *d = (ehd_dev *)calloc(1, sizeof(ehd_dev));
  if (!d)
    return EH_ERR_NOMEM;
  d->device = device;
  d->block = 0; /* chosen per launch from the particle count */
  e = hipSetDevice(device);
  if (e == hipSuccess)
    e = hipStreamCreateWithFlags(&d->stream, hipStreamNonBlocking);
  if (e == hipSuccess)
    e = hipEventCreate(&d->ev0);
  if (e == hipSuccess)
    e = hipEventCreate(&d->ev1);
  if (e == hipSuccess)
    e = hipEventCreate(&d->cev0);
  if (e == hipSuccess)
    e = hipEventCreate(&d->cev1);
  if (e == hipSuccess)
    e = hipEventCreateWithFlags(&d->pev, hipEventDisableTiming);
  if (e != hipSuccess) {
    if (msg && msglen > 0)
      snprintf(msg, msglen, "HIP set-up failed: %s", hipGetErrorString(e));
    free(d);
    return EH_ERR_HIP;
  }
  int rc = ehd_noalloc_init(d);
  if (rc) {
    if (msg && msglen > 0)
      snprintf(msg, msglen, "%s", d->msg);
    ehd_destroy(d);
    return rc;
  }
  *out = d;
  return EH_OK;
}

void ehd_free_collective(ehd_dev *d);

/* teardown: errors are ignored, there is nothing left to undo */
void ehd_destroy(ehd_dev *d) {
  if (!d)
    return;
  (void)hipSetDevice(d->device);
  (void)hipStreamSynchronize(d->stream);
  void *bufs[] = {d->coord[0], d->coord[1], d->coord[2], d->coord[3], d->coord[4], d->coord[5],
                  d->loss_pass, d->loss_code, d->ops, d->counter, d->vdesc, d->chunks, d->perm, d->queue,
                  d->snap[0], d->snap[1], d->snap[2], d->snap[3], d->snap[4], d->snap[5], d->snap_lp, d->snap_lc,
                  d->tile_sum, d->pbuf, d->ids, d->rows, d->rows2, d->order};
  for (size_t k = 0; k < sizeof(bufs) / sizeof(bufs[0]); k++)
    if (bufs[k])
      (void)hipFree(bufs[k]);
  ehd_free_collective(d);
  free(d->host_prog);
  if (d->pstage)
    (void)hipHostFree(d->pstage);
  if (d->pin)
    (void)hipHostFree(d->pin);
  (void)hipEventDestroy(d->pev);
  (void)hipEventDestroy(d->ev0);
  (void)hipEventDestroy(d->ev1);
  (void)hipEventDestroy(d->cev0);
  (void)hipEventDestroy(d->cev1);
  (void)hipStreamDestroy(d->stream);
  free(d);
}

int ehd_alloc_state(ehd_dev *d, int64_t n) {
  d->upload++;
  d->rows_kept = 0;
  HIPCHK(d, hipSetDevice(d->device));
  if (n > d->cap) {
    for (int k = 0; k < 6; k++) {
      if (d->coord[k])
        HIPCHK(d, hipFree(d->coord[k]));
      d->coord[k] = NULL;
    }
    if (d->loss_pass)
      HIPCHK(d, hipFree(d->loss_pass));
    if (d->loss_code)
      HIPCHK(d, hipFree(d->loss_code));
    if (d->ids)
      HIPCHK(d, hipFree(d->ids));
    d->loss_pass = d->loss_code = NULL;
    d->ids = NULL;
    d->cap = 0;
    for (int k = 0; k < 6; k++)
      HIPCHK(d, hipMalloc((void **)&d->coord[k], sizeof(double) * (n > 0 ? n : 1)));
    HIPCHK(d, hipMalloc((void **)&d->loss_pass, sizeof(int32_t) * (n > 0 ? n : 1)));
    HIPCHK(d, hipMalloc((void **)&d->loss_code, sizeof(int32_t) * (n > 0 ? n : 1)));
    HIPCHK(d, hipMalloc((void **)&d->ids, sizeof(double) * (n > 0 ? n : 1)));
    d->cap = n;
  }
  if (!d->counter)
    HIPCHK(d, hipMalloc((void **)&d->counter, sizeof(unsigned long long) * 8));
  d->n = n;
  return EH_OK;
}

int64_t ehd_upload_id(const ehd_dev *d) { return d->upload; }

int ehd_put_state(ehd_dev *d, const double *x, const double *xp, const double *y, const double *yp, const double *s,
                  const double *dp, const int32_t *loss_pass, const int32_t *loss_code, int64_t n) {
  const double *src[6] = {x, xp, y, yp, s, dp};
  if (n != d->n)
    return EH_ERR_STATE;
  HIPCHK(d, hipSetDevice(d->device));
  for (int k = 0; k < 6; k++)
    HIPCHK(d, hipMemcpyAsync(d->coord[k], src[k], sizeof(double) * n, hipMemcpyHostToDevice, d->stream));
  HIPCHK(d, hipMemcpyAsync(d->loss_pass, loss_pass, sizeof(int32_t) * n, hipMemcpyHostToDevice, d->stream));
  HIPCHK(d, hipMemcpyAsync(d->loss_code, loss_code, sizeof(int32_t) * n, hipMemcpyHostToDevice, d->stream));
  HIPCHK(d, hipStreamSynchronize(d->stream));
  return EH_OK;
}

int ehd_get_state(ehd_dev *d, double *x, double *xp, double *y, double *yp, double *s, double *dp,
                  int32_t *loss_pass, int32_t *loss_code, int64_t n) {
  double *dst[6] = {x, xp, y, yp, s, dp};
  if (n != d->n)
    return EH_ERR_STATE;
  HIPCHK(d, hipSetDevice(d->device));
  for (int k = 0; k < 6; k++)
    if (dst[k])
      HIPCHK(d, hipMemcpyAsync(dst[k], d->coord[k], sizeof(double) * n, hipMemcpyDeviceToHost, d->stream));
  if (loss_pass)
    HIPCHK(d, hipMemcpyAsync(loss_pass, d->loss_pass, sizeof(int32_t) * n, hipMemcpyDeviceToHost, d->stream));
  if (loss_code)
    HIPCHK(d, hipMemcpyAsync(loss_code, d->loss_code, sizeof(int32_t) * n, hipMemcpyDeviceToHost, d->stream));
  HIPCHK(d, hipStreamSynchronize(d->stream));
  return EH_OK;
}

/* s, delta and loss pass of particle slot i alone (any may be NULL) */
int ehd_get_one(ehd_dev *d, int64_t i, double *s, double *dp, int32_t *loss_pass) {
  if (i < 0 || i >= d->n)
    return EH_ERR_INVALID;
  HIPCHK(d, hipSetDevice(d->device));
  if (s)
    HIPCHK(d, hipMemcpyAsync(s, d->coord[4] + i, sizeof(double), hipMemcpyDeviceToHost, d->stream));
  if (dp)
    HIPCHK(d, hipMemcpyAsync(dp, d->coord[5] + i, sizeof(double), hipMemcpyDeviceToHost, d->stream));
  if (loss_pass)
    HIPCHK(d, hipMemcpyAsync(loss_pass, d->loss_pass + i, sizeof(int32_t), hipMemcpyDeviceToHost, d->stream));
  HIPCHK(d, hipStreamSynchronize(d->stream));
  return EH_OK;
}

int ehd_get_sdp(ehd_dev *d, double *s, double *dp, int32_t *loss_pass, int64_t n) {
  return ehd_get_state(d, NULL, NULL, NULL, NULL, s, dp, loss_pass, NULL, n);
}

static eh_state state_of(const ehd_dev *d) {
  eh_state st;
  st.x = d->coord[0];
  st.xp = d->coord[1];
  st.y = d->coord[2];
  st.yp = d->coord[3];
  st.s = d->coord[4];
  st.dp = d->coord[5];
  st.loss_pass = d->loss_pass;
  st.loss_code = d->loss_code;
  st.n = d->n;
  return st;
}

static int grow_rows(ehd_dev *d, double **p, int64_t *cap, int64_t count) {
  if (count <= *cap)
    return EH_OK;
  if (*p)
    HIPCHK(d, hipFree(*p));
  *p = NULL;
  *cap = 0;
  HIPCHK(d, hipMalloc((void **)p, sizeof(double) * (size_t)count));
  *cap = count;
  return EH_OK;
}

#define ROW_GRID(n) dim3((unsigned)(((n) + 255) / 256))

void ehd_set_stage_rows(ehd_dev *d, int64_t rows) { d->stage_rows = rows; }

int64_t ehd_stage_rows(const ehd_dev *d, int32_t w) {
  return d->stage_rows > 0 ? d->stage_rows : EHD_STAGE_BYTES / (int64_t)(sizeof(double) * (size_t)(w + 1));
}

int ehd_put_rows(ehd_dev *d, const double *rows, int64_t first, int64_t m, int32_t w, int cull, double Po) {
  d->rows_kept = 0;
  if (first < 0 || m <= 0 || first + m > d->n)
    return EH_ERR_INVALID;
  HIPCHK(d, hipSetDevice(d->device));
  int rc = grow_rows(d, &d->rows, &d->rows_cap, m * (w + 1)); /* and the loss records behind them */
  if (rc)
    return rc;
  HIPCHK(d, hipMemcpyAsync(d->rows, rows, sizeof(double) * (size_t)(m * w), hipMemcpyHostToDevice, d->stream));
  hipLaunchKernelGGL(rows_in, ROW_GRID(m), dim3(256), 0, d->stream, d->rows, first, m, w, cull, Po, state_of(d), d->ids);
  HIPCHK(d, hipGetLastError());
  d->rows_w = w;
  d->rows_kept = m == d->n;
  return EH_OK;
}

static int put_order(ehd_dev *d, const int32_t *order, int64_t n) {
  if (n > d->order_cap) {
    if (d->order)
      HIPCHK(d, hipFree(d->order));
    d->order = NULL;
    d->order_cap = 0;
    HIPCHK(d, hipMalloc((void **)&d->order, sizeof(int32_t) * (size_t)n));
    d->order_cap = n;
  }
  HIPCHK(d, hipMemcpyAsync(d->order, order, sizeof(int32_t) * (size_t)n, hipMemcpyHostToDevice, d->stream));
  return EH_OK;
}

int ehd_get_rows(ehd_dev *d, double *out, int64_t first, int64_t m, const int32_t *order) {
  if (first < 0 || m <= 0 || first + m > d->n)
    return EH_ERR_INVALID;
  HIPCHK(d, hipSetDevice(d->device));
  int rc = grow_rows(d, &d->rows2, &d->rows2_cap, 8 * m);
  if (!rc && order)
    rc = put_order(d, order, m);
  if (rc)
    return rc;
  hipLaunchKernelGGL(rows_out, ROW_GRID(m), dim3(256), 0, d->stream, d->rows2, state_of(d), d->ids, first, m,
                     order ? d->order : (const int32_t *)NULL);
  HIPCHK(d, hipGetLastError());
  HIPCHK(d, hipMemcpyAsync(out, d->rows2, sizeof(double) * 8 * (size_t)m, hipMemcpyDeviceToHost, d->stream));
  HIPCHK(d, hipStreamSynchronize(d->stream));
  return EH_OK;
}

int ehd_rows_kept(const ehd_dev *d) { return d->rows_kept; }

int ehd_rows_back(ehd_dev *d) {
  HIPCHK(d, hipSetDevice(d->device));
  hipLaunchKernelGGL(rows_back, ROW_GRID(d->n), dim3(256), 0, d->stream, d->rows, d->rows_w, state_of(d));
  HIPCHK(d, hipGetLastError());
  return EH_OK;
}

int ehd_fetch_rows(ehd_dev *d, double *out, const int32_t *order) {
  const int64_t n = d->n, w = d->rows_w;
  const double *src = d->rows;
  HIPCHK(d, hipSetDevice(d->device));
  if (order) {
    int rc = grow_rows(d, &d->rows2, &d->rows2_cap, n * w);
    if (!rc)
      rc = put_order(d, order, n);
    if (rc)
      return rc;
    hipLaunchKernelGGL(rows_gather, ROW_GRID(n * w), dim3(256), 0, d->stream, d->rows, d->rows2, n, (int32_t)w,
                       d->order);
    HIPCHK(d, hipGetLastError());
    src = d->rows2;
  }
  HIPCHK(d, hipMemcpyAsync(out, src, sizeof(double) * (size_t)(n * w), hipMemcpyDeviceToHost, d->stream));
  HIPCHK(d, hipStreamSynchronize(d->stream));
  return EH_OK;
}

int ehd_fetch_small(ehd_dev *d, const double **rows, const int32_t **loss_pass, const int32_t **loss_code) {
  const size_t b = sizeof(double) * (size_t)(d->n * (d->rows_w + 1));
  *rows = NULL;
  if (b > EHD_PIN_BYTES)
    return EH_OK;
  HIPCHK(d, hipSetDevice(d->device));
  if (!d->pin)
    HIPCHK(d, hipHostMalloc(&d->pin, EHD_PIN_BYTES, hipHostMallocDefault));
  HIPCHK(d, hipMemcpyAsync(d->pin, d->rows, b, hipMemcpyDeviceToHost, d->stream));
  HIPCHK(d, hipStreamSynchronize(d->stream));
  *rows = (const double *)d->pin;
  *loss_pass = (const int32_t *)(*rows + d->n * d->rows_w);
  *loss_code = *loss_pass + d->n;
  return EH_OK;
}

int ehd_fiducial_times(ehd_dev *d, double Po, double ahead, double *t) {
  HIPCHK(d, hipSetDevice(d->device));
  const int64_t most = ehd_stage_rows(d, 0);
  for (int64_t first = 0; first < d->n; first += most) {
    const int64_t m = d->n - first < most ? d->n - first : most;
    int rc = grow_rows(d, &d->rows2, &d->rows2_cap, m);
    if (rc)
      return rc;
    hipLaunchKernelGGL(fiducial_times, ROW_GRID(m), dim3(256), 0, d->stream, state_of(d), first, m, Po, ahead, d->rows2);
    HIPCHK(d, hipGetLastError());
    HIPCHK(d, hipMemcpyAsync(t + first, d->rows2, sizeof(double) * (size_t)m, hipMemcpyDeviceToHost, d->stream));
  }
  HIPCHK(d, hipStreamSynchronize(d->stream));
  return EH_OK;
}

int ehd_effort(ehd_dev *d, int64_t pass0, int64_t end, int64_t *effort, int64_t *left) {
  unsigned long long h[2];
  HIPCHK(d, hipSetDevice(d->device));
  const int64_t g = (d->n + 255) / 256;
  hipLaunchKernelGGL(clear_counters, dim3(1), dim3(64), 0, d->stream, d->counter);
  hipLaunchKernelGGL(effort_sum, dim3((unsigned)(g < 256 ? g : 256)), dim3(256), 0, d->stream, d->loss_pass, d->n,
                     pass0, end, d->counter);
  HIPCHK(d, hipGetLastError());
  HIPCHK(d, hipMemcpyAsync(h, d->counter, sizeof h, hipMemcpyDeviceToHost, d->stream));
  HIPCHK(d, hipStreamSynchronize(d->stream));
  *effort = (int64_t)h[0];
  *left = (int64_t)h[1];
  return EH_OK;
}

int ehd_put_ops(ehd_dev *d, const eh_op *ops, int32_t nops) {
  /* one record more than there are: the batch kernel reads the header of a
   * variant's first record before it knows that the variant has none */
  const int64_t room = (int64_t)nops + 1;
  HIPCHK(d, hipSetDevice(d->device));
  if (room > d->ops_cap) {
    if (d->ops)
      HIPCHK(d, hipFree(d->ops));
    d->ops = NULL;
    d->ops_cap = 0;
    HIPCHK(d, hipMalloc((void **)&d->ops, sizeof(eh_op) * (size_t)room));
    d->ops_cap = room;
  }
  if (nops > 0)
    HIPCHK(d, hipMemcpyAsync(d->ops, ops, sizeof(eh_op) * nops, hipMemcpyHostToDevice, d->stream));
  HIPCHK(d, hipStreamSynchronize(d->stream));
  d->nops = nops;
  return EH_OK;
}

static size_t up256(size_t b) { return (b + 255) / 256 * 256; }

/* folds the host copy into runs and uploads bodies, runs and positions, laid
 * out in pinned memory, as one copy that nothing waits for (a single-element
 * call spent three copies and a wait here) */
static int upload_program(ehd_dev *d) {
  const int32_t n = d->nflat;
  const size_t m = (size_t)(n > 0 ? n : 1);
  eh_run *runs = (eh_run *)malloc(sizeof(eh_run) * m);
  int32_t *body = (int32_t *)malloc(sizeof(int32_t) * m);
  int32_t nb = 0, nr = -1;
  int rc = EH_OK;
  if (runs && body)
    nr = eh_fold_runs(d->host_prog, n, EH_RUN_MAX_LEN, runs, body, &nb);
  if (nr < 0) {
    rc = EH_ERR_NOMEM;
    snprintf(d->msg, sizeof d->msg, "out of host memory folding the program");
  }
  const size_t o_runs = up256(sizeof(eh_op) * (size_t)nb), o_z = o_runs + up256(sizeof(eh_run) * (size_t)(nr > 0 ? nr : 0)),
               bytes = o_z + sizeof(double) * 2 * m;
  hipError_t e = hipSuccess;
  if (!rc)
    e = hipEventSynchronize(d->pev); /* the last copy has left pstage */
  if (!rc && !e && bytes > d->pbuf_cap) {
    /* kernels in flight may still read the old buffer */
    e = hipStreamSynchronize(d->stream);
    if (!e && d->pbuf)
      e = hipFree(d->pbuf);
    if (!e && d->pstage)
      e = hipHostFree(d->pstage);
    if (!e) {
      d->pbuf = d->pstage = NULL;
      d->pbuf_cap = 0;
      e = hipMalloc(&d->pbuf, bytes);
    }
    if (!e)
      e = hipHostMalloc(&d->pstage, bytes, hipHostMallocDefault);
    if (!e)
      d->pbuf_cap = bytes;
  }
  if (!rc && !e) {
    char *h = (char *)d->pstage, *g = (char *)d->pbuf;
    d->tops = (eh_op *)g;
    d->runs = (eh_run *)(g + o_runs);
    d->zpos = (double *)(g + o_z);
    double *zpos = (double *)(h + o_z);
    for (int32_t j = 0; j < nb; j++)
      memcpy(h + sizeof(eh_op) * (size_t)j, &d->host_prog[body[j]], sizeof(eh_op));
    memcpy(h + o_runs, runs, sizeof(eh_run) * (size_t)nr);
    for (int32_t f = 0; f < n; f++) {
      zpos[2 * f] = d->host_prog[f].z_start;
      zpos[2 * f + 1] = d->host_prog[f].z_end;
    }
    e = hipMemcpyAsync(d->pbuf, d->pstage, bytes, hipMemcpyHostToDevice, d->stream);
    if (!e)
      e = hipEventRecord(d->pev, d->stream);
    if (e) /* pev cannot tell when pstage is free again */
      (void)hipStreamSynchronize(d->stream);
  }
  if (!rc && e)
    rc = hip_fail(d, e, "uploading the tracking program");
  free(runs);
  free(body);
  if (rc) {
    d->nruns = d->ntops = 0;
    d->nflat = 0;
    return rc;
  }
  d->nruns = nr;
  d->ntops = nb;
  return EH_OK;
}

int ehd_put_program(ehd_dev *d, const eh_op *ops, int32_t nops) {
  if (nops < 0 || (nops > 0 && !ops))
    return EH_ERR_INVALID;
  HIPCHK(d, hipSetDevice(d->device));
  if (nops > d->host_prog_cap) {
    eh_op *h = (eh_op *)realloc(d->host_prog, sizeof(eh_op) * (size_t)nops);
    if (!h)
      return EH_ERR_NOMEM;
    d->host_prog = h;
    d->host_prog_cap = nops;
  }
  if (nops > 0)
    memcpy(d->host_prog, ops, sizeof(eh_op) * (size_t)nops);
  for (int32_t f = 0; f < nops; f++)
    eh_op_finish(&d->host_prog[f]);
  d->nflat = nops;
  return upload_program(d);
}

int ehd_patch_op(ehd_dev *d, int32_t index, const eh_op *op) {
  if (index < 0 || index >= d->nflat)
    return EH_ERR_INVALID;
  HIPCHK(d, hipSetDevice(d->device));
  d->host_prog[index] = *op;
  eh_op_finish(&d->host_prog[index]);
  return upload_program(d);
}

int32_t ehd_program_runs(const ehd_dev *d) { return d->nruns; }

/* 64, 128, 192 or 256 lanes per workgroup; 0 = chosen per launch */
void ehd_set_block(ehd_dev *d, int32_t block) {
  if (block == 0 || (block >= 64 && block <= 256 && block % 64 == 0))
    d->block = block;
}

static int track_launch(ehd_dev *d, int64_t pass0, int32_t npasses, int32_t op_first, int32_t op_last, int timed) {
  if (npasses <= 0 || d->n == 0)
    return EH_OK;
  if (op_first < 0 || op_last > d->nflat || op_first > d->nflat || (npasses == 1 && op_first > op_last))
    return EH_ERR_INVALID;
  HIPCHK(d, hipSetDevice(d->device));
  eh_state st;
  st.x = d->coord[0];
  st.xp = d->coord[1];
  st.y = d->coord[2];
  st.yp = d->coord[3];
  st.s = d->coord[4];
  st.dp = d->coord[5];
  st.loss_pass = d->loss_pass;
  st.loss_code = d->loss_code;
  st.n = d->n;
  int block = d->block;
  if (block == 0) {
    /* 256 lanes per workgroup, unless the particles would fill at most one
     * such workgroup per CU: then 64, so the waves spread over all CUs
     * instead of sharing a few (10^4 particles: 157 CUs busy instead of 40,
     * 6 % faster on the FODO ring) */
    if (!d->num_cu) {
      int cu = 0;
      HIPCHK(d, hipDeviceGetAttribute(&cu, hipDeviceAttributeMultiprocessorCount, d->device));
      d->num_cu = cu > 0 ? cu : 256;
    }
    block = d->n <= (int64_t)d->num_cu * 256 ? 64 : 256;
  }
  const int64_t grid = (d->n + block - 1) / block;
  if (timed)
    HIPCHK(d, hipEventRecord(d->ev0, d->stream));
  hipLaunchKernelGGL(eh_track_kernel, dim3((unsigned)grid), dim3(block), 0, d->stream, st, d->tops, d->runs, d->nruns,
                     d->zpos, pass0, npasses, op_first, op_last, d->nflat);
  HIPCHK(d, hipGetLastError());
  if (!timed)
    return EH_OK;
  HIPCHK(d, hipEventRecord(d->ev1, d->stream));
  HIPCHK(d, hipEventSynchronize(d->ev1));
  float ms = 0;
  HIPCHK(d, hipEventElapsedTime(&ms, d->ev0, d->ev1));
  d->track_ms += ms;
  d->track_launches += 1;
  return EH_OK;
}

int ehd_track(ehd_dev *d, int64_t pass0, int32_t npasses, int32_t op_first, int32_t op_last) {
  return track_launch(d, pass0, npasses, op_first, op_last, 1);
}

int ehd_track_single(ehd_dev *d, int64_t pass) { return track_launch(d, pass, 1, 0, 1, 0); }

/* do_match_energy's re-expression of delta against the new central
 * momentum, delta = dp + delta dr, on the particles still in the beam
 * (do_tracking.c:3408-3414) */
__global__ void eh_rescale_dp_kernel(double *dp_, const int32_t *loss_pass, int64_t n, double dp, double dr) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n && loss_pass[i] < 0)
    dp_[i] = dp + dp_[i] * dr;
}

int ehd_rescale_dp(ehd_dev *d, double dp, double dr) {
  if (d->n == 0)
    return EH_OK;
  HIPCHK(d, hipSetDevice(d->device));
  const int64_t grid = (d->n + 255) / 256;
  hipLaunchKernelGGL(eh_rescale_dp_kernel, dim3((unsigned)grid), dim3(256), 0, d->stream, d->coord[5], d->loss_pass,
                     d->n, dp, dr);
  HIPCHK(d, hipGetLastError());
  HIPCHK(d, hipStreamSynchronize(d->stream));
  return EH_OK;
}

__global__ void eh_count_alive_kernel(const int32_t *loss_pass, int64_t n, unsigned long long *out) {
  int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  int alive = (i < n && loss_pass[i] < 0) ? 1 : 0;
  unsigned long long b = __ballot(alive);
  if ((threadIdx.x & 63) == 0 && b)
    atomicAdd(out, (unsigned long long)__popcll(b));
}

int ehd_count_alive(ehd_dev *d, int64_t *n_alive) {
  HIPCHK(d, hipSetDevice(d->device));
  unsigned long long h = 0;
  HIPCHK(d, hipMemcpyAsync(d->counter, &h, sizeof(h), hipMemcpyHostToDevice, d->stream));
  if (d->n > 0) {
    int64_t grid = (d->n + 255) / 256;
    hipLaunchKernelGGL(eh_count_alive_kernel, dim3((unsigned)grid), dim3(256), 0, d->stream, d->loss_pass, d->n,
                       d->counter);
    HIPCHK(d, hipGetLastError());
  }
  HIPCHK(d, hipMemcpyAsync(&h, d->counter, sizeof(h), hipMemcpyDeviceToHost, d->stream));
  HIPCHK(d, hipStreamSynchronize(d->stream));
  *n_alive = (int64_t)h;
  return EH_OK;
}

int ehd_sync(ehd_dev *d) {
  HIPCHK(d, hipSetDevice(d->device));
  HIPCHK(d, hipStreamSynchronize(d->stream));
  return EH_OK;
}

void ehd_timing_reset(ehd_dev *d) {
  d->track_ms = 0;
  d->track_launches = 0;
  d->coll_ms = 0;
  d->coll_launches = 0;
}

int ehd_timing(ehd_dev *d, int64_t *launches, double *ms) {
  *launches = d->track_launches;
  *ms = d->track_ms;
  return EH_OK;
}

const char *ehd_message(const ehd_dev *d) { return d ? d->msg : ""; }

int ehd_batch_setup(ehd_dev *d, const eh_vdesc *v, int32_t nvar, const eh_chunk *chunks, int32_t nchunks) {
  HIPCHK(d, hipSetDevice(d->device));
  if (nvar > d->var_cap) {
    if (d->vdesc)
      HIPCHK(d, hipFree(d->vdesc));
    d->vdesc = NULL;
    HIPCHK(d, hipMalloc((void **)&d->vdesc, sizeof(eh_vdesc) * nvar));
    d->var_cap = nvar;
  }
  if (nchunks > d->chunk_cap) {
    if (d->chunks)
      HIPCHK(d, hipFree(d->chunks));
    d->chunks = NULL;
    HIPCHK(d, hipMalloc((void **)&d->chunks, sizeof(eh_chunk) * nchunks));
    d->chunk_cap = nchunks;
  }
  if (!d->queue)
    HIPCHK(d, hipMalloc((void **)&d->queue, 256));
  if (!d->num_cu) {
    int cu = 0;
    HIPCHK(d, hipDeviceGetAttribute(&cu, hipDeviceAttributeMultiprocessorCount, d->device));
    d->num_cu = cu > 0 ? cu : 256;
  }
  d->dev_nchunks = (int32_t *)d->queue + 32;
  HIPCHK(d, hipMemcpyAsync(d->vdesc, v, sizeof(eh_vdesc) * nvar, hipMemcpyHostToDevice, d->stream));
  HIPCHK(d, hipMemcpyAsync(d->chunks, chunks, sizeof(eh_chunk) * nchunks, hipMemcpyHostToDevice, d->stream));
  HIPCHK(d, hipMemcpyAsync(d->dev_nchunks, &nchunks, sizeof(int32_t), hipMemcpyHostToDevice, d->stream));
  HIPCHK(d, hipStreamSynchronize(d->stream));
  d->nvar = nvar;
  d->nchunks = nchunks;
  d->use_perm = 0;
  return EH_OK;
}

int ehd_batch_compact(ehd_dev *d, const int32_t *perm, int64_t nperm, const eh_chunk *chunks, int32_t nchunks) {
  HIPCHK(d, hipSetDevice(d->device));
  if (nperm > d->perm_cap) {
    if (d->perm)
      HIPCHK(d, hipFree(d->perm));
    d->perm = NULL;
    d->perm_cap = 0;
    HIPCHK(d, hipMalloc((void **)&d->perm, sizeof(int32_t) * (nperm > 0 ? nperm : 1)));
    d->perm_cap = nperm > 0 ? nperm : 1;
  }
  if (nchunks > d->chunk_cap)
    return EH_ERR_INVALID; /* compaction never adds chunks */
  if (nperm > 0)
    HIPCHK(d, hipMemcpyAsync(d->perm, perm, sizeof(int32_t) * nperm, hipMemcpyHostToDevice, d->stream));
  if (nchunks > 0)
    HIPCHK(d, hipMemcpyAsync(d->chunks, chunks, sizeof(eh_chunk) * nchunks, hipMemcpyHostToDevice, d->stream));
  HIPCHK(d, hipMemcpyAsync(d->dev_nchunks, &nchunks, sizeof(int32_t), hipMemcpyHostToDevice, d->stream));
  HIPCHK(d, hipStreamSynchronize(d->stream));
  d->nchunks = nchunks;
  d->use_perm = 1;
  return EH_OK;
}

/* ---- the work queue rebuilt on the device ----
 * The surviving particles, in index order (so grouped by variant, whose
 * particle ranges are contiguous), are listed in perm, and each variant's
 * list is cut into chunks of csize; the count lands in dev_nchunks.  Six
 * small kernels, no host round trip and no memset, so the sequence can sit
 * between the tracking launches of one captured graph. */
#define CT 1024 /* particles per tile of the compaction */

/* alive particles per tile */
__global__ void __launch_bounds__(256) compact_count(const int32_t *__restrict__ lp, int64_t n, int32_t *tile_sum) {
  __shared__ int32_t s[4];
  const int64_t base = (int64_t)blockIdx.x * CT;
  int32_t c = 0;
  for (int k = threadIdx.x; k < CT; k += 256) {
    const int64_t i = base + k;
    c += (i < n && lp[i] < 0) ? 1 : 0;
  }
  for (int off = 32; off > 0; off >>= 1)
    c += __shfl_xor(c, off);
  if ((threadIdx.x & 63) == 0)
    s[threadIdx.x >> 6] = c;
  __syncthreads();
  if (threadIdx.x == 0)
    tile_sum[blockIdx.x] = s[0] + s[1] + s[2] + s[3];
}

/* exclusive scan of the tile sums in place (one workgroup); tile_sum[nt] = total */
__global__ void __launch_bounds__(256) compact_scan(int32_t *tile_sum, int32_t nt) {
  __shared__ int32_t s[256];
  __shared__ int32_t carry;
  if (threadIdx.x == 0)
    carry = 0;
  __syncthreads();
  for (int32_t base = 0; base < nt; base += 256) {
    const int32_t i = base + threadIdx.x;
    const int32_t v = i < nt ? tile_sum[i] : 0;
    s[threadIdx.x] = v;
    __syncthreads();
    for (int off = 1; off < 256; off <<= 1) {
      const int32_t t = (int)threadIdx.x >= off ? s[threadIdx.x - off] : 0;
      __syncthreads();
      s[threadIdx.x] += t;
      __syncthreads();
    }
    const int32_t incl = s[threadIdx.x];
    const int32_t c0 = carry;
    if (i < nt)
      tile_sum[i] = c0 + incl - v;
    __syncthreads();
    if (threadIdx.x == 255)
      carry = c0 + incl;
    __syncthreads();
  }
  if (threadIdx.x == 0)
    tile_sum[nt] = carry;
}

/* perm[position] = index of each alive particle, in index order */
__global__ void __launch_bounds__(256) compact_scatter(const int32_t *__restrict__ lp, int64_t n,
                                                       const int32_t *__restrict__ tile_sum, int32_t *perm) {
  __shared__ int32_t wsum[4];
  const int64_t base = (int64_t)blockIdx.x * CT;
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  int32_t off = tile_sum[blockIdx.x];
  for (int k0 = 0; k0 < CT; k0 += 256) {
    const int64_t i = base + k0 + threadIdx.x;
    const bool a = i < n && lp[i] < 0;
    const unsigned long long m = __ballot(a);
    const int before = __popcll(m & ((1ULL << lane) - 1ULL));
    if (lane == 0)
      wsum[w] = __popcll(m);
    __syncthreads();
    int32_t wbase = 0;
    for (int q = 0; q < w; q++)
      wbase += wsum[q];
    const int32_t tot = wsum[0] + wsum[1] + wsum[2] + wsum[3];
    if (a)
      perm[off + wbase + before] = (int32_t)i;
    __syncthreads();
    off += tot;
  }
}

/* alive particles with index below k, by the workgroup: the tile's prefix
 * plus a count over the start of the tile */
DEV int32_t alive_below(const int32_t *__restrict__ lp, int64_t n, const int32_t *__restrict__ tile_sum, int64_t k,
                        int32_t *red) {
  const int64_t tile = k / CT, base = tile * CT;
  int32_t c = 0;
  for (int64_t i = base + threadIdx.x; i < k && i < n; i += 256)
    c += lp[i] < 0 ? 1 : 0;
  for (int off = 32; off > 0; off >>= 1)
    c += __shfl_xor(c, off);
  __syncthreads();
  if ((threadIdx.x & 63) == 0)
    red[threadIdx.x >> 6] = c;
  __syncthreads();
  return tile_sum[tile] + red[0] + red[1] + red[2] + red[3];
}

/* per variant (one workgroup each): vinfo[4v..] = start in perm, alive, chunks */
__global__ void __launch_bounds__(256) compact_variants(const int32_t *__restrict__ lp, int64_t n,
                                                        const int32_t *__restrict__ tile_sum,
                                                        const eh_vdesc *__restrict__ vars, int32_t csize,
                                                        int32_t *vinfo) {
  __shared__ int32_t red[4];
  const eh_vdesc vd = vars[blockIdx.x];
  const int32_t p0 = alive_below(lp, n, tile_sum, vd.first, red);
  const int32_t p1 = alive_below(lp, n, tile_sum, vd.first + vd.n, red);
  if (threadIdx.x == 0) {
    vinfo[4 * blockIdx.x] = p0;
    vinfo[4 * blockIdx.x + 1] = p1 - p0;
    vinfo[4 * blockIdx.x + 2] = (p1 - p0 + csize - 1) / csize;
  }
}

/* first chunk of each variant (exclusive scan, one workgroup) and the count */
__global__ void __launch_bounds__(256) compact_chunk_offsets(int32_t *vinfo, int32_t nvar, int32_t *nchunks_out) {
  __shared__ int32_t s[256];
  __shared__ int32_t carry;
  if (threadIdx.x == 0)
    carry = 0;
  __syncthreads();
  for (int32_t base = 0; base < nvar; base += 256) {
    const int32_t v = base + threadIdx.x;
    const int32_t c = v < nvar ? vinfo[4 * v + 2] : 0;
    s[threadIdx.x] = c;
    __syncthreads();
    for (int off = 1; off < 256; off <<= 1) {
      const int32_t t = (int)threadIdx.x >= off ? s[threadIdx.x - off] : 0;
      __syncthreads();
      s[threadIdx.x] += t;
      __syncthreads();
    }
    const int32_t incl = s[threadIdx.x];
    const int32_t c0 = carry;
    if (v < nvar)
      vinfo[4 * v + 3] = c0 + incl - c;
    __syncthreads();
    if (threadIdx.x == 255)
      carry = c0 + incl;
    __syncthreads();
  }
  if (threadIdx.x == 0)
    *nchunks_out = carry;
}

/* the chunks of each variant (one workgroup each) */
__global__ void __launch_bounds__(256) compact_write_chunks(const int32_t *__restrict__ vinfo, int32_t csize,
                                                            eh_chunk *chunks) {
  const int32_t v = blockIdx.x;
  const int32_t start = vinfo[4 * v], alive = vinfo[4 * v + 1], nch = vinfo[4 * v + 2], c0 = vinfo[4 * v + 3];
  for (int32_t c = threadIdx.x; c < nch; c += 256) {
    eh_chunk ch;
    ch.variant = v;
    ch.first = (int64_t)start + (int64_t)c * csize;
    ch.count = alive - c * csize < csize ? alive - c * csize : csize;
    chunks[c0 + c] = ch;
  }
}

static int compact_ensure(ehd_dev *d) {
  const int64_t nt = (d->n + CT - 1) / CT;
  if (d->perm_cap < d->n) {
    if (d->perm)
      HIPCHK(d, hipFree(d->perm));
    d->perm = NULL;
    d->perm_cap = 0;
    HIPCHK(d, hipMalloc((void **)&d->perm, sizeof(int32_t) * (d->n > 0 ? d->n : 1)));
    d->perm_cap = d->n > 0 ? d->n : 1;
  }
  if (d->tile_cap < nt + 1 || d->vinfo_cap < d->nvar) {
    if (d->tile_sum)
      HIPCHK(d, hipFree(d->tile_sum));
    d->tile_sum = NULL;
    d->tile_cap = d->vinfo_cap = 0;
    HIPCHK(d, hipMalloc((void **)&d->tile_sum, sizeof(int32_t) * (nt + 1 + 4 * (int64_t)d->nvar)));
    d->tile_cap = nt + 1;
    d->vinfo_cap = d->nvar;
  }
  return EH_OK;
}

static void compact_launch(ehd_dev *d, int32_t csize) {
  const int64_t nt = (d->n + CT - 1) / CT;
  int32_t *vinfo = d->tile_sum + d->tile_cap;
  hipLaunchKernelGGL(compact_count, dim3((unsigned)nt), dim3(256), 0, d->stream, d->loss_pass, d->n, d->tile_sum);
  hipLaunchKernelGGL(compact_scan, dim3(1), dim3(256), 0, d->stream, d->tile_sum, (int32_t)nt);
  hipLaunchKernelGGL(compact_scatter, dim3((unsigned)nt), dim3(256), 0, d->stream, d->loss_pass, d->n, d->tile_sum,
                     d->perm);
  hipLaunchKernelGGL(compact_variants, dim3((unsigned)d->nvar), dim3(256), 0, d->stream, d->loss_pass, d->n,
                     d->tile_sum, d->vdesc, csize, vinfo);
  hipLaunchKernelGGL(compact_chunk_offsets, dim3(1), dim3(256), 0, d->stream, vinfo, d->nvar, d->dev_nchunks);
  hipLaunchKernelGGL(compact_write_chunks, dim3((unsigned)d->nvar), dim3(256), 0, d->stream, vinfo, csize, d->chunks);
}

static int batch_launch(ehd_dev *d, eh_state st, int64_t pass0, int32_t npasses, int32_t ppl, int32_t block,
                        int grid) {
  hipLaunchKernelGGL(eh_queue_reset, dim3(1), dim3(1), 0, d->stream, d->queue);
  const int32_t *perm = d->use_perm ? d->perm : (const int32_t *)NULL;
  if (ppl == 2)
    hipLaunchKernelGGL(eh_batch_kernel<2>, dim3(grid), dim3(block), 0, d->stream, st, d->ops, d->vdesc, d->chunks,
                       d->dev_nchunks, perm, pass0, npasses, d->queue);
  else
    hipLaunchKernelGGL(eh_batch_kernel<1>, dim3(grid), dim3(block), 0, d->stream, st, d->ops, d->vdesc, d->chunks,
                       d->dev_nchunks, perm, pass0, npasses, d->queue);
  return EH_OK;
}

int ehd_batch_track(ehd_dev *d, int64_t pass0, int32_t npasses, int32_t passes_per_launch, int32_t ppl,
                    int32_t block, int32_t use_graph, int32_t device_compact, double *ms_out, int64_t *launches_out) {
  if (npasses <= 0 || d->nchunks <= 0) {
    *ms_out = 0;
    *launches_out = 0;
    return EH_OK;
  }
  if ((ppl != 1 && ppl != 2) || block < 64 || block > 256 || block % 64 || passes_per_launch < 1)
    return EH_ERR_INVALID;
  HIPCHK(d, hipSetDevice(d->device));
  if (device_compact) {
    int rc = compact_ensure(d);
    if (rc)
      return rc;
  }
  eh_state st;
  st.x = d->coord[0];
  st.xp = d->coord[1];
  st.y = d->coord[2];
  st.yp = d->coord[3];
  st.s = d->coord[4];
  st.dp = d->coord[5];
  st.loss_pass = d->loss_pass;
  st.loss_code = d->loss_code;
  st.n = d->n;
  int per_cu = 0;
  if (ppl == 2)
    HIPCHK(d, hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, eh_batch_kernel<2>, block, 0));
  else
    HIPCHK(d, hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, eh_batch_kernel<1>, block, 0));
  if (per_cu < 1)
    per_cu = 1;
  int grid = d->num_cu * per_cu;
  if (grid > d->nchunks)
    grid = d->nchunks;
  int64_t nl = 0;
  hipGraph_t graph = NULL;
  hipGraphExec_t exec = NULL;
  if (use_graph)
    HIPCHK(d, hipStreamBeginCapture(d->stream, hipStreamCaptureModeThreadLocal));
  else
    HIPCHK(d, hipEventRecord(d->ev0, d->stream));
  if (!device_compact) {
    for (int32_t done = 0; done < npasses; done += passes_per_launch) {
      int32_t k = npasses - done < passes_per_launch ? npasses - done : passes_per_launch;
      batch_launch(d, st, pass0 + done, k, ppl, block, grid);
      nl++;
    }
  } else {
    /* launches of 1, 2, 4 ... passes up to passes_per_launch, the queue
     * rebuilt from the survivors on the device after each */
    int32_t done = 0, step = 1;
    while (done < npasses) {
      int32_t k = step < passes_per_launch ? step : passes_per_launch;
      if (k > npasses - done)
        k = npasses - done;
      batch_launch(d, st, pass0 + done, k, ppl, block, grid);
      nl++;
      done += k;
      if (step < passes_per_launch)
        step *= 2;
      if (done < npasses) {
        compact_launch(d, block * ppl);
        d->use_perm = 1;
      }
    }
  }
  if (use_graph) {
    HIPCHK(d, hipStreamEndCapture(d->stream, &graph));
    HIPCHK(d, hipGraphInstantiate(&exec, graph, NULL, NULL, 0));
    HIPCHK(d, hipEventRecord(d->ev0, d->stream));
    HIPCHK(d, hipGraphLaunch(exec, d->stream));
  }
  HIPCHK(d, hipGetLastError());
  HIPCHK(d, hipEventRecord(d->ev1, d->stream));
  HIPCHK(d, hipEventSynchronize(d->ev1));
  float ms = 0;
  HIPCHK(d, hipEventElapsedTime(&ms, d->ev0, d->ev1));
  if (exec)
    HIPCHK(d, hipGraphExecDestroy(exec));
  if (graph)
    HIPCHK(d, hipGraphDestroy(graph));
  d->track_ms += ms;
  d->track_launches += nl;
  *ms_out = ms;
  *launches_out = nl;
  return EH_OK;
}

/* copy of the particle state on the device (autotuning trials restore it) */
int ehd_state_snapshot(ehd_dev *d, int restore) {
  HIPCHK(d, hipSetDevice(d->device));
  if (!restore && d->n > d->snap_cap) {
    for (int k = 0; k < 6; k++) {
      if (d->snap[k])
        HIPCHK(d, hipFree(d->snap[k]));
      d->snap[k] = NULL;
    }
    if (d->snap_lp)
      HIPCHK(d, hipFree(d->snap_lp));
    if (d->snap_lc)
      HIPCHK(d, hipFree(d->snap_lc));
    d->snap_lp = d->snap_lc = NULL;
    for (int k = 0; k < 6; k++)
      HIPCHK(d, hipMalloc((void **)&d->snap[k], sizeof(double) * d->n));
    HIPCHK(d, hipMalloc((void **)&d->snap_lp, sizeof(int32_t) * d->n));
    HIPCHK(d, hipMalloc((void **)&d->snap_lc, sizeof(int32_t) * d->n));
    d->snap_cap = d->n;
  }
  if (restore && d->snap_cap < d->n)
    return EH_ERR_STATE;
  for (int k = 0; k < 6; k++)
    HIPCHK(d, hipMemcpyAsync(restore ? d->coord[k] : d->snap[k], restore ? d->snap[k] : d->coord[k],
                             sizeof(double) * d->n, hipMemcpyDeviceToDevice, d->stream));
  HIPCHK(d, hipMemcpyAsync(restore ? d->loss_pass : d->snap_lp, restore ? d->snap_lp : d->loss_pass,
                           sizeof(int32_t) * d->n, hipMemcpyDeviceToDevice, d->stream));
  HIPCHK(d, hipMemcpyAsync(restore ? d->loss_code : d->snap_lc, restore ? d->snap_lc : d->loss_code,
                           sizeof(int32_t) * d->n, hipMemcpyDeviceToDevice, d->stream));
  HIPCHK(d, hipStreamSynchronize(d->stream));
  return EH_OK;
}

/* ---- device buffers for tests of the device-pointer entry points ---- */
int ehd_test_buffer(ehd_dev *d, int32_t op, void **ptr, void *host, int64_t bytes) {
  HIPCHK(d, hipSetDevice(d->device));
  switch (op) {
  case 0: /* allocate */
    HIPCHK(d, hipMalloc(ptr, bytes > 0 ? bytes : 8));
    return EH_OK;
  case 1: /* free */
    HIPCHK(d, hipFree(*ptr));
    *ptr = NULL;
    return EH_OK;
  case 2: /* host -> device */
    HIPCHK(d, hipMemcpy(*ptr, host, bytes, hipMemcpyHostToDevice));
    return EH_OK;
  case 3: /* device -> host */
    HIPCHK(d, hipMemcpy(host, *ptr, bytes, hipMemcpyDeviceToHost));
    return EH_OK;
  }
  return EH_ERR_INVALID;
}

/* ---- deterministic-math probe (used by tests to compare with the CPU) ---- */
__global__ void eh_math_probe_kernel(int32_t fn, const double *in, const double *in2, double *out, int64_t n) {
  int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n)
    return;
  double v = in[i], r;
  switch (fn) {
  case 0:
    r = em_sin(v);
    break;
  case 1:
    r = em_cos(v);
    break;
  case 2:
    r = em_asin(v);
    break;
  case 3:
    r = em_log(v);
    break;
  case 4:
    r = em_tan(v);
    break;
  case 5:
    r = __builtin_sqrt(v);
    break;
  case 7: /* the unscaled square root the tracking kernels use */
    r = em_sqrt(v);
    break;
  case 8: /* the shared-reciprocal quotient the tracking kernels use */
    r = em_div(v, in2[i], em_recip(in2[i]), em_recip_ok(in2[i]));
    break;
  case 9: /* the same quotient from the rounded reciprocal (bend radii) */
    r = em_div(v, in2[i], 1.0 / in2[i], em_recip_ok(in2[i]));
    break;
  case 10: /* the aperture's integer power, exponent in in2 (0..EH_MAX_AP_EXPONENT) */
    r = ap_ipow(v, (int)in2[i]);
    break;
  case 11: /* the bend's and multipoles' square root with its reciprocal: sqrt(in2) */
    r = em_sqrt_recip_mid(in2[i], &v);
    break;
  case 12: { /* in / sqrt(in2) from that pair */
    double y, g = em_sqrt_recip_mid(in2[i], &y);
    r = em_div_pos(v, g, y);
    break;
  }
  case 13: { /* in / cos(in2), |in2| < 2^-5 */
    const double z = in2[i] * in2[i], c = em_cos_small(in2[i], z);
    const em_small_k k = em_small_coefs();
    r = em_div_pos(v, c, em_recip_cos_small(c, z, &k));
    break;
  }
  default:
    r = v / in2[i];
    break;
  }
  out[i] = r;
}

int ehd_math_probe(ehd_dev *d, int32_t fn, const double *in, const double *in2, double *out, int64_t n) {
  double *din = NULL, *din2 = NULL, *dout = NULL;
  if (n <= 0)
    return EH_OK;
  HIPCHK(d, hipSetDevice(d->device));
  HIPCHK(d, hipMalloc((void **)&din, sizeof(double) * n));
  HIPCHK(d, hipMalloc((void **)&din2, sizeof(double) * n));
  HIPCHK(d, hipMalloc((void **)&dout, sizeof(double) * n));
  HIPCHK(d, hipMemcpyAsync(din, in, sizeof(double) * n, hipMemcpyHostToDevice, d->stream));
  if (in2)
    HIPCHK(d, hipMemcpyAsync(din2, in2, sizeof(double) * n, hipMemcpyHostToDevice, d->stream));
  else
    HIPCHK(d, hipMemcpyAsync(din2, in, sizeof(double) * n, hipMemcpyHostToDevice, d->stream));
  hipLaunchKernelGGL(eh_math_probe_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, d->stream, fn, din, din2,
                     dout, n);
  HIPCHK(d, hipGetLastError());
  HIPCHK(d, hipMemcpyAsync(out, dout, sizeof(double) * n, hipMemcpyDeviceToHost, d->stream));
  HIPCHK(d, hipStreamSynchronize(d->stream));
  HIPCHK(d, hipFree(din));
  HIPCHK(d, hipFree(din2));
  HIPCHK(d, hipFree(dout));
  return EH_OK;
}

} /* extern "C" */
