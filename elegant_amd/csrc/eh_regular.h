/* eh_regular.h -- the integrators for regular particles.
 *
 * Nearly every particle of every beam is regular: inside the apertures, with
 * slopes of milliradians and a momentum within some percent of the reference.
 * For those the general maps spend most of their instructions on what cannot
 * happen: the range scaling and special cases of IEEE division and square root,
 * the branches of the transcendental functions, the loss bookkeeping.  The
 * integrators here leave all of that out, keep one flag per particle that says
 * it stayed regular, and are thrown away for a particle that did not: the caller
 * runs the general integrator for it from the saved entry state.
 *
 * Every result is the general integrator's, bit for bit.  Sums, products and
 * polynomials are the same operations in the same order.  Quotients and roots
 * are correctly rounded here too, by other means:
 *
 *  - RN(a / b) from y = RN(1 / b): q = RN(a y) is within 1.5 ulp, its residual
 *    is exact in one fma, and RN(q + residual y) is the correctly rounded
 *    quotient (P. Markstein, IBM J. Res. Develop. 34 (1990) 111-119), for normal
 *    quotients away from underflow.  The residual is formed with its sign
 *    reversed, which keeps the sign of a zero numerator over a positive b.
 *  - y = RN(1 / b) from y0 within a few ulps: one Newton step y0 + y0 e with
 *    e = 1 - b y0 exact is 1 / b to 2^-101 before its only rounding.  That decides
 *    the rounding unless b = 2^n (1 - k 2^-53) with a small odd k, where 1 / b lies
 *    only k^2 2^-106 above a midpoint; there y must come out above it (the
 *    quotient of a power of two by 1 - 2^-53 is wrong otherwise), which the two
 *    routines below arrange each in its way.  Elsewhere a y off by 2^-27 of a half
 *    ulp more still gives the correctly rounded quotient, since b^2 is then below
 *    4 by more than that.
 *  - RN(sqrt a) from g within a few ulps: g + (a - g g) h with a - g g exact and
 *    h = 1 / (2 g) to 2^-50 is sqrt a to 2^-101 before its only rounding.
 *
 * What bounds these loops is the number of instructions: a dependent FP64 fma
 * issues every 5 cycles from one wavefront and every 4 from several, so that a
 * launch of few particles gains nothing from independent operations and one of
 * many nothing from latency hiding.  A sub-step of a gradient bend takes 144
 * instructions here, 120 of them FP64, against 270 vector and 215 scalar ones in the
 * general integrator, whose branches also keep the compiler from holding the
 * polynomial constants in scalar registers.  Kernel times with the general
 * integrators alone and now (MI355X, MBA ring, fused, 2 turns): 1e6 particles 283 and
 * 137 ms, 30 401 particles (one wavefront on half of the SIMDs) 48.4 and 15.1 ms; FODO
 * ring, 1e4 particles, 40 turns 27.2 and 9.7 ms.
 *
 * A wavefront runs the general integrator as soon as one of its particles is beyond
 * the limits at an element's entry, and both integrators where one leaves them
 * inside.  On a grid filling the aperture of the MBA ring no particle that is not
 * lost ever does; of slopes of 5 mrad rms nearly every wavefront has one.  Kernel
 * times of short lines of such beams, 2 turns, 4e5 particles: quadrupoles and
 * sextupoles, 5 mrad, 0.58 ms (0.60 with the general integrators alone, 0.70 when
 * the other particles of the wavefront went on here); with bends, 3 mrad, 1.54 (1.51,
 * 1.79); 20 mrad, 1.88 (1.85, 2.47).  1e4 particles, one wavefront alone on its SIMD:
 * 0.19 (0.20, 0.24), 0.55 (0.48, 0.65) and 0.66 (0.61, 0.77).  Looking again at every
 * slice would win back 0.04 of the 0.55 and cost regular beams 1 to 3 %.
 *
 * With SYNCH_RAD the momentum changes at every kick; its reciprocal follows by a
 * Newton step from the last one.  MBA ring with radiation and edges, 5e4
 * particles, one turn: 27.1 and 11.2 ms.
 *
 * The starting values need no hardware estimate (v_rcp_f64 and v_rsq_f64 give 24
 * bits and take the issue time of four fma): a bend's and a multipole's root is
 * of (1 + delta)^2 minus a small square, so the binomial series around
 * 1 / (1 + delta), formed once per element, is accurate to the last bits, and a
 * cosine close to one is its own estimate.  Only IEEE +, -, *, and fma are used,
 * so that the host build of these routines gives the same doubles.
 */
#ifndef EH_REGULAR_H
#define EH_REGULAR_H

/* limits of the regular path: 1 + delta; canonical momenta, about the slopes (a
 * bend's QX swings by its sub-step angles on the design orbit already); and the
 * smallest non-zero momentum, whose quotients are far from underflow.  With them
 * |sin phi| < 2^-4 and the series argument of eh_reg_root is < 2^-11 (< 2^-8 with
 * WIDE, where QX takes part), asserted below.  Comparisons are or-ed into one mask
 * (keeping running maxima and minima instead takes fewer scalar instructions, but
 * v_max_f64 and v_min_f64 cost more than v_cmp: 1e6 particles 4 % slower). */
#define EH_REG_B1_MIN 0.875
#define EH_REG_B1_MAX 1.25
#define EH_REG_QMAX 0.0117
#define EH_REG_QXMAX 0.05
#define EH_REG_QMIN 0x1p-340
/* a bend's angles, where eh_sincos is its short series, and the relative change of
 * 1 + delta at a radiation kick */
#define EH_REG_ANGLE 0x1p-4
#define EH_REG_DLOSS 0x1p-18
/* what the host leaves for the slopes of a small beam where the design orbit itself
 * comes near a limit */
#define EH_REG_OWN 1e-3
static_assert(2 * EH_REG_QMAX * EH_REG_QMAX / (EH_REG_B1_MIN * EH_REG_B1_MIN) < 0x1p-11, "series of eh_reg_root");
static_assert((EH_REG_QXMAX * EH_REG_QXMAX + EH_REG_QMAX * EH_REG_QMAX) / (EH_REG_B1_MIN * EH_REG_B1_MIN) < 0x1p-8,
              "series of eh_reg_root<true>");
/* f >= 0.98 (1 + delta) by the above */
static_assert(EH_REG_QXMAX / (0.98 * EH_REG_B1_MIN) < EH_REG_ANGLE, "short series of asin");
/* dense 5 x 5 field block: the terms a gradient alone leaves, (i, j) = (0, 0..4),
 * (1, 0), (1, 2), (1, 3), (2, 2) */
#define EH_LIVE_GRADIENT 0x9bfu

/* RN(a / b) with y = RN(1 / b), b > 0 */
EH_HD double eh_reg_div(double a, double b, double y) {
  const double q = a * y;
  return eh_fma(-eh_fma(q, b, -a), y, q);
}

/* f = RN(sqrt a) and y = RN(1 / f) for a = b1^2 (1 - w) up to its rounding, from
 * rh = RN(1 / b1) and w < 2^-11: the binomial series of (1 - w)^-1/2 to w^4 (the
 * next term is below 2^-56); WIDE: w < 2^-8, to w^6 */
template <bool WIDE = false>
EH_HD void eh_reg_root(double a, double w, double rh, double &f, double &y) {
  double t = 0x1.18p-2;
  if constexpr (WIDE) {
    t = eh_fma(w, 0x1.cep-3, 0x1.f8p-3);
    t = eh_fma(w, t, 0x1.18p-2);
  }
  t = eh_fma(w, t, 0x1.4p-2);
  t = eh_fma(w, t, 0x1.8p-2);
  t = eh_fma(w, t, 0.5);
  const double y0 = eh_fma(rh * w, t, rh);
  const double g = a * y0;
  f = eh_fma(eh_fma(-g, g, a), 0.5 * y0, g);
  /* 2^-80: far below the last bit, far above the 2^-101 by which the step falls
   * short, so that 1 / f just above a midpoint (see the top) rounds up */
  y = eh_fma(eh_fma(-f, y0, 1.0) + 0x1p-80, y0, y0);
}

/* RN(1 / c) for a cosine c = 1 - u, 0 <= u < 2^-9: 2 - c is 1 / c to u^2; one
 * step of third order leaves 3 quarters of an ulp, one of second order the
 * correct rounding.  Starting 2^-51 too high makes 1 - 2^-53 come out right: both
 * steps then end above the midpoint, at 1 + 2^-52. */
EH_HD double eh_reg_recip1(double c) {
  const double y0 = 0x1.0000000000001p1 - c;
  const double e = eh_fma(-c, y0, 1.0);
  const double y1 = eh_fma(y0, eh_fma(e, e, e), y0);
  return eh_fma(eh_fma(-c, y1, 1.0), y1, y1);
}

/* rh = RN(1 / b) within 2^-80 for the quotients above, from the reciprocal of a
 * b within 2^-18 relative (a particle's 1 + delta before a radiation kick); false
 * if it is further off */
EH_HD bool eh_reg_next_recip(double b, double &rh) {
  const double e = eh_fma(-b, rh, 1.0);
  const double y1 = eh_fma(rh, eh_fma(e, e, e), rh);
  rh = eh_fma(eh_fma(-b, y1, 1.0) + 0x1p-80, y1, y1);
  return eh_fabs(e) < EH_REG_DLOSS;
}

/* The coefficients of the short series, opaque to the compiler on the GPU so that
 * it keeps them in scalar registers across a bend: known constants it rebuilds at
 * every use, two s_mov each, which a wavefront alone on its SIMD pays in full (30
 * of the 200 instructions of a sub-step). */
struct eh_reg_series {
  double s1, s2, s3, s4, s5, c2, c3, c4, c5, c6, a1, a2, a3, a4;
};

EH_HD double eh_reg_keep(double c) {
#if defined(__HIP_DEVICE_COMPILE__)
  __asm__ volatile("" : "+s"(c));
#endif
  return c;
}

EH_HD eh_reg_series eh_reg_series_load() {
  return {eh_reg_keep(EH_SIN_1),  eh_reg_keep(EH_SIN_2),  eh_reg_keep(EH_SIN_3),  eh_reg_keep(EH_SIN_4),
          eh_reg_keep(EH_SIN_5),  eh_reg_keep(EH_COS_2),  eh_reg_keep(EH_COS_3),  eh_reg_keep(EH_COS_4),
          eh_reg_keep(EH_COS_5),  eh_reg_keep(EH_COS_6),  eh_reg_keep(EH_ASIN_1), eh_reg_keep(EH_ASIN_2),
          eh_reg_keep(EH_ASIN_3), eh_reg_keep(EH_ASIN_4)};
}

/* eh_sin_poly, and eh_cos_poly with the exact products by 1/2 inside fma */
EH_HD double eh_reg_sin(double r, const eh_reg_series &k) {
  const double z = r * r;
  double q = eh_horner(z, k.s5, k.s4);
  q = eh_horner(z, q, k.s3);
  q = eh_horner(z, q, k.s2);
  q = eh_horner(z, q, k.s1);
  return eh_fma(r * z, q, r);
}

EH_HD double eh_reg_cos(double r, const eh_reg_series &k) {
  const double z = r * r;
  double p = eh_horner(z, k.c6, k.c5);
  p = eh_horner(z, p, k.c4);
  p = eh_horner(z, p, k.c3);
  p = eh_horner(z, p, k.c2);
  const double zl = eh_fma(r, r, -z);
  const double w = eh_fma(-0.5, z, 1.0);
  const double t = eh_fma(-0.5, z, 1.0 - w);
  return w + eh_fma(z * z, p, eh_fma(-0.5, zl, t));
}

/* eh_asin below 2^-4: the two short series of eh_asin_small */
EH_HD double eh_reg_asin(double x, const eh_reg_series &k) {
  const double z = x * x;
  double q = k.a4;
  const bool longer = !(eh_fabs(x) < 0x1p-8);
#if defined(__HIP_DEVICE_COMPILE__)
  if (__ballot(longer))
#else
  if (longer)
#endif
  {
    double p = EH_ASIN_7;
    p = eh_horner(z, p, EH_ASIN_6);
    p = eh_horner(z, p, EH_ASIN_5);
    p = eh_horner(z, p, EH_ASIN_4);
    q = longer ? p : q;
  }
  q = eh_horner(z, q, k.a3);
  q = eh_horner(z, q, k.a2);
  q = eh_horner(z, q, k.a1);
  return eh_fma(x * z, q, x);
}

/* the field of a bend that has a gradient and nothing else, from the nine terms
 * of its dense block in the order of eh_csb_fields_dense; 0 + c y is one fma */
struct eh_grad_field {
  double c0, y1, y2, y3, y4, x1, x1y2, x1y3, x2y2;
};

EH_HD eh_grad_field eh_grad_load(const eh_fterm *__restrict__ cx, const eh_fterm *__restrict__ cy) {
  return {cy[0].coef, cx[1].coef, cy[2].coef, cx[3].coef, cy[4].coef, cy[5].coef, cy[7].coef, cx[8].coef, cy[12].coef};
}

EH_HD void eh_grad_eval(const eh_grad_field &c, double x, double y, double &Fx, double &Fy) {
  const double y2 = y * y, y3 = y2 * y, y4 = y3 * y;
  Fx = eh_fma(c.y1, y, 0.0);
  Fy = c.c0 + c.y2 * y2;
  Fx += c.y3 * y3;
  Fy += c.y4 * y4;
  Fy += c.x1 * x;
  Fy += c.x1y2 * x * y2;
  Fx += c.x1y3 * x * y3;
  Fy += c.x2y2 * (x * x) * y2;
}

/* slopes of regular momenta (convertMomentaToSlopes) */
struct eh_reg_slopes {
  double xp, yp, f, y;
};

EH_HD eh_reg_slopes eh_reg_m2s(double qx, double qy, double b1s, double rh, double rh2) {
  eh_reg_slopes s;
  const double x2 = qx * qx, y2 = qy * qy;
  eh_reg_root(b1s - x2 - y2, (x2 + y2) * rh2, rh, s.f, s.y);
  s.xp = eh_reg_div(qx, s.f, s.y);
  s.yp = eh_reg_div(qy, s.f, s.y);
  return s;
}

/* Whether any of the wavefront's particles is beyond the limits at entry.  It needs
 * the general integrator, which costs the same for all of them: nobody goes on here.
 * How the compiler lays the code out after it decides a few per cent.  Told that the
 * mask is clear behind the vote (multipoles) and that the exit is unlikely (bends) lean
 * kernels gain 1 to 2 % with regular beams (FODO study 9.81 -> 9.71 ms, 30401 particles
 * through the MBA ring 15.25 -> 15.06, batch 30.4 -> 30.0).  In full kernels (FULL) an
 * unlikely exit costs the general integrators 5 to 8 % (elliptical aperture, 1e4
 * particles 11.1 -> 12.0), and a clear mask in the bends, too, gains 1 to 3 % (radiating
 * MBA ring 11.24 -> 11.13). */
EH_HD bool eh_reg_any(bool bad) {
#if defined(__HIP_DEVICE_COMPILE__)
  return __ballot(bad) != 0;
#else
  return bad;
#endif
}

/* zero, or far above underflow */
EH_HD bool eh_reg_sized(double ax) { return (ax >= EH_REG_QMIN) | (ax == 0); }

/* the field sums of one kick of order N, eh_mkick's terms and order (0 + v is
 * v + 0, one fma where v is a product) */
template <int ORDER> EH_HD void eh_reg_mfield(double x, double y, double &Fx, double &Fy) {
  if constexpr (ORDER == 1) {
    Fy = 0.0 + x;
    Fx = 0.0 + y;
  } else if constexpr (ORDER == 2) {
    Fy = eh_fma(0.5, x * x, 0.0);
    Fx = eh_fma(x, y, 0.0);
    Fy += -0.5 * (y * y);
  } else {
    const double x2 = x * x, y2 = y * y;
    Fy = eh_fma(1. / 6., x2 * x, 0.0);
    Fx = eh_fma(0.5 * x2, y, 0.0);
    Fy += -0.5 * x * y2;
    Fx += -(1. / 6.) * (y2 * y);
  }
}

/* integrate_kick_multipole_ordn without losses for a regular particle and one
 * term of the given order: slopes to momenta, the slices, and back; x, xp, y,
 * yp, s advance through the element if it returns true and are left alone
 * otherwise.  (1 + x'^2 + y'^2)^1/2 of a sub-step is (1 + delta) / f up to
 * roundings, which one correction step removes.  The exit's slopes are those of
 * the last kick. */
template <int ORDER, bool RAD>
EH_HD bool eh_mult_regular(const eh_desc &d, int pi, double &x_, double &xp_, double &y_, double &yp_, double &s_,
                           double &dp_) {
  double dp = dp_;
  double x = x_, y = y_, s = 0;
  const double mdx = d.mdx, mdy = d.mdy;
  const double apx = d.reg_apx[pi], apy = d.reg_apy[pi];
  const double h0 = d.reg_h[0], h1 = d.reg_h[1], k0 = d.reg_k[0], k1 = d.reg_k[1];
  const bool steering = d.has_xkick || d.has_ykick;
  double b1 = 1 + dp;
  bool bad = !(b1 >= EH_REG_B1_MIN && b1 <= EH_REG_B1_MAX && eh_fabs(x) <= 10.0 && eh_fabs(y) <= 10.0 &&
               eh_fabs(xp_) <= EH_REG_QMAX && eh_fabs(yp_) <= EH_REG_QMAX && eh_reg_sized(eh_fabs(xp_)) &&
               eh_reg_sized(eh_fabs(yp_)));
  if (eh_reg_any(bad))
    return false;
  bad = false; /* as it is for everyone now */
  double b1s = b1 * b1, rh = 1.0 / b1, rh2 = rh * rh, hrh = 0.5 * rh;
  double qx, qy;
  {
    const double u = eh_sqr(xp_) + eh_sqr(yp_);
    double w, yw;
    eh_reg_root(1 + eh_sqr(xp_) + eh_sqr(yp_), -u, 1.0, w, yw);
    qx = eh_reg_div(b1 * xp_, w, yw);
    qy = eh_reg_div(b1 * yp_, w, yw);
  }
  eh_reg_slopes v = eh_reg_m2s(qx, qy, b1s, rh, rh2);
  /* a particle in the mid-plane stays there, with qy = 0 */
  const bool midplane = (qy == 0) & (y == 0) & !steering;
  const int nsl = d.reg_nsl, nsub = d.reg_nsub;
  for (int ik = 0; ik < nsl; ik++) {
    bad |= !((eh_fabs(x + mdx) <= apx) & (eh_fabs(y + mdy) <= apy));
    for (int step = 0; step < nsub; step++) {
      double dsh = step == 1 || step == 2 ? h1 : h0;
      if (nsub == 8)
        dsh = d.dsh[step];
      x += v.xp * dsh;
      y += v.yp * dsh;
      const double a2 = 1 + eh_sqr(v.xp) + eh_sqr(v.yp);
      const double g = b1 * v.y;
      s += dsh * eh_fma(eh_fma(-g, g, a2), hrh * v.f, g);
      if (step == nsub - 1)
        break;
      double Fx, Fy;
      eh_reg_mfield<ORDER>(x, y, Fx, Fy);
      double K = step == 1 ? k1 : k0;
      if (nsub == 8)
        K = d.kick[step][0];
      double gx = K * Fy, gy = K * Fx; /* the field's increments, for the radiation */
      qx -= gx;
      qy += gy;
      if (steering) {
#if defined(__HIP_DEVICE_COMPILE__)
        __asm__ volatile(""); /* a scalar branch, not selects */
#endif
        /* eh_mkick<0>: the other plane gains a signed zero */
        if (d.has_xkick) {
          qx -= d.xk[step];
          qy += d.xk[step] * 0.0;
        }
        if (d.has_ykick) {
          qx -= d.yk[step] * 0.0;
          qy -= d.yk[step];
        }
      }
      const double ax = eh_fabs(qx), ay = eh_fabs(qy);
      bad |= !((ax <= EH_REG_QMAX) & (ay <= EH_REG_QMAX) & eh_reg_sized(ax) & ((ay >= EH_REG_QMIN) | midplane));
      if constexpr (RAD) {
        /* the energy loss, as the general integrator forms it; squares hide the
         * signs of zeros and anything near underflow */
        v = eh_reg_m2s(qx, qy, b1s, rh, rh2);
        const double kf = step == 1 ? d.reg_kf[1] : d.reg_kf[0], ikf = step == 1 ? d.reg_ikf[1] : d.reg_ikf[0];
        qx = eh_reg_div(qx, b1, rh);
        qy = eh_reg_div(qy, b1, rh);
        gx = eh_reg_div(eh_reg_div(-gx, kf, ikf), d.mdrift, d.reg_idrift);
        gy = eh_reg_div(eh_reg_div(gy, kf, ikf), d.mdrift, d.reg_idrift);
        const double F2 = eh_sqr(gx - d.reg_rxk) + eh_sqr(gy + d.reg_ryk);
        const double a2 = 1 + eh_sqr(v.xp) + eh_sqr(v.yp), g = b1 * v.y;
        const double w = eh_fma(eh_fma(-g, g, a2), hrh * v.f, g) * (d.mdrift * kf);
        dp -= d.rad_coef * b1s * F2 * w;
        b1 = 1 + dp;
        bad |= !(eh_reg_next_recip(b1, rh) & (b1 >= EH_REG_B1_MIN) & (b1 <= EH_REG_B1_MAX));
        b1s = b1 * b1;
        rh2 = rh * rh;
        hrh = 0.5 * rh;
        qx *= b1;
        qy *= b1;
      } else {
        /* the radiation block's division and multiplication by 1 + delta */
        qx = eh_reg_div(qx, b1, rh) * b1;
        qy = eh_reg_div(qy, b1, rh) * b1;
      }
      v = eh_reg_m2s(qx, qy, b1s, rh, rh2);
    }
  }
  bad |= !((eh_fabs(x + mdx) <= apx) & (eh_fabs(y + mdy) <= apy) & (eh_fabs(x) <= 10.0) & (eh_fabs(y) <= 10.0));
  if (bad)
    return false;
  x_ = x;
  xp_ = v.xp;
  y_ = y;
  yp_ = v.yp;
  s_ = s;
  dp_ = dp;
  return true;
}

template <bool RAD>
EH_HD bool eh_mult_regular_n(const eh_desc &d, int pi, double &x, double &xp, double &y, double &yp, double &s,
                             double &dp) {
  if (d.regular == 1)
    return eh_mult_regular<1, RAD>(d, pi, x, xp, y, yp, s, dp);
  if (d.regular == 2)
    return eh_mult_regular<2, RAD>(d, pi, x, xp, y, yp, s, dp);
  return eh_mult_regular<3, RAD>(d, pi, x, xp, y, yp, s, dp);
}

/* integrate_csbend_ordn without losses for a regular particle, slopes to momenta
 * before it and back after it: X, xp, Y, yp and the path `dist` advance through
 * the bend if it returns true and are left alone otherwise.  FIELD as
 * eh_desc.regular. */
template <int FIELD, bool RAD, bool FULL>
EH_HD bool eh_csb_regular(const eh_desc &d, int pi, const eh_fterm *__restrict__ terms, double &X_, double &xp_,
                          double &Y_, double &yp_, double &DP_, double &dist_) {
  double X = X_, QX, Y = Y_, QY, DP = DP_, dist = 0;
  double b1 = 1 + DP;
  bool bad = !(b1 >= EH_REG_B1_MIN && b1 <= EH_REG_B1_MAX && eh_fabs(xp_) <= EH_REG_QMAX &&
               eh_fabs(yp_) <= EH_REG_QMAX && eh_reg_sized(eh_fabs(yp_)));
  if (FULL ? eh_reg_any(bad) : __builtin_expect(eh_reg_any(bad), 0))
    return false;
  if constexpr (FULL)
    bad = false;
  const double rho0 = d.rho0, rho_a = d.rho_actual, r0h = d.rho0_rh, rah = d.rhoa_rh;
  const double apx = d.reg_apx[pi], apy = d.reg_apy[pi];
  const double h0 = d.reg_h[0], h1 = d.reg_h[1], k0 = d.reg_k[0], k1 = d.reg_k[1];
  double b1s = b1 * b1, rh = 1.0 / b1, rh2 = rh * rh;
  eh_grad_field gf;
  if constexpr (FIELD == 2)
    gf = eh_grad_load(terms + d.csb_dx0, terms + d.csb_dy0);
  {
    const double u = eh_sqr(xp_) + eh_sqr(yp_);
    double w, yw;
    eh_reg_root(1 + eh_sqr(xp_) + eh_sqr(yp_), -u, 1.0, w, yw);
    const double c = eh_reg_div(b1, w, yw);
    QX = xp_ * c;
    QY = yp_ * c;
  }
  /* f and 1 / f depend on QY alone, which drifts leave unchanged: formed at
   * entry and after every kick */
  double f, y;
  {
    const double q2 = QY * QY;
    eh_reg_root(b1s - q2, q2 * rh2, rh, f, y);
  }
  const eh_reg_series ks = eh_reg_series_load();
  const int nsl = d.reg_nsl, nsub = d.reg_nsub;
  /* A momentum that stays far above underflow has lost nothing to a tiny, inexact
   * kick.  QY may be zero throughout: always without field terms, in the mid-plane
   * with them. */
  const bool midplane = (QY == 0) & (FIELD == 1 || Y == 0);
  for (int i = 0; i < nsl; i++) {
    bad |= !((eh_fabs(X) <= apx) & (eh_fabs(Y) <= apy) & (eh_fabs(QX) <= EH_REG_QXMAX) &
             (eh_fabs(QX) >= EH_REG_QMIN));
    for (int j = 0; j < nsub; j++) {
      const double sin_phi = eh_reg_div(QX, f, y);
      const double phi = eh_reg_asin(sin_phi, ks);
      double th = j == 1 || j == 2 ? h1 : h0;
      if (nsub == 8)
        th = d.csb_dshr[j];
      const double ang = th + phi;
      bad |= !(eh_fabs(ang) < EH_REG_ANGLE);
      const double sine = eh_reg_sin(ang, ks), cosi = eh_reg_cos(ang, ks);
      const double yc = eh_reg_recip1(cosi);
      const double tang = eh_reg_div(sine, cosi, yc);
      const double cos_phi = eh_reg_cos(phi, ks);
      QX = f * sine;
      const double tphi = eh_reg_div(sin_phi, cos_phi, eh_reg_recip1(cos_phi));
      const double factor = eh_reg_div((rho0 + X) * cos_phi, f, y) * (tang - tphi);
      Y += QY * factor;
      dist += factor * b1;
      const double fr = eh_reg_div(cos_phi, cosi, yc);
      X = rho0 * (fr - 1) + fr * X;
      if (j == nsub - 1)
        break;
      double ds = j == 1 ? k1 : k0;
      if (nsub == 8)
        ds = d.csb_ds[j];
      const double u = ds * (1 + eh_reg_div(X, rho0, r0h));
      double Fx = 0, Fy = 1;
      if constexpr (FIELD == 2)
        eh_grad_eval(gf, X, Y, Fx, Fy);
      if constexpr (FIELD == 3)
        eh_csb_fields(d, terms, X, Y, Fx, Fy);
      QX -= eh_reg_div(u * Fy, rho_a, rah);
      QY += eh_reg_div(u * Fx, rho_a, rah);
      const double ax = eh_fabs(QX), ay = eh_fabs(QY);
      bad |= !((ax <= EH_REG_QXMAX) & (ay <= EH_REG_QMAX) & (ax >= EH_REG_QMIN) & ((ay >= EH_REG_QMIN) | midplane));
      if constexpr (RAD) {
        /* the energy loss of the sub-step as the general integrator forms it; its
         * path factor (h^2 + x'^2 + y'^2)^1/2, h = 1 + X / rho0, is (1 + delta) h / f
         * up to roundings */
        const double hx = 1 + X * d.csb_irho0;
        const double x2 = QX * QX, y2 = QY * QY;
        double f2, yf2;
        eh_reg_root<true>(b1s - x2 - y2, (x2 + y2) * rh2, rh, f2, yf2);
        const double c = eh_reg_div(hx, f2, yf2);
        const double xpr = QX * c, ypr = QY * c;
        const double a2 = eh_sqr(hx) + eh_sqr(xpr) + eh_sqr(ypr);
        const double r0 = 2.0 - hx, e = eh_fma(-hx, r0, 1.0);
        bad |= !(eh_fabs(X * d.csb_irho0) < 0x1p-9);
        const double g = b1 * c, ihx = eh_fma(r0, eh_fma(e, e, e), r0);
        const double w = eh_fma(eh_fma(-g, g, a2), 0.5 * (f2 * rh * ihx), g);
        const double F2 = eh_sqr(Fx) + eh_sqr(Fy);
        QX = eh_reg_div(QX, b1, rh);
        QY = eh_reg_div(QY, b1, rh);
        DP -= d.rad_coef * b1s * F2 * ds * w;
        b1 = 1 + DP;
        bad |= !(eh_reg_next_recip(b1, rh) & (b1 >= EH_REG_B1_MIN) & (b1 <= EH_REG_B1_MAX));
        b1s = b1 * b1;
        rh2 = rh * rh;
        QX *= b1;
        QY *= b1;
      } else {
        /* the radiation block's division and multiplication by 1 + delta */
        QX = eh_reg_div(QX, b1, rh) * b1;
        QY = eh_reg_div(QY, b1, rh) * b1;
      }
      const double q2 = QY * QY;
      eh_reg_root(b1s - q2, q2 * rh2, rh, f, y);
    }
  }
  bad |= !((eh_fabs(X) <= apx) & (eh_fabs(Y) <= apy) & (eh_fabs(QX) <= EH_REG_QMAX));
  if (bad)
    return false;
  const double x2 = QX * QX, y2 = QY * QY;
  eh_reg_root(b1s - x2 - y2, (x2 + y2) * rh2, rh, f, y);
  const double c = eh_reg_div(1.0, f, y);
  X_ = X;
  xp_ = QX * c;
  Y_ = Y;
  yp_ = QY * c;
  DP_ = DP;
  dist_ = dist;
  return true;
}

template <bool RAD, bool FULL>
EH_HD bool eh_csb_regular_n(const eh_desc &d, int pi, const eh_fterm *__restrict__ terms, double &X, double &xp,
                            double &Y, double &yp, double &DP, double &dist) {
  if (d.regular == 2)
    return eh_csb_regular<2, RAD, FULL>(d, pi, terms, X, xp, Y, yp, DP, dist);
  if (d.regular == 1)
    return eh_csb_regular<1, RAD, FULL>(d, pi, terms, X, xp, Y, yp, DP, dist);
  return eh_csb_regular<3, RAD, FULL>(d, pi, terms, X, xp, Y, yp, DP, dist);
}

#endif
