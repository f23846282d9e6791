// vacc_lean.h -- tolerance form of the remap arithmetic (options.fast_arith = 1), host +
// device: the PLM / PPM / PQM reconstructions rewritten for few VALU instructions, and the
// flux-form deposit of one pencil.  The device remap (k_remap_lean) and the CPU checks
// compile the same code.
//
// Reconstructions (cpu_1d_plm.hpp:38-49, cpu_1d_ppm.hpp:35-54, cpu_1d_pqm.hpp:31-173,
// cpu_face_estimates.hpp, cpu_slope_limiters.hpp) in deviations from the cell average v:
// u_l = (left face) - v, u_r = (right face) - v.  The reference's tests keep their meaning:
//   (v[-1] - f_l)(f_l - v) < 0   <=>  u_l outside [-b, 0]    with b = v - v[-1]
//   (v[+1] - f_r)(f_r - v) < 0   <=>  u_r outside [0, a]     with a = v[+1] - v
// each one median of three and a compare.
// and the PQM quartic F(x) = x (c0 + x (c1 + x (c2 + x (c3 + x c4)))) has
//   c0 = v + u_l, c1 = d_l / 2, c2 = -6 u_l - 4 u_r - (3 d_l - d_r) / 2,
//   c3 = 8 u_l + 7 u_r + (3 d_l - 2 d_r) / 2, c4 = -3 (u_l + u_r) + (d_r - d_l) / 2,
// whose monotonicity coefficients are b0 = 6 c2, b1 = 24 c3, b2 = 60 c4 (White & Adcroft
// 2008).  The critical points of F' are then (-2 c3 +- sqrt(4 c3^2 - 10 c2 c4)) / (10 c4) and
// F' = d_l + x (6 c2 + x (12 c3 + x 20 c4)).  The reference tests F' at both critical points
// (with a fallback root for a negative discriminant, sqrt -> b1 + 200 b2); here a Bernstein
// bound passes most cells without either, and the others test the one critical point where
// F' can first take the wrong sign (the same decision: see ReconLean<PQM>::coeffs).
// Multiplies are fused, 1/x and sqrt are the hardware's; results agree with the reference's
// FP32 rounding to a few ulp of the faces.
//
// Deposit (cpu_acc_map.cpp:533-628) in flux form: Lagrangian boundary g of the pencil lies at
// Imin + g dk, t is the next boundary's offset from the current source cell's left edge in
// units of dv, r = dk / dv.  A source cell closes every target whose right boundary it holds
// with F(t) - F(previous boundary in the cell) (plus what earlier cells gave that target) and
// leaves v - F(last boundary) in the open target: every source cell's mass is deposited once,
// with F(1) taken as the cell average v.  The reference evaluates F at both ends of every
// overlap instead, with the Lagrangian coordinates in FP32 (|v| up to 4e6 m/s, ulp 0.25 m/s,
// about 1e-5 of a cell).
#pragma once

#include <math.h>

#include "vacc_common.h"

namespace vacc {

VACC_HD float lean_rcp(float x) {
#if defined(__HIP_DEVICE_COMPILE__)
   return __builtin_amdgcn_rcpf(x);
#else
   return 1.0f / x;
#endif
}
VACC_HD float lean_sqrt(float x) {
#if defined(__HIP_DEVICE_COMPILE__)
   return __builtin_amdgcn_sqrtf(x);
#else
   return sqrtf(x);
#endif
}

// Face estimates with pre-divided weights (cpu_face_estimates.hpp:45-56, :68-78, :160-167).
VACC_HD float lean_h4(const float* v) {   // left face of v[0]
   return fmaf(7.0f / 12.0f, v[-1] + v[0], (-1.0f / 12.0f) * (v[-2] + v[1]));
}
VACC_HD float lean_h8(const float* v) {
   float s = (533.0f / 840.0f) * (v[-1] + v[0]);
   s = fmaf(-139.0f / 840.0f, v[-2] + v[1], s);
   s = fmaf(29.0f / 840.0f, v[-3] + v[2], s);
   return fmaf(-3.0f / 840.0f, v[-4] + v[3], s);
}
// half the h7 face derivative
VACC_HD float lean_h7h(const float* v) {
   float s = (7175.0f / 10080.0f) * (v[0] - v[-1]);
   s = fmaf(-889.0f / 10080.0f, v[1] - v[-2], s);
   s = fmaf(119.0f / 10080.0f, v[2] - v[-3], s);
   return fmaf(-9.0f / 10080.0f, v[3] - v[-4], s);
}

// Half the superbee slope (cpu_slope_limiters.hpp:30-54) of a = v[1] - v[0], b = v[0] - v[-1], with
// ha = a/2 and hb = b/2: the signed superbee max(min(|a|, 2|b|), min(2|a|, |b|)) of two slopes of
// one sign is the median of a, b and twice the smaller one, and med3(a, b, 0) is the smaller
// one, or 0 when the signs differ (the outer median is then 0 as well).  Two instructions with
// the halves carried from cell to cell, in place of ten.
VACC_HD float lean_half_superbee(float a, float b, float ha, float hb) {
   return med3(ha, hb, med3(a, b, 0.0f));
}
// u lies outside the closed interval between 0 and a (a face outside its two cells' averages)
VACC_HD bool lean_outside(float u, float a) { return med3(u, 0.0f, a) != u; }

template <int METHOD>
struct ReconLean;

template <>
struct ReconLean<VACC_PLM> {
   static constexpr int NC = 2;
   float b, hb;   // v[0] - v[-1] and its half
   VACC_HD void start(const float* v) {
      b = v[0] - v[-1];
      hb = 0.5f * b;
   }
   VACC_HD void coeffs(const float* v, float* c) {
      const float a = v[1] - v[0], ha = 0.5f * a;
      const float hd = lean_half_superbee(a, b, ha, hb);
      b = a;
      hb = ha;
      c[0] = v[0] - hd;
      c[1] = hd;
   }
};

template <>
struct ReconLean<VACC_PPM> {
   static constexpr int NC = 3;
   float fl, b, hb;   // h4 left face of the current cell; v[0] - v[-1] and its half
   bool out;          // the left face lies outside [v[-1], v[0]] (the previous cell's right test)
   VACC_HD void start(const float* v) {
      fl = lean_h4(v);
      b = v[0] - v[-1];
      hb = 0.5f * b;
      out = lean_outside(fl - v[0], -b);
   }
   VACC_HD void coeffs(const float* v, float* c) {
      const float vk = v[0];
      const float fr = lean_h4(v + 1);
      const float a = v[1] - vk, ha = 0.5f * a;
      const float hs = lean_half_superbee(a, b, ha, hb);
      float ul = fl - vk, ur = fr - vk;
      // flat cell (zero slope) or a face outside its neighbours: the face moves to v -+ slope/2.
      // The right face's test serves the next cell's left face.
      const bool flat = (hs == 0.0f);
      const bool lout = out;
      out = lean_outside(ur, a);
      ul = (flat | lout) ? -hs : ul;
      ur = (flat | out) ? hs : ur;
      // Colella-Woodward: (p - m)(v - (m + p)/2) > (p - m)^2 / 6  <=>  (u_r - u_l)(u_l + 2 u_r) < 0.
      // After the face checks u_l and u_r have opposite signs (or are 0), so this is |u_l| > 2 |u_r|,
      // and u_l becomes the smaller of u_l and -2 u_r; the right test likewise.
      ul = med3(ul, -2.0f * ur, 0.0f);
      ur = med3(ur, -2.0f * ul, 0.0f);
      fl = fr;
      b = a;
      hb = ha;
      c[0] = vk + ul;
      c[1] = fmaf(-2.0f, ul, -ur);
      c[2] = ul + ur;
   }
};

template <>
struct ReconLean<VACC_PQM> {
   static constexpr int NC = 5;
   float fv, fd, b, hb;   // h8 value and half h7 derivative of the left face; v[0] - v[-1] and its half
   bool out;              // the left face lies outside [v[-1], v[0]] (the previous cell's right test)
   VACC_HD void start(const float* v) {
      fv = lean_h8(v);
      fd = lean_h7h(v);
      b = v[0] - v[-1];
      hb = 0.5f * b;
      out = lean_outside(fv - v[0], -b);
   }
   // c[2..4] from the face deviations and half derivatives gl, gr (d = 2 g): ten operations.  Sharing
   // e = ul + ur, gr - gl and ul + gl between the three takes eight, about 1 % of a step, but rounds
   // otherwise, which 16-bit subcycles carry on to 3e-5 of the momentum.
   VACC_HD static void quartic(float ul, float ur, float gl, float gr, float& c2, float& c3, float& c4) {
      c2 = fmaf(-6.0f, ul, fmaf(-4.0f, ur, fmaf(-3.0f, gl, gr)));
      c3 = fmaf(8.0f, ul, fmaf(7.0f, ur, fmaf(3.0f, gl, -2.0f * gr)));
      c4 = fmaf(-3.0f, ul + ur, gr - gl);
   }
   VACC_HD void coeffs(const float* v, float* c) {
      const float vk = v[0];
      const float fvr = lean_h8(v + 1), fdr = lean_h7h(v + 1);
      const float a = v[1] - vk, ha = 0.5f * a;
      const float hs = lean_half_superbee(a, b, ha, hb);   // half the signed limited slope
      const float bo = b;
      float ul = fv - vk, ur = fvr - vk, gl = fd, gr = fdr;   // gl, gr: half the face derivatives
      fv = fvr;
      fd = fdr;
      b = a;
      hb = ha;
      // flat cell, a face outside its neighbours or a face derivative against the slope: PLM
      // face.  The outside test of a face is the same for both cells that share it, so the right
      // face's result serves the next cell's left face.
      const bool flat = (hs == 0.0f);
      const bool lout = out;
      out = lean_outside(ur, a);
      const bool lp = flat | lout | (hs * gl < 0.0f);
      const bool rp = flat | out | (hs * gr < 0.0f);
      ul = lp ? -hs : ul;
      gl = lp ? hs : gl;
      ur = rp ? hs : ur;
      gr = rp ? hs : gr;
      float c2, c3, c4;
      quartic(ul, ur, gl, gr, c2, c3, c4);
      // monotonicity: the quartic's derivative at its critical points inside [0, 1] must
      // have the sign of psl + psr = 2 (a + b).  F' = 2 gl + x (6 c2 + x (12 c3 + x 20 c4)) has
      // the Bernstein coefficients 2 gl, 2 (gl + c2), 2 (gl + 2 (c2 + c3)), 2 gr on [0, 1]; the
      // end ones carry the sign of a + b (or are 0) after the face checks above.  When the inner
      // two do as well, so does F' on all of [0, 1] (it lies in their convex hull) and the cell
      // passes; otherwise the critical points are tested.  A cell that is not flat has a and b of
      // one sign, and a flat one has c2 = c3 = c4 = 0 and passes, so a's sign serves for a + b's.
      const float bn1 = (gl + c2) * a, bn2 = fmaf(2.0f, c2 + c3, gl) * a;
      bool bad = false;
      if (!(fminf(bn1, bn2) >= 0.0f)) {
         // The critical points are x = (-2 c3 +- sq) / (10 c4), sq = sqrt(4 c3^2 - 10 c2 c4).
         // The third derivative there is +-12 sq, so the + root is the local minimum of F' and
         // the - root its local maximum.  With both ends of F' on the side of a, F' crosses
         // to the other side at a critical point only if it does at the local minimum of
         // a F': the + root for a > 0, the - root for a < 0 (a wrong-signed local maximum
         // of a F' inside [0, 1] has a lower local minimum between it and an end).  A
         // negative discriminant leaves F' monotone between its two well-signed ends, and the
         // reference's fallback root then finds nothing either.  A point outside [0, 1] is
         // moved to the nearer end, where F' has the side of a, in place of the range test.
         const float disc = fmaf(4.0f * c3, c3, -10.0f * (c2 * c4));
         const float x0 = (copysignf(lean_sqrt(fmaxf(disc, 0.0f)), a) - 2.0f * c3) * lean_rcp(10.0f * c4);
         const float x = fminf(fmaxf(x0, 0.0f), 1.0f);
         const float d = fmaf(x, fmaf(x, fmaf(x, 10.0f * c4, 6.0f * c3), 3.0f * c2), gl);   // F'/2
         bad = disc >= 0.0f && d * a < 0.0f;
      }
      if (bad) {
         // repair (cpu_1d_pqm.hpp:79-145) on the side of the smaller one-sided slope
         const bool lft = fabsf(bo) <= fabsf(a);
         const float glx = lft ? (-1.0f / 3.0f) * fmaf(4.0f, ul, ur) : fmaf(-3.0f, ul, -2.0f * ur);
         const float grx = lft ? fmaf(2.0f, ul, 3.0f * ur) : (1.0f / 3.0f) * fmaf(4.0f, ur, ul);
         if (a * glx < 0.0f) {          // left derivative flattened
            gl = 0.0f;
            // products first, then the choice: a choice between two constants would hold
            // both in registers for the whole kernel
            ur = lft ? -4.0f * ul : -1.5f * ul;
            gr = lft ? -10.0f * ul : (-5.0f / 3.0f) * ul;
         } else if (a * grx < 0.0f) {   // right derivative flattened
            gr = 0.0f;
            ul = lft ? -1.5f * ur : -4.0f * ur;
            gl = lft ? (5.0f / 3.0f) * ur : 10.0f * ur;
         } else {
            gl = glx;
            gr = grx;
         }
         quartic(ul, ur, gl, gr, c2, c3, c4);
      }
      c[0] = vk + ul;
      c[1] = gl;
      c[2] = c2;
      c[3] = c3;
      c[4] = c4;
   }
};

// F(x) = x (c0 + x (c1 + ...)), the integral of the reconstruction over [0, x] (units of dv).
template <int NC>
VACC_HD float lean_integral(float x, const float* c) {
   float s = c[NC - 1];
#pragma unroll
   for (int i = NC - 2; i >= 0; --i) s = fmaf(x, s, c[i]);
   return x * s;
}

// Flux-form deposit along one pencil (see the file comment).
template <int NC>
struct Flux {
   float t;        // next boundary, from the current source cell's left edge, in units of dv
   float r;        // dk / dv
   float acc;      // mass of the open target o from earlier source cells
   int o;          // the open target: its right edge is the next boundary

   // x0 = (v0 - Imin) / dk: the Lagrangian coordinate of the first source cell's left edge
   VACC_HD void begin(double x0, float r_) {
      const double fl = floor(x0);
      o = (int)fl;
      t = (float)((fl + 1.0 - x0) * (double)r_);
      r = r_;
      acc = 0.0f;
   }
   // One source cell with integral coefficients c and average v; emit(target, mass) receives
   // each target this cell closes, with the target's whole mass from this pencil.  The receiver
   // stores the emits: the first boundary is handled without a branch, and a cell that holds
   // none emits the open target's mass so far, which the target's closing emit supersedes.
   template <class Emit>
   VACC_HD void cell(const float* c, float v, Emit&& emit) {
      const bool hit = t < 1.0f;
      float Fp = lean_integral<NC>(hit ? t : 0.0f, c);   // F(0) = 0
      const float s = acc + Fp;
      emit(o, s);
      o += hit ? 1 : 0;
      // The boundary moves by r before the cell's width is taken off, not by r - 1 at once: that
      // saves an operation, but rounds differently in the same direction along a whole pencil, which
      // moved the momentum of 16-bit subcycles by 3e-5.
      t = hit ? t + r : t;
      while (t < 1.0f) {        // more boundaries in this cell (dk < dv)
         const float Ft = lean_integral<NC>(t, c);
         emit(o, Ft - Fp);
         Fp = Ft;
         ++o;
         t += r;
      }
      t -= 1.0f;                // from the next cell's left edge
      acc = v + (hit ? -Fp : s);   // without a boundary Fp = 0 and the open target keeps its mass
   }
   // the open target after the pencil's last source cell
   template <class Emit>
   VACC_HD void end(Emit&& emit) {
      emit(o, acc);
   }
};

}  // namespace vacc
