// gqa_math.h -- arithmetic in double with no device builtins: RoPE's sines and cosines and a
// quotient (their errors are measured on the host too).
#pragma once

#include <cmath>

namespace gqa {

// The Taylor coefficients at z = r^2 of sin r = r + r z ps and cos r = 1 - z/2 + z^2 pc.
__host__ __device__ __forceinline__ void sincos_poly(double z, double& ps, double& pc) {
    ps = 1.0 / 355687428096000.0;      // 1/17!
    pc = 1.0 / 20922789888000.0;       // 1/16!
    ps = fma(ps, z, -1.0 / 1307674368000.0);
    pc = fma(pc, z, -1.0 / 87178291200.0);
    ps = fma(ps, z, 1.0 / 6227020800.0);
    pc = fma(pc, z, 1.0 / 479001600.0);
    ps = fma(ps, z, -1.0 / 39916800.0);
    pc = fma(pc, z, -1.0 / 3628800.0);
    ps = fma(ps, z, 1.0 / 362880.0);
    pc = fma(pc, z, 1.0 / 40320.0);
    ps = fma(ps, z, -1.0 / 5040.0);
    pc = fma(pc, z, -1.0 / 720.0);
    ps = fma(ps, z, 1.0 / 120.0);
    pc = fma(pc, z, 1.0 / 24.0);
    ps = fma(ps, z, -1.0 / 6.0);
}

// sin and cos of an angle 4 q quarter turns on from r (sr, cr: r's).
__host__ __device__ __forceinline__ void sincos_quadrant(double q, double sr, double cr, double& s, double& c) {
    const int n = static_cast<int>(4.0 * (q - floor(q)));
    const double a = (n & 1) ? cr : sr, b = (n & 1) ? sr : cr;
    s = (n & 2) ? -a : a;
    c = ((n + 1) & 2) ? -b : b;
}

// sin and cos of an angle in double: reduced to |r| <= pi/4 with a two-part Cody-Waite pi/2
// and fused multiply-adds, then the Taylor series of both (first omitted terms at pi/4: 9e-20
// for the sine, 2.1e-18 for the cosine) and the quadrant.  The reduction runs twice: from
// angles of about 2^46 on the rounding of angle * 2/pi can put k one off, and the second step
// takes that back (on smaller angles its j is 0, or +-1 where r sits at pi/4).  Against 113-bit
// values for every frequency of theta = 500000 at positions up to 400,000: largest error
// 1.2e-16, rms 3.1e-17; over all angles below 2^53 1.9e-16 (the library's sincos of the angle
// reduced modulo 2 pi: 2.5e-16 and 6.2e-17, in about three times the instructions; the kernels
// here wait for one sincos after the other at their start).  From 2^54 on the two parts of pi/2
// are too few bits and the error grows with the angle (1.9e-15 below 2^58); the clamp keeps
// what is left past about 2^105 bounded.
__host__ __device__ __forceinline__ void sincos_f64(double angle, double& s, double& c) {
    const double k = rint(angle * 0.63661977236758134308);    // 2 / pi
    double r = fma(-k, 1.5707963267948965580, angle);          // pi / 2 rounded to double
    r = fma(-k, 6.1232339957367658e-17, r);                    // pi / 2 - that
    const double j = rint(r * 0.63661977236758134308);
    r = fma(-j, 1.5707963267948965580, r);
    r = fma(-j, 6.1232339957367658e-17, r);
    r = r > 0.8 ? 0.8 : r;
    r = r < -0.8 ? -0.8 : r;
    const double z = r * r;
    double ps, pc;
    sincos_poly(z, ps, pc);
    const double sr = fma(r * z, ps, r);
    const double hz = 0.5 * z;
    const double w = 1.0 - hz;
    const double cr = w + fma(z * z, pc, (1.0 - w) - hz);
    // quadrant (k + j) mod 4 (both may exceed the int range, and their sum's last bit a double)
    sincos_quadrant((k * 0.25 - floor(k * 0.25)) + j * 0.25, sr, cr, s, c);
}

// cos and sin of the exact product p * f (|p f| <= kKRopeMaxAngle): sincos_f64 with the product's
// rounding error and the reduced angle's carried along.  Largest error 8e-17.
__host__ __device__ __forceinline__ void rot_exact(double p, double f, double& c, double& s) {
    const double ang = p * f;
    const double k = rint(ang * 0.63661977236758134308);
    const double r1 = fma(-k, 1.5707963267948965580, ang);
    const double t = fma(-k, 6.1232339957367658e-17, fma(p, f, -ang));
    const double r = r1 + t;
    const double rl = t - (r - r1);
    const double z = r * r;
    double ps, pc;
    sincos_poly(z, ps, pc);
    const double hz = 0.5 * z;
    const double w = 1.0 - hz;
    const double sr = r + fma(r * z, ps, fma(-hz, rl, rl));
    const double cr = w + fma(z * z, pc, ((1.0 - w) - hz) - fma(r, rl, 0.5 * fma(r, r, -z)));
    sincos_quadrant(k * 0.25, sr, cr, s, c);
}

// cos and sin of the rounded product pos * f, pos = p + d, from rot_exact(p, f) (bc, bs) and
// rot_exact(d, f) (dc, ds): their product, turned by the rounding error dl of pos * f (the golden
// rotates at the rounded angle).  Of first order in dl, at most half the spacing of doubles
// at the angle: dl^2 / 2 <= 7e-18 up to kKRopeMaxAngle.  Largest error against 113-bit values
// over positions up to 400,000 and theta = 500000: 2.3e-16, rms 4.5e-17 (the library's sincos of
// the reduced angle: 2.5e-16 and 6.0e-17; with the turn after the product, two instructions
// less, 3.4e-16 and 5.6e-17).
constexpr double kKRopeMaxAngle = 67108864.0;            // 2^26
__host__ __device__ __forceinline__ void rot_turn(double bc, double bs, double dc, double ds, double pos, double f,
                                                  double& c, double& s) {
    const double dl = fma(pos, f, -(pos * f));
    const double s0 = fma(bs, dc, bc * ds);
    c = fma(bc, dc, fma(-bs, ds, dl * s0));
    s = fma(bs, dc, fma(bc, ds, -(dl * c)));
}

// a / b from inv = 1 / b: the product, which two roundings leave up to 2 ULP off, and one step
// with its remainder, which rounds once (and equals a / b but for exact ties' neighbours).  32
// quotients by one l take 32 products and 64 fmas, as divisions about 350 instructions.
__host__ __device__ __forceinline__ double quotient(double a, double b, double inv) {
    const double q = a * inv;
    return fma(fma(-q, b, a), inv, q);
}

}  // namespace gqa
