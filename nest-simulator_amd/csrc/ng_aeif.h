// ng_aeif.h -- adaptive Runge-Kutta-Fehlberg 4(5) for aeif_cond_exp, four lanes per neuron.
//
// Stands in for the GSL stepper NEST uses (models/aeif_cond_exp.cpp:386,395,463:
// gsl_odeiv_step_rkf45, gsl_odeiv_control_yp_new(tol, tol), gsl_odeiv_evolve_apply).
// GSL is a third-party library outside the reference tree; its published method is:
//   * Fehlberg's 4(5) tableau, propagating the 5th-order solution, error = 5th - 4th;
//   * y' error control: D_i = eps_abs + eps_rel * |h y'_i|, r = max |yerr_i| / D_i,
//     shrink by S r^(-1/q) (>= 1/5) when r > 1.1, grow by S r^(-1/(q+1)) (<= 5, >= 1)
//     when r < 0.5, S = 0.9, q = 5 (the stepper's order);
//   * evolve: one accepted step towards t1 per call, clipped to t1, retried from the saved
//     state when the controller shrinks h and the shrink moves t by at least one ulp.
// The right-hand side follows aeif_cond_exp_dynamics (models/aeif_cond_exp.cpp:79-124).
//
// Lane c of a neuron's quad of lanes holds component c of the state (V_m, g_ex, g_in, w). The
// stage sums, the error and the final division of each component's derivative are then the
// same instructions in all four lanes, done once instead of four times; the spike current is
// computed in all four; components meet through quad permutes. A neuron's steps are a serial
// chain and the slowest neuron of a network (up to 166 attempted steps in a slice of 15 steps,
// where the mean is 16) decides how long a slice takes, so the chain's length is what counts:
// an attempt takes about 700 instructions per lane instead of 1,300, and its registers fit
// without spilling.
#pragma once

#include "ng_math.h"

namespace nestgpu
{

// x of lane J of the lane's quad / of the lane with quad index c ^ X
template < int CTRL >
__device__ __forceinline__ double
quad_perm( double x )
{
  const uint64_t b = __builtin_bit_cast( uint64_t, x );
  const uint32_t lo = static_cast< uint32_t >(
    __builtin_amdgcn_update_dpp( 0, static_cast< int >( b ), CTRL, 0xf, 0xf, true ) );
  const uint32_t hi = static_cast< uint32_t >(
    __builtin_amdgcn_update_dpp( 0, static_cast< int >( b >> 32 ), CTRL, 0xf, 0xf, true ) );
  return __builtin_bit_cast( double, ( static_cast< uint64_t >( hi ) << 32 ) | lo );
}
template < int J >
__device__ __forceinline__ double
quad_bcast( double x )
{
  return quad_perm< J * 0x55 >( x );
}
template < int J >
__device__ __forceinline__ uint32_t
quad_bcast( uint32_t x )
{
  return static_cast< uint32_t >(
    __builtin_amdgcn_update_dpp( 0, static_cast< int >( x ), J * 0x55, 0xf, 0xf, true ) );
}

// Parameters in one lane. E, m, den: the lane's reversal potential (E_L, E_ex, E_in, E_L),
// its multiplier of V - E (-g_L and a in lanes 0 and 3; lanes 1 and 2 use their conductance)
// and its divisor (C_m, tau_ex, tau_in, tau_w); r_*: refined reciprocals (ng_recip). FAST, below:
// divisions by the constants go through these; otherwise they are plain. zero_fits: a component
// of 0 allows them (aeif_fast_state).
struct AeifLane
{
  int c;
  bool zero_fits;
  double V_peak, V_reset, V_th, Delta_T, gD, I_e, tol;
  double E, m, den, r_den, r_Delta_T;
};

// Whether a step from the lane's component y may divide by reciprocals, where the parameters allow
// it (ParamSet p[18]): y is at least 2^-300 in size; a conductance, and w if a is 0, may also be 0.
// The dividends of such a step are 0 or at least 2^-900, so that ng_div gives every bit of the
// plain quotient:
//   - a stage y + h k is 0 or at least 2^-53 |y|, and 0 where y and k are;
//   - V - E is 0 or at least 2^-354, so every current but the spike current is 0 or at least
//     2^-708, and a sum of them is 0 or at least 2^-761; as is a (V - E_L) - w;
//   - the spike current may be smaller, but counts only if the others are all 0 (V = E_L). It then
//     changes neither V, which is at least 2^-300, nor the step size, whose growth is at its bound.
// Below, bits get lost: a conductance of 0.2 ms without input is less than 2^-1016 after 141 ms,
// where ng_div misses the last bit of 1 to 9 % of the quotients. Overflow gives NaN, which the
// end of the step shows (aeif_finite).
// 6,000 neurons in slices of 15 steps take 4 % longer with it (306 -> 318 us); looking at each
// dividend took 6 %, collecting their range or a branch at each division 9 %.
__device__ __forceinline__ bool
aeif_fast_state( const AeifLane& P, double y )
{
  return fabs( y ) >= 0x1p-300 or ( P.zero_fits and y == 0.0 );
}

__device__ __forceinline__ bool
aeif_finite( double y, double yp )
{
  return fabs( y ) + fabs( yp ) < INFINITY;
}

// g_L Delta_T exp( ( V - V_th ) / Delta_T ) of the effective potential V
template < bool FAST >
__device__ __forceinline__ double
aeif_spike_current( const AeifLane& P, double V )
{
  // a quotient too small for ng_div to be exact leaves the exponential at 1, one that overflows
  // (Delta_T is at least 1e-6) at 0
  const double x = V - P.V_th;
  const double e = P.gD * ng_exp( FAST ? ng_div( x, P.Delta_T, P.r_Delta_T ) : x / P.Delta_T );
  return P.Delta_T == 0. or x < -1e300 ? 0. : e;
}

__device__ __forceinline__ double
aeif_V( const AeifLane& P, bool refractory, double V )
{
  return refractory ? P.V_reset : ( P.V_peak < V ? P.V_peak : V );  // std::min
}

// The lane's component of the right-hand side at effective potential V with spike current
// I_spike; y: the lane's component of the state
template < bool FAST >
__device__ __forceinline__ double
aeif_dynamics( const AeifLane& P, bool refractory, double V, double I_spike, double y )
{
  const double p = ( P.c == 1 or P.c == 2 ? y : P.m ) * ( V - P.E );
  const double I_syn_exc = quad_bcast< 1 >( p );
  const double I_syn_inh = quad_bcast< 2 >( p );
  const double w = quad_bcast< 3 >( y );
  // currents_ carries no CurrentEvents on this path: I_stim_ == 0.0
  double I = p + I_spike - I_syn_exc - I_syn_inh - w + P.I_e + 0.0;
  // only lane 0 uses it: without this the compiler moves the sum and the spike current into a
  // branch of that lane, whose masks and jumps lengthen the chain of every stage
  asm( "" : "+v"( I ) );
  const double num = P.c == 0 ? I : P.c == 3 ? p - y : -y;
  const double f = FAST ? ng_div( num, P.den, P.r_den ) : num / P.den;
  return refractory and P.c == 0 ? 0. : f;
}

// the same at state component y, evaluating the spike current; it is returned in I_spike
template < bool FAST >
__device__ __forceinline__ double
aeif_rhs( const AeifLane& P, bool refractory, double y, double& I_spike )
{
  const double V = aeif_V( P, refractory, quad_bcast< 0 >( y ) );
  I_spike = aeif_spike_current< FAST >( P, V );
  return aeif_dynamics< FAST >( P, refractory, V, I_spike, y );
}

// One attempted step of size h from component y, where the spike current is I_start: the lane's
// component at its end, the error of the embedded 4th-order solution, and the derivative and the
// spike current at the end.
template < bool FAST >
__device__ __forceinline__ double
aeif_step( const AeifLane& P, bool refr, double y, double h, double I_start, double& yerr, double& yp, double& I_end )
{
  const double b21 = 1.0 / 4.0;
  const double b31 = 3.0 / 32.0, b32 = 9.0 / 32.0;
  const double b41 = 1932.0 / 2197.0, b42 = -7200.0 / 2197.0, b43 = 7296.0 / 2197.0;
  const double b51 = 8341.0 / 4104.0, b52 = -32832.0 / 4104.0, b53 = 29440.0 / 4104.0, b54 = -845.0 / 4104.0;
  const double b61 = -6080.0 / 20520.0, b62 = 41040.0 / 20520.0, b63 = -28352.0 / 20520.0, b64 = 9295.0 / 20520.0,
               b65 = -5643.0 / 20520.0;
  const double c1 = 902880.0 / 7618050.0, c3 = 3953664.0 / 7618050.0, c4 = 3855735.0 / 7618050.0,
               c5 = -1371249.0 / 7618050.0, c6 = 277020.0 / 7618050.0;
  const double ec1 = 1.0 / 360.0, ec3 = -128.0 / 4275.0, ec4 = -2197.0 / 75240.0, ec5 = 1.0 / 50.0, ec6 = 2.0 / 55.0;
  double I;
  const double k1 = aeif_dynamics< FAST >( P, refr, aeif_V( P, refr, quad_bcast< 0 >( y ) ), I_start, y );
  const double k2 = aeif_rhs< FAST >( P, refr, y + b21 * h * k1, I );
  const double k3 = aeif_rhs< FAST >( P, refr, y + h * ( b31 * k1 + b32 * k2 ), I );
  const double k4 = aeif_rhs< FAST >( P, refr, y + h * ( b41 * k1 + b42 * k2 + b43 * k3 ), I );
  const double k5 = aeif_rhs< FAST >( P, refr, y + h * ( b51 * k1 + b52 * k2 + b53 * k3 + b54 * k4 ), I );
  const double k6 = aeif_rhs< FAST >( P, refr, y + h * ( b61 * k1 + b62 * k2 + b63 * k3 + b64 * k4 + b65 * k5 ), I );
  const double y1 = y + h * ( c1 * k1 + c3 * k3 + c4 * k4 + c5 * k5 + c6 * k6 );
  yerr = h * ( ec1 * k1 + ec3 * k3 + ec4 * k4 + ec5 * k5 + ec6 * k6 );
  yp = aeif_rhs< FAST >( P, refr, y1, I_end );
  return y1;
}

// y' error control of a step of size h with derivative yp at its end: -1 (decrease), 0 (keep)
// or +1 (increase), and the next step size in *h. The two rules differ in exponent and bounds
// only, so one power serves a wave whose lanes take either.
__device__ __forceinline__ int
aeif_yp_hadjust( double tol, double yerr, double yp, double* h )
{
  const double S = 0.9;
  const double h_old = *h;
  const double D0 = tol * ( 0.0 * fabs( 0.0 ) + 1.0 * fabs( h_old * yp ) ) + tol;
  double rmax = fabs( yerr ) / fabs( D0 );
  // the largest over the components and DBL_MIN; a NaN is passed over, as r > rmax does
  rmax = fmax( rmax, quad_perm< 0xB1 >( rmax ) );
  rmax = fmax( rmax, quad_perm< 0x4E >( rmax ) );
  rmax = fmax( 2.2250738585072014e-308, rmax );
  const bool shrink = rmax > 1.1, grow = rmax < 0.5;
  if ( not( shrink or grow ) )
    return 0;
  double r = S / ng_pow( rmax, shrink ? 1.0 / 5.0 : 1.0 / ( 5.0 + 1.0 ) );
  if ( shrink )
    r = r < 0.2 ? 0.2 : r;
  else
  {
    r = r > 5.0 ? 5.0 : r;
    r = r < 1.0 ? 1.0 : r;
  }
  *h = r * h_old;
  return shrink ? -1 : 1;
}

}  // namespace nestgpu
