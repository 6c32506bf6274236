// ng_models_dev.h -- the device halves of the neuron models.
//
// For each model id registered with ModelManager (ng_model.h), DeviceNode< id > gives what
// nest::Node gives the reference's update loop (nestkernel/node.h:297,572):
//   - receive: handle( SpikeEvent& ) -- the ring-buffer channel an event of weight w (weight
//     times multiplicity) goes to, and the value added there;
//   - load: its state (fields v0..v4 and r of its device index), read when the workgroup starts;
//   - update: update( origin, from, to ) of one neuron over the lags [ph.from, ph.to) of the
//     slice at ph.origin: consume and clear its ring-buffer cells lag by lag, set the bit of
//     every lag it spikes in, store the multimeter samples due (store_sample at lag
//     next_sample, then every mm_int lags) and write the state back. The parameters are the
//     first values (Params) of the ParamSet its host half's pre_run_hook made.
// The slice kernel dispatches on the model id (a compile-time id when a launch holds one
// model), so every model is inlined into the fused kernel. Included by ng_kernels.hip after
// the ring-buffer cell and sampling helpers it uses.
#pragma once

namespace nestgpu
{

template < int ID >
struct DeviceNode;

// The first N values of a parameter set and its refractory steps, in registers. Neurons of a
// wave that share one set (uniform: its index p0) read it through scalar loads, which the
// scalar cache serves for all waves of a CU; others read their own (index pi).
template < int N >
struct ParamValues
{
  double p[ N > 0 ? N : 1 ];
  int32_t refractory_counts;
  __device__ __forceinline__ static ParamValues
  load( const ParamSet* psets, bool uniform, uint32_t p0, uint32_t pi )
  {
    ParamValues v;
    if ( uniform )
      v.read( ( (cptr< const ParamSet >)psets )[ p0 ] );
    else
      v.read( glob( psets )[ pi ] );
    return v;
  }
  template < class PS >
  __device__ __forceinline__ void
  read( PS& ps )
  {
#pragma unroll
    for ( int q = 0; q < N; ++q )
      p[ q ] = ps.p[ q ];
    refractory_counts = ps.refractory_counts;
  }
};

// The device model ids, in the order ModelManager registers them: a model with a DeviceNode
// specialization joins the slice kernel by its entry here. WIDE marks models whose launches
// run one workgroup per CU with up to 256 VGPRs; the others are held to 128 VGPRs, so that
// two workgroups share a CU, spilling what does not fit. BLOCK marks models whose neurons are
// updated by all threads of the workgroup together (update_block) instead of one thread each.
#define NG_DEVICE_MODELS( X ) X( M_IAF_PSC_DELTA ) X( M_IAF_PSC_EXP ) X( M_AEIF_COND_EXP ) X( M_IAF_PSC_ALPHA )
constexpr int N_DEVICE_MODELS = 4;
constexpr int ALL_MODELS = ( 1 << N_DEVICE_MODELS ) - 1;
static_assert( ALL_MODELS < MASK_STDP, "model bits must stay below the stdp bit" );

// the one model id of a launch mask with a single model bit, else -1
template < int MASK >
__device__ constexpr int
single_model()
{
  return ( MASK & ( MASK - 1 ) ) == 0 ? __builtin_ctz( MASK ) : -1;
}

// Runs step( lag, in0, in1 ) over the lags of a slice part with the neuron's input of each
// channel, read and cleared, and collects the lags for which it returns true (a spike) in bits.
// The lags are a serial chain: steps select instead of branching.
// Lags whose cells are all in the LDS window take a loop of one lag per turn with the next lag's
// input in flight; a body unrolled over LB lags was 5 KB of code fetched anew in every launch,
// 890 cycles per lag against 540 (1,777 iaf_psc_exp, slices of ten steps, 16.5 -> 13.9 us with the
// drive in waves of its own). Cells in HBM are read LU lags at a time, so that their loads
// overlap. The words of bits are selected, not indexed: indexed, they lived in scratch memory, 48
// bytes per thread written in every launch and read back before the spike lists (20 ms passes of
// 1,777 iaf_psc_exp 368 -> 349 us, 60 ms of 5,000 iaf_psc_delta 934 -> 859, 200 ms of 100,000
// iaf_psc_exp 21.4 -> 21.0 ms). The words take registers during the update, so the global delivery
// kernels of 80 registers read half as many lags at a time (300,000 iaf_psc_delta 390 -> 382 us
// per slice; 280,000 iaf_psc_alpha 5 % slower, all its variants spilled more).
template < int LU, int NCH, class CELLS, class STEP >
__device__ __forceinline__ void
for_lags( const CELLS& C, const SlicePhase& ph, uint32_t local, uint64_t* bits, STEP&& step )
{
  if ( C.covers( ph.from, ph.to ) )
  {
    lptr< double > p = C.lds + C.win_index( ph.from, 0, local );
    double in0 = p[ 0 ], in1 = NCH > 1 ? p[ C.tb ] : 0.0;
    uint64_t acc = 0;  // spikes in lags [64 w, 64 w + 64) of the current lag
#pragma unroll 1
    for ( int lag = ph.from; lag < ph.to; ++lag )
    {
      const double w0 = in0, w1 = in1;
      p[ 0 ] = 0.0;
      if ( NCH > 1 )
        p[ C.tb ] = 0.0;
      p += C.nct;
      if ( lag + 1 < ph.to )
      {
        in0 = p[ 0 ];
        if ( NCH > 1 )
          in1 = p[ C.tb ];
      }
      acc |= step( lag, w0, w1 ) ? 1ull << ( lag & 63 ) : 0ull;
      if ( ( lag & 63 ) == 63 or lag + 1 == ph.to )
      {
#pragma unroll
        for ( int w = 0; w < 4; ++w )
          bits[ w ] |= ( lag >> 6 ) == w ? acc : 0ull;
        acc = 0;
      }
    }
    return;
  }
  for ( int l0 = ph.from; l0 < ph.to; l0 += LU )
  {
    double w0[ LU ], w1[ LU ];
    uint64_t acc = 0;  // spikes in lags [l0, l0 + LU)
#pragma unroll
    for ( int q = 0; q < LU; ++q )
      if ( l0 + q < ph.to )
      {
        w0[ q ] = C.get( l0 + q, 0, local );
        w1[ q ] = NCH > 1 ? C.get( l0 + q, 1, local ) : 0.0;
      }
#pragma unroll
    for ( int q = 0; q < LU; ++q )
      if ( l0 + q < ph.to )
      {
        C.put( l0 + q, 0, local, 0.0 );
        if ( NCH > 1 )
          C.put( l0 + q, 1, local, 0.0 );
        acc |= step( l0 + q, w0[ q ], w1[ q ] ) ? 1ull << q : 0ull;
      }
#pragma unroll
    for ( int w = 0; w < 4; ++w )
    {
      const int at = l0 - 64 * w;  // the group may cross a word
      bits[ w ] |= at >= 64 or at <= -64 ? 0ull : at >= 0 ? acc << at : acc >> -at;
    }
  }
}

template <>
struct DeviceNode< M_IAF_PSC_DELTA >
{
  static constexpr bool WIDE = false;
  static constexpr bool BLOCK = false;
  static constexpr int GLOBAL_WAVES = 6;
  // iaf_psc_delta::handle( SpikeEvent& ) (iaf_psc_delta.cpp:332-341): one channel, the weight
  __device__ __forceinline__ static void
  receive( double w, uint32_t& ch, double& v )
  {
    ch = 0;
    v = w;
  }
  struct State
  {
    double y3, refr_buf;  // refr_spikes_buffer_
    int32_t r;
  };
  __device__ __forceinline__ static State
  load( const NetDev& d, uint32_t dev )
  {
    return { glob( d.v[ 0 ] )[ dev ], glob( d.v[ 1 ] )[ dev ], glob( d.r )[ dev ] };
  }
  using Params = ParamValues< 9 >;
  template < class CELLS >
  __device__ __forceinline__ static void
  update( const NetDev& d, const Params& ps, const State& st, uint32_t dev, uint32_t local, const CELLS& C,
    const SlicePhase& ph, uint64_t* bits, uint32_t mcol, int next_sample )
  {
    // models/iaf_psc_delta.cpp:272-331
    const double P30 = ps.p[ 0 ], P33 = ps.p[ 1 ], y0I = ps.p[ 2 ], V_th = ps.p[ 3 ], V_reset = ps.p[ 4 ],
                 V_min = ps.p[ 5 ];
    const bool refr_input = ps.p[ 6 ] != 0.0;
    const double h = ps.p[ 7 ], tau_m = ps.p[ 8 ];
    double y3 = st.y3;
    double refr_buf = refr_input ? st.refr_buf : 0.0;
    int32_t r = st.r;
    for_lags< CELLS::WINDOW ? LB : 4, 1 >( C, ph, local, bits,
      [ & ]( int lag, double in, double )
      {
        const bool active = r == 0;
        double y = P30 * y0I + P33 * y3 + in;
        if ( refr_input )
        {
          if ( not active )
            refr_buf += in * ng_exp( -static_cast< double >( r ) * h / tau_m );
          else if ( refr_buf != 0.0 )
          {
            y += refr_buf;
            refr_buf = 0.0;
          }
        }
        y = ( y < V_min ? V_min : y );
        y3 = active ? y : y3;
        r -= active ? 0 : 1;
        const bool spike = y3 >= V_th;
        r = spike ? ps.refractory_counts : r;
        y3 = spike ? V_reset : y3;
        if ( lag == next_sample )
        {
          store_sample( d, mcol, ph.origin + lag + 1, y3, 0.0, 0.0, 0.0 );
          next_sample += d.mm_int;
        }
        return spike;
      } );
    glob( d.v[ 0 ] )[ dev ] = y3;
    if ( refr_input )
      glob( d.v[ 1 ] )[ dev ] = refr_buf;
    glob( d.r )[ dev ] = r;
  }
};

template <>
struct DeviceNode< M_IAF_PSC_EXP >
{
  static constexpr bool WIDE = false;
  static constexpr bool BLOCK = false;
  static constexpr int GLOBAL_WAVES = 4;
  // iaf_psc_exp::handle( SpikeEvent& ) (iaf_psc_exp.cpp:351-362): positive weights to the
  // excitatory channel (1), others to the inhibitory one (0), signed
  __device__ __forceinline__ static void
  receive( double w, uint32_t& ch, double& v )
  {
    ch = w > 0 ? 1u : 0u;
    v = w;
  }
  struct State
  {
    double V, iex, iin;
    int32_t r;
  };
  __device__ __forceinline__ static State
  load( const NetDev& d, uint32_t dev )
  {
    return { glob( d.v[ 0 ] )[ dev ], glob( d.v[ 1 ] )[ dev ], glob( d.v[ 2 ] )[ dev ], glob( d.r )[ dev ] };
  }
  using Params = ParamValues< 10 >;
  template < class CELLS >
  __device__ __forceinline__ static void
  update( const NetDev& d, const Params& ps, const State& st, uint32_t dev, uint32_t local, const CELLS& C,
    const SlicePhase& ph, uint64_t* bits, uint32_t mcol, int next_sample )
  {
    // models/iaf_psc_exp.cpp:288-349 (delta = 0: deterministic threshold)
    const double P22 = ps.p[ 0 ], P21ex = ps.p[ 1 ], P21in = ps.p[ 2 ], P20 = ps.p[ 3 ], P11ex = ps.p[ 4 ],
                 P11in = ps.p[ 5 ], IeI0 = ps.p[ 6 ], Theta = ps.p[ 7 ], V_reset = ps.p[ 8 ], exI1 = ps.p[ 9 ];
    double V = st.V, iex = st.iex, iin = st.iin;
    int32_t r = st.r;
    for_lags< LB, 2 >( C, ph, local, bits,
      [ & ]( int lag, double w_in, double w_ex )
      {
        const bool active = r == 0;
        const double Vn = V * P22 + iex * P21ex + iin * P21in + IeI0 * P20;
        V = active ? Vn : V;
        r -= active ? 0 : 1;
        iex *= P11ex;
        iin *= P11in;
        iex += exI1;
        iex += w_ex;
        iin += w_in;
        const bool spike = V >= Theta;
        r = spike ? ps.refractory_counts : r;
        V = spike ? V_reset : V;
        if ( lag == next_sample )
        {
          store_sample( d, mcol, ph.origin + lag + 1, V, iex, iin, 0.0 );
          next_sample += d.mm_int;
        }
        return spike;
      } );
    glob( d.v[ 0 ] )[ dev ] = V;
    glob( d.v[ 1 ] )[ dev ] = iex;
    glob( d.v[ 2 ] )[ dev ] = iin;
    glob( d.r )[ dev ] = r;
  }
};

template <>
struct DeviceNode< M_AEIF_COND_EXP >
{
  static constexpr bool WIDE = false;
  static constexpr bool BLOCK = true;
  static constexpr int GLOBAL_WAVES = 4;
  static constexpr double LONG_DT = 3.0;  // "close": within this many Delta_T below V_th
  // aeif_cond_exp::handle( SpikeEvent& ) (aeif_cond_exp.cpp:526-541): positive weights to the
  // excitatory conductance (0), others negated to the inhibitory one (1)
  __device__ __forceinline__ static void
  receive( double w, uint32_t& ch, double& v )
  {
    if ( w > 0.0 )
    {
      ch = 0;
      v = w;
    }
    else
    {
      ch = 1;
      v = -w;
    }
  }
  // A neuron that is close to its threshold at the start of a slice will probably take many
  // steps in it.
  __device__ __forceinline__ static bool
  long_update( const NetDev& d, uint32_t dev )
  {
    gref< const ParamSet > ps = glob( d.psets )[ glob( d.pidx )[ dev ] ];
    return glob( d.r )[ dev ] == 0 and glob( d.v[ 0 ] )[ dev ] > ps.p[ 11 ] - LONG_DT * ps.p[ 7 ];
  }
  // Updates the block's aeif_cond_exp neurons with every thread of the workgroup, four lanes
  // per neuron (ng_aeif.h). Neurons need very different numbers of steps (a slice of 15 steps
  // takes 16 attempted steps on average and up to 166), so a quad that finishes its neuron
  // takes the next one of the block from the counter *next (which starts at the number of
  // quads) instead of waiting for the slowest lane of its wave. order: the order in which a block
  // with more neurons than quads takes them (likely long updates first), or null. spk: spike bits of every
  // neuron, [local][words of 64 lags]. Which quad integrates a neuron does not change its
  // operations. Measured on the MI355X (one lane per neuron and a wave per
  // 64 neurons -> this): 6,000 neurons in blocks of 32, slices of 15 steps, 520 -> 325 us per
  // slice; 48 networks in blocks of 512, 1,670 -> 1,050 us. What remains is the chain of the
  // slowest neuron, 2.5 us per attempt.
  template < class CELLS, bool SINGLE >
  __device__ __forceinline__ static void
  update_block( const NetDev& d, uint32_t dev0, uint32_t nb, const CELLS& C, const SlicePhase& ph,
    lptr< uint32_t > next, lptr< unsigned long long > spk, lptr< const uint16_t > order )
  {
    // models/aeif_cond_exp.cpp:443-523
    const int c = static_cast< int >( threadIdx.x & 3u );
    const uint32_t nw = ( static_cast< uint32_t >( d.min_delay ) + 63u ) >> 6;
    const bool channel = c == 1 or c == 2;
    const uint32_t ch = static_cast< uint32_t >( c - 1 );
    gptr< double > const vc = glob( c == 0 ? d.v[ 0 ] : c == 1 ? d.v[ 1 ] : c == 2 ? d.v[ 2 ] : d.v[ 3 ] );
    AeifLane A;
    A.c = c;
    uint32_t pset = NONE;  // parameter set in A
    double b_adapt = 0, V_peak_eff = 0, hstep = 0, I_reset = 0;
    int32_t refractory_counts = 0;
    double y = 0, h = 0, tt = 0, in = 0, I_spk = 0;
    int32_t r = 0;
    int lag = ph.to, guard = 0, next_sample = ph.to;
    uint32_t mcol = NONE;
    unsigned long long bits = 0;  // spikes in lags [64 c, 64 c + 64)
    auto at = [ & ]( uint32_t i ) { return i < nb and order ? static_cast< uint32_t >( order[ i ] ) : i; };
    uint32_t local = at( threadIdx.x >> 2 ), dev = 0;
    auto take = [ & ]
    {
      uint32_t n = 0;
      if ( c == 0 )
        n = __hip_atomic_fetch_add( next, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP );
      local = at( quad_bcast< 0 >( n ) );
    };
    bool have = false;
    // Every iteration is one attempted step of the quad's neuron, preceded by the exchange of
    // a finished neuron for the next one. More than AEIF_MAX_STEPS accepted steps within one
    // time step stop the neuron's lag and raise ERR_AEIF_STEPS, which fails the run (the
    // oracle stops with the same limit). A rejected attempt shrinks h by a factor of at most
    // 0.9 * 1.1^(-1/5) < 0.89 and is accepted once t + h rounds to t or, in a lag's first step
    // (t = 0), once h underflows, after fewer than 6,400 attempts; so every quad finishes.
    for ( ;; )
    {
      if ( lag >= ph.to )
      {
        if ( have )
        {
          vc[ dev ] = y;
          if ( c == 0 )
            glob( d.v[ 4 ] )[ dev ] = h;
          if ( c == 1 )
            glob( d.r )[ dev ] = r;
          if ( static_cast< uint32_t >( c ) < nw )
            spk[ local * nw + c ] = bits;
          take();
        }
        if ( not SINGLE )
          while ( local < nb and glob( d.model )[ dev0 + local ] != M_AEIF_COND_EXP )
            take();
        if ( local >= nb )
          break;
        have = true;
        dev = dev0 + local;
        y = vc[ dev ];
        h = glob( d.v[ 4 ] )[ dev ];
        r = glob( d.r )[ dev ];
        lag = ph.from;
        in = channel ? C.get( lag, ch, local ) : 0.0;
        const uint32_t pi = glob( d.pidx )[ dev ];
        if ( d.mm_int > 0 )
        {
          mcol = glob( d.mm_col )[ dev ];
          next_sample = mcol != NONE ? first_sample_lag( d, ph.origin, ph.from, ph.to ) : ph.to;
        }
        if ( pi != pset )
        {
          pset = pi;
          gref< const ParamSet > ps = glob( d.psets )[ pi ];
          A.V_peak = ps.p[ 0 ];
          A.V_reset = ps.p[ 1 ];
          A.Delta_T = ps.p[ 7 ];
          A.V_th = ps.p[ 11 ];
          A.I_e = ps.p[ 14 ];
          A.tol = ps.p[ 15 ];
          A.gD = ps.p[ 2 ] * ps.p[ 7 ];
          A.E = ps.p[ c == 1 ? 4 : c == 2 ? 5 : 6 ];
          A.m = c == 0 ? -ps.p[ 2 ] : ps.p[ 9 ];
          A.zero_fits = channel or ( c == 3 and ps.p[ 9 ] == 0.0 );
          A.den = ps.p[ c == 0 ? 3 : c == 1 ? 12 : c == 2 ? 13 : 8 ];
          A.r_den = ng_recip( A.den );
          A.r_Delta_T = ng_recip( A.Delta_T );
          b_adapt = ps.p[ 10 ];
          V_peak_eff = ps.p[ 16 ];
          hstep = ps.p[ 17 ];
          refractory_counts = ps.refractory_counts;
          I_reset = aeif_spike_current< false >( A, aeif_V( A, false, A.V_reset ) );
        }
        tt = 0.0;
        guard = 0;
        bits = 0;
        I_spk = aeif_spike_current< false >( A, aeif_V( A, false, quad_bcast< 0 >( y ) ) );
      }
      const bool refr = r > 0;
      const double dt = hstep - tt;
      const bool final_step = h > dt;
      const double h_old = final_step ? dt : h;
      // the spike current at the step's start is the one the last step ended with, or that of the
      // reset potential (inputs change the conductances only)
      double y1, yerr, yp, I_end;
      bool plain = __any( d.plain_div or not aeif_fast_state( A, y ) );
      if ( not plain )
      {
        y1 = aeif_step< true >( A, refr, y, h_old, I_spk, yerr, yp, I_end );
        plain = __any( not aeif_finite( y1, yp ) );
      }
      if ( plain )
        y1 = aeif_step< false >( A, refr, y, h_old, I_spk, yerr, yp, I_end );
      const double tn = final_step ? hstep : tt + h_old;
      double h_new = h_old;
      const int st = aeif_yp_hadjust( A.tol, yerr, yp, &h_new );
      h = h_new;
      if ( st < 0 )
      {
        if ( fabs( h_new ) < fabs( h_old ) and tn + h_new != tn )
          continue;  // again from the same state
        h = h_old;
      }
      y = y1;
      I_spk = I_end;
      tt = tn;
      ++guard;
      const double V = quad_bcast< 0 >( y ), w = quad_bcast< 3 >( y );
      if ( V < -1e3 or w < -1e6 or w > 1e6 )
      {
        if ( c == 0 )
          g_or( &d.counters[ 0 ], ERR_AEIF_INSTABILITY );
        tt = hstep;
      }
      else if ( r > 0 )
      {
        y = c == 0 ? A.V_reset : y;
        I_spk = I_reset;
      }
      else if ( V >= V_peak_eff )
      {
        y = c == 0 ? A.V_reset : c == 3 ? y + b_adapt : y;
        I_spk = I_reset;
        r = refractory_counts > 0 ? refractory_counts + 1 : 0;
        if ( ( lag >> 6 ) == c )
        {
          const unsigned long long bit = 1ull << ( lag & 63 );
          if ( bits & bit )
            g_or( &d.counters[ 0 ], ERR_AEIF_DOUBLE_SPIKE );
          bits |= bit;
        }
      }
      if ( tt < hstep and guard >= AEIF_MAX_STEPS )
      {
        if ( c == 0 )
          g_or( &d.counters[ 0 ], ERR_AEIF_STEPS );
        tt = hstep;
      }
      if ( not( tt < hstep ) )
      {
        if ( r > 0 )
          --r;
        if ( channel )
        {
          y += in;
          C.put( lag, ch, local, 0.0 );
        }
        if ( lag == next_sample )
        {
          store_sample_field( d, mcol, ph.origin + lag + 1, c, y );
          next_sample += d.mm_int;
        }
        ++lag;
        tt = 0.0;
        guard = 0;
        if ( channel and lag < ph.to )
          in = C.get( lag, ch, local );  // arrives while the lag is integrated
      }
    }
  }
  // aeif_cond_exp neurons are loaded and updated by update_block
  struct State
  {
  };
  __device__ __forceinline__ static State
  load( const NetDev&, uint32_t )
  {
    return {};
  }
  using Params = ParamValues< 0 >;
  template < class CELLS >
  __device__ __forceinline__ static void
  update( const NetDev&, const Params&, const State&, uint32_t, uint32_t, const CELLS&, const SlicePhase&, uint64_t*,
    uint32_t, int )
  {
  }
};

template <>
struct DeviceNode< M_IAF_PSC_ALPHA >
{
  static constexpr bool WIDE = false;
  static constexpr bool BLOCK = false;
  static constexpr int GLOBAL_WAVES = 6;
  // iaf_psc_alpha::handle( SpikeEvent& ) (iaf_psc_alpha.cpp:373-383): positive weights to
  // the excitatory channel (1), others to the inhibitory one (0), signed
  __device__ __forceinline__ static void
  receive( double w, uint32_t& ch, double& v )
  {
    ch = w > 0 ? 1u : 0u;
    v = w;
  }
  struct State
  {
    double V, iex, iin, diex, diin;
    int32_t r;
  };
  __device__ __forceinline__ static State
  load( const NetDev& d, uint32_t dev )
  {
    return { glob( d.v[ 0 ] )[ dev ], glob( d.v[ 1 ] )[ dev ], glob( d.v[ 2 ] )[ dev ], glob( d.v[ 3 ] )[ dev ],
      glob( d.v[ 4 ] )[ dev ], glob( d.r )[ dev ] };
  }
  using Params = ParamValues< 16 >;
  template < class CELLS >
  __device__ __forceinline__ static void
  update( const NetDev& d, const Params& ps, const State& st, uint32_t dev, uint32_t local, const CELLS& C,
    const SlicePhase& ph, uint64_t* bits, uint32_t mcol, int next_sample )
  {
    // models/iaf_psc_alpha.cpp:305-370 (the current input y0 is zero: no current sources)
    const double P30 = ps.p[ 0 ], y0I = ps.p[ 1 ], P31ex = ps.p[ 2 ], P32ex = ps.p[ 3 ], P31in = ps.p[ 4 ],
                 P32in = ps.p[ 5 ], expm1_tau_m = ps.p[ 6 ], P21ex = ps.p[ 7 ], P11ex = ps.p[ 8 ],
                 P21in = ps.p[ 9 ], P11in = ps.p[ 10 ], EPSCInit = ps.p[ 11 ], IPSCInit = ps.p[ 12 ],
                 Theta = ps.p[ 13 ], V_reset = ps.p[ 14 ], LowerBound = ps.p[ 15 ];
    double V = st.V, iex = st.iex, iin = st.iin, diex = st.diex, diin = st.diin;
    int32_t r = st.r;
    // its 16 propagators and 5 state variables leave fewer registers for cells of HBM than the
    // other iaf models
    for_lags< CELLS::WINDOW ? 4 : 2, 2 >( C, ph, local, bits,
      [ & ]( int lag, double w_in, double w_ex )
      {
        const bool active = r == 0;
        const double Vn = P30 * y0I + P31ex * diex + P32ex * iex + P31in * diin + P32in * iin + expm1_tau_m * V + V;
        V = active ? ( Vn < LowerBound ? LowerBound : Vn ) : V;
        r -= active ? 0 : 1;
        iex = P21ex * diex + P11ex * iex;  // P22_ex = P11_ex
        diex *= P11ex;
        diex += EPSCInit * w_ex;
        iin = P21in * diin + P11in * iin;
        diin *= P11in;
        diin += IPSCInit * w_in;
        const bool spike = V >= Theta;
        r = spike ? ps.refractory_counts : r;
        V = spike ? V_reset : V;
        if ( lag == next_sample )
        {
          store_sample( d, mcol, ph.origin + lag + 1, V, iex, iin, 0.0 );
          next_sample += d.mm_int;
        }
        return spike;
      } );
    glob( d.v[ 0 ] )[ dev ] = V;
    glob( d.v[ 1 ] )[ dev ] = iex;
    glob( d.v[ 2 ] )[ dev ] = iin;
    glob( d.v[ 3 ] )[ dev ] = diex;
    glob( d.v[ 4 ] )[ dev ] = diin;
    glob( d.r )[ dev ] = r;
  }
};

// models whose update needs the wide register budget
#define NG_WIDE( ID ) | ( DeviceNode< ( ID ) >::WIDE ? ( 1 << ( ID ) ) : 0 )
constexpr int WIDE_MODELS = 0 NG_DEVICE_MODELS( NG_WIDE );
#undef NG_WIDE
// Waves per SIMD of the global delivery kernel of a launch mask: GLOBAL_WAVES of its model. That
// kernel serves networks of more than 512 blocks, whose workgroups mostly wait for run table
// entries and ring cells; at 6 (three workgroups per CU, 80 VGPRs) all blocks of up to 393,000
// neurons are resident at once. Measured per slice with rounds of 1,024 events, 4 against 6 waves
// (rounds of 2,048 at 4 waves before): 300,000 iaf_psc_delta neurons 592 / 390 us (629), 450,000
// - / 986 (1,035); iaf_psc_alpha 300,000 - / 251 (385), 450,000 - / 592 (613); iaf_psc_exp, which
// spills 164 registers at 6, 300,000 195 / 174 (208), 450,000 297 / 353 (325).
template < int MASK >
__host__ __device__ constexpr int
global_waves()
{
  int waves = 4;  // several models
#define NG_WAVES( ID )               \
  if ( MASK == ( 1 << ( ID ) ) )   \
    waves = DeviceNode< ( ID ) >::GLOBAL_WAVES;
  NG_DEVICE_MODELS( NG_WAVES )
#undef NG_WAVES
  return waves;
}
// models updated by the whole workgroup
#define NG_BLOCK( ID ) | ( DeviceNode< ( ID ) >::BLOCK ? ( 1 << ( ID ) ) : 0 )
constexpr int BLOCK_MODELS = 0 NG_DEVICE_MODELS( NG_BLOCK );
#undef NG_BLOCK
static_assert( BLOCK_MODELS == 1 << M_AEIF_COND_EXP, "the slice kernel calls this model's update_block" );

// handle( SpikeEvent& ) of model m
__device__ __forceinline__ void
node_receive( int m, double w, uint32_t& ch, double& v )
{
  ch = 0;
  v = w;
#define NG_RECEIVE( ID )                           \
  if ( m == ( ID ) )                               \
  {                                                \
    DeviceNode< ( ID ) >::receive( w, ch, v );     \
    return;                                        \
  }
  NG_DEVICE_MODELS( NG_RECEIVE )
#undef NG_RECEIVE
}

}  // namespace nestgpu
