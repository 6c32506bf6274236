// ng_kernels.hip -- gfx950 kernel for one min_delay slice of NEST's simulation step.
//
// One workgroup owns a block of `tb` consecutive targets (device index = receive-order
// position) and, for slice s of a chunk:
//   1. delivers the previous slice's spikes to its targets (EventDeliveryManager::
//      deliver_events_, nestkernel/event_delivery_manager.cpp:599-776; Connector::send,
//      connector_base.h:399-428; RingBuffer::add_value, ring_buffer.h:157-161,405-408):
//      it walks the receive-order spike list, reads its own run of each spiking source's
//      out-row, and adds every weight into the target's ring-buffer cell;
//   2. updates its neurons over [from, to) (Node::update of iaf_psc_delta, iaf_psc_exp,
//      aeif_cond_exp) including the spike_generator drive of that slice;
//   3. appends its spikes, in receive order, to its block list for the next slice.
//
// Window delivery: the slots a slice can touch through recurrent synapses are the
// max_delay slots starting at the slice origin (lag + delay - min_delay < max_delay), and
// the update reads the first min_delay of them. In window mode the workgroup copies the wn
// consecutive slots [wa, wa + wn) of those that receive the most events into LDS,
// accumulates there and writes them back once, so the read-modify-write of most synaptic
// events is an LDS operation; cells outside the window are updated in HBM. Global mode
// updates every cell in HBM.
//
// Determinism: NEST adds into one ring-buffer cell in the order (delivery batch, receive
// order of the spike, position in the connector run). A workgroup takes events in that key
// order in rounds of R; each round is bucketed by target, and by slot where a block has few
// targets (LDS counters give every event a place in its bucket), every event finds its rank in
// the bucket ordered by (cell, key), and the first event of each cell's run adds the run in key
// order. No result depends on thread timing or atomics order.
// Built with -ffp-contract=off: every multiply and add rounds as in the reference.

#include <hip/hip_runtime.h>

#include "ng_aeif.h"
#include "ng_device.h"
#include "ng_engine.h"

namespace nestgpu
{

constexpr int IDX_BITS = 11;  // bucket key = slot-channel << 11 | round index: sorted keys group
                              // a bucket's events by cell, in key order within each cell

// Tile shape: chunks and rounds are the same in both variants. With its ring-buffer window, two
// window workgroups fit in the 160 KB of LDS of a CU; global delivery runs two or three
// (global_waves).
template < bool WIN >
struct Tile
{
  static constexpr int BS = static_cast< int >( MAX_TB );  // threads per workgroup
  static constexpr int SPT = 2;                // spikes per thread per chunk
  static constexpr int CH = SPT * BS;          // spikes per chunk
  static constexpr int RQ = 2;                 // events per thread per round
  static constexpr int R = RQ * BS;            // events per round
  static constexpr uint32_t WINDOW = WIN ? WIN_CAP : 1;
  static constexpr uint32_t PMAX = WIN ? PMAX_WIN : PMAX_GLOB;
};
constexpr uint32_t NONE = 0xffffffffu;

// HBM views of the instance's arrays. The pointers in the instance record are generic, and
// generic (FLAT) accesses are counted by the LDS wait counter too: every barrier and every
// LDS read would then wait for all HBM loads in flight. Accessing HBM through global-space
// pointers keeps those loads on the vector-memory counter, so they overlap the LDS phases.
template < class T >
using gptr = __attribute__( ( address_space( 1 ) ) ) T*;
template < class T >
using gref = __attribute__( ( address_space( 1 ) ) ) T&;
// memory that no kernel writes while this one runs: uniform addresses load into scalar registers
template < class T >
using cptr = __attribute__( ( address_space( 4 ) ) ) T*;
template < class T >
using lptr = __attribute__( ( address_space( 3 ) ) ) T*;
template < class T >
__device__ inline gptr< T >
glob( T* p )
{
  return ( gptr< T > )p;
}

// device-scope relaxed atomics on HBM counters (what atomicAdd / atomicOr do, without FLAT)
__device__ inline unsigned long long
g_add( unsigned long long* p, unsigned long long v )
{
  return __hip_atomic_fetch_add( glob( p ), v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT );
}
__device__ inline void
g_add( uint32_t* p, uint32_t v )
{
  __hip_atomic_fetch_add( glob( p ), v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT );
}
__device__ inline void
g_or( unsigned long long* p, unsigned long long v )
{
  __hip_atomic_fetch_or( glob( p ), v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT );
}

// The block's ring buffer as a buffer resource: an access at an offset past its end
// (NO_CELL) moves no data (loads return 0, stores are dropped), so every lane can issue the
// same loads and stores whether or not its event has an HBM cell.
constexpr uint32_t NO_CELL = 0x80000000u;
using v2u = __attribute__( ( ext_vector_type( 2 ) ) ) uint32_t;
__device__ inline double
cell_load( __amdgpu_buffer_rsrc_t r, uint32_t byte_off )
{
  return __builtin_bit_cast( double, __builtin_amdgcn_raw_buffer_load_b64( r, byte_off, 0, 0 ) );
}
__device__ inline void
cell_store( __amdgpu_buffer_rsrc_t r, uint32_t byte_off, double v )
{
  __builtin_amdgcn_raw_buffer_store_b64( __builtin_bit_cast( v2u, v ), r, byte_off, 0, 0 );
}

__device__ inline SynRec
load_rec( gptr< const SynRec > p )
{
  SynRec r;
  r.w_lo = p->w_lo;
  r.w_hi = p->w_hi;
  r.word = p->word;
  return r;
}
// four consecutive entries of a spike list with n entries left, as one load where they are in it
struct Entries
{
  uint32_t x[ 4 ];
};
__device__ inline Entries
load_entries( gptr< const uint32_t > p, uint32_t n )
{
  using v4u = __attribute__( ( ext_vector_type( 4 ), aligned( 4 ) ) ) uint32_t;
  Entries e {};
  if ( n >= 4 )
  {
    const v4u v = *( gptr< const v4u > )p;
#pragma unroll
    for ( int j = 0; j < 4; ++j )
      e.x[ j ] = v[ j ];
  }
  else
#pragma unroll
    for ( uint32_t j = 0; j < 3; ++j )
      e.x[ j ] = j < n ? p[ j ] : 0u;
  return e;
}
// longest spike list that one thread copies. Its turns of four entries are trips to memory of one
// thread, looking the spikes up is one trip for all: 1,000 iaf_psc_exp in blocks of 512, slices of
// 15 steps with 142 spikes per list, 43.0 us copied and 37.0 us looked up; 8,000 in blocks of 64
// with 3 (up to 13) per list 17.3 and 18.0 us.
constexpr uint32_t LIST_COPY = 16;
constexpr int LB = 8;  // lags of ring-buffer input loaded together in the update
static_assert( Tile< false >::R <= ( 1 << IDX_BITS ) and Tile< true >::R <= ( 1 << IDX_BITS ),
  "round index must fit the bucket key" );
static_assert( ( PMAX_GLOB + 1 ) * sizeof( uint32_t ) <= WIN_CAP * sizeof( double ),
  "the window must hold the block prefix of an instance without a window" );

template < bool WIN >
struct SliceLds
{
  static_assert( Tile< WIN >::CH <= Tile< WIN >::R, "a chunk's spikes must fit the sorted keys" );
  using T = Tile< WIN >;
  double win[ T::WINDOW ];  // ring-buffer window [slot - origin][channel][tb]
  unsigned long long log_base;
  uint32_t sh[ T::BS / 64 ];
  uint32_t cnt_base;
  uint32_t pool_next;  // next neuron of a block-wide update
  union
  {
    struct  // delivery
    {
      double sw[ T::R ];             // event values in sorted order
      uint32_t pref[ T::PMAX + 1 ];  // prefix of per-block spike counts
      uint32_t c_g0[ T::CH ];        // first synapse of each chunk spike's run
      uint32_t c_off[ T::CH + 1 ];   // exclusive prefix of run lengths
      uint32_t bk[ T::R ];           // event keys (slot-channel << 11 | round index), by bucket
      uint32_t sk[ T::R ];           // event keys in sorted order; before the rounds of a
                                     // slice of one chunk its spikes
      uint32_t bcnt[ 2 ][ T::BS ];   // events per bucket, alternating between rounds
      alignas( 4 ) uint16_t bst[ T::BS + 2 ];  // bucket starts
      uint16_t c_idx[ T::BS ];       // spike of every 2^sh-th event of the chunk
      uint8_t c_lag[ T::CH ];
    };
    struct  // block-wide update
    {
      unsigned long long spk_bits[ MAX_TB * 4 ];  // spike bits per neuron, 64 lags per word
      uint16_t order[ MAX_TB ];                   // neurons in the order they are taken
    };
  };
};

static_assert( sizeof( SliceLds< true > ) <= 80 * 1024, "two window workgroups share the 160 KB of a CU" );

// XCD-aware block mapping: workgroups are dispatched round-robin over 8 XCDs; give each
// XCD a contiguous range of blocks so neighbouring blocks share its L2. A launch of several
// instances keeps the dispatch order instead: the host puts the instances with the longest
// workgroups first, which then start on different CUs of every XCD, and lighter ones fill up
// (48 networks, half of them aeif_cond_exp, 380 workgroups: 12.8 -> 10.5 ms per 10 slices).
__device__ inline uint32_t
xcd_block( uint32_t w, uint32_t total )
{
  const uint32_t x = w & 7u;
  uint32_t base = 0;
  for ( uint32_t q = 0; q < x; ++q )
    base += ( total - q + 7u ) / 8u;
  return base + ( w >> 3 );
}

__device__ inline uint32_t
upper_bound_u32( const uint32_t* a, uint32_t n, uint32_t v )
{
  uint32_t lo = 0, hi = n;
  while ( lo < hi )
  {
    const uint32_t mid = ( lo + hi ) >> 1;
    if ( a[ mid ] <= v )
      lo = mid + 1;
    else
      hi = mid;
  }
  return lo;
}

// number of records of a delay-ordered run [g0, g0 + len) whose delay offset is below t
__device__ inline uint32_t
run_split( gptr< const SynRec > syn, uint32_t g0, uint32_t len, int t )
{
  if ( t <= 0 )
    return 0;
  uint32_t lo = 0, hi = len;
  while ( lo < hi )
  {
    const uint32_t mid = ( lo + hi ) >> 1;
    if ( static_cast< int >( ( syn[ g0 + mid ].word >> 16 ) & DELAY_MASK ) < t )
      lo = mid + 1;
    else
      hi = mid;
  }
  return lo;
}

// inclusive scan over the 64 lanes of a wave with DPP moves: Hillis-Steele inside each row
// of 16 lanes (row_shr 1, 2, 4, 8; lanes shifted in from outside the row read 0), then the
// last lane of row 0 and 2 is added to row 1 and 3 (row_bcast:15), then the last lane of
// row 1 to rows 2 and 3 (row_bcast:31)
__device__ inline uint32_t
wave_incl_scan( uint32_t x )
{
  x += static_cast< uint32_t >( __builtin_amdgcn_update_dpp( 0, static_cast< int >( x ), 0x111, 0xf, 0xf, false ) );
  x += static_cast< uint32_t >( __builtin_amdgcn_update_dpp( 0, static_cast< int >( x ), 0x112, 0xf, 0xf, false ) );
  x += static_cast< uint32_t >( __builtin_amdgcn_update_dpp( 0, static_cast< int >( x ), 0x114, 0xf, 0xf, false ) );
  x += static_cast< uint32_t >( __builtin_amdgcn_update_dpp( 0, static_cast< int >( x ), 0x118, 0xf, 0xf, false ) );
  x += static_cast< uint32_t >( __builtin_amdgcn_update_dpp( 0, static_cast< int >( x ), 0x142, 0xa, 0xf, false ) );
  x += static_cast< uint32_t >( __builtin_amdgcn_update_dpp( 0, static_cast< int >( x ), 0x143, 0xc, 0xf, false ) );
  return x;
}

// block-wide exclusive scan of one value per thread; returns the total. One barrier: sh must not
// be written again (by the next scan) before another one.
template < int BS >
__device__ inline uint32_t
block_scan( uint32_t v, uint32_t* excl, uint32_t* sh )
{
  const int lane = threadIdx.x & 63;
  const int wid = threadIdx.x >> 6;
  const uint32_t x = wave_incl_scan( v );
  if ( lane == 63 )
    sh[ wid ] = x;
  __syncthreads();
  uint32_t pre = 0, tot = 0;
  for ( int q = 0; q < BS / 64; ++q )
  {
    if ( q < wid )
      pre += sh[ q ];
    tot += sh[ q ];
  }
  *excl = pre + x - v;
  return __builtin_amdgcn_readfirstlane( tot );  // the same in every thread
}

// Poisson count for seeded drive: splitmix64 of (seed, stream, step) gives u in [0, 1), the
// count is the first k with u < cdf[k] (at most kmax). The first KC entries of the table are
// held in registers; the loop continues in HBM only past them.
constexpr int KC = 8;
struct PoissonCache
{
  double c[ KC ];
  uint64_t seed;
  int32_t kmax;
  gptr< const PoissonTable > T;
};

__device__ inline uint32_t
poisson_count( const PoissonCache& P, uint64_t stream, int64_t step )
{
  uint64_t z = P.seed + stream * 0x9E3779B97F4A7C15ull + static_cast< uint64_t >( step ) * 0xD1B54A32D192ED03ull;
  z = ( z ^ ( z >> 30 ) ) * 0xBF58476D1CE4E5B9ull;
  z = ( z ^ ( z >> 27 ) ) * 0x94D049BB133111EBull;
  z = z ^ ( z >> 31 );
  const double u = static_cast< double >( z >> 11 ) * ( 1.0 / 9007199254740992.0 );
  uint32_t k = 0;
#pragma unroll
  for ( int i = 0; i < KC; ++i )
    if ( k == static_cast< uint32_t >( i ) and i < P.kmax and u >= P.c[ i ] )
      k = i + 1;
  if ( k == KC )
    while ( static_cast< int32_t >( k ) < P.kmax and u >= P.T->cdf[ k ] )
      ++k;
  return k;
}

// Ring-buffer cells of one block seen from one slice: slot_rel = absolute step - origin.
// Window mode keeps slots [wa, wa + wn) in LDS (the slots most events of a slice land in);
// all other cells, and every cell in global mode, live in the block's ring in HBM.
template < bool WIN >
struct Cells
{
  static constexpr bool WINDOW = WIN;
  lptr< double > lds;
  gptr< double > rbb;  // block's ring: [slot][channel][tb]
  uint32_t nct;  // doubles per slot (channels * tb)
  uint32_t tb;
  uint32_t s0;  // ring slot of the slice origin
  uint32_t L;
  uint32_t wa, wn;  // window: first slot (relative to the origin) and slots
  bool win;

  __device__ bool
  in_window( uint32_t slot_rel ) const
  {
    return WIN and win and slot_rel - wa < wn;
  }
  // every slot of [from, to) is in the window
  __device__ bool
  covers( int from, int to ) const
  {
    return WIN and win and static_cast< uint32_t >( from ) >= wa and static_cast< uint32_t >( to ) <= wa + wn;
  }
  __device__ uint32_t
  win_index( uint32_t slot_rel, uint32_t ch, uint32_t local ) const
  {
    return ( slot_rel - wa ) * nct + ch * tb + local;
  }
  __device__ uint32_t
  ring_index( uint32_t slot_rel, uint32_t ch, uint32_t local ) const
  {
    uint32_t slot = s0 + slot_rel;
    if ( slot >= L )
      slot -= L;
    return slot * nct + ch * tb + local;
  }
  __device__ double
  get( uint32_t slot_rel, uint32_t ch, uint32_t local ) const
  {
    if ( in_window( slot_rel ) )
      return lds[ win_index( slot_rel, ch, local ) ];
    return rbb[ ring_index( slot_rel, ch, local ) ];
  }
  __device__ void
  put( uint32_t slot_rel, uint32_t ch, uint32_t local, double v ) const
  {
    if ( in_window( slot_rel ) )
      lds[ win_index( slot_rel, ch, local ) ] = v;
    else
      rbb[ ring_index( slot_rel, ch, local ) ] = v;
  }
};

// Cell cache of cache delivery: keys (ring cell index, ~0 empty) and values share the
// window's LDS area.
constexpr uint32_t EMPTY_KEY = 0xffffffffu;
__device__ inline uint32_t
cache_hash( uint32_t cell )
{
  return __umulhi( cell * 2654435761u, CACHE_SLOTS );
}
// slot of cell in the cache, or NONE when the cell is not cached
__device__ inline uint32_t
cache_find( lptr< const uint32_t > keys, uint32_t cell )
{
  uint32_t h = cache_hash( cell );
  for ( uint32_t p = 0; p < CACHE_PROBES; ++p )
  {
    const uint32_t k = keys[ h ];
    if ( k == cell )
      return h;
    if ( k == EMPTY_KEY )
      return NONE;
    h = h + 1 < CACHE_SLOTS ? h + 1 : 0;
  }
  return NONE;
}
// inserts cell; returns its slot if this call inserted it (the caller loads its value), else NONE
__device__ inline uint32_t
cache_insert( lptr< uint32_t > keys, uint32_t cell )
{
  uint32_t h = cache_hash( cell );
  for ( uint32_t p = 0; p < CACHE_PROBES; ++p )
  {
    uint32_t k = EMPTY_KEY;
    if ( __hip_atomic_compare_exchange_strong( keys + h, &k, cell, __ATOMIC_RELAXED, __ATOMIC_RELAXED,
           __HIP_MEMORY_SCOPE_WORKGROUP ) )
      return h;
    if ( k == cell )
      return NONE;
    h = h + 1 < CACHE_SLOTS ? h + 1 : 0;
  }
  return NONE;  // no free slot within the probe limit: the cell stays in the ring
}

// handle( SpikeEvent& ) of model m (the models' device halves, ng_models_dev.h)
__device__ __forceinline__ void node_receive( int m, double w, uint32_t& ch, double& v );

// spike_generator drive of this part: handle() of the target with weight * multiplicity.
// Each lag adds into a different cell, so the cells of LB lags are read together.
// The drive's parameters are read like a model's (ParamValues), its column col with the state.
struct Drive
{
  int64_t t0, n_steps;
  double w;
  int32_t mode, delay, model;
  PoissonCache PC;
  __device__ __forceinline__ static Drive
  load( const NetDev& d, bool uniform, uint32_t p0, uint32_t pi )
  {
    Drive v;
    if ( uniform )
      v.read( d, ( (cptr< const ParamSet >)d.psets )[ p0 ], (cptr< const PoissonTable >)d.ptables );
    else
      v.read( d, glob( d.psets )[ pi ], glob( d.ptables ) );
    return v;
  }
  template < class PS, class TABLES >
  __device__ __forceinline__ void
  read( const NetDev& d, PS& ps, TABLES tables )
  {
    mode = ps.drive_mode;
    model = ps.model;
    t0 = ps.drive_t0;
    n_steps = ps.drive_steps;
    w = ps.drive_w;
    delay = ps.drive_d;
    if ( mode == 2 )
    {
      const int32_t k = ps.drive_table;
      PC.T = glob( d.ptables ) + k;
      PC.seed = tables[ k ].seed;
      PC.kmax = tables[ k ].kmax;
#pragma unroll
      for ( int i = 0; i < KC; ++i )
        PC.c[ i ] = tables[ k ].cdf[ i ];
    }
  }
};

template < class CELLS >
__device__ inline void
drive_adds( const NetDev& d, const Drive& D, uint32_t col, int m, uint32_t local, const CELLS& C, int64_t origin,
  int from, int stride, int to )
{
  const int32_t mode = D.mode;
  if ( mode == 0 or col == NONE )
    return;
  const int64_t t0 = D.t0, n_steps = D.n_steps;
  const double w = D.w;
  const int32_t dd = D.delay;
  const PoissonCache& PC = D.PC;
  // the channel and multiplier of the weight: the model's handle( SpikeEvent& )
  uint32_t ch;
  double sw;
  node_receive( m, w, ch, sw );
  for ( int l0 = from; l0 < to; l0 += LB * stride )
  {
    double add[ LB ];
    bool has[ LB ];
#pragma unroll
    for ( int q = 0; q < LB; ++q )
    {
      has[ q ] = false;
      const int lag = l0 + q * stride;
      const int64_t e = origin + lag;  // emission step; spike stamp e + 1
      if ( lag >= to or e < t0 or e >= t0 + n_steps )
        continue;
      uint32_t c;
      if ( mode == 1 )
        c = glob( d.drive_counts )[ static_cast< uint64_t >( e - t0 ) * d.drive_cols + col ];
      else
        c = poisson_count( PC, col, e );
      if ( c == 0 )
        continue;
      has[ q ] = true;
      add[ q ] = sw * static_cast< double >( c );
    }
    double old[ LB ];
#pragma unroll
    for ( int q = 0; q < LB; ++q )
      if ( has[ q ] )
        old[ q ] = C.get( static_cast< uint32_t >( l0 + q * stride + dd ), ch, local );
#pragma unroll
    for ( int q = 0; q < LB; ++q )
      if ( has[ q ] )
        C.put( static_cast< uint32_t >( l0 + q * stride + dd ), ch, local, old[ q ] + add[ q ] );
  }
}

// Multimeter sample of one neuron after a step (UniversalDataLogger::record_data,
// nestkernel/universal_data_logger_impl.h:343-375): the model's four state fields.
__device__ inline void
store_sample( const NetDev& d, uint32_t col, int64_t stamp, double f0, double f1, double f2, double f3 )
{
  const int64_t row = ( stamp - d.mm_off ) / d.mm_int - d.mm_row0;
  if ( row < 0 or row >= static_cast< int64_t >( d.mm_rows ) )
  {
    g_or( &d.counters[ 0 ], ERR_SAMPLES );
    return;
  }
  gptr< double > p = glob( d.mm_buf ) + ( static_cast< size_t >( row ) * d.mm_cols + col ) * 4;
  p[ 0 ] = f0;
  p[ 1 ] = f1;
  p[ 2 ] = f2;
  p[ 3 ] = f3;
}

// One of the four fields of such a sample.
__device__ inline void
store_sample_field( const NetDev& d, uint32_t col, int64_t stamp, int field, double f )
{
  const int64_t row = ( stamp - d.mm_off ) / d.mm_int - d.mm_row0;
  if ( row < 0 or row >= static_cast< int64_t >( d.mm_rows ) )
  {
    g_or( &d.counters[ 0 ], ERR_SAMPLES );
    return;
  }
  glob( d.mm_buf )[ ( static_cast< size_t >( row ) * d.mm_cols + col ) * 4 + field ] = f;
}

}  // namespace nestgpu

// the neuron models' device halves: update and handle( SpikeEvent& ) per model id
#include "ng_models_dev.h"

namespace nestgpu
{

// Phase timers of the slice kernel, compiled in only with -DNG_PROFILE: per phase, the sum
// over workgroups of wall-clock ticks (read back with nestgpu_profile_read).
#ifdef NG_PROFILE
__device__ unsigned long long g_phase_ticks[ 8 ];
#define NG_PHASE( i )                                                               \
  do                                                                                \
  {                                                                                 \
    __syncthreads();                                                                \
    if ( threadIdx.x == 0 )                                                         \
    {                                                                               \
      const unsigned long long now_ = wall_clock64();                               \
      atomicAdd( &g_phase_ticks[ i ], now_ - t_phase_ );                            \
      t_phase_ = now_;                                                              \
    }                                                                               \
  } while ( 0 )
#else
#define NG_PHASE( i ) \
  do                  \
  {                   \
  } while ( 0 )
#endif

// Two workgroups of 8 waves per CU need at most 128 VGPRs (4 waves per SIMD); instantiations
// with a WIDE model run one workgroup per CU instead.
// ---------------------------------------------------------------- stdp_synapse
// stdp_synapse::send (models/stdp_synapse.h:222-283) for the event of record ridx, emitted at
// step stamp `stamp` in a slice of parity par, to device target tdev over a delay of dsteps:
// facilitation by the target's spikes since the synapse's last presynaptic spike, depression
// by the target's trace. The presynaptic trace and last spike time before this spike come
// from the source's trace row (the source advanced it when it spiked). Returns the new
// weight, which the record keeps. Every record is delivered at most once per slice (a source
// with stdp synapses spikes at most once per slice, checked in the update phase), so no other
// thread touches its weight meanwhile; the target's history is written only in the update
// phase.
constexpr double STDP_EPS = 1.0e-6;  // ConnectionManager::stdp_eps_ (connection_manager.cpp:78)

__device__ inline HistRing
load_ring( gptr< const HistRing > p )
{
  using v4u = __attribute__( ( ext_vector_type( 4 ) ) ) uint32_t;
  const v4u v = *( gptr< const v4u > )p;
  return { v[ 0 ], v[ 1 ], v[ 2 ], v[ 3 ] };
}

__device__ inline double
stdp_event( const NetDev& d, uint32_t ridx, double w, uint32_t tdev, int64_t stamp, uint32_t dsteps, uint32_t par )
{
  gref< const StdpPre > pre = glob( const_cast< const StdpPre* >( d.spre ) )[ glob( d.srow )[ ridx ] ];
  const double kplus = pre.kp[ par ], t_last = pre.tl[ par ];
  const double tau_plus = pre.tau_plus, lambda = pre.lambda, alpha = pre.alpha, Wmax = pre.Wmax;
  const bool mu_p = pre.mu_plus != 0u, mu_m = pre.mu_minus != 0u;
  const double t_spike = d.ms_per_tic * static_cast< double >( stamp * d.tics_per_step );  // Time::get_ms
  const double dd = static_cast< double >( dsteps ) * d.ms_per_step;  // Time::delay_steps_to_ms
  // ArchivingNode::get_history( t_last - d, t_spike - d ): entries t1 + eps <= t < t2 + eps
  const double t1_lim = ( t_last - dd ) + STDP_EPS;
  const double t2_lim = ( t_spike - dd ) + STDP_EPS;
  const HistRing ring = load_ring( glob( d.hist ) + tdev );
  const uint32_t n = ring.n, hm = ring.mask;
  const uint32_t first = n > hm ? n - hm - 1u : 0u;  // entries before first left the ring
  gptr< const double > ht = glob( d.hist_t ) + ring.base;
  gptr< const double > hk = glob( d.hist_k ) + ring.base;
  auto t_at = [ & ]( uint32_t i ) -> double { return ht[ i & hm ]; };
  // the times are increasing: walk back from the newest entry to the range [lo, hi) of
  // entries t1 + eps <= t < t2 + eps, so that an event costs the target spikes in its range
  uint32_t hi = n;
  while ( hi > first and t_at( hi - 1 ) >= t2_lim )
    --hi;
  uint32_t lo = hi;
  while ( lo > first and t_at( lo - 1 ) >= t1_lim )
    --lo;
  // the range (or the latest spike before t2 - eps) may reach past the entries kept
  if ( first > 0 and lo == first )
    g_or( &d.counters[ 0 ], ERR_STDP_HISTORY );
  for ( uint32_t i = lo; i < hi; ++i )
  {
    // facilitate_ (stdp_synapse.h:187-191), oldest entry first
    const double minus_dt = t_last - ( t_at( i ) + dd );
    const double kp = kplus * ng_exp( minus_dt / tau_plus );
    const double norm_w = ( w / Wmax ) + ( lambda * ( mu_p ? 1.0 - ( w / Wmax ) : 1.0 ) * kp );
    w = norm_w < 1.0 ? norm_w * Wmax : Wmax;
  }
  // ArchivingNode::get_K_value( t_spike - d ) (archiving_node.cpp:85-113): the latest spike
  // strictly before (entries from hi on lie after it)
  const double tq = t_spike - dd;
  double K = 0.0;
  for ( uint32_t i = hi; i > first; --i )
  {
    const double th = t_at( i - 1 );
    if ( tq - th > STDP_EPS )
    {
      K = hk[ ( i - 1 ) & hm ] * ng_exp( ( th - tq ) * glob( d.tau_minus_inv )[ tdev ] );
      break;
    }
  }
  // depress_ (stdp_synapse.h:193-198)
  const double norm_w = ( w / Wmax ) - ( alpha * lambda * ( mu_m ? w / Wmax : 1.0 ) * K );
  w = norm_w > 0.0 ? norm_w * Wmax : 0.0;
  uint64_t bits;
  __builtin_memcpy( &bits, &w, sizeof bits );
  gref< SynRec > r = glob( const_cast< SynRec* >( d.syn ) )[ ridx ];
  r.w_lo = static_cast< uint32_t >( bits );
  r.w_hi = static_cast< uint32_t >( bits >> 32 );
  return w;
}

// ArchivingNode::set_spiketime (archiving_node.cpp:196-230) for the spikes of neuron dev at the
// set bits of `bits` (lags of the slice at origin, of parity par, in order), and the source
// side of stdp_synapse::send (stdp_synapse.h:276-279): each of the neuron's presynaptic trace
// rows keeps its state before the spike in slot par and advances Kplus_ and t_lastspike_. A
// neuron with outgoing stdp synapses must spike at most once per slice.
__device__ inline void
stdp_spikes( const NetDev& d, uint32_t dev, int64_t origin, uint32_t par, const uint64_t* bits )
{
  const bool in = glob( d.stdp_in )[ dev ] != 0;
  const uint32_t row0 = glob( d.pre_row0 )[ dev ], row1 = glob( d.pre_row0 )[ dev + 1 ];
  const bool out = row1 > row0;
  if ( not in and not out )
    return;
  double last = glob( d.last_spike )[ dev ];
  const double slice_start = d.ms_per_tic * static_cast< double >( ( origin + 1 ) * d.tics_per_step );
  int count = 0;
  double km = in ? glob( d.kminus )[ dev ] : 0.0;
  HistRing ring {};
  if ( in )
    ring = load_ring( glob( d.hist ) + dev );
  for ( int w = 0; w < 4; ++w )
  {
    uint64_t x = bits[ w ];
    while ( x )
    {
      const int lag = w * 64 + ( __ffsll( static_cast< long long >( x ) ) - 1 );
      x &= x - 1;
      const double t_sp = d.ms_per_tic * static_cast< double >( ( origin + lag + 1 ) * d.tics_per_step );
      if ( out and ( count > 0 or last >= slice_start ) )
        g_or( &d.counters[ 0 ], ERR_STDP_TWICE );
      ++count;
      if ( in )
      {
        km = km * ng_exp( ( last - t_sp ) * glob( d.tau_minus_inv )[ dev ] ) + 1.0;
        const uint32_t at = ring.base + ( ring.n & ring.mask );
        glob( d.hist_t )[ at ] = t_sp;
        glob( d.hist_k )[ at ] = km;
        ++ring.n;
      }
      for ( uint32_t r = row0; r < row1; ++r )
      {
        gref< StdpPre > pre = glob( d.spre )[ r ];
        const double kp = pre.cur_kp, tl = pre.cur_tl;
        pre.kp[ par ] = kp;
        pre.tl[ par ] = tl;
        pre.cur_kp = kp * ng_exp( ( tl - t_sp ) / pre.tau_plus ) + 1.0;
        pre.cur_tl = t_sp;
      }
      last = t_sp;
    }
  }
  if ( count )
  {
    glob( d.last_spike )[ dev ] = last;
    if ( in )
    {
      glob( d.kminus )[ dev ] = km;
      glob( d.hist )[ dev ].n = ring.n;
      if ( ring.n > ring.lim )
        g_or( &d.counters[ 0 ], REQ_HISTORY );
    }
  }
}

// STDP: some instance of the launch has stdp_synapse connections (its own instantiation, so
// that networks without them carry none of that code or its registers)
//
// CACHE: some instance of the launch uses cache delivery; one instantiation, with every model,
// serves these launches, so that the cache costs the others no registers (with it in the window
// kernels, 389 scalar registers spilled into vector lanes).
template < int MASK, bool WIN, bool STDP, bool CACHE >
__global__ void __launch_bounds__( Tile< WIN >::BS,
  ( MASK & WIDE_MODELS ) ? 1 : WIN or STDP ? 4 : global_waves< MASK >() )
  k_slice( const NetDev* __restrict__ nets, const uint32_t* __restrict__ blk_prefix, int n_nets, int s )
{
#ifdef NG_PROFILE
  unsigned long long t_phase_ = wall_clock64();
#endif
  __shared__ SliceLds< WIN > S;
  constexpr int BS = Tile< WIN >::BS;
  constexpr int SPT = Tile< WIN >::SPT;
  constexpr int CH = Tile< WIN >::CH;
  constexpr int RQ = Tile< WIN >::RQ;
  constexpr int R = Tile< WIN >::R;
  constexpr bool SINGLE = single_model< MASK >() >= 0;
  // loads ahead of the delivery: the global kernels held to 80 registers (global_waves) have none
  // left for them; those at 128 were not measured with them
  constexpr bool EARLY = WIN;

  // ---- which instance and block
  const uint32_t gb = n_nets > 1 ? blockIdx.x : xcd_block( blockIdx.x, gridDim.x );
  int lo = 0, hi = n_nets;
  while ( hi - lo > 1 )
  {
    const int mid = ( lo + hi ) >> 1;
    if ( blk_prefix[ mid ] <= gb )
      lo = mid;
    else
      hi = mid;
  }
  const NetDev& d = nets[ lo ];
  const uint32_t b = gb - blk_prefix[ lo ];
  const SlicePhase ph = slice_phase( d, s );
  if ( not ph.active or b >= d.n_blocks )
    return;
  // phase timing (counters[4..6]): thread 0 reads the 100 MHz wall clock at the start, after
  // delivery and at the end of the workgroup's work
  const bool ptime = d.phase_timing != 0;
  unsigned long long tp0 = 0, tp1 = 0;
  const uint32_t P = d.n_blocks;
  const uint32_t tb = d.tb;
  const uint32_t t = threadIdx.x;

  const int par = ph.parity;
  const int ppar = par ^ 1;
  // the first of the loads that the delivery waits for one after the other (list heads, run
  // table, records, ring cells)
  const bool heads = EARLY and P <= static_cast< uint32_t >( BS );  // one thread per block's list
  const size_t my_list = ( static_cast< size_t >( ppar ) * P + t ) * d.spk_cap;
  uint32_t my_n = 0;
  Entries head {};
  if ( heads and t < P and ph.deliver )
  {
    my_n = glob( d.blk_cnt )[ static_cast< size_t >( ppar ) * P + t ];
    head = load_entries( glob( d.blk_spk ) + my_list, d.spk_cap );
  }
  // the block's targets: device indices dev0 .. dev0 + nb - 1
  const uint32_t dev0 = __builtin_amdgcn_readfirstlane( glob( d.bstart )[ b ] );
  const uint32_t nb = __builtin_amdgcn_readfirstlane( glob( d.bstart )[ b + 1 ] ) - dev0;

  Cells< WIN > C;
  C.lds = ( lptr< double > )S.win;
  C.nct = static_cast< uint32_t >( d.nch ) * tb;
  C.tb = tb;
  C.L = static_cast< uint32_t >( d.L );
  C.s0 = static_cast< uint32_t >( ph.origin % d.L );
  C.wa = static_cast< uint32_t >( d.wa );
  C.wn = static_cast< uint32_t >( d.wn );
  C.win = WIN and d.win != 0;
  C.rbb = glob( d.rb ) + static_cast< size_t >( b ) * C.L * C.nct;
  // ring bytes per block < 2^31 (checked on the host), so NO_CELL is always out of range
  const __amdgpu_buffer_rsrc_t rb_rsrc = __builtin_amdgcn_make_buffer_rsrc(
    d.rb + static_cast< size_t >( b ) * C.L * C.nct, 0, static_cast< int >( C.L * C.nct * 8u ), 0x00020000 );

  if ( ptime and threadIdx.x == 0 )
    tp0 = wall_clock64();
  // What the workgroup needs whatever is delivered is loaded now, so that it arrives while the
  // window is staged and the spikes are looked up: the neurons' states, the parameter index and
  // drive column of each thread's neuron (thread t < nb updates neuron t, spare threads add the
  // drive).
  // A load takes about 3,000 cycles here, and a slice of a small network is a chain of them
  // (8-population circuit, 7,700 neurons: 16.7 -> 14.9 us per slice with these loads early).
  const uint32_t local = t;
  const uint32_t dev = dev0 + local;
  // G groups of spare threads, from thread g0 on: from the next whole wave if a group fits
  // there, so that no wave runs the update and the drive one after the other
  uint32_t g0 = ( nb + 63u ) & ~63u;
  if ( g0 + nb > static_cast< uint32_t >( BS ) )
    g0 = nb;
  const uint32_t G = ( static_cast< uint32_t >( BS ) - g0 ) / nb;
  const bool drives = local < nb ? G == 0 : local >= g0 and local < g0 + G * nb;
  const uint32_t ddl = local < nb ? local : drives ? ( local - g0 ) % nb : 0u;  // the drive thread's neuron
  using Node1 = DeviceNode< SINGLE ? single_model< MASK >() : 0 >;
  typename Node1::State st {};
  uint32_t pi = 0, dcol = NONE;
  auto load_neuron = [ & ]
  {
    if ( local < nb or drives )
      pi = glob( d.pidx )[ dev0 + ddl ];
    if ( drives )
      dcol = glob( d.drive_idx )[ dev0 + ddl ];
    if ( SINGLE and local < nb )
      st = Node1::load( d, dev );
  };
  if ( EARLY )
    load_neuron();
  // ================================================================ 0. stage the window
  uint32_t w0 = C.s0 + C.wa;  // ring slot of the window's first slot
  if ( w0 >= C.L )
    w0 -= C.L;
  const uint32_t n_win = C.wn * C.nct;
  const uint32_t before_wrap = ( C.L - w0 ) * C.nct;
  auto ring_of = [ & ]( uint32_t i ) { return i < before_wrap ? w0 * C.nct + i : i - before_wrap; };
  // four cells per thread and step, whose loads are in flight together
  constexpr uint32_t WQ = 4;
  if ( WIN and C.win )
    for ( uint32_t i0 = t; i0 < n_win; i0 += WQ * BS )
    {
      double x[ WQ ];
#pragma unroll
      for ( uint32_t q = 0; q < WQ; ++q )
        x[ q ] = cell_load( rb_rsrc, i0 + q * BS < n_win ? ring_of( i0 + q * BS ) * 8u : NO_CELL );
#pragma unroll
      for ( uint32_t q = 0; q < WQ; ++q )
        if ( i0 + q * BS < n_win )
          S.win[ i0 + q * BS ] = x[ q ];
    }
  // cache delivery: an empty cell cache for this slice (keys, then values, in the window area)
  const bool cache = CACHE and d.cache != 0 and ph.deliver;
  const lptr< uint32_t > ckey = ( lptr< uint32_t > )reinterpret_cast< uint32_t* >( S.win );
  const lptr< double > cval = ( lptr< double > )( S.win + CACHE_SLOTS / 2 );
  if ( cache )
    for ( uint32_t i = t; i < CACHE_SLOTS; i += BS )
      ckey[ i ] = EMPTY_KEY;

  // scratch of every other block scan: the bucket starts, which are not in use at those times
  uint32_t* const sh1 = reinterpret_cast< uint32_t* >( S.bst );

  // ================================================================ 1. delivery
  if ( ph.deliver )
  {
    // prefix of per-block spike counts: an instance with more blocks than threads in the window
    // kernel (it has no window) keeps it in the unused window
    uint32_t* const pref = WIN and P > static_cast< uint32_t >( BS ) ? reinterpret_cast< uint32_t* >( S.win ) : S.pref;
    S.bcnt[ 0 ][ t ] = 0;
    S.bcnt[ 1 ][ t ] = 0;
    int cur = 0;  // counter buffer of the current round
    const bool flat = __builtin_amdgcn_readfirstlane( glob( d.flat_meta )[ 2 + ppar ] ) != 0;
    uint32_t K;
    bool listed = false;   // the slice's spikes are in S.sk, in order
    bool counted = flat;  // K, and the prefix where it is needed, are known
    if ( flat )
      K = __builtin_amdgcn_readfirstlane( glob( d.flat_meta )[ ppar ] );
    else if ( heads )
    {
      // a list too long to be copied counts as more than all spikes in short ones (512 blocks)
      constexpr uint32_t LONG = 1u << 20;
      uint32_t my_k;  // the first spike of block t
      K = block_scan< BS >( my_n > LIST_COPY ? LONG : my_n, &my_k, S.sh );
      // One chunk of spikes in short lists: thread t copies block t's, whose first four it has, and
      // no thread searches the block of its spikes. Others are looked up chunk by chunk.
      listed = K <= static_cast< uint32_t >( CH );
      counted = K < LONG;
      if ( listed )
        for ( uint32_t i = 0; i < my_n; i += 4 )
        {
          const Entries e = i == 0 ? head : load_entries( glob( d.blk_spk ) + my_list + i, d.spk_cap - i );
#pragma unroll
          for ( uint32_t j = 0; j < 4; ++j )
            if ( i + j < my_n )
              S.sk[ my_k + i + j ] = e.x[ j ];
        }
      else if ( counted )
      {
        if ( t < P )
          pref[ t ] = my_k;
        if ( t == 0 )
          pref[ P ] = K;
      }
    }
    if ( not counted )
    {
      // prefix of the per-block spike counts of the delivered slice
      gptr< const uint32_t > cnt = glob( d.blk_cnt ) + static_cast< size_t >( ppar ) * P;
      uint32_t carry = 0;
      if ( heads )
        __syncthreads();  // S.sh is read
      for ( uint32_t p0 = 0; p0 < P; p0 += BS )
      {
        const uint32_t v = p0 + t < P ? cnt[ p0 + t ] : 0;
        uint32_t ex;
        const uint32_t tot = block_scan< BS >( v, &ex, S.sh );
        if ( p0 + t < P )
          pref[ p0 + t ] = carry + ex;
        carry += tot;
        __syncthreads();
      }
      if ( t == 0 )
        pref[ P ] = carry;
      K = carry;
    }
    __syncthreads();
    NG_PHASE( 0 );
    unsigned long long events = 0;
    // A block with few targets splits each target's bucket by slot, up to the number of
    // counters: a bucket's events are compared with each other, and 32 targets alone would make
    // buckets of 32 events (5,000 iaf_psc_delta neurons, 226,000 events per slice: 30 -> 25 us
    // with the sorted arrays and the event index; 100,000 iaf_psc_exp, 4.9M events: 118 -> 103;
    // the full 8-population circuit, 1.75M events: 46 -> 42).
    const uint32_t sub_mask = ( 1u << ( 31 - __builtin_clz( static_cast< uint32_t >( BS ) / nb ) ) ) - 1u;
    // events received in this thread's bucket (local index t % nb), counted while d.rx is set
    uint32_t rxc = 0;
    for ( uint32_t k0 = 0; k0 < K; k0 += CH )
    {
      // each thread resolves SPT consecutive spikes of the chunk: (source, lag), then its
      // run [g0, g1) in the source's row; the loads of one step are independent
      uint32_t src[ SPT ], lag[ SPT ];
      const uint32_t kb = k0 + t * SPT;
      if ( listed )
      {
#pragma unroll
        for ( int q = 0; q < SPT; ++q )
          if ( kb + q < K )
          {
            const uint32_t e = S.sk[ kb + q ];
            src[ q ] = e >> 8;
            lag[ q ] = e & 0xffu;
          }
      }
      else if ( flat )
      {
#pragma unroll
        for ( int q = 0; q < SPT; ++q )
          if ( kb + q < K )
          {
            src[ q ] = glob( d.flat_src )[ kb + q ];
            lag[ q ] = glob( d.flat_lag )[ kb + q ];
          }
      }
      else if ( kb < K )
      {
        uint32_t blk = upper_bound_u32( pref, P + 1, kb ) - 1;
#pragma unroll
        for ( int q = 0; q < SPT; ++q )
        {
          const uint32_t k = kb + q;
          if ( k < K )
          {
            while ( pref[ blk + 1 ] <= k )
              ++blk;
            const size_t at = ( static_cast< size_t >( ppar ) * P + blk ) * d.spk_cap + ( k - pref[ blk ] );
            const uint32_t e = glob( d.blk_spk )[ at ];
            src[ q ] = e >> 8;
            lag[ q ] = e & 0xffu;
          }
        }
      }
      uint32_t g0v[ SPT ], lenv[ SPT ], s1v[ SPT ], s2v[ SPT ];
#pragma unroll
      for ( int q = 0; q < SPT; ++q )
      {
        lenv[ q ] = 0;
        if ( kb + q < K )
        {
          gptr< const uint32_t > bo = glob( d.boff ) + static_cast< size_t >( src[ q ] ) * ( P + 1 ) + b;
          g0v[ q ] = bo[ 0 ];
          lenv[ q ] = bo[ 1 ] - g0v[ q ];
          S.c_lag[ t * SPT + q ] = static_cast< uint8_t >( lag[ q ] );
        }
      }
      // Slot-range passes: pass p takes the events landing in slots [p ws, (p + 1) ws), i.e.
      // delay offsets [p ws - lag, (p + 1) ws - lag): a contiguous part of the delay-ordered
      // run, split at s1 (and s2 for a third pass).
#pragma unroll
      for ( int q = 0; q < SPT; ++q )
      {
        s1v[ q ] = lenv[ q ];
        s2v[ q ] = lenv[ q ];
        if ( d.np > 1 and lenv[ q ] > 0 )
        {
          s1v[ q ] = run_split( glob( d.syn ), g0v[ q ], lenv[ q ], d.ws - static_cast< int >( lag[ q ] ) );
          if ( d.np > 2 )
            s2v[ q ] = run_split( glob( d.syn ), g0v[ q ], lenv[ q ], 2 * d.ws - static_cast< int >( lag[ q ] ) );
        }
      }
      for ( int pass = 0; pass < d.np; ++pass )
      {
      uint32_t lens[ SPT ];
      uint32_t mine = 0;
#pragma unroll
      for ( int q = 0; q < SPT; ++q )
      {
        const uint32_t lo = pass == 0 ? 0u : ( pass == 1 ? s1v[ q ] : s2v[ q ] );
        const uint32_t hi = pass == d.np - 1 ? lenv[ q ] : ( pass == 0 ? s1v[ q ] : s2v[ q ] );
        lens[ q ] = hi - lo;
        if ( lens[ q ] )
          S.c_g0[ t * SPT + q ] = g0v[ q ] + lo;
        mine += lens[ q ];
      }
      uint32_t ex;
      const uint32_t E = block_scan< BS >( mine, &ex, sh1 );
#pragma unroll
      for ( int q = 0; q < SPT; ++q )
      {
        S.c_off[ t * SPT + q ] = ex;
        ex += lens[ q ];
      }
      if ( t == 0 )
        S.c_off[ CH ] = E;
      // The spike of every 2^sh-th event (sh the smallest with at most BS of them): an event's
      // spike is then a table read and a short walk instead of a binary search over the chunk
      // (11 dependent LDS reads per round).
      const int sh = E > static_cast< uint32_t >( BS ) ? 32 - __builtin_clz( ( E - 1 ) / BS ) : 0;
      {
        uint32_t off = ex - mine;
#pragma unroll
        for ( int q = 0; q < SPT; ++q )
        {
          const uint32_t end = off + lens[ q ];
          for ( uint32_t m = ( off + ( 1u << sh ) - 1 ) >> sh; ( m << sh ) < end; ++m )
            S.c_idx[ m ] = static_cast< uint16_t >( t * SPT + q );
          off = end;
        }
      }
      __syncthreads();
      NG_PHASE( 1 );
      events += E;
      if ( cache and E )
      {
        // The cells of this chunk's events join the slice's cell cache. Each thread takes a
        // contiguous span of the events, reads their records (the rounds read them again, from
        // L2) and loads the value of every cell it inserts, all loads in flight together: the
        // rounds then add into LDS only. A cell stays cached for the rest of the slice, so all
        // its later additions go to the cache, after the ones it already holds.
        constexpr int HQ = 8;
        const int umodel = d.uniform_model;
        const uint32_t per = ( E + BS - 1 ) / BS;
        const uint32_t e_beg = min( E, t * per ), e_end = min( E, e_beg + per );
        uint32_t j = e_beg < e_end ? upper_bound_u32( S.c_off, CH + 1, e_beg ) - 1 : 0;
        for ( uint32_t e0 = e_beg; e0 < e_end; e0 += HQ )
        {
          SynRec hr[ HQ ];
          uint32_t hl[ HQ ];
#pragma unroll
          for ( int q = 0; q < HQ; ++q )
          {
            const uint32_t e = e0 + q < e_end ? e0 + q : e_end - 1;
            while ( j + 1 < static_cast< uint32_t >( CH ) and S.c_off[ j + 1 ] <= e )
              ++j;
            hr[ q ] = load_rec( glob( d.syn ) + S.c_g0[ j ] + ( e - S.c_off[ j ] ) );
            hl[ q ] = S.c_lag[ j ];
          }
          uint32_t hcell[ HQ ], hslot[ HQ ];
#pragma unroll
          for ( int q = 0; q < HQ; ++q )
          {
            hslot[ q ] = NONE;
            hcell[ q ] = 0;
            if ( e0 + q < e_end )
            {
              const double w = __hiloint2double( static_cast< int >( hr[ q ].w_hi ), static_cast< int >( hr[ q ].w_lo ) );
              const uint32_t local = hr[ q ].word & 0xffffu;
              const uint32_t slot_rel = hl[ q ] + ( ( hr[ q ].word >> 16 ) & DELAY_MASK );
              const int m = single_model< MASK >() >= 0 ? single_model< MASK >()
                : umodel >= 0                           ? umodel
                                                        : glob( d.model )[ dev0 + local ];
              uint32_t ch;
              double v;
              node_receive( m, w, ch, v );
              hcell[ q ] = C.ring_index( slot_rel, ch, local );
              hslot[ q ] = cache_insert( ckey, hcell[ q ] );
            }
          }
          double hv[ HQ ];
#pragma unroll
          for ( int q = 0; q < HQ; ++q )
            hv[ q ] = cell_load( rb_rsrc, hslot[ q ] != NONE ? hcell[ q ] * 8u : NO_CELL );
#pragma unroll
          for ( int q = 0; q < HQ; ++q )
            if ( hslot[ q ] != NONE )
              cval[ hslot[ q ] ] = hv[ q ];
        }
        __syncthreads();
      }
      // rounds of R events; the synapse records of round r + 1 are loaded while round r
      // is bucketed and applied
      SynRec rec[ RQ ];
      uint32_t rlag[ RQ ];
      uint32_t rid[ STDP ? RQ : 1 ];  // stdp_synapse: the records' indices
      // Every thread issues RQ record loads (events past the end reload the last record):
      // with a fixed number of loads in flight the waits count exactly, instead of draining
      // all outstanding memory operations.
      auto load_round = [ & ]( uint32_t e0 )
      {
        const uint32_t eb = e0 + t * RQ;
        uint32_t j = S.c_idx[ ( eb < E ? eb : E - 1 ) >> sh ];
#pragma unroll
        for ( int q = 0; q < RQ; ++q )
        {
          const uint32_t e = eb + q < E ? eb + q : E - 1;
          while ( j + 1 < static_cast< uint32_t >( CH ) and S.c_off[ j + 1 ] <= e )
            ++j;
          const uint32_t ri = S.c_g0[ j ] + ( e - S.c_off[ j ] );
          rec[ q ] = load_rec( glob( d.syn ) + ri );
          rlag[ q ] = S.c_lag[ j ];
          if constexpr ( STDP )
            rid[ q ] = ri;
        }
      };
      if ( E )
        load_round( 0 );
      const int umodel = d.uniform_model;
      const uint32_t dpar = static_cast< uint32_t >( ph.parity ^ 1 );  // the delivered spikes' slice
      (void)dpar;
      for ( uint32_t e0 = 0; e0 < E; e0 += R, cur ^= 1 )
      {
        // stage: thread t holds events e0 + t*RQ .. + RQ - 1 (key order = round index) and
        // takes an unordered place in its bucket (target and part of the slots)
        uint32_t key[ RQ ], loc[ RQ ], dst[ RQ ], ci[ RQ ], goff[ RQ ];
        double val[ RQ ], cv[ RQ ];
        bool lw[ RQ ];  // the event's cell is in the LDS window
        bool lc[ RQ ];  // the event's cell is in the cell cache (ci = its cache slot)
        const uint32_t eb = e0 + t * RQ;
#pragma unroll
        for ( int q = 0; q < RQ; ++q )
        {
          loc[ q ] = NONE;
          goff[ q ] = NO_CELL;
          lc[ q ] = false;
          if ( eb + q < E )
          {
            double w = __hiloint2double( static_cast< int >( rec[ q ].w_hi ), static_cast< int >( rec[ q ].w_lo ) );
            const uint32_t local = rec[ q ].word & 0xffffu;
            if constexpr ( STDP )
            {
              if ( rec[ q ].word & PLASTIC_BIT )
                w = stdp_event( d, rid[ q ], w, dev0 + local, ph.origin - d.min_delay + rlag[ q ] + 1,
                  ( ( rec[ q ].word >> 16 ) & DELAY_MASK ) + static_cast< uint32_t >( d.min_delay ), dpar );
            }
            const uint32_t slot_rel = rlag[ q ] + ( ( rec[ q ].word >> 16 ) & DELAY_MASK );
            const int m = single_model< MASK >() >= 0 ? single_model< MASK >()
              : umodel >= 0                           ? umodel
                                                      : glob( d.model )[ dev0 + local ];
            uint32_t ch;
            double v;
            node_receive( m, w, ch, v );  // static_synapse: weight * multiplicity 1
            const uint32_t sc = slot_rel * d.nch + ch;
            loc[ q ] = local + nb * ( sc & sub_mask );
            val[ q ] = v;
            key[ q ] = ( sc << IDX_BITS ) | static_cast< uint32_t >( t * RQ + q );
            dst[ q ] = atomicAdd( &S.bcnt[ cur ][ loc[ q ] ], 1u );
            lw[ q ] = C.in_window( slot_rel );
            if ( lw[ q ] )
              ci[ q ] = C.win_index( slot_rel, ch, local );
            else
            {
              ci[ q ] = C.ring_index( slot_rel, ch, local );
              const uint32_t hs = cache ? cache_find( ckey, ci[ q ] ) : NONE;
              if ( hs != NONE )
              {
                lc[ q ] = true;
                ci[ q ] = hs;
              }
              else
                goff[ q ] = ci[ q ] * 8u;
            }
          }
        }
        // the records of this round are consumed: load the next round's now, so they have the
        // whole round to arrive (past the last round: reloads record E - 1, unused)
        load_round( e0 + R );
        __syncthreads();
        NG_PHASE( 2 );  // stage
        // every thread has finished the previous round (its cell stores included): the cells
        // of this round can be read now, while the buckets are formed
#pragma unroll
        for ( int q = 0; q < RQ; ++q )
          cv[ q ] = cell_load( rb_rsrc, goff[ q ] );
        // bucket starts: wave 0 scans the buckets' counts, BS / 64 per lane; the others
        // clear the counters of the next round
        if ( t < 64 )
        {
          constexpr int CPL = BS / 64;
          uint32_t c[ CPL ];
          uint32_t sum = 0;
#pragma unroll
          for ( int j = 0; j < CPL; ++j )
          {
            c[ j ] = S.bcnt[ cur ][ CPL * t + j ];
            sum += c[ j ];
          }
          uint32_t run = wave_incl_scan( sum ) - sum;
#pragma unroll
          for ( int j = 0; j < CPL; ++j )
          {
            S.bst[ CPL * t + j ] = static_cast< uint16_t >( run );
            run += c[ j ];
          }
          if ( t == 63 )
            S.bst[ BS ] = static_cast< uint16_t >( run );
        }
        S.bcnt[ cur ^ 1 ][ t ] = 0;
        if ( d.rx )
          rxc += S.bcnt[ cur ][ t ];
        __syncthreads();
        NG_PHASE( 3 );  // bucket starts
#pragma unroll
        for ( int q = 0; q < RQ; ++q )
          if ( loc[ q ] != NONE )
          {
            dst[ q ] += S.bst[ loc[ q ] ];
            S.bk[ dst[ q ] ] = key[ q ];
          }
        __syncthreads();
        // sorted place of each event in its bucket by (cell, key): the number of smaller keys
        uint32_t srt[ RQ ], bhi[ RQ ];
        bool lead[ RQ ];
#pragma unroll
        for ( int q = 0; q < RQ; ++q )
          if ( loc[ q ] != NONE )
          {
            const uint32_t lo = S.bst[ loc[ q ] ], hi = S.bst[ loc[ q ] + 1 ];
            uint32_t r = 0;
            uint32_t i = lo;
            for ( ; i + 4 <= hi; i += 4 )
            {
              const uint32_t k0 = S.bk[ i ], k1 = S.bk[ i + 1 ], k2 = S.bk[ i + 2 ], k3 = S.bk[ i + 3 ];
              r += ( k0 < key[ q ] ? 1u : 0u ) + ( k1 < key[ q ] ? 1u : 0u ) + ( k2 < key[ q ] ? 1u : 0u )
                + ( k3 < key[ q ] ? 1u : 0u );
            }
            for ( ; i < hi; ++i )
              r += S.bk[ i ] < key[ q ] ? 1u : 0u;
            srt[ q ] = lo + r;
            bhi[ q ] = hi;
            lead[ q ] = r == 0;  // certainly the first of its cell's run
            S.sk[ srt[ q ] ] = key[ q ];
            S.sw[ srt[ q ] ] = val[ q ];
          }
        __syncthreads();
        NG_PHASE( 4 );  // place and rank
        // the first event of each cell's run adds the whole run in key order; runs of
        // different cells proceed in parallel
#pragma unroll
        for ( int q = 0; q < RQ; ++q )
        {
          if ( loc[ q ] == NONE )
            continue;
          const uint32_t sc = key[ q ] >> IDX_BITS;
          if ( not lead[ q ] and ( S.sk[ srt[ q ] - 1 ] >> IDX_BITS ) == sc )
          {
            loc[ q ] = NONE;  // not the first of its run
            goff[ q ] = NO_CELL;
            continue;
          }
          double v = lw[ q ] ? S.win[ ci[ q ] ] : lc[ q ] ? cval[ ci[ q ] ] : cv[ q ];
          v = v + val[ q ];
          for ( uint32_t i = srt[ q ] + 1; i < bhi[ q ] and ( S.sk[ i ] >> IDX_BITS ) == sc; ++i )
            v = v + S.sw[ i ];
          cv[ q ] = v;
        }
#pragma unroll
        for ( int q = 0; q < RQ; ++q )
        {
          if ( loc[ q ] != NONE and lw[ q ] )
            S.win[ ci[ q ] ] = cv[ q ];
          else if ( loc[ q ] != NONE and lc[ q ] )
            cval[ ci[ q ] ] = cv[ q ];
          cell_store( rb_rsrc, goff[ q ], cv[ q ] );  // NO_CELL unless a global run leader
        }
        NG_PHASE( 5 );  // apply
      }
      }  // passes
    }
    if ( cache )
    {
      // write the cached cells back to the ring: the update and the drive read them there
      __syncthreads();
      for ( uint32_t i = t; i < CACHE_SLOTS; i += BS )
      {
        const uint32_t k = ckey[ i ];
        cell_store( rb_rsrc, k != EMPTY_KEY ? k * 8u : NO_CELL, cval[ i ] );
      }
    }
    if ( t == 0 and events )
      g_add( &d.counters[ 1 ], events );
    // a target's events are spread over its buckets t, t + nb, ...: their threads add up in HBM
    // once per slice (with one thread per target that read all its buckets in every round, the
    // first Run of the 8-population circuit at scale 0.384, 39 ms, took 14.8 ms instead of 10.2)
    if ( d.rx and rxc )
      g_add( d.rx + dev0 + t % nb, rxc );
  }
  if ( ( MASK & BLOCK_MODELS ) != 0 and t == 0 )
    S.pool_next = BS / 4;
  __syncthreads();  // window staged and delivered
  if ( ptime and t == 0 )
    tp1 = wall_clock64();

  // ================================================================ 2. update
  // Threads [0, nb) update one neuron each. The spike_generator drive of the slice lands in
  // cells at least min_delay ahead (every delay, the drive's included, is >= min_delay), which
  // the update does not touch, and in distinct cells per lag: when nb <= BS / 2 the spare
  // threads add it concurrently, G groups of nb threads splitting the lags (a wave that held
  // neurons and drive threads ran the two one after the other, 4,000-6,000 cycles more).
  uint64_t bits[ 4 ] = { 0, 0, 0, 0 };
  if ( not EARLY )
    load_neuron();
  // whether the neurons of this wave's threads share one parameter set
  const uint32_t p0 = __builtin_amdgcn_readfirstlane( pi );
  const bool uniform = __ballot( pi != p0 and ( local < nb or drives ) ) == 0;
  if ( local >= nb and drives )
  {
    const uint32_t g = ( local - g0 ) / nb;
    const Drive D = Drive::load( d, uniform, p0, pi );
    const int dm = SINGLE ? single_model< MASK >() : D.model;
    drive_adds( d, D, dcol, dm, ddl, C, ph.origin, ph.from + static_cast< int >( g ), static_cast< int >( G ), ph.to );
  }
  if ( local < nb )
  {
    // multimeter: the next step of this part whose state is sampled (ph.to: none)
    const uint32_t mcol = d.mm_int > 0 ? glob( d.mm_col )[ dev ] : NONE;
    int next_sample = mcol != NONE ? first_sample_lag( d, ph.origin, ph.from, ph.to ) : ph.to;
    const int m = SINGLE ? single_model< MASK >() : glob( d.psets )[ pi ].model;
    // Node::update of the neuron's model (each model of the launch's mask is compiled in)
    if constexpr ( SINGLE )
      Node1::update( d, Node1::Params::load( d.psets, uniform, p0, pi ), st, dev, local, C, ph, bits, mcol, next_sample );
    else
    {
#define NG_UPDATE( ID )                                                                                             \
  if ( ( MASK & ( 1 << ( ID ) ) ) and m == ( ID ) )                                                               \
    DeviceNode< ( ID ) >::update( d, DeviceNode< ( ID ) >::Params::load( d.psets, uniform, p0, pi ),              \
      DeviceNode< ( ID ) >::load( d, dev ), dev, local, C, ph, bits, mcol, next_sample );
      NG_DEVICE_MODELS( NG_UPDATE )
#undef NG_UPDATE
    }
    if ( drives )
      drive_adds( d, Drive::load( d, uniform, p0, pi ), dcol, m, local, C, ph.origin, ph.from, 1, ph.to );
  }
  if ( ( MASK & BLOCK_MODELS ) != 0 and ( SINGLE or d.uniform_model < 0 or d.uniform_model == M_AEIF_COND_EXP ) )
  {
    // the neurons of the model that the workgroup updates together
    using Node = DeviceNode< M_AEIF_COND_EXP >;
    const lptr< uint32_t > next = ( lptr< uint32_t > )&S.pool_next;
    const lptr< unsigned long long > spk = ( lptr< unsigned long long > )S.spk_bits;
    lptr< const uint16_t > order = nullptr;
    if ( nb > static_cast< uint32_t >( BS / 4 ) )
    {
      // More neurons than quads: the ones that will probably take many steps go first, so that
      // no quad starts a long one when the others are done.
      uint32_t before;
      const bool first = local < nb and Node::long_update( d, dev );
      const uint32_t n_first = block_scan< BS >( first ? 1u : 0u, &before, sh1 );
      if ( local < nb )
        S.order[ first ? before : n_first + local - before ] = static_cast< uint16_t >( local );
      order = ( lptr< const uint16_t > )S.order;
      __syncthreads();
    }
    Node::template update_block< Cells< WIN >, SINGLE >( d, dev0, nb, C, ph, next, spk, order );
    __syncthreads();
    if ( local < nb and ( SINGLE or glob( d.model )[ dev ] == M_AEIF_COND_EXP ) )
    {
      const uint32_t nw = ( static_cast< uint32_t >( d.min_delay ) + 63u ) >> 6;
#pragma unroll
      for ( uint32_t w = 0; w < 4; ++w )
        bits[ w ] = w < nw ? S.spk_bits[ local * nw + w ] : 0ull;
    }
  }
  if ( STDP and d.stdp and local < nb )
    stdp_spikes( d, dev, ph.origin, static_cast< uint32_t >( ph.parity ), bits );
  NG_PHASE( 6 );

  // ================================================================ 3. spike lists
  const uint32_t nsp = __popcll( bits[ 0 ] ) + __popcll( bits[ 1 ] ) + __popcll( bits[ 2 ] ) + __popcll( bits[ 3 ] );
  uint32_t ex;
  const uint32_t tot = block_scan< BS >( nsp, &ex, S.sh );  // also orders the update before the write-back
  if ( WIN and C.win )
  {
    for ( uint32_t i = t; i < n_win; i += BS )
      C.rbb[ i < before_wrap ? w0 * C.nct + i : i - before_wrap ] = S.win[ i ];
  }
  if ( t == 0 )
  {
    gptr< uint32_t > cnt = glob( d.blk_cnt ) + static_cast< size_t >( par ) * P + b;
    const uint32_t base = ph.from == 0 ? 0u : *cnt;  // a new slice starts an empty list
    S.cnt_base = base;
    if ( base + tot > d.spk_cap )
      g_or( &d.counters[ 0 ], ERR_SPIKE_LIST );
    *cnt = base + tot < d.spk_cap ? base + tot : d.spk_cap;
    if ( ph.from == 0 and b == 0 )
      glob( d.flat_meta )[ 2 + par ] = 0;
    S.log_base = 0ull;
    if ( tot )
    {
      g_add( &d.counters[ 2 ], static_cast< unsigned long long >( tot ) );
      if ( d.log_enabled )
        S.log_base = g_add( d.log_n, static_cast< unsigned long long >( tot ) );
    }
  }
  __syncthreads();
  const bool log_on = d.log_enabled != 0;
  if ( nsp )
  {
    uint32_t o = S.cnt_base + ex;
    unsigned long long li = S.log_base + ex;
    const size_t list = ( static_cast< size_t >( par ) * P + b ) * d.spk_cap;
    for ( int w = 0; w < 4; ++w )
    {
      unsigned long long x = bits[ w ];
      while ( x )
      {
        const uint32_t lag = w * 64 + ( __ffsll( static_cast< long long >( x ) ) - 1 );
        x &= x - 1;
        if ( o < d.spk_cap )
        {
          glob( d.blk_spk )[ list + o ] = ( dev << 8 ) | lag;
          glob( d.blk_part )[ list + o ] = static_cast< uint8_t >( ph.part );
        }
        ++o;
        if ( log_on )
        {
          if ( li < d.log_cap )
          {
            glob( d.log_src )[ li ] = dev;
            glob( d.log_step )[ li ] = ph.origin + lag + 1;
          }
          else
            g_or( &d.counters[ 0 ], ERR_LOG );
          ++li;
        }
      }
    }
  }
  NG_PHASE( 7 );
  if ( ptime )
  {
    __syncthreads();
    if ( t == 0 )
    {
      const unsigned long long tp2 = wall_clock64();
      g_add( &d.counters[ 4 ], tp1 - tp0 );
      g_add( &d.counters[ 5 ], tp2 - tp0 );
      g_add( &d.counters[ 6 ], 1ull );
    }
  }
}

#ifdef NG_PROFILE
extern "C" int
nestgpu_profile_read( unsigned long long* out8, int reset )
{
  if ( hipMemcpyFromSymbol( out8, HIP_SYMBOL( g_phase_ticks ), sizeof( unsigned long long ) * 8 ) != hipSuccess )
    return 1;
  if ( reset )
  {
    unsigned long long z[ 8 ] = { 0, 0, 0, 0, 0, 0, 0, 0 };
    if ( hipMemcpyToSymbol( HIP_SYMBOL( g_phase_ticks ), z, sizeof z ) != hipSuccess )
      return 1;
  }
  return 0;
}
#endif

#ifndef NG_PART
// A slice split across Run calls: NEST's per-thread registers hold spikes part by part,
// so its receive order is (VP, part, node, lag). Rebuild that order once the slice is
// complete. One workgroup: for each (VP, part), each thread takes one block of the VP's
// range, counts its matching entries, a block scan gives the output offsets, and each
// thread copies its entries in list order.
constexpr int FLATTEN_BS = 1024;

__global__ void __launch_bounds__( FLATTEN_BS )
  k_flatten( NetDev* net, int par, int n_parts )
{
  __shared__ uint32_t sh[ FLATTEN_BS / 64 ];
  const NetDev& d = *net;
  const uint32_t P = d.n_blocks;
  const uint32_t t = threadIdx.x;
  uint32_t o = 0;  // output entries so far (the same in every thread)
  for ( int vp = 0; vp < d.n_vp; ++vp )
  {
    const uint32_t lo = d.vp_begin[ vp ], hi = d.vp_begin[ vp + 1 ];
    if ( lo >= hi )
      continue;
    // the blocks holding device indices lo .. hi - 1
    const uint32_t b0 = upper_bound_u32( d.bstart, P + 1, lo ) - 1;
    const uint32_t b1 = upper_bound_u32( d.bstart, P + 1, hi - 1 );
    for ( int p = 0; p < n_parts; ++p )
      for ( uint32_t c0 = b0; c0 < b1; c0 += FLATTEN_BS )
      {
        const uint32_t b = c0 + t;
        uint32_t n = 0, cnt = 0;
        const uint32_t* lst = nullptr;
        const uint8_t* lpart = nullptr;
        if ( b < b1 )
        {
          n = min( d.blk_cnt[ static_cast< size_t >( par ) * P + b ], d.spk_cap );
          lst = d.blk_spk + ( static_cast< size_t >( par ) * P + b ) * d.spk_cap;
          lpart = d.blk_part + ( static_cast< size_t >( par ) * P + b ) * d.spk_cap;
          for ( uint32_t q = 0; q < n; ++q )
          {
            const uint32_t dev = lst[ q ] >> 8;
            cnt += lpart[ q ] == p and dev >= lo and dev < hi ? 1u : 0u;
          }
        }
        uint32_t ex;
        const uint32_t tot = block_scan< FLATTEN_BS >( cnt, &ex, sh );
        __syncthreads();
        uint32_t w = o + ex;
        for ( uint32_t q = 0; q < n; ++q )
        {
          const uint32_t e = lst[ q ];
          const uint32_t dev = e >> 8;
          if ( lpart[ q ] != p or dev < lo or dev >= hi )
            continue;
          d.flat_src[ w ] = dev;
          d.flat_lag[ w ] = e & 0xffu;
          ++w;
        }
        o += tot;
      }
  }
  if ( t == 0 )
  {
    d.flat_meta[ par ] = o;
    d.flat_meta[ 2 + par ] = 1;
  }
}

#endif  // NG_PART

// ------------------------------------------------------------------ launch wrappers
// This file is compiled once per model set of a launch (NG_PART: the model id, or ALL_MODELS
// for launches with several models), which instantiates that set's slice kernels, and once
// without NG_PART for everything else, so that the instantiations build in parallel.
#define NG_LAUNCH_ARGS                                                                                  \
  const NetDev *nets, const uint32_t *blk_prefix, int n_nets, uint32_t total_blocks, int delivery, bool stdp, \
    int s, size_t dyn_lds, hipStream_t st
template < int MASK >
void launch_models( NG_LAUNCH_ARGS );

#ifdef NG_PART
template < int MASK >
void
launch_models( NG_LAUNCH_ARGS )
{
#define NG_LAUNCH( WIN, STDP, CACHE )                                                                        \
  k_slice< MASK, WIN, STDP, CACHE >                                                                   \
    <<< total_blocks, Tile< WIN >::BS, dyn_lds, st >>>( nets, blk_prefix, n_nets, s )
  if ( delivery == LAUNCH_WINDOW )
    stdp ? NG_LAUNCH( true, true, false ) : NG_LAUNCH( true, false, false );
  else if ( delivery == LAUNCH_GLOBAL )
    stdp ? NG_LAUNCH( false, true, false ) : NG_LAUNCH( false, false, false );
  else if constexpr ( MASK == ALL_MODELS )
    NG_LAUNCH( true, true, true );
#undef NG_LAUNCH
}

template void launch_models< NG_PART >( NG_LAUNCH_ARGS );
#else

// Dynamic LDS that limits the slice kernel to wg_per_cu resident workgroups per CU (0: no
// limit): fewer resident blocks keep the ring buffers they update within the XCD's L2.
size_t
slice_lds_for_occupancy( int wg_per_cu, bool win )
{
  if ( wg_per_cu <= 0 )
    return 0;
  const size_t own = win ? sizeof( SliceLds< true > ) : sizeof( SliceLds< false > );
  const size_t lds_per_cu = 160 * 1024;
  const size_t want = lds_per_cu / static_cast< size_t >( wg_per_cu + 1 ) + 256;  // more than 1/(k+1)
  return want > own ? want - own : 0;
}

hipError_t
launch_slice( const NetDev* nets, const uint32_t* blk_prefix, int n_nets, uint32_t total_blocks, int mask,
  int delivery, int s, size_t dyn_lds, hipStream_t st )
{
  // mask: one bit per model id of the launch, and MASK_STDP for stdp_synapse. A launch of one
  // model takes that model's own instantiation, any other the one with every model.
  const bool stdp = ( mask & MASK_STDP ) != 0;
  switch ( delivery == LAUNCH_CACHE ? ALL_MODELS : mask & ALL_MODELS )
  {
#define NG_ONE( ID )                                                                                                \
  case 1 << ( ID ):                                                                                                 \
    launch_models< 1 << ( ID ) >( nets, blk_prefix, n_nets, total_blocks, delivery, stdp, s, dyn_lds, st );              \
    break;
    NG_DEVICE_MODELS( NG_ONE )
#undef NG_ONE
  default:
    launch_models< ALL_MODELS >( nets, blk_prefix, n_nets, total_blocks, delivery, stdp, s, dyn_lds, st );
  }
  return hipGetLastError();
}

__global__ void
k_status( const NetDev* nets, int n_nets, unsigned long long* out )
{
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if ( i < n_nets )
  {
    out[ 2 * i ] = nets[ i ].counters[ 0 ];
    out[ 2 * i + 1 ] = *nets[ i ].log_n;
  }
}

hipError_t
launch_status( const NetDev* nets, int n_nets, unsigned long long* out, hipStream_t st )
{
  if ( n_nets > 0 )
    k_status<<< ( n_nets + 255 ) / 256, 256, 0, st >>>( nets, n_nets, out );
  return hipGetLastError();
}

// The launch record of a chunk as a kernel argument: 2 us of stream time instead of a copy from
// host memory.
static_assert( sizeof( NetDev ) <= 2048 and sizeof( NetDev ) % 8 == 0, "a launch record is a kernel argument" );
__global__ void
k_stage( const NetDev net, NetDev* out )
{
  const unsigned long long* src = reinterpret_cast< const unsigned long long* >( &net );
  unsigned long long* dst = reinterpret_cast< unsigned long long* >( out );
  for ( uint32_t i = threadIdx.x; i < sizeof( NetDev ) / 8; i += blockDim.x )
    dst[ i ] = src[ i ];
}

hipError_t
launch_stage( const NetDev& net, NetDev* out, hipStream_t st )
{
  k_stage<<< 1, 64, 0, st >>>( net, out );
  return hipGetLastError();
}

// ---- room in the post-spike history rings, between chunks

// doubles as signed integers of the same order
__device__ inline long long
ordered_key( double x )
{
  const long long b = __double_as_longlong( x );
  return b < 0 ? b ^ 0x7fffffffffffffffll : b;
}

// need[t]: (as an ordered key) the least t_lastspike - delay over the stdp synapses onto t, the
// t1 of the next get_history of each. One workgroup per source. stamp0: the source's spikes with
// later stamps are not delivered yet; their synapses will read from the spike before.
__global__ void
k_hist_need( const NetDev d, int64_t stamp0, long long* need )
{
  const uint32_t s = blockIdx.x;
  if ( glob( d.pre_row0 )[ s + 1 ] == glob( d.pre_row0 )[ s ] )
    return;
  gptr< const uint32_t > bo = glob( d.boff ) + static_cast< size_t >( s ) * ( d.n_blocks + 1 );
  for ( uint32_t b = threadIdx.x; b < d.n_blocks; b += blockDim.x )
  {
    const uint32_t dev0 = glob( d.bstart )[ b ], end = bo[ b + 1 ];
    for ( uint32_t k = bo[ b ]; k < end; ++k )
    {
      const uint32_t word = glob( d.syn )[ k ].word;
      if ( not( word & PLASTIC_BIT ) )
        continue;
      gref< const StdpPre > pre = glob( const_cast< const StdpPre* >( d.spre ) )[ glob( d.srow )[ k ] ];
      double t_last = pre.cur_tl;
      const int64_t stamp = llrint( t_last / d.ms_per_step );
      if ( stamp > stamp0 )
        t_last = pre.tl[ ( ( stamp - 1 ) / d.min_delay ) & 1 ];
      const uint32_t dsteps = ( ( word >> 16 ) & DELAY_MASK ) + static_cast< uint32_t >( d.min_delay );
      __hip_atomic_fetch_min( glob( need ) + dev0 + ( word & 0xffffu ),
        ordered_key( t_last - static_cast< double >( dsteps ) * d.ms_per_step ), __ATOMIC_RELAXED,
        __HIP_MEMORY_SCOPE_AGENT );
    }
  }
}

// The ring each neuron wants for chunks of up to span steps: the entries that a synapse has yet
// to read and the one before them (need; null: all entries), and the spikes of one chunk (a
// neuron spikes again after its refractory steps at the earliest), in half the ring: looking
// takes about 2 ms (21 million synapses), so a neuron asks again after half a ring of spikes.
__global__ void
k_hist_plan( const NetDev d, const long long* need, int64_t span, HistRing* plan )
{
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if ( i >= d.n )
    return;
  HistRing r = load_ring( glob( d.hist ) + i );
  if ( not glob( d.stdp_in )[ i ] )
  {
    plan[ i ] = r;
    return;
  }
  uint32_t lo = r.n > r.mask ? r.n - r.mask - 1u : 0u;
  if ( need )
  {
    const uint32_t first = lo;
    uint32_t hi = r.n;
    const long long key = glob( need )[ i ];
    while ( lo < hi )  // the first entry at t1 + eps or later
    {
      const uint32_t mid = lo + ( hi - lo ) / 2;
      const double t = glob( d.hist_t )[ r.base + ( mid & r.mask ) ];
      if ( ordered_key( t - STDP_EPS ) >= key )
        hi = mid;
      else
        lo = mid + 1;
    }
    // one more before it, and one for the rounding of t - eps against t1 + eps
    lo = lo > first + 2u ? lo - 2u : first;
  }
  const int64_t ref = max( glob( d.psets )[ glob( d.pidx )[ i ] ].refractory_counts, 0 );
  const uint64_t chunk = static_cast< uint64_t >( ( span + ref ) / ( ref + 1 ) );
  const uint64_t want = r.n - lo + chunk + 1u;
  uint64_t cap = static_cast< uint64_t >( r.mask ) + 1u;
  while ( want > cap / 2 and cap < ( 1ull << 31 ) )
    cap *= 2;
  r.mask = static_cast< uint32_t >( cap - 1u );
  const uint64_t lim = lo + cap - 1u - chunk;
  r.lim = lim < NONE ? static_cast< uint32_t >( lim ) : NONE - 1u;
  plan[ i ] = r;
}

// Entries into the rings of plan. One wave per neuron.
__global__ void
k_hist_move( const NetDev d, const HistRing* plan, double* hist_t, double* hist_k )
{
  const uint32_t i = ( blockIdx.x * blockDim.x + threadIdx.x ) >> 6;
  if ( i >= d.n or not glob( d.stdp_in )[ i ] )
    return;
  const HistRing r = load_ring( glob( d.hist ) + i ), q = load_ring( glob( plan ) + i );
  const uint32_t first = r.n > r.mask ? r.n - r.mask - 1u : 0u;
  for ( uint32_t k = first + ( threadIdx.x & 63u ); k < r.n; k += 64u )
  {
    const uint32_t from = r.base + ( k & r.mask ), to = q.base + ( k & q.mask );
    glob( hist_t )[ to ] = glob( d.hist_t )[ from ];
    glob( hist_k )[ to ] = glob( d.hist_k )[ from ];
  }
}

hipError_t
launch_hist_need( const NetDev& net, int64_t stamp0, long long* need, hipStream_t st )
{
  k_hist_need<<< net.n, 256, 0, st >>>( net, stamp0, need );
  return hipGetLastError();
}

hipError_t
launch_hist_plan( const NetDev& net, const long long* need, int64_t span, HistRing* plan, hipStream_t st )
{
  k_hist_plan<<< ( net.n + 255 ) / 256, 256, 0, st >>>( net, need, span, plan );
  return hipGetLastError();
}

hipError_t
launch_hist_move( const NetDev& net, const HistRing* plan, double* hist_t, double* hist_k, hipStream_t st )
{
  k_hist_move<<< ( net.n + 3 ) / 4, 256, 0, st >>>( net, plan, hist_t, hist_k );
  return hipGetLastError();
}

hipError_t
launch_flatten( NetDev* net, int par, int n_parts, hipStream_t st )
{
  k_flatten<<< 1, FLATTEN_BS, 0, st >>>( net, par, n_parts );
  return hipGetLastError();
}

#endif  // NG_PART

}  // namespace nestgpu
