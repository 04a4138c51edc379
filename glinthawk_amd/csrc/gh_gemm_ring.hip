// GEMM of up to some hundred activation rows: xout(b, r) = sum_p w(r, p) * x(b, p), f16 or bf16, fp32 accumulate.  Bound by the weights,
// which leave memory once, so everything else is arranged around keeping their loads in flight:
//
//   work-group  8 waves (one work-group per CU) take up to W weight rows, up to X activation rows and one K range, 64 k a step
//   ring        a step's weights and activations go straight from memory into one of S LDS stages (raw buffer loads to LDS, 16 bytes a
//               lane, no registers); S - 1 steps are requested ahead.  One barrier a step: behind it this step's stage has landed for
//               all waves, and the stage of the step before is free and is refilled at once.
//   math        v_mfma_f32_16x16x32, the waves as RG groups of weight rows by TG groups of activation rows
//   k order     with one slab of activation rows, a work-group starts a long K range at a step of its own and wraps around: rows are a power of two apart in memory, and
//               work-groups in lock step on one column range would meet on few channels (7B w1 + w3 at 8 rows: 35 us, rotated 29).  Several slabs read the same
//               weights and keep step, so that L2 serves all but one (7B wo at 1800 rows: 71 us, rotated 100)
//   XCDs        neighbouring work-groups of one K range on one XCD, whose L2 then holds that range of the activations
//
// Measured, cold weights (the streaming kernel, or from 65 rows on a register-staged 128 x 128 tile kernel with two work-groups a CU,
// before): 7B w1 + w3 with the gate at 32 rows 41 -> 30 us (6.0 TB/s), at 77 rows 63 -> 38, w2 at 32 rows 20 -> 17.5; 70B w2 at 64 rows
// 86 -> 77, at 128 rows 113 -> 85; 70B w1 + w3 at 64 rows 146 -> 144, at 128 rows 230 -> 156.  The tiles and the number of stages were
// taken from the same timings; with work-groups handed out in grid order instead, 70B w2 at 128 rows takes 106 us.
//
// Rows of the tile beyond a work-group's share (or the matrix) read as zero by the descriptor's bound and cost no memory traffic, so the
// plan may give work-groups any number of rows that suits the number of CUs.  The fp32 sums of K ranges are added by gemm_reduce_kernel
// (gh_gemm.hip) or the fused epilogues (gh_gemm_fused.hip).  Without a split, w1 and w3 share a launch that applies the SiLU gate.
#include "gh_product.h"

#include <algorithm>
#include <iterator>
#include <type_traits>

namespace gh {

uint64_t gemm_ring_units();

namespace {

typedef __attribute__( ( address_space( 3 ) ) ) void* lds_ptr;

constexpr int RING_THREADS = 512;
// Steps of a K range from which on a work-group starts at one of its own: a short range is over before the channels matter (7B wo, 8 to 16
// steps: 8.6 and 9.4 us either way), and all of its rows are summed in the one order whichever product they are part of.
[[maybe_unused]] constexpr uint32_t RING_TURN_STEPS = 17;
// What a K split costs beside its sums, in ns.  Products of a layer leave sums to the kernel that follows in any case, plain ones only with a split, for
// GEMM_REDUCE_NS, and the plan is the same for both, so that both give the same bits.  This keeps 512 k in one range up to 64 rows (512 x 512,
// plain: 9 us instead of 12) and cuts longer ones; with 2.6 us 2048 x 2048 at 512 rows would stay whole, 25.6 us with its norm instead of 21.8.
constexpr double RING_SPLIT_NS = 1600.0;
constexpr int RING_K = 64; // k a step: 8 chunks of 8 halves
[[maybe_unused]] constexpr uint32_t RING_PAST_ROW = 0x80000000u;  // lane offset of a row that is not there
[[maybe_unused]] constexpr uint32_t RING_PAST_STEP = 0x40000000u; // scalar offset of a step that is not there: no descriptor is longer
                                                                   // (gemm_ring_applicable), and with any lane offset it stays below 2^32

// what a work-group does with its sums
constexpr int RING_STORE = 0;   // round and store xout(b, r)
constexpr int RING_PARTIAL = 1; // fp32 sums of a K range, (splits, b, r)
constexpr int RING_GATE = 2;    // w = [w1 rows | w3 rows]: DType(silu(y1) * y3), as GateRows says (gh_product.h)

// a launch: work unit u = (split * row_blocks + row_block) * slabs + slab
struct RingCut
{
  uint32_t rows;       // weight rows (RING_GATE: output rows) per work-group, a multiple of 4
  uint32_t cols;       // activation rows per slab
  uint32_t row_blocks, slabs, splits;
  uint32_t steps;      // of 64 k per split
};

// loads per wave and step (8 rows each), and LDS stages: what 160 KiB hold (N = 4: four measured faster than five)
constexpr int ring_loads( uint32_t w, uint32_t x ) { return (int)( ( w + x + 63 ) / 64 ); }
constexpr int ring_stages( uint32_t w, uint32_t x ) { return ring_loads( w, x ) == 4 ? 4 : std::min( 6, 20 / ring_loads( w, x ) ); }

template<int W, int X>
struct RingTile
{
  static constexpr int TG = X <= 96 ? 2 : 4, RG = 8 / TG;
  static constexpr int RT = W / ( 16 * RG ), CT = X / ( 16 * TG ); // 16 x 16 tiles of a wave
  static constexpr int N = ring_loads( W, X ), S = ring_stages( W, X );
  static constexpr int SLOTS = N * 64 * 8; // 16 bytes each, per stage
  static_assert( S * SLOTS * 16 <= 160 * 1024 && S <= 6 && S >= 3 );
};

__device__ __forceinline__ uint32_t ring_swizzle( uint32_t row ) { return ( row >> 1 ) & 7; } // 16 neighbouring rows over all slots of 256 bytes

// s % 8 == 0, 16-byte aligned operands, every split at least one step
template<typename E, int W, int X, int MODE>
__global__ __launch_bounds__( RING_THREADS, 1 ) void gemm_ring_kernel( void* __restrict__ out, const E* __restrict__ x, const E* __restrict__ w, uint32_t s, uint32_t r,
                                                                      uint32_t b, GateRows gate, RingCut cut )
{
#if defined( __HIP_DEVICE_COMPILE__ ) // the host's pass does not know the builtins inside the template
  typedef RingTile<W, X> T;
  constexpr int RT = T::RT, CT = T::CT, N = T::N, S = T::S;
  // separate arrays: the compiler keeps an LDS read behind the loads into its own array only
  __shared__ uint4 st0[T::SLOTS], st1[T::SLOTS], st2[T::SLOTS];
  __shared__ uint4 st3[S > 3 ? T::SLOTS : 1], st4[S > 4 ? T::SLOTS : 1], st5[S > 5 ? T::SLOTS : 1];
  typedef typename Mfma<E>::x8 x8;
  const uint32_t units = cut.row_blocks * cut.slabs * cut.splits;
  const uint32_t unit = ( blockIdx.x & 7 ) * ( ( units + 7 ) >> 3 ) + ( blockIdx.x >> 3 ); // work-groups go to the XCDs in turn
  if ( ( blockIdx.x >> 3 ) >= ( units + 7 ) >> 3 || unit >= units ) {
    return; // (whole work-group)
  }
  const uint32_t slab = unit % cut.slabs, row_block = ( unit / cut.slabs ) % cut.row_blocks, split = unit / ( cut.slabs * cut.row_blocks );
  const uint32_t wave = __builtin_amdgcn_readfirstlane( threadIdx.x >> 6 ), lane = threadIdx.x & 63;
  const uint32_t rg = wave / T::TG, tg = wave % T::TG, fr = lane & 15, g4 = lane >> 4;
  const uint32_t ld = s * 2;
  const uint32_t first = row_block * cut.rows, n_rows = min( cut.rows, r - first );
  const uint32_t col0 = slab * cut.cols, n_cols = min( cut.cols, b - col0 );
  const uint32_t all_steps = ( s + RING_K - 1 ) / RING_K;
  const uint32_t step0 = split * cut.steps, n_steps = min( cut.steps, all_steps - step0 );
  const uint32_t start = n_steps < RING_TURN_STEPS || cut.slabs > 1 ? 0 : unit % n_steps;
  // RING_GATE: 16-row tiles of w1 and w3 in turn, so that the factors of an output meet in one lane; a wave loads from one of the two
  const uint64_t w_row0 = first + ( MODE == RING_GATE ? ( ( wave >> 1 ) & 1 ) * (uint64_t)r : 0 );
  const char* w_base = reinterpret_cast<const char*>( w + w_row0 * s );
  const char* x_base = reinterpret_cast<const char*>( x + (uint64_t)col0 * s );
  uint32_t off[N];
  // rows 8 id .. 8 id + 7 of the stage, id = 8 n + wave: the W weight rows, then the activation rows; a lane writes slot lane % 8 of row
  // lane / 8, so it fetches the chunk that the swizzle keeps there (the same for all of its loads)
  const uint32_t chunk = ( lane & 7 ) ^ ring_swizzle( wave * 8 + ( lane >> 3 ) );
#pragma unroll
  for ( int n = 0; n < N; n++ ) {
    const uint32_t row = ( 8 * n + wave ) * 8 + ( lane >> 3 );
    if ( row < W ) {
      const uint32_t of = MODE == RING_GATE ? ( row >> 5 ) * 16 + ( row & 15 ) : row;
      off[n] = of < n_rows ? of * ld + chunk * 16 : RING_PAST_ROW;
    } else {
      off[n] = row - W < n_cols ? ( row - W ) * ld + chunk * 16 : RING_PAST_ROW;
    }
  }
  const bool past_k = chunk >= ( ( s % RING_K ) >> 3 ); // of the last step, where s % 64 != 0: the next row's
  const uint32_t ragged_step = s % RING_K != 0 ? all_steps - 1 : 0xffffffffu;

  auto fetch = [&]( uint4* stage, uint32_t j ) __attribute__( ( always_inline ) ) {
    const __amdgpu_buffer_rsrc_t w_rsrc = __builtin_amdgcn_make_buffer_rsrc( const_cast<char*>( w_base ), 0, (int)( n_rows * ld ), 0x00020000 );
    const __amdgpu_buffer_rsrc_t x_rsrc = __builtin_amdgcn_make_buffer_rsrc( const_cast<char*>( x_base ), 0, (int)( n_cols * ld ), 0x00020000 );
    const uint32_t turned = j + start >= n_steps ? j + start - n_steps : j + start;
    const uint32_t kb = j < n_steps ? ( step0 + turned ) * ( RING_K * 2 ) : RING_PAST_STEP;
    const uint32_t mask = j < n_steps && step0 + turned == ragged_step && past_k ? RING_PAST_ROW : 0u;
#pragma unroll
    for ( int n = 0; n < N; n++ ) {
      const uint32_t id = 8 * n + wave;
      if ( 8 * n + 7 < W / 8 ) { // weights are read once: non-temporal
        __builtin_amdgcn_raw_ptr_buffer_load_lds( w_rsrc, (lds_ptr)( stage + id * 64 ), 16, off[n] | mask, kb, 0, 2 );
      } else {
        __builtin_amdgcn_raw_ptr_buffer_load_lds( x_rsrc, (lds_ptr)( stage + id * 64 ), 16, off[n] | mask, kb, 0, 0 );
      }
    }
  };
  mfma_f32x4 acc[RT][CT];
#pragma unroll
  for ( int i = 0; i < RT; i++ ) {
#pragma unroll
    for ( int c = 0; c < CT; c++ ) {
      acc[i][c] = mfma_f32x4 { 0.0f, 0.0f, 0.0f, 0.0f };
    }
  }
  constexpr int FLY = ( S - 2 ) * N; // this wave's loads behind the stage that a step waits for
  auto step = [&]( const uint4* stage, uint4* freed, uint32_t j ) __attribute__( ( always_inline ) ) {
    __builtin_amdgcn_sched_barrier( 0 );
    __builtin_amdgcn_s_waitcnt( 0x0F70 | ( FLY & 15 ) | ( ( FLY >> 4 ) << 14 ) ); // vmcnt( FLY )
    __builtin_amdgcn_s_barrier(); // this stage is here for all waves, and all are through with the one before
    __builtin_amdgcn_sched_barrier( 0 );
    x8 fw[RT][2], fx[CT][2];
#pragma unroll
    for ( int k = 0; k < 2; k++ ) {
#pragma unroll
      for ( int i = 0; i < RT; i++ ) {
        const uint32_t row = 16 * ( rg * RT + i ) + fr;
        fw[i][k] = __builtin_bit_cast( x8, stage[row * 8 + ( ( 4 * k + g4 ) ^ ring_swizzle( row ) )] );
      }
#pragma unroll
      for ( int c = 0; c < CT; c++ ) {
        const uint32_t row = W + 16 * ( tg * CT + c ) + fr;
        fx[c][k] = __builtin_bit_cast( x8, stage[row * 8 + ( ( 4 * k + g4 ) ^ ring_swizzle( row ) )] );
      }
    }
    fetch( freed, j + S - 1 );
#pragma unroll
    for ( int k = 0; k < 2; k++ ) {
#pragma unroll
      for ( int i = 0; i < RT; i++ ) {
#pragma unroll
        for ( int c = 0; c < CT; c++ ) {
          acc[i][c] = Mfma<E>::k32( fw[i][k], fx[c][k], acc[i][c] );
        }
      }
    }
  };
#define GH_RING_STAGE( i ) ( ( i ) % S == 0 ? st0 : ( i ) % S == 1 ? st1 : ( i ) % S == 2 ? st2 : ( i ) % S == 3 ? st3 : ( i ) % S == 4 ? st4 : st5 )
#pragma unroll
  for ( int i = 0; i < S - 1; i++ ) {
    fetch( GH_RING_STAGE( i ), i );
  }
  uint32_t j = 0;
  for ( ; j + S <= n_steps; j += S ) {
#pragma unroll
    for ( int i = 0; i < S; i++ ) {
      step( GH_RING_STAGE( i ), GH_RING_STAGE( i + S - 1 ), j + i );
    }
  }
#pragma unroll
  for ( int i = 0; i < S - 1; i++ ) {
    if ( j + i < n_steps ) { // uniform across the work-group
      step( GH_RING_STAGE( i ), GH_RING_STAGE( i + S - 1 ), j + i );
    }
  }
#undef GH_RING_STAGE
  __builtin_amdgcn_s_waitcnt( 0x0F70 ); // no load into LDS outlives the work-group
  // acc[i][c][v]: row 16 (rg RT + i) + 4 g4 + v of the tile, activation row 16 (tg CT + c) + fr of the slab
#pragma unroll
  for ( int c = 0; c < CT; c++ ) {
    const uint32_t col = 16 * ( tg * CT + c ) + fr;
    if ( col >= n_cols ) {
      continue;
    }
    if constexpr ( MODE == RING_GATE ) {
      if ( gate.context_rows != nullptr && gate.context_rows[( col0 + col ) / gate.n_tokens] == nullptr ) {
        continue;
      }
#pragma unroll
      for ( int i = 0; i < RT; i += 2 ) {
        const uint32_t row = 16 * ( ( rg * RT + i ) / 2 ) + 4 * g4;
        union
        {
          uint2 raw;
          E h[4];
        } y;
#pragma unroll
        for ( int v = 0; v < 4; v++ ) {
          y.h[v] = gated<E>( gate, acc[i][c][v], acc[i + 1][c][v], min( first + row + v, r - 1 ), r );
        }
        if ( row < n_rows ) { // r % 4 == 0: all four
          *reinterpret_cast<uint2*>( static_cast<E*>( out ) + ( col0 + col ) * gate.stride + first + row ) = y.raw;
        }
      }
    } else {
#pragma unroll
      for ( int i = 0; i < RT; i++ ) {
        const uint32_t row = 16 * ( rg * RT + i ) + 4 * g4;
        const bool whole = row + 3 < n_rows && ( r & 3 ) == 0;
        if constexpr ( MODE == RING_PARTIAL ) {
          float* dst = static_cast<float*>( out ) + ( (uint64_t)split * b + col0 + col ) * r + first + row;
          if ( whole ) {
            *reinterpret_cast<mfma_f32x4*>( dst ) = acc[i][c];
          } else {
#pragma unroll
            for ( int v = 0; v < 4; v++ ) {
              if ( row + v < n_rows ) {
                dst[v] = acc[i][c][v];
              }
            }
          }
        } else {
          E* dst = static_cast<E*>( out ) + ( (uint64_t)col0 + col ) * r + first + row;
          union
          {
            uint2 raw;
            E h[4];
          } y;
#pragma unroll
          for ( int v = 0; v < 4; v++ ) {
            y.h[v] = from_f32<E>( acc[i][c][v] );
          }
          if ( whole ) {
            *reinterpret_cast<uint2*>( dst ) = y.raw;
          } else {
#pragma unroll
            for ( int v = 0; v < 4; v++ ) {
              if ( row + v < n_rows ) {
                dst[v] = y.h[v];
              }
            }
          }
        }
      }
    }
  }
#endif
}

template<typename E, int W, int X>
void ring_launch_tile( int mode, void* out, const E* x, const E* w, uint32_t s, uint32_t r, uint32_t b, const GateRows& gate, const RingCut& cut, hipStream_t st )
{
  const unsigned grid = ( cut.row_blocks * cut.slabs * cut.splits + 7 ) / 8 * 8;
  if ( mode == RING_STORE ) {
    gemm_ring_kernel<E, W, X, RING_STORE><<<grid, RING_THREADS, 0, st>>>( out, x, w, s, r, b, gate, cut );
  } else if ( mode == RING_PARTIAL ) {
    gemm_ring_kernel<E, W, X, RING_PARTIAL><<<grid, RING_THREADS, 0, st>>>( out, x, w, s, r, b, gate, cut );
  } else {
    gemm_ring_kernel<E, W, X, RING_GATE><<<grid, RING_THREADS, 0, st>>>( out, x, w, s, r, b, gate, cut );
  }
}

struct RingPlan
{
  uint32_t w, x; // the tile
  RingCut cut;
  double ns; // estimate: the launch, and the sums of a K split written and read
};

template<typename E>
int ring_launch( int mode, void* out, const E* x, const E* w, uint64_t s, uint64_t r, uint64_t b, const GateRows& gate, const RingPlan& plan, hipStream_t st )
{
  auto go = [&]( auto tile ) {
    ring_launch_tile<E, decltype( tile )::w, decltype( tile )::x>( mode, out, x, w, (uint32_t)s, (uint32_t)r, (uint32_t)b, gate, plan.cut, st );
  };
#define GH_RING_TILE( W, X )                                                                                                                                                     \
  if ( plan.w == W && plan.x == X ) {                                                                                                                                            \
    struct Tile                                                                                                                                                                  \
    {                                                                                                                                                                            \
      enum : int { w = W, x = X };                                                                                                                                               \
    };                                                                                                                                                                           \
    go( Tile {} );                                                                                                                                                               \
    GH_LAUNCH_CHECK();                                                                                                                                                           \
    return GH_OK;                                                                                                                                                                \
  }
  GH_RING_TILE( 128, 32 )
  GH_RING_TILE( 256, 32 )
  GH_RING_TILE( 128, 64 )
  GH_RING_TILE( 256, 64 )
  GH_RING_TILE( 128, 96 )
  GH_RING_TILE( 256, 96 )
  GH_RING_TILE( 128, 128 )
  GH_RING_TILE( 256, 128 )
  GH_RING_TILE( 128, 192 )
  GH_RING_TILE( 128, 256 )
#undef GH_RING_TILE
  return fail( GH_ERR_INVALID, "gh_matmul: no ring kernel of a %u x %u tile", plan.w, plan.x );
}

int g_ring_cus = 0; // tuning override of the CU count the plan balances for (0: the device's)

// The tile, the rows of a work-group and the K split.  A CU takes one work-group at a time, so a launch is as slow as its rounds of
// work-groups.  Fitted to timings of the 7B, 13B and 70B shapes, up to 256 rows with cold weights, and 300 to 7000.  A step costs its
// weights at the CU's share of the memory's rate (4.7 ns a row) and its activations at what L2 delivers to a CU (2 ns a row), but no
// less than a load's time in flight (1.9 us) over the steps requested ahead; 1.5 us with the gate in wide tiles, whose ring_plan() is weighed against two
// launches (2 x 11008 of 4096 k at 77 rows: 37 us so, 43 as two, for which 1.9 us spoke; 2 x 5632 of 2048 at 65: 18 and 23).  With several slabs the weights come from L2 and the
// matrix units set the pace; wide slabs slow each other down.  A round costs what it takes to fill the ring, and a split the fp32 sums
// that are written and read again, and RING_SPLIT_NS.  A work-group that fills three wide stages
// first starts later (4096 x 512 at 256 rows: 16 us for 8 steps), of which the steps of a long range are priced to cover a part.
RingPlan find_ring_plan( uint64_t s, uint64_t r, uint64_t b, bool gate, uint64_t n_cu )
{
  constexpr uint32_t XS[] = { 32, 64, 96, 128, 192, 256 };
  const uint64_t steps = ( s + RING_K - 1 ) / RING_K;
  RingPlan best {};
  for ( uint32_t x : XS ) {
    if ( b <= 256 ? x < b || best.w != 0 : x < 128 ) {
      continue; // up to 256 activation rows: the narrowest tile that takes them at once (a wider one has no more stages)
    }
    const uint64_t slabs = ( b + x - 1 ) / x, cols = ( ( b + slabs - 1 ) / slabs + 15 ) / 16 * 16;
    for ( uint32_t w = 128; w <= ( x <= 128 ? 256u : 128u ); w += 128 ) {
      const uint64_t most = gate ? w / 2 : w;
      for ( uint64_t want = 1; want <= ( gate ? 1u : 16u ); want++ ) {
        const uint64_t per = ( steps + want - 1 ) / want, splits = ( steps + per - 1 ) / per;
        if ( splits != want || ( splits > 1 && per < 4 ) ) {
          continue; // the plan of a smaller split; nothing to pipeline
        }
        // the fewest rounds that hold all rows, and one more
        uint64_t rounds = ( ( ( r + most - 1 ) / most ) * slabs * splits + n_cu - 1 ) / n_cu;
        for ( uint64_t end = rounds + 2; rounds < end; rounds++ ) {
          const uint64_t blocks = std::max<uint64_t>( 1, rounds * n_cu / ( slabs * splits ) );
          const uint64_t rows = std::min<uint64_t>( most, std::max<uint64_t>( 16, ( ( r + blocks - 1 ) / blocks + 3 ) / 4 * 4 ) );
          const uint64_t row_blocks = ( r + rows - 1 ) / rows;
          const double real_rounds = (double)( ( row_blocks * slabs * splits + n_cu - 1 ) / n_cu );
          const double w_rows = (double)( gate ? 2 * rows : rows ), x_rows = (double)std::min<uint64_t>( cols, b );
          const double flight_ns = gate && ring_stages( w, x ) < 6 ? 1500.0 : 1900.0;
          const double step_ns = slabs == 1 ? std::max( 4.7 * w_rows + 2.0 * x_rows, flight_ns / ( ring_stages( w, x ) - 1 ) )
                                            : 1.05 * ( 2.9 * w_rows + 1.05 * ( x_rows + x ) + ( x > 128 ? 20.0 + 7.0 * (double)slabs : 40.0 ) );
          const double start_ns = slabs > 1 ? 3000.0 : x < 192 ? 2000.0 : 2000.0 + 4000.0 * std::min( 1.0, 16.0 / (double)per );
          const double sums_ns = splits > 1 ? (double)( splits * b * r ) * 8.0 / 5000.0 + RING_SPLIT_NS : 0.0;
          const double cost = real_rounds * ( start_ns + (double)per * step_ns ) + sums_ns;
          if ( best.w == 0 || cost < best.ns ) {
            best = RingPlan { w, x, RingCut { (uint32_t)rows, (uint32_t)cols, (uint32_t)row_blocks, (uint32_t)slabs, (uint32_t)splits, (uint32_t)per }, cost };
          }
        }
      }
    }
  }
  return best;
}

// The plan of a product, asked for by the dispatch and again by the launch, and of the same products in every layer and step: the search
// (1 us up to 256 rows, 1.8 beyond) runs only when another product of this thread took the slot in between.  With a search at every call, of
// all widths (5 to 7 us up to 64 rows), the host needed 17 us for a product of 8 rows, 13 so.
RingPlan ring_plan( uint64_t s, uint64_t r, uint64_t b, bool gate )
{
  struct Slot
  {
    uint64_t s, r, b, n_cu;
    bool gate;
    RingPlan plan;
  };
  static thread_local Slot slots[64] {};
  const uint64_t n_cu = gemm_ring_units();
  const uint64_t mixed = ( ( s * 31 + r ) * 31 + b ) * 2 + ( gate ? 1 : 0 );
  Slot& slot = slots[( mixed * 0x9e3779b97f4a7c15ull ) >> 58];
  if ( slot.s != s || slot.r != r || slot.b != b || slot.n_cu != n_cu || slot.gate != gate ) { // (s > 0: an empty slot is no product's)
    slot = Slot { s, r, b, n_cu, gate, find_ring_plan( s, r, b, gate, n_cu ) };
  }
  return slot.plan;
}

} // namespace

// the compute units that plans are balanced for
uint64_t gemm_ring_units() { return g_ring_cus > 0 ? (uint64_t)g_ring_cus : (uint64_t)cu_count(); }

bool gemm_ring_applicable( uint64_t s, uint64_t r, uint64_t b, const void* x, const void* w, const void* xout )
{
  return s % 8 == 0 && s <= ( 1u << 21 ) // 256 rows of a descriptor are at most 2^30 bytes
         && r <= 0x7fffffffull && b <= 0x7fffffffull && ( r / 128 + 1 ) * ( b / 128 + 1 ) * 16 < ( 1ull << 31 )
         && ( ( reinterpret_cast<uintptr_t>( x ) | reinterpret_cast<uintptr_t>( w ) | reinterpret_cast<uintptr_t>( xout ) ) & 15u ) == 0;
}

// *ns: the estimate without the sums of a split
uint32_t gemm_ring_splits( uint64_t s, uint64_t r, uint64_t b, double* ns )
{
  const RingPlan plan = ring_plan( s, r, b, false );
  *ns = plan.cut.splits > 1 ? plan.ns - (double)( plan.cut.splits * b * r ) * 8.0 / 5000.0 - RING_SPLIT_NS : plan.ns;
  return plan.cut.splits;
}

// `partial`: the sums go there (gemm_ring_splits planes of (b, r)), else the rounded result to xout (one split)
template<typename E>
int gemm_ring_launch( E* xout, float* partial, const E* x, const E* w, uint64_t s, uint64_t r, uint64_t b, hipStream_t st )
{
  const RingPlan plan = ring_plan( s, r, b, false );
  GH_REQUIRE( partial != nullptr || plan.cut.splits == 1, "gh_matmul: a K split leaves fp32 sums" );
  return ring_launch<E>( partial ? RING_PARTIAL : RING_STORE, partial ? (void*)partial : (void*)xout, x, w, s, r, b, GateRows {}, plan, st );
}

// hb(b, hidden) = DType(silu(y1) * y3), y1 = x . w1^T, y3 = x . w3^T, w13 = w1 rows then w3 rows, in one launch
bool gemm_ring_gate_applicable( uint64_t s, uint64_t hidden, uint64_t b, const void* x, const void* w13, const void* hb, uint64_t hb_stride )
{
  return hidden % 4 == 0 && hb_stride % 4 == 0 && gemm_ring_applicable( s, 2 * hidden, b, x, w13, hb );
}
double gemm_ring_gate_ns( uint64_t s, uint64_t hidden, uint64_t b ) { return ring_plan( s, hidden, b, true ).ns; }

template<typename E>
int gemm_ring_gate_launch( E* hb, const GateRows& gate, const E* x, const E* w13, uint64_t s, uint64_t hidden, uint64_t b, hipStream_t st )
{
  return ring_launch<E>( RING_GATE, hb, x, w13, s, hidden, b, gate, ring_plan( s, hidden, b, true ), st );
}

void gemm_ring_tuning( int target_wgs )
{
  if ( target_wgs > 0 ) {
    g_ring_cus = target_wgs;
  }
}

int gemm_ring_cut( uint64_t s, uint64_t r, uint64_t b, bool gate, uint32_t* plan )
{
  const RingPlan p = ring_plan( s, r, b, gate );
  const uint32_t out[] = { p.w, p.x, p.cut.rows, p.cut.cols, p.cut.splits, p.cut.steps };
  std::copy( std::begin( out ), std::end( out ), plan );
  return GH_OK;
}

template int gemm_ring_launch<__half>( __half*, float*, const __half*, const __half*, uint64_t, uint64_t, uint64_t, hipStream_t );
template int gemm_ring_launch<__bf16>( __bf16*, float*, const __bf16*, const __bf16*, uint64_t, uint64_t, uint64_t, hipStream_t );
template int gemm_ring_gate_launch<__half>( __half*, const GateRows&, const __half*, const __half*, uint64_t, uint64_t, uint64_t, hipStream_t );
template int gemm_ring_gate_launch<__bf16>( __bf16*, const GateRows&, const __bf16*, const __bf16*, uint64_t, uint64_t, uint64_t, hipStream_t );

} // namespace gh
