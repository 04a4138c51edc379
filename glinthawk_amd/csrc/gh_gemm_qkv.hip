// q, k and v of few activation rows, f16: the product, RoPE and the cache append in one launch.
//
// The ring kernel (gh_gemm_ring.hip) fills the chip by cutting K, which leaves fp32 sums of every K range to be written, and a second kernel to read them, rotate
// and append.  wq, wk and wv together have enough rows for a share of them a CU (40 to 60 of 70B, 7B and 13B), so here a work-group takes its rows over the whole
// K range and finishes them itself.
//
//   work-group  8 waves, one work-group a CU: up to 64 weight rows x up to X activation rows, 128 k a step
//   ring        as in the ring kernel: a step's weights and activations straight into one of S LDS stages, S - 1 steps requested ahead, one barrier a step.  Few
//               weight rows make a short step, so it is twice as long as there: with 64 k the barrier and the trip through LDS (0.24 us) paced it
//   math        v_mfma_f32_16x16x32; the waves as 2 groups of weight rows x 2 of activation rows x 2 halves of a step's k, which read a third less LDS than
//               4 x 2 whole steps; the halves are added at the end
//   k order     every work-group starts at a step of its own and wraps around (rows a power of two apart in memory meet on few channels)
#include "gh_product.h"

#include <algorithm>
#include <type_traits>

namespace gh {

uint32_t gemm_ring_splits( uint64_t s, uint64_t r, uint64_t b, double* ns );
uint64_t gemm_ring_units();
bool gemm_kernel_forced();

namespace {

typedef __attribute__( ( address_space( 3 ) ) ) void* lds_ptr;

constexpr uint32_t QKV_ROWS = 64, QKV_K = 128;
[[maybe_unused]] constexpr uint32_t QKV_PAST_ROW = 0x80000000u;  // lane offset of a row that is not there
[[maybe_unused]] constexpr uint32_t QKV_PAST_STEP = 0x40000000u; // scalar offset of a step that is not there: past every descriptor, and with any lane offset below 2^32

// LDS rows of 64 k: weights of the first half of the step, of the second, activations likewise
template<int X>
struct QkvTile
{
  static constexpr int RT = 2, CT = X / 32;                                          // 16 x 16 tiles of a wave
  static constexpr int LOADS = (int)( 2 * ( QKV_ROWS + X ) / 64 );                    // of a wave a step, 8 rows each
  static constexpr int SLOTS = (int)( 2 * ( QKV_ROWS + X ) * 8 );                     // 16 bytes each, per stage
  static constexpr int S = 160 * 1024 / ( SLOTS * 16 ) < 6 ? 160 * 1024 / ( SLOTS * 16 ) : 6;
  static_assert( X % 32 == 0 && S >= 3 && 8 * CT * 64 <= SLOTS );
};
__device__ __forceinline__ uint32_t qkv_swizzle( uint32_t row ) { return ( row >> 1 ) & 7; } // 16 neighbouring rows over all slots of 256 bytes

// s % 8 == 0, 16-byte aligned operands; dim, kv_dim, head_size % 4 == 0; `share` (a multiple of 4, at most 64) weight rows of a work-group
template<int X>
__global__ __launch_bounds__( 512, 1 ) void gemm_qkv_kernel( __half* __restrict__ q, const __half* __restrict__ x, const __half* __restrict__ w, uint32_t s, uint32_t r, uint32_t b,
                                                             QkvRows rows, uint32_t share, uint32_t units )
{
#if defined( __HIP_DEVICE_COMPILE__ ) // the host's pass does not know the builtins inside the template
  typedef QkvTile<X> T;
  constexpr int RT = T::RT, CT = T::CT, N = T::LOADS, S = T::S;
  // separate arrays: the compiler keeps an LDS read behind the loads into its own array only
  __shared__ uint4 st0[T::SLOTS], st1[T::SLOTS], st2[T::SLOTS];
  __shared__ uint4 st3[S > 3 ? T::SLOTS : 1], st4[S > 4 ? T::SLOTS : 1], st5[S > 5 ? T::SLOTS : 1];
  typedef typename Mfma<__half>::x8 x8;
  const uint32_t unit = ( blockIdx.x & 7 ) * ( ( units + 7 ) >> 3 ) + ( blockIdx.x >> 3 ); // work-groups go to the XCDs in turn
  if ( ( blockIdx.x >> 3 ) >= ( units + 7 ) >> 3 || unit >= units ) {
    return; // (whole work-group)
  }
  const uint32_t wave = __builtin_amdgcn_readfirstlane( threadIdx.x >> 6 ), lane = threadIdx.x & 63;
  const uint32_t kg = wave & 1, tg = ( wave >> 1 ) & 1, rg = wave >> 2, fr = lane & 15, g4 = lane >> 4;
  const uint32_t ld = s * 2;
  const uint32_t first = unit * share, n_rows = min( share, r - first );
  const uint32_t n_steps = ( s + QKV_K - 1 ) / QKV_K, start = unit % n_steps;
  const char* w_base = reinterpret_cast<const char*>( w + (uint64_t)first * s );
  const char* x_base = reinterpret_cast<const char*>( x );

  // a token's cache row and position: here by the time the sums are
  __half* cache[CT];
  uint32_t at[CT];
#pragma unroll
  for ( int c = 0; c < CT; c++ ) {
    const uint32_t token = min( 16 * ( tg * CT + c ) + fr, b - 1 );
    cache[c] = static_cast<__half*>( rows.token_rows[token] );
    at[c] = rows.pos[token];
  }

  // load n of a wave: LDS rows 8 (8 n + wave) ..; a lane writes slot lane % 8 of row lane / 8, so it fetches the chunk that the swizzle keeps there (the same for all of its
  // loads).  Rows past the share (or the matrix) read as zero and cost nothing.
  const uint32_t chunk = ( lane & 7 ) ^ qkv_swizzle( wave * 8 + ( lane >> 3 ) );
  uint32_t off[N];
  bool past_k[N]; // of the last step, where s % 128 != 0: the next row's
#pragma unroll
  for ( int n = 0; n < N; n++ ) {
    const uint32_t row = ( 8 * n + wave ) * 8 + ( lane >> 3 );
    const uint32_t in_x = row - 2 * QKV_ROWS;
    const uint32_t half = n < 2 ? n : in_x / X, of = n < 2 ? row % QKV_ROWS : in_x % X;
    off[n] = of < ( n < 2 ? n_rows : b ) ? of * ld + half * 128 + chunk * 16 : QKV_PAST_ROW;
    past_k[n] = half * 8 + chunk >= ( s % QKV_K ) >> 3;
  }
  const uint32_t ragged_step = s % QKV_K != 0 ? n_steps - 1 : 0xffffffffu;

  auto fetch = [&]( uint4* stage, uint32_t j ) __attribute__( ( always_inline ) ) {
    const __amdgpu_buffer_rsrc_t w_rsrc = __builtin_amdgcn_make_buffer_rsrc( const_cast<char*>( w_base ), 0, (int)( n_rows * ld ), 0x00020000 );
    const __amdgpu_buffer_rsrc_t x_rsrc = __builtin_amdgcn_make_buffer_rsrc( const_cast<char*>( x_base ), 0, (int)( b * ld ), 0x00020000 );
    const uint32_t turned = j + start >= n_steps ? j + start - n_steps : j + start;
    const uint32_t kb = j < n_steps ? turned * ( QKV_K * 2 ) : QKV_PAST_STEP;
    const bool ragged = j < n_steps && turned == ragged_step;
#pragma unroll
    for ( int n = 0; n < N; n++ ) {
      const uint32_t from = off[n] | ( ragged && past_k[n] ? QKV_PAST_ROW : 0u );
      if ( n < 2 ) { // weights are read once: non-temporal
        __builtin_amdgcn_raw_ptr_buffer_load_lds( w_rsrc, (lds_ptr)( stage + ( 8 * n + wave ) * 64 ), 16, from, kb, 0, 2 );
      } else {
        __builtin_amdgcn_raw_ptr_buffer_load_lds( x_rsrc, (lds_ptr)( stage + ( 8 * n + wave ) * 64 ), 16, from, kb, 0, 0 );
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
        const uint32_t row = kg * QKV_ROWS + 16 * ( rg * RT + i ) + fr;
        fw[i][k] = __builtin_bit_cast( x8, stage[row * 8 + ( ( 4 * k + g4 ) ^ qkv_swizzle( row ) )] );
      }
#pragma unroll
      for ( int c = 0; c < CT; c++ ) {
        const uint32_t row = 2 * QKV_ROWS + kg * X + 16 * ( tg * CT + c ) + fr;
        fx[c][k] = __builtin_bit_cast( x8, stage[row * 8 + ( ( 4 * k + g4 ) ^ qkv_swizzle( row ) )] );
      }
    }
    fetch( freed, j + S - 1 );
#pragma unroll
    for ( int k = 0; k < 2; k++ ) {
#pragma unroll
      for ( int i = 0; i < RT; i++ ) {
#pragma unroll
        for ( int c = 0; c < CT; c++ ) {
          acc[i][c] = Mfma<__half>::k32( fw[i][k], fx[c][k], acc[i][c] );
        }
      }
    }
  };
#define GH_QKV_STAGE( i ) ( ( i ) % S == 0 ? st0 : ( i ) % S == 1 ? st1 : ( i ) % S == 2 ? st2 : ( i ) % S == 3 ? st3 : ( i ) % S == 4 ? st4 : st5 )
#pragma unroll
  for ( int i = 0; i < S - 1; i++ ) {
    fetch( GH_QKV_STAGE( i ), i );
  }
  uint32_t j = 0;
  for ( ; j + S <= n_steps; j += S ) {
#pragma unroll
    for ( int i = 0; i < S; i++ ) {
      step( GH_QKV_STAGE( i ), GH_QKV_STAGE( i + S - 1 ), j + i );
    }
  }
#pragma unroll
  for ( int i = 0; i < S - 1; i++ ) {
    if ( j + i < n_steps ) { // uniform across the work-group
      step( GH_QKV_STAGE( i ), GH_QKV_STAGE( i + S - 1 ), j + i );
    }
  }
#undef GH_QKV_STAGE
  __builtin_amdgcn_s_waitcnt( 0x0F70 ); // no load into LDS is under way any more
  __syncthreads();
  // The halves of k: the wave of half kg finishes its 16-row tile kg and hands the other one over.  Tile (i, c): row 16 (2 rg + i) + 4 g4 + v, activation row
  // 16 (CT tg + c) + fr.
  mfma_f32x4* handed = reinterpret_cast<mfma_f32x4*>( st0 );
#pragma unroll
  for ( int c = 0; c < CT; c++ ) {
#pragma unroll
    for ( int v = 0; v < 4; v++ ) {
      reinterpret_cast<float*>( &handed[( wave * CT + c ) * 64 + lane] )[v] = kg == 0 ? acc[1][c][v] : acc[0][c][v];
      acc[0][c][v] = kg == 0 ? acc[0][c][v] : acc[1][c][v];
    }
  }
  __syncthreads();
  const uint32_t row = 16 * ( rg * RT + kg ) + 4 * g4, ch = first + row; // four neighbouring rows of one head
  if ( row >= n_rows ) {
    return;
  }
  const __half *re = static_cast<const __half*>( rows.freq_real ), *im = static_cast<const __half*>( rows.freq_imag );
  union Four
  {
    uint2 raw;
    __half h[4];
  };
#pragma unroll
  for ( int c = 0; c < CT; c++ ) {
    const uint32_t token = 16 * ( tg * CT + c ) + fr;
    const mfma_f32x4 sum = acc[0][c] + handed[( ( wave ^ 1 ) * CT + c ) * 64 + lane];
    if ( token >= b ) {
      continue;
    }
    Four y;
#pragma unroll
    for ( int v = 0; v < 4; v++ ) {
      y.h[v] = from_f32<__half>( sum[v] );
    }
    // an empty context keeps its query unrotated and has no row, as in the unfused ops; v is stored as it is
    if ( ch < rows.dim + rows.kv_dim && cache[c] != nullptr ) {
      const uint64_t k = (uint64_t)at[c] * ( rows.head_size / 2 ) + ( ch % rows.head_size ) / 2;
#pragma unroll
      for ( int v = 0; v < 4; v += 2 ) {
        const float cs = to_f32( re[k + v / 2] ), sn = to_f32( im[k + v / 2] ), y0 = to_f32( y.h[v] ), y1 = to_f32( y.h[v + 1] );
        y.h[v] = from_f32<__half>( y0 * cs - y1 * sn );
        y.h[v + 1] = from_f32<__half>( y0 * sn + y1 * cs );
      }
    }
    if ( ch < rows.dim ) {
      *reinterpret_cast<uint2*>( q + (uint64_t)token * rows.dim + ch ) = y.raw;
    } else if ( cache[c] != nullptr ) {
      __half* dst = cache[c] + ( ch - rows.dim );
      if ( ( reinterpret_cast<uintptr_t>( dst ) & 7u ) == 0 ) {
        *reinterpret_cast<uint2*>( dst ) = y.raw;
      } else {
#pragma unroll
        for ( int v = 0; v < 4; v++ ) {
          dst[v] = y.h[v];
        }
      }
    }
  }
#endif
}

uint64_t qkv_share( uint64_t r )
{
  const uint64_t units = gemm_ring_units();
  return ( ( r + units - 1 ) / units + 3 ) / 4 * 4;
}

} // namespace

// Both routes, us in a graph with cold weights, product over K ranges and epilogue / this kernel, at 1, 32 and 64 rows: 7B (48 rows a CU, 4096 k) 21.7 / 18.3, 22.4 / 19.0,
// 25.7 / 22.8; 13B (60, 5120) 29.8 / 27.9, 32.6 / 30.1, 36.8 / 36.3; 70B (40, 8192) 31.8 / 30.8, 34.7 / 31.6, 39.0 / 39.1; 6144 x 4096 (24 rows a CU) 14.0 / 15.9, 16.0 / 16.2,
// 19.0 / 20.0.  So a step costs its weights at a CU's share of the memory's rate, or weights and activations at what L2 delivers to a CU (50 bytes a ns), but no less than its
// barrier and its trip through LDS; the other route its estimate and the second launch.  Every work-group reads all activations, and behind the kernels of a layer they come from
// beyond L2: from some 640 KB on what is left of the gain is lost there (a layer of 70B at 64 rows 3 us slower).  A tile of more than 64 activation rows gained nothing in a layer.
// Fewer than 32 rows a CU: the other route, also where this one would be a microsecond faster (a short K), so that small models sum in the order that wq and wkv alone have.
constexpr uint32_t QKV_LEAST = 32;
constexpr uint64_t QKV_MOST_BYTES = 640 << 10;
constexpr double QKV_START_NS = 4000.0, QKV_EPILOGUE_NS = 4200.0;
bool gemm_qkv_applicable( uint64_t s, uint64_t b, const void* x, const void* w, const void* q, const QkvRows& rows )
{
  const uint64_t r = rows.dim + 2ull * rows.kv_dim;
  const bool takes = !gemm_kernel_forced() && b > 0 && b <= 64 && b * s * sizeof( __half ) < QKV_MOST_BYTES && r <= 0x7fffffffull && qkv_share( r ) >= QKV_LEAST
         && qkv_share( r ) <= QKV_ROWS && s % 8 == 0 && s <= ( 1u << 21 ) // 64 rows of a descriptor are at most 2^28 bytes
         && rows.dim % 4 == 0 && rows.kv_dim % 4 == 0 && rows.head_size % 4 == 0
         && ( ( reinterpret_cast<uintptr_t>( x ) | reinterpret_cast<uintptr_t>( w ) | reinterpret_cast<uintptr_t>( q ) ) & 15u ) == 0;
  if ( !takes ) {
    return false;
  }
  const double share = (double)qkv_share( r ), steps = (double)( ( s + QKV_K - 1 ) / QKV_K );
  const double ns = QKV_START_NS + steps * std::max( { b <= 32 ? 380.0 : 450.0, share * 256.0 / 25.4, ( share + (double)b ) * 256.0 / 50.0 } );
  double other = 0.0;
  const uint32_t splits = gemm_ring_splits( s, r, b, &other );
  return ns < other + ( splits > 1 ? (double)( splits * b * r ) * 8.0 / 5000.0 : 0.0 ) + QKV_EPILOGUE_NS;
}
int gemm_qkv_launch( void* q, const void* x, const void* w, uint64_t s, uint64_t b, const QkvRows& rows, hipStream_t st )
{
  const uint64_t r = rows.dim + 2ull * rows.kv_dim;
  const uint32_t share = (uint32_t)qkv_share( r ), units = (uint32_t)( ( r + share - 1 ) / share );
  auto go = [&]( auto width ) {
    gemm_qkv_kernel<decltype( width )::value><<<( units + 7 ) / 8 * 8, 512, 0, st>>>( static_cast<__half*>( q ), static_cast<const __half*>( x ), static_cast<const __half*>( w ),
                                                                                     (uint32_t)s, (uint32_t)r, (uint32_t)b, rows, share, units );
  };
  if ( b <= 32 ) {
    go( std::integral_constant<int, 32> {} );
  } else {
    go( std::integral_constant<int, 64> {} );
  }
  GH_LAUNCH_CHECK();
  return GH_OK;
}

} // namespace gh
