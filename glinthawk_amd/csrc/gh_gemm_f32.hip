// fp32 products of a stage, alone and with the op that follows them.  Only small models run in fp32, at a handful of activation rows: a
// product then is a single read of a small matrix and the launch is bound by its one round trip to memory and by being a launch at
// all.  So a wave owns ROWS weight rows and requests the whole of a short row, with its pieces of the activations, before the first
// use, and what follows a product element by element (RoPE and the cache append, the residual add, the SiLU gate) is done where its
// sums are, with no second kernel.  15M model at 4 rows: q, k, v 7.4 + 4.4 us as product and follow-up kernel, 4.5 as one; w1, w3 7.3 + 4.7,
// 3.9; wo and w2 10.7, 3.7 with the add; classifier (32000 x 288) 23.0, 8.2.
//
// The RMS norm in front of a product is a launch of its own for a few rows that every wave of the product reads anyway.  Where a row is requested in
// one go (s <= what KU pieces cover) the wave squares what it holds and norms it before it multiplies, which takes a 15M layer from seven launches to
// five (norm and product as two launches / one, in a graph: 864 x 288 at 4 rows 5.1 / 3.2 us, 32000 x 288 10.4 / 9.2, which zeros in the place of what is past a row's end,
// an instruction an element, made 3.5 and 10.1, 4096 x 512 at 8 rows 5.9 and 7.5).
#include "gh_common.h"

#include <algorithm>

namespace gh {
namespace {

// what a wave does with the sums of its ROWS weight rows for activation row `col`; unit: index of the wave
struct F32Plain
{
  static constexpr bool NORMED = true; // the norm in front of the product may ride along
  float* out;
  uint32_t r;
  template<int ROWS>
  __device__ __forceinline__ uint32_t row( uint32_t unit, int i ) const
  {
    return unit * ROWS + i;
  }
  template<int ROWS>
  __device__ __forceinline__ void store( uint32_t unit, uint32_t col, const float ( &y )[ROWS] ) const
  {
#pragma unroll
    for ( int i = 0; i < ROWS; i++ ) {
      if ( unit * ROWS + i < r ) {
        out[(uint64_t)col * r + unit * ROWS + i] = y[i];
      }
    }
  }
};

struct F32Accum
{
  static constexpr bool NORMED = false;
  float* residual;
  uint32_t r;
  template<int ROWS>
  __device__ __forceinline__ uint32_t row( uint32_t unit, int i ) const
  {
    return unit * ROWS + i;
  }
  template<int ROWS>
  __device__ __forceinline__ void store( uint32_t unit, uint32_t col, const float ( &y )[ROWS] ) const
  {
#pragma unroll
    for ( int i = 0; i < ROWS; i++ ) {
      if ( unit * ROWS + i < r ) {
        residual[(uint64_t)col * r + unit * ROWS + i] += y[i];
      }
    }
  }
};

// half of a wave's rows are of w1, the others the same outputs' of w3
struct F32Gate
{
  static constexpr bool NORMED = true;
  float* hb;
  uint32_t hidden;
  template<int ROWS>
  __device__ __forceinline__ uint32_t row( uint32_t unit, int i ) const
  {
    const uint32_t j = min( unit * ( ROWS / 2 ) + i % ( ROWS / 2 ), hidden - 1 );
    return i < ROWS / 2 ? j : hidden + j;
  }
  template<int ROWS>
  __device__ __forceinline__ void store( uint32_t unit, uint32_t col, const float ( &y )[ROWS] ) const
  {
#pragma unroll
    for ( int i = 0; i < ROWS / 2; i++ ) {
      const uint32_t j = unit * ( ROWS / 2 ) + i;
      if ( j < hidden ) {
        hb[(uint64_t)col * hidden + j] = y[i] / ( 1.0f + __expf( -y[i] ) ) * y[ROWS / 2 + i];
      }
    }
  }
};

// rows [0, dim) q, [dim, dim + kv_dim) k, then v; a wave's rows are whole pairs
struct F32Qkv
{
  static constexpr bool NORMED = true;
  float *q, *kv_out;
  const uint32_t* pos;
  const float *freq_real, *freq_imag;
  void* const* token_rows;
  uint32_t dim, kv_dim, head_size, r;
  template<int ROWS>
  __device__ __forceinline__ uint32_t row( uint32_t unit, int i ) const
  {
    return unit * ROWS + i;
  }
  template<int ROWS>
  __device__ __forceinline__ void store( uint32_t unit, uint32_t col, const float ( &y )[ROWS] ) const
  {
    float* cache = static_cast<float*>( token_rows[col] );
    const uint64_t p = pos[col];
#pragma unroll
    for ( int i = 0; i < ROWS; i += 2 ) {
      const uint32_t c = unit * ROWS + i;
      if ( c >= r ) {
        continue;
      }
      if ( kv_out != nullptr && c >= dim ) { // unrotated
        kv_out[(uint64_t)col * 2 * kv_dim + ( c - dim )] = y[i];
        kv_out[(uint64_t)col * 2 * kv_dim + ( c - dim ) + 1] = y[i + 1];
      }
      // an empty context keeps its query unrotated and has no row, as in the unfused ops; v is stored as it is
      float o0 = y[i], o1 = y[i + 1];
      if ( cache != nullptr && c < dim + kv_dim ) {
        const uint64_t k = p * ( head_size / 2 ) + ( c % head_size ) / 2;
        const float fcr = freq_real[k], fci = freq_imag[k];
        o0 = y[i] * fcr - y[i + 1] * fci;
        o1 = y[i] * fci + y[i + 1] * fcr;
      }
      if ( c < dim ) {
        q[(uint64_t)col * dim + c] = o0;
        q[(uint64_t)col * dim + c + 1] = o1;
      } else if ( cache != nullptr ) {
        cache[c - dim] = o0;
        cache[c - dim + 1] = o1;
      }
    }
  }
};

// Sums over the wave of a value for each of COLS activation rows: the lanes of column_of_lane() = c end up with row c's.  With a sum a row all over the
// wave, a product of a few rows spends more on these than on its dot products.  Instead two rows' halves change places and are added in one go, until a lane holds only its own
// row's (with the norm, 864 x 288 at 4 rows: 4.05 -> 3.5 us, at 8 6.0 -> 4.6; 32000 x 288 at 4: 13.2 -> 8.8, at 8 25.1 -> 13.0).
template<int COLS>
__device__ __forceinline__ uint32_t column_of_lane( uint32_t lane )
{
  return COLS == 1 ? 0 : COLS == 4 ? lane >> 4 : ( lane >> 4 ) + ( ( lane >> 3 ) & 1 ) * 4;
}
template<int COLS>
__device__ __forceinline__ float column_sum( const float ( &v )[COLS], uint32_t lane )
{
  static_assert( COLS == 1 || COLS == 4 || COLS == 8 );
  if constexpr ( COLS == 1 ) {
    return wave_sum( v[0] );
  } else if constexpr ( COLS == 4 ) {
    return row16_sum( sum_rows( sum_halves( v[0], v[2] ), sum_halves( v[1], v[3] ) ) );
  } else {
    const bool high = ( lane & 8 ) != 0;
    float u[4];
#pragma unroll
    for ( int c = 0; c < 4; c++ ) { // the halves of a row of 16 lanes: a rotation by 8
      const float keep = high ? v[c + 4] : v[c], give = high ? v[c] : v[c + 4];
      u[c] = keep + __builtin_bit_cast( float, __builtin_amdgcn_update_dpp( 0, __builtin_bit_cast( int, give ), 0x128, 0xF, 0xF, true ) );
    }
    float s = sum_rows( sum_halves( u[0], u[2] ), sum_halves( u[1], u[3] ) );
    s += dpp_quad_xor1( s );
    s += dpp_quad_xor2( s );
    return s + dpp_half_mirror( s );
  }
}

constexpr int f32_pieces( int rows ) { return rows <= 2 ? 4 : 2; } // of a row under way at once

// V: elements per load (4: s % 4 == 0, 16-byte aligned operands).  COLS activation rows at a time, `cols_per_y` of them per grid row.
// NORM: the activations are x normed by their root mean square, times `norm`; s <= f32_pieces( ROWS ) * 64 * V.
template<int ROWS, int COLS, int V, bool NORM, typename Epilogue>
__global__ __launch_bounds__( 256 ) void gemm_f32_kernel( Epilogue epi, const float* __restrict__ x, const float* __restrict__ norm, const float* __restrict__ w, uint32_t s,
                                                          uint32_t r, uint32_t b, uint32_t units, uint32_t cols_per_y )
{
  constexpr int KU = f32_pieces( ROWS );
  typedef float vec __attribute__( ( ext_vector_type( V ) ) );
  const uint32_t unit = blockIdx.x * 4 + ( threadIdx.x >> 6 );
  if ( unit >= units ) {
    return;
  }
  const uint32_t lane = threadIdx.x & 63;
  const float* wr[ROWS];
#pragma unroll
  for ( int i = 0; i < ROWS; i++ ) {
    wr[i] = w + (uint64_t)min( epi.template row<ROWS>( unit, i ), r - 1 ) * s; // a row past the last repeats it and is not stored
  }
  const uint32_t c_end = min( b, ( blockIdx.y + 1 ) * cols_per_y );
  for ( uint32_t c0 = blockIdx.y * cols_per_y; c0 < c_end; c0 += COLS ) {
    const float* xc[COLS];
#pragma unroll
    for ( int c = 0; c < COLS; c++ ) {
      xc[c] = x + (uint64_t)min( c0 + c, b - 1 ) * s;
    }
    float acc[ROWS][COLS];
#pragma unroll
    for ( int i = 0; i < ROWS; i++ ) {
#pragma unroll
      for ( int c = 0; c < COLS; c++ ) {
        acc[i][c] = 0.0f;
      }
    }
    auto step = [&]( uint32_t k0, auto tail ) __attribute__( ( always_inline ) ) {
      vec a[KU][ROWS], y[KU][COLS], gain[KU];
#pragma unroll
      for ( int u = 0; u < KU; u++ ) {
        const uint32_t p = k0 + ( u * 64 + lane ) * V;
        const bool in = !tail.value || p < s; // past the row's end: the first elements again, as zeros
        const uint32_t at = in ? p : 0;
#pragma unroll
        for ( int i = 0; i < ROWS; i++ ) {
          a[u][i] = *reinterpret_cast<const vec*>( wr[i] + at );
        }
#pragma unroll
        for ( int c = 0; c < COLS; c++ ) {
          y[u][c] = *reinterpret_cast<const vec*>( xc[c] + at );
        }
        if constexpr ( NORM ) {
          gain[u] = *reinterpret_cast<const vec*>( norm + at );
        }
      }
      if constexpr ( NORM ) { // as rmsnorm_kernel: the mean, the root, one rounding of each product
        float ss[COLS];
#pragma unroll
        for ( int c = 0; c < COLS; c++ ) {
          ss[c] = 0.0f;
#pragma unroll
          for ( int u = 0; u < KU; u++ ) {
            if ( ( u * 64 + lane ) * V < s ) {
#pragma unroll
              for ( int e = 0; e < V; e++ ) {
                ss[c] += y[u][c][e] * y[u][c][e];
              }
            }
          }
        }
        const float own = 1.0f / sqrtf( column_sum<COLS>( ss, lane ) / (float)s + 1e-5f );
#pragma unroll
        for ( int c = 0; c < COLS; c++ ) {
          const float inv = lane_value( own, COLS == 1 ? 0 : ( c & 3 ) * 16 + ( c >> 2 ) * 8 );
#pragma unroll
          for ( int u = 0; u < KU; u++ ) {
#pragma unroll
            for ( int e = 0; e < V; e++ ) {
              y[u][c][e] = gain[u][e] * ( inv * y[u][c][e] );
            }
          }
        }
      }
#pragma unroll
      for ( int u = 0; u < KU; u++ ) {
        const bool in = !tail.value || k0 + ( u * 64 + lane ) * V < s;
        // Lanes past the row's end take no part.  With the norm in front everything is here by now and instructions are what counts: they sit a branch out; without it
        // the first piece's products run while the others are under way, and a branch would end that (4096 x 512 at 4 rows 4.1 us, 4.0 with zeros in their place).
        if constexpr ( NORM ) {
          if ( in ) {
#pragma unroll
            for ( int e = 0; e < V; e++ ) {
#pragma unroll
              for ( int i = 0; i < ROWS; i++ ) {
#pragma unroll
                for ( int c = 0; c < COLS; c++ ) {
                  acc[i][c] += a[u][i][e] * y[u][c][e];
                }
              }
            }
          }
        } else {
#pragma unroll
          for ( int e = 0; e < V; e++ ) {
#pragma unroll
            for ( int i = 0; i < ROWS; i++ ) {
              const float av = in ? a[u][i][e] : 0.0f;
#pragma unroll
              for ( int c = 0; c < COLS; c++ ) {
                acc[i][c] += av * ( in ? y[u][c][e] : 0.0f );
              }
            }
          }
        }
      }
    };
    if constexpr ( NORM ) {
      step( 0, std::true_type {} );
    } else {
      uint32_t k0 = 0;
      for ( ; k0 + KU * 64 * V <= s; k0 += KU * 64 * V ) {
        step( k0, std::false_type {} );
      }
      if ( k0 < s ) {
        step( k0, std::true_type {} );
      }
    }
    float mine[ROWS]; // of the activation row that is this lane's
#pragma unroll
    for ( int i = 0; i < ROWS; i++ ) {
      mine[i] = column_sum<COLS>( acc[i], lane );
    }
    const uint32_t col = c0 + column_of_lane<COLS>( lane );
    if ( ( lane & ( COLS == 1 ? 63u : COLS == 4 ? 15u : 7u ) ) == 0 && col < c_end ) {
      epi.template store<ROWS>( unit, col, mine );
    }
  }
}

// Rows per wave: two where that leaves at most two work-groups a CU, i.e. where latency is all there is; else four, which read the
// activations half as often.  8 activation rows at a time where there are more than 4; a single one alone (864 x 288 at 1 row: 3.4 us, 5.0 as four).
template<int ROWS, int COLS, typename Epilogue>
int launch_cols( const Epilogue& epi, const float* x, const float* norm, const float* w, uint64_t s, uint64_t r, uint64_t b, uint64_t units, hipStream_t st )
{
  // Activation rows are shared out over the grid until there are some four work-groups a CU, at most 64 rows in turn to one: 864 x 288 at 16 rows 6.0 -> 4.2 us,
  // at 128 16.5 -> 12.8, 64 x 32 at 128 16 -> 4.3.
  const uint64_t groups = ( units + 3 ) / 4, shares = ( 4 * (uint64_t)cu_count() + groups - 1 ) / groups;
  auto eights = []( uint64_t n, uint64_t parts ) { return ( ( n + parts - 1 ) / parts + 7 ) / 8 * 8; };
  const uint64_t cols = std::max( std::min<uint64_t>( 64, eights( b, shares ) ), eights( b, 65535 ) );
  const dim3 grid( (unsigned)groups, (unsigned)( ( b + cols - 1 ) / cols ) );
  auto go = [&]( auto v, auto normed ) {
    gemm_f32_kernel<ROWS, COLS, decltype( v )::value, decltype( normed )::value>
      <<<grid, 256, 0, st>>>( epi, x, norm, w, (uint32_t)s, (uint32_t)r, (uint32_t)b, (uint32_t)units, (uint32_t)cols );
  };
  const bool whole = s % 4 == 0 && ( ( reinterpret_cast<uintptr_t>( x ) | reinterpret_cast<uintptr_t>( w ) ) & 15u ) == 0;
  if constexpr ( Epilogue::NORMED ) {
    if ( norm != nullptr ) {
      GH_REQUIRE( whole && s <= f32_pieces( ROWS ) * 64 * 4 && ( reinterpret_cast<uintptr_t>( norm ) & 15u ) == 0, "fp32 product: no norm in a launch of this shape" );
      go( std::integral_constant<int, 4> {}, std::true_type {} );
      GH_LAUNCH_CHECK();
      return GH_OK;
    }
  }
  whole ? go( std::integral_constant<int, 4> {}, std::false_type {} ) : go( std::integral_constant<int, 1> {}, std::false_type {} );
  GH_LAUNCH_CHECK();
  return GH_OK;
}
int rows_per_wave( uint64_t weight_rows ) { return weight_rows <= 4096 ? 2 : 4; }
// `outputs`: what the waves share out, `per`: weight rows to one of them
template<typename Epilogue>
int launch_f32( const Epilogue& epi, const float* x, const float* norm, const float* w, uint64_t s, uint64_t r, uint64_t b, uint64_t outputs, uint64_t per, hipStream_t st )
{
  if ( rows_per_wave( outputs * per ) == 2 ) {
    const uint64_t units = ( outputs * per + 1 ) / 2;
    return b == 1   ? launch_cols<2, 1>( epi, x, norm, w, s, r, b, units, st )
           : b <= 4 ? launch_cols<2, 4>( epi, x, norm, w, s, r, b, units, st )
                    : launch_cols<2, 8>( epi, x, norm, w, s, r, b, units, st );
  }
  const uint64_t units = ( outputs * per + 3 ) / 4;
  return b == 1   ? launch_cols<4, 1>( epi, x, norm, w, s, r, b, units, st )
         : b <= 4 ? launch_cols<4, 4>( epi, x, norm, w, s, r, b, units, st )
                  : launch_cols<4, 8>( epi, x, norm, w, s, r, b, units, st );
}

} // namespace

// Whether the norm of the activations can ride in a product of r weight rows (w1 and w3 together): a row in one request, aligned operands.
bool gemm_f32_norm_fits( uint64_t s, uint64_t r, const void* x, const void* norm, const void* w )
{
  return s % 4 == 0 && s <= (uint64_t)f32_pieces( rows_per_wave( r ) ) * 64 * 4
         && ( ( reinterpret_cast<uintptr_t>( x ) | reinterpret_cast<uintptr_t>( norm ) | reinterpret_cast<uintptr_t>( w ) ) & 15u ) == 0;
}

// `norm` (gemm_f32_norm_fits) or NULL: weights of the norm that the activations go through first
int gemm_f32( float* out, const float* x, const float* norm, const float* w, uint64_t s, uint64_t r, uint64_t b, hipStream_t st )
{
  return launch_f32( F32Plain { out, (uint32_t)r }, x, norm, w, s, r, b, r, 1, st );
}
int gemm_f32_accum( float* residual, const float* x, const float* w, uint64_t s, uint64_t r, uint64_t b, hipStream_t st )
{
  return launch_f32( F32Accum { residual, (uint32_t)r }, x, nullptr, w, s, r, b, r, 1, st );
}
int gemm_f32_gate( float* hb, const float* x, const float* norm, const float* w13, uint64_t s, uint64_t hidden, uint64_t b, hipStream_t st )
{
  return launch_f32( F32Gate { hb, (uint32_t)hidden }, x, norm, w13, s, 2 * hidden, b, hidden, 2, st );
}
int gemm_f32_qkv( float* q, float* kv_out, const float* x, const float* norm, const float* wqkv, uint64_t s, uint64_t b, const uint32_t* pos, const float* freq_real,
                  const float* freq_imag, void* const* token_rows, uint32_t dim, uint32_t kv_dim, uint32_t head_size, hipStream_t st )
{
  const uint64_t r = (uint64_t)dim + 2ull * kv_dim;
  return launch_f32( F32Qkv { q, kv_out, pos, freq_real, freq_imag, token_rows, dim, kv_dim, head_size, (uint32_t)r }, x, norm, wqkv, s, r, b, r, 1, st );
}

} // namespace gh
