// fp32 products of a stage, alone and with the op that follows them.  Only small models run in fp32, at a handful of activation rows: a
// product then is a single read of a small matrix and the launch is bound by its one round trip to memory and by being a launch at
// all.  So a wave owns ROWS weight rows and requests the whole of a short row, with its pieces of the activations, before the first
// use, and what follows a product element by element (RoPE and the cache append, the residual add, the SiLU gate) is done where its
// sums are, with no second kernel.  15M model at 4 rows: q, k, v 7.4 + 4.4 us as product and follow-up kernel, 4.5 as one; w1, w3 7.3 + 4.7,
// 3.9; wo and w2 10.7, 3.7 with the add; classifier (32000 x 288) 23.0, 11.4.
#include "gh_common.h"

#include <algorithm>

namespace gh {
namespace {

// what a wave does with the sums of its ROWS weight rows for activation row `col`; unit: index of the wave
struct F32Plain
{
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

// V: elements per load (4: s % 4 == 0, 16-byte aligned operands).  COLS activation rows at a time, `cols_per_y` of them per grid row.
template<int ROWS, int COLS, int V, typename Epilogue>
__global__ __launch_bounds__( 256 ) void gemm_f32_kernel( Epilogue epi, const float* __restrict__ x, const float* __restrict__ w, uint32_t s, uint32_t r, uint32_t b,
                                                          uint32_t units, uint32_t cols_per_y )
{
  constexpr int KU = ROWS <= 2 ? 4 : 2; // pieces of a row under way at once
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
      vec a[KU][ROWS], y[KU][COLS];
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
      }
#pragma unroll
      for ( int u = 0; u < KU; u++ ) {
        const bool in = !tail.value || k0 + ( u * 64 + lane ) * V < s;
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
    };
    uint32_t k0 = 0;
    for ( ; k0 + KU * 64 * V <= s; k0 += KU * 64 * V ) {
      step( k0, std::false_type {} );
    }
    if ( k0 < s ) {
      step( k0, std::true_type {} );
    }
    float mine[ROWS]; // of the activation row that is this lane's: lane c stores row c0 + c
#pragma unroll
    for ( int i = 0; i < ROWS; i++ ) {
      mine[i] = 0.0f;
#pragma unroll
      for ( int c = 0; c < COLS; c++ ) {
        const float sum = wave_sum( acc[i][c] );
        mine[i] = lane == (uint32_t)c ? sum : mine[i];
      }
    }
    if ( lane < COLS && c0 + lane < c_end ) {
      epi.template store<ROWS>( unit, c0 + lane, mine );
    }
  }
}

// Rows per wave: two where that leaves at most two work-groups a CU, i.e. where latency is all there is; else four, which read the
// activations half as often.  8 activation rows at a time where there are more than 4; a single one alone (864 x 288 at 1 row: 3.4 us, 5.0 as four).
template<int ROWS, int COLS, typename Epilogue>
int launch_cols( const Epilogue& epi, const float* x, const float* w, uint64_t s, uint64_t r, uint64_t b, uint64_t units, hipStream_t st )
{
  const uint64_t cols = std::max<uint64_t>( 64, ( ( b + 65534 ) / 65535 + 63 ) / 64 * 64 );
  const dim3 grid( (unsigned)( ( units + 3 ) / 4 ), (unsigned)( ( b + cols - 1 ) / cols ) );
  if ( s % 4 == 0 && ( ( reinterpret_cast<uintptr_t>( x ) | reinterpret_cast<uintptr_t>( w ) ) & 15u ) == 0 ) {
    gemm_f32_kernel<ROWS, COLS, 4><<<grid, 256, 0, st>>>( epi, x, w, (uint32_t)s, (uint32_t)r, (uint32_t)b, (uint32_t)units, (uint32_t)cols );
  } else {
    gemm_f32_kernel<ROWS, COLS, 1><<<grid, 256, 0, st>>>( epi, x, w, (uint32_t)s, (uint32_t)r, (uint32_t)b, (uint32_t)units, (uint32_t)cols );
  }
  GH_LAUNCH_CHECK();
  return GH_OK;
}
// `outputs`: what the waves share out, `per`: weight rows to one of them
template<typename Epilogue>
int launch_f32( const Epilogue& epi, const float* x, const float* w, uint64_t s, uint64_t r, uint64_t b, uint64_t outputs, uint64_t per, hipStream_t st )
{
  if ( outputs * per <= 4096 ) {
    const uint64_t units = ( outputs * per + 1 ) / 2;
    return b == 1   ? launch_cols<2, 1>( epi, x, w, s, r, b, units, st )
           : b <= 4 ? launch_cols<2, 4>( epi, x, w, s, r, b, units, st )
                    : launch_cols<2, 8>( epi, x, w, s, r, b, units, st );
  }
  const uint64_t units = ( outputs * per + 3 ) / 4;
  return b == 1   ? launch_cols<4, 1>( epi, x, w, s, r, b, units, st )
         : b <= 4 ? launch_cols<4, 4>( epi, x, w, s, r, b, units, st )
                  : launch_cols<4, 8>( epi, x, w, s, r, b, units, st );
}

} // namespace

int gemm_f32( float* out, const float* x, const float* w, uint64_t s, uint64_t r, uint64_t b, hipStream_t st )
{
  return launch_f32( F32Plain { out, (uint32_t)r }, x, w, s, r, b, r, 1, st );
}
int gemm_f32_accum( float* residual, const float* x, const float* w, uint64_t s, uint64_t r, uint64_t b, hipStream_t st )
{
  return launch_f32( F32Accum { residual, (uint32_t)r }, x, w, s, r, b, r, 1, st );
}
int gemm_f32_gate( float* hb, const float* x, const float* w13, uint64_t s, uint64_t hidden, uint64_t b, hipStream_t st )
{
  return launch_f32( F32Gate { hb, (uint32_t)hidden }, x, w13, s, 2 * hidden, b, hidden, 2, st );
}
int gemm_f32_qkv( float* q, float* kv_out, const float* x, const float* wqkv, uint64_t s, uint64_t b, const uint32_t* pos, const float* freq_real, const float* freq_imag,
                  void* const* token_rows, uint32_t dim, uint32_t kv_dim, uint32_t head_size, hipStream_t st )
{
  const uint64_t r = (uint64_t)dim + 2ull * kv_dim;
  return launch_f32( F32Qkv { q, kv_out, pos, freq_real, freq_imag, token_rows, dim, kv_dim, head_size, (uint32_t)r }, x, wqkv, s, r, b, r, 1, st );
}

} // namespace gh
