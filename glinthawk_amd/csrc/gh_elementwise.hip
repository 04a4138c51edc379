// Small bandwidth-bound ops of the stage: accum, rmsnorm, silu, argmax, soft_sample, dtype
// conversion and buffer fills.  All math in fp32 on fp16/fp32 storage, one rounding per store,
// following the reference's CPU path (arch/amd64/common/ops.hh).
#include "gh_common.h"

#include <type_traits>
#include <vector>

namespace gh {
namespace {

constexpr int EW_THREADS = 256;

// 16-byte vector of T
template<typename T>
struct Vec16
{
  static constexpr int N = 16 / sizeof( T );
  union
  {
    uint4 raw;
    T v[N];
  };
};

inline unsigned blocks_for( uint64_t items, int per_block, unsigned cap = 65535u * 16u )
{
  uint64_t b = ( items + per_block - 1 ) / per_block;
  if ( b < 1 ) {
    b = 1;
  }
  return (unsigned)( b > cap ? cap : b );
}

// ---- accum ---------------------------------------------------------------------------------
template<typename T>
__global__ __launch_bounds__( EW_THREADS ) void accum_kernel( T* __restrict__ a, const T* __restrict__ b, uint64_t n )
{
  constexpr int N = Vec16<T>::N;
  const uint64_t n_vec = n / N;
  const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
  for ( uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n_vec; i += stride ) {
    Vec16<T> va, vb;
    va.raw = reinterpret_cast<const uint4*>( a )[i];
    vb.raw = reinterpret_cast<const uint4*>( b )[i];
#pragma unroll
    for ( int k = 0; k < N; k++ ) {
      va.v[k] = from_f32<T>( to_f32( va.v[k] ) + to_f32( vb.v[k] ) );
    }
    reinterpret_cast<uint4*>( a )[i] = va.raw;
  }
  for ( uint64_t i = n_vec * N + (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride ) {
    a[i] = from_f32<T>( to_f32( a[i] ) + to_f32( b[i] ) );
  }
}

// ---- silu ----------------------------------------------------------------------------------
__device__ __forceinline__ float silu_mul( float x, float y ) { return x / ( 1.0f + __expf( -x ) ) * y; }

template<typename T>
__global__ __launch_bounds__( EW_THREADS ) void silu_kernel( T* __restrict__ hb, const T* __restrict__ hb2, uint64_t n )
{
  constexpr int N = Vec16<T>::N;
  const uint64_t n_vec = n / N;
  const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
  for ( uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n_vec; i += stride ) {
    Vec16<T> va, vb;
    va.raw = reinterpret_cast<const uint4*>( hb )[i];
    vb.raw = reinterpret_cast<const uint4*>( hb2 )[i];
#pragma unroll
    for ( int k = 0; k < N; k++ ) {
      va.v[k] = from_f32<T>( silu_mul( to_f32( va.v[k] ), to_f32( vb.v[k] ) ) );
    }
    reinterpret_cast<uint4*>( hb )[i] = va.raw;
  }
  for ( uint64_t i = n_vec * N + (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride ) {
    hb[i] = from_f32<T>( silu_mul( to_f32( hb[i] ), to_f32( hb2[i] ) ) );
  }
}

// ---- block reductions -------------------------------------------------------------------------
__device__ __forceinline__ float block_sum( float v, float* smem )
{
  v = wave_sum( v );
  const int wave = threadIdx.x / WAVE;
  const int n_waves = blockDim.x / WAVE;
  if ( threadIdx.x % WAVE == 0 ) {
    smem[wave] = v;
  }
  __syncthreads();
  float total = 0.0f;
  for ( int w = 0; w < n_waves; w++ ) {
    total += smem[w];
  }
  __syncthreads();
  return total;
}

// ---- rmsnorm: one block per row ----------------------------------------------------------------
template<typename T>
__global__ __launch_bounds__( EW_THREADS ) void rmsnorm_kernel( T* __restrict__ out,
                                                               const T* __restrict__ x,
                                                               const T* __restrict__ weight,
                                                               uint32_t size )
{
  __shared__ float smem[EW_THREADS / WAVE];
  constexpr int N = Vec16<T>::N;
  const T* X = x + (uint64_t)blockIdx.x * size;
  T* O = out + (uint64_t)blockIdx.x * size;
  const uint32_t n_vec = ( size % N == 0 ) ? size / N : 0; // vector path only for aligned rows

  float ss = 0.0f;
  for ( uint32_t i = threadIdx.x; i < n_vec; i += blockDim.x ) {
    Vec16<T> v;
    v.raw = reinterpret_cast<const uint4*>( X )[i];
#pragma unroll
    for ( int k = 0; k < N; k++ ) {
      const float f = to_f32( v.v[k] );
      ss += f * f;
    }
  }
  for ( uint32_t i = n_vec * N + threadIdx.x; i < size; i += blockDim.x ) {
    const float f = to_f32( X[i] );
    ss += f * f;
  }
  ss = block_sum( ss, smem );
  ss = ss / (float)size + 1e-5f;
  const float inv = 1.0f / sqrtf( ss );

  for ( uint32_t i = threadIdx.x; i < n_vec; i += blockDim.x ) {
    Vec16<T> v, w;
    v.raw = reinterpret_cast<const uint4*>( X )[i];
    w.raw = reinterpret_cast<const uint4*>( weight )[i];
#pragma unroll
    for ( int k = 0; k < N; k++ ) {
      v.v[k] = from_f32<T>( to_f32( w.v[k] ) * ( inv * to_f32( v.v[k] ) ) );
    }
    reinterpret_cast<uint4*>( O )[i] = v.raw;
  }
  for ( uint32_t i = n_vec * N + threadIdx.x; i < size; i += blockDim.x ) {
    O[i] = from_f32<T>( to_f32( weight[i] ) * ( inv * to_f32( X[i] ) ) );
  }
}

// ---- rows that arrive in page-locked host memory -------------------------------------------------
// The first kernel of a step reads them where the host left them: they go to the device and, normed, to the first product, and the step's tables come along
// in work-groups of their own.  As copies in front of rmsnorm_kernel each is a launch and a hand-over between engines more.  Bound by the bus.
// The copy engine is the faster way over it for 2 MB and more: beyond GH_ROWS_IN_BYTES the rows are copied (f16 with norm, tables and a wait, copied and in place:
// 32 rows of 4096 28.1 and 19.6 us, 64 of 8192 43.4 and 36.8, 128 61.7 and 61.9, 256 99 and 109).
// The sums as rmsnorm_kernel takes them, from registers: a second pass would cross the bus again.  16-byte pieces; PIECES: a thread's.
template<typename T, int PIECES>
__global__ __launch_bounds__( EW_THREADS ) void rows_in_kernel( T* __restrict__ x,
                                                               T* __restrict__ normed,
                                                               const T* __restrict__ host,
                                                               const T* __restrict__ weight,
                                                               uint32_t size,
                                                               uint32_t rows,
                                                               uint4* __restrict__ table,
                                                               const uint4* __restrict__ host_table,
                                                               uint32_t table_pieces )
{
  __shared__ float smem[EW_THREADS / WAVE];
  if ( blockIdx.x >= rows ) {
    const uint32_t i = ( blockIdx.x - rows ) * EW_THREADS + threadIdx.x;
    if ( i < table_pieces ) {
      table[i] = host_table[i];
    }
    return;
  }
  constexpr int N = Vec16<T>::N;
  const uint32_t n_vec = size / N;
  const uint64_t first = (uint64_t)blockIdx.x * n_vec;
  Vec16<T> v[PIECES], w[PIECES];
#pragma unroll
  for ( int p = 0; p < PIECES; p++ ) { // a piece past the row's end is the first again and counts nothing
    const uint32_t i = p * EW_THREADS + threadIdx.x, at = i < n_vec ? i : 0;
    v[p].raw = reinterpret_cast<const uint4*>( host )[first + at];
    w[p].raw = reinterpret_cast<const uint4*>( weight )[at];
  }
  float ss = 0.0f;
#pragma unroll
  for ( int p = 0; p < PIECES; p++ ) {
    const bool in = p * EW_THREADS + threadIdx.x < n_vec;
#pragma unroll
    for ( int k = 0; k < N; k++ ) {
      const float f = to_f32( v[p].v[k] );
      ss += in ? f * f : 0.0f;
    }
  }
  ss = block_sum( ss, smem );
  ss = ss / (float)size + 1e-5f;
  const float inv = 1.0f / sqrtf( ss );
#pragma unroll
  for ( int p = 0; p < PIECES; p++ ) {
    const uint32_t i = p * EW_THREADS + threadIdx.x;
    if ( i < n_vec ) {
      reinterpret_cast<uint4*>( x )[first + i] = v[p].raw;
#pragma unroll
      for ( int k = 0; k < N; k++ ) {
        v[p].v[k] = from_f32<T>( to_f32( w[p].v[k] ) * ( inv * to_f32( v[p].v[k] ) ) );
      }
      reinterpret_cast<uint4*>( normed )[first + i] = v[p].raw;
    }
  }
}

// Rows to page-locked memory, bound by the bus; no size at which the copy engine is faster was found (f16 with the wait, copied and so: 1 row of 8192 16.2 and
// 15.9 us, 32 of 4096 28.4 and 20.8, 64 of 8192 42.2 and 34.8, 256 99 and 92).
__global__ __launch_bounds__( EW_THREADS ) void copy_pieces_kernel( uint4* __restrict__ dst, const uint4* __restrict__ src, uint64_t n )
{
  const uint64_t stride = (uint64_t)gridDim.x * EW_THREADS;
  for ( uint64_t i = (uint64_t)blockIdx.x * EW_THREADS + threadIdx.x; i < n; i += stride ) {
    dst[i] = src[i];
  }
}

// ---- rows of a table by index: one block per row, bytes as they are -------------------------------
// (with a step's table in work-groups of its own, as above)
template<typename P>
__global__ __launch_bounds__( EW_THREADS ) void embed_rows_kernel( P* __restrict__ x, const uint32_t* __restrict__ tokens, const P* __restrict__ table, uint32_t width,
                                                                  uint32_t vocab, uint32_t rows, uint4* __restrict__ step, const uint4* __restrict__ host_step,
                                                                  uint32_t step_pieces )
{
  if ( blockIdx.x >= rows ) {
    const uint32_t i = ( blockIdx.x - rows ) * EW_THREADS + threadIdx.x;
    if ( i < step_pieces ) {
      step[i] = host_step[i];
    }
    return;
  }
  const uint64_t token = tokens[blockIdx.x];
  if ( token >= vocab ) {
    return; // a row without a token stays as it is
  }
  for ( uint32_t c = threadIdx.x; c < width; c += blockDim.x ) {
    x[(uint64_t)blockIdx.x * width + c] = table[token * width + c];
  }
}

// ---- argmax: one block per row, first index of the maximum --------------------------------------
// Bound by latency: a row of 32000 values is one work-group's, so a thread asks for AHEAD pieces of it before it compares the first.  4 fp32
// rows of 32000: 36.8 us with 256 threads that went value by value, 6.1 so.  256 threads where they ask for all of a row at once, with the fewest
// pieces that do (1024 f16 rows of 1000: 4.1 us, 7.5 with eight each; of 4096: 5.0, 9.3, with 1024 threads 17.6), else 1024.  As a loop over the row
// would have it: the lowest index of equal values, NaN never beats anything but stays where the row begins with it.
// V: values per load, n % V == 0 and rows aligned to V values
template<typename T, int V, int ARG_THREADS, int AHEAD>
__global__ __launch_bounds__( ARG_THREADS ) void argmax_kernel( uint32_t* __restrict__ out, const T* __restrict__ v, uint32_t n )
{
  __shared__ float s_val[ARG_THREADS / WAVE];
  __shared__ uint32_t s_idx[ARG_THREADS / WAVE];
  const T* row = v + (uint64_t)blockIdx.x * n;
  struct alignas( sizeof( T ) * V ) Piece
  {
    T e[V];
  };
  const float first = to_f32( row[0] );
  const Piece* pieces = reinterpret_cast<const Piece*>( row );
  const uint32_t n_pieces = n / V;
  float best = -INFINITY;
  uint32_t best_i = 0xffffffffu;
  for ( uint64_t p0 = threadIdx.x; p0 < n_pieces; p0 += ARG_THREADS * AHEAD ) {
    Piece x[AHEAD];
#pragma unroll
    for ( int u = 0; u < AHEAD; u++ ) {
      x[u] = pieces[min( p0 + u * ARG_THREADS, (uint64_t)n_pieces - 1 )]; // past the end: the last one again, which changes nothing
    }
#pragma unroll
    for ( int u = 0; u < AHEAD; u++ ) {
      const uint32_t i0 = (uint32_t)min( p0 + u * ARG_THREADS, (uint64_t)n_pieces - 1 ) * V;
#pragma unroll
      for ( int e = 0; e < V; e++ ) {
        arg_better( best, best_i, to_f32( x[u].e[e] ), i0 + e );
      }
    }
  }
  if ( block_arg<ARG_THREADS>( best, best_i, s_val, s_idx ) ) {
    out[blockIdx.x] = first != first || best_i == 0xffffffffu ? 0u : best_i;
  }
}

// ---- counter-based random numbers (Philox-4x32-10) ----------------------------------------------
__device__ __forceinline__ uint4 philox( uint64_t counter, uint64_t stream_id, uint64_t seed )
{
  uint32_t c0 = (uint32_t)counter, c1 = (uint32_t)( counter >> 32 ), c2 = (uint32_t)stream_id, c3 = (uint32_t)( stream_id >> 32 );
  uint32_t k0 = (uint32_t)seed, k1 = (uint32_t)( seed >> 32 );
#pragma unroll
  for ( int r = 0; r < 10; r++ ) {
    const uint64_t p0 = (uint64_t)0xD2511F53u * c0;
    const uint64_t p1 = (uint64_t)0xCD9E8D57u * c2;
    const uint32_t n0 = (uint32_t)( p1 >> 32 ) ^ c1 ^ k0;
    const uint32_t n1 = (uint32_t)p1;
    const uint32_t n2 = (uint32_t)( p0 >> 32 ) ^ c3 ^ k1;
    const uint32_t n3 = (uint32_t)p0;
    c0 = n0;
    c1 = n1;
    c2 = n2;
    c3 = n3;
    k0 += 0x9E3779B9u;
    k1 += 0xBB67AE85u;
  }
  return make_uint4( c0, c1, c2, c3 );
}

__device__ __forceinline__ float u01( uint32_t bits ) { return ( (float)( bits >> 8 ) + 0.5f ) * ( 1.0f / 16777216.0f ); } // (0,1)

template<typename T>
__global__ __launch_bounds__( EW_THREADS ) void fill_uniform_kernel( T* __restrict__ dst, uint64_t n, float lo, float hi, uint64_t seed )
{
  const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
  const uint64_t n4 = ( n + 3 ) / 4;
  for ( uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n4; i += stride ) {
    const uint4 r = philox( i, 0, seed );
    const uint32_t w[4] = { r.x, r.y, r.z, r.w };
#pragma unroll
    for ( int k = 0; k < 4; k++ ) {
      const uint64_t idx = i * 4 + k;
      if ( idx < n ) {
        dst[idx] = from_f32<T>( lo + ( hi - lo ) * u01( w[k] ) );
      }
    }
  }
}

template<typename T>
__global__ __launch_bounds__( EW_THREADS ) void fill_normal_kernel( T* __restrict__ dst, uint64_t n, float mean, float stdv, uint64_t seed )
{
  const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
  const uint64_t n4 = ( n + 3 ) / 4;
  for ( uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n4; i += stride ) {
    const uint4 r = philox( i, 1, seed );
    // Box-Muller, two pairs
    const float r0 = sqrtf( -2.0f * __logf( u01( r.x ) ) );
    const float r1 = sqrtf( -2.0f * __logf( u01( r.z ) ) );
    float s0, c0, s1, c1;
    __sincosf( 6.2831853071795865f * u01( r.y ), &s0, &c0 );
    __sincosf( 6.2831853071795865f * u01( r.w ), &s1, &c1 );
    const float z[4] = { r0 * c0, r0 * s0, r1 * c1, r1 * s1 };
#pragma unroll
    for ( int k = 0; k < 4; k++ ) {
      const uint64_t idx = i * 4 + k;
      if ( idx < n ) {
        dst[idx] = from_f32<T>( mean + stdv * z[k] );
      }
    }
  }
}

// ---- soft_sample: Gumbel-max noise on rows with temperature > 0 ---------------------------------
template<typename T>
__global__ __launch_bounds__( EW_THREADS ) void gumbel_kernel( T* __restrict__ v, const float* __restrict__ temps, uint32_t vocab, uint64_t seed )
{
  const float temp = temps[blockIdx.y];
  if ( !( temp > 0.0f ) ) {
    return;
  }
  T* row = v + (uint64_t)blockIdx.y * vocab;
  const uint32_t n4 = ( vocab + 3 ) / 4;
  for ( uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < n4; i += gridDim.x * blockDim.x ) {
    const uint4 r = philox( i, 2 + blockIdx.y, seed );
    const uint32_t w[4] = { r.x, r.y, r.z, r.w };
#pragma unroll
    for ( int k = 0; k < 4; k++ ) {
      const uint32_t idx = i * 4 + k;
      if ( idx < vocab ) {
        const float noise = logf( -logf( u01( w[k] ) ) );
        row[idx] = from_f32<T>( to_f32( row[idx] ) / temp - noise );
      }
    }
  }
}

// ---- conversion / zero fill --------------------------------------------------------------------
template<typename D, typename S>
__global__ __launch_bounds__( EW_THREADS ) void convert_kernel( D* __restrict__ dst, const S* __restrict__ src, uint64_t n )
{
  const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
  for ( uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride ) {
    dst[i] = from_f32<D>( to_f32( src[i] ) );
  }
}

__global__ __launch_bounds__( EW_THREADS ) void zero_kernel( uint32_t* __restrict__ dst, uint64_t n_words, uint8_t* tail, uint32_t n_tail )
{
  const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
  for ( uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n_words; i += stride ) {
    dst[i] = 0u;
  }
  if ( blockIdx.x == 0 && threadIdx.x < n_tail ) {
    tail[threadIdx.x] = 0;
  }
}

inline bool aligned16( const void* p ) { return ( reinterpret_cast<uintptr_t>( p ) & 15u ) == 0; }

// Whether kernels can read and write all of this host memory where it is: `bytes` that lie within one page-locked allocation.  Memory that somebody
// registered in part ends in the middle of what is asked about.  (Two queries, 0.1 to 0.2 us together; one of 0.15 us for memory that is not page-locked.)
bool page_locked( const void* p, uint64_t bytes )
{
  hipPointerAttribute_t a {};
  hipDeviceptr_t base = nullptr;
  size_t size = 0;
  if ( hipPointerGetAttributes( &a, p ) != hipSuccess ) {
    (void)hipGetLastError(); // memory the runtime has not heard of: not an error of the next launch
    return false;
  }
  if ( a.type != hipMemoryTypeHost || a.devicePointer != p ) {
    return false;
  }
  if ( hipMemGetAddressRange( &base, &size, a.devicePointer ) != hipSuccess ) {
    (void)hipGetLastError();
    return false;
  }
  const uint64_t before = static_cast<const char*>( p ) - static_cast<const char*>( base );
  return before <= size && bytes <= size - before;
}
// ... and in pieces of 16 bytes, from or to `dev`
bool pieces_in_place( const void* host, const void* dev, uint64_t bytes )
{
  return bytes % 16 == 0 && aligned16( host ) && aligned16( dev ) && page_locked( host, bytes );
}
// the rows of gh_rows_in: at most four pieces a thread
bool rows_in_place( const void* x, const void* normed, const void* host, const void* weight, uint64_t size, uint64_t batch, gh_dtype dt )
{
  const uint64_t bytes = size * dtype_size( dt );
  return bytes % 16 == 0 && bytes <= 4 * 16 * EW_THREADS && batch * bytes <= GH_ROWS_IN_BYTES && aligned16( normed ) && aligned16( weight )
         && pieces_in_place( host, x, batch * bytes );
}

} // namespace
} // namespace gh

using namespace gh;

#define GH_DISPATCH_DT( dt, ... )                                                                                      \
  do {                                                                                                                 \
    if ( ( dt ) == GH_F16 ) {                                                                                          \
      using T = __half;                                                                                                \
      __VA_ARGS__;                                                                                                     \
    } else if ( ( dt ) == GH_F32 ) {                                                                                   \
      using T = float;                                                                                                 \
      __VA_ARGS__;                                                                                                     \
    } else {                                                                                                           \
      return fail( GH_ERR_INVALID, "unsupported dtype %d (f16 and f32 only)", (int)( dt ) );                           \
    }                                                                                                                  \
  } while ( 0 )

// fills also serve the bf16 buffers of the run-time sized designs
#define GH_DISPATCH_FILL( dt, ... )                                                                                    \
  do {                                                                                                                 \
    if ( ( dt ) == GH_BF16 ) {                                                                                         \
      using T = __bf16;                                                                                                \
      __VA_ARGS__;                                                                                                     \
    } else {                                                                                                           \
      GH_DISPATCH_DT( dt, __VA_ARGS__ );                                                                               \
    }                                                                                                                  \
  } while ( 0 )

extern "C" {

int gh_accum( void* a, const void* b, uint64_t size, uint64_t batch, gh_dtype dt, gh_stream stream )
{
  if ( int rc = ensure_init() ) {
    return rc;
  }
  const uint64_t n = size * batch;
  if ( n == 0 ) {
    return GH_OK;
  }
  GH_REQUIRE( a && b, "gh_accum: NULL pointer" );
  GH_REQUIRE( aligned16( a ) && aligned16( b ), "gh_accum: buffers must be 16-byte aligned" );
  GH_DISPATCH_DT( dt, accum_kernel<T><<<blocks_for( n / Vec16<T>::N + 1, EW_THREADS, 8192 ), EW_THREADS, 0, as_stream( stream )>>>(
                        static_cast<T*>( a ), static_cast<const T*>( b ), n ) );
  GH_LAUNCH_CHECK();
  return GH_OK;
}

int gh_silu( void* hb, const void* hb2, uint64_t hidden_dim, uint64_t batch, gh_dtype dt, gh_stream stream )
{
  if ( int rc = ensure_init() ) {
    return rc;
  }
  const uint64_t n = hidden_dim * batch;
  if ( n == 0 ) {
    return GH_OK;
  }
  GH_REQUIRE( hb && hb2, "gh_silu: NULL pointer" );
  GH_REQUIRE( aligned16( hb ) && aligned16( hb2 ), "gh_silu: buffers must be 16-byte aligned" );
  GH_DISPATCH_DT( dt, silu_kernel<T><<<blocks_for( n / Vec16<T>::N + 1, EW_THREADS, 8192 ), EW_THREADS, 0, as_stream( stream )>>>(
                        static_cast<T*>( hb ), static_cast<const T*>( hb2 ), n ) );
  GH_LAUNCH_CHECK();
  return GH_OK;
}

int gh_rmsnorm( void* out, const void* x, const void* weight, uint64_t size, uint64_t batch, gh_dtype dt, gh_stream stream )
{
  if ( int rc = ensure_init() ) {
    return rc;
  }
  if ( batch == 0 || size == 0 ) {
    return GH_OK;
  }
  GH_REQUIRE( out && x && weight, "gh_rmsnorm: NULL pointer" );
  GH_REQUIRE( size <= 0xffffffffull && batch <= 0x7fffffffull, "gh_rmsnorm: shape too large" );
  GH_REQUIRE( aligned16( out ) && aligned16( x ) && aligned16( weight ), "gh_rmsnorm: buffers must be 16-byte aligned" );
  GH_DISPATCH_DT( dt, rmsnorm_kernel<T><<<(unsigned)batch, EW_THREADS, 0, as_stream( stream )>>>(
                        static_cast<T*>( out ), static_cast<const T*>( x ), static_cast<const T*>( weight ), (uint32_t)size ) );
  GH_LAUNCH_CHECK();
  return GH_OK;
}

int gh_rows_in( void* x, void* normed, const void* host, const void* weight, uint64_t size, uint64_t batch, void* table_dev, const void* table_host, uint64_t table_bytes,
                gh_dtype dt, gh_stream stream )
{
  if ( int rc = ensure_init() ) {
    return rc;
  }
  if ( size == 0 ) {
    batch = 0;
  }
  if ( batch == 0 ) {
    dt = GH_F16; // a table alone: bytes as they are
  }
  GH_REQUIRE( batch == 0 || ( x && normed && host && weight ), "gh_rows_in: NULL pointer" );
  GH_REQUIRE( table_bytes == 0 || ( table_dev && table_host ), "gh_rows_in: NULL table" );
  GH_REQUIRE( size <= 0xffffffffull && batch <= 0x7fffffffull && table_bytes <= ( 1ull << 34 ), "gh_rows_in: shape too large" );
  const uint64_t bytes = size * dtype_size( dt ), pieces = ( bytes / 16 + EW_THREADS - 1 ) / EW_THREADS;
  if ( table_bytes > 0 && !pieces_in_place( table_host, table_dev, table_bytes ) ) {
    GH_HIP( hipMemcpyAsync( table_dev, table_host, table_bytes, hipMemcpyHostToDevice, as_stream( stream ) ) );
    table_bytes = 0;
  }
  const uint64_t table_groups = ( table_bytes / 16 + EW_THREADS - 1 ) / EW_THREADS;
  const bool in_place = batch > 0 && rows_in_place( x, normed, host, weight, size, batch, dt );
  const uint64_t rows = in_place ? batch : 0;
  if ( rows + table_groups > 0 ) {
    auto launch = [&]( auto* e, auto count ) {
      using T = std::remove_pointer_t<decltype( e )>;
      rows_in_kernel<T, decltype( count )::value><<<(unsigned)( rows + table_groups ), EW_THREADS, 0, as_stream( stream )>>>(
        static_cast<T*>( x ), static_cast<T*>( normed ), static_cast<const T*>( host ), static_cast<const T*>( weight ), (uint32_t)size, (uint32_t)rows,
        static_cast<uint4*>( table_dev ), static_cast<const uint4*>( table_host ), (uint32_t)( table_bytes / 16 ) );
    };
    GH_DISPATCH_DT( dt, pieces <= 2 ? launch( static_cast<T*>( nullptr ), std::integral_constant<int, 2> {} )
                                    : launch( static_cast<T*>( nullptr ), std::integral_constant<int, 4> {} ) );
    GH_LAUNCH_CHECK();
  }
  if ( batch == 0 || in_place ) {
    return GH_OK;
  }
  GH_HIP( hipMemcpyAsync( x, host, batch * bytes, hipMemcpyHostToDevice, as_stream( stream ) ) );
  return gh_rmsnorm( normed, x, weight, size, batch, dt, stream );
}

int gh_rows_in_place( const void* x, const void* normed, const void* host, const void* weight, uint64_t size, uint64_t batch, gh_dtype dt )
{
  if ( ensure_init() != GH_OK || host == nullptr || size == 0 || size > 0xffffffffull || batch == 0 || batch > 0x7fffffffull || ( dt != GH_F16 && dt != GH_F32 ) ) {
    return 0;
  }
  return rows_in_place( x, normed, host, weight, size, batch, dt ) ? 1 : 0;
}

int gh_host_in_place( const void* host, const void* dev, uint64_t bytes )
{
  return ensure_init() == GH_OK && host != nullptr && pieces_in_place( host, dev, bytes ) ? 1 : 0;
}

int gh_rows_out( void* host, const void* x, uint64_t bytes, gh_stream stream )
{
  if ( int rc = ensure_init() ) {
    return rc;
  }
  if ( bytes == 0 ) {
    return GH_OK;
  }
  GH_REQUIRE( host && x, "gh_rows_out: NULL pointer" );
  if ( pieces_in_place( host, x, bytes ) ) {
    const uint64_t n = bytes / 16;
    copy_pieces_kernel<<<(unsigned)std::min<uint64_t>( ( n + EW_THREADS - 1 ) / EW_THREADS, 1024 ), EW_THREADS, 0, as_stream( stream )>>>(
      static_cast<uint4*>( host ), static_cast<const uint4*>( x ), n );
    GH_LAUNCH_CHECK();
  } else {
    GH_HIP( hipMemcpyAsync( host, x, bytes, hipMemcpyDeviceToHost, as_stream( stream ) ) );
  }
  GH_HIP( hipStreamSynchronize( as_stream( stream ) ) );
  return GH_OK;
}

int gh_embed_rows( void* x, const uint32_t* tokens, const void* table, uint64_t width, uint64_t vocab, uint64_t batch, void* table_dev, const void* table_host,
                   uint64_t table_bytes, gh_dtype dt, gh_stream stream )
{
  if ( int rc = ensure_init() ) {
    return rc;
  }
  if ( width == 0 ) {
    batch = 0;
  }
  GH_REQUIRE( batch == 0 || ( x && tokens && table ), "gh_embed_rows: NULL pointer" );
  GH_REQUIRE( table_bytes == 0 || ( table_dev && table_host ), "gh_embed_rows: NULL table" );
  GH_REQUIRE( width <= 0x7fffffffull && vocab <= 0xffffffffull && batch <= 0x3fffffffull && table_bytes <= ( 1ull << 34 ), "gh_embed_rows: shape too large" );
  if ( table_bytes > 0 && !pieces_in_place( table_host, table_dev, table_bytes ) ) {
    GH_HIP( hipMemcpyAsync( table_dev, table_host, table_bytes, hipMemcpyHostToDevice, as_stream( stream ) ) );
    table_bytes = 0;
  }
  const uint64_t bytes = width * dtype_size( dt ), groups = batch + ( table_bytes / 16 + EW_THREADS - 1 ) / EW_THREADS;
  if ( groups == 0 ) {
    return GH_OK;
  }
  auto launch = [&]( auto piece ) {
    using P = decltype( piece );
    embed_rows_kernel<P><<<(unsigned)groups, EW_THREADS, 0, as_stream( stream )>>>( static_cast<P*>( x ), tokens, static_cast<const P*>( table ),
                                                                                    (uint32_t)( bytes / sizeof( P ) ), (uint32_t)vocab, (uint32_t)batch,
                                                                                    static_cast<uint4*>( table_dev ), static_cast<const uint4*>( table_host ),
                                                                                    (uint32_t)( table_bytes / 16 ) );
  };
  bytes % 16 == 0 && aligned16( x ) && aligned16( table ) ? launch( uint4 {} ) : launch( uint16_t {} );
  GH_LAUNCH_CHECK();
  return GH_OK;
}

int gh_argmax( uint32_t* out_host, uint32_t* out_dev, const void* v, uint64_t n, uint64_t batch, gh_dtype dt, gh_stream stream )
{
  if ( int rc = ensure_init() ) {
    return rc;
  }
  if ( batch == 0 ) {
    return GH_OK;
  }
  GH_REQUIRE( out_dev && v, "gh_argmax: NULL pointer" );
  GH_REQUIRE( n > 0 && n <= 0xfffffffeull && batch <= 0x7fffffffull, "gh_argmax: bad shape" );
  const bool whole = n * dtype_size( dt ) % 16 == 0 && ( reinterpret_cast<uintptr_t>( v ) & 15u ) == 0;
  auto launch = [&]( auto* e, auto per_load ) {
    using T = std::remove_pointer_t<decltype( e )>;
    constexpr int V = decltype( per_load )::value;
    const T* rows = static_cast<const T*>( v );
    auto go = [&]( auto threads, auto ahead ) {
      constexpr int N = decltype( threads )::value, A = decltype( ahead )::value;
      argmax_kernel<T, V, N, A><<<(unsigned)batch, N, 0, as_stream( stream )>>>( out_dev, rows, (uint32_t)n );
    };
    const uint64_t pieces = n / V;
    const std::integral_constant<int, 256> few {};
    const std::integral_constant<int, 1024> many {};
    if ( pieces <= 256 ) {
      go( few, std::integral_constant<int, 1> {} );
    } else if ( pieces <= 512 ) {
      go( few, std::integral_constant<int, 2> {} );
    } else if ( pieces <= 1024 ) {
      go( few, std::integral_constant<int, 4> {} );
    } else if ( pieces <= 2048 ) {
      go( few, std::integral_constant<int, 8> {} );
    } else if ( pieces <= 4096 ) {
      go( many, std::integral_constant<int, 4> {} );
    } else {
      go( many, std::integral_constant<int, 8> {} );
    }
  };
  GH_DISPATCH_DT( dt, whole ? launch( static_cast<T*>( nullptr ), std::integral_constant<int, 16 / sizeof( T )> {} )
                            : launch( static_cast<T*>( nullptr ), std::integral_constant<int, 1> {} ) );
  GH_LAUNCH_CHECK();
  if ( out_host ) {
    GH_HIP( hipMemcpyAsync( out_host, out_dev, batch * sizeof( uint32_t ), hipMemcpyDeviceToHost, as_stream( stream ) ) );
    GH_HIP( hipStreamSynchronize( as_stream( stream ) ) );
  }
  return GH_OK;
}

int gh_soft_sample( void* v, const float* temperatures, uint64_t vocab, uint64_t batch, uint64_t seed, gh_dtype dt, gh_stream stream )
{
  if ( int rc = ensure_init() ) {
    return rc;
  }
  if ( batch == 0 || vocab == 0 ) {
    return GH_OK;
  }
  GH_REQUIRE( v && temperatures, "gh_soft_sample: NULL pointer" );
  GH_REQUIRE( batch <= MAX_BATCH && vocab <= 0xffffffffull, "gh_soft_sample: batch > %llu", (unsigned long long)MAX_BATCH );
  bool any = false;
  for ( uint64_t i = 0; i < batch; i++ ) {
    any = any || temperatures[i] > 0.0f;
  }
  if ( !any ) {
    return GH_OK; // greedy rows are untouched, as in the reference
  }
  void* d_temps = nullptr;
  StageScope scope( as_stream( stream ) );
  if ( int rc = stage_table( temperatures, batch * sizeof( float ), as_stream( stream ), &d_temps ) ) {
    return rc;
  }
  const dim3 grid( blocks_for( vocab / 4 + 1, EW_THREADS, 64 ), (unsigned)batch );
  GH_DISPATCH_DT( dt, gumbel_kernel<T><<<grid, EW_THREADS, 0, as_stream( stream )>>>(
                        static_cast<T*>( v ), static_cast<const float*>( d_temps ), (uint32_t)vocab, seed ) );
  GH_LAUNCH_CHECK();
  return scope.finish();
}

int gh_fill_uniform( void* dst, uint64_t n, float lo, float hi, uint64_t seed, gh_dtype dt, gh_stream stream )
{
  if ( int rc = ensure_init() ) {
    return rc;
  }
  if ( n == 0 ) {
    return GH_OK;
  }
  GH_REQUIRE( dst, "gh_fill_uniform: NULL pointer" );
  GH_DISPATCH_FILL( dt, fill_uniform_kernel<T><<<blocks_for( n / 4 + 1, EW_THREADS, 16384 ), EW_THREADS, 0, as_stream( stream )>>>(
                        static_cast<T*>( dst ), n, lo, hi, seed ) );
  GH_LAUNCH_CHECK();
  return GH_OK;
}

int gh_fill_normal( void* dst, uint64_t n, float mean, float std, uint64_t seed, gh_dtype dt, gh_stream stream )
{
  if ( int rc = ensure_init() ) {
    return rc;
  }
  if ( n == 0 ) {
    return GH_OK;
  }
  GH_REQUIRE( dst, "gh_fill_normal: NULL pointer" );
  GH_DISPATCH_FILL( dt, fill_normal_kernel<T><<<blocks_for( n / 4 + 1, EW_THREADS, 16384 ), EW_THREADS, 0, as_stream( stream )>>>(
                        static_cast<T*>( dst ), n, mean, std, seed ) );
  GH_LAUNCH_CHECK();
  return GH_OK;
}

int gh_memset_zero( void* dst, uint64_t bytes, gh_stream stream )
{
  if ( int rc = ensure_init() ) {
    return rc;
  }
  if ( bytes == 0 ) {
    return GH_OK;
  }
  GH_REQUIRE( dst && ( reinterpret_cast<uintptr_t>( dst ) & 3u ) == 0, "gh_memset_zero: pointer must be 4-byte aligned" );
  const uint64_t words = bytes / 4;
  zero_kernel<<<blocks_for( words + 1, EW_THREADS, 8192 ), EW_THREADS, 0, as_stream( stream )>>>(
    static_cast<uint32_t*>( dst ), words, static_cast<uint8_t*>( dst ) + words * 4, (uint32_t)( bytes % 4 ) );
  GH_LAUNCH_CHECK();
  return GH_OK;
}

int gh_convert( void* dst, gh_dtype dst_dt, const void* src, gh_dtype src_dt, uint64_t n, gh_stream stream )
{
  if ( int rc = ensure_init() ) {
    return rc;
  }
  if ( n == 0 ) {
    return GH_OK;
  }
  GH_REQUIRE( dst && src, "gh_convert: NULL pointer" );
  const unsigned blocks = blocks_for( n, EW_THREADS, 8192 );
  hipStream_t s = as_stream( stream );
  if ( dst_dt == src_dt ) {
    GH_REQUIRE( dst_dt == GH_F16 || dst_dt == GH_F32, "gh_convert: unsupported dtype" );
    GH_HIP( hipMemcpyAsync( dst, src, n * dtype_size( dst_dt ), hipMemcpyDeviceToDevice, s ) );
    return GH_OK;
  }
  if ( dst_dt == GH_F16 && src_dt == GH_F32 ) {
    convert_kernel<__half, float><<<blocks, EW_THREADS, 0, s>>>( static_cast<__half*>( dst ), static_cast<const float*>( src ), n );
  } else if ( dst_dt == GH_F32 && src_dt == GH_F16 ) {
    convert_kernel<float, __half><<<blocks, EW_THREADS, 0, s>>>( static_cast<float*>( dst ), static_cast<const __half*>( src ), n );
  } else {
    return fail( GH_ERR_INVALID, "gh_convert: unsupported dtype pair %d <- %d", (int)dst_dt, (int)src_dt );
  }
  GH_LAUNCH_CHECK();
  return GH_OK;
}

// LlamaOperations::convert_and_copy: the conversion runs on the side that is the device; the host
// side only sees a byte copy of its own dtype.  Everything is queued on the caller's stream, which
// is waited for before the call returns (the reference's conversion is synchronous).
int gh_convert_and_copy( void* dst, gh_dtype dst_dt, const void* src, gh_dtype src_dt, uint64_t n, gh_copy_kind kind, gh_stream stream )
{
  if ( int rc = ensure_init() ) {
    return rc;
  }
  if ( n == 0 ) {
    return GH_OK;
  }
  GH_REQUIRE( dst && src, "gh_convert_and_copy: NULL pointer" );
  GH_REQUIRE( ( dst_dt == GH_F16 || dst_dt == GH_F32 ) && ( src_dt == GH_F16 || src_dt == GH_F32 ), "gh_convert_and_copy: unsupported dtype" );
  GH_REQUIRE( kind == GH_HOST_TO_DEVICE || kind == GH_DEVICE_TO_HOST || kind == GH_DEVICE_TO_DEVICE || kind == GH_HOST_TO_HOST,
              "gh_convert_and_copy: bad copy kind %d", (int)kind );
  if ( dst_dt == src_dt ) {
    return gh_memcpy( dst, src, n * dtype_size( dst_dt ), kind, 0, stream );
  }
  hipStream_t st = as_stream( stream );
  if ( kind == GH_DEVICE_TO_DEVICE ) {
    if ( int rc = gh_convert( dst, dst_dt, src, src_dt, n, stream ) ) {
      return rc;
    }
    GH_HIP( hipStreamSynchronize( st ) );
    return GH_OK;
  }
  // a device target never converts host memory into host memory (LOG(FATAL) "Invalid copy type" in arch/cuda/llama2/ops.cuh:490)
  GH_REQUIRE( kind != GH_HOST_TO_HOST, "gh_convert_and_copy: a converting copy needs a device side" );
  void* tmp = nullptr;
  const gh_dtype tmp_dt = kind == GH_HOST_TO_DEVICE ? src_dt : dst_dt;
  if ( int rc = stream_scratch( st, SCRATCH_CONVERT, n * dtype_size( tmp_dt ), 4ull << 20, &tmp ) ) {
    return rc;
  }
  if ( kind == GH_HOST_TO_DEVICE ) {
    GH_HIP( hipMemcpyAsync( tmp, src, n * dtype_size( src_dt ), hipMemcpyHostToDevice, st ) );
    if ( int rc = gh_convert( dst, dst_dt, tmp, src_dt, n, stream ) ) {
      (void)hipStreamSynchronize( st );
      return rc;
    }
  } else {
    if ( int rc = gh_convert( tmp, dst_dt, src, src_dt, n, stream ) ) {
      return rc;
    }
    GH_HIP( hipMemcpyAsync( dst, tmp, n * dtype_size( dst_dt ), hipMemcpyDeviceToHost, st ) );
  }
  GH_HIP( hipStreamSynchronize( st ) );
  return GH_OK;
}

} // extern "C"
