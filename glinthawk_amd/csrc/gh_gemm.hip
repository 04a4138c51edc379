// Dense projection GEMM of the stage: xout(b, r) = sum_p w(r, p) * x(b, p), w row-major (r, s), fp32 accumulate
// (Operations::matmul / untemplated_matmul, arch/amd64/common/ops.hh:74-93,212-271): which kernel takes a product, and the entry points.
//
//   f16, bf16   s % 8 == 0 and 16-byte aligned operands: the ring kernel (gh_gemm_ring.hip), 128 x 128 tiles (gh_gemm_tile.hip) or 256 x 256 tiles
//               (gh_gemm_tile256.hip), by estimated time: half_plan()
//   otherwise   the kernel of this file.  A work-group owns a 64-row slab of w and a 64-column slab of the batch, walks K in steps of 128,
//               stages both tiles in LDS with 16-byte chunks XOR-swizzled so that the MFMA-operand reads are bank-conflict free, and keeps
//               4 x (16x16) fp32 accumulators per wave (v_mfma_f32_16x16x32_f16 / _bf16).  Where r / 64 is too small to fill the chip K is
//               split across work-groups and an fp32 partial buffer is reduced by a second kernel.
//   f32         gh_gemm_f32.hip
#include "gh_product.h"

#include <cstdlib>
#include <mutex>
#include <type_traits>

namespace gh {

// weights through registers, on request only (gh_gemm_stream.hip)
bool gemm_stream_applicable( uint64_t s, uint64_t r, uint64_t b, const void* x, const void* w, const void* xout );
void gemm_stream_plan( uint64_t s, uint64_t r, uint64_t b, uint32_t* splits_out, uint32_t* k_per_split_out, uint32_t* rows_per_wg_out );
template<typename E>
int gemm_stream_launch( E* xout, float* partial, const E* x, const E* w, uint64_t s, uint64_t r, uint64_t b, uint32_t splits,
                        uint32_t k_per_split, uint32_t rows_per_wg, bool write_partials, hipStream_t st );
void gemm_stream_tuning( int target_wgs, int depth );
void gemm_stream_gate_waves( int waves );
int gemm_stream_gate_waves();
bool gemm_stream_gate_applicable( uint64_t s, uint64_t hidden, uint64_t b, const void* x, const void* w13, const void* hb, uint64_t hb_stride );
template<typename E>
int gemm_stream_gate_launch( E* hb, uint64_t hb_stride, const E* x, const E* w13, uint64_t s, uint64_t hidden, uint64_t b, hipStream_t st );
// 256 x 256 tile kernel for products with enough tiles (gh_gemm_tile256.hip)
bool gemm_tile256_takes( uint64_t s, uint64_t b, const void* x, const void* w, const void* xout );
bool gemm_tile256_fills( uint64_t r, uint64_t b );
double gemm_tile256_ns( uint64_t s, uint64_t r, uint64_t b );
template<typename E>
int gemm_tile256_launch( E* xout, float* partial, const E* x, const E* w, uint64_t s, uint64_t r, uint64_t b, int epilogue, hipStream_t st,
                         uint32_t splits, uint32_t k_len, E* xout2 = nullptr, uint64_t r_first = 0, const GateRows* gate = nullptr, const QkvRows* qkv = nullptr );
bool gemm_tile256_qkv_fits( const QkvRows& q );
uint64_t gemm_tile256_rounds( uint64_t r, uint64_t b );
uint64_t gemm_tile256_tokens( uint64_t r, uint64_t b, uint64_t rounds );
void gemm_tile256_split_plan( uint64_t s, uint64_t r, uint64_t b, uint32_t* splits, uint32_t* k_len, double* ns );
void gemm_tile256_tuning( int rows );
// 128 x 128 tiles, two work-groups a CU (gh_gemm_tile.hip)
bool gemm_tile_applicable( uint64_t s, uint64_t r, uint64_t b, const void* x, const void* w, const void* xout );
void gemm_tile_plan( uint64_t s, uint64_t r, uint64_t b, uint32_t* splits_out, uint32_t* k_per_split_out );
double gemm_tile_ns( uint64_t s, uint64_t r, uint64_t b );
template<typename E>
int gemm_tile_launch( E* xout, float* partial, const E* x, const E* w, uint64_t s, uint64_t r, uint64_t b, uint32_t splits, uint32_t k_per_split, hipStream_t st );
// up to some hundred rows (gh_gemm_ring.hip)
bool gemm_ring_applicable( uint64_t s, uint64_t r, uint64_t b, const void* x, const void* w, const void* xout );
uint32_t gemm_ring_splits( uint64_t s, uint64_t r, uint64_t b, double* ns );
template<typename E>
int gemm_ring_launch( E* xout, float* partial, const E* x, const E* w, uint64_t s, uint64_t r, uint64_t b, hipStream_t st );
double gemm_ring_gate_ns( uint64_t s, uint64_t hidden, uint64_t b );
bool gemm_ring_gate_applicable( uint64_t s, uint64_t hidden, uint64_t b, const void* x, const void* w13, const void* hb, uint64_t hb_stride );
template<typename E>
int gemm_ring_gate_launch( E* hb, const GateRows& gate, const E* x, const E* w13, uint64_t s, uint64_t hidden, uint64_t b, hipStream_t st );
void gemm_ring_tuning( int target_wgs );
int gemm_ring_cut( uint64_t s, uint64_t r, uint64_t b, bool gate, uint32_t* plan );
// fp32 (gh_gemm_f32.hip)
int gemm_f32( float* out, const float* x, const float* norm, const float* w, uint64_t s, uint64_t r, uint64_t b, hipStream_t st );

namespace {

// the 16-bit kernels by their storage type: `run` gets a null pointer of it
template<typename F>
int with_half_type( gh_dtype dt, F&& run )
{
  return dt == GH_BF16 ? run( static_cast<__bf16*>( nullptr ) ) : run( static_cast<__half*>( nullptr ) );
}
inline bool is_half_type( gh_dtype dt ) { return dt == GH_F16 || dt == GH_BF16; }

int g_force_kernel = 0; // 0 auto, 1 small tiled kernel of this file, 2 streaming kernel, 3 128 x 128 tiles (b > 64), 4 256 x 256 tiles, 5 ring kernel
// GLINT_LIBRARY_ROWS in the environment overrides the default (for the command-line profilers, which have no other way in)
uint64_t library_rows_default()
{
  const char* env = getenv( "GLINT_LIBRARY_ROWS" );
  return env != nullptr && *env != '\0' ? strtoull( env, nullptr, 10 ) : 0;
}
uint64_t g_library_rows = library_rows_default(); // 0: never; else plain products of this many rows and more go to the vendor's GEMM library (gh_gemm_set_library_rows)

typedef float f32x4 __attribute__( ( ext_vector_type( 4 ) ) );

constexpr int BM = 64;  // weight rows per work-group
constexpr int BN = 64;  // batch columns per work-group
constexpr int BK = 128; // k per stage (16 chunks of 8 halves)

// split-K partials: a grow-only buffer per stream, so that products queued on different streams never share one
int ensure_workspace( uint64_t bytes, float** out, hipStream_t st )
{
  void* p = nullptr;
  if ( int rc = stream_scratch( st, SCRATCH_GEMM_PARTIALS, bytes, 64ull << 20, &p ) ) {
    return rc;
  }
  *out = static_cast<float*>( p );
  return GH_OK;
}

// Loads one (64 x 128) f16 tile, rows [row0, row0+64) x k [k0, k0+128) of a row-major matrix with
// leading dimension ld, into registers: thread t handles chunk (t % 16) of rows t/16 + 16*i.
// Rows >= n_rows and k >= k_end read as zero.
struct TileRegs
{
  uint4 v[4];
};

template<typename E>
__device__ __forceinline__ TileRegs load_tile( const E* __restrict__ mat, uint64_t ld, uint32_t row0, uint32_t n_rows, uint32_t k0, uint32_t k_end, bool k_vec_ok )
{
  TileRegs t;
  const uint32_t chunk = threadIdx.x & 15;
  const uint32_t k = k0 + chunk * 8;
#pragma unroll
  for ( int i = 0; i < 4; i++ ) {
    const uint32_t row = row0 + ( threadIdx.x >> 4 ) + 16 * i;
    uint4 v = make_uint4( 0, 0, 0, 0 );
    if ( row < n_rows && k < k_end ) {
      const E* p = mat + (uint64_t)row * ld + k;
      if ( k_vec_ok && k + 8 <= k_end ) {
        v = *reinterpret_cast<const uint4*>( p );
      } else {
        union
        {
          uint4 raw;
          E h[8];
        } u;
        u.raw = make_uint4( 0, 0, 0, 0 );
        for ( int e = 0; e < 8; e++ ) {
          if ( k + e < k_end ) {
            u.h[e] = p[e];
          }
        }
        v = u.raw;
      }
    }
    t.v[i] = v;
  }
  return t;
}

__device__ __forceinline__ void store_tile( uint4* lds, const TileRegs& t )
{
  const uint32_t chunk = threadIdx.x & 15;
#pragma unroll
  for ( int i = 0; i < 4; i++ ) {
    const uint32_t row = ( threadIdx.x >> 4 ) + 16 * i;
    lds[row * 16 + ( chunk ^ ( row & 15 ) )] = t.v[i];
  }
}

// grid: (ceil(r / 64), ceil(b / 64), k_splits)
template<typename E, bool SPLIT>
__global__ __launch_bounds__( 256 ) void gemm_mfma_kernel( E* __restrict__ xout,
                                                          float* __restrict__ partial,
                                                          const E* __restrict__ x,
                                                          const E* __restrict__ w,
                                                          uint32_t s,
                                                          uint32_t r,
                                                          uint32_t b,
                                                          uint32_t k_per_split,
                                                          bool k_vec_ok )
{
  __shared__ uint4 s_w[2][BM * 16];
  __shared__ uint4 s_x[2][BN * 16];

  const uint32_t row0 = blockIdx.x * BM;
  const uint32_t col0 = blockIdx.y * BN;
  const uint32_t k_begin = blockIdx.z * k_per_split;
  const uint32_t k_end = min( s, k_begin + k_per_split );
  const uint32_t wave = threadIdx.x >> 6;
  const uint32_t lane = threadIdx.x & 63;
  const uint32_t c = lane & 15;
  const uint32_t g4 = lane >> 4;

  f32x4 acc[4];
#pragma unroll
  for ( int j = 0; j < 4; j++ ) {
    acc[j] = f32x4 { 0.0f, 0.0f, 0.0f, 0.0f };
  }

  TileRegs tw = load_tile( w, s, row0, r, k_begin, k_end, k_vec_ok );
  TileRegs tx = load_tile( x, s, col0, b, k_begin, k_end, k_vec_ok );
  int buf = 0;
  for ( uint32_t k0 = k_begin; k0 < k_end; k0 += BK ) {
    store_tile( s_w[buf], tw );
    store_tile( s_x[buf], tx );
    __syncthreads();
    if ( k0 + BK < k_end ) {
      tw = load_tile( w, s, row0, r, k0 + BK, k_end, k_vec_ok );
      tx = load_tile( x, s, col0, b, k0 + BK, k_end, k_vec_ok );
    }
    const uint4* lw = s_w[buf];
    const uint4* lx = s_x[buf];
    const uint32_t arow = wave * 16 + c;
#pragma unroll
    for ( int kk = 0; kk < 4; kk++ ) {
      const uint32_t ch = 4 * kk + g4;
      const typename Mfma<E>::x8 a = __builtin_bit_cast( typename Mfma<E>::x8, lw[arow * 16 + ( ch ^ ( arow & 15 ) )] );
#pragma unroll
      for ( int j = 0; j < 4; j++ ) {
        const uint32_t brow = 16 * j + c;
        const typename Mfma<E>::x8 bb = __builtin_bit_cast( typename Mfma<E>::x8, lx[brow * 16 + ( ch ^ ( brow & 15 ) )] );
        acc[j] = Mfma<E>::k32( a, bb, acc[j] );
      }
    }
    buf ^= 1; // the other buffer is free: its readers passed the barrier of this iteration
  }

  // acc[j][i] = out(row0 + 16*wave + 4*g4 + i, col0 + 16*j + c)
#pragma unroll
  for ( int j = 0; j < 4; j++ ) {
    const uint32_t col = col0 + 16 * j + c;
    if ( col >= b ) {
      continue;
    }
#pragma unroll
    for ( int i = 0; i < 4; i++ ) {
      const uint32_t row = row0 + 16 * wave + 4 * g4 + i;
      if ( row < r ) {
        if ( SPLIT ) {
          partial[( (uint64_t)blockIdx.z * b + col ) * r + row] = acc[j][i];
        } else {
          xout[(uint64_t)col * r + row] = from_f32<E>( acc[j][i] );
        }
      }
    }
  }
}

template<typename E>
__global__ __launch_bounds__( 256 ) void gemm_reduce_kernel( E* __restrict__ xout, const float* __restrict__ partial, uint64_t n, uint32_t splits )
{
  const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
  for ( uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride ) {
    // ascending order of the split, four loads in flight: a split past the last reads the last again and is not added
    float sum = 0.0f;
    for ( uint32_t k0 = 0; k0 < splits; k0 += 4 ) {
      float p[4];
#pragma unroll
      for ( uint32_t u = 0; u < 4; u++ ) {
        p[u] = partial[(uint64_t)min( k0 + u, splits - 1 ) * n + i];
      }
#pragma unroll
      for ( uint32_t u = 0; u < 4; u++ ) {
        sum += k0 + u < splits ? p[u] : 0.0f;
      }
    }
    xout[i] = from_f32<E>( sum );
  }
}

// Few weight rows (r <= 32: the gates of a recurrent mixer) under many activation rows: bound by the activations, which the tile kernels
// would read with most of their matrix work wasted on rows that are not there.  A work-group takes 32 activation rows, its four waves every
// fourth 64 of the K range, straight from memory in operand order (a row's 64 bytes an instruction, the rest of the line by the next);
// their sums meet in LDS.  What counts is how much is asked for at once: two pieces of 64 k a wave, the next as soon as one is multiplied.  16 rows of 4096 k,
// calls in a row: 8192 activation rows, one piece at a time and 32 bytes of a row an instruction 25.0 us, so 21.7 (3.1 TB/s; the rest of the time is the launch,
// the first loads and the sums); 256 rows 15.2 -> 14.3, 32768 71 -> 63.  Four and eight pieces 21.4 and 22.3, 65 and 68.  The order of the sums is that of
// v_mfma_f32_32x32x16_bf16, two of which in turn are one of the instructions here, bit for bit.  Eight waves with every eighth 64 each (19.8, 14.3 and 57 us) give other bits.
// fp32 output (b, r).  s % 256 == 0, 16-byte aligned operands.  TILES: of 16 weight rows.
constexpr uint32_t SKINNY_ROWS = 32, SKINNY_WAVES = 4, SKINNY_AHEAD = 2;
template<typename E, int TILES>
__global__ __launch_bounds__( SKINNY_WAVES * 64 ) void gemm_skinny_kernel( float* __restrict__ out, const E* __restrict__ x, const E* __restrict__ w, uint32_t s, uint32_t r, uint32_t b )
{
  typedef typename Mfma<E>::x8 x8;
  __shared__ float sums[SKINNY_WAVES][8 * TILES][64];
  const uint32_t wave = threadIdx.x >> 6, lane = threadIdx.x & 63, fr = lane & 15, g = lane >> 4;
  const uint32_t token0 = blockIdx.x * 32;
  const E *xp[2], *wp[TILES]; // rows past the last repeat it and are not stored
#pragma unroll
  for ( uint32_t t = 0; t < 2; t++ ) {
    xp[t] = x + (uint64_t)min( token0 + 16 * t + fr, b - 1 ) * s + 64 * wave + 8 * g;
  }
#pragma unroll
  for ( uint32_t i = 0; i < TILES; i++ ) {
    wp[i] = w + (uint64_t)min( 16 * i + fr, r - 1 ) * s + 64 * wave + 8 * g;
  }
  mfma_f32x4 acc[TILES][2];
#pragma unroll
  for ( int i = 0; i < TILES; i++ ) {
    acc[i][0] = acc[i][1] = mfma_f32x4 { 0.0f, 0.0f, 0.0f, 0.0f };
  }
  x8 xv[SKINNY_AHEAD][2][2], wv[SKINNY_AHEAD][2][TILES];
  auto ask = [&]( int u, uint32_t k ) __attribute__( ( always_inline ) ) { // 64 k
#pragma unroll
    for ( int h = 0; h < 2; h++ ) {
#pragma unroll
      for ( int t = 0; t < 2; t++ ) {
        xv[u][h][t] = *reinterpret_cast<const x8*>( xp[t] + k + 32 * h );
      }
#pragma unroll
      for ( int i = 0; i < TILES; i++ ) {
        wv[u][h][i] = *reinterpret_cast<const x8*>( wp[i] + k + 32 * h );
      }
    }
  };
  auto multiply = [&]( int u ) __attribute__( ( always_inline ) ) {
#pragma unroll
    for ( int h = 0; h < 2; h++ ) {
#pragma unroll
      for ( int i = 0; i < TILES; i++ ) {
#pragma unroll
        for ( int t = 0; t < 2; t++ ) {
          acc[i][t] = Mfma<E>::k32( wv[u][h][i], xv[u][h][t], acc[i][t] );
        }
      }
    }
  };
  constexpr uint32_t STEP = 64 * SKINNY_WAVES;
#pragma unroll
  for ( int u = 0; u < (int)SKINNY_AHEAD; u++ ) {
    if ( u * STEP < s ) {
      ask( u, u * STEP );
    }
  }
  uint32_t k = 0; // (of wave 0; the others' pieces lie behind its)
  for ( ; k + ( 2 * SKINNY_AHEAD - 1 ) * STEP < s; k += SKINNY_AHEAD * STEP ) {
#pragma unroll
    for ( int u = 0; u < (int)SKINNY_AHEAD; u++ ) {
      multiply( u );
      __builtin_amdgcn_sched_barrier( 0 );
      ask( u, k + ( SKINNY_AHEAD + u ) * STEP );
      __builtin_amdgcn_sched_barrier( 0 );
    }
  }
  for ( ; k < s; k += SKINNY_AHEAD * STEP ) {
#pragma unroll
    for ( int u = 0; u < (int)SKINNY_AHEAD; u++ ) {
      if ( k + u * STEP < s ) {
        multiply( u );
      }
      if ( k + ( SKINNY_AHEAD + u ) * STEP < s ) {
        ask( u, k + ( SKINNY_AHEAD + u ) * STEP );
      }
    }
  }
  // acc[i][t][v]: weight row 16 i + 4 g + v, token 16 t + fr
#pragma unroll
  for ( int i = 0; i < TILES; i++ ) {
#pragma unroll
    for ( int t = 0; t < 2; t++ ) {
#pragma unroll
      for ( int v = 0; v < 4; v++ ) {
        sums[wave][8 * i + 4 * t + v][lane] = acc[i][t][v];
      }
    }
  }
  __syncthreads();
#pragma unroll
  for ( uint32_t n = 0; n < 8 * TILES / SKINNY_WAVES; n++ ) {
    const uint32_t at = wave * ( 8 * TILES / SKINNY_WAVES ) + n;
    float y[SKINNY_WAVES];
#pragma unroll
    for ( uint32_t o = 0; o < SKINNY_WAVES; o++ ) {
      y[o] = sums[o][at][lane];
    }
    const float sum = ( y[0] + y[1] ) + ( y[2] + y[3] );
    const uint32_t row = 16 * ( at / 8 ) + 4 * g + at % 4, token = token0 + 16 * ( ( at / 4 ) % 2 ) + fr;
    if ( row < r && token < b ) {
      out[(uint64_t)token * r + row] = sum;
    }
  }
}

} // namespace
} // namespace gh

namespace gh {

// The stores of the ring kernel, 8 bytes a lane with nothing to hide them; what the steps of a long K range are priced at covers part of it
// (32000 x 64 at 7000 rows: 400 us, of which the one step is 20).
static double ring_stores_ns( uint64_t s, uint64_t r, uint64_t b ) { return (double)( b * r ) / 1000.0 * std::min( 1.0, 1024.0 / (double)s ); }

// Which kernel takes a 16-bit product that all of them can take (s % 8 == 0, 16-byte aligned operands), by what each is estimated to need:
// the estimates are fitted to timings of 65 shapes of 64 to 11008 k and 288 to 32000 weight rows at 17 row counts from 65 to 7000, where the
// choice is 1 % off the fastest on average.  The same whether the rounded result is wanted or, for the kernel that follows, its fp32 sums: both
// calls give the same bits.
enum class HalfKernel { ring, tile128, tile256, tile256_split };
struct HalfPlan
{
  HalfKernel kernel { HalfKernel::ring };
  uint32_t splits { 1 }, k_len { 0 };
  double ns { 0.0 };      // to the rounded result
  double sums_ns { 0.0 }; // to the fp32 sums, the reading of them included
};
static HalfPlan half_plan( uint64_t s, uint64_t r, uint64_t b, bool whole_tiles )
{
  const double plane_ns = (double)( b * r ) * 8.0 / 5000.0; // fp32 sums of one K range written and read
  auto priced = [&]( HalfKernel kernel, uint32_t splits, uint32_t k_len, double kernel_ns, double store_ns ) {
    const double sums_ns = kernel_ns + splits * plane_ns;
    return HalfPlan { kernel, splits, k_len, splits > 1 ? sums_ns + GEMM_REDUCE_NS : kernel_ns + store_ns, sums_ns };
  };
  double ns = 0.0;
  uint32_t splits = gemm_ring_splits( s, r, b, &ns ), k_len = 0;
  HalfPlan best = priced( HalfKernel::ring, splits, 0, ns, ring_stores_ns( s, r, b ) );
  auto better = [&]( const HalfPlan& plan ) {
    if ( plan.ns <= best.ns ) {
      best = plan;
    }
  };
  if ( b > 64 ) {
    gemm_tile_plan( s, r, b, &splits, &k_len );
    better( priced( HalfKernel::tile128, splits, k_len, gemm_tile_ns( s, r, b ), 0.0 ) );
  }
  if ( gemm_tile256_takes( s, b, nullptr, nullptr, nullptr ) ) {
    gemm_tile256_split_plan( s, r, b, &splits, &k_len, &ns );
    if ( splits > 1 ) {
      better( priced( HalfKernel::tile256_split, splits, k_len, ns - splits * plane_ns, 0.0 ) );
    }
    if ( whole_tiles ) {
      better( priced( HalfKernel::tile256, 1, 0, gemm_tile256_ns( s, r, b ), 0.0 ) );
    }
  }
  return best;
}

// a product runs on the kernel that was asked for, and no other is tried in front of it
bool gemm_kernel_forced() { return g_force_kernel != 0; }

// Whether a product runs as whole tiles of 256 x 256 (what is left of it once gemm_token_split() has cut it).
static bool tile256_wanted( uint64_t s, uint64_t r, uint64_t b, const void* x, const void* w, const void* xout )
{
  if ( !gemm_tile256_takes( s, b, x, w, xout ) ) {
    return false;
  }
  return g_force_kernel == 4 ? gemm_tile256_fills( r, b ) : g_force_kernel == 0 && half_plan( s, r, b, true ).kernel == HalfKernel::tile256;
}

// Tokens of the first part when a product, `whole_ns` in one, is better run as whole rounds of 256 x 256 tiles and a rest, rest_ns( tokens ); 0 otherwise.
template<typename F>
static uint64_t cut_tokens( uint64_t s, uint64_t r, uint64_t b, double whole_ns, F&& rest_ns )
{
  double best = whole_ns;
  uint64_t best_b1 = 0;
  const uint64_t rounds = gemm_tile256_rounds( r, b );
  for ( uint64_t n = 1; n < 3 && n < rounds; n++ ) { // the first part one round shorter, or two
    const uint64_t b1 = gemm_tile256_tokens( r, b, rounds - n );
    if ( b1 < 192 || ( b1 * r * 2 ) % 16 != 0 ) {
      break;
    }
    // a second launch, and 2 % for what the estimates don't know
    const double cost = ( gemm_tile256_ns( s, r, b1 ) + rest_ns( b - b1 ) + 2000.0 ) * 1.02;
    if ( cost < best ) {
      best = cost;
      best_b1 = b1;
    }
  }
  return best_b1;
}

uint64_t gemm_token_split( uint64_t s, uint64_t r, uint64_t b, gh_dtype dt, const void* x, const void* w, const void* xout )
{
  if ( !is_half_type( dt ) || g_force_kernel != 0 || !gemm_tile256_takes( s, b, x, w, xout ) ) {
    return 0;
  }
  return cut_tokens( s, r, b, half_plan( s, r, b, true ).ns, [&]( uint64_t rest ) { return half_plan( s, r, rest, false ).ns; } );
}

// Which kernel takes w1, w3 and the gate in one launch (what is left of it once gemm_token_split() has cut it); none: two launches.
enum class GateKernel { none, stream, ring, tiles };
static GateKernel gate_kernel( const void* hb, const GateRows& gate, const void* x, const void* w13, uint64_t s, uint64_t hidden, uint64_t b, gh_dtype dt, double* ns )
{
  *ns = 0.0;
  const bool plain_silu = gate.activation == GH_ACT_SILU && gate.bias == nullptr;
  // other gates of many rows: only the tiles have a variant for them, bf16 and over the fp32 sums
  const bool tiles_only = !plain_silu && b >= 192;
  if ( !is_half_type( dt ) || ( tiles_only && ( dt != GH_BF16 || !gate.exact ) ) ) {
    return GateKernel::none;
  }
  if ( ( g_force_kernel == 2 || ( g_force_kernel == 0 && gemm_stream_gate_waves() != 0 ) ) && b <= 64 && plain_silu
       && gemm_stream_gate_applicable( s, hidden, b, x, w13, hb, gate.stride ) ) {
    return GateKernel::stream;
  }
  if ( b > 64 && ( gemm_library_wanted_wide( s, 2 * hidden, b, dt, x, w13, hb ) || gemm_library_wanted( s, hidden, b, dt, x, w13, hb ) ) ) {
    return GateKernel::none;
  }
  const bool rows_of_eight = gate.stride % 8 == 0 && hidden % 8 == 0;
  if ( g_force_kernel != 0 ) {
    return g_force_kernel == 4 && rows_of_eight && tile256_wanted( s, 2 * hidden, b, x, w13, hb ) ? GateKernel::tiles
           : g_force_kernel == 5 && !tiles_only && gemm_ring_gate_applicable( s, hidden, b, x, w13, hb, gate.stride )
             ? GateKernel::ring
             : GateKernel::none;
  }
  if ( !gemm_ring_gate_applicable( s, hidden, b, x, w13, hb, gate.stride ) ) {
    return GateKernel::none;
  }
  // From 192 rows on 256 x 256 tiles where they are enough (70B, 256 rows: 221 us with the gate behind them, the ring kernel 270).  The ring kernel
  // splits no K range here: where too few rows fill the chip (2 x 1024 of 2048 k at 8 rows: 11.6 us) the split of the plain product with the
  // gate's kernel behind it (about 4.5 us) is faster (8.2).  A gate over the fp32 sums of many rows takes such a split only: unsplit products of so
  // many rows leave rounded factors.
  if ( tiles_only ) { // against a product of rounded factors and the gate's kernel, which reads them once more
    const double tile_ns = gemm_tile256_ns( s, 2 * hidden, b ), two_ns = half_plan( s, 2 * hidden, b, false ).ns + 3000.0 + (double)( 3 * b * hidden ) * 2.0 / 5000.0;
    *ns = std::min( tile_ns, two_ns );
    return rows_of_eight && gemm_tile256_takes( s, b, x, w13, hb ) && tile_ns <= two_ns ? GateKernel::tiles : GateKernel::none;
  }
  const bool keeps_sums = gate.exact && b >= PRODUCT_ROUNDED_ROWS;
  const double ring_ns = gemm_ring_gate_ns( s, hidden, b ) + ring_stores_ns( s, hidden, b );
  double two_ns = 0.0;
  if ( keeps_sums ) {
    const uint32_t splits = gemm_ring_splits( s, 2 * hidden, b, &two_ns );
    two_ns = splits > 1 ? two_ns + splits * (double)( 2 * b * hidden ) * 8.0 / 5000.0 + 4500.0 : 1e30;
  } else {
    two_ns = half_plan( s, 2 * hidden, b, false ).sums_ns + 4500.0;
  }
  if ( rows_of_eight && gemm_tile256_takes( s, b, x, w13, hb ) && gemm_tile256_ns( s, 2 * hidden, b ) <= std::min( ring_ns, two_ns ) ) {
    *ns = gemm_tile256_ns( s, 2 * hidden, b );
    return GateKernel::tiles;
  }
  *ns = std::min( ring_ns, two_ns );
  return ring_ns <= two_ns ? GateKernel::ring : GateKernel::none;
}

int gemm_gate_one_launch( void* hb, const GateRows& gate, const void* x, const void* w13, uint64_t s, uint64_t hidden, uint64_t b, gh_dtype dt, hipStream_t st,
                          bool* done )
{
  *done = false;
  if ( !is_half_type( dt ) || overlap( hb, ( ( b - 1 ) * gate.stride + hidden ) * 2, x, b * s * 2 ) ) {
    return GH_OK;
  }
  double ns = 0.0;
  const GateKernel kernel = gate_kernel( hb, gate, x, w13, s, hidden, b, dt, &ns );
  if ( kernel == GateKernel::none ) {
    return GH_OK;
  }
  if ( g_force_kernel == 0 && kernel != GateKernel::stream && gate.context_rows == nullptr // (rows of contexts are counted from the first)
       && gate.stride % 8 == 0 && hidden % 8 == 0 && gemm_tile256_takes( s, b, x, w13, hb ) ) {
    // `rest` tokens after those of the first part; only if the gate rides in both launches
    auto rest_ns = [&]( uint64_t rest ) {
      double first_ns = 0.0, last_ns = 0.0;
      const GateKernel first = gate_kernel( hb, gate, x, w13, s, hidden, b - rest, dt, &first_ns ), last = gate_kernel( hb, gate, x, w13, s, hidden, rest, dt, &last_ns );
      return first != GateKernel::none && last != GateKernel::none ? last_ns : 1e30;
    };
    if ( const uint64_t b1 = cut_tokens( s, 2 * hidden, b, ns, rest_ns ) ) {
      if ( int rc = gemm_gate_one_launch( hb, gate, x, w13, s, hidden, b1, dt, st, done ) ) {
        return rc;
      }
      return gemm_gate_one_launch( static_cast<char*>( hb ) + b1 * gate.stride * 2, gate, static_cast<const char*>( x ) + b1 * s * 2, w13, s, hidden, b - b1, dt, st,
                                   done );
    }
  }
  *done = true;
  return with_half_type( dt, [&]( auto* e ) {
    using E = std::remove_pointer_t<decltype( e )>;
    E* out = static_cast<E*>( hb );
    const E *in = static_cast<const E*>( x ), *mat = static_cast<const E*>( w13 );
    switch ( kernel ) {
      case GateKernel::stream: return gemm_stream_gate_launch<E>( out, gate.stride, in, mat, s, hidden, b, st );
      case GateKernel::tiles: return gemm_tile256_launch<E>( out, nullptr, in, mat, s, hidden, b, 2, st, 1, 0, nullptr, 0, &gate );
      default: return gemm_ring_gate_launch<E>( out, gate, in, mat, s, hidden, b, st );
    }
  } );
}

// Many rows: the large tile kernel with the op that follows the product in its epilogue, 1 = xout += product
// (accum).  *done = false: nothing was launched (shape or alignment not for that kernel), the caller takes
// its other route.
bool gemm_tile_epilogue_applicable( uint64_t s, uint64_t r, uint64_t b, gh_dtype dt, const void* x, const void* w, const void* xout )
{
  if ( !is_half_type( dt ) || r % 8 != 0 || !gemm_tile256_takes( s, b, x, w, xout ) ) {
    return false;
  }
  if ( g_force_kernel != 0 ) {
    return tile256_wanted( s, r, b, x, w, xout );
  }
  // Unsplit 128 x 128 tiles sum in the same order, but would leave fp32 sums here (1024 x 1024, 7000 rows with the norm: 46 us so, 67 with them).
  const HalfPlan plan = half_plan( s, r, b, true );
  return plan.kernel == HalfKernel::tile256
         || ( plan.kernel == HalfKernel::tile128 && plan.splits == 1 && gemm_tile256_ns( s, r, b ) <= plan.sums_ns );
}

int gemm_tile_epilogue_launch( void* xout, const void* x, const void* w, uint64_t s, uint64_t r, uint64_t b, gh_dtype dt, int epilogue, hipStream_t st,
                               bool* done )
{
  *done = false;
  if ( !gemm_tile_epilogue_applicable( s, r, b, dt, x, w, xout ) ) {
    return GH_OK;
  }
  *done = true;
  return with_half_type( dt, [&]( auto* e ) {
    using E = std::remove_pointer_t<decltype( e )>;
    return gemm_tile256_launch<E>( static_cast<E*>( xout ), nullptr, static_cast<const E*>( x ), static_cast<const E*>( w ), s, r, b, epilogue, st, 1, 0 );
  } );
}

// Many rows of q, k and v in one launch that rotates and appends them (f16); *done = false: nothing was launched.
bool gemm_tile_qkv_applicable( uint64_t s, uint64_t b, gh_dtype dt, const void* x, const void* wqkv, const void* q, const QkvRows& rows )
{
  return dt == GH_F16 && gemm_tile256_qkv_fits( rows ) && gemm_tile_epilogue_applicable( s, rows.dim + 2ull * rows.kv_dim, b, dt, x, wqkv, q );
}
int gemm_tile_qkv_launch( void* q, const void* x, const void* wqkv, uint64_t s, uint64_t b, gh_dtype dt, const QkvRows& rows, hipStream_t st, bool* done )
{
  *done = gemm_tile_qkv_applicable( s, b, dt, x, wqkv, q, rows );
  return *done ? gemm_tile256_launch<__half>( static_cast<__half*>( q ), nullptr, static_cast<const __half*>( x ), static_cast<const __half*>( wqkv ), s,
                                              rows.dim + 2ull * rows.kv_dim, b, 4, st, 1, 0, nullptr, 0, nullptr, &rows )
               : GH_OK;
}

static bool skinny_takes( uint64_t s, uint64_t r, uint64_t b, const void* x, const void* w )
{
  return g_force_kernel == 0 && r <= SKINNY_ROWS && b >= 192 && b < ( 1ull << 31 ) && s % 256 == 0
         && ( ( reinterpret_cast<uintptr_t>( x ) | reinterpret_cast<uintptr_t>( w ) ) & 15u ) == 0;
}

// The 16-bit part of gemm_partials(): runs the GEMM proper.  With `want_partials` the result is always left as fp32 partial sums
// `[splits][b][r]` in the library's workspace (*partial_out, *splits_out) for a fused epilogue; otherwise the kernel may store
// DType results straight into `xout` (*splits_out == 0 then).
template<typename E>
int gemm_half_partials( E* xout, const E* x, const E* w, uint64_t s, uint64_t r, uint64_t b, hipStream_t st, bool want_partials, float** partial_out,
                        uint32_t* splits_out )
{
  if ( want_partials && skinny_takes( s, r, b, x, w ) ) {
    float* ws = nullptr;
    if ( int rc = ensure_workspace( b * r * sizeof( float ), &ws, st ) ) {
      return rc;
    }
    *partial_out = ws;
    *splits_out = 1;
    auto kernel = r <= 16 ? gemm_skinny_kernel<E, 1> : gemm_skinny_kernel<E, 2>;
    kernel<<<(unsigned)( ( b + 31 ) / 32 ), SKINNY_WAVES * 64, 0, st>>>( ws, x, w, (uint32_t)s, (uint32_t)r, (uint32_t)b );
    GH_LAUNCH_CHECK();
    return GH_OK;
  }
  const void* out = xout ? static_cast<const void*>( xout ) : x;
  HalfPlan plan;
  bool taken = false; // by one of the kernels for aligned operands
  if ( g_force_kernel == 0 ) {
    taken = gemm_ring_applicable( s, r, b, x, w, out );
    if ( taken ) {
      plan = half_plan( s, r, b, true );
    }
  } else if ( g_force_kernel == 3 ) {
    taken = gemm_tile_applicable( s, r, b, x, w, out );
    GH_REQUIRE( taken, "gh_matmul: the 128 x 128 tile kernel needs b > 64, s %% 8 == 0 and 16-byte aligned operands" );
    plan.kernel = HalfKernel::tile128;
    gemm_tile_plan( s, r, b, &plan.splits, &plan.k_len );
  } else if ( g_force_kernel == 4 ) {
    plan.kernel = HalfKernel::tile256;
    taken = tile256_wanted( s, r, b, x, w, out );
    if ( !taken && gemm_tile256_takes( s, b, x, w, x ) ) {
      plan.kernel = HalfKernel::tile256_split;
      gemm_tile256_split_plan( s, r, b, &plan.splits, &plan.k_len, &plan.ns );
      taken = plan.splits > 1;
    }
    GH_REQUIRE( taken, "gh_matmul: the 256 x 256 tile kernel needs b >= 192, at least 192 tiles with a last round that is not mostly empty, s %% 64 == 0 and 16-byte aligned operands" );
  } else if ( g_force_kernel == 5 ) {
    taken = gemm_ring_applicable( s, r, b, x, w, out );
    GH_REQUIRE( taken, "gh_matmul: the ring kernel needs s %% 8 == 0 and 16-byte aligned operands" );
    plan.splits = gemm_ring_splits( s, r, b, &plan.ns );
  }
  if ( taken ) {
    float* ws = nullptr;
    if ( want_partials || plan.splits > 1 ) {
      if ( int rc = ensure_workspace( (uint64_t)plan.splits * b * r * sizeof( float ), &ws, st ) ) {
        return rc;
      }
      *partial_out = ws;
      *splits_out = plan.splits;
    }
    switch ( plan.kernel ) {
      case HalfKernel::tile128: return gemm_tile_launch( xout, ws, x, w, s, r, b, plan.splits, plan.k_len, st );
      case HalfKernel::tile256: return gemm_tile256_launch( xout, ws, x, w, s, r, b, 0, st, 1, 0 );
      case HalfKernel::tile256_split: return gemm_tile256_launch<E>( nullptr, ws, x, w, s, r, b, 0, st, plan.splits, plan.k_len );
      case HalfKernel::ring: break;
    }
    return gemm_ring_launch( xout, ws, x, w, s, r, b, st );
  }

  if ( g_force_kernel == 2 && gemm_stream_applicable( s, r, b, x, w, xout ? xout : x ) ) {
    uint32_t splits = 1, k_per_split = 0, rows_per_wg = 0;
    gemm_stream_plan( s, r, b, &splits, &k_per_split, &rows_per_wg );
    float* ws = nullptr;
    const bool partial = want_partials || splits > 1;
    if ( partial ) {
      if ( int rc = ensure_workspace( (uint64_t)splits * b * r * sizeof( float ), &ws, st ) ) {
        return rc;
      }
      *partial_out = ws;
      *splits_out = splits;
    }
    return gemm_stream_launch( xout, ws, x, w, s, r, b, splits, k_per_split,
                               rows_per_wg, partial, st );
  }
  GH_REQUIRE( g_force_kernel != 2, "gh_matmul: the streaming kernel needs s %% 256 == 0, r %% 4 == 0 and 16-byte aligned operands" );

  const bool k_vec_ok = ( s % 8 == 0 ) && ( ( reinterpret_cast<uintptr_t>( x ) | reinterpret_cast<uintptr_t>( w ) ) & 15u ) == 0;
  const uint32_t grid_m = (uint32_t)( ( r + BM - 1 ) / BM );
  const uint32_t grid_n = (uint32_t)( ( b + BN - 1 ) / BN );
  GH_REQUIRE( grid_n <= 65535, "gh_matmul: batch too large" );
  // split K until there are about 1024 work-groups (4 per CU), keeping at least 1024 k per split
  uint32_t splits = 1;
  const uint64_t tiles = (uint64_t)grid_m * grid_n;
  if ( tiles < 1024 ) {
    splits = (uint32_t)( ( 1024 + tiles - 1 ) / tiles );
    const uint32_t max_by_k = (uint32_t)std::max<uint64_t>( 1, s / 1024 );
    splits = std::min( splits, max_by_k );
    splits = std::min<uint32_t>( splits, 16 );
  }
  uint32_t k_per_split = (uint32_t)( ( s + splits - 1 ) / splits );
  k_per_split = ( k_per_split + BK - 1 ) / BK * BK;
  splits = (uint32_t)( ( s + k_per_split - 1 ) / k_per_split );

  const dim3 grid( grid_m, grid_n, splits );
  if ( splits == 1 && !want_partials ) {
    gemm_mfma_kernel<E, false><<<grid, 256, 0, st>>>( xout, nullptr, x, w,
                                                 (uint32_t)s, (uint32_t)r, (uint32_t)b, k_per_split, k_vec_ok );
    GH_LAUNCH_CHECK();
    return GH_OK;
  }
  float* ws = nullptr;
  if ( int rc = ensure_workspace( (uint64_t)splits * b * r * sizeof( float ), &ws, st ) ) {
    return rc;
  }
  gemm_mfma_kernel<E, true><<<grid, 256, 0, st>>>( nullptr, ws, x, w, (uint32_t)s, (uint32_t)r,
                                              (uint32_t)b, k_per_split, k_vec_ok );
  GH_LAUNCH_CHECK();
  *partial_out = ws;
  *splits_out = splits;
  return GH_OK;
}

int gemm_partials( void* xout, const void* x, const void* w, uint64_t s, uint64_t r, uint64_t b, gh_dtype dt, hipStream_t st, bool want_partials,
                   float** partial_out, uint32_t* splits_out )
{
  *partial_out = nullptr;
  *splits_out = 0;
  if ( dt == GH_F32 ) {
    float* dst = static_cast<float*>( xout );
    if ( want_partials ) {
      if ( int rc = ensure_workspace( b * r * sizeof( float ), &dst, st ) ) {
        return rc;
      }
      *partial_out = dst;
      *splits_out = 1;
    }
    return gemm_f32( dst, static_cast<const float*>( x ), nullptr, static_cast<const float*>( w ), s, r, b, st );
  }
  GH_REQUIRE( is_half_type( dt ), "gh_matmul: unsupported dtype %d", (int)dt );
  return with_half_type( dt, [&]( auto* e ) {
    using E = std::remove_pointer_t<decltype( e )>;
    return gemm_half_partials<E>( static_cast<E*>( xout ), static_cast<const E*>( x ), static_cast<const E*>( w ), s, r, b, st, want_partials, partial_out, splits_out );
  } );
}

} // namespace gh

namespace gh {
// whether a plain product goes to the vendor's library (gh_gemm_lib.hip)
bool gemm_library_wanted( uint64_t s, uint64_t r, uint64_t b, gh_dtype dt, const void* x, const void* w, const void* xout )
{
  const bool aligned = ( ( reinterpret_cast<uintptr_t>( x ) | reinterpret_cast<uintptr_t>( w ) | reinterpret_cast<uintptr_t>( xout ) ) & 15u ) == 0;
  // measured (13B and 70B shapes): from g_library_rows rows on the library's kernels win nearly everywhere; below, the split-K
  // tile kernel and the two-output launch do (w1 and w3 of the 70B shape at 256 rows as two library products: the decode step
  // of 256 slots 10.07 ms against 9.84)
  // from half that row count on as well unless the weight matrix is much wider than tall (w2): measured with the residual add and
  // the norm behind the product, 384-704 rows, 4-50 % faster for every such product of the 7B, 13B and 70B shapes; for w2 the
  // split-K tile kernel keeps up
  const bool rows_enough = b >= g_library_rows || ( 2 * b >= g_library_rows && 2 * r >= s );
  return dt == GH_F16 && g_force_kernel == 0 && g_library_rows > 0 && rows_enough && s % 8 == 0 && r % 8 == 0 && aligned;
}
// a product with many weight rows (w1 and w3 together) of some hundred activation rows, below gemm_library_wanted()'s row count:
// measured on the 13B and 70B shapes, the library wins there from 128 rows on (1.1-1.6 x), which it does not for narrower products
bool gemm_library_wanted_wide( uint64_t s, uint64_t r, uint64_t b, gh_dtype dt, const void* x, const void* w, const void* xout )
{
  const bool aligned = ( ( reinterpret_cast<uintptr_t>( x ) | reinterpret_cast<uintptr_t>( w ) | reinterpret_cast<uintptr_t>( xout ) ) & 15u ) == 0;
  return dt == GH_F16 && g_force_kernel == 0 && g_library_rows > 0 && b >= 128 && b < g_library_rows && r >= 16384 && s % 8 == 0 && r % 8 == 0 && aligned;
}
} // namespace gh

using namespace gh;

extern "C" {

int gh_gemm_set_tuning( int kernel, int target_workgroups, int tile_rows )
{
  g_force_kernel = kernel;
  gemm_stream_tuning( target_workgroups, 0 );
  gemm_ring_tuning( target_workgroups );
  gemm_tile256_tuning( tile_rows );
  return GH_OK;
}

int gh_gemm_set_gate_waves( int waves )
{
  GH_REQUIRE( waves == 0 || waves == 4 || waves == 8, "gh_gemm_set_gate_waves: %d is not 0, 4 or 8", waves );
  gemm_stream_gate_waves( waves );
  return GH_OK;
}

int gh_gemm_set_library_rows( uint64_t rows )
{
  g_library_rows = rows;
  return GH_OK;
}

uint64_t gh_gemm_library_rows( void ) { return g_library_rows; }

int gh_matmul_fuses_many_rows( uint64_t s, uint64_t r, uint64_t b, gh_dtype dt )
{
  static const char aligned[16] __attribute__( ( aligned( 16 ) ) ) = { 0 };
  return gemm_tile_epilogue_applicable( s, r, b, dt, aligned, aligned, aligned )
             || ( r % 8 == 0 && gemm_token_split( s, r, b, dt, aligned, aligned, aligned ) != 0 )
           ? 1
           : 0;
}

int gh_matmul_qkv_fuses_many_rows( uint64_t s, uint32_t n_kv_heads, uint32_t gqa_size, uint32_t head_size, uint64_t b, gh_dtype dt )
{
  static const char aligned[16] __attribute__( ( aligned( 16 ) ) ) = { 0 };
  QkvRows rows;
  rows.kv_dim = n_kv_heads * head_size;
  rows.dim = rows.kv_dim * gqa_size;
  rows.head_size = head_size;
  if ( gemm_library_wanted( s, rows.dim, b, dt, aligned, aligned, aligned ) || gemm_library_wanted( s, 2ull * rows.kv_dim, b, dt, aligned, aligned, aligned ) ) {
    return 0;
  }
  return gemm_tile_qkv_applicable( s, b, dt, aligned, aligned, aligned, rows )
             || ( dt == GH_F16 && gemm_tile256_qkv_fits( rows ) && gemm_token_split( s, rows.dim + 2ull * rows.kv_dim, b, dt, aligned, aligned, aligned ) != 0 )
           ? 1
           : 0;
}

int gh_gemm_stream_plan( uint64_t s, uint64_t r, uint64_t b, uint32_t* splits, uint32_t* k_per_split, uint32_t* rows_per_workgroup )
{
  GH_REQUIRE( splits && k_per_split && rows_per_workgroup, "gh_gemm_stream_plan: NULL output" );
  GH_REQUIRE( s >= 256 && s % 256 == 0 && r > 0 && b > 0, "gh_gemm_stream_plan: the streaming kernel takes s %% 256 == 0, r > 0, b > 0" );
  gemm_stream_plan( s, r, b, splits, k_per_split, rows_per_workgroup );
  return GH_OK;
}

int gh_gemm_ring_plan( uint64_t s, uint64_t r, uint64_t b, int gated, uint32_t* plan )
{
  static const char aligned[16] __attribute__( ( aligned( 16 ) ) ) = { 0 };
  GH_REQUIRE( plan != nullptr, "gh_gemm_ring_plan: NULL output" );
  GH_REQUIRE( s > 0 && r > 0 && b > 0 && gemm_ring_applicable( s, gated ? 2 * r : r, b, aligned, aligned, aligned ) && ( !gated || r % 4 == 0 ),
              "gh_gemm_ring_plan: the ring kernel takes s %% 8 == 0 up to 2^21, r > 0 (a multiple of 4 with the gate), b > 0" );
  return gemm_ring_cut( s, r, b, gated != 0, plan );
}

int gh_matmul_pair( void* xout_a, void* xout_b, const void* x, const void* w, uint64_t s, uint64_t r_a, uint64_t r_b, uint64_t b, gh_dtype dt,
                    gh_stream stream )
{
  if ( int rc = ensure_init() ) {
    return rc;
  }
  if ( b == 0 ) {
    return GH_OK;
  }
  GH_REQUIRE( xout_a && xout_b && x && w, "gh_matmul_pair: NULL pointer" );
  GH_REQUIRE( is_half_type( dt ) || dt == GH_F32, "gh_matmul_pair: unsupported dtype %d", (int)dt );
  const uint64_t elem = dtype_size( dt );
  const uint64_t r = r_a + r_b;
  GH_REQUIRE( s > 0 && s <= 0x7fffffffull && r <= 0x7fffffffull && b <= 0x7fffffffull, "gh_matmul_pair: bad shape" );
  if ( r_a > 0 && r_b > 0 && gemm_library_wanted( s, r_a, b, dt, x, w, xout_a ) && gemm_library_wanted( s, r_b, b, dt, x, w, xout_b ) ) {
    if ( int rc = gh_matmul( xout_a, x, w, s, r_a, b, dt, stream ) ) { // the library's kernels cut their work finer than whole tiles
      return rc;
    }
    return gh_matmul( xout_b, x, static_cast<const char*>( w ) + r_a * s * elem, s, r_b, b, dt, stream );
  }
  // many rows: one launch of the large tile kernel whose work-groups store to the matrix their rows belong to, so that the two
  // products fill their rounds together (a product of 2048 rows alone leaves most of the chip idle)
  if ( is_half_type( dt ) && g_force_kernel == 0 && r_a > 0 && r_b > 0 && r_a % 8 == 0 && r_b % 8 == 0 && gemm_tile256_takes( s, b, x, w, xout_a )
       && ( reinterpret_cast<uintptr_t>( xout_b ) & 15u ) == 0 ) {
    if ( const uint64_t b1 = gemm_token_split( s, r, b, dt, x, w, xout_a ) ) {
      if ( ( b1 * r_a * elem ) % 16 == 0 && ( b1 * r_b * elem ) % 16 == 0 ) {
        if ( int rc = gh_matmul_pair( xout_a, xout_b, x, w, s, r_a, r_b, b1, dt, stream ) ) {
          return rc;
        }
        return gh_matmul_pair( static_cast<char*>( xout_a ) + b1 * r_a * elem, static_cast<char*>( xout_b ) + b1 * r_b * elem,
                               static_cast<const char*>( x ) + b1 * s * elem, w, s, r_a, r_b, b - b1, dt, stream );
      }
    }
    if ( tile256_wanted( s, r, b, x, w, xout_a ) ) {
      return with_half_type( dt, [&]( auto* e ) {
        using E = std::remove_pointer_t<decltype( e )>;
        return gemm_tile256_launch<E>( static_cast<E*>( xout_a ), nullptr, static_cast<const E*>( x ), static_cast<const E*>( w ), s, r, b, 0, as_stream( stream ),
                                       1, 0, static_cast<E*>( xout_b ), r_a );
      } );
    }
  }
  if ( int rc = gh_matmul( xout_a, x, w, s, r_a, b, dt, stream ) ) {
    return rc;
  }
  return gh_matmul( xout_b, x, static_cast<const char*>( w ) + r_a * s * elem, s, r_b, b, dt, stream );
}

int gh_matmul( void* xout, const void* x, const void* w, uint64_t s, uint64_t r, uint64_t b, gh_dtype dt, gh_stream stream )
{
  if ( int rc = ensure_init() ) {
    return rc;
  }
  if ( b == 0 || r == 0 ) {
    return GH_OK;
  }
  GH_REQUIRE( xout && x && w, "gh_matmul: NULL pointer" );
  GH_REQUIRE( s > 0 && s <= 0x7fffffffull && r <= 0x7fffffffull && b <= 0x7fffffffull, "gh_matmul: bad shape" );
  hipStream_t st = as_stream( stream );
  if ( gemm_library_wanted( s, r, b, dt, x, w, xout ) ) { // a plain product of many rows
    bool done = false;
    if ( int rc = gemm_library( xout, x, w, s, r, b, st, &done ) ) {
      return rc;
    }
    if ( done ) {
      return GH_OK;
    }
  }
  if ( const uint64_t b1 = gemm_token_split( s, r, b, dt, x, w, xout ) ) { // two products along the tokens
    const uint64_t elem = 2;
    if ( int rc = gh_matmul( xout, x, w, s, r, b1, dt, stream ) ) {
      return rc;
    }
    return gh_matmul( static_cast<char*>( xout ) + b1 * r * elem, static_cast<const char*>( x ) + b1 * s * elem, w, s, r, b - b1, dt, stream );
  }
  float* partial = nullptr;
  uint32_t splits = 0;
  if ( int rc = gemm_partials( xout, x, w, s, r, b, dt, st, false, &partial, &splits ) ) {
    return rc;
  }
  if ( splits > 0 ) { // only the 16-bit kernels leave partials when not asked to
    const uint64_t n = b * r;
    const unsigned blocks = (unsigned)std::min<uint64_t>( ( n + 255 ) / 256, 4096 );
    return with_half_type( dt, [&]( auto* e ) -> int {
      using E = std::remove_pointer_t<decltype( e )>;
      gemm_reduce_kernel<E><<<blocks, 256, 0, st>>>( static_cast<E*>( xout ), partial, n, splits );
      GH_LAUNCH_CHECK();
      return GH_OK;
    } );
  }
  return GH_OK;
}

} // extern "C"
