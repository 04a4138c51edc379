// Attention over a sliding window with kept first tokens and a bias by distance (storage type bf16 or fp32, sizes at run time).
//
//   position i sees j <= i with i - j < window or j < keep_first;  score = (q . k) * scale + bias[h][min(i - j, n_dist - 1)]
//
// cache row   [K of every kv head | V of every kv head], each head padded with zeros to a multiple of 8 elements, so that any head size
//             is read in 16-byte (bf16) or 32-byte (fp32) pieces.  Where values are keys (SHARED) a head is there once, as projected: it
//             is read once, is the value, and its score takes 1 / rms of the key as a factor, so no second form of a key exists anywhere.
// keys        a query's visible keys are numbered 0 .. count - 1: first the kept ones in front of the window, then the window
// rows kernel work-group = 4 waves on one (token, kv head, block of query heads, split of the keys); 16 lanes hold one key, eight
//             elements a lane, so a wave takes four keys at a time; every 16-lane group keeps its own running maximum and sum for
//             each of its query heads and they meet once, at the end.  Scores, weights and sums are fp32.
#include "gh_product.h"
#include "gh_window.h"

#include <algorithm>
#include <type_traits>

namespace gh {
namespace {

// cache rows are reached through pointers out of a table: the cast names the address space, so that no flat loads are used
typedef uint32_t u32x4_t __attribute__( ( ext_vector_type( 4 ) ) );
typedef const u32x4_t __attribute__( ( address_space( 1 ) ) ) global_u32x4_t;

// where a row's heads go: heads * vdim columns, rows `stride` elements apart; a factor for each head's output, or NULL
template<typename E>
struct WindowOut
{
  E* out;
  uint64_t stride;
  const float* gates;
  uint32_t heads;
  __device__ __forceinline__ float gate( uint64_t row, uint32_t head ) const { return gates != nullptr ? gates[row * heads + head] : 1.0f; }
};

// ---- q / k norm over the whole projection, cache append ------------------------------------------
// work-group = one token's q, its k or its v (blockIdx.y): columns of the product, normed where there is a norm, to padded heads
struct AppendPart
{
  uint32_t first, cols, dim, pad; // columns of the product; head size and its padded form
  const void* norm;               // (cols) or NULL
};

template<typename E>
__device__ __forceinline__ E* append_target( E* q_out, const WindowRows& wr, const WindowShape& s, uint64_t row )
{
  const uint32_t ctx = (uint32_t)( row / wr.n_tokens ), tok = (uint32_t)( row % wr.n_tokens );
  uint8_t* base = static_cast<uint8_t*>( wr.rows[ctx] );
  if ( base == nullptr ) {
    return nullptr;
  }
  if ( blockIdx.y == 0 ) {
    return q_out + row * s.heads * s.dpad;
  }
  E* cache = reinterpret_cast<E*>( base + wr.offset ) + (uint64_t)( wr.start_pos[ctx] + tok ) * s.row_elems();
  return cache + ( blockIdx.y == 1 ? 0 : s.k_elems() );
}

__device__ __forceinline__ float append_row_sum( float v, float* smem )
{
  v = wave_sum( v );
  if ( ( threadIdx.x & 63 ) == 0 ) {
    smem[threadIdx.x >> 6] = v;
  }
  __syncthreads();
  float total = 0.0f;
  for ( uint32_t w = 0; w < blockDim.x / WAVE; w++ ) {
    total += smem[w];
  }
  return total;
}

// head size, product columns and tables in groups of four; a thread owns NV groups, kept in registers across the norm
template<typename E, typename View, int NV>
__global__ __launch_bounds__( 1024 ) void window_append4_kernel( E* __restrict__ q_out, View y, const E* __restrict__ bias, AppendPart pq, AppendPart pk, AppendPart pv,
                                                                 WindowRows wr, WindowShape s, float eps )
{
  __shared__ float smem[16];
  const uint64_t row = blockIdx.x;
  E* dst = append_target( q_out, wr, s, row );
  if ( dst == nullptr ) {
    return;
  }
  const AppendPart p = blockIdx.y == 0 ? pq : blockIdx.y == 1 ? pk : pv;
  const E* norm = static_cast<const E*>( p.norm );
  float4 v[NV], w[NV];
  float ss = 0.0f;
#pragma unroll
  for ( int g = 0; g < NV; g++ ) {
    const uint32_t c = ( g * blockDim.x + threadIdx.x ) * 4, at = c < p.cols ? c : 0;
    v[g] = y.at4( row, p.first + at );
    w[g] = norm != nullptr ? ProductView<E>::load4( norm + at ) : make_float4( 1.0f, 1.0f, 1.0f, 1.0f );
    if ( bias != nullptr ) {
      const float4 b = ProductView<E>::load4( bias + p.first + at );
      v[g] = make_float4( v[g].x + b.x, v[g].y + b.y, v[g].z + b.z, v[g].w + b.w );
    }
    ss += c < p.cols ? v[g].x * v[g].x + v[g].y * v[g].y + v[g].z * v[g].z + v[g].w * v[g].w : 0.0f;
  }
  const float inv = norm != nullptr ? 1.0f / sqrtf( append_row_sum( ss, smem ) / (float)p.cols + eps ) : 1.0f;
#pragma unroll
  for ( int g = 0; g < NV; g++ ) {
    const uint32_t c = ( g * blockDim.x + threadIdx.x ) * 4;
    if ( c >= p.cols ) {
      continue;
    }
    union
    {
      E e[4];
      uint2 half;
      uint4 full;
    } o;
    o.e[0] = from_f32<E>( v[g].x * inv * w[g].x );
    o.e[1] = from_f32<E>( v[g].y * inv * w[g].y );
    o.e[2] = from_f32<E>( v[g].z * inv * w[g].z );
    o.e[3] = from_f32<E>( v[g].w * inv * w[g].w );
    // (without padding the columns are where they belong already, and the divisions can be saved)
    const bool padded = p.pad != p.dim;
    const uint32_t h = padded ? c / p.dim : 0, e = c - h * p.dim;
    E* at = dst + (uint64_t)h * p.pad + e;
    if constexpr ( sizeof( E ) == 2 ) {
      *reinterpret_cast<uint2*>( at ) = o.half;
    } else {
      *reinterpret_cast<uint4*>( at ) = o.full;
    }
    if ( padded && e + 4 == p.dim ) {
      for ( uint32_t z = p.dim; z < p.pad; z++ ) {
        dst[(uint64_t)h * p.pad + z] = from_f32<E>( 0.0f );
      }
    }
  }
}

// prompts (bias and both norms present): work-group = a token's q, k and v together, the columns of the product in one run; all loads go out
// together and both sums meet at one barrier
template<typename E, typename View, int NV>
__global__ __launch_bounds__( 1024 ) void window_append_row_kernel( E* __restrict__ q_out, View y, const E* __restrict__ bias, AppendPart pq, AppendPart pk, AppendPart pv,
                                                                    WindowRows wr, WindowShape s, float eps )
{
  __shared__ float q_sums[16], k_sums[16];
  const uint64_t row = blockIdx.x;
  const uint32_t ctx = (uint32_t)( row / wr.n_tokens ), tok = (uint32_t)( row % wr.n_tokens );
  uint8_t* base = static_cast<uint8_t*>( wr.rows[ctx] );
  if ( base == nullptr ) {
    return;
  }
  const uint32_t cols = pv.first + pv.cols;
  const E *q_norm = static_cast<const E*>( pq.norm ), *k_norm = static_cast<const E*>( pk.norm );
  float4 v[NV], w[NV];
  float qq = 0.0f, kk = 0.0f;
#pragma unroll
  for ( int g = 0; g < NV; g++ ) {
    const uint32_t c = ( g * blockDim.x + threadIdx.x ) * 4, at = c < cols ? c : 0;
    v[g] = y.at4( row, at );
    const bool is_q = at < pk.first;
    w[g] = ProductView<E>::load4( is_q ? q_norm + at : k_norm + ( at < pv.first ? at - pk.first : 0 ) ); // (v: not used)
    const float4 b = ProductView<E>::load4( bias + at );
    v[g] = make_float4( v[g].x + b.x, v[g].y + b.y, v[g].z + b.z, v[g].w + b.w );
    const float sum = c < pv.first ? v[g].x * v[g].x + v[g].y * v[g].y + v[g].z * v[g].z + v[g].w * v[g].w : 0.0f;
    qq += is_q ? sum : 0.0f;
    kk += is_q ? 0.0f : sum;
  }
  qq = wave_sum( qq );
  kk = wave_sum( kk );
  if ( ( threadIdx.x & 63 ) == 0 ) {
    q_sums[threadIdx.x >> 6] = qq;
    k_sums[threadIdx.x >> 6] = kk;
  }
  __syncthreads();
  qq = kk = 0.0f;
  for ( uint32_t i = 0; i < blockDim.x / WAVE; i++ ) {
    qq += q_sums[i];
    kk += k_sums[i];
  }
  const float q_inv = 1.0f / sqrtf( qq / (float)pq.cols + eps );
  const float k_inv = 1.0f / sqrtf( kk / (float)pk.cols + eps );
  E* q_dst = q_out + row * s.heads * s.dpad;
  E* k_dst = reinterpret_cast<E*>( base + wr.offset ) + (uint64_t)( wr.start_pos[ctx] + tok ) * s.row_elems();
  E* v_dst = k_dst + s.k_elems();
#pragma unroll
  for ( int g = 0; g < NV; g++ ) {
    const uint32_t c = ( g * blockDim.x + threadIdx.x ) * 4;
    if ( c >= cols ) {
      continue;
    }
    const bool is_q = c < pk.first, is_v = c >= pv.first;
    const float inv = is_q ? q_inv : k_inv;
    const uint32_t local = c - ( is_q ? 0 : is_v ? pv.first : pk.first );
    const uint32_t dim = is_v ? pv.dim : pq.dim, pad = is_v ? pv.pad : pq.pad;
    union
    {
      E e[4];
      uint2 half;
      uint4 full;
    } o;
    o.e[0] = from_f32<E>( is_v ? v[g].x : v[g].x * inv * w[g].x );
    o.e[1] = from_f32<E>( is_v ? v[g].y : v[g].y * inv * w[g].y );
    o.e[2] = from_f32<E>( is_v ? v[g].z : v[g].z * inv * w[g].z );
    o.e[3] = from_f32<E>( is_v ? v[g].w : v[g].w * inv * w[g].w );
    const uint32_t h = pad != dim ? local / dim : 0, e = local - h * dim;
    E* at = ( is_q ? q_dst : is_v ? v_dst : k_dst ) + (uint64_t)h * pad + e;
    if constexpr ( sizeof( E ) == 2 ) {
      *reinterpret_cast<uint2*>( at ) = o.half;
    } else {
      *reinterpret_cast<uint4*>( at ) = o.full;
    }
    if ( pad != dim && e + 4 == dim ) {
      for ( uint32_t z = dim; z < pad; z++ ) {
        at[z - e] = from_f32<E>( 0.0f );
      }
    }
  }
}

// Many tokens of long rows, bf16 in one plane: 16 bytes a lane, 4 V columns a group, and a work-group keeps the tables in registers over its tokens, every gridDim.x-th,
// and asks for the next token's columns before it reduces this one's, so that reads pass while stores do.  Bound by memory: 403 MB at 8192 tokens of 3 x 4096 columns,
// 112 us with a work-group for each, 84 so (4.8 TB/s; 87 in a prefill; 82 without the sums' way through LDS, which keeps the order and so the bits of that kernel); 8 bytes a lane and
// tokens in turn 101.
__global__ __launch_bounds__( 1024 ) __attribute__( ( amdgpu_waves_per_eu( 6, 8 ) ) ) void window_append_rows_kernel( __bf16* __restrict__ q_out, ProductView<__bf16> y, const __bf16* __restrict__ bias,
                                                                    AppendPart pq, AppendPart pk, AppendPart pv, WindowRows wr, WindowShape s, float eps, uint32_t rows )
{
  constexpr int NV = 2; // groups of eight columns a thread
  extern __shared__ float fours_sums[]; // of squares, two a group
  __shared__ float q_sums[16], k_sums[16];
  const uint32_t cols = pv.first + pv.cols;
  const __bf16 *q_norm = static_cast<const __bf16*>( pq.norm ), *k_norm = static_cast<const __bf16*>( pk.norm );
  auto run_at = []( const __bf16* p ) __attribute__( ( always_inline ) ) { return *reinterpret_cast<const uint4*>( p ); };
  auto wide = []( const uint4& run, int e ) __attribute__( ( always_inline ) ) { return to_f32( reinterpret_cast<const __bf16*>( &run )[e] ); };
  auto read = [&]( uint32_t c ) __attribute__( ( always_inline ) ) { return c < cols ? c : 0; }; // past the row's end: its first ones
  uint4 ahead[NV], w[NV], add[NV];
  uint32_t col[NV];
#pragma unroll
  for ( int g = 0; g < NV; g++ ) {
    col[g] = ( g * blockDim.x + threadIdx.x ) * 8;
    const uint32_t at = read( col[g] );
    ahead[g] = run_at( y.data + (uint64_t)blockIdx.x * y.stride + at );
    w[g] = run_at( at < pk.first ? q_norm + at : k_norm + ( at < pv.first ? at - pk.first : 0 ) ); // (v: not used)
    add[g] = run_at( bias + at );
  }
  for ( uint32_t row = blockIdx.x; row < rows; row += gridDim.x ) {
    const uint32_t ctx = row / wr.n_tokens, tok = row % wr.n_tokens;
    uint8_t* const base = static_cast<uint8_t*>( wr.rows[ctx] );
    const uint32_t pos = wr.start_pos[ctx] + tok;
    const uint32_t next = min( row + gridDim.x, rows - 1 );
    float v[NV][8];
#pragma unroll
    for ( int g = 0; g < NV; g++ ) { // (nothing that follows from a group's columns is kept from token to token, and the tables as they are, not as the floats that they make)
      asm volatile( "" : "+v"( col[g] ) );
      asm volatile( "" : "+v"( w[g].x ), "+v"( w[g].y ), "+v"( w[g].z ), "+v"( w[g].w ), "+v"( add[g].x ), "+v"( add[g].y ), "+v"( add[g].z ), "+v"( add[g].w ) );
#pragma unroll
      for ( int e = 0; e < 8; e++ ) {
        v[g][e] = wide( ahead[g], e ) + wide( add[g], e );
      }
    }
#pragma unroll
    for ( int g = 0; g < NV; g++ ) {
      ahead[g] = run_at( y.data + (uint64_t)next * y.stride + read( col[g] ) );
    }
#pragma unroll
    for ( int g = 0; g < NV; g++ ) {
#pragma unroll
      for ( int e = 0; e < 8; e += 4 ) {
        const float sum = v[g][e] * v[g][e] + v[g][e + 1] * v[g][e + 1] + v[g][e + 2] * v[g][e + 2] + v[g][e + 3] * v[g][e + 3];
        fours_sums[( col[g] + e ) / 4] = col[g] < pv.first ? sum : 0.0f;
      }
    }
    __syncthreads();
    float qq = 0.0f, kk = 0.0f;
#pragma unroll
    for ( int g = 0; g < 2 * NV; g++ ) { // in the order of a thread with four columns at a time
      const uint32_t f = g * blockDim.x + threadIdx.x;
      const float sum = fours_sums[f];
      qq += 4 * f < pk.first ? sum : 0.0f;
      kk += 4 * f < pk.first ? 0.0f : sum;
    }
    qq = wave_sum( qq );
    kk = wave_sum( kk );
    if ( ( threadIdx.x & 63 ) == 0 ) {
      q_sums[threadIdx.x >> 6] = qq;
      k_sums[threadIdx.x >> 6] = kk;
    }
    __syncthreads(); // (and everyone has read the sums of fours; those of the waves are written again behind the next token's first barrier)
    qq = kk = 0.0f;
    for ( uint32_t i = 0; i < blockDim.x / WAVE; i++ ) {
      qq += q_sums[i];
      kk += k_sums[i];
    }
    if ( base == nullptr ) {
      continue;
    }
    const float q_inv = 1.0f / sqrtf( qq / (float)pq.cols + eps );
    const float k_inv = 1.0f / sqrtf( kk / (float)pk.cols + eps );
    __bf16* q_dst = q_out + (uint64_t)row * s.heads * s.dpad;
    __bf16* k_dst = reinterpret_cast<__bf16*>( base + wr.offset ) + (uint64_t)pos * s.row_elems();
    __bf16* v_dst = k_dst + s.k_elems();
#pragma unroll
    for ( int g = 0; g < NV; g++ ) {
      const uint32_t c = col[g];
      if ( c >= cols ) {
        continue;
      }
      const bool is_q = c < pk.first, is_v = c >= pv.first;
      const float inv = is_q ? q_inv : k_inv;
      union
      {
        __bf16 e[8];
        uint4 run;
      } o;
#pragma unroll
      for ( int e = 0; e < 8; e++ ) {
        o.e[e] = from_f32<__bf16>( is_v ? v[g][e] : v[g][e] * inv * wide( w[g], e ) );
      }
      // (heads are not padded, as they are a multiple of eight)
      *reinterpret_cast<uint4*>( ( is_q ? q_dst : is_v ? v_dst : k_dst ) + ( c - ( is_q ? 0 : is_v ? pv.first : pk.first ) ) ) = o.run;
    }
  }
}

// any sizes: the columns of the part pass through LDS
template<typename E, typename View>
__global__ __launch_bounds__( 256 ) void window_append_any_kernel( E* __restrict__ q_out, View y, const E* __restrict__ bias, AppendPart pq, AppendPart pk, AppendPart pv,
                                                                   WindowRows wr, WindowShape s, float eps )
{
  extern __shared__ float vals[];
  __shared__ float smem[4];
  const uint64_t row = blockIdx.x;
  E* dst = append_target( q_out, wr, s, row );
  if ( dst == nullptr ) {
    return;
  }
  const AppendPart p = blockIdx.y == 0 ? pq : blockIdx.y == 1 ? pk : pv;
  const E* norm = static_cast<const E*>( p.norm );
  float ss = 0.0f;
  for ( uint32_t c = threadIdx.x; c < p.cols; c += blockDim.x ) {
    const float v = y.at( row, p.first + c ) + ( bias != nullptr ? to_f32( bias[p.first + c] ) : 0.0f );
    vals[c] = v;
    ss += v * v;
  }
  const float total = append_row_sum( ss, smem ); // (also the barrier in front of the reads below)
  const float inv = norm != nullptr ? 1.0f / sqrtf( total / (float)p.cols + eps ) : 1.0f;
  for ( uint32_t c = threadIdx.x; c < p.cols / p.dim * p.pad; c += blockDim.x ) {
    const uint32_t h = c / p.pad, e = c % p.pad, src = h * p.dim + e;
    dst[c] = from_f32<E>( e < p.dim ? vals[src] * inv * ( norm != nullptr ? to_f32( norm[src] ) : 1.0f ) : 0.0f );
  }
}

template<typename E, typename View>
int launch_append( E* q, const View& y, const E* bias, const void* q_norm, const void* k_norm, float eps, const WindowRows& wr, const WindowShape& s, uint64_t rows,
                   hipStream_t st )
{
  const uint32_t nq = s.heads * s.dim, nk = s.kv_heads * s.dim, nv = s.kv_heads * s.vdim;
  const AppendPart pq { 0, nq, s.dim, s.dpad, q_norm }, pk { nq, nk, s.dim, s.dpad, k_norm }, pv { nq + nk, nv, s.vdim, s.vpad, nullptr };
  const uint32_t most = std::max( { nq, nk, nv } );
  const dim3 grid( (unsigned)rows, 3 );
  const uintptr_t tables = reinterpret_cast<uintptr_t>( bias ) | reinterpret_cast<uintptr_t>( q_norm ) | reinterpret_cast<uintptr_t>( k_norm );
  if ( s.dim % 4 == 0 && s.vdim % 4 == 0 && y.stride % 4 == 0 && ( tables & 15u ) == 0 && most <= 32768 ) {
    if ( const uint32_t all = ( nq + nk + nv ) / 4; rows >= 1024 && all <= 4096 && bias != nullptr && q_norm != nullptr && k_norm != nullptr ) {
      const uint32_t threads = std::max<uint32_t>( 64, ( ( all + 3 ) / 4 + 63 ) / 64 * 64 );
      bool in_turn = false;
      if constexpr ( std::is_same_v<View, ProductView<__bf16>> ) { // one plane
        // Work-groups that run at a time (six waves a SIMD), each as many tokens as the others: at least six, and long rows.  One token a work-group and several, the call:
        // 3 x 4096 columns at 2048, 3072 and 8192 tokens 44.2, 57.1 and 172 us and 44.2, 56.7 and 146; 10240 at 3072 and 8192 56.5 and 164, 55.9 and 141; 9216 at 8192
        // 108.8 and 110; 6144 at 4096 and 32768 47.2 and 321, 49.9 and 347.
        const uint64_t resident = (uint64_t)cu_count() * std::max( 1u, 1536 / threads ), each = ( rows + resident - 1 ) / resident;
        const uintptr_t runs = reinterpret_cast<uintptr_t>( y.data ) | reinterpret_cast<uintptr_t>( q );
        in_turn = all >= 2560 && each >= 6 && s.dim % 8 == 0 && s.vdim % 8 == 0 && y.stride % 8 == 0 && ( runs & 15u ) == 0;
        if ( in_turn ) {
          window_append_rows_kernel<<<(unsigned)( ( rows + each - 1 ) / each ), threads, 4 * threads * sizeof( float ), st>>>( q, y, bias, pq, pk, pv, wr, s, eps, (uint32_t)rows );
        }
      }
      if ( !in_turn ) {
        window_append_row_kernel<E, View, 4><<<(unsigned)rows, threads, 0, st>>>( q, y, bias, pq, pk, pv, wr, s, eps );
      }
      GH_LAUNCH_CHECK();
      return GH_OK;
    }
    const uint32_t groups = most / 4;
    const uint32_t want = rows >= 1024 ? ( groups + 3 ) / 4 : groups;
    const uint32_t threads = std::min<uint32_t>( 1024, std::max<uint32_t>( 64, ( want + 63 ) / 64 * 64 ) );
    const uint32_t per = ( groups + threads - 1 ) / threads;
    if ( per <= 1 ) {
      window_append4_kernel<E, View, 1><<<grid, threads, 0, st>>>( q, y, bias, pq, pk, pv, wr, s, eps );
    } else if ( per <= 2 ) {
      window_append4_kernel<E, View, 2><<<grid, threads, 0, st>>>( q, y, bias, pq, pk, pv, wr, s, eps );
    } else if ( per <= 4 ) {
      window_append4_kernel<E, View, 4><<<grid, threads, 0, st>>>( q, y, bias, pq, pk, pv, wr, s, eps );
    } else {
      window_append4_kernel<E, View, 8><<<grid, threads, 0, st>>>( q, y, bias, pq, pk, pv, wr, s, eps );
    }
  } else {
    GH_REQUIRE( most <= 15 * 1024, "gh_matmul_window_append: the heads of a token do not fit in LDS" );
    window_append_any_kernel<E, View><<<grid, 256, most * sizeof( float ), st>>>( q, y, bias, pq, pk, pv, wr, s, eps );
  }
  GH_LAUNCH_CHECK();
  return GH_OK;
}

// ---- visible keys ------------------------------------------------------------------------------
struct Visible
{
  uint32_t kept, first, count; // kept keys in front of the window, first key of the window, all of them
  __device__ __forceinline__ uint32_t key( uint32_t idx ) const { return idx < kept ? idx : first + ( idx - kept ); }
};
__device__ __forceinline__ Visible visible_keys( uint32_t pos, const WindowShape& s )
{
  Visible v;
  v.first = pos + 1 > s.window ? pos + 1 - s.window : 0;
  v.kept = min( s.keep_first, v.first );
  v.count = v.kept + ( pos + 1 - v.first );
  return v;
}

template<typename E>
__device__ __forceinline__ void load8( float out[8], const E* p )
{
  if constexpr ( sizeof( E ) == 2 ) {
    union
    {
      uint4 raw;
      E e[8];
    } u;
    u.raw = __builtin_bit_cast( uint4, *(global_u32x4_t*)( p ) );
#pragma unroll
    for ( int i = 0; i < 8; i++ ) {
      out[i] = to_f32( u.e[i] );
    }
  } else {
    const float4 a = __builtin_bit_cast( float4, *(global_u32x4_t*)( p ) ), b = __builtin_bit_cast( float4, *(global_u32x4_t*)( p + 4 ) );
    out[0] = a.x, out[1] = a.y, out[2] = a.z, out[3] = a.w, out[4] = b.x, out[5] = b.y, out[6] = b.z, out[7] = b.w;
  }
}

constexpr float NO_KEY = -1e30f; // running maximum before the first key: exp(NO_KEY - anything real) is 0

// partial result of one split of one (row, head): vpad weighted sums, then the sum of the weights and the maximum
__host__ __device__ inline uint64_t partial_stride( const WindowShape& s ) { return s.vpad + 2; }

// The results of a work-group's NW waves for the query heads h0 .. h0 + nh - 1 of a row, wave w's for head h at
// lds[(w * hq + h) * (vpad + 2)]: added up and stored, as the output or as the partial result of a split.
template<typename E, int NW, int THREADS = 64 * NW>
__device__ __forceinline__ void finish_split( const WindowOut<E>& out, float* partial, const float* lds, uint32_t hq, uint32_t nh, uint64_t row, uint32_t h0, uint32_t split,
                                              uint32_t splits, const WindowShape& s )
{
  const uint32_t stride = s.vpad + 2;
  for ( uint32_t i = threadIdx.x; i < nh * s.vpad; i += THREADS ) {
    const uint32_t h = i / s.vpad, e = i % s.vpad;
    float m = NO_KEY;
#pragma unroll
    for ( int w = 0; w < NW; w++ ) {
      m = fmaxf( m, lds[( w * hq + h ) * stride + s.vpad + 1] );
    }
    float a = 0.0f, sm = 0.0f;
#pragma unroll
    for ( int w = 0; w < NW; w++ ) {
      const float* src = lds + ( w * hq + h ) * stride;
      const float f = __expf( src[s.vpad + 1] - m );
      a += src[e] * f;
      sm += src[s.vpad] * f;
    }
    if ( splits == 1 ) {
      if ( e < s.vdim ) {
        out.out[row * out.stride + ( h0 + h ) * s.vdim + e] = from_f32<E>( a / sm * out.gate( row, h0 + h ) );
      }
    } else {
      float* dst = partial + ( ( row * s.heads + h0 + h ) * splits + split ) * stride;
      dst[e] = a;
      if ( e == 0 ) {
        dst[s.vpad] = sm;
        dst[s.vpad + 1] = m;
      }
    }
  }
}

// HQ query heads at a time; NC pieces of 128 elements per head (a lane holds 8 of each)
template<typename E, int HQ, int NC, bool SHARED>
__global__ __launch_bounds__( 256 ) void window_rows_kernel( WindowOut<E> out,
                                                             float* __restrict__ partial,
                                                             const E* __restrict__ q,
                                                             const float* __restrict__ bias,
                                                             WindowRows wr,
                                                             WindowShape s,
                                                             uint32_t keys_per_split,
                                                             uint32_t splits )
{
  extern __shared__ float lds[]; // 4 waves x HQ x (vpad + 2)
  const uint32_t head_blocks = ( s.group + HQ - 1 ) / HQ;
  const uint32_t g = blockIdx.y / head_blocks, hb = blockIdx.y % head_blocks;
  const uint64_t row = blockIdx.x;
  const uint32_t split = blockIdx.z;
  const uint32_t ctx = (uint32_t)( row / wr.n_tokens ), tok = (uint32_t)( row % wr.n_tokens );
  const uint8_t* base = static_cast<const uint8_t*>( wr.rows[ctx] );
  if ( base == nullptr ) {
    return;
  }
  const uint32_t pos = wr.start_pos[ctx] + tok;
  const Visible vis = visible_keys( pos, s );
  const uint32_t wave = threadIdx.x >> 6, lane = threadIdx.x & 63, l16 = lane & 15, g4 = lane >> 4;
  const uint32_t h0 = g * s.group + hb * HQ;
  const uint32_t nh = min( (uint32_t)HQ, s.group - hb * HQ );
  const E* cache = reinterpret_cast<const E*>( base + wr.offset );
  const uint32_t k_begin = split * keys_per_split, k_end = min( vis.count, k_begin + keys_per_split );

  float qv[HQ][NC][8], acc[HQ][NC][8], mx[HQ], sum[HQ];
#pragma unroll
  for ( int h = 0; h < HQ; h++ ) {
    mx[h] = NO_KEY;
    sum[h] = 0.0f;
#pragma unroll
    for ( int c = 0; c < NC; c++ ) {
#pragma unroll
      for ( int e = 0; e < 8; e++ ) {
        qv[h][c][e] = 0.0f;
        acc[h][c][e] = 0.0f;
      }
      const uint32_t at = c * 128 + l16 * 8;
      if ( (uint32_t)h < nh && at < s.dpad ) {
        load8( qv[h][c], q + ( row * s.heads + h0 + h ) * s.dpad + at );
      }
    }
  }
  // U keys per 16-lane group and step: all their loads go out before the first is used.  A key past the end reads the step's first again
  // and gets no weight.
  constexpr uint32_t U = HQ * NC >= 4 ? 2 : 4;
  const uint32_t at_k = g * s.dpad, at_v = s.k_elems() + g * s.vpad;
  const float* factors = reinterpret_cast<const float*>( base + wr.factors );
  for ( uint32_t i0 = k_begin + wave * 4 * U; i0 < k_end; i0 += 16 * U ) {
    float kv[U][NC][8], vv[SHARED ? 1 : U][NC][8], factor[U];
    uint32_t dist[U];
    bool live[U];
#pragma unroll
    for ( uint32_t u = 0; u < U; u++ ) {
      const uint32_t idx = i0 + 4 * u + g4;
      live[u] = idx < k_end;
      const uint32_t j = vis.key( live[u] ? idx : i0 );
      dist[u] = min( pos - j, s.n_dist - 1 );
      factor[u] = SHARED ? s.scale * factors[factor_index( j, g, s.kv_heads )] : s.scale;
      const E* row_j = cache + (uint64_t)j * s.row_elems();
#pragma unroll
      for ( int c = 0; c < NC; c++ ) {
        const uint32_t at = c * 128 + l16 * 8;
#pragma unroll
        for ( int e = 0; e < 8; e++ ) {
          kv[u][c][e] = 0.0f;
        }
        if ( at < s.dpad ) {
          load8( kv[u][c], row_j + at_k + at );
        }
        if constexpr ( !SHARED ) {
#pragma unroll
          for ( int e = 0; e < 8; e++ ) {
            vv[u][c][e] = 0.0f;
          }
          if ( at < s.vpad ) {
            load8( vv[u][c], row_j + at_v + at );
          }
        }
      }
    }
#pragma unroll
    for ( int h = 0; h < HQ; h++ ) {
      float score[U];
      float m_new = mx[h];
#pragma unroll
      for ( uint32_t u = 0; u < U; u++ ) {
        float dot = 0.0f;
#pragma unroll
        for ( int c = 0; c < NC; c++ ) {
#pragma unroll
          for ( int e = 0; e < 8; e++ ) {
            dot += qv[h][c][e] * kv[u][c][e];
          }
        }
        const float b = bias != nullptr && (uint32_t)h < nh ? bias[(uint64_t)( h0 + h ) * s.n_dist + dist[u]] : 0.0f;
        score[u] = live[u] ? row16_sum( dot ) * factor[u] + b : NO_KEY;
        m_new = fmaxf( m_new, score[u] );
      }
      const float old = __expf( mx[h] - m_new );
      mx[h] = m_new;
      float p[U], p_sum = 0.0f;
#pragma unroll
      for ( uint32_t u = 0; u < U; u++ ) {
        p[u] = live[u] ? __expf( score[u] - m_new ) : 0.0f;
        p_sum += p[u];
      }
      sum[h] = sum[h] * old + p_sum;
#pragma unroll
      for ( int c = 0; c < NC; c++ ) {
#pragma unroll
        for ( int e = 0; e < 8; e++ ) {
          float a = acc[h][c][e] * old;
#pragma unroll
          for ( uint32_t u = 0; u < U; u++ ) {
            a += p[u] * ( SHARED ? kv[u][c][e] : vv[SHARED ? 0 : u][c][e] );
          }
          acc[h][c][e] = a;
        }
      }
    }
  }
  // the four 16-lane groups of the wave, then the four waves
  const uint32_t stride = s.vpad + 2;
#pragma unroll
  for ( int h = 0; h < HQ; h++ ) {
    float m = fmaxf( mx[h], __shfl_xor( mx[h], 16 ) );
    m = fmaxf( m, __shfl_xor( m, 32 ) );
    const float f = __expf( mx[h] - m );
    float sm = sum[h] * f;
    sm += __shfl_xor( sm, 16 );
    sm += __shfl_xor( sm, 32 );
    float* mine = lds + ( wave * HQ + h ) * stride;
#pragma unroll
    for ( int c = 0; c < NC; c++ ) {
      const uint32_t at = c * 128 + l16 * 8;
#pragma unroll
      for ( int e = 0; e < 8; e++ ) {
        float a = acc[h][c][e] * f;
        a += __shfl_xor( a, 16 );
        a += __shfl_xor( a, 32 );
        if ( g4 == 0 && at + e < s.vpad ) {
          mine[at + e] = a;
        }
      }
    }
    if ( lane == 0 ) {
      mine[s.vpad] = sm;
      mine[s.vpad + 1] = m;
    }
  }
  __syncthreads();
  finish_split<E, 4>( out, partial, lds, HQ, nh, row, h0, split, splits, s );
}

// One wave per (row, head): lane k holds maximum and sum of split k (at most 64), and eight splits' values are requested at once (one row of 32 heads, 1025
// keys: 16.5 us with the attention, with a split after the other 18.6).
template<typename E>
__global__ __launch_bounds__( 256 ) void window_merge_kernel( WindowOut<E> out, const float* __restrict__ partial, WindowRows wr, WindowShape s, uint32_t splits,
                                                              uint64_t pairs )
{
  const uint64_t pair = (uint64_t)blockIdx.x * 4 + ( threadIdx.x >> 6 );
  if ( pair >= pairs || wr.rows[pair / s.heads / wr.n_tokens] == nullptr ) {
    return;
  }
  const uint32_t lane = threadIdx.x & 63, stride = s.vpad + 2;
  const float* src = partial + pair * splits * stride;
  const float* own = src + min( lane, splits - 1 ) * stride + s.vpad;
  const float own_sum = own[0], own_max = own[1];
  const uint64_t row = pair / s.heads;
  const uint32_t head = (uint32_t)( pair % s.heads );
  const float gate = out.gate( row, head );
  const float m = wave_max( own_max ); // (the last split's repeated in the lanes beyond)
  const float weight = lane < splits ? __expf( own_max - m ) : 0.0f;
  const float sm = wave_sum( lane < splits ? own_sum * weight : 0.0f );
  // No lane leaves before the end: each holds a split's weight, and what makes it may move into a loop that only the lanes with a value enter.
  for ( uint32_t e0 = 0; e0 < s.vdim; e0 += 64 ) {
    const uint32_t e = min( e0 + lane, s.vdim - 1 );
    float a = 0.0f;
    for ( uint32_t k0 = 0; k0 < splits; k0 += 8 ) {
      float v[8];
#pragma unroll
      for ( uint32_t u = 0; u < 8; u++ ) { // a split past the last reads the last again and is not added
        v[u] = src[min( k0 + u, splits - 1 ) * stride + e];
      }
#pragma unroll
      for ( uint32_t u = 0; u < 8; u++ ) {
        a += k0 + u < splits ? v[u] * lane_value( weight, min( k0 + u, splits - 1 ) ) : 0.0f;
      }
    }
    if ( e0 + lane < s.vdim ) {
      out.out[row * out.stride + head * s.vdim + e] = from_f32<E>( a / sm * gate );
    }
  }
}

// ---- many tokens: key tiles on the matrix cores (bf16, head sizes up to 128) -----------------------------------------------------
//
// work-group  4 waves on one (context, kv head), 32 query columns a wave; a column is (token, query head) with the query heads of a group side
//             by side where their number is a power of two, else one query head per work-group
// keys        64 at a time: the tiles of the kept first tokens in front of the window, then those of the window of the work-group's
//             tokens.  A wave leaves out a tile that none of its columns sees, takes no mask for one that all of them see whole, and a
//             constant bias for one farther away than the bias table is long.  Else the table's copy in LDS has entries in front of
//             distance 0 and behind the last, where they fit: a lane reads the biases of its 32 keys with one address and offsets.
// scores^T    K Q^T by v_mfma_f32_32x32x16_bf16 (K out of LDS, Q in registers): a lane holds 32 of the tile's 64 scores of ITS column, the
//             lane 32 further on the others, so maximum and sum stay in the lane but for one exchange
// values      O^T += V^T P^T: the weights are, as they lie, the right operand; V^T comes out of LDS by transposing reads.  The weights
//             are fp32: they enter as two bf16 terms (16 bits of mantissa), their sum is taken in fp32.
// LDS         rows of 256 bytes whatever the head size (the rest is zero), 16-byte chunks XORed with bits of the row; the next tile's
//             rows are in registers while this one is multiplied, and two work-groups share a CU.  Where values are keys both products
//             read one tile: the low four bits of the row, pairs exchanged, keep the plain reads (16 rows, one chunk) and the
//             transposing ones (4 rows, 4 chunks) apart.
// order       the longest work-groups of up to eight pairs of an XCD start first, then those of the next eight.  Those of one pair next to each other leave
//             the last pairs' long ones to the end, 4.9 of 8 waves in flight on average where there are few; those of all pairs at once need all keys at a
//             time, which come out of HBM again for every block once they are more than the Infinity Cache holds.  Heads of 128, us: pair by pair, eight, all:
//             8 x 1024 tokens of window 1024 198, 149, 153; 32 x 1024 of it 783, 642, 775; 16 x 2048 1131, 1020, 1294; 8 x 4096 1970, 1818, 2107; 64 heads, 16 x
//             2048 of window 1024 1884, 1791, 2238; 2 x 8192 1812, 1751, 1755; keys as values 16 x 2048 979, 898, 933.  Groups of 4 to 16 are within 4 %, of 2 and 48 behind.
// rounding    scale and bias are one fused multiplication in every tile, the reference point is taken off behind it.  Both in one for tiles with a constant bias
//             saves 32 of a tile's instructions and no time (8 x 1024 tokens 166 us against 165), and bits differ from one form of tile to the other.
// bound       vector and matrix work of two waves a SIMD, which overlap little.  8 x 1024 tokens, 32 heads of 128, window 1024, 512 distances:
//             221 us -> 200 with fewer vector instructions (702 -> 540 a tile and wave) -> 161 with the order; 4 x 2048 tokens without a
//             bias: 309 -> 239, keys as values 293 -> 222 (calls in a row, their keys in the Infinity Cache; in prefills 182 and, keys as values, 270).  The products run at 0.9 PFLOP/s there, both terms counted.
//             Other priorities for the waves in their products: no change.
constexpr float LOG2E = 1.4426950408889634f;
constexpr float LAZY = 8.0f; // the reference point of a column's exponentials moves when its maximum has grown by 2^LAZY
constexpr uint32_t TILE_KEYS = 64;
constexpr uint32_t GROUP_PAIRS = 8;
constexpr uint32_t BIAS_LDS = 8192; // floats of bias table a work-group can hold
// Entries around a head's table, where they fit: from a wave's 32 tokens to the keys of a tile that touches the table the distances reach 94 before its start and behind its end
constexpr uint32_t BIAS_PAD = 96;
typedef __attribute__( ( address_space( 3 ) ) ) char lds_char;
typedef short v4s __attribute__( ( ext_vector_type( 4 ) ) );
typedef __attribute__( ( address_space( 3 ) ) ) v4s* lds_v4s;
typedef Mfma<__bf16>::x8 bf16x8;

__device__ __forceinline__ uint32_t shared_swizzle( uint32_t row ) { return ( ( row & 3 ) << 2 ) | ( ( row >> 2 ) & 3 ); }

// KS: steps of 16 of the query/key size; VB: blocks of 32 of the value size
template<int KS, int VB, bool SHARED>
__global__ __launch_bounds__( 256, 2 ) void window_tiles_kernel( WindowOut<__bf16> out,
                                                                 const __bf16* __restrict__ q,
                                                                 const float* __restrict__ bias,
                                                                 WindowRows wr,
                                                                 WindowShape s,
                                                                 uint32_t head_cols,  // query heads side by side in the columns
                                                                 uint32_t col_blocks, // work-groups along the tokens of a pair
                                                                 uint32_t n_pairs,    // contexts x kv heads x (query heads of a group / head_cols)
                                                                 uint32_t group_pairs, // pairs of an XCD whose blocks are in one order
                                                                 uint32_t bias_row,   // floats of a head's bias table in LDS; 0: no bias
                                                                 uint32_t bias_pad )  // its entries in front of distance 0 and behind the last one
{
  extern __shared__ uint4 lds16[];
  uint4* s_k = lds16;
  uint4* s_v = SHARED ? s_k : s_k + TILE_KEYS * 16;
  float* s_factor = reinterpret_cast<float*>( s_v + TILE_KEYS * 16 );  // SHARED: of the tile's keys, times scale and log2(e)
  float* s_bias = s_factor + ( SHARED ? TILE_KEYS : 0 );               // (head_cols, bias_row), times log2(e)

  // all column blocks of a pair on one XCD; the longest blocks of a group of pairs first
  const uint32_t xcd = blockIdx.x & 7, slot = blockIdx.x >> 3;
  const uint32_t group = slot / ( group_pairs * col_blocks ), in_group = slot % ( group_pairs * col_blocks );
  const uint32_t pairs = min( group_pairs, ( n_pairs + 7 ) / 8 - group * group_pairs );
  const uint32_t cb = col_blocks - 1 - in_group / pairs;
  const uint32_t pair = ( group * group_pairs + in_group % pairs ) * 8 + xcd;
  if ( pair >= n_pairs ) {
    return;
  }
  const uint32_t per_group = s.group / head_cols;
  const uint32_t ctx = pair / ( s.kv_heads * per_group );
  const uint32_t g = pair / per_group % s.kv_heads;
  const uint32_t h0 = g * s.group + pair % per_group * head_cols;
  const uint8_t* base = static_cast<const uint8_t*>( wr.rows[ctx] );
  if ( base == nullptr ) {
    return;
  }
  const __bf16* cache = reinterpret_cast<const __bf16*>( base + wr.offset );
  const uint32_t start = wr.start_pos[ctx];
  const uint32_t wave = threadIdx.x >> 6, lane = threadIdx.x & 63, r = lane & 31, g2 = lane >> 5;
  const uint32_t tok_wg = cb * ( 128 / head_cols );
  const uint32_t tok_last = min( wr.n_tokens, tok_wg + 128 / head_cols ) - 1;
  const uint32_t colnum = wave * 32 + r;
  const uint32_t tok = tok_wg + colnum / head_cols, hc = colnum % head_cols;
  const bool col_ok = tok < wr.n_tokens;
  const uint32_t pos = start + ( col_ok ? tok : tok_last ); // a column without a query does as the last one and is not stored
  const uint32_t pos_first = start + tok_wg, pos_last = start + tok_last;
  // those of the wave's own columns
  const uint32_t wave_col = __builtin_amdgcn_readfirstlane( wave ) * 32;
  const uint32_t wave_first = start + min( tok_wg + wave_col / head_cols, tok_last ), wave_last = start + min( tok_wg + ( wave_col + 31 ) / head_cols, tok_last );

  if ( bias_row == 0 && threadIdx.x == 0 ) {
    s_bias[0] = 0.0f;
  }
  for ( uint32_t c = 0; c < ( bias_row > 0 ? head_cols : 0 ); c++ ) {
    for ( uint32_t i = threadIdx.x; i < bias_row; i += 256 ) { // distances before 0 as 0, those past the table as its last
      s_bias[c * bias_row + i] = bias[(uint64_t)( h0 + c ) * s.n_dist + min( i - min( i, bias_pad ), s.n_dist - 1 )] * LOG2E;
    }
  }

  bf16x8 qb[KS];
  {
    const __bf16* qp = q + ( ( (uint64_t)ctx * wr.n_tokens + ( col_ok ? tok : tok_last ) ) * s.heads + h0 + hc ) * s.dpad;
#pragma unroll
    for ( int k = 0; k < KS; k++ ) {
      const uint32_t ch = 2 * k + g2;
      u32x4_t v = { 0, 0, 0, 0 };
      if ( ch * 8 < s.dpad ) {
        v = *(global_u32x4_t*)( qp + ch * 8 );
      }
      qb[k] = __builtin_bit_cast( bf16x8, v );
    }
  }

  // tiles: kept keys [0, kept), then [first, pos_last]
  const uint32_t first = pos_first + 1 > s.window ? pos_first + 1 - s.window : 0;
  const uint32_t kept = min( s.keep_first, first );
  const uint32_t kept_tiles = ( kept + TILE_KEYS - 1 ) / TILE_KEYS;
  const uint32_t tiles = kept_tiles + ( pos_last + 1 - first + TILE_KEYS - 1 ) / TILE_KEYS;
  auto tile_at = [&]( uint32_t i ) { return i < kept_tiles ? i * TILE_KEYS : first + ( i - kept_tiles ) * TILE_KEYS; };

  // a thread's four 16-byte pieces of a tile of K and of V: row threadIdx / 16 + 16 i, chunk threadIdx % 16
  const uint32_t ld_chunk = threadIdx.x & 15, ld_row = threadIdx.x >> 4;
  const uint32_t row_bytes = s.row_elems() * sizeof( __bf16 );
  const uint32_t at_k = ( g * s.dpad + ld_chunk * 8 ) * sizeof( __bf16 ), at_v = ( s.k_elems() + g * s.vpad + ld_chunk * 8 ) * sizeof( __bf16 );
  const bool k_chunk = ld_chunk * 8 < s.dpad && ld_chunk < 2 * KS, v_chunk = ld_chunk * 8 < s.vpad && ld_chunk < 4 * VB; // a thread past the head's size keeps its zeros
  u32x4_t rk[4] = {}, rv[SHARED ? 1 : 4] = {};
  const float* factors = reinterpret_cast<const float*>( base + wr.factors );
  float rf = 0.0f;
  auto load = [&]( uint32_t i ) {
    const uint32_t t0 = tile_at( i ), end = i < kept_tiles ? kept : pos_last + 1;
    if ( SHARED && threadIdx.x < TILE_KEYS ) {
      rf = factors[factor_index( min( t0 + threadIdx.x, end - 1 ), g, s.kv_heads )];
    }
    const char* tile = reinterpret_cast<const char*>( cache ) + (uint64_t)t0 * row_bytes;
    auto load_row = [&]( int k, const char* at, uint32_t lane_offset ) __attribute__( ( always_inline ) ) {
      if ( k_chunk ) {
        rk[k] = *(global_u32x4_t*)( at + ( lane_offset + at_k ) );
      }
      if constexpr ( !SHARED ) {
        if ( v_chunk ) {
          rv[k] = *(global_u32x4_t*)( at + ( lane_offset + at_v ) );
        }
      }
    };
    if ( t0 + TILE_KEYS <= end ) { // whole: one address for the wave and the lane's row
#pragma unroll
      for ( int k = 0; k < 4; k++ ) {
        load_row( k, tile + (uint64_t)( 16 * k ) * row_bytes, ld_row * row_bytes );
      }
    } else { // (past the last key that key again: no column sees it there)
#pragma unroll
      for ( int k = 0; k < 4; k++ ) {
        load_row( k, tile, min( ld_row + 16 * k, end - 1 - t0 ) * row_bytes );
      }
    }
  };
  const float scale_log2e = s.scale * LOG2E;
  auto store = [&] {
#pragma unroll
    for ( int k = 0; k < 4; k++ ) {
      const uint32_t row = ld_row + 16 * k;
      s_k[row * 16 + ( ld_chunk ^ ( SHARED ? shared_swizzle( row ) : row & 15 ) )] = __builtin_bit_cast( uint4, rk[k] );
      if constexpr ( !SHARED ) {
        s_v[row * 16 + ( ld_chunk ^ ( 4 * ( row & 3 ) ) )] = __builtin_bit_cast( uint4, rv[k] );
      }
    }
    if ( SHARED && threadIdx.x < TILE_KEYS ) {
      s_factor[threadIdx.x] = rf * scale_log2e;
    }
  };
  const uint32_t tr_e = ( lane & 15 ) >> 2, tr_q = lane & 3, tr_grp = ( lane >> 4 ) & 1;
  const uint32_t v_lane = ( 4 * g2 + tr_e ) * 256 + ( ( ( 2 * tr_grp + ( tr_q >> 1 ) ) ^ ( 4 * tr_e ) ^ ( SHARED ? g2 : 0 ) ) * 16 ) + ( tr_q & 1 ) * 8;

  mfma_f32x16 acc[VB];
#pragma unroll
  for ( int vb = 0; vb < VB; vb++ ) {
#pragma unroll
    for ( int v = 0; v < 16; v++ ) {
      acc[vb][v] = 0.0f;
    }
  }
  float m = NO_KEY, l = 0.0f;
  const float* my_bias = s_bias + hc * bias_row + bias_pad;
  const uint32_t n_dist = bias_row > 0 ? s.n_dist : 1;
  auto offset_of = []( int sub, int v ) { return 32 * sub + 8 * ( v / 4 ) + v % 4; }; // of a register's key from key_l

  load( 0 );
  for ( uint32_t i = 0; i < tiles; i++ ) {
    __syncthreads(); // the last tile's readers are done (and the bias table is written)
    store();
    __syncthreads();
    if ( i + 1 < tiles ) {
      load( i + 1 );
    }
    const uint32_t t0 = tile_at( i );
    const uint32_t last_key = t0 + TILE_KEYS - 1;
    const bool in_window = i >= kept_tiles;
    if ( in_window && ( t0 > wave_last || ( t0 >= s.keep_first && wave_first - min( last_key, wave_first ) >= s.window ) ) ) {
      continue; // keys that none of the wave's columns sees
    }
    const bool far = bias_row == 0 || ( last_key <= wave_first && wave_first - last_key >= n_dist - 1 ); // every distance in the table's last row
    const bool past_window = in_window && wave_last - t0 >= s.window && last_key >= s.keep_first;
    const bool edge = in_window ? last_key > wave_first || past_window : last_key >= kept;
    mfma_f32x16 sx[2];
#pragma unroll
    for ( int k = 0; k < KS; k++ ) { // (the two halves in turn: a product that waits for the one before it leaves the matrix unit idle)
#pragma unroll
      for ( int sub = 0; sub < 2; sub++ ) {
        const uint32_t row = 32 * sub + r;
        const bf16x8 a = __builtin_bit_cast( bf16x8, s_k[row * 16 + ( ( 2 * k + g2 ) ^ ( SHARED ? shared_swizzle( row ) : row & 15 ) )] );
        const mfma_f32x16 zero = { 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0 };
        sx[sub] = Mfma<__bf16>::k16( a, qb[k], k == 0 ? zero : sx[sub] );
      }
    }
    float st[2][16];
#pragma unroll
    for ( int sub = 0; sub < 2; sub++ ) {
#pragma unroll
      for ( int v = 0; v < 16; v++ ) {
        st[sub][v] = sx[sub][v];
      }
    }
    // ---- scale, bias by distance, mask (log2 domain)
    const uint32_t key_l = t0 + 4 * g2; // key of register v: key_l + offset_of( sub, v )
    const int32_t dist_l = (int32_t)( pos - key_l );
    auto scores = [&]( auto bias_of ) __attribute__( ( always_inline ) ) {
#pragma unroll
      for ( int sub = 0; sub < 2; sub++ ) {
#pragma unroll
        for ( int q4 = 0; q4 < 4; q4++ ) {
          float4 f = make_float4( scale_log2e, scale_log2e, scale_log2e, scale_log2e );
          if constexpr ( SHARED ) { // a factor for each key
            f = *reinterpret_cast<const float4*>( s_factor + 32 * sub + 8 * q4 + 4 * g2 );
          }
          const float factor[4] = { f.x, f.y, f.z, f.w };
#pragma unroll
          for ( int e = 0; e < 4; e++ ) {
            st[sub][4 * q4 + e] = __builtin_fmaf( st[sub][4 * q4 + e], factor[e], bias_of( offset_of( sub, 4 * q4 + e ) ) );
          }
        }
      }
    };
    if ( far ) {
      const float b = my_bias[n_dist - 1];
      scores( [&]( int ) __attribute__( ( always_inline ) ) { return b; } );
    } else if ( bias_pad > 0 ) { // from the distance of the last key up, one address for all
      const float* row = my_bias + dist_l - ( (int)TILE_KEYS - 5 );
      scores( [&]( int o ) __attribute__( ( always_inline ) ) { return row[(int)TILE_KEYS - 5 - o]; } );
    } else {
      scores( [&]( int o ) __attribute__( ( always_inline ) ) { return my_bias[min( pos - min( key_l + o, pos ), n_dist - 1 )]; } );
    }
    if ( edge ) { // the hidden keys of a column are those before or behind one offset, which a register's is compared with
      auto hide = [&]( auto hidden ) __attribute__( ( always_inline ) ) {
#pragma unroll
        for ( int sub = 0; sub < 2; sub++ ) {
#pragma unroll
          for ( int v = 0; v < 16; v++ ) {
            st[sub][v] = hidden( (int32_t)offset_of( sub, v ) ) ? -INFINITY : st[sub][v];
          }
        }
      };
      const int32_t end = in_window ? dist_l + 1 : (int32_t)( kept - key_l );
      hide( [&]( int32_t o ) __attribute__( ( always_inline ) ) { return o >= end; } );
      if ( in_window && past_window ) {
        const int32_t outside = dist_l - (int32_t)s.window, keep = (int32_t)( s.keep_first - min( s.keep_first, key_l ) );
        hide( [&]( int32_t o ) __attribute__( ( always_inline ) ) { return ( o <= outside ) & ( o >= keep ); } );
      }
    }
    // ---- online softmax
    float mx4[4];
#pragma unroll
    for ( int c = 0; c < 4; c++ ) {
      mx4[c] = st[c >> 1][8 * ( c & 1 )];
#pragma unroll
      for ( int e = 1; e < 8; e++ ) {
        mx4[c] = fmaxf( mx4[c], st[c >> 1][8 * ( c & 1 ) + e] );
      }
    }
    const float mx = half_wave_max( fmaxf( fmaxf( mx4[0], mx4[1] ), fmaxf( mx4[2], mx4[3] ) ) );
    if ( __builtin_amdgcn_ballot_w64( mx > m + LAZY ) != 0 ) {
      const float m_new = fmaxf( m, mx );
      const float alpha = __builtin_amdgcn_exp2f( m - m_new );
      m = m_new;
      l *= alpha;
#pragma unroll
      for ( int vb = 0; vb < VB; vb++ ) {
#pragma unroll
        for ( int v = 0; v < 16; v++ ) {
          acc[vb][v] *= alpha;
        }
      }
    }
#pragma unroll
    for ( int kk = 0; kk < 4; kk++ ) { // 16 keys
      union
      {
        uint32_t pair[4];
        bf16x8 x;
      } hi, lo;
#pragma unroll
      for ( int e = 0; e < 4; e++ ) {
        const float p0 = __builtin_amdgcn_exp2f( st[kk >> 1][8 * ( kk & 1 ) + 2 * e] - m );
        const float p1 = __builtin_amdgcn_exp2f( st[kk >> 1][8 * ( kk & 1 ) + 2 * e + 1] - m );
        l += p0;
        l += p1;
        hi.pair[e] = rounded_pair<__bf16>( p0, p1 );
        asm( "" : "+v"( hi.pair[e] ) ); // (taken apart again below: the compiler would convert the two once more instead)
        lo.pair[e] = rounded_pair<__bf16>( p0 - __builtin_bit_cast( float, hi.pair[e] << 16 ), p1 - __builtin_bit_cast( float, hi.pair[e] & 0xffff0000u ) );
      }
#pragma unroll
      for ( int vp = 0; vp < VB; vp += 2 ) { // (two blocks in turn: a product that waits for the one before it leaves the matrix unit idle)
        union
        {
          v4s half[2];
          bf16x8 x;
        } a[2];
#pragma unroll
        for ( int c = 0; c < min( 2, VB - vp ); c++ ) {
#pragma unroll
          for ( int hf = 0; hf < 2; hf++ ) {
            a[c].half[hf] = __builtin_amdgcn_ds_read_tr16_b64_v4i16( (lds_v4s)( (lds_char*)s_v + ( v_lane ^ ( 64 * ( vp + c ) ) ^ ( SHARED ? 32 * hf : 0 ) ) + ( 16 * kk + 8 * hf ) * 256 ) );
          }
        }
#pragma unroll
        for ( int c = 0; c < min( 2, VB - vp ); c++ ) {
          acc[vp + c] = Mfma<__bf16>::k16( a[c].x, lo.x, acc[vp + c] );
        }
#pragma unroll
        for ( int c = 0; c < min( 2, VB - vp ); c++ ) {
          acc[vp + c] = Mfma<__bf16>::k16( a[c].x, hi.x, acc[vp + c] );
        }
      }
    }
  }
  l += __shfl_xor( l, 32 );
  if ( !col_ok ) {
    return;
  }
  const uint64_t row = (uint64_t)ctx * wr.n_tokens + tok;
  const float inv = 1.0f / l * out.gate( row, h0 + hc );
  __bf16* o = out.out + row * out.stride + ( h0 + hc ) * s.vdim;
  const bool wide = s.vdim % 4 == 0 && out.stride % 4 == 0;
#pragma unroll
  for ( int vb = 0; vb < VB; vb++ ) {
#pragma unroll
    for ( int q4 = 0; q4 < 4; q4++ ) {
      const uint32_t d = 32 * vb + 8 * q4 + 4 * g2;
      union
      {
        __bf16 e[4];
        uint2 raw;
      } y;
#pragma unroll
      for ( int e = 0; e < 4; e++ ) {
        y.e[e] = (__bf16)( acc[vb][4 * q4 + e] * inv );
      }
      if ( wide && d < s.vdim ) {
        *reinterpret_cast<uint2*>( o + d ) = y.raw;
      } else if ( !wide ) {
        for ( int e = 0; e < 4; e++ ) {
          if ( d + e < s.vdim ) {
            o[d + e] = y.e[e];
          }
        }
      }
    }
  }
}

// ---- few tokens: one query row at a time on the matrix cores (bf16, head sizes up to 128) ---------------------------------------
//
// The products of the tile kernel in 16 x 16 blocks, with the query heads of a group as the columns (where the group is small most of them
// stay empty: the kernel streams keys, and the matrix cores keep up with that many times over).  A wave takes every NW-th tile of 32 of the
// row's visible keys, numbered as in the rows kernel, so nothing needs a mask but the end; its tiles pass through LDS of its own, the next
// one's rows on their way into registers meanwhile, without a barrier.  Two blocks of scores are, as they lie, the right operand of
// the product with the values: slot 8 g + e of its 32 keys is key 4 g + e for e < 4, else key 16 + 4 g + e - 4 (g = lane / 16).
constexpr uint32_t STEP_KEYS = 32;
constexpr uint32_t STEP_COLS = 16; // query heads of a work-group
// LDS of a work-group in 16-byte units: the waves' tiles, and the factors of their keys behind them; the results of the waves take its place
// at the end
constexpr uint32_t step_lds( int waves, bool shared ) { return waves * ( STEP_KEYS * ( shared ? 16 : 32 ) + ( shared ? STEP_KEYS / 4 : 0 ) ); }
static_assert( step_lds( 1, true ) * 16 >= STEP_COLS * ( 128 + 2 ) * sizeof( float ), "the results of a wave, heads of up to 128" );
// 16-byte chunks of a key's 256 bytes are XORed with this: 16 rows at one chunk (plain reads) and 8 rows at one pair of chunks (transposing
// reads) lie in different banks
__device__ __forceinline__ uint32_t step_swizzle( uint32_t row ) { return ( ( row & 7 ) << 1 ) | ( ( row >> 3 ) & 1 ); }

// maximum over the four lanes of a column (lane, lane ^ 16, lane ^ 32, lane ^ 48), in all of them
__device__ __forceinline__ float column_max( float v )
{
  const unsigned bits = __builtin_bit_cast( unsigned, v );
  const auto rows = __builtin_amdgcn_permlane16_swap( bits, bits, false, false );
  const unsigned even = rows[0], odd = rows[1];
  return half_wave_max( fmaxf( __builtin_bit_cast( float, even ), __builtin_bit_cast( float, odd ) ) );
}

// D: head size up to which the kernel goes; NW waves, HB blocks of head_cols heads side by side, NW / HB waves on the keys of each
template<int D, bool SHARED, int NW, int HB>
__global__ __launch_bounds__( 64 * NW, SHARED ? 4 : 2 ) void window_decode_kernel( WindowOut<__bf16> out,
                                                                                         float* __restrict__ partial,
                                                                                         const __bf16* __restrict__ q,
                                                                                         const float* __restrict__ bias,
                                                                                         WindowRows wr,
                                                                                         WindowShape s,
                                                                                         uint32_t head_cols,
                                                                                         uint32_t keys_per_split,
                                                                                         uint32_t splits )
{
  constexpr int KS = D / 32, VB = D / 16; // steps of 32 of the query/key size, blocks of 16 of the value size
  __shared__ uint4 tiles[step_lds( NW, SHARED )]; // K and V of each wave, 256 bytes a key
  const uint32_t head_blocks = s.heads / ( head_cols * HB );
  const uint32_t hb = blockIdx.x % head_blocks, split = blockIdx.x / head_blocks % splits;
  const uint64_t row = blockIdx.x / head_blocks / splits;
  const uint32_t ctx = (uint32_t)( row / wr.n_tokens ), tok = (uint32_t)( row % wr.n_tokens );
  const uint8_t* base = static_cast<const uint8_t*>( wr.rows[ctx] );
  if ( base == nullptr ) {
    return;
  }
  const __bf16* cache = reinterpret_cast<const __bf16*>( base + wr.offset );
  const uint32_t wave = __builtin_amdgcn_readfirstlane( threadIdx.x >> 6 ), block = wave % HB, turn = wave / HB;
  const uint32_t h0 = ( hb * HB + block ) * head_cols, g = h0 / s.group;
  const uint32_t pos = wr.start_pos[ctx] + tok;
  const Visible vis = visible_keys( pos, s );
  const uint32_t k_begin = split * keys_per_split, k_end = min( vis.count, k_begin + keys_per_split );
  const uint32_t lane = threadIdx.x & 63, r = lane & 15, g4 = lane >> 4;
  const uint32_t hc = min( r, head_cols - 1 ); // columns beyond do as the last one and are not stored
  uint4* s_k = tiles + wave * STEP_KEYS * ( SHARED ? 16 : 32 );
  uint4* s_v = SHARED ? s_k : s_k + STEP_KEYS * 16;
  float* s_factor = reinterpret_cast<float*>( tiles + NW * STEP_KEYS * ( SHARED ? 16 : 32 ) ) + wave * STEP_KEYS; // times scale and log2(e)

  bf16x8 qb[KS];
#pragma unroll
  for ( int k = 0; k < KS; k++ ) {
    const uint32_t ch = 4 * k + g4;
    u32x4_t v = { 0, 0, 0, 0 };
    if ( ch * 8 < s.dpad ) {
      v = *(global_u32x4_t*)( q + ( row * s.heads + h0 + hc ) * s.dpad + ch * 8 );
    }
    qb[k] = __builtin_bit_cast( bf16x8, v );
  }
  const bool k_chunk = r * 8 < s.dpad && r < D / 8, v_chunk = r * 8 < s.vpad && r < D / 8;
  const uint32_t row_bytes = s.row_elems() * sizeof( __bf16 );
  const uint32_t at_k = ( g * s.dpad + r * 8 ) * sizeof( __bf16 ), at_v = ( s.k_elems() + g * s.vpad + r * 8 ) * sizeof( __bf16 );
  u32x4_t rk[8], rv[SHARED ? 1 : 8]; // chunks beyond a head's size stay zero
#pragma unroll
  for ( int k = 0; k < 8; k++ ) {
    rk[k] = u32x4_t { 0, 0, 0, 0 };
    rv[SHARED ? 0 : k] = u32x4_t { 0, 0, 0, 0 };
  }
  const float* factors = reinterpret_cast<const float*>( base + wr.factors );
  float rf = 0.0f;
  auto load_row = [&]( int k, const char* row_k, uint32_t off ) {
    if ( k_chunk ) {
      rk[k] = __builtin_nontemporal_load( (global_u32x4_t*)( row_k + ( off + at_k ) ) );
    }
    if constexpr ( !SHARED ) {
      if ( v_chunk ) {
        rv[k] = __builtin_nontemporal_load( (global_u32x4_t*)( row_k + ( off + at_v ) ) );
      }
    }
  };
  auto load = [&]( uint32_t i0 ) {
    if constexpr ( SHARED ) {
      rf = factors[factor_index( vis.key( min( i0 + ( lane & 31 ), k_end - 1 ) ), g, s.kv_heads )];
    }
    if ( i0 + STEP_KEYS <= k_end && ( i0 >= vis.kept || i0 + STEP_KEYS <= vis.kept ) ) { // neighbouring rows: one address for the wave
      const char* tile = reinterpret_cast<const char*>( cache ) + (uint64_t)vis.key( i0 ) * row_bytes;
#pragma unroll
      for ( int k = 0; k < 8; k++ ) {
        load_row( k, tile + 4 * k * row_bytes, g4 * row_bytes );
      }
    } else {
#pragma unroll
      for ( int k = 0; k < 8; k++ ) {
        const uint32_t j = vis.key( min( i0 + g4 + 4 * k, k_end - 1 ) ); // past the end: the last key again, without weight
        load_row( k, reinterpret_cast<const char*>( cache ) + (uint64_t)j * row_bytes, 0 );
      }
    }
  };
  // a lane's bytes in a tile: of the row it writes first, of the key it reads for the scores, and of the transposing reads (16 lanes bring
  // 4 keys of 16 value columns, lane i gets column i).  The other places are a few bits and rows away.
  const uint32_t w_home = g4 * 256 + ( r ^ step_swizzle( g4 ) ) * 16;
  const uint32_t k_home = r * 256 + ( g4 ^ step_swizzle( r ) ) * 16;
  const uint32_t v_row = 4 * g4 + ( r >> 2 );
  const uint32_t v_home = v_row * 256 + ( ( ( ( r & 3 ) >> 1 ) ^ step_swizzle( v_row ) ) * 16 ) + ( r & 1 ) * 8;
  const float scale_log2e = s.scale * LOG2E;
  const float* my_bias = bias != nullptr ? bias + (uint64_t)( h0 + hc ) * s.n_dist : nullptr;
  const float far_bias = bias != nullptr ? my_bias[s.n_dist - 1] * LOG2E : 0.0f;

  mfma_f32x4 acc[VB];
#pragma unroll
  for ( int vb = 0; vb < VB; vb++ ) {
    acc[vb] = mfma_f32x4 { 0.0f, 0.0f, 0.0f, 0.0f };
  }
  float m = NO_KEY, l = 0.0f;
  uint32_t i0 = k_begin + turn * STEP_KEYS;
  if ( i0 < k_end ) {
    load( i0 );
  }
  for ( ; i0 < k_end; i0 += NW / HB * STEP_KEYS ) {
    uint32_t w_lane = w_home, k_lane = k_home, v_lane = v_home;
    asm( "" : "+v"( w_lane ), "+v"( k_lane ), "+v"( v_lane ) ); // the addresses beside these are made where they are used, not kept in registers
#pragma unroll
    for ( int k = 0; k < 8; k++ ) {
      const uint32_t at = ( w_lane ^ ( 16 * step_swizzle( 4 * k ) ) ) + 4 * k * 256;
      *reinterpret_cast<uint4*>( reinterpret_cast<char*>( s_k ) + at ) = __builtin_bit_cast( uint4, rk[k] );
      if constexpr ( !SHARED ) {
        *reinterpret_cast<uint4*>( reinterpret_cast<char*>( s_v ) + at ) = __builtin_bit_cast( uint4, rv[k] );
      }
    }
    if ( SHARED && lane < STEP_KEYS ) {
      s_factor[lane] = rf * scale_log2e;
    }
    if ( i0 + NW / HB * STEP_KEYS < k_end ) {
      load( i0 + NW / HB * STEP_KEYS );
    }
    __builtin_amdgcn_fence( __ATOMIC_RELEASE, "wavefront" );
    float st[8]; // of key i0 + 16 (e / 4) + 4 g4 + e % 4
#pragma unroll
    for ( int t = 0; t < 2; t++ ) {
      mfma_f32x4 d = { 0.0f, 0.0f, 0.0f, 0.0f };
#pragma unroll
      for ( int k = 0; k < KS; k++ ) {
        const uint4 a = *reinterpret_cast<const uint4*>( reinterpret_cast<const char*>( s_k ) + ( k_lane ^ ( 64 * k ) ) + 16 * t * 256 );
        d = Mfma<__bf16>::k32( __builtin_bit_cast( bf16x8, a ), qb[k], d );
      }
      float4 f = make_float4( scale_log2e, scale_log2e, scale_log2e, scale_log2e );
      if constexpr ( SHARED ) {
        f = *reinterpret_cast<const float4*>( s_factor + 16 * t + 4 * g4 );
      }
      st[4 * t] = d[0] * f.x, st[4 * t + 1] = d[1] * f.y, st[4 * t + 2] = d[2] * f.z, st[4 * t + 3] = d[3] * f.w;
    }
    if ( bias != nullptr ) {
      // every distance of the tile in the bias table's last row?
      const uint32_t nearest = vis.key( min( i0 + STEP_KEYS, k_end ) - 1 );
      if ( pos - nearest >= s.n_dist - 1 ) {
#pragma unroll
        for ( int e = 0; e < 8; e++ ) {
          st[e] += far_bias;
        }
      } else {
#pragma unroll
        for ( int e = 0; e < 8; e++ ) {
          const uint32_t j = vis.key( min( i0 + 16 * ( e / 4 ) + 4 * g4 + e % 4, k_end - 1 ) );
          st[e] += my_bias[min( pos - j, s.n_dist - 1 )] * LOG2E;
        }
      }
    }
    if ( i0 + STEP_KEYS > k_end ) {
#pragma unroll
      for ( int e = 0; e < 8; e++ ) {
        st[e] = i0 + 16 * ( e / 4 ) + 4 * g4 + e % 4 < k_end ? st[e] : -INFINITY;
      }
    }
    const float mx = column_max( fmaxf( fmaxf( fmaxf( st[0], st[1] ), fmaxf( st[2], st[3] ) ), fmaxf( fmaxf( st[4], st[5] ), fmaxf( st[6], st[7] ) ) ) );
    if ( __builtin_amdgcn_ballot_w64( mx > m + LAZY ) != 0 ) {
      const float m_new = fmaxf( m, mx );
      const float alpha = __builtin_amdgcn_exp2f( m - m_new );
      m = m_new;
      l *= alpha;
#pragma unroll
      for ( int vb = 0; vb < VB; vb++ ) {
#pragma unroll
        for ( int v = 0; v < 4; v++ ) {
          acc[vb][v] *= alpha;
        }
      }
    }
    bf16x8 hi, lo;
#pragma unroll
    for ( int e = 0; e < 8; e++ ) {
      const float p = __builtin_amdgcn_exp2f( st[e] - m );
      l += p;
      hi[e] = (__bf16)p;
      lo[e] = (__bf16)( p - (float)hi[e] );
    }
#pragma unroll
    for ( int vb = 0; vb < VB; vb++ ) {
      union
      {
        v4s half[2];
        bf16x8 x;
      } a;
#pragma unroll
      for ( int t = 0; t < 2; t++ ) {
        a.half[t] = __builtin_amdgcn_ds_read_tr16_b64_v4i16( (lds_v4s)( (lds_char*)s_v + ( v_lane ^ ( 32 * vb ) ) + 16 * t * 256 ) );
      }
      acc[vb] = Mfma<__bf16>::k32( a.x, lo, acc[vb] );
      acc[vb] = Mfma<__bf16>::k32( a.x, hi, acc[vb] );
    }
    __builtin_amdgcn_fence( __ATOMIC_ACQUIRE, "wavefront" );
  }
  l += __shfl_xor( l, 16 );
  l += __shfl_xor( l, 32 );
  __syncthreads(); // the tiles' LDS takes the waves' results
  float* results = reinterpret_cast<float*>( tiles );
  if ( r < head_cols ) {
    float* mine = results + ( wave * head_cols + r ) * ( s.vpad + 2 );
#pragma unroll
    for ( int vb = 0; vb < VB; vb++ ) {
#pragma unroll
      for ( int v = 0; v < 4; v++ ) {
        const uint32_t d = 16 * vb + 4 * g4 + v;
        if ( d < s.vpad ) {
          mine[d] = acc[vb][v];
        }
      }
    }
    if ( g4 == 0 ) {
      mine[s.vpad] = l;
      mine[s.vpad + 1] = m * ( 1.0f / LOG2E ); // the sums are joined in natural units
    }
  }
  __syncthreads();
  finish_split<__bf16, NW / HB, 64 * NW>( out, partial, results, HB * head_cols, HB * head_cols, row, hb * HB * head_cols, split, splits, s );
}

// ---- few tokens of heads that share their keys with no other: dot products in the vector ALU -------------------------------------
//
// With one query head to a kv head the matrix cores above would multiply one column of sixteen, and a tile's way there is through LDS.  Here 16 lanes hold one
// key, eight elements a lane, straight from memory, and the vector ALU keeps up with it.  A wave walks a range of the visible keys in tiles of
// 4 U, from one of its own on (work-groups in step on rows a power of two apart meet on few channels), the next tile under way; lane c of a row of lanes owns the
// score of key c % U, so that a tile is one exponential.  Scores, weights and sums are fp32, and the weights enter the sums whole.
// Bound by memory, and by the vector ALU next: with the products of the scores unpacked to fp32, where v_dot2_f32_bf16 takes two at a time, values that are keys
// took 49.5 us instead of 43.5 at 32 contexts x 32 heads x 1025 keys (6.2 TB/s; 46.6 by the kernel above), K and V apart 87.2 instead of 84.9 (6.3; 92.2).
typedef __bf16 bf16x2_t __attribute__( ( ext_vector_type( 2 ) ) );
template<bool SHARED, int NW, int HB>
__global__ __launch_bounds__( 64 * NW, 4 ) void window_dot_kernel( WindowOut<__bf16> out,
                                                                   float* __restrict__ partial,
                                                                   const __bf16* __restrict__ q,
                                                                   const float* __restrict__ bias,
                                                                   WindowRows wr,
                                                                   WindowShape s,
                                                                   uint32_t keys_per_split,
                                                                   uint32_t splits )
{
  constexpr int U = SHARED ? 8 : 4; // keys of a row of lanes in a tile: 8 KB of a wave either way
  constexpr uint32_t TILE = 4 * U;
  __shared__ float results[NW * ( 128 + 2 )];
  const uint32_t head_blocks = s.heads / HB, hb = blockIdx.x % head_blocks, split = blockIdx.x / head_blocks % splits;
  const uint64_t row = blockIdx.x / head_blocks / splits;
  const uint32_t ctx = (uint32_t)( row / wr.n_tokens ), tok = (uint32_t)( row % wr.n_tokens );
  const uint8_t* base = static_cast<const uint8_t*>( wr.rows[ctx] );
  const uint32_t pos = wr.start_pos[ctx] + tok; // (read before the branch: one round trip for the two)
  if ( base == nullptr ) {
    return;
  }
  const uint32_t wave = __builtin_amdgcn_readfirstlane( threadIdx.x >> 6 ), lane = threadIdx.x & 63, r = lane >> 4, c = lane & 15;
  const uint32_t head = hb * HB + wave % HB, turn = wave / HB;
  const Visible vis = visible_keys( pos, s );
  const uint32_t s_begin = split * keys_per_split, s_end = min( vis.count, s_begin + keys_per_split );
  const uint32_t s_keys = s_end > s_begin ? s_end - s_begin : 0;
  const uint32_t per_wave = ( s_keys + NW / HB * TILE - 1 ) / ( NW / HB * TILE ) * TILE;
  const uint32_t k_begin = s_begin + turn * per_wave, k_end = min( s_end, k_begin + per_wave );

  const char* cache = reinterpret_cast<const char*>( base + wr.offset );
  const uint32_t row_bytes = s.row_elems() * sizeof( __bf16 );
  const bool k_chunk = c * 8 < s.dpad, v_chunk = c * 8 < s.vpad;
  const uint32_t at_k = ( head * s.dpad + c * 8 ) * sizeof( __bf16 ), at_v = ( s.k_elems() + head * s.vpad + c * 8 ) * sizeof( __bf16 );
  const float* factors = reinterpret_cast<const float*>( base + wr.factors );
  u32x4_t qr = { 0, 0, 0, 0 };
  if ( k_chunk ) {
    qr = *(global_u32x4_t*)( q + ( row * s.heads + head ) * s.dpad + c * 8 );
  }

  u32x4_t kn[U], vn[SHARED ? 1 : U]; // chunks beyond a head's size stay zero
#pragma unroll
  for ( int j = 0; j < U; j++ ) {
    kn[j] = u32x4_t { 0, 0, 0, 0 };
    vn[SHARED ? 0 : j] = u32x4_t { 0, 0, 0, 0 };
  }
  float fn = 0.0f;
  const uint32_t own = 4 * ( c % U ) + r; // key of the tile whose score is this lane's
  auto load_row = [&]( int j, const char* key_row, uint32_t off ) __attribute__( ( always_inline ) ) {
    if ( k_chunk ) {
      kn[j] = __builtin_nontemporal_load( (global_u32x4_t*)( key_row + ( off + at_k ) ) );
    }
    if constexpr ( !SHARED ) {
      if ( v_chunk ) {
        vn[j] = __builtin_nontemporal_load( (global_u32x4_t*)( key_row + ( off + at_v ) ) );
      }
    }
  };
  auto load = [&]( uint32_t i0 ) __attribute__( ( always_inline ) ) {
    if constexpr ( SHARED ) {
      fn = factors[factor_index( vis.key( min( i0 + own, k_end - 1 ) ), head, s.kv_heads )];
    }
    if ( i0 + TILE <= k_end && ( i0 >= vis.kept || i0 + TILE <= vis.kept ) ) { // neighbouring rows: one address for the wave
      const char* tile = cache + (uint64_t)vis.key( i0 ) * row_bytes;
#pragma unroll
      for ( int j = 0; j < U; j++ ) {
        load_row( j, tile + 4 * j * row_bytes, r * row_bytes );
      }
    } else {
#pragma unroll
      for ( int j = 0; j < U; j++ ) { // past the end: the last key again, without weight
        load_row( j, cache + (uint64_t)vis.key( min( i0 + 4 * j + r, k_end - 1 ) ) * row_bytes, 0 );
      }
    }
  };
  const float scale_log2e = s.scale * LOG2E;
  const float* my_bias = bias != nullptr ? bias + (uint64_t)head * s.n_dist : nullptr;
  const float far_bias = bias != nullptr ? my_bias[s.n_dist - 1] * LOG2E : 0.0f;

  float acc[8];
#pragma unroll
  for ( int e = 0; e < 8; e++ ) {
    acc[e] = 0.0f;
  }
  float m = NO_KEY, l = 0.0f; // m: of a row of lanes; l: of this lane's keys
  const uint32_t n_tiles = k_begin < k_end ? ( k_end - k_begin + TILE - 1 ) / TILE : 0;
  uint32_t i0 = n_tiles > 0 ? k_begin + (uint32_t)( ( row * 5 + turn * 3 ) * 7 ) % n_tiles * TILE : 0;
  if ( n_tiles > 0 ) {
    load( i0 );
  }
  for ( uint32_t n = 0; n < n_tiles; n++ ) {
    const uint32_t next = i0 + TILE < k_end ? i0 + TILE : k_begin;
    u32x4_t kc[U], vc[SHARED ? 1 : U];
#pragma unroll
    for ( int j = 0; j < U; j++ ) {
      kc[j] = kn[j];
      vc[SHARED ? 0 : j] = vn[SHARED ? 0 : j];
    }
    const float f = SHARED ? fn * scale_log2e : scale_log2e;
    if ( n + 1 < n_tiles ) {
      load( next );
    }
    auto unpacked = []( u32x4_t raw, float( &v )[8] ) __attribute__( ( always_inline ) ) {
#pragma unroll
      for ( int e = 0; e < 4; e++ ) {
        v[2 * e] = __builtin_bit_cast( float, raw[e] << 16 );
        v[2 * e + 1] = __builtin_bit_cast( float, raw[e] & 0xffff0000u );
      }
    };
    float sc = 0.0f;
#pragma unroll
    for ( int j = 0; j < U; j++ ) {
      float dot = 0.0f;
#pragma unroll
      for ( int e = 0; e < 4; e++ ) {
        const uint32_t kw = kc[j][e], qw = qr[e];
        dot = __builtin_amdgcn_fdot2_f32_bf16( __builtin_bit_cast( bf16x2_t, kw ), __builtin_bit_cast( bf16x2_t, qw ), dot, false );
      }
      dot = row16_sum( dot );
      sc = j == 0 || c % U == (uint32_t)j ? dot : sc;
    }
    sc *= f;
    if ( bias != nullptr ) {
      // every distance of the tile in the bias table's last row?
      const uint32_t nearest = vis.key( min( i0 + TILE, k_end ) - 1 );
      sc += pos - nearest >= s.n_dist - 1 ? far_bias : my_bias[min( pos - vis.key( min( i0 + own, k_end - 1 ) ), s.n_dist - 1 )] * LOG2E;
    }
    sc = i0 + own < k_end ? sc : -INFINITY;
    const float mx = row16_max( sc );
    if ( __builtin_amdgcn_ballot_w64( mx > m + LAZY ) != 0 ) {
      const float m_new = fmaxf( m, mx );
      const float alpha = __builtin_amdgcn_exp2f( m - m_new );
      m = m_new;
      l *= alpha;
#pragma unroll
      for ( int e = 0; e < 8; e++ ) {
        acc[e] *= alpha;
      }
    }
    const float p = __builtin_amdgcn_exp2f( sc - m );
    l += c < U ? p : 0.0f;
    auto add = [&]( auto j ) __attribute__( ( always_inline ) ) {
      constexpr int J = decltype( j )::value;
      float v8[8];
      unpacked( SHARED ? kc[J] : vc[SHARED ? 0 : J], v8 );
      const float pj = __builtin_bit_cast( float, __builtin_amdgcn_update_dpp( 0, __builtin_bit_cast( int, p ), 0x150 + J, 0xF, 0xF, true ) ); // lane J of the row
#pragma unroll
      for ( int e = 0; e < 8; e++ ) {
        acc[e] += pj * v8[e];
      }
    };
    add( std::integral_constant<int, 0> {} ), add( std::integral_constant<int, 1> {} ), add( std::integral_constant<int, 2> {} ), add( std::integral_constant<int, 3> {} );
    if constexpr ( U == 8 ) {
      add( std::integral_constant<int, 4> {} ), add( std::integral_constant<int, 5> {} ), add( std::integral_constant<int, 6> {} ), add( std::integral_constant<int, 7> {} );
    }
    i0 = next;
  }
  // the rows of lanes added up against the wave's maximum: lane (r, c) ends up with elements 8 c + r and 8 c + 4 + r
  const float m_all = column_max( m ), f = __builtin_amdgcn_exp2f( m - m_all );
  l = row16_sum( l ) * f;
  l = ( lane_value( l, 0 ) + lane_value( l, 16 ) ) + ( lane_value( l, 32 ) + lane_value( l, 48 ) );
#pragma unroll
  for ( int e = 0; e < 8; e++ ) {
    acc[e] *= f;
  }
  float* mine = results + wave * ( s.vpad + 2 );
#pragma unroll
  for ( int k = 0; k < 2; k++ ) {
    const float sum = sum_rows( sum_halves( acc[4 * k], acc[4 * k + 2] ), sum_halves( acc[4 * k + 1], acc[4 * k + 3] ) );
    const uint32_t d = 8 * c + 4 * k + r;
    if ( d < s.vpad ) {
      mine[d] = sum;
    }
  }
  if ( lane == 0 ) {
    mine[s.vpad] = l;
    mine[s.vpad + 1] = m_all * ( 1.0f / LOG2E ); // the sums are joined in natural units
  }
  __syncthreads();
  finish_split<__bf16, NW / HB, 64 * NW>( out, partial, results, HB, HB, row, hb * HB, split, splits, s );
}

template<typename E, int NC, bool SHARED>
void launch_rows( int hq, dim3 grid, hipStream_t st, const WindowOut<E>& out, float* partial, const E* q, const float* bias, const WindowRows& wr, const WindowShape& s,
                  uint32_t keys_per_split, uint32_t splits )
{
  const size_t lds = 4ull * hq * ( s.vpad + 2 ) * sizeof( float );
  if constexpr ( NC <= 1 ) {
    if ( hq == 8 ) {
      window_rows_kernel<E, 8, NC, SHARED><<<grid, 256, lds, st>>>( out, partial, q, bias, wr, s, keys_per_split, splits );
      return;
    }
  }
  if constexpr ( NC <= 2 ) {
    if ( hq == 4 ) {
      window_rows_kernel<E, 4, NC, SHARED><<<grid, 256, lds, st>>>( out, partial, q, bias, wr, s, keys_per_split, splits );
      return;
    }
    if ( hq == 2 ) {
      window_rows_kernel<E, 2, NC, SHARED><<<grid, 256, lds, st>>>( out, partial, q, bias, wr, s, keys_per_split, splits );
      return;
    }
  }
  window_rows_kernel<E, 1, NC, SHARED><<<grid, 256, lds, st>>>( out, partial, q, bias, wr, s, keys_per_split, splits );
}

// Splits of the visible keys of a call's rows, and room for their partial results: as many as give every CU two work-groups, of at
// least `least` keys each.
struct SplitPlan
{
  uint32_t keys { 0 }, splits { 1 };
  float* partial { nullptr };
};
int cut_keys( const WindowShape& s, uint64_t rows, uint64_t most, uint64_t splits, hipStream_t st, SplitPlan* plan )
{
  plan->keys = (uint32_t)( ( ( most + splits - 1 ) / splits + 31 ) / 32 * 32 );
  plan->splits = (uint32_t)( ( most + plan->keys - 1 ) / plan->keys );
  if ( plan->splits > 1 ) {
    void* p = nullptr;
    if ( int rc = stream_scratch( st, SCRATCH_MIXER, rows * s.heads * plan->splits * partial_stride( s ) * sizeof( float ), 1ull << 20, &p ) ) {
      return rc;
    }
    plan->partial = static_cast<float*>( p );
  }
  return GH_OK;
}
int plan_splits( const WindowShape& s, uint64_t rows, uint64_t head_blocks, uint32_t max_pos, uint64_t least, hipStream_t st, SplitPlan* plan )
{
  const uint64_t most = std::min<uint64_t>( (uint64_t)max_pos + 1, (uint64_t)s.window + s.keep_first );
  const uint64_t splits = std::max<uint64_t>( 1, 2ull * cu_count() / std::max<uint64_t>( 1, rows * head_blocks ) );
  return cut_keys( s, rows, most, std::min( { splits, std::max<uint64_t>( 1, most / least ), (uint64_t)64 } ), st, plan );
}
template<typename E>
int merge_splits( const WindowOut<E>& out, const SplitPlan& plan, const WindowRows& wr, const WindowShape& s, uint64_t rows, hipStream_t st )
{
  if ( plan.splits > 1 ) {
    const uint64_t pairs = rows * s.heads;
    window_merge_kernel<E><<<(unsigned)( ( pairs + 3 ) / 4 ), 256, 0, st>>>( out, plan.partial, wr, s, plan.splits, pairs );
    GH_LAUNCH_CHECK();
  }
  return GH_OK;
}

// Few rows of bf16 whose query heads have a kv head each, of 65 to 128.  us, 32 heads of 128, against window_decode_kernel, K and V apart | values that are keys:
//   1 row    1025 keys 13.9 -> 11.7, 4097 25.7 -> 18.5 | 11.7 -> 10.1, 16.5 -> 14.0
//   8 rows    300 13.4 -> 10.9, 1025 31.9 -> 25.4, 4097 91 -> 85 | 9.5 -> 8.6, 20.6 -> 15.1, 52 -> 46
//   16 rows  1025 50 -> 45, 4097 170 -> 158 | 26.7 -> 24.8, 88 -> 81
//   32 rows    64 10.7 -> 9.2, 1025 91 -> 84, 4097 325 -> 317 | 8.2 -> 6.8, 45.5 -> 44.4, 169 -> 164
//   48 rows   300 48.5 -> 38.5, 1025 129 -> 122 | 25.1 -> 22.2, 65 -> 64
// What counts is the waves on the chip, some 4 to 8 a CU, and that work-groups come out even over the CUs; beyond that neighbouring heads in a work-group, which read
// neighbouring pieces of a cache row.  So eight waves, on one head while there are no more streams of keys than CUs (cut further where that leaves CUs idle and a stream
// is long: the merge is a launch), on two heads up to twice as many and on four up to four times.
struct DotPlan
{
  uint32_t waves, heads; // of a work-group
  uint64_t splits;
};
DotPlan plan_dot( const WindowShape& s, uint64_t rows, uint64_t most )
{
  const uint64_t streams = rows * s.heads, cus = (uint64_t)cu_count(), weight = most * ( s.values_are_keys ? 1 : 2 );
  DotPlan p { 8, streams <= cus ? 1u : streams <= 2 * cus ? 2u : streams <= 4 * cus ? 4u : 2u, 1 };
  // (16 rows of 4097 keys 163 | 84.7 us with four ranges of a head's keys, 158 | 81.1 with two; 48 rows of 64 13.4 | 9.7 and 11.3 | 7.6)
  if ( p.heads == 2 && ( streams <= 2 * cus ? most > 3072 : most <= 192 ) ) {
    p.waves = 4;
  }
  while ( s.heads % p.heads != 0 ) {
    p.heads /= 2;
  }
  // Many short streams of an odd number of heads: of eight waves on one head most have no keys (120 rows of 5 heads, 33 keys 7.5 | 7.8 us, 5.9 | 5.6 with four).
  if ( p.heads == 1 && streams > 2 * cus && most <= 192 ) {
    p.waves = 4;
  }
  // Splits of 128 keys, from sixteen of them on of 256 (2 rows of 5 heads, 2500 keys 13.6 | 12.5 us in 27 splits, 11.2 | 10.4 in 16; one of 6 of 96, 16385 keys 20.0 | 15.2 in
  // 16, 18.1 | 15.1 in 32).
  if ( const uint64_t idle = cus / streams; idle >= 2 && weight >= ( idle >= 4 ? 1024u : 2048u ) ) {
    p.splits = std::max<uint64_t>( 1, std::min( { idle, most / 128, std::max<uint64_t>( 16, most / 256 ), (uint64_t)64 } ) );
  }
  // Long streams whose work-groups leave a third of the CUs without one, in their only round or in the last: a CU takes in some 35 GB/s, so that is lost.  Four waves on two
  // heads then, in as many splits as make two a CU; more work-groups than CUs are cut by three.  11 rows of 12 heads, 16385 keys 238 | 118 us, 182 | 96 so (195 | 107 by
  // window_decode_kernel), 4097 keys 62 | 33 and 51 | 30 (57 | 33); 43 rows of 6 of 96, 16385 keys 476 | 238 and 293 | 150 (451 | 250); 100 of them, values that are keys,
  // 445 and 352 (413).
  const uint64_t groups = streams / p.heads, rounds = ( groups + cus - 1 ) / cus;
  if ( s.heads % 2 == 0 && weight >= 4096 && 8 * groups >= 3 * cus && 100 * groups <= 69 * rounds * cus ) {
    if ( groups <= cus ) {
      p.waves = 4;
      p.heads = streams <= 2 * cus ? 2 : p.heads;
      p.splits = std::max<uint64_t>( 1, 2 * cus / ( streams / p.heads ) );
    } else {
      p.splits = 3;
    }
  }
  return p;
}
int attend_dot( const WindowOut<__bf16>& out, const __bf16* q, const float* bias, const WindowRows& wr, const WindowShape& s, uint64_t rows, uint32_t max_pos, hipStream_t st )
{
  const uint64_t most = std::min<uint64_t>( (uint64_t)max_pos + 1, (uint64_t)s.window + s.keep_first );
  const auto [waves, heads, splits] = plan_dot( s, rows, most );
  SplitPlan plan;
  if ( int rc = cut_keys( s, rows, most, splits, st, &plan ) ) {
    return rc;
  }
  const uint64_t grid = rows * ( s.heads / heads ) * plan.splits;
  GH_REQUIRE( grid < ( 1ull << 31 ), "gh_attn_window: grid too large" );
  auto launch = [&]( auto nw, auto hb ) {
    constexpr int NW = decltype( nw )::value, HB = decltype( hb )::value;
    if ( s.values_are_keys ) {
      window_dot_kernel<true, NW, HB><<<(unsigned)grid, 64 * NW, 0, st>>>( out, plan.partial, q, bias, wr, s, plan.keys, plan.splits );
    } else {
      window_dot_kernel<false, NW, HB><<<(unsigned)grid, 64 * NW, 0, st>>>( out, plan.partial, q, bias, wr, s, plan.keys, plan.splits );
    }
  };
  const std::integral_constant<int, 4> four {};
  const std::integral_constant<int, 8> eight {};
  const std::integral_constant<int, 2> two {};
  const std::integral_constant<int, 1> one {};
  if ( heads == 4 ) {
    waves == 4 ? launch( four, four ) : launch( eight, four );
  } else if ( heads == 2 ) {
    waves == 4 ? launch( four, two ) : launch( eight, two );
  } else {
    waves == 4 ? launch( four, one ) : launch( eight, one );
  }
  GH_LAUNCH_CHECK();
  return merge_splits( out, plan, wr, s, rows, st );
}

// few rows of bf16 with heads of up to 128
int attend_decode( const WindowOut<__bf16>& out, const __bf16* q, const float* bias, const WindowRows& wr, const WindowShape& s, uint64_t rows, uint32_t max_pos, hipStream_t st )
{
  if ( s.group == 1 && std::max( s.dpad, s.vpad ) > 64 ) {
    return attend_dot( out, q, bias, wr, s, rows, max_pos, st );
  }
  uint32_t head_cols = s.group; // the largest divisor of the group that fits
  while ( head_cols > STEP_COLS || s.group % head_cols != 0 ) {
    head_cols--;
  }
  const uint64_t blocks = s.heads / head_cols, groups = rows * blocks, most = std::min<uint64_t>( (uint64_t)max_pos + 1, (uint64_t)s.window + s.keep_first );
  // Eight waves on the keys of a row where work-groups of four would leave room on the CUs and a row has four tiles or more (below eight tiles some of the
  // waves have none); with K and V apart a CU holds one such work-group, which pays only while they are few.  us, rows x keys, four waves / eight.  32 heads of 64 with keys of
  // their own, values that are keys: 1 x 300 8.7 / 6.1, 8 x 300 10.0 / 6.6, 24 x 300 10.2 / 12.0, 32 x 1025 29.6 / 28.8, 48 x 1025 41.0 / 39.7; both: 1 x 300 9.9 / 8.0, 8 x 300
  // 11.8 / 8.8, 8 x 1025 20.2 / 22.0.  32 heads of 128 in groups of four, values that are keys: 24 x 300 12.3 / 8.4, 48 x 300 11.7 / 11.4; both: 8 x 1025 14.8 / 13.5, 8 x 2048 19.0 /
  // 22.2, 24 x 300 14.9 / 10.9, 48 x 300 17.1 / 20.4.
  const bool wide = s.values_are_keys ? ( groups < 16ull * cu_count() && most >= 16 * STEP_KEYS ) || ( groups <= (uint64_t)cu_count() && most >= 4 * STEP_KEYS )
                                      : most >= 4 * STEP_KEYS && ( 4 * groups <= (uint64_t)cu_count() || ( groups <= (uint64_t)cu_count() && most <= 16 * STEP_KEYS ) );
  // Two heads a work-group where there are more work-groups than the CUs hold and few keys to each: half as many starts (32 heads of 64 with keys of their own: 32 x 64
  // 10.5 -> 7.4, 32 x 300 22.8 -> 18.0; longer rows gain up to a fifth or nothing, 32 x 2048 100 -> 85, 48 x 1025 80 -> 80, and stay as they were).
  const bool pair = !s.values_are_keys && !wide && blocks % 2 == 0 && groups >= 3ull * cu_count() && most <= 16 * STEP_KEYS;
  const uint64_t head_blocks = pair ? blocks / 2 : blocks;
  SplitPlan plan;
  if ( int rc = plan_splits( s, rows, head_blocks, max_pos, ( wide ? 8 : pair ? 2 : 4 ) * STEP_KEYS, st, &plan ) ) {
    return rc;
  }
  const uint64_t grid = rows * head_blocks * plan.splits;
  GH_REQUIRE( grid < ( 1ull << 31 ), "gh_attn_window: grid too large" );
#define GH_WINDOW_DECODE( D, SHARED, NW, HB ) \
  window_decode_kernel<D, SHARED, NW, HB><<<(unsigned)grid, 64 * NW, 0, st>>>( out, plan.partial, q, bias, wr, s, head_cols, plan.keys, plan.splits )
  auto launch = [&]( auto size ) {
    constexpr int D = decltype( size )::value;
    if ( s.values_are_keys ) {
      wide ? GH_WINDOW_DECODE( D, true, 8, 1 ) : GH_WINDOW_DECODE( D, true, 4, 1 );
    } else if ( pair ) {
      GH_WINDOW_DECODE( D, false, 4, 2 );
    } else {
      wide ? GH_WINDOW_DECODE( D, false, 8, 1 ) : GH_WINDOW_DECODE( D, false, 4, 1 );
    }
  };
  s.dpad <= 64 && s.vpad <= 64 ? launch( std::integral_constant<int, 64> {} ) : launch( std::integral_constant<int, 128> {} );
#undef GH_WINDOW_DECODE
  GH_LAUNCH_CHECK();
  return merge_splits( out, plan, wr, s, rows, st );
}

template<typename E, bool SHARED>
int attend_rows( const WindowOut<E>& out, const E* q, const float* bias, const WindowRows& wr, const WindowShape& s, uint64_t rows, uint32_t max_pos, hipStream_t st )
{
  const uint32_t widest = std::max( s.dpad, s.vpad );
  const int max_hq = widest <= 128 ? 8 : widest <= 256 ? 4 : 1;
  int hq = 1;
  while ( hq < max_hq && hq < (int)s.group ) {
    hq *= 2;
  }
  const uint32_t head_blocks = s.kv_heads * ( ( s.group + hq - 1 ) / hq );
  GH_REQUIRE( head_blocks <= 65535, "gh_attn_window: too many heads" );
  SplitPlan plan;
  if ( int rc = plan_splits( s, rows, head_blocks, max_pos, 64, st, &plan ) ) {
    return rc;
  }
  const uint32_t per = plan.keys;
  const uint32_t splits = plan.splits;
  float* partial = plan.partial;
  const dim3 grid( (unsigned)rows, head_blocks, (unsigned)splits );
  if ( widest <= 128 ) {
    launch_rows<E, 1, SHARED>( hq, grid, st, out, partial, q, bias, wr, s, per, (uint32_t)splits );
  } else if ( widest <= 256 ) {
    launch_rows<E, 2, SHARED>( hq, grid, st, out, partial, q, bias, wr, s, per, (uint32_t)splits );
  } else {
    launch_rows<E, 4, SHARED>( hq, grid, st, out, partial, q, bias, wr, s, per, (uint32_t)splits );
  }
  GH_LAUNCH_CHECK();
  return merge_splits( out, plan, wr, s, rows, st );
}

// Whether the tile kernel serves a call; its launch.
uint32_t tile_head_cols( const WindowShape& s )
{
  uint32_t cols = s.group <= 32 && ( s.group & ( s.group - 1 ) ) == 0 ? s.group : 1;
  while ( cols > 1 && (uint64_t)cols * s.n_dist > BIAS_LDS ) { // as many as have their bias tables fit
    cols /= 2;
  }
  return cols;
}
bool tiles_applicable( const WindowShape& s, const float* bias, uint32_t n_tokens )
{
  return n_tokens >= 16 && s.dpad <= 128 && s.vpad <= 128 && ( bias == nullptr || (uint64_t)tile_head_cols( s ) * s.n_dist <= BIAS_LDS );
}
int attend_tiles( const WindowOut<__bf16>& out, const __bf16* q, const float* bias, const WindowRows& wr, const WindowShape& s, uint64_t batch, hipStream_t st )
{
  const uint32_t head_cols = tile_head_cols( s );
  const uint32_t col_blocks = ( wr.n_tokens + 128 / head_cols - 1 ) / ( 128 / head_cols );
  const uint64_t n_pairs = batch * s.kv_heads * ( s.group / head_cols );
  const uint64_t grid = ( n_pairs + 7 ) / 8 * 8 * col_blocks;
  GH_REQUIRE( grid < ( 1ull << 31 ), "gh_attn_window: grid too large" );
  const uint64_t xcd_pairs = ( n_pairs + 7 ) / 8, groups = ( xcd_pairs + GROUP_PAIRS - 1 ) / GROUP_PAIRS;
  const uint32_t group_pairs = (uint32_t)( ( xcd_pairs + groups - 1 ) / groups ); // as many in each
  const uint32_t bias_pad = bias != nullptr && (uint64_t)head_cols * ( s.n_dist + 2 * BIAS_PAD ) <= BIAS_LDS ? BIAS_PAD : 0;
  const uint32_t bias_row = bias == nullptr ? 0 : s.n_dist + 2 * bias_pad, bias_floats = head_cols * bias_row;
  const size_t lds = ( s.values_are_keys ? TILE_KEYS * ( 256 + sizeof( float ) ) : 2 * TILE_KEYS * 256 ) + std::max( bias_floats, 1u ) * sizeof( float );
#define GH_WINDOW_TILES( KS, VB, SHARED ) \
  window_tiles_kernel<KS, VB, SHARED><<<(unsigned)grid, 256, lds, st>>>( out, q, bias, wr, s, head_cols, col_blocks, (uint32_t)n_pairs, group_pairs, bias_row, bias_pad )
  if ( s.values_are_keys ) {
    if ( s.dpad <= 64 ) {
      GH_WINDOW_TILES( 4, 2, true );
    } else if ( s.dpad <= 96 ) {
      GH_WINDOW_TILES( 6, 3, true );
    } else {
      GH_WINDOW_TILES( 8, 4, true );
    }
  } else if ( s.dpad <= 64 && s.vpad <= 64 ) {
    GH_WINDOW_TILES( 4, 2, false );
  } else if ( s.vpad <= 64 ) {
    GH_WINDOW_TILES( 8, 2, false );
  } else {
    GH_WINDOW_TILES( 8, 4, false );
  }
#undef GH_WINDOW_TILES
  GH_LAUNCH_CHECK();
  return GH_OK;
}

} // namespace
} // namespace gh

using namespace gh;

extern "C" {

uint64_t gh_window_row_bytes( const gh_window_attn* a, gh_dtype dt ) { return (uint64_t)window_shape( a ).row_elems() * dtype_size( dt ); }

uint64_t gh_window_factor_bytes( const gh_window_attn* a ) { return a->values_are_keys ? (uint64_t)a->kv_heads * sizeof( float ) : 0; }

uint64_t gh_window_query_elements( const gh_window_attn* a ) { return (uint64_t)a->heads * window_shape( a ).dpad; }

int gh_matmul_window_append( void* q, const void* x, const void* wqkv, const void* bias, uint64_t width, const gh_window_attn* a, const void* q_norm,
                             const void* k_norm, float eps, void* const* context_rows_dev, uint64_t cache_offset, const uint32_t* start_pos_dev, uint64_t batch,
                             uint32_t n_tokens, gh_dtype dt, gh_stream stream )
{
  if ( int rc = ensure_init() ) {
    return rc;
  }
  const uint64_t rows = batch * n_tokens;
  if ( rows == 0 ) {
    return GH_OK;
  }
  GH_REQUIRE( q && x && wqkv && a && context_rows_dev && start_pos_dev, "gh_matmul_window_append: NULL pointer" );
  GH_REQUIRE( dt == GH_BF16 || dt == GH_F32, "gh_matmul_window_append: unsupported dtype %d", (int)dt );
  GH_REQUIRE( window_shape_ok( a ) && rows < ( 1ull << 31 ) && cache_offset % 16 == 0 && !a->values_are_keys, "gh_matmul_window_append: bad shape" );
  const WindowShape s = window_shape( a );
  const uint64_t r = (uint64_t)s.heads * s.dim + (uint64_t)s.kv_heads * ( s.dim + s.vdim );
  hipStream_t st = as_stream( stream );
  Product y;
  if ( int rc = make_product( x, wqkv, width, r, rows, dt, false, st, &y ) ) {
    return rc;
  }
  const WindowRows wr { context_rows_dev, cache_offset, 0, start_pos_dev, n_tokens };
  return with_product( dt, y, [&]( auto tag, auto view ) -> int {
    using E = decltype( tag );
    return launch_append<E>( static_cast<E*>( q ), view, static_cast<const E*>( bias ), q_norm, k_norm, eps, wr, s, rows, st );
  } );
}

int gh_attn_window( void* out, uint64_t out_stride, const float* head_gates, const void* q, const gh_window_attn* a, const float* distance_bias_dev,
                    void* const* context_rows_dev, uint64_t cache_offset, uint64_t factor_offset, const uint32_t* start_pos_dev, uint64_t batch, uint32_t n_tokens,
                    uint32_t max_start_pos, gh_dtype dt, gh_stream stream )
{
  if ( int rc = ensure_init() ) {
    return rc;
  }
  const uint64_t rows = batch * n_tokens;
  if ( rows == 0 ) {
    return GH_OK;
  }
  GH_REQUIRE( out && q && a && context_rows_dev && start_pos_dev, "gh_attn_window: NULL pointer" );
  GH_REQUIRE( dt == GH_BF16 || dt == GH_F32, "gh_attn_window: unsupported dtype %d", (int)dt );
  GH_REQUIRE( window_shape_ok( a ) && rows < ( 1ull << 31 ) && cache_offset % 16 == 0, "gh_attn_window: bad shape" );
  const WindowShape s = window_shape( a );
  GH_REQUIRE( out_stride >= (uint64_t)s.heads * s.vdim && factor_offset % 16 == 0, "gh_attn_window: bad stride or offset" );
  const WindowRows wr { context_rows_dev, cache_offset, factor_offset, start_pos_dev, n_tokens };
  const uint32_t max_pos = max_start_pos + n_tokens - 1;
  hipStream_t st = as_stream( stream );
  if ( dt == GH_F32 ) {
    const WindowOut<float> to { static_cast<float*>( out ), out_stride, head_gates, s.heads };
    const float* qf = static_cast<const float*>( q );
    return s.values_are_keys ? attend_rows<float, true>( to, qf, distance_bias_dev, wr, s, rows, max_pos, st )
                             : attend_rows<float, false>( to, qf, distance_bias_dev, wr, s, rows, max_pos, st );
  }
  const WindowOut<__bf16> to { static_cast<__bf16*>( out ), out_stride, head_gates, s.heads };
  const __bf16* qb = static_cast<const __bf16*>( q );
  if ( tiles_applicable( s, distance_bias_dev, n_tokens ) ) {
    return attend_tiles( to, qb, distance_bias_dev, wr, s, batch, st );
  }
  if ( s.dpad <= 128 && s.vpad <= 128 ) {
    return attend_decode( to, qb, distance_bias_dev, wr, s, rows, max_pos, st );
  }
  return s.values_are_keys ? attend_rows<__bf16, true>( to, qb, distance_bias_dev, wr, s, rows, max_pos, st )
                           : attend_rows<__bf16, false>( to, qb, distance_bias_dev, wr, s, rows, max_pos, st );
}

} // extern "C"
