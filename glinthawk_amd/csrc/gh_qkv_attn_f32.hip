// fp32, few and short rows: norm, wq, wk, wv, RoPE, cache append and decode attention of a layer in one launch.
//
// Small models at a handful of contexts are a chain of launches, each bound by being one and by its round trips to memory.  A query head of a context
// needs 3 x head_size of the weight rows, its own cache rows and nothing of any other, so a work-group that makes q, k and v itself can go on to the
// attention: a head's weights are read once per context (from L2, but for the first), which costs less than the launch that it saves while a
// work-group's share is short.  The old keys and values do not depend on the product, so they are requested with the weights, in front of it; that no other
// work-group of the launch writes one of them, i.e. that a context stands in the batch once, is up to the caller.
//
//   work-group  8 waves on one (query head, context); 16 lanes share a row of x, of the weights or of a key, four elements a piece
//   product     a row of lanes takes the weight rows j, j + 32, ... of the head's q | k | v rows, all requested at once
//   attention   a turn is 5 to 8 keys a row of lanes, up to 256 in all; the new key and value come out of LDS and take their place behind the last old one
//
// Bound by what one CU takes in (a head of the 15M model: 166 KB of weights, 56 of keys and values at 150 keys) and by the chain weights, product, scores,
// values.  A row past its end is masked a piece at a time and turns without keys are left out, as instructions count here: 8.7 us with a select an element.
// Two launches / this one, us, in a graph, 6 heads of 48 of 288, 20, 150 and 256 keys: 2 contexts 6.8 7.5 7.9 / 5.6 6.4 7.1, 4 contexts 6.9 7.7 7.9 / 5.7 6.4
// 7.2, 16 contexts 8.3 9.1 9.4 / 5.8 6.6 7.4; a step of the 15M model at 4 contexts 162 / 153.
#include "gh_common.h"

#include <type_traits>

namespace gh {

bool attn_decode_forced(); // gh_attn_decode.hip

namespace {

constexpr float LOG2E = 1.4426950408889634f;
constexpr uint32_t QA_WAVES = 8, QA_GROUPS = QA_WAVES * 4; // rows of 16 lanes
constexpr uint32_t QA_PIECES = 5;                          // of four elements a lane holds of a row of x or of the weights
constexpr uint32_t QA_WIDTH = 64 * QA_PIECES, QA_HEAD = 64;
typedef float f4 __attribute__( ( ext_vector_type( 4 ) ) );
// cache rows come out of a table: the cast names the address space, so that no flat loads are used; offsets in bytes, 32 bits from one base
typedef const __attribute__( ( address_space( 1 ) ) ) char* global_bytes;
typedef const __attribute__( ( address_space( 1 ) ) ) f4* global_f4;
typedef const __attribute__( ( address_space( 1 ) ) ) float* global_f32;
__device__ __forceinline__ f4 load4( global_bytes base, uint32_t at ) { return *(global_f4)( base + at ); }

// R: weight rows of a row of lanes (3 head_size <= 32 R)
template<int R>
__global__ __launch_bounds__( 64 * QA_WAVES ) void qkv_attn_f32_kernel( const float* __restrict__ x,
                                                                       const float* __restrict__ norm,
                                                                       const float* __restrict__ w,
                                                                       const float* const* __restrict__ layer_rows,
                                                                       float* const* __restrict__ token_rows,
                                                                       const uint32_t* __restrict__ pos,
                                                                       const float* __restrict__ freq_real,
                                                                       const float* __restrict__ freq_imag,
                                                                       float* __restrict__ xb,
                                                                       uint32_t s,
                                                                       uint32_t n_kv_heads,
                                                                       uint32_t gqa,
                                                                       uint32_t head_size,
                                                                       uint32_t seq_len,
                                                                       float scale_log2e )
{
  constexpr int P = QA_PIECES, U = R <= 4 ? 8 : R == 5 ? 7 : 5; // keys of a row of lanes at once: what 256 registers hold
  __shared__ __attribute__( ( aligned( 16 ) ) ) float s_qkv[3 * QA_HEAD];
  __shared__ float s_out[QA_WAVES][QA_HEAD], s_m[QA_WAVES], s_l[QA_WAVES];
  const uint32_t head = blockIdx.x, ctx = blockIdx.y, h = head / gqa;
  const uint32_t wave = threadIdx.x >> 6, lane = threadIdx.x & 63, r = lane >> 4, c = lane & 15, group = wave * 4 + r;
  const uint32_t n_heads = n_kv_heads * gqa, dim = n_heads * head_size, kv_dim = n_kv_heads * head_size;
  const float* base = layer_rows[ctx];
  float* appended = token_rows[ctx];
  const uint32_t last = pos[ctx];

  f4 xv[P], gain[P], wv[R][P];
  uint32_t at[P];
#pragma unroll
  for ( int k = 0; k < P; k++ ) {
    at[k] = 4 * min( 4 * ( c + 16 * k ), s - 4 ); // past the row's end: its last elements again, as zeros
    xv[k] = load4( (global_bytes)( x + (uint64_t)ctx * s ), at[k] );
    gain[k] = load4( (global_bytes)norm, at[k] );
  }
#pragma unroll
  for ( int i = 0; i < R; i++ ) {
    const uint32_t j = min( group + QA_GROUPS * i, 3 * head_size - 1 );
    const uint32_t row = j < head_size ? head * head_size + j : j < 2 * head_size ? dim + h * head_size + ( j - head_size ) : dim + kv_dim + h * head_size + ( j - 2 * head_size );
#pragma unroll
    for ( int k = 0; k < P; k++ ) {
      wv[i][k] = load4( (global_bytes)w, row * ( 4 * s ) + at[k] );
    }
  }

  // An empty context has no rows: it goes through the motions and stores nothing.  Without an old key the weights are read in the place of one.
  const bool here = base != nullptr;
  const uint32_t old = here ? min( last, seq_len - 1 ) : 0; // keys in front of the new one
  const global_bytes keys = (global_bytes)( old > 0 ? base + h * head_size : w ), values = keys + 4 * kv_dim;
  const uint32_t d = 4 * c;
  const bool in_head = d < head_size;
  const uint32_t piece = min( d, head_size - 4 );
  const uint32_t freq_at = ( here ? last : 0 ) * ( head_size / 2 ) + piece / 2;
  const float re[2] = { freq_real[freq_at], freq_real[freq_at + 1] }, im[2] = { freq_imag[freq_at], freq_imag[freq_at + 1] };

  auto rest = [&]( auto aligned ) __attribute__( ( always_inline ) ) {
    auto piece_at = [&]( global_bytes p, uint32_t byte ) __attribute__( ( always_inline ) ) {
      if constexpr ( aligned.value ) {
        return load4( p, byte );
      } else {
        const global_f32 one = (global_f32)( p + byte );
        return f4 { one[0], one[1], one[2], one[3] };
      }
    };
    f4 kp[U] = {}, vp[U] = {};
    auto load = [&]( uint32_t t0 ) __attribute__( ( always_inline ) ) {
#pragma unroll
      for ( int u = 0; u < U; u++ ) {
        const uint32_t byte = min( t0 + QA_GROUPS * u + group, max( old, 1u ) - 1 ) * ( 8 * kv_dim ) + 4 * piece;
        if ( u == 0 || t0 + QA_GROUPS * u < old ) { // (uniform; the others have no old key, and are not looked at or are the new one)
          kp[u] = piece_at( keys, byte );
          vp[u] = piece_at( values, byte );
        }
      }
    };
    load( 0 );
    __builtin_amdgcn_sched_barrier( 0 );

    // ---- x normed as rmsnorm does (the mean, the root, one rounding of each product), then this row of lanes' rows of q | k | v
    auto dot4 = []( f4 a, f4 b ) __attribute__( ( always_inline ) ) { return a[0] * b[0] + a[1] * b[1] + a[2] * b[2] + a[3] * b[3]; };
    float ss = 0.0f;
#pragma unroll
    for ( int k = 0; k < P; k++ ) {
      const float sum = dot4( xv[k], xv[k] );
      ss += 4 * ( c + 16 * k ) < s ? sum : 0.0f;
    }
    const float inv_rms = 1.0f / sqrtf( row16_sum( ss ) / (float)s + 1e-5f );
#pragma unroll
    for ( int k = 0; k < P; k++ ) {
#pragma unroll
      for ( int e = 0; e < 4; e++ ) {
        xv[k][e] = gain[k][e] * ( inv_rms * xv[k][e] );
      }
    }
#pragma unroll
    for ( int i = 0; i < R; i++ ) {
      float dot = 0.0f;
#pragma unroll
      for ( int k = 0; k < P; k++ ) {
        const float sum = dot4( wv[i][k], xv[k] );
        dot += 4 * ( c + 16 * k ) < s ? sum : 0.0f;
      }
      dot = row16_sum( dot );
      if ( c == 0 && group + QA_GROUPS * i < 3 * head_size ) {
        s_qkv[group + QA_GROUPS * i] = dot;
      }
    }
    __syncthreads();

    // ---- this lane's piece of the rotated query and key, and of the value
    auto turned = [&]( f4 v ) __attribute__( ( always_inline ) ) {
      return f4 { v[0] * re[0] - v[1] * im[0], v[0] * im[0] + v[1] * re[0], v[2] * re[1] - v[3] * im[1], v[2] * im[1] + v[3] * re[1] };
    };
    const f4 q = turned( *reinterpret_cast<const f4*>( s_qkv + piece ) );
    const f4 k_new = turned( *reinterpret_cast<const f4*>( s_qkv + head_size + piece ) );
    const f4 v_new = *reinterpret_cast<const f4*>( s_qkv + 2 * head_size + piece );
    if ( appended != nullptr && head % gqa == 0 && group == 0 && in_head ) {
      float* row = appended + h * head_size + piece;
      if constexpr ( aligned.value ) {
        *reinterpret_cast<f4*>( row ) = k_new;
        *reinterpret_cast<f4*>( row + kv_dim ) = v_new;
      } else {
#pragma unroll
        for ( int e = 0; e < 4; e++ ) {
          row[e] = k_new[e];
          row[kv_dim + e] = v_new[e];
        }
      }
    }

    // ---- online softmax over the old keys and, behind them, the new one; m: of the wave, l: of this lane's keys
    float acc[4] = { 0.0f, 0.0f, 0.0f, 0.0f }, m = -INFINITY, l = 0.0f;
    auto turn = [&]( uint32_t t0 ) __attribute__( ( always_inline ) ) {
      float sc[U], most = -INFINITY;
#pragma unroll
      for ( int u = 0; u < U; u++ ) {
        const uint32_t key0 = t0 + QA_GROUPS * u, key = key0 + group;
        sc[u] = 0.0f;
        if ( key0 > old ) { // uniform, as the next
          continue;
        }
        if ( old - key0 < QA_GROUPS ) {
#pragma unroll
          for ( int e = 0; e < 4; e++ ) {
            kp[u][e] = key == old ? k_new[e] : kp[u][e];
            vp[u][e] = key == old ? v_new[e] : vp[u][e];
          }
        }
        const float dot = dot4( kp[u], q );
        sc[u] = row16_sum( in_head ? dot : 0.0f ) * scale_log2e;
        most = key <= old ? fmaxf( most, sc[u] ) : most;
      }
      const float m_new = fmaxf( m, fmaxf( fmaxf( lane_value( most, 0 ), lane_value( most, 16 ) ), fmaxf( lane_value( most, 32 ), lane_value( most, 48 ) ) ) );
      const float m_ref = m_new == -INFINITY ? 0.0f : m_new; // a score of -inf weighs 0, also where no finite one came before it
      const float alpha = __builtin_amdgcn_exp2f( m - m_ref );
      l *= alpha;
#pragma unroll
      for ( int e = 0; e < 4; e++ ) {
        acc[e] *= alpha;
      }
#pragma unroll
      for ( int u = 0; u < U; u++ ) {
        const bool in = t0 + QA_GROUPS * u + group <= old;
        if ( t0 + QA_GROUPS * u > old ) {
          continue;
        }
        const float p = in ? __builtin_amdgcn_exp2f( sc[u] - m_ref ) : 0.0f;
        l += p;
#pragma unroll
        for ( int e = 0; e < 4; e++ ) {
          acc[e] += in ? p * vp[u][e] : 0.0f;
        }
      }
      m = m_new;
    };
    turn( 0 );
    for ( uint32_t t0 = QA_GROUPS * U; t0 <= old; t0 += QA_GROUPS * U ) {
      load( t0 );
      turn( t0 );
    }
    // the rows of lanes added up: lane (r, c) ends up with element 4 c + r
    float out = sum_rows( sum_halves( acc[0], acc[2] ), sum_halves( acc[1], acc[3] ) );
    l = ( lane_value( l, 0 ) + lane_value( l, 16 ) ) + ( lane_value( l, 32 ) + lane_value( l, 48 ) );
    s_out[wave][lane] = out;
    if ( lane == 0 ) {
      s_m[wave] = m;
      s_l[wave] = l;
    }
    __syncthreads();
    if ( wave != 0 || !here ) {
      return;
    }
    float m_all = s_m[0];
#pragma unroll
    for ( int v = 1; v < (int)QA_WAVES; v++ ) {
      m_all = fmaxf( m_all, s_m[v] );
    }
    const float m_ref = m_all == -INFINITY ? 0.0f : m_all;
    l = 0.0f, out = 0.0f;
#pragma unroll
    for ( int v = 0; v < (int)QA_WAVES; v++ ) { // a wave without keys: maximum -inf, sums of zero
      const float f = __builtin_amdgcn_exp2f( s_m[v] - m_ref );
      l += s_l[v] * f;
      out += s_out[v][lane] * f;
    }
    const uint32_t element = 4 * c + r;
    if ( element < head_size ) {
      xb[( (uint64_t)ctx * n_heads + head ) * head_size + element] = out * ( 1.0f / l );
    }
  };
  ( ( reinterpret_cast<uintptr_t>( base ) | reinterpret_cast<uintptr_t>( appended ) ) & 15u ) == 0 ? rest( std::true_type {} ) : rest( std::false_type {} );
}

} // namespace
} // namespace gh

using namespace gh;

extern "C" {

// Wider rows or heads and more work-groups than CUs would have a CU take in more than the saved launch is worth.  A single context's product is the
// cheapest as it is (6 heads of 48, 20, 150 and 256 keys: 5.9 6.5 6.7 us as two launches, 5.6 6.3 7.1 as one; 5 of 64: 5.6 6.4 6.8 and 5.8 6.6 7.2): only for heads
// whose share is small (8 of 40 over 4: 5.8 6.5 6.7 and 5.2 6.0 6.5; 4 of 16: 5.6 6.5 6.7 and 4.5 5.2 5.7).
int gh_rmsnorm_qkv_attn_rides( uint64_t b, const gh_shape* shape, gh_dtype dt )
{
  return shape != nullptr && dt == GH_F32 && b > 0 && b <= 65535 && shape->dim <= QA_WIDTH && shape->dim % 4 == 0 && shape->head_size <= QA_HEAD
             && shape->head_size % 4 == 0 && ( b > 1 || shape->head_size <= 40 ) && b * shape->n_heads <= (uint64_t)cu_count()
             && (uint64_t)shape->seq_len * shape->kv_dim <= ( 1ull << 28 ) // (offsets of 32 bits)
           ? 1
           : 0;
}

// The work-group of a (head, context) walks all of its keys, a turn after the other, where the attention by itself cuts them over idle CUs.  Two launches / one, us, in a graph,
// 512, 768, 1024 and 2048 keys: 6 heads of 48, 2 contexts 11.3 11.5 11.7 11.9 / 9.9 11.5 12.9 19.4, 8 contexts 12.8 13.9 15.0 19.0 / 10.1 11.8 13.6 21.2; 5 of 64, 2 contexts 11.0
// 11.7 11.6 11.9 / 10.0 11.5 13.4 19.8; 4 of 16, one context 9.0 8.9 8.9 9.8 / 7.6 8.9 10.1 16.8; 8 of 40 over 8, 16 contexts 16.3 18.7 21.2 31.6 / 11.5 13.9 16.8 27.5.  Up to 512 keys
// one is faster for every shape tried; beyond, it depends on how many CUs the cut would fill.
constexpr uint32_t QA_KEYS = 512;
int gh_rmsnorm_qkv_attn_preferred( uint64_t b, uint32_t max_pos, const gh_shape* shape, gh_dtype dt )
{
  return max_pos < QA_KEYS && !attn_decode_forced() && gh_rmsnorm_qkv_attn_rides( b, shape, dt ) == 1 ? 1 : 0;
}

int gh_rmsnorm_qkv_attn( void* xb, const void* x, const void* norm_weight, const void* wqkv, uint64_t b, const uint32_t* pos_dev, const void* freq_real,
                         const void* freq_imag, const void* const* layer_rows_dev, void* const* token_rows_dev, const gh_shape* shape, gh_dtype dt,
                         gh_stream stream )
{
  if ( int rc = ensure_init() ) {
    return rc;
  }
  if ( b == 0 ) {
    return GH_OK;
  }
  GH_REQUIRE( shape != nullptr && xb && x && norm_weight && wqkv && pos_dev && freq_real && freq_imag && layer_rows_dev && token_rows_dev, "gh_rmsnorm_qkv_attn: NULL pointer" );
  GH_REQUIRE( shape->n_kv_heads > 0 && shape->gqa_size > 0 && shape->head_size > 0 && shape->seq_len > 0, "gh_rmsnorm_qkv_attn: zero dimension" );
  GH_REQUIRE( shape->n_heads == shape->n_kv_heads * shape->gqa_size && shape->kv_dim == shape->n_kv_heads * shape->head_size
                && shape->dim == shape->n_heads * shape->head_size,
              "gh_rmsnorm_qkv_attn: the heads do not make up the dimensions" );
  GH_REQUIRE( gh_rmsnorm_qkv_attn_rides( b, shape, dt ) == 1, "gh_rmsnorm_qkv_attn: no single launch for this shape" );
  GH_REQUIRE( ( ( reinterpret_cast<uintptr_t>( x ) | reinterpret_cast<uintptr_t>( norm_weight ) | reinterpret_cast<uintptr_t>( wqkv ) ) & 15u ) == 0,
              "gh_rmsnorm_qkv_attn: operands not 16-byte aligned" );
  GH_REQUIRE( !overlap( xb, b * shape->dim * sizeof( float ), x, b * shape->dim * sizeof( float ) ), "gh_rmsnorm_qkv_attn: output over the activations" );
  const dim3 grid( shape->n_heads, (unsigned)b );
  const float scale = LOG2E / sqrtf( (float)shape->head_size );
  auto go = [&]( auto rows ) {
    qkv_attn_f32_kernel<decltype( rows )::value><<<grid, 64 * QA_WAVES, 0, as_stream( stream )>>>(
      static_cast<const float*>( x ), static_cast<const float*>( norm_weight ), static_cast<const float*>( wqkv ), reinterpret_cast<const float* const*>( layer_rows_dev ),
      reinterpret_cast<float* const*>( token_rows_dev ), pos_dev, static_cast<const float*>( freq_real ), static_cast<const float*>( freq_imag ), static_cast<float*>( xb ), shape->dim, shape->n_kv_heads,
      shape->gqa_size, shape->head_size, shape->seq_len, scale );
  };
  const uint32_t rows = ( 3 * shape->head_size + QA_GROUPS - 1 ) / QA_GROUPS;
  if ( rows <= 2 ) {
    go( std::integral_constant<int, 2> {} );
  } else if ( rows <= 4 ) {
    go( std::integral_constant<int, 4> {} );
  } else if ( rows == 5 ) {
    go( std::integral_constant<int, 5> {} );
  } else {
    go( std::integral_constant<int, 6> {} );
  }
  GH_LAUNCH_CHECK();
  return GH_OK;
}

} // extern "C"
