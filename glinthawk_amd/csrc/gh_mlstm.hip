// Matrix-memory LSTM (the mLSTM of xLSTM: Beck et al., "xLSTM: Extended Long Short-Term Memory"): exponential input gate and sigmoid
// forget gate in log space with a running maximum m (starting at 0), a matrix S and a vector n per head.
//
//   m' = max(f + m, i);  S' = e^(f + m - m') S + e^(i - m') k v^T;  n' likewise with k;  o = S'^T q / (max(|n' . q|, e^(-m')) + 1e-6)
//
// gates   i = cap tanh((. + b) / cap), f = logsigmoid(cap tanh((. + b) / cap))
// state   fp32, per context and head: S (dim x vdim_padded), then n (heads x dim), then m (heads); zero at position 0, which the kernels
//         take from the position (a slot that is used again needs no clearing)
// walk    work-group = 64 columns of v of one (context, head); it keeps its (dim x 64) part of S in registers over all the tokens of the
//         call (one for decode) and streams it in and out of memory once.  n and m are needed by every column slice: each slice carries
//         its own copy and the finishing kernel writes them back, so no slice reads what another one has already replaced.
//         Bound by the state, read and written once.  Decode of 32 contexts with 8 heads of 256 x 512 (268 MB): 53.8 -> 49.5 us, 5.4 TB/s, with the slices
//         of a head on one XCD and stores that pass the cache by; that order alone 85 -> 76 us for the whole call, those stores alone 76, both 75; 8
//         contexts 31 -> 29, 32 and 28; 64 contexts 139 -> 131, 135 and 132; 13 contexts 42 -> 40, 40 and 36.  Loads past the cache lose (64: 171).
// finish  one work-group per token: each head's output divided by its root mean square, times a weight, times sigmoid(g)
#include "gh_product.h"

#include <algorithm>
#include <type_traits>

namespace gh {
namespace {

constexpr uint32_t SLICE = 64;          // columns of v per work-group
typedef float f4 __attribute__( ( ext_vector_type( 4 ) ) );
constexpr uint32_t CHUNKED_TOKENS = 24; // from this many tokens per context on, bf16 runs in chunks on the matrix cores

struct MlstmShape
{
  uint32_t heads, dim, vdim, vpad;
  float cap, eps, q_scale;
  // elements of the state of one context
  __host__ __device__ uint64_t n_off() const { return (uint64_t)heads * dim * vpad; }
  __host__ __device__ uint64_t m_off() const { return n_off() + (uint64_t)heads * dim; }
  __host__ __device__ uint64_t elements() const { return m_off() + heads; }
};

__device__ __forceinline__ float soft_cap( float z, float cap ) { return cap * tanhf( z / cap ); }
// log(sigmoid(z)), stable for either sign
__device__ __forceinline__ float log_sigmoid( float z ) { return fminf( z, 0.0f ) - log1pf( expf( -fabsf( z ) ) ); }

// columns of the products: [q | k | v | g] in one, [i | f] in the other
struct MlstmCols
{
  uint32_t q, k, v, g, i, f;
};

// the gates as their product left them
template<typename E>
struct MlstmGates
{
  ProductView<float> y;
  MlstmCols col;
  const E *bias_i, *bias_f;
  float cap;
  __device__ __forceinline__ float log_input( float z, uint32_t h ) const { return soft_cap( z + ( bias_i != nullptr ? to_f32( bias_i[h] ) : 0.0f ), cap ); }
  __device__ __forceinline__ float log_forget( float z, uint32_t h ) const
  {
    return log_sigmoid( soft_cap( z + ( bias_f != nullptr ? to_f32( bias_f[h] ) : 0.0f ), cap ) );
  }
};

// `gates`: (rows, 2 heads) fp32, the log input gates of a token's heads, then its log forget gates (mlstm_gates_kernel); NULL: the kernel makes them itself
template<typename E, typename View>
struct MlstmIn
{
  View main;
  const float* gates;
  MlstmCols col;
};

template<typename E>
__global__ __launch_bounds__( 256 ) void mlstm_gates_kernel( float* __restrict__ out,
                                                             MlstmGates<E> in,
                                                             uint32_t heads,
                                                             uint64_t rows )
{
  const uint64_t total = rows * 2 * heads, stride = (uint64_t)gridDim.x * blockDim.x;
  for ( uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < total; i += stride ) {
    const uint64_t row = i / ( 2 * heads );
    const uint32_t g = (uint32_t)( i % ( 2 * heads ) );
    out[i] = g < heads ? in.log_input( in.y.at( row, in.col.i + g ), g ) : in.log_forget( in.y.at( row, in.col.f + g - heads ), g - heads );
  }
}

struct MlstmState
{
  void* const* rows;         // state region of each context; NULL: no context
  uint64_t offset;           // bytes from there to this layer's state
  const uint32_t* start_pos; // position of the first token of the call
  uint32_t n_tokens;
};

// RPT: rows of S per thread kept in registers (0: S stays in memory, any dim)
template<typename E, typename View, int RPT>
__global__ __launch_bounds__( 256 ) void mlstm_walk_kernel( float* __restrict__ o_out, float* __restrict__ nm_out, MlstmIn<E, View> in, MlstmGates<E> raw, MlstmState st, MlstmShape s )
{
  extern __shared__ float lds[];
  __shared__ float g_s[2];        // the gates of one token
  const uint32_t dim4 = ( s.dim + 3 ) / 4 * 4; // v_s and red are read as float4
  float* q_s = lds;               // dim
  float* k_s = q_s + dim4;        // dim
  float* n_s = k_s + dim4;        // dim
  float* v_s = n_s + s.dim;       // SLICE
  float* nq_s = v_s + SLICE;      // 16
  float* red = nq_s + 16;         // 16 x SLICE
  uint32_t slice = blockIdx.x, h = blockIdx.y, ctx = blockIdx.z;
  // The slices of a (context, head) on one XCD, as far as there are eight pairs for eight XCDs: together they are whole rows of S, that is whole pages,
  // and one L2 holds q, k and n of the head.
  const uint32_t slices = gridDim.x, pairs = gridDim.y * gridDim.z, id = ( ctx * gridDim.y + h ) * slices + slice;
  if ( (uint64_t)pairs * slices <= UINT32_MAX && id < ( pairs & ~7u ) * slices ) {
    const uint32_t nth = id >> 3, pair = nth / slices * 8 + ( id & 7 );
    slice = nth % slices;
    h = pair % gridDim.y;
    ctx = pair / gridDim.y;
  }
  uint8_t* base = static_cast<uint8_t*>( st.rows[ctx] );
  if ( base == nullptr ) {
    return;
  }
  float* S = reinterpret_cast<float*>( base + st.offset );
  const float* n_in = S + s.n_off() + (uint64_t)h * s.dim;
  const float* m_in = S + s.m_off() + h;
  S += (uint64_t)h * s.dim * s.vpad;
  const bool fresh = st.start_pos[ctx] == 0;
  const uint32_t t = threadIdx.x;
  const uint32_t cl = t & 15, rg = t >> 4;
  const uint32_t c0 = slice * SLICE + cl * 4;
  const bool col_live = c0 < s.vpad;
  // The gates' sums, a K range a lane (the input gate's in the lower half of the wave), requested in front of the state: one token of a context
  float gate_part = 0.0f;
  if ( in.gates == nullptr && t < WAVE ) {
    const uint32_t k = t & 31;
    const float* sums = raw.y.data + ctx * raw.y.stride + ( ( t & 32 ) == 0 ? raw.col.i : raw.col.f ) + h;
    gate_part = k < raw.y.planes() ? sums[k * raw.y.plane] : 0.0f;
    for ( uint32_t more = k + 32; more < raw.y.planes(); more += 32 ) {
      gate_part += sums[more * raw.y.plane];
    }
  }
  constexpr int R = RPT > 0 ? RPT : 1;
  float4 reg[R];
  if constexpr ( RPT > 0 ) {
#pragma unroll
    for ( int r = 0; r < RPT; r++ ) {
      const uint32_t row = rg + 16 * r;
      reg[r] = make_float4( 0.0f, 0.0f, 0.0f, 0.0f );
      if ( !fresh && row < s.dim && col_live ) {
        reg[r] = *reinterpret_cast<const float4*>( S + (uint64_t)row * s.vpad + c0 );
      }
    }
  } else if ( fresh && col_live ) {
    for ( uint32_t row = rg; row < s.dim; row += 16 ) {
      *reinterpret_cast<float4*>( S + (uint64_t)row * s.vpad + c0 ) = make_float4( 0.0f, 0.0f, 0.0f, 0.0f );
    }
  }
  gate_part = row16_sum( gate_part );
  for ( uint32_t d = t; d < s.dim; d += 256 ) {
    n_s[d] = fresh ? 0.0f : n_in[d];
  }
  float m = fresh ? 0.0f : *m_in;

  for ( uint32_t tok = 0; tok < st.n_tokens; tok++ ) {
    const uint64_t row_in = (uint64_t)ctx * st.n_tokens + tok;
    __syncthreads(); // the previous token's readers are done (and n_s is written)
    for ( uint32_t d = t; d < s.dim; d += 256 ) {
      q_s[d] = in.main.at( row_in, in.col.q + h * s.dim + d ) * s.q_scale;
      k_s[d] = in.main.at( row_in, in.col.k + h * s.dim + d );
    }
    if ( t < SLICE ) {
      const uint32_t c = slice * SLICE + t;
      v_s[t] = c < s.vdim ? in.main.at( row_in, in.col.v + h * s.vdim + c ) : 0.0f;
    }
    float gi = 0.0f, gf = 0.0f;
    if ( in.gates != nullptr ) {
      gi = in.gates[row_in * 2 * s.heads + h];
      gf = in.gates[( row_in * 2 + 1 ) * s.heads + h];
    } else if ( t < WAVE ) { // one wave for all: some 200 instructions
      g_s[0] = raw.log_input( lane_value( gate_part, 0 ) + lane_value( gate_part, 16 ), h );
      g_s[1] = raw.log_forget( lane_value( gate_part, 32 ) + lane_value( gate_part, 48 ), h );
    }
    __syncthreads();
    if ( in.gates == nullptr ) {
      gi = g_s[0], gf = g_s[1];
    }
    const float m_new = fmaxf( gf + m, gi );
    const float decay = expf( gf + m - m_new ), inp = expf( gi - m_new );
    m = m_new;
    const float4 v4 = *reinterpret_cast<const float4*>( v_s + cl * 4 );
    float4 acc = make_float4( 0.0f, 0.0f, 0.0f, 0.0f );
    auto row_step = [&]( float4& x, uint32_t row ) {
      const float kk = inp * k_s[row], qq = q_s[row];
      x.x = decay * x.x + kk * v4.x;
      x.y = decay * x.y + kk * v4.y;
      x.z = decay * x.z + kk * v4.z;
      x.w = decay * x.w + kk * v4.w;
      acc.x += qq * x.x;
      acc.y += qq * x.y;
      acc.z += qq * x.z;
      acc.w += qq * x.w;
    };
    if constexpr ( RPT > 0 ) {
#pragma unroll
      for ( int r = 0; r < RPT; r++ ) {
        const uint32_t row = rg + 16 * r;
        if ( row < s.dim ) {
          row_step( reg[r], row );
        }
      }
    } else if ( col_live ) {
      for ( uint32_t row = rg; row < s.dim; row += 16 ) {
        float4* p = reinterpret_cast<float4*>( S + (uint64_t)row * s.vpad + c0 );
        float4 x = *p;
        row_step( x, row );
        *p = x;
      }
    }
    // n: one owner per element; its product with q by the sixteen row groups
    float nq = 0.0f;
    for ( uint32_t row = rg + 16 * cl; row < s.dim; row += 256 ) {
      const float x = decay * n_s[row] + inp * k_s[row];
      n_s[row] = x;
      nq += x * q_s[row];
    }
    nq = row16_sum( nq );
    if ( cl == 0 ) {
      nq_s[rg] = nq;
    }
    *reinterpret_cast<float4*>( red + rg * SLICE + cl * 4 ) = acc;
    __syncthreads();
    if ( t < SLICE && slice * SLICE + t < s.vdim ) {
      float num = 0.0f, den = 0.0f;
#pragma unroll
      for ( int r = 0; r < 16; r++ ) {
        num += red[r * SLICE + t];
        den += nq_s[r];
      }
      o_out[row_in * s.heads * s.vdim + h * s.vdim + slice * SLICE + t] = num / ( fmaxf( fabsf( den ), expf( -m ) ) + 1e-6f );
    }
  }
  if constexpr ( RPT > 0 ) {
#pragma unroll
    for ( int r = 0; r < RPT; r++ ) {
      const uint32_t row = rg + 16 * r;
      if ( row < s.dim && col_live ) {
        __builtin_nontemporal_store( f4 { reg[r].x, reg[r].y, reg[r].z, reg[r].w }, reinterpret_cast<f4*>( S + (uint64_t)row * s.vpad + c0 ) );
      }
    }
  }
  if ( slice == 0 ) {
    float* dst = nm_out + ( (uint64_t)ctx * s.heads + h ) * ( s.dim + 1 );
    for ( uint32_t row = t; row < s.dim; row += 256 ) { // (the owners wrote before the last barrier)
      dst[row] = n_s[row];
    }
    if ( t == 0 ) {
      dst[s.dim] = m;
    }
  }
}

// ---- many tokens: chunks of 64 on the matrix cores (bf16 products) -------------------------------------------------------------
//
// With b_t the sum of the log forget gates of the chunk up to token t, c_s = i_s - b_s and M_t = max(m0, c_1 .. c_t) (m0: the running
// maximum in front of the chunk), the recurrence unrolls to m_t = b_t + M_t and
//
//   S_t = e^(m0 - M_t) S_0 + sum_(s <= t) e^(c_s - M_t) k_s v_s^T                      (n_t likewise)
//   o_t = (e^(m0 - M_t) S_0^T q_t + sum_(s <= t) e^(c_s - M_t) (k_s . q_t) v_s) / (max(|n_t . q_t|, e^(-m_t)) + 1e-6)
//
// Three kernels:
//   scan    the gates, b, c and M of every token, a work-group for a (context, head), a wave for a chunk
//   scores  a work-group for a chunk: the weights of the keys P[t][s] = e^(c_s - M_t) (k_s . q_t), their sums over s, and what the chunk
//           adds to n.  They do not depend on v: made here once instead of by all the columns of v.
//   states  4 waves on one (context, head, 64 columns of v) walk the chunks, O = a Q S + P V, then S = decay S + K^T (w V); a wave owns
//           16 columns, its part of S (dim x 16, fp32) stays in accumulator registers from the first chunk to the last.  Two work-groups
//           per CU: two waves a SIMD cover each other's reads of LDS and waits.
//           n is carried by every slice of the columns, a thread an element; each makes the denominators of its share of the tokens.
// exactness   q, k, v are bf16 already.  What enters the state (the weighted values) meets k as three bf16 terms, 24 bits: the state's sums are
//             those of fp32 operands at the rate of bf16 matrix instructions.  What is read out of it for the output (S, the weights of
//             the keys) meets q and v as two terms, 16 bits.  n and its products are fp32.
// loads       k of a chunk is requested at its head and needed behind Q S and P V; q and v of the next one are requested behind those and needed
//             at the next one's head.
// order       of the sums: terms of 16 keys or dims at a time, the lower term first, as v_mfma_f32_32x32x16_bf16 takes them (eight of a lane, lanes 0 .. 31 in
//             front).  v_mfma_f32_16x16x32_bf16 is two of those in turn, bit for bit, so its lanes 32 .. 63 hold the next term of the same 16, or the first of the
//             next, instead of 16 others: permlane32_swap brings a lane's terms there.  Models depend on the last bits (behind a thousand tokens and two
//             layers they are more than a tenth of the logits of 3 tokens in 960, in either order as far off 64 bits), so the order is kept whatever the tile.
// operands    an accumulator tile of v_mfma_f32_16x16x32_bf16 (lane = column, registers = rows 4 (lane / 16) + v) is, with the tile of the next quads,
//             an operand of the next product over those rows when the other operand takes its rows in the same order:
//               scores^T = K Q^T        lane = query, registers = keys   -> left operand of   P V     (V out of LDS transposed)
//               S                       lane = column of v, registers = dim -> right operand of Q S   (Q out of LDS in pieces of 4)
//             S += K^T (w V): both operands out of LDS with transposing reads (ds_read_b64_tr_b16).
// LDS         64 rows each of q, k and v, 16-byte chunks XORed with bits of the row so that row reads (16 rows) and transposing reads (8 rows, two chunks
//             each) both touch every bank once; straight from memory (buffer_load ... lds; rows past the sequence and padding read as zero).
// bound       8 contexts of 1024 tokens, 8 heads of 256 x 512: 310 us in one kernel, whose waves, one a SIMD, made gates, weights and n once for every 32
//             columns; now, in a prefill, scan 10, scores 24 and states 162 us (calls in a row 391 -> 293, with scores of 15, whose q and k the last call left in
//             the caches; 1 of 2048 tokens 528 -> 230, 32 of 24 tokens 117 -> 83).  States: waits of four waves for each other, twice a chunk, and for LDS, 330 reads a chunk and wave, with two waves a SIMD; the matrix cores are busy for a quarter of it.
//             With 32 keys or dims of one term in a product, whose bits differ: 200 reads fewer and 129 us.  A third operand of k out of LDS instead of one
//             selected from two: 235 us at 1 x 2048 tokens instead of 230, 8 x 1024 even.
constexpr int CHUNK = 64;
typedef __attribute__( ( address_space( 3 ) ) ) void* lds_ptr;
typedef __attribute__( ( address_space( 3 ) ) ) char lds_char;
typedef short v4s __attribute__( ( ext_vector_type( 4 ) ) );
typedef __attribute__( ( address_space( 3 ) ) ) v4s* lds_v4s;
typedef Mfma<__bf16>::x8 bf16x8;

// slot of 16-byte chunk `chunk` of row `row` in a tile of `BYTES` a row, 128, 256 or 512: eight rows in a row and those `FAR` further on apart
template<uint32_t BYTES, uint32_t FAR = 8>
__device__ __forceinline__ uint32_t swizzle( uint32_t row, uint32_t chunk )
{
  return BYTES == 128 ? chunk ^ ( ( ( ( row >> 1 ) & 3 ) << 1 ) | ( ( row / FAR ) & 1 ) ) : chunk ^ ( ( ( row & 7 ) << 1 ) | ( ( row / FAR ) & 1 ) );
}
// eight rows in a row and a chunk and the next but one apart
template<uint32_t BYTES>
__device__ __forceinline__ uint32_t swizzle_pair( uint32_t row, uint32_t chunk )
{
  return BYTES == 128 ? chunk ^ ( ( ( row >> 1 ) & 1 ) | ( row & 4 ) ) : chunk ^ ( ( row & 1 ) | ( ( row & 6 ) << 1 ) );
}

// Eight fp32 values as N bf16 terms each, 8 bits of mantissa a term; taken two at a time, as the conversion instruction does.
typedef float f32x2 __attribute__( ( ext_vector_type( 2 ) ) );
typedef __bf16 bf16x2 __attribute__( ( ext_vector_type( 2 ) ) );
template<int N>
struct Split
{
  union
  {
    bf16x2 pair[4];
    bf16x8 x;
  } t[N];
  __device__ __forceinline__ void set( int k, float x0, float x1 ) // elements 2 k, 2 k + 1
  {
#pragma unroll
    for ( int n = 0; n < N; n++ ) {
      const bf16x2 b = __builtin_convertvector( ( f32x2 { x0, x1 } ), bf16x2 );
      t[n].pair[k] = b;
      x0 -= (float)b[0];
      x1 -= (float)b[1];
    }
  }
};
__device__ __forceinline__ double shfl_up_f64( double v, int by )
{
  const uint64_t bits = __builtin_bit_cast( uint64_t, v );
  const uint32_t lo = __shfl_up( (uint32_t)bits, by ), hi = __shfl_up( (uint32_t)( bits >> 32 ), by );
  return __builtin_bit_cast( double, ( (uint64_t)hi << 32 ) | lo );
}
__device__ __forceinline__ double last_lane_f64( double v )
{
  const uint64_t bits = __builtin_bit_cast( uint64_t, v );
  const uint32_t lo = __builtin_amdgcn_readlane( (uint32_t)bits, 63 ), hi = __builtin_amdgcn_readlane( (uint32_t)( bits >> 32 ), 63 );
  return __builtin_bit_cast( double, ( (uint64_t)hi << 32 ) | lo );
}

// What the three kernels and the finishing one hand on, by (context, head) = pair.
struct MlstmChunks
{
  float* token;   // planes of (pairs, chunks x 64): see below
  float* decay;   // (pairs, chunks): factor of the state over a chunk
  float* n;       // (pairs, chunks, dim): what a chunk adds to n
  uint4* weights; // (pairs, chunks, WEIGHT_TILES, 64 lanes): P as the left operands of P V
  uint32_t chunks;
  uint64_t plane;
  enum
  {
    C,     // c_s - M of the chunk's last token; -inf past the sequence
    W,     // e to the power of it
    A,     // factor of the state in front of the chunk
    M,     // M_t - M of the chunk's last token
    FLOOR, // e^(-m_t)
    DEN,   // sum of the weights of the keys
    OVER,  // 1 / denominator
    PLANES
  };
  __device__ __forceinline__ float* tokens( int which, uint32_t pair, uint32_t chunk ) const { return token + which * plane + ( (uint64_t)pair * chunks + chunk ) * CHUNK; }
};
constexpr uint32_t WEIGHT_TILES = 10; // 16 queries x 16 keys, both terms, up to the queries' own
__device__ __forceinline__ constexpr uint32_t weight_tile( uint32_t queries, uint32_t keys ) { return queries * ( queries + 1 ) / 2 + keys; }

// Lanes 0 .. 31 of both operands in the first, lanes 32 .. 63 of both in the second: [a | A], [b | B] -> [a | b], [A | B]
__device__ __forceinline__ void swap_halves( bf16x8& first, bf16x8& second )
{
  typedef uint32_t u32x4_t __attribute__( ( ext_vector_type( 4 ) ) );
  u32x4_t a = __builtin_bit_cast( u32x4_t, first ), b = __builtin_bit_cast( u32x4_t, second );
#pragma unroll
  for ( int k = 0; k < 4; k++ ) {
    const auto ab = __builtin_amdgcn_permlane32_swap( a[k], b[k], false, false );
    a[k] = ab[0], b[k] = ab[1];
  }
  first = __builtin_bit_cast( bf16x8, a ), second = __builtin_bit_cast( bf16x8, b );
}

// The tokens of a chunk, lane <-> token: the sums b of the log forget gates, c, and the largest c so far (without what lies in front of the chunk).
struct ChunkScan
{
  double b, c, M;
  bool live;
  __device__ __forceinline__ ChunkScan( const MlstmGates<__bf16>& in, const MlstmState& st, uint32_t ctx, uint32_t h, uint32_t tok, uint32_t lane )
  {
    live = tok < st.n_tokens;
    const uint64_t row = (uint64_t)ctx * st.n_tokens + ( live ? tok : 0 );
    const float gi = in.log_input( in.y.at( row, in.col.i + h ), h ), gf = in.log_forget( in.y.at( row, in.col.f + h ), h );
    b = live ? (double)gf : 0.0;
#pragma unroll
    for ( int by = 1; by < 64; by *= 2 ) {
      const double up = shfl_up_f64( b, by );
      b += (int)lane >= by ? up : 0.0;
    }
    c = live ? (double)gi - b : -1e300;
    M = c;
#pragma unroll
    for ( int by = 1; by < 64; by *= 2 ) {
      const double up = shfl_up_f64( M, by );
      M = (int)lane >= by && up > M ? up : M;
    }
  }
  // what the other kernels take, with the running maximum in front of the chunk
  __device__ __forceinline__ void finish( const MlstmChunks& out, uint32_t pair, uint32_t chunk, uint32_t lane, double before, float& c_rel, float& w, float& M_rel )
  {
    M = before > M ? before : M;
    const double M_end = last_lane_f64( M );
    c_rel = live ? (float)( c - M_end ) : -INFINITY;
    w = expf( c_rel );
    M_rel = (float)( M - M_end );
    out.tokens( MlstmChunks::C, pair, chunk )[lane] = c_rel;
    out.tokens( MlstmChunks::W, pair, chunk )[lane] = w;
    out.tokens( MlstmChunks::A, pair, chunk )[lane] = expf( (float)( before - M ) );
    out.tokens( MlstmChunks::M, pair, chunk )[lane] = M_rel;
    out.tokens( MlstmChunks::FLOOR, pair, chunk )[lane] = expf( -(float)( b + M ) );
    if ( lane == 0 ) {
      out.decay[(uint64_t)pair * out.chunks + chunk] = expf( (float)( before - M_end ) );
    }
  }
};
__device__ __forceinline__ double max_in_front( const uint8_t* base, const MlstmState& st, const MlstmShape& s, uint32_t ctx, uint32_t h )
{
  return st.start_pos[ctx] == 0 ? 0.0 : (double)reinterpret_cast<const float*>( base + st.offset )[s.m_off() + h];
}

// work-group <-> (head, context), wave <-> chunk, lane <-> token
__global__ __launch_bounds__( 1024 ) void mlstm_scan_kernel( float* __restrict__ nm_out, MlstmGates<__bf16> in, MlstmState st, MlstmShape s, MlstmChunks out )
{
  __shared__ double s_b[16], s_M[16]; // of a chunk: sum of its log forget gates, largest c without what lies in front of it
  const uint32_t h = blockIdx.x, ctx = blockIdx.y, pair = ctx * s.heads + h;
  const uint8_t* base = static_cast<const uint8_t*>( st.rows[ctx] );
  if ( base == nullptr ) {
    return;
  }
  const uint32_t wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  double m0 = max_in_front( base, st, s, ctx, h );
  for ( uint32_t c0 = 0; c0 < out.chunks; c0 += 16 ) {
    const uint32_t chunk = c0 + wave;
    ChunkScan scan( in, st, ctx, h, chunk * CHUNK + lane, lane );
    __syncthreads(); // everyone has read the last sixteen chunks'
    if ( lane == 63 ) {
      s_b[wave] = scan.b;
      s_M[wave] = scan.M;
    }
    __syncthreads();
    double before = m0; // running maximum in front of this wave's chunk
#pragma unroll
    for ( uint32_t k = 0; k < 16; k++ ) { // (chunks past the last: nothing to add, nothing as large)
      before = k == wave ? m0 : before;
      m0 = s_b[k] + ( s_M[k] > m0 ? s_M[k] : m0 );
    }
    if ( chunk < out.chunks ) {
      float c_rel, w, M_rel;
      scan.finish( out, pair, chunk, lane, before, c_rel, w, M_rel );
    }
  }
  if ( threadIdx.x == 0 ) {
    nm_out[(uint64_t)pair * ( s.dim + 1 ) + s.dim] = (float)m0;
  }
}

// work-group <-> chunk of a (context, head), wave <-> 16 queries.  KS: steps of 32 of dim.  dim % 8 == 0, 16-byte aligned product rows.
// ALONE: the call has one chunk, whose gates the work-group scans itself beside its loads, without a launch in front (2 contexts of 24 tokens, 4 heads of 64:
// 27.2 -> 22.5 us for the call; 16 of 64 tokens, 4 heads of 128 x 256: 36.9 -> 31.5).
template<int KS, bool ALONE>
__global__ __launch_bounds__( 256 ) void mlstm_scores_kernel( float* __restrict__ nm_out, MlstmIn<__bf16, ProductView<__bf16>> in, MlstmGates<__bf16> raw, MlstmState st, MlstmShape s,
                                                              MlstmChunks ch, uint32_t n_pairs )
{
  constexpr uint32_t PIECES = 4 * KS; // 8 dims each
  constexpr uint32_t RB = KS * 64;                         // bytes of a row in LDS
  __shared__ uint4 s_k[CHUNK * RB / 16]; // then the sums for n of eight keys each
  __shared__ __attribute__( ( aligned( 16 ) ) ) float s_c[CHUNK], s_w[CHUNK], s_M[CHUNK];
  // on the XCD that walks the chunks
  const uint32_t pair = ( blockIdx.x >> 3 ) / ch.chunks * 8 + ( blockIdx.x & 7 ), chunk = ( blockIdx.x >> 3 ) % ch.chunks;
  if ( pair >= n_pairs ) {
    return;
  }
  const uint32_t h = pair % s.heads, ctx = pair / s.heads;
  const uint8_t* base = static_cast<const uint8_t*>( st.rows[ctx] );
  if ( base == nullptr ) {
    return;
  }
  const uint32_t wave = __builtin_amdgcn_readfirstlane( threadIdx.x >> 6 ), lane = threadIdx.x & 63, r = lane & 15, g = lane >> 4;
  const uint32_t rows = min( (uint32_t)CHUNK, st.n_tokens - chunk * CHUNK );
  const uint32_t ld_bytes = (uint32_t)( in.main.stride * 2 );
  const __bf16* first = in.main.data + ( (uint64_t)ctx * st.n_tokens + chunk * CHUNK ) * in.main.stride;
  const int bytes = (int)( ( rows - 1 ) * ld_bytes + s.dim * 2 ); // rows past the sequence read as zero
  const __amdgpu_buffer_rsrc_t q_rsrc = __builtin_amdgcn_make_buffer_rsrc( const_cast<__bf16*>( first + in.col.q + h * s.dim ), 0, bytes, 0x00020000 );
  const __amdgpu_buffer_rsrc_t k_rsrc = __builtin_amdgcn_make_buffer_rsrc( const_cast<__bf16*>( first + in.col.k + h * s.dim ), 0, bytes, 0x00020000 );
  constexpr uint32_t PAST_THE_END = 0x80000000u; // an offset beyond any descriptor
  typedef uint32_t u32x4_t __attribute__( ( ext_vector_type( 4 ) ) );
  bf16x8 qb[KS];
#pragma unroll
  for ( int k = 0; k < KS; k++ ) {
    qb[k] = __builtin_bit_cast( bf16x8, (u32x4_t)__builtin_amdgcn_raw_buffer_load_b128( q_rsrc, ( 4 * k + g ) * 8 < s.dim ? ( 16 * wave + r ) * ld_bytes + ( 4 * k + g ) * 16 : PAST_THE_END, 0, 0 ) );
  }
  constexpr uint32_t ROWS = 1024 / RB; // rows of one instruction of one wave
#pragma unroll
  for ( uint32_t i = 0; i < CHUNK / ( 4 * ROWS ); i++ ) {
    const uint32_t row0 = ( 4 * i + wave ) * ROWS, row = row0 + lane / PIECES, piece = swizzle<RB, 32>( row, lane % PIECES );
    __builtin_amdgcn_raw_ptr_buffer_load_lds( k_rsrc, (lds_ptr)( s_k + row0 * PIECES ), 16, piece * 8 < s.dim ? row * ld_bytes + piece * 16 : PAST_THE_END, 0, 0, 0 );
  }
  auto k_at = [&]( uint32_t row, uint32_t piece ) __attribute__( ( always_inline ) ) { return __builtin_bit_cast( bf16x8, s_k[row * PIECES + swizzle<RB, 32>( row, piece )] ); };
  if ( wave == 0 ) {
    float c_rel, w, M_rel;
    if constexpr ( ALONE ) {
      ChunkScan scan( raw, st, ctx, h, lane, lane );
      scan.finish( ch, pair, 0, lane, max_in_front( base, st, s, ctx, h ), c_rel, w, M_rel );
      if ( lane == 63 ) {
        nm_out[(uint64_t)pair * ( s.dim + 1 ) + s.dim] = (float)( scan.b + scan.M );
      }
    } else {
      c_rel = ch.tokens( MlstmChunks::C, pair, chunk )[lane], w = ch.tokens( MlstmChunks::W, pair, chunk )[lane], M_rel = ch.tokens( MlstmChunks::M, pair, chunk )[lane];
    }
    s_c[lane] = c_rel, s_w[lane] = w, s_M[lane] = M_rel;
  }
  __builtin_amdgcn_s_waitcnt( 0x0F70 ); // vmcnt(0): this wave's part of k has landed
  __syncthreads();
  const float Mq = s_M[16 * wave + r];
  // lane group g: keys 32 (g / 2) + 8 kt + 4 (g % 2) + e
  const uint32_t key_l = 32 * ( g >> 1 ) + 4 * ( g & 1 ), key_r = 32 * ( r >> 3 ) + 4 * ( ( r >> 2 ) & 1 ) + ( r & 3 ), query = 16 * wave + r;
  float dot[4][4], weight[4][4], p[4][4];
#pragma unroll
  for ( uint32_t kt = 0; kt < 4; kt++ ) {
#pragma unroll
    for ( int e = 0; e < 4; e++ ) {
      dot[kt][e] = weight[kt][e] = p[kt][e] = 0.0f;
    }
    if ( wave > 0 || kt < 2 ) { // (the first 16 queries see none of the others' keys)
      mfma_f32x4 sc = { 0, 0, 0, 0 };
#pragma unroll
      for ( int k = 0; k < KS; k++ ) {
        sc = Mfma<__bf16>::k32( k_at( key_r + 8 * kt, 4 * k + g ), qb[k], sc );
      }
      const float4 ck = *reinterpret_cast<const float4*>( &s_c[key_l + 8 * kt] );
      const float cks[4] = { ck.x, ck.y, ck.z, ck.w };
#pragma unroll
      for ( int e = 0; e < 4; e++ ) {
        dot[kt][e] = sc[e] * s.q_scale, weight[kt][e] = __expf( cks[e] - Mq );
        p[kt][e] = key_l + 8 * kt + e <= query ? dot[kt][e] * weight[kt][e] : 0.0f;
      }
    }
  }
  // their sum, the quads of keys of an even number and those of an odd one each in their order: lanes 32 further on go on from where these end
  float den = 0.0f;
#pragma unroll
  for ( int k = 0; k < 16; k++ ) { // (the last 32 queries see all of the first 32 keys)
    den = wave >= 2 ? __builtin_fmaf( dot[k / 4][k % 4], weight[k / 4][k % 4], den ) : den + p[k / 4][k % 4];
  }
  den = __shfl_xor( den, 32 );
#pragma unroll
  for ( int k = 0; k < 16; k++ ) {
    den += p[k / 4][k % 4];
  }
  den += __shfl_xor( den, 16 );
  if ( g == 2 ) {
    ch.tokens( MlstmChunks::DEN, pair, chunk )[query] = den;
  }
  // as operands: the lower term of 16 keys in lanes 0 .. 31, the upper one of the same keys in the others
  uint4* dst = ch.weights + ( (uint64_t)pair * ch.chunks + chunk ) * ( WEIGHT_TILES * 64 ) + lane;
#pragma unroll
  for ( uint32_t j = 0; j < 2; j++ ) {
    Split<2> f;
#pragma unroll
    for ( int k = 0; k < 4; k++ ) {
      f.set( k, p[2 * j + ( k >> 1 )][2 * ( k & 1 )], p[2 * j + ( k >> 1 )][2 * ( k & 1 ) + 1] );
    }
    swap_halves( f.t[1].x, f.t[0].x );
#pragma unroll
    for ( uint32_t n = 0; n < 2; n++ ) { // keys 32 n + 16 j ..
      if ( 2 * n + j <= wave ) {
        dst[weight_tile( wave, 2 * n + j ) * 64] = __builtin_bit_cast( uint4, f.t[1 - n].x );
      }
    }
  }
  // what the chunk adds to n: eight keys and eight dims a thread
  const uint32_t piece = threadIdx.x % PIECES, set = threadIdx.x / PIECES;
  float sum[8];
  if ( set < 8 ) { // of the quads 4 (set / 2) + set % 2 and the next but one
    const uint32_t key0 = 16 * ( set >> 1 ) + 4 * ( set & 1 );
    bf16x8 k[8];
#pragma unroll
    for ( int i = 0; i < 8; i++ ) {
      k[i] = k_at( key0 + i + 4 * ( i / 4 ), piece );
    }
    const float4 w0 = *reinterpret_cast<const float4*>( &s_w[key0] ), w1 = *reinterpret_cast<const float4*>( &s_w[key0 + 8] );
#pragma unroll
    for ( int e = 0; e < 8; e++ ) {
      sum[e] = (float)k[0][e] * w0.x + (float)k[1][e] * w0.y + (float)k[2][e] * w0.z + (float)k[3][e] * w0.w + (float)k[4][e] * w1.x + (float)k[5][e] * w1.y + (float)k[6][e] * w1.z
               + (float)k[7][e] * w1.w;
    }
  }
  float* s_n = reinterpret_cast<float*>( s_k );
  __syncthreads(); // everyone has read k
  if ( set < 8 ) {
#pragma unroll
    for ( int e = 0; e < 8; e += 4 ) {
      *reinterpret_cast<float4*>( s_n + set * ( 8 * PIECES ) + piece * 8 + e ) = make_float4( sum[e], sum[e + 1], sum[e + 2], sum[e + 3] );
    }
  }
  __syncthreads();
  if ( threadIdx.x < s.dim ) {
    float n[2] = { 0.0f, 0.0f };
#pragma unroll
    for ( uint32_t k = 0; k < 8; k++ ) {
      n[k & 1] += s_n[k * ( 8 * PIECES ) + threadIdx.x];
    }
    ch.n[( (uint64_t)pair * ch.chunks + chunk ) * s.dim + threadIdx.x] = n[0] + n[1];
  }
}

// KS: steps of 32 of dim, dim <= 32 KS.  dim % 8 == 0, vdim % 8 == 0, 16-byte aligned product rows.
template<int KS>
__global__ __launch_bounds__( 256, 2 ) void mlstm_states_kernel( float* __restrict__ o_out, float* __restrict__ nm_out, MlstmIn<__bf16, ProductView<__bf16>> in, MlstmState st,
                                                                 MlstmShape s, MlstmChunks ch, uint32_t slices, uint32_t n_pairs )
{
  constexpr uint32_t RB = KS * 64; // bytes of a q or k row in LDS
  __shared__ uint4 s_k[CHUNK * RB / 16], s_q[CHUNK * RB / 16];
  __shared__ uint4 s_v[CHUNK * 8];
  __shared__ __attribute__( ( aligned( 16 ) ) ) float s_n[256]; // n in front of the chunk
  __shared__ __attribute__( ( aligned( 16 ) ) ) float s_a[CHUNK], s_w[2][CHUNK]; // (w is read behind the second barrier of a chunk, when another wave may write the next one's)

  // the slices of a (context, head) read the same q and k: all on one XCD, next to each other in time
  const uint32_t pair = ( blockIdx.x >> 3 ) / slices * 8 + ( blockIdx.x & 7 ), slice = ( blockIdx.x >> 3 ) % slices;
  if ( pair >= n_pairs ) {
    return;
  }
  const uint32_t h = pair % s.heads, ctx = pair / s.heads;
  uint8_t* base = static_cast<uint8_t*>( st.rows[ctx] );
  if ( base == nullptr ) {
    return;
  }
  float* S_mem = reinterpret_cast<float*>( base + st.offset );
  const bool fresh = st.start_pos[ctx] == 0;
  float n = !fresh && threadIdx.x < s.dim ? S_mem[s.n_off() + (uint64_t)h * s.dim + threadIdx.x] : 0.0f; // thread <-> element
  const float* n_chunk = ch.n + (uint64_t)pair * ch.chunks * s.dim + threadIdx.x;
  S_mem += (uint64_t)h * s.dim * s.vpad;
  const uint32_t wave = __builtin_amdgcn_readfirstlane( threadIdx.x >> 6 );
  const uint32_t lane = threadIdx.x & 63, r = lane & 15, g = lane >> 4;
  const uint32_t col = slice * 64 + wave * 16 + r; // this lane's column of v

  constexpr uint32_t PAST_THE_END = 0x80000000u; // an offset beyond any descriptor: reads zero, stores nothing
  const uint64_t S_at = reinterpret_cast<uint64_t>( S_mem ); // (said to be uniform: else every access below becomes a loop over the lanes' addresses)
  S_mem = reinterpret_cast<float*>( (uint64_t)__builtin_amdgcn_readfirstlane( (uint32_t)( S_at >> 32 ) ) << 32 | (uint32_t)__builtin_amdgcn_readfirstlane( (uint32_t)S_at ) );
  const __amdgpu_buffer_rsrc_t S_rsrc = __builtin_amdgcn_make_buffer_rsrc( S_mem, 0, (int)( s.dim * s.vpad * 4 ), 0x00020000 );
  // tile d: rows 32 (d / 2) + 8 (d % 2) + 16 (g / 2) + 4 (g % 2) + v, so that a lane holds both quads of eight rows apart, lanes 32 further on those of 16 rows further on
  const uint32_t S_off = col < s.vpad ? ( ( 16 * ( g >> 1 ) + 4 * ( g & 1 ) ) * s.vpad + col ) * 4 : PAST_THE_END;
  mfma_f32x4 S[2 * KS];
#pragma unroll
  for ( int d = 0; d < 2 * KS; d++ ) {
#pragma unroll
    for ( int v = 0; v < 4; v++ ) {
      S[d][v] = __builtin_bit_cast( float, __builtin_amdgcn_raw_buffer_load_b32( S_rsrc, fresh ? PAST_THE_END : S_off, ( 32 * ( d / 2 ) + 8 * ( d % 2 ) + v ) * s.vpad * 4, 0 ) );
    }
  }
  const uint64_t row_first = (uint64_t)ctx * st.n_tokens;
  const uint32_t ld_bytes = (uint32_t)( in.main.stride * 2 );

  // rows [0, rows) x `chunks` 16-byte chunks of the product at `p`, LDS rows of BYTES; the rest reads as zero
  auto fetch = [&]( uint4* tile, const __bf16* p, uint32_t rows, uint32_t chunks, auto row_bytes_tag, auto slot ) __attribute__( ( always_inline ) ) {
    constexpr uint32_t BYTES = decltype( row_bytes_tag )::value;
    const __amdgpu_buffer_rsrc_t rsrc = __builtin_amdgcn_make_buffer_rsrc( const_cast<__bf16*>( p ), 0, (int)( ( rows - 1 ) * ld_bytes + chunks * 16 ), 0x00020000 );
    constexpr uint32_t ROWS = 1024 / BYTES; // rows of one instruction of one wave
    constexpr uint32_t FORMS = BYTES == 512 ? 2 : 1; // 16 rows on a lane's chunk is the same again, so those are an offset of the wave's
#pragma unroll
    for ( uint32_t form = 0; form < FORMS; form++ ) {
      const uint32_t row = ( 4 * form + wave ) * ROWS + lane / ( BYTES / 16 );
      const uint32_t chunk = slot( row, lane % ( BYTES / 16 ) ); // the swizzle is its own inverse
      const uint32_t off = chunk < chunks ? row * ld_bytes + chunk * 16 : PAST_THE_END;
#pragma unroll
      for ( uint32_t i = 0; i < CHUNK / ( 4 * ROWS * FORMS ); i++ ) {
        const uint32_t on = 4 * ROWS * FORMS * i; // rows
        __builtin_amdgcn_raw_ptr_buffer_load_lds( rsrc, (lds_ptr)( tile + ( ( 4 * form + wave ) * ROWS + on ) * ( BYTES / 16 ) ), 16, off, on * ld_bytes, 0, 0 );
      }
    }
  };
  auto fetch_qv = [&]( uint32_t t0 ) __attribute__( ( always_inline ) ) {
    const uint32_t rows = min( (uint32_t)CHUNK, st.n_tokens - t0 );
    const __bf16* first = in.main.data + ( row_first + t0 ) * in.main.stride;
    fetch( s_q, first + in.col.q + h * s.dim, rows, s.dim / 8, std::integral_constant<uint32_t, RB> {}, swizzle<RB> );
    fetch( s_v, first + in.col.v + h * s.vdim + slice * 64, rows, min( 8u, ( s.vdim - slice * 64 ) / 8 ), std::integral_constant<uint32_t, 128> {}, swizzle<128> );
  };

  // 16 columns of keys, transposed: a lane gets its column's rows 4 (g % 2) + e and 8 + 4 (g % 2) + e.  Lane 4 e + q of a 16-lane group points at row e of
  // its four, columns 4 q .. 4 q + 3: of the 16 of this wave (v), or of the rows of a tile of S (k).
  const uint32_t tr_row = 4 * ( g & 1 ) + ( r >> 2 ), tr_q = r & 3;
  const uint32_t upper = 16 * ( g >> 1 ); // rows further on for lanes 32 .. 63, where an operand is of 32 keys
  auto transposed = [&]( const uint4* tile, uint32_t first, uint32_t second ) __attribute__( ( always_inline ) ) {
    union
    {
      v4s half[2];
      bf16x8 x;
    } u;
    u.half[0] = __builtin_amdgcn_ds_read_tr16_b64_v4i16( (lds_v4s)( (lds_char*)tile + first ) );
    u.half[1] = __builtin_amdgcn_ds_read_tr16_b64_v4i16( (lds_v4s)( (lds_char*)tile + second ) );
    return u.x;
  };
  // Byte addresses: a part of the lane, its low bits XORed with a constant, and a constant.  Computed where they are used: kept in registers over the loop there
  // are too many of them.
  auto opaque = []( uint32_t v ) __attribute__( ( always_inline ) ) {
    asm volatile( "" : "+v"( v ) );
    return v;
  };
  const uint32_t v_lane = tr_row * 128 + swizzle<128>( tr_row, 2 * wave + ( tr_q >> 1 ) ) * 16 + ( tr_q & 1 ) * 8;
  auto v_at = [&]( uint32_t lane_part ) __attribute__( ( always_inline ) ) { return transposed( s_v, lane_part, ( lane_part ^ 16 ) + 8 * 128 ); }; // (eight rows on: the swizzle's low bit)
  const uint32_t k_lane = tr_row * RB + swizzle_pair<RB>( tr_row, 2 * ( tr_q >> 1 ) ) * 16 + ( tr_q & 1 ) * 8;
  // a query's quads g % 2 of 16 dims.  The four tiles of queries apart from each other: two reads of 8 bytes at a constant distance would become one instruction
  // whose two halves meet in the same banks, and whose results have to be moved into their operands' registers.
  const uint32_t q_lane = r * RB + swizzle<RB>( r, 0 ) * 16 + ( g & 1 ) * 8;
  constexpr uint32_t PERIOD = RB == 128 ? 128 : 256; // bytes that the swizzles act on
  auto slot = [&]( uint32_t lane_part, uint32_t chunk ) __attribute__( ( always_inline ) ) { return ( lane_part ^ ( 16 * chunk % PERIOD ) ) + 16 * chunk / PERIOD * PERIOD; };

  float a1 = ch.tokens( MlstmChunks::A, pair, 0 )[lane], w1 = ch.tokens( MlstmChunks::W, pair, 0 )[lane]; // of token `lane`
  fetch_qv( 0 );
  __builtin_amdgcn_s_waitcnt( 0x0F70 ); // vmcnt(0)
  constexpr int STORES = 16; // of O, each an instruction of its own: the rows of a tile are whole rows of the output apart
  for ( uint32_t c = 0; c < ch.chunks; c++ ) {
    const uint32_t t0 = c * CHUNK, rows = min( (uint32_t)CHUNK, st.n_tokens - t0 );
    s_n[threadIdx.x] = n;
    if ( wave == 0 ) {
      s_a[lane] = a1;
      s_w[c & 1][lane] = w1;
    }
    // This wave's part of q and v has landed: behind its requests are AT LEAST the last chunk's STORES (memory operations of a wave end in their order).
    __builtin_amdgcn_s_waitcnt( ( STORES & 15 ) | ( STORES >> 4 ) << 14 | 0x0F70 );
    asm volatile( "s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory" ); // everyone's; and everyone is through with the last chunk's k
    const uint4* weights = ch.weights + ( (uint64_t)pair * ch.chunks + c ) * ( WEIGHT_TILES * 64 ) + lane;
    uint4 P[WEIGHT_TILES];
#pragma unroll
    for ( uint32_t i = 0; i < WEIGHT_TILES; i++ ) {
      P[i] = weights[i * 64];
    }
    const float den1 = ch.tokens( MlstmChunks::DEN, pair, c )[lane], floor1 = ch.tokens( MlstmChunks::FLOOR, pair, c )[lane]; // of token `lane`
    const float decay = ch.decay[(uint64_t)pair * ch.chunks + c];
    const float n_more = threadIdx.x < s.dim ? n_chunk[(uint64_t)c * s.dim] : 0.0f;
    fetch( s_k, in.main.data + ( row_first + t0 ) * in.main.stride + in.col.k + h * s.dim, rows, s.dim / 8, std::integral_constant<uint32_t, RB> {}, swizzle_pair<RB> );
    __builtin_amdgcn_sched_barrier( 0 ); // (else the scheduler moves the requests down to where their results are used)

    // ---- Q S (state in front of the chunk): 16 queries a tile
    mfma_f32x4 O[4];
    uint32_t q_row[4];
#pragma unroll
    for ( int i = 0; i < 4; i++ ) {
      O[i] = mfma_f32x4 { 0, 0, 0, 0 };
      q_row[i] = opaque( 16 * i * RB + q_lane );
    }
#pragma unroll
    for ( int j = 0; j < KS; j++ ) {
      if ( j % 2 == 0 ) {
        __builtin_amdgcn_sched_barrier( 0 ); // (without these fences the scheduler asks for all operands of a phase at once and spills)
      }
      Split<2> sp;
#pragma unroll
      for ( int k = 0; k < 4; k++ ) {
        sp.set( k, S[2 * j + ( k >> 1 )][2 * ( k & 1 )], S[2 * j + ( k >> 1 )][2 * ( k & 1 ) + 1] );
      }
      swap_halves( sp.t[1].x, sp.t[0].x ); // both terms of the lower 16 rows, the lower term in front; both of the upper 16
#pragma unroll
      for ( int n2 = 1; n2 >= 0; n2-- ) {
        union
        {
          uint2 p[2];
          bf16x8 x;
        } a[4];
#pragma unroll
        for ( int i = 0; i < 4; i++ ) {
#pragma unroll
          for ( int hf = 0; hf < 2; hf++ ) {
            a[i].p[hf] = *reinterpret_cast<const uint2*>( reinterpret_cast<const char*>( s_q ) + slot( q_row[i], 4 * j + 2 * ( 1 - n2 ) + hf ) );
          }
        }
#pragma unroll
        for ( int i = 0; i < 4; i++ ) { // (the tiles in turn: a product that waits for the one before it leaves the matrix unit idle)
          O[i] = Mfma<__bf16>::k32( a[i].x, sp.t[n2].x, O[i] );
        }
      }
    }
    // ---- denominators of this slice's tokens: n . q, four lanes a token, a quarter of the dims each
    if ( slice + slices * wave < rows ) {
      const uint32_t ln = opaque( lane );
      const uint32_t token = slice + slices * ( wave + ( ln & ~3u ) ), t = min( token, (uint32_t)CHUNK - 1 );
      const uint32_t half = ( ln >> 1 ) & 1, quad = ln & 1; // of the head's dims, of eight
      const uint32_t q_token = t * RB + swizzle<RB>( t, 2 * KS * half ) * 16 + quad * 8;
      const float* nk = s_n + 16 * KS * half + 4 * quad;
      float nq = 0.0f;
#pragma unroll
      for ( uint32_t k = 0; k < KS; k++ ) { // 16 dims
        if ( k % 4 == 0 ) {
          __builtin_amdgcn_sched_barrier( 0 );
        }
        union
        {
          uint2 p[2];
          bf16x8 x;
        } a;
        const float4 n0 = *reinterpret_cast<const float4*>( nk + 16 * k ), n1 = *reinterpret_cast<const float4*>( nk + 16 * k + 8 );
#pragma unroll
        for ( uint32_t hf = 0; hf < 2; hf++ ) {
          a.p[hf] = *reinterpret_cast<const uint2*>( reinterpret_cast<const char*>( s_q ) + slot( q_token, 2 * k + hf ) );
        }
        nq += (float)a.x[0] * n0.x + (float)a.x[1] * n0.y + (float)a.x[2] * n0.z + (float)a.x[3] * n0.w + (float)a.x[4] * n1.x + (float)a.x[5] * n1.y + (float)a.x[6] * n1.z
              + (float)a.x[7] * n1.w;
      }
      nq += __shfl_xor( nq, 1 );
      nq += __shfl_xor( nq, 2 );
      const float over = 1.0f / ( fmaxf( fabsf( nq * s.q_scale * s_a[t] + __shfl( den1, t ) ), __shfl( floor1, t ) ) + 1e-6f );
      if ( ( ln & 3 ) == 0 && token < rows ) {
        ch.tokens( MlstmChunks::OVER, pair, c )[t] = over;
      }
    }
    // ---- O = a Q S + P V
    bf16x8 V[4];
#pragma unroll
    for ( int k = 0; k < 4; k++ ) {
      V[k] = v_at( v_lane + 16 * k * 128 );
    }
#pragma unroll
    for ( uint32_t i = 0; i < 4; i++ ) {
      const float4 a4 = *reinterpret_cast<const float4*>( &s_a[16 * i + 4 * g] );
      const float f[4] = { a4.x, a4.y, a4.z, a4.w };
#pragma unroll
      for ( int e = 0; e < 4; e++ ) {
        O[i][e] *= f[e] * s.q_scale;
      }
#pragma unroll
      for ( uint32_t k = 0; k <= i; k++ ) {
        O[i] = Mfma<__bf16>::k32( __builtin_bit_cast( bf16x8, P[weight_tile( i, k )] ), V[k], O[i] );
      }
    }
    bf16x8 V2[2]; // the keys of 32 over the lanes: a half's terms are made in it, and change places with the other's
#pragma unroll
    for ( int k = 0; k < 2; k++ ) {
      V2[k] = v_at( v_lane + ( 32 * k + upper ) * 128 );
    }
    __builtin_amdgcn_s_waitcnt( 0x0F70 ); // vmcnt(0): this wave's part of k has landed
    __syncthreads();                      // everyone's; and everyone has read q and v
    if ( t0 + CHUNK < st.n_tokens ) {
      a1 = ch.tokens( MlstmChunks::A, pair, c + 1 )[lane], w1 = ch.tokens( MlstmChunks::W, pair, c + 1 )[lane];
      fetch_qv( t0 + CHUNK );
    }
    __builtin_amdgcn_sched_barrier( 0 ); // the stores stay behind the requests
    const uint32_t hv = s.heads * s.vdim;
    const __amdgpu_buffer_rsrc_t o_rsrc
      = __builtin_amdgcn_make_buffer_rsrc( o_out + ( row_first + t0 ) * hv + h * s.vdim, 0, (int)( ( ( rows - 1 ) * hv + s.vdim ) * 4 ), 0x00020000 );
    const uint32_t o_off = col < s.vdim ? ( 4 * g * hv + col ) * 4 : PAST_THE_END;
    static_assert( sizeof( O ) == STORES * sizeof( float ), "the wait at a chunk's head counts on one store for each element" );
#pragma unroll
    for ( int i = 0; i < 4; i++ ) {
#pragma unroll
      for ( int e = 0; e < 4; e++ ) {
        __builtin_amdgcn_raw_buffer_store_b32( __builtin_bit_cast( unsigned, (float)O[i][e] ), o_rsrc, o_off, ( 16 * i + e ) * hv * 4, 0 );
      }
    }
    n = n * decay + n_more;
    // ---- S behind the chunk
    // 32 keys are three products: lower and middle term of the first 16; their upper term and the lower one of the others; the others' middle and upper term
    bf16x8 wv[2][3];
#pragma unroll
    for ( int j = 0; j < 2; j++ ) {
      Split<3> terms;
#pragma unroll
      for ( int hf = 0; hf < 2; hf++ ) {
        const float4 w = *reinterpret_cast<const float4*>( &s_w[c & 1][32 * j + upper + 8 * hf + 4 * ( g & 1 )] );
        terms.set( 2 * hf, (float)V2[j][4 * hf] * w.x, (float)V2[j][4 * hf + 1] * w.y );
        terms.set( 2 * hf + 1, (float)V2[j][4 * hf + 2] * w.z, (float)V2[j][4 * hf + 3] * w.w );
      }
      bf16x8 lower = terms.t[1].x, others = terms.t[1].x; // the middle terms of either, in all lanes
      swap_halves( lower, others );
      const bool first = lane < 32;
      wv[j][0] = first ? terms.t[2].x : lower;
      wv[j][1] = first ? terms.t[0].x : terms.t[2].x;
      wv[j][2] = first ? others : terms.t[0].x;
    }
#pragma unroll
    for ( int d0 = 0; d0 < 2 * KS; d0 += 4 ) { // (four tiles in turn, as above)
      __builtin_amdgcn_sched_barrier( 0 );
#pragma unroll
      for ( int d = d0; d < d0 + 4; d++ ) {
#pragma unroll
        for ( int v = 0; v < 4; v++ ) {
          S[d][v] *= decay;
        }
      }
      const uint32_t k_both = opaque( k_lane );
#pragma unroll
      for ( int j = 0; j < 2; j++ ) {
        bf16x8 a[3][4];
#pragma unroll
        for ( int d = 0; d < 4; d++ ) {
          const uint32_t at = slot( k_both, 4 * ( ( d0 + d ) / 2 ) + d % 2 ) + 32 * j * RB;
          a[0][d] = transposed( s_k, at, at + 8 * RB );
          a[2][d] = transposed( s_k, at + 16 * RB, at + 24 * RB );
          a[1][d] = lane < 32 ? a[0][d] : a[2][d];
        }
#pragma unroll
        for ( int n3 = 0; n3 < 3; n3++ ) {
#pragma unroll
          for ( int d = 0; d < 4; d++ ) {
            S[d0 + d] = Mfma<__bf16>::k32( a[n3][d], wv[j][n3], S[d0 + d] );
          }
        }
      }
    }
  }

  uint32_t vpad = s.vpad; // (the row offsets anew: kept from the loads above they would occupy the scalar registers all along)
  asm volatile( "" : "+s"( vpad ) );
#pragma unroll
  for ( int d = 0; d < 2 * KS; d++ ) {
#pragma unroll
    for ( int v = 0; v < 4; v++ ) {
      __builtin_amdgcn_raw_buffer_store_b32( __builtin_bit_cast( unsigned, (float)S[d][v] ), S_rsrc, S_off, ( 32 * ( d / 2 ) + 8 * ( d % 2 ) + v ) * vpad * 4, 0 );
    }
  }
  if ( slice == 0 && threadIdx.x < s.dim ) {
    nm_out[(uint64_t)pair * ( s.dim + 1 ) + threadIdx.x] = n;
  }
}

// one wave per (token, head); V: columns at a time; CHUNKED: `o` is not divided by its denominators yet
template<typename E, typename View, int V, bool CHUNKED>
__global__ __launch_bounds__( 256 ) void mlstm_finish_kernel( E* __restrict__ out,
                                                              const float* __restrict__ o,
                                                              const float* __restrict__ nm,
                                                              MlstmIn<E, View> in,
                                                              const E* __restrict__ norm,
                                                              MlstmState st,
                                                              MlstmShape s,
                                                              MlstmChunks ch )
{
  const uint64_t row = blockIdx.x;
  const uint32_t h = blockIdx.y * 4 + ( threadIdx.x >> 6 ), lane = threadIdx.x & 63;
  const uint32_t ctx = (uint32_t)( row / st.n_tokens ), tok = (uint32_t)( row % st.n_tokens );
  uint8_t* base = static_cast<uint8_t*>( st.rows[ctx] );
  if ( base == nullptr || h >= s.heads ) {
    return;
  }
  const float* oh = o + row * s.heads * s.vdim + (uint64_t)h * s.vdim;
  E* dst = out + row * s.heads * s.vdim + (uint64_t)h * s.vdim;
  float over = 1.0f;
  if constexpr ( CHUNKED ) {
    over = ch.tokens( MlstmChunks::OVER, ctx * s.heads + h, tok / CHUNK )[tok % CHUNK];
  }
  if constexpr ( V == 4 ) { // vdim <= 1024, everything in groups of four
    float4 v[4], g[4], w[4];
    float ss = 0.0f;
#pragma unroll
    for ( int k = 0; k < 4; k++ ) {
      const uint32_t c = ( k * 64 + lane ) * 4, at = c < s.vdim ? c : 0;
      v[k] = *reinterpret_cast<const float4*>( oh + at );
      g[k] = in.main.at4( row, in.col.g + h * s.vdim + at );
      w[k] = ProductView<E>::load4( norm + h * s.vdim + at );
    }
#pragma unroll
    for ( int k = 0; k < 4; k++ ) {
      v[k].x *= over, v[k].y *= over, v[k].z *= over, v[k].w *= over;
      ss += ( k * 64 + lane ) * 4 < s.vdim ? squares<false>( v[k] ) : 0.0f;
    }
    const float inv = 1.0f / sqrtf( wave_sum( ss ) / (float)s.vdim + s.eps );
#pragma unroll
    for ( int k = 0; k < 4; k++ ) {
      const uint32_t c = ( k * 64 + lane ) * 4;
      union
      {
        E e[4];
        uint2 half;
        uint4 full;
      } y;
      y.e[0] = from_f32<E>( v[k].x * inv * w[k].x / ( 1.0f + expf( -g[k].x ) ) );
      y.e[1] = from_f32<E>( v[k].y * inv * w[k].y / ( 1.0f + expf( -g[k].y ) ) );
      y.e[2] = from_f32<E>( v[k].z * inv * w[k].z / ( 1.0f + expf( -g[k].z ) ) );
      y.e[3] = from_f32<E>( v[k].w * inv * w[k].w / ( 1.0f + expf( -g[k].w ) ) );
      if ( c < s.vdim ) {
        if constexpr ( sizeof( E ) == 2 ) {
          *reinterpret_cast<uint2*>( dst + c ) = y.half;
        } else {
          *reinterpret_cast<uint4*>( dst + c ) = y.full;
        }
      }
    }
  } else {
    float ss = 0.0f;
    for ( uint32_t c = lane; c < s.vdim; c += 64 ) {
      ss += oh[c] * over * ( oh[c] * over );
    }
    const float inv = 1.0f / sqrtf( wave_sum( ss ) / (float)s.vdim + s.eps );
    for ( uint32_t c = lane; c < s.vdim; c += 64 ) {
      const float g = in.main.at( row, in.col.g + h * s.vdim + c );
      dst[c] = from_f32<E>( oh[c] * over * inv * to_f32( norm[h * s.vdim + c] ) / ( 1.0f + expf( -g ) ) );
    }
  }
  if ( tok + 1 == st.n_tokens ) {
    float* S = reinterpret_cast<float*>( base + st.offset );
    const float* src = nm + ( (uint64_t)ctx * s.heads + h ) * ( s.dim + 1 );
    for ( uint32_t d = lane; d < s.dim; d += 64 ) {
      S[s.n_off() + (uint64_t)h * s.dim + d] = src[d];
    }
    if ( lane == 0 ) {
      S[s.m_off() + h] = src[s.dim];
    }
  }
}

MlstmShape shape_of( const gh_mlstm* m )
{
  MlstmShape s;
  s.heads = m->heads;
  s.dim = m->dim;
  s.vdim = m->vdim;
  s.vpad = ( m->vdim + 3 ) / 4 * 4;
  s.cap = m->gate_cap;
  s.eps = m->eps;
  s.q_scale = 1.0f / sqrtf( (float)m->dim );
  return s;
}

} // namespace
} // namespace gh

using namespace gh;

extern "C" {

uint64_t gh_mlstm_state_bytes( const gh_mlstm* m ) { return shape_of( m ).elements() * sizeof( float ); }

uint64_t gh_mlstm_weight_rows( const gh_mlstm* m, uint64_t* gate_row )
{
  const uint64_t main = 2ull * m->heads * m->dim + 2ull * m->heads * m->vdim;
  const uint64_t first = ( main + 7 ) / 8 * 8;
  if ( gate_row != nullptr ) {
    *gate_row = first;
  }
  return first + ( 2ull * m->heads + 7 ) / 8 * 8;
}

int gh_mlstm_forward( void* out, const void* x, const void* w, uint64_t width, const gh_mlstm* m, const void* bias_i, const void* bias_f, const void* norm,
                      void* const* context_rows_dev, uint64_t state_offset, const uint32_t* start_pos_dev, uint64_t batch, uint32_t n_tokens, gh_dtype dt,
                      gh_stream stream )
{
  if ( int rc = ensure_init() ) {
    return rc;
  }
  const uint64_t rows = batch * n_tokens;
  if ( rows == 0 ) {
    return GH_OK;
  }
  GH_REQUIRE( out && x && w && m && norm && context_rows_dev && start_pos_dev, "gh_mlstm_forward: NULL pointer" );
  GH_REQUIRE( dt == GH_BF16 || dt == GH_F32, "gh_mlstm_forward: unsupported dtype %d", (int)dt );
  GH_REQUIRE( m->heads > 0 && m->dim > 0 && m->vdim > 0 && m->heads <= 65535 && batch <= 65535 && m->dim <= 4096, "gh_mlstm_forward: bad shape" );
  GH_REQUIRE( m->gate_cap > 0.0f && state_offset % 16 == 0, "gh_mlstm_forward: bad gate cap or state offset" );
  const MlstmShape s = shape_of( m );
  hipStream_t st = as_stream( stream );
  uint64_t gate_row = 0;
  const uint64_t r = gh_mlstm_weight_rows( m, &gate_row );
  const uint32_t hd = s.heads * s.dim, hv = s.heads * s.vdim;
  MlstmCols col { 0, hd, 2 * hd, 2 * hd + hv, (uint32_t)gate_row, (uint32_t)gate_row + s.heads };
  Product y, gates;
  const bool chunked = dt == GH_BF16 && n_tokens >= CHUNKED_TOKENS && s.dim <= 256 && s.dim % 8 == 0 && s.vdim % 8 == 0;
  if ( dt == GH_BF16 && ( chunked || rows >= PRODUCT_ROUNDED_ROWS ) ) { // the gates stay fp32 sums
    if ( int rc = make_product( x, w, width, gate_row, rows, dt, false, st, &y, 1 ) ) {
      return rc;
    }
    if ( int rc = make_product( x, static_cast<const char*>( w ) + gate_row * width * dtype_size( dt ), width, r - gate_row, rows, dt, true, st, &gates ) ) {
      return rc;
    }
    col.i = 0;
    col.f = s.heads;
  } else {
    if ( int rc = make_product( x, w, width, r, rows, dt, false, st, &y ) ) {
      return rc;
    }
    gates = y;
  }
  void* scratch = nullptr;
  const uint64_t o_bytes = ( rows * hv * sizeof( float ) + 255 ) / 256 * 256;
  const uint64_t nm_bytes = ( batch * s.heads * ( s.dim + 1ull ) * sizeof( float ) + 255 ) / 256 * 256;
  const uint64_t n_pairs = batch * s.heads, n_chunks = ( (uint64_t)n_tokens + CHUNK - 1 ) / CHUNK, all_chunks = chunked ? n_pairs * n_chunks : 0;
  const uint64_t weight_bytes = all_chunks * WEIGHT_TILES * 64 * sizeof( uint4 ), token_bytes = MlstmChunks::PLANES * all_chunks * CHUNK * sizeof( float );
  // chunks: 12 KB and a head's n, whatever the size of its values (a tenth of the call's workspace at 512 columns of v, two fifths at 64)
  const uint64_t more = chunked ? weight_bytes + token_bytes + all_chunks * ( s.dim + 1ull ) * sizeof( float ) : rows * 2 * s.heads * sizeof( float );
  if ( int rc = stream_scratch( st, SCRATCH_MIXER, o_bytes + nm_bytes + more, 1ull << 20, &scratch ) ) {
    return rc;
  }
  float* o = static_cast<float*>( scratch );
  float* nm = reinterpret_cast<float*>( static_cast<char*>( scratch ) + o_bytes );
  char* behind = static_cast<char*>( scratch ) + o_bytes + nm_bytes;
  float* log_gates = reinterpret_cast<float*>( behind );
  MlstmChunks chunks {};
  if ( chunked ) {
    chunks.weights = reinterpret_cast<uint4*>( behind );
    chunks.token = reinterpret_cast<float*>( behind + weight_bytes );
    chunks.decay = reinterpret_cast<float*>( behind + weight_bytes + token_bytes );
    chunks.n = chunks.decay + all_chunks;
    chunks.chunks = (uint32_t)n_chunks;
    chunks.plane = all_chunks * CHUNK;
  }
  const MlstmState state { context_rows_dev, state_offset, start_pos_dev, n_tokens };
  return with_product( dt, y, [&]( auto tag, auto view ) -> int {
    using E = decltype( tag );
    using View = decltype( view );
    const MlstmGates<E> raw { ProductView<float>( gates ), col, static_cast<const E*>( bias_i ), static_cast<const E*>( bias_f ), s.cap };
    // One token of a context: every work-group of a head makes the two gates again beside its loads of the state, which is less than a launch in front of it
    // (32 contexts: 4.6 us).
    const bool gates_made = n_tokens > 1 && !chunked;
    if ( gates_made ) {
      mlstm_gates_kernel<E><<<(unsigned)std::min<uint64_t>( ( rows * 2 * s.heads + 255 ) / 256, 4096 ), 256, 0, st>>>( log_gates, raw, s.heads, rows );
      GH_LAUNCH_CHECK();
    }
    const MlstmIn<E, View> in { view, gates_made ? log_gates : nullptr, col };
    const dim3 grid( ( s.vpad + SLICE - 1 ) / SLICE, s.heads, (unsigned)batch );
    bool walked = false;
    if constexpr ( std::is_same_v<View, ProductView<__bf16>> ) {
      if ( chunked ) {
        const unsigned groups = (unsigned)( ( n_pairs + 7 ) / 8 * 8 * grid.x ), score_groups = (unsigned)( ( n_pairs + 7 ) / 8 * 8 * n_chunks );
        const bool alone = n_chunks == 1;
        if ( !alone ) {
          mlstm_scan_kernel<<<dim3( s.heads, (unsigned)batch ), 1024, 0, st>>>( nm, raw, state, s, chunks );
          GH_LAUNCH_CHECK();
        }
        auto walk = [&]( auto steps ) -> int {
          constexpr int KS = decltype( steps )::value;
          auto scores = alone ? mlstm_scores_kernel<KS, true> : mlstm_scores_kernel<KS, false>;
          scores<<<score_groups, 256, 0, st>>>( nm, in, raw, state, s, chunks, (uint32_t)n_pairs );
          GH_LAUNCH_CHECK();
          mlstm_states_kernel<KS><<<groups, 256, 0, st>>>( o, nm, in, state, s, chunks, grid.x, (uint32_t)n_pairs );
          return GH_OK;
        };
        const int rc = s.dim <= 64 ? walk( std::integral_constant<int, 2> {} )
                       : s.dim <= 128 ? walk( std::integral_constant<int, 4> {} ) : walk( std::integral_constant<int, 8> {} );
        if ( rc ) {
          return rc;
        }
        walked = true;
      }
    }
    const size_t lds = ( 3 * ( ( s.dim + 3 ) / 4 * 4 ) + SLICE + 16 + 16 * SLICE ) * sizeof( float );
    if ( walked ) {
      // the chunks' kernels have done it
    } else if ( s.dim <= 64 ) {
      mlstm_walk_kernel<E, View, 4><<<grid, 256, lds, st>>>( o, nm, in, raw, state, s );
    } else if ( s.dim <= 128 ) {
      mlstm_walk_kernel<E, View, 8><<<grid, 256, lds, st>>>( o, nm, in, raw, state, s );
    } else if ( s.dim <= 256 ) {
      mlstm_walk_kernel<E, View, 16><<<grid, 256, lds, st>>>( o, nm, in, raw, state, s );
    } else {
      mlstm_walk_kernel<E, View, 0><<<grid, 256, lds, st>>>( o, nm, in, raw, state, s );
    }
    GH_LAUNCH_CHECK();
    const dim3 finish( (unsigned)rows, ( s.heads + 3 ) / 4 );
    auto finish_rows = [&]( auto columns ) {
      constexpr int V = decltype( columns )::value;
      if constexpr ( std::is_same_v<View, ProductView<__bf16>> ) {
        if ( walked ) {
          mlstm_finish_kernel<E, View, V, true><<<finish, 256, 0, st>>>( static_cast<E*>( out ), o, nm, in, static_cast<const E*>( norm ), state, s, chunks );
          return;
        }
      }
      mlstm_finish_kernel<E, View, V, false><<<finish, 256, 0, st>>>( static_cast<E*>( out ), o, nm, in, static_cast<const E*>( norm ), state, s, chunks );
    };
    if ( s.vdim % 4 == 0 && s.vdim <= 1024 && view.stride % 4 == 0 && col.g % 4 == 0 && ( reinterpret_cast<uintptr_t>( norm ) & 15u ) == 0
         && ( reinterpret_cast<uintptr_t>( out ) & 15u ) == 0 ) {
      finish_rows( std::integral_constant<int, 4> {} );
    } else {
      finish_rows( std::integral_constant<int, 1> {} );
    }
    GH_LAUNCH_CHECK();
    return GH_OK;
  } );
}

} // extern "C"
