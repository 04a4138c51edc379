// Tile GEMM for many activation rows: a 256 x 256 (weight rows x tokens) output tile per work-group, i.e. per CU, for products with
// enough such tiles to fill the chip.
//
//   work-group  8 waves, two per SIMD, as two groups of four: group g owns weight rows 64 g .. + 63 of either half of the tile, wave w of a
//               group tokens 32 w .. + 31 of either half: 64 x 32 outputs in each of the four quadrants, 2 x 4 x 8 accumulators of
//               v_mfma_f32_16x16x32 (128 registers).
//   schedule    A 64-k step is two phases, one per half of the weight rows: the memory part reads the phase's operands from LDS and
//               requests later ones, then 32 MFMAs multiply them.  The second group runs one barrier behind the first, so that at
//               any moment one wave of a SIMD multiplies while the other reads: neither waits for the other's instructions, and all a
//               barrier costs is its own latency.  24 LDS reads, 64 MFMAs and 4 barriers a wave and step.
//   operands    global -> LDS directly (`buffer_load ... lds`, 16 bytes a lane), two 64-k stages.  A half tile is requested again as soon
//               as both groups have read it, i.e. nearly two steps ahead; waits count loads instead of draining them (8 stay
//               in flight, 128 KiB of LDS are all but 16 KiB outstanding or in use).  16-byte chunks are XORed with bits of their row through
//               the address a lane fetches, so that the operand reads are free of bank conflicts.
//   output      MFMA row m of a lane's four row tiles is mapped to weight row 32 (i / 2) + 8 (m / 4) + 4 (i % 2) + m % 4: a lane then holds
//               8 neighbouring rows of a token and 4 lanes 64 contiguous bytes, which leave as 16-byte stores straight from the
//               registers.  LDS takes no part, so the next tile's first two steps are requested behind the last steps of this
//               one and arrive under its stores: one work-group per CU walks tile after tile without draining (K ranges of an
//               even number of steps; others take one tile per work-group).
//   tile order  each XCD owns every 8th row tile and walks them in patches of 32 tiles that are resident together; the row tiles beyond a
//               multiple of 8 are cut into 8 equal runs of tiles.
//   what binds  the power budget.  Counters at 8192 x 8192 x 8192 (pipes busy of 4, clock): this loop 3.74 at 1.47 GHz; in four phases a step,
//               i.e. twice the barriers, 2.95 at 1.59 GHz; those four phases with v_mfma_f32_32x32x16 3.28 at 1.40 GHz: half the accumulator
//               traffic a flop buys 13 % of clock.  PFLOP/s, interleaved on one box: 8192 x 8192 x 8192 1.49 (1.25 with the kernels this
//               one replaced, v_mfma_f32_32x32x16 in four waves of 128 x 128 or eight of 96 x 128 without phases), 15360 x 5120 at 16384
//               tokens 1.45 (1.24), 13824 x 5120 1.43 (1.24), 22016 x 4096 at 8192 tokens 1.43 (1.20), 28672 x 8192 at 3328 tokens 1.43
//               (1.14), 8192 x 28672 at 3328 (1.6 rounds) 1.33 (1.13).  Of that: reads in front of the loads of a part 1 %; tile after
//               tile without draining 1-2 %; the output's addresses once a tile instead of once a store 3 %.  Not kept: raised wave
//               priority around the MFMAs (-2 %), the loads between the MFMAs (-3 %), four loads in either phase instead of 2 and 6 (0).
#include "gh_product.h"

#include <algorithm>
#include <type_traits>

namespace gh {

typedef __attribute__( ( address_space( 3 ) ) ) void* lds_ptr;

namespace {

constexpr int TM2 = 256; // weight rows per work-group
constexpr int TN2 = 256; // tokens per work-group
constexpr int TKS = 64;  // k per step
constexpr int T256_THREADS = 512;

// XCD x owns row tiles x, x + 8, ... of the first `owned` and walks (row tile, token tile) in strips of gm row tiles and, inside a strip, in
// patches of gm x gn, token direction fastest.  The row tiles left over (fewer than 8, or none) are cut into 8 equal runs of tiles, one
// per XCD, in patches of (all of those rows) x rest_gn.
struct TileOrder
{
  uint32_t token_tiles, gm, gn;
  uint32_t owned;
  uint32_t rest_rows, rest_share, rest_gn; // left-over row tiles; tiles of them per XCD
};

// Tile `idx` of an XCD's list; false: past its end.
__device__ __forceinline__ bool tile_of_index( const TileOrder& ord, uint32_t xcd, uint32_t idx, uint32_t& row_tile, uint32_t& token_tile )
{
  const uint32_t rows = ( ord.owned + 7 - xcd ) / 8;
  if ( idx < rows * ord.token_tiles ) {
    const uint32_t per_strip = ord.gm * ord.token_tiles; // gm row tiles over all tokens; the last strip and each strip's last patch may be narrower
    const uint32_t strip = idx / per_strip, in_strip = idx % per_strip;
    const uint32_t height = min( ord.gm, rows - strip * ord.gm );
    const uint32_t patch = in_strip / ( height * ord.gn ), in_patch = in_strip % ( height * ord.gn );
    const uint32_t width = min( ord.gn, ord.token_tiles - patch * ord.gn );
    row_tile = ( strip * ord.gm + in_patch / width ) * 8 + xcd;
    token_tile = patch * ord.gn + in_patch % width;
    return true;
  }
  const uint32_t mine = idx - rows * ord.token_tiles;
  const uint32_t u = xcd * ord.rest_share + mine;
  if ( mine >= ord.rest_share || u >= ord.rest_rows * ord.token_tiles ) {
    return false;
  }
  const uint32_t per_patch_col = ord.rest_rows * ord.rest_gn; // the last one may be narrower
  const uint32_t patch_col = u / per_patch_col, in_col = u % per_patch_col;
  const uint32_t width = min( ord.rest_gn, ord.token_tiles - patch_col * ord.rest_gn );
  row_tile = ord.owned + in_col / width;
  token_tile = patch_col * ord.rest_gn + in_col % width;
  return true;
}

// What a work-group does with its sums: xout = DType(sum); the reference's next op on top of that,
// xout = DType(float(xout) + float(DType(sum))) (accum; only with r % 8 == 0); or the fp32 sums, (splits, b, r).
// Or the SiLU gate over two products, w = [w1 rows | w3 rows], as GateRows says (gh_product.h), without a bias: a tile is 128 rows of w1 and the same 128 of
// w3, whose sums a lane holds side by side; half as many stores, and no kernel that reads both factors
// again (13B, 16384 tokens: 271 us a layer; the pass of four 36.9 -> 35.5 ms).  With one work-group per CU nothing hides the epilogue, so a
// gate that takes longer is a variant of its own, bf16: the tanh gate, and biases, kept in LDS since the tile before (8192 rows, 2 x 11008 of
// 4096 k: 1083 us as a rounded product and a kernel behind it, 984 so; 1024 rows of 2 x 2816 of 1024 k 33.8 and 26.1).
// The gate's epilogue is 1475 vector instructions a wave with the general division and every factor also rounded for the case that it counts, 866 as it is (bf16;
// f16, which rounds the factors, 1410 and 1061): some 3 of a 64-step tile's 95 us, of which the power budget takes back a part (4 x 2048 tokens of the design whose gate
// is half of its time 4851 -> 4799 us, 26 x 128 of 70B 17.55 -> 17.47 ms, both with two instructions an output fewer, whose gates of factors below -87.3 were 0).
// Or q, k and v as QkvRows says, 16-byte pieces of a token's heads to its query and its cache row: the two kernels that read the product again, append and
// rotate took 260 us a layer at 13B and 16384 tokens (3 x 5120 rows of 5120), this epilogue 55 of the product's 1785 (1730 with plain stores).
constexpr int EPI_STORE = 0, EPI_ACCUM = 1, EPI_GATE = 2, EPI_PARTIAL = 3, EPI_QKV = 4, EPI_BIAS_GATE = 5;

struct TileOut
{
  void* xout;      // rows [0, r_first), a (b, r_first) matrix
  void* xout2;     // rows from r_first on, as rows 0.. of a (b, r - r_first) matrix; r_first == r: one output
  float* partial;  // EPI_PARTIAL
  uint32_t r, b, r_first; // the gates: r rows of each factor
  GateRows gate;
  QkvRows qkv;
};

// LDS slot (16 bytes) of a chunk: rows of 8 chunks.  A wave's 16-byte reads are served in four passes of 16 lanes (0-3, 12-15, 20-23, 24-27 first);
// a pass covers two neighbouring chunks of the rows below, and the XORs spread it over all 16 slots of 256 bytes.
__device__ __forceinline__ uint32_t x_swizzle( uint32_t row ) { return ( row >> 1 ) & 7; }                           // 16 neighbouring rows
__device__ __forceinline__ uint32_t w_swizzle( uint32_t row ) { return ( ( row >> 1 ) & 1 ) | ( ( row >> 2 ) & 6 ); } // rows 8 (m / 4) + m % 4 (+ 4), m < 16

__device__ __forceinline__ void drain_loads_and_stores() { __builtin_amdgcn_s_waitcnt( 0x0F70 ); } // vmcnt(0)

// acc[a][h][i][j][v]: row 128 a + 64 group + 32 (i / 2) + 8 (lane / 16) + 4 (i % 2) + v, token 128 h + 32 wave + 16 j + lane % 16.
// Returns whether the tile left by exactly 16 (the gates: 8) stores of this wave behind its last load (not EPI_PARTIAL); else nothing is outstanding, so that
// also the compiler, which waits before it reads what loads leave in LDS, may count those stores: with one path of fewer stores it has the next
// tile's second reads wait for nearly all of them (4096 x 1024 at 8192 tokens 61 -> 59 us, 2 x 11008 x 4096 with the gate 1 %).
// tokens: LDS, EPI_QKV: the cache rows of the tile's 256 tokens, then their positions; those past the last hold the last one's.
// EPI_BIAS_GATE: the biases (float) of the tile's 128 rows of w1, then those of w3
template<typename E, int EPI>
__device__ __forceinline__ bool store_tile( const mfma_f32x4 ( &acc )[2][2][4][2], const TileOut& o, uint32_t tile_row0, uint32_t tile_col0, uint32_t group, uint32_t wave,
                                            uint32_t lane, uint32_t split, const uint32_t* tokens )
{
  const uint32_t row0 = tile_row0 + 64 * group + 8 * ( lane >> 4 ), col0 = tile_col0 + 32 * wave + ( lane & 15 );
  union Chunk
  {
    uint4 raw;
    uint32_t pair[4];
    E h[8];
  };
  auto rounded = [&]( int a, int h, int i, int j ) __attribute__( ( always_inline ) ) {
    Chunk y;
#pragma unroll
    for ( int e = 0; e < 8; e += 2 ) {
      y.pair[e / 2] = rounded_pair<E>( acc[a][h][2 * i + ( e >> 2 )][j][e & 3], acc[a][h][2 * i + ( e >> 2 )][j][( e & 3 ) + 1] );
    }
    return y;
  };
  auto added = []( Chunk y, const Chunk& old ) __attribute__( ( always_inline ) ) { // the op that follows the product, on the rounded product
#pragma unroll
    for ( int e = 0; e < 8; e += 2 ) {
      y.pair[e / 2] = rounded_pair<E>( to_f32<E>( old.h[e] ) + to_f32<E>( y.h[e] ), to_f32<E>( old.h[e + 1] ) + to_f32<E>( y.h[e + 1] ) );
    }
    return y;
  };
  if constexpr ( EPI == EPI_PARTIAL ) {
#pragma unroll
    for ( int n = 0; n < 16; n++ ) {
      const int h = n >> 3, j = ( n >> 2 ) & 1, a = ( n >> 1 ) & 1, i = n & 1;
      const uint32_t row = row0 + 128 * a + 32 * i, col = col0 + 128 * h + 16 * j;
      float* dst = o.partial + ( (uint64_t)split * o.b + col ) * o.r + row;
      if ( row + 7 < o.r && col < o.b && ( o.r & 3 ) == 0 ) {
        *reinterpret_cast<mfma_f32x4*>( dst ) = acc[a][h][2 * i][j];
        *reinterpret_cast<mfma_f32x4*>( dst + 4 ) = acc[a][h][2 * i + 1][j];
      } else if ( col < o.b ) {
#pragma unroll
        for ( int e = 0; e < 8; e++ ) {
          if ( row + e < o.r ) {
            dst[e] = acc[a][h][2 * i + ( e >> 2 )][j][e & 3];
          }
        }
      }
    }
    return false;
  }
  if constexpr ( EPI == EPI_GATE || EPI == EPI_BIAS_GATE ) { // tile_row0: of the output
    constexpr bool BIAS = EPI == EPI_BIAS_GATE;
    auto values = [&]( int h, int i, int j, auto act, auto exact ) __attribute__( ( always_inline ) ) {
      Chunk y, y1, y3; // (the rounded factors)
      if constexpr ( !BIAS && !exact.value ) {
        y1 = rounded( 0, h, i, j ), y3 = rounded( 1, h, i, j );
      }
      float g[8];
#pragma unroll
      for ( int e = 0; e < 8; e++ ) {
        const float a1 = acc[0][h][2 * i + ( e >> 2 )][j][e & 3], a3 = acc[1][h][2 * i + ( e >> 2 )][j][e & 3];
        if constexpr ( BIAS ) {
          const float* bias = reinterpret_cast<const float*>( tokens ) + 64 * group + 8 * ( lane >> 4 ) + 32 * i + e;
          g[e] = activate<E>( a1 + bias[0], act ) * ( a3 + bias[TM2 / 2] );
        } else if constexpr ( exact.value ) {
          g[e] = sigmoid_times( a1, a1 ) * a3;
        } else {
          g[e] = sigmoid_times( to_f32<E>( y1.h[e] ), to_f32<E>( y1.h[e] ) ) * to_f32<E>( y3.h[e] );
        }
      }
#pragma unroll
      for ( int e = 0; e < 8; e += 2 ) {
        y.pair[e / 2] = rounded_pair<E>( g[e], g[e + 1] );
      }
      return y;
    };
    E* base = static_cast<E*>( o.xout ) + (uint64_t)col0 * o.gate.stride + row0;
    auto store = [&]( auto all, auto act, auto exact ) __attribute__( ( always_inline ) ) {
#pragma unroll
      for ( int n = 0; n < 8; n++ ) { // (with biases the four outputs of a row in turn)
        const int h = BIAS ? ( n >> 1 ) & 1 : n >> 2, j = BIAS ? n & 1 : ( n >> 1 ) & 1, i = BIAS ? n >> 2 : n & 1;
        const uint32_t col = col0 + 128 * h + 16 * j;
        const Chunk y = values( h, i, j, act, exact );
        if ( all.value
             || ( row0 + 32 * i < o.r && col < o.b && ( o.gate.context_rows == nullptr || o.gate.context_rows[col / o.gate.n_tokens] != nullptr ) ) ) {
          *reinterpret_cast<uint4*>( base + ( 128 * h + 16 * j ) * o.gate.stride + 32 * i ) = y.raw; // r % 8 == 0: eight rows
        }
      }
    };
    if ( ( tile_row0 + TM2 / 2 <= o.r ) & ( tile_col0 + TN2 <= o.b ) & ( o.gate.context_rows == nullptr ) ) {
      if ( BIAS && o.gate.activation == GH_ACT_GELU_TANH ) {
        store( std::true_type {}, std::integral_constant<int, GH_ACT_GELU_TANH> {}, std::true_type {} );
      } else if ( BIAS || o.gate.exact ) {
        store( std::true_type {}, std::integral_constant<int, GH_ACT_SILU> {}, std::true_type {} );
      } else {
        store( std::true_type {}, std::integral_constant<int, GH_ACT_SILU> {}, std::false_type {} );
      }
      return true;
    }
    if ( BIAS || o.gate.exact ) {
      store( std::false_type {}, o.gate.activation, std::true_type {} );
    } else {
      store( std::false_type {}, o.gate.activation, std::false_type {} );
    }
    drain_loads_and_stores();
    return false;
  }
  if constexpr ( EPI == EPI_QKV ) { // a tile's rows are all of q, of k or of v, and 128 rows of whole heads: the angles of rows 128 further on are the same
    const bool to_q = tile_row0 < o.qkv.dim, turn = tile_row0 < o.qkv.dim + o.qkv.kv_dim;
    const E *re = static_cast<const E*>( o.qkv.freq_real ), *im = static_cast<const E*>( o.qkv.freq_imag );
    auto cache_of = [&]( int h, int j ) __attribute__( ( always_inline ) ) {
      return reinterpret_cast<E*>( reinterpret_cast<const uint64_t*>( tokens )[128 * h + 32 * wave + 16 * j + ( lane & 15 )] );
    };
    auto takes_pieces = []( const void* cache ) __attribute__( ( always_inline ) ) { return ( cache != nullptr ) & ( ( reinterpret_cast<uintptr_t>( cache ) & 15u ) == 0 ); };
    // every store of the tile unconditional: all tokens are there, and all their rows take 16 bytes at a time
    const bool aligned = takes_pieces( cache_of( 0, 0 ) ) & takes_pieces( cache_of( 0, 1 ) ) & takes_pieces( cache_of( 1, 0 ) ) & takes_pieces( cache_of( 1, 1 ) );
    const bool whole = ( tile_col0 + TN2 <= o.b ) & ( to_q | (bool)__all( aligned ) );
    union Angles
    {
      uint2 raw;
      E h[4];
    };
    auto store = [&]( auto turned, auto all ) __attribute__( ( always_inline ) ) {
      Angles cs[2][2][2], sn[2][2][2]; // [token half][token][32 rows]
      if constexpr ( turned.value ) {
#pragma unroll
        for ( int n = 0; n < 8; n++ ) {
          const int h = n >> 2, j = ( n >> 1 ) & 1, i = n & 1;
          const uint32_t at = cache_of( h, j ) != nullptr ? tokens[2 * TN2 + 128 * h + 32 * wave + 16 * j + ( lane & 15 )] : 0;
          const uint64_t k = (uint64_t)at * ( o.qkv.head_size / 2 ) + ( ( row0 + 32 * i ) % o.qkv.head_size ) / 2;
          cs[h][j][i].raw = *reinterpret_cast<const uint2*>( re + k );
          sn[h][j][i].raw = *reinterpret_cast<const uint2*>( im + k );
        }
      }
#pragma unroll
      for ( int n = 0; n < 16; n++ ) {
        const int h = n >> 3, j = ( n >> 2 ) & 1, a = ( n >> 1 ) & 1, i = n & 1;
        const uint32_t row = row0 + 128 * a + 32 * i, col = col0 + 128 * h + 16 * j;
        E* const own = cache_of( h, j );
        Chunk y = rounded( a, h, i, j );
        if ( turned.value && own != nullptr ) {
#pragma unroll
          for ( int e = 0; e < 4; e++ ) {
            const float c = to_f32<E>( cs[h][j][i].h[e] ), s = to_f32<E>( sn[h][j][i].h[e] ), y0 = to_f32<E>( y.h[2 * e] ), y1 = to_f32<E>( y.h[2 * e + 1] );
            y.h[2 * e] = from_f32<E>( y0 * c - y1 * s );
            y.h[2 * e + 1] = from_f32<E>( y0 * s + y1 * c );
          }
        }
        E* dst = to_q ? static_cast<E*>( o.xout ) + (uint64_t)col * o.qkv.dim + row : own + ( row - o.qkv.dim );
        if ( all.value || ( col < o.b && ( to_q || takes_pieces( own ) ) ) ) {
          *reinterpret_cast<uint4*>( dst ) = y.raw;
        } else if ( col < o.b && own != nullptr ) {
#pragma unroll
          for ( int e = 0; e < 8; e++ ) {
            dst[e] = y.h[e];
          }
        }
      }
    };
    if ( whole & turn ) {
      store( std::true_type {}, std::true_type {} );
      return true;
    }
    if ( whole ) {
      store( std::false_type {}, std::true_type {} );
      return true;
    }
    turn ? store( std::true_type {}, std::false_type {} ) : store( std::false_type {}, std::false_type {} );
    drain_loads_and_stores();
    return false;
  }
  // two products that share their activations in one launch: a tile of one of them, or of both
  const bool second = tile_row0 >= o.r_first;
  if ( ( tile_row0 + TM2 <= o.r ) & ( tile_col0 + TN2 <= o.b ) & ( ( o.r & 7 ) == 0 ) & ( second | ( tile_row0 + TM2 <= o.r_first ) ) ) {
    const uint64_t ld = second ? o.r - o.r_first : o.r_first;
    E* base = static_cast<E*>( second ? o.xout2 : o.xout ) + (uint64_t)col0 * ld + ( row0 - ( second ? o.r_first : 0 ) );
    Chunk old[EPI == EPI_ACCUM ? 16 : 1]; // all of them before the first store, which a load behind it would wait for
    if constexpr ( EPI == EPI_ACCUM ) {
#pragma unroll
      for ( int n = 0; n < 16; n++ ) {
        old[n].raw = *reinterpret_cast<const uint4*>( base + ( 128 * ( n >> 3 ) + 16 * ( ( n >> 2 ) & 1 ) ) * ld + 128 * ( ( n >> 1 ) & 1 ) + 32 * ( n & 1 ) );
      }
    }
#pragma unroll
    for ( int n = 0; n < 16; n++ ) {
      const int h = n >> 3, j = ( n >> 2 ) & 1, a = ( n >> 1 ) & 1, i = n & 1;
      Chunk y = rounded( a, h, i, j );
      if constexpr ( EPI == EPI_ACCUM ) {
        y = added( y, old[n] );
      }
      *reinterpret_cast<uint4*>( base + ( 128 * h + 16 * j ) * ld + 128 * a + 32 * i ) = y.raw;
    }
    return true;
  }
#pragma unroll
  for ( int n = 0; n < 16; n++ ) {
    const int h = n >> 3, j = ( n >> 2 ) & 1, a = ( n >> 1 ) & 1, i = n & 1;
    const uint32_t row = row0 + 128 * a + 32 * i, col = col0 + 128 * h + 16 * j;
    if ( row >= o.r || col >= o.b ) {
      continue;
    }
    Chunk y = rounded( a, h, i, j );
    if ( ( o.r & 7 ) == 0 ) { // (r_first % 8 == 0: eight rows never straddle the two outputs)
      const bool in_second = row >= o.r_first;
      uint4* dst = reinterpret_cast<uint4*>( in_second ? static_cast<E*>( o.xout2 ) + (uint64_t)col * ( o.r - o.r_first ) + ( row - o.r_first )
                                                       : static_cast<E*>( o.xout ) + (uint64_t)col * o.r_first + row );
      if ( EPI == EPI_ACCUM ) {
        Chunk old;
        old.raw = *dst;
        y = added( y, old );
      }
      *dst = y.raw;
    } else { // (one output only: the launch refuses two, and the residual add, with r % 8 != 0)
#pragma unroll
      for ( int e = 0; e < 8; e++ ) {
        if ( row + e < o.r ) {
          static_cast<E*>( o.xout )[(uint64_t)col * o.r + row + e] = y.h[e];
        }
      }
    }
  }
  drain_loads_and_stores();
  return false;
}

// grid: 8 x (work-groups of one XCD) by K splits (more than one only with EPI_PARTIAL: split z leaves its sums in partial[z]).
// k_len: k per split.  s % 64 == 0, k_len % 64 == 0, at least two steps a split, 16-byte aligned operands.
// WALK: a work-group takes tile after tile; an even number of steps, so that a tile finds the stages as the last one did, and one split.
template<typename E, int EPI, bool WALK>
__global__ __launch_bounds__( T256_THREADS, 1 ) void gemm_tile256_kernel( const E* __restrict__ x, const E* __restrict__ w, uint32_t s, uint32_t k_len, TileOut out, TileOrder ord )
{
  // Separate arrays: the compiler keeps an LDS read behind the loads into its own array only.  W: the weight rows' halves, X: all tokens.
  __shared__ uint4 s_wa0[128 * 8], s_wb0[128 * 8], s_x0[256 * 8];
  __shared__ uint4 s_wa1[128 * 8], s_wb1[128 * 8], s_x1[256 * 8];
  // EPI_QKV: cache rows and positions of a tile's tokens, left here at the end of the tile before: read where they are needed they would be one more round
  // trip a tile with nothing beside it.  Two of them, as a wave may be through with a tile while others still store it.
  // EPI_BIAS_GATE: its biases, likewise.
  __shared__ __align__( 16 ) uint32_t s_tokens[2][EPI == EPI_QKV ? 3 * TN2 : EPI == EPI_BIAS_GATE ? TM2 : 1];
  constexpr bool GATE = EPI == EPI_GATE || EPI == EPI_BIAS_GATE;
  typedef typename Mfma<E>::x8 x8;
  const uint32_t xcd = blockIdx.x & 7; // work-groups go to the XCDs in turn
  uint32_t idx = blockIdx.x >> 3;
  uint32_t row_tile = 0, token_tile = 0;
  if ( !tile_of_index( ord, xcd, idx, row_tile, token_tile ) ) {
    return; // (whole work-group)
  }
  const uint32_t all_waves = __builtin_amdgcn_readfirstlane( threadIdx.x >> 6 );
  const uint32_t lane = threadIdx.x & 63, group = all_waves >> 2, wave = all_waves & 3;
  const uint32_t fr = lane & 15, g4 = lane >> 4;
  const uint32_t ld_bytes = s * 2;
  const uint32_t k0 = blockIdx.y * k_len;
  const uint32_t n_steps = min( k_len, s - k0 ) / TKS;
  // Half tiles: 128 rows, two instructions of 64 rows (8 a wave); a lane writes slot lane % 8 of row lane / 8, so it fetches the chunk
  // that the swizzle keeps there.
  uint32_t w_off[4], x_off[4];
#pragma unroll
  for ( int i = 0; i < 4; i++ ) {
    const uint32_t row = threadIdx.x >> 3, slot = threadIdx.x & 7;
    w_off[i] = ( row + 64 * i ) * ld_bytes + ( slot ^ w_swizzle( row ) ) * 16;
    x_off[i] = ( row + 64 * i ) * ld_bytes + ( slot ^ x_swizzle( row ) ) * 16;
  }
  constexpr uint32_t ROWS = GATE ? TM2 / 2 : TM2; // output rows of a tile
  const uint64_t w3_bytes = (uint64_t)out.r * ld_bytes;      // the gates: from a row of w1 to its row of w3
  struct Operands // of a tile: first byte of this split's k range and bytes from there to the end of its last row
  {
    const char *w, *x;
    uint32_t w_bytes, x_bytes;
  };
  auto operands_of = [&]( uint32_t rt, uint32_t tt ) __attribute__( ( always_inline ) ) {
    Operands p;
    p.w = reinterpret_cast<const char*>( w + (uint64_t)rt * ROWS * s + k0 );
    p.x = reinterpret_cast<const char*>( x + (uint64_t)tt * TN2 * s + k0 );
    p.w_bytes = min( ROWS, out.r - rt * ROWS ) * ld_bytes - k0 * 2;
    p.x_bytes = min( (uint32_t)TN2, out.b - tt * TN2 ) * ld_bytes - k0 * 2;
    return p;
  };
  Operands cur = operands_of( row_tile, token_tile ), next = cur;
  bool more = false; // `next` holds another tile
  // half tile `half` of a step; the steps behind the last are the first of the next tile, or nothing: an offset past the descriptor's end
  // (the scalar offset takes part in the range check) reads zero and costs no traffic
  auto k_bytes = [&]( uint32_t step ) __attribute__( ( always_inline ) ) {
    return step < n_steps ? step * ( TKS * 2 ) : WALK && more ? ( step - n_steps ) * ( TKS * 2 ) : 0x80000000u;
  };
  auto fetch_w = [&]( uint4* tile, int half, uint32_t step ) __attribute__( ( always_inline ) ) {
    const Operands& p = WALK && step >= n_steps ? next : cur;
    const char* base = GATE && half == 1 ? p.w + w3_bytes : p.w;
    const int row = GATE ? 0 : 2 * half;
    const __amdgpu_buffer_rsrc_t rsrc = __builtin_amdgcn_make_buffer_rsrc( const_cast<char*>( base ), 0, (int)p.w_bytes, 0x00020000 );
    const uint32_t kb = k_bytes( step );
    __builtin_amdgcn_raw_ptr_buffer_load_lds( rsrc, (lds_ptr)( tile + 64 * all_waves ), 16, w_off[row], kb, 0, 0 );
    __builtin_amdgcn_raw_ptr_buffer_load_lds( rsrc, (lds_ptr)( tile + 64 * 8 + 64 * all_waves ), 16, w_off[row + 1], kb, 0, 0 );
  };
  auto fetch_x = [&]( uint4* tile, int half, uint32_t step ) __attribute__( ( always_inline ) ) {
    const Operands& p = WALK && step >= n_steps ? next : cur;
    const __amdgpu_buffer_rsrc_t rsrc = __builtin_amdgcn_make_buffer_rsrc( const_cast<char*>( p.x ), 0, (int)p.x_bytes, 0x00020000 );
    const uint32_t kb = k_bytes( step );
    __builtin_amdgcn_raw_ptr_buffer_load_lds( rsrc, (lds_ptr)( tile + 128 * 8 * half + 64 * all_waves ), 16, x_off[2 * half], kb, 0, 0 );
    __builtin_amdgcn_raw_ptr_buffer_load_lds( rsrc, (lds_ptr)( tile + 128 * 8 * half + 64 * 8 + 64 * all_waves ), 16, x_off[2 * half + 1], kb, 0, 0 );
  };

  mfma_f32x4 acc[2][2][4][2];
  x8 fw[4][2], fx[2][2][2]; // [row tile][k half], [token half][token tile][k half]
  const uint32_t w_row = 64 * group + 8 * ( fr >> 2 ) + ( fr & 3 ), x_row = 32 * wave + fr;
  auto read_w = [&]( const uint4* tile ) __attribute__( ( always_inline ) ) {
#pragma unroll
    for ( int k = 0; k < 2; k++ ) {
#pragma unroll
      for ( int i = 0; i < 4; i++ ) {
        const uint32_t row = w_row + 32 * ( i >> 1 ) + 4 * ( i & 1 );
        fw[i][k] = __builtin_bit_cast( x8, tile[row * 8 + ( ( 4 * k + g4 ) ^ w_swizzle( row ) )] );
      }
    }
  };
  auto read_x = [&]( const uint4* tile ) __attribute__( ( always_inline ) ) {
#pragma unroll
    for ( int h = 0; h < 2; h++ ) {
#pragma unroll
      for ( int k = 0; k < 2; k++ ) {
#pragma unroll
        for ( int j = 0; j < 2; j++ ) {
          const uint32_t row = x_row + 16 * j;
          fx[h][j][k] = __builtin_bit_cast( x8, tile[( 128 * h + row ) * 8 + ( ( 4 * k + g4 ) ^ x_swizzle( row ) )] );
        }
      }
    }
  };
  auto multiply = [&]( auto a, int h ) __attribute__( ( always_inline ) ) {
#pragma unroll
    for ( int k = 0; k < 2; k++ ) {
#pragma unroll
      for ( int i = 0; i < 4; i++ ) {
#pragma unroll
        for ( int j = 0; j < 2; j++ ) {
          acc[a.value][h][i][j] = Mfma<E>::k32( fw[i][k], fx[h][j][k], acc[a.value][h][i][j] );
        }
      }
    }
  };
  constexpr std::integral_constant<int, 0> upper {};
  constexpr std::integral_constant<int, 1> lower {};
  auto barrier = []() __attribute__( ( always_inline ) ) {
    __builtin_amdgcn_sched_barrier( 0 );
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier( 0 );
  };
  // The end of a memory part: this wave's reads are here, and all of its loads but the youngest 8, which leaves what the next part reads
  // in LDS (the barrier makes that all waves').  `stores`: the last tile's stores are still counted behind the loads this waits for.
  constexpr int STORES = GATE ? 8 : 16;
  auto arrive = [&]( bool stores ) __attribute__( ( always_inline ) ) {
    __builtin_amdgcn_sched_barrier( 0 );
    if ( stores ) {
      __builtin_amdgcn_s_waitcnt( 0x0070 | ( ( 8 + STORES ) & 15 ) | ( ( ( 8 + STORES ) >> 4 ) << 14 ) ); // lgkmcnt(0), vmcnt(8 + STORES)
    } else {
      __builtin_amdgcn_s_waitcnt( 0x0078 ); // lgkmcnt(0), vmcnt(8)
    }
    barrier();
  };
  auto step = [&]( uint4* wa, uint4* wb, uint4* xs, uint4* wb_other, uint32_t j, bool stores ) __attribute__( ( always_inline ) ) {
    read_w( wa );
    read_x( xs );
    __builtin_amdgcn_sched_barrier( 0 ); // the reads first: behind the loads they would wait for room in the address unit's queue
    fetch_w( wb_other, 1, j + 1 );
    arrive( stores );
    multiply( upper, 0 );
    multiply( upper, 1 );
    barrier();
    read_w( wb );
    __builtin_amdgcn_sched_barrier( 0 );
    fetch_w( wa, 0, j + 2 );
    fetch_x( xs, 0, j + 2 );
    fetch_x( xs, 1, j + 2 );
    arrive( stores );
    multiply( lower, 1 );
    multiply( lower, 0 );
    barrier();
  };
  // (no branch around loads and stores: what the compiler cannot count it waits for)
  struct Token
  {
    uint64_t row;
    uint32_t pos;
    float bias;
  };
  auto token_of = [&]( uint32_t rt, uint32_t tt ) __attribute__( ( always_inline ) ) {
    Token token { 0, 0, 0.0f };
    if constexpr ( EPI == EPI_QKV ) {
      const uint32_t col = min( tt * TN2 + ( threadIdx.x & ( TN2 - 1 ) ), out.b - 1 );
      token.row = reinterpret_cast<const uint64_t*>( out.qkv.token_rows )[col];
      token.pos = out.qkv.pos[col];
    }
    if constexpr ( EPI == EPI_BIAS_GATE ) { // (without biases any value that can be read)
      const uint32_t row = min( rt * ROWS + ( threadIdx.x & ( ROWS - 1 ) ), out.r - 1 );
      const E* bias = out.gate.bias != nullptr ? static_cast<const E*>( out.gate.bias ) : w;
      const float value = to_f32<E>( bias[( threadIdx.x & ROWS ) != 0 ? (uint64_t)out.r + row : row] );
      token.bias = out.gate.bias != nullptr ? value : 0.0f;
    }
    return token;
  };
  auto keep_token = [&]( uint32_t* tokens, const Token& token ) __attribute__( ( always_inline ) ) {
    if constexpr ( EPI == EPI_QKV ) { // (by two threads each)
      reinterpret_cast<uint64_t*>( tokens )[threadIdx.x & ( TN2 - 1 )] = token.row;
      tokens[2 * TN2 + ( threadIdx.x & ( TN2 - 1 ) )] = token.pos;
    }
    if constexpr ( EPI == EPI_BIAS_GATE ) {
      reinterpret_cast<float*>( tokens )[threadIdx.x & ( TM2 - 1 )] = token.bias;
    }
  };
  keep_token( s_tokens[0], token_of( row_tile, token_tile ) );
  fetch_w( s_wa0, 0, 0 );
  fetch_x( s_x0, 0, 0 );
  fetch_x( s_x0, 1, 0 );
  fetch_w( s_wb0, 1, 0 );
  fetch_w( s_wa1, 0, 1 );
  fetch_x( s_x1, 0, 1 );
  fetch_x( s_x1, 1, 1 );
  // vmcnt(8): step 0 up to its second half of weight rows.  WALK: vmcnt(0), as what is outstanding here is what the compiler, which waits before it reads
  // what loads leave in LDS, allows for in every tile: the first reads of the second and later ones would wait for the stores in between.
  __builtin_amdgcn_s_waitcnt( WALK ? 0x0F70 : 0x0F78 );
  barrier();
  if ( group == 1 ) {
    barrier();
  }
  auto clear = [&]() __attribute__( ( always_inline ) ) {
#pragma unroll
    for ( int n = 0; n < 32; n++ ) {
      acc[n >> 4][( n >> 3 ) & 1][( n >> 1 ) & 3][n & 1] = mfma_f32x4 { 0.0f, 0.0f, 0.0f, 0.0f };
    }
  };
  uint32_t j = 0;
  if constexpr ( WALK ) {
    bool stores = false;
    for ( uint32_t tile = 0;; tile++ ) {
      uint32_t next_row = 0, next_token = 0;
      idx += gridDim.x >> 3;
      more = tile_of_index( ord, xcd, idx, next_row, next_token );
      if ( more ) {
        next = operands_of( next_row, next_token );
      }
      clear();
      j = 0;
      do { // (an even number of steps)
        step( s_wa0, s_wb0, s_x0, s_wb1, j, stores && j == 0 );
        step( s_wa1, s_wb1, s_x1, s_wb0, j + 1, false );
        j += 2;
      } while ( j < n_steps );
      if ( !more ) {
        __builtin_amdgcn_s_waitcnt( 0x0F70 ); // vmcnt(0): no load-to-LDS outlives the work-group
      }
      const Token token = token_of( more ? next_row : row_tile, more ? next_token : token_tile );
      stores = store_tile<E, EPI>( acc, out, row_tile * ROWS, token_tile * TN2, group, wave, lane, 0, s_tokens[tile & 1] );
      keep_token( s_tokens[( tile + 1 ) & 1], token );
      if ( !more ) {
        break;
      }
      cur = next;
      row_tile = next_row;
      token_tile = next_token;
    }
  } else {
    clear();
    for ( ; j + 2 <= n_steps; j += 2 ) {
      step( s_wa0, s_wb0, s_x0, s_wb1, j, false );
      step( s_wa1, s_wb1, s_x1, s_wb0, j + 1, false );
    }
    if ( j < n_steps ) {
      step( s_wa0, s_wb0, s_x0, s_wb1, j, false );
    }
    __builtin_amdgcn_s_waitcnt( 0x0F70 );
    store_tile<E, EPI>( acc, out, row_tile * ROWS, token_tile * TN2, group, wave, lane, blockIdx.y, s_tokens[0] );
  }
  if ( group == 0 ) {
    barrier();
  }
}

int g_tile_rows = 0; // tuning hook: non-zero leaves every product whole (no cut along the tokens)

uint64_t cus_per_xcd() { return std::max<uint64_t>( 1, (uint64_t)cu_count() / 8 ); } // 32

// Rounds of one work-group per CU that an XCD runs for its share of the tiles.
uint64_t rounds_per_xcd( uint64_t r, uint64_t b )
{
  const uint64_t row_tiles = ( r + TM2 - 1 ) / TM2, token_tiles = ( b + TN2 - 1 ) / TN2;
  const uint64_t tiles = ( row_tiles / 8 ) * token_tiles + ( ( row_tiles % 8 ) * token_tiles + 7 ) / 8;
  return ( tiles + cus_per_xcd() - 1 ) / cus_per_xcd();
}

} // namespace

void gemm_tile256_tuning( int rows ) { g_tile_rows = rows; }

bool gemm_tile256_takes( uint64_t s, uint64_t b, const void* x, const void* w, const void* xout )
{
  return b >= 192 && s % TKS == 0 && s >= 2 * TKS && s < ( 1u << 22 )
         && ( ( reinterpret_cast<uintptr_t>( x ) | reinterpret_cast<uintptr_t>( w ) | reinterpret_cast<uintptr_t>( xout ) ) & 15u ) == 0;
}

// Enough tiles to fill the chip without a K split, and no last round that is mostly empty: what the forced kernel takes.
bool gemm_tile256_fills( uint64_t r, uint64_t b )
{
  const uint64_t tiles = ( ( r + TM2 - 1 ) / TM2 ) * ( ( b + TN2 - 1 ) / TN2 );
  const uint64_t cus = (uint64_t)cu_count(), rounds = ( tiles + cus - 1 ) / cus;
  return 4 * tiles >= 3 * cus && 10 * tiles >= 6 * rounds * cus;
}

// `rounds` of one work-group per CU, `units` work-groups in all.  A step of 64 k takes 1 us while few CUs multiply and 1.37 when all do and
// the clock drops (70B w2, 448 steps: 200 tokens 483 us, 1024 511, 2048 616, 3328 in two rounds 1155), a round's ends 3.5, and up to 3 more that a
// long K range hides (14 rounds of 2, 8, 16 and 32 steps, 32000 rows at 7000 tokens: 126, 248, 383 and 667 us).  With a single row of
// token tiles no work-group shares its weights and all of them come from memory at once: 2 us when all CUs ask (256 tokens of 57344 x 8192,
// 224 tiles, 128 steps: 1.83 us a step; 32000 x 8192, 125 tiles: 1.48; 10240 x 8192, 40: 1.1), less with fewer tokens beside them (28672 x 8192, 112
// tiles: 1.47 at 256 tokens, 1.41 at 224, 1.27 at 192), but not where a K split asks in several places (8192 x 28672 in 8 at 192 tokens: 1.9).
static double rounds_ns( uint64_t rounds, uint64_t units, uint64_t steps, uint64_t b, bool split )
{
  const double busy = (double)units / (double)( rounds * (uint64_t)cu_count() );
  const double step_ns = b > TN2 ? 1000.0 + 370.0 * busy * busy : 1000.0 + busy * ( split ? 1000.0 : 1800.0 * (double)b / TN2 - 800.0 );
  return (double)rounds * ( (double)steps * step_ns + 3500.0 + 3000.0 * std::min( 1.0, 16.0 / (double)steps ) ) + 1000.0;
}
double gemm_tile256_ns( uint64_t s, uint64_t r, uint64_t b )
{
  return rounds_ns( rounds_per_xcd( r, b ), ( ( r + TM2 - 1 ) / TM2 ) * ( ( b + TN2 - 1 ) / TN2 ), s / TKS, b, false );
}

// A launch is as slow as its number of rounds, so a product whose tiles leave the last round partly empty pays for a whole round there:
// 8192 rows x 3328 tokens are 416 tiles, 1.6 rounds, and take 2.  Such a product may be cut in two along the tokens: the first part as
// many tokens as fill `rounds` rounds, the rest a product of its own (the K range split over work-groups, or smaller tiles).  Returns
// those tokens, 0 if there are none.
uint64_t gemm_tile256_tokens( uint64_t r, uint64_t b, uint64_t rounds )
{
  for ( uint64_t t = ( b - 1 ) / TN2; g_tile_rows == 0 && t >= 1; t-- ) {
    if ( rounds_per_xcd( r, t * TN2 ) <= rounds ) {
      return t * TN2;
    }
  }
  return 0;
}
uint64_t gemm_tile256_rounds( uint64_t r, uint64_t b ) { return rounds_per_xcd( r, b ); }

// The K range of each tile split over several work-groups, the fp32 sums of each split to partial[split].  *splits = 0: not for this
// shape.  The sums are written and read.
void gemm_tile256_split_plan( uint64_t s, uint64_t r, uint64_t b, uint32_t* splits, uint32_t* k_len, double* ns )
{
  *splits = 0;
  *k_len = 0;
  *ns = 0.0;
  const uint64_t tiles = ( ( r + TM2 - 1 ) / TM2 ) * ( ( b + TN2 - 1 ) / TN2 );
  const uint64_t cus = (uint64_t)cu_count(), steps = s / TKS;
  if ( b < 192 || tiles > 2 * cus || s % TKS != 0 || s >= ( 1u << 22 ) ) {
    return;
  }
  for ( uint64_t want = 2; want <= 16; want++ ) {
    const uint64_t per = ( steps + want - 1 ) / want, n = ( steps + per - 1 ) / per;
    if ( per < 12 || n != want ) {
      continue;
    }
    const double cost = rounds_ns( ( tiles * n + cus - 1 ) / cus, tiles * n, per, b, true ) + (double)( n * b * r ) * 8.0 / 5000.0;
    if ( *splits == 0 || cost < *ns ) {
      *splits = (uint32_t)n;
      *k_len = (uint32_t)( per * TKS );
      *ns = cost;
    }
  }
  if ( b > 3 * TN2 ) { // 3 to 10 % less than that where four and more token tiles share weights (5120 x 5120: 1000 tokens 63 us, the ring kernel 76; 1500: 83 and 91)
    *ns *= 0.96;
  }
}

// Tiles that lie in one of q, k and v, whole heads in 128 rows, angles that are read four at a time.
bool gemm_tile256_qkv_fits( const QkvRows& q )
{
  return q.dim % TM2 == 0 && q.kv_dim % TM2 == 0 && q.head_size >= 8 && 128 % q.head_size == 0
         && ( ( reinterpret_cast<uintptr_t>( q.freq_real ) | reinterpret_cast<uintptr_t>( q.freq_imag ) ) & 7u ) == 0;
}

// `partial` != nullptr: fp32 sums (splits, b, r) instead of xout; else `epilogue` 0 stores, 1 accumulates into xout (needs r % 8 == 0), 2 gates
// (2 r weight rows, `gate`), 4 rotates and appends (`qkv`; xout: q).
// splits > 1 (from gemm_tile256_split_plan, with its k_len) needs `partial`.
template<typename E>
int gemm_tile256_launch( E* xout, float* partial, const E* x, const E* w, uint64_t s, uint64_t r, uint64_t b, int epilogue, hipStream_t st, uint32_t splits,
                         uint32_t k_len, E* xout2, uint64_t r_first, const GateRows* gate, const QkvRows* qkv )
{
  if ( xout2 == nullptr ) {
    r_first = r;
  }
  GH_REQUIRE( xout2 == nullptr || ( partial == nullptr && epilogue == EPI_STORE && splits == 1 && r % 8 == 0 && r_first % 8 == 0 && r_first > 0 && r_first < r ),
              "gh_matmul: two outputs need plain stores, no K split and row counts that are multiples of 8" );
  GH_REQUIRE( splits >= 1 && ( splits == 1 || ( partial != nullptr && k_len % TKS == 0 && (uint64_t)k_len * splits >= s && (uint64_t)k_len * ( splits - 1 ) < s ) ),
              "gh_matmul: bad K split for the 256-token tile kernel" );
  if ( splits == 1 ) {
    k_len = (uint32_t)s;
  }
  const bool plain_gate = gate != nullptr && gate->activation == GH_ACT_SILU && gate->bias == nullptr;
  const int epi = partial != nullptr ? EPI_PARTIAL : epilogue == EPI_GATE && !plain_gate ? EPI_BIAS_GATE : epilogue;
  GH_REQUIRE( epi == EPI_STORE || epi == EPI_ACCUM || epi == EPI_PARTIAL || ( epi == EPI_QKV && qkv != nullptr && gemm_tile256_qkv_fits( *qkv ) )
                || ( ( epi == EPI_GATE || ( epi == EPI_BIAS_GATE && gate != nullptr && gate->exact && std::is_same_v<E, __bf16> ) ) && r % 8 == 0 && gate->stride % 8 == 0 ),
              "gh_matmul: unknown tile epilogue %d", epi );
  GH_REQUIRE( epi != EPI_ACCUM || r % 8 == 0, "gh_matmul: the accumulating tile epilogue needs r %% 8 == 0" );
  const uint64_t tile_rows = epi == EPI_GATE || epi == EPI_BIAS_GATE ? TM2 / 2 : TM2;
  const uint32_t row_tiles = (uint32_t)( ( r + tile_rows - 1 ) / tile_rows );
  TileOrder ord;
  ord.token_tiles = (uint32_t)( ( b + TN2 - 1 ) / TN2 );
  // Whole row tiles per XCD, the weights of each read into one L2 only, where that takes no more rounds of the XCD's 32 CUs than an even
  // share of all tiles (13824 x 5120 at 16384 tokens, 54 row tiles: 14 either way, 1 % faster); else the row tiles beyond a multiple
  // of 8 are shared out (20 row tiles: 5 rounds against 6; with 4 splits of 3 token tiles 32 work-groups per XCD against 36, 110 us against 149).
  const uint64_t tokens = ord.token_tiles, even = ( row_tiles / 8 ) * tokens + ( ( row_tiles % 8 ) * tokens + 7 ) / 8, whole = ( row_tiles + 7 ) / 8 * tokens;
  const uint64_t per_cu = cus_per_xcd();
  ord.rest_rows = ( whole * splits + per_cu - 1 ) / per_cu <= ( even * splits + per_cu - 1 ) / per_cu ? 0 : row_tiles % 8;
  ord.owned = row_tiles - ord.rest_rows;
  // The 32 tiles an XCD works on at a time read gm + gn operand strips into its L2: strips of equal height, at most 6 row tiles, and
  // patches of equal width that make 32 tiles with that (6 x 5: 11 strips; heights of 4 and 2 with patches 8 wide: 12 and 18).
  auto even_part = []( uint32_t n, uint32_t most ) { return n == 0 ? 1 : ( n + ( n + most - 1 ) / most - 1 ) / ( ( n + most - 1 ) / most ); };
  ord.gm = even_part( ( ord.owned + 7 ) / 8, 6 );
  ord.gn = even_part( ord.token_tiles, ( 32 + ord.gm / 2 ) / ord.gm );
  ord.rest_gn = even_part( ord.token_tiles, ( 32 + ord.rest_rows / 2 ) / std::max( 1u, ord.rest_rows ) );
  ord.rest_share = (uint32_t)( ( (uint64_t)ord.rest_rows * tokens + 7 ) / 8 );
  const uint64_t per_xcd = ord.rest_rows == 0 ? whole : even; // the longest list
  GH_REQUIRE( 8 * per_xcd < ( 1ull << 31 ), "gh_matmul: grid too large" );
  const TileOut out { xout, xout2, partial, (uint32_t)r, (uint32_t)b, (uint32_t)r_first, gate != nullptr ? *gate : GateRows {}, qkv != nullptr ? *qkv : QkvRows {} };
  const bool walk = per_xcd > per_cu && epi != EPI_PARTIAL && s % ( 2 * TKS ) == 0;
  const dim3 grid( (unsigned)( 8 * ( walk ? per_cu : per_xcd ) ), splits );
#define GH_TILE256( EP, WALK ) gemm_tile256_kernel<E, EP, WALK><<<grid, T256_THREADS, 0, st>>>( x, w, (uint32_t)s, k_len, out, ord )
  switch ( epi ) {
    case EPI_STORE: walk ? GH_TILE256( EPI_STORE, true ) : GH_TILE256( EPI_STORE, false ); break;
    case EPI_ACCUM: walk ? GH_TILE256( EPI_ACCUM, true ) : GH_TILE256( EPI_ACCUM, false ); break;
    case EPI_GATE: walk ? GH_TILE256( EPI_GATE, true ) : GH_TILE256( EPI_GATE, false ); break;
    case EPI_BIAS_GATE:
      if constexpr ( std::is_same_v<E, __bf16> ) {
        walk ? GH_TILE256( EPI_BIAS_GATE, true ) : GH_TILE256( EPI_BIAS_GATE, false );
      }
      break;
    case EPI_QKV:
      if constexpr ( std::is_same_v<E, __half> ) {
        walk ? GH_TILE256( EPI_QKV, true ) : GH_TILE256( EPI_QKV, false );
      }
      break;
    default: GH_TILE256( EPI_PARTIAL, false ); break;
  }
#undef GH_TILE256
  GH_LAUNCH_CHECK();
  return GH_OK;
}

template int gemm_tile256_launch<__half>( __half*, float*, const __half*, const __half*, uint64_t, uint64_t, uint64_t, int, hipStream_t, uint32_t, uint32_t,
                                          __half*, uint64_t, const GateRows*, const QkvRows* );
template int gemm_tile256_launch<__bf16>( __bf16*, float*, const __bf16*, const __bf16*, uint64_t, uint64_t, uint64_t, int, hipStream_t, uint32_t, uint32_t,
                                          __bf16*, uint64_t, const GateRows*, const QkvRows* );

} // namespace gh
