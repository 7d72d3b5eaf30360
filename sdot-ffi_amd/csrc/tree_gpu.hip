// The BSP tree built on the device, no host round trip: median cut on the longest axis, leaf <= `leaf`, perfect binary tree
// in preorder, each leaf's seeds in ascending user index.
//
// How ( this build's own scheme; the reference's card builder is `gpu/Bsp2D.cuh:367` ):
//   1. a stable LSD radix sort of the seeds along each axis, the axes in the same launches ( 64-bit order-preserving keys of the
//      doubles, 8 passes of 8 bits; the in-tile rank of an element among its digit's is found with wave64 ballots; a pass is
//      histogram / scan of each digit's tiles / scatter );
//   2. per level, every node's slice is a contiguous segment of EVERY sorted list, so its box is read off the segments' ends; the
//      median cut on the longest axis takes the first half of that axis' list as is, and the other lists are stably partitioned by
//      the flags the cut writes ( an exclusive scan over all positions ): the lists stay sorted inside every child. Five launches a
//      level: the nodes, the flags, the scan in two, the partition, which also hands each position its child;
//   3. the leaves' seeds sorted by user index, the preorder numbering and the rank tables.
// Everything stays on the device; the host only issues launches ( their count is a function of `n` ) and waits for none of them.
// A cloud of at most `SMALL_TREE` seeds is built by ONE workgroup with its lists in LDS ( `k_small_tree` ): the ~100 launches take ~0.25 ms
// whatever they do. The line is where the two cross: the workgroup's sorting networks double at every power of two. Masses of a Voronoi
// diagram, us a call by one workgroup / by launches: 2D 500 seeds 266 / 398, 2000 333 / 475, 4096 418 / 520; 3D 500 356 / 470, 2000 490 / 597,
// 4096 663 / 704; with room for 8192 in it, 2D 5000 555 / 560, 8192 600 / 562; 3D 5000 895 / 761, 8192 1110 / 923.

#include "tree.h"
#include "tree3.h"

namespace sdot_amd {

namespace {

constexpr int RS_THREADS = 256;
constexpr int RS_ITEMS = 8;
constexpr int RS_TILE = RS_THREADS * RS_ITEMS;

__device__ __forceinline__ unsigned long long dkey( double x ) {
    unsigned long long u = __double_as_longlong( x );
    return ( u >> 63 ) ? ~u : ( u | 0x8000000000000000ull );
}

/// the keys of every axis ( `dim` coordinates a seed; the grid's second index ), and the identity permutation
__global__ void k_keys( I64 n, const double *pos, int dim, unsigned long long *key, int *val ) {
    const I64 i = I64( blockIdx.x ) * blockDim.x + threadIdx.x;
    if ( i >= n ) return;
    const int axis = blockIdx.y;
    key[ axis * n + i ] = dkey( pos[ dim * i + axis ] );
    val[ axis * n + i ] = int( i );
}

/// histogram of digit `shift` per tile: `hist[ ( axis 256 + digit ) nt + tile ]`
__global__ __launch_bounds__( RS_THREADS ) void k_rs_hist( I64 n, const unsigned long long *keys, int shift, int nt, unsigned *hist ) {
    __shared__ unsigned h[ 256 ];
    h[ threadIdx.x ] = 0;
    __syncthreads();
    const unsigned long long *key = keys + blockIdx.y * n;
    const I64 base = I64( blockIdx.x ) * RS_TILE;
    for ( int j = 0; j < RS_ITEMS; ++j ) {
        const I64 i = base + j * RS_THREADS + threadIdx.x;
        if ( i < n ) atomicAdd( &h[ ( key[ i ] >> shift ) & 255 ], 1u );
    }
    __syncthreads();
    hist[ ( size_t( blockIdx.y ) * 256 + threadIdx.x ) * nt + blockIdx.x ] = h[ threadIdx.x ];
}

__device__ __forceinline__ unsigned wave_inclusive( unsigned v ) {
    const int lane = threadIdx.x & 63;
    for ( int o = 1; o < 64; o <<= 1 ) { const unsigned t = __shfl_up( v, o, 64 ); if ( lane >= o ) v += t; }
    return v;
}
/// the exclusive prefix of `v` over the block's `T` threads, and the block's total ( `sh`: one word a wave )
template<int T>
__device__ __forceinline__ unsigned block_exclusive( unsigned v, unsigned *sh, unsigned &total ) {
    const unsigned inc = wave_inclusive( v );
    __syncthreads();
    if ( ( threadIdx.x & 63 ) == 63 ) sh[ threadIdx.x >> 6 ] = inc;
    __syncthreads();
    unsigned before = 0;
    total = 0;
    for ( int w = 0; w < T / 64; ++w ) { const unsigned x = sh[ w ]; before += w < int( threadIdx.x >> 6 ) ? x : 0; total += x; }
    return before + inc - v;
}

/// the tiles' counts of one digit made offsets, its total kept ( one block a digit and axis; one block over all counts of 1M keys took
/// 118 us a pass )
__global__ __launch_bounds__( RS_THREADS ) void k_rs_scan( int nt, unsigned *hist, unsigned *total ) {
    __shared__ unsigned sh[ RS_THREADS / 64 ];
    unsigned *v = hist + ( size_t( blockIdx.y ) * 256 + blockIdx.x ) * nt;
    unsigned carry = 0;
    for ( int b = 0; b < nt; b += RS_THREADS ) {
        const int i = b + int( threadIdx.x );
        const unsigned x = i < nt ? v[ i ] : 0u;
        unsigned t;
        const unsigned e = block_exclusive<RS_THREADS>( x, sh, t );
        if ( i < nt ) v[ i ] = carry + e;
        carry += t;
    }
    if ( threadIdx.x == 0 ) total[ blockIdx.y * 256 + blockIdx.x ] = carry;
}

/// the stable scatter of one pass: a tile is read in rounds of 256 elements in order; inside a round the
/// rank of an element among the same digit comes from wave ballots ( 8 bits -> the mask of its peers )
/// plus the counts of the waves before it and of the earlier rounds
__global__ __launch_bounds__( RS_THREADS ) void k_rs_scatter( I64 n, const unsigned long long *keys, const int *vals, int shift, int nt,
                                                            const unsigned *offs, const unsigned *total, unsigned long long *keys_out, int *vals_out ) {
    __shared__ unsigned running[ 256 ], sh[ RS_THREADS / 64 ];
    __shared__ unsigned wcount[ RS_THREADS / 64 ][ 256 ];
    const unsigned long long *key = keys + blockIdx.y * n;
    const int *val = vals + blockIdx.y * n;
    unsigned long long *key_out = keys_out + blockIdx.y * n;
    int *val_out = vals_out + blockIdx.y * n;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    unsigned all;
    const unsigned first = block_exclusive<RS_THREADS>( total[ blockIdx.y * 256 + threadIdx.x ], sh, all );
    running[ threadIdx.x ] = first + offs[ ( size_t( blockIdx.y ) * 256 + threadIdx.x ) * nt + blockIdx.x ];
    const I64 base = I64( blockIdx.x ) * RS_TILE;
    const unsigned long long lt = lane ? ( ~0ull >> ( 64 - lane ) ) : 0ull;
    for ( int j = 0; j < RS_ITEMS; ++j ) {
        for ( int w = 0; w < RS_THREADS / 64; ++w ) wcount[ w ][ threadIdx.x ] = 0;
        __syncthreads();
        const I64 i = base + j * RS_THREADS + threadIdx.x;
        const bool live = i < n;
        const unsigned long long k = live ? key[ i ] : 0ull;
        const unsigned d = unsigned( ( k >> shift ) & 255 );
        unsigned long long peers = __ballot( live );
        for ( int b = 0; b < 8; ++b ) {
            const unsigned long long m = __ballot( ( d >> b ) & 1 );
            peers &= ( ( d >> b ) & 1 ) ? m : ~m;
        }
        const unsigned r_in = __popcll( peers & lt );
        if ( live && r_in == 0 ) wcount[ wave ][ d ] = __popcll( peers );
        __syncthreads();
        if ( live ) {
            unsigned r = running[ d ] + r_in;
            for ( int w = 0; w < wave; ++w ) r += wcount[ w ][ d ];
            key_out[ r ] = k;
            val_out[ r ] = val[ i ];
        }
        __syncthreads();
        unsigned add = 0;
        for ( int w = 0; w < RS_THREADS / 64; ++w ) add += wcount[ w ][ threadIdx.x ];
        running[ threadIdx.x ] += add;
        __syncthreads();
    }
}

/// the stable sorts of `axes` lists of `n` ( key, id ) pairs by key ( eight passes: the result is back in `k0`, `v0` )
void radix_sort( I64 n, int axes, unsigned long long *k0, int *v0, unsigned long long *k1, int *v1, unsigned *hist, unsigned *total, hipStream_t st ) {
    const int nt = int( ( n + RS_TILE - 1 ) / RS_TILE );
    for ( int pass = 0; pass < 8; ++pass ) {
        const int shift = 8 * pass;
        k_rs_hist<<<dim3( nt, axes ), RS_THREADS, 0, st>>>( n, k0, shift, nt, hist );
        k_rs_scan<<<dim3( 256, axes ), RS_THREADS, 0, st>>>( nt, hist, total );
        k_rs_scatter<<<dim3( nt, axes ), RS_THREADS, 0, st>>>( n, k0, v0, shift, nt, hist, total, k1, v1 );
        std::swap( k0, k1 );
        std::swap( v0, v1 );
    }
    check_launch( "radix_sort" );
}

// ---- the levels ------------------------------------------------------------------------------------------

// ( every array over the lists holds `n` entries an axis )

/// the slice of node `j` of level `L`, from its parent's slice and cut
__device__ __forceinline__ void slice_of( int L, int j, I64 n, const int *hbeg, const int *hend, const int *hmid, int &b, int &e ) {
    b = 0;
    e = int( n );
    if ( L == 0 ) return;
    const int p = ( 1 << ( L - 1 ) ) - 1 + j / 2;
    b = j & 1 ? hmid[ p ] : hbeg[ p ];
    e = j & 1 ? hend[ p ] : hmid[ p ];
}

/// a node's box ( the ends of its segments of the lists ), the axis it is cut along ( the first longest ) and where ( its end: not cut )
template<int D, class ID>
__device__ __forceinline__ void node_cut( int b, int e, const double *pos, const ID *ids, I64 stride, int leaf, double *lo, double *hi, int &axis,
                                          int &mid ) {
    axis = 0;
    mid = e;
    for ( int d = 0; d < D; ++d ) lo[ d ] = hi[ d ] = 0;
    if ( e <= b ) return;
    for ( int d = 0; d < D; ++d ) {
        lo[ d ] = pos[ D * size_t( ids[ d * stride + b ] ) + d ];
        hi[ d ] = pos[ D * size_t( ids[ d * stride + e - 1 ] ) + d ];
    }
    for ( int d = 1; d < D; ++d ) if ( hi[ d ] - lo[ d ] > hi[ axis ] - lo[ axis ] ) axis = d;
    if ( e - b > leaf && hi[ axis ] > lo[ axis ] ) mid = b + ( e - b ) / 2;
}

/// the nodes of level `L`, in heap order
template<int D>
__global__ void k_level_nodes( int L, I64 n, const double *pos, const int *ids, int leaf, double *hbox, int *haxis, int *hmid, int *hbeg, int *hend ) {
    const int j = blockIdx.x * blockDim.x + threadIdx.x;
    if ( j >= 1 << L ) return;
    const int node = ( 1 << L ) - 1 + j;
    int b, e, axis, mid;
    slice_of( L, j, n, hbeg, hend, hmid, b, e );
    double lo[ D ], hi[ D ];
    node_cut<D>( b, e, pos, ids, n, leaf, lo, hi, axis, mid );
    for ( int d = 0; d < D; ++d ) { hbox[ 2 * D * size_t( node ) + d ] = lo[ d ]; hbox[ 2 * D * size_t( node ) + D + d ] = hi[ d ]; }
    hbeg[ node ] = b;
    hend[ node ] = e;
    haxis[ node ] = axis;
    hmid[ node ] = mid;
}

/// the side of every seed from its node's cut list: `flag[ id ] = position < mid`
__global__ void k_flags( I64 n, int L, const int *seg, const int *haxis, const int *hmid, const int *ids, unsigned char *flag ) {
    const I64 p = I64( blockIdx.x ) * blockDim.x + threadIdx.x;
    if ( p >= n ) return;
    const int node = ( 1 << L ) - 1 + ( L ? seg[ p ] : 0 );
    flag[ ids[ haxis[ node ] * n + p ] ] = p < hmid[ node ];
}

/// the lists a level partitions: in 2D the one that is not cut, position by position ( one scan ); in 3D all three, the cut one's partition
/// being the identity
template<int D>
__device__ __forceinline__ I64 list_at( I64 n, I64 p, int axis ) { return D == 2 ? ( 1 - axis ) * n + p : blockIdx.y * n + p; }

/// the exclusive scan of the left flags in the lists' order: inside each 1024 positions, and their sums
template<int D>
__global__ __launch_bounds__( 1024 ) void k_scan_blocks( I64 n, int L, const int *seg, const int *haxis, const int *ids, const unsigned char *flag,
                                                       unsigned *s, unsigned *bsum ) {
    __shared__ unsigned sh[ 16 ];
    const I64 p = I64( blockIdx.x ) * 1024 + threadIdx.x;
    unsigned v = 0;
    if ( p < n ) v = flag[ ids[ list_at<D>( n, p, D == 2 ? haxis[ ( 1 << L ) - 1 + ( L ? seg[ p ] : 0 ) ] : 0 ) ] ];
    unsigned total;
    const unsigned e = block_exclusive<1024>( v, sh, total );
    if ( p < n ) s[ blockIdx.y * n + p ] = e;
    if ( threadIdx.x == 0 ) bsum[ blockIdx.y * gridDim.x + blockIdx.x ] = total;
}

/// the blocks' sums scanned, one block a list
__global__ __launch_bounds__( 1024 ) void k_scan_sums( int m, unsigned *bsum ) {
    __shared__ unsigned sh[ 16 ];
    unsigned *v = bsum + size_t( blockIdx.x ) * m, carry = 0;
    for ( int b = 0; b < m; b += 1024 ) {
        const int i = b + int( threadIdx.x );
        const unsigned x = i < m ? v[ i ] : 0u;
        unsigned t;
        const unsigned e = block_exclusive<1024>( x, sh, t );
        if ( i < m ) v[ i ] = carry + e;
        carry += t;
    }
}

/// the stable partition of the lists inside every segment, and the next level's node of every position
template<int D>
__global__ void k_partition( I64 n, int L, const int *seg, const int *haxis, const int *hbeg, const int *hmid, const int *ids,
                             const unsigned char *flag, const unsigned *s, const unsigned *bsum, int nsb, int *out, int *seg_out ) {
    const I64 p = I64( blockIdx.x ) * blockDim.x + threadIdx.x;
    if ( p >= n ) return;
    const int j = L ? seg[ p ] : 0, node = ( 1 << L ) - 1 + j;
    const int b = hbeg[ node ], m = hmid[ node ], axis = haxis[ node ];
    const unsigned *sl = s + blockIdx.y * n, *bl = bsum + size_t( blockIdx.y ) * nsb;
    const I64 from = list_at<D>( n, p, axis );
    const int id = ids[ from ];
    const bool left = flag[ id ];
    const unsigned before = ( sl[ p ] + bl[ p / 1024 ] ) - ( sl[ b ] + bl[ b / 1024 ] );
    const int q = left ? b + int( before ) : m + int( ( p - b ) - before );
    out[ from - p + q ] = id;
    if ( D == 2 ) out[ axis * n + p ] = ids[ axis * n + p ];
    if ( blockIdx.y == 0 ) seg_out[ p ] = 2 * j + ( p >= m );
}

/// the leaves' seeds in ascending user index, and the outputs in rank order
__global__ void k_leaves( int count, int first, const int *hbeg, const int *hend, int *ids, int *leaf_of ) {
    const int j = blockIdx.x * blockDim.x + threadIdx.x;
    if ( j >= count ) return;
    const int b = hbeg[ first + j ], e = hend[ first + j ];
    if ( leaf_of ) for ( int i = b; i < e; ++i ) leaf_of[ i ] = j;
    for ( int i = b + 1; i < e; ++i ) {                   // insertion sort, a handful of seeds
        const int v = ids[ i ];
        int k = i;
        for ( ; k > b && ids[ k - 1 ] > v; --k ) ids[ k ] = ids[ k - 1 ];
        ids[ k ] = v;
    }
}

template<int D>
__device__ __forceinline__ double4 seed_of( const double *pos, int u ) {
    if ( D == 2 ) return make_double4( pos[ 2 * size_t( u ) ], pos[ 2 * size_t( u ) + 1 ], 0.0, 0.0 );
    return make_double4( pos[ 3 * size_t( u ) ], pos[ 3 * size_t( u ) + 1 ], pos[ 3 * size_t( u ) + 2 ], 0.0 );
}

template<int D>
__global__ void k_rank_tables( I64 n, const int *ids, const double *pos, int *order, int *rank_of, double4 *seeds ) {
    const I64 k = I64( blockIdx.x ) * blockDim.x + threadIdx.x;
    if ( k >= n ) return;
    const int u = ids[ k ];
    order[ k ] = u;
    rank_of[ u ] = int( k );
    seeds[ k ] = seed_of<D>( pos, u );
}

/// the preorder index of node `j` of level `L` in a tree `depth` high: a left child is 1 after its parent, a right one `2^( height - 1 )`
__device__ __forceinline__ int preorder_of( int j, int L, int depth ) { return 2 * ( j << ( depth - 1 - L ) ) + L - __popc( unsigned( j ) ); }

/// the tree's arrays from the heap's, in preorder, and the nodes level by level
__global__ void k_to_preorder( I64 N, int depth, int box, const int *hbeg, const int *hend, const double *hbox, int *beg, int *end, double *out,
                               int *lvl_nodes ) {
    const I64 h = I64( blockIdx.x ) * blockDim.x + threadIdx.x;
    if ( h >= N ) return;
    const int L = 31 - __clz( int( h ) + 1 ), p = preorder_of( int( h ) + 1 - ( 1 << L ), L, depth );
    lvl_nodes[ h ] = p;
    beg[ p ] = hbeg[ h ];
    end[ p ] = hend[ h ];
    for ( int c = 0; c < box; ++c ) out[ box * size_t( p ) + c ] = hbox[ box * size_t( h ) + c ];
}

// ---- a small cloud's tree by one workgroup ----------------------------------------------------------------------------

constexpr int SMALL_T = 1024, SMALL_NODES = 1024;
constexpr int SMALL_PER = SMALL_TREE / SMALL_T;        ///< a thread's consecutive positions in a scan

struct SmallOut {
    int *beg, *end, *lvl_nodes, *order, *rank_of, *leaf_of;
    double *box;
    double4 *seeds;
};

/// THE SAME TREE in one launch: each axis sorted by a bitonic network over ( key, user index ), the lists and their partitions in LDS,
/// the levels separated by barriers, each thread four consecutive positions of a scan. It is bound by its barriers and LDS: 2k seeds 114
/// us, which made a call that measures 2k cells 0.79 -> 0.44 ms
template<int D>
__global__ __launch_bounds__( SMALL_T ) void k_small_tree( int n, const double *pos, int leaf, int depth, SmallOut out ) {
    typedef unsigned short u16;
    __shared__ unsigned long long keys[ SMALL_TREE ];
    __shared__ u16 lists[ D ][ SMALL_TREE ];
    __shared__ u16 nbeg[ SMALL_NODES ], nend[ SMALL_NODES ], nmid[ SMALL_NODES ], npre[ SMALL_NODES ], pbeg[ SMALL_NODES / 2 ], pend[ SMALL_NODES / 2 ],
        pmid[ SMALL_NODES / 2 ];
    __shared__ unsigned char naxis[ SMALL_NODES ];
    __shared__ unsigned sh[ SMALL_T / 64 ];
    const int tid = threadIdx.x;
    int n2 = 2;
    while ( n2 < n ) n2 *= 2;
    for ( int d = 0; d < D; ++d ) {
        u16 *id = lists[ d ];
        for ( int i = tid; i < n2; i += SMALL_T ) { keys[ i ] = i < n ? dkey( pos[ D * i + d ] ) : ~0ull; id[ i ] = u16( i ); }
        __syncthreads();
        for ( int k = 2; k <= n2; k *= 2 )
            for ( int j = k / 2; j > 0; j /= 2 ) {
                for ( int t = tid; t < n2 / 2; t += SMALL_T ) {
                    const int a = 2 * t - ( t & ( j - 1 ) ), b = a + j;
                    const unsigned long long ka = keys[ a ], kb = keys[ b ];
                    const u16 ia = id[ a ], ib = id[ b ];
                    const bool greater = ka > kb || ( ka == kb && ia > ib );
                    if ( greater == ! ( a & k ) ) { keys[ a ] = kb; keys[ b ] = ka; id[ a ] = ib; id[ b ] = ia; }
                }
                __syncthreads();
            }
    }
    // ( the keys' room: the partitions' output, the segments, the flags )
    u16 *alt = reinterpret_cast<u16 *>( keys );                       // [ D ][ SMALL_TREE ]
    unsigned char *flag = reinterpret_cast<unsigned char *>( alt + 3 * SMALL_TREE );
    u16 *cur = &lists[ 0 ][ 0 ];
    const int p0 = SMALL_PER * tid;
    int seg[ SMALL_PER ];
    for ( int u = 0; u < SMALL_PER; ++u ) seg[ u ] = 0;
    for ( int L = 0; L < depth; ++L ) {
        const int count = 1 << L;
        if ( tid < count ) {
            const int j = tid;
            int b = 0, e = n, axis, mid;
            if ( L ) {
                b = j & 1 ? pmid[ j / 2 ] : pbeg[ j / 2 ];
                e = j & 1 ? pend[ j / 2 ] : pmid[ j / 2 ];
            }
            double lo[ D ], hi[ D ];
            node_cut<D>( b, e, pos, cur, SMALL_TREE, leaf, lo, hi, axis, mid );
            const int p = preorder_of( j, L, depth );
            out.lvl_nodes[ count - 1 + j ] = p;
            out.beg[ p ] = b;
            out.end[ p ] = e;
            for ( int d = 0; d < D; ++d ) { out.box[ 2 * D * p + d ] = lo[ d ]; out.box[ 2 * D * p + D + d ] = hi[ d ]; }
            nbeg[ j ] = u16( b );
            nend[ j ] = u16( e );
            nmid[ j ] = u16( mid );
            naxis[ j ] = ( unsigned char )( axis );
        }
        __syncthreads();
        if ( L + 1 == depth ) break;
        for ( int u = 0; u < SMALL_PER; ++u )
            if ( p0 + u < n ) flag[ cur[ naxis[ seg[ u ] ] * SMALL_TREE + p0 + u ] ] = p0 + u < nmid[ seg[ u ] ];
        __syncthreads();
        for ( int d = 0; d < D; ++d ) {
            const u16 *in = cur + d * SMALL_TREE;
            u16 *to = alt + d * SMALL_TREE;
            unsigned f = 0, c = 0, all;
            for ( int u = 0; u < SMALL_PER; ++u )
                if ( p0 + u < n && flag[ in[ p0 + u ] ] ) { f |= 1u << u; ++c; }
            const unsigned before = block_exclusive<SMALL_T>( c, sh, all );
            // the prefix at each segment's start, from the thread that holds it
            for ( int u = 0; u < SMALL_PER; ++u )
                if ( p0 + u < n && p0 + u == nbeg[ seg[ u ] ] ) npre[ seg[ u ] ] = u16( before + __popc( f & ( ( 1u << u ) - 1 ) ) );
            __syncthreads();
            for ( int u = 0; u < SMALL_PER; ++u ) {
                if ( p0 + u >= n ) continue;
                const int j = seg[ u ], lb = int( before ) + __popc( f & ( ( 1u << u ) - 1 ) ) - npre[ j ];
                to[ f >> u & 1 ? nbeg[ j ] + lb : nmid[ j ] + ( p0 + u - nbeg[ j ] ) - lb ] = in[ p0 + u ];
            }
            __syncthreads();
        }
        for ( int u = 0; u < SMALL_PER; ++u )
            if ( p0 + u < n ) seg[ u ] = 2 * seg[ u ] + ( p0 + u >= nmid[ seg[ u ] ] );
        __syncthreads();
        if ( tid < count ) { pbeg[ tid ] = nbeg[ tid ]; pend[ tid ] = nend[ tid ]; pmid[ tid ] = nmid[ tid ]; }
        // ( the flags lie past the partitions' output and are written anew before the lists change places again )
        for ( int d = 0; d < D; ++d )
            for ( int i = tid; i < n; i += SMALL_T ) cur[ d * SMALL_TREE + i ] = alt[ d * SMALL_TREE + i ];
        __syncthreads();
    }
    // the leaves' seeds in ascending user index, then the rank tables
    if ( tid < 1 << ( depth - 1 ) ) {
        const int b = nbeg[ tid ], e = nend[ tid ];
        for ( int i = b + 1; i < e; ++i ) {
            const u16 v = cur[ i ];
            int k = i;
            for ( ; k > b && cur[ k - 1 ] > v; --k ) cur[ k ] = cur[ k - 1 ];
            cur[ k ] = v;
        }
        if ( out.leaf_of ) for ( int i = b; i < e; ++i ) out.leaf_of[ i ] = tid;
    }
    __syncthreads();
    for ( int k = tid; k < n; k += SMALL_T ) {
        const int u = cur[ k ];
        out.order[ k ] = u;
        out.rank_of[ u ] = k;
        out.seeds[ k ] = seed_of<D>( pos, u );
    }
}

/// the tree of `D`-dimensional seeds into the arrays of `o` ( see the file's header )
template<int D>
void build_into( const SmallOut &o, I64 n, const double *pos, int leaf, int depth, hipStream_t st ) {
    const I64 N = ( I64( 1 ) << depth ) - 1;
    if ( n <= SMALL_TREE && ( 1 << ( depth - 1 ) ) <= SMALL_NODES ) {
        k_small_tree<D><<<1, SMALL_T, 0, st>>>( int( n ), pos, leaf, depth, o );
        check_launch( "k_small_tree" );
        return;
    }
    Arena &A = arena();
    // scratch ( one build at a time on a thread's arena ), `D` lists an array
    unsigned long long *ka = A.get<unsigned long long>( "tb.ka", size_t( n ) * D ), *kb = A.get<unsigned long long>( "tb.kb", size_t( n ) * D );
    int *va = A.get<int>( "tb.va", size_t( n ) * D ), *vb = A.get<int>( "tb.vb", size_t( n ) * D );
    const int nt = int( ( n + RS_TILE - 1 ) / RS_TILE ), nsb = int( ( n + 1023 ) / 1024 ), lists = D == 2 ? 1 : D;
    unsigned *hist = A.get<unsigned>( "tb.hist", size_t( 256 ) * nt * D ), *total = A.get<unsigned>( "tb.total", 256 * D );
    int *hbeg = A.get<int>( "tb.hbeg", size_t( N ) ), *hend = A.get<int>( "tb.hend", size_t( N ) );
    int *haxis = A.get<int>( "tb.haxis", size_t( N ) ), *hmid = A.get<int>( "tb.hmid", size_t( N ) );
    double *hbox = A.get<double>( "tb.hbox", size_t( N ) * 2 * D );
    int *seg = A.get<int>( "tb.seg", size_t( n ) ), *seg2 = A.get<int>( "tb.seg2", size_t( n ) );
    unsigned char *flag = A.get<unsigned char>( "tb.flag", size_t( n ) );
    unsigned *s = A.get<unsigned>( "tb.s", size_t( n ) * lists ), *bsum = A.get<unsigned>( "tb.bsum", size_t( nsb ) * lists );
    const unsigned nbk = blocks_for( n, 256 );
    k_keys<<<dim3( nbk, D ), 256, 0, st>>>( n, pos, D, ka, va );
    radix_sort( n, D, ka, va, kb, vb, hist, total, st );
    for ( int L = 0; L < depth; ++L ) {
        k_level_nodes<D><<<blocks_for( I64( 1 ) << L, 256 ), 256, 0, st>>>( L, n, pos, va, leaf, hbox, haxis, hmid, hbeg, hend );
        if ( L + 1 == depth ) break;
        k_flags<<<nbk, 256, 0, st>>>( n, L, seg, haxis, hmid, va, flag );
        k_scan_blocks<D><<<dim3( nsb, lists ), 1024, 0, st>>>( n, L, seg, haxis, va, flag, s, bsum );
        k_scan_sums<<<lists, 1024, 0, st>>>( nsb, bsum );
        k_partition<D><<<dim3( nbk, lists ), 256, 0, st>>>( n, L, seg, haxis, hbeg, hmid, va, flag, s, bsum, nsb, vb, seg2 );
        check_launch( "tree level" );
        std::swap( va, vb );
        std::swap( seg, seg2 );
    }
    const int L = depth - 1;
    k_leaves<<<blocks_for( I64( 1 ) << L, 256 ), 256, 0, st>>>( 1 << L, ( 1 << L ) - 1, hbeg, hend, va, o.leaf_of );
    k_rank_tables<D><<<nbk, 256, 0, st>>>( n, va, pos, o.order, o.rank_of, o.seeds );
    k_to_preorder<<<blocks_for( N, 256 ), 256, 0, st>>>( N, depth, 2 * D, hbeg, hend, hbox, o.beg, o.end, o.box, o.lvl_nodes );
    check_launch( "tree finish" );
}

} // namespace

void build_tree_device3( DevTree3 &t, I64 n, const double *pos, int leaf, hipStream_t st, const std::string &tag ) {
    SDOT_CHECK( n >= 1, "a tree needs at least one seed" );
    SDOT_CHECK( n < ( I64( 1 ) << 31 ) - 8, "more seeds than 32-bit ranks can index" );
    const int depth = max_depth_for( n, leaf );
    const I64 N = ( I64( 1 ) << depth ) - 1;
    t.n = n; t.depth = depth; t.leaf = leaf; t.nb_nodes = N;
    Arena &A = arena();
    t.nodes = A.get<NodeRec3>( tag + ".nodes3", size_t( N ) );
    t.node_box = A.get<double>( tag + ".node_box3", size_t( N ) * 6 );
    t.node_beg = A.get<int>( tag + ".node_beg3", size_t( N ) );
    t.node_end = A.get<int>( tag + ".node_end3", size_t( N ) );
    t.lvl_nodes = A.get<int>( tag + ".lvl_nodes3", size_t( N ) );
    t.order = A.get<int>( tag + ".order3", size_t( n ) );
    t.rank_of = A.get<int>( tag + ".rank_of3", size_t( n ) );
    t.seeds = A.get<double4>( tag + ".seeds3", size_t( n ) );
    t.stat = A.get<double>( tag + ".stat3", size_t( N ) * 16 );
    t.fit = A.get<double>( tag + ".fit3", size_t( N ) * 3 );
    t.rkeys = A.get<unsigned long long>( tag + ".rkeys3", size_t( N ) * 3 );
    build_into<3>( SmallOut{ t.node_beg, t.node_end, t.lvl_nodes, t.order, t.rank_of, nullptr, t.node_box, t.seeds }, n, pos, leaf, depth, st );
}

void build_tree_device( DevTree &t, I64 n, const double *pos, int leaf, hipStream_t st, const std::string &tag ) {
    SDOT_CHECK( n >= 1, "a tree needs at least one seed" );
    SDOT_CHECK( n < ( I64( 1 ) << 31 ) - 8, "more seeds than 32-bit ranks can index" );
    const int depth = max_depth_for( n, leaf );
    const I64 N = ( I64( 1 ) << depth ) - 1;
    t.n = n; t.depth = depth; t.leaf = leaf; t.nb_nodes = N;
    Arena &A = arena();
    t.nodes = A.get<NodeRec>( tag + ".nodes", size_t( N ) );
    t.nodes32 = A.get<NodeF>( tag + ".nodes32", size_t( N ) );
    t.node_box = A.get<double>( tag + ".node_box", size_t( N ) * 4 );
    t.node_beg = A.get<int>( tag + ".node_beg", size_t( N ) );
    t.node_end = A.get<int>( tag + ".node_end", size_t( N ) );
    t.lvl_nodes = A.get<int>( tag + ".lvl_nodes", size_t( N ) );
    t.order = A.get<int>( tag + ".order", size_t( n ) );
    t.rank_of = A.get<int>( tag + ".rank_of", size_t( n ) );
    t.leaf_of = A.get<int>( tag + ".leaf_of", size_t( n ) );
    t.seeds = A.get<double4>( tag + ".seeds", size_t( n ) );
    t.stat = A.get<double>( tag + ".stat", size_t( N ) * 11 );
    t.fit = A.get<double>( tag + ".fit", size_t( N ) * 2 );
    t.rkeys = A.get<unsigned long long>( tag + ".rkeys", size_t( N ) * 3 );
    build_into<2>( SmallOut{ t.node_beg, t.node_end, t.lvl_nodes, t.order, t.rank_of, t.leaf_of, t.node_box, t.seeds }, n, pos, leaf, depth, st );
}

} // namespace sdot_amd
