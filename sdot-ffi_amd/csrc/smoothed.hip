// The Newton direction by flexible CG preconditioned with one V-cycle of smoothed aggregation.
//
// The aggregates are `pack` consecutive tree ranks, as in the reference's CPU multigrid ( `src/sdot/include/sdot/sdotplan/
// Multigrid.h:11-18` ), and so is the idea of smoothing the prolongation and dropping its small entries ( `:331-368` ). Against the
// K-cycle over plain aggregates ( multigrid.hip ) it trades a dearer setup, once per system, for an iteration of a third of the
// launches and fewer of them. On a 200k-seed image Laplacian, relative residual 1e-6 ( the same cycles emulated on the CPU ):
// 63 iterations of ~70 launches with the K-cycle; 38 of ~21 with aggregates of 8; 27 with a first level of 4.
//
// What a level does:
//   * `P = ( I - 2/3 D^-1 A ) P0`, a row's entries below 0.1 of its largest dropped ( 0.2 to 0.25 where rows are long, in 3D: there the
//     coarse rows would outgrow their room ), the rest scaled to a unit sum ( `k_prolongator` ); the restriction is `P^T`,
//     listed per coarse row in increasing order of the fine rows;
//   * the Galerkin row `P^T A P` by one wave: its columns found by an LDS hash, each column's sum taken in whole numbers of
//     a bound's 2^-60, so the result does not depend on the hash's races ( `k_galerkin` );
//   * two damped Jacobi sweeps before ( from zero: one pass ) and after, Chebyshev dampings; the correction scaled by 1.2, which
//     saves 10 % of the iterations ( 1.15 to 1.45 measured alike ), as truncated prolongations under-correct;
//   * THE BOTTOM: the first level of at most 2048 rows is one product with a dense operator, the V-cycle over the levels below
//     applied to every unit vector at setup ( `k_bottom_op`, two columns a workgroup, the vectors in LDS ). A product of 2048^2
//     floats takes ~6 us spread over the chip ( each XCD's eighth of it stays in its L2 ), where the levels below as launches take
//     ~12 x 5 us, and as one workgroup 17-48 us.
// Small levels are bound by their launches ( ~5 us each whatever they do ), the finest one by HBM and its gathers.
//
// The outer iteration fuses the direction into the product: a lane reads its neighbours' `z` and `p` and forms `z + beta p` itself
// ( `k_direction` ); the convergence test runs in the cycle's first kernel. Every scalar is summed from fixed-shape partials by each
// block that needs it; a stop flag turns the launches after convergence into no-ops.

#include "smoothed.h"

#include <algorithm>
#include <type_traits>

namespace sdot_amd {

namespace {

constexpr int SA_PMAX = 8;          ///< entries of a prolongation row
constexpr int SA_TMAX = 128;        ///< fine rows that interpolate from one coarse row
constexpr int SA_SMAX = 255;        ///< entries of a coarse row, at most
constexpr int SA_HASH = 512;        ///< slots of the Galerkin row's hash
constexpr I64 SA_BOTTOM = 2048;     ///< rows of the dense bottom, at most
constexpr int SA_DENSE = 64;        ///< rows of the coarsest level, at most
constexpr int SA_LEVELS = 16;
constexpr int SA_BLOCKS = 2048;     ///< partial sums: eight waves a SIMD, one row per lane below 512k rows
constexpr int TH = 256;

/// the outer iteration's device state, and the partial sums' slots
enum { S_PQ = 0, S_NB, S_ERR, S_DONE, S_IT, S_TOL, S_FAILED, S_BAD, S_TRUE, S_NB_STATE };
enum { P_PQ = 0, P_PR, P_RR, P_ZQ, P_NB };

/// a level's matrix: entry `q` of row `i` at `( row_off ? row_off[ i ] : i rs ) + q step`; the off-diagonal entries are `-val`
template<class R>
struct Rows {
    I64 n = 0, step = 1;
    int rs = 0;
    const int *row_off = nullptr, *cnt = nullptr, *col = nullptr;
    const R *val = nullptr, *dia = nullptr;
    __device__ __forceinline__ I64 base( I64 i ) const { return row_off ? I64( row_off[ i ] ) : i * rs; }
};

/// a level: its matrix, the inverse diagonal, the prolongation from the next level ( entry `q` of row `i` at `q n + i` ), the
/// restriction into it from the level above ( row `I`'s list at `I SA_TMAX` ), the cycle's vectors
template<class P>
struct Level {
    Rows<P> A;
    P *dinv = nullptr;
    int *pn = nullptr, *pcol = nullptr;
    P *pval = nullptr;
    int *tn = nullptr, *tcol = nullptr;
    P *tval = nullptr;
    P *r = nullptr, *y = nullptr, *x = nullptr, *t = nullptr, *e = nullptr;
};

__device__ __forceinline__ double wave_sum( double v ) {
    for ( int o = 32; o > 0; o >>= 1 ) v += __shfl_xor( v, o, 64 );
    return v;
}
/// the block's sum ( 4 waves ), the same in every thread
__device__ __forceinline__ double sum_block( double v, double *sh ) {
    v = wave_sum( v );
    __syncthreads();
    if ( ( threadIdx.x & 63 ) == 0 ) sh[ threadIdx.x >> 6 ] = v;
    __syncthreads();
    return ( sh[ 0 ] + sh[ 1 ] ) + ( sh[ 2 ] + sh[ 3 ] );
}
__device__ __forceinline__ double sum_partials( const double *p, int nb, double *sh ) {
    double a = 0;
    for ( int j = threadIdx.x; j < nb; j += TH ) a += p[ j ];
    return sum_block( a, sh );
}

/// the block's place when the blocks of one XCD take consecutive places ( they are dealt round-robin to the 8 XCDs, and a row's
/// neighbours, near ranks, are then read from the same L2 )
__device__ __forceinline__ int xcd_block() {
    const int nblk = int( gridDim.x ), b = int( blockIdx.x );
    const int per = nblk / 8, rem = nblk % 8, xcd = b % 8, slot = b / 8;
    return xcd < rem ? xcd * ( per + 1 ) + slot : rem * ( per + 1 ) + ( xcd - rem ) * per + slot;
}

/// `sum_q val_q f( col_q )` over a row of `c` entries, four entries' loads in flight at a time
template<class R, class F>
__device__ __forceinline__ double row_sum( const Rows<R> &A, I64 b, int c, F f ) {
    double s = 0;
    for ( int q = 0; q < c; q += 4 ) {
        double v[ 4 ], x[ 4 ];
#pragma unroll
        for ( int k = 0; k < 4; ++k ) {
            const I64 e = b + I64( q + k < c ? q + k : c - 1 ) * A.step;
            v[ k ] = double( A.val[ e ] );
            x[ k ] = f( A.col[ e ] );
        }
#pragma unroll
        for ( int k = 0; k < 4; ++k ) s += q + k < c ? v[ k ] * x[ k ] : 0.0;
    }
    return s;
}

/// the same over a row shared by `G` lanes ( entry `q` to lane `q % G` ), the sum in each of them
template<int G, class R, class F>
__device__ __forceinline__ double row_sum_lanes( const Rows<R> &A, I64 b, int c, int lane, F f ) {
    double s = 0;
    for ( int q = lane; q < c; q += G ) {
        const I64 e = b + I64( q ) * A.step;
        s += double( A.val[ e ] ) * f( A.col[ e ] );
    }
    for ( int o = G / 2; o > 0; o >>= 1 ) s += __shfl_xor( s, o, G );
    return s;
}

// ---- the hierarchy ------------------------------------------------------------------------------------------------------

__global__ void k_sa_zero( int n, int *v, double *state ) {
    const int i = int( blockIdx.x ) * blockDim.x + threadIdx.x;
    if ( i < n ) v[ i ] = 0;
    if ( i < S_NB_STATE ) state[ i ] = 0;
}

template<class P>
__global__ void k_sa_dinv( I64 n, const P *dia, P *dinv ) {
    const I64 i = I64( blockIdx.x ) * blockDim.x + threadIdx.x;
    if ( i < n ) dinv[ i ] = P( 1.0 / double( dia[ i ] ) );
}

/// THE PROLONGATION'S ROWS, `G` lanes a row: `( 1 - omega ) e_own + omega / d sum_j c_ij e_agg(j)`, the entries of one aggregate
/// summed in the row's order ( each lane adds up those equal to its own ), small ones dropped, at most `SA_PMAX` kept; each row
/// is then added to the lists of the coarse rows it reads ( in the order the lanes come: `k_galerkin` sorts them ). A row past
/// `G E - 1` entries leaves the last ones out: any unit-sum row is a prolongation
template<class P, int G, int E>
__global__ __launch_bounds__( TH ) void k_prolongator( Rows<P> A, int pack, double omega, double theta, int *pn, int *pcol, P *pval, int *tn, int *tcol ) {
    const int lane = threadIdx.x & ( G - 1 );
    const I64 i = ( I64( xcd_block() ) * TH + threadIdx.x ) / G;
    const bool live = i < A.n;
    const int gsh = ( threadIdx.x & 63 ) & ~( G - 1 );
    const unsigned long long gmask = G == 64 ? ~0ull : ( ( 1ull << G ) - 1 );
    int key[ E ];
    P w[ E ], tot[ E ];
    bool first[ E ];
    const int own = live ? int( i / pack ) : -1;
    const int cnt = live ? min( A.cnt[ i ], G * E - 1 ) : -1;
    const I64 b = live ? A.base( i ) : 0;
    const double d = live ? double( A.dia[ i ] ) : 1.0;
    const double f = d > 0 ? omega / d : 0.0;
#pragma unroll
    for ( int e = 0; e < E; ++e ) {
        const int q = lane + G * e;
        key[ e ] = -1;
        w[ e ] = tot[ e ] = 0;
        first[ e ] = q <= cnt;
        if ( q < cnt ) { key[ e ] = A.col[ b + I64( q ) * A.step ] / pack; w[ e ] = P( f * double( A.val[ b + I64( q ) * A.step ] ) ); }
        else if ( q == cnt ) { key[ e ] = own; w[ e ] = P( 1 - omega ); }
    }
#pragma unroll
    for ( int g = 0; g < E; ++g ) {
        if ( ! __any( key[ g ] >= 0 ) ) break;
        for ( int k = 0; k < G; ++k ) {
            const int kk = __shfl( key[ g ], k, G );
            const P ww = __shfl( w[ g ], k, G );
#pragma unroll
            for ( int e = 0; e < E; ++e )
                if ( kk == key[ e ] ) {
                    tot[ e ] += ww;
                    if ( g < e || ( g == e && k < lane ) ) first[ e ] = false;
                }
        }
    }
    P m = 0;
#pragma unroll
    for ( int e = 0; e < E; ++e ) if ( first[ e ] ) m = max( m, P( fabs( double( tot[ e ] ) ) ) );
    for ( int o = G / 2; o > 0; o >>= 1 ) m = max( m, P( __shfl_xor( m, o, G ) ) );
    // the threshold, raised while too many entries pass it
    P thr = P( theta ) * m;
    int pos[ E ], total = 0;
    for ( int pass = 0; pass < 6; ++pass ) {
        total = 0;
#pragma unroll
        for ( int e = 0; e < E; ++e ) {
            const bool keep = first[ e ] && P( fabs( double( tot[ e ] ) ) ) >= thr;
            const unsigned long long bal = ( __ballot( keep ) >> gsh ) & gmask;
            pos[ e ] = keep ? total + __popcll( bal & ( ( 1ull << lane ) - 1 ) ) : SA_PMAX;
            total += __popcll( bal );
        }
        if ( ! __any( total > SA_PMAX ) ) break;
        if ( total > SA_PMAX ) thr = thr * P( 1.5 ) < m ? thr * P( 1.5 ) : m;
    }
    P s = 0;
#pragma unroll
    for ( int e = 0; e < E; ++e ) if ( pos[ e ] < SA_PMAX ) s += tot[ e ];
    for ( int o = G / 2; o > 0; o >>= 1 ) s += __shfl_xor( s, o, G );
    if ( ! live ) return;
    if ( ! ( s > P( 0.25 ) ) ) {                         // ( no sum to scale by: the plain aggregate )
        if ( lane == 0 ) {
            pn[ i ] = 1; pcol[ i ] = own; pval[ i ] = 1;
            const int at = atomicAdd( &tn[ own ], 1 );
            if ( at < SA_TMAX ) tcol[ I64( own ) * SA_TMAX + at ] = int( i );
        }
        return;
    }
    const P inv = P( 1 ) / s;
#pragma unroll
    for ( int e = 0; e < E; ++e )
        if ( pos[ e ] < SA_PMAX ) {
            pcol[ I64( pos[ e ] ) * A.n + i ] = key[ e ];
            pval[ I64( pos[ e ] ) * A.n + i ] = tot[ e ] * inv;
            const int at = atomicAdd( &tn[ key[ e ] ], 1 );
            if ( at < SA_TMAX ) tcol[ I64( key[ e ] ) * SA_TMAX + at ] = int( i );
        }
    if ( lane == 0 ) pn[ i ] = min( total, SA_PMAX );
}

/// the fine rows that read coarse row `I`, listed by `k_prolongator` in any order: sorted ( `si`, LDS ), their weights found ( `sw` ) and
/// both written back as the restriction's row; one wave. Returns the list's length
template<class P>
__device__ __forceinline__ int sorted_list( I64 I, I64 nf, const int *pn, const int *pcol, const P *pval, const int *tn, int *tcol, P *tval, int *raw,
                                            int *si, double *sw ) {
    const int lane = threadIdx.x;
    const int cnt = min( tn[ I ], SA_TMAX );
    int mine[ 2 ], rank[ 2 ] = { 0, 0 };
    for ( int u = 0; u < 2; ++u ) {
        const int k = lane + 64 * u;
        mine[ u ] = k < cnt ? tcol[ I * SA_TMAX + k ] : 0x7fffffff;
        raw[ k ] = mine[ u ];
    }
    __syncthreads();
    for ( int k = 0; k < cnt; ++k ) { rank[ 0 ] += raw[ k ] < mine[ 0 ]; rank[ 1 ] += raw[ k ] < mine[ 1 ]; }
    for ( int u = 0; u < 2; ++u )
        if ( lane + 64 * u < cnt ) si[ rank[ u ] ] = mine[ u ];
    __syncthreads();
    for ( int u = 0; u < 2; ++u ) {
        const int k = lane + 64 * u;
        if ( k >= cnt ) continue;
        const int i = si[ k ], np = pn[ i ];
        P w = 0;
        for ( int q = 0; q < np; ++q ) if ( pcol[ I64( q ) * nf + i ] == int( I ) ) w = pval[ I64( q ) * nf + i ];
        sw[ k ] = double( w );
        tcol[ I * SA_TMAX + k ] = i;
        tval[ I * SA_TMAX + k ] = w;
    }
    __syncthreads();
    return cnt;
}

/// THE GALERKIN ROWS, one wave a coarse row ( see the file's header ): the terms `P_iI a_ij P_jK` of the fine rows `i` of its list, eight
/// lanes a fine row, added in LDS at their column's place in a hash of the columns met ( at most `SA_SMAX + 1` ). The sums are 64-bit
/// whole numbers of `2^-60` of a guess of the row's terms' size ( `P`'s rows sum to 1, a Laplacian's row to twice its diagonal ), so that the
/// atomics' order does not matter: the row is the same in every run, and each sum is within `2^-61` of the guess a term, where a sum in
/// double rounds by `2^-53` of itself. Entries of both signs can pass the guess ( 1M 3D seeds in a thin slab ), so the terms' sizes are summed
/// too, in double: below `2^62` units no column's sum wraps. `state[ S_BAD ]` beyond it, and when a list or a row outgrows its room.
/// ( Terms staged in LDS and added up by their column's lane, every lane looking at every term: 1M rows 2.05 ms a hierarchy, 0.90 so )
template<class P>
__global__ __launch_bounds__( 64 ) void k_galerkin( Rows<P> A, const int *pn, const int *pcol, const P *pval, int *tn, int *tcol, P *tval, int room,
                                                   int *ccnt, int *ccol, P *cval, P *cdia, P *cdinv, double *state ) {
    __shared__ unsigned long long sum[ SA_HASH ];
    __shared__ double sw[ SA_TMAX ];
    __shared__ int raw[ SA_TMAX ], si[ SA_TMAX ], hk[ SA_HASH ], ck[ SA_SMAX + 1 ], at[ SA_SMAX + 1 ], nkeys;
    const int lane = threadIdx.x;
    const I64 I = xcd_block();
    const bool over = tn[ I ] > SA_TMAX;
    for ( int h = lane; h < SA_HASH; h += 64 ) { hk[ h ] = -1; sum[ h ] = 0; }
    if ( lane == 0 ) nkeys = 0;
    const int cnt = sorted_list( I, A.n, pn, pcol, pval, tn, tcol, tval, raw, si, sw );
    double bound = 0;
    for ( int k = lane; k < cnt; k += 64 ) bound += 2 * fabs( sw[ k ] * double( A.dia[ si[ k ] ] ) );
    for ( int o = 32; o; o >>= 1 ) bound += __shfl_xor( bound, o, 64 );
    const int ex = bound > 0 && bound < 1e300 ? max( ilogb( bound ) + 1, -900 ) : 0;
    double size = 0;
    const double scale = ldexp( 1.0, 60 - ex ), unit = ldexp( 1.0, ex - 60 );
    const int g = lane >> 3, sub = lane & 7;
    for ( int base = 0; base < cnt && nkeys <= SA_SMAX + 1; base += 8 ) {   // ( past any room the hash would fill up )
        if ( base + g < cnt ) {
            const int i = si[ base + g ];
            const double wi = sw[ base + g ] * scale;
            const int rc = A.cnt[ i ];
            const I64 b = A.base( i );
            for ( int q = sub; q <= rc; q += 8 ) {
                int j = i;
                double a;
                if ( q < rc ) { j = A.col[ b + I64( q ) * A.step ]; a = -double( A.val[ b + I64( q ) * A.step ] ); }
                else a = double( A.dia[ i ] );
                const int np = pn[ j ];
                for ( int e = 0; e < np; ++e ) {
                    const int K = pcol[ I64( e ) * A.n + j ];
                    const double t = wi * a * double( pval[ I64( e ) * A.n + j ] );
                    const long long term = __double2ll_rn( t );
                    size += fabs( t );
                    unsigned h = ( unsigned( K ) * 2654435761u ) >> 23;
                    for ( int probe = 0; probe < SA_HASH; ++probe, h = ( h + 1 ) & ( SA_HASH - 1 ) ) {
                        int prev = hk[ h ];
                        if ( prev == -1 ) {
                            prev = atomicCAS( &hk[ h ], -1, K );
                            if ( prev == -1 ) {
                                const int id = atomicAdd( &nkeys, 1 );
                                if ( id <= SA_SMAX ) { ck[ id ] = K; at[ id ] = int( h ); }
                                prev = K;
                            }
                        }
                        if ( prev == K ) { atomicAdd( &sum[ h ], static_cast<unsigned long long>( term ) ); break; }
                    }
                }
            }
        }
        __syncthreads();
    }
    size = wave_sum( size );
    const int m = min( nkeys, SA_SMAX + 1 );
    bool diag = false;
    for ( int id = lane; id < m; id += 64 ) {
        const int K = ck[ id ];
        const double v = double( static_cast<long long>( sum[ at[ id ] ] ) ) * unit;
        if ( K == int( I ) ) {
            const P d = P( v > 0 ? v : 1.0 );
            cdia[ I ] = d;
            cdinv[ I ] = P( 1.0 / double( d ) );
            diag = true;
            continue;
        }
        int r = 0;
        for ( int k = 0; k < m; ++k ) r += ck[ k ] < K && ck[ k ] != int( I );
        if ( r < room ) { ccol[ I * room + r ] = K; cval[ I * room + r ] = P( -v ); }
    }
    const bool has_diag = __any( diag );
    if ( lane == 0 ) {
        if ( ! has_diag ) { cdia[ I ] = 1; cdinv[ I ] = 1; }
        ccnt[ I ] = min( max( m - ( has_diag ? 1 : 0 ), 0 ), room );
        if ( over ) tn[ I ] = SA_TMAX;
        if ( over || nkeys > room + 1 || ! ( size < 0x1p62 ) ) state[ S_BAD ] = 1;
    }
}

/// THE GALERKIN ROWS BELOW THE BOTTOM'S LEVEL, where rows are long and few ( at most `SA_DENSE_COLS` columns ): `AP` as a dense matrix, one
/// lane an entry, the row's terms in its order; `P` is read as a dense matrix too ( `k_dense_p` ). The hash's waves took 0.5 ms a level there
constexpr int SA_DENSE_COLS = 256;

template<class P>
__global__ void k_dense_p( int n, int nc, const int *pn, const int *pcol, const P *pval, P *pd ) {
    const int k = int( blockIdx.x ) * blockDim.x + threadIdx.x;
    if ( k >= n * nc ) return;
    const int i = k / nc, K = k % nc, np = pn[ i ];
    P v = 0;
    for ( int q = 0; q < np; ++q ) if ( pcol[ I64( q ) * n + i ] == K ) v = pval[ I64( q ) * n + i ];
    pd[ k ] = v;
}

template<class P>
__global__ void k_dense_ap( Rows<P> A, int nc, const P *pd, double *ap ) {
    const int k = int( blockIdx.x ) * blockDim.x + threadIdx.x;
    if ( k >= int( A.n ) * nc ) return;
    const int i = k / nc, K = k % nc;
    ap[ k ] = double( A.dia[ i ] ) * double( pd[ k ] ) -
              row_sum( A, A.base( i ), A.cnt[ i ], [&]( int j ) { return double( pd[ j * nc + K ] ); } );
}

/// `P^T ( A P )`, one wave a coarse row, a lane the columns `lane + 64 u`; the entries that are not 0 kept, in increasing columns
template<class P>
__global__ __launch_bounds__( 64 ) void k_dense_ptap( Rows<P> A, int nc, const double *ap, const int *pn, const int *pcol, const P *pval, int *tn,
                                                     int *tcol, P *tval, int room, int *ccnt, int *ccol, P *cval, P *cdia, P *cdinv, double *state ) {
    __shared__ int raw[ SA_TMAX ], si[ SA_TMAX ];
    __shared__ double sw[ SA_TMAX ];
    const int lane = threadIdx.x, I = int( blockIdx.x );
    const bool over = tn[ I ] > SA_TMAX;
    const int cnt = sorted_list( I64( I ), A.n, pn, pcol, pval, tn, tcol, tval, raw, si, sw );
    double acc[ SA_DENSE_COLS / 64 ] = {};
    for ( int t = 0; t < cnt; ++t ) {
        const double w = sw[ t ];
        const double *row = ap + I64( si[ t ] ) * nc;
#pragma unroll
        for ( int u = 0; u < SA_DENSE_COLS / 64; ++u ) if ( lane + 64 * u < nc ) acc[ u ] += w * row[ lane + 64 * u ];
    }
    int at = 0;
#pragma unroll
    for ( int u = 0; u < SA_DENSE_COLS / 64; ++u ) {
        const int K = lane + 64 * u;
        const bool keep = K < nc && K != I && acc[ u ] != 0;
        const unsigned long long bal = __ballot( keep );
        const int r = at + __popcll( bal & ( ( 1ull << lane ) - 1 ) );
        if ( keep && r < room ) { ccol[ I64( I ) * room + r ] = K; cval[ I64( I ) * room + r ] = P( -acc[ u ] ); }
        at += __popcll( bal );
        if ( K == I ) {
            const P d = P( acc[ u ] > 0 ? acc[ u ] : 1.0 );
            cdia[ I ] = d;
            cdinv[ I ] = P( 1.0 / double( d ) );
        }
    }
    if ( lane == 0 ) {
        ccnt[ I ] = min( at, room );
        if ( over ) tn[ I ] = SA_TMAX;
        if ( over || at > room ) state[ S_BAD ] = 1;
    }
}

/// the inverse of `A_c + alpha 1 1^T` on the coarsest level ( `alpha` the mean diagonal over `n`: the rank-one term removes the
/// constants, the kernel of a Laplacian ), by Gauss-Jordan in place in LDS, one workgroup; row-major
template<class P>
__global__ __launch_bounds__( TH ) void k_sa_inverse( Rows<P> C, double *inv ) {
    __shared__ double M[ SA_DENSE ][ SA_DENSE + 1 ], rowp[ SA_DENSE ], colp[ SA_DENSE ], sh[ 4 ];
    const int n = int( C.n );
    double s = 0;
    for ( int i = threadIdx.x; i < n; i += TH ) s += double( C.dia[ i ] );
    const double alpha = sum_block( s, sh ) / double( n ) / double( n );
    for ( int k = threadIdx.x; k < n * n; k += TH ) M[ k / n ][ k % n ] = alpha;
    __syncthreads();
    if ( int( threadIdx.x ) < n ) {
        const int i = threadIdx.x;
        M[ i ][ i ] += double( C.dia[ i ] );
        const I64 b = C.base( i );
        for ( int q = 0; q < C.cnt[ i ]; ++q ) M[ i ][ C.col[ b + q * C.step ] ] -= double( C.val[ b + q * C.step ] );
    }
    __syncthreads();
    for ( int p = 0; p < n; ++p ) {
        if ( int( threadIdx.x ) < n ) {
            rowp[ threadIdx.x ] = M[ p ][ threadIdx.x ] / M[ p ][ p ];
            colp[ threadIdx.x ] = M[ threadIdx.x ][ p ];
        }
        __syncthreads();
        const double piv = 1.0 / colp[ p ];
        for ( int k = threadIdx.x; k < n * n; k += TH ) {
            const int r = k / n, c = k % n;
            M[ r ][ c ] = r == p ? ( c == p ? piv : rowp[ c ] ) : ( c == p ? -colp[ r ] * piv : M[ r ][ c ] - colp[ r ] * rowp[ c ] );
        }
        __syncthreads();
    }
    for ( int k = threadIdx.x; k < n * n; k += TH ) inv[ k ] = M[ k / n ][ k % n ];
}

// ---- the dense bottom -----------------------------------------------------------------------------------------------------

template<class P>
struct BottomLevels {
    int nl = 0;
    double w0 = 0, w1 = 0, over = 1;
    const double *inv = nullptr;
    int at[ SA_LEVELS ] = {};                            ///< each level's first row in the LDS vectors
    Level<P> L[ SA_LEVELS ];
};
constexpr int BOP_THREADS = 1024, BOP_LANES = 8;

/// THE BOTTOM'S OPERATOR: columns `NR b .. NR b + NR - 1` of the V-cycle over `B`'s levels, one workgroup, the vectors in LDS ( `NR`
/// values a row: what bounds it is the matrices' reads from L2, which the `NR` columns share ), 8 lanes a row. The first two sweeps
/// on a unit vector touch its row's neighbours alone. Row `c` of `op` is the cycle applied to the unit vector `c`: the cycle is
/// symmetric, so rows serve as columns
template<class P, int NR>
__global__ __launch_bounds__( BOP_THREADS ) void k_bottom_op( BottomLevels<P> B, int rows, P *op ) {
    extern __shared__ char raw[];
    // ( `x` and `t` of every level, then `r` of the levels below the first: there it is a unit vector )
    P *X = reinterpret_cast<P *>( raw ), *T = X + size_t( rows ) * NR, *R = T + size_t( rows ) * NR;
    const int n0 = int( B.L[ 0 ].A.n ), c0 = int( blockIdx.x ) * NR;
    const int lane = threadIdx.x & ( BOP_LANES - 1 ), grp = threadIdx.x / BOP_LANES, ngrp = BOP_THREADS / BOP_LANES;
    auto rhs = [&]( int l, int i, int k ) -> double {
        return l == 0 ? ( i == c0 + k ? 1.0 : 0.0 ) : double( R[ ( B.at[ l ] - n0 + i ) * NR + k ] );
    };
    auto all_lanes = [&]( double *s ) {
#pragma unroll
        for ( int k = 0; k < NR; ++k )
            for ( int o = BOP_LANES / 2; o > 0; o >>= 1 ) s[ k ] += __shfl_xor( s[ k ], o, BOP_LANES );
    };
    auto pick = [&]( const double *s ) {                 // ( lane `k` takes column `k`'s sum )
        double v = s[ 0 ];
#pragma unroll
        for ( int k = 1; k < NR; ++k ) v = lane == k ? s[ k ] : v;
        return v;
    };
    auto product = [&]( const Rows<P> &A, int i, double *s, auto f ) {          // `s_k = sum_j val f( j, k )`, in every lane
#pragma unroll
        for ( int k = 0; k < NR; ++k ) s[ k ] = 0;
        const int c = A.cnt[ i ];
        const I64 b = A.base( i );
        for ( int q = lane; q < c; q += 4 * BOP_LANES ) {
            double v[ 4 ];
            int j[ 4 ];
#pragma unroll
            for ( int u = 0; u < 4; ++u ) {
                const int e = q + u * BOP_LANES < c ? q + u * BOP_LANES : q;
                v[ u ] = double( A.val[ b + e ] );
                j[ u ] = A.col[ b + e ];
            }
#pragma unroll
            for ( int u = 0; u < 4; ++u )
                if ( q + u * BOP_LANES < c )
#pragma unroll
                    for ( int k = 0; k < NR; ++k ) s[ k ] += v[ u ] * f( j[ u ], k );
        }
        all_lanes( s );
    };
    for ( int l = 0; l + 1 < B.nl; ++l ) {
        const Level<P> &L = B.L[ l ], &C = B.L[ l + 1 ];
        P *x = X + size_t( B.at[ l ] ) * NR, *t = T + size_t( B.at[ l ] ) * NR, *rc = R + size_t( B.at[ l + 1 ] - n0 ) * NR;
        const int n = int( L.A.n );
        double s[ NR ];
        if ( l == 0 ) {
            for ( int k = threadIdx.x; k < n * NR; k += BOP_THREADS ) x[ k ] = 0;
            __syncthreads();
            for ( int k = 0; k < NR && c0 + k < n; ++k ) {
                const int c = c0 + k, cnt = L.A.cnt[ c ];
                const double y = B.w0 * double( L.dinv[ c ] );
                for ( int q = threadIdx.x; q <= cnt; q += BOP_THREADS ) {
                    const int i = q < cnt ? L.A.col[ L.A.base( c ) + q ] : c;
                    const double e = q < cnt ? double( L.A.val[ L.A.base( c ) + q ] ) * y : 1 - double( L.A.dia[ c ] ) * y;
                    x[ i * NR + k ] = P( ( q < cnt ? 0.0 : y ) + B.w1 * double( L.dinv[ i ] ) * e );
                }
            }
        } else
            for ( int i = grp; i < n; i += ngrp ) {
                product( L.A, i, s, [&]( int j, int k ) { return B.w0 * double( L.dinv[ j ] ) * rhs( l, j, k ); } );
                if ( lane < NR ) {
                    const double ri = rhs( l, i, lane ), di = double( L.dinv[ i ] ), y = B.w0 * di * ri;
                    x[ i * NR + lane ] = P( y + B.w1 * di * ( ri - ( double( L.A.dia[ i ] ) * y - pick( s ) ) ) );
                }
            }
        __syncthreads();
        for ( int i = grp; i < n; i += ngrp ) {
            product( L.A, i, s, [&]( int j, int k ) { return double( x[ j * NR + k ] ); } );
            if ( lane < NR ) t[ i * NR + lane ] = P( rhs( l, i, lane ) - ( double( L.A.dia[ i ] ) * double( x[ i * NR + lane ] ) - pick( s ) ) );
        }
        __syncthreads();
        for ( int I = grp; I < int( C.A.n ); I += ngrp ) {
#pragma unroll
            for ( int k = 0; k < NR; ++k ) s[ k ] = 0;
            const int c = C.tn[ I ];
            for ( int q = lane; q < c; q += BOP_LANES ) {
                const double v = double( C.tval[ I64( I ) * SA_TMAX + q ] );
                const int j = C.tcol[ I64( I ) * SA_TMAX + q ];
#pragma unroll
                for ( int k = 0; k < NR; ++k ) s[ k ] += v * double( t[ j * NR + k ] );
            }
            all_lanes( s );
            if ( lane < NR ) rc[ I * NR + lane ] = P( pick( s ) );
        }
        __syncthreads();
    }
    {
        const int a = B.at[ B.nl - 1 ], nd = int( B.L[ B.nl - 1 ].A.n );
        for ( int k = threadIdx.x; k < nd * NR; k += BOP_THREADS ) {
            const int i = k / NR, c = k % NR;
            double v = 0;
            for ( int j = 0; j < nd; ++j ) v += B.inv[ i * nd + j ] * rhs( B.nl - 1, j, c );
            T[ size_t( a + i ) * NR + c ] = P( v );
        }
        __syncthreads();
    }
    for ( int l = B.nl - 2; l >= 0; --l ) {
        const Level<P> &L = B.L[ l ];
        const P *xc = T + size_t( B.at[ l + 1 ] ) * NR;
        P *x = X + size_t( B.at[ l ] ) * NR, *t = T + size_t( B.at[ l ] ) * NR;
        const int n = int( L.A.n );
        for ( int k = threadIdx.x; k < n * NR; k += BOP_THREADS ) {
            const int i = k / NR, c = k % NR, np = L.pn[ i ];
            double v = 0;
            for ( int q = 0; q < np; ++q ) v += double( L.pval[ I64( q ) * n + i ] ) * double( xc[ L.pcol[ I64( q ) * n + i ] * NR + c ] );
            t[ k ] = P( double( x[ k ] ) + B.over * v );
        }
        __syncthreads();
        P *in = t, *out = x;
        for ( int sweep = 0; sweep < 2; ++sweep ) {
            const double w = sweep ? B.w1 : B.w0;
            double s[ NR ];
            for ( int i = grp; i < n; i += ngrp ) {
                product( L.A, i, s, [&]( int j, int k ) { return double( in[ j * NR + k ] ); } );
                if ( lane < NR ) {
                    const double xi = double( in[ i * NR + lane ] );
                    out[ i * NR + lane ] = P( xi + w * double( L.dinv[ i ] ) * ( rhs( l, i, lane ) - ( double( L.A.dia[ i ] ) * xi - pick( s ) ) ) );
                }
            }
            __syncthreads();
            P *sw = in; in = out; out = sw;              // ( two sweeps: the last lands in `t` )
        }
    }
    for ( int k = 0; k < NR && c0 + k < n0; ++k )
        for ( int i = threadIdx.x; i < n0; i += BOP_THREADS ) op[ size_t( c0 + k ) * n0 + i ] = T[ size_t( i ) * NR + k ];
}

/// `x = op r`, one wave a row ( HBM / L2: 4 `n^2` bytes )
template<class P>
__global__ __launch_bounds__( TH ) void k_bottom_apply( int n, const P *op, const P *r, P *x, const double *state ) {
    if ( state[ S_DONE ] != 0 ) return;
    const int row = int( blockIdx.x ) * ( TH / 64 ) + int( threadIdx.x >> 6 ), lane = threadIdx.x & 63;
    if ( row >= n ) return;
    const P *o = op + size_t( row ) * n;
    double s0 = 0, s1 = 0, s2 = 0, s3 = 0;
    int j = lane;
    for ( ; j + 192 < n; j += 256 ) {
        s0 += double( o[ j ] ) * double( r[ j ] );
        s1 += double( o[ j + 64 ] ) * double( r[ j + 64 ] );
        s2 += double( o[ j + 128 ] ) * double( r[ j + 128 ] );
        s3 += double( o[ j + 192 ] ) * double( r[ j + 192 ] );
    }
    for ( ; j < n; j += 64 ) s0 += double( o[ j ] ) * double( r[ j ] );
    const double s = wave_sum( ( s0 + s1 ) + ( s2 + s3 ) );
    if ( lane == 0 ) x[ row ] = P( s );
}

// ---- the cycle's passes ---------------------------------------------------------------------------------------------------
// The finest level: one row a lane, each block a contiguous range of rows, the XCDs contiguous ranges of blocks.

/// the rows of the calling block when `n` rows are cut in `gridDim.x` ranges of whole blocks of `TH`
struct Range { I64 lo, hi; };
__device__ __forceinline__ Range range_of( I64 n ) {
    const I64 chunk = ( n + I64( gridDim.x ) * TH - 1 ) / ( I64( gridDim.x ) * TH ) * TH;
    const I64 lo = xcd_block() * chunk;
    return { lo, lo + chunk < n ? lo + chunk : n };
}

/// the first two sweeps from zero: `y = w0 D^-1 r` is given, `x = y + w1 D^-1 ( r - A y )`. `TEST`: the outer iteration's convergence
/// test first, on the partials of `r . r` ( every block takes the same decision, one writes it down )
template<class P, bool TEST>
__global__ __launch_bounds__( TH ) void k_fine_two( Rows<P> A, const P *dinv, const P *r, const P *y, P *x, double w1, const double *part, int nblk,
                                                   double *state ) {
    __shared__ double sh[ 4 ];
    if ( TEST ? block_stopped( &state[ S_DONE ] ) : state[ S_DONE ] != 0 ) return;
    if ( TEST ) {
        const double err = sqrt( sum_partials( part + P_RR * SA_BLOCKS, nblk, sh ) ) / state[ S_NB ];
        const bool done = err <= state[ S_TOL ];
        if ( blockIdx.x == 0 && threadIdx.x == 0 ) {
            state[ S_ERR ] = err;
            state[ S_IT ] += 1;
            if ( done ) state[ S_DONE ] = 1;
        }
        if ( done ) return;
    }
    const Range g = range_of( A.n );
    for ( I64 i = g.lo + threadIdx.x; i < g.hi; i += TH ) {
        const double yi = double( y[ i ] );
        const double s = double( A.dia[ i ] ) * yi - row_sum( A, A.base( i ), A.cnt[ i ], [&]( int j ) { return double( y[ j ] ); } );
        x[ i ] = P( yi + w1 * double( dinv[ i ] ) * ( double( r[ i ] ) - s ) );
    }
}

/// `e = r - A x`
template<class P>
__global__ __launch_bounds__( TH ) void k_fine_res( Rows<P> A, const P *r, const P *x, P *e, const double *state ) {
    if ( state[ S_DONE ] != 0 ) return;
    const Range g = range_of( A.n );
    for ( I64 i = g.lo + threadIdx.x; i < g.hi; i += TH )
        e[ i ] = P( double( r[ i ] ) - ( double( A.dia[ i ] ) * double( x[ i ] ) -
                                         row_sum( A, A.base( i ), A.cnt[ i ], [&]( int j ) { return double( x[ j ] ); } ) ) );
}

/// one sweep, `xo = x + w D^-1 ( r - A x )`; `DOT`: the partials of `xo . q` too ( the flexible CG's `z . q` )
template<class P, bool DOT, class R>
__global__ __launch_bounds__( TH ) void k_fine_sweep( Rows<P> A, const P *dinv, const P *r, const P *x, P *xo, double w, const R *q, double *part,
                                                     const double *state ) {
    __shared__ double sh[ 4 ];
    if ( state[ S_DONE ] != 0 ) return;
    double acc = 0;
    const Range g = range_of( A.n );
    for ( I64 i = g.lo + threadIdx.x; i < g.hi; i += TH ) {
        const double xi = double( x[ i ] );
        const double s = double( A.dia[ i ] ) * xi - row_sum( A, A.base( i ), A.cnt[ i ], [&]( int j ) { return double( x[ j ] ); } );
        const P v = P( xi + w * double( dinv[ i ] ) * ( double( r[ i ] ) - s ) );
        xo[ i ] = v;
        if ( DOT ) acc += double( v ) * double( q[ i ] );
    }
    if ( DOT ) {
        const double s = sum_block( acc, sh );
        if ( threadIdx.x == 0 ) part[ P_ZQ * SA_BLOCKS + blockIdx.x ] = s;
    }
}

/// `t = x + over P xc`, one row a lane
template<class P>
__global__ __launch_bounds__( TH ) void k_prolong( I64 n, const int *pn, const int *pcol, const P *pval, const P *xc, const P *x, double over, P *t,
                                                  const double *state ) {
    if ( state[ S_DONE ] != 0 ) return;
    const I64 i = I64( xcd_block() ) * TH + threadIdx.x;
    if ( i >= n ) return;
    const int np = pn[ i ];
    double s = 0;
    for ( int q = 0; q < np; ++q ) s += double( pval[ I64( q ) * n + i ] ) * double( xc[ pcol[ I64( q ) * n + i ] ] );
    t[ i ] = P( double( x[ i ] ) + over * s );
}

/// `r = P^T e` and `y = w0 D^-1 r` on the level below, eight lanes a row
template<class P>
__global__ __launch_bounds__( TH ) void k_restrict_to( I64 nc, const int *tn, const int *tcol, const P *tval, const P *e, const P *dinv, double w0,
                                                      P *r, P *y, const double *state ) {
    if ( state[ S_DONE ] != 0 ) return;
    const I64 I = ( I64( xcd_block() ) * TH + threadIdx.x ) >> 3;
    const int lane = threadIdx.x & 7;
    if ( I >= nc ) return;
    const int c = tn[ I ];
    double s = 0;
    for ( int q = lane; q < c; q += 8 ) s += double( tval[ I * SA_TMAX + q ] ) * double( e[ tcol[ I * SA_TMAX + q ] ] );
    for ( int o = 4; o > 0; o >>= 1 ) s += __shfl_xor( s, o, 8 );
    if ( lane == 0 ) { r[ I ] = P( s ); y[ I ] = P( w0 * double( dinv[ I ] ) * s ); }
}

/// the passes of a coarser level, `G` lanes a row: the first two sweeps ( MODE 0 ), the residual ( 1 ), a sweep ( 2 )
template<class P, int G, int MODE>
__global__ __launch_bounds__( TH ) void k_coarse_pass( Rows<P> A, const P *dinv, const P *r, const P *x, P *xo, double w, const double *state ) {
    if ( state[ S_DONE ] != 0 ) return;
    const I64 i = ( I64( xcd_block() ) * TH + threadIdx.x ) / G;
    const int lane = threadIdx.x & ( G - 1 );
    if ( i >= A.n ) return;
    const double s = row_sum_lanes<G>( A, A.base( i ), A.cnt[ i ], lane, [&]( int j ) { return double( x[ j ] ); } );
    if ( lane ) return;
    const double xi = double( x[ i ] ), e = double( r[ i ] ) - ( double( A.dia[ i ] ) * xi - s );
    xo[ i ] = P( MODE == 1 ? e : xi + w * double( dinv[ i ] ) * e );
}

// ---- the outer iteration --------------------------------------------------------------------------------------------------

template<class P>
__global__ __launch_bounds__( TH ) void k_outer_init( I64 n, const double *b, const P *dinv, double w0, double *d, double *r, double *p, P *rp, P *y,
                                                     double *part ) {
    __shared__ double sh[ 4 ];
    double acc = 0;
    const Range g = range_of( n );
    for ( I64 i = g.lo + threadIdx.x; i < g.hi; i += TH ) {
        const double v = b[ i ];
        d[ i ] = 0;
        p[ i ] = 0;
        r[ i ] = v;
        rp[ i ] = P( v );
        y[ i ] = P( w0 * double( dinv[ i ] ) * v );
        acc += v * v;
    }
    const double s = sum_block( acc, sh );
    if ( threadIdx.x == 0 ) part[ blockIdx.x ] = s;
}

/// ( a system whose hierarchy could not be built stops here: the iterations queued behind are no-ops )
__global__ __launch_bounds__( TH ) void k_outer_start( const double *part, int nblk, double *state, double tol ) {
    __shared__ double sh[ 4 ];
    const double bb = sum_partials( part, nblk, sh );
    if ( threadIdx.x == 0 ) {
        state[ S_NB ] = sqrt( bb );
        state[ S_ERR ] = 1;
        state[ S_DONE ] = bb > 0 && state[ S_BAD ] == 0 ? 0.0 : 1.0;
        state[ S_TOL ] = tol;
    }
}

/// `p = z + beta p_old` formed for the row and each neighbour, `q = A p`, the partials of `p . q` and `p . r`; `beta = -z . q / p . q`
/// summed by every block ( 0 at the first iteration )
template<class P>
__global__ __launch_bounds__( TH ) void k_direction( Rows<double> A, const P *z, const double *po, const double *r, double *pn, double *q, double *part,
                                                    int nblk, const double *state ) {
    __shared__ double sh[ 4 ];
    if ( state[ S_DONE ] != 0 ) return;
    const double zq = sum_partials( part + P_ZQ * SA_BLOCKS, nblk, sh ), pq0 = state[ S_PQ ];
    const double beta = state[ S_IT ] > 0 && pq0 > 0 ? -zq / pq0 : 0.0;
    double pq = 0, pr = 0;
    const Range g = range_of( A.n );
    for ( I64 i = g.lo + threadIdx.x; i < g.hi; i += TH ) {
        const double pi = double( z[ i ] ) + beta * po[ i ];
        const double s = A.dia[ i ] * pi - row_sum( A, A.base( i ), A.cnt[ i ], [&]( int j ) { return double( z[ j ] ) + beta * po[ j ]; } );
        pn[ i ] = pi;
        q[ i ] = s;
        pq += pi * s;
        pr += pi * r[ i ];
    }
    pq = sum_block( pq, sh );
    pr = sum_block( pr, sh );
    if ( threadIdx.x == 0 ) { part[ P_PQ * SA_BLOCKS + blockIdx.x ] = pq; part[ P_PR * SA_BLOCKS + blockIdx.x ] = pr; }
}

/// `alpha = p . r / p . q`, `d += alpha p`, `r -= alpha q`, the cycle's copies of `r` and `w0 D^-1 r`, the partials of `r . r`.
/// `p . q <= 0` ( a breakdown ) stops the iteration as a failure
template<class P>
__global__ __launch_bounds__( TH ) void k_update( I64 n, const double *p, const double *q, const P *dinv, double w0, double *d, double *r, P *rp, P *y,
                                                 double *part, int nblk, double *state ) {
    __shared__ double sh[ 4 ];
    if ( block_stopped( &state[ S_DONE ] ) ) return;
    const double pq = sum_partials( part + P_PQ * SA_BLOCKS, nblk, sh ), pr = sum_partials( part + P_PR * SA_BLOCKS, nblk, sh );
    if ( ! ( pq > 0 ) ) {
        if ( blockIdx.x == 0 && threadIdx.x == 0 ) { state[ S_PQ ] = pq; state[ S_DONE ] = 1; state[ S_FAILED ] = 1; }
        return;
    }
    const double alpha = pr / pq;
    if ( blockIdx.x == 0 && threadIdx.x == 0 ) state[ S_PQ ] = pq;
    double acc = 0;
    const Range g = range_of( n );
    for ( I64 i = g.lo + threadIdx.x; i < g.hi; i += TH ) {
        d[ i ] += alpha * p[ i ];
        const double v = r[ i ] - alpha * q[ i ];
        r[ i ] = v;
        rp[ i ] = P( v );
        y[ i ] = P( w0 * double( dinv[ i ] ) * v );
        acc += v * v;
    }
    const double s = sum_block( acc, sh );
    if ( threadIdx.x == 0 ) part[ P_RR * SA_BLOCKS + blockIdx.x ] = s;
}

/// the partials of `| b - A d |^2`, then the true relative residual ( the recurrence only estimates it )
__global__ __launch_bounds__( TH ) void k_true( Rows<double> A, const double *b, const double *d, double *part ) {
    __shared__ double sh[ 4 ];
    double acc = 0;
    const Range g = range_of( A.n );
    for ( I64 i = g.lo + threadIdx.x; i < g.hi; i += TH ) {
        const double e = b[ i ] - ( A.dia[ i ] * d[ i ] - row_sum( A, A.base( i ), A.cnt[ i ], [&]( int j ) { return d[ j ]; } ) );
        acc += e * e;
    }
    const double s = sum_block( acc, sh );
    if ( threadIdx.x == 0 ) part[ blockIdx.x ] = s;
}
__global__ __launch_bounds__( TH ) void k_true_end( const double *part, int nblk, double *state ) {
    __shared__ double sh[ 4 ];
    const double ee = sum_partials( part, nblk, sh );
    if ( threadIdx.x == 0 ) state[ S_TRUE ] = state[ S_NB ] > 0 ? sqrt( ee ) / state[ S_NB ] : 0.0;
}

/// the levels' sizes: `n[ 0 ]` the system's, `lb` the dense bottom, the last one at most `SA_DENSE`. The first aggregates hold 4
/// ranks where that takes no more levels above the bottom than 8 ( 27 iterations against 38 on the 200k image Laplacian, the same
/// launches ), 8 elsewhere and below ( a level more costs six launches an iteration ). In 3D only where the level they make is the bottom itself:
/// its rows have up to 120 entries, and the next level's then 280 and more, past any room ( from 12k seeds on every system was handed over
/// to the K-cycle; three systems of 20k / 60k / 250k / 1M uniform seeds: 28.9 / 44.7 / 80 / 140 ms so, 4.0 / 5.4 / 11.6 / 37 ms with 8 )
struct Sizes { int nl = 0, lb = 0; I64 n[ SA_LEVELS ]; int pack[ SA_LEVELS ]; };
Sizes sizes_of( I64 n, bool wide ) {
    auto above = [&]( I64 p ) { int k = 1; for ( I64 m = ( n + p - 1 ) / p; m > SA_BOTTOM; m = ( m + 7 ) / 8 ) ++k; return k; };
    Sizes s;
    s.n[ 0 ] = n;
    s.pack[ 0 ] = above( 4 ) == above( 8 ) && ! ( wide && above( 4 ) > 1 ) ? 4 : 8;
    s.lb = above( s.pack[ 0 ] );
    int l = 0;
    while ( l < s.lb || s.n[ l ] > SA_DENSE ) {
        if ( l ) s.pack[ l ] = 8;
        s.n[ l + 1 ] = ( s.n[ l ] + s.pack[ l ] - 1 ) / s.pack[ l ];
        ++l;
        SDOT_CHECK( l + 1 < SA_LEVELS, "smoothed aggregation: too many levels" );
    }
    s.nl = l + 1;
    return s;
}

/// the entries a row of level `l + 1` has room for. 2D: 17 to 22 a row on the first coarse level, 30 to 60 on the next; 3D, at most: 100 ( 120
/// with packs of 4 ), 150, 180 ( 1M seeds ); below the bottom's level rows may be full
int room_of( const Sizes &sz, int l, bool wide ) { return l >= sz.lb ? SA_DENSE_COLS : wide && l ? SA_SMAX : wide || l ? 192 : 96; }

/// the prolongation's rows drop what is below this part of their largest entry: more where rows are long, in 3D, and more still between the
/// levels above the bottom there ( the 1M seeds' third level has rows of 180 entries so, of 260 at 0.2 )
double theta_of( const Sizes &sz, int l, bool wide ) { return ! wide ? 0.1 : l && l < sz.lb ? 0.25 : 0.2; }

template<class P>
FcgResult solve_with( const Csr &L, const P *val, const P *dia, const double *b, double *d, double tol, int maxit, const MgOptions &o, hipStream_t st,
                      int &nb_levels, int prev_its, double drop, const std::string &pfx ) {
    constexpr bool same = std::is_same<P, double>::value;
    Arena &A = arena();
    const I64 n = L.n;
    const bool wide = L.nnz > 10 * n;                    // ( 3D: 15.5 entries a row, 2D: 6 )
    const Sizes sz = sizes_of( n, wide );
    const double omega = 2.0 / 3, over = 1.2;
    // the sweeps' dampings: the Chebyshev nodes of [ 0.2, 2 ] ( 2 bounds the spectrum of `D^-1 A` )
    const double th = 1.1, de = 0.9, pi = 3.14159265358979323846;
    const double w0 = 1 / ( th + de * std::cos( pi / 4 ) ), w1 = 1 / ( th + de * std::cos( 3 * pi / 4 ) );

    double *state = A.get<double>( pfx + ".state", S_NB_STATE );
    double *hs = pinned<double>( pfx + ".hstate", S_NB_STATE );
    double *part = A.get<double>( pfx + ".part", size_t( P_NB ) * SA_BLOCKS );
    Level<P> V[ SA_LEVELS ];
    V[ 0 ].A.n = n; V[ 0 ].A.step = L.step; V[ 0 ].A.row_off = L.row_off; V[ 0 ].A.cnt = L.row_cnt; V[ 0 ].A.col = L.col;
    V[ 0 ].A.val = val; V[ 0 ].A.dia = dia;
    I64 lists = 0;
    for ( int l = 1; l < sz.nl; ++l ) lists += sz.n[ l ];
    int *tn = A.get<int>( pfx + ".tn", size_t( lists ) );
    k_sa_zero<<<blocks_for( std::max<I64>( lists, S_NB_STATE ), TH ), TH, 0, st>>>( int( lists ), tn, state );
    V[ 0 ].dinv = A.get<P>( pfx + ".dinv0", size_t( n ) );
    k_sa_dinv<P><<<blocks_for( n, TH ), TH, 0, st>>>( n, dia, V[ 0 ].dinv );
    for ( int l = 0; l + 1 < sz.nl; ++l ) {
        Level<P> &F = V[ l ], &C = V[ l + 1 ];
        const size_t nf = size_t( sz.n[ l ] ), nc = size_t( sz.n[ l + 1 ] );
        const std::string tag = pfx + "." + std::to_string( l );
        const int room = room_of( sz, l, wide );
        const double theta = std::min( drop * theta_of( sz, l, wide ), 0.9 );
        F.pn = A.get<int>( tag + ".pn", nf );
        F.pcol = A.get<int>( tag + ".pcol", nf * SA_PMAX );
        F.pval = A.get<P>( tag + ".pval", nf * SA_PMAX );
        C.tn = tn; tn += nc;
        C.tcol = A.get<int>( tag + ".tcol", nc * SA_TMAX );
        C.tval = A.get<P>( tag + ".tval", nc * SA_TMAX );
        int *cnt = A.get<int>( tag + ".cnt", nc ), *col = A.get<int>( tag + ".col", nc * room );
        P *cval = A.get<P>( tag + ".val", nc * room ), *cdia = A.get<P>( tag + ".dia", nc );
        C.dinv = A.get<P>( tag + ".dinv", nc );
        C.A.n = I64( nc ); C.A.rs = room; C.A.cnt = cnt; C.A.col = col; C.A.val = cval; C.A.dia = cdia;
        // lanes a row by its expected length: 6 and 15.5 entries on the finest level, 17 to 80 below
        if ( l == 0 && ! wide ) k_prolongator<P, 8, 4><<<blocks_for( 8 * I64( nf ), TH ), TH, 0, st>>>( F.A, sz.pack[ l ], omega, theta, F.pn, F.pcol, F.pval, C.tn, C.tcol );
        else if ( l == 0 )      k_prolongator<P, 16, 4><<<blocks_for( 16 * I64( nf ), TH ), TH, 0, st>>>( F.A, sz.pack[ l ], omega, theta, F.pn, F.pcol, F.pval, C.tn, C.tcol );
        else                    k_prolongator<P, 32, 4><<<blocks_for( 32 * I64( nf ), TH ), TH, 0, st>>>( F.A, sz.pack[ l ], omega, theta, F.pn, F.pcol, F.pval, C.tn, C.tcol );
        if ( l >= sz.lb && nc <= size_t( SA_DENSE_COLS ) ) {
            P *pd = A.get<P>( pfx + ".pd", size_t( SA_BOTTOM ) * SA_DENSE_COLS );
            double *ap = A.get<double>( pfx + ".ap", size_t( SA_BOTTOM ) * SA_DENSE_COLS );
            const unsigned db = blocks_for( I64( nf * nc ), TH );
            k_dense_p<P><<<db, TH, 0, st>>>( int( nf ), int( nc ), F.pn, F.pcol, F.pval, pd );
            k_dense_ap<P><<<db, TH, 0, st>>>( F.A, int( nc ), pd, ap );
            k_dense_ptap<P><<<unsigned( nc ), 64, 0, st>>>( F.A, int( nc ), ap, F.pn, F.pcol, F.pval, C.tn, C.tcol, C.tval, room, cnt, col, cval, cdia,
                                                           C.dinv, state );
        } else
            k_galerkin<P><<<unsigned( nc ), 64, 0, st>>>( F.A, F.pn, F.pcol, F.pval, C.tn, C.tcol, C.tval, room, cnt, col, cval, cdia, C.dinv, state );
        check_launch( "k_galerkin" );
    }
    // the bottom: the coarsest level's inverse, then the operator of the levels from `lb`
    double *inv = A.get<double>( pfx + ".inv", size_t( SA_DENSE ) * SA_DENSE );
    k_sa_inverse<P><<<1, TH, 0, st>>>( V[ sz.nl - 1 ].A, inv );
    const int nb = int( sz.n[ sz.lb ] );
    P *op = A.get<P>( pfx + ".op", size_t( nb ) * nb );
    BottomLevels<P> B;
    B.nl = sz.nl - sz.lb; B.w0 = w0; B.w1 = w1; B.over = over; B.inv = inv;
    int brows = 0;
    for ( int l = sz.lb; l < sz.nl; ++l ) { B.L[ l - sz.lb ] = V[ l ]; B.at[ l - sz.lb ] = brows; brows += int( sz.n[ l ] ); }
    constexpr int NR = same ? 2 : 4;                     // ( at most 2048 + 288 rows: 79 KB of LDS, two workgroups a CU )
    k_bottom_op<P, NR><<<blocks_for( nb, NR ), BOP_THREADS, size_t( 3 * brows - nb ) * NR * sizeof( P ), st>>>( B, brows, op );
    check_launch( "k_bottom_op" );
    nb_levels = sz.nl;

    // the vectors
    for ( int l = 0; l <= sz.lb; ++l ) {
        const size_t m = size_t( sz.n[ l ] );
        const std::string tag = pfx + ".v" + std::to_string( l );
        V[ l ].x = A.get<P>( tag + ".x", m ); V[ l ].y = A.get<P>( tag + ".y", m );
        if ( l || ! same ) V[ l ].r = A.get<P>( tag + ".r", m );
        if ( l < sz.lb ) { V[ l ].t = A.get<P>( tag + ".t", m ); V[ l ].e = A.get<P>( tag + ".e", m ); }
    }
    double *r = A.get<double>( pfx + ".r", size_t( n ) ), *q = A.get<double>( pfx + ".q", size_t( n ) );
    double *p0 = A.get<double>( pfx + ".p0", size_t( n ) ), *p1 = A.get<double>( pfx + ".p1", size_t( n ) );
    if constexpr ( same ) V[ 0 ].r = r;
    Rows<double> A0;
    A0.n = n; A0.step = L.step; A0.row_off = L.row_off; A0.cnt = L.row_cnt; A0.col = L.col; A0.val = L.val; A0.dia = L.dia;
    const int nblk = int( std::min<I64>( blocks_for( n, TH ), SA_BLOCKS ) );

    // one cycle on `V[ 0 ].r` into `V[ 0 ].x`
    auto cycle = [&]( hipStream_t s, bool test ) {
        const Level<P> &F = V[ 0 ];
        if ( test ) k_fine_two<P, true><<<nblk, TH, 0, s>>>( F.A, F.dinv, F.r, F.y, F.x, w1, part, nblk, state );
        else        k_fine_two<P, false><<<nblk, TH, 0, s>>>( F.A, F.dinv, F.r, F.y, F.x, w1, part, nblk, state );
        k_fine_res<P><<<nblk, TH, 0, s>>>( F.A, F.r, F.x, F.e, state );
        for ( int l = 1; l <= sz.lb; ++l ) {
            const Level<P> &C = V[ l ];
            k_restrict_to<P><<<blocks_for( 8 * C.A.n, TH ), TH, 0, s>>>( C.A.n, C.tn, C.tcol, C.tval, V[ l - 1 ].e, C.dinv, w0, C.r, C.y, state );
            if ( l == sz.lb ) { k_bottom_apply<P><<<blocks_for( nb, TH / 64 ), TH, 0, s>>>( nb, op, C.r, C.x, state ); break; }
            // ( eight lanes a row of ~17 entries, sixteen from the next level on and in 3D )
            if ( l == 1 && ! wide ) {
                k_coarse_pass<P, 8, 0><<<blocks_for( 8 * C.A.n, TH ), TH, 0, s>>>( C.A, C.dinv, C.r, C.y, C.x, w1, state );
                k_coarse_pass<P, 8, 1><<<blocks_for( 8 * C.A.n, TH ), TH, 0, s>>>( C.A, C.dinv, C.r, C.x, C.e, 0.0, state );
            } else {
                k_coarse_pass<P, 16, 0><<<blocks_for( 16 * C.A.n, TH ), TH, 0, s>>>( C.A, C.dinv, C.r, C.y, C.x, w1, state );
                k_coarse_pass<P, 16, 1><<<blocks_for( 16 * C.A.n, TH ), TH, 0, s>>>( C.A, C.dinv, C.r, C.x, C.e, 0.0, state );
            }
        }
        for ( int l = sz.lb - 1; l >= 1; --l ) {
            const Level<P> &C = V[ l ];
            k_prolong<P><<<blocks_for( C.A.n, TH ), TH, 0, s>>>( C.A.n, C.pn, C.pcol, C.pval, V[ l + 1 ].x, C.x, over, C.t, state );
            if ( l == 1 && ! wide ) {
                k_coarse_pass<P, 8, 2><<<blocks_for( 8 * C.A.n, TH ), TH, 0, s>>>( C.A, C.dinv, C.r, C.t, C.e, w0, state );
                k_coarse_pass<P, 8, 2><<<blocks_for( 8 * C.A.n, TH ), TH, 0, s>>>( C.A, C.dinv, C.r, C.e, C.x, w1, state );
            } else {
                k_coarse_pass<P, 16, 2><<<blocks_for( 16 * C.A.n, TH ), TH, 0, s>>>( C.A, C.dinv, C.r, C.t, C.e, w0, state );
                k_coarse_pass<P, 16, 2><<<blocks_for( 16 * C.A.n, TH ), TH, 0, s>>>( C.A, C.dinv, C.r, C.e, C.x, w1, state );
            }
        }
        k_prolong<P><<<blocks_for( n, TH ), TH, 0, s>>>( n, F.pn, F.pcol, F.pval, V[ 1 ].x, F.x, over, F.t, state );
        k_fine_sweep<P, false, double><<<nblk, TH, 0, s>>>( F.A, F.dinv, F.r, F.t, F.e, w0, nullptr, nullptr, state );
        k_fine_sweep<P, true, double><<<nblk, TH, 0, s>>>( F.A, F.dinv, F.r, F.e, F.x, w1, q, part, state );
    };
    k_outer_init<P><<<nblk, TH, 0, st>>>( n, b, V[ 0 ].dinv, w0, d, r, p0, V[ 0 ].r, V[ 0 ].y, part );
    k_outer_start<<<1, TH, 0, st>>>( part, nblk, state, tol );
    // ( `q` is read by the cycle's last kernel: the first cycle's `z . q` is not used )
    SDOT_HIP( hipMemcpyAsync( q, r, sizeof( double ) * size_t( n ), hipMemcpyDeviceToDevice, st ) );
    cycle( st, false );
    check_launch( "smoothed aggregation: start" );
    constexpr int batch = 4;                             // ( even: `p0` and `p1` change places each iteration )
    auto iterations = [&]( hipStream_t s, bool timed_first ) {
        for ( int c = 0; c < batch; ++c ) {
            Timing::Pending tp;
            const bool timed = timed_first && c == 0 && timing().begin( TK_SPMV, s, tp );
            k_direction<P><<<nblk, TH, 0, s>>>( A0, V[ 0 ].x, c % 2 ? p1 : p0, r, c % 2 ? p0 : p1, q, part, nblk, state );
            if ( timed ) {
                timing().end( tp, s );
                // ( offsets, counts and diagonal; `z`, both directions, `r` and `q`; the entries )
                timing().spmv_bytes += double( n ) * ( 4 + 4 + 8 + sizeof( P ) + 4 * 8 ) + double( L.nnz ) * ( 4 + 8 );
            }
            k_update<P><<<nblk, TH, 0, s>>>( n, c % 2 ? p0 : p1, q, V[ 0 ].dinv, w0, d, r, V[ 0 ].r, V[ 0 ].y, part, nblk, state );
            cycle( s, true );
        }
    };
    hipGraphExec_t exec = nullptr;
    if ( o.graphs ) {
        Key key;
        key.val( int( 0x5a ) ); key.val( int( sizeof( P ) ) ); key.val( n ); key.val( L.step ); key.val( wide );
        key.val( L.row_off ); key.val( L.row_cnt ); key.val( L.col ); key.val( L.val ); key.val( L.dia ); key.val( val ); key.val( dia );
        for ( int l = 0; l <= sz.lb; ++l ) {
            const Level<P> &W = V[ l ];
            key.val( sz.n[ l ] ); key.val( W.A.cnt ); key.val( W.A.col ); key.val( W.A.val ); key.val( W.A.dia ); key.val( W.A.rs );
            key.val( W.dinv ); key.val( W.pn ); key.val( W.pcol ); key.val( W.pval ); key.val( W.tn ); key.val( W.tcol ); key.val( W.tval );
            key.val( W.r ); key.val( W.y ); key.val( W.x ); key.val( W.t ); key.val( W.e );
        }
        key.val( op ); key.val( part ); key.val( state ); key.val( r ); key.val( q ); key.val( p0 ); key.val( p1 ); key.val( d );
        exec = g_graphs.find( key.b );
        hipStream_t cs = exec ? nullptr : g_capture.get();
        if ( ! exec && cs && hipStreamBeginCapture( cs, hipStreamCaptureModeThreadLocal ) == hipSuccess ) {
            hipGraph_t g = nullptr;
            iterations( cs, false );
            const hipError_t e = hipStreamEndCapture( cs, &g );
            if ( e == hipSuccess && g && hipGraphInstantiate( &exec, g, nullptr, nullptr, 0 ) == hipSuccess ) {
                g_graphs.put( key.b, g, exec );
                timing().graph_captures += 1;
            } else {                                     // ( no graph: the batches are launched one by one )
                exec = nullptr;
                if ( g ) (void) hipGraphDestroy( g );
            }
        }
        (void) hipGetLastError();
    }
    FcgResult res;
    int launched = 0;
    // batches queued before the first look at the state: most of what the last system took ( launches past convergence are no-ops )
    int ahead = std::max( 1, std::min( prev_its, maxit ) * 7 / 8 / batch );
    for ( ;; ) {
        for ( ; ahead > 0; --ahead, launched += batch ) {
            // ( with live timing on, the first batch is launched one by one, its product timed )
            if ( ( launched == 0 && timing().on ) || ! exec ) iterations( st, launched == 0 );
            else {
                SDOT_HIP( hipGraphLaunch( exec, st ) );
                timing().graph_replays += 1;
            }
        }
        ahead = 1;
        check_launch( "smoothed aggregation: iterations" );
        SDOT_HIP( hipMemcpyAsync( hs, state, sizeof( double ) * S_NB_STATE, hipMemcpyDeviceToHost, st ) );
        SDOT_HIP( hipStreamSynchronize( st ) );
        if ( hs[ S_BAD ] != 0 ) { res.bad = true; return res; }
        if ( hs[ S_DONE ] != 0 || launched >= maxit ) break;
    }
    k_true<<<nblk, TH, 0, st>>>( A0, b, d, part );
    k_true_end<<<1, TH, 0, st>>>( part, nblk, state );
    check_launch( "k_true" );
    SDOT_HIP( hipMemcpyAsync( hs, state, sizeof( double ) * S_NB_STATE, hipMemcpyDeviceToHost, st ) );
    SDOT_HIP( hipStreamSynchronize( st ) );
    res.its = int( hs[ S_IT ] );
    res.err = hs[ S_ERR ];
    res.true_err = hs[ S_TRUE ];
    res.failed = hs[ S_FAILED ] != 0;
    return res;
}

} // namespace

double smoothed_bytes( I64 n, bool wide, double s ) {
    // ( a flat 3D cloud's rows are a 2D cloud's, and may grow within a solve: the smaller aggregates, the longer rows )
    const Sizes sz = sizes_of( n, false );
    const double m = double( n ), nb = double( sz.n[ sz.lb ] );
    double b = 8 * S_NB_STATE + 8.0 * P_NB * SA_BLOCKS + s * m + 8.0 * SA_DENSE * SA_DENSE + s * nb * nb + 4 * 8 * m;
    if ( sz.nl - 1 > sz.lb ) b += double( SA_BOTTOM ) * SA_DENSE_COLS * ( s + 8 );
    for ( int l = 0; l + 1 < sz.nl; ++l ) {
        const double nf = double( sz.n[ l ] ), nc = double( sz.n[ l + 1 ] );
        b += nf * ( 4 + SA_PMAX * ( 4 + s ) ) + nc * ( 4 + SA_TMAX * ( 4 + s ) + 4 + room_of( sz, l, wide ) * ( 4 + s ) + 2 * s );
    }
    for ( int l = 0; l <= sz.lb; ++l ) b += s * double( sz.n[ l ] ) * ( 2 + ( l || s < 8 ? 1 : 0 ) + ( l < sz.lb ? 2 : 0 ) );
    return b;
}

FcgResult smoothed_solve( const Csr &L, const float *valf, const float *diaf, const double *b, double *d, double tol, int maxit, const MgOptions &o,
                          hipStream_t st, int &nb_levels, int prev_its, double drop ) {
    if ( valf ) return solve_with<float>( L, valf, diaf, b, d, tol, maxit, o, st, nb_levels, prev_its, drop, "saf" );
    return solve_with<double>( L, L.val, L.dia, b, d, tol, maxit, o, st, nb_levels, prev_its, drop, "sad" );
}

} // namespace sdot_amd
