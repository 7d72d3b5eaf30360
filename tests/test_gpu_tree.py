"""The device's tree builds ( one workgroup's, for at most 4096 seeds; the launches' beyond ) against the oracle's tree."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _by_median( pos, leaf = 10 ):
    """the tree by its definition: a node of more than `leaf` seeds is cut along its box's ( first ) longest side into the first half of its
    seeds and the rest, by ( coordinate, user index ); the leaves by user index"""
    n = len( pos )
    depth = 1
    while leaf << ( depth - 1 ) < n: depth += 1
    order, beg, end = np.zeros( n, int ), [], []
    def node( ids, at, h ):
        beg.append( at )
        end.append( at + len( ids ) )
        if h == 1:
            order[ at:at + len( ids ) ] = np.sort( ids )
            return
        cut = len( ids )
        if cut > leaf:
            side = np.ptp( pos[ ids ], axis = 0 )
            d = int( side[ 1 ] > side[ 0 ] )
            if side[ d ] > 0:
                ids = ids[ np.lexsort( ( ids, pos[ ids, d ] ) ) ]
                cut //= 2
        node( ids[ :cut ], at, h - 1 )
        node( ids[ cut: ], at + cut, h - 1 )
    node( np.arange( n ), 0, depth )
    return order, np.array( beg ), np.array( end )


# one seed, a leaf, two leaves, one seed past a power of two and past a scan's block, and both sides of the one workgroup's 4096;
# `grid`: coordinates with many ties ( where the oracle cuts by its own order among the tied ), `line`: an axis without any extent,
# `same`: all seeds in one place ( no node is cut )
@pytest.mark.parametrize( "n", [ 1, 2, 10, 11, 129, 1025, 4095, 4096, 4097, 8191, 8192, 8193, 70_000 ] )
@pytest.mark.parametrize( "kind", [ "uniform", "grid", "line", "same" ] )
def test_the_tree_is_the_one_defined( native, oracle, n, kind ):
    rng = np.random.default_rng( n )
    pos = rng.uniform( -1, 1, ( n, 2 ) )
    if kind == "grid": pos = np.round( 8 * pos ) / 8 + 0.0
    if kind == "line": pos[ :, 1 ] = -0.25
    if kind == "same": pos[ : ] = [ 0.5, 0.25 ]
    print( f"case tree n={ n } { kind }", flush = True )
    t = { k: v.cpu().numpy() for k, v in native.build_tree_2d( pos ).items() }
    order, beg, end = _by_median( pos )
    assert np.array_equal( t[ "seed_indices" ], order )
    assert np.array_equal( t[ "rank_of" ][ order ], np.arange( n ) )
    assert np.array_equal( t[ "node_begin" ], beg ) and np.array_equal( t[ "node_end" ], end )
    for b, e, box in zip( beg, end, t[ "node_box" ] ):
        if e > b: assert np.array_equal( box, [ pos[ order[ b:e ] ].min( 0 ), pos[ order[ b:e ] ].max( 0 ) ] )
    if kind == "uniform":
        assert np.array_equal( t[ "seed_indices" ], oracle.build_tree( pos )[ "order" ] )


@pytest.mark.parametrize( "leaf", [ 1, 3, 64 ] )
def test_other_leaves( native, oracle, leaf ):
    pos = np.random.default_rng( leaf ).uniform( 0, 1, ( 2000, 2 ) )
    t = { k: v.cpu().numpy() for k, v in native.build_tree_2d( pos, leaf = leaf ).items() }
    to = oracle.build_tree( pos, leaf = leaf )
    assert np.array_equal( t[ "seed_indices" ], to[ "order" ] ) and np.array_equal( t[ "node_end" ], to[ "end" ] )


# the 3D tree through the counts of the walk over it ( the nodes tried and pruned, the cuts: another tree has others )
@pytest.mark.parametrize( "n", [ 1, 10, 11, 1025, 4096, 4097, 8192, 8193 ] )
def test_the_3d_walk_counts_the_oracles( native, oracle, n ):
    from sdot import UniformBox
    pos = np.random.default_rng( n ).uniform( 0, 1, ( n, 3 ) )
    print( f"case 3D tree n={ n }", flush = True )
    m, ev = native.measures_3d( pos, None, [ 0, 0, 0, 1, 1, 1 ], UniformBox( [ 0 ] * 3, [ 1 ] * 3 ), events = True )
    mo, evo = oracle.measures_3d( pos, events = True )
    assert np.allclose( m.cpu().numpy(), mo, rtol = 1e-10, atol = 1e-16 )
    for k in ( "side_tests", "node_visits", "cuts" ):     # ( the few cells of a second pass are walked, and counted, twice )
        assert abs( ev[ k ] - evo[ k ] ) <= 0.01 * evo[ k ], k


# the 3D tree, seed for seed: each cell's facets come in the order of the cuts that made them, which is the order its walk met the leaves and
# their seeds in ( another tree has another )
@pytest.mark.parametrize( "n", [ 1, 10, 11, 1025, 4096, 4097, 8192, 8193, 30_000 ] )
def test_the_3d_cells_are_cut_in_the_oracles_order( native, oracle, n ):
    from sdot import UniformBox
    rng = np.random.default_rng( n )
    pos = rng.uniform( 0, 1, ( n, 3 ) ) * [ 1.0, 0.5, 1.0 ]
    w = 0.1 * n ** ( -2 / 3 ) * rng.uniform( -1, 1, n )
    print( f"case 3D tree n={ n }", flush = True )
    m, ( fi, fj, _ ) = native.measures_3d( pos, w, [ 0, 0, 0, 1, 1, 1 ], UniformBox( [ 0 ] * 3, [ 1 ] * 3 ), facets = True )
    mo, ( oi, oj, _ ) = oracle.measures_3d( pos, w, facets = True )
    assert np.allclose( m.cpu().numpy(), mo, rtol = 1e-10, atol = 1e-16 )
    assert np.array_equal( fi.cpu().numpy(), oi ) and np.array_equal( fj.cpu().numpy(), oj )
