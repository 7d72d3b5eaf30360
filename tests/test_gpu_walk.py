"""The first pass's walk by groups of lanes and by one lane a cell ( chosen by the cells' count ): the FP64 cells equal to the oracle's to
the bit on either side of each threshold, the second pass's whole-wave walk included, and majorants that keep a node's slope where the
reference drops it changing no cell."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _unit():
    from sdot import UniformBox
    return UniformBox( [ 0, 0 ], [ 1, 1 ] )


# one seed, a leaf, two leaves ( the shortest way down ), a group's remainder in a wave and a block; both sides of the
# thresholds 2^15 and 2^18 and of the buffer of polygons
@pytest.mark.parametrize( "n", [ 1, 3, 10, 11, 21, 255, 257, 32768, 32769, 262144, 262145 ] )
def test_masses_are_the_oracles_to_the_bit( native, oracle, n ):
    rng = np.random.default_rng( n )
    pos = rng.uniform( 0, 1, ( n, 2 ) )
    w = 0.01 * np.sin( 6 * pos[ :, 0 ] ) * np.cos( 5 * pos[ :, 1 ] ) + 0.2 / n * rng.uniform( -0.5, 0.5, n )
    print( f"case walk n={ n }", flush = True )
    m = native.measures_2d( pos, w, [ 0, 0, 1, 1 ], _unit() ).cpu().numpy()
    assert np.array_equal( m, oracle.measures( pos, w ) )


def test_many_sided_cells_by_whole_waves_and_by_lanes( native, oracle ):
    # a seed amid a ring of `k`: its cell has `k` sides ( 17 to 96: the second pass; beyond: the third ); a few such cells are walked by whole
    # waves, 1200 of them by one lane each
    for k, cells in ( ( 17, 1 ), ( 40, 3 ), ( 65, 2 ), ( 96, 1 ), ( 97, 1 ), ( 18, 1200 ) ):
        g = int( np.ceil( np.sqrt( cells ) ) )
        a = 2 * np.pi * ( np.arange( k ) + 0.37 ) / k
        ring = np.concatenate( [ [ [ 0.0, 0.0 ] ], 0.3 * np.stack( [ np.cos( a ), np.sin( a ) ], 1 ) ] )
        at = np.array( [ ( i % g + 0.5, i // g + 0.5 ) for i in range( cells ) ] )
        pos = ( ( at[ :, None ] + ring[ None ] ) / g ).reshape( -1, 2 ) + 1e-7 * np.random.default_rng( k ).uniform( -1, 1, ( cells * ( k + 1 ), 2 ) )
        print( f"case { cells } cells of { k } sides", flush = True )
        m = native.measures_2d( pos, None, [ 0, 0, 1, 1 ], _unit() ).cpu().numpy()
        assert np.array_equal( m, oracle.measures( pos, None ) )


@pytest.mark.parametrize( "n, scale, shift", [ ( 60_000, 0.02, 0.0 ), ( 60_000, 0.02, 1e3 ), ( 60_000, 0.02, -1e6 ), ( 3_000, 30.0, 5.0 ) ] )
def test_kept_slopes_change_no_cell( native, oracle, n, scale, shift ):
    # weights that vary slowly over the square: most nodes under a hundredth of it have their slope dropped by the reference's rule
    # ( the oracle's ); a large common weight cancels in the majorants
    rng = np.random.default_rng( 3 )
    L = np.sqrt( scale / 0.02 )
    pos = rng.uniform( 0, L, ( n, 2 ) )
    w = scale * np.sin( 2 * np.pi * pos[ :, 0 ] / L ) * np.cos( 2 * np.pi * pos[ :, 1 ] / L ) + 0.2 * L * L / n * rng.uniform( -0.5, 0.5, n ) + shift
    from sdot import UniformBox
    dens = UniformBox( [ 0, 0 ], [ L, L ], target_mass = L * L )
    m = native.measures_2d( pos, w, [ 0, 0, L, L ], dens ).cpu().numpy()
    mo = oracle.measures( pos, w, lo = ( 0, 0 ), hi = ( L, L ) )
    # ( a seed whose plane passes within rounding of a vertex may cut a sliver in one walk and be pruned in the other: the weights' own
    # rounding, an ulp of `shift`, against a facet's length over the seeds' distance )
    tol = 8 * max( np.spacing( abs( shift ) + scale ), np.spacing( L * L ) )
    assert np.abs( m - mo ).max() <= tol
    m32 = native.measures_2d( pos, w, [ 0, 0, L, L ], dens, precision = 1 ).cpu().numpy()
    assert np.abs( m32 - mo ).max() <= 1e-9 * L * L / n + tol


# `along`: weights `slope ( x - y )` plus a constant. On the diagonal the majorants' two terms cancel, and on a lattice every vertex is met by a
# plane that passes it within rounding: a majorant or a test below its own rounding loses slivers
@pytest.mark.parametrize( "at", [ ( 0.0, 0.0 ), ( 1e4, 1e4 ), ( 1e5, 0.0 ), ( 1e5, 1e5 ), ( -1e5, 1e5 ), ( 3.3e4, 7.7e5 ), ( 1e6, 1e6 ) ] )
@pytest.mark.parametrize( "slope, constant", [ ( 0.1, 0.0 ), ( 1e-3, 1e-3 ), ( 0.0, 1e-3 ) ] )
def test_a_lattice_far_from_the_origin_loses_no_sliver( native, at, slope, constant ):
    import torch
    from sdot import UniformBox
    at = np.array( at )
    for k in ( 50, 141 ):
        pos = np.stack( np.meshgrid( *[ ( np.arange( k ) + 0.5 ) / k ] * 2, indexing = "ij" ), -1 ).reshape( -1, 2 ) + at
        w = slope * ( ( pos - at ) @ [ 1.0, -1.0 ] ) + constant
        # ( counting the walk's steps takes the reference's majorants )
        got = native.measures_2d( pos, w, [ *at, *( at + 1 ) ], UniformBox( at, at + 1 ), facets = True )
        ref = native.measures_2d( pos, w, [ *at, *( at + 1 ) ], UniformBox( at, at + 1 ), facets = True, events = True )
        pairs = [ torch.sort( r[ 1 ][ 0 ] * len( pos ) + r[ 1 ][ 1 ] )[ 0 ] for r in ( got, ref ) ]
        assert torch.equal( *pairs ) and torch.equal( got[ 0 ], ref[ 0 ] )
