"""The smoothed-aggregation V-cycle ( the Newton systems' default preconditioner ) through `sdot_amd_linear_solves_2d`, on the
Laplacians of power diagrams in tree order: against a dense solve where that is quick, against the Jacobi-PCG elsewhere."""
import numpy as np
import pytest

import helpers as H

pytestmark = pytest.mark.gpu


def _system( native, n, d, seed ):
    """the Laplacian of a Voronoi diagram, rows in tree order, as CSR, and a right-hand side of zero sum"""
    import torch
    rng = np.random.default_rng( seed )
    pos = rng.uniform( 0, 1, ( n, d ) )
    if d == 2:
        from sdot import UniformBox
        order = native.build_tree_2d( pos )[ "seed_indices" ].cpu().numpy()
        _, ( fi, fj, fc ) = native.measures_2d( pos, None, [ 0, 0, 1, 1 ], UniformBox( [ 0, 0 ], [ 1, 1 ] ), facets = True )
    else:
        # ( boxes of a few seeds in a serpentine order: near neighbours near, as the tree's ranks )
        k = max( 1, round( ( n / 8 ) ** ( 1 / 3 ) ) )
        c = np.floor( pos * k ).astype( int )
        order = np.lexsort( ( c[ :, 2 ], c[ :, 1 ] // 2, c[ :, 0 ] // 2 ) )
        _, ( fi, fj, fc ) = native.measures_3d( pos, None, [ 0, 0, 0, 1, 1, 1 ], None, facets = True )
    rank = np.empty( n, np.int64 )
    rank[ order ] = np.arange( n )
    i, j, c = rank[ fi.cpu().numpy() ], rank[ fj.cpu().numpy() ], fc.cpu().numpy()
    at = np.lexsort( ( j, i ) )
    i, j, c = i[ at ], j[ at ], c[ at ]
    row = np.concatenate( [ [ 0 ], np.cumsum( np.bincount( i, minlength = n ) ) ] )
    dia = np.bincount( i, weights = c, minlength = n )
    b = rng.normal( size = n )
    return row, j, c, dia, torch.as_tensor( b - b.mean() )


def _cycles_since( native, before ):
    """the systems that the smoothed cycle ran on, and that the K-cycle was tried on, since `before`"""
    now = native.cycle_counts()
    return now[ "smoothed" ] - before[ "smoothed" ], now[ "kcycle" ] - before[ "kcycle" ]


# the sizes: one level over the coarsest ( 65: the smallest the cycle takes ), a bottom of one level and of two, the first
# aggregates of 4 and of 8 ( 8192 / 8193 ), a level between the finest and the bottom, 3D rows
@pytest.mark.parametrize( "n, d", [ ( 65, 2 ), ( 256, 2 ), ( 261, 2 ), ( 2049, 2 ), ( 8192, 2 ), ( 8193, 2 ), ( 40_003, 2 ), ( 150_001, 2 ), ( 700, 3 ), ( 9_001, 3 ) ] )
@pytest.mark.parametrize( "fp32", [ False, True ] )
def test_smoothed_cycle_solves_the_laplacian( native, n, d, fp32 ):
    print( f"case smoothed n={ n } d={ d } fp32={ fp32 }", flush = True )
    row, col, val, dia, b = _system( native, n, d, n + d )
    tol = 1e-10
    x, its = native.linear_solves_2d( row, col, val, dia, b, tol = tol, method = "mg", smoothed = True, fp32 = fp32 )
    x = x[ 0 ].cpu().numpy()
    bh = b.numpy()
    assert 0 < its[ 0 ] < 120
    # the true residual: the recurrence's, at most `tol`, is accepted when the true one is within 10 times it
    Ax = dia * x - np.bincount( np.repeat( np.arange( n ), np.diff( row ) ), weights = val * x[ col ], minlength = n )
    assert np.linalg.norm( bh - Ax ) <= 10 * tol * np.linalg.norm( bh )
    assert x[ 0 ] == 0
    if n <= 2100:
        M = np.diag( dia )
        np.add.at( M, ( np.repeat( np.arange( n ), np.diff( row ) ), col ), -val )
        ref = np.zeros( n )
        ref[ 1: ] = np.linalg.solve( M[ 1:, 1: ], bh[ 1: ] )
        # ( the error is at most the residual over the smallest eigenvalue of the grounded matrix )
        lam = np.linalg.eigvalsh( ( M + M.T )[ 1:, 1: ] / 2 )[ 0 ]
        assert np.linalg.norm( x - ref ) <= 10 * tol * np.linalg.norm( bh ) / lam + 1e-12 * np.linalg.norm( ref )


def test_smoothed_cycle_is_bitwise_reproducible( native ):
    row, col, val, dia, b = _system( native, 30_011, 2, 5 )
    x = [ native.linear_solves_2d( row, col, val, dia, b, tol = 1e-8, method = "mg", smoothed = True, fp32 = True )[ 0 ].cpu().numpy() for _ in range( 3 ) ]
    assert np.array_equal( x[ 0 ], x[ 1 ] ) and np.array_equal( x[ 0 ], x[ 2 ] )


def test_rows_without_room_go_to_the_other_solvers( native ):
    # seeds in a random order: aggregates of far seeds, whose coarse rows outgrow any room
    n = 9_000
    row, col, val, dia, b = _system( native, n, 2, 7 )
    p = np.random.default_rng( 8 ).permutation( n )
    inv = np.argsort( p )
    i = np.repeat( np.arange( n ), np.diff( row ) )
    i2, j2 = inv[ i ], inv[ col ]
    at = np.lexsort( ( j2, i2 ) )
    row2 = np.concatenate( [ [ 0 ], np.cumsum( np.bincount( i2, minlength = n ) ) ] )
    before = native.cycle_counts()
    x, its = native.linear_solves_2d( row2, j2[ at ], val[ at ], dia[ p ], b.numpy()[ p ], tol = 1e-9, method = "mg", smoothed = True, fp32 = True )
    x = x[ 0 ].cpu().numpy()
    assert its[ 0 ] > 0 and _cycles_since( native, before ) == ( 0, 1 )
    r = b.numpy()[ p ] - ( dia[ p ] * x - np.bincount( i2, weights = val * x[ j2 ], minlength = n ) )
    assert np.linalg.norm( r ) <= 1e-8 * np.linalg.norm( b.numpy() )


@pytest.mark.parametrize( "fp32", [ False, True ] )
def test_a_breakdown_leaves_the_solution_untouched( native, fp32 ):
    # a negative definite system breaks down at its first step: every block of the update has to take that decision, none a step
    # ( small beside the 1 that stands in for a coarse diagonal that is not positive, so that the hierarchy is built )
    row, col, val, dia, b = _system( native, 150_001, 2, 3 )
    before = native.cycle_counts()
    x, its = native.linear_solves_2d( row, col, -1e-6 * val, -1e-6 * dia, b, tol = 1e-8, method = "mg", smoothed = True, fp32 = fp32 )
    assert its[ 0 ] == -1 and not x.any().item() and _cycles_since( native, before ) == ( 1, 1 )


@pytest.mark.parametrize( "fp32", [ False, True ] )
def test_a_missed_tolerance_goes_to_the_k_cycle( native, fp32 ):
    # coefficients over twenty orders of magnitude: no cycle brings them to the tolerance, each is tried
    row, col, val, dia, b = _system( native, 9_000, 2, 7 )
    i = np.repeat( np.arange( 9_000 ), np.diff( row ) )
    far = np.exp( 4 * np.random.default_rng( 1 ).normal( size = 9_000 ) )
    val = val * far[ i ] * far[ col ]
    before = native.cycle_counts()
    _, its = native.linear_solves_2d( row, col, val, np.bincount( i, weights = val ), b, tol = 1e-8, method = "mg", smoothed = True, fp32 = fp32 )
    assert its[ 0 ] == -1 and _cycles_since( native, before ) == ( 1, 1 )


@pytest.mark.parametrize( "fp32", [ False, True ] )
def test_rows_past_the_whole_numbers_room_build_no_hierarchy( native, fp32 ):
    # a diagonal of a thousandth of its row: the Galerkin terms pass what their unit was made for, hundreds of times
    row, col, val, dia, b = _system( native, 9_000, 2, 7 )
    before = native.cycle_counts()
    native.linear_solves_2d( row, col, val, 1e-3 * dia, b, tol = 1e-8, method = "mg", smoothed = True, fp32 = fp32 )
    assert _cycles_since( native, before ) == ( 0, 1 )


@pytest.mark.parametrize( "tuning", [ dict(), dict( mg_precision = "double" ), dict( mg_kcycle = 2 ) ] )
def test_handed_over_systems_stay_within_the_byte_model( native, tuning ):
    # a linear tolerance below rounding: every system goes through the smoothed cycle ( or the K-cycle that the options ask for, in FP32 ), the
    # FP64 K-cycle and Jacobi-PCG
    import sdot
    from sdot import memory
    rng = np.random.default_rng( 5 )
    dens = sdot.UniformBox( [ 0, 0 ], [ 1, 1 ] )
    it = sdot.Iterative( tol = 1e-9, on_failure = "ignore", tuning = sdot.Tuning( linear_tol = 1e-18, **tuning ) )
    print( f"case handed over { tuning }", flush = True )
    native.release()
    before = native.cycle_counts()
    sol = sdot.OtProblem( sdot.SumOfDiracs( rng.uniform( 0, 1, ( 9_000, 2 ) ) ), dens ).solve( it )
    smoothed, kcycle = _cycles_since( native, before )
    assert kcycle >= sol.stats[ "nb_iter" ] >= 3 and smoothed == ( 0 if "mg_kcycle" in tuning else kcycle )
    assert native.device_bytes() <= sum( memory.solve_bytes( 9_000, 2, dens, it ).values() )


@pytest.mark.parametrize( "d, n, kind", [ ( 3, 20_000, "uniform" ), ( 3, 60_000, "uniform" ), ( 3, 60_000, "clusters" ), ( 2, 300_000, "clusters" ) ] )
def test_3d_and_clustered_clouds_keep_the_smoothed_cycle( native, d, n, kind ):
    # their coarse rows grow past the room where the prolongations are those of a 2D uniform cloud
    import sdot
    rng = np.random.default_rng( n )
    pos = rng.uniform( 0, 1, ( n, d ) )
    if kind == "clusters":
        centre, size, at = rng.uniform( 0.1, 0.9, ( 20, d ) ), 10 ** rng.uniform( -3, -1, 20 ), rng.integers( 0, 20, n )
        pos = np.clip( centre[ at ] + size[ at, None ] * rng.normal( size = ( n, d ) ), 1e-9, 1 - 1e-9 )
    print( f"case { kind } n={ n } d={ d }", flush = True )
    before = native.cycle_counts()
    sol = sdot.OtProblem( sdot.SumOfDiracs( pos ), sdot.UniformBox( [ 0 ] * d, [ 1 ] * d ) ).solve( sdot.Iterative( tol = 1e-3 / n, max_iter = 2, on_failure = "ignore" ) )
    smoothed, kcycle = _cycles_since( native, before )
    assert smoothed >= 2 and kcycle == 0 and sol.stats[ "lin_nb_iter" ] < 60 * smoothed


def test_rows_that_no_prolongation_fits_go_to_the_other_solvers( native ):
    # a random graph of ~40 neighbours a row: its coarse rows are full whatever is dropped
    import torch
    n = 9_000
    rng = np.random.default_rng( 4 )
    i, j = rng.integers( 0, n, ( 2, 20 * n ) )
    keep = i != j
    pair = np.unique( np.minimum( i, j )[ keep ] * n + np.maximum( i, j )[ keep ] )
    i, j = np.concatenate( [ pair // n, pair % n ] ), np.concatenate( [ pair % n, pair // n ] )
    at = np.lexsort( ( j, i ) )
    i, j = i[ at ], j[ at ]
    row = np.concatenate( [ [ 0 ], np.cumsum( np.bincount( i, minlength = n ) ) ] )
    val, dia = np.ones( len( i ) ), np.bincount( i, minlength = n ).astype( float )
    b = rng.normal( size = n )
    b -= b.mean()
    before = native.cycle_counts()
    x, its = native.linear_solves_2d( row, j, val, dia, torch.as_tensor( b ), tol = 1e-9, method = "mg", smoothed = True, fp32 = True )
    x = x[ 0 ].cpu().numpy()
    assert its[ 0 ] > 0 and _cycles_since( native, before ) == ( 0, 1 )
    assert np.linalg.norm( b - ( dia * x - np.bincount( i, weights = val * x[ j ], minlength = n ) ) ) <= 1e-8 * np.linalg.norm( b )


def test_a_flat_3d_cloud_stays_within_the_byte_model( native ):
    # seeds in one layer: rows of 2D length, whose hierarchy is a 2D cloud's
    import sdot
    from sdot import memory
    rng = np.random.default_rng( 6 )
    n = 20_000
    pos = np.column_stack( [ rng.uniform( 0, 1, ( n, 2 ) ), 0.5 + 1e-7 * rng.uniform( -1, 1, n ) ] )
    dens, it = sdot.UniformBox( [ 0 ] * 3, [ 1 ] * 3 ), sdot.Iterative( tol = 1e-7, max_iter = 3, on_failure = "ignore" )
    native.release()
    sol = sdot.OtProblem( sdot.SumOfDiracs( pos ), dens ).solve( it )
    assert sol.stats[ "lin_nb_iter" ] > 0
    assert native.device_bytes() <= sum( memory.solve_bytes( n, 3, dens, it ).values() )
