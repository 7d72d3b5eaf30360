"""The search of exact duplicates on the device ( the rows' prints in a hash table ) against the host's."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


# a table of two slots, full half and just past it, a large one; one pair far apart, many, all rows equal, a pair of zeros' signs
@pytest.mark.parametrize( "n", [ 1, 2, 3, 1024, 1025, 300_001 ] )
@pytest.mark.parametrize( "d", [ 1, 2, 3 ] )
def test_duplicates_are_the_hosts( native, n, d ):
    import torch
    from sdot.SdotPlanNd import exact_duplicates
    rng = np.random.default_rng( n + d )
    pos = rng.uniform( -1, 1, ( n, d ) )
    zeros = pos.copy()
    zeros[ 0 ], zeros[ -1 ] = 0.0, -0.0
    for P in ( pos, np.concatenate( [ pos, pos[ :1 ] ] ), np.concatenate( [ pos, pos ] ), np.ones( ( n, d ) ), zeros ):
        print( f"case prints { P.shape }", flush = True )
        dup, rep = exact_duplicates( torch.as_tensor( P ).cuda() )
        dup_h, rep_h = exact_duplicates( P )
        assert np.array_equal( dup, dup_h ) and np.array_equal( rep, rep_h )
    assert native.equal_prints( torch.as_tensor( np.ones( ( 2, d ) ) ).cuda() ) and not native.equal_prints( torch.as_tensor( pos ).cuda() )


@pytest.mark.parametrize( "d", [ 2, 3 ] )
def test_the_search_holds_no_memory_of_its_own( native, d ):
    import sdot
    import torch
    from sdot import memory
    from sdot.SdotPlanNd import exact_duplicates
    pos = torch.as_tensor( np.random.default_rng( d ).uniform( 0, 1, ( 300_001, d ) ) ).cuda()
    native.equal_prints( pos[ :2 ] )
    native.release()
    torch.cuda.reset_peak_memory_stats()
    before = torch.cuda.memory_allocated()
    exact_duplicates( pos )
    assert torch.cuda.max_memory_allocated() - before <= 4096     # ( the answer, and torch's rounding of its size )
    # what it took of the library's is the solve's: the whole stays within the solve's model
    dens, it = sdot.UniformBox( [ 0 ] * d, [ 1 ] * d ), sdot.Iterative( tol = 1e-9 )
    sdot.OtProblem( sdot.SumOfDiracs( pos ), dens ).solve( it )
    assert native.device_bytes() <= sum( memory.solve_bytes( 300_001, d, dens, it ).values() )
