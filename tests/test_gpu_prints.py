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
