"""The linear solvers' stop flag, in the kernels' source: a kernel that sets it reads it once for the whole block ( `block_stopped` ). Where each
thread reads it, a wave may see it set by another block of the same launch after the wave before it saw it clear, and leave the block's
barriers to the others, which then sum slots that were never written."""
import pathlib
import re

import pytest

CSRC = pathlib.Path( __file__ ).resolve().parent.parent / "sdot-ffi_amd" / "csrc"


def _kernels( text ):
    """( name, body ) of every kernel of a source"""
    for m in re.finditer( r"__global__[^;{]*?\b(k_\w+)\s*\(", text ):
        at = text.index( "{", text.index( ")", m.end() ) )
        depth, i = 1, at + 1
        while depth:
            depth += { "{": 1, "}": -1 }.get( text[ i ], 0 )
            i += 1
        yield m.group( 1 ), text[ at:i ]


@pytest.mark.parametrize( "source", [ "smoothed.hip", "multigrid.hip", "solver.hip" ] )
def test_a_kernel_that_sets_the_stop_flag_reads_it_by_block( source ):
    setters = []
    for name, body in _kernels( ( CSRC / source ).read_text() ):
        flag = r"(?:state|cg)\[ (?:S|CG)_DONE \]"
        if not re.search( flag + r" = ", body ):
            continue
        setters.append( name )
        own_reads = [ l for l in body.splitlines() if re.search( flag + r" != 0", l ) and "block_stopped" not in l ]
        assert not own_reads, ( name, own_reads )
    assert setters
