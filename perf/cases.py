"""The work that a user of this package has it do, as cases that can be timed: transport solves, batches of them, and single
power diagrams with their masses, moments and gradients, in 2D and 3D, over the sizes they are used at.

`listed()` gives the cases, `draw( rng )` one more of the same ranges, `prepare( case, seed )` what a program has in hand before
the call, `run( state )` one pass through the public entry points, `work( case )` what a pass cannot do without, `tolerance( case )`
how far two correct results may differ, `exact( case, seed )` the same outputs in plain torch and 64 bits."""

import math
import os
import sys

import numpy as np
import torch

sys.path.insert( 0, os.path.join( os.path.dirname( os.path.dirname( os.path.abspath( __file__ ) ) ), "sdot-ffi_amd" ) )

import sdot  # noqa: E402


def listed():
    return [
        # the flagship: a million Diracs onto a 1024^2 image, direct ( no width continuation ), from a cold start
        dict( name = "solve_image_1m", op = "solve", dim = 2, n = 1_000_000, density = "image", res = 1024, continuation = "never", tol = 1e-9 ),
        # an ordinary served request, all settings at their defaults
        dict( name = "solve_image_40k", op = "solve", dim = 2, n = 40_013, density = "image", res = 256, continuation = "auto", tol = 1e-9 ),
        # the uniform ( Lebesgue ) target: blue-noise sampling, equal-area partitions
        dict( name = "solve_uniform_500k", op = "solve", dim = 2, n = 500_000, density = "uniform", res = 0, continuation = "auto", tol = 1e-9 ),
        # the smallest solves: an interactive call, where latency counts
        dict( name = "solve_uniform_1k", op = "solve", dim = 2, n = 1_000, density = "uniform", res = 0, continuation = "auto", tol = 1e-10 ),
        # 3D: a few Gaussians, with the widths' continuation
        dict( name = "solve_gauss3d_10k", op = "solve", dim = 3, n = 10_007, density = "gauss", res = 0, continuation = "auto", tol = 1e-9 ),
        # 3D: a voxel image, as served requests have it
        dict( name = "solve_voxel3d_6k", op = "solve", dim = 3, n = 6_000, density = "image", res = 64, continuation = "auto", tol = 1e-9 ),
        # many small problems at once, each with its own image
        dict( name = "batch_12", op = "batch", dim = 2, n = 1_000, n_max = 40_000, count = 12, res = 256, tol = 1e-9 ),
        # one large diagram against an image: the inner call of a program with its own optimiser
        dict( name = "masses_image_1m", op = "masses", dim = 2, n = 1_000_000, density = "image", res = 1024, float = "float64" ),
        # one small diagram: latency
        dict( name = "masses_uniform_2k", op = "masses", dim = 2, n = 2_003, density = "uniform", res = 0, float = "float64" ),
        # masses and their gradients ( weights and positions ): a loss on the masses, forward and backward
        dict( name = "grad_image_60k", op = "grad", dim = 2, n = 60_001, density = "image", res = 256, float = "float64" ),
        # a large 3D diagram: cell volumes
        dict( name = "masses3d_uniform_300k", op = "masses", dim = 3, n = 300_000, density = "uniform", res = 0, float = "float64" ),
        # masses, barycentres and second moments of 3D cells against Gaussians: the cost of a 3D plan
        dict( name = "moments3d_gauss_20k", op = "moments", dim = 3, n = 20_011, density = "gauss", res = 0, float = "float64" ),
    ]


def _log( rng, lo, hi ):
    return int( round( math.exp( rng.uniform( math.log( lo ), math.log( hi ) ) ) ) )


def draw( rng ):
    kind = rng.choice( [ "solve2", "solve2", "solve2", "solve3", "batch", "masses2", "masses2", "grad", "masses3", "moments" ] )
    if kind == "solve2":
        density = rng.choice( [ "image", "image", "uniform" ] )
        n = _log( rng, 500, 700_000 if density == "uniform" else 70_000 )
        c = dict( op = "solve", dim = 2, n = n, density = density, res = rng.choice( [ 128, 200, 256, 333, 512 ] ) if density == "image" else 0,
                  continuation = "auto", tol = 1e-10 if n <= 4_000 else 1e-9 )
    elif kind == "solve3":
        density = rng.choice( [ "gauss", "image", "uniform" ] )
        c = dict( op = "solve", dim = 3, n = _log( rng, 500, 12_000 ), density = density,
                  res = rng.choice( [ 32, 48, 64 ] ) if density == "image" else 0, continuation = "auto", tol = 1e-9 )
    elif kind == "batch":
        c = dict( op = "batch", dim = 2, n = rng.choice( [ 500, 1_000, 2_000 ] ), n_max = _log( rng, 8_000, 40_000 ), count = rng.randint( 4, 12 ),
                  res = rng.choice( [ 128, 200, 256 ] ), tol = 1e-9 )
    elif kind == "masses2":
        density = rng.choice( [ "image", "uniform", "gauss" ] )
        c = dict( op = "masses", dim = 2, n = _log( rng, 500, 1_000_000 ), density = density,
                  res = rng.choice( [ 128, 333, 512, 1024 ] ) if density == "image" else 0, float = rng.choice( [ "float64", "float64", "float32" ] ) )
    elif kind == "grad":
        density = rng.choice( [ "image", "uniform" ] )
        c = dict( op = "grad", dim = 2, n = _log( rng, 500, 400_000 ), density = density, res = rng.choice( [ 128, 256, 500 ] ) if density == "image" else 0,
                  float = "float64" )
    elif kind == "masses3":
        density = rng.choice( [ "uniform", "gauss", "image" ] )
        c = dict( op = "masses", dim = 3, n = _log( rng, 500, 300_000 if density == "uniform" else 60_000 ), density = density,
                  res = rng.choice( [ 32, 64 ] ) if density == "image" else 0, float = "float64" )
    else:
        dim = rng.choice( [ 2, 3 ] )
        density = rng.choice( [ "uniform", "image", "gauss" ] if dim == 2 else [ "uniform", "gauss" ] )
        c = dict( op = "moments", dim = dim, n = _log( rng, 500, 300_000 if dim == 2 else 40_000 ), density = density,
                  res = rng.choice( [ 128, 256 ] ) if density == "image" else 0, float = "float64" )
    return c


# ---- what a program has in hand before the call -------------------------------------------------------------------------------


def _generator( seed ):
    g = torch.Generator( device = "cuda" )
    g.manual_seed( int( seed ) )
    return g


def _uniform( g, shape, lo = 0.0, hi = 1.0 ):
    return lo + ( hi - lo ) * torch.rand( shape, dtype = torch.float64, device = "cuda", generator = g )


def _bumps( g, dim, res ):
    """a `res^dim` image: a floor of 0.1 and isotropic bumps, first index along x ( host array )"""
    k = 8 if dim == 2 and res > 512 else 4
    c = _uniform( g, ( k, dim ), *( ( 0.0, 1.0 ) if dim == 2 else ( 0.2, 0.8 ) ) )
    s = _uniform( g, ( k, ), *( ( 0.05, 0.15 ) if k == 8 else ( 0.08, 0.2 ) ) )
    x = ( torch.arange( res, dtype = torch.float64, device = "cuda" ) + 0.5 ) / res
    v = torch.full( ( res, ) * dim, 0.1, dtype = torch.float64, device = "cuda" )
    for q in range( k ):
        e = None
        for d in range( dim ):
            f = torch.exp( -( x - c[ q, d ] ) ** 2 / ( 2 * s[ q ] ** 2 ) ).reshape( [ -1 if a == d else 1 for a in range( dim ) ] )
            e = f if e is None else e * f
        v += e
    return v.cpu().numpy()


def _density( case, g ):
    """`( target, raw )`: the target distribution and the plain arrays it was made of"""
    dim, res = case[ "dim" ], case[ "res" ]
    lo, hi = [ 0.0 ] * dim, [ 1.0 ] * dim
    if case[ "density" ] == "image":
        v = _bumps( g, dim, res )
        return sdot.Image( v, origin = lo, frame = np.eye( dim ) / res ), v
    if case[ "density" ] == "gauss":
        mu = _uniform( g, ( 4, dim ), 0.2, 0.8 ).cpu().numpy()
        sigma = _uniform( g, ( 4, ), 0.1, 0.2 ).cpu().numpy()
        mass = _uniform( g, ( 4, ), 0.5, 1.5 ).cpu().numpy()
        return sdot.SumOfGaussians( mu, sigma, mass, support_box = ( lo, hi ) ), ( mu, sigma, mass )
    return sdot.UniformBox( lo, hi ), None


def _weights( pos, g ):
    """weights as a solve meets them: a smooth potential that carries cells away from their seeds, and noise of a cell's size"""
    n, dim = pos.shape
    a = 0.02 * _uniform( g, ( 2, ), 0.5, 1.0 )
    w = a[ 0 ] * torch.sin( 2 * math.pi * pos[ :, 0 ] ) * torch.cos( 2 * math.pi * pos[ :, 1 ] ) + a[ 1 ] * torch.cos( 2 * math.pi * pos[ :, -1 ] )
    return w + 0.2 * n ** ( -2 / dim ) * ( _uniform( g, ( n, ) ) - 0.5 )


def _batch_sizes( case ):
    """`count` sizes from `n` to `n_max`, spread over their logarithm, none round"""
    return [ int( s ) + q for q, s in enumerate( np.geomspace( case[ "n" ], case[ "n_max" ], case[ "count" ] ) ) ]


def prepare( case, seed ):
    g = _generator( seed )
    op = case[ "op" ]
    if op == "batch":
        items = []
        for n in _batch_sizes( case ):
            v = _bumps( g, 2, case[ "res" ] )
            items.append( ( _uniform( g, ( int( n ), 2 ) ), sdot.Image( v, origin = [ 0, 0 ], frame = np.eye( 2 ) / case[ "res" ] ) ) )
        return dict( op = op, items = items, settings = sdot.Iterative( tol = case[ "tol" ], on_failure = "ignore" ) )
    pos = _uniform( g, ( case[ "n" ], case[ "dim" ] ) )
    target, raw = _density( case, g )
    state = dict( op = op, pos = pos, target = target, raw = raw )
    if op == "solve":
        state[ "settings" ] = sdot.Iterative( tol = case[ "tol" ], continuation = case[ "continuation" ], on_failure = "ignore" )
        return state
    state[ "w" ] = _weights( pos, g )
    state[ "float" ] = case[ "float" ]
    if op == "grad":
        state[ "cotangent" ] = torch.randn( case[ "n" ], dtype = torch.float64, device = "cuda", generator = g )
        state[ "pos" ].requires_grad_( True )
        state[ "w" ].requires_grad_( True )
    return state


def run( state ):
    op = state[ "op" ]
    if op == "solve":
        plan = sdot.OtProblem( sdot.SumOfDiracs( state[ "pos" ] ), state[ "target" ] ).solve( state[ "settings" ] )
        return dict( weights = plan.weights, masses = plan.cell_masses, barycenters = plan.barycenters, cost = float( plan.cost ) )
    if op == "batch":
        plans = sdot.solve_batch( [ sdot.OtProblem( sdot.SumOfDiracs( p ), t ) for p, t in state[ "items" ] ], state[ "settings" ] )
        return [ dict( weights = p.weights, masses = p.cell_masses, barycenters = p.barycenters, cost = float( p.cost ) ) for p in plans ]
    pd = sdot.PowerDiagram( state[ "pos" ], state[ "w" ], distribution = state[ "target" ], kernel_dtype = state[ "float" ] )
    if op == "masses":
        return pd.measures
    if op == "moments":
        m, f, s = pd.moments
        return dict( masses = m, first = f, second = s )
    m = pd.measures
    gp, gw = torch.autograd.grad( m, ( state[ "pos" ], state[ "w" ] ), state[ "cotangent" ] )
    return dict( masses = m.detach(), grad_positions = gp, grad_weights = gw )


# ---- what a pass cannot do without --------------------------------------------------------------------------------------------


def work( case ):
    """Bytes: the inputs read once, the outputs written once. Flops: a cell's own neighbours alone ( 6 in 2D, 15.5 in 3D ): its
    bisectors, its vertices, their tests and its measures; a solve: at least five diagrams, and for each a Newton system in the
    work of ten products with its matrix."""
    if case[ "op" ] == "batch":
        total = sum( _batch_sizes( case ) )
        one = work( dict( case, op = "solve", n = total, density = "image" ) )
        return { "bytes": one[ "bytes" ] + 8 * ( case[ "count" ] - 1 ) * case[ "res" ] ** 2, "flops": one[ "flops" ] }
    n, dim = case[ "n" ], case[ "dim" ]
    nbr = 6.0 if dim == 2 else 15.5
    cell = 6 * 40 if dim == 2 else 15.5 * 12 + 27 * 60
    points = { "uniform": 0, "image": 40, "gauss": 600 if dim == 2 else 1500 }[ case[ "density" ] ]
    flops = n * ( cell + nbr * points )
    vector = 8 * n
    image = 8 * case[ "res" ] ** dim if case[ "density" ] == "image" else 0
    given = vector * dim + image
    if case[ "op" ] == "solve":
        return { "bytes": given + vector * ( 2 + dim ), "flops": 5 * ( flops + 10 * n * ( 2 * nbr + 8 ) ) }
    given += vector
    if case[ "op" ] == "masses":
        return { "bytes": given + vector, "flops": flops }
    if case[ "op" ] == "moments":
        return { "bytes": given + vector * ( 2 + dim ), "flops": flops * 1.5 }
    return { "bytes": given + vector + vector * ( 2 + dim ), "flops": flops * 2 }


def tolerance( case ):
    """A solve stops anywhere under its absolute tolerance, `n tol` of a cell's mass; few cells are at that limit. Measured between the
    default solves and FP64 cells with another multigrid ( aggregates of 4 ): 1M image ( n tol 1e-3 ) rel 2.6e-6, max 3.5e-4; the
    others, which end further below, 3e-11 and 1e-9. Diagrams: against `exact`, 4e-14 ( masses ) and 4e-13 ( gradients ) at 60k,
    growing with the cells' number; the float kernel re-solves its vertices in double and differs where floats decide a degenerate cut."""
    n = case[ "n_max" ] if case[ "op" ] == "batch" else case[ "n" ]
    if case[ "op" ] in ( "solve", "batch" ):
        return { "rel": max( 1e-9, 1e-2 * n * case[ "tol" ] ), "max": max( 4e-8, 2 * n * case[ "tol" ] ) }
    if case[ "float" ] == "float32":
        return { "rel": 1e-9 }
    return { "rel": 1e-11 if case[ "dim" ] == 3 else 2e-12 + 3e-17 * n }


# ---- the same outputs in plain torch, 64 bits ---------------------------------------------------------------------------------
#
# A cell is the box cut by the bisectors of its nearest seeds, and again by those of the seeds that still own one of its vertices,
# until there is none; all cells are cut together as padded arrays, in coordinates about their seeds. In 3D each face is cut out of
# its plane the same way, and a cell is the sum of the signed tetrahedra from its seed to its faces' triangles.


def _nearest( pos, k ):
    """the `k` nearest seeds of each ( itself left out ), nearest first"""
    n = pos.shape[ 0 ]
    k = min( k, n - 1 )
    step = max( 1, 50_000_000 // n )

    def squares( p ):                                    # ( not `torch.cdist`: its results are wrong past ~4096 rows on this card )
        return sum( ( p[ :, None, d ] - pos[ None, :, d ] ) ** 2 for d in range( pos.shape[ 1 ] ) )

    return torch.cat( [ squares( pos[ a:a + step ] ).topk( k + 1, largest = False ).indices[ :, 1: ] for a in range( 0, n, step ) ] )


def _intruders( pos, w, cell, x ):
    """the seeds that own a point `x` of a cell before the cell's own does: `( cell, seed )`, each pair once"""
    step = max( 1, 50_000_000 // len( pos ) )
    found = []
    for a in range( 0, len( cell ), step ):
        c, z = cell[ a:a + step ], x[ a:a + step ]
        power, seed = ( sum( ( z[ :, None, d ] - pos[ None, :, d ] ) ** 2 for d in range( pos.shape[ 1 ] ) ) - w[ None, : ] ).min( 1 )
        out = power < ( ( z - pos[ c ] ) ** 2 ).sum( 1 ) - w[ c ] - 1e-13
        found.append( torch.unique( c[ out ] * len( pos ) + seed[ out ] ) )
    both = torch.unique( torch.cat( found ) )
    return both // len( pos ), both % len( pos )


def _more( near, cell, seed ):
    """`near` with the seeds `seed` added to the rows `cell` ( increasing ), the other rows filled with -1"""
    at = torch.arange( len( cell ), device = cell.device ) - torch.searchsorted( cell, cell )
    extra = torch.full( ( len( near ), int( at.max() ) + 1 ), -1, device = near.device )
    extra[ cell, at ] = seed
    return torch.cat( [ near, extra ], 1 )


def _cut( P, nb, ids, dirs, off, cut_id ):
    """convex polygons `P [ m, V, 2 ]` ( the first `nb` vertices of each; `ids` names the cut of the edge leaving a vertex ) cut by
    `dirs . x <= off`, the new edge named `cut_id`"""
    m, V = ids.shape
    slot = torch.arange( V, device = P.device )
    real = slot < nb[ :, None ]
    nxt = torch.where( slot + 1 < nb[ :, None ], slot + 1, 0 ).expand( m, V )
    s = ( P * dirs[ :, None, : ] ).sum( -1 ) - off[ :, None ]
    s1 = torch.gather( s, 1, nxt )
    P1 = torch.gather( P, 1, nxt[ :, :, None ].expand( m, V, 2 ) )
    inside, inside1 = ( s <= 0 ) & real, s1 <= 0
    cross = real & ( inside != inside1 )
    t = torch.where( cross, s / torch.where( cross, s - s1, 1.0 ), 0.0 )
    X = P + t[ :, :, None ] * ( P1 - P )
    both = torch.stack( [ P, X ], 2 ).reshape( m, 2 * V, 2 )
    keep = torch.stack( [ inside, cross ], 2 ).reshape( m, 2 * V )
    # ( leaving the half-plane starts the new edge, coming back carries on with the old one )
    name = torch.stack( [ ids, torch.where( inside, cut_id[ :, None ], ids ) ], 2 ).reshape( m, 2 * V )
    order = torch.argsort( ( ~keep ).to( torch.int8 ), dim = 1, stable = True )[ :, :V ]
    nb = keep.sum( 1 )
    if int( nb.max() ) > V:
        raise RuntimeError( "a polygon with more vertices than there is room for" )
    return torch.gather( both, 1, order[ :, :, None ].expand( m, V, 2 ) ), nb, torch.gather( name, 1, order )


def _cells( pos, w, near, room = 28 ):
    """the 2D cells about their seeds: `( P [ n, room, 2 ], nb, ids )`, the box's sides named -1 .. -4"""
    n = pos.shape[ 0 ]
    box = torch.tensor( [ [ 0.0, 0.0 ], [ 1.0, 0.0 ], [ 1.0, 1.0 ], [ 0.0, 1.0 ] ], dtype = torch.float64, device = pos.device )
    P = torch.cat( [ box[ None ] - pos[ :, None ], torch.zeros( n, room - 4, 2, dtype = torch.float64, device = pos.device ) ], 1 )
    nb = torch.full( ( n, ), 4, device = pos.device )
    ids = torch.arange( -1, -room - 1, -1, device = pos.device ).expand( n, room )
    for q in range( near.shape[ 1 ] ):
        j = near[ :, q ]
        d = pos[ j ] - pos
        P, nb, ids = _cut( P, nb, ids, d, torch.where( j < 0, 1e3, ( ( d * d ).sum( 1 ) + w - w[ j ] ) / 2 ), j )
    return P, nb, ids


def _all_cells( pos, w, near = 40 ):
    near = _nearest( pos.detach(), near )
    while True:
        with torch.no_grad():
            cell, a, _, _ = _edges( pos, *_cells( pos, w, near ) )
            cell, seed = _intruders( pos, w, cell, a )
        if not len( cell ):
            return _cells( pos, w, near )
        near = _more( near, cell, seed )


def _edges( pos, P, nb, ids ):
    """the edges of all cells: `( cell, a, b, cut )`, absolute coordinates"""
    m, V = ids.shape
    slot = torch.arange( V, device = P.device )
    nxt = torch.where( slot + 1 < nb[ :, None ], slot + 1, 0 ).expand( m, V )
    P1 = torch.gather( P, 1, nxt[ :, :, None ].expand( m, V, 2 ) )
    cell, k = torch.nonzero( slot < nb[ :, None ], as_tuple = True )
    return cell, pos[ cell ] + P[ cell, k ], pos[ cell ] + P1[ cell, k ], ids[ cell, k ]


_GL = { k: tuple( torch.tensor( ( v + 1 ) / 2 if i == 0 else v / 2 ) for i, v in enumerate( np.polynomial.legendre.leggauss( k ) ) ) for k in ( 3, 8, 16 ) }


class _Field:
    """the density in 2D: along a row, `int rho`, `int s rho`, `int s^2 rho` up to `x` from the column of `x_ref` ( powers 0, 1, 2 ), and
    the points an edge is integrated at"""

    def __init__( self, case, raw, device ):
        self.kind = case[ "density" ]
        if self.kind == "image":
            self.res = case[ "res" ]
            self.v = torch.as_tensor( raw, dtype = torch.float64, device = device )
            self.v = self.v * ( self.res ** 2 / self.v.sum() )
            x = torch.arange( self.res + 1, dtype = torch.float64, device = device ) / self.res
            self.pre = []
            for p in range( 3 ):
                c = torch.zeros( self.res + 1, self.res, dtype = torch.float64, device = device )
                c[ 1: ] = torch.cumsum( self.v * ( ( x[ 1: ] ** ( p + 1 ) - x[ :-1 ] ** ( p + 1 ) ) / ( p + 1 ) )[ :, None ], 0 )
                self.pre.append( c )
        elif self.kind == "gauss":
            mu, sigma, mass = ( torch.as_tensor( a, dtype = torch.float64, device = device ) for a in raw )
            self.gauss = ( mu, sigma, mass / mass.sum() )

    def at( self, x, y ):
        if self.kind == "uniform":
            return torch.ones_like( x )
        if self.kind == "image":
            i, j = ( ( c.detach() * self.res ).floor().long().clamp( 0, self.res - 1 ) for c in ( x, y ) )
            return self.v[ i, j ]
        mu, sigma, mass = self.gauss
        return sum( mass[ q ] / ( 2 * math.pi * sigma[ q ] ** 2 ) * torch.exp( -( ( x - mu[ q, 0 ] ) ** 2 + ( y - mu[ q, 1 ] ) ** 2 ) / ( 2 * sigma[ q ] ** 2 ) )
                    for q in range( len( mass ) ) )

    def row( self, p, x, y, x_ref ):
        if self.kind == "uniform":
            return ( x ** ( p + 1 ) - x_ref ** ( p + 1 ) ) / ( p + 1 )
        if self.kind == "image":
            i, j, r = ( ( c.detach() * self.res ).floor().long().clamp( 0, self.res - 1 ) for c in ( x, y, x_ref ) )
            return self.pre[ p ][ i, j ] - self.pre[ p ][ r, j ] + self.v[ i, j ] * ( x ** ( p + 1 ) - ( i.double() / self.res ) ** ( p + 1 ) ) / ( p + 1 )
        mu, sigma, mass = self.gauss
        total = 0
        for q in range( len( mass ) ):
            s, m = sigma[ q ], mu[ q, 0 ]

            def prim( z ):
                e = math.sqrt( math.pi / 2 ) * s * torch.erf( ( z - m ) / ( math.sqrt( 2 ) * s ) )
                g = s * s * torch.exp( -( z - m ) ** 2 / ( 2 * s * s ) )
                return e if p == 0 else m * e - g if p == 1 else ( m * m + s * s ) * e - ( z + m ) * g
            total = total + mass[ q ] / ( 2 * math.pi * s * s ) * torch.exp( -( y - mu[ q, 1 ] ) ** 2 / ( 2 * s * s ) ) * ( prim( x ) - prim( x_ref ) )
        return total

    def points( self, a, b ):
        """`( t, weight )` `[ E, Q ]` along each edge: Gauss points on each of its pieces in one pixel, or on the whole"""
        x, g = ( v.to( a.device ) for v in _GL[ 16 if self.kind == "gauss" else 3 ] )
        if self.kind != "image":
            return x.expand( len( a ), -1 ), g.expand( len( a ), -1 )
        ts = [ torch.zeros( len( a ), 1, dtype = torch.float64, device = a.device ), torch.ones( len( a ), 1, dtype = torch.float64, device = a.device ) ]
        for d in range( 2 ):
            u, e = a[ :, d ] * self.res, ( b - a )[ :, d ] * self.res
            lo, hi = torch.minimum( u, u + e ).detach(), torch.maximum( u, u + e ).detach()
            first = lo.floor() + 1
            count = int( ( hi.ceil() - first ).clamp( min = 0 ).max() )
            line = first[ :, None ] + torch.arange( count, device = a.device )
            ok = line < hi[ :, None ]
            ts.append( torch.where( ok, ( line - u[ :, None ] ) / torch.where( ok, e[ :, None ], 1.0 ), 1.0 ) )
        t = torch.sort( torch.cat( ts, 1 ), 1 ).values
        d = t[ :, 1: ] - t[ :, :-1 ]
        return ( t[ :, :-1, None ] + d[ :, :, None ] * x ).flatten( 1 ), ( d[ :, :, None ] * g ).flatten( 1 )


def _measures( n, pos, field, edges, moments = False ):
    """masses, or `( masses, int x rho, int |x|^2 rho )`, by Green's theorem along the edges"""
    cell, a, b, _ = edges
    parts = []
    for s in range( 0, len( cell ), 400_000 ):
        c, u, v = cell[ s:s + 400_000 ], a[ s:s + 400_000 ], b[ s:s + 400_000 ]
        t, g = field.points( u, v )
        x, y = ( u[ :, None, d ] + t * ( v - u )[ :, None, d ] for d in range( 2 ) )
        ref = pos.detach()[ c, 0 ][ :, None ].expand_as( x )
        g = g * ( v - u )[ :, None, 1 ]
        f = [ field.row( 0, x, y, ref ) ]
        if moments:
            f += [ field.row( 1, x, y, ref ), y * f[ 0 ], field.row( 2, x, y, ref ) + y * y * f[ 0 ] ]
        parts.append( torch.stack( [ ( g * q ).sum( 1 ) for q in f ], 1 ) )
    out = torch.zeros( n, 4 if moments else 1, dtype = torch.float64, device = pos.device ).index_add( 0, cell, torch.cat( parts ) )
    return ( out[ :, 0 ], out[ :, 1:3 ], out[ :, 3 ] ) if moments else out[ :, 0 ]


def _solve( case, state, field ):
    """the plan by a damped Newton with dense systems, every cell cut by every other seed"""
    pos = state[ "pos" ]
    n = len( pos )
    near = _nearest( pos, n - 1 )
    nu = torch.full( ( n, ), 1.0 / n, dtype = torch.float64, device = pos.device )

    def diagram( w ):
        e = _edges( pos, *_cells( pos, w, near ) )
        return e, _measures( n, pos, field, e )

    w = torch.zeros( n, dtype = torch.float64, device = pos.device )
    e, m = diagram( w )
    floor = 0.5 * min( float( m.min() ), 1 / n )
    for _ in range( 60 ):
        r = nu * ( m.sum() / nu.sum() ) - m
        if float( r.abs().max() ) < 1e-15:
            break
        cell, a, b, cut = ( q[ e[ 3 ] >= 0 ] for q in e )
        t, g = field.points( a, b )
        x, y = ( a[ :, None, d ] + t * ( b - a )[ :, None, d ] for d in range( 2 ) )
        c = ( g * field.at( x, y ) ).sum( 1 ) * ( b - a ).norm( dim = 1 ) / ( 2 * ( pos[ cut ] - pos[ cell ] ).norm( dim = 1 ) )
        L = torch.zeros( n, n, dtype = torch.float64, device = pos.device ).index_put_( ( cell, cut ), -c, accumulate = True )
        L = ( L + L.T ) / 2
        L = L - torch.diag( L.sum( 1 ) )
        step = torch.zeros_like( w )
        step[ 1: ] = torch.linalg.solve( L[ 1:, 1: ], r[ 1: ] )
        size, t = float( r.norm() ), 1.0
        while t > 1e-9:
            e2, m2 = diagram( w + t * step )
            r2 = float( ( nu * ( m2.sum() / nu.sum() ) - m2 ).norm() )
            if float( m2.min() ) >= floor and r2 < size:
                break
            t /= 2
        if r2 >= size:
            break
        w, e, m = w + t * step, e2, m2
    m, first, second = _measures( n, pos, field, e, moments = True )
    cost = second - 2 * ( pos * first ).sum( 1 ) + ( pos * pos ).sum( 1 ) * m
    return dict( weights = w - w[ 0 ], masses = m, barycenters = first / m[ :, None ], cost = float( cost.sum() ) )


def _faces3( pos, w, cells, near, room ):
    """the faces of the 3D cells `cells` about their seeds: `( X [ F, room, 3 ], nb, cell, height )`, the cell's place in `cells`, the
    signed distance from its seed to the face"""
    dev = pos.device
    axes = torch.cat( [ torch.eye( 3, dtype = torch.float64, device = dev ), -torch.eye( 3, dtype = torch.float64, device = dev ) ] )
    p = pos[ cells ]
    to = pos[ near ] - p[ :, None ]
    d = torch.cat( [ axes[ None ].expand( len( p ), 6, 3 ), to ], 1 )
    off = torch.cat( [ 1 - p, p, torch.where( near < 0, 1e3, ( to ** 2 ).sum( -1 ) / 2 + ( w[ cells, None ] - w[ near ] ) / 2 ) ], 1 )
    # the plane of each cut: its point nearest the seed, two unit directions in it
    size = d.norm( dim = -1 )
    unit = d / size[ :, :, None ]
    height = off / size
    centre = unit * height[ :, :, None ]
    u = torch.linalg.cross( unit, torch.nn.functional.one_hot( unit.abs().argmin( -1 ), 3 ).to( unit.dtype ) )
    u = u / u.norm( dim = -1, keepdim = True )
    v = torch.linalg.cross( unit, u )
    m, K = off.shape
    P = torch.zeros( m * K, room, 2, dtype = torch.float64, device = dev )
    P[ :, :4 ] = torch.tensor( [ [ -3.0, -3.0 ], [ 3.0, -3.0 ], [ 3.0, 3.0 ], [ -3.0, 3.0 ] ], dtype = torch.float64, device = dev )
    nb = torch.full( ( m * K, ), 4, device = dev )
    face = torch.arange( m * K, device = dev )
    centre, u, v = ( z.reshape( -1, 3 ) for z in ( centre, u, v ) )
    for q in range( K ):
        c = face // K
        dq = d[ c, q ]
        dirs = torch.stack( [ ( u[ face ] * dq ).sum( 1 ), ( v[ face ] * dq ).sum( 1 ) ], 1 )
        # ( a face is not cut by its own plane )
        o = torch.where( face % K == q, 1e3, off[ c, q ] - ( centre[ face ] * dq ).sum( 1 ) )
        P, nb, _ = _cut( P, nb, torch.zeros( len( face ), room, dtype = torch.long, device = dev ), torch.where( ( face % K == q )[ :, None ], 0.0, dirs ), o, face )
        left = nb >= 3
        P, nb, face = P[ left ], nb[ left ], face[ left ]
    X = centre[ face ][ :, None ] + P[ :, :, :1 ] * u[ face ][ :, None ] + P[ :, :, 1: ] * v[ face ][ :, None ]
    return X, nb, face // K, height.reshape( -1 )[ face ]


def _moments3( case, raw, pos, w, near = 100, room = 20 ):
    """`( masses, int x rho, int |x|^2 rho )` of 3D cells against a constant or a sum of Gaussians"""
    n, dev = len( pos ), pos.device
    nearest = _nearest( pos, near )
    out = torch.zeros( n, 5, dtype = torch.float64, device = dev )
    x1, g1 = ( v.to( dev ) for v in _GL[ 8 ] )
    step = max( 1, 400_000 // nearest.shape[ 1 ] )
    for s in range( 0, n, step ):
        cells = torch.arange( s, min( s + step, n ), device = dev )
        k = nearest[ s:s + step ]
        while True:
            X, nb, c, height = _faces3( pos, w, cells, k, room )
            f, t = torch.nonzero( torch.arange( room, device = dev ) < nb[ :, None ], as_tuple = True )
            cell, seed = _intruders( pos, w, cells[ c[ f ] ], pos[ cells[ c[ f ] ] ] + X[ f, t ] )
            if not len( cell ):
                break
            k = _more( k, cell - s, seed )
        f, t = torch.nonzero( torch.arange( 1, room - 1, device = dev ) + 1 < nb[ :, None ], as_tuple = True )
        a, b, e = X[ f, 0 ], X[ f, t + 1 ], X[ f, t + 2 ]
        cell = cells[ c[ f ] ]
        o = pos[ cell ]
        vol = torch.linalg.cross( b - a, e - a ).norm( dim = 1 ) / 6 * height[ f ]     # ( signed by the seed's side of the face )
        if case[ "density" ] == "uniform":
            total, squares = a + b + e, ( a * a + b * b + e * e + a * b + b * e + e * a ).sum( 1 )
            first = vol[ :, None ] * ( o + total / 4 )
            second = vol * ( squares / 10 + ( o * total ).sum( 1 ) / 2 + ( o * o ).sum( 1 ) )
            part = torch.cat( [ vol[ :, None ], first, second[ :, None ] ], 1 )
        else:
            mu, sigma, mass = ( torch.as_tensor( q, dtype = torch.float64, device = dev ) for q in raw )
            mass = mass / mass.sum()
            part = torch.zeros( len( cell ), 5, dtype = torch.float64, device = dev )
            for i in range( 512 ):                       # ( the cube's point ( r, h, l ) on the tetrahedron, its volume's factor 6 r^2 h )
                q = ( i // 64, i // 8 % 8, i % 8 )
                r, h, l = x1[ q[ 0 ] ], x1[ q[ 1 ] ], x1[ q[ 2 ] ]
                z = o + r * ( a + h * ( ( b - a ) + l * ( e - b ) ) )
                rho = sum( mass[ j ] / ( 2 * math.pi * sigma[ j ] ** 2 ) ** 1.5 * torch.exp( -( ( z - mu[ j ] ) ** 2 ).sum( 1 ) / ( 2 * sigma[ j ] ** 2 ) )
                           for j in range( len( mass ) ) )
                wt = 6 * r * r * h * g1[ q[ 0 ] ] * g1[ q[ 1 ] ] * g1[ q[ 2 ] ] * vol * rho
                part += wt[ :, None ] * torch.cat( [ torch.ones_like( z[ :, :1 ] ), z, ( z * z ).sum( 1, keepdim = True ) ], 1 )
        out.index_add_( 0, cell, part )
    return out[ :, 0 ], out[ :, 1:4 ], out[ :, 4 ]


def exact( case, seed ):
    op, n, dim = case[ "op" ], case[ "n" ], case[ "dim" ]
    # ( past these sizes it takes over 20 seconds, as do the 3D solves and the batches; a voxel image would be cut voxel by voxel )
    if op == "batch" or ( dim == 3 and ( op == "solve" or n > 21_000 or case[ "density" ] == "image" ) ) or n > ( 1_200 if op == "solve" else 120_000 ):
        return None
    state = prepare( case, seed )
    pos = state[ "pos" ]
    if dim == 3:
        m, f, s = _moments3( case, state[ "raw" ], pos, state[ "w" ] )
        return m if op == "masses" else dict( masses = m, first = f, second = s )
    field = _Field( case, state[ "raw" ], pos.device )
    if op == "solve":
        return _solve( case, state, field )
    w = state[ "w" ]
    edges = _edges( pos, *_all_cells( pos, w ) )
    if op == "moments":
        m, f, s = _measures( n, pos, field, edges, moments = True )
        return dict( masses = m, first = f, second = s )
    m = _measures( n, pos, field, edges )
    if op == "masses":
        return m
    gp, gw = torch.autograd.grad( m, ( pos, w ), state[ "cotangent" ] )
    return dict( masses = m.detach(), grad_positions = gp, grad_weights = gw )
