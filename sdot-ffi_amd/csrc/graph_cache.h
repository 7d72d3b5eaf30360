// The flexible CG's batches of iterations as HIP graphs, shared by the two multigrid cycles.
#pragma once

#include "common.h"

#include <algorithm>
#include <cstdint>
#include <vector>

namespace sdot_amd {

/// THE ITERATIONS AS A GRAPH: a batch of flexible CG iterations is ~100 launches of small kernels, whose issue costs
/// more than their work on the coarse levels; replayed from a HIP graph it is one launch. A graph is valid as long as
/// every kernel argument is: its key is the full record of them ( the hierarchy's levels, vectors and sizes, the options,
/// the storage type ), written field by field ( no padding bytes ) and compared whole, so that two different argument sets
/// never share a graph. The arena keeps the buffers of a solve of the same size, so Newton's successive systems ( two slots
/// of rows ) replay two graphs per storage type. A few per thread are kept ( least recently used out ).
struct GraphCache {
    struct Entry { std::vector<unsigned char> key; hipGraphExec_t exec; hipGraph_t graph; uint64_t used; };
    std::vector<Entry> entries;
    uint64_t clock = 0;
    ~GraphCache() {
        for ( auto &e : entries ) { (void) hipGraphExecDestroy( e.exec ); (void) hipGraphDestroy( e.graph ); }
    }
    hipGraphExec_t find( const std::vector<unsigned char> &key ) {
        for ( auto &e : entries ) if ( e.key == key ) { e.used = ++clock; return e.exec; }
        return nullptr;
    }
    void put( const std::vector<unsigned char> &key, hipGraph_t g, hipGraphExec_t x ) {
        if ( entries.size() >= 8 ) {
            auto old = std::min_element( entries.begin(), entries.end(), []( const Entry &a, const Entry &b ) { return a.used < b.used; } );
            (void) hipGraphExecDestroy( old->exec );
            (void) hipGraphDestroy( old->graph );
            entries.erase( old );
        }
        entries.push_back( Entry{ key, x, g, ++clock } );
    }
};
inline thread_local GraphCache g_graphs;

/// the stream graphs are captured on ( a capture needs a stream of its own: the legacy default stream cannot be
/// captured ); one per thread, default priority
struct CaptureStream {
    hipStream_t s = nullptr;
    ~CaptureStream() { if ( s ) (void) hipStreamDestroy( s ); }
    hipStream_t get() {
        if ( ! s && hipStreamCreateWithFlags( &s, hipStreamNonBlocking ) != hipSuccess ) { (void) hipGetLastError(); s = nullptr; }
        return s;
    }
};
inline thread_local CaptureStream g_capture;

/// a graph's key: the values of the kernels' arguments appended one by one ( scalars and pointers, never a struct with
/// padding )
struct Key {
    std::vector<unsigned char> b;
    template<class T> void val( const T &v ) {
        const unsigned char *c = reinterpret_cast<const unsigned char *>( &v );
        b.insert( b.end(), c, c + sizeof( T ) );
    }
};

/// what one flexible-CG solve reports
struct FcgResult {
    int its = 0;
    bool bad = false, failed = false;    ///< no hierarchy ( a coarse row past its room ); a breakdown ( `p . q <= 0` )
    double err = 0, true_err = 0;        ///< relative residual by the recurrence, and the true one
};

} // namespace sdot_amd
