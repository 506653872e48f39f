// svlg_tiles.hpp -- host description of the node tiles of the fused explicit kernel.
#pragma once

#include <cstdint>
#include <vector>

namespace svlg {

struct HostTiles {
    int ntiles = 0, ncolors = 0;
    int max_stage = 0, max_own = 0, max_elem = 0;
    std::vector<int32_t> perm;       // device node -> original node
    std::vector<int32_t> inv;        // original node -> device node
    std::vector<int32_t> own_ptr;    // [ntiles+1] device node range owned by tile
    std::vector<int32_t> nplain;     // [ntiles] plain nodes at the start of the range
    std::vector<int32_t> halo_ptr;   // [ntiles+1]
    std::vector<int32_t> halo_node;  // device node of each halo slot
    std::vector<int32_t> elem_ptr;   // [ntiles+1]
    std::vector<int32_t> elem_id;    // original element index (tag order)
    std::vector<uint16_t> elem_lconn;// [elems*nen] staged slot of each corner
    std::vector<int32_t> color_ptr;  // [ntiles*(ncolors+1)] offsets inside the tile's elements
};

// What the default tile size depends on beside the counts.
struct TileTraits {
    bool bricks = false;           // the elements are parallelepipeds
    bool j2 = false;               // a J2 element
    bool lumped = true;            // lumped mass
    bool implicit = false;         // only implicit integrators take it: consistent mass or stiffness-proportional damping
    bool corner_unique = true;     // no node is the same corner of two elements (else: colour-phase kernel)
};

// Node-tile size when the caller names none. 3D: 160 nodes fill the chip and recompute 0.7
// elements per element; up to 12,000 nodes smaller tiles spread the mesh over the 256 CUs and leave
// room for the second ring of the multi-step kernel (8,125 nodes: 36 to 48 nodes 3.6 us per
// step, 64 nodes 3.8, 160 nodes 5.7). 2D: one tile while a workgroup holds the mesh, then tiles that
// give about a workgroup per CU (5,151 nodes: 64 nodes 1.37 us, 128 nodes 1.43; 20,301 nodes: 128 nodes
// 1.42, 64 nodes 1.64), 400 nodes where the rings of the multi-step kernel need the room
// (80,601 nodes: 400 nodes 2.2 us, 128 nodes 3.2), and 192 nodes above a million, where single steps
// of small workgroups hide their latencies best (1.77M nodes: 192 nodes 29.4 us; 448 nodes 28 us when
// no tile touches more than 512 elements, 52 us when one does).
// Gauss-point hexahedra (256 registers, one wave per SIMD) take 96 nodes, whose elements are three
// waves: 16,128 nodes 9.5 us per step against 12.9 with 160 and 12.2 with 64 nodes, 62,279 nodes 18.0
// against 23.3 and 24.1.
// Gauss-point quadrilaterals leave the multi-step kernel at a chip full of tiles; single steps take 192 nodes
// from there on (208,921 nodes: 192 nodes 11.7 us per step, 400 nodes 13.2; 0.55M: 24.3 and 25.6).
// The colour-phase kernel pays for every colour of a workgroup's elements and holds 512 threads: its
// quads stay at 400 nodes or more (208,921 nodes: 400 nodes 8.5 us per step, 448 nodes 9.3; distorted
// 15.5 and 12.3; 1.4M nodes, 448 nodes 38 and 192 nodes 66, distorted 58 and 86), its bricks at 160 above
// 9,000 (11,648 nodes 15.8 against 17.0 with 40); general hexahedra, of which a CU holds one
// workgroup, take the smallest of 40, 96 and 160 whose tiles are one round of the CUs (8,625 nodes 18.0 /
// 18.5 / 22.0 us; 10,125 nodes 33.4 / 18.5 / 22.0; 26,381 nodes 49.7 / 34.5 / 22.0; 0.52M nodes 299 with 96, 222
// with 160).
// Models with J2 elements keep one size: the tiles set the order of the solver's dot products, and
// a yielding point's elastic or plastic branch can follow their last bits.
// Models that only the implicit integrators take: quadrilateral bricks above 36,000 nodes 448, the fewest tiles
// whose elements fit a workgroup (microseconds per iteration, 400 against 448 nodes: 60,501 nodes
// Jacobi 12.7, 11.7; 0.56M 42.8, 40.7, learned 195, 170; 1.3M with 192 nodes 81.3, 75.3, learned 449, 402;
// 120,701 nodes learned 76.5, 79.8); other quadrilaterals touch too many elements at 448. Large lumped
// hexahedral bricks: 330 nodes, whose operator has fewer partials to add up and less to recompute (64^3
// block: Jacobi 48.9 -> 40.2 us per iteration, the learned preconditioner's operator 32 -> 24.5, its
// layers 11.7 -> 10.5); below 512 such tiles the CUs need the smaller ones.
int default_tile_nodes(int ndim, int nnodes, const TileTraits &q);

// special[n] != 0 marks nodes that need the general update (restrained DOF, dashpot,
// Rayleigh mass damping, point load).
void make_tiles(int ndim, int nnodes, int nelem, int nen, const double *X, const int32_t *conn,
                const int32_t *color, int ncolors, const uint8_t *special, int max_own, HostTiles &t);

// The tiles of a model: of at most tile_nodes nodes, or of the default size (tile_nodes <= 0), which
// must leave the corner-slot kernels possible where smaller tiles do (512 elements a tile; flat or
// long tiles touch more).
void plan_tiles(int ndim, int nnodes, int nelem, int nen, const double *X, const int32_t *conn, const int32_t *color,
                int ncolors, const uint8_t *special, int tile_nodes, const TileTraits &q, HostTiles &t);

// What the multi-step plan is made from, in device numbering (empty: the model has no plan).
struct MultiInput {
    std::vector<int32_t> conn;         // [nelem*nen]
    std::vector<int32_t> n2e_ptr, n2e; // [nnodes+1], node -> element * nen + corner in ascending element order
    std::vector<int32_t> own_ptr;      // [ntiles+1]
    std::vector<uint8_t> special;      // [nnodes] nodes that take the general update
    std::vector<double> lam, mu;       // [nelem] Lame constants, times the volume scale on the table paths
    std::vector<uint16_t> gid;         // [nelem] geometry-table entry (empty: none)
};

// Deep-halo plan of the multi-step explicit kernel over the same tiles: every tile's nodes in
// rings around its owned nodes (ring d: reached through d layers of elements) and its elements in
// layers (layer d: touching a node of ring d or nearer), so that a workgroup can advance its owned
// nodes by up to `depth` steps from one staging.
struct HostMulti {
    struct Tile {
        std::vector<int32_t> node, elem;  // device nodes by ring, elements (tag order) by layer
        std::vector<int32_t> ncnt, ecnt;  // nodes up to ring 0..depth, elements up to layer 0..depth-1
        std::vector<uint16_t> conn;       // [elements * nen] staged slot of each corner
    };
    int depth = 0, nen = 0;
    int ns = 0, ne = 0, nu = 0;  // strides: staged nodes, elements, updated nodes (rings < depth)
    std::vector<Tile> tiles;
};

// False if a tile needs more than max_threads staged nodes or elements, or if memory ran out in a
// worker (in the caller's thread: std::bad_alloc).
bool make_multi(const MultiInput &in, int nen, int depth, int max_threads, HostMulti &t);

// The plan's arrays as the kernel reads them, all of fixed strides per tile.
struct MultiArrays {
    int32_t *cnt;            // [ntiles][2 (depth + 1)]: ncnt, ecnt, 0
    int32_t *node;           // [ntiles][ns] device node, the sign bit set on special nodes
    uint16_t *econn;         // [ntiles][ne][nen] staged slot of each corner
    uint16_t *ncor;          // [ntiles][nu][nen] tile element whose corner a the node is, or none
    uint16_t *egeo;          // [ntiles][ne]
    double *elam, *emu;      // [ntiles][ne], 0 on the padding
};
void fill_multi(const HostMulti &t, const MultiInput &in, int none, const MultiArrays &o);

}  // namespace svlg
