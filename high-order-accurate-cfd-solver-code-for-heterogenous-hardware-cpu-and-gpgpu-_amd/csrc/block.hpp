// Structured-block data shared by the block kernels and the block / batch host objects.
#pragma once
#include <hip/hip_runtime.h>

#include <cstdint>

#include "ctx.hpp"
#include "physics.hpp"

namespace cfdx {
namespace blk {

// Tile shapes compiled into the kernels; a launch list picks one of each at run time (the
// autotuner times them on the actual grids). All tiles have 256 threads.
//   face sweep along i: (TA lines across = j, TB faces along i); variant 0: the next 256 faces of the lines one
//   after the other (line_tile), four lines of 64
//   face sweeps along j and k: (TA lines across = i, TB faces along j or k)
//   node kernels: (TX along i, TY along j) at one k
constexpr int N_FACE_I = 3, N_FACE_JK = 4, N_NODE = 4;
constexpr int FACE_I_TILES[N_FACE_I][2] = {{4, 64}, {2, 128}, {8, 32}};
constexpr int FACE_JK_TILES[N_FACE_JK][2] = {{16, 16}, {32, 8}, {64, 4}, {8, 32}};
constexpr int NODE_TILES[N_NODE][2] = {{64, 4}, {32, 8}, {128, 2}, {256, 1}};

struct TileCfg {
    int face[3] = {0, 0, 0};   // variant of the i, j, k face sweeps
    int node = 0;              // variant of the node kernels
    // node tile order: strips of this many tile rows (0: whole planes). Strips of 4 rows by
    // default: a thin block's planes, split over the 8 XCDs, would otherwise give each XCD only a
    // few planes, whose k +- 2 neighbours another XCD reads (C-grid 384x128x32: +1-2 %)
    int strip = 4;
    bool operator==(const TileCfg &o) const
    {
        return face[0] == o.face[0] && face[1] == o.face[1] && face[2] == o.face[2] && node == o.node &&
               strip == o.strip;
    }
};

// Device-side view of one block: sizes, array pointers and per-block run parameters.
// P, Fv and FH hold the flux type (double or float); everything else is double.
struct BlockDev {
    int ni, nj, nk;             // owned nodes
    uint32_t n;                 // the length of every array
    int pi, pj;                 // stored rows: their pitch, and how many to a plane (index strides)
    int off[3];                 // ghost layers before the first owned node along i, j, k (3, or 0 if periodic)
    const uint8_t *code;        // bounded blocks: per stored node 0 interior, 1 boundary node, 100 ghost
    int bc[6];                  // side conditions (CFDX_BC_*) of i-, i+, j-, j+, k-, k+
    int cut_i0, cut_i1;         // wall range of a CFDX_BC_WALL_CUT side
    double cos_aoa, sin_aoa;    // far-field flow direction
    uint32_t tile0[4];          // first global tile of this block: node tiles, face tiles x, y, z
    uint32_t stream;            // the list's non-temporal switch, for the face sweeps
    uint32_t strip;             // node tiles: rows of tiles per strip walked plane by plane (0: whole planes)
    const double *det;          // det at the node
    const double *m[9];         // node metrics zeta_x .. xi_z
    const double *kf[3][3];     // face metric row of direction d at the +1/2 face (zeta_?ip, eta_?jp, xi_?kp)
    const double *df[3];        // half-point det at ip, jp, kp
    const float *geo32;         // mixed blocks: float copies of the 22 geometry arrays above, in their
                                // order (det, m, kf, df); null in FP64 blocks
    void *P[5];                 // rho, u, v, w, p used by the flux kernels
    double *U0[5];              // RK base det*Q
    double *Us[5];              // stage vector U1 / U2
    void *Fv[3][4];             // viscous fluxes, components 1..4 (the mass component is identically 0)
    double *mu;
    void *FH[3][5];             // face fluxes F-hat at the +1/2 faces
    double *mon;                // residual monitor: per-wave max |du|, |dv|, |de| of the last step (null: off)
    double del_t, mach, eps;
    int viscous;
    cfdx::dev::ViscParams vp;
};

// Thickness of the shell of a bounded block: the loc-selected derivative forms differ from the
// central ones only at a side's boundary node (every direction) and at the node next to it (the
// form that reaches the ghost layers); two nodes from the side the stencil's outer points are the
// boundary node and the interior, which select the central form.
constexpr uint32_t SHELL = 2;

// The shell of a bounded block (the nodes within SHELL of a side along a bounded direction; the tiled node
// kernels leave them to shell tiles) in two parts: the k planes and j rows, along which i runs, and the i
// columns left; 0 for a periodic block.
__host__ __device__ inline uint32_t shell_rows(const BlockDev &B)
{
    if (!B.code) return 0;
    const uint32_t ni = B.ni, nj = B.nj, nk = B.nk, kb = B.off[2] ? SHELL : 0u;
    return (B.off[2] ? 2 * SHELL * ni * nj : 0u) + (B.off[1] ? 2 * SHELL * ni * (nk - 2 * kb) : 0u);
}
__host__ __device__ inline uint32_t shell_columns(const BlockDev &B)
{
    if (!B.code || !B.off[0]) return 0;
    return 2 * SHELL * ((uint32_t)B.nj - (B.off[1] ? 2 * SHELL : 0u)) * ((uint32_t)B.nk - (B.off[2] ? 2 * SHELL : 0u));
}

// Shell tiles: 256 nodes of the rows, 64 or 256 of the columns. A column node's neighbours share no cache line
// with the next node's, so a wave's loads take 32 lines each and few columns are bound by the address rate of
// the few CUs they are on: up to COLUMNS_SPREAD nodes they go over four times the CUs. C-grids, us a step with 256
// and with 64, FP64: 128x64x16 (3840 column nodes) 168 and 146, 192x96x24 (8832) 352 and 347, 192x96x28 (10304) 427 and 426,
// 224x112x28 (12096) 634 and 637, 256x112x30 (12960) 722 and 725, 256x128x32 (15872) 857 and 863; mixed: 132 and 104, 258 and
// 241, 282 and 268, 359 and 354, 438 and 435, 552 and 549. The line lies where the two types' gain and loss meet.
constexpr uint32_t SHELL_TILE = 256, COLUMNS_SPREAD = 12288;
__host__ __device__ inline uint32_t shell_column_tile(const BlockDev &B) { return shell_columns(B) <= COLUMNS_SPREAD ? 64u : 256u; }
__host__ __device__ inline uint32_t shell_row_tiles(const BlockDev &B) { return (shell_rows(B) + SHELL_TILE - 1) / SHELL_TILE; }
__host__ __device__ inline uint32_t shell_tile_count(const BlockDev &B)
{
    const uint32_t c = shell_column_tile(B);
    return shell_row_tiles(B) + (shell_columns(B) + c - 1) / c;
}
// The wave of the residual monitor's slots that wave w of shell tile s has: four a row tile, then those of the
// column tiles.
__host__ __device__ inline uint32_t shell_wave(const BlockDev &B, uint32_t s, uint32_t w)
{
    const uint32_t rows = shell_row_tiles(B);
    return s < rows ? 4 * s + w : 4 * rows + (s - rows) * (shell_column_tile(B) / 64) + w;
}

// How the kernels of a list go over its blocks: with shell tiles beside the node tiles if some block has a bounded
// direction, and with non-temporal accesses to what a kernel touches once if the list streams.
enum : int { LIST_PLAIN, LIST_STREAM, LIST_BOUNDED, LIST_BOUNDED_STREAM };
constexpr bool list_streams(int k) { return (k & 1) != 0; }
constexpr bool list_bounded(int k) { return (k & 2) != 0; }

// Bytes of a stored node that a stage reads and writes (FP64: 22 geometry arrays, U0, Us, P, Fv, FH; mixed:
// the float geometry, det, U0, Us and the 32 float arrays).
__host__ __device__ inline uint64_t stage_bytes(uint64_t n, bool mixed) { return n * (mixed ? 304 : 512); }
__host__ __device__ inline uint64_t stage_bytes(const BlockDev &B) { return stage_bytes(B.n, B.geo32 != nullptr); }

// The size past which a block or a list streams: below it a stage's arrays stay in the 256 MB last-level
// cache (and the L2s) from one stage to the next, and the hint gives that up. FP64: 64^3 197 us a step
// with the hint, 177 without; 80^3 (262 MB) 449 and 391; 96^3 (453 MB) 708 and 731; 256^3 12.88 and 13.09 ms.
// Mixed: 64^3 125 and 112 us, 96^3 (269 MB) 400 and 369, 112^3 (427 MB) 622 and 643, 128^3 889 and 937.
// C-grids, FP64: 192x96x24 (288 MB) 423 and 378, 256x128x32 (575 MB) 889 and 904, 384x128x32 1284 and 1306; mixed:
// 256x128x32 (341 MB) 588 and 572, 384x128x32 (508 MB) 829 and 843.
// Past it, rows that are not whole 64-byte pieces cost as well (row_layout): below, the pieces that two rows share
// are found in the cache, and end to end the arrays take less of it.
constexpr uint64_t STREAM_BYTES = (uint64_t)384 << 20;

// Whether a block takes non-temporal accesses: past that size, with rows of whole 64-byte pieces. With others the hint
// drops lines that the neighbouring rows still need (FP64 161x131x127 1.5 % slower, 255x200x160 2.5 %, mixed 4 and 5 %).
inline bool streams_past_cache(const BlockDev &B)
{
    return (uint64_t)B.pi * (B.geo32 ? 4 : 8) % 64 == 0 && stage_bytes(B) > STREAM_BYTES;
}

// One launch over a list of blocks.
struct LaunchList {
    const BlockDev *blks = nullptr;   // device array
    const uint32_t *prefix[4] = {};   // device arrays of nblk+1 tile offsets (node, face x, y, z)
    uint32_t nblk = 0;
    uint32_t total[4] = {};
    uint32_t grid_cap = 0;            // 0: one workgroup per tile; else persistent grid of this size
    TileCfg tiles;
    uint32_t bc_face = 0;             // largest side face (owned nodes) of the bounded blocks; 0 if none
    uint32_t bc_face_d[3] = {};       // the same per direction (0: no block bounded in that direction)
    uint32_t bc_planes = 0;           // largest nk of the blocks bounded along i
    uint32_t shell_tiles = 0;         // most shell tiles of a bounded block
    bool stream = false;              // past the cache: non-temporal accesses
    double *Lout = nullptr;           // mode 3 (a single block): the right-hand side, 5 x owned nodes
};

// kernels (block_kernels.hip)
// ev (optional): 6 events recorded before the viscous kernel, after it, after each face sweep
// and after the update
// ov (optional, ignored when timing with ev): the viscous node kernel and the face sweeps run together:
// in one launch with the default tile shapes and grid, else the viscous kernel on ov->aux, forked from
// st before the sweeps and joined back before the update
// Returns the number of kernels launched.
struct Overlap {
    hipStream_t aux;
    hipEvent_t fork, join;
};
int stage(const LaunchList &L, int precision, int mode, hipStream_t st, bool any_visc, hipEvent_t *ev,
          const Overlap *ov = nullptr);
// whether stage() puts the viscous kernel on the second stream: other tile shapes than the defaults or a
// capped grid, with the overlap on
bool stage_forks(const LaunchList &L, const Overlap *ov);
// the float copies of the geometry of a mixed block (after every write of its double geometry)
// after every geometry write: face arrays to unit normal and det_f |k|, then the float copy
void geometry_finalize(const BlockDev &B, hipStream_t st);
// P and U0 of the owned nodes from double primitives staged component-major in owned order
void base(const BlockDev &B, int precision, hipStream_t st, const double *stage);
// rows of w doubles, end to end in src, to rows of a pitch in dst
void spread_rows(const double *src, double *dst, size_t rows, uint32_t w, uint32_t pitch, hipStream_t st);
void prims(const BlockDev &B, int precision, hipStream_t st, double *out);
// *count += the number of workgroups that found a value that is not finite in p[0..n)
void count_nonfinite(const double *p, size_t n, unsigned *count, hipStream_t st);
// FLOW records (cfdx_flow) of the owned nodes, owned order, into device memory
void flow_out(const BlockDev &B, int precision, hipStream_t st, cfdx_flow *out, double mach);
uint32_t tiles_of(const BlockDev &B, int kind, const TileCfg &cfg);
// side conditions of the bounded blocks of a list (mode 0..2 after that RK stage, mode 2 also
// refreshing U0), side by side in the order i-, i+, j-, j+, k-, k+; stage() runs it after the update
void boundary(const LaunchList &L, int precision, int mode, hipStream_t st);
// out[0..2] (device) = maxima of count per-wave monitor triples
void monitor_reduce(const double *mon, uint32_t count, double *out, hipStream_t st);

// device-side set-up (init_kernels.hip)
void init_geometry(const BlockDev &B, const double L[3], double amp, const double ph[3], hipStream_t st);
void init_state(const BlockDev &B, const double L[3], double amp, const double ph[3], int kind, double mach, double beta,
                double xc, double yc, hipStream_t st);
int cfl_parts(const BlockDev &B);
void cfl_radius(const BlockDev &B, double *part, hipStream_t st);

}  // namespace blk
}  // namespace cfdx
