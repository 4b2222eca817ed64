// Structured-block kernels. Each block is one ni x nj x nk grid, periodic or bounded, held in HBM as
// structure-of-arrays; a launch covers a list of blocks (one for cfdx_block_step, many for a
// batch), every workgroup taking one tile of one block through a prefix table of tile counts.
//   k_flux        a stage's viscous tiles and face tiles in one launch (default tile shapes); apart:
//   k_visc        node kernel: Fv, Ev, Gv (+ mu) from the stage vector U (Viscous.cl)
//   k_face<DIR>   one thread per face (i+1/2 along DIR): characteristic WCNS reconstruction,
//                 LLF and the 6th-order midpoint correction (Weno.cl), LDS-staged tiles
//   k_update      flux differences + viscous divergence -> L, SSP-RK3 stage j, primitives
//                 (Weno.cl:3060-3135)
//   k_bc_ij, k_bc side conditions of bounded blocks after each stage
// Each face flux is computed once and shared by its two nodes (the reference computes it
// twice, once from each side, with identical operands).
// S is the flux arithmetic / storage type: double (plain form) or float (mixed form). The RK
// base U0, the stage vector Us, the metrics and the L accumulation are double in both.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "block.hpp"

using namespace cfdx::dev;

namespace cfdx {
namespace blk {

// Loads and stores at a 32-bit element index from a uniform base pointer, so the compiler
// emits SGPR-base + VGPR-offset accesses (a block holds < 2^29 nodes). The array pointers come
// from a descriptor in memory, so they are cast to the global address space explicitly: global
// (not flat) instructions count only on the vector-memory wait counter, not on the LDS one.
#define CFDX_GLOBAL __attribute__((address_space(1)))
template <typename T>
__device__ __forceinline__ T ld(const T *base, uint32_t i)
{
    const CFDX_GLOBAL char *p = (const CFDX_GLOBAL char *)base;
    return *(const CFDX_GLOBAL T *)(p + i * (uint32_t)sizeof(T));
}
template <typename T>
__device__ __forceinline__ void st(T *base, uint32_t i, T v)
{
    CFDX_GLOBAL char *p = (CFDX_GLOBAL char *)base;
    *(CFDX_GLOBAL T *)(p + i * (uint32_t)sizeof(T)) = v;
}

// Streaming forms for data a kernel touches once (geometry read at its own node, outputs): the
// non-temporal hint lets the L2 evict these lines first, keeping the stencil neighbours that
// adjacent tiles read again. For the lists of blocks that streams_past_cache chooses.
template <bool NT, typename T>
__device__ __forceinline__ T ldx(const T *base, uint32_t i)
{
    if constexpr (NT)
        return __builtin_nontemporal_load((const CFDX_GLOBAL T *)((const CFDX_GLOBAL char *)base + i * (uint32_t)sizeof(T)));
    else
        return ld(base, i);
}
template <bool NT, typename T>
__device__ __forceinline__ void stx(T *base, uint32_t i, T v)
{
    if constexpr (NT)
        __builtin_nontemporal_store(v, (CFDX_GLOBAL T *)((CFDX_GLOBAL char *)base + i * (uint32_t)sizeof(T)));
    else
        st(base, i, v);
}

// Geometry array a (0 det, 1-9 node metrics, 10-18 face metric rows, 19-21 face dets) in the flux
// type: the double arrays in an FP64 block, their float copies in a mixed block (the flux
// arithmetic reads the metrics in S; the copies hold the same roundings a conversion at the load
// would give, in half the bytes).
template <typename S>
__device__ __forceinline__ const S *geo(const BlockDev &B, int a);
template <>
__device__ __forceinline__ const double *geo<double>(const BlockDev &B, int a) { return B.det + (size_t)a * B.n; }
template <>
__device__ __forceinline__ const float *geo<float>(const BlockDev &B, int a) { return B.geo32 + (size_t)a * B.n; }

__device__ __forceinline__ int wrapi(int i, int n) { return i < 0 ? i + n : (i >= n ? i - n : i); }

// stored index of owned coordinates (i, j, k); a bounded direction may go 3 nodes beyond the
// owned range into its ghost layers
__device__ __forceinline__ uint32_t node_index(const BlockDev &B, int i, int j, int k)
{
    return (uint32_t)(i + B.off[0]) + (uint32_t)B.pi * ((uint32_t)(j + B.off[1]) + (uint32_t)B.pj * (uint32_t)(k + B.off[2]));
}

// owned coordinate c + o along a direction of n owned nodes: wrapped if the direction is periodic
__device__ __forceinline__ int along_shift(const BlockDev &B, int d, int c, int o, int n)
{
    return B.off[d] ? c + o : wrapi(c + o, n);
}

__device__ __forceinline__ uint32_t shifted(const BlockDev &B, int i, int j, int k, int d, int o)
{
    if (d == 0) i = along_shift(B, 0, i, o, B.ni);
    else if (d == 1) j = along_shift(B, 1, j, o, B.nj);
    else k = along_shift(B, 2, k, o, B.nk);
    return node_index(B, i, j, k);
}

// number of +1/2 faces a sweep along d computes per line: one more than the owned nodes in a
// bounded direction (the face between the first owned node and its ghost)
__device__ __host__ __forceinline__ int faces_along(const BlockDev &B, int d)
{
    const int n = d == 0 ? B.ni : d == 1 ? B.nj : B.nk;
    return B.off[d] ? n + 1 : n;
}

// The form that the loc codes select for a derivative along d at a node (loc_derivative, Viscous.cl:285-435 and
// with weno_form Weno.cl:2732-2856): four points at offsets o and the weights of the three differences from each to the
// next, found without a branch, so that a shell node reads its codes in one memory round trip and its points in
// another (a branch per form, with seven points each, made the shell tiles the longest of a small launch: C-grid
// 128x64x16 update 26 us a stage). Every form's weights sum to zero, so differences carry it whole: they are exact for
// points near each other, and a uniform state gives exactly 0. Error against exact arithmetic on operands of order 1 that
// vary by 1e-3, rms: one-sided forms 8e-20, loc_derivative's sums of the values 6e-17 .. 1.5e-16; the central form's bits
// are those of the tiles (8 d is exact). The weights are held twelve times larger, with one factor for all forms: with
// a factor of its own to each form the mixed k_flux takes 98 registers instead of 96, 4 waves a SIMD instead of 5 (C-grid
// 384x128x32 864 us a step instead of 814). No match: zero weights on the node itself.
struct LocForm {
    int o[4];
    double w[3];
    // the derivative from the values at the four points
    __device__ __forceinline__ double of(const double (&f)[4]) const
    {
        return (1.0 / 12.0) * (w[0] * (f[0] - f[1]) + w[1] * (f[1] - f[2]) + w[2] * (f[2] - f[3]));
    }
};
__device__ __forceinline__ LocForm loc_form(int LI, int LM2, int LM1, int LP1, int LP2, bool weno_form)
{
    const bool side = LI > 0 && LI <= 52, in = LI == 0;
    const bool hi = side && LP1 == 100, lo = side && LM1 == 100;
    const bool by_hi = in && LP1 > 0 && LP1 <= 52 && LP2 == 100;
    const bool by_lo = in && LM1 > 0 && (!weno_form || LM1 <= 52) && LM2 == 100;
    const bool mid = LM2 != 100 && LM1 != 100 && LP2 != 100 && LP1 != 100 && (in || (!weno_form && LI > 0));
    LocForm f = {{0, 0, 0, 0}, {0.0, 0.0, 0.0}};
    auto take = [&](bool c, int o0, int o1, int o2, int o3, double w0, double w1, double w2) {
        f.o[0] = c ? o0 : f.o[0]; f.o[1] = c ? o1 : f.o[1]; f.o[2] = c ? o2 : f.o[2]; f.o[3] = c ? o3 : f.o[3];
        f.w[0] = c ? w0 : f.w[0]; f.w[1] = c ? w1 : f.w[1]; f.w[2] = c ? w2 : f.w[2];
    };
    // in the reference's order, a later match over an earlier one
    take(hi, 0, -1, -2, -3, 22.0, -14.0, 4.0);
    take(lo, 0, 1, 2, 3, -22.0, 14.0, -4.0);
    take(by_hi, 1, 0, -1, -2, 4.0, 10.0, -2.0);
    take(by_lo, -1, 0, 1, 2, -4.0, -10.0, 2.0);
    take(mid, 1, -1, 2, -2, 8.0, 0.0, -1.0);
    return f;
}
// the forms of a node along the three directions
__device__ __forceinline__ void loc_forms(const BlockDev &B, int i, int j, int k, bool weno_form, LocForm (&f)[3])
{
    const int LI = ld(B.code, node_index(B, i, j, k));
    int c[3][4];
#pragma unroll
    for (int d = 0; d < 3; ++d)
#pragma unroll
        for (int q = 0; q < 4; ++q) c[d][q] = ld(B.code, shifted(B, i, j, k, d, q < 2 ? q - 2 : q - 1));
#pragma unroll
    for (int d = 0; d < 3; ++d) f[d] = loc_form(LI, c[d][0], c[d][1], c[d][2], c[d][3], weno_form);
}

// The shell of a bounded block: the nodes within SHELL of a side along a bounded direction (the
// only nodes where a loc-selected form can differ from the central one). The node kernels skip it and
// the shell kernels cover it, so the tiled kernels carry no loc branches. Enumeration: the k shell
// planes (if k is bounded), then the j shell rows inside the k range left, then the i shell
// columns inside the j and k ranges left; i runs fastest in the first two parts.
__device__ __forceinline__ bool in_shell(const BlockDev &B, int i, int j, int k)
{
    const int c[3] = {i, j, k}, n[3] = {B.ni, B.nj, B.nk};
    bool s = false;
#pragma unroll
    for (int q = 0; q < 3; ++q) s |= B.off[q] && (c[q] < (int)SHELL || c[q] > n[q] - 1 - (int)SHELL);
    return s;
}

// Thread's node of shell tile s of the block, if it has one.
__device__ __forceinline__ bool shell_node(const BlockDev &B, uint32_t s, int &i, int &j, int &k)
{
    const uint32_t ni = B.ni, nj = B.nj, nk = B.nk, rows = shell_row_tiles(B), tid = threadIdx.x;
    const uint32_t kb = B.off[2] ? SHELL : 0u, jb = B.off[1] ? SHELL : 0u, w = 2 * SHELL;
    auto layer = [](uint32_t m, uint32_t n) { return (int)(m < SHELL ? m : n - 2 * SHELL + m); };
    if (s < rows) {
        uint32_t t = s * SHELL_TILE + tid;
        if (t >= shell_rows(B)) return false;
        const uint32_t planes = B.off[2] ? w * ni * nj : 0u;
        i = (int)(t % ni);
        if (t < planes) {
            j = (int)((t / ni) % nj);
            k = layer(t / (ni * nj), nk);
        } else {
            t -= planes;   // a multiple of ni
            j = layer((t / ni) % w, nj);
            k = (int)(kb + t / (w * ni));
        }
        return true;
    }
    const uint32_t c = shell_column_tile(B), t = (s - rows) * c + tid;
    if (tid >= c || t >= shell_columns(B)) return false;
    i = layer(t % w, ni);
    j = (int)(jb + (t / w) % (nj - 2 * jb));
    k = (int)(kb + t / (w * (nj - 2 * jb)));
    return true;
}

// Workgroups are dispatched round-robin over the 8 XCDs (workgroup b runs on XCD b % 8), each
// with its own L2. Remap the linear workgroup id so XCD x takes one contiguous range of tiles
// (a slab of k planes of one block). Bijective for any count.
__device__ __forceinline__ uint32_t xcd_tile(uint32_t b, uint32_t nb)
{
    const uint32_t q = nb >> 3, r = nb & 7u, x = b & 7u, l = b >> 3;
    return x * q + (x < r ? x : r) + l;
}

// Node tile lt of a block: (i0, j0) of its first node and its plane k. Tiles run along i, then
// (with B.strip = S > 0) through strips of S tile rows, each strip plane by plane, so that the
// k +- 2 planes of a strip are recent in the L2 of the XCD that walks it; S = 0: plane by plane.
__device__ __forceinline__ void node_tile(const BlockDev &B, uint32_t lt, int TX, int TY, int &i0, int &j0, int &k)
{
    const uint32_t ntx = (B.ni + TX - 1) / TX, nty = (B.nj + TY - 1) / TY, nk = (uint32_t)B.nk;
    const uint32_t S = B.strip;
    if (S == 0 || S >= nty) {
        i0 = (int)((lt % ntx) * TX);
        j0 = (int)(((lt / ntx) % nty) * TY);
        k = (int)(lt / (ntx * nty));
        return;
    }
    const uint32_t per_full = ntx * S * nk, full = nty / S;
    uint32_t sidx, r, rows;
    if (lt < full * per_full) { sidx = lt / per_full; r = lt % per_full; rows = S; }
    else { sidx = full; r = lt - full * per_full; rows = nty - full * S; }
    k = (int)(r / (ntx * rows));
    const uint32_t q = r % (ntx * rows);
    i0 = (int)((q % ntx) * TX);
    j0 = (int)((sidx * S + q / ntx) * TY);
}

// Runs f on the tiles of a launch: one workgroup per tile, or (LOOP) a smaller grid striding over all
// of them. The loop is a form of its own because the compiler moves everything a tile does not change
// (constants, index arithmetic) before it and then holds it throughout: the mixed i sweep takes 96
// registers with the loop.
template <bool LOOP, typename F>
__device__ __forceinline__ void each_tile(uint32_t all, const F &f)
{
    if constexpr (LOOP) {
        for (uint32_t wg = blockIdx.x; wg < all; wg += gridDim.x) f(wg);
    } else {
        f(blockIdx.x);
    }
}

// block of a global tile id: the largest b with prefix[b] <= t (prefix[0] = 0, prefix[nblk] = total)
__device__ __forceinline__ uint32_t find_block(const uint32_t *__restrict__ prefix, uint32_t nblk, uint32_t t)
{
    uint32_t lo = 0, hi = nblk;
    while (hi - lo > 1) {
        const uint32_t mid = (lo + hi) >> 1;
        if (prefix[mid] <= t) lo = mid; else hi = mid;
    }
    return lo;
}

// ---------------------------------------------------------------------------
// viscous node kernel (Viscous.cl:285-631 on a periodic block: central 4th order)
// ---------------------------------------------------------------------------
// Fv, Ev, Gv (+ mu) of one node. LOC: a shell node of a bounded block (loc-selected forms near
// the sides); otherwise the central forms.
// PT: the stage vector of the node's in-plane stencil (i and j offsets -2 .. 2) is read from a
// plane tile in LDS: pt[(c * rows + ty + 2 + dj) * cols + tx + 2 + di] (the same doubles the global
// loads would give); the k offsets are read from global memory.
template <typename S, bool LOC, bool NT, bool PT = false>
__device__ __forceinline__ void visc_node(const BlockDev &B, int i, int j, int k, int mode, const double *pt = nullptr,
                                          int tx = 0, int ty = 0, int cols = 0, int rows = 0)
{
    const uint32_t g = node_index(B, i, j, k);
    // stage vector into the viscous kernel: U0 at j = 0, the raw U1 / U2 after (Solver.cpp:427-435)
    const double *const *Uin = (mode == 0 || mode == 3) ? B.U0 : B.Us;
    auto tile = [&](int c, int d, int o) -> double {
        return pt[(c * rows + ty + 2 + (d == 1 ? o : 0)) * cols + tx + 2 + (d == 0 ? o : 0)];
    };
    double U[5];
#pragma unroll
    for (int c = 0; c < 5; ++c) U[c] = PT ? tile(c, 0, 0) : ld(Uin[c], g);
    const double iU0 = pinv_(U[0]);
    // the differences are taken in double; the flux arithmetic runs in S
    S Uv[5];
#pragma unroll
    for (int c = 0; c < 5; ++c) Uv[c] = S(U[c]);
    const NodeRatios<S> nr = node_ratios(Uv);
    S m[9], G[4][3] = {}, sk[3];
    // adds direction d from the neighbours at d -+ 1 (a, b) and the differences dU; gives the magnitude of
    // the MTS scale-similarity term of momentum component d + 1 along d (Viscous.cl:493-495)
    auto add = [&](int d, double Ud, const S(&dU)[5], double a0, double b0, double ad, double bd, S mx, S my, S mz) -> S {
        const double x = (Ud * iU0) - ((0.25 * ad + 0.5 * Ud + 0.25 * bd) * pinv_(0.25 * a0 + 0.5 * U[0] + 0.25 * b0));
        S r = S(fabs_(x));
        pin_(r);   // or the whole term would sink, with its operands alive, to its use after the loop
        add_gradient(dU, nr, mx, my, mz, G);
#pragma unroll
        for (int c = 0; c < 4; ++c)
#pragma unroll
            for (int e = 0; e < 3; ++e) pin_(G[c][e]);
        return r;
    };
    if constexpr (LOC) {
        LocForm form[3];
        loc_forms(B, i, j, k, false, form);
#pragma unroll
        for (int d = 0; d < 3; ++d) {
            uint32_t x[4];
#pragma unroll
            for (int q = 0; q < 4; ++q) x[q] = shifted(B, i, j, k, d, form[d].o[q]);
            const uint32_t m1 = shifted(B, i, j, k, d, -1), p1 = shifted(B, i, j, k, d, 1);
            const double a0 = ld(Uin[0], m1), b0 = ld(Uin[0], p1), ad = ld(Uin[1 + d], m1), bd = ld(Uin[1 + d], p1);
            const S mx = ld(geo<S>(B, 1 + 3 * d), g), my = ld(geo<S>(B, 2 + 3 * d), g), mz = ld(geo<S>(B, 3 + 3 * d), g);
            S dU[5];
#pragma unroll
            for (int c = 0; c < 5; ++c) {
                const double *u = Uin[c];
                dU[c] = S(form[d].of({ld(u, x[0]), ld(u, x[1]), ld(u, x[2]), ld(u, x[3])}));
            }
            sk[d] = add(d, U[1 + d], dU, a0, b0, ad, bd, mx, my, mz);
        }
        uint32_t g2 = g;
        pin_(g2);   // the metrics again, not held through the gradients
#pragma unroll
        for (int c = 0; c < 9; ++c) m[c] = ld(geo<S>(B, 1 + c), g2);
    } else {
#pragma unroll
        for (int q = 0; q < 3; ++q) {
            const int d = 2 - q;   // k first: its neighbours come from global memory
            const uint32_t m2 = shifted(B, i, j, k, d, -2), m1 = shifted(B, i, j, k, d, -1);
            const uint32_t p1 = shifted(B, i, j, k, d, 1), p2 = shifted(B, i, j, k, d, 2);
            double a0, b0, ad, bd;
            S dU[5];
#pragma unroll
            for (int c = 3 * d; c < 3 * d + 3; ++c) m[c] = ldx<NT>(geo<S>(B, 1 + c), g);
#pragma unroll
            for (int c = 0; c < 5; ++c) {
                const double *u = Uin[c];
                double a, b, a2, b2;
                if (PT && d < 2) {
                    a = tile(c, d, -1); b = tile(c, d, 1); a2 = tile(c, d, -2); b2 = tile(c, d, 2);
                } else {
                    a = ld(u, m1); b = ld(u, p1); a2 = ld(u, m2); b2 = ld(u, p2);
                }
                dU[c] = S((1.0 / 12.0) * (8.0 * (b - a) - (b2 - a2)));
                if (c == 0) { a0 = a; b0 = b; }
                if (c == d + 1) { ad = a; bd = b; }
            }
            sk[d] = add(d, U[1 + d], dU, a0, b0, ad, bd, m[3 * d], m[3 * d + 1], m[3 * d + 2]);
        }
    }
    S fv[3][5];
    // the node velocity: away from the sides, from the stage vector already in registers (U_m /
    // U_0, the primitives of P up to rounding) instead of three more loads; near the sides the
    // side conditions set P apart from the stage vector, so it is read from P
    S vel[3];
#pragma unroll
    for (int c = 0; c < 3; ++c) vel[c] = LOC ? ld((const S *)B.P[1 + c], g) : S(U[1 + c] * iU0);
    const S mu = viscous_fluxes(G, Uv, nr, vel[0], vel[1], vel[2], m, ldx<NT>(geo<S>(B, 0), g), sk, B.vp, fv);
#pragma unroll
    for (int d = 0; d < 3; ++d)
#pragma unroll
        for (int c = 1; c < 5; ++c) stx<NT>((S *)B.Fv[d][c - 1], g, fv[d][c]);
    if (mode >= 2) stx<NT>(B.mu, g, (double)mu);
}

// Doubles of LDS a node tile of the viscous kernel stages: tiles of at least 4 rows hold the stage
// vector of the tile and its in-plane halo (each state loaded once per tile instead of once per node
// that reaches it).
template <int TX, int TY>
constexpr int VISC_LDS = TY >= 4 ? 5 * (TY + 4) * (TX + 4) : 1;

// Viscous node fluxes of the nodes of tile lt of block B; plane: VISC_LDS<TX, TY> doubles of LDS.
template <typename S, int TX, int TY, int K>
__device__ __forceinline__ void visc_tile(const BlockDev &B, uint32_t lt, int mode, double *plane)
{
    constexpr bool BND = list_bounded(K), NT = list_streams(K);
    constexpr int PC = TX + 4, PR = TY + 4;
    int i0, j0, k;
    node_tile(B, lt, TX, TY, i0, j0, k);
    const int tx = (int)(threadIdx.x % TX), ty = (int)(threadIdx.x / TX);
    const int i = i0 + tx, j = j0 + ty;
    if constexpr (TY >= 4) {
        // the stage vector of the tile and its in-plane halo (2 nodes on each side, corners
        // left out) into LDS; points past the last node a tile node reaches are skipped
        const double *const *Uin = (mode == 0 || mode == 3) ? B.U0 : B.Us;
        __syncthreads();   // the LDS of the previous tile fully read
        for (int p = (int)threadIdx.x; p < PR * PC; p += TX * TY) {
            const int r = p / PC, q = p % PC;
            const bool hi = q >= 2 && q < TX + 2, hj = r >= 2 && r < TY + 2;
            if (!hi && !hj) continue;
            if (i0 + q - 2 > B.ni + 1 || j0 + r - 2 > B.nj + 1) continue;
            const uint32_t x = node_index(B, along_shift(B, 0, i0, q - 2, B.ni), along_shift(B, 1, j0, r - 2, B.nj), k);
#pragma unroll
            for (int c = 0; c < 5; ++c) plane[(c * PR + r) * PC + q] = ld(Uin[c], x);
        }
        __syncthreads();
    }
    if (i >= B.ni || j >= B.nj) return;
    if (BND && B.code && in_shell(B, i, j, k)) return;   // a shell tile's node
    if constexpr (TY >= 4) visc_node<S, false, NT, true>(B, i, j, k, mode, plane, tx, ty, PC, PR);
    else visc_node<S, false, NT>(B, i, j, k, mode);
}

// Viscous node fluxes of shell tile s of the list (block = s / shell_tiles).
template <typename S>
__device__ __forceinline__ void visc_shell_tile(const BlockDev *__restrict__ blks, uint32_t s, int mode, uint32_t shell_tiles)
{
    const BlockDev &B = blks[s / shell_tiles];
    int i, j, k;
    if (B.viscous && B.code && shell_node(B, s % shell_tiles, i, j, k)) visc_node<S, true, false>(B, i, j, k, mode);
}

// Node tiles of the list first (tile ids through the XCD remap), then, for lists with bounded
// blocks, nblk x shell_tiles shell tiles of up to TX * TY shell nodes each (SHELL_TILE; block = id / shell_tiles),
// dispatched last in plain order so that they spread over the XCDs at the end of the launch.
template <typename S, int TX, int TY, int K, bool LOOP>
__global__ void __launch_bounds__(TX *TY, ((TY >= 4 && !(LOOP && list_bounded(K))) || sizeof(S) == 4 ? 4 : 3))
    k_visc(const BlockDev *__restrict__ blks, const uint32_t *__restrict__ prefix, uint32_t nblk, uint32_t total, int mode,
           uint32_t shell_tiles)
{
    constexpr bool BND = list_bounded(K);
    __shared__ double plane[VISC_LDS<TX, TY>];
    const uint32_t all = total + (BND ? nblk * shell_tiles : 0u);
    auto tile = [&](uint32_t wg) {
        if (BND && wg >= total) {
            visc_shell_tile<S>(blks, wg - total, mode, shell_tiles);
            return;
        }
        const uint32_t t = xcd_tile(wg, total);
        const BlockDev &B = blks[find_block(prefix, nblk, t)];
        if (B.viscous) visc_tile<S, TX, TY, K>(B, t - B.tile0[0], mode, plane);
    };
    each_tile<LOOP>(all, tile);
}

// ---------------------------------------------------------------------------
// face kernel: F-hat at the +1/2 face of every node along DIR. A tile is TB faces along DIR
// times TA lines across it. Phase 1 stages the conserved state Q and the node flux F_DIR of the
// TB+5 stencil points of every line in LDS (each point computed once per tile); phase 2 gives
// each thread one face, reading its six stencil points from LDS.
// ---------------------------------------------------------------------------
template <int DIR, int TA, int TB>
__device__ __forceinline__ int lds_at(int c, int s, int a)
{
    constexpr int NP = TB + 5;
    return DIR == 0 ? (c * TA + a) * NP + s : (c * NP + s) * TA + a;
}

template <int DIR>
__device__ __forceinline__ uint32_t tile_node(const BlockDev &B, int along, int across, int fixed)
{
    if (DIR == 0) return node_index(B, along, across, fixed);
    if (DIR == 1) return node_index(B, across, along, fixed);
    return node_index(B, across, fixed, along);
}

// Mixed form: the Roe state's inputs (rho, u, v, w, h) of the stencil points are staged too, so
// phase 2 reads the two centre nodes from LDS; FP64 derives them from the conserved states of
// the two centre nodes, which phase 2 holds in registers anyway (no primitive loads; staging
// them in FP64 would cost a wave per SIMD).
template <typename S>
constexpr bool STAGE_ROE = std::is_same<S, float>::value;

// Values of LDS a point of a face tile takes: Q, the node flux and (mixed form) the Roe inputs.
template <typename S>
constexpr int POINT_VALUES = STAGE_ROE<S> ? 15 : 10;
template <typename S, int TA, int TB>
constexpr int FACE_LDS = POINT_VALUES<S> * (TB + 5) * TA;

// Phase 1: the values of the point at stored node x, handed to put(value, its place).
template <typename S, int DIR, typename Put>
__device__ __forceinline__ void stage_point(const BlockDev &B, uint32_t x, const Put &put)
{
    const S rho = ld((const S *)B.P[0], x), u = ld((const S *)B.P[1], x), v = ld((const S *)B.P[2], x), w = ld((const S *)B.P[3], x),
            pr = ld((const S *)B.P[4], x);
    S q[5], f[5];
    prim_to_q(rho, u, v, w, pr, q);
    node_flux_e(rho, u, v, w, pr, q[4] + pr, ld(geo<S>(B, 1 + 3 * DIR), x), ld(geo<S>(B, 2 + 3 * DIR), x),
                ld(geo<S>(B, 3 + 3 * DIR), x), ld(geo<S>(B, 0), x), f);
#pragma unroll
    for (int c = 0; c < 5; ++c) {
        put(c, q[c]);
        put(5 + c, f[c]);
    }
    if constexpr (STAGE_ROE<S>) {
        put(10, rho); put(11, u); put(12, v); put(13, w);
        put(14, enthalpy(rho, u, v, w, pr));
    }
}

// Phase 2: the flux of the face at stored node gl; get(m, v) is value v of its stencil point m (0..5).
template <typename S, int DIR, typename Get>
__device__ __forceinline__ void face_at(const BlockDev &B, uint32_t gl, const Get &get)
{
    auto q = [&](int m, int c) { return get(m, c); };
    S roe[5], irho;
    if constexpr (STAGE_ROE<S>) {
        // the face's two centre nodes are stencil points 2 and 3
        irho = roe_average(get(2, 10), get(2, 11), get(2, 12), get(2, 13), get(2, 14), get(3, 10), get(3, 11), get(3, 12), get(3, 13),
                           get(3, 14), roe);
    } else {
        // from the conserved states of the two centre nodes
        S qa[5], qb[5], ia, ib, ua, va, wa, ha, ub, vb, wb, hb;
#pragma unroll
        for (int c = 0; c < 5; ++c) { qa[c] = q(2, c); qb[c] = q(3, c); }
        pinv2_(qa[0], qb[0], ia, ib);
        q_roe_inputs(qa, ia, ua, va, wa, ha);
        q_roe_inputs(qb, ib, ub, vb, wb, hb);
        irho = roe_average(qa[0], ua, va, wa, ha, qb[0], ub, vb, wb, hb, roe);
    }
    // unit face normal and det_f |k| (the stored face arrays after geometry_finalize)
    S fg[4];
    if (!B.stream) {
#pragma unroll
        for (int c = 0; c < 3; ++c) fg[c] = ld(geo<S>(B, 10 + 3 * DIR + c), gl);
        fg[3] = ld(geo<S>(B, 19 + DIR), gl);
    } else {
#pragma unroll
        for (int c = 0; c < 3; ++c) fg[c] = ldx<true>(geo<S>(B, 10 + 3 * DIR + c), gl);
        fg[3] = ldx<true>(geo<S>(B, 19 + DIR), gl);
    }
    S llf[5];
    face_llf(q, roe, irho, fg[0], fg[1], fg[2], fg[3], S(B.eps), llf);
    S fh[5];
#pragma unroll
    for (int c = 0; c < 5; ++c)
        fh[c] = S(llf[c] + midpoint_correction(get(0, 5 + c), get(1, 5 + c), get(2, 5 + c), get(3, 5 + c), get(4, 5 + c), get(5, 5 + c)));
    if (!B.stream) {
#pragma unroll
        for (int c = 0; c < 5; ++c) st((S *)B.FH[DIR][c], gl, fh[c]);
    } else {
#pragma unroll
        for (int c = 0; c < 5; ++c) stx<true>((S *)B.FH[DIR][c], gl, fh[c]);
    }
}

// Lines to a row of the j and k sweeps' tiles: the sweeps go over the lines of all rows one after the other, so that
// the last tile of a row is not partly empty (a tile takes TA lines, 97 nodes would be seven tiles of 16; us a step with
// those and with these, FP64 and mixed: 97x83x61 344 and 337, 222 and 218; 50x70x90 255 and 230, 154 and 147; rows of whole
// tiles are unchanged). Blocks that stream keep a tile's lines in a row, on whole pieces of memory.
__device__ __host__ __forceinline__ int line_row(const BlockDev &B, int TA)
{
    return stage_bytes(B) > STREAM_BYTES ? (B.ni + TA - 1) / TA * TA : B.ni;
}

// The faces of tile lt of block B along DIR; sq: FACE_LDS<S, TA, TB> values of LDS.
template <typename S, int DIR, int TA, int TB>
__device__ __forceinline__ void face_tile(const BlockDev &B, uint32_t lt, S *sq)
{
    static_assert(TA * TB == 256, "face tiles have 256 threads");
    constexpr int NP = TB + 5;
    const int tid = threadIdx.x;
    const int n_along = DIR == 0 ? B.ni : DIR == 1 ? B.nj : B.nk;
    // face f of a line is the +1/2 face of along-coordinate f - sh (sh = 1 in a bounded
    // direction: the first face lies between the first owned node and its ghost)
    const int nfa = faces_along(B, DIR), sh = B.off[DIR] ? 1 : 0;
    // tiles run along the lines' direction before the fixed coordinate, so that the next tile of
    // an XCD re-reads the stencil halo planes of this one from its L2
    const uint32_t ntb = (nfa + TB - 1) / TB, nta = DIR == 0 ? (B.nj + TA - 1) / TA : (B.ni + TA - 1) / TA;
    const int tb = DIR == 0 ? tid % TB : tid / TA, ta = DIR == 0 ? tid / TB : tid % TA;
    int b0, a0, fixed, across = 0;
    bool line;
    if (DIR == 0) {
        b0 = (lt % ntb) * TB; a0 = ((lt / ntb) % nta) * TA; fixed = lt / (ntb * nta);
        line = a0 + ta < B.nj;
    } else {
        // a row of tiles takes the next nta * TA lines, whose across coordinate i runs on from one fixed coordinate
        // to the next after row lines
        const int row = line_row(B, TA), nfix = DIR == 1 ? B.nk : B.nj;
        const uint32_t r = lt / (nta * ntb), rest = lt - r * (nta * ntb), tile_b = rest / nta, a = rest - tile_b * nta;
        b0 = tile_b * TB;
        a0 = 0;
        fixed = (int)r;
        across = (int)(a * TA) + ta;
        if (row != (int)(nta * TA)) {
            const uint32_t l0 = (r * nta + a) * TA;
            fixed = (int)(l0 / (uint32_t)row);
            across = (int)(l0 - (uint32_t)fixed * (uint32_t)row) + ta;
            while (across >= row) { across -= row; ++fixed; }
        }
        line = across < B.ni && fixed < nfix;
    }

    __syncthreads();   // the previous tile's LDS fully consumed
    for (int p = tid; p < NP * TA; p += 256) {
        const int s = DIR == 0 ? p % NP : p / TA;
        const int a = DIR == 0 ? p / NP : ta;
        if (DIR == 0 ? a0 + a >= B.nj : !line) continue;
        // the points past the stencil of the tile's last computed face feed no face: skip them
        // (a bounded line ends 3 ghost nodes past its last owned node; a periodic line shorter
        // than the tile would wrap more than once)
        if (s > nfa - b0 + 4) continue;
        const int along = along_shift(B, DIR, b0 - sh, s - 2, n_along);
        const uint32_t x = tile_node<DIR>(B, along, DIR == 0 ? a0 + a : across, fixed);
        stage_point<S, DIR>(B, x, [&](int v, S y) { sq[lds_at<DIR, TA, TB>(v, s, a)] = y; });
    }
    __syncthreads();

    if (b0 + tb < nfa && line) {
        face_at<S, DIR>(B, tile_node<DIR>(B, b0 + tb - sh, DIR == 0 ? a0 + ta : across, fixed),
                        [&](int m, int v) { return sq[lds_at<DIR, TA, TB>(v, tb + m, ta)]; });
    }
}

// Variant 0 of the i sweep: a tile is the next line_faces() faces of the block's lines one after the other, whatever
// their length, so that no tile but the last is partly empty. (Tiles of 4 lines by 64 faces gave the 385 faces of a
// bounded line of 384 nodes 7 tiles, and 97 faces 2; us a step with those and with these, FP64 and mixed: C-grids
// 128x64x16 146 and 141, 107 and 103; 384x128x32 1279 and 1257, 825 and 807; 97x83x61 353 and 344, 226 and 221; sizes of
// whole tiles 0-0.5 %.) The stencil points of its faces are the points of the lines' own sequence, row = nf + 5 to
// a line, from that of its first face on.
constexpr int LINE_POINTS = 336;
__device__ __host__ __forceinline__ uint32_t line_faces(uint32_t nf)
{
    // 256 faces reach over 16 lines of 17, 256 + 16 x 5 points; shorter lines: n faces touch up to n / nf + 2
    return nf >= 17 ? 256u : (LINE_POINTS - 10) * nf / (nf + 5);
}

template <typename S>
__device__ __forceinline__ void line_tile(const BlockDev &B, uint32_t lt, S *sq)
{
    const uint32_t tid = threadIdx.x, nf = faces_along(B, 0), row = nf + 5, lines = (uint32_t)B.nj * (uint32_t)B.nk;
    const int sh = B.off[0] ? 1 : 0;
    const uint32_t faces = line_faces(nf), F0 = lt * faces, count = min(faces, nf * lines - F0);
    const uint32_t l0 = F0 / nf, f0 = F0 - l0 * nf;               // first line, and its first face here
    const uint32_t last = (f0 + count - 1) / nf;                  // lines after it
    const uint32_t points = last * row + (f0 + count - 1 - last * nf) + 6 - f0;
    const int j0 = (int)(l0 % (uint32_t)B.nj), k0 = (int)(l0 / (uint32_t)B.nj);
    // item x of len to a line, counted from the first line: lines after it (into s) and the item of that line. Past
    // the first line x is below LINE_POINTS, where the product with the reciprocal is exact.
    auto split = [](uint32_t &x, uint32_t len, float inv) -> uint32_t {
        if (x < len) return 0;
        x -= len;
        const uint32_t s = (uint32_t)(((float)x + 0.5f) * inv);
        x -= s * len;
        return s + 1;
    };
    auto node = [&](uint32_t s, int i) -> uint32_t {
        int j = j0 + (int)s, k = k0;
        while (j >= B.nj) { j -= B.nj; ++k; }
        return node_index(B, i, j, k);
    };
    const float inv_row = 1.0f / (float)row, inv_nf = 1.0f / (float)nf;

    __syncthreads();   // the previous tile's LDS fully consumed
    for (uint32_t p = tid; p < points; p += 256) {
        uint32_t x = f0 + p;
        const uint32_t s = split(x, row, inv_row);
        stage_point<S, 0>(B, node(s, along_shift(B, 0, (int)x - sh, -2, B.ni)), [&](int v, S y) { sq[v * LINE_POINTS + p] = y; });
    }
    __syncthreads();

    if (tid < count) {
        uint32_t f = f0 + tid;
        const uint32_t s = split(f, nf, inv_nf), p = s * row + f - f0;
        face_at<S, 0>(B, node(s, (int)f - sh), [&](int m, int v) { return sq[v * LINE_POINTS + p + m]; });
    }
}

// Tile lt of the sweep along DIR: variant 0 of the i sweep is a line tile, every other a rectangular one.
template <int DIR, int TA, int TB>
constexpr bool LINE_TILE = DIR == 0 && TA == FACE_I_TILES[0][0] && TB == FACE_I_TILES[0][1];
template <typename S, int DIR, int TA, int TB>
constexpr int SWEEP_LDS = LINE_TILE<DIR, TA, TB> ? POINT_VALUES<S> *LINE_POINTS : FACE_LDS<S, TA, TB>;
template <typename S, int DIR, int TA, int TB>
__device__ __forceinline__ void sweep_tile(const BlockDev &B, uint32_t lt, S *lds)
{
    if constexpr (LINE_TILE<DIR, TA, TB>) line_tile<S>(B, lt, lds);
    else face_tile<S, DIR, TA, TB>(B, lt, lds);
}

template <typename S, int DIR, int TA, int TB, bool LOOP>
__global__ void __launch_bounds__(256, (TA == 64 ? 3 : 4)) k_face(const BlockDev *__restrict__ blks, const uint32_t *__restrict__ prefix,
                                              uint32_t nblk, uint32_t total)
{
    __shared__ S lds[SWEEP_LDS<S, DIR, TA, TB>];
    auto tile = [&](uint32_t wg) {
        const uint32_t t = xcd_tile(wg, total);
        const BlockDev &B = blks[find_block(prefix, nblk, t)];
        sweep_tile<S, DIR, TA, TB>(B, t - B.tile0[1 + DIR], lds);
    };
    each_tile<LOOP>(total, tile);
}

// The viscous node tiles and the three face sweeps of a stage in one launch (tile variants 0). They
// depend on nothing of each other, and apart each launch ends with a tail and a gap. Untimed steps of the same build, apart
// and together, us, FP64: 64^3 213 and 176, 96^3 766 and 686, 128^3 1615 and 1548, 160^3 3153 and 3088, 256^3 12745 and
// 12880, 320^3 25227 and 25608; mixed: 146 and 111, 407 and 354, 938 and 872, 1809 and 1776, 7234 and 7206, 14009 and
// 14136: from 256^3 on it no longer pays, by 1 to 1.5 % in FP64. At 256^3 it takes 2.9 ms FP64 and 1.6 mixed, moves 11.0
// and 5.9 GB through the L2 (its kinds apart 11.2 and 6.1) and issues 8.6e8 and 7.9e8 wave instructions: FP64 62 % of the
// issue slots at the 1.9 GHz that the card's power limit leaves, 3.8 TB/s; mixed all of them (an FP32 instruction takes
// an issue slot like an FP64 one). Each XCD takes its own contiguous share of every kind of tile and runs through them
// FLUX_CHUNK tiles of a kind at a time: with the kinds alternating tile by tile they fall into step
// with the CUs (each CU draws tiles of one kind; 256^3 8 % slower in FP64, 23 % mixed), 4 and 16 are
// best, a kind's whole share at a time 1 % slower at 256^3 FP64 and 3 % at 128^3 mixed.
constexpr uint32_t FLUX_CHUNK = 16;
struct FluxTotals {
    const uint32_t *prefix[4];
    uint32_t total[4];   // tiles of the node kernel and of the i, j, k sweeps
    uint32_t chunk;      // tiles of a kind that an XCD takes at a time
};

template <typename S, bool VISC, int K>
__global__ void __launch_bounds__(256, 4) k_flux(const BlockDev *__restrict__ blks, FluxTotals T, uint32_t nblk, int mode,
                                                 uint32_t shell_tiles)
{
    constexpr int IA = FACE_I_TILES[0][0], IB = FACE_I_TILES[0][1], JA = FACE_JK_TILES[0][0], JB = FACE_JK_TILES[0][1];
    constexpr int TX = NODE_TILES[0][0], TY = NODE_TILES[0][1];
    constexpr int L0 = VISC ? VISC_LDS<TX, TY> * (int)sizeof(double) : 0, L1 = SWEEP_LDS<S, 0, IA, IB> * (int)sizeof(S),
                  L2 = FACE_LDS<S, JA, JB> * (int)sizeof(S);
    __shared__ __align__(16) char lds[L0 > L1 ? (L0 > L2 ? L0 : L2) : (L1 > L2 ? L1 : L2)];
    constexpr bool BND = list_bounded(K);
    constexpr uint32_t KINDS = VISC ? 4 : 3;
    uint32_t wg = blockIdx.x;
    if (VISC && BND) {
        // the shell tiles first (a multiple of 8 workgroups, so that the others keep their XCDs): their long
        // chains would otherwise be the tail of the launch
        const uint32_t shell = nblk * shell_tiles, first = (shell + 7) & ~7u;
        if (wg < shell) visc_shell_tile<S>(blks, wg, mode, shell_tiles);
        if (wg < first) return;
        wg -= first;
    }
    const uint32_t x = wg & 7u, l = wg >> 3, kind = (l % (KINDS * T.chunk)) / T.chunk + (4 - KINDS),
                   r = (l / (KINDS * T.chunk)) * T.chunk + l % T.chunk;
    const uint32_t total = T.total[kind], q = total >> 3, rem = total & 7u;
    if (r >= q + (x < rem ? 1u : 0u)) return;
    const uint32_t t = x * q + (x < rem ? x : rem) + r;
    const BlockDev &B = blks[find_block(T.prefix[kind], nblk, t)];
    const uint32_t lt = t - B.tile0[kind];
    if (kind == 0) {
        if (B.viscous) visc_tile<S, TX, TY, K>(B, lt, mode, (double *)lds);
    } else if (kind == 1) {
        sweep_tile<S, 0, IA, IB>(B, lt, (S *)lds);
    } else if (kind == 2) {
        sweep_tile<S, 1, JA, JB>(B, lt, (S *)lds);
    } else {
        sweep_tile<S, 2, JA, JB>(B, lt, (S *)lds);
    }
}

// ---------------------------------------------------------------------------
// update kernel: L and the SSP-RK3 stage (Weno.cl:3060-3135), in double. Bound by memory: 256^3 FP64 1.41 ms, 7.0
// GB (6.4 with every value once), 5.0 TB/s; mixed 0.81 ms, 4.3 GB, 5.3 TB/s (a copy of 4 GiB: 4.7).
//   mode 0..2: RK stage j; mode 3: write L only, to Lout (owned order, component-major)
// ---------------------------------------------------------------------------
// L and the SSP-RK3 stage of one node; mdu / mdv / mde: the node's monitor values (mode 2 with
// the monitor on). LOC as in visc_node.
template <typename S, bool LOC, bool NT>
__device__ __forceinline__ void update_node(const BlockDev &B, int i, int j, int k, int mode, double *Lout, double &mdu,
                                            double &mdv, double &mde)
{
    const uint32_t g = node_index(B, i, j, k);
    double L[5] = {0, 0, 0, 0, 0};
#pragma unroll
    for (int d = 0; d < 3; ++d) {
        const uint32_t m1 = shifted(B, i, j, k, d, -1);
#pragma unroll
        for (int c = 0; c < 5; ++c) {
            const S *fh = (const S *)B.FH[d][c];
            L[c] += (double)ld(fh, g) - (double)ld(fh, m1);
        }
    }
    if (B.viscous) {
        if constexpr (LOC) {
            // bounded block: the loc-selected forms of Weno.cl:2732-2856
            LocForm form[3];
            loc_forms(B, i, j, k, true, form);
            // across a wake cut the row -m of column i is the row m of column ni - 1 - i, where eta runs the
            // other way: its flux along j, negated
            const bool cut = B.bc[2] == CFDX_BC_WALL_CUT && !(i >= B.cut_i0 && i <= B.cut_i1);
#pragma unroll
            for (int d = 0; d < 3; ++d) {
                uint32_t x[4];
                bool across[4];
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    const int o = form[d].o[q];
                    across[q] = d == 1 && cut && j + o < 0;
                    x[q] = across[q] ? node_index(B, B.ni - 1 - i, -(j + o), k) : shifted(B, i, j, k, d, o);
                }
#pragma unroll
                for (int c = 1; c < 5; ++c) {
                    const S *f = (const S *)B.Fv[d][c - 1];
                    double y[4];
#pragma unroll
                    for (int q = 0; q < 4; ++q) {
                        y[q] = (double)ld(f, x[q]);
                        y[q] = across[q] ? -y[q] : y[q];
                    }
                    L[c] += form[d].of(y);
                }
            }
        } else {
#pragma unroll
            for (int d = 0; d < 3; ++d) {
                const uint32_t m2 = shifted(B, i, j, k, d, -2), m1 = shifted(B, i, j, k, d, -1);
                const uint32_t p1 = shifted(B, i, j, k, d, 1), p2 = shifted(B, i, j, k, d, 2);
#pragma unroll
                for (int c = 1; c < 5; ++c) {
                    const S *f = (const S *)B.Fv[d][c - 1];
                    L[c] += (1.0 / 12.0) * (8.0 * ((double)ld(f, p1) - (double)ld(f, m1)) - ((double)ld(f, p2) - (double)ld(f, m2)));
                }
            }
        }
    }
#pragma unroll
    for (int c = 0; c < 5; ++c) L[c] = -L[c];
    if (mode == 3) {
        const size_t no = (size_t)B.ni * B.nj * B.nk, o = (size_t)i + (size_t)B.ni * ((size_t)j + (size_t)B.nj * k);
#pragma unroll
        for (int c = 0; c < 5; ++c) Lout[c * no + o] = L[c];
    } else {
        const double del_t = B.del_t;
        double un[5], u0[5];
#pragma unroll
        for (int c = 0; c < 5; ++c) u0[c] = ldx<NT>(B.U0[c], g);
        if (mode == 0) {
#pragma unroll
            for (int c = 0; c < 5; ++c) { un[c] = u0[c] + del_t * L[c]; stx<NT>(B.Us[c], g, un[c]); }
        } else if (mode == 1) {
#pragma unroll
            for (int c = 0; c < 5; ++c) { un[c] = 0.75 * u0[c] + 0.25 * ldx<NT>(B.Us[c], g) + 0.25 * del_t * L[c]; stx<NT>(B.Us[c], g, un[c]); }
        } else {
#pragma unroll
            for (int c = 0; c < 5; ++c) un[c] = (u0[c] * (1.0 / 3.0)) + ((2.0 / 3.0) * ldx<NT>(B.Us[c], g)) + (2.0 / 3.0) * (del_t * L[c]);
        }
        const double det = ldx<NT>(B.det, g);
        const double idet = 1.0 / det;
        const double rho = idet * un[0], ir = 1.0 / rho;
        const double u = (idet * un[1]) * ir, v = (idet * un[2]) * ir, w = (idet * un[3]) * ir;
        const double e = (idet * un[4]) * ir - 0.5 * (u * u + v * v + w * w);
        const double p = e * rho * 0.4;
        stx<NT>((S *)B.P[0], g, S(rho)); stx<NT>((S *)B.P[1], g, S(u)); stx<NT>((S *)B.P[2], g, S(v)); stx<NT>((S *)B.P[3], g, S(w)); stx<NT>((S *)B.P[4], g, S(p));
        if (mode == 2) {
            // next step's RK base: U_Q recomputes det*Q from the new primitives (Solver.cpp:377-388)
            double q[5];
            prim_to_q(rho, u, v, w, p, q);
#pragma unroll
            for (int c = 0; c < 5; ++c) stx<NT>(B.U0[c], g, det * q[c]);
            if (B.mon) {
                const double r0 = idet * u0[0], ir0 = 1.0 / r0;
                const double uo = (idet * u0[1]) * ir0, vo = (idet * u0[2]) * ir0, wo = (idet * u0[3]) * ir0;
                const double eo = (idet * u0[4]) * ir0 - 0.5 * (uo * uo + vo * vo + wo * wo);
                mdu = fabs(u - uo); mdv = fabs(v - vo); mde = fabs(e - eo);
            }
        }
    }
}

// one maximum per wave of the monitor values (every lane takes part), written by lane 0 at slot
__device__ __forceinline__ void monitor_wave(const BlockDev &B, uint32_t slot, double mdu, double mdv, double mde)
{
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
        mdu = fmax(mdu, __shfl_xor(mdu, o));
        mdv = fmax(mdv, __shfl_xor(mdv, o));
        mde = fmax(mde, __shfl_xor(mde, o));
    }
    if ((threadIdx.x & 63) == 0) {
        double *m = B.mon + 3 * (size_t)slot;
        m[0] = mdu; m[1] = mdv; m[2] = mde;
    }
}

// tiles as in k_visc; the shell tiles' monitor slots follow the block's node tiles' (tiles x
// waves per tile)
template <typename S, int TX, int TY, int K, bool LOOP>
__global__ void __launch_bounds__(TX *TY) k_update(const BlockDev *__restrict__ blks, const uint32_t *__restrict__ prefix,
                                                   uint32_t nblk, uint32_t total, int mode, uint32_t shell_tiles,
                                                   double *Lout)
{
    constexpr bool BND = list_bounded(K), NT = list_streams(K);
    const uint32_t shell = BND ? nblk * shell_tiles : 0u, first = (shell + 7) & ~7u, all = first + total;
    auto tile = [&](uint32_t wg) {
        // residual monitor of the step (Solver.cpp:546-573): |du|, |dv|, |de| against the RK base
        double mdu = 0.0, mdv = 0.0, mde = 0.0;
        if (BND && wg < first) {   // the shell tiles first, as in k_flux
            if (wg >= shell) return;
            const BlockDev &B = blks[wg / shell_tiles];
            const uint32_t s = wg % shell_tiles;
            if (!B.code || s >= shell_tile_count(B)) return;
            int i, j, k;
            if (shell_node(B, s, i, j, k)) update_node<S, true, false>(B, i, j, k, mode, Lout, mdu, mdv, mde);
            if (mode == 2 && B.mon && threadIdx.x < (s < shell_row_tiles(B) ? SHELL_TILE : shell_column_tile(B))) {
                const uint32_t main_slots = ((B.ni + TX - 1) / TX) * ((B.nj + TY - 1) / TY) * B.nk * (uint32_t)(TX * TY / 64);
                monitor_wave(B, main_slots + shell_wave(B, s, threadIdx.x / 64), mdu, mdv, mde);
            }
            return;
        }
        const uint32_t t = xcd_tile(wg - first, total);
        const BlockDev &B = blks[find_block(prefix, nblk, t)];
        const uint32_t lt = t - B.tile0[0];
        int i0, j0, k;
        node_tile(B, lt, TX, TY, i0, j0, k);
        const int i = i0 + (int)(threadIdx.x % TX), j = j0 + (int)(threadIdx.x / TX);
        if (i < B.ni && j < B.nj && !(BND && B.code && in_shell(B, i, j, k)))
            update_node<S, false, NT>(B, i, j, k, mode, Lout, mdu, mdv, mde);
        if (mode == 2 && B.mon) monitor_wave(B, lt * (TX * TY / 64) + threadIdx.x / 64, mdu, mdv, mde);
    };
    each_tile<LOOP>(all, tile);
}

// maxima over the per-wave monitor values: out[0..2] = max |du|, |dv|, |de|; one workgroup, four triples of
// each thread in flight (bound by memory latency)
constexpr int MON_THREADS = 1024;
__global__ void __launch_bounds__(MON_THREADS) k_mon_reduce(const double *__restrict__ mon, uint32_t count, double *__restrict__ out)
{
    __shared__ double sh[3][MON_THREADS / 64];
    double m[3] = {0.0, 0.0, 0.0};
#pragma unroll 4
    for (uint32_t q = threadIdx.x; q < count; q += MON_THREADS) {
#pragma unroll
        for (int r = 0; r < 3; ++r) m[r] = fmax(m[r], mon[3 * (size_t)q + r]);
    }
#pragma unroll
    for (int r = 0; r < 3; ++r) {
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) m[r] = fmax(m[r], __shfl_xor(m[r], o));
        if ((threadIdx.x & 63) == 0) sh[r][threadIdx.x / 64] = m[r];
    }
    __syncthreads();
    if (threadIdx.x < 3) {
        double x = 0.0;
        for (int w = 0; w < MON_THREADS / 64; ++w) x = fmax(x, sh[threadIdx.x][w]);
        out[threadIdx.x] = x;
    }
}

// owned node o (i-fastest over ni x nj x nk) -> stored index
__device__ __forceinline__ uint32_t owned_node(const BlockDev &B, uint32_t o)
{
    const int i = (int)(o % (uint32_t)B.ni), j = (int)((o / (uint32_t)B.ni) % (uint32_t)B.nj), k = (int)(o / ((uint32_t)B.ni * B.nj));
    return node_index(B, i, j, k);
}

__device__ __forceinline__ uint32_t owned_count(const BlockDev &B) { return (uint32_t)B.ni * B.nj * B.nk; }

// set_flow: double primitives staged component-major in owned order (stage[c * n_owned + o]) ->
// P (type S) and U0 = det * Q(P) in double
template <typename S>
__global__ void k_base(BlockDev B, const double *__restrict__ stage)
{
    const uint32_t o = blockIdx.x * blockDim.x + threadIdx.x, no = owned_count(B);
    if (o >= no) return;
    const uint32_t g = owned_node(B, o);
    const double rho = stage[o], u = stage[no + o], v = stage[2 * (size_t)no + o], w = stage[3 * (size_t)no + o],
                 p = stage[4 * (size_t)no + o];
    double q[5];
    prim_to_q(rho, u, v, w, p, q);
    const double det = ld(B.det, g);
#pragma unroll
    for (int c = 0; c < 5; ++c) st(B.U0[c], g, det * q[c]);
    st((S *)B.P[0], g, S(rho)); st((S *)B.P[1], g, S(u)); st((S *)B.P[2], g, S(v)); st((S *)B.P[3], g, S(w)); st((S *)B.P[4], g, S(p));
}

// get_flow of the mixed form: primitives from the double RK base U0 / det, owned order
__global__ void k_prims(BlockDev B, double *__restrict__ out)
{
    const uint32_t o = blockIdx.x * blockDim.x + threadIdx.x, no = owned_count(B);
    if (o >= no) return;
    const uint32_t g = owned_node(B, o);
    const double idet = 1.0 / ld(B.det, g);
    const double rho = idet * ld(B.U0[0], g), ir = 1.0 / rho;
    const double u = (idet * ld(B.U0[1], g)) * ir, v = (idet * ld(B.U0[2], g)) * ir, w = (idet * ld(B.U0[3], g)) * ir;
    const double e = (idet * ld(B.U0[4], g)) * ir - 0.5 * (u * u + v * v + w * w);
    out[o] = rho; out[no + o] = u; out[2 * (size_t)no + o] = v; out[3 * (size_t)no + o] = w; out[4 * (size_t)no + o] = e * rho * 0.4;
}

// get_flow of the plain form: the primitives of the last stage, owned order
__global__ void k_copy_prims(BlockDev B, double *__restrict__ out)
{
    const uint32_t o = blockIdx.x * blockDim.x + threadIdx.x, no = owned_count(B);
    if (o >= no) return;
    const uint32_t g = owned_node(B, o);
#pragma unroll
    for (int c = 0; c < 5; ++c) out[(size_t)c * no + o] = ld((const double *)B.P[c], g);
}

// ---------------------------------------------------------------------------
// side conditions of bounded blocks (Flow_Initialisation.cpp face rules; the C-grid wake cut)
// ---------------------------------------------------------------------------
template <typename S>
__device__ __forceinline__ void get_prim(const BlockDev &B, uint32_t g, double (&w)[5])
{
#pragma unroll
    for (int c = 0; c < 5; ++c) w[c] = (double)ld((const S *)B.P[c], g);
}

// primitives of a boundary or ghost node; its RK base (mode 2) or stage vector (modes 0, 1)
// follows from them, as U_Q rebuilds U from FLOW (ghost stage vectors are not defined by the
// reference at stages 1 and 2; here they are det * Q of the side condition's state). The
// primitives are rounded to S first, as if read back from the stored arrays.
template <typename S>
__device__ __forceinline__ void put_node(const BlockDev &B, uint32_t g, const double (&w)[5], int mode, bool ghost)
{
    double r[5];
#pragma unroll
    for (int c = 0; c < 5; ++c) r[c] = (double)S(w[c]);
    const bool u = mode == 2 || ghost;
    const double det = u ? ld(B.det, g) : 0.0;
#pragma unroll
    for (int c = 0; c < 5; ++c) st((S *)B.P[c], g, S(w[c]));
    if (!u) return;
    double q[5];
    prim_to_q(r[0], r[1], r[2], r[3], r[4], q);
#pragma unroll
    for (int c = 0; c < 5; ++c) st(mode == 2 ? B.U0[c] : B.Us[c], g, det * q[c]);
}

// the node across a wake cut into a ghost or duplicate node: primitives copied, the stage vector
// and RK base carry the same Q with the destination's own det (U = det Q). Every value is loaded
// before the first store.
template <typename S>
__device__ __forceinline__ void copy_node(const BlockDev &B, uint32_t dst, uint32_t src)
{
    const double ratio = ld(B.det, dst) / ld(B.det, src);
    S p[5];
    double us[5], u0[5];
#pragma unroll
    for (int c = 0; c < 5; ++c) {
        p[c] = ld((const S *)B.P[c], src);
        us[c] = ld(B.Us[c], src);
        u0[c] = ld(B.U0[c], src);
    }
#pragma unroll
    for (int c = 0; c < 5; ++c) {
        st((S *)B.P[c], dst, p[c]);
        st(B.Us[c], dst, us[c] * ratio);
        st(B.U0[c], dst, u0[c] * ratio);
    }
}

// One node of side hi (0: low, 1: high) of direction d: face node (a, bq) and layer m (0: the boundary
// node, 1..3: the ghost layers). The nodes a side
// writes are its boundary nodes and ghost layers; it reads the first owned layers in from its
// side (a bounded direction has >= 7 nodes), so the two sides of a direction are independent and
// the directions run one after the other (i, then j, then k: a node on two sides ends with the
// later direction's value).
template <typename S>
__device__ __forceinline__ void bc_node(const BlockDev &B, int d, int hi, int a, int bq, int m, int mode)
{
    const int side = 2 * d + hi;
    const int n = d == 0 ? B.ni : d == 1 ? B.nj : B.nk;
    auto at = [&](int c) -> uint32_t {
        if (d == 0) return node_index(B, c, a, bq);
        if (d == 1) return node_index(B, a, c, bq);
        return node_index(B, a, bq, c);
    };
    const int c0 = hi ? n - 1 : 0, in = hi ? -1 : 1;   // boundary node; step into the block
    int kind = B.bc[side];
    if (kind == CFDX_BC_WALL_CUT) {
        if (a >= B.cut_i0 && a <= B.cut_i1) {
            kind = CFDX_BC_WALL;
        } else {
            // wake cut (j- side, a = i): node (i, -m) is node (ni-1-i, m); row 0 of the lower half
            // copies the upper half
            const int im = B.ni - 1 - a;
            if (m > 0) copy_node<S>(B, node_index(B, a, -m, bq), node_index(B, im, m, bq));
            else if (a < im) copy_node<S>(B, node_index(B, a, 0, bq), node_index(B, im, 0, bq));
            return;
        }
    }
    const double M2 = 1.4 * B.mach * B.mach;
    double w[5];
    if (kind == CFDX_BC_WALL || kind == CFDX_BC_EXTRAP) {
        get_prim<S>(B, at(c0 + in * (m ? m : 1)), w);
        if (m == 0) {
            if (kind == CFDX_BC_WALL) {
                const double t1 = M2 * (w[4] / w[0]);
                w[0] = M2 * (w[4] / t1); w[1] = 0.0; w[2] = 0.0; w[3] = 0.0;
            }
        } else if (kind == CFDX_BC_WALL) {
            w[1] = -w[1]; w[2] = -w[2]; w[3] = -w[3];
        }
    } else if (kind == CFDX_BC_FARFIELD) {
        const double p = 1.0 / M2;
        w[0] = M2 * (p / 1.0); w[1] = B.cos_aoa; w[2] = B.sin_aoa; w[3] = 0.0; w[4] = p;
    } else {   // CFDX_BC_OUTFLOW
        get_prim<S>(B, at(c0 + in), w);
        const double t1 = M2 * (w[4] / w[0]);
        w[0] = M2 * (w[4] / t1);
    }
    put_node<S>(B, at(c0 - in * m), w, mode, m > 0);
}

// One direction's two sides (blockIdx.z), one thread per node of a side's face and layer.
template <typename S>
__global__ void __launch_bounds__(256) k_bc(const BlockDev *__restrict__ blks, int d, int mode)
{
    const BlockDev &B = blks[blockIdx.y];
    if (!B.off[d]) return;
    const int na = d == 0 ? B.nj : B.ni, nb = d == 2 ? B.nj : B.nk;
    const uint32_t nf = (uint32_t)na * (uint32_t)nb;
    const uint32_t t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= 4 * nf) return;
    // i sides: the four layers of a face node are adjacent in memory, so they go to four adjacent
    // threads; j and k sides: adjacent threads take adjacent i of one layer
    const int m = d == 0 ? (int)(t & 3u) : (int)(t / nf);
    const uint32_t r = d == 0 ? t >> 2 : t - (uint32_t)m * nf;
    bc_node<S>(B, d, (int)blockIdx.z, (int)(r % (uint32_t)na), (int)(r / (uint32_t)na), m, mode);
}

// The side conditions of the i and j directions of blocks bounded in either, in one launch: i first, then
// j, as k_bc one after the other. Workgroups 0 .. planes - 1 take the two i sides of a k plane each and,
// after them, the j sides of the four columns at either end, the only ones that read what the i sides
// wrote or write what they read; the other workgroups take the j sides of the columns between. 384x128x32: 15.6 us,
// where two launches of 7.2 us each were: a plane's workgroup does its i sides and then its end columns, so the launch
// saves the gap between two and no kernel time.
constexpr int BC_IJ = 512, BC_END = 4;
template <typename S>
__global__ void __launch_bounds__(BC_IJ) k_bc_ij(const BlockDev *__restrict__ blks, uint32_t planes, int mode)
{
    const BlockDev &B = blks[blockIdx.y];
    const int ni = B.ni, nj = B.nj, nk = B.nk;
    if (blockIdx.x < planes) {
        const int k = (int)blockIdx.x;
        if (!B.off[0] || k >= nk) return;
        // the four layers of a face node are adjacent in memory, so they go to four adjacent threads
        for (int t = (int)threadIdx.x; t < 8 * nj; t += BC_IJ) bc_node<S>(B, 0, (t >> 2) >= nj, (t >> 2) % nj, k, t & 3, mode);
        if (!B.off[1]) return;
        __syncthreads();
        const int cols = min(2 * BC_END, ni);
        for (int t = (int)threadIdx.x; t < 8 * cols; t += BC_IJ) {
            const int c = t % cols, r = t / cols;
            bc_node<S>(B, 1, r >> 2, c < BC_END ? c : ni - cols + c, k, r & 3, mode);
        }
        return;
    }
    if (!B.off[1]) return;
    const uint32_t first = B.off[0] ? BC_END : 0, cols = B.off[0] ? (uint32_t)max(ni - 2 * BC_END, 0) : (uint32_t)ni;
    const uint32_t t = (blockIdx.x - planes) * BC_IJ + threadIdx.x;
    if (t >= 8 * cols * (uint32_t)nk) return;
    const uint32_t c = t % cols, r = t / cols;
    bc_node<S>(B, 1, (int)((r / (uint32_t)nk) >> 2), (int)(first + c), (int)(r % (uint32_t)nk), (int)((r / (uint32_t)nk) & 3u), mode);
}

// The kernels launched.
template <typename S>
int launch_bc(const LaunchList &L, int mode, hipStream_t st)
{
    int n = 0;
    const bool ij = L.bc_face_d[0] && L.bc_face_d[1];
    if (ij) {
        const uint32_t js = (8 * L.bc_face_d[1] + BC_IJ - 1) / BC_IJ;
        hipLaunchKernelGGL(k_bc_ij<S>, dim3(L.bc_planes + js, L.nblk), dim3(BC_IJ), 0, st, L.blks, L.bc_planes, mode);
        ++n;
    }
    for (int d = ij ? 2 : 0; d < 3; ++d)
        if (L.bc_face_d[d]) {
            hipLaunchKernelGGL(k_bc<S>, dim3((4 * L.bc_face_d[d] + 255) / 256, L.nblk, 2), dim3(256), 0, st, L.blks, d, mode);
            ++n;
        }
    return n;
}

// ---------------------------------------------------------------------------
// host launchers
// ---------------------------------------------------------------------------
template <typename S, int DIR, int TA, int TB>
void launch_face(const LaunchList &L, hipStream_t st)
{
    const uint32_t n = L.total[1 + DIR];
    if (L.grid_cap && L.grid_cap < n)
        hipLaunchKernelGGL((k_face<S, DIR, TA, TB, true>), dim3(L.grid_cap), dim3(256), 0, st, L.blks, L.prefix[1 + DIR], L.nblk, n);
    else
        hipLaunchKernelGGL((k_face<S, DIR, TA, TB, false>), dim3(n), dim3(256), 0, st, L.blks, L.prefix[1 + DIR], L.nblk, n);
}
// cap: workgroups of the launch (0: one per tile)
template <typename S, int V, int K>
void launch_node_k(const LaunchList &L, uint32_t cap, hipStream_t st, bool visc_kernel, int mode)
{
    constexpr int TX = NODE_TILES[V][0], TY = NODE_TILES[V][1];
    static_assert(TX * TY == 256, "node tiles have 256 threads");
    const uint32_t shell_tiles = list_bounded(K) ? L.shell_tiles : 0u;
    // one workgroup per shell tile too
    const uint32_t shell = L.nblk * shell_tiles, all = L.total[0] + (visc_kernel ? shell : (shell + 7) & ~7u);
    const bool loop = cap && cap < all;
    auto go = [&](auto kernel, auto... out) {
        hipLaunchKernelGGL(kernel, dim3(loop ? cap : all), dim3(TX * TY), 0, st, L.blks, L.prefix[0], L.nblk, L.total[0], mode,
                           shell_tiles, out...);
    };
    if (visc_kernel && loop) go(k_visc<S, TX, TY, K, true>);
    else if (visc_kernel) go(k_visc<S, TX, TY, K, false>);
    else if (loop) go(k_update<S, TX, TY, K, true>, L.Lout);
    else go(k_update<S, TX, TY, K, false>, L.Lout);
}
// lists without bounded blocks run the node kernels without the loc-code branches
template <typename S, int V>
void launch_node(const LaunchList &L, uint32_t cap, hipStream_t st, bool visc_kernel, int mode)
{
    if (L.bc_face && L.stream) launch_node_k<S, V, LIST_BOUNDED_STREAM>(L, cap, st, visc_kernel, mode);
    else if (L.bc_face) launch_node_k<S, V, LIST_BOUNDED>(L, cap, st, visc_kernel, mode);
    else if (L.stream) launch_node_k<S, V, LIST_STREAM>(L, cap, st, visc_kernel, mode);
    else launch_node_k<S, V, LIST_PLAIN>(L, cap, st, visc_kernel, mode);
}

template <typename S>
void node_kernel(const LaunchList &L, uint32_t cap, hipStream_t st, bool visc_kernel, int mode)
{
    switch (L.tiles.node) {
    case 1: launch_node<S, 1>(L, cap, st, visc_kernel, mode); break;
    case 2: launch_node<S, 2>(L, cap, st, visc_kernel, mode); break;
    case 3: launch_node<S, 3>(L, cap, st, visc_kernel, mode); break;
    default: launch_node<S, 0>(L, cap, st, visc_kernel, mode);
    }
}

template <typename S>
void face_i(const LaunchList &L, hipStream_t st)
{
    constexpr auto &T = FACE_I_TILES;
    switch (L.tiles.face[0]) {
    case 1: launch_face<S, 0, T[1][0], T[1][1]>(L, st); break;
    case 2: launch_face<S, 0, T[2][0], T[2][1]>(L, st); break;
    default: launch_face<S, 0, T[0][0], T[0][1]>(L, st);
    }
}

template <typename S, int DIR>
void face_jk(const LaunchList &L, hipStream_t st)
{
    constexpr auto &T = FACE_JK_TILES;
    switch (L.tiles.face[DIR]) {
    case 1: launch_face<S, DIR, T[1][0], T[1][1]>(L, st); break;
    case 2: launch_face<S, DIR, T[2][0], T[2][1]>(L, st); break;
    case 3: launch_face<S, DIR, T[3][0], T[3][1]>(L, st); break;
    default: launch_face<S, DIR, T[0][0], T[0][1]>(L, st);
    }
}

// The grid of k_flux over a list: every kind's tiles per XCD rounded up to the same whole number of chunks. A
// launch holds fewer than 2^32 threads; lists past that (thin blocks of tens of millions of nodes, whose
// tiles of 256 points are nearly empty) run the kernels apart.
constexpr uint64_t MAX_GRID = ((uint64_t)1 << 32) / 256 - 1;
struct FluxGrid {
    uint32_t chunk, shell_tiles;
    uint64_t wgs;
};
FluxGrid flux_grid(const LaunchList &L, bool any_visc)
{
    uint32_t most = 0;
    for (int q = any_visc ? 0 : 1; q < 4; ++q) most = std::max(most, L.total[q]);
    FluxGrid g;
    const uint32_t share = most / 8 + (most % 8 != 0);
    g.chunk = std::max(std::min(FLUX_CHUNK, share), 1u);
    const uint64_t slots = (uint64_t)(share + g.chunk - 1) / g.chunk * g.chunk;
    g.shell_tiles = L.bc_face && any_visc ? L.shell_tiles : 0u;
    g.wgs = (uint64_t)8 * (any_visc ? 4 : 3) * slots + (((uint64_t)L.nblk * g.shell_tiles + 7) & ~(uint64_t)7);
    return g;
}

bool stage_forks(const LaunchList &L, const Overlap *ov)
{
    const TileCfg &t = L.tiles;
    return ov && (L.grid_cap || t.face[0] || t.face[1] || t.face[2] || t.node || flux_grid(L, true).wgs > MAX_GRID);
}

template <typename S>
void launch_flux(const LaunchList &L, int mode, hipStream_t st, bool any_visc)
{
    const FluxGrid fg = flux_grid(L, any_visc);
    FluxTotals T;
    for (int q = 0; q < 4; ++q) {
        T.prefix[q] = L.prefix[q];
        T.total[q] = L.total[q];
    }
    T.chunk = fg.chunk;
    const dim3 g((uint32_t)fg.wgs);
    auto go = [&](auto kernel) { hipLaunchKernelGGL(kernel, g, dim3(256), 0, st, L.blks, T, L.nblk, mode, fg.shell_tiles); };
    if (!any_visc) go(k_flux<S, false, LIST_PLAIN>);   // the sweeps alone take the blocks' own switch
    else if (L.bc_face && L.stream) go(k_flux<S, true, LIST_BOUNDED_STREAM>);
    else if (L.bc_face) go(k_flux<S, true, LIST_BOUNDED>);
    else if (L.stream) go(k_flux<S, true, LIST_STREAM>);
    else go(k_flux<S, true, LIST_PLAIN>);
}

template <typename S>
int launch_stage(const LaunchList &L, int mode, hipStream_t st, bool any_visc, hipEvent_t *ev, const Overlap *ov)
{
    auto rec = [&](int s) { if (ev) (void)hipEventRecord(ev[s], st); };
    rec(0);
    // the viscous node kernel reads the stage vector, primitives and geometry and writes Fv and mu;
    // the face sweeps read the primitives and geometry and write F-hat: independent until the update
    const bool overlap = ov && !ev, together = overlap && !stage_forks(L, ov);
    int n = together ? 2 : any_visc ? 5 : 4;   // kernels launched
    hipStream_t vs = st;
    if (together) {
        launch_flux<S>(L, mode, st, any_visc);
    } else if (any_visc) {
        if (overlap) {
            // other tile shapes or a capped grid: beside the sweeps on the second stream
            (void)hipEventRecord(ov->fork, st);
            (void)hipStreamWaitEvent(ov->aux, ov->fork, 0);
            vs = ov->aux;
        }
        node_kernel<S>(L, L.grid_cap, vs, true, mode);
    }
    if (vs != st) (void)hipEventRecord(ov->join, vs);
    rec(1);
    if (!together) face_i<S>(L, st);
    rec(2);
    if (!together) face_jk<S, 1>(L, st);
    rec(3);
    if (!together) face_jk<S, 2>(L, st);
    rec(4);
    if (vs != st) (void)hipStreamWaitEvent(st, ov->join, 0);
    node_kernel<S>(L, L.grid_cap, st, false, mode);
    if (L.bc_face && mode <= 2) n += launch_bc<S>(L, mode, st);
    rec(5);
    return n;
}

int stage(const LaunchList &L, int precision, int mode, hipStream_t st, bool any_visc, hipEvent_t *ev, const Overlap *ov)
{
    return precision == CFDX_MIXED ? launch_stage<float>(L, mode, st, any_visc, ev, ov)
                                   : launch_stage<double>(L, mode, st, any_visc, ev, ov);
}

void base(const BlockDev &B, int precision, hipStream_t st, const double *stage)
{
    const unsigned nb = (unsigned)(((uint32_t)B.ni * B.nj * B.nk + 255) / 256);
    if (precision == CFDX_MIXED) hipLaunchKernelGGL(k_base<float>, dim3(nb), dim3(256), 0, st, B, stage);
    else hipLaunchKernelGGL(k_base<double>, dim3(nb), dim3(256), 0, st, B, stage);
}

void boundary(const LaunchList &L, int precision, int mode, hipStream_t st)
{
    if (!L.bc_face) return;
    if (precision == CFDX_MIXED) launch_bc<float>(L, mode, st);
    else launch_bc<double>(L, mode, st);
}

// get_flow: the reference's FLOW record of every owned node, owned order (Weno.cl:3126-3135 for
// t, a, e; mu of the last viscous pass). The primitives are those of the last stage (plain form)
// or recovered in double from the RK base (mixed form).
__global__ void k_flow_out(BlockDev B, cfdx_flow *__restrict__ out, double mach, int from_base)
{
    const uint32_t o = blockIdx.x * blockDim.x + threadIdx.x, no = owned_count(B);
    if (o >= no) return;
    const uint32_t g = owned_node(B, o);
    double rho, u, v, w, p;
    if (from_base) {
        const double idet = 1.0 / ld(B.det, g);
        rho = idet * ld(B.U0[0], g);
        const double ir = 1.0 / rho;
        u = (idet * ld(B.U0[1], g)) * ir; v = (idet * ld(B.U0[2], g)) * ir; w = (idet * ld(B.U0[3], g)) * ir;
        const double e = (idet * ld(B.U0[4], g)) * ir - 0.5 * (u * u + v * v + w * w);
        p = e * rho * 0.4;
    } else {
        rho = ld((const double *)B.P[0], g); u = ld((const double *)B.P[1], g); v = ld((const double *)B.P[2], g);
        w = ld((const double *)B.P[3], g); p = ld((const double *)B.P[4], g);
    }
    // the record's 9 doubles in order u, v, w, p, t, rho, mu, a, e (out is 8-byte aligned)
    double *r = (double *)out + 9 * (size_t)o;
    r[0] = u; r[1] = v; r[2] = w; r[3] = p;
    r[4] = (1.4 * mach * mach) * (p / rho);
    r[5] = rho;
    r[6] = ld(B.mu, g);
    r[7] = sqrt(1.4 * p / rho);
    r[8] = p / (0.4 * rho);
}

void flow_out(const BlockDev &B, int precision, hipStream_t st, cfdx_flow *out, double mach)
{
    const unsigned nb = (unsigned)(((uint32_t)B.ni * B.nj * B.nk + 255) / 256);
    hipLaunchKernelGGL(k_flow_out, dim3(nb), dim3(256), 0, st, B, out, mach, precision == CFDX_MIXED ? 1 : 0);
}

// number of workgroups that met a value that is not finite among p[0..n)
__global__ void __launch_bounds__(256) k_nonfinite(const double *__restrict__ p, size_t n, unsigned *__restrict__ count)
{
    bool bad = false;
    for (size_t q = (size_t)blockIdx.x * blockDim.x + threadIdx.x; q < n; q += (size_t)gridDim.x * blockDim.x)
        bad |= !__builtin_isfinite(p[q]);
    if (__syncthreads_or(bad) && threadIdx.x == 0) atomicAdd(count, 1u);
}

void count_nonfinite(const double *p, size_t n, unsigned *count, hipStream_t st)
{
    const unsigned nb = (unsigned)std::min<size_t>((n + 255) / 256, 4096);
    hipLaunchKernelGGL(k_nonfinite, dim3(nb), dim3(256), 0, st, p, n, count);
}

__global__ void __launch_bounds__(256) k_geo32(const double *__restrict__ src, float *__restrict__ dst, size_t n)
{
    for (size_t q = (size_t)blockIdx.x * blockDim.x + threadIdx.x; q < n; q += (size_t)gridDim.x * blockDim.x)
        dst[q] = (float)src[q];
}

// The face arrays (metric row k of the +1/2 face along each direction, arrays 10-18, and its det
// det_f, arrays 19-21) into the form the face sweeps use: the unit normal k / |k| and det_f |k|.
// A stored node with no face (k = 0) keeps zeros.
__global__ void __launch_bounds__(256) k_unit_normals(double *__restrict__ geo, size_t n)
{
    for (size_t g = (size_t)blockIdx.x * blockDim.x + threadIdx.x; g < n; g += (size_t)gridDim.x * blockDim.x) {
#pragma unroll
        for (int d = 0; d < 3; ++d) {
            double *k = geo + (size_t)(10 + 3 * d) * n + g, *df = geo + (size_t)(19 + d) * n + g;
            const double a = k[0], b = k[n], c = k[2 * n];
            const double kn = sqrt(a * a + b * b + c * c);
            if (kn > 0.0) {
                k[0] = a / kn;
                k[n] = b / kn;
                k[2 * n] = c / kn;
                df[0] = df[0] * kn;
            }
        }
    }
}

__global__ void __launch_bounds__(256) k_spread_rows(const double *__restrict__ src, double *__restrict__ dst, size_t n,
                                                     uint32_t w, uint32_t pitch)
{
    for (size_t q = (size_t)blockIdx.x * blockDim.x + threadIdx.x; q < n; q += (size_t)gridDim.x * blockDim.x)
        dst[q / w * pitch + q % w] = src[q];
}

void spread_rows(const double *src, double *dst, size_t rows, uint32_t w, uint32_t pitch, hipStream_t st)
{
    const size_t n = rows * w;
    const unsigned nb = (unsigned)std::min<size_t>((n + 255) / 256, 8192);
    hipLaunchKernelGGL(k_spread_rows, dim3(nb), dim3(256), 0, st, src, dst, n, w, pitch);
}

void geometry_finalize(const BlockDev &B, hipStream_t st)
{
    const size_t n = B.n;
    const unsigned nf = (unsigned)std::min<size_t>((n + 255) / 256, 8192);
    hipLaunchKernelGGL(k_unit_normals, dim3(nf), dim3(256), 0, st, const_cast<double *>(B.det), n);
    if (!B.geo32) return;
    const size_t n22 = (size_t)22 * B.n;
    const unsigned nb = (unsigned)std::min<size_t>((n22 + 255) / 256, 8192);
    hipLaunchKernelGGL(k_geo32, dim3(nb), dim3(256), 0, st, B.det, const_cast<float *>(B.geo32), n22);
}

void prims(const BlockDev &B, int precision, hipStream_t st, double *out)
{
    const unsigned nb = (unsigned)(((uint32_t)B.ni * B.nj * B.nk + 255) / 256);
    if (precision == CFDX_MIXED) hipLaunchKernelGGL(k_prims, dim3(nb), dim3(256), 0, st, B, out);
    else hipLaunchKernelGGL(k_copy_prims, dim3(nb), dim3(256), 0, st, B, out);
}

void monitor_reduce(const double *mon, uint32_t count, double *out, hipStream_t st)
{
    hipLaunchKernelGGL(k_mon_reduce, dim3(1), dim3(MON_THREADS), 0, st, mon, count, out);
}

uint32_t tiles_of(const BlockDev &B, int kind, const TileCfg &cfg)
{
    if (kind == 0) {
        const int TX = NODE_TILES[cfg.node][0], TY = NODE_TILES[cfg.node][1];
        return (uint32_t)(((B.ni + TX - 1) / TX) * ((B.nj + TY - 1) / TY) * B.nk);
    }
    auto f = [&](const int (&t)[2], int along, int across, int fix) {
        return (uint32_t)(((across + t[0] - 1) / t[0]) * ((along + t[1] - 1) / t[1]) * fix);
    };
    if (kind == 1 && cfg.face[0] == 0) {
        const uint32_t nf = (uint32_t)faces_along(B, 0), faces = line_faces(nf);
        return (nf * (uint32_t)B.nj * (uint32_t)B.nk + faces - 1) / faces;
    }
    if (kind == 1) return f(FACE_I_TILES[cfg.face[0]], faces_along(B, 0), B.nj, B.nk);
    // rows of tiles over the block's lines, nta tiles to a row
    auto rows = [&](const int (&t)[2], int along, int fix) {
        const uint32_t nta = (uint32_t)((B.ni + t[0] - 1) / t[0]), lines = (uint32_t)line_row(B, t[0]) * (uint32_t)fix;
        return (lines + nta * t[0] - 1) / (nta * t[0]) * nta * (uint32_t)((along + t[1] - 1) / t[1]);
    };
    if (kind == 2) return rows(FACE_JK_TILES[cfg.face[1]], faces_along(B, 1), B.nk);
    return rows(FACE_JK_TILES[cfg.face[2]], faces_along(B, 2), B.nj);
}

}  // namespace blk
}  // namespace cfdx
