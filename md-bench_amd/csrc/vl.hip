// Verlet-list scheme on gfx950: ghost map, binning, neighbour build, LJ (full/half), EAM,
// velocity Verlet and the kinetic-energy reduction.  All arrays stay on the device between
// calls.  Layouts: x, v, f AoS (3 doubles per atom, the reference's ATOM_POSITION_AOS);
// neighbour list SoA (entry k of atom i at k*Nlocal + i), the reference's GPU layout; bins CSR.
//
// Strict kernels keep the reference's evaluation order and never fuse multiply-adds (the whole
// file is built with -ffp-contract=off), so FP64 results are bit-identical to MD-Bench compiled
// the same way.  Fast kernels spread each atom's list over LPA lanes and use explicit fma().
#include <hip/hip_runtime.h>

#include <algorithm>
#include <climits>
#include <cmath>
#include <cstring>
#include <type_traits>

#include "mdgfx950.h"
#include "block_scan.h"
#include "fp64.h"
#include "runtime.h"

using namespace mdg;

namespace {

constexpr int BLOCK     = 256;
constexpr int MAXTYPES2 = 64;  // ntypes <= 8
// LJ passes of full lists stage their neighbours' positions in LDS (k_force_lj_staged, k_stage_build)
// above STAGE_MIN atoms, where the list is kept for STAGE_USES force calls or more: at 1.05 M atoms a
// call gains 84 us and the tables cost 250 us per list; whole steps with a list per 20 measured 323 us
// without and 255 with, at 702 k atoms 218 and 170, at 562 k 148 and 137, at 500 k (the list just fits
// the last-level cache) 126 and 127.
constexpr int STAGE_MIN = 520000, STAGE_USES = 8, STAGE_RETRY = 32;
constexpr int FUSE_GHOSTS_EAM = 300000;  // EAM systems up to this size move ghosts in the force call
constexpr int FAST_LPA  = 4;   // lanes per atom in the fast force kernels of large systems

struct Grid {
    double off[3];     // pad * binsize + 1e-9 (coord2bin, neighbor.c:386-400)
    double bininv[3];
    int mbinx, mbiny, mbinz, mbins;
};

struct Tables {
    double eps[MAXTYPES2], sig6[MAXTYPES2], cutf[MAXTYPES2], cutn[MAXTYPES2];
};

struct State {
    bool ready = false;
    // grid (setupNeighborGFX950)
    Grid g{};
    double binsize[3]{};
    int pad[3]{}, nstencil = 0;
    int* d_stencil = nullptr;
    size_t stencil_cap = 0;
    double prd[3]{}, cutneigh = 0;
    // atoms
    size_t cap_all = 0, cap_ghost = 0, cap_v = 0;
    // second position buffer: a force call that also integrates the next step writes the new
    // local positions there (its other lanes still read the current ones) and the two swap
    double* d_xn  = nullptr;
    size_t cap_xn = 0;
    // fast half lists: force accumulators of the local atoms, zero between calls
    double* d_acc  = nullptr;
    size_t cap_acc = 0;
    // atom sort: the bin-ordered copies of x, v and f (9 doubles per atom) and of the types
    double* d_sort    = nullptr;
    size_t cap_sort   = 0;
    int* d_sort_t     = nullptr;
    size_t cap_sort_t = 0;
    int ntypes = 0;
    int ncu    = 0;  // compute units, rounded up to a multiple of 8 (persistent EAM grids)
    bool uniform = true;  // every type pair has the same LJ parameters
    Tables tab{};
    // bins
    int* d_bin_of = nullptr;
    size_t cap_bin_of = 0;
    int* d_bincount = nullptr;
    int* d_binstart = nullptr;
    size_t cap_bins = 0, cap_binstart = 0;
    int *d_binatoms = nullptr, *d_binslots = nullptr;  // in index order; as scattered
    size_t cap_binatoms = 0, cap_binslots = 0;
    int* d_binplace = nullptr;  // each atom's place in its bin as scattered
    double* d_xs    = nullptr;  // positions in the order of d_binatoms: all x, all y, all z
    size_t cap_binplace = 0, cap_xs = 0;
    bool binned = false;
    // per-atom EAM energies (training labels for the learned potential)
    double* d_eatom = nullptr;
    size_t cap_eatom = 0;
    bool eatom_on = false;
    // ghosts
    int* d_gcnt = nullptr;
    int* d_goff = nullptr;
    size_t cap_gcnt = 0, cap_goff = 0;
    int* d_pbc = nullptr;
    size_t cap_pbc = 0;
    // locals and ghosts of the last setupPbcGFX950, which d_gcnt, d_goff and d_pbc describe
    // (-1: none)
    int gmap_nlocal = -1, gmap_nghost = -1;
    bool ghosts_current = false;  // the last call moved no local atom or moved its ghosts with it
    // neighbour list capacity (elements)
    size_t cap_nb = 0, cap_numneigh = 0;
    // staged neighbour positions (k_stage_build): per block of atoms the atoms its lists name, and
    // each list entry's place among them; stage_nlocal atoms of stage_max entries (-1: none)
    int *d_stage = nullptr, *d_stage_n = nullptr;
    unsigned short* d_hint = nullptr;
    size_t cap_stage = 0, cap_stage_n = 0, cap_hint = 0;
    int stage_nlocal = -1, stage_max = 0;
    // whether tables pay is judged by the last lists (speed only, the results are the same): the force
    // calls of the last two, overflowing blocks (a running count, see k_stage_build), lists to leave out
    int list_uses = -1, last_uses = -1, stage_over = 0, stage_skip = 0;
    // EAM
    double* d_fp = nullptr;
    size_t cap_fp = 0;
    double *d_rhor = nullptr, *d_frho = nullptr, *d_z2r = nullptr;
    int nr = 0, nrho = 0;
    double rdr = 0, rdrho = 0;
    // reductions and status
    double* d_red = nullptr;
    size_t cap_red = 0;
    double* d_ev = nullptr;
    // [0] flags, [1] max numneigh, [2] scan total, [3] staging overflows, [4] go (k_ghost_setup),
    // [ST_OUTSIDE]
    int* d_status = nullptr;
    int* h_status = nullptr;  // pinned
    int* h_flag   = nullptr;  // pinned, written by kernels (HF_*)
    int xs_ld = 0;            // length of d_xs's three runs
    double* h_red = nullptr;  // pinned
    bool ev_on = false;
    double ev_last[2]{};
};

State S;

enum { ST_BIN_RANGE = 1, ST_NB_OVERFLOW = 2 };
// Status word set by a binning with an atom outside the grid, zero between calls: whoever reads it set
// clears it.  (The other flags are cleared between the binning and the list build; with a host word
// for the binning kernels to set, a list of 32,000 atoms took about 2 us more.)
constexpr int ST_OUTSIDE = 5;

// ---------------------------------------------------------------- helpers
__device__ inline int coord2bin(const Grid& g, double x, double y, double z)
{
    int ix = (int)((x + g.off[0]) * g.bininv[0]);
    int iy = (int)((y + g.off[1]) * g.bininv[1]);
    int iz = (int)((z + g.off[2]) * g.bininv[2]);
    return iz * g.mbiny * g.mbinx + iy * g.mbinx + ix;
}

template <int W>
__device__ inline double group_sum(double v)
{
#pragma unroll
    for (int o = W / 2; o > 0; o >>= 1)
        v += __shfl_xor(v, o, W);
    return v;
}

__device__ inline double block_sum(double v, double* sh)
{
    v                = group_sum<64>(v);
    const int lane   = threadIdx.x & 63, w = threadIdx.x >> 6;
    if (lane == 0) sh[w] = v;
    __syncthreads();
    double r = 0;
    if (threadIdx.x == 0)
        for (int k = 0; k < (int)(blockDim.x >> 6); k++)
            r += sh[k];
    __syncthreads();
    return r;  // valid in thread 0
}

// ---------------------------------------------------------------- integrate (integrate.c:21-42)
__global__ void k_initial_integrate(int n3, double* __restrict__ x, double* __restrict__ v,
    const double* __restrict__ f, double dt, double dtforce)
{
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n3) return;
    double vv = v[i] + dtforce * f[i];
    v[i]      = vv;
    x[i]      = x[i] + dt * vv;
}

__global__ void k_final_integrate(int n3, double* __restrict__ v, const double* __restrict__ f,
    double dtforce)
{
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n3) return;
    v[i] = v[i] + dtforce * f[i];
}

// ---------------------------------------------------------------- pbc (pbc.c:42-232)
__global__ void k_wrap(int n3, double* __restrict__ x, double xprd, double yprd, double zprd)
{
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n3) return;
    int d      = i % 3;
    double prd = d == 0 ? xprd : (d == 1 ? yprd : zprd);
    double xx  = x[i];
    if (xx < 0.0) xx += prd;
    else if (xx >= prd) xx -= prd;
    x[i] = xx;
}

// The 26 ghost images in the reference's order: 6 planes, 8 corners, 12 edges.  Each entry:
// required side per axis (0 none, 1 low -> shift +1, 2 high -> shift -1).
__constant__ signed char c_ghost_side[26][3] = {
    { 1, 0, 0 }, { 2, 0, 0 }, { 0, 1, 0 }, { 0, 2, 0 }, { 0, 0, 1 }, { 0, 0, 2 },
    { 1, 1, 1 }, { 1, 2, 1 }, { 1, 1, 2 }, { 1, 2, 2 }, { 2, 1, 1 }, { 2, 2, 1 }, { 2, 1, 2 },
    { 2, 2, 2 },
    { 1, 0, 1 }, { 1, 0, 2 }, { 2, 0, 1 }, { 2, 0, 2 }, { 0, 1, 1 }, { 0, 1, 2 }, { 0, 2, 1 },
    { 0, 2, 2 }, { 1, 1, 0 }, { 2, 1, 0 }, { 1, 2, 0 }, { 2, 2, 0 } };

__device__ inline unsigned ghost_mask(const double* xi, const double* prd, double cut)
{
    unsigned lo[3], hi[3];
#pragma unroll
    for (int d = 0; d < 3; d++) {
        lo[d] = xi[d] < cut;
        hi[d] = xi[d] >= (prd[d] - cut);
    }
    unsigned m = 0;
#pragma unroll
    for (int c = 0; c < 26; c++) {
        bool ok = true;
#pragma unroll
        for (int d = 0; d < 3; d++) {
            int s = c_ghost_side[c][d];
            if (s == 1) ok = ok && lo[d];
            if (s == 2) ok = ok && hi[d];
        }
        if (ok) m |= 1u << c;
    }
    return m;
}

struct Prd {
    double p[3];
};

// (wrap: the atom back into the box first, as k_wrap does)
__global__ void k_ghost_count(int nlocal, double* __restrict__ x, Prd prd, double cut,
    int* __restrict__ cnt, int wrap)
{
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= nlocal) return;
    double xi[3] = { x[3 * i], x[3 * i + 1], x[3 * i + 2] };
    if (wrap)
#pragma unroll
        for (int d = 0; d < 3; d++) {
            if (xi[d] < 0.0) x[3 * i + d] = xi[d] += prd.p[d];
            else if (xi[d] >= prd.p[d]) x[3 * i + d] = xi[d] -= prd.p[d];
        }
    cnt[i] = __popc(ghost_mask(xi, prd.p, cut));
}

// (the ghosts' positions too, as k_update_pbc writes them)
__global__ void k_ghost_fill(int nlocal, double* x, Prd prd, double cut,
    const int* __restrict__ off, int* __restrict__ border_map, int* __restrict__ pbc,
    int* __restrict__ type, const int* __restrict__ go = nullptr)
{
    if (go && !*go) return;
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= nlocal) return;
    double xi[3] = { x[3 * i], x[3 * i + 1], x[3 * i + 2] };
    unsigned m   = ghost_mask(xi, prd.p, cut);
    int g        = off[i];
    int ti       = type[i];
    for (int c = 0; c < 26; c++) {
        if (!(m & (1u << c))) continue;
        border_map[g] = i;
#pragma unroll
        for (int d = 0; d < 3; d++) {
            int s          = c_ghost_side[c][d];
            const int p    = s == 1 ? 1 : (s == 2 ? -1 : 0);
            pbc[3 * g + d] = p;
            x[3 * (nlocal + g) + d] = xi[d] + p * prd.p[d];
        }
        type[nlocal + g] = ti;
        g++;
    }
}

// After a ghost count: whether room suffices (see k_ghost_setup), and clean words for the list build
__global__ void k_ghost_go(int room, int* __restrict__ status, int* __restrict__ go)
{
    status[0] = status[1] = 0;
    *go       = status[2] <= room;
}

// The ghosts' counts and offsets of a small system in one block (and, with wrap, the atoms' return
// into the box before): thread t owns atoms t * per onwards, so that the ghosts stay in the order of
// their owners.  The total goes to the host's word too.  More than room ghosts: go is set to 0 and
// the launches behind this one, made before the host knows the total, do nothing.
// Launches bound a small system's rebuild (about 5 us each with the gap before it): wrap, count,
// scan and the status copy were four (9.5 us of kernels for 256 atoms, 3.5 here).
constexpr int SETUP_T = 1024, SETUP_I = 8, SETUP_SMALL = SETUP_T * SETUP_I;
enum { HF_TOTAL, HF_OVERFLOW, HF_RANGE };  // words that kernels write for the host

__global__ void __launch_bounds__(SETUP_T) k_ghost_setup(int n, double* __restrict__ x, int wrap,
    Prd prd, double cut, int* __restrict__ cnt, int* __restrict__ off, int* __restrict__ status,
    int room, int* __restrict__ go, int* __restrict__ host)
{
    __shared__ int sh[33];
    const int per = (n + SETUP_T - 1) / SETUP_T;
    const int b   = threadIdx.x * per;
    int c[SETUP_I], sum = 0;
    double r[SETUP_I][3];  // (all loads first)
#pragma unroll
    for (int k = 0; k < SETUP_I; k++)
        if (k < per)
#pragma unroll
            for (int d = 0; d < 3; d++)
                r[k][d] = x[3 * min(b + k, n - 1) + d];
#pragma unroll
    for (int k = 0; k < SETUP_I; k++) {
        c[k] = 0;
        if (k >= per || b + k >= n) continue;
        const int i = b + k;
        int prod    = 1;
#pragma unroll
        for (int d = 0; d < 3; d++) {
            double xx = r[k][d];
            if (wrap) {  // (k_wrap)
                if (xx < 0.0) x[3 * i + d] = xx += prd.p[d];
                else if (xx >= prd.p[d]) x[3 * i + d] = xx -= prd.p[d];
            }
            prod *= 1 + (xx < cut) + (xx >= (prd.p[d] - cut));
        }
        c[k] = prod - 1;  // = the bits of ghost_mask
        sum += c[k];
    }
    int total;
    int at = block_excl_scan(sum, sh, &total);
#pragma unroll
    for (int k = 0; k < SETUP_I; k++) {
        if (k >= per || b + k >= n) continue;
        cnt[b + k] = c[k];
        off[b + k] = at;
        at += c[k];
    }
    if (threadIdx.x == 0) {
        status[0] = status[1] = 0;
        status[2] = total;
        *go       = total <= room;
        host[HF_TOTAL] = total;
    }
}

// k_ghost_fill with a thread per atom and image: with a thread per atom, 256 atoms of up to seven
// images took 6.9 us (3.1 so).
__global__ void __launch_bounds__(BLOCK) k_ghost_fill_small(int nlocal, double* x, Prd prd, double cut,
    const int* __restrict__ off, int* __restrict__ border_map, int* __restrict__ pbc,
    int* __restrict__ type, const int* __restrict__ go)
{
    if (!*go) return;
    const int i = (blockIdx.x * BLOCK + threadIdx.x) >> 5, c = threadIdx.x & 31;
    if (i >= nlocal) return;  // (for the two halves of a wavefront by themselves)
    double xi[3] = { x[3 * i], x[3 * i + 1], x[3 * i + 2] };
    const unsigned m = ghost_mask(xi, prd.p, cut);
    if (!(m >> c & 1)) return;
    const int g   = off[i] + __popc(m & ((1u << c) - 1));
    border_map[g] = i;
#pragma unroll
    for (int d = 0; d < 3; d++) {
        const int s             = c_ghost_side[c][d];
        const int p             = s == 1 ? 1 : (s == 2 ? -1 : 0);
        pbc[3 * g + d]          = p;
        x[3 * (nlocal + g) + d] = xi[d] + p * prd.p[d];
    }
    type[nlocal + g] = type[i];
}

__global__ void k_update_pbc(int nlocal, int nghost, double* __restrict__ x,
    const int* __restrict__ border_map, const int* __restrict__ pbc, Prd prd)
{
    int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= 3 * nghost) return;
    int g               = k / 3, d = k % 3;
    int b               = border_map[g];
    x[3 * (nlocal + g) + d] = x[3 * b + d] + pbc[3 * g + d] * prd.p[d];
}

// ---------------------------------------------------------------- binning (neighbor.c:386-464)
// Each atom's bin and its place among the bin's atoms as they arrive (one atomic per atom: with a
// second one in the scatter the two took 29 us each at 1M atoms).  An atom outside the grid is in no
// bin, and sets *outside where the caller asks for it.
__global__ void k_bin_count(int nlocal, const int* __restrict__ nghost, const double* __restrict__ x, Grid g, int* __restrict__ bin_of,
    int* __restrict__ place, int* __restrict__ count, int* __restrict__ outside,
    const int* __restrict__ go)
{
    if (go && !*go) return;
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= nlocal + (nghost ? *nghost : 0)) return;
    int b = coord2bin(g, x[3 * i], x[3 * i + 1], x[3 * i + 2]);
    if (b < 0 || b >= g.mbins) {
        if (outside) *outside = 1;
        bin_of[i] = -1;
        return;
    }
    bin_of[i] = b;
    place[i]  = atomicAdd(&count[b], 1);
}

__global__ void k_bin_scatter(int nlocal, const int* __restrict__ nghost, const int* __restrict__ bin_of,
    const int* __restrict__ place, const int* __restrict__ binstart, int* __restrict__ slots,
    const int* __restrict__ go)
{
    if (go && !*go) return;
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= nlocal + (nghost ? *nghost : 0)) return;
    int b = bin_of[i];
    if (b < 0) return;
    slots[binstart[b] + place[i]] = i;
}

// Atoms arrive in a bin in arbitrary order; the reference fills bins in atom-index order, so each
// atom goes to its rank among its bin's (a handful of atoms).  One atom per thread: with one bin
// per thread (an insertion sort in memory) it took 13 us for 256 atoms and their ghosts.  The
// positions are copied to the same order (xs: n x, n y, n z), in which the list build's candidates
// are contiguous.  clear: two status words zeroed for the list build that follows.
__global__ void k_bin_rank(int n, const int* __restrict__ bin_of, const int* __restrict__ binstart,
    const int* __restrict__ slots, const double* __restrict__ x, int* __restrict__ binatoms,
    double* __restrict__ xs, const int* __restrict__ total, int* __restrict__ clear,
    const int* __restrict__ go = nullptr)
{
    if (go && !*go) return;
    const int m = blockIdx.x * blockDim.x + threadIdx.x;
    if (clear && m < 2) clear[m] = 0;
    if (m >= n || m >= *total) return;
    const int a = slots[m], b = bin_of[a];
    const int s = binstart[b], e = binstart[b + 1];
    int r = s;
    for (int k = s; k < e; k++)
        r += slots[k] < a;
    binatoms[r] = a;
#pragma unroll
    for (int d = 0; d < 3; d++)
        xs[(size_t)d * n + r] = x[3 * a + d];
}

// Counts, scan and scatter in one block for a small system, with the counts and starts in LDS and an
// atom's bin and place in registers; ORDER (up to BIN1_ORDER atoms): the slots in LDS too, and
// k_bin_rank's work.  n: nlocal plus the ghosts counted by k_ghost_setup where nghost is not null.
// 256 atoms and 1500 ghosts: 15 us in four launches, 7.7 in one.  4000 atoms and 5500 ghosts: 25 us in
// four launches, 17.5 in two, 24 in one (6 for the ranks and 9 for the writes, which many blocks share
// better).  outside: as for k_bin_count; clear: two status words zeroed for the list build that follows.
constexpr int BIN1_T = 1024, BIN1_I = 16, BIN1_N = BIN1_T * BIN1_I, BIN1_BINS = 16384;
constexpr int BIN1_ORDER = 4 * BIN1_T;

template <bool ORDER>
__global__ void __launch_bounds__(BIN1_T) k_bin_single(int nlocal, const int* __restrict__ nghost,
    int ld, const double* __restrict__ x, Grid g, int* __restrict__ binstart,
    int* __restrict__ bin_of, int* __restrict__ slots, int* __restrict__ binatoms,
    double* __restrict__ xs, int* __restrict__ outside, int* __restrict__ clear,
    const int* __restrict__ go)
{
    constexpr int NI = ORDER ? BIN1_ORDER / BIN1_T : BIN1_I;
    __shared__ int s_bin[BIN1_BINS];  // atoms per bin, then the bins' starts
    __shared__ int s_slot[ORDER ? BIN1_ORDER : 1];
    __shared__ int sh[33];
    if (go && !*go) return;
    const int n   = nlocal + (nghost ? *nghost : 0);
    const int tid = threadIdx.x;
    for (int b = tid; b < g.mbins; b += BIN1_T)
        s_bin[b] = 0;
    __syncthreads();
    int bin[NI], place[NI];
    double r[4][3];  // (four atoms' loads together)
#pragma unroll
    for (int k = 0; k < NI; k++) {
        bin[k] = -1;
        if (k * BIN1_T >= n) continue;  // (uniform)
        if ((k & 3) == 0)
#pragma unroll
            for (int q = 0; q < 4; q++)
#pragma unroll
                for (int d = 0; d < 3; d++)
                    r[q][d] = x[3 * min((k + q) * BIN1_T + tid, n - 1) + d];
        const int i = k * BIN1_T + tid;
        if (i >= n) continue;
        const int b = coord2bin(g, r[k & 3][0], r[k & 3][1], r[k & 3][2]);
        if (b < 0 || b >= g.mbins) {
            if (outside) *outside = 1;
            continue;
        }
        bin[k]   = b;
        place[k] = atomicAdd(&s_bin[b], 1);
    }
    __syncthreads();
    // thread t's bins t * per onwards
    const int per = (g.mbins + BIN1_T - 1) / BIN1_T;
    const int b0 = tid * per, b1 = min(b0 + per, g.mbins);
    int sum = 0, total;
    for (int b = b0; b < b1; b++)
        sum += s_bin[b];
    int at = block_excl_scan(sum, sh, &total);
    for (int b = b0; b < b1; b++) {
        const int c = s_bin[b];
        s_bin[b]    = at;
        at += c;
    }
    __syncthreads();
    for (int b = tid; b < g.mbins; b += BIN1_T)
        binstart[b] = s_bin[b];
    if (tid == 0) {
        binstart[g.mbins] = total;
        if (clear) clear[0] = clear[1] = 0;
    }
#pragma unroll
    for (int k = 0; k < NI; k++) {
        const int i = k * BIN1_T + tid;
        if (!ORDER && i < n) bin_of[i] = bin[k];
        if (bin[k] >= 0) (ORDER ? s_slot : slots)[s_bin[bin[k]] + place[k]] = i;
    }
    if (!ORDER) return;
    __syncthreads();
#pragma unroll
    for (int k = 0; k < NI; k++) {
        if (bin[k] < 0) continue;
        const int i = k * BIN1_T + tid;
        const int s = s_bin[bin[k]], e = bin[k] + 1 < g.mbins ? s_bin[bin[k] + 1] : total;
        int m = s;
        for (int q = s; q < e; q++)
            m += s_slot[q] < i;
        binatoms[m] = i;
#pragma unroll
        for (int d = 0; d < 3; d++)
            xs[(size_t)d * ld + m] = r[k][d];
    }
}

// Launches the binning of up to BIN1_N atoms (nlocal and *nghost), max_n at most, in few launches.
void launch_bins_small(int nlocal, const int* nghost, int max_n, const double* x, int* outside,
    int* clear, const int* go)
{
    hipStream_t s = stream();
    if (max_n <= BIN1_ORDER) {
        k_bin_single<true><<<1, BIN1_T, 0, s>>>(nlocal, nghost, S.xs_ld, x, S.g, S.d_binstart,
            S.d_bin_of, S.d_binslots, S.d_binatoms, S.d_xs, outside, clear, go);
    } else {
        k_bin_single<false><<<1, BIN1_T, 0, s>>>(nlocal, nghost, S.xs_ld, x, S.g, S.d_binstart,
            S.d_bin_of, S.d_binslots, S.d_binatoms, S.d_xs, outside, clear, go);
        k_bin_rank<<<blocks_for(max_n, BLOCK), BLOCK, 0, s>>>(S.xs_ld, S.d_bin_of, S.d_binstart,
            S.d_binslots, x, S.d_binatoms, S.d_xs, S.d_binstart + S.g.mbins, nullptr, go);
    }
    MDG_LAUNCH_CHECK("binatoms");
}

// sortAtom (neighbor.c:466-536): new slot p takes the atom at position p of the bin-major list of
// the local atoms (in index order within a bin), with its position, velocity, force and type.
__global__ void k_sort_gather(int n, const int* __restrict__ order, const double* __restrict__ x,
    const double* __restrict__ v, const double* __restrict__ f, const int* __restrict__ type,
    double* __restrict__ xs, double* __restrict__ vs, double* __restrict__ fs,
    int* __restrict__ ts)
{
    const int p = blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= n) return;
    const int o = order[p];
#pragma unroll
    for (int d = 0; d < 3; d++) {
        xs[3 * p + d] = x[3 * o + d];
        vs[3 * p + d] = v[3 * o + d];
        fs[3 * p + d] = f[3 * o + d];
    }
    ts[p] = type[o];
}

// ---------------------------------------------------------------- neighbour build
// (neighbor.c:260-352): stencil bins in order, atoms in bin order, rsq <= cutneighsq.
// One block per bin, its local atoms (32 at a time, bin order) in LDS.  The candidates of the bin's
// stencil are flattened in the reference's loop order (stencil bins in order, atoms in bin order)
// and taken in segments of NB_SEG, in four passes over the block's threads:
//   1. the candidates farther from the local atoms' bounding box than the cutoff drop out (about
//      half of the stencil's; the margin keeps every pair whose own test could pass); the others
//      stay in order;
//   2. the rest against every local atom, a ballot per atom and 64 candidates kept in LDS;
//   3. the ballots' running counts per local atom;
//   4. each accepted candidate to its place in that atom's list.
// For small systems, whose few bins leave the chip idle: the passes' latency bounds it (one
// wavefront per bin with every candidate tested against every atom, as before, took 40 us for 256
// atoms; this takes 17, of 16384 atoms 35 us; the wavefront kernel below 27 and 41 us, but from
// 32000 atoms on 50 us against 56, and 794 against 1650 us at 1M).
constexpr int NB_T = 256, NB_SEG = 1024, NB_Q = 32;
constexpr int NB_SMALL = 24000;  // atoms up to which the block kernel builds the lists
constexpr int NB_BINS  = 16384;  // and bins (see small_lists)

__global__ void __launch_bounds__(NB_T) k_build_neighbor(int nlocal, int ld, const double* __restrict__ xs,
    const int* __restrict__ type, int ntypes, Tables tab, int uniform, double cnmax, int mbins,
    const int* __restrict__ binstart, const int* __restrict__ binatoms,
    const int* __restrict__ stencil, int nstencil, int half, int maxneighs,
    int* __restrict__ neighbors, int* __restrict__ numneigh, int* __restrict__ status,
    int* __restrict__ host, const int* __restrict__ go)
{
    __shared__ int s_m[NB_SEG], s_cj[NB_SEG];
    __shared__ unsigned long long s_mask[NB_Q][NB_SEG / 64];
    __shared__ int s_off[NB_Q][NB_SEG / 64];
    __shared__ double s_x[NB_Q][3];
    __shared__ int s_id[NB_Q], s_t[NB_Q], s_cnt[NB_Q], s_scan[33], s_w[NB_T / 64], s_nq;
    const double* ys = xs + ld;
    const double* zs = ys + ld;
    const int b      = blockIdx.x;
    if (b >= mbins || (go && !*go)) return;
    if (b == 0 && threadIdx.x == 0 && status[ST_OUTSIDE]) host[HF_RANGE] = 1;
    const int beg = binstart[b], end = binstart[b + 1];
    // index order inside a bin: its local atoms come first
    if (beg >= end || binatoms[beg] >= nlocal) return;
    const int tid = threadIdx.x, w = tid >> 6, lane = tid & 63;
    const unsigned long long lt = (lane == 0) ? 0ull : (~0ull >> (64 - lane));
    for (int q0 = beg; q0 < end; q0 += NB_Q) {
        __syncthreads();
        if (w == 0) {
            const int m0 = q0 + lane;
            int i0       = -1;
            if (lane < NB_Q && m0 < end) i0 = binatoms[m0];
            const bool isloc = i0 >= 0 && i0 < nlocal;
            const unsigned long long lb = __ballot(isloc);
            if (isloc) {
                const int q = __popcll(lb & lt);
                s_id[q]     = i0;
                s_t[q]      = type[i0];
                s_x[q][0]   = xs[m0];
                s_x[q][1]   = ys[m0];
                s_x[q][2]   = zs[m0];
            }
            if (lane < NB_Q) s_cnt[lane] = 0;
            if (lane == 0) s_nq = __popcll(lb);
        }
        __syncthreads();
        const int nq = s_nq;
        if (nq == 0) break;
        double lo3[3] = { s_x[0][0], s_x[0][1], s_x[0][2] }, hi3[3] = { lo3[0], lo3[1], lo3[2] };
        for (int q = 1; q < nq; q++)
#pragma unroll
            for (int d = 0; d < 3; d++) {
                const double v = s_x[q][d];
                lo3[d]         = fmin(lo3[d], v);
                hi3[d]         = fmax(hi3[d], v);
            }
        for (int c0 = 0; c0 < nstencil; c0 += NB_T) {
            int lo = 0, cc = 0;
            if (c0 + tid < nstencil) {
                const int jb = b + stencil[c0 + tid];
                if (jb < 0 || jb >= mbins) {
                    host[HF_RANGE] = 1;
                } else {
                    lo = binstart[jb];
                    cc = binstart[jb + 1] - lo;
                }
            }
            int total;
            const int pre = block_excl_scan(cc, s_scan, &total);
            for (int g0 = 0; g0 < total; g0 += NB_SEG) {
                const int segn = min(NB_SEG, total - g0);
                for (int t = max(pre, g0); t < min(pre + cc, g0 + segn); t++)
                    s_m[t - g0] = lo + (t - pre);
                __syncthreads();
                // 1. the candidates near the local atoms' box, in order
                int nc = 0;
                for (int t0 = 0; t0 < segn; t0 += NB_T) {
                    const int t = t0 + tid;
                    bool near   = false;
                    int m       = 0;
                    if (t < segn) {
                        m                  = s_m[t];
                        const double xj[3] = { xs[m], ys[m], zs[m] };
                        double d2          = 0.0;
#pragma unroll
                        for (int d = 0; d < 3; d++) {
                            const double g = fmax(fmax(lo3[d] - xj[d], xj[d] - hi3[d]), 0.0);
                            d2             = fma(g, g, d2);
                        }
                        near = d2 <= cnmax;
                    }
                    const unsigned long long bal = __ballot(near);
                    if (lane == 0) s_w[w] = __popcll(bal);
                    __syncthreads();
                    int at = nc;
#pragma unroll
                    for (int k = 0; k < NB_T / 64; k++) {
                        if (k < w) at += s_w[k];
                        nc += s_w[k];
                    }
                    if (near) s_cj[at + __popcll(bal & lt)] = m;
                    __syncthreads();
                }
                const int nb = (nc + 63) >> 6;
                // 2. against every local atom, half of the atoms per turn of a wavefront
                const int qh = (nq + 1) >> 1;
                for (int u = w; u < 2 * nb; u += NB_T / 64) {
                    const int bt = u >> 1, qb = (u & 1) * qh, qe = min(nq, qb + qh);
                    const bool cand = bt * 64 + lane < nc;
                    int j = 0, tj = 0;
                    double xj = 0.0, yj = 0.0, zj = 0.0;
                    if (cand) {
                        const int m = s_cj[bt * 64 + lane];
                        j           = binatoms[m];
                        xj          = xs[m];
                        yj          = ys[m];
                        zj          = zs[m];
                        if (!uniform) tj = type[j];
                    }
                    for (int q = qb; q < qe; q++) {
                        const int i      = s_id[q];
                        const double dx  = s_x[q][0] - xj;
                        const double dy  = s_x[q][1] - yj;
                        const double dz  = s_x[q][2] - zj;
                        const double rsq = dx * dx + dy * dy + dz * dz;
                        const double cn  = uniform ? tab.cutn[0] : tab.cutn[s_t[q] * ntypes + tj];
                        const bool pass  = cand && j != i && !(half && j < i) && rsq <= cn;
                        const unsigned long long bq = __ballot(pass);
                        if (lane == 0) s_mask[q][bt] = bq;
                    }
                }
                __syncthreads();
                // 3. running counts
                if (tid < nq) {
                    int n = s_cnt[tid];
                    for (int bt = 0; bt < nb; bt++) {
                        s_off[tid][bt] = n;
                        n += __popcll(s_mask[tid][bt]);
                    }
                    s_cnt[tid] = n;
                }
                __syncthreads();
                // 4. the accepted ones to their lists
                for (int bt = 0; bt < nb; bt++) {
                    const int j = bt * 64 + lane < nc ? binatoms[s_cj[bt * 64 + lane]] : 0;
                    for (int q = w; q < nq; q += NB_T / 64) {
                        const unsigned long long m = s_mask[q][bt];
                        const int pos              = s_off[q][bt] + __popcll(m & lt);
                        if ((m >> lane & 1) && pos < maxneighs)
                            neighbors[(size_t)pos * nlocal + s_id[q]] = j;
                    }
                }
                __syncthreads();
            }
        }
        if (tid < nq) {
            const int n         = s_cnt[tid];
            numneigh[s_id[tid]] = n;
            if (n > maxneighs) {
                host[HF_OVERFLOW] = 1;
                atomicMax(&status[1], n);
            }
        }
    }
}

// The same for large systems, one wavefront per bin and no barriers: the stencil columns' lanes
// write the candidates' entries to LDS (each candidate found its column by a binary search of
// dependent cross-lane reads before), the ones near the local atoms' box are kept in place, in
// order, and only those are tested against every local atom.  880 -> 794 us for 1M atoms, 147 ->
// 120 us for 131,000.  The tests' vector instructions (1640 per bin, 400 us) and the texture
// path's work (the scattered list stores and the candidates' loads, 600 us busy) bound it; bins
// of one XCD adjacent made it slower (895 us: slabs of ghost bins leave an XCD idle).
// Up to NB_FEW local atoms (bins of half the list cutoff, in boxes read from a file) are tested against
// every candidate at once: choosing the near ones costs as much as those tests.  us per list with 2, 3,
// 4 and 5 (without: 1319; the kernel before: 1205) for 1.05 M atoms in such bins 1255, 1263, 1223, 1216, for
// 131,000 136, 137, 134, 135 (141; 128); bins of seven atoms unchanged.
constexpr int NBW_SEG = 1024, NB_FEW = 4;
struct NbLocal {
    double x, y, z;
    int id, type;
};

__device__ inline void wave_fence()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

__global__ void __launch_bounds__(BLOCK) k_build_neighbor_wave(int nlocal, int ld,
    const double* __restrict__ xs, const int* __restrict__ type, int ntypes, Tables tab, int uniform,
    double cnmax, int mbins, const int* __restrict__ binstart, const int* __restrict__ binatoms,
    const int* __restrict__ stencil, int nstencil, int half, int maxneighs,
    int* __restrict__ neighbors, int* __restrict__ numneigh, int* __restrict__ status,
    const int* __restrict__ go)
{
    __shared__ int s_c[BLOCK / 64][NBW_SEG];
    __shared__ __align__(16) NbLocal s_l[BLOCK / 64][NB_Q];
    const int w = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int b = __builtin_amdgcn_readfirstlane(blockIdx.x * (BLOCK / 64) + w);
    if (b >= mbins || (go && !*go)) return;
    const int beg = binstart[b], end = binstart[b + 1];
    if (beg >= end || binatoms[beg] >= nlocal) return;
    const unsigned long long lt = (lane == 0) ? 0ull : (~0ull >> (64 - lane));
    const double* ys = xs + ld;
    const double* zs = ys + ld;
    int* s_m         = s_c[w];
    NbLocal* loc = s_l[w];
    for (int q0 = beg; q0 < end; q0 += NB_Q) {
        // this chunk's local atoms, in bin order, and their box
        const int m0 = q0 + lane;
        int i0       = -1;
        if (lane < NB_Q && m0 < end) i0 = binatoms[m0];
        const bool isloc = i0 >= 0 && i0 < nlocal;
        const int nq     = __popcll(__ballot(isloc));
        if (nq == 0) break;  // index order inside a bin: ghosts from here on
        double lo3[3] = { 1e300, 1e300, 1e300 }, hi3[3] = { -1e300, -1e300, -1e300 };
        if (isloc) {  // lanes 0 .. nq - 1
            NbLocal l{ xs[m0], ys[m0], zs[m0], i0, type[i0] };
            loc[lane] = l;
            lo3[0] = hi3[0] = l.x;
            lo3[1] = hi3[1] = l.y;
            lo3[2] = hi3[2] = l.z;
        }
#pragma unroll
        for (int o = 1; o < NB_Q; o <<= 1)
#pragma unroll
            for (int d = 0; d < 3; d++) {
                lo3[d] = fmin(lo3[d], __shfl_xor(lo3[d], o, 64));
                hi3[d] = fmax(hi3[d], __shfl_xor(hi3[d], o, 64));
            }
#pragma unroll
        for (int d = 0; d < 3; d++) {  // lanes 32 .. 63 read those of lanes 0 .. 31
            lo3[d] = __shfl(lo3[d], lane & (NB_Q - 1), 64);
            hi3[d] = __shfl(hi3[d], lane & (NB_Q - 1), 64);
        }
        int cnt = 0;  // lane q < nq: length of atom q's list so far
        for (int s0 = 0; s0 < nstencil; s0 += 64) {
            int lo = 0, cc = 0;
            if (s0 + lane < nstencil) {
                const int jb = b + stencil[s0 + lane];
                if (jb < 0 || jb >= mbins) {
                    atomicOr(&status[0], ST_BIN_RANGE);
                } else {
                    lo = binstart[jb];
                    cc = binstart[jb + 1] - lo;
                }
            }
            const int inc   = wave_incl_scan(cc);
            const int total = __shfl(inc, 63, 64);
            const int pre   = inc - cc;
            for (int g0 = 0; g0 < total; g0 += NBW_SEG) {
                const int segn = min(NBW_SEG, total - g0);
                const int t1   = min(inc, g0 + segn);
                wave_fence();
                for (int t = max(pre, g0); t < t1; t++)
                    s_m[t - g0] = lo + (t - pre);
                wave_fence();
                // the candidates near the box stay, in order (a batch is read before its places,
                // at or below it, are written); all of them for few local atoms
                int nc = nq <= NB_FEW ? segn : 0;
                for (int t0 = nc; t0 < segn; t0 += 64) {
                    bool near = false;
                    int m     = 0;
                    if (t0 + lane < segn) {
                        m                  = s_m[t0 + lane];
                        const double xj[3] = { xs[m], ys[m], zs[m] };
                        double d2          = 0.0;
#pragma unroll
                        for (int d = 0; d < 3; d++) {
                            const double g = fmax(fmax(lo3[d] - xj[d], xj[d] - hi3[d]), 0.0);
                            d2             = fma(g, g, d2);
                        }
                        near = d2 <= cnmax;
                    }
                    const unsigned long long bal = __ballot(near);
                    wave_fence();
                    if (near) s_m[nc + __popcll(bal & lt)] = m;
                    wave_fence();
                    nc += __popcll(bal);
                }
                for (int t0 = 0; t0 < nc; t0 += 64) {
                    const bool cand = t0 + lane < nc;
                    int j = -1, tj = 0;
                    double xj = 0.0, yj = 0.0, zj = 0.0;
                    if (cand) {
                        const int m = s_m[t0 + lane];
                        j           = binatoms[m];
                        xj          = xs[m];
                        yj          = ys[m];
                        zj          = zs[m];
                        if (!uniform) tj = type[j];
                    }
                    for (int q = 0; q < nq; q++) {
                        const NbLocal l  = loc[q];
                        const double dx  = l.x - xj;
                        const double dy  = l.y - yj;
                        const double dz  = l.z - zj;
                        const double rsq = dx * dx + dy * dy + dz * dz;
                        const double cn  = uniform ? tab.cutn[0] : tab.cutn[l.type * ntypes + tj];
                        const bool pass  = cand && j != l.id && !(half && j < l.id) && rsq <= cn;
                        const unsigned long long bq = __ballot(pass);
                        const int base = __builtin_amdgcn_readlane(cnt, q);
                        if (pass) {
                            const int pos = base + __popcll(bq & lt);
                            if (pos < maxneighs) neighbors[(size_t)pos * nlocal + l.id] = j;
                        }
                        if (lane == q) cnt += __popcll(bq);
                    }
                }
            }
        }
        if (lane < nq) {
            numneigh[i0] = cnt;
            if (cnt > maxneighs) {
                atomicOr(&status[0], ST_NB_OVERFLOW);
                atomicMax(&status[1], cnt);
            }
        }
        wave_fence();
    }
}

// The run loop's integration inside a full-list force kernel: with v set, the lane that writes
// an atom's total force also applies finalIntegrate (integrate.c:61-86) and the next step's
// initialIntegrate (integrate.c:29-59) with it, the same FP64 operations in the same order as
// k_final_integrate then k_initial_integrate, and writes the new position to xn.
// With gcnt set (the ghosts of setupPbcGFX950: atom i's images are goff[i] .. goff[i] + gcnt[i])
// the atom's lanes also write its images' new positions, as k_update_pbc does afterwards: a step
// is then one launch instead of two (the ghost update is 3.8 us of a 256-atom step and 5.2 us of
// a 1M-atom one, nearly all of it the launch).
struct Fuse0 {
    double* v;
    double* xn;
    double dt, dtforce;
};
struct Fuse : Fuse0 {
    const int* gcnt;
    const int* goff;
    const int* pbc;
    double prd[3];
};

template <bool GH>
using FuseOf = std::conditional_t<GH, Fuse, Fuse0>;

// v0 (loaded at the kernel's start, so its latency hides behind the neighbour loop) and x0 are
// the atom's velocity and position, fx, fy, fz its total force: the same in all of its LPA lanes.
template <int LPA, bool GH>
__device__ inline void fused_integrate(const FuseOf<GH>& fu, int nlocal, int i, int lane,
    const double* v0, const double* x0, int ng, int g0, double fx, double fy, double fz)
{
    const double fr[3] = { fx, fy, fz };
    double xn[3];
#pragma unroll
    for (int d = 0; d < 3; d++) {
        double vv = v0[d] + fu.dtforce * fr[d];
        vv        = vv + fu.dtforce * fr[d];
        xn[d]     = x0[d] + fu.dt * vv;
        if (lane == 0) {
            fu.v[3 * i + d]  = vv;
            fu.xn[3 * i + d] = xn[d];
        }
    }
    if constexpr (GH)
        for (int k = lane; k < ng; k += LPA) {
            const int g = g0 + k;
#pragma unroll
            for (int d = 0; d < 3; d++)
                fu.xn[3 * (nlocal + g) + d] = xn[d] + fu.pbc[3 * g + d] * fu.prd[d];
        }
}

// What fused_integrate needs of atom i, loaded ahead of the neighbour loop.
template <bool GH>
__device__ inline void fused_load(const FuseOf<GH>& fu, int i, double* v0, int* ng, int* g0)
{
#pragma unroll
    for (int d = 0; d < 3; d++)
        v0[d] = fu.v[3 * i + d];
    if constexpr (GH)
        if (fu.gcnt) {
            *ng = fu.gcnt[i];
            *g0 = fu.goff[i];
        }
}

// A lane's list entries (lane, lane + LPA, ... of atom i) in order.  The loads have no branch around
// them, which would make the compiler wait for all loads in flight: behind the list's end the first
// entry is read again.
template <int LPA>
struct ListWalk {
    const int *p, *p0;
    size_t step;
    int nn;
    __device__ ListWalk(const int* neighbors, int nlocal, int i, int lane, int n)
        : p(neighbors + (size_t)lane * nlocal + i), p0(neighbors + i), step((size_t)LPA * nlocal),
          nn(n)
    {
    }
    __device__ int next(int k)
    {
        const int j = *(k < nn ? p : p0);
        p += step;
        return j;
    }
};

// The value of the neighbouring lane (lane ^ 1)
__device__ inline int swap1(int v) { return __builtin_amdgcn_update_dpp(0, v, 0xB1, 0xf, 0xf, false); }
__device__ inline double swap1(double v)
{
    const long long b = __double_as_longlong(v);
    const int lo = swap1((int)b), hi = swap1((int)(b >> 32));
    return __longlong_as_double(((long long)hi << 32) | (unsigned)lo);
}

// What two neighbouring lanes load together of their two atoms j (both lanes active): each 16 bytes of
// the even lane's atom, then of the odd lane's.  A load's cost is the cache lines that neighbouring
// lanes name, a lookup per clock: a lane alone needs two for its atom's 24 or 32 bytes, two together
// one for each of the two.  The lanes exchange halves when the values are used (registers still
// being loaded are not touched before).
struct alignas(8) Pos2 {
    double a, b;
};
template <bool PAIR>
struct GatherPos {  // position j of x: even lane (x, y), odd lane (y, z)
    Pos2 p, q;
    __device__ void load(const double* __restrict__ x, int j, bool odd)
    {
        const int jo = PAIR ? swap1(j) : j;
        p = *reinterpret_cast<const Pos2*>(x + 3 * (size_t)(odd ? jo : j) + odd);
        q = *reinterpret_cast<const Pos2*>(x + 3 * (size_t)(odd ? j : jo) + (PAIR ? odd : 1));
    }
    __device__ double3 get(bool odd) const
    {
        if (!PAIR) return make_double3(p.a, p.b, q.b);
        const double r = swap1(odd ? p.b : q.a);
        return make_double3(odd ? r : p.a, odd ? q.a : p.b, odd ? q.b : r);
    }
};
template <bool PAIR>
struct GatherRow {  // row j of four doubles
    double2 p, q;
    __device__ void load(const double2* __restrict__ rows, int j, bool odd)
    {
        const int jo = PAIR ? swap1(j) : j;
        p            = rows[2 * (size_t)(odd ? jo : j) + odd];
        q            = rows[2 * (size_t)(odd ? j : jo) + (PAIR ? odd : 1)];
    }
    __device__ void get(bool odd, double2* r0, double2* r1) const
    {
        if (!PAIR) {
            *r0 = p;
            *r1 = q;
            return;
        }
        double2 t = odd ? p : q;
        t.x       = swap1(t.x);
        t.y       = swap1(t.y);
        *r0       = odd ? t : p;
        *r1       = odd ? q : t;
    }
};

// ---------------------------------------------------------------- LJ (force_lj.c:17-206)
// One atom per LPA lanes.  STRICT: LPA == 1, reference order, no fma; HALF: strict half lists (the
// fast ones are k_force_lj_half's).
template <int LPA, bool STRICT, bool HALF, bool EV>
__global__ void __launch_bounds__(BLOCK) k_force_lj(int nlocal, const double* __restrict__ x,
    const int* __restrict__ type, int ntypes, Tables tab, int uniform,
    const int* __restrict__ neighbors, const int* __restrict__ numneigh, double* __restrict__ f,
    double* __restrict__ ev, Fuse fu)
{
    static_assert(!STRICT || LPA == 1, "the strict kernels sum in list order");
    static_assert(!HALF || STRICT, "fast half lists have a kernel of their own");
    __shared__ double s_tab[3][MAXTYPES2];
    __shared__ double s_red[16];
    if (!uniform) {
        const int nt2 = ntypes * ntypes;
        for (int k = threadIdx.x; k < nt2; k += blockDim.x) {
            s_tab[0][k] = tab.eps[k];
            s_tab[1][k] = tab.sig6[k];
            s_tab[2][k] = tab.cutf[k];
        }
        __syncthreads();
    }
    const int gid  = blockIdx.x * blockDim.x + threadIdx.x;
    const int i    = gid / LPA;
    const int lane = gid % LPA;
    const bool act = i < nlocal;
    double fix = 0, fiy = 0, fiz = 0, e = 0, w = 0;
    double v0[3] = {}, x0[3] = {};
    int ng = 0, g0 = 0;
    if (!HALF && fu.v && act && (lane == 0 || fu.gcnt)) fused_load<true>(fu, i, v0, &ng, &g0);
    if (act) {
        const double xt = x[3 * i], yt = x[3 * i + 1], zt = x[3 * i + 2];
        x0[0] = xt;
        x0[1] = yt;
        x0[2] = zt;
        const int ti    = uniform ? 0 : type[i];
        const int nn    = numneigh[i];
        const double eps0 = tab.eps[0], sig0 = tab.sig6[0], cut0 = tab.cutf[0];
        for (int k = lane; k < nn; k += LPA) {
            const int j = neighbors[(size_t)k * nlocal + i];
            double dx   = xt - x[3 * j];
            double dy   = yt - x[3 * j + 1];
            double dz   = zt - x[3 * j + 2];
            double rsq;
            if (STRICT) rsq = dx * dx + dy * dy + dz * dz;
            else rsq = fma(dx, dx, fma(dy, dy, dz * dz));
            double eps = eps0, sig6 = sig0, cutf = cut0;
            if (!uniform) {
                int tij = ti * ntypes + type[j];
                eps     = s_tab[0][tij];
                sig6    = s_tab[1][tij];
                cutf    = s_tab[2][tij];
            }
            if (rsq < cutf) {
                double sr2   = STRICT || EV ? 1.0 / rsq : recip_normal(rsq);
                double sr6   = sr2 * sr2 * sr2 * sig6;
                double force = 48.0 * sr6 * (sr6 - 0.5) * sr2 * eps;
                if (STRICT) {
                    fix += dx * force;
                    fiy += dy * force;
                    fiz += dz * force;
                } else {
                    fix = fma(dx, force, fix);
                    fiy = fma(dy, force, fiy);
                    fiz = fma(dz, force, fiz);
                }
                if (HALF && j < nlocal) {
                    atomicAdd(&f[3 * j], -(dx * force));
                    atomicAdd(&f[3 * j + 1], -(dy * force));
                    atomicAdd(&f[3 * j + 2], -(dz * force));
                }
                if (EV) {
                    double wgt = (HALF && j < nlocal) ? 1.0 : 0.5;
                    e += wgt * 4.0 * eps * sr6 * (sr6 - 1.0);
                    w += wgt * rsq * force;
                }
            }
        }
    }
    if (LPA > 1) {
        fix = group_sum<LPA>(fix);
        fiy = group_sum<LPA>(fiy);
        fiz = group_sum<LPA>(fiz);
    }
    if (act && lane == 0) {
        if (HALF) {
            atomicAdd(&f[3 * i], fix);
            atomicAdd(&f[3 * i + 1], fiy);
            atomicAdd(&f[3 * i + 2], fiz);
        } else {
            f[3 * i]     = fix;
            f[3 * i + 1] = fiy;
            f[3 * i + 2] = fiz;
        }
    }
    if (!HALF && fu.v && act && (lane == 0 || fu.gcnt))
        fused_integrate<LPA, true>(fu, nlocal, i, lane, v0, x0, ng, g0, fix, fiy, fiz);
    if (EV) {
        double be = block_sum(e, s_red);
        double bw = block_sum(w, s_red);
        if (threadIdx.x == 0) {
            atomicAdd(&ev[0], be);
            atomicAdd(&ev[1], bw);
        }
    }
}

// ---------------------------------------------------------------- staged neighbour positions
// A large system's force pass is bound by the texture path's address rate: two loads of 64 different
// lines for the positions of 64 pairs.  So a block of STAGE_T threads takes STAGE_A consecutive atoms
// (of one region of the box in the lattice's order), reads the positions of all the distinct atoms
// that its lists name into LDS once, and its pairs read them there.  Which atoms those are, and each
// list entry's place among them, is worked out when the list is built (k_stage_build).  Both are
// only hints: a pair uses the staged position only if the staged atom is the one its list entry
// names, and loads it from memory otherwise (a list written by someone else, a region with more than
// STAGE_CAP distinct neighbours).  1.05 M atoms: 276 us per call with the positions gathered, 192
// staged, bound by HBM (676 MB a call at 3.5 TB/s, 480 of them list and hints; VALU 60 %).  The two blocks
// that a CU's LDS and waves hold set STAGE_CAP; a 256-atom lattice block names 1300 - 1700.  Blocks
// of 512 threads and 128 atoms took the same, three or four sets of entries ahead too.
constexpr int STAGE_T = 1024, STAGE_A = 256, STAGE_CAP = 2000, STAGE_LOG = 10;

// tab: STAGE_CAP atoms per block, tab_n: how many (0: too many), hint[k * nlocal + i]: the place.
// Atoms are taken by pages of 64: a block's neighbours lie in a hundred or two of them, found in a
// small hash table; a page's members are bits of a word, so that a list entry is entered with an OR
// and an atom's place is its page's first plus the members below it (pages in table order).  LDS and
// the lists' two readings bound it: 252 us at 1.05 M atoms (800 us for the list itself), 17 more where
// every entry is an OR without the read before it.
__global__ void __launch_bounds__(STAGE_T) k_stage_build(int nlocal,
    const int* __restrict__ neighbors, const int* __restrict__ numneigh, int maxneighs,
    int* __restrict__ tab, int* __restrict__ tab_n, unsigned short* __restrict__ hint,
    int* __restrict__ overflows)
{
    constexpr int SLOTS = STAGE_T, LPA = STAGE_T / STAGE_A, PROBES = 16;
    __shared__ int s_page[SLOTS];
    __shared__ unsigned long long s_bits[SLOTS];
    __shared__ unsigned short s_first[SLOTS];
    __shared__ int s_scan[33], s_bad;
    s_page[threadIdx.x] = -1;
    s_bits[threadIdx.x] = 0ull;
    if (threadIdx.x == 0) s_bad = 0;
    __syncthreads();
    const int i    = blockIdx.x * STAGE_A + threadIdx.x / LPA;
    const int lane = threadIdx.x % LPA;
    const int nn   = i < nlocal ? min(numneigh[i], maxneighs) : 0;
    auto start     = [](int p) { return ((unsigned)p * 2654435761u) >> (32 - STAGE_LOG); };
    auto enter = [&](int j) {
        const int p = j >> 6;
        unsigned h  = start(p);
        int left    = PROBES;
        for (; left; left--, h = (h + 1) & (SLOTS - 1)) {
            int key = __hip_atomic_load(&s_page[h], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
            if (key == -1) {
                key = atomicCAS(&s_page[h], -1, p);
                if (key == -1) key = p;
            }
            if (key == p) break;
        }
        // (most entries name an atom that is there already: a read instead of an atomic)
        const unsigned long long bit = 1ull << (j & 63);
        if (!left) s_bad = 1;
        else if (!(__hip_atomic_load(&s_bits[h], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP) & bit))
            atomicOr(&s_bits[h], bit);
    };
    // (list entries two ahead in two registers: 305 -> 252 us; four: 255)
    auto walk = [&](auto use) {
        ListWalk<LPA> list(neighbors, nlocal, i < nlocal ? i : 0, lane, nn);
        int ja = list.next(lane), jb = list.next(lane + LPA);
        for (int k = lane; k < nn; k += 2 * LPA) {
            const int j0 = ja;
            ja           = list.next(k + 2 * LPA);
            use(k, j0);
            const int j1 = jb;
            jb           = list.next(k + 3 * LPA);
            if (k + LPA < nn) use(k + LPA, j1);
        }
    };
    walk([&](int, int j) { enter(j); });
    __syncthreads();
    unsigned long long bits = s_bits[threadIdx.x];
    int n;
    int at = block_excl_scan(__popcll(bits), s_scan, &n);
    const bool ok = n <= STAGE_CAP && !s_bad;
    if (threadIdx.x == 0) {
        tab_n[blockIdx.x] = ok ? n : 0;
        if (!ok) atomicAdd(overflows, 1);
    }
    if (!ok) return;
    s_first[threadIdx.x] = (unsigned short)at;
    const int page = s_page[threadIdx.x];
    for (; bits; bits &= bits - 1)
        tab[(size_t)blockIdx.x * STAGE_CAP + at++] = page * 64 + __ffsll((long long)bits) - 1;
    __syncthreads();
    auto place = [&](int j) {
        const int p = j >> 6;
        unsigned h  = start(p);
        for (int left = PROBES; left > 1 && s_page[h] != p; left--)
            h = (h + 1) & (SLOTS - 1);
        return (unsigned short)(s_first[h] + __popcll(s_bits[h] & ((1ull << (j & 63)) - 1)));
    };
    walk([&](int k, int j) { hint[(size_t)k * nlocal + i] = place(j); });
}

// LJ, full lists, fast, without energies: the pairs, their order and arithmetic are those of
// k_force_lj with four lanes per atom.
template <bool UNIFORM>
__global__ void __launch_bounds__(STAGE_T) k_force_lj_staged(int nlocal, int nall, int nblocks,
    const double* __restrict__ x, const int* __restrict__ type, int ntypes, Tables tab,
    const int* __restrict__ neighbors, const int* __restrict__ numneigh, int maxneighs,
    const int* __restrict__ stage, const int* __restrict__ stage_n,
    const unsigned short* __restrict__ hint, double* __restrict__ f, Fuse fu)
{
    constexpr int LPA = STAGE_T / STAGE_A;
    __shared__ double s_pos[3 * STAGE_CAP + 3];
    __shared__ int s_key[STAGE_CAP + 1];  // the one behind the last: no atom
    __shared__ unsigned char s_type[UNIFORM ? 1 : STAGE_CAP + 1];
    __shared__ double s_tab[3][UNIFORM ? 1 : MAXTYPES2];
    // blocks of one XCD adjacent (the grid is a multiple of 8)
    const int per = gridDim.x >> 3;
    const int b   = (blockIdx.x & 7) * per + (blockIdx.x >> 3);
    if (b >= nblocks) return;
    if (!UNIFORM)
        for (int k = threadIdx.x; k < ntypes * ntypes; k += STAGE_T) {
            s_tab[0][k] = tab.eps[k];
            s_tab[1][k] = tab.sig6[k];
            s_tab[2][k] = tab.cutf[k];
        }
    const int ns = stage_n[b];
    if (threadIdx.x == 0) s_key[ns] = -1;
    for (int k = threadIdx.x; k < ns; k += STAGE_T) {
        const int j = stage[(size_t)b * STAGE_CAP + k];
        const bool in = (unsigned)j < (unsigned)nall;
        s_key[k]      = in ? j : -1;
        if (in) {
            s_pos[3 * k]     = x[3 * j];
            s_pos[3 * k + 1] = x[3 * j + 1];
            s_pos[3 * k + 2] = x[3 * j + 2];
            if (!UNIFORM) s_type[k] = (unsigned char)type[j];
        }
    }
    const int i    = b * STAGE_A + threadIdx.x / LPA;
    const int lane = threadIdx.x % LPA;
    const bool act = i < nlocal;
    double fix = 0, fiy = 0, fiz = 0;
    double v0[3] = {}, x0[3] = {};
    int ng = 0, g0 = 0, nn = 0, ti = 0;
    if (act) {
        if (fu.v && (lane == 0 || fu.gcnt)) fused_load<true>(fu, i, v0, &ng, &g0);
        x0[0] = x[3 * i];
        x0[1] = x[3 * i + 1];
        x0[2] = x[3 * i + 2];
        nn    = numneigh[i];
        if (!UNIFORM) ti = type[i] * ntypes;
    }
    __syncthreads();
    // Entries and hints two iterations ahead, in two sets of registers.  The loads are unconditional
    // (a lane behind its list's end reads the row's first entry, as all such lanes do) and a memory
    // fallback waits where it is, so that the waits in the loop are for the older set alone: with a
    // branch around the loads the compiler waited for all of them in every iteration (207 us).
    const unsigned at = lane * (unsigned)nlocal + (act ? i : 0);
    auto next = [&](int k0, int* j, unsigned* h) {
        const unsigned e = k0 + lane < nn ? at : 0;
        const size_t row = (size_t)min(k0, maxneighs - 1) * nlocal;
        *j = *(const int*)((const char*)(neighbors + row) + 4u * e);
        *h = *(const unsigned short*)((const char*)(hint + row) + 2u * e);
    };
    auto pair = [&](int k0, int* pj, unsigned* ph) {
        const int j      = *pj;
        const unsigned h = min(*ph, (unsigned)ns);
        double xj = s_pos[3 * h], yj = s_pos[3 * h + 1], zj = s_pos[3 * h + 2];
        int tj = 0;
        if (!UNIFORM) tj = s_type[h];
        const int key = s_key[h];
        next(k0 + 2 * LPA, pj, ph);
        // (kept as LDS reads: the compiler would merge them with the loads below into flat loads,
        // which take the texture path again)
        asm volatile("" : "+v"(xj), "+v"(yj), "+v"(zj));
        const bool in = k0 + lane < nn;
        if (__builtin_expect(in && key != j, 0)) {
            xj = x[3 * j];
            yj = x[3 * j + 1];
            zj = x[3 * j + 2];
            if (!UNIFORM) tj = type[j];
            asm volatile("" : "+v"(xj), "+v"(yj), "+v"(zj), "+v"(tj));
        }
        const double dx = x0[0] - xj, dy = x0[1] - yj, dz = x0[2] - zj;
        const double rsq  = fma(dx, dx, fma(dy, dy, dz * dz));
        const double cutf = UNIFORM ? tab.cutf[0] : s_tab[2][ti + tj];
        if (in && rsq < cutf) {
            const double eps   = UNIFORM ? tab.eps[0] : s_tab[0][ti + tj];
            const double sig6  = UNIFORM ? tab.sig6[0] : s_tab[1][ti + tj];
            const double sr2   = recip_normal(rsq);
            const double sr6   = sr2 * sr2 * sr2 * sig6;
            const double force = 48.0 * sr6 * (sr6 - 0.5) * sr2 * eps;
            fix                = fma(dx, force, fix);
            fiy                = fma(dy, force, fiy);
            fiz                = fma(dz, force, fiz);
        }
    };
    int j1, j2;
    unsigned h1, h2;
    next(0, &j1, &h1);
    next(LPA, &j2, &h2);
    for (int k0 = 0; k0 + lane < nn; k0 += 2 * LPA) {
        pair(k0, &j1, &h1);
        pair(k0 + LPA, &j2, &h2);
    }
    fix = group_sum<LPA>(fix);
    fiy = group_sum<LPA>(fiy);
    fiz = group_sum<LPA>(fiz);
    if (act && lane == 0) {
        f[3 * i]     = fix;
        f[3 * i + 1] = fiy;
        f[3 * i + 2] = fiz;
    }
    if (fu.v && act && (lane == 0 || fu.gcnt))
        fused_integrate<LPA, true>(fu, nlocal, i, lane, v0, x0, ng, g0, fix, fiy, fiz);
}

// Half lists, fast: a block takes HALF_T / LPA consecutive atoms (of one region of the box, in the
// lattice's or the bin sort's order) and adds the forces on their listed neighbours in LDS, those
// of its own atoms in place, those of other atoms in a hash table keyed by the atom, and only then
// adds each touched atom to memory once.  One FP64 atomic per pair and axis to memory instead took
// 121 us a call for 35,700 atoms (1.4M pairs), nearly all of it the atomics; this takes
// 18.5 us and 5.3 for the gather of the accumulators (with the integration).
// LDS atomics and the latency of the list's loads bound it.  A pair that finds no slot within
// HALF_PROBE tries adds to memory directly.  acc: zero on entry.
// fghost: the ghosts' rows of the forces, which are zero (cleared here, beside the lists' loads; as more
// blocks of k_take_half it cost 0.8 us more at 6912 atoms).
constexpr int HALF_T = 1024, HALF_PROBE = 8;

template <int LPA, bool EV>
__global__ void __launch_bounds__(HALF_T) k_force_lj_half(int nlocal, const double* __restrict__ x,
    const int* __restrict__ type, int ntypes, Tables tab, int uniform,
    const int* __restrict__ neighbors, const int* __restrict__ numneigh, double* __restrict__ acc,
    double* __restrict__ ev, int nghost, double* __restrict__ fghost)
{
    constexpr int A = HALF_T / LPA, LOG = LPA <= 8 ? 11 : 10, SLOTS = 1 << LOG;
    __shared__ double s_tab[3][MAXTYPES2];
    __shared__ double s_red[16];
    __shared__ int s_key[SLOTS];
    __shared__ double s_f[3 * SLOTS];
    __shared__ double s_own[3 * A];
    if (!uniform)
        for (int k = threadIdx.x; k < ntypes * ntypes; k += HALF_T) {
            s_tab[0][k] = tab.eps[k];
            s_tab[1][k] = tab.sig6[k];
            s_tab[2][k] = tab.cutf[k];
        }
    for (int k = threadIdx.x; k < SLOTS; k += HALF_T)
        s_key[k] = -1;
    for (int k = threadIdx.x; k < 3 * SLOTS; k += HALF_T)
        s_f[k] = 0.0;
    for (int k = threadIdx.x; k < 3 * A; k += HALF_T)
        s_own[k] = 0.0;
    for (int k = blockIdx.x * HALF_T + threadIdx.x; k < 3 * nghost; k += gridDim.x * HALF_T)
        fghost[k] = 0.0;
    __syncthreads();
    const int i0   = blockIdx.x * A;
    const int i    = i0 + threadIdx.x / LPA;
    const int lane = threadIdx.x % LPA;
    double fix = 0, fiy = 0, fiz = 0, e = 0, w = 0;
    if (i < nlocal) {
        const double xt = x[3 * i], yt = x[3 * i + 1], zt = x[3 * i + 2];
        const int ti    = uniform ? 0 : type[i];
        const int nn    = numneigh[i];
        const double eps0 = tab.eps[0], sig0 = tab.sig6[0], cut0 = tab.cutf[0];
        for (int k = lane; k < nn; k += LPA) {
            const int j      = neighbors[(size_t)k * nlocal + i];
            const double dx  = xt - x[3 * j];
            const double dy  = yt - x[3 * j + 1];
            const double dz  = zt - x[3 * j + 2];
            const double rsq = fma(dx, dx, fma(dy, dy, dz * dz));
            double eps = eps0, sig6 = sig0, cutf = cut0;
            if (!uniform) {
                const int tij = ti * ntypes + type[j];
                eps           = s_tab[0][tij];
                sig6          = s_tab[1][tij];
                cutf          = s_tab[2][tij];
            }
            if (!(rsq < cutf)) continue;
            const double sr2   = EV ? 1.0 / rsq : recip_normal(rsq);
            const double sr6   = sr2 * sr2 * sr2 * sig6;
            const double force = 48.0 * sr6 * (sr6 - 0.5) * sr2 * eps;
            fix = fma(dx, force, fix);
            fiy = fma(dy, force, fiy);
            fiz = fma(dz, force, fiz);
            if (EV) {
                const double wgt = j < nlocal ? 1.0 : 0.5;
                e += wgt * 4.0 * eps * sr6 * (sr6 - 1.0);
                w += wgt * rsq * force;
            }
            if (j >= nlocal) continue;
            double* dst = nullptr;
            if (j >= i0 && j < i0 + A) {
                dst = &s_own[3 * (j - i0)];
            } else {
                unsigned h = ((unsigned)j * 2654435761u) >> (32 - LOG);
                for (int p = 0; p < HALF_PROBE && !dst; p++, h = (h + 1) & (SLOTS - 1)) {
                    int key = __hip_atomic_load(&s_key[h], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
                    if (key == -1) {
                        key = atomicCAS(&s_key[h], -1, j);
                        if (key == -1) key = j;
                    }
                    if (key == j) dst = &s_f[3 * h];
                }
            }
            if (dst) {
                atomicAdd(dst, -(dx * force));
                atomicAdd(dst + 1, -(dy * force));
                atomicAdd(dst + 2, -(dz * force));
            } else {
                atomicAdd(&acc[3 * j], -(dx * force));
                atomicAdd(&acc[3 * j + 1], -(dy * force));
                atomicAdd(&acc[3 * j + 2], -(dz * force));
            }
        }
    }
    fix = group_sum<LPA>(fix);
    fiy = group_sum<LPA>(fiy);
    fiz = group_sum<LPA>(fiz);
    if (i < nlocal && lane == 0) {
        double* own = &s_own[3 * (i - i0)];
        atomicAdd(own, fix);
        atomicAdd(own + 1, fiy);
        atomicAdd(own + 2, fiz);
    }
    __syncthreads();
    for (int k = threadIdx.x; k < 3 * A; k += HALF_T)
        if (3 * i0 + k < 3 * nlocal) atomicAdd(&acc[3 * i0 + k], s_own[k]);
    for (int k = threadIdx.x; k < 3 * SLOTS; k += HALF_T) {
        const int j = s_key[k / 3];
        if (j >= 0) atomicAdd(&acc[3 * j + k % 3], s_f[k]);
    }
    if (EV) {
        const double be = block_sum(e, s_red);
        const double bw = block_sum(w, s_red);
        if (threadIdx.x == 0) {
            atomicAdd(&ev[0], be);
            atomicAdd(&ev[1], bw);
        }
    }
}

// The half list's total forces from the accumulators, which are cleared for the next call; with v
// set also the kicks, the drift and the ghosts of fused_integrate (in place: nothing else reads
// the positions).
__global__ void k_take_half(int nlocal, double* __restrict__ acc, double* __restrict__ f, double* x,
    Fuse fu)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= nlocal) return;
    double fr[3];
#pragma unroll
    for (int d = 0; d < 3; d++) {
        fr[d]          = acc[3 * i + d];
        acc[3 * i + d] = 0.0;
        f[3 * i + d]   = fr[d];
    }
    if (!fu.v) return;
    double v0[3];
    int ng = 0, g0 = 0;
    fused_load<true>(fu, i, v0, &ng, &g0);
    const double x0[3] = { x[3 * i], x[3 * i + 1], x[3 * i + 2] };
    fused_integrate<1, true>(fu, nlocal, i, 0, v0, x0, ng, g0, fr[0], fr[1], fr[2]);
}

// ---------------------------------------------------------------- EAM (force_eam.c:19-228)
// Spline knot of a pair distance (force_eam.c:72-76, 154-158): row m and offset p in [0, 1].
__device__ inline int eam_knot(double r, double rdr, int nr, double* p)
{
    double pp = r * rdr + 1.0;
    int m     = (int)pp;
    m         = m < nr - 1 ? m : nr - 1;
    pp -= m;
    *p = pp < 1.0 ? pp : 1.0;
    return m;
}

// rho_j(r) from the value coefficients (c3..c6) of its row (force_eam.c:85-88)
__device__ inline double eam_rho(const double* c, double p)
{
    return ((c[0] * p + c[1]) * p + c[2]) * p + c[3];
}

// The pair force over r (force_eam.c:188-206) from the derivative coefficients c0..c2 of the rho
// row (cr) and the full z2r row (cz); phi for the energy
__device__ inline double eam_fpair(const double* cr, const double* cz, double p, double recip,
    double fpi, double fpj, double* phi_out)
{
    double rhoip = (cr[0] * p + cr[1]) * p + cr[2];
    double z2p   = (cz[0] * p + cz[1]) * p + cz[2];
    double z2    = ((cz[3] * p + cz[4]) * p + cz[5]) * p + cz[6];
    double phi   = z2 * recip;
    double phip  = z2p * recip - phi * recip;
    double psip  = fpi * rhoip + fpj * rhoip + phip;
    *phi_out     = phi;
    return -psip * recip;
}

template <int LPA, bool STRICT, bool EV>
__global__ void __launch_bounds__(BLOCK) k_eam_density(int nlocal, const double* __restrict__ x,
    const int* __restrict__ neighbors, const int* __restrict__ numneigh, double cutforcesq,
    const double* __restrict__ rs, const double* __restrict__ fs, int nr, int nrho, double rdr,
    double rdrho, double* __restrict__ fp, double* __restrict__ ev, double* __restrict__ eatom,
    const int* __restrict__ gcnt, const int* __restrict__ goff)
{
    __shared__ double s_red[16];
    const int gid  = blockIdx.x * blockDim.x + threadIdx.x;
    const int i    = gid / LPA;
    const int lane = gid % LPA;
    const bool act = i < nlocal;
    double rhoi    = 0, e = 0;
    int ng = 0, g0 = 0;
    if (act) {
        if (gcnt) {
            ng = gcnt[i];
            g0 = goff[i];
        }
        const double xt = x[3 * i], yt = x[3 * i + 1], zt = x[3 * i + 2];
        const int nn    = numneigh[i];
        for (int k = lane; k < nn; k += LPA) {
            const int j = neighbors[(size_t)k * nlocal + i];
            double dx   = xt - x[3 * j];
            double dy   = yt - x[3 * j + 1];
            double dz   = zt - x[3 * j + 2];
            double rsq  = STRICT ? dx * dx + dy * dy + dz * dz : fma(dx, dx, fma(dy, dy, dz * dz));
            if (rsq < cutforcesq) {
                double p;
                const int m = eam_knot(sqrt(rsq), rdr, nr, &p);
                rhoi += eam_rho(rs + m * 7 + 3, p);
            }
        }
    }
    if (LPA > 1) rhoi = group_sum<LPA>(rhoi);
    if (act && (lane == 0 || lane < ng)) {
        double p = 1.0 * rhoi * rdrho + 1.0;
        int m    = (int)p;
        m        = m < nrho - 1 ? m : nrho - 1;
        m        = m > 1 ? m : 1;
        p -= m;
        p                = p < 1.0 ? p : 1.0;
        const double* c  = fs + m * 7;
        const double fpi = (c[0] * p + c[1]) * p + c[2];
        // the atom's images too (else k_ghost_copy copies them)
        for (int k = lane; k < ng; k += LPA)
            fp[nlocal + g0 + k] = fpi;
        if (lane == 0) fp[i] = fpi;
        if (EV && lane == 0) {
            e = ((c[3] * p + c[4]) * p + c[5]) * p + c[6];
            if (eatom) eatom[i] = e;
        }
    }
    if (EV) {
        double be = block_sum(e, s_red);
        if (threadIdx.x == 0) atomicAdd(&ev[0], be);
    }
}

__global__ void k_ghost_copy(int nlocal, int nghost, double* __restrict__ a,
    const int* __restrict__ border_map)
{
    int g = blockIdx.x * blockDim.x + threadIdx.x;
    if (g >= nghost) return;
    a[nlocal + g] = a[border_map[g]];
}

// The ghosts' rows (position, F' of the owner) of the table passes
__global__ void k_ghost_rows(int nlocal, int nghost, const double* __restrict__ x,
    double2* __restrict__ xf, const int* __restrict__ border_map)
{
    const int g = blockIdx.x * blockDim.x + threadIdx.x;
    if (g >= nghost) return;
    const size_t i = (size_t)nlocal + g;
    xf[2 * i]      = make_double2(x[3 * i], x[3 * i + 1]);
    xf[2 * i + 1]  = make_double2(x[3 * i + 2], xf[2 * (size_t)border_map[g] + 1].y);
}

// GH: with the ghosts' positions (a variant of its own: in one kernel with the other the energy pass of
// 442,000 atoms took 234 us for 226).
template <int LPA, bool STRICT, bool EV, bool GH>
__global__ void __launch_bounds__(BLOCK) k_eam_force(int nlocal, const double* __restrict__ x,
    const int* __restrict__ neighbors, const int* __restrict__ numneigh, double cutforcesq,
    const double* __restrict__ rs, const double* __restrict__ zs, int nr, double rdr,
    const double* __restrict__ fp, double* __restrict__ f, double* __restrict__ ev,
    double* __restrict__ eatom, FuseOf<GH> fu)
{
    __shared__ double s_red[16];
    const int gid  = blockIdx.x * blockDim.x + threadIdx.x;
    const int i    = gid / LPA;
    const int lane = gid % LPA;
    const bool act = i < nlocal;
    double fix = 0, fiy = 0, fiz = 0, e = 0, w = 0;
    double v0[3] = {}, x0[3] = {};
    int ng = 0, g0 = 0;
    if (fu.v && act && (lane == 0 || GH)) fused_load<GH>(fu, i, v0, &ng, &g0);
    if (act) {
        const double xt = x[3 * i], yt = x[3 * i + 1], zt = x[3 * i + 2];
        x0[0] = xt;
        x0[1] = yt;
        x0[2] = zt;
        const double fpi = fp[i];
        const int nn     = numneigh[i];
        for (int k = lane; k < nn; k += LPA) {
            const int j = neighbors[(size_t)k * nlocal + i];
            double dx   = xt - x[3 * j];
            double dy   = yt - x[3 * j + 1];
            double dz   = zt - x[3 * j + 2];
            double rsq  = STRICT ? dx * dx + dy * dy + dz * dz : fma(dx, dx, fma(dy, dy, dz * dz));
            if (rsq < cutforcesq) {
                double r, recip;
                if (STRICT || EV) {
                    r     = sqrt(rsq);
                    recip = 1.0 / r;
                } else {
                    recip = root_recip_normal(rsq, &r);
                }
                double p, phi;
                const int m        = eam_knot(r, rdr, nr, &p);
                const double fpair = eam_fpair(rs + m * 7, zs + m * 7, p, recip, fpi, fp[j], &phi);
                if (STRICT) {
                    fix += dx * fpair;
                    fiy += dy * fpair;
                    fiz += dz * fpair;
                } else {
                    fix = fma(dx, fpair, fix);
                    fiy = fma(dy, fpair, fiy);
                    fiz = fma(dz, fpair, fiz);
                }
                if (EV) {
                    e += 0.5 * phi;
                    w += 0.5 * rsq * fpair;
                }
            }
        }
    }
    if (LPA > 1) {
        fix = group_sum<LPA>(fix);
        fiy = group_sum<LPA>(fiy);
        fiz = group_sum<LPA>(fiz);
    }
    double ea = 0.0;
    if (EV && eatom) ea = LPA > 1 ? group_sum<LPA>(e) : e;
    if (act && lane == 0) {
        f[3 * i]     = fix;
        f[3 * i + 1] = fiy;
        f[3 * i + 2] = fiz;
        if (EV && eatom) eatom[i] += ea;
    }
    if (fu.v && act && (lane == 0 || GH))
        fused_integrate<LPA, GH>(fu, nlocal, i, lane, v0, x0, ng, g0, fix, fiy, fiz);
    if (EV) {
        double be = block_sum(e, s_red);
        double bw = block_sum(w, s_red);
        if (threadIdx.x == 0) {
            atomicAdd(&ev[0], be);
            atomicAdd(&ev[1], bw);
        }
    }
}

// The same two passes with the spline rows staged in LDS (no energy): the per-pair table rows
// (32 B in the density pass, 80 B in the force pass) then come from LDS, and the texture path
// serves only the neighbour gathers.  The tables take 64 KB and 160,000 B for nr <= TAB_NR, so
// the blocks are persistent: TAB_BLOCK threads, one block per 64 KB / 160 KB of a CU's LDS,
// each over a contiguous range of atoms (ranges of one XCD adjacent, as in the cluster-pair
// kernels).  Operations and their order are those of k_eam_density / k_eam_force.
// The density pass leaves a row of 32 bytes per atom, its position and F', for the force pass: one
// aligned row in one cache line instead of a position and an F'.  Both passes load list entries two
// or three pairs ahead and positions or rows one, in two sets of registers, and two neighbouring
// lanes load their two atoms together (GatherPos, GatherRow): they were bound by the L1's lookups,
// one per lane and load, and the force pass (one block per CU, 4 waves per SIMD) by latency.  Force
// pass at 1.05 M atoms 451 -> 288 us (377 loading ahead, 343 with rows, 299 without branches around
// the list loads), at 131 k 53 -> 41; density 255 -> 262 (the rows cost 6; loads ahead alone 270) and
// 30 -> 28.  Bound now: FP64 instructions and lookups alike.
constexpr int TAB_BLOCK = 1024;
constexpr int TAB_NR    = 2000;

template <int LPA, bool STRICT>
__global__ void __launch_bounds__(TAB_BLOCK) k_eam_density_tab(int nlocal, int per_block,
    const double* __restrict__ x, const int* __restrict__ neighbors,
    const int* __restrict__ numneigh, double cutforcesq, const double* __restrict__ rs,
    const double* __restrict__ fs, int nr, int nrho, double rdr, double rdrho,
    double2* __restrict__ xf)
{
    __shared__ double s_rs[TAB_NR * 4];  // value coefficients c3..c6 of each rho row
    for (int k = threadIdx.x; k < nr * 4; k += TAB_BLOCK)
        s_rs[k] = rs[(k >> 2) * 7 + 3 + (k & 3)];
    __syncthreads();
    const int per   = gridDim.x >> 3;
    const int lb    = (blockIdx.x & 7) * per + (blockIdx.x >> 3);
    const int begin = lb * per_block;
    const int end   = min(nlocal, begin + per_block);
    const int lane  = threadIdx.x % LPA;
    for (int base = begin; base < end; base += TAB_BLOCK / LPA) {
        const int i    = base + threadIdx.x / LPA;
        const bool act = i < end;
        double rhoi    = 0;
        if (act) {
            const double xt = x[3 * i], yt = x[3 * i + 1], zt = x[3 * i + 2];
            const int nn    = numneigh[i];
            // the list two or three entries ahead, positions one, in two sets of registers
            ListWalk<LPA> list(neighbors, nlocal, i, lane, nn);
            GatherPos<(LPA > 1)> pa, pb;
            const bool odd = LPA > 1 && (lane & 1);
            auto pair = [&](int k, const GatherPos<(LPA > 1)>& w) {
                const double3 q  = w.get(odd);
                const double dx  = xt - q.x;
                const double dy  = yt - q.y;
                const double dz  = zt - q.z;
                const double rsq = STRICT ? dx * dx + dy * dy + dz * dz
                                          : fma(dx, dx, fma(dy, dy, dz * dz));
                if (k < nn && rsq < cutforcesq) {
                    double p;
                    const int m = eam_knot(sqrt(rsq), rdr, nr, &p);
                    rhoi += eam_rho(s_rs + m * 4, p);
                }
            };
            int ja = list.next(lane), jb = list.next(lane + LPA);
            pa.load(x, nn > 0 ? ja : i, odd);
            ja = list.next(lane + 2 * LPA);
            for (int k = lane; k - lane < nn; k += 2 * LPA) {  // (all lanes of the atom)
                pb.load(x, jb, odd);
                jb = list.next(k + 3 * LPA);
                pair(k, pa);
                pa.load(x, ja, odd);
                ja = list.next(k + 4 * LPA);
                pair(k + LPA, pb);
            }
        }
        if (LPA > 1) rhoi = group_sum<LPA>(rhoi);
        if (act && lane == 0) {
            double p = 1.0 * rhoi * rdrho + 1.0;
            int m    = (int)p;
            m        = m < nrho - 1 ? m : nrho - 1;
            m        = m > 1 ? m : 1;
            p -= m;
            p               = p < 1.0 ? p : 1.0;
            const double* c = fs + m * 7;
            xf[2 * i]       = make_double2(x[3 * i], x[3 * i + 1]);
            xf[2 * i + 1]   = make_double2(x[3 * i + 2], (c[0] * p + c[1]) * p + c[2]);
        }
    }
}

// GH: with the ghosts' positions (a variant of its own: in one kernel with the other, the large
// systems' passes, which do not write them, ran 1 % slower).
template <int LPA, bool STRICT, bool GH>
__global__ void __launch_bounds__(TAB_BLOCK) k_eam_force_tab(int nlocal, int per_block,
    const double2* __restrict__ xf, const int* __restrict__ neighbors,
    const int* __restrict__ numneigh, double cutforcesq, const double* __restrict__ rs,
    const double* __restrict__ zs, int nr, double rdr, double* __restrict__ f, FuseOf<GH> fu)
{
    __shared__ double s_t[TAB_NR * 10];  // per row: rho c0..c2, then z2r c0..c6
    for (int k = threadIdx.x; k < nr * 10; k += TAB_BLOCK) {
        const int row = k / 10, c = k - 10 * row;
        s_t[k]        = c < 3 ? rs[row * 7 + c] : zs[row * 7 + c - 3];
    }
    __syncthreads();
    const int per   = gridDim.x >> 3;
    const int lb    = (blockIdx.x & 7) * per + (blockIdx.x >> 3);
    const int begin = lb * per_block;
    const int end   = min(nlocal, begin + per_block);
    const int lane  = threadIdx.x % LPA;
    for (int base = begin; base < end; base += TAB_BLOCK / LPA) {
        const int i    = base + threadIdx.x / LPA;
        const bool act = i < end;
        double fix = 0, fiy = 0, fiz = 0;
        double v0[3] = {}, x0[3] = {};
        int ng = 0, g0 = 0;
        if (fu.v && act && (lane == 0 || GH)) fused_load<GH>(fu, i, v0, &ng, &g0);
        if (act) {
            const double2 ri0 = xf[2 * i], ri1 = xf[2 * i + 1];
            const double xt = ri0.x, yt = ri0.y, zt = ri1.x;
            x0[0]            = xt;
            x0[1]            = yt;
            x0[2]            = zt;
            const double fpi = ri1.y;
            const int nn     = numneigh[i];
            // the list two or three entries ahead, rows one, in two sets of registers
            ListWalk<LPA> list(neighbors, nlocal, i, lane, nn);
            GatherRow<(LPA > 1)> ra, rb;
            const bool odd = LPA > 1 && (lane & 1);
            auto pair = [&](int k, const GatherRow<(LPA > 1)>& w) {
                double2 r0, r1;
                w.get(odd, &r0, &r1);
                const double dx  = xt - r0.x;
                const double dy  = yt - r0.y;
                const double dz  = zt - r1.x;
                const double rsq = STRICT ? dx * dx + dy * dy + dz * dz
                                          : fma(dx, dx, fma(dy, dy, dz * dz));
                if (k < nn && rsq < cutforcesq) {
                    double r, recip;
                    if (STRICT) {
                        r     = sqrt(rsq);
                        recip = 1.0 / r;
                    } else {
                        recip = root_recip_normal(rsq, &r);
                    }
                    double p, phi;
                    const int m        = eam_knot(r, rdr, nr, &p);
                    const double* row  = s_t + m * 10;
                    const double fpair = eam_fpair(row, row + 3, p, recip, fpi, r1.y, &phi);
                    if (STRICT) {
                        fix += dx * fpair;
                        fiy += dy * fpair;
                        fiz += dz * fpair;
                    } else {
                        fix = fma(dx, fpair, fix);
                        fiy = fma(dy, fpair, fiy);
                        fiz = fma(dz, fpair, fiz);
                    }
                }
            };
            int ja = list.next(lane), jb = list.next(lane + LPA);
            ra.load(xf, nn > 0 ? ja : i, odd);
            ja = list.next(lane + 2 * LPA);
            for (int k = lane; k - lane < nn; k += 2 * LPA) {  // (all lanes of the atom)
                rb.load(xf, jb, odd);
                jb = list.next(k + 3 * LPA);
                pair(k, ra);
                ra.load(xf, ja, odd);
                ja = list.next(k + 4 * LPA);
                pair(k + LPA, rb);
            }
        }
        if (LPA > 1) {
            fix = group_sum<LPA>(fix);
            fiy = group_sum<LPA>(fiy);
            fiz = group_sum<LPA>(fiz);
        }
        if (act && lane == 0) {
            f[3 * i]     = fix;
            f[3 * i + 1] = fiy;
            f[3 * i + 2] = fiz;
        }
        if (fu.v && act && (lane == 0 || GH))
            fused_integrate<LPA, GH>(fu, nlocal, i, lane, v0, x0, ng, g0, fix, fiy, fiz);
    }
}

// ---------------------------------------------------------------- thermo (thermo.c:76-81)
__global__ void __launch_bounds__(BLOCK) k_ksum_partial(int n, const double* __restrict__ v,
    double mass, double* __restrict__ part)
{
    __shared__ double s_red[16];
    double t = 0;
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x)
        t += (v[3 * i] * v[3 * i] + v[3 * i + 1] * v[3 * i + 1] + v[3 * i + 2] * v[3 * i + 2]) * mass;
    double b = block_sum(t, s_red);
    if (threadIdx.x == 0) part[blockIdx.x] = b;
}

__global__ void k_sum_partials(int n, double* __restrict__ part)
{
    __shared__ double s_red[16];
    double t = 0;
    for (int k = threadIdx.x; k < n; k += blockDim.x)
        t += part[k];
    double b = block_sum(t, s_red);
    if (threadIdx.x == 0) part[0] = b;
}

// ---------------------------------------------------------------- host helpers
bool ensure_status()
{
    if (!S.d_status) {
        MDG_HIP(hipMalloc(&S.d_status, 16 * sizeof(int)));
        MDG_HIP(hipHostMalloc(&S.h_status, 16 * sizeof(int), hipHostMallocDefault));
        MDG_HIP(hipHostMalloc(&S.h_flag, 16 * sizeof(int), hipHostMallocCoherent));
        MDG_HIP(hipMalloc(&S.d_ev, 4 * sizeof(double)));
        MDG_HIP(hipHostMalloc(&S.h_red, 4 * sizeof(double), hipHostMallocDefault));
        if (failed()) return false;
        fill_i32(S.d_status, 0, 16);
    }
    return !failed();
}

void stage_release()
{
    dfree(S.d_stage);
    dfree(S.d_stage_n);
    dfree(S.d_hint);
    S.d_stage = S.d_stage_n = nullptr;
    S.d_hint    = nullptr;
    S.cap_stage = S.cap_stage_n = S.cap_hint = 0;
    S.stage_nlocal = -1;
}

// For grow, which has no room left: a system that fits the device without the tables runs without them.
bool stage_give_back()
{
    if (!S.d_stage && !S.d_stage_n && !S.d_hint) return false;
    MDG_HIP(hipStreamSynchronize(stream()));
    stage_release();
    return !failed();
}

// Room for n elements, or false (no error: see stage_give_back).
template <typename T>
bool stage_room(T** p, size_t* cap, size_t n)
{
    if (n <= *cap) return true;
    dfree(*p);
    *cap = 0;
    if (hipMalloc((void**)p, n * sizeof(T)) != hipSuccess) {
        (void)hipGetLastError();
        *p = nullptr;
        return false;
    }
    *cap = n;
    return true;
}

void read_status()
{
    MDG_HIP(hipMemcpyAsync(S.h_status, S.d_status, 16 * sizeof(int), hipMemcpyDeviceToHost,
        stream()));
    MDG_HIP(hipStreamSynchronize(stream()));
}

void launch_ghost_copy(double* a, Atom* atom)
{
    if (atom->Nghost <= 0) return;
    k_ghost_copy<<<blocks_for(atom->Nghost, BLOCK), BLOCK, 0, stream()>>>(atom->Nlocal,
        atom->Nghost, a, atom->d_atom.border_map);
    MDG_LAUNCH_CHECK("ghost_copy");
}

}  // namespace

// ================================================================ C ABI
extern "C" {

void initDeviceGFX950(Parameter* param, Atom* atom, Neighbor* neighbor)
{
    if (failed() || !stream()) return;
    if (!ensure_status()) return;
    {
        int dev = 0, cu = 0;
        MDG_HIP(hipGetDevice(&dev));
        MDG_HIP(hipDeviceGetAttribute(&cu, hipDeviceAttributeMultiprocessorCount, dev));
        if (failed()) return;
        S.ncu = (cu + 7) / 8 * 8;
    }
    set_give_back(stage_give_back);
    DeviceAtom* d   = &atom->d_atom;
    memset(d, 0, sizeof(*d));
    S.cap_all = S.cap_v = 0;
    size_t n  = (size_t)(atom->Nmax > atom->Nlocal + atom->Nghost ? atom->Nmax
                                                                    : atom->Nlocal + atom->Nghost);
    size_t c  = 0;
    grow_n(&d->x, &c, 3 * n, 0);
    c = 0;
    grow_n(&d->fx, &c, 3 * n, 0);
    c = 0;
    grow_n(&d->type, &c, n, 0);
    c = 0;
    grow_n(&d->vx, &c, 3 * (size_t)atom->Nlocal + 3, 0);
    S.cap_v   = 3 * (size_t)atom->Nlocal + 3;
    S.cap_all = n;
    if (failed()) return;
    fill_f64(d->fx, 0.0, 3 * n);

    // type-pair tables (atom.c:125-142)
    S.ntypes = atom->ntypes;
    if (S.ntypes * S.ntypes > MAXTYPES2) {
        set_error(MDG_ERR_ARG, "ntypes %d > 8 not supported", S.ntypes);
        return;
    }
    S.uniform = true;
    for (int k = 0; k < S.ntypes * S.ntypes; k++) {
        S.tab.eps[k]  = atom->epsilon[k];
        S.tab.sig6[k] = atom->sigma6[k];
        S.tab.cutf[k] = atom->cutforcesq[k];
        S.tab.cutn[k] = atom->cutneighsq[k];
        if (atom->epsilon[k] != atom->epsilon[0] || atom->sigma6[k] != atom->sigma6[0] ||
            atom->cutforcesq[k] != atom->cutforcesq[0] || atom->cutneighsq[k] != atom->cutneighsq[0])
            S.uniform = false;
    }
    size_t t2 = (size_t)S.ntypes * S.ntypes;
    MDG_HIP(hipMalloc(&d->epsilon, t2 * sizeof(double)));
    MDG_HIP(hipMalloc(&d->sigma6, t2 * sizeof(double)));
    MDG_HIP(hipMalloc(&d->cutforcesq, t2 * sizeof(double)));
    MDG_HIP(hipMalloc(&d->cutneighsq, t2 * sizeof(double)));
    if (failed()) return;
    MDG_HIP(hipMemcpyAsync(d->epsilon, atom->epsilon, t2 * 8, hipMemcpyHostToDevice, stream()));
    MDG_HIP(hipMemcpyAsync(d->sigma6, atom->sigma6, t2 * 8, hipMemcpyHostToDevice, stream()));
    MDG_HIP(hipMemcpyAsync(d->cutforcesq, atom->cutforcesq, t2 * 8, hipMemcpyHostToDevice, stream()));
    MDG_HIP(hipMemcpyAsync(d->cutneighsq, atom->cutneighsq, t2 * 8, hipMemcpyHostToDevice, stream()));

    // neighbour list
    DeviceNeighbor* dn = &neighbor->d_neighbor;
    dn->neighbors      = nullptr;
    dn->numneigh       = nullptr;
    S.cap_nb = S.cap_numneigh = 0;
    grow_n(&dn->neighbors, &S.cap_nb, (size_t)atom->Nlocal * neighbor->maxneighs, 0);
    grow_n(&dn->numneigh, &S.cap_numneigh, (size_t)atom->Nlocal, 0);
    S.binned = false;
    S.ready  = true;
    S.gmap_nlocal  = -1;
    S.stage_nlocal = S.list_uses = S.last_uses = -1;
    S.stage_skip   = 0;
    copyDataToGFX950Device(param, atom);
}

void freeDeviceGFX950(Atom* atom, Neighbor* neighbor)
{
    if (S.d_status) (void)hipStreamSynchronize(stream());
    if (atom) {
        DeviceAtom* d = &atom->d_atom;
        dfree(d->x);
        dfree(d->vx);
        dfree(d->fx);
        dfree(d->type);
        dfree(d->border_map);
        dfree(d->epsilon);
        dfree(d->sigma6);
        dfree(d->cutforcesq);
        dfree(d->cutneighsq);
        memset(d, 0, sizeof(*d));
    }
    if (neighbor) {
        dfree(neighbor->d_neighbor.neighbors);
        dfree(neighbor->d_neighbor.numneigh);
        neighbor->d_neighbor.neighbors = nullptr;
        neighbor->d_neighbor.numneigh  = nullptr;
    }
    dfree(S.d_xn);
    dfree(S.d_acc);
    dfree(S.d_sort);
    dfree(S.d_sort_t);
    dfree(S.d_stencil);
    dfree(S.d_bin_of);
    dfree(S.d_bincount);
    dfree(S.d_binstart);
    dfree(S.d_binatoms);
    dfree(S.d_binslots);
    dfree(S.d_binplace);
    dfree(S.d_xs);
    dfree(S.d_eatom);
    dfree(S.d_gcnt);
    dfree(S.d_goff);
    dfree(S.d_pbc);
    stage_release();
    dfree(S.d_fp);
    dfree(S.d_rhor);
    dfree(S.d_frho);
    dfree(S.d_z2r);
    dfree(S.d_red);
    dfree(S.d_ev);
    dfree(S.d_status);
    if (S.h_status) (void)hipHostFree(S.h_status);
    if (S.h_flag) (void)hipHostFree(S.h_flag);
    if (S.h_red) (void)hipHostFree(S.h_red);
    S = State();
}

void uploadNeighborGFX950(Atom* atom, Neighbor* neighbor)
{
    if (failed() || !S.ready) return;
    const int nlocal = atom->Nlocal, mn = neighbor->maxneighs;
    grow_n(&neighbor->d_neighbor.neighbors, &S.cap_nb, (size_t)nlocal * mn, 0);
    grow_n(&neighbor->d_neighbor.numneigh, &S.cap_numneigh, (size_t)nlocal, 0);
    if (failed()) return;
    // the host list is AoS (neighbors[i * maxneighs + k]); the device list is SoA
    int* soa = (int*)malloc((size_t)nlocal * mn * sizeof(int) + 4);
    if (!soa) {
        set_error(MDG_ERR_CAPACITY, "uploadNeighborGFX950: host buffer");
        return;
    }
    for (int i = 0; i < nlocal; i++)
        for (int k = 0; k < neighbor->numneigh[i]; k++)
            soa[(size_t)k * nlocal + i] = neighbor->neighbors[(size_t)i * mn + k];
    MDG_HIP(hipMemcpyAsync(neighbor->d_neighbor.neighbors, soa, (size_t)nlocal * mn * sizeof(int),
        hipMemcpyHostToDevice, stream()));
    MDG_HIP(hipMemcpyAsync(neighbor->d_neighbor.numneigh, neighbor->numneigh,
        (size_t)nlocal * sizeof(int), hipMemcpyHostToDevice, stream()));
    MDG_HIP(hipStreamSynchronize(stream()));
    free(soa);
}

void copyDataToGFX950Device(Parameter* param, Atom* atom)
{
    (void)param;
    if (failed() || !S.ready) return;
    S.ghosts_current = false;
    size_t nall = (size_t)atom->Nlocal + atom->Nghost;
    DeviceAtom* d = &atom->d_atom;
    MDG_HIP(hipMemcpyAsync(d->x, atom->x, 3 * nall * sizeof(double), hipMemcpyHostToDevice, stream()));
    MDG_HIP(hipMemcpyAsync(d->vx, atom->vx, 3 * (size_t)atom->Nlocal * sizeof(double),
        hipMemcpyHostToDevice, stream()));
    MDG_HIP(hipMemcpyAsync(d->type, atom->type, nall * sizeof(int), hipMemcpyHostToDevice, stream()));
    MDG_HIP(hipStreamSynchronize(stream()));
}

void copyDataFromGFX950Device(Parameter* param, Atom* atom)
{
    (void)param;
    if (failed() || !S.ready) return;
    DeviceAtom* d = &atom->d_atom;
    size_t nl     = (size_t)atom->Nlocal;
    MDG_HIP(hipMemcpyAsync(atom->x, d->x, 3 * nl * sizeof(double), hipMemcpyDeviceToHost, stream()));
    MDG_HIP(hipMemcpyAsync(atom->vx, d->vx, 3 * nl * sizeof(double), hipMemcpyDeviceToHost, stream()));
    MDG_HIP(hipMemcpyAsync(atom->fx, d->fx, 3 * nl * sizeof(double), hipMemcpyDeviceToHost, stream()));
    MDG_HIP(hipMemcpyAsync(atom->type, d->type, nl * sizeof(int), hipMemcpyDeviceToHost, stream()));
    MDG_HIP(hipStreamSynchronize(stream()));
}

// setupNeighbor (neighbor.c:101-258), restated for the host; the stencil goes to the device.
void setupNeighborGFX950(Parameter* param)
{
    if (failed()) return;
    if (!ensure_status()) return;
    const double FACTOR = 0.999;
    double cutneigh     = param->cutneigh;
    double xprd = param->nx * param->lattice, yprd = param->ny * param->lattice,
           zprd = param->nz * param->lattice;
    double bs[3], inv[3];
    int nb[3];
    if (param->input_file != NULL) {
        double lo[3] = { param->xlo, param->ylo, param->zlo };
        double hi[3] = { param->xhi, param->yhi, param->zhi };
        xprd = param->xprd;
        yprd = param->yprd;
        zprd = param->zprd;
        for (int d = 0; d < 3; d++) {
            bs[d] = cutneigh * 0.5;
            nb[d] = (int)((hi[d] - lo[d]) / bs[d]);
            if (nb[d] == 0) nb[d] = 1;
            inv[d] = nb[d] / (hi[d] - lo[d]);
        }
    } else {
        const double neighscale = 5.0 / 6.0;
        int nxyz[3]             = { param->nx, param->ny, param->nz };
        double prd[3]           = { xprd, yprd, zprd };
        for (int d = 0; d < 3; d++) {
            double t = neighscale * nxyz[d];
            nb[d]    = (int)(t > 1 ? t : 1);
            bs[d]    = prd[d] / nb[d];
            inv[d]   = 1.0 / bs[d];
        }
    }
    int pad[3], next[3];
    for (int d = 0; d < 3; d++) {
        pad[d] = (int)(cutneigh * inv[d]);
        while (pad[d] * bs[d] < FACTOR * cutneigh)
            pad[d]++;
    }
    for (int d = 0; d < 3; d++) {
        next[d] = (int)(cutneigh * inv[d]);
        while (next[d] * bs[d] < FACTOR * cutneigh) {
            next[d]++;
            pad[d]++;
        }
    }
    int mb[3];
    for (int d = 0; d < 3; d++) {
        mb[d] = nb[d] + 4 * pad[d];
        if (mb[d] < 1) mb[d] = 1;
    }
    double cutneighsq = cutneigh * cutneigh;
    int st[1024];
    int ns = 0;
    for (int k = -next[2]; k <= next[2]; k++)
        for (int j = -next[1]; j <= next[1]; j++)
            for (int i = -next[0]; i <= next[0]; i++) {
                int ijk[3] = { i, j, k };
                double dd[3];
                for (int d = 0; d < 3; d++)
                    dd[d] = ijk[d] > 0 ? (ijk[d] - 1) * bs[d] : (ijk[d] == 0 ? 0.0 : (ijk[d] + 1) * bs[d]);
                double dist = dd[0] * dd[0] + dd[1] * dd[1] + dd[2] * dd[2];
                if (dist < cutneighsq) {
                    if (ns >= 1024) {
                        set_error(MDG_ERR_ARG, "stencil larger than 1024 bins");
                        return;
                    }
                    st[ns++] = k * mb[1] * mb[0] + j * mb[0] + i;
                }
            }
    for (int d = 0; d < 3; d++) {
        S.binsize[d]  = bs[d];
        S.g.bininv[d] = inv[d];
        S.pad[d]      = pad[d];
        S.g.off[d]    = fabs(0.0 - pad[d] * bs[d]) + 1e-9;
    }
    S.g.mbinx  = mb[0];
    S.g.mbiny  = mb[1];
    S.g.mbinz  = mb[2];
    S.g.mbins  = mb[0] * mb[1] * mb[2];
    S.nstencil = ns;
    S.prd[0]   = param->xprd;
    S.prd[1]   = param->yprd;
    S.prd[2]   = param->zprd;
    S.cutneigh = cutneigh;
    grow_n(&S.d_stencil, &S.stencil_cap, (size_t)ns, 0);
    if (failed()) return;
    MDG_HIP(hipMemcpyAsync(S.d_stencil, st, ns * sizeof(int), hipMemcpyHostToDevice, stream()));
    MDG_HIP(hipStreamSynchronize(stream()));
    S.binned = false;
}

// Room for the bins of n atoms
static void grow_bins(size_t n)
{
    const size_t mb = (size_t)S.g.mbins, cap0 = S.cap_bins;
    grow_n(&S.d_binplace, &S.cap_binplace, n, 0);
    grow_n(&S.d_xs, &S.cap_xs, 3 * n, 0);
    grow_n(&S.d_bin_of, &S.cap_bin_of, n, 0);
    grow_n(&S.d_bincount, &S.cap_bins, mb + 1, 0);
    grow_n(&S.d_binstart, &S.cap_binstart, mb + 1, 0);
    grow_n(&S.d_binatoms, &S.cap_binatoms, n + 1, 0);
    grow_n(&S.d_binslots, &S.cap_binslots, n + 1, 0);
    if (failed()) return;
    // (all zero between binnings: the scan clears them)
    if (S.cap_bins != cap0) fill_i32(S.d_bincount, 0, S.cap_bins);
}

// What a binning is for: lists (their status words are cleared on the way, and lists_done reports an
// atom outside the grid), the sort (which reports one), or the caller's own use.
enum BinFor { BIN_CALLER, BIN_SORT, BIN_LISTS };

// Launches the binning of nlocal and *nghost atoms (null: none), max_n at most.
static void launch_bins(int nlocal, const int* nghost, int max_n, const double* x, BinFor use,
    const int* go)
{
    const int mb = S.g.mbins;
    int* outside = use == BIN_CALLER ? nullptr : S.d_status + ST_OUTSIDE;
    int* clear   = use == BIN_LISTS ? S.d_status : nullptr;
    if (max_n <= BIN1_N && mb <= BIN1_BINS) {
        launch_bins_small(nlocal, nghost, max_n, x, outside, clear, go);
        return;
    }
    hipStream_t s       = stream();
    const unsigned grid = blocks_for(max_n, BLOCK);
    k_bin_count<<<grid, BLOCK, 0, s>>>(nlocal, nghost, x, S.g, S.d_bin_of, S.d_binplace,
        S.d_bincount, outside, go);
    exclusive_scan_take(S.d_bincount, S.d_binstart, mb, S.d_binstart + mb);
    k_bin_scatter<<<grid, BLOCK, 0, s>>>(nlocal, nghost, S.d_bin_of, S.d_binplace, S.d_binstart,
        S.d_binslots, go);
    k_bin_rank<<<grid, BLOCK, 0, s>>>(S.xs_ld, S.d_bin_of, S.d_binstart, S.d_binslots, x,
        S.d_binatoms, S.d_xs, S.d_binstart + mb, clear, go);
    MDG_LAUNCH_CHECK("binatoms");
}

static void bin_atoms(Atom* atom, BinFor use)
{
    if (failed() || !S.ready || S.g.mbins == 0) {
        if (!failed()) set_error(MDG_ERR_ARG, "binatomsGFX950 before setupNeighborGFX950");
        return;
    }
    TimedRegion tr(F_BINNING);
    const int nall = atom->Nlocal + atom->Nghost;
    grow_bins((size_t)nall);
    if (failed()) return;
    S.xs_ld  = nall;
    S.binned = true;
    launch_bins(nall, nullptr, nall, atom->d_atom.x, use, nullptr);
}

void binatomsGFX950(Atom* atom) { bin_atoms(atom, BIN_CALLER); }

void sortAtomGFX950(Atom* atom)
{
    // sortAtom (neighbor.c:466-536) with the caller's Nghost = 0 of main.c:92-95 and 372-381
    // done here: the local atoms are binned alone and re-stored in bin order
    if (failed() || !S.ready) return;
    const int n  = atom->Nlocal;
    atom->Nghost = 0;
    S.gmap_nlocal    = -1;
    S.ghosts_current = false;
    if (n <= 0) return;
    bin_atoms(atom, BIN_SORT);
    if (failed()) return;
    read_status();
    if (failed()) return;
    if (S.h_status[ST_OUTSIDE]) {
        fill_i32(S.d_status + ST_OUTSIDE, 0, 1);
        set_error(MDG_ERR_BIN, "sortAtomGFX950: an atom lies outside the bin grid");
        return;
    }
    grow_n(&S.d_sort, &S.cap_sort, 9 * (size_t)n, 0);
    grow_n(&S.d_sort_t, &S.cap_sort_t, (size_t)n, 0);
    if (failed()) return;
    DeviceAtom* d     = &atom->d_atom;
    hipStream_t st    = stream();
    double* xs        = S.d_sort;
    double* vs        = S.d_sort + 3 * (size_t)n;
    double* fs        = S.d_sort + 6 * (size_t)n;
    k_sort_gather<<<blocks_for(n, BLOCK), BLOCK, 0, st>>>(n, S.d_binatoms, d->x, d->vx, d->fx,
        d->type, xs, vs, fs, S.d_sort_t);
    MDG_LAUNCH_CHECK("sort_gather");
    MDG_HIP(hipMemcpyAsync(d->x, xs, 24 * (size_t)n, hipMemcpyDeviceToDevice, st));
    MDG_HIP(hipMemcpyAsync(d->vx, vs, 24 * (size_t)n, hipMemcpyDeviceToDevice, st));
    MDG_HIP(hipMemcpyAsync(d->fx, fs, 24 * (size_t)n, hipMemcpyDeviceToDevice, st));
    MDG_HIP(hipMemcpyAsync(d->type, S.d_sort_t, 4 * (size_t)n, hipMemcpyDeviceToDevice, st));
    S.binned = false;  // the bins name the old indices
}

// The staging tables of a full list just built (after a wait for the stream), where they pay: not
// for lists that are soon replaced, and not while most blocks' neighbours do not fit (atoms in the
// bin sort's order, rows of one bin's width: 321 us per step with the tables tried on every list,
// 311 without); those try again after STAGE_RETRY lists.
static void stage_build(int nlocal, Neighbor* neighbor)
{
    const int over = S.h_status[3] - S.stage_over;
    const int uses = S.last_uses < 0 ? STAGE_USES : std::max(S.list_uses, S.last_uses);
    const int nb   = (nlocal + STAGE_A - 1) / STAGE_A;
    S.stage_over   = S.h_status[3];
    S.last_uses    = S.list_uses;
    S.list_uses    = 0;
    if (S.stage_nlocal == nlocal && over > nb / 2) S.stage_skip = STAGE_RETRY;
    S.stage_nlocal = -1;
    if (neighbor->half_neigh || strict_mode() || nlocal <= STAGE_MIN || nlocal > (1 << 27) || S.d_rhor)
        return;
    if (uses < STAGE_USES) return;
    if (S.stage_skip > 0) {
        S.stage_skip--;
        return;
    }
    const int mn = neighbor->maxneighs;
    if (!stage_room(&S.d_stage, &S.cap_stage, (size_t)nb * STAGE_CAP) ||
        !stage_room(&S.d_stage_n, &S.cap_stage_n, (size_t)nb) ||
        !stage_room(&S.d_hint, &S.cap_hint, (size_t)nlocal * mn)) {
        stage_release();
        return;
    }
    TimedRegion tr(F_NEIGHBOR);
    k_stage_build<<<nb, STAGE_T, 0, stream()>>>(nlocal, neighbor->d_neighbor.neighbors,
        neighbor->d_neighbor.numneigh, mn, S.d_stage, S.d_stage_n, S.d_hint, S.d_status + 3);
    MDG_LAUNCH_CHECK("stage_build");
    S.stage_nlocal = nlocal;
    S.stage_max    = mn;
}

// Whether the block kernel builds the lists: for few atoms, and few bins, since it spends a block on
// each bin, empty ones too.  Boxes read from a file have bins of half the list cutoff, and may be mostly
// empty.  us per list (kernel), a block and a wavefront per bin:
//     atoms    bins
//       256   17576   11.7   14.4
//       256   64000   22.4   14.9
//      2048   17576   14.9   16.2
//      2048   29791   21.4   19.8
//      6912   10648   21.6   31.2
//      6912   17576   28.1   22.5
//     16384   15625   33.9   41.7
//     16384   29791   63.5   33.1
//     16384  328509   125    37
static bool small_lists(int nlocal) { return nlocal <= NB_SMALL && S.g.mbins <= NB_BINS; }

// Launches the list build over the bins; go: see k_ghost_setup.
static void launch_lists(Atom* atom, Neighbor* neighbor, const int* go)
{
    const int nlocal = atom->Nlocal;
    // the largest list cutoff squared, with a margin over the rounding of a distance to a box
    double cnmax = 0.0;
    for (int k = 0; k < S.ntypes * S.ntypes; k++)
        cnmax = std::max(cnmax, S.tab.cutn[k]);
    cnmax *= 1.0 + 1e-12;
    grow_n(&neighbor->d_neighbor.neighbors, &S.cap_nb, (size_t)nlocal * neighbor->maxneighs, 0);
    grow_n(&neighbor->d_neighbor.numneigh, &S.cap_numneigh, (size_t)nlocal, 0);
    if (failed()) return;
    TimedRegion tr(F_NEIGHBOR);
#define MDG_NB(K, G, T, ...)                                                                     \
    K<<<G, T, 0, stream()>>>(nlocal, S.xs_ld, S.d_xs, atom->d_atom.type, S.ntypes, S.tab,        \
        S.uniform ? 1 : 0, cnmax, S.g.mbins, S.d_binstart, S.d_binatoms, S.d_stencil,            \
        S.nstencil, neighbor->half_neigh, neighbor->maxneighs, neighbor->d_neighbor.neighbors,   \
        neighbor->d_neighbor.numneigh, __VA_ARGS__)
    if (small_lists(nlocal)) {
        S.h_flag[HF_OVERFLOW] = S.h_flag[HF_RANGE] = 0;  // (no earlier list build is running)
        MDG_NB(k_build_neighbor, S.g.mbins, NB_T, S.d_status, S.h_flag, go);
    } else {
        MDG_NB(k_build_neighbor_wave, blocks_for(S.g.mbins, BLOCK / 64), BLOCK, S.d_status, go);
    }
#undef MDG_NB
    MDG_LAUNCH_CHECK("build_neighbor");
}

// Waits for the list build; false: the lists were too short and have been given more room.  An atom
// outside the grid is an error: it is in no bin, and its own list has not been written.
static bool lists_done(int nlocal, Neighbor* neighbor, bool waited = false)
{
    bool range, overflow;
    if (small_lists(nlocal)) {
        if (!waited) MDG_HIP(hipStreamSynchronize(stream()));
        if (failed()) return true;
        range    = S.h_flag[HF_RANGE] != 0;
        overflow = S.h_flag[HF_OVERFLOW] != 0;
        if (overflow) read_status();  // the longest list
    } else {
        if (!waited) read_status();
        range    = (S.h_status[0] & ST_BIN_RANGE) != 0 || S.h_status[ST_OUTSIDE] != 0;
        overflow = (S.h_status[0] & ST_NB_OVERFLOW) != 0;
    }
    if (failed()) return true;
    if (range) {
        fill_i32(S.d_status + ST_OUTSIDE, 0, 1);
        set_error(MDG_ERR_BIN, "an atom lies outside the bin grid (coord2bin out of range)");
        return true;
    }
    if (!overflow) {
        stage_build(nlocal, neighbor);
        return true;
    }
    // neighbor.c:336-345: grow to 1.2x the largest count and rebuild
    neighbor->maxneighs = (int)(S.h_status[1] * 1.2) + 1;
    stage_release();  // room for the list first
    fill_i32(S.d_status, 0, 2);
    return false;
}

void buildNeighborGFX950(Atom* atom, Neighbor* neighbor)
{
    if (failed() || !S.ready) return;
    bin_atoms(atom, BIN_LISTS);
    for (int attempt = 0; attempt < 8; attempt++) {
        if (failed()) return;
        launch_lists(atom, neighbor, nullptr);
        if (failed() || lists_done(atom->Nlocal, neighbor)) return;
    }
    set_error(MDG_ERR_CAPACITY, "neighbour list did not converge");
}

void setupPbcGFX950(Atom* atom, Parameter* param)
{
    if (failed() || !S.ready) return;
    TimedRegion tr(F_PBC);
    const int nlocal = atom->Nlocal;
    S.gmap_nlocal    = -1;
    S.ghosts_current = false;
    Prd prd{ { param->xprd, param->yprd, param->zprd } };
    grow_n(&S.d_gcnt, &S.cap_gcnt, (size_t)nlocal + 1, 0);
    grow_n(&S.d_goff, &S.cap_goff, (size_t)nlocal + 1, 0);
    if (failed()) return;
    hipStream_t s    = stream();
    const bool small = nlocal <= SETUP_SMALL;
    int nghost;
    if (small) {
        k_ghost_setup<<<1, SETUP_T, 0, s>>>(nlocal, atom->d_atom.x, 0, prd, param->cutneigh,
            S.d_gcnt, S.d_goff, S.d_status, INT_MAX, S.d_status + 4, S.h_flag);
        MDG_LAUNCH_CHECK("ghost_setup");
        MDG_HIP(hipStreamSynchronize(s));
        if (failed()) return;
        nghost = S.h_flag[HF_TOTAL];
    } else {
        k_ghost_count<<<blocks_for(nlocal, BLOCK), BLOCK, 0, s>>>(nlocal, atom->d_atom.x, prd,
            param->cutneigh, S.d_gcnt, 0);
        exclusive_scan(S.d_gcnt, S.d_goff, nlocal, S.d_status + 2);
        read_status();
        if (failed()) return;
        nghost = S.h_status[2];
    }
    // grow atom arrays (keep the locals), ghost map and shifts
    size_t need = (size_t)nlocal + nghost;
    if (need > S.cap_all) {
        int keep_ghost = atom->Nghost;
        atom->Nghost   = 0;  // only locals carry data worth keeping
        DeviceAtom* d  = &atom->d_atom;
        size_t cx = S.cap_all * 3, cf = cx, ct = S.cap_all;
        grow_n(&d->x, &cx, 3 * need, 3 * (size_t)nlocal);
        grow_n(&d->fx, &cf, 3 * need, 0);
        grow_n(&d->type, &ct, need, (size_t)nlocal);
        // (with the headroom: a rebuild whose ghosts have room waits once)
        S.cap_all    = failed() ? S.cap_all : std::min({ cx / 3, cf / 3, ct });
        atom->Nghost = keep_ghost;
    }
    size_t gc = S.cap_ghost;
    grow_n(&atom->d_atom.border_map, &gc, (size_t)nghost + 1, 0);
    S.cap_ghost = gc;
    grow_n(&S.d_pbc, &S.cap_pbc, 3 * (size_t)nghost + 3, 0);
    if (failed()) return;
    if (small)
        k_ghost_fill_small<<<blocks_for(32LL * nlocal, BLOCK), BLOCK, 0, s>>>(nlocal, atom->d_atom.x,
            prd, param->cutneigh, S.d_goff, atom->d_atom.border_map, S.d_pbc, atom->d_atom.type,
            S.d_status + 4);
    else
        k_ghost_fill<<<blocks_for(nlocal, BLOCK), BLOCK, 0, s>>>(nlocal, atom->d_atom.x, prd,
            param->cutneigh, S.d_goff, atom->d_atom.border_map, S.d_pbc, atom->d_atom.type);
    MDG_LAUNCH_CHECK("ghost_fill");
    atom->Nghost  = nghost;
    S.gmap_nlocal = nlocal;
    S.gmap_nghost = nghost;
    S.ghosts_current = true;
}

// A run's rebuild: updateAtomsPbcGFX950, setupPbcGFX950, updatePbcGFX950 and buildNeighborGFX950.  Where
// the buffers have room for the ghosts, everything is launched before the host waits (once, for the
// lists): the launches behind the ghosts' count take it from device memory, and do nothing if the
// room turns out too small.  With the small systems' kernels of few launches a rebuild takes 16 us
// less for 256 atoms (of about 75) and 25 for 4000; larger ones 8 less at 11,000 atoms, 14 at 62,000 and
// 131,000, 27 (of 1200, a force call included) at 1.05 M.
void mdg_vl_reneighbour(Parameter* param, Atom* atom, Neighbor* neighbor)
{
    if (failed() || !S.ready) return;
    const int nlocal = atom->Nlocal, mb = S.g.mbins;
    const bool small = nlocal <= SETUP_SMALL && mb <= BIN1_BINS;
    const size_t ld  = std::min(S.cap_all, (size_t)(small ? BIN1_N : INT_MAX / 3));
    const size_t room = std::min({ ld - std::min(ld, (size_t)nlocal), S.cap_ghost, S.cap_pbc / 3 });
    if (nlocal <= 0 || mb <= 0 || room == 0) {
        updateAtomsPbcGFX950(atom, param, true);
        setupPbcGFX950(atom, param);
        if (!S.ghosts_current) updatePbcGFX950(atom, param, true);
        buildNeighborGFX950(atom, neighbor);
        return;
    }
    S.gmap_nlocal    = -1;
    S.ghosts_current = false;
    S.binned         = false;
    S.xs_ld          = (int)ld;
    const Prd prd{ { param->xprd, param->yprd, param->zprd } };
    grow_n(&S.d_gcnt, &S.cap_gcnt, (size_t)nlocal + 1, 0);
    grow_n(&S.d_goff, &S.cap_goff, (size_t)nlocal + 1, 0);
    grow_bins(ld);
    if (failed()) return;
    hipStream_t s = stream();
    int* go       = S.d_status + 4;
    DeviceAtom* d = &atom->d_atom;
    if (small) {
        TimedRegion tr(F_PBC);
        k_ghost_setup<<<1, SETUP_T, 0, s>>>(nlocal, d->x, 1, prd, param->cutneigh, S.d_gcnt, S.d_goff,
            S.d_status, (int)room, go, S.h_flag);
        k_ghost_fill_small<<<blocks_for(32LL * nlocal, BLOCK), BLOCK, 0, s>>>(nlocal, d->x, prd,
            param->cutneigh, S.d_goff, d->border_map, S.d_pbc, d->type, go);
        MDG_LAUNCH_CHECK("ghost_setup");
    } else {
        TimedRegion tr(F_PBC);
        const unsigned grid = blocks_for(nlocal, BLOCK);
        k_ghost_count<<<grid, BLOCK, 0, s>>>(nlocal, d->x, prd, param->cutneigh, S.d_gcnt, 1);
        exclusive_scan(S.d_gcnt, S.d_goff, nlocal, S.d_status + 2);
        k_ghost_go<<<1, 1, 0, s>>>((int)room, S.d_status, go);
        k_ghost_fill<<<grid, BLOCK, 0, s>>>(nlocal, d->x, prd, param->cutneigh, S.d_goff,
            d->border_map, S.d_pbc, d->type, go);
        MDG_LAUNCH_CHECK("ghost_setup");
    }
    {
        TimedRegion tr(F_BINNING);
        launch_bins(nlocal, S.d_status + 2, (int)ld, d->x, BIN_LISTS, go);
    }
    if (failed()) return;
    launch_lists(atom, neighbor, go);
    if (failed()) return;
    const bool flags = small_lists(nlocal);  // (lists_done's two ways)
    if (small && flags) MDG_HIP(hipStreamSynchronize(s));
    else read_status();
    if (failed()) return;
    const int nghost = small ? S.h_flag[HF_TOTAL] : S.h_status[2];
    if ((size_t)nghost > room) {  // nothing was built (the atoms are in the box)
        setupPbcGFX950(atom, param);
        buildNeighborGFX950(atom, neighbor);
        return;
    }
    atom->Nghost     = nghost;
    S.gmap_nlocal    = nlocal;
    S.gmap_nghost    = nghost;
    S.ghosts_current = true;
    S.binned         = true;
    for (int attempt = 1; !lists_done(nlocal, neighbor, attempt == 1); attempt++) {
        if (attempt == 8) {
            set_error(MDG_ERR_CAPACITY, "neighbour list did not converge");
            return;
        }
        launch_lists(atom, neighbor, nullptr);
        if (failed()) return;
    }
}

void updatePbcGFX950(Atom* atom, Parameter* param, bool doReneighbor)
{
    (void)doReneighbor;
    if (failed() || !S.ready || atom->Nghost <= 0) return;
    TimedRegion tr(F_PBC);
    Prd prd{ { param->xprd, param->yprd, param->zprd } };
    k_update_pbc<<<blocks_for(3LL * atom->Nghost, BLOCK), BLOCK, 0, stream()>>>(atom->Nlocal,
        atom->Nghost, atom->d_atom.x, atom->d_atom.border_map, S.d_pbc, prd);
    MDG_LAUNCH_CHECK("update_pbc");
}

void updateAtomsPbcGFX950(Atom* atom, Parameter* param, bool doReneighbor)
{
    (void)doReneighbor;
    if (failed() || !S.ready) return;
    S.ghosts_current = false;
    TimedRegion tr(F_PBC);
    k_wrap<<<blocks_for(3LL * atom->Nlocal, BLOCK), BLOCK, 0, stream()>>>(3 * atom->Nlocal,
        atom->d_atom.x, param->xprd, param->yprd, param->zprd);
    MDG_LAUNCH_CHECK("wrap");
}

// Lanes per atom of the fast full-list LJ kernel without energies.  A small system leaves the chip
// idle and waits on the chain of loads along each lane's share of the list, so its lists go to more
// lanes; a large one fills the chip with 4, and more lanes only make the list rows' loads narrower.
// us per step (force, integration and ghosts in one launch, 76 listed neighbours) with
//     atoms     4     8    16    32    64 lanes
//       256  13.2   8.9   6.2   5.3   4.7
//      2048  14.4   8.6   6.3   5.3   5.3
//      6912  13.8   8.7   7.0   7.2   8.5
//     16384  14.3  10.2   8.9  10.9  17.2
//     32000  16.9  11.8  14.4  19.4  29.0
//     55296  19.5  16.3  22.8  30.0  45.7
//    131072  28.5  35.1  49.1  67.2 102.7
// (before: 4 lanes and a ghost update of 3.8 us a step at every size).
static int lanes_per_atom(int nlocal)
{
    return nlocal <= 1500    ? 64
           : nlocal <= 5000  ? 32
           : nlocal <= 24000 ? 16
           : nlocal <= 80000 ? 8
                             : FAST_LPA;
}

// The same choice for the fast half-list kernel without energies.  us per step (force, gather and
// integration with the ghosts; 38 listed neighbours) with
//     atoms     4     8    16    32 lanes
//       256  16.5  13.7  11.8  10.8
//      6912  23.4  15.6  12.5  11.6
//     16384  22.6  15.6  13.8  16.0
//     32000  24.0  17.4  18.8  23.4
//     55296  25.6  22.9  28.7  36.5
//    131072  36.6  41.8  51.5  72.7
static int half_lanes(int nlocal)
{
    return nlocal <= 10000 ? 32 : nlocal <= 24000 ? 16 : nlocal <= 80000 ? 8 : 4;
}

static double force_lj(Parameter* param, Atom* atom, Neighbor* neighbor, Fuse fu)
{
    (void)param;
    if (failed() || !S.ready) return 0.0;
    const double t0 = wtime();
    const int nlocal = atom->Nlocal;
    const int nall   = nlocal + atom->Nghost;
    const bool strict = strict_mode();
    hipStream_t s    = stream();
    if (S.list_uses >= 0) S.list_uses++;
    if (S.ev_on) fill_f64(S.d_ev, 0.0, 2);
    const int half = neighbor->half_neigh;
    if (half && strict) fill_f64(atom->d_atom.fx, 0.0, 3 * (size_t)nall);
    if (half && !strict) {
        const size_t cap0 = S.cap_acc;
        grow_n(&S.d_acc, &S.cap_acc, 3 * (size_t)nlocal, 0);
        if (failed()) return 0.0;
        if (S.cap_acc != cap0) fill_f64(S.d_acc, 0.0, S.cap_acc);
    }
    {
        TimedRegion tr(F_FORCE_LJ);
#define MDG_LJ(L, ST, H, E)                                                                      \
    k_force_lj<L, ST, H, E><<<blocks_for((long long)nlocal * L, BLOCK), BLOCK, 0, s>>>(nlocal, atom->d_atom.x, atom->d_atom.type,    \
        S.ntypes, S.tab, S.uniform ? 1 : 0, neighbor->d_neighbor.neighbors,                      \
        neighbor->d_neighbor.numneigh, atom->d_atom.fx, S.d_ev, fu)
#define MDG_LJH(L, E)                                                                            \
    k_force_lj_half<L, E><<<blocks_for(nlocal, HALF_T / L), HALF_T, 0, s>>>(nlocal,              \
        atom->d_atom.x, atom->d_atom.type, S.ntypes, S.tab, S.uniform ? 1 : 0,                   \
        neighbor->d_neighbor.neighbors, neighbor->d_neighbor.numneigh, S.d_acc, S.d_ev,           \
        atom->Nghost, atom->d_atom.fx + 3 * (size_t)nlocal)
        if (strict) {
            if (half) {
                if (S.ev_on) MDG_LJ(1, true, true, true);
                else MDG_LJ(1, true, true, false);
            } else {
                if (S.ev_on) MDG_LJ(1, true, false, true);
                else MDG_LJ(1, true, false, false);
            }
        } else {
            if (half) {
                const int lanes = half_lanes(nlocal);
                if (S.ev_on) MDG_LJH(4, true);
                else if (lanes == 32) MDG_LJH(32, false);
                else if (lanes == 16) MDG_LJH(16, false);
                else if (lanes == 8) MDG_LJH(8, false);
                else MDG_LJH(4, false);
                k_take_half<<<blocks_for(nlocal, BLOCK), BLOCK, 0, s>>>(nlocal, S.d_acc,
                    atom->d_atom.fx, atom->d_atom.x, fu);
            } else if (S.ev_on) {
                MDG_LJ(FAST_LPA, false, false, true);
            } else {
                const int lanes = lanes_per_atom(nlocal);
                if (lanes == 64) MDG_LJ(64, false, false, false);
                else if (lanes == 32) MDG_LJ(32, false, false, false);
                else if (lanes == 16) MDG_LJ(16, false, false, false);
                else if (lanes == 8) MDG_LJ(8, false, false, false);
                else if (S.stage_nlocal == nlocal && S.stage_max == neighbor->maxneighs) {
                    const int nb        = (nlocal + STAGE_A - 1) / STAGE_A;
                    const unsigned grid = ((unsigned)nb + 7) & ~7u;
#define MDG_LJS(U)                                                                               \
    k_force_lj_staged<U><<<grid, STAGE_T, 0, s>>>(nlocal, nall, nb, atom->d_atom.x,              \
        atom->d_atom.type, S.ntypes, S.tab, neighbor->d_neighbor.neighbors,                      \
        neighbor->d_neighbor.numneigh, S.stage_max, S.d_stage, S.d_stage_n, S.d_hint,            \
        atom->d_atom.fx, fu)
                    if (S.uniform) MDG_LJS(true);
                    else MDG_LJS(false);
#undef MDG_LJS
                } else MDG_LJ(FAST_LPA, false, false, false);
            }
        }
#undef MDG_LJH
#undef MDG_LJ
        MDG_LAUNCH_CHECK("force_lj");
    }
    return wtime() - t0;
}

double computeForceLJGFX950(Parameter* param, Atom* atom, Neighbor* neighbor, Stats* stats)
{
    (void)stats;
    return force_lj(param, atom, neighbor, Fuse{});
}

void setEamTablesGFX950(int nr, int nrho, double rdr, double rdrho, const double* rhor_spline,
    const double* frho_spline, const double* z2r_spline, int nr_tot, int nrho_tot)
{
    if (failed() || !stream()) return;
    dfree(S.d_rhor);
    dfree(S.d_frho);
    dfree(S.d_z2r);
    S.d_rhor = S.d_frho = S.d_z2r = nullptr;
    MDG_HIP(hipMalloc(&S.d_rhor, (size_t)nr_tot * 8));
    MDG_HIP(hipMalloc(&S.d_z2r, (size_t)nr_tot * 8));
    MDG_HIP(hipMalloc(&S.d_frho, (size_t)nrho_tot * 8));
    if (failed()) return;
    MDG_HIP(hipMemcpy(S.d_rhor, rhor_spline, (size_t)nr_tot * 8, hipMemcpyHostToDevice));
    MDG_HIP(hipMemcpy(S.d_z2r, z2r_spline, (size_t)nr_tot * 8, hipMemcpyHostToDevice));
    MDG_HIP(hipMemcpy(S.d_frho, frho_spline, (size_t)nrho_tot * 8, hipMemcpyHostToDevice));
    S.nr    = nr;
    S.nrho  = nrho;
    S.rdr   = rdr;
    S.rdrho = rdrho;
}

// Lanes per atom of the fast EAM passes.  The LDS-table passes read the whole spline tables into
// every block first (64 and 160 KB, ~12 us a pass however few atoms there are), so up to 20000
// atoms (40000 with tables that do not fit) the passes read the rows from L2 instead, with an atom's
// list on as many lanes as the system leaves idle; the density pass then also writes the ghosts' F'.
// us per step (both passes, integration, ghosts; 75 listed neighbours) with
//     atoms  LDS tables, 4     8    16    32    64 lanes
//       500      30.4        19.8  12.6  10.2   8.9
//      4000      32.1        20.2  13.3  12.3  13.2
//      8788      34.6        24.5  18.4  18.3  23.3
//     16384      33.9        24.3  22.7  29.1  41.8
//     32000      40.6        35.6  44.1  54.1  74.6
//     55296      49.3        60.5  70.0  87.0 120.3
// (the tables' column before two lanes loaded a neighbour together; since then 28.2 against 29.5 with
// 8 lanes at 23328, 29.7 against 35.4 at 32000 and 34.9 against 45.5 at 37044).
static int eam_lanes(int nlocal, bool tab)
{
    return nlocal <= 1500             ? 64
           : nlocal <= 9000           ? 32
           : nlocal <= 20000          ? 16
           : !tab && nlocal <= 40000  ? 8
                                      : FAST_LPA;
}

// The same for the passes with energies, whose blocks each end with atomics on the same words: fewer
// lanes are fewer blocks.  us per call (both passes, 75 listed neighbours) with
//     atoms     4     8    16    32 lanes
//       256  28.4  19.7  14.9  13.2
//       864  30.5  20.1  15.5  15.3
//      2048  29.9  20.1  18.0  20.5
//      4000  30.8  22.3  22.4  30.3
//     10976  33.0  30.5  40.4  69.8
//     19652  39.8  44.3  65.0   108
//     32000  50.7  63.9   102   169
static int eam_energy_lanes(int nlocal)
{
    return nlocal <= 1000 ? 32 : nlocal <= 3000 ? 16 : nlocal <= 10000 ? 8 : FAST_LPA;
}

static double force_eam(Parameter* param, Atom* atom, Neighbor* neighbor, Fuse fu)
{
    if (failed() || !S.ready) return 0.0;
    if (!S.d_rhor) {
        set_error(MDG_ERR_ARG, "computeForceEamGFX950 before setEamTablesGFX950");
        return 0.0;
    }
    const double t0 = wtime();
    const int nlocal = atom->Nlocal;
    const int nall   = nlocal + atom->Nghost;
    grow_n(&S.d_fp, &S.cap_fp, 4 * (size_t)nall + 1, 0);  // F', or rows of position and F'
    if (failed()) return 0.0;
    const bool strict = strict_mode();
    hipStream_t s     = stream();
    double cutf       = param->cutforce * param->cutforce;
    double* eatom = nullptr;
    if (S.eatom_on) {
        grow_n(&S.d_eatom, &S.cap_eatom, (size_t)nlocal + 1, 0);
        if (failed()) return 0.0;
        eatom = S.d_eatom;
    }
    const bool ev = S.ev_on || S.eatom_on;
    if (ev) fill_f64(S.d_ev, 0.0, 2);
    TimedRegion tr(F_FORCE_EAM);
#define MDG_EAM_F(L, ST, E, G)                                                                   \
    k_eam_force<L, ST, E, G><<<grid, BLOCK, 0, s>>>(nlocal, atom->d_atom.x,                      \
        neighbor->d_neighbor.neighbors, neighbor->d_neighbor.numneigh, cutf, S.d_rhor, S.d_z2r,  \
        S.nr, S.rdr, S.d_fp, atom->d_atom.fx, S.d_ev, eatom, fu)
#define MDG_EAM(L, ST, E)                                                                        \
    do {                                                                                         \
        const unsigned grid = blocks_for((long long)nlocal * L, BLOCK);                          \
        k_eam_density<L, ST, E><<<grid, BLOCK, 0, s>>>(nlocal, atom->d_atom.x,                   \
            neighbor->d_neighbor.neighbors, neighbor->d_neighbor.numneigh, cutf, S.d_rhor,       \
            S.d_frho, S.nr, S.nrho, S.rdr, S.rdrho, S.d_fp, S.d_ev, eatom,                       \
            gmap ? S.d_gcnt : nullptr, S.d_goff);                                                \
        if (!gmap) launch_ghost_copy(S.d_fp, atom);                                              \
        if (fu.gcnt) MDG_EAM_F(L, ST, E, true);                                                  \
        else MDG_EAM_F(L, ST, E, false);                                                         \
    } while (0)
    // without the energy and for tables of up to TAB_NR rows: the LDS-table passes
#define MDG_EAM_FT(L, ST, G)                                                                     \
    k_eam_force_tab<L, ST, G><<<gf, TAB_BLOCK, 0, s>>>(nlocal, pf, xf,                           \
        neighbor->d_neighbor.neighbors, neighbor->d_neighbor.numneigh, cutf, S.d_rhor, S.d_z2r,  \
        S.nr, S.rdr, atom->d_atom.fx, fu)
#define MDG_EAM_TAB(L, ST)                                                                       \
    do {                                                                                         \
        const unsigned gd = 2u * (unsigned)S.ncu, gf = (unsigned)S.ncu;                          \
        const int pd = (int)((nlocal + gd - 1) / gd), pf = (int)((nlocal + gf - 1) / gf);        \
        k_eam_density_tab<L, ST><<<gd, TAB_BLOCK, 0, s>>>(nlocal, pd, atom->d_atom.x,            \
            neighbor->d_neighbor.neighbors, neighbor->d_neighbor.numneigh, cutf, S.d_rhor,       \
            S.d_frho, S.nr, S.nrho, S.rdr, S.rdrho, xf);                                         \
        if (atom->Nghost > 0) {                                                                  \
            k_ghost_rows<<<blocks_for(atom->Nghost, BLOCK), BLOCK, 0, s>>>(nlocal, atom->Nghost, \
                atom->d_atom.x, xf, atom->d_atom.border_map);                                    \
            MDG_LAUNCH_CHECK("ghost_rows");                                                      \
        }                                                                                        \
        if (fu.gcnt) MDG_EAM_FT(L, ST, true);                                                    \
        else MDG_EAM_FT(L, ST, false);                                                           \
    } while (0)
    double2* xf     = (double2*)S.d_fp;
    const bool tab  = !ev && S.nr <= TAB_NR && S.ncu > 0 && nlocal > 0;
    const bool gmap = S.gmap_nlocal == nlocal && S.gmap_nghost == atom->Nghost;
    const int lanes = eam_lanes(nlocal, tab);
    if (strict) {
        if (ev) MDG_EAM(1, true, true);
        else if (tab) MDG_EAM_TAB(1, true);
        else MDG_EAM(1, true, false);
    } else if (ev) {
        const int el = eam_energy_lanes(nlocal);
        if (el == 32) MDG_EAM(32, false, true);
        else if (el == 16) MDG_EAM(16, false, true);
        else if (el == 8) MDG_EAM(8, false, true);
        else MDG_EAM(FAST_LPA, false, true);
    } else if (lanes == 64) {
        MDG_EAM(64, false, false);
    } else if (lanes == 32) {
        MDG_EAM(32, false, false);
    } else if (lanes == 16) {
        MDG_EAM(16, false, false);
    } else if (lanes == 8) {
        MDG_EAM(8, false, false);
    } else if (tab) {
        MDG_EAM_TAB(FAST_LPA, false);
    } else {
        MDG_EAM(FAST_LPA, false, false);
    }
#undef MDG_EAM_TAB
#undef MDG_EAM_FT
#undef MDG_EAM
#undef MDG_EAM_F
    MDG_LAUNCH_CHECK("force_eam");
    return wtime() - t0;
}

double computeForceEamGFX950(Parameter* param, Atom* atom, Neighbor* neighbor, Stats* stats)
{
    (void)stats;
    return force_eam(param, atom, neighbor, Fuse{});
}

double computeForceFinalInitialGFX950(Parameter* param, Atom* atom, Neighbor* neighbor,
    Stats* stats)
{
    if (failed() || !S.ready) return 0.0;
    const bool eam = param->force_field == FF_EAM;
    if (strict_mode()) {
        // the strict kernels run the three calls in order
        const double t = eam ? computeForceEamGFX950(param, atom, neighbor, stats)
                             : computeForceLJGFX950(param, atom, neighbor, stats);
        finalIntegrateGFX950(false, param, atom);
        initialIntegrateGFX950(false, param, atom);
        return t;
    }
    // a half list's positions are moved after its forces are complete, in place
    const bool in_place = !eam && neighbor->half_neigh;
    if (!in_place) grow_n(&S.d_xn, &S.cap_xn, 3 * S.cap_all, 0);
    if (failed()) return 0.0;
    Fuse fu{ { atom->d_atom.vx, in_place ? atom->d_atom.x : S.d_xn, param->dt, param->dtforce } };
    // (not for large EAM systems: the images' writes in the border atoms' tails hold up their
    // persistent blocks by 15 us a step at 1M atoms, more than the 5 us of the ghost update)
    const bool ghosts = S.gmap_nlocal == atom->Nlocal && S.gmap_nghost == atom->Nghost &&
                        !(eam && atom->Nlocal > FUSE_GHOSTS_EAM);
    if (ghosts) {
        fu.gcnt   = S.d_gcnt;
        fu.goff   = S.d_goff;
        fu.pbc    = S.d_pbc;
        fu.prd[0] = param->xprd;
        fu.prd[1] = param->yprd;
        fu.prd[2] = param->zprd;
    }
    const double t = eam ? force_eam(param, atom, neighbor, fu) : force_lj(param, atom, neighbor, fu);
    // the new local positions become the current ones; ghost positions written too if their map
    // is known, else they follow at updatePbc
    if (!in_place) {
        std::swap(atom->d_atom.x, S.d_xn);
        S.cap_xn = 3 * S.cap_all;
    }
    S.ghosts_current = ghosts && !failed();
    return t;
}

// For the run loop: the last call was setupPbcGFX950, or a fused force call that also moved the
// ghosts.
int mdg_vl_ghosts_current(void) { return S.ghosts_current; }

void requestEamAtomEnergyGFX950(int on)
{
    S.eatom_on = on != 0;
}

int downloadEamAtomEnergyGFX950(Atom* atom, double* out)
{
    if (failed() || !S.ready) return -1;
    if (!S.eatom_on || !S.d_eatom) {
        set_error(MDG_ERR_ARG, "per-atom EAM energies were not requested before the force call");
        return -1;
    }
    MDG_HIP(hipMemcpyAsync(out, S.d_eatom, (size_t)atom->Nlocal * 8, hipMemcpyDeviceToHost,
        stream()));
    MDG_HIP(hipStreamSynchronize(stream()));
    return failed() ? -1 : 0;
}

void initialIntegrateGFX950(bool reneigh, Parameter* param, Atom* atom)
{
    (void)reneigh;
    if (failed() || !S.ready) return;
    S.ghosts_current = false;
    TimedRegion tr(F_INTEGRATE);
    int n3 = 3 * atom->Nlocal;
    k_initial_integrate<<<blocks_for(n3, BLOCK), BLOCK, 0, stream()>>>(n3, atom->d_atom.x,
        atom->d_atom.vx, atom->d_atom.fx, param->dt, param->dtforce);
    MDG_LAUNCH_CHECK("initial_integrate");
}

void finalIntegrateGFX950(bool reneigh, Parameter* param, Atom* atom)
{
    (void)reneigh;
    if (failed() || !S.ready) return;
    TimedRegion tr(F_INTEGRATE);
    int n3 = 3 * atom->Nlocal;
    k_final_integrate<<<blocks_for(n3, BLOCK), BLOCK, 0, stream()>>>(n3, atom->d_atom.vx,
        atom->d_atom.fx, param->dtforce);
    MDG_LAUNCH_CHECK("final_integrate");
}

double kineticSumGFX950(Parameter* param, Atom* atom)
{
    if (failed() || !S.ready) return 0.0;
    TimedRegion tr(F_THERMO);
    const int nb = 512;
    grow_n(&S.d_red, &S.cap_red, (size_t)nb, 0);
    if (failed()) return 0.0;
    k_ksum_partial<<<nb, BLOCK, 0, stream()>>>(atom->Nlocal, atom->d_atom.vx, param->mass, S.d_red);
    k_sum_partials<<<1, BLOCK, 0, stream()>>>(nb, S.d_red);
    MDG_LAUNCH_CHECK("ksum");
    MDG_HIP(hipMemcpyAsync(S.h_red, S.d_red, sizeof(double), hipMemcpyDeviceToHost, stream()));
    MDG_HIP(hipStreamSynchronize(stream()));
    return failed() ? 0.0 : S.h_red[0];
}

void requestEnergyVirialGFX950(int on)
{
    if (!ensure_status()) return;
    S.ev_on = on != 0;
}

void energyVirialGFX950(double* epot, double* virial)
{
    double h[2] = { 0, 0 };
    if (!failed() && S.d_ev) {
        MDG_HIP(hipMemcpyAsync(h, S.d_ev, 2 * sizeof(double), hipMemcpyDeviceToHost, stream()));
        MDG_HIP(hipStreamSynchronize(stream()));
    }
    if (epot) *epot = h[0];
    if (virial) *virial = h[1];
}

int downloadVLStateGFX950(Atom* atom, Neighbor* neighbor, double* x, double* f, double* v,
    int* border_map, int* pbc, int* numneigh, int* neighbors_csr, long long csr_cap)
{
    if (failed() || !S.ready) return -1;
    hipStream_t s = stream();
    size_t nl = atom->Nlocal, nall = nl + atom->Nghost;
    if (x) MDG_HIP(hipMemcpyAsync(x, atom->d_atom.x, 3 * nall * 8, hipMemcpyDeviceToHost, s));
    if (f) MDG_HIP(hipMemcpyAsync(f, atom->d_atom.fx, 3 * nl * 8, hipMemcpyDeviceToHost, s));
    if (v) MDG_HIP(hipMemcpyAsync(v, atom->d_atom.vx, 3 * nl * 8, hipMemcpyDeviceToHost, s));
    if (border_map && atom->Nghost)
        MDG_HIP(hipMemcpyAsync(border_map, atom->d_atom.border_map, atom->Nghost * 4,
            hipMemcpyDeviceToHost, s));
    if (pbc && atom->Nghost)
        MDG_HIP(hipMemcpyAsync(pbc, S.d_pbc, 3 * (size_t)atom->Nghost * 4, hipMemcpyDeviceToHost, s));
    int rc = 0;
    if (numneigh && neighbors_csr) {
        int* nn = (int*)malloc(nl * sizeof(int));
        size_t tot = nl * (size_t)neighbor->maxneighs;
        int* soa   = (int*)malloc(tot * sizeof(int) + 4);
        MDG_HIP(hipMemcpyAsync(nn, neighbor->d_neighbor.numneigh, nl * 4, hipMemcpyDeviceToHost, s));
        MDG_HIP(hipMemcpyAsync(soa, neighbor->d_neighbor.neighbors, tot * 4, hipMemcpyDeviceToHost, s));
        MDG_HIP(hipStreamSynchronize(s));
        long long k = 0;
        for (size_t i = 0; i < nl && rc == 0; i++) {
            numneigh[i] = nn[i];
            for (int m = 0; m < nn[i]; m++) {
                if (k >= csr_cap) {
                    rc = -2;
                    break;
                }
                neighbors_csr[k++] = soa[(size_t)m * nl + i];
            }
        }
        free(nn);
        free(soa);
        if (rc == 0) rc = (int)(k > 0x7fffffff ? -3 : k);
    }
    MDG_HIP(hipStreamSynchronize(s));
    return failed() ? -1 : rc;
}

int downloadBinsGFX950(int* binstart, int mbins_cap, int* binatoms, int nall_cap)
{
    if (failed() || !S.binned) return -1;
    int mb = S.g.mbins;
    if (mbins_cap < mb + 1) return -2;
    MDG_HIP(hipMemcpy(binstart, S.d_binstart, (mb + 1) * sizeof(int), hipMemcpyDeviceToHost));
    int tot = binstart[mb];
    if (tot > nall_cap) return -3;
    MDG_HIP(hipMemcpy(binatoms, S.d_binatoms, tot * sizeof(int), hipMemcpyDeviceToHost));
    return failed() ? -1 : mb;
}

}  // extern "C"
