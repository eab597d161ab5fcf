// mdx_sor_lds.hip -- LDS-resident red-black SOR for gfx950 with multi-sweep temporal blocking.
//
// The streaming sweeps (mdx_sor.hip) read and write the whole grid once per colour; on the wavy
// channel (2.4 M cells) that is a few microseconds of HBM/MALL traffic, but every launch also pays
// dispatch latency.  Here every workgroup owns one subdomain for a whole batch of iterations: its
// Phi tile lives in LDS with a halo two cells deep, and its right-hand side and face coefficients
// (the IBM geometry is z-invariant, so one x-y plane of mu suffices) in registers of the threads
// that own its z-columns (the pair form keeps the coefficients in an LDS table).
//
// Temporal blocking: an iteration relaxes colour 0 on the subdomain AND on the one-cell ring of
// face cells around it (recomputing what the neighbours compute for those cells, from the same old
// values, so the results are identical), then colour 1 on the subdomain, whose neighbours are then
// all up to date.  One halo exchange per iteration therefore suffices instead of one per colour.
// The ring cells read the second halo layer and the halo edge lines, so a workgroup exchanges with
// up to 18 neighbours: 6 faces two layers deep and 12 edges one cell thick.  Only the colour-1
// cells of those regions travel: the ring's colour-0 cells are the only colour-0 halo cells any
// relaxation reads, and this workgroup forms them itself (the recomputation above), so half of the
// halo is exchanged.
//
// Exchange: every published word carries the number of the iteration it belongs to (a 32-bit
// payload and a 32-bit tag in one 64-bit agent-scope atomic store), and a consumer polls the face
// data itself until every word it needs shows the expected tag: one store and one load per
// hand-off, with no acknowledgement wait and no separate counter.  Faces are double-buffered by
// iteration parity; a producer cannot overwrite a buffer before its consumers have read it,
// because it first needs their next layers.  All workgroups must be co-resident: the plan never
// holds more workgroups than the CUs take at once (runtime occupancy), and every wait is bounded
// (a spin limit sets an error flag and the kernel runs to completion).
//
// The arithmetic per cell is sor_residual_core(), the same expressions the streaming sweeps use,
// and the relaxation factor -omega/denom is formed from the same values, so the iterates are
// bit-identical to the streaming sweeps (and to the oracle).
#include <algorithm>
#include <map>
#include <type_traits>

#include "mdx_sor_core.h"

namespace mdx {

static constexpr int RB_THREADS = 512;
static constexpr int RB_HE = 6;      // exchanged values per thread (a subdomain's colour-1 halo <= RB_HE * RB_THREADS)
static constexpr int RB_MAXR = 3;    // colour-0 ring cells per thread
static constexpr int RB_G = 3;       // cells relaxed per group (loads issued together)
static constexpr int RB_H = 2;       // halo depth
// column forms: cells per thread and colour, for a whole column (bz <= 2 * RB_ZC1 - 2) and for a half
// column (bz <= 4 * RB_ZC2 - 4)
static constexpr int RB_ZC1 = 13, RB_ZC2 = 7;
// plan codes (in place of the pairs per thread) of the column forms
static constexpr int RB_COLS = -1, RB_COLS2 = -2;
static constexpr int RB_XSTRIDE = RB_HE * RB_THREADS;   // exchange entries per workgroup and buffer
// Fixed LDS geometry: a tile row has room for RB_BX values and a plane for RB_BY rows, whatever the
// subdomain (bx + 4 <= RB_BX, by + 4 <= RB_BY), so every stencil and coefficient-plane offset is an
// immediate of the LDS instruction; the coefficient table uses the same plane shape.  The box is the
// 24 x 16 tile of the 192 x 128 x 96 channel on 256 workgroups with its halo.
//
// Row and plane strides are chosen for the 32 banks.  In the column forms a wave's lanes are
// neighbouring columns, 20 interior ones to a row of that tile, at planes that alternate with the
// colour.  FP32 (32 lanes at a time): rows of 36 and planes of 720 values put the next row's lanes
// exactly behind the first's, where rows of 28 and planes of 560 took 3.5 cycles instead of 2.6 a
// load.  FP64 (16 lanes at a time; 160 KB hold rows of 28): planes of 568 instead of 560 take 4.2
// cycles instead of 5.4.  Per iteration at 192 x 128 x 96, FP32 / FP64: 4.5 / 6.5 us before, 4.3 / 6.4 now.
static constexpr int RB_BX = 28, RB_BY = 20;
struct RbStride {
    int row, plane;
};
__host__ __device__ constexpr RbStride rb_stride(bool fp32, bool half_columns) {
    return half_columns ? (fp32 ? RbStride{36, 720} : RbStride{28, 568}) : RbStride{28, 560};
}

// LDS index of the dummy cell, past the tile
__host__ __device__ inline int rb_dummy(int plane, int bz) { return plane * (bz + 2 * RB_H) + plane + 1; }

template <typename T>
struct RbArgs {
    Dims d;
    int px, py, pz;          // workgroups along x, y, z
    int bx, by, bz;          // the largest subdomain (its extents lay out the exchange buffers)
    int per_y;
    SorConst<T> s;
    T omega;
    const T *mu_u, *mu_v, *mu_w;   // z-invariant plane tables (IBM) or nullptr
    T *x;                    // solution (interior layout), updated in place
    const T *rhs;
    int zero_init;           // x starts at zero (the defect equation)
    int iters;               // full red+black iterations
    int md;                  // leading pair entries of every thread that lie in the deep box
    unsigned long long *faces;   // [wg][buffer][word of the value][exchange entry], tagged words
    int total;               // exchange entries in use per workgroup (faces two deep, then edges)
    const int *xl;           // exchange lists of the plan: [wg][entry] publish words, then pull words
    unsigned tag0;           // iteration s of this launch publishes tag tag0 + s + 1 (never 0)
    int *err;
    int spin_limit;          // polls of a neighbour wait before it gives up and sets *err
    // Check epilogue: after the last iteration and one more halo exchange the residual check that
    // follows the batch is formed here, from the tile in LDS.  FP32 batches (the mixed solve): the
    // corrected iterate phi_out = phi_in + e, the new defect r_out = (float)(rhs64 - L_mu phi_out)
    // and max |defect|, with the arithmetic of the separate defect kernel (cell_residual over
    // phi_in + (double)e), instead of writing e back for that kernel.  FP64 batches: the iterate
    // itself goes to phi_out and max |rhs64 - L_mu phi_out| is sor_residual64_kernel's.
    int defect;
    GridK g;
    MuK<double> mu64;
    SorConst<double> s64;
    const double *phi_in, *rhs64;
    double *phi_out, *max_part;
    float *r_out;
    // workgroup 0 folds the workgroups' maxima into red_max[0] and the host slot, with the error
    // word red_max[1], then writes seq to host_slot[2]
    unsigned long long *red_max;
    double *host_slot;
    unsigned long long seq;
    // skip: return at once when the previous check, red_max[0], is not >= skip_tol (converged, or
    // not a number): a batch queued ahead of the host's read of that check then costs one launch
    int skip;
    double skip_tol;
    // half-column form: overlap the interior columns' halo-free cells with the exchange
    int ovl;
};

// a value as tagged 64-bit words: the tag in the high half, 32 payload bits in the low half
template <typename T> struct Tagged;
template <> struct Tagged<float> {
    static constexpr int NW = 1;
    __device__ static void pack(float v, unsigned tag, unsigned long long *o) {
        o[0] = ((unsigned long long)tag << 32) | __float_as_uint(v);
    }
    __device__ static float unpack(const unsigned long long *o) { return __uint_as_float((unsigned)o[0]); }
};
template <> struct Tagged<double> {
    static constexpr int NW = 2;
    __device__ static void pack(double v, unsigned tag, unsigned long long *o) {
        const unsigned long long b = (unsigned long long)__double_as_longlong(v);
        o[0] = ((unsigned long long)tag << 32) | (b & 0xffffffffull);
        o[1] = ((unsigned long long)tag << 32) | (b >> 32);
    }
    __device__ static double unpack(const unsigned long long *o) {
        return __longlong_as_double((long long)((o[1] << 32) | (o[0] & 0xffffffffull)));
    }
};

// Exchange direction q: 0-5 faces (x-, x+, y-, y+, z-, z+), two layers deep; 6-17 edges, one cell.
__host__ __device__ inline void rb_dir(int q, int &dx, int &dy, int &dz) {
    dx = dy = dz = 0;
    if (q < 6) {
        const int sgn = (q & 1) ? 1 : -1;
        if (q < 2) dx = sgn; else if (q < 4) dy = sgn; else dz = sgn;
        return;
    }
    const int e = q - 6, s1 = (e & 1) ? 1 : -1, s2 = (e & 2) ? 1 : -1;
    if (e < 4) { dx = s1; dy = s2; }          // x-y edges (lines along z)
    else if (e < 8) { dx = s1; dz = s2; }     // x-z edges (lines along y)
    else { dy = s1; dz = s2; }                // y-z edges (lines along x)
}

// extents of direction q's region: the subdomain size along axes where the direction is 0, else
// the depth (2 for faces, 1 for edges)
__host__ __device__ inline void rb_extent(int q, int bx, int by, int bz, int &ex, int &ey, int &ez) {
    int dx, dy, dz;
    rb_dir(q, dx, dy, dz);
    const int h = q < 6 ? RB_H : 1;
    ex = dx ? h : bx;
    ey = dy ? h : by;
    ez = dz ? h : bz;
}

// exchange entries per workgroup: the colour-1 half of the 18 regions of the largest subdomain
// (a line of an odd number of cells counts its longer half)
__host__ __device__ inline int rb_xchg_total(int bx, int by, int bz) {
    int t = 0;
    for (int q = 0; q < 18; ++q) {
        int ex, ey, ez;
        rb_extent(q, bx, by, bz, ex, ey, ez);
        t += (ex * ey * ez + 1) / 2;
    }
    return t;
}

// Part w of n cells cut into p parts: origin o and size b.  Every part starts on an even cell, so a
// cell's colour depends on its local coordinates alike in every workgroup along the axis; the
// first parts take one pair more where p does not divide the pairs, the last one an odd cell.
__host__ __device__ inline void rb_part(int n, int p, int w, int &o, int &b) {
    const int np = n / 2, base = np / p, rem = np % p;
    o = 2 * (w * base + (w < rem ? w : rem));
    b = 2 * (base + (w < rem ? 1 : 0)) + (w == p - 1 ? n & 1 : 0);
}
__host__ inline int rb_part_max(int n, int p) {
    int o, b, c;
    rb_part(n, p, 0, o, b);
    rb_part(n, p, p - 1, o, c);
    return b > c ? b : c;
}
__host__ inline int rb_part_min(int n, int p) {
    const int b = 2 * (n / 2 / p);
    return p == 1 ? n : b;
}

// colour-0 ring cells: on each face ring, half of by*bz (x faces), bx*bz (y) or bx*by (z) cells
__host__ __device__ inline int rb_ring_total(int bx, int by, int bz) { return by * bz + bx * bz + bx * by; }

// COLS: column form.  A thread owns one column (i, j) of the subdomain or of the face ring and
// marches it in z, relaxing every other cell; the face coefficients of the column stay in
// registers (z-invariant tables) and the z neighbour between two cells of one colour is loaded
// once, so a cell costs six LDS loads and one store instead of thirteen loads and a store.
// Otherwise (pair form) a thread owns MAXP x-pairs and up to RB_MAXR ring cells anywhere in the
// tile and reads their coefficients from an LDS table; the pair form also relaxes the deep box's
// colour 0 while the halo is in flight.
// FORM: 0 pair form, 1 column form, 2 column form with two threads per column (the lower and the
// upper half of its z range) in workgroups of twice the threads.
// STRETCH (the half-column form only): the y coefficients of a stretched grid's row in registers.
template <typename T, bool IBM, int MAXP, int FORM, bool STRETCH>
__global__ __launch_bounds__(FORM == 2 ? 2 * RB_THREADS : RB_THREADS) void rb_lds_kernel(RbArgs<T> a) {
    // threads per workgroup, exchange entries per thread (the face buffer layout is the same for
    // every form) and, in the column forms, cells per thread and colour
    constexpr bool COLS = FORM > 0;
    constexpr int NT = FORM == 2 ? 2 * RB_THREADS : RB_THREADS, HE = RB_XSTRIDE / NT;
    constexpr int ZC = FORM == 2 ? RB_ZC2 : RB_ZC1;
    if (a.skip) {
        // every workgroup reads the same word: the previous kernel's result, which this launch's
        // workgroup 0 overwrites only after all workgroups have published their epilogue maxima
        const unsigned long long rb = __hip_atomic_load(&a.red_max[0], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if (!(__longlong_as_double((long long)rb) >= a.skip_tol)) return;
    }
    extern __shared__ unsigned char smem_raw[];
    using TW = Tagged<T>;
    constexpr int NW = TW::NW;
    const Dims d = a.d;
    constexpr int TXP = rb_stride(sizeof(T) == 4, FORM == 2).row, PLANE = rb_stride(sizeof(T) == 4, FORM == 2).plane;
    constexpr int cw = TXP, cpl = PLANE;   // coefficient table: local i, j in [0, b+1]
    T *X = reinterpret_cast<T *>(smem_raw);
    // Unused slots of the pair form's cell lists point at a dummy cell past the tile, whose stencil
    // reads and writes stay inside a padding of 2 planes + 3 values, so its relax loops need no
    // branches; the column forms mask absent cells off (colour()) and only mark them by it.  The
    // same cell in every workgroup, past the largest tile.
    const int dummy = rb_dummy(PLANE, a.bz);
    T *C = X + dummy + PLANE + 2;   // IBM pair form: 6 planes of cpl values
                                       // (planes: threads read at pair stride)
    const int nwg = a.px * a.py * a.pz;
    // XCD-aware placement: workgroups are dispatched round-robin over the 8 XCDs, so consecutive
    // subdomain ids (neighbours along x first) are given to workgroups on the same XCD.
    const int per_xcd = nwg / RB_XCDS;
    const int b = blockIdx.x;
    const int w = (nwg % RB_XCDS == 0) ? (b % RB_XCDS) * per_xcd + b / RB_XCDS : b;
    const int wx = w % a.px, wy = (w / a.px) % a.py, wz = w / (a.px * a.py);
    int ox, oy, oz, bx, by, bz;   // this workgroup's subdomain
    rb_part(d.nx, a.px, wx, ox, bx);
    rb_part(d.ny, a.py, wy, oy, by);
    rb_part(d.nz, a.pz, wz, oz, bz);
    const int tx = bx + 2 * RB_H, ty = by + 2 * RB_H, tz = bz + 2 * RB_H;   // tile extent in use
    const int t = threadIdx.x;
    const bool per_y = a.per_y != 0;
    // LDS index of local cell (i, j, k); the subdomain is 1..b, the halo -1..0 and b+1..b+2
    auto L = [&](int i, int j, int k) { return (i + 1) + TXP * (j + 1) + PLANE * (k + 1); };
    // periodic image in 1..n of a coordinate within one period of the domain (-n < g <= 2n)
    auto wrap = [](int g, int n) { return g < 1 ? g + n : (g > n ? g - n : g); };
    // the workgroup in direction (dx, dy, dz), or -1 beyond a wall
    auto neighbour = [&](int dx, int dy, int dz) {
        int ny_ = wy + dy;
        if (ny_ < 0 || ny_ >= a.py) {
            if (!per_y) return -1;
            ny_ = (ny_ + a.py) % a.py;
        }
        return (wx + dx + a.px) % a.px + a.px * (ny_ + a.py * ((wz + dz + a.pz) % a.pz));
    };
    auto wall_bits = [&](int gj) { return (!per_y && gj == d.ny ? 1 : 0) | (!per_y && gj == 1 ? 2 : 0); };

    // ---- load the tile (subdomain and halo) from the global solution, in LDS order over the fixed
    // row and plane (constant divisors; values past the tile extent in a row or plane are zero)
    for (int q = t; q < PLANE * tz; q += NT) {
        const int xi = q % PLANE % TXP, yi = q % PLANE / TXP;
        const int li = xi - 1, lj = yi - 1, lk = q / PLANE - 1;
        T v = T(0);
        if (!a.zero_init && xi < tx && yi < ty) {
            const int gi = wrap(ox + li, d.nx), gk = wrap(oz + lk, d.nz);
            int gj = oy + lj;
            if (per_y) gj = wrap(gj, d.ny);
            if (gj >= 1 && gj <= d.ny) v = a.x[d.in(gi, gj, gk)];
        }
        X[q] = v;
    }
    // ---- face coefficient table (one x-y plane, ring included): mui, muip, mvj, mvjp, mw, -omega/denom
    T qconst = T(0);
    if (IBM && !COLS) {
        const int sx = d.sx;
        for (int q0 = t; q0 < (bx + 2) * (by + 2); q0 += NT) {
            const int li = q0 % (bx + 2), lj = q0 / (bx + 2), q = li + cw * lj;
            const int gi = wrap(ox + li, d.nx);
            int gj = oy + lj;
            if (per_y) gj = wrap(gj, d.ny);
            T mui = 1, muip = 1, mvj = 1, mvjp = 1, mw = 1, qq = 0;
            if (gj >= 1 && gj <= d.ny) {   // rows beyond a wall are never relaxed
                const int gip = gi == d.nx ? 1 : gi + 1;
                const int gjp = (per_y && gj == d.ny) ? 1 : gj + 1;
                mui = a.mu_u[(size_t)gi + (size_t)sx * gj];
                muip = a.mu_u[(size_t)gip + (size_t)sx * gj];
                mvj = a.mu_v[(size_t)gi + (size_t)sx * gj];
                mvjp = a.mu_v[(size_t)gi + (size_t)sx * gjp];
                mw = a.mu_w[(size_t)gi + (size_t)sx * gj];
                const T denom = (mui + muip) * a.s.idx2 + (mw + mw) * a.s.idz2 + (mvj + mvjp) * a.s.idy2;
                qq = -a.omega / denom;
            }
            C[q] = mui; C[q + cpl] = muip; C[q + 2 * cpl] = mvj; C[q + 3 * cpl] = mvjp; C[q + 4 * cpl] = mw;
            C[q + 5 * cpl] = qq;
        }
    } else {
        const T one = T(1);
        const T denom = (one + one) * a.s.idx2 + (one + one) * a.s.idz2 + (one + one) * a.s.idy2;
        qconst = -a.omega / denom;
    }

    // ---- subdomain pairs of this thread, packed in one word: LDS index of the colour-0 cell
    // (bits 0-15), its coefficient-table index (bits 16-27), wall flags (bits 28-29) and whether
    // the pair's colour-1 cell is at -1 (bit 30)
    // Pair order: first the pairs of the deep box (x-pairs 1..hbx-2, rows 2..by-1, planes 2..bz-1),
    // whose colour-0 cells read no halo, then the shell around it.  Entries m < a.md of every thread
    // are deep (a.md: whole relax groups), so their colour 0 can run while the halo is in flight.
    const int hbx = bx / 2, npairs = hbx * by * bz;
    const int dpx = hbx > 2 ? hbx - 2 : 0, dpy = by > 2 ? by - 2 : 0, dpz = bz > 2 ? bz - 2 : 0;
    const int ndeep = dpx * dpy * dpz;
    auto pair_of = [&](int p, int &pi, int &j, int &k) {
        if (p < ndeep) {
            pi = 1 + p % dpx;
            j = 2 + (p / dpx) % dpy;
            k = 2 + p / (dpx * dpy);
            return;
        }
        int q = p - ndeep;
        if (ndeep == 0) {   // no deep box: natural order
            pi = q % hbx;
            j = (q / hbx) % by + 1;
            k = q / (hbx * by) + 1;
            return;
        }
        const int s1 = 2 * hbx * by;   // planes 1 and bz
        if (q < s1) {
            k = q < hbx * by ? 1 : bz;
            const int r = q % (hbx * by);
            pi = r % hbx;
            j = r / hbx + 1;
            return;
        }
        q -= s1;
        const int rr = 2 * hbx + 2 * (by - 2);   // shell of a middle plane: rows 1, by and the end pairs
        k = q / rr + 2;
        int r = q % rr;
        if (r < 2 * hbx) {
            j = r < hbx ? 1 : by;
            pi = r % hbx;
        } else {
            r -= 2 * hbx;
            j = r / 2 + 2;
            pi = (r & 1) ? hbx - 1 : 0;
        }
    };
    auto pack = [](int c, int ti, int walls, int neg) { return c | (ti << 16) | (walls << 28) | (neg << 30); };
    constexpr int NP = COLS ? 1 : MAXP, NR = COLS ? 1 : RB_MAXR;
    int pw[NP];
    T rh[NP][2];
#pragma unroll
    for (int m = 0; m < NP; ++m) {
        const int p = t + m * NT;
        pw[m] = pack(dummy, 0, 0, 0);
        rh[m][0] = rh[m][1] = T(0);
        if (!COLS && p < npairs) {
            int pi, j, k;
            pair_of(p, pi, j, k);
            const int i0 = 2 * pi + 1;
            const int gj = oy + j;
            // colour c relaxes the cell with (gi + gj + gk + c) odd
            const int off0 = ((ox + i0 + gj + oz + k) & 1) ? 0 : 1;
            pw[m] = pack(L(i0 + off0, j, k), (i0 + off0) + cw * j, wall_bits(gj), off0);
            rh[m][0] = a.rhs[d.in(ox + i0 + off0, gj, oz + k)];
            rh[m][1] = a.rhs[d.in(ox + i0 + 1 - off0, gj, oz + k)];
        }
    }
    // ---- colour-0 cells of the face ring owned by neighbours, recomputed here.  Face f has fixed
    // coordinate 0 or b+1 along its axis A and spans 1..bU x 1..bV (U = y for x faces, else x);
    // with bU even each U-line holds bU/2 colour-0 cells.
    int rw[NR];   // packed as the pair words
    T rr[NR];
#pragma unroll
    for (int m = 0; m < NR; ++m) {
        rw[m] = pack(dummy, 0, 0, 0);
        rr[m] = T(0);
    }
    if (!COLS) {
        const int nr = rb_ring_total(bx, by, bz);
#pragma unroll
        for (int m = 0; m < NR; ++m) {
            int e = t + m * NT;
            rw[m] = pack(dummy, 0, 0, 0);
            rr[m] = T(0);
            if (e < nr) {
                int f;   // 0 x faces, 1 y faces, 2 z faces; two faces per axis
                if (e < by * bz) f = 0;
                else if ((e -= by * bz) < bx * bz) f = 1;
                else { e -= bx * bz; f = 2; }
                const int bU = f == 0 ? by : bx, bV = f == 2 ? by : bz;
                const int half = bU / 2 * bV, side = e / half;
                const int r = e - side * half, v = r / (bU / 2) + 1, uq = r % (bU / 2);
                const int dxn = f == 0 ? (side ? 1 : -1) : 0, dyn = f == 1 ? (side ? 1 : -1) : 0,
                          dzn = f == 2 ? (side ? 1 : -1) : 0;
                if (neighbour(dxn, dyn, dzn) >= 0) {
                    // local coordinates with u = 2 uq + 1 + s (s picks the colour-0 cell)
                    int li, lj, lk;
                    const int cA = side ? (f == 0 ? bx + 1 : (f == 1 ? by + 1 : bz + 1)) : 0;
                    if (f == 0) { li = cA; lj = 2 * uq + 1; lk = v; }
                    else if (f == 1) { li = 2 * uq + 1; lj = cA; lk = v; }
                    else { li = 2 * uq + 1; lj = v; lk = cA; }
                    const int s = ((ox + li + oy + lj + oz + lk) & 1) ? 0 : 1;
                    if (f == 0) lj += s; else li += s;
                    const int gi = wrap(ox + li, d.nx), gk = wrap(oz + lk, d.nz);
                    int gj = oy + lj;
                    if (per_y) gj = wrap(gj, d.ny);
                    rw[m] = pack(L(li, lj, lk), li + cw * lj, wall_bits(gj), 0);
                    rr[m] = a.rhs[d.in(gi, gj, gk)];
                }
            }
        }
    }
    // ---- column form: the column of this thread.  The subdomain's columns march z from 0 to bz+1
    // in colour 0 (the two end cells are the z faces of the ring) and from 1 to bz in colour 1;
    // after them come the columns of the ring's x faces (2*by) and y faces (2*bx), colour 0 only, z
    // from 1 to bz, none beyond a wall.  FORM 2 orders the subdomain's columns interior first:
    // those at least 3 cells from every x and y face (i in 3..bx-2, j in 3..by-2), padded to whole
    // wavefronts where the threads allow, then the frame of the two outer rings.
    // The cells of one colour in a thread's range are its end cell, next to the z face the range
    // ends at (the lowest; the highest in FORM 2's upper halves), and the rest, marched upward.  In
    // a wavefront of interior columns only (csplit), the rest of each colour reads no halo value
    // and sends none (colour 0 is at least 2 cells from every face, colour 1 at least 3), so it
    // relaxes while the halo exchange is in flight: colour 1's after the publish, the next
    // iteration's colour 0 after that.  A thread without a column has the dummy cell as its end
    // cell and no rest; cells that are not there are masked off, and a wave without any skips the
    // pass.
    int cb0 = dummy, cr0 = dummy, nr0 = 0;   // colour 0: end cell, first of the rest, their count
    int cb1 = dummy, cr1 = dummy, nr1 = 0;   // colour 1
    bool csplit = false;
    T cmui = 1, cmuip = 1, cmvj = 1, cmvjp = 1, cmw = 1, cq = qconst, can = T(0), cas = T(0);
    T rb0 = T(0), rb1 = T(0);
    T r0[COLS ? ZC - 1 : 1], r1[COLS ? ZC - 1 : 1];
#pragma unroll
    for (int n = 0; n < (COLS ? ZC - 1 : 1); ++n) r0[n] = r1[n] = T(0);
    if (COLS) {
        // FORM 2: threads tc and tc + RB_THREADS share column tc, the lower and the upper half of its
        // z range
        const int tc = t % RB_THREADS, half = t / RB_THREADS;
        const int nin = bx * by, nxf = 2 * by, nyf = 2 * bx;
        int nI = 0, nIp = 0;   // interior columns, and the threads they take with their padding
        if (FORM == 2 && bx > 4 && by > 4) {
            nI = (bx - 4) * (by - 4);
            nIp = (nI + 63) / 64 * 64;
            if (nIp + (nin - nI) + nxf + nyf > RB_THREADS) nIp = nI;
        }
        const int nsub = nIp + nin - nI;   // threads of the subdomain's columns, padding included
        int cli = 0, clj = 0, kz0 = 0, kz1 = -1, kc0 = 1, kc1 = bz;   // colour-0 and colour-1 z ranges
        bool inner = false;
        if (tc < nsub) {
            if (tc < nI) {
                cli = 3 + tc % (bx - 4); clj = 3 + tc / (bx - 4); inner = true;
            } else if (tc >= nIp) {
                const int f = tc - nIp;
                if (nI == 0) {   // natural order
                    cli = f % bx + 1; clj = f / bx + 1;
                } else if (f < 4 * bx) {   // rows 1, 2, by-1, by
                    const int r = f / bx;
                    cli = f % bx + 1; clj = r < 2 ? r + 1 : by - 3 + r;
                } else {   // columns 1, 2, bx-1, bx of rows 3 .. by-2
                    const int g2 = f - 4 * bx, c = g2 % 4;
                    clj = 3 + g2 / 4; cli = c < 2 ? c + 1 : bx - 3 + c;
                }
                inner = true;
            }
            if (inner) { kz0 = 0; kz1 = bz + 1; }
        } else if (tc < nsub + nxf) {
            const int e = tc - nsub;
            cli = e < by ? 0 : bx + 1; clj = e % by + 1; kz0 = 1; kz1 = bz;
        } else if (tc < nsub + nxf + nyf) {
            const int e = tc - nsub - nxf;
            clj = e < bx ? 0 : by + 1; cli = e % bx + 1;
            if (neighbour(0, clj == 0 ? -1 : 1, 0) >= 0) { kz0 = 1; kz1 = bz; }
        }
        // the wavefront's threads tc are 64 consecutive ones: all interior (or padding)
        csplit = FORM == 2 && a.ovl && ((tc >> 6) + 1) * 64 <= nIp;
        const bool top = FORM == 2 && half == 1;   // the end cell is the highest of the range
        if (FORM == 2) {
            const int h0 = (kz1 - kz0 + 2) / 2, h1 = bz / 2;   // positions in the lower halves
            if (half == 0) { kz1 = kz0 + h0 - 1; kc1 = h1; }
            else { kz0 += h0; kc0 = h1 + 1; }
        }
        if (kz1 >= kz0) {
            const int gi = wrap(ox + cli, d.nx);
            int gj = oy + clj;
            if (per_y) gj = wrap(gj, d.ny);
            const int par = (ox + cli + oy + clj + oz) & 1;   // colour c relaxes (par + lk + c) odd
            // colour 0: cells k0, k0 + 2, ..., n0 of them
            const int k0 = kz0 + (((par + kz0) & 1) ? 0 : 1);
            const int n0 = k0 <= kz1 ? (kz1 - k0) / 2 + 1 : 0;
            if (n0 > 0) {
                const int kb = top ? k0 + 2 * (n0 - 1) : k0, kr = top ? k0 : k0 + 2;
                cb0 = L(cli, clj, kb);
                rb0 = a.rhs[d.in(gi, gj, wrap(oz + kb, d.nz))];
                nr0 = n0 - 1;
                if (nr0 > 0) cr0 = L(cli, clj, kr);
#pragma unroll
                for (int n = 0; n < ZC - 1; ++n)
                    r0[n] = n < nr0 ? a.rhs[d.in(gi, gj, wrap(oz + kr + 2 * n, d.nz))] : T(0);
            }
            if (inner) {
                const int k1 = kc0 + (((par + kc0) & 1) ? 1 : 0);   // colour 1: (par + lk) even
                const int n1 = k1 <= kc1 ? (kc1 - k1) / 2 + 1 : 0;
                if (n1 > 0) {
                    const int kb = top ? k1 + 2 * (n1 - 1) : k1, kr = top ? k1 : k1 + 2;
                    cb1 = L(cli, clj, kb);
                    rb1 = a.rhs[d.in(gi, gj, oz + kb)];
                    nr1 = n1 - 1;
                    if (nr1 > 0) cr1 = L(cli, clj, kr);
#pragma unroll
                    for (int n = 0; n < ZC - 1; ++n) r1[n] = n < nr1 ? a.rhs[d.in(gi, gj, oz + kr + 2 * n)] : T(0);
                }
            }
            if (IBM) {   // the face coefficients of the column, as the streaming sweeps form them
                const int sx = d.sx, gip = gi == d.nx ? 1 : gi + 1, gjp = (per_y && gj == d.ny) ? 1 : gj + 1;
                cmui = a.mu_u[(size_t)gi + (size_t)sx * gj];
                cmuip = a.mu_u[(size_t)gip + (size_t)sx * gj];
                cmvj = a.mu_v[(size_t)gi + (size_t)sx * gj];
                cmvjp = a.mu_v[(size_t)gi + (size_t)sx * gjp];
                cmw = a.mu_w[(size_t)gi + (size_t)sx * gj];
            }
            if (STRETCH) {
                can = (T)(a.g.ihv[gj + 1] * a.g.ihc[gj]);
                cas = (T)(a.g.ihv[gj] * a.g.ihc[gj]);
                const T denom = (cmui + cmuip) * a.s.idx2 + (cmw + cmw) * a.s.idz2 + (cmvj * cas + cmvjp * can);
                cq = -a.omega / denom;
            } else if (IBM) {
                const T denom = (cmui + cmuip) * a.s.idx2 + (cmw + cmw) * a.s.idz2 + (cmvj + cmvjp) * a.s.idy2;
                cq = -a.omega / denom;
            }
            // no flux through a wall face: a zero coefficient (the denominator keeps the face, as the
            // streaming sweeps' does; the halo row behind the wall holds zeros)
            const int wb = wall_bits(gj);
            if (wb & 1) cmvjp = T(0);
            if (wb & 2) cmvj = T(0);
        }
    }
    // ---- exchange lists (built once per plan by rb_xlist_kernel): entry e = t + jj * NT
    __shared__ int nbr_from[19];   // the workgroup that sends direction q's region to this one (18: none)
    if (t < 18) {
        int dx, dy, dz;
        rb_dir(t, dx, dy, dz);
        nbr_from[t] = neighbour(-dx, -dy, -dz);
    }
    if (t == 18) nbr_from[18] = w;
    int xpub[HE], xdst[HE];
#pragma unroll
    for (int jj = 0; jj < HE; ++jj) {
        const size_t e = (size_t)t + (size_t)jj * NT;
        xpub[jj] = a.xl[(size_t)w * RB_XSTRIDE + e];
        xdst[jj] = a.xl[((size_t)nwg + w) * RB_XSTRIDE + e];
    }
    bool failed = false;
    __syncthreads();
    // per entry: whether it waits for a sender, the sender's word (of the even buffer; of no use to an
    // entry that does not wait) and the cell
    bool xwait[HE];
    unsigned xsrc[HE];
#pragma unroll
    for (int jj = 0; jj < HE; ++jj) {
        xwait[jj] = (xdst[jj] >> 25) & 1;
        xsrc[jj] = (unsigned)(nbr_from[(xdst[jj] >> 20) & 31] * 2 * RB_XSTRIDE * NW + t + jj * NT);
        xdst[jj] &= 0xfffff;
    }

    // relax the cell of packed word pw shifted by dlt (0: the colour-0 cell, +-1: its pair partner)
    auto relax = [&](int pwd, int dlt, T rhs) -> T {
        const int c = (pwd & 0xffff) + dlt, ti = ((pwd >> 16) & 0xfff) + dlt;
        T mui = 1, muip = 1, mvj = 1, mvjp = 1, mw = 1, q = qconst;
        if (IBM) {
            mui = C[ti]; muip = C[ti + cpl]; mvj = C[ti + 2 * cpl]; mvjp = C[ti + 3 * cpl]; mw = C[ti + 4 * cpl];
            q = C[ti + 5 * cpl];
        }
        T denom;
        const T p0 = X[c];
        const T r = sor_residual_core<T, false>(p0, X[c + 1], X[c - 1], X[c + TXP], X[c - TXP],
                                                X[c + PLANE], X[c - PLANE], mui, muip, mvj, mvjp, mw, mw,
                                                (pwd >> 28) & 1,
                                                (pwd >> 29) & 1, rhs, a.s, T(0), T(0), denom);
        return p0 + r * q;
    };
    auto partner = [](int pwd) { return ((pwd >> 30) & 1) ? -1 : 1; };
    // Column form: the cells of one colour in this thread's range, the end cell ce and / or the rest
    // (n cells upward from c0, two planes apart; the upper z neighbour of a cell is the lower one of
    // the next).  The pass is bound by VALU issue (25 operations a cell, four cycles each per wave),
    // so it spends nothing on cells that are not there: a lane without a cell is masked off, a wave
    // without any skips the pass, and every operand is an immediate offset from the thread's one
    // address.  Cells of one colour never read each other: where every working lane of the wave has
    // them (nmin, wave-uniform), two or three cells' operands are loaded before the first is stored,
    // since the compiler cannot move an LDS load above a store.  Per iteration, FP32 / FP64, against
    // every lane relaxing every slot (absent cells in a dummy): 4.9 -> 4.5 / 6.9 -> 6.5 us at
    // 192 x 128 x 96, 4.4 -> 3.0 / 6.2 -> 3.6 us at 96 x 64 x 48.
    struct Ops {
        T p, xp, xm, yp, ym, zl, zh;
    };
    auto relax_ops = [&](const Ops &o, T rhs) -> T {
        T denom;
        const T r = sor_residual_core<T, STRETCH>(o.p, o.xp, o.xm, o.yp, o.ym, o.zh, o.zl, cmui, cmuip, cmvj, cmvjp,
                                                  cmw, cmw, false, false, rhs, a.s, can, cas, denom);
        return o.p + r * cq;
    };
    auto fetch = [&](const T *B, Ops &o) {   // B: the cell one plane below
        o.ym = B[PLANE - TXP];
        o.xm = B[PLANE - 1];
        o.p = B[PLANE];
        o.xp = B[PLANE + 1];
        o.yp = B[PLANE + TXP];
        o.zh = B[2 * PLANE];
    };
    auto colour = [&](auto end_, auto rest_, bool has, int ce, T re, int c0, int n, int nmin, const T *rhs) {
        constexpr bool END = decltype(end_)::value, REST = decltype(rest_)::value;
        if (!has) return;
        if (END) {
            Ops e;
            T *E = X + (ce - PLANE);
            e.zl = E[0];
            fetch(E, e);
            E[PLANE] = relax_ops(e, re);
        }
        if (!REST) return;
        T *R = X + (c0 - PLANE);
        T zlo = R[0];
        auto cells = [&](auto first_, auto count_) {
            constexpr int g = decltype(first_)::value, CN = decltype(count_)::value;
            if (g >= ZC - 1) return;
            if (CN > 1 && nmin >= g + CN) {
                Ops o[CN];
#pragma unroll
                for (int u = 0; u < CN; ++u) {
                    o[u].zl = zlo;
                    fetch(R + 2 * PLANE * (g + u), o[u]);
                    zlo = o[u].zh;
                }
#pragma unroll
                for (int u = 0; u < CN; ++u) R[2 * PLANE * (g + u) + PLANE] = relax_ops(o[u], rhs[g + u]);
                return;
            }
#pragma unroll
            for (int u = 0; u < CN; ++u) {
                if (g + u < n) {
                    Ops o;
                    o.zl = zlo;
                    fetch(R + 2 * PLANE * (g + u), o);
                    zlo = o.zh;
                    R[2 * PLANE * (g + u) + PLANE] = relax_ops(o, rhs[g + u]);
                }
            }
        };
        using std::integral_constant;
        cells(integral_constant<int, 0>{}, integral_constant<int, 3>{});
        if (FORM == 2) {   // six cells, of which the last is often some lanes' only
            cells(integral_constant<int, 3>{}, integral_constant<int, 2>{});
            cells(integral_constant<int, 5>{}, integral_constant<int, 1>{});
        } else {
            cells(integral_constant<int, 3>{}, integral_constant<int, 3>{});
            cells(integral_constant<int, 6>{}, integral_constant<int, 3>{});
            cells(integral_constant<int, 9>{}, integral_constant<int, 3>{});
        }
    };
    static_assert(RB_ZC2 == 7 && RB_ZC1 == 13, "the chunks of colour() cover a range");
    constexpr std::true_type yes{};
    constexpr std::false_type no{};
    const bool has0 = COLS && cb0 != dummy, has1 = COLS && cb1 != dummy;
    // cells that every lane of the wave with any has
    auto wave_min = [&](bool has, int n) {
        int m = 0;
        while (m < ZC - 1 && !__any(has && n <= m)) ++m;
        return __builtin_amdgcn_readfirstlane(m);
    };
    const int nm0 = COLS ? wave_min(has0, nr0) : 0, nm1 = COLS ? wave_min(has1, nr1) : 0;
    if (COLS && nr0 == 0) cr0 = cb0;   // addresses inside the tile
    if (COLS && nr1 == 0) cr1 = cb1;

    unsigned long long *F = a.faces;
    // publish the colour-1 layer cells, tagged with iteration s, into buffer s & 1
    auto publish = [&](int s) {
        const unsigned tag = a.tag0 + (unsigned)s + 1u;
        const size_t mybase = ((size_t)(w * 2 + (s & 1)) * RB_XSTRIDE) * NW;
        // every layer value first (one LDS wait), then the stores, the words of an FP64 value in
        // separate runs so that each store instruction fills whole lines (interleaved: 9.4 us per
        // FP64 iteration at 192 x 128 x 96 instead of 7.1)
        T val[HE];
#pragma unroll
        for (int jj = 0; jj < HE; ++jj) val[jj] = X[xpub[jj]];
#pragma unroll
        for (int jj = 0; jj < HE; ++jj) asm volatile("" : "+v"(val[jj]));
#pragma unroll
        for (int jj = 0; jj < HE; ++jj) {
            if (t + jj * NT >= a.total) break;   // (whole waves but one)
            unsigned long long wv[NW];
            TW::pack(val[jj], tag, wv);
            unsigned long long *dst = F + mybase + (size_t)(t + jj * NT);
#pragma unroll
            for (int q = 0; q < NW; ++q)
                __hip_atomic_store(dst + q * RB_XSTRIDE, wv[q], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
    };
    for (int s = 0; s < a.iters; ++s) {
        // The packed words are loop-invariant; left visible, the compiler would keep every address
        // derived from them (13 per cell and colour) live across the loop and run out of registers.
        // An empty asm that claims to redefine them makes the few address adds happen per use.
#pragma unroll
        for (int m = 0; m < NP; ++m) asm volatile("" : "+v"(pw[m]));
#pragma unroll
        for (int m = 0; m < NR; ++m) asm volatile("" : "+v"(rw[m]));
#pragma unroll
        for (int jj = 0; jj < HE; ++jj) asm volatile("" : "+v"(xpub[jj]), "+v"(xdst[jj]), "+v"(xsrc[jj]));
        // ---- colour 0 on the subdomain and the face ring.  Cells of one colour never neighbour
        // each other, so each is stored as soon as it is formed; groups of RB_G cells with a
        // scheduling barrier between them bound the loads in flight (registers).  After the first
        // iteration the deep groups (g < a.md) were relaxed while the halo was in flight.
        if (COLS) {
            // column data: loop-invariant, kept from being hoisted as per-cell addresses (as above)
            asm volatile("" : "+v"(cb0), "+v"(cr0), "+v"(cb1), "+v"(cr1));
            // colour 0: the end cells, and the rest where the last exchange's wait has not relaxed it
            if (!csplit || s == 0) colour(yes, yes, has0, cb0, rb0, cr0, nr0, nm0, r0);
            else colour(yes, no, has0, cb0, rb0, cr0, nr0, nm0, r0);
            __syncthreads();
            // colour 1: the end cells, and the rest where it is not left for the exchange's flight
            if (!csplit) colour(yes, yes, has1, cb1, rb1, cr1, nr1, nm1, r1);
            else colour(yes, no, has1, cb1, rb1, cr1, nr1, nm1, r1);
            __syncthreads();
        }
#pragma unroll
        for (int g = 0; g < NP; g += RB_G) {
            if (COLS) break;
            if (s > 0 && g < a.md) continue;
            T nv[RB_G];
#pragma unroll
            for (int u = 0; u < RB_G; ++u) nv[u] = relax(pw[g + u], 0, rh[g + u][0]);
#pragma unroll
            for (int u = 0; u < RB_G; ++u) X[pw[g + u] & 0xffff] = nv[u];
            __builtin_amdgcn_sched_barrier(0);
        }
        if (!COLS) {
            T nv[NR];
#pragma unroll
            for (int m = 0; m < NR; ++m) nv[m] = relax(rw[m], 0, rr[m]);
#pragma unroll
            for (int m = 0; m < NR; ++m) X[rw[m] & 0xffff] = nv[m];
            __syncthreads();
        }
        // ---- colour 1 on the subdomain: its neighbours are subdomain or ring cells, all updated
#pragma unroll
        for (int g = 0; g < NP; g += RB_G) {
            if (COLS) break;
            T nv[RB_G];
#pragma unroll
            for (int u = 0; u < RB_G; ++u) nv[u] = relax(pw[g + u], partner(pw[g + u]), rh[g + u][1]);
#pragma unroll
            for (int u = 0; u < RB_G; ++u) X[(pw[g + u] & 0xffff) + partner(pw[g + u])] = nv[u];
            __builtin_amdgcn_sched_barrier(0);
        }
        if (!COLS) __syncthreads();
        // the last iteration needs no exchange, unless the defect epilogue reads the final halo
        if (s == a.iters - 1 && !a.defect) {
            if (COLS && a.ovl) {   // the rest of colour 1 in the split wavefronts, before the write-back
                if (csplit) colour(no, yes, has1, cb1, rb1, cr1, nr1, nm1, r1);
                __syncthreads();
            }
            break;
        }

        // ---- publish this subdomain's colour-1 layer cells
        const int buf = s & 1;
        const unsigned tag = a.tag0 + (unsigned)s + 1u;
        publish(s);
        // ---- column form, split wavefronts: the rest of colour 1, then (after every colour-1 cell
        // it reads is final) the next iteration's rest of colour 0, while the layers travel.  The
        // publish reads only colour-1 layer cells, which neither writes, and the halo the pull
        // writes is read by neither.
        if (COLS && a.ovl) {
            if (csplit) colour(no, yes, has1, cb1, rb1, cr1, nr1, nm1, r1);
            if (s < a.iters - 1) {
                __syncthreads();
                if (csplit) colour(no, yes, has0, cb0, rb0, cr0, nr0, nm0, r0);
            }
        }
        // ---- the next iteration's colour 0 on the deep groups, while the neighbours' layers travel:
        // those cells read only subdomain cells of colour 1, final for this iteration; the barrier
        // lets the publish read its layers first
        if (!COLS && s < a.iters - 1) {
            __syncthreads();
#pragma unroll
            for (int g = 0; g < NP; g += RB_G) {
                if (g >= a.md) continue;
                T nv[RB_G];
#pragma unroll
                for (int u = 0; u < RB_G; ++u) nv[u] = relax(pw[g + u], 0, rh[g + u][0]);
#pragma unroll
                for (int u = 0; u < RB_G; ++u) X[pw[g + u] & 0xffff] = nv[u];
                __builtin_amdgcn_sched_barrier(0);
            }
        }
        // ---- pull the neighbours' layers: poll the tagged words until all carry this tag
        // source word of entry jj: the sender's buffer `buf`, entry e, in words
        const unsigned long long *S = F + (size_t)buf * RB_XSTRIDE * NW;   // the senders' buffer of this parity
        unsigned long long got[HE][NW];
#pragma unroll
        for (int jj = 0; jj < HE; ++jj) {
#pragma unroll
            for (int q = 0; q < NW; ++q) got[jj][q] = 0;
            if (!xwait[jj]) continue;
#pragma unroll
            for (int q = 0; q < NW; ++q)
                got[jj][q] = __hip_atomic_load(S + (xsrc[jj] + (unsigned)(q * RB_XSTRIDE)), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
        for (int spins = 0; !failed; ++spins) {
            bool ready = true;
#pragma unroll
            for (int jj = 0; jj < HE; ++jj)
#pragma unroll
                for (int q = 0; q < NW; ++q)
                    ready = ready && (!xwait[jj] || (unsigned)(got[jj][q] >> 32) == tag);
            if (ready) break;
            if (spins >= a.spin_limit) {   // a neighbour never published: flag it and run to the end
                __hip_atomic_store(a.err, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                failed = true;
                break;
            }
            __builtin_amdgcn_s_sleep(1);
#pragma unroll
            for (int jj = 0; jj < HE; ++jj)
#pragma unroll
                for (int q = 0; q < NW; ++q)
                    if (xwait[jj] && (unsigned)(got[jj][q] >> 32) != tag)
                        got[jj][q] = __hip_atomic_load(S + (xsrc[jj] + (unsigned)(q * RB_XSTRIDE)), __ATOMIC_RELAXED,
                                                       __HIP_MEMORY_SCOPE_AGENT);
        }
#pragma unroll
        for (int jj = 0; jj < HE; ++jj)
            if (xwait[jj]) X[xdst[jj]] = TW::unpack(got[jj]);
        __syncthreads();
    }
    if (!a.defect) {
        // ---- write the subdomain back
        for (int q = t; q < bx * by * bz; q += NT) {
            const int i = q % bx + 1, j = (q / bx) % by + 1, k = q / (bx * by) + 1;
            a.x[d.in(ox + i, oy + j, oz + k)] = X[L(i, j, k)];
        }
        return;
    }
    // ---- check epilogue: the halo holds the neighbours' final values (exchanged above).  A thread
    // owns a column (i, j) of the subdomain, or half of its planes where the workgroup has the
    // threads (EP = 2), and marches k, keeping Phi = phi_in + e of planes k-1, k, k+1 of its column;
    // the face coefficients of a column do not change with k (z-invariant tables).  The pointers
    // are declared unaliased so the loads of the next plane may issue before this plane's stores.
    // The operands handed to sor_residual_core are those cell_residual forms, so the defect equals
    // the separate kernel's.
    double mx = 0.0;
    const int ncol = bx * by;
    const int EP = NT >= 2 * ncol ? 2 : 1;
    if (t < EP * ncol) {
        const int col = t % ncol, part = t / ncol;
        const int li = col % bx + 1, lj = col / bx + 1;
        const int hz = (bz + EP - 1) / EP;
        const int lk0 = 1 + part * hz, lk1 = lk0 + hz - 1 < bz ? lk0 + hz - 1 : bz;
        const int i = ox + li, j = oy + lj, nx = d.nx, ny = d.ny, nz = d.nz;
        const bool per2 = per_y;
        const int ip = i == nx ? 1 : i + 1, im = i == 1 ? nx : i - 1;
        int jp = j + 1, jm = j - 1;
        if (per2) {
            if (jp > ny) jp = 1;
            if (jm < 1) jm = ny;
        }
        const bool wn_ = !per2 && j == ny, ws_ = !per2 && j == 1;
        const int jn = wn_ ? j : jp, js = ws_ ? j : jm;
        const int ljn = wn_ ? lj : lj + 1, ljs = ws_ ? lj : lj - 1;   // LDS rows of the y neighbours
        double mui = 1, muip = 1, mvj = 1, mvjp = 1, mwk = 1, mwkp = 1;
        if (IBM) {
            mui = a.mu64.u[a.mu64.at(i, j, 1)];
            muip = a.mu64.u[a.mu64.at(ip, j, 1)];
            mvj = a.mu64.v[a.mu64.at(i, j, 1)];
            mvjp = a.mu64.v[a.mu64.at(i, jp, 1)];
            mwk = a.mu64.w[a.mu64.at(i, j, 1)];
            mwkp = mwk;   // z-invariant table
        }
        const double *__restrict__ pin = a.phi_in;
        const double *__restrict__ r64 = a.rhs64;
        double *__restrict__ pout = a.phi_out;
        float *__restrict__ rout = a.r_out;
        // the iterate of one cell: phi_in + e (FP32 batches), or the tile's own value
        constexpr bool F64 = sizeof(T) == 8;
        auto Pc = [&](int gi, int gj, int gk, int xi, int xj, int xk) {
            return F64 ? (double)X[L(xi, xj, xk)] : pin[d.in(gi, gj, gk)] + (double)X[L(xi, xj, xk)];
        };
        double an = 0.0, as = 0.0;
        if (STRETCH) {
            an = a.g.ihv[j + 1] * a.g.ihc[j];
            as = a.g.ihv[j] * a.g.ihc[j];
        }
        auto kw = [&](int k) { return k < 1 ? k + nz : (k > nz ? k - nz : k); };
        // z neighbours of the first plane: below the subdomain the lower neighbour wraps periodically
        double pm = Pc(i, j, kw(oz + lk0 - 1), li, lj, lk0 - 1), pc = Pc(i, j, oz + lk0, li, lj, lk0);
#pragma unroll 2
        for (int lk = lk0; lk <= lk1; ++lk) {
            const int k = oz + lk;
            const double pn = Pc(i, j, kw(k + 1), li, lj, lk + 1);
            const double pxp = Pc(ip, j, k, li + 1, lj, lk), pxm = Pc(im, j, k, li - 1, lj, lk);
            const double pyp = Pc(i, jn, k, li, ljn, lk), pym = Pc(i, js, k, li, ljs, lk);
            const size_t c = d.in(i, j, k);
            double denom;
            const double r = sor_residual_core<double, STRETCH>(pc, pxp, pxm, pyp, pym, pn, pm, mui, muip, mvj, mvjp,
                                                                mwk, mwkp, wn_, ws_, r64[c], a.s64, an, as, denom);
            pout[c] = pc;
            if (!F64) rout[c] = (float)r;
            mx = nanmax_any(mx, fabs(r));
            pm = pc;
            pc = pn;
        }
    }
    // ---- the maximum over workgroups without fences: every workgroup publishes its partial as two
    // tagged words (tag0 + iters + 1, unique to this launch) after the face buffers; workgroup 0
    // polls them all (bounded) and writes the result to red_max[0] and the host slot
    __shared__ double wred[NT / 64];
    for (int off = 32; off > 0; off >>= 1) mx = nanmax_any(mx, __shfl_xor(mx, off, 64));
    if ((t & 63) == 0) wred[t >> 6] = mx;
    __syncthreads();
    const unsigned mtag = a.tag0 + (unsigned)a.iters + 1u;
    unsigned long long *MP = a.faces + (size_t)nwg * 2 * RB_XSTRIDE * NW;   // 2 words per workgroup
    if (t == 0) {
        double m = wred[0];
        for (int q = 1; q < NT / 64; ++q) m = nanmax_any(m, wred[q]);
        unsigned long long wv[2];
        Tagged<double>::pack(m, mtag, wv);
        __hip_atomic_store(MP + 2 * w, wv[0], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __hip_atomic_store(MP + 2 * w + 1, wv[1], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    if (blockIdx.x != 0) return;
    double m = 0.0;
    for (int q = t; q < nwg; q += NT) {
        unsigned long long wv[2];
        for (int spins = 0;; ++spins) {
            wv[0] = __hip_atomic_load(MP + 2 * q, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            wv[1] = __hip_atomic_load(MP + 2 * q + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            if ((unsigned)(wv[0] >> 32) == mtag && (unsigned)(wv[1] >> 32) == mtag) break;
            if (failed || spins >= a.spin_limit) {
                __hip_atomic_store(a.err, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                failed = true;
                break;
            }
            __builtin_amdgcn_s_sleep(1);
        }
        m = nanmax_any(m, Tagged<double>::unpack(wv));
    }
    __syncthreads();   // wred reused
    for (int off = 32; off > 0; off >>= 1) m = nanmax_any(m, __shfl_xor(m, off, 64));
    if ((t & 63) == 0) wred[t >> 6] = m;
    __syncthreads();
    if (t == 0) {
        for (int q = 1; q < NT / 64; ++q) m = nanmax_any(m, wred[q]);
        m = nanmax_any(wred[0], m);
        const unsigned long long errw = __hip_atomic_load(&a.red_max[1], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        a.red_max[0] = (unsigned long long)__double_as_longlong(m);
        a.host_slot[0] = m;
        a.host_slot[1] = __longlong_as_double((long long)errw);
        __threadfence_system();
        reinterpret_cast<volatile unsigned long long *>(a.host_slot)[2] = a.seq;
    }
}

// Exchange lists of workgroup w (subdomain id), entry e of the colour-1 cells of the 18 regions
// (faces two layers deep, then edges one cell thick; entry e = t + jj * threads of thread t).
// Neighbours share the extents along their common face or edge, so a region has the same cells on
// both sides whatever the two subdomains' other extents, and its entries the same numbers.
// Publish word: the LDS cell this workgroup sends for its neighbour in direction D (bits 0-19).
// Pull word: the halo cell where the region that the neighbour in direction -D sent lands (bits
// 0-19), D (bits 20-24) and whether to wait for it (bit 25).  Colour 1 has an even global
// coordinate sum; cells 2k and 2k+1 of a region's natural order are neighbours along its first
// extent above one, of opposite colours, and entry k of the region is the one of the two of
// colour 1, on both sides alike.
// An entry of the list without a cell to send publishes the dummy cell, one past the list's end is
// not sent; an entry with no sender (beyond a wall, or past the end) neither loads nor stores.  Its
// direction is 18, this workgroup itself, so that its word has an address in the buffer like any
// other's (with a real direction there, the kernel came out 1% slower at 100 x 70 x 54).
// Built once per plan; the batch kernel only loads it.
struct RbGeom {
    int nx, ny, nz, px, py, pz, bx, by, bz, per_y, total, dummy;
    RbStride st;
};

__global__ __launch_bounds__(256) void rb_xlist_kernel(RbGeom g, int *xl) {
    const int w = blockIdx.y, nwg = g.px * g.py * g.pz;
    const int e = blockIdx.x * 256 + threadIdx.x;
    if (e >= RB_XSTRIDE) return;
    const int wx = w % g.px, wy = (w / g.px) % g.py, wz = w / (g.px * g.py);
    int ox, oy, oz, bx, by, bz;
    rb_part(g.nx, g.px, wx, ox, bx);
    rb_part(g.ny, g.py, wy, oy, by);
    rb_part(g.nz, g.pz, wz, oz, bz);
    auto L = [&](int i, int j, int k) { return (i + 1) + g.st.row * (j + 1) + g.st.plane * (k + 1); };
    auto has_sender = [&](int dx, int dy, int dz) {   // the neighbour in direction -D exists
        (void)dx;
        (void)dz;
        const int ny_ = wy - dy;
        return g.per_y || (ny_ >= 0 && ny_ < g.py);
    };
    int xpub = g.dummy, xdst = g.dummy | (18 << 20);
    if (e < g.total) {
        int q = 0, off = 0, ex = 0, ey = 0, ez = 0;
        for (; q < 18; ++q) {   // the regions start at the offsets of the largest subdomain
            rb_extent(q, g.bx, g.by, g.bz, ex, ey, ez);
            if (e < off + (ex * ey * ez + 1) / 2) break;
            off += (ex * ey * ez + 1) / 2;
        }
        rb_extent(q, bx, by, bz, ex, ey, ez);
        int dx, dy, dz;
        rb_dir(q, dx, dy, dz);
        const int h = q < 6 ? RB_H : 1;
        const int col = 1, k2 = 2 * (e - off);
        auto cell = [&](int r, auto side, int &cx, int &cy, int &cz) {
            cx = side(dx, r % ex, bx, h);
            cy = side(dy, (r / ex) % ey, by, h);
            cz = side(dz, r / (ex * ey), bz, h);
        };
        // sender side: the layer next to its face D; receiver side: the halo beyond face -D
        auto snd = [](int dd, int rr_, int bb, int hh) { return dd > 0 ? bb - hh + 1 + rr_ : 1 + rr_; };
        auto rcv = [](int dd, int rr_, int bb, int hh) {
            return dd < 0 ? bb + 1 + rr_ : (dd > 0 ? 1 - hh + rr_ : 1 + rr_);
        };
        auto colour = [&](int cx, int cy, int cz) { return ((ox + cx + oy + cy + oz + cz) & 1) ? 0 : 1; };
        // entry k2 / 2 of a region of n cells: the colour-1 one of cells k2 and k2 + 1 (none past
        // the region's end)
        const int n = ex * ey * ez;
        int cx, cy, cz;
        auto pick = [&](auto side) {
            if (k2 >= n) return false;
            cell(k2, side, cx, cy, cz);
            if (colour(cx, cy, cz) == col) return true;
            if (k2 + 1 >= n) return false;
            cell(k2 + 1, side, cx, cy, cz);
            return true;
        };
        if (pick(snd)) xpub = L(cx, cy, cz);
        if (has_sender(dx, dy, dz) && pick(rcv)) xdst = L(cx, cy, cz) | (q << 20) | (1 << 25);
    }
    xl[(size_t)w * RB_XSTRIDE + e] = xpub;
    xl[((size_t)nwg + w) * RB_XSTRIDE + e] = xdst;
}

// ------------------------------------------------------------------------------- host side
static size_t rb_lds_bytes(int plane, int bz, size_t tsize, bool ibm) {
    return ((size_t)rb_dummy(plane, bz) + plane + 2 + (ibm ? 6 * (size_t)plane : 0)) * tsize;
}

template <typename T, bool IBM, int MAXP, int FORM = 0, bool STRETCH = false>
static const void *rb_fn() {
    return reinterpret_cast<const void *>(&rb_lds_kernel<T, IBM, MAXP, FORM, STRETCH>);
}

// pairs per thread: multiples of the group size RB_G; RB_COLS, RB_COLS2: the column forms (only the
// half-column form serves a stretched grid)
template <typename T, bool IBM>
static const void *rb_fn_for(int maxp, bool stretch) {
    if (stretch) return rb_fn<T, IBM, RB_G, 2, true>();
    switch (maxp) {
    case RB_COLS: return rb_fn<T, IBM, RB_G, 1>();
    case RB_COLS2: return rb_fn<T, IBM, RB_G, 2>();
    case 3: return rb_fn<T, IBM, 3>();
    case 6: return rb_fn<T, IBM, 6>();
    case 9: return rb_fn<T, IBM, 9>();
    case 12: return rb_fn<T, IBM, 12>();
    default: return rb_fn<T, IBM, 15>();
    }
}

// threads per workgroup of a plan's kernel form
static int rb_threads(int maxp) { return maxp == RB_COLS2 ? 2 * RB_THREADS : RB_THREADS; }

static int rb_maxp_class(int need) {
    const int c = (need + RB_G - 1) / RB_G * RB_G;
    return c < RB_G ? RB_G : (c <= 15 ? c : 0);
}

// workgroups of this kernel variant that fit on one CU (registers, LDS, waves), from the runtime
static int rb_occupancy(bool fp32, bool ibm, int maxp, bool stretch, size_t lds) {
    const void *fn = fp32 ? (ibm ? rb_fn_for<float, true>(maxp, stretch) : rb_fn_for<float, false>(maxp, stretch))
                          : (ibm ? rb_fn_for<double, true>(maxp, stretch) : rb_fn_for<double, false>(maxp, stretch));
    if (lds > 65536 && hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds) != hipSuccess) {
        (void)hipGetLastError();
        return 0;
    }
    int nb = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&nb, fn, rb_threads(maxp), lds) != hipSuccess) {
        (void)hipGetLastError();
        return 0;
    }
    return nb;
}

// Choose the decomposition: every workgroup co-resident (runtime occupancy) on `share` CUs (0: all
// of them, several workgroups on a CU where they fit),
// the fewest cells per CU, then the smallest exchange.  The half-column form takes any cut of the
// grid into parts of at least 4 cells (rb_part); the pair and whole-column forms, whose lists are
// sized by one shape, need equal even parts.  `why` receives the reason when nothing fits.
bool rb_plan(const mdx_handle *h, bool fp32, int share, RbPlanOut &out, std::string &why) {
    const int nx = h->d.nx, ny = h->d.ny, nz = h->d.nz;
    // single attributes: reading all device properties takes longer than the search below
    auto attr = [&](hipDeviceAttribute_t a) {
        int v = -1;
        if (hipDeviceGetAttribute(&v, a, h->device) != hipSuccess) (void)hipGetLastError();
        return v;
    };
    const int all_cus = attr(hipDeviceAttributeMultiprocessorCount), lds_block = attr(hipDeviceAttributeMaxSharedMemoryPerBlock),
              lds_cu = attr(hipDeviceAttributeMaxSharedMemoryPerMultiprocessor);
    if (all_cus < 1 || lds_block < 1) { why = "no device properties"; return false; }
    if (h->rb_coop && attr(hipDeviceAttributeCooperativeLaunch) != 1) {
        why = "device reports no cooperative launch";
        return false;
    }
    if (h->cfg.periodic[1] && ny % 2) { why = "odd periodic y"; return false; }
    const int cus = share > 0 ? std::min(share, all_cus) : all_cus;
    const size_t lds_max = (size_t)std::max(lds_cu, lds_block);
    const size_t ts = fp32 ? 4 : 8;
    bool found = false;
    double best_cells = 1e300, best_x = 1e300;
    std::map<std::pair<int, size_t>, int> occupancy;   // by form and LDS size
    why = "no decomposition fits (cus=" + std::to_string(cus) + ", lds/block=" + std::to_string(lds_block) +
          ", lds/cu=" + std::to_string(lds_cu) + ")";
    const long max_wg = 4L * cus;
    for (int px = 1; px <= nx / 2; ++px) {
        const int bx = rb_part_max(nx, px);
        if (bx + 2 * RB_H > RB_BX) continue;   // the fixed LDS row
        for (int py = 1; py <= std::max(1, ny / 2); ++py) {
            if ((long)px * py > max_wg) break;
            const int by = rb_part_max(ny, py);
            if (by + 2 * RB_H > RB_BY) continue;   // the fixed LDS plane
            for (int pz = 1; pz <= nz / 2; ++pz) {
                const int bz = rb_part_max(nz, pz);
                if ((long)px * py * pz > max_wg) break;
                const int nwg = px * py * pz;
                // a share: a CU for every workgroup, so that no other launch's workgroups, however
                // they are spread, take the place one of these waits for
                if (share > 0 && nwg > cus) break;
                const bool equal = (nx / 2) % px == 0 && ny % 2 == 0 && (ny / 2) % py == 0 && (nz / 2) % pz == 0;
                // the column form where a thread per column (subdomain and face ring) fits
                const bool colfit = bx * by + 2 * (bx + by) <= RB_THREADS && rb_part_min(nx, px) >= 4 &&
                                    rb_part_min(ny, py) >= 4 && rb_part_min(nz, pz) >= 4;
                int maxp = equal ? rb_maxp_class((bx / 2 * by * bz + RB_THREADS - 1) / RB_THREADS) : 0;
                if (colfit && h->rb_form == 0 && bz <= 4 * RB_ZC2 - 4) maxp = RB_COLS2;
                if (colfit && h->rb_form == 2 && equal && bz <= 2 * RB_ZC1 - 2) maxp = RB_COLS;
                if (!maxp || (h->stretched && maxp != RB_COLS2)) continue;
                // the column forms keep the face coefficients in registers: no LDS table
                const int plane = rb_stride(fp32, maxp == RB_COLS2).plane;
                // packed per-cell words: LDS index (dummy cell and its padding included) < 2^16,
                // coefficient-table index < 2^12
                if (rb_dummy(plane, bz) + plane + 2 >= 65536 || plane >= 4096) continue;
                const size_t lds = rb_lds_bytes(plane, bz, ts, h->ibm_on && maxp > 0);
                if (lds > lds_max) continue;
                if (rb_ring_total(bx, by, bz) > RB_MAXR * RB_THREADS) continue;
                const int total = rb_xchg_total(bx, by, bz);
                if (total > RB_HE * RB_THREADS) continue;
                const double rounds = std::ceil((double)nwg / cus);
                const double cells = rounds * bx * by * bz;
                // a column form where one fits: the pair form relaxes absent cells too (48 x 32 x 24:
                // 4.0 against 2.3 us per FP32 iteration)
                const bool better = (maxp < 0) != (found && out.maxp < 0)
                                        ? maxp < 0 || !found
                                        : cells < best_cells - 0.5 || (cells < best_cells + 0.5 && total < best_x);
                if (!better) continue;
                const auto key = std::make_pair(maxp, lds);
                if (!occupancy.count(key))
                    occupancy[key] = rb_occupancy(fp32, h->ibm_on, maxp, h->stretched, lds);
                const int per_cu = occupancy[key];
                if (per_cu < 1 || nwg > per_cu * cus) continue;
                best_cells = cells;
                best_x = total;
                out = RbPlanOut{px, py, pz, bx, by, bz, maxp, lds, total};
                found = true;
            }
        }
    }
    return found;
}

// the exchange lists of plan p into xl (2 * workgroups * RB_XSTRIDE ints), on the handle's stream
hipError_t rb_build_xlists(mdx_handle *h, const RbPlanOut &p, bool fp32, int *xl) {
    const RbStride st = rb_stride(fp32, p.maxp == RB_COLS2);
    const int nwg = p.px * p.py * p.pz;
    const RbGeom g{h->d.nx, h->d.ny, h->d.nz, p.px, p.py, p.pz, p.bx, p.by, p.bz, h->cfg.periodic[1] ? 1 : 0, p.total,
                   rb_dummy(st.plane, p.bz), st};
    hipLaunchKernelGGL(rb_xlist_kernel, dim3((RB_XSTRIDE + 255) / 256, nwg), dim3(256), 0, h->stream, g, xl);
    return hipGetLastError();
}

size_t rb_xlist_bytes(const RbPlanOut &p) { return 2 * (size_t)p.px * p.py * p.pz * RB_XSTRIDE * sizeof(int); }

size_t rb_faces_bytes(const RbPlanOut &p, bool fp32) {
    const size_t nwg = (size_t)p.px * p.py * p.pz;
    return nwg * 2 * (size_t)RB_XSTRIDE * 8 * (fp32 ? 1 : 2) + nwg * 16;   // faces, then the maxima
}

template <typename T>
static hipError_t rb_launch_t(mdx_handle *h, const RbPlanOut &pl, T *x, const T *rhs, int zero_init, int iters,
                              T *const *mu, const RbDefect *df) {
    RbSet &S = *h->rb;
    RbArgs<T> a;
    a.defect = df != nullptr;
    a.g = grid_k(h);
    a.mu64.u = h->ibm_on ? h->mu64[0] : nullptr;
    a.mu64.v = h->ibm_on ? h->mu64[1] : nullptr;
    a.mu64.w = h->ibm_on ? h->mu64[2] : nullptr;
    a.mu64.plane = h->coef_plane ? 1 : 0;
    a.mu64.sx = h->d.sx;
    a.mu64.sy = h->d.sy;
    a.s64 = SorConst<double>{1.0 / h->dx * (1.0 / h->dx), 1.0 / h->dy * (1.0 / h->dy), 1.0 / h->dz * (1.0 / h->dz)};
    a.phi_in = df ? df->phi_in : nullptr;
    a.rhs64 = h->rhs;
    a.phi_out = df ? df->phi_out : nullptr;
    a.max_part = h->max_part;
    a.r_out = h->r32;
    a.red_max = h->red_max;
    a.host_slot = df ? df->host_slot : nullptr;
    a.seq = df ? df->seq : 0;
    a.skip = df ? df->skip : 0;
    a.skip_tol = df ? df->skip_tol : 0.0;
    a.ovl = h->rb_overlap ? 1 : 0;
    a.d = h->d;
    a.px = pl.px; a.py = pl.py; a.pz = pl.pz;
    a.bx = pl.bx; a.by = pl.by; a.bz = pl.bz;
    a.per_y = h->cfg.periodic[1] ? 1 : 0;
    const double ix2 = 1.0 / h->dx * (1.0 / h->dx), iy2 = 1.0 / h->dy * (1.0 / h->dy), iz2 = 1.0 / h->dz * (1.0 / h->dz);
    if (sizeof(T) == 4)
        a.s = SorConst<T>{(T)(1.0 / (h->dx * h->dx)), (T)(1.0 / (h->dy * h->dy)), (T)(1.0 / (h->dz * h->dz))};
    else
        a.s = SorConst<T>{(T)ix2, (T)iy2, (T)iz2};
    a.omega = (T)(sizeof(T) == 4 ? h->inner_omega : h->cfg.omega);
    a.mu_u = h->ibm_on ? mu[0] : nullptr;
    a.mu_v = h->ibm_on ? mu[1] : nullptr;
    a.mu_w = h->ibm_on ? mu[2] : nullptr;
    a.x = x;
    a.rhs = rhs;
    a.zero_init = zero_init;
    a.iters = iters;
    {
        const int hbx = pl.bx / 2, dpx = hbx > 2 ? hbx - 2 : 0, dpy = pl.by > 2 ? pl.by - 2 : 0,
                  dpz = pl.bz > 2 ? pl.bz - 2 : 0;
        a.md = (dpx * dpy * dpz / RB_THREADS) / RB_G * RB_G;   // whole relax groups only
    }
    a.faces = reinterpret_cast<unsigned long long *>(S.mem);
    a.total = pl.total;
    a.xl = sizeof(T) == 4 ? S.xl32 : S.xl64;
    // tags of this launch: tag + 1 .. tag + iters + 1 (the last for the maxima); before the
    // 32-bit tag would wrap to 0 the face buffer is cleared and the count restarts
    if (S.tag + (unsigned long long)iters + 2ull > 0xffffffffull) {
        hipError_t e = hipMemsetAsync(S.mem, 0, S.faces_bytes, h->stream);
        if (e != hipSuccess) return e;
        S.tag = 0;
    }
    a.tag0 = (unsigned)S.tag;
    S.tag += (unsigned long long)iters + 1ull;
    a.err = h->rb_err;
    a.spin_limit = h->rb_spin_limit;
    const void *fn = h->ibm_on ? rb_fn_for<T, true>(pl.maxp, h->stretched) : rb_fn_for<T, false>(pl.maxp, h->stretched);
    hipError_t e = hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)pl.lds);
    if (e != hipSuccess) return e;
    void *args[] = {&a};
    // The plan holds at most as many workgroups as the CUs take at once (runtime occupancy), and a
    // dispatch waits for nothing but earlier work on this stream, so every workgroup becomes
    // resident with an ordinary launch; the cooperative launch gives the same guarantee formally
    // at about 30 us of extra dispatch time per launch.  Every neighbour wait is bounded and
    // raises the error word, so a workgroup that never arrived ends the batch with an error.
    if (h->rb_coop)
        return hipLaunchCooperativeKernel(fn, dim3(pl.px * pl.py * pl.pz), dim3(rb_threads(pl.maxp)), args,
                                          (unsigned)pl.lds, h->stream);
    return hipLaunchKernel(fn, dim3(pl.px * pl.py * pl.pz), dim3(rb_threads(pl.maxp)), args, (size_t)pl.lds,
                           h->stream);
}

hipError_t launch_rb_lds(mdx_handle *h, bool fp32, int iters, int zero_init, const RbDefect *df) {
    const RbPlanOut &pl = fp32 ? h->rb->plan32 : h->rb->plan64;
    if (fp32) return rb_launch_t<float>(h, pl, h->e32, h->r32, zero_init, iters, h->mu32, df);
    return rb_launch_t<double>(h, pl, h->phi, h->rhs, zero_init, iters, h->mu64, df);
}

}  // namespace mdx

// ------------------------------------------------------------------------------- LDS read rate
// The chip's sustained LDS read bandwidth, the ceiling of the LDS-resident sweeps: every thread of
// 8 workgroups per CU reads 16-byte vectors of a 64 KB LDS array in a rotating, bank-conflict-free
// pattern (index masked into the array) and folds them, so nothing is optimised away.
namespace mdx {
static constexpr int LDSR_VEC = 4096, LDSR_ITERS = 4096;
__global__ __launch_bounds__(256) void lds_read_rate_kernel(float *out) {
    __shared__ float4 buf[LDSR_VEC];
    for (int q = threadIdx.x; q < LDSR_VEC; q += 256) buf[q] = make_float4((float)q, (float)q + 1.f, 0.f, 1.f);
    __syncthreads();
    float4 acc = make_float4(0.f, 0.f, 0.f, 0.f);
    int idx = threadIdx.x;
#pragma unroll 8
    for (int i = 0; i < LDSR_ITERS; ++i) {
        const float4 v = buf[idx & (LDSR_VEC - 1)];
        acc.x += v.x;
        acc.y += v.y;
        acc.z += v.z;
        acc.w += v.w;
        idx += 256;
    }
    out[blockIdx.x * 256 + threadIdx.x] = acc.x + acc.y + acc.z + acc.w;
}
}  // namespace mdx

extern "C" int mdx_lds_read_rate(double *bytes_per_s, double *bytes_per_clock_per_cu) {
    using namespace mdx;
    if (!bytes_per_s) {
        mdx_set_error("mdx_lds_read_rate: null argument");
        return MDX_ERR_ARG;
    }
    int dev = 0;
    MDX_HIP(hipGetDevice(&dev));
    hipDeviceProp_t p;
    MDX_HIP(hipGetDeviceProperties(&p, dev));
    const int blocks = p.multiProcessorCount * 8;
    float *out = nullptr;
    MDX_HIP(hipMalloc(&out, (size_t)blocks * 256 * sizeof(float)));
    hipEvent_t e0 = nullptr, e1 = nullptr;
    hipError_t e = hipEventCreate(&e0);
    if (e == hipSuccess) e = hipEventCreate(&e1);
    if (e == hipSuccess) {
        hipLaunchKernelGGL(lds_read_rate_kernel, dim3(blocks), dim3(256), 0, nullptr, out);   // warm-up
        e = hipEventRecord(e0, nullptr);
    }
    for (int r = 0; r < 10 && e == hipSuccess; ++r) {
        hipLaunchKernelGGL(lds_read_rate_kernel, dim3(blocks), dim3(256), 0, nullptr, out);
        e = hipGetLastError();
    }
    if (e == hipSuccess) e = hipEventRecord(e1, nullptr);
    if (e == hipSuccess) e = hipEventSynchronize(e1);
    float ms = 0.f;
    if (e == hipSuccess) e = hipEventElapsedTime(&ms, e0, e1);
    if (e0) (void)hipEventDestroy(e0);
    if (e1) (void)hipEventDestroy(e1);
    (void)hipFree(out);
    MDX_HIP(e);
    const double bytes = 10.0 * blocks * 256.0 * LDSR_ITERS * 16.0;
    *bytes_per_s = bytes / (ms * 1e-3);
    if (bytes_per_clock_per_cu) *bytes_per_clock_per_cu = *bytes_per_s / (p.clockRate * 1e3) / p.multiProcessorCount;
    return MDX_OK;
}
