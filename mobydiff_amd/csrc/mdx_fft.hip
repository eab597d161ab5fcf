// mdx_fft.hip -- FFT(x,z) + Thomas(y) pressure solve for gfx950 (FP64).
//
// Replaces build_fft_rhs + the FFTW/cuFFT 2-D r2c/c2r + solve_tridiagonal_y + scaling +
// apply_fft_pressure_correction (pressure_solver.f90:77-173, pressure_fft.f90:102-148,
// pressure_backend_fftw.f90:51-93) with five kernels:
//   1. divergence of u* fused with the real x-FFT of each (j,k) row          rhs -> hat
//   2. z-FFT of each (kx, j) line, TX lines per workgroup                    hat -> hat
//   3. Thomas forward elimination / back substitution per (kx,kz) line       hat -> hat
//   4. inverse z-FFT                                                         hat -> hat
//   5. inverse real x-FFT with the 1/(nx nz) scaling per row                 hat -> phi
//   6. projection u = (u* - dtg grad phi)/(1 + dtg coef), p += phi
// (2. to 4. are one launch on small grids, column_solve_kernel).
// Transforms of 16 to 1024 points hold 16 points per thread in registers (fft_line: one LDS
// exchange for 32 to 256 points, two above); shorter ones are radix-4 Stockham (self-sorting) in
// LDS.  hat keeps the reference's half-spectrum layout plane_hat(nxh, nz, ny), kx fastest, each kx
// row padded to whole 128-byte lines (fft_stride).
#include <type_traits>

#include "mdx_internal.h"

namespace mdx {

// complex element types of the transforms: FP64 for the plain solve, FP32 for the defect solves
template <typename C> struct Cx;
template <> struct Cx<double2> {
    using R = double;
    static __device__ inline double2 mk(double a, double b) { return make_double2(a, b); }
};
template <> struct Cx<float2> {
    using R = float;
    static __device__ inline float2 mk(float a, float b) { return make_float2(a, b); }
};

// Stockham (self-sorting) transform of LINES lines of length n = 2^p held in LDS (a, b ping-pong),
// line q at q * ls: one radix-2 pass when p is odd, then radix-4 passes.  A pass combining groups
// of ns points reads r inputs n/r apart and writes them r-interleaved with twiddles
// w^(q kk n / (r ns)), kk = position in the group.  Returns the buffer holding the result.
// tw[m] = exp(-2 pi i m / n), m < n/2, staged in LDS by the caller (stage_twiddles); larger
// exponents use w^(m + n/2) = -w^m.
template <typename C>
__device__ inline C *stockham(C *a, C *b, int n, int lines, int ls, const C *tw, bool inverse, int tid,
                              int nthr) {
    using R = typename Cx<C>::R;
    const int half = n >> 1, quarter = n >> 2;
    int ns = 1;
    if (__builtin_ctz(n) & 1) {   // radix-2 pass
        for (int t = tid; t < half * lines; t += nthr) {
            const int line = t / half, jj = t - line * half;
            const C x0 = a[line * ls + jj], x1 = a[line * ls + jj + half];
            b[line * ls + 2 * jj] = Cx<C>::mk(x0.x + x1.x, x0.y + x1.y);
            b[line * ls + 2 * jj + 1] = Cx<C>::mk(x0.x - x1.x, x0.y - x1.y);
        }
        __syncthreads();
        C *t2 = a;
        a = b;
        b = t2;
        ns = 2;
    }
    auto twid = [&](int m) {   // w^m for 0 <= m < n
        C w = m < half ? tw[m] : Cx<C>::mk(-tw[m - half].x, -tw[m - half].y);
        if (inverse) w.y = -w.y;
        return w;
    };
    for (; ns < n; ns <<= 2) {
        const int stride = n / (4 * ns);
        for (int t = tid; t < quarter * lines; t += nthr) {
            const int line = t / quarter, jj = t - line * quarter;
            const int kk = jj & (ns - 1);
            const C *src = a + line * ls + jj;
            const C x0 = src[0], x1 = src[quarter], x2 = src[2 * quarter], x3 = src[3 * quarter];
            const C w1 = twid(kk * stride), w2 = twid(2 * kk * stride), w3 = twid(3 * kk * stride);
            const R y1r = x1.x * w1.x - x1.y * w1.y, y1i = x1.x * w1.y + x1.y * w1.x;
            const R y2r = x2.x * w2.x - x2.y * w2.y, y2i = x2.x * w2.y + x2.y * w2.x;
            const R y3r = x3.x * w3.x - x3.y * w3.y, y3i = x3.x * w3.y + x3.y * w3.x;
            // 4-point DFT; the forward transform multiplies by (-i)^(pq), the inverse by i^(pq)
            const R s02r = x0.x + y2r, s02i = x0.y + y2i, d02r = x0.x - y2r, d02i = x0.y - y2i;
            const R s13r = y1r + y3r, s13i = y1i + y3i, d13r = y1r - y3r, d13i = y1i - y3i;
            const R jr = inverse ? -d13i : d13i, ji = inverse ? d13r : -d13r;   // -i (or +i) * d13
            C *dst = b + line * ls + ((jj - kk) << 2) + kk;
            dst[0] = Cx<C>::mk(s02r + s13r, s02i + s13i);
            dst[ns] = Cx<C>::mk(d02r + jr, d02i + ji);
            dst[2 * ns] = Cx<C>::mk(s02r - s13r, s02i - s13i);
            dst[3 * ns] = Cx<C>::mk(d02r - jr, d02i - ji);
        }
        __syncthreads();
        C *t2 = a;
        a = b;
        b = t2;
    }
    return a;
}

static constexpr int FFT_THREADS = 256;

// the n/2 twiddles into LDS (read by every butterfly of every pass)
template <typename C>
__device__ inline void stage_twiddles(C *dst, const C *__restrict__ tw, int n) {
    for (int t = threadIdx.x; t < n / 2; t += FFT_THREADS) dst[t] = tw[t];
}

// ------------------------------------------------------------------------------- register transforms
// An N-point line (N = 16 M, M = 1 .. 64) on M threads with 16 points each.  In every pass thread t
// of the line holds the points t + M s (s = 0 .. 15), which are whole butterflies of every radix
// used: radix M first for N <= 256 (1, 2, 4, 8 or 16), radix N / 256 and 16 above, and 16 last.  A
// pass is one to two of stockham's radix-2 and radix-4 steps done in registers, with its twiddles and
// its order of operations, so a line's transform has the same bits (the FP32 passes of the defect
// correction leave the same phi).  Between passes the points go through LDS once, instead of once
// per radix-4 step with the whole line read from and written to LDS each time; a thread's first
// loads and last stores are its own points, so no staging either.  LDS addresses are padded by one
// element in 16, which keeps the radix-16 scatter (16 elements apart) and the gather (consecutive)
// free of bank conflicts.  At 256 x 192 x 256 in FP64 the LDS kernels took 129 us (x, with the
// right-hand side), 94 us (z, either way) and 89 us (x inverse); these take 105, 43 (37 inverse) and
// 36 us in a step: 3.9, 4.9 (5.7) and 5.8 TB/s by the counters, which see 1.02 to 1.04 times the fields
// and the spectrum read and written once.  In FP32: 49 us (x), 62 (z) and 62 (x inverse, adding to phi)
// before, 26, 32 (26 inverse) and 26 (to zero; 40 adding) now.
template <typename C, bool INV> __device__ inline C ctw(C a, C w) {   // a w (forward) or a conj(w)
    const typename Cx<C>::R wi = INV ? -w.y : w.y;
    return Cx<C>::mk(a.x * w.x - a.y * wi, a.x * wi + a.y * w.x);
}
// 4-point transform; the forward one multiplies by (-i)^(pq), the inverse one by i^(pq)
template <typename C, bool INV> __device__ inline void dft4(C &a, C &b, C &c, C &d) {
    const C s02 = Cx<C>::mk(a.x + c.x, a.y + c.y), d02 = Cx<C>::mk(a.x - c.x, a.y - c.y),
            s13 = Cx<C>::mk(b.x + d.x, b.y + d.y), d13 = Cx<C>::mk(b.x - d.x, b.y - d.y),
            j = INV ? Cx<C>::mk(-d13.y, d13.x) : Cx<C>::mk(d13.y, -d13.x);
    a = Cx<C>::mk(s02.x + s13.x, s02.y + s13.y);
    b = Cx<C>::mk(d02.x + j.x, d02.y + j.y);
    c = Cx<C>::mk(s02.x - s13.x, s02.y - s13.y);
    d = Cx<C>::mk(d02.x - j.x, d02.y - j.y);
}

template <int N, int TH> struct RFft {   // TH threads per workgroup
    static constexpr int M = N / 16;                       // threads per line
    static constexpr int LPW = TH / M;                     // lines per workgroup
    static constexpr int LS = N + M + 1;                   // LDS elements per line (padded)
    static constexpr int R0 = M <= 16 ? M : M / 16;        // first radix
    static constexpr int TW = 3 * N / 4;                   // twiddles w^m in LDS
    static constexpr bool TW0 = M == 1 || R0 >= 8;         // the first pass needs them
};
__device__ inline int rf_pad(int q) { return q + (q >> 4); }

// one pass of radix R on the thread's 16 points, as radix-2 and radix-4 steps in registers (the
// groups of ns points become groups of R ns), and the scatter to line (LDS) unless it is the last
// pass.  tw[m] = w^m, 0 <= m < 3 N / 4.
template <typename C, int N, int R, int NS, bool INV, bool LAST>
__device__ inline void rf_pass(C (&e)[16], int t, const C *tw, C *line) {
    constexpr int M = N / 16, U = 16 / R;
#pragma unroll
    for (int u = 0; u < U; ++u) {
        const int b = t + u * M, kk = b & (NS - 1);
        C v[R];
#pragma unroll
        for (int q = 0; q < R; ++q) v[q] = e[u + q * U];
        if constexpr (R == 2 || R == 8) {   // radix 2, groups of 1
            constexpr int H = R / 2;
#pragma unroll
            for (int q = 0; q < H; ++q) {
                const C x0 = v[q], x1 = v[q + H];
                v[q] = Cx<C>::mk(x0.x + x1.x, x0.y + x1.y);
                v[q + H] = Cx<C>::mk(x0.x - x1.x, x0.y - x1.y);
            }
        }
        if constexpr (R == 8) {   // radix 4, groups of 2: v[q + 4 p] -> v[p + 2 q']
#pragma unroll
            for (int q = 1; q < 4; ++q) v[q + 4] = ctw<C, INV>(v[q + 4], tw[q * (N / 8)]);
            dft4<C, INV>(v[0], v[1], v[2], v[3]);
            dft4<C, INV>(v[4], v[5], v[6], v[7]);
            const C w[8] = {v[0], v[4], v[1], v[5], v[2], v[6], v[3], v[7]};
#pragma unroll
            for (int q = 0; q < 8; ++q) v[q] = w[q];
        }
        if constexpr (R == 4 || R == 16) {   // radix 4, groups of NS
            constexpr int Q = R / 4;
#pragma unroll
            for (int a = 0; a < Q; ++a) {
                if (NS > 1) {
#pragma unroll
                    for (int q = 1; q < 4; ++q) v[a + q * Q] = ctw<C, INV>(v[a + q * Q], tw[q * kk * (N / (4 * NS))]);
                }
                dft4<C, INV>(v[a], v[a + Q], v[a + 2 * Q], v[a + 3 * Q]);
            }
        }
        if constexpr (R == 16) {   // radix 4, groups of 4 NS: v[a + 4 c] -> v[c + 4 d]
#pragma unroll
            for (int c = 0; c < 4; ++c) {
                if (NS > 1 || c > 0) {
#pragma unroll
                    for (int a = 1; a < 4; ++a)
                        v[a + 4 * c] = ctw<C, INV>(v[a + 4 * c], tw[a * (kk + NS * c) * (N / (16 * NS))]);
                }
                dft4<C, INV>(v[4 * c], v[4 * c + 1], v[4 * c + 2], v[4 * c + 3]);
            }
#pragma unroll
            for (int c = 0; c < 4; ++c)
#pragma unroll
                for (int d = 0; d < c; ++d) {
                    const C x = v[4 * c + d];
                    v[4 * c + d] = v[4 * d + c];
                    v[4 * d + c] = x;
                }
        }
        const int o = (b - kk) * R + kk;
#pragma unroll
        for (int q = 0; q < R; ++q) {
            if (LAST) e[u + q * U] = v[q];
            else line[rf_pad(o + q * NS)] = v[q];
        }
    }
}
template <typename C, int N>
__device__ inline void rf_gather(C (&e)[16], int t, const C *line) {
#pragma unroll
    for (int s = 0; s < 16; ++s) e[s] = line[rf_pad(t + N / 16 * s)];
}
// the transform of the line whose points t + M s thread t holds in e; line: the line's LDS, tw: the
// twiddles in LDS (staged by the caller before the barrier in here); threads with
// `on` false hold no line and only join the barriers
template <typename C, int N, bool INV>
__device__ inline void fft_line(C (&e)[16], int t, const C *tw, C *line, bool on = true) {
    using F = RFft<N, 64>;
    if constexpr (F::M == 1) {
        __syncthreads();
        if (on) rf_pass<C, N, 16, 1, INV, true>(e, t, tw, line);
    } else {
        if constexpr (F::TW0) __syncthreads();
        if (on) rf_pass<C, N, F::R0, 1, INV, false>(e, t, tw, line);
        __syncthreads();
        if (on) rf_gather<C, N>(e, t, line);
        if constexpr (F::M > 16) {
            __syncthreads();
            if (on) rf_pass<C, N, 16, F::R0, INV, false>(e, t, tw, line);
            __syncthreads();
            if (on) rf_gather<C, N>(e, t, line);
        }
        if (on) rf_pass<C, N, 16, F::M, INV, true>(e, t, tw, line);
    }
}
// the twiddles of fft_line into LDS (tw: w^m, m < N / 2; w^(m + N/2) = -w^m)
template <typename C, int N, int TH, int W = 1>
__device__ inline void rf_stage(C *dst, const C *__restrict__ tw) {
    for (int q = threadIdx.x; q < RFft<N, TH>::TW; q += TH * W) {
        const C w = tw[q < N / 2 ? q : q - N / 2];
        dst[q] = q < N / 2 ? w : Cx<C>::mk(-w.x, -w.y);
    }
}
// Two real rows are one complex line: row r in the real parts, row r + 1 (the next plane's) in the
// imaginary ones, so the x-transforms do half the work of real rows taken as complex lines.
// F(m) = A(m) + i B(m), A(m) = (F(m) + conj F(N - m)) / 2, B(m) = (F(m) - conj F(N - m)) / 2i.
// The line is in LDS in natural order; the rows' half spectra go to a and b.
template <typename C, int N>
__device__ inline void rf_split(const C *line, int m, C &a, C &b) {
    using T = typename Cx<C>::R;
    const C f = line[rf_pad(m)], g = line[rf_pad((N - m) & (N - 1))];
    a = Cx<C>::mk(T(0.5) * (f.x + g.x), T(0.5) * (f.y - g.y));
    b = Cx<C>::mk(T(0.5) * (f.y + g.y), T(0.5) * (g.x - f.x));
}
// rows 2 P and 2 P + 1 of the thread's line from its transform e to hat; every thread of the
// workgroup calls it (barriers)
// (TR: into the transposed spectrum of the column solves, kx slowest, `stride` values to a kx)
template <typename C, int N, int TH, int W = 1, bool TR = false>
__device__ inline void rf_store_rows(C (&e)[16], int t, C *lds, int l, int P0, int npairs, int stride, C *hat) {
    using F = RFft<N, TH>;
    C *line = lds + (size_t)l * F::LS;
    __syncthreads();
    if (W == 1 || l < F::LPW) {
#pragma unroll
        for (int s = 0; s < 16; ++s) line[rf_pad(t + F::M * s)] = e[s];
    }
    __syncthreads();
    constexpr int H = N / 2 + 1;
    for (int q = threadIdx.x; q < F::LPW * H; q += TH * W) {
        const int ll = TR ? q % F::LPW : q / H, m = TR ? q / F::LPW : q - ll * H, P = P0 + ll;
        if (P >= npairs) {
            if (TR) continue;
            break;
        }
        C a, b;
        rf_split<C, N>(lds + (size_t)ll * F::LS, m, a, b);
        if (TR) {
            hat[(size_t)stride * m + 2 * P] = a;
            hat[(size_t)stride * m + 2 * P + 1] = b;
        } else {
            hat[(size_t)stride * (2 * P) + m] = a;
            hat[(size_t)stride * (2 * P + 1) + m] = b;
        }
    }
}
// the thread's points of the inverse line of rows 2 P and 2 P + 1, from their half spectra (the real
// parts of the kx = 0 and kx = nx / 2 coefficients, Hermitian extension of the rest)
template <typename C, int N>
__device__ inline void rf_load_rows(C (&e)[16], int t, int P, int stride, const C *__restrict__ hat) {
    const C *A = hat + (size_t)stride * (2 * P), *B = A + stride;
#pragma unroll
    for (int s = 0; s < 16; ++s) {
        const int q = t + N / 16 * s;
        if (s < 8) {
            C a = A[q], b = B[q];
            if (s == 0 && q == 0) a.y = b.y = 0;
            e[s] = Cx<C>::mk(a.x - b.y, a.y + b.x);
        } else {
            C a = A[N - q], b = B[N - q];
            if (s == 8 && 2 * q == N) a.y = b.y = 0;
            e[s] = Cx<C>::mk(a.x + b.y, b.x - a.y);
        }
    }
}

// complex elements per kx row of the spectrum: nx / 2 + 1 rounded up to 128 bytes, so every row and
// every tile of 8 (FP64) or 16 (FP32) columns starts on a line (unpadded, the z-transform fetched
// 1.9 times its data)
template <typename C> static int fft_stride_t(int nx) {
    const int per = 128 / (int)sizeof(C);
    return (nx / 2 + 1 + per - 1) / per * per;
}
int fft_stride(int nx, bool fp32) { return fp32 ? fft_stride_t<float2>(nx) : fft_stride_t<double2>(nx); }

// a / d with r = 1 / d rounded: the quotient corrected once by its residual, which is a / d rounded
// (Markstein) for all but the ends of the exponent range: 3 operations where the division takes a
// dozen.  A plain a * r would put the rounding of r into every cell alike.
__device__ inline double div_by(double a, double d, double r) {
    const double q = a * r;
    return fma(fma(-q, d, a), r, q);
}

// 1. rhs(i,k,j) = div u* / dtg and the forward x-transform, two rows (planes k, k + 1) per line.
//    wrap: u*'s ghosts are taken as apply_bc fills them (periodic in x and z, v* = 0 on the walls)
//    instead of read; inside a step nothing else reads them, so their fill is left to its end.
//    The workgroups past `lines` form the flow-rate partial sums of u* instead, tile by tile as the
//    momentum kernel would (64 x 4 columns, mkz planes): on the grids where it is faster without.
struct FlowSum {
    int lines, mkz;
    double *part;
};
__device__ inline void flow_sum_tile(const GridK &g, const double *__restrict__ us, const FlowSum &f, double *s) {
    const Dims d = g.d;
    const int ntx = (d.nx + 63) / 64, nty = (d.ny + 3) / 4;
    const int wg = (int)blockIdx.x - f.lines, tx = wg % ntx, ty = wg / ntx % nty, tz = wg / ntx / nty;
    const int i = tx * 64 + threadIdx.x % 64 + 1, j = ty * 4 + threadIdx.x / 64 + 1, k0 = tz * f.mkz + 1;
    const int nk = k0 + f.mkz - 1 < d.nz ? f.mkz : d.nz - k0 + 1;
    double fa = 0.0, fb = 0.0;
    if (i <= d.nx && j <= d.ny) {
        const double hj = g.ihc ? 1.0 / g.ihc[j] : g.dy;
        const double *u = us + d.g(i, j, k0);
        const size_t sz = (size_t)d.sx * d.sy;
#pragma unroll 4
        for (int k = 0; k < nk; ++k) {
            fa += u[k * sz] * hj;
            fb += hj;
        }
    }
    flow_tile_sum<4>(fa, fb, threadIdx.x, s, f.part, (size_t)wg);
}
template <int N, int TH, int W, bool STRETCH, bool TR>
__global__ __launch_bounds__(TH * W) void rhs_xfft_reg_kernel(GridK g, const double *__restrict__ us,
                                                              const double *__restrict__ vs,
                                                              const double *__restrict__ ws, double dtg, int wrap,
                                                              FlowSum fsum, const double2 *__restrict__ tw, int stride,
                                                              double2 *__restrict__ hat) {
    using F = RFft<N, TH>;
    extern __shared__ __align__(16) unsigned char lds_raw[];
    if ((int)blockIdx.x >= fsum.lines) {
        static_assert(TH * W == 256, "the sums' 64 x 4 columns");
        flow_sum_tile(g, us, fsum, reinterpret_cast<double *>(lds_raw));
        return;
    }
    double2 *lds = reinterpret_cast<double2 *>(lds_raw), *twl = lds + F::LPW * F::LS;
    const Dims d = g.d;
    const int npairs = d.ny * d.nz / 2, t = threadIdx.x % F::M, l = threadIdx.x / F::M;
    const int P0 = blockIdx.x * F::LPW;
    const double it = 1.0 / dtg, ix = 1.0 / g.dx, iy = 1.0 / g.dy, iz = 1.0 / g.dz;
    const size_t sy = d.sx, sz = (size_t)d.sx * d.sy;
    // the lines in row order (a wave's loads are consecutive cells), each thread 16 / W cell pairs
#pragma unroll
    for (int s = 0; s < 16 / W; ++s) {
        const int q = threadIdx.x + TH * W * s, ll = q / N, i = q % N, P = P0 + ll;
        double2 r = make_double2(0.0, 0.0);
        if (P < npairs) {
            const int k = (2 * P) % d.nz + 1, j = (2 * P) / d.nz + 1;
            const size_t c0 = d.g(1 + i, j, k);
            const double *u = us + c0, *v = vs + c0, *w = ws + c0;
            const double w1 = w[sz], ih = STRETCH ? g.ihc[j] : 0.0;
            const int up = wrap && i == N - 1 ? 1 - N : 1;
            const double w2 = wrap && k + 1 == d.nz ? (w - (size_t)(k - 1) * sz)[0] : w[2 * sz];
            double va = v[0], vb = v[sz], vc = v[sy], vd = v[sz + sy];
            if (wrap && j == 1) va = vb = 0.0;
            if (wrap && j == d.ny) vc = vd = 0.0;
            auto rhs = [&](double du, double dv, double dw) {
                const double dy = STRETCH ? dv * ih : div_by(dv, g.dy, iy);
                return div_by(div_by(du, g.dx, ix) + dy + div_by(dw, g.dz, iz), dtg, it);
            };
            r.x = rhs(u[up] - u[0], vc - va, w1 - w[0]);
            r.y = rhs(u[sz + up] - u[sz], vd - vb, w2 - w1);
        }
        lds[(size_t)ll * F::LS + rf_pad(i)] = r;
    }
    rf_stage<double2, N, TH, W>(twl, tw);
    __syncthreads();
    const bool on = W == 1 || l < F::LPW;
    double2 *line = lds + (on ? l : 0) * F::LS;
    double2 e[16];
    if (on) rf_gather<double2, N>(e, t, line);
    if constexpr (!F::TW0) __syncthreads();   // the lines are read before they are written again
    fft_line<double2, N, false>(e, t, twl, line, on);
    rf_store_rows<double2, N, TH, W, TR>(e, t, lds, l, P0, npairs, stride, hat);
}

// 1. (FP32) forward x-transform of a real FP64 field in (nx, nz, ny) layout, a row per line (two rows
// in one line would mix their roundings, and a pass of the defect correction is only as accurate)
template <int N, int TH>
__global__ __launch_bounds__(TH) void xfft32_reg_kernel(Dims d, const double *__restrict__ in,
                                                        const float2 *__restrict__ tw, int stride,
                                                        float2 *__restrict__ hat) {
    using F = RFft<N, TH>;
    extern __shared__ __align__(16) unsigned char lds_raw[];
    float2 *lds = reinterpret_cast<float2 *>(lds_raw), *twl = lds + F::LPW * F::LS;
    const int nrows = d.ny * d.nz, t = threadIdx.x % F::M, r = blockIdx.x * F::LPW + threadIdx.x / F::M;
    rf_stage<float2, N, TH>(twl, tw);
    float2 e[16];
    const double *a = in + (size_t)N * (r < nrows ? r : 0) + t;
#pragma unroll
    for (int s = 0; s < 16; ++s) e[s] = make_float2((float)a[F::M * s], 0.f);
    fft_line<float2, N, false>(e, t, twl, lds + threadIdx.x / F::M * F::LS);
    if (r >= nrows) return;
    float2 *h = hat + (size_t)stride * r + t;
#pragma unroll
    for (int s = 0; s < 8; ++s) h[F::M * s] = e[s];
    if (t == 0) h[N / 2] = e[8];
}

// 5. inverse x-transform: phi (nx, nz, ny) = scaled rows, two per line
template <int N, int TH>
__global__ __launch_bounds__(TH) void ixfft_reg_kernel(Dims d, const double2 *__restrict__ hat,
                                                       const double2 *__restrict__ tw, int stride, double scale,
                                                       double *__restrict__ phi) {
    using F = RFft<N, TH>;
    extern __shared__ __align__(16) unsigned char lds_raw[];
    double2 *lds = reinterpret_cast<double2 *>(lds_raw), *twl = lds + F::LPW * F::LS;
    const int npairs = d.ny * d.nz / 2, t = threadIdx.x % F::M, l = threadIdx.x / F::M;
    const int P = blockIdx.x * F::LPW + l;
    rf_stage<double2, N, TH>(twl, tw);
    double2 e[16];
    rf_load_rows<double2, N>(e, t, P < npairs ? P : 0, stride, hat);
    fft_line<double2, N, true>(e, t, twl, lds + l * F::LS);
    if (P >= npairs) return;
    double *p = phi + (size_t)N * (2 * P) + t;
#pragma unroll
    for (int s = 0; s < 16; ++s) {
        p[F::M * s] = e[s].x * scale;
        p[N + F::M * s] = e[s].y * scale;
    }
}
// The same from the transposed spectrum (column_solve_kernel) for its small grids: 64 threads hold the
// lines, and 256 load them (neighbouring lanes on neighbouring lines, 32 bytes each) and store phi's
// rows, through LDS.  64^3: 4.0 us above, 5.2 here (6.6 with the 64 threads alone).
template <int N, int TH, int W>
__global__ __launch_bounds__(TH * W) void ixfft_columns_kernel(Dims d, const double2 *__restrict__ hat,
                                                               const double2 *__restrict__ tw, int stride,
                                                               double scale, double *__restrict__ phi) {
    using F = RFft<N, TH>;
    extern __shared__ __align__(16) unsigned char lds_raw[];
    double2 *lds = reinterpret_cast<double2 *>(lds_raw), *twl = lds + F::LPW * F::LS;
    const int npairs = d.ny * d.nz / 2, t = threadIdx.x % F::M, l = threadIdx.x / F::M, P0 = blockIdx.x * F::LPW;
    rf_stage<double2, N, TH, W>(twl, tw);
    for (int q = threadIdx.x; q < F::LPW * (N / 2 + 1); q += TH * W) {
        const int ll = q % F::LPW, m = q / F::LPW;
        double2 *line = lds + ll * F::LS;
        double2 a = make_double2(0.0, 0.0), b = a;
        if (P0 + ll < npairs) {
            const double2 *h = hat + (size_t)stride * m + 2 * (P0 + ll);
            a = h[0];
            b = h[1];
        }
        if (m == 0 || 2 * m == N) {   // real
            line[rf_pad(m)] = make_double2(a.x, b.x);
        } else {
            line[rf_pad(m)] = make_double2(a.x - b.y, a.y + b.x);
            line[rf_pad(N - m)] = make_double2(a.x + b.y, b.x - a.y);
        }
    }
    __syncthreads();
    const bool on = l < F::LPW;
    double2 *line = lds + (on ? l : 0) * F::LS;
    double2 e[16];
    if (on) rf_gather<double2, N>(e, t, line);
    if constexpr (!F::TW0) __syncthreads();   // the lines are read before they are written again
    fft_line<double2, N, true>(e, t, twl, line, on);
    __syncthreads();
    if (on) {
#pragma unroll
        for (int s = 0; s < 16; ++s) line[rf_pad(t + F::M * s)] = e[s];
    }
    __syncthreads();
    for (int q = threadIdx.x; q < 2 * F::LPW * N; q += TH * W) {
        const int r = q / N, x = q % N;
        if (2 * P0 + r >= 2 * npairs) break;
        const double2 v = lds[r / 2 * F::LS + rf_pad(x)];
        phi[(size_t)N * (2 * P0 + r) + x] = (r % 2 ? v.y : v.x) * scale;
    }
}
// 5. (FP32) inverse x-transform of each row, scaled, and the mean mode's solution added to the FP64 phi
// (FIRST: to zero)
template <int N, int TH, bool FIRST>
__global__ __launch_bounds__(TH) void ixfft32_add_reg_kernel(Dims d, const float2 *__restrict__ hat,
                                                             const float2 *__restrict__ tw, int stride, float scale,
                                                             const double *__restrict__ mean, double *__restrict__ phi) {
    using F = RFft<N, TH>;
    extern __shared__ __align__(16) unsigned char lds_raw[];
    float2 *lds = reinterpret_cast<float2 *>(lds_raw), *twl = lds + F::LPW * F::LS;
    const int nrows = d.ny * d.nz, t = threadIdx.x % F::M, r = blockIdx.x * F::LPW + threadIdx.x / F::M;
    const double mj = mean[r < nrows ? r / d.nz : 0];
    rf_stage<float2, N, TH>(twl, tw);
    const float2 *h = hat + (size_t)stride * (r < nrows ? r : 0);
    double *p = phi + (size_t)N * (r < nrows ? r : 0) + t;
    float2 e[16];
    double a[16];
#pragma unroll
    for (int s = 0; s < 16; ++s) {
        const int q = t + F::M * s;
        if (s < 8) {
            e[s] = h[q];
            if (s == 0 && q == 0) e[s].y = 0.f;
        } else {
            const float2 c = h[N - q];
            e[s] = make_float2(c.x, s == 8 && 2 * q == N ? 0.f : -c.y);
        }
        a[s] = FIRST ? mj : p[F::M * s] + mj;
    }
    fft_line<float2, N, true>(e, t, twl, lds + threadIdx.x / F::M * F::LS);
    if (r >= nrows) return;
#pragma unroll
    for (int s = 0; s < 16; ++s) p[F::M * s] = a[s] + (double)(e[s].x * scale);
}

// 2./4. z-transform in place.  The first `tiles` workgroups take CW consecutive kx columns (CW = 16,
// or the lines of a workgroup or half the x points if fewer) of LPW / CW planes; the others the nrem
// columns past the last whole tile (one, the highest kx, where CW divides nx / 2), a plane per line:
// in a tile of its own it would leave 15 of 16 threads idle.  The line index runs fastest over the
// threads, so a load or store of one kz moves the CW columns' consecutive values.
template <typename C, int N, int TH, bool INV>
__global__ __launch_bounds__(TH) void zfft_reg_kernel(int ny, int stride, int cw, int ntx, int tiles, int nrem,
                                                              const C *__restrict__ tw, C *__restrict__ hat) {
    using F = RFft<N, TH>;
    extern __shared__ __align__(16) unsigned char lds_raw[];
    C *lds = reinterpret_cast<C *>(lds_raw), *twl = lds + F::LPW * F::LS;
    const int l = threadIdx.x % F::LPW, t = threadIdx.x / F::LPW;
    int kx, j;
    bool live;
    if ((int)blockIdx.x < tiles) {
        const int pw = F::LPW / cw, tx = blockIdx.x % ntx, ty = blockIdx.x / ntx;
        kx = tx * cw + l % cw;
        j = ty * pw + l / cw;
        live = j < ny;
    } else {
        const int q = (blockIdx.x - tiles) * F::LPW + l;
        kx = ntx * cw + q / ny;
        j = q % ny;
        live = q < nrem * ny;
    }
    rf_stage<C, N, TH>(twl, tw);
    C *p = hat + (size_t)stride * N * (live ? j : 0) + (live ? kx : 0);
    C e[16];
#pragma unroll
    for (int s = 0; s < 16; ++s) e[s] = p[(size_t)stride * (t + F::M * s)];
    fft_line<C, N, INV>(e, t, twl, lds + l * F::LS);
    if (!live) return;
#pragma unroll
    for (int s = 0; s < 16; ++s) p[(size_t)stride * (t + F::M * s)] = e[s];
}

// 1. rhs(i,k,j) = [(u*(i+1)-u*(i))/dx + (v*(j+1)-v*(j))/dy + (w*(k+1)-w*(k))/dz]/dtg, then the
//    r2c x-transform; rows r = (k-1) + nz (j-1) are contiguous in hat.
template <bool STRETCH>
__global__ __launch_bounds__(FFT_THREADS) void rhs_xfft_kernel(GridK g, const double *__restrict__ us,
                                                              const double *__restrict__ vs,
                                                              const double *__restrict__ ws, double dtg, int wrap,
                                                              const double2 *__restrict__ tw, int lines,
                                                              int stride, double2 *hat) {
    extern __shared__ __align__(16) unsigned char lds_raw[];
    double2 *lds = reinterpret_cast<double2 *>(lds_raw);
    const Dims d = g.d;
    const int n = d.nx, nxh = n / 2 + 1;
    const int nrows = d.ny * d.nz;
    double2 *a = lds, *b = lds + (size_t)lines * n, *twl = b + (size_t)lines * n;
    stage_twiddles(twl, tw, n);
    for (int t = threadIdx.x; t < lines * n; t += FFT_THREADS) {
        const int line = t / n, i = t - line * n + 1;
        const int r = blockIdx.x * lines + line;
        double v = 0.0;
        if (r < nrows) {
            const int k = r % d.nz + 1, j = r / d.nz + 1;
            const int ip = wrap && i == n ? 1 : i + 1, kp = wrap && k == d.nz ? 1 : k + 1;
            const double vn = wrap && j == d.ny ? 0.0 : vs[d.g(i, j + 1, k)], vc = wrap && j == 1 ? 0.0 : vs[d.g(i, j, k)];
            const double dv = STRETCH ? (vn - vc) * g.ihc[j] : (vn - vc) / g.dy;
            v = ((us[d.g(ip, j, k)] - us[d.g(i, j, k)]) / g.dx + dv +
                 (ws[d.g(i, j, kp)] - ws[d.g(i, j, k)]) / g.dz) / dtg;
        }
        a[t] = make_double2(v, 0.0);
    }
    __syncthreads();
    double2 *res = stockham(a, b, n, lines, n, twl, false, threadIdx.x, FFT_THREADS);
    for (int t = threadIdx.x; t < lines * nxh; t += FFT_THREADS) {
        const int line = t / nxh, m = t - line * nxh;
        const int r = blockIdx.x * lines + line;
        if (r < nrows) hat[(size_t)stride * r + m] = res[line * n + m];
    }
}

// 2./4. z-transform of TX consecutive kx columns of one j plane.
template <typename C>
__global__ __launch_bounds__(FFT_THREADS) void zfft_kernel(Dims d, C *hat, const C *__restrict__ tw, int tx,
                                                           int inverse, int stride) {
    extern __shared__ __align__(16) unsigned char lds_raw[];
    C *lds = reinterpret_cast<C *>(lds_raw);
    const int nz = d.nz, nxh = d.nx / 2 + 1;
    const int tiles = (nxh + tx - 1) / tx;
    const int j = blockIdx.x / tiles, kx0 = (blockIdx.x % tiles) * tx;
    // columns nz + 1 apart in LDS: the transposing loads and stores (tx columns of one kz row)
    // fall in different banks
    const int ls = nz + 1;
    C *a = lds, *b = lds + (size_t)tx * ls, *twl = b + (size_t)tx * ls;
    C *plane = hat + (size_t)stride * nz * j;
    stage_twiddles(twl, tw, nz);
    for (int t = threadIdx.x; t < tx * nz; t += FFT_THREADS) {
        const int c = t % tx, kz = t / tx;
        const int kx = kx0 + c;
        a[c * ls + kz] = kx < nxh ? plane[(size_t)kx + (size_t)stride * kz] : Cx<C>::mk(0, 0);
    }
    __syncthreads();
    C *res = stockham(a, b, nz, tx, ls, twl, inverse != 0, threadIdx.x, FFT_THREADS);
    for (int t = threadIdx.x; t < tx * nz; t += FFT_THREADS) {
        const int c = t % tx, kz = t / tx;
        const int kx = kx0 + c;
        if (kx < nxh) plane[(size_t)kx + (size_t)stride * kz] = res[c * ls + kz];
    }
}

// 3. pressure_fft.f90:102-148 with precomputed cp/den_inv (pressure_fft.f90:20-100); one thread
//    per (kx,kz) line, consecutive kx in consecutive lanes (coalesced), in place.  The recurrences
//    run in blocks of TB planes whose loads are all issued before the block's stores (a load after
//    a store through the same pointer cannot be hoisted above it), so TB loads are in flight at a
//    time instead of one; the arithmetic and its order are those of the plane-by-plane loops.
static constexpr int TB = 8;

__global__ __launch_bounds__(64) void tridiag_kernel(Dims d, int stride, double2 *hat, const double *__restrict__ cp,
                                                     const double *__restrict__ den_inv,
                                                     const double *__restrict__ arow) {
    const int nxh = d.nx / 2 + 1, ny = d.ny, nz = d.nz;
    const int t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= nxh * nz) return;
    const int kx = t % nxh, kz = t / nxh;
    const size_t hs = (size_t)stride * nz;                  // stride between j planes in hat
    const size_t cs = (size_t)nxh;                          // stride between j in cp/den_inv
    const size_t h0 = (size_t)kx + (size_t)stride * kz;
    const size_t c0 = (size_t)kx + (size_t)nxh * (size_t)ny * kz;
    double2 dp;
    if (kx == 0 && kz == 0) {
        dp = make_double2(0.0, 0.0);
    } else {
        const double2 r = hat[h0];
        const double di = den_inv[c0];
        dp = make_double2(r.x * di, r.y * di);
    }
    hat[h0] = dp;
    // forward elimination, planes 2..ny
    for (int jb = 2; jb <= ny; jb += TB) {
        double2 rr[TB];
        double aa[TB], dd[TB];
#pragma unroll
        for (int q = 0; q < TB; ++q) {
            const int jj = jb + q;
            if (jj <= ny) {
                rr[q] = hat[h0 + hs * (jj - 1)];
                aa[q] = arow[jj - 1];
                dd[q] = den_inv[c0 + cs * (jj - 1)];
            }
        }
#pragma unroll
        for (int q = 0; q < TB; ++q) {
            const int jj = jb + q;
            if (jj <= ny) {
                dp = make_double2((rr[q].x - aa[q] * dp.x) * dd[q], (rr[q].y - aa[q] * dp.y) * dd[q]);
                hat[h0 + hs * (jj - 1)] = dp;
            }
        }
    }
    // back substitution, planes ny-1..1 (hat(ny) = dp(ny))
    double2 nxt = dp;
    for (int jb = ny - 1; jb >= 1; jb -= TB) {
        double2 qq[TB];
        double cc[TB];
#pragma unroll
        for (int q = 0; q < TB; ++q) {
            const int jj = jb - q;
            if (jj >= 1) {
                qq[q] = hat[h0 + hs * (jj - 1)];
                cc[q] = cp[c0 + cs * (jj - 1)];
            }
        }
#pragma unroll
        for (int q = 0; q < TB; ++q) {
            const int jj = jb - q;
            if (jj >= 1) {
                nxt = make_double2(qq[q].x - cc[q] * nxt.x, qq[q].y - cc[q] * nxt.y);
                hat[h0 + hs * (jj - 1)] = nxt;
            }
        }
    }
}

// 3'. The same tridiagonal solves with one wavefront per (kx,kz) line, every value of the line in
//     registers: the spectrum is read once and written once (16 B per cell), against twice each
//     plus the two FP64 tables for the thread-per-line recurrence.  Lane l holds rows
//     j = l, l + 64, ..., l + 64 (M-1) (0-based) with a_j (sub-diagonal), b_j = bd_j - k
//     (k = lamx[kx] + lamz[kz], the modified wavenumbers of pressure_fft.f90:20-100), c_j and the
//     complex right-hand side; rows past ny, and neighbours past the ends, are identity rows.
//       * Parallel cyclic reduction, six steps (coupling distance 1, 2, ..., 32, the neighbours'
//         coefficients by cross-lane shuffles), leaves every row coupled only to the rows 64 away:
//         each lane then holds an independent M-row system, solved by Thomas.
//       * One step of iterative refinement in the same precision: the residual d - A x with the
//         original rows (neighbours x_(j-1), x_(j+1) by shuffles) goes through the same reduction,
//         whose multipliers and Thomas factors were kept in registers, and the correction is added.
//     Reduction alone left residuals 100-1000x larger than the serial recurrence's on the
//     tanh-stretched grid (weakly dominant low-wavenumber rows); with the refinement step they are
//     within 2x of it.  Every lane works through the whole solve (no serial chain across lanes:
//     a line's serial recurrence in one wave would cost 64 lanes' worth of FP64 issue per step).
//     The mean mode (kx = kz = 0) pins row 1 to zero, as the reference does (dp(1) = 0), by making
//     it an identity row.  A workgroup takes 16 consecutive lines and stages them through LDS: for
//     a fixed row the 16 lines' values are contiguous in the spectrum (256 B in FP64), so the loads
//     and stores move whole cache lines, and each wave then reads its line's rows from LDS
//     (rows of a line contiguous, padded by one value so the transposed copy is conflict-free).
template <typename T>
__device__ inline T shfl_any(T v, int src) {
    return __shfl(v, src, 64);
}
template <>
__device__ inline double2 shfl_any<double2>(double2 v, int src) {
    return make_double2(__shfl(v.x, src, 64), __shfl(v.y, src, 64));
}
template <>
__device__ inline float2 shfl_any<float2>(float2 v, int src) {
    return make_float2(__shfl(v.x, src, 64), __shfl(v.y, src, 64));
}

// a workgroup of TW_WAVES waves solves TW_LINES consecutive lines, staged through LDS
static constexpr int TW_WAVES = 4, TW_LINES = 16, TW_STEPS = 6;

// the value of row i - delta (lo) or i + delta (hi) for row set q, from the shuffled copies of all
// row sets (rows across the lane wrap belong to set q - 1 / q + 1; beyond the ends: `edge`)
template <int M, typename V>
__device__ inline V pick_lo(const V (&sh)[M], int q, bool wrap, V edge) {
    return !wrap ? sh[q] : (q > 0 ? sh[q > 0 ? q - 1 : 0] : edge);
}
template <int M, typename V>
__device__ inline V pick_hi(const V (&sh)[M], int q, bool wrap, V edge) {
    return !wrap ? sh[q] : (q + 1 < M ? sh[q + 1 < M ? q + 1 : q] : edge);
}

// C: double2 (the FP64 solve; the mean mode pins row 1) or float2 (the FP32 defect solves; the
// mean mode is solved apart in FP64, so its line is zeroed, MEAN_ZERO)
template <typename C, int M, bool MEAN_ZERO>
__global__ __launch_bounds__(64 * TW_WAVES) void tridiag_wave_kernel(int nlines, int stride, int nxh, int ny, size_t plane, C *hat,
                                                                    const typename Cx<C>::R *__restrict__ lamx,
                                                                    const typename Cx<C>::R *__restrict__ lamz,
                                                                    const typename Cx<C>::R *__restrict__ arow,
                                                                    const typename Cx<C>::R *__restrict__ bdrow,
                                                                    const typename Cx<C>::R *__restrict__ crow) {
    using R = typename Cx<C>::R;
    extern __shared__ __align__(16) unsigned char lds_raw[];
    C *tile = reinterpret_cast<C *>(lds_raw);   // [TW_LINES][ny + 1]: line-major, rows contiguous
    const int ldt = ny + 1;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int t0 = blockIdx.x * TW_LINES;
    const C zero2 = Cx<C>::mk(R(0), R(0));
    // ---- the TW_LINES lines of this workgroup into LDS: for each row, the lines' values are
    // consecutive in the spectrum (TW_LINES * sizeof(C) contiguous bytes per row)
    {
        const int tt = threadIdx.x % TW_LINES, jj = threadIdx.x / TW_LINES;
        const int t = t0 + tt;
        for (int j = jj; j < ny; j += 64 * TW_WAVES / TW_LINES)
            tile[tt * ldt + j] = t < nlines ? hat[(size_t)t + plane * j] : zero2;
    }
    __syncthreads();
    // ---- every wave solves its lines from LDS (lane l: rows l, l + 64, ...)
    for (int l = wave; l < TW_LINES; l += TW_WAVES) {
        const int t = t0 + l;
        if (t >= nlines) break;   // whole waves
        if (t % stride >= nxh) continue;   // the padding of a kx row
        C *line = tile + (size_t)l * ldt;
        if (MEAN_ZERO && t == 0) {
            for (int j = lane; j < ny; j += 64) line[j] = zero2;
            continue;
        }
        const int kx = t % stride, kz = t / stride;
        const R k = lamx[kx] + lamz[kz];
        // the original rows (kept for the residual) and the right-hand side
        R a0[M], b0[M], c0[M];
        C d0[M];
#pragma unroll
        for (int q = 0; q < M; ++q) {
            const int j = lane + 64 * q;
            if (j < ny && !(t == 0 && j == 0)) {
                a0[q] = arow[j];
                c0[q] = crow[j];
                b0[q] = bdrow[j] - k;
                d0[q] = line[j];
            } else {
                a0[q] = R(0);
                c0[q] = R(0);
                b0[q] = R(1);
                d0[q] = zero2;
            }
        }
        // reduction of the rows, keeping the multipliers of every step
        R a[M], b[M], c[M], k1s[TW_STEPS][M], k2s[TW_STEPS][M];
#pragma unroll
        for (int q = 0; q < M; ++q) {
            a[q] = a0[q];
            b[q] = b0[q];
            c[q] = c0[q];
        }
#pragma unroll
        for (int s = 0; s < TW_STEPS; ++s) {
            const int delta = 1 << s;
            const int lo = (lane - delta) & 63, hi = (lane + delta) & 63;
            const bool wlo = lane < delta, whi = lane + delta >= 64;
            R rb[M], la[M], lc[M], lr[M], ha[M], hc[M], hr[M];
#pragma unroll
            for (int q = 0; q < M; ++q) rb[q] = R(1) / b[q];
#pragma unroll
            for (int q = 0; q < M; ++q) {
                la[q] = shfl_any(a[q], lo);
                lc[q] = shfl_any(c[q], lo);
                lr[q] = shfl_any(rb[q], lo);
                ha[q] = shfl_any(a[q], hi);
                hc[q] = shfl_any(c[q], hi);
                hr[q] = shfl_any(rb[q], hi);
            }
#pragma unroll
            for (int q = 0; q < M; ++q) {
                const R na = pick_lo<M>(la, q, wlo, R(0)), nc = pick_lo<M>(lc, q, wlo, R(0)),
                        nr = pick_lo<M>(lr, q, wlo, R(1));
                const R pa = pick_hi<M>(ha, q, whi, R(0)), pc = pick_hi<M>(hc, q, whi, R(0)),
                        pr = pick_hi<M>(hr, q, whi, R(1));
                const R k1 = a[q] * nr, k2 = c[q] * pr;
                k1s[s][q] = k1;
                k2s[s][q] = k2;
                a[q] = -na * k1;
                b[q] = b[q] - nc * k1 - pa * k2;
                c[q] = -pc * k2;
            }
        }
        // Thomas factors of the lane's M-row system (row q couples to rows q - 1 and q + 1 only)
        R cp[M], rden[M];
#pragma unroll
        for (int q = 0; q < M; ++q) {
            const R den = q > 0 ? b[q] - a[q] * cp[q - 1] : b[q];
            rden[q] = R(1) / den;
            cp[q] = c[q] * rden[q];
        }
        // a right-hand side through the kept reduction and Thomas factors
        auto solve = [&](C (&d)[M]) {
#pragma unroll
            for (int s = 0; s < TW_STEPS; ++s) {
                const int delta = 1 << s;
                const int lo = (lane - delta) & 63, hi = (lane + delta) & 63;
                const bool wlo = lane < delta, whi = lane + delta >= 64;
                C ld[M], hd[M];
#pragma unroll
                for (int q = 0; q < M; ++q) {
                    ld[q] = shfl_any(d[q], lo);
                    hd[q] = shfl_any(d[q], hi);
                }
#pragma unroll
                for (int q = 0; q < M; ++q) {
                    const C nd = pick_lo<M>(ld, q, wlo, zero2), pd = pick_hi<M>(hd, q, whi, zero2);
                    d[q] = Cx<C>::mk(d[q].x - nd.x * k1s[s][q] - pd.x * k2s[s][q],
                                     d[q].y - nd.y * k1s[s][q] - pd.y * k2s[s][q]);
                }
            }
#pragma unroll
            for (int q = 0; q < M; ++q) {
                if (q > 0) d[q] = Cx<C>::mk(d[q].x - a[q] * d[q - 1].x, d[q].y - a[q] * d[q - 1].y);
                d[q] = Cx<C>::mk(d[q].x * rden[q], d[q].y * rden[q]);
            }
#pragma unroll
            for (int q = M - 2; q >= 0; --q)
                d[q] = Cx<C>::mk(d[q].x - cp[q] * d[q + 1].x, d[q].y - cp[q] * d[q + 1].y);
        };
        C x[M];
#pragma unroll
        for (int q = 0; q < M; ++q) x[q] = d0[q];
        solve(x);
        // refinement: r = d - A x with the original rows, solved the same way, added
        {
            const int lo = (lane - 1) & 63, hi = (lane + 1) & 63;
            const bool wlo = lane < 1, whi = lane + 1 >= 64;
            C lx[M], hx[M], r[M];
#pragma unroll
            for (int q = 0; q < M; ++q) {
                lx[q] = shfl_any(x[q], lo);
                hx[q] = shfl_any(x[q], hi);
            }
#pragma unroll
            for (int q = 0; q < M; ++q) {
                const C xm = pick_lo<M>(lx, q, wlo, zero2), xp = pick_hi<M>(hx, q, whi, zero2);
                r[q] = Cx<C>::mk(d0[q].x - (a0[q] * xm.x + b0[q] * x[q].x + c0[q] * xp.x),
                                 d0[q].y - (a0[q] * xm.y + b0[q] * x[q].y + c0[q] * xp.y));
            }
            solve(r);
#pragma unroll
            for (int q = 0; q < M; ++q) x[q] = Cx<C>::mk(x[q].x + r[q].x, x[q].y + r[q].y);
        }
#pragma unroll
        for (int q = 0; q < M; ++q) {
            const int j = lane + 64 * q;
            if (j < ny) line[j] = x[q];
        }
    }
    __syncthreads();
    // ---- back to the spectrum, as loaded
    {
        const int tt = threadIdx.x % TW_LINES, jj = threadIdx.x / TW_LINES;
        const int t = t0 + tt;
        if (t < nlines)
            for (int j = jj; j < ny; j += 64 * TW_WAVES / TW_LINES) hat[(size_t)t + plane * j] = tile[tt * ldt + j];
    }
}

// The partitioned Thomas recurrence: a line's rows are cut into segments of M consecutive rows, a
// thread each, whose rows stay in its registers (rows past ny are identity rows).  A segment's
// interior rows (1 .. M-2) are eliminated by the Thomas recurrence with three right-hand sides: the
// data, and the couplings to the segment's first row F (through a_1) and last row E (through
// c_(M-2)), so every interior value is p + q F + s E.  Substituted into the first and last rows,
// that leaves a tridiagonal system in F_0, E_0, F_1, E_1, ... of two rows per segment.
// KEEP: what the elimination of another right-hand side needs stays too.
template <typename C, int M, bool KEEP> struct TriSegment {
    using R = typename Cx<C>::R;
    static_assert(M >= 3, "a segment has interior rows");
    R cp[M], qq[M], ss[M], rd[KEEP ? M : 1];
    R a0, b0, c0, aL, bL, cL;
    // coef(r, a, b, c): row r of the segment; p: the data
    template <typename F> __device__ inline void eliminate(const F &coef, C (&p)[M]) {
        coef(0, a0, b0, c0);
        coef(M - 1, aL, bL, cL);
#pragma unroll
        for (int r = 1; r <= M - 2; ++r) {
            R a, b, c;
            coef(r, a, b, c);
            const R rden = R(1) / (r > 1 ? b - a * cp[r - 1] : b);
            if (KEEP) rd[KEEP ? r : 0] = rden;
            cp[r] = r < M - 2 ? c * rden : R(0);
            p[r] = r > 1 ? Cx<C>::mk((p[r].x - a * p[r - 1].x) * rden, (p[r].y - a * p[r - 1].y) * rden)
                         : Cx<C>::mk(p[r].x * rden, p[r].y * rden);
            qq[r] = (r == 1 ? -a : -a * qq[r - 1]) * rden;
            ss[r] = ((r == M - 2 ? -c : R(0)) - (r > 1 ? a * ss[r - 1] : R(0))) * rden;
        }
#pragma unroll
        for (int r = M - 3; r >= 1; --r) {
            p[r] = Cx<C>::mk(p[r].x - cp[r] * p[r + 1].x, p[r].y - cp[r] * p[r + 1].y);
            qq[r] -= cp[r] * qq[r + 1];
            ss[r] -= cp[r] * ss[r + 1];
        }
    }
    // the same elimination of another right-hand side
    template <typename F> __device__ inline void again(const F &coef, C (&p)[M]) const {
#pragma unroll
        for (int r = 1; r <= M - 2; ++r) {
            R a, b, c;
            coef(r, a, b, c);
            const R rden = rd[KEEP ? r : 0];
            p[r] = r > 1 ? Cx<C>::mk((p[r].x - a * p[r - 1].x) * rden, (p[r].y - a * p[r - 1].y) * rden)
                         : Cx<C>::mk(p[r].x * rden, p[r].y * rden);
        }
#pragma unroll
        for (int r = M - 3; r >= 1; --r) p[r] = Cx<C>::mk(p[r].x - cp[r] * p[r + 1].x, p[r].y - cp[r] * p[r + 1].y);
    }
    // the two rows of the reduced system (a, b, c) and their data
    __device__ inline void first(R &a, R &b, R &c) const {
        a = a0;
        b = b0 + c0 * qq[1];
        c = c0 * ss[1];
    }
    __device__ inline void last(R &a, R &b, R &c) const {
        a = aL * qq[M - 2];
        b = bL + aL * ss[M - 2];
        c = cL;
    }
    __device__ inline C first(const C (&p)[M]) const { return Cx<C>::mk(p[0].x - c0 * p[1].x, p[0].y - c0 * p[1].y); }
    __device__ inline C last(const C (&p)[M]) const {
        return Cx<C>::mk(p[M - 1].x - aL * p[M - 2].x, p[M - 1].y - aL * p[M - 2].y);
    }
    // row r of the solution
    __device__ inline C row(const C (&p)[M], int r, C F, C E) const {
        return r == 0 ? F : r == M - 1 ? E
               : Cx<C>::mk(p[r].x + qq[r] * F.x + ss[r] * E.x, p[r].y + qq[r] * F.y + ss[r] * E.y);
    }
};
// the residual of a segment's rows into r: data(q) less the rows (coef) applied to x, whose neighbours
// past the segment's ends are xm and xp
template <typename C, int M, typename F, typename G>
__device__ inline void tri_residual(const F &coef, const G &data, const C (&x)[M], C xm, C xp, C (&r)[M]) {
#pragma unroll
    for (int q = 0; q < M; ++q) {
        typename Cx<C>::R a, b, c;
        coef(q, a, b, c);
        C l = xm, u = xp;
        if (q > 0) l = x[q > 0 ? q - 1 : 0];
        if (q < M - 1) u = x[q < M - 1 ? q + 1 : q];
        const C d = data(q);
        r[q] = Cx<C>::mk(d.x - (a * l.x + b * x[q].x + c * u.x), d.y - (a * l.y + b * x[q].y + c * u.y));
    }
}

// 3''. The same solves as a partitioned Thomas recurrence (TriSegment).  A workgroup of 256 threads
//     takes 16 consecutive lines and gives each line 16 segments; a row of the 16 lines is 256
//     contiguous bytes, so loads and stores move whole cache lines without staging.  The reduced
//     system (32 unknowns per line) is solved by one thread per line, TP_CH rows' operands read
//     ahead of the chain; the segments then form their interior values.  The serial chain per
//     line is 2 (M - 2) + 64 steps instead of 2 ny, the work about twice the plain recurrence's, and
//     the spectrum moves once each way.  The mean mode pins row 1 as the wave solve does; MEAN_ZERO
//     zeroes that line.  256 x 192 x 256 in FP64: 92 us with the lines staged in LDS (70 KB, two
//     workgroups per CU) and the reduced system's operands read step by step; 57 now (FP32: 50 and
//     31), 64^3 13.1 and 7.8.
//     REFINE: one step of iterative refinement, as in the wave solve, which the FP64 lines of fewer
//     than 64 rows took before.  Over ny = 16 .. 63, uniform spacing in a 4 pi x 2 x 2 pi box, the
//     slowest modes' rms error is 3.7e-14 without the step, 1.2e-14 with it and 1.2e-14 in the wave
//     solve; from 64 rows on the recurrence alone is as accurate as it was.
static constexpr int TP_LINES = 16, TP_SEGS = 16, TP_CH = 8;
template <typename C, int M, bool MEAN_ZERO, bool REFINE>
__global__ __launch_bounds__(TP_LINES * TP_SEGS, M <= 12 ? 3 : 2) void tridiag_part_kernel(int nlines, int stride, int nxh, int ny,
                                                                        size_t plane, C *hat,
                                                                        const typename Cx<C>::R *__restrict__ lamx,
                                                                        const typename Cx<C>::R *__restrict__ lamz,
                                                                        const typename Cx<C>::R *__restrict__ arow,
                                                                        const typename Cx<C>::R *__restrict__ bdrow,
                                                                        const typename Cx<C>::R *__restrict__ crow) {
    using R = typename Cx<C>::R;
    constexpr int NR = 2 * TP_SEGS;   // reduced rows per line
    __shared__ R ra[NR][TP_LINES], rb[NR][TP_LINES], rc[NR][TP_LINES];
    __shared__ C rd[NR][TP_LINES];
    const int tt = threadIdx.x % TP_LINES, sg = threadIdx.x / TP_LINES;
    const int t = blockIdx.x * TP_LINES + tt;
    const bool live = t < nlines && t % stride < nxh;   // a line, not the padding of a kx row
    const bool ident_line = !live || (MEAN_ZERO && t == 0);
    const int j0 = sg * M;
    const C zero = Cx<C>::mk(R(0), R(0));
    // row r of the segment: (a, b, c) and the data
    auto solved = [&](int r) { return !ident_line && j0 + r < ny && !(t == 0 && j0 + r == 0); };
    C p[M], d[REFINE ? M : 1];
    C *h = hat + (size_t)(t < nlines ? t : 0) + plane * j0;
#pragma unroll
    for (int r = 0; r < M; ++r) {
        p[r] = zero;
        if (solved(r)) p[r] = h[plane * r];
        if (REFINE) d[REFINE ? r : 0] = p[r];
    }
    const R k = live ? lamx[t % stride] + lamz[t / stride] : R(0);
    auto coef = [&](int r, R &a, R &b, R &c) {
        const int j = j0 + r;
        if (solved(r)) {
            a = arow[j];
            b = bdrow[j] - k;
            c = crow[j];
        } else {
            a = R(0);
            b = R(1);
            c = R(0);
        }
    };
    TriSegment<C, M, REFINE> seg;
    seg.eliminate(coef, p);
    seg.first(ra[2 * sg][tt], rb[2 * sg][tt], rc[2 * sg][tt]);
    rd[2 * sg][tt] = seg.first(p);
    seg.last(ra[2 * sg + 1][tt], rb[2 * sg + 1][tt], rc[2 * sg + 1][tt]);
    rd[2 * sg + 1][tt] = seg.last(p);
    __syncthreads();
    // the reduced system of each line, one thread per line (Thomas; solution into rd); again: with the
    // factors of the first time (rb: reciprocal denominators)
    auto reduced = [&](auto again_) {
        constexpr bool again = decltype(again_)::value;
        R cprev = R(0);
        C dprev = zero;
        for (int r0 = 0; r0 < NR; r0 += TP_CH) {
            R a[TP_CH], b[TP_CH], c[TP_CH];
            C e[TP_CH];
#pragma unroll
            for (int u = 0; u < TP_CH; ++u) {
                a[u] = ra[r0 + u][tt];
                b[u] = rb[r0 + u][tt];
                if (!again) c[u] = rc[r0 + u][tt];
                e[u] = rd[r0 + u][tt];
            }
#pragma unroll
            for (int u = 0; u < TP_CH; ++u) {
                R rden = b[u];
                if (!again) {
                    const R den = b[u] - a[u] * cprev;
                    rden = R(1) / den;
                    cprev = c[u] * rden;
                    rc[r0 + u][tt] = cprev;
                    if (REFINE) rb[r0 + u][tt] = rden;
                }
                dprev = Cx<C>::mk((e[u].x - a[u] * dprev.x) * rden, (e[u].y - a[u] * dprev.y) * rden);
                rd[r0 + u][tt] = dprev;
            }
        }
        C xn = dprev;
        for (int r0 = NR - TP_CH; r0 >= 0; r0 -= TP_CH) {
            R c[TP_CH];
            C e[TP_CH];
#pragma unroll
            for (int u = 0; u < TP_CH; ++u) {
                c[u] = rc[r0 + u][tt];
                e[u] = rd[r0 + u][tt];
            }
#pragma unroll
            for (int u = TP_CH - 1; u >= 0; --u) {
                if (r0 + u == NR - 1) continue;
                xn = Cx<C>::mk(e[u].x - c[u] * xn.x, e[u].y - c[u] * xn.y);
                rd[r0 + u][tt] = xn;
            }
        }
    };
    if (sg == 0) reduced(std::false_type{});
    __syncthreads();
    // ---- every row of the segment from F and E
    const C F = rd[2 * sg][tt], E = rd[2 * sg + 1][tt];
    if constexpr (REFINE) {
        C x[M];
#pragma unroll
        for (int r = 0; r < M; ++r) x[r] = seg.row(p, r, F, E);
        C xm = zero, xp = zero;
        if (sg > 0) xm = rd[2 * sg - 1][tt];
        if (sg < TP_SEGS - 1) xp = rd[2 * sg + 2][tt];
        tri_residual<C, M>(coef, [&](int r) { return d[REFINE ? r : 0]; }, x, xm, xp, p);
        seg.again(coef, p);
        __syncthreads();   // the neighbours' ends have been read
        rd[2 * sg][tt] = seg.first(p);
        rd[2 * sg + 1][tt] = seg.last(p);
        __syncthreads();
        if (sg == 0) reduced(std::true_type{});
        __syncthreads();
        const C dF = rd[2 * sg][tt], dE = rd[2 * sg + 1][tt];
        if (!live) return;
#pragma unroll
        for (int r = 0; r < M; ++r) {
            const C e = seg.row(p, r, dF, dE);
            if (j0 + r < ny) h[plane * r] = Cx<C>::mk(x[r].x + e.x, x[r].y + e.y);
        }
    } else {
        if (!live) return;
#pragma unroll
        for (int r = 0; r < M; ++r)
            if (j0 + r < ny) h[plane * r] = seg.row(p, r, F, E);
    }
}

// 2. - 4. in one launch, where a kx column of the spectrum (all planes and kz, transposed: kx slowest)
//     fits a CU's LDS and the launches are short: z-transforms of the column's lines, its tridiagonal
//     solves as tridiag_part_kernel does them (CS_SEGS segments of M rows; the reduced rows' data in the
//     tile, at the rows they stand for), and the transforms back, one workgroup per kx.  Bound by
//     latency: 64^3 18.2 us in three launches, 13.0 in one; 128 x 97 x 64 26.2 and 17.1.
//     REFINE as there (rms error over ny = 16 .. 63 2.3e-14 without the step, 1.2e-14 with it; from 64
//     rows on, without, 6.4e-14 against 8.0e-14 with 16 segments): 64 x 48 x 64 11.0 us without, 15.2.
static constexpr int CS_T = 512, CS_SEGS = 8;
template <int N, int M> constexpr size_t column_lds() {
    return (size_t)CS_SEGS * M * RFft<N, CS_T>::LS * 16 + RFft<N, CS_T>::TW * 16 + 3 * 2 * CS_SEGS * (N < 64 ? N : 64) * 8;
}
template <int N, int M, bool REFINE>
__global__ __launch_bounds__(CS_T) void column_solve_kernel(int ny, const double2 *__restrict__ tw,
                                                            const double *__restrict__ lamx,
                                                            const double *__restrict__ lamz,
                                                            const double *__restrict__ arow,
                                                            const double *__restrict__ bdrow,
                                                            const double *__restrict__ crow, double2 *__restrict__ hat) {
    using F = RFft<N, CS_T>;
    using C2 = Cx<double2>;
    constexpr int NK = N < 64 ? N : 64, NR = 2 * CS_SEGS;   // kz at a time, reduced rows
    static_assert(NK * CS_SEGS <= CS_T, "a thread per segment");
    extern __shared__ __align__(16) unsigned char lds_raw[];
    double2 *tile = reinterpret_cast<double2 *>(lds_raw), *twl = tile + CS_SEGS * M * F::LS;
    double *ra = reinterpret_cast<double *>(twl + F::TW), *rb = ra + NR * NK, *rc = rb + NR * NK;
    const int kx = blockIdx.x, t = threadIdx.x % F::M, l = threadIdx.x / F::M;
    double2 *col = hat + (size_t)kx * ny * N;
    rf_stage<double2, N, CS_T>(twl, tw);
    if constexpr (!F::TW0) __syncthreads();
    for (int j0 = 0; j0 < ny; j0 += F::LPW) {
        const int j = j0 + l;
        const bool on = j < ny;
        double2 *line = tile + (on ? j : 0) * F::LS;
        double2 e[16];   // (one for both loops would keep idle lanes' values through the solves: spills)
        if (on) {
#pragma unroll
            for (int s = 0; s < 16; ++s) e[s] = col[(size_t)j * N + t + F::M * s];
        }
        fft_line<double2, N, false>(e, t, twl, line, on);
        __syncthreads();
        if (on) {
#pragma unroll
            for (int s = 0; s < 16; ++s) line[rf_pad(t + F::M * s)] = e[s];
        }
    }
    const int tk = threadIdx.x % NK, sg = threadIdx.x / NK, r0 = sg * M;
    for (int k0 = 0; k0 < N; k0 += NK) {
        const int kz = k0 + tk;
        const bool mine = sg < CS_SEGS;
        double2 *c = tile + rf_pad(kz);
        const double k = lamx[kx] + lamz[kz];
        const double2 zero = make_double2(0.0, 0.0);
        auto solved = [&](int r) { return r0 + r < ny && !(kx == 0 && kz == 0 && r0 + r == 0); };
        auto coef = [&](int r, double &a, double &b, double &cc) {
            a = cc = 0.0;
            b = 1.0;
            if (solved(r)) {
                a = arow[r0 + r];
                b = bdrow[r0 + r] - k;
                cc = crow[r0 + r];
            }
        };
        double2 p[M], df = zero, dl = zero;
        TriSegment<double2, M, REFINE> seg;
        __syncthreads();
        if (mine) {
#pragma unroll
            for (int r = 0; r < M; ++r) {
                p[r] = zero;
                if (solved(r)) p[r] = c[(r0 + r) * F::LS];
            }
            df = p[0];
            dl = p[M - 1];
            seg.eliminate(coef, p);
            const int f = 2 * sg * NK + tk, g = f + NK;
            seg.first(ra[f], rb[f], rc[f]);
            c[r0 * F::LS] = seg.first(p);
            seg.last(ra[g], rb[g], rc[g]);
            c[(r0 + M - 1) * F::LS] = seg.last(p);
        }
        // the reduced rows of a kz, by the first segment's thread; again: with the kept factors
        auto reduced = [&](auto again_) {
            constexpr bool again = decltype(again_)::value;
            auto row = [&](int r) -> double2 & { return c[(r / 2 * M + (r % 2 ? M - 1 : 0)) * F::LS]; };
            constexpr int CH = REFINE ? 8 : NR;   // rows read ahead of the chain
            double cs[CH], cprev = 0.0;
            double2 ds[CH], dprev = zero;
#pragma unroll
            for (int q = 0; q < NR; q += CH) {
#pragma unroll
                for (int u = 0; u < CH; ++u) ds[u] = row(q + u);
#pragma unroll
                for (int u = 0; u < CH; ++u) {
                    const int o = (q + u) * NK + tk;
                    const double a = ra[o];
                    double rden = rb[o];
                    if (!again) {
                        rden = 1.0 / (rden - a * cprev);
                        cs[u] = cprev = rc[o] * rden;
                        if (REFINE) {
                            rb[o] = rden;
                            rc[o] = cprev;
                        }
                    }
                    ds[u] = dprev = C2::mk((ds[u].x - a * dprev.x) * rden, (ds[u].y - a * dprev.y) * rden);
                    if (REFINE) row(q + u) = dprev;
                }
                if (REFINE) __builtin_amdgcn_sched_barrier(0);
            }
            if (!REFINE) row(NR - 1) = dprev;
#pragma unroll
            for (int q = NR - CH; q >= 0; q -= CH) {
                if (REFINE) {
#pragma unroll
                    for (int u = 0; u < CH; ++u) {
                        ds[u] = row(q + u);
                        cs[u] = rc[(q + u) * NK + tk];
                    }
                }
#pragma unroll
                for (int u = CH - 1; u >= 0; --u) {
                    if (q + u == NR - 1) continue;
                    dprev = C2::mk(ds[u].x - cs[u] * dprev.x, ds[u].y - cs[u] * dprev.y);
                    row(q + u) = dprev;
                }
                if (REFINE) __builtin_amdgcn_sched_barrier(0);
            }
        };
        __syncthreads();
        if (sg == 0) reduced(std::false_type{});
        __syncthreads();
        if constexpr (REFINE) {
            double2 x[M];
            if (mine) {
                const double2 f = c[r0 * F::LS], g = c[(r0 + M - 1) * F::LS];
                double2 xm = zero, xp = zero;
                if (sg > 0) xm = c[(r0 - 1) * F::LS];
                if (sg < CS_SEGS - 1) xp = c[(r0 + M) * F::LS];
#pragma unroll
                for (int r = 0; r < M; ++r) x[r] = seg.row(p, r, f, g);
                // (the interior rows' data are still in the tile)
                auto data = [&](int r) {
                    double2 v = zero;
                    if (r == 0) v = df;
                    else if (r == M - 1) v = dl;
                    else if (solved(r)) v = c[(r0 + r) * F::LS];
                    return v;
                };
                tri_residual<double2, M>(coef, data, x, xm, xp, p);
                seg.again(coef, p);
            }
            __syncthreads();   // the neighbours' ends have been read
            if (mine) {
                c[r0 * F::LS] = seg.first(p);
                c[(r0 + M - 1) * F::LS] = seg.last(p);
            }
            __syncthreads();
            if (sg == 0) reduced(std::true_type{});
            __syncthreads();
            if (mine) {
                const double2 f = c[r0 * F::LS], g = c[(r0 + M - 1) * F::LS];
#pragma unroll
                for (int r = 0; r < M; ++r) {
                    const double2 v = seg.row(p, r, f, g);
                    if (r0 + r < ny) c[(r0 + r) * F::LS] = C2::mk(x[r].x + v.x, x[r].y + v.y);
                }
            }
        } else if (mine) {
            const double2 f = c[r0 * F::LS], g = c[(r0 + M - 1) * F::LS];
#pragma unroll
            for (int r = 1; r <= M - 2; ++r)
                if (r0 + r < ny) c[(r0 + r) * F::LS] = seg.row(p, r, f, g);
        }
    }
    __syncthreads();
    for (int j0 = 0; j0 < ny; j0 += F::LPW) {
        const int j = j0 + l;
        const bool on = j < ny;
        double2 *line = tile + (on ? j : 0) * F::LS;
        double2 e[16];
        if (on) rf_gather<double2, N>(e, t, line);
        if constexpr (!F::TW0) __syncthreads();
        fft_line<double2, N, true>(e, t, twl, line, on);
        if (on) {
#pragma unroll
            for (int s = 0; s < 16; ++s) col[(size_t)j * N + t + F::M * s] = e[s];
        }
        __syncthreads();
    }
}

// launches the partitioned solve for ny <= 256, in FP32 for ny >= 64 (false: the caller takes another
// solver).  Below 64 rows a line's segments past ny idle, and still FP64, with its refinement step,
// takes 14.1 us at 128 x 33 x 128 where a wave per line took 28.8; the FP32 passes of the defect
// correction keep the wave's rounding there.
template <typename C, bool MEAN_ZERO>
static bool launch_tridiag_part(hipStream_t st, const Dims &d, C *hat, const typename Cx<C>::R *lamx,
                                const typename Cx<C>::R *lamz, const typename Cx<C>::R *a,
                                const typename Cx<C>::R *bd, const typename Cx<C>::R *c) {
    if ((sizeof(C) == 8 && d.ny < 64) || d.ny > 256) return false;
    const int nxh = d.nx / 2 + 1, stride = fft_stride_t<C>(d.nx), nlines = stride * d.nz, m = (d.ny + TP_SEGS - 1) / TP_SEGS;
    const size_t plane = (size_t)nlines;
    const dim3 grid((nlines + TP_LINES - 1) / TP_LINES), blk(TP_LINES * TP_SEGS);
#define TP_LAUNCH(MM, REF)                                                                                         \
    hipLaunchKernelGGL((tridiag_part_kernel<C, MM, MEAN_ZERO, REF>), grid, blk, 0, st, nlines, stride, nxh, d.ny, \
                       plane, hat, lamx, lamz, a, bd, c)
    if (d.ny < 64) {
        if constexpr (sizeof(C) == 16) TP_LAUNCH(4, true);
        return true;
    }
#define TP_CASE(MM)           \
    if (m <= MM) {            \
        TP_LAUNCH(MM, false); \
        return true;          \
    }
    TP_CASE(4) TP_CASE(8) TP_CASE(12) TP_CASE(16)
#undef TP_CASE
#undef TP_LAUNCH
    return false;
}

// launches the one-wave-per-line solve for ny <= 256 (false: the caller runs the Thomas kernel)
template <typename C, bool MEAN_ZERO>
static bool launch_tridiag_wave(hipStream_t st, const Dims &d, C *hat, const typename Cx<C>::R *lamx,
                                const typename Cx<C>::R *lamz, const typename Cx<C>::R *a,
                                const typename Cx<C>::R *bd, const typename Cx<C>::R *c) {
    const int nxh = d.nx / 2 + 1, stride = fft_stride_t<C>(d.nx), nlines = stride * d.nz, m = (d.ny + 63) / 64;
    const size_t plane = (size_t)nlines;
    const dim3 grid((nlines + TW_LINES - 1) / TW_LINES), blk(64 * TW_WAVES);
    const size_t lds = (size_t)TW_LINES * (d.ny + 1) * sizeof(C);   // <= 66 KB (ny <= 256)
#define TW_CASE(MM)                                                                                            \
    case MM: {                                                                                                 \
        if (allow_lds<tridiag_wave_kernel<C, MM, MEAN_ZERO>>(lds) != hipSuccess) return false;                 \
        hipLaunchKernelGGL((tridiag_wave_kernel<C, MM, MEAN_ZERO>), grid, blk, lds, st, nlines, stride, nxh, d.ny, plane, \
                           hat, lamx, lamz, a, bd, c);                                                         \
        return true;                                                                                           \
    }
    switch (m) {
    TW_CASE(1) TW_CASE(2) TW_CASE(3) TW_CASE(4)
    default: return false;
    }
#undef TW_CASE
}

// 5. c2r along x: the real parts of the kx=0 and kx=nx/2 coefficients, Hermitian extension of the
//    rest, inverse transform, times 1/(nx nz); phi in rhs layout (nx, nz, ny).
__global__ __launch_bounds__(FFT_THREADS) void ixfft_kernel(Dims d, const double2 *__restrict__ hat,
                                                           const double2 *__restrict__ tw, int lines,
                                                           int stride, double scale, double *phi) {
    extern __shared__ __align__(16) unsigned char lds_raw[];
    double2 *lds = reinterpret_cast<double2 *>(lds_raw);
    const int n = d.nx, nxh = n / 2 + 1;
    const int nrows = d.ny * d.nz;
    double2 *a = lds, *b = lds + (size_t)lines * n, *twl = b + (size_t)lines * n;
    stage_twiddles(twl, tw, n);
    for (int t = threadIdx.x; t < lines * n; t += FFT_THREADS) {
        const int line = t / n, m = t - line * n;
        const int r = blockIdx.x * lines + line;
        double2 v = make_double2(0.0, 0.0);
        if (r < nrows) {
            const double2 *row = hat + (size_t)stride * r;
            if (m == 0 || 2 * m == n) v = make_double2(row[m].x, 0.0);
            else if (m < nxh) v = row[m];
            else v = make_double2(row[n - m].x, -row[n - m].y);
        }
        a[t] = v;
    }
    __syncthreads();
    double2 *res = stockham(a, b, n, lines, n, twl, true, threadIdx.x, FFT_THREADS);
    for (int t = threadIdx.x; t < lines * n; t += FFT_THREADS) {
        const int line = t / n, i = t - line * n;
        const int r = blockIdx.x * lines + line;
        if (r < nrows) phi[(size_t)n * r + i] = res[t].x * scale;
    }
}

// workgroup shape of the k-marching fft_div_rhs_kernel: 64 x FC_Y cells, FC_KZ planes
static constexpr int FC_Y = 4, FC_KZ = 16;

// a plane's sum from the partial sums of fft_plane_sum_kernel
static constexpr int PLANE_CHUNKS = 16;
__device__ inline double plane_sum(const double *part, int j) {
    double a = 0.0;
    for (int c = 0; c < PLANE_CHUNKS; ++c) a += part[j * PLANE_CHUNKS + c];
    return a;
}

// 6. u = (u* - dtg grad phi)/(1 + dtg coef) and p += phi (pressure_solver.f90:129-173).  Each thread
// takes one column (i,j) of a 64 x 4 tile and marches `kz` planes, FC_CH planes' loads in flight at
// a time (phi(k-1) stays in a register).  Inside a step (FftStep) the same pass also
//   * shifts u* by the flow-rate correction, folded here from the partial sums in every workgroup's
//     own order-fixed way (a uniform shift drops out of the divergence, so the right-hand side does
//     not need it; a pass of its own read and wrote u* once more, 54 us at 256 x 192 x 256), and
//     stores it if the step leaves u* visible (store_us);
//   * writes the ghosts of the new fields as apply_bc fills them, from the cells at the boundary
//     (the separate fill took three launches and 31 us, 10 at 64^3).
// pin: the plane sums whose mean (plane 1) is taken off phi, where the solve leaves that to this pass.
// Bound by HBM: 9 arrays once, 72 B per cell.
static constexpr int FC_CH = 4;
struct FftStep {
    const double *part = nullptr;   // flow-rate partial sums, nparts pairs (none: no shift)
    int nparts = 0;
    double norm = 1.0, target = 0.0;
    double *out = nullptr;          // bulk velocity, mean mu_u, du
    int store_us = 0, ghosts = 0;
    const double *pin = nullptr;
};
template <bool STRETCH, bool IBM>
__global__ __launch_bounds__(256) void fft_correct_kernel(GridK g, const double *__restrict__ phi, double *us,
                                                          const double *__restrict__ vs,
                                                          const double *__restrict__ ws,
                                                          const double *__restrict__ cu,
                                                          const double *__restrict__ cv,
                                                          const double *__restrict__ cw, double dtg, int kz,
                                                          FftStep fs, double *un, double *vn, double *wn, double *pn) {
    const Dims d = g.d;
    int tx, ty, tz;
    if (!xcd_tile(d.nx, d.ny, (d.nz + kz - 1) / kz, 64, 4, tx, ty, tz)) return;   // uniform per workgroup
    const int nx = d.nx, ny = d.ny, nz = d.nz;
    const int i0 = tx * 64 + threadIdx.x + 1, j0 = ty * 4 + threadIdx.y + 1;
    const int i = i0 < nx ? i0 : nx, j = j0 < ny ? j0 : ny;   // threads past the grid load the last cells'
    const int k0 = tz * kz + 1, k1 = k0 + kz - 1 < nz ? k0 + kz - 1 : nz;
    const size_t sz = (size_t)d.sx * d.sy;
    const double rx = 1.0 / g.dx, ry = 1.0 / g.dy, rz = 1.0 / g.dz, ih = STRETCH ? g.ihv[j] : 0.0;
    // phi(i,k,j) in (nx, nz, ny) layout, its x neighbour and the row below
    const double *p = phi + (size_t)(i - 1) + (size_t)nx * ((size_t)(k0 - 1) + (size_t)nz * (size_t)(j - 1));
    const ptrdiff_t om = i == 1 ? nx - 1 : -1, oj = j >= 2 ? -(ptrdiff_t)nx * nz : 0;
    size_t c = d.g(i, j, k0);
    double pp[FC_CH], px[FC_CH], py[FC_CH], a[FC_CH], b[FC_CH], e[FC_CH], q[FC_CH];
    auto load = [&](int k) {   // planes k .. k + FC_CH - 1 (past the end: the last one again, unused)
#pragma unroll
        for (int u = 0; u < FC_CH; ++u) {
            const int w = k + u <= k1 ? u : k1 - k;
            const size_t cc = c + w * sz;
            pp[u] = p[w * (ptrdiff_t)nx];
            px[u] = p[w * (ptrdiff_t)nx + om];
            py[u] = p[w * (ptrdiff_t)nx + oj];
            a[u] = us[cc];
            b[u] = j >= 2 ? vs[cc] : 0.0;
            e[u] = ws[cc];
            q[u] = pn[cc];
        }
    };
    load(k0);   // before the folds, whose loads and barriers take as long
    const double pkm = k0 > 1 ? p[-(ptrdiff_t)nx] : p[(ptrdiff_t)nx * (nz - k0)];
    double du = 0.0;
    if (fs.part) {
        __shared__ double s1[256], s2[256];
        double o[3];
        flow_fold(fs.part, fs.nparts, fs.norm, fs.target, threadIdx.x + 64 * threadIdx.y, s1, s2, o);
        du = o[2];
        if (blockIdx.x == 0 && threadIdx.x + threadIdx.y == 0) {
            fs.out[0] = o[0];
            fs.out[1] = o[1];
            fs.out[2] = o[2];
        }
    }
    const double pc = fs.pin ? plane_sum(fs.pin, 0) / (double)((long)nx * nz) : 0.0;
    if (i0 > nx || j0 > ny) return;
    double pm = pkm - pc;
    const int xi = i == nx ? -nx : i == 1 ? nx : 0;   // to the column's x image, if it has one
    auto put = [&](double *f, size_t cc, double v, ptrdiff_t zi) {   // a value and its periodic images
        f[cc] = v;
        if (!fs.ghosts) return;
        if (xi) f[cc + xi] = v;
        if (zi) {
            f[cc + zi] = v;
            if (xi) f[cc + zi + xi] = v;
        }
    };
    for (int k = k0;;) {
#pragma unroll
        for (int u = 0; u < FC_CH; ++u) {
            if (k + u > k1) break;
            const size_t cc = c + u * sz;
            const ptrdiff_t zi = k + u == nz ? -(ptrdiff_t)(nz * sz) : k + u == 1 ? (ptrdiff_t)(nz * sz) : 0;
            const double p0 = pp[u] - pc;
            if (fs.part) {
                a[u] = a[u] + du;
                if (fs.store_us) us[cc] = a[u];
            }
            double U = a[u] - div_by(dtg * (p0 - (px[u] - pc)), g.dx, rx);
            double W = e[u] - div_by(dtg * (p0 - pm), g.dz, rz);
            const double gy = dtg * (p0 - (py[u] - pc));
            double V = b[u] - (STRETCH ? gy * ih : div_by(gy, g.dy, ry));
            if (IBM) {
                U = U / (1.0 + dtg * cu[cc]);
                W = W / (1.0 + dtg * cw[cc]);
                V = V / (1.0 + dtg * cv[cc]);
            }
            put(un, cc, U, zi);
            put(wn, cc, W, zi);
            put(pn, cc, q[u] + p0, zi);
            if (j >= 2) put(vn, cc, V, zi);
            if (fs.ghosts) {
                if (j == 1) {
                    put(un, cc - d.sx, -U, zi);
                    put(wn, cc - d.sx, -W, zi);
                    put(vn, cc, 0.0, zi);
                }
                if (j == ny) {
                    put(un, cc + d.sx, -U, zi);
                    put(wn, cc + d.sx, -W, zi);
                    put(vn, cc + d.sx, 0.0, zi);
                }
            }
            pm = p0;
        }
        k += FC_CH;
        if (k > k1) break;
        c += FC_CH * sz;
        p += FC_CH * (ptrdiff_t)nx;
        load(k);
    }
}

bool fft_sums(const mdx_handle *h) {
    return h->cfg.precision != MDX_PREC_MIXED && h->d.nx >= 16 && momentum_sums_apart(h);
}

// whether the projection takes u*'s ghosts as filled and writes the new fields' itself
static int fft_wrap(const mdx_handle *h) { return h->step_bc && h->fused_bc; }

// the flow-rate shift the projection of a step makes
static FftStep fft_step(const mdx_handle *h) {
    FftStep fs;
    if (!h->step_bc || !h->step_parts) return fs;
    fs.part = h->fr_part;
    fs.nparts = h->step_parts;
    fs.norm = (double)h->d.nx * (double)h->d.nz * h->cfg.flow_height;
    fs.target = h->cfg.ub_target;
    fs.out = h->red_part + 2048;
    fs.store_us = h->step_last;
    return fs;
}

// Planes per workgroup of the correction: up to 16 (the phi(k-1) loads and the folds are per
// workgroup), down to one chunk while the workgroups would not give every CU four: 7.5 us at 64^3
// with 4 planes against 9.9 with 1; 214 us at 256 x 192 x 256 with 4 as with 16 or 32.
static hipError_t launch_correct(mdx_handle *h, const double *phi, double dtg, const double *pin) {
    GridK g = grid_k(h);
    const Dims d = h->d;
    int kz = 16;
    while (kz > FC_CH && xcd_grid(d.nx, d.ny, (d.nz + kz - 1) / kz, 64, 4) < 1024) kz /= 2;
    FftStep fs = fft_step(h);
    fs.ghosts = fft_wrap(h);
    fs.pin = pin;
#define MDX_CORR(S, I)                                                                                             \
    hipLaunchKernelGGL((fft_correct_kernel<S, I>), dim3(xcd_grid(d.nx, d.ny, (d.nz + kz - 1) / kz, 64, 4)),        \
                       dim3(64, 4), 0, h->stream, g, phi, h->us, h->vs, h->ws, h->cu, h->cv, h->cw, dtg, kz, fs,   \
                       h->un, h->vn, h->wn, h->pn)
    if (h->stretched) { if (h->ibm_on) MDX_CORR(true, true); else MDX_CORR(true, false); }
    else { if (h->ibm_on) MDX_CORR(false, true); else MDX_CORR(false, false); }
#undef MDX_CORR
    h->apply_wrote_bc = fs.ghosts;
    return hipGetLastError();
}

static int rows_per_block(int n) {
    int lines = (4 * FFT_THREADS) / n;   // n/4 radix-4 butterflies per line, FFT_THREADS threads
    if (lines < 1) lines = 1;
    return lines;
}

static int z_tile(int nz) {
    int tx = 2048 / nz;                  // 2 buffers x tx x (nz + 1) x 16 B, about 64 KB
    if (tx < 1) tx = 1;
    if (tx > 16) tx = 16;
    return tx;
}

// dynamic LDS of the transforms: two ping-pong buffers of `lines` lines (stride ls) and the twiddles
template <typename C>
static size_t fft_lds(int lines, int ls, int n) {
    return (2 * (size_t)lines * ls + (size_t)(n / 2)) * sizeof(C);
}

// a kernel of the register transforms on `blocks` workgroups
template <typename C, int N, int TH, auto FN, int W = 1, typename... A>
static hipError_t rf_launch(hipStream_t st, unsigned blocks, A... args) {
    using F = RFft<N, TH>;
    const size_t lds = ((size_t)F::LPW * F::LS + F::TW) * sizeof(C);
    const hipError_t e = allow_lds<FN>(lds);
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(FN, dim3(blocks), dim3(TH * W), lds, st, args...);
    return hipGetLastError();
}
// CALL(N) for the register transforms' lengths (it returns); shorter lines fall through
#define RF_SIZES(n, CALL)  \
    switch (n) {           \
    case 16: CALL(16);     \
    case 32: CALL(32);     \
    case 64: CALL(64);     \
    case 128: CALL(128);   \
    case 256: CALL(256);   \
    case 512: CALL(512);   \
    case 1024: CALL(1024); \
    default: break;        \
    }

template <int N, int TH>
static unsigned rf_row_blocks(const Dims &d, int rows = 2) {   // rows: rows per line
    return (unsigned)((d.ny * d.nz / rows + RFft<N, TH>::LPW - 1) / RFft<N, TH>::LPW);
}
// Workgroups of one transforming wavefront (64 threads; the x-transform with the right-hand side adds
// three that only load and store) where those of 256 would leave CUs without two: `blocks256` is the
// number of the latter.  Measured at 64^3 (32 to 36 workgroups of 256): z 10.2 us -> 5.0 us, x with
// the right-hand side 17.3 -> 7.5, x inverse 5.8 -> 4.2; 128 x 97 x 64: 10.9 -> 6.8, 18.2 -> 9.5,
// 6.4 -> 5.1.  At 256 x 192 x 256 (1536 and more) x does not depend on it; in z a wavefront alone has
// 4 columns, 64 bytes, of each kz: FP64 56 and 51 us against 48 and 42 with 256 threads and 41 and 38
// with the 128 taken there, whose 8 columns are one cache line (FP32: 16 columns, 256 threads).
static bool rf_small(unsigned blocks256) {
    return blocks256 < 512;
}

template <typename C, int N, int TH, bool INV>
static hipError_t rf_zfft_t(hipStream_t st, const Dims &d, C *hat, const C *tw) {
    using F = RFft<N, TH>;
    const int nxh = d.nx / 2 + 1;
    int cw = F::LPW < 16 ? F::LPW : 16;
    while (cw > d.nx / 2) cw /= 2;
    const int pw = F::LPW / cw, ntx = nxh / cw, nrem = nxh - ntx * cw;
    const int tiles = ntx * ((d.ny + pw - 1) / pw), rem = (nrem * d.ny + F::LPW - 1) / F::LPW;
    return rf_launch<C, N, TH, zfft_reg_kernel<C, N, TH, INV>>(st, (unsigned)(tiles + rem), d.ny, fft_stride_t<C>(d.nx), cw,
                                                               ntx, tiles, nrem, tw, hat);
}
template <typename C, int N, bool INV>
static hipError_t rf_zfft(hipStream_t st, const Dims &d, C *hat, const C *tw) {
    return rf_small((unsigned)((d.nx / 2 + 1) * d.ny / RFft<N, 256>::LPW)) ? rf_zfft_t<C, N, 64, INV>(st, d, hat, tw)
                                                                         : rf_zfft_t<C, N, sizeof(C) == 16 ? 128 : 256, INV>(st, d, hat, tw);
}
// z-transform of the whole spectrum
template <typename C, bool INV>
static hipError_t launch_zfft(hipStream_t st, const Dims &d, C *hat, const C *tw) {
#define ZF(N) return rf_zfft<C, N, INV>(st, d, hat, tw)
    RF_SIZES(d.nz, ZF)
#undef ZF
    const int tx = z_tile(d.nz), nxh = d.nx / 2 + 1;
    const size_t shz = fft_lds<C>(tx, d.nz + 1, d.nz);
    hipLaunchKernelGGL(zfft_kernel<C>, dim3(d.ny * ((nxh + tx - 1) / tx)), dim3(FFT_THREADS), shz, st, d, hat, tw, tx,
                       INV ? 1 : 0, fft_stride_t<C>(d.nx));
    return hipGetLastError();
}

// the x points of a column-solved grid
static constexpr int COLUMN_NX = 256;

// (TRK: into the transposed spectrum of the column solves)
template <bool TRK> static hipError_t launch_rhs_xfft(mdx_handle *h, double dtg) {
    GridK g = grid_k(h);
    const Dims d = h->d;
    const int stride = fft_stride_t<double2>(d.nx);
#define XF_(N, TH, W, S)                                                                                              \
    do {                                                                                                              \
        const unsigned nb = rf_row_blocks<N, TH>(d);                                                                  \
        const FlowSum fsum{(int)nb, h->mom_kz, h->fr_part};                                                           \
        return rf_launch<double2, N, TH, rhs_xfft_reg_kernel<N, TH, W, S, W == 4 && TRK>, W>(                         \
            h->stream, nb + (h->step_sum ? momentum_tiles(h) : 0), g, (const double *)h->us, (const double *)h->vs,   \
            (const double *)h->ws, dtg, fft_wrap(h), fsum, (const double2 *)h->tw_x, TRK ? d.ny * d.nz : stride,       \
            (double2 *)h->hat);                                                                                       \
    } while (0)
#define XF(N)                                                  \
    if constexpr (!TRK || N <= COLUMN_NX) {                    \
        if (TRK || rf_small(rf_row_blocks<N, 256>(d))) {       \
            if (h->stretched) XF_(N, 64, 4, true);             \
            XF_(N, 64, 4, false);                              \
        }                                                      \
    }                                                          \
    if constexpr (!TRK) {                                      \
        if (h->stretched) XF_(N, 256, 1, true);                \
        XF_(N, 256, 1, false);                                 \
    }                                                          \
    break
    RF_SIZES(d.nx, XF)
#undef XF
#undef XF_
    if (TRK) return hipErrorInvalidValue;   // (columns_fit)
    const int lines = rows_per_block(d.nx);
    const int nrows = d.ny * d.nz;
    const size_t shx = fft_lds<double2>(lines, d.nx, d.nx);
    if (h->stretched)
        hipLaunchKernelGGL(rhs_xfft_kernel<true>, dim3((nrows + lines - 1) / lines), dim3(FFT_THREADS), shx,
                           h->stream, g, h->us, h->vs, h->ws, dtg, fft_wrap(h), (const double2 *)h->tw_x, lines, stride,
                           (double2 *)h->hat);
    else
        hipLaunchKernelGGL(rhs_xfft_kernel<false>, dim3((nrows + lines - 1) / lines), dim3(FFT_THREADS), shx,
                           h->stream, g, h->us, h->vs, h->ws, dtg, fft_wrap(h), (const double2 *)h->tw_x, lines, stride,
                           (double2 *)h->hat);
    return hipGetLastError();
}

static hipError_t launch_ixfft(mdx_handle *h, double *phi) {
    const Dims d = h->d;
    const int stride = fft_stride_t<double2>(d.nx);
    const double scale = 1.0 / (double)(d.nx * d.nz);
#define IX_(N, TH)                                                                                                  \
    return rf_launch<double2, N, TH, ixfft_reg_kernel<N, TH>>(h->stream, rf_row_blocks<N, TH>(d), d,                 \
                                                              (const double2 *)h->hat, (const double2 *)h->tw_x,    \
                                                              stride, scale, phi)
#define IX(N)                                                \
    if (rf_small(rf_row_blocks<N, 256>(d))) IX_(N, 64);      \
    IX_(N, 256)
    RF_SIZES(d.nx, IX)
#undef IX
#undef IX_
    const int lines = rows_per_block(d.nx);
    const int nrows = d.ny * d.nz;
    const size_t shx = fft_lds<double2>(lines, d.nx, d.nx);
    hipLaunchKernelGGL(ixfft_kernel, dim3((nrows + lines - 1) / lines), dim3(FFT_THREADS), shx, h->stream, d,
                       (const double2 *)h->hat, (const double2 *)h->tw_x, lines, stride, scale, phi);
    return hipGetLastError();
}

// the LDS a column may take
static constexpr size_t COLUMN_LDS = 160 * 1024 - 1024;
template <int N, int M> static hipError_t column_solve(mdx_handle *h) {
    const Dims d = h->d;
    constexpr size_t lds = column_lds<N, M>();
    auto launch = [&](auto refine) {
        constexpr auto FN = column_solve_kernel<N, M, decltype(refine)::value>;
        const hipError_t e = allow_lds<FN>(lds);
        if (e != hipSuccess) return e;
        hipLaunchKernelGGL(FN, dim3(d.nx / 2 + 1), dim3(CS_T), lds, h->stream, d.ny, (const double2 *)h->tw_z, h->lamx,
                           h->lamz, h->tw_a, h->bdrow, h->crow, (double2 *)h->hat);
        return hipGetLastError();
    };
    if constexpr (CS_SEGS * M < 64) return launch(std::true_type{});
    else if constexpr (CS_SEGS * (M - 1) >= 63) return launch(std::false_type{});
    else return d.ny < 64 ? launch(std::true_type{}) : launch(std::false_type{});
}
// Rows per segment: the fewest that reach ny (every further one is a step of all chains and a line of
// LDS), from 4 to 16, what a thread's registers hold; the larger ones only where the column fits.
template <int N, int M = 4> static bool column_fits(int m) {
    if constexpr (M > 16 || column_lds<N, M>() > COLUMN_LDS) return false;
    else return m <= M || column_fits<N, M + 1>(m);
}
template <int N, int M = 4> static hipError_t column_solve_rows(mdx_handle *h, int m) {
    if constexpr (M > 16 || column_lds<N, M>() > COLUMN_LDS) return hipErrorInvalidValue;
    else return m <= M ? column_solve<N, M>(h) : column_solve_rows<N, M + 1>(h, m);
}
// Whether (2.) to (4.) go column by column in one launch: FP64 grids whose x-transforms take the
// small workgroups, with a kx column in LDS.  A step against the three launches: 128 and 163 us at
// 64^3, 204 and 250 at 128 x 97 x 64, 219 and 246 at 128 x 120 x 64, 224 and 264 at 256 x 60 x 64, 110 and 129 at
// 32 x 24 x 32, 154 and 160 at 16 x 96 x 64 (nine columns).
static bool columns_fit(const mdx_handle *h) {
    const Dims d = h->d;
    if (!h->wave_tridiag || !h->part_tridiag || d.nx < 16 || d.nx > COLUMN_NX) return false;
    const int lines = 256 * 16 / d.nx;   // RFft<nx, 256>::LPW
    if (!rf_small((unsigned)((d.ny * d.nz / 2 + lines - 1) / lines))) return false;
    const int m = (d.ny + CS_SEGS - 1) / CS_SEGS;
    switch (d.nz) {
    case 32: return column_fits<32>(m);
    case 64: return column_fits<64>(m);
    case 128: return column_fits<128>(m);
    default: return false;
    }
}
static hipError_t launch_columns(mdx_handle *h) {
    const int m = (h->d.ny + CS_SEGS - 1) / CS_SEGS;
    switch (h->d.nz) {
    case 32: return column_solve_rows<32>(h, m);
    case 64: return column_solve_rows<64>(h, m);
    case 128: return column_solve_rows<128>(h, m);
    default: return hipErrorInvalidValue;
    }
}

static hipError_t launch_ixfft_columns(mdx_handle *h, double *phi) {
    const Dims d = h->d;
    const double scale = 1.0 / (double)(d.nx * d.nz);
#define IX(N)                                                                                                       \
    if constexpr (N <= COLUMN_NX)                                                                                   \
        return rf_launch<double2, N, 64, ixfft_columns_kernel<N, 64, 4>, 4>(h->stream, rf_row_blocks<N, 64>(d), d,  \
                                                                            (const double2 *)h->hat,                \
                                                                            (const double2 *)h->tw_x, d.ny * d.nz,  \
                                                                            scale, phi);                            \
    break
    RF_SIZES(d.nx, IX)
#undef IX
    return hipErrorInvalidValue;
}

hipError_t launch_fft_forward(mdx_handle *h, double dtg) {
    if (columns_fit(h)) return launch_rhs_xfft<true>(h, dtg);
    const hipError_t e = launch_rhs_xfft<false>(h, dtg);
    return e != hipSuccess ? e
                           : launch_zfft<double2, false>(h->stream, h->d, (double2 *)h->hat, (const double2 *)h->tw_z);
}

hipError_t launch_tridiag(mdx_handle *h) {
    if (columns_fit(h)) return launch_columns(h);   // with both z-transforms
    const Dims d = h->d;
    const int nlines = (d.nx / 2 + 1) * d.nz;
    if (h->wave_tridiag && h->part_tridiag &&
        launch_tridiag_part<double2, false>(h->stream, d, (double2 *)h->hat, h->lamx, h->lamz, h->tw_a, h->bdrow,
                                            h->crow))
        return hipGetLastError();
    if (h->wave_tridiag && launch_tridiag_wave<double2, false>(h->stream, d, (double2 *)h->hat, h->lamx, h->lamz, h->tw_a,
                                                     h->bdrow, h->crow))
        return hipGetLastError();
    hipLaunchKernelGGL(tridiag_kernel, dim3((nlines + 63) / 64), dim3(64), 0, h->stream, d, fft_stride_t<double2>(d.nx),
                       (double2 *)h->hat, h->cp, h->den_inv, h->arow);
    return hipGetLastError();
}

hipError_t launch_fft_backward_correct(mdx_handle *h, double dtg) {
    hipError_t e;
    if (columns_fit(h)) {
        e = launch_ixfft_columns(h, h->fft_rhs);
    } else {
        e = launch_zfft<double2, true>(h->stream, h->d, (double2 *)h->hat, (const double2 *)h->tw_z);
        if (e == hipSuccess) e = launch_ixfft(h, h->fft_rhs);
    }
    return e != hipSuccess ? e : launch_correct(h, h->fft_rhs, dtg, nullptr);
}

// ------------------------------------------------------------------------------- mixed precision
// FP32 transforms and Thomas solves inside an FP64 defect correction.  Each pass takes the residual
// r = rhs - L phi, formed in FP64 with the discrete operator the transforms diagonalise (3-point
// second differences in x and z, the tridiagonal rows in y).  Its mean mode (kx = kz = 0), whose
// system is singular and pinned by phi_hat(y_1) = 0 (pressure_fft.f90:92-96, 119-121), is solved in
// FP64 from the plane sums of r; the other modes go through the FP32 transforms and Thomas solves.

// rhs(i,k,j) of rhs_xfft_kernel, in FP64, layout (nx, nz, ny).  A 64 x FC_Y workgroup owns rows
// j0 .. j0+FC_Y-1 of a 64-cell x segment and marches FC_KZ planes: w*(k+1) becomes w*(k) of the
// next plane in a register and u*(i+1) comes from the lane above (lane 63 reads it), so w* and u*
// are fetched about once; v*(j+1) is the row above's v*(j) (a cache hit).  wrap: as in
// rhs_xfft_reg_kernel; fs: the flow-rate shift of u*, added before the differences (it drops out of
// them but for rounding, which the FP32 passes would turn into differences of their own precision).
// The first pass starts from phi = 0, whose residual is the right-hand side, so max |rhs| is formed here.
template <bool STRETCH>
__global__ __launch_bounds__(64 * FC_Y) void fft_div_rhs_kernel(GridK g, const double *__restrict__ us,
                                                               const double *__restrict__ vs,
                                                               const double *__restrict__ ws, double dtg, int wrap,
                                                               FftStep fs, double *__restrict__ rhs, double *part) {
    static_assert(64 * FC_Y == 256, "the fold's threads");
    const Dims d = g.d;
    double du = 0.0;
    if (fs.part) {
        __shared__ double s1[256], s2[256];
        double o[3];
        flow_fold(fs.part, fs.nparts, fs.norm, fs.target, threadIdx.x + 64 * threadIdx.y, s1, s2, o);
        du = o[2];
    }
    const int lane = threadIdx.x;
    const int i = blockIdx.x * 64 + lane + 1;
    const int j = blockIdx.y * FC_Y + threadIdx.y + 1;
    const int k0 = blockIdx.z * FC_KZ + 1, k1 = k0 + FC_KZ - 1 < d.nz ? k0 + FC_KZ - 1 : d.nz;
    const bool act = i <= d.nx && j <= d.ny;
    double wk = act ? ws[d.g(i, j, k0)] : 0.0, m = 0.0;
    for (int k = k0; k <= k1; ++k) {
        double uc = 0.0, up = 0.0, vj = 0.0, vjp = 0.0, wkp = 0.0;
        if (act) {
            uc = us[d.g(i, j, k)];
            if (fs.part) uc = uc + du;
            vj = wrap && j == 1 ? 0.0 : vs[d.g(i, j, k)];
            vjp = wrap && j == d.ny ? 0.0 : vs[d.g(i, j + 1, k)];
            wkp = ws[d.g(i, j, wrap && k == d.nz ? 1 : k + 1)];
        }
        up = __shfl_down(uc, 1, 64);
        if (act && (lane == 63 || i == d.nx)) {
            up = us[d.g(wrap && i == d.nx ? 1 : i + 1, j, k)];
            if (fs.part) up = up + du;
        }
        if (act) {
            const double dv = STRETCH ? (vjp - vj) * g.ihc[j] : (vjp - vj) / g.dy;
            const double r = ((up - uc) / g.dx + dv + (wkp - wk) / g.dz) / dtg;
            rhs[(size_t)(i - 1) + (size_t)d.nx * ((size_t)(k - 1) + (size_t)d.nz * (size_t)(j - 1))] = r;
            m = nanmax_any(m, fabs(r));
        }
        wk = wkp;
    }
    block_max_part(m, part);
}

// partial sums of the (nx, nz) planes: workgroup (plane j, chunk c) sums chunk c of PLANE_CHUNKS
// equal parts of plane j into part[j * PLANE_CHUNKS + c]; consumers fold a plane's chunks in order
__global__ __launch_bounds__(256) void fft_plane_sum_kernel(Dims d, const double *__restrict__ rhs, double *part) {
    __shared__ double s[256];
    const long plane = (long)d.nx * d.nz;
    const int j = blockIdx.x / PLANE_CHUNKS, c = blockIdx.x % PLANE_CHUNKS;
    const long lo = plane * c / PLANE_CHUNKS, hi = plane * (c + 1) / PLANE_CHUNKS;
    const double *p = rhs + plane * j;
    double a = 0.0;
    for (long q = lo + threadIdx.x; q < hi; q += 256) a += p[q];
    s[threadIdx.x] = a;
    __syncthreads();
    for (int w = 128; w > 0; w >>= 1) {
        if (threadIdx.x < w) s[threadIdx.x] += s[threadIdx.x + w];
        __syncthreads();
    }
    if (threadIdx.x == 0) part[blockIdx.x] = s[0];
}

// the kx = kz = 0 line of tridiag_kernel in FP64 on the plane sums; mean[j-1] = x_j / (nx nz).
// The operands are staged in LDS first, so the sequential recurrences do not wait on global memory.
static constexpr int MEAN_MAX_NY = 1024;   // 40 KB of LDS
__global__ __launch_bounds__(256) void fft_mean_mode_kernel(Dims d, const double *__restrict__ part,
                                                            const double *__restrict__ cp,
                                                            const double *__restrict__ den_inv,
                                                            const double *__restrict__ arow, double scale,
                                                            double *mean) {
    __shared__ double ss[MEAN_MAX_NY], sa[MEAN_MAX_NY], sd[MEAN_MAX_NY], sc[MEAN_MAX_NY], sm[MEAN_MAX_NY];
    const int ny = d.ny;
    const size_t cs = (size_t)(d.nx / 2 + 1);   // stride between j of line (0, 0) in cp / den_inv
    for (int q = threadIdx.x; q < ny; q += 256) {
        ss[q] = plane_sum(part, q);
        sa[q] = arow[q];
        sd[q] = den_inv[cs * q];
        sc[q] = cp[cs * q];
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        double dp = 0.0;
        sm[0] = 0.0;
        for (int jj = 2; jj <= ny; ++jj) {
            dp = (ss[jj - 1] - sa[jj - 1] * dp) * sd[jj - 1];
            sm[jj - 1] = dp;
        }
        double nxt = dp;
        sm[ny - 1] = nxt * scale;
        for (int jj = ny - 1; jj >= 1; --jj) {
            nxt = sm[jj - 1] - sc[jj - 1] * nxt;
            sm[jj - 1] = nxt;
        }
        for (int jj = 1; jj < ny; ++jj) sm[jj - 1] *= scale;
    }
    __syncthreads();
    for (int q = threadIdx.x; q < ny; q += 256) mean[q] = sm[q];
}

// max |rhs - L phi| (FP64) per workgroup, and with STORE the residual itself, which only a further pass
// reads; layout (nx, nz, ny), x and z periodic.  A thread takes a column (i, k) of a 64 x 4 tile and
// marches jm rows, FR_CH rows' loads in flight and phi(j-1), phi(j) in registers.  Bound by HBM: 16 B
// per cell, 24 with STORE (256 x 192 x 256: 121 us before, a thread per cell with 64-bit index divisions
// and always storing; 51 and 68 now).
static constexpr int FR_CH = 4;
template <bool STRETCH, bool STORE>
__global__ __launch_bounds__(256) void fft_residual_kernel(GridK g, const double *__restrict__ rhs,
                                                           const double *__restrict__ phi, const double *__restrict__ arow,
                                                           int jm, double *__restrict__ res, double *part) {
    const Dims d = g.d;
    const int nx = d.nx, ny = d.ny, nz = d.nz;
    const int i0 = blockIdx.x * 64 + threadIdx.x, k0 = blockIdx.y * 4 + threadIdx.y;   // 0-based
    const bool act = i0 < nx && k0 < nz;
    const int i = act ? i0 : 0, k = act ? k0 : 0;
    const int j0 = blockIdx.z * jm, j1 = j0 + jm < ny ? j0 + jm : ny;
    const double idx2 = 1.0 / (g.dx * g.dx), idz2 = 1.0 / (g.dz * g.dz);
    const ptrdiff_t sp = (ptrdiff_t)nx * nz;
    const ptrdiff_t xp = i + 1 == nx ? 1 - nx : 1, xm = i == 0 ? nx - 1 : -1;
    const ptrdiff_t zp = k + 1 == nz ? (ptrdiff_t)nx * (1 - nz) : nx, zm = k == 0 ? (ptrdiff_t)nx * (nz - 1) : -(ptrdiff_t)nx;
    const size_t q0 = (size_t)i + (size_t)nx * ((size_t)k + (size_t)nz * (size_t)j0);
    const double *p = phi + q0, *f = rhs + q0;
    double m = 0.0, pm = j0 > 0 ? p[-sp] : 0.0, p0 = p[0];
    for (int j = j0; j < j1; j += FR_CH, p += FR_CH * sp, f += FR_CH * sp) {
        double py[FR_CH], a[FR_CH], b[FR_CH], c[FR_CH], e[FR_CH], r[FR_CH];
#pragma unroll
        for (int u = 0; u < FR_CH; ++u) {   // past the end: the last row again, unused
            const int w = j + u < j1 ? u : j1 - 1 - j;
            const double *q = p + w * sp;
            a[u] = q[xp];
            b[u] = q[xm];
            c[u] = q[zp];
            e[u] = q[zm];
            r[u] = f[w * sp];
            py[u] = j + w + 1 < ny ? q[sp] : 0.0;
        }
#pragma unroll
        for (int u = 0; u < FR_CH; ++u) {
            const int jj = j + u;
            if (jj >= j1) break;
            double ly = 0.0;
            if (jj > 0) ly += arow[jj] * (pm - p0);
            if (jj < ny - 1) ly += (STRETCH ? g.ihv[jj + 2] * g.ihc[jj + 1] : arow[jj + 1]) * (py[u] - p0);
            const double lap = (a[u] - 2.0 * p0 + b[u]) * idx2 + (c[u] - 2.0 * p0 + e[u]) * idz2 + ly;
            const double rr = r[u] - lap;
            if (STORE && act) res[q0 + (size_t)(jj - j0) * sp] = rr;
            m = nanmax_any(m, fabs(rr));
            pm = p0;
            p0 = py[u];
        }
    }
    block_max_part(act ? m : 0.0, part);
}

// 1. (FP32) r2c x-transform of a real FP64 field in (nx, nz, ny) layout
__global__ __launch_bounds__(FFT_THREADS) void xfft32_kernel(Dims d, const double *__restrict__ in,
                                                             const float2 *__restrict__ tw, int lines, int stride,
                                                             float2 *hat) {
    extern __shared__ __align__(16) unsigned char lds_raw[];
    float2 *lds = reinterpret_cast<float2 *>(lds_raw);
    const int n = d.nx, nxh = n / 2 + 1;
    const int nrows = d.ny * d.nz;
    float2 *a = lds, *b = lds + (size_t)lines * n, *twl = b + (size_t)lines * n;
    stage_twiddles(twl, tw, n);
    for (int t = threadIdx.x; t < lines * n; t += FFT_THREADS) {
        const int line = t / n, i = t - line * n;
        const int r = blockIdx.x * lines + line;
        a[t] = make_float2(r < nrows ? (float)in[(size_t)n * r + i] : 0.f, 0.f);
    }
    __syncthreads();
    float2 *res = stockham(a, b, n, lines, n, twl, false, threadIdx.x, FFT_THREADS);
    for (int t = threadIdx.x; t < lines * nxh; t += FFT_THREADS) {
        const int line = t / nxh, m = t - line * nxh;
        const int r = blockIdx.x * lines + line;
        if (r < nrows) hat[(size_t)stride * r + m] = res[line * n + m];
    }
}

// 3. (FP32) Thomas per (kx, kz) line with FP32 tables; the mean mode line is set to zero (it is
//    solved in FP64 separately)
__global__ __launch_bounds__(64) void tridiag32_kernel(Dims d, int stride, float2 *hat, const float *__restrict__ cp,
                                                       const float *__restrict__ den_inv,
                                                       const float *__restrict__ arow) {
    const int nxh = d.nx / 2 + 1, ny = d.ny, nz = d.nz;
    const int t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= nxh * nz) return;
    const int kx = t % nxh, kz = t / nxh;
    const size_t hs = (size_t)stride * nz, cs = (size_t)nxh;
    const size_t h0 = (size_t)kx + (size_t)stride * kz;
    const size_t c0 = (size_t)kx + (size_t)nxh * (size_t)ny * kz;
    if (kx == 0 && kz == 0) {
        for (int jj = 1; jj <= ny; ++jj) hat[h0 + hs * (jj - 1)] = make_float2(0.f, 0.f);
        return;
    }
    float2 dp;
    {
        const float2 r = hat[h0];
        const float di = den_inv[c0];
        dp = make_float2(r.x * di, r.y * di);
    }
    hat[h0] = dp;
    for (int jb = 2; jb <= ny; jb += TB) {
        float2 rr[TB];
        float aa[TB], dd[TB];
#pragma unroll
        for (int q = 0; q < TB; ++q) {
            const int jj = jb + q;
            if (jj <= ny) {
                rr[q] = hat[h0 + hs * (jj - 1)];
                aa[q] = arow[jj - 1];
                dd[q] = den_inv[c0 + cs * (jj - 1)];
            }
        }
#pragma unroll
        for (int q = 0; q < TB; ++q) {
            const int jj = jb + q;
            if (jj <= ny) {
                dp = make_float2((rr[q].x - aa[q] * dp.x) * dd[q], (rr[q].y - aa[q] * dp.y) * dd[q]);
                hat[h0 + hs * (jj - 1)] = dp;
            }
        }
    }
    float2 nxt = dp;
    for (int jb = ny - 1; jb >= 1; jb -= TB) {
        float2 qq[TB];
        float cc[TB];
#pragma unroll
        for (int q = 0; q < TB; ++q) {
            const int jj = jb - q;
            if (jj >= 1) {
                qq[q] = hat[h0 + hs * (jj - 1)];
                cc[q] = cp[c0 + cs * (jj - 1)];
            }
        }
#pragma unroll
        for (int q = 0; q < TB; ++q) {
            const int jj = jb - q;
            if (jj >= 1) {
                nxt = make_float2(qq[q].x - cc[q] * nxt.x, qq[q].y - cc[q] * nxt.y);
                hat[h0 + hs * (jj - 1)] = nxt;
            }
        }
    }
}

// 5. (FP32) c2r x-transform, scaled, and the mean mode's solution added to the FP64 phi (first: to zero)
__global__ __launch_bounds__(FFT_THREADS) void ixfft32_add_kernel(Dims d, const float2 *__restrict__ hat,
                                                                  const float2 *__restrict__ tw, int lines, int stride,
                                                                  float scale, const double *__restrict__ mean, int first,
                                                                  double *phi) {
    extern __shared__ __align__(16) unsigned char lds_raw[];
    float2 *lds = reinterpret_cast<float2 *>(lds_raw);
    const int n = d.nx, nxh = n / 2 + 1;
    const int nrows = d.ny * d.nz;
    float2 *a = lds, *b = lds + (size_t)lines * n, *twl = b + (size_t)lines * n;
    stage_twiddles(twl, tw, n);
    for (int t = threadIdx.x; t < lines * n; t += FFT_THREADS) {
        const int line = t / n, m = t - line * n;
        const int r = blockIdx.x * lines + line;
        float2 v = make_float2(0.f, 0.f);
        if (r < nrows) {
            const float2 *row = hat + (size_t)stride * r;
            if (m == 0 || 2 * m == n) v = make_float2(row[m].x, 0.f);
            else if (m < nxh) v = row[m];
            else v = make_float2(row[n - m].x, -row[n - m].y);
        }
        a[t] = v;
    }
    __syncthreads();
    float2 *res = stockham(a, b, n, lines, n, twl, true, threadIdx.x, FFT_THREADS);
    for (int t = threadIdx.x; t < lines * n; t += FFT_THREADS) {
        const int line = t / n, i = t - line * n;
        const int r = blockIdx.x * lines + line;
        if (r < nrows) {
            const double p = (first ? 0.0 : phi[(size_t)n * r + i]) + mean[r / d.nz];
            phi[(size_t)n * r + i] = p + (double)(res[t].x * scale);
        }
    }
}

// the FP64 right-hand side -> h->fft_rhs; its max |.| into the max reduction
hipError_t launch_fft_mixed_setup(mdx_handle *h, double dtg, double *host_slot, unsigned long long seq) {
    GridK g = grid_k(h);
    const Dims d = h->d;
    dim3 blk(64, FC_Y), grd((d.nx + 63) / 64, (d.ny + FC_Y - 1) / FC_Y, (d.nz + FC_KZ - 1) / FC_KZ);
#define MDX_RHS(S)                                                                                              \
    hipLaunchKernelGGL(fft_div_rhs_kernel<S>, grd, blk, 0, h->stream, g, h->us, h->vs, h->ws, dtg, fft_wrap(h), \
                       fft_step(h), h->fft_rhs, h->max_part)
    if (h->stretched) MDX_RHS(true);
    else MDX_RHS(false);
#undef MDX_RHS
    const hipError_t e = hipGetLastError();
    return e != hipSuccess ? e : launch_max_final(h, grd.x * grd.y * grd.z, host_slot, seq);
}

// max |rhs - L phi| into the max reduction, or (store) the residual into h->fft_res
hipError_t launch_fft_residual(mdx_handle *h, bool store, double *host_slot, unsigned long long seq) {
    GridK g = grid_k(h);
    const Dims d = h->d;
    int jm = 16;   // rows per workgroup, fewer while that leaves CUs without four workgroups
    auto groups = [&](int m) { return (unsigned)((d.nx + 63) / 64 * ((d.nz + 3) / 4) * ((d.ny + m - 1) / m)); };
    while (jm > FR_CH && groups(jm) < 1024) jm /= 2;
    const dim3 grd((d.nx + 63) / 64, (d.nz + 3) / 4, (d.ny + jm - 1) / jm);
#define MDX_RES(S, T)                                                                                           \
    hipLaunchKernelGGL((fft_residual_kernel<S, T>), grd, dim3(64, 4), 0, h->stream, g, h->fft_rhs, h->fft_phi,  \
                       h->arow, jm, h->fft_res, h->max_part)
    if (h->stretched) { if (store) MDX_RES(true, true); else MDX_RES(true, false); }
    else { if (store) MDX_RES(false, true); else MDX_RES(false, false); }
#undef MDX_RES
    const hipError_t e = hipGetLastError();
    return e != hipSuccess || store ? e : launch_max_final(h, groups(jm), host_slot, seq);
}

// the FP32 x-transforms of the defect solves
static hipError_t launch_xfft32(mdx_handle *h, const double *res) {
    const Dims d = h->d;
    const int stride = fft_stride_t<float2>(d.nx);
#define XF_(N, TH)                                                                                               \
    return rf_launch<float2, N, TH, xfft32_reg_kernel<N, TH>>(h->stream, rf_row_blocks<N, TH>(d, 1), d,          \
                                                              res,                                               \
                                                              (const float2 *)h->tw_x32, stride, (float2 *)h->hat32)
#define XF(N)                                                \
    if (rf_small(rf_row_blocks<N, 256>(d, 1))) XF_(N, 64);   \
    XF_(N, 256)
    RF_SIZES(d.nx, XF)
#undef XF
#undef XF_
    const int lines = rows_per_block(d.nx), nrows = d.ny * d.nz;
    hipLaunchKernelGGL(xfft32_kernel, dim3((nrows + lines - 1) / lines), dim3(FFT_THREADS),
                       fft_lds<float2>(lines, d.nx, d.nx), h->stream, d, res, (const float2 *)h->tw_x32, lines,
                       stride, (float2 *)h->hat32);
    return hipGetLastError();
}

static hipError_t launch_ixfft32_add(mdx_handle *h, const double *mean, bool first) {
    const Dims d = h->d;
    const int stride = fft_stride_t<float2>(d.nx);
    const float scale = 1.0f / (float)(d.nx * d.nz);
#define IX_(N, TH, FIRST)                                                                                        \
    return rf_launch<float2, N, TH, ixfft32_add_reg_kernel<N, TH, FIRST>>(h->stream, rf_row_blocks<N, TH>(d, 1), \
                                                                          d, (const float2 *)h->hat32,           \
                                                                          (const float2 *)h->tw_x32, stride,     \
                                                                          scale, mean, h->fft_phi)
#define IX(N)                                                \
    if (rf_small(rf_row_blocks<N, 256>(d, 1))) {             \
        if (first) IX_(N, 64, true);                         \
        IX_(N, 64, false);                                   \
    }                                                        \
    if (first) IX_(N, 256, true);                            \
    IX_(N, 256, false)
    RF_SIZES(d.nx, IX)
#undef IX
#undef IX_
    const int lines = rows_per_block(d.nx), nrows = d.ny * d.nz;
    hipLaunchKernelGGL(ixfft32_add_kernel, dim3((nrows + lines - 1) / lines), dim3(FFT_THREADS),
                       fft_lds<float2>(lines, d.nx, d.nx), h->stream, d, (const float2 *)h->hat32,
                       (const float2 *)h->tw_x32, lines, stride, scale, mean, (int)first, h->fft_phi);
    return hipGetLastError();
}

// one defect-correction pass on res = rhs - L phi (first: phi = 0 and res = rhs): the mean mode in FP64
// (plane sums, pinned Thomas), the other modes by FP32 transforms and Thomas; both corrections added
// to h->fft_phi
hipError_t launch_fft32_solve_add(mdx_handle *h, bool first) {
    const Dims d = h->d;
    if (d.ny > MEAN_MAX_NY) return hipErrorInvalidValue;
    const double *res = first ? h->fft_rhs : h->fft_res;
    hipLaunchKernelGGL(fft_plane_sum_kernel, dim3(d.ny * PLANE_CHUNKS), dim3(256), 0, h->stream, d, res, h->fft_mean);
    double *mean = h->fft_mean + (size_t)d.ny * PLANE_CHUNKS;
    hipLaunchKernelGGL(fft_mean_mode_kernel, dim3(1), dim3(256), 0, h->stream, d, h->fft_mean, h->cp, h->den_inv,
                       h->arow, 1.0 / (double)(d.nx * d.nz), mean);
    hipError_t e = launch_xfft32(h, res);
    if (e != hipSuccess) return e;
    if ((e = launch_zfft<float2, false>(h->stream, d, (float2 *)h->hat32, (const float2 *)h->tw_z32)) != hipSuccess)
        return e;
    const int nlines = (d.nx / 2 + 1) * d.nz;
    if (!(h->wave_tridiag && h->part_tridiag &&
          launch_tridiag_part<float2, true>(h->stream, d, (float2 *)h->hat32, h->lamx32, h->lamz32, h->tw_a32,
                                            h->bdrow32, h->crow32)) &&
        !(h->wave_tridiag && launch_tridiag_wave<float2, true>(h->stream, d, (float2 *)h->hat32, h->lamx32, h->lamz32,
                                                     h->tw_a32, h->bdrow32, h->crow32)))
        hipLaunchKernelGGL(tridiag32_kernel, dim3((nlines + 63) / 64), dim3(64), 0, h->stream, d,
                           fft_stride_t<float2>(d.nx), (float2 *)h->hat32, h->cp32, h->den32, h->arow32);
    if ((e = launch_zfft<float2, true>(h->stream, d, (float2 *)h->hat32, (const float2 *)h->tw_z32)) != hipSuccess)
        return e;
    return launch_ixfft32_add(h, mean, first);
}

// the plane sums of phi in plane 1: the mean that launch_fft_correct takes off phi, which re-imposes the
// pin phi_hat(y_1) = 0 exactly (the FP32 inverse transforms leave plane means of the order of their
// rounding, and a constant is invisible to the residual; velocities see only differences)
hipError_t launch_fft_pin(mdx_handle *h) {
    hipLaunchKernelGGL(fft_plane_sum_kernel, dim3(PLANE_CHUNKS), dim3(256), 0, h->stream, h->d, h->fft_phi, h->fft_mean);
    return hipGetLastError();
}

// the projection with the FP64 phi of the defect correction (step 6); pin: less its mean in plane 1
hipError_t launch_fft_correct(mdx_handle *h, double dtg, bool pin) {
    return launch_correct(h, h->fft_phi, dtg, pin ? h->fft_mean : nullptr);
}

}  // namespace mdx
