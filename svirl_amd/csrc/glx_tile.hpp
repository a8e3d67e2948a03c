// TDGL time steps on register tiles: grids whose nodes fit in the registers
// of the chip are swept without re-reading the fields from memory.
//
// A workgroup of NW waves owns one tile: 64 columns (one per lane)
// by NW * NR rows, wave w holding rows w*NR .. w*NR + NR-1 of its
// lanes' columns in registers, with the outer H columns and rows a halo of
// the neighbouring tiles. A Jacobi sweep is straight-line code over a lane's
// NR nodes: the lateral neighbours come from the adjacent lanes (DPP shifts),
// the vertical ones from the lane's own registers, and the rows above and
// below a wave's rows from its neighbour waves through LDS. Values beyond
// the tile are unknown, so each sweep spoils one more ring of halo; after up
// to H sweeps the tiles exchange rings through memory (neighbours only) and
// go on. Link factors, right-hand sides and diagonals stay in registers for
// the whole solve, and one launch runs all steps of a run.
//
// The FP64 arithmetic is that of the row-marching passes (psi_rows, a_rows):
// results and every sweep count equal theirs to the bit.
//
// FP32 psi solves carry, from their sweep PSI_TURN on, the change d of a sweep
// and the sum D of the changes instead of psi and its right-hand side: the
// solve is linear in psi, so d' = M d, and psi^{n+1} is the iterate at the
// turn plus D. That costs the same registers and instructions, D is rounded at
// the size of the changes that are left, and the stop rule's 1e-6 is tested on
// values whose own rounding is 1e-13, where the difference of two rounded
// iterates is off by up to 1e-7 and makes about 2 of 100 solves go a sweep too
// far. The first sweeps carry psi itself because a step may shrink psi by
// much (4 times a step where A outgrows the vortices): changes summed from
// psi^n are rounded at its size, not psi^{n+1}'s, and after 20 such steps the
// error against 64 bits was 1.6 times that of the row-marching solves, which
// carry psi throughout (513^2: 5.8e-7 against 3.4e-7; with the turn 3.5e-7).
// Over 70 runs of 10 steps on 65 x 65 to 1025 x 1025: tiles 2.4e-7 at most and
// 2.0e-7 in the mean, no sweep count off; rows 8.2e-7, 2.5e-7 and 19 of 700 off.
#pragma once

#include "glx_td.hpp"

namespace glx {

// A FP32 psi solve carries changes from this sweep on; from its first one if
// the previous step took PSI_FEW sweeps or fewer (psi hardly changes then,
// and the stop rule is met among the first sweeps).
constexpr int PSI_TURN = 2, PSI_FEW = 4;

// A tile shape: NW waves of NR rows each, halo H.
template <int NR_, int H_, int NW_> struct TileOf {
    static constexpr int NR = NR_, H = H_, NW = NW_;
    static constexpr int COLS = WAVE - 2 * H, ROWS = NW * NR - 2 * H;  // of the tile's own
    static_assert(NW >= 4 && H <= NR && ROWS > 0, "tile shape");
};

// What the tiles of one instance need to meet: a flag word per workgroup
// (epoch of its last published ring), check words and group words (epoch <<
// 32 | unconverged-sweep bits), two arrays of each used in turn, and the
// error flag.
struct TileSync {
    unsigned long long *flag, *chk[2], *grp[2];
    int *err;
};

// The workgroup's tile: (tx, ty) of ntx x nty = nwg; the instance's words
// start at flag, chk[.] + base and grp[.] + gbase.
struct TileTeam {
    int base, gbase, nwg, tx, ty, ntx, nty;
};

template <typename R, typename SH> struct TileLds {
    static constexpr int NR = SH::NR, NW = SH::NW;
    // first and last rows of every wave (slots 2 w + 1 and 2 w + 2) between
    // two rows of zeros that stand for what lies beyond the tile, two copies
    // used in turn
    cplx<R> edge[2][2 * NW + 2][WAVE];
    // FP64: the right-hand side and the diagonal of every node (each lane
    // reads its own)
    static constexpr int KW = std::is_same<R, double>::value ? NW : 1;
    static constexpr int KR = std::is_same<R, double>::value ? NR : 1;
    cplx<R> rhs[KW][KR][WAVE];
    R den[KW][KR][WAVE];
    // FP32: the right-hand side of every node up to the turn, psi at the turn
    // from there on
    static constexpr int TW = std::is_same<R, double>::value ? 1 : NW;
    static constexpr int TR = std::is_same<R, double>::value ? 1 : NR;
    cplx<R> base[TW][TR][WAVE];
    unsigned bits[NW], all;
    int fail;
};

// ---- memory the tiles share: written through, read past the caches ---------
__device__ __forceinline__ void st_shared_mem(float *p, float v) {
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void st_shared_mem(double *p, double v) {
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void st_shared_mem(cplx<float> *p, cplx<float> v) {
    unsigned long long u = ((unsigned long long)__float_as_uint(v.im) << 32) | __float_as_uint(v.re);
    __hip_atomic_store(reinterpret_cast<unsigned long long *>(p), u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void st_shared_mem(cplx<double> *p, cplx<double> v) {
    st_shared_mem(&p->re, v.re);
    st_shared_mem(&p->im, v.im);
}
template <typename R> __device__ __forceinline__ R ld_shared_mem(const R *p) {
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ cplx<float> ld_shared_mem(const cplx<float> *p) {
    const unsigned long long u = ld_relaxed(reinterpret_cast<const unsigned long long *>(p));
    return {__uint_as_float((unsigned)u), __uint_as_float((unsigned)(u >> 32))};
}
__device__ __forceinline__ cplx<double> ld_shared_mem(const cplx<double> *p) {
    return {ld_shared_mem(&p->re), ld_shared_mem(&p->im)};
}

// A uniform (scalar register) or per-lane value that the compiler cannot
// trace: what is derived from it is formed where it is used, not hoisted
// out of the step loop. The masks and addresses of every row of a tile,
// each a register pair, would otherwise all be kept through the sweeps.
__device__ __forceinline__ int fresh_s(int x) {
    asm volatile("" : "+s"(x));
    return x;
}
__device__ __forceinline__ int fresh_v(int x) {
    asm volatile("" : "+v"(x));
    return x;
}

template <typename R> __device__ __forceinline__ R fresh_r(R x) {
    asm volatile("" : "+v"(x));
    return x;
}

// A copy of *p through the scalar cache, from a pointer laundered like
// fresh_s: the phases of a step each load the arguments they use, instead
// of keeping all of them in scalar registers through the step loop. *p is
// constant while the kernel runs.
template <typename T> __device__ __forceinline__ T fresh_args(const T *p) {
    static_assert(sizeof(T) % 4 == 0, "copied as words");
    uint64_t a = reinterpret_cast<uint64_t>(p);
    asm volatile("" : "+s"(a));
    typedef const __attribute__((address_space(4))) uint32_t *Words;
    const Words w = (Words)a;
    T v;
    uint32_t *d = reinterpret_cast<uint32_t *>(&v);
#pragma unroll
    for (unsigned k = 0; k < sizeof(T) / 4; ++k) d[k] = w[k];
    return v;
}

// One argument field through the scalar cache. What the tiles branch on
// and index with (these, buffer indices, the words of a meeting) is made
// uniform explicitly: read from memory or LDS like lane data it would turn
// every loop of a solve into one over execution masks.
template <typename T> __device__ __forceinline__ T arg(const T *p) {
    return *(const __attribute__((address_space(4))) T *)(uintptr_t)p;
}
__device__ __forceinline__ int uniform(int x) { return __builtin_amdgcn_readfirstlane(x); }

// x where bit r of `on` is set, else 0.
__device__ __forceinline__ float tile_mask(float x, unsigned on, int r) {
    const int m = -(int)((on >> r) & 1u);
    return __int_as_float(__float_as_int(x) & m);
}
__device__ __forceinline__ double tile_mask(double x, unsigned on, int r) {
    const long long m = -(int)((on >> r) & 1u);
    return __longlong_as_double(__double_as_longlong(x) & m);
}

// Column and row context of a lane in its tile.
struct TileCtx {
    int c, lane;  // the lane's column, its index
    int j0, w;    // the global row of the wave's row 0, the wave's index
    __device__ __forceinline__ TileCtx fresh() const { return {fresh_v(c), fresh_v(lane), fresh_s(j0), fresh_s(w)}; }
    __device__ __forceinline__ bool first() const { return w == 0; }  // the wave at the tile's top / bottom
    template <typename SH> __device__ __forceinline__ bool last() const { return w == SH::NW - 1; }
    // the column, its a links exist; the column belongs to this tile
    __device__ __forceinline__ bool col(int Nx) const { return (unsigned)c < (unsigned)Nx; }
    __device__ __forceinline__ bool hasa(int Nx) const { return (unsigned)c < (unsigned)(Nx - 1); }
    template <typename SH> __device__ __forceinline__ bool own(int Nx) const {
        return col(Nx) && lane >= SH::H && lane < WAVE - SH::H;
    }
    // column clamped to the nodes / to the a links
    __device__ __forceinline__ uint32_t cc(int Nx) const { return (uint32_t)min(max(c, 0), Nx - 1); }
    __device__ __forceinline__ uint32_t ca(int Nx) const { return (uint32_t)min(max(c, 0), Nx - 2); }
    // the wave's rows [r0, r1) that belong to this tile
    template <typename SH> __device__ __forceinline__ int r0() const { return max(first() ? SH::H : 0, -j0); }
    template <typename SH> __device__ __forceinline__ int r1(int Ny) const {
        return min(last<SH>() ? SH::NR - SH::H : SH::NR, Ny - j0);
    }
};

template <typename SH> __device__ __forceinline__ TileCtx tile_ctx(int tx, int ty) {
    const int lane = threadIdx.x & (WAVE - 1), w = wave_id();
    return {tx * SH::COLS - SH::H + lane, lane, ty * SH::ROWS - SH::H + w * SH::NR, w};
}

// sincos_r with its FP64 constants read from memory through the scalar cache
// (the same values, so the same results): as literals they are loaded into
// some forty registers ahead of the step loop and kept there.
struct SinCosTab {
    double k[22];
};
__device__ const SinCosTab sincos_tab = {{
    0.6366197723675814, 1.5707963267341256, 6.077100506303966e-11, 2.0222662487959506e-21,
    1.0 / 355687428096000.0, -1.0 / 1307674368000.0, 1.0 / 6227020800.0, -1.0 / 39916800.0, 1.0 / 362880.0,
    -1.0 / 5040.0, 1.0 / 120.0, -1.0 / 6.0,
    -1.0 / 6402373705728000.0, 1.0 / 20922789888000.0, -1.0 / 87178291200.0, 1.0 / 479001600.0, -1.0 / 3628800.0,
    1.0 / 40320.0, -1.0 / 720.0, 1.0 / 24.0, -0.5, 1.0}};
template <typename R> struct TileSinCos {
    __device__ __forceinline__ void load() {}
    __device__ __forceinline__ void operator()(R x, R *s, R *c) const { sincos_r(x, s, c); }
};
template <> struct TileSinCos<double> {
    SinCosTab t;
    __device__ __forceinline__ void load() { t = fresh_args(&sincos_tab); }
    __device__ __forceinline__ void operator()(double x, double *s, double *c) const {
        const double k = rint(x * t.k[0]);
        double r = fma(-k, t.k[1], x);
        r = fma(-k, t.k[2], r);
        r = fma(-k, t.k[3], r);
        const double z = r * r;
        double ps = t.k[4];
#pragma unroll
        for (int n = 5; n < 12; ++n) ps = fma(ps, z, t.k[n]);
        const double sr = fma(r * z, ps, r);
        double pc = t.k[12];
#pragma unroll
        for (int n = 13; n < 21; ++n) pc = fma(pc, z, t.k[n]);
        const double cr = fma(z, pc, t.k[21]);
        const int q = (int)((long long)k & 3);
        const double sv = (q & 1) ? cr : sr, cv = (q & 1) ? sr : cr;
        *s = (q & 2) ? -sv : sv;
        *c = ((q + 1) & 2) ? -cv : cv;
    }
};

// The lane's part of a psi solve: psi, the link factors of a(c, j) and
// b(c, j) (FP32: scaled by dt/dx^2, dt/dy^2; zero where the link touches no
// material), those of b above row 0, and the diagonals. FP32 keeps
// 1/den, and psi in p and rhs/den in rd up to the turn, from there on the
// change of the last sweep in p and the sum of all in rd; FP64 1/den and, in
// LDS, rhs and den.
template <typename R, typename SH> struct PsiTile {
    static constexpr int NR = SH::NR;
    cplx<R> p[NR], rd[NR];
    R ca[NR], sa[NR], cb[NR], sb[NR];
    R cbu, sbu;
    R rden[NR];
    unsigned ena, enb;  // bit r: a(c, j) / b(c, j) touches the material
};

// Row j of an array of n rows of `stride` elements, j clamped into it.
template <typename T> __device__ __forceinline__ const T *tile_row(const T *p, int j, int n, int stride) {
    return p + (size_t)stride * (size_t)(uint32_t)min(max(j, 0), n - 1);
}

// The material flag of cell (c, j) from its mask byte (0 outside the grid).
__device__ __forceinline__ bool tile_cell(bool has_mt, int byte, bool hasa, int j, int Ny) {
    return hasa && j >= 0 && j < Ny - 1 && (!has_mt || byte != 0);
}

// The link factors of the tile from the vector potential ab.
template <typename R, bool GAUGE, typename SH>
__device__ __forceinline__ void tile_links(const PsiSweepArgs<R> *Ap, const R *ab, const TileCtx &X0, PsiTile<R, SH> &t) {
    constexpr int NR = SH::NR;
    constexpr bool FOLD = std::is_same<R, float>::value;
    const PsiSweepArgs<R> A = fresh_args(Ap);
    const TileCtx X = X0.fresh();
    const int Nx = A.Nx, Ny = A.Ny, Nxa = Nx - 1;
    const R *b = ab + (size_t)Nxa * Ny;
    const bool has_mt = A.mt != nullptr, hasa = X.hasa(Nx);
    const uint8_t *mtp = has_mt ? A.mt : reinterpret_cast<const uint8_t *>(ab);  // any readable bytes
    const uint32_t ca = X.ca(Nx), oa = ca * (uint32_t)sizeof(R), ob = X.cc(Nx) * (uint32_t)sizeof(R);
    const R gb = GAUGE ? gauge_phase_b<R>(A, X.c) : R(0);
    const R kxa = FOLD ? A.dt * A.idx2 : R(1), kyb = FOLD ? A.dt * A.idy2 : R(1);
    TileSinCos<R> sincos;
    sincos.load();
    auto byte_at = [&](int j) { return (int)at(tile_row(mtp, j, Ny - 1, Nxa), ca); };
    auto b_link = [&](R v, bool on, R &cv, R &sv) {
        sincos(link_phase<R, GAUGE>(A.dy, v, gb), &sv, &cv);
        mask_link(on, cv, sv);
        if constexpr (FOLD) {
            cv *= kyb;
            sv *= kyb;
        }
    };
    R av[NR], bv[NR];
    int mc[NR];
    const R bu = at(tile_row(b, X.j0 - 1, Ny - 1, Nx), ob);
    const int mu = byte_at(X.j0 - 1);
#pragma unroll
    for (int r = 0; r < NR; ++r) {
        av[r] = at(tile_row(ab, X.j0 + r, Ny, Nxa), oa);
        bv[r] = at(tile_row(b, X.j0 + r, Ny - 1, Nx), ob);
        mc[r] = byte_at(X.j0 + r);
    }
    bool cellm = tile_cell(has_mt, mu, hasa, X.j0 - 1, Ny);
    b_link(bu, shfl_up1((int)cellm) != 0 || cellm, t.cbu, t.sbu);
    t.ena = t.enb = 0u;
#pragma unroll
    for (int r = 0; r < NR; ++r) {
        const int j = X.j0 + r;
        const bool cellc = tile_cell(has_mt, mc[r], hasa, j, Ny);
        const bool ona = cellm || cellc, onb = shfl_up1((int)cellc) != 0 || cellc;
        sincos(link_phase<R, GAUGE>(A.dx, av[r], GAUGE ? gauge_phase_a<R>(A, j) : R(0)), &t.sa[r], &t.ca[r]);
        mask_link(ona, t.ca[r], t.sa[r]);
        if constexpr (FOLD) {
            t.ca[r] *= kxa;
            t.sa[r] *= kxa;
        }
        b_link(bv[r], onb, t.cb[r], t.sb[r]);
        t.ena |= ona ? 1u << r : 0u;
        t.enb |= onb ? 1u << r : 0u;
        cellm = cellc;
        __builtin_amdgcn_sched_barrier(0);
    }
}

// psi of the tile from a state buffer, with the right-hand sides and
// diagonals of a step that starts there.
template <typename R, typename SH>
__device__ __forceinline__ void tile_psi_load(const PsiSweepArgs<R> *Ap, const cplx<R> *psi, const TileCtx &X0,
                                              PsiTile<R, SH> &t, TileLds<R, SH> &S) {
    constexpr int NR = SH::NR;
    constexpr bool FOLD = std::is_same<R, float>::value;
    const PsiSweepArgs<R> A = fresh_args(Ap);
    const TileCtx X = X0.fresh();
    const int Nx = A.Nx, Ny = A.Ny, Nxa = Nx - 1;
    const bool has_mt = A.mt != nullptr, hasa = X.hasa(Nx), col = X.col(Nx), has_em = A.eps_map != nullptr;
    const uint8_t *mtp = has_mt ? A.mt : reinterpret_cast<const uint8_t *>(psi);  // any readable bytes
    const R *emp = has_em ? A.eps_map : reinterpret_cast<const R *>(psi);          // when absent
    const uint32_t ca = X.ca(Nx), oc = X.cc(Nx) * (uint32_t)sizeof(R);
    R ev[NR];
    int mc[NR];
    const int mu = (int)at(tile_row(mtp, X.j0 - 1, Ny - 1, Nxa), ca);
#pragma unroll
    for (int r = 0; r < NR; ++r) {
        t.p[r] = ld_at(tile_row(psi, X.j0 + r, Ny, Nx), 2 * oc);
        ev[r] = at(tile_row(emp, X.j0 + r, Ny, Nx), oc);
        mc[r] = (int)at(tile_row(mtp, X.j0 + r, Ny - 1, Nxa), ca);
    }
    bool cellm = tile_cell(has_mt, mu, hasa, X.j0 - 1, Ny), leftm = shfl_up1((int)cellm) != 0;
#pragma unroll
    for (int r = 0; r < NR; ++r) {
        const int j = X.j0 + r;
        const bool cellc = tile_cell(has_mt, mc[r], hasa, j, Ny), leftc = shfl_up1((int)cellc) != 0;
        const bool in = col && j >= 0 && j < Ny;
        t.p[r] = {in ? t.p[r].re : R(0), in ? t.p[r].im : R(0)};
        // outside the material (and beyond the grid) the sweep gives 0: all
        // four link factors are zero there, so is the right-hand side, and
        // the diagonal is 1 (with eps it would be 0 where dt eps = 1, and
        // 0 / 0 would spread from there)
        const bool inside = leftm || leftc || cellm || cellc;
        const cplx<R> rh = {inside ? t.p[r].re : R(0), inside ? t.p[r].im : R(0)};
        const R e = has_em ? ev[r] : A.eps;
        const R den = psi_den(A, rh, inside ? e : R(0), leftm, leftc, cellm, cellc);
        if constexpr (FOLD) {
            t.rden[r] = den;
            t.rd[r] = {rh.re * den, rh.im * den};
            S.base[X.w][r][X.lane] = rh;
        } else {
            t.rden[r] = R(1) / den;
            S.rhs[X.w][r][X.lane] = rh;
            S.den[X.w][r][X.lane] = den;
        }
        cellm = cellc;
        leftm = leftc;
        __builtin_amdgcn_sched_barrier(0);
    }
}

// U(-dy b) psi of a node: its part in the sum of the node above it.
template <typename R> __device__ __forceinline__ cplx<R> tile_psi_up(const cplx<R> &p, R cb, R sb) {
    return {cb * p.re - sb * p.im, cb * p.im + sb * p.re};
}

// One node: psi^{j+1} (FP32: its neighbours' part in it) from its own value,
// the part m of the row below, the row above (pp) and the lanes either side.
template <typename R, typename SH>
__device__ __forceinline__ cplx<R> tile_psi_node(const PsiSweepArgs<R> &A, const PsiTile<R, SH> &t, int r,
                                                 const cplx<R> &p, const cplx<R> &m, const cplx<R> &pp,
                                                 const cplx<R> &rhs, R den) {
    const R ca = t.ca[r], sa = t.sa[r], cb = t.cb[r], sb = t.sb[r];
    const R pr_re = shfl_dn1(p.re), pr_im = shfl_dn1(p.im);
    // this lane's part in the sum of the lane to the right
    const R l_re = ca * p.re - sa * p.im, l_im = ca * p.im + sa * p.re;
    if constexpr (std::is_same<R, float>::value) {
        float re = fmaf(ca, pr_re, m.re), im = fmaf(ca, pr_im, m.im);
        re = fmaf(sa, pr_im, re);
        im = fmaf(-sa, pr_re, im);
        re += shfl_up1(l_re);
        im += shfl_up1(l_im);
        re = fmaf(cb, pp.re, re);
        im = fmaf(cb, pp.im, im);
        re = fmaf(sb, pp.im, re);
        im = fmaf(-sb, pp.re, im);
        return {re, im};
    } else {
        const R m0r = shfl_up1(l_re), m0i = shfl_up1(l_im);
        const R p0r = ca * pr_re + sa * pr_im, p0i = ca * pr_im - sa * pr_re;
        const R q0pr = cb * pp.re + sb * pp.im, q0pi = cb * pp.im - sb * pp.re;
        const R nre = rhs.re + A.dt * (A.idx2 * (m0r + p0r) + A.idy2 * (m.re + q0pr));
        const R nim = rhs.im + A.dt * (A.idx2 * (m0i + p0i) + A.idy2 * (m.im + q0pi));
        return {div_by(nre, den, t.rden[r]), div_by(nim, den, t.rden[r])};
    }
}

// Largest |change| by row group: rows that belong to the tile in every wave
// (mid), in all but the first (top), all but the last (bot) and all but both
// (both) are told apart at compile time.
template <typename R> struct TileRes {
    R mid, top, bot, both;
    template <typename SH> __device__ __forceinline__ void add(int r, R v) {
        constexpr int NR = SH::NR, H = SH::H;
        if (r < H && r >= NR - H) both = fmax(both, v);
        else if (r < H) top = fmax(top, v);
        else if (r >= NR - H) bot = fmax(bot, v);
        else mid = fmax(mid, v);
    }
    template <typename SH> __device__ __forceinline__ R of(const TileCtx &X) const {
        R v = mid;
        v = X.first() ? v : fmax(v, top);
        v = X.last<SH>() ? v : fmax(v, bot);
        v = (X.first() || X.last<SH>()) ? v : fmax(v, both);
        return v;
    }
};

// The first and last rows of every wave for its neighbours (copy `par`).
template <typename R, typename SH>
__device__ __forceinline__ void tile_edges_out(TileLds<R, SH> &S, int par, const TileCtx &X, const cplx<R> &lo,
                                               const cplx<R> &hi) {
    S.edge[par][2 * X.w + 1][X.lane] = lo;
    S.edge[par][2 * X.w + 2][X.lane] = hi;
}

// n psi sweeps on the tile, the first of them the solve's sweep j (FP32 carries
// changes from sweep `turn` on); bit s of the result: sweep s left a change of
// at least thr at some node of the tile that belongs to this wave. `par` is the
// LDS copy the first sweep reads (the caller's edges are there, behind a
// barrier) and, on return, the one to be used next.
template <typename R, typename SH>
__device__ __forceinline__ unsigned tile_psi_sweeps(const PsiSweepArgs<R> *Ap, PsiTile<R, SH> &t, TileLds<R, SH> &S,
                                                    const TileCtx &X, int n, R thr, int &par_, int j, int turn) {
    constexpr int NR = SH::NR;
    int par = uniform(par_);
    constexpr bool F64 = std::is_same<R, double>::value;
    const PsiSweepArgs<R> A = fresh_args(Ap);
    unsigned bits = 0u;
    const cplx<R>(*rl)[WAVE] = S.rhs[F64 ? X.w : 0];
    const R(*dl)[WAVE] = S.den[F64 ? X.w : 0];
    auto sweep = [&](auto changes, int s, bool first) {
        constexpr bool CHANGES = decltype(changes)::value;
        // the rows above and below the wave's (unknown beyond the tile)
        const cplx<R> up = S.edge[par][2 * X.w][X.lane], dn = S.edge[par][2 * X.w + 3][X.lane];
        TileRes<R> res{R(0), R(0), R(0), R(0)};
        auto node = [&](int r, const cplx<R> &p, const cplx<R> &m, const cplx<R> &pp) {
            const cplx<R> q = tile_psi_node<R, SH>(A, t, r, p, m, pp, rl[F64 ? r : 0][X.lane],
                                                 dl[F64 ? r : 0][X.lane]);
            cplx<R> v = q, d = {q.re - p.re, q.im - p.im};
            if constexpr (!F64) {
                v = {fmaf(q.re, t.rden[r], t.rd[r].re), fmaf(q.im, t.rden[r], t.rd[r].im)};
                d = CHANGES ? cplx<R>{q.re * t.rden[r], q.im * t.rden[r]} : cplx<R>{v.re - p.re, v.im - p.im};
                if constexpr (CHANGES) {
                    t.rd[r] = v;
                    v = d;
                }
            }
            res.template add<SH>(r, fmax(fabs(d.re), fabs(d.im)));
            return v;
        };
        // rows 1 .. NR-1, then row 0: `up` and `dn` have the middle rows to
        // arrive in. A row's part in the sum of the next is formed before its
        // new value, which then takes its place in the registers (formed with
        // the next row it keeps the old value alive, and the loop moves two
        // registers a row: 24 of 384 instructions a sweep of 14 rows)
        const cplx<R> old1 = t.p[1];
        cplx<R> m = tile_psi_up(t.p[0], t.cb[0], t.sb[0]);
#pragma unroll
        for (int r = 1; r < NR; ++r) {
            const cplx<R> cur = t.p[r], below = m;
            if (r + 1 < NR) m = tile_psi_up(cur, t.cb[r], t.sb[r]);
            t.p[r] = node(r, cur, below, r + 1 < NR ? t.p[r + 1 < NR ? r + 1 : r] : dn);
        }
        t.p[0] = node(0, t.p[0], tile_psi_up(up, t.cbu, t.sbu), old1);
        if constexpr (CHANGES) {
            if (first) {  // the first change has the own value's part too
                res = {R(0), R(0), R(0), R(0)};
#pragma unroll
                for (int r = 0; r < NR; ++r) {
                    t.p[r] = t.rd[r];
                    res.template add<SH>(r, fmax(fabs(t.p[r].re), fabs(t.p[r].im)));
                }
            }
        }
        par ^= 1;
        tile_edges_out<R, SH>(S, par, X, t.p[0], t.p[NR - 1]);
        const bool open = X.own<SH>(A.Nx) && res.template of<SH>(X) >= thr;
        bits |= __ballot(open) != 0ull ? 1u << s : 0u;
        __syncthreads();
    };
    int s = 0;
    for (; s < n && (F64 || j + s < turn); ++s) sweep(std::false_type{}, s, false);
    if constexpr (!F64)
        for (; s < n; ++s) {
            const bool first = j + s == turn;
            if (first) {  // rhs/den - psi, rounded once
#pragma unroll
                for (int r = 0; r < NR; ++r) {
                    const cplx<R> rh = S.base[X.w][r][X.lane];
                    S.base[X.w][r][X.lane] = t.p[r];
                    t.rd[r] = {fmaf(rh.re, t.rden[r], -t.p[r].re), fmaf(rh.im, t.rden[r], -t.p[r].im)};
                }
            }
            sweep(std::true_type{}, s, first);
        }
    par_ = par;
    return bits;
}

// ---- A ------------------------------------------------------------------------
//
// The lane's part of an A solve: both links of every node, and the part of
// their updates that the source fixes, S = rhs + dt rho (J_s + H source).
template <typename R, typename SH> struct ATile {
    static constexpr int NR = SH::NR;
    R a[NR], b[NR], Sa[NR], Sb[NR];
};

// The links of the tile from a vector potential buffer.
template <typename R, typename SH>
__device__ __forceinline__ void tile_a_load(int Nx, int Ny, const R *ab, const TileCtx &X0, ATile<R, SH> &t) {
    constexpr int NR = SH::NR;
    const TileCtx X = X0.fresh();
    const int Nxa = Nx - 1;
    const R *b = ab + (size_t)Nxa * Ny;
    const bool col = X.col(Nx), hasa = X.hasa(Nx);
    const uint32_t oa = X.ca(Nx) * (uint32_t)sizeof(R), ob = X.cc(Nx) * (uint32_t)sizeof(R);
#pragma unroll
    for (int r = 0; r < NR; ++r) {
        t.a[r] = at(tile_row(ab, X.j0 + r, Ny, Nxa), oa);
        t.b[r] = at(tile_row(b, X.j0 + r, Ny - 1, Nx), ob);
    }
#pragma unroll
    for (int r = 0; r < NR; ++r) {
        const int j = X.j0 + r;
        t.a[r] = (hasa && j >= 0 && j < Ny) ? t.a[r] : R(0);
        t.b[r] = (col && j >= 0 && j < Ny - 1) ? t.b[r] : R(0);
    }
}

// Those of them that do not belong to the tile, as its neighbours
// published them.
template <typename R, typename SH>
__device__ __forceinline__ void tile_a_halo(int Nx, int Ny, const R *ab, const TileCtx &X0, ATile<R, SH> &t) {
    constexpr int NR = SH::NR;
    const TileCtx X = X0.fresh();
    const int Nxa = Nx - 1;
    const R *b = ab + (size_t)Nxa * Ny;
    const bool col = X.col(Nx), hasa = X.hasa(Nx), own = X.own<SH>(Nx);
    const uint32_t cc = X.cc(Nx);
    const int r0 = X.r0<SH>(), r1 = X.r1<SH>(Ny);
#pragma unroll
    for (int r = 0; r < NR; ++r) {
        const int j = X.j0 + r;
        if (j >= 0 && j < Ny) {
            const bool halo = !(own && r >= r0 && r < r1);
            if (halo && hasa) t.a[r] = ld_shared_mem(ab + (size_t)Nxa * j + cc);
            if (halo && col && j < Ny - 1) t.b[r] = ld_shared_mem(b + (size_t)Nx * j + cc);
        }
    }
}

// The fixed parts Sa, Sb of a pair of sweeps whose source is the current
// (a, b); A^n is read from `rhs`. psi_dn: psi of the row below the wave's
// last one.
template <typename R, bool GAUGE, typename SH>
__device__ __forceinline__ void tile_a_source(const ASweepArgs<R> *Ap, const cplx<R> (&p)[SH::NR], unsigned ena,
                                              unsigned enb, const cplx<R> &psi_dn, const R *rhs, const TileCtx &X0,
                                              ATile<R, SH> &t) {
    constexpr int NR = SH::NR;
    const ASweepArgs<R> A = fresh_args(Ap);
    const TileCtx X = X0.fresh();
    const int Nx = A.Nx, Ny = A.Ny, Nxa = Nx - 1;
    const R *rhs_b = rhs + (size_t)Nxa * Ny;
    const bool col = X.col(Nx), hasa = X.hasa(Nx);
    const uint32_t oa = X.ca(Nx) * (uint32_t)sizeof(R), ob = X.cc(Nx) * (uint32_t)sizeof(R);
    const R gb = GAUGE ? gauge_phase_b<R>(A, X.c) : R(0);
    TileSinCos<R> sincos;
    sincos.load();
    ena = (unsigned)fresh_v((int)ena);
    enb = (unsigned)fresh_v((int)enb);
    const R rhb = X.c == 0 ? -A.rh_b : (X.c + 1 == Nx ? A.rh_b : R(0));
#pragma unroll
    for (int r = 0; r < NR; ++r) {
        t.Sa[r] = at(tile_row(rhs, X.j0 + r, Ny, Nxa), oa);
        t.Sb[r] = at(tile_row(rhs_b, X.j0 + r, Ny - 1, Nx), ob);
    }
#pragma unroll
    for (int r = 0; r < NR; ++r) {
        const int j = X.j0 + r;
        R sn, cs;
        sincos(link_phase<R, GAUGE>(A.dx, t.a[r], GAUGE ? gauge_phase_a<R>(A, j) : R(0)), &sn, &cs);
        // psi is the same for every pair of sweeps: without the fresh copies
        // its products would be kept from one pair to the next
        const cplx<R> pr = {fresh_r(p[r].re), fresh_r(p[r].im)};
        const R jla = tile_mask(link_current(A.idx, pr, shfl_dn1(pr.re), shfl_dn1(pr.im), cs, sn), ena, r);
        sincos(link_phase<R, GAUGE>(A.dy, t.b[r], gb), &sn, &cs);
        const cplx<R> pu = r + 1 < NR ? p[r + 1 < NR ? r + 1 : r] : psi_dn;
        const R jlb = tile_mask(link_current(A.idy, pr, pu.re, pu.im, cs, sn), enb, r);
        const R rha = j == 0 ? A.rh_a : (j + 1 == Ny ? -A.rh_a : R(0));
        const R va = t.Sa[r] + A.dt_rho * (jla + rha), vb = t.Sb[r] + A.dt_rho * (jlb + rhb);
        t.Sa[r] = (hasa && j >= 0 && j < Ny) ? va : R(0);
        t.Sb[r] = (col && j >= 0 && j < Ny - 1) ? vb : R(0);
        __builtin_amdgcn_sched_barrier(0);
    }
}

// One A sweep with the source parts in t.Sa, t.Sb; up, dn: (a, b) of the
// rows above and below the wave's (unknown beyond the tile). EDGE: the
// wave's rows reach the grid's first or last row or beyond.
template <typename R, bool EDGE, typename SH>
__device__ __forceinline__ void tile_a_sweep(const ASweepArgs<R> &A, ATile<R, SH> &t, const TileCtx &X, R Ka, R Kb,
                                             const cplx<R> &up, const cplx<R> &dn, R rden_a, R rden_b,
                                             TileRes<R> &res) {
    constexpr int NR = SH::NR;
    const int j0 = EDGE ? fresh_s(X.j0) : 0;
    // links (a, b) of a row, (am, bm) of the row below it in index, ap of
    // the row after it -> the updated pair
    auto links = [&](int r, R a, R b, R am, R bm, R ap, R &va, R &vb) {
        R Ta, Tb;
        if constexpr (std::is_same<R, double>::value) {
            const R P = A.idxy * b, Pm = A.idxy * bm;
            const R t1 = A.idy2 * am - Pm + shfl_dn1(Pm);
            const R t2 = A.idy2 * ap + P - shfl_dn1(P);
            Ta = t1 + t2;
            const R W = A.idx2 * b, Z = A.idxy * a, Zp = A.idxy * ap;
            const R u1 = shfl_up1(W) - shfl_up1(Z) + shfl_up1(Zp);
            const R u2 = shfl_dn1(W) + Z - Zp;
            Tb = u1 + u2;
        } else {
            const R D = b - shfl_dn1(b), Dm = bm - shfl_dn1(bm), E = a - ap;
            Ta = fmaf(A.idxy, D - Dm, A.idy2 * (am + ap));
            Tb = fmaf(A.idxy, E - shfl_up1(E), A.idx2 * (shfl_up1(b) + shfl_dn1(b)));
        }
        if constexpr (EDGE) {
            // 0 where the row has no such link, 2 on the boundary rows (ghost cell)
            const int j = j0 + r, Ny = A.Ny;
            Ta *= (j < 0 || j >= Ny) ? R(0) : ((j == 0 || j == Ny - 1) ? R(2) : R(1));
            Tb *= (j < 0 || j >= Ny - 1) ? R(0) : R(1);
        }
        if constexpr (std::is_same<R, double>::value) {
            va = div_by(t.Sa[r] + Ka * Ta, A.den_a, rden_a);
            vb = div_by(t.Sb[r] + Kb * Tb, A.den_b, rden_b);
        } else {
            // in_vgpr: the change below is that of the rounded values (an fma
            // of the unrounded product would be off by up to half an ulp,
            // 5e-7 where |A| nears 16, and the stop criterion of 1e-6 would
            // never be met on large grids)
            va = in_vgpr(fmaf(Ka, Ta, t.Sa[r]) * A.iden_a);
            vb = in_vgpr(fmaf(Kb, Tb, t.Sb[r]) * A.iden_b);
        }
        res.template add<SH>(r, fmax(fabs(va - a), fabs(vb - b)));
    };
    const R a0 = t.a[0], b0 = t.b[0], a1 = t.a[1];
    R pa = a0, pb = b0;
#pragma unroll
    for (int r = 1; r < NR; ++r) {
        const R a = t.a[r], b = t.b[r];
        links(r, a, b, pa, pb, r + 1 < NR ? t.a[r + 1 < NR ? r + 1 : r] : dn.re, t.a[r], t.b[r]);
        pa = a;
        pb = b;
    }
    links(0, a0, b0, up.re, up.im, a1, t.a[0], t.b[0]);
}

// n A sweeps; result as tile_psi_sweeps. The LDS edges hold (a, b) of a
// wave's first and last rows.
template <typename R, typename SH>
__device__ __forceinline__ unsigned tile_a_sweeps(const ASweepArgs<R> *Ap, ATile<R, SH> &t, TileLds<R, SH> &S,
                                                  const TileCtx &X, int n, R thr, int &par_, R rden_a, R rden_b) {
    constexpr int NR = SH::NR;
    int par = uniform(par_);
    const ASweepArgs<R> A = fresh_args(Ap);
    unsigned bits = 0u;
    // dt rho kappa^2 times the ghost factor of the b links' column; 0 where
    // the column has no such link
    const R Ka = X.hasa(A.Nx) ? A.dt_rho_kappa2 : R(0);
    const R Kb = X.col(A.Nx) ? ((X.c == 0 || X.c + 1 == A.Nx) ? R(2) * A.dt_rho_kappa2 : A.dt_rho_kappa2) : R(0);
    const bool edge = X.j0 < 1 || X.j0 + NR > A.Ny - 1;
    for (int s = 0; s < n; ++s) {
        const cplx<R> up = S.edge[par][2 * X.w][X.lane], dn = S.edge[par][2 * X.w + 3][X.lane];
        TileRes<R> res{R(0), R(0), R(0), R(0)};
        if (edge) tile_a_sweep<R, true, SH>(A, t, X, Ka, Kb, up, dn, rden_a, rden_b, res);
        else tile_a_sweep<R, false, SH>(A, t, X, Ka, Kb, up, dn, rden_a, rden_b, res);
        par ^= 1;
        tile_edges_out<R, SH>(S, par, X, cplx<R>{t.a[0], t.b[0]}, cplx<R>{t.a[NR - 1], t.b[NR - 1]});
        const bool open = X.own<SH>(A.Nx) && res.template of<SH>(X) >= thr;
        bits |= __ballot(open) != 0ull ? 1u << s : 0u;
        __syncthreads();
    }
    par_ = par;
    return bits;
}

// ---- publishing and meeting -----------------------------------------------------

// Whether row r of the wave is in the ring of width H along the tile's top
// and bottom edges that its neighbours read.
template <typename SH> __device__ __forceinline__ bool tile_ring_row(const TileCtx &X, int r) {
    const int tr = X.w * SH::NR + r;  // row in the tile
    return tr < 2 * SH::H || tr >= SH::NW * SH::NR - 2 * SH::H;
}

// The tile's nodes (all of them, or just the ring) to a psi buffer. `all` is
// laundered: a copy of the code for each of its values would cost more in
// instruction fetches, once a solve, than the lane masks do. The wait ahead
// of the stores is for loads long past: without it the compiler waits, on
// the common counter, ahead of every store (each value was once loaded on
// some path), and the stores go out one at a time: 1.6 instead of 0.6 us for
// the A links of 4 rows, and as long again until the last one is through.
template <typename R, typename SH>
__device__ __forceinline__ void tile_psi_publish(int Nx, int Ny, cplx<R> *out, const TileCtx &X0,
                                                 const cplx<R> (&p)[SH::NR], bool all) {
    constexpr int NR = SH::NR, H = SH::H;
    const TileCtx X = X0.fresh();
    const bool own = X.own<SH>(Nx), side = fresh_v(all) || X.lane < 2 * H || X.lane >= WAVE - 2 * H;
    const uint32_t cc = X.cc(Nx);
    const int r0 = X.r0<SH>(), r1 = X.r1<SH>(Ny);
    __builtin_amdgcn_s_waitcnt(0);
#pragma unroll
    for (int r = 0; r < NR; ++r)
        if (r >= r0 && r < r1 && own && (side || tile_ring_row<SH>(X, r)))
            st_shared_mem(out + (size_t)Nx * (X.j0 + r) + cc, p[r]);
}

// psi of a FP32 solve past its turn at the nodes of the tile.
template <typename R, typename SH>
__device__ __forceinline__ void tile_psi_total(const TileLds<R, SH> &S, const TileCtx &X, const PsiTile<R, SH> &t,
                                               cplx<R> (&p)[SH::NR]) {
#pragma unroll
    for (int r = 0; r < SH::NR; ++r) {
        const cplx<R> b = S.base[X.w][r][X.lane];
        p[r] = {b.re + t.rd[r].re, b.im + t.rd[r].im};
    }
}
template <typename R, typename SH>
__device__ __forceinline__ void tile_a_publish(int Nx, int Ny, R *out, const TileCtx &X0, const ATile<R, SH> &t,
                                               bool all) {
    constexpr int NR = SH::NR, H = SH::H;
    const TileCtx X = X0.fresh();
    const int Nxa = Nx - 1;
    R *out_b = out + (size_t)Nxa * Ny;
    const bool own = X.own<SH>(Nx), side = fresh_v(all) || X.lane < 2 * H || X.lane >= WAVE - 2 * H, hasa = X.hasa(Nx);
    const uint32_t cc = X.cc(Nx);
    const int r0 = X.r0<SH>(), r1 = X.r1<SH>(Ny);
    __builtin_amdgcn_s_waitcnt(0);
#pragma unroll
    for (int r = 0; r < NR; ++r)
        if (r >= r0 && r < r1 && own && (side || tile_ring_row<SH>(X, r))) {
            const int j = X.j0 + r;
            if (hasa) st_shared_mem(out + (size_t)Nxa * j + cc, t.a[r]);
            if (j < Ny - 1) st_shared_mem(out_b + (size_t)Nx * j + cc, t.b[r]);
        }
}

// The halo nodes of the tile from a psi buffer its neighbours published.
template <typename R, typename SH>
__device__ __forceinline__ void tile_psi_halo(int Nx, int Ny, const cplx<R> *psi, const TileCtx &X0,
                                              PsiTile<R, SH> &t) {
    constexpr int NR = SH::NR;
    const TileCtx X = X0.fresh();
    const bool col = X.col(Nx), own = X.own<SH>(Nx);
    const uint32_t cc = X.cc(Nx);
    const int r0 = X.r0<SH>(), r1 = X.r1<SH>(Ny);
#pragma unroll
    for (int r = 0; r < NR; ++r) {
        const int j = X.j0 + r;
        if (j >= 0 && j < Ny && col && !(own && r >= r0 && r < r1))
            t.p[r] = ld_shared_mem(psi + (size_t)Nx * j + cc);
    }
}

// One poll of a word until its epoch is at least `epoch`. Returns false
// when the run is being aborted or the wait is past its bound.
__device__ __forceinline__ bool tile_poll(const unsigned long long *w, unsigned long long epoch, int *err,
                                          unsigned long long &v) {
    const unsigned long long t0 = wall_clock64();
    while (((v = ld_relaxed(w)) >> 32) < epoch) {
        if (ld_relaxed(err)) return false;
        if (wall_clock64() - t0 > BARRIER_TIMEOUT_TICKS) {
            __hip_atomic_store(err, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            return false;
        }
        __builtin_amdgcn_s_sleep(1);
    }
    return true;
}

// What this workgroup published is in memory (the stores are written
// through; every wave waits for its own), then its flag says so.
__device__ __forceinline__ void tile_signal(unsigned long long *w, unsigned long long v) {
    __builtin_amdgcn_s_waitcnt(0);
    __syncthreads();
    if (threadIdx.x == 0) __hip_atomic_store(w, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Publish epoch `epoch` to the neighbours and wait for theirs. A tile is at
// most one epoch ahead of its neighbours: it has read their rings of epoch
// e before it signals e + 1, and they wait for that before they overwrite
// the buffer of epoch e with that of e + 2.
template <typename R, typename SH>
__device__ __forceinline__ bool tile_meet_neighbours(const TileSync &ts, const TileTeam &tm, unsigned long long epoch,
                                                     TileLds<R, SH> &S) {
    unsigned long long *flag = ts.flag + tm.base + tm.ty * tm.ntx + tm.tx;
    tile_signal(flag, epoch << 32);
    bool ok = true;
    if (threadIdx.x == 0) ok = ld_relaxed(ts.err) == 0;
    if (threadIdx.x < 9 && threadIdx.x != 4) {
        const int x = tm.tx + (int)threadIdx.x % 3 - 1, y = tm.ty + (int)threadIdx.x / 3 - 1;
        if (x >= 0 && x < tm.ntx && y >= 0 && y < tm.nty) {
            unsigned long long v;
            ok = tile_poll(flag + (y - tm.ty) * tm.ntx + (x - tm.tx), epoch, ts.err, v) && ok;
        }
    }
    return uniform(__syncthreads_or(!ok)) == 0;
}

// All workgroups of the instance meet: `bits` (per wave) are or-ed over all
// of them. Everything they published is visible to plain loads afterwards.
// Two levels: the first workgroup of every TILE_GROUP gathers its group's
// words into a group word, and every workgroup waits for all group words.
// (With every workgroup polling every word, 484 workgroups took 22 us: a
// thousand cache lines each asked for by all of them.)
constexpr int TILE_GROUP = 32;
template <typename R, typename SH>
__device__ __forceinline__ bool tile_meet_all(const TileSync &ts, const TileTeam &tm, unsigned long long epoch,
                                              TileLds<R, SH> &S, unsigned bits, unsigned &out) {
    const int lane = threadIdx.x & (WAVE - 1), w = wave_id();
    if (lane == 0) S.bits[w] = bits;
    __builtin_amdgcn_s_waitcnt(0);
    __syncthreads();
    if (w == 0) {
        unsigned mine = 0u;
#pragma unroll
        for (int k = 0; k < SH::NW; ++k) mine |= S.bits[k];
        unsigned long long *words = ts.chk[epoch & 1] + tm.base, *groups = ts.grp[epoch & 1] + tm.gbase;
        const int local = tm.ty * tm.ntx + tm.tx, g0 = local - local % TILE_GROUP;
        const int ng = (tm.nwg + TILE_GROUP - 1) / TILE_GROUP;
        if (lane == 0)
            __hip_atomic_store(words + local, (epoch << 32) | mine, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        bool ok = ld_relaxed(ts.err) == 0;
        auto all = [&](unsigned v) {
#pragma unroll
            for (int off = 32; off > 0; off >>= 1) v |= (unsigned)__shfl_xor((int)v, off, WAVE);
            return v;
        };
        unsigned long long v = 0ull;
        if (local == g0) {
            if (ok && lane < TILE_GROUP && g0 + lane < tm.nwg) ok = tile_poll(words + g0 + lane, epoch, ts.err, v);
            mine = all(mine | (unsigned)v);
            if (!__any(!ok) && lane == 0)
                __hip_atomic_store(groups + g0 / TILE_GROUP, (epoch << 32) | mine, __ATOMIC_RELAXED,
                                   __HIP_MEMORY_SCOPE_AGENT);
        }
        for (int k = lane; k < ng && ok; k += WAVE) {
            ok = tile_poll(groups + k, epoch, ts.err, v);
            mine |= (unsigned)v;
        }
        mine = all(mine);
        const bool fail = __any(!ok);
        if (lane == 0) {
            S.all = mine;
            S.fail = fail;
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
        }
    }
    __syncthreads();
    out = (unsigned)uniform((int)S.all);
    return uniform(S.fail) == 0;
}

// ---- the run --------------------------------------------------------------------

// Where a solve stands: sweeps done, the first sweep of the bits gathered
// since the last check, and the sweep to check at next. The first check is
// at the previous step's count; the ones after it one, two, ... sweeps on.
struct TileSched {
    int j, j0, next, beyond;
    __device__ __forceinline__ TileSched(int pred, int most, int max_sweeps)
        : j(0), j0(0), next(min(min(pred > 0 ? pred : most, 32), max_sweeps)), beyond(pred > 0 ? 1 : most) {}
    // the first sweep of the window that met the stop rule everywhere (bits
    // of the sweeps that did not), 0 if none did
    __device__ __forceinline__ int met(unsigned open) const {
        const int len = j - j0;
        const unsigned done = ~open & (len >= 32 ? ~0u : (1u << len) - 1u);
        return done ? j0 + __ffs((int)done) : 0;
    }
    // the solve once more, up to sweep m
    __device__ __forceinline__ void again(int m) {
        j = j0 = 0;
        next = m;
    }
    // after a check without convergence
    __device__ __forceinline__ void extend(int pred, int max_sweeps) {
        j0 = j;
        next = (j < pred) ? min(pred, j + 32) : j + beyond;
        if (j >= pred) beyond = min(2 * beyond, 8);
        next = min(next, max_sweeps);
    }
};

// All steps of a run on this workgroup's tile. FP32 with WITHA holds A in
// the gauge-shifted form (link_phase).
template <typename R, bool WITHA, typename SH>
__device__ __forceinline__ void tile_run(const TDSolveArgs<R> *T, const TileSync &ts, const TileTeam &tm, int nsteps,
                                         R thr_psi, R thr_a, int *st, int *sweeps, int stride, bool passes, TileLds<R, SH> &S) {
    constexpr int NR = SH::NR, H = SH::H;
    constexpr bool GAUGE = WITHA && RunForm<R>::has_gauge;
    constexpr bool F64 = std::is_same<R, double>::value;
    constexpr int HA = H & ~1;  // A sweeps between exchanges: even, as the source changes with every second sweep
    const int Nx = arg(&T->psi.Nx), Ny = arg(&T->psi.Ny), max_sweeps = arg(&T->max_sweeps);
    const TileCtx X = tile_ctx<SH>(tm.tx, tm.ty);
    if (X.w < 4)  // the rows of zeros; a barrier follows before any is read
        S.edge[X.w >> 1][(X.w & 1) ? 2 * SH::NW + 1 : 0][X.lane] = {R(0), R(0)};
    PsiTile<R, SH> t;
    int pc = uniform(st[ST_PSI]), qc = uniform(st[ST_AB]), pred = 0, pred_a = 0, par = 0;
    int redo = 0, redo_a = 0, done_steps = 0;
    unsigned long long ef = 0, ec = 0;  // epochs of the flag and check words
    bool ok = true;
    R rden_a = R(0), rden_b = R(0);
    if constexpr (F64 && WITHA) {
        rden_a = R(1) / arg(&T->A.den_a);
        rden_b = R(1) / arg(&T->A.den_b);
    }
    for (int step = 0; step < nsteps && ok; ++step) {
        // -- psi
        const int o1 = (pc + 1) % 3, o2 = (pc + 2) % 3;
        int cur = pc;  // the buffer published last
        {
            if (WITHA || step == 0) tile_links<R, GAUGE, SH>(&T->psi, arg(&T->Q[uniform(qc)]), X, t);
            TileSched sc(pred, H, max_sweeps);
            unsigned bits = 0u;
            int nsw = 0, stop = 0;  // stop: the sweep a redone solve ends at
            const int turn = pred > 0 && pred <= PSI_FEW ? 0 : PSI_TURN;
            bool again;
            do {
                again = false;
                tile_psi_load<R, SH>(&T->psi, arg(&T->P[uniform(pc)]), X, t, S);
                for (;;) {
                    par ^= 1;
                    tile_edges_out<R, SH>(S, par, X, t.p[0], t.p[NR - 1]);
                    __syncthreads();
                    const int n = uniform(min(sc.next - sc.j, H));
                    bits |= tile_psi_sweeps<R, SH>(&T->psi, t, S, X, n, thr_psi, par, uniform(sc.j), uniform(turn)) << (sc.j - sc.j0);
                    sc.j += n;
                    const bool check = uniform(sc.j) == uniform(sc.next);
                    cur = cur == o1 ? o2 : o1;
                    // FP32: all of psi^{n+1} goes out at a check, the ring of
                    // psi or changes where the solve goes on
                    if (F64 || check) {
                        cplx<R> v[NR];
#pragma unroll
                        for (int r = 0; r < NR; ++r) v[r] = t.p[r];
                        if (!F64 && uniform(sc.j) > uniform(turn)) tile_psi_total<R, SH>(S, X, t, v);
                        tile_psi_publish<R, SH>(Nx, Ny, arg(&T->P[uniform(cur)]), X, v, check);
                    }
                    if (check) {
                        unsigned all = 0u;
                        if (!(ok = tile_meet_all<R, SH>(ts, tm, ++ec, S, bits, all))) break;
                        nsw = sc.j;
                        if (stop) break;  // a redone solve is over
                        const int m = sc.met(all);
                        if (m == sc.j || (!m && sc.j >= max_sweeps)) break;
                        bits = 0u;
                        if (m) {  // an earlier sweep met the stop rule: again from psi^n, up to that sweep
                            ++redo;
                            sc.again(stop = m);
                            again = true;
                            break;
                        }
                        sc.extend(pred, max_sweeps);
                        if constexpr (!F64) cur = cur == o1 ? o2 : o1;
                    }
                    if (!(F64 && check)) {
                        if constexpr (!F64) tile_psi_publish<R, SH>(Nx, Ny, arg(&T->P[uniform(cur)]), X, t.p, false);
                        if (!(ok = tile_meet_neighbours<R, SH>(ts, tm, ++ef, S))) break;
                    }
                    tile_psi_halo<R, SH>(Nx, Ny, arg(&T->P[uniform(cur)]), X, t);
                }
            } while (again);
            if (!ok) break;
            if (!F64 && uniform(nsw) > uniform(turn)) tile_psi_total<R, SH>(S, X, t, t.p);
            pred = nsw;
            if (threadIdx.x == 0 && tm.tx == 0 && tm.ty == 0) sweeps[(long)step * stride] = nsw;
        }
        pc = cur;
        // -- A
        if constexpr (WITHA) {
            const int q1 = (qc + 1) % 3, q2 = (qc + 2) % 3;
            const R *Q = arg(&T->Q[uniform(qc)]);
            int qcur = qc;
            ATile<R, SH> u;
            // psi beyond the tile, and of the row below the wave's last one
            tile_psi_halo<R, SH>(Nx, Ny, arg(&T->P[uniform(pc)]), X, t);
            par ^= 1;
            tile_edges_out<R, SH>(S, par, X, t.p[0], t.p[NR - 1]);
            __syncthreads();
            const cplx<R> pdn = S.edge[par][2 * X.w + 3][X.lane];
            TileSched sc(pred_a, HA, max_sweeps);
            unsigned bits = 0u;
            int nsw = 0, stop = 0;
            bool again;
            do {
                again = false;
                tile_a_load<R, SH>(Nx, Ny, Q, X, u);
                int seg = HA;  // sweeps since the halo was read
                for (;;) {
                    // rings are exchanged at even sweeps only, where the source
                    // parts are formed anew: between, those of the halo are as
                    // old as the halo
                    if (sc.j % 2 == 0) {
                        seg = 0;
                        par ^= 1;
                        tile_edges_out<R, SH>(S, par, X, cplx<R>{u.a[0], u.b[0]}, cplx<R>{u.a[NR - 1], u.b[NR - 1]});
                        __syncthreads();
                    }
                    do {
                        if (sc.j % 2 == 0) tile_a_source<R, GAUGE, SH>(&T->A, t.p, t.ena, t.enb, pdn, Q, X, u);
                        const int n = uniform(min(sc.next - sc.j, 2 - sc.j % 2));
                        bits |= tile_a_sweeps<R, SH>(&T->A, u, S, X, n, thr_a, par, rden_a, rden_b) << (sc.j - sc.j0);
                        sc.j += n;
                        seg += n;
                    } while (sc.j < sc.next && seg < HA);
                    const bool check = uniform(sc.j) == uniform(sc.next);
                    qcur = qcur == q1 ? q2 : q1;
                    tile_a_publish<R, SH>(Nx, Ny, arg(&T->Q[uniform(qcur)]), X, u, check);
                    if (!check) {
                        if (!(ok = tile_meet_neighbours<R, SH>(ts, tm, ++ef, S))) break;
                    } else {
                        unsigned all = 0u;
                        if (!(ok = tile_meet_all<R, SH>(ts, tm, ++ec, S, bits, all))) break;
                        nsw = sc.j;
                        if (stop) break;
                        const int m = sc.met(all);
                        if (m == sc.j || (!m && sc.j >= max_sweeps)) break;
                        bits = 0u;
                        if (m) {
                            ++redo_a;
                            sc.again(stop = m);
                            again = true;
                            break;
                        }
                        sc.extend(pred_a, max_sweeps);
                    }
                    if (sc.j % 2 == 0) tile_a_halo<R, SH>(Nx, Ny, arg(&T->Q[uniform(qcur)]), X, u);
                }
            } while (again);
            if (!ok) break;
            qc = qcur;
            pred_a = nsw;
            if (threadIdx.x == 0 && tm.tx == 0 && tm.ty == 0) sweeps[(long)step * stride + 1] = nsw;
        } else {
            if (threadIdx.x == 0 && tm.tx == 0 && tm.ty == 0) sweeps[(long)step * stride + 1] = 0;
        }
        ++done_steps;
    }
    if (threadIdx.x == 0 && tm.tx == 0 && tm.ty == 0) {
        if (!ok) {
            st[ST_ERRSTEP] = done_steps + 1;
            return;
        }
        st[ST_PSI] = pc;
        st[ST_AB] = qc;
        if (!passes) return;
        st[ST_PASS_PSI] = nsteps + redo;
        st[ST_REDO_PSI] = redo;
        st[ST_PASS_A] = WITHA ? nsteps + redo_a : 0;
        st[ST_REDO_A] = redo_a;
    }
}

template <typename R, bool WITHA, typename SH>
__global__ void __launch_bounds__(SH::NW * WAVE, 2)
    k_td_tiles(TDSolveArgs<R> T_, TileSync ts, int ntx, int nty, int nsteps, R thr_psi, R thr_a) {
    __shared__ TileLds<R, SH> S;
    // the arguments where they lie in constant memory (T_ is the first one)
    const TDSolveArgs<R> *T = (const TDSolveArgs<R> *)__builtin_amdgcn_kernarg_segment_ptr();
    const int wg = xcd_block();
    const TileTeam tm{0, 0, ntx * nty, wg % ntx, wg / ntx, ntx, nty};
    tile_run<R, WITHA, SH>(T, ts, tm, nsteps, thr_psi, thr_a, T_.sc.state, T_.sc.sweeps, 2, true, S);
}

// A batch: the tiles of many instances in one launch, each instance with
// its own words, state and sweep counts. Instance k of the launch has the
// workgroups from inst[k].b0 on; where its arguments, state and sweeps lie
// is numbered by inst[k].id.
struct TileInst {
    int b0, ntx, nty, gbase, id, pad;
    double thr_psi, thr_a;
};

template <typename R, bool WITHA, typename SH>
__global__ void __launch_bounds__(SH::NW * WAVE, 2)
    k_batch_td_tiles(const TDSolveArgs<R> *args, const TileInst *inst, int ninst, TileSync ts, int *state, int *sweeps,
                     int n, int nsteps) {
    __shared__ TileLds<R, SH> S;
    const int wg = xcd_block();
    int lo = 0, hi = ninst;  // the last instance that begins at or before wg
    while (hi - lo > 1) {
        const int mid = (lo + hi) / 2;
        if (arg(&inst[mid].b0) <= wg) lo = mid;
        else hi = mid;
    }
    const TileInst I = fresh_args(inst + lo);
    const int local = wg - I.b0;
    const TileTeam tm{I.b0, I.gbase, I.ntx * I.nty, local % I.ntx, local / I.ntx, I.ntx, I.nty};
    tile_run<R, WITHA, SH>(args + I.id, ts, tm, nsteps, R(I.thr_psi), R(I.thr_a), state + 8 * I.id,
                           sweeps + 2 * I.id, 2 * n, false, S);
}

// A <-> A - A_g of the batch's instances that evolve A (args[k].solveA), one
// row of workgroups each; the buffer is the one the state says.
template <typename R> __global__ void __launch_bounds__(256) k_batch_gauge_shift(const TDSolveArgs<R> *args, const int *state, double sign) {
    const int k = blockIdx.y;
    const TDSolveArgs<R> &T = args[k];
    if (!T.solveA) return;
    gauge_shift<R>(pick3(T.Q, state[8 * k + ST_AB]), T.A.Nx, T.A.Ny, T.A.gH, T.A.gdx, T.A.gdy, T.A.gx0, T.A.gy0, sign);
}

}  // namespace glx
