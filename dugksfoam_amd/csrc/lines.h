// lines.h -- the step kernels over velocity columns (included by dugks_engine.hip).
//
// The velocity set is a tensor product, so along its last axis (z in 3-D, y in 2-D, x in 1-D)
// everything a kernel needs of a velocity is a factor or a polynomial of the one coordinate that
// changes.  Here a lane owns a column of velocities: it keeps the other coordinates, so that the
// Gaussian products, the Shakhov polynomials and xi.S of every face of a cell reduce to one or two
// operations per velocity, and the velocity sums of a column need only the powers 0..3 of the last
// coordinate (4 sums instead of 14); the other factors are applied once, when the column ends.
// A lane that takes any velocity and rebuilds all of it is bound by its vector instructions, about
// three times as many; and the face moments ride along in the pass that forms the face values instead
// of reading them back from HBM.  A step before (k_face_values, k_face_moments, k_cell) and now, ms:
//   48^3 cells, 24^3 velocities, FP64    46.9  35.9      20000 triangles, 64^2, FP64    5.77  4.48
//   48^3 cells, 24^3 velocities, FP32    36.6  28.2      64 cavities, 28^2, FP64        6.19  5.16
//   21^3 cells, 13^3, g and h, FP64      1.77  1.11      60^2 cells, 41^2, FP64        0.310 0.266
//
// Cells of up to 6 faces (3-D) or 4 (2-D, 1-D) in face-value mode take this path: the per-face
// constants of a loop iteration and the per-face sums then fit the register files.  General
// polyhedra, the rebuilding mode and DUGKS_FACE_MFMA=0 keep the kernels of dugks_engine.hip.
#pragma once

#include "lane_sums.h"

// The column of one lane of a tile: iteration i of the tile is velocity 64 (titer[tile] + i) + lane of
// a row, at loop-axis position l + i dl; i < n (the other lanes' entries are padding).
struct alignas(8) LineRec {
    uint8_t ix, iy;   // the fixed axes (none in 1-D, x in 2-D, x and y in 3-D)
    uint8_t l, dl;
    int32_t n;
};

// Values a column's sums expand to: density, momentum / central first moment (D), second moments
// (D (D + 1) / 2), Q (D) and, where h is carried, its energy sum.
template <int D, bool H>
constexpr int line_nval()
{
    return 1 + D + D * (D + 1) / 2 + D + (H ? 1 : 0);
}

constexpr int LINE_MAXW = 8;             // waves per workgroup
constexpr int LINE_MAXNT = 64 * LINE_MAXW;

// LDS by its own address space, where one value comes from LDS or from memory: through generic pointers the
// compiler merges the two loads into one flat load behind a null check.
#define LDS_AS __attribute__((address_space(3)))

template <typename T>
DEVI T ld_at(const T *base, unsigned byte_off)
{
    return *(const T *)((const char *)base + byte_off);
}

template <typename TS>
DEVI void st_at_stream(TS *base, unsigned byte_off, double v)
{
    TS *q = (TS *)((char *)base + byte_off);
    if (DUGKS_NT_STORE) __builtin_nontemporal_store((TS)v, q);
    else *q = (TS)v;
}

// Keeps a wave-uniform value in scalar registers across the loops that use it.  Without it the compiler
// loads it again from the scalar cache in every iteration, and every wait for such a load (they return
// out of order) stalls the wave.
DEVI int pin_word(int u)
{
    asm volatile("" : "+v"(u));
    return __builtin_amdgcn_readfirstlane(u);
}

template <typename T>
DEVI void pin(T &v)
{
    if constexpr (sizeof(T) == 4) {
        v = __builtin_bit_cast(T, pin_word(__builtin_bit_cast(int, v)));
    } else {
        const uint64_t b = __builtin_bit_cast(uint64_t, v);
        const uint32_t lo = pin_word((int)(uint32_t)b), hi = pin_word((int)(uint32_t)(b >> 32));
        v = __builtin_bit_cast(T, (uint64_t)hi << 32 | lo);
    }
}

// A column's sums (line_add): n[m] = sum w_l c_l^m g for m = 0..2 of the loop axis (c = coordinate -
// reference), n[3] = sum w_l c_l (c_l^2 g + h) and, where h is carried, n[4] = sum w_l h.
template <bool H>
constexpr int line_nsum()
{
    return H ? 5 : 4;
}

template <bool H>
DEVI void line_add(double *n, const double *wl, double g, double h)
{
#pragma unroll
    for (int m = 0; m < 4; ++m) n[m] = fma(g, wl[m], n[m]);
    if (H) {
        n[3] = fma(h, wl[1], n[3]);
        n[4] = fma(h, wl[0], n[4]);
    }
}

// Sums of a finished column -> its NV values, with w and cx, cy the lane's fixed factors.
// Order: 1; c (D); c c^T (upper triangle); c (|c|^2 g + h) (D); h.
template <int D, bool H>
DEVI void line_expand(const double *n, double w, double cx, double cy, double *o)
{
    const double N0 = w * n[0], N1 = w * n[1], N2 = w * n[2], N3 = w * n[3];
    const double h0 = H ? w * n[4] : 0.0;
    int m = 0;
    o[m++] = N0;
    if constexpr (D == 3) {
        const double bx = cx * N0, by = cy * N0, r2 = cx * cx + cy * cy;
        o[m++] = bx; o[m++] = by; o[m++] = N1;
        o[m++] = cx * bx; o[m++] = cx * by; o[m++] = cx * N1;
        o[m++] = cy * by; o[m++] = cy * N1; o[m++] = N2;
        const double e = r2 * N0 + N2 + h0;
        o[m++] = cx * e; o[m++] = cy * e; o[m++] = r2 * N1 + N3;
    } else if constexpr (D == 2) {
        const double bx = cx * N0;
        o[m++] = bx; o[m++] = N1;
        o[m++] = cx * bx; o[m++] = cx * N1; o[m++] = N2;
        o[m++] = cx * (cx * bx + N2 + h0); o[m++] = cx * cx * N1 + N3;
    } else {
        o[m++] = N1;
        o[m++] = N2;
        o[m++] = N3;
    }
    if (H) o[m++] = h0;
}

// NV totals about Ur -> the moment record of acc_moments (density, momentum, energy, Q, P about Ur).
template <int D, bool H>
DEVI void line_record(const double *t, const double *Ur, double *a)
{
#pragma clang fp contract(on)
    constexpr int c1 = 1, c2 = 1 + D, q0 = c2 + D * (D + 1) / 2;
    const double n = t[0];
    double tr = 0.0, ub = 0.0, uu = 0.0;
    int m = c2;
    for (int i = 0; i < D; ++i) {
        tr += t[m];
        m += D - i;
        ub += Ur[i] * t[c1 + i];
        uu += Ur[i] * Ur[i];
    }
    if (H) tr += t[q0 + D];
    a[0] = n;
    for (int i = 0; i < D; ++i) {
        a[1 + i] = t[c1 + i] + n * Ur[i];
        a[D + 2 + i] = 0.5 * t[q0 + i];
    }
    a[D + 1] = 0.5 * (tr + 2.0 * ub + n * uu);
    for (int i = 0; i < D * (D + 1) / 2; ++i) a[2 * D + 2 + i] = 0.5 * t[c2 + i];
}

// Adds the record r (about Ur) to a (about Uh): density, momentum and energy are absolute; P and Q
// shift exactly with d = Uh - Ur and the record's own sums.
template <int D>
DEVI void record_add(double *a, const double *r, const double *Ur, const double *Uh)
{
#pragma clang fp contract(on)
    const double n = r[0];
    double d[D], b[D], dd = 0.0, db = 0.0, uj = 0.0, uu = 0.0;
    for (int i = 0; i < D; ++i) {
        d[i] = Uh[i] - Ur[i];
        b[i] = 0.5 * (r[1 + i] - n * Ur[i]);
        dd += d[i] * d[i];
        db += d[i] * b[i];
        uj += Ur[i] * r[1 + i];
        uu += Ur[i] * Ur[i];
    }
    const double A = r[D + 1] - uj + 0.5 * uu * n;   // sum w (|c|^2 g + h) / 2 about Ur
    double Pm[D][D];
    int m = 2 * D + 2;
    for (int i = 0; i < D; ++i)
        for (int j = i; j < D; ++j) {
            Pm[i][j] = Pm[j][i] = r[m];
            a[m] += r[m] - b[i] * d[j] - d[i] * b[j] + 0.5 * n * d[i] * d[j];
            ++m;
        }
    for (int i = 0; i < D; ++i) {
        double pd = 0.0;
        for (int j = 0; j < D; ++j) pd += Pm[i][j] * d[j];
        a[D + 2 + i] += r[D + 2 + i] - 2.0 * pd + dd * b[i] - d[i] * A + 2.0 * d[i] * db - 0.5 * n * d[i] * dd;
        a[1 + i] += r[1 + i];
    }
    a[0] += n;
    a[D + 1] += r[D + 1];
}

// A lane's column: the fixed coordinates, weights and row-offset factors.
template <int D>
struct Column {
    double x, y;        // fixed coordinates (3-D: x, y; 2-D: x)
    double w, mo;       // product of the fixed axes' weights / FP32 row-offset factors
    int ix, iy;
};

template <int D, typename TS>
DEVI Column<D> column_at(const P<TS> &p, const LineRec &r, const double *vt)
{
    Column<D> c;
    const int nxi = p.nxi, nax = p.nax;
    c.ix = r.ix;
    c.iy = r.iy;
    c.x = D >= 2 ? vt[c.ix] : 0.0;
    c.y = D == 3 ? vt[nxi + c.iy] : 0.0;
    c.w = D >= 2 ? vt[nax + c.ix] : 1.0;
    if (D == 3) c.w *= vt[nax + nxi + c.iy];
    c.mo = 1.0;
    if (sizeof(TS) == 4) {
        const double *e = vt + 2 * nax;
        if (D >= 2) c.mo = e[c.ix];
        if (D == 3) c.mo *= e[nxi + c.iy];
    }
    return c;
}

// The loop-axis table in LDS: LT doubles per axis position.
//   [0] coordinate, [1..4] w (z - Ur)^m, m = 0..3, [5] FP32 row-offset factor, [6] cell equilibrium's
//   exp factor, [7] index in the per-axis tables, [8 + j] face j's exp factor
// One address and immediate offsets serve every entry of an iteration.
template <int NS>
constexpr int line_lt()
{
    return 8 + NS + (NS & 1);
}

template <int LT, typename TS>
DEVI void stage_axis(const P<TS> &p, int la0, double Ur, double *tab)
{
    for (int t = threadIdx.x; t < p.nxi; t += blockDim.x) {
        const double z = p.axis[la0 + t], c = z - Ur;
        double w = p.axw[la0 + t], *e = tab + t * LT;
        e[0] = z;
#pragma unroll
        for (int m = 0; m < 4; ++m) {
            e[1 + m] = w;
            w *= c;
        }
        e[5] = p.moff[la0 + t];
    }
}

// A wave's walk over its columns, tile by tile: begin(tile, column), then for each iteration
// body(column, byte offset into a row, loop-axis table entry, loaded values) on the lanes whose column
// holds a velocity, then end(tile, column).  load(byte offset, values) issues an iteration's loads.
template <int D, int LT, typename R, typename TS, typename BEGIN, typename LOAD, typename BODY, typename END>
DEVI void walk_columns(const P<TS> &p, const double *vt, const double *tab, BEGIN begin, LOAD load, BODY body, END end)
{
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), nwv = blockDim.x >> 6;
    for (int t = wave; t < p.ntile; t += nwv) {
        const int q0 = __builtin_amdgcn_readfirstlane(p.titer[t]), its = __builtin_amdgcn_readfirstlane(p.titer[t + 1]) - q0;
        const LineRec lr = p.rec[t * 64 + lane];
        unsigned ko = (unsigned)(q0 * 64 + lane) * (unsigned)sizeof(TS);
        constexpr unsigned STEP = 64 * sizeof(TS);
        const Column<D> col = column_at<D>(p, lr, vt);
        begin(t, col);
        const double *e = tab + lr.l * LT;
        const int de = lr.dl * LT, n = lr.n;
#pragma unroll 1
        for (int i = 0; i < its; ++i, ko += STEP, e += de) {
            R cur;
            load(ko, cur);
            if (i < n) body(col, ko, e, cur);
        }
        end(t, col);
    }
}

// Stored value + row offset; the offset is 0 with FP64 storage.
template <typename TS>
DEVI double plus_off(double v, double o)
{
    return sizeof(TS) == 8 ? v : v + o;
}

// FP32 row offset (row_off) of a column's velocity: loop-axis factor at e[5]
template <typename TS>
DEVI double col_off(double mo, const double *e, double pre)
{
    return sizeof(TS) == 8 ? 0.0 : mo * e[5] * pre;
}

// ---------------------------------------------------------------------------------------------
// k_face_lines: S2 face values and the S6 face-moment sums, cell-wise (the work of k_face_values,
// k_face_moments_mx and k_face_moments).  Every face value is written by its upwind cell, with the
// selection of k_face_values; the cell's share of each face's moments (the values it wrote) is
// summed about the cell's previous velocity and left in spart[cell NS + face], one record each.
// Bound by memory at 3-D sizes (48^3 x 24^3 FP64: 16.3 ms, 5.3 TB/s, against 15.1 + 6.9 of the two passes), by
// latency and vector issue at a few thousand cells.  The open faces ride in the first workgroups: alone
// they are one short kernel of few waves (75 x 25 cells: 13 us of a 110 us step).
// ---------------------------------------------------------------------------------------------
#ifndef KFL_WAVES
#define KFL_WAVES 4
#endif
template <int D, bool H, int NS, typename TS>
__global__ __launch_bounds__(LINE_MAXNT) __attribute__((amdgpu_waves_per_eu(D == 3 && H ? 3 : KFL_WAVES, 8))) void k_face_lines(P<TS> p)
{
    constexpr int NV = line_nval<D, H>(), V = NS * NV, NQ = (V + 63) / 64, NM = NMom<D>::v, NA = line_nsum<H>(), LT = 6;
    extern __shared__ __align__(16) double tabs[];   // [velocity table | axis table | sums of the waves]
    double *vt = tabs, *tab = vt + 3 * p.nax + 2, *red = tab + LT * p.nxi;
    const int nob = (p.nopen + NXCD - 1) / NXCD * NXCD;
    if ((int)blockIdx.x < nob) {
        // an open face: k_face_open's values, and their moment record about the owner cell's velocity
        const int i = blockIdx.x;
        if (i >= p.nopen) return;
        stage_vt(p, vt);
        __syncthreads();
        double a[NM];
#pragma unroll
        for (int m = 0; m < NM; ++m) a[m] = 0.0;
        open_face<D, H, NS, true>(p, i, threadIdx.x, p.nvp, blockDim.x, vt, a);
        block_sum<NM>(a, tab + NM, tab);
        if ((int)threadIdx.x < NM) p.opart[(size_t)i * NM + threadIdx.x] = tab[threadIdx.x];
        return;
    }
    int pos, b;
    if (!xcd_block(p.nc, 1, pos, b, nob)) return;
    stage_vt(p, vt);
    const int c = cptr(p.corder)[pos];
    const int la0 = (D - 1) * p.nxi;
    const double Ur[3] = {cptr(p.cU)[3 * c], cptr(p.cU)[3 * c + 1], cptr(p.cU)[3 * c + 2]};
    stage_axis<LT>(p, la0, Ur[D - 1], tab);
    __syncthreads();
    const double dt = cptr(p.dtc)[cptr(p.ccase)[c]];
    const CONST_AS CellSt *st = cptr(p.cst) + c;
    const CONST_AS LineGeo *LG = cptr(p.lgeo) + (size_t)c * NS;
    const CONST_AS Slot *SL = cptr(p.slots) + cptr(p.cs)[c];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), nwv = blockDim.x >> 6;
    const bool inner = st->inner;
    const TS *rowC = p.gb_in + (size_t)c * p.nvp, *hrowC = H ? p.hb_in + (size_t)c * p.nvp : nullptr;
    // the stencil: rows of the neighbours, faces, outward area vectors; with few faces also the
    // gradient and face vectors (the others come from LDS)
    int64_t off[NS];
    int face[NS];
    double Sx[NS], Sy[NS], Sl[NS];
    constexpr bool VEC = D * NS <= 8;
    double Lv[VEC ? NS : 1][D], dv[VEC ? NS : 1][D];
#pragma unroll
    for (int j = 0; j < NS; ++j) {
        off[j] = st->off[j];
        face[j] = LG[j].face;
        Sl[j] = LG[j].Sl;
        Sx[j] = D >= 2 ? LG[j].S[0] : 0.0;
        Sy[j] = D == 3 ? LG[j].S[1] : 0.0;
        if constexpr (VEC) {
            pin(off[j]);
            pin(face[j]);
            pin(Sl[j]);
            if (D >= 2) pin(Sx[j]);
#pragma unroll
            for (int d = 0; d < D; ++d) {
                Lv[j][d] = st->L[j][d];
                dv[j][d] = LG[j].dC[d];
                pin(Lv[j][d]);
                pin(dv[j][d]);
            }
        }
    }
    double tot[NQ];
#pragma unroll
    for (int i = 0; i < NQ; ++i) tot[i] = 0.0;
    double n[NS][NA];
    struct Rows {
        TS g, h, vg[NS], vh[H ? NS : 1];
    };

    auto begin = [&](int, const Column<D> &) {
#pragma unroll
        for (int j = 0; j < NS; ++j)
#pragma unroll
            for (int m = 0; m < NA; ++m) n[j][m] = 0.0;
    };
    auto load = [&](unsigned ko, Rows &r) {
        r.g = ld_at(rowC, ko);
        if (H) r.h = ld_at(hrowC, ko);
#pragma unroll
        for (int j = 0; j < NS; ++j) {
            r.vg[j] = ld_at(p.gb_in + off[j], ko);
            if (H) r.vh[j] = ld_at(p.hb_in + off[j], ko);
        }
    };
    // BND: the cell has boundary faces
    auto body = [&](auto bnd, const Column<D> &col, unsigned ko, const double *e, const Rows &r) {
        constexpr bool BND = decltype(bnd)::value;
        const double z = e[0], gC = r.g, hC = H ? (double)r.h : 0.0;
        auto Lvec = [&](int j, int d) { return VEC ? Lv[VEC ? j : 0][d] : st->L[j][d]; };
        auto dvec = [&](int j, int d) { return VEC ? dv[VEC ? j : 0][d] : LG[j].dC[d]; };
        // outward xi.S without contraction, (x Sx + y Sy) + z Sz
        auto flux_dir = [&](int j) {
#pragma clang fp contract(off)
            const double l = z * Sl[j];
            if (D == 1) return l;
            if (D == 2) return col.x * Sx[j] + l;
            return (col.x * Sx[j] + col.y * Sy[j]) + l;
        };
        // velocities along a face: |xi.S| < VSMALL (none of a slot past the cell's faces: xi.S is a NaN)
        bool mid = false;
#pragma unroll
        for (int j = 0; j < NS; ++j) mid = mid || fabs(flux_dir(j)) < VSMALL;
        const bool anymid = __any(mid);
        double GC[3] = {0, 0, 0}, HC[3] = {0, 0, 0};
        const int wm = BND ? st->wmask : 0;
#pragma unroll
        for (int j = 0; j < NS; ++j) {
            double dg, dh = 0.0;
            if (BND && (wm & (1 << j))) {
                const double a = st->a[j];
                dg = (gC + r.vg[j] * a) - gC;
                if (H) dh = (hC + r.vh[j] * a) - hC;
            } else {
                dg = (double)r.vg[j] - gC;
                if (H) dh = (double)r.vh[j] - hC;
            }
#pragma unroll
            for (int d = 0; d < D; ++d) {
                const double l = Lvec(j, d);
                GC[d] = fma(l, dg, GC[d]);
                if (H) HC[d] = fma(l, dh, HC[d]);
            }
        }
        const double og = col_off<TS>(col.mo, e, vt[3 * p.nax]), oh = H ? col_off<TS>(col.mo, e, vt[3 * p.nax + 1]) : 0.0;
        // g - G.(xi dt / 2); the face values add G.(Cf - C)
        const double hz = 0.5 * z * dt;
        const double hx[3] = {D == 1 ? hz : 0.5 * col.x * dt, D == 2 ? hz : 0.5 * col.y * dt, hz};
        double ga = gC, ha = hC;
#pragma unroll
        for (int d = 0; d < D; ++d) {
            ga = fma(-GC[d], hx[d], ga);
            if (H) ha = fma(-HC[d], hx[d], ha);
        }
        // the face value, stored (own) and added to the face's sums as k_cell will read it
        auto put = [&](int j, bool own, double part, double gf, double hf) {
            if (own) {
                st_at_stream(p.fvg + (size_t)face[j] * p.nvp, ko, gf);
                if (H) st_at_stream(p.fvh + (size_t)face[j] * p.nvp, ko, hf);
            }
            double g = plus_off<TS>((double)(TS)gf, og), h = H ? plus_off<TS>((double)(TS)hf, oh) : 0.0;
            if (anymid) {
                g *= part;
                h *= part;
            }
            line_add<H>(n[j], e + 1, g, h);
        };
#pragma unroll
        for (int j = 0; j < NS; ++j) {
            const double s = flux_dir(j);
            double gf = ga, hf = ha;
#pragma unroll
            for (int d = 0; d < D; ++d) {
                const double dc = dvec(j, d);
                gf = fma(GC[d], dc, gf);
                if (H) hf = fma(HC[d], dc, hf);
            }
            const int kind = BND || anymid ? LG[j].kind : KIND_OWN;
            // the values this cell writes: where it is upwind (outward xi.S; never on KIND_NONE)
            bool mine = s > 0.0, own = true;
            double part = 1.0;
            if (anymid && (kind == KIND_OWN || kind == KIND_NEI)) {
                // |xi.S| < VSMALL: the mean of both reconstructions (discreteVelocity.C:505-515).  Its
                // flux is 0, so that only its moments matter: each cell adds half of its own
                // reconstruction, and the owner's is stored
                const bool m = fabs(s) < VSMALL;
                mine = mine || m;
                own = kind == KIND_OWN || s > 0.0;
                part = m ? 0.5 : 1.0;
            }
            if (BND) {
                if (grad_row(kind)) {
                    // the next step's lagged fixedGradient row n . grad(gbar)
                    const CONST_AS Slot &S = SL[j];
                    double ng = GC[0] * S.dCo[0], nhv = HC[0] * S.dCo[0];
#pragma unroll
                    for (int d = 1; d < D; ++d) {
                        ng += GC[d] * S.dCo[d];
                        nhv += HC[d] * S.dCo[d];
                    }
                    *(TS *)((char *)(p.gBg_out + (size_t)S.bidx * p.nvp) + ko) = (TS)ng;
                    if (H) *(TS *)((char *)(p.gBh_out + (size_t)S.bidx * p.nvp) + ko) = (TS)nhv;
                }
                if (kind == KIND_ZG) {
                    mine = true;
                    gf = gC;
                    hf = hC;
                } else if (kind == KIND_CYC) {
                    mine = true;
                    if (__any(!(s > VSMALL))) {
                        const CONST_AS Slot &S = SL[j];
                        const double dCs[3] = {S.dCs[0], S.dCs[1], S.dCs[2]};
                        const int o = S.other;
                        const unsigned k = ko / (unsigned)sizeof(TS);
                        const double gO = ld_at(p.gb_in + (size_t)o * p.nvp, ko);
                        const double hO = H ? ld_at(p.hb_in + (size_t)o * p.nvp, ko) : 0.0;
                        double GO[3] = {0, 0, 0}, HO[3] = {0, 0, 0};
                        grad_at<D, H, NS>(p, o, k, gO, hO, GO, HO);
                        gf = face_value<D>(KIND_CYC, s, gC, GC, dCs, gO, GO, dCs, S.aux, hx);
                        if (H) hf = face_value<D>(KIND_CYC, s, hC, HC, dCs, hO, HO, dCs, S.aux, hx);
                    }
                }
            }
            if (mine) put(j, own, part, gf, hf);
        }
    };
    auto end =
        [&](int, const Column<D> &col) {
            // the column's sums -> the faces' values, summed over the lanes; with an even number of
            // faces, j and j + NS / 2 together are the first step of lane_sums on their values
            const double cx = col.x - Ur[0], cy = col.y - Ur[1];
            if constexpr (NS % 2 == 0) {
                double v[V / 2];
#pragma unroll
                for (int j = 0; j < NS / 2; ++j) {
                    double e0[NV], e1[NV];
                    line_expand<D, H>(n[j], col.w, cx, cy, e0);
                    line_expand<D, H>(n[j + NS / 2], col.w, cx, cy, e1);
#pragma unroll
                    for (int m = 0; m < NV; ++m) {
                        swap_halves<32>(e0[m], e1[m]);
                        v[j * NV + m] = e0[m] + e1[m];
                    }
                }
                lane_halve<V / 2, 16>(v, lane);
#pragma unroll
                for (int i = 0; i < NQ; ++i) tot[i] += v[i];
            } else {
                double v[V];
#pragma unroll
                for (int j = 0; j < NS; ++j) line_expand<D, H>(n[j], col.w, cx, cy, v + j * NV);
                lane_sums<V>(v, lane);
#pragma unroll
                for (int i = 0; i < NQ; ++i) tot[i] += v[i];
            }
        };
    if (inner)
        walk_columns<D, LT, Rows>(p, vt, tab, begin, load,
                                  [&](const Column<D> &col, unsigned ko, const double *e, const Rows &r) {
                                      body(std::false_type{}, col, ko, e, r);
                                  },
                                  end);
    else
        walk_columns<D, LT, Rows>(p, vt, tab, begin, load,
                                  [&](const Column<D> &col, unsigned ko, const double *e, const Rows &r) {
                                      body(std::true_type{}, col, ko, e, r);
                                  },
                                  end);
#pragma unroll
    for (int i = 0; i < NQ; ++i) {
        const int q = lane_value<V>(lane, i);
        if (q >= 0) red[wave * V + q] = tot[i];
    }
    __syncthreads();
    for (int q = threadIdx.x; q < V; q += blockDim.x) {
        double s = 0.0;
        for (int w = 0; w < nwv; ++w) s += red[w * V + q];
        red[q] = s;
    }
    __syncthreads();
    if ((int)threadIdx.x < NS) {
        double a[NM];
        line_record<D, H>(red + threadIdx.x * NV, Ur, a);
        double *o = p.spart + ((size_t)c * NS + threadIdx.x) * NM;
        for (int m = 0; m < NM; ++m) o[m] = a[m];
    }
}

// Along a column, with z the loop coordinate, an equilibrium's factors are
//   c2 - D - 2 = z (z invRT + B) + P0,  pc = z qz + q0,  Gaussian = t0 * (loop-axis table entry).
// P0 and q0 of a lane from the expanded constants of a face (FaceEq) or a cell:
template <int D, typename FE>
DEVI void line_fixed(const FE &fe, double x, double y, double &P0, double &q0)
{
#pragma clang fp contract(on)
    P0 = fe.C0;
    q0 = fe.Q0;
    if (D >= 2) {
        P0 += x * (x * fe.invRT + fe.B[0]);
        q0 += x * fe.qc[0];
    }
    if (D == 3) {
        P0 += y * (y * fe.invRT + fe.B[1]);
        q0 += y * fe.qc[1];
    }
}

// The cell equilibrium in expanded form.
struct CellEq {
    double invRT, RT, pre, B[3], C0, Q0, qc[3];
};

// What the column form of k_cell needs of the state that formed gbar: the cell equilibrium and
// kr = r / (1 - r) of g~ (s8_cell).  Written by k_face_fin.
struct alignas(64) LineCell {
    double invRT, B[3], qc[3], RT, kr, pre, C0, Q0, dtV, pad[3];
};
static_assert(sizeof(LineCell) == 128, "linecell size");

template <int D>
DEVI void cell_eq(double rho, const double *U, double T, const double *q, double R, double Pr, CellEq &e)
{
#pragma clang fp contract(on)
    EqC k;
    eq_consts(rho, U, T, q, R, Pr, D, k);
    e.invRT = k.invRT;
    e.RT = k.RT;
    e.pre = k.pre;
    double uu = 0.0, uq = 0.0;
    for (int d = 0; d < 3; ++d) {
        e.B[d] = -2.0 * U[d] * k.invRT;
        e.qc[d] = k.qc[d];
        uu += U[d] * U[d];
        uq += U[d] * k.qc[d];
    }
    e.C0 = uu * k.invRT - (D + 2);
    e.Q0 = -uq;
}

// -1/3 g~ + 4/3 gbar with g~ = (gbar - r geq) / (1 - r) = gbar - kr (geq - gbar).  In this form the rounding
// of kr takes nothing from the cell's sums, which geq - gbar does not hold: with cA gbar + cB geq, cA + cB is
// 1 within the last place of cA only, a loss of mass in every step that grows without bound as r nears 1.
DEVI double s8_cell(double g, double geq, double kr)
{
    const double gt = fma(-kr, geq - g, g);
    return fma(4.0 / 3, g, -1.0 / 3 * gt);
}

template <int D, typename TS>
DEVI void line_cell(const P<TS> &p, int c)
{
    const double dt = p.dtc[p.ccase[c]];
    CellEq e;
    cell_eq<D>(p.crho[c], p.cU + 3 * (size_t)c, p.cT[c], p.cq + 3 * (size_t)c, p.R, p.Pr, e);
    const double r = s1_r(dt, p.ctau[c]);
    LineCell lc;
    lc.invRT = e.invRT;
    lc.RT = e.RT;
    lc.pre = e.pre;
    lc.C0 = e.C0;
    lc.Q0 = e.Q0;
    for (int d = 0; d < 3; ++d) {
        lc.B[d] = e.B[d];
        lc.qc[d] = e.qc[d];
    }
    lc.kr = r / (1.0 - r);
    lc.dtV = dt / p.cV[c];
    lc.pad[0] = lc.pad[1] = lc.pad[2] = 0.0;
    p.lcell[c] = lc;
}

// Shakhov equilibrium of a column's velocity (the polynomial form of face_relax).
template <bool H>
DEVI void line_geq(double z, double invRT, double B, double qz, double RT, double P0, double q0, double gB, double kc,
                   double kc2K, double &geq, double &heq)
{
    const double Pv = fma(z, fma(z, invRT, B), P0);
    const double pc = fma(z, qz, q0);
    geq = fma(pc, Pv, 1.0) * gB;
    heq = H ? fma(pc, fma(Pv, kc, kc2K), kc) * (gB * RT) : 0.0;   // kc2K = 2 kc - 2 K
}

// Cell equilibrium's exp factors: fixed axes in tabC, the loop axis in entry 6 of the axis table, and its index
// in entry 7.
template <int LT, typename TS>
DEVI void stage_cell_exp(const P<TS> &p, int la0, const double *U, double invRT, double *tabC, double *tab)
{
    for (int t = threadIdx.x; t < p.nax; t += blockDim.x) {
        const int ax = t / p.nxi;
        const double u = U[ax] - p.axis[t - ax * p.nxi];
        const double e = exp(-(u * u) * (0.5 * invRT));
        if (t >= la0) {
            tab[(t - la0) * LT + 6] = e;
            tab[(t - la0) * LT + 7] = t;
        } else {
            tabC[t] = e;
        }
    }
}

// Product of the fixed axes' entries of a per-axis exp table with stride SD.
template <int D, int SD>
DEVI double column_exp(const double *tab, int nxi, const Column<D> &c)
{
    double e = 1.0;
    if (D >= 2) e = tab[c.ix * SD];
    if (D == 3) e *= tab[(nxi + c.iy) * SD];
    return e;
}

// S1 of the next step over the columns of one cell: row <- (1 - r) g~ + r geq.  g~ of the first
// p.ntl tiles is in LDS (rowL: 64 values, or 64 of g and 64 of h, an iteration), of the others in the
// output row itself.
template <int D, bool H, int LT, bool LDS, typename TS>
DEVI void line_s1(const P<TS> &p, int c, const CellEq &e, const double *tabC, const double *tab, const double *vt,
                  double rn, TS *rowL)
{
    TS *__restrict__ go = p.gb_out + (size_t)c * p.nvp;
    TS *__restrict__ ho = H ? p.hb_out + (size_t)c * p.nvp : nullptr;
    const double mog = vt[3 * p.nax], moh = vt[3 * p.nax + 1], kc2K = 2.0 * p.kc - 2.0 * p.K;
    double g0, P0, q0;
    bool inL = false;
    LDS_AS TS *const rL = (LDS_AS TS *)rowL, *rl = rL;
    struct None {};
    walk_columns<D, LT, None>(
        p, vt, tab,
        [&](int t, const Column<D> &col) {
            g0 = e.pre * column_exp<D, 1>(tabC, p.nxi, col);
            line_fixed<D>(e, col.x, col.y, P0, q0);
            if (LDS) {
                inL = t < p.ntl;
                rl = rL + (inL ? __builtin_amdgcn_readfirstlane(p.titer[t]) : 0) * (H ? 128 : 64) + (threadIdx.x & 63);
            }
        },
        [](unsigned, None &) {},
        [&](const Column<D> &col, unsigned ko, const double *ea, const None &) {
            double gv, hv = 0.0;
            if (LDS && inL) {
                gv = rl[0];
                if (H) hv = rl[64];
                rl += H ? 128 : 64;
            } else {
                gv = ld_at(go, ko);
                if (H) hv = ld_at(ho, ko);
            }
            double geq, heq;
            line_geq<H>(ea[0], e.invRT, e.B[D - 1], e.qc[D - 1], e.RT, P0, q0, g0 * ea[6], p.kc, kc2K, geq, heq);
            const double og = col_off<TS>(col.mo, ea, mog), oh = H ? col_off<TS>(col.mo, ea, moh) : 0.0;
            st_at_stream(go, ko, s1_value(gv, og, rn, geq));
            if (H) st_at_stream(ho, ko, s1_value(hv, oh, rn, heq));
        },
        [](int, const Column<D> &) {});
}

// ---------------------------------------------------------------------------------------------
// k_cell_lines: S7 face relaxation, S8 update and S9 cell moments over velocity columns (k_cell's
// work), one workgroup per cell.  Bound by memory (48^3 x 24^3 FP64: 24.7 -> 19.7 ms, 5.6 TB/s with what
// the L2 misses).  With F1 it also forms the cell macros and the next step's S1;
// the new row of the first p.ntl tiles then stays in LDS and is written to HBM once.
// Dynamic LDS: [velocity table (3 nax + 2) | axis table (LT nxi) | face tables of the fixed axes (NS la0) |
// cell table of the fixed axes (la0) | incoming wall tables (NS nax) | row].
// ---------------------------------------------------------------------------------------------
#ifndef KCL_WAVES
#define KCL_WAVES 4
#endif
template <int D, bool H, int NS, typename TS, bool F1>
__global__ __launch_bounds__(LINE_MAXNT) __attribute__((amdgpu_waves_per_eu(D == 3 && H ? 3 : KCL_WAVES, 8))) void k_cell_lines(P<TS> p)
{
    constexpr int NV = line_nval<D, H>(), NC = NMom<D>::v, NA = line_nsum<H>(), LT = line_lt<NS>();
    static_assert(NV <= 64, "one value per lane");
    extern __shared__ __align__(16) double tabs[];
    __shared__ double red[LINE_MAXW * NV];
    const int nax = p.nax, nxi = p.nxi, la0 = (D - 1) * p.nxi;
    int pos, b;
    if (!xcd_block(p.nc, 1, pos, b)) return;
    double *vt = tabs;
    double *tab = vt + 3 * nax + 2;
    double *tabF = tab + LT * nxi;
    double *tabC = tabF + NS * la0;
    double *tabW = tabC + la0;
    TS *rowL = (TS *)(tabW + NS * nax);
    stage_vt(p, vt);
    const int c = cptr(p.corder)[pos];
    const int cas = cptr(p.ccase)[c];
    const double dt = cptr(p.dtc)[cas];
    const int s0 = cptr(p.cs)[c];
    const int ns = cptr(p.cs)[c + 1] - s0;
    const CONST_AS LineGeo *LG = cptr(p.lgeo) + (size_t)c * NS;
    const TS *__restrict__ rowC = p.gb_in + (size_t)c * p.nvp;
    const TS *__restrict__ hrowC = H ? p.hb_in + (size_t)c * p.nvp : nullptr;
    TS *__restrict__ go = p.gb_out + (size_t)c * p.nvp;
    TS *__restrict__ ho = H ? p.hb_out + (size_t)c * p.nvp : nullptr;

    // state that formed gbar: macros of the previous step
    const double Uc[3] = {cptr(p.cU)[3 * c], cptr(p.cU)[3 * c + 1], cptr(p.cU)[3 * c + 2]};
    const CONST_AS LineCell *LC = cptr(p.lcell) + c;
    stage_axis<LT>(p, la0, Uc[D - 1], tab);
    stage_cell_exp<LT>(p, la0, Uc, LC->invRT, tabC, tab);
    // per face the relaxation factors r pre exp(...) (the first axis carries r pre; the loop axis goes
    // to the axis table) and, on walls, the incoming rho_w pre_w Maxwellian; entries past the cell's
    // faces are 0
    for (int t = threadIdx.x; t < NS * nax; t += blockDim.x) {
        const int j = t / nax, a = t - j * nax;
        const int ax = a / nxi;
        double e = 0.0;
        if (j < ns) {
            const Slot &sj = p.slots[s0 + j];
            const FaceEq &fe = p.feq[sj.face];
            const double u = fe.U[ax] - p.axis[a - ax * nxi];
            e = exp(-(u * u) * (0.5 * fe.invRT));
            if (ax == 0) e *= fe.r * fe.pre;
            if (sj.kind == KIND_WALL) {
                double w = p.wexp[(size_t)sj.bidx * nax + a];
                if (ax == 0) w *= fe.rho_w * fe.pad[1];
                tabW[a * NS + j] = w;
            }
        }
        if (a >= la0) tab[(a - la0) * LT + 8 + j] = e;
        else tabF[a * NS + j] = e;
    }
    __syncthreads();
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), nwv = blockDim.x >> 6;
    const double kc2K = 2.0 * p.kc - 2.0 * p.K;
    const bool plain = cptr(p.cst)[c].plain;
    double tot = 0.0;
    // per lane and face: fixed part of the Gaussian, the polynomials and the flux factor
    double f0[NS], fP[NS], fq[NS], fs[NS], n[NA], c0, cP0, cq0;
    constexpr bool VEC = D * NS <= 8;   // few faces: their constants stay in scalar registers
    // rows of the faces' values (entries past the cell's faces: its first face)
    const TS *fpg[NS], *fph[H ? NS : 1];
#pragma unroll
    for (int j = 0; j < NS; ++j) {
        fpg[j] = p.fvg + (size_t)LG[j].face * p.nvp;
        if (VEC) pin(fpg[j]);
        if (H) {
            fph[j] = p.fvh + (size_t)LG[j].face * p.nvp;
            if (VEC) pin(fph[j]);
        }
    }
    // the faces along the loop axis (in scalar registers with few faces), and the cell
    LineFace LF[VEC ? NS : 1];
#pragma unroll
    for (int j = 0; j < (VEC ? NS : 0); ++j) {
        const CONST_AS LineFace &f = cptr(p.lface)[(size_t)c * NS + j];
        LF[j] = {f.invRT, f.B, f.qz, f.omr, f.Sl, H ? f.RT : 0.0, {0.0, 0.0}};
        pin(LF[j].invRT);
        pin(LF[j].B);
        pin(LF[j].qz);
        pin(LF[j].omr);
        pin(LF[j].Sl);
        if (H) pin(LF[j].RT);
    }
    double kr = LC->kr, cinvRT = LC->invRT, cBl = LC->B[D - 1], cqz = LC->qc[D - 1], cRT = H ? LC->RT : 0.0;
    if (VEC) {
        pin(kr);
        pin(cinvRT);
        pin(cBl);
        pin(cqz);
        if (H) pin(cRT);
    }
    bool inL = false;
    LDS_AS TS *const rL = (LDS_AS TS *)rowL, *rl = rL;

    struct Rows {
        TS g, h, fg[NS], fh[H ? NS : 1];
    };
    walk_columns<D, LT, Rows>(
        p, vt, tab,
        [&](int t, const Column<D> &col) {
            c0 = LC->pre * column_exp<D, 1>(tabC, nxi, col);
            line_fixed<D>(*LC, col.x, col.y, cP0, cq0);
#pragma unroll
            for (int j = 0; j < NS; ++j) {
                const CONST_AS FaceEq &fe = cptr(p.feq)[LG[j].face];
                // 1-D: the loop axis carries everything
                f0[j] = column_exp<D, NS>(tabF + j, nxi, col);
                line_fixed<D>(fe, col.x, col.y, fP[j], fq[j]);
                fs[j] = 0.0;
                if (D >= 2) fs[j] = -col.x * (LG[j].S[0] * LC->dtV);
                if (D == 3) fs[j] = fma(-col.y, LG[j].S[1] * LC->dtV, fs[j]);
            }
#pragma unroll
            for (int m = 0; m < NA; ++m) n[m] = 0.0;
            if (F1) {
                inL = t < p.ntl;
                rl = rL + (inL ? __builtin_amdgcn_readfirstlane(p.titer[t]) : 0) * (H ? 128 : 64) + lane;
            }
        },
        [&](unsigned ko, Rows &r) {
            // the row (no other workgroup reads it) and the values of all faces
            r.g = __builtin_nontemporal_load((const TS *)((const char *)rowC + ko));
            if (H) r.h = __builtin_nontemporal_load((const TS *)((const char *)hrowC + ko));
#pragma unroll
            for (int j = 0; j < NS; ++j) {
                r.fg[j] = ld_at(fpg[j], ko);
                if (H) r.fh[j] = ld_at(fph[j], ko);
            }
        },
        [&](const Column<D> &col, unsigned ko, const double *e, const Rows &r) {
            double gC = r.g, hC = H ? (double)r.h : 0.0;
            const TS *gf = r.fg, *hf = r.fh;
            const double z = e[0];
            const double og = col_off<TS>(col.mo, e, vt[3 * nax]), oh = H ? col_off<TS>(col.mo, e, vt[3 * nax + 1]) : 0.0;
            gC = plus_off<TS>(gC, og);
            if (H) hC = plus_off<TS>(hC, oh);
            double geq, heq;
            line_geq<H>(z, cinvRT, cBl, cqz, cRT, cP0, cq0, c0 * e[6], p.kc, kc2K, geq, heq);
            // S8 (discreteVelocity.C:937-975): -1/3 g~ + 4/3 gbar with g~ = (gbar - r geq) / (1 - r)
            double ag = s8_cell(gC, geq, kr);
            double ah = H ? s8_cell(hC, heq, kr) : 0.0;
            if (plain) {
#pragma unroll
                for (int j = 0; j < NS; ++j) {
                    // S7: (1 - r) g + r geq; S8: the outward flux +-xi.S dt / V
                    const CONST_AS LineFace *lfm = cptr(p.lface) + (size_t)c * NS + j;
                    const LineFace lf = VEC ? LF[VEC ? j : 0] : LineFace{lfm->invRT, lfm->B, lfm->qz, lfm->omr, lfm->Sl, H ? lfm->RT : 0.0, {0.0, 0.0}};
                    double rg, rh;
                    line_geq<H>(z, lf.invRT, lf.B, lf.qz, lf.RT, fP[j], fq[j], f0[j] * e[8 + j], p.kc, kc2K, rg, rh);
                    const double s = fma(z, lf.Sl, fs[j]);
                    ag = fma(s, fma(lf.omr, plus_off<TS>(gf[j], og), rg), ag);
                    if (H) ah = fma(s, fma(lf.omr, plus_off<TS>(H ? hf[j] : 0.0, oh), rh), ah);
                }
            } else {
#pragma unroll
                for (int j = 0; j < NS; ++j) {
                    if (j >= ns) continue;
                    const CONST_AS LineFace *lfm = cptr(p.lface) + (size_t)c * NS + j;
                    const LineFace lf = VEC ? LF[VEC ? j : 0] : LineFace{lfm->invRT, lfm->B, lfm->qz, lfm->omr, lfm->Sl, H ? lfm->RT : 0.0, {0.0, 0.0}};
                    const CONST_AS Slot &S = cptr(p.slots)[s0 + j];
                    const int kind = S.kind;
                    const double Sv[3] = {S.S[0], S.S[1], S.S[2]};
                    const double so = dotnc(D == 1 ? z : col.x, D == 2 ? z : (D == 3 ? col.y : 0.0), D == 3 ? z : 0.0, Sv);
                    double g = plus_off<TS>(gf[j], og), h = H ? plus_off<TS>(hf[j], oh) : 0.0;
                    // S7 (discreteVelocity.C:867-920): on symmetry, far-field, fixed and zeroGradient
                    // patches and walls only the outgoing values relax (their operators are no-ops);
                    // incoming wall values are rho_w M_w; on a symmetryPlane every value relaxes (the
                    // field operation, 880-881), the outgoing ones once more (905-920)
                    const bool all = kind == KIND_OWN || kind == KIND_NEI || kind == KIND_CYC || kind == KIND_SPL;
                    if (kind == KIND_WALL && !(so > 0)) {
                        g = tabW[(int)e[7] * NS + j];
                        if (D >= 2) g *= tabW[col.ix * NS + j];
                        if (D == 3) g *= tabW[(nxi + col.iy) * NS + j];
                        if (H) h = g * (p.R * cptr(p.feq)[S.face].pad[0]) * p.kc;
                    } else if (all || so > 0) {
                        double rg, rh;
                        line_geq<H>(z, lf.invRT, lf.B, lf.qz, lf.RT, fP[j], fq[j], f0[j] * e[8 + j], p.kc, kc2K, rg, rh);
                        g = fma(lf.omr, g, rg);
                        if (H) h = fma(lf.omr, h, rh);
                        if (kind == KIND_SPL && so > 0) {
                            g = fma(lf.omr, g, rg);
                            if (H) h = fma(lf.omr, h, rh);
                        }
                    }
                    const double s = fma(z, lf.Sl, fs[j]);
                    ag = fma(s, g, ag);
                    if (H) ah = fma(s, h, ah);
                }
            }
            const TS sg = (TS)(sizeof(TS) == 8 ? ag : ag - og), sh = (TS)(sizeof(TS) == 8 ? ah : ah - oh);
            if (F1 && inL) {
                rl[0] = sg;
                if (H) rl[64] = sh;
                rl += H ? 128 : 64;
            } else {
                *(TS *)((char *)go + ko) = sg;
                if (H) *(TS *)((char *)ho + ko) = sh;
            }
            line_add<H>(n, e + 1, ag, ah);
        },
        [&](int, const Column<D> &col) {
            double v[NV];
            line_expand<D, H>(n, col.w, col.x - Uc[0], col.y - Uc[1], v);
            lane_sums<NV>(v, lane);
            tot += v[0];
        });
    {
        const int q = lane_value<NV>(lane, 0);
        if (q >= 0) red[wave * NV + q] = tot;
    }
    __syncthreads();
    double tv[NV];
#pragma unroll
    for (int q = 0; q < NV; ++q) {
        double s = 0.0;
        for (int w = 0; w < nwv; ++w) s += red[w * NV + q];
        tv[q] = s;
    }
    double a[NC];
    line_record<D, H>(tv, Uc, a);
    if (!F1) {
        if (threadIdx.x == 0)
            for (int m = 0; m < NC; ++m) p.cpart[(size_t)c * NC + m] = a[m];
        return;
    }
    // F1: the work of k_cell_fin and k_cell_s1_lines for this cell, with their arithmetic
    double rho, U[3], T, tau, q[3];
    finish_moments<D>(a, Uc, p.R, p.K, p.muc[cas], p.omega, p.Tref, rho, U, T, tau, q);
    const double fqc = q_fac(tau, dt * p.Pr);
    for (int d = 0; d < 3; ++d) q[d] = fqc * q[d];
    if (threadIdx.x == 0) {
        p.crho[c] = rho;
        p.cT[c] = T;
        p.ctau[c] = tau;
        for (int d = 0; d < 3; ++d) {
            p.cU[3 * c + d] = U[d];
            p.cq[3 * c + d] = q[d];
        }
        if (!(rho > 0.0) || !(T > 0.0) || !isfinite(rho) || !isfinite(T) || !isfinite(tau)) p.flag[0] = 1;
    }
    CellEq en;
    cell_eq<D>(rho, U, T, q, p.R, p.Pr, en);
    // every lane is past the velocity loop (the barrier above): the cell's exp factors can be rebuilt
    stage_cell_exp<LT>(p, la0, U, en.invRT, tabC, tab);
    __syncthreads();
    line_s1<D, H, LT, true>(p, c, en, tabC, tab, vt, s1_r(dt, tau), rowL);
}

// k_cell_s1_lines: the next step's S1 as a kernel of its own (DUGKS_FUSE_S1=0), with the arithmetic
// of k_cell_lines' tail.
template <int D, bool H, typename TS>
__global__ __launch_bounds__(LINE_MAXNT) void k_cell_s1_lines(P<TS> p)
{
    constexpr int LT = 8;
    __shared__ double tab[LT * 64];
    __shared__ double tabC[NAXMAX];
    __shared__ double vt[VT_SIZE];
    const int c = blockIdx.x, la0 = (D - 1) * p.nxi;
    stage_vt(p, vt);
    const double dt = cptr(p.dtc)[cptr(p.ccase)[c]];
    const double Un[3] = {cptr(p.cU)[3 * c], cptr(p.cU)[3 * c + 1], cptr(p.cU)[3 * c + 2]};
    const double qn[3] = {cptr(p.cq)[3 * c], cptr(p.cq)[3 * c + 1], cptr(p.cq)[3 * c + 2]};
    CellEq en;
    cell_eq<D>(cptr(p.crho)[c], Un, cptr(p.cT)[c], qn, p.R, p.Pr, en);
    stage_axis<LT>(p, la0, Un[D - 1], tab);
    stage_cell_exp<LT>(p, la0, Un, en.invRT, tabC, tab);
    __syncthreads();
    line_s1<D, H, LT, false>(p, c, en, tabC, tab, vt, s1_r(dt, cptr(p.ctau)[c]), (TS *)tab);
}
