// gf_therm.h -- the proven thermal step (FP64 temperature) as marching column strips.
//
// src/fl_therm.f90:393-598: the reference's in-place Gauss-Seidel update reads the NEW
// values of (j-1,i), (j,i-1) and (j+1,i-1).  Here one wave of 64 lanes holds 64
// consecutive rows of one column, one node a lane, and marches from column to column
// in the reference's order.  When it comes to column i, its values of column i-1 are
// final, so only the coupling down the column is left to iterate: the wave applies the
// update to its column until no bit changes (each application moves the new values one
// row on; the coupling of rows is weak, so three to five do).  Everything lives in registers:
// the row above and below come by lane shifts (DPP), the element column just formed is
// kept for the next node column, and the loads of the columns ahead are in flight while
// a column is computed.  There is no LDS traffic and no barrier.
//
// What bounds it: VALU issue where the mesh fills the SIMDs, about 270 FP64 operations
// and 150 others (lane shifts among them) a column; the latency of that chain, 1.3 us a
// column, where a SIMD holds one wave.  The tiles it replaced (64 x 16 nodes in LDS, a
// workgroup barrier per application, 58% of the nodes evaluated in halos) waited on LDS
// and barriers; their thermal step took 137 us on 2001x1001 nodes, this one 95, and on
// square cells (902x302 nodes), where their four halo columns needed a second pass in
// every step, 125 us against 30.
//
// Strips: rows are cut into strips of 64 lanes that overlap by 2 * TS_HB rows (none at
// the mesh's top and bottom), columns into strips of `w` output columns that start
// some halo columns (therm_halo) and one ring column further left.  The ring and
// the outermost rows only hold the starting iterate.  A strip's values in its halo rows and columns are not exact; what
// it saves of them (its border) is compared with the values of the strips that own
// those nodes (therm_check_one), which proves the assembled result.
#pragma once

#define TS_HB 6                  // rows of a strip above and below its output rows: one ring row, five halo rows
#define TS_HI_MAX 8              // most halo columns left of its output columns (after one ring column)
#define TS_OJ (64 - 2 * TS_HB)   // output rows of an inner strip
#define TS_SWEEP0 2              // applications before the first stillness test
#define TS_MAXSWEEP 48
#define TS_NB(w) (2 * (w) + 64)  // border values of a strip: row above, row below, column to the left

// The boundary conditions (:575-598) overwrite rows 1 and nz and columns 1 and nx.  The
// values before them are what the border check and a further pass read, and what the
// next call's rows 1 and nz start from; they go to a ring buffer of GF_NPRE slots of
// 2 nx + 2 nz values: row 1, row nz, column 1, column nx.
#define GF_NPRE 4
// slots of a call: pass p writes slot[p & 1]; the last two calls' final values (hist of
// them are valid)
struct ThermSlots {
    int cur[2], prev, prev2, hist;
};
// consecutive calls number `call` turn three slots over; an odd pass uses the fourth
__host__ __device__ inline ThermSlots therm_slots(int call, int hist)
{
    const int c = call % 3;
    return ThermSlots{{c, 3}, (c + 2) % 3, (c + 1) % 3, hist};
}
GF_DEV double *therm_pre(const GfDevParams *P, const GfDevArrays &A, int slot)
{
    return A.tpre + (long)slot * 2 * (P->nx + P->nz);
}

// Halo columns of a strip: each damps what the ring's start leaves by the coupling of
// columns c = diff dt / dx^2, and that error is some 1e-5 of a value's change (rows 1
// and nz, whose start follows the last two calls).  Enough of them that c^hi <= 1e-11
// (at least 2): at c = 1.3e-2 (901x301 cells of 333 m) 4, 5 and 6 columns need a further
// pass in 45%, 2% and none of the steps; more columns only cost their own time, and
// what a strip leaves unsettled the border check finds.
GF_DEV int therm_halo(const GfDevParams *P, double dt)
{
    const double dx = P->rxbo / (double)(P->nx - 1), c = P->diff_max * dt / (dx * dx);
    int hi = 2;
    for (double v = c * c; v > 1.0e-11 && hi < TS_HI_MAX; v *= c) hi++;
    return hi;
}

struct ThermGeo {
    int nz, nx, w, nr, ns;  // row strips, column strips
};
GF_DEV ThermGeo therm_geo(const GfDevParams *P, int w)
{
    ThermGeo g;
    g.nz = P->nz;
    g.nx = P->nx;
    g.w = w;
    g.nr = g.nz <= 64 ? 1 : (g.nz - 2 * TS_HB + TS_OJ - 1) / TS_OJ;
    g.ns = (g.nx + w - 1) / w;
    return g;
}
// strip t (row strips fastest): row of lane 0, first and last output lane, output columns
struct ThermStrip {
    int jb, fo, lo, c0, c1;
    bool top, bot;  // it holds the mesh's first, last row
};
GF_DEV ThermStrip therm_strip_of(const ThermGeo &g, int t)
{
    ThermStrip s;
    const int r = t % g.nr, c = t / g.nr;
    s.jb = 1 + r * TS_OJ;
    s.top = r == 0;
    s.bot = r == g.nr - 1;
    s.fo = s.top ? 0 : TS_HB;
    s.lo = s.bot ? g.nz - s.jb : 63 - TS_HB;
    s.c0 = c * g.w + 1;
    s.c1 = min(s.c0 + g.w - 1, g.nx);
    return s;
}

// lane l gets the value of lane l-1 (row above; 0 in lane 0) or of lane l+1 (row below;
// 0 in lane 63)
GF_DEV int lane_up(int v) { return __builtin_amdgcn_update_dpp(0, v, 0x138, 0xf, 0xf, true); }
GF_DEV int lane_dn(int v) { return __builtin_amdgcn_update_dpp(0, v, 0x130, 0xf, 0xf, true); }
GF_DEV double lane_up(double v) { return __hiloint2double(lane_up(__double2hiint(v)), lane_up(__double2loint(v))); }
GF_DEV double lane_dn(double v) { return __hiloint2double(lane_dn(__double2hiint(v)), lane_dn(__double2loint(v))); }

// K(a,b) products, ra13, P = dummye ra13 and Q = 0.5 diff / area of one triangle
struct ThermTri {
    double k11, k12, k13, k22, k23, k33, ra, p, q;
};
// ar, inv: area entry and its reciprocal (both 0 where there is no element: every value
// is then 0 and the triangle adds nothing, bit for bit)
GF_DEV ThermTri therm_tri(const double d[6], double inv, double dm, double hdf)
{
    ThermTri t;
    t.ra = div_fma(inv, 6.0, GF_RSIX);
    t.p = dm * t.ra;
    t.q = hdf * inv;
    t.k11 = KAB(d, 1, 1);
    t.k12 = KAB(d, 1, 2);
    t.k13 = KAB(d, 1, 3);
    t.k22 = KAB(d, 2, 2);
    t.k23 = KAB(d, 2, 3);
    t.k33 = KAB(d, 3, 3);
    return t;
}

// 1 / d, correctly rounded for an operand that rcp_safe accepts: two Newton steps from
// the hardware's estimate and a last step from the exact remainder (the steps of an IEEE
// division without the scaling that keeps extreme exponents in range)
GF_DEV double rcp_core(double d)
{
    double y = __builtin_amdgcn_rcp(d);
    y = __builtin_fma(__builtin_fma(-d, y, 1.0), y, y);
    y = __builtin_fma(__builtin_fma(-d, y, 1.0), y, y);
    return __builtin_fma(__builtin_fma(-d, y, 1.0), y, y);
}
// |d| in [2^-400, 2^400], and a significand that is not all ones (the operands for which
// the last step need not round correctly: Markstein's exception)
GF_DEV bool rcp_safe(double d)
{
    const unsigned h = (unsigned)__double2hiint(d), e = (h >> 20) & 0x7ffu;
    return e - (1023u - 400u) <= 800u && ((h | 0xfff00000u) & (unsigned)__double2loint(d)) != 0xffffffffu;
}
// 1 / a where a = RN(1 / d), correctly rounded where rcp_safe(a): the remainder 1 - a d is
// exact and d is within one ulp of 1 / a, so one step from d does
GF_DEV double rcp_back(double a, double d) { return __builtin_fma(__builtin_fma(-a, d, 1.0), d, d); }

struct ThermIter {
    const double *xin;  // starting iterate of a pass > 0
    double *xout;
    int arp;            // the areas of the last move are pending (formed from the coordinates)
    int pass;
};

// One strip.  MODE, the start: 0 the old temperature, 1 xin, 2 the extrapolation
// 2 temp - temp0.  sPh: den, cp, 0.5 diff, 1 / cp per phase (LDS).
template <bool DIS, int MODE>
GF_DEV void therm_strip(const GfDevParams *__restrict__ P, GfDevClock *ck, const GfDevArrays &A, const ThermGeo &g,
                        int t, const ThermIter &it, const ThermSlots &sl, double *bord, double dt,
                        const double (*sPh)[GF_MAXPH])
{
    t = __builtin_amdgcn_readfirstlane(t);
    const int lane = threadIdx.x % 64;
    const ThermStrip s = therm_strip_of(g, t);
    const int nz = g.nz, nx = g.nx, row = s.jb + lane;
    const unsigned nn = (unsigned)nz * nx, ne = (unsigned)(nz - 1) * (nx - 1);
    constexpr unsigned OOB = 0x80000000u;  // past every array: loads read 0, stores are dropped
    const unsigned nvo = row <= nz ? (unsigned)(row - 1) * 8u : OOB;
    const bool erow = row < nz && lane < 63;
    const unsigned evo = erow ? (unsigned)(row - 1) * 8u : OOB, evi = erow ? (unsigned)(row - 1) * 4u : OOB;
    const Buf bT = mkbuf(A.temp, 8ull * nn), bC = mkbuf(A.cord, 16ull * nn),
              bG = mkbuf(MODE == 1 ? it.xin : A.temp0, 8ull * nn), bX = mkbuf(it.xout, 8ull * nn),
              bA = mkbuf(A.area, 16ull * ne), bS = mkbuf(A.source, 8ull * ne), bI = mkbuf(A.iphase, 4ull * ne),
              bH = mkbuf(A.shrheat, 8ull * ne);
    const unsigned npre = 2u * (nx + nz);
    const bool edge = s.top || s.bot;  // (uniform)
    const bool erow1 = row == 1, erown = row == nz;
    // start of rows 1 and nz: the values before the boundary conditions of the last two
    // calls, carried on (pass 0), or those of the last pass (the iterate's own boundary
    // rows hold the conditions)
    const int pslot = MODE == 1 ? sl.cur[(it.pass - 1) & 1] : sl.prev;
    const Buf bP = mkbuf(A.tpre + (long)pslot * npre, 8ull * npre),
              bP2 = mkbuf(A.tpre + (long)sl.prev2 * npre, 8ull * npre),
              bW = mkbuf(A.tpre + (long)sl.cur[it.pass & 1] * npre, 8ull * npre);
    const unsigned pvo = erow1 ? 0u : erown ? 8u * nx : OOB;  // row arrays, + 8 (i - 1)
    const unsigned pco = row <= nz ? 8u * (2 * nx + row - 1) : OOB;  // column arrays, + 8 nz for column nx
    const bool pedge = edge && (MODE == 1 || (MODE == 2 && sl.hist > 0));
    const bool plin = MODE == 2 && sl.hist > 1;

    struct Node {
        double x, y, t, g, p, p2;
    };
    auto load_node = [&](int i) {
        Node n{0, 0, 0, 0, 0, 0};
        if (i <= min(nx, s.c1 + 1)) {  // (uniform; i >= 1)
            const unsigned so = (unsigned)nz * (unsigned)(i - 1) * 8u;
            n.x = bld(bC, nvo, so);
            n.y = bld(bC, nvo, so + 8u * nn);
            n.t = bld(bT, nvo, so);
            if (MODE != 0) n.g = bld(bG, nvo, so);
            if (pedge) {
                n.p = bld(bP, pvo, 8u * (i - 1));
                if (plin) n.p2 = bld(bP2, pvo, 8u * (i - 1));
            }
            if (MODE == 1 && (i == 1 || i == nx)) {  // (the iterate's boundary columns, likewise)
                n.g = bld(bP, pco, i == 1 ? 0u : 8u * nz);
            }
        }
        return n;
    };
    struct Elem {
        double a0, a1, src, sh;
        int ph;
    };
    auto load_elem = [&](int i) {
        Elem e{0, 0, 0, 0, 1};
        if (i <= min(nx - 1, s.c1)) {
            const unsigned ec = (unsigned)(nz - 1) * (unsigned)(i - 1);
            e.src = bld(bS, evo, ec * 8u);
            e.ph = bldi(bI, evi, ec * 4u);
            if (!it.arp) {
                e.a0 = bld(bA, evo, ec * 8u);
                e.a1 = bld(bA, evo, (ec + ne) * 8u);
            }
            if (DIS) e.sh = bld(bH, evo, ec * 8u);
        }
        return e;
    };
    auto start_of = [&](const Node &n) {
        double v = MODE == 0 ? n.t : MODE == 1 ? n.g : 2.0 * n.t - n.g;
        if (pedge && (erow1 || erown)) v = plin ? 2.0 * n.p - n.p2 : n.p;
        return v;
    };

    const int hi = __builtin_amdgcn_readfirstlane(therm_halo(P, dt));
    const int ib = max(1, s.c0 - hi - 1);
    const bool has_ring = s.c0 - hi > 1;  // column ib only holds the start
    // lanes that hold the start in every column (the ring rows), or no node
    const bool hold = (lane == 0 && !s.top) || (lane == 63 && !s.bot) || row > nz;

    Node n0 = load_node(ib), n1 = load_node(ib + 1);
    Elem e0 = load_elem(ib);
    double ydn0 = lane_dn(n0.y), xdn0 = lane_dn(n0.x), tdn0 = lane_dn(n0.t);
    double xl = 0.0, xd = 0.0;  // X(j, i-1), X(j+1, i-1)
    // element column i-1: triangle B one row up, A and B of this row
    double lB13 = 0, lB23 = 0, lB33 = 0, lBp = 0, lBq = 0, lBr = 0;
    double mA13 = 0, mA23 = 0, mA33 = 0, mAp = 0, mAq = 0, mAr = 0;
    double mB11 = 0, mB12 = 0, mB13 = 0, mBp = 0, mBq = 0, mBr = 0;
    bool still = true;
    for (int i = ib; i <= s.c1; i++) {
        // the loads of the columns ahead
        const Node n2 = load_node(i + 2);
        const Elem e1 = load_elem(i + 1);
        // ---- element column i (between node columns i and i+1)
        const double ydn1 = lane_dn(n1.y), xdn1 = lane_dn(n1.x), tdn1 = lane_dn(n1.t);
        const int phs = e0.ph >= 1 && e0.ph <= GF_MAXPH ? e0.ph - 1 : 0;  // (0 where there is no element)
        const bool eok = erow && i < nx;
        ThermTri ta, tb;
        {
            double ar0 = e0.a0, ar1 = e0.a1, inv0, inv1;
            if (it.arp) {
                const double xc[5] = {0.0, n0.x, xdn0, n1.x, xdn1}, yc[5] = {0.0, n0.y, ydn0, n1.y, ydn1};
                const double det0 = move_det(xc, yc, 0), det1 = move_det(xc, yc, 1);
                ar0 = rcp_core(det0);
                ar1 = rcp_core(det1);
                inv0 = rcp_back(ar0, det0);
                inv1 = rcp_back(ar1, det1);
                if (__any(eok && !(rcp_safe(det0) && rcp_safe(det1) && rcp_safe(ar0) && rcp_safe(ar1)))) {
                    ar0 = 1.0 / det0;
                    ar1 = 1.0 / det1;
                    inv0 = 1.0 / ar0;
                    inv1 = 1.0 / ar1;
                }
            } else {
                inv0 = rcp_core(ar0);
                inv1 = rcp_core(ar1);
                if (__any(eok && !(rcp_safe(ar0) && rcp_safe(ar1)))) {
                    inv0 = 1.0 / ar0;
                    inv1 = 1.0 / ar1;
                }
            }
            ar0 = eok ? ar0 : 0.0;
            ar1 = eok ? ar1 : 0.0;
            inv0 = eok ? inv0 : 0.0;
            inv1 = eok ? inv1 : 0.0;
            // dummye = (source + dissip / den) / cp (:405-414; + 0 without shear heating)
            const double sd = DIS ? e0.src + e0.sh / sPh[0][phs] : e0.src + 0.0, cp = sPh[1][phs];
            double dm = div_fma(sd, cp, sPh[3][phs]);
            if (__any(eok && sd != 0.0 && !(rcp_safe(sd) && rcp_safe(cp)))) dm = sd / cp;
            dm = eok ? dm : 0.0;
            const double hdf = sPh[2][phs];
            const double y1 = n0.y, y2 = ydn0, y3 = n1.y, y4 = ydn1, x1 = n0.x, x2 = xdn0, x3 = n1.x, x4 = xdn1;
            const double da[6] = {(y2 - y3) * ar0, (y3 - y1) * ar0, (y1 - y2) * ar0,
                                  (x3 - x2) * ar0, (x1 - x3) * ar0, (x2 - x1) * ar0};
            const double db[6] = {(y2 - y4) * ar1, (y4 - y3) * ar1, (y3 - y2) * ar1,
                                  (x4 - x2) * ar1, (x3 - x4) * ar1, (x2 - x3) * ar1};
            ta = therm_tri(da, inv0, dm, hdf);
            tb = therm_tri(db, inv1, dm, hdf);
        }
        // one row up: element row j-1 for node row j
        const double uA12 = lane_up(ta.k12), uA22 = lane_up(ta.k22), uA23 = lane_up(ta.k23);
        const double uAp = lane_up(ta.p), uAq = lane_up(ta.q), uAr = lane_up(ta.ra);
        const double uB12 = lane_up(tb.k12), uB22 = lane_up(tb.k22), uB23 = lane_up(tb.k23);
        const double uBp = lane_up(tb.p), uBq = lane_up(tb.q), uBr = lane_up(tb.ra);
        double x = start_of(n0);
        if (!(has_ring && i == ib)) {  // (uniform)
            // ---- node column i: t1 B of (j-1,i-1), t2 A of (j-1,i), t3 B of (j-1,i),
            // t4 A of (j,i-1), t5 B of (j,i-1), t6 A of (j,i)
            const double tme = n0.t, tur = lane_up(n1.t);  // T(j,i), T(j-1,i+1)
            const double area_n = (((((0.0 + lBr) + uAr) + uBr) + mAr) + mBr) + ta.ra;
            // a lane that holds its start: told = start, 1/area = 0 (a zero increment)
            double rarea = rcp_core(area_n);
            if (__any(!hold && !rcp_safe(area_n))) rarea = 1.0 / area_n;
            rarea = hold ? 0.0 : rarea;
            const double told = hold ? x : tme;
            const double xl12 = xl * lB23, c13 = tme * lB33;             // t1: K13 K23 K33
            const double c22 = tme * uA22, c23 = tur * uA23;             // t2
            const double qs3 = uBq * (tur * uB12 + tme * uB22 + n1.t * uB23);
            const double qs4 = mAq * ((xl * mA13 + xd * mA23) + tme * mA33);
            const double qs5 = mBq * ((tme * mB11 + xd * mB12) + tdn0 * mB13);
            const double qs6 = ta.q * (tme * ta.k11 + tdn0 * ta.k12 + n1.t * ta.k13);
            auto eval = [&](double xu) {
                double rhs = 0.0;
                rhs = rhs + lBp - lBq * ((xu * lB13 + xl12) + c13);
                rhs = rhs + uAp - uAq * ((xu * uA12 + c22) + c23);
                rhs = rhs + uBp - qs3;
                rhs = rhs + mAp - qs4;
                rhs = rhs + mBp - qs5;
                rhs = rhs + ta.p - qs6;
                return told + div_fma(rhs * dt, area_n, rarea);
            };
            int nsweep = 0;
#pragma unroll
            for (; nsweep < TS_SWEEP0; nsweep++) x = eval(lane_up(x));
            for (;;) {
                const double xn = eval(lane_up(x));
                const bool ch = __double_as_longlong(xn) != __double_as_longlong(x);
                x = xn;
                nsweep++;
                if (!__any(ch)) break;
                if (nsweep >= TS_MAXSWEEP) {
                    still = false;
                    break;
                }
            }
        }
        // ---- results of column i
        if (i >= s.c0) {
            const bool out = lane >= s.fo && lane <= s.lo;
            const unsigned so = (unsigned)nz * (unsigned)(i - 1) * 8u;
            const unsigned vo = out ? nvo : OOB;
            double v = x;
            if (edge) {
                // before the conditions: kept apart
                bst(bW, out ? pvo : OOB, 8u * (i - 1), x);
                double vb = P->bot_bc;
                if (P->itemp_bc != 1) {
                    vb = x;
                    if (P->itemp_bc == 2) {
                        const int phu = lane_up(phs);
                        vb = lane_up(x) + P->bot_bc * (lane_up(n0.y) - n0.y) / PHASE(phu + 1).conduct;
                    }
                }
                if (erown) v = vb;
                if (erow1) v = P->t_top;
            }
            // the side columns take their neighbours' values (:590-598)
            if (i == 1 || i == nx) {
                bst(bW, out ? pco : OOB, i == 1 ? 0u : 8u * nz, x);
            } else {
                bst(bX, vo, so, v);
                if (i == 2) bst(bX, vo, 0u, v);
                if (i == nx - 1) bst(bX, vo, so + 8u * nz, v);
            }
            // border: the row above the output rows, the row below them
            if (g.nr > 1) {
                const unsigned k = (unsigned)(i - s.c0);
                const int b = lane == s.fo - 1 ? 0 : lane == s.lo + 1 ? 1 : -1;
                if (b >= 0 && !(b == 0 && s.top) && !(b == 1 && s.bot)) bord[b * g.w + k] = x;
            }
        } else if (i == s.c0 - 1) {
            bord[2 * g.w + lane] = x;
        }
        // ---- on to column i+1
        xl = x;
        xd = lane_dn(x);
        lB13 = lane_up(tb.k13); lB23 = uB23; lB33 = lane_up(tb.k33); lBp = uBp; lBq = uBq; lBr = uBr;
        mA13 = ta.k13; mA23 = ta.k23; mA33 = ta.k33; mAp = ta.p; mAq = ta.q; mAr = ta.ra;
        mB11 = tb.k11; mB12 = tb.k12; mB13 = tb.k13; mBp = tb.p; mBq = tb.q; mBr = tb.ra;
        n0 = n1;
        n1 = n2;
        e0 = e1;
        xdn0 = xdn1;
        ydn0 = ydn1;
        tdn0 = tdn1;
    }
    if (!still && lane == 0) atomicOr(&ck->therm_pass_changed[it.pass], 2u);
}

// by the lanes of one wave, for that wave
GF_DEV void therm_phase_table(const GfDevParams *__restrict__ P, double (*sPh)[GF_MAXPH])
{
    const int q = threadIdx.x % 64;
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();  // (the wave's reads of another model's table are done)
    if (q < GF_MAXPH) {
        sPh[0][q] = P->ph[q].den;
        sPh[1][q] = P->ph[q].cp;
        sPh[2][q] = 0.5 * P->ph[q].diff;
        sPh[3][q] = 1.0 / P->ph[q].cp;
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

// pass 0 (mode 0 or 2) or, with launches per phase, a fallback pass: one wave a strip
template <bool DIS, int MODE>
__global__ void __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(3)))
k_therm_strip(const GfDevParams *__restrict__ P, GfDevClock *ck, GfDevArrays A, int w, int pass, int arp, ThermSlots sl,
              int ops)
{
    if (ops && blockIdx.x == 0 && threadIdx.x == 0) clock_op(ck, ops);  // (fields nothing here reads)
    __shared__ double sPh[4][GF_MAXPH];
    if (pass > 0 && ck->therm_pass_changed[pass - 1] == 0u) return;  // already proven
    const ThermGeo g = therm_geo(P, w);
    const int nt = g.nr * g.ns, q = (nt + 7) / 8;  // XCD x runs strips [x q, (x+1) q)
    const int t = (int)(blockIdx.x % 8) * q + (int)(blockIdx.x / 8);
    if ((int)(blockIdx.x / 8) >= q || t >= nt) return;
    therm_phase_table(P, sPh);
    const ThermIter it{pass % 2 == 1 ? A.xa : A.xb, pass % 2 == 0 ? A.xa : A.xb, arp, pass};
    therm_strip<DIS, MODE>(P, ck, A, g, t, it, sl, A.tbord + (long)t * TS_NB(w), ck->dt, sPh);
}

// Compares border value t of the strips with the value its owner wrote.  A node whose
// values differ is harmless when every output node of this strip that reads it still
// satisfies x = F(x) with the global values: those (at most three) are evaluated again
// here.  Any remaining difference (or a strip that did not settle) asks for another
// pass.
GF_DEV void therm_check_one(const GfDevParams *__restrict__ P, GfDevClock *ck, const GfDevArrays &A,
                            const ThermGeo &g, long t, int pass, int arp, const ThermSlots &sl)
{
    const int nb = TS_NB(g.w);
    if (t >= (long)g.nr * g.ns * nb) return;
    const int strip = (int)((unsigned)t / (unsigned)nb), k = (int)((unsigned)t % (unsigned)nb);
    const ThermStrip s = therm_strip_of(g, strip);
    int lane, i;
    if (k < g.w) {  // the row above the output rows
        if (s.top) return;
        lane = s.fo - 1;
        i = s.c0 + k;
    } else if (k < 2 * g.w) {  // the row below them (read from the next column: not the last)
        if (s.bot) return;
        lane = s.lo + 1;
        i = s.c0 + k - g.w;
        if (i >= s.c1) return;
    } else {  // the column to the left: the output rows and the one below
        lane = k - 2 * g.w;
        i = s.c0 - 1;
        if (i < 1 || lane < s.fo || lane > s.lo + (s.bot ? 0 : 1)) return;
    }
    if (i > s.c1) return;
    const int nz = g.nz, nx = g.nx, j = s.jb + lane;
    const double *__restrict__ x = (pass % 2 == 0) ? A.xa : A.xb;
    const double *__restrict__ pre = therm_pre(P, A, sl.cur[pass & 1]);
    // the pass's value before the boundary conditions
    auto X = [&](int jj, int ii) -> double {
        if (jj == 1) return pre[ii - 1];
        if (jj == nz) return pre[nx + ii - 1];
        if (ii == 1) return pre[2 * nx + jj - 1];
        if (ii == nx) return pre[2 * nx + nz + jj - 1];
        return x[IN(jj, ii)];
    };
    const long long a = __double_as_longlong(A.tbord[t]), b = __double_as_longlong(X(j, i));
    if (a == b) return;
    const int dj[3] = {1, 0, -1}, di[3] = {0, 1, 1};  // read as up, left, left-down
    const double dt = ck->dt;
    auto T = [&](int jj, int ii) { return A.temp[IN(jj, ii)]; };  // the old temperature
    bool bad = false;
#pragma unroll
    for (int q = 0; q < 3; q++) {
        const int mj = j + dj[q], mi = i + di[q];
        if (mj < s.jb + s.fo || mj > s.jb + s.lo || mi < s.c0 || mi > s.c1) continue;
        ThermCoef c;
        therm_coef(P, A, mj, mi, T, c, arp);
        const double xu = mj > 1 ? X(mj - 1, mi) : 0.0;
        const double xl = mi > 1 ? X(mj, mi - 1) : 0.0;
        const double xd = (mi > 1 && mj < nz) ? X(mj + 1, mi - 1) : 0.0;
        const double f = therm_eval(c, xu, xl, xd, dt);
        bad |= __double_as_longlong(f) != __double_as_longlong(X(mj, mi));
    }
    atomicAdd(&ck->therm_mismatch, 1ull);  // (statistics)
    atomicMax(&ck->therm_mismatch_ulp, (unsigned long long)(a > b ? a - b : b - a));
    if (bad) atomicOr(&ck->therm_pass_changed[pass], 1u);
}

__global__ void __launch_bounds__(256) k_therm_check(const GfDevParams *__restrict__ P, GfDevClock *ck, GfDevArrays A,
                                                    int w, int pass, int arp, ThermSlots sl, long total)
{
    if (pass > 0 && ck->therm_pass_changed[pass - 1] == 0u) return;  // that pass did not run
    const ThermGeo g = therm_geo(P, w);
    const long t = (long)blockIdx.x * 256 + threadIdx.x;
    if (t < total) therm_check_one(P, ck, A, g, t, pass, arp, sl);
}
// The check of pass 0 as the first `grid` workgroups of a launch that neither reads the
// temperature nor writes what the check reads (grid 0: none; a multiple of 8, so that the
// others keep their XCDs)
struct ThermChk {
    int grid, w, arp;
    ThermSlots sl;
    double *temp, *xa;  // the call's old temperature and its result
};
GF_DEV void therm_chk_block(const GfDevParams *__restrict__ P, GfDevClock *ck, GfDevArrays A, const ThermChk &c)
{
    A.temp = c.temp;
    A.xa = c.xa;
    const ThermGeo g = therm_geo(P, c.w);
    therm_check_one(P, ck, A, g, (long)blockIdx.x * 256 + threadIdx.x, 0, c.arp, c.sl);
}

// The call's outcome, once: statistics, and GF_ERR_THERM_SWEEPS where no pass was proven
GF_DEV void therm_outcome(GfDevClock *ck, int proven)
{
    if (proven < 0) {
        atomicAdd(&ck->therm_unconverged, 1ull);
        raise_error(ck, GF_ERR_THERM_SWEEPS, 0);
    } else if (proven > 0) {
        atomicAdd(&ck->therm_extra_passes, (unsigned long long)proven);
    }
}
// ... and, after an odd last pass, its result (iterate xb, slot 3) into xa and the call's slot
GF_DEV void therm_settle(const GfDevParams *__restrict__ P, const GfDevArrays &A, const ThermSlots &sl, int last,
                         long tid, long nthr)
{
    if (last % 2 == 0) return;
    for (long t = tid; t < NN; t += nthr) A.xa[t] = A.xb[t];
    const double *from = therm_pre(P, A, sl.cur[1]);
    double *to = therm_pre(P, A, sl.cur[0]);
    for (long t = tid; t < 2L * (P->nx + P->nz); t += nthr) to[t] = from[t];
}

// The rest of the call after pass 0 and its check, in one launch of at most one
// workgroup per CU.  When pass 0 is proven it returns at once.  Otherwise the further
// passes run here, each over all strips and followed by its border check, with grid
// barriers between the phases, until one is proven or npass ran.  The flags that decide
// another pass are read with coherent loads after a barrier, so every workgroup takes
// the same decision; flag 0 was written by earlier launches.
template <bool DIS>
__global__ void __launch_bounds__(256) k_therm_rest(const GfDevParams *__restrict__ P, GfDevClock *ck, GfDevArrays A,
                                                    int w, int arp, ThermSlots sl, int npass)
{
    if (ck->therm_pass_changed[0] == 0u) return;
    __shared__ double sPhw[4][4][GF_MAXPH];  // (a table a wave)
    double(*sPh)[GF_MAXPH] = sPhw[threadIdx.x / 64];
    therm_phase_table(P, sPh);
    const ThermGeo g = therm_geo(P, w);
    const int nt = g.nr * g.ns;
    const long nb = (long)nt * TS_NB(w);
    const long tid = (long)blockIdx.x * blockDim.x + threadIdx.x, nthr = (long)gridDim.x * blockDim.x;
    int proven = -1, pass = 1;
    for (; pass < npass; pass++) {
        const ThermIter it{pass % 2 == 1 ? A.xa : A.xb, pass % 2 == 0 ? A.xa : A.xb, arp, pass};
        for (int t = (int)(tid / 64); t < nt; t += (int)(nthr / 64))
            therm_strip<DIS, 1>(P, ck, A, g, t, it, sl, A.tbord + (long)t * TS_NB(w), ck->dt, sPh);
        if (!grid_sync(ck)) return;  // every strip's iterate is written
        for (long t = tid; t < nb; t += nthr) therm_check_one(P, ck, A, g, t, pass, arp, sl);
        if (!grid_sync(ck)) return;  // every border is checked
        if (__hip_atomic_load(&ck->therm_pass_changed[pass], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == 0u) {
            proven = pass;
            break;
        }
    }
    if (tid == 0) therm_outcome(ck, proven);
    therm_settle(P, A, sl, proven < 0 ? npass - 1 : proven, tid, nthr);
}

// the end of a call whose further passes ran as launches of their own
__global__ void __launch_bounds__(256) k_therm_last(const GfDevParams *__restrict__ P, GfDevClock *ck, GfDevArrays A,
                                                    ThermSlots sl, int npass)
{
    int proven = -1;
    for (int k = npass - 1; k >= 0; k--)
        if (ck->therm_pass_changed[k] == 0u) proven = k;
    const long tid = (long)blockIdx.x * blockDim.x + threadIdx.x, nthr = (long)gridDim.x * blockDim.x;
    if (tid == 0) therm_outcome(ck, proven);
    therm_settle(P, A, sl, proven < 0 ? npass - 1 : proven, tid, nthr);
}

// While a batch's table holds the context's array pointers the result is copied to temp
// instead of the buffers turning over (src/fl_therm.f90:52 copies temp to temp0)
__global__ void __launch_bounds__(256) k_therm_copy(const GfDevParams *__restrict__ P, GfDevArrays A)
{
    const long t = xcd_lin();
    if (t >= NN) return;
    A.temp0[t] = A.temp[t];
    A.temp[t] = A.xa[t];
}
