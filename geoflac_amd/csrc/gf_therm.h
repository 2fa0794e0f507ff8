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
// and barriers; their thermal step took 137 us on 2001x1001 nodes, the strips take 68 (and 6
// for the rest of the call), and on square cells (902x302 nodes), where their four halo
// columns needed a second pass in every step, 125 us against 27.
//
// Strips: rows are cut into strips of 64 lanes that overlap by 2 * TS_HB rows (none at
// the mesh's top and bottom), columns into strips of `w` output columns that start
// some halo columns (therm_halo) and one ring column further left.  The ring and
// the outermost rows only hold the starting iterate.  A strip's values in its halo rows and columns are not exact; what
// it saves of them (its border) is compared with the values of the strips that own
// those nodes (therm_check_one), which proves the assembled result.
#pragma once

#define TS_HB 6                  // rows of a strip above and below its output rows: one ring row, five halo rows
#define TS_HI_MAX 12             // most halo columns left of its output columns (after one ring column)
#define TS_HI_FEW 8              // ... where more would not be enough either
#define TS_OJ (64 - 2 * TS_HB)   // output rows of an inner strip
#define TS_SWEEP0 2              // applications before the first stillness test
#define TS_MAXSWEEP 48
#define TS_NB(w) (2 * (w) + 64)  // border values of a strip: row above, row below, column to the left

// The boundary conditions (:575-598) overwrite rows 1 and nz and columns 1 and nx.  The
// values before them are what the border check and a further pass read, and what the
// next call's rows 1 and nz start from; they go to a ring buffer of GF_NPRE slots of
// 2 nx + 2 nz values: row 1, row nz, column 1, column nx.
#define GF_NPRE 4
// slots of a call: pass p writes of(p); the last two calls' final values (hist of them are
// valid)
struct ThermSlots {
    int cur, prev, prev2, hist;
    int flag;  // first flag of the call's passes; the other set's are cleared by pass 0
    GF_DEVM int of(int pass) const { return pass & 1 ? GF_NPRE - 1 : cur; }
    GF_DEVM int flag_of(int pass) const { return flag + pass % GF_THERM_FLAGS; }
};
// consecutive calls number `call` turn three slots over; an odd pass uses the fourth
__host__ __device__ inline ThermSlots therm_slots(int call, int hist, int set = 0)
{
    const int c = call % 3;
    return ThermSlots{c, (c + 2) % 3, (c + 1) % 3, hist, set ? GF_THERM_FLAGS : 0};
}
// the flags of the next call (those of the one before this, whose passes are over), and the
// counters of this call's further passes
GF_DEV void therm_clear_other(GfDevClock *ck, const ThermSlots &sl)
{
    if (blockIdx.x == 0 && threadIdx.x == 0) ck->q_next = ck->q_done = 0u;
    if (blockIdx.x == 0 && threadIdx.x < GF_THERM_FLAGS)
        ck->therm_pass_changed[(sl.flag ^ GF_THERM_FLAGS) + threadIdx.x] = 0u;
}
GF_DEV double *therm_pre(const GfDevParams *P, const GfDevArrays &A, int slot)
{
    return A.tpre + (long)slot * 2 * (P->nx + P->nz);
}

struct ThermGeo {
    int nz, nx, w, nr, ns;  // row strips, column strips
};
__host__ __device__ inline ThermGeo therm_geo(int nz, int nx, int w)
{
    ThermGeo g;
    g.nz = nz;
    g.nx = nx;
    g.w = w;
    g.nr = nz <= 64 ? 1 : (nz - 2 * TS_HB + TS_OJ - 1) / TS_OJ;
    g.ns = (nx + w - 1) / w;
    return g;
}
// Halo columns of a strip: each damps what the ring's start leaves by the coupling of
// columns c = diff dt / dx^2.  That error is some 1e-5 of a value's change (rows 1 and nz,
// whose start follows the last two calls), and grows as c^2 itself, the second difference in
// time that the extrapolated start leaves out.  Enough of them that c^hi <= 1e-11 and
// c^(hi + 2) <= 1e-15 (at least 2): at c = 1.3e-2 (901x301 cells of 333 m) 4, 5 and 6 columns
// need a further pass in 45%, 2% and none of the steps.  The second bound tells from c = 1e-2
// on: at c = 3e-2 to 6e-2 (200-360 x 34-60 cells of 25-45 m) the first one's 8 or fewer need
// one in 3-100% of the steps, its 9 to 11 in 0-12%.  Where TS_HI_MAX are not enough (c > 8.5e-2)
// further passes run in every step anyway, and TS_HI_FEW cost less: 131x70 cells at c = 0.11
// take 127 us a step with 8, 150 with 12.  What a strip leaves unsettled the border check
// finds.
__host__ __device__ inline int therm_halo(double diff_max, double rxbo, int nx, double dt)
{
    const double dx = rxbo / (double)(nx - 1), c = diff_max * dt / (dx * dx);
    double v = c * c;
    for (int hi = 2; hi <= TS_HI_MAX; hi++, v *= c)
        if (v <= 1.0e-11 && v * c * c <= 1.0e-15) return hi;
    return TS_HI_FEW;
}
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

struct ThermIter {
    const double *xin;  // starting iterate of a pass > 0
    double *xout;
    int arp;            // the areas of the last move are pending (formed from the coordinates)
    int pass;
};

// What a wave knows of its strip, and its loads and stores.  MODE, the start: 0 the old
// temperature, 1 xin, 2 the extrapolation 2 temp - temp0.
template <bool DIS, int MODE>
struct ThermWave {
    const GfDevParams *__restrict__ P;
    ThermGeo g;
    ThermStrip s;
    int hi, lane, row, nz, nx, arp;
    unsigned nn, ne, nvo, evo, evi, pvo, pco;
    bool erow, edge, erow1, erown, pedge, plin;
    // lanes that hold the start in every column (the ring rows), or no node
    bool hold;
    Buf bT, bC, bG, bX, bA, bS, bI, bH, bP, bP2, bW;
    double *bord;

    static constexpr unsigned OOB = 0x80000000u;  // past every array: loads read 0, stores are dropped
    struct Node {
        double x, y, t, g, p, p2;
    };
    struct Elem {
        double a0, a1, src, sh;
        int ph;
    };

    GF_DEVM ThermWave(const GfDevParams *__restrict__ P_, const GfDevArrays &A, const ThermGeo &g_, int t,
                      const ThermIter &it, const ThermSlots &sl, double *bord_, int hi_)
        : P(P_), g(g_), hi(hi_), bord(bord_)
    {
        s = therm_strip_of(g, t);
        lane = threadIdx.x % 64;
        nz = g.nz;
        nx = g.nx;
        arp = it.arp;
        row = s.jb + lane;
        nn = (unsigned)nz * nx;
        ne = (unsigned)(nz - 1) * (nx - 1);
        nvo = row <= nz ? (unsigned)(row - 1) * 8u : OOB;
        erow = row < nz && lane < 63;
        evo = erow ? (unsigned)(row - 1) * 8u : OOB;
        evi = erow ? (unsigned)(row - 1) * 4u : OOB;
        edge = s.top || s.bot;  // (uniform)
        erow1 = row == 1;
        erown = row == nz;
        hold = (lane == 0 && !s.top) || (lane == 63 && !s.bot) || row > nz;
        bT = mkbuf(A.temp, 8ull * nn);
        bC = mkbuf(A.cord, 16ull * nn);
        bG = mkbuf(MODE == 1 ? it.xin : A.temp0, 8ull * nn);
        bX = mkbuf(it.xout, 8ull * nn);
        bA = mkbuf(A.area, 16ull * ne);
        bS = mkbuf(A.source, 8ull * ne);
        bI = mkbuf(A.iphase, 4ull * ne);
        bH = mkbuf(A.shrheat, 8ull * ne);
        // start of rows 1 and nz: the values before the boundary conditions of the last two
        // calls, carried on (pass 0), or those of the last pass (the iterate's own boundary
        // rows hold the conditions)
        const unsigned npre = 2u * (nx + nz);
        const int pslot = MODE == 1 ? sl.of(it.pass - 1) : sl.prev;
        bP = mkbuf(A.tpre + (long)pslot * npre, 8ull * npre);
        bP2 = mkbuf(A.tpre + (long)sl.prev2 * npre, 8ull * npre);
        bW = mkbuf(A.tpre + (long)sl.of(it.pass) * npre, 8ull * npre);
        pvo = erow1 ? 0u : erown ? 8u * nx : OOB;               // row arrays, + 8 (i - 1)
        pco = row <= nz ? 8u * (2 * nx + row - 1) : OOB;        // column arrays, + 8 nz for column nx
        pedge = edge && (MODE == 1 || (MODE == 2 && sl.hist > 0));
        plin = MODE == 2 && sl.hist > 1;
    }
    // node column i (i >= 1; 0 past the mesh and past the strip's last neighbours)
    GF_DEVM Node node(int i) const
    {
        Node n{0, 0, 0, 0, 0, 0};
        if (i <= min(nx, s.c1 + 1)) {  // (uniform)
            const unsigned so = (unsigned)nz * (unsigned)(i - 1) * 8u;
            n.x = bld(bC, nvo, so);
            n.y = bld(bC, nvo, so + 8u * nn);
            n.t = bld(bT, nvo, so);
            if (MODE != 0) n.g = bld(bG, nvo, so);
            if (pedge) {
                n.p = bld(bP, pvo, 8u * (i - 1));
                if (plin) n.p2 = bld(bP2, pvo, 8u * (i - 1));
            }
            if (MODE == 1 && (i == 1 || i == nx))  // (the iterate's boundary columns, likewise)
                n.g = bld(bP, pco, i == 1 ? 0u : 8u * nz);
        }
        return n;
    }
    GF_DEVM Elem elem(int i) const
    {
        Elem e{0, 0, 0, 0, 1};
        if (i <= min(nx - 1, s.c1)) {
            const unsigned ec = (unsigned)(nz - 1) * (unsigned)(i - 1);
            e.src = bld(bS, evo, ec * 8u);
            e.ph = bldi(bI, evi, ec * 4u);
            if (!arp) {
                e.a0 = bld(bA, evo, ec * 8u);
                e.a1 = bld(bA, evo, (ec + ne) * 8u);
            }
            if (DIS) e.sh = bld(bH, evo, ec * 8u);
        }
        return e;
    }
    GF_DEVM double start(const Node &n) const
    {
        double v = MODE == 0 ? n.t : MODE == 1 ? n.g : 2.0 * n.t - n.g;
        if (pedge && (erow1 || erown)) v = plin ? 2.0 * n.p - n.p2 : n.p;
        return v;
    }
    // Element column i between node columns n0 and n1 (yd, xd: their rows below).
    // sPh: den, cp, 0.5 diff, 1 / cp per phase (LDS).
    GF_DEVM void tris(int i, const Node &n0, const Node &n1, double xd0, double yd0, double xd1, double yd1,
                      const Elem &e, int phs, const double (*sPh)[GF_MAXPH], ThermTri &ta, ThermTri &tb) const
    {
        const bool eok = erow && i < nx;
        double ar0 = e.a0, ar1 = e.a1, inv0, inv1;
        if (arp) {
            const double xc[5] = {0.0, n0.x, xd0, n1.x, xd1}, yc[5] = {0.0, n0.y, yd0, n1.y, yd1};
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
        const double sd = DIS ? e.src + e.sh / sPh[0][phs] : e.src + 0.0, cp = sPh[1][phs];
        double dm = div_fma(sd, cp, sPh[3][phs]);
        if (__any(eok && sd != 0.0 && !(rcp_safe(sd) && rcp_safe(cp)))) dm = sd / cp;
        dm = eok ? dm : 0.0;
        const double hdf = sPh[2][phs];
        const double y1 = n0.y, y2 = yd0, y3 = n1.y, y4 = yd1, x1 = n0.x, x2 = xd0, x3 = n1.x, x4 = xd1;
        const double da[6] = {(y2 - y3) * ar0, (y3 - y1) * ar0, (y1 - y2) * ar0,
                              (x3 - x2) * ar0, (x1 - x3) * ar0, (x2 - x1) * ar0};
        const double db[6] = {(y2 - y4) * ar1, (y4 - y3) * ar1, (y3 - y2) * ar1,
                              (x4 - x2) * ar1, (x3 - x4) * ar1, (x2 - x3) * ar1};
        ta = therm_tri(da, inv0, dm, hdf);
        tb = therm_tri(db, inv1, dm, hdf);
    }
    // 1 / area of a node, 0 in the lanes that hold their start (a zero increment)
    GF_DEVM double rarea(double area_n) const
    {
        double r = rcp_core(area_n);
        if (__any(!hold && !rcp_safe(area_n))) r = 1.0 / area_n;
        return hold ? 0.0 : r;
    }
    // the result x of column i and the border values it holds
    GF_DEVM void store(int i, double x, double y, int phs) const
    {
        if (i < s.c0) {
            if (i == s.c0 - 1) bord[2 * g.w + lane] = x;
            return;
        }
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
                    vb = lane_up(x) + P->bot_bc * (lane_up(y) - y) / PHASE(phu + 1).conduct;
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
    }
};
GF_DEV int therm_phs(int ph) { return ph >= 1 && ph <= GF_MAXPH ? ph - 1 : 0; }  // (0 where there is no element)

// What node column i+1 takes of element column i: triangle B one row up (t1), A and B of
// its own row (t4, t5)
struct ThermLeft {
    double b13, b23, b33, bp, bq, br;
    double a13, a23, a33, ap, aq, ar;
    double c11, c12, c13, cp, cq, cr;
};
// What node column i takes of element column i from the row above (t2 A, t3 B)
struct ThermUp {
    double a12, a22, a23, ap, aq, ar, b12, b22, b23, bp, bq, br;
};
GF_DEV ThermUp therm_up(const ThermTri &ta, const ThermTri &tb)
{
    return ThermUp{lane_up(ta.k12), lane_up(ta.k22), lane_up(ta.k23), lane_up(ta.p), lane_up(ta.q), lane_up(ta.ra),
                   lane_up(tb.k12), lane_up(tb.k22), lane_up(tb.k23), lane_up(tb.p), lane_up(tb.q), lane_up(tb.ra)};
}
GF_DEV ThermLeft therm_left(const ThermTri &ta, const ThermTri &tb, const ThermUp &u)
{
    return ThermLeft{lane_up(tb.k13), u.b23, lane_up(tb.k33), u.bp, u.bq, u.br, ta.k13, ta.k23, ta.k33,
                     ta.p, ta.q, ta.ra, tb.k11, tb.k12, tb.k13, tb.p, tb.q, tb.ra};
}

// One strip by one wave.
template <bool DIS, int MODE>
GF_DEV void therm_strip(const GfDevParams *__restrict__ P, GfDevClock *ck, const GfDevArrays &A, const ThermGeo &g,
                        int t, const ThermIter &it, const ThermSlots &sl, double *bord, double dt,
                        const double (*sPh)[GF_MAXPH])
{
    typedef ThermWave<DIS, MODE> W;
    const W w(P, A, g, __builtin_amdgcn_readfirstlane(t), it, sl, bord,
              __builtin_amdgcn_readfirstlane(therm_halo(P->diff_max, P->rxbo, P->nx, dt)));
    const int ib = max(1, w.s.c0 - w.hi - 1);
    const bool has_ring = w.s.c0 - w.hi > 1;  // column ib only holds the start
    typename W::Node n0 = w.node(ib), n1 = w.node(ib + 1);
    typename W::Elem e0 = w.elem(ib);
    double ydn0 = lane_dn(n0.y), xdn0 = lane_dn(n0.x), tdn0 = lane_dn(n0.t);
    double xl = 0.0, xd = 0.0;  // X(j, i-1), X(j+1, i-1)
    ThermLeft l{};              // of element column i-1 (none at the mesh's left)
    bool still = true;
    for (int i = ib; i <= w.s.c1; i++) {
        // the loads of the columns ahead
        const typename W::Node n2 = w.node(i + 2);
        const typename W::Elem e1 = w.elem(i + 1);
        const double ydn1 = lane_dn(n1.y), xdn1 = lane_dn(n1.x), tdn1 = lane_dn(n1.t);
        const int phs = therm_phs(e0.ph);
        ThermTri ta, tb;
        w.tris(i, n0, n1, xdn0, ydn0, xdn1, ydn1, e0, phs, sPh, ta, tb);
        const ThermUp u = therm_up(ta, tb);
        double x = w.start(n0);
        if (!(has_ring && i == ib)) {  // (uniform)
            // t1 B of (j-1,i-1), t2 A of (j-1,i), t3 B of (j-1,i), t4 A of (j,i-1),
            // t5 B of (j,i-1), t6 A of (j,i)
            const double tme = n0.t, tur = lane_up(n1.t);  // T(j,i), T(j-1,i+1)
            const double area_n = (((((0.0 + l.br) + u.ar) + u.br) + l.ar) + l.cr) + ta.ra;
            const double rarea = w.rarea(area_n);
            const double told = w.hold ? x : tme;
            const double xl12 = xl * l.b23, c13 = tme * l.b33;           // t1: K13 K23 K33
            const double c22 = tme * u.a22, c23 = tur * u.a23;           // t2
            const double qs3 = u.bq * (tur * u.b12 + tme * u.b22 + n1.t * u.b23);
            const double qs4 = l.aq * ((xl * l.a13 + xd * l.a23) + tme * l.a33);
            const double qs5 = l.cq * ((tme * l.c11 + xd * l.c12) + tdn0 * l.c13);
            const double qs6 = ta.q * (tme * ta.k11 + tdn0 * ta.k12 + n1.t * ta.k13);
            auto eval = [&](double xu) {
                double rhs = 0.0;
                rhs = rhs + l.bp - l.bq * ((xu * l.b13 + xl12) + c13);
                rhs = rhs + u.ap - u.aq * ((xu * u.a12 + c22) + c23);
                rhs = rhs + u.bp - qs3;
                rhs = rhs + l.ap - qs4;
                rhs = rhs + l.cp - qs5;
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
        w.store(i, x, n0.y, phs);
        // on to column i+1
        xl = x;
        xd = lane_dn(x);
        l = therm_left(ta, tb, u);
        n0 = n1;
        n1 = n2;
        e0 = e1;
        xdn0 = xdn1;
        ydn0 = ydn1;
        tdn0 = tdn1;
    }
    if (!still && w.lane == 0) atomicOr(&ck->therm_pass_changed[sl.flag_of(it.pass)], 2u);
}

// One strip by one workgroup, a wave a column, for meshes of so few strips that each has a
// CU of its own: a wave's march from column to column (1.3 us each) leaves 3 of a CU's 4
// SIMDs idle there.  Column
// c0 - hi - 1 + q is wave q's.  The waves form their element columns at the same time, hand
// the next column its share through LDS, and apply the update together from the last
// iterate of the column to the left (a barrier each time) until no bit of the strip changes:
// more applications than the march takes, but all columns in one of them.  The same fixed
// point, borders and proof.  Bound by latency: the loads and element columns some 3 us, 6 to
// 8 applications 0.4 us each.  At 4 + 4 columns the kernel takes 6.9 us where the march took
// 12 (60x20 cells), 7.4 for 12 (151x47) and 9.3 for 13 (400x100); a step there 39.3 -> 36.2,
// 49.4 -> 44.9 and 37.1 -> 33.2 us.  2, 3 and 4 output columns are within 2% at the two
// smaller meshes; 400x100 cells take 34.8, 34.3 and 33.2 us a step (400 workgroups to 200).
#define TC_W 9   // waves (columns) of a workgroup: output columns, halo columns, the ring
#define TC_HI 4  // most halo columns (fewer are used where therm_halo says so)
struct ThermColLds {
    double ph[4][GF_MAXPH];
    double left[TC_W - 1][18][64];
    double x[2][TC_W][64];
    int flag[3];
};
template <bool DIS, int MODE>
GF_DEV void therm_cols(const GfDevParams *__restrict__ P, GfDevClock *ck, const GfDevArrays &A, const ThermGeo &g,
                       int t, const ThermIter &it, const ThermSlots &sl, double *bord, ThermColLds &L)
{
    typedef ThermWave<DIS, MODE> W;
    const int q = __builtin_amdgcn_readfirstlane((int)(threadIdx.x / 64));
    const W w(P, A, g, t, it, sl, bord, TC_W - 1 - g.w);
    const int i = w.s.c0 - w.hi - 1 + q;
    const bool in = i >= 1 && i <= w.s.c1;  // (uniform in a wave; the others only keep the barriers)
    const double dt = ck->dt;
    typename W::Node n0{}, n1{};
    typename W::Elem e0{};
    if (in) {
        n0 = w.node(i);
        n1 = w.node(i + 1);
        e0 = w.elem(i);
    }
    if (threadIdx.x < GF_MAXPH) {
        const int k = threadIdx.x;
        L.ph[0][k] = P->ph[k].den;
        L.ph[1][k] = P->ph[k].cp;
        L.ph[2][k] = 0.5 * P->ph[k].diff;
        L.ph[3][k] = 1.0 / P->ph[k].cp;
    }
    if (threadIdx.x < 3) L.flag[threadIdx.x] = 0;
    // (dt, and so the halo, come after the loads on purpose: columns beyond it are let go)
    const int hi = min(w.hi, __builtin_amdgcn_readfirstlane(therm_halo(P->diff_max, P->rxbo, P->nx, dt)));
    const bool work = in && i >= w.s.c0 - hi;  // (the ring and what is beyond it only hold the start)
    __syncthreads();
    const double ydn0 = lane_dn(n0.y), xdn0 = lane_dn(n0.x), tdn0 = lane_dn(n0.t);
    const int phs = therm_phs(e0.ph);
    ThermTri ta, tb;
    w.tris(i, n0, n1, xdn0, ydn0, lane_dn(n1.x), lane_dn(n1.y), e0, phs, L.ph, ta, tb);
    const ThermUp u = therm_up(ta, tb);
    double x = w.start(n0);
    {
        const ThermLeft l = therm_left(ta, tb, u);
        const double v[18] = {l.b13, l.b23, l.b33, l.bp, l.bq, l.br, l.a13, l.a23, l.a33,
                              l.ap, l.aq, l.ar, l.c11, l.c12, l.c13, l.cp, l.cq, l.cr};
        if (q < TC_W - 1) {
#pragma unroll
            for (int k = 0; k < 18; k++) L.left[q][k][w.lane] = v[k];
        }
        L.x[0][q][w.lane] = x;
        L.x[1][q][w.lane] = x;
    }
    lds_barrier();
    ThermLeft l{};
    if (q > 0 && i > 1) {
        double v[18];
#pragma unroll
        for (int k = 0; k < 18; k++) v[k] = L.left[q - 1][k][w.lane];
        l = ThermLeft{v[0], v[1], v[2], v[3], v[4], v[5], v[6], v[7], v[8],
                      v[9], v[10], v[11], v[12], v[13], v[14], v[15], v[16], v[17]};
    }
    const double tme = n0.t, tur = lane_up(n1.t);
    const double area_n = (((((0.0 + l.br) + u.ar) + u.br) + l.ar) + l.cr) + ta.ra;
    const double rarea = w.rarea(work ? area_n : 1.0);
    const double told = w.hold ? x : tme;
    const double c13 = tme * l.b33, c22 = tme * u.a22, c23 = tur * u.a23, c43 = tme * l.a33, c51 = tme * l.c11,
                 c53 = tdn0 * l.c13;
    const double qs3 = u.bq * (tur * u.b12 + tme * u.b22 + n1.t * u.b23);
    const double qs6 = ta.q * (tme * ta.k11 + tdn0 * ta.k12 + n1.t * ta.k13);
    int cur = 0, nsweep = 0;
    bool still = false;
    while (nsweep < TS_MAXSWEEP) {
        if (work) {
            const double xl = q > 0 ? L.x[cur][q - 1][w.lane] : 0.0, xd = lane_dn(xl), xu = lane_up(x);
            double rhs = 0.0;
            rhs = rhs + l.bp - l.bq * ((xu * l.b13 + xl * l.b23) + c13);
            rhs = rhs + u.ap - u.aq * ((xu * u.a12 + c22) + c23);
            rhs = rhs + u.bp - qs3;
            rhs = rhs + l.ap - l.aq * ((xl * l.a13 + xd * l.a23) + c43);
            rhs = rhs + l.cp - l.cq * ((c51 + xd * l.c12) + c53);
            rhs = rhs + ta.p - qs6;
            const double xn = told + div_fma(rhs * dt, area_n, rarea);
            if (nsweep >= TS_SWEEP0 && __any(__double_as_longlong(xn) != __double_as_longlong(x)) && w.lane == 0)
                L.flag[nsweep % 3] = 1;
            x = xn;
            L.x[cur ^ 1][q][w.lane] = x;
        }
        lds_barrier();
        // (flag nsweep % 3 is raised before the barrier and read after it; the one of two
        // applications on is cleared meanwhile)
        const int any = nsweep < TS_SWEEP0 ? 1 : L.flag[nsweep % 3];
        if (threadIdx.x == 0) L.flag[(nsweep + 2) % 3] = 0;
        cur ^= 1;
        nsweep++;
        if (!any) {
            still = true;
            break;
        }
    }
    if (in) w.store(i, x, n0.y, phs);
    if (!still && threadIdx.x == 0) atomicOr(&ck->therm_pass_changed[sl.flag_of(it.pass)], 2u);
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

// pass 0 (mode 0 or 2), one wave a strip
template <bool DIS, int MODE>
__global__ void __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(3)))
k_therm_strip(const GfDevParams *__restrict__ P, GfDevClock *ck, GfDevArrays A, ThermGeo g, int arp, ThermSlots sl,
              ClockOps ops)
{
    therm_clear_other(ck, sl);
    if (blockIdx.x == 0 && threadIdx.x == 0) clock_op(ck, ops);  // (fields nothing here reads)
    __shared__ double sPh[4][GF_MAXPH];
    const int nt = g.nr * g.ns, q = (nt + 7) / 8;  // XCD x runs strips [x q, (x+1) q)
    const int t = (int)(blockIdx.x % 8) * q + (int)(blockIdx.x / 8);
    if ((int)(blockIdx.x / 8) >= q || t >= nt) return;
    therm_phase_table(P, sPh);
    const ThermIter it{A.xb, A.xa, arp, 0};
    therm_strip<DIS, MODE>(P, ck, A, g, t, it, sl, A.tbord + (long)t * TS_NB(g.w), ck->dt, sPh);
}
// pass 0, one workgroup a strip
template <bool DIS, int MODE>
__global__ void __launch_bounds__(64 * TC_W)
k_therm_cols(const GfDevParams *__restrict__ P, GfDevClock *ck, GfDevArrays A, ThermGeo g, int arp, ThermSlots sl,
             ClockOps ops)
{
    therm_clear_other(ck, sl);
    if (blockIdx.x == 0 && threadIdx.x == 0) clock_op(ck, ops);  // (fields nothing here reads)
    __shared__ ThermColLds L;
    const int nt = g.nr * g.ns, q = (nt + 7) / 8, t = (int)(blockIdx.x % 8) * q + (int)(blockIdx.x / 8);
    if ((int)(blockIdx.x / 8) >= q || t >= nt) return;
    const ThermIter it{A.xb, A.xa, arp, 0};
    therm_cols<DIS, MODE>(P, ck, A, g, t, it, sl, A.tbord + (long)t * TS_NB(g.w), L);
}

// the same bits; not-a-numbers count as the same (which of them a diverged model holds is no
// matter, and no reason for further passes)
GF_DEV bool therm_same(double a, double b)
{
    return __double_as_longlong(a) == __double_as_longlong(b) || (a != a && b != b);
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
    const double *__restrict__ pre = therm_pre(P, A, sl.of(pass));
    // the pass's value before the boundary conditions
    auto X = [&](int jj, int ii) -> double {
        if (jj == 1) return pre[ii - 1];
        if (jj == nz) return pre[nx + ii - 1];
        if (ii == 1) return pre[2 * nx + jj - 1];
        if (ii == nx) return pre[2 * nx + nz + jj - 1];
        return x[IN(jj, ii)];
    };
    const double xb = A.tbord[t], xo = X(j, i);
    if (therm_same(xb, xo)) return;
    const long long a = __double_as_longlong(xb), b = __double_as_longlong(xo);
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
        bad |= !therm_same(f, X(mj, mi));
    }
    atomicAdd(&ck->therm_mismatch, 1ull);  // (statistics)
    atomicMax(&ck->therm_mismatch_ulp, (unsigned long long)(a > b ? a - b : b - a));
    if (bad) atomicOr(&ck->therm_pass_changed[sl.flag_of(pass)], 1u);
}

__global__ void __launch_bounds__(256) k_therm_check(const GfDevParams *__restrict__ P, GfDevClock *ck, GfDevArrays A,
                                                    ThermGeo g, int arp, ThermSlots sl, long total)
{
    const long t = (long)blockIdx.x * 256 + threadIdx.x;
    if (t < total) therm_check_one(P, ck, A, g, t, 0, arp, sl);
}
// The check of pass 0 as the first `grid` workgroups of a launch that neither reads the
// temperature nor writes what the check reads (grid 0: none; a multiple of 8, so that the
// others keep their XCDs)
struct ThermChk {
    int grid, arp;
    ThermGeo g;
    ThermSlots sl;
    double *temp, *xa;  // the call's old temperature and its result
};
GF_DEV void therm_chk_block(const GfDevParams *__restrict__ P, GfDevClock *ck, GfDevArrays A, const ThermChk &c)
{
    A.temp = c.temp;
    A.xa = c.xa;
    therm_check_one(P, ck, A, c.g, (long)blockIdx.x * 256 + threadIdx.x, 0, c.arp, c.sl);
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
    const double *from = therm_pre(P, A, sl.of(1));
    double *to = therm_pre(P, A, sl.of(0));
    for (long t = tid; t < 2L * (P->nx + P->nz); t += nthr) to[t] = from[t];
}

// The rest of the call after pass 0 and its check, in one launch.  When pass 0 is proven it
// returns at once.  Otherwise the further passes run here in phases of R.grid units each
// (queue_take): phase 2 (p - 1) runs the strips of pass p, phase 2 p - 1 checks its borders,
// and the phase after the pass that ends the call settles its result.  The flag that decides
// another pass is read with coherent loads once the phases before are done, so every unit
// takes the same decision (strips of pass p clear the one of pass p + 1); flag 0 was written
// by earlier launches.  No workgroup needs the others resident, so that models and batches
// may run their passes at the same time, on streams of their own; grid barriers after each
// phase did, and were slower: 12 models of 200-360 x 34-60 cells in a batch, a further pass
// in nearly every step, 241 us a step to 203.
//
// As many passes as the proof takes (therm_pass_limit), two at most in nearly every call.
// In a start that is the same in every column, though, some row's sum may lie so near a
// rounding tie that the last bit of a value hangs on the value to its left all along the
// row: the serial order's bit then moves on by a strip, or its halo, a pass.
__host__ __device__ inline int therm_pass_limit(const ThermGeo &g) { return g.nx + 4; }  // (some 3 columns a pass or more)
struct ThermRest {
    int grid, arp, npass;
    ThermGeo g;
    ThermSlots sl;
};
template <bool DIS>
GF_DEV void therm_rest_body(const GfDevParams *__restrict__ P, GfDevClock *ck, const GfDevArrays &A, const ThermRest &R)
{
    const ThermSlots sl = R.sl;
    if (ck->therm_pass_changed[sl.flag] == 0u) return;
    const ThermGeo g = R.g;
    const int npass = R.npass;
    __shared__ double sPhw[4][4][GF_MAXPH];  // (a table a wave)
    double(*sPh)[GF_MAXPH] = sPhw[threadIdx.x / 64];
    therm_phase_table(P, sPh);
    const int nt = g.nr * g.ns;
    const long nb = (long)nt * TS_NB(g.w);
    const unsigned units = (unsigned)R.grid;
    const long nthr = (long)units * 256;
    for (;;) {
        const unsigned unit = queue_take(ck), phase = unit / units;
        const long tid = (long)(unit % units) * 256 + threadIdx.x;
        if (phase > 2u * (unsigned)(npass - 1)) return;
        if (!queue_wait(ck, phase * units)) {  // (not expected)
            if (threadIdx.x == 0) __hip_atomic_fetch_or(&ck->q_timeout, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            return;
        }
        // passes up to `checked` are checked
        const int checked = (int)(phase / 2u), pass = checked + 1;
        const bool open = __hip_atomic_load(&ck->therm_pass_changed[sl.flag_of(checked)], __ATOMIC_RELAXED,
                                            __HIP_MEMORY_SCOPE_AGENT) != 0u;
        if ((checked > 0 && !open) || pass == npass) {
            if (phase % 2u != 0u) return;  // (settled)
            if (tid == 0) therm_outcome(ck, checked > 0 && !open ? checked : -1);
            therm_settle(P, A, sl, checked, tid, nthr);
        } else if (phase % 2u == 0u) {
            if (tid == 0)
                __hip_atomic_store(&ck->therm_pass_changed[sl.flag_of(pass + 1)], 0u, __ATOMIC_RELAXED,
                                   __HIP_MEMORY_SCOPE_AGENT);
            const ThermIter it{pass % 2 == 1 ? A.xa : A.xb, pass % 2 == 0 ? A.xa : A.xb, R.arp, pass};
            for (int t = (int)(tid / 64); t < nt; t += (int)(nthr / 64))
                therm_strip<DIS, 1>(P, ck, A, g, t, it, sl, A.tbord + (long)t * TS_NB(g.w), ck->dt, sPh);
        } else {
            for (long t = tid; t < nb; t += nthr) therm_check_one(P, ck, A, g, t, pass, R.arp, sl);
        }
        queue_done(ck);
    }
}
template <bool DIS>
__global__ void __launch_bounds__(256) k_therm_rest(const GfDevParams *__restrict__ P, GfDevClock *ck, GfDevArrays A,
                                                    ThermRest R)
{
    therm_rest_body<DIS>(P, ck, A, R);
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
