// gf_batch.h -- many independent models advanced by the same launches.
//
// A parameter sweep holds hundreds of small models of different mesh sizes.  One
// launch per kernel of the step covers all of them: the launch's index range is the
// concatenation of the models' elements (or nodes, thermal tiles, border entries),
// each model's range starting at a multiple of 256.  A workgroup therefore lies in
// one model, which it reads from a table of the model of each 256-index chunk (one
// load, the same for every lane, so the model's entry is read with scalar loads).
// Every model keeps its own parameters, clock (dt, time, reductions) and arrays, so
// the models stay independent; the kernel bodies are the single-model ones.
#pragma once
#include "gf_kernels.h"
#include "gf_phase.h"

// The temperature turns over three buffers and the coordinates two, as in a model alone,
// but in the table: kb_begin turns them at the start of each step, so that a captured step
// can be replayed.  Within a step A.temp is the step's result (formed by the thermal
// launches) and A.temp0 its old temperature; A.cord are the coordinates before the move and
// cord_next those after it (the current ones between steps; where the grid does not move,
// A.cord throughout).
struct BatchEntry {
    const GfDevParams *P;
    GfDevClock *ck;
    GfDevArrays A;
    double *tprev;      // the starting temperature of the call before (the next call's result)
    double *cord_next;
    ThermGeo tg;        // thermal strips
    GfDevClock *host;   // the model's clock in page-locked memory
    long pe, pn, pt, pb, pm;  // first global index: elements, nodes, thermal tiles, border entries, markers
    long ce, cn, ct, cb, cm;  // counts of the same
};

enum { BK_ELEM = 0, BK_NODE = 1, BK_TILE = 2, BK_BORD = 3, BK_MARK = 4 };
#define BATCH_ALIGN 256  // each model's element, node and border ranges start at a multiple

// model of each 256-index chunk of the element, node and border ranges, and of each tile
struct BatchMap {
    const int *chunk[5];
    int nm, pad;
};

template <int F>
GF_DEV long bprefix(const BatchEntry &b)
{
    return F == BK_ELEM ? b.pe : F == BK_NODE ? b.pn : F == BK_TILE ? b.pt : F == BK_BORD ? b.pb : b.pm;
}
template <int F>
GF_DEV long bcount(const BatchEntry &b)
{
    return F == BK_ELEM ? b.ce : F == BK_NODE ? b.cn : F == BK_TILE ? b.ct : F == BK_BORD ? b.cb : b.cm;
}

// the entry of model m (m uniform across the workgroup), read through the constant
// address space: the table is never written while a kernel runs, so its fields load
// with scalar loads and the buffer descriptors built from them stay uniform (read as
// ordinary global memory, the compiler cannot prove them uniform once the kernel has
// stored anything and wraps every buffer access in a loop over distinct values)
typedef const __attribute__((address_space(4))) BatchEntry ConstBatchEntry;
GF_DEV const BatchEntry &bentry(const BatchEntry *tab, int m)
{
    return *(const BatchEntry *)&((ConstBatchEntry *)tab)[m];
}

// workgroup k is dispatched to XCD k % 8: give each XCD one contiguous run of the
// index range (the first G % 8 XCDs one workgroup more), so that the node rows two
// neighbouring workgroups share stay in one L2 (a bijection for any grid size G)
// (skip, a multiple of 8: the first workgroups of the launch do something else)
GF_DEV unsigned xcd_block(unsigned skip = 0)
{
    const unsigned G = gridDim.x - skip, k = blockIdx.x - skip, x = k % 8, q = G / 8, r = G % 8;
    return x * q + min(x, r) + k / 8;
}

// calls fn(entry, local index) for the global index of this thread (workgroups of at
// most BATCH_ALIGN threads, dividing it)
template <int F, typename Fn>
GF_DEV void batch_apply(const BatchEntry *__restrict__ tab, const BatchMap &map, Fn fn)
{
    const long g0 = (long)xcd_block() * blockDim.x;
    const int m = __builtin_amdgcn_readfirstlane(map.chunk[F][g0 / BATCH_ALIGN]);
    const BatchEntry &b = bentry(tab, m);
    const long l = g0 + threadIdx.x - bprefix<F>(b);
    if (l >= bcount<F>(b)) return;
    fn(b, l);
}

__global__ void kb_clock(const BatchEntry *__restrict__ tab, BatchMap map, int op)
{
    const int m = blockIdx.x * blockDim.x + threadIdx.x;
    if (m < map.nm) clock_op(tab[m].ck, op);
}
// the boundary values that earlier thermal calls left are not this batch's
__global__ void kb_fresh(const BatchEntry *__restrict__ tab, BatchMap map)
{
    const int m = blockIdx.x * blockDim.x + threadIdx.x;
    if (m < map.nm) tab[m].ck->th_hist = 0;
}
// the start of a step: clock updates, the buffers turned over (cord: the coordinates
// too), the thermal calls counted
__global__ void kb_begin(BatchEntry *tab, BatchMap map, int op, int cord)
{
    const int m = blockIdx.x * blockDim.x + threadIdx.x;
    if (m >= map.nm) return;
    BatchEntry &b = tab[m];
    clock_op(b.ck, op);
    b.ck->th_call = (b.ck->th_call + 1) % 3;
    b.ck->th_hist = min(b.ck->th_hist + 1, 3);
    b.ck->th_last = 0;
    b.ck->q_next = b.ck->q_done = 0u;  // (kb_therm_rest)
    double *t = b.tprev;
    b.tprev = b.A.temp0;
    b.A.temp0 = b.A.temp;
    b.A.temp = t;
    if (cord) {
        double *c = b.A.cord;
        b.A.cord = b.cord_next;
        b.cord_next = c;
    }
}

// the arrays as the thermal kernels name them (temp the old temperature, xa the result,
// temp0 the call before's old temperature), and as the kernels after the move do
GF_DEV GfDevArrays bthermal(const BatchEntry &b)
{
    GfDevArrays A = b.A;
    A.temp = b.A.temp0;
    A.xa = b.A.temp;
    A.temp0 = b.tprev;
    return A;
}
GF_DEV GfDevArrays bmoved(const BatchEntry &b)
{
    GfDevArrays A = b.A;
    A.cord = b.cord_next;
    return A;
}
GF_DEV ThermSlots bslots(const BatchEntry &b) { return therm_slots(b.ck->th_call, b.ck->th_hist - 1); }

// The proven thermal step of every model (k_therm_strip, k_therm_check, k_therm_rest):
// one wave a strip over the strips of all models
template <bool DIS, int MODE>
__global__ void __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(3)))
kb_therm_strip(const BatchEntry *__restrict__ tab, BatchMap map, int total, int arp)
{
    __shared__ double sPh[4][GF_MAXPH];
    const int q = (total + 7) / 8, g = (int)(blockIdx.x % 8) * q + (int)(blockIdx.x / 8);
    if ((int)(blockIdx.x / 8) >= q || g >= total) return;
    const BatchEntry &b = bentry(tab, __builtin_amdgcn_readfirstlane(map.chunk[BK_TILE][g]));
    const GfDevArrays A = bthermal(b);
    therm_phase_table(b.P, sPh);
    const ThermIter it{A.xb, A.xa, arp, 0};
    const int t = g - (int)b.pt;
    therm_strip<DIS, MODE>(b.P, b.ck, A, b.tg, t, it, bslots(b), A.tbord + (long)t * TS_NB(b.tg.w), b.ck->dt,
                           sPh);
}
__global__ void __launch_bounds__(256) kb_therm_check(const BatchEntry *__restrict__ tab, BatchMap map, int arp)
{
    batch_apply<BK_BORD>(tab, map, [&](const BatchEntry &b, long t) {
        therm_check_one(b.P, b.ck, bthermal(b), b.tg, t, 0, arp, bslots(b));
    });
}
// Returns at once when every model's pass 0 is proven.  Otherwise the further passes of
// the models that are not, in the phases of k_therm_rest over the strips and borders of all
// of them (queue_take on the first model's counters).
template <bool DIS>
__global__ void __launch_bounds__(256) kb_therm_rest(const BatchEntry *__restrict__ tab, BatchMap map, int total,
                                                     long border, int arp, int npass)
{
    // of a batch, whose calls all use the first set (bslots)
    auto flag = [&](GfDevClock *ck, int pass) { return &ck->therm_pass_changed[pass % GF_THERM_FLAGS]; };
    auto is_open = [&](GfDevClock *ck, int pass) {  // (written by other workgroups of this launch too)
        return __hip_atomic_load(flag(ck, pass), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0u;
    };
    // whether a model's pass is not proven (nor any before it: later flags stay 0 then)
    auto any_open = [&](int pass) {
        int any = 0;
        for (int m = threadIdx.x; m < map.nm; m += 256) any |= is_open(tab[m].ck, pass);
        return __syncthreads_or(any) != 0;
    };
    if (!any_open(0)) return;
    __shared__ double sPhw[4][4][GF_MAXPH];
    double(*sPh)[GF_MAXPH] = sPhw[threadIdx.x / 64];
    GfDevClock *queue = tab[0].ck;
    const unsigned units = gridDim.x;
    const long nthr = (long)units * 256;
    for (;;) {
        const unsigned unit = queue_take(queue), phase = unit / units;
        const long tid = (long)(unit % units) * 256 + threadIdx.x;
        if (phase > 2u * (unsigned)(npass - 1)) return;
        if (!queue_wait(queue, phase * units)) {  // (not expected; no model's result is known then)
            for (int m = threadIdx.x; m < map.nm; m += 256)
                __hip_atomic_fetch_or(&tab[m].ck->q_timeout, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            return;
        }
        // passes up to `checked` are checked
        const int checked = (int)(phase / 2u), pass = checked + 1;
        if (pass == npass || (checked > 0 && !any_open(checked))) {
            if (phase % 2u != 0u) return;  // (settled)
            for (int m = 0; m < map.nm; m++) {
                GfDevClock *ck = tab[m].ck;
                const int last = __hip_atomic_load(&ck->th_last, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                const bool open = is_open(ck, checked);
                if (!open && last == 0) continue;
                if (tid == 0) therm_outcome(ck, open ? -1 : last);
                therm_settle(tab[m].P, bthermal(tab[m]), bslots(tab[m]), last, tid, nthr);
            }
        } else if (phase % 2u == 0u) {
            if (unit % units == 0u)
                for (int m = threadIdx.x; m < map.nm; m += 256)
                    __hip_atomic_store(flag(tab[m].ck, pass + 1), 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            for (int g = (int)(tid / 64); g < total; g += (int)(nthr / 64)) {
                const BatchEntry &b = bentry(tab, __builtin_amdgcn_readfirstlane(map.chunk[BK_TILE][g]));
                if (!is_open(b.ck, pass - 1)) continue;
                const GfDevArrays A = bthermal(b);
                therm_phase_table(b.P, sPh);
                const ThermIter it{pass % 2 == 1 ? A.xa : A.xb, pass % 2 == 0 ? A.xa : A.xb, arp, pass};
                const int t = g - (int)b.pt;
                if (t == 0 && threadIdx.x % 64 == 0)
                    __hip_atomic_store(&b.ck->th_last, pass, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                therm_strip<DIS, 1>(b.P, b.ck, A, b.tg, t, it, bslots(b), A.tbord + (long)t * TS_NB(b.tg.w),
                                    b.ck->dt, sPh);
            }
        } else {
            for (long g = tid - threadIdx.x; g < border; g += nthr) {
                const BatchEntry &b = bentry(tab, __builtin_amdgcn_readfirstlane(map.chunk[BK_BORD][g / BATCH_ALIGN]));
                const long t = g + threadIdx.x - b.pb;
                if (t < b.cb && is_open(b.ck, pass - 1))
                    therm_check_one(b.P, b.ck, bthermal(b), b.tg, t, pass, arp, bslots(b));
            }
        }
        queue_done(queue);
    }
}

// FP32-arithmetic mode: the thermal pipeline over the tiles of all models (k_therm_pipe,
// one workgroup per CU walking a list of tiles)
template <bool DIS>
__global__ void __launch_bounds__(1024) kb_therm_pipe(const BatchEntry *__restrict__ tab, BatchMap map, long total,
                                                      double stol, int arp, int fold)
{
    __shared__ ThermRaw raw;
    __shared__ double sU[TH_NF * TH_NE];
    __shared__ int sFlag[3];
    const long q = (total + 7) / 8, x = blockIdx.x % 8, r = blockIdx.x / 8, RW = gridDim.x / 8;
    const long first = x * q + r, end = min((x + 1) * q, total);
    if (first >= end) return;
    auto entry = [&](long t) -> const BatchEntry & { return bentry(tab, __builtin_amdgcn_readfirstlane(map.chunk[BK_TILE][t])); };
    {
        const BatchEntry &b = entry(first);
        therm_store_raw<DIS>(therm_prefetch<DIS>(b.P, b.ck, bthermal(b), (int)(first - b.pt), arp), raw);
    }
    for (long t = first; t < end; t += RW) {
        lds_barrier();  // this tile's inputs are in; the previous tile is done with sU
        const BatchEntry &b = entry(t);
        const long tn = t + RW;
        const BatchEntry &bn = entry(tn < end ? tn : t);
        therm_tile_pipe<DIS>(b.P, b.ck, bthermal(b), (int)(t - b.pt), bn.P, bn.ck, bthermal(bn),
                             tn < end ? (int)(tn - bn.pt) : -1, raw, sU, sFlag, stol, arp, fold);
    }
}
// its boundary conditions where the tiles do not apply them
__global__ void __launch_bounds__(256) kb_therm_bc(const BatchEntry *__restrict__ tab, BatchMap map)
{
    batch_apply<BK_NODE>(tab, map, [&](const BatchEntry &b, long t) { therm_bc_node(b.P, bthermal(b), t); });
}

template <int M>
__global__ void __launch_bounds__(256) kb_visc(const BatchEntry *__restrict__ tab, BatchMap map, int rot)
{
    batch_apply<BK_ELEM>(tab, map, [&](const BatchEntry &b, long e) { visc_body<M>(b.P, b.ck, b.A, e, rot); });
}

// rot: the batch's last element move left its stress/strain rotation to this kernel.
// chk: its first workgroups check the thermal borders of all models (`border` entries),
// as k_rheol1's do: the check's launch took 9.4 us of a step of 12 FP64 models.
// FP32 arithmetic: three waves per SIMD (168 VGPRs, with a few spills) where a model alone
// takes two: 24 models of 100-600 x 40-150 cells keep them all busy, 197 -> 191 us a step;
// 1000x250 cells alone lost 1.4 of 69 us that way.
template <bool SHEARH, int M>
__global__ void __launch_bounds__(256, M == 1 ? 3 : 2)
kb_rheol(const BatchEntry *__restrict__ tab, BatchMap map, int avgsr, int rot, int chk, long border, int arp)
{
    if (M != 1 && blockIdx.x < (unsigned)chk) {
        const long g = (long)blockIdx.x * blockDim.x;
        if (g >= border) return;
        const BatchEntry &b = bentry(tab, __builtin_amdgcn_readfirstlane(map.chunk[BK_BORD][g / BATCH_ALIGN]));
        const long t = g + threadIdx.x - b.pb;
        if (t < b.cb) therm_check_one(b.P, b.ck, bthermal(b), b.tg, t, 0, arp, bslots(b));
        return;
    }
    __shared__ RheolPhases phs;
    const long g0 = (long)xcd_block((unsigned)chk) * blockDim.x;
    const BatchEntry &b = bentry(tab, __builtin_amdgcn_readfirstlane(map.chunk[BK_ELEM][g0 / BATCH_ALIGN]));
    const long e = g0 + threadIdx.x - b.pe;
    rheol_single<SHEARH, typename Prec<M>::SV, typename Prec<M>::AT>(
        b.P, phs, b.ck, b.A, min(e, b.ce - 1), avgsr, rot, e < b.ce, [&]() {
            for (int k = threadIdx.x; k < RP_N * GF_MAXPH; k += blockDim.x)
                (&phs.f[0][0])[k] = rheol_phase_value(b.P, k);
            lds_barrier();
        });
}

// move: the coordinates move into cord_next as the node has its velocity (and the move's
// dt is recorded, for the rotation and the areas left pending)
template <int M>
__global__ void __launch_bounds__(256) kb_node(const BatchEntry *__restrict__ tab, BatchMap map, int move)
{
    batch_apply<BK_NODE>(tab, map, [&](const BatchEntry &b, long t) {
        node_body<M>(b.P, b.ck, b.A, t, move ? b.cord_next : nullptr);
        if (move && t == 0) b.ck->dt_move = b.ck->dt;
    });
}
// the negative-area STOP of moves whose areas are still pending (coordinates only)
__global__ void __launch_bounds__(256) kb_area_check(const BatchEntry *__restrict__ tab, BatchMap map)
{
    batch_apply<BK_ELEM>(tab, map, [&](const BatchEntry &b, long e) { area_check_body(b.P, b.ck, bmoved(b), e); });
}

__global__ void kb_clock_out(const BatchEntry *__restrict__ tab) { clock_out(tab[blockIdx.x].ck, tab[blockIdx.x].host); }

// the masses and dt minima after the step's move (arp: its areas are pending)
template <int M>
__global__ void __launch_bounds__(256) kb_dens(const BatchEntry *__restrict__ tab, BatchMap map, int rot)
{
    batch_apply<BK_ELEM>(tab, map, [&](const BatchEntry &b, long e) { dens_body<M>(b.P, b.ck, bmoved(b), e, rot); });
}

__global__ void __launch_bounds__(256) kb_rmass(const BatchEntry *__restrict__ tab, BatchMap map, int arp)
{
    batch_apply<BK_NODE>(tab, map, [&](const BatchEntry &b, long t) { rmass_body(b.P, b.ck, bmoved(b), t, arp); });
}

__global__ void __launch_bounds__(256) kb_amass(const BatchEntry *__restrict__ tab, BatchMap map, int arp)
{
    batch_apply<BK_NODE>(tab, map, [&](const BatchEntry &b, long t) { amass_body(b.P, b.ck, bmoved(b), t, arp); });
}
// both masses, with the dt scalars from the maxima of kb_dt_reduce (k_masses)
__global__ void __launch_bounds__(256) kb_masses(const BatchEntry *__restrict__ tab, BatchMap map, int arp)
{
    batch_apply<BK_NODE>(tab, map, [&](const BatchEntry &b, long t) {
        const double dlmin = dlmin_of(__longlong_as_double((long long)b.ck->dly_bits));
        const DtScal ds{dlmin, __longlong_as_double((long long)b.ck->velmax_bits), dt_elastic_of(b.P, b.ck, dlmin)};
        if (t == 0) dt_scalars_body(b.P, b.ck, dlmin);  // (nothing else here reads what it stores)
        masses_body(b.P, ds, bmoved(b), t, arp);
    });
}

// dt minima: `per` workgroups of 256 threads per model
#define BATCH_DT_BLOCKS 16
template <typename SV>
__global__ void __launch_bounds__(256) kb_dt_reduce(const BatchEntry *__restrict__ tab, BatchMap map, int arp)
{
    const int m = blockIdx.x / BATCH_DT_BLOCKS;
    if (m >= map.nm) return;
    const BatchEntry &b = bentry(tab, m);
    dt_reduce_body<SV>(b.P, b.ck, bmoved(b), blockIdx.x % BATCH_DT_BLOCKS, BATCH_DT_BLOCKS, arp);
}

__global__ void kb_dt_scalars(const BatchEntry *__restrict__ tab, BatchMap map)
{
    const int m = blockIdx.x * blockDim.x + threadIdx.x;
    if (m < map.nm)
        dt_scalars_body(tab[m].P, tab[m].ck, dlmin_of(__longlong_as_double((long long)tab[m].ck->dly_bits)));
}

// change_phase of every model with markers (gf_phase.h)
__global__ void __launch_bounds__(256) kb_phase_rules(const BatchEntry *__restrict__ tab, BatchMap map)
{
    batch_apply<BK_MARK>(tab, map, [&](const BatchEntry &b, long kk) { phase_rules_body(b.P, b.ck, b.A, kk); });
}
// the plan writes the model's active planes into its parameter block
__global__ void kb_phase_plan(const BatchEntry *__restrict__ tab, BatchMap map)
{
    const int m = blockIdx.x * blockDim.x + threadIdx.x;
    if (m < map.nm && tab[m].A.phstamp) phase_plan_body(const_cast<GfDevParams *>(tab[m].P), tab[m].ck);
}
__global__ void __launch_bounds__(256) kb_phase_update(const BatchEntry *__restrict__ tab, BatchMap map)
{
    batch_apply<BK_ELEM>(tab, map, [&](const BatchEntry &b, long e) {
        if (!b.A.phstamp) return;
        if (b.ck->ph_replan) phase_replane_body(b.P, b.ck, b.A, e);
        phase_recount_body(b.P, b.ck, b.A, e);
    });
}
