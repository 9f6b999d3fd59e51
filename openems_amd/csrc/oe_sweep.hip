// oe_sweep.hip -- a parameter sweep: many structures (each an oe_engine with
// its CPML, lumped-port DFT and excitations) stepped together.
//
// The reference runs one Simulation at a time (Simulation::run,
// src/fdtd/simulation.rs:255-326, batching timesteps per call,
// src/fdtd/batch.rs:17-34); it has no multi-structure launcher.  Here a
// half-step of all active structures is one launch: the work-groups of each
// structure's own launch (its tiles, and as riders its port DFT and source
// values) stand one after the other, found through a table.  Structures that
// need scalar lanes or have no material table go in launches per kernel
// variant beside it, sources and DFTs too large to ride in a point launch
// after it.  The step sequence between two termination checks is captured
// once as a HIP graph and replayed; structures that together outgrow the
// cache behind the L2s run it in sets that do not, one set after the other.  Each structure stops on its own energy decay or at
// max_steps; stopped structures leave the tables.  Checks fall on the
// engines' absolute timesteps and the peak is kept in the engine, so a run
// can continue where an earlier one stopped with the same result as one run.

#include "oe_objects.h"

#include <algorithm>
#include <chrono>
#include <cmath>
#include <cstring>
#include <memory>
#include <vector>

using namespace oe;

namespace {

struct Item {
    oe_engine* eng;
    oe_extension* cpml;
    oe_extension* port;
    std::vector<SweepExc> exc;              // target filled at run time
    std::vector<std::vector<float>> samples;
    std::vector<size_t> exc_off;            // element offsets of the targets
    // of the running run
    bool unit = false;       // in a UnitGroup
    bool fold = false;       // sources added by the E launch
    bool ride_port = false;  // port DFT carried by the launches
};

struct UnitGroup {  // one launch: the grids of one kind
    int axes;
    bool ragged;
    std::vector<SweepUnit> units;
    std::vector<int> wg_unit;
    int rows_h = 0, rows_e = 0;  // largest material tables
    const SweepUnit* d_unit = nullptr;  // device copies
    const int* d_wg = nullptr;
};

struct Group {      // one launch: all boxes of one (vec, axes) kind
    int vec, axes;
    std::vector<SweepBox> boxes;
    std::vector<int> wg_box;
    int n_wg = 0;
    const SweepBox* d_box = nullptr;  // device copies
    const int* d_wg = nullptr;
};

// Structures stepped together from check to check.
struct Set {
    std::vector<int> ids;
    std::vector<Group> groups;
    std::vector<UnitGroup> unit_groups;
    int stream_own = 1;
    uint64_t* step = nullptr;         // step under way, steps whose E half has begun
    int first_point = 0, n_point = 0;  // its structures in the point launch's tables
    hipGraph_t graph = nullptr;
    hipGraphExec_t exec = nullptr;
};

inline int ceil_div(int a, int b) { return (a + b - 1) / b; }

#define HIP_RET(expr)                          \
    do {                                       \
        const hipError_t e_ = (expr);          \
        if (e_ != hipSuccess) return e_;       \
    } while (0)

}  // namespace

struct oe_sweep {
    int device = 0;
    hipStream_t stream = nullptr;
    std::vector<Item> items;
    // planes per work-group along i: 32 microstrips of 0.2 to 1.3 M cells
    // take 301 / 295 / 299 / 324 us a step at 1 / 2 / 4 / 8
    int ci = 2;
    int xcd_remap = 1;
    // largest material table per half of the structures outside the units
    // (0: some structure reads its coefficient arrays, so every one does)
    int rows_h = 0, rows_e = 0;
    double tune_ms[4] = {0, 0, 0, 0};
    int tune_ci[4] = {1, 2, 4, 8};
    // device state of a run
    DevBuf structs, tables, rides, excs, exc_first, exc_serial, exc_samples, dfts, dft_of, ids, partials, energy, step;
    double* energy_host = nullptr;
    size_t energy_host_n = 0;
    std::vector<Set> sets;
    std::vector<Ride> ride_host;  // per structure, of the run (n_wg 0: none)
    // per structure, the (timestep, E + H energy) of every check of the last run
    std::vector<std::vector<std::pair<uint64_t, double>>> history;
    int graph_steps = 0;  // of every set's graph (0: not captured)
    // The CPML slab launches of a half-step run beside the interior launch,
    // each on a side stream of its own (forked and joined by events; graph
    // branches under capture).  OE_SWEEP_OVERLAP=1: all slab launches on one
    // side stream; 0: every launch on the sweep stream.
    int overlap = 2;
    hipStream_t side[3] = {nullptr, nullptr, nullptr};
    hipEvent_t ev_fork = nullptr, ev_join[3] = {nullptr, nullptr, nullptr};

    void drop_graph() {
        for (Set& t : sets) {
            if (t.exec) (void)hipGraphExecDestroy(t.exec);
            if (t.graph) (void)hipGraphDestroy(t.graph);
            t.exec = nullptr;
            t.graph = nullptr;
        }
        graph_steps = 0;
    }
    ~oe_sweep() {
        for (hipStream_t q : side)
            if (q) {
                (void)hipSetDevice(device);
                (void)hipStreamSynchronize(q);
            }
        if (stream) {
            (void)hipSetDevice(device);
            (void)hipStreamSynchronize(stream);
        }
        drop_graph();
        if (energy_host) (void)hipHostFree(energy_host);
        if (ev_fork) (void)hipEventDestroy(ev_fork);
        for (hipEvent_t q : ev_join)
            if (q) (void)hipEventDestroy(q);
        for (hipStream_t q : side)
            if (q) (void)hipStreamDestroy(q);
        if (stream) (void)hipStreamDestroy(stream);
    }
};

namespace {

// Boxes of one structure: with CPML the x-face slabs, the y-face slabs, the
// corner columns and the interior (z faces only), each with the kernel
// variant compiled for the faces it can hold; without CPML the whole grid
// (plain kernel).
void structure_boxes(const oe_sweep* sw, int sid, const Item& it, std::vector<Group>& groups) {
    const Grid& g = it.eng->g;
    const int vec = sweep_lanes(g, !it.cpml || it.cpml->cpml.zvec);
    const int nzv = ceil_div(g.nz, vec);
    SweepBox proto{};
    proto.sid = sid;
    proto.bx = std::min(64, nzv);
    proto.by = 256 / proto.bx;
    proto.n_kb = ceil_div(nzv, proto.bx);
    proto.ci = std::min(sw->ci, g.nx);
    auto add = [&](int axes, int i0, int i1, int j0, int j1) {
        if (i1 <= i0 || j1 <= j0) return;
        Group* G = nullptr;
        for (auto& q : groups)
            if (q.vec == vec && q.axes == axes) G = &q;
        if (!G) {
            groups.push_back(Group{vec, axes, {}, {}, 0, nullptr, nullptr});
            G = &groups.back();
        }
        SweepBox b = proto;
        b.i0 = i0; b.i1 = i1; b.j0 = j0; b.j1 = j1;
        // A box thinner in j than a work-group's rows (the y-face slabs and
        // corner columns: `layers` rows) stacks several i-chunks in one
        // work-group instead of leaving the surplus rows idle.
        const int rows = 256 / b.bx;
        b.by = std::min(rows, j1 - j0);
        b.ns = rows / b.by;
        b.n_jb = ceil_div(j1 - j0, b.by);
        const int n_ib = ceil_div(i1 - i0, b.ci * b.ns);
        b.first = G->n_wg;
        const int n = b.n_kb * b.n_jb * n_ib;
        for (int q = 0; q < n; ++q) G->wg_box.push_back((int)G->boxes.size());
        G->boxes.push_back(b);
        G->n_wg += n;
    };
    const CpmlArgs* cp = it.cpml ? &it.cpml->cpml : nullptr;
    if (!cp) {
        add(0, 0, g.nx, 0, g.ny);
        return;
    }
    const int m = cp->on_mask;
    const int ix0 = (m & 1) ? cp->L[0] : 0, ix1 = (m & 2) ? cp->g0[1] : g.nx;
    const int jy0 = (m & 4) ? cp->L[2] : 0, jy1 = (m & 8) ? cp->g0[3] : g.ny;
    // x slabs without the y-slab rows (x and z faces), y slabs without the
    // x-slab planes (y and z faces), the four corner columns (all faces):
    // the lighter kernels keep 3 waves per SIMD where the all-faces one has 2.
    const int all = AX_X | AX_Y | AX_Z;
    add(AX_X | AX_Z, 0, ix0, jy0, jy1);
    add(AX_X | AX_Z, ix1, g.nx, jy0, jy1);
    add(AX_Y | AX_Z, ix0, ix1, 0, jy0);
    add(AX_Y | AX_Z, ix0, ix1, jy1, g.ny);
    add(all, 0, ix0, 0, jy0);
    add(all, 0, ix0, jy1, g.ny);
    add(all, ix1, g.nx, 0, jy0);
    add(all, ix1, g.nx, jy1, g.ny);
    add((m & 48) ? AX_Z : 0, ix0, ix1, jy0, jy1);
}

// The active structures in sets.  State comes faster from the 256 MB behind
// the L2s than from memory, so where all structures together outgrow it and
// there are several steps from check to check, they are dealt to sets of up
// to 200 MB (32 microstrips of 450 MB: 318 us a step in one set, 294 in three,
// 357 in sets of 80 MB, whose launches are too small; 64 of 930 MB: 654 in
// one, 627 in sets of 240 MB, 611 in sets of 200).
void deal_sets(oe_sweep* sw, const std::vector<int>& active, uint64_t check) {
    sw->drop_graph();
    sw->sets.clear();
    auto state = [&](int sid) {
        const Item& it = sw->items[sid];
        return grid_state(it.eng, it.cpml ? &it.cpml->cpml : nullptr);
    };
    size_t total = 0;
    for (int sid : active) total += state(sid);
    const size_t most = (size_t)200 << 20;
    const bool deal = stream_state(total) && total > most && check >= 8;
    const size_t target = deal ? total / ((total + most - 1) / most) : total;
    size_t held = 0;
    for (int sid : active) {
        const size_t b = state(sid);
        if (sw->sets.empty() || (deal && held > 0 && (held + b > most || held + b / 2 > target))) {
            sw->sets.emplace_back();
            held = 0;
        }
        sw->sets.back().ids.push_back(sid);
        held += b;
        sw->sets.back().stream_own = stream_state(held);
    }
}

// Launch tables of the active structures, uploaded into sw->tables, and the
// sets' step counters after `done` steps.
oe_status build_tables(oe_sweep* sw, const std::vector<int>& active, uint64_t check, uint64_t done) {
    deal_sets(sw, active, check);
    const size_t n_sets = sw->sets.size();
    if (sw->step.bytes < 2 * n_sets * sizeof(uint64_t)) HIP_OK(sw->step.alloc(2 * n_sets * sizeof(uint64_t)));
    std::vector<uint64_t> counters;
    for (size_t q = 0; q < n_sets; ++q) {
        sw->sets[q].step = sw->step.as<uint64_t>() + 2 * q;
        counters.push_back(done - 1);  // -1 at first: the first H launch makes it 0
        counters.push_back(done);
    }
    for (Set& set : sw->sets) {
        for (int sid : set.ids) {
            const Item& it = sw->items[sid];
            sw->ride_host[sid].step_a = set.step;
            sw->ride_host[sid].step_b = set.step + 1;
            if (!it.unit) {
                structure_boxes(sw, sid, it, set.groups);
                continue;
            }
            SweepUnit u{};
            int axes = 0;
            if (!one_launch_plan(it.eng, it.cpml ? &it.cpml->cpml : nullptr, sw->ci, &u.a, &axes))
                return fail(OE_ERR_CONFIG, "structure %d has no single launch", sid);
            if (it.cpml) u.c = it.cpml->cpml;
            u.a.xcd_remap = 0;
            const Ride& r = sw->ride_host[sid];
            if (r.n_wg > 0) {
                u.a.ride = sw->rides.as<Ride>() + sid;
                u.a.n_ride = r.n_wg;
                u.a.src_val = r.src_val;
                u.a.n_src = r.n_src;
                for (int q = 0; q < r.n_src; ++q) u.a.src_idx[q] = (uint32_t)(it.exc_off[q] % it.eng->g.N);
            }
            UnitGroup* G = nullptr;
            for (auto& q : set.unit_groups)
                if (q.axes == axes && q.ragged == (u.a.ragged != 0)) G = &q;
            if (!G) {
                set.unit_groups.emplace_back();
                G = &set.unit_groups.back();
                G->axes = axes;
                G->ragged = u.a.ragged != 0;
            }
            u.first = (int)G->wg_unit.size();
            G->wg_unit.insert(G->wg_unit.end(), u.a.n_ride + u.a.first[u.a.nbox], (int)G->units.size());
            G->units.push_back(u);
            G->rows_h = std::max(G->rows_h, u.a.n_mat_h);
            G->rows_e = std::max(G->rows_e, u.a.n_mat_e);
        }
    }
    std::vector<char> host;
    auto put = [&](const void* p, size_t bytes) {
        const size_t at = host.size();
        host.resize((at + bytes + 63) / 64 * 64);
        std::memcpy(host.data() + at, p, bytes);
        return at;
    };
    std::vector<std::pair<size_t, size_t>> at;
    for (const Set& set : sw->sets) {
        for (const auto& G : set.groups) {
            const size_t b = put(G.boxes.data(), G.boxes.size() * sizeof(SweepBox));
            at.push_back({b, put(G.wg_box.data(), G.wg_box.size() * sizeof(int))});
        }
        for (const auto& G : set.unit_groups) {
            const size_t b = put(G.units.data(), G.units.size() * sizeof(SweepUnit));
            at.push_back({b, put(G.wg_unit.data(), G.wg_unit.size() * sizeof(int))});
        }
    }
    if (sw->tables.bytes < host.size()) HIP_OK(sw->tables.alloc(host.size()));
    HIP_OK(hipMemcpyAsync(sw->tables.p, host.data(), host.size(), hipMemcpyHostToDevice, sw->stream));
    HIP_OK(hipMemcpyAsync(sw->step.p, counters.data(), counters.size() * sizeof(uint64_t), hipMemcpyHostToDevice,
                          sw->stream));
    HIP_OK(hipMemcpyAsync(sw->rides.p, sw->ride_host.data(), sw->ride_host.size() * sizeof(Ride), hipMemcpyHostToDevice,
                          sw->stream));
    HIP_OK(hipStreamSynchronize(sw->stream));
    const char* base = sw->tables.as<char>();
    size_t q = 0;
    for (Set& set : sw->sets) {
        for (auto& G : set.groups) {
            G.d_box = reinterpret_cast<const SweepBox*>(base + at[q].first);
            G.d_wg = reinterpret_cast<const int*>(base + at[q++].second);
        }
        for (auto& G : set.unit_groups) {
            G.d_unit = reinterpret_cast<const SweepUnit*>(base + at[q].first);
            G.d_wg = reinterpret_cast<const int*>(base + at[q++].second);
        }
    }
    return OE_OK;
}

// The first launch advances the half's step counter.  The launches of one
// half write disjoint cells and read only the other field, so with
// sw->overlap the slab groups (x/y CPML faces) go to side streams, forked
// from and joined back into the sweep stream around its interior launch.
hipError_t yee_half(oe_sweep* sw, const Set& set, bool h) {
    uint64_t* inc = set.step + (h ? 0 : 1);
    for (const auto& G : set.unit_groups) {
        const UnitArgs a{G.d_unit, G.d_wg, sw->xcd_remap, set.stream_own, inc};
        inc = nullptr;
        HIP_RET(launch_units(h, a, (int)G.wg_unit.size(), G.axes, G.ragged, h ? G.rows_h : G.rows_e, sw->stream));
    }
    if (set.groups.empty()) return hipSuccess;
    const bool ov = sw->overlap && set.groups.size() > 1;
    const int n_side = sw->overlap == 2 ? 3 : 1;
    int used = 0;  // side streams forked so far
    if (ov) HIP_RET(hipEventRecord(sw->ev_fork, sw->stream));
    for (const auto& G : set.groups) {
        SweepArgs a{};
        a.st = sw->structs.as<SweepStruct>();
        a.box = G.d_box;
        a.wg_box = G.d_wg;
        a.xcd_remap = sw->xcd_remap;
        a.step_inc = inc;
        inc = nullptr;
        hipStream_t st = sw->stream;
        if (ov && (G.axes & (AX_X | AX_Y)) != 0) {
            // slab group: the next side stream (or the one side stream)
            const int q = std::min(used, n_side - 1);
            if (q == used) {
                HIP_RET(hipStreamWaitEvent(sw->side[q], sw->ev_fork, 0));
                ++used;
            }
            st = sw->side[q];
        }
        hipError_t e = launch_sweep(h, a, G.n_wg, G.axes, G.vec, h ? sw->rows_h : sw->rows_e, st);
        if (e != hipSuccess) return e;
    }
    for (int q = 0; q < used; ++q) {
        HIP_RET(hipEventRecord(sw->ev_join[q], sw->side[q]));
        HIP_RET(hipStreamWaitEvent(sw->stream, sw->ev_join[q], 0));
    }
    return hipSuccess;
}

// Point and DFT tables of the active structures, set by set.
oe_status build_step_tables(oe_sweep* sw, const std::vector<int>& active) {
    std::vector<SweepExc> ex;
    std::vector<int> first{0};
    std::vector<int> serial, dft_of;
    std::vector<SweepDft> dft;
    int n = 0;
    for (Set& set : sw->sets) {
        set.first_point = n;
        set.n_point = 0;
        for (int sid : set.ids) {
            const Item& it = sw->items[sid];
            const bool own_exc = !it.fold && !it.exc.empty(), own_dft = it.port && !it.ride_port;
            if (!own_exc && !own_dft) continue;
            ++n;
            ++set.n_point;
            if (own_exc)
                for (const auto& e : it.exc) ex.push_back(e);
            first.push_back((int)ex.size());
            // sources on one cell apply in list order: then one thread does them all
            std::vector<const float*> cells;
            if (own_exc)
                for (const auto& e : it.exc) cells.push_back(e.target);
            std::sort(cells.begin(), cells.end());
            serial.push_back(std::adjacent_find(cells.begin(), cells.end()) != cells.end() ? 1 : 0);
            dft_of.push_back(own_dft ? (int)dft.size() : -1);
            if (own_dft) {
                SweepDft d{};
                d.F = it.eng->F;
                d.N = it.eng->g.N;
                d.d = it.port->dft;
                d.sample0 = it.port->dft_count;
                d.t0 = (double)it.eng->timestep;
                dft.push_back(d);
            }
    }
    }
    if (sw->excs.bytes < std::max<size_t>(ex.size(), 1) * sizeof(SweepExc))
        HIP_OK(sw->excs.alloc(std::max<size_t>(ex.size(), 1) * sizeof(SweepExc)));
    if (sw->exc_first.bytes < first.size() * sizeof(int)) HIP_OK(sw->exc_first.alloc(first.size() * sizeof(int)));
    const size_t nb_struct = std::max<size_t>(active.size(), 1) * sizeof(int);
    if (sw->exc_serial.bytes < nb_struct) HIP_OK(sw->exc_serial.alloc(nb_struct));
    if (sw->dft_of.bytes < nb_struct) HIP_OK(sw->dft_of.alloc(nb_struct));
    if (n > 0) {
        HIP_OK(hipMemcpyAsync(sw->exc_serial.p, serial.data(), serial.size() * sizeof(int), hipMemcpyHostToDevice,
                              sw->stream));
        HIP_OK(hipMemcpyAsync(sw->dft_of.p, dft_of.data(), dft_of.size() * sizeof(int), hipMemcpyHostToDevice,
                              sw->stream));
    }
    if (sw->dfts.bytes < std::max<size_t>(dft.size(), 1) * sizeof(SweepDft))
        HIP_OK(sw->dfts.alloc(std::max<size_t>(dft.size(), 1) * sizeof(SweepDft)));
    if (!ex.empty()) HIP_OK(hipMemcpyAsync(sw->excs.p, ex.data(), ex.size() * sizeof(SweepExc), hipMemcpyHostToDevice, sw->stream));
    HIP_OK(hipMemcpyAsync(sw->exc_first.p, first.data(), first.size() * sizeof(int), hipMemcpyHostToDevice, sw->stream));
    if (!dft.empty()) HIP_OK(hipMemcpyAsync(sw->dfts.p, dft.data(), dft.size() * sizeof(SweepDft), hipMemcpyHostToDevice, sw->stream));
    if (sw->ids.bytes < std::max<size_t>(active.size(), 1) * sizeof(int))
        HIP_OK(sw->ids.alloc(std::max<size_t>(active.size(), 1) * sizeof(int)));
    if (!active.empty())
        HIP_OK(hipMemcpyAsync(sw->ids.p, active.data(), active.size() * sizeof(int), hipMemcpyHostToDevice, sw->stream));
    HIP_OK(hipStreamSynchronize(sw->stream));
    return OE_OK;
}

// One timestep of a set's structures (no host synchronisation; capturable).
hipError_t sweep_step(oe_sweep* sw, const Set& set, double dt) {
    // the first H launch advances the step counter (from -1: step st reads st)
    HIP_RET(yee_half(sw, set, true));
    HIP_RET(yee_half(sw, set, false));
    if (set.n_point == 0) return hipSuccess;
    return launch_sweep_point(sw->excs.as<SweepExc>(), sw->exc_first.as<int>() + set.first_point,
                              sw->exc_serial.as<int>() + set.first_point, sw->dfts.as<SweepDft>(),
                              sw->dft_of.as<int>() + set.first_point, set.n_point, set.step, dt, sw->stream);
}

oe_status capture(oe_sweep* sw, double dt, int steps) {
    sw->drop_graph();
    for (Set& set : sw->sets) {
        HIP_OK(hipStreamBeginCapture(sw->stream, hipStreamCaptureModeThreadLocal));
        hipError_t err = hipSuccess;
        for (int q = 0; q < steps && err == hipSuccess; ++q) err = sweep_step(sw, set, dt);
        hipGraph_t g = nullptr;
        const hipError_t ec = hipStreamEndCapture(sw->stream, &g);
        if (err != hipSuccess || ec != hipSuccess) {
            if (g) (void)hipGraphDestroy(g);
            return fail(OE_ERR_DEVICE, "sweep graph capture failed: %s", hipGetErrorString(err != hipSuccess ? err : ec));
        }
        set.graph = g;
        HIP_OK(hipGraphInstantiate(&set.exec, set.graph, nullptr, nullptr, 0));
    }
    sw->graph_steps = steps;
    return OE_OK;
}

// The riders of the run: port DFTs and source values of the structures in
// units (build_tables adds the set's counters and uploads them).  Samples are on the device (it.exc[q].samples).
oe_status build_rides(oe_sweep* sw, uint64_t t0, double dt) {
    const size_t n = sw->items.size();
    sw->ride_host.assign(n, Ride{});
    std::vector<PointExc> src;
    for (auto& it : sw->items) {
        const Grid& g = it.eng->g;
        YeeArgs a;
        int axes;
        it.unit = one_launch_plan(it.eng, it.cpml ? &it.cpml->cpml : nullptr, 1, &a, &axes);
        const bool riding = it.unit && it.eng->ride;
        it.fold = riding && !it.exc.empty() && it.exc.size() <= (size_t)MAX_FOLD_SOURCES;
        for (size_t off : it.exc_off) {  // cells the E update writes
            const size_t cell = off % g.N, plane = (size_t)g.ny * g.nz;
            if (cell < plane || cell % plane < (size_t)g.nz) it.fold = false;
        }
        it.ride_port = riding && it.port && dft_rides(it.port);
        if (it.fold) src.resize(src.size() + it.exc.size());
    }
    const size_t src_off = (n * sizeof(Ride) + 63) / 64 * 64;
    const size_t val_off = (src_off + src.size() * sizeof(PointExc) + 63) / 64 * 64;
    const size_t bytes = val_off + n * MAX_FOLD_SOURCES * sizeof(SourceValue);
    if (sw->rides.bytes < bytes) HIP_OK(sw->rides.alloc(bytes));
    size_t at = 0;
    for (size_t s = 0; s < n; ++s) {
        const Item& it = sw->items[s];
        Ride& r = sw->ride_host[s];
        r.F = it.eng->F;
        r.g = it.eng->g;
        r.t0 = (double)t0;
        r.dt = dt;
        if (it.fold) {
            r.n_src = (int)it.exc.size();
            r.src = reinterpret_cast<const PointExc*>(sw->rides.as<char>() + src_off) + at;
            r.src_val = reinterpret_cast<SourceValue*>(sw->rides.as<char>() + val_off) + s * MAX_FOLD_SOURCES;
            for (size_t q = 0; q < it.exc.size(); ++q) {
                PointExc& x = src[at++];
                x.idx = (uint32_t)(it.exc_off[q] % it.eng->g.N);
                x.comp = (uint32_t)(it.exc_off[q] / it.eng->g.N);
                x.soft = it.exc[q].soft;
                x.zero_after = 1;  // as the point launch does
                x.samples = it.exc[q].samples;
                x.n_samples = it.exc[q].n_samples;
            }
        }
        r.first_dft = it.fold ? 1 : 0;
        if (it.ride_port) r.dft[r.n_dft++] = RideDft{it.port->dft, it.port->dft_count};
        r.first_ade = r.first_mur = r.n_wg = r.first_dft + r.n_dft;
    }
    if (!src.empty())
        HIP_OK(hipMemcpyAsync(sw->rides.as<char>() + src_off, src.data(), src.size() * sizeof(PointExc),
                              hipMemcpyHostToDevice, sw->stream));
    HIP_OK(hipStreamSynchronize(sw->stream));
    return OE_OK;
}

// The E signals of the last step of structures that stop.
oe_status ride_last(oe_sweep* sw, const std::vector<int>& stopping) {
    std::vector<int> ids;
    for (int s : stopping)
        if (sw->items[s].ride_port) ids.push_back(s);
    if (ids.empty()) return OE_OK;
    if (sw->ids.bytes < ids.size() * sizeof(int)) HIP_OK(sw->ids.alloc(ids.size() * sizeof(int)));
    HIP_OK(hipMemcpyAsync(sw->ids.p, ids.data(), ids.size() * sizeof(int), hipMemcpyHostToDevice, sw->stream));
    HIP_OK(launch_ride_last_many(sw->rides.as<Ride>(), sw->ids.as<int>(), (int)ids.size(), 2, sw->stream));
    HIP_OK(hipStreamSynchronize(sw->stream));
    return OE_OK;
}

oe_status energies(oe_sweep* sw, int n) {
    if (n <= 0) return OE_OK;
    const size_t need = (size_t)n * 2 * energy_blocks() * sizeof(double);
    if (sw->partials.bytes < need) HIP_OK(sw->partials.alloc(need));
    if (sw->energy.bytes < (size_t)n * 2 * sizeof(double)) HIP_OK(sw->energy.alloc((size_t)n * 2 * sizeof(double)));
    if (sw->energy_host_n < (size_t)n) {
        if (sw->energy_host) (void)hipHostFree(sw->energy_host);
        sw->energy_host = nullptr;
        sw->energy_host_n = 0;
        HIP_OK(hipHostMalloc(&sw->energy_host, (size_t)n * 2 * sizeof(double), hipHostMallocDefault));
        sw->energy_host_n = n;
    }
    HIP_OK(launch_sweep_energy(sw->structs.as<SweepStruct>(), sw->ids.as<int>(), n, sw->partials.as<double>(),
                               sw->energy.as<double>(), sw->stream));
    HIP_OK(hipMemcpyAsync(sw->energy_host, sw->energy.p, (size_t)n * 2 * sizeof(double), hipMemcpyDeviceToHost, sw->stream));
    HIP_OK(hipStreamSynchronize(sw->stream));
    return OE_OK;
}

}  // namespace

extern "C" {

oe_status oe_sweep_create(int device, oe_sweep** out) {
    if (!out) return fail(OE_ERR_CONFIG, "null argument");
    int n = 0;
    if (hipGetDeviceCount(&n) != hipSuccess || n <= 0) return fail(OE_ERR_DEVICE, "no HIP device available");
    if (device < 0 || device >= n) return fail(OE_ERR_CONFIG, "device %d out of range", device);
    std::unique_ptr<oe_sweep> sw(new oe_sweep());
    sw->device = device;
    HIP_OK(hipSetDevice(device));
    HIP_OK(hipStreamCreateWithFlags(&sw->stream, hipStreamNonBlocking));
    if (const char* v = getenv("OE_SWEEP_OVERLAP")) sw->overlap = std::min(std::max(atoi(v), 0), 2);
    if (sw->overlap) {
        HIP_OK(hipEventCreateWithFlags(&sw->ev_fork, hipEventDisableTiming));
        for (int q = 0; q < (sw->overlap == 2 ? 3 : 1); ++q) {
            HIP_OK(hipStreamCreateWithFlags(&sw->side[q], hipStreamNonBlocking));
            HIP_OK(hipEventCreateWithFlags(&sw->ev_join[q], hipEventDisableTiming));
        }
    }
    *out = sw.release();
    return OE_OK;
}

void oe_sweep_destroy(oe_sweep* sw) { delete sw; }

oe_status oe_sweep_add(oe_sweep* sw, oe_engine* e, oe_extension* cpml, oe_extension* port,
                       const oe_excitation* exc, size_t n_exc, size_t* index) {
    if (!sw || !e) return fail(OE_ERR_CONFIG, "null argument");
    if (n_exc && !exc) return fail(OE_ERR_CONFIG, "excitations is null");
    if (e->device != sw->device) return fail(OE_ERR_CONFIG, "engine on another device");
    for (const auto& it : sw->items)
        if (it.eng == e) return fail(OE_ERR_CONFIG, "engine already in the sweep");
    if (!sw->items.empty() && std::fabs(e->dt - sw->items[0].eng->dt) > 1e-12 * sw->items[0].eng->dt)
        return fail(OE_ERR_CONFIG, "all structures of a sweep share one timestep (dt differs)");
    if (cpml) {
        if (cpml->kind != EXT_CPML || cpml->eng != e) return fail(OE_ERR_CONFIG, "cpml is not this engine's CPML");
        if (!cpml->cpml.physical) return fail(OE_ERR_CONFIG, "a sweep runs the physical CPML mode only");
    }
    if (port) {
        if (port->kind != EXT_DFT || port->eng != e) return fail(OE_ERR_CONFIG, "port is not a DFT of this engine");
        if (port->dft.n_sig > 256) return fail(OE_ERR_CONFIG, "a sweep DFT holds at most 256 signals");
        if (port->dft_stride != 1) return fail(OE_ERR_CONFIG, "a sweep DFT samples every step");
    }
    Item it{};
    it.eng = e;
    it.cpml = cpml;
    it.port = port;
    for (size_t q = 0; q < n_exc; ++q) {
        const oe_excitation& x = exc[q];
        if (x.i >= (uint32_t)e->g.nx || x.j >= (uint32_t)e->g.ny || x.k >= (uint32_t)e->g.nz || x.direction > 2)
            return fail(OE_ERR_CONFIG, "excitation %zu out of the grid", q);
        if (x.n_samples && !x.samples) return fail(OE_ERR_CONFIG, "excitation %zu has no samples", q);
        SweepExc s{};
        s.n_samples = x.n_samples;
        s.soft = x.soft ? 1u : 0u;
        it.exc.push_back(s);
        it.samples.emplace_back(x.samples, x.samples + x.n_samples);
        it.exc_off.push_back((size_t)x.direction * e->g.N + ((size_t)x.i * e->g.ny + x.j) * e->g.nz + x.k);
    }
    sw->items.push_back(std::move(it));
    if (index) *index = sw->items.size() - 1;
    return OE_OK;
}

oe_status oe_sweep_run(oe_sweep* sw, const oe_sweep_config* cfg, oe_sweep_entry* results) {
    if (!sw || !cfg || !results) return fail(OE_ERR_CONFIG, "null argument");
    if (sw->items.empty()) return fail(OE_ERR_CONFIG, "empty sweep");
    if (cfg->max_steps == 0) return fail(OE_ERR_CONFIG, "max_steps must be positive");
    HIP_OK(hipSetDevice(sw->device));
    const auto t0 = std::chrono::steady_clock::now();
    const int n = (int)sw->items.size();
    const uint64_t check = cfg->check_interval ? cfg->check_interval : 100;
    const double dt = sw->items[0].eng->dt;
    const uint64_t T0 = sw->items[0].eng->timestep;  // timestep of the run's first step
    for (auto& it : sw->items) {
        if (it.eng->timestep != T0)
            return fail(OE_ERR_CONFIG, "structures of a sweep run start at one timestep (%llu and %llu)",
                        (unsigned long long)T0, (unsigned long long)it.eng->timestep);
        HIP_OK(hipStreamSynchronize(it.eng->stream));
    }

    // static device data: structures, excitation samples
    std::vector<SweepStruct> st(n);
    size_t total = 0;
    for (int s = 0; s < n; ++s) {
        const Item& it = sw->items[s];
        st[s].g = it.eng->g;
        st[s].F = it.eng->F;
        st[s].Cf = it.eng->Cf;
        if (it.cpml) st[s].c = it.cpml->cpml;
        if (it.eng->mat) {
            st[s].mat_e = it.eng->mat;
            st[s].mat_h = it.eng->mat + it.eng->g.N;
            st[s].tab_e = it.eng->mtab;
            st[s].tab_h = it.eng->mtab + (size_t)MAX_MAT_ROWS * 6;
            st[s].n_mat_e = it.eng->n_mat[0];
            st[s].n_mat_h = it.eng->n_mat[1];
            if (it.eng->mat8) {
                if (st[s].n_mat_e >= 2 && st[s].n_mat_e <= 256) st[s].mat8_e = it.eng->mat8;
                if (st[s].n_mat_h >= 2 && st[s].n_mat_h <= 256) st[s].mat8_h = it.eng->mat8 + it.eng->g.N;
            }
        }
        for (const auto& v : it.samples) total += v.size();
    }
    HIP_OK(sw->structs.alloc(n * sizeof(SweepStruct)));
    HIP_OK(hipMemcpyAsync(sw->structs.p, st.data(), n * sizeof(SweepStruct), hipMemcpyHostToDevice, sw->stream));
    HIP_OK(sw->exc_samples.alloc(std::max<size_t>(total, 1) * sizeof(float)));
    size_t off = 0;
    for (auto& it : sw->items)
        for (size_t q = 0; q < it.exc.size(); ++q) {
            it.exc[q].target = it.eng->F + it.exc_off[q];
            it.exc[q].samples = sw->exc_samples.as<float>() + off;
            if (!it.samples[q].empty())
                HIP_OK(hipMemcpyAsync(sw->exc_samples.as<float>() + off, it.samples[q].data(),
                                      it.samples[q].size() * sizeof(float), hipMemcpyHostToDevice, sw->stream));
            off += it.samples[q].size();
        }
    OE_TRY(build_rides(sw, T0, dt));
    sw->rows_e = sw->rows_h = 0;
    bool all_e = true, all_h = true;
    for (int s = 0; s < n; ++s) {
        if (sw->items[s].unit) continue;
        all_e = all_e && st[s].n_mat_e > 0;
        all_h = all_h && st[s].n_mat_h > 0;
        sw->rows_e = std::max(sw->rows_e, st[s].n_mat_e);
        sw->rows_h = std::max(sw->rows_h, st[s].n_mat_h);
    }
    if (!all_e) sw->rows_e = 0;
    if (!all_h) sw->rows_h = 0;

    std::vector<int> active(n);
    for (int s = 0; s < n; ++s) active[s] = s;
    std::vector<double> peak(n, 0.0);
    for (int s = 0; s < n; ++s) peak[s] = sw->items[s].eng->peak_persistent;
    sw->history.assign(n, {});
    for (int s = 0; s < n; ++s) {
        results[s] = oe_sweep_entry{};
        results[s].termination_reason = OE_TERM_STEPS_COMPLETED;
    }

    // The i-depth of the work-groups, timed over the run's own first steps
    // after its first check (no result depends on it), TUNE_STEPS of each
    // candidate.
    struct Events {
        hipEvent_t a = nullptr, b = nullptr;
        ~Events() {
            if (a) (void)hipEventDestroy(a);
            if (b) (void)hipEventDestroy(b);
        }
    } ev;
    constexpr int TUNE_STEPS = 5;
    int tune_next = cfg->autotune ? 0 : 4, tune_best = 0;
    if (cfg->autotune) {
        HIP_OK(hipEventCreate(&ev.a));
        HIP_OK(hipEventCreate(&ev.b));
        for (double& ms : sw->tune_ms) ms = 0.0;
    }

    OE_TRY(build_tables(sw, active, check, 0));
    OE_TRY(build_step_tables(sw, active));
    uint64_t done = 0;
    sw->drop_graph();
    while (!active.empty() && done < cfg->max_steps) {
        // Energy is sampled after the steps whose timestep is a multiple of
        // check (0, check, 2 check, ...), as a single engine with
        // sample_interval = check_interval does: from timestep 0, step 0
        // alone, then chunks of check steps.
        const uint64_t ts = T0 + done;                            // timestep of the next step
        const uint64_t next_check = (ts + check - 1) / check * check;  // first check at or after it
        const uint64_t chunk = std::min<uint64_t>(next_check - ts + 1, cfg->max_steps - done);
        uint64_t ran = 0;
        while (tune_next < 4 && done > 0 && chunk - ran >= TUNE_STEPS) {
            const int q = tune_next++;
            sw->ci = sw->tune_ci[q];
            OE_TRY(build_tables(sw, active, check, done + ran));
            OE_TRY(build_step_tables(sw, active));
            HIP_OK(hipEventRecord(ev.a, sw->stream));
            for (const Set& set : sw->sets)
                for (int w = 0; w < TUNE_STEPS; ++w) HIP_OK(sweep_step(sw, set, dt));
            HIP_OK(hipEventRecord(ev.b, sw->stream));
            HIP_OK(hipEventSynchronize(ev.b));
            float ms = 0.f;
            HIP_OK(hipEventElapsedTime(&ms, ev.a, ev.b));
            sw->tune_ms[q] = ms / TUNE_STEPS;
            if (sw->tune_ms[q] < sw->tune_ms[tune_best]) tune_best = q;
            ran += TUNE_STEPS;
            if (tune_next == 4 || chunk - ran < TUNE_STEPS) {
                sw->ci = sw->tune_ci[tune_best];
                OE_TRY(build_tables(sw, active, check, done + ran));
                OE_TRY(build_step_tables(sw, active));
            }
        }
        if (cfg->use_graph && chunk == check && done > 0 && ran == 0) {
            // the graph holds a divisor of the check interval (at most 25
            // steps) and is launched check / gsteps times: the active set
            // changes at many checks, and instantiating a short graph costs
            // a fraction of a long one
            int gsteps = 1;
            for (int q = 1; q <= 25; ++q)
                if (check % q == 0) gsteps = q;
            if (sw->graph_steps != gsteps) OE_TRY(capture(sw, dt, gsteps));
            for (const Set& set : sw->sets)
                for (uint64_t q = 0; q < chunk / gsteps; ++q) HIP_OK(hipGraphLaunch(set.exec, sw->stream));
        } else {
            for (const Set& set : sw->sets)
                for (uint64_t q = ran; q < chunk; ++q) HIP_OK(sweep_step(sw, set, dt));
        }
        done += chunk;
        const uint64_t cur = T0 + done - 1;  // timestep of the last step run
        if (cur % check != 0) continue;  // max_steps reached between checks
        OE_TRY(energies(sw, (int)active.size()));
        std::vector<int> keep;
        for (size_t q = 0; q < active.size(); ++q) {
            const int s = active[q];
            const double E = sw->energy_host[2 * q] + sw->energy_host[2 * q + 1];
            peak[s] = std::max(peak[s], E);
            sw->history[s].push_back({cur, E});
            results[s].final_energy = E;
            results[s].peak_energy = peak[s];
            bool stop = false;
            // src/fdtd/basic_engine.rs:128-141, with the engine's persistent peak
            if (cfg->has_energy_decay_db && cur > 0 && peak[s] > 0.0 && E > 0.0) {
                const double ddb = 10.0 * std::log10(E / peak[s]);
                if (ddb < -std::fabs(cfg->energy_decay_db)) {
                    stop = true;
                    results[s].termination_reason = OE_TERM_ENERGY_DECAY;
                    results[s].final_decay_db = ddb;
                }
            }
            if (stop) results[s].timesteps_executed = done;
            else keep.push_back(s);
        }
        if (keep.size() != active.size()) {
            std::vector<int> stopping;
            for (int s : active)
                if (results[s].termination_reason == OE_TERM_ENERGY_DECAY) stopping.push_back(s);
            OE_TRY(ride_last(sw, stopping));
            active.swap(keep);
            if (!active.empty()) {
                OE_TRY(build_tables(sw, active, check, done));
                OE_TRY(build_step_tables(sw, active));
            }
        }
    }
    OE_TRY(ride_last(sw, active));
    HIP_OK(hipStreamSynchronize(sw->stream));
    for (int s : active) results[s].timesteps_executed = done;
    // Engines and port DFTs advance by the steps each structure ran.
    for (int s = 0; s < n; ++s) {
        Item& it = sw->items[s];
        it.eng->timestep += results[s].timesteps_executed;
        it.eng->peak_persistent = peak[s];
        if (it.port) {
            it.port->dft_count += results[s].timesteps_executed;
            it.port->dft_seen += results[s].timesteps_executed;
        }
    }
    sw->drop_graph();
    const double wall = std::chrono::duration<double>(std::chrono::steady_clock::now() - t0).count();
    for (int s = 0; s < n; ++s) results[s].elapsed_seconds = wall;
    return OE_OK;
}

oe_status oe_sweep_tuning(const oe_sweep* sw, int* ci, double ms_per_step[4], int candidates[4]) {
    if (!sw) return fail(OE_ERR_CONFIG, "null argument");
    if (ci) *ci = sw->ci;
    for (int q = 0; q < 4; ++q) {
        if (ms_per_step) ms_per_step[q] = sw->tune_ms[q];
        if (candidates) candidates[q] = sw->tune_ci[q];
    }
    return OE_OK;
}

oe_status oe_sweep_energy_history(const oe_sweep* sw, size_t index, uint64_t* timesteps, double* energies,
                                  size_t capacity, size_t* n) {
    if (!sw) return fail(OE_ERR_CONFIG, "null argument");
    if (index >= sw->history.size()) return fail(OE_ERR_CONFIG, "structure %zu has no history (run the sweep first)", index);
    const auto& h = sw->history[index];
    if (n) *n = h.size();
    const size_t m = std::min(capacity, h.size());
    for (size_t q = 0; q < m; ++q) {
        if (timesteps) timesteps[q] = h[q].first;
        if (energies) energies[q] = h[q].second;
    }
    return OE_OK;
}

oe_status oe_sweep_set_ci(oe_sweep* sw, int ci) {
    if (!sw) return fail(OE_ERR_CONFIG, "null argument");
    if (ci < 1 || ci > 1024) return fail(OE_ERR_CONFIG, "ci out of range");
    sw->ci = ci;
    return OE_OK;
}

}  // extern "C"
