// Device-side phonon transport for gfx950.
//
// One lane owns one phonon.  The event loop is psim's ModelSimulator::simulatePhonon
// (psim/src/modelSimulator.cpp:139-198) with handleImpacts (:205-225), nextImpact (:87-122),
// scatter (:124-137), the surface handlers (psim/src/surface.cpp:23-109,
// compositeSurface.cpp:47-66, cell.cpp:103-108) and the geometry predicates of
// psim/src/geometry.cpp.  Every floating-point expression keeps the reference's operation
// order (the library is built with -ffp-contract=off), so a lane reproduces the CPU oracle's
// trajectory bit for bit given the same Philox stream.
//
// Phonon state lives in registers for a whole launch window of measurement steps and is
// written back to the structure-of-arrays pool only when the window ends.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "psim_gpu.h"
#include "psim_math.h"
#include "psim_rng.h"

namespace psim_dev {

constexpr double GEOEPS = __DBL_EPSILON__ * 1E9;  // utils.h:10
constexpr double SCALING_FACTOR = 1e9;  // modelSimulator.cpp:17
constexpr double VELOCITY_EPS = 0.01;  // modelSimulator.cpp:23
constexpr int MAX_COLLISIONS = 100;  // modelSimulator.cpp:25
constexpr double HBAR = 1.054517e-34;  // material.cpp:12
constexpr double BOLTZ = 1.38065e-23;  // material.cpp:13
constexpr int NBINS = PSIM_NUM_FREQ_BINS;
constexpr int GUIDE = 2048;  // guide-table cells per frequency table (a power of two)

enum : int { POL_LA = 0, POL_TA = 1 };
enum : int { FATE_ABSORBED = 1, FATE_EXPIRED = 2, FATE_NOT_STARTED = 3, FATE_STALLED = 4 };

// Phonon record word: bits 0-9 frequency bin (emission pool), bit 10 TA, bit 11 negative sign, bit 12
// impurities scatter it (Rates::impurity), bits 16-31 random-stream index (the model's index in a batch, 0 otherwise).
constexpr uint32_t META_BIN = (1u << 10) - 1u;
constexpr uint32_t META_TA = 1u << 10;
constexpr uint32_t META_NEG = 1u << 11;
constexpr uint32_t META_IMPURITY = 1u << 12;
constexpr int META_STREAM_SHIFT = 16;

// A cell whose three edges run from corner to corner, as the impact search and the surface stage read
// it: one cache line.  The corners stand once, so what the edges' tests need of each (its differences to
// the path, the side of the path it lies on, its place against the path's box) is computed once, not for
// the two edges that meet there.
struct __attribute__((aligned(128))) Tri {
    double2 corner[3];  // edge b runs from corner b to corner (b + 1) % 3
    int32_t sub_begin[3];  // of each edge's sub-surfaces, transitions first
    uint32_t info;  // their numbers, TRI_SUB_BITS bits each, then a bit for each vertical edge
    double2 line[3];  // slope and intercept; a vertical edge's x instead of its slope
    double pad_[2];
};
constexpr int TRI_SUB_BITS = 4;  // a model with an edge of more than 15 sub-surfaces uses Edge

// One of a cell's three edges, for models whose cells are not all such triangles.
// `vert`: its ends have the same x up to rounding (rel_equals, tested once at upload).
struct __attribute__((aligned(16))) Edge {
    double p1x, p1y, p2x, p2y;
    double slope, intercept;  // a vertical edge's x instead of its slope
    int32_t vert;
    int32_t sub_begin, n_sub;  // its sub-surfaces, transitions first
    int32_t pad_;
};

// What a phonon reflects off: an edge's or a sub-surface's normal and specularity.
struct __attribute__((aligned(16))) Wall {
    double nx, ny, spec, pad_;
};

// A sub-surface: the line its containment test needs, then what a hit on it does.  The neighbour's
// sensor stands beside the neighbour, so a transition needs no lookup of the cell entered.
struct __attribute__((aligned(16))) Sub {
    double p1x, p1y, p2x, p2y;
    int32_t kind, target, target_sensor, same_material;
    double start, duration;
    double max_freq_la, max_freq_ta;
};

// What scattering in a sensor reads, its material's constants among it: one record, one address, so
// the loads of a scattering phonon go out together instead of sensor first, material next.
struct __attribute__((aligned(16))) Sensor {
    double b_l, t3;
    double b_tn, t4;
    double b_tu, b_i;
    double w, tk;  // tk = t_init x BOLTZ
    double r_tk, pad0_;  // 1 / tk, rounded to nearest
    int32_t material, scatter_table, flight_cap, pad_;
};

// A frequency bin of a material, with the material's bin width.
struct __attribute__((aligned(16))) Bin {
    double freq, vel_la, vel_ta, width;
};

// A frequency table: cumulative distribution, LA share of each bin and the start indices of the
// frequency search.
struct __attribute__((aligned(16))) Table {
    double cdf[NBINS], frac[NBINS];
    uint16_t guide[GUIDE + 1], pad_[7];
};

struct Model {
    const psim_cell* __restrict__ cells;
    const Tri* __restrict__ tris;  // [n_cells], read where every cell is one (TRI)
    const Edge* __restrict__ edges;  // [3 * n_cells]
    const Wall* __restrict__ walls;  // [3 * n_cells] of the edges, then [n_subs] of the sub-surfaces
    const Sub* __restrict__ subs;
    const Sensor* __restrict__ sensors;
    const Bin* __restrict__ bins;  // [n_materials][NBINS]
    const Table* __restrict__ tables;
    const psim_source* __restrict__ sources;
    int32_t guided;  // every table has its guide (else, some not monotone, the bisection runs as written)
    int32_t sub_walls;  // 3 * n_cells
    int32_t n_sources;
    int32_t n_sensors;
    int32_t full;
    int32_t phasor;
    int32_t N;  // measurement steps (validated to fit int32 at upload)
    int32_t adj;
    int32_t R;
    // Steady state: phonons whose step lies below `stop` (= adj - 1, else 0) fly across the
    // measurement boundaries below it without stopping; those boundaries only count steps.
    int32_t stop;
    double sim_time;
    double step_time;
    double t_eq;
    double r_N;  // 1 / N, rounded to nearest
};

// The emission pool, indexed by phonon id: a 64-byte record (one cache line half, four vector loads)
// and the two words that are looked at apart.  A newborn phonon has no scattering time yet (0).
struct __attribute__((aligned(16))) PoolRec {
    double2 pos, dir;  // px py, dx dy
    double2 fv;  // freq, vel
    double age;
    int32_t cell;  // -1: never starts
    int32_t sensor;
};

struct Pool {
    PoolRec* __restrict__ rec;
    uint2* __restrict__ ms;  // meta, id within the phonon's random stream (id - source id_base)
};

struct Ph {
    double px, py, dx, dy, freq, vel;
    int32_t cell, bin, pol, sign;
    int32_t step;
};

// ---- division ---------------------------------------------------------------------------
// Correctly rounded quotients by a divisor that several of them share (Markstein's method: with r
// close enough to 1 / d, one remainder step in fused arithmetic rounds n / d correctly).  A full
// division costs 11 FP64 instructions here; a quotient by a known reciprocal costs three.  For
// finite n and d away from the ends of the exponent range, which callers see to.
__device__ __forceinline__ double recip(double d) { return psim_recip(d); }
__device__ __forceinline__ double div_by(double n, double d, double r) { return psim_div_by(n, d, r); }
__device__ __forceinline__ double div_normal(double n, double d) { return PSIM_DIV(n, d); }

// Makes values arrive here: a load stays before the branches that follow, and goes out beside its
// neighbours instead of where one branch or another first needs it.
template <typename T>
__device__ __forceinline__ void pin(T& x) {
    asm volatile("" : "+v"(x));
}
template <typename T, typename... U>
__device__ __forceinline__ void pin(T& x, U&... more) {
    pin(x);
    pin(more...);
}

// ---- geometry (psim/src/geometry.cpp) ------------------------------------------------

__device__ __forceinline__ double get_slope(double x1, double y1, double x2, double y2) {  // :325-327
    return (fabs(x1 - x2) < GEOEPS) ? 0. : (y1 - y2) / (x1 - x2);
}

// crossProduct of (p2 - p1) and (p - p1), :291-300, :311-313
__device__ __forceinline__ double line_cross(double x1, double y1, double x2, double y2, double px, double py) {
    const double ax = x2 - x1, ay = y2 - y1;
    const double bx = px - x1, by = py - y1;
    return ax * by - bx * ay;
}

__device__ __forceinline__ bool on_line(double x1, double y1, double x2, double y2, double px, double py) {
    return fabs(line_cross(x1, y1, x2, y2, px, py)) < GEOEPS;
}

__host__ __device__ __forceinline__ bool rel_equals(double a, double b) {  // :108-110
    return fabs(a - b) <= ((fabs(a) < fabs(b) ? fabs(b) : fabs(a)) * GEOEPS);
}

// ---- phonon updates -------------------------------------------------------------------

// Material::freqIndex (material.cpp:64-75): a bisection over the cumulative table that keeps
// cdf[low] <= rand < cdf[high] and returns `high`.  For a non-decreasing table that is the first
// index whose value exceeds rand, clamped to [1, NBINS - 1] (bin 0 folds into bin 1, as in the
// reference).  With a guide table (guide[g] = first index whose value exceeds g / GUIDE, for
// g = 0..GUIDE) that index lies in [guide[g], guide[g + 1]] for g = floor(rand * GUIDE), which a
// short scan finds: one dependent load in place of ten.  Tables that are not non-decreasing
// have no guide and run the bisection.
template <typename T>
__device__ __forceinline__ void freq_index(const T& t, bool guided, psim_stream& st, int& bin, int& pol) {
    const auto* __restrict__ cdf = t.cdf;
    double rand, upol;  // the bisection's draw and the branch draw, one block
    psim_urand2(&st, &rand, &upol);
    int high;
    if (guided) {
        const int g = (int)(rand * (double)GUIDE);
        int i = t.guide[g];
        const int end = t.guide[g + 1];
        // the first two candidates in one round trip: a guide cell seldom spans more
        const double c0 = cdf[i < NBINS ? i : NBINS - 1], c1 = cdf[i + 1 < NBINS ? i + 1 : NBINS - 1];
        if (i < end && !(rand < c0)) {
            ++i;
            if (i < end && !(rand < c1)) {
                ++i;
                while (i < end && !(rand < cdf[i])) { ++i; }
            }
        }
        high = i < 1 ? 1 : (i > NBINS - 1 ? NBINS - 1 : i);
    } else {
        int low = 0;
        high = NBINS - 1;
        int mid = low + (high - low) / 2;
        while (high - low > 1) {
            if (rand < cdf[mid]) {
                high = mid;
            } else {
                low = mid;
            }
            mid = (low + high) / 2;
        }
    }
    bin = high;
    pol = (upol <= t.frac[high]) ? POL_LA : POL_TA;
}

// SensorController::initialUpdate / scatterUpdate with Material::getFreq, sensorController.cpp:28-55,
// material.cpp:77-80
template <typename T, typename B>
__device__ __forceinline__ void resample(const Model& m, const T& table, const B* bins, Ph& p, psim_stream& st) {
    int bin, pol;
    freq_index(table, m.guided != 0, st, bin, pol);
    const B& bn = bins[bin];
    const double f0 = bn.freq, vla = bn.vel_la, vta = bn.vel_ta, width = bn.width;
    p.freq = m.full ? f0 : f0 + (2. * psim_urand(&st) - 1.) * width / 2.;
    p.bin = bin;
    p.pol = pol;
    p.vel = (pol == POL_LA) ? vla : vta;  // material.cpp:82-84
}

__device__ __forceinline__ void set_rand_direction(Ph& p, psim_stream& st) {  // phonon.cpp:28-31
    double u1, u2;
    psim_urand2(&st, &u1, &u2);
    p.dx = 2. * u1 - 1.;
    p.dy = PSIM_SQRT(1. - p.dx * p.dx) * psim_cos2pi(u2);
}

__device__ __forceinline__ void redirect(double nx, double ny, Ph& p, psim_stream& st) {  // surface.cpp:23-30
    double rand, u2;
    psim_urand2(&st, &rand, &u2);
    const double new_dx = PSIM_SQRT(rand);
    const double new_dy = PSIM_SQRT(1. - rand) * psim_cos2pi(u2);
    p.dx = nx * new_dx - ny * new_dy;
    p.dy = ny * new_dx + nx * new_dy;
}

// Cell::handleSurfaceCollision -> CompositeSurface::handlePhonon (cell.cpp:103-108,
// compositeSurface.cpp:47-66): the first edge the point of impact lies on, its first sub-surface the
// point lies on, and what becomes of the phonon there.  Only the search and what moves the phonon
// on stand here: a reflection waits for reflect(), which a wave runs together with its
// scatters' draws and new directions.  `wall` is the index of the surface to reflect off, its
// complement where a transition sends the phonon back (no specular reflection); `sensor` follows
// the phonon into the cell it enters.
enum : int { HIT_PASSED = 0, HIT_WALL = 1, HIT_ABSORBED = 2 };

template <bool TRI>
__device__ __forceinline__ int surface_hit(const Model& m, Ph& p, int& sensor, int& wall) {
    int on = 3, begin = 0, n_sub = 0;
    if constexpr (TRI) {
        const Tri& t = m.tris[p.cell];
        const double2 v0 = t.corner[0], v1 = t.corner[1], v2 = t.corner[2];
        int32_t b0 = t.sub_begin[0], b1 = t.sub_begin[1], b2 = t.sub_begin[2];
        uint32_t info = t.info;
        const bool on0 = on_line(v0.x, v0.y, v1.x, v1.y, p.px, p.py);
        const bool on1 = on_line(v1.x, v1.y, v2.x, v2.y, p.px, p.py);
        const bool on2 = on_line(v2.x, v2.y, v0.x, v0.y, p.px, p.py);
        pin(b0, b1, b2, info);
        on = on0 ? 0 : on1 ? 1 : on2 ? 2 : 3;
        begin = on0 ? b0 : on1 ? b1 : b2;
        n_sub = (int)(info >> (TRI_SUB_BITS * on) & ((1u << TRI_SUB_BITS) - 1u));
    } else {
        #pragma unroll 1
        for (int b = 2; b >= 0; --b) {
            const Edge& e = m.edges[3 * p.cell + b];
            if (on_line(e.p1x, e.p1y, e.p2x, e.p2y, p.px, p.py)) {
                on = b;
                begin = e.sub_begin;
                n_sub = e.n_sub;
            }
        }
    }
    if (on == 3) { return HIT_PASSED; }
    wall = 3 * p.cell + on;
    for (int i = begin; i < begin + n_sub; ++i) {
        Sub s = m.subs[i];  // whole, at once
        pin(s.kind, s.target, s.target_sensor, s.same_material);
        pin(s.start, s.duration, s.max_freq_la, s.max_freq_ta);
        if (!on_line(s.p1x, s.p1y, s.p2x, s.p2y, p.px, p.py)) { continue; }
        wall = m.sub_walls + i;
        if (s.kind == 0) {  // TransitionSurface::handlePhonon, surface.cpp:71-109
            const double max_freq = (p.pol == POL_LA) ? s.max_freq_la : s.max_freq_ta;
            if (!s.same_material && p.freq > max_freq) {
                wall = ~wall;
                return HIT_WALL;
            }
            p.cell = s.target;
            sensor = s.target_sensor;
            return HIT_PASSED;
        }
        // EmitSurface::handlePhonon, surface.cpp:61-65
        const double phonon_time = (double)p.step * m.step_time;
        return phonon_time < s.start || phonon_time + m.step_time > s.start + s.duration ? HIT_WALL : HIT_ABSORBED;
    }
    return HIT_WALL;
}

// The geometric part of ModelSimulator::nextImpact (modelSimulator.cpp:87-117): the nearest edge
// crossing of the path p -> p + v * time.  On a hit the phonon is moved to the point of impact
// and the impact time is returned in out_time; the collision itself is handled separately
// (modelSimulator.cpp:118).
// Each edge runs Line::getIntersection (geometry.cpp:104-138: boxesIntersect :282-289,
// doesSegmentCrossLine :302-306 both ways, then the point) with the reference's operations and
// roundings; what depends on the path alone (its box, slope, direction, the reciprocals of its
// velocity) is computed once, and differences that only change sign are shared (negation is exact).
// The predicates of all three edges come first, without branches, so that their loads share one wait;
// the points of those crossed follow, with their slopes' loads in another.
template <bool TRI>
__device__ __forceinline__ bool find_impact(const Model& m, Ph& p, double time, double& out_time) {
    const double vx = p.dx * p.vel;
    const double vy = p.dy * p.vel;
    const double sx = p.px, sy = p.py;
    const double ex = p.px + time * vx, ey = p.py + time * vy;
    const double ddx = sx - ex, ddy = sy - ey;
    if (ddx * ddx + ddy * ddy < GEOEPS * GEOEPS) { return false; }  // pt_eq(start, end)
    const double os = (fabs(ddx) < GEOEPS) ? 0. : div_normal(ddy, ddx);  // the path's slope and intercept
    const double oi = sy - os * sx;
    const bool o_vert = rel_equals(sx, ex);
    // the path's box, drawn in by GEOEPS
    const double hix = ((ex <= sx) ? sx : ex) - GEOEPS, lox = ((ex <= sx) ? ex : sx) + GEOEPS;
    const double hiy = ((ey <= sy) ? sy : ey) - GEOEPS, loy = ((ey <= sy) ? ey : sy) + GEOEPS;
    const bool move_x = vx > VELOCITY_EPS || vx < -VELOCITY_EPS;
    const bool move_y = vy > VELOCITY_EPS || vy < -VELOCITY_EPS;
    const double rvx = recip(vx), rvy = recip(vy);  // used where move_x / move_y
    bool reach[3];
    if constexpr (TRI) {
        const Tri& t = m.tris[p.cell];
        double vx[3], vy[3], bx[3], by[3];
        bool near[3], side[3], left[3], right[3], below[3], above[3];
        #pragma unroll
        for (int k = 0; k < 3; ++k) {
            const double2 v = t.corner[k];
            vx[k] = v.x;
            vy[k] = v.y;
        }
        #pragma unroll
        for (int k = 0; k < 3; ++k) {
            bx[k] = sx - vx[k];
            by[k] = sy - vy[k];
            const double d = ddx * by[k] - bx[k] * ddy;  // the corner against the path's line
            near[k] = fabs(d) < GEOEPS;
            side[k] = d < 0.;
            left[k] = vx[k] <= hix;
            right[k] = vx[k] >= lox;
            below[k] = vy[k] <= hiy;
            above[k] = vy[k] >= loy;
        }
        #pragma unroll
        for (int b = 0; b < 3; ++b) {
            const int e = (b + 1) % 3;
            const bool box = (left[b] | left[e]) & (right[b] | right[e]) & (below[b] | below[e]) & (above[b] | above[e]);
            const double ax = vx[e] - vx[b], ay = vy[e] - vy[b];
            const double c1 = ax * by[b] - bx[b] * ay;  // path ends against the edge's line
            const double c2 = ax * (ey - vy[b]) - (ex - vx[b]) * ay;
            reach[b] = box & ((fabs(c1) < GEOEPS) | (fabs(c2) < GEOEPS) | ((c1 < 0.) != (c2 < 0.)))
                       & (near[b] | near[e] | (side[b] != side[e]));
        }
    } else {
        uint32_t set = 0;
        #pragma unroll 1
        for (int b = 0; b < 3; ++b) {
            const Edge& s = m.edges[3 * p.cell + b];
            const double p1x = s.p1x, p1y = s.p1y, p2x = s.p2x, p2y = s.p2y;
            const bool box = ((p1x <= hix) | (p2x <= hix)) & ((p1x >= lox) | (p2x >= lox)) & ((p1y <= hiy) | (p2y <= hiy))
                             & ((p1y >= loy) | (p2y >= loy));
            const double ax = p2x - p1x, ay = p2y - p1y;
            const double b1x = sx - p1x, b1y = sy - p1y, b2x = ex - p1x, b2y = ey - p1y;
            const double c1 = ax * b1y - b1x * ay, c2 = ax * b2y - b2x * ay;
            const double f2x = p2x - sx, f2y = p2y - sy;
            const double d1 = ddx * b1y - b1x * ddy, d2 = f2x * ddy - ddx * f2y;
            const bool cross = ((fabs(c1) < GEOEPS) | (fabs(c2) < GEOEPS) | ((c1 < 0.) != (c2 < 0.)))
                               & ((fabs(d1) < GEOEPS) | (fabs(d2) < GEOEPS) | ((d1 < 0.) != (d2 < 0.)));
            set |= (uint32_t)(box & cross) << b;
        }
        #pragma unroll
        for (int b = 0; b < 3; ++b) { reach[b] = (set >> b & 1u) != 0; }
    }
    if (!(reach[0] | reach[1] | reach[2])) { return false; }
    bool hit = false;
    double ix = 0., iy = 0.;
    double slope[3], icept[3];
    uint32_t vert = 0;  // a bit for each edge
    if constexpr (TRI) {
        const Tri& t = m.tris[p.cell];
        #pragma unroll
        for (int b = 0; b < 3; ++b) {
            const double2 l = t.line[b];
            slope[b] = l.x;
            icept[b] = l.y;
        }
        vert = t.info >> (3 * TRI_SUB_BITS);
    } else {
        #pragma unroll
        for (int b = 0; b < 3; ++b) {
            const Edge& s = m.edges[3 * p.cell + b];
            slope[b] = s.slope;
            icept[b] = s.intercept;
            vert |= (uint32_t)s.vert << b;
        }
    }
    pin(slope[0], slope[1], slope[2], icept[0], icept[1], icept[2]);
    pin(vert);
    #pragma unroll
    for (int b = 0; b < 3; ++b) {
        if (!reach[b]) { continue; }
        const double ss = slope[b], si = icept[b];
        const bool s_vert = (vert >> b & 1u) != 0;
        double qx, qy;
        if (o_vert && !s_vert) {  // the path vertical
            const Edge& s = m.edges[3 * p.cell + b];
            const double mm = get_slope(s.p1x, s.p1y, s.p2x, s.p2y);
            qx = sx;
            qy = mm * sx + (s.p1y - mm * s.p1x);
        } else {
            if (s_vert ? o_vert : rel_equals(ss, os)) { continue; }
            qx = s_vert ? ss : div_normal(oi - si, ss - os);
            qy = (s_vert ? os : ss) * qx + (s_vert ? oi : si);
        }
        const double gx = qx - sx, gy = qy - sy;
        if (gx * gx + gy * gy < GEOEPS * GEOEPS) { continue; }  // pt_eq(point, start)
        const double tx = move_x ? div_by(gx, vx, rvx) : time;
        const double ty = move_y ? div_by(gy, vy, rvy) : time;
        const double it = (tx <= ty) ? tx : ty;
        if (it <= time) {
            time = it;
            ix = qx;
            iy = qy;
            hit = true;
        }
    }
    if (hit) {
        p.px = ix;
        p.py = iy;
        out_time = time;
    }
    return hit;
}

// Material::relaxRates at the sensor temperature (material.cpp:54-56, 207-239) and what a scatter
// and a scattering time need of them: the shares of the total rate up to which a scatter
// resamples (a, (r0 + r1) / total) and keeps its direction (b, r0 / total), whether impurities
// scatter at all, and the time to the next scatter, SCALING_FACTOR * -log(u) / total
// (modelSimulator.cpp:124-137, 158-162).  The three quotients share their divisor.
struct Rates {
    double a, b;
    bool impurity;
};

template <bool UNI, typename S>  // S: Sensor, in global or (UNI) constant memory
__device__ __forceinline__ double relax_rates(const S& s, double freq, int pol, double& r0, double& r1, double& r2) {
    double b_l = s.b_l, t3 = s.t3, b_tn = s.b_tn, t4 = s.t4, b_tu = s.b_tu, b_i = s.b_i, w = s.w, tk = s.tk, r_tk = s.r_tk;
    if constexpr (!UNI) { pin(b_l, t3, b_tn, t4, b_tu, b_i, w, tk, r_tk); }
    if (pol == POL_LA) {
        r0 = b_l * freq * freq * t3;
        r1 = r0;
    } else {
        r0 = (freq < w) ? b_tn * freq * t4 : 0.;
        r1 = (freq >= w) ? b_tu * freq * freq / psim_sinh(div_by(HBAR * freq, tk, r_tk)) : 0.;
    }
    r2 = b_i * psim_pow4(freq);
    return 0. + r0 + r1 + r2;
}

template <bool UNI, typename S>
__device__ __forceinline__ double scatter_time(const S& s, const Ph& p, double u, Rates& r) {
    double r0, r1, r2;
    const double total = relax_rates<UNI>(s, p.freq, p.pol, r0, r1, r2);
    const double n = SCALING_FACTOR * -psim_log(u);
    r.impurity = r2 > 0.;
    if (u > 0. && total > 1e-100 && total < 1e100) {
        const double rt = recip(total);
        r.a = div_by(r0 + r1, total, rt);
        r.b = div_by(r0, total, rt);
        return div_by(n, total, rt);
    }
    r.a = (r0 + r1) / total;
    r.b = r0 / total;
    return n / total;
}

// The same where a frequency can only be a bin's and all sensors are alike (full simulations of one
// material): a block works out its bins' rates once, for both polarizations.
struct __attribute__((aligned(16))) BinRates {
    double a, b;  // b negative (-0 too) where impurities do not scatter
    double total, r_total;  // the total's reciprocal, 0 near the ends of the exponent range
};

__device__ __forceinline__ BinRates bin_rates(const Sensor& s, double freq, int pol) {
    double r0, r1, r2;
    BinRates q;
    q.total = relax_rates<false>(s, freq, pol, r0, r1, r2);
    q.a = (r0 + r1) / q.total;
    q.b = copysign(r0 / q.total, r2 > 0. ? 1. : -1.);
    q.r_total = q.total > 1e-100 && q.total < 1e100 ? recip(q.total) : 0.;
    return q;
}

__device__ __forceinline__ double scatter_time(const BinRates& q, double u, Rates& r) {
    const double n = SCALING_FACTOR * -psim_log(u);
    const double a = q.a, b = q.b, total = q.total, r_total = q.r_total;
    r.a = a;
    r.b = fabs(b);
    r.impurity = !signbit(b);
    return u > 0. && r_total != 0. ? div_by(n, total, r_total) : n / total;
}

// A new direction: Surface::redirectPhonon off a wall (surface.cpp:23-30), before its rotation to
// the wall's normal, or Phonon::setRandDirection (phonon.cpp:28-31).  Both take the next block and
// end in sqrt(..) cos(2 pi u); one pass serves lanes of either kind.
__device__ __forceinline__ void new_direction(bool off_wall, double& dx, double& dy, psim_stream& st) {
    double u1, u2;
    psim_urand2(&st, &u1, &u2);
    const double along = 2. * u1 - 1.;
    const double c = psim_cos2pi(u2);
    dy = PSIM_SQRT(1. - (off_wall ? u1 : along * along)) * c;
    dx = off_wall ? PSIM_SQRT(u1) : along;
}

}  // namespace psim_dev
