// mcg_box.h -- the step and the wavefront loop of scenes that are one
// axis-aligned box: the slab, the bar, the film, the bulk cell and the porous
// film (included by mcg_kernels.hip, in its anonymous namespace).
//
// The general step (flight_step / collide_step) reads everything about a
// bundle's cell from LDS, because neighbouring lanes may be in different
// cells, and tests each face against a plane record.  With one box all of
// that is the same for every lane: the bounds, the face kinds and the tally's
// geometry are wavefront-uniform (BoxCell, held in scalar registers), and a
// step reads LDS only for what an event draws (the alias table, the mode's
// mean free path and velocity) and for a diffuse face's rotation.  A specular
// or periodic face needs no random numbers, so a wavefront whose events are
// all of those kinds skips the Philox block and the direction draw.
//
// What bounds it: vector issue and, in a solve's drain, the latency of one
// bundle's chain of dependent instructions (a dependent vector instruction
// issues every 9 cycles from a lone wavefront, an independent one every 5);
// the general step spends both on what one box does not need: LDS reads of the
// cell (28 words) behind every step, address arithmetic per tally row, ~70
// spilled scalars read back lane by lane, and per-step checks for traces.
// Measured, general kernel (before it had a drain of its own) against this one
// with its drain, launch shapes and claims, a whole solve, same box: bar 1e7
// bundles FP32 5.75 -> 3.73 ms, 1e6 FP64 4.20 -> 1.99 ms, slab 1e5 FP64 725 ->
// 351 us, slab 1e4 FP32 295 -> 148 us, porous film 1e7 64 x 64 85.5 -> 66.1 ms,
// film 1e6 (12 x 6 map, bundles of thousands of steps) 21.4 -> 8.0 ms.
//
// Results: FP32 flight takes the same rounded operations on every quantity a
// trajectory depends on as the general step, and FP64 the oracle's, so
// bundles take the same events bundle for bundle; the places where an
// operation of the general step is left out (products with exact zeros and
// ones) are noted where they are.
#pragma once

// Event kinds beyond mcg_bdry_kind, and the codes of the events a flight
// finds: 4 x (2 axis + upper side) for a face, then the intrinsic event and
// the pore wall.  A code is the bit offset of the event's kind in
// BoxCell::kinds.
enum : uint32_t { kKindIntrinsic = 8, kKindPore = 9 };
enum : uint32_t { kCodeIntrinsic = 24, kCodePore = 28 };

// Walking lanes below which a walk phase of a four-row map ends (kWalkQuorum
// for fewer rows).  Four FP64 LDS adds a crossing bound such a map: the LDS
// takes 10 cycles for an add of 20 lanes and 20 for one of 64 (bank conflicts
// even out), so fuller phases pay although they leave fewer lanes to step.
// Porous film 1e7, 64 x 64, quorum 28 / 32 / 36 / 40 / 44: 68.0 / 67.2 / 65.9 /
// 65.6 / 64.7 ms; 24 mixed solves replayed 10.2 / 10.1 / 10.1 / 10.4 / 10.6 ms.
// One row at a time (a 128 x 128 map in parts) is bound by the steps: quorum
// 20 / 28 / 36 / 44: 9.6 / 9.8 / 10.2 / 11.3 ms.
constexpr int kBoxWalkQuorum4 = 36;

// Threads of a box kernel's workgroup at most (kThreads).  The FP64 kernels of
// grids hold a walk besides a bundle (and the drain its draws and a flight): two
// wavefronts a SIMD with 256 registers each run them without spills, four with
// 128 spill 50 to 100.  A lone bundle's step takes 1.21 us with two and 1.52 us
// with four (12 x 6 film), so solves whose longest bundles bound them take two:
// up to kNarrowPerLane bundles a lane of four (a batch, whose solves end
// together, kNarrowBatch).  Film 1e4 1.82 -> 1.26 ms, 1e5 4.3 -> 3.1 ms, 1e6 25.2
// -> 21.5 ms, porous film 1e5 3.04 -> 2.76 ms (1e6 the other way, 15.4 -> 16.9
// ms), 16 porous films of 3e3 in a batch 14.2 -> 10.4 ms (with grabs of 256);
// beyond, four hide each other's waits better: porous film 4e6 56 ms (two: 62),
// 1e7 127 ms (147), 16 of 5e4 in a batch 18.3 ms (19.2).  1-D tallies keep four
// throughout (bar 1e7 FP64: 7.5 ms, two 8.5).
constexpr int kNarrowThreads = 512, kNarrowPerLane = 5, kNarrowBatch = 1;
template <typename F>
bool box_narrow(int axes, double bundles, int cus, int per_lane) {
    return sizeof(F) == 8 && axes != 0 && bundles <= per_lane * 1024.0 * cus;
}


// LDS row stride of a 1-D tally and of its difference array, in doubles: a
// compile-time stride puts the rows of one column at immediate offsets of one
// address (4 addresses a step instead of 16).
constexpr int kBoxCols = 256;

// Per-face data a step reads from LDS.
template <typename F>
struct BoxFace {
    F rot[9];           // rotation taking z onto the inward normal
    F pt[3];            // periodic translation
    uint32_t spec_thr;
    uint32_t pad[3];
};

// Wavefront-uniform description of the box and its tally.
template <typename F>
struct BoxCell {
    F lo[3], hi[3];          // face positions
    F klo[3], khi[3];        // FP32: positions beyond which a bundle is lost
    F eps;                   // FP64: the kill tolerance
    uint32_t kinds;          // 4 bits per event code
    uint32_t planes;         // plane number of each face code, 4 bits each
    uint32_t maxscat, maxloop;
    uint32_t k0, k1;
    int32_t nmodes;
    int32_t counts;          // per-bundle counts are recorded
    int32_t partial;         // some wall is partially specular
    // tally: 0 none, 1 along one axis (a single cell is one axis of one
    // cell), 2 a grid walked over its divided axes
    // rowmask: the quantities tallied (bit 0 T, 1-3 the flux components);
    // rows, cols: shape of the LDS tally, from row0, col0 of the solve's map
    // of gcols columns (the whole map, or the part of it this workgroup tallies)
    int32_t tally, rowmask, rows, cols, row0, col0, gcols;
    int32_t part, parts, colparts;   // see box_part
    unsigned long long* next;        // claim counter of the part
    uint32_t comp[3][3];                   // per tally axis: mask of each position component
    int32_t last[3], stride[3];            // largest index, column stride
    F o[3], inv[3], div[3];                // cell coordinate = div (inv (p - o))
    // pore (kind of its wall, or -1)
    int32_t pore;
    F cx, cy, r2, rin2;      // axis, radius^2, (radius - tolerance)^2
    F r;
    uint32_t pore_thr;
};

// A quotient by a common divisor: the correctly rounded a / b of the IEEE
// division sequence (reciprocal estimate, two Newton steps, quotient,
// remainder correction) without its scaling steps, which leave operands of
// this size unchanged; the reciprocal is shared by all quotients.
struct Quotient {
    double b, r;
    __device__ __forceinline__ explicit Quotient(double d) : b(d) {
        double x = __builtin_amdgcn_rcp(d);
        x = __builtin_fma(x, __builtin_fma(-d, x, 1.0), x);
        r = __builtin_fma(x, __builtin_fma(-d, x, 1.0), x);
    }
    __device__ __forceinline__ double operator()(double a) const {
        const double q = a * r;
        return __builtin_fma(__builtin_fma(-b, q, a), r, q);
    }
};

template <typename F>
struct BoxLane {
    dev::V3<F> pos, dir;
    F path;                  // free path left
    F vel;                   // FP32: sign / velocity (a flight's signed time is one product); FP64: velocity
    F sg;                    // the bundle's sign
    uint32_t nscat, nbdry, nstep;
    int64_t id;
};

// Parameter along a flight, 0 to 1, of a walk.  An axis's crossings follow one
// another by a fixed step; FP64 adds up steps in fixed point, 2^-62 a unit,
// where adding them up in double puts the flight's last shares off by an ulp
// per crossing.  Largest error of a share at 64 / 160 cells, against extended
// precision: double steps 1.8e-15 / 4.4e-15, a quotient per crossing 1.3e-16 /
// 2.7e-16, fixed point 8.3e-17 / 1.3e-16.  It costs 2 to 8 % of an FP64 map's
// time (porous film 64 x 64, 1e6 bundles 17.0 -> 17.6 ms, 4e6 54.1 -> 58.4;
// film 1e6 12.2 -> 12.5 ms).
template <typename F>
struct BoxParam {
    using T = F;
    static constexpr F kOne = F(1), kNone = F(2);   // kNone: no crossing left
    __device__ static __forceinline__ double length(F to, F from) { return double(to - from); }
    static constexpr double kUnit = 1.0;            // length() of a whole flight is 1 / kUnit
};
template <>
struct BoxParam<double> {
    using T = uint64_t;
    static constexpr uint64_t kOne = 1ull << 62, kNone = ~0ull;
    static constexpr double kUnit = 0x1p-62;
    // x in [0, 1], or below for a step
    __device__ static __forceinline__ uint64_t of(double x) {
        const double s = x * 0x1p30, h = floor(s);
        return (uint64_t(uint32_t(h)) << 32) | uint32_t((s - h) * 0x1p32);
    }
    // the difference, which rounding of the steps may leave just below zero
    __device__ static __forceinline__ double length(uint64_t to, uint64_t from) {
        const uint64_t d = to - from;
        return __builtin_fma(double(int32_t(d >> 32)), 0x1p32, double(uint32_t(d)));
    }
};

// A grid walk in progress (see WalkN).  `left` counts the entries still to
// add (crossings and the last segment): the lane walks while it is positive.
template <typename F, int NA>
struct BoxWalk {
    using T = typename BoxParam<F>::T;
    T t[NA], dt[NA];         // next crossing parameter per axis and the step between crossings
    int32_t n[NA], dcol[NA];
    int32_t left;
    int32_t idx;
    T prev;
    double amt[kMaxRows];    // per unit of BoxParam::length
};
// Without a grid: the share of the last flight in its last cell, kept back (the
// next flight of the bundle starts in that cell) until the lane leaves it.
template <typename F>
struct BoxWalk<F, 0> {
    int32_t left;            // no walk: always 0
    int32_t cell;            // the cell, -1 for none
    double held[kMaxRows];
};

template <typename F>
struct BoxView {
    const uint64_t* scat;
    const F* mfp;
    const F* vel;            // FP32 in LDS: 1 / velocity; else velocity
    const BoxFace<F>* faces;
    double* tally;
};

template <typename F>
__device__ __forceinline__ dev::V3<F> unit_of(const dev::V3<F>& v) {
    if constexpr (sizeof(F) == 4) {
        // the directions normalised here have length one up to rounding, so
        // normalized()'s test for the zero vector is left out
        const F s = __builtin_amdgcn_rsqf(v.x * v.x + v.y * v.y + v.z * v.z);
        return dev::V3<F>{v.x * s, v.y * s, v.z * s};
    } else {
        const F n2 = v.x * v.x + v.y * v.y + v.z * v.z;
        const Quotient q(sqrt(n2));
        return n2 > F(0) ? dev::V3<F>{q(v.x), q(v.y), q(v.z)} : v;
    }
}

// The pore wall's normal at p, away from the axis (FP64 divides by the radius
// as the oracle does).
template <typename F>
__device__ __forceinline__ dev::V3<F> box_wall_normal(const BoxCell<F>& B, const dev::V3<F>& p) {
    if constexpr (sizeof(F) == 8) {
        const Quotient q(B.r);
        return unit_of(dev::V3<F>{q(p.x - B.cx), q(p.y - B.cy), F(0)});
    } else {
        return dev::normalized(dev::V3<F>{p.x - B.cx, p.y - B.cy, F(0)});
    }
}

// A value the compiler must keep as it is: uniform parameters would otherwise
// be read again from memory inside the step (a wait each), and what is derived
// from them (the Philox round keys) held across the loop and spilled.
// Scalar registers are short in these kernels and vector registers are not,
// so what the vector instructions of a step use as operands is kept in vector
// registers.
template <typename T>
__device__ __forceinline__ void in_vector(T& x) {
    asm volatile("" : "+v"(x));
}
template <typename T>
__device__ __forceinline__ void in_scalar(T& x) {
    asm volatile("" : "+s"(x));
}

template <typename F, int kAxes>
__device__ __forceinline__ void box_pin(BoxCell<F>& B) {
    in_scalar(B.kinds);
    in_scalar(B.maxscat);
    in_scalar(B.maxloop);
    in_scalar(B.cols);
    if constexpr (sizeof(F) == 8 && kAxes != 0) return;   // these kernels have no vector registers left
#pragma unroll
    for (int a = 0; a < 3; ++a) {
        in_vector(B.lo[a]);
        in_vector(B.hi[a]);
        if constexpr (sizeof(F) == 4) {
            in_vector(B.klo[a]);
            in_vector(B.khi[a]);
        }
    }
    if constexpr (sizeof(F) == 8) in_vector(B.eps);
#pragma unroll
    for (int q = 0; q < (kAxes == 0 ? 1 : kAxes); ++q) {
        in_vector(B.o[q]);
        in_vector(B.inv[q]);
        in_vector(B.div[q]);
        in_vector(B.last[q]);
    }
}

// floor(x) as an int (the hardware's one instruction in FP32).
__device__ __forceinline__ int cell_of(float x) {
    int i;
    asm("v_cvt_flr_i32_f32 %0, %1" : "=v"(i) : "v"(x));
    return i;
}
__device__ __forceinline__ int cell_of(double x) { return int(floor(x)); }

// The component of v a tally axis runs along: the masks are all ones for it
// and zero for the others.
__device__ __forceinline__ float pick3(const uint32_t (&m)[3], const dev::V3<float>& v) {
    return __uint_as_float((__float_as_uint(v.x) & m[0]) | (__float_as_uint(v.y) & m[1]) | (__float_as_uint(v.z) & m[2]));
}
__device__ __forceinline__ double pick3(const uint32_t (&m)[3], const dev::V3<double>& v) {
    const uint32_t lo = (uint32_t(__double2loint(v.x)) & m[0]) | (uint32_t(__double2loint(v.y)) & m[1]) |
                        (uint32_t(__double2loint(v.z)) & m[2]);
    const uint32_t hi = (uint32_t(__double2hiint(v.x)) & m[0]) | (uint32_t(__double2hiint(v.y)) & m[1]) |
                        (uint32_t(__double2hiint(v.z)) & m[2]);
    return __hiloint2double(int(hi), int(lo));
}

// One entry of a walk: the share up to the next crossing to the current cell,
// then the axis of that crossing advances.  Crossings of two axes at the same
// parameter are two entries, the first axis first, the second of zero length.
// Written without branches: after the last segment the advance changes
// nothing that is read again.
template <int kRows, typename F, int NA>
__device__ __forceinline__ void box_walk_next(BoxWalk<F, NA>& W, const BoxCell<F>& B, double* tally) {
    using P = BoxParam<F>;
    typename P::T tm = W.t[0], dt = W.dt[0];
    int32_t n = W.n[0], dcol = W.dcol[0];
    bool later[NA];   // the crossing is of axis q or a later one
    later[0] = true;
#pragma unroll
    for (int q = 1; q < NA; ++q) {
        later[q] = W.t[q] < tm;
        tm = later[q] ? W.t[q] : tm;
        dt = later[q] ? W.dt[q] : dt;
        n = later[q] ? W.n[q] : n;
        dcol = later[q] ? W.dcol[q] : dcol;
    }
    const double seg = P::length(W.left == 1 ? P::kOne : tm, W.prev);
    double* p = tally + W.idx;
    if constexpr (kRows == kMaxRows) {
#pragma unroll
        for (int j = 0; j < kMaxRows; ++j) {
            unsafeAtomicAdd(p, W.amt[j] * seg);
            p += B.cols;
        }
    } else if (uint32_t(W.idx) < uint32_t(B.cols)) {   // perhaps a range of the columns
        if constexpr (kRows == 1) {
            unsafeAtomicAdd(p, W.amt[0] * seg);
        } else {
#pragma unroll
            for (int j = 0; j < kMaxRows; ++j) {
                if (B.rowmask >> j & 1) {
                    unsafeAtomicAdd(p, W.amt[j] * seg);
                    p += B.cols;
                }
            }
        }
    }
    W.left--;
    W.prev = tm;
    W.idx += dcol;
    n--;
    const typename P::T t = n > 0 ? tm + dt : P::kNone;
#pragma unroll
    for (int q = 0; q < NA; ++q) {
        bool mine = later[q];
#pragma unroll
        for (int r = q + 1; r < NA; ++r) mine = mine && !later[r];
        W.t[q] = mine ? t : W.t[q];
        W.n[q] = mine ? n : W.n[q];
    }
}

template <int U, int kRows, typename F, int NA>
__device__ __forceinline__ void box_walk_some(BoxWalk<F, NA>& W, const BoxCell<F>& B, double* tally) {
    if (W.left > 0) {
        box_walk_next<kRows>(W, B, tally);
        if constexpr (U > 1) box_walk_some<U - 1, kRows>(W, B, tally);
    }
}

// Adds one row of a 1-D flight: the first and last cells' shares and the
// crossed interior as a range.
template <typename F>
struct Span {
    double *first, *last, *beg, *end;   // row 0's addresses: cells, range start and end in the difference array
    F fb, fe, scale;                    // shares of the end cells; FP32: 1 / cells crossed
    bool one, range;
};

template <int kRow, typename F>
__device__ __forceinline__ void add_row(const Span<F>& s, F amt, F ca) {
    unsafeAtomicAdd(s.first + kRow * kBoxCols, double(s.one ? amt : ca * s.fb));
    if (!s.one) unsafeAtomicAdd(s.last + kRow * kBoxCols, double(ca * s.fe));
    if (s.range) {
        unsafeAtomicAdd(s.beg + kRow * kBoxCols, double(ca));
        unsafeAtomicAdd(s.end + kRow * kBoxCols, -double(ca));
    }
}

// Adds what a lane holds back of its last cell.
template <int kRows, typename F>
__device__ __forceinline__ void box_release(BoxWalk<F, 0>& W, const BoxCell<F>& B, double* tally) {
    if (W.cell >= 0) {
#pragma unroll
        for (int j = 0; j < kMaxRows; ++j)
            if (kRows == kMaxRows || B.rowmask >> j & 1) unsafeAtomicAdd(tally + W.cell + j * kBoxCols, W.held[j]);
    }
#pragma unroll
    for (int j = 0; j < kMaxRows; ++j) W.held[j] = 0.0;
}

// The tally of a flight pre -> L.pos of length dmin: added at once along one
// axis, set up in W for a grid.
template <typename F, int kAxes, int kRows, bool kHold = false>
__device__ __forceinline__ void box_tally(const BoxCell<F>& B, const BoxView<F>& V, const BoxLane<F>& L,
                                          const dev::V3<F>& pre, F dmin, BoxWalk<F, kAxes>& W) {
    F dt;
    if constexpr (sizeof(F) == 4) dt = dmin * L.vel;
    else dt = L.sg * Quotient(L.vel)(dmin);
    const F dx = L.sg * (L.pos.x - pre.x), dy = L.sg * (L.pos.y - pre.y), dz = L.sg * (L.pos.z - pre.z);
    // the one row's amount
    const F only = B.rowmask & 1 ? dt : (B.rowmask & 2 ? dx : (B.rowmask & 4 ? dy : dz));
    if constexpr (kAxes == 0) {
        if (B.tally == 0) return;
        const F b = B.div[0] * (B.inv[0] * (pick3(B.comp[0], pre) - B.o[0]));
        const F e = B.div[0] * (B.inv[0] * (pick3(B.comp[0], L.pos) - B.o[0]));
        const int bb = min(max(cell_of(b), 0), B.last[0]);
        const int ee = min(max(cell_of(e), 0), B.last[0]);
        const bool up = bb < ee;
        const int lo = min(bb, ee) + 1, hi = max(bb, ee);
        if constexpr (kHold) {
            static_assert(sizeof(F) == 4, "FP32 only");
            // What bounds a 1-D FP32 solve with full wavefronts is the LDS (an
            // FP64 add of 64 lanes takes 20 cycles; 16 of them a flight, the
            // LDS active 92 % of the time outside the drain): a flight's last
            // share waits in registers for the next flight's first, and
            // flights inside one cell add nothing.  Bar 1e7 4.31 -> 3.90 ms,
            // 256 slabs 13.0 -> 12.4 ms.  FP64, whose steps are twice as
            // long, adds at once (bar 1e6 held back: 1.98 -> 1.99 ms).
            const bool one = bb == ee;
            const F fbb = F(bb), fee = F(ee);
            const F db = (up ? fbb + F(1) : fbb) - b, de = e - (up ? fee : fee + F(1));
            // a flight inside one cell: its whole amounts to that cell
            const F rad = one ? F(1) : __builtin_amdgcn_rcpf(fabsf(e - b));
            const F fb = one ? F(1) : (up ? db : -db), fe = up ? de : -de;
            const F ca[kMaxRows] = {dt * rad, dx * rad, dy * rad, dz * rad};
            if (bb != W.cell) {   // another bundle, or moved by a periodic face
                box_release<kRows>(W, B, V.tally);
                W.cell = bb;
            }
            double *const first = V.tally + bb, *const beg = V.tally + kMaxRows * kBoxCols + lo,
                           *const end = V.tally + kMaxRows * kBoxCols + hi;
#pragma unroll
            for (int j = 0; j < kMaxRows; ++j) W.held[j] += double(ca[j] * fb);
            if (!one) {
#pragma unroll
                for (int j = 0; j < kMaxRows; ++j)
                    if (kRows == kMaxRows || B.rowmask >> j & 1) unsafeAtomicAdd(first + j * kBoxCols, W.held[j]);
#pragma unroll
                for (int j = 0; j < kMaxRows; ++j) W.held[j] = double(ca[j] * fe);
                W.cell = ee;
                if (lo < hi) {
#pragma unroll
                    for (int j = 0; j < kMaxRows; ++j)
                        if (kRows == kMaxRows || B.rowmask >> j & 1) {
                            unsafeAtomicAdd(beg + j * kBoxCols, double(ca[j]));
                            unsafeAtomicAdd(end + j * kBoxCols, -double(ca[j]));
                        }
                }
            }
            return;
        }
        Span<F> s;
        s.one = bb == ee;
        s.range = lo < hi;
        s.fb = up ? F(1 + bb) - b : b - F(bb);
        s.fe = up ? e - F(ee) : F(1 + ee) - e;
        s.first = V.tally + bb;
        s.last = V.tally + ee;
        s.beg = V.tally + kMaxRows * kBoxCols + lo;
        s.end = V.tally + kMaxRows * kBoxCols + hi;
        if constexpr (sizeof(F) == 4) {
            const F rad = __builtin_amdgcn_rcpf(fabsf(e - b));
            if (kRows == kMaxRows || B.rowmask & 1) add_row<0>(s, dt, dt * rad);
            if (kRows == kMaxRows || B.rowmask & 2) {
                add_row<1>(s, dx, dx * rad);
                add_row<2>(s, dy, dy * rad);
                add_row<3>(s, dz, dz * rad);
            }
        } else {
            const Quotient q(fabs(e - b));
            if (kRows == kMaxRows || B.rowmask & 1) add_row<0>(s, dt, q(dt));
            if (kRows == kMaxRows || B.rowmask & 2) {
                add_row<1>(s, dx, q(dx));
                add_row<2>(s, dy, q(dy));
                add_row<3>(s, dz, q(dz));
            }
        }
    } else {
        int idx = 0, left = 1;
#pragma unroll
        for (int q = 0; q < kAxes; ++q) {
            const F b = B.div[q] * (B.inv[q] * (pick3(B.comp[q], pre) - B.o[q]));
            const F e = B.div[q] * (B.inv[q] * (pick3(B.comp[q], L.pos) - B.o[q]));
            const int bk = min(max(cell_of(b), 0), B.last[q]);
            const int ek = min(max(cell_of(e), 0), B.last[q]);
            const F dc = e - b;
            const bool up = bk < ek;
            idx += bk * B.stride[q];
            const F first = F(up ? bk + 1 : bk) - b;
            const int n = up ? ek - bk : bk - ek;
            bool none;
            if constexpr (sizeof(F) == 4) {
                none = (fabsf(dc) < FLT_MIN) | (n == 0);
                const F r = __builtin_amdgcn_rcpf(dc);
                W.dt[q] = fabsf(r);
                W.t[q] = none ? F(2) : first * r;
            } else {
                none = (fabs(dc) < DBL_MIN) | (n == 0);
                const Quotient d(none ? F(1) : dc);
                // the step is used from two crossings on, where it is below
                // one: 1 / |dc| and, to the fixed point's last bits, the
                // remainder of that reciprocal
                const double rest = __builtin_fma(-d.b, d.r, 1.0) * d.r * 0x1p62;
                const int64_t dt = int64_t(BoxParam<F>::of(fabs(d.r))) + int32_t(dc < F(0) ? -rest : rest);
                W.dt[q] = uint64_t(dt);
                W.t[q] = none ? BoxParam<F>::kNone : BoxParam<F>::of(d(first));
            }
            W.n[q] = none ? 0 : n;
            left += none ? 0 : n;
            W.dcol[q] = up ? B.stride[q] : -B.stride[q];
        }
        W.idx = kRows == kMaxRows ? idx : idx - B.col0;
        W.prev = 0;
        W.left = left;
        constexpr double kUnit = BoxParam<F>::kUnit;   // a power of two: exact
        W.amt[0] = kUnit * double(kRows == 1 ? only : dt);
        W.amt[1] = kUnit * double(dx);
        W.amt[2] = kUnit * double(dy);
        W.amt[3] = kUnit * double(dz);
    }
}

// The flight of a scatter-step (problem.cpp:401-416, flight_step): the face
// ahead on each axis, the pore, the free path; moves L and returns the event's
// code.  pre and dmin describe the flight; outside is the kill test.
template <typename F>
__device__ __forceinline__ uint32_t box_flight(const BoxCell<F>& B, BoxLane<F>& L, dev::V3<F>& pre, F& dmin_out,
                                               bool& outside_out) {
    const F p[3] = {L.pos.x, L.pos.y, L.pos.z}, u[3] = {L.dir.x, L.dir.y, L.dir.z};
    F dmin = L.path;
    uint32_t hit = kCodeIntrinsic;
    int plane = -1;
#pragma unroll
    for (int a = 0; a < 3; ++a) {
        const bool up = u[a] > F(0);
        const uint32_t code = up ? 8u * a + 4u : 8u * a;
        if constexpr (sizeof(F) == 4) {
            // a face that rounding left just behind is met where the bundle stands
            const F ta = ((up ? B.hi[a] : B.lo[a]) - p[a]) * __builtin_amdgcn_rcpf(u[a]);
            const F t = fmaxf(ta, F(0));
            const bool take = (u[a] != F(0)) & (t < dmin);
            dmin = take ? t : dmin;
            hit = take ? code : hit;
        } else {
            // -(c + n.p) / (n.u) of the oracle's face loop: the normal's
            // other components are zeros and its sign cancels.  Equal
            // parameters keep the lower face number.
            const F t = Quotient(u[a])((up ? B.hi[a] : B.lo[a]) - p[a]);
            const int pl = int((B.planes >> code) & 15u);
            const bool take = (u[a] != F(0)) & ((t < dmin) | ((t == dmin) & (plane >= 0) & (pl < plane)));
            dmin = take ? t : dmin;
            hit = take ? code : hit;
            plane = take ? pl : plane;
        }
    }
    if (B.pore >= 0) {
        const F dx = p[0] - B.cx, dy = p[1] - B.cy;
        const F bq = dx * u[0] + dy * u[1];
        const F aq = u[0] * u[0] + u[1] * u[1];
        const F cq = dx * dx + dy * dy - B.r2;
        const F disc = bq * bq - aq * cq;
        if ((bq < F(0)) & (disc >= F(0))) {
            // a start on (or, by rounding, just inside) the wall heading in
            // meets it at once
            const F t = cq <= F(0) ? F(0) : dev::Real<F>::div(cq, dev::Real<F>::sqrt_(disc) - bq);
            hit = t < dmin ? uint32_t(kCodePore) : hit;
            dmin = t < dmin ? t : dmin;
        }
    }
    L.path -= dmin;
    if (L.path < dev::Real<F>::kMin) L.path = F(0);
    pre = L.pos;
    dmin_out = dmin;
    L.pos = dev::V3<F>{pre.x + dmin * u[0], pre.y + dmin * u[1], pre.z + dmin * u[2]};
    L.nstep++;
    // kill test (subdomain.cpp:186-190)
    bool outside;
    if constexpr (sizeof(F) == 4) {
        outside = (L.pos.x < B.klo[0]) | (L.pos.x > B.khi[0]) | (L.pos.y < B.klo[1]) | (L.pos.y > B.khi[1]) |
                  (L.pos.z < B.klo[2]) | (L.pos.z > B.khi[2]);
    } else {
        outside = (dmin < -B.eps) | (L.pos.x - B.lo[0] < -B.eps) | (B.hi[0] - L.pos.x < -B.eps) |
                  (L.pos.y - B.lo[1] < -B.eps) | (B.hi[1] - L.pos.y < -B.eps) | (L.pos.z - B.lo[2] < -B.eps) |
                  (B.hi[2] - L.pos.z < -B.eps);
    }
    if (B.pore >= 0) {
        const F dx = L.pos.x - B.cx, dy = L.pos.y - B.cy;
        outside |= dx * dx + dy * dy < B.rin2;
    }
    outside_out = outside;
    return hit;
}

// What an event may draw: the isotropic and the Lambertian direction (about
// z), the free path and speed of a scattered mode, the word of the
// partial-specularity test.
template <typename F>
struct Draws {
    dev::V3<F> iso, lam;
    F path, vel;
    uint32_t spec;
};

template <typename F, bool kLdsTables>
__device__ __forceinline__ F box_mode_speed(const BoxView<F>& V, uint32_t mode) {
    const F vel = V.vel[mode];
    if constexpr (sizeof(F) == 8 || kLdsTables) return vel;
    else return __builtin_amdgcn_rcpf(vel);
}

template <typename F>
__device__ __forceinline__ dev::Event box_event_stream(const BoxCell<F>& B, uint32_t event, int64_t id) {
    uint32_t k0 = B.k0, k1 = B.k1;
    in_scalar(k0);
    in_scalar(k1);
    return dev::Event{k0, k1, event, uint32_t(id), uint32_t(uint64_t(id) >> 32)};
}

// All draws of one event, whatever its kind (the drain's draws ahead).
template <typename F, bool kLdsTables>
__device__ __forceinline__ Draws<F> box_draws(const BoxCell<F>& B, const BoxView<F>& V, uint32_t event, int64_t id) {
    const dev::Event ev = box_event_stream(B, event, id);
    const uint4 b0 = ev.block(0), b1 = low_block<F>(ev, 1);
    Draws<F> D;
    D.spec = b1.w;
    if constexpr (sizeof(F) == 4)
        if (B.partial) D.spec = ev.block(1).w;
    const F r = dev::Real<F>::symmetric(b0.x, b1.x);
    const F ar = r < F(0) ? -r : r;
    const F si = dev::Real<F>::sqrt_(F(1) - r * r), sl = dev::Real<F>::sqrt_(ar);
    const F q = dev::Real<F>::symmetric(b0.y, b1.y);
    F sq, cq;
    dev::Real<F>::sincos_pi(q, sq, cq);
    D.iso = dev::V3<F>{si * cq, si * sq, r};
    D.lam = dev::V3<F>{sl * cq, sl * sq, dev::Real<F>::sqrt_(F(1) - ar)};
    const uint32_t mode = dev::alias_draw(V.scat, uint32_t(B.nmodes), b0.w);
    D.path = draw_path<F>(ev, b0, b1, V.mfp[mode]);
    D.vel = box_mode_speed<F, kLdsTables>(V, mode);
    return D;
}

// The event of a scatter-step (problem.cpp:418-433, collide_step), with its
// draws given (kAhead) or made here as far as the event needs them.  Returns
// the bundle's fate, kAlive while it lives.
template <typename F, bool kLdsTables, bool kAhead>
__device__ __forceinline__ uint32_t box_event(const BoxCell<F>& B, const BoxView<F>& V, uint32_t hit, BoxLane<F>& L,
                                              const Draws<F>& ahead) {
    uint32_t kind = (B.kinds >> hit) & 15u;
    const bool intr = kind == kKindIntrinsic;
    bool pore = false;
    if (B.pore >= 0) {
        pore = kind == kKindPore;
        kind = pore ? uint32_t(B.pore) : kind;
    }
    const BoxFace<F>& P = V.faces[hit < kCodeIntrinsic ? hit >> 2 : 0u];
    const dev::Event ev = box_event_stream(B, L.nstep, L.id);
    if (B.partial) {
        if (kind == MCG_PARTIAL) {
            uint32_t w;
            if constexpr (kAhead) w = ahead.spec;
            else w = ev.block(1).w;
            kind = w < (pore ? B.pore_thr : P.spec_thr) ? uint32_t(MCG_SPEC) : uint32_t(MCG_DIFF);
        }
    }
    if (sizeof(F) == 8 || B.counts) L.nbdry += intr ? 0u : 1u;
    dev::V3<F> d = L.dir;
    if (intr | (kind == MCG_DIFF)) {
        // isotropic cos(theta) = r or Lambertian sin^2(theta) = |r| about z,
        // then turned onto the normal
        F path = F(0), vel = F(0);
        if constexpr (kAhead) {
            d = dev::V3<F>{intr ? ahead.iso.x : ahead.lam.x, intr ? ahead.iso.y : ahead.lam.y,
                           intr ? ahead.iso.z : ahead.lam.z};
            path = ahead.path;
            vel = ahead.vel;
        } else {
            const uint4 b0 = ev.block(0), b1 = low_block<F>(ev, 1);
            const F r = dev::Real<F>::symmetric(b0.x, b1.x);
            const F ar = r < F(0) ? -r : r;
            const F sinT = dev::Real<F>::sqrt_(intr ? F(1) - r * r : ar);
            const F cosT = intr ? r : dev::Real<F>::sqrt_(F(1) - ar);
            const F q = dev::Real<F>::symmetric(b0.y, b1.y);
            F sq, cq;
            dev::Real<F>::sincos_pi(q, sq, cq);
            d = dev::V3<F>{sinT * cq, sinT * sq, cosT};
            if (intr) {
                const uint32_t mode = dev::alias_draw(V.scat, uint32_t(B.nmodes), b0.w);
                const F mfp = V.mfp[mode];
                vel = box_mode_speed<F, kLdsTables>(V, mode);
                path = draw_path<F>(ev, b0, b1, mfp);
            }
        }
        L.nscat++;
        if (intr) {
            L.path = path;
            L.vel = sizeof(F) == 4 ? L.sg * vel : vel;
        } else {
            F m[9];
#pragma unroll
            for (int i = 0; i < 9; ++i) m[i] = P.rot[i];
            if (pore) rotation_to_wall(box_wall_normal(B, L.pos), m);
            d = dev::matvec(m, d);
        }
    }
    if (kind == MCG_SPEC) {
        // I - 2 n n^T of an axis: the component's sign
        const uint32_t axis = hit >> 3;
        d.x = axis == 0u ? -d.x : d.x;
        d.y = axis == 1u ? -d.y : d.y;
        d.z = axis == 2u ? -d.z : d.z;
        if (pore) {
            F m[9];
            reflection_off(box_wall_normal(B, L.pos), m);
            d = dev::matvec(m, L.dir);
        }
    }
    if (kind == MCG_PERI) {
        // the map's rotation is the identity (box_cell takes no other)
        L.pos = dev::V3<F>{L.pos.x + P.pt[0], L.pos.y + P.pt[1], L.pos.z + P.pt[2]};
    }
    L.dir = unit_of(d);
    uint32_t fate = L.nstep >= B.maxloop ? uint32_t(MCG_MAXLOOP) : kAlive;
    fate = L.nscat >= B.maxscat ? uint32_t(MCG_MAXSCAT) : fate;
    fate = kind == MCG_ISOT ? uint32_t(MCG_ABSORBED) : fate;
    return fate;
}

// One scatter-step.
template <typename F, bool kLdsTables, int kAxes, int kRows>
__device__ __forceinline__ uint32_t box_step(const BoxCell<F>& B, const BoxView<F>& V, BoxLane<F>& L,
                                             BoxWalk<F, kAxes>& W) {
    dev::V3<F> pre;
    F dmin;
    bool outside;
    const uint32_t hit = box_flight(B, L, pre, dmin, outside);
    uint32_t fate = MCG_ESCAPED;
    if (!outside) {
        box_tally<F, kAxes, kRows, sizeof(F) == 4>(B, V, L, pre, dmin, W);
        fate = box_event<F, kLdsTables, false>(B, V, hit, L, Draws<F>{});
    }
    return fate;
}

// Kernel parameters read where they are used: the pointer goes through an
// opaque move, so that the loads stay in the (rare) emission rounds instead of
// being held in scalar registers across the loop and spilled.
template <typename F>
using ParamPtr = const __attribute__((address_space(4))) KParams<F>*;

template <typename F>
__device__ __forceinline__ ParamPtr<F> params_here(ParamPtr<F> kp) {
    asm volatile("" : "+s"(kp));
    return kp;
}

// A pointer that the parameters hold, known to point to global memory (read
// from memory it would be addressed as generic).
template <typename T>
__device__ __forceinline__ T* in_global(T* p) {
    return (T*)(__attribute__((address_space(1))) T*)p;
}

// LDS layout: [scat alias | mfp | vel] (when kLdsTables), faces, tally.
template <typename F>
__host__ __device__ inline size_t box_lds_tables(int nmodes) {
    return (size_t(nmodes) * (8 + 2 * sizeof(F)) + 15) & ~size_t(15);
}

// doubles of the LDS tally: fixed strides for a 1-D tally, rows x cols for a grid
template <typename F>
__host__ __device__ inline int box_tally_doubles(const BoxCell<F>& B) {
    return B.tally == 1 ? 2 * kMaxRows * kBoxCols : (B.tally == 2 ? B.rows * B.cols : 0);
}

template <typename F, bool kLdsTables>
__device__ __forceinline__ BoxView<F> box_stage(ParamPtr<F> kp, const BoxCell<F>& B, unsigned char* lds,
                                                int tid, int nthreads) {
    const uint64_t* const g_scat = in_global(kp->scat_alias);
    const F* const g_mfp = in_global(kp->mode_mfp);
    const F* const g_vel = in_global(kp->mode_vel);
    BoxView<F> v;
    size_t off = 0;
    if constexpr (kLdsTables) {
        const int n = B.nmodes;
        uint64_t* s = reinterpret_cast<uint64_t*>(lds);
        F* m = reinterpret_cast<F*>(lds + 8 * size_t(n));
        F* q = m + n;
        for (int i = tid; i < n; i += nthreads) {
            s[i] = g_scat[i];
            m[i] = g_mfp[i];
            const F vel = g_vel[i];
            if constexpr (sizeof(F) == 4) q[i] = __builtin_amdgcn_rcpf(vel);
            else q[i] = vel;
        }
        v.scat = s;
        v.mfp = m;
        v.vel = q;
        off = box_lds_tables<F>(n);
    } else {
        v.scat = g_scat;
        v.mfp = g_mfp;
        v.vel = g_vel;
    }
    BoxFace<F>* f = reinterpret_cast<BoxFace<F>*>(lds + off);
    if (tid < 6) {
        const DevPlane<F>& P = in_global(kp->planes)[(B.planes >> (4 * tid)) & 15u];
        for (int i = 0; i < 9; ++i) f[tid].rot[i] = P.rot[i];
        for (int i = 0; i < 3; ++i) f[tid].pt[i] = P.pt[i];
        f[tid].spec_thr = P.spec_thr;
    }
    v.faces = f;
    v.tally = reinterpret_cast<double*>(lds + off + 6 * sizeof(BoxFace<F>));
    const int nt = box_tally_doubles(B);
    for (int i = tid; i < nt; i += nthreads) v.tally[i] = 0.0;
    return v;
}

// Adds a workgroup's LDS tally into the solve's global tally (after a barrier).
template <typename F>
__device__ __forceinline__ void box_flush(ParamPtr<F> kp, const BoxCell<F>& B, const double* tally, int tid,
                                          int nthreads) {
    double* const direct = in_global(kp->direct);
    double* const diff = in_global(kp->diff);
    if (B.tally == 1) {
        const int r0 = B.rowmask & 1 ? 0 : 1;   // LDS row j is the quantity j
        for (int i = tid; i < B.rows * kBoxCols; i += nthreads) {
            const int r = i / kBoxCols, c = i % kBoxCols;
            const double a = tally[(r0 + r) * kBoxCols + c], d = tally[(kMaxRows + r0 + r) * kBoxCols + c];
            if (a != 0.0 && c < B.cols) unsafeAtomicAdd(direct + r * B.cols + c, a);
            if (d != 0.0 && c <= B.cols) unsafeAtomicAdd(diff + r * (B.cols + 1) + c, d);
        }
    } else if (B.tally == 2) {
        for (int r = 0; r < B.rows; ++r)
            for (int c = tid; c < B.cols; c += nthreads) {
                const double a = tally[r * B.cols + c];
                if (a != 0.0) unsafeAtomicAdd(direct + size_t(B.row0 + r) * B.gcols + B.col0 + c, a);
            }
    }
}

// Emission into a box lane (emit of the general path).
template <typename F, bool kLdsTables>
__device__ __forceinline__ void box_emit(ParamPtr<F> kp, const BoxCell<F>& B, const BoxView<F>& V, int64_t n,
                                         BoxLane<F>& L) {
    KParams<F> K;
    K.emitters = in_global(kp->emitters);
    K.emit_cdf = in_global(kp->emit_cdf);
    K.sdoms = in_global(kp->sdoms);
    K.pores = in_global(kp->pores);
    K.nemitter = kp->nemitter;
    K.npore = kp->npore;
    K.nmodes = B.nmodes;
    K.k0 = kp->k0;
    K.k1 = kp->k1;
    Lane<F> T;
    emit<F>(K, in_global(kp->flux_alias), V.mfp, n, T);
    L.pos = T.pos;
    L.dir = T.dir;
    L.path = T.scat_next;
    L.sg = F(T.sign);
    if constexpr (sizeof(F) == 8) L.vel = V.vel[T.mode];
    else if constexpr (kLdsTables) L.vel = L.sg * V.vel[T.mode];
    else L.vel = L.sg * __builtin_amdgcn_rcpf(V.vel[T.mode]);
    L.nscat = L.nbdry = L.nstep = 0;
    L.id = n;
}

// Lane l's value of x as lane addr / 4 of the wavefront holds it (all lanes
// take part).
__device__ __forceinline__ int lane_pull(int addr, int x) { return __builtin_amdgcn_ds_bpermute(addr, x); }
__device__ __forceinline__ uint32_t lane_pull(int addr, uint32_t x) { return uint32_t(lane_pull(addr, int(x))); }
__device__ __forceinline__ float lane_pull(int addr, float x) {
    return __int_as_float(lane_pull(addr, __float_as_int(x)));
}
__device__ __forceinline__ int64_t lane_pull(int addr, int64_t x) {
    const uint32_t lo = lane_pull(addr, uint32_t(uint64_t(x))), hi = lane_pull(addr, uint32_t(uint64_t(x) >> 32));
    return int64_t(uint64_t(lo) | (uint64_t(hi) << 32));
}
__device__ __forceinline__ double lane_pull(int addr, double x) {
    return __hiloint2double(lane_pull(addr, __double2hiint(x)), lane_pull(addr, __double2loint(x)));
}
template <typename F>
__device__ __forceinline__ dev::V3<F> lane_pull(int addr, const dev::V3<F>& v) {
    return dev::V3<F>{lane_pull(addr, v.x), lane_pull(addr, v.y), lane_pull(addr, v.z)};
}

struct BoxStats {   // wavefront-uniform
    unsigned long long steps = 0, ended = 0, absorbed = 0, escaped = 0;
};

// Books the lanes whose bundle ended (fate not kAlive); all lanes call.
template <typename F>
__device__ __forceinline__ void box_end(const BoxCell<F>& B, ParamPtr<F> kp, const BoxLane<F>& L, uint32_t fate,
                                        bool& active, BoxStats& st) {
    const uint64_t ended = __ballot(fate != kAlive);
    if (ended == 0ull) return;
    st.ended += popc(ended);
    st.absorbed += popc(__ballot(fate == MCG_ABSORBED));
    st.escaped += popc(__ballot(fate == MCG_ESCAPED));
    if (fate != kAlive) {
        active = false;
        if (B.counts && B.part == 0) {
            const ParamPtr<F> k = params_here<F>(kp);
            const int64_t i = L.id - k->first;
            in_global(k->c_nscat)[i] = L.nscat;
            in_global(k->c_nbdry)[i] = L.nbdry;
            in_global(k->c_nstep)[i] = L.nstep;
            in_global(k->c_fate)[i] = fate;
        }
    }
}

// The drain of a wavefront: its last bundles, at most kDrainLanes, with no id
// left to claim.  What bounds it is the chain of a step's instructions, one
// bundle each, while most lanes are idle; so the idle lanes take over what does
// not depend on the bundle's path.  The bundles sit in the first `span` lanes
// (a power of two) and step together;
//  - the draws of a bundle's next 64 / span events (they depend on the id and
//    the event's number alone) are made by 64 / span lanes at once, and a step
//    fetches its event's;
//  - a flight's tally is left to a lane of its own, and the 64 lanes' flights
//    are tallied (and their grid walks walked) together once all hold one.
// A step is then its flight and its event's turn.
// A lone bundle's step, before and now (us, FP32 / FP64): slab 1.19 / 2.08 and
// 0.78 / 1.02, film (12 x 6 map) 1.87 / 2.87 and 0.81 / 1.52, porous film
// (64 x 64) 2.92 / 3.77 and 0.92 / 1.72; bar 1e6 FP64 3.24 -> 2.01 ms, film 1e6
// 12.5 -> 7.75 ms.  8, 16 or 32 lanes: bar FP64 2.11 / 2.01 / 1.96 ms, film
// 7.84 / 7.75 / 7.70 ms, 256 slabs 13.05 / 12.99 / 13.08 ms.
#ifndef MCG_DRAIN_LANES
#define MCG_DRAIN_LANES 16
#endif
constexpr int kDrainLanes = MCG_DRAIN_LANES;

template <typename F, bool kLdsTables, int kAxes, int kRows>
__device__ __forceinline__ void box_drain(const BoxCell<F>& B, ParamPtr<F> kp, const BoxView<F>& V, int lane,
                                          uint64_t lt_mask, BoxLane<F>& L, bool active, BoxStats& st) {
    int span = 2 * kDrainLanes, shift = 0;   // lanes the bundles sit in; log2 of the draws ahead per bundle
    int at = 0, ahead = 0;                   // next event among the draws ahead, how many there are
    int slot = 0;                            // lanes holding a flight to tally
    Draws<F> D;
    dev::V3<F> fpre, fpos;                   // this lane's flight to tally
    F fdmin = F(0), fvel = F(0);
    bool pending = false;
    for (;;) {
        const uint64_t live = __ballot(active);
        if (live == 0ull || slot + span > kWave) {
            // the flights held are tallied together
            BoxWalk<F, kAxes> W;
            W.left = 0;
            if (pending) {
                BoxLane<F> T;
                T.pos = fpos;
                T.sg = fvel < F(0) ? F(-1) : F(1);
                T.vel = sizeof(F) == 4 ? fvel : fabs(fvel);
                box_tally<F, kAxes, kRows>(B, V, T, fpre, fdmin, W);
            }
            if constexpr (kAxes != 0)
                while (__ballot(W.left > 0) != 0ull) box_walk_some<kWalkUnroll, kRows>(W, B, V.tally);
            pending = false;
            slot = 0;
        }
        if (live == 0ull) return;
        const int n = popc(live);
        if (2 * n <= span) {
            // the live bundles into the first lanes, in order
            const int to = active ? popc(live & lt_mask) : n + popc(~live & lt_mask);
            const int from = 4 * __builtin_amdgcn_ds_permute(4 * to, lane);
            L.pos = lane_pull(from, L.pos);
            L.dir = lane_pull(from, L.dir);
            L.path = lane_pull(from, L.path);
            L.vel = lane_pull(from, L.vel);
            L.sg = lane_pull(from, L.sg);
            L.nscat = lane_pull(from, L.nscat);
            L.nbdry = lane_pull(from, L.nbdry);
            L.nstep = lane_pull(from, L.nstep);
            L.id = lane_pull(from, L.id);
            active = lane < n;
            span = 1;
            shift = 6;
            while (span < n) {
                span *= 2;
                --shift;
            }
            ahead = at = 0;
        }
        if (at == ahead) {
            // lane l draws event number l % (64 / span) ahead of bundle l / (64 / span)
            const int of = 4 * (lane >> shift);
            const int64_t id = lane_pull(of, L.id);
            const uint32_t event = lane_pull(of, L.nstep) + 1u + uint32_t(lane & ((1 << shift) - 1));
            D = box_draws<F, kLdsTables>(B, V, event, id);
            at = 0;
            ahead = 1 << shift;
        }
        // (pulled by every lane: a lane that is switched off passes nothing on)
        Draws<F> E;
        const int src = 4 * (((lane << shift) + at) & (kWave - 1));
        E.iso = lane_pull(src, D.iso);
        E.lam = lane_pull(src, D.lam);
        E.path = lane_pull(src, D.path);
        E.vel = lane_pull(src, D.vel);
        E.spec = B.partial ? lane_pull(src, D.spec) : 0u;
        ++at;
        dev::V3<F> pre = L.pos;
        F dmin = F(0);
        bool outside = true;
        uint32_t hit = kCodeIntrinsic;
        if (active) hit = box_flight(B, L, pre, dmin, outside);
        st.steps += n;
        // flights to lanes slot .. slot + span - 1
        const bool flown = active && !outside;
        const uint64_t flights = __ballot(flown);
        const int give = lane - slot;
        const int giver = 4 * (give & (kWave - 1));
        const dev::V3<F> gpre = lane_pull(giver, pre), gpos = lane_pull(giver, L.pos);
        const F gdmin = lane_pull(giver, dmin), gvel = lane_pull(giver, sizeof(F) == 4 ? L.vel : L.sg * L.vel);
        if (uint32_t(give) < uint32_t(span) && (flights >> (give & (kWave - 1)) & 1ull)) {
            fpre = gpre;
            fpos = gpos;
            fdmin = gdmin;
            fvel = gvel;
            pending = true;
        }
        slot += span;
        uint32_t fate = kAlive;
        if (flown) fate = box_event<F, kLdsTables, true>(B, V, hit, L, E);
        else if (active) fate = MCG_ESCAPED;
        box_end(B, kp, L, fate, active, st);
    }
}

// A wavefront's loop over the bundles it claims (trajectory_kernel's loop).
// The refill is looked at only when some lane has run out of work since the
// last look: a wavefront left with a few long-lived bundles goes from step to
// step without it.
template <typename F, bool kLdsTables, int kAxes, int kRows>
__device__ __forceinline__ void box_run(const BoxCell<F>& B, ParamPtr<F> kp, const BoxView<F>& V, int lane) {
    const uint64_t lt_mask = (lane == 0) ? 0ull : (~0ull >> (kWave - lane));
    int64_t pool_base = 0, pool_lim = 0, seen = 0;
    bool active = false, full = false, drained = false;
    BoxLane<F> L, N;
    BoxWalk<F, kAxes> W;
    W.left = 0;
    if constexpr (kAxes == 0) {
        W.cell = -1;
        for (int j = 0; j < kMaxRows; ++j) W.held[j] = 0.0;
    }
    BoxStats st;
    uint64_t busy = ~0ull, last_busy = 0ull;
    for (;;) {
        if (busy != last_busy || busy == 0ull) {
            const bool walking = W.left > 0;
            const ParamPtr<F> k = params_here<F>(kp);
            const int64_t count = k->count;
            unsigned long long* const next = in_global(B.next);
            if constexpr (sizeof(F) == 4) {
                if (!active && !walking && full) {
                    L = N;
                    full = false;
                    active = true;
                }
                const bool near_end = count - seen < k->tail;
                const bool empty = !full && !drained && (!near_end || (!active && !walking));
                const uint64_t me = __ballot(empty);
                if (me != 0ull && (popc(me) >= kSlotQuorum || popc(__ballot(empty && !active && !walking)) >= kEmitQuorum ||
                                   __ballot(active || walking) == 0ull)) {
                    const int64_t mine = claim(empty, lane, lt_mask, pool_base, pool_lim, next, k->chunk, count,
                                               k->guide, k->tail, seen);
                    if (empty) {
                        if (mine < count) {
                            box_emit<F, kLdsTables>(k, B, V, k->first + mine, N);
                            full = true;
                        } else {
                            drained = true;
                        }
                    }
                    if (!active && !walking && full) {
                        L = N;
                        full = false;
                        active = true;
                    }
                }
                if (__ballot(active || walking || full || !drained) == 0ull) break;
            } else {
                const bool need = !active && !drained && !walking;
                if (emit_now<kEmitQuorumFp64>(need, active || walking)) {
                    const int64_t mine = claim(need, lane, lt_mask, pool_base, pool_lim, next, k->chunk, count,
                                               k->guide, 0, seen);
                    if (need) {
                        if (mine < count) {
                            box_emit<F, kLdsTables>(k, B, V, k->first + mine, L);
                            active = true;
                        } else {
                            drained = true;
                        }
                    }
                }
                if (__ballot(active || walking) == 0ull) break;
            }
            last_busy = __ballot(active || walking);
            // no id left (one lane found none) and few bundles: the drain
            if (__ballot(drained) != 0ull && __ballot(full) == 0ull && popc(__ballot(active)) <= kDrainLanes) {
                if constexpr (kAxes != 0) {
                    while (__ballot(W.left > 0) != 0ull) box_walk_some<kWalkUnroll, kRows>(W, B, V.tally);
                } else if constexpr (sizeof(F) == 4) {
                    box_release<kRows>(W, B, V.tally);
                    W.cell = -1;
                }
                box_drain<F, kLdsTables, kAxes, kRows>(B, kp, V, lane, lt_mask, L, active, st);
                break;
            }
        }
        const bool go = active && !(W.left > 0);
        st.steps += popc(__ballot(go));
        uint32_t fate = kAlive;
        if (go) fate = box_step<F, kLdsTables, kAxes, kRows>(B, V, L, W);
        box_end(B, kp, L, fate, active, st);
        if constexpr (kAxes != 0) {
            // the walk phase (walk_phase): while kWalkQuorum lanes walk or no
            // other lane has a step to take
            for (;;) {
                const uint64_t m = __ballot(W.left > 0);
                if (m == 0ull || (popc(m) < (kRows == kMaxRows ? kBoxWalkQuorum4 : kWalkQuorum) && __ballot(active && !(W.left > 0)) != 0ull)) break;
                box_walk_some<kWalkUnroll, kRows>(W, B, V.tally);
            }
        }
        busy = __ballot(active || W.left > 0);
    }
    if constexpr (kAxes == 0 && sizeof(F) == 4) box_release<kRows>(W, B, V.tally);
    if (lane == 0 && st.ended != 0 && B.part == 0) {
        unsigned long long* const c = in_global(params_here<F>(kp)->counters);
        atomicAdd(c + C_STEPS, st.steps);
        atomicAdd(c + C_ESC, st.escaped);
        atomicAdd(c + C_ABS, st.absorbed);
        atomicAdd(c + C_TRUNC, st.ended - st.absorbed - st.escaped);
        atomicAdd(c + C_BUNDLES, st.ended);
    }
}

// A map larger than the LDS is tallied in parts (rows of it, or column ranges
// of a row), each by its own workgroups, which run all of the solve's bundles
// and add only to their part: workgroup w takes part w % parts.  The bundles'
// counts and statistics are those of part 0.
//
// Why: adding in global memory is bound by the rate of FP64 atomics past the
// LDS, 1.1e10 a second for the whole GPU, four per cell a flight crosses, so a
// 128 x 128 map ran at 2e8 scatter-steps a second; running the bundles once per
// part and adding in LDS costs parts / (parts running at once) more steps.
// Porous film, 2e5 bundles, 128 x 128 Multi map (4 parts): 153 -> 6.0 ms.
template <typename F>
__host__ __device__ inline void box_part(BoxCell<F>& B, uint32_t w) {
    if (B.parts == 1) return;
    B.part = int32_t(w % uint32_t(B.parts));
    const int32_t r = B.part / B.colparts, c = B.part % B.colparts;
    if (B.colparts > 1) {   // one row, a range of its columns
        B.row0 = r;
        B.col0 = c * B.cols;
        B.cols = B.cols < B.gcols - B.col0 ? B.cols : B.gcols - B.col0;
    } else {
        B.row0 = r * B.rows;
    }
    // the quantities of rows [row0, row0 + rows) among those tallied
    int32_t mask = 0, row = 0;
    for (int j = 0; j < kMaxRows; ++j) {
        if (!(B.rowmask >> j & 1)) continue;
        if (row >= B.row0 && row < B.row0 + B.rows) mask |= 1 << j;
        ++row;
    }
    B.rows = B.rows < row - B.row0 ? B.rows : row - B.row0;
    B.rowmask = mask;
}

// A solve of a one-box scene (the kernel parameters come first: params_here
// reads them through the kernel-argument segment).
template <typename F, bool kLdsTables, int kAxes, int kRows, int kThreads = 1024>
__global__ void __launch_bounds__(kThreads) box_kernel(KParams<F> Karg, BoxCell<F> Barg) {
    extern __shared__ __align__(16) unsigned char lds[];
    const int tid = threadIdx.x;
    const ParamPtr<F> kp = (ParamPtr<F>)__builtin_amdgcn_kernarg_segment_ptr();
    BoxCell<F> B = Barg;
    if constexpr (kAxes != 0) box_part(B, blockIdx.x);
    B.next = B.part == 0 ? kp->next : kp->part_next + (B.part - 1);
    B.k0 = kp->k0;
    B.k1 = kp->k1;
    box_pin<F, kAxes>(B);
    const BoxView<F> V = box_stage<F, kLdsTables>(params_here<F>(kp), B, lds, tid, blockDim.x);
    __syncthreads();
    box_run<F, kLdsTables, kAxes, kRows>(B, kp, V, tid & (kWave - 1));
    __syncthreads();
    box_flush(params_here<F>(kp), B, V.tally, tid, blockDim.x);
}

// ------------------------------------------------------------------ batches
// Many one-box solves in one persistent launch.  A workgroup stages a solve,
// runs the bundles it claims until none are left, adds its LDS tally to the
// solve's and takes the next solve.  Each visit costs the staging and a drain
// (the last bundles' remaining steps, during which lanes idle), so a workgroup
// should make few visits and those where most work is left:
//  - it starts at the solve its share of the estimated work lies in
//    (BoxSolve::work_before), so solves begin with workgroups in proportion,
//    and goes on to those that begin in its share, so small solves are visited
//    once each;
//  - then it takes the solve with the most estimated work left per workgroup
//    already on it, and leaves a solve to the workgroups on it when what is
//    left is no more than one bundle per lane of theirs.  A solve is taken by
//    an atomic count of its visitors: workgroups that look at the same moment
//    do not all go to the same one.
// Every solve is finished: one with unclaimed bundles and no visitor is always
// taken (the first to count itself as a visitor stays), and a visitor leaves
// only when nothing is unclaimed (a stale read of a counter can only add a
// visit that finds nothing).
// Every solve visited in turn by the general step, before, and this: 256 slabs
// 17.7 -> 12.1 ms a call, 24 mixed solves replayed 19.9 -> 10.3 ms, same box.
// Many small solves, every one visited in turn / picked without shares and
// takes / this (ms): 4000 slabs of 200 FP32 38.6 / 20.5 / 0.57, FP64 3.9 / 34.7 /
// 1.5; 512 of 1e3 FP64 0.94 / 1.28 / 0.38.
template <typename F>
struct BoxSolve {
    KParams<F> K;                  // first: box_run reads it through ParamPtr
    BoxCell<F> B;
    uint32_t* visitors;            // workgroups on the solve
    double work_before, work;      // estimated work of the solves before this one, and of one bundle
    int32_t tables, pad;           // sampling tables staged in LDS
};

template <typename F, bool kLdsTables, int kAxes, int kRows>
__device__ __forceinline__ void box_visit(const BoxCell<F>& cell, ParamPtr<F> kp, unsigned char* lds, int tid,
                                          int nthreads) {
    BoxCell<F> B = cell;
    box_pin<F, kAxes>(B);
    const BoxView<F> V = box_stage<F, kLdsTables>(params_here<F>(kp), B, lds, tid, nthreads);
    __syncthreads();
    box_run<F, kLdsTables, kAxes, kRows>(B, kp, V, tid & (kWave - 1));
    __syncthreads();
    box_flush(params_here<F>(kp), B, V.tally, tid, nthreads);
    __syncthreads();
}

// The solve with the most estimated work left per workgroup on it, -1 when no
// solve needs another workgroup (uniform over the workgroup; LDS is free).
template <typename F>
__device__ int box_pick(const BoxSolve<F>* solves, int n, unsigned char* lds, int tid, int nthreads) {
    unsigned long long* const key = reinterpret_cast<unsigned long long*>(lds);
    if (tid == 0) *key = 0ull;
    __syncthreads();
    unsigned long long best = 0ull;
    for (int i = tid; i < n; i += nthreads) {
        const BoxSolve<F>& s = solves[i];
        const int64_t left =
            s.K.count - int64_t(__hip_atomic_load(s.B.next, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
        if (left <= 0) continue;
        const uint32_t v = __hip_atomic_load(s.visitors, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if (v != 0 && left <= int64_t(v) * nthreads) continue;
        // spread workgroups that look at the same moment
        const uint32_t mix = (blockIdx.x * 2654435761u + uint32_t(i) * 40503u) >> 24;
        const float score = float(double(left) * s.work) / float(v + 1) * (1.0f + float(mix) * (1.0f / 512.0f));
        const unsigned long long k = (uint64_t(__float_as_uint(fmaxf(score, FLT_MIN))) << 32) | uint32_t(i);
        best = k > best ? k : best;
    }
    if (best != 0ull) atomicMax(key, best);
    __syncthreads();
    best = *key;
    __syncthreads();
    return best == 0ull ? -1 : int(uint32_t(best));
}

// The last solve whose work begins at or before the middle of workgroup w's
// share of the whole.
template <typename F>
__device__ __forceinline__ int box_share(const BoxSolve<F>* solves, int n, unsigned w) {
    const double total = solves[n - 1].work_before + solves[n - 1].work * double(solves[n - 1].K.count);
    const double at = total * ((double(w) + 0.5) / double(gridDim.x));
    int lo = 0, hi = n - 1;
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (solves[mid].work_before <= at) lo = mid;
        else hi = mid - 1;
    }
    return lo;
}

// Counts this workgroup as a visitor of the solve if it needs one more (uniform
// over the workgroup; LDS is free).
template <typename F>
__device__ bool box_take(const BoxSolve<F>& s, unsigned char* lds, int tid, int nthreads) {
    int* const taken = reinterpret_cast<int*>(lds);
    if (tid == 0) {
        uint32_t* const visitors = in_global(s.visitors);
        const int64_t left =
            s.K.count - int64_t(__hip_atomic_load(in_global(s.B.next), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
        bool ok = left > 0;
        if (ok) {
            const uint32_t v = atomicAdd(visitors, 1u);
            ok = v == 0 || left > int64_t(v) * nthreads;
            if (!ok) atomicSub(visitors, 1u);
        }
        *taken = ok ? 1 : 0;
    }
    __syncthreads();
    const bool ok = *taken != 0;
    __syncthreads();
    return ok;
}

// kAxes: axes of the grids among the solves (0 when all tallies are 1-D).
template <typename F, int kAxes, int kThreads = 1024>
__global__ void __launch_bounds__(kThreads) box_batch_kernel(const BoxSolve<F>* solves, int n) {
    extern __shared__ __align__(16) unsigned char lds[];
    const int tid = threadIdx.x, nthreads = blockDim.x;
    // this workgroup's share of the solves: from the last one whose work begins
    // at or before the middle of its share of the work, to the next workgroup's
    const int first = blockIdx.x == 0 ? 0 : box_share(solves, n, blockIdx.x);
    int last = -1;   // looked up when it is needed: a search of global memory
    if (tid == 0) atomicAdd(in_global(solves[first].visitors), 1u);
    for (int si = first, own = first; si >= 0;) {
        const auto* sv = (const __attribute__((address_space(4))) BoxSolve<F>*)(solves + __builtin_amdgcn_readfirstlane(si));
        const ParamPtr<F> kp = (ParamPtr<F>)sv;
        BoxCell<F> B = *(const BoxCell<F>*)&sv->B;
        B.k0 = kp->k0;
        B.k1 = kp->k1;
        if (kAxes == 0 || B.tally != 2) {
            if (B.rowmask == 15) box_visit<F, true, 0, kMaxRows>(B, kp, lds, tid, nthreads);
            else box_visit<F, true, 0, 0>(B, kp, lds, tid, nthreads);
        } else if constexpr (kAxes != 0) {
            if (sv->tables) {
                if (B.rowmask == 15) box_visit<F, true, kAxes, kMaxRows>(B, kp, lds, tid, nthreads);
                else box_visit<F, true, kAxes, 0>(B, kp, lds, tid, nthreads);
            } else {
                if (B.rowmask == 15) box_visit<F, false, kAxes, kMaxRows>(B, kp, lds, tid, nthreads);
                else box_visit<F, false, kAxes, 0>(B, kp, lds, tid, nthreads);
            }
        }
        if (tid == 0) atomicSub(in_global(sv->visitors), 1u);
        // the next solve: of this workgroup's share, then the one most in need
        si = -1;
        if (last < 0) last = blockIdx.x + 1 == gridDim.x ? n : box_share(solves, n, blockIdx.x + 1);
        while (si < 0 && own + 1 < last) {
            ++own;
            if (box_take(solves[own], lds, tid, nthreads)) si = own;
        }
        while (si < 0) {
            const int pick = box_pick(solves, n, lds, tid, nthreads);
            if (pick < 0) break;
            if (box_take(solves[pick], lds, tid, nthreads)) si = pick;
        }
    }
}
