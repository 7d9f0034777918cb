// Division-free walks of strided views as rows, shared by the full
// reductions and the map-reductions.  A view (RowsView, built on the host)
// is `rows` rows of `cols` elements under up to three outer dimensions;
// threads walk it in units -- 16-byte vectors of 4 elements when rows are
// contiguous, single elements otherwise -- tracking two linear forms over
// the row digits: `off`, the element offset of the walked operand, and
// `off2`, a second form (a logical index, or a second operand's offset).
#pragma once

#include "hx_device.hpp"
#include "hx_internal.hpp"

namespace hx {

// Unit u of a row sits at element u * ustride (form 1) and u * ustride2
// (form 2).  The walker's step of `step` units is split on the host into
// whole rows (as outer digits, innermost first, with their offsets
// step_off / step_off2) and leftover units (step_units, step_uoff /
// step_uoff2), so a step is adds and compares only.  ospan[k] =
// oshape[k] * ostride[k], and the same for form 2.
struct RowsGeom {
    uint64_t rows, cols, units;
    int64_t ustride, units_span, cstride2, ustride2, units_span2;
    uint32_t orank;
    uint64_t oshape[3];
    int64_t ostride[3], ospan[3], ostride2[3], ospan2[3];
    uint64_t step_units, step_rows;
    uint64_t step_digits[3];
    int64_t step_uoff, step_off, step_uoff2, step_off2;
};

// Walks a thread's units of a RowsGeom view: unit `item` is unit
// item % units of row item / units.  Divisions only at the start; each
// advance adds the precomputed step with carries.  `off` and `off2` are
// the two forms at the walker's unit.
struct RowWalker {
    uint64_t unit;
    uint64_t dig[3]; // outer digits of the row, innermost first (the outermost unwrapped)
    int64_t off, off2;
    __device__ __forceinline__ void init(const RowsGeom &g, int64_t base, int64_t base2, uint64_t item) {
        const uint64_t row = item / g.units;
        unit = item - row * g.units;
        off = base + (int64_t)unit * g.ustride;
        off2 = base2 + (int64_t)unit * g.ustride2;
        uint64_t r = row;
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            if ((uint32_t)k + 1 < g.orank) {
                const uint64_t q = r / g.oshape[k];
                dig[k] = r - q * g.oshape[k];
                r = q;
            } else {
                dig[k] = r;
                r = 0;
            }
            if ((uint32_t)k < g.orank) {
                off += (int64_t)dig[k] * g.ostride[k];
                off2 += (int64_t)dig[k] * g.ostride2[k];
            }
        }
    }
    __device__ __forceinline__ void advance(const RowsGeom &g) {
        unit += g.step_units;
        off += g.step_uoff + g.step_off;
        off2 += g.step_uoff2 + g.step_off2;
        uint64_t carry = 0;
        if (unit >= g.units) {
            unit -= g.units;
            off -= g.units_span;
            off2 -= g.units_span2;
            carry = 1;
        }
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            if ((uint32_t)k < g.orank) {
                dig[k] += g.step_digits[k] + carry;
                if (carry) {
                    off += g.ostride[k];
                    off2 += g.ostride2[k];
                }
                carry = 0;
                if ((uint32_t)k + 1 < g.orank && dig[k] >= g.oshape[k]) {
                    dig[k] -= g.oshape[k];
                    off -= g.ospan[k];
                    off2 -= g.ospan2[k];
                    carry = 1;
                }
            }
        }
    }
};

// The walker geometry of a row view: units per row (vectors of 4 elements
// or single elements) and a step of `step` units as whole rows, outer
// digits of those rows (innermost first; the outermost unwrapped) and
// leftover units.
inline RowsGeom rows_geom(const RowsView &v, bool vec, uint64_t step) {
    RowsGeom g{};
    g.rows = v.rows;
    g.cols = v.cols;
    g.units = vec ? ceil_div(v.cols, 4) : v.cols;
    g.ustride = vec ? 4 : v.cstride;
    g.units_span = (int64_t)g.units * g.ustride;
    g.cstride2 = v.cstride2;
    g.ustride2 = vec ? 4 * v.cstride2 : v.cstride2;
    g.units_span2 = (int64_t)g.units * g.ustride2;
    g.orank = v.orank;
    for (int k = 0; k < 3; ++k) {
        g.oshape[k] = v.oshape[k];
        g.ostride[k] = v.ostride[k];
        g.ospan[k] = (int64_t)v.oshape[k] * v.ostride[k];
        g.ostride2[k] = v.ostride2[k];
        g.ospan2[k] = (int64_t)v.oshape[k] * v.ostride2[k];
    }
    g.step_units = step % g.units;
    g.step_rows = step / g.units;
    g.step_uoff = (int64_t)g.step_units * g.ustride;
    g.step_uoff2 = (int64_t)g.step_units * g.ustride2;
    uint64_t r = g.step_rows;
    for (uint32_t k = 0; k < 3; ++k) {
        if (k + 1 < g.orank) {
            g.step_digits[k] = r % g.oshape[k];
            r /= g.oshape[k];
        } else if (k + 1 == g.orank) {
            g.step_digits[k] = r;
            r = 0;
        } else {
            g.step_digits[k] = 0;
        }
        if (k < g.orank) {
            g.step_off += (int64_t)g.step_digits[k] * g.ostride[k];
            g.step_off2 += (int64_t)g.step_digits[k] * g.ostride2[k];
        }
    }
    return g;
}

// Matrices: views of `rows` rows of `cols` contiguous elements, one distance
// apart (slices, sub-blocks, padded rows).  Here a step is one compare and a
// few adds -- the rows need no digits -- and a thread keeps one walker, whose W
// next units' loads go out together.  The general walker's 64-bit digits
// cost more vector instructions per 16-byte unit than the reductions
// themselves.  f32, us, general walker -> this one, sum / dot / L2 norm /
// argmax: the 4094 x 4094 inside of a 4096-wide matrix 18.2 / 34.2 / 25.3 /
// 23.4 -> 14.8 / 25.5 / 15.0 / 16.7 (4.5 to 5.3 TB/s); 832191 rows of 71 of 79
// 53.5 / 98.6 / 72.6 / 72.4 -> 42.9 / 81.6 / 42.9 / 45.1 (5.5 to 6.4 TB/s of the
// lines touched); 114 rows of 674 6.4 / 5.8 / 5.6 / 9.3 -> 4.2 / 3.9 / 3.9 / 5.5.
// Two units in flight: 18.8 / 27.4 / 18.9 / 16.6 for the first; eight 14.5 /
// 25.9 / 14.8 / 16.3, but 2 to 5% slower beyond 256 MB.  It wins down to rows of
// one vector and a tail: 2^24 elements in rows of 5 / 9 / 17 / 33, one element
// apart, sum 27.0 / 24.6 / 23.5 / 21.6 -> 16.5 / 15.6 / 15.1 / 13.9, dot of rows of
// 5 46.4 -> 28.9.
//
// A row's last unit, when cols is no multiple of 4, is the vector that ends
// at the row's end: its first `shift` elements belong to the unit before and
// are masked.  So every load is a whole vector inside its row, and no lane
// branches around one.
struct MatrixWalk {
    uint64_t items;          // rows * units
    uint32_t units;          // 16-byte units per row
    uint32_t tail;           // shift of a row's last unit, 0 to 3
    uint64_t trips;          // trips of W units that every thread takes in full
    int64_t row_a, row_b;    // distance between rows of a (and b)
    int64_t step_a, wrap_a;  // offset of one step, and of a step that passes the row's end beyond it
    int64_t step_b, wrap_b;
    uint32_t step_units;
    uint32_t cols, step_i, wrap_i; // the same for the row-major index (mod 2^32)
};

// `nthreads` threads, W units a trip.
inline MatrixWalk matrix_walk(const RowsView &v, uint64_t nthreads, uint32_t W) {
    MatrixWalk m{};
    m.units = (uint32_t)ceil_div(v.cols, 4);
    m.tail = (uint32_t)((4 - v.cols % 4) % 4);
    m.items = v.rows * m.units;
    m.trips = m.items / (nthreads * W);
    m.row_a = v.ostride[0];
    m.row_b = v.ostride2[0];
    const uint64_t rows = nthreads / m.units;
    m.step_units = (uint32_t)(nthreads % m.units);
    m.step_a = (int64_t)rows * m.row_a + 4 * (int64_t)m.step_units;
    m.step_b = (int64_t)rows * m.row_b + 4 * (int64_t)m.step_units;
    m.wrap_a = m.row_a - 4 * (int64_t)m.units;
    m.wrap_b = m.row_b - 4 * (int64_t)m.units;
    m.cols = (uint32_t)v.cols;
    m.step_i = (uint32_t)(rows * v.cols + 4 * (uint64_t)m.step_units);
    m.wrap_i = (uint32_t)(v.cols - 4 * (uint64_t)m.units);
    return m;
}
// Rows of contiguous elements under one outer dimension, at least one vector
// long.
inline bool is_matrix_walk(const RowsView &v) {
    return v.orank == 1 && v.cstride == 1 && v.cols >= 4 && v.cols <= 0xFFFFFFF0ull;
}

// Calls visit(x, y, shift, index) for thread `tid`'s units: x (and y, with
// TWO) the unit's vectors of a and b, elements below `shift` (4: all) to be
// left out, `index` the row-major index of x's first element.
template <typename T, int W, bool TWO, typename Visit>
__device__ __forceinline__ void walk_matrix(const MatrixWalk &g, const T *a, const T *b, uint64_t tid,
                                            uint64_t nthreads, Visit &&visit) {
    using V = typename Vec4A4<T>::type;
    uint64_t row;
    uint32_t unit;
    if (g.items <= 0xFFFFFFFFull) {
        const uint32_t r = (uint32_t)tid / g.units; // tid < items, or nothing is read
        unit = (uint32_t)tid - r * g.units;
        row = r;
    } else {
        row = tid / g.units;
        unit = (uint32_t)(tid - row * g.units);
    }
    int64_t oa = (int64_t)row * g.row_a + 4 * (int64_t)unit;
    int64_t ob = TWO ? (int64_t)row * g.row_b + 4 * (int64_t)unit : 0;
    uint32_t index = (uint32_t)row * g.cols + 4 * unit;
    auto step = [&]() {
        unit += g.step_units;
        oa += g.step_a;
        if constexpr (TWO) ob += g.step_b;
        index += g.step_i;
        if (unit >= g.units) {
            unit -= g.units;
            oa += g.wrap_a;
            if constexpr (TWO) ob += g.wrap_b;
            index += g.wrap_i;
        }
    };
    V x[W], y[W];
    uint32_t shift[W], first[W];
    for (uint64_t t = 0; t < g.trips; ++t) {
#pragma unroll
        for (int k = 0; k < W; ++k) {
            shift[k] = unit + 1 == g.units ? g.tail : 0u;
            first[k] = index - shift[k];
            x[k] = load_a4<true>((const V *)(a + (oa - shift[k])));
            if constexpr (TWO) y[k] = load_a4<true>((const V *)(b + (ob - shift[k])));
            step();
        }
#pragma unroll
        for (int k = 0; k < W; ++k) visit(x[k], TWO ? y[k] : x[k], shift[k], first[k]);
    }
    // The rest: units past the end read the view's first vector.
    uint64_t j = tid + g.trips * W * nthreads;
    if (j >= g.items) return;
#pragma unroll
    for (int k = 0; k < W; ++k) {
        const bool live = j < g.items;
        shift[k] = !live ? 4u : unit + 1 == g.units ? g.tail : 0u;
        first[k] = index - shift[k];
        x[k] = load_a4<true>((const V *)(a + (live ? oa - shift[k] : 0)));
        if constexpr (TWO) y[k] = load_a4<true>((const V *)(b + (live ? ob - shift[k] : 0)));
        step();
        j += nthreads;
    }
#pragma unroll
    for (int k = 0; k < W; ++k) visit(x[k], TWO ? y[k] : x[k], shift[k], first[k]);
}

} // namespace hx
