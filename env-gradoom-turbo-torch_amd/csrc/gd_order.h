// A sorting network for a thread's registers: K. E. Batcher, "Sorting networks and their applications" (1968), the merge of odd and even places; and the walk
// over what it ordered.  Host code as well, which the tests compile.
#ifndef GD_ORDER_H
#define GD_ORDER_H

#ifdef __HIPCC__
#define GD_ORDER_FN __device__ __attribute__((always_inline)) inline
#else
#define GD_ORDER_FN inline
#endif

// two numbers in order
GD_ORDER_FN void order_two(double &low, double &high) {
    const double a = low, b = high;
#ifdef __HIPCC__
    asm("v_min_f64 %0, %1, %2" : "=v"(low) : "v"(a), "v"(b));      // plain minima of numbers that are none of them NaN: fmin() would ask first
    asm("v_max_f64 %0, %1, %2" : "=v"(high) : "v"(a), "v"(b));
#else
    low = a < b ? a : b; high = a < b ? b : a;
#endif
}
// LOW .. LOW + SPAN (a power of two) of `v`, STEP apart
template <int LOW, int SPAN, int STEP, int COUNT> GD_ORDER_FN void order_merge(double (&v)[COUNT]) {
    if constexpr (2 * STEP < SPAN) {
        order_merge<LOW, SPAN, 2 * STEP>(v);
        order_merge<LOW + STEP, SPAN, 2 * STEP>(v);
#pragma unroll
        for (int at = LOW + STEP; at + STEP < LOW + SPAN; at += 2 * STEP) order_two(v[at], v[at + STEP]);
    } else {
        order_two(v[LOW], v[LOW + STEP]);
    }
}
template <int LOW, int SPAN, int COUNT> GD_ORDER_FN void order_part(double (&v)[COUNT]) {
    if constexpr (SPAN > 1) {
        order_part<LOW, SPAN / 2>(v);
        order_part<LOW + SPAN / 2, SPAN / 2>(v);
        order_merge<LOW, SPAN, 1>(v);
    }
}
// Numbers, a power of two of them, the smallest first.
template <int COUNT> GD_ORDER_FN void order_up(double (&v)[COUNT]) {
    static_assert((COUNT & (COUNT - 1)) == 0, "order_up: a power of two");
    order_part<0, COUNT>(v);
}
// The smallest of two ordered runs, as many as each holds, in order, in `v`: the pairs from opposite ends hold them and rise, then fall.
template <int COUNT> GD_ORDER_FN void order_merge_lowest(double (&v)[COUNT], const double (&other)[COUNT]) {
#pragma unroll
    for (int k = 0; k < COUNT; ++k) {
        double most = other[COUNT - 1 - k];
        order_two(v[k], most);
    }
#pragma unroll
    for (int step = COUNT / 2; step > 0; step /= 2)
#pragma unroll
        for (int k = 0; k < COUNT; ++k)
            if (!(k & step)) order_two(v[k], v[k + step]);
}

// Rows `from` .. `held` of an ordered window, some at a time, until the last of them is farther than enough(): true if it came to that, so that what lies beyond
// the window is farther still.  row(k) gives a row, which has a distance; look() is asked about every one and told whether it is there.  Rows from `held` on are
// read with the last ones and hold anything: they neither end a walk nor keep it from ending.  ADVANCE: `from` moves past those leading ones that are no
// farther than `passed`.
#define WINDOW_WALK_ROWS 4
template <bool ADVANCE, typename Row, typename Look, typename Enough>
GD_ORDER_FN bool window_walk(int &from, int held, float passed, Row row, Look look, Enough enough) {
    bool leading = true, more = true;
    for (int k = from; k < held && more; k += WINDOW_WALK_ROWS) {
        decltype(row(0)) rows[WINDOW_WALK_ROWS];
#pragma unroll
        for (int j = 0; j < WINDOW_WALK_ROWS; ++j) rows[j] = row(k + j);
        float last = rows[0].dist;
#pragma unroll
        for (int j = 0; j < WINDOW_WALK_ROWS; ++j) {
            const bool there = k + j < held;
            if (ADVANCE) { leading = leading && there && !(rows[j].dist > passed); from += leading ? 1 : 0; }
            last = there ? rows[j].dist : last;
            look(rows[j], there);
        }
        more = !(last > enough());
    }
    return !more;
}

#endif
