// A sorting network for a thread's registers: K. E. Batcher, "Sorting networks and their applications" (1968), the merge of odd and even places.
// Host code as well, which the tests compile.
#ifndef GD_ORDER_H
#define GD_ORDER_H

#ifdef __HIPCC__
#define GD_ORDER_FN __host__ __device__ __attribute__((always_inline)) inline
#else
#define GD_ORDER_FN inline
#endif

// LOW .. LOW + SPAN (a power of two) of the first COUNT of `v`, STEP apart.  What lies beyond COUNT counts as larger than anything, so that no exchange
// with it is ever made.
template <int COUNT, int LOW, int SPAN, int STEP> GD_ORDER_FN void order_merge(unsigned (&v)[COUNT]) {
    auto exchange = [&](int a, int b) {
        const unsigned low = v[a] < v[b] ? v[a] : v[b], high = v[a] < v[b] ? v[b] : v[a];
        v[a] = low; v[b] = high;
    };
    if constexpr (2 * STEP < SPAN) {
        order_merge<COUNT, LOW, SPAN, 2 * STEP>(v);
        order_merge<COUNT, LOW + STEP, SPAN, 2 * STEP>(v);
#pragma unroll
        for (int at = LOW + STEP; at + STEP < LOW + SPAN; at += 2 * STEP)
            if (at + STEP < COUNT) exchange(at, at + STEP);
    } else if constexpr (LOW + STEP < COUNT) {
        exchange(LOW, LOW + STEP);
    }
}
template <int COUNT, int LOW, int SPAN> GD_ORDER_FN void order_part(unsigned (&v)[COUNT]) {
    if constexpr (SPAN > 1 && LOW + 1 < COUNT) {
        order_part<COUNT, LOW, SPAN / 2>(v);
        order_part<COUNT, LOW + SPAN / 2, SPAN / 2>(v);
        order_merge<COUNT, LOW, SPAN, 1>(v);
    }
}
// Up to 64 numbers, the smallest first.
template <int COUNT> GD_ORDER_FN void order_up(unsigned (&v)[COUNT]) {
    static_assert(COUNT <= 64, "order_up: a network for up to 64");
    order_part<COUNT, 0, COUNT <= 32 ? 32 : 64>(v);
}

#endif
