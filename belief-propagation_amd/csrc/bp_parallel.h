/*
 * bp_parallel.h -- host threads for the passes over a graph's padded arrays
 * (bp_parallel.cpp).
 */
#pragma once

#include <algorithm>
#include <cstddef>
#include <functional>

/* Calls f(i) for i < parts on the calling thread and up to 15 others, which
 * wait for further calls for a second and then end.  Calls from several
 * threads share them.  f must not throw. */
void bp_parallel(unsigned parts, const std::function<void(unsigned)> &f);

/* f(begin, end) over [0, n) in parts of at least `grain`. */
template <typename F> static void par_for(size_t n, size_t grain, F f)
{
    const unsigned parts = (unsigned)std::min<size_t>(16, n / std::max<size_t>(grain, 1));
    if (parts < 2) {
        f((size_t)0, n);
        return;
    }
    bp_parallel(parts, [&](unsigned i) { f(n * i / parts, n * (i + 1) / parts); });
}
