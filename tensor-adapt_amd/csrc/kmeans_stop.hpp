// kmeans_stop.hpp — the stop flag of the centroid merge's Lloyd passes.
//
// Every block of pass `it` reads the flag when it starts, and block 0 of the
// same launch may store it when its pass changes nothing.  The waves of a
// block then meet at barriers, so all of them have to come to the same
// decision whenever each reads.  The flag therefore holds the first pass that
// has nothing to do: pass `it` stores it + 1, which its own launch reads as "go
// on" just like the value before the store, and only later launches stop.
#pragma once
#include <stdint.h>

namespace ta {

constexpr int32_t kKmeansRunning = 0x7fffffff;
constexpr int32_t kmeans_stop_after(int it) { return it + 1; }
constexpr bool kmeans_stopped(int32_t flag, int it) { return flag <= it; }

}  // namespace ta
