// lanes.h — which search lanes run side by side (host code, no HIP).
#pragma once

namespace jhq {

// use[0 .. result): the lanes of `lanes` that have a hardware queue of their own,
// lane 0 first; 0 if a measurement failed.  span(ls, m, brief, &ms) runs one
// probe kernel on each of the m lanes ls at once and gives the time from the
// first's start to the last's end: about one kernel's time if no two of the lanes
// share a queue, about twice that if some do.  A host that stalls while it
// enqueues lengthens a span, which is short (270 us; with 24 busy processes on 16
// cores, one index of 60 lost a lane by it), so a kernel's own time and the refusal
// of a lane take two runs that agree.
template <class Span>
int pick_lanes(int lanes, int* use, Span span) {
    // the shortest of up to 4 runs, until one is below `enough` or two agree
    auto settled = [&](const int* ls, int m, float enough, float* ms) {
        float t = 0.f;
        for (int run = 0; run < 4; run++) {
            if (!span(ls, m, false, &t)) return false;
            const float hi = run && *ms > t ? *ms : t, lo = run && *ms < t ? *ms : t;
            const bool done = t < enough || (run && hi - lo <= 0.1f * lo);
            *ms = lo;
            if (done) break;
        }
        return true;
    };
    float t1 = 0.f, t = 0.f;
    // (a lane's first launch is slower, and the very first loads the kernel)
    for (int l = 0; l < lanes; l++)
        if (!span(&l, 1, true, &t)) return 0;
    use[0] = 0;
    if (!settled(use, 1, 0.f, &t1) || !(t1 > 0.f)) return 0;
    int n = 1;
    for (int j = 1; j < lanes; j++) {
        use[n] = j;
        if (!settled(use, n + 1, 1.5f * t1, &t)) return 0;
        if (t < 1.5f * t1) n++;
    }
    return n;
}

}  // namespace jhq
