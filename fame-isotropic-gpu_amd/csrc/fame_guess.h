/*
 * fame_guess.h -- how many iterations the next CG solve is expected to take.
 *
 * A solve's launches are queued for the expected count before the host first asks
 * how it went.  One too many costs three launches that return at once (10 us), one
 * too few a round trip (40 us), so the counts are kept per tolerance and iteration
 * limit: a refinement to 1e-16 in between must not be what the next solve to
 * 1e-12 expects.  Two pairs at a time, the less recent one gives way.
 */
#pragma once
#include <algorithm>

struct CgGuess {
    struct Entry {
        double tol = 0.0;
        int maxit = 0, predict = 0, last = 0;     /* 0: not known */
        unsigned used = 0;
    };
    Entry e[2];
    unsigned clock = 0;

    Entry& at(double tol, int maxit) {
        Entry* old = &e[0];
        for (Entry& x : e) {
            if (x.used && x.tol == tol && x.maxit == maxit) { x.used = ++clock; return x; }
            if (x.used < old->used) old = &x;
        }
        *old = Entry();
        old->tol = tol; old->maxit = maxit; old->used = ++clock;
        return *old;
    }
    /* counts that go up and down by one: the larger.  A solve in which no problem
     * iterated (right-hand sides below the tolerance) says nothing of the next    */
    static void took(Entry& x, int its) {
        if (its < 1) return;
        x.predict = std::max(its, std::min(x.last, its + 1));
        x.last = its;
    }
};
