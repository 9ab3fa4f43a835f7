// Walks the K loop of the persistent grouped GEMM kernel as csrc/k_schedule.hpp describes it, for two tiles in a row, and
// prints every access to an operand tile in LDS that is ordered by time only.  All waves run the same sequence and may be
// anywhere between two barriers; a wave's own loads retire in order.
//   -DPLANT_NO_BARRIER   leaves out the barrier in front of the loop
//   -DPLANT_IN_FLIGHT    lets the waits of barrier B leave one load more in flight
#include <cstdio>
#include <vector>

#include "k_schedule.hpp"

using namespace xma_rocm::k_schedule;

enum Kind { LOAD, ROW, READ, READS_BACK, WAIT, BARRIER, STAGING, NEED_ROWS };
struct Event {
    Kind kind;
    int place, piece, what; // place: half + 4 * stage; what: tile * 1000 + step (LOAD, READ), loads left in flight (WAIT)
};

static std::vector<Event> walk(int KT, bool ovl, int tile) {
    std::vector<Event> ev;
    auto load = [&](Load l, int kt) {
        if (l.piece < 0) return;
        const int step = l.ahead == NEXT_TILE ? 0 : kt + l.ahead, t = l.ahead == NEXT_TILE ? tile + 1 : tile;
        ev.push_back({LOAD, l.piece / 4 + 4 * (step & 1), l.piece, t * 1000 + step});
    };
    auto read = [&](int half, int step) { ev.push_back({READ, half + 4 * (step & 1), 0, tile * 1000 + step}); };
    auto wait = [&](int left) {
        if (left >= 0) ev.push_back({WAIT, 0, 0, left});
        ev.push_back({READS_BACK, 0, 0, 0});
    };
    auto barrier = [&] { ev.push_back({BARRIER, 0, 0, 0}); };
    ev.push_back({WAIT, 0, 0, 0});
    barrier();
    if (!ovl)
        for (int i = 0; i < ROW_LOADS; ++i) ev.push_back({ROW, 0, 0, 0});
    read(Q0, 0), read(P0, 0);
    for (int s = 0; s < 16; ++s) load(load_before_loop(s), 0);
    wait(-1);
#ifndef PLANT_NO_BARRIER
    if (BARRIER_BEFORE_LOOP) barrier();
#endif
    for (int kt = 0; kt < KT; ++kt) {
        const int mode = !ovl ? (kt == 0 ? CHECKED_FIRST : CHECKED)
                              : kt == 0 ? OVL_FIRST : kt == 1 ? OVL_SECOND : kt == KT - 1 ? OVL_LAST : kt == KT - 2 ? OVL_DRAIN : STEADY;
        if (mode == OVL_LAST) ev.push_back({NEED_ROWS, 0, 0, 0});
        for (int phase = 0; phase < 4; ++phase) {
            const bool reads = phase < 2 || reads_ahead(mode);
            for (int slot = 0; slot < 8; ++slot) { // fragments are read in slots 0 to 5, in front of the slot's load
                if (reads && slot < 6) read(read_of(phase), kt + (phase >= 2 ? 1 : 0));
                load(load_of(mode, phase, slot), kt);
                if (row_load_of(mode, phase, slot) >= 0) ev.push_back({ROW, 0, 0, 0});
            }
            if (phase == 0) wait(-1);
            if (phase == 1) {
#ifdef PLANT_IN_FLIGHT
                wait(in_flight_b(mode) + 1), barrier();
#else
                wait(in_flight_b(mode)), barrier();
#endif
            }
            if (phase == 3 && mode != OVL_LAST) wait(in_flight_a(mode)), barrier();
        }
    }
    if (!ovl) {
        wait(0), barrier();
        ev.push_back({NEED_ROWS, 0, 0, 0});
        for (int n = 0; n < 16; ++n) load({ordered(n), NEXT_TILE}, 0);
    }
    ev.push_back({STAGING, 0, 0, 0}); // the epilogue writes and reads stage 1
    ev.push_back({READS_BACK, 0, 0, 0});
    return ev;
}

static int check(const std::vector<Event> &ev, int KT, bool first, bool second) {
    int bad = 0;
    const int n = (int)ev.size();
    auto report = [&](const char *what, int i) {
        if (bad++ < 4) printf("KT=%d overlap=%d,%d: %s (event %d, place %d, step %d)\n", KT, first, second, what, i, ev[i].place, ev[i].what);
    };
    auto is_load = [&](int i) { return ev[i].kind == LOAD || ev[i].kind == ROW; };
    // first event at which load l has landed in the wave that issued it
    auto landed = [&](int l) {
        int younger = 0;
        for (int i = l + 1; i < n; ++i) {
            if (is_load(i)) ++younger;
            if (ev[i].kind == WAIT && younger >= ev[i].what) return i;
        }
        return n;
    };
    auto next_of = [&](Kind k, int i) {
        while (i < n && ev[i].kind != k) ++i;
        return i;
    };
    for (int i = 0; i < n; ++i) {
        if (ev[i].kind == LOAD || ev[i].kind == STAGING) { // overwrites: all earlier reads are over in every wave
            for (int r = 0; r < i; ++r) {
                const bool staging = ev[r].kind == STAGING || ev[i].kind == STAGING;
                const int place = ev[i].kind == STAGING ? ev[r].place : ev[i].place;
                if (!(ev[r].kind == READ && ev[r].place == place) && !(ev[r].kind == STAGING && place >= 4)) continue;
                if (staging && place < 4) continue;
                if (ev[i].kind == STAGING && ev[r].kind == STAGING) continue; // private to a wave
                if (next_of(BARRIER, next_of(READS_BACK, r)) > i) {
                    report("overwritten while another wave may still read it", i);
                    break;
                }
            }
        }
        if (ev[i].kind == LOAD || ev[i].kind == READ || ev[i].kind == STAGING) { // earlier loads into the place have landed
            int fresh = 0;
            for (int l = i - 1; l >= 0; --l) {
                if (ev[l].kind == STAGING && ev[i].kind == READ && ev[i].place >= 4) break;
                if (ev[l].kind != LOAD || (ev[i].kind == STAGING ? ev[l].place < 4 : ev[l].place != ev[i].place)) continue;
                const int land = landed(l);
                if (ev[i].kind == LOAD) {
                    if (ev[l].piece == ev[i].piece && land > i) report("loaded while an older load into the place is in flight", i);
                } else if (next_of(BARRIER, land) > i) {
                    report("used before the loads into it have landed in every wave", i);
                    break;
                } else if (ev[i].kind == READ) {
                    if (fresh < 4 && ev[l].what == ev[i].what) ++fresh;
                    else if (fresh < 4) break;
                }
            }
            if (ev[i].kind == READ && fresh < 4 && ev[i].what % 1000 < KT) report("read without four loads of this step", i);
        }
        if (ev[i].kind == NEED_ROWS) {
            for (int l = 0; l < i; ++l)
                if (ev[l].kind == ROW && landed(l) > i) report("row loads in flight where their values are needed", i);
        }
    }
    return bad;
}

int main() {
    int bad = 0, walks = 0;
    for (int KT = 1; KT <= 12; ++KT)
        for (int first = 0; first < 2; ++first)
            for (int second = 0; second < 2; ++second) {
                if ((first || second) && (KT < 4 || KT % 2)) continue;
                std::vector<Event> ev;
                for (int n = 0; n < 16; ++n) ev.push_back({LOAD, ordered(n) / 4, ordered(n), 0}); // the first tile's step 0
                for (const Event &e : walk(KT, first, 0)) ev.push_back(e);
                for (const Event &e : walk(KT, second, 1)) ev.push_back(e);
                bad += check(ev, KT, first, second);
                ++walks;
            }
    printf("%d walks, %d faults\n", walks, bad);
    return bad != 0;
}
