// What the tiled samplers stage of a window's rows, replayed on the host under
// AddressSanitizer and UndefinedBehaviorSanitizer: tables in the list's order,
// with pixels taken out, with buckets moved and with buckets shared.  A row
// that row_span accepts stages positions of the list only and holds every one
// of its buckets; a row that is no run of the list is not accepted.
#include <algorithm>
#include <cstdio>
#include <random>
#include <vector>

#include "epcq_common.h"
#include "epcq_sampler.h"

int main() {
    std::mt19937 rng(7);
    auto below = [&](int n) { return (int)(rng() % (unsigned)n); };
    int bad = 0, runs = 0, others = 0;
    for (int round = 0; round < 4000; ++round) {
        const int W = 1 + below(40), kind = round % 4;
        std::vector<int> count(W);
        for (int& c : count) c = below(3) ? below(9) : 0;
        std::vector<int2> table(W, make_int2(-1, -1));
        std::vector<int> place(W);
        for (int i = 0; i < W; ++i) place[i] = i;
        if (kind == 2) std::shuffle(place.begin(), place.end(), rng);
        int n = 0;
        for (int i : place) {
            if (count[i]) table[i] = make_int2(n, count[i]);
            n += count[i];
        }
        if (kind == 1)
            for (int2& e : table)
                if (below(3) == 0) e = make_int2(-1, -1);
        if (kind == 3)
            for (int i = 0; i < 3; ++i) table[below(W)] = table[below(W)];
        std::vector<int> list(n, 1);
        const int c0 = below(W), cols = 1 + below(W - c0);
        int lo, hi, end = -1;
        bool ordered = true;
        for (int c = c0; c < c0 + cols; ++c) {
            if (table[c].y <= 0) continue;
            ordered = ordered && table[c].x >= end;
            end = table[c].x + table[c].y;
        }
        const bool run = epcq::row_span(table.data() + c0, cols, lo, hi);
        bad += run != ordered;
        if (!run) {
            ++others;
            continue;
        }
        ++runs;
        std::vector<int> staged;
        for (int j = lo; j < hi; ++j) staged.push_back(list.at(j));
        for (int c = c0; c < c0 + cols; ++c)
            for (int j = 0; j < table[c].y; ++j) bad += staged.at(table[c].x - lo + j) != 1;
    }
    std::printf("row spans: %d runs, %d others, %s\n", runs, others, bad || runs < 1000 || others < 300 ? "FAILED" : "ok");
    return bad || runs < 1000 || others < 300;
}
