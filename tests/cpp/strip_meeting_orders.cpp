// Every order in which the touches of the word by the parts of a strip can fall (csrc/strip_meeting.h), on the host: the word
// ends at zero, every part's projection is run once (without a projection: one part goes on), and no part goes on before all
// have arrived.  Prints what it has seen; exit status 1 where something else happened.
#include <cstdio>
#include <map>
#include <set>
#include <vector>

#include "strip_meeting.h"

namespace {

struct Touch {
    bool clears;
    uint32_t value;
};

// Hands a part the answers it has had so far; the first touch behind them is thrown to the scheduler.
struct Replayed {
    const std::vector<uint32_t> *answers;
    size_t *at;
    uint32_t touch(Touch t) {
        if (*at == answers->size()) throw t;
        return (*answers)[(*at)++];
    }
    uint32_t add(uint32_t v) { return touch({false, v}); }
    void clear() { touch({true, 0}); }
    void pause() {}
};

struct Outcome {
    bool done = false;
    Touch next{};
    std::vector<int> projected;  // parts whose projection it has begun
    bool went_on = false;
};

Outcome part_until_next_touch(int part, int parts, bool projecting, int spin, const std::vector<uint32_t> &answers) {
    Outcome o;
    size_t at = 0;
    Replayed word{&answers, &at};
    try {
        const uint32_t was = word.add(et::kMeetArrived);
        const int others = et::meet_wait(word, was, part, parts, projecting, spin);
        if (others >= 0) {
            o.went_on = true;
            if (projecting) o.projected.push_back(part);
            for (int p = 0; p < parts; p++)
                if (others >> p & 1) o.projected.push_back(p);
            et::meet_through(word, parts);
        }
        o.done = true;
    } catch (const Touch &t) {
        o.next = t;
    }
    return o;
}

using State = std::pair<uint32_t, std::vector<std::vector<uint32_t>>>;

long walk(int parts, bool projecting, int spin, uint32_t &worst) {
    std::set<State> seen;
    std::vector<State> todo{{0u, std::vector<std::vector<uint32_t>>((size_t)parts)}};
    long bad = 0;
    while (!todo.empty()) {
        State s = std::move(todo.back());
        todo.pop_back();
        if (!seen.insert(s).second) continue;
        std::vector<Outcome> now;
        std::map<int, int> projected;
        bool all_done = true, all_here = true;
        int on = 0;
        for (int p = 0; p < parts; p++) {
            now.push_back(part_until_next_touch(p, parts, projecting, spin, s.second[(size_t)p]));
            all_done = all_done && now.back().done;
            all_here = all_here && !s.second[(size_t)p].empty();
            on += now.back().went_on;
            for (int q : now.back().projected) projected[q]++;
        }
        if (on && !all_here) bad++;
        if (all_done) {
            bool once = projecting ? (int)projected.size() == parts : on == 1;
            for (const auto &q : projected) once = once && q.second == 1;
            if (!once || s.first != 0) {
                bad++;
                worst = s.first;
            }
            continue;
        }
        for (int p = 0; p < parts; p++) {
            if (now[(size_t)p].done) continue;
            State next = s;
            next.second[(size_t)p].push_back(s.first);
            next.first = now[(size_t)p].next.clears ? 0u : s.first + now[(size_t)p].next.value;
            todo.push_back(std::move(next));
        }
    }
    std::printf("%d parts, %s, %d looks: %zu states, %ld wrong, last word 0x%x\n", parts, projecting ? "projecting" : "normalising", spin, seen.size(), bad, worst);
    return bad;
}

}  // namespace

int main() {
    long bad = 0;
    for (int parts = 2; parts <= 3; parts++)
        for (int projecting = 0; projecting < 2; projecting++)
            for (int spin = 0; spin <= (parts == 2 ? 3 : 2); spin++) {
                uint32_t worst = 0;
                bad += walk(parts, projecting != 0, spin, worst);
            }
    return bad != 0;
}
