// Engines come, go, step, are waited for and are captured in a random order; whenever one launches, the launches of the others that
// the runtime does not order before it must fit on the chip beside it.  Prints "ok <launches in turns> <refused turns>" or the fault.
// With the argument "claim": whether one engine gets the route, which it then holds until its input ends.
#include "resident_gate.hip"
#include <memory>
#include <random>

using namespace mrs;

namespace {
struct Engine {
    ResidentSeat seat;
    ModelStream stream;
    int workgroups = 0;
    long last = 0;        // number of its last launch on its stream, 0: none that the host has not waited for
    bool turns = false, own_capture = false;
};

const char *launch(Engine &e, std::vector<std::unique_ptr<Engine>> &all, int live, long &ordered, long &refused) {
    Model &m = model();
    m.acting = &e.stream;
    const ResidentTurn turn(e.turns ? &e.seat : nullptr);
    if (!turn.go()) { refused += !e.stream.capturing; return nullptr; }
    if (e.turns && e.stream.capturing && !e.own_capture) return "a launch in a caller's capture";
    if (!e.turns || e.stream.capturing) return nullptr;   // a kernel chain, or nothing that runs now
    auto &own = e.stream.before;
    if ((int)own.size() <= e.stream.id) own.resize(e.stream.id + 1, 0);
    int together = e.workgroups;
    for (auto &o : all)
        if (o.get() != &e && o->last && ((int)own.size() <= o->stream.id || own[o->stream.id] < o->last)) together += o->workgroups;
    if (together > m.places) return "launches that do not fit together are not ordered";
    ordered += live > m.places;
    e.last = ++own[e.stream.id];
    return nullptr;
}
// The host waits for an engine's stream: what comes before its end there is over, whoever launched it.
void host_wait(Engine &e, std::vector<std::unique_ptr<Engine>> &all) {
    auto &own = e.stream.before;
    for (auto &o : all)
        if ((int)own.size() > o->stream.id && o->last <= own[o->stream.id]) o->last = 0;
    e.last = 0;
}
}  // namespace

int main(int argc, char **argv) {
    if (!strcmp(argv[1], "claim")) {
        ResidentSeat seat;
        ModelStream stream{0};
        printf("%d\n", resident_claim(seat, 0, 64, &stream));
        fflush(stdout);
        while (getchar() != EOF) {}
        return 0;
    }
    std::mt19937 rng((unsigned)atoi(argv[1]));
    Model &m = model();
    m.fail_every = argc > 2 ? atoi(argv[2]) : 0;
    std::vector<std::unique_ptr<Engine>> all;
    std::vector<std::unique_ptr<Engine>> gone;   // streams keep their numbers
    int ids = 0;
    long ordered = 0, refused = 0;
    for (int n = 0; n < 20000; n++) {
        int live = 0;
        for (auto &e : all) live += e->turns ? e->workgroups : 0;
        const int what = (int)(rng() % 100);
        if (all.empty() || (what < 4 && all.size() < 5)) {
            auto e = std::make_unique<Engine>();
            e->stream.id = ids++;
            const int sizes[] = {4, 64, 128, 256, 257};
            e->workgroups = sizes[rng() % 5];
            e->turns = resident_claim(e->seat, 0, e->workgroups, &e->stream);
            if (e->turns != (e->workgroups <= m.places)) return printf("claim of %d workgroups: %d\n", e->workgroups, e->turns), 1;
            all.push_back(std::move(e));
            continue;
        }
        const size_t at = rng() % all.size();
        Engine &e = *all[at];
        if (what < 7) {
            e.stream.capturing = false;
            host_wait(e, all);
            resident_release(e.seat);
            gone.push_back(std::move(all[at]));
            all.erase(all.begin() + at);
        } else if (what < 15) {
            e.stream.capturing = !e.stream.capturing;
            e.own_capture = e.seat.recording = e.stream.capturing && rng() % 2;
        } else if (what < 30) {
            if (e.stream.capturing) continue;   // (a captured stream cannot be waited for)
            host_wait(e, all);
            resident_idle(e.seat);
        } else if (const char *fault = launch(e, all, live, ordered, refused)) {
            return printf("operation %d: %s\n", n, fault), 1;
        }
        if (m.joined) return printf("operation %d: a capturing stream was joined\n", n), 1;
        if (m.touched) return printf("operation %d: another engine's stream was touched\n", n), 1;
    }
    printf("ok %ld %ld\n", ordered, refused);
    return 0;
}
