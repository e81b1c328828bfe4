// Who may run resident decode steps, and when (resident_gate.hip).
#pragma once
#include <hip/hip_runtime_api.h>

namespace mrs {

// An engine's place at its GPU's gate, from resident_claim to resident_release.
struct ResidentSeat {
    int device = -1, workgroups = 0;   // device < 0: no claim, the engine's steps are kernel chains
    hipStream_t stream = nullptr;      // the engine's stream
    bool open = false;                 // launches that no event covers and that the host has not waited for
    bool recording = false;            // the engine captures a step for itself
    bool unseen = false;               // launches whose fault word the host has not looked at
    bool off = false;                  // a launch was called off: kernel chains until the engine is reset
    bool told = false;                 // the caller has had the error for a fault
};
bool resident_claim(ResidentSeat &seat, int device, int workgroups, hipStream_t stream);
void resident_release(ResidentSeat &seat);   // the engine has waited for its stream
void resident_idle(ResidentSeat &seat);      // the same, and goes on

// An engine's turn: made before a resident launch (or the replay of a graph that holds one) and dropped right behind it.  go()
// false: no launch now -- the step is the kernel chain, which waits for nobody.  An engine without a seat always goes.  In a
// capture only the engine's own recording goes: its replays take turns.  A caller's graph is replayed with no turn and gets the chain.
class ResidentTurn {
public:
    explicit ResidentTurn(ResidentSeat *seat);
    ~ResidentTurn();
    bool go() const { return go_; }
    ResidentTurn(const ResidentTurn &) = delete;
    ResidentTurn &operator=(const ResidentTurn &) = delete;
private:
    ResidentSeat *seat_;
    bool go_, locked_ = false;
};

// While an engine captures a step for itself.
struct ResidentRecording {
    ResidentSeat *seat;
    explicit ResidentRecording(ResidentSeat *s) : seat(s) { if (seat) seat->recording = true; }
    ~ResidentRecording() { if (seat) seat->recording = false; }
    ResidentRecording(const ResidentRecording &) = delete;
    ResidentRecording &operator=(const ResidentRecording &) = delete;
};

}  // namespace mrs
