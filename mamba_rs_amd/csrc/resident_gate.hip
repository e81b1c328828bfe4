// Who may run resident decode steps (the four kernels that include resident.hpp), and when.
//
// A resident launch's workgroups wait for each other, so they must all get a place on the GPU.  One launch alone always does (an
// engine takes the route only while its workgroups are at most as many as the compute units, one each); two launches that hold
// half of the places each would wait until they give up.  So
//   * one process per GPU has the route: the first to ask binds an abstract socket named after the GPU's PCI address, which the
//     system takes back when the process ends, whatever way it ends; another process's engines keep the kernel chains (of those that
//     share a network namespace: two containers on one GPU do not see each other, and launches that meet there are called off);
//   * an engine whose kernels may not use all compute units -- a mask on its stream or in the environment -- keeps the chains;
//   * inside the process, while the live engines' launches do not all fit together, they go one after the other: every launch is
//     followed by an event on its own stream, and the next engine's launch waits for it (on the GPU).  An engine touches no
//     stream but its own: another one's may be in a capture, which an event recorded from here would join.
//   * launches from before there were that many engines carry no event.  Until the host has waited for them, or their engine has
//     launched again, the other engines' steps are kernel chains;
//   * a step that a caller captures on an engine's stream is the kernel chain: the caller's replays take no turns.
// An engine's own steps, on its one stream, follow each other anyway, and ordinary kernels on other streams end by themselves.
#include "resident_gate.hpp"
#include <errno.h>
#include <mutex>
#include <stddef.h>
#include <stdint.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>
#include <sys/socket.h>
#include <sys/un.h>
#include <unistd.h>
#include <vector>

namespace mrs {
namespace {

constexpr int kMaxDevices = 64;
struct Gate {
    std::mutex m;
    bool asked = false, ours = false;
    int places = 0, live = 0;             // compute units; workgroups of the live engines' launches
    std::vector<ResidentSeat *> seats;
    const ResidentSeat *last = nullptr;   // whose launch `event` was recorded behind
    hipEvent_t event = nullptr;
};
Gate g_gates[kMaxDevices];

bool bind_gpu(int device) {
    char bus[64] = {0};
    if (hipDeviceGetPCIBusId(bus, (int)sizeof bus - 1, device) != hipSuccess) return false;
    const int fd = socket(AF_UNIX, SOCK_DGRAM | SOCK_CLOEXEC, 0);
    if (fd < 0) return false;
    sockaddr_un a;
    memset(&a, 0, sizeof a);
    a.sun_family = AF_UNIX;
    const int n = snprintf(a.sun_path + 1, sizeof a.sun_path - 1, "mamba_hip.resident.%s", bus);   // (a leading zero byte: no file)
    if (bind(fd, reinterpret_cast<sockaddr *>(&a), (socklen_t)(offsetof(sockaddr_un, sun_path) + 1 + n)) != 0) {
        close(fd);
        return false;
    }
    return true;   // held until the process ends
}

// Whether kernels on a stream may use all `units` compute units.
bool whole_gpu(hipStream_t stream, int units) {
    const char *e = getenv("HSA_CU_MASK");   // (applied below HIP, which does not report it)
    if (e && *e) return false;
    uint32_t mask[32] = {0};   // (1024 units)
    if (hipExtStreamGetCUMask(stream, 32, mask) != hipSuccess) {
        (void)hipGetLastError();
        return false;
    }
    int may = 0;
    for (uint32_t m : mask) may += __builtin_popcount(m);
    return may >= units;
}

}  // namespace

bool resident_claim(ResidentSeat &seat, int device, int workgroups, hipStream_t stream) {
    if (device < 0 || device >= kMaxDevices) return false;
    Gate &g = g_gates[device];
    std::lock_guard<std::mutex> lock(g.m);
    if (!g.asked) {
        g.asked = true;
        g.ours = hipDeviceGetAttribute(&g.places, hipDeviceAttributeMultiprocessorCount, device) == hipSuccess &&
                 hipEventCreateWithFlags(&g.event, hipEventDisableTiming) == hipSuccess && bind_gpu(device);
    }
    if (!g.ours || workgroups > g.places || !whole_gpu(stream, g.places)) return false;
    try { g.seats.push_back(&seat); } catch (...) { return false; }
    seat.device = device; seat.workgroups = workgroups; seat.stream = stream; seat.open = seat.unseen = seat.off = seat.told = false;
    g.live += workgroups;
    return true;
}

void resident_release(ResidentSeat &seat) {
    if (seat.device < 0) return;
    Gate &g = g_gates[seat.device];
    std::lock_guard<std::mutex> lock(g.m);
    g.live -= seat.workgroups;
    for (size_t i = 0; i < g.seats.size(); i++)
        if (g.seats[i] == &seat) { g.seats.erase(g.seats.begin() + i); break; }
    if (g.last == &seat) g.last = nullptr;   // (its work is done)
    seat.device = -1;
}

void resident_idle(ResidentSeat &seat) {
    if (seat.device < 0) return;
    std::lock_guard<std::mutex> lock(g_gates[seat.device].m);
    seat.open = false;
}

ResidentTurn::ResidentTurn(ResidentSeat *seat) : seat_(seat), go_(true) {
    if (!seat || seat->device < 0) return;
    hipStreamCaptureStatus cap = hipStreamCaptureStatusNone;
    if (hipStreamIsCapturing(seat->stream, &cap) != hipSuccess) { go_ = false; return; }
    if (cap != hipStreamCaptureStatusNone) { go_ = seat->recording; return; }   // recorded, not run
    if (seat->off) { go_ = false; return; }
    Gate &g = g_gates[seat->device];
    g.m.lock();
    if (g.live > g.places) {
        for (const ResidentSeat *s : g.seats)
            if (s != seat && s->open) go_ = false;
        if (go_ && g.last && g.last != seat && hipStreamWaitEvent(seat->stream, g.event, 0) != hipSuccess) {
            (void)hipGetLastError();
            go_ = false;
        }
    }
    if (go_) locked_ = true;
    else g.m.unlock();
}

ResidentTurn::~ResidentTurn() {
    if (!locked_) return;
    Gate &g = g_gates[seat_->device];
    seat_->open = seat_->unseen = true;
    if (g.live > g.places) {
        if (hipEventRecord(g.event, seat_->stream) == hipSuccess) {
            seat_->open = false;
            g.last = seat_;
        } else (void)hipGetLastError();
    }
    g.m.unlock();
}

}  // namespace mrs
