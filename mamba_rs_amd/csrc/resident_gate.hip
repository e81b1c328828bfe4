// Who may run resident decode steps (resident_step.hip, resident_m3_step.hip), and when.
//
// A resident launch's workgroups wait for each other, so they must all get a place on the GPU.  One launch alone always does (an
// engine takes the route only while its workgroups are at most as many as the compute units, one each); two launches that hold
// half of the places each would wait until their spin limit.  So
//   * one process per GPU has the route: the first to ask binds an abstract socket named after the GPU's PCI address, which the
//     system takes back when the process ends, whatever way it ends; another process's engines keep the kernel chains;
//   * inside the process, engines whose launches do not all fit together take turns: a launch waits (on the GPU, with an event)
//     for what the previous engine's stream holds.  An engine's own steps, on its one stream, follow each other anyway, and
//     ordinary kernels on other streams end by themselves and only delay a launch.
#include "common.hpp"
#include <errno.h>
#include <mutex>
#include <string.h>
#include <stddef.h>
#include <sys/socket.h>
#include <sys/un.h>
#include <unistd.h>

namespace mrs {
namespace {

constexpr int kMaxDevices = 64;
struct Gate {
    std::mutex m;
    bool asked = false, ours = false;
    int places = 0, live = 0;         // compute units; workgroups of the live engines' launches
    hipStream_t last = nullptr;       // stream of the last launch
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

}  // namespace

bool resident_claim(int device, int workgroups) {
    if (device < 0 || device >= kMaxDevices) return false;
    Gate &g = g_gates[device];
    std::lock_guard<std::mutex> lock(g.m);
    if (!g.asked) {
        g.asked = true;
        g.ours = hipDeviceGetAttribute(&g.places, hipDeviceAttributeMultiprocessorCount, device) == hipSuccess &&
                 hipEventCreateWithFlags(&g.event, hipEventDisableTiming) == hipSuccess && bind_gpu(device);
    }
    if (!g.ours || workgroups > g.places) return false;
    g.live += workgroups;
    return true;
}

void resident_release(int device, int workgroups, hipStream_t st) {
    Gate &g = g_gates[device];
    std::lock_guard<std::mutex> lock(g.m);
    g.live -= workgroups;
    if (g.last == st) g.last = nullptr;   // (its work is done: the engine has waited for its stream)
}

ResidentTurn::ResidentTurn(int device, hipStream_t st) : device_(device) {
    Gate &g = g_gates[device];
    g.m.lock();
    if (g.last && g.last != st && g.live > g.places) {
        hipStreamCaptureStatus cap = hipStreamCaptureStatusNone;
        if (hipStreamIsCapturing(st, &cap) == hipSuccess && cap == hipStreamCaptureStatusNone && hipEventRecord(g.event, g.last) == hipSuccess)
            (void)hipStreamWaitEvent(st, g.event, 0);
    }
    g.last = st;
}
ResidentTurn::~ResidentTurn() { g_gates[device_].m.unlock(); }

}  // namespace mrs
