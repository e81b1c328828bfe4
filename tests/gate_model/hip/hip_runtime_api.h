// What csrc/resident_gate.hip needs of the runtime, as a model that runs on the host (model.cpp): streams and events are vector
// clocks, and an operation that joins somebody's capture or touches another engine's stream is counted.
#pragma once
#include <stdint.h>
#include <stdlib.h>
#include <string.h>
#include <vector>

enum hipError_t { hipSuccess = 0, hipErrorUnknown = 999 };
enum hipStreamCaptureStatus { hipStreamCaptureStatusNone = 0, hipStreamCaptureStatusActive = 1 };
enum hipDeviceAttribute_t { hipDeviceAttributeMultiprocessorCount };
constexpr unsigned hipEventDisableTiming = 2;

struct ModelStream {
    int id;
    bool capturing = false;
    std::vector<long> before;   // before[s]: the operations of stream s that come before the next one of this stream
};
struct ModelEvent { std::vector<long> before; };
typedef ModelStream *hipStream_t;
typedef ModelEvent *hipEvent_t;

struct Model {
    int places = 256;
    const ModelStream *acting = nullptr;       // the stream of the engine whose call this is
    long joined = 0, touched = 0, waits = 0, records = 0;
    int fail_every = 0, calls = 0;             // every n-th record or wait fails
};
inline Model &model() { static Model m; return m; }
inline bool model_fails() { Model &m = model(); return m.fail_every && ++m.calls % m.fail_every == 0; }
inline void model_merge(std::vector<long> &a, const std::vector<long> &b) {
    if (a.size() < b.size()) a.resize(b.size(), 0);
    for (size_t i = 0; i < b.size(); i++) if (b[i] > a[i]) a[i] = b[i];
}
inline hipError_t hipGetLastError() { return hipSuccess; }
inline hipError_t hipDeviceGetPCIBusId(char *s, int n, int) { strncpy(s, getenv("MODEL_BUS") ? getenv("MODEL_BUS") : "model", n); return hipSuccess; }
inline hipError_t hipDeviceGetAttribute(int *v, hipDeviceAttribute_t, int) { *v = model().places; return hipSuccess; }
inline hipError_t hipExtStreamGetCUMask(hipStream_t, uint32_t n, uint32_t *mask) {
    const char *e = getenv("MODEL_CU_MASK");   // the first word
    for (uint32_t i = 0; i < n; i++) mask[i] = i * 32 >= (uint32_t)model().places ? 0 : i == 0 && e ? (uint32_t)strtoul(e, nullptr, 16) : ~0u;
    return hipSuccess;
}
inline hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned) { *e = new ModelEvent; return hipSuccess; }
inline hipError_t hipStreamIsCapturing(hipStream_t s, hipStreamCaptureStatus *c) {
    *c = s->capturing ? hipStreamCaptureStatusActive : hipStreamCaptureStatusNone;
    return hipSuccess;
}
inline hipError_t hipEventRecord(hipEvent_t e, hipStream_t s) {
    Model &m = model();
    m.records++; m.joined += s->capturing; m.touched += s != m.acting;
    if (model_fails()) return hipErrorUnknown;
    e->before = s->before;
    return hipSuccess;
}
inline hipError_t hipStreamWaitEvent(hipStream_t s, hipEvent_t e, unsigned) {
    Model &m = model();
    m.waits++; m.joined += s->capturing; m.touched += s != m.acting;
    if (model_fails()) return hipErrorUnknown;
    model_merge(s->before, e->before);
    return hipSuccess;
}
