// Graphs behind forward_graph.h.

#include "forward_graph.h"

#include "direct_dispatch.h"
#include "pack.h"

#include <mutex>

namespace paella {

bool timing_armed();  // ops_misc.hip

void* forward_graph_record(int (*launch)(void* stream, void* arg), void* arg) {
    // One stream of the library's own, for recording only; thread-local mode leaves other threads' allocations alone.
    static std::mutex mutex;
    static hipStream_t stream = nullptr;
    std::lock_guard<std::mutex> lock(mutex);
    if (!stream && hipStreamCreateWithFlags(&stream, hipStreamNonBlocking) != hipSuccess) {
        (void)hipGetLastError();
        stream = nullptr;
        return nullptr;
    }
    if (hipStreamBeginCapture(stream, hipStreamCaptureModeThreadLocal) != hipSuccess) {
        (void)hipGetLastError();
        return nullptr;
    }
    const int rc = launch(stream, arg);
    hipGraph_t graph = nullptr;
    const hipError_t ended = hipStreamEndCapture(stream, &graph);
    hipGraphExec_t exec = nullptr;
    if (rc == 0 && ended == hipSuccess && hipGraphInstantiate(&exec, graph, nullptr, nullptr, 0) != hipSuccess) exec = nullptr;
    if (graph) (void)hipGraphDestroy(graph);
    (void)hipGetLastError();
    return exec;
}

bool forward_graph_allowed(void* handle) {
    if (direct_queue_lookup(handle) || timing_armed() || g_pack_recording) return false;
    hipStreamCaptureStatus status = hipStreamCaptureStatusNone;
    return !handle || (hipStreamIsCapturing(static_cast<hipStream_t>(handle), &status) == hipSuccess && status == hipStreamCaptureStatusNone);
}

int forward_graph_replay(void* graph, void* stream) { return (int)hipGraphLaunch(static_cast<hipGraphExec_t>(graph), static_cast<hipStream_t>(stream)); }

void forward_graph_destroy(void* graph) { (void)hipGraphExecDestroy(static_cast<hipGraphExec_t>(graph)); }

}  // namespace paella
