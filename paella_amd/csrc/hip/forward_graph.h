#pragma once
// A forward pass recorded once and replayed.
//
// A kernel launch costs the calling thread about 3.3 us, a node of a replayed graph 1: eight ResNet-50 passes on eight streams spent
// 1.2 of their 1.9 ms in the calling thread, which could keep only two of them running at a time (now 1.4 ms).  A pass alone is faster
// launched kernel by kernel: its first kernel starts at once and the thread stays ahead of the device, where a replay starts when the
// whole graph has been handed over (Inception-v3 alone 396 against 415 us).

namespace paella {

// Records what launch(stream, arg) enqueues.  nullptr if it cannot be recorded.
void* forward_graph_record(int (*launch)(void* stream, void* arg), void* arg);
// False when a pass on this handle has to be launched kernel by kernel: a direct-dispatch queue, a stream that is being captured, armed
// timing events.
bool forward_graph_allowed(void* stream);
int forward_graph_replay(void* graph, void* stream);
void forward_graph_destroy(void* graph);

}  // namespace paella
