// The executor (csrc/models/executor.cpp) on the scripted device, launches and graphs taken by the functions below (an executable's
// definitions come before a library's).  `exec_check refuse|allow`: two requests of one model pass in turn, on buffers that move once;
// prints how often a recording was tried and how many passes were launched kernel by kernel and replayed.

#include "paella_models.h"

#include <cstdio>
#include <cstring>

namespace {
bool g_refuse = false;
int g_recorded = 0, g_launches = 0, g_replayed = 0;
}  // namespace

namespace paella {
void* forward_graph_record(int (*)(void*, void*), void*) {
    ++g_recorded;
    return g_refuse ? nullptr : &g_recorded;
}
bool forward_graph_allowed(void*) { return true; }
int forward_graph_replay(void*, void*) {
    ++g_replayed;
    return 0;
}
void forward_graph_destroy(void*) {}
}  // namespace paella

extern "C" int paella_exec_launch_stage(paella_exec*, int, void*, uint32_t, void*) {
    ++g_launches;
    return 0;
}

int main(int argc, char** argv) {
    g_refuse = argc > 1 && std::strcmp(argv[1], "refuse") == 0;
    paella_model* m = nullptr;
    paella_exec* e[2] = {nullptr, nullptr};
    if (paella_model_get("squeezenet1_1", 1, &m) || paella_exec_create(m, &e[0]) || paella_exec_create(m, &e[1])) return 1;
    alignas(16) static float moved[4];
    for (int turn = 0; turn < 2; ++turn) {
        for (int pass = 0; pass < 10; ++pass)
            for (paella_exec* x : e)
                if (paella_exec_forward(x, nullptr)) return 1;
        std::printf("%d %d %d\n", g_recorded, g_launches / paella_model_num_stages(m), g_replayed);
        for (paella_exec* x : e)
            if (paella_exec_bind_input(x, moved)) return 1;
    }
    for (paella_exec* x : e) paella_exec_destroy(x);
    return 0;
}
