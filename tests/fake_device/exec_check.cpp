// The executor (csrc/models/executor.cpp) on the scripted device, launches and graphs taken by the functions below (an executable's
// definitions come before a library's).  `exec_check refuse|allow`: two requests of one model pass in turn, on buffers that move once;
// prints how often a recording was tried and how many passes were launched kernel by kernel and replayed.
// `exec_check copies`: host_store, host_settle and host_load (csrc/hip/host_io.h) on host memory, up to the last byte in front of a page that may not
// be touched; prints the number of lengths checked.
// `exec_check launches <model> <takes|refuses> [first last notifier]...`: what paella_exec_launch_stages returns and issues for each range: a stage's number, with
// "*<job id>" where it reports to the notifier, or "pooled" for a conv and its pool as one launch (refuses: as that launch does for operands that overlap).

#include "../../paella_amd/csrc/hip/host_io.h"
#include "paella_models.h"

#include <sys/mman.h>

#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <string>
#include <vector>

namespace {
bool g_refuse = false;
int g_recorded = 0, g_launches = 0, g_replayed = 0;
std::string g_issued;
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

extern "C" int paella_exec_launch_stage(paella_exec*, int stage, void*, uint32_t job_id, void* notifier) {
    ++g_launches;
    g_issued += " " + std::to_string(stage);
    if (notifier || job_id) g_issued += "*" + std::to_string(job_id);
    return 0;
}

extern "C" int paella_conv2d_launch_pooled(const paella_conv_plan*, const paella_pool_desc*, const float*, const void*, const float*, const float*, float*, void*) {
    if (g_refuse) return PAELLA_ENOSUP;
    g_issued += " pooled";
    return 0;
}

static int check_launches(int argc, char** argv) {
    g_refuse = std::strcmp(argv[3], "refuses") == 0;
    paella_model* m = nullptr;
    paella_exec* e = nullptr;
    if (paella_model_get(argv[2], 1, &m) || paella_exec_create(m, &e)) return 1;
    char notifier;
    for (int i = 4; i + 2 < argc; i += 3) {
        const bool reports = std::atoi(argv[i + 2]) != 0;
        const int rc = paella_exec_launch_stages(e, std::atoi(argv[i]), std::atoi(argv[i + 1]), nullptr, reports ? 7 : 0, reports ? &notifier : nullptr);
        std::printf("%d%s\n", rc, g_issued.c_str());
        g_issued.clear();
    }
    return paella_exec_destroy(e);
}

static int check_copies() {
    constexpr size_t kRoom = 16384;
    char* const room = static_cast<char*>(mmap(nullptr, kRoom + 4096, PROT_READ | PROT_WRITE, MAP_PRIVATE | MAP_ANONYMOUS, -1, 0));
    if (room == MAP_FAILED || mprotect(room + kRoom, 4096, PROT_NONE) != 0) return 1;
    std::vector<char> src(kRoom + 1), back(kRoom);
    for (size_t i = 0; i < src.size(); ++i) src[i] = (char)(i * 7 + i / 251);
    int checked = 0;
    for (size_t n : {0, 1, 4, 15, 16, 17, 63, 64, 65, 127, 784 * 4, 4095, 4096, 4097, 4160, 4161, 12288, 16383, 16384}) {
        char* const dst = room + (kRoom - n) / 64 * 64;
        std::memset(room, 0x55, kRoom);
        paella::host_store(dst, src.data() + 1, n);
        paella::host_settle(dst, n);
        if (std::memcmp(dst, src.data() + 1, n) != 0) return 1;
        for (char* p = room; p < room + kRoom; ++p)
            if ((p < dst || p >= dst + n) && *p != 0x55) return 1;
        std::fill(back.begin(), back.end(), (char)0x33);
        paella::host_load(back.data(), dst, n);
        if (std::memcmp(back.data(), src.data() + 1, n) != 0) return 1;
        for (size_t i = n; i < kRoom; ++i)
            if (back[i] != 0x33) return 1;
        ++checked;
    }
    std::printf("%d\n", checked);
    return 0;
}

int main(int argc, char** argv) {
    if (argc > 1 && std::strcmp(argv[1], "copies") == 0) return check_copies();
    if (argc > 3 && std::strcmp(argv[1], "launches") == 0) return check_launches(argc, argv);
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
