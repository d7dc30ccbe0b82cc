#pragma once
// ModelJob -- the job definition shared by the model adapters: copy the request in, run the model one
// operator per scheduler stage, copy the result out and wake the client.  It has the shape of the
// reference's TVM adapters (reference jobs/tvm_mnist/tvm_mnist.cpp:10-64): same sizes, same stage
// sequence mem -> kernels -> mem(pre-notify), same extern "C" init_job entry point; the kernels come from
// the executor in paella_models.h instead of a TVM module.
//
// Differences, on purpose:
//  * the device-to-host stage copies the model OUTPUT (the reference copies its input buffer back);
//  * PAELLA_INPUT_RESIDENT=1 (measurement only) drops the host-to-device stage: the input stays in device memory;
//  * a tensor of at most PAELLA_ZERO_COPY_BYTES (default 64 KiB) gets no copy stage: the first kernel reads the input
//    from, the last kernel writes the output to, the pinned staging buffer across PCIe (the small CNN then has 5 stages
//    instead of 7, ResNet-18 no device-to-host stage); pre-notify moves to the last kernel;
//  * a model whose kernels all have at most PAELLA_GROUP_THREADS work-items (default 65536, an eighth of what the device
//    holds; 0 = off) is one scheduler stage: its kernels are issued together, in order on one queue, and only the last
//    one reports to the scheduler.  Scheduling kernel by kernel pays off for kernels that fill the device; for the small
//    CNN (5 kernels, 3 launches of at most 49 workgroups) each trip through the scheduler costs more than the kernel;
//  * request buffers in the client's shared-memory pool cannot be registered with the runtime on this
//    platform, so both copies go through a per-instance pinned staging buffer, unless the host addresses the
//    device's memory and writes the input there (filled on the server
//    thread just before the H2D copy is issued -- or, under a stage-by-stage scheduler, by a helper thread as a copy stage
//    of its own -- and drained in on_complete());
//  * under a scheduler that issues a whole job at once (fifo), PAELLA_DISPATCH=direct puts the job's kernels, in order, on one
//    of the operator library's direct-dispatch queues with the barrier bit set (a queue then behaves like a stream), the
//    input upload being a copy kernel on the same queue: plain per-request stream serving on the same launch path as the
//    stage-by-stage schedulers, so that a comparison with them is one of policy and not of launch cost.  Default there: HIP
//    streams and launches.

#include <llis/job/context.h>
#include <llis/job/coroutine_job.h>
#include <llis/server/sm_resources.h>

#include "paella_hip.h"
#include "paella_models.h"

#include <algorithm>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <stdexcept>
#include <string>
#include <vector>

namespace paella {

class ModelJob : public llis::job::CoroutineJob {
  public:
    // onnx_stem: file name (without ".onnx") of the model's ONNX zoo file.  If $LLIS_MODELS_DIR/<stem>.onnx is readable
    // the adapter serves that file -- its graph and trained weights -- instead of the built-in seeded model; the
    // reference looks in the same directory for "<stem>-cuda_llis-pack.so" (reference jobs/tvm_mnist/tvm_mnist.cpp:27).
    explicit ModelJob(const char* model_name, const char* onnx_stem = nullptr) : name_(resolve(model_name, onnx_stem)) {
        if (paella_model_io_bytes(name_.c_str(), &in_bytes_, &out_bytes_) != 0) throw std::invalid_argument("cannot load model " + name_);
    }

    // An idle instance's device memory goes back with it; one that is stopped with work in flight keeps it (the kernels of a
    // direct-dispatch queue are not waited for by the runtime's free).
    ~ModelJob() override {
        if (is_running() || has_next()) return;
        if (exec_) paella_exec_destroy(exec_);
        if (staging_) llis_hip_host_free(staging_);
    }

    static std::string resolve(const char* model_name, const char* onnx_stem) {
        const char* dir = std::getenv("LLIS_MODELS_DIR");
        if (dir && *dir && onnx_stem) {
            const std::string path = std::string(dir) + "/" + onnx_stem + ".onnx";
            if (FILE* f = std::fopen(path.c_str(), "rb")) {
                std::fclose(f);
                return "onnx:" + path;
            }
        }
        return model_name;
    }

    size_t get_input_size() override { return in_bytes_; }
    size_t get_output_size() override { return out_bytes_; }
    size_t get_param_size() override { return 4; }

    void one_time_init() override {
        const char* seed_env = std::getenv("LLIS_MODEL_SEED");
        const uint64_t seed = seed_env ? std::strtoull(seed_env, nullptr, 10) : 1;
        check(paella_model_get(name_.c_str(), seed, &model_), "paella_model_get");
        check(paella_exec_create(model_, &exec_), "paella_exec_create");
        void* p = nullptr;
        out_off_ = (in_bytes_ + 255) / 256 * 256;
        check(llis_hip_host_alloc_pinned(&p, out_off_ + out_bytes_), "pinned staging");
        staging_ = reinterpret_cast<char*>(p);
        num_stages_ = paella_model_num_stages(model_);
        const char* grp = std::getenv("PAELLA_GROUP_THREADS");
        const unsigned long group_limit = grp ? std::strtoul(grp, nullptr, 10) : 65536;
        // Only a model made of small kernels throughout is issued in one piece.  Grouping the small kernels of a large
        // model (ResNet-18's projections and its global pool) was measured too: 13.9 -> 12.8 k requests/s at saturation,
        // because a member that must wait for its predecessor stalls everything behind it in its queue.
        bool all_small = group_limit > 0;
        dims_.resize((size_t)num_stages_);
        pooled_.resize((size_t)num_stages_);
        for (int s = 0; s < num_stages_; ++s) {
            paella_launch_dims& d = dims_[(size_t)s];
            paella_model_stage_dims(model_, s, &d);
            all_small = all_small && (unsigned long)d.grid * d.block <= group_limit;
            paella_launch_dims& p = pooled_[(size_t)s];
            if (paella_model_pooled_dims(model_, s, &p) != 0) p = {};
        }
        // A conv and its pool as one launch have workgroups of their own (49 for 25 of the small CNN's first conv, up to six times as many
        // elsewhere), held to the same limit: they go out as two where it does not allow that.
        apart_.assign((size_t)num_stages_, 0);
        for (int s = 0; s < num_stages_; ++s) apart_[(size_t)s] = all_small && (unsigned long)pooled_[(size_t)s].grid * pooled_[(size_t)s].block > group_limit;
        group_end_.assign((size_t)num_stages_, 0);
        for (int s = 0; s < num_stages_; ++s) group_end_[(size_t)s] = all_small ? num_stages_ - 1 : s;
        // Kernels go out as AQL packets on the operator library's own queues unless PAELLA_DISPATCH=hip; the
        // copies stay on the pooled HIP stream.  Only under a scheduler that orders a job's stages through the
        // notification ring (fifo2, full3): the queues have no ordering of their own, and fifo relies on the stream.
        const char* resident = std::getenv("PAELLA_INPUT_RESIDENT");
        input_resident_ = resident && std::strcmp(resident, "1") == 0;
        const char* zc = std::getenv("PAELLA_ZERO_COPY_BYTES");
        const size_t zero_copy_limit = zc ? std::strtoull(zc, nullptr, 10) : 65536;
        zero_in_ = !input_resident_ && in_bytes_ <= zero_copy_limit && paella_exec_bind_input(exec_, staging_) == 0;
        zero_out_ = out_bytes_ <= zero_copy_limit && paella_exec_bind_output(exec_, staging_ + out_off_) == 0;
        timed_ = llis::job::Context::get_gpu2sched_block_time_channel()->is_connected();  // server runs with --measure_block_time
        const char* starts = std::getenv("PAELLA_UNFIT_STARTS");
        unfit_starts_ = starts && std::strcmp(starts, "1") == 0;
        const char* dispatch = std::getenv("PAELLA_DISPATCH");
        direct_ = !(dispatch && std::strcmp(dispatch, "hip") == 0) && llis::job::Context::is_stage_by_stage();
        // whole-job issue on an ordered direct queue: asked for by name, and only when no copy has to stay on the HIP stream
        // behind the kernels (every model's output here is small enough to be written by its last kernel)
        whole_job_direct_ = !llis::job::Context::is_stage_by_stage() && dispatch && std::strcmp(dispatch, "direct") == 0 && zero_out_ &&
                            in_bytes_ % sizeof(float) == 0;
        if (direct_ || whole_job_direct_) {
            void* probe = nullptr;
            if (paella_direct_queue_shared(&probe) != 0) {
                std::fprintf(stderr, "[llis] model job: direct dispatch unavailable, using HIP launches\n");
                direct_ = whole_job_direct_ = false;
            }
        }
        // Nothing of a request outlives it.  Only with direct dispatch, where instances that outlive their client spare the next one's first
        // requests 0.1 to 0.3 ms each (2 to 3 ms of p99 in every third run of 10 000 requests at 48 k/s).  With HIP launches they cost the
        // small CNN's p99 in the 9 : 1 mix 10 to 25 % at 17 k requests/s, and the rate at a p99 of 260 us and 7.93 ms falls from 16.7 to
        // 14.5 k (medians of 12 searches each; the saturation rate stays); what the runtime does with the older allocations is not known.
        if (!input_resident_ && direct_) set_shareable();
        // (Sixteen at once are another 3 to 5 % for a request alone, but twice as long in a newcomer's way; four lose 10 %.)
        uncrowded_stages_ = direct_ && !timed_ && group_limit > 0 ? 8 : 1;
        // Conv launches of different requests share launches (paella_pack_enable) unless PAELLA_PACK=0: the serving thread
        // holds them and lets them go from its loop.
        const char* pack = std::getenv("PAELLA_PACK");
        pack_ = direct_ && !(pack && std::strcmp(pack, "0") == 0);
        if (pack_) llis::job::Context::add_poll_hook(&paella_pack_poll_hook);  // one address for every adapter library: registered once
        if (direct_) llis::job::Context::set_report_hook(&paella_direct_report_hook);
        // The staging copy of an input too large for zero-copy leaves the serving thread unless PAELLA_STAGE_THREAD=0; only
        // under a scheduler that waits for a stage's completion before it issues the next one.
        const char* st = std::getenv("PAELLA_STAGE_THREAD");
        stage_off_thread_ = llis::job::Context::is_stage_by_stage() && !(st && std::strcmp(st, "0") == 0);
        // ... and needs no staging where the host addresses device memory (PAELLA_ZERO_COPY_BYTES=0 asks for copy stages throughout)
        store_input_ = direct_ && zero_copy_limit > 0 && (stage_off_thread_ || zero_in_) && !input_resident_ && paella_exec_host_io(exec_) == 0;
        if (store_input_ && zero_in_) check(paella_exec_bind_input(exec_, nullptr), "input buffer");
    }

    void body(void* io_ptr) override {
        io_ptr_ = io_ptr;
        if (zero_in_) {
            // no stage of its own: staged just before the first kernel is issued, below
        } else if (!input_resident_) {
            set_is_mem();
            // From the third input on (the first store to a page of the aperture takes a fault, 1.5 us) it is written where the kernels
            // read it: one pass instead of the copy into the staging buffer, the DMA and its marker.  ResNet-18 under load 16.1 -> 18.9 k
            // requests/s, Inception-v3 alone 481 -> 427 us.
            const bool stored = store_input_ && ++inputs_ > 2;
            if (stored) {
                set_completes_itself();
                set_stage_span(2);  // of a request whose input is staged
                yield();
                const int rc = paella_exec_store_input(exec_, io_ptr, &ModelJob::staged, static_cast<llis::job::Job*>(this));
                if (rc == PAELLA_ENOSUP) {  // not on this platform
                    store_input_ = false;
                    check(llis_hip_memcpy(paella_exec_input(exec_), io_ptr, in_bytes_, LLIS_HIP_H2D), "input");
                    staged(static_cast<llis::job::Job*>(this));
                } else {
                    check(rc, "input");
                }
                unset_completes_itself();
            } else if (stage_off_thread_) {
                // The host-side copy into the staging buffer is a copy stage of its own, done by the operator library's helper
                // thread, which reports it to the scheduler like a finished copy: the serving thread keeps reading its rings.
                set_completes_itself();
                yield();
                const int rc = paella_host_copy_submit(staging_, io_ptr, in_bytes_, &ModelJob::staged, static_cast<llis::job::Job*>(this));
                if (rc == PAELLA_EBUSY) {  // the helper sleeps: a quiet moment, the copy is done here
                    std::memcpy(staging_, io_ptr, in_bytes_);
                    staged(static_cast<llis::job::Job*>(this));
                } else {
                    check(rc, "staging copy");
                }
                unset_completes_itself();
                yield();
            } else {
                yield();
                std::memcpy(staging_, io_ptr, in_bytes_);
            }
            if (whole_job_direct_) {
                // the upload as a kernel that reads the pinned staging buffer, first packet of this job on its queue (the
                // scheduler's completion marker for the copy stage goes to the idle HIP stream and counts at once; the job
                // ends when its last kernel's workgroups have reported)
                check(paella_direct_queue_shared(&job_queue_), "direct queue");
                paella_direct_queue_set_ordered(job_queue_, 1);
                check(paella_copy_launch(reinterpret_cast<const float*>(staging_), reinterpret_cast<float*>(paella_exec_input(exec_)),
                                         in_bytes_ / sizeof(float), job_queue_, 0, nullptr), "upload kernel");
            } else if (!stored) {
                check(llis_hip_memcpy_async(paella_exec_input(exec_), staging_, in_bytes_, LLIS_HIP_H2D, stream()), "H2D");
            }
            unset_is_mem();
        } else if (!input_uploaded_) {
            // Measurement mode PAELLA_INPUT_RESIDENT=1: the instance's input is uploaded once, from its first
            // request, and every request then runs kernels + the result copy only (no host-to-device stage).
            check(llis_hip_memcpy(paella_exec_input(exec_), io_ptr, in_bytes_, LLIS_HIP_H2D), "initial H2D");
            input_uploaded_ = true;
        }

        for (int s = 0; s < num_stages_;) {
            int last = group_end_[(size_t)s];
            // One of few requests in flight is not kept waiting for the scheduler after every kernel, which is 4 us of a stage's 8 to 9,
            // and its kernels but the group's last, which report to nobody, take the tiles of a launch without a server.  Requests/s
            // with one / two / four in flight: Inception-v3 1250 / 2150 / 3420 -> 2140 / 3480 / 4740, DenseNet-121 710 / 1320 / 2310
            // -> 1270 / 2370 / 3810, ResNet-18 3280 / 5920 / 9500 -> 5060 / 7960 / 12030.
            const bool group = uncrowded_stages_ > 1 && last == s && llis::job::Context::is_uncrowded();
            if (group) last = std::min(s + uncrowded_stages_, num_stages_) - 1;
            // Admitted and accounted as its last kernel, or, where no limit bounds the others, as the largest.
            const paella_launch_dims& d = group ? largest(s, last) : dims_[(size_t)last];
            set_num_blocks(d.grid);
            set_num_threads_per_block(d.block);
            set_smem_size_per_block(d.lds_bytes);
            set_num_registers_per_thread(d.vgprs);
            if (group) {
                set_stage_span((unsigned)(last - s + 1));
                set_num_reporting_blocks(dims_[(size_t)last].grid);
            }
            if (zero_out_ && last == num_stages_ - 1) set_pre_notify();
            yield();
            if (zero_in_ && s == 0) stage_small_input(io_ptr);
            // Workgroup starts are reported only on request (PAELLA_UNFIT_STARTS=1), and then only by a kernel admitted beyond
            // the occupancy budget ("unfit"), whose over-subscription credit full3 returns once all its workgroups are resident;
            // without start messages the credit returns when the kernel ends (reference src/server/scheduler_full3.cpp:196-204).
            const uint32_t id = get_id() | (is_unfit() && unfit_starts_ ? 0u : PAELLA_JOB_ID_NO_START) | (timed_ ? PAELLA_JOB_ID_TIME_BLOCKS : 0u);
            void* target = stream();
            if (direct_) check(paella_direct_queue_shared(&target), "direct queue");
            if (whole_job_direct_) {
                if (!job_queue_) {  // no upload stage came first
                    check(paella_direct_queue_shared(&job_queue_), "direct queue");
                    paella_direct_queue_set_ordered(job_queue_, 1);
                }
                target = job_queue_;
            }
            if (pack_) enable_packing_on_this_thread();
            // members of a group wait for what is ahead of them in the queue (a stream orders by itself); the first one
            // too, so that it is not held back for packing while the others go out
            if (direct_ && last > s) paella_direct_queue_set_ordered(target, 1);
            // ... and the whole group is recorded, to go out together with the same group of other requests of this model
            const bool recording = pack_ && last > s && !group && paella_pack_sequence_begin(model_, target) == 0;
            for (int k = s, to; k <= last; k = to + 1) {
                for (to = k; to < last && !apart_[(size_t)to];) ++to;
                check(paella_exec_launch_stages(exec_, k, to, target, to == last ? id : 0, to == last ? get_finished_block_notifier() : nullptr), "stage launch");
            }
            if (recording) check(paella_pack_sequence_end(), "end of the recorded launch sequence");
            if (direct_ && last > s) paella_direct_queue_set_ordered(target, 0);
            s = last + 1;
        }
        if (job_queue_) {  // the whole job is out (the scheduler drained this coroutine in one go): the queue is the next job's
            paella_direct_queue_set_ordered(job_queue_, 0);
            job_queue_ = nullptr;
        }

        if (zero_out_) return;
        set_is_mem();
        set_pre_notify();
        yield();
        check(llis_hip_memcpy_async(staging_ + out_off_, paella_exec_output(exec_), out_bytes_, LLIS_HIP_D2H, stream()), "D2H");
    }

    // The output sits right after the input bytes of the request slot (what the client library reads).
    void on_complete() override { std::memcpy(reinterpret_cast<char*>(io_ptr_) + in_bytes_, staging_ + out_off_, out_bytes_); }

  private:
    // An input small enough that the serving thread moves it itself: 4 KB to device memory takes 0.3 us, and no kernel fetches it over
    // the bus (the small CNN alone 25.9 -> 24.9 us a request).
    void stage_small_input(void* io_ptr) {
        if (store_input_) {
            const int rc = paella_exec_store_input(exec_, io_ptr, nullptr, nullptr);
            if (rc != PAELLA_ENOSUP) {
                check(rc, "input");
                return;
            }
            store_input_ = false;  // not on this platform: the kernels read the staging buffer
            check(paella_exec_bind_input(exec_, staging_), "input buffer");
        }
        std::memcpy(staging_, io_ptr, in_bytes_);
    }

    // The launch of first..last that takes the largest share of the device, by the resource it takes most of.
    const paella_launch_dims& largest(int first, int last) const {
        using R = llis::server::SmResources;
        const paella_launch_dims* at = &dims_[(size_t)last];
        double most = 0;
        auto look = [&](const paella_launch_dims& d) {
            const double share = d.grid * std::max({(double)R::wg_threads(d.block) / (R::kSimdsPerCu * R::kMaxWavesPerSimd * R::kWaveLanes),
                                                    (double)R::wg_regs(d.block, d.vgprs) / (R::kSimdsPerCu * R::kVgprsPerSimdLane * R::kWaveLanes),
                                                    (double)R::wg_lds(d.lds_bytes) / (160 * 1024)});
            if (share > most) {
                most = share;
                at = &d;
            }
        };
        for (int k = first; k <= last; ++k) {
            look(dims_[(size_t)k]);
            if (k + 1 < last) look(pooled_[(size_t)k]);  // (a pool that reports goes out by itself)
        }
        return *at;
    }

    void* stream() { return reinterpret_cast<void*>(get_cuda_stream()); }

    static void staged(void* job) { llis::job::Context::post_mem_completion(static_cast<llis::job::Job*>(job)); }

    // Packing is a property of the launching thread (the serving thread, which also runs pack_poll from its loop).
    static void enable_packing_on_this_thread() {
        static thread_local bool on = false;
        if (!on) {
            paella_pack_enable(1);
            on = true;
        }
    }

    static void check(int rc, const char* what) {
        if (rc != 0) {
            std::fprintf(stderr, "[llis] model job: %s failed: %d (%s)\n", what, rc, rc > 0 ? llis_hip_error_string(rc) : "bad argument");
            std::abort();
        }
    }

    std::string name_;
    size_t in_bytes_ = 0, out_bytes_ = 0, out_off_ = 0;
    paella_model* model_ = nullptr;
    paella_exec* exec_ = nullptr;
    char* staging_ = nullptr;
    void* io_ptr_ = nullptr;
    int num_stages_ = 0;
    std::vector<paella_launch_dims> dims_;  // per kernel
    std::vector<paella_launch_dims> pooled_;  // per kernel: of it and the pool behind it as one launch, no workgroups where that is never done
    std::vector<char> apart_;      // per kernel: it goes out by itself in a group, although the pool behind it could be in the same launch
    std::vector<int> group_end_;   // per kernel: index of the last kernel of the group it is issued with
    bool direct_ = true;
    bool whole_job_direct_ = false;
    void* job_queue_ = nullptr;    // whole-job issue: the ordered queue this request's kernels are going to
    bool pack_ = false;
    bool stage_off_thread_ = false;
    bool store_input_ = false;     // inputs can go to device memory without a staging buffer
    unsigned inputs_ = 0;
    bool timed_ = false;
    int uncrowded_stages_ = 1;     // kernels issued at once for a request that shares the device with few others
    bool unfit_starts_ = false;
    bool input_resident_ = false, input_uploaded_ = false;
    bool zero_in_ = false, zero_out_ = false;
};

}  // namespace paella

#define PAELLA_DEFINE_MODEL_JOB(ClassName, model_name, onnx_stem)                                        \
    class ClassName : public paella::ModelJob {                                                          \
      public:                                                                                            \
        ClassName() : paella::ModelJob(model_name, onnx_stem) {}                                         \
    };                                                                                                   \
    extern "C" __attribute__((visibility("default"))) llis::job::Job* init_job() { return new ClassName(); }
