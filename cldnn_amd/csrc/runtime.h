// Engine, buffer and event objects behind the C handles of cldnn_hip.h.
#pragma once
#include <atomic>
#include <condition_variable>
#include <mutex>
#include <utility>
#include <vector>

#include "common.h"

struct cldnn_hip_engine_s {
    std::atomic<int> refs{1};
    int device = 0;
    bool profiling = false;
    hipStream_t stream = nullptr;
    hipDeviceProp_t props{};
    std::atomic<int64_t> used{0}, max_used{0};
    std::mutex pool_mutex;
    std::vector<hipEvent_t> event_pool;  // recycled hipEvents (the reference pools its cl events too)
    // this device's copy of the scratch array inside the code object, looked up when the engine is created, so that
    // cldnn_hip_conv_enqueue_static_scratch only launches
    void* static_scratch = nullptr;

    // A mark is a number the stream writes into pinned host memory when everything before it is done; waiting for it is
    // reading that memory.  Marks of one engine are reached in order.
    std::mutex mark_mutex;
    uint64_t marks = 0;
    uint64_t* reached = nullptr;

    hipEvent_t take_event();
    void give_event(hipEvent_t ev);
    uint64_t mark();
    bool has_reached(uint64_t m) const { return __atomic_load_n(reached, __ATOMIC_ACQUIRE) >= m; }
    void wait_for(uint64_t m) const;
    void make_current() const;
    // where a launch of this thread goes: the stream, or what the thread is recording (cldnn_hip_engine_record_begin)
    hipStream_t launch_stream() const;
};

// The launches of a recording as an instantiated graph.
struct cldnn_hip_recording_s {
    cldnn_hip_engine engine = nullptr;
    hipGraphExec_t exec = nullptr;
};

struct cldnn_hip_buffer_s {
    std::atomic<int> refs{1};
    cldnn_hip_engine engine = nullptr;
    void* dev = nullptr;
    size_t bytes = 0;
    std::mutex lock_mutex;
    int lock_count = 0;
    void* shadow = nullptr;  // pinned host mirror, allocated on first lock
    // which copy is current.  DEVICE also stands for "not known": whoever holds the device pointer may have written.
    enum copy_state { DEVICE, HOST, BOTH };
    copy_state newest = DEVICE;
    bool read_in_place = false;  // since the host wrote the shadow a kernel has read it where it is
    bool is_result = false;      // the last use wrote it: what the host maps it for is most likely to read it
    uint64_t uploaded = 0;       // the engine's mark behind the last copy that an unmap started

    void need_shadow();
    void upload();  // shadow -> device on the engine's stream, not waited for
};

struct cldnn_hip_event_s {
    std::atomic<int> refs{1};
    cldnn_hip_engine engine = nullptr;
    bool user = false;
    std::atomic<bool> user_set{false};
    uint64_t mark = 0;           // of the engine, or 0: the end is `stop`
    hipEvent_t start = nullptr;  // only with profiling
    hipEvent_t stop = nullptr;
    // a deferred event stands for work that has not been submitted yet: it is recorded later, and whoever waits for
    // it first waits for that
    bool deferred = false;
    std::mutex deferred_mutex;
    std::condition_variable deferred_cv;
    bool deferred_pending = false;
    std::mutex handler_mutex;
    bool handlers_fired = false;
    std::vector<std::pair<cldnn_hip_event_handler, void*>> handlers;
};

namespace chip {
// translate exceptions at the C boundary (same idea as the reference's exception_handler,
// src/include/api_impl.h:63-110)
template <class F>
cldnn_hip_status guarded(F&& f)
{
    try {
        f();
        return CLDNN_HIP_SUCCESS;
    } catch (const error& e) {
        set_last_error(e.what());
        return e.status;
    } catch (const std::bad_alloc&) {
        set_last_error("host allocation failed");
        return CLDNN_HIP_OUT_OF_RESOURCES;
    } catch (const std::exception& e) {
        set_last_error(e.what());
        return CLDNN_HIP_ERROR;
    }
}
}  // namespace chip
