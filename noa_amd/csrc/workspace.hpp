// Device workspaces of single calls (volume copies, partial sums, work items): kept from one call for the next on the
// same stream instead of being allocated and freed each time.
#pragma once

#include <hip/hip_runtime.h>

#include <cstddef>
#include <list>

namespace noa_hip {

// A device buffer for the work enqueued on `stream` until this object is destroyed. data() is null where no memory was
// left. Allocating takes 0.1 to 0.4 ms once the runtime has given freed memory back, and a free in stream order can hold
// the host until the stream has caught up, so the buffers are kept: at most WORKSPACE_LIMIT bytes per device, over all
// streams. When that is reached, the stream's own buffers and those whose last use has ended on the GPU make room, the
// longest unused first; a buffer still in use by another stream's work is neither taken nor waited for, and the call
// allocates and frees its own in stream order, as do larger calls and all calls on a stream that is being captured. Safe from several threads: a buffer
// belongs to one call at a time, and a call waits, on its stream, for the event recorded behind the buffer's last use.
class CallWorkspace {
public:
    CallWorkspace() = default;
    CallWorkspace(size_t bytes, hipStream_t stream);
    ~CallWorkspace();
    CallWorkspace(CallWorkspace&& other) noexcept;
    CallWorkspace& operator=(CallWorkspace&& other) noexcept;
    CallWorkspace(const CallWorkspace&) = delete;
    CallWorkspace& operator=(const CallWorkspace&) = delete;

    template<class T = void> T* data() const { return static_cast<T*>(m_data); }
    explicit operator bool() const { return m_data != nullptr; }

    struct Kept {
        void* data;
        size_t bytes;
        hipStream_t stream;        // of the last use
        hipEvent_t event;          // behind it
    };

private:
    void release() noexcept;

    void* m_data{};
    hipStream_t m_stream{};
    std::list<Kept> m_kept;        // one element, moved from and to the idle buffers; empty: not kept
    int m_device{};
};

constexpr size_t WORKSPACE_LIMIT = size_t(1) << 30;

// Gives the kept buffers of a device that no call is using back to the runtime; returns their bytes.
size_t workspace_trim(int device);

} // namespace noa_hip
