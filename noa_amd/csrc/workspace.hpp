// Device workspaces of single calls (volume copies, partial sums, work items): kept from one call for the next on the
// same stream instead of being allocated and freed each time.
#pragma once

#include <hip/hip_runtime.h>

#include <cstddef>

namespace noa_hip {

// A device buffer for the work enqueued on `stream` until this object is destroyed. data() is null where no memory was
// left. Freeing a stream-ordered allocation waits for the stream here (hipFreeAsync returned after the kernel that used
// the buffer: the host then enqueues nothing while the GPU runs), and allocating takes 0.1 to 0.4 ms once the runtime has
// given the memory back, so the buffers are kept: at most WORKSPACE_LIMIT bytes per device, the ones of other streams
// given back first when that is reached; larger buffers, and all of them while a stream is being captured, are allocated
// and freed in stream order. Safe from several threads: a buffer belongs to one call at a time, and a call waits, on its
// stream, for the event recorded behind the buffer's last use.
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

private:
    void release();

    void* m_data{};
    size_t m_bytes{};
    hipStream_t m_stream{};
    hipEvent_t m_event{};      // null: not kept
    int m_device{};
};

constexpr size_t WORKSPACE_LIMIT = size_t(1) << 30;

// Gives the kept buffers of a device that no call is using back to the runtime; returns their bytes.
size_t workspace_trim(int device);

} // namespace noa_hip
