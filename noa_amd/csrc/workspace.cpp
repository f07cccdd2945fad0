#include "workspace.hpp"

#include <map>
#include <mutex>
#include <utility>

namespace noa_hip {
namespace {

using Kept = CallWorkspace::Kept;

struct Device {
    std::list<Kept> idle;      // the most recently used first
    size_t total{};            // bytes of the idle buffers and of those in use
};
std::mutex g_mutex;            // held for list operations and event queries only: no allocation, free or wait
std::map<int, Device> g_devices;

// The events order the GPU's work on device memory only: without the fence to the host, recording one takes 1.1 instead
// of 2.9 us of the stream's time.
constexpr unsigned EVENT_FLAGS = hipEventDisableTiming | hipEventDisableSystemFence;
constexpr size_t GRANULE = size_t(2) << 20;

bool capturing(hipStream_t stream) {
    hipStreamCaptureStatus status = hipStreamCaptureStatusNone;
    return hipStreamIsCapturing(stream, &status) == hipSuccess && status != hipStreamCaptureStatusNone;
}

// Moves idle buffers to `out`, the longest unused first, until the device's total is at most `target` (g_mutex held): the
// ones last used on `stream`, which frees them behind that use, and the ones whose last use has ended on the GPU. Another
// thread may be capturing in the mode that forbids event queries to all threads.
void make_room(Device& dev, size_t target, hipStream_t stream, std::list<Kept>& out) {
    hipStreamCaptureMode mode = hipStreamCaptureModeRelaxed;
    (void)hipThreadExchangeStreamCaptureMode(&mode);
    for (auto it = dev.idle.end(); dev.total > target && it != dev.idle.begin();) {
        const auto at = std::prev(it);
        if (at->stream == stream || hipEventQuery(at->event) == hipSuccess) {
            dev.total -= at->bytes;
            out.splice(out.end(), dev.idle, at);
        } else {
            it = at;
        }
    }
    (void)hipThreadExchangeStreamCaptureMode(&mode);
    (void)hipGetLastError();                           // of a query: not ready
}

// Frees buffers in the order of `stream` (g_mutex not held).
void give_back(std::list<Kept>& buffers, hipStream_t stream) {
    for (const Kept& k : buffers) {
        (void)hipStreamWaitEvent(stream, k.event, 0);   // nothing to wait for, but where the handle is a new stream's
        (void)hipFreeAsync(k.data, stream);
        (void)hipEventDestroy(k.event);
    }
    buffers.clear();
}

void* allocate(size_t bytes, hipStream_t stream) {
    void* data = nullptr;
    if (hipMallocAsync(&data, bytes, stream) == hipSuccess) return data;
    (void)hipGetLastError();
    return nullptr;
}

} // namespace

CallWorkspace::CallWorkspace(size_t bytes, hipStream_t stream) : m_stream(stream) {
    if (bytes == 0) return;
    (void)hipGetDevice(&m_device);
    if (capturing(stream)) {
        m_data = allocate(bytes, stream);
        return;
    }
    const size_t size = (bytes + GRANULE - 1) / GRANULE * GRANULE;
    std::list<Kept> freed;
    bool keep = false;
    {
        std::lock_guard<std::mutex> lock(g_mutex);
        Device& dev = g_devices[m_device];
        // The smallest idle buffer of this stream that holds the call and is not much larger.
        auto best = dev.idle.end();
        for (auto it = dev.idle.begin(); it != dev.idle.end(); ++it)
            if (it->stream == stream && it->bytes >= size && it->bytes <= 2 * size + 8 * GRANULE &&
                (best == dev.idle.end() || it->bytes < best->bytes))
                best = it;
        // The wait costs nothing on the same stream; a new stream may have the handle of one that was destroyed.
        if (best != dev.idle.end() && hipStreamWaitEvent(stream, best->event, 0) == hipSuccess) {
            m_kept.splice(m_kept.end(), dev.idle, best);
            m_data = m_kept.front().data;
            return;
        }
        if (size <= WORKSPACE_LIMIT) {
            if (dev.total + size > WORKSPACE_LIMIT) make_room(dev, WORKSPACE_LIMIT - size, stream, freed);
            keep = dev.total + size <= WORKSPACE_LIMIT;
            if (keep) {
                m_kept.push_back({nullptr, size, stream, nullptr});
                dev.total += size;                     // this call's, also while it allocates
            }
        }
    }
    give_back(freed, stream);
    m_data = allocate(keep ? size : bytes, stream);
    if (!m_data) {
        // Out of memory: the buffers kept for others may be what is missing.
        {
            std::lock_guard<std::mutex> lock(g_mutex);
            make_room(g_devices[m_device], 0, stream, freed);
        }
        give_back(freed, stream);
        m_data = allocate(keep ? size : bytes, stream);
    }
    if (!keep) return;
    m_kept.front().data = m_data;
    if (!m_data || hipEventCreateWithFlags(&m_kept.front().event, EVENT_FLAGS) != hipSuccess) {
        (void)hipGetLastError();
        m_kept.clear();                                // without an event: freed after the call
        std::lock_guard<std::mutex> lock(g_mutex);
        g_devices[m_device].total -= size;
    }
}

void CallWorkspace::release() noexcept {
    if (!m_data) return;
    if (m_kept.empty()) {
        (void)hipFreeAsync(m_data, m_stream);
    } else {
        Kept& kept = m_kept.front();
        kept.stream = m_stream;
        const bool recorded = hipEventRecord(kept.event, m_stream) == hipSuccess;
        {
            std::lock_guard<std::mutex> lock(g_mutex);
            Device& dev = g_devices.find(m_device)->second;
            if (recorded) dev.idle.splice(dev.idle.begin(), m_kept);
            else dev.total -= kept.bytes;
        }
        give_back(m_kept, m_stream);                   // where nothing could be recorded: freed in stream order
    }
    m_data = nullptr;
}

CallWorkspace::~CallWorkspace() { release(); }

CallWorkspace::CallWorkspace(CallWorkspace&& other) noexcept { *this = std::move(other); }

CallWorkspace& CallWorkspace::operator=(CallWorkspace&& other) noexcept {
    if (this != &other) {
        release();
        m_data = std::exchange(other.m_data, nullptr);
        m_stream = other.m_stream;
        m_kept.splice(m_kept.end(), other.m_kept);
        m_device = other.m_device;
    }
    return *this;
}

size_t workspace_trim(int device) {
    std::list<Kept> buffers;
    {
        std::lock_guard<std::mutex> lock(g_mutex);
        const auto it = g_devices.find(device);
        if (it == g_devices.end()) return 0;
        for (const Kept& k : it->second.idle) it->second.total -= k.bytes;
        buffers.swap(it->second.idle);
    }
    int current = 0;
    (void)hipGetDevice(&current);
    (void)hipSetDevice(device);
    size_t bytes = 0;
    for (const Kept& k : buffers) {
        bytes += k.bytes;
        (void)hipEventSynchronize(k.event);
    }
    give_back(buffers, nullptr);
    (void)hipStreamSynchronize(nullptr);
    (void)hipSetDevice(current);
    return bytes;
}

} // namespace noa_hip
