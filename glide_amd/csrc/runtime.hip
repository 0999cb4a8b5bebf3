// Library/device helpers of the C ABI: memory, streams, events, fills, error strings.
#include <cstdio>
#include <cstring>
#include <list>
#include <map>
#include <mutex>
#include <unordered_map>
#include "host_util.hpp"

namespace {
// Freed device memory kept for the next allocation of about its size.  A build makes and frees two dozen arrays and workspaces
// of a few megabytes to a gigabyte; at 30 to 600 us each for mapping and unmapping that was 2.3 of the 8.9 ms of an index of
// 20 000 rows and 3.6 of 25.8 ms of one of 100 000 (5 us each from here).
// What freeing promises stays: all work of the device has ended before it returns, as with hipFree, so whoever gets the
// memory next, on whatever stream or thread, gets it unused.  At most kMostHeld bytes a device are held, the least recently
// freed go first; larger blocks are never held.  Everything goes back when an allocation fails and by
// glide_hip_release_memory; held memory is reported as free.
constexpr size_t kMostHeld = size_t{2} << 30;

class DeviceMemory {
public:
    int allocate(void** ptr, size_t bytes) {
        int device = 0;
        GLIDE_HIP_TRY(hipGetDevice(&device));
        {
            std::lock_guard<std::mutex> guard(mutex_);
            Device& d = devices_[device];
            auto it = d.by_size.lower_bound(bytes);
            if (it != d.by_size.end() && it->first - bytes <= bytes / 4 + 4096) {   // a fifth of it unused at most
                const Entry e = it->second;
                *ptr = *e;
                live_[*ptr] = Block{it->first, device};
                drop(d, it);
                return GLIDE_OK;
            }
        }
        hipError_t rc = hipMalloc(ptr, bytes);
        if (rc == hipErrorOutOfMemory) {
            (void) hipGetLastError();
            release();
            rc = hipMalloc(ptr, bytes);
        }
        if (rc != hipSuccess) {
            (void) hipGetLastError();   // reported here, not by the next launch
            return static_cast<int>(rc);
        }
        std::lock_guard<std::mutex> guard(mutex_);
        live_[*ptr] = Block{bytes, device};
        return GLIDE_OK;
    }

    int free(void* ptr) {
        Block block{0, -1};
        {
            std::lock_guard<std::mutex> guard(mutex_);
            const auto it = live_.find(ptr);
            if (it != live_.end()) {
                block = it->second;
                live_.erase(it);
            } else if (holds(ptr)) {
                return static_cast<int>(hipErrorInvalidValue);   // freed twice
            }
        }
        int device = 0;
        // memory of other making, of another device than the current one, or where the device cannot be waited for
        if (block.device < 0 || block.bytes > kMostHeld || hipGetDevice(&device) != hipSuccess || device != block.device || hipDeviceSynchronize() != hipSuccess) {
            (void) hipGetLastError();
            GLIDE_HIP_TRY(hipFree(ptr));
            return GLIDE_OK;
        }
        std::list<void*> out;
        {
            std::lock_guard<std::mutex> guard(mutex_);
            Device& d = devices_[device];
            d.by_age.push_back(ptr);
            d.by_size.emplace(block.bytes, std::prev(d.by_age.end()));
            d.held += block.bytes;
            while (d.held > kMostHeld) {
                const Entry oldest = d.by_age.begin();
                for (auto it = d.by_size.begin(); it != d.by_size.end(); ++it) {
                    if (it->second == oldest) {
                        out.push_back(*oldest);
                        drop(d, it);
                        break;
                    }
                }
            }
        }
        for (void* p : out) GLIDE_HIP_TRY(hipFree(p));
        return GLIDE_OK;
    }

    size_t held() {   // on the current device
        int device = 0;
        if (hipGetDevice(&device) != hipSuccess) return 0;
        std::lock_guard<std::mutex> guard(mutex_);
        const auto it = devices_.find(device);
        return it == devices_.end() ? 0 : it->second.held;
    }

    void release() {
        std::list<void*> out;
        {
            std::lock_guard<std::mutex> guard(mutex_);
            for (auto& entry : devices_) {
                out.splice(out.end(), entry.second.by_age);
                entry.second.by_size.clear();
                entry.second.held = 0;
            }
        }
        for (void* p : out) (void) hipFree(p);
    }

private:
    struct Block { size_t bytes; int device; };
    using Entry = std::list<void*>::iterator;
    struct Device {
        std::list<void*> by_age;               // least recently freed first
        std::multimap<size_t, Entry> by_size;
        size_t held = 0;
    };
    void drop(Device& d, std::multimap<size_t, Entry>::iterator it) {
        d.held -= it->first;
        d.by_age.erase(it->second);
        d.by_size.erase(it);
    }
    bool holds(void* ptr) const {
        for (const auto& entry : devices_)
            for (void* p : entry.second.by_age)
                if (p == ptr) return true;
        return false;
    }
    std::mutex mutex_;
    std::map<int, Device> devices_;
    std::unordered_map<void*, Block> live_;
};
// never destroyed: arrays may be freed by destructors that run after this file's
DeviceMemory& device_memory() {
    static DeviceMemory* const memory = new DeviceMemory;
    return *memory;
}

__global__ void fill_u32_kernel(uint32_t* p, uint32_t v, size_t n) {
    size_t i = static_cast<size_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    const size_t stride = static_cast<size_t>(gridDim.x) * blockDim.x;
    for (; i < n; i += stride) p[i] = v;
}
}  // namespace

using namespace glide;

extern "C" {

const char* glide_hip_version(void) { return "glide-hip 0.1 (gfx950)"; }

const char* glide_hip_error_string(int code) {
    switch (code) {
        case GLIDE_OK: return "success";
        case GLIDE_ERR_UNSUPPORTED: return "size outside the supported range";
        case GLIDE_ERR_BAD_ARGUMENT: return "bad argument";
        case GLIDE_ERR_NO_DEVICE: return "no HIP device";
        default: return code > 0 ? hipGetErrorString(static_cast<hipError_t>(code)) : "unknown error";
    }
}

int glide_hip_set_device(int device) {
    int n = 0;
    if (hipGetDeviceCount(&n) != hipSuccess || n == 0) return GLIDE_ERR_NO_DEVICE;
    GLIDE_HIP_TRY(hipSetDevice(device));
    return GLIDE_OK;
}

int glide_hip_device_info(char* name, size_t name_len, int* compute_units, size_t* total_mem) {
    int dev = 0;
    GLIDE_HIP_TRY(hipGetDevice(&dev));
    hipDeviceProp_t prop;
    GLIDE_HIP_TRY(hipGetDeviceProperties(&prop, dev));
    if (name && name_len) {
        std::snprintf(name, name_len, "%s (%s)", prop.name, prop.gcnArchName);
    }
    if (compute_units) *compute_units = prop.multiProcessorCount;
    if (total_mem) *total_mem = prop.totalGlobalMem;
    return GLIDE_OK;
}

int glide_hip_mem_info(size_t* free_bytes, size_t* total_bytes) {
    size_t f = 0, t = 0;
    GLIDE_HIP_TRY(hipMemGetInfo(&f, &t));
    f += device_memory().held();   // an allocation that needs it gets it
    if (free_bytes) *free_bytes = f;
    if (total_bytes) *total_bytes = t;
    return GLIDE_OK;
}

int glide_hip_malloc(void** ptr, size_t bytes) {
    if (!ptr) return GLIDE_ERR_BAD_ARGUMENT;
    try {
        return device_memory().allocate(ptr, bytes ? bytes : 1);
    } catch (...) {   // no host memory for the bookkeeping
        return static_cast<int>(hipErrorOutOfMemory);
    }
}
int glide_hip_free(void* ptr) {
    try {
        return device_memory().free(ptr);
    } catch (...) {
        return static_cast<int>(hipErrorOutOfMemory);
    }
}
int glide_hip_release_memory(void) {
    device_memory().release();
    return GLIDE_OK;
}
int glide_hip_host_alloc_pinned(void** ptr, size_t bytes) {
    if (!ptr) return GLIDE_ERR_BAD_ARGUMENT;
    GLIDE_HIP_TRY(hipHostMalloc(ptr, bytes ? bytes : 1, hipHostMallocDefault));
    return GLIDE_OK;
}
int glide_hip_host_free_pinned(void* ptr) {
    GLIDE_HIP_TRY(hipHostFree(ptr));
    return GLIDE_OK;
}
int glide_hip_memcpy_h2d(void* dst, const void* src, size_t bytes, void* stream) {
    GLIDE_HIP_TRY(hipMemcpyAsync(dst, src, bytes, hipMemcpyHostToDevice, as_stream(stream)));
    GLIDE_HIP_TRY(hipStreamSynchronize(as_stream(stream)));
    return GLIDE_OK;
}
int glide_hip_memcpy_d2h(void* dst, const void* src, size_t bytes, void* stream) {
    GLIDE_HIP_TRY(hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToHost, as_stream(stream)));
    GLIDE_HIP_TRY(hipStreamSynchronize(as_stream(stream)));
    return GLIDE_OK;
}
int glide_hip_memcpy_d2d(void* dst, const void* src, size_t bytes, void* stream) {
    GLIDE_HIP_TRY(hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToDevice, as_stream(stream)));
    return GLIDE_OK;
}
int glide_hip_memcpy_h2d_async(void* dst, const void* src, size_t bytes, void* stream) {
    GLIDE_HIP_TRY(hipMemcpyAsync(dst, src, bytes, hipMemcpyHostToDevice, as_stream(stream)));
    return GLIDE_OK;
}
int glide_hip_memcpy_d2h_async(void* dst, const void* src, size_t bytes, void* stream) {
    GLIDE_HIP_TRY(hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToHost, as_stream(stream)));
    return GLIDE_OK;
}
int glide_hip_stream_wait_event(void* stream, void* event) {
    GLIDE_HIP_TRY(hipStreamWaitEvent(as_stream(stream), static_cast<hipEvent_t>(event), 0));
    return GLIDE_OK;
}
int glide_hip_fill_u32(uint32_t* ptr, uint32_t value, size_t count, void* stream) {
    if (!ptr) return GLIDE_ERR_BAD_ARGUMENT;
    if (count == 0) return GLIDE_OK;
    const unsigned blocks = static_cast<unsigned>(count / 256 + 1 > 4096 ? 4096 : count / 256 + 1);
    hipLaunchKernelGGL(fill_u32_kernel, dim3(blocks), dim3(256), 0, as_stream(stream), ptr, value, count);
    return launch_status();
}
int glide_hip_stream_create(void** stream) {
    if (!stream) return GLIDE_ERR_BAD_ARGUMENT;
    hipStream_t s;
    GLIDE_HIP_TRY(hipStreamCreate(&s));  // default priority
    *stream = s;
    return GLIDE_OK;
}
int glide_hip_stream_destroy(void* stream) {
    GLIDE_HIP_TRY(hipStreamDestroy(as_stream(stream)));
    return GLIDE_OK;
}
int glide_hip_stream_synchronize(void* stream) {
    GLIDE_HIP_TRY(hipStreamSynchronize(as_stream(stream)));
    return GLIDE_OK;
}
int glide_hip_event_create(void** event) {
    if (!event) return GLIDE_ERR_BAD_ARGUMENT;
    hipEvent_t e;
    GLIDE_HIP_TRY(hipEventCreate(&e));
    *event = e;
    return GLIDE_OK;
}
int glide_hip_event_destroy(void* event) {
    GLIDE_HIP_TRY(hipEventDestroy(static_cast<hipEvent_t>(event)));
    return GLIDE_OK;
}
int glide_hip_event_record(void* event, void* stream) {
    GLIDE_HIP_TRY(hipEventRecord(static_cast<hipEvent_t>(event), as_stream(stream)));
    return GLIDE_OK;
}
int glide_hip_event_elapsed_ms(void* start, void* stop, float* ms) {
    if (!ms) return GLIDE_ERR_BAD_ARGUMENT;
    GLIDE_HIP_TRY(hipEventSynchronize(static_cast<hipEvent_t>(stop)));
    GLIDE_HIP_TRY(hipEventElapsedTime(ms, static_cast<hipEvent_t>(start), static_cast<hipEvent_t>(stop)));
    return GLIDE_OK;
}

}  // extern "C"
