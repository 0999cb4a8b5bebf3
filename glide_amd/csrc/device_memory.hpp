// Device memory kept between allocations (glide_hip_malloc, glide_hip_free).
#pragma once
#include <list>
#include <map>
#include <mutex>
#include <unordered_map>
#include "host_util.hpp"

namespace glide {

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
        try {
            std::lock_guard<std::mutex> guard(mutex_);
            live_[*ptr] = Block{bytes, device};
        } catch (...) {
            (void) hipFree(*ptr);
            throw;
        }
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
        std::list<void*> out;   // what does not fit any more; filled without allocating
        try {
            std::list<void*> entry{ptr};
            std::lock_guard<std::mutex> guard(mutex_);
            Device& d = devices_[device];
            d.by_size.emplace(block.bytes, entry.begin());   // the iterator goes on to name the element where it is moved to
            d.by_age.splice(d.by_age.end(), entry);
            d.held += block.bytes;
            while (d.held > kMostHeld) {
                const Entry oldest = d.by_age.begin();
                auto it = d.by_size.begin();
                while (it->second != oldest) ++it;   // every element of one is in the other
                d.held -= it->first;
                d.by_size.erase(it);
                out.splice(out.end(), d.by_age, oldest);
            }
        } catch (...) {   // no host memory for the bookkeeping: not held
            GLIDE_HIP_TRY(hipFree(ptr));
            return GLIDE_OK;
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

}  // namespace glide
