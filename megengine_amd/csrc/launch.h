// Kernel launches of the library: every launch goes through launch_kernel(), which either hands it to the HIP runtime or,
// while the calling thread binds an operator call (mi355_convbias_s8_bind), notes it down instead -- kernel, grid, dynamic
// LDS and a copy of the arguments -- so that a later call replays it without walking validation, tile choice and argument
// set-up again.
//
// hipLaunchKernel is called directly: the <<<>>> form pushes and pops a launch configuration around the same call and
// needs a hipGetLastError after it (0.15 us of a 2.7 us launch on the host of an MI355X).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>
#include <string.h>

#include <tuple>
#include <utility>
#include <vector>

namespace mi355 {

// The launches of one operator call, in order.
class LaunchList {
public:
    void add(const void* fn, dim3 grid, dim3 block, unsigned lds, void* const* args, const uint32_t* sizes, uint32_t nargs) {
        Item it{fn, grid, block, lds, (uint32_t)arg_at_.size(), nargs};
        for (uint32_t i = 0; i < nargs; ++i) {
            const size_t at = blob_.size();
            blob_.resize(at + (sizes[i] + 15) / 16);
            memcpy(&blob_[at], args[i], sizes[i]);
            arg_at_.push_back((uint32_t)at);
        }
        items_.push_back(it);
    }
    // after the last add(): argument addresses are final from here on
    void seal() {
        ptrs_.clear();
        for (uint32_t at : arg_at_) ptrs_.push_back(&blob_[at]);
    }
    hipError_t replay(hipStream_t st) const {
        for (const Item& it : items_) {
            const hipError_t e = hipLaunchKernel(it.fn, it.grid, it.block, const_cast<void**>(&ptrs_[it.first]), it.lds, st);
            if (e != hipSuccess) {
                (void)hipGetLastError();
                return e;
            }
        }
        return hipSuccess;
    }

private:
    struct Item {
        const void* fn;
        dim3 grid, block;
        unsigned lds;
        uint32_t first, nargs;
    };
    struct alignas(16) Unit {
        unsigned char b[16];
    };
    std::vector<Item> items_;
    std::vector<Unit> blob_;
    std::vector<uint32_t> arg_at_;
    std::vector<void*> ptrs_;
};

// non-null while the calling thread binds an operator call (set and cleared by mi355_convbias_s8_bind only)
extern thread_local LaunchList* t_binding;

template <class... P, class... A>
int launch_kernel(void (*kern)(P...), dim3 grid, dim3 block, unsigned lds, hipStream_t st, A&&... args) {
    static_assert(sizeof...(P) == sizeof...(A), "one argument per kernel parameter");
    std::tuple<P...> vals(std::forward<A>(args)...);
    const void* fn = reinterpret_cast<const void*>(kern);
    return std::apply(
            [&](auto&... v) -> int {
                void* ptrs[] = {const_cast<void*>(static_cast<const void*>(&v))...};
                if (t_binding) {
                    const uint32_t sizes[] = {(uint32_t)sizeof(v)...};
                    t_binding->add(fn, grid, block, lds, ptrs, sizes, (uint32_t)sizeof...(P));
                    return 0;
                }
                const hipError_t e = hipLaunchKernel(fn, grid, block, ptrs, lds, st);
                if (e != hipSuccess) (void)hipGetLastError();
                return (int)e;
            },
            vals);
}

}  // namespace mi355
