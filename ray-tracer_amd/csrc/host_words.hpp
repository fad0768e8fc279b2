// host_words.hpp -- page-locked host words that a kernel writes and the host
// polls.  Host code without HIP headers: the runtime calls come in as
// arguments, so their failures can be tested on the CPU.
#pragma once
#include <cstddef>
#include <cstdint>
#include <cstring>

namespace rsh {

// Both addresses are set, or neither is.
struct HostWords {
    uint32_t* host = nullptr;
    uint32_t* dev = nullptr;       // the device address of the same words
};

// alloc(void**, bytes), address(void** device, void* host) and release(void*)
// return 0 on success.  Cleared words in w, or the failing call's error and w
// as it was: words without a device address are given back.
template <class Alloc, class Address, class Release>
auto acquire_words(HostWords& w, size_t bytes, Alloc alloc, Address address, Release release)
    -> decltype(alloc((void**)nullptr, bytes)) {
    using Error = decltype(alloc((void**)nullptr, bytes));
    if (w.host) return Error{};
    void *host = nullptr, *dev = nullptr;
    Error e = alloc(&host, bytes);
    if (e != Error{}) return e;
    std::memset(host, 0, bytes);
    e = address(&dev, host);
    if (e != Error{}) {
        (void)release(host);
        return e;
    }
    w.host = static_cast<uint32_t*>(host);
    w.dev = static_cast<uint32_t*>(dev);
    return Error{};
}

}  // namespace rsh
