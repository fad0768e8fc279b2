// with_less.hpp -- a call that is made again with less memory held.  Host code
// without HIP headers, so that it can be tested on the CPU.
#pragma once

namespace rsh {

// call() returns 0 or an error; where it failed for want of memory (lacks()) and
// give_back() had something to free, it is made again.
template <class Call, class Lacks, class GiveBack>
auto with_less(Call call, Lacks lacks, GiveBack give_back) -> decltype(call()) {
    for (;;) {
        const auto r = call();
        if (r == decltype(call()){} || !lacks() || !give_back()) return r;
    }
}

}  // namespace rsh
