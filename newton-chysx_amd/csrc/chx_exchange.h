// Numbers, slots and tags of what the resident PCG's workgroups exchange.
// Plain C++ for the kernel and for the host's tests.
#pragma once

namespace chx {

// A word's tag: the launch number (8 bits, never 0) and the low 8 bits of
// the exchange's number.
constexpr unsigned exchange_tag(unsigned launch, unsigned number) { return launch << 8 | (number & 255u); }
constexpr unsigned exchange_slot(unsigned number) { return number & 1u; }

// A solve's exchanges.  Every one has sums; not every one has halo rows (the
// two-reduction solver sends none with rho).  Each kind is numbered by
// itself, so the word that a reader waits for last held the one of two
// numbers before, whose tag is another one.  (With one number for both, the
// two-reduction solver's iterations leave the rows of even numbers alone, and
// a refinement 256 numbers after the set-up would find its tag already there.)
struct Exchange {
    unsigned sums = ~0u, rows = ~0u;  // numbers of the last ones
    constexpr void next(bool with_rows) {
        ++sums;
        if (with_rows) ++rows;
    }
};

// The number of the next launch, 1 .. kResEpochs, and whether old tags have to
// be cleared before it: numbers start over, so no word may keep one.  Not
// every launch that counts runs the resident kernel (an assembly by itself,
// the streaming kernels), so the flag stays until that kernel has run, and so
// cleared: `solved`, the instances that it finished since the last number, is
// not zero then.  (The kernel taking the flag back itself cost 2 us a solve.)
constexpr unsigned kResEpochs = 255u;
struct Launch {
    unsigned long long number, clear;
};
constexpr Launch next_launch(Launch last, unsigned long long solved) {
    return last.number >= kResEpochs ? Launch{1ull, 1ull}
                                     : Launch{last.number + 1ull, solved != 0ull ? 0ull : last.clear};
}

}  // namespace chx
