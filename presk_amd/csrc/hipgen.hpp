// The generic path: any PSK-Kernel nest printed as HIP source for gfx950 and
// built with hiprtc -- the executor's counterpart of the reference's LLVM
// backend, which prints a kernel as C and builds it with clang
// (crates/presk-llvm/src/lib.rs:240-304, after the C printer of
// crates/presk-export-c/src/lib.rs:291-369).
//
// Each printed kernel performs exactly the operations of the kernel
// interpreter (crates/presk-kernel/src/exec.rs:619-869) in the same order:
// f32 arithmetic for f32/bf16/f16/e8m15 storage, f64 for f64, exact widening
// loads, stores rounded once, the overflow guard, the fdlibm-method
// functions.  It is parallel only over loops whose iterations write disjoint
// output elements (`Kernel::parallel_at`, ir.rs:375-492) and carry no scalar
// from one iteration to the next, so every output element is computed by the
// same statements in the same order: bit-identical to the interpreter.
#pragma once

#include <string>
#include <vector>

#include "ir.hpp"

namespace presk {

constexpr int kMaxBufs = 24;

// What one launch of a printed phase needs: the parallel loops mapped to the
// grid (outermost first) and whether the outermost takes the [lo, hi) split.
struct Phase {
    std::string fn;                   // the __global__ function's name
    std::vector<int64_t> bounds;      // parallel loop bounds, outermost first (empty: one thread)
    bool split = false;               // bounds[0] is the KernelFn split loop
};

struct Generated {
    std::string src;
    std::vector<Phase> phases;
    bool fast_fns = false;            // an f32 exp or erf printed as FAST mode's function
};

// Prints `k`.  Returns false and sets `err` for a kernel the printer refuses.
// `fast_fns` (FAST mode): f32 exp and erf as pk_expf_fast / pk_erff_fast,
// whose results lie within a stated bound of the interpreter's, in place of
// its bits.
bool generate_hip(const Kernel& k, Generated* out, std::string* err, bool fast_fns = false);

// A nest that is one elementwise pass: its loops are the output's axes in
// order, all on the grid, `vec` consecutive elements a thread, and its one
// store is unconditional, so thread t writes elements [t vec, t vec + vec) of
// the flat output.  `same`: the inputs it reads at the output's own index only.
struct FlatNest {
    int vec = 0;
    int64_t numel = 0;
    std::vector<bool> same;
};
bool flat_nest(const Kernel& k, FlatNest* out);

// One launch for a run of such nests over one element count and vector width:
// kernels[j] after kernels[j - 1] in each thread.  from[j][b]: the earlier
// kernel whose output input b is (its `same`), taken from that kernel's
// registers, as stored; -1: memory.  Every kernel's output is written.  The
// pointers are the kernels' buffers in order, inputs then output, without the
// inputs taken from registers (`slots`: kernel and buffer of each).  FAST mode's
// exp and erf.  The source is one kernel, for chain_source to put beside others.
bool generate_chain(const std::vector<const Kernel*>& kernels, const std::vector<std::vector<int>>& from, Generated* out,
                    std::vector<std::pair<int, int>>* slots, std::string* err);
// The source of several chains' kernels as one module, the i-th under
// chain_name(i).
std::string chain_source(const std::vector<std::string>& chains);
std::string chain_name(size_t i);

// The argument block every printed phase takes (by value).
struct PhaseArgs {
    void* buf[kMaxBufs];
    unsigned* flag;
    long long lo, hi;
};

}  // namespace presk
