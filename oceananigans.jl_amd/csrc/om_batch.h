// om_batch.h — one kernel body, two launch forms: a launch for one model, and a launch over a
// table of members (an ensemble of independent models of any sizes) that covers every member's
// blocks in one grid.
//
// A kernel kind K is a struct with kThreads, kMinBlocks and a __device__ `run(const A &, const Blk &)`
// that reads its block coordinates from the Blk it is given, never from blockIdx/gridDim.
//   k_one<K, A>(a)          hardware block coordinates
//   k_many<K, A>(tab, n)    a flat 1-D grid; member m owns blocks [tab[m].begin, tab[m].begin +
//                           gx·gy·gz) with begin a multiple of 8, so that a member's block id keeps
//                           its residue mod 8 (the XCD the dispatcher gives it) and XCD-aware tile
//                           orders stay valid; the blocks between members exit at once.
// Host launches go through launch_k<K>(grid, block, lds, stream, args).  With a Recorder installed
// on the calling thread, the launch is appended to it instead (kind, grid, block, LDS bytes and the
// argument bytes), so an ensemble can replay every member's launch sequence as one member-table
// launch per position.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <cstring>
#include <type_traits>
#include <vector>

#include "om_internal.h"

namespace om {

struct Blk {
    uint32_t x, y, z, gx, gy, gz;
};

template <class A> struct BatchEntry {
    A a;
    uint32_t gx, gy, gz, begin;
};

// The arguments of a kind that declares kArgsInMemory are read where the launch put them (the
// kernel-argument segment, or the batch's table), in the constant address space, so that the kind may
// read them again (ConstArgs) instead of holding them all in scalar registers.
template <class K, class = void> struct ArgsInMemory { static constexpr bool value = false; };
template <class K> struct ArgsInMemory<K, std::enable_if_t<K::kArgsInMemory>> { static constexpr bool value = true; };

template <class A> struct ConstArgs {
    const OM_CONSTANT A *p;
    __device__ __forceinline__ explicit ConstArgs(const A &a) : p((const OM_CONSTANT A *)&a) {}
    // the arguments, read anew from here on: what was loaded before need not stay in registers
    __device__ __forceinline__ const A &again() const {
        const OM_CONSTANT A *q = p;
        asm volatile("" : "+s"(q));
        return *(const A *)q;
    }
};

template <class K, class A> __global__ void __launch_bounds__(K::kThreads, K::kMinBlocks) k_one(A a) {
    const Blk B{blockIdx.x, blockIdx.y, blockIdx.z, gridDim.x, gridDim.y, gridDim.z};
    if constexpr (ArgsInMemory<K>::value)   // (the only argument: the segment starts with it)
        K::run(*(const A *)(const OM_CONSTANT A *)__builtin_amdgcn_kernarg_segment_ptr(), B);
    else
        K::run(a, B);
}

template <class K, class A>
__global__ void __launch_bounds__(K::kThreads, K::kMinBlocks) k_many(const BatchEntry<A> *__restrict__ tab, int n) {
    const uint32_t id = blockIdx.x;
    int lo = 0, hi = n - 1;   // the last member whose range starts at or before id
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (tab[mid].begin <= id) lo = mid;
        else hi = mid - 1;
    }
    const BatchEntry<A> &E = tab[__builtin_amdgcn_readfirstlane(lo)];
    const uint32_t local = id - E.begin;
    if (local >= E.gx * E.gy * E.gz) return;
    const uint32_t x = local % E.gx, r = local / E.gx;
    K::run(E.a, Blk{x, r % E.gy, r / E.gy, E.gx, E.gy, E.gz});
}

// ---------------------------------------------------------------------------------------------
// recording
// ---------------------------------------------------------------------------------------------
struct LaunchRec {
    const void *kind;                                  // identifies K's family and A
    dim3 grid, block;
    size_t lds;
    std::vector<unsigned char> args;                   // the A bytes
    size_t entry_size;                                 // sizeof(BatchEntry<A>)
    void (*fill)(unsigned char *dst, const LaunchRec &r, uint32_t begin);
    void (*launch_many)(const void *tab, int n, uint32_t blocks, dim3 block, size_t lds, hipStream_t st);
};

struct Recorder {
    std::vector<LaunchRec> recs;
};

// the recorder of the calling thread (nullptr: launches run)
Recorder *&thread_recorder();

template <class K, class A> void batch_fill(unsigned char *dst, const LaunchRec &r, uint32_t begin) {
    BatchEntry<A> e;
    std::memset(&e, 0, sizeof e);
    std::memcpy(&e.a, r.args.data(), sizeof(A));
    e.gx = r.grid.x; e.gy = r.grid.y; e.gz = r.grid.z; e.begin = begin;
    std::memcpy(dst, &e, sizeof e);
}

template <class K, class A> void batch_launch_many(const void *tab, int n, uint32_t blocks, dim3 block, size_t lds, hipStream_t st) {
    hipLaunchKernelGGL((k_many<K, A>), dim3(blocks), block, lds, st, static_cast<const BatchEntry<A> *>(tab), n);
}

// A kernel kind may name a family (`using Family = …`): variants that do the same work of the step on
// members of different sizes.  Members whose recorded launches agree in kind share a position of a
// batch; launch_many tells the variants apart, and each variant is one launch of that position.
template <class K, class = void> struct KindFamily { using type = K; };
template <class K> struct KindFamily<K, std::void_t<typename K::Family>> { using type = typename K::Family; };
template <class F, class A> inline const char kind_tag = 0;

template <class K, class A> void launch_k(dim3 grid, dim3 block, size_t lds, hipStream_t st, const A &a) {
    if (Recorder *R = thread_recorder()) {
        LaunchRec r;
        r.kind = &kind_tag<typename KindFamily<K>::type, A>;
        r.grid = grid; r.block = block; r.lds = lds;
        r.args.resize(sizeof(A));
        std::memcpy(r.args.data(), &a, sizeof(A));
        r.entry_size = sizeof(BatchEntry<A>);
        r.fill = &batch_fill<K, A>;
        r.launch_many = &batch_launch_many<K, A>;
        R->recs.push_back(std::move(r));
        return;
    }
    hipLaunchKernelGGL((k_one<K, A>), grid, block, lds, st, a);
}

}  // namespace om
