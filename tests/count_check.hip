// Reference counts at and beyond their ceiling (run by test_counts_gpu.py).
// One block inserts nodes that share a few children through
// small_find_insert, as the small merge levels and the parallel spine do.
// The children's counts start below, at and far above the ceiling, the last
// within one addition of the end of 32 bits: below it they must grow by the
// number of nodes, from it on they must stay.  Prints "ok" or the first
// failure.
#include "merge_device.h"

#include <cstdio>
#include <vector>

using namespace svdag;

#define TRY(call)                                                        \
    do {                                                                 \
        const hipError_t e_ = (call);                                    \
        if (e_ != hipSuccess) {                                          \
            std::printf("%s: %s\n", #call, hipGetErrorString(e_));      \
            return 1;                                                    \
        }                                                                \
    } while (0)

constexpr uint32_t kNodes = 700, kShared = 6;

// Node i: children shared[i % kShared] and unique[i].
__global__ void __launch_bounds__(kSmallBlock) insert_nodes(DagDev dag, const uint32_t* shared, const uint32_t* unique,
                                                            uint32_t* result)
{
    __shared__ TableDev sTab[kRefTables];
    __shared__ SmallShared<kSmallBlock> sh;
    if (threadIdx.x == 0)
        sh.inserted = sh.oom = 0u;
    tables_stage(sTab, dag);
    __syncthreads();
    uint32_t n[kNodeStride] = {};
    const bool active = threadIdx.x < kNodes;
    if (active) {
        n[0] = 0x03u;
        n[1] = shared[threadIdx.x % kShared];
        n[2] = unique[threadIdx.x];
    }
    small_find_insert(dag, sTab, n, threadIdx.x, true, active, kRoleParentOfNodes, 0u, sh, [] {});
    if (threadIdx.x == 0) {
        result[0] = sh.inserted;
        result[1] = sh.oom;
    }
}

int main()
{
    constexpr uint32_t kTables = 8, kBuckets = 1024, kCap = 4096; // item sizes 2 .. 9
    std::vector<TableDev> tabs(kTables);
    for (uint32_t i = 0; i < kTables; ++i) {
        TableDev& t = tabs[i];
        t = TableDev {};
        t.itemWords = 2u + i;
        t.numBuckets = kBuckets;
        t.slabCap = kCap;
        t.slots = line_slots(t.itemWords);
        t.tagWords = line_tag_words(t.slots);
        std::vector<uint32_t> lines((size_t)kCap * kLineWords, 0u);
        for (uint32_t l = 0; l < kCap; ++l)
            lines[(size_t)l * kLineWords + t.tagWords] = kNoSlab;
        const AllocState a { kBuckets, 0, 0u, 0u };
        TRY(hipMalloc(t.lines.slot(), lines.size() * 4));
        TRY(hipMalloc(t.freeList.slot(), kCap * 4));
        TRY(hipMalloc(t.alloc.slot(), sizeof a));
        TRY(hipMalloc(t.refs.slot(), (size_t)kCap * kMaxSlots * 4));
        TRY(hipMalloc(t.roles.slot(), (size_t)kCap * kMaxSlots));
        TRY(hipMemcpy(t.lines, lines.data(), lines.size() * 4, hipMemcpyHostToDevice));
        TRY(hipMemcpy(t.alloc, &a, sizeof a, hipMemcpyHostToDevice));
        TRY(hipMemset(t.refs, 0, (size_t)kCap * kMaxSlots * 4));
        TRY(hipMemset(t.roles, 0, (size_t)kCap * kMaxSlots));
    }
    DagDev dag {};
    dag.numTables = kTables;
    TableDev* dTabs = nullptr;
    TRY(hipMalloc(&dTabs, sizeof(TableDev) * kTables));
    TRY(hipMemcpy(dTabs, tabs.data(), sizeof(TableDev) * kTables, hipMemcpyHostToDevice));
    dag.tables = dTabs;

    // The children are items of two words: only their handles and counts
    // matter here, so they need no words of their own.
    const uint32_t start[kShared] = { 0u, kStickyRefs - 1u, kStickyRefs, 5000u, 0xFFFFFFF0u, 0xFFFFFFFFu };
    std::vector<uint32_t> shared(kShared), unique(kNodes), refs((size_t)kCap * kMaxSlots, 0u);
    for (uint32_t k = 0; k < kShared; ++k) {
        shared[k] = node_handle((k + 1u) << kSlotBits, 2u);
        refs[(k + 1u) << kSlotBits] = start[k];
    }
    for (uint32_t i = 0; i < kNodes; ++i)
        unique[i] = node_handle((100u + i) << kSlotBits, 2u);
    TRY(hipMemcpy(tabs[0].refs, refs.data(), refs.size() * 4, hipMemcpyHostToDevice));
    uint32_t *dShared = nullptr, *dUnique = nullptr, *dResult = nullptr;
    TRY(hipMalloc(&dShared, kShared * 4));
    TRY(hipMalloc(&dUnique, kNodes * 4));
    TRY(hipMalloc(&dResult, 8));
    TRY(hipMemcpy(dShared, shared.data(), kShared * 4, hipMemcpyHostToDevice));
    TRY(hipMemcpy(dUnique, unique.data(), kNodes * 4, hipMemcpyHostToDevice));
    insert_nodes<<<1, kSmallBlock>>>(dag, dShared, dUnique, dResult);
    TRY(hipGetLastError());
    TRY(hipDeviceSynchronize());

    uint32_t result[2] = {};
    TRY(hipMemcpy(result, dResult, 8, hipMemcpyDeviceToHost));
    if (result[0] != kNodes || result[1] != 0u) {
        std::printf("inserted %u of %u, out of memory %u\n", result[0], kNodes, result[1]);
        return 1;
    }
    TRY(hipMemcpy(refs.data(), tabs[0].refs, refs.size() * 4, hipMemcpyDeviceToHost));
    for (uint32_t k = 0; k < kShared; ++k) {
        const uint32_t parents = kNodes / kShared + (k < kNodes % kShared ? 1u : 0u);
        const uint32_t want = start[k] < kStickyRefs ? start[k] + parents : start[k];
        const uint32_t got = refs[(k + 1u) << kSlotBits];
        if (got != want) {
            std::printf("child %u: count %u -> %u, not %u\n", k, start[k], got, want);
            return 1;
        }
    }
    for (uint32_t i = 0; i < kNodes; ++i)
        if (refs[(100u + i) << kSlotBits] != 1u) {
            std::printf("unique child %u: count %u\n", i, refs[(100u + i) << kSlotBits]);
            return 1;
        }
    std::printf("ok\n");
    return 0;
}
