// Device code shared by the level kernels (dag.hip) and the spine kernels
// (fused.hip) of the bottom-up merge: descriptors and reference counts summed
// in LDS, and the find-or-insert of a small level in one block.
#pragma once
#include "dag_internal.h"

namespace svdag {

// The tables' descriptors in LDS: a lane's probe then waits for its record,
// not for its record and then a descriptor.
__device__ inline void tables_stage(TableDev* sTab, const DagDev& dag)
{
    const uint32_t* src = reinterpret_cast<const uint32_t*>(dag.tables);
    uint32_t* dst = reinterpret_cast<uint32_t*>(sTab);
    for (uint32_t i = threadIdx.x; i < dag.numTables * (sizeof(TableDev) / 4u); i += blockDim.x)
        dst[i] = src[i];
}

__device__ inline const uint32_t* staged_node(const TableDev* sTab, uint32_t h)
{
    return table_item_ptr(sTab[node_handle_size(h) - 2u], node_handle_ptr(h));
}
__device__ inline const uint32_t* staged_leaf(const TableDev* sTab, const DagDev& dag, uint32_t h)
{
    return table_item_ptr(sTab[leaf_handle_size(dag, h) - 2u], leaf_handle_ptr(dag, h));
}

// Reference counts summed per block before they reach the tables.
constexpr uint32_t kRefSlots = 2048; // 256 items have at most 2048 children
template <uint32_t kSlots>
struct BlockRefs {
    uint32_t child[kSlots], add[kSlots];
};

__device__ inline uint32_t* child_count(const DagDev& dag, const TableDev* sTab, uint32_t c, uint8_t role)
{
    const bool leaf = role == kRoleParentOfLeaves;
    const uint32_t s = leaf ? leaf_handle_size(dag, c) : node_handle_size(c);
    return sTab[s - 2].refs + (leaf ? leaf_handle_ptr(dag, c) : node_handle_ptr(c));
}

template <uint32_t kSlots>
__device__ inline void block_ref_add(BlockRefs<kSlots>& refs, uint32_t slotMask, const DagDev& dag,
                                     const TableDev* sTab, uint32_t c, uint8_t role)
{
    uint32_t p = (c * 0x9E3779B1u) >> 21;
    for (uint32_t tries = 0; tries < 8; ++tries) {
        p &= slotMask;
        uint32_t v = __hip_atomic_load(&refs.child[p], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        if (v == kSentinel)
            v = atomicCAS(&refs.child[p], kSentinel, c);
        if (v == kSentinel || v == c) {
            atomicAdd(&refs.add[p], 1u);
            return;
        }
        ++p;
    }
    uint32_t* cnt = child_count(dag, sTab, c, role);
    if (ld_filter(cnt) < kStickyRefs)
        atomicAdd(cnt, 1u);
}

// The block's sums (after a barrier) to the tables: one update per child, none
// for a count at its ceiling -- it is never taken back, so it would grow with
// every item that shares the child until it wrapped.  Every count the thread
// updates is loaded before the first update.
template <uint32_t kBlock, uint32_t kSlots>
__device__ inline void block_refs_flush(const BlockRefs<kSlots>& refs, uint32_t slotMask, const DagDev& dag,
                                        const TableDev* sTab, uint8_t role)
{
    constexpr uint32_t kPer = kSlots / kBlock;
    uint32_t* cnt[kPer];
    uint32_t seen[kPer], add[kPer];
#pragma unroll
    for (uint32_t k = 0; k < kPer; ++k) {
        const uint32_t q = k * kBlock + threadIdx.x;
        const uint32_t c = q <= slotMask ? refs.child[q] : kSentinel;
        seen[k] = kStickyRefs;
        if (c != kSentinel) {
            cnt[k] = child_count(dag, sTab, c, role);
            add[k] = refs.add[q];
            seen[k] = ld_filter(cnt[k]);
        }
    }
#pragma unroll
    for (uint32_t k = 0; k < kPer; ++k)
        if (seen[k] < kStickyRefs)
            atomicAdd(cnt[k], add[k]);
}

// ---------------------------------------------------------------- small levels
// Levels of at most kSmallBlock items run in one block, one thread per item,
// the item's words in registers from its record to its insert: what the
// level kernels pass through the workspace (records, representatives,
// handles, the dedup table, the full flags) stays in LDS, and a level waits
// for the bucket's line, a compare and a CAS only.
constexpr uint32_t kSmallBlock = 1024;
template <uint32_t kItems>
struct SmallShared {
    uint32_t word[kNodeStride][kItems];
    uint32_t hash[kItems];
    uint32_t first[2 * kItems];
    uint32_t rep[2][kItems], handle[2][kItems]; // by level parity
    uint8_t created[2][kItems];
    BlockRefs<kRefSlots> refs[2];
    uint32_t inserted, oom;
};

// The contents n of the block's items (one per thread, active where there is
// one): equal ones collapse, each is found in the DAG (unless isNew) or
// inserted.  Item `slot` has its representative in sh.rep[parity][slot], and that one's
// handle and created flag beside it (kSentinel: empty, or the arena is
// exhausted, with sh.oom set), all visible after the call's last barrier.
// Every thread of the block (kSmallBlock of them) calls it; betweenPhases
// runs while the finds' loads are done and the inserts have not begun.
template <uint32_t kItems, typename Between>
__device__ inline void small_find_insert(const DagDev& dag, const TableDev* sTab, const uint32_t (&n)[kNodeStride],
                                         uint32_t slot, bool works, bool active, uint8_t role, uint32_t parity,
                                         SmallShared<kItems>& sh, Between&& betweenPhases)
{
    BlockRefs<kRefSlots>& refs = sh.refs[parity];
    const bool holds = active && (n[0] & 0xFFu) != 0u;
    uint32_t s = 2, h = 0;
    for (uint32_t q = threadIdx.x; q < 2 * kItems; q += kSmallBlock)
        sh.first[q] = 0u;
    for (uint32_t q = threadIdx.x; q < kRefSlots; q += kSmallBlock) {
        refs.child[q] = kSentinel;
        refs.add[q] = 0u;
    }
    if (holds) {
        s = node_size_from_header(n[0]);
        h = lane_hash<(int)kNodeStride>(n, s);
#pragma unroll
        for (uint32_t k = 0; k < kNodeStride; ++k)
            sh.word[k][slot] = n[k];
        sh.hash[slot] = h;
    }
    __syncthreads();
    uint32_t rep = slot;
    if (holds) {
        uint32_t p = mix32(h) & (2 * kItems - 1u);
        while (true) {
            uint32_t v = __hip_atomic_load(&sh.first[p], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
            if (v == 0u)
                v = atomicCAS(&sh.first[p], 0u, slot + 1u);
            if (v == 0u)
                break;
            if (sh.hash[v - 1u] == h) {
                bool eq = true;
#pragma unroll
                for (uint32_t k = 0; k < kNodeStride; ++k)
                    eq &= k >= s || sh.word[k][v - 1u] == n[k];
                if (eq) {
                    rep = v - 1u;
                    break;
                }
            }
            p = (p + 1u) & (2 * kItems - 1u);
        }
    }
    const bool leads = holds && rep == slot;
    uint32_t ptr = kNotFound, line = kNoSlab;
    LineHead head {};
    if (leads) {
        const TableDev& t = sTab[s - 2];
        if (n[9] == 0u) {
            ptr = lane_find_hint<(int)kNodeStride>(t, n, s, h, line, head, role);
        } else { // a node with a child this merge inserted is new: no find
            line = h % t.numBuckets;
            line_head_load(head, t.lines + (size_t)line * kLineWords, t.tagWords);
        }
    }
    // Every find before any insert: an insert claims a slot's tag before it
    // writes the item.
    __syncthreads();
    betweenPhases();
    if (works) {
        uint32_t handle = kSentinel;
        const bool inserts = leads && ptr == kNotFound;
        if (inserts) {
            const TableDev& t = sTab[s - 2];
            ptr = lane_insert_at<(int)kNodeStride>(t, n, s, h, line, head);
            if (ptr == kNotFound) {
                sh.oom = 1u;
            } else {
                t.roles[ptr] = role;
#pragma unroll
                for (uint32_t k = 0; k < 8; ++k)
                    if (k + 1u < s)
                        block_ref_add(refs, kRefSlots - 1u, dag, sTab, n[1 + k], role);
                atomicAdd(&sh.inserted, 1u);
            }
        }
        if (leads && ptr != kNotFound)
            handle = node_handle(ptr, s);
        sh.rep[parity][slot] = holds ? rep : kSentinel;
        sh.handle[parity][slot] = handle;
        sh.created[parity][slot] = inserts ? 1u : 0u;
    }
    __syncthreads();
    block_refs_flush<kSmallBlock>(refs, kRefSlots - 1u, dag, sTab, role);
}

} // namespace svdag
