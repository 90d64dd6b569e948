// Fused multi-edit waves: many pending edits, one SVO build and one merge.
//
// Semantics are those of applying the edits one after another
// (editMyHashDag, my_gpu_hash_dag_edits.cu:633-671, per edit); the fused form
// changes only how the work is scheduled.
//
// Split level S.  Every edit of a batch spans at most two level-S cells per
// axis (S is chosen from the largest edit).  An edit's SVO then has at most
// eight items on every level above S (its "spine"); below S it owns the
// subtrees of its level-S cells.
//
// Waves.  A wave is a run of consecutive edits whose level-S cells are
// disjoint from the voxel bounds of every earlier edit of the wave.  For a
// geometric editor (sphere / box add and remove, sphere paint) a node is
// changed only if it intersects the editor's bounds, and its decision at a
// node depends only on the node and the editor; so the subtrees below S that
// edit k builds and merges are the same whether the earlier edits of the wave
// have run or not.  One wave is therefore
//   fused_seed   for each edit and level-S cell: walk from the wave's input
//                root to the cell and decide it as the parent would
//                (svo_inner_level); subdivided cells become level-S work
//                items tagged with their edit;
//   joint levels the SVO build and merge kernels over levels S .. leaf for all
//                edits of the wave at once, with the fully-filled gate and
//                the no-leaf rule kept per edit;
//   fused_spine  one wave64 replays the edits in order on levels 0 .. S-1:
//                top-down SVO decisions against the current root, then the
//                bottom-up merge (payload cleared, gated full discovery,
//                in-level dedup, DAG find / insert), and publishes each
//                edit's root.
// Copy edits read the live DAG outside their own region and run on their
// own, as does an edit the spine cannot take (more than eight items on a
// level, which the choice of S rules out).
#include "merge_device.h"
#include <algorithm>
#include <cstring>

namespace svdag {

constexpr uint32_t kSpineItems = 8;
constexpr uint32_t kMaxWave = 256;

// Reset the wave's joint level table and status and its edits' counters.
__global__ void __launch_bounds__(256) wave_begin(WsDev ws, FusedDev f, EditStatus* status)
{
    const uint2 wv = f.waves[*f.waveIdx];
    const uint32_t t = threadIdx.x;
    if (t < kMaxLevels)
        ws.lvl[t] = LevelDesc {};
    if (t == 0)
        *ws.status = EditStatus {};
    for (uint32_t k = wv.x; k < wv.y; ++k) {
        if (t < kMaxLevels) {
            ws.edCount[k * kMaxLevels + t] = 0u;
            ws.edFull[k * kMaxLevels + t] = 0u;
        }
        if (t < 8)
            f.seedWork[k * 8 + t] = kSentinel;
        if (t == 0)
            status[k] = EditStatus {};
    }
}

// One lane per (edit, level-S cell slot).
__global__ void __launch_bounds__(256) fused_seed(WsDev ws, DagDev dag, const EditorDev* eds, FusedDev f,
                                                  const uint32_t* rootPtr)
{
    const uint2 wv = f.waves[*f.waveIdx];
    const uint32_t t = blockIdx.x * blockDim.x + threadIdx.x;
    const uint32_t k = wv.x + t / 8u, j = t & 7u;
    if (k >= wv.y)
        return;
    const SeedDesc sd = f.seeds[k];
    const uint32_t d[3] = { (j >> 2) & 1u, (j >> 1) & 1u, j & 1u };
    if (d[0] >= sd.n[0] || d[1] >= sd.n[1] || d[2] >= sd.n[2])
        return;
    const uint32_t S = f.S;
    const uint32_t cx = sd.lo[0] + d[0], cy = sd.lo[1] + d[1], cz = sd.lo[2] + d[2];
    uint32_t h = *rootPtr;
    for (uint32_t l = 0; l < S && h != kSentinel; ++l) {
        const uint32_t sh = S - 1u - l;
        const uint32_t c = (((cx >> sh) & 1u) << 2) | (((cy >> sh) & 1u) << 1) | ((cz >> sh) & 1u);
        const uint32_t* node = dag_node_ptr(dag, h);
        const uint32_t mask = node[0] & 0xFFu;
        h = ((mask >> c) & 1u) ? node[1 + __builtin_popcount(mask & ((1u << c) - 1u))] : kSentinel;
    }
    NState st = NS_PARTIAL;
    uint32_t stMat = 0;
    if (h == kSentinel)
        st = NS_EMPTY;
    else if (S != dag.leafLevel && eds[k].kind == EK_PAINT) // only paint reads Filled vs Partial
        st = header_full(dag_node_ptr(dag, h)[0], dag.M, stMat) ? NS_FILLED : NS_PARTIAL;
    uint32_t fillMat = 0;
    if (decide(eds[k], cx, cy, cz, dag.levels - S, st, fillMat) != OP_SUBDIVIDE)
        return;
    const uint32_t g = atomicAdd(&ws.lvl[S].count, 1u);
    atomicAdd(&ws.edCount[k * kMaxLevels + S], 1u);
    if (g < ws.capWork && (S != dag.leafLevel || g < ws.capLeaf)) {
        ws.work[g] = make_uint4(cx, cy, cz, h);
        ws.editOf[g] = k;
        f.seedWork[k * 8 + j] = g;
    } else {
        atomicOr(&ws.status->overflow, 1u);
    }
}

// ------------------------------------------------------------------ parallel spine
// The spine of a wave of sphere and box edits, built one level at a time for
// all edits at once instead of edit after edit.
//
// Why it is the same DAG.  Above S these tools decide by geometry alone (a
// node there is larger than any edit of the wave, so it is neither contained
// nor left untouched by state), so every edit's spine SVO is the same against
// the wave's input root as against the root the edits before it left.  The
// node an edit k builds at spine position P takes each child c either from
// its own level below (c subdivided by k) or from the DAG as the edits
// before k left it: the version of c built by the latest earlier edit whose
// spine contains c, or c's handle in the input DAG.  So level l needs only
// level l + 1 of every edit, and all edits' nodes of one level are built,
// deduplicated and found / inserted together: S sequential steps instead of
// S per edit.  Paint reads node state above S, and anything unexpected (a
// fill above S, more than eight items on a level, a missing seed) leaves the
// wave to the sequential spine.
constexpr uint32_t kParEdits = 64;
constexpr uint32_t kParItems = kParEdits * kSpineItems;
constexpr uint32_t kParThreads = kSmallBlock;

struct SpineItem {
    uint32_t x, y, z;       // position at its level
    uint32_t sub;           // children this edit subdivides
    uint32_t dep;           // paint: children whose decision read their state (empty or not)
    uint32_t ref[8];        // per subdivided child: its item one level down, or its seed work item at S
    uint32_t och[8];        // its children in the wave's input DAG (kSentinel: none)
};
struct SpineScratch {
    SpineItem item[kParEdits][kMaxLevels][kSpineItems];
    uint32_t cnt[kParEdits][kMaxLevels];
};

size_t spine_scratch_bytes()
{
    return sizeof(SpineScratch);
}

__global__ void __launch_bounds__(kParThreads) fused_spine_par(WsDev ws, DagDev dag, const EditorDev* eds, FusedDev f,
                                                               uint32_t* rootPtr, EditStatus* status,
                                                               LevelDesc* levels)
{
    __shared__ uint32_t sPos[kParItems][3];
    __shared__ uint4 sItem[2][kParItems]; // top-down: a level's positions and input-DAG handles, by level parity
    __shared__ uint32_t sCnt[2][kParEdits];
    __shared__ uint32_t sSub[kParItems], sChildNew[kParItems], sChildH[kParItems][8];
    __shared__ uint32_t sPosHash[2 * kParItems], sPosOf[kParItems], sPrev[kParItems];
    __shared__ unsigned long long sPosEdits[kParItems];
    __shared__ uint32_t sFullCnt[2][kParEdits], sDropped[kParEdits]; // full items by level parity
    __shared__ uint32_t sOk, sBad;
    __shared__ uint32_t sStop[2]; // top-down, by level parity: a level sets its flag while waves still read the last one's
    __shared__ TableDev sTab[kRefTables];
    __shared__ SmallShared<kParItems> sh;
    const uint32_t t = threadIdx.x;
    tables_stage(sTab, dag); // read after the barriers below
    const uint2 wv = f.waves[*f.waveIdx];
    const uint32_t K = wv.y - wv.x, S = f.S;
    const uint32_t leafLevel = dag.leafLevel;
    SpineScratch& sc = *reinterpret_cast<SpineScratch*>(f.spine);
    const EditStatus joint = *ws.status;
    if (t == 0) {
        sOk = K >= 1 && K <= kParEdits && S >= 1 && S <= leafLevel && !joint.overflow && !joint.oom;
        sBad = sStop[0] = sStop[1] = 0u;
        sh.oom = 0u;
        sh.inserted = 0u;
    }
    __syncthreads();
    if (sOk && t < K) {
        const uint32_t kind = eds[wv.x + t].kind;
        if (!(kind == EK_SPHERE_ADD || kind == EK_SPHERE_REMOVE || kind == EK_BOX_ADD || kind == EK_BOX_REMOVE
              || kind == EK_PAINT))
            atomicOr(&sBad, 1u);
    }
    __syncthreads();
    if (!sOk || sBad)
        return; // the sequential spine takes the wave
    const uint32_t root0 = *rootPtr;
    // An edit's level may end up without items (an edit off the volume
    // subdivides nothing), so every count starts at zero.
    for (uint32_t q = t; q < K * kMaxLevels; q += blockDim.x)
        sc.cnt[q / kMaxLevels][q % kMaxLevels] = q % kMaxLevels == 0u ? 1u : 0u;
    if (t < K) {
        sItem[0][t * kSpineItems] = make_uint4(0u, 0u, 0u, root0);
        sCnt[0][t] = 1u;
        sDropped[t] = ws.edCount[(wv.x + t) * kMaxLevels + leafLevel] == 0u ? 1u : 0u;
    }
    __syncthreads();

    // ---- top-down: every edit's spine items on levels 0 .. S-1, eight lanes
    // per item, one per child (13 us a level with one thread per item).
    for (uint32_t l = 0; l < S; ++l) {
        const uint32_t par = l & 1u, c = t & 7u;
        for (uint32_t p = t >> 3; p < K * kSpineItems; p += kParThreads / 8u) {
            const uint32_t pk = p / kSpineItems, pi = p % kSpineItems;
            const bool active = pi < sCnt[par][pk];
            uint32_t child = kSentinel;
            bool sub = false, dep = false;
            uint4 item = make_uint4(0u, 0u, 0u, kSentinel);
            if (active) {
                item = sItem[par][p];
                const EditGeom ed = eds[wv.x + pk];
                if (item.w != kSentinel) {
                    const uint32_t* node = dag_node_ptr(dag, item.w);
                    const uint32_t mask = node[0] & 0xFFu;
                    if ((mask >> c) & 1u)
                        child = node[1 + __builtin_popcount(mask & ((1u << c) - 1u))];
                }
                // Sphere and box decide by geometry alone above S.  Paint
                // reads the child's state (svo_inner_level's NodeDesc), here
                // from the wave's input DAG; the bottom-up checks that the
                // edits before it in the wave left that state as it was.
                const bool paint = ed.kind == EK_PAINT;
                NState st = NS_PARTIAL;
                uint32_t stMat = 0;
                if (paint) {
                    if (child == kSentinel)
                        st = NS_EMPTY;
                    else if (l + 1u != leafLevel)
                        st = header_full(dag_node_ptr(dag, child)[0], dag.M, stMat) ? NS_FILLED : NS_PARTIAL;
                }
                uint32_t fm = 0;
                const Op op = decide_geom(ed, (item.x << 1) | ((c >> 2) & 1u), (item.y << 1) | ((c >> 1) & 1u),
                                          (item.z << 1) | (c & 1u), dag.levels - (l + 1), st, fm);
                sub = op == OP_SUBDIVIDE;
                if (!(sub || op == OP_KEEP || (paint && op == OP_EMPTY && st == NS_EMPTY)))
                    atomicOr(&sStop[par], 1u); // a fill above S: the sequential spine takes the wave
                dep = paint && op != OP_KEEP;
            }
            const uint32_t subm = group_ballot<8>(sub, t & 56u), depm = group_ballot<8>(dep, t & 56u);
            sChildH[p][c] = child;
            if (c == 0)
                sSub[p] = subm;
            if (active) {
                SpineItem& it = sc.item[pk][l][pi];
                it.och[c] = child;
                if (c == 0) {
                    it.x = item.x;
                    it.y = item.y;
                    it.z = item.z;
                    it.sub = subm;
                    it.dep = depm;
                }
            }
        }
        __syncthreads();
        for (uint32_t p = t >> 3; p < K * kSpineItems; p += kParThreads / 8u) {
            const uint32_t pk = p / kSpineItems, pi = p % kSpineItems;
            uint32_t before = 0, total = 0;
            for (uint32_t q = 0; q < kSpineItems; ++q) {
                const uint32_t n = (uint32_t)__builtin_popcount(sSub[pk * kSpineItems + q]);
                before += q < pi ? n : 0u;
                total += n;
            }
            const uint32_t subm = sSub[p];
            if ((subm >> c) & 1u) {
                const uint4 item = sItem[par][p];
                const uint32_t cx = (item.x << 1) | ((c >> 2) & 1u), cy = (item.y << 1) | ((c >> 1) & 1u),
                               cz = (item.z << 1) | (c & 1u);
                uint32_t ref = before + (uint32_t)__builtin_popcount(subm & ((1u << c) - 1u));
                if (l + 1 < S) {
                    if (ref < kSpineItems)
                        sItem[par ^ 1u][pk * kSpineItems + ref] = make_uint4(cx, cy, cz, sChildH[p][c]);
                } else {
                    const SeedDesc sd = f.seeds[wv.x + pk];
                    const uint32_t dx = cx - sd.lo[0], dy = cy - sd.lo[1], dz = cz - sd.lo[2];
                    const bool inRange = dx < sd.n[0] && dy < sd.n[1] && dz < sd.n[2];
                    ref = inRange ? f.seedWork[(wv.x + pk) * 8 + ((dx << 2) | (dy << 1) | dz)] : kSentinel;
                    if (ref == kSentinel)
                        atomicOr(&sStop[par], 1u);
                }
                sc.item[pk][l][pi].ref[c] = ref;
            }
            if (pi == 0 && c == 0 && l + 1 < S) {
                sCnt[par ^ 1u][pk] = total < kSpineItems ? total : kSpineItems;
                sc.cnt[pk][l + 1] = total < kSpineItems ? total : kSpineItems;
                if (total > kSpineItems)
                    atomicOr(&sStop[par], 1u);
            }
        }
        __syncthreads();
        if (sStop[par])
            return; // nothing written outside the scratch: the sequential spine takes the wave
    }
    const uint32_t k = t >> 3, i = t & 7u; // one (edit, item) pair per thread from here on

    // ---- bottom-up: levels S-1 .. 0, every edit's nodes of a level at once.
    // An item of the SVO does not change any more, so the next level's is
    // loaded while this one is found and inserted.
    const uint32_t idx = t; // (edit k, item i) = (t / 8, t % 8)
    struct Ahead {
        uint32_t cnt, x, y, z, sub, dep, ref[8], och[8];
    };
    auto load = [&](uint32_t l, Ahead& a) {
        a.cnt = k < K ? sc.cnt[k][l] : 0u;
        const SpineItem& it = sc.item[k < K ? k : 0u][l][i];
        a.x = it.x;
        a.y = it.y;
        a.z = it.z;
        a.sub = it.sub;
        a.dep = it.dep;
#pragma unroll
        for (uint32_t c = 0; c < 8; ++c) {
            a.ref[c] = it.ref[c];
            a.och[c] = it.och[c];
        }
    };
    const bool paint = k < K && eds[wv.x + k].kind == EK_PAINT;
    if (t < kParEdits)
        sFullCnt[S & 1u][t] = t < K ? ws.edFull[(wv.x + t) * kMaxLevels + S] : 0u;
    Ahead next;
    load(S - 1u, next);
    for (int l = (int)S - 1; l >= 0; --l) {
        const Ahead it = next;
        if (l > 0)
            load((uint32_t)l - 1u, next);
        const uint32_t parity = (uint32_t)l & 1u;
        const bool here = k < K && i < it.cnt;
        const bool active = here && !sDropped[k];
        const bool childLevelS = (uint32_t)l + 1 == S;
        const bool leafChildren = (uint32_t)l + 1 == leafLevel;
        // Stage the level in LDS: positions, and the subdivided children with
        // their merge results.  A skipped (no-leaf) edit rebuilds nothing, so
        // it stages no subdivided children.
        if (t < kParItems) {
            uint32_t subm = 0, newm = 0;
            sPos[t][0] = kSentinel;
            if (here) {
                sPos[t][0] = it.x;
                sPos[t][1] = it.y;
                sPos[t][2] = it.z;
            }
            if (active) {
                subm = it.sub;
                uint32_t rep[8], h[8], cr[8];
#pragma unroll
                for (uint32_t c = 0; c < 8; ++c) {
                    rep[c] = h[c] = kSentinel;
                    cr[c] = 0u;
                }
                if (childLevelS) {
#pragma unroll
                    for (uint32_t c = 0; c < 8; ++c)
                        if ((subm >> c) & 1u)
                            rep[c] = ws.rep[it.ref[c]];
#pragma unroll
                    for (uint32_t c = 0; c < 8; ++c)
                        if (rep[c] != kSentinel) {
                            h[c] = ws.handle[rep[c]];
                            cr[c] = ws.created[rep[c]] & 1u;
                        }
                } else {
#pragma unroll
                    for (uint32_t c = 0; c < 8; ++c)
                        if ((subm >> c) & 1u) {
                            rep[c] = sh.rep[parity ^ 1u][k * kSpineItems + it.ref[c]];
                            if (rep[c] != kSentinel) {
                                h[c] = sh.handle[parity ^ 1u][rep[c]];
                                cr[c] = sh.created[parity ^ 1u][rep[c]];
                            }
                        }
                }
#pragma unroll
                for (uint32_t c = 0; c < 8; ++c)
                    if ((subm >> c) & 1u) {
                        sChildH[t][c] = h[c];
                        newm |= cr[c] << c;
                    }
            }
            sSub[t] = subm;
            sChildNew[t] = newm;
            sPosEdits[t] = 0ull;
        }
        for (uint32_t h = t; h < 2 * kParItems; h += blockDim.x)
            sPosHash[h] = 0u;
        if (t < kParEdits)
            sFullCnt[parity][t] = 0u;
        __syncthreads();
        // Group the level's items by position: the first item to claim a
        // position names it, and collects the set of edits with an item there.
        if (t < kParItems && sPos[t][0] != kSentinel) {
            const uint32_t px = sPos[t][0], py = sPos[t][1], pz = sPos[t][2];
            uint32_t p = mix32(px * 0x9E3779B1u ^ mix32(py * 0x85EBCA77u ^ mix32(pz))) & (2 * kParItems - 1u);
            uint32_t owner = t;
            while (true) {
                uint32_t v = sPosHash[p];
                if (v == 0u) {
                    v = atomicCAS(&sPosHash[p], 0u, t + 1u);
                    if (v == 0u)
                        break;
                }
                if (sPos[v - 1u][0] == px && sPos[v - 1u][1] == py && sPos[v - 1u][2] == pz) {
                    owner = v - 1u;
                    break;
                }
                p = (p + 1u) & (2 * kParItems - 1u);
            }
            sPosOf[t] = owner;
            atomicOr(&sPosEdits[owner], 1ull << (t / kSpineItems));
        }
        __syncthreads();
        // Each item's predecessor: the same position's item in the latest
        // earlier edit that has one.
        if (t < kParItems) {
            uint32_t prev = kSentinel;
            if (sPos[t][0] != kSentinel) {
                const uint32_t e = t / kSpineItems;
                const unsigned long long before = sPosEdits[sPosOf[t]] & ((1ull << e) - 1ull);
                if (before != 0ull) {
                    const uint32_t j = 63u - (uint32_t)__builtin_clzll(before);
                    for (uint32_t q = 0; q < kSpineItems; ++q) {
                        const uint32_t o = j * kSpineItems + q;
                        if (sPos[o][0] != kSentinel && sPosOf[o] == sPosOf[t]) {
                            prev = o;
                            break;
                        }
                    }
                }
            }
            sPrev[t] = prev;
        }
        __syncthreads();
        uint32_t rec[kNodeStride];
#pragma unroll
        for (uint32_t w = 0; w < kNodeStride; ++w)
            rec[w] = 0u;
        if (active) {
            const uint32_t mySub = sSub[idx];
            uint32_t ver[8];
#pragma unroll
            for (uint32_t c = 0; c < 8; ++c)
                ver[c] = ((mySub >> c) & 1u) ? sChildH[idx][c] : it.och[c];
            // A child this edit leaves alone is the version the latest earlier
            // edit rebuilt, else the input DAG's: walk the position's
            // predecessors until every such child has its version.
            uint32_t left = ~mySub & 0xFFu;
            for (uint32_t o = sPrev[idx]; left != 0u && o != kSentinel; o = sPrev[o]) {
                const uint32_t hit = sSub[o] & left;
#pragma unroll
                for (uint32_t c = 0; c < 8; ++c)
                    if ((hit >> c) & 1u)
                        ver[c] = sChildH[o][c];
                left &= ~hit;
            }
            uint32_t n = 0, newMask = 0;
#pragma unroll
            for (uint32_t c = 0; c < 8; ++c) {
                if (ver[c] == kSentinel)
                    continue;
#pragma unroll
                for (uint32_t q = 0; q <= c; ++q)
                    if (q == n)
                        rec[1 + q] = ver[c];
                ++n;
                newMask |= 1u << c;
            }
            // Discovery, gated on this edit's full items one level down.
            bool full = false;
            uint32_t fm = 0;
            if (sFullCnt[parity ^ 1u][k] != 0u && newMask == 0xFFu) {
                full = true;
#pragma unroll
                for (uint32_t j = 0; j < 8; ++j) {
                    if (!full || (j > 0 && rec[1 + j] == rec[1]))
                        continue;
                    uint32_t m = 0;
                    const bool fj = leafChildren ? leaf_is_full(dag_leaf_ptr(dag, rec[1 + j]), dag.M, m)
                                                 : header_full(dag_node_ptr(dag, rec[1 + j])[0], dag.M, m);
                    if (j == 0)
                        fm = m;
                    full = fj && m == fm;
                }
            }
            rec[0] = full ? header_make_full(0xFFu, fm, dag.M) : header_make(newMask, 0u, dag.M);
            rec[9] = sChildNew[idx] != 0u ? 1u : 0u;
            if (full)
                atomicAdd(&sFullCnt[parity][k], 1u);
        }
        // A paint item decided its state-dependent children on the input
        // DAG's state; the edits before it in the wave may have made such a
        // child empty or non-empty.  The DAG would come out the same (the
        // paint's own cells are disjoint from those edits), but its SVO would
        // not, so such a wave goes to the sequential spine, which decides on
        // the current state.  Nothing of the wave is published before the
        // last level, and what was inserted below is what the sequential
        // spine builds again and finds.
        if (here && paint) {
            uint32_t need = it.dep, prior[8];
#pragma unroll
            for (uint32_t c = 0; c < 8; ++c)
                prior[c] = it.och[c];
            for (uint32_t o = sPrev[idx]; need != 0u && o != kSentinel; o = sPrev[o]) {
                const uint32_t hit = sSub[o] & need;
#pragma unroll
                for (uint32_t c = 0; c < 8; ++c)
                    if ((hit >> c) & 1u)
                        prior[c] = sChildH[o][c];
                need &= ~hit;
            }
#pragma unroll
            for (uint32_t c = 0; c < 8; ++c)
                if (((it.dep >> c) & 1u) && (prior[c] == kSentinel) != (it.och[c] == kSentinel))
                    atomicOr(&sBad, 1u);
        }
        __syncthreads();
        if (sBad)
            break; // the sequential spine takes the wave
        small_find_insert(dag, sTab, rec, idx, t < kParItems, active, node_role(dag, (uint32_t)l), parity, sh, [] {});
        if (sh.oom)
            break;
    }
    __syncthreads();
    if (t == 0 && sh.inserted)
        atomicAdd(dag.stored, (unsigned long long)sh.inserted);
    if (sBad)
        return;

    // ---- per-edit results, in edit order.
    if (sh.oom) {
        if (t == 0) {
            EditStatus st {};
            st.oom = 1u;
            st.rootBefore = st.rootAfter = root0;
            status[wv.x] = st;
            *ws.poison = 1u;
            *f.spineDone = 1u;
        }
        return;
    }
    for (uint32_t q = t; q < K * kMaxLevels; q += blockDim.x) {
        const uint32_t e = q / kMaxLevels, lev = q % kMaxLevels;
        LevelDesc d {};
        d.count = lev < S ? sc.cnt[e][lev] : ws.edCount[(wv.x + e) * kMaxLevels + lev];
        levels[(wv.x + e) * kMaxLevels + lev] = d;
    }
    if (t == 0) {
        uint32_t root = root0;
        for (uint32_t e = 0; e < K; ++e) {
            EditStatus st {};
            st.done = 1u;
            st.rootBefore = root;
            if (!sDropped[e]) {
                st.applied = 1u;
                st.leafCount = ws.edCount[(wv.x + e) * kMaxLevels + leafLevel];
                const uint32_t rep = sh.rep[0][e * kSpineItems];
                root = rep == kSentinel ? kSentinel : sh.handle[0][rep];
            }
            st.rootAfter = root;
            status[wv.x + e] = st;
        }
        *rootPtr = root;
        *f.spineDone = 1u;
    }
}

// One wave64 (the whole block) replays the wave's edits on levels 0 .. S-1.
__global__ void __launch_bounds__(64) fused_spine(WsDev ws, DagDev dag, const EditorDev* eds, FusedDev f,
                                                  uint32_t* rootPtr, EditStatus* status, LevelDesc* levels)
{
    __shared__ uint4 sItem[kMaxLevels][kSpineItems];
    __shared__ uint32_t sRec[kMaxLevels][kSpineItems][kNodeStride];
    __shared__ uint32_t sHandle[kMaxLevels][kSpineItems];
    __shared__ uint32_t sCreated[kMaxLevels][kSpineItems]; // 1: the spine inserted it
    __shared__ uint32_t sHasNew[kSpineItems];               // item has a created child
    __shared__ uint32_t sCnt[kMaxLevels];
    __shared__ RefArrays sRa;
    const uint32_t lane = threadIdx.x;
    ref_arrays_stage(sRa, dag); // read after the barriers below
    if (*f.spineDone) {
        // The parallel spine took this wave.
        __syncthreads();
        if (lane == 0) {
            *f.spineDone = 0u;
            *f.waveIdx += 1u;
        }
        return;
    }
    const uint2 wv = f.waves[*f.waveIdx];
    const uint32_t S = f.S;
    const uint32_t leafLevel = dag.leafLevel;
    uint32_t root = *rootPtr;
    const EditStatus joint = *ws.status;
    if (joint.overflow || joint.oom) {
        // Nothing of the wave is applied; the host grows what ran out and
        // runs the edits again from the wave's first one.
        if (lane == 0) {
            EditStatus st {};
            st.overflow = joint.overflow;
            st.oom = joint.oom;
            st.rootBefore = st.rootAfter = root;
            status[wv.x] = st;
            *ws.poison = 1u;
        }
        if (lane < kMaxLevels)
            levels[wv.x * kMaxLevels + lane] = ws.lvl[lane];
        __syncthreads();
        if (lane == 0)
            *f.waveIdx += 1u;
        return;
    }
    const uint32_t i8 = lane >> 3, c8 = lane & 7u, gbase = lane & ~7u;
    for (uint32_t k = wv.x; k < wv.y; ++k) {
        const EditorDev& ed = eds[k];
        const SeedDesc sd = f.seeds[k];
        // ---- top-down: the edit's SVO on levels 0 .. S-1 (svo_inner_level).
        if (lane == 0) {
            sItem[0][0] = make_uint4(0u, 0u, 0u, root);
            sCnt[0] = 1u;
        }
        __syncthreads();
        bool bad = false;
        for (uint32_t l = 0; l < S; ++l) {
            const uint32_t n = sCnt[l];
            const bool active = i8 < n;
            const uint32_t childLevel = l + 1u;
            const bool leafChildren = childLevel == leafLevel;
            const uint4 item = active ? sItem[l][i8] : make_uint4(0u, 0u, 0u, kSentinel);
            uint32_t childHandle = kSentinel;
            if (item.w != kSentinel) {
                const uint32_t* node = dag_node_ptr(dag, item.w);
                const uint32_t mask = node[0] & 0xFFu;
                if ((mask >> c8) & 1u)
                    childHandle = node[1 + __builtin_popcount(mask & ((1u << c8) - 1u))];
            }
            const uint32_t cx = (item.x << 1) | ((c8 >> 2) & 1u);
            const uint32_t cy = (item.y << 1) | ((c8 >> 1) & 1u);
            const uint32_t cz = (item.z << 1) | (c8 & 1u);
            NState st = NS_PARTIAL;
            uint32_t stMat = 0;
            if (childHandle == kSentinel)
                st = NS_EMPTY;
            else if (!leafChildren && ed.kind == EK_PAINT) // only paint reads Filled vs Partial
                st = header_full(dag_node_ptr(dag, childHandle)[0], dag.M, stMat) ? NS_FILLED : NS_PARTIAL;
            uint32_t fillMat = 0;
            const Op op = active ? decide(ed, cx, cy, cz, dag.levels - childLevel, st, fillMat) : OP_KEEP;
            const bool sub = active && op == OP_SUBDIVIDE;
            const unsigned long long subBal = __ballot(sub);
            const uint32_t gsub = (uint32_t)(subBal >> gbase) & 0xFFu;
            uint32_t ref = childHandle;
            if (sub) {
                if (childLevel < S) {
                    const uint32_t idx = (uint32_t)__builtin_popcountll(subBal & ((1ull << lane) - 1ull));
                    if (idx < kSpineItems)
                        sItem[childLevel][idx] = make_uint4(cx, cy, cz, childHandle);
                    ref = idx;
                } else {
                    const uint32_t dx = cx - sd.lo[0], dy = cy - sd.lo[1], dz = cz - sd.lo[2];
                    const bool inRange = dx < sd.n[0] && dy < sd.n[1] && dz < sd.n[2];
                    ref = inRange ? f.seedWork[k * 8 + ((dx << 2) | (dy << 1) | dz)] : kSentinel;
                    bad |= ref == kSentinel;
                }
            } else if (op == OP_EMPTY) {
                ref = kSentinel;
            } else if (op == OP_FILL) {
                ref = dag.fullyFilled[childLevel * dag.numMaterials + fillMat];
            }
            const bool out = active && ref != kSentinel;
            const uint32_t cmask = (uint32_t)(__ballot(out) >> gbase) & 0xFFu;
            if (active) {
                uint32_t* rec = sRec[l][i8];
                const uint32_t nOut = __builtin_popcount(cmask);
                if (out)
                    rec[1 + __builtin_popcount(cmask & ((1u << c8) - 1u))] = ref;
                if (c8 >= nOut)
                    rec[1 + c8] = 0u;
                if (c8 == 0) {
                    rec[0] = cmask ? header_make(cmask, gsub, dag.M) : 0u;
                    rec[9] = 0u;
                }
            }
            const uint32_t total = (uint32_t)__builtin_popcountll(subBal);
            if (childLevel < S && total > kSpineItems)
                bad = true;
            if (lane == 0 && childLevel < S)
                sCnt[childLevel] = min(total, kSpineItems);
            __syncthreads();
        }
        if (__ballot(bad) != 0) {
            // Hand the edit back to the host, which runs it on its own.
            if (lane == 0) {
                EditStatus st {};
                st.fallback = 1u;
                st.rootBefore = st.rootAfter = root;
                status[k] = st;
                *ws.poison = 1u;
            }
            break;
        }
        if (lane < kMaxLevels) {
            LevelDesc d {};
            d.count = lane < S ? sCnt[lane] : ws.edCount[k * kMaxLevels + lane];
            levels[k * kMaxLevels + lane] = d;
        }
        const uint32_t leafCount = ws.edCount[k * kMaxLevels + leafLevel];
        if (leafCount == 0) {
            // No leaf: the edit is dropped (my_gpu_hash_dag_edits.cu:651).
            if (lane == 0) {
                EditStatus st {};
                st.done = 1u;
                st.seqSpine = 1u;
                st.rootBefore = st.rootAfter = root;
                status[k] = st;
            }
            __syncthreads();
            continue;
        }
        // ---- bottom-up merge of levels S-1 .. 0.
        uint32_t prevFull = ws.edFull[k * kMaxLevels + S];
        bool oom = false;
        for (int l = (int)S - 1; l >= 0; --l) {
            const uint32_t n = sCnt[l];
            const bool childSeed = (uint32_t)l + 1u == S;
            const bool leafChildren = (uint32_t)l + 1u == leafLevel;
            // updateChildPointers + gated discover_fully_filled: one lane per item.
            bool full = false;
            if (lane < n) {
                uint32_t* rec = sRec[l][lane];
                const uint32_t hdr = rec[0];
                const uint32_t mask = hdr & 0xFFu;
                if (mask) {
                    const uint32_t imask = header_payload(hdr, dag.M) & 0xFFu;
                    uint32_t outH[8];
                    uint32_t nOut = 0, newMask = 0, q = 0, newChild = 0;
                    for (uint32_t c = 0; c < 8; ++c) {
                        if (!((mask >> c) & 1u))
                            continue;
                        uint32_t h = rec[1 + q++];
                        if ((imask >> c) & 1u) {
                            if (childSeed) {
                                const uint32_t r = ws.rep[h];
                                h = (r == kSentinel) ? kSentinel : ws.handle[r];
                                if (r != kSentinel)
                                    newChild |= ws.created[r] & 1u;
                            } else {
                                newChild |= sCreated[l + 1][h];
                                h = sHandle[l + 1][h];
                            }
                        }
                        if (h != kSentinel) {
                            outH[nOut++] = h;
                            newMask |= 1u << c;
                        }
                    }
                    uint32_t fm = 0;
                    if (prevFull != 0 && newMask == 0xFFu) {
                        full = true;
                        for (uint32_t j = 0; j < 8 && full; ++j) {
                            uint32_t m = 0;
                            const bool fj = leafChildren ? leaf_is_full(dag_leaf_ptr(dag, outH[j]), dag.M, m)
                                                         : header_full(dag_node_ptr(dag, outH[j])[0], dag.M, m);
                            if (j == 0)
                                fm = m;
                            full = fj && m == fm;
                        }
                    }
                    rec[0] = full ? header_make_full(0xFFu, fm, dag.M) : header_make(newMask, 0u, dag.M);
                    for (uint32_t j = 0; j < 8; ++j)
                        rec[1 + j] = j < nOut ? outH[j] : 0u;
                    sHasNew[lane] = newChild;
                }
            }
            prevFull = (uint32_t)__builtin_popcountll(__ballot(full));
            __syncthreads();
            // In-level dedup, then DAG find / insert: eight lanes per item.
            bool empty = true;
            uint32_t repIdx = i8;
            if (i8 < n) {
                const uint32_t* rec = sRec[l][i8];
                empty = (rec[0] & 0xFFu) == 0u;
                for (uint32_t j = 0; j < i8 && !empty; ++j) {
                    bool eq = true;
                    for (uint32_t w = 0; w < kNodeStride && eq; ++w)
                        eq = sRec[l][j][w] == rec[w];
                    if (eq) {
                        repIdx = j;
                        break;
                    }
                }
            }
            uint32_t handle = kSentinel, created = 0;
            const bool mine = i8 < n && !empty && repIdx == i8;
            const uint8_t role = node_role(dag, (uint32_t)l);
            uint32_t r = kNotFound, hint = kNoSlab, s = 0, h = 0;
            Needle<8> nd;
            if (mine) {
                const uint32_t* rec = sRec[l][i8];
                s = node_size_from_header(rec[0]);
                needle_load(nd, rec, s, c8);
                h = needle_hash(nd, s, c8);
                // A node with a child inserted by this merge is new: no find.
                if (sHasNew[i8] == 0u)
                    r = table_find_group_hint<8>(dag.tables[s - 2], nd, s, h, c8, gbase, hint, role);
            }
            // Every find before any insert: an insert claims a slot's tag
            // before it writes the item.
            __syncthreads();
            if (mine && r == kNotFound) {
                r = table_insert_group<8>(dag.tables[s - 2], nd, s, h, c8, gbase, hint);
                created = 1u;
                if (r != kNotFound) {
                    refs_on_insert(dag, sRa, nd, s, r, role, c8);
                    if (c8 == 0)
                        atomicAdd(dag.stored, 1ull);
                }
            }
            if (mine) {
                if (r == kNotFound)
                    oom = true;
                else
                    handle = node_handle(r, s);
            }
            if (c8 == 0 && i8 < n) {
                sHandle[l][i8] = handle;
                sCreated[l][i8] = created;
            }
            __syncthreads();
            if (c8 == 0 && i8 < n && !empty && repIdx != i8) {
                sHandle[l][i8] = sHandle[l][repIdx];
                sCreated[l][i8] = sCreated[l][repIdx];
            }
            __syncthreads();
            if (__ballot(oom) != 0)
                break;
        }
        if (__ballot(oom) != 0) {
            if (lane == 0) {
                EditStatus st {};
                st.oom = 1u;
                st.rootBefore = st.rootAfter = root;
                status[k] = st;
                *ws.poison = 1u;
            }
            break;
        }
        const uint32_t newRoot = sHandle[0][0];
        if (lane == 0) {
            EditStatus st {};
            st.done = 1u;
            st.applied = 1u;
            st.seqSpine = 1u;
            st.rootBefore = root;
            st.rootAfter = newRoot;
            st.leafCount = leafCount;
            status[k] = st;
        }
        root = newRoot;
        __syncthreads();
    }
    __syncthreads();
    if (lane == 0) {
        *rootPtr = root;
        *f.waveIdx += 1u;
    }
}

// ======================================================================== host

static uint32_t ceil_log2(uint64_t v)
{
    uint32_t p = 0;
    while ((1ull << p) < v)
        ++p;
    return p;
}

// Edits whose bounds span more than a quarter of the volume on an axis run
// on their own, so that one huge edit does not pull S up for the batch.
constexpr int kMinSplit = 2;

static uint64_t max_span(const Bounds& b)
{
    uint64_t m = 0;
    for (int a = 0; a < 3; ++a)
        m = std::max<uint64_t>(m, (uint64_t)(b.hi[a] - b.lo[a] + 1));
    return m;
}

static bool fusable(const svdag_ctx* ctx, const EditorDev& e)
{
    if (!(e.kind == EK_SPHERE_ADD || e.kind == EK_SPHERE_REMOVE || e.kind == EK_BOX_ADD || e.kind == EK_BOX_REMOVE
          || e.kind == EK_PAINT))
        return false;
    return (int)ctx->dag.levels - (int)ceil_log2(max_span(edit_bounds(ctx, e))) >= kMinSplit;
}

uint32_t plan_batch(svdag_ctx* ctx, const EditorDev* eds, uint32_t first, uint32_t n, std::vector<BatchStep>& steps,
                    const std::vector<uint8_t>& alone, uint32_t waveBase)
{
    steps.clear();
    const uint32_t D = ctx->dag.levels;
    uint64_t maxSpan = 0;
    for (uint32_t k = first; k < n; ++k)
        if (fusable(ctx, eds[k]) && !alone[k])
            maxSpan = std::max<uint64_t>(maxSpan, max_span(edit_bounds(ctx, eds[k])));
    int S = maxSpan ? (int)D - (int)ceil_log2(maxSpan) : 0;
    S = std::min<int>(S, (int)ctx->dag.leafLevel);
    if (S < 1) {
        for (uint32_t k = first; k < n; ++k)
            steps.push_back({ k, k + 1, false });
        return 0;
    }
    SeedDesc* seeds = reinterpret_cast<SeedDesc*>(ctx->hFused);
    uint2* waves = reinterpret_cast<uint2*>(seeds + ctx->batchCap);
    uint32_t nWaves = waveBase;
    const uint32_t sh = D - (uint32_t)S;
    std::vector<Bounds> members;
    uint32_t waveStart = first;
    bool open = false;
    auto close = [&](uint32_t end) {
        if (!open)
            return;
        steps.push_back({ waveStart, end, true });
        waves[nWaves++] = make_uint2(waveStart, end);
        members.clear();
        open = false;
    };
    for (uint32_t k = first; k < n; ++k) {
        if (!fusable(ctx, eds[k]) || alone[k]) {
            close(k);
            steps.push_back({ k, k + 1, false });
            continue;
        }
        const Bounds b = edit_bounds(ctx, eds[k]);
        SeedDesc sd {};
        int64_t cellLo[3], cellHi[3];
        for (int a = 0; a < 3; ++a) {
            const int64_t lo = b.lo[a] >> sh, hi = b.hi[a] >> sh;
            sd.lo[a] = (uint32_t)lo;
            sd.n[a] = (uint32_t)(hi - lo + 1);
            cellLo[a] = lo << sh;
            cellHi[a] = ((hi + 1) << sh) - 1;
        }
        seeds[k] = sd;
        bool conflict = false;
        for (const Bounds& m : members) {
            bool overlap = true;
            for (int a = 0; a < 3; ++a)
                overlap &= cellLo[a] <= m.hi[a] && m.lo[a] <= cellHi[a];
            if (overlap) {
                conflict = true;
                break;
            }
        }
        if (conflict || members.size() >= kMaxWave)
            close(k);
        if (!open) {
            open = true;
            waveStart = k;
        }
        members.push_back(b);
    }
    close(n);
    return (uint32_t)S;
}

// The wave's launch sequence.  levelItems == nullptr: fixed grids (every
// kernel walks its device-side count with a grid-stride loop), as captured
// into a graph that serves any wave of the same split level.
// part: 0 the whole wave, 1 its SVO build (wave_begin .. leaf level), 2
// its merge and spine.  The build only reads items the root reaches; the
// merge, which finds and inserts, waits for mergeAfter when given.
static int enqueue_wave(svdag_ctx* ctx, uint32_t S, const uint64_t* levelItems, uint32_t seedLanes,
                        hipEvent_t mergeAfter = nullptr, int part = 0)
{
    const DagDev& dag = ctx->dag;
    const hipStream_t st = ctx->stream;
    WsDev ws = ctx->ws;
    ws.edCount = ctx->dEdCount;
    ws.edFull = ctx->dEdFull;
    const FusedDev f { ctx->dWaves, ctx->dWaveIdx, ctx->dSeeds, ctx->dSeedWork, S, ctx->dWaveIdx + 1, ctx->dSpine };
    if (part != 2) {
        wave_begin<<<1, 256, 0, st>>>(ws, f, ctx->dStatusArr);
        fused_seed<<<(seedLanes + 255) / 256, 256, 0, st>>>(ws, dag, ctx->dEditors, f, ctx->dRoot);
    }
    if (levelItems) {
        SVDAG_TRY(launch_joint_levels(ctx, ws, ctx->dEditors, S, levelItems, ctx->maxBlocks, mergeAfter, part));
    } else {
        // Grids for any wave of this split level: a wave holds at most
        // kMaxWave edits of at most 8 level-S cells each, and every item has
        // at most 8 children, so level L holds at most 8 kMaxWave 8^(L-S)
        // items (the grid-stride loops cover the counts either way).
        uint64_t bound[kMaxLevels];
        uint64_t b = 8ull * kMaxWave;
        for (uint32_t L = 0; L < kMaxLevels; ++L) {
            bound[L] = L < S ? 0ull : b;
            if (L >= S)
                b = std::min<uint64_t>(b * 8ull, 1ull << 40);
        }
        SVDAG_TRY(launch_joint_levels(ctx, ws, ctx->dEditors, S, bound, 2048, mergeAfter, part));
    }
    if (part != 1) {
        fused_spine_par<<<1, kParThreads, 0, st>>>(ws, dag, ctx->dEditors, f, ctx->dRoot, ctx->dStatusArr,
                                                   ctx->dLevelArr);
        fused_spine<<<1, 64, 0, st>>>(ws, dag, ctx->dEditors, f, ctx->dRoot, ctx->dStatusArr, ctx->dLevelArr);
    }
    SVDAG_HIP(hipGetLastError());
    return SVDAG_OK;
}

void release_wave_graphs(svdag_ctx* ctx)
{
    for (auto& g : ctx->waveGraphs) {
        (void)hipGraphExecDestroy(g.exec);
        (void)hipGraphExecDestroy(g.merge);
    }
    ctx->waveGraphs.clear();
}

// One part of the wave's launch sequence captured and instantiated.
static int capture_wave_part(svdag_ctx* ctx, uint32_t S, int part, hipGraphExec_t& out)
{
    hipGraph_t graph = nullptr;
    SVDAG_HIP(hipStreamBeginCapture(ctx->stream, hipStreamCaptureModeThreadLocal));
    const int rc = enqueue_wave(ctx, S, nullptr, 8u * kMaxWave, nullptr, part);
    const hipError_t e = hipStreamEndCapture(ctx->stream, &graph);
    if (rc != SVDAG_OK) {
        if (graph)
            (void)hipGraphDestroy(graph);
        return rc;
    }
    SVDAG_HIP(e);
    const hipError_t ie = hipGraphInstantiate(&out, graph, nullptr, nullptr, 0);
    (void)hipGraphDestroy(graph);
    SVDAG_HIP(ie);
    return SVDAG_OK;
}

// The wave's graphs for split level S: its SVO build and its merge, replayed
// one after the other (so that the merge can wait for an event in between).
static int wave_graph(svdag_ctx* ctx, uint32_t S, hipGraphExec_t& build, hipGraphExec_t& merge)
{
    for (auto it = ctx->waveGraphs.begin(); it != ctx->waveGraphs.end();) {
        if (it->generation != ctx->bufferGeneration) {
            (void)hipGraphExecDestroy(it->exec);
            (void)hipGraphExecDestroy(it->merge);
            it = ctx->waveGraphs.erase(it);
            continue;
        }
        if (it->S == S && it->groupSize == ctx->groupSize) {
            build = it->exec;
            merge = it->merge;
            return SVDAG_OK;
        }
        ++it;
    }
    SVDAG_TRY(capture_wave_part(ctx, S, 1, build));
    const int rc = capture_wave_part(ctx, S, 2, merge);
    if (rc != SVDAG_OK) {
        (void)hipGraphExecDestroy(build);
        return rc;
    }
    ctx->waveGraphs.push_back({ S, ctx->groupSize, ctx->bufferGeneration, build, merge });
    return SVDAG_OK;
}

int launch_wave(svdag_ctx* ctx, const EditorDev* hEds, const BatchStep& step, uint32_t S, hipEvent_t mergeAfter)
{
    if (ctx->batchMode == SVDAG_BATCH_FUSED_GRAPH) {
        hipGraphExec_t build = nullptr, merge = nullptr;
        SVDAG_TRY(wave_graph(ctx, S, build, merge));
        SVDAG_HIP(hipGraphLaunch(build, ctx->stream));
        if (mergeAfter)
            SVDAG_HIP(hipStreamWaitEvent(ctx->stream, mergeAfter, 0));
        SVDAG_HIP(hipGraphLaunch(merge, ctx->stream));
        return SVDAG_OK;
    }
    uint64_t levelItems[kMaxLevels] {};
    for (uint32_t k = step.first; k < step.end; ++k) {
        const Bounds b = edit_bounds(ctx, hEds[k]);
        for (uint32_t L = S; L <= ctx->dag.leafLevel; ++L)
            levelItems[L] += level_bound(ctx, b, L);
    }
    return enqueue_wave(ctx, S, levelItems, 8u * (step.end - step.first), mergeAfter);
}

} // namespace svdag
