// hploc.hip - H-PLOC BVH2 construction (Benthin et al. 2024).
//
// Replaces BuildBVH2Kernel and its helpers (NexusBVH/src/Cuda/BinaryBuilder.cu:
// FindParentId/Delta 16-40, LoadIndices/StoreIndices 42-69,
// MergeClustersCreateBVH2Node 72-124, FindNearestNeighbor 127-163,
// PlocMerge 165-197, kernel 200-273).
//
// One lane per sorted primitive climbs the LBVH bottom-up (Apetrei 2014):
// the first child to reach a parent (atomic exchange on parent[]) retires,
// the second continues with the union range. Whenever a lane's range holds
// more than C primitives (or is the whole scene) its clusters are merged
// with PLOC++ by a group of lanes:
//   * NXB_MERGE_WAVE32: groups of 32 lanes, C = 16 -- the reference schedule.
//     A wave64 runs two independent groups, i.e. two merge tasks at once.
//   * NXB_MERGE_WAVE64: one group of 64 lanes, C = 32.
// The structure built depends only on the LBVH and the geometry, not on the
// order in which tasks run.
//
// Node ids without atomics: the reference takes ids from one global counter
// (BinaryBuilder.cu:85-91); on MI355X one hot address caps at ~10^8
// atomics/s, which would dominate the build. Here every cluster carries a
// representative (the smallest sorted position it covers; lists stay ordered
// by it). Merging clusters i < j retires rep(j); every position but 0 is
// retired exactly once, so id = n - 1 + rep(j) numbers the internal nodes
// bijectively onto [n, 2n-2], deterministically. The root goes to 2n-2; the
// node that retired position n-1 is parked in a spare slot (kMoved) and
// moved to the root's natural id when the root is made.
//
// Nearest neighbours: the reference's shuffle scheme yields, for cluster i,
// the first minimum of union areas (compared as uint32 bits) in the order
// i+1, i-1, i+2, i-2, ..., i+R, i-R. Here every lane writes its box to LDS and
// computes the R forward areas a(i, i+r); the backward ones a(i-r, i) come from
// lane i-r through lane shifts (nearest()). Unions use IEEE minimum/maximum,
// so a(i-r, i) == a(i, i-r) bit for bit.
//
// Batched builds (many independent meshes in one launch): the sorted keys
// are 64-bit (mesh << 30 | 30-bit Morton code) and each mesh's positions
// form a contiguous range [lo, lo + cnt). A merge task never leaves its mesh
// (the climb treats the mesh range as the whole array) and numbers its nodes
// with the mesh's own representatives: local id L = cnt - 1 + (rep - lo),
// stored at global id base + L. Leaves come first (leaf g = primitive g),
// then the internal nodes of mesh 0, 1, ...: base = N + lo - mesh - cnt. A
// single mesh is the case lo = 0, cnt = n, base = 0.
//
// Memory ordering across waves: everything one wave hands to another through
// a parent exchange (the cluster records and sizes a merge leaves) is
// written with agent-scope atomic stores and read with agent-scope atomic
// loads, which are coherent across XCDs without cache maintenance. A wave
// waits for its stores to complete before its next exchange; the reader's
// loads are issued only after its exchange returned. Leaves (written by an
// earlier kernel) use plain loads, and so do the internal nodes' stores,
// which only later kernels read (see create_node for the one exception).
//
// BVH8 builds of one mesh write each internal node as a 64-byte wide record
// (both children's boxes, ids and primitive counts) for the collapse, in
// place of its BVH2 node and size: at 28.1M triangles the records cost
// H-PLOC 0.25 ms and save the collapse 0.64 ms.
//
// What bounds it: up to about a million primitives the chain of merges to the
// root (a step is an exchange, key and record loads, 2 to 5 rounds of search
// and merge, and the stores' completion: some 3 us each); above, the vector
// units (60-70% busy) and requests to memory. Times in us before and after the
// last changes (search, merge rounds, loads and stores below):
//   BVH2, 12.7M 32-bit keys     1550 -> 1300    BVH8, 28.1M   3172 -> 2570
//   BVH8, 300K                   177 -> 159     BVH8, 2,003     86 -> 77
//   2,048 meshes, 19.7M         1890 -> 1690
#include <type_traits>

#include "device_common.h"
#include "nxb_internal.h"

namespace nxb {

// Two waves per block; each wave is persistent and works through its own
// range of sorted positions.
constexpr int kHplocThreads = 128;
constexpr int kHplocWaves = kHplocThreads / 64;
constexpr int kMaxRadius = 16;

constexpr uint32_t kInfBits = 0x7F800000u;  // areas at or above it as bits: infinite, NaN or negative
constexpr uint32_t kMoved = 0xFFFFFFFDu;  // temporary id of the node that retired n-1
constexpr uint32_t kRefill = 32;           // free lanes that make a wave start new positions
// Resident blocks per CU (6 waves per SIMD): at 28.1M primitives a BVH8 build's
// H-PLOC (tasks of 32 lanes, staged records, 80 registers) takes 2.60 ms with 12,
// 2.84 with 10, 3.04 with 8; 14 (72 registers) took 3.73. Tasks of 64 lanes, with
// 57 to 71 registers, keep the same limit: they were not measured with more.
constexpr uint32_t kHplocBlocksPerCu = kHplocMaxBlocksPerCu;
constexpr uint32_t kHplocMaxChunk = 1024;
// Primitives from which wide records go through the stage: below, its LDS round
// trip lengthens every merge round (1.1M primitives: 266 us direct, 284 staged;
// 2,003: 77 and 84); above, requests for memory bound the kernel (16M blobs:
// 1944 and 1709 us; uniform 1806 and 1436). The two meet at 2.5M to 4M. BVH2
// nodes, two stores of 16 bytes, gained nothing staged (12.7M: 1300 and 1298).
constexpr uint32_t kStagedPrims = 3u << 20;
constexpr uint32_t kHplocRegions = 8;         // XCDs of the chip
constexpr uint32_t kHplocCounterStride = 32;  // words between region counters (own 128-byte line)

// What a build keeps besides the BVH2: nothing more; the primitive count of
// every internal node; or a wide record in place of every internal node, stored
// by the lane that merges or (kKeepStaged) through LDS by four lanes each.
// Without counts a merge neither loads, carries nor stores them.
enum HplocKeep { kKeepNodes, kKeepSizes, kKeepRecords, kKeepStaged };

// Wide records of one merge round on their way to memory (kKeepStaged).
// Record r's quarter q stands at column (q + r / 4) % 4 of row r, so that 16
// lanes storing one quarter each cover all banks.
struct RecStage {
    uint4 q[32 * 4];
    uint32_t at[32];  // record index, or kInvalid: nothing to store
};
struct NoStage {};

template <int GW, HplocKeep KEEP>
struct HplocLds {
    // Cluster boxes by slot, in two planes (lx ly lz hx | hy hz) so that the
    // loads of neighbouring slots are free of bank conflicts (32 bytes a slot
    // made each take twice as long). Each group has GW slots and kMaxRadius
    // more that always hold a NaN box, so that the neighbour search reads
    // slot + r unconditionally.
    static constexpr uint32_t kStride = GW + kMaxRadius;
    float4 boxa[64 / GW * kStride];
    float2 boxb[64 / GW * kStride];
    uint2 id[64];                     // cluster id, representative
    uint32_t sz[64];                  // primitives in the cluster
    // in-wave hand-over of the parent exchange
    uint32_t mlane[64];               // slot & 63 -> a lane that posted it
    uint32_t mslot[64];               // lane -> slot it exchanges at rightwards this step, or kInvalid
    uint32_t mclaim[64];              // lane -> range end handed to it, or kInvalid
    std::conditional_t<KEEP == kKeepStaged, RecStage, NoStage> rec;
};

// Delta (BinaryBuilder.cu:16-40) between the sorted positions a and a + 1, their
// keys read by one load. 32-bit keys: the keys' bits, then the positions'.
// 64-bit keys: the keys', or of equal keys the positions'.
__device__ __forceinline__ uint64_t delta_next(const uint32_t* m, uint32_t a, uint32_t) {
    struct Pair { uint32_t k[2]; } p;
    __builtin_memcpy(&p, m + a, sizeof(p));
    return ((uint64_t)(p.k[0] ^ p.k[1]) << 32) | (a ^ (a + 1));
}
__device__ __forceinline__ uint64_t delta_next(const uint64_t* m, uint32_t a, uint32_t) {
    struct Pair { uint64_t k[2]; } p;
    __builtin_memcpy(&p, m + a, sizeof(p));
    const uint64_t d = p.k[0] ^ p.k[1];
    return d ? d : (uint64_t)(a ^ (a + 1));
}
// Batched keys (mesh << 30 | 30-bit code): the 32-bit Delta of the mesh alone,
// with positions local to the mesh (first position lo). Both keys lie in one
// mesh, so the mesh bits in their low words cancel in the XOR.
__device__ __forceinline__ uint64_t delta_next_batch(const uint64_t* m, uint32_t a, uint32_t lo) {
    struct Pair { uint32_t k[4]; } p;
    __builtin_memcpy(&p, m + a, sizeof(p));
    return ((uint64_t)(p.k[0] ^ p.k[2]) << 32) | ((a - lo) ^ (a + 1 - lo));
}

template <int GW, HplocKeep KEEP>
__device__ __forceinline__ void lds_put_box(HplocLds<GW, KEEP>& s, uint32_t i, const Box& b) {
    s.boxa[i] = make_float4(b.lx, b.ly, b.lz, b.hx);
    s.boxb[i] = make_float2(b.hy, b.hz);
}
template <int GW, HplocKeep KEEP>
__device__ __forceinline__ Box lds_get_box(const HplocLds<GW, KEEP>& s, uint32_t i) {
    float4 a = s.boxa[i];
    float2 c = s.boxb[i];
    Box b;
    b.lx = a.x; b.ly = a.y; b.lz = a.z; b.hx = a.w; b.hy = c.x; b.hz = c.y;
    return b;
}

// The value of the lane below; lane 0 takes lane 63's.
__device__ __forceinline__ uint32_t from_lane_below(uint32_t v) {
    return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x13C, 0xF, 0xF, true);
}

// FindNearestNeighbor (BinaryBuilder.cu:127-163) without branching on lanes:
// the reference's choice is the first minimum of the areas in the order
// forward a(i, i+1), backward a(i-1, i), a(i, i+2), a(i-2, i), ... Distances
// are taken from the largest to 1. Lane i + r receives a(i, i + r) as its
// backward area by r shifts of one lane: the running minimum `bb` and the lane
// `src` it came from move up a lane before distance r is taken in, so what is
// taken in at distance r ends r lanes up after the shift that follows distance
// 1. Taking an equal area at a smaller distance leaves each side's first
// minimum; between the sides an equal area goes to the smaller distance, then
// forward. The shifts are VALU moves (DPP), most of them folded into the
// minimum or the select that follows.
//
// Slots past the group's clusters hold NaN boxes, whose areas are NaN: as bits
// above every finite area, so with MASK == false nothing is compared against
// the group's end. A wave whose minima are all finite has the reference's
// choice; any other (areas that overflow) searches with MASK == true, where
// candidates that are not clusters of the group, or lie beyond the lane's own
// radius (the task's, uniform over its group), become kInvalid explicitly. A
// taken-in area's target is a slot of the same group, so nothing valid crosses
// into another group.
//
// Each backward area fetched through LDS and scanned in the reference's order
// took 8 LDS round trips and 78 registers; shifts of distances and a compare
// with the group's end per distance 26 VALU instructions per distance, now 20.
template <uint32_t UNROLL, bool MASK, int GW, HplocKeep KEEP>
__device__ __forceinline__ uint32_t nearest(const HplocLds<GW, KEEP>& s, const Box& own, uint32_t slot, uint32_t gl,
                                            int lim, uint32_t top, uint32_t& best) {
    uint32_t bf = kInvalid, bb = kInvalid, rf = 0, src = gl;
#pragma unroll UNROLL
    for (uint32_t r = top; r >= 1; --r) {
        uint32_t a = __float_as_uint(box_area(box_union(own, lds_get_box(s, slot + r))));
        if (MASK) a = (int)r < lim ? a : kInvalid;
        bb = min(from_lane_below(bb), a);
        asm("" : "+v"(bb));  // one use of the shifted value, so that the shift folds into the minimum
        src = from_lane_below(src);
        src = bb == a ? gl : src;
        bf = min(bf, a);
        rf = bf == a ? r : rf;
    }
    bb = from_lane_below(bb);
    src = from_lane_below(src);
    best = min(bf, bb);
    const bool fwd = bf < bb || (bf == bb && rf <= gl - src);
    return fwd ? gl + rf : src;
}

struct NodeStore {
    nxb_bvh2_node* nodes;
    bool wide_ok;              // node_count * 32 bytes fits a 32-bit buffer offset
    nxb_bvh2_node* moved;      // spare slot per mesh for kMoved
    uint32_t* moved_parent;    // per mesh: id of the node whose child is kMoved
    uint32_t* moved_size;      // per mesh: primitive count of the kMoved node
    uint32_t* nsize;           // kKeepSizes: primitive count of internal node id (index id - n)
    uint32_t n;                // leaves (all meshes)
    uint32_t node_count;       // nodes (all meshes): 2n - meshes
    uint4* rec8;               // kKeepRecords, kKeepStaged (one mesh): wide record of internal node id at id - n
    uint4* moved_rec;          // spare wide record for kMoved
};

// The mesh of a merge task: sorted positions [lo, lo + cnt), local node id L
// stored at base + L.
struct MeshCtx {
    uint32_t lo, cnt, mesh, base;
};

// 16-byte agent-coherent accesses. The relaxed agent-scope atomics of 64-bit
// words compile to plain loads/stores with the sc1 cache policy; the same
// policy on 16-byte buffer loads/stores moves 32 bytes in two memory
// transactions instead of four. A buffer covers its whole array: offsets past
// it read zeros and drop stores.
constexpr int kCachePolicySc1 = 16;
constexpr int kRawBufferWord3 = 0x00020000;
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));

// Cluster records. After a merge over a range, position p of the range
// holds one of the clusters the merge left (the first `count` positions):
// its box, id and representative. The parent merge reads them from their
// positions in one round of loads, without a second, dependent load of the
// boxes by id. A merged range's first cluster always holds the range's first
// leaf, so its representative is the range start; that record's
// representative word carries the cluster count instead.
// Records are two planes of 16 bytes per position (plane A: lx ly lz hx;
// plane B: hy hz id rep), so that the 16-byte access of consecutive lanes to
// consecutive positions covers whole 64-byte segments: one store instruction
// writes 16 lanes x 16 bytes contiguously instead of every other 16 bytes.
// Positions never merged have no record: their cluster is the leaf, read by
// id from the sorted permutation and the leaf nodes.
struct ClusterRec {
    Box b;
    uint32_t cid, rep;
};

__device__ __forceinline__ ClusterRec load_rec(const NodeStore& ns, const uint32_t* recs, uint32_t p) {
    ClusterRec r;
    if (ns.wide_ok) {
        const __amdgpu_buffer_rsrc_t ra =
            __builtin_amdgcn_make_buffer_rsrc(const_cast<uint32_t*>(recs), (short)0, (int)(ns.n * 16u), kRawBufferWord3);
        const __amdgpu_buffer_rsrc_t rb = __builtin_amdgcn_make_buffer_rsrc(
            const_cast<uint32_t*>(recs + (size_t)ns.n * 4), (short)0, (int)(ns.n * 16u), kRawBufferWord3);
        u32x4 a = __builtin_amdgcn_raw_buffer_load_b128(ra, (int)(p * 16u), 0, kCachePolicySc1);
        u32x4 c = __builtin_amdgcn_raw_buffer_load_b128(rb, (int)(p * 16u), 0, kCachePolicySc1);
        r.b.lx = __uint_as_float(a.x); r.b.ly = __uint_as_float(a.y); r.b.lz = __uint_as_float(a.z);
        r.b.hx = __uint_as_float(a.w); r.b.hy = __uint_as_float(c.x); r.b.hz = __uint_as_float(c.y);
        r.cid = c.z;
        r.rep = c.w;
    } else {
        const uint64_t* qa = reinterpret_cast<const uint64_t*>(recs + (size_t)p * 4);
        const uint64_t* qb = reinterpret_cast<const uint64_t*>(recs + (size_t)ns.n * 4 + (size_t)p * 4);
        uint64_t w0 = load_agent64(qa), w1 = load_agent64(qa + 1), w2 = load_agent64(qb), w3 = load_agent64(qb + 1);
        r.b.lx = __uint_as_float((uint32_t)w0); r.b.ly = __uint_as_float((uint32_t)(w0 >> 32));
        r.b.lz = __uint_as_float((uint32_t)w1); r.b.hx = __uint_as_float((uint32_t)(w1 >> 32));
        r.b.hy = __uint_as_float((uint32_t)w2); r.b.hz = __uint_as_float((uint32_t)(w2 >> 32));
        r.cid = (uint32_t)w3;
        r.rep = (uint32_t)(w3 >> 32);
    }
    return r;
}
__device__ __forceinline__ void store_rec(const NodeStore& ns, uint32_t* recs, uint32_t p, const Box& b, uint32_t cid,
                                          uint32_t rep) {
    if (ns.wide_ok) {
        const __amdgpu_buffer_rsrc_t ra =
            __builtin_amdgcn_make_buffer_rsrc(recs, (short)0, (int)(ns.n * 16u), kRawBufferWord3);
        const __amdgpu_buffer_rsrc_t rb =
            __builtin_amdgcn_make_buffer_rsrc(recs + (size_t)ns.n * 4, (short)0, (int)(ns.n * 16u), kRawBufferWord3);
        u32x4 a = {__float_as_uint(b.lx), __float_as_uint(b.ly), __float_as_uint(b.lz), __float_as_uint(b.hx)};
        u32x4 c = {__float_as_uint(b.hy), __float_as_uint(b.hz), cid, rep};
        __builtin_amdgcn_raw_buffer_store_b128(a, ra, (int)(p * 16u), 0, kCachePolicySc1);
        __builtin_amdgcn_raw_buffer_store_b128(c, rb, (int)(p * 16u), 0, kCachePolicySc1);
    } else {
        uint64_t* qa = reinterpret_cast<uint64_t*>(recs + (size_t)p * 4);
        uint64_t* qb = reinterpret_cast<uint64_t*>(recs + (size_t)ns.n * 4 + (size_t)p * 4);
        store_agent64(qa, (uint64_t)__float_as_uint(b.lx) | ((uint64_t)__float_as_uint(b.ly) << 32));
        store_agent64(qa + 1, (uint64_t)__float_as_uint(b.lz) | ((uint64_t)__float_as_uint(b.hx) << 32));
        store_agent64(qb, (uint64_t)__float_as_uint(b.hy) | ((uint64_t)__float_as_uint(b.hz) << 32));
        store_agent64(qb + 1, (uint64_t)cid | ((uint64_t)rep << 32));
    }
}

__device__ __forceinline__ void load_node_agent(const nxb_bvh2_node* p, uint64_t w[4]) {
    const uint64_t* q = reinterpret_cast<const uint64_t*>(p);
    w[0] = load_agent64(q); w[1] = load_agent64(q + 1); w[2] = load_agent64(q + 2); w[3] = load_agent64(q + 3);
}
__device__ __forceinline__ void store_words_agent(nxb_bvh2_node* p, const uint64_t w[4]) {
    uint64_t* q = reinterpret_cast<uint64_t*>(p);
    store_agent64(q, w[0]); store_agent64(q + 1, w[1]); store_agent64(q + 2, w[2]); store_agent64(q + 3, w[3]);
}

// Wide record of an internal node, read by the BVH8 collapse of the same
// build: words 0-5 the left child's box, 6-11 the right child's, then the
// left and right ids and their primitive counts (64 bytes, one segment).
__device__ __forceinline__ void rec8_words(const Box& lb, const Box& rb, uint32_t left, uint32_t right,
                                           uint32_t lsz, uint32_t rsz, uint4 q[4]) {
    q[0] = make_uint4(__float_as_uint(lb.lx), __float_as_uint(lb.ly), __float_as_uint(lb.lz), __float_as_uint(lb.hx));
    q[1] = make_uint4(__float_as_uint(lb.hy), __float_as_uint(lb.hz), __float_as_uint(rb.lx), __float_as_uint(rb.ly));
    q[2] = make_uint4(__float_as_uint(rb.lz), __float_as_uint(rb.hx), __float_as_uint(rb.hy), __float_as_uint(rb.hz));
    q[3] = make_uint4(left, right, lsz, rsz);
}
__device__ __forceinline__ void store_rec8_agent(uint4* p, const uint4 q[4]) {
    uint64_t* w = reinterpret_cast<uint64_t*>(p);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        store_agent64(w + 2 * i, (uint64_t)q[i].x | ((uint64_t)q[i].y << 32));
        store_agent64(w + 2 * i + 1, (uint64_t)q[i].z | ((uint64_t)q[i].w << 32));
    }
}

// Creates the node merging clusters (left, right) with box b and size
// primitives (lb, rb, lsz, rsz: the two clusters' boxes and primitive
// counts, for the wide record). Returns its id. A wide record goes to row
// `row` of the stage; store_records() stores it.
template <HplocKeep KEEP, typename Lds>
__device__ __forceinline__ uint32_t create_node(Lds& s, uint32_t row, const NodeStore& ns, const MeshCtx& mc,
                                                const Box& b, uint32_t left, uint32_t right, uint32_t right_rep,
                                                uint32_t size, bool root_step, uint32_t* flags, const Box& lb,
                                                const Box& rb, uint32_t lsz, uint32_t rsz) {
    if constexpr (KEEP == kKeepStaged) s.rec.at[row] = kInvalid;
    const uint32_t n = ns.n;
    const uint32_t local = mc.cnt - 1 + (right_rep - mc.lo);
    const uint32_t root_local = 2 * mc.cnt - 2;
    const uint32_t natural = mc.base + local;
    uint32_t id = root_step ? mc.base + root_local : (local == root_local ? kMoved : natural);
    if (local > root_local || natural >= ns.node_count) { atomic_or_agent(flags, kFlagBadIndex); return 0; }
    uint32_t* moved_parent = ns.moved_parent + mc.mesh;
    if constexpr (KEEP >= kKeepRecords) {
        // BVH8 build: the wide record stands for the internal node (its box
        // is the union of the children's, its size their sum); the same
        // parking of kMoved, on records.
        if (root_step && local != root_local) {
            const uint64_t* mr = reinterpret_cast<const uint64_t*>(ns.moved_rec);
            uint64_t* dst = reinterpret_cast<uint64_t*>(ns.rec8 + 4ull * (natural - n));
#pragma unroll
            for (int i = 0; i < 8; ++i) dst[i] = load_agent64(mr + i);
            if (left == kMoved) {
                left = natural;
            } else if (right == kMoved) {
                right = natural;
            } else {
                const uint32_t p = load_agent(moved_parent);
                if (p < ns.node_count && p >= n) {
                    // the ids are the record's words 12 and 13
                    uint64_t* q = reinterpret_cast<uint64_t*>(ns.rec8 + 4ull * (p - n) + 3);
                    const uint64_t lr = load_agent64(q);
                    uint32_t pl = (uint32_t)lr, pr = (uint32_t)(lr >> 32);
                    if (pl == kMoved) pl = natural;
                    else if (pr == kMoved) pr = natural;
                    else atomic_or_agent(flags, kFlagBadIndex);
                    store_agent64(q, (uint64_t)pl | ((uint64_t)pr << 32));
                } else {
                    atomic_or_agent(flags, kFlagBadIndex);
                }
            }
        } else if (left == kMoved || right == kMoved) {
            store_agent(moved_parent, id);
        }
        uint4 q[4];
        rec8_words(lb, rb, left, right, lsz, rsz, q);
        if (id == kMoved) {
            store_rec8_agent(ns.moved_rec, q);
        } else if (left == kMoved || right == kMoved) {
            store_rec8_agent(ns.rec8 + 4ull * (id - n), q);
        } else {
            if constexpr (KEEP == kKeepStaged) {
                s.rec.at[row] = id - n;
#pragma unroll
                for (uint32_t i = 0; i < 4; ++i) s.rec.q[4 * row + ((i + row / 4) & 3)] = q[i];
            } else {
                uint4* p = ns.rec8 + 4ull * (id - n);
                p[0] = q[0]; p[1] = q[1]; p[2] = q[2]; p[3] = q[3];
            }
        }
        return id;
    }
    nxb_bvh2_node* moved = ns.moved + mc.mesh;
    uint32_t* moved_size = ns.moved_size + mc.mesh;
    if (root_step && local != root_local) {
        // the parked node takes the root's natural id
        uint64_t w[4];
        load_node_agent(moved, w);
        store_words_agent(ns.nodes + natural, w);
        if constexpr (KEEP == kKeepSizes) ns.nsize[natural - n] = load_agent(moved_size);
        if (left == kMoved) {
            left = natural;
        } else if (right == kMoved) {
            right = natural;
        } else {
            uint32_t p = load_agent(moved_parent);
            if (p < ns.node_count) {
                uint64_t* q = reinterpret_cast<uint64_t*>(ns.nodes + p) + 3;
                uint64_t lr = load_agent64(q);
                uint32_t pl = (uint32_t)lr, pr = (uint32_t)(lr >> 32);
                if (pl == kMoved) pl = natural;
                else if (pr == kMoved) pr = natural;
                else atomic_or_agent(flags, kFlagBadIndex);
                store_agent64(q, (uint64_t)pl | ((uint64_t)pr << 32));
            } else {
                atomic_or_agent(flags, kFlagBadIndex);
            }
        }
    } else if (left == kMoved || right == kMoved) {
        store_agent(moved_parent, id);
    }
    // No wave of this kernel reads a node back, except the root step, which
    // rewrites the child ids of the node that points at the parked one: that
    // node is stored agent-coherently; every other node is a plain store
    // (whole lines in L2, written back when the kernel ends).
    if (id == kMoved) store_node_agent(moved, 0, b, left, right);
    else if (left == kMoved || right == kMoved) store_node_agent(ns.nodes, id, b, left, right);
    else store_node(ns.nodes, id, b, left, right);
    if constexpr (KEEP == kKeepSizes) {
        if (id == kMoved) store_agent(moved_size, size);
        else ns.nsize[id - n] = size;
    }
    return id;
}

// Stores the staged records of a round (`count` rows), a 64-byte segment per
// four lanes. Stored by the lane that made it, a record took four stores of 16
// bytes to as many segments as lanes.
__device__ __forceinline__ void store_records(const RecStage& st, const NodeStore& ns, uint32_t count) {
    const uint32_t lane = __lane_id();
    for (uint32_t r = lane / 4; r - lane / 4 < count; r += 16) {
        const uint32_t at = r < count ? st.at[r] : kInvalid;
        const uint4 v = st.q[4 * r + (lane & 3)];
        if (at != kInvalid) ns.rec8[4ull * at + ((lane - r / 4) & 3)] = v;
    }
}

// Per-segment radius policy: a merge task over sorted positions
// [l_start, r_end) within one segment's span takes the radius of the segment
// of l_start; wider tasks (the upper levels of the tree) and table entries 0
// take the fixed radius.
__device__ __forceinline__ uint32_t radius_for(const RadiusParams& rp, uint32_t l_start, uint32_t r_end) {
    uint32_t r = rp.radius;
    if (rp.table && r_end - l_start <= (1u << rp.seg_log2)) {
        uint32_t seg = l_start >> rp.seg_log2;
        if (seg < rp.table_len) {
            uint32_t t = rp.table[seg];
            if (t >= 1) r = t;
        }
    }
    return r > (uint32_t)kMaxRadius ? (uint32_t)kMaxRadius : r;
}

// PlocMerge for the group this lane belongs to. All lanes of the wave call
// it together; a group with has_task == false does nothing.
//   GW  : lanes per group (32 or 64), C = GW / 2
//   gl  : lane index within the group; gbase: first lane of the group
//   gmask: 64-bit mask of the group's lanes
template <int GW, HplocKeep KEEP>
__device__ __forceinline__ void ploc_merge(HplocLds<GW, KEEP>& s, bool has_task, uint32_t l_start, uint32_t split,
                                           uint32_t r_end, bool final, uint32_t gl, uint32_t gbase,
                                           uint64_t gmask, const uint32_t* cluster, uint32_t* recs, uint32_t* csizes,
                                           const NodeStore& ns, const MeshCtx& mc, const RadiusParams& rp,
                                           uint32_t* flags) {
    constexpr uint32_t C = GW / 2;
    const uint32_t bbase = gbase / GW * HplocLds<GW, KEEP>::kStride;  // the group's first box slot
    const float nan = __builtin_nanf("");
    uint32_t num;

    // LoadIndices (BinaryBuilder.cu:42-57): the left child's clusters, then
    // the right child's. A child of at most C primitives was never merged:
    // its clusters are its leaves in sorted order (one primitive each), read
    // through the sorted permutation. A merged child left its clusters'
    // records at the front of its range, their count in the first record.
    // Lanes [0, C) read the left child's clusters and lanes [C, 2C) the
    // right child's, all at once; the valid entries are then compacted in
    // that order through LDS, where the group's other slots get NaN boxes.
    {
        const bool lhalf = gl < C;
        const uint32_t k = lhalf ? gl : gl - C;
        const uint32_t first = lhalf ? l_start : split;
        const uint32_t span = lhalf ? split - l_start : r_end - split;
        const bool merged = span > C;
        const uint32_t pos = first + k;
        bool v = has_task && k < min(span, C);
        // Leaves (written by an earlier kernel: plain loads) and records are
        // both in flight at once; one after the other cost a task that has
        // both kinds a third memory latency.
        uint32_t leaf = 0, lsz = 1u;
        ClusterRec r = {};
        if (v && !merged) leaf = cluster[pos];
        if (v && merged) {
            r = load_rec(ns, recs, pos);
            if constexpr (KEEP != kKeepNodes) lsz = load_agent(&csizes[pos]);
        }
        Box lb = {};
        if (v && !merged) {
            if (leaf >= ns.n) { atomic_or_agent(flags, kFlagBadIndex); leaf = 0; }
            lb = load_box(ns.nodes, leaf);
        }
        const uint32_t lcid = merged ? r.cid : leaf;
        // the half's first lane holds the child's cluster count (merged child)
        const uint32_t count = (uint32_t)__shfl((int)r.rep, (int)(gbase + (lhalf ? 0u : C)));
        const uint32_t lrep = merged ? (k == 0 ? first : r.rep) : pos;
        v = v && (!merged || k < count) && lcid != kInvalid;
        if (v && lcid - ns.node_count < kMoved - ns.node_count) atomic_or_agent(flags, kFlagBadIndex);
        Box b = merged ? r.b : lb;
        const uint64_t vm = ballot(v) & gmask;
        num = (uint32_t)__popcll(vm);
        const uint32_t rank = mask_rank(vm), dst = v ? rank : num + gl - rank;
        b.lx = v ? b.lx : nan;
        lds_put_box(s, bbase + dst, b);
        s.id[gbase + dst] = make_uint2(lcid, lrep);
        if constexpr (KEEP != kKeepNodes) s.sz[gbase + dst] = lsz;
        wave_lds_sync();
    }
    const uint32_t slot = bbase + gl;
    Box own = lds_get_box(s, slot);
    uint32_t cid = s.id[gbase + gl].x, rep = s.id[gbase + gl].y, sz = 0;
    if constexpr (KEEP != kKeepNodes) sz = s.sz[gbase + gl];

    const uint32_t threshold = final ? 1u : C;
    // The radius is uniform over a group. The search runs to the larger of the
    // wave's two, unrolled for 8; only where a table gave two tasks different
    // ones (plain_r == 0) does each lane mask the distances past its own (two of
    // 22 instructions a distance). Masked whenever there was a table: learned
    // radii at 1.9M primitives 508 -> 473 us with the policy's kernels, one task
    // a wave 560 -> 511.
    uint32_t R = min(rp.radius, (uint32_t)kMaxRadius), r_wave = R, plain_r = R;
    if (rp.table) {
        R = has_task ? radius_for(rp, l_start, r_end) : 0u;
        const uint32_t r0 = __builtin_amdgcn_readfirstlane(R), r1 = GW == 64 ? r0 : __builtin_amdgcn_readlane(R, 32);
        r_wave = max(r0, r1);
        plain_r = min(r0, r1) != 0 && r0 != r1 ? 0u : r_wave;
    }

    // The group's first num slots hold own/id/sz of its clusters here and after
    // every compaction below, its other slots NaN boxes. All lanes of the wave
    // take part in every round (lane shifts read them); a group that is done
    // (num <= threshold) merges nothing.
    for (;;) {
        const bool run = num > threshold && gl < num;
        if (!ballot(run)) break;
        // ---- FindNearestNeighbor (BinaryBuilder.cu:127-163) ----
        uint32_t nn, best;
        if (plain_r == 8) nn = nearest<8, false>(s, own, slot, gl, 0, 8u, best);
        else if (plain_r) nn = nearest<2, false>(s, own, slot, gl, 0, plain_r, best);
        else nn = nearest<2, true>(s, own, slot, gl, (int)R + 1, r_wave, best);
        if (ballot(run && best >= kInfBits)) {
            nn = nearest<1, true>(s, own, slot, gl, min((int)num - (int)gl, (int)R + 1), r_wave, best);
            if (best == kInvalid) nn = kInvalid;
        }

        // ---- MergeClustersCreateBVH2Node (BinaryBuilder.cu:72-124) ----
        // the neighbour's neighbour, from its lane
        const uint32_t theirs = (uint32_t)__builtin_amdgcn_ds_bpermute((int)((gbase + nn) * 4u), (int)nn);
        const bool mutual = run && nn < (uint32_t)GW && theirs == gl;
        const bool merge = mutual && gl < nn;
        const uint64_t merges = ballot(merge);
        const uint32_t mcount = (uint32_t)__popcll(merges & gmask);
        const bool root_step = final && num - mcount == 1;
        if (merge) {
            const Box nb = lds_get_box(s, bbase + nn);
            const uint2 nid = s.id[gbase + nn];
            uint32_t nsz = 0;
            if constexpr (KEEP != kKeepNodes) nsz = s.sz[gbase + nn];
            const Box ob = own;
            own = box_union(own, nb);
            cid = create_node<KEEP>(s, mask_rank(merges), ns, mc, own, cid, nid.x, nid.y, sz + nsz, root_step, flags,
                                    ob, nb, sz, nsz);
            sz += nsz;
        }
        const bool valid = gl < num && (merge || !mutual);
        const uint64_t vm = ballot(valid) & gmask;
        num -= mcount;
        const uint32_t rank = mask_rank(vm), dst = valid ? rank : num + gl - rank;
        own.lx = valid ? own.lx : nan;
        wave_lds_sync();
        lds_put_box(s, bbase + dst, own);
        s.id[gbase + dst] = make_uint2(cid, rep);
        if constexpr (KEEP != kKeepNodes) s.sz[gbase + dst] = sz;
        wave_lds_sync();
        own = lds_get_box(s, slot);
        cid = s.id[gbase + gl].x;
        rep = s.id[gbase + gl].y;
        if constexpr (KEEP != kKeepNodes) sz = s.sz[gbase + gl];
        if constexpr (KEEP == kKeepStaged) store_records(s.rec, ns, (uint32_t)__popcll(merges));
    }

    // StoreIndices (BinaryBuilder.cu:59-69), as records: the num clusters
    // left, the count in the first record's representative word.
    if (gl < num) {
        store_rec(ns, recs, l_start + gl, own, cid, gl == 0 ? num : rep);
        if constexpr (KEEP != kKeepNodes) store_agent(&csizes[l_start + gl], sz);
    }
}

template <typename K, int GW, bool BATCH, HplocKeep KEEP>
__global__ __launch_bounds__(kHplocThreads) __attribute__((amdgpu_waves_per_eu(6))) void k_hploc(const K* __restrict__ keys, const uint32_t* cluster,
                                                         uint32_t* recs, uint32_t* csizes, uint32_t* parent,
                                                         NodeStore ns, const uint32_t* __restrict__ mesh_lo,
                                                         uint32_t meshes, RadiusParams rp, uint32_t* flags,
                                                         uint32_t* next_chunk, uint32_t first, uint32_t chunk) {
    __shared__ HplocLds<GW, KEEP> lds[kHplocWaves];
    constexpr uint32_t C = GW / 2;
    const uint32_t tid = threadIdx.x;
    HplocLds<GW, KEEP>& s = lds[tid >> 6];
    const uint32_t lane = tid & 63;
    const uint32_t n = ns.n;

    // Persistent waves. The sorted positions are cut into kHplocRegions
    // regions, one per XCD (blocks are dispatched to XCDs round-robin, so
    // block b runs on XCD b % kHplocRegions and the merges of a region stay
    // in one L2). A wave starts positions in order, a batch of free lanes at
    // a time, so that it keeps most lanes busy even though most climbs end
    // after a step or two. Its first `first` positions are fixed by its
    // index in the region; then it takes chunks of `chunk` positions from
    // the region's counter (dynamic chunks keep the waves level where the
    // merge cost varies along the array, e.g. with per-segment radii), and
    // once its region is used up and all its lanes are idle, from the next
    // regions'.
    const uint32_t region_len = (((n + kHplocRegions - 1) / kHplocRegions) + 63u) & ~63u;
    uint32_t region = blockIdx.x % kHplocRegions, tried = 0;
    uint32_t next = 0, end = 0;  // the wave's current chunk (wave-uniform)
    bool more = true;            // chunks may be left (wave-uniform)
    bool have_pf = false;        // lane 0's pf holds the next counter value of the home region
    uint32_t pf = 0;
    {
        const uint32_t j = (blockIdx.x / kHplocRegions) * kHplocWaves + (tid >> 6);
        const uint64_t lo_r = (uint64_t)region * region_len;
        const uint64_t hi_r = min((uint64_t)n, lo_r + region_len);
        const uint64_t c = lo_r + (uint64_t)j * first;
        if (c < hi_r) {
            next = (uint32_t)c;
            end = (uint32_t)min(hi_r, c + first);
        }
    }

    uint32_t left = 0, right = 0, split = 0;
    bool active = false;
    bool pending = false;        // a merge's stores may be in flight (wave-uniform)
    uint32_t lo = 0, hi = n - 1, mesh = 0;  // this lane's mesh [lo, hi] (the whole array for a single build)

    s.mlane[lane] = lane;
    s.mclaim[lane] = kInvalid;
    for (uint32_t i = lane; i < 64 / GW * HplocLds<GW, KEEP>::kStride; i += 64)
        s.boxa[i] = make_float4(__builtin_nanf(""), 0.0f, 0.0f, 0.0f);
    wave_lds_sync();

    uint32_t g, gl, gbase;
    uint64_t gmask;
    if (GW == 32) {
        g = lane >> 5;
        gl = lane & 31;
        gbase = g * 32;
        gmask = g ? 0xFFFFFFFF00000000ull : 0x00000000FFFFFFFFull;
    } else {
        g = 0;
        gl = lane;
        gbase = 0;
        gmask = ~0ull;
    }

    for (;;) {
        // Start the next positions on the free lanes (at least kRefill of
        // them, or all lanes free).
        const uint64_t free_lanes = ballot(!active);
        const uint32_t nfree = (uint32_t)__popcll(free_lanes);
        while (more && next >= end && (tried == 0 ? nfree >= kRefill : nfree == 64u)) {
            // the region's dynamic chunks start after the first positions of
            // its waves
            const uint32_t waves_r =
                gridDim.x > region ? ((gridDim.x - region + kHplocRegions - 1) / kHplocRegions) * kHplocWaves : 0u;
            const uint64_t lo_r = (uint64_t)region * region_len;
            const uint64_t hi_r = min((uint64_t)n, lo_r + region_len);
            uint32_t* ctr = &next_chunk[region * kHplocCounterStride];
            const uint64_t base = lo_r + (uint64_t)waves_r * first;
            uint32_t c = 0;
            if (have_pf) {
                c = pf;  // lane 0's, taken with the stores of the refill that used up the last chunk
                have_pf = false;
            } else if (lane == 0) {
                // When stealing, a plain read first: the counter only grows,
                // so a region it shows used up is used up, and idle waves add
                // no atomics to the counters still in use.
                c = tried ? load_agent(ctr) : 0u;
                if (base + c < hi_r) c = atomic_add_agent(ctr, chunk);
            }
            c = __builtin_amdgcn_readfirstlane(c);
            const uint64_t pos = base + c;
            if (pos < hi_r) {
                next = (uint32_t)pos;
                end = (uint32_t)min(hi_r, pos + chunk);
            } else if (++tried == kHplocRegions) {
                more = false;
            } else {
                region = (region + 1) % kHplocRegions;
            }
        }
        if (next < end && (nfree >= kRefill || free_lanes == ~0ull)) {
            const uint32_t i = next + mask_rank(free_lanes);
            if (!active && i < end) {
                left = right = i;
                split = 0;
                active = true;
                if constexpr (BATCH) {
                    const uint32_t m = (uint32_t)((uint64_t)keys[i] >> 30);
                    if (m < meshes) {
                        mesh = m;
                        lo = mesh_lo[m];
                        hi = mesh_lo[m + 1] - 1;
                    } else {
                        atomic_or_agent(flags, kFlagBadIndex);
                        active = false;
                    }
                }
            }
            next = min(end, next + nfree);
            if (next >= end && more && tried == 0 && !have_pf) {
                // this batch uses up the chunk: take the next one now, so
                // that the atomic's latency hides behind the climb
                if (lane == 0) pf = atomic_add_agent(&next_chunk[region * kHplocCounterStride], chunk);
                have_pf = true;
            }
        }
        if (!ballot(active)) {
            if (!more && next >= end) break;
            continue;
        }
        bool to_right = false;
        if (active) {
            const auto d = [&](uint32_t at) {
                if constexpr (BATCH) return delta_next_batch(keys, at, lo);
                else return delta_next(keys, at, 0u);
            };
            to_right = left == lo || (right != hi && d(right) < d(left - 1));
        }
        // Two lanes of this wave that reach the same parent slot in this step
        // (the range ending at it going right, the one starting after it
        // going left) meet in LDS instead of exchanging through memory: the
        // left-going lane hands its range end over and stops. Each slot has
        // one candidate per side, so a lane found through the slot hash is
        // the partner iff it posted the same slot; every other lane takes
        // the exchange. The wave's stores are complete (the wait just below),
        // so the continuing lane reads the partner's clusters as it
        // would after an exchange. Skipped (wave-uniform) unless the wave
        // has lanes going both ways, as on the serial climb near the root.
        if (pending) {
            pending = false;
            wait_memory_ops();
        }
        if (ballot(active && to_right) != 0 && ballot(active && !to_right) != 0) {
            const uint32_t slot = to_right ? right : left - 1;
            s.mslot[lane] = (active && to_right) ? slot : kInvalid;
            if (active && to_right) s.mlane[slot & 63u] = lane;
            wave_lds_sync();
            if (active && !to_right) {
                const uint32_t p = s.mlane[slot & 63u] & 63u;
                if (s.mslot[p] == slot) {
                    s.mclaim[p] = right;
                    active = false;
                }
            }
            wave_lds_sync();
        }
        bool handed = false;
        if (active && to_right) {
            const uint32_t c = s.mclaim[lane];
            if (c != kInvalid) {
                s.mclaim[lane] = kInvalid;
                split = right + 1;
                right = c;
                handed = true;
            }
        }
        if (active && !handed) {
            const uint32_t at = to_right ? right : left - 1;
            uint32_t prev = atomic_xchg_agent(&parent[at], to_right ? left : right);
            if (prev == kInvalid) {
                active = false;
            } else {
                if (prev > hi || prev < lo) {
                    atomic_or_agent(flags, kFlagBadIndex);
                    prev = to_right ? hi : lo;
                }
                split = at + 1;
                if (to_right) right = prev;
                else left = prev;
            }
        }
        uint32_t size = right - left + 1;
        bool final = active && size == hi - lo + 1;
        uint64_t tasks = ballot(active && (size > C || final));
        if (!tasks) continue;

        compiler_barrier();  // cluster/node reads stay after the exchanges
        while (tasks) {
            uint32_t t0 = (uint32_t)__builtin_ctzll(tasks);
            tasks &= tasks - 1;
            uint32_t t1 = 64;
            if (GW == 32 && tasks) {
                t1 = (uint32_t)__builtin_ctzll(tasks);
                tasks &= tasks - 1;
            }
            uint32_t my = (g == 0) ? t0 : t1;
            bool has = my < 64;
            const uint32_t tsel = (g && t1 < 64) ? t1 : t0;  // lane whose task this group runs
            uint32_t l0 = __builtin_amdgcn_readlane(left, t0), s0 = __builtin_amdgcn_readlane(split, t0);
            uint32_t r0 = __builtin_amdgcn_readlane(right, t0);
            uint32_t f0 = __builtin_amdgcn_readlane((uint32_t)final, t0);
            uint32_t l1 = l0, s1 = s0, r1 = r0, f1 = f0;
            if (t1 < 64) {
                l1 = __builtin_amdgcn_readlane(left, t1);
                s1 = __builtin_amdgcn_readlane(split, t1);
                r1 = __builtin_amdgcn_readlane(right, t1);
                f1 = __builtin_amdgcn_readlane((uint32_t)final, t1);
            }
            uint32_t tl = g ? l1 : l0, ts = g ? s1 : s0, tr = g ? r1 : r0;
            bool tf = (g ? f1 : f0) != 0;
            MeshCtx tm{0u, n, 0u, 0u};
            if constexpr (BATCH) {
                // the task's mesh (lanes of the other group run another task)
                tm.lo = __shfl(lo, (int)tsel);
                tm.cnt = __shfl(hi, (int)tsel) + 1 - tm.lo;
                tm.mesh = __shfl(mesh, (int)tsel);
                tm.base = n + tm.lo - tm.mesh - tm.cnt;
            }
            ploc_merge<GW, KEEP>(s, has, tl, ts, tr + 1, tf, gl, gbase, gmask, cluster, recs, csizes, ns, tm, rp,
                                 flags);
        }
        // Merge outputs are agent-scope atomic stores; they must be complete
        // before this wave's next parent exchange hands the subtree over. The
        // wait stands after the next step's key loads, whose latency it covers.
        pending = true;
    }
}

// One resident block per slot of the chip (persistent waves): at most
// kHplocBlocksPerCu per CU and no more than the kernel's occupancy allows (a
// block that is not resident would start its fixed positions late), fewer
// when the input gives a wave less than 64 positions. The kernel is a template
// argument, so that each has its own occupancy here: kernels of one signature share
// a type.
template <auto KERNEL>
static uint32_t hploc_grid(uint32_t n, uint32_t blocks_per_cu) {
    static const int per_cu = [] {  // the same on every gfx950 device
        int blocks = 0;
        const hipError_t e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&blocks, KERNEL, kHplocThreads, 0);
        return e == hipSuccess && blocks > 0 ? blocks : 1;
    }();
    const uint32_t want = blocks_per_cu ? min(blocks_per_cu, kHplocBlocksPerCu) : kHplocBlocksPerCu;
    const uint32_t resident = device_cu_count() * min((uint32_t)per_cu, want);
    const uint32_t most = (n + kHplocThreads - 1) / kHplocThreads;
    return most < resident ? most : resident;
}

// Positions per wave: three quarters of a wave's share fixed, the rest in
// chunks of an eighth of a share (multiples of 64, chunks at most
// kHplocMaxChunk). At 1.1M primitives a half share fixed was 15% slower
// (chunk grabs on the critical path) and at 28.1M a full share fixed was 5%
// slower (waves uneven).
struct HplocChunks {
    uint32_t first, chunk;
};
static HplocChunks hploc_chunks(uint32_t n, uint32_t grid) {
    const uint64_t share = (n + (uint64_t)grid * kHplocWaves - 1) / ((uint64_t)grid * kHplocWaves);
    auto round64 = [](uint64_t v) { return v < 64 ? 64ull : (v + 63) & ~63ull; };
    const uint64_t first = round64(share * 3 / 4), chunk = round64(share / 8);
    return HplocChunks{(uint32_t)first, (uint32_t)(chunk > kHplocMaxChunk ? kHplocMaxChunk : chunk)};
}

template <typename K, int GW, bool BATCH, HplocKeep KEEP>
static hipError_t launch_hploc_kernel(const K* keys, uint32_t* cluster, uint32_t n, const uint32_t* mesh_lo,
                                      uint32_t meshes, const NodeStore& ns, RadiusParams rp, uint32_t blocks_per_cu,
                                      HplocScratch sc, hipStream_t s) {
    const auto kernel = k_hploc<K, GW, BATCH, KEEP>;
    const uint32_t grid = hploc_grid<k_hploc<K, GW, BATCH, KEEP>>(n, blocks_per_cu);
    const HplocChunks cp = hploc_chunks(n, grid);
    hipLaunchKernelGGL(kernel, dim3(grid), dim3(kHplocThreads), 0, s, keys, cluster, sc.recs, sc.csizes, sc.parent,
                       ns, mesh_lo, meshes, rp, sc.flags, sc.next_chunk, cp.first, cp.chunk);
    return hipGetLastError();
}

template <typename K, bool BATCH, HplocKeep KEEP>
static hipError_t launch_hploc_mode(const void* keys, uint32_t* cluster, uint32_t n, const uint32_t* mesh_lo,
                                    uint32_t meshes, const NodeStore& ns, uint32_t merge_mode, RadiusParams rp,
                                    uint32_t blocks_per_cu, HplocScratch sc, hipStream_t s) {
    const K* k = static_cast<const K*>(keys);
    return merge_mode == NXB_MERGE_WAVE64
               ? launch_hploc_kernel<K, 64, BATCH, KEEP>(k, cluster, n, mesh_lo, meshes, ns, rp, blocks_per_cu, sc, s)
               : launch_hploc_kernel<K, 32, BATCH, KEEP>(k, cluster, n, mesh_lo, meshes, ns, rp, blocks_per_cu, sc, s);
}

hipError_t launch_hploc(const void* keys, uint32_t key_bits, uint32_t* cluster, uint32_t n, nxb_bvh2_node* nodes,
                        uint32_t merge_mode, RadiusParams rp, uint32_t blocks_per_cu, HplocScratch sc,
                        hipStream_t s) {
    if (n == 0) return hipSuccess;
    if (sc.nsize) return hipErrorInvalidValue;  // no caller wants them for one mesh
    const bool rec = sc.rec8 && sc.moved_rec;
    const NodeStore ns{nodes, 2ull * n - 1 < (1ull << 27), sc.moved, sc.moved_parent, sc.moved_size, nullptr, n,
                       2 * n - 1, sc.rec8, sc.moved_rec};
    const auto launch = key_bits == 32
                            ? (!rec                ? launch_hploc_mode<uint32_t, false, kKeepNodes>
                               : n < kStagedPrims  ? launch_hploc_mode<uint32_t, false, kKeepRecords>
                                                   : launch_hploc_mode<uint32_t, false, kKeepStaged>)
                            : (!rec                ? launch_hploc_mode<uint64_t, false, kKeepNodes>
                               : n < kStagedPrims  ? launch_hploc_mode<uint64_t, false, kKeepRecords>
                                                   : launch_hploc_mode<uint64_t, false, kKeepStaged>);
    return launch(keys, cluster, n, nullptr, 1u, ns, merge_mode, rp, blocks_per_cu, sc, s);
}

hipError_t launch_hploc_batch(const uint64_t* keys, uint32_t* cluster, uint32_t n, const uint32_t* mesh_lo,
                              uint32_t meshes, nxb_bvh2_node* nodes, uint32_t merge_mode, RadiusParams rp,
                              uint32_t blocks_per_cu, HplocScratch sc, hipStream_t s) {
    if (n == 0) return hipSuccess;
    const NodeStore ns{nodes, 2ull * n - meshes < (1ull << 27), sc.moved, sc.moved_parent, sc.moved_size, sc.nsize, n,
                       2 * n - meshes, nullptr, nullptr};
    const auto launch =
        sc.nsize ? launch_hploc_mode<uint64_t, true, kKeepSizes> : launch_hploc_mode<uint64_t, true, kKeepNodes>;
    return launch(keys, cluster, n, mesh_lo, meshes, ns, merge_mode, rp, blocks_per_cu, sc, s);
}

}  // namespace nxb
