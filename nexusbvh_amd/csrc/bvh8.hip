// bvh8.hip - BVH2 -> compressed 8-wide BVH (Ylitie et al. 2017).
//
// Replaces BuildBVH8Kernel and its helpers (NexusBVH/src/Cuda/WideConverter.cu:
// GetCost 25-30, GreedyAssignment 106-153, CreateBVH8Node 156-206,
// CreateBVH8SingleLeaf 209-222, kernel 225-414).
//
// Per BVH8 node: collapse up to 8 BVH2 descendants (push both children of
// the current node, the smaller-area one into the popped slot, then pop the
// highest-index inner slot), greedy octant slot assignment, then 8-bit
// child-box quantization against the node's box.
//
// Scheduling (gfx950): persistent waves. A work item is one BVH8 *inner*
// node; its slot index is its BVH8 node index, so work[k] holds the BVH2
// node that BVH8 node k is built from. Lanes take node indices in increasing
// order from an atomic counter and wait on work[k] until the parent (always
// a smaller index, already taken by a running lane) publishes it with an
// agent-scope store. The producing lane keeps its first inner child and
// builds it next (depth-first, no publish/poll round trip on that path),
// marking the slot kTaken so whoever drew it moves on. Leaf children are
// written to primIdx by the parent directly, so leaves cost no work item.
// Leaf ranges in primIdx are fixed top-down from subtree primitive counts
// (no atomics). Node indices and completion share one 64-bit counter
// (finished << 32 | allocated), updated once per wave iteration for all its
// lanes (a hot address takes only ~10^8 atomics/s on MI355X); waiting lanes
// stop when finished == allocated. Waits are bounded by spin_limit; hitting
// it sets the timeout flag and exits.
#include "device_common.h"
#include "nxb_internal.h"

namespace nxb {

constexpr int kBvh8Threads = 256;
constexpr uint32_t kNoSlot = 0xFFFFFFFFu;
// work[k] value of a node that its producer builds itself (depth-first).
constexpr uint32_t kTaken = 0xFFFFFFFEu;

__device__ __forceinline__ uint32_t nib(uint32_t x, uint32_t i) { return (x >> (4 * i)) & 0xFu; }
__device__ __forceinline__ uint32_t bits_below(uint32_t x, uint32_t i) {
    return (uint32_t)__popc(x & ((1u << i) - 1u));
}
// CeilLog2 / InvPow2 (BuilderUtils.h:335-347).
__device__ __forceinline__ uint32_t ceil_log2(float x) {
    uint32_t ix = __float_as_uint(x);
    return ((ix >> 23) & 0xFFu) + ((ix & 0x7FFFFFu) != 0);
}
__device__ __forceinline__ float inv_pow2(uint32_t e) { return __uint_as_float((uint32_t)(254 - (int)e) << 23); }

// GetCost (WideConverter.cu:25-30): exact +-1 products, FMA-neutral.
__device__ __forceinline__ float slot_cost(uint32_t s, float ox, float oy, float oz) {
    float sx = ((s >> 2) & 1) ? -1.0f : 1.0f;
    float sy = ((s >> 1) & 1) ? -1.0f : 1.0f;
    float sz = (s & 1) ? -1.0f : 1.0f;
    return sx * ox + sy * oy + sz * oz;
}

__device__ __forceinline__ uint32_t with_nib(uint32_t x, uint32_t i, uint32_t v) {
    return (x & ~(0xFu << (4 * i))) | (v << (4 * i));
}

constexpr uint32_t kAuctionMaxBids = 4096;   // per epsilon phase
constexpr uint32_t kAuctionMaxPhases = 16;

// Auction slot assignment (the reference's compiled-out alternative to the
// greedy one, WideConverter.cu:52-102 with its cost table at 336-361;
// Bertsekas' auction algorithm with epsilon scaling, theta = 8). Children
// bid for slots with reward cost(c, s) - price(s); the winner's price rises
// by (best - second best) + epsilon and an outbid child bids again. Bounded:
// at most kAuctionMaxPhases phases of kAuctionMaxBids bids; children left
// unassigned (or non-finite costs) take the first free slots in child order.
// ox/oy/oz: (parent min + max) - (child min + max) per child.
__device__ __forceinline__ uint32_t auction_assign(const Box& pb, const float ox[8], const float oy[8],
                                                   const float oz[8], uint32_t n) {
    const float max_dim = fmaxf(fmaxf(pb.hx - pb.lx, pb.hy - pb.ly), pb.hz - pb.lz);
    const float scale = (max_dim == 0.0f ? 0.0f : 10.0f / max_dim) * 0.5f;
    float cx[8], cy[8], cz[8];
    float max_cost = -3.402823466e+38f;
#pragma unroll
    for (uint32_t k = 0; k < 8; ++k) {
        cx[k] = ox[k] * scale;
        cy[k] = oy[k] * scale;
        cz[k] = oz[k] * scale;
        const float cost = fabsf(cx[k]) + fabsf(cy[k]) + fabsf(cz[k]);
        if (k < n && cost > max_cost) max_cost = cost;
    }
    float prices[8];
#pragma unroll
    for (uint32_t s = 0; s < 8; ++s) prices[s] = 0.0f;
    const float threshold = 1.0f / (float)n;
    float epsilon = fmaxf(max_cost, threshold);
    uint32_t assign = 0xFFFFFFFFu;
    bool done = !(epsilon < INFINITY);  // non-finite costs: first free slots
    for (uint32_t phase = 0; !done && epsilon >= threshold && phase < kAuctionMaxPhases; ++phase) {
        assign = 0xFFFFFFFFu;
        uint32_t bidders = 0x76543210u, left = n;
        for (uint32_t bids = 0; left > 0; ++bids) {
            if (bids == kAuctionMaxBids) { done = true; break; }
            const uint32_t c = nib(bidders, --left);
            float ccx = 0.0f, ccy = 0.0f, ccz = 0.0f;
#pragma unroll
            for (uint32_t k = 0; k < 8; ++k)
                if (k == c) { ccx = cx[k]; ccy = cy[k]; ccz = cz[k]; }
            float win = -3.402823466e+38f, second = -3.402823466e+38f;
            uint32_t ws = 0xFu;
#pragma unroll
            for (uint32_t t = 0; t < 8; ++t) {
                const float reward = slot_cost(t, ccx, ccy, ccz) - prices[t];
                if (reward > win) { second = win; win = reward; ws = t; }
                else if (reward > second) second = reward;
            }
            if (ws == 0xFu) { done = true; break; }
            float raise = (win - second) + epsilon;
            uint32_t prev = 0xFu;
#pragma unroll
            for (uint32_t t = 0; t < 8; ++t)
                if (t == ws) { prices[t] = prices[t] + raise; prev = nib(assign, t); }
            assign = with_nib(assign, ws, c);
            if (prev != 0xFu) bidders = with_nib(bidders, left++, prev);
        }
        epsilon *= 0.125f;
    }
    // children without a slot (bid limit, non-finite costs): first free slots
    for (uint32_t k = 0; k < n; ++k) {
        bool placed = false;
        for (uint32_t t = 0; t < 8; ++t) placed |= nib(assign, t) == k;
        if (placed) continue;
        for (uint32_t t = 0; t < 8; ++t)
            if (nib(assign, t) == 0xFu) { assign = with_nib(assign, t, k); break; }
    }
    return assign;
}

__device__ __forceinline__ uint32_t q_floor(float v) { return ((uint32_t)floorf(v)) & 0xFFu; }
__device__ __forceinline__ uint32_t q_ceil(float v) { return ((uint32_t)ceilf(v)) & 0xFFu; }

// Boxes of the children of the node each lane collapses, in LDS (child t of
// lane i at [t][i]): loaded once during the collapse, read again by the slot
// assignment and the quantization without another global load.
struct ChildBoxes {
    float4 a[8][kBvh8Threads];  // lx, ly, lz, hx
    float2 b[8][kBvh8Threads];  // hy, hz
};
__device__ __forceinline__ void put_child_box(ChildBoxes& cb, uint32_t t, uint32_t tid, const Box& b) {
    cb.a[t][tid] = make_float4(b.lx, b.ly, b.lz, b.hx);
    cb.b[t][tid] = make_float2(b.hy, b.hz);
}
__device__ __forceinline__ Box get_child_box(const ChildBoxes& cb, uint32_t t, uint32_t tid) {
    const float4 a = cb.a[t][tid];
    const float2 c = cb.b[t][tid];
    Box b;
    b.lx = a.x; b.ly = a.y; b.lz = a.z; b.hx = a.w; b.hy = c.x; b.hz = c.y;
    return b;
}

// CreateBVH8Node (WideConverter.cu:156-206) into 20 words; empty slots keep
// all-zero meta and quantization bytes.
__device__ __forceinline__ void write_bvh8_node(nxb_bvh8_node* out, uint32_t k, const Box& pb, const ChildBoxes& cbx,
                                                uint32_t tid, uint32_t child_base, uint32_t prim_base,
                                                uint32_t assign, uint32_t inner_mask, uint32_t leaf_mask) {
    const float qstep = 1.0f / 255.0f;
    uint32_t e0 = ceil_log2((pb.hx - pb.lx) * qstep) & 0xFFu;
    uint32_t e1 = ceil_log2((pb.hy - pb.ly) * qstep) & 0xFFu;
    uint32_t e2 = ceil_log2((pb.hz - pb.lz) * qstep) & 0xFFu;
    float ix = inv_pow2(e0), iy = inv_pow2(e1), iz = inv_pow2(e2);
    uint32_t meta[2] = {0, 0}, qlx[2] = {0, 0}, qly[2] = {0, 0}, qlz[2] = {0, 0};
    uint32_t qhx[2] = {0, 0}, qhy[2] = {0, 0}, qhz[2] = {0, 0};
#pragma unroll
    for (uint32_t i = 0; i < 8; ++i) {
        uint32_t a = nib(assign, i);
        if (a == 0xFu) continue;
        uint32_t m;
        if (inner_mask & (1u << i)) m = (1u << 5) | (24 + i);
        else m = (1u << 5) | bits_below(leaf_mask, i);
        const Box cb = get_child_box(cbx, a, tid);
        const uint32_t w = i >> 2, sh = 8 * (i & 3);
        meta[w] |= m << sh;
        qlx[w] |= q_floor((cb.lx - pb.lx) * ix) << sh;
        qly[w] |= q_floor((cb.ly - pb.ly) * iy) << sh;
        qlz[w] |= q_floor((cb.lz - pb.lz) * iz) << sh;
        qhx[w] |= q_ceil((cb.hx - pb.lx) * ix) << sh;
        qhy[w] |= q_ceil((cb.hy - pb.ly) * iy) << sh;
        qhz[w] |= q_ceil((cb.hz - pb.lz) * iz) << sh;
    }
    uint4* o = reinterpret_cast<uint4*>(out + k);
    o[0] = make_uint4(__float_as_uint(pb.lx), __float_as_uint(pb.ly), __float_as_uint(pb.lz),
                      e0 | (e1 << 8) | (e2 << 16) | (inner_mask << 24));
    o[1] = make_uint4(child_base, prim_base, meta[0], meta[1]);
    o[2] = make_uint4(qlx[0], qlx[1], qly[0], qly[1]);
    o[3] = make_uint4(qlz[0], qlz[1], qhx[0], qhx[1]);
    o[4] = make_uint4(qhy[0], qhy[1], qhz[0], qhz[1]);
}

// Collapse + slot assignment of one inner BVH2 node (WideConverter.cu:284-379).
struct Collapsed {
    Box pb;              // the node's box
    uint32_t child[8];   // BVH2 children in push order
    uint32_t cleft[8];   // their left fields (kInvalid for a leaf)
    uint32_t cright[8];  // their right fields (primitive index of a leaf)
    uint32_t count;
    uint32_t assign;     // nibble s = child index in slot s, 0xF = empty
    uint32_t im, lm;     // inner / leaf slot masks
};

// GreedyAssignment (WideConverter.cu:106-153), or the auction, of the
// c.count collapsed children; inner: their inner-child bits by child index.
__device__ __forceinline__ void assign_slots(Collapsed& c, const ChildBoxes& cbx, uint32_t tid, uint32_t slot_mode,
                                             uint32_t inner) {
    const uint32_t count = c.count;
    const Box& pb = c.pb;
    const float pcx = pb.lx + pb.hx, pcy = pb.ly + pb.hy, pcz = pb.lz + pb.hz;
    uint32_t assign = 0xFFFFFFFFu;
    if (slot_mode == NXB_SLOT_AUCTION) {
        float ox[8], oy[8], oz[8];
#pragma unroll
        for (uint32_t k = 0; k < 8; ++k) {
            ox[k] = oy[k] = oz[k] = 0.0f;
            if (k < count) {
                const Box cb = get_child_box(cbx, k, tid);
                ox[k] = pcx - (cb.lx + cb.hx);
                oy[k] = pcy - (cb.ly + cb.hy);
                oz[k] = pcz - (cb.lz + cb.hz);
            }
        }
        assign = auction_assign(pb, ox, oy, oz, count);
    }
#pragma unroll
    for (uint32_t k = 0; k < 8; ++k) {
        if (slot_mode == NXB_SLOT_AUCTION || k >= count) break;
        const Box cb = get_child_box(cbx, k, tid);
        float ox = pcx - (cb.hx + cb.lx), oy = pcy - (cb.hy + cb.ly), oz = pcz - (cb.hz + cb.lz);
        float best_cost = -3.402823466e+38f;
        uint32_t best = 0xFu, first_free = 0xFu;
#pragma unroll
        for (uint32_t s = 0; s < 8; ++s) {
            if (nib(assign, s) != 0xFu) continue;
            if (first_free == 0xFu) first_free = s;
            float cost = slot_cost(s, ox, oy, oz);
            if (cost > best_cost) { best_cost = cost; best = s; }
        }
        if (best == 0xFu) best = first_free;
        assign = (assign & ~(0xFu << (4 * best))) | (k << (4 * best));
    }
    uint32_t im = 0, lm = 0;
#pragma unroll
    for (uint32_t s = 0; s < 8; ++s) {
        uint32_t a = nib(assign, s);
        if (a == 0xFu) continue;
        uint32_t bit = (inner >> a) & 1u;
        im |= bit << s;
        lm |= (bit ^ 1u) << s;
    }
    c.assign = assign;
    c.im = im;
    c.lm = lm;
}

// have_lr: x's children (gl, gr) come with the work item, so their loads do
// not wait for x's (whose box is needed only after the expansion).
__device__ __forceinline__ bool collapse_node(const nxb_bvh2_node* b2, uint32_t node_count, uint32_t x,
                                              Collapsed& c, ChildBoxes& cbx, uint32_t tid, uint32_t slot_mode,
                                              bool have_lr = false, uint32_t gl = 0, uint32_t gr = 0) {
    uint32_t xl, xr;
    load_node(b2, x, c.pb, xl, xr);
    if (have_lr) {
        xl = gl;
        xr = gr;
    }
    if (xl == kInvalid) return false;  // a leaf is never a work item
#pragma unroll
    for (int t = 0; t < 8; ++t) { c.child[t] = 0; c.cright[t] = 0; c.cleft[t] = 0; }
    uint32_t inner = 0, count = 0;
    int msb = 0;
    uint32_t lr0 = xl, lr1 = xr;
    for (;;) {
        if (lr0 >= node_count || lr1 >= node_count) return false;
        Box b0, b1;
        uint32_t l0, r0, l1, r1;
        load_node(b2, lr0, b0, l0, r0);
        load_node(b2, lr1, b1, l1, r1);
        bool first_is_1 = !(box_area(b0) < box_area(b1));
        uint32_t ia = (uint32_t)msb, ib = count + 1;
        uint32_t na = first_is_1 ? lr1 : lr0, nb = first_is_1 ? lr0 : lr1;
        uint32_t la = first_is_1 ? l1 : l0, lb = first_is_1 ? l0 : l1;
        uint32_t ra = first_is_1 ? r1 : r0, rb = first_is_1 ? r0 : r1;
        put_child_box(cbx, ia, tid, first_is_1 ? b1 : b0);
        put_child_box(cbx, ib, tid, first_is_1 ? b0 : b1);
#pragma unroll
        for (uint32_t t = 0; t < 8; ++t) {
            if (t == ia) { c.child[t] = na; c.cleft[t] = la; c.cright[t] = ra; }
            if (t == ib) { c.child[t] = nb; c.cleft[t] = lb; c.cright[t] = rb; }
        }
        if (la != kInvalid) inner |= 1u << ia;
        if (lb != kInvalid) inner |= 1u << ib;
        count += 2;
        msb = inner ? 31 - __clz(inner) : -1;
        if (msb < 0 || count == 8) break;
        inner &= ~(1u << msb);
        --count;
#pragma unroll
        for (uint32_t t = 0; t < 8; ++t)
            if (t == (uint32_t)msb) { lr0 = c.cleft[t]; lr1 = c.cright[t]; }
    }
    c.count = count;
    assign_slots(c, cbx, tid, slot_mode, inner);
    return true;
}

// The wide record of a BVH8 build's internal node: both children's boxes, ids
// (a leaf's is its primitive index, below n) and primitive counts.
__device__ __forceinline__ void load_rec8(const uint4* rec, uint32_t i, Box& l, Box& r, uint32_t& li, uint32_t& ri,
                                          uint32_t& ls, uint32_t& rs) {
    const uint4* p = rec + 4ull * i;
    const uint4 q0 = p[0], q1 = p[1], q2 = p[2], q3 = p[3];
    l.lx = __uint_as_float(q0.x); l.ly = __uint_as_float(q0.y); l.lz = __uint_as_float(q0.z);
    l.hx = __uint_as_float(q0.w); l.hy = __uint_as_float(q1.x); l.hz = __uint_as_float(q1.y);
    r.lx = __uint_as_float(q1.z); r.ly = __uint_as_float(q1.w); r.lz = __uint_as_float(q2.x);
    r.hx = __uint_as_float(q2.y); r.hy = __uint_as_float(q2.z); r.hz = __uint_as_float(q2.w);
    li = q3.x; ri = q3.y; ls = q3.z; rs = q3.w;
}

// Publishes the inner children of BVH8 node k (the first one is kept by this
// lane, depth-first), writes its leaves to primIdx and writes the node.
// Primitive ranges are fixed top-down: the subtree of a node owns a range of
// primIdx as long as its primitive count; the node's own leaves take the
// front, then each inner child (in slot order) takes a range of its size.
// Primitive counts of a node's inner children, per output slot (0 for leaf
// and free slots).
__device__ __forceinline__ void load_child_sizes(const Collapsed& c, const uint32_t* nsize, uint32_t n,
                                                 uint32_t node_count, uint32_t sz[8]) {
#pragma unroll
    for (uint32_t s = 0; s < 8; ++s) {
        sz[s] = 0;
        const uint32_t a = nib(c.assign, s);
        if (a == 0xFu || !(c.im & (1u << s))) continue;
        uint32_t ch = 0;
#pragma unroll
        for (uint32_t t = 0; t < 8; ++t)
            if (t == a) ch = c.child[t];
        if (ch >= n && ch < node_count) sz[s] = nsize[ch - n];
    }
}

__device__ __forceinline__ void emit_node(const ChildBoxes& cbx, uint32_t tid, const Collapsed& c, uint32_t k,
                                          uint32_t child_base, uint32_t prim_base, uint32_t leaf_count,
                                          const uint32_t sz[8], nxb_bvh8_node* out, uint32_t* prim_idx,
                                          uint32_t n, uint32_t capacity, uint64_t* work, uint32_t* flags,
                                          uint32_t& keep_slot, uint32_t& keep_x, uint32_t& keep_base) {
    keep_slot = kNoSlot;
    keep_x = kInvalid;
    keep_base = 0;
    uint32_t next_base = prim_base + leaf_count;
#pragma unroll
    for (uint32_t s = 0; s < 8; ++s) {
        uint32_t a = nib(c.assign, s);
        if (a == 0xFu) continue;
        uint32_t ch = 0, pr = 0;
#pragma unroll
        for (uint32_t t = 0; t < 8; ++t)
            if (t == a) { ch = c.child[t]; pr = c.cright[t]; }
        if (c.im & (1u << s)) {
            uint32_t slot = child_base + bits_below(c.im, s);
            const uint32_t size = sz[s];
            if (slot >= capacity || size < 2 || next_base + size > n) {
                atomic_or_agent(flags, kFlagBadIndex);
            } else if (keep_slot == kNoSlot) {
                keep_slot = slot;
                keep_x = ch;
                keep_base = next_base;
                store_agent64(&work[slot], ((uint64_t)next_base << 32) | kTaken);
            } else {
                store_agent64(&work[slot], ((uint64_t)next_base << 32) | ch);
            }
            next_base += size;
        } else {
            uint32_t p = prim_base + bits_below(c.lm, s);
            if (p < n) prim_idx[p] = pr;
            else atomic_or_agent(flags, kFlagBadIndex);
        }
    }
    write_bvh8_node(out, k, c.pb, cbx, tid, child_base, leaf_count ? prim_base : 0u, c.assign, c.im, c.lm);
}

// The value N lanes back in the same row of 16 (row_shr:N), 0 at its start and
// from inactive lanes: never inside a branch or a ?: arm.
template <int N>
__device__ __forceinline__ uint32_t lane_back(uint32_t v) {
    return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x110 + N, 0xF, 0xF, true);
}

// Inclusive sum over the 64 lanes of a wave, by lane shifts of the vector units
// (rows of 16, then the rows' totals); six shuffles through LDS took six round
// trips. All lanes of the wave are active.
__device__ __forceinline__ uint32_t wave_inclusive_sum(uint32_t v) {
    v += lane_back<1>(v);
    v += lane_back<2>(v);
    v += lane_back<4>(v);
    v += lane_back<8>(v);
    v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x142, 0xA, 0xF, false);  // row_bcast:15 to rows 1, 3
    v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x143, 0xC, 0xF, false);  // row_bcast:31 to rows 2, 3
    return v;
}

// Barrier of the block for data in LDS alone: global stores in flight, which
// only later kernels read, are not waited for as __syncthreads() does.
__device__ __forceinline__ void lds_barrier() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// n leaves; node_count = 2n - 1 for one BVH2, 2n - (trees) for a forest
// whose roots seed work[0..trees).
template <uint32_t SLOT>
__global__ __launch_bounds__(kBvh8Threads) void k_bvh8(const nxb_bvh2_node* __restrict__ b2, uint32_t n,
                                                       uint32_t node_count, nxb_bvh8_node* __restrict__ out,
                                                       uint32_t* prim_idx, uint32_t capacity, uint64_t* work,
                                                       unsigned long long* ctr, uint32_t* grab,
                                                       const uint32_t* __restrict__ nsize, uint32_t* flags,
                                                       uint32_t spin_limit) {
    __shared__ ChildBoxes cbx;
    const uint32_t tid = threadIdx.x;
    if (n == 1) {
        // CreateBVH8SingleLeaf (WideConverter.cu:209-222).
        if (blockIdx.x == 0 && tid == 0) {
            Box pb = load_box(b2, 0);
            put_child_box(cbx, 0, tid, pb);
            prim_idx[0] = 0;
            write_bvh8_node(out, 0, pb, cbx, tid, 0, 0, 0xFFFFFFF0u, 0u, 1u);
        }
        return;
    }
    uint32_t slot = kNoSlot;  // BVH8 node this lane builds next
    uint32_t x = kInvalid;    // its BVH2 node, once known
    uint32_t pbase = 0;       // first primIdx entry of its subtree
    bool done = false;
    uint32_t spins = 0, idle = 0, witer = 0;
    for (;;) {
        if (!ballot(!done)) break;
        bool need = !done && slot == kNoSlot;
        uint64_t nm = ballot(need);
        if (nm) {
            uint32_t leader = (uint32_t)__builtin_ctzll(nm);
            uint32_t base = 0;
            if (lane_id() == leader) base = atomic_add_agent(grab, (uint32_t)__popcll(nm));
            base = __shfl(base, (int)leader);
            if (need) slot = base + mask_rank(nm);
        }
        bool waiting = false;
        if (!done && x == kInvalid) {
            if (slot >= capacity) {
                done = true;
            } else {
                uint64_t v = load_agent64(&work[slot]);
                uint32_t lo = (uint32_t)v;
                if (lo == kTaken) {
                    slot = kNoSlot;  // its producer builds it
                    spins = 0;
                } else if (lo != kInvalid) {
                    x = lo;
                    pbase = (uint32_t)(v >> 32);
                } else {
                    waiting = true;
                    if (++spins >= spin_limit) {
                        atomic_or_agent(flags, kFlagTimeout);
                        done = true;
                        waiting = false;
                    }
                }
            }
        }
        // Completion: every allocated node finished (one load per wave).
        ++witer;
        if ((witer & 7u) == 0 && ballot(waiting)) {
            unsigned long long cv = 0;
            if (lane_id() == 0) cv = __hip_atomic_load(ctr, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            uint32_t lo = __shfl((uint32_t)cv, 0), hi = __shfl((uint32_t)(cv >> 32), 0);
            if (waiting && lo == hi) done = true;
        }
        bool have = !done && x != kInvalid;
        if (!ballot(have)) {
            if (!ballot(!done && slot == kNoSlot)) {
                // the whole wave waits on unpublished nodes
                if (++idle > 8) __builtin_amdgcn_s_sleep(24);
                else __builtin_amdgcn_s_sleep(2);
            }
            continue;
        }
        idle = 0;
        Collapsed c;
        bool ok = false;
        if (have) {
            spins = 0;
            ok = x < node_count && collapse_node(b2, node_count, x, c, cbx, tid, SLOT);
            if (!ok) atomic_or_agent(flags, kFlagBadIndex);
        }
        // One atomic per wave iteration: allocate the inner children of all
        // lanes and count their nodes as finished.
        uint32_t ic = ok ? (uint32_t)__popc(c.im) : 0u;
        uint32_t packed = (ic << 16) | (have ? 1u : 0u);
        uint32_t incl = wave_inclusive_sum(packed);
        uint32_t total = __shfl(incl, 63);
        uint32_t excl = incl - packed;
        unsigned long long old = 0;
        if (lane_id() == 0)
            old = __hip_atomic_fetch_add(ctr, ((unsigned long long)(total & 0xFFFFu) << 32) | (total >> 16),
                                         __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        uint32_t node_base = __shfl((uint32_t)old, 0);
        if (have) {
            uint32_t ks = kNoSlot, kx = kInvalid, kb = 0;
            if (ok) {
                uint32_t child_base = ic ? node_base + (excl >> 16) : 0u;
                uint32_t sz[8];
                load_child_sizes(c, nsize, n, node_count, sz);
                emit_node(cbx, tid, c, slot, child_base, pbase, c.count - ic, sz, out, prim_idx, n, capacity, work,
                          flags, ks, kx, kb);
            }
            slot = ks;
            x = kx;
            pbase = kb;
        }
    }
}

// ---- level-synchronous construction (single builds) -------------------------
//
// One kernel per BVH8 level: every node of the level is collapsed by one
// lane; a block allocates the inner children of all its lanes with one
// atomic add on the next level's counter (block scan of the counts). Level
// l holds the ids [base_l, base_l + cnt[l]) with base_l = cnt[0] + ... +
// cnt[l-1], so a level's kernel finds its range from counters that earlier
// kernels completed, and no lane ever waits on another (no polling, no spin
// limit). The total node count is the sum of the counters.
//
// Inputs: a whole build (one mesh) collapses the wide records its H-PLOC
// wrote instead of BVH2 nodes: one aligned 64-byte load per expansion (both
// children's boxes, ids and primitive counts) replaces two 32-byte node
// loads (leaves in input order, a line each) and the size lookups. At 28.1M
// triangles this took the collapse from 1.94 to 1.31 ms. The stage entry
// point and batched forests collapse BVH2 nodes.
//
// What bounds it: every record is read once and every node written once (2.2 GB
// at 28.1M triangles), 64 bytes at a time all over memory, by lanes that wait
// for one record before they ask for the next. The children are kept in
// registers and a node is put together in LDS (36 KB a block, four blocks per
// CU; the children's boxes in LDS took 48 KB, three blocks, and 2,970 vector
// instructions per wave, now 2,400), and four lanes fetch a record in one
// request. Collapse of 28.1M triangles 1323 -> 1278 -> 1165 us, 12.7M 828 -> 770
// -> 722, 2.9M 338 -> 308 -> 293; queued children put in order before their
// store, 1% less, was not worth its lines.
constexpr uint32_t kMaxLevels = kBvh8LevelWords - 1;  // BVH8 levels; each consumes at least one BVH2 level

// Exclusive scan over a 256-thread block; *total gets the block sum.
template <bool LDS_ONLY = false>
__device__ __forceinline__ uint32_t block_scan_256(uint32_t v, uint32_t* tmp, uint32_t* total) {
    const uint32_t tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
    const uint32_t incl = wave_inclusive_sum(v);
    if (lane == 63) tmp[w] = incl;
    if (LDS_ONLY) lds_barrier();
    else __syncthreads();
    uint32_t before = 0, all = 0;
#pragma unroll
    for (uint32_t k = 0; k < kBvh8Threads / 64; ++k) {
        const uint32_t t = tmp[k];
        if (k < w) before += t;
        all += t;
    }
    if (LDS_ONLY) lds_barrier();
    else __syncthreads();
    *total = all;
    return before + incl - v;
}

// The children of the node a lane collapses, in registers: box, id and primitive
// count (0: a leaf). Only ever indexed by constants.
struct Kids {
    Box box[8];
    uint32_t id[8], prims[8];
};

// Records idx of the wave's lanes (kInvalid: none), four lanes fetching each:
// straight to LDS, 16 bytes a lane, so that a record is one 64-byte request. Its
// own lane fetching it made four of as many lines as lanes. buf: 260 words of
// the wave's own; record of lane 4i + j at 65 j + 4 i (conflict-free). All lanes
// of the wave take part.
template <uint32_t J>
__device__ __forceinline__ uint32_t of_quad(uint32_t v) {  // the value of the four's lane J
    return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, J * 0x55, 0xF, 0xF, true);
}
__device__ __forceinline__ void fetch16(const uint4* from, uint4* buf) {
    __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)from,
                                     (__attribute__((address_space(3))) void*)buf, 16, 0, 0);
}
template <uint32_t J>
__device__ __forceinline__ void fetch_rec(const uint4* rec, uint32_t idx, uint4* buf) {
    const uint32_t of = of_quad<J>(idx);
    if (of != kInvalid) fetch16(rec + 4ull * of + (__lane_id() & 3u), buf + 65 * J);
}
__device__ __forceinline__ void load_rec8_quads(const uint4* rec, uint32_t idx, uint4* buf, Box& l, Box& r,
                                                uint32_t& li, uint32_t& ri, uint32_t& ls, uint32_t& rs) {
    fetch_rec<0>(rec, idx, buf);
    fetch_rec<1>(rec, idx, buf);
    fetch_rec<2>(rec, idx, buf);
    fetch_rec<3>(rec, idx, buf);
    wait_memory_ops();
    wave_lds_sync();
    const uint32_t lane = __lane_id();
    const uint4* p = buf + 65 * (lane & 3u) + 4 * (lane >> 2);
    const uint4 q0 = p[0], q1 = p[1], q2 = p[2], q3 = p[3];
    wave_lds_sync();
    l.lx = __uint_as_float(q0.x); l.ly = __uint_as_float(q0.y); l.lz = __uint_as_float(q0.z);
    l.hx = __uint_as_float(q0.w); l.hy = __uint_as_float(q1.x); l.hz = __uint_as_float(q1.y);
    r.lx = __uint_as_float(q1.z); r.ly = __uint_as_float(q1.w); r.lz = __uint_as_float(q2.x);
    r.hx = __uint_as_float(q2.y); r.hy = __uint_as_float(q2.z); r.hz = __uint_as_float(q2.w);
    li = q3.x; ri = q3.y; ls = q3.z; rs = q3.w;
}

// Collapse of internal node x (record x - n), in the push/pop order of
// collapse_node: the pair's larger child goes on top (slot t + 1 in step t), the
// smaller into the popped slot, which selects find. The node's box is the union
// of its children's (as H-PLOC formed it, bit for bit). False for an id out of
// range.
__device__ __forceinline__ bool collapse_kids(const uint4* rec, uint32_t n, uint32_t node_count, uint32_t x, Kids& K,
                                              Box& pb, uint32_t& count, uint32_t& inner, uint4* buf) {
    count = 0;
    inner = 0;
    bool ok = x >= n && x < node_count, live = ok;
    uint32_t msb = 0, cur = x;
#pragma unroll
    for (uint32_t t = 0; t < 7; ++t) {
        if (!ballot(live)) break;
        Box b0, b1;
        uint32_t i0, i1, s0, s1;
        load_rec8_quads(rec, live ? cur - n : kInvalid, buf, b0, b1, i0, i1, s0, s1);
        if (live && max(i0, i1) >= node_count) {
            ok = false;
            live = false;
        }
        if (!live) continue;
        if (t == 0) pb = box_union(b0, b1);
        const bool first_is_1 = !(box_area(b0) < box_area(b1));
        const uint32_t small = first_is_1 ? i1 : i0, large = first_is_1 ? i0 : i1;
        const uint32_t psmall = small >= n ? (first_is_1 ? s1 : s0) : 0u;
        const Box bs = first_is_1 ? b1 : b0;
        K.box[t + 1] = first_is_1 ? b0 : b1;
        K.id[t + 1] = large;
        K.prims[t + 1] = large >= n ? (first_is_1 ? s0 : s1) : 0u;
        uint32_t older = 0;  // the highest inner child below the popped slot
        inner |= (small >= n ? 1u << msb : 0u) | (large >= n ? 2u << t : 0u);
        const uint32_t top = 31u - (uint32_t)__clz(inner | 1u);
#pragma unroll
        for (uint32_t j = 0; j <= t; ++j) {
            const bool here = msb == j;
            K.box[j].lx = here ? bs.lx : K.box[j].lx;
            K.box[j].ly = here ? bs.ly : K.box[j].ly;
            K.box[j].lz = here ? bs.lz : K.box[j].lz;
            K.box[j].hx = here ? bs.hx : K.box[j].hx;
            K.box[j].hy = here ? bs.hy : K.box[j].hy;
            K.box[j].hz = here ? bs.hz : K.box[j].hz;
            K.id[j] = here ? small : K.id[j];
            K.prims[j] = here ? psmall : K.prims[j];
            older = top == j ? K.id[j] : older;
        }
        count = t + 2;
        live = inner != 0;
        if (t < 6 && live) {
            cur = large >= n ? large : older;
            msb = top;
            inner &= ~(1u << top);
        }
    }
    return ok;
}

// GreedyAssignment (WideConverter.cu:106-153): each child in push order takes
// the free slot of the largest cost (GetCost 25-30), the lowest on a tie; with
// no comparable cost the first free slot. Slots s and 7 - s have opposite
// costs, bit for bit, so four sums give all eight. box(k): child k's box (any
// from count on). Nibble k of the result is child k's slot; used: the slots.
template <typename BoxOf>
__device__ __forceinline__ uint32_t greedy_slots(const Box& pb, uint32_t count, uint32_t& used, const BoxOf& box) {
    const float lowest = -3.402823466e+38f;
    const float pcx = pb.lx + pb.hx, pcy = pb.ly + pb.hy, pcz = pb.lz + pb.hz;
    uint32_t slots = 0, taken = 0;
#pragma unroll
    for (uint32_t k = 0; k < 8; ++k) {
        const Box cb = box(k);
        const float ox = pcx - (cb.hx + cb.lx), oy = pcy - (cb.hy + cb.ly), oz = pcz - (cb.hz + cb.lz);
        const float p = ox + oy, m = ox - oy;
        const float c[4] = {p + oz, p - oz, m + oz, m - oz};
        // the largest cost of the free slots (a NaN is dropped), then the
        // lowest slot that has it
        float cost[8], most = lowest;
#pragma unroll
        for (uint32_t s = 0; s < 8; ++s) {
            cost[s] = (taken & (1u << s)) ? lowest : (s < 4 ? c[s & 3] : -c[(7 - s) & 3]);
            most = fmaxf(most, cost[s]);
        }
        uint32_t best = 8u;
#pragma unroll
        for (int s = 7; s >= 0; --s) best = cost[s] == most ? (uint32_t)s : best;
        if (!(most > lowest)) best = (uint32_t)__builtin_ctz(~taken | 0x100u);
        if (k < count) {
            taken |= 1u << best;
            slots |= best << (4 * k);
        }
    }
    used = taken;
    return slots;
}

// Auction slots (auction_assign) of the same.
template <typename BoxOf>
__device__ __forceinline__ uint32_t auction_slots(const Box& pb, uint32_t count, uint32_t& used, const BoxOf& box) {
    const float pcx = pb.lx + pb.hx, pcy = pb.ly + pb.hy, pcz = pb.lz + pb.hz;
    float ox[8], oy[8], oz[8];
#pragma unroll
    for (uint32_t k = 0; k < 8; ++k) {
        const Box cb = box(k);
        ox[k] = k < count ? pcx - (cb.lx + cb.hx) : 0.0f;
        oy[k] = k < count ? pcy - (cb.ly + cb.hy) : 0.0f;
        oz[k] = k < count ? pcz - (cb.lz + cb.hz) : 0.0f;
    }
    const uint32_t assign = auction_assign(pb, ox, oy, oz, count);
    uint32_t slots = 0, taken = 0;
#pragma unroll
    for (uint32_t s = 0; s < 8; ++s) {
        const uint32_t a = nib(assign, s);
        if (a == 0xFu) continue;
        taken |= 1u << s;
        slots |= s << (4 * a);
    }
    used = taken;
    return slots;
}
template <uint32_t SLOT, typename BoxOf>
__device__ __forceinline__ uint32_t choose_slots(const Box& pb, uint32_t count, uint32_t& used, const BoxOf& box) {
    if constexpr (SLOT == NXB_SLOT_AUCTION) return auction_slots(pb, count, used, box);
    else return greedy_slots(pb, count, used, box);
}

// A wave's nodes on their way to memory, and their children by slot.
struct NodeStage {
    uint4 w[5 * kBvh8Threads];  // lane's node: five words from 5 * lane
    uint2 kid[8][kBvh8Threads];  // id, primitive count (0: a leaf)
};

// Exponents of a node's quantization grid (CreateBVH8Node, WideConverter.cu:156-206).
__device__ __forceinline__ uint32_t grid_exponents(const Box& pb, float& ix, float& iy, float& iz) {
    const float qstep = 1.0f / 255.0f;
    const uint32_t e0 = ceil_log2((pb.hx - pb.lx) * qstep) & 0xFFu;
    const uint32_t e1 = ceil_log2((pb.hy - pb.ly) * qstep) & 0xFFu;
    const uint32_t e2 = ceil_log2((pb.hz - pb.lz) * qstep) & 0xFFu;
    ix = inv_pow2(e0);
    iy = inv_pow2(e1);
    iz = inv_pow2(e2);
    return e0 | (e1 << 8) | (e2 << 16);
}

// Puts the lane's node into the stage's words w, byte by byte at its slots,
// without the child and primitive bases.
template <typename KidsOf>
__device__ __forceinline__ void stage_node(uint4* w, const Box& pb, const KidsOf& K, uint32_t count, uint32_t slots,
                                           uint32_t im, uint32_t lm) {
    float ix, iy, iz;
    const uint32_t e = grid_exponents(pb, ix, iy, iz);
    w[0] = make_uint4(__float_as_uint(pb.lx), __float_as_uint(pb.ly), __float_as_uint(pb.lz), e | (im << 24));
#pragma unroll
    for (uint32_t i = 1; i < 5; ++i) w[i] = make_uint4(0, 0, 0, 0);
#pragma unroll
    for (uint32_t k = 0; k < 8; ++k) {
        if (k >= count) break;
        const uint32_t s = nib(slots, k);
        const Box& b = K.box[k];
        uint8_t* q = reinterpret_cast<uint8_t*>(w) + 24 + s;
        q[0] = (uint8_t)((1u << 5) | ((im >> s) & 1u ? 24u + s : bits_below(lm, s)));
        q[8] = (uint8_t)q_floor((b.lx - pb.lx) * ix);
        q[16] = (uint8_t)q_floor((b.ly - pb.ly) * iy);
        q[24] = (uint8_t)q_floor((b.lz - pb.lz) * iz);
        q[32] = (uint8_t)q_ceil((b.hx - pb.lx) * ix);
        q[40] = (uint8_t)q_ceil((b.hy - pb.ly) * iy);
        q[48] = (uint8_t)q_ceil((b.hz - pb.lz) * iz);
    }
}

// What collapse_nodes works on: a level's nodes and where they go.
struct LevelIo {
    const uint4* rec;
    uint32_t n, node_count;
    nxb_bvh8_node* out;
    uint32_t* prim_idx;
    uint32_t capacity;
    uint64_t* work;
    uint32_t* flags;
};

// Makes the BVH8 nodes k0 + lane < hi of the block (a whole block, one node a
// lane): x and pbase of each lane's node, ids(total) the first id of the block's
// inner children, in LDS or known to all lanes after its barrier.
template <uint32_t SLOT, typename Ids>
__device__ __forceinline__ uint32_t collapse_nodes(NodeStage& st, uint32_t* scan_tmp, const LevelIo& io, uint32_t k0,
                                                   bool has, uint32_t x, uint32_t pbase, const Ids& ids) {
    const uint32_t tid = threadIdx.x, lane = tid & 63u, w0 = tid & ~63u;
    Kids K = {};
    Box pb = {0, 0, 0, 0, 0, 0};
    uint32_t count = 0, inner = 0;
    const bool ok =
        collapse_kids(io.rec, io.n, io.node_count, has ? x : 0u, K, pb, count, inner, st.w + 5 * w0);
    if (has && !ok) atomic_or_agent(io.flags, kFlagBadIndex);
    const uint32_t ic = ok ? (uint32_t)__popc(inner) : 0u;
    uint32_t total = 0;
    const uint32_t excl = block_scan_256<true>(ic, scan_tmp, &total);
    ids.take(total);
    uint32_t im = 0, used = 0;
    if (ok) {
        const uint32_t slots = choose_slots<SLOT>(pb, count, used, [&](uint32_t i) { return K.box[i]; });
#pragma unroll
        for (uint32_t i = 0; i < 8; ++i) im |= ((inner >> i) & 1u) << nib(slots, i);
        stage_node(st.w + 5 * tid, pb, K, count, slots, im, used & ~im);
#pragma unroll
        for (uint32_t i = 0; i < 8; ++i)
            if (i < count) st.kid[nib(slots, i)][tid] = make_uint2(K.id[i], K.prims[i]);
    }
    lds_barrier();
    const uint32_t base = ids.first() + excl;
    if (ok) {
        const uint32_t leaves = count - ic;
        uint32_t next_base = pbase + leaves, leaf = pbase, child = base;
        bool good = true;
#pragma unroll
        for (uint32_t s = 0; s < 8; ++s) {
            const uint2 kid = st.kid[s][tid];
            if ((im >> s) & 1u) {
                if (child < io.capacity && kid.y >= 2 && next_base + kid.y <= io.n)
                    io.work[child] = ((uint64_t)next_base << 32) | kid.x;  // read by the next level
                else good = false;
                next_base += kid.y;
                ++child;
            } else if ((used >> s) & 1u) {
                if (leaf < io.n) io.prim_idx[leaf] = kid.x;
                else good = false;
                ++leaf;
            }
        }
        if (!good) atomic_or_agent(io.flags, kFlagBadIndex);
        *reinterpret_cast<uint2*>(&st.w[5 * tid + 1]) = make_uint2(ic ? base : 0u, leaves ? pbase : 0u);
    }
    const uint64_t oks = ballot(ok);
    wave_lds_sync();
    // the wave's nodes are consecutive: 16 bytes a lane, five times
    uint4* o = reinterpret_cast<uint4*>(io.out + k0 + w0);
#pragma unroll
    for (uint32_t i = 0; i < 5; ++i) {
        const uint32_t c = lane + 64 * i;
        if ((oks >> (c / 5u)) & 1ull) o[c] = st.w[5 * w0 + c];
    }
    return total;
}

// Ids of a block's inner children from the next level's counter.
struct IdsFromCounter {
    uint32_t* slot;     // one word of LDS
    uint32_t* counter;
    uint32_t from;      // the next level's first id
    __device__ __forceinline__ void take(uint32_t total) const {
        if (threadIdx.x == 0) *slot = total ? from + atomic_add_agent(counter, total) : 0u;
    }
    __device__ __forceinline__ uint32_t first() const { return *slot; }
};
struct IdsInOrder {
    uint32_t from;
    __device__ __forceinline__ void take(uint32_t) const {}
    __device__ __forceinline__ uint32_t first() const { return from; }
};

// The top levels of one tree in one block: the level counters initialized
// (cnt[0] = 1, the root; the rest 0), then levels 0..kBvh8TopLevels-1 (at most 1,
// 8 and 64 nodes) one after another, the children's ids taken from a running
// count instead of a global atomic. Saves the launches and counter round trips
// of the levels whose time is all latency.
template <uint32_t SLOT>
__global__ __launch_bounds__(kBvh8Threads) void k_bvh8_top(LevelIo io, uint32_t* cnt) {
    __shared__ NodeStage st;
    __shared__ uint32_t scan_tmp[kBvh8Threads / 64];
    const uint32_t tid = threadIdx.x;
    for (uint32_t i = tid; i <= kMaxLevels; i += kBvh8Threads) cnt[i] = i == 0 ? 1u : 0u;
    uint32_t lo = 0, m = 1;
    for (uint32_t level = 0; level < kBvh8TopLevels && m != 0; ++level) {
        const uint32_t hi = lo + m;
        uint32_t next = 0;
        for (uint32_t k0 = lo; k0 < hi; k0 += kBvh8Threads) {
            const bool has = k0 + tid < hi && k0 + tid < io.capacity;
            // the root, primitive base 0; below, written by this block's previous
            // level (agent-scope loads: not through the CU's L1)
            uint64_t v = io.node_count - 1;
            if (level > 0 && has) v = load_agent64(&io.work[k0 + tid]);
            next += collapse_nodes<SLOT>(st, scan_tmp, io, k0, has, (uint32_t)v, (uint32_t)(v >> 32),
                                         IdsInOrder{hi + next});
            __syncthreads();  // the work items are written before the next level reads them
        }
        if (tid == 0) cnt[level + 1] = next;
        lo = hi;
        m = next;
    }
}

// (second bound: waves per SIMD, four as the LDS allows; the auction needs the
// registers of three)
template <uint32_t SLOT>
__global__ __launch_bounds__(kBvh8Threads, SLOT == NXB_SLOT_AUCTION ? 3 : 4) void k_bvh8_level(
    LevelIo io, uint32_t* cnt, uint32_t level) {
    __shared__ NodeStage st;
    __shared__ uint32_t scan_tmp[kBvh8Threads / 64];
    __shared__ uint32_t sbase;
    const uint32_t tid = threadIdx.x;
    const uint32_t m = cnt[level];
    if (m == 0) return;
    uint32_t lo = 0;
    for (uint32_t j = 0; j < level; ++j) lo += cnt[j];
    const uint32_t hi = lo + m;
    if (level + 1 > kMaxLevels) {
        if (blockIdx.x == 0 && tid == 0) atomic_or_agent(io.flags, kFlagBadIndex);
        return;
    }
    for (uint32_t k0 = lo + blockIdx.x * kBvh8Threads; k0 < hi; k0 += gridDim.x * kBvh8Threads) {
        const bool has = k0 + tid < hi && k0 + tid < io.capacity;
        const uint64_t v = has ? io.work[k0 + tid] : 0ull;
        collapse_nodes<SLOT>(st, scan_tmp, io, k0, has, (uint32_t)v, (uint32_t)(v >> 32),
                             IdsFromCounter{&sbase, &cnt[level + 1], hi});
        lds_barrier();  // sbase and the stage are read before the next nodes
    }
}

// ---- every node expanded first (single builds of small meshes) --------------
//
// What a BVH8 node looks like depends on its BVH2 node alone, except for the
// numbers of its children and primitives. So one launch makes the BVH8 node of
// every internal BVH2 node, side by side: the chain of seven record loads, the
// slots and the quantization are waited for once instead of once per level. The
// levels that follow only hand out numbers: a level inside a block is two loads,
// a count and the writes (~2,500 cycles, 1,300 to 2,700 of them the loads'),
// where collapsing the nodes took ~17,000. 2,003 primitives: 10 us and 18 us;
// 300K: 34 us and four launches of 6 to 20 us.

// Primitives up to which a build takes this path, above a launch per level: all
// internal BVH2 nodes are about five times those that the BVH8 needs, but at
// once. Collapse stage in us, on a surface, blobs and slivers, this / levels:
// 31/115, 29/95, 28/87 at 2,003; 51/158, 47/153, 46/145 at 48K; 93/165, 105/193,
// 94/168 at 300K; 178/200, 196/223, 180/200 at 900K; 211/214, 225/239, 195/203
// at 2^20; 206/205, 240/251, 205/205 at 1.1M; 238/208, 265/258, 246/217 at 1.3M;
// 337/247, 365/286, 343/252 at 2M: the line lies just below where they meet.
// With auction slots 108/505, 153/571, 114/420
// at 2,003; 269/1119, 264/1218, 202/850 at 300K; 616/1314, 600/1424, 455/883 at
// 2^20; 632/1315, 612/1488, 469/908 at 1.1M; 995/1319, 979/1498, 792/947 at 2M.
constexpr uint32_t kSmallPrims = 1u << 20;
bool bvh8_small(uint32_t n) { return n <= kSmallPrims; }

// The children of the node each lane collapses, in LDS (child t of lane i at
// [t][i]): box, id (a leaf is an id below n, its primitive index) and
// primitive count. Indexed by slot when they are read back, which in
// registers would take a select over all eight per field.
struct RecChildren {
    float4 a[8][kBvh8Threads];  // lx, ly, lz, hx
    uint4 b[8][kBvh8Threads];   // hy, hz, id, primitives
};
__device__ __forceinline__ void put_rec_child(RecChildren& ch, uint32_t t, uint32_t tid, const Box& b, uint32_t id,
                                              uint32_t prims) {
    ch.a[t][tid] = make_float4(b.lx, b.ly, b.lz, b.hx);
    ch.b[t][tid] = make_uint4(__float_as_uint(b.hy), __float_as_uint(b.hz), id, prims);
}
__device__ __forceinline__ Box get_child_box(const RecChildren& ch, uint32_t t, uint32_t tid) {
    const float4 a = ch.a[t][tid];
    const uint2 c = *reinterpret_cast<const uint2*>(&ch.b[t][tid]);
    Box b;
    b.lx = a.x; b.ly = a.y; b.lz = a.z; b.hx = a.w; b.hy = __uint_as_float(c.x); b.hz = __uint_as_float(c.y);
    return b;
}

// Collapse of internal node x (record x - n). Same push/pop order as
// collapse_node; the node's box is the union of its children's (as H-PLOC
// formed it, bit for bit). False for an id out of range.
__device__ __forceinline__ bool collapse_children(const uint4* rec, uint32_t n, uint32_t node_count, uint32_t x,
                                                  Box& pb, uint32_t& count, uint32_t& inner, RecChildren& ch,
                                                  uint32_t tid) {
    if (x < n || x >= node_count) return false;
    inner = 0;
    uint32_t top = 0, msb = 0, cur = x;  // top: the last slot in use
    for (;;) {
        Box b0, b1;
        uint32_t i0, i1, s0, s1;
        load_rec8(rec, cur - n, b0, b1, i0, i1, s0, s1);
        if (max(i0, i1) >= node_count) return false;
        // the smaller child into the popped slot, the larger on top
        const bool first_is_1 = !(box_area(b0) < box_area(b1));
        const uint32_t na = first_is_1 ? i1 : i0, nb = first_is_1 ? i0 : i1;
        if (top == 0) pb = box_union(b0, b1);
        ++top;
        put_rec_child(ch, msb, tid, first_is_1 ? b1 : b0, na, first_is_1 ? s1 : s0);
        put_rec_child(ch, top, tid, first_is_1 ? b0 : b1, nb, first_is_1 ? s0 : s1);
        inner |= (na >= n ? 1u << msb : 0u) | (nb >= n ? 1u << top : 0u);
        if (inner == 0 || top == 7) break;
        // the highest inner slot is expanded next: the larger child just
        // pushed, else the smaller one, else an older child
        msb = 31u - (uint32_t)__clz(inner);
        cur = nb >= n ? nb : na;
        if (cur < n) cur = ch.b[msb][tid].z;
        inner &= ~(1u << msb);
    }
    count = top + 1;
    return true;
}

// Work items passed on inside a block. place: the node's BVH8 id, and its level
// from bit kLevelBit up. (Each node has its own level: a block's share of the
// queue comes from blocks that followed their subtrees for any number of levels.)
constexpr uint32_t kLevelBit = 24, kIdMask = (1u << kLevelBit) - 1u;
static_assert(kSmallPrims <= 1u << kLevelBit && kMaxLevels < 1u << (32 - kLevelBit), "an id and a level in one word");
struct BlockQueue {
    uint32_t x[kBvh8Threads], base[kBvh8Threads], place[kBvh8Threads];
};

// Where a level's children go: ids[0..] in the order of the nodes' slots, to
// the block's queue (keep) or to the queue positions from `queue` on.
struct ChildSink {
    BlockQueue* bq;
    bool keep;
    uint32_t ids, queue;
    uint64_t *work, *work2;
    uint32_t capacity, n;

    __device__ __forceinline__ bool put(uint32_t at, uint32_t level, uint32_t x, uint32_t base,
                                        uint32_t prims) const {
        const uint32_t cid = ids + at;
        bool good = cid < capacity && prims >= 2 && base + prims <= n;
        const uint32_t cx = good ? x : kInvalid;  // an invalid item is flagged, not followed
        if (keep) {
            bq->x[at] = cx;
            bq->base[at] = base;
            bq->place[at] = (level << kLevelBit) | (cid & kIdMask);
        } else if (queue + at < capacity) {
            work[queue + at] = ((uint64_t)base << 32) | cx;
            work2[queue + at] = (level << kLevelBit) | (cid & kIdMask);
        } else {
            good = false;
        }
        return good;
    }
};

// A node's 80 bytes without the child and primitive bases, and its children by
// slot: id (kInvalid: free) and primitive count (0: a leaf or free).
struct PackedNode {
    uint4 w[5];
    uint32_t kid[8], prims[8];
};
__device__ __forceinline__ PackedNode pack_node(const RecChildren& ch, uint32_t tid, const Box& pb, uint32_t inner,
                                                uint32_t assign) {
    PackedNode r;
    float ix, iy, iz;
    const uint32_t e = grid_exponents(pb, ix, iy, iz);
    uint32_t leaves = 0, im = 0;
    uint32_t meta[2] = {0, 0}, qlx[2] = {0, 0}, qly[2] = {0, 0}, qlz[2] = {0, 0};
    uint32_t qhx[2] = {0, 0}, qhy[2] = {0, 0}, qhz[2] = {0, 0};
#pragma unroll
    for (uint32_t s = 0; s < 8; ++s) {
        // (an empty slot computes on child 7's words and keeps zeros)
        const uint32_t a = nib(assign, s) & 7u;
        const bool used = nib(assign, s) != 0xFu, in = used && ((inner >> a) & 1u);
        const float4 ca = ch.a[a][tid];
        const uint4 cb = ch.b[a][tid];
        const uint32_t w = s >> 2, sh = 8 * (s & 3);
        auto put = [&](uint32_t* q, uint32_t v) { q[w] |= used ? v << sh : 0u; };
        put(qlx, q_floor((ca.x - pb.lx) * ix));
        put(qly, q_floor((ca.y - pb.ly) * iy));
        put(qlz, q_floor((ca.z - pb.lz) * iz));
        put(qhx, q_ceil((ca.w - pb.lx) * ix));
        put(qhy, q_ceil((__uint_as_float(cb.x) - pb.ly) * iy));
        put(qhz, q_ceil((__uint_as_float(cb.y) - pb.lz) * iz));
        put(meta, (1u << 5) | (in ? 24u + s : leaves));
        r.kid[s] = used ? cb.z : kInvalid;
        r.prims[s] = in ? cb.w : 0u;
        im |= in ? 1u << s : 0u;
        leaves += used && !in ? 1u : 0u;
    }
    r.w[0] = make_uint4(__float_as_uint(pb.lx), __float_as_uint(pb.ly), __float_as_uint(pb.lz), e | (im << 24));
    r.w[1] = make_uint4(0u, 0u, meta[0], meta[1]);
    r.w[2] = make_uint4(qlx[0], qlx[1], qly[0], qly[1]);
    r.w[3] = make_uint4(qlz[0], qlz[1], qhx[0], qhx[1]);
    r.w[4] = make_uint4(qhy[0], qhy[1], qhz[0], qhz[1]);
    return r;
}

// Per internal BVH2 node x, at x - n: its BVH8 node.
//   kids: 8 ids by slot (kInvalid: free), 8 primitive counts (0: a leaf or free)
//   node: its 80 bytes, without the child and primitive bases
struct Expanded {
    uint4* kids;  // 4 each
    uint4* node;  // 5 each
};

template <uint32_t SLOT>
__global__ __launch_bounds__(kBvh8Threads) void k_bvh8_expand(const uint4* __restrict__ rec, uint32_t n,
                                                              uint32_t node_count, Expanded ex, uint32_t* flags) {
    __shared__ RecChildren ch;
    const uint32_t tid = threadIdx.x;
    for (uint32_t i = blockIdx.x * kBvh8Threads + tid; i < n - 1; i += gridDim.x * kBvh8Threads) {
        Box pb = {0, 0, 0, 0, 0, 0};
        uint32_t count = 0, inner = 0;
        if (!collapse_children(rec, n, node_count, n + i, pb, count, inner, ch, tid)) {
            atomic_or_agent(flags, kFlagBadIndex);
            const uint4 none = make_uint4(kInvalid, kInvalid, kInvalid, kInvalid), zero = make_uint4(0, 0, 0, 0);
            ex.kids[4ull * i] = none;
            ex.kids[4ull * i + 1] = none;
            ex.kids[4ull * i + 2] = zero;
            ex.kids[4ull * i + 3] = zero;
            continue;
        }
        uint32_t used, assign = 0xFFFFFFFFu;
        const auto box = [&](uint32_t k) { return get_child_box(ch, k, tid); };
        const uint32_t slots = choose_slots<SLOT>(pb, count, used, box);
#pragma unroll
        for (uint32_t k = 0; k < 8; ++k)
            if (k < count) assign = with_nib(assign, nib(slots, k), k);
        const PackedNode r = pack_node(ch, tid, pb, inner, assign);
        uint4* k = ex.kids + 4ull * i;
        k[0] = make_uint4(r.kid[0], r.kid[1], r.kid[2], r.kid[3]);
        k[1] = make_uint4(r.kid[4], r.kid[5], r.kid[6], r.kid[7]);
        k[2] = make_uint4(r.prims[0], r.prims[1], r.prims[2], r.prims[3]);
        k[3] = make_uint4(r.prims[4], r.prims[5], r.prims[6], r.prims[7]);
        uint4* o = ex.node + 5ull * i;
#pragma unroll
        for (uint32_t j = 0; j < 5; ++j) o[j] = r.w[j];
    }
}

// Levels that a block follows while the queue grows, by queued nodes: a node's
// children hold about 1/2, 1/4, 1/8, ... of its primitives (the larger child is
// expanded each time), so a block that went on alone with a large one would
// hold up the launch. One level more for each measured within 5%.
constexpr uint32_t kThreeLevelNodes = 2048, kTwoLevelNodes = 32768;
__device__ __forceinline__ uint32_t levels_to_follow(uint32_t m) {
    return m <= kThreeLevelNodes ? 3u : m <= kTwoLevelNodes ? 2u : 1u;
}

// Numbers the nodes from the root down. A block reserves the ids of its nodes'
// inner children with one atomic add on the node counter alloc (the nodes below
// the root, node 0; zero before launch 0) and passes the children on to itself,
// through LDS, while they fit its lanes, else to the next launch through a queue
// in global memory: work[q] = (first primitive << 32 | BVH2 id), work2[q] = the
// place word of queue position q. Launch l takes the positions
// [cnt[1] + ... + cnt[l-1], +cnt[l]), counts that earlier launches completed, so
// no lane ever waits on another (no polling, no spin limit); launch 0 is the
// root.
//
// Eight lanes take a node, one its slot: a block's pass places 32 nodes, and a
// node's words go out in three coalesced stores. (One lane per node: 38 us at
// 2,003 primitives and 105 at 300K for both kernels, now 31 and 93.) At least
// kPlaceShare nodes per block: each block and level costs two atomic adds on the
// same two counters (10 ns each).
__global__ __launch_bounds__(kBvh8Threads) void k_bvh8_place(Expanded ex, uint32_t n, uint32_t node_count,
                                                             nxb_bvh8_node* __restrict__ out,
                                                             uint32_t* __restrict__ prim_idx, uint32_t capacity,
                                                             uint64_t* work, uint64_t* work2, uint32_t* cnt,
                                                             uint32_t launch, uint32_t* alloc, uint32_t* flags) {
    constexpr uint32_t kPlaceNodes = kBvh8Threads / 8, kPlacePasses = 8, kPlaceShare = 4;
    __shared__ BlockQueue bq[2];
    __shared__ uint32_t scan_tmp[2][kBvh8Threads / 64];
    __shared__ uint32_t sids, squeue;
    const uint32_t tid = threadIdx.x, lane = tid & 63u, w = tid >> 6, s = tid & 7u, g = tid >> 3;
    const uint32_t m = launch == 0 ? 1u : min(cnt[launch], capacity);
    if (m == 0) return;
    uint32_t lo = 0;
    for (uint32_t j = 1; j < launch; ++j) lo += cnt[j];
    const uint32_t hi = launch == 0 ? 0u : lo + m;
    const bool follow = m <= gridDim.x * kBvh8Threads;
    uint32_t left = kMaxLevels;
    if (launch != 0 && (launch == 1 || m >= cnt[launch - 1])) left = levels_to_follow(m);
    const uint32_t per = follow ? max((m + gridDim.x - 1) / gridDim.x, kPlaceShare) : (uint32_t)kBvh8Threads;
    for (uint32_t i0 = blockIdx.x * per; i0 < m; i0 += gridDim.x * per) {
        uint32_t nodes = min(per, m - i0), cur = 0;
        uint32_t below = 1;  // launch 0, one block: ids given out
        if (launch == 0) {
            if (tid == 0) {  // the root
                bq[0].x[0] = node_count - 1;
                bq[0].base[0] = 0;
                bq[0].place[0] = 0;
            }
        } else {
            if (tid < nodes) {
                const bool has = lo + i0 + tid < capacity;
                const uint64_t v = has ? work[lo + i0 + tid] : (uint64_t)kInvalid;
                bq[0].x[tid] = (uint32_t)v;
                bq[0].base[tid] = (uint32_t)(v >> 32);
                bq[0].place[tid] = has ? (uint32_t)work2[lo + i0 + tid] : 0u;
            }
        }
        lds_barrier();
        for (;;) {
            // what each lane places: slot s of the node of its eight in pass p
            uint32_t kid[kPlacePasses], prims[kPlacePasses], img[kPlacePasses][3], ic = 0;
#pragma unroll
            for (uint32_t p = 0; p < kPlacePasses; ++p) {
                kid[p] = kInvalid;
                prims[p] = 0;
                img[p][0] = img[p][1] = img[p][2] = 0;
                const uint32_t j = p * kPlaceNodes + g;
                if (p * kPlaceNodes < nodes && j < nodes) {
                    const uint32_t x = bq[cur].x[j], place = bq[cur].place[j];
                    if (x >= n && x < node_count && (place & kIdMask) < capacity &&
                        place >> kLevelBit < kMaxLevels) {
                        const uint32_t* k = reinterpret_cast<const uint32_t*>(ex.kids + 4ull * (x - n));
                        const uint32_t* o = reinterpret_cast<const uint32_t*>(ex.node + 5ull * (x - n));
                        prims[p] = k[8 + s];
                        kid[p] = k[s];
                        img[p][0] = o[s];
                        img[p][1] = o[8 + s];
                        img[p][2] = o[16 + (s & 3u)];
                    } else {
                        atomic_or_agent(flags, kFlagBadIndex);
                    }
                }
            }
#pragma unroll
            for (uint32_t p = 0; p < kPlacePasses; ++p)
                if (p * kPlaceNodes < nodes) ic += (uint32_t)__popcll(ballot(prims[p] != 0));
            if (lane == 0) scan_tmp[cur][w] = ic;
            lds_barrier();
            uint32_t at = 0, total = 0;
#pragma unroll
            for (uint32_t k = 0; k < kBvh8Threads / 64; ++k) {
                const uint32_t t = scan_tmp[cur][k];
                at += k < w ? t : 0u;
                total += t;
            }
            const bool keep = follow && --left != 0 && total <= (uint32_t)kBvh8Threads;
            uint32_t ids = below, queue = 0;
            if (launch == 0) {
                below += total;
                if (tid == 0 && !(keep && total)) {
                    *alloc = below - 1;
                    cnt[1] = total;
                }
            } else {
                if (tid == 0) sids = total ? 1u + atomic_add_agent(alloc, total) : 0u;
                if (tid == 64) squeue = total && !keep ? hi + atomic_add_agent(&cnt[launch + 1], total) : 0u;
                lds_barrier();
                ids = sids;
                queue = squeue;
            }
            const ChildSink sink{&bq[cur ^ 1], keep, ids, queue, work, work2, capacity, n};
            bool good = true;
#pragma unroll
            for (uint32_t p = 0; p < kPlacePasses; ++p) {
                if (p * kPlaceNodes >= nodes) break;
                const uint32_t j = min(p * kPlaceNodes + g, nodes - 1);
                const uint32_t x = bq[cur].x[j], base = bq[cur].base[j], place = bq[cur].place[j];
                const uint32_t id = place & kIdMask, level = place >> kLevelBit;
                const bool ok = p * kPlaceNodes + g < nodes && x >= n && x < node_count && id < capacity &&
                                level < kMaxLevels;
                const bool in = prims[p] != 0, leaf = !in && kid[p] != kInvalid;
                const uint64_t ib = ballot(in);
                const uint32_t im = (uint32_t)(ib >> (lane & 56u)) & 0xFFu;
                const uint32_t lm = (uint32_t)(ballot(leaf) >> (lane & 56u)) & 0xFFu;
                const uint32_t leaves = (uint32_t)__popc(lm);
                const uint32_t first = at + (uint32_t)__popcll(ib & ((1ull << (lane & 56u)) - 1ull));  // its children
                uint32_t before = prims[p];  // primitives of the inner slots up to this one
                const uint32_t back1 = lane_back<1>(before);  // (all lanes take part in each shift)
                before += s >= 1 ? back1 : 0u;
                const uint32_t back2 = lane_back<2>(before);
                before += s >= 2 ? back2 : 0u;
                const uint32_t back4 = lane_back<4>(before);
                before += s >= 4 ? back4 : 0u;
                if (in)
                    good &= sink.put(first + bits_below(im, s), level + 1, kid[p], base + leaves + before - prims[p],
                                     prims[p]);
                if (leaf) {
                    const uint32_t q = base + bits_below(lm, s);
                    if (q < n) prim_idx[q] = kid[p];
                    else good = false;
                }
                if (ok) {
                    uint32_t* dst = reinterpret_cast<uint32_t*>(out + id);
                    uint32_t v = img[p][0];
                    if (s == 4) v = im ? ids + first : 0u;
                    if (s == 5) v = leaves ? base : 0u;
                    dst[s] = v;
                    dst[8 + s] = img[p][1];
                    if (s < 4) dst[16 + s] = img[p][2];
                }
                at += (uint32_t)__popcll(ib);
            }
            if (!good) atomic_or_agent(flags, kFlagBadIndex);
            if (!keep || total == 0) break;
            lds_barrier();  // the next level's queue is written
            nodes = total;
            cur ^= 1;
        }
        lds_barrier();  // the queue is read before the next share fills it
    }
}

// `count` consecutive values per lane from one counter per tree (node ids,
// primIdx slots): each run of consecutive lanes with the same tree takes its
// values with one atomic (issued by the run's last lane) and every lane gets
// the first of its `count`. Lanes with tree == kInvalid take none. Whole wave
// only.
__device__ __forceinline__ uint32_t alloc_tree_ids(uint32_t* ctr, uint32_t tree, uint32_t count) {
    const uint32_t lane = lane_id();
    const uint32_t prev = __shfl_up(tree, 1);
    const uint64_t heads = ballot(lane == 0 || prev != tree);
    const uint32_t first = 63u - (uint32_t)__clzll((long long)(heads & (~0ull >> (63u - lane))));
    uint32_t v = count;  // inclusive sum over the run
#pragma unroll
    for (uint32_t off = 1; off < 64; off <<= 1) {
        const uint32_t t = __shfl_up(v, off);
        if (lane >= first + off) v += t;
    }
    const bool tail = lane == 63u || ((heads >> (lane + 1u)) & 1ull);
    const uint64_t tails = ballot(tail);
    const uint32_t last = (uint32_t)__ffsll((long long)(tails & (~0ull << lane))) - 1u;
    uint32_t base = 0;
    if (tail && tree != kInvalid && v != 0) base = atomic_add_agent(&ctr[tree], v);
    return __shfl(base, last) + v - count;
}

// Work items of one block's top levels (k_bvh8_tree_top), in LDS: BVH2
// node, the node's children, tree and node id.
constexpr uint32_t kTopQueue = kBvh8Threads;
struct TopQueue {
    uint32_t x[kTopQueue], l[kTopQueue], r[kTopQueue], tree[kTopQueue], self[kTopQueue];
};

// One BVH8 node of tree `tree` (batched builds): node `self` of the tree's
// region out, children's work items at queue positions qbase.., their node
// ids nbase.. (tree-local), its leaves at primIdx slots prim_base.. (local to
// the tree; each node takes its own from the tree's counter, so no subtree
// sizes are read). The children go to the level queue in work2/work3
// (positions below capacity), or with lq to a block's LDS queue (positions
// below kTopQueue).
// ti = {first primitive, primitive count, region start, region capacity}.
__device__ __forceinline__ void emit_tree_node(const ChildBoxes& cbx, uint32_t tid, const Collapsed& c,
                                               uint32_t tree, uint32_t self, uint32_t qbase, uint32_t nbase,
                                               uint32_t prim_base, uint4 ti, nxb_bvh8_node* out,
                                               uint32_t* prim_idx, uint32_t capacity, uint64_t* work2,
                                               uint64_t* work3, uint32_t* flags, TopQueue* lq = nullptr) {
    const uint32_t ic = (uint32_t)__popc(c.im);
    const uint32_t leaf_count = c.count - ic;
    if (self >= ti.w || (ic != 0 && nbase + ic > ti.w) || (leaf_count != 0 && prim_base + leaf_count > ti.y)) {
        atomic_or_agent(flags, kFlagBadIndex);
        return;
    }
    bool bad = false;
#pragma unroll
    for (uint32_t s = 0; s < 8; ++s) {
        const uint32_t a = nib(c.assign, s);
        if (a == 0xFu) continue;
        uint32_t ch = 0, pl = 0, pr = 0;
#pragma unroll
        for (uint32_t t = 0; t < 8; ++t)
            if (t == a) { ch = c.child[t]; pl = c.cleft[t]; pr = c.cright[t]; }
        if (c.im & (1u << s)) {
            const uint32_t rank = bits_below(c.im, s);
            const uint32_t q = qbase + rank;
            if (q >= (lq ? kTopQueue : capacity)) {
                bad = true;
            } else if (lq) {
                // read by this block's next level
                lq->x[q] = ch;
                lq->l[q] = pl;
                lq->r[q] = pr;
                lq->tree[q] = tree;
                lq->self[q] = nbase + rank;
            } else {
                // read by the next level's kernel
                work2[q] = ((uint64_t)pr << 32) | pl;
                work3[q] = ((uint64_t)tree << 32) | (nbase + rank);
            }
        } else {
            const uint32_t p = prim_base + bits_below(c.lm, s);
            if (p < ti.y) prim_idx[ti.x + p] = pr;
            else bad = true;
        }
    }
    if (bad) atomic_or_agent(flags, kFlagBadIndex);
    write_bvh8_node(out + ti.z, self, c.pb, cbx, tid, ic ? nbase : 0u, leaf_count ? prim_base : 0u, c.assign, c.im,
                    c.lm);
}

// As Kids, of BVH2 nodes: an inner child's children, a leaf's kInvalid and
// primitive index.
struct TreeKids {
    Box box[8];
    uint32_t left[8], right[8];
};

// Two nodes per lane (c0, c1; kInvalid: none) as load_rec8_quads fetches a
// record: two lanes each.
template <uint32_t J>
__device__ __forceinline__ void fetch_pair(const uint4* nodes, uint32_t c0, uint32_t c1, uint4* buf) {
    const uint32_t o0 = of_quad<J>(c0), o1 = of_quad<J>(c1), q = __lane_id() & 3u;
    if (o0 != kInvalid) fetch16(nodes + 2ull * (q & 2u ? o1 : o0) + (q & 1u), buf + 65 * J);
}
__device__ __forceinline__ void load_pair_quads(const nxb_bvh2_node* b2, uint32_t c0, uint32_t c1, uint4* buf, Box& b0,
                                                Box& b1, uint32_t& l0, uint32_t& r0, uint32_t& l1, uint32_t& r1) {
    const uint4* nodes = reinterpret_cast<const uint4*>(b2);
    fetch_pair<0>(nodes, c0, c1, buf);
    fetch_pair<1>(nodes, c0, c1, buf);
    fetch_pair<2>(nodes, c0, c1, buf);
    fetch_pair<3>(nodes, c0, c1, buf);
    wait_memory_ops();
    wave_lds_sync();
    const uint32_t lane = __lane_id();
    const uint4* p = buf + 65 * (lane & 3u) + 4 * (lane >> 2);
    const uint4 q0 = p[0], q1 = p[1], q2 = p[2], q3 = p[3];
    wave_lds_sync();
    b0.lx = __uint_as_float(q0.x); b0.ly = __uint_as_float(q0.y); b0.lz = __uint_as_float(q0.z);
    b0.hx = __uint_as_float(q0.w); b0.hy = __uint_as_float(q1.x); b0.hz = __uint_as_float(q1.y);
    b1.lx = __uint_as_float(q2.x); b1.ly = __uint_as_float(q2.y); b1.lz = __uint_as_float(q2.z);
    b1.hx = __uint_as_float(q2.w); b1.hy = __uint_as_float(q3.x); b1.hz = __uint_as_float(q3.y);
    l0 = q1.z; r0 = q1.w; l1 = q3.z; r1 = q3.w;
}

// collapse_kids from BVH2 nodes, of the node with children c0 and c1.
__device__ __forceinline__ bool collapse_tree_kids(const nxb_bvh2_node* b2, uint32_t node_count, bool has, uint32_t c0,
                                                   uint32_t c1, TreeKids& K, Box& pb, uint32_t& count, uint32_t& inner,
                                                   uint4* buf) {
    count = 0;
    inner = 0;
    bool ok = has, live = has;
    uint32_t msb = 0;
#pragma unroll
    for (uint32_t t = 0; t < 7; ++t) {
        if (live && max(c0, c1) >= node_count) {
            ok = false;
            live = false;
        }
        if (!ballot(live)) break;
        Box b0, b1;
        uint32_t l0, r0, l1, r1;
        load_pair_quads(b2, live ? c0 : kInvalid, c1, buf, b0, b1, l0, r0, l1, r1);
        if (!live) continue;
        if (t == 0) pb = box_union(b0, b1);
        const bool first_is_1 = !(box_area(b0) < box_area(b1));
        const uint32_t sl = first_is_1 ? l1 : l0, sr = first_is_1 ? r1 : r0;
        const Box bs = first_is_1 ? b1 : b0;
        K.box[t + 1] = first_is_1 ? b0 : b1;
        K.left[t + 1] = first_is_1 ? l0 : l1;
        K.right[t + 1] = first_is_1 ? r0 : r1;
        inner |= (sl != kInvalid ? 1u << msb : 0u) | (K.left[t + 1] != kInvalid ? 2u << t : 0u);
        const uint32_t top = 31u - (uint32_t)__clz(inner | 1u);
        c0 = K.left[t + 1];  // of the highest inner child
        c1 = K.right[t + 1];
#pragma unroll
        for (uint32_t j = 0; j <= t; ++j) {
            const bool here = msb == j;
            K.box[j].lx = here ? bs.lx : K.box[j].lx;
            K.box[j].ly = here ? bs.ly : K.box[j].ly;
            K.box[j].lz = here ? bs.lz : K.box[j].lz;
            K.box[j].hx = here ? bs.hx : K.box[j].hx;
            K.box[j].hy = here ? bs.hy : K.box[j].hy;
            K.box[j].hz = here ? bs.hz : K.box[j].hz;
            K.left[j] = here ? sl : K.left[j];
            K.right[j] = here ? sr : K.right[j];
            c0 = top == j ? K.left[j] : c0;
            c1 = top == j ? K.right[j] : c1;
        }
        count = t + 2;
        live = inner != 0;
        if (t < 6 && live) {
            msb = top;
            inner &= ~(1u << top);
        }
    }
    return ok;
}

// A level of a forest whose trees each own an output region (batched
// builds). Queue position k (level order, as in k_bvh8_level) holds work2[k] =
// its BVH2 node's children and work3[k] = (tree << 32 | tree-local node id);
// tree t writes its nodes to out + info[t].z and its
// primitives to prim_idx + info[t].x, so each tree's BVH8 is contiguous with
// root 0 and needs no compaction afterwards. Node ids come from ids[t] and
// each node's primIdx slots for its leaves from prims[t]. Children, fetches and
// node words as in collapse_nodes, the children's BVH2 ids not kept at all (162
// registers, three waves per SIMD; held to 128 it spills and takes 1,400 us):
// levels 3 and below of 2,048 meshes 1,080 -> 880 us.
template <uint32_t SLOT>
__global__ __launch_bounds__(kBvh8Threads) void k_bvh8_tree_level(
    const nxb_bvh2_node* __restrict__ b2, uint32_t node_count, nxb_bvh8_node* __restrict__ out,
    uint32_t* __restrict__ prim_idx, uint32_t capacity, uint64_t* work2, uint64_t* work3, uint32_t* cnt,
    uint32_t level, const uint4* __restrict__ info, uint32_t trees, uint32_t* ids, uint32_t* prims, uint32_t* flags) {
    __shared__ uint4 words[5 * kBvh8Threads];
    __shared__ uint32_t dest[kBvh8Threads];  // node of each lane, from out; kInvalid: none
    __shared__ uint32_t scan_tmp[kBvh8Threads / 64];
    __shared__ uint32_t sbase;
    const uint32_t tid = threadIdx.x, lane = tid & 63u, w0 = tid & ~63u;
    const uint32_t m = cnt[level];
    if (m == 0) return;
    uint32_t lo = 0;
    for (uint32_t j = 0; j < level; ++j) lo += cnt[j];
    const uint32_t hi = lo + m;
    if (level + 1 > kMaxLevels) {
        if (blockIdx.x == 0 && tid == 0) atomic_or_agent(flags, kFlagBadIndex);
        return;
    }
    for (uint32_t k0 = lo + blockIdx.x * kBvh8Threads; k0 < hi; k0 += gridDim.x * kBvh8Threads) {
        const uint32_t k = k0 + tid;
        TreeKids K = {};
        Box pb = {0, 0, 0, 0, 0, 0};
        uint32_t tree = kInvalid, self = 0, count = 0, inner = 0;
        uint4 ti = make_uint4(0, 0, 0, 0);
        uint64_t lr = 0;
        bool has = k < hi && k < capacity;
        if (has) {
            const uint64_t t3 = work3[k];
            lr = work2[k];
            self = (uint32_t)t3;
            tree = (uint32_t)(t3 >> 32);
            ti = info[min(tree, trees - 1u)];
            has = tree < trees;
        }
        const bool ok = collapse_tree_kids(b2, node_count, has, (uint32_t)lr, (uint32_t)(lr >> 32), K, pb, count,
                                           inner, words + 5 * w0);
        if (!ok) {
            tree = kInvalid;
            if (k < hi) atomic_or_agent(flags, kFlagBadIndex);
        }
        const uint32_t ic = ok ? (uint32_t)__popc(inner) : 0u;
        const uint32_t leaves = ok ? count - ic : 0u;
        uint32_t total = 0;
        const uint32_t excl = block_scan_256<true>(ic, scan_tmp, &total);
        // lanes without inner children or leaves stay in their tree's run
        // (count 0), so a wave whose nodes lie in one tree takes its ids and
        // its primIdx slots with one atomic each
        const uint32_t nbase = alloc_tree_ids(ids, tree, ic);
        const uint32_t pbase = alloc_tree_ids(prims, tree, leaves);
        if (tid == 0) sbase = total ? hi + atomic_add_agent(&cnt[level + 1], total) : 0u;
        const bool fits = ok && self < ti.w && (ic == 0 || nbase + ic <= ti.w) &&
                          (leaves == 0 || pbase + leaves <= ti.y);
        if (ok && !fits) atomic_or_agent(flags, kFlagBadIndex);
        uint32_t im = 0, used = 0, slots = 0;
        if (fits) {
            slots = choose_slots<SLOT>(pb, count, used, [&](uint32_t i) { return K.box[i]; });
#pragma unroll
            for (uint32_t i = 0; i < 8; ++i) im |= ((inner >> i) & 1u) << nib(slots, i);
            stage_node(words + 5 * tid, pb, K, count, slots, im, used & ~im);
            *reinterpret_cast<uint2*>(&words[5 * tid + 1]) = make_uint2(ic ? nbase : 0u, leaves ? pbase : 0u);
        }
        dest[tid] = fits ? ti.z + self : kInvalid;
        lds_barrier();
        if (fits) {
            const uint32_t qbase = sbase + excl, lm = used & ~im;
            bool good = qbase + ic <= capacity;
#pragma unroll
            for (uint32_t i = 0; i < 8; ++i) {
                if (i >= count) break;
                const uint32_t s = nib(slots, i);
                if ((inner >> i) & 1u) {
                    const uint32_t rank = bits_below(im, s), q = qbase + rank;
                    if (q < capacity) {  // read by the next level's kernel
                        work2[q] = ((uint64_t)K.right[i] << 32) | K.left[i];
                        work3[q] = ((uint64_t)tree << 32) | (nbase + rank);
                    }
                } else {
                    prim_idx[ti.x + pbase + bits_below(lm, s)] = K.right[i];
                }
            }
            if (!good) atomic_or_agent(flags, kFlagBadIndex);
        }
        // 16 bytes a lane: a tree's nodes are consecutive for the most part
        uint4* o = reinterpret_cast<uint4*>(out);
#pragma unroll
        for (uint32_t i = 0; i < 5; ++i) {
            const uint32_t c = lane + 64 * i, to = dest[w0 + c / 5u];
            if (to != kInvalid) o[5ull * to + c % 5u] = words[5 * w0 + c];
        }
        lds_barrier();  // sbase, dest and the words are read before the next nodes
    }
}

// Levels 0..kTreeTopLevels-1 of a forest with per-tree regions, one block
// per kTopTrees trees: at most 4 roots, 32 level-1 and 256 level-2 nodes,
// so each level is one pass of the block's lanes. The block seeds its roots,
// keeps the work items of levels 1 and 2 in LDS and numbers those levels'
// nodes with LDS counters (no global atomics, no launches between these
// levels), then appends level 3's work items to the level queue from
// position 0 (cnt[0..2] stay 0, cnt[3] counts them) and hands its trees'
// node and primIdx counts to ids[] and prims[] for the level kernels.
constexpr uint32_t kTopTrees = 4;

template <uint32_t SLOT>
__global__ __launch_bounds__(kBvh8Threads) void k_bvh8_tree_top(
    const nxb_bvh2_node* __restrict__ b2, uint32_t n, uint32_t node_count, nxb_bvh8_node* __restrict__ out,
    uint32_t* prim_idx, uint32_t capacity, uint64_t* work2, uint64_t* work3, uint32_t* cnt,
    const uint4* __restrict__ info, uint32_t trees, const uint32_t* __restrict__ mesh_lo, uint32_t* ids,
    uint32_t* prims, uint32_t* flags) {
    __shared__ ChildBoxes cbx;
    __shared__ TopQueue tq[2];
    __shared__ uint32_t scan_tmp[kBvh8Threads / 64];
    __shared__ uint32_t s_ids[kTopTrees], s_prims[kTopTrees];
    __shared__ uint32_t s_cnt[2];
    __shared__ uint32_t sbase;
    const uint32_t tid = threadIdx.x;
    const uint32_t t0 = blockIdx.x * kTopTrees;
    if (t0 >= trees) return;
    const uint32_t nt = min(kTopTrees, trees - t0);
    if (tid < nt) {
        // the root of tree t is its last internal node, n + lo - t + cnt - 2
        const uint32_t t = t0 + tid;
        const uint32_t lo = mesh_lo[t], c = mesh_lo[t + 1] - lo;
        tq[0].x[tid] = n + lo - t + c - 2;
        tq[0].l[tid] = 0;
        tq[0].r[tid] = 0;
        tq[0].tree[tid] = t;
        tq[0].self[tid] = 0;
        s_ids[tid] = 1;
        s_prims[tid] = 0;
    }
    if (tid == 0) s_cnt[0] = nt;
    __syncthreads();
    for (uint32_t level = 0; level < kTreeTopLevels; ++level) {
        const uint32_t cur = level & 1u;
        const uint32_t m = s_cnt[cur];
        const bool last = level + 1 == kTreeTopLevels;
        Collapsed c;
        bool ok = false;
        uint32_t tree = kInvalid, self = 0;
        uint4 ti = make_uint4(0, 0, 0, 0);
        if (tid < m) {
            const uint32_t x = tq[cur].x[tid], t = tq[cur].tree[tid];
            self = tq[cur].self[tid];
            ti = info[min(t, trees - 1u)];
            ok = t >= t0 && t < t0 + nt && x < node_count &&
                 collapse_node(b2, node_count, x, c, cbx, tid, SLOT, level > 0, tq[cur].l[tid], tq[cur].r[tid]);
            if (ok) tree = t;
            else atomic_or_agent(flags, kFlagBadIndex);
        }
        const uint32_t ic = ok ? (uint32_t)__popc(c.im) : 0u;
        const uint32_t leaves = ok ? c.count - ic : 0u;
        uint32_t total = 0;
        const uint32_t excl = block_scan_256(ic, scan_tmp, &total);
        uint32_t nbase = 0, pbase = 0;
        if (ic) nbase = atomicAdd(&s_ids[tree - t0], ic);
        if (leaves) pbase = atomicAdd(&s_prims[tree - t0], leaves);
        if (tid == 0) {
            if (last) sbase = total ? atomic_add_agent(&cnt[kTreeTopLevels], total) : 0u;
            else s_cnt[cur ^ 1u] = total;
        }
        __syncthreads();  // this level's queue is read; sbase and the next count are set
        if (ok)
            emit_tree_node(cbx, tid, c, tree, self, last ? sbase + excl : excl, nbase, pbase, ti, out, prim_idx,
                           capacity, work2, work3, flags, last ? nullptr : &tq[cur ^ 1u]);
        __syncthreads();  // the next level's queue is written
    }
    if (tid < nt) {
        ids[t0 + tid] = s_ids[tid];
        prims[t0 + tid] = s_prims[tid];
    }
}

// Primitive counts of the internal nodes of any BVH2: parents first, then a
// bottom-up climb where the second child to arrive at a node sums the two
// counts (distinct-address atomics only).
__global__ void k_parents(const nxb_bvh2_node* __restrict__ b2, uint32_t n, uint32_t* parent, uint32_t* arrive,
                          uint32_t* flags) {
    uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i == 0) parent[2 * n - 2] = kInvalid;
    if (i < n - 1) {
        uint32_t x = n + i;
        arrive[i] = 0;
        uint32_t l = b2[x].left, r = b2[x].right;
        if (l < 2 * n - 1 && r < 2 * n - 1) {
            parent[l] = x;
            parent[r] = x;
        } else {
            atomic_or_agent(flags, kFlagBadIndex);
        }
    }
}

__global__ void k_sizes(const nxb_bvh2_node* __restrict__ b2, uint32_t n, const uint32_t* __restrict__ parent,
                        uint32_t* arrive, uint32_t* nsize) {
    uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    uint32_t p = parent[i];
    for (uint32_t guard = 0; p != kInvalid && p >= n && p < 2 * n - 1 && guard < n; ++guard) {
        wait_memory_ops();
        if (atomic_add_agent(&arrive[p - n], 1u) == 0) return;  // first arrival: the sibling finishes p
        compiler_barrier();
        uint32_t l = b2[p].left, r = b2[p].right;
        uint32_t sl = l < n ? 1u : load_agent(&nsize[l - n]);
        uint32_t sr = r < n ? 1u : load_agent(&nsize[r - n]);
        store_agent(&nsize[p - n], sl + sr);
        p = parent[p];
    }
}

hipError_t launch_subtree_sizes(const nxb_bvh2_node* bvh2, uint32_t n, uint32_t* parent, uint32_t* arrive,
                                uint32_t* nsize, uint32_t* flags, hipStream_t s) {
    if (n < 2) return hipSuccess;
    uint32_t g = (n + 255) / 256;
    hipLaunchKernelGGL(k_parents, dim3(g), dim3(256), 0, s, bvh2, n, parent, arrive, flags);
    hipLaunchKernelGGL(k_sizes, dim3(g), dim3(256), 0, s, bvh2, n, parent, arrive, nsize);
    return hipGetLastError();
}

__global__ void k_bvh8_init(unsigned long long* ctr, uint32_t* grab, uint64_t* work, uint32_t root) {
    *ctr = 1;   // one node allocated (the root), none finished
    *grab = 0;
    work[0] = root;  // primitive base 0
}

hipError_t launch_bvh8_prep(uint32_t n, uint32_t capacity, Bvh8Scratch sc, hipStream_t s) {
    if (n == 0) return hipSuccess;
    hipError_t e = launch_fill_u32(reinterpret_cast<uint32_t*>(sc.work), kInvalid, 2ull * capacity, s);
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(k_bvh8_init, dim3(1), dim3(1), 0, s, sc.ctr, sc.grab, sc.work, 2 * n - 2);
    return hipGetLastError();
}

hipError_t launch_bvh8_run(const nxb_bvh2_node* bvh2, uint32_t n, nxb_bvh8_node* out, uint32_t* prim_idx,
                           uint32_t capacity, uint32_t spin_limit, Bvh8Scratch sc, hipStream_t s) {
    if (n == 0) return hipSuccess;
    // Fewer, busier waves: lanes of a wave that build nodes in the same
    // iteration share one counter atomic.
    uint32_t lanes = capacity / 16;
    lanes = max(lanes, 4096u);
    lanes = min(lanes, device_cu_count() * 512u);
    lanes = min(lanes, capacity);
    uint32_t grid = (lanes + kBvh8Threads - 1) / kBvh8Threads;
    if (n == 1) grid = 1;
    hipLaunchKernelGGL(sc.slot_mode == NXB_SLOT_AUCTION ? k_bvh8<NXB_SLOT_AUCTION> : k_bvh8<NXB_SLOT_GREEDY>,
                       dim3(grid), dim3(kBvh8Threads), 0, s, bvh2, n, 2 * n - 1, out, prim_idx, capacity, sc.work,
                       sc.ctr, sc.grab, sc.nsize, sc.flags, spin_limit);
    return hipGetLastError();
}

hipError_t launch_bvh8_forest(const nxb_bvh2_node* bvh2, uint32_t n, uint32_t trees, nxb_bvh8_node* out,
                              uint32_t* prim_idx, uint32_t capacity, uint32_t lanes, uint32_t spin_limit,
                              Bvh8Scratch sc, hipStream_t s) {
    if (n < 2) return hipErrorInvalidValue;
    lanes = min(max(lanes, 256u), capacity);
    uint32_t grid = (lanes + kBvh8Threads - 1) / kBvh8Threads;
    hipLaunchKernelGGL(sc.slot_mode == NXB_SLOT_AUCTION ? k_bvh8<NXB_SLOT_AUCTION> : k_bvh8<NXB_SLOT_GREEDY>,
                       dim3(grid), dim3(kBvh8Threads), 0, s, bvh2, n, 2 * n - trees, out, prim_idx, capacity,
                       sc.work, sc.ctr, sc.grab, sc.nsize, sc.flags, spin_limit);
    return hipGetLastError();
}

hipError_t launch_bvh8_collapse(const nxb_bvh2_node* bvh2, uint32_t n, nxb_bvh8_node* out, uint32_t* prim_idx,
                                uint32_t capacity, Bvh8Scratch sc, uint32_t* cnt, uint32_t* alloc, uint32_t from,
                                uint32_t count, hipStream_t s) {
    if (n == 0) return hipSuccess;
    if (n == 1) {
        if (from == 0)
            hipLaunchKernelGGL(k_bvh8<NXB_SLOT_GREEDY>, dim3(1), dim3(kBvh8Threads), 0, s, bvh2, n, 1u, out,
                               prim_idx, capacity, sc.work, sc.ctr, sc.grab, sc.nsize, sc.flags, 1u);
        return hipGetLastError();
    }
    if (!sc.rec8 || !sc.work2) return hipErrorInvalidValue;
    const bool auction = sc.slot_mode == NXB_SLOT_AUCTION;
    if (bvh8_small(n)) {
        if (!sc.ex_kids || !sc.ex_node) return hipErrorInvalidValue;
        const Expanded ex{sc.ex_kids, sc.ex_node};
        if (from == 0)  // two blocks of 64 KB LDS per CU
            hipLaunchKernelGGL(auction ? k_bvh8_expand<NXB_SLOT_AUCTION> : k_bvh8_expand<NXB_SLOT_GREEDY>,
                               dim3(min((n - 2) / kBvh8Threads + 1, device_cu_count() * 2u)), dim3(kBvh8Threads), 0, s,
                               sc.rec8, n, 2 * n - 1, ex, sc.flags);
        const uint32_t grid = min((capacity + kBvh8Threads - 1) / kBvh8Threads, device_cu_count() * 4u);
        const uint32_t end = min(from + count, kMaxLevels);
        for (uint32_t l = from; l < end; ++l)
            hipLaunchKernelGGL(k_bvh8_place, dim3(l == 0 ? 1u : grid), dim3(kBvh8Threads), 0, s, ex, n, 2 * n - 1, out,
                               prim_idx, capacity, sc.work, sc.work2, cnt, l, alloc, sc.flags);
        return hipGetLastError();
    }
    const LevelIo io{sc.rec8, n, 2 * n - 1, out, prim_idx, capacity, sc.work, sc.flags};
    // four 36 KB blocks per CU; a level of m nodes uses ceil(m / 256) blocks
    const uint32_t grid = min((capacity + kBvh8Threads - 1) / kBvh8Threads, device_cu_count() * 4u);
    if (from == 0) {
        hipLaunchKernelGGL(auction ? k_bvh8_top<NXB_SLOT_AUCTION> : k_bvh8_top<NXB_SLOT_GREEDY>, dim3(1),
                           dim3(kBvh8Threads), 0, s, io, cnt);
        from = kBvh8TopLevels;
        count = count > kBvh8TopLevels ? count - kBvh8TopLevels : 0u;
    }
    auto level = auction ? k_bvh8_level<NXB_SLOT_AUCTION> : k_bvh8_level<NXB_SLOT_GREEDY>;
    const uint32_t end = min(from + count, kMaxLevels);
    for (uint32_t l = from; l < end; ++l)
        hipLaunchKernelGGL(level, dim3(grid), dim3(kBvh8Threads), 0, s, io, cnt, l);
    return hipGetLastError();
}

// Level counters of a forest: k_bvh8_tree_top counts the first level of the queue.
__global__ void k_bvh8_forest_level_init(uint32_t* cnt) {
    for (uint32_t i = threadIdx.x; i <= kMaxLevels; i += blockDim.x) cnt[i] = 0u;
}

// Node total into the low word of *ctr; a non-empty level past the last one
// launched means the forest was deeper than the launch covered
// (kFlagDeeper: the caller launches again with more levels).
__global__ void k_bvh8_level_total(const uint32_t* cnt, uint32_t levels, unsigned long long* ctr, uint32_t* flags) {
    uint32_t total = 0;
    for (uint32_t l = 0; l < levels; ++l) total += cnt[l];
    *ctr = total;
    if (cnt[levels] != 0) atomic_or_agent(flags, kFlagDeeper);
}

hipError_t launch_bvh8_tree_levels(const nxb_bvh2_node* bvh2, uint32_t n, uint32_t trees, nxb_bvh8_node* out,
                                   uint32_t* prim_idx, uint32_t capacity, uint32_t levels, Bvh8Scratch sc,
                                   uint32_t* cnt, uint64_t* work3, const uint4* info, const uint32_t* mesh_lo,
                                   uint32_t* ids, uint32_t* prims, hipStream_t s) {
    if (n < 2 || trees == 0 || levels < kTreeTopLevels || levels > kMaxLevels || !sc.work2 || !work3 || !info ||
        !mesh_lo || !ids || !prims)
        return hipErrorInvalidValue;
    const uint32_t grid = min((capacity + kBvh8Threads - 1) / kBvh8Threads, device_cu_count() * 3u);
    const bool auction = sc.slot_mode == NXB_SLOT_AUCTION;
    hipLaunchKernelGGL(k_bvh8_forest_level_init, dim3(1), dim3(128), 0, s, cnt);
    auto top = auction ? k_bvh8_tree_top<NXB_SLOT_AUCTION> : k_bvh8_tree_top<NXB_SLOT_GREEDY>;
    hipLaunchKernelGGL(top, dim3((trees + kTopTrees - 1) / kTopTrees), dim3(kBvh8Threads), 0, s, bvh2, n,
                       2 * n - trees, out, prim_idx, capacity, sc.work2, work3, cnt, info, trees, mesh_lo,
                       ids, prims, sc.flags);
    auto level = auction ? k_bvh8_tree_level<NXB_SLOT_AUCTION> : k_bvh8_tree_level<NXB_SLOT_GREEDY>;
    for (uint32_t l = kTreeTopLevels; l < levels; ++l)
        hipLaunchKernelGGL(level, dim3(grid), dim3(kBvh8Threads), 0, s, bvh2, 2 * n - trees, out, prim_idx,
                           capacity, sc.work2, work3, cnt, l, info, trees, ids, prims, sc.flags);
    hipLaunchKernelGGL(k_bvh8_level_total, dim3(1), dim3(1), 0, s, cnt, levels, sc.ctr, sc.flags);
    return hipGetLastError();
}

uint32_t bvh8_launches(uint32_t n, const uint32_t* cnt_host, uint32_t below_host, uint32_t launched,
                       uint32_t* node_total) {
    *node_total = n;
    if (n <= 1) return 1;
    // the counts of launches (levels) up to `launched` are final; an empty
    // one ends the tree
    uint32_t total = bvh8_small(n) ? 0u : 1u;
    for (uint32_t l = 1; l <= launched; ++l) {
        if (cnt_host[l] == 0) {
            *node_total = bvh8_small(n) ? 1u + below_host : total;
            return l;
        }
        total += cnt_host[l];
    }
    return 0;
}

hipError_t launch_bvh8(const nxb_bvh2_node* bvh2, uint32_t n, nxb_bvh8_node* out, uint32_t* prim_idx,
                       uint32_t capacity, uint32_t spin_limit, Bvh8Scratch sc, hipStream_t s) {
    hipError_t e = launch_bvh8_prep(n, capacity, sc, s);
    if (e != hipSuccess) return e;
    return launch_bvh8_run(bvh2, n, out, prim_idx, capacity, spin_limit, sc, s);
}

}  // namespace nxb
