// trace.hip — closest-hit traversal of the LBVH on gfx950 (the extend phase
// of the wavefront path tracer and the parity entry aurora_trace_closest).
//
// Two persistent kernels, both over grids sized to the resident capacity of
// the chip, whose waves claim rays from WaveClaims' counters:
//   k_query / k_extend_group  the group walk (traverse.hpp): four lanes per ray
//     on the four-wide tree.  Uncounted ray queries, but those of many rays on
//     small scenes (k_query_lanes, one lane per ray; query_walk says which), and
//     the bounces of renders of larger scenes.
//   k_extend  one lane per ray: the binary tree (render bounces), the four-wide
//     tree for small scenes' bounces, and every run that counts fetches (their
//     counts are those of this visit order).  When enough lanes of a wave64
//     have finished, the wave hands out new rays by ballot rank.  A four-wide
//     step fetches a 128-byte node (one cache line, four child boxes), tests
//     the four slabs, intersects leaf primitives at once and descends to the
//     nearest hit child, pushing the others farthest first.  The stack lives in
//     LDS (kLds entries per lane, laid out [level][thread] so a wave's pushes
//     hit 64 consecutive banks) and spills deeper levels to a per-thread global
//     array.
//
// What the group walk gave (queries of random rays in a row, one lane per ray
// before -> after): 2^20 sorted rays on 1.2 M overlapping primitives 12.0 -> 6.4
// ms; 2^20 rays on 190 k scattered primitives 0.80 -> 0.54 ms; 100,001 rays on a
// serving scene of 50 k 226 -> 67 us; 1000 rays on 485 spheres 73 -> 5 us (13 us for
// one call alone), of which the packing kernels and the upload of a scene record,
// with its synchronisation, were 40.  The first of these issues 4.26e9 VALU
// instructions at 645 G/s (one kind alone reaches 614 G/s, pairs 1229) with 52 of
// 64 lanes active; 27 of 64 before, when the L1 address path was busy 75% of the
// time.
//
// Reference counterpart: the per-ray linear scan over all triangles,
// experiments/rt.cpp:209-218, with are::Triangle::intersect_ray
// (src/object/triangle.cpp:82-121) as the primitive test.
#include "internal.hpp"
#include "traverse.hpp"

namespace aur {

namespace {

constexpr int kBlock = 256;
constexpr int kLds = 16;
constexpr int kMaxStack = 96;  // three pushes per level of a tree of depth <= 64
constexpr int kRefill = 8;
constexpr uint32_t kPickWord = 1;  // of the work counters (which are kPoolStride apart): the walk that k_query_pick took
constexpr uint32_t kNone = 0xffffffffu;
constexpr uint32_t kNoPrim = 0x7fffffffu;

// ONE: every ray belongs to the first scene record, whose fields are then
// wave-uniform (scalar registers, loaded once); otherwise each claimed ray
// loads its scene's record.
//
// WIDE: walk the four-wide tree (ray queries, memory bound); otherwise the
// binary tree, one 64-byte child pair per step (render bounces, issue bound).
template <bool COUNT, bool ONE, bool WIDE>
__global__ __launch_bounds__(kBlock) void k_extend(ExtendArgs a) {
    __shared__ uint32_t stk[kLds][kBlock];
    const uint32_t n = a.count ? *a.count : a.n;
    if (a.zero_after && blockIdx.x == 0 && threadIdx.x == 0) *a.zero_after = 0u;
    const int tid = threadIdx.x;
    const int lane = tid & 63;
    uint32_t* spill = a.spill + (size_t)blockIdx.x * kBlock + tid;
    const size_t sstride = a.spill_stride;
    const float tmax = a.tmax;
    float tmin = 0.0f;  // the scene's ray offset
    // the scene of the lane's current ray
    const float4* N = nullptr;  // the wide nodes (WIDE) or the binary nodes
    const float4* S = nullptr;
    const float4* Qd = nullptr;
    uint32_t n_spheres = 0, n_nodes = 0, n_prims = 0;
    if constexpr (ONE) {
        const SceneRec& rec = a.recs[0];
        tmin = rec.tmin;
        N = WIDE ? rec.sc.wide : rec.sc.nodes;
        S = rec.sc.spheres;
        Qd = rec.sc.quads;
        n_spheres = rec.sc.n_spheres;
        n_nodes = WIDE ? rec.sc.n_wide : rec.sc.n_nodes;
        n_prims = rec.sc.n_spheres + rec.sc.n_quads;
    }

    uint32_t ri = kNone;
    bool done = false;
    v3 o = V(0, 0, 0), d = V(0, 0, 0), inv = V(0, 0, 0);
    float best_t = tmax;
    uint32_t best_id = kNoPrim;
    uint32_t cur = 0;
    int sp = 0;
    uint32_t cn = 0, cs = 0, cq = 0;                  // per-ray counts
    unsigned long long tn = 0, ts = 0, tq = 0;        // per-lane totals

    // te: the entry distance of the primitive's box; a hit before it does not
    // count (this makes the closest hit independent of the visit order)
    // (an id past the primitives, which no well-formed tree holds, reads
    // primitive 0 and is neither counted nor taken)
    auto test_prim = [&](uint32_t id, float te) {
        const bool valid = id < n_prims;
        const uint32_t k = valid ? id : 0u;
        float t = 0.0f;
        bool h;
        if (k < n_spheres) {
            if (COUNT) cs += valid ? 1u : 0u;
            h = hit_sphere_t(ldg4(S, k), o, d, tmin, tmax, t);
        } else {
            if (COUNT) cq += valid ? 1u : 0u;
            const size_t q = 3 * (size_t)(k - n_spheres);
            h = hit_quad_t(ldg4(Qd, q), ldg4(Qd, q + 1), ldg4(Qd, q + 2), o, d, tmin, tmax, t);
        }
        const bool take = valid & h & (t >= te) & ((t < best_t) | ((t == best_t) & (id < best_id)));
        best_t = take ? t : best_t;
        best_id = take ? id : best_id;
    };
    auto finish = [&]() {
        const bool miss = best_id == kNoPrim;
        a.hit[ri] = make_float2(miss ? tmax : best_t, __int_as_float(miss ? AURORA_MISS : (int)best_id));
        if (COUNT) {
            if (a.counts) {
                a.counts[3 * (size_t)ri] = cn;
                a.counts[3 * (size_t)ri + 1] = cs;
                a.counts[3 * (size_t)ri + 2] = cq;
            }
            tn += cn;
            ts += cs;
            tq += cq;
        }
        ri = kNone;
    };

    WaveClaims claims;
    claims.init(a.pool, n, 64u);
    for (;;) {
        const bool idle = (ri == kNone) && !done;
        const uint64_t im = __ballot(idle);
        const uint64_t am = __ballot(ri != kNone);
        if (im != 0 && (am == 0 || __popcll(im) >= kRefill)) {
            claims.refill();
            const uint32_t avail = claims.next < claims.end ? claims.end - claims.next : 0u;
            const uint32_t rank = lanes_below(im);
            if (idle) {
                if (avail == 0) {
                    done = true;
                } else if (rank < avail) {
                    ri = claims.next + rank;
                    if (a.order) ri = a.order[ri];
                    const float4 ro = a.ray_o[ri], rd = a.ray_d[ri];
                    o = xyz(ro);
                    d = xyz(rd);
                    if constexpr (!ONE) {
                        const SceneRec& rec = a.recs[__float_as_uint(rd.w)];
                        tmin = rec.tmin;
                        N = WIDE ? rec.sc.wide : rec.sc.nodes;
                        S = rec.sc.spheres;
                        Qd = rec.sc.quads;
                        n_spheres = rec.sc.n_spheres;
                        n_nodes = WIDE ? rec.sc.n_wide : rec.sc.n_nodes;
                        n_prims = rec.sc.n_spheres + rec.sc.n_quads;
                    }
                    inv = V(rcp_rn(d.x), rcp_rn(d.y), rcp_rn(d.z));
                    best_t = tmax;
                    best_id = kNoPrim;
                    sp = 0;
                    cn = cs = cq = 0;
                    if (n_nodes == 0) {
                        finish();
                    } else if constexpr (WIDE) {
                        cur = 0;  // the root of the four-wide tree
                    } else {
                        const float4 r0 = ldg4(N, 0), r1 = ldg4(N, 1);
                        if (COUNT) ++cn;
                        float tr;
                        const uint32_t rc = __float_as_uint(r0.w);
                        if (!slab(r0, r1, o, inv, tmin, best_t, tr)) {
                            finish();
                        } else if (rc & AURORA_NODE_LEAF) {
                            test_prim(rc & ~AURORA_NODE_LEAF, tr);
                            finish();
                        } else {
                            cur = rc;
                        }
                    }
                }
            }
            claims.next += min(avail, (uint32_t)__popcll(im));
        }
        if (__ballot((ri != kNone) || !done) == 0) break;
        if (ri == kNone) continue;

        auto push = [&](uint32_t v) {
            // the tree is shallow enough that the bound only keeps every
            // access inside the stack arrays
            if (sp < kLds) stk[sp][tid] = v;
            else if (sp < kMaxStack) spill[(size_t)(sp - kLds) * sstride] = v;
            if (sp < kMaxStack) ++sp;
        };
        auto pop_or_finish = [&]() {
            if (sp == 0) {
                finish();
            } else {
                --sp;
                if (sp < kLds) cur = stk[sp][tid];
                else cur = ldg1(spill, (size_t)(sp - kLds) * sstride);
            }
        };
        if constexpr (WIDE) {
            // a well-formed tree only refers to nodes below n_wide; any other
            // value ends the ray instead of reading out of bounds
            if (cur >= n_nodes) {
                finish();
                continue;
            }
            // one step: the four slots of wide node cur
            uint32_t r0, r1, r2, r3;
            const int m = wide_step(N, cur, o, inv, tmin, best_t, test_prim, r0, r1, r2, r3);
            if (COUNT) cn += 4;
            if (m == 0) {
                pop_or_finish();
                continue;
            }
            // the others farthest first
            if (m > 3) push(r3);
            if (m > 2) push(r2);
            if (m > 1) push(r1);
            cur = r0;
        } else {
            // a well-formed tree only holds even pair indices below n_nodes;
            // any other value ends the ray instead of reading out of bounds
            if ((cur & 1u) || cur + 1 >= n_nodes) {
                finish();
                continue;
            }
            // one step: the child pair at nodes[cur], nodes[cur+1]
            const float4 a0 = ldg4(N, 2 * (size_t)cur), a1 = ldg4(N, 2 * (size_t)cur + 1);
            const float4 b0 = ldg4(N, 2 * (size_t)cur + 2), b1 = ldg4(N, 2 * (size_t)cur + 3);
            if (COUNT) cn += 2;
            float ta, tb;
            bool ha = slab(a0, a1, o, inv, tmin, best_t, ta);
            bool hb = slab(b0, b1, o, inv, tmin, best_t, tb);
            const uint32_t ca = __float_as_uint(a0.w), cb = __float_as_uint(b0.w);
            if (ha && (ca & AURORA_NODE_LEAF)) {
                test_prim(ca & ~AURORA_NODE_LEAF, ta);
                ha = false;
            }
            if (hb && (cb & AURORA_NODE_LEAF)) {
                test_prim(cb & ~AURORA_NODE_LEAF, tb);
                hb = false;
            }
            if (ha && hb) {
                const bool bnear = tb < ta;
                push(bnear ? ca : cb);
                cur = bnear ? cb : ca;
            } else if (ha) {
                cur = ca;
            } else if (hb) {
                cur = cb;
            } else {
                pop_or_finish();
            }
        }
    }
    if (COUNT && a.totals) {
#pragma unroll
        for (int off = 32; off >= 1; off >>= 1) {
            tn += __shfl_xor(tn, off);
            ts += __shfl_xor(ts, off);
            tq += __shfl_xor(tq, off);
        }
        if (lane == 0) {
            atomicAdd(&a.totals[0], tn);
            atomicAdd(&a.totals[1], ts);
            atomicAdd(&a.totals[2], tq);
        }
    }
}

constexpr int kGroupFlush = 48;   // lanes with a leaf before leaves are tested (32: 6848, 40: 6761, 48: 6754 us)


// Closest hits over the four-wide tree by the group walk.  IO names the rays,
// their scenes and where the hits go.  A wave fetches kGroupBatch rays at a
// time, one per lane and one batch ahead, and keeps them in shared memory for
// its groups: fetched by the group that takes it, each ray stopped all 16
// walks for a memory latency (short walks then ran at a quarter of the speed).
constexpr int kGroupBatch = 16;   // 32 and 64 leave room for fewer waves (sorted queries 6.6, 7.0, 7.8 ms)
struct QueryShared {
    GroupShared g;
    float ray[9][kGroupBatch];
    uint32_t id[kGroupBatch], scene[kGroupBatch];
};
template <class IO>
__device__ __forceinline__ void group_trace(const IO& io, uint32_t n, uint32_t* pool, float tmax, uint32_t* spill,
                                            uint32_t spill_stride) {
    __shared__ QueryShared shared[kBlock / 64];
    const int lane = threadIdx.x & 63, ray = lane >> 2, slot = lane & 3;
    QueryShared& sh = shared[threadIdx.x >> 6];
    const size_t stride = spill_stride / 4;
    GroupWalk w;
    group_init(w, sh.g, spill + 2 * (size_t)(blockIdx.x * kGroupBlockRays + (threadIdx.x >> 2)), ray, slot);
    GroupScene sc = io.scene();
    WaveClaims claims;
    claims.init(pool, n, kGroupRays);
    uint32_t ri = kNone;
    uint32_t head = 0, tail = 0;  // the batch's rays not yet taken
    // the next batch, in registers
    v3 no = V(0, 0, 0), nd = V(0, 0, 0);
    uint32_t ni = 0, ns = 0, n_next = 0;
    auto fetch = [&]() {
        claims.refill();
        n_next = claims.next < claims.end ? min(claims.end - claims.next, (uint32_t)kGroupBatch) : 0u;
        if ((uint32_t)lane < n_next) ni = io.ray(claims.next + lane, no, nd, ns);
        claims.next += n_next;
    };
    fetch();
    for (;;) {
        const uint64_t im = __ballot(ri == kNone);
        if (im != 0) {
            if (head == tail && n_next != 0) {
                if ((uint32_t)lane < n_next) {
                    sh.ray[0][lane] = no.x;
                    sh.ray[1][lane] = no.y;
                    sh.ray[2][lane] = no.z;
                    sh.ray[3][lane] = nd.x;
                    sh.ray[4][lane] = nd.y;
                    sh.ray[5][lane] = nd.z;
                    sh.ray[6][lane] = rcp_rn(nd.x);
                    sh.ray[7][lane] = rcp_rn(nd.y);
                    sh.ray[8][lane] = rcp_rn(nd.z);
                    sh.id[lane] = ni;
                    if constexpr (!IO::kOneScene) sh.scene[lane] = ns;
                }
                head = 0;
                tail = n_next;
                group_sync();
                fetch();
            }
            if (head < tail) {
                const uint32_t at = head + (lanes_below(im) >> 2);
                if (ri == kNone && at < tail) {
                    ri = sh.id[at];
                    if constexpr (!IO::kOneScene) sc = io.scene(sh.scene[at]);
                    group_begin(w, sh.g, sc, V(sh.ray[0][at], sh.ray[1][at], sh.ray[2][at]),
                                V(sh.ray[3][at], sh.ray[4][at], sh.ray[5][at]),
                                V(sh.ray[6][at], sh.ray[7][at], sh.ray[8][at]), tmax, ray, slot);
                }
                head = min(tail, head + ((uint32_t)__popcll(im) >> 2));
            } else if (im == ~0ull) {
                break;
            }
        }
        group_sync();
        group_step<IO::kOneScene>(w, sh.g, sc, ray, slot, stride);
        group_sync();
        // leaves are tested when enough lanes have one, when a ray has no room
        // for more, or when no ray can go on without
        const uint64_t pend = __ballot(group_pending(w, slot));
        if (pend != 0 && (__popcll(pend) >= kGroupFlush || __ballot(group_full(w)) != 0 ||
                          __ballot(group_walking(w)) == 0))
            group_leaves(w, sh.g, sc, tmax, ray, slot);
        if (w.st == 0u && ri != kNone) {
            const bool miss = w.best_id == kNoPrim;
            if (slot == 0) io.hit(ri, miss ? tmax : w.best_t, miss ? AURORA_MISS : (int)w.best_id);
            ri = kNone;
        }
    }
}

struct QueryIO {
    static constexpr bool kOneScene = true;
    const QueryArgs& a;
    __device__ __forceinline__ GroupScene scene() const { return a.sc; }
    __device__ __forceinline__ uint32_t ray(uint32_t i, v3& o, v3& d, uint32_t&) const {
        if (a.order) i = a.order[i];
        o = load3(a.org, i);
        d = load3(a.dir, i);
        return i;
    }
    __device__ __forceinline__ void hit(uint32_t i, float t, int prim) const {
        a.t[i] = t;
        a.prim[i] = prim;
    }
};
__global__ __launch_bounds__(kBlock) void k_query(QueryArgs a) {
    if (a.pick && a.pool[kPickWord] != 0u) return;
    group_trace(QueryIO{a}, a.n, a.pool, a.tmax, a.spill, a.spill_stride);
}

// The same with one lane per ray.  Where the rays of a wave go the same way its
// 64 lanes walk together, and the group walk's four lanes per ray only give the
// wave a quarter of the rays (query_walk has the figures).
__global__ __launch_bounds__(kBlock) void k_query_lanes(QueryArgs a) {
    if (a.pick && a.pool[kPickWord] == 0u) return;
    __shared__ uint32_t stk[kTravLds * kBlock];
    const QueryIO io{a};
    uint32_t* spill = a.spill + (size_t)blockIdx.x * kBlock + threadIdx.x;
    DevScene sc{};
    sc.wide = a.sc.wide;
    sc.spheres = a.sc.spheres;
    sc.quads = a.sc.quads;
    sc.n_wide = a.sc.n_wide;
    sc.n_spheres = a.sc.n_spheres;
    sc.n_quads = a.sc.n_prims - a.sc.n_spheres;
    uint32_t ri = kNone;
    bool done = false;
    v3 o = V(0, 0, 0), d = V(0, 0, 0);
    WideWalk w{};
    WaveClaims claims;
    claims.init(a.pool, a.n, 64u);
    for (;;) {
        const bool idle = (ri == kNone) && !done;
        const uint64_t im = __ballot(idle);
        const uint64_t am = __ballot(ri != kNone);
        if (im != 0 && (am == 0 || __popcll(im) >= kRefill)) {
            claims.refill();
            const uint32_t avail = claims.next < claims.end ? claims.end - claims.next : 0u;
            const uint32_t rank = lanes_below(im);
            if (idle) {
                if (avail == 0) {
                    done = true;
                } else if (rank < avail) {
                    uint32_t sid = 0u;
                    ri = io.ray(claims.next + rank, o, d, sid);
                    wide_walk_start(w, d, a.tmax);
                }
            }
            claims.next += min(avail, (uint32_t)__popcll(im));
        }
        if (__ballot((ri != kNone) || !done) == 0) break;
        if (ri == kNone) continue;
        if (wide_walk_step(w, sc, o, d, a.sc.tmin, a.tmax, stk + threadIdx.x, kBlock, spill, a.spill_stride)) {
            float t;
            int prim;
            wide_walk_result(w, a.tmax, t, prim);
            io.hit(ri, t, prim);
            ri = kNone;
        }
    }
}

// Clears the work counters and decides which of the two walks runs: 1024 pairs of
// rays that a wave would hold together, 31 places apart in claim order; lanes when
// three quarters of them start within a sixteenth of the scene's extent and go
// within 8 degrees (a pinhole image's neighbours do, also past the ends of its
// rows; random, bounced or shadow rays of an area light do not).
__global__ __launch_bounds__(1024) void k_query_pick(QueryArgs a) {
    const uint32_t i = threadIdx.x;
    if (i < kPools) a.pool[kPoolStride * i] = 0u;
    const QueryIO io{a};
    const uint32_t p = (uint32_t)(((uint64_t)a.n * i) / 1024u);
    v3 o0, d0, o1, d1;
    uint32_t sid = 0u;
    (void)io.ray(p, o0, d0, sid);
    (void)io.ray(min(a.n - 1u, p + 31u), o1, d1, sid);
    const float4 lo = a.box[0], hi = a.box[1];
    const float reach = fmaxf(fmaxf(hi.x - lo.x, hi.y - lo.y), hi.z - lo.z) * 0.0625f;
    const v3 s = o1 - o0;
    const float c = dot(d0, d1);
    const bool same = dot(s, s) <= reach * reach && c > 0.0f && (c * c >= 0.98f * dot(d0, d0) * dot(d1, d1));
    const int n_same = __syncthreads_count(same);
    if (i == 0) a.pool[kPickWord] = n_same >= 768 ? 1u : 0u;
}

// the live queue of a wavefront bounce
template <bool ONE>
struct QueueIO {
    static constexpr bool kOneScene = ONE;
    const ExtendArgs& a;
    __device__ __forceinline__ GroupScene scene() const { return ONE ? group_scene(a.recs[0]) : GroupScene{}; }
    __device__ __forceinline__ GroupScene scene(uint32_t sid) const { return group_scene(a.recs[sid]); }
    __device__ __forceinline__ uint32_t ray(uint32_t i, v3& o, v3& d, uint32_t& sid) const {
        const float4 ro = a.ray_o[i], rd = a.ray_d[i];
        o = xyz(ro);
        d = xyz(rd);
        sid = __float_as_uint(rd.w);
        return i;
    }
    __device__ __forceinline__ void hit(uint32_t i, float t, int prim) const {
        a.hit[i] = make_float2(t, __int_as_float(prim));
    }
};
template <bool ONE>
__global__ __launch_bounds__(kBlock) void k_extend_group(ExtendArgs a) {
    if (a.zero_after && blockIdx.x == 0 && threadIdx.x == 0) *a.zero_after = 0u;
    group_trace(QueueIO<ONE>{a}, a.count ? *a.count : a.n, a.pool, a.tmax, a.spill, a.spill_stride);
}

__global__ void k_clear_pool(uint32_t* pool) {
    if (threadIdx.x < kPools) pool[kPoolStride * threadIdx.x] = 0u;
}

__global__ __launch_bounds__(kBlock) void k_brute(DevScene sc, const float4* ro, const float4* rd, uint32_t n,
                                                  float tmin, float tmax, float2* hit) {
    const uint32_t i = blockIdx.x * kBlock + threadIdx.x;
    if (i >= n) return;
    const v3 o = xyz(ro[i]), d = xyz(rd[i]);
    const v3 inv = V(rcp_rn(d.x), rcp_rn(d.y), rcp_rn(d.z));
    float best_t = tmax;
    uint32_t best_id = kNoPrim;
    const uint32_t np = sc.n_spheres + sc.n_quads;
    for (uint32_t id = 0; id < np; ++id) {
        // the rule of the tree traversals: the ray must enter the
        // primitive's box, and a hit before the box's entry does not count
        v3 lo, hi;
        prim_box(sc, id, lo, hi);
        float te;
        if (!slab(make_float4(lo.x, lo.y, lo.z, 0.0f), make_float4(hi.x, hi.y, hi.z, 0.0f), o, inv, tmin, tmax, te))
            continue;
        float t;
        bool h;
        if (id < sc.n_spheres) {
            h = hit_sphere(sc.spheres[id], o, d, tmin, tmax, t);
        } else {
            const float4* q = sc.quads + 3 * (size_t)(id - sc.n_spheres);
            float al, be;
            h = hit_quad(q[0], q[1], q[2], o, d, tmin, tmax, t, al, be);
        }
        if (h && t >= te && (t < best_t || (t == best_t && id < best_id))) {
            best_t = t;
            best_id = id;
        }
    }
    const bool miss = best_id == kNoPrim;
    hit[i] = make_float2(miss ? tmax : best_t, __int_as_float(miss ? AURORA_MISS : (int)best_id));
}

__device__ __forceinline__ uint32_t spread9(uint32_t v) {
    // bits 0..8 of v to every third bit
    v &= 0x1ffu;
    v = (v | (v << 16)) & 0x030000ffu;
    v = (v | (v << 8)) & 0x0300f00fu;
    v = (v | (v << 4)) & 0x030c30c3u;
    v = (v | (v << 2)) & 0x09249249u;
    return v;
}

__device__ __forceinline__ uint32_t cell9(float x, float lo, float hi) {
    const float e = hi - lo;
    const float u = e > 0.0f ? (x - lo) / e : 0.0f;
    return (uint32_t)fminf(fmaxf(u * 512.0f, 0.0f), 511.0f);
}

__global__ __launch_bounds__(kBlock) void k_ray_keys(const float* ro, const float* rd, uint32_t n,
                                                     const float4* nodes, uint32_t* keys, uint32_t* vals) {
    const uint32_t i = blockIdx.x * kBlock + threadIdx.x;
    if (i >= n) return;
    const float4 lo = nodes[0], hi = nodes[1];
    const v3 o = load3(ro, i), d = load3(rd, i);
    const uint32_t m = (spread9(cell9(o.x, lo.x, hi.x)) << 2) | (spread9(cell9(o.y, lo.y, hi.y)) << 1) |
                       spread9(cell9(o.z, lo.z, hi.z));
    const uint32_t oct = (d.x < 0.0f ? 4u : 0u) | (d.y < 0.0f ? 2u : 0u) | (d.z < 0.0f ? 1u : 0u);
    keys[i] = (m << 3) | oct;
    vals[i] = i;
}

}  // namespace

Status launch_ray_keys(const float* ro, const float* rd, uint32_t n, const float4* nodes, uint32_t* keys,
                       uint32_t* vals, hipStream_t s) {
    if (n == 0) return Status::ok();
    k_ray_keys<<<(n + kBlock - 1) / kBlock, kBlock, 0, s>>>(ro, rd, n, nodes, keys, vals);
    AUR_HIP(hipGetLastError());
    return Status::ok();
}

static_assert(kExtendBlock == kBlock && kExtendSpillLevels >= kMaxStack - kLds, "extend shape constants");
int extend_block() { return kBlock; }
int extend_spill_levels() { return kExtendSpillLevels; }

Status launch_extend(const ExtendArgs& a, int grid, hipStream_t s) {
    if ((size_t)grid * kBlock > a.spill_stride) return Status{AURORA_ERR_RUNTIME, "extend grid exceeds spill stride"};
    const bool count = a.counts || a.totals;
    const int v = (count ? 4 : 0) | (a.one_scene ? 2 : 0) | (a.wide ? 1 : 0);
    void (*const ks[8])(ExtendArgs) = {k_extend<false, false, false>, k_extend<false, false, true>,
                                       k_extend<false, true, false>,  k_extend<false, true, true>,
                                       k_extend<true, false, false>,  k_extend<true, false, true>,
                                       k_extend<true, true, false>,   k_extend<true, true, true>};
    if (a.group && a.wide && !count) {
        auto k = a.one_scene ? k_extend_group<true> : k_extend_group<false>;
        k<<<grid, kBlock, 0, s>>>(a);
    } else {
        ks[v]<<<grid, kBlock, 0, s>>>(a);
    }
    AUR_HIP(hipGetLastError());
    return Status::ok();
}

// Which walk a query takes (us; camera: the rays of a 512x512 pinhole image,
// random: 262,144 and 2^20 rays of random origin and direction).
// - As many rays as the group walk's grid holds, or fewer: group.  The call is
//   as long as its longest ray, and four lanes shorten it: 10^5 camera rays on 500,
//   8 k and 50 k primitives 26, 52, 88 against 73, 118, 168 by lanes (packing them),
//   random ones 33, 74, 123 against 98, 157, 241.
// - Fewer than 1,024 primitives: lanes.  500 primitives: camera 120 by groups, 62 by
//   lanes; random 107 and 239, 88 and 211.
// - 32,768 or more: group.  50 k primitives: camera 174 and, by lanes, 209; random 211
//   and 443, 295 and 592.
// - Between these, lanes where the rays of a wave go the same way and groups where
//   they do not.  2,000 primitives: camera 155 by groups, 82 by lanes; 2^21 random
//   rays 449 and 486.  8,000: camera 175 and 125; random 161 and 335, 201 and 430.
//   The look at the rays and the idle walk's launch cost 3 to 8 us.
constexpr uint32_t kLaneAlwaysPrims = 1024, kLaneMaxPrims = 32768;
QueryWalk query_walk(uint32_t n, uint32_t n_prims, uint32_t groups) {
    if (n <= groups || n_prims >= kLaneMaxPrims) return QueryWalk::Group;
    return n_prims < kLaneAlwaysPrims ? QueryWalk::Lanes : QueryWalk::Pick;
}

size_t query_spill_bytes(QueryWalk walk, int blocks) {
    return walk == QueryWalk::Lanes ? (size_t)blocks * kBlock * (kTravMaxStack - kTravLds) * 4
                                    : (size_t)blocks * kGroupBlockRays * kGroupSpillBytes;
}
static_assert(kGroupSpillBytes == (kGroupMaxStack - kGroupStack) * 8 &&
                  kGroupBlockRays * kGroupSpillBytes <= kBlock * kExtendSpillLevels * 4,
              "group spill: no more than k_extend_group's share of ExtendArgs::spill");

Status launch_query(const QueryArgs& args, QueryWalk walk, int group_grid, int lane_grid, hipStream_t s) {
    QueryArgs a = args;
    a.pick = walk == QueryWalk::Pick ? 1u : 0u;
    if (walk == QueryWalk::Group && (uint64_t)group_grid * kGroupBlockRays >= a.n)
        a.pool = nullptr;  // one ray per place: nothing to claim
    else if (a.pick)
        k_query_pick<<<1, 1024, 0, s>>>(a);
    else
        k_clear_pool<<<1, 64, 0, s>>>(a.pool);
    if (walk != QueryWalk::Group) {
        a.spill_stride = (uint32_t)(lane_grid * kBlock);
        k_query_lanes<<<lane_grid, kBlock, 0, s>>>(a);
    }
    if (walk != QueryWalk::Lanes) {
        a.spill_stride = (uint32_t)(group_grid * kBlock);
        k_query<<<group_grid, kBlock, 0, s>>>(a);
    }
    AUR_HIP(hipGetLastError());
    return Status::ok();
}

Status launch_brute(const DevScene& sc, const float4* o, const float4* d, uint32_t n, float tmin, float tmax,
                    float2* hit, hipStream_t s) {
    if (n == 0) return Status::ok();
    k_brute<<<(n + kBlock - 1) / kBlock, kBlock, 0, s>>>(sc, o, d, n, tmin, tmax, hit);
    AUR_HIP(hipGetLastError());
    return Status::ok();
}

}  // namespace aur
