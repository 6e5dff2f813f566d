// BVH8 traversal kernels of the HIP intersector (gfx950, wave64).
//
// k_closest*    : closest hit, replaces EmbreeAccel::intersect
//                 (reference src/core/accel.cpp:348-407; interface
//                 HitableInterface::intersect, src/core/hitable.h:12-13)
// k_occluded*   : any hit in [tmin, tmax], replaces HitableInterface::occluded
//                 (src/core/hitable.h:15-33)
// k_trace_pair  : both, for one bounce of the integrator
//
// Design:
//  - persistent lanes: every lane owns one ray at a time; finished lanes are
//    refilled from a global ray counter, one atomic per wave (ballot +
//    prefix count), so incoherent rays do not leave idle lanes behind;
//  - a per-lane short stack in LDS (kStack group entries); deeper entries
//    spill to a per-lane region in HBM, so any BVH depth works;
//  - 128-byte nodes: seven 16-byte loads per visit (each lane loads its own
//    near and far planes by the ray's octant; the leaf words are read only
//    when leaf children are tested), 16-bit child boxes decoded with one fma
//    per plane; the nearest hit inner child is visited next and the others go
//    on the stack as one group, visited in octant order (children sit in
//    octant slots) and culled as a group by their nearest entry distance;
//  - watertight ray/triangle test (Woop, Benthin, Wald 2013) with contraction
//    disabled, so its result is bit-identical to the host oracle's;
//  - closest hit is the smallest t, ties broken by the lowest primitive
//    index, which makes the answer independent of traversal order.
#include <hip/hip_runtime.h>

#include <mutex>

#include "kp_feed.h"
#include "kp_kernels.h"
#include "kp_layout.h"

#pragma clang fp contract(off)

namespace kp {

// Scratch of the allocation-free closest-hit entry point
// (kp_intersect_closest_noalloc): work counter at byte 0, error word at byte
// 256, per-lane stack spill area from byte KP_SCRATCH_SPILL_OFFSET.  Each
// device holds its own copy for the life of the process; host code must use
// the address noalloc_scratch() returns for the device, never this name.
static __device__ __align__(256) unsigned char scratch[KP_SCRATCH_BYTES];

hipError_t noalloc_scratch(int device, void** ptr) {
    static std::mutex mu;
    static void* per_device[KP_SCRATCH_MAX_DEVICES] = {};
    if (device < 0 || device >= KP_SCRATCH_MAX_DEVICES) return hipErrorInvalidDevice;
    std::lock_guard<std::mutex> lock(mu);
    if (!per_device[device]) {
        // the caller has made `device` current
        void* p = nullptr;
        const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (e != hipSuccess) return e;
        per_device[device] = p;
    }
    *ptr = per_device[device];
    return hipSuccess;
}


struct RayPre {
    float ox, oy, oz, tmin, dx, dy, dz, tmax;
    float ix, iy, iz;
    float Sx, Sy, Sz;
    uint32_t k;   // the triangle test's axes: kx | ky << 2 | kz << 4
};

__device__ __forceinline__ float pick3(float a, float b, float c, int k) {
    return k == 0 ? a : (k == 1 ? b : c);
}

__device__ __forceinline__ float safe_rcp(float d) {
    float dd = fabsf(d) < 1e-20f ? copysignf(1e-20f, d) : d;
    return 1.0f / dd;
}

__device__ __forceinline__ float fast_rcp(float d) {
    const float dd = fabsf(d) < 1e-20f ? copysignf(1e-20f, d) : d;
    const float q = __builtin_amdgcn_rcpf(dd);
    return fmaf(fmaf(-dd, q, 1.0f), q, q);
}

// Rays with a non-finite origin or direction, a zero direction or a NaN
// interval bound miss everything (same rule as the oracle).
__device__ __forceinline__ bool ray_valid(const float4 a, const float4 b) {
    const bool fin = isfinite(a.x) && isfinite(a.y) && isfinite(a.z) && isfinite(b.x) &&
                     isfinite(b.y) && isfinite(b.z);
    const bool nz = b.x != 0.0f || b.y != 0.0f || b.z != 0.0f;
    return fin && nz && !isnan(a.w) && !isnan(b.w);
}

__device__ __forceinline__ void setup_ray(const float4 a, const float4 b, RayPre& r) {
    r.ox = a.x; r.oy = a.y; r.oz = a.z; r.tmin = a.w;
    r.dx = b.x; r.dy = b.y; r.dz = b.z; r.tmax = b.w;
    const float ax = fabsf(r.dx), ay = fabsf(r.dy), az = fabsf(r.dz);
    int kz = (ax >= ay) ? ((ax >= az) ? 0 : 2) : ((ay >= az) ? 1 : 2);
    int kx = (kz == 2) ? 0 : kz + 1;
    int ky = (kx == 2) ? 0 : kx + 1;
    const float dkz = pick3(r.dx, r.dy, r.dz, kz);
    if (dkz < 0.0f) { int t = kx; kx = ky; ky = t; }
    r.k = (uint32_t)(kx | ky << 2 | kz << 4);
    r.Sx = pick3(r.dx, r.dy, r.dz, kx) / dkz;
    r.Sy = pick3(r.dx, r.dy, r.dz, ky) / dkz;
    r.Sz = 1.0f / dkz;
    // Reciprocals for the box tests only: the hardware estimate (1 ulp) and one
    // Newton step, within a hair of the rounded quotient; the boxes' widening
    // covers far more.  The estimate flushes denormal results, so a direction
    // that large (practically never) takes the divisions.
    r.ix = fast_rcp(r.dx);
    r.iy = fast_rcp(r.dy);
    r.iz = fast_rcp(r.dz);
    if (__ballot(fmaxf(fmaxf(ax, ay), az) > 1e37f) != 0ull) {
        r.ix = safe_rcp(r.dx);
        r.iy = safe_rcp(r.dy);
        r.iz = safe_rcp(r.dz);
    }
}

// Watertight test; same operation order as the host oracle.
__device__ __forceinline__ bool tri_test(const RayPre& r, const float4 a, const float4 b,
                                         const float4 c, float tmax_incl, float& t_out,
                                         float& u_out, float& v_out) {
    const int kx = (int)(r.k & 3u), ky = (int)((r.k >> 2) & 3u), kz = (int)(r.k >> 4);
    const float A0 = a.x - r.ox, A1 = a.y - r.oy, A2 = a.z - r.oz;
    const float B0 = b.x - r.ox, B1 = b.y - r.oy, B2 = b.z - r.oz;
    const float C0 = c.x - r.ox, C1 = c.y - r.oy, C2 = c.z - r.oz;
    const float Akz = pick3(A0, A1, A2, kz), Bkz = pick3(B0, B1, B2, kz), Ckz = pick3(C0, C1, C2, kz);
    const float Ax = pick3(A0, A1, A2, kx) - r.Sx * Akz;
    const float Ay = pick3(A0, A1, A2, ky) - r.Sy * Akz;
    const float Bx = pick3(B0, B1, B2, kx) - r.Sx * Bkz;
    const float By = pick3(B0, B1, B2, ky) - r.Sy * Bkz;
    const float Cx = pick3(C0, C1, C2, kx) - r.Sx * Ckz;
    const float Cy = pick3(C0, C1, C2, ky) - r.Sy * Ckz;
    float U = Cx * By - Cy * Bx;
    float V = Ax * Cy - Ay * Cx;
    float W = Bx * Ay - By * Ax;
    if (U == 0.0f || V == 0.0f || W == 0.0f) {
        const double CxBy = (double)Cx * (double)By, CyBx = (double)Cy * (double)Bx;
        U = (float)(CxBy - CyBx);
        const double AxCy = (double)Ax * (double)Cy, AyCx = (double)Ay * (double)Cx;
        V = (float)(AxCy - AyCx);
        const double BxAy = (double)Bx * (double)Ay, ByAx = (double)By * (double)Ax;
        W = (float)(BxAy - ByAx);
    }
    if ((U < 0.0f || V < 0.0f || W < 0.0f) && (U > 0.0f || V > 0.0f || W > 0.0f)) return false;
    const float det = U + V + W;
    if (det == 0.0f) return false;
    const float Az = r.Sz * Akz, Bz = r.Sz * Bkz, Cz = r.Sz * Ckz;
    const float T = U * Az + V * Bz + W * Cz;
    const float t = T / det;
    if (!(t >= r.tmin && t <= tmax_incl)) return false;
    t_out = t;
    u_out = V / det;
    v_out = W / det;
    return true;
}


// Per-ray node-test constants: the ray direction's octant (bit k set when
// direction k is negative) and the byte offset in a node of each near / far
// plane word (planes lo.x lo.y lo.z hi.x hi.y hi.z are the 16-byte words
// 2..7), one byte each, so each lane loads its own near and far planes
// instead of selecting them per child.
struct NodeTest {
    uint32_t oct;
    uint32_t offa;   // bytes: near x, far x, near y, far y
    uint32_t offb;   // bytes: near z, far z
};

__device__ __forceinline__ NodeTest node_test_setup(const RayPre& r) {
    NodeTest t;
    const bool nx = r.ix < 0.0f, ny = r.iy < 0.0f, nz = r.iz < 0.0f;
    t.oct = (nx ? 1u : 0u) | (ny ? 2u : 0u) | (nz ? 4u : 0u);
    t.offa = (nx ? 0x2050u : 0x5020u) | ((ny ? 0x3060u : 0x6030u) << 16);
    t.offb = nz ? 0x4070u : 0x7040u;
    return t;
}

// The node array as a buffer resource: a node visit addresses its words by
// 32-bit byte offsets from one scalar base (no 64-bit address arithmetic per
// load); the range is left open, as every node index is valid.
typedef __amdgpu_buffer_rsrc_t NodeBuf;

__device__ __forceinline__ NodeBuf node_buffer(const uint4* nodes) {
    return __builtin_amdgcn_make_buffer_rsrc((void*)nodes, (short)0, (int)0xFFFFFFFF, 0x00020000);
}

__device__ __forceinline__ uint4 node_word(NodeBuf nb, uint32_t byte_off) {
    return __builtin_bit_cast(uint4, __builtin_amdgcn_raw_buffer_load_b128(nb, byte_off, 0, 0));
}

// Plane value of a slot: a binary16 integer read straight from its half of
// the word (the fma below becomes one mixed-precision fma, no conversion).
__device__ __forceinline__ float qplane(const uint4& plane, int slot) {
    const uint32_t d = (slot >> 1) == 0 ? plane.x : (slot >> 1) == 1 ? plane.y : (slot >> 1) == 2 ? plane.z : plane.w;
    const unsigned short h = (slot & 1) ? (unsigned short)(d >> 16) : (unsigned short)(d & 0xFFFFu);
    return (float)__builtin_bit_cast(_Float16, h);
}

// Relative widening of a far distance, 2*gamma(3) (Ize 2013): tf + |tf| * eps.
#define KP_FAR_EPS 3.5762793e-7f

// Result of one node visit.
struct NodeHits {
    uint32_t group;      // first inner child | inner mask << 24
    uint32_t inner;      // inner children hit (slot bits)
    uint32_t leaves;     // leaf children hit (slot bits)
    int32_t near_key;    // (tnear key | slot) of the nearest inner child hit
    int32_t next_key;    // the same for the second nearest (kNoKey if none)
};

// Order key of a child entry distance, as a signed integer: non-negative
// distances by their bits (monotone), negative ones (sign bit set: negative
// as integers) all first.
constexpr int32_t kNoKey = 0x7FFFFFFF;
__device__ __forceinline__ int32_t tkey(float tn, uint32_t slot) {
    return (int32_t)((__float_as_uint(tn) & 0xFFFFFFF8u) | slot);
}

// (the compiler does not form it from min and max here)
__device__ __forceinline__ int32_t median3(int32_t a, int32_t b, int32_t c) {
    int32_t m;
    asm("v_med3_i32 %0, %1, %2, %3" : "=v"(m) : "v"(a), "v"(b), "v"(c));
    return m;
}

// Tests the 8 children of node `idx` against [tmin, tmax].  Measured on the
// 4.2 M incoherent rays (1,148,576 triangles): the vector ALU issues in 89 %
// of its cycles and the L1's data return is busy in 89 % of its own, so a
// visit's instructions and its loads both cost time.  With seven loads (leaf
// words only where leaves are tested), signed order keys (no clamp at zero),
// the running second minimum as a median, and the hit kept in LDS instead of
// four registers: 1,284 -> 1,188 us a launch (1,145 with the leaf runs below
// and the keys formed after the slots).
__device__ __forceinline__ void visit_node(NodeBuf nb, uint32_t idx, const RayPre& r, const NodeTest& nt,
                                           float tmax, NodeHits& h) {
    const uint32_t p = idx << 7;   // 128-byte nodes
    const uint4 w0 = node_word(nb, p);
    const uint4 nx = node_word(nb, p + (nt.offa & 0xFFu)), fx = node_word(nb, p + ((nt.offa >> 8) & 0xFFu));
    const uint4 ny = node_word(nb, p + ((nt.offa >> 16) & 0xFFu)), fy = node_word(nb, p + (nt.offa >> 24));
    const uint4 nz = node_word(nb, p + (nt.offb & 0xFFu)), fz = node_word(nb, p + (nt.offb >> 8));
    const float px = __uint_as_float(w0.x), py = __uint_as_float(w0.y), pz = __uint_as_float(w0.z);
    const int ex = (int)(int8_t)(w0.x & 0xFF), ey = (int)(int8_t)(w0.y & 0xFF), ez = (int)(int8_t)(w0.z & 0xFF);
    // ix 2^ex: a product with a power of two, exact as the multiplication
    const float ax = ldexpf(r.ix, ex), ay = ldexpf(r.iy, ey), az = ldexpf(r.iz, ez);
    const float bx = (px - r.ox) * r.ix, by = (py - r.oy) * r.iy, bz = (pz - r.oz) * r.iz;
    const uint32_t imask = w0.w >> 24;
    uint32_t hit = 0u;
    float tns[8];
#pragma unroll
    for (int s = 0; s < 8; ++s) {
        const float tnx = fmaf(qplane(nx, s), ax, bx);
        const float tfx = fmaf(qplane(fx, s), ax, bx);
        const float tny = fmaf(qplane(ny, s), ay, by);
        const float tfy = fmaf(qplane(fy, s), ay, by);
        const float tnz = fmaf(qplane(nz, s), az, bz);
        const float tfz = fmaf(qplane(fz, s), az, bz);
        const float tn = fmaxf(fmaxf(tnx, tny), fmaxf(tnz, r.tmin));
        const float tf = fminf(fminf(tfx, tfy), fminf(tfz, tmax));
        hit |= tn <= fmaf(fabsf(tf), KP_FAR_EPS, tf) ? (1u << s) : 0u;
        tns[s] = tn;
    }
    // order keys of the hit inner children, the others kNoKey: the mask bit
    // spread over the word selects (two instructions a slot; a compare and a
    // conditional move on both conditions take four, occlusion launches 5 %).
    // k1 <= k2, so the second smallest of {k1, k2, key} is their median.
    int32_t k1 = kNoKey, k2 = kNoKey;
    const uint32_t m = hit & imask;
#pragma unroll
    for (int s = 0; s < 8; ++s) {
        const uint32_t mask = (uint32_t)__builtin_amdgcn_sbfe((int)m, s, 1);
        const int32_t key = (int32_t)(((uint32_t)tkey(tns[s], (uint32_t)s) & mask) | ((uint32_t)kNoKey & ~mask));
        k2 = median3(k1, k2, key);
        k1 = min(k1, key);
    }
    // Empty slots hold inverted boxes (lower plane 2047, upper plane 0), which
    // miss unless the far-distance widening exceeds the node's extent; such a
    // slot then counts as a leaf child with no triangles and tests nothing.
    h.group = w0.w;
    h.inner = hit & imask;
    h.leaves = hit & ~imask;
    h.near_key = k1;
    h.next_key = k2;
}

__device__ __forceinline__ uint32_t inner_child(uint32_t child_base, uint32_t imask, uint32_t slot) {
    return child_base + __popc(imask & ((1u << slot) - 1u));
}

// Slot bits reordered by rank = slot ^ oct (an involution).
__device__ __forceinline__ uint32_t oct_permute(uint32_t m, uint32_t oct) {
    if (oct & 1u) m = ((m & 0x55u) << 1) | ((m >> 1) & 0x55u);
    if (oct & 2u) m = ((m & 0x33u) << 2) | ((m >> 2) & 0x33u);
    if (oct & 4u) m = ((m & 0x0Fu) << 4) | ((m >> 4) & 0x0Fu);
    return m;
}

// Stack entry (a group of inner children of one node still to visit):
//   x = child_base (24 bits) | inner mask << 24
//   y = lower bound of the group's entry distances (float bits, low 8 bits
//       cleared: a truncation toward zero, or -inf) | remaining children as
//       octant-rank bits (8 bits).
__device__ __forceinline__ uint32_t group_bound_bits(int32_t key2) {
    return key2 < 0 ? 0xFF800000u : (uint32_t)key2 & 0xFFFFFF00u;   // a negative distance: -inf
}

// Entry distance of one child slot of node `idx` (the same arithmetic as
// visit_node), for a top-level leaf child that names an instance.
__device__ __forceinline__ float slot_tnear(const uint4* __restrict__ nodes, uint32_t idx, uint32_t slot,
                                            const RayPre& r, const NodeTest& nt) {
    const uint4* p = nodes + (size_t)idx * 8;
    const uint4 w0 = p[0];
    const uint4 nx = p[(nt.offa & 0xFFu) >> 4], ny = p[((nt.offa >> 16) & 0xFFu) >> 4], nz = p[(nt.offb & 0xFFu) >> 4];
    const int ex = (int)(int8_t)(w0.x & 0xFF), ey = (int)(int8_t)(w0.y & 0xFF), ez = (int)(int8_t)(w0.z & 0xFF);
    const float ax = ldexpf(r.ix, ex), ay = ldexpf(r.iy, ey), az = ldexpf(r.iz, ez);
    const float bx = (__uint_as_float(w0.x) - r.ox) * r.ix, by = (__uint_as_float(w0.y) - r.oy) * r.iy,
                bz = (__uint_as_float(w0.z) - r.oz) * r.iz;
    const int s = (int)slot;
    const float tnx = fmaf(qplane(nx, s), ax, bx);
    const float tny = fmaf(qplane(ny, s), ay, by);
    const float tnz = fmaf(qplane(nz, s), az, bz);
    return fmaxf(fmaxf(tnx, tny), fmaxf(tnz, r.tmin));
}

// World ray to an instance's object space: o' = M o + m, d' = M d with the
// row-major 3x4 world-to-object matrix in inst[0..2] (FP32, no contraction,
// the same order as the oracle); the interval [tmin, tmax] is unchanged.
__device__ __forceinline__ void ray_to_object(const float4* __restrict__ inst, const float4 a, const float4 b,
                                              float4& oa, float4& ob) {
    const float4 m0 = inst[0], m1 = inst[1], m2 = inst[2];
    oa.x = ((m0.x * a.x + m0.y * a.y) + m0.z * a.z) + m0.w;
    oa.y = ((m1.x * a.x + m1.y * a.y) + m1.z * a.z) + m1.w;
    oa.z = ((m2.x * a.x + m2.y * a.y) + m2.z * a.z) + m2.w;
    oa.w = a.w;
    ob.x = (m0.x * b.x + m0.y * b.y) + m0.z * b.z;
    ob.y = (m1.x * b.x + m1.y * b.y) + m1.z * b.z;
    ob.z = (m2.x * b.x + m2.y * b.y) + m2.z * b.z;
    ob.w = b.w;
}

// Special stack entries of the two-level traversal (low byte of y zero; a
// group entry always has remaining-child bits there):
//   instance entry  x = instance record, y = bound of its box entry distance
//   return marker   x = kReturnMarker, y = -inf: back to the world-space ray
//   same-space end  x = kReturnSame, y = -inf: an identity placement ends
//   top level       x = kEnterTop, y = -inf: the meshes are done, go to the
//                   top level's root (same space and primitive base)
constexpr uint32_t kReturnMarker = 0xFFFFFFFFu;
constexpr uint32_t kReturnSame = 0xFFFFFFFEu;
constexpr uint32_t kEnterTop = 0xFFFFFFFDu;
// Instance record flag (bits of the third word of its fourth float4): the
// world-to-object matrix is exactly the identity, so the ray is used as is.
constexpr uint32_t kInstIdentity = 1u;

template <int S>
struct Stack {
    uint2 (*lds)[KP_TRACE_BLOCK];
    uint2* spill;
    uint32_t cap;
    int sp;
    int tid;

    __device__ __forceinline__ bool push(uint32_t a, uint32_t b) {
        if (sp >= S) {
            if ((uint32_t)(sp - S) >= cap) return false;
            spill[sp - S] = lds[sp & (S - 1)][tid];
        }
        lds[sp & (S - 1)][tid] = make_uint2(a, b);
        ++sp;
        return true;
    }
    __device__ __forceinline__ void push_lds(uint32_t a, uint32_t b) {   // sp < S
        lds[sp][tid] = make_uint2(a, b);
        ++sp;
    }
    __device__ __forceinline__ uint2 top() const { return lds[(sp - 1) & (S - 1)][tid]; }
    __device__ __forceinline__ void set_top_y(uint32_t y) { lds[(sp - 1) & (S - 1)][tid].y = y; }
    __device__ __forceinline__ void drop() {
        --sp;
        if (sp >= S) lds[sp & (S - 1)][tid] = spill[sp - S];
    }
};

constexpr int kStack = KP_TRACE_STACK;

// Work distribution of the persistent kernels.  A wave takes chunks of
// consecutive rays: a first chunk by its index (about half the rays split
// evenly over the waves), then chunks of kChunk from the global counter (one
// atomic per chunk; kTailChunk once fewer than one kChunk per wave remained
// after the wave's last chunk, so the waves run dry at about the same time),
// and hands them to its lanes from a wave-uniform cursor; every lane keeps
// its next ray prefetched in registers, so replacing a finished ray costs no
// memory round trip.  All members except the prefetch are wave-uniform.
struct RayFeeder {
    uint32_t next, end, n;
    uint32_t dyn_base;  // first ray handed out by the counter (after the static chunks)
    uint32_t waves;     // waves that share the queue
    bool drained;
    uint32_t* counter;
    const float4* rays;
    const uint32_t* roots;
    uint32_t pid, proot;   // prefetched ray of this lane (pid KP_INVALID: none) and its root
    float4 p0, p1;

    // block / blocks: this block's index among the blocks that share the queue
    __device__ __forceinline__ void init(uint32_t* ctr, const float4* rs, const uint32_t* rts, uint32_t count,
                                         uint32_t block, uint32_t blocks, uint32_t simds, uint32_t thin_one,
                                         uint32_t thin_most, bool even) {
        counter = ctr;
        rays = rs;
        roots = rts;
        proot = 0u;
        n = count;
        pid = KP_INVALID;
        // Wave w's first chunk is rays [w F, (w+1) F) without an atomic
        // (every wave of the grid would otherwise hit the one counter address
        // at start); the counter hands out the rays after all first chunks,
        // and a wave whose first chunk lies beyond the rays has none.
        waves = blocks * (KP_TRACE_BLOCK / 64);
        const uint32_t wave = block * (KP_TRACE_BLOCK / 64) + (threadIdx.x >> 6);
        const uint32_t first = first_chunk(n, waves, simds, thin_one, thin_most, even);
        dyn_base = waves * first;
        next = wave * first;
        if (next < n) {
            end = next + first < n ? next + first : n;
            drained = false;
        } else {
            next = end = 0;
            drained = true;
        }
        assign();
    }
    // Gives a prefetched ray to every lane without one, as far as rays last.
    __device__ __forceinline__ void assign() {
        const uint64_t m = __ballot(pid == KP_INVALID);
        if (m == 0 || drained) return;
        if (next >= end) {
            if (dyn_base >= n) {   // the first chunks covered every ray
                drained = true;
                return;
            }
            // the last chunk taken ended at `end`: small chunks once fewer
            // than kChunk rays per wave were left after it
            const uint64_t late = (uint64_t)waves * kChunk;
            const uint32_t size = (uint64_t)end + late >= n ? kTailChunk : kChunk;
            uint32_t base = 0;
            if (__lane_id() == 0) base = atomicAdd(counter, size);
            base = dyn_base + __builtin_amdgcn_readfirstlane(base);
            if (base >= n) {
                drained = true;
                return;
            }
            next = base;
            end = base + size < n ? base + size : n;
        }
        const uint32_t avail = end - next;
        const uint32_t want = (uint32_t)__popcll(m);
        const uint32_t prefix = (uint32_t)__popcll(m & ((1ull << __lane_id()) - 1ull));
        if (pid == KP_INVALID && prefix < avail) {
            pid = next + prefix;
            p0 = rays[2 * (size_t)pid];
            p1 = rays[2 * (size_t)pid + 1];
            if (roots) proot = roots[pid];
        }
        next += want < avail ? want : avail;
    }
};

// Lanes holding postponed leaf children before the wave tests them together.
constexpr int kLeafBatch = 16;
// Lanes with nothing but postponed leaves left (they wait) before the wave
// tests them; a wave test has a fixed cost of about 150 instructions and an
// idle lane costs a 64th of an iteration, so waiting for a fuller batch pays.
constexpr uint32_t kStuckBatch = 8u;

// LDS of the wave-wide leaf test (per block): the item map of each wave and,
// per lane, the merged result of the triangles tested for its ray.
struct LeafLds {
    uint32_t map[KP_TRACE_BLOCK];             // wave's 64 entries: owner lane << 8 | item of the owner
    unsigned long long key[KP_TRACE_BLOCK];   // closest hit: minimum hit key of the lane's ray, ~0 if none;
                                              // any hit: nonzero once hit
    union {
        float4 hit[KP_TRACE_BLOCK];           // closest hit: {t, u, v} of the minimum key
        struct {                              // any hit, connecting: rays found unoccluded
            uint32_t n[KP_TRACE_BLOCK / 64];
            uint32_t ray[KP_TRACE_BLOCK / 64][128];   // < 64 left over + at most one per lane and pass
        } open;
    };
};

__device__ __forceinline__ unsigned long long hit_key(float t, uint32_t prim);

// A closest-hit lane reads the leaf words of a set when the wave tests it, an
// occlusion lane when it finds the set (three registers more; the closest-hit
// builds have none to spare: with the words in registers they spill in the
// loop and the 4.2 M incoherent rays take 1,272 us instead of 1,228).
template <bool kAny>
constexpr bool kLazyLeaves = !kAny;

// Inclusive prefix sum and prefix maximum over the wave's 64 lanes, all of
// them active: four steps within rows of 16 lanes, two across rows.
template <bool kMax>
__device__ __forceinline__ uint32_t wave_scan(uint32_t x) {
#define KP_SCAN_STEP(ctrl, rows)                                                                  \
    {                                                                                             \
        const uint32_t y = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, ctrl, rows, 0xf, false); \
        x = kMax ? max(x, y) : x + y;                                                             \
    }
    KP_SCAN_STEP(0x111, 0xf)   // row_shr:1
    KP_SCAN_STEP(0x112, 0xf)   // row_shr:2
    KP_SCAN_STEP(0x114, 0xf)   // row_shr:4
    KP_SCAN_STEP(0x118, 0xf)   // row_shr:8
    KP_SCAN_STEP(0x142, 0xa)   // row_bcast:15 into rows 1 and 3
    KP_SCAN_STEP(0x143, 0xc)   // row_bcast:31 into rows 2 and 3
#undef KP_SCAN_STEP
    return x;
}

// The triangles of a leaf set: a node's leaf triangles are stored in slot
// order, so the set is tested as the run from its first to its last slot.
// Leaf slots between them that were not hit are tested too (their triangles
// are missed, or hit beyond their box's distance, as any other triangle); a
// run needs no per-slot bookkeeping, and a test round has idle lanes.
__device__ __forceinline__ void leaf_run(uint32_t slots, const uint4& w, uint32_t& first, uint32_t& count) {
    const uint32_t lo = __ffs(slots) - 1u, hi = 31u - (uint32_t)__clz((int)slots);
    const uint32_t a = __builtin_amdgcn_perm(w.z, w.y, lo | 0x0c0c0c00u);   // meta byte of slot lo
    const uint32_t b = __builtin_amdgcn_perm(w.z, w.y, hi | 0x0c0c0c00u);
    first = w.x + (a & 31u);
    count = (b & 31u) + (b >> 5) - (a & 31u);
}

// Triangles of a set's slots alone (what the counted variant counts).
__device__ __forceinline__ uint32_t leaf_set_tris(uint32_t slots, const uint4& w) {
    uint32_t n = 0u;
    for (uint32_t s = 0u; s < 8u; ++s)
        if ((slots >> s) & 1u) n += (((s < 4u ? w.y : w.z) >> ((s & 3u) * 8u)) & 0xFFu) >> 5;
    return n;
}

// Tests the postponed leaf sets of the wave's lanes together; all 64 lanes
// must call it, those without a set as well.  Each lane holds up to two sets
// (node << 8 | its hit leaf slots, 0 if none; the second is the one found in
// the current iteration), at most two runs of 32 triangles; the runs are laid
// out as one list (exclusive prefix sums over the lanes) and dealt out to the
// 64 lanes, so the triangle tests run with nearly every lane busy instead of
// one loop per lane at the pace of its longest set.  An item's owner is found
// by a prefix maximum over marks that the owners leave at the start of their
// part of the list.  A tester reads the owner's ray and closest distance from
// the owner's registers (lane permutes) and merges a hit into the owner's LDS
// slot: the 64-bit minimum of the (distance, primitive) key, then the t, u, v
// of the lane whose key is the minimum.  The slot lasts as long as the ray
// (key ~0: no hit yet), so a lane keeps only its closest distance in a
// register.  Every triangle is tested against the owner's closest distance at
// the start of the batch, so the slot holds the minimum key over all hits, the
// same as testing them one after another.
//
// With per-slot item lists, ballots per bit for the prefix sums and only the
// active lanes as testers this was about 40 % of the kernel's instructions:
// 4.2 M incoherent rays 1,190 us then and 1,150 now, 2.07 M camera rays 535 and
// 458, one million shadow rays 238 and 207, 262,147 two-level rays 247 and 193.
template <bool kAny, bool kCount>
__device__ __forceinline__ void test_leaves_wave(NodeBuf nb, const float4* __restrict__ tris, const RayPre& r,
                                                 uint32_t set1, const uint4& pw, uint32_t set2, float& best_t, bool& occl,
                                                 uint64_t& cnt_tris, uint32_t prim_off, LeafLds& L, int tid) {
    const uint32_t lane = __lane_id();
    uint32_t d1 = 0u, t1 = 0u, d2 = 0u, t2 = 0u;   // runs: first triangle, count
    const bool open = !(kAny && occl);
    if (set1 && open) {
        uint4 w = pw;
        if (kLazyLeaves<kAny>) w = node_word(nb, ((set1 >> 8) << 7) + 16u);
        leaf_run(set1 & 0xFFu, w, d1, t1);
        if (kCount) cnt_tris += leaf_set_tris(set1 & 0xFFu, w);
    }
    if (__ballot(set2 != 0u) != 0ull) {
        if (set2 && open) {
            const uint4 w = node_word(nb, ((set2 >> 8) << 7) + 16u);
            leaf_run(set2 & 0xFFu, w, d2, t2);
            if (kCount) cnt_tris += leaf_set_tris(set2 & 0xFFu, w);
        }
    }
    const uint32_t T = t1 + t2;
    const uint32_t incl = wave_scan<false>(T);
    const uint32_t E = incl - T;   // the lane's part of the list is [E, incl)
    const uint32_t P = __builtin_amdgcn_readlane(incl, 63);
    if (P == 0u) return;
    const uint32_t cut = E + t1;   // items below: the first run
    d1 -= E;                       // list position + d1 / d2 = triangle
    d2 -= cut;
    const int wbase = tid & ~63;
    uint32_t* map = &L.map[wbase];
    if (kAny && T != 0u) L.key[tid] = 0ull;
    for (uint32_t base = 0u; base < P; base += 64u) {
        map[lane] = 0u;
        __builtin_amdgcn_wave_barrier();
        const uint32_t mark = max(E, base);
        if (mark < min(incl, base + 64u)) map[mark - base] = lane;
        __builtin_amdgcn_wave_barrier();
        // (lane 0 as owner leaves the mark 0, which is also the filling:
        // it can only be the list's first owner)
        const uint32_t pos = base + lane;
        const int ow = (int)wave_scan<true>(map[lane]);
        const uint32_t o_cut = __shfl(cut, ow), o_d1 = __shfl(d1, ow), o_d2 = __shfl(d2, ow);
        RayPre o;
        o.ox = __shfl(r.ox, ow);
        o.oy = __shfl(r.oy, ow);
        o.oz = __shfl(r.oz, ow);
        o.tmin = __shfl(r.tmin, ow);
        o.Sx = __shfl(r.Sx, ow);
        o.Sy = __shfl(r.Sy, ow);
        o.Sz = __shfl(r.Sz, ow);
        o.k = __shfl(r.k, ow);
        const float o_best = __shfl(best_t, ow);
        const uint32_t o_off = __shfl(prim_off, ow);
        if (pos < P) {
            const uint32_t tri = pos + (pos < o_cut ? o_d1 : o_d2);
            const float4* tp = tris + 3 * (size_t)tri;
            const float4 ta = tp[0], tb = tp[1], tc = tp[2];
            float t, u, v;
            if (tri_test(o, ta, tb, tc, o_best, t, u, v)) {
                const int ot = wbase + ow;
                if (kAny) {
                    L.key[ot] = 1ull;
                } else {
                    const unsigned long long hk = hit_key(t, __float_as_uint(ta.w) + o_off);
                    // (no other triangle of the ray has this key)
                    __hip_atomic_fetch_min(&L.key[ot], hk, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WAVEFRONT);
                    __builtin_amdgcn_wave_barrier();
                    if (__hip_atomic_load(&L.key[ot], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WAVEFRONT) == hk)
                        L.hit[ot] = make_float4(t, u, v, 0.0f);
                }
            }
        }
        __builtin_amdgcn_wave_barrier();
    }
    if (T != 0u) {
        const unsigned long long k = __hip_atomic_load(&L.key[tid], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WAVEFRONT);
        if (kAny) {
            if (k != 0ull) occl = true;
        } else if (k != ~0ull) {
            best_t = L.hit[tid].x;
        }
    }
}

// Order key of a closest-hit candidate: distance first (float bits mapped to
// unsigned order, -0 taken as +0 as the comparisons do), then primitive, so
// the minimum key is the closest hit with the lowest primitive among equal
// distances (the tie rule).
__device__ __forceinline__ unsigned long long hit_key(float t, uint32_t prim) {
    uint32_t b = __float_as_uint(t);
    if (b == 0x80000000u) b = 0u;
    b ^= (b & 0x80000000u) ? 0xFFFFFFFFu : 0x80000000u;
    return ((unsigned long long)b << 32) | prim;
}

// Writes a ray's hit record from its slot's key and {t, u, v}.
__device__ __forceinline__ void write_hit(float4* out, unsigned long long key, const float4& h) {
    const bool none = key == ~0ull;
    *out = none ? make_float4(__int_as_float(0x7f800000), __uint_as_float(KP_INVALID), 0.0f, 0.0f)
                : make_float4(h.x, __uint_as_float((uint32_t)key), h.y, h.z);
}

// Position of the set bit of rank r (0-based) in m; r < popcount(m).
__device__ __forceinline__ uint32_t nth_set_bit(unsigned long long m, uint32_t r) {
    uint32_t pos = 0u;
    uint32_t c = __popc((uint32_t)m);
    if (r >= c) { r -= c; m >>= 32; pos += 32u; }
    c = __popc((uint32_t)m & 0xFFFFu);
    if (r >= c) { r -= c; m >>= 16; pos += 16u; }
    c = __popc((uint32_t)m & 0xFFu);
    if (r >= c) { r -= c; m >>= 8; pos += 8u; }
    c = __popc((uint32_t)m & 0xFu);
    if (r >= c) { r -= c; m >>= 4; pos += 4u; }
    c = __popc((uint32_t)m & 0x3u);
    if (r >= c) { r -= c; m >>= 2; pos += 2u; }
    return pos + (r >= ((uint32_t)m & 1u) ? 1u : 0u);
}

// LDS of one traversal block (31 KB, so five blocks fit a CU).  Split rays
// (one level) and world-space rays (two-level) never meet in one kernel.
struct SplitLds {
    unsigned long long key[KP_TRACE_BLOCK];       // owner: minimum helper hit key
    float4 hit[KP_TRACE_BLOCK];                   // owner: {t, u, v} of that key
    uint32_t role[KP_TRACE_BLOCK];                // owner thread | kHelper | kDonated | kWaiting
    unsigned long long busy[KP_TRACE_BLOCK / 64];   // wave: owners with helpers at work
};
struct TraceLds {
    uint2 stack[KP_TRACE_STACK][KP_TRACE_BLOCK];
    LeafLds leaf;
    union {
        SplitLds split;
        float4 wray[2][KP_TRACE_BLOCK];   // world ray per lane (two-level)
    };
};

// Lane roles of a split closest-hit ray (low 8 bits: block thread of the
// lane that owns the ray).
constexpr uint32_t kHelper = 1u << 8;    // traverses a group of another lane's ray
constexpr uint32_t kDonated = 1u << 9;   // owner whose ray has had groups handed out
constexpr uint32_t kWaiting = 1u << 10;  // owner done with its part, helpers still at work
constexpr uint32_t kStepsWaiting = 0xFFFFFFFFu;   // step count of a waiting owner (skips the traversal)

// Rays on the wave's list of unoccluded ones (written by any of its lanes).
__device__ __forceinline__ uint32_t open_count(LeafLds& L, int tid) {
    return __hip_atomic_load(&L.open.n[tid >> 6], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WAVEFRONT);
}
__device__ __forceinline__ void set_open_count(LeafLds& L, int tid, uint32_t n) {
    __hip_atomic_store(&L.open.n[tid >> 6], n, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WAVEFRONT);
}

// Ends an occlusion ray: its flag, or (connecting) a place on the list if it
// is not occluded.
template <bool kConnect>
__device__ __forceinline__ void finish_any(const TraceArgs& args, LeafLds& L, uint32_t ray, bool occl, int tid) {
    if (!kConnect) {
        args.occl[ray] = occl ? 1u : 0u;
        return;
    }
    const unsigned long long m = __ballot(!occl);
    if (!occl) {
        const uint32_t base = open_count(L, tid);
        L.open.ray[tid >> 6][base + (uint32_t)__popcll(m & ((1ull << __lane_id()) - 1ull))] = ray;
        __builtin_amdgcn_wave_barrier();
        set_open_count(L, tid, base + (uint32_t)__popcll(m));
    }
}

// A split ray's slot, written by other lanes of the wave.
__device__ __forceinline__ unsigned long long skey_load(unsigned long long* key, uint32_t i) {
    return __hip_atomic_load(&key[i], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WAVEFRONT);
}
__device__ __forceinline__ void skey_store(unsigned long long* key, uint32_t i, unsigned long long v) {
    __hip_atomic_store(&key[i], v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WAVEFRONT);
}

// Adds the contributions of up to 64 of the wave's listed unoccluded rays to
// their paths (the last ones of the list) and shortens the list.  Every lane
// of the wave must call it.
__device__ __forceinline__ void connect_open(const TraceArgs& args, LeafLds& L, uint32_t open, int tid) {
    const uint32_t left = open > 64u ? open - 64u : 0u;
    const uint32_t i = left + __lane_id();
    if (i < open) {
        const float4 c = args.scontrib[L.open.ray[tid >> 6][i]];
        float4* l = args.radiance + __float_as_uint(c.w);
        float4 x = *l;
        x.x += c.x;
        x.y += c.y;
        x.z += c.z;
        *l = x;
    }
    __builtin_amdgcn_wave_barrier();
    set_open_count(L, tid, left);
    __builtin_amdgcn_wave_barrier();
}

// Persistent traversal shared by closest hit (kAny = false) and occlusion
// (kAny = true).  A node visit tests the 8 children; the nearest hit inner
// child is visited next and the other hit inner children are pushed as one
// group entry, taken later in octant order (the builder puts children in
// octant slots) and skipped as a whole when their nearest entry distance lies
// beyond the closest hit so far.  Hit leaf children are postponed (one set
// per lane) and tested wave-wide (test_leaves_wave) when at least kLeafBatch
// lanes of the wave hold some, when kStuckBatch lanes (or every lane in the
// loop) have nothing else left, or when a lane finds a second set, so the
// triangle tests run with many lanes active instead of one or two.
//
// Two-level variant (kInst): a ray first traverses the BVH of the meshes
// (world_root, one-level, in world space) with a top-level marker below it on
// the stack; nodes below args.n_tlas form the top level, whose leaf children
// are instances.  Each lane keeps its world-space ray in LDS, read back on
// entering and leaving an instance.  A hit instance is pushed as an instance
// entry (culled later like a group by its entry distance); taking it pushes a
// return marker, moves the ray to the instance's object space and continues
// at the instance's root; reaching the marker restores the world-space ray
// (refetched from the ray buffer).  An identity placement keeps the ray and
// only switches the primitive base.  Postponed leaf children are tested
// before any of these switches, so a set is always tested in the space and
// with the primitive base it was found in.
//
// Split rays (kSplit; one level): once the rays are handed out, lanes
// whose rays are done would idle while the wave finishes its longest rays.
// Such a lane takes a child of the top group entry of a lane still at work
// (the whole group where no more lanes are idle than can give) and traverses
// it for the same ray (read from the donor's registers) with the donor's
// closest distance so far; the children are disjoint subtrees, so every
// triangle is still tested by exactly one lane.  A drain is bound by latency:
// about eight passes of 5,000 to 8,000 cycles for the longest rays of a small
// image, so a pass should spread a ray as far as there are lanes and a helper
// start at once.  With the ray read again and set up anew, the group taken in
// one pass and its first child visited in the next 1,000 closest-hit rays
// took 27.6 us, 65,536 90.7, 2,000 occlusion rays 44.1 and a 160 x 120 preview
// 343; with the ray from the donor and the first child visited at once 19.2,
// 77.7, 36.0 and 304; with thin occlusion launches 27.0 (occlusion) and 268;
// with single children handed out 15.2, 76.2, 22.0 and 255 (4.2 M rays lose
// 1 % by the registers, so the axes of the triangle test share one: 1,117 us
// before, 1,130, 1,115 now).  Two node visits between passes: 17.7, 82.3, 26.7
// and 262.  A helper
// merges its closest hit into its owner's slot in LDS (64-bit minimum of the
// (distance, primitive) key, then the t, u, v of the winning key); the owner
// writes the ray's hit once no helper of its ray is left.  The result is the
// minimum key over all triangles the ray hits in [tmin, tmax], the same as
// without splitting.  A helper also culls with its owner's closest distance
// once that is nearer (read at every pass of the drain phase).  An occlusion
// ray's slot holds only whether a part of it has hit; its helpers then stop.
// Occlusion splits in the integrator's pair launches and, in launches of its
// own, up to kSplitRays rays per block (in the loop it has six spilled
// registers, the build without has none): 400,000 rays 121 us one launch at a
// time and 67.1 with three in flight without, 111 and 66.0 with; 1,000,003 rays
// 199 and 133 without, 189 and 137 with.
//
// Connect (kConnect, occlusion): instead of a flag per ray, a ray that is not
// occluded adds its contribution to its path's radiance.  The finished rays
// are listed in LDS and added 64 at a time, so the two dependent loads
// (contribution, radiance) are waited for once per 64 rays, not once per
// loop pass.  A path has at most one ray in the queue: no two adds meet.
template <bool kAny, bool kCount, bool kInst, bool kConnect = false, bool kSplit = !kAny && !kInst>
__device__ __forceinline__ void traverse(const TraceArgs& args, TraceLds& S, uint32_t block, uint32_t blocks) {
    static_assert(!(kSplit && kInst), "the split state and the world-space rays share their LDS");
    LeafLds& leafl = S.leaf;
    float4 (&wray)[2][KP_TRACE_BLOCK] = S.wray;
    unsigned long long (&skey)[KP_TRACE_BLOCK] = S.split.key;
    float4 (&shit)[KP_TRACE_BLOCK] = S.split.hit;
    uint32_t (&srole)[KP_TRACE_BLOCK] = S.split.role;
    unsigned long long (&sbusy)[KP_TRACE_BLOCK / 64] = S.split.busy;
    const int tid = threadIdx.x;
    const uint32_t gl = blockIdx.x * KP_TRACE_BLOCK + tid;
    Stack<kStack> st;
    st.lds = S.stack;
    st.spill = args.spill + (size_t)gl * args.spill_cap;
    st.cap = args.spill_cap;
    st.sp = 0;
    st.tid = tid;
    const uint4* __restrict__ nodes = args.nodes;
    const NodeBuf nbuf = node_buffer(nodes);
    const uint32_t n_rays = args.n_dev ? *args.n_dev : args.n;   // device-side count for queues
    const float4* __restrict__ tris = args.tris;

    uint32_t ray_id = KP_INVALID;
    RayPre r;
    NodeTest nt;
    float best_t = 0.0f;                                   // closest distance so far (the hit itself is in LDS)
    uint32_t cur = KP_INVALID, steps = 0;
    uint32_t pend = 0u;                                    // postponed leaf children: node << 8 | slots
    uint4 pw = make_uint4(0u, 0u, 0u, 0u);                 // the leaf words of that node (!kLazyLeaves)
    uint32_t inst_pbase = 0u;                              // primitive base of the instance entered
    bool occl = false;
    bool split_on = false;   // rays are being split (wave-uniform; roles live in srole)
    uint64_t cnt_nodes = 0, cnt_tris = 0;
    RayFeeder feed;
    // (the counted variant measures the visits a ray needs: no thin launches,
    // which trade visits for latency)
    feed.init(args.counter, args.rays, args.roots, n_rays, block, blocks, args.simds, kThinOne<kAny>,
              kSplit && !kCount ? kThinMost<kAny> : 0u, args.n_dev != nullptr && blocks == gridDim.x);
    if (kConnect) {
        set_open_count(leafl, tid, 0u);
        __builtin_amdgcn_wave_barrier();
    }

    for (;;) {
        if (kConnect) {
            const uint32_t open = open_count(leafl, tid);
            if (open >= 64u) connect_open(args, leafl, open, tid);
        }
        if (ray_id == KP_INVALID && feed.pid != KP_INVALID) {
            ray_id = feed.pid;
            setup_ray(feed.p0, feed.p1, r);
            nt = node_test_setup(r);
            best_t = r.tmax;
            if (!kAny) leafl.key[tid] = ~0ull;
            occl = false;
            pend = 0u;
            inst_pbase = 0u;
            cur = ray_valid(feed.p0, feed.p1) ? feed.proot : KP_INVALID;   // root
            st.sp = 0;
            steps = 0;
            if (kSplit && split_on) {
                srole[tid] = (uint32_t)tid;
                skey[tid] = ~0ull;
            }
            feed.pid = KP_INVALID;
            if (kInst) {
                wray[0][tid] = feed.p0;
                wray[kInst ? 1 : 0][tid] = feed.p1;
                if (cur != KP_INVALID && args.world_root != KP_INVALID) {
                    st.push(kEnterTop, 0xFF800000u);   // the top level, after the meshes
                    cur = args.world_root;
                }
            }
        }
        feed.assign();
        if (kSplit && feed.drained) {
            const uint32_t lane = __lane_id();
            if (!split_on) {   // every ray in flight is its own owner
                split_on = true;
                srole[tid] = (uint32_t)tid;
                skey[tid] = ~0ull;
            }
            uint32_t role = srole[tid];
            if (kAny) {
                // a part of the ray has hit: its helpers stop, its owner waits for that
                const bool hit = ray_id != KP_INVALID && skey_load(skey, role & 0xFFu) != ~0ull;
                if (hit && (role & kHelper)) {
                    ray_id = KP_INVALID;
                    pend = 0u;
                } else if (hit && !(role & kWaiting)) {
                    role |= kWaiting;
                    srole[tid] = role;
                    steps = kStepsWaiting;
                    pend = 0u;
                }
            }
            unsigned long long* busy_w = &sbusy[tid >> 6];
            if (__ballot(ray_id != KP_INVALID && (role & kWaiting)) != 0ull) {
                // owners whose helpers are all done write their ray's hit (the
                // lanes of a wave reach LDS in instruction order)
                if (lane == 0u) __hip_atomic_store(busy_w, 0ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WAVEFRONT);
                __builtin_amdgcn_wave_barrier();
                if (ray_id != KP_INVALID && (role & kHelper))
                    __hip_atomic_fetch_or(busy_w, 1ull << (role & 63u), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WAVEFRONT);
                __builtin_amdgcn_wave_barrier();
                const unsigned long long busy = __hip_atomic_load(busy_w, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WAVEFRONT);
                if (ray_id != KP_INVALID && (role & kWaiting) && !((busy >> lane) & 1ull)) {
                    if (kAny) {
                        finish_any<kConnect>(args, leafl, ray_id, skey_load(skey, tid) != ~0ull, tid);
                    } else {
                        const unsigned long long k = skey[tid], own = leafl.key[tid];
                        write_hit(args.hits + ray_id, k < own ? k : own, k < own ? shit[tid] : leafl.hit[tid]);
                    }
                    ray_id = KP_INVALID;
                }
            }
            if (!kAny) {
                // a helper culls with its owner's closest distance once that
                // is nearer; its own hit, farther than the owner's, cannot win
                const float ob = __shfl(best_t, (int)(role & 63u));
                if (ray_id != KP_INVALID && (role & kHelper) && ob < best_t) {
                    best_t = ob;
                    leafl.key[tid] = ~0ull;
                }
            }
            // idle lanes take the top group entry of lanes still at work
            const unsigned long long idle = __ballot(ray_id == KP_INVALID && feed.pid == KP_INVALID);
            if (idle != 0ull) {
                const bool can = ray_id != KP_INVALID && !(role & kWaiting) && st.sp > 0;
                uint2 e = make_uint2(0u, 0u);
                if (can) e = st.top();
                const bool donor = can && !(__uint_as_float(e.y & 0xFFFFFF00u) > best_t);
                const unsigned long long donors = __ballot(donor);
                if (donors != 0ull) {
                    // the idle lane of rank i takes child i / donors of the
                    // group of donor i % donors, if the group has as many (or
                    // all of the group where every idle lane has its donor)
                    const uint32_t n_idle = (uint32_t)__popcll(idle), n_don = (uint32_t)__popcll(donors);
                    const unsigned long long below = (1ull << lane) - 1ull;
                    const float inv = __builtin_amdgcn_rcpf((float)n_don);
                    const uint32_t rank = (uint32_t)__popcll(idle & below);
                    const uint32_t kth = (uint32_t)(((float)rank + 0.5f) * inv);
                    const bool is_idle = (idle >> lane) & 1ull;
                    const int src = is_idle ? (int)nth_set_bit(donors, rank - kth * n_don) : (int)lane;
                    const uint32_t mine = (uint32_t)__popcll(donors & below);
                    const bool give = donor && mine < n_idle;
                    const bool whole = n_idle <= n_don;
                    const uint32_t gx = __shfl(e.x, src), gy = __shfl(e.y, src);
                    const uint32_t rid = __shfl(ray_id, src);
                    const float bt = __shfl(best_t, src);
                    const uint32_t own = __shfl(role & 0xFFu, src);
                    const bool take = is_idle && kth < (uint32_t)__popc(gy & 0xFFu);
                    if (give) {
                        uint32_t c = (uint32_t)(((float)(n_idle - mine - 1u) + 0.5f) * inv) + 1u;
                        uint32_t rest = whole ? 0u : e.y & 0xFFu;
                        while (c != 0u && rest != 0u) {
                            rest &= rest - 1u;
                            --c;
                        }
                        if (rest) st.set_top_y((e.y & 0xFFFFFF00u) | rest);
                        else st.drop();
                        srole[tid] = role | kDonated;
                    }
                    // the ray as its donor holds it (the others read themselves)
                    r.ox = __shfl(r.ox, src);
                    r.oy = __shfl(r.oy, src);
                    r.oz = __shfl(r.oz, src);
                    r.tmin = __shfl(r.tmin, src);
                    r.ix = __shfl(r.ix, src);
                    r.iy = __shfl(r.iy, src);
                    r.iz = __shfl(r.iz, src);
                    r.Sx = __shfl(r.Sx, src);
                    r.Sy = __shfl(r.Sy, src);
                    r.Sz = __shfl(r.Sz, src);
                    r.k = __shfl(r.k, src);
                    if (take) {
                        ray_id = rid;
                        srole[tid] = own | kHelper;
                        nt = node_test_setup(r);
                        best_t = bt;
                        if (!kAny) leafl.key[tid] = ~0ull;
                        occl = false;
                        pend = 0u;
                        steps = 0;
                        st.sp = 0;
                        uint32_t pm = gy & 0xFFu;
                        for (uint32_t k = 0u; k < kth; ++k) pm &= pm - 1u;
                        cur = inner_child(gx & 0x00FFFFFFu, gx >> 24, (__ffs(pm) - 1u) ^ nt.oct);
                        pm &= pm - 1u;
                        if (whole && pm) st.push_lds(gx, (gy & 0xFFFFFF00u) | pm);
                    }
                }
            }
        }
        if (__ballot(ray_id != KP_INVALID || feed.pid != KP_INVALID) == 0) break;
        // Iterations of the whole wave: lanes without work (busy false: no ray,
        // or an owner waiting for its helpers) stay in the loop and test
        // other lanes' triangles.
        {
            bool busy = ray_id != KP_INVALID && steps != kStepsWaiting;
            // nothing left to hand out and nothing to split: run to the end
            const bool more = !feed.drained || __ballot(feed.pid != KP_INVALID) != 0ull;
            while (__ballot(busy) != 0ull) {
                bool fault = false;
                uint32_t pend2 = 0u;   // a second leaf set found this iteration
                if (busy && cur != KP_INVALID) {
                    NodeHits h;
                    visit_node(nbuf, cur, r, nt, best_t, h);
                    if (kCount) cnt_nodes++;
                    const uint32_t vis = cur;
                    cur = KP_INVALID;
                    // (steps are node visits: a lane whose postponed leaves
                    // wait for the wave's test may wait for any number of the
                    // wave's other rays)
                    ++steps;
                    if (kInst && h.leaves && vis < args.n_tlas) {
                        // top-level leaves: push every instance they name
                        uint32_t lm = h.leaves;
                        const uint4 w1 = node_word(nbuf, (vis << 7) + 16u);
                        while (lm && !fault) {
                            const uint32_t s = __ffs(lm) - 1u;
                            lm &= lm - 1u;
                            const uint32_t mw = s < 4u ? w1.y : w1.z;
                            const uint32_t meta = (mw >> ((s & 3u) * 8u)) & 0xFFu;
                            const uint32_t first = w1.x + (meta & 31u), count = meta >> 5;
                            const uint32_t gy = group_bound_bits(tkey(slot_tnear(nodes, vis, s, r, nt), 0u));
                            for (uint32_t i = 0; i < count; ++i) {
                                if (!st.push(args.tlas_inst[first + i], gy)) {
                                    atomicOr(args.err, 1u);
                                    fault = true;
                                    break;
                                }
                            }
                        }
                    } else if (h.leaves) {
                        // (the words' load is waited for with the next visit's)
                        const uint32_t set = (vis << 8) | h.leaves;
                        if (pend == 0u) {
                            pend = set;
                            if (!kLazyLeaves<kAny>) pw = node_word(nbuf, (vis << 7) + 16u);
                        } else {   // this lane already holds a set: the wave tests both below
                            pend2 = set;
                        }
                    }
                    if (h.inner && !fault && !(kAny && occl)) {
                        const uint32_t s1 = (uint32_t)h.near_key & 7u;
                        const uint32_t rest = h.inner & ~(1u << s1);
                        if (rest) {
                            const uint32_t gy = group_bound_bits(h.next_key) | oct_permute(rest, nt.oct);
                            if (__ballot(st.sp >= kStack) == 0ull) {   // nearly always: no lane spills
                                st.push_lds(h.group, gy);
                            } else if (!st.push(h.group, gy)) {
                                atomicOr(args.err, 1u);
                                fault = true;
                            }
                        }
                        cur = inner_child(h.group & 0x00FFFFFFu, h.group >> 24, s1);
                    }
                }
                if (busy && !fault && cur == KP_INVALID && !(kAny && occl)) {
                    while (st.sp > 0) {
                        const uint2 e = st.top();
                        const float bound = __uint_as_float(e.y & 0xFFFFFF00u);
                        if (!kAny && bound > best_t) {   // every child of the group is beyond the hit
                            st.drop();
                            continue;
                        }
                        if (kInst && (e.y & 0xFFu) == 0u) {
                            if (e.x == kEnterTop) {   // same space and base: leaves may stay postponed
                                st.drop();
                                cur = 0u;
                                break;
                            }
                            // postponed leaves belong to the current space and
                            // base: the lane waits (no node) until the wave tests them
                            if (pend != 0u) break;
                            st.drop();
                            if (e.x == kReturnSame) {
                                inst_pbase = 0u;
                                continue;
                            }
                            if (e.x == kReturnMarker) {   // leave the instance: world-space ray again
                                const float4 wa = wray[0][tid], wb = wray[kInst ? 1 : 0][tid];
                                setup_ray(wa, wb, r);
                                nt = node_test_setup(r);
                                inst_pbase = 0u;
                                continue;
                            }
                            const float4* inst = args.insts + 4 * (size_t)e.x;
                            const float4 rec = inst[3];
                            if (__float_as_uint(rec.z) & kInstIdentity) {
                                if (!st.push(kReturnSame, 0xFF800000u)) {
                                    atomicOr(args.err, 1u);
                                    fault = true;
                                    break;
                                }
                            } else {
                                const float4 wa = wray[0][tid], wb = wray[kInst ? 1 : 0][tid];
                                float4 oa, ob;
                                ray_to_object(inst, wa, wb, oa, ob);
                                if (!ray_valid(oa, ob)) continue;   // degenerate in object space: misses
                                if (!st.push(kReturnMarker, 0xFF800000u)) {
                                    atomicOr(args.err, 1u);
                                    fault = true;
                                    break;
                                }
                                setup_ray(oa, ob, r);
                                nt = node_test_setup(r);
                            }
                            inst_pbase = __float_as_uint(rec.y);
                            cur = __float_as_uint(rec.x);
                            break;
                        }
                        uint32_t pm = e.y & 0xFFu;
                        const uint32_t s = (__ffs(pm) - 1u) ^ nt.oct;
                        pm &= pm - 1u;
                        if (pm) st.set_top_y((e.y & 0xFFFFFF00u) | pm);
                        else st.drop();
                        cur = inner_child(e.x & 0x00FFFFFFu, e.x >> 24, s);
                        break;
                    }
                }
                // postponed leaves: tested together once enough lanes hold some,
                // once kStuckBatch lanes (or every busy lane) have nothing but
                // leaves left, or when a lane found a second set (held for
                // this iteration only; the wave tests both sets)
                // (lanes that are not busy hold no set)
                const bool stuck = pend != 0u && (cur == KP_INVALID || fault);
                const uint32_t n_stuck = (uint32_t)__popcll(__ballot(stuck));
                const uint32_t n_busy = (uint32_t)__popcll(__ballot(busy));
                if (n_stuck >= min(kStuckBatch, n_busy) || __ballot(pend2 != 0u) != 0ull ||
                    __popcll(__ballot(pend != 0u)) >= kLeafBatch) {
                    test_leaves_wave<kAny, kCount>(nbuf, tris, r, pend, pw, pend2, best_t, occl, cnt_tris, inst_pbase,
                                                   leafl, tid);
                    pend = 0u;
                }
                bool done = busy && (fault || (kAny && occl) || (cur == KP_INVALID && pend == 0u && st.sp == 0));
                if (busy && !done && steps > args.max_steps) {
                    atomicOr(args.err, 2u);
                    done = true;
                }
                if (done) {
                    const uint32_t role = kSplit && split_on ? srole[tid] : 0u;
                    if (kAny) {
                        if (kSplit && (role & kHelper)) {
                            if (occl) skey_store(skey, role & 0xFFu, 0ull);
                        } else if (kSplit && (role & kDonated)) {
                            if (occl) skey_store(skey, tid, 0ull);
                            srole[tid] = role | kWaiting;   // finished once the helpers are done
                            steps = kStepsWaiting;
                        } else {
                            finish_any<kConnect>(args, leafl, ray_id, occl, tid);
                        }
                    } else if (kSplit && (role & kHelper)) {
                        // merge into the owner's slot: minimum key, then the
                        // t, u, v of the lane whose key is the minimum
                        const uint32_t o = role & 0xFFu;
                        const unsigned long long k = leafl.key[tid];
                        if (k != ~0ull) {
                            __hip_atomic_fetch_min(&skey[o], k, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WAVEFRONT);
                            __builtin_amdgcn_wave_barrier();
                            if (__hip_atomic_load(&skey[o], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WAVEFRONT) == k)
                                shit[o] = leafl.hit[tid];
                        }
                    } else if (kSplit && (role & kDonated)) {
                        srole[tid] = role | kWaiting;   // the hit is written once the helpers are done
                        steps = kStepsWaiting;
                    } else {
                        write_hit(args.hits + ray_id, leafl.key[tid], leafl.hit[tid]);
                    }
                    if (!kSplit || steps != kStepsWaiting) ray_id = KP_INVALID;
                    pend = 0u;
                    busy = false;
                }
                if (__popcll(__ballot(busy)) < args.refill_below && (kSplit || more)) break;
            }
        }
    }
    if (kConnect) {
        // (waiting owners may have joined the list after the pass's check, so
        // up to 127 rays are left)
        for (uint32_t open = open_count(leafl, tid); open != 0u; open = open_count(leafl, tid))
            connect_open(args, leafl, open, tid);
    }
    if (kCount) {
        atomicAdd((unsigned long long*)&args.counters[0], (unsigned long long)cnt_nodes);
        atomicAdd((unsigned long long*)&args.counters[1], (unsigned long long)cnt_tris);
    }
}

template <bool kCount>
__global__ __launch_bounds__(KP_TRACE_BLOCK) void k_closest(TraceArgs args) {
    __shared__ TraceLds lds;
    traverse<false, kCount, false>(args, lds, blockIdx.x, gridDim.x);
}

// The traversals compiled for 5 waves per SIMD (96 registers; the closest-hit
// build spills one register, the splitting occlusion build seven): more waves
// hide more of the node fetches' latency.  Launched everywhere but for the
// counted and the allocation-free closest hit.
__global__ __launch_bounds__(KP_TRACE_BLOCK) __attribute__((amdgpu_waves_per_eu(5))) void k_closest5(
    TraceArgs args) {
    __shared__ TraceLds lds;
    traverse<false, false, false>(args, lds, blockIdx.x, gridDim.x);
}

template <bool kSplit>
__global__ __launch_bounds__(KP_TRACE_BLOCK) __attribute__((amdgpu_waves_per_eu(5))) void k_occluded5(
    TraceArgs args) {
    __shared__ TraceLds lds;
    traverse<true, false, false, false, kSplit>(args, lds, blockIdx.x, gridDim.x);
}

// The two-level traversals compiled for 5 waves per SIMD (96 registers,
// spilling 24 and 44 B per lane; 31 KB of LDS per block, so 5 blocks fit a CU): the
// integrator's two-level render of C3's terrain runs 2.3 % faster than with
// the 4-wave build.
__global__ __launch_bounds__(KP_TRACE_BLOCK) __attribute__((amdgpu_waves_per_eu(5))) void k_closest_inst5(
    TraceArgs args) {
    __shared__ TraceLds lds;
    traverse<false, false, true>(args, lds, blockIdx.x, gridDim.x);
}

__global__ __launch_bounds__(KP_TRACE_BLOCK) __attribute__((amdgpu_waves_per_eu(5))) void k_occluded_inst5(
    TraceArgs args) {
    __shared__ TraceLds lds;
    traverse<true, false, true>(args, lds, blockIdx.x, gridDim.x);
}

// A bounce's two traversals in one launch: blocks [0, n_closest) trace the
// path rays (closest hit), the others the shadow rays of the vertices before
// them (occlusion, connecting).  The two queues do not depend on each other,
// and a persistent launch ends with a drain (its longest rays) in which the
// machine empties: with both in one launch the shadow blocks start on every
// CU as its closest-hit blocks run out, so a bounce has one drain, not two
// (about 20 us each: most of a bounce of a small image).  The two-level build
// spills 30 registers and is still faster than two launches: a two-level
// terrain render 29.5 ms with two launches, 27.4 with one.
template <bool kInst>
__global__ __launch_bounds__(KP_TRACE_BLOCK) __attribute__((amdgpu_waves_per_eu(5))) void k_trace_pair(
    TraceArgs args, ShadowQueue q, uint32_t n_closest) {
    __shared__ TraceLds lds;
    if (blockIdx.x < n_closest) {
        traverse<false, false, kInst>(args, lds, blockIdx.x, n_closest);
    } else {
        args.rays = q.rays;
        args.n_dev = q.n_dev;
        args.counter = q.counter;
        args.roots = q.roots;
        args.scontrib = q.contrib;
        args.radiance = q.radiance;
        traverse<true, false, kInst, true, !kInst>(args, lds, blockIdx.x - n_closest, gridDim.x - n_closest);
    }
}

template <bool kCount>
__global__ __launch_bounds__(KP_TRACE_BLOCK) void k_closest_inst(TraceArgs args) {
    __shared__ TraceLds lds;
    traverse<false, kCount, true>(args, lds, blockIdx.x, gridDim.x);
}

__global__ __launch_bounds__(256) void k_copy16(uint4* __restrict__ dst, const uint4* __restrict__ src,
                                                uint64_t n) {
    const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) dst[i] = src[i];
}

hipError_t launch_copy16(void* dst, const void* src, uint64_t n16, int cus, hipStream_t s) {
    const uint64_t want = (n16 + 255) / 256;
    const uint64_t cap = (uint64_t)(cus > 0 ? cus : 256) * 16;
    const uint32_t grid = (uint32_t)(want < cap ? (want ? want : 1) : cap);
    hipLaunchKernelGGL(k_copy16, dim3(grid), dim3(256), 0, s, (uint4*)dst, (const uint4*)src, n16);
    return hipGetLastError();
}

__global__ void k_reset_u32(uint32_t* p, uint32_t n) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = 0u;
}

// The host's last word on a call: one kernel behind its work instead of a
// blocking 4- to 16-byte copy per value after the wait (about 13 us each).
__global__ void k_status(const uint32_t* err, const uint32_t* noalloc_err, const unsigned long long* totals,
                         const uint32_t* train_records, HostStatus* out) {
    if (threadIdx.x != 0) return;
    HostStatus h{};
    if (totals) {
        h.totals[0] = totals[0];
        h.totals[1] = totals[1];
    }
    if (err) h.err = *err;
    if (noalloc_err) h.noalloc_err = *noalloc_err;
    if (train_records) h.train_records = *train_records;
    *out = h;
}

hipError_t launch_status(const uint32_t* err, const uint32_t* noalloc_err, const unsigned long long* totals,
                         const uint32_t* train_records, HostStatus* out, hipStream_t s) {
    hipLaunchKernelGGL(k_status, dim3(1), dim3(64), 0, s, err, noalloc_err, totals, train_records, out);
    return hipGetLastError();
}

// ---------------------------------------------------------------- launch --
// Whether the launch's feeders take rays from the counter: not while first
// chunks hold every ray (RayFeeder::init), so small launches need no clearing
// launch before them (5 us; 1,000 rays with three launches in flight 11.3 us
// a launch with it).
static bool uses_counter(const TraceArgs& a, uint32_t grid) {
    return a.n_dev || !first_chunks_hold_all(a.n, grid * (KP_TRACE_BLOCK / 64));
}

hipError_t launch_closest(const TraceArgs& a, uint32_t grid, bool count, bool reset, hipStream_t s) {
    if (grid == 0 || grid > a.spill_blocks) return hipErrorInvalidValue;   // lanes without a spill slice
    if (reset && uses_counter(a, grid)) hipLaunchKernelGGL(k_reset_u32, dim3(1), dim3(64), 0, s, a.counter, 1u);
    if (a.insts) {
        if (count) hipLaunchKernelGGL(k_closest_inst<true>, dim3(grid), dim3(KP_TRACE_BLOCK), 0, s, a);
        else if (a.five_waves) hipLaunchKernelGGL(k_closest_inst5, dim3(grid), dim3(KP_TRACE_BLOCK), 0, s, a);
        else hipLaunchKernelGGL(k_closest_inst<false>, dim3(grid), dim3(KP_TRACE_BLOCK), 0, s, a);
        return hipGetLastError();
    }
    if (count) hipLaunchKernelGGL(k_closest<true>, dim3(grid), dim3(KP_TRACE_BLOCK), 0, s, a);
    else if (a.five_waves) hipLaunchKernelGGL(k_closest5, dim3(grid), dim3(KP_TRACE_BLOCK), 0, s, a);
    else hipLaunchKernelGGL(k_closest<false>, dim3(grid), dim3(KP_TRACE_BLOCK), 0, s, a);
    return hipGetLastError();
}

hipError_t launch_occluded(const TraceArgs& a, uint32_t grid, hipStream_t s) {
    if (grid == 0 || grid > a.spill_blocks) return hipErrorInvalidValue;   // lanes without a spill slice
    if (uses_counter(a, grid)) hipLaunchKernelGGL(k_reset_u32, dim3(1), dim3(64), 0, s, a.counter, 1u);
    if (a.insts) hipLaunchKernelGGL(k_occluded_inst5, dim3(grid), dim3(KP_TRACE_BLOCK), 0, s, a);
    else if ((uint64_t)a.n <= (uint64_t)grid * kSplitRays)
        hipLaunchKernelGGL(k_occluded5<true>, dim3(grid), dim3(KP_TRACE_BLOCK), 0, s, a);
    else hipLaunchKernelGGL(k_occluded5<false>, dim3(grid), dim3(KP_TRACE_BLOCK), 0, s, a);
    return hipGetLastError();
}

hipError_t launch_pair(const TraceArgs& a, const ShadowQueue& q, uint32_t grid_closest, uint32_t grid_occluded,
                       hipStream_t s) {
    if (grid_closest == 0 || grid_occluded == 0 || grid_closest + grid_occluded > a.spill_blocks)
        return hipErrorInvalidValue;   // lanes without a spill slice
    const dim3 grid(grid_closest + grid_occluded);
    if (a.insts) hipLaunchKernelGGL(k_trace_pair<true>, grid, dim3(KP_TRACE_BLOCK), 0, s, a, q, grid_closest);
    else hipLaunchKernelGGL(k_trace_pair<false>, grid, dim3(KP_TRACE_BLOCK), 0, s, a, q, grid_closest);
    return hipGetLastError();
}

hipError_t trace_occupancy(int* blocks_per_cu_closest) {
    return hipOccupancyMaxActiveBlocksPerMultiprocessor(blocks_per_cu_closest, k_closest<false>, KP_TRACE_BLOCK, 0);
}

// Blocks per CU of the 5-wave builds: the smaller of the one-level and the
// two-level kernel's, so a grid of that size stays resident for either.
hipError_t trace_occupancy_five(int* blocks_per_cu_closest, int* blocks_per_cu_occluded) {
    int one = 0, two = 0;
    hipError_t e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&one, k_closest5, KP_TRACE_BLOCK, 0);
    if (e == hipSuccess) e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&two, k_closest_inst5, KP_TRACE_BLOCK, 0);
    if (e != hipSuccess) return e;
    *blocks_per_cu_closest = one < two ? one : two;
    e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&one, k_occluded5<true>, KP_TRACE_BLOCK, 0);
    if (e == hipSuccess) e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&two, k_occluded_inst5, KP_TRACE_BLOCK, 0);
    if (e != hipSuccess) return e;
    *blocks_per_cu_occluded = one < two ? one : two;
    return hipSuccess;
}

hipError_t launch_reset_u32(uint32_t* p, uint32_t n, hipStream_t s) {
    hipLaunchKernelGGL(k_reset_u32, dim3((n + 255) / 256), dim3(256), 0, s, p, n);
    return hipGetLastError();
}

}  // namespace kp
