// Data layout of the HIP intersector (host and device visible).
//
// BVH8 node record (host): 128 bytes, 16-byte aligned:
//   dword 0-2  p.xyz       float    origin of the quantisation grid; the low
//                                   byte of each is the axis's exponent e
//                                   (the builder picks such an origin)
//   dword 3    e.x,e.y,e.z int8     per-axis power-of-two scale exponents
//              imask       uint8    bit i set = child slot i is an inner node
//   dword 4    child_base  uint32   index of the first inner child; inner
//                                   children are stored contiguously in slot
//                                   order (child = base + rank of slot i)
//   dword 5    prim_base   uint32   first triangle of the leaf children
//   dword 6-7  meta[8]     uint8    leaf slot: (count << 5) | offset,
//                                   count 1..7 triangles at prim_base+offset;
//                                   inner slot: 1; empty slot: 0
//   dword 8-31 q[6][8]     binary16 child boxes, planes lo.x lo.y lo.z hi.x
//                                   hi.y hi.z, each 8 slots, holding integers
//                                   0..2047 (exact in binary16, so the
//                                   mixed-precision fma reads them without a
//                                   conversion); decoded bound = p + q * 2^e
//                                   (conservative by construction); an empty
//                                   slot has lo = 2047, hi = 0 and meta 0.
// Device node: the same 128 bytes with the header regrouped so that a visit
// needs only its first 16 bytes beside the planes:
//   dword 0-2  p.xyz       (low byte: e)
//   dword 3    child_base (24 bits) | imask << 24
//   dword 4    prim_base          read only for nodes whose leaf children
//   dword 5-6  meta[8]            are hit (empty slots: a valid offset)
//   dword 7    0
//   dword 8-31 planes
// One lane reads its node with 16-byte loads from one 128-byte line; the L1
// takes about one cycle per lane and load, which bounds traversal as much as
// the vector ALU does, so a visit's loads are worth saving: seven instead of
// eight.
// Inner children sit in octant slots: bit k of the slot set = the child lies
// on the high side of axis k (as nearly as the builder can arrange).
// Triangle record: 48 bytes = three float4 {v0.xyz, prim}, {v1.xyz, 0},
// {v2.xyz, 0}; `prim` is the caller-visible primitive index (bit pattern).
#pragma once
#include <stdint.h>

#define KP_NODE_BYTES 128u
#define KP_TRI_BYTES 48u
#define KP_LEAF_FLAG 0x80000000u
#define KP_INVALID 0xFFFFFFFFu
#define KP_MAX_LEAF 7u

struct alignas(16) KpNode8 {
    float px, py, pz;
    int8_t ex, ey, ez;
    uint8_t imask;
    uint32_t child_base;
    uint32_t prim_base;
    uint8_t meta[8];
    uint16_t q[6][8];
};
static_assert(sizeof(KpNode8) == KP_NODE_BYTES, "node must be 128 bytes");

// The device form of a node record (above).
static inline void kp_device_node(const KpNode8& n, uint32_t out[32]) {
    __builtin_memcpy(out, &n, KP_NODE_BYTES);
    const uint32_t prim_base = out[5], meta0 = out[6], meta1 = out[7];
    out[3] = (out[4] & 0x00FFFFFFu) | ((uint32_t)n.imask << 24);
    out[4] = prim_base;
    out[5] = meta0;
    out[6] = meta1;
    out[7] = 0u;
    // An empty slot's meta byte: no triangles, at the offset of the leaf slots
    // before it.  Its inverted box can be hit (the far distance is widened), and
    // a leaf set is tested as the run from its first to its last slot.
    uint8_t* meta = (uint8_t*)(out + 5);
    uint32_t off = 0u;
    for (int s = 0; s < 8; ++s) {
        if (meta[s] == 0u) meta[s] = (uint8_t)off;
        else if (!((n.imask >> s) & 1u)) off = (meta[s] & 31u) + (meta[s] >> 5);
    }
}

// A leaf reference packs a triangle start (28 bits) and count-1 (3 bits).
static inline uint32_t kp_leaf_ref(uint32_t first, uint32_t count) {
    return KP_LEAF_FLAG | (first << 3) | (count - 1u);
}
