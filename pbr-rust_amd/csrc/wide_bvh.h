// 8-wide BVH collapsed from the binary build tree, and its traversal.
#pragma once

#include "pbrtm_device.h"
#include "pbrtm_internal.h"
#include "wide_box.h"

namespace pbrtm {

namespace pt {
struct DShape;
}

constexpr int kWide = 8;
constexpr uint32_t kWideLeaf = 0x80000000u;
constexpr uint32_t kWideEmpty = 0xFFFFFFFFu;

// 128 bytes = one cache line. Child boxes are quantized to 8 bits per plane
// against the node's origin (the union's lower corner) and a power-of-two step
// per axis: plane = fmaf(q, 2^exp, org), rounded outwards at encoding so that
// every decoded box contains the child's exact FP32 box. Then one (word0,
// word1) reference per child slot. Interior child: word0 = wide node index,
// word1 = 0. Leaf child: word0 = kWideLeaf | first leaf position, word1 =
// primitive count. Unused slot: word0 = kWideEmpty, inverted box. Slots hold
// the collapsed binary subtree's frontier in left-to-right order.
struct alignas(128) WNode {
    float org[3];
    int8_t exp[3];
    uint8_t pad;
    uint8_t q[6][kWide];  // lo_x, lo_y, lo_z, hi_x, hi_y, hi_z per slot
    uint32_t ref[kWide][2];
};
static_assert(sizeof(WNode) == 128, "WNode is one cache line");

// Per wide node and ray octant (bit k = direction k negative): the order in
// which the reference's depth-first, near-child-first binary traversal reaches
// the slots, as 8 nibbles (position p -> slot), 0xF past the last slot.
struct WideBvh {
    DevBuf nodes, order;
    uint32_t num_nodes = 0;
    uint32_t max_depth = 0;   // wide levels on the longest root-to-leaf path
    uint32_t collapse_levels = 0;
};

// Collapses the binary tree (preorder-reserved ids, root 0, n primitives).
hipError_t collapse_wide(const BNode *bnodes, uint32_t n, WideBvh &out, DevBuf &scratch, uint32_t *err,
                         hipStream_t stream);

struct WideTrace {
    const WNode *nodes;
    const uint32_t *order;
    const float *tri_leaf;
    const uint32_t *prim_order;
    const pt::DShape *shapes;  // analytic primitives (leaf pad word = index + 1), null for triangle-only trees
    uint32_t num_nodes, num_prims, max_depth;
    TreeBox box;
    uint2 *spill;           // per-ray stack overflow area (max_depth - kLdsStack entries per ray), may be null
    uint32_t spill_per_ray;
    uint32_t grid_quarters; // persistent traversal grid: this many quarters of the resident maximum (0 = all)
};

// counts (device, nullable): adds [wide nodes visited, child box tests, triangle tests];
// a node whose boxes are tested again after a hit in one of its leaves is no new visit.
// queue (device, n entries) and queue_len (device, one word zeroed by the caller) hold the
// compacted active rays and their number; heads (device, kHeadWords words zeroed by the
// caller, 64-byte aligned) count the rows handed out.
constexpr uint32_t kHeads = 32;       // counters of rows, each serving its share of them
constexpr uint32_t kHeadStride = 16;  // words between two: a cache line of their own
constexpr uint32_t kHeadWords = kHeads * kHeadStride;
hipError_t trace_wide(const WideTrace &B, const float *rays, uint32_t n, int any_hit, uint32_t *prim_out,
                      float *t_out, float *bary_out, uint32_t *err, unsigned long long *counts, uint32_t *queue,
                      uint32_t *queue_len, uint32_t *heads, hipStream_t stream);

// The rays of a queue filled by the caller (*queue_len of at most n entries; heads have to
// be zero, rows below a head left from another traversal would be skipped). Ray i of
// several jobs is traced against jobs[ray_job[i >> job_shift]] (nodes, order, tri_leaf,
// prim_order, num_nodes, num_prims, box); B supplies the spill area.
hipError_t trace_wide_multi_queued(const WideTrace &B, const WideTrace *jobs, const uint32_t *ray_job,
                                   uint32_t job_shift, const float *rays, uint32_t n, int any_hit, uint32_t *prim_out,
                                   float *t_out, float *bary_out, uint32_t *err, const uint32_t *queue,
                                   const uint32_t *queue_len, uint32_t *heads, hipStream_t stream);
// The same for one tree (queue, queue_len and heads as above).
// counts (device, nullable): adds [nodes visited, child box tests, primitive tests].
hipError_t trace_wide_queued(const WideTrace &B, const float *rays, uint32_t n, int any_hit, uint32_t *prim_out,
                             float *t_out, float *bary_out, uint32_t *err, const uint32_t *queue,
                             const uint32_t *queue_len, uint32_t *heads, hipStream_t stream,
                             unsigned long long *counts = nullptr);

constexpr uint32_t kLdsStack = 12;

}  // namespace pbrtm
