// Host-side launch interfaces shared by the kernel translation units
// (kernels_grid.hip, kernels_transfer.hip, kernels_particles.hip) and the C ABI
// implementation (slosh_api.hip): the device buffers each launcher takes and
// the launchers themselves.
#pragma once

#include "common.h"

// ---- grid sort (kernels_grid.hip) ---------------------------------------------
struct GridBuffers {
    uint32_t *keys, *prev_keys;
    uint32_t *blist, *nbr, *cell_cnt, *cell_start, *blk_start, *blk_cnt;
    uint32_t *pslot, *prank, *perm, *counters;
    uint32_t *tile_sums;  // ceil(cap / 4096) words
    unsigned long long *rsum;  // REGIONS
};

// `fast`: the previous substep's fused kernels prepared this table. `ev` (optional)
// brackets the whole sequence.
hipError_t launch_grid_build(const GridBuffers &g, const float4 *pos, uint32_t n, float h, uint32_t batched,
                             uint32_t cap, bool fast, const PassEvents *ev, hipStream_t stream);

// ---- transfers (kernels_transfer.hip) ------------------------------------------
struct TransferBuffers {
    uint32_t fast;  // steady-state substep (members from stayer ranges and mover lists)
    const uint32_t *keys, *blist, *nbr, *counters;
    const uint32_t *perm;                             // full sort
    uint32_t *cell_cnt, *blk_start, *blk_cnt, *stay;  // this table
    // The steady state: this table's regional block lists, what the previous substep
    // left for each block (see NextTableBuffers), the previous table's keys and stayers;
    // written by P2G: the flat list and its length, the neighbour tables, each block's
    // range (start, count), stayers and movers.
    const uint2 *rlist;
    const uint4 *arrive;
    const uint32_t *rcnt, *prev_keys, *prev_stay;
    uint32_t rshift;
    uint32_t *blist_out, *num_blocks, *nbr_out;
    uint4 *bin;
    // Per region, the sums of its blocks' particles (high word) and items (low word),
    // and each block's place in them.
    unsigned long long *rsum;
    uint2 *rel;
    uint32_t *items;  // the fused G2P kernel's items (max_items of ITEM_WORDS words)
    uint32_t *n_items, *taken;
    const uint32_t *mlist, *ovf_slot, *ovf_hid;
    uint32_t *errors;  // this substep's error word
    float4 *tiles, *nodes;
    void *coll_prev, *coll_cur;
    float *fdt;
};

// Most items n particles in at most cap blocks can give: a block's entries are
// its candidates and listed movers (at most n of each over all blocks), in 64s.
inline size_t max_items(size_t n, size_t cap) { return 2 * n / 64 + (n < cap ? n : cap) + 1; }

struct ParticleBuffers {
    float4 *pos, *vm;
    float *C, *F, *vgd, *dps;
    uint32_t *ids;
};

struct StaticBuffers {
    const float4 *prop, *model, *dp0, *dp1;
    const float4 *scene_rec;  // batched: 4 records (prop, model, dp0, dp1) per scene id
};

struct ColliderBuffers {
    const float4 *shapes, *poses;
    const uint2 *mats;
    uint32_t count;
    const float4 *mesh_vtx;    // trimesh collision vertices (x, y, z, pad)
    const uint32_t *mesh_idx;  // trimesh collision indices
    // Per node of every trimesh body: its box, entry and exit (2 float4), and a leaf's
    // triangle and its index (3 float4); per collider its first node, then per
    // collider how its closest triangles are found (MESH_*) and its largest coordinate.
    const float4 *mesh_nodes, *mesh_leaves;
    const uint32_t *mesh_base;
};

struct BodyBuffers {
    float4 *poses, *vels;
    const float4 *mprops, *local_com;
    int *impulses;
    uint32_t count;
};

// The next substep's table and sort inputs, prepared by this substep's grid update
// (reset) and fused G2P (insertion, block lists, movers).
struct NextTableBuffers {
    uint32_t *keys, *counters;
    // Per block: the movers it receives; its slot in the table before and its range there
    // (start, count), if it has stayers (else SLOSH_NONE).
    uint4 *arrive;
    uint32_t *mlist;                // the first MOVER_CAP movers of each block
    uint32_t *ovf_slot, *ovf_hid;   // the others
    uint2 *rlist;                   // regional block lists (slot, key)
    uint32_t *rcnt;
    unsigned long long *rsum;
    uint32_t rshift, prime;
};

hipError_t launch_p2g(const StepParams &P, const ParticleBuffers &pb, uint32_t pcap, const TransferBuffers &t,
                      const PassEvents *ev, hipStream_t stream);
hipError_t launch_grid_update(const StepParams &P, const TransferBuffers &t, const ColliderBuffers &c,
                              const NextTableBuffers &next, uint32_t mode, uint32_t do_update, const PassEvents *ev,
                              hipStream_t stream);
// The BVH of one trimesh body (its `count` nodes' boxes and vertices at vtx, links and
// triangles at idx) in the layout of the grid update: ColliderBuffers::mesh_nodes, mesh_leaves.
hipError_t launch_pack_mesh(const float4 *vtx, const uint32_t *idx, uint32_t count, float4 *nodes, float4 *leaves,
                            hipStream_t stream);
hipError_t launch_g2p_update(const StepParams &P, const ParticleBuffers &in, const ParticleBuffers &out,
                             const StaticBuffers &s, uint32_t pcap, const TransferBuffers &t,
                             const NextTableBuffers &next, const BodyBuffers &bb, const PassEvents *ev,
                             hipStream_t stream);
hipError_t launch_g2p(const StepParams &P, const ParticleBuffers &b, uint32_t pcap, const TransferBuffers &t,
                      const PassEvents *ev, hipStream_t stream);
hipError_t launch_particle_update(const StepParams &P, const ParticleBuffers &b, const StaticBuffers &s, uint32_t pcap,
                                  float *fdt, const PassEvents *ev, hipStream_t stream);
hipError_t launch_rigid_update(const StepParams &P, const BodyBuffers &bb, const PassEvents *ev, hipStream_t stream);
// Per-scene record table: for each run of equal scene ids among storage slots
// [slot0, slot0 + n) of a particle buffer, the by-id records of the run's first
// particle (read only while every scene has one record), then each scene's mass
// (the largest of those particles' masses) in the plastic record's z (read only
// while every scene's particles have mass = enabled ? its mass : +0).
hipError_t launch_scene_records(const float4 *pos, const float4 *vm, const uint32_t *ids, uint32_t slot0, uint32_t n,
                                const StaticBuffers &s, float4 *scene_rec, hipStream_t stream);
hipError_t launch_timestep_bound(const StepParams &P, const ParticleBuffers &b, const StaticBuffers &s, uint32_t pcap,
                                 uint32_t *out, hipStream_t stream);
// Two passes over partial minima, one per TSB_CHUNK particles, in `partials`
// (div_up(n, TSB_CHUNK) words); *out = the bound, 0xffffffff with no enabled
// particle. Neither buffer needs clearing first.
hipError_t launch_timestep_bound_partials(const StepParams &P, const ParticleBuffers &b, const StaticBuffers &s,
                                          uint32_t pcap, uint32_t *partials, uint32_t *out, hipStream_t stream);

// ---- particle storage (kernels_particles.hip) ------------------------------------
struct CompactArgs {
    // current and destination particle sets (slot order)
    float4 *pos[2], *vm[2];
    float *C[2], *F[2], *vgd[2], *dps[2], *fdt[2];
    uint32_t *ids[2];
    // by-id static records, current and destination
    float4 *prop[2], *model[2], *dp0[2], *dp1[2];
    uint32_t *keep_slot, *keep_id, *keep_id2, *tile_sums, *total;
};
hipError_t launch_compact(const CompactArgs &a, uint32_t n, uint32_t pcap, uint32_t mode, const uint8_t *dead,
                          uint32_t lo, uint32_t hi, hipStream_t st);

struct GatherArgs {
    float4 *pos, *vm;
    float *C, *F, *vgd, *dps, *fdt;
    uint32_t *ids;
    // staging (count entries per component)
    float4 *s_pos, *s_vm;
    float *s_C, *s_F, *s_vgd, *s_dps, *s_fdt;
    uint32_t *rank_id, *tile_sums, *total;
};
// `strip`: clear the positions' flag bits.
hipError_t launch_scene_gather(const GatherArgs &a, uint32_t n, uint32_t pcap, uint32_t scene, uint32_t count,
                               uint32_t strip, hipStream_t st);
// Reference records of the particles with ids [lo, lo + count) into `out`, in id
// order; of `bad` (mapped host memory) word 0 becomes `mark` if an id is not below n,
// word 1 if `counters` (both tables') report an overflow.
enum { READ_POSITIONS = 0, READ_KINEMATICS, READ_DEF_GRAD };
hipError_t launch_read_records(const GatherArgs &a, uint32_t n, uint32_t pcap, uint32_t kind, uint32_t lo,
                               uint32_t count, void *out, const uint32_t *counters, uint32_t *bad, uint32_t mark,
                               hipStream_t st);
uint32_t scan_tiles(uint32_t n);
