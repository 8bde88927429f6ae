// lvn_kernels.h — launch interface of the gfx950 kernels (host side).
#pragma once

#include <hip/hip_runtime.h>

#include "lvn_shared.h"

namespace lvn {

// Arguments common to every stage kernel (passed by value).
struct KArgs {
    char* arena;             // chunk slot 0; slot i starts at arena + i * L.slot_bytes
    SlotLayout L;
    Geometry G;
    Caps caps;
    const ChunkDesc* chunks;
    Counters* counters;
    const DevOp* ops;
    const int* op_index;
    FieldParams F;
    const uint8_t* perm;     // 65,536 bytes
    const float4* grads;     // decoded gradients, one per stored table byte
    int defmat;
    int fp16;                // density stored as sign-preserving FP16
    int ysplit;              // density kernel: y segments per column
    int precise;             // QEF: compensated FP32 sums + FP64 re-solve
    unsigned long long* work;  // optional work counters (see lvn_batch_work), else null
    int* queue;              // kNumQueues work-queue heads, zeroed by launch_clear_counters
    int* item_prefix;        // chunks + 1 edge-item offsets (k_edge_data)
    int* special;            // the chunks with brushes or a cached field: their number, then them
    int cus;                 // compute units of the device
    int persist_per_cu;      // persistent workgroups per CU (edge crossing)
    int density_per_cu;      // persistent workgroups per CU (density), 0 = by the number of items
    int load;                // chunk_load of the launch's chunks, 0 = their number
    int height_lines;        // 1: x/z-edge sample heights evaluated once per line (k_height_lines)
    const int* slot_map;     // batch entry -> arena slot, or null for the identity
    int row_blocks;          // workgroups over the batch for the bookkeeping kernels
    int voxel_blocks;        // workgroups over the batch for the per-voxel kernels
    int cross_lanes;         // lanes per edge in the crossing stage (1, 2, 4, 8; 16 = sample-parallel), 0 = by batch size
    int dens_cols;           // 1: a field without the cave term stores no density; crossings form
                             // their end samples as y - H from the column heights (h_cols)
    int mat_free;            // 1: a fresh chunk without brushes stores no materials; the density
                             // pass writes its solid bits as planes, which k_solid_rows turns
                             // into rows and the QEF reads corners from
};

// Global work-queue heads (queue[1]: the edge-crossing items; the density and
// line-height passes share their items within workgroups instead; the rest are spare).
constexpr int kNumQueues = 8;

void launch_clear_counters(const KArgs& a, int n, hipStream_t s);

constexpr int kNumStages = LVN_NUM_STAGES;
extern const char* const kStageNames[kNumStages];
// Launch stage `i` (0..kNumStages-1) of the pipeline.
void launch_stage(const KArgs& a, int chunks, int i, hipStream_t s);
// Stages 6 to 8 launch nothing: the voxels' rows, scan and list go with the edges' (2, 3 and 4).
constexpr bool stage_launches(int i) { return i < 6 || i > 8; }

// Stage launchers: `chunks` chunk slots [0, chunks) processed by one launch each.
void launch_density(const KArgs& a, int chunks, hipStream_t s);
void launch_csg(const KArgs& a, int chunks, hipStream_t s);
void launch_rows(const KArgs& a, int chunks, hipStream_t s);             // solid, edge and voxel rows
void launch_scan_rows(const KArgs& a, int chunks, hipStream_t s);        // edge rows and voxel segments
void launch_compact(const KArgs& a, int chunks, hipStream_t s);          // edge lists and voxel codes
void launch_edge_cross(const KArgs& a, int chunks, hipStream_t s);
void launch_qef(const KArgs& a, int chunks, hipStream_t s);
void launch_scan_quads_seams(const KArgs& a, int chunks, hipStream_t s);
void launch_emit(const KArgs& a, int chunks, hipStream_t s);

// y-segments per density column when the launch shapes leave it open.
int default_ysplit(const Geometry& G, int field_kind, int chunks);
// Density workgroups per CU when the launch shapes leave it open.
int default_density_per_cu(const Geometry& G, int ysplit, int chunks, int cus);
// What `chunks` chunks count for in the crossing stage's choices, `coarse` being the sum of
// their sample scales / 4.
inline int chunk_load(int field_kind, long chunks, long coarse) {
    const long load = field_kind == LVN_FIELD_TERRAIN_CAVES ? chunks + coarse : chunks;
    return (int)(load < (1L << 24) ? load : 1L << 24);
}
// Lanes per edge in the crossing stage when the launch shapes leave it open.
int default_cross_lanes(const Geometry& G, int field_kind, int load);
// 1: line heights (k_height_lines) when the launch shapes leave it open.
int default_height_lines(const Geometry& G, int field_kind, int load);
// cross_lanes value of the sample-parallel crossing kernel (16 lanes per edge in the
// search, 6 in the normal).
constexpr int kCrossSampleParallel = 16;

// A mesh's three arrays (vertices, triangles, seam nodes) copied by one launch; pinned host
// memory or device memory on either side, addresses and sizes multiples of 4.
struct MeshCopy {
    const char* src[3];
    char* dst[3];
    uint64_t bytes[3];
};
void launch_copy_mesh(const MeshCopy& c, hipStream_t s);

// Chunk slot 0's counters and, back to back from kExportHeader bytes on, the mesh that
// generateChunkMesh exports of it into `out` (pinned host memory).
constexpr int kExportHeader = 64;
void launch_export(const KArgs& a, char* out, hipStream_t s);

// Chunk slot 0's descriptor and its op batch from pinned host memory into a.chunks, a.ops
// and a.op_index, counters cleared.
void launch_stage_chunk(const KArgs& a, const ChunkDesc* chunk, const DevOp* ops, const int* index, hipStream_t s);

// The pipeline's stages for chunk slots [0, chunks).
void launch_stages(const KArgs& a, int chunks, hipStream_t s);
// The same, counters cleared first.
void launch_pipeline(const KArgs& a, int chunks, hipStream_t s);

}  // namespace lvn
