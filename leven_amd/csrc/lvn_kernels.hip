// lvn_kernels.hip — the chunk-mesher stages as gfx950 kernels.
//
// Every kernel takes the chunk from blockIdx.y (or, in the persistent kernels,
// from a work item), so one launch serves one chunk (plain form) or a whole
// batch (batched form).  Compaction is deterministic: a classification kernel
// writes 64-bit masks and counts per row (edges: x/y/z masks of a hermite row;
// voxels, quads, seams: one mask per 64 elements), one workgroup per chunk scans
// the counts, and element i lands at base[row] + popcount(mask bits below i).
// The element order is therefore the reference's linear order everywhere
// (cl/density_field.cl:52-53, cl/octree.cl:153, cl/octree.cl:398-439).

#include "lvn_device.hpp"
#include "lvn_kernels.h"

#include <hip/hip_fp16.h>

#include <algorithm>

namespace lvn {

namespace {

// Batch entry `chunk` lives in arena slot slot_map[chunk] (identity without a map).
template <typename T>
__device__ __forceinline__ T* slot_ptr(const KArgs& a, int chunk, uint64_t off) {
    const uint64_t slot = a.slot_map ? (uint64_t)a.slot_map[chunk] : (uint64_t)chunk;
    return reinterpret_cast<T*>(a.arena + slot * a.L.slot_bytes + off);
}

__device__ __forceinline__ int field_index(const Geometry& G, int x, int y, int z) {
    return x + G.F * (y + G.F * z);
}

// Division by H or F (runtime values) as a multiply-high: exact for n < 2^21
// since (n * ceil(2^32/d)) / 2^32 - n/d < n / 2^32 < 1/d for d < 2^11.
__device__ __forceinline__ int div_magic(int n, uint32_t magic) { return (int)__umulhi((uint32_t)n, magic); }

// Voxel v = x + N (y + N z) with N = 2^depth.
__device__ __forceinline__ void decode_voxel(const Geometry& G, int v, int& x, int& y, int& z) {
    x = v & (G.N - 1);
    y = (v >> G.depth) & (G.N - 1);
    z = v >> (2 * G.depth);
}

__device__ __forceinline__ uint64_t lanemask_lt(int lane) { return lane == 0 ? 0ull : (~0ull >> (64 - lane)); }

// Dense lookup of a compacted element through its segment's mask word m (bit `lane`)
// and base: its index, or -1.
__device__ __forceinline__ int dense_index_of(uint64_t m, int base, int lane) {
    return ((m >> lane) & 1ull) ? base + __popcll(m & lanemask_lt(lane)) : -1;
}

// Work split of a chunk over the x dimension of its grid (blockIdx.y is the chunk).
__device__ __forceinline__ int wave_in_chunk() { return (int)(blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6)); }
__device__ __forceinline__ int waves_per_chunk() { return (int)(gridDim.x * (blockDim.x >> 6)); }
__device__ __forceinline__ int thread_in_chunk() { return (int)(blockIdx.x * blockDim.x + threadIdx.x); }
__device__ __forceinline__ int threads_per_chunk() { return (int)(gridDim.x * blockDim.x); }

// Bits x + 1 of a 66-bit sample row (lo = x 0..63, hi = x 64, 65) moved to bit x.
__device__ __forceinline__ uint64_t shift_next(uint64_t lo, uint64_t hi) { return (lo >> 1) | (hi << 63); }

// Items of the queued crossing kernel: wave w of the grid starts with grab w (`per_grab`
// consecutive items), without the queue, and takes later grabs from the atomic counter.
// One counter serves about 77 grabs per us, so when every wave of a full grid (3,072 for
// one chunk) took its first, mostly failing, grab there, that alone was 40 us.  Waves are
// numbered across the workgroups, so few items spread over the CUs.
__device__ __forceinline__ int grid_waves() { return (int)(gridDim.x * (blockDim.x >> 6)); }
__device__ __forceinline__ int first_grab(int per_grab) {
    return __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6) * (int)gridDim.x + (int)blockIdx.x) * per_grab;
}

// FP16 store that keeps the sign of every negative sample (an underflow to -0
// would turn a solid sample into air under the reference's `density < 0` test,
// cl/density_field.cl:34).
__device__ __forceinline__ __half to_half_keep_sign(float d) {
    __half h = __float2half_rn(d);
    if (d < 0.f && !(__half2float(h) < 0.f)) h = __ushort_as_half((unsigned short)0x8001u);
    return h;
}

// cl/shared_constants.cl:4-9 / cl/octree.cl:227-232
__constant__ int kEdgeMap[12][2] = {{0, 4}, {1, 5}, {2, 6}, {3, 7}, {0, 2}, {1, 3},
                                    {4, 6}, {5, 7}, {0, 1}, {2, 3}, {4, 5}, {6, 7}};

}  // namespace

// ---------------------------------------------------------------------------
// Density + default material (GenerateDefaultField, cl/density_field.cl:11-37)
// ---------------------------------------------------------------------------
// One thread per (x, z) column segment: the height term depends on x and z
// only, so it is evaluated once and reused down the column.  A wave takes 64
// consecutive columns (group g, column x + F z = 64 g + lane) over one y-segment.
__device__ __forceinline__ bool chunk_mat_free(const KArgs& a, const ChunkDesc& cd) {
    return a.mat_free && cd.op_count == 0 && cd.mode != kModeCached;
}

// A chunk whose samples the density pass found all solid or all air (and no brush or cached
// field changes): it has no edges and no voxels, and the bookkeeping kernels pass it by.  Half
// of a clipmap's chunks are such.
__device__ __forceinline__ bool chunk_uniform(const KArgs& a, int chunk) {
    return chunk_mat_free(a, a.chunks[chunk]) && a.counters[chunk].sides != (kSomeSolid | kSomeAir);
}

// The least of the wave's values, in every lane.
__device__ __forceinline__ uint32_t wave_min(uint32_t x) {
#define LVN_LEAST(ctrl) x = min(x, (uint32_t)__builtin_amdgcn_update_dpp((int)x, (int)x, ctrl, 0xf, 0xf, false));
    LVN_LEAST(0x111)  // row_shr 1, 2, 4, 8: lane 15 of a row holds the row's
    LVN_LEAST(0x112)
    LVN_LEAST(0x114)
    LVN_LEAST(0x118)
    LVN_LEAST(0x142)  // row_bcast 15 and 31: lane 63 holds the wave's
    LVN_LEAST(0x143)
#undef LVN_LEAST
    return (uint32_t)__builtin_amdgcn_readlane((int)x, 63);
}

template <bool kCount, int kKind>
__device__ __forceinline__ void density_column(const KArgs& a, const NoiseLds& T, int chunk, int seg, int g) {
    const Geometry& G = a.G;
    const int F = G.F;
    const int lane = threadIdx.x & 63;
    const bool valid = g * 64 + lane < F * F;     // the last group is partial
    const int col = valid ? g * 64 + lane : F * F - 1;
    const int seg_len = (F + a.ysplit - 1) / a.ysplit;
    const ChunkDesc cd = a.chunks[chunk];  // a copy: the loops below store through pointers that could alias it
    const int z = div_magic(col, G.magic_f);
    const int x = col - z * F;
    const int y0 = seg * seg_len;
    const int y1 = min(F, y0 + seg_len);
    uint8_t* mat = slot_ptr<uint8_t>(a, chunk, a.L.mat);
    uint8_t* orig = slot_ptr<uint8_t>(a, chunk, a.L.orig);
    // the materials before CSG are read only to find edges a brush touched: chunks
    // without ops skip them (uniform over a 64-column item, which lies in one chunk)
    const bool keep_orig = cd.op_count > 0;
    if (cd.mode == kModeCached) {  // a cached field: its materials, no density
        const uint8_t* old = reinterpret_cast<const uint8_t*>(cd.old_mat);
        for (int y = y0; y < y1 && valid; ++y) {
            const int idx = field_index(G, x, y, z);
            const uint8_t m = old[idx];
            mat[idx] = m;
            if (keep_orig) orig[idx] = m;
        }
        return;
    }
    // A chunk without brushes in a batch stores no materials (uniform over the wave): its
    // "not air" bits go to the planes, one ballot per y, and lane j keeps the word of
    // y = y0 + 64 k + j until the wave stores them together.
    const bool planes = chunk_mat_free(a, cd);
    uint64_t* P = slot_ptr<uint64_t>(a, chunk, a.L.planes) + (long)g * F;
    const float wx = (float)(x * cd.scale + cd.off[0]);
    const float wz = (float)(z * cd.scale + cd.off[2]);
    const float H = height_term<kKind>(a.F, T, wx, wz);
    if (seg == 0 && valid) slot_ptr<float>(a, chunk, a.L.h_cols)[col] = H;  // read by the crossing kernels
    float* dens = slot_ptr<float>(a, chunk, a.L.density);
    __half* dens16 = slot_ptr<__half>(a, chunk, a.L.density);
    unsigned caves = 0;
    uint64_t word = 0, solid = 0, air = 0;
    const uint64_t all = __ballot(valid);
    const uint64_t can_be = a.defmat == kAir ? 0ull : all;  // a default material of air leaves no solid sample
    constexpr bool kCaves = kKind == LVN_FIELD_TERRAIN_CAVES || kKind == kAnyField;
    if (!kCaves && planes && a.dens_cols) {
        // Nothing but the planes is stored, of the sign of wy - H, and wy rises with y: a
        // column's solid samples are its first n, found by halving, and only the planes
        // between the least and the largest n of the 64 columns are looked at one by one.
        // (Sample by sample, 38 vector and 32 scalar instructions each, this loop was the
        // pass's time: 591 -> 195 us on the reference's terrain, 1,800 chunks.)
        const int len = max(y1 - y0, 0);  // the last of many y-segments may be empty
        int n = 0;
#pragma unroll
        for (int step = 64; step > 0; step >>= 1) {
            const float wy = (float)((y0 + n + step - 1) * cd.scale + cd.off[1]);
            if (n + step <= len && wy - H < 0.f) n += step;
        }
        if (!can_be) n = 0;
        const int least = (int)wave_min(valid ? (uint32_t)n : (uint32_t)len);
        const int most = len - (int)wave_min((uint32_t)(len - (valid ? n : 0)));
        for (int base = 0; base < len; base += 64) {
            word = base + lane < least ? all : 0ull;
            for (int y = max(least, base); y < min(most, base + 64); ++y) {
                const uint64_t bits = __ballot(valid && n > y);
                if (lane == y - base) word = bits;
            }
            if (base + lane < len) P[y0 + base + lane] = word;
        }
        solid = most > 0;
        air = least < len;
    } else {
        auto keep = [&](int y, uint64_t bits) {  // the solid bits of plane y
            solid |= bits;
            air |= all & ~bits;
            const int j = (y - y0) & 63;
            if (lane == j) word = bits;
            if ((j == 63 || y == y1 - 1) && lane <= j) P[y - j + lane] = word;
        };
        int idx = field_index(G, x, y0, z), v = y0 * cd.scale + cd.off[1];
        for (int y = y0; y < y1; ++y, v += cd.scale, idx += F) {
            const float wy = (float)v;
            const float d = combine<kKind>(a.F, T, wy - H, wx, wy, wz);
            if constexpr (kCount) caves += (a.F.kind == LVN_FIELD_TERRAIN_CAVES && !((wy - H) > a.F.cave_cut)) ? 1u : 0u;
            if (valid) {
                if (a.fp16)
                    dens16[idx] = to_half_keep_sign(d);
                else if (!a.dens_cols)
                    dens[idx] = d;
                if (!planes) {
                    const uint8_t m = d < 0.f ? (uint8_t)a.defmat : (uint8_t)kAir;
                    mat[idx] = m;
                    if (keep_orig) orig[idx] = m;
                }
            }
            if (planes) keep(y, __ballot(d < 0.f) & can_be);
        }
    }
    if (planes && lane == 0)
        slot_ptr<uint8_t>(a, chunk, a.L.sides)[seg * G.col_groups + g] =
            (uint8_t)((solid ? kSomeSolid : 0) | (air ? kSomeAir : 0));
    if constexpr (kCount) {
        if (valid) {
            atomicAdd(&a.work[0], 1ull);
            atomicAdd(&a.work[1], (unsigned long long)caves);
            atomicAdd(&a.work[5], (unsigned long long)(y1 > y0 ? y1 - y0 : 0));
        }
    }
}

// Items of a persistent kernel shared within the workgroup: workgroup b owns items b,
// b + gridDim.x, ... (`total` items in all; interleaved, so every workgroup gets items
// of every chunk and their totals even out) and its waves take them through the LDS
// counter `next` (zeroed before the workgroup's first barrier).  No global atomic per
// item: one shared counter serves only about 77,000 grabs per ms on MI355X, and each
// grab is a round trip to memory.  Returns the item, or -1 when the workgroup's are done.
__device__ __forceinline__ int wg_next_item(int* next, int total) {
    const int mine = (total - (int)blockIdx.x + (int)gridDim.x - 1) / (int)gridDim.x;
    int j = 0;
    if ((threadIdx.x & 63) == 0) j = atomicAdd(next, 1);
    j = __builtin_amdgcn_readfirstlane(j);
    return j < mine ? (int)blockIdx.x + (int)gridDim.x * j : -1;
}

// Persistent: the grid fills the machine once (one or two 1024-thread workgroups per
// CU, a launch-shape parameter), each workgroup loads the noise tables once, and its
// waves take 64-column items from the workgroup's share (wg_next_item: 1.01-1.04 ms ->
// 0.99-1.00 ms against one global queue).
// kCount adds the work counters of lvn_batch_work (a separate instantiation, so
// the timed kernels carry no counting code).
// At most 80 SGPRs and 64 VGPRs: two 1024-thread workgroups then fit a CU (8 waves per
// SIMD; 50 to 54 SGPRs spill into VGPR lanes), which the tuner takes where the pass is a
// chain of height-term lookups per column (the reference's terrain field: 0.69 -> 0.57 ms
// on its clipmap batch); the cave field's pass takes the same time either way.
template <bool kCount, int kKind>
__global__ __launch_bounds__(1024) __attribute__((amdgpu_num_sgpr(80), amdgpu_waves_per_eu(8, 8))) void k_density(
    KArgs a, int chunks) {
    __shared__ NoiseLds T;
    __shared__ int next_local;
    if (threadIdx.x == 0) next_local = 0;
    load_noise_tables(T, a.perm, a.grads);  // ends with a barrier
    const int groups = a.G.col_groups;
    const int items_per_chunk = groups * a.ysplit;  // (y-segment, column group) pairs
    const int total = items_per_chunk * chunks;
    for (;;) {
        const int item = wg_next_item(&next_local, total);
        if (item < 0) break;
        const int chunk = item / items_per_chunk;
        const int r = item - chunk * items_per_chunk;
        const int seg = r / groups;
        density_column<kCount, kKind>(a, T, chunk, seg, r - seg * groups);
    }
}

// ---------------------------------------------------------------------------
// Brushes.  A chunk's op list is walked by whole waves: 64 ops are loaded at once, one per
// lane, and each is then read lane by lane into scalar registers, so an op costs a dozen
// v_readlane instead of two dependent memory round trips.
// ---------------------------------------------------------------------------
struct WaveOps {
    const DevOp* ops;
    const int* index;
    int n, group;       // ops in the list; the group of 64 held, or -1
    uint32_t w[16];     // the lane's op

    __device__ __forceinline__ WaveOps(const KArgs& a, const ChunkDesc& cd)
        : ops(a.ops), index(a.op_index + cd.op_start), n(cd.op_count), group(-1) {}
    // Holds ops 64 g .. 64 g + 63 of the list (a lane past its end holds the last op).
    __device__ __forceinline__ void hold(int g) {
        if (g == group) return;
        group = g;
        const int k = min(64 * g + (int)(threadIdx.x & 63), n - 1);
        const uint4* p = reinterpret_cast<const uint4*>(ops + index[k]);
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const uint4 v = p[q];
            w[4 * q] = v.x;
            w[4 * q + 1] = v.y;
            w[4 * q + 2] = v.z;
            w[4 * q + 3] = v.w;
        }
    }
    __device__ __forceinline__ DevOp mine() const {
        DevOp op;
        __builtin_memcpy(&op, w, sizeof(op));
        return op;
    }
    // Op k of the list, the same in every lane.
    __device__ __forceinline__ DevOp at(int k) {
        static_assert(sizeof(DevOp) == 64, "16 words");
        hold(k >> 6);
        uint32_t u[16];
#pragma unroll
        for (int i = 0; i < 16; ++i) u[i] = (uint32_t)__builtin_amdgcn_readlane((int)w[i], k & 63);
        DevOp op;
        __builtin_memcpy(&op, u, sizeof(op));
        return op;
    }
};

// The chunks with brushes or a cached field (k_clear_counters): special[0] of them, in
// special[1 ..].
__device__ __forceinline__ int special_chunks(const KArgs& a) { return a.special[0]; }
__device__ __forceinline__ int special_chunk(const KArgs& a, int i) {
    return __builtin_amdgcn_readfirstlane(a.special[1 + i]);
}

// Deals items 0, 1, ... of one list after another round `waves` waves: the first item of the
// current list for this wave, given how many earlier lists' items were dealt.
__device__ __forceinline__ int first_dealt(int wave, int dealt, int waves) {
    return wave >= dealt ? wave - dealt : wave - dealt + waves;
}

// The sum over this lane and those below it.
__device__ __forceinline__ int wave_upto(int v) {
#define LVN_UPTO(ctrl, rows) v += __builtin_amdgcn_update_dpp(0, v, ctrl, rows, 0xf, false);
    LVN_UPTO(0x111, 0xf)  // row_shr 1, 2, 4, 8: within a row of 16
    LVN_UPTO(0x112, 0xf)
    LVN_UPTO(0x114, 0xf)
    LVN_UPTO(0x118, 0xf)
    LVN_UPTO(0x142, 0xa)  // row_bcast 15: rows 0 and 2 into 1 and 3
    LVN_UPTO(0x143, 0xc)  // row_bcast 31: the first two rows into the others
#undef LVN_UPTO
    return v;
}

// ---------------------------------------------------------------------------
// CSG material override (CSG_HermiteIndices + BrushMaterial,
// cl/apply_csg_operation.cl:114-140,179-210): the last op whose brush contains a sample sets
// its material.  A wave takes a run of tiles of 16 x 4 x 8 samples along z, finds the ops whose
// bounding sphere reaches the run's column (64 tests at a time), then those that reach a tile,
// and walks these from the last to the first, a sample being settled by the first that holds
// it.  Runs of all brushed chunks are dealt flat over the grid's waves: a wave reads only the
// chunks of its own runs (when every wave went through the whole list of brushed chunks, two
// dependent reads each, the list's length was the time where ops are few: 92 us for 124
// chunks).  A run is one tile until every wave has two of them, then longer, so most columns
// of a chunk under a few ops cost one test.  Bound by vector issue.  Stage times in us, ops one
// after another over each chunk with a barrier after each / every wave through the list / this:
// one chunk of the reference's terrain under 60 brushes 100 / 18 / 18.5, 24 such chunks 104 / 35 /
// 27.5, its clipmap 107 / 44 / 30; 512 cave chunks under 256 brushes 34.5 / 92 / 32.5, under 1,024
// boxes 104 / 134 / 82; the cave clipmap 35 / 61 / 28.  (2,048 workgroups: 41 us for the 512 cave
// chunks, 37 for the 24; tiles in runs along x, tested one by one: 48 and 48.)
// ---------------------------------------------------------------------------
constexpr int kCsgX = 16, kCsgY = 4, kCsgZ = 8;  // 64 lanes over x and y, 8 layers each
constexpr int kCsgBlocks = 4096;
constexpr int kCsgRunsPerWave = 2;

// Squared distance from a point's coordinate to the stretch [lo, hi]; NaN for a coordinate that
// is no number, which a brush's distance ignores along its axes: such a brush reaches anywhere.
__device__ __forceinline__ float off_stretch(float lo, float hi, float o) {
    const float d = fmaxf(fmaxf(lo - o, o - hi), 0.f);
    return d * d + (o - o);
}

// The tiles of column (jx, jy) from layer l0 to below l1.
__device__ __forceinline__ void csg_run(const KArgs& a, const ChunkDesc& cd, WaveOps& list, uint8_t* mat, int jx, int jy,
                                        int l0, int l1) {
    const int F = a.G.F, lane = threadIdx.x & 63, n = cd.op_count;
    const int x0 = jx * kCsgX, y0 = jy * kCsgY;
    const int x = x0 + (lane & (kCsgX - 1)), y = y0 + lane / kCsgX;
    // the column's sides and each tile's are positions of its own samples, rounded as these
    // are: from 2^24 voxels on a sum of rounded numbers could leave some outside
    const float lox = (float)(x0 * cd.scale + cd.off[0]), hix = (float)((x0 + kCsgX - 1) * cd.scale + cd.off[0]);
    const float loy = (float)(y0 * cd.scale + cd.off[1]), hiy = (float)((y0 + kCsgY - 1) * cd.scale + cd.off[1]);
    const float px = (float)(x * cd.scale + cd.off[0]), py = (float)(y * cd.scale + cd.off[1]);
    float r2 = 0.f, d2 = 0.f, oz = 0.f;  // of the lane's op of the group held: reach, distance from the column
    uint64_t reach = 0;                  // the ops of the group that reach the column
    auto hold = [&](int g) {
        list.hold(g);
        const DevOp op = list.mine();
        const float r = op.radius + 1.f;
        r2 = r * r;
        oz = op.oz;
        d2 = off_stretch(lox, hix, op.ox) + off_stretch(loy, hiy, op.oy) + (oz - oz);
        reach = __ballot(64 * g + lane < n && !(d2 > r2));
    };
    const int last = (n - 1) >> 6;
    if (last == 0) {
        hold(0);
        if (!reach) return;
    }
    for (int l = l0; l < l1; ++l) {
        const int z0 = l * kCsgZ;
        const float loz = (float)(z0 * cd.scale + cd.off[2]), hiz = (float)((z0 + kCsgZ - 1) * cd.scale + cd.off[2]);
        unsigned outside = x < F && y < F ? 0u : 0xffu;  // a bit per layer of samples
        if (z0 + kCsgZ > F) outside |= 0xffu << (F - z0);
        unsigned settled = outside;
        int to[kCsgZ] = {};
        for (int g = last; g >= 0; --g) {
            if (last) hold(g);
            uint64_t near = reach & __ballot(!(d2 + off_stretch(loz, hiz, oz) > r2));
            while (near && __ballot((settled & 0xffu) != 0xffu)) {
                const int b = 63 - (int)__builtin_clzll(near);
                near &= ~(1ull << b);
                const DevOp u = list.at(64 * g + b);
                const int newm = u.type == 0 ? (int)(uint8_t)u.material : kAir;
#pragma unroll
                for (int k = 0; k < kCsgZ; ++k) {
                    const float pz = (float)((z0 + k) * cd.scale + cd.off[2]);
                    const bool take = !((settled >> k) & 1u) && brush_density(u, px, py, pz) <= 0.f;
                    to[k] = take ? newm : to[k];
                    settled |= take ? 1u << k : 0u;
                }
            }
        }
        const unsigned write = settled & ~outside;
#pragma unroll
        for (int k = 0; k < kCsgZ; ++k)
            if ((write >> k) & 1u) mat[field_index(a.G, x, y, z0 + k)] = (uint8_t)to[k];
    }
}

__global__ __launch_bounds__(256) void k_csg(KArgs a) {
    const int F = a.G.F;
    const int waves = grid_waves();
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6) * (int)gridDim.x + (int)blockIdx.x);
    const int tx = (F + kCsgX - 1) / kCsgX, ty = (F + kCsgY - 1) / kCsgY, tz = (F + kCsgZ - 1) / kCsgZ;
    const int columns = tx * ty, lists = special_chunks(a);
    const int runs = max(1, min(tz, (int)((long)kCsgRunsPerWave * waves / max(1, columns * lists))));
    const int per = (tz + runs - 1) / runs;  // tiles of a run
    const int items = columns * runs, total = lists * items;
    for (int i = wave; i < total; i += waves) {
        const int q = i / items, j = i - q * items;
        const int chunk = special_chunk(a, q);
        const ChunkDesc cd = a.chunks[chunk];  // a copy: the stores could alias it
        if (cd.op_count == 0) continue;
        const int run = j / columns, c = j - run * columns, jy = c / tx;
        WaveOps list(a, cd);
        csg_run(a, cd, list, slot_ptr<uint8_t>(a, chunk, a.L.mat), c - jy * tx, jy, run * per, min(tz, run * per + per));
    }
}

// ---------------------------------------------------------------------------
// Edge classification (FindFieldEdges, cl/density_field.cl:41-76) as bit rows.
// k_solid_rows packs the post-CSG "not air" test of every sample into rows of
// F bits (y, z fixed); k_rows turns three neighbouring rows into the x, y
// and z edge masks of a hermite row with a few 64-bit operations, so a chunk's
// 3 H^3 edge slots are classified by H^2 threads.
// ---------------------------------------------------------------------------
constexpr int kRowsPerBlock = 16;  // sample rows staged per wave

// Rows [16 b, 16 b + 16) of a chunk from its materials, by one wave; `stage` is the wave's.
__device__ __forceinline__ void solid_block(const KArgs& a, int chunk, int b, uint32_t* stage) {
    const Geometry& G = a.G;
    const int F = G.F, lane = threadIdx.x & 63;
    const uint32_t* mat = slot_ptr<const uint32_t>(a, chunk, a.L.mat);
    uint64_t* S = slot_ptr<uint64_t>(a, chunk, a.L.solid);
    const uint8_t* bytes = reinterpret_cast<const uint8_t*>(stage);
    const int words_total = G.field_samples >> 2;  // F is even, so F^3 is a multiple of 8
    const int block_words = (kRowsPerBlock * F) >> 2;
    // bytes [16 F b, 16 F (b + 1)): 4-byte aligned
    const int w0 = b * block_words;
    for (int j = lane; j < block_words; j += 64)
        if (w0 + j < words_total) stage[j] = mat[w0 + j];
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    // The block's rows are 2 * rows consecutive words of S: lane 2k keeps row k's low
    // word and lane 2k + 1 its high word, and one store writes them all.
    const int rows = min(kRowsPerBlock, G.field_rows - b * kRowsPerBlock);
    uint64_t word = 0;
    for (int k = 0; k < rows; ++k) {
        const bool s0 = lane < F && bytes[k * F + lane] != kAir;
        const bool s1 = lane + 64 < F && bytes[k * F + lane + 64] != kAir;
        const uint64_t lo = __ballot(s0), hi = __ballot(s1);
        if (lane == 2 * k) word = lo;
        if (lane == 2 * k + 1) word = hi;
    }
    if (lane < 2 * rows) S[2 * b * kRowsPerBlock + lane] = word;
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
}

// A batch's chunks without brushes have solid planes, each turned by its own workgroups.  So
// are the blocks of those with materials while a chunk has a wave for each; in larger batches
// these, which are few, are dealt round all waves of the launch: a brushed chunk's five
// workgroups took 14 blocks a wave one after another, and the launch waited for them (1,800
// clipmap chunks 64 -> 30 us, 512 cave chunks 56 -> 44; 16 chunks 8 us, dealt 12).
__global__ __launch_bounds__(256) void k_solid_rows(KArgs a) {
    __shared__ uint32_t stage[4][kRowsPerBlock * 66 / 4];
    const int chunk = blockIdx.y;
    const Geometry& G = a.G;
    const int F = G.F;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int blocks = (G.field_rows + kRowsPerBlock - 1) / kRowsPerBlock;
    const bool planes = chunk_mat_free(a, a.chunks[chunk]);  // uniform over the workgroup
    const bool deal = a.mat_free && waves_per_chunk() < blocks;
    if (!planes && !deal)
        for (int b = wave_in_chunk(); b < blocks; b += waves_per_chunk()) solid_block(a, chunk, b, stage[wave]);
    if (planes) {
        // the sides its items met, for the kernels from here on (an atomic per item instead
        // cost the density pass 50 us on 1,800 chunks)
        uint64_t* S = slot_ptr<uint64_t>(a, chunk, a.L.solid);
        const uint8_t* met = slot_ptr<const uint8_t>(a, chunk, a.L.sides);
        int mine = 0;
        for (int i = lane; i < G.col_groups * a.ysplit; i += 64) mine |= met[i];
        const int sides = (__ballot(mine & kSomeSolid) ? kSomeSolid : 0) | (__ballot(mine & kSomeAir) ? kSomeAir : 0);
        if (blockIdx.x == 0 && threadIdx.x == 0) a.counters[chunk].sides = sides;
        // Row (y, z) is bits [F z, F z + F) of plane y: a 64-bit window of two or three
        // consecutive group words, then F - 64 bits above it (none when F <= 64).
        const uint64_t* P = slot_ptr<const uint64_t>(a, chunk, a.L.planes);
        const uint64_t lo_mask = F >= 64 ? ~0ull : ((1ull << F) - 1ull);
        const uint64_t hi_mask = F > 64 ? ((1ull << (F - 64)) - 1ull) : 0ull;
        const int rows = sides == (kSomeSolid | kSomeAir) ? G.field_rows : 0;
        for (int r = thread_in_chunk(); r < rows; r += threads_per_chunk()) {
            const int z = div_magic(r, G.magic_f), y = r - z * F;
            const int t0 = F * z, g0 = t0 >> 6, sh = t0 & 63;
            const uint64_t w0 = P[g0 * F + y];
            const uint64_t w1 = g0 + 1 < G.col_groups ? P[(g0 + 1) * F + y] : 0ull;
            const uint64_t w2 = g0 + 2 < G.col_groups ? P[(g0 + 2) * F + y] : 0ull;
            const uint64_t lo = sh ? (w0 >> sh) | (w1 << (64 - sh)) : w0;
            const uint64_t hi = sh ? (w1 >> sh) | (w2 << (64 - sh)) : w1;
            S[2 * r] = lo & lo_mask;
            S[2 * r + 1] = hi & hi_mask;
        }
    }
    if (!deal) return;
    const int lists = special_chunks(a), waves = (int)(gridDim.x * gridDim.y * (blockDim.x >> 6));
    // consecutive workgroups take distant blocks, so a few blocks spread over the CUs
    const int first = __builtin_amdgcn_readfirstlane((int)((threadIdx.x >> 6) * gridDim.x + blockIdx.x) * (int)gridDim.y +
                                                     (int)blockIdx.y);
    for (int i = first; i < lists * blocks; i += waves)
        solid_block(a, special_chunk(a, i / blocks), i % blocks, stage[wave]);
}

// Edge rows by the first `edge_blocks` workgroups of a chunk, voxel rows by the others: both
// read only the solid rows, so one launch serves both (and the kernels after it: one scan,
// one compaction), three launches of about 5 us less for one chunk.  A row without edges
// stores its count alone, which spares 70% of the 243 MB of words of a clipmap batch: its
// words are whatever the slot held before.  The line heights and the lists skip such a row by
// its count; the QEF loads the words of all four rows round a voxel, and uses a row's only for
// an edge between corners of different sign, and such an edge is in the row.
// Row counts are packed: edges in the low half, y-edges in the high half.
__device__ __forceinline__ void edge_rows(const KArgs& a, int chunk, int thread, int threads) {
    const Geometry& G = a.G;
    const int H = G.H, F = G.F;
    const uint64_t* S = slot_ptr<const uint64_t>(a, chunk, a.L.solid);
    uint64_t* E = slot_ptr<uint64_t>(a, chunk, a.L.e_rows);
    uint32_t* count = slot_ptr<uint32_t>(a, chunk, a.L.e_count);
    const uint64_t mlo = H >= 64 ? ~0ull : ((1ull << H) - 1ull);  // x in [0, H)
    const uint64_t mhi = H > 64 ? 1ull : 0ull;                     // x = 64
    for (int r = thread; r < G.edge_rows; r += threads) {
        const int z = div_magic(r, G.magic_h), y = r - z * H;
        const int s0 = y + F * z;
        const uint64_t alo = S[2 * s0], ahi = S[2 * s0 + 1];                   // (y, z)
        const uint64_t blo = S[2 * (s0 + 1)], bhi = S[2 * (s0 + 1) + 1];       // (y + 1, z)
        const uint64_t clo = S[2 * (s0 + F)], chi = S[2 * (s0 + F) + 1];       // (y, z + 1)
        const uint64_t xlo = (alo ^ shift_next(alo, ahi)) & mlo;
        const uint64_t xhi = (ahi ^ (ahi >> 1)) & mhi;
        const uint64_t ylo = (alo ^ blo) & mlo, yhi = (ahi ^ bhi) & mhi;
        const uint64_t zlo = (alo ^ clo) & mlo, zhi = (ahi ^ chi) & mhi;
        const uint64_t hi = xhi | (yhi << 1) | (zhi << 2);
        const int ny = __popcll(ylo) + (int)((hi >> 1) & 1ull);
        const int n = __popcll(xlo) + __popcll(ylo) + __popcll(zlo) + __popcll(hi);
        if (n) {
            E[4 * r] = xlo;
            E[4 * r + 1] = ylo;
            E[4 * r + 2] = zlo;
            E[4 * r + 3] = hi;
        }
        count[r] = (uint32_t)n | ((uint32_t)ny << 16);
    }
}

// A voxel is active when its 8 corners are not all solid or all air (FindActiveVoxels,
// cl/octree.cl:142-223): over a voxel row, the AND and OR of the four sample rows around it
// and their x + 1 shifts.  Segment `seg` of 64 voxels holds 64 / N voxel rows.
__device__ __forceinline__ void voxel_rows(const KArgs& a, int chunk, int thread, int threads) {
    const Geometry& G = a.G;
    const int N = G.N, F = G.F;
    const uint64_t* S = slot_ptr<const uint64_t>(a, chunk, a.L.solid);
    uint64_t* vmask = slot_ptr<uint64_t>(a, chunk, a.L.v_mask);
    const int per_seg = N >= 64 ? 1 : 64 / N;
    const uint64_t nmask = N >= 64 ? ~0ull : ((1ull << N) - 1ull);
    for (int seg = thread; seg < G.voxel_segs; seg += threads) {
        uint64_t m = 0;
        for (int k = 0; k < per_seg; ++k) {
            const int vr = seg * per_seg + k;  // voxel row y + N z
            const int y = vr & (N - 1), z = vr >> G.depth;
            const int s0 = y + F * z;
            const int rows[4] = {s0, s0 + 1, s0 + F, s0 + F + 1};
            uint64_t all = ~0ull, any = 0ull;
#pragma unroll
            for (int c = 0; c < 4; ++c) {
                const uint64_t lo = S[2 * rows[c]], hi = S[2 * rows[c] + 1];
                const uint64_t nx = shift_next(lo, hi);
                all &= lo & nx;
                any |= lo | nx;
            }
            m |= ((any & ~all) & nmask) << (k * N);
        }
        vmask[seg] = m;
    }
}

__global__ __launch_bounds__(256) void k_rows(KArgs a, int edge_blocks) {
    const int chunk = blockIdx.y;
    if (chunk_uniform(a, chunk)) return;
    if ((int)blockIdx.x < edge_blocks)
        edge_rows(a, chunk, thread_in_chunk(), edge_blocks * 256);
    else
        voxel_rows(a, chunk, thread_in_chunk() - edge_blocks * 256, ((int)gridDim.x - edge_blocks) * 256);
}

// ---------------------------------------------------------------------------
// Exclusive scans, one workgroup per chunk and list (replaces the recursive Scan /
// ExclusiveScan with its blocking readback, src/compute.cpp:344-396).
// ---------------------------------------------------------------------------
// Two counts scanned at once, in the halves of a 64-bit sum: get(i) for i in [0, n), put(i,
// sum before i); the total is returned to every thread.  Each of the 1,024 threads sums a
// run of elements, its wave scans the sums by shuffles, and one barrier joins the waves (the
// 10-step scan through LDS with two barriers a step, once per count, took 8.5 us for a
// 64^3 chunk's rows; this takes 4).
constexpr int kScanThreads = 1024;
template <typename Get, typename Put>
__device__ __forceinline__ uint64_t block_scan(int n, uint64_t* wsum, Get get, Put put) {
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int per = (n + kScanThreads - 1) / kScanThreads;
    const int b0 = min(n, tid * per), b1 = min(n, b0 + per);
    uint64_t sum = 0;
    for (int i = b0; i < b1; ++i) sum += get(i);
    uint64_t run = sum;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
        const uint64_t u = __shfl_up(run, off);
        if (lane >= off) run += u;
    }
    __syncthreads();  // wsum may still be read from an earlier scan
    if (lane == 63) wsum[wave] = run;
    __syncthreads();
    uint64_t before = 0, total = 0;
#pragma unroll
    for (int w = 0; w < kScanThreads / 64; ++w) {
        const uint64_t v = wsum[w];
        if (w < wave) before += v;
        total += v;
    }
    uint64_t at = before + run - sum;
    for (int i = b0; i < b1; ++i) {
        put(i, at);
        at += get(i);
    }
    return total;
}
__device__ __forceinline__ uint64_t halves(uint32_t packed) { return (packed & 0xffffu) | ((uint64_t)(packed >> 16) << 32); }

// Edge rows (blockIdx.x 0) and voxel segments (1).
__global__ __launch_bounds__(kScanThreads) void k_scan_rows(KArgs a) {
    __shared__ uint64_t wsum[kScanThreads / 64];
    const int chunk = blockIdx.y;
    if (chunk_uniform(a, chunk)) return;  // its counters stay cleared
    Counters* cnt = a.counters + chunk;
    if (blockIdx.x == 0) {
        const uint32_t* count = slot_ptr<const uint32_t>(a, chunk, a.L.e_count);
        int2* base = slot_ptr<int2>(a, chunk, a.L.e_base);
        const uint64_t t = block_scan(a.G.edge_rows, wsum, [&](int i) { return halves(count[i]); },
                                      [&](int i, uint64_t at) { base[i] = make_int2((int)(uint32_t)at, (int)(at >> 32)); });
        if (threadIdx.x == 0) {
            const int n = (int)(uint32_t)t;
            cnt->edges = min(n, a.caps.edges);
            cnt->edges_y = min((int)(t >> 32), a.caps.edges);
            if (n > a.caps.edges) atomicOr(&cnt->status, kStatusEdgeOverflow);
        }
    } else {
        const uint64_t* mask = slot_ptr<const uint64_t>(a, chunk, a.L.v_mask);
        int* base = slot_ptr<int>(a, chunk, a.L.v_base);
        const int n = (int)block_scan(a.G.voxel_segs, wsum, [&](int i) { return (uint64_t)__popcll(mask[i]); },
                                      [&](int i, uint64_t at) { base[i] = (int)at; });
        if (threadIdx.x == 0) {
            cnt->voxels = min(n, a.caps.voxels);
            if (n > a.caps.voxels) atomicOr(&cnt->status, kStatusVoxelOverflow);
        }
    }
}

// ---------------------------------------------------------------------------
// Edge compaction (CompactEdges, cl/density_field.cl:80-92): the edge id is
// ((x | y << S | z << 2S) << 2) | axis (cl/density_field.cl:63,74).
// ---------------------------------------------------------------------------
// The ids of every hermite row's edges in slot order (x, then axis), and each edge's
// crossing position (y-edges first, then x and z edges).  A wave takes 64 consecutive
// rows r = y + H z and loads their words together (lane j: row j).  Where its live rows
// are dense (kDenseRow edges or more on average) it walks them in order with lane x
// holding position x of the row: an edge's rank in the row is the popcount of the three
// edge words below its lane (lower x) plus the lower axes at its own x.  Where they are
// sparse, each lane takes one edge of the wave's run of the list: it finds the edge's row
// among the 64 bases and the edge within the row by halving the words, so 64 edges cost
// about 140 instructions however they are spread (a lane walking each row's edges cost
// 550 on the clipmap, whose rows hold a few edges each, and scattered their stores).
// Either way a store instruction writes one contiguous stretch of the ids.  `split` waves
// share 64 rows where a batch is too small to fill the chip.  Measured for the whole kernel:
// 1,800 clipmap chunks 150 -> 80 us, 512 cave chunks 160 -> 118, one 64^3 chunk 11.3 -> 5.4.
// (Dense lists, bound by their stores, gain nothing: 1,890 coarse cave chunks of 136,000 edges
// take 1,535 us, an edge kernel and a voxel kernel with 4-byte order entries took 1,525.)
constexpr int kDenseRow = 32;

__device__ __forceinline__ int wave_sum(int v) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o);
    return __builtin_amdgcn_readfirstlane(v);
}
__device__ __forceinline__ uint64_t readlane64(uint64_t v, int j) {
    const uint32_t lo = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)v, j);
    const uint32_t hi = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(v >> 32), j);
    return ((uint64_t)hi << 32) | lo;
}

// The n-th edge (from 0) of a row in slot order: its x and axis, from the row's words w
// (x, y, z edge bits of x < 64) and hi (the edges at x = 64).
__device__ __forceinline__ void nth_edge(const uint64_t w[3], uint32_t hi, int n, int& x, int& axis) {
    uint32_t b[3] = {(uint32_t)w[0], (uint32_t)w[1], (uint32_t)w[2]};
    x = 0;
    int c = __popc(b[0]) + __popc(b[1]) + __popc(b[2]);
    if (n >= c) {
        n -= c;
        x = 32;
#pragma unroll
        for (int i = 0; i < 3; ++i) b[i] = (uint32_t)(w[i] >> 32);
        c = __popc(b[0]) + __popc(b[1]) + __popc(b[2]);
        if (n >= c) {  // the three bits at x = 64
            n -= c;
            x = 64;
#pragma unroll
            for (int i = 0; i < 3; ++i) b[i] = (hi >> i) & 1;
        }
    }
#pragma unroll
    for (int s = 16; s > 0; s >>= 1) {
        const uint32_t m = (1u << s) - 1;
        c = __popc(b[0] & m) + __popc(b[1] & m) + __popc(b[2] & m);
        const int up = n >= c ? s : 0;  // (never taken at x = 64: its bits lie lowest)
        n -= up ? c : 0;
        x += up;
#pragma unroll
        for (int i = 0; i < 3; ++i) b[i] >>= up;
    }
    const int b0 = b[0] & 1, b1 = b[1] & 1;
    axis = b0 && n == 0 ? 0 : b1 && n == b0 ? 1 : 2;
}

// Last lane whose value (ascending over the lanes) is not above v.
__device__ __forceinline__ int last_lane_at(int value, int v) {
    int r = 0;
#pragma unroll
    for (int step = 32; step > 0; step >>= 1)
        if (__shfl(value, r + step) <= v) r += step;
    return r;
}

__device__ __forceinline__ void edge_compact(const KArgs& a, int chunk, int wave, int waves, int split, uint4 (*stage)[2]) {
    const Geometry& G = a.G;
    const uint64_t* E = slot_ptr<const uint64_t>(a, chunk, a.L.e_rows);
    const uint32_t* count = slot_ptr<const uint32_t>(a, chunk, a.L.e_count);
    const int2* base = slot_ptr<const int2>(a, chunk, a.L.e_base);
    int* ids = slot_ptr<int>(a, chunk, a.L.e_ids);
    int2* order = slot_ptr<int2>(a, chunk, a.L.e_order);
    const int S = G.shift, cap = a.caps.edges, order_cap = a.caps.order, ey_total = a.counters[chunk].edges_y;
    const int lane = threadIdx.x & 63;
    const uint64_t lt = lanemask_lt(lane);
    // rank k in id order; crossing position: y-edges first, then x and z edges
    auto put = [&](int k, int ky, int id, bool is_y) {
        if (k < cap) {
            ids[k] = id;
            const int pos = is_y ? ky : ey_total + (k - ky);
            if (pos < order_cap) order[pos] = make_int2(k, id);
        }
    };
    const int units = ((G.edge_rows + 63) >> 6) * split;
    for (int u = wave; u < units; u += waves) {
        const int g = u / split, part = u - g * split;
        const int rl = (g << 6) + lane;
        const int cnt = rl < G.edge_rows ? (int)(count[rl] & 0xffffu) : 0;
        uint64_t live = __ballot(cnt != 0);
        if (!live) continue;
        int kb = 0x7fffffff, kyb = 0;
        uint64_t w0 = 0, w1 = 0, w2 = 0, w3 = 0;
        if (rl < G.edge_rows) {
            const int2 b = base[rl];
            kb = b.x;
            kyb = b.y;
        }
        if (cnt) {  // a row without edges has no words
            w0 = E[4 * rl];
            w1 = E[4 * rl + 1];
            w2 = E[4 * rl + 2];
            w3 = E[4 * rl + 3];
        }
        const int total = wave_sum(cnt);
        if (total < kDenseRow * __popcll(live)) {  // sparse rows: one lane per edge
            stage[lane][0] = make_uint4((uint32_t)w0, (uint32_t)(w0 >> 32), (uint32_t)w1, (uint32_t)(w1 >> 32));
            stage[lane][1] = make_uint4((uint32_t)w2, (uint32_t)(w2 >> 32), (uint32_t)w3, (uint32_t)kyb);
            __builtin_amdgcn_wave_barrier();  // read by the wave's other lanes
            const int k_first = __builtin_amdgcn_readlane(kb, 0);
            for (int i0 = part << 6; i0 < total; i0 += split << 6) {
                const int k = k_first + min(i0 + lane, total - 1);
                const int j = last_lane_at(kb, k);  // of equal bases the last: the row with edges
                const int n = k - __shfl(kb, j);
                const uint4 p = stage[j][0], q = stage[j][1];
                const uint64_t w[3] = {(uint64_t)p.y << 32 | p.x, (uint64_t)p.w << 32 | p.z, (uint64_t)q.y << 32 | q.x};
                int x, axis;
                nth_edge(w, q.z, n, x, axis);
                const int at_x = x < 64 ? (int)(w[1] >> x) & 1 : (int)(q.z >> 1) & 1;  // the y-edge at the same x
                const int ky = (int)q.w + __popcll(w[1] & (x < 64 ? lanemask_lt(x) : ~0ull)) + (axis == 2 ? at_x : 0);
                const int r = (g << 6) + j, z = div_magic(r, G.magic_h), y = r - z * G.H;
                if (i0 + lane < total) put(k, ky, (x | y << S | z << (2 * S)) << 2 | axis, axis == 1);
            }
            __builtin_amdgcn_wave_barrier();
            continue;
        }
        for (int skip = 0; live; ++skip) {
            const int j = (int)__builtin_ctzll(live);
            live &= live - 1ull;
            if (skip % split != part) continue;
            const int r = (g << 6) + j;
            const int z = div_magic(r, G.magic_h), y = r - z * G.H;
            const int row_id = (y << S) | (z << (2 * S));
            const uint64_t ex = readlane64(w0, j), ey = readlane64(w1, j), ez = readlane64(w2, j);
            const uint64_t hi = readlane64(w3, j);
            const int k0 = __builtin_amdgcn_readlane(kb, j), ky0 = __builtin_amdgcn_readlane(kyb, j);
            const int bx = (int)((ex >> lane) & 1ull), by = (int)((ey >> lane) & 1ull), bz = (int)((ez >> lane) & 1ull);
            int k = k0 + __popcll(ex & lt) + __popcll(ey & lt) + __popcll(ez & lt);
            int ky = ky0 + __popcll(ey & lt);
            const int id = (lane | row_id) << 2;
            if (bx) put(k, ky, id, false);
            k += bx;
            if (by) put(k, ky, id | 1, true);
            k += by;
            ky += by;
            if (bz) put(k, ky, id | 2, false);
            if (hi != 0 && lane == 0) {  // x = 64 (N = 64 only): after every x < 64
                int kh = k0 + __popcll(ex) + __popcll(ey) + __popcll(ez), kyh = ky0 + __popcll(ey);
                const int id64 = (64 | row_id) << 2;
                for (int axis = 0; axis < 3; ++axis) {
                    if (!((hi >> axis) & 1ull)) continue;
                    put(kh, kyh, id64 | axis, axis == 1);
                    ++kh;
                    kyh += axis == 1 ? 1 : 0;
                }
            }
        }
    }
}

// ---------------------------------------------------------------------------
// Edge crossing + normal
// ---------------------------------------------------------------------------

// Heights along the lines of x- and z-edges.  An x-edge (x, y, z) samples the height
// term at (x + k/16, z) and a z-edge at (x, z + k/16): the same values for every y, and
// caves give a line about three crossing edges.  So the interior samples k = 1..15 of
// every line holding a crossing x- or z-edge are evaluated once, before the crossing
// kernels, by the expressions those kernels use (bit-identical values), and read back
// there.  Line (sel, x, z), sel 0 for x-edges and 1 for z-edges, starts at:
__device__ __forceinline__ int hline_index(int H, int sel, int x, int z) { return ((sel * H + z) * H + x) * kLineStride; }

// Position of the j-th set bit (from 0) of m; m has more than j set bits.
__device__ __forceinline__ int nth_bit(uint64_t m, int j) {
    int pos = 0;
#pragma unroll
    for (int w = 32; w >= 1; w >>= 1) {
        const uint64_t low = m & ((1ull << w) - 1ull);
        const int c = __popcll(low);
        if (j >= c) {
            j -= c;
            m >>= w;
            pos += w;
        } else {
            m = low;
        }
    }
    return pos;
}

// Item = (chunk, sel, z).  Items are short (a few hundred height evaluations), and a
// shared atomic queue serves only about 77,000 grabs per ms, which would bound this pass
// at 0.86 ms for 512 chunks; a static stride over the waves leaves many idle (the items
// of one wave then come from one layer of chunks, all sky or all caves).  So workgroup b
// takes items b, b + gridDim.x, ... (chunks of every layer) and its waves share them
// through an LDS counter.  The lines
// needed are the OR over y of the chunk's edge rows (x-edge or z-edge words); the lanes
// run over their samples only.  Chunks whose edges take no density crossings (the
// cached-field form) are skipped.
template <bool kCount, int kKind>
__global__ __launch_bounds__(1024) void k_height_lines(KArgs a, int chunks) {
    __shared__ NoiseLds T;
    __shared__ int next_local;
    if (threadIdx.x == 0) next_local = 0;
    load_noise_tables(T, a.perm, a.grads);  // ends with a barrier
    const Geometry& G = a.G;
    const int H = G.H;
    const int per_chunk = 2 * H;
    const int total = per_chunk * chunks;
    const int lane = threadIdx.x & 63;
    for (;;) {
        const int item = wg_next_item(&next_local, total);
        if (item < 0) break;
        const int chunk = item / per_chunk;
        const int r = item - chunk * per_chunk;
        const int sel = r / H, z = r - sel * H;
        const ChunkDesc cd = a.chunks[chunk];  // a copy: the sample loop's stores could alias it
        if (cd.mode == kModeCached || a.counters[chunk].edges == 0) continue;  // uniform over the wave
        const uint32_t* count = slot_ptr<const uint32_t>(a, chunk, a.L.e_count);
        const uint64_t* E = slot_ptr<const uint64_t>(a, chunk, a.L.e_rows);
        const int word = sel == 0 ? 0 : 2;  // x-edge or z-edge bits of x < 64
        uint64_t lo = 0, hi = 0;
        for (int y = lane; y < H; y += 64) {
            const int row = y + H * z;
            if ((count[row] & 0xffffu) == 0) continue;  // its words are not stored
            lo |= E[4 * row + word];
            hi |= (E[4 * row + 3] >> word) & 1ull;  // bit 0: x-edge, bit 2: z-edge at x = 64
        }
#pragma unroll
        for (int m = 32; m >= 1; m >>= 1) {
            lo |= __shfl_xor(lo, m);
            hi |= __shfl_xor(hi, m);
        }
        float* out = slot_ptr<float>(a, chunk, a.L.h_lines) + hline_index(H, sel, 0, z);
        const int n_lo = __popcll(lo), n = n_lo + (int)(hi & 1ull);  // hi is set only when H > 64
        unsigned nh = 0;
        for (int p = lane; p < n * kLineSamples; p += 64) {
            const int j = p / kLineSamples, k = p - j * kLineSamples + 1;
            const int x = j < n_lo ? nth_bit(lo, j) : 64;
            const int w0x = x * cd.scale + cd.off[0], w0z = z * cd.scale + cd.off[2];
            const float p0x = (float)w0x, p0z = (float)w0z;
            const float p1x = (float)(w0x + (sel == 0 ? cd.scale : 0));
            const float p1z = (float)(w0z + (sel == 1 ? cd.scale : 0));
            const float cur = (float)k * 0.0625f;  // = the sequential scan's running sum (exact)
            out[x * kLineStride + (k - 1)] = height_term<kKind>(a.F, T, p0x + (p1x - p0x) * cur, p0z + (p1z - p0z) * cur);
            ++nh;
        }
        if constexpr (kCount) atomicAdd(&a.work[2], (unsigned long long)nh);
    }
}

// The normal of FindEdgeIntersectionInfo (cl/density_field.cl:131-150): central
// differences with h = 0.001 at the arg-min sample t of the edge p0 -> p1, whose height
// term `Hbest` is reused when it was evaluated there.
template <int kKind>
__device__ __forceinline__ float4 crossing_normal(const FieldParams& Fp, const NoiseLds& T, int axis, bool ends_known,
                                                  float tbest, float Hbest, float p0x, float p0y, float p0z, float p1x,
                                                  float p1y, float p1z, unsigned& nh, unsigned& nc) {
    const float px = p0x + (p1x - p0x) * tbest;
    const float py = p0y + (p1y - p0y) * tbest;
    const float pz = p0z + (p1z - p0z) * tbest;
    const float h = 0.001f;
    // The height at the arg-min sample is only known when it was evaluated there.
    const bool hb_known = axis == 1 || !(ends_known && (tbest == 0.f || tbest == 1.f));
    const float H0 = hb_known ? Hbest : height_small<kKind>(Fp, T, px, pz);
    const float x[3] = {px, px + h, px - h}, y[3] = {py, py + h, py - h}, z[3] = {pz, pz + h, pz - h};
    float H[4];
    height_near<kKind>(Fp, T, x, z, H);
    nh += hb_known ? 4u : 5u;
    // the six samples, combine() each
    float d[6] = {py - H[0], py - H[1], y[1] - H0, y[2] - H0, py - H[2], py - H[3]};
    if (field_kind<kKind>(Fp) == LVN_FIELD_TERRAIN_CAVES) {
        constexpr int ix[6] = {1, 2, 0, 0, 0, 0}, iy[6] = {0, 0, 1, 2, 0, 0}, iz[6] = {0, 0, 0, 0, 1, 2};
#pragma unroll
        for (int i = 0; i < 6; ++i) {
            nc += !(d[i] > Fp.cave_cut) ? 1u : 0u;
            d[i] = combine<kKind>(Fp, T, d[i], x[ix[i]], y[iy[i]], z[iz[i]]);
        }
    }
    const float3 n = normalize_or_zero(d[0] - d[1], d[2] - d[3], d[4] - d[5]);
    return make_float4(n.x, n.y, n.z, tbest);
}

// FindEdgeIntersectionInfo, cl/density_field.cl:96-151: first arg-min of |d|
// over t = k/16, then a central-difference normal with h = 0.001.  The height
// term of samples that share (x, z) is evaluated once: per column (`colH`, a y-edge's, from
// the density pass), and per x- or z-edge line (`hl`, k_height_lines); the two end samples are the stored field
// samples when the field is FP32.
template <int kKind>
__device__ __forceinline__ float4 density_crossing(const KArgs& a, const NoiseLds& T, const ChunkDesc& cd, int x, int y, int z,
                                   int axis, bool ends_known, float d_start, float d_end, const float* hl,
                                   float colH, unsigned& nh, unsigned& nc) {
    const FieldParams& Fp = a.F;
    const bool caves = field_kind<kKind>(Fp) == LVN_FIELD_TERRAIN_CAVES;
    const int w0x = x * cd.scale + cd.off[0], w0y = y * cd.scale + cd.off[1], w0z = z * cd.scale + cd.off[2];
    const float p0x = (float)w0x, p0y = (float)w0y, p0z = (float)w0z;
    const float p1x = (float)(w0x + (axis == 0 ? cd.scale : 0));
    const float p1y = (float)(w0y + (axis == 1 ? cd.scale : 0));
    const float p1z = (float)(w0z + (axis == 2 ? cd.scale : 0));
    float minV = 3.402823466e+38f, tbest = 0.f, Hbest = colH, cur = 0.f;
    const bool lines = a.height_lines != 0 && axis != 1;
    // Without the cave term a sample is y - H, and every H is at hand for a y-edge (its
    // column's) and with line heights, which lie in one 64-byte line and are loaded together
    // (one after another, the 15 loads' latency was the larger part of an x- or z-edge item).
    if (!caves && ends_known && (lines || axis == 1)) {
        float Hl[kLineStride];
        if (lines) {
#pragma unroll
            for (int q = 0; q < kLineStride / 4; ++q) {
                const float4 v = reinterpret_cast<const float4*>(hl)[q];  // 16-byte aligned: lines are 64 bytes
                Hl[4 * q] = v.x;
                Hl[4 * q + 1] = v.y;
                Hl[4 * q + 2] = v.z;
                Hl[4 * q + 3] = v.w;
            }
        }
#pragma unroll
        for (int k = 0; k <= 16; ++k) {
            const float t = (float)k * 0.0625f;  // = the running sum below (exact)
            const float H = lines && k >= 1 && k <= kLineSamples ? Hl[k >= 1 && k <= kLineSamples ? k - 1 : 0] : colH;
            const float py = p0y + (p1y - p0y) * t;
            const float d = k == 0 ? fabsf(d_start) : k == 16 ? fabsf(d_end) : fabsf(py - H);
            if (d < minV) {
                tbest = t;
                minV = d;
                Hbest = H;
            }
        }
        return crossing_normal<kKind>(Fp, T, axis, ends_known, tbest, Hbest, p0x, p0y, p0z, p1x, p1y, p1z, nh, nc);
    }
    float Hn = lines ? hl[0] : 0.f;  // the next interior sample's line height, loaded a sample ahead
    for (int k = 0; k <= 16; ++k) {
        const float px = p0x + (p1x - p0x) * cur;
        const float py = p0y + (p1y - p0y) * cur;
        const float pz = p0z + (p1z - p0z) * cur;
        float d, H = colH;
        if (ends_known && k == 0) {
            d = fabsf(d_start);
        } else if (ends_known && k == 16) {
            d = fabsf(d_end);
        } else {
            if (axis != 1) {
                if (lines && k >= 1 && k <= kLineSamples) {
                    H = Hn;
                    if (k < kLineSamples) Hn = hl[k];
                } else {
                    H = height_term<kKind>(Fp, T, px, pz);
                    ++nh;
                }
            }
            nc += (caves && !((py - H) > Fp.cave_cut)) ? 1u : 0u;
            d = fabsf(combine<kKind>(Fp, T, py - H, px, py, pz));
        }
        if (d < minV) {
            tbest = cur;
            minV = d;
            Hbest = H;
        }
        cur = cur + 0.0625f;
    }
    return crossing_normal<kKind>(Fp, T, axis, ends_known, tbest, Hbest, p0x, p0y, p0z, p1x, p1y, p1z, nh, nc);
}

// The distance from an edge's middle sample to its farther end, both as they are rounded:
// half an edge below 2^23 voxels; beyond, where the middle of a short edge is no FP32 number,
// up to a whole one.  (Every sample lies between the ends: the sum that places it rounds
// monotonically.)
__device__ __forceinline__ float farther_end(float p0x, float p0y, float p0z, float ex, float ey, float ez, float mx,
                                             float my, float mz) {
    // along the edge's axis; the two across add +0
    const float back = ((mx - p0x) + (my - p0y)) + (mz - p0z);
    return fmaxf(back, ((ex + ey) + ez) - back);
}

// FindEdgeIntersectionInfo of the CSG program, cl/apply_csg_operation.cl:443-477,
// with BrushZeroCrossing (:86-110) and BrushNormal (:144-175): the first (t, op) in
// the reference's t-outer, op-inner scan whose |d| is smallest, t = k/16; then the
// normal of the last op holding that point.  Only t matters of the pair, so the scan's
// answer is the smallest k among the samples of the smallest |d|, whatever order they are
// visited in: the ops are the outer loop here (each read once instead of 17 times), and an
// op is sampled along the edge only when it can still win.  A brush's distance is
// 1-Lipschitz (a rounded rotation and the FP32 steps stay within 1e-5 of the magnitudes
// that enter it), so with |d| = m at the edge's middle no sample of the edge, at most half
// an edge away, is below m - half: an op for which that exceeds the running minimum is
// passed by.  All edges of the wave are one chunk's, `list` its ops.
__device__ __forceinline__ float4 brush_crossing(WaveOps& list, const ChunkDesc& cd, bool live, int x, int y, int z,
                                                 int axis) {
    const int w0x = x * cd.scale + cd.off[0], w0y = y * cd.scale + cd.off[1], w0z = z * cd.scale + cd.off[2];
    const float p0x = (float)w0x, p0y = (float)w0y, p0z = (float)w0z;
    const float ex = (float)(w0x + (axis == 0 ? cd.scale : 0)) - p0x;
    const float ey = (float)(w0y + (axis == 1 ? cd.scale : 0)) - p0y;
    const float ez = (float)(w0z + (axis == 2 ? cd.scale : 0)) - p0z;
    const int n = cd.op_count;
    constexpr int kMid = 8;
    float minD = 3.402823466e+38f;
    int kbest = 0;
    const float mx = p0x + ex * 0.5f, my = p0y + ey * 0.5f, mz = p0z + ez * 0.5f;
    const float half = farther_end(p0x, p0y, p0z, ex, ey, ez, mx, my, mz);
    for (int k = 0; k < n; ++k) {
        const DevOp op = list.at(k);
        const float d = fabsf(brush_density(op, mx, my, mz));
        if (d < minD) {
            minD = d;
            kbest = kMid;
        }
    }
    for (int k = 0; k < n; ++k) {
        const DevOp op = list.at(k);
        const float slack = 1e-5f * (((fabsf(mx - op.ox) + fabsf(my - op.oy)) + (fabsf(mz - op.oz) + half)) +
                                     ((fabsf(op.dx) + fabsf(op.dy)) + fabsf(op.dz)));
        const float reach = half + slack;
        const float m = fabsf(brush_density(op, mx, my, mz));
        if (__ballot(live && !(m - reach > minD)) == 0) continue;  // also taken for NaN distances
        for (int i = 0; i <= 16; ++i) {
            const float t = (float)i * 0.0625f;  // = the scan's running sum (exact)
            const float d = fabsf(brush_density(op, p0x + ex * t, p0y + ey * t, p0z + ez * t));
            if (d < minD || (d == minD && i < kbest)) {
                minD = d;
                kbest = i;
            }
        }
    }
    const float crossing = (float)kbest * 0.0625f;
    const float px = p0x + ex * crossing;
    const float py = p0y + ey * crossing;
    const float pz = p0z + ez * crossing;
    const float h = 0.001f;
    float3 nrm = make_float3(0.f, 0.f, 0.f);
    bool open = live;  // the last op holding the point decides: the first one found from the end
    for (int k = n - 1; k >= 0 && __ballot(open) != 0; --k) {
        const DevOp op = list.at(k);
        if (!open || brush_density(op, px, py, pz) > 0.f) continue;
        const float dx = brush_density(op, px + h, py, pz) - brush_density(op, px - h, py, pz);
        const float dy = brush_density(op, px, py + h, pz) - brush_density(op, px, py - h, pz);
        const float dz = brush_density(op, px, py, pz + h) - brush_density(op, px, py, pz - h);
        const float flip = op.type == 0 ? 1.f : -1.f;
        const float3 u = normalize_or_zero(dx, dy, dz);
        nrm = make_float3(flip * u.x, flip * u.y, flip * u.z);
        open = false;
    }
    return make_float4(nrm.x, nrm.y, nrm.z, crossing);
}

// The least of the wave's non-negative values, in every lane (their bits order like they do,
// and a NaN loses to any number).
__device__ __forceinline__ float wave_least(float v) { return __uint_as_float(wave_min(__float_as_uint(v))); }

// The same for one edge, the same in every lane: the ops lie one per lane, so the distances
// of 64 of them at a point are one evaluation, and an op that can win is sampled with a
// sample per lane.  About 310 instructions an edge up to 64 ops; 64 edges by the form above
// take about 180 per op, and 500 for each op that can win for any of them.
__device__ __forceinline__ float4 brush_crossing_one(WaveOps& list, const ChunkDesc& cd, int x, int y, int z, int axis) {
    const int lane = threadIdx.x & 63;
    const int w0x = x * cd.scale + cd.off[0], w0y = y * cd.scale + cd.off[1], w0z = z * cd.scale + cd.off[2];
    const float p0x = (float)w0x, p0y = (float)w0y, p0z = (float)w0z;
    const float ex = (float)(w0x + (axis == 0 ? cd.scale : 0)) - p0x;
    const float ey = (float)(w0y + (axis == 1 ? cd.scale : 0)) - p0y;
    const float ez = (float)(w0z + (axis == 2 ? cd.scale : 0)) - p0z;
    const int n = cd.op_count, groups = (n + 63) >> 6;
    constexpr float kFar = 3.402823466e+38f;
    const float mx = p0x + ex * 0.5f, my = p0y + ey * 0.5f, mz = p0z + ez * 0.5f;
    const float half = farther_end(p0x, p0y, p0z, ex, ey, ez, mx, my, mz);
    float mid = kFar;  // the lane's op's |d| at the middle (of the last group held)
    float least = kFar;
    for (int g = 0; g < groups; ++g) {
        list.hold(g);
        mid = 64 * g + lane < n ? fabsf(brush_density(list.mine(), mx, my, mz)) : kFar;
        least = fminf(least, mid);
    }
    least = wave_least(least);
    const float t = (float)min(lane, 16) * 0.0625f;  // the lane's sample (= the scan's running sum, exact)
    const float sx = p0x + ex * t, sy = p0y + ey * t, sz = p0z + ez * t;
    float best = kFar;
    for (int g = 0; g < groups; ++g) {
        if (groups > 1) {
            list.hold(g);
            mid = fabsf(brush_density(list.mine(), mx, my, mz));
        }
        const DevOp own = list.mine();
        const float slack = 1e-5f * (((fabsf(mx - own.ox) + fabsf(my - own.oy)) + (fabsf(mz - own.oz) + half)) +
                                     ((fabsf(own.dx) + fabsf(own.dy)) + fabsf(own.dz)));
        const float reach = half + slack;
        uint64_t left = __ballot(64 * g + lane < n && !(mid - reach > least));  // also taken for NaN distances
        while (left) {
            const DevOp op = list.at(64 * g + (int)__builtin_ctzll(left));
            left &= left - 1;
            const float d = fabsf(brush_density(op, sx, sy, sz));
            if (d < best) best = d;
        }
    }
    if (lane > 16) best = kFar;
    const float found = wave_least(best);
    const int kbest = (int)__builtin_ctzll(__ballot(best == found));
    const float crossing = (float)kbest * 0.0625f;
    const float px = p0x + ex * crossing;
    const float py = p0y + ey * crossing;
    const float pz = p0z + ez * crossing;
    const float h = 0.001f;
    for (int g = groups - 1; g >= 0; --g) {  // the last op holding the point decides
        list.hold(g);
        const uint64_t in = __ballot(64 * g + lane < n && !(brush_density(list.mine(), px, py, pz) > 0.f));
        if (!in) continue;
        const DevOp op = list.at(64 * g + 63 - (int)__builtin_clzll(in));
        // lanes 0 .. 5: the points h before and behind along each axis
        const float step = lane & 1 ? -h : h;
        const float d = brush_density(op, lane >> 1 == 0 ? px + step : px, lane >> 1 == 1 ? py + step : py,
                                      lane >> 1 == 2 ? pz + step : pz);
        float q[6];
#pragma unroll
        for (int i = 0; i < 6; ++i) q[i] = __uint_as_float((uint32_t)__builtin_amdgcn_readlane((int)__float_as_uint(d), i));
        const float flip = op.type == 0 ? 1.f : -1.f;
        const float3 u = normalize_or_zero(q[0] - q[1], q[2] - q[3], q[4] - q[5]);
        return make_float4(flip * u.x, flip * u.y, flip * u.z, crossing);
    }
    return make_float4(0.f, 0.f, 0.f, crossing);
}

// The end samples of edge (x, y, z, axis), field indices i0 and i1: the stored field, or,
// for a field without the cave term whose density a batch does not store (dens_cols),
// y - H with H from the column heights: density_column's expression, bit for bit (its
// sample is combine(wy - H) = wy - H for such a field).
__device__ __forceinline__ float2 edge_ends(const KArgs& a, int chunk, const ChunkDesc& cd, int x, int y, int z, int axis,
                                           int i0, int i1) {
    if (a.dens_cols) {
        const float* hc = slot_ptr<const float>(a, chunk, a.L.h_cols);
        const int F = a.G.F;
        const float H0 = hc[x + F * z];
        const float H1 = axis == 1 ? H0 : hc[(x + (axis == 0 ? 1 : 0)) + F * (z + (axis == 2 ? 1 : 0))];
        const float wy0 = (float)(y * cd.scale + cd.off[1]);
        const float wy1 = (float)((y + (axis == 1 ? 1 : 0)) * cd.scale + cd.off[1]);
        return make_float2(wy0 - H0, wy1 - H1);
    }
    const float* dens = slot_ptr<const float>(a, chunk, a.L.density);
    return make_float2(dens[i0], dens[i1]);
}

// The hermite point, axis and field indices of an edge id.
struct EdgeAt {
    int x, y, z, axis, i0, i1;
};
__device__ __forceinline__ bool decode_edge(const Geometry& G, int id, EdgeAt& e) {
    e.axis = id & 3;
    const int hidx = id >> 2, msk = (1 << G.shift) - 1;
    e.x = hidx & msk;
    e.y = (hidx >> G.shift) & msk;
    e.z = (hidx >> (2 * G.shift)) & msk;
    e.i0 = field_index(G, e.x, e.y, e.z);
    e.i1 = e.i0 + (e.axis == 0 ? 1 : e.axis == 1 ? G.F : G.F * G.F);
    return e.x < G.H && e.y < G.H && e.z < G.H && e.axis <= 2;  // always so for the ids of the edge lists
}

// An edge with an endpoint whose material a brush changed takes brush data
// (src/compute_csg.cpp:97-217).
__device__ __forceinline__ bool edge_touched(const KArgs& a, int chunk, const ChunkDesc& cd, int i0, int i1) {
    if (cd.op_count == 0) return false;
    const uint8_t* mat = slot_ptr<const uint8_t>(a, chunk, a.L.mat);
    const uint8_t* orig = slot_ptr<const uint8_t>(a, chunk, a.L.orig);
    return mat[i0] != orig[i0] || mat[i1] != orig[i1];
}

// One compacted edge's density crossing; edges with brush data are k_edge_data's.
template <bool kCount, int kKind>
__device__ __forceinline__ void cross_edge(const KArgs& a, const NoiseLds& T, int chunk, int i, int id) {
    const Geometry& G = a.G;
    const ChunkDesc& cd = a.chunks[chunk];
    EdgeAt e;
    if (!decode_edge(G, id, e)) {
        atomicOr(&a.counters[chunk].status, kStatusLookupMiss);
        return;
    }
    if (edge_touched(a, chunk, cd, e.i0, e.i1)) return;
    const bool ends = !a.fp16;
    const float2 de = ends ? edge_ends(a, chunk, cd, e.x, e.y, e.z, e.axis, e.i0, e.i1) : make_float2(0.f, 0.f);
    const float* hl = slot_ptr<const float>(a, chunk, a.L.h_lines) + hline_index(G.H, e.axis == 2 ? 1 : 0, e.x, e.z);
    const float colH = e.axis == 1 ? slot_ptr<const float>(a, chunk, a.L.h_cols)[e.x + G.F * e.z] : 0.f;
    unsigned nh = 0, nc = 0;
    const float4 out = density_crossing<kKind>(a, T, cd, e.x, e.y, e.z, e.axis, ends, de.x, de.y, hl, colH, nh, nc);
    if constexpr (kCount) {
        atomicAdd(&a.work[2], (unsigned long long)nh);
        atomicAdd(&a.work[3], (unsigned long long)nc);
        atomicAdd(&a.work[6], 1ull);
    }
    slot_ptr<float4>(a, chunk, a.L.e_data)[i] = out;
}

// A chunk's edges are crossed in two runs, its y-edges (one height evaluation per
// edge) and its x and z edges (one per sample), so that a wave holds one kind and
// skips the per-sample height work when all its edges are y-edges.
// The chunks of a launch whose crossings come from the field: not the cached ones.
__device__ __forceinline__ int edge_items_y(const Counters& c, int per_item) {
    return (min(c.edges_y, c.edges) + per_item - 1) / per_item;
}
__device__ __forceinline__ int edge_items_xz(const Counters& c, int per_item) {
    return (c.edges - min(c.edges_y, c.edges) + per_item - 1) / per_item;
}
// Slot `e` of the chunk's item j: the edge's rank (index into e_ids / e_data) and id, rank -1
// past the end.
__device__ __forceinline__ int2 edge_of_item(const KArgs& a, int chunk, int j, int e, int per_item) {
    const Counters& c = a.counters[chunk];
    const int ey = min(c.edges_y, c.edges), ny = (ey + per_item - 1) / per_item;
    const int pos = j < ny ? j * per_item + e : ey + (j - ny) * per_item + e;
    if (j < ny ? pos >= ey : pos >= c.edges) return make_int2(-1, 0);
    if (pos >= a.caps.order) return make_int2(-1, 0);  // more edges than the chunk's voxels can have: refused
    const int2 o = slot_ptr<const int2>(a, chunk, a.L.e_order)[pos];
    return (unsigned)o.x < (unsigned)c.edges ? o : make_int2(-1, 0);  // entries past a capped list are not written
}

// The last chunk c with prefix[c] <= item (prefix ascends from 0, item < prefix[chunks]): the
// wave looks at 64 chunks spread over the range at once, so 4,096 chunks take two loads,
// where a binary search waits for 11 one after another.
__device__ __forceinline__ int chunk_of_item(const int* prefix, int chunks, int item) {
    const int lane = threadIdx.x & 63;
    int lo = 0, n = chunks;
    while (n > 1) {
        const int step = (n + 63) >> 6, at = lane * step;
        const int found = __popcll(__ballot(at < n && prefix[lo + at] <= item));  // >= 1: lane 0's holds
        lo += (found - 1) * step;
        n = min(step, n - (found - 1) * step);
    }
    return lo;
}

// Items of `per_item` edges (64 / lanes per edge) over all chunks: item_prefix[c] =
// sum over earlier chunks of the chunk's y-edge and x/z-edge items, item_prefix[chunks] =
// total; a cached chunk has none.  One workgroup of 256 threads.
constexpr int kEdgeDataThreads = 256;
__device__ __forceinline__ void edge_items(const KArgs& a, int chunks, int per_item, int* wsum) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    int carry = 0;
    for (int base = 0; base < chunks; base += kEdgeDataThreads) {
        const int c = base + (int)threadIdx.x;
        int v = 0;
        if (c < chunks && a.chunks[c].mode != kModeCached)
            v = edge_items_y(a.counters[c], per_item) + edge_items_xz(a.counters[c], per_item);
        const int sum = wave_upto(v);
        if (lane == 63) wsum[wave] = sum;
        __syncthreads();
        int before = carry, all = carry;
#pragma unroll
        for (int w = 0; w < kEdgeDataThreads / 64; ++w) {
            if (w < wave) before += wsum[w];
            all += wsum[w];
        }
        if (c < chunks) a.item_prefix[c] = before + sum - v;
        carry = all;
        __syncthreads();
    }
    if (threadIdx.x == 0) a.item_prefix[chunks] = carry;
}

// The edges whose hermite data needs no field evaluation: those a brush touched, and in
// the cached form every other one, which keeps its data from the old edge list.  The last
// workgroup counts the crossing kernels' items meanwhile.  The others deal the 64-edge items
// of the chunks that have such edges round the grid's waves.  Beside the crossing kernels' density path this one is short of
// neither registers nor LDS, and a few brushed chunks of a batch (whose edges each scan the
// chunk's op list) no longer hold a wave of the density queue: those were its tail.  One
// brushed 64^3 chunk of the reference's terrain meshed in 598 -> 325 us, a two-step edit of
// a cached chunk (no field evaluation at all) in 1,104 -> 761 us, 24 chunks under 256
// brushes staged, meshed and fetched in 1,554 -> 1,285 us.
// A wave finds its items among 64 lists at a time, a list per lane: three reads and a scan for
// all of them.  (Going through the lists one by one, each with two dependent reads, took 70 us
// of 124 brushed chunks' time: crossing stage 2,075 -> 2,005 us; of 24 chunks 145 -> 137, of
// 64 680 -> 666.)
// Of a few chunks, those under many brushes take short items and their touched edges one by
// one, an op per lane: 64 edges of one wave scanning 60 ops one after another were the time
// of a one-chunk call while most of the chip was idle.  One 64^3 chunk under 60 brushes 54 us
// by 64 edges a wave, 33 by items of 16 edges, 16 by 4 and by 2.  Under fewer than 20 brushes
// the scan is the shorter chain, and with more chunks it costs fewer instructions: 24 chunks
// 85 against 92 us, 64 chunks 137 against 206.  (Its own kernel: beside it the scan alone
// took 5 to 10% longer.)
constexpr int kOneEdgeItem = 4;
constexpr int kFewChunks = 8, kOneEdgeOps = 20;
template <bool kCount, bool kFew>
__global__ __launch_bounds__(kEdgeDataThreads) void k_edge_data(KArgs a, int chunks, int per_item) {
    __shared__ int wsum[kEdgeDataThreads / 64];
    if (blockIdx.x == gridDim.x - 1) {
        edge_items(a, chunks, per_item, wsum);
        return;
    }
    const Geometry& G = a.G;
    const int lane = threadIdx.x & 63;
    const int waves = (int)((gridDim.x - 1) * (blockDim.x >> 6));
    // waves are numbered across the workgroups, so a few items spread over the CUs
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6) * (int)(gridDim.x - 1) + (int)blockIdx.x);
    const int lists = special_chunks(a);
    int dealt = 0;  // items of earlier lists, modulo the number of waves
    for (int first = 0; first < lists; first += 64) {
        // 64 lists at a time, one per lane: its chunk, edges, and the items up to and with it
        int own_chunk = 0, own_edges = 0, own_items = 0;
        if (first + lane < lists) {
            own_chunk = a.special[1 + first + lane];
            own_edges = a.counters[own_chunk].edges;
            const int per = kFew && a.chunks[own_chunk].op_count >= kOneEdgeOps ? kOneEdgeItem : 64;
            own_items = (own_edges + per - 1) / per;
        }
        const int upto = wave_upto(own_items), total = __builtin_amdgcn_readlane(upto, 63);
        for (int t = first_dealt(wave, dealt, waves); t < total; t += waves) {
            const int q = __popcll(__ballot(upto <= t));  // the list of item t
            const int chunk = __builtin_amdgcn_readlane(own_chunk, q), edges = __builtin_amdgcn_readlane(own_edges, q);
            const int j = t - (__builtin_amdgcn_readlane(upto, q) - __builtin_amdgcn_readlane(own_items, q));
            const ChunkDesc cd = a.chunks[chunk];
            const bool cached = cd.mode == kModeCached;
            const bool one = kFew && cd.op_count >= kOneEdgeOps;
            const int per = one ? kOneEdgeItem : 64;  // edges of an item
            const int* ids = slot_ptr<const int>(a, chunk, a.L.e_ids);
            float4* data = slot_ptr<float4>(a, chunk, a.L.e_data);
            const int* oid = reinterpret_cast<const int*>(cd.old_ids);
            const float4* odata = reinterpret_cast<const float4*>(cd.old_data);
            WaveOps list(a, cd);
            const int i = per * j + lane;
            const bool in = lane < per && i < edges;
            const int id = in ? ids[i] : 0;
            EdgeAt e;
            const bool live = decode_edge(G, id, e) && in;
            if (in && !live) atomicOr(&a.counters[chunk].status, kStatusLookupMiss);
            const bool touched = live && edge_touched(a, chunk, cd, e.i0, e.i1);
            uint64_t left = __ballot(touched);
            if (kFew && left && one) {
                float4 out = make_float4(0.f, 0.f, 0.f, 0.f);
                while (left) {
                    const int b = (int)__builtin_ctzll(left);
                    left &= left - 1;
                    EdgeAt at;
                    decode_edge(G, __builtin_amdgcn_readlane(id, b), at);
                    const float4 v = brush_crossing_one(list, cd, at.x, at.y, at.z, at.axis);
                    if (lane == b) out = v;
                }
                if (touched) data[i] = out;
            } else if (left) {
                const float4 out = brush_crossing(list, cd, touched, e.x, e.y, e.z, e.axis);
                if (touched) data[i] = out;
            }
            if (cached && live && !touched) {
                int lo = 0, hi = cd.old_edges;
                while (lo < hi) {
                    const int mid = (lo + hi) >> 1;
                    if (oid[mid] < id) lo = mid + 1; else hi = mid;
                }
                if (lo < cd.old_edges && oid[lo] == id) {
                    data[i] = odata[lo];
                } else {
                    data[i] = make_float4(0.f, 0.f, 0.f, 0.f);
                    atomicOr(&a.counters[chunk].status, kStatusLookupMiss);
                }
            }
            if constexpr (kCount) {
                if (touched) atomicAdd(&a.work[4], (unsigned long long)(17 * cd.op_count));
                if (touched || (cached && live)) atomicAdd(&a.work[6], 1ull);
            }
        }
        dealt = (dealt + total) % waves;
    }
}

// Persistent like k_density: waves pull 64-edge items of any chunk.  768-thread
// workgroups: at the kernel's register count (6 waves per SIMD) two of them fit a
// CU beside their two 64 KiB tables, where one 1024-thread workgroup would leave
// a third of the wave slots empty.
constexpr int kCrossThreads = 768;

template <bool kCount, int kKind>
__global__ __attribute__((amdgpu_waves_per_eu(6, 8))) __launch_bounds__(kCrossThreads) void k_edge_cross(KArgs a,
                                                                                                          int chunks) {
    __shared__ NoiseLds T;
    __shared__ int next_local;
    const int total = a.item_prefix[chunks];
    if ((int)blockIdx.x >= total) return;  // no wave of this workgroup has an item
    if (threadIdx.x == 0) next_local = 0;
    load_noise_tables(T, a.perm, a.grads);  // ends with a barrier
    const int lane = threadIdx.x & 63;
    // Cave items cost several times more underground than above, so they come from the one
    // global queue (sharing within workgroups measured slower: clipmap 93.2 -> 94.5 ms), in
    // grabs that shrink as the work runs out: half a wave's share of what is left when the
    // wave last looked, from 16 items down to 1.  Without the cave term items are short
    // and alike, and 82,000 of them through a counter that serves 77 grabs per us were the
    // whole of the kernel's time (0.92 ms on the reference's clipmap, its waves waiting 78%
    // of it): there each workgroup owns every gridDim-th block of items (of 8 once its
    // waves have 8 each, so that neighbours share a chunk's lines) and its waves share them
    // through an LDS counter.
    constexpr bool kQueue = kKind == LVN_FIELD_TERRAIN_CAVES || kKind == kAnyField;
    const int block_log = total >= 96 * (int)gridDim.x ? 3 : 0;
    const int waves = grid_waves();
    auto share = [&](int from) { return min(16, max(1, (total - from) / (2 * waves))); };
    const int given = share(0) * waves;  // the waves' first grabs
    int item, end = 0;
    auto local_item = [&]() {
        int j = 0;
        if (lane == 0) j = atomicAdd(&next_local, 1);
        j = __builtin_amdgcn_readfirstlane(j);
        const long at = ((((long)(j >> block_log) * gridDim.x) + blockIdx.x) << block_log) + (j & ((1 << block_log) - 1));
        return at < total ? (int)at : total;
    };
    auto next_of = [&](int cur) {  // the wave's item after `cur`, or total
        if constexpr (!kQueue) return local_item();
        if (cur + 1 < end) return cur + 1;
        if (given >= total) return total;
        const int n = share(cur);
        int at = 0;
        if (lane == 0) at = atomicAdd(&a.queue[1], n);
        at = given + __builtin_amdgcn_readfirstlane(at);
        end = min(at + n, total);
        return min(at, total);
    };
    if constexpr (kQueue) {
        item = first_grab(share(0));
        end = min(item + share(0), total);
    } else {
        item = local_item();
    }
    if (item >= total) return;
    int chunk = chunk_of_item(a.item_prefix, chunks, item);
    int2 o = edge_of_item(a, chunk, item - a.item_prefix[chunk], lane, 64);
    for (;;) {
        // the next item's edges are on their way while this one's are crossed
        const int next = next_of(item);
        int next_chunk = chunk;
        int2 o_next = make_int2(-1, 0);
        if (next < total) {
            if (next < item || a.item_prefix[chunk + 1] <= next) next_chunk = chunk_of_item(a.item_prefix, chunks, next);
            o_next = edge_of_item(a, next_chunk, next - a.item_prefix[next_chunk], lane, 64);
        }
        if (o.x >= 0) cross_edge<kCount, kKind>(a, T, chunk, o.x, o.y);
        if (next >= total) break;
        item = next;
        chunk = next_chunk;
        o = o_next;
    }
}

// Small batches: kG lanes share one edge, so a chunk's few hundred edge items become
// kG times as many waves with kG times shorter dependency chains.  Lane `sub`
// evaluates samples k = sub, sub + kG, ... of the 17; the group reduces to the first
// arg-min (smallest |d|, then smallest k, as the sequential scan decides), then the
// six normal samples are spread over the group.  Every value is computed by the
// same expression as in density_crossing, so results are identical.
template <bool kCount, int kKind, int kG>
__device__ __forceinline__ void cross_edge_group(const KArgs& a, const NoiseLds& T, int chunk, int i, int id,
                                                 int sub) {
    const Geometry& G = a.G;
    const ChunkDesc& cd = a.chunks[chunk];
    EdgeAt e;
    if (!decode_edge(G, id, e)) {
        if (sub == 0) atomicOr(&a.counters[chunk].status, kStatusLookupMiss);
        return;
    }
    const int x = e.x, y = e.y, z = e.z, axis = e.axis, i0 = e.i0, i1 = e.i1;
    if (edge_touched(a, chunk, cd, i0, i1)) return;  // k_edge_data's
    const FieldParams& Fp = a.F;
    const bool caves = field_kind<kKind>(Fp) == LVN_FIELD_TERRAIN_CAVES;
    const bool ends = !a.fp16;
    const float2 de = ends ? edge_ends(a, chunk, cd, x, y, z, axis, i0, i1) : make_float2(0.f, 0.f);
    const float d_start = de.x, d_end = de.y;
    const int w0x = x * cd.scale + cd.off[0], w0y = y * cd.scale + cd.off[1], w0z = z * cd.scale + cd.off[2];
    const float p0x = (float)w0x, p0y = (float)w0y, p0z = (float)w0z;
    const float p1x = (float)(w0x + (axis == 0 ? cd.scale : 0));
    const float p1y = (float)(w0y + (axis == 1 ? cd.scale : 0));
    const float p1z = (float)(w0z + (axis == 2 ? cd.scale : 0));
    unsigned nh = 0, nc = 0;
    const float colH = axis == 1 ? slot_ptr<const float>(a, chunk, a.L.h_cols)[x + G.F * z] : 0.f;
    const float* hl = slot_ptr<const float>(a, chunk, a.L.h_lines) + hline_index(G.H, axis == 2 ? 1 : 0, x, z);
    float minV = 3.402823466e+38f, Hbest = colH;
    int kbest = 17;
    const int k_first = sub == 0 ? kG : sub;  // this lane's first interior sample
    const bool lines = a.height_lines != 0 && axis != 1;
    float Hn = (lines && k_first <= kLineSamples) ? hl[k_first - 1] : 0.f;
    for (int k = sub; k <= 16; k += kG) {
        const float cur = (float)k * 0.0625f;  // = the sequential scan's running sum (exact)
        const float px = p0x + (p1x - p0x) * cur;
        const float py = p0y + (p1y - p0y) * cur;
        const float pz = p0z + (p1z - p0z) * cur;
        float d, H = colH;
        if (ends && k == 0) {
            d = fabsf(d_start);
        } else if (ends && k == 16) {
            d = fabsf(d_end);
        } else {
            if (axis != 1) {
                if (lines && k >= 1 && k <= kLineSamples) {
                    H = Hn;
                    if (k + kG <= kLineSamples) Hn = hl[k + kG - 1];
                } else {
                    H = height_term<kKind>(Fp, T, px, pz);
                    ++nh;
                }
            }
            nc += (caves && !((py - H) > Fp.cave_cut)) ? 1u : 0u;
            d = fabsf(combine<kKind>(Fp, T, py - H, px, py, pz));
        }
        if (d < minV) {
            minV = d;
            kbest = k;
            Hbest = H;
        }
    }
#pragma unroll
    for (int m = 1; m < kG; m <<= 1) {
        const float ov = __shfl_xor(minV, m, kG);
        const int ok = __shfl_xor(kbest, m, kG);
        const float oh = __shfl_xor(Hbest, m, kG);
        if (ov < minV || (ov == minV && ok < kbest)) {
            minV = ov;
            kbest = ok;
            Hbest = oh;
        }
    }
    const float tbest = (float)kbest * 0.0625f;
    const float px = p0x + (p1x - p0x) * tbest;
    const float py = p0y + (p1y - p0y) * tbest;
    const float pz = p0z + (p1z - p0z) * tbest;
    const float h = 0.001f;
    const bool hb_known = axis == 1 || !(ends && (kbest == 0 || kbest == 16));
    constexpr int kR = (6 + kG - 1) / kG;
    float vals[kR];
#pragma unroll
    for (int r = 0; r < kR; ++r) vals[r] = 0.f;
#pragma unroll 1
    for (int r = 0; r < kR; ++r) {  // one copy of the field's code
        const int j = r * kG + sub;  // normal sample j: +x, -x, +y, -y, +z, -z
        if (j >= 6) continue;
        const float sx = j == 0 ? h : j == 1 ? -h : 0.f;
        const float sz = j == 4 ? h : j == 5 ? -h : 0.f;
        const float qx = j < 2 ? px + sx : px;
        const float qy = j == 2 ? py + h : j == 3 ? py - h : py;
        const float qz = j >= 4 ? pz + sz : pz;
        float H = Hbest;  // the two samples above and below lie in the arg-min sample's column
        if (!(hb_known && (j == 2 || j == 3))) {
            H = height_term<kKind>(Fp, T, qx, qz);
            nh += j == 3 ? 0u : 1u;
        }
        const float aa = qy - H;
        nc += (caves && !(aa > Fp.cave_cut)) ? 1u : 0u;
        const float val = combine<kKind>(Fp, T, aa, qx, qy, qz);
#pragma unroll
        for (int q = 0; q < kR; ++q) vals[q] = q == r ? val : vals[q];
    }
    float v[6];
#pragma unroll
    for (int j = 0; j < 6; ++j) v[j] = __shfl(vals[j / kG], j % kG, kG);
    const float3 n = normalize_or_zero(v[0] - v[1], v[2] - v[3], v[4] - v[5]);
    if constexpr (kCount) {
        atomicAdd(&a.work[2], (unsigned long long)nh);
        atomicAdd(&a.work[3], (unsigned long long)nc);
        if (sub == 0) atomicAdd(&a.work[6], 1ull);
    }
    if (sub == 0) slot_ptr<float4>(a, chunk, a.L.e_data)[i] = make_float4(n.x, n.y, n.z, tbest);
}

template <bool kCount, int kKind, int kG>
__global__ __attribute__((amdgpu_waves_per_eu(6, 8))) __launch_bounds__(kCrossThreads) void k_edge_cross_group(
    KArgs a, int chunks) {
    __shared__ NoiseLds T;
    __shared__ int next_local;
    constexpr int kPerItem = 64 / kG;
    const int total = a.item_prefix[chunks];
    if ((int)blockIdx.x >= total) return;  // no wave of this workgroup has an item
    if (threadIdx.x == 0) next_local = 0;
    load_noise_tables(T, a.perm, a.grads);  // ends with a barrier
    const int lane = threadIdx.x & 63;
    for (int item = wg_next_item(&next_local, total); item >= 0; item = wg_next_item(&next_local, total)) {
        const int lo = chunk_of_item(a.item_prefix, chunks, item);
        const int2 o = edge_of_item(a, lo, item - a.item_prefix[lo], lane / kG, kPerItem);
        if (o.x >= 0) cross_edge_group<kCount, kKind, kG>(a, T, lo, o.x, o.y, lane & (kG - 1));
    }
}

// Sample-parallel search.  Lanes of different edges evaluate points a voxel or more
// apart (32 voxels in a coarse chunk), so their noise-table reads hit unrelated LDS
// addresses and conflict; lanes of one edge evaluate points a fraction of a voxel apart
// and mostly read the same table entries.  A wave takes a 64-edge item: each lane first
// loads its own edge (edges with brush data are k_edge_data's); the search then runs four edges at a time, 16 lanes each
// (lane s evaluates interior sample s + 1, lane 15 the end samples, read from the stored
// field when it is FP32), reduced over the row to the first arg-min (smallest |d|, then
// smallest k: the sequential scan's rule); finally each lane computes its own edge's
// normal from the search's result (crossing_normal).  Every value comes from the same
// expression as in density_crossing, so results are identical.  A y-edge's height term is
// its column's, stored by the density pass.
constexpr int kSpWaves = kCrossThreads / 64;

// v from the lane kN places further round its row of 16 (DPP row_ror).
template <int kN>
__device__ __forceinline__ int row_ror(int v) {
    return __builtin_amdgcn_update_dpp(v, v, 0x120 + kN, 0xf, 0xf, false);
}

// One step of the row's arg-min: keep the smaller (|d| bits, k) pair and its height.
template <int kN>
__device__ __forceinline__ void argmin_step(uint32_t& d, int& k, float& H) {
    const uint32_t od = (uint32_t)row_ror<kN>((int)d);
    const int ok = row_ror<kN>(k);
    const float oh = __int_as_float(row_ror<kN>(__float_as_int(H)));
    const bool take = od < d || (od == d && ok < k);
    d = take ? od : d;
    k = take ? ok : k;
    H = take ? oh : H;
}

template <bool kCount, int kKind>
__global__ __attribute__((amdgpu_waves_per_eu(6, 8))) __launch_bounds__(kCrossThreads) void k_edge_cross_sp(KArgs a,
                                                                                                             int chunks) {
    __shared__ NoiseLds T;
    __shared__ int next_local;
    __shared__ int sp_k[kSpWaves][64];    // per wave: kbest of each edge of the item
    __shared__ float sp_h[kSpWaves][64];  // and the height term there
    const int total = a.item_prefix[chunks];
    if ((int)blockIdx.x >= total) return;  // no wave of this workgroup has an item
    if (threadIdx.x == 0) next_local = 0;
    load_noise_tables(T, a.perm, a.grads);  // ends with a barrier
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int row = lane >> 4, sub = lane & 15;
    const FieldParams& Fp = a.F;
    const bool caves = field_kind<kKind>(Fp) == LVN_FIELD_TERRAIN_CAVES;
    const bool ends = !a.fp16;
    const Geometry& G = a.G;
    unsigned nh = 0, nc = 0, ne = 0;
    for (int item = wg_next_item(&next_local, total); item >= 0; item = wg_next_item(&next_local, total)) {
        const int lo = chunk_of_item(a.item_prefix, chunks, item);
        const int chunk = lo;
        const ChunkDesc& cd = a.chunks[chunk];
        // ---- each lane loads its own edge
        const int2 o = edge_of_item(a, chunk, item - a.item_prefix[chunk], lane, 64);
        int ei = o.x;
        int exyz = 0;
        float eH = 0.f, eS = 0.f, eE = 0.f;
        if (ei >= 0) {
            EdgeAt e;
            if (!decode_edge(G, o.y, e)) {
                atomicOr(&a.counters[chunk].status, kStatusLookupMiss);
                ei = -1;
            } else if (edge_touched(a, chunk, cd, e.i0, e.i1)) {  // k_edge_data's
                ei = -1;
            } else {
                exyz = e.x | (e.y << 8) | (e.z << 16) | (e.axis << 24);
                eH = e.axis == 1 ? slot_ptr<const float>(a, chunk, a.L.h_cols)[e.x + G.F * e.z] : 0.f;
                if (ends) {
                    const float2 de = edge_ends(a, chunk, cd, e.x, e.y, e.z, e.axis, e.i0, e.i1);
                    eS = de.x;
                    eE = de.y;
                }
            }
        }
        // ---- search: four edges at a time, 16 lanes each
        for (int r = 0; r < 16; ++r) {
            const int src = 4 * r + row;
            // every lane takes part in the shuffles: a lane of a row that skips the round
            // may be the source of another row's edge
            const int i = __shfl(ei, src);
            const int xyz = __shfl(exyz, src);
            const float colH = __shfl(eH, src);
            const float dS = __shfl(eS, src), dE = __shfl(eE, src);
            if (i < 0) continue;  // uniform over the row
            const int x = xyz & 255, y = (xyz >> 8) & 255, z = (xyz >> 16) & 255, axis = xyz >> 24;
            const int w0x = x * cd.scale + cd.off[0], w0y = y * cd.scale + cd.off[1], w0z = z * cd.scale + cd.off[2];
            const float p0x = (float)w0x, p0y = (float)w0y, p0z = (float)w0z;
            const float p1x = (float)(w0x + (axis == 0 ? cd.scale : 0));
            const float p1y = (float)(w0y + (axis == 1 ? cd.scale : 0));
            const float p1z = (float)(w0z + (axis == 2 ? cd.scale : 0));
            const bool lines = a.height_lines != 0 && axis != 1;
            // the lane's candidate: (|d| bits, k, H); none = (FLT_MAX, 17, colH)
            uint32_t md = 0x7f7fffffu;
            int mk = 17;
            float mh = colH;
            const int nk = sub < 15 ? 1 : 2;
            for (int q = 0; q < nk; ++q) {
                const int k = sub < 15 ? sub + 1 : 16 * q;
                const float cur = (float)k * 0.0625f;  // = the sequential scan's running sum (exact)
                float d, H = colH;
                if (ends && k == 0) {
                    d = fabsf(dS);
                } else if (ends && k == 16) {
                    d = fabsf(dE);
                } else {
                    const float px = p0x + (p1x - p0x) * cur;
                    const float py = p0y + (p1y - p0y) * cur;
                    const float pz = p0z + (p1z - p0z) * cur;
                    if (axis != 1) {
                        if (lines && k >= 1 && k <= kLineSamples) {
                            H = slot_ptr<const float>(a, chunk, a.L.h_lines)[hline_index(G.H, axis == 2 ? 1 : 0, x, z) +
                                                                             (k - 1)];
                        } else {
                            H = height_term<kKind>(Fp, T, px, pz);
                            ++nh;
                        }
                    }
                    nc += (caves && !((py - H) > Fp.cave_cut)) ? 1u : 0u;
                    d = fabsf(combine<kKind>(Fp, T, py - H, px, py, pz));
                }
                // the scan takes a sample only when |d| < its running minimum (from FLT_MAX):
                // lane 15 tries sample 0 before sample 16
                if (d < __uint_as_float(md)) {
                    md = __float_as_uint(d);
                    mk = k;
                    mh = H;
                }
            }
            // |d| >= 0, so its bits order like its values
            argmin_step<1>(md, mk, mh);
            argmin_step<2>(md, mk, mh);
            argmin_step<4>(md, mk, mh);
            argmin_step<8>(md, mk, mh);
            if (sub == 0) {
                sp_k[wave][src] = mk == 17 ? 0 : mk;  // no sample taken: the scan keeps t = 0
                sp_h[wave][src] = mh;
            }
        }
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        // ---- normal: each lane its own edge
        if (ei >= 0) {
            const int kb = sp_k[wave][lane];
            const float hb = sp_h[wave][lane];
            const int x = exyz & 255, y = (exyz >> 8) & 255, z = (exyz >> 16) & 255, axis = exyz >> 24;
            const int w0x = x * cd.scale + cd.off[0], w0y = y * cd.scale + cd.off[1], w0z = z * cd.scale + cd.off[2];
            const float p1x = (float)(w0x + (axis == 0 ? cd.scale : 0));
            const float p1y = (float)(w0y + (axis == 1 ? cd.scale : 0));
            const float p1z = (float)(w0z + (axis == 2 ? cd.scale : 0));
            slot_ptr<float4>(a, chunk, a.L.e_data)[ei] =
                crossing_normal<kKind>(Fp, T, axis, ends, (float)kb * 0.0625f, hb, (float)w0x, (float)w0y, (float)w0z, p1x, p1y,
                                p1z, nh, nc);
            ++ne;
        }
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    }
    if constexpr (kCount) {
        atomicAdd(&a.work[2], (unsigned long long)nh);
        atomicAdd(&a.work[3], (unsigned long long)nc);
        atomicAdd(&a.work[6], (unsigned long long)ne);
    }
}

// ---------------------------------------------------------------------------
// Active voxels (FindActiveVoxels + CompactVoxels, cl/octree.cl:142-223)
// ---------------------------------------------------------------------------

__device__ __forceinline__ int corner_materials(const KArgs& a, const uint8_t* mat, int x, int y, int z, int* cm) {
    const Geometry& G = a.G;
    int corners = 0;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        cm[i] = mat[field_index(G, x + ((i >> 2) & 1), y + ((i >> 1) & 1), z + (i & 1))];
        corners |= (cm[i] == kAir ? 0 : 1) << i;
    }
    return corners;
}

// The corners' solid bits from the solid rows, for a chunk that stores no materials: a
// sample's material is then the default material where it is not air (density < 0) and air
// elsewhere.  Two neighbouring bits of each of the voxel's four rows.
__device__ __forceinline__ int corners_from_rows(const KArgs& a, const uint64_t* S, int x, int y, int z) {
    int corners = 0;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const int jy = j & 1, jz = j >> 1;
        const ulonglong2 w = *reinterpret_cast<const ulonglong2*>(S + 2 * ((y + jy) + a.G.F * (z + jz)));
        const int t = (int)(uint32_t)(w.x >> x) | (x == 63 ? (int)((uint32_t)w.y << 1) : 0);
        corners |= (t & 1) << (2 * jy + jz) | ((t >> 1) & 1) << (4 + 2 * jy + jz);
    }
    return corners;
}

// The edges with a sign change, bit e for the corners kEdgeMap[e].
__device__ __forceinline__ int edges_of_corners(int corners) {
    const int x = corners ^ (corners >> 4), y = corners ^ (corners >> 2), z = corners ^ (corners >> 1);
    return (x & 15) | ((y & 3) | ((y >> 2) & 12)) << 4 |
           ((z & 1) | ((z >> 1) & 2) | ((z >> 2) & 4) | ((z >> 3) & 8)) << 8;
}

// FindDominantMaterial, cl/octree.cl:78-138.  The reference sorts the eight corner
// materials by insertion; any correct sort yields the same sequence, and Batcher's
// odd-even merge network (19 compare-exchanges, min/max pairs) does it without the
// insertion sort's data-dependent loops, which diverge across a wave.
__device__ __forceinline__ void sort_exchange(int& a, int& b) {
    const int lo = min(a, b), hi = max(a, b);
    a = lo;
    b = hi;
}

__device__ __forceinline__ int dominant_material(const int* m) {
    int d[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) d[i] = m[i];
    sort_exchange(d[0], d[1]); sort_exchange(d[2], d[3]); sort_exchange(d[4], d[5]); sort_exchange(d[6], d[7]);
    sort_exchange(d[0], d[2]); sort_exchange(d[1], d[3]); sort_exchange(d[4], d[6]); sort_exchange(d[5], d[7]);
    sort_exchange(d[1], d[2]); sort_exchange(d[5], d[6]);
    sort_exchange(d[0], d[4]); sort_exchange(d[1], d[5]); sort_exchange(d[2], d[6]); sort_exchange(d[3], d[7]);
    sort_exchange(d[2], d[4]); sort_exchange(d[3], d[5]);
    sort_exchange(d[1], d[2]); sort_exchange(d[3], d[4]); sort_exchange(d[5], d[6]);
    int current = d[0], count = 1, maxCount = 0, maxMaterial = 0;
#pragma unroll
    for (int i = 1; i < 8; ++i) {
        const int v = d[i];
        if (v == kAir || v == kNone) continue;
        if (current != v) {
            if (count > maxCount) {
                maxCount = count;
                maxMaterial = current;
            }
            current = v;
            count = 1;
        } else {
            ++count;
        }
    }
    if (count > maxCount) maxMaterial = current;
    return maxMaterial;
}

// The octree codes of every segment's active voxels in linear order; the corner
// materials, edge mask and dominant material are found by the QEF kernel, which reads
// the corners anyway.  A wave takes 64 consecutive segments and loads their masks and
// bases together (lane j: segment j).  Where its live segments are dense (kDenseRow
// voxels or more on average) it walks them in order with lane b holding the segment's
// voxel b: its rank is the popcount of the mask below b.  Where they are sparse, each lane
// takes one voxel of the wave's run of the list, found as the edges are.
__device__ __forceinline__ void voxel_compact(const KArgs& a, int chunk, int wave, int waves, int split) {
    const Geometry& G = a.G;
    const uint64_t* vmask = slot_ptr<const uint64_t>(a, chunk, a.L.v_mask);
    const int* vbase = slot_ptr<const int>(a, chunk, a.L.v_base);
    int* vcode = slot_ptr<int>(a, chunk, a.L.v_code);
    const int cap = a.caps.voxels;
    const int lane = threadIdx.x & 63;
    const uint64_t lt = lanemask_lt(lane);
    const int units = ((G.voxel_segs + 63) >> 6) * split;
    for (int u = wave; u < units; u += waves) {
        const int g = u / split, part = u - g * split;
        const int sl = (g << 6) + lane;
        const uint64_t ml = sl < G.voxel_segs ? vmask[sl] : 0;
        uint64_t live = __ballot(ml != 0);
        if (!live) continue;
        const int bl = sl < G.voxel_segs ? vbase[sl] : 0x7fffffff;
        const int total = wave_sum(__popcll(ml));
        if (total < kDenseRow * __popcll(live)) {  // sparse: one lane per voxel
            const int i_first = __builtin_amdgcn_readlane(bl, 0);
            for (int i0 = part << 6; i0 < total; i0 += split << 6) {
                const int i = i_first + min(i0 + lane, total - 1);
                const int j = last_lane_at(bl, i);
                int n = i - __shfl(bl, j);
                const uint32_t lo = (uint32_t)__shfl((int)(uint32_t)ml, j), hi = (uint32_t)__shfl((int)(uint32_t)(ml >> 32), j);
                const int c = __popc(lo);
                int b = n >= c ? 32 : 0;
                uint32_t m = n >= c ? hi : lo;
                n -= n >= c ? c : 0;
#pragma unroll
                for (int s = 16; s > 0; s >>= 1) {
                    const int below = __popc(m & ((1u << s) - 1)), up = n >= below ? s : 0;
                    n -= up ? below : 0;
                    b += up;
                    m >>= up;
                }
                int x, y, z;
                decode_voxel(G, (((g << 6) + j) << 6) + b, x, y, z);
                if (i0 + lane < total && i < cap) vcode[i] = (int)code_for_position(x, y, z, G.depth);
            }
            continue;
        }
        for (int skip = 0; live; ++skip) {
            const int j = (int)__builtin_ctzll(live);
            live &= live - 1ull;
            if (skip % split != part) continue;
            const int seg = (g << 6) + j;
            const uint64_t m = readlane64(ml, j);
            const int i = __builtin_amdgcn_readlane(bl, j) + __popcll(m & lt);
            if (((m >> lane) & 1ull) && i < cap) {
                int x, y, z;
                decode_voxel(G, (seg << 6) + lane, x, y, z);
                vcode[i] = (int)code_for_position(x, y, z, G.depth);
            }
        }
    }
}

// Edge lists by the first `edge_blocks` workgroups of a chunk, voxel codes by the others.
__global__ __launch_bounds__(256) void k_compact(KArgs a, int edge_blocks, int split) {
    __shared__ uint4 stage[4][64][2];  // a wave's 64 edge rows
    const int chunk = blockIdx.y;
    const Counters& c = a.counters[chunk];
    if ((int)blockIdx.x < edge_blocks) {
        if (c.edges) edge_compact(a, chunk, wave_in_chunk(), edge_blocks * 4, split, stage[threadIdx.x >> 6]);
    } else {
        if (c.voxels) voxel_compact(a, chunk, wave_in_chunk() - edge_blocks * 4, ((int)gridDim.x - edge_blocks) * 4, split);
    }
}

// ---------------------------------------------------------------------------
// QEF build + solve (CreateLeafNodes + SolveQEFs, cl/octree.cl:236-331,
// cl/qef.cl).  Edge data is found through the edge segment masks instead of a
// cuckoo hash (cl/cuckoo.cl:73-104).
// ---------------------------------------------------------------------------

struct Q4 {
    float x, y, z, w;
};

__device__ __forceinline__ float dot4(const Q4& a, const Q4& b) {
    return ((a.x * b.x + a.y * b.y) + a.z * b.z) + a.w * b.w;
}

// Both square roots have arguments >= 1 and the cosine's divisor lies in [1, sqrt 2]
// (|tn| <= 1), so they take the short correctly rounded forms; the other two
// divisions see any magnitude (tau overflows to inf for a tiny apq).
__device__ __forceinline__ void givens(float app, float apq, float aqq, float& c, float& s) {  // cl/qef.cl:31-42
    const float tau = (aqq - app) / (2.f * apq);
    const float stt = sqrt_ge1(1.f + tau * tau);
    const float tn = 1.f / ((tau >= 0.f) ? (tau + stt) : (tau - stt));
    c = recip_1_2(sqrt_ge1(1.f + tn * tn));
    s = tn * c;
}

// svd_rotate, cl/qef.cl:58-86, for the pair (A, B); U/W are the other two
// off-diagonal entries rotated with it (vtav[0][3-b], vtav[1-a][2]).
#define LVN_ROTATE(AA, BB, AB, U, W, VA0, VB0, VA1, VB1, VA2, VB2)                   \
    if (AB != 0.f) {                                                                   \
        float c, s;                                                                    \
        givens(AA, AB, BB, c, s);                                                      \
        const float cc = c * c, ss = s * s;                                            \
        const float mx = ((2.f * c) * s) * AB;                                         \
        const float u0 = AA, w0 = BB;                                                  \
        AA = (cc * u0 - mx) + ss * w0;                                                 \
        BB = (ss * u0 + mx) + cc * w0;                                                 \
        const float u1 = U, w1 = W;                                                    \
        U = c * u1 - s * w1;                                                           \
        W = s * u1 + c * w1;                                                           \
        AB = 0.f;                                                                      \
        float uu = VA0, ww = VB0;                                                      \
        VA0 = c * uu - s * ww;                                                         \
        VB0 = s * uu + c * ww;                                                         \
        uu = VA1; ww = VB1;                                                            \
        VA1 = c * uu - s * ww;                                                         \
        VB1 = s * uu + c * ww;                                                         \
        uu = VA2; ww = VB2;                                                            \
        VA2 = c * uu - s * ww;                                                         \
        VB2 = s * uu + c * ww;                                                         \
    }

__device__ __forceinline__ float invdet(float x) {  // svd_invdet, cl/qef.cl:107-109
    return (fabsf(x) < 0.1f || fabsf(1.f / x) < 0.1f) ? 0.f : 1.f / x;
}

// Edge e's bit in a voxel's presence word, 5 bits each: row j = y + 2 z and slot s = 3 x + axis
// of its lower end's corner.
constexpr uint64_t kSlotOfEdge = 0ull | 16ull << 5 | 8ull << 10 | 24ull << 15 |         // x edges
                                 1ull << 20 | 17ull << 25 | 4ull << 30 | 20ull << 35 |  // y edges
                                 2ull << 40 | 10ull << 45 | 5ull << 50 | 13ull << 55;   // z edges

__device__ __forceinline__ void qef_fast(const KArgs& a, int chunk, const ChunkDesc& cd, int3 p, int emask, float4& out,
                                         float4& nrm) {
    const Geometry& G = a.G;
    const uint64_t* erows = slot_ptr<const uint64_t>(a, chunk, a.L.e_rows);
    const int2* eb = slot_ptr<const int2>(a, chunk, a.L.e_base);
    const float4* ed = slot_ptr<float4>(a, chunk, a.L.e_data);
    const float fscale = (float)cd.scale;

    // The voxel's edges start at its corners, so they lie in four edge rows, (y or y + 1,
    // z or z + 1), at x and x + 1: row j's six possible edges are bits 8 j .. 8 j + 5 of
    // `have` in list order, and first[j] is the list index of the first of them.  Both are
    // meaningless for a row without edges, whose words are not written (edge_rows);
    // no edge of emask lies in one, since emask and the rows come from the same solid bits.
    uint32_t have = 0;
    int first[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const int r = (p.y + (j & 1)) + G.H * (p.z + (j >> 1));
        const uint64_t ex = erows[4 * r], ey = erows[4 * r + 1], ez = erows[4 * r + 2], hi = erows[4 * r + 3];
        const uint64_t lt = lanemask_lt(p.x);
        first[j] = eb[r].x + __popcll(ex & lt) + __popcll(ey & lt) + __popcll(ez & lt);
        const uint32_t bx = (uint32_t)(ex >> p.x), by = (uint32_t)(ey >> p.x), bz = (uint32_t)(ez >> p.x);
        uint32_t b = (bx & 1) | (by & 1) << 1 | (bz & 1) << 2 | (bx & 2) << 2 | (by & 2) << 3 | (bz & 2) << 4;
        if (p.x == 63) b |= ((uint32_t)hi & 7) << 3;
        have |= b << (8 * j);
    }
    // The edge's point is a0 + (a1 - a0) t per component (cl/octree.cl:266-272), scaled.  Its
    // end corners differ by exactly 1 along the edge's axis and by exactly 0 across it, and t
    // is a finite crossing in [0, 1], so (a1 - a0) t is t along the axis and +0 across it:
    // the across components are fscale * a0 (six per voxel, formed once) and the w lane is
    // +0, which leaves the dot product's fourth term +0 and makes the w sums count edges.
    const float fx = (float)p.x, fy = (float)p.y, fz = (float)p.z;
    const float sx0 = fscale * fx, sx1 = fscale * (float)(p.x + 1);
    const float sy0 = fscale * fy, sy1 = fscale * (float)(p.y + 1);
    const float sz0 = fscale * fz, sz1 = fscale * (float)(p.z + 1);
    float ata0 = 0.f, ata1 = 0.f, ata2 = 0.f, ata3 = 0.f, ata4 = 0.f, ata5 = 0.f;
    Q4 atb = {0.f, 0.f, 0.f, 0.f}, mass = {0.f, 0.f, 0.f, 0.f}, nsum = {0.f, 0.f, 0.f, 0.f};
    int count = 0;
    // Each lane walks its own edges in the order of e, the next one's data in flight: a wave
    // takes as many steps as its busiest voxel has edges (7 or 8 of the 12), where a step per
    // possible edge computed all twelve indices and waited for twelve loads in turn.  The
    // kernel is bound by vector issue (1,300 of about 2,060 instructions a segment are the
    // rotations below): 1,800 clipmap chunks 337 -> 297 us, 512 cave chunks 488 -> 461.
    uint32_t left = (uint32_t)emask;
    int slot = 0;
    bool used = false;
    float4 d = make_float4(0.f, 0.f, 0.f, 0.f);
    auto next = [&]() {  // the lowest edge left
        const int e = __builtin_ctz(left);
        left &= left - 1;
        slot = (int)(kSlotOfEdge >> (5 * e)) & 31;
        const int j = slot >> 3;
        const int row = j == 0 ? first[0] : j == 1 ? first[1] : j == 2 ? first[2] : first[3];
        const int k = row + __popc((have >> (8 * j)) & ((1u << (slot & 7)) - 1));
        used = ((have >> slot) & 1) && k >= 0 && k < a.caps.edges;
        if (used) d = ed[k];
    };
    bool more = left != 0;
    if (more) next();
    while (more) {
        const float4 c = d;
        const int at = slot;
        const bool take = used;
        more = left != 0;
        if (more) next();
        if (!take) continue;
        const int s = at & 7, axis = s >= 3 ? s - 3 : s;
        const float along = fscale * ((axis == 0 ? fx : axis == 1 ? fy : fz) + c.w);
        Q4 pos, n;
        pos.x = axis == 0 ? along : s >= 3 ? sx1 : sx0;
        pos.y = axis == 1 ? along : (at & 8) ? sy1 : sy0;
        pos.z = axis == 2 ? along : (at & 16) ? sz1 : sz0;
        n.x = c.x;
        n.y = c.y;
        n.z = c.z;
        // qef_add_point, cl/qef.cl:170-191
        ata0 = ata0 + n.x * n.x;
        ata1 = ata1 + n.x * n.y;
        ata2 = ata2 + n.x * n.z;
        ata3 = ata3 + n.y * n.y;
        ata4 = ata4 + n.y * n.z;
        ata5 = ata5 + n.z * n.z;
        const float b = (((pos.x * n.x + pos.y * n.y) + pos.z * n.z) + 0.f);
        atb.x = atb.x + n.x * b;
        atb.y = atb.y + n.y * b;
        atb.z = atb.z + n.z * b;
        mass.x = mass.x + pos.x;
        mass.y = mass.y + pos.y;
        mass.z = mass.z + pos.z;
        nsum.x = nsum.x + n.x;
        nsum.y = nsum.y + n.y;
        nsum.z = nsum.z + n.z;
        ++count;
    }
    mass.w = (float)count;  // the sums of 1 per edge
    nsum.w = (float)count;
    // qef_create_from_points tail (cl/qef.cl:302), then qef_solve's divide by max(w, 1) (:244).
    {
        const float w = mass.w;
        mass.x = mass.x / w;
        mass.y = mass.y / w;
        mass.z = mass.z / w;
        mass.w = mass.w / w;
        const float mw = fmaxf(mass.w, 1.f);
        mass.x = mass.x / mw;
        mass.y = mass.y / mw;
        mass.z = mass.z / mw;
        mass.w = mass.w / mw;
    }
    Q4 amp;
    {
        const Q4 row = {ata0, ata1, ata2, 0.f};
        amp.x = atb.x - dot4(row, mass);
        amp.y = atb.y - ((ata1 * mass.x + ata3 * mass.y) + ata4 * mass.z);
        amp.z = atb.z - ((ata2 * mass.x + ata4 * mass.y) + ata5 * mass.z);
        amp.w = atb.w - 0.f;
    }
    // svd_solve_sym, 10 cyclic sweeps (cl/qef.cl:88-105).
    float v00 = ata0, v01 = ata1, v02 = ata2, v11 = ata3, v12 = ata4, v22 = ata5;
    float V00 = 1.f, V01 = 0.f, V02 = 0.f, V10 = 0.f, V11 = 1.f, V12 = 0.f, V20 = 0.f, V21 = 0.f, V22 = 1.f;
    for (int sweep = 0; sweep < 10; ++sweep) {
        LVN_ROTATE(v00, v11, v01, v02, v12, V00, V01, V10, V11, V20, V21)
        LVN_ROTATE(v00, v22, v02, v01, v12, V00, V02, V10, V12, V20, V22)
        LVN_ROTATE(v11, v22, v12, v01, v02, V01, V02, V11, V12, V21, V22)
    }
    const float d0 = invdet(v00), d1 = invdet(v11), d2 = invdet(v22);
    const float Vm[3][3] = {{V00, V01, V02}, {V10, V11, V12}, {V20, V21, V22}};
    float x[3];
#pragma unroll
    for (int r = 0; r < 3; ++r) {
        Q4 row;
        row.x = ((Vm[r][0] * d0) * Vm[0][0] + (Vm[r][1] * d1) * Vm[0][1]) + (Vm[r][2] * d2) * Vm[0][2];
        row.y = ((Vm[r][0] * d0) * Vm[1][0] + (Vm[r][1] * d1) * Vm[1][1]) + (Vm[r][2] * d2) * Vm[1][2];
        row.z = ((Vm[r][0] * d0) * Vm[2][0] + (Vm[r][1] * d1) * Vm[2][1]) + (Vm[r][2] * d2) * Vm[2][2];
        row.w = 0.f;
        x[r] = dot4(row, amp);
    }
    out.x = ((x[0] + mass.x) * 4.f) + (float)cd.min[0];
    out.y = ((x[1] + mass.y) * 4.f) + (float)cd.min[1];
    out.z = ((x[2] + mass.z) * 4.f) + (float)cd.min[2];
    out.w = 1.f;
    const float nw = nsum.w;
    nrm = make_float4(nsum.x / nw, nsum.y / nw, nsum.z / nw, 0.f);
}

// ---------------------------------------------------------------------------
// Precision form of the QEF (LVN_CTX_PRECISE_QEF).  The normal equations are
// formed about the mass point, A = sum n n^T and r = sum n (n . (p - m)) (the
// same least-squares problem as ATb - ATA m, without its cancellation), with
// every product split exactly by an FMA (TwoProduct) and summed with Neumaier
// compensation.  The Jacobi pseudo-inverse runs in FP32; a vertex with an eigenvalue
// within kThresholdWindow |A|_F of the truncation thresholds 0.1 and 10 is re-solved
// entirely in FP64.
// ---------------------------------------------------------------------------

__device__ __forceinline__ void neumaier(float& s, float& c, float x) {
    const float t = s + x;
    c += fabsf(s) >= fabsf(x) ? (s - t) + x : (x - t) + s;
    s = t;
}

__device__ __forceinline__ void add_product(float& s, float& c, float a, float b) {
    const float p = a * b;
    const float e = fmaf(a, b, -p);  // exact error of the product
    neumaier(s, c, p);
    c += e;
}

template <typename T>
__device__ __forceinline__ void jacobi_rotate(T& aa, T& bb, T& ab, T& u, T& w, T& va0, T& vb0, T& va1, T& vb1, T& va2,
                                              T& vb2) {
    if (ab == (T)0) return;
    const T tau = (bb - aa) / ((T)2 * ab);
    const T stt = sqrt((T)1 + tau * tau);
    const T tn = (T)1 / ((tau >= (T)0) ? (tau + stt) : (tau - stt));
    const T c = (T)1 / sqrt((T)1 + tn * tn);
    const T s = tn * c;
    const T cc = c * c, ss = s * s, mx = (((T)2 * c) * s) * ab;
    const T u0 = aa, w0 = bb;
    aa = (cc * u0 - mx) + ss * w0;
    bb = (ss * u0 + mx) + cc * w0;
    const T u1 = u, w1 = w;
    u = c * u1 - s * w1;
    w = s * u1 + c * w1;
    ab = (T)0;
    T x = va0, y = vb0;
    va0 = c * x - s * y;
    vb0 = s * x + c * y;
    x = va1; y = vb1;
    va1 = c * x - s * y;
    vb1 = s * x + c * y;
    x = va2; y = vb2;
    va2 = c * x - s * y;
    vb2 = s * x + c * y;
}

// 10 cyclic Jacobi sweeps + truncated pseudo-inverse applied to r (cl/qef.cl:88-144).
template <typename T>
__device__ __forceinline__ void qef_pinv_solve(const T A[6], const T r[3], T x[3], T sig[3]) {
    T v00 = A[0], v01 = A[1], v02 = A[2], v11 = A[3], v12 = A[4], v22 = A[5];
    T V[3][3] = {{1, 0, 0}, {0, 1, 0}, {0, 0, 1}};
    for (int sweep = 0; sweep < 10; ++sweep) {
        jacobi_rotate<T>(v00, v11, v01, v02, v12, V[0][0], V[0][1], V[1][0], V[1][1], V[2][0], V[2][1]);
        jacobi_rotate<T>(v00, v22, v02, v01, v12, V[0][0], V[0][2], V[1][0], V[1][2], V[2][0], V[2][2]);
        jacobi_rotate<T>(v11, v22, v12, v01, v02, V[0][1], V[0][2], V[1][1], V[1][2], V[2][1], V[2][2]);
    }
    sig[0] = v00;
    sig[1] = v11;
    sig[2] = v22;
    const T tol = (T)0.1;
    T d[3];
#pragma unroll
    for (int i = 0; i < 3; ++i)
        d[i] = (fabs(sig[i]) < tol || fabs((T)1 / sig[i]) < tol) ? (T)0 : (T)1 / sig[i];
#pragma unroll
    for (int i = 0; i < 3; ++i) {
        T acc = 0;
#pragma unroll
        for (int j = 0; j < 3; ++j)
            acc += ((V[i][0] * d[0]) * V[j][0] + (V[i][1] * d[1]) * V[j][1] + (V[i][2] * d[2]) * V[j][2]) * r[j];
        x[i] = acc;
    }
}

// The truncated pseudo-inverse keeps eigenvalues in [0.1, 10] (svd_invdet, cl/qef.cl:107-109),
// so the retained ones have a condition number of at most 100 and FP32 solves them well;
// what FP32 can get wrong is which eigenvalues are retained.  FP32 Jacobi's eigenvalues
// are within a small multiple of eps * |A|_F of the exact ones (backward stable, about 30
// rotations here): an eigenvalue that close to 0.1 or 10 is re-solved in FP64.
constexpr float kThresholdWindow = 256.f * 5.9604645e-8f;  // 256 eps, times |A|_F

__device__ __forceinline__ bool near_threshold(float s, float w) {
    const float a = fabsf(s);
    return fabsf(a - 0.1f) <= w || fabsf(a - 10.f) <= w;
}

// qef_fast's walk of a voxel's edges, for more than one pass: the precision form walks them
// twice instead of keeping twelve points and normals, 104 registers instead of 188 and four
// waves per SIMD instead of two: 64 chunks 168 -> 121 us.  (qef_fast keeps its own loop: by
// this one a lone chunk's 11 us became 18.)  As there, `have` and `first` of a row without edges
// are meaningless, and no edge of emask lies in one.
struct EdgeWalk {
    uint32_t have;
    int first[4];
    float sx0, sx1, sy0, sy1, sz0, sz1, fx, fy, fz, fscale;

    __device__ __forceinline__ EdgeWalk(const KArgs& a, int chunk, int3 p, float scale) : have(0), fscale(scale) {
        const Geometry& G = a.G;
        const uint64_t* erows = slot_ptr<const uint64_t>(a, chunk, a.L.e_rows);
        const int2* eb = slot_ptr<const int2>(a, chunk, a.L.e_base);
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int r = (p.y + (j & 1)) + G.H * (p.z + (j >> 1));
            const uint64_t ex = erows[4 * r], ey = erows[4 * r + 1], ez = erows[4 * r + 2], hi = erows[4 * r + 3];
            const uint64_t lt = lanemask_lt(p.x);
            first[j] = eb[r].x + __popcll(ex & lt) + __popcll(ey & lt) + __popcll(ez & lt);
            const uint32_t bx = (uint32_t)(ex >> p.x), by = (uint32_t)(ey >> p.x), bz = (uint32_t)(ez >> p.x);
            uint32_t b = (bx & 1) | (by & 1) << 1 | (bz & 1) << 2 | (bx & 2) << 2 | (by & 2) << 3 | (bz & 2) << 4;
            if (p.x == 63) b |= ((uint32_t)hi & 7) << 3;
            have |= b << (8 * j);
        }
        fx = (float)p.x, fy = (float)p.y, fz = (float)p.z;
        sx0 = fscale * fx, sx1 = fscale * (float)(p.x + 1);
        sy0 = fscale * fy, sy1 = fscale * (float)(p.y + 1);
        sz0 = fscale * fz, sz1 = fscale * (float)(p.z + 1);
    }
    // f(point, normal) for each edge of emask with hermite data.
    template <class F>
    __device__ __forceinline__ void each(const KArgs& a, const float4* ed, int emask, F f) const {
        uint32_t left = (uint32_t)emask;
        int slot = 0;
        bool used = false;
        float4 d = make_float4(0.f, 0.f, 0.f, 0.f);
        auto next = [&]() {  // the lowest edge left
            const int e = __builtin_ctz(left);
            left &= left - 1;
            slot = (int)(kSlotOfEdge >> (5 * e)) & 31;
            const int j = slot >> 3;
            const int row = j == 0 ? first[0] : j == 1 ? first[1] : j == 2 ? first[2] : first[3];
            const int k = row + __popc((have >> (8 * j)) & ((1u << (slot & 7)) - 1));
            used = ((have >> slot) & 1) && k >= 0 && k < a.caps.edges;
            if (used) d = ed[k];
        };
        bool more = left != 0;
        if (more) next();
        while (more) {
            const float4 c = d;
            const int at = slot;
            const bool take = used;
            more = left != 0;
            if (more) next();
            if (!take) continue;
            const int s = at & 7, axis = s >= 3 ? s - 3 : s;
            const float along = fscale * ((axis == 0 ? fx : axis == 1 ? fy : fz) + c.w);
            const float3 pos = make_float3(axis == 0 ? along : s >= 3 ? sx1 : sx0, axis == 1 ? along : (at & 8) ? sy1 : sy0,
                                           axis == 2 ? along : (at & 16) ? sz1 : sz0);
            f(pos, make_float3(c.x, c.y, c.z));
        }
    }
};

__device__ __forceinline__ void qef_precise(const KArgs& a, int chunk, const ChunkDesc& cd, int3 p, int emask, float4& out,
                                            float4& nrm) {
    const float4* ed = slot_ptr<const float4>(a, chunk, a.L.e_data);
    const EdgeWalk walk(a, chunk, p, (float)cd.scale);
    float cnt = 0.f;
    float sx = 0.f, cx = 0.f, sy = 0.f, cy = 0.f, sz = 0.f, cz = 0.f;
    float nsx = 0.f, nsy = 0.f, nsz = 0.f;
    walk.each(a, ed, emask, [&](float3 q, float3 n) {
        cnt += 1.f;
        neumaier(sx, cx, q.x);
        neumaier(sy, cy, q.y);
        neumaier(sz, cz, q.z);
        nsx = nsx + n.x;
        nsy = nsy + n.y;
        nsz = nsz + n.z;
    });
    const float mx = (sx + cx) / cnt, my = (sy + cy) / cnt, mz = (sz + cz) / cnt;
    float As[6] = {0, 0, 0, 0, 0, 0}, Ac[6] = {0, 0, 0, 0, 0, 0}, rs[3] = {0, 0, 0}, rc[3] = {0, 0, 0};
    walk.each(a, ed, emask, [&](float3 q, float3 n) {
        add_product(As[0], Ac[0], n.x, n.x);
        add_product(As[1], Ac[1], n.x, n.y);
        add_product(As[2], Ac[2], n.x, n.z);
        add_product(As[3], Ac[3], n.y, n.y);
        add_product(As[4], Ac[4], n.y, n.z);
        add_product(As[5], Ac[5], n.z, n.z);
        const float b = fmaf(n.x, q.x - mx, fmaf(n.y, q.y - my, n.z * (q.z - mz)));
        add_product(rs[0], rc[0], n.x, b);
        add_product(rs[1], rc[1], n.y, b);
        add_product(rs[2], rc[2], n.z, b);
    });
    float A[6], r[3], x[3], sig[3];
#pragma unroll
    for (int i = 0; i < 6; ++i) A[i] = As[i] + Ac[i];
#pragma unroll
    for (int i = 0; i < 3; ++i) r[i] = rs[i] + rc[i];
    qef_pinv_solve<float>(A, r, x, sig);
    const float normf = sqrtf((A[0] * A[0] + A[3] * A[3] + A[5] * A[5]) + 2.f * (A[1] * A[1] + A[2] * A[2] + A[4] * A[4]));
    const float w = kThresholdWindow * normf;
    if (near_threshold(sig[0], w) || near_threshold(sig[1], w) || near_threshold(sig[2], w)) {
        double n = 0, mxd = 0, myd = 0, mzd = 0;
        walk.each(a, ed, emask, [&](float3 q, float3) {
            n += 1.0;
            mxd += (double)q.x;
            myd += (double)q.y;
            mzd += (double)q.z;
        });
        mxd /= n;
        myd /= n;
        mzd /= n;
        double Ad[6] = {0, 0, 0, 0, 0, 0}, rd[3] = {0, 0, 0}, xd[3], sd[3];
        walk.each(a, ed, emask, [&](float3 q, float3 v) {
            const double a0 = v.x, a1 = v.y, a2 = v.z;
            Ad[0] += a0 * a0;
            Ad[1] += a0 * a1;
            Ad[2] += a0 * a2;
            Ad[3] += a1 * a1;
            Ad[4] += a1 * a2;
            Ad[5] += a2 * a2;
            const double b = a0 * ((double)q.x - mxd) + a1 * ((double)q.y - myd) + a2 * ((double)q.z - mzd);
            rd[0] += a0 * b;
            rd[1] += a1 * b;
            rd[2] += a2 * b;
        });
        qef_pinv_solve<double>(Ad, rd, xd, sd);
        out = make_float4((float)((xd[0] + mxd) * 4.0 + (double)cd.min[0]),
                          (float)((xd[1] + myd) * 4.0 + (double)cd.min[1]),
                          (float)((xd[2] + mzd) * 4.0 + (double)cd.min[2]), 1.f);
        atomicAdd(&a.counters[chunk].resolved, 1);
    } else {
        out = make_float4(((x[0] + mx) * 4.f) + (float)cd.min[0], ((x[1] + my) * 4.f) + (float)cd.min[1],
                          ((x[2] + mz) * 4.f) + (float)cd.min[2], 1.f);
    }
    // the vertex normal is the reference's unnormalised mean of the edge normals
    const float nw = cnt;
    nrm = make_float4(nsx / nw, nsy / nw, nsz / nw, 0.f);
}

// ---------------------------------------------------------------------------
// Per active voxel, one pass: corner materials and edge mask (CreateLeafNodes,
// cl/octree.cl:236-283), dominant material (cl/octree.cl:78-138), the QEF vertex
// written straight into the vertex buffer (GenerateMeshVertexBuffer,
// cl/octree.cl:475-496), the voxel's quad flags (GenerateMesh, cl/octree.cl:398-439)
// and seam flag (FindSeamNodes, cl/octree.cl:500-518).  Per 64-voxel segment the
// quad count and the seam mask go to the quad and seam scans.
// ---------------------------------------------------------------------------

__device__ __forceinline__ int quad_flag(const Geometry& G, int3 p, int emask, int axis) {
    const int pa = axis == 0 ? p.y : axis == 1 ? p.z : p.x;
    const int pb = axis == 0 ? p.z : axis == 1 ? p.x : p.y;
    if (pa == G.N - 1 || pb == G.N - 1) return 0;  // isEdgeVoxel, cl/octree.cl:411-417
    return (emask >> (axis * 4 + 3)) & 1;
}

template <bool kPrecise>
__global__ __launch_bounds__(256) void k_qef(KArgs a) {
    const int chunk = blockIdx.y;
    const Geometry& G = a.G;
    const int V = a.counters[chunk].voxels;
    const ChunkDesc cd = a.chunks[chunk];
    const int* vcode = slot_ptr<const int>(a, chunk, a.L.v_code);
    const uint8_t* mat = slot_ptr<const uint8_t>(a, chunk, a.L.mat);
    const uint64_t* S = slot_ptr<const uint64_t>(a, chunk, a.L.solid);
    const bool rows = chunk_mat_free(a, cd);  // corners from the solid rows
    int* vemask = slot_ptr<int>(a, chunk, a.L.v_emask);
    int* vmat = slot_ptr<int>(a, chunk, a.L.v_mat);
    float4* verts = slot_ptr<float4>(a, chunk, a.L.verts);
    uint32_t* qcount = slot_ptr<uint32_t>(a, chunk, a.L.q_count);
    uint64_t* smask = slot_ptr<uint64_t>(a, chunk, a.L.s_mask);
    const int lane = threadIdx.x & 63;
    const int N = G.N;
    for (int base = wave_in_chunk() << 6; base < V; base += waves_per_chunk() << 6) {
        const int vi = base + lane;
        int qbits = 0, seam = 0;
        if (vi < V) {
            const int3 p = position_for_code((uint32_t)vcode[vi], G.depth);
            int corners, dominant;
            if (rows && a.defmat < kNone) {  // the default material sorts before air and is the only one
                corners = corners_from_rows(a, S, p.x, p.y, p.z);
                dominant = corners ? a.defmat : kAir;
            } else {
                int cm[8];
                if (rows) {
                    corners = corners_from_rows(a, S, p.x, p.y, p.z);
#pragma unroll
                    for (int i = 0; i < 8; ++i) cm[i] = (corners >> i) & 1 ? a.defmat : kAir;
                } else {
                    corners = corner_materials(a, mat, p.x, p.y, p.z, cm);
                }
                dominant = dominant_material(cm);
            }
            const int emask = edges_of_corners(corners);
            const int m = (dominant << 8) | corners;
            float4 pos, nrm;
            if constexpr (kPrecise)
                qef_precise(a, chunk, cd, p, emask, pos, nrm);
            else
                qef_fast(a, chunk, cd, p, emask, pos, nrm);
#pragma unroll
            for (int axis = 0; axis < 3; ++axis) qbits |= quad_flag(G, p, emask, axis) << axis;
            seam = p.x == 0 || p.x == N - 1 || p.y == 0 || p.y == N - 1 || p.z == 0 || p.z == N - 1;
            vemask[vi] = emask | (qbits << 12);
            vmat[vi] = m;
            verts[3 * vi] = pos;
            verts[3 * vi + 1] = nrm;
            verts[3 * vi + 2] = make_float4(cd.colour[0], cd.colour[1], cd.colour[2], (float)(m >> 8));
        }
        const int nq = __popc(qbits);
        const uint64_t b0 = __ballot(nq & 1), b1 = __ballot(nq & 2), sm = __ballot(seam);
        if (lane == 0) {
            const int seg = base >> 6;
            qcount[seg] = (uint32_t)(__popcll(b0) + 2 * __popcll(b1)) | ((uint32_t)__popcll(sm) << 16);
            smask[seg] = sm;
        }
    }
}

// Quad and seam scans of one chunk in one workgroup (the segment count is the
// chunk's voxel count, known only on the device).
__global__ __launch_bounds__(kScanThreads) void k_scan_quads_seams(KArgs a) {
    __shared__ uint64_t wsum[kScanThreads / 64];
    const int chunk = blockIdx.y;
    Counters* cnt = a.counters + chunk;
    const int n = (cnt->voxels + 63) >> 6;
    if (n == 0) return;  // the counters stay cleared
    const uint32_t* count = slot_ptr<const uint32_t>(a, chunk, a.L.q_count);
    int2* base = slot_ptr<int2>(a, chunk, a.L.q_base);
    const uint64_t t = block_scan(n, wsum, [&](int i) { return halves(count[i]); },
                                  [&](int i, uint64_t at) { base[i] = make_int2((int)(uint32_t)at, (int)(at >> 32)); });
    if (threadIdx.x == 0) {
        const int q = (int)(uint32_t)t, sn = (int)(t >> 32);
        cnt->quads = min(q, a.caps.quads);
        if (q > a.caps.quads) atomicOr(&cnt->status, kStatusQuadOverflow);
        cnt->seams = min(sn, a.caps.seams);
        if (sn > a.caps.seams) atomicOr(&cnt->status, kStatusSeamOverflow);
    }
}

// cl/octree.cl:376-381
__constant__ int kEdgeNodeOffsets[3][4][3] = {{{0, 0, 0}, {0, 0, 1}, {0, 1, 0}, {0, 1, 1}},
                                              {{0, 0, 0}, {1, 0, 0}, {0, 0, 1}, {1, 0, 1}},
                                              {{0, 0, 0}, {0, 1, 0}, {1, 0, 0}, {1, 1, 0}}};

// Quads (GenerateMesh + CompactMeshTriangles, cl/octree.cl:335-464) in (voxel,
// axis) order, and seam nodes (ExtractSeamNodeInfo, cl/octree.cl:529-551) in
// voxel order.  A segment's quads fill one contiguous run of the index buffer
// (at most 3 per voxel): each wave builds its run in LDS and copies it out with
// 8-byte stores of consecutive addresses, so every store instruction writes whole
// lines instead of 64 scattered 12-byte pieces.
constexpr int kEmitWaves = 4;                  // waves per k_emit workgroup
constexpr int kEmitStageInts = 64 * 3 * 6;     // one segment's quads, 6 indices each
__global__ __launch_bounds__(64 * kEmitWaves) void k_emit(KArgs a) {
    __shared__ int2 stage_all[kEmitWaves][kEmitStageInts / 2];
    int* stage = reinterpret_cast<int*>(stage_all[threadIdx.x >> 6]);
    const int chunk = blockIdx.y;
    const Geometry& G = a.G;
    const int V = a.counters[chunk].voxels;
    const int* vcode = slot_ptr<const int>(a, chunk, a.L.v_code);
    const int* vemask = slot_ptr<const int>(a, chunk, a.L.v_emask);
    const int* vmat = slot_ptr<const int>(a, chunk, a.L.v_mat);
    const uint64_t* vm = slot_ptr<const uint64_t>(a, chunk, a.L.v_mask);
    const int* vb = slot_ptr<const int>(a, chunk, a.L.v_base);
    const int2* qbase = slot_ptr<const int2>(a, chunk, a.L.q_base);  // quads, seam nodes
    const uint64_t* smask = slot_ptr<const uint64_t>(a, chunk, a.L.s_mask);
    const float4* verts = slot_ptr<const float4>(a, chunk, a.L.verts);
    int* tris = slot_ptr<int>(a, chunk, a.L.tris);
    float4* seams = slot_ptr<float4>(a, chunk, a.L.seams);
    const int lane = threadIdx.x & 63;
    const uint64_t lt = lanemask_lt(lane);
    for (int base = wave_in_chunk() << 6; base < V; base += waves_per_chunk() << 6) {
        const int vi = base + lane, seg = base >> 6;
        // the voxel's own words, loaded together (a lane past the end reads the last voxel)
        const int vc = min(vi, V - 1);
        const int em = vemask[vc], code = vcode[vc], m = vmat[vc];
        const int2 qs = qbase[seg];
        const int qb = qs.x;
        const uint64_t sm = smask[seg];
        const int qbits = vi < V ? (em >> 12) & 7 : 0;
        const int nq = __popc(qbits);
        const uint64_t b0 = __ballot(nq & 1), b1 = __ballot(nq & 2);
        const bool seam = (sm >> lane) & 1ull;
        const int run = __popcll(b0) + 2 * __popcll(b1);  // the segment's quads
        if (vi < V && (qbits || seam)) {
            const int3 p = position_for_code((uint32_t)code, G.depth);
            int qi = __popcll(b0 & lt) + 2 * __popcll(b1 & lt);  // within the segment's run
            // The nine neighbour lookups (three per axis) are loaded together, before any is
            // used: one memory round trip instead of one per axis and step.  An index is
            // clamped into the grid, so an axis without a quad reads a valid, unused word (a
            // quad's neighbours all lie in the grid: quad_flag excludes the last layers).
            uint64_t nw[3][3];
            int nb[3][3], nl[3][3];
            if (G.N == 64) {
                // A segment is the voxel row (y, z): the nine neighbours (kEdgeNodeOffsets) lie
                // in the rows (y, z), (y + 1, z), (y, z + 1) and (y + 1, z + 1), at x or x + 1.
                const int r = p.y + 64 * p.z, rmax = 64 * 64 - 1;
                const int r10 = min(r + 1, rmax), r01 = min(r + 64, rmax), r11 = min(r + 65, rmax);
                const uint64_t m00 = vm[r], m10 = vm[r10], m01 = vm[r01], m11 = vm[r11];
                const int b00 = vb[r], b10 = vb[r10], b01 = vb[r01], b11 = vb[r11];
                const int x0 = p.x, x1 = (p.x + 1) & 63;
                nw[0][0] = m01; nb[0][0] = b01; nl[0][0] = x0;  // (0, 0, 1)
                nw[0][1] = m10; nb[0][1] = b10; nl[0][1] = x0;  // (0, 1, 0)
                nw[0][2] = m11; nb[0][2] = b11; nl[0][2] = x0;  // (0, 1, 1)
                nw[1][0] = m00; nb[1][0] = b00; nl[1][0] = x1;  // (1, 0, 0)
                nw[1][1] = m01; nb[1][1] = b01; nl[1][1] = x0;  // (0, 0, 1)
                nw[1][2] = m01; nb[1][2] = b01; nl[1][2] = x1;  // (1, 0, 1)
                nw[2][0] = m10; nb[2][0] = b10; nl[2][0] = x0;  // (0, 1, 0)
                nw[2][1] = m00; nb[2][1] = b00; nl[2][1] = x1;  // (1, 0, 0)
                nw[2][2] = m10; nb[2][2] = b10; nl[2][2] = x1;  // (1, 1, 0)
            } else {
                const int last = G.N * G.N * G.N - 1;
                #pragma unroll
                for (int axis = 0; axis < 3; ++axis) {
                    #pragma unroll
                    for (int n = 1; n < 4; ++n) {
                        const int x = p.x + kEdgeNodeOffsets[axis][n][0];
                        const int y = p.y + kEdgeNodeOffsets[axis][n][1];
                        const int z = p.z + kEdgeNodeOffsets[axis][n][2];
                        const int i = min(x + G.N * (y + G.N * z), last);
                        nw[axis][n - 1] = vm[i >> 6];
                        nb[axis][n - 1] = vb[i >> 6];
                        nl[axis][n - 1] = i & 63;
                    }
                }
            }
            #pragma unroll
            for (int axis = 0; axis < 3; ++axis) {
                if (!((qbits >> axis) & 1)) continue;
                int nodes[4];
                nodes[0] = vi;
                bool ok = true;
                #pragma unroll
                for (int n = 1; n < 4; ++n) {
                    nodes[n] = dense_index_of(nw[axis][n - 1], nb[axis][n - 1], nl[axis][n - 1]);
                    ok = ok && nodes[n] >= 0;
                }
                int3* out = reinterpret_cast<int3*>(stage + 6 * qi);  // two 12-byte LDS stores
                if (!ok) {  // cannot happen: all four voxels around a sign-changing interior edge are active
                    atomicOr(&a.counters[chunk].status, kStatusLookupMiss);
                    out[0] = out[1] = make_int3(0, 0, 0);
                } else {
                    const int edge = axis * 4 + 3;
                    const int flip = ((m >> kEdgeMap[edge][0]) & 1) != 0 ? 1 : 0;  // ProcessEdge, cl/octree.cl:335-372
                    if (flip) {
                        out[0] = make_int3(nodes[0], nodes[3], nodes[1]);
                        out[1] = make_int3(nodes[0], nodes[2], nodes[3]);
                    } else {
                        out[0] = make_int3(nodes[0], nodes[1], nodes[3]);
                        out[1] = make_int3(nodes[0], nodes[3], nodes[2]);
                    }
                }
                ++qi;
            }
            if (seam) {
                const int si = qs.y + __popcll(sm & lt);
                if (si < a.caps.seams) {
                    const float4 pos = verts[3 * vi], nrm = verts[3 * vi + 1];
                    reinterpret_cast<int4*>(seams)[3 * si] = make_int4(p.x, p.y, p.z, m);
                    seams[3 * si + 1] = pos;
                    seams[3 * si + 2] = nrm;
                }
            }
        }
        // The run's LDS stores are complete before any lane of the wave reads them back.
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        // Copy the run to quads [qb, qb + run), clipped at the quad capacity; 6 indices
        // per quad make it a whole number of 8-byte pairs at an 8-byte aligned address.
        const int keep = max(0, min(run, a.caps.quads - qb));
        int2* dst = reinterpret_cast<int2*>(tris + 6 * (long)qb);
        const int2* src = reinterpret_cast<const int2*>(stage);
        for (int i = lane; i < 3 * keep; i += 64) dst[i] = src[i];
        // ... and every lane has read the run before the next segment overwrites it.
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    }
}

// One mesh read back into the caller's pinned buffers by one launch and one wait.  Bound by
// the host link (57 GB/s).  Three hipMemcpy calls and a read of the chunk's counters, each
// waited for, took 64 chunks of 1.2 MB 3.3 ms; this and counters read once per run take 1.9.
// Copies in the widest units that addresses and sizes allow.
template <typename Word>
__device__ __forceinline__ void copy_words(const char* src, char* dst, uint64_t bytes) {
    const Word* s = reinterpret_cast<const Word*>(src);
    Word* d = reinterpret_cast<Word*>(dst);
    const uint64_t n = bytes / sizeof(Word), step = (uint64_t)gridDim.x * blockDim.x;
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += step) d[i] = s[i];
}
__global__ __launch_bounds__(256) void k_copy_mesh(MeshCopy c) {
    const uint64_t odd = (uint64_t)c.src[blockIdx.y] | (uint64_t)c.dst[blockIdx.y] | c.bytes[blockIdx.y];
    if ((odd & 15) == 0)
        copy_words<uint4>(c.src[blockIdx.y], c.dst[blockIdx.y], c.bytes[blockIdx.y]);
    else if ((odd & 7) == 0)
        copy_words<uint2>(c.src[blockIdx.y], c.dst[blockIdx.y], c.bytes[blockIdx.y]);
    else
        copy_words<uint32_t>(c.src[blockIdx.y], c.dst[blockIdx.y], c.bytes[blockIdx.y]);
}

// The one-chunk forms' export as the pipeline's last kernel: the counters and the mesh in one
// pass to the host, so the caller waits once instead of for the counters, then three device
// copies into the mesh cache and one read-back; the cache's copy now runs beside the host's.
// Bound by the host link: 2 MB of a 64^3 cave chunk in 45 us.  With k_stage_chunk that call
// went 297 -> 286 us, a two-step edit 779 -> 720, a 16^3 chunk 145 -> 125.
__global__ __launch_bounds__(256) void k_export(KArgs a, char* out) {
    const Counters k = a.counters[0];
    if (blockIdx.x == 0 && blockIdx.y == 0 && threadIdx.x == 0) *reinterpret_cast<Counters*>(out) = k;
    if (k.status || k.edges == 0) return;
    const uint64_t bv = k.quads > 0 ? 48ull * k.voxels : 0, bt = 24ull * k.quads, bs = 48ull * k.seams;
    char* at = out + kExportHeader;
    if (blockIdx.y == 0)
        copy_words<uint4>(slot_ptr<const char>(a, 0, a.L.verts), at, bv);
    else if (blockIdx.y == 1)
        copy_words<uint2>(slot_ptr<const char>(a, 0, a.L.tris), at + bv, bt);
    else
        copy_words<uint2>(slot_ptr<const char>(a, 0, a.L.seams), at + bv + bt, bs);
}

static inline unsigned ceil_div(long a, long b) { return (unsigned)((a + b - 1) / b); }

// Zero the per-chunk counters (a kernel rather than a memset node, so that a
// captured graph clears them correctly on every replay).
// The first workgroup also lists the chunks with brushes or a cached field, which are few in
// a batch: k_csg and k_edge_data walk that list instead of every descriptor (28 us of 1,800).
constexpr int kClearThreads = 1024;
__global__ __launch_bounds__(kClearThreads) void k_clear_counters(Counters* c, int n, int* queue, const ChunkDesc* chunks,
                                                                  int* special) {
    __shared__ int wcount[kClearThreads / 64];
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) c[i] = Counters{};
    if (blockIdx.x) return;
    if (i < kNumQueues) queue[i] = 0;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    int count = 0;
    for (int base = 0; base < n; base += kClearThreads) {
        const int k = base + (int)threadIdx.x;
        const bool listed = k < n && (chunks[k].op_count > 0 || chunks[k].mode == kModeCached);
        const uint64_t hits = __ballot(listed);
        if (lane == 0) wcount[wave] = __popcll(hits);
        __syncthreads();
        int before = count, all = count;
        for (int w = 0; w < kClearThreads / 64; ++w) {
            before += w < wave ? wcount[w] : 0;
            all += wcount[w];
        }
        if (listed) special[1 + before + __popcll(hits & lanemask_lt(lane))] = k;
        count = all;
        __syncthreads();
    }
    if (threadIdx.x == 0) special[0] = count;
}

// The one-chunk forms' inputs, read from pinned host memory by the pipeline's first kernel
// (a descriptor and 68 bytes an op) instead of up to three copies and a clear launched ahead
// of it: about 20 us of a one-chunk call were spent before its first stage.
__global__ __launch_bounds__(256) void k_stage_chunk(const ChunkDesc* chunk, const DevOp* ops, const int* index,
                                                     ChunkDesc* d_chunk, DevOp* d_ops, int* d_index, Counters* c,
                                                     int* queue, int* special) {
    static_assert(sizeof(ChunkDesc) % 4 == 0 && sizeof(DevOp) == 64, "copied in words");
    const int t = threadIdx.x, n = chunk->op_count;
    if (t < (int)(sizeof(ChunkDesc) / 4)) reinterpret_cast<uint32_t*>(d_chunk)[t] = reinterpret_cast<const uint32_t*>(chunk)[t];
    if (t == 0) {
        *c = Counters{};
        special[0] = n > 0 || chunk->mode == kModeCached ? 1 : 0;
        special[1] = 0;
    }
    if (t < kNumQueues) queue[t] = 0;
    for (int i = t; i < 4 * n; i += 256) reinterpret_cast<uint4*>(d_ops)[i] = reinterpret_cast<const uint4*>(ops)[i];
    for (int i = t; i < n; i += 256) d_index[i] = index[i];
}

// ---------------------------------------------------------------------------
// Launchers
// ---------------------------------------------------------------------------

void launch_stage_chunk(const KArgs& a, const ChunkDesc* chunk, const DevOp* ops, const int* index, hipStream_t s) {
    hipLaunchKernelGGL(k_stage_chunk, dim3(1), dim3(256), 0, s, chunk, ops, index, const_cast<ChunkDesc*>(a.chunks),
                       const_cast<DevOp*>(a.ops), const_cast<int*>(a.op_index), a.counters, a.queue, a.special);
}

void launch_clear_counters(const KArgs& a, int n, hipStream_t s) {
    hipLaunchKernelGGL(k_clear_counters, dim3(ceil_div(std::max(n, 1), kClearThreads)), dim3(kClearThreads), 0, s,
                       a.counters, n, a.queue, a.chunks, a.special);
}

// A kernel over the field, built for the launch's field kind; the work-counting form takes
// any kind.  Further template arguments follow the kind.
#define LVN_LAUNCH_KIND(kernel, grid, block, ...)                                                                 \
    do {                                                                                                          \
        if (a.work)                                                                                               \
            hipLaunchKernelGGL((kernel<true, kAnyField __VA_OPT__(, ) __VA_ARGS__>), grid, block, 0, s, a, chunks);  \
        else if (a.F.kind == LVN_FIELD_LEVEN_TERRAIN)                                                             \
            hipLaunchKernelGGL((kernel<false, LVN_FIELD_LEVEN_TERRAIN __VA_OPT__(, ) __VA_ARGS__>), grid, block, 0,  \
                               s, a, chunks);                                                                     \
        else if (a.F.kind == LVN_FIELD_TERRAIN_CAVES)                                                             \
            hipLaunchKernelGGL((kernel<false, LVN_FIELD_TERRAIN_CAVES __VA_OPT__(, ) __VA_ARGS__>), grid, block, 0,  \
                               s, a, chunks);                                                                     \
        else                                                                                                      \
            hipLaunchKernelGGL((kernel<false, LVN_FIELD_HEIGHTFIELD __VA_OPT__(, ) __VA_ARGS__>), grid, block, 0, s, \
                               a, chunks);                                                                        \
    } while (0)

// per_cu workgroups per CU (at most two: the LDS table limit), fewer when the work is
// small.
static unsigned persistent_blocks(const KArgs& a, int per_cu, long items) {
    return (unsigned)std::max(1L, std::min((long)per_cu * a.cus, (items + 15) / 16));
}

// A column item evaluates the height term once and then its y-segment.  With the cave term
// the segment is the cost (a 66-sample column is 0.18 ms of dependent octaves), so few
// chunks are cut finely, down to two samples, until about 20,000 items fill the chip, and
// never below three segments, which balance caves against sky; without it each segment
// repeats the whole height term, so a cut pays only where samples are stored (one chunk, or
// chunks under brushes) and until about 3,400 items are in flight.
// Measured with caves (density stage, us): one chunk 29 with 6 segments, 15 with these; 8
// chunks 41 -> 36; 24 chunks 73 -> 69; 96 chunks 271 with one, 198 with these; 500 chunks 944
// -> 844 (with the workgroups below).  Reference terrain, one chunk with stored samples 14
// with 6 segments, 12 with these; batches of solid planes alone take 11 us up to 16 chunks
// and 55 for 500 whole, 1.7 times that in two segments.
int default_ysplit(const Geometry& G, int field_kind, int chunks) {
    const long items = (long)G.col_groups * std::max(1, chunks);
    if (field_kind == LVN_FIELD_TERRAIN_CAVES) return (int)std::clamp(20000L / items, 3L, (long)G.F / 2);
    return (int)std::clamp(3400L / items, 1L, std::min(11L, (long)G.F / 2));
}
// Two workgroups per CU once one per CU has every wave busy (500 chunks: 904 -> 844 us
// with caves, 59 -> 55 without); below that a second one only loads tables.
int default_density_per_cu(const Geometry& G, int ysplit, int chunks, int cus) {
    return (long)G.col_groups * ysplit * chunks > 16L * cus ? 2 : 1;
}

void launch_density(const KArgs& a, int chunks, hipStream_t s) {
    const long items = (long)a.G.col_groups * a.ysplit * chunks;
    // density_per_cu workgroups per CU (two fit, by the kernel's register caps), or one per
    // item where there are fewer items than that.
    const int per_cu = a.density_per_cu ? a.density_per_cu : default_density_per_cu(a.G, a.ysplit, chunks, a.cus);
    const unsigned blocks = (unsigned)std::max(1L, std::min((long)per_cu * a.cus, items));
    LVN_LAUNCH_KIND(k_density, dim3(blocks), dim3(1024));
}
void launch_copy_mesh(const MeshCopy& c, hipStream_t s) {
    const uint64_t most = std::max(c.bytes[0], std::max(c.bytes[1], c.bytes[2]));
    const unsigned blocks = std::clamp(ceil_div((long)(most / 16), 256), 1u, 256u);
    hipLaunchKernelGGL(k_copy_mesh, dim3(blocks, 3), dim3(256), 0, s, c);
}
void launch_export(const KArgs& a, char* out, hipStream_t s) {
    hipLaunchKernelGGL(k_export, dim3(128, 3), dim3(256), 0, s, a, out);
}
void launch_csg(const KArgs& a, int chunks, hipStream_t s) {
    // a few chunks have no more tiles than that many waves
    const long tiles = (long)((a.G.F + kCsgX - 1) / kCsgX) * ((a.G.F + kCsgY - 1) / kCsgY) * ((a.G.F + kCsgZ - 1) / kCsgZ);
    hipLaunchKernelGGL(k_csg, dim3((unsigned)std::min((long)kCsgBlocks, ceil_div(tiles * chunks, 4) + 0L)), dim3(256), 0, s, a);
}
// Workgroups per chunk for a kernel that loops over `threads` work items of 256-thread
// workgroups: all of them for a few chunks, about `target` workgroups over a large batch.
static unsigned chunk_blocks(int chunks, long threads, int target) {
    const long full = std::max(1L, (threads + 255) / 256);
    const long share = std::max(1L, ((long)target + chunks - 1) / chunks);
    return (unsigned)std::min(full, share);
}

void launch_rows(const KArgs& a, int chunks, hipStream_t s) {
    const long solid_waves = (a.G.field_rows + kRowsPerBlock - 1) / kRowsPerBlock;
    hipLaunchKernelGGL(k_solid_rows, dim3(chunk_blocks(chunks, 64L * solid_waves, a.row_blocks), chunks), dim3(256), 0, s, a);
    const unsigned eb = chunk_blocks(chunks, a.G.edge_rows, a.row_blocks);
    const unsigned vb = chunk_blocks(chunks, a.G.voxel_segs, a.row_blocks);
    hipLaunchKernelGGL(k_rows, dim3(eb + vb, chunks), dim3(256), 0, s, a, (int)eb);
}
void launch_scan_rows(const KArgs& a, int chunks, hipStream_t s) {
    hipLaunchKernelGGL(k_scan_rows, dim3(2, chunks), dim3(kScanThreads), 0, s, a);
}
void launch_scan_quads_seams(const KArgs& a, int chunks, hipStream_t s) {
    hipLaunchKernelGGL(k_scan_quads_seams, dim3(1, chunks), dim3(kScanThreads), 0, s, a);
}
void launch_compact(const KArgs& a, int chunks, hipStream_t s) {
    // A wave per 64 rows, or four while one each does not fill the chip (32 waves per CU):
    // one chunk 9.5 -> 5.4 us, 24 chunks 11 -> 7; but 1,800 chunks 80 -> 139 us, whose rows
    // are mostly empty and looked at four times.
    const long edge_groups = (a.G.edge_rows + 63) / 64, voxel_groups = (a.G.voxel_segs + 63) / 64;
    const int split = (edge_groups + voxel_groups) * chunks < 32L * a.cus ? 4 : 1;
    const unsigned eb = chunk_blocks(chunks, 64L * edge_groups * split, a.row_blocks);
    const unsigned vb = chunk_blocks(chunks, 64L * voxel_groups * split, a.row_blocks);
    hipLaunchKernelGGL(k_compact, dim3(eb + vb, chunks), dim3(256), 0, s, a, (int)eb, split);
}
// Lanes per edge of the crossing stage: the tuned value, else by field and batch size (a
// typical 64^3 chunk has a few hundred 64-edge items, a chunk of N^3 about (N / 64)^2 of
// that; kG lanes multiply the waves and divide each wave's chain of dependent octaves).
// Crossing stage measured at 1 / 2 / 4 / 8 lanes (us): heightfield, 8 chunks 36/33/28/25,
// 32 chunks 52/42/35/35, 200 chunks 88/84/98/108, 500 chunks 196/198/253/302; caves, 1 chunk
// 131/67/46/32, 8 chunks 86/87/75/74, 64 chunks 415/339/382/406, 96 chunks 501/519/594/638;
// the reference's terrain, whose 14 octaves a term make the longest chains, chunks spread over
// its clipmap, 24 chunks 91/58/48/38, 64 chunks 91/69/58/55, 90 chunks 111/80/78/79, 120 chunks
// 152/118/125/127, 300 chunks 290/235/268/284, 1,800 chunks 956-1,017/927-933/1,198/1,311; the
// chunks nearest its surface, 64 chunks 206/170/171/166, 200 chunks 243/202/211/211, 400 chunks
// 348/311/362/378.
// Sampled coarsely, caves cross more of the edges (17,000 a chunk at voxel size 1, 170,000
// and more at 32: 50 such chunks 2,485 us with 1 lane, 2,700 with 2), hence chunk_load.
static long full_chunks(const Geometry& G, int load) { return std::max(1L, (long)load * G.N * G.N / 4096); }

int default_cross_lanes(const Geometry& G, int field_kind, int load) {
    const long n = full_chunks(G, load);
    if (field_kind == LVN_FIELD_LEVEN_TERRAIN) return n <= 100 ? 8 : 2;
    if (field_kind == LVN_FIELD_TERRAIN_CAVES) return n <= 10 ? 8 : n <= 80 ? 2 : 1;
    return n <= 12 ? 8 : n <= 48 ? 4 : n <= 400 ? 2 : 1;
}

// Line heights pay where several crossings share a line, as caves make them, and the pass
// before the crossings is short beside these: 200 chunks of caves 1,406 -> 1,219 us, 32
// chunks 263 -> 254, one chunk 131 -> 136.  A surface crosses a line about once: 1,800
// chunks of the reference's terrain 903 without, 944 with.
int default_height_lines(const Geometry& G, int field_kind, int load) {
    return field_kind == LVN_FIELD_TERRAIN_CAVES && full_chunks(G, load) >= 64 ? 1 : 0;
}

static int cross_lanes(const KArgs& a, int chunks) {
    return a.cross_lanes > 0 ? a.cross_lanes : default_cross_lanes(a.G, a.F.kind, a.load ? a.load : chunks);
}

constexpr int kEdgeDataBlocks = 1024;

template <int kG>
static void launch_cross_group(const KArgs& a, int chunks, hipStream_t s) {
    const dim3 grid(persistent_blocks(a, a.persist_per_cu, 512L * kG * chunks));
    LVN_LAUNCH_KIND(k_edge_cross_group, grid, dim3(kCrossThreads), kG);
}

void launch_edge_cross(const KArgs& a, int chunks, hipStream_t s) {
    if (a.height_lines) {
        const long line_items = 2L * a.G.H * chunks;
        const dim3 line_grid(persistent_blocks(a, 2, line_items));  // 63 SGPRs: two workgroups per CU stay resident
        LVN_LAUNCH_KIND(k_height_lines, line_grid, dim3(1024));
    }
    const int g = cross_lanes(a, chunks);
    // 1,024 waves of brush and cached edges (of a few chunks: 96 KB of hermite data), and
    // one workgroup that counts the items
    const dim3 data_grid(kEdgeDataBlocks + 1), data_block(kEdgeDataThreads);
    const int per_item = g == kCrossSampleParallel ? 64 : 64 / g;
    auto* const data_kernel = a.work ? (chunks <= kFewChunks ? k_edge_data<true, true> : k_edge_data<true, false>)
                                     : (chunks <= kFewChunks ? k_edge_data<false, true> : k_edge_data<false, false>);
    hipLaunchKernelGGL(data_kernel, data_grid, data_block, 0, s, a, chunks, per_item);
    // the item count is on the device; size the grid for 512 edge items per chunk
    switch (g) {
    case 2: launch_cross_group<2>(a, chunks, s); return;
    case 4: launch_cross_group<4>(a, chunks, s); return;
    case 8: launch_cross_group<8>(a, chunks, s); return;
    case kCrossSampleParallel: {
        const dim3 grid(persistent_blocks(a, a.persist_per_cu, 512L * chunks));
        LVN_LAUNCH_KIND(k_edge_cross_sp, grid, dim3(kCrossThreads));
        return;
    }
    default: break;
    }
    const dim3 grid(persistent_blocks(a, a.persist_per_cu, 512L * chunks));
    LVN_LAUNCH_KIND(k_edge_cross, grid, dim3(kCrossThreads));
}
// The kernels below loop up to the chunk's voxel count, known only on the device.
void launch_qef(const KArgs& a, int chunks, hipStream_t s) {
    const dim3 grid(chunk_blocks(chunks, a.caps.voxels, a.voxel_blocks), chunks);
    if (a.precise)
        hipLaunchKernelGGL(k_qef<true>, grid, dim3(256), 0, s, a);
    else
        hipLaunchKernelGGL(k_qef<false>, grid, dim3(256), 0, s, a);
}
void launch_emit(const KArgs& a, int chunks, hipStream_t s) {
    hipLaunchKernelGGL(k_emit, dim3(chunk_blocks(chunks, a.caps.voxels, a.voxel_blocks), chunks), dim3(64 * kEmitWaves), 0,
                       s, a);
}

const char* const kStageNames[kNumStages] = {
    "density", "csg", "edge_rows", "scan_edges", "edge_compact", "edge_cross",
    "voxel_rows", "scan_voxels", "voxel_compact", "qef", "scan_quads_seams", "emit"};

void launch_stage(const KArgs& a, int chunks, int i, hipStream_t s) {
    switch (i) {
    case 0: launch_density(a, chunks, s); break;
    case 1: launch_csg(a, chunks, s); break;
    case 2: launch_rows(a, chunks, s); break;  // edge and voxel rows
    case 3: launch_scan_rows(a, chunks, s); break;
    case 4: launch_compact(a, chunks, s); break;
    case 5: launch_edge_cross(a, chunks, s); break;
    case 6:
    case 7:
    case 8: break;  // stage_launches
    case 9: launch_qef(a, chunks, s); break;
    case 10: launch_scan_quads_seams(a, chunks, s); break;
    default: launch_emit(a, chunks, s); break;
    }
}

void launch_stages(const KArgs& a, int chunks, hipStream_t s) {
    for (int i = 0; i < kNumStages; ++i) launch_stage(a, chunks, i, s);
}

void launch_pipeline(const KArgs& a, int chunks, hipStream_t s) {
    launch_clear_counters(a, chunks, s);
    launch_stages(a, chunks, s);
}

}  // namespace lvn
