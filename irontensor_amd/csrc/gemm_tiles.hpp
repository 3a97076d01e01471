// What the GEMM translation units share: operand loads, the tile order, and the grouped form's
// arguments and schedule.
#pragma once

#include <algorithm>
#include <cmath>

#include "epilogue.hpp"
#include "internal.hpp"
#include "mfma.hpp"

namespace it {

// Several independent GEMMs of one layout in one launch. Workgroup w runs on XCD w % 8, and each
// XCD has its own L2, so the blocks are scheduled per XCD: XCD x runs blocks j = 0 .. xn[x] - 1
// (workgroup j * 8 + x), an equal share of the group's tiles x splits, as contiguous chunks. Chunk c
// gives blocks jstart.. of its XCD the tiles t0, t0 + 1, ... (grouped raster order) of split `split`
// of problem gi, until the next chunk of that XCD starts. A problem's split then sits on one XCD
// (or two, where a share ends inside it), and its operand panels are fetched into one L2 instead of
// eight.
constexpr int GEMM_GROUP_MAX = 8;
constexpr int GROUP_CHUNKS = 96;
struct GroupChunk {
    uint16_t jstart;
    uint8_t gi, split;
    uint16_t t0, unused;
};
struct GemmGroupArgs {
    GemmArgs g[GEMM_GROUP_MAX];
    int *arrive;                         // FP32 groups: the split-K arrival counters (zero),
    int cstart[GEMM_GROUP_MAX + 1];      // problem g's tiles at arrive[cstart[g]] ..
    int count;
    uint16_t xn[8];                      // blocks of XCD x
    uint16_t xstart[9];                  // its chunks: chunk[xstart[x]] .. chunk[xstart[x + 1] - 1]
    GroupChunk chunk[GROUP_CHUNKS];
};

namespace {

constexpr int NTHREADS = 256;
constexpr int ROW_PITCH = 144;  // LDS bytes per row of a [rows][BK] tile (128 data + 16 pad)

template <typename T>
struct ET;
template <>
struct ET<float> {
    static constexpr int VEC = 4;    // elements per 16 bytes
    static constexpr int BK = 32;    // k per tile
    static constexpr int KSTEP = 16; // k per fragment step (4 lane groups x 4)
};
template <>
struct ET<uint16_t> {
    static constexpr int VEC = 8;
    static constexpr int BK = 64;
    static constexpr int KSTEP = 32;
};


// Loads VEC consecutive elements starting at base[off]; elements at positions c + e >= clim (or the
// whole vector when !row_ok) read as zero.
template <typename T>
__device__ __forceinline__ u32x4 load_vec(const T *base, int64_t off, bool row_ok, int64_t c,
                                          int64_t clim, bool vec_ok) {
    constexpr int VEC = ET<T>::VEC;
    if (row_ok && vec_ok && c + VEC <= clim) return *(const u32x4 *)(base + off);
    u32x4 v = {0u, 0u, 0u, 0u};
    if (row_ok) {
        if constexpr (sizeof(T) == 4) {
#pragma unroll
            for (int e = 0; e < 4; ++e)
                if (c + e < clim) v[e] = __float_as_uint(base[off + e]);
        } else {
#pragma unroll
            for (int e = 0; e < 8; ++e)
                if (c + e < clim) v[e >> 1] |= (uint32_t)base[off + e] << ((e & 1) * 16);
        }
    }
    return v;
}

// How an operand tile is read from global memory:
//   LOAD_EXACT   every tile is whole and aligned: plain 128-bit loads;
//   LOAD_MASKED  16-byte vectors are aligned and never straddle an edge, so a vector is either
//                wholly in bounds or wholly out: branch-free load of a safe address + select;
//   LOAD_CHECKED anything else: per-element bounds checks.
//   LOAD_RSRC    (FP32, 16-byte vectors as LOAD_MASKED, K a multiple of the k-tile where an operand
//                is k-contiguous) buffer loads through a descriptor that ends where the operand's
//                valid rows (k-contiguous) or k (mn-contiguous) end, from 32-bit offsets formed once
//                per block: the hardware's range check returns zeros past that end, with no
//                per-load address arithmetic or selects. The descriptor spans exactly the
//                operand's elements (first to last, not whole row strides, which can reach past the
//                allocation for a strided head). An mn-contiguous operand's columns past M (or N)
//                read the next row's elements, or zeros past the last element; they reach only
//                output rows (columns) past M (N), which the epilogue never stores.
enum LoadMode : int { LOAD_EXACT = 0, LOAD_MASKED = 1, LOAD_CHECKED = 2, LOAD_RSRC = 3 };

template <int MODE, typename T>
__device__ __forceinline__ u32x4 load_mode(const T *base, int64_t off, bool row_ok, int64_t c,
                                           int64_t clim, bool vec_ok) {
    if constexpr (MODE == LOAD_EXACT) {
        return *(const u32x4 *)(base + off);
    } else if constexpr (MODE == LOAD_MASKED) {
        const bool ok = row_ok && c < clim;
        const u32x4 v = *(const u32x4 *)(base + (ok ? off : 0));
        return ok ? v : u32x4{0u, 0u, 0u, 0u};
    } else {
        return load_vec<T>(base, off, row_ok, c, clim, vec_ok);
    }
}

// Grouped raster order: tile `idx` of groups of 8 tile rows, column-major within a group.
__device__ __forceinline__ void raster_tile(int idx, int tiles_m, int tiles_n, int &tm, int &tn) {
    constexpr int GROUP = 8;
    const int span = GROUP * tiles_n;
    const int first_m = (idx / span) * GROUP;
    const int gsize = min(tiles_m - first_m, GROUP);
    const int in = idx % span;
    tm = first_m + in % gsize;
    tn = in / gsize;
}

// Tile order: XCD-aware remap (workgroup w runs on XCD w % 8, which then takes a contiguous range
// of the grouped order) then the grouped raster.
__device__ __forceinline__ void map_tile(int pid, int tiles_m, int tiles_n, int &tm, int &tn) {
    constexpr int NXCD = 8;
    const int total = tiles_m * tiles_n;
    if (total % NXCD == 0) pid = (pid % NXCD) * (total / NXCD) + pid / NXCD;
    raster_tile(pid, tiles_m, tiles_n, tm, tn);
}

namespace sg {
constexpr int VALU = 0x002, MFMA = 0x008, VMEM_READ = 0x020, DS_READ = 0x100, DS_WRITE = 0x200;
}

constexpr int CP_DEVICE_SCOPE = 16;  // cache-policy bit sc1 of the buffer intrinsics: device scope

// The map_tile index whose tile is number r of the grouped raster order (map_tile's XCD remap
// undone: the group's schedule has already placed the block on its XCD).
__device__ __forceinline__ int raster_pid(int r, int total) {
    if (total % 8 != 0) return r;
    const int q = total / 8;
    return (r % q) * 8 + r / q;
}

// This block's problem, split and map_tile index under the group's XCD schedule; false for a block
// past its XCD's share.
__device__ __forceinline__ bool group_block(const GemmGroupArgs &grp, int &gi, int &split, int &tile) {
    const int x = (int)blockIdx.x & 7, j = (int)blockIdx.x >> 3;
    if (j >= grp.xn[x]) return false;
    int c = grp.xstart[x];
    while (c + 1 < grp.xstart[x + 1] && grp.chunk[c + 1].jstart <= j) ++c;
    gi = grp.chunk[c].gi;
    split = grp.chunk[c].split;
    const GemmArgs &p = grp.g[gi];
    tile = raster_pid(grp.chunk[c].t0 + (j - grp.chunk[c].jstart), p.tiles_m * p.tiles_n);
    return true;
}

int64_t cdiv(int64_t a, int64_t b) { return (a + b - 1) / b; }

// Tiles need no bounds checks when every tile (and every split's k range) is whole and aligned.
bool tiles_exact(const GemmArgs &a, int bm, int bn, int bk) {
    return a.M % bm == 0 && a.N % bn == 0 && a.K % bk == 0 && a.k_per_split % bk == 0 &&
           a.a_vec_ok && a.b_vec_ok;
}

// The group's XCD schedule (GemmGroupArgs): the blocks of every problem (tiles x splits, in call
// and split order) cut into eight equal shares, one per XCD. Returns the grid size, or 0 when the
// schedule does not fit the table (the caller then launches the calls separately).
int xcd_schedule(GemmGroupArgs &grp) {
    int64_t total = 0;
    for (int i = 0; i < grp.count; ++i) {
        const int64_t tiles = (int64_t)grp.g[i].tiles_m * grp.g[i].tiles_n;
        if (tiles > 65535 || grp.g[i].splits > 255) return 0;
        total += tiles * grp.g[i].splits;
    }
    const int64_t per = cdiv(total, 8);
    if (total == 0 || per > 65535) return 0;
    int x = 0, nch = 0;
    int64_t filled = 0;
    grp.xstart[0] = 0;
    for (int i = 0; i < grp.count; ++i) {
        const int64_t tiles = (int64_t)grp.g[i].tiles_m * grp.g[i].tiles_n;
        for (int sp = 0; sp < grp.g[i].splits; ++sp)
            for (int64_t t = 0; t < tiles;) {
                if (filled == per) {  // this XCD's share is full: the next one starts
                    if (x == 7) return 0;
                    grp.xn[x++] = (uint16_t)per;
                    grp.xstart[x] = (uint16_t)nch;
                    filled = 0;
                }
                if (nch == GROUP_CHUNKS) return 0;
                grp.chunk[nch++] = GroupChunk{(uint16_t)filled, (uint8_t)i, (uint8_t)sp, (uint16_t)t, 0};
                const int64_t take = std::min(tiles - t, per - filled);
                t += take;
                filled += take;
            }
    }
    grp.xn[x] = (uint16_t)filled;
    for (int y = x + 1; y < 8; ++y) {
        grp.xn[y] = 0;
        grp.xstart[y] = (uint16_t)nch;
    }
    grp.xstart[8] = (uint16_t)nch;
    return (int)(8 * per);
}

}  // namespace
}  // namespace it
