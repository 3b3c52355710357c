// Records the update kernels read from device memory, and the launch geometry
// shared by host and device code.  gfx950 only.
#pragma once
#include <stddef.h>
#include <stdint.h>

#include "../../include/ramtorch_sr_adamw.h"

namespace rt {

constexpr int kThreads = 256;                       // 4 wavefronts of 64
constexpr int kVec = 8;                             // elements per lane per vector (128 bit of bf16)
constexpr int kItersPerChunk = 4;                   // vectors per lane per chunk
constexpr uint32_t kChunkElems = kThreads * kVec * kItersPerChunk;  // 8192

// One tensor (or contiguous piece of one) as the kernels see it: half a cache line.
struct alignas(16) TensorRec {
    uint64_t p, g, m, v;    // device addresses
    uint64_t numel;
    uint64_t block_base;    // elem_offset / 8: first Philox block of this piece
    uint32_t tensor_id4;    // tensor_id * 4; + {0,1,2} selects p / m / v noise
    uint32_t set_idx;       // index into the DevScalars array
    uint32_t first_piece;   // number of its first piece within the launch (see kPieceElems)
    uint32_t dtypes;        // p | g << 2 | m << 4 | v << 6 (RT_DT_*), read by the runtime-typed kernel
};
static_assert(sizeof(TensorRec) == 64, "TensorRec layout");

// What only some tensors have, in an array of its own at the same index; a table image without
// explicit noise, debug outputs and centralization has no such array.
struct alignas(16) TensorExtra {
    uint64_t np, nm, nv;        // explicit noise (uint16 per element) or 0
    uint64_t dp, dm, dv;        // optional fp32 debug outputs or 0
    uint64_t row_mean;          // fp32 row means for centralization or 0
    uint64_t row_len;
};
static_assert(sizeof(TensorExtra) == 64, "TensorExtra layout");

// rt_scalars of one param group at one step count, plus that step (Philox counter word 3).
struct alignas(16) DevScalars {
    rt_scalars s;
    uint32_t step;
    uint32_t pad[3];
};
static_assert(sizeof(DevScalars) == 64, "DevScalars layout");

// One workgroup's unit of work in the generic, runtime-typed and norm kernels: chunk `chunk`
// (kChunkElems elements) of tensor `tensor`.
struct ChunkRef {
    uint32_t tensor;
    uint32_t chunk;
};

// Fast kernel: a workgroup owns one unit of kFastUnitElems consecutive elements of one tensor.
// Which tensor is found by searching a list with one entry per tensor that has whole units: the
// index of its first unit within the launch (ascending); such tensors come first among the launch's
// records, so an entry's place is its record's.  A few hundred bytes for a transformer's parameter set,
// so the search runs out of cache, where a per-workgroup table entry would be a fresh HBM line.
// (Units of two or four chunks per workgroup were measured 1.5 % and 2.5 % slower on the 8B set.)
constexpr int kFastIters = kItersPerChunk;           // vectors per lane per fast unit
constexpr uint32_t kFastUnitElems = kThreads * kVec * kFastIters;

// Piece: at most kPieceElems consecutive elements, owned by one wavefront -- a whole short tensor, or part of
// what a tensor leaves over after its whole fast units.  A list names each piece's tensor; where in the
// tensor it lies follows from the record (piece q of the launch is number q - first_piece of those that
// begin at the last multiple of kFastUnitElems).  Every templated layout and the centralizing instance have
// pieces: as chunks of the generic kernel the leftovers cost a second launch that starts when the first
// has drained (17.7 M elements in 160 ragged fp32 tensors: 66 + 10.5 us of kernels, 66 us with pieces).
constexpr uint32_t kPieceElems = 64 * kVec;  // 512: one 128-bit vector per lane

// How much of the gradients the passes before an update leave in the memory-side cache: the part that the update reads
// first (see ldg128_keep).  A clipped step's norm and update over bf16 p, m and fp32 g, v, in us with 0 / 256 MB / 512 MB /
// everything kept: 0.24 GB of gradients 248 / 226 / 225 / 225, 0.87 GB 900 / 865 / 860 / 869, 1.7 GB 1804 / 1772 / 1761 /
// 1790, 3.5 GB 3633 / 3606 / 3591 / 3648, 7 GB 7381 / 7339 / 7311 / 7414, 32 GB 30.40 / 30.47 / 30.41 / 30.74 ms.
constexpr uint64_t kKeptBytes = 512ull << 20;

// Sets of scalars that travel as kernel arguments.  They are what changes from step to step while the tensors
// stay where they are: as part of the table they cost a copy in front of every launch (2.5 us of host time and as much
// on the GPU).  Four cover two param groups at two step counts; 64 bytes of arguments cost 0.04 us a launch.
constexpr uint32_t kArgSets = 4;

// Kernel arguments of the update kernels (passed by value).
struct LaunchArgs {
    const TensorRec* tensors;       // the launch's records; tensors with whole units first
    const TensorExtra* extras;      // same index, or NULL
    const DevScalars* sets;
    const uint32_t* first;          // first unit (row-wise kernel: first row) of each of the first n_ranges tensors, ascending
    const uint32_t* piece_tensor;   // record index of each piece
    const ChunkRef* chunks;         // generic / runtime-typed kernels
    const float* clip_coef;         // optional device float: grads are multiplied by it
    const uint32_t* skip;           // optional device flag: non-zero leaves everything untouched
    uint32_t n_ranges, n_pieces, n_piece_wgs;
    uint32_t piece_rate;            // how piece workgroups are spread over the launch, see unit_or_pieces
    uint32_t n_wgs;                 // workgroups' worth of work (units, and groups of four pieces) in the launch; see sr_adamw_link_kernel
    uint32_t seed_lo, seed_hi;
    uint32_t n_arg_sets;            // 1: every tensor of the launch uses arg_sets[0]; 2 .. kArgSets: the launch's sets; 0: they are in `sets`
    uint32_t n_rows;                // row-wise kernel: rows in the launch
    DevScalars arg_sets[kArgSets];
};

}  // namespace rt
