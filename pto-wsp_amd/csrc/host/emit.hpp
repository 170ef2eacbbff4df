// HIP source emission for one launch of a traced kernel.
#pragma once

#include <string>
#include <tuple>
#include <vector>

#include "analysis.hpp"
#include "plan.hpp"

namespace ptowsp {

// Launch-time facts a kernel is specialized on.
struct EmitSpec {
    int vec_width = 1;                 // row programs: 4, 2 or 1 floats per access
    bool row_unit_cols = false;        // row programs: full-row and column-vector params have unit column stride
    std::vector<int> indirect_count;   // per tensor ordinal: indirect index terms (in dim order)
    std::vector<int> inner_dyn_term;   // per inner loop: indirect term index of its extent, or -1
    int threads = 256;
    // Run every task of the launch in program order in one workgroup: used
    // when tasks of the grid write overlapping memory (the result then
    // depends on the reference's sequential order).
    bool serial = false;
    // Row programs: the kernel's in-kernel (P.seq) loops run inside each row's
    // lane team (the host has checked that rows do not depend on each other).
    bool row_loops = false;
    // Serial launches: the grid variables (bit v) iterated in program order
    // inside a workgroup; the others are decoded from the block index, one
    // group of tasks per workgroup.  0 means all of them.
    uint32_t seq_mask = 0;
    // The launch runs the grid tasks listed in A.tlist (ascending), not all
    // of them: a task mask from a cond on grid variables.
    bool task_list = false;
    // Row programs: cap on passes per wave iteration, and non-temporal
    // (streaming) global accesses for full-row tiles.
    int row_up = 8;
    bool nontemporal = false;
    // Tile programs: matmul ops of MFMA shape (M, N multiples of 32) on the
    // matrix cores (tile_mma) instead of the scalar loop.
    bool tile_mma = true;
    // GEMM family on MFMA (only when strides and alignment allow it).
    bool gemm = false;
    // GEMM: the grid variables along which the tasks continue one C matrix
    // downwards / to the right (-1: none); C is cut into blocks of gemm_bm x
    // gemm_bn whatever the task tiles are (gemm_edge: the last ones are not
    // whole), in rings of gemm_ring LDS stages, each holding gemm_kf task K
    // steps (consecutive ones, adjacent in A's columns and B's rows, in the
    // accumulate form).  gemm_split: parts of the K range summed by blocks of
    // their own.
    int gemm_vm = -1, gemm_vn = -1;
    int gemm_bm = 256, gemm_bn = 256, gemm_kf = 1, gemm_ring = 2, gemm_split = 1;
    bool gemm_edge = false;
    // GEMM: 256x256 blocks with K step 32 or 64 and A / B row pitches that
    // are multiples of 64 elements run as a two-group ping-pong block.
    bool gemm_pingpong = false;
    // Decode family (online softmax over pages): the in-kernel page loop of
    // every unit is split over the resident waves.
    bool decode = false;
    // Decode: the next launch (a NormInfo kernel over the same grid and o / l
    // views) is folded in; its output tensor is argument slot ntens + 1.
    bool decode_norm = false;
    // Decode: pages in each wave's register ring, and waves per block (4:
    // one per SIMD; 8: two per SIMD, 256 VGPRs each).
    int decode_ring = 4;
    int decode_waves = 4;
    bool decode_ordered = false;  // release / acquire fences around the unit completion count
    bool decode_few = false;      // bf16, more than 16 query rows: so few units that the launch uses fewer waves

    bool operator==(const EmitSpec& o) const {
        auto all = [](const EmitSpec& s) {
            return std::tie(s.vec_width, s.row_unit_cols, s.indirect_count, s.inner_dyn_term, s.threads, s.serial, s.row_loops, s.seq_mask,
                            s.task_list, s.row_up, s.nontemporal, s.tile_mma, s.gemm, s.gemm_vm, s.gemm_vn, s.gemm_bm, s.gemm_bn, s.gemm_kf,
                            s.gemm_ring, s.gemm_split, s.gemm_edge, s.gemm_pingpong, s.decode, s.decode_norm, s.decode_ring, s.decode_waves,
                            s.decode_ordered, s.decode_few);
        };
        return all(*this) == all(o);
    }
};

// Units (grid tasks) of one decode launch at most: every block holds their
// page-count prefix in LDS (DecodeSplit::kMaxUnits on the device).
constexpr int kDecodeMaxUnits = 4096;
// Scheduling cost of starting a unit, in pages (DecodeSplit::kUnitCost).
constexpr int kDecodeUnitCost = 3;

// Counters at the start of a program's launch scratch: one per decode unit,
// or per C block of a GEMM launch with split K.
constexpr int kScratchCounters = kDecodeMaxUnits;

// Waves of a GEMM block: 2 along M (1 for 32-row blocks), 4 along N for
// 256-wide and 32-row blocks, else 2.
inline int gemm_waves_n(int bm, int bn) { return bn >= 256 || (bm == 32 && bn >= 128) ? 4 : 2; }
inline int gemm_waves_m(int bm) { return bm == 32 ? 1 : 2; }

struct EmittedKernel {
    std::string source;
    std::string whole_entry;    // GEMM with K in parts: the kernel that takes K whole
    std::string entry;          // kernel symbol
    int threads = 256;
    int rows_per_chunk = 0;     // row programs: rows handled per wave iteration
    int waves_per_block = 4;
    bool row_program = false;
    int part_floats = 0;        // decode: floats per partial (m, l, o of one unit)
    int blocks_per_task = 1;    // row blocks: workgroups per task
    int tasks_per_block = 1;    // row blocks: tasks per workgroup
    size_t lds_bytes = 0;
    // Tile programs: bytes of global scratch per workgroup for the tiles that
    // do not fit in LDS (base[ntens] of the launch; the grid is capped so
    // that blocks x gtile_bytes stays bounded).
    size_t gtile_bytes = 0;
};

EmittedKernel emit_launch(const Module& m, const KernelAnalysis& a, const LaunchSpec& L, const EmitSpec& spec);

// A chain of launches over the same grid whose rows are independent, run as
// one kernel.  Params that are the same view share a slot: what one launch
// stores, the next reads from registers.  With matmuls the chain runs as row
// blocks (RowBlockInfo, emit_rowblock), without as a row program
// (emit_rowchain), whose launches may also loop, each `loop` times: over
// their in-kernel loop, or over an innermost grid variable of their own.
struct RowChain {
    struct Seg {
        const KernelAnalysis* a = nullptr;
        std::vector<int> slot;  // tensor ordinal -> slot
        int scal0 = 0;          // its first scalar argument
        bool loops = false;
    };
    struct Slot {
        DType dtype = DType::F32;
        bool vec = false;        // unit columns, 16-byte aligned rows
        bool moves = false;      // the loop moves it (coef[slot][ng])
        bool written = false;
        bool uniform = false;    // all tasks read the same tile
        int stage_mode = 0;      // how rv_stage reads it as a right operand
    };
    std::vector<Seg> segs;
    std::vector<Slot> slots;
    int ng = 0;                      // grid loop variables
    int loop = 1;
    int vec_width = 1;               // row program: as EmitSpec
    bool unit_cols = false, nontemporal = false;
    bool late = false;               // row blocks: right operands after the first are staged when they are used
};

// Emits the kernel of a chain; false when its values need more registers, or
// its right operands more LDS, than a wave or workgroup has to give, or its
// body more code than the instruction cache holds.
bool emit_rowblock(const RowChain& c, EmittedKernel& ek);
bool emit_rowchain(const RowChain& c, EmittedKernel& ek);

// Parameters of the row-program layout for a row of `cols` floats with
// accesses `vw` wide: lanes per row G, chunks per lane NV, unrolled passes UP.
struct RowLayout {
    int vw = 1, g = 1, nv = 1, up = 1;
    bool masked = false;  // the team's last chunks reach past the row's end
};
// unit_cols: every full-row access has unit column stride, so that accesses
// of 4 elements, aligned to one, may be used where the width is not even.
RowLayout row_layout(int cols, int vw, int up_cap = 8, bool unit_cols = false);

}  // namespace ptowsp
