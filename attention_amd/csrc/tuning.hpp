// Process-wide tuning values of the launchers.  Each starts from an environment variable that is read once,
// when the first launcher asks; ahpc_hip_set_tuning changes it afterwards (tests use that to reach code paths
// that ordinary problem sizes would need a large GPU job for).  None of them changes results
// by more than the order in which sums are taken.
#pragma once

#include <atomic>
#include <cstdint>

namespace ahpc {

struct Tuning {
    // forward, causal: a workgroup takes a late query tile and then an early one once the launch has at least
    // this many query tiles; 0 (default) = by shape in dense launches, from 1024 tiles on in ragged ones.  The kernels that
    // share a workgroup's walk out (two walks, fp32 with 32 rows) never pair.  (AHPC_FLASH_PAIR_MIN)
    std::atomic<int64_t> flash_pair_min_tiles;
    // decode: wavefronts per workgroup, 1..8 (AHPC_DECODE_WAVES, default 0 = the launcher's choice)
    std::atomic<int64_t> decode_waves;
    // decode: tokens per context chunk when the caller passes none (AHPC_DECODE_CHUNK, default 0 = by shape)
    std::atomic<int64_t> decode_chunk;
    // decode, groups of up to 16: wavefronts that share a chunk, 1 (none), 2, 4 or 8; 0 (default) = by shape, none with decode_waves set
    // (AHPC_DECODE_SHARE)
    std::atomic<int64_t> decode_share;
    // decode: query heads per K/V head from which on the matrix-core kernels are taken where they apply (16-bit pool,
    // d > 32, pages of 16).  Default 2: timed on 8 pool heads, the page-by-page matrix-core kernel reaches 0.65-0.72
    // of 8 TB/s for groups of 2, 4 and 8 where the lane-per-element kernel reaches 0.58, 0.55 and 0.36; with one
    // query head per pool head the lane-per-element kernel stays ahead by 1-2 %.  Groups of more than 8 take
    // the matrix-core kernels whatever it says.  (AHPC_DECODE_MFMA_MIN_GROUP)
    std::atomic<int64_t> decode_matrix_min_group;
    // backward: dK and dV in one walk over the query tiles (1), in two (2), or the launcher's choice (0, the default:
    // by shape: one walk up to d = 128, two at d = 256, and for fp32 launches that leave CUs idle the kernels whose
    // workgroups own 32 rows and share the walk, which 3 asks for; 4 = one walk by two sets of wavefronts, where that exists).  (AHPC_BWD_SPLIT)
    std::atomic<int64_t> bwd_split;
    // forward with a dense mask on the matrix-core kernel: 1 (default) = the mask is packed to one bit per element in
    // front of the launch, into device memory the library keeps; 0 = the kernel reads the caller's fp32 mask in place
    // (what a stream under graph capture gets in any case).  (AHPC_MASK_PACK)
    std::atomic<int64_t> mask_pack;
    // backward, causal launches: 1 = the dQ and dK/dV workgroups take a long and a short tile of their head each (equal work
    // for all), 0 = one tile per workgroup, long tiles first, 2 (default) = by shape (bwd_pair_by_shape).  (AHPC_BWD_PAIR)
    std::atomic<int64_t> bwd_pair;
    // forward on the 16-bit matrix-core kernel: query rows per workgroup, 128 (4 wavefronts, two workgroups per CU) or
    // 256 (8 wavefronts, one workgroup per CU: one stream of K/V tiles feeds twice the rows); fp32 forward: 128, or 32 (the
    // wavefronts of a workgroup share the walk over the keys); 0 (default) = by shape.  (AHPC_FLASH_ROWS)
    std::atomic<int64_t> flash_rows;
    // forward on the 16-bit matrix-core kernel with 128 rows, no mask, d <= 128: 1 = one set of wavefronts per workgroup, 2 = two that
    // share the walk over the keys, 0 (default) = by shape.  (AHPC_FLASH_WALKS)
    std::atomic<int64_t> flash_walks;
    // KV block pool (host class): 1 (default) = slabs are address ranges that grow in place where the device has virtual
    // memory management; 0 = plain allocations that grow by reallocation and a device copy.  Read when a pool is
    // created.  (AHPC_POOL_IN_PLACE)
    std::atomic<int64_t> pool_in_place;
    Tuning();
};

Tuning& tuning();

// Thresholds of query tiles for flash_plan_launch.
constexpr int64_t kAlwaysPair = 1, kNeverPair = int64_t(1) << 40;
// The threshold of a dense launch: the tuning value when it was set, else what the launch's shape asks for.
inline int64_t pair_threshold(bool paired_by_shape) {
    const int64_t t = tuning().flash_pair_min_tiles.load();
    return t > 0 ? t : paired_by_shape ? kAlwaysPair : kNeverPair;
}
// Of a ragged batch: two rounds of two workgroups on each of 256 CUs (its own shape is not known on the host).
inline int64_t ragged_pair_threshold() {
    const int64_t t = tuning().flash_pair_min_tiles.load();
    return t > 0 ? t : 1024;
}

}  // namespace ahpc
