// Build-time tuning knobs of the fused Adam kernels (defaults = measured best on MI355X).
#ifndef PS_CONFIG_H
#define PS_CONFIG_H

#ifndef PS_BLOCK
#define PS_BLOCK 64  // threads per workgroup
#endif
#ifndef PS_LANE_ELEMS
#define PS_LANE_ELEMS 4  // elements per lane per vector step (4 or 8)
#endif
#ifndef PS_UNROLL
#define PS_UNROLL 1  // vector steps per lane per tile
#endif
#ifndef PS_MAX_WAVES_PER_EU
#define PS_MAX_WAVES_PER_EU 0  // cap on resident waves per SIMD (0: no cap; the LDS request below does the capping)
#endif
#ifndef PS_LDS_KB
#define PS_LDS_KB 17  // KiB of (unused) dynamic LDS requested per workgroup: caps resident workgroups per CU at floor(160 / PS_LDS_KB) = 9
#endif
#ifndef PS_NEAR_LDS_KB
#define PS_NEAR_LDS_KB 14  // the same for the one-launch tensor lists: 11 workgroups per CU (their waves take longer to their first load)
#endif
#ifndef PS_STREAM_LDS_KB
#define PS_STREAM_LDS_KB 14  // PS_LDS_KB of the kernels that stream past the caches: 11 workgroups per CU
#endif
#ifndef PS_STREAM_NEAR_LDS_KB
#define PS_STREAM_NEAR_LDS_KB 12  // PS_NEAR_LDS_KB of those: 13 workgroups per CU
#endif
// Launch shape of the inf/nan probe kernels (pure read streams).  Measured on 3.2 GB of fp16 payloads: single-wave
// workgroups with 8 loads per lane and 6 resident workgroups per CU read 6.85 TB/s; 256 threads x 4 loads, uncapped,
// 6.29 TB/s.
#ifndef PS_SCAN_BLOCK
#define PS_SCAN_BLOCK 64  // threads per workgroup (64 or a multiple of it)
#endif
#ifndef PS_SCAN_UNROLL
#define PS_SCAN_UNROLL 8  // 16-byte loads per lane per tile
#endif
#ifndef PS_RESIDENT_TILES
#define PS_RESIDENT_TILES 8192  // launches of up to so many workgroups of the update are not capped
#endif
#ifndef PS_SCAN_LDS_KB
#define PS_SCAN_LDS_KB 26  // KiB of unused dynamic LDS per workgroup (0: no cap on resident workgroups)
#endif
#ifndef PS_COPY_BLOCK
#define PS_COPY_BLOCK 256  // threads per workgroup of the backward-side gradient copy (64: 43 us instead of 40 for 64 Mi fp16 elements off the slot's phase)
#endif
#ifndef PS_SMALL_WAVES
#define PS_SMALL_WAVES 16  // waves of a workgroup of the step in one launch: one for the state, the others a tile each
#endif
#ifndef PS_SMALL_TILES
#define PS_SMALL_TILES 280  // longest list (256-element tiles) that is probed, stepped and rescaled in one launch
#endif
#ifndef PS_SMALL_TILES_ALONE
#define PS_SMALL_TILES_ALONE 80  // the same by one workgroup, where the caller has no scratch memory for several to share
#endif
#if PS_MAX_WAVES_PER_EU > 0
#define PS_OCCUPANCY __attribute__((amdgpu_waves_per_eu(1, PS_MAX_WAVES_PER_EU)))
#else
#define PS_OCCUPANCY
#endif

#endif  // PS_CONFIG_H
