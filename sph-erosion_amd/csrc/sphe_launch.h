// sphe_launch.h -- kernel launchers of sphe_kernels.hip used by the runtime.
#pragma once

#include <hip/hip_runtime.h>

#include "sphe_device.h"

// e0 / e1 (optional): profiling events that take the start of the first and
// the end of the last kernel a launcher issues.
void sphe_launch_hash(const DevState& D, hipStream_t st, hipEvent_t e0 = nullptr, hipEvent_t e1 = nullptr);
// The particle scan: counts -> cell records, the pool's claim counter reset; in
// its last launch also the terrain heights (heights), and the status word is
// cleared (first), so that no launch of it before may set a status bit.
void sphe_launch_scan_cells(const DevState& D, bool heights, bool first, hipStream_t st, hipEvent_t e0 = nullptr,
                            hipEvent_t e1 = nullptr);
// tiles of n counts at the smallest tile size (the size of the per-tile arrays)
int64_t sphe_scan_partials(int64_t n);
void sphe_launch_scatter(const DevState& D, hipStream_t st, hipEvent_t e0 = nullptr, hipEvent_t e1 = nullptr);
void sphe_launch_reorder(const DevState& D, hipStream_t st, hipEvent_t e0 = nullptr, hipEvent_t e1 = nullptr);
void sphe_launch_density(const DevState& D, int block, int remap, int lanes, hipStream_t st,
                         hipEvent_t e0 = nullptr, hipEvent_t e1 = nullptr);
void sphe_launch_force(const DevState& D, int block, int lanes, hipStream_t st, hipEvent_t e0 = nullptr,
                       hipEvent_t e1 = nullptr);
void sphe_launch_heights(const DevState& D, hipStream_t st, hipEvent_t e0 = nullptr, hipEvent_t e1 = nullptr);
void sphe_launch_two_phase(const DevState& D, hipStream_t st, hipEvent_t e0 = nullptr, hipEvent_t e1 = nullptr);
void sphe_launch_clear_status(const DevState& D, hipStream_t st);
void sphe_launch_terrain_mesh(const float* H, int nx, int nz, float cell, float ox, float oz, float* out,
                              hipStream_t st);
// The 112-byte record's values of the particle at sorted slot *slotp (device
// memory) into out[0 .. 28]; out[22] = -1 when *slotp names no slot.  lists:
// the neighbour lists are still the last step's.
void sphe_launch_inspect(const DevState& D, const int32_t* slotp, int lanes, bool lists, double* out, hipStream_t st);
// id -> slot map of the current state for those of the scenes at slots p0 ..
// p1-1 (whole scenes) that have one, entries m0 .. m1-1; unique: every entry of
// these belongs to exactly one particle.
void sphe_launch_idmap(const DevState& D, int64_t p0, int64_t p1, int32_t* map, int64_t m0, int64_t m1, bool unique,
                       hipStream_t st);
// Positions (what 0) or velocities (1) of the n particles at slots p0 ..
// p0+n-1, whose ids are 0 .. n-1, as 3 floats at out[3 id]; their last
// densities (2) as one float at out[id].
void sphe_launch_feed(const DevState& D, int64_t p0, int64_t n, int what, float* out, hipStream_t st);
// The same n floats (what 0, 1: 3 per particle) by a scene's part of the id
// map, written in order: out may be mapped host memory.
void sphe_launch_gather(const DevState& D, const int32_t* map, int64_t n, int what, float* out, hipStream_t st);
// Sorted slot of one particle id of a scene by a search over its slots.
void sphe_launch_find_id(const DevState& D, int scene, int32_t id, int32_t* slot_out, hipStream_t st);
void sphe_launch_accel(const DevState& D, int scene, int lanes, double* out, hipStream_t st);
void sphe_launch_neighbours(const DevState& D, int scene, const int64_t* off, int32_t* counts, int32_t* idx,
                            hipStream_t st);
void sphe_launch_keys(const DevState& D, int scene, int32_t* keys, hipStream_t st);
int sphe_mass_blocks();
void sphe_launch_mass(const DevState& D, int scene, double* part, double* out, hipStream_t st);
// Blocks per scene of the all-scene bookkeeping: part holds
// 3 * SPHE_MASS_BLOCKS_PER_SCENE * nscenes doubles, out 3 * nscenes (terrain
// volumes of all scenes, then their sediment, then their unit sums).
#define SPHE_MASS_BLOCKS_PER_SCENE 32
void sphe_launch_mass_scenes(const DevState& D, double* part, double* out, hipStream_t st);
// Most scenes sphe_mass_all_noalloc serves from the library's static scratch
// (3 * (SPHE_MASS_BLOCKS_PER_SCENE + 1) doubles per scene, 3.2 MiB in all).
#define SPHE_NOALLOC_MAX_SCENES 4096
// Device address of that scratch on `device`, which must be the current
// device: looked up with hipGetSymbolAddress on the first call for the
// device and kept per device.  *doubles = its size.  0, or -1 when the
// lookup failed.
int sphe_noalloc_scratch(int device, double** ptr, size_t* doubles);
void sphe_launch_copy(const void* a, void* b, int64_t n16, hipStream_t st);
