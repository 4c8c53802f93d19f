// forage_batch.hpp -- the batch object behind the opaque abm_forage_batch handle.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <vector>

#include "../../include/abm_amd.h"

struct abm_forage_batch {
    int32_t n_replicas = 0;
    int32_t n_agents_total = 0;
    int64_t field_words = 0;
    int32_t max_agents = 0;
    int32_t max_rays = 0;
    int device = 0;
    int cus = 0;                       // compute units of the device
    void* reps_dev = nullptr;
    void* order_dev = nullptr;        // replicas by descending cost: the blocks' update order
    int32_t* agent_offset_host = nullptr;
    int64_t* field_offset_host = nullptr;
    // Replicas the update kernel takes (the first n_plain of order_dev), those
    // with visual exclusion, which the occlude kernel takes (the next n_occl) or
    // the step kernel (the next n_crowd), and the ones beyond one workgroup's
    // LDS, updated over the whole GPU.
    int32_t n_plain = 0, n_occl = 0, n_crowd = 0;
    int32_t plain_max_agents = 0, plain_max_rays = 0, occl_max_agents = 0, occl_max_rays = 0;
    int32_t crowd_max_agents = 0, crowd_max_rays = 0;
    int32_t path = 0;                  // ABM_FORAGE_PATH_*
    std::vector<int32_t> rep_n, rep_r; // agents and rays of every replica
    std::vector<int32_t> order_host;   // every replica: update kernel's, occlude kernel's, step kernel's, wide
    std::vector<uint8_t> too_big;      // [b]: beyond one workgroup's LDS
    std::vector<uint8_t> exclusion;    // [b]: visual exclusion
    std::vector<int32_t> wide;         // replicas updated over the whole GPU
    int32_t wide_chunks = 0, wide_max_rays = 0;   // their 64-agent chunks, their largest field
    int64_t wide_keys = 0;             // words of their generators' twisted keys
    void* wide_mem = nullptr;          // their map, cues, drives, counts, words, control
    int64_t wide_steps = 0;            // replica updates made that way under earlier plans
};

// The resource patches' per-replica constants and pending-placement scratch
// behind the opaque abm_forage_world handle.
struct abm_forage_world {
    abm_forage_batch* batch = nullptr;
    int32_t n_replicas = 0;
    int64_t patch_total = 0;
    size_t member_lds = 0;           // bytes of the largest replica's membership masks
    size_t world_lds = 0;            // LDS of the world kernel's workgroups
    int32_t threads = 0;             // their threads
    int32_t wide_reps = 0, wide_blocks = 0;   // replicas whose loop runs over the whole GPU, their blocks
    int64_t wide_chunks = 0;         // their 64-agent chunks
    void* wide_mem = nullptr;        // their scratch (the control words zeroed once)
    size_t collide_lds = 0;          // LDS of the collision kernel (0: no replica collides)
    void* wreps_dev = nullptr;
    int32_t* kill_rank = nullptr;    // [patch_total], -1 = not killed
    int32_t* pend = nullptr;         // [2 * n_replicas]: kind, count
    int32_t* pend_id = nullptr;      // [patch_total]
    int64_t* patch_offset_host = nullptr;
};
