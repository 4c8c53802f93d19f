// forage_batch.hpp -- the batch object behind the opaque abm_forage_batch handle.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <atomic>
#include <mutex>
#include <vector>

#include "../../include/abm_amd.h"

// Replicas updated over the whole GPU, their 64-agent chunks, largest field and
// words of twisted generator keys, and the scratch of their launches on the null
// stream (and the lists that every scratch shares): allocated when a path first
// needs it and then kept while the batch lives, since a captured step keeps its
// address.
struct WidePlan {
    std::vector<int32_t> reps;
    int32_t chunks = 0, max_rays = 0;
    int64_t keys = 0;
    void* mem = nullptr;
    bool clean = false;                // its cue counts are 0 (each step leaves them so)
};

// Scratch of a plan's steps elsewhere than on the null stream: one for all other
// streams (capture 0), and one for the steps that a capture of a stream records,
// whose graph may run beside any other call.
struct WideScratch {
    int plan = 0;
    unsigned long long capture = 0;
    hipStream_t stream = nullptr;
    void* mem = nullptr;
    bool clean = false;                // as WidePlan's
    WideScratch* next = nullptr;
};

// Replicas that one kernel takes, a workgroup each: order_dev[first, first + count).
struct ForageClass {
    int32_t first = 0, count = 0, max_agents = 0, max_rays = 0;
};

struct abm_forage_batch {
    int32_t n_replicas = 0;
    int32_t n_agents_total = 0;
    int64_t field_words = 0;
    int32_t max_agents = 0;
    int32_t max_rays = 0;
    int device = 0;
    int cus = 0;                       // compute units of the device
    void* reps_dev = nullptr;
    void* order_dev = nullptr;         // the classes' replicas by descending cost, fixed at creation
    int32_t* agent_offset_host = nullptr;
    int64_t* field_offset_host = nullptr;
    // Replicas that fit one workgroup's LDS: those without visual exclusion,
    // which the update kernel takes, the ones of them that the launches over
    // the whole GPU cannot take (rays), and those with it, which the occlude
    // kernel or the step kernel takes.
    ForageClass plain, narrow, occl, crowd;
    WidePlan wide[2];                  // replicas beyond that LDS; those and the plain ones but the narrow
    int32_t path = 0;                  // ABM_FORAGE_PATH_*
    std::atomic<bool> spread{false};   // the path in use takes wide[1] (and narrow in the place of plain)
    bool spread_auto = false;          // what ABM_FORAGE_PATH_AUTO takes
    // Calls may come from several threads and streams, each with its own state.
    // One at a time issues its launches; the null stream has wide[].mem to itself,
    // the other streams wait for each other's launches.
    mutable std::mutex wide_lock;
    hipEvent_t wide_done = nullptr;    // after the launches of the last call on another stream
    WideScratch* scratch = nullptr;
    int32_t n_captures = 0;
    std::vector<int32_t> rep_n, rep_r; // agents and rays of every replica
    std::vector<uint8_t> too_big;      // [b]: beyond one workgroup's LDS
    std::vector<uint8_t> exclusion;    // [b]: visual exclusion
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
