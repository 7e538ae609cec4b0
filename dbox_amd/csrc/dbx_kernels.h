// dbx_kernels.h -- host-callable launchers of the step kernels.
#pragma once

#include <hip/hip_runtime.h>

#include "dbx_device.h"

namespace dbx {

constexpr int kMaxBlock = 1024;

// Step kernels over the worlds order[worldOffset .. worldOffset + nworlds); lead
// selects the instantiation that profiles report for the lead (largest) tier.
struct WideBp;
// wide: the tier's worlds too big for one workgroup, whose first Collide pass
// runs over the whole device first
hipError_t launch_collide(const Dev &d, int cur, int worldOffset, int nworlds, int ldsBytes, int block, bool lead,
                          hipStream_t s, const WideBp *wide, int nwide);
size_t islands_scratch_bytes(int bodies, int contacts);
size_t solve_wave_lds_bytes(int bodies, int constraints, int levels, int islands);
hipError_t configure_kernels(int maxDynamicLds);
hipError_t launch_islands(const Dev &d, int cur, int ordered, int worldOffset, int nworlds, int ldsBytes, bool lead,
                          hipStream_t s);
// exact order: the island search of the tier's worlds too big for one workgroup
// (no joints), one island per wave
hipError_t launch_islands_wide(const Dev &d, int cur, const WideBp *wide, int nwide, hipStream_t s);
hipError_t launch_solve(const Dev &d, int cur, const StepParams &sp, int worldOffset, int nworlds, int block,
                        int ldsBytes, bool lead, hipStream_t s);
// waves: 1 to 8 per world
hipError_t launch_solve_wave(const Dev &d, int cur, const StepParams &sp, int worldOffset, int nworlds, int waves,
                             int ldsBytes, bool lead, hipStream_t s);
// exact order with kStepGrouped: the islands of the tier's big worlds (no joints)
// solved by groups of workgroups; the solve launches above skip those worlds
hipError_t launch_solve_groups(const Dev &d, int cur, const StepParams &sp, const WideBp *wide, int nwide,
                               int ldsBytes, bool lead, hipStream_t s);
// The phases named by `what` of a step of worlds that fit one workgroup (at most
// kStepBodies bodies), in one launch: what the launches above do in as many.
// ldsBytes: at least step_lds_bytes().
// Larger worlds gain little from fewer launches (a pyramid of 121 bodies: 700 us a step in
// a launch per phase, 690 in one) and more from the eight waves of their own solve.
constexpr int kStepBodies = 128;
enum : int { kStepCollide = 1, kStepSolve = 2, kStepOrdered = 4, kStepToi = 8 };
int step_lds_bytes();
hipError_t launch_step(const Dev &d, int cin, const StepParams &sp, int worldOffset, int nworlds, int ldsBytes, int what,
                       bool lead, hipStream_t s);
// a tier in which some worlds have joints, in one launch (waves as for launch_solve_wave)
hipError_t launch_solve_mixed(const Dev &d, int cur, const StepParams &sp, int worldOffset, int nworlds, int waves,
                              int ldsBytes, bool lead, hipStream_t s);
// the joint worlds [first, first + nworlds) of Dev.jointOrder, 64 to 256 threads each
// (launch_solve and launch_solve_wave skip joint worlds)
size_t solve_joint_lds_bytes(int bodies, int constraints, int joints);
hipError_t launch_solve_joint(const Dev &d, int cur, const StepParams &sp, int first, int nworlds, int threads,
                              int ldsBytes, bool lead, hipStream_t s);
size_t broadphase_scratch_bytes(int proxies);

// A world whose broadphase scratch does not fit in one workgroup's LDS: its pairs
// are found by a pass spread over the whole device (sort, sweep and pair sort in
// global memory) before k_broadphase adds them as contacts.
struct WideBp {
    int world;              // world index
    WorldDesc desc;         // its descriptor (fixture and pair ranges)
    int n;                  // proxies (fixtures)
    int P;                  // power of two >= n: sorted proxy keys
    int cap;                // the world's pair capacity
    int Pcap;               // power of two >= cap: sorted pair keys
    int nblk;               // 256-proxy blocks of the sweep count
    unsigned long long *keys; // P
    int *cur;               // n + 1 candidate offsets
    int *bsum;              // nblk block sums
    float4 *part;           // bounds partials, one per bounds workgroup
    int *ctr;               // [0] pairs found, [1] candidates, [2] sweep axis
    unsigned long long *pkeys; // Pcap
    // Collide's compaction and contact lists, and the continuous pass's lists of
    // the contacts made after Collide, over the whole device
    int nchunk;             // contact chunks of kWideCollideChunk (contact capacity)
    int2 *chunk;            // nchunk + 1: kept / touching contacts per chunk, then their offsets
    int *lcnt, *loff;       // bodyCount + 1: new contacts per body, then offsets
    int *lent;              // 2 * contact capacity: (2 * slot + side) per body
    // AddPair over the device: per pair its accept flag, per chunk of pairs the
    // accepted count, then its first contact slot
    int npchunk;            // pair chunks of kWideCollideChunk (pair capacity)
    int *pacc;              // pair capacity
    int2 *pchunk;           // npchunk + 1
    int tierFirst;          // 1 when the world is the first of its tier's launch order
};
constexpr int kWideCollideChunk = 1024;
// b.n, b.cap and b.desc set
size_t wide_scratch_bytes(const WideBp &b);
void wide_carve(WideBp &b, char *p);
hipError_t launch_broadphase(const Dev &d, int cur, int worldOffset, int nworlds, int ldsBytes, int block, bool lead,
                             hipStream_t s, const WideBp *wide = nullptr, int nwide = 0);
// b2World.SolveTOI (continuous physics) after the step's broadphase.
hipError_t launch_toi(const Dev &d, int cur, const StepParams &sp, int worldOffset, int nworlds, bool lead,
                      hipStream_t s, const WideBp *wide, int nwide);
// working memory of launch_bp_single for n proxies
size_t bp_single_scratch_bytes(int n);
hipError_t launch_bp_single(const float4 *fat, const int *moved, int n, char *scratch, int2 *out, int cap, int *total,
                            hipStream_t s);
hipError_t launch_collide_pairs(const Shape *sa, const float *xa, const Shape *sb, const float *xb, int n, float *out,
                                hipStream_t s);
hipError_t launch_max_penetration(const Dev &d, int cur, float *out, hipStream_t s);

// Read-backs and body writes through pinned host memory that the kernels write and
// read themselves; the last kernel of a read ends with host_signal (dbx_device.h).
// dbx_body_state records of the bodies [base, base + n)
hipError_t launch_read_bodies(const Dev &d, int base, int n, void *out, HostSignal sig, hipStream_t s);
// *head = the world's contact count; its dbx_contact records, newest first, when
// they fit in outBytes.  rows: an estimate of the count, for the launch's size only
hipError_t launch_read_contacts(const Dev &d, int buf, int w, int rows, int *head, void *out, size_t outBytes,
                                HostSignal sig, hipStream_t s);
// What dbx_read_events assembles its list from, one after the other behind the
// world's state in *head: the list Collide walked, the same before Collide (pre, or
// null), each solved constraint's contact slot, its contact (zero flags for a slot out
// of range), the continuous pass's log (log 0: none).  Written when they fit in outBytes.
struct EventRead {
    int walkedBuf, nowBuf, w;
    const Contact *pre;
    int solved, log; // whether constraints were solved and whether the pass's log is valid
};
__host__ __device__ inline void event_sizes(const EventRead &r, const WorldState &S, int logCap, int &walked, int &solved,
                                            int &log) {
    walked = S.collideCount;
    solved = r.solved ? S.constraints : 0;
    log = r.log ? (S.toiCallbacks < logCap ? S.toiCallbacks : logCap) : 0;
}
__host__ __device__ inline size_t event_words(const EventRead &r, int walked, int solved, int log) {
    return 20 * (size_t)walked * (r.pre ? 2 : 1) + 21 * (size_t)solved + 8 * (size_t)log;
}
hipError_t launch_read_events(const Dev &d, const EventRead &r, int rows, WorldState *head, void *out, size_t outBytes,
                              HostSignal sig, hipStream_t s);
// What dbx_sync looks at: the phase-stamp counter, the first world with an error and
// its error word, then the stamps of the steps seen .. seen + steps - 1 (the last
// kProfSlots of them)
struct SyncHead {
    unsigned long long profCount;
    int errorWorld, error; // -1: none
};
hipError_t launch_read_sync(const Dev &d, unsigned long long seen, int steps, SyncHead *head, unsigned long long *stamps,
                            HostSignal sig, hipStream_t s);
// dbx_write_bodies from n dbx_body_state records (and force / torque triples, or
// null) in pinned memory, with the fixtures' refit
hipError_t launch_write_bodies(const Dev &d, int w, int bodies, int fixtures, const void *in, const float *force3,
                               hipStream_t s);

} // namespace dbx
