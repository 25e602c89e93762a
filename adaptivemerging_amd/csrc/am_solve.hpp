// am_solve.hpp - argument blocks and launchers of the solve-side kernels.
#pragma once

#include "am_internal.hpp"

namespace am {

// Inputs of the record set-up (b, D, mu in sweep order) and of the unpack.
struct SetupArgs {
    BodiesView B;
    ContactsView C;
    const int* n_contacts;
    const int* order;    // sweep position -> contact index
    double* rec;         // kRecDoubles per sweep position
    int* meta;           // int4 per sweep position: solve body a, solve body b, clamp, 0
    const int* pos_a;    // first solve body of the group of each sweep position
    int* sstate;         // contact state per sweep position
    double dt;
    double feedback;
    double compliance;
    double rest_val;
    double fric_val;
    int rest_ovr;
    int fric_ovr;
    int post;
    int in_collection;
    const double* lam_alt;  // unpack: odd-sweep lambda of the dataflow schedule, stride 4 (null: coloured)
    const int* scene_used = nullptr;  // unpack with lam_alt: sweeps used per scene (null: the same for all)
};

// Inputs of the persistent coloured PGS kernel.
struct PgsArgs {
    const int* colour_start;  // kMaxColours + 2 entries over sorted group positions
    const int* group_desc;    // int4 per sorted group: first, end sweep position, solve bodies A, B
    const int* meta;
    double* rec;
    int* sstate;
    double* dv;
    const double* minv;
    const double* jinv;
    const int* bflags;
    int iterations;
    int check_tolerance;      // main solve: early exit and changes
    int warm_start;           // apply confidentWarmStart first
    double tolerance;
    double omega;
    double sliding;
    double compliance;
    unsigned long long* iter_max;  // per sweep, bit pattern of max |dl|
    int* iters_used;
    unsigned* barrier;             // grid-barrier counter (zeroed before launch)
    int* error;                    // set if a barrier spin limit is hit
    // Independent scenes that stop one by one (PGS.java:190 per scene): with
    // per_scene set, a group whose scene has converged skips the remaining
    // sweeps.  Arrays are indexed by scene s; scene_max[s * iterations + t]
    // is sweep t+1's max |dl| over the scene's groups, scene_done[s *
    // (iterations + 1) + p] the scene's groups that finished pass p.
    int per_scene = 0;
    int n_scenes = 1;
    const int* g_scene = nullptr;              // scene of each sorted group
    unsigned long long* scene_max = nullptr;
    // per scene and sweep (dataflow schedule): groups done in the high 32
    // bits, those whose max |dl| was not under the tolerance in the low 32
    unsigned long long* scene_done = nullptr;
    const unsigned* scene_groups = nullptr;    // groups per scene
    int* scene_used = nullptr;                 // sweeps each scene used (written after the solve)
};

// Inputs of the dataflow PGS kernel (the same sweeps without grid barriers).
// A group's updated deltaV of each dynamic body goes to its own slot
// (kSlotDoubles doubles per incidence 2 q + side, one set per pass parity);
// the body's next update polls that slot until it is no longer empty, takes
// the value and empties the slot again.
constexpr int kSlotDoubles = 8;
constexpr unsigned long long kSlotEmpty = 0xFFF5A5A5A5A5A5A5ull;  // a signalling NaN: no arithmetic result
constexpr int kPassWords = 8;  // the pass words spread the waves' adds over this many addresses
constexpr int kPassStride = 16;  // resident kernel: arrival words are a cache line (128 B) apart

// The resident kernel: LDS doubles a workgroup can hold and steps a wave can;
// a workgroup is 4 sweeping waves and the pass keeper.
constexpr int kResidentDoubles = 4 * 4912;
constexpr int kResidentSteps = 40;
constexpr int kResidentThreads = 320;
constexpr int kResidentMaxWaves = 1024;
constexpr int kResidentMaxSweeps = 65536;

// Words behind the colour starts (kMaxColours + 2 of them), read back with them:
// the resident kernel's plan (2), whether groups are left without a colour, and
// whether some group's two solve bodies are one dynamic body.
constexpr int kWordPlan = kMaxColours + 2, kWordLeft = kMaxColours + 4, kWordOneBody = kMaxColours + 5,
              kLayoutWords = kMaxColours + 6;

struct FlowArgs {
    PgsArgs P;
    const int* flow;       // int4 per sorted group: rank_a, deg_a, rank_b, deg_b
    const int* pred;       // int2 per sorted group: incidence of the previous update of A, of B
    double* slot;          // 2 parities x 2 n_groups incidences x kSlotDoubles (all empty at launch)
    int n_groups;
    double* dv_alt;        // deltaV of odd passes (a copy of dv at launch)
    double* lam_alt;       // lambda of odd sweeps, 4 per sweep position (3 used)
    // per pass, kPassWords words (zeroed before launch): waves that have
    // finished it in the high 32 bits, those whose max |dl| was not under the
    // tolerance in the low; wave w adds to word w % kPassWords
    // (the resident kernel: the verdict word, then kPassWords arrival words per
    // sweep, kPassStride apart, counting workgroups)
    unsigned long long* pass_done;
    const int* resident_used;  // resident kernel: LDS doubles of each wave (launch_resident_plan)
    unsigned n_waves;
};

void fill_int(hipStream_t s, int* p, int n, int v);
void fill_double(hipStream_t s, double* p, int n, double v);
void fill_u64(hipStream_t s, void* p, size_t n, unsigned long long v);

// Fills and device copies that do not depend on each other, up to 12 to a
// launch: a launch costs the host about 5 us, more than any of them takes at
// the sizes of most scenes.  Sizes are multiples of 4 bytes.
class MemBatch {
public:
    static constexpr int kMax = 12;
    struct Job {
        void* dst;
        const void* src;  // null: fill
        unsigned long long value;
        size_t words;  // of 4 bytes
        unsigned end;  // first workgroup past it
    };
    struct Jobs {
        Job job[kMax];
        int n;
    };
    explicit MemBatch(hipStream_t s) : s_(s) { j_.n = 0; }
    void fill_int(int* p, size_t n, int v) { add(p, nullptr, (unsigned)v | (unsigned long long)(unsigned)v << 32, n); }
    void fill_u64(void* p, size_t n, unsigned long long v) { add(p, nullptr, v, 2 * n); }
    void copy(void* dst, const void* src, size_t bytes) { add(dst, src, 0, bytes / 4); }
    void run();

private:
    void add(void* dst, const void* src, unsigned long long v, size_t words);
    hipStream_t s_;
    Jobs j_;
};
void launch_groups(hipStream_t s, int cap, const int* n_contacts, const int* cb1, const int* cb2, const int* slot,
                   const int* parent, int* flags, int* scanned, int* group_start, int* group_a, int* group_b,
                   int* d_n_groups, void* scan_temp);
void launch_incidence(hipStream_t s, bool fill, int n_groups, const int* ga, const int* gb, const int* bflags,
                      int* inc_count, const int* inc_start, int* inc_cursor, int* inc_items);
// Colours taken at a body: those of its groups in parallel colours, and how many are in the tail
struct TakenColours {
    unsigned long long set, in_tail;
};
// colour[] and blocker[] start at -1, taken[] (by body) at 0; blocker is for
// layers, taken and rank (2 n_groups) for none.  *remaining: some group has no
// colour yet (launch again); its thread gave up after max_polls polls
constexpr int kColourPolls = 20000;  // each a memory round trip
void launch_colour(hipStream_t s, int n_groups, const int* ga, const int* gb, const int* bflags, const int* inc_start,
                   const int* inc_count, const int* inc_items, int* colour, TakenColours* taken, int* rank,
                   int* remaining, const int* layer, int* blocker, bool again, int max_polls);
// The whole layout of at most kSmallLayout groups in one workgroup: as many as
// its LDS holds.  us of a layout and its read-back, here / by the launches, for
// 300, 1,000, 2,000 and 4,096 groups of a pile (13 colours): 56 / 110, 63 / 112,
// 80 / 125, 113 / 134, the same with 1,000 and with 150,000 bodies.  Groups that
// all share one dynamic body wait for each other in turn: 230 / 362, 843 / 1,026,
// 2,245 / 1,911, 7,007 / 3,802 (no scene here has such a body; with one launch per
// round of the colouring each of its groups took a round).
// A wave that polled max_polls times gives up and sets the kWordLeft word instead
// of a layout (0 with one); nothing is laid out then.
constexpr int kSmallLayout = 4096;
constexpr int kSmallPolls = 1 << 22;  // each a few LDS round trips
struct SmallLayoutArgs {
    int n_groups, waves;  // waves: of the resident kernel (0: no plan)
    int max_polls;
    const int *ga, *gb, *bflags, *group_start, *layer;
    int *inc_count, *inc_start;  // by body
    int *colour_start, *pos_start, *order, *pos_a, *group_desc, *flow, *pred, *used;
};
void launch_layout_small(hipStream_t s, const SmallLayoutArgs& A);
void launch_colour_keys(hipStream_t s, int n_groups, const int* colour, const int* group_start, uint64_t* keys);
void launch_colour_layout(hipStream_t s, int n_groups, const uint64_t* sorted, const int* group_start,
                          const int* group_a, const int* group_b, int* colour_start, int* sizes, int* pos_start,
                          int* order, int* group_desc, int* pos_a, int* spos, int* d_total, void* scan_temp);
void launch_setup(hipStream_t s, const SetupArgs& S, int cap);
// scene of every sorted group (from its first contact's body 1) and the group count per scene
void launch_group_scene(hipStream_t s, const int* group_desc, int n_groups, const int* order, const int* cb1,
                        const am_body_desc* desc, int n_scenes, int* g_scene, unsigned* scene_groups);
// sweeps used per scene (first sweep under the tolerance, else all)
void launch_scene_finish(hipStream_t s, const PgsArgs& P);
void launch_unpack(hipStream_t s, const SetupArgs& S, int cap);
// the sweeps used, then deltaV and the contacts from the last sweep's buffers
struct FlowArgs;
void launch_flow_end(hipStream_t s, const FlowArgs& F, const SetupArgs& S, int cap, int n_dv);
int pgs_max_blocks(int block, bool* ok);
// one_body: some group's two solve bodies are the same one
hipError_t launch_pgs(hipStream_t s, const PgsArgs& P, int grid, int block, bool plain, bool one_body);
int pgs_flow_max_blocks(bool* ok);
// block 64: k_pgs_flow; kResidentThreads: the resident kernel
hipError_t launch_pgs_flow(hipStream_t s, const FlowArgs& F, int grid, int block, bool plain);
int pgs_resident_max_blocks(bool* ok);
// what `waves` resident waves would hold: used[] LDS doubles of each, plan[0]
// those of the fullest workgroup, plan[1] steps of the busiest wave
void launch_resident_plan(hipStream_t s, const int* colour_start, const int* group_desc, int waves, int* used,
                          int* plan);
void launch_flow_ranks(hipStream_t s, int n_groups, const int* bflags, const int* inc_start,
                       const int* inc_count, const int* inc_items, const int* spos, const int* group_desc,
                       int* flow, int* pred, int* one_body);
void launch_map_insert(hipStream_t s, const OldContactsView& O, int* table);
// O.first: one word for each old contact, INT_MAX before the call; match: 2 n words
void launch_warm_start(hipStream_t s, BodiesView B, ContactsView C, OldContactsView O, int n, int post, int* match,
                       int* counters);
void launch_redo_warm(hipStream_t s, ContactsView C, const int* n, int cap, int zero);
void launch_clear(hipStream_t s, BodiesView B);
void launch_gravity(hipStream_t s, BodiesView B, const int* targets, int n, double gx, double gy, double gz);
void launch_advance(hipStream_t s, BodiesView B, const int* targets, int n, double dt, bool positions);
// the listed entities' poses advanced by dt with deltaV as the velocities
void launch_advance_post(hipStream_t s, BodiesView B, const int* targets, int n, double dt);
// every entity's pose advanced by dt into xa (3 per entity) and Ra (9 per entity)
void launch_advanced_poses(hipStream_t s, BodiesView B, double dt, double* xa, double* Ra);
void launch_springs(hipStream_t s, BodiesView B, const am_spring* springs, int n, double ks, double ds);
// a force held for the next external-force pass (am_impulse_add)
struct ImpulseRec {
    int body;
    int pad;
    double p[3];
    double f[3];
};
void launch_kinematic(hipStream_t s, BodiesView B, const am_kinematic* k, int n, double t);
void launch_impulses(hipStream_t s, BodiesView B, const ImpulseRec* I, int n);
void launch_viscous(hipStream_t s, BodiesView B, const int* targets, int n, double a1, double a2);
void launch_update_jinv(hipStream_t s, BodiesView B);
void launch_metric(hipStream_t s, BodiesView B, const int* pairs, int n, double* out);

// am_detect.hip
void launch_buckets(hipStream_t s, const int* cell, int n, int* count, const int* start, int* cursor, int* items,
                    bool scatter);
void launch_contacts_set(hipStream_t s, BodiesView B, int n, const int* b1, const int* b2, const double* pw,
                         const double* nw, const double* viol, const int* info, const int* bv1, const int* bv2,
                         ContactsView C, int* overflow);

}  // namespace am
