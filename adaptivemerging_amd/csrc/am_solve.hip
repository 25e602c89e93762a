// am_solve.hip - solve groups, greedy Jones-Plassmann colouring of the
// group-body graph, the persistent coloured projected Gauss-Seidel kernel,
// the warm start, integration, gravity and the relative-motion metric.
//
// Coloured Gauss-Seidel: contacts are grouped by the pair of solve bodies they
// act on (a "group"; contacts of one body pair are contiguous in the contact
// list).  Groups that share a dynamic body get different colours.  A sweep
// runs the colours in order; inside a colour every group is independent and
// one lane processes the contacts of its group sequentially.  The result is
// bit-identical to a sequential PGS sweep (PGS.java:100-193) over the contacts
// in (colour, group, contact) order, because each contact reads and writes
// exactly the deltaV values that order would give it.
#include "am_solve.hpp"

namespace am {

// ---------------------------------------------------------------------------
// small utility kernels
__global__ void k_fill_int(int* p, int n, int v) {
    int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k < n) p[k] = v;
}
__global__ void k_fill_double(double* p, int n, double v) {
    int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k < n) p[k] = v;
}
void fill_int(hipStream_t s, int* p, int n, int v) {
    if (n > 0) hipLaunchKernelGGL(k_fill_int, dim3((n + 255) / 256), dim3(256), 0, s, p, n, v);
}
void fill_double(hipStream_t s, double* p, int n, double v) {
    if (n > 0) hipLaunchKernelGGL(k_fill_double, dim3((n + 255) / 256), dim3(256), 0, s, p, n, v);
}
__global__ void k_fill_u64(unsigned long long* p, size_t n, unsigned long long v) {
    const size_t k = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (k < n) p[k] = v;
}
void fill_u64(hipStream_t s, void* p, size_t n, unsigned long long v) {
    if (n > 0)
        hipLaunchKernelGGL(k_fill_u64, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, (unsigned long long*)p, n,
                           v);
}

constexpr unsigned kMemWords = 1024;  // of a workgroup: 16 bytes a thread
__global__ __launch_bounds__(256) void k_mem_batch(MemBatch::Jobs J) {
    int k = 0;
    unsigned first = 0;
    while (blockIdx.x >= J.job[k].end) first = J.job[k++].end;
    const MemBatch::Job& j = J.job[k];
    const size_t w0 = (size_t)(blockIdx.x - first) * kMemWords + 4 * threadIdx.x;
    unsigned* dst = (unsigned*)j.dst;
    const unsigned* src = (const unsigned*)j.src;
    const unsigned lo = (unsigned)j.value, hi = (unsigned)(j.value >> 32);
    if (w0 + 4 <= j.words && (((uintptr_t)dst | (uintptr_t)src) & 15) == 0) {
        *(uint4*)(dst + w0) = src ? *(const uint4*)(src + w0) : make_uint4(lo, hi, lo, hi);
        return;
    }
    for (size_t w = w0; w < w0 + 4 && w < j.words; w++) dst[w] = src ? src[w] : (w & 1) ? hi : lo;
}
void MemBatch::add(void* dst, const void* src, unsigned long long v, size_t words) {
    if (words == 0) return;
    if (j_.n == kMax) run();
    const unsigned first = j_.n ? j_.job[j_.n - 1].end : 0;
    j_.job[j_.n++] = Job{dst, src, v, words, first + (unsigned)((words + kMemWords - 1) / kMemWords)};
}
void MemBatch::run() {
    if (j_.n) hipLaunchKernelGGL(k_mem_batch, dim3(j_.job[j_.n - 1].end), dim3(256), 0, s_, j_);
    j_.n = 0;
}

// ---------------------------------------------------------------------------
// Groups: runs of contacts with the same unordered slot pair (solve bodies are
// the top-level entities), or with the same unordered physical body pair when
// slot and parent are null (the single sweep inside collections).
// slot == nullptr: physical body pairs (computeInCollection)
AMD_INLINE int starts_group(int k, const int* cb1, const int* cb2, const int* slot) {
    if (k == 0) return 1;
    const int a = slot ? slot[cb1[k]] : cb1[k], b = slot ? slot[cb2[k]] : cb2[k];
    const int pa = slot ? slot[cb1[k - 1]] : cb1[k - 1], pb = slot ? slot[cb2[k - 1]] : cb2[k - 1];
    return min(a, b) != min(pa, pb) || max(a, b) != max(pa, pb) ? 1 : 0;
}
struct GroupArgs {
    int cap;
    const int *n_contacts, *cb1, *cb2, *slot, *parent;
    int *flags, *scanned, *group_start, *group_a, *group_b, *d_n_groups;
};
AMD_INLINE void begin_group(const GroupArgs& A, int g, int k) {
    A.group_start[g] = k;
    const int a = A.cb1[k], b = A.cb2[k];
    if (A.group_a) A.group_a[g] = (A.parent && A.parent[a] >= 0) ? A.parent[a] : a;
    if (A.group_b) A.group_b[g] = (A.parent && A.parent[b] >= 0) ? A.parent[b] : b;
}
__global__ void k_group_flags(GroupArgs A) {
    int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k < A.cap) A.flags[k] = k < *A.n_contacts ? starts_group(k, A.cb1, A.cb2, A.slot) : 0;
}

__global__ void k_group_build(GroupArgs A) {
    int k = blockIdx.x * blockDim.x + threadIdx.x;
    int n = *A.n_contacts;
    if (k >= n) return;
    if (A.flags[k]) begin_group(A, A.scanned[k], k);
    if (k == n - 1) A.group_start[A.scanned[k] + A.flags[k]] = n;
}
// All of it by one workgroup, 4,096 contacts at a time (8 us each): one launch for three
// that take 10 us for 5,000 contacts and cost the host 5 each.
constexpr int kGroupsAtOnce = 8192;
__global__ __launch_bounds__(1024) void k_groups_small(GroupArgs A) {
    constexpr int kItems = 4;
    __shared__ int wave_sum[16];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, n = min(*A.n_contacts, A.cap);
    if (n <= 0) {
        for (int k = threadIdx.x; k < A.cap; k += blockDim.x) A.flags[k] = 0, A.scanned[k] = 0;
        if (threadIdx.x == 0) *A.d_n_groups = 0;
        return;
    }
    int before = 0;  // groups of the contacts before this turn's
    for (int k0 = 0; k0 < A.cap; k0 += 1024 * kItems) {
        const int k = k0 + threadIdx.x * kItems;
        // the pairs of the contacts from k - 1 on, loaded without a branch between them
        int a[kItems + 1], b[kItems + 1], f[kItems], sum = 0;
#pragma unroll
        for (int u = 0; u <= kItems; u++) {
            const int i = max(0, min(k + u - 1, n - 1));
            a[u] = A.cb1[i];
            b[u] = A.cb2[i];
        }
        if (A.slot)
#pragma unroll
            for (int u = 0; u <= kItems; u++) {
                a[u] = A.slot[a[u]];
                b[u] = A.slot[b[u]];
            }
#pragma unroll
        for (int u = 0; u < kItems; u++) {
            const bool same = min(a[u], b[u]) == min(a[u + 1], b[u + 1]) && max(a[u], b[u]) == max(a[u + 1], b[u + 1]);
            f[u] = k + u < n && (k + u == 0 || !same) ? 1 : 0;
            sum += f[u];
        }
        int inc = sum;
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) {
            const int v = __shfl_up(inc, o, 64);
            if (lane >= o) inc += v;
        }
        if (lane == 63) wave_sum[wave] = inc;
        __syncthreads();
        int at = before + inc - sum;
        for (int v = 0; v < 16; v++) {
            at += v < wave ? wave_sum[v] : 0;
            before += wave_sum[v];
        }
        __syncthreads();
#pragma unroll
        for (int u = 0; u < kItems; u++) {
            if (k + u >= A.cap) break;
            A.flags[k + u] = f[u];
            A.scanned[k + u] = at;
            if (f[u]) begin_group(A, at, k + u);
            at += f[u];
            if (k + u == n - 1) A.group_start[at] = n;
        }
    }
    if (threadIdx.x == 0) *A.d_n_groups = before;
}

void launch_groups(hipStream_t s, int cap, const int* n_contacts, const int* cb1, const int* cb2, const int* slot,
                   const int* parent, int* flags, int* scanned, int* group_start, int* group_a, int* group_b,
                   int* d_n_groups, void* scan_temp) {
    if (cap <= 0) return;
    const GroupArgs A{cap, n_contacts, cb1, cb2, slot, parent, flags, scanned, group_start, group_a, group_b, d_n_groups};
    if (cap <= kGroupsAtOnce) {
        hipLaunchKernelGGL(k_groups_small, dim3(1), dim3(1024), 0, s, A);
        return;
    }
    dim3 g((cap + 255) / 256), b(256);
    hipLaunchKernelGGL(k_group_flags, g, b, 0, s, A);
    exclusive_scan(s, flags, scanned, cap, d_n_groups, scan_temp);
    hipLaunchKernelGGL(k_group_build, g, b, 0, s, A);
}

// ---------------------------------------------------------------------------
// Colouring.
AMD_INLINE bool dynamic_body(const int* flags, int e) { return (flags[e] & AM_BODY_PINNED) == 0; }

// A body's list names a group once, also where both its solve bodies are that body
// (contacts given between members of one collection): ranks count groups.
__global__ void k_incidence_count(int n_groups, const int* ga, const int* gb, const int* bflags, int* inc_count) {
    int g = blockIdx.x * blockDim.x + threadIdx.x;
    if (g >= n_groups) return;
    if (dynamic_body(bflags, ga[g])) atomicAdd(&inc_count[ga[g]], 1);
    if (gb[g] != ga[g] && dynamic_body(bflags, gb[g])) atomicAdd(&inc_count[gb[g]], 1);
}
__global__ void k_incidence_fill(int n_groups, const int* ga, const int* gb, const int* bflags, const int* inc_start,
                                 int* inc_cursor, int* inc_items) {
    int g = blockIdx.x * blockDim.x + threadIdx.x;
    if (g >= n_groups) return;
    int a = ga[g], b = gb[g];
    if (dynamic_body(bflags, a)) inc_items[inc_start[a] + atomicAdd(&inc_cursor[a], 1)] = g;
    if (b != a && dynamic_body(bflags, b)) inc_items[inc_start[b] + atomicAdd(&inc_cursor[b], 1)] = g;
}

AMD_INLINE uint32_t prio(uint32_t g) {
    uint32_t h = g * 0x9E3779B1u;
    h ^= h >> 16;
    h *= 0x85EBCA6Bu;
    h ^= h >> 13;
    return h;
}
AMD_INLINE bool higher(uint32_t h, uint32_t g) {
    uint32_t ph = prio(h), pg = prio(g);
    return ph > pg || (ph == pg && h > g);
}

// Jones-Plassmann colouring: a group whose neighbours of higher priority all
// have their colours takes the smallest one unused by them.  Its neighbours of
// lower priority wait for it, so its colour follows from the priorities alone,
// whatever the order in which groups get there: there are no rounds, every
// group polls until it can be coloured.
//
// A body's groups get their colours in order of priority, so a group is ready
// when as many groups of each of its bodies have theirs as come before it there
// (its rank), and the colours to avoid are all those taken at the two bodies.
// A body's state is the set of its taken colours and the number of its groups in
// the sequential tail.  A group adds to one of the two, in one store (nobody else
// writes there until it has), so their sum is the rank only when both are final.
// priority rank of a group on a body: item(i) is the body's i-th group
template <class Item>
AMD_INLINE int colour_rank(int g, int deg, Item item) {
    constexpr int kAhead = 4;
    int rank = 0;
    for (int i0 = 0; i0 < deg; i0 += kAhead) {
        int h[kAhead];
#pragma unroll
        for (int u = 0; u < kAhead; u++) h[u] = item(min(i0 + u, deg - 1));
#pragma unroll
        for (int u = 0; u < kAhead; u++) rank += i0 + u < deg && higher((uint32_t)h[u], (uint32_t)g) ? 1 : 0;
    }
    return rank;
}
// sequential tail if all 64 parallel colours are taken
AMD_INLINE int free_colour(unsigned long long used) { return ~used != 0 ? __ffsll((long long)~used) - 1 : kMaxColours; }

// With layers (the single sweep's breadth-first layers), a group also waits
// for its neighbours of lower layers and takes a colour above all of theirs,
// so along every body the sweep visits the groups layer by layer; only
// neighbours of its own layer compete for colours.  Colours then may pass
// the parallel ones: those groups run in the sequential tail in colour order.
// A quad of lanes holds a group and goes through the lists of its two bodies 16
// neighbours at a time.  colour_of(h), item(i), layer_of(h): the colour of a
// group (negative: none yet), entry i of the bodies' lists, a group's layer.
// try_layered gives the group's colour, or -1 and the neighbour it waits for.
struct ColourLists {
    int start_a, n_a, start_b, n_b;
};
constexpr int kQuadSwap1 = 0xB1, kQuadSwap2 = 0x4E;  // quad_perm: lanes 0-1 and 2-3, then the pairs
AMD_INLINE unsigned quad_or(unsigned v) {
    v |= (unsigned)__builtin_amdgcn_mov_dpp((int)v, kQuadSwap1, 0xF, 0xF, true);
    return v | (unsigned)__builtin_amdgcn_mov_dpp((int)v, kQuadSwap2, 0xF, 0xF, true);
}
AMD_INLINE int quad_max(int v) {
    v = max(v, __builtin_amdgcn_mov_dpp(v, kQuadSwap1, 0xF, 0xF, true));
    return max(v, __builtin_amdgcn_mov_dpp(v, kQuadSwap2, 0xF, 0xF, true));
}
template <class Colour, class Item, class Layer>
AMD_INLINE int try_layered(int g, const ColourLists& b, Colour colour_of, Item item, Layer layer_of, int& blocker) {
    constexpr int kAhead = 4;
    const int lane = threadIdx.x & 3, n = b.n_a + b.n_b, lg = layer_of(g);
    int lo = 0;                   // the colour must be at least lo (above every lower-layer neighbour)
    unsigned long long used = 0;  // colours lo .. lo + 63 taken by same-layer neighbours
    for (int pass = 0; pass < 2; pass++) {
        for (int i0 = 0; i0 < n; i0 += 4 * kAhead) {
            int h[kAhead], ch[kAhead], lh[kAhead];
#pragma unroll
            for (int u = 0; u < kAhead; u++) {
                const int i = min(i0 + 4 * u + lane, n - 1);
                h[u] = item(i < b.n_a ? b.start_a + i : b.start_b + i - b.n_a);
            }
#pragma unroll
            for (int u = 0; u < kAhead; u++) {
                ch[u] = colour_of(h[u]);
                lh[u] = layer_of(h[u]);
            }
            int wait = -1;
#pragma unroll
            for (int u = 0; u < kAhead; u++) {
                if (h[u] == g) continue;
                if (pass == 0) {
                    if (lh[u] >= lg) continue;
                    if (ch[u] < 0) wait = h[u];
                    else lo = max(lo, ch[u] + 1);
                } else {
                    if (lh[u] != lg) continue;
                    if (ch[u] < 0) {
                        if (higher((uint32_t)h[u], (uint32_t)g)) wait = h[u];
                    } else if (ch[u] >= lo && ch[u] - lo < 64) {
                        used |= 1ull << (ch[u] - lo);
                    }
                }
            }
            wait = quad_max(wait);
            if (wait >= 0) {
                blocker = wait;
                return -1;
            }
        }
        lo = quad_max(lo);
    }
    used = ((unsigned long long)quad_or((unsigned)(used >> 32)) << 32) | quad_or((unsigned)used);
    return lo + free_colour(used);
}
AMD_INLINE int ld_int(const int* p) { return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }
AMD_INLINE void st_int(int* p, int v) { __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }
AMD_INLINE unsigned long long ld_u64(const unsigned long long* p) {
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
AMD_INLINE void st_u64(unsigned long long* p, unsigned long long v) {
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
// colour[] starts negative, taken[] (by body) empty.  A thread's groups are
// g, g + threads, ...; it polls those without a colour in turn, a bounded number
// of times: if some are left then (workgroups that were not resident together),
// *remaining is set and the launch is repeated.  What bounds it is the chain of
// groups each waiting for another, a link of which costs a store and the load
// that sees it (settled 20,000-box pile, 104,000 groups: 84 us; a launch per
// round of the colouring, which went through the lists again, took 1500).
// rank[2 g + side]: the group's priority rank on its body, -1 for a pinned one (or the other side's body again)
__global__ void k_colour_ranks(int n_groups, const int* ga, const int* gb, const int* bflags, const int* inc_start,
                               const int* inc_count, const int* inc_items, int* rank) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x, g = i >> 1;
    if (g >= n_groups) return;
    const int e = (i & 1) ? gb[g] : ga[g];
    int r = -1;
    if (dynamic_body(bflags, e) && !((i & 1) && e == ga[g])) {
        const int* list = &inc_items[inc_start[e]];
        r = colour_rank(g, inc_count[e], [&](int k) { return list[k]; });
    }
    rank[i] = r;
}
__global__ __launch_bounds__(256) void k_colour(int n_groups, const int* ga, const int* gb, const int* rank,
                                                int* colour, TakenColours* taken, int* remaining, int max_polls) {
    const int threads = gridDim.x * blockDim.x, first = blockIdx.x * blockDim.x + threadIdx.x;
    struct Group {
        int a, b, ra, rb;
    };
    auto load = [&](int g) { return Group{ga[g], gb[g], rank[2 * g], rank[2 * g + 1]}; };
    // true once the group has its colour
    auto attempt = [&](int g, const Group& m) {
        unsigned long long set_a = 0, set_b = 0, tail_a = 0, tail_b = 0;
        if (m.ra >= 0) {
            set_a = ld_u64(&taken[m.a].set);
            tail_a = ld_u64(&taken[m.a].in_tail);
        }
        if (m.rb >= 0) {
            set_b = ld_u64(&taken[m.b].set);
            tail_b = ld_u64(&taken[m.b].in_tail);
        }
        if ((m.ra >= 0 && __popcll(set_a) + (int)tail_a != m.ra) || (m.rb >= 0 && __popcll(set_b) + (int)tail_b != m.rb))
            return false;
        const int c = free_colour(set_a | set_b);
        colour[g] = c;
        if (c < kMaxColours) {
            if (m.ra >= 0) st_u64(&taken[m.a].set, set_a | 1ull << c);
            if (m.rb >= 0) st_u64(&taken[m.b].set, set_b | 1ull << c);
        } else {
            if (m.ra >= 0) st_u64(&taken[m.a].in_tail, tail_a + 1);
            if (m.rb >= 0) st_u64(&taken[m.b].in_tail, tail_b + 1);
        }
        return true;
    };
    // the thread's first group (its only one up to 500,000 groups) in registers
    Group m = {0, 0, -1, -1};
    bool done = first >= n_groups || colour[first] >= 0;
    if (!done) m = load(first);
    for (int polls = 0;; polls++) {
        if (!done) done = attempt(first, m);
        bool left = !done;
        for (int g = first + threads; g < n_groups; g += threads)
            if (colour[g] < 0 && !attempt(g, load(g))) left = true;
        if (!__any(left)) return;
        if (polls >= max_polls) {
            *remaining = 1;
            return;
        }
    }
}
// with layers: a quad per group, polling colour[] itself
__global__ __launch_bounds__(256) void k_colour_layered(int n_groups, const int* ga, const int* gb, const int* bflags,
                                                        const int* inc_start, const int* inc_count,
                                                        const int* inc_items, int* colour, int* remaining,
                                                        const int* layer, int* blocker, int max_polls) {
    const int quads = gridDim.x * (blockDim.x / 4), quad = (blockIdx.x * blockDim.x + threadIdx.x) / 4;
    for (int polls = 0;; polls++) {
        bool left = false;
        for (int g = quad; g < n_groups; g += quads) {
            if (ld_int(&colour[g]) >= 0) continue;
            // the neighbour that kept this group waiting keeps it waiting while it is uncoloured
            int bl = ld_int(&blocker[g]);
            int c = -1;
            if (bl < 0 || quad_max(ld_int(&colour[bl])) >= 0) {
                const int a = ga[g], b = gb[g];
                ColourLists l = {0, 0, 0, 0};
                if (dynamic_body(bflags, a)) l.start_a = inc_start[a], l.n_a = inc_count[a];
                if (dynamic_body(bflags, b)) l.start_b = inc_start[b], l.n_b = inc_count[b];
                c = try_layered(
                    g, l, [&](int h) { return ld_int(&colour[h]); }, [&](int i) { return inc_items[i]; },
                    [&](int h) { return layer[h]; }, bl);
                if (c >= 0) st_int(&colour[g], c);
                else st_int(&blocker[g], bl);
            }
            left = left || c < 0;
        }
        if (!__any(left)) return;
        if (polls >= max_polls) {
            *remaining = 1;
            return;
        }
    }
}

// Sort key of a group: colour, then (inside a parallel colour, where groups
// commute) larger groups first, then group index.  Equal-sized groups end up
// side by side, so a step of consecutive groups wastes few contact slots.
constexpr uint32_t kKeyGroupMask = 0x0FFFFFFFu;
__global__ void k_colour_keys(int n_groups, const int* colour, const int* group_start, uint64_t* keys) {
    int g = blockIdx.x * blockDim.x + threadIdx.x;
    if (g >= n_groups) return;
    const int c = colour[g];
    const uint32_t size = (uint32_t)min(group_start[g + 1] - group_start[g], 15);
    const uint32_t rank = c < kMaxColours ? 15u - size : 0u;
    keys[g] = ((uint64_t)(uint32_t)c << 32) | (rank << 28) | (uint32_t)g;
}

// colour_start[c] = first sorted position with colour >= c, c = 0..kMaxColours;
// colour_start[kMaxColours + 1] = n_groups (the tail holds every colour from
// kMaxColours on, in colour order); the words after it (kWordPlan ...) are
// cleared for the kernels that follow
__global__ void k_colour_starts(int n_groups, const uint64_t* sorted, int* colour_start) {
    int c = threadIdx.x;
    if (c > kMaxColours + 1) {
        if (c < kLayoutWords && c != kWordLeft) colour_start[c] = 0;
        return;
    }
    if (c == kMaxColours + 1) {
        colour_start[c] = n_groups;
        return;
    }
    int lo = 0, hi = n_groups;
    while (lo < hi) {
        int mid = (lo + hi) >> 1;
        if ((int)(sorted[mid] >> 32) < c) lo = mid + 1;
        else hi = mid;
    }
    colour_start[c] = lo;
}

__global__ void k_sorted_sizes(int n_groups, const uint64_t* sorted, const int* group_start, int* sizes) {
    int q = blockIdx.x * blockDim.x + threadIdx.x;
    if (q == n_groups) sizes[q] = 0;
    if (q >= n_groups) return;
    int g = (int)((uint32_t)sorted[q] & kKeyGroupMask);
    sizes[q] = group_start[g + 1] - group_start[g];
}

__global__ void k_solve_order(int n_groups, const uint64_t* sorted, const int* group_start, const int* pos_start,
                              const int* group_a, const int* group_b, int* order, int* group_desc, int* pos_a,
                              int* spos) {
    int q = blockIdx.x * blockDim.x + threadIdx.x;
    if (q >= n_groups) return;
    int g = (int)((uint32_t)sorted[q] & kKeyGroupMask);
    spos[g] = q;
    int s = group_start[g], e = group_start[g + 1], o = pos_start[q];
    for (int k = s; k < e; k++) {
        order[o + (k - s)] = k;
        pos_a[o + (k - s)] = group_a[g];
    }
    reinterpret_cast<int4*>(group_desc)[q] = make_int4(o, o + (e - s), group_a[g], group_b[g]);
}

// Dataflow ranks: for every dynamic body a with deg_a incident groups, the rank
// of each of its groups among them in sorted (colour-major) order.  flow[q] =
// {rank_a, deg_a, rank_b, deg_b} for sorted group q with solve bodies A, B
// (deg 0 for a pinned body: never waited on, never written).  pred[2 q + s]
// is the incidence (2 q' + s') of the update of that body just before this
// one: the group ranked one lower, or for rank 0 the body's last group, whose
// update of the previous pass comes first.
//
// The rank of group q on a body, and the position of the one before it (for
// rank 0 the body's last): spos_of(i) is the position of the body's i-th group.
template <class Spos>
AMD_INLINE int flow_rank(int q, int deg, Spos spos_of, int& pred) {
    constexpr int kAhead = 4;
    int rank = 0, before = -1, last = -1;
    for (int i0 = 0; i0 < deg; i0 += kAhead) {
        int qi[kAhead];
#pragma unroll
        for (int u = 0; u < kAhead; u++) qi[u] = spos_of(min(i0 + u, deg - 1));
#pragma unroll
        for (int u = 0; u < kAhead; u++) {
            if (qi[u] < q) {
                rank += i0 + u < deg ? 1 : 0;
                before = max(before, qi[u]);
            }
            last = max(last, qi[u]);
        }
    }
    pred = before >= 0 ? before : last;
    return rank;
}
// A thread per group and side: the lists are short, and the loads of several
// entries are in flight together (a thread per body, one entry at a time, took
// 193 us on the settled 20,000-box pile; this takes 17).
__global__ void k_flow_ranks(int n_groups, const int* bflags, const int* inc_start, const int* inc_count,
                             const int* inc_items, const int* spos, const int* group_desc, int* flow, int* pred,
                             int* one_body) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x, q = i >> 1, side = i & 1;
    if (q >= n_groups) return;
    const int e = group_desc[4 * q + 2 + side];
    int rank = 0, deg = 0, before = 0;
    if (dynamic_body(bflags, e)) {
        const int start = inc_start[e];
        deg = inc_count[e];
        int of;
        rank = flow_rank(q, deg, [&](int k) { return spos[inc_items[start + k]]; }, of);
        before = 2 * of + (group_desc[4 * of + 2] == e ? 0 : 1);
        if (side && e == group_desc[4 * q + 2]) *one_body = 1;
    }
    reinterpret_cast<int2*>(flow)[i] = make_int2(rank, deg);
    pred[i] = before;
}

void launch_flow_ranks(hipStream_t s, int n_groups, const int* bflags, const int* inc_start, const int* inc_count,
                       const int* inc_items, const int* spos, const int* group_desc, int* flow, int* pred,
                       int* one_body) {
    if (n_groups > 0)
        hipLaunchKernelGGL(k_flow_ranks, dim3((2 * n_groups + 255) / 256), dim3(256), 0, s, n_groups, bflags, inc_start,
                           inc_count, inc_items, spos, group_desc, flow, pred, one_body);
}

// The division (D lambda - omega (b + J.dv)) / (D + C) of a row.  The
// denominator is fixed during a solve, so the denominator-only half of the
// hardware division sequence (reciprocal estimate and two Newton steps) is
// done once per row in setup; per sweep the quotient is then q0 = n y,
// r = fma(-d, q0, n), q = fma(r, y, q0), the same operations the sequence
// performs when v_div_scale leaves its operands unscaled and v_div_fixup has
// nothing to fix.  Both |n| and |d| in [2^-250, 2^250] guarantees that (no
// exponent gap near 768, no denormal quotient or reciprocal, nonzero finite
// operands); anything else takes the full division.  The result is the
// correctly rounded quotient either way.
AMD_INLINE double div_recip(double den) {
    const double a = fabs(den);
    if (!(a >= 0x1p-250 && a <= 0x1p250)) return 0.0;  // 0: always divide
    double y = __builtin_amdgcn_rcp(den);
    double e = __builtin_fma(-den, y, 1.0);
    y = __builtin_fma(y, e, y);
    e = __builtin_fma(-den, y, 1.0);
    return __builtin_fma(y, e, y);
}
AMD_INLINE double div_row(double num, double den, double y) {
    const double a = fabs(num);
    const bool fast = y != 0.0 && a >= 0x1p-250 && a <= 0x1p250;
    const double q0 = num * y;
    const double r = __builtin_fma(-den, q0, num);
    double q = __builtin_fma(r, y, q0);
    if (__builtin_expect(!__all(fast), 0)) {
        if (!fast) q = num / den;
    }
    return q;
}

// ---------------------------------------------------------------------------
// Per-contact solve records in sweep order (Contact.computeB,
// Contact.computeJMinvJt, the friction rule of PGS.java:128-142).
AMD_INLINE double contact_mu(const am_body_desc& d1, const am_body_desc& d2, int fovr, double fval) {
    if (fovr) return fval;
    double f1 = d1.friction, f2 = d2.friction;
    if (f1 < 0.2 || f2 < 0.2) return jmin(f1, f2);
    if (f1 > 1. || f2 > 1.) return jmax(f1, f2);
    return (f1 + f2) / 2.;
}

__global__ void k_setup(SetupArgs S) {
    int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= *S.n_contacts) return;
    const BodiesView& B = S.B;
    const ContactsView& C = S.C;
    int c = S.order[k];
    int b1 = C.b1[c], b2 = C.b2[c];
    int a = (B.parent[b1] >= 0 && !S.in_collection) ? B.parent[b1] : b1;
    int b = (B.parent[b2] >= 0 && !S.in_collection) ? B.parent[b2] : b2;
    double* J = &C.J[(size_t)c * 36];
    // CollisionProcessor.updateJacobiansThatNeedUpdating (:326-334): contacts
    // touching a collection rebuild the world frame from body-1 coordinates.
    if (B.parent[b1] >= 0 || B.parent[b2] >= 0) {
        m33 R = ldm(&B.R[b1 * 9]);
        d3 x = ld3(&B.x[b1 * 3]);
        d3 pW = xform(R, x, ld3(&C.pB1[c * 3]));
        d3 nW = mul(R, ld3(&C.nB1[c * 3]));
        d3 t1 = mul(R, ld3(&C.t1B1[c * 3]));
        d3 t2 = mul(R, ld3(&C.t2B1[c * 3]));
        d3 r1 = sub(pW, ld3(&B.x[a * 3]));
        d3 r2 = sub(pW, ld3(&B.x[b * 3]));
        const d3 dirs[3] = {nW, t1, t2};
#pragma unroll
        for (int row = 0; row < 3; row++) {
            d3 d = dirs[row];
            st3(J + row * 12 + 0, mk(-1.0 * d.x, -1.0 * d.y, -1.0 * d.z));
            st3(J + row * 12 + 3, cross(d, r1));
            st3(J + row * 12 + 6, d);
            st3(J + row * 12 + 9, cross(r2, d));
        }
    }
    double Jr[36];
#pragma unroll
    for (int i = 0; i < 36; i++) Jr[i] = J[i];
    // b (Contact.computeB, Contact.java:279-326)
    double bn = 0, bt1 = 0, bt2 = 0;
    if (S.post) {
        bn = S.feedback * C.viol[c];
        bt1 = 0.;
        bt2 = 0.;
    } else {
        double restitution = (B.desc[b1].restitution + B.desc[b2].restitution) / 2.;
        if (S.rest_ovr) restitution = S.rest_val;
        const int ids[2] = {a, b};
#pragma unroll
        for (int s = 0; s < 2; s++) {
            int e = ids[s];
            const double* Jn = Jr + 0 + s * 6;
            const double* Jt1 = Jr + 12 + s * 6;
            const double* Jt2 = Jr + 24 + s * 6;
            double sc = B.minv[e] * S.dt;
            d3 tmp = scale_add(sc, ld3(&B.f[e * 3]), ld3(&B.v[e * 3]));
            bn += dot(tmp, ld3(Jn));
            bt1 += dot(tmp, ld3(Jt1));
            bt2 += dot(tmp, ld3(Jt2));
            tmp = mul(ldm(&B.jinv[e * 9]), ld3(&B.t[e * 3]));
            tmp = mk(tmp.x * S.dt, tmp.y * S.dt, tmp.z * S.dt);
            tmp = add(tmp, ld3(&B.w[e * 3]));
            bn += dot(tmp, ld3(Jn + 3));
            bt1 += dot(tmp, ld3(Jt1 + 3));
            bt2 += dot(tmp, ld3(Jt2 + 3));
            double bounce = dot(ld3(&B.v[e * 3]), ld3(Jn)) + dot(ld3(&B.w[e * 3]), ld3(Jn + 3));
            bounce *= restitution;
            bn += bounce;
        }
        bn += S.feedback * C.viol[c];
    }
    // D (Contact.computeJMinvJt, Contact.java:340-354); the jinv products are
    // kept for the sweep's deltaV updates (PGS.updateDeltaVwithLambdai).
    m33 ja_inv = ldm(&B.jinv[a * 9]);
    m33 jb_inv = ldm(&B.jinv[b * 9]);
    double D[3];
    d3 ta[3], tb[3];
#pragma unroll
    for (int row = 0; row < 3; row++) {
        const double* ja = Jr + row * 12;
        const double* jb = Jr + row * 12 + 6;
        ta[row] = mul(ja_inv, ld3(ja + 3));
        tb[row] = mul(jb_inv, ld3(jb + 3));
        D[row] = B.minv[a] * dot(ld3(ja), ld3(ja)) + dot(ld3(ja + 3), ta[row]) + B.minv[b] * dot(ld3(jb), ld3(jb)) +
                 dot(ld3(jb + 3), tb[row]);
    }
    // Records are oriented so that their first body is the group's first
    // body A; a contact listed the other way round stores jb.w, ja.v (= -jb.v
    // exactly), ja.w and the swapped jinv products.  Every product of the
    // update is unchanged and J.dv only swaps its two (commuting) halves, so
    // the sweep stays bit-exact without swapping body registers per contact.
    const bool flip = a != S.pos_a[k];
    double* rec = &S.rec[(size_t)k * kRecDoubles];
#pragma unroll
    for (int row = 0; row < 3; row++) {
        const double* J0 = Jr + row * 12;
        double* q = rec + row * kRecRow;
        if (!flip) {
            st3(q + kRecBv, ld3(J0 + 6));
            st3(q + kRecAw, ld3(J0 + 3));
            st3(q + kRecBw, ld3(J0 + 9));
            st3(q + kRecTa, ta[row]);
            st3(q + kRecTb, tb[row]);
        } else {
            st3(q + kRecBv, ld3(J0 + 0));  // ja.v = -jb.v
            st3(q + kRecAw, ld3(J0 + 9));
            st3(q + kRecBw, ld3(J0 + 3));
            st3(q + kRecTa, tb[row]);
            st3(q + kRecTb, ta[row]);
        }
    }
    const int ea = flip ? b : a, eb = flip ? a : b;
    const double bs[3] = {bn, bt1, bt2};
    rec[kRecMu] = contact_mu(B.desc[b1], B.desc[b2], S.fric_ovr, S.fric_val);
#pragma unroll
    for (int r = 0; r < 3; r++) rec[kRecLambda + r] = C.lam[c * 3 + r];
    bool clamp = !(B.flags[b1] & AM_BODY_MAGNET_ACTIVE) && !(B.flags[b2] & AM_BODY_MAGNET_ACTIVE);
    rec[kRecAB] = __longlong_as_double((long long)(((uint64_t)(uint32_t)eb << 32) | (uint32_t)ea));
    bool recips = true;
#pragma unroll
    for (int r = 0; r < 3; r++) {
        double* q = rec + r * kRecRow;
        const double den = D[r] + S.compliance, y = div_recip(den);
        q[kRecB] = bs[r];
        q[kRecD] = D[r];
        q[kRecDen] = den;
        q[kRecY] = y;
        recips = recips && y != 0.0;
    }
    // 0: not clamped; 1: clamped, every row's reciprocal stored (the
    // dataflow kernel's fast update may take it); 2: clamped otherwise
    rec[kRecClamp] = !clamp ? 0.0 : recips ? 1.0 : 2.0;
    rec[kRecDoubles - 1] = 0.0;
    reinterpret_cast<int4*>(S.meta)[k] = make_int4(ea, eb, clamp ? 1 : 0, 0);
    S.sstate[k] = C.state[c];
}

void launch_setup(hipStream_t s, const SetupArgs& S, int cap) {
    if (cap <= 0) return;
    hipLaunchKernelGGL(k_setup, dim3((cap + 127) / 128), dim3(128), 0, s, S);
}

// Results back to list order.
AMD_INLINE void unpack(const SetupArgs& S, int k, int iters_used) {
    int c = S.order[k];
    double* rec = &S.rec[(size_t)k * kRecDoubles];
    ContactsView C = S.C;
    const int used = S.scene_used ? S.scene_used[S.B.desc[S.C.b1[c]].scene] : iters_used;
    if (S.lam_alt && (used & 1)) {
        // dataflow schedule: an odd last sweep left lambda in the odd-sweep buffer
#pragma unroll
        for (int r = 0; r < 3; r++) rec[kRecLambda + r] = S.lam_alt[4 * k + r];
    }
#pragma unroll
    for (int r = 0; r < 3; r++) {
        C.lam[c * 3 + r] = rec[kRecLambda + r];
        C.b[c * 3 + r] = rec[r * kRecRow + kRecB];
        C.D[c * 3 + r] = rec[r * kRecRow + kRecD];
    }
    C.state[c] = S.sstate[k];
}
__global__ void k_unpack(SetupArgs S) {
    int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k < *S.n_contacts) unpack(S, k, 0);  // the coloured schedule has one buffer
}

void launch_unpack(hipStream_t s, const SetupArgs& S, int cap) {
    if (cap <= 0) return;
    hipLaunchKernelGGL(k_unpack, dim3((cap + 255) / 256), dim3(256), 0, s, S);
}

// ---------------------------------------------------------------------------
// The sweep.
struct BodyRegs {
    double dv[6];
    double minv;
    bool dyn;
};

// deltaV crosses workgroups between colours: it is read and written with
// agent-scope relaxed atomics (coherent at device level, global_load/store
// ... sc1), so the barrier needs no L2 write-back or invalidation and the
// read-only contact records stay resident in each XCD's L2 across sweeps.
AMD_INLINE double ld_coherent(const double* p) {
    return __hip_atomic_load(const_cast<double*>(p), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
AMD_INLINE void st_coherent(double* p, double v) { __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }

AMD_INLINE void load_body(const PgsArgs& P, int e, BodyRegs& r) {
#pragma unroll
    for (int i = 0; i < 6; i++) r.dv[i] = ld_coherent(&P.dv[e * 6 + i]);
    r.minv = P.minv[e];
    r.dyn = (P.bflags[e] & AM_BODY_PINNED) == 0;
}
AMD_INLINE void store_body(const PgsArgs& P, int e, const BodyRegs& r) {
    if (!r.dyn) return;
#pragma unroll
    for (int i = 0; i < 6; i++) st_coherent(&P.dv[e * 6 + i], r.dv[i]);
}

// One row of a contact record: aw = ja.w, bv = jb.v (ja.v = -jb.v),
// bw = jb.w, ta = jinv_a ja.w, tb = jinv_b jb.w.
struct Row {
    d3 aw, bv, bw, ta, tb;
};
AMD_INLINE Row row_of(const double* rec, int r) {
    const double* q = rec + r * kRecRow;
    return Row{ld3(q + kRecAw), ld3(q + kRecBv), ld3(q + kRecBw), ld3(q + kRecTa), ld3(q + kRecTb)};
}

// PGS.updateDeltaVwithLambdai (PGS.java:221-245).  one: both sides are the same
// body, whose deltaV takes A's half first, then B's.
AMD_INLINE void apply_row(const Row& R, double lambda, BodyRegs& A, BodyRegs& Bb, bool one) {
    double s1 = A.minv * lambda;
    A.dv[0] = s1 * -R.bv.x + A.dv[0];
    A.dv[1] = s1 * -R.bv.y + A.dv[1];
    A.dv[2] = s1 * -R.bv.z + A.dv[2];
    A.dv[3] = lambda * R.ta.x + A.dv[3];
    A.dv[4] = lambda * R.ta.y + A.dv[4];
    A.dv[5] = lambda * R.ta.z + A.dv[5];
    if (one)
#pragma unroll
        for (int i = 0; i < 6; i++) Bb.dv[i] = A.dv[i];
    double s2 = Bb.minv * lambda;
    Bb.dv[0] = s2 * R.bv.x + Bb.dv[0];
    Bb.dv[1] = s2 * R.bv.y + Bb.dv[1];
    Bb.dv[2] = s2 * R.bv.z + Bb.dv[2];
    Bb.dv[3] = lambda * R.tb.x + Bb.dv[3];
    Bb.dv[4] = lambda * R.tb.y + Bb.dv[4];
    Bb.dv[5] = lambda * R.tb.z + Bb.dv[5];
    if (one)
#pragma unroll
        for (int i = 0; i < 6; i++) A.dv[i] = Bb.dv[i];
}
// Contact.getJdv (Contact.java:362-378)
AMD_INLINE double jdv(const Row& R, const BodyRegs& A, const BodyRegs& Bb) {
    double da = (-R.bv.x * A.dv[0] + -R.bv.y * A.dv[1] + -R.bv.z * A.dv[2]) +
                (R.aw.x * A.dv[3] + R.aw.y * A.dv[4] + R.aw.z * A.dv[5]);
    double db = (R.bv.x * Bb.dv[0] + R.bv.y * Bb.dv[1] + R.bv.z * Bb.dv[2]) +
                (R.bw.x * Bb.dv[3] + R.bw.y * Bb.dv[4] + R.bw.z * Bb.dv[5]);
    return da + db;
}

constexpr int kRec2 = kRecDoubles / 2;  // 16-byte words per record
struct Rec {
    double v[kRecDoubles];
};
AMD_INLINE void load_rec(const double2* src, Rec& r) {
#pragma unroll
    for (int i = 0; i < kRec2; i++) {
        double2 t = src[i];
        r.v[2 * i] = t.x;
        r.v[2 * i + 1] = t.y;
    }
}

// One group (the contacts of one body pair): mode 0 is confidentWarmStart
// (PGS.java:250-256), mode 1 one PGS pass (PGS.java:100-184).  recs points at
// the group's first record; lambda and the contact state are written back at
// sweep position k.  kOneBody: groups may have one body on both sides.
template <bool kOneBody>
AMD_INLINE void process_group(const PgsArgs& P, int4 gd, const double2* recs, int mode, bool last_iter, double& mx) {
    const int k0 = gd.x, k1 = gd.y, A = gd.z, Bi = gd.w;
    BodyRegs ra, rb;
    load_body(P, A, ra);
    load_body(P, Bi, rb);
    const bool one = kOneBody && A == Bi;
    bool nan = false;
    for (int k = k0; k < k1; k++) {
        Rec cur;
        load_rec(recs + (size_t)(k - k0) * kRec2, cur);
        const double* rec = cur.v;
        double lam[3] = {rec[kRecLambda + 0], rec[kRecLambda + 1], rec[kRecLambda + 2]};
        if (mode == 0) {
#pragma unroll
            for (int r = 0; r < 3; r++) apply_row(row_of(rec, r), lam[r], ra, rb, one);
        } else {
            const bool clamp = rec[kRecClamp] != 0.0;
            const double mu = rec[kRecMu];
            const double omega = P.omega;
#pragma unroll
            for (int r = 0; r < 3; r++) {
                Row R = row_of(rec, r);
                double Jd = jdv(R, ra, rb);
                double prev = lam[r];
                double Dr = rec[r * kRecRow + kRecD];
                double l = (Dr * lam[r] - omega * (rec[r * kRecRow + kRecB] + Jd)) / (Dr + P.compliance);
                if (clamp) {
                    if (r == 0) {
                        l = jmax(0, l);
                    } else {
                        double limit = mu * lam[0];
                        l = jmax(l, -limit);
                        l = jmin(l, limit);
                    }
                }
                lam[r] = l;
                double diff = l - prev;
                apply_row(R, diff, ra, rb, one);
                // Math.max over |diff| (PGS.java:125); a NaN is carried separately
                mx = fmax(mx, fabs(diff));
                nan = nan || diff != diff;
            }
            double* dst = &P.rec[(size_t)k * kRecDoubles + kRecLambda];
            dst[0] = lam[0];
            dst[1] = lam[1];
            dst[2] = lam[2];
            if (last_iter) {
                // Contact.updateContactState (Contact.java:385-398)
                double w1 = rec[kRecRow + kRecB] + jdv(row_of(rec, 1), ra, rb);
                double w2 = rec[2 * kRecRow + kRecB] + jdv(row_of(rec, 2), ra, rb);
                int st;
                if (fabs(lam[0]) <= 1e-14) st = AM_STATE_BROKEN;
                else if (fabs(w1) > P.sliding) st = AM_STATE_ONEDGE;
                else if (fabs(w2) > P.sliding) st = AM_STATE_ONEDGE;
                else st = AM_STATE_CLEAR;
                P.sstate[k] = st;
            }
        }
    }
    if (nan) mx = __longlong_as_double(0x7ff8000000000000ll);
    store_body(P, A, ra);
    store_body(P, Bi, rb);
}

AMD_INLINE double wave_max(double v) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v = jmax(v, __shfl_xor(v, o, 64));
    return v;
}

// Grid barrier for a co-resident (cooperatively launched) grid.  The caller
// has already waited for its deltaV stores (s_waitcnt) and passed a workgroup
// barrier, so lane 0 arrives on a monotonically increasing counter right
// away and spins on a coherent load until all blocks of this instance have
// arrived.  A spin limit turns a barrier that cannot complete into an error
// flag.
template <bool kSingleBlock>
AMD_INLINE bool grid_barrier(const PgsArgs& P, unsigned& epoch) {
    if (kSingleBlock) return true;
    __shared__ int bail;
    epoch += gridDim.x;
    if (threadIdx.x == 0) {
        bail = 0;
        __hip_atomic_fetch_add(P.barrier, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        long spins = 0;
        while (__hip_atomic_load(P.barrier, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) < epoch) {
            if (++spins > 20000000L) {
                atomicOr(P.error, 1);
                bail = 1;
                break;
            }
            // another workgroup gave up: leave now instead of at our own limit
            if ((spins & 1023) == 0 && __hip_atomic_load(P.error, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT))
                break;
            __builtin_amdgcn_s_sleep(1);
        }
        if (__hip_atomic_load(P.error, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) bail = 1;
    }
    __syncthreads();
    return bail == 0;
}

// Persistent kernel: warm-start pass then up to `iterations` sweeps; one grid
// barrier per non-empty colour.  Groups of a colour are dealt block-cyclically
// (group j of the colour goes to block j % grid, lane j / grid) so every
// workgroup, hence every CU in use, gets a share.  The per-sweep max |delta
// lambda| is reduced with an integer atomic max on the bit pattern (non-
// negative doubles order as their bits) into a slot per sweep.  kOneBody: for
// contact sets where some group's two solve bodies are the same one (contacts
// given between members of one collection).  Only this kernel knows such groups:
// a thread holds both sides, where the dataflow kernels' lanes keep a deltaV each.
template <bool kSingleBlock, bool kOneBody>
__global__ __launch_bounds__(256) void k_pgs(PgsArgs P) {
    const int* cs = P.colour_start;
    const int slot0 = threadIdx.x * gridDim.x + blockIdx.x;
    const int stride = gridDim.x * blockDim.x;
    const int4* gdesc = reinterpret_cast<const int4*>(P.group_desc);
    const double2* grec = reinterpret_cast<const double2*>(P.rec);
    __shared__ int s_cols[kMaxColours];
    __shared__ int s_ncols;
    if (threadIdx.x == 0) {
        int nc = 0;
        for (int c = 0; c < kMaxColours; c++)
            if (cs[c + 1] > cs[c]) s_cols[nc++] = c;
        s_ncols = nc;
    }
    __syncthreads();
    const int ncols = s_ncols;
    const bool has_tail = cs[kMaxColours + 1] > cs[kMaxColours];
    const bool lane0 = blockIdx.x == 0 && threadIdx.x == 0;
    unsigned epoch = 0;
    // this lane's first group of the next colour: its descriptor does not
    // depend on other workgroups, so it is read before the barrier
    int4 head = make_int4(0, 0, 0, 0);
    bool have = false;
    auto prefetch = [&](int ci) {
        const int c = s_cols[ci];
        const int q = cs[c] + slot0;
        have = q < cs[c + 1];
        if (have) head = gdesc[q];
    };
    int it = 0;
    // one group; with per-scene exits a sweep skips the groups of a scene
    // whose previous sweep was under the tolerance (that sweep is final
    // after the grid barrier), and each group's max goes to its scene too
    auto run_group = [&](int q, int4 gd, int mode, bool last, double& mx) {
        if (!P.per_scene || mode == 0) {
            process_group<kOneBody>(P, gd, grec + (size_t)gd.x * kRec2, mode, last, mx);
            return;
        }
        const int sc = P.g_scene[q];
        if (it > 0) {
            const double prev = __longlong_as_double((long long)__hip_atomic_load(
                &P.scene_max[(size_t)sc * P.iterations + it - 1], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
            if (prev < P.tolerance) return;
        }
        double gmx = 0.0;
        process_group<kOneBody>(P, gd, grec + (size_t)gd.x * kRec2, mode, last, gmx);
        if (!(gmx <= 0))
            atomicMax(&P.scene_max[(size_t)sc * P.iterations + it], (unsigned long long)__double_as_longlong(gmx));
        mx = gmx != gmx ? gmx : fmax(mx, gmx);
    };
    auto run_colour = [&](int ci, int mode, bool last, double& mx) {
        const int c = s_cols[ci];
        if (have) run_group(cs[c] + slot0, head, mode, last, mx);
        for (int q = cs[c] + slot0 + stride; q < cs[c + 1]; q += stride) run_group(q, gdesc[q], mode, last, mx);
    };
    auto run_tail = [&](int mode, bool last, double& mx) {
        if (lane0)
            for (int q = cs[kMaxColours]; q < cs[kMaxColours + 1]; q++) run_group(q, gdesc[q], mode, last, mx);
    };
    // Ends a colour: wait for this lane's deltaV stores, read the next
    // colour's descriptor, meet the other workgroups.
    auto next = [&](int ci_next) -> bool {
        __builtin_amdgcn_s_waitcnt(0);
        if (ci_next >= 0) prefetch(ci_next);
        __syncthreads();
        return grid_barrier<kSingleBlock>(P, epoch);
    };

    if (ncols > 0) prefetch(0);
    const int first_after_tail = ncols > 0 ? 0 : -1;
    if (P.warm_start) {
        double dummy = 0;
        for (int ci = 0; ci < ncols; ci++) {
            run_colour(ci, 0, false, dummy);
            const int nx = ci + 1 < ncols ? ci + 1 : (has_tail ? -1 : first_after_tail);
            if (!next(nx)) return;
        }
        if (has_tail) {
            run_tail(0, false, dummy);
            if (!next(first_after_tail)) return;
        }
    }
    for (; it < P.iterations; it++) {
        const bool last = (it == P.iterations - 1);
        double mx = 0;
        for (int ci = 0; ci < ncols; ci++) {
            run_colour(ci, 1, last, mx);
            if (ci == ncols - 1 && !has_tail) {
                double wm = wave_max(mx);
                if ((threadIdx.x & 63) == 0 && !(wm <= 0))
                    atomicMax(&P.iter_max[it], (unsigned long long)__double_as_longlong(wm));
            }
            const int nx = ci + 1 < ncols ? ci + 1 : (has_tail ? -1 : first_after_tail);
            if (!next(nx)) return;
        }
        if (has_tail) {
            run_tail(1, last, mx);
            double wm = wave_max(mx);
            if ((threadIdx.x & 63) == 0 && !(wm <= 0))
                atomicMax(&P.iter_max[it], (unsigned long long)__double_as_longlong(wm));
            if (!next(first_after_tail)) return;
        }
        if (ncols == 0 && !has_tail) {
            if (!next(-1)) return;
        }
        double m = __longlong_as_double((long long)__hip_atomic_load(&P.iter_max[it], __ATOMIC_RELAXED,
                                                                      __HIP_MEMORY_SCOPE_AGENT));
        if (P.check_tolerance && m < P.tolerance) {
            it++;
            break;
        }
    }
    if (lane0) *P.iters_used = it;
}

int pgs_max_blocks(int block, bool* ok) {
    int dev = 0, n_cu = 0, per_cu = 0;
    (void)hipGetDevice(&dev);
    (void)hipDeviceGetAttribute(&n_cu, hipDeviceAttributeMultiprocessorCount, dev);
    int one_body = 0;
    (void)hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, k_pgs<false, false>, block, 0);
    (void)hipOccupancyMaxActiveBlocksPerMultiprocessor(&one_body, k_pgs<false, true>, block, 0);
    per_cu = std::min(per_cu, one_body);
    *ok = per_cu > 0;
    return n_cu * (per_cu > 0 ? per_cu : 1);
}

hipError_t launch_pgs(hipStream_t s, const PgsArgs& P, int grid, int block, bool plain, bool one_body) {
    void (*single)(PgsArgs) = one_body ? k_pgs<true, true> : k_pgs<true, false>;
    void (*kernel)(PgsArgs) = one_body ? k_pgs<false, true> : k_pgs<false, false>;
    if (grid <= 1) {
        hipLaunchKernelGGL(single, dim3(1), dim3(block), 0, s, P);
        return hipGetLastError();
    }
    if (plain) {
        // the caller clamps grid to the co-resident limit; the barrier's spin
        // limit turns a grid that is not co-resident into an error
        hipLaunchKernelGGL(kernel, dim3(grid), dim3(block), 0, s, P);
        return hipGetLastError();
    }
    void* args[] = {(void*)&P};
    return hipLaunchCooperativeKernel((const void*)kernel, dim3(grid), dim3(block), args, 0, s);
}

// ---------------------------------------------------------------------------
// Dataflow schedule of the same sweeps.
//
// Each dynamic body receives its group updates in sorted (colour-major) order,
// the order the coloured schedule and the exported sweep order define, and
// groups on disjoint bodies commute: the result is bit-identical to the
// coloured schedule, with no grid-wide barrier.  The order is kept by handing
// a body's deltaV from each update to the next through slots: sorted group q
// writes its updated deltaV of each dynamic body to its own slot (incidence
// 2 q + side, one set of slots per pass parity), and the body's next update
// (one rank higher, or for rank 0 the body's last group of the previous pass:
// pred[]) polls that slot until it no longer holds the empty pattern, takes
// the value and empties the slot for its next writer.  Pass 0 is
// confidentWarmStart, passes 1..iterations are sweeps.
//
// A wave runs steps of up to four groups of one colour, one group per 16-lane
// row (lanes hold one deltaV component each, quads A.v, A.w, B.v, B.w), so a
// row's J.dv is a product per lane and a fixed-shape DPP reduction in the
// reference's summation order.  Wave w runs steps w, w + W, ... pass by pass
// in order; the global minimum (pass, step) not yet done always has its
// inputs, so with every wave resident the schedule cannot deadlock, and
// bounded spins turn a wave that stops making progress into an error flag
// instead of a hang.
//
// Early exit (PGS.java:190) needs the max |dl| of sweep t before sweep t+1 is
// final.  Sweeps double-buffer lambda (odd sweeps in lam_alt) and deltaV (odd
// passes in dv_alt), and a wave starts sweep p only once sweep p-2 is known not
// to have converged, so at most one sweep runs speculatively and its buffers
// are simply not selected.  The last sweep (contact states) waits for the
// verdict on the one before it, so it never runs speculatively.

AMD_INLINE double* slot_at(const FlowArgs& F, int parity, int incidence) {
    return F.slot + ((size_t)parity * 2 * F.n_groups + incidence) * kSlotDoubles;
}
AMD_INLINE unsigned long long ld_cnt64(const unsigned long long* p) {
    return __hip_atomic_load(const_cast<unsigned long long*>(p), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
AMD_INLINE int uniform(int v) { return __builtin_amdgcn_readfirstlane(v); }
// DPP move of a double (bound_ctrl: lanes without a source read 0)
template <int kCtrl>
AMD_INLINE double dpp_d(double v) {
    const long long b = __double_as_longlong(v);
    const int lo = __builtin_amdgcn_mov_dpp((int)b, kCtrl, 0xF, 0xF, true);
    const int hi = __builtin_amdgcn_mov_dpp((int)(b >> 32), kCtrl, 0xF, 0xF, true);
    return __longlong_as_double(((long long)hi << 32) | (unsigned)lo);
}
constexpr int kQuadLane0 = 0x00, kQuadLane1 = 0x55, kQuadLane2 = 0xAA;  // quad_perm broadcasts
constexpr int kRowHalfMirror = 0x141, kRowMirror = 0x140;

// Contact.getJdv (Contact.java:362-378) for the group held by a 16-lane row.
// Quads of the row hold A.v, A.w, B.v, B.w (lanes 0-2 of each quad, lane 3
// idle), p = J_i dv_i.  Every lane of the row gets the reference's sum
// ((p0 + p1) + p2) per quad, (v + w) per body, then A + B; the partner quads
// come through mirrors, which only swap the operands of an addition, and IEEE
// addition commutes.
AMD_INLINE double row_jdv(double p) {
    const double s = (dpp_d<kQuadLane0>(p) + dpp_d<kQuadLane1>(p)) + dpp_d<kQuadLane2>(p);
    const double h = s + dpp_d<kRowHalfMirror>(s);
    return h + dpp_d<kRowMirror>(h);
}

constexpr long kFlowSpinLimit = 1L << 22;  // polls of one wait (each a memory round trip)
// Turns of a wait that may look at LDS only, and are shorter: the pass keeper's, and the sweeping waves' for it.  A wave that stops making
// progress meets the limit above first, and its error flag ends these.
constexpr long kLdsSpinLimit = 16 * kFlowSpinLimit;

// Per-contact operands of one row: this lane's J entries and update
// coefficients of the three rows, and the contact's uniform values.
struct WaveRec {
    double jc[6];  // as stored: the A.v lanes flip the sign on use (J)
    unsigned sign;
    double b[3], d[3], den[3], y[3], mu, clamp, lam[3];
};
// Where a lane's entries sit in a record: quads hold A.v, A.w, B.v, B.w;
// J entries ja.v = -jb.v, ja.w, jb.v, jb.w; coefficients -jb.v, jinv_a ja.w,
// jb.v, jinv_b jb.w (the v lanes' coefficient is their J entry, scaled by
// minv*dl at update time).
struct LaneMap {
    int jofs, cofs;
    unsigned sign;  // sign bit flipped on A.v lanes
};
AMD_INLINE LaneMap lane_map(int li) {
    const int q = li >> 2, j = (li & 3) < 3 ? (li & 3) : 0;
    LaneMap m;
    m.jofs = (q == 1 ? kRecAw : q == 3 ? kRecBw : kRecBv) + j;
    m.cofs = q == 1 ? kRecTa + j : q == 3 ? kRecTb + j : m.jofs;
    m.sign = q == 0 ? 0x80000000u : 0u;
    return m;
}
AMD_INLINE double flip(double v, unsigned sign) {
    const long long b = __double_as_longlong(v) ^ ((long long)sign << 32);
    return __longlong_as_double(b);
}
AMD_INLINE const double* lam_src(const FlowArgs& F, int k, int p) {
    const bool from_alt = p >= 1 && ((p - 1) & 1);
    return from_alt ? &F.lam_alt[4 * k] : &F.P.rec[(size_t)k * kRecDoubles + kRecLambda];
}
// rec: the row's record (LDS or global); lam: its lambda for this pass
AMD_INLINE double J(const WaveRec& c, int i) { return flip(c.jc[i], c.sign); }
AMD_INLINE void read_wave_rec(const double* rec, const double* lam, const LaneMap& m, WaveRec& w) {
    w.sign = m.sign;
#pragma unroll
    for (int r = 0; r < 3; r++) {
        const double* q = rec + r * kRecRow;
        w.jc[2 * r] = q[m.jofs];
        w.jc[2 * r + 1] = q[m.cofs];
        w.b[r] = q[kRecB];
        w.d[r] = q[kRecD];
        w.den[r] = q[kRecDen];
        w.y[r] = q[kRecY];
        w.lam[r] = lam[r];
    }
    w.mu = rec[kRecMu];
    w.clamp = rec[kRecClamp];
}

// A step's records are copied into LDS with DMA loads (16 B per lane, lane
// l's bytes at 16 l) before the wave waits for its dependencies: per contact
// slot, two blocks of two rows' 512-byte records, and a block with each row's
// lambda when the pass reads the odd-sweep buffer.
constexpr int kDmaSlots = 8;
typedef __attribute__((address_space(3))) void lds_void;
struct DmaSlot {
    double2 rec[2][64];
    double2 lam[64];
};

// A contact's new lambdas go to this pass's buffer; the last sweep also sets
// its state (Contact.updateContactState, Contact.java:385-398).
AMD_INLINE double* lam_dst(const FlowArgs& F, int k, int p) {
    return (p & 1) ? &F.lam_alt[4 * k] : &F.P.rec[(size_t)k * kRecDoubles + kRecLambda];
}
AMD_INLINE void contact_state(const FlowArgs& F, const WaveRec& c, int k, bool last, bool lead,
                              const double (&lam)[3], double dv) {
    const PgsArgs& P = F.P;
    if (last) {
        const double w1 = c.b[1] + row_jdv(J(c, 2) * dv);
        const double w2 = c.b[2] + row_jdv(J(c, 4) * dv);
        if (lead) {
            int st;
            if (fabs(lam[0]) <= 1e-14) st = AM_STATE_BROKEN;
            else if (fabs(w1) > P.sliding) st = AM_STATE_ONEDGE;
            else if (fabs(w2) > P.sliding) st = AM_STATE_ONEDGE;
            else st = AM_STATE_CLEAR;
            P.sstate[k] = st;
        }
    }
}
AMD_INLINE void contact_done(const FlowArgs& F, const WaveRec& c, int k, int p, bool last, bool lead,
                             const double (&lam)[3], double dv) {
    // every lane of the row stores the same values to the same place
    double* dst = lam_dst(F, k, p);
    dst[0] = lam[0];
    dst[1] = lam[1];
    dst[2] = lam[2];
    contact_state(F, c, k, last, lead, lam, dv);
}

// One contact of a row-held group in pass p (PGS.java:100-184; pass 0 is
// confidentWarmStart, PGS.java:250-256).  dv is this lane's deltaV component,
// f its body's minv on v lanes and 1 on w lanes (PGS.java:221-245 scales the
// v part by minv*dl and the w part by dl; 1*dl == dl exactly).  mx is the
// running max |dl| with NaN tracked apart (Math.max keeps a NaN).
AMD_INLINE void row_contact(const FlowArgs& F, const WaveRec& c, int k, int p, bool last, bool lead, double f,
                            double& dv, double& mx, bool& nan) {
    const PgsArgs& P = F.P;
    double lam[3] = {c.lam[0], c.lam[1], c.lam[2]};
    if (p == 0) {
#pragma unroll
        for (int r = 0; r < 3; r++) dv = (f * lam[r]) * J(c, 2 * r + 1) + dv;
        return;
    }
#pragma unroll
    for (int r = 0; r < 3; r++) {
        const double jd = row_jdv(J(c, 2 * r) * dv);
        const double prev = lam[r];
        const double num = c.d[r] * lam[r] - P.omega * (c.b[r] + jd);
        double l = div_row(num, c.den[r], c.y[r]);
        // projection (PGS.java:111-113, 150-158), selected without a branch.
        // Math.max(0, l) is (l <= 0) ? +0 : l for every l (NaN and -0
        // included).  For a limit that is neither NaN nor -0, Math.max(l,
        // -limit) and Math.min(., limit) are the plain selects below (NaN l
        // falls through both, and the only zero tie, -0 against +0, resolves
        // the Java way); other limits take the full Java forms.
        double lc;
        if (r == 0) {
            lc = l <= 0.0 ? 0.0 : l;
        } else {
            const double limit = c.mu * lam[0];
            const bool plain = limit > 0.0 || __double_as_longlong(limit) == 0;
            const double a = l < -limit ? -limit : l;
            lc = a > limit ? limit : a;
            if (__builtin_expect(!__all(plain), 0)) {
                if (!plain) lc = jmin(jmax(l, -limit), limit);
            }
        }
        l = c.clamp != 0.0 ? lc : l;
        lam[r] = l;
        const double diff = l - prev;
        dv = (f * diff) * J(c, 2 * r + 1) + dv;
        mx = fmax(mx, fabs(diff));
        nan = nan || diff != diff;
    }
    contact_done(F, c, k, p, last, lead, lam, dv);
}

// The same update where the step has been found to need none of the general
// forms: every row's |numerator| in [2^-250, 2^250) with a nonzero stored
// reciprocal (the quotient is then q0 = n y, r = fma(-d, q0, n), q = fma(r, y,
// q0), exactly the division), every friction limit a finite value >= +0 (the
// plain selects are then Math.max/Math.min), and every contact clamped (its
// record's clamp flag 1, which also says every row's reciprocal is stored).  The
// conditions are gathered per lane into FastCheck without a branch; the step
// checks them once at its end and, if any failed, runs again from its start
// with row_contact.
struct FastCheck {
    unsigned num_hi_max = 0;            // high words of |numerator|
    unsigned num_hi_min = 0xffffffffu;
    unsigned limit_hi_max = 0;          // high words of the friction limits (sign included)
    bool plain = true;                  // every contact's clamp flag 1
    AMD_INLINE bool ok() const {
        return plain && num_hi_min >= 0x30500000u && num_hi_max < 0x4F900000u && limit_hi_max < 0x7FF00000u;
    }
};
AMD_INLINE unsigned hi_word(double v) { return (unsigned)((unsigned long long)__double_as_longlong(v) >> 32); }
AMD_INLINE void row_contact_fast(const FlowArgs& F, const WaveRec& c, int k, int p, bool last, bool lead, double f,
                                 double& dv, double& mx, FastCheck& chk, double (&lam)[3]) {
    const PgsArgs& P = F.P;
    lam[0] = c.lam[0];
    lam[1] = c.lam[1];
    lam[2] = c.lam[2];
    chk.plain = chk.plain && c.clamp == 1.0;
#pragma unroll
    for (int r = 0; r < 3; r++) {
        const double jd = row_jdv(J(c, 2 * r) * dv);
        const double prev = lam[r];
        const double num = c.d[r] * lam[r] - P.omega * (c.b[r] + jd);
        const unsigned h = hi_word(num) & 0x7fffffffu;
        chk.num_hi_max = max(chk.num_hi_max, h);
        chk.num_hi_min = min(chk.num_hi_min, h);
        const double q0 = num * c.y[r];
        const double rr = __builtin_fma(-c.den[r], q0, num);
        double l = __builtin_fma(rr, c.y[r], q0);
        if (r == 0) {
            // l is finite and nonzero here (nonzero finite quotient), so
            // max(l, +0) is Math.max(0, l)
            l = __builtin_fmax(l, 0.0);
        } else {
            const double limit = c.mu * lam[0];
            chk.limit_hi_max = max(chk.limit_hi_max, hi_word(limit));
            l = __builtin_fmin(__builtin_fmax(l, -limit), limit);
        }
        lam[r] = l;
        const double diff = l - prev;
        dv = (f * diff) * J(c, 2 * r + 1) + dv;
        // finite whenever the step's conditions hold (a NaN or infinite
        // numerator fails them), so no NaN is tracked here
        mx = fmax(mx, fabs(diff));
    }
    contact_state(F, c, k, last, lead, lam, dv);
}

// Steps: up to 4 consecutive sorted groups of one parallel colour (no shared
// dynamic body), one per 16-lane row of a wave.  A colour with fewer groups
// than there are waves, and the sequential tail colour, give one group per
// step: a step starts when all its groups' inputs are there, and the long
// chains of dependent updates run through the small late colours, where a
// group would otherwise wait for its step-mates' inputs.  Wave w runs steps
// w, w + W, ... of every pass in order.
constexpr int kRowsPerWave = 4;

// kScenes: a batched solve with per-scene exits (P.per_scene set); the
// single-scene kernel carries none of their code.
template <bool kScenes>
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(1, 2))) void k_pgs_flow(FlowArgs F) {
    const PgsArgs& P = F.P;
    const int* cs = P.colour_start;
    __shared__ int s_sp[kMaxColours + 2];  // first step of each colour, then the total
    __shared__ int s_per[kMaxColours + 1];  // groups per step of each colour
    const int W = gridDim.x;
    if (threadIdx.x == 0) {
        int n = 0;
        for (int c = 0; c <= kMaxColours; c++) {
            s_sp[c] = n;
            const int g = cs[c + 1] - cs[c];
            const int per = c < kMaxColours && g >= W ? kRowsPerWave : 1;
            s_per[c] = per;
            n += (g + per - 1) / per;
        }
        s_sp[kMaxColours + 1] = n;
    }
    __syncthreads();
    const int n_steps = s_sp[kMaxColours + 1];
    const int w = blockIdx.x;
    const int lane = threadIdx.x;
    const int row = lane >> 4, li = lane & 15, quad = li >> 2, jj = li & 3;
    const bool lead = li == 0;
    const bool mine = jj < 3;               // holds a deltaV component
    const bool side_b = quad >= 2;
    const bool vlane = (quad & 1) == 0;     // a linear-velocity component
    const int comp = (quad & 1) * 3 + (jj < 3 ? jj : 0);
    const int first = P.warm_start ? 0 : 1;
    const int lastp = P.iterations;
    const int4* gdesc = reinterpret_cast<const int4*>(P.group_desc);
    const int4* fdesc = reinterpret_cast<const int4*>(F.flow);
    __shared__ DmaSlot s_dma[kDmaSlots];
    __shared__ double s_lam[kRowsPerWave][kDmaSlots][4];  // fast-update lambdas of the step
    const int2* gpred = reinterpret_cast<const int2*>(F.pred);
    const LaneMap lmap = lane_map(li);
    int chk = 0;  // sweeps 1..chk are known not to have converged

    // per-scene exits: the scene counter this lane's row still has to add
    // its group to (added once the step after it has waited for its memory
    // operations, or at the end of the pass)
    unsigned long long* pend_done = nullptr;
    unsigned long long pend_add = 0;
    for (int p = first; p <= lastp; p++) {
        // pass gates: sweep p-2 must be known not converged (p-1 for the last sweep)
        if (P.check_tolerance) {
            const int need = (p == lastp && p >= 2) ? p - 1 : p - 2;
            long spins = 0;
            while (chk < need) {
                // the waves done with sweep chk + 1 and those over the
                // tolerance there (the sweep converged if none was), summed
                // over the sweep's words (read together)
                unsigned long long wd = 0;
                const unsigned long long* pw = &F.pass_done[(size_t)(chk + 1) * kPassWords];
#pragma unroll
                for (int q = 0; q < kPassWords; q++) wd += ld_cnt64(&pw[q]);
                const unsigned d = (unsigned)uniform((int)(unsigned)(wd >> 32));
                if (d == F.n_waves) {
                    if (uniform((int)(unsigned)wd) == 0) return;  // converged at sweep chk + 1
                    chk++;
                    spins = 0;
                    continue;
                }
                if (++spins > kFlowSpinLimit ||
                    ((spins & 255) == 0 && uniform(__hip_atomic_load(P.error, __ATOMIC_RELAXED,
                                                                      __HIP_MEMORY_SCOPE_AGENT)))) {
                    if (lane == 0) atomicOr(P.error, 1);
                    return;
                }
            }
        }
        double mx = 0.0;
        bool nan = false;
        double* cur = (p & 1) ? F.dv_alt : P.dv;
        double* prv = (p & 1) ? P.dv : F.dv_alt;
        int c = 0;  // colour of the current step (steps ascend)
        // this row's group of a step (the colour cursor advances with st)
        auto step_group = [&](int st, bool& act) {
            while (s_sp[c + 1] <= st) c++;
            const int per = s_per[c];
            const int q0 = cs[c] + (st - s_sp[c]) * per;
            const int count = min(per, cs[c + 1] - q0);
            act = row < count;
            return q0 + (act ? row : 0);
        };
        bool nx_active = false;
        int4 nx_gd = make_int4(0, 0, 0, 0), nx_fd = make_int4(0, 0, 0, 0);
        int2 nx_pr = make_int2(0, 0);
        int nx_sc = 0, nx_q = 0;
        if (w < n_steps) {
            const int q = step_group(w, nx_active);
            nx_q = q;
            nx_gd = gdesc[q];
            nx_fd = fdesc[q];
            nx_pr = gpred[q];
            if (kScenes) nx_sc = P.g_scene[q];
        }
        for (int st = w; st < n_steps; st += W) {
            // descriptors of this step were loaded during the previous one
            const bool has_group = nx_active;
            const int4 gd = nx_gd;
            const int4 fd = nx_fd;
            const int2 pr = nx_pr;
            const int sc = nx_sc, qg = nx_q;
            if (st + W < n_steps) {
                const int q = step_group(st + W, nx_active);
                nx_q = q;
                nx_gd = gdesc[q];
                nx_fd = fdesc[q];
                nx_pr = gpred[q];
                if (kScenes) nx_sc = P.g_scene[q];
            }
            // Per-scene exits: a row whose scene was under the tolerance at
            // sweep p-2 or p-3 (or p-1 before the last sweep) skips this
            // pass.  A skipped sweep leaves the scene's max at 0, so with
            // p-3 checked too a scene that skipped once skips every later
            // pass (its first sweep under the tolerance is final; a later
            // sweep over it must not bring back a scene whose groups
            // published nothing for the pass before).  Lane 0 of the row
            // learns it while the wave polls for its inputs below: it waits
            // until every group of the scene has finished those sweeps, then
            // reads the scene's max.  Every group it waits for comes earlier
            // in the (pass, step) order, so the earliest undone step can
            // always run.  Until then the row counts as active (its records
            // are copied and its inputs polled for).
            bool active = has_group;
            int n = active ? gd.y - gd.x : 0;
            int nmax = n;
            nmax = max(nmax, __shfl_xor(nmax, 16, 64));
            nmax = max(nmax, __shfl_xor(nmax, 32, 64));
            // the step's records do not depend on other waves: copy them into
            // LDS while the wave waits.  Lane l of a record block copies word
            // l & 31 of row 2i + (l >> 5)'s record.
            const int staged = min(nmax, kDmaSlots);
            const bool odd_lam = p >= 1 && ((p - 1) & 1);
            {
                int kb[kRowsPerWave], nl[kRowsPerWave];
#pragma unroll
                for (int r = 0; r < kRowsPerWave; r++) {
                    kb[r] = __builtin_amdgcn_readlane(gd.x, r * 16);
                    nl[r] = max(__builtin_amdgcn_readlane(n, r * 16) - 1, 0);
                }
                const bool upper = lane >= 32;
                for (int t = 0; t < staged; t++) {
#pragma unroll
                    for (int i = 0; i < 2; i++) {
                        const int r0 = 2 * i, r1 = 2 * i + 1;
                        const int k = upper ? kb[r1] + min(t, nl[r1]) : kb[r0] + min(t, nl[r0]);
                        const double* src = P.rec + (size_t)k * kRecDoubles + 2 * (lane & 31);
                        __builtin_amdgcn_global_load_lds((const void*)src, (lds_void*)&s_dma[t].rec[i][0], 16, 0, 0);
                    }
                    if (odd_lam) {
                        const int k = gd.x + min(t, max(n - 1, 0));  // this lane's row
                        const double* src = &F.lam_alt[4 * k + (li == 1 ? 2 : 0)];
                        __builtin_amdgcn_global_load_lds((const void*)src, (lds_void*)&s_dma[t].lam[0], 16, 0, 0);
                    }
                }
            }
            // Each lane of a dynamic body takes its deltaV component from the
            // slot of that body's previous update (this pass's, or for the
            // body's first group the previous pass's last): it polls until
            // the slot is filled, then empties it for the slot's next writer.
            // The body's first update of the launch, and pinned bodies, read
            // the launch buffers instead.
            const int e = side_b ? gd.w : gd.z;
            const int rank = side_b ? fd.z : fd.x;
            const int deg = side_b ? fd.w : fd.y;
            double dv = 0.0, f = 1.0;
            bool dyn = false;
            double* src = nullptr;
            if (active && mine) {
                if (vlane) f = P.minv[e];
                dyn = deg != 0;
                if (dyn && !(p == first && rank == 0))
                    src = slot_at(F, rank == 0 ? ((p - 1) & 1) : (p & 1), side_b ? pr.y : pr.x) + comp;
                else
                    dv = ld_coherent(&prv[e * 6 + comp]);
            }
            {
                bool got = src == nullptr;
                long spins = 0;
                auto spin = [&]() -> bool {  // false: give up (error flag set)
                    __builtin_amdgcn_s_sleep(1);
                    if (++spins > kFlowSpinLimit ||
                        ((spins & 255) == 0 && uniform(__hip_atomic_load(P.error, __ATOMIC_RELAXED,
                                                                          __HIP_MEMORY_SCOPE_AGENT)))) {
                        if (lane == 0) atomicOr(P.error, 1);
                        __builtin_amdgcn_s_waitcnt(0);  // this step's LDS copies land before the wave ends
                        return false;
                    }
                    return true;
                };
                auto poll = [&]() {
                    if (!got) {
                        const double v = ld_coherent(src);
                        if ((unsigned long long)__double_as_longlong(v) != kSlotEmpty) {
                            dv = v;
                            got = true;
                        }
                    }
                };
                const int t1 = p - 2, t2 = (p == lastp) ? p - 1 : 0;
                if (!(kScenes && p >= 1 && P.check_tolerance && (t1 >= 1 || t2 >= 1))) {
                    while (true) {
                        poll();
                        if (__all(got)) break;
                        if (!spin()) return;
                    }
                } else {
                    // lane 0 of each row resolves its scene's exit check
                    // while the row polls; a skipped row reads no inputs (its
                    // scene's other groups skip this pass too and publish none)
                    bool resolved = !(has_group && li == 0), skip = false;
                    const unsigned want = has_group ? P.scene_groups[sc] : 0u;
                    const unsigned long long* cnt = &P.scene_done[(size_t)sc * (P.iterations + 1)];
                    // sweeps checked: t1, t1 - 1 and t2 where they exist (a
                    // missing one repeats t1 or t2)
                    const int ta = t1 >= 1 ? t1 : t2, tb = t1 >= 2 ? t1 - 1 : ta, tc = t2 >= 1 ? t2 : ta;
                    while (true) {
                        // the slot and the scene's words are read together; a
                        // sweep's word is final once all the scene's groups
                        // have counted themselves in it, and the scene was
                        // under the tolerance there if none was over it
                        double v = 0.0;
                        if (!got) v = ld_coherent(src);
                        unsigned long long wa = 0, wb = 0, wc = 0;
                        if (!resolved) {
                            wa = ld_cnt64(&cnt[ta]);
                            wb = ld_cnt64(&cnt[tb]);
                            wc = ld_cnt64(&cnt[tc]);
                        }
                        if (!got && (unsigned long long)__double_as_longlong(v) != kSlotEmpty) {
                            dv = v;
                            got = true;
                        }
                        if (!resolved && (unsigned)(wa >> 32) == want && (unsigned)(wb >> 32) == want &&
                            (unsigned)(wc >> 32) == want) {
                            skip = (unsigned)wa == 0u || (unsigned)wb == 0u || (unsigned)wc == 0u;
                            resolved = true;
                        }
                        const bool row_resolved = __shfl(resolved, row * 16, 64);
                        const bool row_skip = __shfl(skip, row * 16, 64);
                        if (__all(row_resolved && (row_skip || got))) break;
                        if (!spin()) return;
                    }
                    if (__shfl(skip, row * 16, 64) && has_group) {
                        active = false;
                        n = 0;
                        src = nullptr;
                    }
                }
            }
            const bool last = p == lastp;
            __builtin_amdgcn_s_waitcnt(0);  // LDS copies landed
            if (kScenes && pend_done) {
                // the previous step's scene max has landed (the wait above)
                __hip_atomic_fetch_add(pend_done, pend_add, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                pend_done = nullptr;
            }
            // rows with fewer contacts idle; contacts past the LDS slots
            // (groups of more than kDmaSlots contacts) read global memory
            double smx = 0.0;  // this step's max |dl| and NaN flag (row-uniform)
            bool snan = false;
            // Contacts in the LDS slots and the rest (read from global
            // memory) run in separate loops, so that the first one waits on
            // LDS reads only and never on the lambda stores in flight.
            const int in_lds = min(nmax, kDmaSlots);
            auto lds_rec = [&](int t, WaveRec& rc) {
                const double* rl = reinterpret_cast<const double*>(&s_dma[t].rec[row >> 1][(row & 1) * 32]);
                const double* ll = odd_lam ? reinterpret_cast<const double*>(&s_dma[t].lam[row * 16]) : rl + kRecLambda;
                read_wave_rec(rl, ll, lmap, rc);
            };
            auto global_rec = [&](int t, WaveRec& rc) {
                const int k = gd.x + min(t, max(n - 1, 0));
                read_wave_rec(P.rec + (size_t)k * kRecDoubles, lam_src(F, k, p), lmap, rc);
            };
            // sweeps try the fast update first, which keeps the lambdas of the
            // contacts in the LDS slots in LDS; the general update stores its
            // lambdas at once (over the few the fast one stored directly, in
            // the same places from the same lanes, if the step runs again)
            bool general = p == 0;
            if (!general) {
                const double dv_start = dv;
                FastCheck fc;
                // the next contact's record is read while this one runs
                // (two buffers used in turn, so nothing is copied)
                WaveRec ra, rb;
                if (in_lds > 0) lds_rec(0, ra);
                double lam[3];
                for (int t = 0; t < in_lds; t += 2) {
                    if (t + 1 < in_lds) lds_rec(t + 1, rb);
                    if (t < n) {
                        row_contact_fast(F, ra, gd.x + t, p, last, lead, f, dv, smx, fc, lam);
                        // every lane of the row writes the same values to the same place
                        s_lam[row][t][0] = lam[0];
                        s_lam[row][t][1] = lam[1];
                        s_lam[row][t][2] = lam[2];
                    }
                    if (t + 1 >= in_lds) break;
                    if (t + 2 < in_lds) lds_rec(t + 2, ra);
                    if (t + 1 < n) {
                        row_contact_fast(F, rb, gd.x + t + 1, p, last, lead, f, dv, smx, fc, lam);
                        s_lam[row][t + 1][0] = lam[0];
                        s_lam[row][t + 1][1] = lam[1];
                        s_lam[row][t + 1][2] = lam[2];
                    }
                }
                for (int t = kDmaSlots; t < nmax; t++) {
                    global_rec(t, ra);
                    if (t < n) {
                        row_contact_fast(F, ra, gd.x + t, p, last, lead, f, dv, smx, fc, lam);
                        double* dst = lam_dst(F, gd.x + t, p);
                        dst[0] = lam[0];
                        dst[1] = lam[1];
                        dst[2] = lam[2];
                    }
                }
                if (__builtin_expect(!__all(fc.ok()), 0)) {
                    general = true;
                    dv = dv_start;
                    smx = 0.0;
                    snan = false;
                    __builtin_amdgcn_s_waitcnt(0);
                }
            }
            if (general) {
                for (int t = 0; t < in_lds; t++) {
                    WaveRec rc;
                    lds_rec(t, rc);
                    if (t < n) row_contact(F, rc, gd.x + t, p, last, lead, f, dv, smx, snan);
                }
                for (int t = kDmaSlots; t < nmax; t++) {
                    WaveRec rc;
                    global_rec(t, rc);
                    if (t < n) row_contact(F, rc, gd.x + t, p, last, lead, f, dv, smx, snan);
                }
            }
            mx = fmax(mx, smx);
            nan = nan || snan;
            // Publish deltaV to this group's slots.  The body's last update of
            // the pass also goes to the pass's buffer, which holds the result
            // when this is the last sweep.
            if (active && mine && dyn) {
                st_coherent(slot_at(F, p & 1, 2 * qg + (side_b ? 1 : 0)) + comp, dv);
                if (rank == deg - 1) st_coherent(&cur[e * 6 + comp], dv);
            }
            // The slot that was read is emptied behind the values that the next
            // update waits for.  It must be seen empty before its next writer
            // fills it; that writer comes after this group's own publish of the
            // next pass (the body's updates are one chain), and the stores of
            // this pass have landed by the wait after that pass's poll.
            if (src) st_coherent(src, __longlong_as_double((long long)kSlotEmpty));
            if (!general && active && li < 3) {
                const int nl = min(n, kDmaSlots);
                for (int t = 0; t < nl; t++) {
                    lam_dst(F, gd.x + t, p)[li] = s_lam[row][t][li];
                }
            }
            // per-scene exits, after the publish (which is what later steps
            // wait for): the scene's max for this sweep now, the group's
            // count once a later wait has seen the max land
            if (kScenes && p >= 1 && has_group && lead) {
                if (active && !(smx <= 0))
                    atomicMax(&P.scene_max[(size_t)sc * P.iterations + p - 1],
                              (unsigned long long)__double_as_longlong(
                                  snan ? __longlong_as_double(0x7ff8000000000000ll) : smx));
                pend_done = &P.scene_done[(size_t)sc * (P.iterations + 1) + p];
                // over the tolerance (NaN included), as the scene's max would be
                const bool over = active && !(smx <= 0) && (snan || !(smx < P.tolerance));
                pend_add = (1ull << 32) | (over ? 1ull : 0ull);
            }
        }
        if (kScenes && pend_done) {
            __builtin_amdgcn_s_waitcnt(0);
            __hip_atomic_fetch_add(pend_done, pend_add, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            pend_done = nullptr;
        }
        if (p >= 1) {
            if (__any(nan)) mx = __longlong_as_double(0x7ff8000000000000ll);
            mx = wave_max(mx);
            if (lane == 0) {
                if (!(mx <= 0))  // NaN included
                    atomicMax(&P.iter_max[p - 1], (unsigned long long)__double_as_longlong(mx));
                // the wait also lands this wave's lambda stores before its next
                // pass reads them back
                __builtin_amdgcn_s_waitcnt(0);
                const bool over = !(mx <= 0) && !(mx < P.tolerance);  // NaN over
                __hip_atomic_fetch_add(&F.pass_done[(size_t)p * kPassWords + (w % kPassWords)],
                                       (1ull << 32) | (over ? 1ull : 0ull), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            }
        }
    }
}

// ---------------------------------------------------------------------------
// The dataflow schedule with everything that a wave needs resident in LDS.
//
// Where the solve fits (kResDoubles of LDS for the four waves of each CU: 55,000
// contacts where the waves get equal shares, as in one colour; 46,000 in a wall of
// boxes, under 33,000 in 80 batched scenes), every wave keeps its groups' records, lambdas and
// bookkeeping in LDS for the whole solve, and a pass reads no global memory
// but the slots.  What bounds it is the chain of dependent group updates, a
// link of which costs the handoff of deltaV (0.4 us between CUs) and the
// contacts' arithmetic.  So the arithmetic is laid out for latency:
//  - A quad of lanes holds a group (A.v, A.w, B.v, B.w, three components
//    each): a row's J.dv is three products and two additions per lane and two
//    DPP exchanges, where a 16-lane row with one component per lane needs two
//    more stages.  16 groups of a colour share a wave's instructions.
//  - Friction limits are applied with min and max, not compares and selects
//    (46 cycles a bound, against 10).
//  - The next contact's record is read while the current one runs, the first
//    one's while the wave waits for its inputs.
//  - Nothing waits before a publish, and the slot that was read is emptied
//    after it.  It must be seen empty before its next writer fills it; that
//    writer comes after this group's own publish of the next pass (the body's
//    updates are one chain), and the stores of this pass have landed by the
//    wait after that pass's poll.
//  - A body with a single group hands its deltaV to itself through LDS.
// The gates between passes are kept by a fifth wave of each workgroup: it
// reports the passes its workgroup's waves have finished, follows the sweeps'
// verdicts, and leaves both in LDS, where a sweeping wave finds them without
// a global read.
//
// Groups are spread over all waves: a step takes ceil(groups of the colour /
// waves) groups, at most 16, so a colour is one step per wave while it can be.
// Measured (per sweep, against k_pgs_flow): see the dispatch in pgs_shape.
constexpr int kResWaves = 4;                        // sweeping waves of a workgroup
constexpr int kQuads = 16;                          // groups of a step
constexpr int kResDoubles = kResidentDoubles;       // LDS of a workgroup's waves together
// A contact in LDS.  Per row, what each kind of lane reads (its J entries, then
// its update coefficients) as 6 doubles in a row, three 16-byte reads: jb.v
// twice for the v lanes, ja.w and jinv_a ja.w, jb.w and jinv_b jb.w; then b, D,
// D + C and its reciprocal of each row; then lambda and mu, once for even and
// once for odd passes.  A wave issues an LDS read every 20 cycles or so, so a
// contact is laid out for few of them (17; 21 with the records' own layout).
constexpr int kResRow = 18, kResV = 0, kResAw = 6, kResBw = 12;
constexpr int kResScalars = 3 * kResRow;  // 4 a row
constexpr int kResLam = kResScalars + 12, kResLamOdd = kResLam + 4;
constexpr int kResContact = kResLamOdd + 4;
// per group, for each side: deltaV (6) of a body that is only this group's or
// pinned, minv, {LDS offset of the first contact, contacts}, {body, incidence of
// its previous update, flags, scene (side A) or the scene's groups (side B)}
constexpr int kResSide = 10, kResGroup = 2 * kResSide;
constexpr int kResF = 6, kResFirst = 7, kResInts = 8;
enum { kSideDyn = 1, kSideSelf = 2, kSideRank0 = 4, kSideLast = 8 };

struct ResidentSteps {
    int n[kMaxColours + 1], per[kMaxColours + 1], first[kMaxColours + 1];
    int start[kMaxColours + 2];  // first sorted group of each colour
    int colours;                 // up to the last one that has groups
};
struct ResidentLds {
    double2 region[kResDoubles / 2];       // the waves' groups, each wave as much as the plan counted for it
    // LDS offset of its groups, first sorted group, groups | every contact's clamp
    // flag is 1 << 7 | contacts of its largest << 8, contacts; first sweep position
    int4 step[kResWaves][kResidentSteps];
    int step_k0[kResWaves][kResidentSteps];
    ResidentSteps steps;
    double pass_max[4][kResWaves * kQuads];  // by pass % 4: max |dl| of each quad
    int done[kResWaves];                   // passes that each wave has finished
    int published;  // passes up to this one are reported
    int known;      // sweeps 1..known are known not to have converged
    int stop;       // the sweep that converged
    int failed;
};
static_assert(sizeof(ResidentLds) <= 160 * 1024, "LDS of a CU");

// The steps of W waves: colour c has n[c] of per[c] groups each (one each in the
// sequential tail), and step i of it belongs to wave (first[c] + i) % W.  While
// there is a wave for every step they follow each other.  Otherwise the colours
// start 5/8 of the waves apart, as each begins with its largest groups: those of
// 8 colours in a row then fall to different waves.  27,000 contacts of 48 batched
// scenes need 25,000 doubles in the fullest workgroup when they follow each other,
// and fit like this.  Where both fit, a sweep takes the same within 3 % (piles of
// 8,900 to 26,800 contacts 1 to 2 % less, ropes and walls up to 3 % more).  A wave
// takes its steps colour by colour.
// Called by a whole workgroup of more than kMaxColours threads.
AMD_INLINE void resident_steps(const int* cs, int W, ResidentSteps& S) {
    const int c = threadIdx.x;
    if (c <= kMaxColours) {
        const int start = cs[c], g = cs[c + 1] - start;
        const int per = c < kMaxColours ? max(1, min(kQuads, (g + W - 1) / W)) : 1;
        S.start[c] = start;
        if (c == kMaxColours) S.start[c + 1] = start + g;
        S.per[c] = per;
        S.n[c] = (g + per - 1) / per;
    }
    __syncthreads();
    if (c <= kMaxColours) {
        int before = 0, total = 0, used = 0;
        for (int k = 0; k <= kMaxColours; k++) {
            const int n = S.n[k];
            before = k == c ? total : before;
            used = n ? k + 1 : used;
            total += n;
        }
        S.first[c] = total > W ? (int)((long)(c & 7) * 5 * W / 8) % W : before % W;
        if (c == 0) S.colours = used;
    }
    __syncthreads();
}
struct StepWalk {
    int c = -1, i = 0;
    // the wave's next step: its first sorted group and its groups; false at the end
    AMD_INLINE bool next(const ResidentSteps& S, int W, int w, int& q0, int& count) {
        if (c >= 0) i += W;
        while (c < 0 || i >= S.n[c]) {
            if (++c >= S.colours) return false;
            i = w - S.first[c];
            if (i < 0) i += W;
        }
        q0 = S.start[c] + i * S.per[c];
        count = min(S.per[c], S.start[c + 1] - q0);
        return true;
    }
};

// used[w] = LDS doubles of wave w; plan[0] = those of the fullest workgroup,
// plan[1] = steps of the busiest wave (counted only as far as the limits)
__global__ __launch_bounds__(256) void k_resident_plan(const int* cs, const int* group_desc, int W, int* used,
                                                       int* plan) {
    __shared__ ResidentSteps S;
    resident_steps(cs, W, S);
    const int w = blockIdx.x * blockDim.x + threadIdx.x;
    if (w >= W) return;  // W is a multiple of kResWaves, which divides the wavefront
    const int4* gdesc = reinterpret_cast<const int4*>(group_desc);
    int sum = 0, steps = 0, q0, count;
    StepWalk walk;
    while (walk.next(S, W, w, q0, count)) {
        const int contacts = gdesc[q0 + count - 1].y - gdesc[q0].x;
        sum += count * kResGroup + min(contacts, kResDoubles) * kResContact;
        steps++;
        if (sum > kResDoubles || steps > kResidentSteps) break;
    }
    used[w] = sum;
    int total = sum;
#pragma unroll
    for (int o = 1; o < kResWaves; o <<= 1) total += __shfl_xor(total, o, 64);
    if (w % kResWaves == 0) atomicMax(&plan[0], total);
    atomicMax(&plan[1], steps);
}
void launch_resident_plan(hipStream_t s, const int* colour_start, const int* group_desc, int waves, int* used,
                          int* plan) {
    hipLaunchKernelGGL(k_resident_plan, dim3((waves + 255) / 256), dim3(256), 0, s, colour_start, group_desc, waves,
                       used, plan);
}

// LDS operations of one wave are performed in order: only the compiler is held back
AMD_INLINE void lds_order() { asm volatile("" ::: "memory"); }
// ---------------------------------------------------------------------------
// The layout of a small contact set in one workgroup: incidence lists, colours,
// sorted groups, sweep order, flow ranks and the resident kernel's plan, which
// are some 20 launches otherwise (and were up to 100, with a launch per
// colouring round).  What bounds it is latency: the colouring's chain of
// groups, each waiting for a neighbour, runs in LDS (20 us for 3 groups, 56 for
// 1,700).
constexpr int kSmallThreads = 1024, kSmallWaves = kSmallThreads / 64;
constexpr int kSmallBins = kMaxColours * 16 + 1;  // (colour, 15 - size), then the tail
struct SmallLds {
    short colour[kSmallLayout];             // then each group's sorted position
    short sorted[kSmallLayout];             // with layers the group waited for; then the group at each sorted position
    unsigned short item[2 * kSmallLayout];  // each body's groups
    union {
        struct {  // a body's, at the start of its groups (TakenColours)
            unsigned long long set[2 * kSmallLayout];
            unsigned short in_tail[2 * kSmallLayout];
        };
        struct {
            unsigned short start_a, n_a, start_b, n_b;
        } lists[kSmallLayout];
        struct {
            unsigned short hist[kSmallWaves][kSmallBins + 7];
            int pos[kSmallLayout + 1];
        };
    };
    int wave_sum[kSmallWaves];
    int cs[kMaxColours + 2];
    int n_items;
    int gave_up;
    int plan[2];
    int one_body;
    ResidentSteps steps;
};
static_assert(sizeof(SmallLds) <= 160 * 1024, "LDS of a CU");

// exclusive sum of v over the workgroup; wave_sum is scratch
AMD_INLINE int small_exclusive(int v, int* wave_sum) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    int inc = v;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const int t = __shfl_up(inc, o, 64);
        if (lane >= o) inc += t;
    }
    __syncthreads();
    if (lane == 63) wave_sum[wave] = inc;
    __syncthreads();
    int before = 0;
    for (int k = 0; k < kSmallWaves; k++) before += k < wave ? wave_sum[k] : 0;
    return before + inc - v;
}
// the lanes of the wave with this lane's key (of 11 bits) that are in
AMD_INLINE unsigned long long same_key(int key, bool in) {
    unsigned long long m = __ballot(in);
#pragma unroll
    for (int b = 0; b < 11; b++) {
        const unsigned long long v = __ballot((key >> b) & 1);
        m &= (key >> b) & 1 ? v : ~v;
    }
    return m;
}
static_assert(kSmallBins <= 1 << 11, "same_key");

__global__ __launch_bounds__(kSmallThreads) void k_layout_small(SmallLayoutArgs A) {
    __shared__ SmallLds L;
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6, n = A.n_groups;
    constexpr int kPer = kSmallLayout / kSmallThreads;

    // Incidence lists: a body's groups in any order.  Only bodies with groups are
    // looked at: the groups clear their bodies' counts, and the first one counted at
    // a body takes its place in the list.
    if (t == 0) L.n_items = L.gave_up = 0;
    int body[kPer][2], at[kPer][2], count[kPer][2];  // this thread's groups; -1: a pinned body
#pragma unroll
    for (int k = 0; k < kPer; k++) {
        const int g = t + k * kSmallThreads;
        body[k][0] = g < n ? A.ga[g] : -1;
        body[k][1] = g < n ? A.gb[g] : -1;
    }
#pragma unroll
    for (int k = 0; k < kPer; k++)
#pragma unroll
        for (int s = 0; s < 2; s++)
            if (body[k][s] >= 0 && !dynamic_body(A.bflags, body[k][s])) body[k][s] = -1;
#pragma unroll
    for (int k = 0; k < kPer; k++)
        if (body[k][1] == body[k][0]) body[k][1] = -1;
#pragma unroll
    for (int k = 0; k < kPer; k++)
#pragma unroll
        for (int s = 0; s < 2; s++)
            if (body[k][s] >= 0) st_int(&A.inc_count[body[k][s]], 0);
    __builtin_amdgcn_s_waitcnt(0);
    __syncthreads();
#pragma unroll
    for (int k = 0; k < kPer; k++) {
        const int g = t + k * kSmallThreads;
#pragma unroll
        for (int s = 0; s < 2; s++) at[k][s] = body[k][s] >= 0 ? atomicAdd(&A.inc_count[body[k][s]], 1) : 0;
        if (g < n) {
            L.colour[g] = -1;
            L.sorted[g] = -1;
        }
    }
    __builtin_amdgcn_s_waitcnt(0);
    __syncthreads();
#pragma unroll
    for (int k = 0; k < kPer; k++)
#pragma unroll
        for (int s = 0; s < 2; s++)
            count[k][s] = body[k][s] >= 0 ? ld_int(&A.inc_count[body[k][s]]) : 0;
#pragma unroll
    for (int k = 0; k < kPer; k++)
#pragma unroll
        for (int s = 0; s < 2; s++) {
            if (body[k][s] < 0 || at[k][s] != 0) continue;
            const int start = atomicAdd(&L.n_items, count[k][s]);
            st_int(&A.inc_start[body[k][s]], start);
            if (!A.layer) {
                L.set[start] = 0;
                L.in_tail[start] = 0;
            }
        }
    __builtin_amdgcn_s_waitcnt(0);
    __syncthreads();
    int start[kPer][2];
#pragma unroll
    for (int k = 0; k < kPer; k++)
#pragma unroll
        for (int s = 0; s < 2; s++) start[k][s] = body[k][s] >= 0 ? ld_int(&A.inc_start[body[k][s]]) : 0;
#pragma unroll
    for (int k = 0; k < kPer; k++) {
        const int g = t + k * kSmallThreads;
#pragma unroll
        for (int s = 0; s < 2; s++)
            if (body[k][s] >= 0) L.item[start[k][s] + at[k][s]] = (unsigned short)g;
        if (A.layer && g < n) {
            L.lists[g].start_a = (unsigned short)start[k][0];
            L.lists[g].n_a = (unsigned short)count[k][0];
            L.lists[g].start_b = (unsigned short)start[k][1];
            L.lists[g].n_b = (unsigned short)count[k][1];
        }
    }
    __syncthreads();

    // colours
    if (!A.layer) {
        // as k_colour
        int rank[kPer][2];
        bool done[kPer];
#pragma unroll
        for (int k = 0; k < kPer; k++) {
            const int g = t + k * kSmallThreads;
            done[k] = g >= n;
#pragma unroll
            for (int s = 0; s < 2; s++)
                rank[k][s] = body[k][s] >= 0 ? colour_rank(g, count[k][s],
                                                           [&](int i) { return (int)L.item[start[k][s] + i]; })
                                             : 0;
        }
        bool left = true;
        for (int polls = 0; left; polls++) {
            if (polls > A.max_polls) {
                L.gave_up = 1;
                break;
            }
            left = false;
#pragma unroll
            for (int k = 0; k < kPer; k++) {
                unsigned long long set[2] = {0, 0};
                int tail[2] = {0, 0};
                bool ready = !done[k];
#pragma unroll
                for (int s = 0; s < 2; s++)
                    if (!done[k] && body[k][s] >= 0) {
                        set[s] = __hip_atomic_load(&L.set[start[k][s]], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
                        tail[s] = __hip_atomic_load(&L.in_tail[start[k][s]], __ATOMIC_RELAXED,
                                                    __HIP_MEMORY_SCOPE_WORKGROUP);
                        ready = ready && __popcll(set[s]) + tail[s] == rank[k][s];
                    }
                if (ready) {
                    const int c = free_colour(set[0] | set[1]);
                    L.colour[t + k * kSmallThreads] = (short)c;
#pragma unroll
                    for (int s = 0; s < 2; s++) {
                        if (body[k][s] < 0) continue;
                        if (c < kMaxColours)
                            __hip_atomic_store(&L.set[start[k][s]], set[s] | 1ull << c, __ATOMIC_RELAXED,
                                               __HIP_MEMORY_SCOPE_WORKGROUP);
                        else
                            __hip_atomic_store(&L.in_tail[start[k][s]], (unsigned short)(tail[s] + 1), __ATOMIC_RELAXED,
                                               __HIP_MEMORY_SCOPE_WORKGROUP);
                    }
                    done[k] = true;
                }
                left = left || __any(!done[k]);
            }
        }
    } else {
        auto get = [](const short* p) {
            return (int)__hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        };
        auto set = [](short* p, int v) {
            __hip_atomic_store(p, (short)v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        };
        bool left = true;
        for (int polls = 0; __any(left); polls++) {
            if (polls > A.max_polls) {
                L.gave_up = 1;
                break;
            }
            left = false;
            for (int g = t / 4; g < n; g += kSmallThreads / 4) {
                if (get(&L.colour[g]) >= 0) continue;
                int bl = get(&L.sorted[g]);
                int c = -1;
                if (bl < 0 || get(&L.colour[bl]) >= 0) {
                    const auto l = L.lists[g];
                    c = try_layered(
                        g, ColourLists{l.start_a, l.n_a, l.start_b, l.n_b}, [&](int h) { return get(&L.colour[h]); },
                        [&](int i) { return (int)L.item[i]; }, [&](int h) { return A.layer[h]; }, bl);
                    if (c >= 0) set(&L.colour[g], c);
                    else set(&L.sorted[g], bl);
                }
                left = left || c < 0;
            }
        }
    }
    __syncthreads();
    if (L.gave_up) {
        if (t == 0) A.colour_start[kWordLeft] = 1;
        return;
    }

    // sorted positions: a stable counting sort over (colour, larger groups first)
    for (int i = t; i < kSmallWaves * (kSmallBins + 7); i += kSmallThreads) (&L.hist[0][0])[i] = 0;
    __syncthreads();
    const int chunk = ((n + kSmallThreads - 1) / kSmallThreads) * 64;  // of a wave
    auto bin_of = [&](int g) {
        const int c = L.colour[g];
        return c < kMaxColours ? c * 16 + 15 - min(A.group_start[g + 1] - A.group_start[g], 15) : kSmallBins - 1;
    };
    int bin[kPer];
#pragma unroll
    for (int k = 0; k < kPer; k++) {
        const int g = wave * chunk + 64 * k + lane;
        const bool in = 64 * k < chunk && g < n;
        bin[k] = in ? bin_of(g) : 0;
        const unsigned long long m = same_key(bin[k], in);
        if (in && __ffsll((long long)m) - 1 == lane) L.hist[wave][bin[k]] += (unsigned short)__popcll(m);
        lds_order();
    }
    __syncthreads();
    {
        int sum = 0;
        for (int v = 0; v < kSmallWaves; v++) sum += L.hist[v][t];
        const int base = small_exclusive(sum, L.wave_sum);
        int run = base;
        for (int v = 0; v < kSmallWaves; v++) {
            const int count = L.hist[v][t];
            L.hist[v][t] = (unsigned short)run;
            run += count;
        }
        if (t % 16 == 0) L.cs[t / 16] = base;
        if (t == kSmallThreads - 1) {  // the tail's bin
            L.cs[kMaxColours] = run;
            L.cs[kMaxColours + 1] = n;
            for (int v = 0; v < kSmallWaves; v++) {
                const int count = L.hist[v][kSmallBins - 1];
                L.hist[v][kSmallBins - 1] = (unsigned short)run;
                run += count;
            }
        }
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < kPer; k++) {
        const int g = wave * chunk + 64 * k + lane;
        const bool in = 64 * k < chunk && g < n;
        const unsigned long long m = same_key(bin[k], in);
        const int q = L.hist[wave][bin[k]] + __popcll(m & ((1ull << lane) - 1));
        lds_order();
        if (in && __ffsll((long long)m) - 1 == lane) L.hist[wave][bin[k]] += (unsigned short)__popcll(m);
        lds_order();
        if (in) L.sorted[q] = (short)g;
    }
    __syncthreads();
    // the tail in the order of its colours
    const int tail = L.cs[kMaxColours], n_tail = n - tail;
    if (A.layer && n_tail > 1) {
        int to[kPer], who[kPer];
#pragma unroll
        for (int k = 0; k < kPer; k++) {
            const int i = t + k * kSmallThreads;
            if (i >= n_tail) continue;
            who[k] = L.sorted[tail + i];
            const int c = L.colour[who[k]];
            int before = 0;
            for (int j = 0; j < n_tail; j++) {
                const int cj = L.colour[L.sorted[tail + j]];
                before += cj < c || (cj == c && j < i) ? 1 : 0;
            }
            to[k] = before;
        }
        __syncthreads();
#pragma unroll
        for (int k = 0; k < kPer; k++)
            if (t + k * kSmallThreads < n_tail) L.sorted[tail + to[k]] = (short)who[k];
        __syncthreads();
    }

    // positions of the groups and their contacts
    {
        int size[kPer], sum = 0;
#pragma unroll
        for (int k = 0; k < kPer; k++) {
            const int q = t * kPer + k;
            size[k] = 0;
            if (q < n) {
                const int g = L.sorted[q];
                L.colour[g] = (short)q;
                size[k] = A.group_start[g + 1] - A.group_start[g];
            }
            sum += size[k];
        }
        int run = small_exclusive(sum, L.wave_sum);
#pragma unroll
        for (int k = 0; k < kPer; k++) {
            const int q = t * kPer + k;
            if (q <= n) {
                L.pos[q] = run;
                A.pos_start[q] = run;
            }
            run += size[k];
        }
        if (t == kSmallThreads - 1 && n == kSmallLayout) {
            L.pos[n] = run;
            A.pos_start[n] = run;
        }
    }
    if (t <= kMaxColours + 1) A.colour_start[t] = L.cs[t];
    if (t < 2) L.plan[t] = 0;
    if (t == 2) L.one_body = 0;
    __syncthreads();
    for (int q = t / 4; q < n; q += kSmallThreads / 4) {
        const int g = L.sorted[q], o = L.pos[q], size = L.pos[q + 1] - o, k0 = A.group_start[g];
        const int a = A.ga[g], b = A.gb[g];
        for (int k = t & 3; k < size; k += 4) {
            A.order[o + k] = k0 + k;
            A.pos_a[o + k] = a;
        }
        if ((t & 3) == 0) reinterpret_cast<int4*>(A.group_desc)[q] = make_int4(o, o + size, a, b);
    }
    // flow ranks (k_flow_ranks): a thread per group and side
    for (int i = t; i < 2 * n; i += kSmallThreads) {
        const int q = i >> 1, g = L.sorted[q], e = (i & 1) ? A.gb[g] : A.ga[g];
        int rank = 0, deg = 0, pred = 0;
        if (dynamic_body(A.bflags, e)) {
            const int s0 = ld_int(&A.inc_start[e]);
            deg = ld_int(&A.inc_count[e]);
            int of;
            rank = flow_rank(q, deg, [&](int k) { return (int)L.colour[L.item[s0 + k]]; }, of);
            pred = 2 * of + (A.ga[L.sorted[of]] == e ? 0 : 1);
            if ((i & 1) && e == A.ga[g]) L.one_body = 1;
        }
        reinterpret_cast<int2*>(A.flow)[i] = make_int2(rank, deg);
        A.pred[i] = pred;
    }
    // the resident kernel's plan
    if (A.waves > 0) {
        resident_steps(L.cs, A.waves, L.steps);
        if (t < A.waves) {
            int sum = 0, steps = 0, q0, count;
            StepWalk walk;
            while (walk.next(L.steps, A.waves, t, q0, count)) {
                sum += count * kResGroup + min(L.pos[q0 + count] - L.pos[q0], kResDoubles) * kResContact;
                steps++;
                if (sum > kResDoubles || steps > kResidentSteps) break;
            }
            A.used[t] = sum;
            int total = sum;
#pragma unroll
            for (int o = 1; o < kResWaves; o <<= 1) total += __shfl_xor(total, o, 64);
            atomicMax(&L.plan[0], total);
            atomicMax(&L.plan[1], steps);
        }
    }
    __syncthreads();
    if (t < 2) A.colour_start[kWordPlan + t] = L.plan[t];
    if (t == 2) A.colour_start[kWordOneBody] = L.one_body;
    if (t == 3) A.colour_start[kWordLeft] = 0;
}
void launch_layout_small(hipStream_t s, const SmallLayoutArgs& A) {
    hipLaunchKernelGGL(k_layout_small, dim3(1), dim3(kSmallThreads), 0, s, A);
}

AMD_INLINE int lds_int(const int* p) { return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP); }
AMD_INLINE void set_lds_int(int* p, int v) { __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP); }
AMD_INLINE void lds_landed() { __builtin_amdgcn_s_waitcnt(0xC07F); }  // lgkmcnt(0)

// One contact as a lane of its quad needs it: its three J entries and update
// coefficients per row, and the contact's scalars.
typedef double d2v __attribute__((ext_vector_type(2)));
struct QuadRec {
    double j[3][3], c[3][3];
    double b[3], d[3], den[3], y[3], mu, lam[3];
};
struct QuadMap {
    int ofs;        // of this kind of lane in a row
    unsigned sign;  // A.v lanes: their entries are -jb.v
};
// at: the contact in LDS; lam: its lambda and mu for this pass
AMD_INLINE void read_quad_rec(const double* at, const double* lam, const QuadMap& m, QuadRec& w) {
#pragma unroll
    for (int r = 0; r < 3; r++) {
        const d2v* q = reinterpret_cast<const d2v*>(at + r * kResRow + m.ofs);
        const d2v q0 = q[0], q1 = q[1], q2 = q[2];
        w.j[r][0] = q0.x;
        w.j[r][1] = q0.y;
        w.j[r][2] = q1.x;
        w.c[r][0] = q1.y;
        w.c[r][1] = q2.x;
        w.c[r][2] = q2.y;
        const d2v* sc = reinterpret_cast<const d2v*>(at + kResScalars + 4 * r);
        const d2v s0 = sc[0], s1 = sc[1];
        w.b[r] = s0.x;
        w.d[r] = s0.y;
        w.den[r] = s1.x;
        w.y[r] = s1.y;
    }
    const d2v* l = reinterpret_cast<const d2v*>(lam);
    const d2v l0 = l[0], l1 = l[1];
    w.lam[0] = l0.x;
    w.lam[1] = l0.y;
    w.lam[2] = l1.x;
    w.mu = l1.y;
}
// The places (one or two, else -1) in a contact in LDS of double d of its record.
AMD_INLINE void resident_places(int d, int& first, int& second) {
    first = second = -1;
    if (d >= kRecLambda) {
        if (d < kRecLambda + 3) {
            first = kResLam + d - kRecLambda;
            second = kResLamOdd + d - kRecLambda;
        }
        return;
    }
    const int r = d / kRecRow, q = (d % kRecRow) / 4, i = d % 4, row = r * kResRow;
    if (i == 3) {
        if (q < 4) {
            first = kResScalars + 4 * r + q;  // b, D, D + C, its reciprocal
        } else if (r == 0) {
            first = kResLam + 3;
            second = kResLamOdd + 3;
        }
        return;
    }
    if (q == 0) {
        first = row + kResV + i;
        second = row + kResV + 3 + i;
    } else {
        first = row + i + (q == 1 ? kResAw : q == 2 ? kResBw : q == 3 ? kResAw + 3 : kResBw + 3);
    }
}
static_assert(kRecB == 3 && kRecD == 7 && kRecDen == 11 && kRecY == 15 && kRecMu == 19, "resident_places");
// Contact.getJdv (Contact.java:362-378), the same sum in every lane of the
// quad.  kExact flips the A.v lanes' entries; otherwise their sum is flipped,
// which differs only in the sign of a zero.
template <bool kExact>
AMD_INLINE double quad_jdv(const double (&j)[3], unsigned sign, const double (&dv)[3]) {
    double s;
    if (kExact) {
        s = flip(j[0], sign) * dv[0] + flip(j[1], sign) * dv[1] + flip(j[2], sign) * dv[2];
    } else {
        s = flip(j[0] * dv[0] + j[1] * dv[1] + j[2] * dv[2], sign);
    }
    const double h = s + dpp_d<kQuadSwap1>(s);
    return h + dpp_d<kQuadSwap2>(h);
}
// f: minv on v lanes, 1 on w lanes, negative on A.v lanes ((-f dl) c is (f dl)
// (-c) exactly)
AMD_INLINE void quad_apply(const double (&c)[3], double f, double dl, double (&dv)[3]) {
    const double s = f * dl;
#pragma unroll
    for (int i = 0; i < 3; i++) dv[i] = s * c[i] + dv[i];
}

// row_contact_fast on a quad: the conditions are those of FastCheck, with the
// numerators' range as one unsigned distance from its lower end.  There a
// numerator is normal and nonzero, so the sign of a zero J.dv changes nothing,
// and min and max are the plain selects (a limit of +0 against -l gives -0 in
// both).
struct QuadCheck {
    unsigned num = 0;    // max of 2 |numerator|'s high word - 2 * 0x30500000
    unsigned limit = 0;  // max high word of the friction limits (sign included)
    AMD_INLINE bool ok() const { return num < 2u * (0x4F900000u - 0x30500000u) && limit < 0x7FF00000u; }
};
AMD_INLINE void quad_contact_fast(double omega, const QuadRec& c, unsigned sign, double f, double (&dv)[3], double& mx,
                                  QuadCheck& chk, double (&lam)[3]) {
#pragma unroll
    for (int r = 0; r < 3; r++) {
        const double jd = quad_jdv<false>(c.j[r], sign, dv);
        const double num = c.d[r] * c.lam[r] - omega * (c.b[r] + jd);
        unsigned h = hi_word(num);
        asm("" : "+v"(h));  // else the shift becomes a 64-bit one
        chk.num = max(chk.num, (h << 1) - 2u * 0x30500000u);
        const double q0 = num * c.y[r];
        const double rr = __builtin_fma(-c.den[r], q0, num);
        double l = __builtin_fma(rr, c.y[r], q0);
        if (r == 0) {
            l = __builtin_fmax(l, 0.0);
        } else {
            const double limit = c.mu * lam[0];
            chk.limit = max(chk.limit, hi_word(limit));
            l = __builtin_fmin(__builtin_fmax(l, -limit), limit);
        }
        lam[r] = l;
        const double diff = l - c.lam[r];
        quad_apply(c.c[r], f, diff, dv);
        mx = fmax(mx, fabs(diff));
    }
}
// row_contact on a quad: every form of the update
AMD_INLINE void quad_contact(double omega, const QuadRec& c, bool clamp, unsigned sign, double f, double (&dv)[3],
                             double& mx, bool& nan, double (&lam)[3]) {
#pragma unroll
    for (int r = 0; r < 3; r++) {
        const double jd = quad_jdv<true>(c.j[r], sign, dv);
        const double prev = c.lam[r];
        const double num = c.d[r] * prev - omega * (c.b[r] + jd);
        double l = div_row(num, c.den[r], c.y[r]);
        double lc;
        if (r == 0) {
            lc = jmax(0, l);
        } else {
            const double limit = c.mu * lam[0];
            lc = jmin(jmax(l, -limit), limit);
        }
        l = clamp ? lc : l;
        lam[r] = l;
        const double diff = l - prev;
        quad_apply(c.c[r], f, diff, dv);
        mx = fmax(mx, fabs(diff));
        nan = nan || diff != diff;
    }
}

// The pass keeper: one wave of the workgroup.  Workgroups count themselves in
// at a sweep's arrival words (kPassWords of them, a cache line apart); workgroup
// 0's keeper alone reads those, and leaves the verdict in one word that the
// others read: with every keeper polling the arrival words, the adds took
// longer to get through than a pass.
AMD_INLINE void keep_passes(const FlowArgs& F, ResidentLds& L, int lane) {
    const PgsArgs& P = F.P;
    const int lastp = P.iterations;
    unsigned long long* verdict = F.pass_done;  // sweeps known not to have converged | converged sweep << 32
    unsigned long long* arrive = F.pass_done + kPassStride;
    int a = 1;    // next sweep of this workgroup to report
    int chk = 0;  // sweeps 1..chk are known not to have converged
    long spins = 0;
    while (true) {
        bool moved = false;
        if (a <= lastp && __all(lds_int(&L.done[lane & (kResWaves - 1)]) >= a)) {
            // Math.max over the quads, by the bits (non-negative doubles order as
            // their bits, a NaN above all)
            unsigned long long mx = (unsigned long long)__double_as_longlong(
                __hip_atomic_load(&L.pass_max[a & 3][lane], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP));
#pragma unroll
            for (int o = 32; o > 0; o >>= 1) {
                const unsigned long long v = __shfl_xor(mx, o, 64);
                mx = v > mx ? v : mx;
            }
            if (lane == 0) {
                const bool over = mx && !(__longlong_as_double((long long)mx) < P.tolerance);  // NaN over
                if (P.check_tolerance)
                    __hip_atomic_fetch_add(&arrive[((size_t)a * kPassWords + blockIdx.x % kPassWords) * kPassStride],
                                           (1ull << 32) | (over ? 1ull : 0ull), __ATOMIC_RELAXED,
                                           __HIP_MEMORY_SCOPE_AGENT);
                if (mx) atomicMax(&P.iter_max[a - 1], mx);
                // the ring's entries are written again four passes on, which wait for this
                set_lds_int(&L.published, a);
            }
            a++;
            moved = true;
        }
        if (P.check_tolerance && chk < lastp - 1) {
            int known = chk, stop = 0;
            if (blockIdx.x == 0) {
                if (chk + 1 < a) {
                    const unsigned long long v =
                        lane < kPassWords ? ld_cnt64(&arrive[((size_t)(chk + 1) * kPassWords + lane) * kPassStride]) : 0;
                    int here = (int)(v >> 32), over = (int)(unsigned)v;
#pragma unroll
                    for (int o = 1; o < kPassWords; o <<= 1) {
                        here += __shfl_xor(here, o, 64);
                        over += __shfl_xor(over, o, 64);
                    }
                    if (uniform(here) == (int)gridDim.x) {
                        if (uniform(over) == 0) stop = chk + 1;
                        else known = chk + 1;
                        if (lane == 0)
                            __hip_atomic_store(verdict, ((unsigned long long)stop << 32) | (unsigned)known,
                                               __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                    }
                }
            } else if (chk + 1 < a) {
                const unsigned long long v = ld_cnt64(verdict);
                known = uniform((int)(unsigned)v);
                stop = uniform((int)(v >> 32));
            }
            if (known != chk) {
                chk = known;
                if (lane == 0) set_lds_int(&L.known, chk);
                moved = true;
            }
            if (stop) {
                if (lane == 0) set_lds_int(&L.stop, stop);
                return;
            }
        } else if (a > lastp) {
            return;
        }
        if (moved) {
            spins = 0;
            continue;
        }
        if (uniform(lds_int(&L.failed))) return;
        if (++spins > kLdsSpinLimit ||
            ((spins & 255) == 0 && uniform(__hip_atomic_load(P.error, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)))) {
            if (lane == 0) {
                atomicOr(P.error, 1);
                set_lds_int(&L.failed, 1);
            }
            return;
        }
        __builtin_amdgcn_s_sleep(1);
    }
}

template <bool kScenes>
__global__ __launch_bounds__((kResWaves + 1) * 64) __attribute__((amdgpu_waves_per_eu(1, 2))) void k_pgs_resident(
    FlowArgs F) {
    __shared__ ResidentLds L;
    const PgsArgs& P = F.P;
    const int* cs = P.colour_start;
    const int W = gridDim.x * kResWaves;
    const int wave = uniform((int)threadIdx.x >> 6), lane = threadIdx.x & 63;
    if (threadIdx.x == 0) {
        L.published = L.known = L.stop = L.failed = 0;
        for (int i = 0; i < kResWaves; i++) L.done[i] = 0;
    }
    resident_steps(cs, W, L.steps);
    if (wave == kResWaves) {
        keep_passes(F, L, lane);
        return;
    }
    const int w = blockIdx.x * kResWaves + wave;
    const int quad = lane >> 2, lt = lane & 3, side = lt >> 1, wpart = lt & 1;
    const bool lead = lt == 0;
    const int first = P.warm_start ? 0 : 1;
    const int lastp = P.iterations;
    const double omega = P.omega;
    const int4* gdesc = reinterpret_cast<const int4*>(P.group_desc);
    double* reg = reinterpret_cast<double*>(&L.region[0]);
    int room = 0;  // this wave's part of the region ends there
    int off = 0;
    for (int v = 0; v <= wave; v++) {
        off = room;
        room += F.resident_used[blockIdx.x * kResWaves + v];
    }
    room = min(room, kResDoubles);
    QuadMap map;
    map.ofs = lt == 1 ? kResAw : lt == 3 ? kResBw : kResV;
    map.sign = lt == 0 ? 0x80000000u : 0u;

    // take this wave's groups into LDS
    int n_steps = 0;
    {
        const double* start_dv = (first & 1) ? P.dv : F.dv_alt;
        const int4* fdesc = reinterpret_cast<const int4*>(F.flow);
        const int2* gpred = reinterpret_cast<const int2*>(F.pred);
        const double2* recs = reinterpret_cast<const double2*>(P.rec);
        // a lane copies 16 bytes of a record, the two halves of the wave two records
        int to[4];
        resident_places(2 * (lane & 31), to[0], to[1]);
        resident_places(2 * (lane & 31) + 1, to[2], to[3]);
        StepWalk walk;
        int q0 = 0, count = 0;
        int4 gd = make_int4(0, 0, 0, 0), fd = gd;
        int2 pr = make_int2(0, 0);
        auto fetch = [&]() -> bool {
            if (!walk.next(L.steps, W, w, q0, count)) return false;
            const int q = q0 + (quad < count ? quad : 0);
            gd = gdesc[q];
            fd = fdesc[q];
            pr = gpred[q];
            return true;
        };
        bool more = fetch();
        while (more) {
            const int4 g = gd, fl = fd;
            const int2 pd = pr;
            const int q_first = q0, n_groups = count;
            more = fetch();
            const bool has = quad < n_groups;
            const int k0 = uniform(g.x), contacts = __builtin_amdgcn_readlane(g.y, 4 * (n_groups - 1)) - k0;
            const int first_contact = off + n_groups * kResGroup;
            if (n_steps >= kResidentSteps || contacts > kResDoubles ||
                first_contact + contacts * kResContact > room) {  // the plan allows none of these
                if (lane == 0) {
                    atomicOr(P.error, 1);
                    set_lds_int(&L.failed, 1);
                }
                return;
            }
            const int e = side ? g.w : g.z, rank = side ? fl.z : fl.x, deg = side ? fl.w : fl.y;
            double v[3], minv = 0.0;
            int extra = 0;
            if (has) {
#pragma unroll
                for (int i = 0; i < 3; i++) v[i] = ld_coherent(&start_dv[e * 6 + 3 * wpart + i]);
                minv = P.minv[e];
                if (kScenes) {
                    extra = P.g_scene[q_first + quad];
                    if (side) extra = (int)P.scene_groups[extra];
                }
            }
            bool plain = true;
            constexpr int kAhead = 4;  // pairs of records in flight
            for (int i0 = 0; i0 < contacts; i0 += 2 * kAhead) {
                double2 d[kAhead];
#pragma unroll
                for (int u = 0; u < kAhead; u++) {
                    const int i = min(i0 + 2 * u + (lane >> 5), contacts - 1);
                    d[u] = recs[(size_t)(k0 + i) * kRec2 + (lane & 31)];
                }
#pragma unroll
                for (int u = 0; u < kAhead; u++) {
                    const int i = min(i0 + 2 * u + (lane >> 5), contacts - 1);
                    double* at = reg + first_contact + i * kResContact;
                    if (to[0] >= 0) at[to[0]] = d[u].x;
                    if (to[1] >= 0) at[to[1]] = d[u].x;
                    if (to[2] >= 0) at[to[2]] = d[u].y;
                    if (to[3] >= 0) at[to[3]] = d[u].y;
                    if ((lane & 31) == kRecClamp / 2) plain = plain && (kRecClamp % 2 ? d[u].y : d[u].x) == 1.0;
                }
            }
            int nmax = has ? g.y - g.x : 0;
#pragma unroll
            for (int o = 4; o < 64; o <<= 1) nmax = max(nmax, __shfl_xor(nmax, o, 64));
            plain = __all(plain);
            if (lane == 0) {
                L.step[wave][n_steps] =
                    make_int4(off, q_first, n_groups | (plain ? 0x80 : 0) | (nmax << 8), contacts);
                L.step_k0[wave][n_steps] = k0;
            }
            if (has) {
                double* blk = reg + off + quad * kResGroup + side * kResSide;
#pragma unroll
                for (int i = 0; i < 3; i++) blk[3 * wpart + i] = v[i];
                if (wpart == 0) {
                    const int flags = (deg ? kSideDyn : 0) | (deg == 1 ? kSideSelf : 0) | (rank == 0 ? kSideRank0 : 0) |
                                      (rank == deg - 1 ? kSideLast : 0);
                    auto pack = [](int lo, int hi) {
                        return __longlong_as_double(((long long)hi << 32) | (unsigned)lo);
                    };
                    blk[kResF] = minv;
                    blk[kResFirst] = pack(first_contact + (g.x - k0) * kResContact, g.y - g.x);
                    blk[kResInts] = pack(e, side ? pd.y : pd.x);
                    blk[kResInts + 1] = pack(flags, extra);
                }
            }
            off = first_contact + contacts * kResContact;
            n_steps++;
        }
    }

    // bookkeeping of the next step
    struct Next {
        int q0, count, nmax;
        bool plain;
        double* blk;
        double f;
        long long where, who, what;  // first contact and contacts; body and incidence; flags and extra
    } nx;
    auto next_step = [&](int s) {
        const int4 T = L.step[wave][s];
        const int goff = uniform(T.x);
        nx.q0 = uniform(T.y);
        nx.count = uniform(T.z) & 0x7f;
        nx.plain = uniform(T.z) & 0x80;
        nx.nmax = uniform(T.z) >> 8;
        nx.blk = reg + goff + (quad < nx.count ? quad : 0) * kResGroup + side * kResSide;
        nx.f = nx.blk[kResF];
        nx.where = __double_as_longlong(nx.blk[kResFirst]);
        nx.who = __double_as_longlong(nx.blk[kResInts]);
        nx.what = __double_as_longlong(nx.blk[kResInts + 1]);
    };
    if (n_steps > 0) next_step(0);
    for (int p = first; p <= lastp; p++) {
        // pass gates: sweep p-2 must be known not converged (p-1 for the last
        // sweep), and the workgroup's pass ring must have room
        if (p >= 2) {
            const int need = !P.check_tolerance ? 0 : p == lastp ? p - 1 : p - 2;
            bool leave = false;
            for (long spins = 0;; spins++) {
                const int stop = uniform(lds_int(&L.stop)), known = uniform(lds_int(&L.known)),
                          pub = uniform(lds_int(&L.published));
                // every wave runs the sweep after the converged one and leaves then
                leave = (stop && stop <= need) || uniform(lds_int(&L.failed));
                if (leave || (known >= need && pub >= p - 3)) break;
                if (spins > 4 * kLdsSpinLimit) {  // the keeper gives up long before
                    if (lane == 0) atomicOr(P.error, 1);
                    leave = true;
                    break;
                }
                __builtin_amdgcn_s_sleep(1);
            }
            if (leave) break;
        }
        const bool last = p == lastp;
        const int lam_r = (p >= 1 && ((p - 1) & 1)) ? kResLamOdd : kResLam, lam_w = (p & 1) ? kResLamOdd : kResLam;
        double* cur = (p & 1) ? F.dv_alt : P.dv;
        const double* prv = (p & 1) ? P.dv : F.dv_alt;
        double mx = 0.0;
        bool nan = false;
        for (int s = 0; s < n_steps; s++) {
            // this step's bookkeeping was read during the one before
            const int q0 = nx.q0, nmax = nx.nmax;
            const bool plain = nx.plain;
            // A quad without a group runs the first one's again and keeps the
            // result to itself: a wave with most of its lanes switched off takes
            // longer over a contact, not less (1000 to 1600 cycles, against 670).
            const bool owner = quad < nx.count;
            const int group = q0 + (owner ? quad : 0);
            bool skipped = false;
            double* blk = nx.blk;
            const int e = (int)nx.who, pred = (int)(nx.who >> 32), flags = (int)nx.what, extra = (int)(nx.what >> 32);
            const double f = wpart ? 1.0 : lead ? -nx.f : nx.f;
            double* rec = reg + (int)nx.where;
            int n = (int)(nx.where >> 32);
            auto load = [&](int t, QuadRec& rc) {
                const double* at = rec + min(t, max(n - 1, 0)) * kResContact;
                read_quad_rec(at, at + lam_r, map, rc);
            };
            QuadRec ra, rb;
            // inputs: LDS for pinned bodies and bodies of this group alone, the
            // launch buffer for a body's first update, else the slot of the
            // body's previous update
            double dv[3] = {blk[3 * wpart], blk[3 * wpart + 1], blk[3 * wpart + 2]};
            double* src = nullptr;
            const bool own = !(flags & kSideDyn) || (flags & kSideSelf);
            if (!own) {
                if (p == first && (flags & kSideRank0)) {
#pragma unroll
                    for (int i = 0; i < 3; i++) dv[i] = ld_coherent(&prv[e * 6 + 3 * wpart + i]);
                } else {
                    src = slot_at(F, (flags & kSideRank0) ? ((p - 1) & 1) : (p & 1), pred) + 4 * wpart;
                }
            }
            // the first poll is on its way while the first record is read
            double v0 = 0.0, v1 = 0.0, v2 = 0.0;
            if (src) {
                v0 = ld_coherent(src);
                v1 = ld_coherent(src + 1);
                v2 = ld_coherent(src + 2);
            }
            load(0, ra);
            {
                bool got = src == nullptr;
                long spins = 0;
                auto spin = [&]() -> bool {  // false: give up (error flag set)
                    __builtin_amdgcn_s_sleep(1);
                    if (!got) {
                        v0 = ld_coherent(src);
                        v1 = ld_coherent(src + 1);
                        v2 = ld_coherent(src + 2);
                    }
                    if (++spins > kFlowSpinLimit ||
                        ((spins & 255) == 0 &&
                         uniform(__hip_atomic_load(P.error, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)))) {
                        if (lane == 0) {
                            atomicOr(P.error, 1);
                            set_lds_int(&L.failed, 1);
                        }
                        return false;
                    }
                    return true;
                };
                auto poll = [&]() {
                    if (!got) {
                        auto filled = [](double v) { return (unsigned long long)__double_as_longlong(v) != kSlotEmpty; };
                        if (filled(v0) && filled(v1) && filled(v2)) {
                            dv[0] = v0;
                            dv[1] = v1;
                            dv[2] = v2;
                            got = true;
                        }
                    }
                };
                const int t1 = p - 2, t2 = last ? p - 1 : 0;
                if (!(kScenes && p >= 1 && P.check_tolerance && (t1 >= 1 || t2 >= 1))) {
                    while (true) {
                        poll();
                        if (__all(got)) break;
                        if (!spin()) return;
                    }
                } else {
                    // Per-scene exits, as in k_pgs_flow: a group whose scene was
                    // under the tolerance at sweep p-2 or p-3 (p-1 before the
                    // last) skips this pass and every later one.
                    bool resolved = !lead, skip = false;
                    unsigned want = 0;
                    if (lead) want = (unsigned)(__double_as_longlong(blk[kResSide + kResInts + 1]) >> 32);
                    const unsigned long long* cnt = &P.scene_done[(size_t)(lead ? extra : 0) * (P.iterations + 1)];
                    const int ta = t1 >= 1 ? t1 : t2, tb = t1 >= 2 ? t1 - 1 : ta, tc = t2 >= 1 ? t2 : ta;
                    while (true) {
                        poll();
                        if (!resolved) {
                            const unsigned long long wa = ld_cnt64(&cnt[ta]), wb = ld_cnt64(&cnt[tb]),
                                                     wc = ld_cnt64(&cnt[tc]);
                            if ((unsigned)(wa >> 32) == want && (unsigned)(wb >> 32) == want &&
                                (unsigned)(wc >> 32) == want) {
                                skip = (unsigned)wa == 0u || (unsigned)wb == 0u || (unsigned)wc == 0u;
                                resolved = true;
                            }
                        }
                        const int flagged = (resolved ? 1 : 0) | (skip ? 2 : 0);
                        const int of_quad = __builtin_amdgcn_mov_dpp(flagged, kQuadLane0, 0xF, 0xF, true);
                        if (__all((of_quad & 1) && ((of_quad & 2) || got))) {
                            if (of_quad & 2) {
                                skipped = true;
                                n = 0;
                                src = nullptr;
                            }
                            break;
                        }
                        if (!spin()) return;
                    }
                }
            }
            // the inputs were the last loads: this wave's stores of the pass before have landed
            __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0)
            double smx = 0.0;
            bool snan = false;
            double lam[3];
            // every lane of the quad writes the same values to the same place
            auto keep_lambda = [&](int t) {
                double* to = rec + t * kResContact + lam_w;
                to[0] = lam[0];
                to[1] = lam[1];
                to[2] = lam[2];
            };
            // Contact.updateContactState (Contact.java:385-398)
            auto state = [&](int t, const QuadRec& c) {
                const double w1 = c.b[1] + quad_jdv<true>(c.j[1], map.sign, dv);
                const double w2 = c.b[2] + quad_jdv<true>(c.j[2], map.sign, dv);
                if (lead && owner) {
                    int st;
                    if (fabs(lam[0]) <= 1e-14) st = AM_STATE_BROKEN;
                    else if (fabs(w1) > P.sliding) st = AM_STATE_ONEDGE;
                    else if (fabs(w2) > P.sliding) st = AM_STATE_ONEDGE;
                    else st = AM_STATE_CLEAR;
                    P.sstate[gdesc[group].x + t] = st;
                }
            };
            // sweeps but the last (whose contacts get their states) try the
            // fast update; the general one runs again from the step's start
            lds_landed();
            bool general = p == 0 || last || !plain;
            if (!general) {
                const double dv0[3] = {dv[0], dv[1], dv[2]};
                QuadCheck chk;
                // A record is read while the one before it runs; the wait for it
                // stands before the reads of the one after it (their number is
                // more than the counter of LDS operations tells apart)
                auto one = [&](int t, const QuadRec& now, QuadRec& then) {
                    if (t < n) {
                        load(t + 1, then);
                        quad_contact_fast(omega, now, map.sign, f, dv, smx, chk, lam);
                    }
                    lds_landed();
                    if (t < n) keep_lambda(t);
                };
                for (int t = 0; t < nmax; t += 2) {
                    one(t, ra, rb);
                    if (t + 1 >= nmax) break;
                    one(t + 1, rb, ra);
                }
                if (__builtin_expect(!__all(chk.ok()), 0)) {
                    dv[0] = dv0[0];
                    dv[1] = dv0[1];
                    dv[2] = dv0[2];
                    smx = 0.0;
                    general = true;
                }
            }
            if (general) {
                for (int t = 0; t < nmax; t++) {
                    load(t, ra);
                    if (t >= n) continue;
                    if (p == 0) {
                        // confidentWarmStart (PGS.java:250-256)
#pragma unroll
                        for (int r = 0; r < 3; r++) quad_apply(ra.c[r], f, ra.lam[r], dv);
                        continue;
                    }
                    const bool clamp = P.rec[(size_t)(gdesc[group].x + t) * kRecDoubles + kRecClamp] != 0.0;
                    quad_contact(omega, ra, clamp, map.sign, f, dv, smx, snan, lam);
                    keep_lambda(t);
                    if (last) state(t, ra);
                }
            }
            // publish: the next update's slot, or LDS for a body of this group
            // alone; the body's last update of a pass also to the pass's buffer
            if (owner && !skipped && (flags & kSideDyn)) {
                if (flags & kSideSelf) {
#pragma unroll
                    for (int i = 0; i < 3; i++) blk[3 * wpart + i] = dv[i];
                } else {
                    double* dst = slot_at(F, p & 1, 2 * group + side) + 4 * wpart;
#pragma unroll
                    for (int i = 0; i < 3; i++) st_coherent(dst + i, dv[i]);
                }
                if (flags & kSideLast)
#pragma unroll
                    for (int i = 0; i < 3; i++) st_coherent(&cur[e * 6 + 3 * wpart + i], dv[i]);
            }
            // the slot that was read is empty again only now, behind the values
            // that the next update waits for
            if (src && owner)
#pragma unroll
                for (int i = 0; i < 3; i++) st_coherent(src + i, __longlong_as_double((long long)kSlotEmpty));
            if (n_steps > 1) next_step(s + 1 < n_steps ? s + 1 : 0);
            mx = fmax(mx, smx);
            nan = nan || snan;
            if (kScenes && p >= 1 && P.per_scene && owner && lead) {
                const size_t sc = (size_t)extra;
                if (!skipped && !(smx <= 0))
                    atomicMax(&P.scene_max[sc * P.iterations + p - 1],
                              (unsigned long long)__double_as_longlong(
                                  snan ? __longlong_as_double(0x7ff8000000000000ll) : smx));
                // over the tolerance (NaN included), as the scene's max would be
                const bool over = !skipped && !(smx <= 0) && (snan || !(smx < P.tolerance));
                __hip_atomic_fetch_add(&P.scene_done[sc * (P.iterations + 1) + p], (1ull << 32) | (over ? 1ull : 0ull),
                                       __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            }
        }
        if (p >= 1) {
            if (nan) mx = __longlong_as_double(0x7ff8000000000000ll);
            L.pass_max[p & 3][wave * kQuads + quad] = mx;  // the same from every lane of the quad
            lds_order();
            set_lds_int(&L.done[wave], p);
        }
    }
    // lambdas of the last even and the last odd pass; k_unpack takes the one
    // that the sweeps used say
    for (int s = 0; s < n_steps; s++) {
        const int4 T = L.step[wave][s];
        const int goff = uniform(T.x), count = uniform(T.z) & 0x7f, contacts = uniform(T.w);
        const int k0 = uniform(L.step_k0[wave][s]);
        const double* at = reg + goff + count * kResGroup;
        for (int i = lane; i < 3 * contacts; i += 64) {
            const int t = i / 3, r = i - 3 * t;
            P.rec[(size_t)(k0 + t) * kRecDoubles + kRecLambda + r] = at[t * kResContact + kResLam + r];
            if (lastp >= 1) F.lam_alt[4 * (size_t)(k0 + t) + r] = at[t * kResContact + kResLamOdd + r];
        }
    }
}

int pgs_resident_max_blocks(bool* ok) {
    int dev = 0, n_cu = 0, a = 0, b = 0;
    (void)hipGetDevice(&dev);
    (void)hipDeviceGetAttribute(&n_cu, hipDeviceAttributeMultiprocessorCount, dev);
    (void)hipOccupancyMaxActiveBlocksPerMultiprocessor(&a, k_pgs_resident<false>, (kResWaves + 1) * 64, 0);
    (void)hipOccupancyMaxActiveBlocksPerMultiprocessor(&b, k_pgs_resident<true>, (kResWaves + 1) * 64, 0);
    *ok = std::min(a, b) > 0;
    return n_cu * std::min(a, b);
}

// Sweeps used: the first converged sweep, else all (threads that fall below it find nothing)
AMD_INLINE int first_converged(const PgsArgs& P) {
    int used = P.iterations;
    if (P.check_tolerance)
        for (int t = 1 + (int)threadIdx.x; t <= P.iterations; t += blockDim.x)
            if (__longlong_as_double((long long)P.iter_max[t - 1]) < P.tolerance) {
                used = t;
                break;
            }
    for (int o = 32; o > 0; o >>= 1) used = min(used, __shfl_xor(used, o, 64));
    return used;
}
__global__ void k_flow_finish(PgsArgs P) {
    const int used = first_converged(P);
    if (threadIdx.x == 0) *P.iters_used = used;
}
// The buffers of the last pass become the results.  With find, every workgroup
// looks the sweeps up by itself (up to kFindSweeps of them), which saves a launch.
constexpr int kFindSweeps = 4096;
__global__ __launch_bounds__(256) void k_flow_end(FlowArgs F, SetupArgs S, int n_dv, int cap, int find) {
    __shared__ int wave_used[4];
    int used;
    if (find) {
        used = first_converged(F.P);
        if ((threadIdx.x & 63) == 0) wave_used[threadIdx.x >> 6] = used;
        __syncthreads();
        used = min(min(wave_used[0], wave_used[1]), min(wave_used[2], wave_used[3]));
        if (blockIdx.x == 0 && threadIdx.x == 0) *F.P.iters_used = used;
    } else {
        used = *F.P.iters_used;
    }
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n_dv) {
        const int u = S.scene_used ? S.scene_used[S.B.desc[i / 6].scene] : used;
        if (u & 1) F.P.dv[i] = F.dv_alt[i];
    }
    if (i < cap) unpack(S, i, used);
}

// Sweeps used per scene: the first sweep whose max |dl| over the scene was
// under the tolerance, else all (a scene's skipped sweeps read 0).
__global__ void k_scene_finish(PgsArgs P) {
    int s = blockIdx.x * blockDim.x + threadIdx.x;
    if (s >= P.n_scenes) return;
    int used = P.iterations;
    for (int t = 1; t <= P.iterations; t++)
        if (__longlong_as_double((long long)P.scene_max[(size_t)s * P.iterations + t - 1]) < P.tolerance) {
            used = t;
            break;
        }
    P.scene_used[s] = used;
}
void launch_scene_finish(hipStream_t s, const PgsArgs& P) {
    if (P.per_scene && P.n_scenes > 0)
        hipLaunchKernelGGL(k_scene_finish, dim3((P.n_scenes + 63) / 64), dim3(64), 0, s, P);
}

// Groups are counted per scene in an LDS histogram per workgroup (when the
// scenes fit), so each workgroup adds to a scene's global count once instead
// of every group contending for its scene's counter.
constexpr int kSceneHist = 4096;
__global__ __launch_bounds__(1024) void k_group_scene(const int* group_desc, int n_groups, const int* order,
                                                      const int* cb1, const am_body_desc* desc, int n_scenes,
                                                      int* g_scene, unsigned* scene_groups) {
    __shared__ unsigned hist[kSceneHist];
    const bool local = n_scenes <= kSceneHist;
    if (local)
        for (int i = threadIdx.x; i < n_scenes; i += blockDim.x) hist[i] = 0;
    __syncthreads();
    for (int q = blockIdx.x * blockDim.x + threadIdx.x; q < n_groups; q += gridDim.x * blockDim.x) {
        const int sc = desc[cb1[order[group_desc[q * 4]]]].scene;
        g_scene[q] = sc;
        if (local) atomicAdd(&hist[sc], 1u);
        else atomicAdd(&scene_groups[sc], 1u);
    }
    __syncthreads();
    if (local)
        for (int i = threadIdx.x; i < n_scenes; i += blockDim.x)
            if (hist[i]) atomicAdd(&scene_groups[i], hist[i]);
}
void launch_group_scene(hipStream_t s, const int* group_desc, int n_groups, const int* order, const int* cb1,
                        const am_body_desc* desc, int n_scenes, int* g_scene, unsigned* scene_groups) {
    if (n_groups > 0)
        hipLaunchKernelGGL(k_group_scene, dim3(std::min((n_groups + 4095) / 4096, 256)), dim3(1024), 0, s, group_desc,
                           n_groups, order, cb1, desc, n_scenes, g_scene, scene_groups);
}

int pgs_flow_max_blocks(bool* ok) {
    int dev = 0, n_cu = 0, per_cu = 0;
    (void)hipGetDevice(&dev);
    (void)hipDeviceGetAttribute(&n_cu, hipDeviceAttributeMultiprocessorCount, dev);
    int per_cu_scenes = 0;
    (void)hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, k_pgs_flow<false>, 64, 0);
    (void)hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu_scenes, k_pgs_flow<true>, 64, 0);
    per_cu = std::min(per_cu, per_cu_scenes);
    *ok = per_cu > 0;
    return n_cu * (per_cu > 0 ? per_cu : 1);
}

hipError_t launch_pgs_flow(hipStream_t s, const FlowArgs& F, int grid, int block, bool plain) {
    const bool resident = block != 64;
    void (*kernel)(FlowArgs) = resident ? (F.P.per_scene ? k_pgs_resident<true> : k_pgs_resident<false>)
                                        : (F.P.per_scene ? k_pgs_flow<true> : k_pgs_flow<false>);
    if (plain) {
        hipLaunchKernelGGL(kernel, dim3(grid), dim3(block), 0, s, F);
    } else {
        void* args[] = {(void*)&F};
        hipError_t e = hipLaunchCooperativeKernel((const void*)kernel, dim3(grid), dim3(block), args, 0, s);
        if (e != hipSuccess) return e;
    }
    return hipGetLastError();
}
void launch_flow_end(hipStream_t s, const FlowArgs& F, const SetupArgs& S, int cap, int n_dv) {
    const bool find = F.P.iterations <= kFindSweeps;
    if (!find) hipLaunchKernelGGL(k_flow_finish, dim3(1), dim3(64), 0, s, F.P);
    launch_scene_finish(s, F.P);
    hipLaunchKernelGGL(k_flow_end, dim3((std::max(cap, n_dv) + 255) / 256), dim3(256), 0, s, F, S, n_dv, cap,
                       find ? 1 : 0);
}

// ---------------------------------------------------------------------------
// Warm start (CollisionProcessor.java:443-665).
AMD_INLINE uint64_t mix64(uint64_t z) {
    z += 0x9e3779b97f4a7c15ull;
    z = (z ^ (z >> 30)) * 0xbf58476d1ce4e5b9ull;
    z = (z ^ (z >> 27)) * 0x94d049bb133111ebull;
    return z ^ (z >> 31);
}
struct CKey {
    int lo, hi, bvlo, bvhi, info;
};
// Contact.hashCode/equals (Contact.java:543-572): swap-invariant identity.
AMD_INLINE CKey make_key(int b1, int b2, int bv1, int bv2, int info) {
    CKey k;
    if (b1 < b2) {
        k.lo = b1; k.hi = b2; k.bvlo = bv1; k.bvhi = bv2;
    } else {
        k.lo = b2; k.hi = b1; k.bvlo = bv2; k.bvhi = bv1;
    }
    k.info = info;
    return k;
}
AMD_INLINE uint64_t key_hash(const CKey& k) {
    uint64_t h = mix64(((uint64_t)(uint32_t)k.lo << 32) | (uint32_t)k.hi);
    h = mix64(h ^ (((uint64_t)(uint32_t)k.bvlo << 32) | (uint32_t)k.bvhi));
    return mix64(h ^ (uint64_t)(uint32_t)k.info);
}
AMD_INLINE bool key_eq_old(const CKey& k, const OldContactsView& O, int i) {
    CKey o = make_key(O.b1[i], O.b2[i], O.bv1[i], O.bv2[i], O.info[i]);
    return k.lo == o.lo && k.hi == o.hi && k.bvlo == o.bvlo && k.bvhi == o.bvhi && k.info == o.info;
}

// updateContactsMap (CollisionProcessor.java:443-448): insert every old
// contact; for equal keys the later list position wins, like HashMap.put.
__global__ void k_map_insert(OldContactsView O, int* table) {
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= O.n) return;
    CKey k = make_key(O.b1[i], O.b2[i], O.bv1[i], O.bv2[i], O.info[i]);
    int s = (int)(key_hash(k) & (uint64_t)O.table_mask);
    for (;;) {
        int cur = atomicCAS(&table[s], -1, i);
        if (cur == -1) return;
        if (key_eq_old(k, O, cur)) {
            atomicMax(&table[s], i);
            return;
        }
        s = (s + 1) & O.table_mask;
    }
}

void launch_map_insert(hipStream_t s, const OldContactsView& O, int* table) {
    if (O.n <= 0) return;
    hipLaunchKernelGGL(k_map_insert, dim3((O.n + 255) / 256), dim3(256), 0, s, O, table);
}

AMD_INLINE int old_lookup(const OldContactsView& O, const CKey& k) {
    if (O.n <= 0) return -1;
    int s = (int)(key_hash(k) & (uint64_t)O.table_mask);
    for (;;) {
        int i = O.table[s];
        if (i < 0) return -1;
        if (key_eq_old(k, O, i)) return i;
        s = (s + 1) & O.table_mask;
    }
}

AMD_INLINE void set_lambda(ContactsView& C, int c, const double* l) {
#pragma unroll
    for (int r = 0; r < 3; r++) {
        C.lam[c * 3 + r] = l ? l[r] : 0.0;
        C.lamw[c * 3 + r] = l ? l[r] : 0.0;
    }
}

// Whether a contact side (body, bv id) is a composite part that is not a box
// (Contact.csb1 / csb2 set and not RigidBodyGeomBox); AM_BV_SUB carries the part.
AMD_INLINE bool non_box_part(const BodiesView& B, int body, int bv) {
    const am_body_desc& d = B.desc[body];
    if (d.geom != AM_GEOM_COMPOSITE || bv > -3) return false;
    const int s = (-3 - bv) >> 16;
    return B.sub_desc[d.tree_first + s].geom != AM_GEOM_BOX;
}

AMD_INLINE d3 world_point(const BodiesView& B, int body, d3 pB1) {
    return xform(ldm(&B.R[body * 9]), ld3(&B.x[body * 3]), pB1);
}

// The warm start takes two passes with a lane per contact.  Which old contact a
// contact takes does not depend on the lambdas, so every contact looks for its own
// at once.  A box-box contact takes the lambda and zeroes it ("take and zero"), so of
// the contacts that want one old contact the first in list order has its lambda and
// the later ones zero: O.first[o] is that first one.
//
// A lane per group, contact by contact, took 60 us for 5,000 contacts of boxes and
// 115 for sphere trees with 60 contacts a pair: the chain of lookups of its largest
// group.  The two passes take 21 and 13.
__global__ void k_warm_match(BodiesView B, ContactsView C, OldContactsView O, int n, int post, int2* match,
                             int* counters) {
    const int c = blockIdx.x * blockDim.x + threadIdx.x;
    int bad = 0, rep = 0;
    if (c < n) {
        int taken = -1, plain = -1;  // old contacts: zeroed, left as they are
        int b1 = C.b1[c], b2 = C.b2[c];
        // box or composite on both sides takes the box-box path (CollisionProcessor.java:489-493)
        const int g1 = B.desc[b1].geom, g2 = B.desc[b2].geom;
        const bool boxish = (g1 == AM_GEOM_BOX || g1 == AM_GEOM_COMPOSITE) && (g2 == AM_GEOM_BOX || g2 == AM_GEOM_COMPOSITE);
        CKey key = make_key(b1, b2, C.bv1[c], C.bv2[c], C.info[c]);
        const int same = old_lookup(O, key);
        auto vanilla = [&]() {
            plain = same;
            C.is_new[c] = same >= 0 ? 0 : 1;
        };
        // a part that is not a box: body 1's takes the vanilla start only
        // (:497-500), body 2's the vanilla start and then the box-box path (:501-503)
        if (!boxish || non_box_part(B, b1, C.bv1[c])) {
            vanilla();
        } else {
            if (non_box_part(B, b2, C.bv2[c])) vanilla();
            d3 pNew = world_point(B, b1, ld3(&C.pB1[c * 3]));
            int o = same;
            if (o >= 0) {
                d3 pOld = world_point(B, O.b1[o], ld3(&O.pB1[o * 3]));
                double dist = distance(pNew, pOld);
                if (dist > 0.05) {
                    bad++;
                    int myInfo = C.info[c];
                    double best = dist;
                    int bestInfo = myInfo, bestOld = o;
                    for (int info = 0; info < 9; info++) {
                        if (info == myInfo) continue;
                        key.info = info;
                        int oo = old_lookup(O, key);
                        if (oo < 0) break;
                        pOld = world_point(B, O.b1[oo], ld3(&O.pB1[oo * 3]));
                        dist = distance(pNew, pOld);
                        if (dist < best) {
                            best = dist;
                            bestInfo = info;
                            bestOld = oo;
                        }
                    }
                    if (bestInfo != myInfo) rep++;
                    o = bestOld;
                    dist = best;
                }
                if (dist < 0.05) taken = o;
                else C.is_new[c] = 1;
            } else {
                double best = 1.7976931348623157e308;
                int bestInfo = -1, bestOld = -1;
                for (int info = 0; info < 9; info++) {
                    key.info = info;
                    int oo = old_lookup(O, key);
                    if (oo < 0) break;
                    d3 pOld = world_point(B, O.b1[oo], ld3(&O.pB1[oo * 3]));
                    double dist = distance(pNew, pOld);
                    if (dist < best) {
                        best = dist;
                        bestInfo = info;
                        bestOld = oo;
                    }
                }
                if (bestInfo != -1) {
                    rep++;
                    if (best < 0.05) taken = bestOld;
                } else {
                    C.is_new[c] = 1;
                }
            }
        }
        if (plain >= 0) {
            set_lambda(C, c, &O.lam[plain * 3]);
            C.prev_viol[c] = post ? O.prev_viol[plain] : O.viol[plain];
        }
        if (taken >= 0) {
            C.is_new[c] = 0;
            C.prev_viol[c] = post ? O.prev_viol[taken] : O.viol[taken];
            atomicMin(&O.first[taken], c);
        }
        match[c] = make_int2(taken, plain);
    }
    if (bad) atomicAdd(&counters[0], bad);
    if (rep) atomicAdd(&counters[1], rep);
}
__global__ void k_warm_take(ContactsView C, OldContactsView O, int n, const int2* match) {
    const int c = blockIdx.x * blockDim.x + threadIdx.x;
    if (c >= n) return;
    const int2 m = match[c];
    if (m.x >= 0) {
        const bool mine = O.first[m.x] == c;
        set_lambda(C, c, mine ? &O.lam[m.x * 3] : nullptr);
        if (mine)
#pragma unroll
            for (int r = 0; r < 3; r++) O.lam[m.x * 3 + r] = 0.0;
    } else if (m.y >= 0 && O.first[m.y] < c) {
        set_lambda(C, c, nullptr);  // zeroed by an earlier contact
    }
}

void launch_warm_start(hipStream_t s, BodiesView B, ContactsView C, OldContactsView O, int n, int post, int* match,
                       int* counters) {
    if (n <= 0) return;
    const dim3 g((n + 127) / 128), b(128);
    hipLaunchKernelGGL(k_warm_match, g, b, 0, s, B, C, O, n, post, (int2*)match, counters);
    hipLaunchKernelGGL(k_warm_take, g, b, 0, s, C, O, n, (const int2*)match);
}

// redoWarmStart / noWarmStart (CollisionProcessor.java:453-470)
__global__ void k_redo_warm(ContactsView C, const int* n, int zero) {
    int c = blockIdx.x * blockDim.x + threadIdx.x;
    if (c >= *n) return;
#pragma unroll
    for (int r = 0; r < 3; r++) C.lam[c * 3 + r] = zero ? 0.0 : C.lamw[c * 3 + r];
}
void launch_redo_warm(hipStream_t s, ContactsView C, const int* n, int cap, int zero) {
    if (cap <= 0) return;
    hipLaunchKernelGGL(k_redo_warm, dim3((cap + 255) / 256), dim3(256), 0, s, C, n, zero);
}

// ---------------------------------------------------------------------------
// Forces and integration.
// RigidBody.clear (RigidBody.java:226-230)
__global__ void k_clear(BodiesView B) {
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= B.n) return;
#pragma unroll
    for (int a = 0; a < 3; a++) {
        B.f[i * 3 + a] = 0.0;
        B.t[i * 3 + a] = 0.0;
    }
#pragma unroll
    for (int a = 0; a < 6; a++) B.dv[i * 6 + a] = 0.0;
}
void launch_clear(hipStream_t s, BodiesView B) {
    if (B.n > 0) hipLaunchKernelGGL(k_clear, dim3((B.n + 255) / 256), dim3(256), 0, s, B);
}

// RigidBodySystem.applyGravityForce (RigidBodySystem.java:276-290): listed
// entities and the members of listed collections.
__global__ void k_gravity(BodiesView B, const int* targets, int n, d3 dir) {
    int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= n) return;
    int i = targets[k];
    double m = -B.desc[i].mass;
    B.f[i * 3 + 0] = B.f[i * 3 + 0] + m * dir.x;
    B.f[i * 3 + 1] = B.f[i * 3 + 1] + m * dir.y;
    B.f[i * 3 + 2] = B.f[i * 3 + 2] + m * dir.z;
}
void launch_gravity(hipStream_t s, BodiesView B, const int* targets, int n, double gx, double gy, double gz) {
    if (n > 0) hipLaunchKernelGGL(k_gravity, dim3((n + 255) / 256), dim3(256), 0, s, B, targets, n, d3{gx, gy, gz});
}

// RigidBody.applyForceW (RigidBody.java:335-340)
AMD_INLINE void apply_force_w(BodiesView B, int e, d3 p, d3 F) {
    st3(&B.f[e * 3], add(ld3(&B.f[e * 3]), F));
    const d3 r = sub(p, ld3(&B.x[e * 3]));
    st3(&B.t[e * 3], add(ld3(&B.t[e * 3]), cross(r, F)));
}
// RigidBodySystem.applySpringForces (RigidBodySystem.java:309-322) with
// Spring.applyOneBody / applyTwoBodies (Spring.java:165-214).  One thread walks
// the springs in list order, so every accumulator receives the reference's
// sequence of additions.
__global__ void k_springs(BodiesView B, const am_spring* S, int n, double ks, double ds) {
    if (threadIdx.x != 0 || blockIdx.x != 0) return;
    for (int i = 0; i < n; i++) {
        const am_spring sp = S[i];
        const int b1 = sp.body1;
        const d3 p1w = xform(ldm(&B.R[b1 * 9]), ld3(&B.x[b1 * 3]), ld3(sp.pb1));
        if (sp.type != AM_SPRING_BODYBODY) {
            const d3 disp = sub(ld3(sp.pw), p1w);
            const double len = length(disp);
            if (len < 1e-3) continue;
            const d3 vel = spatial_velocity(B, b1, p1w);
            const double scl = -(sp.k * ks * (len - sp.l0 * sp.ls) - sp.d * ds * (dot(vel, disp) / len)) / len;
            const d3 F = scale(-scl, disp);
            apply_force_w(B, b1, p1w, F);
            if (B.parent[b1] >= 0) apply_force_w(B, B.parent[b1], p1w, F);
        } else {
            const int b2 = sp.body2;
            const d3 p2w = xform(ldm(&B.R[b2 * 9]), ld3(&B.x[b2 * 3]), ld3(sp.pb2));
            d3 disp = sub(p2w, p1w);
            const double dist = length(disp);
            if (dist < 1e-3) continue;
            disp = scale(1. / dist, disp);
            const d3 v2 = spatial_velocity(B, b2, p2w);
            const d3 v1 = spatial_velocity(B, b1, p1w);
            const d3 rel = sub(v2, v1);
            const double fi = sp.k * ks * (dist - sp.l0 * sp.ls) + sp.d * ds * dot(rel, disp);
            d3 F = scale(fi, disp);
            apply_force_w(B, b1, p1w, F);
            if (B.parent[b1] >= 0) apply_force_w(B, B.parent[b1], p1w, F);
            F = scale(-fi, disp);
            apply_force_w(B, b2, p2w, F);
            if (B.parent[b2] >= 0) apply_force_w(B, B.parent[b2], p2w, F);
        }
    }
}
void launch_springs(hipStream_t s, BodiesView B, const am_spring* springs, int n, double ks, double ds) {
    if (n > 0) hipLaunchKernelGGL(k_springs, dim3(1), dim3(64), 0, s, B, springs, n, ks, ds);
}

// RigidBody.advanceVelocities (RigidBody.java:409-417)
__global__ void k_advance_velocities(BodiesView B, const int* targets, int n, double dt) {
    int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= n) return;
    int i = targets[k];
    double s = dt * B.minv[i];
    d3 v = scale_add(s, ld3(&B.f[i * 3]), ld3(&B.v[i * 3]));
    v = add(v, ld3(&B.dv[i * 6]));
    st3(&B.v[i * 3], v);
    d3 dom = mul(ldm(&B.jinv[i * 9]), ld3(&B.t[i * 3]));
    dom = mk(dom.x * dt, dom.y * dt, dom.z * dt);
    d3 w = add(ld3(&B.w[i * 3]), dom);
    w = add(w, ld3(&B.dv[i * 6 + 3]));
    st3(&B.w[i * 3], w);
}

// Sine and cosine of the rotation angle (expRodrigues calls Math.sin and
// Math.cos).  Computed by fdlibm 5.3's algorithm (Sun Microsystems, 1993),
// which defines java.lang.StrictMath.sin/cos: Cody-Waite reduction by pi/2 in
// up to three steps (e_rem_pio2.c, |x| <= 2^19 pi/2) and the minimax kernels
// of k_sin.c / k_cos.c.  Larger arguments, which no physical step reaches,
// take the three-step reduction with a floating-point quotient.  Written out
// here rather than calling the device library so that every rounding is
// fixed by the source, whatever the library version.
namespace fdm {
__device__ __forceinline__ int hi(double x) { return (int)(__double_as_longlong(x) >> 32); }
__device__ __forceinline__ double from_hi(int h) { return __longlong_as_double((long long)(unsigned)h << 32); }
constexpr double S1 = -1.66666666666666324348e-01, S2 = 8.33333333332248946124e-03,
                 S3 = -1.98412698298579493134e-04, S4 = 2.75573137070700676789e-06,
                 S5 = -2.50507602534068634195e-08, S6 = 1.58969099521155010221e-10;
constexpr double C1 = 4.16666666666666019037e-02, C2 = -1.38888888888741095749e-03,
                 C3 = 2.48015872894767294178e-05, C4 = -2.75573143513906633035e-07,
                 C5 = 2.08757232129817482790e-09, C6 = -1.13596475577881948265e-11;
constexpr double invpio2 = 6.36619772367581382433e-01, pio2_1 = 1.57079632673412561417e+00,
                 pio2_1t = 6.07710050650619224932e-11, pio2_2 = 6.07710050630396597660e-11,
                 pio2_2t = 2.02226624879595063154e-21, pio2_3 = 2.02226624871116645580e-21,
                 pio2_3t = 8.47842766036889956997e-32;
// high words of the doubles nearest n pi/2, n = 1..32
__constant__ int npio2_hw[32] = {
    0x3ff921fb, 0x400921fb, 0x4012d97c, 0x401921fb, 0x401f6a7a, 0x4022d97c, 0x4025fdbb, 0x402921fb,
    0x402c463a, 0x402f6a7a, 0x4031475c, 0x4032d97c, 0x40346b9c, 0x4035fdbb, 0x40378fdb, 0x403921fb,
    0x403ab41b, 0x403c463a, 0x403dd85a, 0x403f6a7a, 0x40407e4c, 0x4041475c, 0x4042106c, 0x4042d97c,
    0x4043a28c, 0x40446b9c, 0x404534ac, 0x4045fdbb, 0x4046c6cb, 0x40478fdb, 0x404858eb, 0x404921fb};

__device__ double k_sin(double x, double y, bool tail) {
    int ix = hi(x) & 0x7fffffff;
    if (ix < 0x3e400000 && (int)x == 0) return x;
    double z = x * x, v = z * x;
    double r = S2 + z * (S3 + z * (S4 + z * (S5 + z * S6)));
    if (!tail) return x + v * (S1 + z * r);
    return x - ((z * (0.5 * y - v * r) - y) - v * S1);
}
__device__ double k_cos(double x, double y) {
    int ix = hi(x) & 0x7fffffff;
    if (ix < 0x3e400000 && (int)x == 0) return 1.0;
    double z = x * x;
    double r = z * (C1 + z * (C2 + z * (C3 + z * (C4 + z * (C5 + z * C6)))));
    if (ix < 0x3fd33333) return 1.0 - (0.5 * z - (z * r - x * y));
    double qx = ix > 0x3fe90000 ? 0.28125 : from_hi(ix - 0x00200000);
    double hz = 0.5 * z - qx, a = 1.0 - qx;
    return a - (hz - (z * r - x * y));
}
// x = n pi/2 + y0 + y1 for |x| >= pi/4; returns n
__device__ int rem_pio2(double x, double& y0, double& y1) {
    int hx = hi(x), ix = hx & 0x7fffffff;
    if (ix < 0x4002d97c) {  // |x| < 3pi/4
        const double s = hx > 0 ? 1.0 : -1.0;
        double z = x - s * pio2_1;
        if (ix != 0x3ff921fb) {
            y0 = z - s * pio2_1t;
            y1 = (z - y0) - s * pio2_1t;
        } else {
            z = z - s * pio2_2;
            y0 = z - s * pio2_2t;
            y1 = (z - y0) - s * pio2_2t;
        }
        return hx > 0 ? 1 : -1;
    }
    double t = fabs(x);
    const bool medium = ix <= 0x413921fb;
    double fn;
    int n;
    if (medium) {
        n = (int)(t * invpio2 + 0.5);
        fn = (double)n;
    } else {
        fn = floor(t * invpio2 + 0.5);
        n = (int)(fn - 4.0 * floor(fn * 0.25));
    }
    double r = t - fn * pio2_1;
    double w = fn * pio2_1t;
    y0 = r - w;
    if (!(medium && n < 32 && ix != npio2_hw[n - 1])) {
        const int j = ix >> 20;
        int i = j - ((hi(y0) >> 20) & 0x7ff);
        if (i > 16 || !medium) {
            t = r;
            w = fn * pio2_2;
            r = t - w;
            w = fn * pio2_2t - ((t - r) - w);
            y0 = r - w;
            i = j - ((hi(y0) >> 20) & 0x7ff);
            if (i > 49 || !medium) {
                t = r;
                w = fn * pio2_3;
                r = t - w;
                w = fn * pio2_3t - ((t - r) - w);
                y0 = r - w;
            }
        }
    }
    y1 = (r - y0) - w;
    if (hx < 0) {
        y0 = -y0;
        y1 = -y1;
        return -n;
    }
    return n;
}
// both at once: the reduction is shared
__device__ void sincos(double x, double& s, double& c) {
    int ix = hi(x) & 0x7fffffff;
    if (ix <= 0x3fe921fb) {
        s = k_sin(x, 0.0, false);
        c = k_cos(x, 0.0);
        return;
    }
    if (ix >= 0x7ff00000) {
        s = c = x - x;
        return;
    }
    double y0, y1;
    const int q = rem_pio2(x, y0, y1) & 3;
    const double ks = k_sin(y0, y1, true), kc = k_cos(y0, y1);
    switch (q) {
        case 0: s = ks; c = kc; break;
        case 1: s = kc; c = -ks; break;
        case 2: s = -ks; c = -kc; break;
        default: s = -kc; c = ks; break;
    }
}
}  // namespace fdm

// Prescribed motion of the kinematic bodies at time t:
// x = x0 + (a sin(w t + phase)) dir, v = (a w cos(w t + phase)) dir, omega = 0.
__global__ void k_kinematic(BodiesView B, const am_kinematic* K, int n, double t) {
    int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= n) return;
    const am_kinematic q = K[k];
    double s, c;
    fdm::sincos(q.omega * t + q.phase, s, c);
    const double ds = q.amplitude * s;
    const double vs = q.amplitude * q.omega * c;
    const int e = q.body;
#pragma unroll
    for (int a = 0; a < 3; a++) {
        B.x[e * 3 + a] = q.x0[a] + ds * q.dir[a];
        B.v[e * 3 + a] = vs * q.dir[a];
        B.w[e * 3 + a] = 0.0;
    }
}
void launch_kinematic(hipStream_t s, BodiesView B, const am_kinematic* k, int n, double t) {
    if (n > 0) hipLaunchKernelGGL(k_kinematic, dim3((n + 63) / 64), dim3(64), 0, s, B, k, n, t);
}

// RigidBodySystem.applyImpulse (RigidBodySystem.java:262-267): each held
// force goes to its body's top-level entity through RigidBody.applyForceW.
// One thread, so forces on one entity add in the order they were held.
__global__ void k_impulses(BodiesView B, const ImpulseRec* I, int n) {
    if (blockIdx.x != 0 || threadIdx.x != 0) return;
    for (int k = 0; k < n; k++) {
        const int b = I[k].body;
        const int e = B.parent[b] >= 0 ? B.parent[b] : b;
        apply_force_w(B, e, ld3(I[k].p), ld3(I[k].f));
    }
}
void launch_impulses(hipStream_t s, BodiesView B, const ImpulseRec* I, int n) {
    if (n > 0) hipLaunchKernelGGL(k_impulses, dim3(1), dim3(64), 0, s, B, I, n);
}

// RigidBodySystem.applyViscousDecay (RigidBodySystem.java:428-435): v and
// omega of the listed (top-level) entities scaled (Vector3d.scale).
__global__ void k_viscous(BodiesView B, const int* targets, int n, double a1, double a2) {
    int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= n) return;
    const int e = targets[k];
#pragma unroll
    for (int a = 0; a < 3; a++) {
        B.v[e * 3 + a] = a1 * B.v[e * 3 + a];
        B.w[e * 3 + a] = a2 * B.w[e * 3 + a];
    }
}
void launch_viscous(hipStream_t s, BodiesView B, const int* targets, int n, double a1, double a2) {
    if (n > 0) hipLaunchKernelGGL(k_viscous, dim3((n + 255) / 256), dim3(256), 0, s, B, targets, n, a1, a2);
}

// The pose update of RigidBody.advancePositions (RigidBody.java:427-437):
// Rodrigues rotation (expRodrigues, RigidBody.java:382-401) and
// Matrix3d.normalizeCP.  Returns whether R changed.
__device__ __forceinline__ bool advance_pose(d3& x, m33& R, d3 v, d3 om, double dt) {
    x = scale_add(dt, v, x);
    double t = length(om) * dt;
    d3 d = normalized(om);
    if (t > 1e-8) {
        double s, c;
        fdm::sincos(t, s, c);
        const double c1 = 1 - c;
        double wX = d.x, wY = d.y, wZ = d.z;
        m33 dR;
        dR.m[0] = c + wX * wX * c1;
        dR.m[3] = wZ * s + wX * wY * c1;
        dR.m[6] = -wY * s + wX * wZ * c1;
        dR.m[1] = -wZ * s + wX * wY * c1;
        dR.m[4] = c + wY * wY * c1;
        dR.m[7] = wX * s + wY * wZ * c1;
        dR.m[2] = wY * s + wX * wZ * c1;
        dR.m[5] = -wX * s + wY * wZ * c1;
        dR.m[8] = c + wZ * wZ * c1;
        dR = mmul(dR, R);
        double mag = 1.0 / sqrt(dR.m[0] * dR.m[0] + dR.m[3] * dR.m[3] + dR.m[6] * dR.m[6]);
        R.m[0] = dR.m[0] * mag;
        R.m[3] = dR.m[3] * mag;
        R.m[6] = dR.m[6] * mag;
        mag = 1.0 / sqrt(dR.m[1] * dR.m[1] + dR.m[4] * dR.m[4] + dR.m[7] * dR.m[7]);
        R.m[1] = dR.m[1] * mag;
        R.m[4] = dR.m[4] * mag;
        R.m[7] = dR.m[7] * mag;
        R.m[2] = R.m[3] * R.m[7] - R.m[4] * R.m[6];
        R.m[5] = R.m[1] * R.m[6] - R.m[0] * R.m[7];
        R.m[8] = R.m[0] * R.m[4] - R.m[1] * R.m[3];
        return true;
    }
    return false;
}

// RigidBody.advancePositions (RigidBody.java:427-441) of the listed entities;
// with from_dv the velocities are deltaV's parts
// (advancePositionsPostStabilization, RigidBody.java:423-425).
__global__ void k_advance_positions(BodiesView B, const int* targets, int n, double dt, int from_dv) {
    int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= n) return;
    int i = targets[k];
    d3 x = ld3(&B.x[i * 3]);
    m33 R = ldm(&B.R[i * 9]);
    const d3 v = from_dv ? ld3(&B.dv[i * 6]) : ld3(&B.v[i * 3]);
    const d3 om = from_dv ? ld3(&B.dv[i * 6 + 3]) : ld3(&B.w[i * 3]);
    const bool turned = advance_pose(x, R, v, om, dt);
    st3(&B.x[i * 3], x);
    if (turned) stm(&B.R[i * 9], R);
    stm(&B.jinv[i * 9], rm0rt(R, ldm(B.desc[i].jinv0)));
}

// Every entity's pose advanced by dt without changing the body state (the
// copies body1Advanced / body2Advanced of MotionMetricProcessor.java:79-83).
__global__ void k_advanced_poses(BodiesView B, double dt, double* xa, double* Ra) {
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= B.n) return;
    d3 x = ld3(&B.x[i * 3]);
    m33 R = ldm(&B.R[i * 9]);
    advance_pose(x, R, ld3(&B.v[i * 3]), ld3(&B.w[i * 3]), dt);
    st3(&xa[i * 3], x);
    stm(&Ra[i * 9], R);
}
void launch_advance_post(hipStream_t s, BodiesView B, const int* targets, int n, double dt) {
    if (n > 0) hipLaunchKernelGGL(k_advance_positions, dim3((n + 127) / 128), dim3(128), 0, s, B, targets, n, dt, 1);
}
void launch_advanced_poses(hipStream_t s, BodiesView B, double dt, double* xa, double* Ra) {
    if (B.n > 0) hipLaunchKernelGGL(k_advanced_poses, dim3((B.n + 127) / 128), dim3(128), 0, s, B, dt, xa, Ra);
}

void launch_advance(hipStream_t s, BodiesView B, const int* targets, int n, double dt, bool positions) {
    if (n <= 0) return;
    if (positions) hipLaunchKernelGGL(k_advance_positions, dim3((n + 127) / 128), dim3(128), 0, s, B, targets, n, dt, 0);
    else hipLaunchKernelGGL(k_advance_velocities, dim3((n + 255) / 256), dim3(256), 0, s, B, targets, n, dt);
}

// jinv = R jinv0 R^T for non-pinned entities, zero for pinned.
__global__ void k_update_jinv(BodiesView B) {
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= B.n) return;
    if (B.flags[i] & AM_BODY_PINNED) {
#pragma unroll
        for (int a = 0; a < 9; a++) B.jinv[i * 9 + a] = 0.0;
        return;
    }
    stm(&B.jinv[i * 9], rm0rt(ldm(&B.R[i * 9]), ldm(B.desc[i].jinv0)));
}
void launch_update_jinv(hipStream_t s, BodiesView B) {
    if (B.n > 0) hipLaunchKernelGGL(k_update_jinv, dim3((B.n + 255) / 256), dim3(256), 0, s, B);
}

// ---------------------------------------------------------------------------
// MotionMetricProcessor.getLargestVelocityNorm (MotionMetricProcessor.java:39-73)
__global__ void k_metric(BodiesView B, const int* pairs, int n, double* out) {
    int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= n) return;
    int a = pairs[k * 2], b = pairs[k * 2 + 1];
    out[k] = b < 0 ? metric_one(B, a) : metric_two(B, a, b);
}
void launch_metric(hipStream_t s, BodiesView B, const int* pairs, int n, double* out) {
    if (n > 0) hipLaunchKernelGGL(k_metric, dim3((n + 127) / 128), dim3(128), 0, s, B, pairs, n, out);
}

// ---------------------------------------------------------------------------
// Colouring driver pieces
void launch_incidence(hipStream_t s, bool fill, int n_groups, const int* ga, const int* gb, const int* bflags,
                      int* inc_count, const int* inc_start, int* inc_cursor, int* inc_items) {
    if (n_groups <= 0) return;
    dim3 g((n_groups + 255) / 256), b(256);
    if (!fill) hipLaunchKernelGGL(k_incidence_count, g, b, 0, s, n_groups, ga, gb, bflags, inc_count);
    else hipLaunchKernelGGL(k_incidence_fill, g, b, 0, s, n_groups, ga, gb, bflags, inc_start, inc_cursor, inc_items);
}
void launch_colour(hipStream_t s, int n_groups, const int* ga, const int* gb, const int* bflags, const int* inc_start,
                   const int* inc_count, const int* inc_items, int* colour, TakenColours* taken, int* rank,
                   int* remaining, const int* layer, int* blocker, bool again, int max_polls) {
    if (n_groups <= 0) return;
    // at most 8 workgroups on each of 256 CUs (workgroups that wait for others that
    // are not resident give up in the end and leave room for them)
    const int per = layer ? 64 : 256;
    const dim3 g(std::min((n_groups + per - 1) / per, 2048)), b(256);
    if (layer) {
        hipLaunchKernelGGL(k_colour_layered, g, b, 0, s, n_groups, ga, gb, bflags, inc_start, inc_count, inc_items,
                           colour, remaining, layer, blocker, max_polls);
        return;
    }
    if (!again)
        hipLaunchKernelGGL(k_colour_ranks, dim3((2 * n_groups + 255) / 256), b, 0, s, n_groups, ga, gb, bflags,
                           inc_start, inc_count, inc_items, rank);
    hipLaunchKernelGGL(k_colour, g, b, 0, s, n_groups, ga, gb, rank, colour, taken, remaining, max_polls);
}
void launch_colour_keys(hipStream_t s, int n_groups, const int* colour, const int* group_start, uint64_t* keys) {
    if (n_groups > 0)
        hipLaunchKernelGGL(k_colour_keys, dim3((n_groups + 255) / 256), dim3(256), 0, s, n_groups, colour,
                           group_start, keys);
}
void launch_colour_layout(hipStream_t s, int n_groups, const uint64_t* sorted, const int* group_start,
                          const int* group_a, const int* group_b, int* colour_start, int* sizes, int* pos_start,
                          int* order, int* group_desc, int* pos_a, int* spos, int* d_total, void* scan_temp) {
    hipLaunchKernelGGL(k_colour_starts, dim3(1), dim3(128), 0, s, n_groups, sorted, colour_start);
    if (n_groups <= 0) return;
    dim3 g((n_groups + 255) / 256), b(256);
    hipLaunchKernelGGL(k_sorted_sizes, dim3((n_groups + 256) / 256), b, 0, s, n_groups, sorted, group_start, sizes);
    exclusive_scan(s, sizes, pos_start, n_groups + 1, d_total, scan_temp);
    hipLaunchKernelGGL(k_solve_order, g, b, 0, s, n_groups, sorted, group_start, pos_start, group_a, group_b, order,
                       group_desc, pos_a, spos);
}

}  // namespace am
