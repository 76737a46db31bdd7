// kmst_union.hip -- the direct solve: a whole minimum spanning forest in one
// launch of resident workgroups (and two short ones: a fill of the counters
// before it, their publication after it), on undirected edge lists over a
// union-find parent array.
//
// Phases (every size is read on the device; a grid barrier between phases):
//
//   init     parent[v] = v, minima and edge marks cleared, weight pivots from
//            a sample of the weights;
//   light    one pass over the input: validation, every vertex's lightest
//            record and row, and the forward (src < dst) records of the one to
//            three lightest weight classes, each wave listing its own;
//   rounds   hook and relabel (below) on the first class's edges until none is
//            left;
//   flatten  every vertex points at its root;
//   cross    the next class, at last the rest of the input: the edges that
//            still join different components, followed by their rounds
//            (boruvka_recursive, hybrid_boruvka_edgefilter.hpp:227-330, with
//            the classes as its levels);
//   output   the marked input positions in order: the input is sorted by
//            (src, dst), so this is the MST sorted by (min, max).
//
// A list holds each undirected edge once as (a, b, key) with a and b roots of
// the parent array; best[v] is the smallest key of the edges at root v.
//   hook     an edge that is the minimum of one of its ends hooks that end
//            onto the other; of a mutual pair the lower end stays root (the
//            lower-endpoint rule of determine_mst_edges,
//            include/algorithms/gbbs_reimplementation.hpp:100-130).  The
//            edges that hook an end are MST edges.  Keys order edges
//            strictly, so every component of the hooks holds exactly one
//            mutual pair, whose lower end is the only root that lives on: it
//            clears its minimum of the next round.
//   relabel  both ends walk to their roots (shortening the walked paths, as
//            update_parents, gbbs_reimplementation.hpp:162-169), self-loops
//            drop (relabel_edges / filter_out_self_loops, :184-219), and the
//            kept edges offer their keys to the minima of the next round.
// Against the sort-based rounds this moves each undirected edge once instead
// of both directed records, and needs no vertex renumbering, sort, pass over
// the vertices or read-back.
//
// What bounds it: a small or medium solve is a chain of dependent memory
// round trips (about 0.7 us each) and barriers.  A barrier costs 2.1 us at 16
// workgroups and 2.6 us at 256, because what workgroups share between phases
// (parent, minima, marks, counters) is accessed with agent-scope relaxed
// atomics, which are coherent by themselves; with plain accesses each barrier
// needs an agent-scope fence per workgroup, an L2 write-back, and costs 2.4 to
// 11.4 us.  A launch per phase costs 4 us and more.  Agent-scope gathers run
// at the rate of plain ones (250 10^9/s from a 4 MB table, 58 10^9/s from 64
// MB); atomic minima run at 26 10^9/s spread out and 12 10^6/s on one address.
// A large one is bound by random accesses, 8 to 16 bytes of 64 to 128 MB tables
// for every listed edge and round, and by the light pass.
// Measured a whole solve, this against the round loop: 256 vertices, 4.4 10^3
// records 50 / 185 us (union_small_kernel); 2^14, 5.2 10^5 208 / 534 us; 2^17, 2.1 10^6 317 / 1394
// us; 10^6, 3.2 10^7 729 / 2628 us (a copy of its bytes: 81 us); 2^24, 5.4 10^8
// 6.75 / 10.5 ms (1.36 ms).
// Lists are private to a wave, so they need no coherence, counters or
// workgroup barriers, and their compaction is in place (plain accesses: a wave's
// range changes hands once, behind a release and an acquire).
#include "kmst_kernels.hpp"
#include "kmst_rows.hpp"
#include "kmst_walks.hpp"

namespace kmst {

namespace {

constexpr int UT = UNION_THREADS;  // 1024: one workgroup per CU
constexpr int UW = UT / WAVE;
constexpr u64 WALL_TICKS_PER_MS = 100000;              // 100 MHz wall clock
constexpr u64 BARRIER_TICKS = 10000 * WALL_TICKS_PER_MS;  // bound of a barrier's wait
constexpr u64 JOIN_TICKS = 5 * WALL_TICKS_PER_MS;      // bound of the first one's
constexpr int DEEP_SHIFT = 35;  // in a relabel's payload, above the edges of all waves

// wave index, in a scalar register: what follows from it (a wave's units, list
// and counts) is then wave-uniform to the compiler too
__device__ __forceinline__ u32 wave_index() {
  return __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE);
}

// ------------------------------------------------------------ shared data
template <typename T>
__device__ __forceinline__ T get(const T* p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
template <typename T>
__device__ __forceinline__ void put(T* p, T v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Element i of a per-vertex array: with at most UNION_VERTICES_MAX vertices the
// byte offset fits 32 bits, so the access takes a scalar base and one register.
template <typename T>
__device__ __forceinline__ T* at(T* base, u32 i) {
  return reinterpret_cast<T*>(reinterpret_cast<char*>(base) + u32(i * u32(sizeof(T))));
}
template <typename T>
__device__ __forceinline__ const T* at(const T* base, u32 i) {
  return reinterpret_cast<const T*>(reinterpret_cast<const char*>(base) + u32(i * u32(sizeof(T))));
}
__device__ __forceinline__ u64* minima(const UnionArgs& a, int which) {
  return which ? a.best[1] : a.best[0];
}

__device__ __forceinline__ void lower(u64* best, u32 v, u64 k) {
  (void)__hip_atomic_fetch_min(at(best, v), k, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void offer(u64* best, u32 v, u64 k) {
  if (k < get(at(best, v))) lower(best, v, k);
}

// Lane shifts by DPP: one instruction, where a shuffle is a round trip through
// the LDS.  Lanes without a source keep `old`.
constexpr int DPP_WAVE_SHL1 = 0x130, DPP_WAVE_SHR1 = 0x138;  // from the lane after, before
constexpr int DPP_ROW_SHR = 0x110;                           // + o: from o lanes before, of 16
constexpr int DPP_ROW_BCAST15 = 0x142, DPP_ROW_BCAST31 = 0x143;
template <int CTRL, int ROWS = 0xF>
__device__ __forceinline__ u32 dpp(u32 old, u32 x) {
  return static_cast<u32>(__builtin_amdgcn_update_dpp(static_cast<int>(old), static_cast<int>(x),
                                                      CTRL, ROWS, 0xF, false));
}

// ------------------------------------------------------------ barrier
// Workgroups arrive on one of eight group words (workgroup id mod 8, one XCD
// each) and a group's last arrival adds the group to the root word, so that no
// address takes more than 32 arrivals.  The words also sum a payload, returned
// to every workgroup.  Group words are cleared by their last arrival; the root
// words rotate, and workgroup 0 clears the one after next (nobody arrives on
// it before workgroup 0 has arrived on the next).
// Every wave waits for its own stores and atomics (vmcnt 0) before its
// workgroup arrives.  The first barrier is the admission check: an ordinary
// launch does not promise that all workgroups are resident together, so if
// they are not within JOIN_TICKS the launch is called off, by one atomic
// decision that later arrivals see, and every workgroup leaves with nothing
// changed but scratch.  Once it has passed, all are resident, and the other
// barriers complete (their wait is bounded all the same).
constexpr u32 GROUPS = 8;
constexpr u32 LINE = 16;  // u64 words per 128-byte line
constexpr u64 PAYLOAD_SHIFT = 16;

struct Barrier {
  u64* words;  // root words at lines 0..3, group words at lines 4..11
  u32 k = 0;
  u32* err;
};

// (thread 0's payload counts)
__device__ __forceinline__ bool sync_grid(Barrier& bar, u64 payload, u64& sum) {
  __shared__ u64 s_sum;
  __shared__ u32 s_ok;
  __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0)
  __syncthreads();
  if (gridDim.x == 1) {
    if (threadIdx.x == 0) s_sum = payload;
    __syncthreads();
    sum = s_sum;
    return true;
  }
  if (threadIdx.x == 0) {
    const u32 g = blockIdx.x % GROUPS, groups = min(GROUPS, gridDim.x);
    const u32 members = (gridDim.x - g + GROUPS - 1) / GROUPS;
    u64* root = bar.words + (bar.k & 3) * LINE;
    u64* grp = bar.words + (4 + g) * LINE;
    const u64 mine = (payload << PAYLOAD_SHIFT) | 1;
    const u64 now = __hip_atomic_fetch_add(grp, mine, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) + mine;
    if ((now & 0xFFFF) == members) {
      put(grp, u64{0});
      __builtin_amdgcn_s_waitcnt(0x0F70);  // cleared before the group's next arrivals
      (void)__hip_atomic_fetch_add(root, (now & ~u64{0xFFFF}) | 1, __ATOMIC_RELAXED,
                                   __HIP_MEMORY_SCOPE_AGENT);
    }
    const u64 t0 = wall_clock64();
    u32 ok = 1;
    u64 r;
    while (((r = get(root)) & 0xFFFF) != groups) {
      if (wall_clock64() - t0 > BARRIER_TICKS || (get(bar.err) & ERR_SPIN)) {
        atomicOr(bar.err, ERR_SPIN);
        ok = 0;
        break;
      }
      __builtin_amdgcn_s_sleep(1);
    }
    if (blockIdx.x == 0) put(bar.words + ((bar.k + 2) & 3) * LINE, u64{0});
    s_sum = r >> PAYLOAD_SHIFT;
    s_ok = ok;
  }
  ++bar.k;
  __syncthreads();
  sum = s_sum;
  return s_ok != 0;
}

// Block-wide sum of a wave-uniform value, in thread 0 (all threads call).
__device__ __forceinline__ u64 block_total(u64 wave_value) {
  __shared__ u64 s_v[UW];
  __syncthreads();  // thread 0 may still be adding the call before
  if (lane_id() == 0) s_v[wave_index()] = wave_value;
  __syncthreads();
  u64 t = 0;
  if (threadIdx.x == 0)
    for (int w = 0; w < UW; ++w) t += s_v[w];
  return t;
}

__device__ __forceinline__ bool join_grid(u32* joined) {
  __shared__ u32 s_join;
  if (threadIdx.x == 0) {
    u32 ok = 1;
    if (gridDim.x > 1) {
      u32 seen = __hip_atomic_fetch_add(joined, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) + 1;
      const u64 t0 = wall_clock64();
      while (seen != gridDim.x && !(seen & UNION_CALLED_OFF)) {
        if (wall_clock64() - t0 > JOIN_TICKS)
          (void)atomicCAS(joined, seen, seen | UNION_CALLED_OFF);  // fails if someone joined: look again
        else
          __builtin_amdgcn_s_sleep(1);
        seen = get(joined);
      }
      ok = seen & UNION_CALLED_OFF ? 0u : 1u;
    }
    s_join = ok;
  }
  __syncthreads();
  return s_join != 0;
}

// ------------------------------------------------------------ loads
// Four consecutive words, with the alignment of one: global_load_dwordx4
// needs 4-byte alignment only, so arrays at any address take the wide loads.
// The passes over the input read each word once: non-temporal loads leave
// the parent array and the minima in the L2s.
typedef u32 u32x4 __attribute__((ext_vector_type(4), aligned(4)));
__device__ __forceinline__ void load4(const u32* p, u32 (&x)[4]) {
  const u32x4 v = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(p));
#pragma unroll
  for (int e = 0; e < 4; ++e) x[e] = v[e];
}

// One wave's 256 consecutive records, lane l those at 4l .. 4l + 3; past the
// end copies of the last record, which change no minimum.  With `before`, lane
// 0 also gets the record before them ((0, 0), which no valid record precedes,
// before the first); by vector loads: LDS accesses would wait for scalar ones.
struct Unit {
  u32 s[4], d[4], w[4];
  u32 ps, pd;
};
__device__ __forceinline__ void load_unit(Unit& x, const UnionArgs& a, u64 unit, bool before) {
  const u64 r0 = unit * UNION_UNIT + 4 * lane_id();
  if ((unit + 1) * UNION_UNIT <= a.m) {
    load4(a.src + r0, x.s);
    load4(a.dst + r0, x.d);
    load4(a.wt + r0, x.w);
  } else {
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const u64 i = min(r0 + e, a.m - 1);
      x.s[e] = a.src[i];
      x.d[e] = a.dst[i];
      x.w[e] = a.wt[i];
    }
  }
  if (before) {
    x.ps = x.pd = 0;
    if (r0 != 0) {
      x.ps = a.src[min(r0, a.m) - 1];
      x.pd = a.dst[min(r0, a.m) - 1];
    }
  }
}

// ------------------------------------------------------------ union-find
// Roots of N vertices, their walks in lockstep so that a step's dependent
// loads are in flight together; a walk that has ended loads no more (the
// longest of a wave's walks is several times the mean).  A walk stores nothing
// but every eighth step (a load waits for the stores before it, a round trip to
// memory per step; the stores that remain let walks over a long chain double),
// and the root it found where (x's hash ^ salt) & thin is 0.  False where a
// walk takes more than `limit` steps.
template <int N, int STORE = 8>
__device__ __forceinline__ bool find_roots(u32* parent, u32 (&x)[N], u32 thin, u32 salt,
                                           u32 limit) {
  u32 p[N];
#pragma unroll
  for (int j = 0; j < N; ++j) p[j] = get(at(parent, x[j]));
  u32 open = 0, moved = 0;  // bit j: walk j has not ended / has left its first parent
#pragma unroll
  for (int j = 0; j < N; ++j) open |= p[j] != x[j] ? 1u << j : 0u;
  // (unrolled as far as a constant limit the loop costs 10^6 spokes of a wheel 475 us, not 405)
#pragma unroll 1
  for (u32 step = 1; __any(open != 0); ++step) {
    u32 y[N];
#pragma unroll
    for (int j = 0; j < N; ++j) {
      y[j] = p[j];
      if ((open >> j) & 1) y[j] = get(at(parent, p[j]));
    }
#pragma unroll
    for (int j = 0; j < N; ++j) {
      if (y[j] == p[j]) {
        open &= ~(1u << j);
      } else {
        moved |= 1u << j;
        p[j] = y[j];
        if (step % STORE == 0) put(at(parent, x[j]), y[j]);
      }
    }
    if (step > limit) return false;
  }
#pragma unroll
  for (int j = 0; j < N; ++j) {
    if (((moved >> j) & 1) && ((((x[j] * 0x9E3779B1u) >> 16) ^ salt) & thin) == 0)
      put(at(parent, x[j]), p[j]);
    x[j] = p[j];
  }
  return true;
}

// ------------------------------------------------------------ minima in LDS
// Minima of a workgroup's offers by vertex: few roots share many edges in
// late rounds, and atomics on one address take about 80 ns each.  First come,
// first served: an offer whose slot belongs to another vertex goes to the
// shared minimum at once.
constexpr int TABLE_BITS = 12;
struct OfferTable {
  static constexpr u32 SIZE = 1u << TABLE_BITS;
  u32 id[SIZE];
  u64 key[SIZE];
};
__device__ __forceinline__ void table_clear(OfferTable& t) {
  for (u32 i = threadIdx.x; i < t.SIZE; i += UT) {
    t.id[i] = NONE32;
    t.key[i] = VAL_NONE;
  }
}
__device__ __forceinline__ void table_offer(OfferTable& t, u64* best, u32 v, u64 k) {
  const u32 slot = (v * 0x9E3779B1u) >> (32 - TABLE_BITS);
  u32 owner = t.id[slot];
  if (owner == NONE32) owner = atomicCAS(&t.id[slot], NONE32, v);
  if (owner == NONE32 || owner == v) {
    if (k < t.key[slot])
      atomicMin(reinterpret_cast<unsigned long long*>(&t.key[slot]),
                static_cast<unsigned long long>(k));
    // keeps the two atomics apart: merged, they become one flat access
    asm volatile("; lds offer");
  } else {
    offer(best, v, k);
  }
}
__device__ __forceinline__ void table_flush(OfferTable& t, u64* best) {
  for (u32 i = threadIdx.x; i < t.SIZE; i += UT)
    if (t.id[i] != NONE32) offer(best, t.id[i], t.key[i]);
}

// ------------------------------------------------------------ pivots
// The sampled weights at the classes' ranks (a rank at or past `samples`: all
// ones, everything is below), by workgroup 0: a radix select over 8-bit
// digits, histograms of the samples still in the running from the highest
// digit that is not zero everywhere.  A class's size strays by the square root
// of its rank, and the first class is a few percent of a dense input: 4096
// samples where a solve takes long enough to pay for them.
constexpr u32 PIVOT_PER_THREAD = 4;
constexpr u32 PIVOT_SAMPLES_MAX = UT * PIVOT_PER_THREAD;
// Samples are runs of 16 records: 4096 records far apart are as many pages to
// one CU, 40 us (1024: 10 us).
constexpr u32 SAMPLE_RUN = 16;

__device__ __forceinline__ void pick_pivots(const UnionArgs& a) {
  __shared__ u32 h[256];
  __shared__ u32 s_scan[UW];
  __shared__ u32 s_digit, s_below, s_max, s_far, s_runs, s_hub;
  const u32 t = threadIdx.x, samples = a.samples;
  const u32 runs_of = (samples + SAMPLE_RUN - 1) / SAMPLE_RUN;
  if (t == 0) s_max = s_far = s_runs = s_hub = 0;
  __syncthreads();
  u32 x[PIVOT_PER_THREAD], mx = 0, far = 0, runs = 0;
#pragma unroll
  for (u32 j = 0; j < PIVOT_PER_THREAD; ++j) {
    const u32 q = j * UT + t;
    x[j] = 0;
    if (j * UT >= samples) continue;
    const u32 r = min(q, samples - 1);
    const u64 i = min((u64(r / SAMPLE_RUN) * a.m) / runs_of + r % SAMPLE_RUN, a.m - 1);
    x[j] = a.wt[i];
    mx = max(mx, x[j]);
    if (q < samples) {
      const u32 s = a.src[i], d = a.dst[i];
      far += max(s, d) - min(s, d) >= FAR_SPAN ? 1u : 0u;
      runs += i == 0 || a.src[i - 1] != s ? 1u : 0u;
      if (q % SAMPLE_RUN == 0 && q && a.src[(u64(q / SAMPLE_RUN - 1) * a.m) / runs_of] == s)
        atomicAdd(&s_hub, 1u);  // the row reaches back to the run before
    }
  }
#pragma unroll
  for (int o = WAVE / 2; o > 0; o >>= 1) {
    mx = max(mx, __shfl_xor(mx, o, WAVE));
    far += __shfl_xor(far, o, WAVE);
    runs += __shfl_xor(runs, o, WAVE);
  }
  if (lane_id() == 0) {
    atomicMax(&s_max, mx);
    atomicAdd(&s_far, far);
    atomicAdd(&s_runs, runs);
  }
  __syncthreads();
  if (t == 0) {
    put(a.ctl + UC_FAR, s_far);
    put(a.ctl + UC_RUNS, s_runs);
    put(a.ctl + UC_HUB, 5 * s_hub > runs_of ? 1u : 0u);
  }
  const int top = s_max >> 24 ? 24 : s_max >> 16 ? 16 : s_max >> 8 ? 8 : 0;
  u32 pivot = NONE32;
#pragma unroll
  for (u32 which = 0; which < UNION_CLASSES; ++which) {
    u32 want = a.rank[which];
    if (want >= samples) pivot = NONE32;
    else if (which == 0 || want != a.rank[which - 1]) {
      u32 prefix = 0;
      for (int shift = top; shift >= 0; shift -= 8) {
        if (t < 256) h[t] = 0;
        __syncthreads();
#pragma unroll
        for (u32 j = 0; j < PIVOT_PER_THREAD; ++j)
          if (j * UT + t < samples && (shift == top || (x[j] >> (shift + 8)) == prefix))
            atomicAdd(&h[(x[j] >> shift) & 255], 1u);
        __syncthreads();
        const u32 c = t < 256 ? h[t] : 0u;
        const u32 incl = wave_inclusive_sum(c);
        if (lane_id() == WAVE - 1) s_scan[wave_id()] = incl;
        __syncthreads();
        if (t < 256) {
          u32 below = incl - c;
          for (int w = 0; w < wave_id(); ++w) below += s_scan[w];
          if (want >= below && want < below + c) {
            s_digit = t;
            s_below = below;
          }
        }
        __syncthreads();
        prefix = (prefix << 8) | s_digit;
        want -= s_below;
        __syncthreads();
      }
      pivot = prefix;
    }
    if (t == 0) put(a.ctl + UC_PIVOT + which, pivot);
  }
}

// ------------------------------------------------------------ light pass
// Bound: 12 bytes per record from HBM, which it reads at 3.3 of the 4.9 TB/s of
// a copy at 10^6 vertices (3.2 10^7 records, 122 us) and at 2^24 (5.4 10^8, 1.87
// ms; 16 records per vertex 68 us and 1.0 ms).  The loads alone take 68 us at
// 10^6; listing the light edges adds 20 us, rows 13 us, minima 20 us (vector
// instructions fill 60 % of the issue slots; 143 us with shuffles through the
// LDS, wave-wide error masks, scalar loads that LDS accesses waited for, and
// atomics at the chunks' ends one by one).  Two units per step were slower (140).
//
// A list edge's key is (weight << 32) | the record's position.  Positions
// follow (min, max), so keys order the edges by (weight, min, max), parallel
// copies of one weight (the same triple) by position.
// The first minima are (weight << 32) | dst over a vertex's records in both
// directions: among the edges at one vertex v, dst < v sorts by min = dst
// before dst > v by max = dst, so (weight, dst) orders them as (weight, min,
// max) does, and no record needs its twin's position.  The input is sorted by
// src, so the minima are a segmented minimum over runs: a run inside a chunk of
// a.chunk consecutive units, which one wave takes, is stored; only the runs at
// the chunk's ends take an atomic.  Those wait in LDS and leave together: the
// next loads' wait includes an atomic's, some 5 us among streaming loads (at
// 2^24 vertices, 5.4 10^8 records, 32 chunks per wave: 0.3 of 1.95 ms).
__device__ __forceinline__ u64 dst_key(u32 w, u32 d) { return (u64(w) << 32) | d; }

// A run's lightest record so far; equal weights: the first one, as dst ascends.
// With `inside` the run began in this chunk, after its first record or with it.
struct Run {
  u32 s, w, d, inside;
};

// The run a chunk's next unit may continue (wave-uniform).
struct Carry {
  Run run;
  bool any;  // false at the chunk's first unit
};

// A wave's offers of its chunks' first and last runs.
struct Ends {
  u32 s[WAVE];
  u64 k[WAVE];
};
constexpr u32 ENDS_PER_UNIT = 4;  // at most: the carry, a lane's head, a lane's tail, the last tail

// The lanes' runs that end (sources at or past n share word n; every lane calls).
__device__ __forceinline__ void end_run(u64* best, u32 n, bool ends, const Run& r, Ends& pending,
                                        u32& count) {
  const u64 b = __ballot(ends && !r.inside);
  if (ends) {
    const u32 s = min(r.s, n);
    const u64 k = dst_key(r.w, r.d);
    if (r.inside) {
      put(at(best, s), k);
    } else {
      pending.s[count + mbcnt(b)] = s;
      pending.k[count + mbcnt(b)] = k;
    }
  }
  count += static_cast<u32>(__popcll(b));
}
__device__ __forceinline__ void offer_ends_of_chunks(u64* best, const Ends& pending, u32& count) {
  if (lane_id() < static_cast<int>(count)) lower(best, pending.s[lane_id()], pending.k[lane_id()]);
  count = 0;
}

// Segmented minimum over the lanes, a step: an open lane (its run began before
// it) takes over what the lane at the step's distance knows of the run.
template <int CTRL, int ROWS = 0xF>
__device__ __forceinline__ void scan_step(Run& r, u32& open) {
  const u32 w = dpp<CTRL, ROWS>(r.w, r.w), d = dpp<CTRL, ROWS>(r.d, r.d);
  const u32 in = dpp<CTRL, ROWS>(r.inside, r.inside), still = dpp<CTRL, ROWS>(open, open);
  if (open) {
    const bool first = w <= r.w;
    r.w = first ? w : r.w;
    r.d = first ? d : r.d;
    r.inside = in;
    open = still;
  }
}

// Minima of a unit.
__device__ __forceinline__ void run_minima(const Unit& x, bool first_unit, bool last_of_chunk,
                                           u32 n, u64* best, Carry& c, Ends& pending, u32& count) {
  const u32 lane = lane_id();
  Run tail{x.s[0], x.w[0], x.d[0], 1}, head = tail;
  bool multi = false;  // the lane's records hold more than one run
#pragma unroll
  for (int e = 1; e < 4; ++e) {
    if (x.s[e] != tail.s) {
      if (!multi) head = tail;
      else put(at(best, min(tail.s, n)), dst_key(tail.w, tail.d));  // a run inside the lane
      multi = true;
      tail = Run{x.s[e], x.w[e], x.d[e], 1};
    } else if (x.w[e] < tail.w) {
      tail.w = x.w[e];
      tail.d = x.d[e];
    }
  }
  // the run before a lane's: the previous lane's last one, or the carry
  bool joins = dpp<DPP_WAVE_SHR1>(0, tail.s) == x.s[0];
  u32 began = 1;  // the lane's first run began inside the chunk, if it joins none
  if (lane == 0) {
    joins = c.any && c.run.s == x.s[0];
    began = c.any || first_unit || x.ps != x.s[0] ? 1u : 0u;
    if (joins && !multi && c.run.w <= tail.w) {
      tail.w = c.run.w;
      tail.d = c.run.d;
    }
    if (!multi) tail.inside = joins ? c.run.inside : began;
  }
  end_run(best, n, lane == 0 && c.any && !joins, c.run, pending, count);
  u32 open = lane > 0 && joins && !multi ? 1u : 0u;
  scan_step<DPP_ROW_SHR + 1>(tail, open);
  scan_step<DPP_ROW_SHR + 2>(tail, open);
  scan_step<DPP_ROW_SHR + 4>(tail, open);
  scan_step<DPP_ROW_SHR + 8>(tail, open);
  scan_step<DPP_ROW_BCAST15, 0xA>(tail, open);
  scan_step<DPP_ROW_BCAST31, 0xC>(tail, open);
  const u32 pw = dpp<DPP_WAVE_SHR1>(c.run.w, tail.w), pd = dpp<DPP_WAVE_SHR1>(c.run.d, tail.d);
  const u32 pin = dpp<DPP_WAVE_SHR1>(c.run.inside, tail.inside);
  const u32 next_s = dpp<DPP_WAVE_SHL1>(tail.s, x.s[0]);
  if (multi) {
    if (joins && pw <= head.w) {
      head.w = pw;
      head.d = pd;
    }
    head.inside = joins ? pin : began;
  }
  end_run(best, n, multi, head, pending, count);
  const u32 inside = tail.inside;
  if (lane == WAVE - 1) tail.inside = 0;  // the next chunk may continue it
  end_run(best, n, lane < WAVE - 1 ? next_s != tail.s : last_of_chunk, tail, pending, count);
  c.run.s = __builtin_amdgcn_readlane(tail.s, WAVE - 1);
  c.run.w = __builtin_amdgcn_readlane(tail.w, WAVE - 1);
  c.run.d = __builtin_amdgcn_readlane(tail.d, WAVE - 1);
  c.run.inside = __builtin_amdgcn_readlane(inside, WAVE - 1);
  c.any = !last_of_chunk;
}

// What a workgroup found in the input.
struct Found {
  u64 hash_fwd, hash_rev;
  u32 fwd, bad, dup;
};

// A wave's own lists, in its range of `cap` edges of both buffers: c edges
// from `base` of the first one on; the later light classes' rest1 and rest2 edges from
// the range's end down, the second class in the second buffer and the third in
// the first.  Every edge comes from one of the wave's own records, so cap
// (their number) is never exceeded, whatever the input.
struct WaveLists {
  u64 base, cap;
  u32 c, rest1, rest2;
};

// The units of a wave: chunks of `chunk` consecutive units, the chunks dealt
// to the waves in turn.
struct UnitWalk {
  u64 unit, end, left_in_chunk, skip;
  u32 chunk;
  __device__ __forceinline__ UnitWalk(const UnionArgs& a, u64 wave, u64 waves, u64 units)
      : unit(wave * a.chunk), end(units), left_in_chunk(a.chunk), skip((waves - 1) * a.chunk),
        chunk(a.chunk) {}
  __device__ __forceinline__ bool valid() const { return unit < end; }
  __device__ __forceinline__ bool first_of_chunk() const { return left_in_chunk == chunk; }
  __device__ __forceinline__ bool last_of_chunk() const {
    return left_in_chunk == 1 || unit + 1 == end;
  }
  __device__ __forceinline__ void next() {
    ++unit;
    if (--left_in_chunk == 0) {
      unit += skip;
      left_in_chunk = chunk;
    }
  }
};

// A wave's taken edges wait in LDS and leave 64 at a time, in whole lines
// (stored as they were taken, a few per unit, they cost 70 of 178 us at 10^6
// vertices, 3.2 10^7 records).  Class c at [c * STAGE, (c + 1) * STAGE).
constexpr u32 STAGE = 2 * WAVE;
struct Stage {
  u32 s[UNION_CLASSES * STAGE], d[UNION_CLASSES * STAGE];
  u64 v[UNION_CLASSES * STAGE];
  Ends ends;
};

// The first min(n, 64) staged edges of a class to its list, the rest (fewer
// than 64) to the front.
template <int CLASS>
__device__ __forceinline__ void drain(const UnionArgs& a, WaveLists& l, Stage& st, u32& n) {
  const u32 lane = lane_id(), at = CLASS * STAGE + lane, out = min<u32>(n, WAVE);
  if (lane < out) {
    const u64 q = CLASS ? l.base + l.cap - 1 - ((CLASS == 1 ? l.rest1 : l.rest2) + lane)
                        : l.base + l.c + lane;
    a.s[CLASS & 1][q] = st.s[at];
    a.d[CLASS & 1][q] = st.d[at];
    a.v[CLASS & 1][q] = st.v[at];
  }
  (CLASS == 0 ? l.c : CLASS == 1 ? l.rest1 : l.rest2) += out;
  n -= out;
  if (lane < n) {
    st.s[at] = st.s[at + WAVE];
    st.d[at] = st.d[at + WAVE];
    st.v[at] = st.v[at + WAVE];
  }
}

__device__ __forceinline__ void light_pass(const UnionArgs& a, WaveLists& l, UnitWalk walk, Stage& st,
                                           Found& out) {
  __shared__ Found s_found[UW];
  const int lane = lane_id();
  const u32 q0 = get(a.ctl + UC_PIVOT), q1 = get(a.ctl + UC_PIVOT + 1),
            q2 = get(a.ctl + UC_PIVOT + 2);
  u32* const span = reinterpret_cast<u32*>(a.span);
  u32 top = 0, loop = NONE32;  // the largest id, the smallest src ^ dst of the lane's records
  u32 unordered = 0, dup = 0, fwd = 0;  // wave-uniform
  u64 hf = 0, hall = 0;  // hash sums of the forward and of all records
  Carry carry{{0, 0, 0, 0}, false};
  Ends& ends = st.ends;
  u32 n0 = 0, n1 = 0, n2 = 0;  // staged edges of the classes
  u32 n_ends = 0;
  Unit next;
  u32 last_s = 0, last_d = 0;  // of the unit before, in the same chunk
  if (walk.valid()) load_unit(next, a, walk.unit, true);
  while (walk.valid()) {
    Unit x = next;
    if (!walk.first_of_chunk()) {
      x.ps = last_s;
      x.pd = last_d;
    }
    last_s = __builtin_amdgcn_readlane(x.s[3], WAVE - 1);
    last_d = __builtin_amdgcn_readlane(x.d[3], WAVE - 1);
    const u64 unit = walk.unit;
    const bool last = walk.last_of_chunk();
    walk.next();
    if (walk.valid()) load_unit(next, a, walk.unit, walk.first_of_chunk());
    const u64 r0 = unit * UNION_UNIT + 4 * lane;
    const bool full = (unit + 1) * UNION_UNIT <= a.m;
    u32 ps = dpp<DPP_WAVE_SHR1>(x.ps, x.s[3]), pd = dpp<DPP_WAVE_SHR1>(x.pd, x.d[3]);
    u64 listed[4], descents = 0;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const u32 s = x.s[e], d = x.d[e], w = x.w[e];
      const u64 in = full ? ~0ull : __ballot(r0 + e < a.m);
      const u32 lo = min(s, d), hi = max(s, d);
      top = max(top, hi);
      loop = min(loop, s ^ d);
      descents |= __ballot(((u64(ps) << 32) | pd) >= ((u64(s) << 32) | d)) & in;
      if (ps != s) {  // (the first record's predecessor is (0, 0): row 0 ends, or begins, at 0)
        put(at(span, 2 * min(ps, a.n) + 1), static_cast<u32>(r0 + e));
        put(at(span, 2 * min(s, a.n)), static_cast<u32>(r0 + e));
      }
      ps = s;
      pd = d;
      const u64 f = __ballot(s < d) & in;
      u64 h = sym_hash(lo, hi, w);
      if (!full && r0 + e >= a.m) h = 0;
      fwd += static_cast<u32>(__popcll(f));
      hf += s < d ? h : 0ull;
      hall += h;
      listed[e] = f & __ballot(w <= q2);
    }
    if (r0 < a.m && r0 + 4 >= a.m) put(at(span, 2 * min(x.s[3], a.n) + 1), static_cast<u32>(a.m));
    if (descents) {  // parallel records or disorder (or record 0 is (0, 0): a self-loop)
      ps = dpp<DPP_WAVE_SHR1>(x.ps, x.s[3]);
      pd = dpp<DPP_WAVE_SHR1>(x.pd, x.d[3]);
      for (int e = 0; e < 4; ++e) {
        const bool here = r0 + e < a.m;
        const u64 prev = (u64(ps) << 32) | pd, now = (u64(x.s[e]) << 32) | x.d[e];
        unordered |= __any(here && prev > now) ? 1u : 0u;
        dup |= __any(here && prev == now) ? 1u : 0u;
        ps = x.s[e];
        pd = x.d[e];
      }
    }
    if (n_ends > WAVE - ENDS_PER_UNIT) offer_ends_of_chunks(a.best[0], ends, n_ends);
    run_minima(x, unit == 0, last, a.n, a.best[0], carry, ends, n_ends);
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      if (!listed[e]) continue;
      const u32 w = x.w[e];
      const u64 b0 = listed[e] & __ballot(w <= q0), b1 = listed[e] & __ballot(w <= q1) & ~b0,
                b2 = listed[e] & ~(b0 | b1);
      if ((listed[e] >> lane) & 1) {
        u32 q = n0 + mbcnt(b0);
        if (w > q0) q = w > q1 ? 2 * STAGE + n2 + mbcnt(b2) : STAGE + n1 + mbcnt(b1);
        st.s[q] = x.s[e];
        st.d[q] = x.d[e];
        st.v[q] = (u64(w) << 32) | (r0 + e);
      }
      n0 += static_cast<u32>(__popcll(b0));
      n1 += static_cast<u32>(__popcll(b1));
      n2 += static_cast<u32>(__popcll(b2));
      if (n0 >= WAVE) drain<0>(a, l, st, n0);
      if (n1 >= WAVE) drain<1>(a, l, st, n1);
      if (n2 >= WAVE) drain<2>(a, l, st, n2);
    }
  }
  offer_ends_of_chunks(a.best[0], ends, n_ends);
  if (n0) drain<0>(a, l, st, n0);
  if (n1) drain<1>(a, l, st, n1);
  if (n2) drain<2>(a, l, st, n2);
#pragma unroll
  for (int o = WAVE / 2; o > 0; o >>= 1) {
    hf += __shfl_xor(hf, o, WAVE);
    hall += __shfl_xor(hall, o, WAVE);
    top = max(top, __shfl_xor(top, o, WAVE));
    loop = min(loop, __shfl_xor(loop, o, WAVE));
  }
  if (lane == 0)
    s_found[wave_index()] = Found{hf, hall - hf, fwd,
                                  (top >= a.n || loop == 0 ? u32(ERR_INVALID) : 0u) |
                                      (unordered ? u32(ERR_UNSORTED) : 0u),
                                  dup};
  __syncthreads();
  if (threadIdx.x == 0) {
    Found f{0, 0, 0, 0, 0};
    for (int w = 0; w < UW; ++w) {
      f.hash_fwd += s_found[w].hash_fwd;
      f.hash_rev += s_found[w].hash_rev;
      f.fwd += s_found[w].fwd;
      f.bad |= s_found[w].bad;
      f.dup |= s_found[w].dup;
    }
    out = f;
  }
}

// ------------------------------------------------------------ crossing edges
// Nearly every crossing edge touches one giant component, whose minimum would
// take one atomic per edge at one address.  It gets none: a root without a
// minimum hooks nowhere, and the components that choose an edge to it hook
// onto it, which is all a round needs to make progress.  Any root may be the
// passive one: the most frequent root of 64 sampled vertices.
// The flatten marks its component in a bitmap (n / 8 bytes); most records lie
// inside it.
// Neither changes in these passes: after an acquire at agent scope plain loads
// are current, and the gathers of a source's records hit the L1.
__device__ __forceinline__ u32 most_frequent(u32 x) {
  u32 votes = 0;
  for (int i = 0; i < WAVE; ++i) votes += __shfl(x, i, WAVE) == x ? 1u : 0u;
  u32 most = votes;
#pragma unroll
  for (int o = WAVE / 2; o > 0; o >>= 1) most = max(most, __shfl_xor(most, o, WAVE));
  return __shfl(x, __ffsll(static_cast<unsigned long long>(__ballot(votes == most))) - 1, WAVE);
}
__device__ __forceinline__ u32 pick_giant(const UnionArgs& a) {
  // (the roots do not change meanwhile: every workgroup picks the same)
  u32 x[1] = {static_cast<u32>((u64(lane_id()) * a.n) / WAVE)};
  (void)find_roots<1>(a.parent, x, NONE32, 0, WALK_LIMIT);
  return most_frequent(x[0]);
}
// A graph of unconnected parts has a giant each, one wave per part picks it.
// They are marked by a byte each, and their minima in both arrays are 0, which no
// offer lowers and no edge's key equals but that of the lightest edge of all, a
// true minimum of its ends.
__device__ __forceinline__ void pick_giants(const UnionArgs& a, u64 wave, u64 waves, bool again) {
  for (u64 p = wave; p < a.parts; p += waves) {
    const u32 v0 = a.part_off[p], len = a.part_off[p + 1] - v0;
    const bool lead = lane_id() == 0;
    if (again && lead) {
      const u32 old = get(a.part_giant + p);
      if (old != NONE32) put(a.giants + old, u8{0});
    }
    u32 g = NONE32;
    if (len) {
      u32 x[1] = {v0 + static_cast<u32>((u64(lane_id()) * len) / WAVE)};
      (void)find_roots<1>(a.parent, x, NONE32, 0, WALK_LIMIT);
      g = most_frequent(x[0]);
    }
    if (!lead) continue;
    put(a.part_giant + p, g);
    if (g != NONE32) put(a.giants + g, u8{1});
  }
}

__device__ __forceinline__ void offer_ends(u64* best, u32 s, u32 d, u64 k, u32 giant) {
  if (s != giant) offer(best, s, k);
  if (d != giant) offer(best, d, k);
}

// Appends to the wave's list the edges of four per lane whose ends (roots,
// 0 / 0 where a lane has none) differ, with their offers.
__device__ __forceinline__ void append_crossing(const UnionArgs& a, WaveLists& l, const u32 (&s)[4],
                                                const u32 (&d)[4], const u64 (&k)[4], u64* best,
                                                u32 giant) {
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const u64 b = __ballot(s[e] != d[e]);
    if (!b) continue;
    if (s[e] != d[e]) {
      const u64 q = l.base + l.c + mbcnt(b);
      a.s[0][q] = s[e];
      a.d[0][q] = d[e];
      a.v[0][q] = k[e];
      offer_ends(best, s[e], d[e], k[e], giant);
    }
    l.c += static_cast<u32>(__popcll(b));
  }
}

// A later light class: the wave's own list, from its low end up (the third
// class's crossing edges go to the same range's front: what is appended never
// reaches what is still to be read).
// With `filter`, where most vertices are inside the giant, an edge's ends are
// first looked up in its bitmap, which stays in the L2s where the parent array
// does not.  At 2^24 vertices, 2.5 10^7 edges of the third class, 0.88 of the
// vertices inside: 550 us without, 410 with the lookup; of the second class, half
// of the vertices inside, 350 either way.
__device__ __forceinline__ void cross_list(const UnionArgs& a, WaveLists& l, u32 cls, u64* best,
                                           u32 giant, bool filter) {
  const bool second = cls == 1;
  const u32 *ls = second ? a.s[1] : a.s[0], *ld = second ? a.d[1] : a.d[0];
  const u64* lv = second ? a.v[1] : a.v[0];
  const u32 listed = second ? l.rest1 : l.rest2;
  const u64 lo = l.base + l.cap - listed;
  for (u32 j0 = 0; j0 < listed; j0 += 4 * WAVE) {
    u32 x[8], s[4], d[4];
    u64 k[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const u64 q = lo + min<u32>(j0 + e * WAVE + lane_id(), listed - 1);
      x[e] = ls[q];
      x[4 + e] = ld[q];
      k[e] = lv[q];
    }
    u32 skip = 0;  // bit e: both ends inside
    if (filter) {
      u32 b[8];
      const u32* bits = reinterpret_cast<const u32*>(a.bits);
#pragma unroll
      for (int e = 0; e < 8; ++e) b[e] = *at(bits, x[e] >> 5);
#pragma unroll
      for (int e = 0; e < 4; ++e)
        skip |= ((b[e] >> (x[e] & 31)) & (b[4 + e] >> (x[4 + e] & 31)) & 1u) << e;
    }
    if (__all(skip == 15)) continue;
#pragma unroll
    for (int e = 0; e < 8; ++e)
      if (!((skip >> (e & 3)) & 1)) x[e] = *at(a.parent, x[e]);
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const bool in = j0 + e * WAVE + lane_id() < listed && !((skip >> e) & 1);
      s[e] = in ? x[e] : 0u;
      d[e] = in ? x[4 + e] : 0u;
    }
    append_crossing(a, l, s, d, k, best, giant);
  }
}

// The rest of the input where the giant leaves many records outside, or rows
// too long for one wave: the wave's own forward records above the pivot, two
// units per step, every load of a kind in flight before the next kind's.
__device__ __forceinline__ void cross_input(const UnionArgs& a, WaveLists& l, UnitWalk walk,
                                            u64* best, u32 giant) {
  constexpr int U = 2;
  const u32 pivot = get(a.ctl + UC_PIVOT + UNION_CLASSES - 1);
  while (walk.valid()) {
    Unit x[U];
    u64 r0[U];
    int have = 0;  // (wave-uniform)
#pragma unroll
    for (int u = 0; u < U; ++u) {
      r0[u] = a.m;
      if (walk.valid()) {
        r0[u] = walk.unit * UNION_UNIT + 4 * lane_id();
        load_unit(x[u], a, walk.unit, false);
        walk.next();
        have = u + 1;
      }
    }
    u32 live = 0;  // bit 4u + e
#pragma unroll
    for (int u = 0; u < U; ++u)
      if (u < have)
#pragma unroll
        for (int e = 0; e < 4; ++e)
          live |= r0[u] + e < a.m && x[u].w[e] > pivot && x[u].s[e] < x[u].d[e] ? 1u << (4 * u + e) : 0u;
    {
      u64 bd[4 * U], bs[4 * U];
#pragma unroll
      for (int k = 0; k < 4 * U; ++k) {
        bd[k] = 0;
        bs[k] = 0;
        if ((live >> k) & 1) {
          bd[k] = a.bits[x[k / 4].d[k % 4] >> 6];
          bs[k] = a.bits[x[k / 4].s[k % 4] >> 6];
        }
      }
#pragma unroll
      for (int k = 0; k < 4 * U; ++k)
        if ((bd[k] >> (x[k / 4].d[k % 4] & 63)) & (bs[k] >> (x[k / 4].s[k % 4] & 63)) & 1)
          live &= ~(1u << k);
    }
    if (!__any(live != 0)) continue;
    u32 s[U][4], d[U][4];
#pragma unroll
    for (int k = 0; k < 4 * U; ++k) {
      s[k / 4][k % 4] = d[k / 4][k % 4] = 0;
      if ((live >> k) & 1) {
        s[k / 4][k % 4] = *at(a.parent, x[k / 4].s[k % 4]);
        d[k / 4][k % 4] = *at(a.parent, x[k / 4].d[k % 4]);
      }
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      if (u >= have) continue;
      u64 k[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) k[e] = (u64(x[u].w[e]) << 32) | (r0[u] + e);
      append_crossing(a, l, s[u], d[u], k, best, giant);
    }
  }
}

// The rest of the input where the giant leaves few records outside: a crossing
// edge has an end outside, so the rows of the vertices outside hold them all.
// A wave takes 64 vertices at a time (the flatten's share of the wave), and its
// lanes spread over the records of their rows together.  An edge with one end
// inside is found from its outer end; its key is the position of its forward
// record, which a binary search of the inner end's row finds (no parallel
// records: the position is unique).  At 10^6 vertices, 3.2 10^7 records: 12 us,
// a pass over the input 146 us; at 2^24, 5.4 10^8: 130 to 200 us and 3.1 ms.
constexpr u64 ROW_LONG = 4096;   // a longer row outside: cross_input instead
constexpr u64 ROWS_SHARE = 4;    // also with more than 1/4 of the records outside
struct Rows {
  u32 upto[WAVE];   // records of the group's rows up to this one's end
  u32 shift[WAVE];  // position of the row's j-th record of the group: shift + j
  u32 root[WAVE];
};
__device__ __forceinline__ void cross_rows(const UnionArgs& a, WaveLists& l, u64 wave, u64 waves,
                                           u64* best, u32 giant, Rows& rows) {
  const u32 pivot = get(a.ctl + UC_PIVOT + UNION_CLASSES - 1);
  const u64 groups = (u64(a.n) + WAVE - 1) / WAVE;
  const u32 lane = lane_id();
  for (u64 g0 = wave; g0 < groups; g0 += waves * WAVE) {
    const u64 own = g0 + lane * waves;
    const u64 word = own < groups ? a.bits[own] : ~0ull;
    for (u64 todo = __ballot(word != ~0ull); todo; todo &= todo - 1) {
      const u32 i = static_cast<u32>(__ffsll(static_cast<unsigned long long>(todo)) - 1);
      const u64 v0 = (g0 + i * waves) * WAVE;
      const u64 in = __shfl(static_cast<unsigned long long>(word), i, WAVE);
      u32 begin = 0, len = 0, root = 0;
      if (!((in >> lane) & 1) && v0 + lane < a.n) {
        const u64 sp = a.span[v0 + lane];
        begin = static_cast<u32>(sp);
        len = static_cast<u32>(sp >> 32) - begin;
        root = *at(a.parent, static_cast<u32>(v0) + lane);
      }
      const u32 upto = wave_inclusive_sum(len);
      const u32 total = __shfl(upto, WAVE - 1, WAVE);
      rows.upto[lane] = upto;
      rows.shift[lane] = begin - (upto - len);
      rows.root[lane] = root;
      __builtin_amdgcn_wave_barrier();
      for (u32 j0 = 0; j0 < total; j0 += 4 * WAVE) {
        u32 s[4], d[4], rs[4], w[4], p[4];
        bool ok[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const u32 j = min(j0 + e * WAVE + lane, total - 1);
          u32 r = 0;
#pragma unroll
          for (u32 h = WAVE / 2; h > 0; h >>= 1) r += rows.upto[r + h - 1] <= j ? h : 0u;
          p[e] = rows.shift[r] + j;
          rs[e] = rows.root[r];
          s[e] = static_cast<u32>(v0) + r;
          d[e] = a.dst[p[e]];
          w[e] = a.wt[p[e]];
          ok[e] = j0 + e * WAVE + lane < total;
        }
        u32 rd[4];
        bool inner[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          ok[e] = ok[e] && w[e] > pivot;
          inner[e] = ok[e] && ((a.bits[d[e] >> 6] >> (d[e] & 63)) & 1);
        }
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          rd[e] = rs[e];
          if (ok[e] && (inner[e] || s[e] < d[e])) rd[e] = *at(a.parent, d[e]);
          ok[e] = rd[e] != rs[e];
        }
        // positions of the forward records
        u32 lo[4], hi[4];
        u32 open = 0;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          lo[e] = p[e];
          hi[e] = p[e];
          if (ok[e] && s[e] > d[e]) {
            const u64 sp = a.span[d[e]];
            lo[e] = row_first(sp);
            hi[e] = row_last(sp);
          }
        }
        do {
          u32 x[4];
          open = 0;
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            x[e] = 0;
            if (lo[e] < hi[e]) x[e] = a.dst[lo[e] + (hi[e] - lo[e]) / 2];
          }
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            if (lo[e] >= hi[e]) continue;
            const u32 mid = lo[e] + (hi[e] - lo[e]) / 2;
            if (x[e] < s[e]) lo[e] = mid + 1;
            else hi[e] = mid;
            open |= lo[e] < hi[e] ? 1u : 0u;
          }
        } while (__any(open != 0));
        u64 k[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          k[e] = (u64(w[e]) << 32) | lo[e];
          if (!ok[e]) rs[e] = rd[e];
        }
        append_crossing(a, l, rs, rd, k, best, giant);
      }
      __builtin_amdgcn_wave_barrier();
    }
  }
}

// ------------------------------------------------------------ rounds
constexpr int UR = 4;  // rows of one edge per lane a wave loads before use

// With `first` the minima are the light pass's, (weight << 32) | the other
// end; parallel copies of one weight then share a minimum, so with copies in
// the input the hook claims its child and one of them is taken.  Returns the
// wave's roots that live on, with `note` listed from the start of the wave's range
// of the second buffer (the later class lies at its end: both fit).
__device__ __forceinline__ u32 hook(const UnionArgs& a, const WaveLists& l, int cur, bool first,
                                    bool copies, u32 giant, u32* parent, bool note) {
  const u64* best = minima(a, cur);
  u64* next = minima(a, cur ^ 1);
  u32 live = 0;
  for (u32 j0 = 0; j0 < l.c; j0 += UR * WAVE) {
    u32 x[UR], y[UR];
    u64 k[UR], bx[UR], by[UR];
#pragma unroll
    for (int u = 0; u < UR; ++u) {
      const u64 i = l.base + min<u32>(j0 + u * WAVE + lane_id(), l.c - 1);
      x[u] = a.s[0][i];
      y[u] = a.d[0][i];
      k[u] = a.v[0][i];
    }
#pragma unroll
    for (int u = 0; u < UR; ++u) {
      bx[u] = get(at(best, x[u]));
      by[u] = get(at(best, y[u]));
    }
#pragma unroll
    for (int u = 0; u < UR; ++u) {
      const u32 w = static_cast<u32>(k[u] >> 32);
      // (the passive root's word is an old minimum)
      const bool mx = bx[u] == (first ? dst_key(w, y[u]) : k[u]) && x[u] != giant;
      const bool my = by[u] == (first ? dst_key(w, x[u]) : k[u]) && y[u] != giant;
      u32 child = x[u], other = y[u];
      bool lives = false;
      if (j0 + u * WAVE + lane_id() < l.c && (mx || my)) {
        if (mx && my) {
          child = max(x[u], y[u]);
          other = min(x[u], y[u]);
        } else if (my) {
          child = y[u];
          other = x[u];
        }
        bool hooked = true;
        if (copies) {
          // a wave's lanes hold the copies of one edge together: the first of them
          // claims its child, if no other wave has (claims of one address take 12 ns each:
          // 10^6 copies between two vertices 12 ms, without the look and the choice)
          const u32 lead = __builtin_amdgcn_readfirstlane(child);
          const u64 same = __ballot(child == lead);
          hooked = (child != lead || mbcnt(same) == 0) && get(at(parent, child)) == child &&
                   atomicCAS(at(parent, child), child, other) == child;
        } else {
          put(at(parent, child), other);
        }
        if (hooked) {
          lives = mx && my;
          if (lives) put(at(next, other), VAL_NONE);  // the root that lives on
          const u32 pos = static_cast<u32>(k[u]);
          (void)__hip_atomic_fetch_or(a.marks + (pos >> 5), 1u << (pos & 31), __ATOMIC_RELAXED,
                                      __HIP_MEMORY_SCOPE_AGENT);
        }
      }
      const u64 b = __ballot(lives);
      if (note && lives) a.s[1][l.base + live + mbcnt(b)] = other;
      live += static_cast<u32>(__popcll(b));
    }
  }
  return live;
}

// Rounds with at most this many live roots fold their offers in LDS; with
// more, most offers of a workgroup are to distinct roots.
// So do inputs where one vertex has a fifth of the records, whatever the roots: every
// wave's minimum goes to it, 80 ns each.  Wheels of 10^6 vertices, hub edges the heaviest, at the
// lowest and the highest id: 1950 and 2054 us, with the fold 1063 and 1768 (round loop
// 1595 and 1224); of 2^17 457 and 427, 396 and 275 (690 and 674).  With an eighth of the
// records, beside a band of 2^17 vertices, the fold makes no difference (505 us; 800).
constexpr u64 TABLE_LIVE = u64{1} << TABLE_BITS;

// Every vertex onto its root, 24 steps of all walks at a time: where all
// vertices of a chain walk together and store every third step, a chain's length
// falls to a quarter in three steps.  More vertices than threads take walk in
// turn, hence the passes.
constexpr u32 SHORTEN_STEPS = 24;
constexpr u32 SHORTEN_PASSES = 32;  // 25^32: more is a corrupted forest
__device__ __forceinline__ bool shorten_chains(const UnionArgs& a, Barrier& bar, u32 gthread,
                                               u32 threads) {
  for (u32 pass = 0; pass < SHORTEN_PASSES; ++pass) {
    bool open = false;
    for (u64 v0 = gthread; v0 < a.n; v0 += 4 * threads) {
      u32 x[4];
#pragma unroll
      for (u32 j = 0; j < 4; ++j)
        x[j] = static_cast<u32>(v0 + j * threads < a.n ? v0 + j * threads : v0);
      if (!find_roots<4, 3>(a.parent, x, 0, 0, SHORTEN_STEPS)) open = true;
    }
    u64 sum;
    if (!sync_grid(bar, block_total(__any(open) ? 1 : 0), sum)) return false;
    if (!sum) return true;
  }
  if (gthread == 0) atomicOr(a.err, ERR_SPIN);
  return false;
}

// True where the wave met a deep chain: its edges from there on are kept as they
// were.  After shorten_chains the same call finishes the round (what it offered
// before, it offers again).
__device__ __forceinline__ bool relabel(const UnionArgs& a, WaveLists& l, int out, u64 live,
                                        bool table, OfferTable& t, u32 giant, u32 wave) {
  u64* best = minima(a, out);
  // with few roots every wave meets the same ones: some waves' stores do
  const u32 thin = live > TABLE_LIVE ? 0u : live > 1024 ? 3u : live > 128 ? 31u : 255u;
  if (table) {
    table_clear(t);
    __syncthreads();
  }
  u32 kept = 0;
  bool deep = false;
  for (u32 j0 = 0; j0 < l.c; j0 += UR * WAVE) {
    u32 xy[2 * UR];
    u64 k[UR];
#pragma unroll
    for (int u = 0; u < UR; ++u) {
      const u64 i = l.base + min<u32>(j0 + u * WAVE + lane_id(), l.c - 1);
      xy[u] = a.s[0][i];
      xy[UR + u] = a.d[0][i];
      k[u] = a.v[0][i];
    }
    deep = deep || !find_roots<2 * UR>(a.parent, xy, thin, wave, WALK_DEEP);
#pragma unroll
    for (int u = 0; u < UR; ++u) {
      const u32 x = xy[u], y = xy[UR + u];
      const bool keep = j0 + u * WAVE + lane_id() < l.c && x != y;
      const u64 b = __ballot(keep);
      if (keep) {
        // in place: the rows up to here have been read
        const u64 q = l.base + kept + mbcnt(b);
        a.s[0][q] = x;
        a.d[0][q] = y;
        a.v[0][q] = k[u];
        if (deep) {
        } else if (table) {
          if (x != giant) table_offer(t, best, x, k[u]);
          if (y != giant) table_offer(t, best, y, k[u]);
        } else {
          offer_ends(best, x, y, k[u], giant);
        }
      }
      kept += static_cast<u32>(__popcll(b));
    }
  }
  l.c = kept;
  if (table) {
    __syncthreads();
    table_flush(t, best);
  }
  return deep;
}

// Every one of `count` parents in LDS onto its root (all threads call, *open is 0
// before; ends with a barrier), and beside(i) for each.  A walk stops after LDS_WALK
// steps and all walk again from where they are: a chain falls to a sixteenth.  Walked to
// the end in one go, with the root at the highest id, a band of 4096 vertices took 435 us a
// call (60 now), a ring of 8192 1700 (78); random trees, some ten deep, take one pass and 0.2
// us a round for the look at *open (2^8 vertices 47.9 -> 48.9 us).  A store every step
// costs those 3 us a round.
constexpr u32 LDS_WALK = 16;
constexpr u32 LDS_PASSES = 6;  // 16^6: more is a cycle
template <typename F>
__device__ __forceinline__ void roots_in_lds(u32* parent, u32 count, u32* open, F&& beside) {
  for (u32 pass = 1;; ++pass) {
    for (u32 i = threadIdx.x; i < count; i += UT) {
      // (others shorten the walked paths meanwhile)
      u32 r = parent[i], steps = 0;
      for (u32 p; (p = parent[r]) != r && steps < LDS_WALK; ++steps) r = p;
      parent[i] = r;
      beside(i);
      if (steps == LDS_WALK) *open = pass;
    }
    __syncthreads();
    if (*open < pass || pass == LDS_PASSES) return;
  }
}

// Few roots: with at most DENSE_MAX of them left in the first class's rounds,
// the lists hold dense ids.  A round's hooks then lie over few words, which every
// workgroup reads into its LDS and resolves there, where a step of a walk takes a
// tenth of the time (the trees of a round are some ten hooks deep); and its
// offers meet in LDS before they go to the shared minima.  A graph of at most
// DENSE_MAX vertices begins this way, its ids being the vertices.
// At 10^6 vertices, 2 10^5 edges left, rounds of 1500 roots and less relabel in 9
// to 7 us, 40 to 9 as walks with a hashed table of minima; at 2^14, 3 10^4 edges, in 8
// to 5 us, 18 to 7.  Entering takes two barriers more: not worth it with few
// edges (geometric graphs, 13 us of 570 at 10^6 vertices), nor with more ids for every workgroup to
// read (with 8192 a solve of 2^17 vertices takes 15 us more than with 4096).
constexpr u32 DENSE_MAX = 4096;
constexpr u64 DENSE_EDGES = 16, DENSE_EDGES_MIN = 4096;  // edges per root, and in all, at least
struct DenseRound {
  u32 root[DENSE_MAX];
  u64 best[DENSE_MAX];
  u32 open;
};
// With `enter` the lists still hold vertices.  True where the wave met a deep
// chain: it keeps the edges from there on as vertices, marked by UNRESOLVED.
constexpr u32 UNRESOLVED = 0x80000000u;
static_assert(UNION_VERTICES_MAX <= UNRESOLVED, "bit 31 of a vertex is free");
__device__ __forceinline__ bool relabel_dense(const UnionArgs& a, WaveLists& l, int out, u32 ids,
                                              bool enter, const u32* parent, DenseRound& t,
                                              u32 wave) {
  u64* best = minima(a, out);
  if (threadIdx.x == 0) t.open = 0;
  for (u32 i = threadIdx.x; i < ids; i += UT) t.best[i] = VAL_NONE;
  if (!enter) {
    u32 p[DENSE_MAX / UT];  // all in flight together
#pragma unroll
    for (u32 j = 0; j < DENSE_MAX / UT; ++j)
      if (j * UT < ids) p[j] = get(at(parent, min(j * UT + threadIdx.x, ids - 1)));
#pragma unroll
    for (u32 j = 0; j < DENSE_MAX / UT; ++j)
      if (j * UT + threadIdx.x < ids) t.root[j * UT + threadIdx.x] = p[j];
  }
  __syncthreads();
  if (!enter) {
    roots_in_lds(t.root, ids, &t.open, [](u32) {});
  }
  u32 kept = 0;
  bool deep = false;
  for (u32 j0 = 0; j0 < l.c; j0 += UR * WAVE) {
    u32 xy[2 * UR];
    u64 k[UR];
#pragma unroll
    for (int u = 0; u < UR; ++u) {
      const u64 i = l.base + min<u32>(j0 + u * WAVE + lane_id(), l.c - 1);
      xy[u] = a.s[0][i];
      xy[UR + u] = a.d[0][i];
      k[u] = a.v[0][i];
    }
    if (enter) {
      deep = deep || !find_roots<2 * UR>(a.parent, xy, 31, wave, WALK_DEEP);
      u32 id[2 * UR];
#pragma unroll
      for (int u = 0; u < 2 * UR; ++u) id[u] = get(at(a.dense_id, xy[u]));
#pragma unroll
      for (int u = 0; u < 2 * UR; ++u)  // (a root without an id: none, if symmetric)
        xy[u] = deep ? xy[u] | UNRESOLVED : min(id[u], ids - 1);
    } else {
#pragma unroll
      for (int u = 0; u < 2 * UR; ++u) xy[u] = t.root[xy[u]];
    }
#pragma unroll
    for (int u = 0; u < UR; ++u) {
      const u32 x = xy[u], y = xy[UR + u];
      const bool keep = j0 + u * WAVE + lane_id() < l.c && x != y;
      const u64 b = __ballot(keep);
      if (keep) {
        // in place: the rows up to here have been read
        const u64 q = l.base + kept + mbcnt(b);
        a.s[0][q] = x;
        a.d[0][q] = y;
        a.v[0][q] = k[u];
        if (!deep && k[u] < t.best[x])
          atomicMin(reinterpret_cast<unsigned long long*>(&t.best[x]),
                    static_cast<unsigned long long>(k[u]));
        if (!deep && k[u] < t.best[y])
          atomicMin(reinterpret_cast<unsigned long long*>(&t.best[y]),
                    static_cast<unsigned long long>(k[u]));
      }
      kept += static_cast<u32>(__popcll(b));
    }
  }
  l.c = kept;
  __syncthreads();
  u64 k[DENSE_MAX / UT], b[DENSE_MAX / UT];
#pragma unroll
  for (u32 j = 0; j < DENSE_MAX / UT; ++j) {
    const u32 i = j * UT + threadIdx.x;
    k[j] = i < ids ? t.best[i] : VAL_NONE;
    b[j] = 0;
    if (k[j] != VAL_NONE) b[j] = get(at(best, i));
  }
#pragma unroll
  for (u32 j = 0; j < DENSE_MAX / UT; ++j)
    if (k[j] < b[j]) lower(best, j * UT + threadIdx.x, k[j]);
  return deep;
}

// The edges that a wave kept as vertices, after shorten_chains.
__device__ __forceinline__ void convert_rest(const UnionArgs& a, const WaveLists& l, u32 ids) {
  for (u32 j = lane_id(); j < l.c; j += WAVE)
    for (u32* x : {a.s[0] + l.base + j, a.d[0] + l.base + j})
      if (*x & UNRESOLVED)
        *x = min(get(at(a.dense_id, get(at(a.parent, *x & ~UNRESOLVED)))), ids - 1);
}

// ------------------------------------------------------------ output
// A wave's 64 mark words: 2048 input positions.
constexpr u32 WINDOW = WAVE * 32;
struct Window {
  u16 pos[WINDOW];             // the marked positions
  u32 bits[WAVE], before[WAVE];  // the mark words, the marks before each
};
// Sources of a window's marked records, from the rows of its vertices: the
// gather of a third array would fetch nearly every line of it (an MST has one
// record in 16 or 32).  A solve of 2^24 vertices 6.95 -> 6.65 ms, geometric 4.75
// -> 4.55, of 10^6 745 -> 728 us.
// False, with nothing written, where many vertices without records lie between.
__device__ __forceinline__ bool window_sources(const UnionArgs& a, const Window& win, u64 base,
                                               u32 v0, u32 v1, u64 at) {
  if (v1 - v0 > 2 * WINDOW) return false;
  auto rank = [&](u64 p) {  // marks of the window before position p
    const u32 x = static_cast<u32>(p - base);
    return win.before[x / 32] + static_cast<u32>(__popc(win.bits[x / 32] & ((1u << (x & 31)) - 1)));
  };
  for (u32 w = v0; w <= v1; w += WAVE) {
    const u32 v = w + lane_id();
    u32 first = 0, last = 0;
    if (v <= v1) {
      const u64 sp = get(a.span + v);
      const u64 b = max(u64(static_cast<u32>(sp)), base);
      const u64 e = min(sp >> 32, base + WINDOW);
      if (b < e) {
        first = rank(b);
        last = rank(e - 1) + ((win.bits[(e - 1 - base) / 32] >> ((e - 1) & 31)) & 1u);
      }
    }
    const bool many = last - first > 16;  // a hub: the wave writes it together
    if (!many)
      for (u32 k = first; k < last; ++k)
        a.out_s[at + k] = v;
    for (u64 hubs = __ballot(many); hubs; hubs &= hubs - 1) {
      const int i = __ffsll(static_cast<unsigned long long>(hubs)) - 1;
      const u32 f = __shfl(first, i, WAVE), l = __shfl(last, i, WAVE), s = w + i;
      for (u32 k = f + lane_id(); k < l; k += WAVE) a.out_s[at + k] = s;
    }
  }
  return true;
}

// ------------------------------------------------------------ the solve
union Scratch {
  Stage stage[UW];
  OfferTable table;
  DenseRound dense;
  Window window[UW];
  Rows rows[UW];
};

// The kernel's arguments, loaded anew: held over all phases they fill the
// scalar registers, and what spills costs vector instructions in every loop.
__device__ __forceinline__ UnionArgs arguments() {
  typedef const UnionArgs __attribute__((address_space(4))) * Pointer;
  Pointer p = (Pointer)__builtin_amdgcn_kernarg_segment_ptr();
  asm volatile("" : "+s"(p));
  return *(const UnionArgs*)p;
}

// Sum over the waves before this one of what the workgroups put in their fourth
// found word, a barrier ago, and this workgroup's waves in s_waves.
__device__ __forceinline__ u64 waves_before(const UnionArgs& a, const u64* s_waves, u64& s_base) {
  if (wave_index() == 0) {
    u64 before = 0;
    for (u32 b = lane_id(); b < blockIdx.x; b += WAVE) before += get(a.found + b * 4 + 3);
#pragma unroll
    for (int o = WAVE / 2; o > 0; o >>= 1) before += __shfl_xor(before, o, WAVE);
    if (lane_id() == 0) s_base = before;
  }
  __syncthreads();
  u64 sum = s_base;
  for (u32 w = 0; w < wave_index(); ++w) sum += s_waves[w];
  return sum;
}

__global__ __launch_bounds__(UT) void union_solve_kernel(UnionArgs) {
  __shared__ Scratch s_x;
  __shared__ Found s_all;
  __shared__ u64 s_waves[UW], s_base;  // prefix sums over the waves
  __shared__ u32 s_giant, s_hub;
  UnionArgs a = arguments();
  if (!join_grid(a.joined)) return;
  Barrier bar{a.bar, 0, a.err};
  const u32 n = a.n;
  const int lane = lane_id();
  const u32 G = gridDim.x, gthread = blockIdx.x * UT + threadIdx.x, threads = G * UT;
  const u32 wave = blockIdx.x * UW + wave_index(), waves = G * UW;
  u64 sum;

  // init
  for (u64 v = gthread; v < n; v += threads) {
    put(a.parent + v, static_cast<u32>(v));
    put(a.best[0] + v, VAL_NONE);
    put(a.span + v, u64{0});
    if (a.parts) put(a.giants + v, u8{0});
  }
  for (u64 i = gthread; i < (a.m + 31) / 32; i += threads) put(a.marks + i, 0u);
  if (blockIdx.x == 0) pick_pivots(a);
  if (!sync_grid(bar, 0, sum)) return;

  // light pass
  a = arguments();
  const u64 units = (a.m + UNION_UNIT - 1) / UNION_UNIT;
  // a wave's range of the list buffers: as many edges as its chunks have
  // records (only the input's last chunk may be short)
  const u64 chunks = (units + a.chunk - 1) / a.chunk;
  const u64 q = chunks / waves, rem = chunks % waves;
  WaveLists l;
  l.base = (wave * q + min(wave, rem)) * a.chunk * UNION_UNIT;
  l.cap = (q + (wave < rem ? 1 : 0)) * a.chunk * UNION_UNIT;
  l.c = l.rest1 = l.rest2 = 0;
  Found mine{};
  light_pass(a, l, UnitWalk(a, wave, waves, units), s_x.stage[wave_index()], mine);
  if (threadIdx.x == 0) {
    u64* f = a.found + blockIdx.x * 4;
    put(f, mine.hash_fwd);
    put(f + 1, mine.hash_rev);
    put(f + 2, (u64(mine.bad) << 32) | mine.dup);
  }
  if (!sync_grid(bar, mine.fwd, sum)) return;
  if (wave_id() == 0) {
    u64 hf = 0, hr = 0, bd = 0;
    const u32 hub = get(a.ctl + UC_HUB);
    for (u32 b = lane; b < G; b += WAVE) {
      hf += get(a.found + b * 4);
      hr += get(a.found + b * 4 + 1);
      bd |= get(a.found + b * 4 + 2);
    }
#pragma unroll
    for (int o = WAVE / 2; o > 0; o >>= 1) {
      hf += __shfl_xor(hf, o, WAVE);
      hr += __shfl_xor(hr, o, WAVE);
      bd |= __shfl_xor(bd, o, WAVE);
    }
    if (lane == 0) s_hub = hub;
    if (lane == 0)
      s_all = Found{hf, hr, static_cast<u32>(sum), static_cast<u32>(bd >> 32), static_cast<u32>(bd)};
  }
  __syncthreads();
  const Found all = s_all;
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    *a.fwd_count = all.fwd;
    a.hsum[0] = all.hash_fwd;
    a.hsum[1] = all.hash_rev;
    if (all.bad) atomicOr(a.err, all.bad);
  }
  // the minima of a malformed input may hook a cycle: leave, the host reports
  if (all.bad || u64(all.fwd) * 2 != a.m || all.hash_fwd != all.hash_rev) return;

  // rounds of each class
  a = arguments();
  const bool copies = all.dup != 0;
  u32 round = 0, giant = NONE32;
  int cur = 0;
  u64 live = n;  // roots, where this is known
  for (u32 phase = 0; phase < a.classes + (a.has_heavy ? 1 : 0); ++phase) {
    a = arguments();
    const bool last = phase == a.classes;
    if (phase > 0) {
      // the minima are cleared for every root: one that took no part in the last
      // round holds an old one
      // cross_rows moves the lists' ranges to other waves: a line that one XCD's
      // L2 still holds dirty would be written back over what another wrote since
      if (last && wave_index() == 0) __builtin_amdgcn_fence(__ATOMIC_RELEASE, "agent");
      if (a.parts) {
        pick_giants(a, wave, waves, phase > 1);
        if (!sync_grid(bar, 0, sum)) return;
      } else {
        if (wave_index() == 0) s_giant = pick_giant(a);
        __syncthreads();
        giant = s_giant;
      }
      // last: the wave's records in rows outside it; else its vertices inside
      u64 count = 0;
      u32 roots = 0;
      for (u64 v0 = gthread; v0 < n; v0 += 4 * threads) {
        u32 x[4];
#pragma unroll
        for (u32 j = 0; j < 4; ++j)
          x[j] = static_cast<u32>(v0 + j * threads < n ? v0 + j * threads : v0);
        if (!find_roots<4>(a.parent, x, 0, 0, WALK_LIMIT)) atomicOr(a.err, ERR_SPIN);
#pragma unroll
        for (u32 j = 0; j < 4; ++j) {
          const u64 v = v0 + j * threads;  // consecutive over a wave, from a multiple of 64
          const bool in = v < n && (a.parts ? get(at(a.giants, x[j])) != 0 : x[j] == giant);
          const u64 b = __ballot(in);
          const bool root = v < n && x[j] == v;
          if (root && a.parts && in) {
            put(minima(a, cur) + v, u64{0});
            put(minima(a, cur ^ 1) + v, u64{0});
          } else if (root) {
            put(minima(a, cur) + v, VAL_NONE);
          }
          roots += static_cast<u32>(__popcll(__ballot(root)));
          if (lane == 0 && v < n) put(a.bits + v / 64, b);
          if (!last && lane == 0) count += static_cast<u64>(__popcll(b));
          if (last && v < n && !in) {
            const u64 sp = get(a.span + v), len = (sp >> 32) - static_cast<u32>(sp);
            count += len > ROW_LONG ? a.m : len;
          }
        }
      }
#pragma unroll
      for (int o = WAVE / 2; o > 0; o >>= 1) count += __shfl_xor(count, o, WAVE);
      if (lane == 0) s_waves[wave_index()] = count;
      count = min(block_total(count), a.m);
      const u64 block_roots = block_total(roots);
      if (threadIdx.x == 0) {
        put(a.found + blockIdx.x * 4 + 2, block_roots);
        put(a.found + blockIdx.x * 4 + 3, count);
      }
      if (!sync_grid(bar, count, sum)) return;
      // one wave acquires for the CU: the L1 is its workgroup's alone
      if (wave_index() == 0) __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
      __syncthreads();
      if (wave == 0) {  // (for the log)
        live = 0;
        for (u32 b = lane; b < G; b += WAVE) live += get(a.found + b * 4 + 2);
#pragma unroll
        for (int o = WAVE / 2; o > 0; o >>= 1) live += __shfl_xor(live, o, WAVE);
      }
      a = arguments();
      if (!last) {
        cross_list(a, l, phase, minima(a, cur), giant, 6 * sum > 5 * u64(n));
      } else if (copies || sum * ROWS_SHARE > a.m) {
        cross_input(a, l, UnitWalk(a, wave, waves, (a.m + UNION_UNIT - 1) / UNION_UNIT), minima(a, cur), giant);
      } else {
        // a wave's list holds as many edges as its rows have records
        l.base = waves_before(a, s_waves, s_base);
        cross_rows(a, l, wave, waves, minima(a, cur), giant, s_x.rows[wave_index()]);
      }
    }
    a = arguments();
    u64 edges;
    if (!sync_grid(bar, block_total(l.c), edges)) return;
    // dense ids of the first class's rounds (0: none yet), and whether they are the vertices
    u32 ids = phase == 0 && n <= DENSE_MAX ? n : 0;
    const bool identity = ids != 0;
    bool resolved = false;  // the last relabel resolved them in LDS
    u64 known = n;  // bound of the roots
    // the round enters the dense ids; its lists hold vertices still
    bool enter = false, convert = false;
    while (edges) {
      if (__builtin_expect(!(edges >> DEEP_SHIFT), 1)) {
        if (blockIdx.x == 0 && threadIdx.x == 0 && round < UNION_LOG) a.log[round] = edges | (live << 32);
        const bool first = phase == 0 && round == 0;
        const bool note = phase == 0 && !ids && known <= 8 * DENSE_MAX;
        const u32 lw = hook(a, l, cur, first, first && copies, giant,
                            ids && !identity ? a.dense_parent : a.parent, note);
        const u64 block_live = block_total(lw);
        if (note) {
          if (lane == 0) s_waves[wave_index()] = lw;
          if (threadIdx.x == 0) put(a.found + blockIdx.x * 4 + 3, block_live);
        }
        if (!sync_grid(bar, block_live, live)) return;
        known = live;
        enter = note && live <= DENSE_MAX && edges >= DENSE_EDGES_MIN && edges >= DENSE_EDGES * live;
        convert = enter;
        if (enter) {
          // the survivors' ids: their order over the waves
          u64 id = waves_before(a, s_waves, s_base);
          for (u32 i = lane; i < lw; i += WAVE) {
            const u32 v = a.s[1][l.base + i], x = static_cast<u32>(id) + i;
            put(at(a.dense_id, v), x);
            put(a.dense_vertex + x, v);
            put(a.dense_parent + x, x);
            put(minima(a, cur ^ 1) + x, VAL_NONE);
          }
          ids = static_cast<u32>(live);
          u64 none;
          if (!sync_grid(bar, 0, none)) return;
        }
        cur ^= 1;
        ++round;
      } else {  // a wave met a deep chain: the same round's relabel again
        if (!shorten_chains(a, bar, gthread, threads)) return;
        if (convert) convert_rest(a, l, ids);
        convert = false;
        if (blockIdx.x == 0 && threadIdx.x == 0 && round <= UNION_LOG) a.log[round - 1] |= UNION_CHAINS;
      }
      a = arguments();
      bool deep;
      if (ids)
        deep = relabel_dense(a, l, cur, ids, convert, identity ? a.parent : a.dense_parent, s_x.dense,
                             wave);
      else deep = relabel(a, l, cur, live, live <= TABLE_LIVE || s_hub, s_x.table, giant, wave);
      resolved = ids && !enter;
      if (!sync_grid(bar, block_total(l.c | (deep ? u64{1} << DEEP_SHIFT : 0)), edges)) return;
      if (round >= UNION_ROUNDS_MAX) {
        // every round at least halves the components that have edges
        if (gthread == 0) atomicOr(a.err, ERR_SPIN);
        return;
      }
    }
    if (blockIdx.x == 0 && threadIdx.x == 0) a.log[UNION_LOG + phase] = round;
    if (resolved) {
      for (u64 i = gthread; i < ids; i += threads) {
        const u32 r = s_x.dense.root[i];
        if (r != i) {
          if (identity) put(a.parent + i, r);
          else put(at(a.parent, get(a.dense_vertex + i)), get(a.dense_vertex + r));
        }
      }
      // (the identity's walks end at the same roots before and after)
      if (!identity && !sync_grid(bar, 0, sum)) return;
    }
  }

  a = arguments();
  // output: workgroups own equal contiguous parts of the mark words, their
  // waves equal parts of those
  const u64 words = (a.m + 31) / 32;
  const u64 rows = (words + WAVE - 1) / WAVE;  // rows of 64 words
  const u64 r0 = (wave * rows) / waves, r1 = ((wave + 1) * rows) / waves;
  u32 cnt = 0;
  for (u64 r = r0; r < r1; ++r) {
    const u64 w = r * WAVE + lane;
    cnt += w < words ? static_cast<u32>(__popc(get(a.marks + w))) : 0u;
  }
#pragma unroll
  for (int o = WAVE / 2; o > 0; o >>= 1) cnt += __shfl_xor(cnt, o, WAVE);
  if (lane == 0) s_waves[wave_id()] = cnt;
  const u64 block_count = block_total(cnt);
  if (threadIdx.x == 0) put(a.found + blockIdx.x * 4 + 3, block_count);
  u64 total;
  if (!sync_grid(bar, block_count, total)) return;
  if (total > a.out_cap) {  // the host refuses the call: the caller's arrays stay as they are
    if (gthread == 0) {
      *a.count = static_cast<u32>(total);
      a.ctl[UC_DONE] = 1;
    }
    return;
  }
  u64 at = waves_before(a, s_waves, s_base);
  Window& win = s_x.window[wave_index()];
  u64 weight = 0;
  for (u64 r = r0; r < r1; ++r) {
    const u64 w = r * WAVE + lane, base = r * WINDOW;
    const u32 bits = w < words ? get(a.marks + w) : 0u;
    const u32 v0 = a.src[base], v1 = a.src[min(base + WINDOW, a.m) - 1];
    const u32 c = static_cast<u32>(__popc(bits));
    const u32 incl = wave_inclusive_sum(c);
    const u32 row = __shfl(incl, WAVE - 1, WAVE);
    u32 p = incl - c;
    win.bits[lane] = bits;
    win.before[lane] = p;
    for (u32 b = bits; b; b &= b - 1) win.pos[p++] = static_cast<u16>(lane * 32 + __ffs(b) - 1);
    __builtin_amdgcn_wave_barrier();
    const bool gather = row && !window_sources(a, win, base, v0, v1, at);
    for (u32 j = lane; j < row; j += WAVE) {
      const u64 e = base + win.pos[j], o = at + j;
      const u32 wt = a.wt[e];
      weight += wt;
      if (gather) a.out_s[o] = a.src[e];
      a.out_d[o] = a.dst[e];
      a.out_w[o] = wt;
    }
    __builtin_amdgcn_wave_barrier();
    at += row;
  }
#pragma unroll
  for (int o = WAVE / 2; o > 0; o >>= 1) weight += __shfl_xor(weight, o, WAVE);
  const u64 block_weight = block_total(weight);
  if (threadIdx.x == 0) {
    a.found[blockIdx.x * 4] = block_weight;
    if (blockIdx.x == 0) {
      *a.count = static_cast<u32>(total);
      a.ctl[UC_DONE] = 1;
    }
  }
}

// Sums the workgroups' weights and counts the smaller endpoints with more
// than MST_GROUP_SMALL edges in the output (the edge MST_GROUP_SMALL past the
// first of its group counts the group).  The last workgroup to end publishes
// the counters and the log, as publish_words does.  What it reads of other
// workgroups are agent-scope atomics, awaited before the workgroup counts as
// ended: a fence per workgroup (a write-back of its L2) took 30 us of 29 MB
// read by 61 workgroups, 66 us with 244.
__global__ __launch_bounds__(UT) void union_finish_kernel(UnionArgs a, u32 blocks, u64* total,
                                                          u32* groups, u32* ended, Publication p) {
  __shared__ u32 s_last;
  const u64 count = a.ctl[UC_DONE] && *a.count <= a.out_cap ? *a.count : 0;
  u32 c = 0;
#pragma unroll 2
  for (u64 i = u64(blockIdx.x) * UT + threadIdx.x + MST_GROUP_SMALL; i < count;
       i += u64(gridDim.x) * UT) {
    const u32 s = a.out_s[i], first = a.out_s[i - MST_GROUP_SMALL];
    const u32 before = a.out_s[max(i, MST_GROUP_SMALL + u64{1}) - MST_GROUP_SMALL - 1];
    c += s == first && (i == MST_GROUP_SMALL || before != s) ? 1u : 0u;
  }
  if (c) (void)__hip_atomic_fetch_add(groups, c, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  if (blockIdx.x == 0 && wave_id() == 0) {
    u64 w = 0;
    for (u32 b = lane_id(); b < blocks; b += WAVE) w += a.found[b * 4];
#pragma unroll
    for (int o = WAVE / 2; o > 0; o >>= 1) w += __shfl_xor(w, o, WAVE);
    if (lane_id() == 0) put(total, w);
  }
  if (!p.host) return;
  __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0)
  __syncthreads();
  if (threadIdx.x == 0)
    s_last = __hip_atomic_fetch_add(ended, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) + 1 ==
                     gridDim.x
                 ? 1u
                 : 0u;
  __syncthreads();
  if (!s_last) return;
  for (u32 i = threadIdx.x; i < 64; i += UT) p.host[i] = get(a.ctr + i);
  const u32* lg = reinterpret_cast<const u32*>(a.log);
  for (u32 i = threadIdx.x; i < 2 * UNION_LOG_TOTAL; i += UT) p.host[p.extra_at + i] = get(lg + i);
  __threadfence_system();
  __syncthreads();
  if (threadIdx.x == 0)
    __hip_atomic_store(p.host + p.seq_at, p.seq, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
}

// ------------------------------------------------------------ small inputs
// One workgroup, one launch: the records stay in registers (record k * UT + t
// with thread t), the parents, minima and marks in LDS, so a round is four
// workgroup barriers and no memory round trip.  The general solve's phases cost
// 3 us each for those: 256 vertices, 4.4 10^3 records take 84 us a call with it
// (three launches) and 46 with this one (one launch, no counters to clear).
// Every edge takes part from the first round on: a second class would cost more
// rounds.  The limit is where the records fill the registers.
constexpr int SMALL_SLOTS = static_cast<int>(UNION_SMALL_RECORDS) / UT;
constexpr u32 SMALL_WORDS = static_cast<u32>(UNION_SMALL_RECORDS / 32);

__global__ __launch_bounds__(UT) void union_small_kernel(UnionArgs a, u64* total, u32* groups,
                                                         Publication p) {
  __shared__ u32 s_parent[UNION_SMALL_VERTICES];
  __shared__ u64 s_best[UNION_SMALL_VERTICES];
  __shared__ u32 s_marks[SMALL_WORDS], s_before[SMALL_WORDS];
  __shared__ u64 s_fwd_hash, s_rev_hash, s_weight;
  __shared__ u32 s_fwd, s_bad, s_live[3], s_open, s_count, s_groups;
  __shared__ u64 s_log[UNION_LOG];
  __shared__ u32 s_scan[UW];
  const u32 t = threadIdx.x, lane = lane_id(), n = a.n, m = static_cast<u32>(a.m);
  u32 s[SMALL_SLOTS], d[SMALL_SLOTS], w[SMALL_SLOTS];
#pragma unroll
  for (int k = 0; k < SMALL_SLOTS; ++k) {
    s[k] = d[k] = w[k] = 0;
    if (k * UT + t < m) {
      s[k] = a.src[k * UT + t];
      d[k] = a.dst[k * UT + t];
      w[k] = a.wt[k * UT + t];
    }
  }
  if (t == 0) {
    s_fwd_hash = s_rev_hash = s_weight = 0;
    s_fwd = s_bad = s_count = s_groups = 0;
    s_live[0] = s_live[1] = s_live[2] = 0;
  }
  for (u32 v = t; v < n; v += UT) {
    s_parent[v] = v;
    s_best[v] = VAL_NONE;
  }
  for (u32 i = t; i < SMALL_WORDS; i += UT) s_marks[i] = 0;
  __syncthreads();

  // validation
  u64 hf = 0, hr = 0;
  u32 bad = 0, fwd = 0, alive = 0;  // alive, bit k: record k is a forward one and joins two roots
#pragma unroll
  for (int k = 0; k < SMALL_SLOTS; ++k) {
    if (k * UT >= m) continue;
    const u32 i = k * UT + t;
    u32 ps = dpp<DPP_WAVE_SHR1>(0, s[k]), pd = dpp<DPP_WAVE_SHR1>(0, d[k]);
    if (i < m) {
      if (lane == 0 && i > 0) {
        ps = a.src[i - 1];
        pd = a.dst[i - 1];
      }
      const u32 lo = min(s[k], d[k]), hi = max(s[k], d[k]);
      if (lo == hi || hi >= n) bad |= ERR_INVALID;
      if (((u64(ps) << 32) | pd) > ((u64(s[k]) << 32) | d[k])) bad |= ERR_UNSORTED;
      const u64 h = sym_hash(lo, hi, w[k]);
      if (s[k] < d[k]) {
        hf += h;
        ++fwd;
        alive |= 1u << k;
      } else {
        hr += h;
      }
    }
  }
#pragma unroll
  for (int o = WAVE / 2; o > 0; o >>= 1) {
    hf += __shfl_xor(hf, o, WAVE);
    hr += __shfl_xor(hr, o, WAVE);
    fwd += __shfl_xor(fwd, o, WAVE);
    bad |= __shfl_xor(bad, o, WAVE);
  }
  if (lane == 0) {
    atomicAdd(reinterpret_cast<unsigned long long*>(&s_fwd_hash), static_cast<unsigned long long>(hf));
    atomicAdd(reinterpret_cast<unsigned long long*>(&s_rev_hash), static_cast<unsigned long long>(hr));
    atomicAdd(&s_fwd, fwd);
    atomicOr(&s_bad, bad);
  }
  __syncthreads();
  const bool good = !s_bad && 2 * s_fwd == m && s_fwd_hash == s_rev_hash;

  // rounds: the roots an edge joins, x | y << 16
  u32 ends[SMALL_SLOTS];
#pragma unroll
  for (int k = 0; k < SMALL_SLOTS; ++k) ends[k] = s[k] | (d[k] << 16);
  u32 round = 0, live = good ? s_fwd : 0, roots = n;
  while (live && round < UNION_ROUNDS_MAX) {
    if (t == 0 && round < UNION_LOG) s_log[round] = live | (u64(roots) << 32);
#pragma unroll
    for (int k = 0; k < SMALL_SLOTS; ++k) {
      if (!((alive >> k) & 1)) continue;
      const u64 key = (u64(w[k]) << 32) | (k * UT + t);
      const u32 x = ends[k] & 0xFFFF, y = ends[k] >> 16;
      if (key < s_best[x])
        atomicMin(reinterpret_cast<unsigned long long*>(&s_best[x]), static_cast<unsigned long long>(key));
      if (key < s_best[y])
        atomicMin(reinterpret_cast<unsigned long long*>(&s_best[y]), static_cast<unsigned long long>(key));
    }
    if (t == 0) s_live[(round + 1) % 3] = s_open = 0;
    __syncthreads();
    u32 mine = 0;  // edges that stay | roots that live on << 16
#pragma unroll
    for (int k = 0; k < SMALL_SLOTS; ++k) {
      if (!((alive >> k) & 1)) continue;
      const u32 i = k * UT + t, x = ends[k] & 0xFFFF, y = ends[k] >> 16;
      const u64 key = (u64(w[k]) << 32) | i;
      const bool mx = s_best[x] == key, my = s_best[y] == key;
      if (!mx && !my) continue;
      u32 child = mx ? x : y, other = mx ? y : x;
      if (mx && my) {  // the lower end stays root
        child = max(x, y);
        other = min(x, y);
        mine += 1u << 16;
      }
      s_parent[child] = other;
      atomicOr(&s_marks[i / 32], 1u << (i & 31));
    }
    __syncthreads();
    roots_in_lds(s_parent, n, &s_open, [&](u32 v) { s_best[v] = VAL_NONE; });
#pragma unroll
    for (int k = 0; k < SMALL_SLOTS; ++k) {
      if (!((alive >> k) & 1)) continue;
      const u32 x = s_parent[ends[k] & 0xFFFF], y = s_parent[ends[k] >> 16];
      ends[k] = x | (y << 16);
      if (x == y) alive &= ~(1u << k);
      else ++mine;
    }
#pragma unroll
    for (int o = WAVE / 2; o > 0; o >>= 1) mine += __shfl_xor(mine, o, WAVE);
    if (lane == 0 && mine) atomicAdd(&s_live[round % 3], mine);
    ++round;
    __syncthreads();
    live = s_live[(round - 1) % 3] & 0xFFFF;
    roots = s_live[(round - 1) % 3] >> 16;
  }
  // output: the marked records in order; s_best counts the edges of a smaller endpoint
  u32 *count = reinterpret_cast<u32*>(s_best);
  for (u32 v = t; v < n; v += UT) count[v] = 0;
  const u32 c = t < SMALL_WORDS ? static_cast<u32>(__popc(s_marks[t])) : 0u;
  const u32 incl = wave_inclusive_sum(c);
  if (lane == WAVE - 1) s_scan[wave_index()] = incl;
  __syncthreads();
  u32 before = incl - c;
  for (u32 i = 0; i < wave_index(); ++i) before += s_scan[i];
  if (t < SMALL_WORDS) s_before[t] = before;
  if (t == SMALL_WORDS - 1) s_count = before + c;
  __syncthreads();
  const bool room = s_count <= a.out_cap;  // else the host refuses the call
  u64 weight = 0;
#pragma unroll
  for (int k = 0; k < SMALL_SLOTS; ++k) {
    const u32 i = k * UT + t;
    if (i >= m || !((s_marks[i / 32] >> (i & 31)) & 1)) continue;
    const u32 o = s_before[i / 32] + static_cast<u32>(__popc(s_marks[i / 32] & ((1u << (i & 31)) - 1)));
    weight += w[k];
    if (room) {  // past the L2: the caller may go on before this launch has ended
      put(a.out_s + o, s[k]);
      put(a.out_d + o, d[k]);
      put(a.out_w + o, w[k]);
    }
    if (atomicAdd(&count[s[k]], 1u) == MST_GROUP_SMALL) atomicAdd(&s_groups, 1u);
  }
#pragma unroll
  for (int o = WAVE / 2; o > 0; o >>= 1) weight += __shfl_xor(weight, o, WAVE);
  if (lane == 0 && weight)
    atomicAdd(reinterpret_cast<unsigned long long*>(&s_weight), static_cast<unsigned long long>(weight));
  __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0): the output
  __syncthreads();

  // the counter words and the log, to the device's or the host's
  u32* const ctr = p.host ? p.host : a.ctr;
  u32* const lg = p.host ? p.host + p.extra_at : reinterpret_cast<u32*>(a.log);
  auto word = [&](const void* at) { return static_cast<u32>(static_cast<const u32*>(at) - a.ctr); };
  if (t < 64) {
    u32 x = 0;
    // (every round at least halves the components that have edges)
    if (t == word(a.err)) x = s_bad | (live ? u32(ERR_SPIN) : 0u);
    if (t == word(a.fwd_count)) x = s_fwd;
    if (t == word(a.hsum)) x = static_cast<u32>(s_fwd_hash);
    if (t == word(a.hsum) + 1) x = static_cast<u32>(s_fwd_hash >> 32);
    if (t == word(a.hsum) + 2) x = static_cast<u32>(s_rev_hash);
    if (t == word(a.hsum) + 3) x = static_cast<u32>(s_rev_hash >> 32);
    if (t == word(total)) x = static_cast<u32>(s_weight);
    if (t == word(total) + 1) x = static_cast<u32>(s_weight >> 32);
    if (t == word(groups)) x = s_groups;
    if (t == word(a.count)) x = s_count;
    if (t == word(a.ctl) + UC_DONE) x = good && !live ? 1u : 0u;
    if (t - word(a.ctl) - UC_PIVOT < UNION_CLASSES) x = NONE32;
    ctr[t] = x;
  }
  for (u32 i = t; i < 2 * UNION_LOG_TOTAL; i += UT) {
    const u32 r = i / 2;
    const u64 x = r < min(round, UNION_LOG) ? s_log[r] : r == UNION_LOG ? u64{round} : 0;
    lg[i] = static_cast<u32>(i & 1 ? x >> 32 : x);
  }
  if (!p.host) return;
  __threadfence_system();
  __syncthreads();
  if (t == 0)
    __hip_atomic_store(p.host + p.seq_at, p.seq, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
}

}  // namespace

void union_solve_small(hipStream_t st, const UnionArgs& a, u64* total, u32* groups,
                       const Publication& p) {
  if (a.m > UNION_SMALL_RECORDS || a.n > UNION_SMALL_VERTICES)
    throw Error(KMST_EINVAL, "small direct solve: size");
  KTScope t(st, K_PERSIST, 24.0 * a.m + 24.0 * a.n);
  union_small_kernel<<<1, UT, 0, st>>>(a, total, groups, p);
  KMST_HIP(hipGetLastError());
}

u64 union_mark_words(u64 m) { return (m + 31) / 32; }
u32 union_samples(u64 m) {
  return static_cast<u32>(std::min<u64>(m >= (u64{1} << 22) ? PIVOT_SAMPLES_MAX : UT, m));
}

u32 union_blocks(u64 m, u32 cus) {
  // three units per wave at least: fewer workgroups make the barriers and the
  // offers of few roots cheaper (2^17 vertices, 2.1 10^6 records: 350 us with 171
  // workgroups, 359 with 256, 369 with 64; 2^14, 4.9 10^5: 205 with 41, 203 with
  // 61, 232 with 16)
  const u64 want = (m + 3 * UW * UNION_UNIT - 1) / (3 * UW * UNION_UNIT);
  return static_cast<u32>(std::max<u64>(1, std::min<u64>({want, cus, UNION_BLOCKS_MAX})));
}

u32 union_chunk(u64 m, u32 blocks) {
  // long chunks spare atomics at their ends, several chunks per wave even out
  // how many edges the waves list: at most four chunks up to 64 units per wave
  const u64 waves = u64(blocks) * UW, units = (m + UNION_UNIT - 1) / UNION_UNIT;
  return static_cast<u32>(
      std::max<u64>(1, std::min<u64>((units + 4 * waves - 1) / (4 * waves), UNION_CHUNK_MAX)));
}

void union_solve(hipStream_t st, const UnionArgs& a, u32 blocks, u64* total, u32* groups,
                 u32* ended, const Publication& p) {
  if (blocks == 0 || blocks > UNION_BLOCKS_MAX) throw Error(KMST_EINVAL, "direct solve: workgroups");
  {
    KTScope t(st, K_PERSIST, 24.0 * a.m + 24.0 * a.n);
    union_solve_kernel<<<blocks, UT, 0, st>>>(a);
    KMST_HIP(hipGetLastError());
  }
  KTScope t(st, K_OTHER, 8.0 * a.n);
  const u32 grid = static_cast<u32>(std::max<u64>(1, std::min<u64>((a.n + 4 * UT - 1) / (4 * UT), 256)));
  union_finish_kernel<<<grid, UT, 0, st>>>(a, blocks, total, groups, ended, p);
  KMST_HIP(hipGetLastError());
}

}  // namespace kmst
