// Map update: VoxelMap::update / build (voxel_map.cpp:200-256) with
// VoxelGrid::pushPoint / updatePlane / merge (voxel_map.cpp:42-186), executed
// for a batch of independent sessions as a pipeline of data-parallel stages
// plus, for the scans that need them, the evictions' decisions and the merge
// replay (one workgroup per session each).
//
// Points of all sessions in a batch share one global index space, session
// after session (g = off[s] + i); times inside a session are its point
// indices i, which is the order the reference loops in.
//
//   K1 ins_keys      per point: fp32 insertion transform (PCL order), key,
//                    hash find-or-insert in the session's table
//   K2 sort          per session, stable radix sort by hash slot: each key's
//                    points become a contiguous segment in point order
//   K3/K4 segments   segment heads, the existing voxel of each segment, new
//                    keys flagged at their first point
//   K5 create        creation events in point order; where the LRU can
//                    overflow, one workgroup per session decides all creations
//                    and evictions against the LRU queue at once
//   K6 replay        each voxel's points through the pushPoint state machine;
//                    the voxels whose walk reaches a refit (known from counts)
//                    take the FP64 moment path (a wave or a lane each), the
//                    others a light one that queues their points
//   K7/K8 merge      see vmp_merge.hpp
//   K9 finalize      dirty bits, LRU queue append, hash tombstones, free list
// Every ordering decision (LRU order, victims, group ids, merge order) is
// therefore the reference's point order.
#pragma once
#include "vmp_common.hpp"
#include "vmp_observe.hpp"

namespace vmp {

constexpr int kMapThreads = 256;
constexpr int32_t kNever = 0x7fffffff;

struct MapCounters {
  int64_t size;            // live voxels
  uint64_t group_counter;  // VoxelGrid::count
  int64_t point_base;      // global point index of this scan's point 0 (LRU stamps)
  int64_t ring_head, ring_tail;
  int32_t free_top, bump;
  int32_t used_entries;    // non-empty hash slots, tombstones included
  int32_t pad0;
  int32_t tag;             // scan tag
  int32_t error;           // bit 1 hash probe overflow, 2 range, 4 capacity, 8 pool, 16 replay queue,
                           // 32 replay class (cannot happen)
  // per-scan outputs
  int32_t nseg, ncreate_ev, ncre, nevict, ncand;
  int32_t refits, merge_calls, merge_evals, merges, dropped;
  int32_t fast;            // 1: this scan's creations took the parallel (no-eviction) path
  int32_t pad1;
  int32_t merge_windows;   // windows of the merge replay
  int32_t merge_requeued;  // window entries sent back for re-evaluation
  int32_t merge_max_acting;  // most acting entries in one window of the merge replay
  int32_t pad_ctr;
};

// one session's map (device pointers)
struct MapDev {
  HashEntry* table;
  uint32_t hmask;
  int32_t pool;
  VoxHot* hot;
  VoxState* vs;
  double* plane;      // [pool][kPlaneD]
  double* mom;        // [pool][kMomD]
  float* pend;        // [pool][pend_cap][kPendF] points added since the moments' last update
  int32_t pend_cap;   // update_size_thresh - 1
  int32_t* freelist;  // [pool]
  int32_t* ring_vid;  // [qcap]
  uint64_t* ring_stamp;
  int64_t qcap;
  MapCounters* ctr;
  int32_t capacity;
  int32_t max_pt, upd_pt;
  int32_t hbits;      // log2 of the table size
  double plane_thresh, merge_a, merge_d, vs64;
};

// one session of a batch
struct SessInfo {
  const float* x;
  const float* y;
  const float* z;
  const UpdParams* prm;
  int32_t n, off;     // points, global offset of point 0
  int32_t is_build;
  int32_t seg_lo, seg_hi;  // its segments in the batch segment list
  int32_t cre_lo, cre_hi;  // its creation events in the batch creation list
  int32_t spl_lo, spl_hi;  // its acting merge candidates in spl
  int32_t ftop0, bump0;    // free-list top and bump pointer before its fast creations
};

// batch workspace, all arrays sized for the batch's total points
struct BatchBufs {
  int32_t ntot;
  int32_t nsess;
  int32_t hbits;       // bits of the largest hash-slot index in the batch
  int32_t cand_sshift; // position of the session bits in a batch candidate key (25 + time bits)
  uint64_t* skey_in;   // (session << hbits) | hash slot, per point
  int32_t* sval_in;    // global point index
  uint64_t* skey_out;
  int32_t* sval_out;
  int32_t* flags;      // scratch flag / value array
  int32_t* sel;        // compaction output (ascending global indices)
  int32_t* cnt;        // counts: [0] segments, [1] creation events, [2] LRU appends,
                       // [5] refitting voxels, [6] the long ones of these
  int32_t* seg_start;  // segment -> first sorted position
  int32_t* seg_end;
  int32_t* seg_sess;
  int32_t* seg_vid;
  int32_t* seg_entry;
  int32_t* cre_t;      // creation events: local point index, segment
  int32_t* cre_seg;
  int4* co;            // resolved creations in order, per session at its offset:
                       // (vid, segment, point time, evicted incarnation or -1);
                       // the r-th takes group id group_counter - ncre + r
  int32_t* ev_vid;     // evicted voxels in order, per session at its offset
  uint64_t* cand_in;   // merge candidates, see cand_key(), at session offset + point time (~0 none)
  uint64_t* cand_out;  // keys of the acting ones, in order
  int32_t* cand_nbr;   // per candidate record: 6 eligible neighbour ids at its time
  int32_t* spl;        // records (cand_nbr) of the candidates that act on the pre-replay state, in order
  int32_t* seg_ct;     // per segment: its candidate times (up to 7, ascending)
  int32_t* seg_nct;
  int2* seg_nbr;       // per segment: the six neighbour voxels, see nbr_eligible()
  int4* hlist;         // refitting voxels as (vid, start, length, session), see k_create_init
  uint32_t* seg_cls;   // per segment: how its voxel replays (replay_class)
  int32_t* seg_old;    // per segment: its voxel before this scan's creations (-1: none)
  // per acting candidate (its index in spl, the first pre_cap of them): for
  // each record r (its six eligible neighbours, then itself) and each
  // neighbour j of r (j = 6: r itself), the voxel X there at the candidate's
  // time, X's segment in this scan (-1: none or evicted) and X's first
  // merge() call after that time; none of these depends on merges
  int32_t* pre_x;
  int32_t* pre_seg;
  int32_t* pre_tn;
  int32_t pre_cap;
  int32_t pad1;
  // live LRU ring entries from the head of each evicting session: (vid,
  // first touch in this scan or kNever, segment, ring position - head).
  // lv holds them per 64-entry ring chunk (chunk k of a session at
  // 2 * off + 64 k, two entries per point; lv_cnt: its count, at
  // lv_cnt_base()), lv2 all of them in ring order at 2 * off
  int4* lv;
  int4* lv2;
  int32_t* lv_cnt;
  int32_t* prim;       // work entries of the compaction / radix sort (prim_ws_entries)
  // per point in key-sorted order: its insertion point relative to its
  // voxel's centre (fp32, as the replays fold it in), its index in the scan
  // and its fp32 world covariance, (q.x, q.y, q.z, index bits, C0..C5, -, -),
  // formed once by k_seg_info
  float4* qc;
};
__host__ __device__ inline int64_t lv_cnt_base(int off, int s) { return (int64_t(2) * off >> 6) + s; }

// sessions of one batch: the merge-candidate key holds a session in 15 bits
constexpr int kMaxBatchSessions = 1 << 15;

// merge-candidate key: session (15 bits) | point time (24 bits) | voxel (25 bits)
__host__ __device__ inline uint64_t cand_key(int s, int t, int32_t vid) {
  return (uint64_t(uint32_t(s)) << 49) | (uint64_t(uint32_t(t)) << 25) | uint64_t(uint32_t(vid));
}
__host__ __device__ inline int cand_t(uint64_t k) { return int((k >> 25) & 0xFFFFFFull); }
__host__ __device__ inline int32_t cand_vid(uint64_t k) { return int32_t(k & 0x1FFFFFFull); }
// In the batch's candidate list the session sits right above the point time
// (at bit cand_sshift, 25 + the bits of the largest scan), so the sort reads
// no constant bits; the local part (time, voxel) is cand_key(0, t, vid).
__host__ __device__ inline uint64_t cand_key_batch(int s, int t, int32_t vid, int sshift) {
  return (uint64_t(uint32_t(s)) << sshift) | (uint64_t(uint32_t(t)) << 25) | uint64_t(uint32_t(vid));
}
__host__ __device__ inline uint64_t cand_local(uint64_t k, int sshift) { return k & ((uint64_t(1) << sshift) - 1); }

__device__ inline int sess_of(const SessInfo* si, int nsess, int g) {
  int lo = 0, hi = nsess - 1;
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (si[mid].off <= g) lo = mid;
    else hi = mid - 1;
  }
  return lo;
}

// ------------------------------------------------------------ helpers -----
// Grid-stride loop whose trip count is the same for every lane of a block,
// so wave-level operations inside see the whole wave; `valid` marks the
// lanes with an item.
#define VMP_UNIFORM_LOOP(i, valid, n)                                                            \
  for (int i##_0 = blockIdx.x * blockDim.x; i##_0 < (n); i##_0 += gridDim.x * blockDim.x)         \
    for (int i = i##_0 + int(threadIdx.x), valid = (i < (n)), i##_once = 1; i##_once; i##_once = 0)

// Fetch-add on counters, aggregated over the wave: the lanes that add to the
// same counter do so with one atomic, and each lane gets the counter's value
// before its own contribution (lanes in lane order).  Every lane of the wave
// calls it; a lane with v = 0 contributes nothing.
__device__ inline int wave_fetch_add(int* p, int v) {
  const int lane = threadIdx.x & 63;
  uint64_t pending = __ballot(v != 0);
  const uint64_t pv = reinterpret_cast<uint64_t>(p);
  int out = 0;
  while (pending) {
    const int leader = __ffsll((unsigned long long)pending) - 1;
    const uint32_t lo = uint32_t(__shfl(int(uint32_t(pv)), leader, 64));
    const uint32_t hi = uint32_t(__shfl(int(uint32_t(pv >> 32)), leader, 64));
    const uint64_t pl = uint64_t(lo) | (uint64_t(hi) << 32);
    const bool in = ((pending >> lane) & 1ull) && pv == pl;
    const uint64_t grp = __ballot(in);
    const int x = in ? v : 0;
    int incl = x;
    for (int o = 1; o < 64; o <<= 1) {
      const int u = __shfl_up(incl, o, 64);
      if (lane >= o) incl += u;
    }
    const int total = __shfl(incl, 63, 64);
    int base = 0;
    if (lane == leader) base = atomicAdd(reinterpret_cast<int*>(pl), total);
    base = __shfl(base, leader, 64);
    if (in) out = base + incl - x;
    pending &= ~grp;
  }
  return out;
}

__device__ inline uint64_t bits_below(int l) { return l == 0 ? 0ull : (~0ull >> (64 - l)); }

// LDS written by some lanes of a wave and read by others of the same wave
__device__ inline void wave_lds_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// *inserted = 1 when this call claimed the empty slot (the caller counts
// used_entries); with inserted == nullptr the count is added here
__device__ inline int32_t hash_find_or_insert(HashEntry* table, uint32_t mask, uint64_t key, MapCounters* ctr,
                                              int* inserted = nullptr) {
  const HashSeq seq = hash_seq(key);
  uint32_t h = hash_home(seq, mask);
  // The probes up to the first empty slot on loads that the caches may serve:
  // no kernel that inserts removes or replaces a key, so only a slot seen
  // empty can hold something else by now, and is looked at again below.
  uint32_t probe = 0;
  while (probe <= mask) {
    const unsigned long long k = __hip_atomic_load(reinterpret_cast<unsigned long long*>(&table[h].key),
                                                   __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    if (k == key) return int32_t(h);
    if (k == kKeyEmpty) break;
    h = hash_probe(seq, ++probe, mask);
  }
  while (probe <= mask) {
    unsigned long long* kp = reinterpret_cast<unsigned long long*>(&table[h].key);
    unsigned long long k = __hip_atomic_load(kp, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (k == key) return int32_t(h);
    if (k == kKeyEmpty) {
      unsigned long long old = atomicCAS(kp, (unsigned long long)kKeyEmpty, (unsigned long long)key);
      if (old == kKeyEmpty) {
        if (inserted) *inserted = 1;
        else atomicAdd(&ctr->used_entries, 1);
        return int32_t(h);
      }
      if (old == key) return int32_t(h);
    }
    h = hash_probe(seq, ++probe, mask);
  }
  atomicOr(&ctr->error, 1);
  return -1;
}

__device__ inline int32_t hash_find_slot(const HashEntry* table, uint32_t mask, uint64_t key) {
  const HashSeq seq = hash_seq(key);
  uint32_t h = hash_home(seq, mask);
  for (uint32_t probe = 0; probe <= mask;) {
    const uint64_t k = table[h].key;
    if (k == key) return int32_t(h);
    if (k == kKeyEmpty) return -1;
    h = hash_probe(seq, ++probe, mask);
  }
  return -1;
}

// symmetric 3x3 index (xx xy xz yy yz zz)
__host__ __device__ constexpr int s6(int a, int b) {
  return a <= b ? (a == 0 ? b : (a == 1 ? 2 + b : 5)) : (b == 0 ? a : (b == 1 ? 2 + a : 5));
}

// One Jacobi rotation in the plane (p, q): apq becomes zero, apr and aqr are
// the elements coupling p and q to the third axis, vp and vq the columns of V.
// The angle comes from cos and sin of twice the angle, two reciprocal square
// roots in sequence (the textbook form's chain is three divisions and two
// square roots, over three times as long); rows and columns change by
// a' = a - s (b + tau a), tau = s / (1 + c), which rounds less than
// c a - s b.
__device__ inline void jacobi_rotate(double& app, double& aqq, double& apq, double& apr, double& aqr, double* vp,
                                     double* vq) {
  const double d = aqq - app, h = 2.0 * apq;
  const double z = fma(d, d, h * h);
  if (!(z > 1e-290)) return;  // nothing left to rotate
  const double x = rsqrt_pos(z);
  const double u = fma(0.5 * fabs(d), x, 0.5);  // cos^2 of the angle
  const double y = rsqrt_pos(u);
  const double c = u * y;
  double s = 0.5 * fabs(h) * x * y;
  if ((d < 0.0) != (h < 0.0) && d != 0.0) s = -s;
  if (d == 0.0 && h < 0.0) s = -s;
  const double ta = s * y * apq;
  app -= ta;
  aqq += ta;
  apq = 0.0;
  const double tau = s * rcp_pos(1.0 + c);
  auto turn = [&](double& a, double& b) {
    const double a0 = a, b0 = b;
    a = fma(-s, fma(tau, a0, b0), a0);
    b = fma(s, fma(-tau, b0, a0), b0);
  };
  turn(apr, aqr);
  for (int k = 0; k < 3; ++k) turn(vp[k], vq[k]);
}

// Cyclic Jacobi on a symmetric 3x3 (the oracle's method and sweep order;
// eigenvalues ascending, eigenvectors in columns of V row-major).  Over
// 500,000 covariances of planar, thick and degenerate point sets: eigenvalues
// within 5e-16 of the largest one (1.9e-15 with the textbook rotations),
// normals times the eigenvalue gap within 4.4e-16 (7.4e-16).
__device__ inline void eigh3_dev(const double Ain[9], double ev[3], double V[9]) {
  double a00 = Ain[0], a11 = Ain[4], a22 = Ain[8];
  double a01 = 0.5 * (Ain[1] + Ain[3]), a02 = 0.5 * (Ain[2] + Ain[6]), a12 = 0.5 * (Ain[5] + Ain[7]);
  double v0[3] = {1.0, 0.0, 0.0}, v1[3] = {0.0, 1.0, 0.0}, v2[3] = {0.0, 0.0, 1.0};  // columns
  for (int sweep = 0; sweep < 64; ++sweep) {
    const double off = a01 * a01 + a02 * a02 + a12 * a12;
    const double dia = a00 * a00 + a11 * a11 + a22 * a22;
    if (off <= 1e-36 * dia || off == 0.0) break;
    jacobi_rotate(a00, a11, a01, a02, a12, v0, v1);
    jacobi_rotate(a00, a22, a02, a01, a12, v0, v2);
    jacobi_rotate(a11, a22, a12, a01, a02, v1, v2);
  }
  // ascending order by three exchanges (ties keep index order)
  auto order = [](double& x, double& y, double* p, double* q) {
    if (!(y < x)) return;
    const double t = x;
    x = y;
    y = t;
    for (int k = 0; k < 3; ++k) {
      const double w = p[k];
      p[k] = q[k];
      q[k] = w;
    }
  };
  order(a00, a11, v0, v1);
  order(a11, a22, v1, v2);
  order(a00, a11, v0, v1);
  ev[0] = a00;
  ev[1] = a11;
  ev[2] = a22;
  for (int k = 0; k < 3; ++k) {
    V[3 * k] = v0[k];
    V[3 * k + 1] = v1[k];
    V[3 * k + 2] = v2[k];
  }
}

__device__ inline void write_hot(const MapDev& m, int32_t vid, uint32_t flags) {
  const double* pl = m.plane + size_t(vid) * kPlaneD;
  int64_t kx, ky, kz;
  unpack_key(m.vs[vid].key, kx, ky, kz);
  VoxHot h;
  h.mx = float(pl[0] - double(kx) * m.vs64);
  h.my = float(pl[1] - double(ky) * m.vs64);
  h.mz = float(pl[2] - double(kz) * m.vs64);
  h.flags = flags;
  h.nx = float(pl[3]);
  h.ny = float(pl[4]);
  h.nz = float(pl[5]);
  h.pad = 0.f;
  m.hot[vid] = h;
}

#define VMP_GRID_LOOP(i, n) for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < (n); i += gridDim.x * blockDim.x)

// what a session's counters start a scan from
__device__ inline void begin_scan(MapCounters* c) {
  c->tag += 1;
  c->fast = 0;
  c->nseg = c->ncreate_ev = c->ncre = c->nevict = c->ncand = 0;
  c->refits = c->merge_calls = c->merge_evals = c->merges = c->dropped = 0;
  c->merge_windows = c->merge_requeued = c->merge_max_acting = 0;
}
__global__ void k_fill_i32(int32_t* p, int32_t v, int n) {
  VMP_GRID_LOOP(i, n) p[i] = v;
}

// A session whose creation events all fit under its capacity (no LRU
// eviction in this scan) takes its new voxels from the free-list top down,
// then from the bump pointer.  Its counters advance as soon as its creation
// count is known; the free-list top and bump pointer they started from stay
// in S for k_create_init.  Other sessions keep fast = 0 and go through
// k_create_evict.
__device__ inline void create_fast_counters(const MapDev& m, SessInfo& S, int nc) {
  MapCounters* c = m.ctr;
  if (c->size + nc > m.capacity) return;
  const int ftop = c->free_top, bump = c->bump;
  S.ftop0 = ftop;
  S.bump0 = bump;
  if (nc <= ftop) {
    c->free_top = ftop - nc;
  } else {
    c->bump = bump + (nc - ftop);
    c->free_top = 0;
  }
  if (c->bump > m.pool) atomicOr(&c->error, 8);
  c->size += nc;
  c->group_counter += uint64_t(nc);
  c->ncre = nc;
  c->nevict = 0;
  c->fast = 1;
}

// per-session [lo, hi) of an ascending list of n global indices
// which: 0 segments, 1 creation events
__device__ inline void session_range(const MapDev* maps, SessInfo* si, int s, const int32_t* list, int n,
                                     int which) {
  auto lb = [&](int v) {
    int lo = 0, hi = n;
    while (lo < hi) {
      const int mid = (lo + hi) >> 1;
      if (list[mid] < v) lo = mid + 1;
      else hi = mid;
    }
    return lo;
  };
  const int lo = lb(si[s].off), hi = lb(si[s].off + si[s].n);
  MapCounters* c = maps[s].ctr;
  if (which == 0) {
    si[s].seg_lo = lo;
    si[s].seg_hi = hi;
    c->nseg = hi - lo;
  } else {
    si[s].cre_lo = lo;
    si[s].cre_hi = hi;
    c->ncreate_ev = hi - lo;
    create_fast_counters(maps[s], si[s], hi - lo);
  }
}
__global__ void k_ranges(const MapDev* maps, SessInfo* si, int nsess, const int32_t* list, const int32_t* count,
                         int which) {
  const int s = blockIdx.x * blockDim.x + threadIdx.x;
  if (s < nsess) session_range(maps, si, s, list, *count, which);
}
// The same, inside the compaction that produces the list: a session's first
// list position is the number of items selected before its first point,
// which the thread holding that point knows once its tile's prefix is known
// (sfirst[t] .. sfirst[t + 1] - 1 are the sessions starting in tile t); the
// last tile to finish sets each session's end (the next one's start, or the
// count) and its counter.  Sessions starting at or past nitems (empty
// trailing sessions) start at the count.
__device__ inline int32_t* range_lo(SessInfo& S, int which) {
  return which == 0 ? &S.seg_lo : &S.cre_lo;
}
struct TailRanges {
  const MapDev* maps;
  SessInfo* si;
  int nsess;
  const int32_t* list;
  int which;
  const int32_t* sfirst;
  int nitems;
  static constexpr bool kActive = true;
  __device__ void at_tile(int tile, int base, int pos, const int32_t (&v)[kPrimIpt]) const {
    const int s1 = sfirst[tile + 1];
    for (int s = sfirst[tile]; s < s1; ++s) {
      const int o = si[s].off;
      if (o < base || o >= base + kPrimIpt) continue;
      int p = pos;
#pragma unroll
      for (int k = 0; k < kPrimIpt; ++k)
        if (k < o - base && v[k] != 0) ++p;
      *range_lo(si[s], which) = p;
    }
  }
  __device__ void operator()(int n) const {
    for (int s = threadIdx.x; s < nsess; s += blockDim.x) {
      const int lo = si[s].off >= nitems ? n : *range_lo(si[s], which);
      const int hi = s + 1 < nsess ? (si[s + 1].off >= nitems ? n : *range_lo(si[s + 1], which)) : n;
      if (si[s].off >= nitems) *range_lo(si[s], which) = lo;
      MapCounters* c = maps[s].ctr;
      if (which == 0) {
        si[s].seg_hi = hi;
        c->nseg = hi - lo;
      } else {
        si[s].cre_hi = hi;
        c->ncreate_ev = hi - lo;
        create_fast_counters(maps[s], si[s], hi - lo);
      }
    }
  }
};

// ------------------------------------------------------------------ K1 ----
// The map stage's first kernel: also starts every session's counters (this
// kernel itself touches their error and used_entries only), the stage's
// clock, and the counts and flags of the later passes.
__global__ void k_ins_keys(const MapDev* maps, const SessInfo* si, int nsess, BatchBufs b, uint64_t* clk) {
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    clk[1] = wall_clock64();
    b.cnt[5] = 0;
    b.cnt[6] = 0;
  }
  VMP_GRID_LOOP(s, nsess) begin_scan(maps[s].ctr);
  // claimed slots: one atomic per block for a session alone (one per wave of a
  // 120,000-point scan queued up behind each other), else per wave and session
  __shared__ int claimed;
  if (threadIdx.x == 0) claimed = 0;
  __syncthreads();
  VMP_UNIFORM_LOOP(g, valid, b.ntot) {
    int ins = 0;
    const int s = valid ? sess_of(si, nsess, g) : 0;
    if (valid) {
    const SessInfo& S = si[s];
    const MapDev m = maps[s];
    const int i = g - S.off;
    const UpdParams& P = *S.prm;
    float pw[3];
    ins_transform(P.m, P.t, S.x[i], S.y[i], S.z[i], pw);
    int64_t k[3];
    bool ok = true;
    for (int r = 0; r < 3; ++r) {
      k[r] = int64_t(floor(double(pw[r]) / m.vs64));
      ok &= key_ok(k[r]);
    }
    int32_t e = -1;
    if (ok) e = hash_find_or_insert(m.table, m.hmask, pack_key(k[0], k[1], k[2]), m.ctr, &ins);
    else atomicOr(&m.ctr->error, 2);
    b.skey_in[g] = (uint64_t(s) << b.hbits) | uint64_t(uint32_t(e < 0 ? 0 : e));
    b.sval_in[g] = g;
    b.flags[g] = 0;
    }
    if (nsess > 1) {
      wave_fetch_add(&maps[s].ctr->used_entries, ins);
    } else {
      const uint64_t bal = __ballot(ins);
      if ((threadIdx.x & 63) == 0 && bal) atomicAdd(&claimed, __popcll(bal));
    }
  }
  __syncthreads();
  if (threadIdx.x == 0 && claimed) atomicAdd(&maps[0].ctr->used_entries, claimed);
}

// ------------------------------------------------------------------ K3 ----
// Segment heads: a key-sorted point whose key differs from the one before it
// (a key holds its session, so sessions begin segments too).
struct PredHead {
  const uint64_t* key;
  __device__ int32_t operator()(int i) const { return i == 0 || key[i] != key[i - 1] ? 1 : 0; }
};
__global__ void k_seg_heads(BatchBufs b) {
  const PredHead head{b.skey_out};
  VMP_GRID_LOOP(j, b.ntot) b.flags[j] = head(j);
}

// Whether this scan's walk of a voxel reaches a refit (updatePlane with
// n >= update_size_thresh, voxel_map.cpp:42-95), from counts alone: an
// uninitialised voxel refits when n reaches the threshold, an initialised
// enabled one when newly_add does, before the walk stops at the freeze
// point (n >= max_point_thresh); a build refits every voxel with enough
// points once at the end.
__device__ inline bool walk_refits(int n0, int newly0, uint32_t flags, int len, int upd, int mx, bool build) {
  if (build) return n0 + len >= upd;
  if ((flags & kInit) && !(flags & kEnable)) return false;
  if (!(flags & kInit)) return len > upd - n0 - 1;
  const int jr = upd - newly0 - 1;                  // walk index of the next refit
  const int f = mx - n0 - 1 > 0 ? mx - n0 - 1 : 0;  // walk index of the freeze point
  return jr < (len < f + 1 ? len : f + 1);
}

// How a voxel's points of this scan replay: 0 not at all (no voxel), class 1
// frozen before the scan (counted only), 2 .. kClsHeavy - 1 the light walk of
// class - 1 points (clamped), kClsHeavy and above the moment path, by length.
constexpr uint32_t kClsHeavy = 64;
__device__ inline uint32_t replay_class(const MapDev& m, int n0, int newly0, uint32_t flags, int len, bool build) {
  if (walk_refits(n0, newly0, flags, len, m.upd_pt, m.max_pt, build))
    return kClsHeavy + min(uint32_t(len), kClsHeavy - 1);
  if (!build && (flags & kInit) && !(flags & kEnable)) return 1;
  return 1 + min(uint32_t(len), kClsHeavy - 2);
}

// ------------------------------------------------------------------ K4 ----
// Item j: segment j's record (the existing voxel's fields of this scan, its
// replay class; a creation event at the first point of a segment without a
// voxel), and the replays' input of sorted point j (so a voxel's points are
// contiguous): the point relative to its voxel's centre, its world covariance
// (calcBodyCov's z = 0 -> 0.001 applies to the covariance only,
// commons.cpp:20-23) and its index in the scan, (q.x, q.y, q.z, index bits,
// C0..C5, -, -).  The transform and the key are k_ins_keys' expressions, so
// the voxel is the one the point was keyed to.
__global__ void k_seg_info(const MapDev* maps, const SessInfo* si, int nsess, BatchBufs b) {
  const int nseg = b.cnt[0];
  VMP_GRID_LOOP(j, b.ntot) {
    if (j < nseg) {
      const int q = j;
      const int start = b.sel[q];
      const int s = sess_of(si, nsess, start);
      const SessInfo& S = si[s];
      const int lim = S.off + S.n;
      const int end = (q + 1 < nseg && b.sel[q + 1] < lim) ? b.sel[q + 1] : lim;
      const MapDev m = maps[s];
      const uint32_t e = uint32_t(b.skey_out[start] & ((uint64_t(1) << b.hbits) - 1));
      const int first = b.sval_out[start] - S.off;
      b.seg_start[q] = start;
      b.seg_end[q] = end;
      b.seg_sess[q] = s;
      b.seg_entry[q] = int32_t(e);
      const int32_t vid = m.table[e].vid;
      b.seg_vid[q] = vid;
      b.seg_old[q] = vid;
      uint32_t cls = 0;
      if (vid >= 0) {  // this scan's fields (three vector stores)
        VoxState* st = m.vs + vid;
        cls = replay_class(m, st->n, st->newly_add, st->flags, end - start, S.is_build != 0);
        st_global2(&st->merge_pos, kNever, -2);
        st_global4(&st->tag, m.ctr->tag, -1, kNever, -1);
        st_global4(&st->prev_vid, -1, first, q, 0);
      } else {
        b.flags[S.off + first] = q + 1;  // creation event at its first point (array cleared before)
      }
      b.seg_cls[q] = cls;
    }
    const int s = sess_of(si, nsess, j);
    const SessInfo& S = si[s];
    const double vs64 = maps[s].vs64;
    const UpdParams& P = *S.prm;
    const int i = b.sval_out[j] - S.off;
    const float x = S.x[i], y = S.y[i], z = S.z[i];
    float pw[3];
    ins_transform(P.m, P.t, x, y, z, pw);
    float qv[3];
    for (int r = 0; r < 3; ++r) {
      const int64_t k = int64_t(floor(double(pw[r]) / vs64));
      qv[r] = float(double(pw[r]) - (double(k) + 0.5) * vs64);
    }
    const float pz = z == 0.0f ? 0.001f : z;
    float C[6];
    point_world_cov(P.rwl32, P.Prr, P.Ppp, P.s2, P.rv, x, y, pz, C);
    b.qc[3 * size_t(j)] = make_float4(qv[0], qv[1], qv[2], __int_as_float(i));
    b.qc[3 * size_t(j) + 1] = make_float4(C[0], C[1], C[2], C[3]);
    b.qc[3 * size_t(j) + 2] = make_float4(C[4], C[5], 0.0f, 0.0f);
  }
}

__global__ void k_cre_split(const SessInfo* si, int nsess, BatchBufs b) {
  const int nc = b.cnt[1];
  VMP_GRID_LOOP(r, nc) {
    const int g = b.sel[r];
    const int s = sess_of(si, nsess, g);
    b.cre_t[r] = g - si[s].off;
    b.cre_seg[r] = b.flags[g] - 1;
  }
}
// the same as the output of the compaction of the creation events (v: the
// event's flag, its segment + 1)
struct OutCre {
  int32_t* sel;
  int32_t* cre_t;
  int32_t* cre_seg;
  const SessInfo* si;
  int nsess;
  __device__ void operator()(int r, int g, int32_t v) const {
    sel[r] = g;
    cre_t[r] = g - si[sess_of(si, nsess, g)].off;
    cre_seg[r] = v - 1;
  }
};

// ------------------------------------------------------------------ K5 ----
// Chunks of the ring that k_ring_live compacts for a session: enough for the
// creations of most scans at a few stale entries per victim, within the
// session's two entries per point; k_create_evict reads the ring itself
// beyond them.
__device__ inline int64_t lv_chunks(const MapCounters* c, const SessInfo& S) {
  const int64_t used = c->ring_tail - c->ring_head;
  const int64_t want = int64_t(6) * (S.cre_hi - S.cre_lo) + 4096;
  return min(min((used + 63) >> 6, (want + 63) >> 6), (int64_t(2) * S.n) >> 6);
}

// The ring entry `rel` places after the head as (vid, first touch in this
// scan or kNever, segment, rel); vid -1 if it is past the tail or stale.  An
// entry is live while its voxel is alive, still carries the entry's stamp
// and has not been evicted in this scan; no decision of k_create_evict makes
// another entry live.
__device__ inline int4 ring_entry(const MapDev& m, int64_t head, int64_t tail, int tag, int64_t rel) {
  int4 e = make_int4(-1, kNever, -1, int32_t(rel));
  if (head + rel >= tail) return e;
  const int64_t ph = (head + rel) % m.qcap;
  const int32_t v = m.ring_vid[ph];
  const uint64_t stp = m.ring_stamp[ph];
  const VoxState& st = m.vs[v];
  const bool cur = st.tag == tag;
  if ((st.flags & kAlive) && st.stamp == stp && !(cur && st.evict_t != kNever)) e.x = v;
  if (cur && st.create_t < 0) e.y = st.first_t;
  e.z = st.seg;
  return e;
}

constexpr int kLvWaves = 4;   // waves per block of k_ring_live
constexpr int kLvBlocks = 32; // blocks per session

// The live ring entries ahead of the head (grid: kLvBlocks x sessions), one
// wave per 64-entry chunk, compacted within the chunk.
__global__ void __launch_bounds__(64 * kLvWaves) k_ring_live(const MapDev* maps, const SessInfo* si, int nsess,
                                                              BatchBufs b) {
  const int s = blockIdx.y;
  if (s >= nsess) return;
  const MapDev m = maps[s];
  const MapCounters* c = m.ctr;
  if (c->fast) return;
  const SessInfo S = si[s];
  const int64_t nch = lv_chunks(c, S);
  const int64_t head = c->ring_head, tail = c->ring_tail;
  const int tag = c->tag;
  const int lane = threadIdx.x & 63;
  int4* out0 = b.lv + int64_t(2) * S.off;
  for (int64_t k = int64_t(blockIdx.x) * kLvWaves + (threadIdx.x >> 6); k < nch;
       k += int64_t(gridDim.x) * kLvWaves) {
    const int4 e = ring_entry(m, head, tail, tag, k * 64 + lane);
    const uint64_t bal = __ballot(e.x >= 0);
    if (e.x >= 0) out0[k * 64 + __popcll(bal & bits_below(lane))] = e;
    if (lane == 0) b.lv_cnt[lv_cnt_base(S.off, s) + k] = __popcll(bal);
  }
}

// Creations and evictions in order, one workgroup per session that may
// overflow.  LRU order is the descending order of last-touch stamps; the
// ring holds (vid, stamp) in ascending stamp order with stale entries skipped
// lazily.  The victim of each creation is the oldest live voxel not yet
// touched by an earlier point of this scan; a victim touched later comes back
// as a new voxel at its first touch (another creation event).
//
// All decisions are taken at once.  Let the events (creations and
// re-creations) in time order be T_0 < T_1 < ..., Z the creations that still
// fit under the capacity, f_i the first touch of the live ring entry i in
// this scan (kNever: none) and r_i the number of victims before i.  The ring
// pointer reaches i with the event Z + r_i, so i is a victim if and only if
// f_i > T_(Z + r_i), that is, if at least Z + r_i + 1 events precede f_i; an
// untouched entry always is, while events are left.  Only the touched
// entries need deciding, and whether one is a victim changes r of the
// entries after it and the events after its first touch only.  So: one bit
// per live entry (victim) and per point time (event), all touched entries
// evaluated against prefix counts of both, the changed bits flipped, until a
// round changes none.
//
// Such a state is the sequential result: by induction over i, r_i is right,
// and a victim behind i returns after the event that reaches i.  And the
// rounds end: once the entries before i are settled, one behind i that is
// wrongly held a victim with a first touch before T_(Z + r_i) is dropped by
// the next round if no other such entry has an earlier first touch, and
// without such entries i itself is right.  Their number grows with the logarithm
// of the touched entries: a restatement on the CPU took up to 6 for 2,400 random
// scans of 60,000 points, and for 60,000 touched entries 13 in random order, 18
// with the first touches descending along the ring, 3 to 8 nearly ascending.
//
// For 6,300 evictions of a 60k-point scan 30 us, bound by the chain of round
// trips and barriers; one decision after the other (about 1 us for each step
// of up to 64 of them) took 181 us.
constexpr int kCeThreads = 1024;  // k_create_evict block
constexpr int kCeWaves = kCeThreads / 64;
constexpr int kEvWords = 4096;    // words of each bit table that fit in LDS (262,144 bits)
constexpr int kEvUnroll = 8;      // ring chunks a wave loads per round trip
constexpr uint64_t kCandWrong = uint64_t(1) << 31;  // above the 26 bits of a live entry's index
struct EvTables {
  uint64_t* ev;  // bit t: an event at point time t
  uint64_t* vw;  // bit i: live entry i is a victim
  int32_t* evp;  // bits set before each word
  int32_t* vp;
};

// marks an evicted voxel in its record (one lane); cur: the record already
// carries this scan's fields
__device__ inline void evict_write(const MapDev& m, int tag, int32_t victim, bool cur, int t) {
  VoxState* st = m.vs + victim;
  if (cur) {
    *as_global(&st->evict_t) = t;
  } else {  // this scan's fields start here (three vector stores)
    st_global2(&st->merge_pos, kNever, -2);
    st_global4(&st->tag, tag, -1, t, -1);
    st_global4(&st->prev_vid, -1, kNever, -1, 0);
  }
}

// a bit table's word: in LDS, or in global memory, where the flips are
// device-scope atomics that plain loads could miss
template <bool kLds>
__device__ inline uint64_t ev_word(const uint64_t* p) {
  return kLds ? *p : __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// exclusive prefix counts of the set bits of w[0 .. n) into p; returns the
// total (a block of kCeThreads, four words each per pass)
template <bool kLds>
__device__ inline int bits_scan(const uint64_t* w, int n, int32_t* p, int32_t* wsum) {
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  int carry = 0;
  for (int i0 = 0; i0 < n; i0 += 4 * kCeThreads) {
    const int i = i0 + 4 * tid;
    int v[4], sum = 0;
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      v[u] = i + u < n ? __popcll(ev_word<kLds>(w + i + u)) : 0;
      sum += v[u];
    }
    int incl = sum;
    for (int o = 1; o < 64; o <<= 1) {
      const int x = __shfl_up(incl, o, 64);
      if (lane >= o) incl += x;
    }
    if (lane == 63) wsum[wave] = incl;
    __syncthreads();
    int run = carry + incl - sum;
#pragma unroll
    for (int q = 0; q < kCeWaves; ++q) {
      const int x = wsum[q];
      run += q < wave ? x : 0;
      carry += x;
    }
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      if (i + u < n) p[i + u] = run;
      run += v[u];
    }
    __syncthreads();
  }
  return carry;
}

// The decisions over nlive packed live entries (b.lv2, at 2 * off): the
// events into b.co, the victims into b.ev_vid and their records, the
// session's counters.  With too few victims in the whole ring the scan
// touches more new voxels than the LRU can evict: error 4, nothing changed.
template <bool kLds>
__device__ inline void evict_decide(const MapDev& m, const SessInfo& S, const BatchBufs& b, int nlive, int Z,
                                    const EvTables& T, int32_t* wsum, int* ncand) {
  MapCounters* c = m.ctr;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int clo = S.cre_lo, ncre_ev = S.cre_hi - clo, off = S.off;
  const int nw = (S.n + 63) >> 6, nk = (nlive + 63) >> 6;
  const int4* lv = b.lv2 + int64_t(2) * off;
  uint64_t* cand = b.cand_in + off;  // touched entries: (first touch << 32) | entry
  auto flip = [](uint64_t* p, int bit) {
    atomicXor(reinterpret_cast<unsigned long long*>(p), 1ull << bit);
  };
  for (int i = tid; i < nw; i += kCeThreads) T.ev[i] = 0;
  if (tid == 0) *ncand = 0;
  __syncthreads();
  for (int r = tid; r < ncre_ev; r += kCeThreads) {
    const int t = b.cre_t[clo + r];
    flip(T.ev + (t >> 6), t & 63);
  }
  for (int k = wave; k < nk; k += kCeWaves) {
    const int i = 64 * k + lane;
    const int f = i < nlive ? lv[i].y : kNever;
    const uint64_t bt = __ballot(f != kNever), bu = __ballot(i < nlive && f == kNever);
    if (lane == 0) T.vw[k] = bu;
    if (bt) {
      int base = 0;
      if (lane == 0) base = atomicAdd(ncand, __popcll(bt));
      base = __builtin_amdgcn_readfirstlane(base);
      if (f != kNever) cand[base + __popcll(bt & bits_below(lane))] = (uint64_t(uint32_t(f)) << 32) | uint32_t(i);
    }
  }
  __syncthreads();
  const int nt = *ncand;
  auto victim_bit = [&](int i) { return (ev_word<kLds>(T.vw + (i >> 6)) >> (i & 63)) & 1ull; };
  auto rank = [&](int i) { return T.vp[i >> 6] + __popcll(ev_word<kLds>(T.vw + (i >> 6)) & bits_below(i & 63)); };
  auto events_before = [&](int t) {
    return T.evp[t >> 6] + __popcll(ev_word<kLds>(T.ev + (t >> 6)) & bits_below(t & 63));
  };
  int nev, nvict;
  while (true) {
    nev = bits_scan<kLds>(T.ev, nw, T.evp, wsum);
    nvict = bits_scan<kLds>(T.vw, nk, T.vp, wsum);
    // every evaluation of a round precedes its flips: a wrong bit is noted in
    // the entry's bit 31 (its own thread flips it after the barrier)
    int wrong = 0;
    for (int q = tid; q < nt; q += kCeThreads) {
      const uint64_t cq = cand[q];
      const int f = int(cq >> 32), i = int(uint32_t(cq));
      if (int(events_before(f) >= Z + rank(i) + 1) != int(victim_bit(i))) {
        cand[q] = cq | kCandWrong;
        wrong = 1;
      }
    }
    if (!__syncthreads_or(wrong)) break;
    for (int q = tid; wrong && q < nt; q += kCeThreads) {
      uint64_t cq = cand[q];
      if (!(cq & kCandWrong)) continue;
      cand[q] = cq &= ~kCandWrong;
      const int f = int(cq >> 32), i = int(uint32_t(cq));
      flip(T.vw + (i >> 6), i & 63);
      flip(T.ev + (f >> 6), f & 63);
    }
    __syncthreads();
  }
  const int need = nev - Z;  // one victim per event from the Z-th on
  if (nvict < need || nev > S.n) {
    if (tid == 0) atomicOr(&c->error, 4);
    return;
  }
  // ---- the events in order: the j-th takes the j-th free slot
  const int ftop = c->free_top, bump = c->bump;
  int err = 0;
  auto slot_of = [&](int j) {
    const int32_t vid = j < ftop ? m.freelist[ftop - 1 - j] : bump + (j - ftop);
    if (vid >= m.pool) err = 8;
    return vid;
  };
  for (int r = tid; r < ncre_ev; r += kCeThreads) {
    const int t = b.cre_t[clo + r], seg = b.cre_seg[clo + r];
    const int j = events_before(t);
    b.co[off + j] = make_int4(slot_of(j), seg, t, -1);
  }
  for (int q = tid; q < nt; q += kCeThreads) {
    const int i = int(uint32_t(cand[q]));
    if (!victim_bit(i)) continue;
    const int4 e = lv[i];
    const int j = events_before(e.y);
    b.co[off + j] = make_int4(slot_of(j), e.z, e.y, e.x);
  }
  if (err) atomicOr(&c->error, err);
  __syncthreads();
  // ---- the victims in order: the r-th goes at the event Z + r
  const int tag = c->tag;
  int last = -1;
  for (int k = wave; k < nk; k += kCeWaves) {
    if (T.vp[k] >= need) break;
    const int i = 64 * k + lane;
    const int r = rank(i);
    if (!victim_bit(i) || r >= need) continue;
    const int4 e = lv[i];
    const int t = b.co[off + Z + r].z;
    evict_write(m, tag, e.x, e.y != kNever, t);
    b.ev_vid[off + r] = e.x;
    if (r == need - 1) last = e.w;
  }
  __syncthreads();  // every read of the counters precedes their update
  if (last >= 0) {  // the thread of the last victim
    c->size += Z;
    c->group_counter += uint64_t(nev);
    c->free_top = max(0, ftop - nev);
    c->bump = bump + max(0, nev - ftop);
    c->ring_head += last + 1;
    c->ncre = nev;
    c->nevict = need;
  }
}

__global__ void __launch_bounds__(kCeThreads) k_create_evict(const MapDev* maps, const SessInfo* si, int nsess,
                                                             BatchBufs b) {
  const int s = blockIdx.x;
  if (s >= nsess) return;
  const MapDev m = maps[s];
  const MapCounters* c = m.ctr;
  if (c->fast) return;
  __shared__ uint64_t s_ev[kEvWords], s_vw[kEvWords];
  __shared__ int32_t s_evp[kEvWords], s_vp[kEvWords];
  __shared__ int32_t wsum[kCeWaves], wt[kCeWaves];
  __shared__ int ncand;
  const SessInfo S = si[s];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int off = S.off, ncre_ev = S.cre_hi - S.cre_lo;
  const int Z = int(max(int64_t(0), int64_t(m.capacity) - c->size));  // below ncre_ev: the session is not a fast one
  // ---- the live entries from the head on, packed in ring order, up to
  //      where the untouched ones alone could serve every creation and every
  //      return of a touched one before them (creations and touched old
  //      voxels have distinct first points, so that is at most 2 n entries)
  const int64_t nch = lv_chunks(c, S);
  const int64_t head = c->ring_head, tail = c->ring_tail, used = tail - head;
  const int tag = c->tag;
  const int4* lvc = b.lv + int64_t(2) * off;
  const int32_t* lcnt = b.lv_cnt + lv_cnt_base(off, s);
  int4* packed = b.lv2 + int64_t(2) * off;
  const int lim = 2 * S.n;
  int nl = 0, nt = 0;
  for (int64_t k0 = 0; 64 * k0 < used; k0 += kCeWaves * kEvUnroll) {
    const int64_t kw = k0 + wave * kEvUnroll;
    int4 e[kEvUnroll];
    if (kw + kEvUnroll <= nch) {  // compacted ahead: every load of the round first
      int cn[kEvUnroll];
#pragma unroll
      for (int u = 0; u < kEvUnroll; ++u) {
        cn[u] = lcnt[kw + u];
        e[u] = lvc[(kw + u) * 64 + lane];
      }
#pragma unroll
      for (int u = 0; u < kEvUnroll; ++u)
        if (lane >= cn[u]) e[u] = make_int4(-1, kNever, -1, 0);
    } else {
#pragma unroll
      for (int u = 0; u < kEvUnroll; ++u) e[u] = ring_entry(m, head, tail, tag, (kw + u) * 64 + lane);
    }
    int su = 0, stt = 0;
#pragma unroll
    for (int u = 0; u < kEvUnroll; ++u) {
      su += __popcll(__ballot(e[u].x >= 0));
      stt += __popcll(__ballot(e[u].x >= 0 && e[u].y != kNever));
    }
    if (lane == 0) {
      wsum[wave] = su;
      wt[wave] = stt;
    }
    __syncthreads();
    int at = nl;
    for (int q = 0; q < kCeWaves; ++q) {
      at += q < wave ? wsum[q] : 0;
      nl += wsum[q];
      nt += wt[q];
    }
#pragma unroll
    for (int u = 0; u < kEvUnroll; ++u) {
      const uint64_t bal = __ballot(e[u].x >= 0);
      const int i = at + __popcll(bal & bits_below(lane));
      if (e[u].x >= 0 && i < lim) packed[i] = e[u];
      at += __popcll(bal);
    }
    __syncthreads();
    if (nl - nt >= ncre_ev - Z + nt) break;
  }
  const int nlive = min(nl, lim);
  const int nw = (S.n + 63) >> 6, nk = (nlive + 63) >> 6;
  if (nw <= kEvWords && nk <= kEvWords) {
    evict_decide<true>(m, S, b, nlive, Z, EvTables{s_ev, s_vw, s_evp, s_vp}, wsum, &ncand);
  } else {  // the tables of a larger scan in the candidate stage's scratch, free until then
    uint64_t* ev = reinterpret_cast<uint64_t*>(b.cand_nbr + size_t(off) * 6);
    int32_t* evp = reinterpret_cast<int32_t*>(ev + nw + nk);
    evict_decide<false>(m, S, b, nlive, Z, EvTables{ev, ev + nw, evp, evp + nw}, wsum, &ncand);
  }
}

// Initialise created voxels and point their hash slots at them; a session
// whose LRU cannot overflow in this scan (fast, set with its counters where
// the creation events were counted) takes its voxel ids here.  Then every
// segment has its voxel and its replay class, and the refitting voxels are
// listed as (vid, start, length, session) records: all of them from the front
// of hlist (cnt[5] counts them) and, from its back, those with at least
// long_seg points (cnt[6]; 0 lists none).  The two parts cannot meet: a long
// segment holds two points or more.  A segment is listed by the thread of its
// creation, or by its own if its voxel was there before and stays; the two
// read nothing that the other writes (seg_old and the evict time).
__global__ void __launch_bounds__(kMapThreads) k_create_init(const MapDev* maps, const SessInfo* si, int nsess,
                                                             BatchBufs b, int long_seg) {
  constexpr int kW = kMapThreads / 64;
  __shared__ int woff[2][kW];
  __shared__ int bbase[2];
  const int nseg = b.cnt[0];
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  VMP_UNIFORM_LOOP(p, valid, b.ntot) {
    int4 rec[2] = {make_int4(-1, 0, 0, 0), make_int4(-1, 0, 0, 0)};
    if (valid) {
      const int s = sess_of(si, nsess, p);
      const SessInfo& S = si[s];
      const MapDev m = maps[s];
      const int r = p - S.off;
      const int ncre = m.ctr->ncre;
      if (r < ncre) {
        int4 co;
        if (m.ctr->fast) {
          const int k = S.cre_lo + r, ftop = S.ftop0;
          co = make_int4(r < ftop ? m.freelist[ftop - 1 - r] : S.bump0 + (r - ftop), b.cre_seg[k], b.cre_t[k], -1);
        } else {
          co = b.co[p];
        }
        const int32_t vid = co.x;
        const int q = co.y;
        if (vid >= 0 && vid < m.pool && q >= 0) {  // else the error is already flagged
          const int32_t e = b.seg_entry[q];
          const int start = b.seg_start[q], len = b.seg_end[q] - start;
          VoxState st;
          st.key = m.table[e].key;
          st.group_id = m.ctr->group_counter - uint64_t(ncre) + uint64_t(r);
          st.stamp = 0;
          st.n = 0;
          st.newly_add = 0;
          st.flags = kEnable | kAlive;
          st.pad = 0;
          st.tag = m.ctr->tag;
          st.create_t = co.z;
          st.evict_t = kNever;
          st.freeze_t = -1;
          st.prev_vid = co.w;
          st.first_t = co.z;
          st.seg = q;
          st.merge_pos = kNever;
          st.dirty_t = -2;
          st.pad1 = 0;
          m.vs[vid] = st;
          // the plane record and the moments are not cleared here: the voxel
          // has points in this scan, and the replay starts a voxel with n = 0
          // from zero
          VoxHot h{};
          h.flags = kEnable | kAlive;
          m.hot[vid] = h;
          m.table[e].vid = vid;
          b.seg_vid[q] = vid;
          const uint32_t cls = replay_class(m, 0, 0, kEnable | kAlive, len, S.is_build != 0);
          b.seg_cls[q] = cls;
          if (cls >= kClsHeavy) rec[0] = make_int4(vid, start, len, s);
        }
      }
      // the merge stage's per-point slots start empty (k_candidates fills
      // them; k_create_evict kept its touched entries there before)
      b.cand_in[p] = ~0ull;
      if (p < nseg) {
        const int32_t vid = b.seg_old[p];
        if (vid >= 0) {
          const int qs = b.seg_sess[p];
          const MapDev qm = maps[qs];
          const bool stays = qm.ctr->fast || qm.vs[vid].evict_t == kNever;
          if (stays && b.seg_cls[p] >= kClsHeavy)
            rec[1] = make_int4(vid, b.seg_start[p], b.seg_end[p] - b.seg_start[p], qs);
        }
      }
    }
    // the block's share of each list, wave by wave
    const bool hv[2] = {rec[0].x >= 0, rec[1].x >= 0};
    const bool lg[2] = {hv[0] && long_seg > 0 && rec[0].z >= long_seg, hv[1] && long_seg > 0 && rec[1].z >= long_seg};
    const uint64_t bh[2] = {__ballot(hv[0]), __ballot(hv[1])}, bl[2] = {__ballot(lg[0]), __ballot(lg[1])};
    if (lane == 0) {
      woff[0][wv] = __popcll(bh[0]) + __popcll(bh[1]);
      woff[1][wv] = __popcll(bl[0]) + __popcll(bl[1]);
    }
    __syncthreads();
    if (threadIdx.x < 2) {
      int run = 0;
      for (int w = 0; w < kW; ++w) {
        const int c = woff[threadIdx.x][w];
        woff[threadIdx.x][w] = run;
        run += c;
      }
      bbase[threadIdx.x] = run ? atomicAdd(&b.cnt[5 + threadIdx.x], run) : 0;
    }
    __syncthreads();
    const uint64_t below = bits_below(lane);
    int h0 = bbase[0] + woff[0][wv], l0 = bbase[1] + woff[1][wv];
#pragma unroll
    for (int k = 0; k < 2; ++k) {
      if (hv[k]) b.hlist[h0 + __popcll(bh[k] & below)] = rec[k];
      if (lg[k]) b.hlist[b.ntot - 1 - (l0 + __popcll(bl[k] & below))] = rec[k];
      h0 += __popcll(bh[k]);
      l0 += __popcll(bl[k]);
    }
    __syncthreads();
  }
}

// ------------------------------------------------------------------ K6 ----
struct Moments {
  double s1[3], s2[6], c0[6], c1[3][6], c2[6][6];
};

__device__ inline void mom_load(const double* src, Moments& M) {
  int o = 0;
  for (int a = 0; a < 3; ++a) M.s1[a] = src[o++];
  for (int a = 0; a < 6; ++a) M.s2[a] = src[o++];
  for (int a = 0; a < 6; ++a) M.c0[a] = src[o++];
  for (int a = 0; a < 3; ++a)
    for (int l = 0; l < 6; ++l) M.c1[a][l] = src[o++];
  for (int a = 0; a < 6; ++a)
    for (int l = 0; l < 6; ++l) M.c2[a][l] = src[o++];
}
__device__ inline void mom_zero(Moments& M) {
  for (int a = 0; a < 3; ++a) M.s1[a] = 0.0;
  for (int a = 0; a < 6; ++a) M.s2[a] = 0.0;
  for (int a = 0; a < 6; ++a) M.c0[a] = 0.0;
  for (int a = 0; a < 3; ++a)
    for (int l = 0; l < 6; ++l) M.c1[a][l] = 0.0;
  for (int a = 0; a < 6; ++a)
    for (int l = 0; l < 6; ++l) M.c2[a][l] = 0.0;
}
__device__ inline void mom_store(double* dst, const Moments& M) {
  int o = 0;
  for (int a = 0; a < 3; ++a) dst[o++] = M.s1[a];
  for (int a = 0; a < 6; ++a) dst[o++] = M.s2[a];
  for (int a = 0; a < 6; ++a) dst[o++] = M.c0[a];
  for (int a = 0; a < 3; ++a)
    for (int l = 0; l < 6; ++l) dst[o++] = M.c1[a][l];
  for (int a = 0; a < 6; ++a)
    for (int l = 0; l < 6; ++l) dst[o++] = M.c2[a][l];
}
// A point's contribution to every moment is one fused multiply-add of two
// of 16 factors, F = (1, q, q q^T (rounded, xx xy xz yy yz zz), C): each
// moment c takes F[mom_i1(c)] * F[mom_i2(c)].  Both the per-lane walk and
// the per-wave walk accumulate exactly these terms in point order, so the
// two give the same bits.  The moments are this library's own intermediate,
// not a quantity the reference rounds in a particular order.
constexpr int kMomC = 69;  // moment components (S1q S2q S0C S1C S2C)
constexpr int kMomF = 16;  // factors per point
__host__ __device__ constexpr int mom_i1(int c) {
  return c < 3 ? 1 + c
               : (c < 9 ? 1 + (c - 3 < 3 ? 0 : (c - 3 < 5 ? 1 : 2))
                        : (c < 15 ? 10 + (c - 9) : (c < 33 ? 1 + (c - 15) / 6 : 4 + (c - 33) / 6)));
}
__host__ __device__ constexpr int mom_i2(int c) {
  return c < 3 ? 0
               : (c < 9 ? 1 + (c - 3 < 3 ? c - 3 : (c - 3 < 5 ? c - 5 : 2))
                        : (c < 15 ? 0 : 10 + (c < 33 ? (c - 15) % 6 : (c - 33) % 6)));
}
__device__ inline void mom_factors(const float q[3], const float C[6], double F[kMomF]) {
  F[0] = 1.0;
  for (int a = 0; a < 3; ++a) F[1 + a] = double(q[a]);
  for (int a = 0; a < 3; ++a)
    for (int bb = a; bb < 3; ++bb) F[4 + s6(a, bb)] = F[1 + a] * F[1 + bb];
  for (int l = 0; l < 6; ++l) F[10 + l] = double(C[l]);
}
__device__ inline void mom_add(Moments& M, const float q[3], const float C[6]) {
  double F[kMomF];
  mom_factors(q, C, F);
  for (int a = 0; a < 3; ++a) M.s1[a] = fma(F[mom_i1(a)], F[mom_i2(a)], M.s1[a]);
  for (int a = 0; a < 6; ++a) M.s2[a] = fma(F[mom_i1(3 + a)], F[mom_i2(3 + a)], M.s2[a]);
  for (int l = 0; l < 6; ++l) M.c0[l] = fma(F[mom_i1(9 + l)], F[mom_i2(9 + l)], M.c0[l]);
  for (int a = 0; a < 3; ++a)
    for (int l = 0; l < 6; ++l) M.c1[a][l] = fma(F[mom_i1(15 + 6 * a + l)], F[mom_i2(15 + 6 * a + l)], M.c1[a][l]);
  for (int a = 0; a < 6; ++a)
    for (int l = 0; l < 6; ++l) M.c2[a][l] = fma(F[mom_i1(33 + 6 * a + l)], F[mom_i2(33 + 6 * a + l)], M.c2[a][l]);
}

// updatePlane (voxel_map.cpp:97-136) from moments.  Plane::cov is kept as the
// traces of its two diagonal blocks: the normal block's trace
// sum_i tr(F_i C_i F_i^T) is a quadratic form of d_i = p_i - mean, rebuilt
// from sum q q C, sum q C, sum C; the centre block adds tr(C_i)/n^2.
struct RefitOut {
  double tn, tm;   // increments of the two traces
  double nrm[3];   // the oriented normal
  bool plane;
};
__device__ inline RefitOut refit_eval(const MapDev& m, const Moments& M, int n, const double center[3]) {
  RefitOut o;
  o.plane = false;
  const double invn = 1.0 / double(n);
  double mu[3];
  for (int a = 0; a < 3; ++a) mu[a] = M.s1[a] * invn;
  double cov[9];
  for (int a = 0; a < 3; ++a)
    for (int bb = 0; bb < 3; ++bb) cov[a * 3 + bb] = M.s2[s6(a, bb)] * invn - mu[a] * mu[bb];
  double ev[3], V[9];
  eigh3_dev(cov, ev, V);
  if (ev[0] > m.plane_thresh) return o;
  o.plane = true;
  // the covariance moments are read after the eigen solve, not hoisted
  // above it (they would hold 120 registers through the Jacobi sweeps)
  asm volatile("" ::: "memory");
  // With d_i = q_i - mu and T[ab][lm] = sum_i d_a d_b C_lm
  //   = S2C[ab][lm] - mu_a S1C[b][lm] - mu_b S1C[a][lm] + mu_a mu_b S0C[lm],
  // and W(w,x) the symmetric weights of w x^T (xx xy xz yy yz zz; the
  // off-diagonal ones w_a x_b + w_b x_a), the numerator for eigenvector e is
  //   sum_{ab,lm} T[ab][lm] (W(n,n)[lm] W(e,e)[ab] + 2 W(e,n)[lm] W(e,n)[ab]
  //                          + W(e,e)[lm] W(n,n)[ab]),
  // formed one row ab of T at a time (T is not stored).
  const double nn[3] = {V[0], V[3], V[6]};
  auto W = [](const double* w, const double* x, double w6[6]) {
    for (int l = 0; l < 3; ++l)
      for (int mm = l; mm < 3; ++mm) w6[s6(l, mm)] = l == mm ? w[l] * x[l] : w[l] * x[mm] + w[mm] * x[l];
  };
  double Wnn[6], We[2][6], Wen[2][6];
  W(nn, nn, Wnn);
  for (int k = 0; k < 2; ++k) {
    const double e[3] = {V[1 + k], V[4 + k], V[7 + k]};
    W(e, e, We[k]);
    W(e, nn, Wen[k]);
  }
  double num[2] = {0.0, 0.0};
  for (int a = 0; a < 3; ++a)
    for (int bb = a; bb < 3; ++bb) {
      const int ab = s6(a, bb);
      double r1 = 0.0, r2[2] = {0.0, 0.0}, r3[2] = {0.0, 0.0};
      for (int l = 0; l < 6; ++l) {
        const double t = M.c2[ab][l] - mu[a] * M.c1[bb][l] - mu[bb] * M.c1[a][l] + mu[a] * mu[bb] * M.c0[l];
        r1 += t * Wnn[l];
        for (int k = 0; k < 2; ++k) {
          r2[k] += t * Wen[k][l];
          r3[k] += t * We[k][l];
        }
      }
      for (int k = 0; k < 2; ++k) num[k] += We[k][ab] * r1 + 2.0 * Wen[k][ab] * r2[k] + Wnn[ab] * r3[k];
    }
  double tn_inc = 0.0;
  for (int k = 0; k < 2; ++k) {
    const double den = double(n) * (ev[0] - ev[1 + k]);
    tn_inc += num[k] / (den * den);
  }
  o.tn = tn_inc;
  o.tm = (M.c0[0] + M.c0[3] + M.c0[5]) * invn * invn;
  double mw[3];
  for (int a = 0; a < 3; ++a) mw[a] = center[a] + mu[a];
  double axis = -(mw[0] * nn[0] + mw[1] * nn[1] + mw[2] * nn[2]);
  const double sg = axis < 0.0 ? -1.0 : 1.0;
  for (int a = 0; a < 3; ++a) o.nrm[a] = sg * nn[a];
  return o;
}
// A refit's effect on the voxel: every refit initialises it; a plane refit
// adds to the two traces and replaces the normal, a non-plane one clears
// the plane flag.  A voxel's refits apply in walk order.
__device__ inline void refit_apply(const RefitOut& o, uint32_t& flags, double* pl) {
  flags |= kInit;
  if (!o.plane) {
    flags &= ~kPlane;
    return;
  }
  flags |= kPlane;
  pl[6] += o.tn;
  pl[7] += o.tm;
  for (int a = 0; a < 3; ++a) pl[3 + a] = o.nrm[a];
}
__device__ inline void refit(const MapDev& m, Moments& M, int n, uint32_t& flags, double* pl,
                             const double center[3], int& refits) {
  if (n < m.upd_pt) return;
  ++refits;
  refit_apply(refit_eval(m, M, n, center), flags, pl);
}

// The whole walk of a voxel in this scan from counts alone (the state
// machine of the lane walk in k_replay_heavy, voxel_map.cpp:42-95): the
// walk index of the refit that initialises the voxel, then of the first
// refit of the initialised voxel (one every update_size_thresh points after
// it), of the point that freezes it, how many points the walk adds before a
// frozen voxel stops it, and newly_add after it.  A build adds every point
// and refits once at the end (not listed here).
struct WalkPlan {
  int walk;      // points the walk adds
  int init_j;    // refit that initialises the voxel (-1: none)
  int per_j;     // first refit of the initialised voxel (kNever: none)
  int freeze_j;  // point that freezes the voxel (-1: none)
  int newly;     // newly_add after the walk
  bool stopped;  // the segment's rest reaches a frozen voxel
};
__device__ inline WalkPlan walk_plan(int n0, int newly0, uint32_t flags, int len, int upd, int mx, bool build) {
  WalkPlan p{len, -1, kNever, -1, newly0, false};
  if (build) return p;
  int js = 0;  // first walk index on the initialised path
  if (!(flags & kInit)) {
    const int ji = max(0, upd - n0 - 1);  // n reaches update_size_thresh
    if (ji >= len) return p;
    p.init_j = ji;
    js = ji + 1;
  }
  if (!(flags & kEnable)) {  // frozen once initialised
    p.walk = min(len, js);
    p.stopped = js < len;
    return p;
  }
  const int jf = max(js, mx - n0 - 1);  // n reaches max_point_thresh
  p.walk = min(len, jf + 1);
  p.stopped = jf + 1 < len;
  if (jf < len) p.freeze_j = jf;
  if (p.walk > js) {
    const int j1 = js + max(0, upd - 1 - newly0);
    if (j1 < p.walk) {
      p.per_j = j1;
      p.newly = (p.walk - 1 - j1) % upd;
    } else {
      p.newly = newly0 + (p.walk - js);
    }
  }
  return p;
}

// The voxels that refit in this scan replay their pending points and then their points of this scan in
// order through the pushPoint state machine, with FP64 moments and refits
// from them, in one of two forms that give the same bits:
//  - one wave per voxel (heavy_wave): lane c keeps moment c (lanes 0-4 also
//    moment 64 + c) and adds the points' terms in order from factors that
//    the wave stages in LDS 64 points at a time; at each refit point (known
//    from counts, walk_plan) it stores a snapshot of the moments, and up to
//    kSnap refits then run side by side, one per lane, applied in walk order.
//    The chain is a few memory round trips and one refit, whatever the
//    segment's length.
//  - one lane per voxel (heavy_lane): a walk per lane, the refits of the
//    wave's lanes taken together in rounds.  For steps with more than
//    wave_max refitting voxels, those whose segment has fewer than long_seg
//    points walk this way, so the FP64 refits run for 64 voxels at once.
constexpr int kHeavyChunk = 4;  // points of a heavy voxel's lane walk loaded together
constexpr int kLightChunk = 8;  // the same for the light walk
constexpr int kSnap = 16;       // refits evaluated together by heavy_wave
constexpr int kAccChunk = 8;    // points whose factors heavy_wave reads together
struct HeavyLds {
  double F[64][kMomF + 1];    // factors of 64 consecutive points of the walk (rows padded
                              // to an odd number of doubles: a lane per row, no bank conflicts)
  double snap[kSnap][kMomC];  // moments at refit points
  int snapn[kSnap];           // point count at each of those refits
};

__device__ inline double readlane_d(double v, int k) {
  const uint64_t u = uint64_t(__double_as_longlong(v));
  const uint32_t lo = uint32_t(__builtin_amdgcn_readlane(int(uint32_t(u)), k));
  const uint32_t hi = uint32_t(__builtin_amdgcn_readlane(int(uint32_t(u >> 32)), k));
  return __longlong_as_double((long long)(uint64_t(lo) | (uint64_t(hi) << 32)));
}

__device__ inline void write_hot_pl(const MapDev& m, int32_t vid, uint32_t flags, const double* pl, int64_t kx,
                                    int64_t ky, int64_t kz) {
  VoxHot h;
  h.mx = float(pl[0] - double(kx) * m.vs64);
  h.my = float(pl[1] - double(ky) * m.vs64);
  h.mz = float(pl[2] - double(kz) * m.vs64);
  h.flags = flags;
  h.nx = float(pl[3]);
  h.ny = float(pl[4]);
  h.nz = float(pl[5]);
  h.pad = 0.f;
  m.hot[vid] = h;
}

__device__ inline void heavy_lane(const MapDev& m, const SessInfo& S, const BatchBufs& b, int32_t vid, int start, int end,
                                  int& refits, int& calls, int& dropped) {
  if (vid >= 0) {
    VoxState st = m.vs[vid];
    double* pl = m.plane + size_t(vid) * kPlaneD;
    double* mo = m.mom + size_t(vid) * kMomD;
    double plv[kPlaneD];
    Moments M;
    const int cnt = st.n > 0 ? int(mo[kMomPend]) : 0;
    if (st.n > 0) {
      for (int k = 0; k < kPlaneD; ++k) plv[k] = pl[k];
    } else {  // a new voxel (its records were not cleared at creation)
      for (int k = 0; k < kPlaneD; ++k) plv[k] = 0.0;
    }
    if (st.n - cnt > 0) mom_load(mo, M);
    else mom_zero(M);  // no point has reached the moments yet
    if (cnt > m.pend_cap) atomicOr(&m.ctr->error, 32);
    const float* pd = m.pend + size_t(vid) * m.pend_cap * kPendF;
    const int npd = min(cnt, m.pend_cap);
    for (int k0 = 0; k0 < npd; k0 += kHeavyChunk) {  // a chunk of pending points loaded together
      float v[kHeavyChunk][kPendF];
#pragma unroll
      for (int u = 0; u < kHeavyChunk; ++u) {
        const int k = min(k0 + u, npd - 1);
#pragma unroll
        for (int a = 0; a < kPendF; ++a) v[u][a] = pd[k * kPendF + a];
      }
#pragma unroll
      for (int u = 0; u < kHeavyChunk; ++u)
        if (k0 + u < npd) mom_add(M, v[u], v[u] + 3);
    }
    int64_t kx, ky, kz;
    unpack_key(st.key, kx, ky, kz);
    const double center[3] = {(double(kx) + 0.5) * m.vs64, (double(ky) + 0.5) * m.vs64,
                              (double(kz) + 0.5) * m.vs64};
    uint32_t flags = st.flags;
    int n = st.n, newly = st.newly_add;
    int merge_pos = kNever, freeze_t = -1;
    // Points are replayed in rounds: each lane advances to its next refit
    // (or the end of its segment), then the lanes that reached one refit
    // together, so the wave runs the FP64 refit once per round instead of
    // whenever any lane needs it.  Per lane the order of operations is the
    // reference's: add the point, refit, then the freeze check.
    int pos = start;
    bool active = true;
    while (__any(active)) {
      bool need = false;
      while (active && !need) {
        // the next kHeavyChunk points of the segment, loaded together
        // (contiguous in key order); a refit ends the chunk early
        float4 qa[kHeavyChunk], qb[kHeavyChunk], qd[kHeavyChunk];
#pragma unroll
        for (int u = 0; u < kHeavyChunk; ++u) {
          const size_t p3 = 3 * size_t(min(pos + u, end - 1));
          qa[u] = b.qc[p3];
          qb[u] = b.qc[p3 + 1];
          qd[u] = b.qc[p3 + 2];
        }
#pragma unroll
        for (int u = 0; u < kHeavyChunk; ++u) {
          if (!active || need) break;
          if (pos >= end) {
            active = false;
            break;
          }
          if ((flags & kInit) && !(flags & kEnable) && !S.is_build) {
            if (flags & kPlane) {
              merge_pos = pos - start;
              calls += end - pos;
            } else {
              dropped += end - pos;
            }
            active = false;
            break;
          }
          const int i = __float_as_int(qa[u].w);
          ++pos;
          const float qv[3] = {qa[u].x, qa[u].y, qa[u].z};
          const float C[6] = {qb[u].x, qb[u].y, qb[u].z, qb[u].w, qd[u].x, qd[u].y};
          mom_add(M, qv, C);
          ++n;
          if (S.is_build) continue;
          if (!(flags & kInit)) {
            // updatePlane after every point until the voxel initialises
            need = n >= m.upd_pt;
            continue;
          }
          ++newly;
          if (newly >= m.upd_pt) {
            need = true;
            newly = 0;
          }
          if (n >= m.max_pt) {
            flags &= ~kEnable;
            freeze_t = i;
          }
        }
      }
      if (need) refit(m, M, n, flags, plv, center, refits);
    }
    if (S.is_build) refit(m, M, n, flags, plv, center, refits);
    const double invn = 1.0 / double(n);
    for (int a = 0; a < 3; ++a) plv[a] = fma(M.s1[a], invn, center[a]);
    mom_store(mo, M);
    for (int a = 0; a < 3; ++a) mo[kMomRun + a] = M.s1[a];
    mo[kMomPend] = 0.0;
    for (int k = 0; k < kPlaneD; ++k) pl[k] = plv[k];
    st.flags = flags;
    st.n = n;
    st.newly_add = newly;
    st.freeze_t = freeze_t;
    st.merge_pos = merge_pos;
    m.vs[vid] = st;
    write_hot(m, vid, flags);
  }
}

// The ks refits whose snapshots are in L, lane k evaluating the k-th, then
// applied in order to the wave-uniform flags and plane record.
__device__ inline void heavy_flush(const MapDev& m, HeavyLds& L, int ks, const double center[3], uint32_t& flags,
                                   double plv[kPlaneD]) {
  wave_lds_sync();
  const int lane = threadIdx.x & 63;
  RefitOut o{};
  // the snapshot rows have the layout of Moments: the refit reads them from LDS
  if (lane < ks) o = refit_eval(m, *reinterpret_cast<const Moments*>(L.snap[lane]), L.snapn[lane], center);
  wave_lds_sync();
  for (int k = 0; k < ks; ++k) {
    RefitOut r;
    r.plane = __builtin_amdgcn_readlane(int(o.plane), k) != 0;
    r.tn = readlane_d(o.tn, k);
    r.tm = readlane_d(o.tm, k);
    for (int a = 0; a < 3; ++a) r.nrm[a] = readlane_d(o.nrm[a], k);
    refit_apply(r, flags, plv);
  }
}

// One voxel on one wave; the counts go to lane 0's refits/calls/dropped.
__device__ inline void heavy_wave(const MapDev& m, bool build, const BatchBufs& b, int32_t vid, int start, int len,
                                  HeavyLds& L, int& refits, int& calls, int& dropped) {
  const int lane = threadIdx.x & 63;
  // segment point `lane` and pending point `lane`, loaded with the voxel's
  // state (before the pending count is known) for the first 64 rows
  float4 s0a = make_float4(0.f, 0.f, 0.f, 0.f), s0b = s0a, s0d = s0a;
  if (lane < len) {
    const size_t p3 = 3 * size_t(start + lane);
    s0a = b.qc[p3];
    s0b = b.qc[p3 + 1];
    s0d = b.qc[p3 + 2];
  }
  const float* pd = m.pend + size_t(vid) * m.pend_cap * kPendF;
  float pv0[kPendF];
  for (int a = 0; a < kPendF; ++a) pv0[a] = lane < m.pend_cap ? pd[lane * kPendF + a] : 0.f;
  const VoxState st = m.vs[vid];
  double* pl = m.plane + size_t(vid) * kPlaneD;
  double* mo = m.mom + size_t(vid) * kMomD;
  const int cnt = st.n > 0 ? int(mo[kMomPend]) : 0;
  if (cnt > m.pend_cap && lane == 0) atomicOr(&m.ctr->error, 32);
  const int npd = min(cnt, m.pend_cap);
  // lane c holds moment c and, on lanes 0-4, moment 64 + c
  const bool has_mom = st.n - cnt > 0;  // some point has reached the moments
  const int c2 = 64 + min(lane, kMomC - 65);
  double Ma = has_mom ? mo[lane] : 0.0;
  double Mb = has_mom ? mo[c2] : 0.0;
  const int ia1 = mom_i1(lane), ia2 = mom_i2(lane), ib1 = mom_i1(c2), ib2 = mom_i2(c2);
  double plv[kPlaneD];
  for (int k = 0; k < kPlaneD; ++k) plv[k] = st.n > 0 ? pl[k] : 0.0;  // a new voxel's record is not cleared
  int64_t kx, ky, kz;
  unpack_key(st.key, kx, ky, kz);
  const double center[3] = {(double(kx) + 0.5) * m.vs64, (double(ky) + 0.5) * m.vs64, (double(kz) + 0.5) * m.vs64};
  const WalkPlan P = walk_plan(st.n, st.newly_add, st.flags, len, m.upd_pt, m.max_pt, build);
  uint32_t flags = st.flags;
  // the pending points, then the walk's points of this scan, as rows of F
  // 64 at a time
  const int total = npd + P.walk;
  int next = P.init_j >= 0 ? P.init_j : P.per_j;  // walk index of the next refit
  int ks = 0, nref = 0;
  if (lane < npd) mom_factors(pv0, pv0 + 3, L.F[lane]);
  if (lane < P.walk && npd + lane < 64) {
    const float qv[3] = {s0a.x, s0a.y, s0a.z};
    const float C[6] = {s0b.x, s0b.y, s0b.z, s0b.w, s0d.x, s0d.y};
    mom_factors(qv, C, L.F[npd + lane]);
  }
  for (int p0 = 0; p0 < total; p0 += 64) {
    const int x = p0 + lane;
    if (p0 > 0 && x < total) {
      float qv[3], C[6];
      if (x < npd) {
        for (int a = 0; a < 3; ++a) qv[a] = pd[x * kPendF + a];
        for (int l = 0; l < 6; ++l) C[l] = pd[x * kPendF + 3 + l];
      } else {
        const size_t p3 = 3 * size_t(start + x - npd);
        const float4 qa = b.qc[p3], qb = b.qc[p3 + 1], qd = b.qc[p3 + 2];
        qv[0] = qa.x, qv[1] = qa.y, qv[2] = qa.z;
        C[0] = qb.x, C[1] = qb.y, C[2] = qb.z, C[3] = qb.w, C[4] = qd.x, C[5] = qd.y;
      }
      mom_factors(qv, C, L.F[lane]);
    }
    wave_lds_sync();
    const int np = min(64, total - p0);
    for (int t0 = 0; t0 < np; t0 += kAccChunk) {
      // the refits among the chunk's points must fit beside the snapshots held
      int nc = 0;
      for (int nx = next, j0 = p0 + t0 - npd; nx < j0 + kAccChunk && nx < P.walk;
           nx = nx == P.init_j ? P.per_j : nx + m.upd_pt)
        ++nc;
      if (ks + nc > kSnap) {
        heavy_flush(m, L, ks, center, flags, plv);
        ks = 0;
      }
      double fa[kAccChunk][2], fb[kAccChunk][2];  // the chunk's factors, read together
#pragma unroll
      for (int u = 0; u < kAccChunk; ++u) {
        const double* f = L.F[min(t0 + u, np - 1)];
        fa[u][0] = f[ia1];
        fa[u][1] = f[ia2];
        fb[u][0] = f[ib1];
        fb[u][1] = f[ib2];
      }
#pragma unroll
      for (int u = 0; u < kAccChunk; ++u) {
        if (t0 + u >= np) break;
        Ma = fma(fa[u][0], fa[u][1], Ma);
        Mb = fma(fb[u][0], fb[u][1], Mb);
        const int j = p0 + t0 + u - npd;
        if (j == next) {
          if (st.n + j + 1 >= m.upd_pt) {  // (the lane walk's refit() is a no-op below the threshold)
            L.snap[ks][lane] = Ma;
            if (lane < kMomC - 64) L.snap[ks][64 + lane] = Mb;
            L.snapn[ks] = st.n + j + 1;
            ++ks;
            ++nref;
          }
          next = j == P.init_j ? P.per_j : j + m.upd_pt;
        }
      }
    }
    wave_lds_sync();
  }
  if (ks == kSnap) {
    heavy_flush(m, L, ks, center, flags, plv);
    ks = 0;
  }
  const int n = st.n + P.walk;
  if (build && n >= m.upd_pt) {  // a build refits once with all the points
    L.snap[ks][lane] = Ma;
    if (lane < kMomC - 64) L.snap[ks][64 + lane] = Mb;
    L.snapn[ks] = n;
    ++ks;
    ++nref;
  }
  if (ks) heavy_flush(m, L, ks, center, flags, plv);
  const double invn = 1.0 / double(n);
  for (int a = 0; a < 3; ++a) plv[a] = fma(readlane_d(Ma, a), invn, center[a]);
  if (P.freeze_j >= 0) flags &= ~kEnable;
  int merge_pos = kNever;
  if (P.stopped) {
    if (flags & kPlane) {
      merge_pos = P.walk;
      if (lane == 0) calls += len - P.walk;
    } else if (lane == 0) {
      dropped += len - P.walk;
    }
  }
  const int freeze_t = P.freeze_j >= 0 ? __float_as_int(b.qc[3 * size_t(start + P.freeze_j)].w) : -1;
  mo[lane] = Ma;
  if (lane < kMomC - 64) mo[64 + lane] = Mb;
  if (lane < 3) mo[kMomRun + lane] = Ma;
  if (lane == 0) mo[kMomPend] = 0.0;
  double pv = plv[0];
  for (int k = 1; k < kPlaneD; ++k) pv = lane == k ? plv[k] : pv;
  if (lane < kPlaneD) pl[lane] = pv;
  if (lane == 0) {
    VoxState& vs = m.vs[vid];
    vs.flags = flags;
    vs.n = n;
    vs.newly_add = P.newly;
    vs.freeze_t = freeze_t;
    vs.merge_pos = merge_pos;
    write_hot_pl(m, vid, flags, plv, kx, ky, kz);
    refits += nref;
  }
}

// Orders a block's items by class, descending (n items per class counted in
// LDS, then placed by a scan), so that the lanes of a wave walk voxels with
// similar numbers of points; items of class 0 come last.  Returns the item
// that this thread takes.  An order over all segments took a histogram and a
// radix pass, 14 us.  The order decides nothing else, every voxel replays on
// its own.
struct SortLds {
  int cnt[kClsHeavy];
  int item[kMapThreads];
};
__device__ inline int block_order(uint32_t cls, SortLds& L) {
  const int tid = threadIdx.x;
  __syncthreads();
  if (tid < int(kClsHeavy)) L.cnt[tid] = 0;
  __syncthreads();
  const int k = int(kClsHeavy - 1 - cls);
  const int r = atomicAdd(&L.cnt[k], 1);
  __syncthreads();
  if (tid < 64) {
    const int c = L.cnt[tid];
    int incl = c;
    for (int o = 1; o < 64; o <<= 1) {
      const int u = __shfl_up(incl, o, 64);
      if (tid >= o) incl += u;
    }
    L.cnt[tid] = incl - c;
  }
  __syncthreads();
  L.item[L.cnt[k] + r] = tid;
  __syncthreads();
  return L.item[tid];
}

// The counts of a replay's voxels (refits, merge() calls, drops): summed in a
// block for a session alone, else added per wave and session.  With an atomic
// per voxel on the one counter those of 2,800 refits of a 120,000-point scan
// queued up for a third of the time of k_replay (55 us, 34 now).
__device__ inline void replay_count(const MapDev& m, int* lds, int refits, int calls, int dropped) {
  if (lds) {
    if (refits) atomicAdd(&lds[0], refits);
    if (calls) atomicAdd(&lds[1], calls);
    if (dropped) atomicAdd(&lds[2], dropped);
  } else {
    wave_fetch_add(&m.ctr->refits, refits);
    wave_fetch_add(&m.ctr->merge_calls, calls);
    wave_fetch_add(&m.ctr->dropped, dropped);
  }
}

// One wave per voxel of hlist: every refitting voxel when there are at most
// wave_max of them, else the long ones (cnt[6], at hlist's back).  A
// one-session step reads its map's record without waiting for the list.
__device__ inline void replay_waves(const MapDev* maps, const SessInfo* si, const BatchBufs& b, int wave_max,
                                    int block, int nblocks, HeavyLds* lds, int* cnt) {
  constexpr int kWpb = kMapThreads / 64;
  const int nh = b.cnt[5];
  const bool all = nh <= wave_max;
  const int nw = all ? nh : b.cnt[6];
  const int wv = threadIdx.x >> 6;
  const MapDev m0 = maps[0];
  const bool build0 = si[0].is_build != 0;
  for (int u = block * kWpb + wv; u < nw; u += nblocks * kWpb) {
    int refits = 0, calls = 0, dropped = 0;
    const int4 r = b.hlist[all ? u : b.ntot - 1 - u];
    MapDev m;
    bool build;
    if (b.nsess == 1) {
      m = m0;
      build = build0;
    } else {
      m = maps[r.w];
      build = si[r.w].is_build != 0;
    }
    heavy_wave(m, build, b, r.x, r.y, r.z, lds[wv], refits, calls, dropped);
    replay_count(m, cnt, refits, calls, dropped);
  }
}

// The rest of the refitting voxels, one per lane (a kernel of its own: the
// walk takes all the registers of a wave per SIMD, and together with
// heavy_wave it spilled).  Left out where a scan has no more than wave_max
// points.
__global__ void __launch_bounds__(kMapThreads)
k_replay_heavy(const MapDev* maps, const SessInfo* si, BatchBufs b, int wave_max, int long_seg) {
  __shared__ SortLds sort;
  const int nh = b.cnt[5];
  if (nh <= wave_max) return;
  for (int i0 = blockIdx.x * kMapThreads; i0 < nh; i0 += gridDim.x * kMapThreads) {
    const int i = i0 + int(threadIdx.x);
    int len = i < nh ? b.hlist[i].z : 0;
    if (long_seg > 0 && len >= long_seg) len = 0;  // replayed by a wave
    const int j = i0 + block_order(min(uint32_t(len), kClsHeavy - 1), sort);
    int4 r = j < nh ? b.hlist[j] : make_int4(-1, 0, 0, 0);
    if (long_seg > 0 && r.z >= long_seg) r.x = -1;
    int refits = 0, calls = 0, dropped = 0;
    const MapDev& m = maps[r.w];
    heavy_lane(m, si[r.w], b, r.x, r.y, r.y + r.z, refits, calls, dropped);
    wave_fetch_add(&m.ctr->refits, refits);
    wave_fetch_add(&m.ctr->merge_calls, calls);
    wave_fetch_add(&m.ctr->dropped, dropped);
  }
}

// The other voxels: frozen ones count their points as merge() calls or drops;
// the rest add points without reaching a refit, so only the count, the
// running mean and the freeze state change, and each point (relative to the
// voxel centre, with its world cov) joins the pending list that the voxel's
// next refit folds into the moments.
__device__ inline void replay_light(const MapDev* maps, const SessInfo* si, const BatchBufs& b, int block,
                                    int nblocks, SortLds& sort, int* cnt) {
  const int nseg = b.cnt[0];
  // a one-session step reads its map's record once, before the voxels
  const MapDev m0 = maps[0];
  const int build0 = si[0].is_build;
  for (int q0 = block * kMapThreads; q0 < nseg; q0 += nblocks * kMapThreads) {
    int calls = 0, dropped = 0;
    const uint32_t cls = q0 + int(threadIdx.x) < nseg ? b.seg_cls[q0 + threadIdx.x] : 0;
    const int q = min(q0 + block_order(cls >= kClsHeavy ? 0u : cls, sort), nseg - 1);
    const bool mine = q0 + sort.item[threadIdx.x] < nseg && b.seg_cls[q] < kClsHeavy;
    const int32_t vid = mine ? b.seg_vid[q] : -1;
    const int start = b.seg_start[q], end = b.seg_end[q];
    MapDev m;
    int s, is_build;
    if (b.nsess == 1) {
      s = 0;
      m = m0;
      is_build = build0;
    } else {
      s = mine ? b.seg_sess[q] : 0;
      m = maps[s];
      is_build = si[s].is_build;
    }
    VoxState st = m.vs[vid < 0 ? 0 : vid];
    const bool frozen0 = vid >= 0 && !is_build && (st.flags & kInit) && !(st.flags & kEnable);
    if (frozen0) {
      // frozen before this scan: every point is a merge() call (plane) or dropped
      const int len = end - start;
      if (st.flags & kPlane) {
        m.vs[vid].merge_pos = 0;
        calls += len;
      } else {
        dropped += len;
      }
    } else if (vid >= 0) {
      double* pl = m.plane + size_t(vid) * kPlaneD;
      double nrm[3];  // the plane's normal, kept (zero for a new voxel)
      for (int a = 0; a < 3; ++a) nrm[a] = st.n > 0 ? pl[3 + a] : 0.0;
      int64_t kx, ky, kz;
      unpack_key(st.key, kx, ky, kz);
      const double center[3] = {(double(kx) + 0.5) * m.vs64, (double(ky) + 0.5) * m.vs64,
                                (double(kz) + 0.5) * m.vs64};
      double* mo = m.mom + size_t(vid) * kMomD;
      double s1[3] = {0.0, 0.0, 0.0};
      int cnt = 0;
      if (st.n > 0) {
        for (int a = 0; a < 3; ++a) s1[a] = mo[kMomRun + a];
        cnt = int(mo[kMomPend]);
      }
      float* pd = m.pend + size_t(vid) * m.pend_cap * kPendF;
      uint32_t flags = st.flags;
      int n = st.n, newly = st.newly_add;
      int merge_pos = kNever, freeze_t = -1;
      bool walking = true;
      for (int p0 = start; p0 < end && walking; p0 += kLightChunk) {
       // a chunk of the segment's points loaded together (contiguous in key order)
       float4 qa[kLightChunk], qb[kLightChunk], qd[kLightChunk];
#pragma unroll
       for (int u = 0; u < kLightChunk; ++u) {
         const size_t p3 = 3 * size_t(min(p0 + u, end - 1));
         qa[u] = b.qc[p3];
         qb[u] = b.qc[p3 + 1];
         qd[u] = b.qc[p3 + 2];
       }
#pragma unroll
       for (int u = 0; u < kLightChunk; ++u) {
        const int pos = p0 + u;
        if (pos >= end || !walking) break;
        if ((flags & kInit) && !(flags & kEnable) && !is_build) {
          if (flags & kPlane) {
            merge_pos = pos - start;
            calls += end - pos;
          } else {
            dropped += end - pos;
          }
          walking = false;
          break;
        }
        const int i = __float_as_int(qa[u].w);
        const float qv[3] = {qa[u].x, qa[u].y, qa[u].z};
        const float C[6] = {qb[u].x, qb[u].y, qb[u].z, qb[u].w, qd[u].x, qd[u].y};
        if (cnt < m.pend_cap) {
          for (int a = 0; a < 3; ++a) pd[cnt * kPendF + a] = qv[a];
          for (int a = 0; a < 6; ++a) pd[cnt * kPendF + 3 + a] = C[a];
        } else {
          atomicOr(&m.ctr->error, 32);
        }
        ++cnt;
        for (int a = 0; a < 3; ++a) s1[a] += double(qv[a]);
        ++n;
        if (is_build) continue;
        if (!(flags & kInit)) {
          if (n >= m.upd_pt) atomicOr(&m.ctr->error, 32);  // a refit: the other kernel's voxel
          continue;
        }
        ++newly;
        if (newly >= m.upd_pt) atomicOr(&m.ctr->error, 32);
        if (n >= m.max_pt) {
          flags &= ~kEnable;
          freeze_t = i;
        }
       }
      }
      for (int a = 0; a < 3; ++a) mo[kMomRun + a] = s1[a];
      mo[kMomPend] = double(cnt);
      const double invn = 1.0 / double(n);
      double plv[6];
      for (int a = 0; a < 3; ++a) plv[a] = center[a] + s1[a] * invn;
      for (int a = 0; a < 3; ++a) plv[3 + a] = nrm[a];
      for (int a = 0; a < 3; ++a) pl[a] = plv[a];
      if (st.n == 0)  // a new voxel: its plane record was not cleared at creation
        for (int k = 3; k < kPlaneD; ++k) pl[k] = 0.0;
      st.flags = flags;
      st.n = n;
      st.newly_add = newly;
      st.freeze_t = freeze_t;
      st.merge_pos = merge_pos;
      m.vs[vid] = st;
      write_hot_pl(m, vid, flags, plv, kx, ky, kz);
    }
    replay_count(m, cnt, 0, calls, dropped);
  }
}

// Both in one launch: blocks below hblocks take refitting voxels, the others
// those that do not refit, so the light walks fill in where the long chains of the
// refits leave the card idle.
__global__ void __launch_bounds__(kMapThreads) __attribute__((amdgpu_waves_per_eu(2, 2)))
k_replay(const MapDev* maps, const SessInfo* si, BatchBufs b, int wave_max, int hblocks) {
  __shared__ HeavyLds lds[kMapThreads / 64];
  __shared__ SortLds sort;
  __shared__ int cnt[3];
  if (threadIdx.x < 3) cnt[threadIdx.x] = 0;
  __syncthreads();
  int* lc = b.nsess == 1 ? cnt : nullptr;
  if (int(blockIdx.x) < hblocks)
    replay_waves(maps, si, b, wave_max, blockIdx.x, hblocks, lds, lc);
  else
    replay_light(maps, si, b, int(blockIdx.x) - hblocks, int(gridDim.x) - hblocks, sort, lc);
  if (!lc) return;
  __syncthreads();
  MapCounters* c = maps[0].ctr;
  int* out[3] = {&c->refits, &c->merge_calls, &c->dropped};
  if (threadIdx.x < 3 && cnt[threadIdx.x]) atomicAdd(out[threadIdx.x], cnt[threadIdx.x]);
}

}  // namespace vmp

#include "vmp_merge.hpp"

namespace vmp {

// ------------------------------------------------------------------ K9 ----
// The scan's last fields of every touched voxel and the marks of their LRU
// appends, then (sessions that evict) the evicted voxels' slots: hash
// tombstones and the free list.
__global__ void k_finalize(const MapDev* maps, const SessInfo* si, int nsess, BatchBufs b, int evict) {
  const int nseg = b.cnt[0];
  VMP_GRID_LOOP(q, nseg) {
    const int32_t vid = b.seg_vid[q];
    const int s = b.seg_sess[q];
    const MapDev m = maps[s];
    const int last_t = b.sval_out[b.seg_end[q] - 1] - si[s].off;
    // LRU append marker (array cleared before); a segment left without a
    // voxel by an error appends an entry that no voxel's stamp can match
    b.flags[si[s].off + last_t] = vid < 0 ? -1 : vid + 1;
    if (vid < 0) continue;
    VoxState& st = m.vs[vid];
    const bool calls = st.merge_pos != kNever;
    const bool frozen_plane = (st.flags & kPlane) && !(st.flags & kEnable) && (st.flags & kInit);
    // a dirtying event is resolved by a later (evaluated) merge() call
    const bool dirty = frozen_plane && st.dirty_t > -2 && !(calls && last_t > st.dirty_t);
    if (dirty) st.flags |= kDirty;
    else st.flags &= ~kDirty;
    st.stamp = uint64_t(m.ctr->point_base + last_t);
  }
  if (!evict) return;
  VMP_GRID_LOOP(p, b.ntot) {
    const int s = sess_of(si, nsess, p);
    const MapDev m = maps[s];
    const MapCounters* c = m.ctr;
    const int r = p - si[s].off;
    if (r >= c->nevict) continue;
    const int32_t v = b.ev_vid[p];
    VoxState& st = m.vs[v];
    const int32_t e = hash_find_slot(m.table, m.hmask, st.key);
    if (e >= 0 && m.table[e].vid == v) {
      m.table[e].vid = -1;
      m.table[e].key = kKeyTomb;
    }
    st.flags = 0;
    m.hot[v].flags = 0;
    m.freelist[c->free_top + r] = v;
  }
}

// LRU queue append, as the output of the compaction of the marks: one entry
// per segment, so a session's first is its first segment's number.
struct OutLru {
  const MapDev* maps;
  const SessInfo* si;
  int nsess;
  __device__ void operator()(int r, int g, int32_t v) const {
    const int s = sess_of(si, nsess, g);
    const MapDev& m = maps[s];
    const int64_t ph = (m.ctr->ring_tail + (r - si[s].seg_lo)) % m.qcap;
    m.ring_vid[ph] = v < 0 ? 0 : v - 1;
    m.ring_stamp[ph] = v < 0 ? ~uint64_t(0) : uint64_t(m.ctr->point_base + (g - si[s].off));
  }
};
__global__ void k_lru_append(OutLru out, BatchBufs b) {
  const int nsel = b.cnt[2];
  VMP_GRID_LOOP(r, nsel) out(r, b.sel[r], b.flags[b.sel[r]]);
}

// ---------------------------------------------------- housekeeping -----
// Hash rebuild of the listed sessions (grid row y: session l.s[y] of the
// batch): a cleared table, then every live voxel of the pool inserted again.
// Two launches whatever the number of sessions, nothing read back.  Each
// block counts what it inserted and adds it once: with an atomic per voxel
// on the one counter the insertion of 200,000 voxels took 318 us, 32 us now.
constexpr int kMaintRows = 60;
struct MaintList {
  uint16_t s[kMaintRows];
};
__device__ inline void rehash_clear(const MapDev& m) {
  if (blockIdx.x == 0 && threadIdx.x == 0) m.ctr->used_entries = 0;
  for (uint32_t h = blockIdx.x * blockDim.x + threadIdx.x; h <= m.hmask; h += gridDim.x * blockDim.x) {
    m.table[h].key = kKeyEmpty;
    m.table[h].vid = -1;
  }
}
__global__ void k_hash_init(MapDev m) { rehash_clear(m); }
__global__ void k_rehash_clear(const MapDev* maps, MaintList l) { rehash_clear(maps[l.s[blockIdx.y]]); }
__global__ void __launch_bounds__(kMapThreads) k_rehash_insert(const MapDev* maps, MaintList l) {
  const MapDev m = maps[l.s[blockIdx.y]];
  int n = 0;
  VMP_GRID_LOOP(v, m.pool) {
    if (!(m.vs[v].flags & kAlive)) continue;
    int ins = 0;
    const int32_t e = hash_find_or_insert(m.table, m.hmask, m.vs[v].key, m.ctr, &ins);
    if (e >= 0) m.table[e].vid = v;
    n += ins;
  }
  __shared__ int sum;
  if (threadIdx.x == 0) sum = 0;
  __syncthreads();
  if (n) atomicAdd(&sum, n);
  __syncthreads();
  if (threadIdx.x == 0 && sum) atomicAdd(&m.ctr->used_entries, sum);
}

// LRU ring compaction.  An entry stays when its voxel is alive and still
// carries the entry's stamp (older entries of a re-touched voxel are stale).
// Pass 1 linearises the circular range [head, head + used) into tv/ts and
// flags the survivors; a stable select gives their positions; pass 2 writes
// them back to the front of the ring, so ascending stamp order is kept.
__global__ void k_ring_mark(MapDev m, int64_t head, int64_t used, int32_t* tv, uint64_t* ts, int32_t* keep) {
  for (int64_t r = int64_t(blockIdx.x) * blockDim.x + threadIdx.x; r < used; r += int64_t(gridDim.x) * blockDim.x) {
    const int64_t ph = (head + r) % m.qcap;
    const int32_t v = m.ring_vid[ph];
    const uint64_t s = m.ring_stamp[ph];
    tv[r] = v;
    ts[r] = s;
    keep[r] = (v >= 0 && v < m.pool && (m.vs[v].flags & kAlive) && m.vs[v].stamp == s) ? 1 : 0;
  }
}
__global__ void k_ring_scatter(MapDev m, const int32_t* tv, const uint64_t* ts, const int32_t* sel, const int32_t* cnt) {
  const int n = *cnt;
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    m.ctr->ring_head = 0;
    m.ctr->ring_tail = n;
  }
  VMP_GRID_LOOP(j, n) {
    const int32_t r = sel[j];
    m.ring_vid[j] = tv[r];
    m.ring_stamp[j] = ts[r];
  }
}

}  // namespace vmp
