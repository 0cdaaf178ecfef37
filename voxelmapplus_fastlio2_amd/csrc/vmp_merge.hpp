// Merge stages of the map update: VoxelGrid::merge (voxel_map.cpp:138-186)
// is called for every point that lands in a frozen plane voxel, reads the six
// face neighbours "at that moment" and may rewrite both planes and the
// neighbour's group id, so its calls are ordered by point index.
//
// Which calls can act:  a call is a no-op if the previous evaluated call on
// the same voxel was one and nothing in its closed neighbourhood changed
// since.  Changes are (a) a voxel freezing as a plane (known after the
// per-voxel replay) and (b) merges themselves.  Evictions only remove
// neighbours and new incarnations start unfrozen, so neither can turn an idle
// call into an acting one.
//   k_candidates   candidates = the first call after each (a)-event of the
//                  voxel or its neighbours, plus the first call of voxels
//                  still dirty from earlier scans; also caches each touched
//                  voxel's six neighbours and its candidate times
//   k_spec_eval    every candidate evaluated in parallel on the state before
//                  any merge of this scan: its eligible neighbours at its
//                  time (existence, incarnation, frozen-ness and plane-ness
//                  do not depend on merges) and whether it would merge
//   k_merge_replay one workgroup per session walks, in point order, the
//                  candidates that would merge plus the calls a real merge
//                  makes necessary: for every voxel whose closed
//                  neighbourhood a merge changed ("tainted"), its next call
//                  and all its later candidates, whose speculative result
//                  assumed the unchanged neighbourhood.
#pragma once

namespace vmp {

// incarnation of a key at point time t (-1: none)
__device__ inline int32_t vid_at(const MapDev& m, int32_t vid, int tag, int t) {
  if (vid < 0) return -1;
  const VoxState& st = m.vs[vid];
  if (st.tag == tag && st.create_t > t) vid = st.prev_vid;
  if (vid < 0) return -1;
  const VoxState& s2 = m.vs[vid];
  if (s2.tag == tag && s2.evict_t <= t) return -1;
  return vid;
}

// first merge() call of segment q strictly after local point t (kNever if none).
// The segment's point times ascend; the search narrows the range by sixteen
// independent samples per step (one memory round trip each) instead of a
// binary search's chain of dependent loads.
__device__ inline int first_call_in(const BatchBufs& b, int start, int end, int t, int off) {
  int lo = start, hi = end;  // answer in [lo, hi], hi = none
  const int tg = t + off;                          // compare global indices
  while (hi - lo > 16) {
    const int step = (hi - lo + 15) >> 4;
    int v[16];
#pragma unroll
    for (int k = 0; k < 16; ++k) v[k] = b.sval_out[min(lo + (k + 1) * step - 1, hi - 1)];
    int k = 0;
    while (k < 16 && v[k] <= tg) ++k;
    if (k == 16) return kNever;  // the last sample is hi - 1
    const int nhi = min(lo + (k + 1) * step - 1, hi - 1);
    lo = k == 0 ? lo : lo + k * step;
    hi = nhi;  // sval_out[nhi] > tg: the answer is at most nhi
    if (lo >= hi) return b.sval_out[hi] - off;
    ++hi;      // search [lo, nhi] inclusive as the half-open [lo, nhi + 1)
  }
  int v[16];
#pragma unroll
  for (int k = 0; k < 16; ++k) v[k] = lo + k < hi ? b.sval_out[lo + k] : 0x7fffffff;
  for (int k = 0; k < 16; ++k)
    if (lo + k < hi && v[k] > tg) return v[k] - off;
  return kNever;
}

__device__ inline int first_call_after(const BatchBufs& b, int q, int merge_pos, int t, int off) {
  return first_call_in(b, b.seg_start[q] + merge_pos, b.seg_end[q], t, off);
}

__device__ inline int32_t lookup_vid(const MapDev& m, uint64_t key) {
  const int32_t e = hash_find_slot(m.table, m.hmask, key);
  return e < 0 ? -1 : m.table[e].vid;
}

// neighbour j of a voxel if merge() may consider it at time t: it exists,
// is frozen (update_enable false), initialised and a plane; else -1
__device__ inline int32_t eligible_at(const MapDev& m, int32_t cur, int tag, int t) {
  const int32_t nv = vid_at(m, cur, tag, t);
  if (nv < 0) return -1;
  const VoxState& ns = m.vs[nv];
  const bool frozen = !(ns.flags & kEnable) && !(ns.tag == tag && ns.freeze_t > t);
  return (frozen && (ns.flags & kPlane) && (ns.flags & kInit)) ? nv : -1;
}
// A face neighbour of a voxel of this scan, as k_candidates leaves it in
// seg_nbr: (its current incarnation, -1 none; the point time from which it is
// eligible, kNever if at no time).  Nothing here depends on merges.  A
// neighbour that was evicted or that came back in this scan carries kNbrSlow:
// its state at a time is read from the records.
constexpr int32_t kNbrSlow = -2;
__device__ inline int32_t nbr_eligible(const MapDev& m, int2 nb, int tag, int t) {
  if (nb.x < 0) return -1;
  if (nb.y == kNbrSlow) return eligible_at(m, nb.x, tag, t);
  return t >= nb.y ? nb.x : -1;
}
__device__ inline int32_t nbr_at(const MapDev& m, uint64_t vkey, int j, int tag, int t) {
  if (!key_neighbour_ok(vkey, j)) return -1;
  return eligible_at(m, lookup_vid(m, key_neighbour(vkey, j)), tag, t);
}

// The six face neighbours' voxel ids (-1: none), as lookup_vid gives them;
// the six home-slot entries are loaded together, then the next probes of the
// neighbours that collided, together again.
__device__ inline void lookup_nbrs6(const MapDev& m, uint64_t vkey, int32_t nv[6]) {
  uint64_t nk[6];
  HashSeq q[6];
  HashEntry e[6];
#pragma unroll
  for (int j = 0; j < 6; ++j) {
    nk[j] = key_neighbour_ok(vkey, j) ? key_neighbour(vkey, j) : kKeyEmpty;
    q[j] = hash_seq(nk[j]);
    e[j] = m.table[hash_home(q[j], m.hmask)];
    nv[j] = -1;
  }
  uint32_t open = 0;  // neighbours whose sequence goes on
#pragma unroll
  for (int j = 0; j < 6; ++j) {
    if (nk[j] == kKeyEmpty) continue;
    if (e[j].key == nk[j]) nv[j] = e[j].vid;
    else if (e[j].key != kKeyEmpty) open |= 1u << j;
  }
  for (uint32_t probe = 1; open != 0 && probe <= m.hmask; ++probe) {
#pragma unroll
    for (int j = 0; j < 6; ++j)
      if (open & (1u << j)) e[j] = m.table[hash_probe(q[j], probe, m.hmask)];
#pragma unroll
    for (int j = 0; j < 6; ++j) {
      if (!(open & (1u << j))) continue;
      if (e[j].key == nk[j]) nv[j] = e[j].vid;
      if (e[j].key == nk[j] || e[j].key == kKeyEmpty) open &= ~(1u << j);
    }
  }
}

// eligible_at for six voxel ids, their records read in three rounds of six
// loads (the incarnation's creation fields, then the eligibility fields of
// the incarnation at time t) instead of a chain per neighbour
__device__ inline void eligible6(const MapDev& m, const int32_t cur[6], int tag, int t, int32_t out[6]) {
  int32_t v[6];
#pragma unroll
  for (int j = 0; j < 6; ++j) {
    const VoxState& r = m.vs[cur[j] < 0 ? 0 : cur[j]];
    const int rt = r.tag, ct = r.create_t, pv = r.prev_vid;
    v[j] = cur[j] < 0 ? -1 : ((rt == tag && ct > t) ? pv : cur[j]);
  }
#pragma unroll
  for (int j = 0; j < 6; ++j) {
    const VoxState& r = m.vs[v[j] < 0 ? 0 : v[j]];
    const int rt = r.tag, ev = r.evict_t, fz = r.freeze_t;
    const uint32_t fl = r.flags;
    const bool gone = v[j] < 0 || (rt == tag && ev <= t);
    const bool frozen = !(fl & kEnable) && !(rt == tag && fz > t);
    out[j] = (!gone && frozen && (fl & kPlane) && (fl & kInit)) ? v[j] : -1;
  }
}

// angle and distance gates (voxel_map.cpp:147-155); planes as kPlaneD records
__device__ inline bool merge_gate(const double* pv, const double* pn, double ma, double md) {
  double dn = pn[3] * pv[3];
  dn += pn[4] * pv[4];
  dn += pn[5] * pv[5];
  const double norm_distance = 1.0 - dn;
  double a1 = pn[3] * pn[0];
  a1 += pn[4] * pn[1];
  a1 += pn[5] * pn[2];
  double a0 = pv[3] * pv[0];
  a0 += pv[4] * pv[1];
  a0 += pv[5] * pv[2];
  const double axis_distance = fabs(a1 - a0);
  return !(norm_distance > ma || axis_distance > md);
}

// trace-weighted fusion (voxel_map.cpp:157-183), written to both records.
// Operator precedence as in the reference: new_mean = tm0*m_n + (tm1*m_v)/(tm0+tm1)
// and likewise for the normal, which is not re-normalised.
__device__ inline void merge_fuse(double* pv, double* pn) {
  const double tn0 = pv[6], tm0 = pv[7], tn1 = pn[6], tm1 = pn[7];
  const double tc0 = tn0 + tm0, tc1 = tn1 + tm1;
  double nm[3], nrm[3];
  for (int k = 0; k < 3; ++k) {
    nm[k] = tm0 * pn[k] + (tm1 * pv[k]) / (tm0 + tm1);
    nrm[k] = tn0 * pn[3 + k] + (tn1 * pv[3 + k]) / (tn0 + tn1);
  }
  const double den = (tc0 + tc1) * (tc0 + tc1);
  const double ntn = (tc0 * tc0 * tn1 + tc1 * tc1 * tn0) / den;
  const double ntm = (tc0 * tc0 * tm1 + tc1 * tc1 * tm0) / den;
  double dd = nm[0] * nrm[0];
  dd += nm[1] * nrm[1];
  dd += nm[2] * nrm[2];
  if (-dd < 0.0)
    for (int k = 0; k < 3; ++k) nrm[k] = -nrm[k];
  for (int k = 0; k < 3; ++k) {
    pv[k] = nm[k];
    pv[3 + k] = nrm[k];
    pn[k] = nm[k];
    pn[3 + k] = nrm[k];
  }
  pv[6] = pn[6] = ntn;
  pv[7] = pn[7] = ntm;
}

// ------------------------------------------------------------------ K7 ----
// Eight lanes per touched voxel: lane j < 6 its face neighbour j (id, record,
// and the first call after the neighbour's freezing), lane 6 its own freezing
// and carried dirty mark; the distinct call times are then sorted within the
// eight lanes.  Bound by the chain of round trips of one lane; with a lane per
// voxel the searches of up to seven call times ran one after the other
// (22 us at 120,000 points, 13 now).
constexpr int kCandLanes = 8;
__global__ void __launch_bounds__(kMapThreads) k_candidates(const MapDev* maps, const SessInfo* si, BatchBufs b) {
  const int nseg = b.cnt[0];
  const MapDev m0 = maps[0];  // a one-session step reads its map's record once
  __shared__ int cands;       // and adds its candidates once per block
  if (threadIdx.x == 0) cands = 0;
  __syncthreads();
  constexpr int kPer = kMapThreads / kCandLanes;
  const int j = threadIdx.x % kCandLanes, lane = threadIdx.x & 63, g0 = lane & ~(kCandLanes - 1);
  for (int q0 = blockIdx.x * kPer; q0 < nseg; q0 += gridDim.x * kPer) {
    const int q = q0 + int(threadIdx.x) / kCandLanes;
    const bool valid = q < nseg;
    const int32_t vid = valid ? b.seg_vid[q] : -1;
    const int s = b.nsess == 1 || !valid ? 0 : b.seg_sess[q];
    MapDev m;
    if (b.nsess == 1) m = m0;
    else m = maps[s];
    MapCounters* c = m.ctr;
    constexpr int kNone = -2;
    int after = kNone;  // a candidate is the first call after this time
    int dirty = -2, call = kNever;
    int2 nb = make_int2(-1, kNever);
    if (vid >= 0) {
      const int tag = c->tag, off = si[s].off;
      VoxState& st = m.vs[vid];
      const int start = b.seg_start[q], end = b.seg_end[q];
      const uint32_t flags = st.flags;
      const int freeze_t = st.freeze_t, merge_pos = st.merge_pos;
      const bool own_freeze = freeze_t >= 0 && (flags & kPlane);
      if (j == 6) {
        dirty = (flags & kDirty) ? -1 : -2;
        if (own_freeze) dirty = freeze_t;
        if ((flags & kDirty) || own_freeze) after = -1;
      } else if (j < 6 && key_neighbour_ok(st.key, j)) {
        const int32_t nv = lookup_vid(m, key_neighbour(st.key, j));
        if (nv >= 0) {
          const VoxState& ns = m.vs[nv];
          const int ntag = ns.tag, nfrz = ns.freeze_t, ncre = ns.create_t, nevt = ns.evict_t, nprv = ns.prev_vid;
          const uint32_t nflg = ns.flags;
          const bool cur = ntag == tag;
          const bool frozen_plane = !(nflg & kEnable) && (nflg & kPlane) && (nflg & kInit);
          nb = make_int2(nv, frozen_plane ? (cur ? max(ncre, nfrz) : -1) : kNever);
          if (cur && (nevt != kNever || nprv >= 0)) nb.y = kNbrSlow;
          if (cur && nfrz >= 0 && (nflg & kPlane)) dirty = after = nfrz;
          // a frozen plane marks its untouched live neighbours dirty for later
          // scans (only their kDirty bit changes: this kernel reads kPlane and
          // kAlive of neighbours, and the own flags of touched voxels only)
          if (own_freeze && !cur && (nflg & kAlive)) atomicOr(&m.vs[nv].flags, kDirty);
        }
      }
      if (after != kNone && merge_pos != kNever) call = first_call_in(b, start + merge_pos, end, after, off);
    }
    if (valid && j < 6) b.seg_nbr[q * 6 + j] = nb;
    // one candidate per distinct call, ascending
    int tv[kCandLanes];
#pragma unroll
    for (int o = 0; o < kCandLanes; ++o) tv[o] = __shfl(call, g0 + o, 64);
    bool emits = call != kNever;
#pragma unroll
    for (int o = 0; o < kCandLanes; ++o) emits &= !(o < j && tv[o] == call);
    const uint64_t all = __ballot(emits);
    const uint32_t em = uint32_t(all >> g0) & ((1u << kCandLanes) - 1u);
    int pos = 0;
#pragma unroll
    for (int o = 0; o < kCandLanes; ++o) pos += ((em >> o) & 1u) && tv[o] < call ? 1 : 0;
#pragma unroll
    for (int o = 1; o < kCandLanes; o <<= 1) dirty = max(dirty, __shfl_xor(dirty, o, 64));
    if (valid && j == 0) b.seg_nct[q] = __popc(em);
    if (vid >= 0 && j == 6) m.vs[vid].dirty_t = dirty;
    // the session's candidate count; each candidate goes to its session's
    // offset plus its point time (a call time belongs to one voxel), so the
    // filled slots are in sorted order
    if (b.nsess > 1) wave_fetch_add(&c->ncand, emits ? 1 : 0);
    else if (lane == 0 && all) atomicAdd(&cands, __popcll(all));
    if (emits) {
      const int off = si[s].off;
      if (call < si[s].n) b.cand_in[off + call] = cand_key_batch(s, call, vid, b.cand_sshift);
      else atomicOr(&c->error, 16);
      b.seg_ct[q * 7 + pos] = call;
    }
  }
  __syncthreads();
  if (threadIdx.x == 0 && cands) atomicAdd(&m0.ctr->ncand, cands);
}

// ------------------------------------------------------------------ K8 ----
// The call at point time t is made by the voxel that received point t and its
// candidate sits at its session's offset plus t, so the filled slots in order
// are the candidates sorted on (session, time).  A tile's candidates are
// packed in LDS, evaluated a thread each, and the acting ones compacted over
// the tiles (one launch; two compactions with the evaluation between them took
// 15 us on a 2,003-point scan, 22 on 20,000 points, 27 on 120,000): spl[k]
// and cand_out[k] are the k-th acting candidate's record (its eligible
// neighbours, cand_nbr) and key.  The last tile sets the sessions' ranges.
__device__ inline int spec_eval(const MapDev& m, const BatchBufs& b, uint64_t local, int tag, int32_t nv[6]) {
  const int t = cand_t(local);
  const int32_t V = cand_vid(local);
  const VoxState& vst = m.vs[V];
  const uint64_t gV = vst.group_id;
  double pv[kPlaneD];
  for (int k = 0; k < kPlaneD; ++k) pv[k] = m.plane[size_t(V) * kPlaneD + k];
  // the six neighbours (cached ids of a voxel touched in this scan, else
  // looked up), their eligibility at t, then the gate, each step with the
  // six neighbours' loads together
  if (vst.tag == tag && vst.seg >= 0) {
    int2 nb[6];
#pragma unroll
    for (int j = 0; j < 6; ++j) nb[j] = b.seg_nbr[vst.seg * 6 + j];
#pragma unroll
    for (int j = 0; j < 6; ++j) nv[j] = nbr_eligible(m, nb[j], tag, t);
  } else {
    int32_t nc[6];
    lookup_nbrs6(m, vst.key, nc);
    eligible6(m, nc, tag, t, nv);
  }
  int spec = 0;
#pragma unroll
  for (int j = 0; j < 6; ++j)
    if (nv[j] >= 0 && m.vs[nv[j]].group_id != gV &&
        merge_gate(pv, m.plane + size_t(nv[j]) * kPlaneD, m.merge_a, m.merge_d))
      spec = 1;
  return spec;
}
__global__ void __launch_bounds__(kPrimThreads) k_spec_eval(const MapDev* maps, SessInfo* si, BatchBufs b, PrimWs ws) {
  using Scan = rocprim::block_scan<int32_t, kPrimThreads>;
  __shared__ typename Scan::storage_type st;
  __shared__ uint64_t ck[kPrimTile];
  constexpr int kWords = kPrimTile / 64;
  static_assert(kWords <= 64, "the acting bits' scan runs in one wave");
  __shared__ uint64_t abits[kWords];
  __shared__ int apre[kWords];
  __shared__ int s_tile, s_last;
  __shared__ uint32_t s_prefix;
  const int nt = gridDim.x, n = b.ntot, lane = threadIdx.x & 63;
  if (threadIdx.x == 0) s_tile = take_ticket(ws.ctl, nt);
  if (threadIdx.x < kWords) abits[threadIdx.x] = 0;
  __syncthreads();
  const int tile = s_tile, tile0 = tile * kPrimTile;
  const int base = tile0 + threadIdx.x * kPrimIpt;
  uint64_t v[kPrimIpt];
  int32_t c = 0, pos = 0, cnt = 0;
#pragma unroll
  for (int k = 0; k < kPrimIpt; ++k) {
    v[k] = base + k < n ? b.cand_in[base + k] : ~uint64_t(0);
    c += v[k] != ~uint64_t(0) ? 1 : 0;
  }
  Scan().exclusive_scan(c, pos, 0, cnt, st);
#pragma unroll
  for (int k = 0; k < kPrimIpt; ++k)
    if (v[k] != ~uint64_t(0)) ck[pos++] = v[k];
  __syncthreads();
  for (int i0 = 0; i0 < cnt; i0 += kPrimThreads) {
    const int i = i0 + int(threadIdx.x);
    int spec = 0;
    if (i < cnt) {
      const int s = int(ck[i] >> b.cand_sshift);
      const MapDev m = maps[s];
      int32_t nv[6];
      spec = spec_eval(m, b, cand_local(ck[i], b.cand_sshift), m.ctr->tag, nv);
      if (spec)
        for (int j = 0; j < 6; ++j) b.cand_nbr[size_t(tile0 + i) * 6 + j] = nv[j];
    }
    const uint64_t bal = __ballot(spec);
    if (lane == 0) abits[(i0 + int(threadIdx.x)) >> 6] = bal;
  }
  __syncthreads();
  if (threadIdx.x < 64) {
    const int x = lane < kWords ? __popcll(abits[min(lane, kWords - 1)]) : 0;
    int incl = x;
    for (int o = 1; o < 64; o <<= 1) {
      const int u = __shfl_up(incl, o, 64);
      if (lane >= o) incl += u;
    }
    if (lane < kWords) apre[lane] = incl - x;
    const uint32_t agg = uint32_t(__shfl(incl, 63, 64));
    uint32_t prefix = 0;
    if (tile > 0) {
      if (lane == 0) st_store(ws.status + tile, kStAgg | agg);
      prefix = look_back_wave(ws.status, tile, ws.ctl);
    }
    if (lane == 0) {
      st_store(ws.status + tile, kStInc | (prefix + agg));
      s_prefix = prefix;
      if (tile == nt - 1) b.cnt[4] = int32_t(prefix + agg);
    }
  }
  __syncthreads();
  for (int i = threadIdx.x; i < cnt; i += kPrimThreads) {
    const uint64_t w = abits[i >> 6];
    if (!((w >> (i & 63)) & 1)) continue;
    const int k = int(s_prefix) + apre[i >> 6] + __popcll(w & bits_below(i & 63));
    b.spl[k] = tile0 + i;
    b.cand_out[k] = ck[i];
  }
  if (!finish_tile(ws.ctl, nt, ws.status, nt, nullptr, 0, &s_last, true)) return;
  // the sessions' ranges: each starts behind the last key of an earlier one.
  // A thread sets those of the sessions between two keys; where they are many
  // (sessions without a candidate), all threads do, gap after gap: 2,048
  // sessions without one took a single thread 104 us.
  constexpr int kWalk = 16;
  static_assert(kMaxBatchSessions <= 1 << 15 && kMaxBatchSessions / kWalk <= kPrimTile, "gaps fit in ck");
  __shared__ int s_gaps;
  if (threadIdx.x == 0) s_gaps = 0;
  __syncthreads();
  const int na = b.cnt[4];
  auto set = [&](int s, int k) {
    si[s].spl_lo = k;
    if (s > 0) si[s - 1].spl_hi = k;
  };
  for (int k = threadIdx.x; k <= na; k += kPrimThreads) {
    const int s0 = k == 0 ? 0 : int(b.cand_out[k - 1] >> b.cand_sshift) + 1;
    const int s1 = k == na ? b.nsess - 1 : int(b.cand_out[k] >> b.cand_sshift);
    if (s1 - s0 < kWalk) {
      for (int s = s0; s <= s1; ++s) set(s, k);
    } else {
      ck[atomicAdd(&s_gaps, 1)] = (uint64_t(k) << 30) | (uint64_t(s0) << 15) | uint64_t(s1);
    }
    if (k == na) si[b.nsess - 1].spl_hi = na;
  }
  __syncthreads();
  for (int i = 0; i < s_gaps; ++i) {
    const uint64_t g = ck[i];
    for (int s = int(g >> 15 & 0x7fff) + int(threadIdx.x); s <= int(g & 0x7fff); s += kPrimThreads) set(s, int(g >> 30));
  }
}

// The merge-independent part of the taint phase of every acting candidate,
// in parallel ahead of the replay (see BatchBufs::pre_x).
constexpr int kPreItems = 49;  // 7 records x (6 neighbours + itself)
__global__ void k_spl_prefetch(const MapDev* maps, const SessInfo* si, BatchBufs b) {
  const int npre = min(b.cnt[4], b.pre_cap);
  VMP_GRID_LOOP(it, npre * kPreItems) {
    const int k = it / kPreItems, r = it % kPreItems, cj = r / 7, j = r % 7;
    const int pos = b.spl[k];
    const uint64_t cur = b.cand_out[k];
    const int s = int(cur >> b.cand_sshift);
    const MapDev m = maps[s];
    const int tag = m.ctr->tag, off = si[s].off;
    const int t = cand_t(cand_local(cur, b.cand_sshift));
    const int32_t base = cj == 6 ? cand_vid(cur) : b.cand_nbr[size_t(pos) * 6 + cj];
    int32_t X = -1;
    bool simple = false;  // its record alone says whether it exists at t
    if (base >= 0) {
      if (j == 6) {
        X = base;
      } else {
        const VoxState& bs = m.vs[base];
        if (bs.tag == tag && bs.seg >= 0) {
          const int2 nb = b.seg_nbr[bs.seg * 6 + j];
          simple = nb.y != kNbrSlow;
          X = simple ? nb.x : vid_at(m, nb.x, tag, t);
        } else if (key_neighbour_ok(bs.key, j)) {
          X = vid_at(m, lookup_vid(m, key_neighbour(bs.key, j)), tag, t);
        }
      }
    }
    int xseg = -1, tn = kNever;
    if (simple && X >= 0 && m.vs[X].tag == tag && m.vs[X].create_t > t) X = -1;
    if (X >= 0) {
      const VoxState& xs = m.vs[X];
      if (xs.tag == tag && xs.seg >= 0 && xs.evict_t == kNever) {
        xseg = xs.seg;
        if (xs.merge_pos != kNever) tn = first_call_after(b, xs.seg, xs.merge_pos, t, off);
      }
    }
    b.pre_x[it] = X;
    b.pre_seg[it] = xseg;
    b.pre_tn[it] = tn;
  }
}

constexpr int kMrWaves = 8;      // waves of one session's merge replay: acting entries evaluated per window
constexpr int kMrThreads = 64 * kMrWaves;
constexpr int kWin = 36;         // window entries (36 x 7 records <= 512 threads)
constexpr int kSPre = 2 * kWin;  // static candidates and pool entries merged per window
constexpr int kStat = 1024;      // static candidates held in LDS
constexpr int kPoolCap = 2048;   // pending re-evaluations, kept sorted
constexpr int kTaintPer = 49;    // up to 7 changed voxels x their closed neighbourhood
constexpr int kKeysPer = 8;      // keys a tainted voxel can give: its next call and its candidates
constexpr int kNewCap = kMrWaves * kTaintPer * kKeysPer;  // keys one window's commits can create
constexpr int kPlS = kPlaneD + 1;  // doubles per plane record in LDS (odd: a lane per record, no bank conflicts)
static_assert(kWin * 7 <= kMrThreads, "one thread per window record");
static_assert(kWin <= 64, "window bookkeeping runs in one wave");
static_assert(kTaintPer <= 64, "an acting entry's taint phase takes a lane per item");
static_assert(128 + kSPre <= kMrThreads && 2 * kSPre <= 3 * 64, "the window's merge");

__device__ inline int rank_lt(const uint64_t* a, int n, uint64_t v) {  // elements < v
  int lo = 0, hi = n;
  while (lo < hi) {
    const int mid = (lo + hi) >> 1;
    if (a[mid] < v) lo = mid + 1;
    else hi = mid;
  }
  return lo;
}
__device__ inline int rank_le(const uint64_t* a, int n, uint64_t v) {  // elements <= v
  int lo = 0, hi = n;
  while (lo < hi) {
    const int mid = (lo + hi) >> 1;
    if (a[mid] <= v) lo = mid + 1;
    else hi = mid;
  }
  return lo;
}

// One workgroup per session replays, in point order, the merge() calls that
// act.  Windowed speculation with in-order commit:
//   fill     the next kWin keys of the static list (acting candidates) merged
//            with the sorted pool of re-evaluations, duplicates dropped;
//   records  each entry's voxel and six eligible neighbours (group, plane);
//   gates    every entry's six gates in parallel: an entry acts if one passes;
//   act      the first kMrWaves acting entries, a wave each: the merge() on a
//            copy of the current state and, a lane per item, the
//            re-evaluations its merges make necessary (new keys and the
//            voxels' dirty marks, held in registers until it commits);
//   commit   in point order.  An entry whose records, or (if it acts) the
//            records its taint phase read, were changed by an earlier entry
//            of the window, or that a new key must precede, or that acts and
//            got no wave, stops the commit: it and every later entry return
//            to the pool.
// A committed entry therefore saw exactly the state the serial order gives
// it, and its taint phase read the same records a serial one would.
//
// Bound by the chain of a window: a merge's re-evaluations mostly come before
// the rest of the window, so a window commits 2 to 3 acting entries (of some
// 20) and a scan with 30 merges takes about 15.  Hence eight barriers a
// window, the window's merge in one wave, the statics in LDS, and the taint
// phase's loads beside the merge's arithmetic: 11 us a window (15.5 with a
// lane per entry for the merges, twenty barriers and a hash of first writers),
// of which the acting waves' loads (three to five round trips) take 4.5.
__global__ void __launch_bounds__(kMrThreads) k_merge_replay(const MapDev* maps, const SessInfo* si, int nsess,
                                                             BatchBufs b) {
  const int s = blockIdx.x;
  if (s >= nsess) return;
  const MapDev m = maps[s];
  MapCounters* c = m.ctr;
  const int tag = c->tag, off = si[s].off;
  const int spl_hi = si[s].spl_hi;
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
  __shared__ uint64_t pool[2][kPoolCap];
  __shared__ uint64_t skey[kStat];  // statics from sbase on
  __shared__ int spos[kStat];
  __shared__ uint64_t wkey[kWin];
  __shared__ int wpos[kWin];
  __shared__ int wspl[kWin];  // index of a static entry in spl (-1: pool entry)
  __shared__ double pl[kWin][7][kPlS];
  __shared__ uint64_t grp[kWin][7];
  __shared__ int32_t nbv[kWin][7];
  __shared__ int32_t rseg[kWin][7];  // record voxels: segment of this scan (-1 none), key, flags
  __shared__ uint64_t rkey[kWin][7];
  __shared__ uint32_t rflg[kWin][7];
  __shared__ int gates[kWin];        // gates passed on the window's state (bit j)
  __shared__ int conf[kWin];
  __shared__ uint64_t minkey[kMrWaves];  // first new key of the waves' entries
  __shared__ int actw[kMrWaves];     // the waves' entries (kWin: none)
  __shared__ int clos[kMrWaves];     // their changed records (bit j)
  __shared__ int2 wr[kMrWaves * 7];  // the voxels they change, with the entry
  __shared__ uint64_t gbuf[kNewCap + kWin];
  __shared__ uint64_t mk[2 * kSPre];  // fill: statics and pool entries merged
  __shared__ int mspl[2 * kSPre];
  __shared__ int sh_i[5];
  int sp = si[s].spl_lo, sbase = sp, pb = 0, ph = 0, pn = 0;
  int evals = 0, merges = 0, windows = 0, requeued = 0, max_acting = 0, err = 0;
  uint64_t last = ~0ull;
  for (int k = tid; k < min(kStat, spl_hi - sbase); k += kMrThreads) {
    skey[k] = cand_local(b.cand_out[sbase + k], b.cand_sshift);
    spos[k] = b.spl[sbase + k];
  }
  __syncthreads();
  while (true) {
    // ---- fill the window: the next statics and pool entries merged in
    //      parallel (merge path; statics first on equal keys), duplicates and
    //      keys beyond what is taken in dropped, the first kWin taken
    const int ns = min(kSPre, spl_hi - sp), np = min(kSPre, pn - ph);
    if (sp + ns > sbase + kStat) {
      sbase = sp;
      for (int k = tid; k < min(kStat, spl_hi - sbase); k += kMrThreads) {
        skey[k] = cand_local(b.cand_out[sbase + k], b.cand_sshift);
        spos[k] = b.spl[sbase + k];
      }
      __syncthreads();
    }
    const uint64_t* sseg = skey + (sp - sbase);
    const uint64_t* pseg = &pool[pb][ph];
    const int M = ns + np;
    if (tid < ns) {
      const int p = tid + rank_lt(pseg, np, sseg[tid]);
      mk[p] = sseg[tid];
      mspl[p] = sp + tid;
    } else if (tid >= 128 && tid - 128 < np) {
      const int j = tid - 128;
      const int p = j + rank_le(sseg, ns, pseg[j]);
      mk[p] = pseg[j];
      mspl[p] = -1;
    }
    __syncthreads();
    // valid: not over the limit, not a duplicate of the previous key; one
    // wave, three positions a lane
    if (wv == 0) {
      uint64_t lim = ~0ull;  // keys above a static or pool entry left out wait
      if (spl_hi - sp > kSPre) lim = sseg[ns - 1];
      if (pn - ph > kSPre && pseg[np - 1] < lim) lim = pseg[np - 1];
      int total = 0, statics = 0, cut = M, used = 0;
      bool full = false;
#pragma unroll
      for (int q = 0; q < 3; ++q) {
        const int p = 64 * q + lane;
        const bool in = p < M;
        const uint64_t key = in ? mk[p] : ~0ull;
        const bool over = in && key > lim;
        const bool ok = in && !over && key != (p == 0 ? last : mk[p - 1]);
        const bool stat = in && !over && mspl[p] >= 0;
        const uint64_t bok = __ballot(ok), bst = __ballot(stat), bov = __ballot(over);
        const int pre = total + __popcll(bok & bits_below(lane));
        if (ok && pre < kWin) {
          wkey[pre] = key;
          wspl[pre] = mspl[p];
          wpos[pre] = mspl[p] >= 0 ? spos[mspl[p] - sbase] : -1;
        }
        const uint64_t bend = __ballot(ok && pre == kWin - 1);  // the kWin-th taken key ends the range
        if (bend) {
          const int e = __ffsll((unsigned long long)bend) - 1;
          full = true;
          cut = 64 * q + e + 1;
          used = statics + __popcll(bst & (bits_below(e) | (1ull << e)));
        }
        if (bov && !full && cut == M) cut = 64 * q + __ffsll((unsigned long long)bov) - 1;
        total += __popcll(bok);
        statics += __popcll(bst);
      }
      if (!full) used = statics;  // statics counted only below the limit
      if (lane < kWin) {
        gates[lane] = 0;
        conf[lane] = 0;
      }
      if (lane < kMrWaves) minkey[lane] = ~0ull;
      if (lane == 0) {
        sh_i[0] = total < kWin ? total : kWin;
        sh_i[1] = used;
        sh_i[2] = cut;
        sh_i[3] = 0;  // keys for the pool
        sh_i[4] = 0;  // changed voxels
      }
    }
    __syncthreads();
    const int n = sh_i[0], used = sh_i[1], cut = sh_i[2];
    sp += used;
    ph += cut - used;
    if (n == 0) {
      if (cut == 0) break;  // nothing left
      __syncthreads();      // (sh_i is read before the next fill writes it)
      continue;             // only duplicates of the last key were taken in
    }
    ++windows;
    // ---- records: thread w*7+j, j = 6 is the voxel itself
    const int rw = tid / 7, rj = tid - 7 * rw;
    int32_t rv = -1;
    double rp[kPlaneD];
    if (tid < n * 7) {
      const uint64_t cur = wkey[rw];
      const int t = cand_t(cur);
      const int32_t V = cand_vid(cur);
      if (rj == 6) {
        rv = V;
      } else if (wpos[rw] >= 0) {
        rv = b.cand_nbr[size_t(wpos[rw]) * 6 + rj];
      } else {  // a re-evaluation
        const VoxState& vst = m.vs[V];
        rv = (vst.tag == tag && vst.seg >= 0) ? nbr_eligible(m, b.seg_nbr[vst.seg * 6 + rj], tag, t)
                                              : nbr_at(m, vst.key, rj, tag, t);
      }
      nbv[rw][rj] = rv;
      if (rv >= 0) {
        const VoxState& ns_ = m.vs[rv];
        for (int k = 0; k < kPlaneD; ++k) rp[k] = m.plane[size_t(rv) * kPlaneD + k];
        grp[rw][rj] = ns_.group_id;
        rseg[rw][rj] = (ns_.tag == tag && ns_.seg >= 0) ? ns_.seg : -1;
        rkey[rw][rj] = ns_.key;
        rflg[rw][rj] = ns_.flags;
        for (int k = 0; k < kPlaneD; ++k) pl[rw][rj][k] = rp[k];
      }
    }
    __syncthreads();
    // ---- gates on the window's state (an entry no neighbour passes changes
    //      nothing)
    if (rv >= 0 && rj < 6 && grp[rw][rj] != grp[rw][6]) {
      double pv[6];
      for (int k = 0; k < 6; ++k) pv[k] = pl[rw][6][k];
      if (merge_gate(pv, rp, m.merge_a, m.merge_d)) atomicOr(&gates[rw], 1 << rj);
    }
    __syncthreads();
    uint64_t am = __ballot(lane < n && gates[min(lane, kWin - 1)] != 0);  // the acting entries
    max_acting = max(max_acting, __popcll(am));
    int w = kWin, nlim = n;  // this wave's entry; the first acting one without a wave
    {
      uint64_t r = am;
      for (int a = 0; a < kMrWaves && r; ++a) {
        const int e = __ffsll((unsigned long long)r) - 1;
        if (a == wv) w = e;
        r &= r - 1;
      }
      if (r) nlim = __ffsll((unsigned long long)r) - 1;
    }
    w = __builtin_amdgcn_readfirstlane(w);
    int32_t X = -1;  // this lane's taint item: a voxel of a record's closed neighbourhood
    bool need = false;
    int nl = 0, xseg = -1;
    uint64_t loc[kKeysPer];
    int cl = 0;
    if (w < kWin) {
      const int t = cand_t(wkey[w]);
      // ---- taint item r: voxel j (6: itself) next to record cj.  What does
      //      not depend on the merge is loaded before it; nothing here is
      //      written before the commit.
      const int cj = lane / 7, j = lane - 7 * cj;
      const bool item = lane < kTaintPer && nbv[w][min(cj, 6)] >= 0;
      int pre_tn = kNever;
      const bool pre = wspl[w] >= 0 && wspl[w] < b.pre_cap;  // a static entry's come precomputed
      bool simple = false;
      if (item) {
        if (pre) {
          const int at = wspl[w] * kPreItems + lane;
          X = b.pre_x[at];
          xseg = b.pre_seg[at];
          pre_tn = b.pre_tn[at];
        } else if (j == 6) {
          X = nbv[w][cj];
        } else {
          const int bseg = rseg[w][cj];
          if (bseg >= 0) {
            const int2 nb = b.seg_nbr[bseg * 6 + j];
            simple = nb.y != kNbrSlow;
            X = simple ? nb.x : vid_at(m, nb.x, tag, t);
          } else if (key_neighbour_ok(rkey[w][cj], j)) {
            X = vid_at(m, lookup_vid(m, key_neighbour(rkey[w][cj], j)), tag, t);
          }
        }
      }
      uint32_t xflags = 0;
      uint64_t xkey = 0, xgrp = 0;
      int xmp = kNever;
      double px[kPlaneD];
      int nct = 0, ct[7], xs0 = 0, xs1 = 0;
      if (X >= 0) {
        const VoxState* xv = m.vs + X;
        const int xtag = xv->tag, xsg = xv->seg, xev = xv->evict_t, xct = xv->create_t;
        xflags = xv->flags;
        xkey = xv->key;
        xgrp = xv->group_id;
        xmp = xv->merge_pos;
        for (int k = 0; k < kPlaneD; ++k) px[k] = m.plane[size_t(X) * kPlaneD + k];
        if (!pre) {
          xseg = (xtag == tag && xsg >= 0 && xev == kNever) ? xsg : -1;
          if (simple && xtag == tag && xct > t) X = -1;  // created later in the scan
        }
        if (xseg >= 0) {
          nct = b.seg_nct[xseg];
          for (int k = 0; k < 7; ++k) ct[k] = b.seg_ct[xseg * 7 + k];
          xs0 = b.seg_start[xseg];
          xs1 = b.seg_end[xseg];
        }
      }
      // ---- merge(): the six neighbours in order against the entry's own
      //      plane (the gates after a merge on the fused plane)
      double pv[kPlaneD];
      for (int k = 0; k < kPlaneD; ++k) pv[k] = pl[w][6][k];
      const uint64_t g6 = grp[w][6];
      const int cand = lane < 6 && nbv[w][min(lane, 5)] >= 0 && grp[w][min(lane, 5)] != g6;
      uint64_t pass = uint64_t(uint32_t(gates[w]));
      while (pass) {
        const int jj = __ffsll((unsigned long long)pass) - 1;
        double pn[kPlaneD];
        for (int k = 0; k < kPlaneD; ++k) pn[k] = pl[w][jj][k];
        merge_fuse(pv, pn);
        wave_lds_sync();
        if (lane == 0)
          for (int k = 0; k < kPlaneD; ++k) pl[w][jj][k] = pn[k];
        wave_lds_sync();
        cl |= 1 << jj;
        bool ok = cand && lane > jj;
        if (ok) {
          double pq[6];
          for (int k = 0; k < 6; ++k) pq[k] = pl[w][lane][k];
          ok = merge_gate(pv, pq, m.merge_a, m.merge_d);
        }
        pass = __ballot(ok);
      }
      cl |= 1 << 6;
      wave_lds_sync();
      if (lane == 0)
        for (int k = 0; k < kPlaneD; ++k) pl[w][6][k] = pv[k];
      wave_lds_sync();
      // ---- for each changed voxel and each voxel X of its closed
      //      neighbourhood: X re-evaluates its next call and its later
      //      candidates if X changed itself, or if X (a plane not in the
      //      group) passes the gates against a new record.  A voxel of the
      //      scan records its dirty time, one outside is marked dirty.
      if (!(item && ((cl >> cj) & 1))) X = -1;
      if (X >= 0) {
        int64_t ax, ay, az;
        unpack_key(xkey, ax, ay, az);
        for (int cc = 0; cc < 7; ++cc) {
          if (!((cl >> cc) & 1)) continue;
          if (nbv[w][cc] == X) need = true;
          if (need || !(xflags & kPlane) || !(xflags & kInit) || xgrp == g6) continue;
          int64_t bx, by, bz;
          unpack_key(rkey[w][cc], bx, by, bz);
          const int64_t dist = (ax > bx ? ax - bx : bx - ax) + (ay > by ? ay - by : by - ay) +
                               (az > bz ? az - bz : bz - az);
          if (dist != 1) continue;
          double pc[6];
          for (int k = 0; k < 6; ++k) pc[k] = pl[w][cc][k];
          if (merge_gate(px, pc, m.merge_a, m.merge_d)) need = true;
        }
        need = need && (xseg >= 0 || (xflags & kAlive));
        if (need && xseg >= 0) {
          const int tn = pre ? pre_tn : (xmp != kNever ? first_call_in(b, xs0 + xmp, xs1, t, off) : kNever);
          uint64_t first = ~0ull;
#pragma unroll
          for (int k = 0; k < kKeysPer; ++k) {
            const int tc = k == 0 ? tn : ct[k > 0 ? k - 1 : 0];
            const bool use = k == 0 ? tn != kNever : (k <= nct && tc > t);
            loc[k] = use ? cand_key(0, tc, X) : ~0ull;
            nl += use ? 1 : 0;
            if (loc[k] < first) first = loc[k];
          }
          if (nl > 0) atomicMin(reinterpret_cast<unsigned long long*>(&minkey[wv]), (unsigned long long)first);
        }
      }
    }
    if (lane == 0) {
      actw[wv] = w;
      clos[wv] = cl;
    }
    if (w < kWin) {
      int at = lane == 0 ? atomicAdd(&sh_i[4], __popc(unsigned(cl))) : 0;
      at = __builtin_amdgcn_readfirstlane(at);
      if (lane < 7 && ((cl >> lane) & 1)) wr[at + __popc(unsigned(cl) & ((1u << lane) - 1u))] = make_int2(nbv[w][lane], w);
    }
    __syncthreads();
    // ---- conflicts: an entry whose records, or whose taint items, an earlier
    //      entry of the window changes
    {
      const int me = rv >= 0 ? rw : -1, mx = X >= 0 ? w : -1, nw = sh_i[4];
      bool hit_r = false, hit_x = false;
#pragma unroll 8
      for (int q = 0; q < nw; ++q) {
        const int2 u = wr[q];
        hit_r |= (u.x == rv) & (u.y < me);
        hit_x |= (u.x == X) & (u.y < mx);
      }
      if (hit_r) conf[me] = 1;
      if (hit_x) conf[w] = 1;
    }
    __syncthreads();
    // ---- commit in point order, all at once: the first entry in conflict, or
    //      that an earlier entry's new key must precede, stops it.  The
    //      entries before it commit together: their write sets are disjoint
    //      (an entry that writes a voxel also read it).  Every wave finds the
    //      stop for itself.
    int stop;
    {
      const int l = min(lane, kWin - 1);
      const uint64_t key = wkey[l];
      bool late = conf[l] != 0;
#pragma unroll
      for (int a = 0; a < kMrWaves; ++a) late |= (actw[a] < l) & (minkey[a] <= key);
      const uint64_t bm = __ballot(lane < n && late);
      stop = bm ? __ffsll((unsigned long long)bm) - 1 : n;
      stop = min(stop, nlim);
      // the statics from the stop on are read again from the static list
      // (with their precomputed taint data) rather than sent to the pool;
      // consumed statics ascend, so they are the last ones
      sp -= __popcll(__ballot(lane >= stop && lane < n && wspl[l] >= 0));
    }
    evals += stop;
    requeued += n - stop;
#pragma unroll
    for (int a = 0; a < kMrWaves; ++a) merges += actw[a] < stop ? __popc(unsigned(clos[a])) - 1 : 0;
    if (w < stop) {
      if (lane < 7 && ((cl >> lane) & 1)) {  // a lane per changed record
        const int32_t Y = nbv[w][lane];
        double q[kPlaneD];
        for (int k = 0; k < kPlaneD; ++k) q[k] = pl[w][lane][k];
        for (int k = 0; k < kPlaneD; ++k) m.plane[size_t(Y) * kPlaneD + k] = q[k];
        m.vs[Y].group_id = grp[w][6];
        // an atomic bit set: another entry of this commit may set kDirty on Y
        atomicOr(&m.vs[Y].flags, kMerged);
        // the observe record from the LDS copies (merges never change the
        // plane bit, which is all the observe pass reads of the flags)
        int64_t kx, ky, kz;
        unpack_key(rkey[w][lane], kx, ky, kz);
        write_hot_pl(m, Y, rflg[w][lane] | kMerged, q, kx, ky, kz);
      }
      if (need) {
        VoxState& xs = m.vs[X];
        if (xseg >= 0) atomicMax(&xs.dirty_t, cand_t(wkey[w]));
        else atomicOr(&xs.flags, kDirty);
      }
      if (nl > 0) {
        int at = atomicAdd(&sh_i[3], nl);
#pragma unroll
        for (int k = 0; k < kKeysPer; ++k)
          if (loc[k] != ~0ull) gbuf[at++] = loc[k];
      }
    }
    // ---- pool := pool[ph, pn) merged with the committed entries' new keys and
    //      the pool entries sent back (duplicates are dropped at the next fill)
    if (tid >= stop && tid < n && wspl[tid] < 0) gbuf[atomicAdd(&sh_i[3], 1)] = wkey[tid];
    // duplicates of a key sent back must not be dropped against it: the last
    // processed key is the last committed one
    if (stop > 0) last = wkey[stop - 1];
    __syncthreads();
    const int g = sh_i[3], rest = pn - ph;
    if (g + rest > kPoolCap) {
      err |= 16;
      break;
    }
    const uint64_t* prest = &pool[pb][ph];
    uint64_t* dst = pool[1 - pb];
    for (int k = tid; k < g; k += kMrThreads) {  // ties by index
      const uint64_t v = gbuf[k];
      int rk = rank_lt(prest, rest, v);
#pragma unroll 4
      for (int q = 0; q < g; ++q) rk += (gbuf[q] < v) || (gbuf[q] == v && q < k);
      dst[rk] = v;
    }
    for (int k = tid; k < rest; k += kMrThreads) {
      const uint64_t v = prest[k];
      int rk = k;
#pragma unroll 4
      for (int q = 0; q < g; ++q) rk += gbuf[q] <= v;
      dst[rk] = v;
    }
    pb = 1 - pb;
    ph = 0;
    pn = g + rest;
    __syncthreads();
  }
  if (tid == 0) {
    c->merge_evals += evals;
    c->merges += merges;
    c->merge_windows += windows;
    c->merge_requeued += requeued;
    c->merge_max_acting = max(c->merge_max_acting, max_acting);
    if (err) atomicOr(&c->error, err);
  }
}

}  // namespace vmp
