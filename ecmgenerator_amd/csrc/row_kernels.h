// row_kernels.h -- the plain step's per-agent passes with 16 lanes per agent,
// for crowds that leave the chip idle at one agent per lane; row_rule.h says
// up to which size.  Included by sim_kernels.hip inside namespace ecm.
//
// At one agent per lane, a crowd of up to some 65,000 agents fills at most one
// wavefront per SIMD, and a pass lasts as long as one wavefront's chain of
// dependent loads and unrolled code: 82-85 us for the neighbour search and
// ORCA at 500 agents as at 5,000 (k 10), plus the queue kernels of the
// agents that need the 3D LP.  Here a row of 16 lanes (one DPP row) works on
// one agent, four agents per wavefront: the lanes test candidate cells,
// obstacle edges, path segments and LP constraints side by side, so the
// chain is a few tens of loads and a rolled loop of a few KB of code, and
// the 3D LP follows in place.  Each value is computed with the operations,
// and each list kept in the order, of the one-lane form; results are equal
// bit for bit.

constexpr int kRow = 16;
// Candidates buffered per agent in the neighbour search, kRowTrip a lane at a
// time: selected down to k (at most 16) when the next might not fit.
constexpr int kRowTrip = 4;
constexpr int kRowCand = 96;
constexpr int kRowLdsBytes = (kRowCand + 4 + kRow) * 12;      // (d2, id) and sorted position of each candidate, with
                                                              // room behind them, and of the k selected
template <int N>
__device__ __forceinline__ int row_ror(int v) {
    return __builtin_amdgcn_mov_dpp(v, 0x120 + N, 0xf, 0xf, true);
}
// Reductions over the 16 lanes, the result in every lane.
__device__ __forceinline__ int row_min(int v) {
    v = min(v, row_ror<8>(v)); v = min(v, row_ror<4>(v)); v = min(v, row_ror<2>(v));
    return min(v, row_ror<1>(v));
}
__device__ __forceinline__ int row_max(int v) {
    v = max(v, row_ror<8>(v)); v = max(v, row_ror<4>(v)); v = max(v, row_ror<2>(v));
    return max(v, row_ror<1>(v));
}
// Floats (no NaN) as integers of the same order, and back: the integer
// minimum takes one DPP instruction a step, the float one also quiets.
__device__ __forceinline__ int order_of(float v) {
    const int b = __float_as_int(v);
    return b ^ ((b >> 31) & 0x7fffffff);
}
__device__ __forceinline__ float of_order(int v) { return __int_as_float(v ^ ((v >> 31) & 0x7fffffff)); }
// The row's bits of the wavefront's ballot.
__device__ __forceinline__ uint32_t row_ballot(bool b) {
    return (uint32_t)(__ballot(b) >> (__lane_id() & 48u)) & 0xffffu;
}
__device__ __forceinline__ V2 row_get(V2 v, int lane) { return mk(__shfl(v.x, lane, kRow), __shfl(v.y, lane, kRow)); }
// Orders the row's LDS accesses for the compiler (the hardware runs one
// wavefront's in order).
__device__ __forceinline__ void row_fence() {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

// ------------------------------------------------------------- attraction
// locate_cell, 16 listed cells at a time: each list ascends, so its first
// cell that contains p is the lowest lane's, and the collection's first is
// the lower of the two lists'.
__device__ __forceinline__ int row_locate_cell(const EnvDesc& s, V2 p, int l, uint32_t& fallback) {
    if (s.n_cells == 0) return -1;
    const int bx = grid_cell(p.x, s.eg.x0, s.eg.inv_cell, s.eg.side);
    const int by = grid_cell(p.y, s.eg.y0, s.eg.inv_cell, s.eg.side);
    const int b = by * s.eg.side + bx;
    const uint32_t key = (p.y == 0.0f) ? 0u : __float_as_uint(p.y);
    uint32_t h = hash_u32(key) & (uint32_t)s.yhash_mask;
    uint32_t kk = 0xffffffffu;
    if (s.yhash_mask >= 0) kk = s.yhash_key[h];
    const int i0 = s.ebucket_start[b], ie = s.ebucket_start[b + 1];
    int best = INT_MAX;
    auto scan = [&](const int* list, int a, int e) {
        for (int i = a; i < e; i += kRow) {
            bool in = false;
            int c = INT_MAX;
            if (i + l < e) {
                c = list[i + l];
                const float4 A = s.cellA[c], B = s.cellB[c];
                in = quad_contains(p, mk(A.x, A.y), mk(A.z, A.w), mk(B.x, B.y), mk(B.z, B.w));
            }
            const uint32_t m = row_ballot(in);
            if (m) {
                best = min(best, __shfl(c, __ffs((int)m) - 1, kRow));
                return;
            }
        }
    };
    scan(s.ebucket_cells, i0, ie);
    while (kk != 0xffffffffu) {
        if (kk == key) {
            const int j0 = s.yhash_off[h];
            scan(s.ycells, j0, j0 + s.yhash_cnt[h]);
            fallback = 1;
            break;
        }
        h = (h + 1u) & (uint32_t)s.yhash_mask;
        kk = s.yhash_key[h];
    }
    return best == INT_MAX ? -1 : best;
}

// irm_attraction with one path segment per lane, 16 from the end at a time.
__device__ __forceinline__ bool row_irm(const EnvDesc& s, V2 pos, int cell, const float2* path, int np, int l, V2& out) {
    if (cell < 0) return false;
    V2 rl = mk(0.0f, 0.0f), oa, ob;
    if (!retract(s, pos, cell, rl, oa, ob)) return false;
    const V2 co = closest_on_segment(rl, oa, ob);
    const float clearance = len(rl - co);
    const float clr2 = clearance * clearance;
    const float2 g = path[np - 1];
    const V2 goal = mk(g.x, g.y);
    if (len2(goal - rl) < clr2) { out = goal; return true; }
    bool success = false;
    for (int hi = np - 1; hi > 0; hi -= kRow) {
        const int lo = max(hi - kRow, 0);
        const int i = lo + l;
        bool met = false, hit = false;
        V2 at = mk(0.0f, 0.0f);
        if (i < hi) {
            const float2 pa = path[i], pb = path[i + 1];
            const V2 q1 = mk(pa.x, pa.y) - rl;
            const V2 q2 = mk(pb.x, pb.y) - rl;
            const V2 ed = q2 - q1;
            const float el2 = len2(ed);
            const float dm = det(q1, q2);
            const float disc = clr2 * el2 - dm * dm;
            met = !(disc < kEps);
            if (met) {
                const float sgn = ed.y < 0.0f ? -1.0f : 1.0f;
                const float sq = sqrtf(disc);
                const V2 i1 = mk((dm * ed.y + sgn * ed.x * sq) / el2, (-dm * ed.x + fabsf(ed.y) * sq) / el2);
                const V2 i2 = mk((dm * ed.y - sgn * ed.x * sq) / el2, (-dm * ed.x - fabsf(ed.y) * sq) / el2);
                const V2 g1 = q1 + rl, g2 = q2 + rl;
                const V2 gi1 = i1 + rl, gi2 = i2 + rl;
                const V2 edg = g2 - g1;
                const float t1 = dot(gi1 - g1, edg) / el2;
                const float t2 = dot(gi2 - g1, edg) / el2;
                const bool v1 = t1 >= 0.0f && t1 <= 1.0f;
                const bool v2 = t2 >= 0.0f && t2 <= 1.0f && t2 > (v1 ? t1 : -1.0f);
                hit = v1 || v2;
                at = v2 ? gi2 : gi1;
            }
        }
        success |= row_ballot(met) != 0u;
        const uint32_t m = row_ballot(hit);
        if (m) {
            out = row_get(at, 31 - __clz((int)m));
            return true;
        }
    }
    return success;
}

// attr_agent with 16 lanes.
__device__ __forceinline__ void row_attr_agent(const DevState& s, int t, int l, const AttrIn& in) {
    const V2 pos = mk(in.pr.x, in.pr.y);
    const EnvDesc& E = env_of_sorted(s, in.sv);
    const int np = in.pc.y;
    const float2* path = s.path_pts + in.pc.x;
    const float2 gg = path[np - 1];
    uint32_t fb = 0;
    const int cell = row_locate_cell(E, pos, l, fb);
    const float gx = pos.x - gg.x, gy = pos.y - gg.y;
    const float dGoal = gx * gx + gy * gy;
    V2 attr = mk(in.a0.x, in.a0.y);
    bool alive = true, event = false;
    if (dGoal < s.arrival_r2) {
        attr = mk(gg.x, gg.y);
        if (dGoal < s.delete_r2) alive = false;
        fb = 0;
    } else {
        V2 ap = mk(0.0f, 0.0f);
        if (row_irm(E, pos, cell, path, np, l, ap)) attr = ap;
        else event = true;
    }
    if (l != 0) return;
    // UpdatePath(e, currentPosition, goal) with the step-start position
    if (event) put_event(s, __float_as_int(in.pr.w), __float_as_int(pos.x), __float_as_int(pos.y), t);
    s.attr_s[t] = make_float2(attr.x, attr.y);
    if (fb) atomicAdd(&s.stats[2], 1u);
    s.dead_s[t] = alive ? 0 : 1;
    if (!alive) {
        retire_agent(s, in, attr);
        return;
    }
    const V2 des = normalize(attr - pos) * in.sv.z;
    s.pref_vel_s[t] = make_float2(des.x, des.y);
}

// k_attr and k_scatter_attr with 16 lanes per agent: 14 -> 10 us at 500 agents
// and 18 -> 13 at 5,000; at 37,000 40 instead of 21 (four times the
// wavefronts wait on the same loads), so larger crowds keep one lane.
__global__ __launch_bounds__(256) void k_attr_row(DevState s) {
    const int n_active = (int)s.cell_start[s.n_keys];
    const int per = blockDim.x / kRow, l = threadIdx.x & (kRow - 1);
    for (int t = xcd_block() * per + (int)threadIdx.x / kRow; t < n_active; t += gridDim.x * per)
        row_attr_agent(s, t, l, attr_in(s, t));
    publish_if_last(s, gridDim.x);
}

__global__ __launch_bounds__(256) void k_scatter_attr_row(DevState s, uint32_t blocks) {
    __shared__ __align__(16) uint32_t top[kTopMax];
    if (blockIdx.x >= blocks) { write_starts(s, blockIdx.x - blocks); return; }
    const int n_old = (int)(uint32_t)s.acc[14], n = n_old + (int)(uint32_t)s.acc[15];
    const int per = blockDim.x / kRow, l = threadIdx.x & (kRow - 1);
    int t = xcd_block((int)blocks) * per + (int)threadIdx.x / kRow;
    Moved M = moved_agent(s, t, n_old, n);
    const Starts S = scatter_starts(s, top);
    while (t < n) {
        if (M.m != kInvalidKey) {
            const int slot = (int)(S.pre[M.m / kScanCells] + M.in_cell);
            if (l == 0) store_moved(s, M.in, slot);
            row_attr_agent(s, slot, l, M.in);
        }
        t += (int)blocks * per;
        M = moved_agent(s, t, n_old, n);
    }
    publish_if_last(s, blocks);
}

// ------------------------------------------------------------- neighbours
// One agent's candidates in LDS, (d2, id) pairs and sorted positions, and the
// selected ones.
struct RowCand {
    float2 *di, *best;
    int *slot, *best_slot;
};
__device__ __forceinline__ RowCand row_cand(float4* lds) {
    float2* di = reinterpret_cast<float2*>(lds);
    int* slot = reinterpret_cast<int*>(di + kRowCand + 4 + kRow);
    return RowCand{di, di + kRowCand + 4, slot, slot + kRowCand + 4};
}

// Keeps the k best of the m buffered candidates, in (d2, id) order from
// entry 0 on: each lane ranks its entries against all, four per trip.
__device__ __forceinline__ void row_select(const RowCand& B, int k, int l, int& m, float& thr) {
    // the up to three entries behind the last rank behind every real one
    if (l < 3) B.di[m + l] = make_float2(INFINITY, __int_as_float(INT_MAX));
    row_fence();
    const float4* two = reinterpret_cast<const float4*>(B.di);
    for (int e = l; e - l < m; e += kRow) {
        const float2 own = e < m ? B.di[e] : make_float2(INFINITY, __int_as_float(INT_MAX));
        const int id = __float_as_int(own.y);
        int rank = 0;
        for (int i = 0; i < m; i += 4) {
            const float4 a = two[i / 2], b = two[i / 2 + 1];
            rank += (int)nb_better(a.x, __float_as_int(a.y), own.x, id) +
                    (int)nb_better(a.z, __float_as_int(a.w), own.x, id) +
                    (int)nb_better(b.x, __float_as_int(b.y), own.x, id) +
                    (int)nb_better(b.z, __float_as_int(b.w), own.x, id);
        }
        if (e < m && rank < k) {
            B.best[rank] = own;
            B.best_slot[rank] = B.slot[e];
        }
    }
    row_fence();
    m = min(m, k);
    if (l < m) {
        B.di[l] = B.best[l];
        B.slot[l] = B.best_slot[l];
    }
    row_fence();
    if (m == k) thr = fminf(thr, B.di[k - 1].x);
}

// The exact k nearest of the agent at sorted position t: the candidates of
// knn_query / knn_query_seeded (d2 > eps, within the seeds' bound when there
// is one, else ring by ring until the unvisited region is beyond the k-th),
// a cell per lane, collected in LDS and ranked by (d2, id).  Returns the
// count; lane r < count holds the r-th neighbour's sorted position in slot.
__device__ __forceinline__ int row_knn(const DevState& s, const EnvDesc& E, int t, int q, V2 p, int l,
                                       const RowCand& B, int& slot) {
    const int k = s.k;
    const GridDesc& g = E.ag;
    float thr = INFINITY;
    {
        // the seeds (q: the agent's last sorted position), every level's
        // loads issued together, out-of-range entries reading entry 0
        const bool had = q >= 0 && q < s.n_slots;
        const int had_n = s.nbr_cnt_prev[had ? q : 0];
        const int os = s.nbr_prev[(size_t)min(l, k - 1) * s.n_slots + (had ? q : 0)];
        const bool in = os >= 0 && os < s.n_slots;
        const int f = s.fwd[in ? os : 0];
        const bool on = in && f >= 0 && f < s.n_slots;
        const float4 c = s.sorted_pr[on ? f : 0];
        const float dx = c.x - p.x, dy = c.y - p.y;
        const float d2 = dx * dx + dy * dy;
        bool ok = had && had_n >= k && on && d2 > kEps;
        if (s.agent_env) ok = ok && __float_as_int(s.sorted_v[on ? f : 0].w) == __float_as_int(s.sorted_v[t].w);
        if (row_ballot(!ok) == 0u) thr = __int_as_float(row_max(__float_as_int(d2)));       // d2 > 0
    }
    int m = 0;
    const float wmax = kKnnWalkCells * g.cell;
    // one rectangle of cells around the bound's circle, which holds every
    // candidate (knn_query_seeded), or rings around the agent's cell, until
    // the unvisited region is beyond the k-th (knn_query)
    const bool rect = thr <= wmax * wmax;
    const float guard = 2e-3f;
    int cx = grid_cell(p.x, g.x0, g.inv_cell, g.side);
    int cy = grid_cell(p.y, g.y0, g.inv_cell, g.side);
    int w = 1, nc = 1;
    if (rect) {
        const float rr = __builtin_amdgcn_sqrtf(thr) * 1.0001f + guard;
        cx = grid_cell(p.x - rr, g.x0, g.inv_cell, g.side);
        cy = grid_cell(p.y - rr, g.y0, g.inv_cell, g.side);
        w = grid_cell(p.x + rr, g.x0, g.inv_cell, g.side) - cx + 1;
        nc = w * (grid_cell(p.y + rr, g.y0, g.inv_cell, g.side) - cy + 1);
    }
    // q / w for the rectangle's few hundred cells: half a cell from any
    // whole quotient, far more than the reciprocal's error
    const float inv_w = __builtin_amdgcn_rcpf((float)w);
    for (int r = 0;; ++r) {
        if (!rect) nc = r == 0 ? 1 : 8 * r;
        float prune2 = INFINITY;
        if (thr < INFINITY) {
            const float rr = __builtin_amdgcn_sqrtf(thr) * 1.0001f + guard;
            prune2 = rr * rr;
        }
        for (int q0 = 0; q0 < nc; q0 += kRow) {
            const int q = q0 + l;
            int x, y;
            if (rect) { const int yy = (int)(((float)q + 0.5f) * inv_w); x = cx + (q - yy * w); y = cy + yy; }
            else if (r == 0) { x = cx; y = cy; }
            else if (q < 2 * r + 1) { x = cx - r + q; y = cy + r; }
            else if (q < 4 * r + 2) { x = cx - r + (q - (2 * r + 1)); y = cy - r; }
            else if (q < 6 * r + 1) { x = cx - r; y = cy - r + 1 + (q - (4 * r + 2)); }
            else { x = cx + r; y = cy - r + 1 + (q - (6 * r + 1)); }
            uint32_t a = 0, b = 0;
            if (q < nc && x >= 0 && y >= 0 && x < g.side && y < g.side &&
                band_d2(p.x, g.x0, g.cell, x, g.side) + band_d2(p.y, g.y0, g.cell, y, g.side) <= prune2) {
                const uint32_t key = E.cell_base + morton2((uint32_t)x, (uint32_t)y);
                a = s.cell_start[key];
                b = s.cell_start[key + 1];
            }
            // a cell's agents [a, b) per lane, the lanes in step, kRowTrip at
            // a time with their loads together
            while (row_ballot(a < b)) {
                if (m > kRowCand - kRow * kRowTrip) row_select(B, k, l, m, thr);
                float4 c[kRowTrip];
#pragma unroll
                for (int u = 0; u < kRowTrip; ++u) c[u] = s.sorted_pr[a < b ? min(a + u, b - 1u) : 0u];
#pragma unroll
                for (int u = 0; u < kRowTrip; ++u) {
                    const float dx = c[u].x - p.x, dy = c[u].y - p.y;
                    const float d2 = dx * dx + dy * dy;
                    const bool keep = a + u < b && d2 > kEps && d2 <= thr;
                    const uint32_t bal = row_ballot(keep);
                    if (keep) {
                        const int e = m + __popc(bal & ((1u << l) - 1u));
                        B.di[e] = make_float2(d2, c[u].w);
                        B.slot[e] = (int)(a + u);
                    }
                    m += __popc(bal);
                }
                a += kRowTrip;
            }
        }
        const int xl = cx - r, xh = cx + r, yl = cy - r, yh = cy + r;
        const bool all = rect || (xl <= 0 && yl <= 0 && xh >= g.side - 1 && yh >= g.side - 1);
        if (all || m >= k) row_select(B, k, l, m, thr);
        if (all) break;
        if (thr < INFINITY) {
            float bnd = INFINITY;
            if (xl > 0) bnd = fminf(bnd, p.x - (g.x0 + (float)xl * g.cell));
            if (yl > 0) bnd = fminf(bnd, p.y - (g.y0 + (float)yl * g.cell));
            if (xh < g.side - 1) bnd = fminf(bnd, (g.x0 + (float)(xh + 1) * g.cell) - p.x);
            if (yh < g.side - 1) bnd = fminf(bnd, (g.y0 + (float)(yh + 1) * g.cell) - p.y);
            bnd -= guard;
            if (bnd > 0.0f && bnd * bnd > thr) {
                if (m < k) row_select(B, k, l, m, thr);
                break;
            }
        }
    }
    slot = l < m ? B.slot[l] : -1;
    row_fence();                                     // the buffer is reused
    return m;
}

// -------------------------------------------------------------------- LPs
// A row's constraint list in the reference's order: nO obstacle constraints
// in LDS (ob, the first 16 also in on / op of lane c), then na agent
// constraints, number a in an / ap of lane a; pool is LDS for 16 of those.
struct RowList {
    const float4* ob;
    float4* pool;
    int nO, na;
    V2 on, op;
};

__device__ __forceinline__ V2 ob_n(const float4& c) { return mk(c.x, c.y); }
__device__ __forceinline__ V2 ob_p(const float4& c) { return mk(c.z, c.w); }

// The first constraint from index i < nO + na on that `test` holds for, or
// nO + na; agent constraints outside the bits of aval are passed over.
template <typename F>
__device__ __forceinline__ int row_first(const RowList& C, V2 an, V2 ap, uint32_t aval, int i, int l, F&& test) {
    const bool va = ((aval >> l) & 1u) && test(an, ap);
    if (C.nO <= kRow) {
        // both of a lane's constraints at once
        const bool vo = l < C.nO && test(C.on, C.op);
        const uint32_t m = (row_ballot(vo) | (row_ballot(va) << C.nO)) & (~0u << i);
        return m ? __ffs((int)m) - 1 : C.nO + C.na;
    }
    for (int c0 = i & ~(kRow - 1); c0 < C.nO; c0 += kRow) {
        const int c = c0 + l;
        bool v = false;
        if (c >= i && c < C.nO) {
            const float4 q = C.ob[c];
            v = test(ob_n(q), ob_p(q));
        }
        const uint32_t m = row_ballot(v);
        if (m) return c0 + __ffs((int)m) - 1;
    }
    const uint32_t m = row_ballot(va && l >= i - C.nO);
    return m ? C.nO + __ffs((int)m) - 1 : C.nO + C.na;
}

// RandomizedLP (ORCA.cpp:428-587) over the list: the loop over every i
// becomes the next violated i (the others leave the velocity unchanged), and
// the loop over j < i one step of all lanes with a row minimum and maximum:
// the bounds only tighten, so the reference's test within the loop fails
// exactly when the final bounds cross.  Equal zeros of different sign
// resolve to the first in list order, as std::min / std::max keep it.
template <bool DIR>
__device__ __forceinline__ int row_lp(const RowList& C, V2 an, V2 ap, uint32_t aval, V2 opt, float maxSpeed, int l,
                                      V2& out) {
    if (DIR) out = opt * maxSpeed;
    else if (len(opt) > maxSpeed) out = normalized(opt) * maxSpeed;
    else out = opt;
    C.pool[l] = make_float4(an.x, an.y, ap.x, ap.y);
    row_fence();
    const int n = C.nO + C.na;
    int i = 0;
    while (i < n) {
        i = row_first(C, an, ap, aval, i, l, [&](V2 cn, V2 cp) { return !(det(right(cn), cp - out) <= 0.0f); });
        if (i >= n) return n;
        const float4 h = *(i < C.nO ? C.ob + i : C.pool + (i - C.nO));
        const V2 hn = ob_n(h), hp = ob_p(h);
        const V2 dir = right(hn);
        const float dpd = dot(dir, hp);
        const float disc = dpd * dpd + maxSpeed * maxSpeed - dot(hp, hp);
        if (disc <= 0.0f) return i;
        const float sq = exp_within(disc, -96, 96) ? root_from(disc, __builtin_amdgcn_rsqf(disc)) : sqrtf(disc);
        float lo = -INFINITY, hi = INFINITY;
        int klo = INT_MAX, khi = INT_MAX;           // 2 index + sign of the lane's bound
        bool bad = false;
        auto narrow = [&](int j, V2 jn, V2 jp) {
            const float den = det(right(hn), right(jn));
            const float num = det(right(jn), hp - jp);
            if (fabsf(den) <= kEps) {
                bad |= num < 0.0f;
            } else {
                const float t = num / den;
                const int key = 2 * j + (int)(__float_as_uint(t) >> 31);
                if (den >= 0.0f) { if (t < hi) { hi = t; khi = key; } }
                else if (t > lo) { lo = t; klo = key; }
            }
        };
        const int oi = min(i, C.nO);
        if (l < oi) narrow(l, C.on, C.op);
        for (int c = l + kRow; c < oi; c += kRow) { const float4 q = C.ob[c]; narrow(c, ob_n(q), ob_p(q)); }
        if (l < i - C.nO && ((aval >> l) & 1u)) narrow(C.nO + l, an, ap);
        if (row_ballot(bad)) return i;
        float tl = of_order(row_max(order_of(lo))), tr = of_order(row_min(order_of(hi)));
        if (tl == 0.0f || tr == 0.0f) {
            if (tl == 0.0f) tl = row_min(lo == 0.0f ? klo : INT_MAX) & 1 ? -0.0f : 0.0f;
            if (tr == 0.0f) tr = row_min(hi == 0.0f ? khi : INT_MAX) & 1 ? -0.0f : 0.0f;
        }
        const float lft = std_max(-dpd - sq, tl);
        const float rgt = std_min(-dpd + sq, tr);
        if (lft > rgt) return i;
        float t;
        if (DIR) {
            t = dot(opt, dir) > 0 ? rgt : lft;
        } else {
            t = dot(dir, opt - hp);
            t = t < lft ? lft : (t > rgt ? rgt : t);
        }
        out = hp + dir * t;
        ++i;
    }
    return n;
}

// RandomizedLP3D (ORCA.cpp:592-669): the bisectors with the agent
// constraints before ci, one per lane, keep their places in the list.
__device__ __forceinline__ void row_lp3d(const RowList& C, V2 an, V2 ap, float maxSpeed, int failed, int l, V2& out) {
    const int n = C.nO + C.na;
    const uint32_t all = (1u << C.na) - 1u;
    float maxPen = 0.0f;
    int i = failed;
    while (i < n) {
        i = row_first(C, an, ap, all, i, l, [&](V2 cn, V2 cp) { return !(det(right(cn), cp - out) <= maxPen); });
        if (i >= n) return;
        V2 cn, cp;
        if (i < C.nO) { const float4 q = C.ob[i]; cn = ob_n(q); cp = ob_p(q); }
        else { cn = row_get(an, i - C.nO); cp = row_get(ap, i - C.nO); }
        V2 pn = mk(0.0f, 0.0f), pp = mk(0.0f, 0.0f);
        bool has = false;
        if (l < i - C.nO) {
            const float d = det(right(cn), right(an));
            if (fabsf(d) <= kEps) {
                if (!(dot(cn, an) > 0)) {
                    pp = (cp + ap) * 0.5f;
                    pn = normalized(an - cn);
                    has = true;
                }
            } else {
                const float tt = det(right(an), cp - ap) / d;
                pp = cp + right(cn) * tt;
                pn = normalized(an - cn);
                has = true;
            }
        }
        const uint32_t pval = row_ballot(has);
        const V2 temp = out;
        if (row_lp<true>(C, pn, pp, pval, cn, maxSpeed, l, out) < n) out = temp;
        maxPen = det(right(cn), cp - out);
        ++i;
    }
}

// The obstacle edge of a lane: its loads, apart from its constraint.
struct RowEdge {
    int e;                    // -1: none
    float4 a, b, c;
};
__device__ __forceinline__ RowEdge row_edge(const EnvDesc& E, int q, int e1) {
    RowEdge r;
    r.e = q < e1 ? E.obucket_edges[q] : -1;
    const int at = max(r.e, 0);
    r.a = E.oe0[at];
    r.b = E.oe1[at];
    r.c = E.oe2[at];
    return r;
}

// Neighbour search, ORCA, both LPs and the integration of the agent at
// sorted position t.  lds: the row's share, room for maxo obstacle and 16
// agent constraints and for the candidate buffer (used one after the other).  The
// loads of the obstacle edges go out before the neighbour search and those
// of the neighbours before the edges' half-planes: a lone wavefront waits for
// each level of dependent loads, 500-900 cycles, and there are a dozen.
__device__ __forceinline__ void row_step_agent(const DevState& s, int t, int l, float4* lds, int maxo) {
    const float4 pr = s.sorted_pr[t];
    const float4 sv = s.sorted_v[t];
    const int prev = s.prev_of[t];
    const float2 pv = s.pref_vel_s[t];
    if (s.dead_s[t]) {                               // destroyed this step: state unchanged
        if (l == 0) {
            s.nbr_cnt[t] = 0;
            s.pos_s[t] = make_float2(pr.x, pr.y);
            s.vel_s[t] = make_float2(sv.x, sv.y);
        }
        return;
    }
    const V2 position = mk(pr.x, pr.y);
    const V2 velocity = mk(sv.x, sv.y);
    const float rad = pr.z;
    const float maxSpeed = s.max_speed_from_pref ? sv.z : s.max_speed;
    const EnvDesc& E = env_of_sorted(s, sv);
    const bool obst = E.n_obst_edges > 0;
    int e0 = 0, e1 = 0;
    RowEdge edge;
    if (obst) {
        obstacle_bucket(E, position, e0, e1);
        edge = row_edge(E, e0 + l, e1);
    }
    int slot;
    const RowCand B = row_cand(lds);
    const int cnt = row_knn(s, E, t, prev, position, l, B, slot);
    const float4 q = s.sorted_pr[l < cnt ? slot : t];
    const float2 qv = sorted_vel(s, l < cnt ? slot : t);
    if (l < cnt) s.nbr[(size_t)l * s.n_slots + t] = slot;
    if (l == 0) s.nbr_cnt[t] = cnt;

    RowList C;
    C.ob = lds;
    C.pool = lds + maxo;
    C.nO = 0;
    C.na = cnt;
    // the edges of the bucket, one per lane, kept in bucket order
    if (obst) {
        const float range = s.time_horizon_obst * maxSpeed + rad;          // ORCA.cpp:27
        for (int q0 = e0; q0 < e1; q0 += kRow) {
            if (q0 > e0) edge = row_edge(E, q0 + l, e1);
            bool made = false;
            V2 cp = mk(0.0f, 0.0f), cn = mk(0.0f, 0.0f);
            float dd;
            if (edge.e >= 0 && edge_near(edge.a, position, range * range, dd))
                made = edge_constraint(s, edge.a, edge.b, edge.c, position, velocity, rad, cp, cn);
            const uint32_t m = row_ballot(made);
            const int at = C.nO + __popc(m & ((1u << l) - 1u));
            if (made && at < maxo) lds[at] = make_float4(cn.x, cn.y, cp.x, cp.y);
            C.nO += __popc(m);
        }
        C.nO = min(C.nO, maxo);                      // maxo covers the longest bucket
    }
    V2 an = mk(0.0f, 0.0f), ap = mk(0.0f, 0.0f);
    if (l < cnt && !(s.inv_dt != 0.0f && agent_constraint_common(s, position, velocity, rad, q, qv, ap, an)))
        agent_constraint(s, position, velocity, rad, q, qv, ap, an);
    row_fence();
    const float4 own = l < C.nO ? lds[l] : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    C.on = ob_n(own);
    C.op = ob_p(own);
    V2 o;
    const int n = C.nO + cnt;
    const int fail = row_lp<false>(C, an, ap, (1u << cnt) - 1u, mk(pv.x, pv.y), maxSpeed, l, o);
    if (fail < n) row_lp3d(C, an, ap, maxSpeed, fail, l, o);
    // the counters of the one-lane passes: 3D LPs, agents past the main
    // pass's obstacle slots, and both
    uint32_t* ws = s.wstats + kStatStride * (blockIdx.x % kStatSlots);
    wave_count(ws + kStat3d, l == 0 && fail < n);
    wave_count(ws + kStatOvf, l == 0 && C.nO > kRowStatObst);
    wave_count(ws + kStatBig, l == 0 && fail < n && C.nO > kRowStatObst);
    if (l == 0) integrate(s, t, position, velocity, o);
    row_fence();                                     // lds is reused by the next agent
}

// One wavefront per block: four agents at a time, strided over the grid.
__global__ __launch_bounds__(64, 5) void k_row_step(DevState s, int maxo, int row_f4) {
    extern __shared__ float4 row_lds[];
    const int n_active = (int)s.cell_start[s.n_keys];
    const int r = threadIdx.x / kRow, l = threadIdx.x & (kRow - 1);
    for (int t = xcd_block() * 4 + r; t < n_active; t += gridDim.x * 4)
        row_step_agent(s, t, l, row_lds + r * row_f4, maxo);
}
