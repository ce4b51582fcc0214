// vxs_split.h — wide rows (vocabulary above 8192) sampled by several workgroups each, for batches too
// small to fill the chip with one workgroup per row. Included by vxs_wide.hip, inside its namespace.
//
// A row is cut into segments of 1024 NC consecutive entries, one 256-thread workgroup each, which keeps
// its segment in registers (thread t the entries 1024 c + 4 t + j of it) after one read and one
// transform (S1-S4). What the segments of a row tell each other goes through a record per segment in a
// workspace, between arrivals at counters of the row:
//   greedy, top-k <= 256   each segment publishes its maximum, or the entries that can be among the
//                          row's k largest (at least its own k largest, in index order); the last to
//                          arrive finishes the row alone, with the ordered pass's tail.
//   nucleus (no top-k)     the segments meet four times: row maximum; the mass of 160 buckets a quarter
//                          octave wide, which locate the top-p cut; 128 parts of the bucket that holds
//                          it; the few entries of that part. Then every workgroup knows the exact cut
//                          and each segment's kept mass, and the one whose segment holds the draw
//                          finds it in its registers.
// What bounds it: with few rows the chain of reads, meetings (about 2 us each) and the finish, not the
// bytes; 64 nucleus rows of 151936 entries take 45.7 us (one workgroup per row: 1361), of which the one
// read of 39 MB is 8; 16 top-k rows 22.1 (76). Segments stay in registers so that no stage reads the
// row again, which holds them to 128 registers (four workgroups per compute unit): larger segments with
// three per unit took 47.6 to 61 us.
//
// Masses are the fixed-point ones of the other kernels (multiples of 2^-F, exact sums in any order).
// A top-k above 256 goes through the same stages over counts first, to its k-th largest value, and then on
// as a nucleus row over what is left. Rows that none of this fits (more ties than the exact regime or a list holds, top-p
// not above 0) are sampled by the last workgroup to leave, with the general algorithm.
//
// A meeting is a bounded wait: workgroups are dispatched in order, so a row's arrive together unless
// other work holds the chip, and one that has waited meet_ticks gives the row up for all its workgroups
// (a compare-and-swap that only succeeds while the meeting is incomplete, so they agree); the last to
// leave then samples it. Nothing waits for that.

constexpr int kSplitMaxSegs = 64;                       // one lane each
constexpr int kSegList = 1152;                          // top-k entries a segment can publish
constexpr int kCoarse = 160;                            // quarter-octave buckets: 4 per octave, up to 39 octaves and 1.0
constexpr int kSub = 128;                               // parts of one of them
constexpr int kSegPart = 256;                           // entries of the cut's part per segment ...
constexpr int kRowPart = 768;                           // ... and per row
constexpr int kMine = 4096;                             // indices of the cut's part kept in LDS per segment
constexpr int kFineMass = kCoarse * 16;                 // LDS histogram: 64 buckets per octave
constexpr uint32_t kAbandoned = 0x80000000u;

struct alignas(64) SplitRow {  // zero between calls
    uint32_t meet[8];
    uint32_t left;
    // the row's counts (top-k above kKMax) and masses, summed up by its segments
    alignas(64) uint64_t coarse[2][kCoarse], sub[2][kSub];
};
struct alignas(16) SplitSeg {
    uint32_t maxkey, cnt, bad, n;     // largest key; finite entries; 1 non-finite, 2 bad history id; entries listed
    uint32_t bkey, argi, kmin, kmax;  // top-k: a key with the segment's share of k entries at or above; greedy: index; keys of the cut's part
    uint64_t kept, pad;
    union {
        uint64_t list[kSegList];      // top-k: key << 32 | index, in index order
        uint64_t part[kSegPart];      // nucleus: the entries of the cut's part, the same way (any order)
    };
};

// Records are written and read with device-scope relaxed atomics, which go through to (come from) the
// level all XCDs share; a wave's stores are acknowledged before it lets its workgroup count itself
// (published), so whoever sees the count reads them. (Fences of that scope would write back and
// invalidate the XCD's whole L2 each time: with fences 634 us where it took 91 without, 64 nucleus rows
// of 151936 entries.)
template <class T>
__device__ __forceinline__ void put(T& at, T x) {
    __hip_atomic_store(&at, x, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
template <class T>
__device__ __forceinline__ T get(const T& at) {
    return __hip_atomic_load(&at, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void sum_up(uint64_t& at, uint64_t x) {
    __hip_atomic_fetch_add(&at, x, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void published() {
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
}

// One count at *w once everything this workgroup put is visible; true in the last of S.
__device__ __forceinline__ bool arrive_last(uint32_t* w, int S, const BlkW& g, WideSmem& s) {
    published();
    if (g.t == 0) s.wcomp[0] = __hip_atomic_fetch_add(w, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == (uint32_t)S - 1;
    __syncthreads();
    return s.wcomp[0] != 0;
}
// All S workgroups of the row (true), or the row was given up (false for all of them).
__device__ __forceinline__ bool meet(uint32_t* w, int S, uint32_t ticks, const BlkW& g, WideSmem& s) {
    published();
    if (g.t == 0) {
        uint32_t cur = __hip_atomic_fetch_add(w, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        cur = cur & kAbandoned ? cur : cur + 1;
        const uint64_t t0 = __builtin_amdgcn_s_memrealtime();
        while (!(cur & kAbandoned) && cur != (uint32_t)S) {
            if (__builtin_amdgcn_s_memrealtime() - t0 > ticks) {
                if (__hip_atomic_compare_exchange_strong(w, &cur, cur | kAbandoned, __ATOMIC_RELAXED, __ATOMIC_RELAXED,
                                                         __HIP_MEMORY_SCOPE_AGENT))
                    cur |= kAbandoned;
                continue;  // on failure cur holds the count now: complete, abandoned or higher
            }
            __builtin_amdgcn_s_sleep(1);
            cur = get(*w);
        }
        s.wcomp[0] = cur == (uint32_t)S;
    }
    __syncthreads();
    return s.wcomp[0] != 0;
}

// The bitmap (bit i - lo) of the row's history ids inside [lo, lo + len), len a multiple of 32; false when
// any id lies outside [0, V). `first` holds the ids at h0 + thread + 256 k, loaded ahead. All threads
// call it.
constexpr int kIdsAhead = 8;
__device__ __forceinline__ bool build_segment_bitmap(const BlkW& g, const SampleArgs& a, const HistRange& hr, int V, int lo, int len,
                                                     const int (&first)[kIdsAhead], uint32_t* bm) {
    for (int w = g.t; w < len / 32; w += kTW) bm[w] = 0;
    __syncthreads();
    bool bad = false;
    auto mark = [&](int h, int id) {
        const unsigned o = (unsigned)(id - lo);
        bad |= h < hr.h1 && (unsigned)id >= (unsigned)V;
        if (h < hr.h1 && o < (unsigned)len) atomicOr(&bm[o >> 5], 1u << (o & 31));
    };
#pragma unroll
    for (int k = 0; k < kIdsAhead; k++) mark(hr.h0 + k * kTW + g.t, first[k]);
    for (int hb = hr.h0 + kIdsAhead * kTW; hb < hr.h1; hb += 8 * kTW) {  // eight ids per thread in flight
        int id[8];
#pragma unroll
        for (int k = 0; k < 8; k++) {
            const int h = hb + k * kTW + g.t;
            id[k] = h < hr.h1 ? a.hist_ids[h] : 0;
        }
#pragma unroll
        for (int k = 0; k < 8; k++) mark(hb + k * kTW + g.t, id[k]);
    }
    return !g.any(bad);
}

// The segment that holds position p of the concatenated lists: before[] (LDS) the positions before each.
__device__ __forceinline__ int segment_at(const uint32_t* before, uint32_t p) {
    int sg = 0;
#pragma unroll
    for (int step = kSplitMaxSegs / 2; step; step >>= 1)  // (before[] holds the total from S on)
        sg += before[sg + step] <= p ? step : 0;
    return sg;
}

// Top-k finish, by the last workgroup to arrive: the segments' lists through the waves (a quarter of the
// segments each) into registers in index order, then the ordered pass's tail. True: the general algorithm
// must sample the row (nothing written).
__device__ __forceinline__ bool split_topk_finish(const SampleArgs& a, int vec, int r, const vxs_params& P, const RowX& X, BlkW& g,
                                                  WideSmem& s, const SplitSeg* segs, int S, const float* __restrict__ xrow, double u) {
    const int K = P.top_k;
    const bool in = g.lane < S;
    const uint32_t my_n = in ? get(segs[g.lane].n) : 0u;
    const uint32_t cnt = wave_sum(in ? get(segs[g.lane].cnt) : 0u);
    const uint32_t bad = in ? get(segs[g.lane].bad) : 0u;
    const uint32_t tau = wave_umin(in ? get(segs[g.lane].bkey) : 0xffffffffu);  // at least K entries reach it
    if (__ballot((bad & 2u) != 0)) {
        if (g.t == 0) put_id(a, r, VXS_ERR_ID_OUT_OF_RANGE);
        return false;
    }
    if (__ballot(bad != 0)) {
        if (g.t == 0) put_id(a, r, VXS_ERR_NONFINITE);
        return false;
    }
    if (cnt == 0) {  // every entry -inf: the reference's draw returns the last id
        if (g.t == 0) put_id(a, r, a.vocab - 1);
        return false;
    }
    if (__ballot(my_n > (uint32_t)kSegList)) return true;  // more entries than a list holds: ties, mostly
    uint32_t* wkey = s.wkey[g.wv];
    int32_t* widx = s.widx[g.wv];
    int wn = 0;
    uint32_t bound = tau;
    bool ok = true;
    // keep the entries of the full buffer at or above a lower bound of their k-th largest
    auto compact = [&]() {
        wave_sync();
        uint32_t kk[kPerL];
        int32_t ii[kPerL];
        uint32_t klo = 0xffffffffu, khi = 0;
#pragma unroll
        for (int q = 0; q < kPerL; q++) {
            const bool have = g.lane + 64 * q < wn;
            kk[q] = have ? wkey[g.lane + 64 * q] : 0u;
            ii[q] = widx[g.lane + 64 * q];
            klo = have ? min(klo, kk[q]) : klo;
            khi = max(khi, kk[q]);
        }
        bound = max(bound, wave_bound_regs(kk, wave_umin(klo), wave_umax(khi), K, 32));
        wave_sync();
        uint32_t m = 0;
#pragma unroll
        for (int q = 0; q < kPerL; q++) {
            const bool keep = kk[q] >= bound && kk[q] != 0u;
            const uint64_t bal = __ballot(keep);
            if (keep) {
                const uint32_t pos = m + __builtin_amdgcn_mbcnt_hi((uint32_t)(bal >> 32),
                                                                   __builtin_amdgcn_mbcnt_lo((uint32_t)bal, 0u));
                wkey[pos] = kk[q];
                widx[pos] = ii[q];
            }
            m += (uint32_t)__builtin_popcountll(bal);
        }
        wave_sync();
        wn = __builtin_amdgcn_readfirstlane((int)m);
    };
    // the concatenated lists, a quarter of the positions per wave, ten 64-entry pieces in flight
    uint32_t* before = reinterpret_cast<uint32_t*>(&s.ex.cp[0]);
    const uint32_t incl = wave_incl_sum(my_n), N = readlane(incl, 63);
    if (g.wv == 0) before[g.lane] = incl - my_n;
    __syncthreads();
    constexpr int kAt = 10;
    const uint32_t p1 = (uint32_t)((uint64_t)N * (g.wv + 1) / kWW);
#pragma unroll 1
    for (uint32_t p0 = (uint32_t)((uint64_t)N * g.wv / kWW); p0 < p1; p0 += 64 * kAt) {
        uint64_t e[kAt];
#pragma unroll
        for (int q = 0; q < kAt; q++) {
            const uint32_t p = min(p0 + 64 * q + g.lane, p1 - 1);  // unconditional, so that the searches overlap
            const int sg = segment_at(before, p);
            e[q] = get(segs[sg].list[p - before[sg]]);
        }
#pragma unroll
        for (int q = 0; q < kAt; q++) e[q] = p0 + 64 * q + g.lane < p1 ? e[q] : 0ull;
#pragma unroll
        for (int q = 0; q < kAt; q++) {
            const uint32_t key = (uint32_t)(e[q] >> 32);
            int c = __builtin_popcountll(__ballot(key >= bound && key != 0u));
            if (wn + c > kCapW && ok) {
                compact();
                c = __builtin_popcountll(__ballot(key >= bound && key != 0u));
                ok = wn + c <= kCapW;
            }
            const bool keep = ok && key >= bound && key != 0u;
            const uint64_t bal = __ballot(keep);
            if (keep) {
                const uint32_t pos = (uint32_t)wn + __builtin_amdgcn_mbcnt_hi((uint32_t)(bal >> 32),
                                                                             __builtin_amdgcn_mbcnt_lo((uint32_t)bal, 0u));
                wkey[pos] = key;
                widx[pos] = (int32_t)(uint32_t)e[q];
            }
            wn = __builtin_amdgcn_readfirstlane(wn + (int)__builtin_popcountll(bal));
        }
    }
    wave_sync();
    uint32_t kk[kPerL];
    int32_t ii[kPerL];
    uint32_t klo = 0xffffffffu, khi = 0;
#pragma unroll
    for (int q = 0; q < kPerL; q++) {
        const bool have = g.lane + 64 * q < wn;
        kk[q] = have ? wkey[g.lane + 64 * q] : 0u;
        ii[q] = widx[g.lane + 64 * q];
        klo = have ? min(klo, kk[q]) : klo;
        khi = max(khi, kk[q]);
    }
    klo = wave_umin(klo);
    khi = wave_umax(khi);
    if (g.lane == 0) {
        s.wklo[g.wv] = klo;
        s.wkhi[g.wv] = khi;
        s.wbad[g.wv] = ok ? 0 : 1;
    }
    s.h.h3[g.t] = 0u;  // the first histogram of the k-th largest select
    __syncthreads();
    bool any_full = false;
#pragma unroll
    for (int w = 0; w < kWW; w++) {
        klo = min(klo, s.wklo[w]);
        khi = max(khi, s.wkhi[w]);
        any_full = any_full || s.wbad[w] != 0;
    }
    if (any_full) return true;
    return ordered_tail(a, vec, r, P, X, g, s, kk, ii, klo, khi, K, (uint32_t)K < cnt, g.wv == 0, nullptr, nullptr, xrow, [&]() { return u; });
}

// What is left to do for a row when its workgroup's part is done.
enum SplitEnd : int {
    kEndGone,      // nothing (the row's counters are clear, or another workgroup of the row sees to them)
    kEndGeneral,   // as kEndGone, but this workgroup must sample the row with the general algorithm
    kEndLeave,     // leave with the others: the last clears the counters ...
    kEndUnsampled  // ... and samples the row with the general algorithm (every workgroup of the row ends so)
};

template <int NC>
__device__ __forceinline__ SplitEnd split_row(const SampleArgs& a, int vec, int r, int seg, int S, SplitRow& row, SplitSeg* segs,
                                              BlkW& g, WideSmem& s, uint32_t* bm_dyn) {
    // the nucleus stages' arrays over the candidate buffers and the exact regime's
    uint64_t* lds64 = reinterpret_cast<uint64_t*>(&s.wkey[0][0]);
    static_assert(offsetof(WideSmem, slot) >= sizeof(uint64_t) * kFineMass, "histogram storage");
    static_assert(kFineMass >= 2 * kRowPart + kSplitMaxSegs + kSplitMaxSegs / 2 + 256 + kRowPart / 2, "list storage");
    static_assert(sizeof(uint64_t) * (kFineMass - kSub) >= sizeof(int32_t) * kMine, "index storage");
    constexpr int L = 1024 * NC, NE = 4 * NC;
    SplitSeg& me = segs[seg];
    const int V = a.vocab;
    const float* __restrict__ xrow = a.logits + (int64_t)r * a.ld;
    const int lo = seg * L, hi = min(V, lo + L);

    // ---- the segment, read once (raw buffer loads bounded by its end: entries past it read zero)
    typedef float f4 __attribute__((ext_vector_type(4)));
    const __amdgpu_buffer_rsrc_t rowbuf =
        __builtin_amdgcn_make_buffer_rsrc((void*)xrow, (short)0, hi * (int)sizeof(float), 0x00020000);
    float v[NE];
#pragma unroll
    for (int c = 0; c < NC; c++) {
        const f4 q = __builtin_bit_cast(f4, __builtin_amdgcn_raw_buffer_load_b128(rowbuf, (lo + 1024 * c + 4 * g.t) * 4, 0, 2));
#pragma unroll
        for (int j = 0; j < 4; j++) v[4 * c + j] = q[j];
    }
    // A row without a penalty reads nothing of its history (a caller need not have filled it); with one,
    // the first ids are on their way while the segment is.
    const vxs_params P = a.params[(int64_t)r * a.params_stride];
    const bool pen_on = P.rep_penalty != 1.0f && has_history(a);
    HistRange hr{0, 0};
    if (pen_on) hr = history_range(a, r);
    int first[kIdsAhead];
#pragma unroll
    for (int k = 0; k < kIdsAhead; k++) {
        const int h = hr.h0 + k * kTW + g.t;
        first[k] = h < hr.h1 ? a.hist_ids[h] : 0;
    }
    const bool greedy = !P.do_sample;
    const double u = greedy ? 0.0 : readlane_d(row_uniform(a, r), 0);  // before any workgroup can end the row's step
    RowX X;
    X.bm = nullptr;
    X.rho = P.rep_penalty;
    X.rinv = 1.0f / P.rep_penalty;
    X.fastdiv = __builtin_fabsf(P.rep_penalty) >= 0x1p-60f && __builtin_fabsf(P.rep_penalty) <= 0x1p60f;
    bool bad_id = false;
    if (pen_on) {
        bad_id = !build_segment_bitmap(g, a, hr, V, lo, L, first, bm_dyn);
        X.bm = bm_dyn - (lo >> 5);  // indexed by vocabulary entry
    }
    X.sb = max(P.supp_begin, 0);
    X.se = min(P.supp_end, V);
    if (!(P.supp_begin < P.supp_end)) X.sb = X.se = 0;
    X.keep = P.keep_id;
    X.ban = P.ban_id;
    X.invT = row_inv_temp(P);

    // ---- S1-S4 in registers; statistics
    bool bad = false;
    float tmx = kNegInf;
    int bi = 0x7fffffff;  // greedy: the first index of this thread's largest entry
    uint32_t fin = 0;     // wave-uniform count of finite entries
#pragma unroll
    for (int c = 0; c < NC; c++) {
        const int base = lo + 1024 * c, i0 = base + 4 * g.t;
        if (X.bm) {
            const uint32_t nib = (X.bm[i0 >> 5] >> (i0 & 31)) & 15u;
            if (nib) {
#pragma unroll
                for (int j = 0; j < 4; j++)
                    if ((nib >> j) & 1u) v[4 * c + j] = penalize(v[4 * c + j], X.rho, X.rinv, X.fastdiv);
            }
        }
        if ((base < X.se && base + 1024 > X.sb) || (X.ban >= base && X.ban < base + 1024)) {
#pragma unroll
            for (int j = 0; j < 4; j++) {
                const int i = i0 + j;
                if ((i >= X.sb && i < X.se && i != X.keep) || i == X.ban) v[4 * c + j] = kNegInf;
            }
        }
#pragma unroll
        for (int j = 0; j < 4; j++) v[4 * c + j] *= X.invT;
        if (base + 1024 > hi) {
#pragma unroll
            for (int j = 0; j < 4; j++) v[4 * c + j] = i0 + j < hi ? v[4 * c + j] : kNegInf;
        }
        if (greedy) {
#pragma unroll
            for (int j = 0; j < 4; j++) {
                bad |= v[4 * c + j] != v[4 * c + j];
                const bool take = i0 + j < hi && (v[4 * c + j] > tmx || bi == 0x7fffffff);
                tmx = take ? v[4 * c + j] : tmx;
                bi = take ? i0 + j : bi;
            }
        } else {
#pragma unroll
            for (int j = 0; j < 4; j++) {
                bad |= __builtin_amdgcn_class(v[4 * c + j], 0x203);  // NaN or +inf
                tmx = fmaxf(tmx, v[4 * c + j]);
                fin += (uint32_t)__builtin_popcountll(__ballot(v[4 * c + j] != kNegInf));
            }
        }
        __builtin_amdgcn_sched_barrier(0);
    }
    const uint32_t badw = (wave_any(bad) ? 1u : 0u) | (bad_id ? 2u : 0u);
    const uint32_t badf = (uint32_t)g.combine(badw, [](uint64_t p, uint64_t q) { return p | q; });
    const int K = P.top_k;

    if (greedy) {
        const float wbv = wave_fmax(tmx);
        const uint32_t wbi = wave_umin(tmx == wbv ? (uint32_t)bi : 0xffffffffu);
        if (g.lane == 0) {
            s.slot[2][g.wv] = f2key(wbv);
            s.slot[3][g.wv] = wbi;
        }
        __syncthreads();
        if (g.t == 0) {
            uint32_t best = 0, besti = 0xffffffffu;
            for (int w = 0; w < kWW; w++) {
                const uint32_t k = (uint32_t)s.slot[2][w], i = (uint32_t)s.slot[3][w];
                if (k > best || (k == best && i < besti)) {
                    best = k;
                    besti = i;
                }
            }
            put(me.maxkey, best);
            put(me.argi, besti);
            put(me.bad, badf);
        }
        if (!arrive_last(&row.meet[0], S, g, s)) return kEndGone;
        if (g.t == 0) put(row.meet[0], 0u);
        if (g.wv != 0) return kEndGone;
        const bool in = g.lane < S;
        const uint32_t flags = in ? get(segs[g.lane].bad) : 0u, key = in ? get(segs[g.lane].maxkey) : 0u;
        const uint32_t best = wave_umax(key);
        const uint32_t besti = wave_umin(in && key == best ? get(segs[g.lane].argi) : 0xffffffffu);
        const bool bid = __ballot((flags & 2u) != 0) != 0, nan = __ballot(flags != 0) != 0;
        if (g.lane == 0) put_id(a, r, bid ? VXS_ERR_ID_OUT_OF_RANGE : nan ? VXS_ERR_NONFINITE : (int)besti);
        return kEndGone;
    }
    const uint32_t cnt = (uint32_t)g.combine(fin, [](uint64_t p, uint64_t q) { return p + q; });

    if (K > 0 && K <= kKMax && K < V) {
        // ---- top-k: this segment's entries at or above a lower bound of its k-th largest (all finite ones
        // when there are at most k): the k-th largest of the thread maxima. As k nears their number the bound
        // falls to the least of them and the list overflows, at once for k from 250 on; two maxima per
        // thread, of the even and of the odd sweeps, keep it. Their search takes 2 us more, which rows of many
        // segments get back from shorter lists (us, one / two: 16 x 151936 k = 150 34.9 / 34.3, 200 43.8 / 38.8,
        // 240 62 / 44, 256 182 / 48; 64 x 20000 k = 200 24.6 / 27.4, 240 29.3 / 28.6, 256 82 / 29.4; 1 x 8193
        // k = 200 22.1 / 24.2, 240 23.1 / 25.1, 256 55 / 25.6).
        // this segment's share of k by length: the shares add up to k and more, and a short last segment's
        // is no harder to reach than the others' (64 x 9001, the same share for all: k = 50 17.1 -> 16.6, 240 28.6 -> 27.6)
        const int Kq = (K * (hi - lo) + V - 1) / V;
        float Tb = kNegInf;
        uint32_t bq = 0;  // a key of which at least Kq entries of this segment are at or above (0: fewer are finite)
        float* tm = reinterpret_cast<float*>(&s.wkey[0][0]);
        auto bounds = [&](auto per_thread) {
            constexpr int N = decltype(per_thread)::value * kTW / 64;
            __syncthreads();
            uint32_t mk[N];
            uint32_t mlo = 0xffffffffu, mhi = 0;
#pragma unroll
            for (int q = 0; q < N; q++) {
                mk[q] = f2key(tm[g.lane + 64 * q]);
                mlo = min(mlo, mk[q]);
                mhi = max(mhi, mk[q]);
            }
            mlo = wave_umin(mlo);
            mhi = wave_umax(mhi);
            if (cnt > (uint32_t)K) Tb = key2f(wave_bound_regs4(mk, mlo, mhi, K, 8));
            if (cnt >= (uint32_t)Kq) bq = wave_bound_regs4(mk, mlo, mhi, Kq, 4);
        };
        if (K <= (S > 5 ? 192 : 240)) {
            tm[g.t] = tmx;
            bounds(std::integral_constant<int, 1>());
        } else {
            float odd = kNegInf;
            tmx = kNegInf;
#pragma unroll
            for (int c = 0; c < NC; c++)
#pragma unroll
                for (int j = 0; j < 4; j++) (c & 1 ? odd : tmx) = fmaxf(c & 1 ? odd : tmx, v[4 * c + j]);
            tm[g.t] = tmx;
            tm[kTW + g.t] = odd;
            bounds(std::integral_constant<int, 2>());
        }
        constexpr int NH = (NC + 3) / 4;
        uint64_t excl[NH], totals[NH];
        uint32_t tot = 0;
#pragma unroll
        for (int h = 0; h < NH; h++) {
            uint64_t mine = 0;  // 16-bit counts per sweep, four sweeps a scan
#pragma unroll
            for (int c = 4 * h; c < NC && c < 4 * h + 4; c++) {
                uint32_t m = 0;
#pragma unroll
                for (int j = 0; j < 4; j++) m += v[4 * c + j] >= Tb && v[4 * c + j] != kNegInf ? 1u : 0u;
                mine |= (uint64_t)m << (16 * (c - 4 * h));
            }
            excl[h] = g.excl(mine, totals[h]);
#pragma unroll
            for (int c = 4 * h; c < NC && c < 4 * h + 4; c++) tot += (uint32_t)((totals[h] >> (16 * (c - 4 * h))) & 0xffffu);
        }
        if (tot <= (uint32_t)kSegList) {
            uint32_t base = 0;
#pragma unroll
            for (int c = 0; c < NC; c++) {
                const int h = c / 4, f = 16 * (c % 4);
                uint32_t off = base + (uint32_t)((excl[h] >> f) & 0xffffu);
#pragma unroll
                for (int j = 0; j < 4; j++)
                    if (v[4 * c + j] >= Tb && v[4 * c + j] != kNegInf)
                        put(me.list[off++], ((uint64_t)f2key(v[4 * c + j]) << 32) | (uint32_t)(lo + 1024 * c + 4 * g.t + j));
                base += (uint32_t)((totals[h] >> f) & 0xffffu);
            }
        }
        if (g.t == 0) {
            put(me.n, tot <= (uint32_t)kSegList ? tot : 0xffffffffu);
            put(me.cnt, cnt);
            put(me.bad, badf);
            put(me.bkey, bq);
        }
        if (!arrive_last(&row.meet[0], S, g, s)) return kEndGone;
        if (g.t == 0) put(row.meet[0], 0u);
        return split_topk_finish(a, vec, r, P, X, g, s, segs, S, xrow, u) ? kEndGeneral : kEndGone;
    }

    // ---- nucleus. Meeting 0: the row's maximum and finite count
    const bool topp = P.top_p < 1.0f;
    {
        const float wmx = wave_fmax(tmx);
        if (g.lane == 0) s.slot[2][g.wv] = f2key(wmx);
        for (int i = g.t; i < kFineMass; i += kTW) lds64[i] = 0;
        __syncthreads();
        if (g.t == 0) {
            put(me.maxkey, max(max((uint32_t)s.slot[2][0], (uint32_t)s.slot[2][1]), max((uint32_t)s.slot[2][2], (uint32_t)s.slot[2][3])));
            put(me.cnt, cnt);
            put(me.bad, badf);
        }
    }
    const bool in = g.lane < S;  // lane l of every wave reads segment l's record
    if (!meet(&row.meet[0], S, a.meet_ticks, g, s)) return kEndUnsampled;
    float mx;
    bool count_first;  // top-k above kKMax: the k-th largest first, by the same stages over counts
    {
        const uint32_t flags = in ? get(segs[g.lane].bad) : 0u;
        const uint32_t rcnt = wave_sum(in ? get(segs[g.lane].cnt) : 0u);
        mx = key2f(wave_umax(in ? get(segs[g.lane].maxkey) : 0u));
        const bool bid = __ballot((flags & 2u) != 0) != 0, nf = __ballot(flags != 0) != 0;
        if (bid || nf || rcnt == 0) {  // (every entry -inf: the reference's draw returns the last id)
            if (seg == 0 && g.t == 0) put_id(a, r, bid ? VXS_ERR_ID_OUT_OF_RANGE : nf ? VXS_ERR_NONFINITE : V - 1);
            return kEndLeave;
        }
        count_first = K > 0 && K < V && (uint32_t)K < rcnt;
    }
    const double thr = (double)(1.0f - P.top_p);
    if (topp && !(thr < 1.0)) return kEndUnsampled;

    // ---- masses in place of the values: multiples of 2^-F, as integers of that unit
    const int F = min(51, 53 - (32 - __clz(V - 1)));
    const float Cb = mass_bias(F);
    const double unit = __builtin_ldexp(1.0, 52 - F);
    auto units = [&](float q) -> uint64_t {
        asm volatile("" : "+v"(q));  // formed where it is used: 64 bits per entry are not kept
        return (uint64_t)__double_as_longlong((double)q + unit) - (uint64_t)__double_as_longlong(unit);
    };
    auto part_of = [](float q) -> uint32_t {
        asm volatile("" : "+v"(q));  // (the same)
        return __float_as_uint(q) >> 14;
    };
    const uint32_t base17 = (uint32_t)(127 - F) << 6;  // bits >> 17 of the smallest mass, 2^-F
#pragma unroll
    for (int c = 0; c < NC; c++) {
#pragma unroll
        for (int j = 0; j < 4; j++) v[4 * c + j] = mass_of(exp_neg(v[4 * c + j] - mx), Cb);
        __builtin_amdgcn_sched_barrier(0);  // (kept apart: the registers must hold two sweeps' work, not all)
    }
    uint32_t qcut = 0;        // bits >> 14 of the cut's part; the masses above it are kept, those in it ...
    uint32_t ckey = 0;        // ... from (key, index) = (ckey, cidx) on
    uint32_t cidx = 0;
    bool tied = false;        // all of the cut's part have one key
    int own_n = 0;            // this segment's entries of the part
    double kept_l = 0.0;      // lane l: the kept mass of segment l
    // The entries that go, by a bit each in LDS: those of the cut's part that are below (ckey, cidx) (with
    // ties the ones before the cut index, else this segment's list decides).
    auto drop = [&]() {
        uint32_t* gone = reinterpret_cast<uint32_t*>(lds64);
        __syncthreads();
        for (int w = g.t; w < L / 32; w += kTW) {
            const int k = tied ? min(max((int)cidx - (lo + 32 * w), 0), 32) : 0;
            gone[w] = k == 32 ? ~0u : (1u << k) - 1u;
        }
        __syncthreads();
        if (!tied) {
            for (int j = g.t; j < own_n; j += kTW) {
                const uint64_t k = get(me.part[j]);
                const uint32_t o = (uint32_t)k - (uint32_t)lo;
                if (k < (((uint64_t)ckey << 32) | cidx)) atomicOr(&gone[o >> 5], 1u << (o & 31));
            }
            __syncthreads();
        }
#pragma unroll
        for (int c = 0; c < NC; c++) {
            const uint32_t nib = gone[32 * c + (g.t >> 3)] >> (4 * (g.t & 7));
#pragma unroll
            for (int j = 0; j < 4; j++) {
                const uint32_t q = part_of(v[4 * c + j]);
                const uint32_t first_kept = qcut + ((nib >> j) & 1u);
                v[4 * c + j] = q < first_kept ? 0.0f : v[4 * c + j];
            }
            __builtin_amdgcn_sched_barrier(0);
        }
        __syncthreads();
    };
    // Stage 0 (top-k above kKMax): weights 1, the cut at the k-th largest value, ties kept; entries of mass
    // zero count as below it (they have no part in any sum). Stage 1: the top-p cut, weights the masses.
    auto locate = [&](auto which) -> bool {
        constexpr int stage = decltype(which)::value;
        uint32_t* meets = &row.meet[1 + 3 * stage];
        auto weight = [&](float q) -> uint64_t { return stage ? units(q) : 1ull; };
#pragma unroll
        for (int e = 0; e < NE; e++) {
            if (e % 4 == 0) __builtin_amdgcn_sched_barrier(0);
            const uint32_t b = __float_as_uint(v[e]);
            if (b) atomicAdd((unsigned long long*)&lds64[(b >> 17) - base17], (unsigned long long)weight(v[e]));
        }
        __syncthreads();
        uint64_t own = 0;  // thread t: this segment's mass in bucket t
        if (g.t < kCoarse) {
#pragma unroll
            for (int i = 0; i < 16; i++) own += lds64[16 * g.t + ((i + g.t) & 15)];
            if (own) sum_up(row.coarse[stage][g.t], own);
        }
        if (!meet(&meets[0], S, a.meet_ticks, g, s)) return false;
        // the bucket where the ascending cumulative mass crosses T
        auto crossing = [&](uint64_t h, double rest, double& below, double& total) -> int {
            const double run = g.excl((double)h, total);
            // (rest negative: T itself is sought)
            const double t0 = rest >= 0.0 ? rest : stage ? floor(thr * total) : total - (double)K;
            if (h != 0 && run <= t0 && t0 - run < (double)h) {
                s.wcand[0] = g.t;
                s.slot[2][0] = (uint64_t)__double_as_longlong(run);
            }
            __syncthreads();
            total = readlane_d(total, 0);  // (uniform: in scalar registers from here)
            below = readlane_d(__longlong_as_double((long long)s.slot[2][0]), 0);
            return __builtin_amdgcn_readfirstlane(s.wcand[0]);
        };
        uint64_t h = g.t < kCoarse ? get(row.coarse[stage][g.t]) : 0ull;
        double below, total;
        const int bc = crossing(h, -1.0, below, total);
        const double T = stage ? floor(thr * total) : total - (double)K;
        if (T >= total) return false;  // top-p so small that only the last entry stays
        if (T < 0.0) {                         // at most K entries have mass: all of them stay
            __syncthreads();
            for (int i = g.t; i < kFineMass; i += kTW) lds64[i] = 0;
            __syncthreads();
            return true;
        }
        double kept = readlane_d(g.dsum(g.t > bc ? (double)own : 0.0), 0);  // this segment's mass above the bucket
        // its 128 parts
        if (g.t < kSub) lds64[g.t] = 0;
        __syncthreads();
        const uint32_t q21 = (uint32_t)bc + (base17 >> 4);
#pragma unroll
        for (int e = 0; e < NE; e++) {
            if (e % 4 == 0) __builtin_amdgcn_sched_barrier(0);
            const uint32_t b = __float_as_uint(v[e]);
            if ((b >> 21) == q21) atomicAdd((unsigned long long*)&lds64[(b >> 14) & (kSub - 1)], (unsigned long long)weight(v[e]));
        }
        __syncthreads();
        own = g.t < kSub ? lds64[g.t] : 0;
        if (own) sum_up(row.sub[stage][g.t], own);
        if (!meet(&meets[1], S, a.meet_ticks, g, s)) return false;
        h = g.t < kSub ? get(row.sub[stage][g.t]) : 0ull;
        double sub_below, sub_total;
        const int bf = crossing(h, T - below, sub_below, sub_total);
        below += sub_below;
        qcut = (q21 << 7) + (uint32_t)bf;
        kept += readlane_d(g.dsum(g.t > bf ? (double)own : 0.0), 0);
        // the part's entries as (d, index) keys (stage 0: by value): their indices first, then their values
        // read again, all at once (few: one each per thread)
        auto key_of = [&](int i) -> uint32_t {
            const float x = X(i, xrow[i]);
            return f2key(stage ? x - mx : x);
        };
        auto mass_of_key = [&](uint32_t key) -> float { return mass_of(exp_neg(stage ? key2f(key) : key2f(key) - mx), Cb); };
        if (g.t == 0) s.n = 0;
        int32_t* mine = reinterpret_cast<int32_t*>(lds64 + kSub);  // indices of this segment's entries of the part
        __syncthreads();
#pragma unroll
        for (int c = 0; c < NC; c++) {
            bool is[4];
            int n4 = 0;
#pragma unroll
            for (int j = 0; j < 4; j++) {
                is[j] = part_of(v[4 * c + j]) == qcut;
                n4 += is[j] ? 1 : 0;
            }
            if (n4) {
                int at = atomicAdd(&s.n, n4);
#pragma unroll
                for (int j = 0; j < 4; j++)
                    if (is[j]) mine[at++ & (kMine - 1)] = lo + 1024 * c + 4 * g.t + j;
            }
            __builtin_amdgcn_sched_barrier(0);
        }
        __syncthreads();
        uint32_t kmin = 0xffffffffu, kmax = 0;
        own_n = __builtin_amdgcn_readfirstlane(s.n);
        if (own_n <= kMine) {
            for (int j = g.t; j < own_n; j += kTW) {
                const int i = mine[j];
                const uint32_t key = key_of(i);
                kmin = min(kmin, key);
                kmax = max(kmax, key);
                if (j < kSegPart) put(me.part[j], ((uint64_t)key << 32) | (uint32_t)i);
            }
        } else {  // many: ties, most likely; each thread reads its own
#pragma unroll 4
            for (int e = 0; e < NE; e++) {
                const int i = lo + 1024 * (e / 4) + 4 * g.t + (e & 3);
                bool in_part = false;
#pragma unroll
                for (int q = 0; q < NE; q++) in_part |= q == e && part_of(v[q]) == qcut;
                const uint32_t key = in_part ? key_of(i) : 0u;
                kmin = in_part ? min(kmin, key) : kmin;
                kmax = max(kmax, key);
            }
        }
        kmin = g.umin(kmin);
        kmax = g.umax(kmax);
        if (g.t == 0) {
            put(me.n, (uint32_t)own_n);
            put(me.kmin, kmin);
            put(me.kmax, kmax);
            put(me.kept, (uint64_t)kept);
        }
        if (!meet(&meets[2], S, a.meet_ticks, g, s)) return false;
        const uint32_t n_l = in ? get(segs[g.lane].n) : 0u;
        const uint32_t n = wave_sum(n_l);
        kept_l = in ? (double)get(segs[g.lane].kept) : 0.0;
        kmin = wave_umin(in ? get(segs[g.lane].kmin) : 0xffffffffu);
        kmax = wave_umax(in ? get(segs[g.lane].kmax) : 0u);
        tied = kmin == kmax;
        if (tied) {
            // one key (ties, or one entry): the crossing follows index order among them
            const double w = (double)weight(mass_of_key(kmin));
            const uint32_t nth = (uint32_t)((T - below) / w);  // entries of the part that go (exact integers)
            const uint32_t before = wave_incl_sum(n_l) - n_l;
            const uint32_t go_l = min(n_l, nth > before ? nth - before : 0u);
            kept_l += w * (double)(n_l - go_l);
            ckey = kmin;
            const uint32_t go = readlane(go_l, seg);  // this segment's first `go` tied entries in index order go
            cidx = 0;
            if (!stage) {
                // (ties at the k-th largest are kept)
            } else if (go == (uint32_t)own_n) {
                cidx = 0x7fffffffu;
            } else if (go) {  // uniform: the index of entry number `go` among them
                uint32_t run = 0;
#pragma unroll 1
                for (int c = 0; c < NC; c++) {
                    uint32_t m4 = 0;
#pragma unroll
                    for (int e = 0; e < NE; e++)
                        if (e / 4 == c) m4 |= part_of(v[e]) == qcut ? 1u << (e & 3) : 0u;
                    uint32_t t4;
                    const uint32_t ex = run + g.excl((uint32_t)__builtin_popcount(m4), t4);
                    if (go >= ex && go < ex + (uint32_t)__builtin_popcount(m4)) {
                        for (uint32_t k = go - ex; k; k--) m4 &= m4 - 1;
                        s.wcand[1] = lo + 1024 * c + 4 * g.t + __builtin_ctz(m4);
                    }
                    run += t4;
                }
                __syncthreads();
                cidx = (uint32_t)s.wcand[1];
            }
        } else if (n > (uint32_t)kRowPart || __ballot(n_l > (uint32_t)kSegPart)) {
            return false;
        } else {
            uint64_t* list = lds64;                   // [n] keys
            uint64_t* mass = lds64 + kRowPart;        // [n] their masses
            uint64_t* kept_s = lds64 + 2 * kRowPart;  // [S]
            uint32_t* before = reinterpret_cast<uint32_t*>(kept_s + kSplitMaxSegs);  // [S]
            uint64_t* digit = lds64 + 2 * kRowPart + kSplitMaxSegs + kSplitMaxSegs / 2;  // [256] masses by the next 8 bits
            int32_t* few = reinterpret_cast<int32_t*>(digit + 256);                       // positions of the crossing digit's entries
            __syncthreads();
            if (g.wv == 0) before[g.lane] = wave_incl_sum(n_l) - n_l;
            if (g.t == 0) s.n = 0;
            digit[g.t] = 0;
            __syncthreads();
            if (g.t < S) kept_s[g.t] = get(segs[g.t].kept);
#pragma unroll 1
            for (uint32_t p = g.t; p < n; p += kTW) {  // (a few hundred entries at most: one round, mostly)
                const int sg = segment_at(before, p);
                const uint64_t k = get(segs[sg].part[p - before[sg]]);
                const float m = mass_of_key((uint32_t)(k >> 32));
                list[p] = k;
                mass[p] = weight(m);
                atomicAdd((unsigned long long*)&digit[(__float_as_uint(m) >> 6) & 255u], (unsigned long long)weight(m));
            }
            __syncthreads();
            // the digit that holds the crossing, then its entries (a few) compared with each other
            double digit_below, digit_total;
            const uint32_t dc = (uint32_t)crossing(digit[g.t], T - below, digit_below, digit_total);
#pragma unroll 1
            for (uint32_t p = g.t; p < n; p += kTW)
                if (((__float_as_uint(mass_of_key((uint32_t)(list[p] >> 32))) >> 6) & 255u) == dc)
                    few[atomicAdd(&s.n, 1)] = (int32_t)p;
            __syncthreads();
            const int m = s.n;
            const uint64_t rest = (uint64_t)(T - below - digit_below);
            for (int j = g.t; j < m; j += kTW) {
                const int pj = few[j];
                const uint64_t k = list[pj];
                uint64_t lower = 0;
                for (int i = 0; i < m; i++) lower += list[few[i]] < k ? mass[few[i]] : 0ull;
                if (lower <= rest && rest - lower < mass[pj]) s.slot[3][0] = k;  // exactly one entry
            }
            __syncthreads();
            const uint64_t cut = s.slot[3][0];
#pragma unroll 1
            for (uint32_t p = g.t; p < n; p += kTW)
                if (list[p] >= cut)
                    atomicAdd((unsigned long long*)&kept_s[(uint32_t)list[p] / (uint32_t)L], (unsigned long long)mass[p]);
            __syncthreads();
            kept_l = in ? (double)kept_s[g.lane] : 0.0;
            ckey = (uint32_t)(cut >> 32);
            cidx = stage ? (uint32_t)cut : 0u;
        }
        if (!stage) {
            drop();
            for (int i = g.t; i < kFineMass; i += kTW) lds64[i] = 0;  // stage 1's histogram
            __syncthreads();
        }
        return true;
    };
    if (count_first && !locate(std::integral_constant<int, 0>())) return kEndUnsampled;
    if (topp && !locate(std::integral_constant<int, 1>())) return kEndUnsampled;
    if (!topp) {
        double ls = 0.0;
#pragma unroll
        for (int e = 0; e < NE; e++) {
            if (e % 4 == 0) __builtin_amdgcn_sched_barrier(0);
            ls += (double)units(v[e]);
        }
        ls = g.dsum(ls);
        if (g.t == 0) put(me.kept, (uint64_t)ls);
        if (!meet(&row.meet[7], S, a.meet_ticks, g, s)) return kEndUnsampled;
        kept_l = in ? (double)get(segs[g.lane].kept) : 0.0;
    }

    // ---- draw: the first kept entry whose inclusive prefix mass exceeds floor(u * kept mass)
    const double incl = wave_incl_sum(kept_l);
    const double D = floor(u * readlane_d(incl, 63));
    const uint64_t holds = __ballot(D >= incl - kept_l && D - (incl - kept_l) < kept_l);
    if (!holds) return kEndUnsampled;  // no crossing (u at or above 1, NaN)
    if ((int)__builtin_ctzll(holds) != seg) return kEndLeave;
    const double rest = D - readlane_d(incl - kept_l, seg);
    if (topp) drop();
    double* sweep = reinterpret_cast<double*>(lds64);  // [NC][waves]
    __syncthreads();
#pragma unroll
    for (int c = 0; c < NC; c++) {
        double w = 0.0;
#pragma unroll
        for (int j = 0; j < 4; j++) w += (double)units(v[4 * c + j]);
        w = wave_sum(w);
        if (g.lane == 0) sweep[kWW * c + g.wv] = w;
    }
    __syncthreads();
    // (sweep, wave) that holds the draw, in index order
    static_assert(NC * kWW <= 64, "one lane each");
    const double sw = g.lane < NC * kWW ? sweep[g.lane] : 0.0;
    const double sw_before = wave_incl_sum(sw) - sw;
    const uint64_t holds_sw = __ballot(rest >= sw_before && rest - sw_before < sw);
    const int at = holds_sw ? (int)__builtin_ctzll(holds_sw) : 0;  // (one does: the sums are exact)
    const double run = readlane_d(sw_before, at);
    if (at % kWW == g.wv) {
        double w[4] = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
        for (int c = 0; c < NC; c++)
            if (c == at / kWW)
#pragma unroll
                for (int j = 0; j < 4; j++) w[j] = (double)units(v[4 * c + j]);
        const double mine = w[0] + w[1] + w[2] + w[3];
        double acc = run + wave_incl_sum(mine) - mine;
        if (rest >= acc && rest - acc < mine) {
            const double a1 = acc + w[0], a2 = a1 + w[1], a3 = a2 + w[2];
            const int j = rest < a1 ? 0 : rest < a2 ? 1 : rest < a3 ? 2 : 3;
            put_id(a, r, lo + 1024 * (at / kWW) + 4 * g.t + j);
        }
    }
    return kEndLeave;
}

template <int NC>
__global__ __launch_bounds__(kTW) __attribute__((amdgpu_waves_per_eu(4))) void sample_split_kernel(SampleArgs a, int vec, int S,
                                                                                                  SplitRow* rows, SplitSeg* all) {
    extern __shared__ uint32_t bm_dyn[];  // penalised-id bitmap (the general algorithm: of the whole row)
    __shared__ WideSmem s;
    BlkW g;
    g.t = threadIdx.x;
    g.lane = g.t & 63;
    g.wv = __builtin_amdgcn_readfirstlane(g.t >> 6);
    g.s = &s;
    const int r = (int)(blockIdx.x / (unsigned)S), seg = (int)(blockIdx.x % (unsigned)S);
    SplitRow& row = rows[r];
    SplitEnd end = split_row<NC>(a, vec, r, seg, S, row, all + (int64_t)r * S, g, s, bm_dyn);
    if (end == kEndGone) return;
    __syncthreads();
    if (end != kEndGeneral) {
        if (!arrive_last(&row.left, S, g, s)) return;
        // clear the row for the next call
        for (int i = g.t; i < 2 * kCoarse; i += kTW) put(row.coarse[0][i], uint64_t(0));
        for (int i = g.t; i < 2 * kSub; i += kTW) put(row.sub[0][i], uint64_t(0));
        if (g.t < 8) put(row.meet[g.t], 0u);
        if (g.t == 0) put(row.left, 0u);
        if (end == kEndLeave) return;
    }
    wide_general_row(a, vec, r, g, s, bm_dyn);
}
