// rs_tree.hip -- whole split trees of small buckets in one kernel.  Included by
// rs_engine.hip after the level kernels, whose group functions it uses.
//
// A bucket of 100 keys at l = 8 needs about 30,000 key evaluations over 20 nodes: as
// level launches (one for every tree level, with node lists, search states and a
// partition between levels) its nodes cost more in tickets, atomics on their state
// and memory round trips than in hashing (1M keys at l = 8, b = 100: 5,000 cycles per
// evaluation on the rotation level).  Here one wavefront takes a bucket through its
// whole tree with its keys in LDS: duplicate check, then node by node in DFS preorder
// the search, the partition of the keys and the descriptor length.  Nothing is shared
// between waves, so there are no atomics but the bucket tickets, and the node lists,
// the per-bucket sort and the expansion go.
//
// What it costs: a node is searched by one wave, so a bucket's time is its own chain
// of searches.  The host uses it where a bucket's expected work is small
// (tree_fits in rs_engine.hip).

namespace rsa {

struct TreeArgs {
    const uint64_t *acc;        // bucket key offsets, nb + 1
    const uint64_t *node_base;  // bucket slot offsets, nb + 1
    const uint64_t *sorted;     // `second` values grouped by bucket, any order inside
    uint64_t *seeds;
    uint16_t *node_m;
    uint64_t *bits;             // descriptor bits per bucket
    unsigned long long *evals;  // [0, kNumKinds) evaluations, [kNumKinds, 2 kNumKinds) seeds, as k_bucket_bits
    unsigned long long *work;   // executed evaluations per kind (kNumKinds)
    const uint32_t *memo;       // Golomb-Rice memo, then node counts by size
    uint32_t *err;
    uint32_t *ctl;              // [0] bucket tickets
    uint64_t nb;
    SplitParams P;
    int rotate;
    uint32_t min_m, max_m;      // bucket sizes this launch takes
    uint32_t cap;               // LDS keys of a bucket (>= max_m; a multiple of 8)
    uint32_t scratch;           // LDS bytes beside them (partition, duplicate table, a lone wave's staged queue)
    uint32_t queue;             // LDS bytes of a staged queue
    uint32_t batch;             // buckets per ticket
    uint32_t up_fb, up_magic, lo_fb, lo_magic;  // packed counters of the two aggregation levels (32 bits)
    const unsigned long long *clock0;  // time limit, as SearchArgs
    unsigned long long limit_ticks;
    const uint32_t *stop;
    uint32_t stop_mask;
    const uint32_t *max_bucket;  // optional: the largest bucket's size; below min_m the launch does nothing
};

// Entries of the duplicate table of a bucket of at most cap keys.
__host__ __device__ inline uint32_t tree_dup_entries(uint32_t cap) {
    uint32_t t = 64;
    while (t < 2 * cap) t <<= 1;
    return t;
}

__device__ __forceinline__ void lds_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// True if two of the m keys are equal: every key enters a hash table of key indexes
// (open addressing; the table has at least 2 m entries, so a probe sequence ends).
__device__ __forceinline__ bool tree_duplicates(const uint64_t *k, uint32_t m, uint32_t *table, uint32_t entries) {
    const uint32_t lane = lane_id();
    for (uint32_t i = lane; i < entries; i += 64) table[i] = 0xFFFFFFFFu;
    lds_sync();
    bool dup = false;
    const uint32_t shift = 32 - (31 - __clz(entries));
    for (uint32_t i = lane; i < m; i += 64) {
        const uint64_t key = k[i];
        uint32_t at = (((uint32_t)key ^ (uint32_t)(key >> 32) * 0x85ebca6bu) * 0x9E3779B1u) >> shift;
        for (;;) {
            const uint32_t j = atomicCAS(&table[at], 0xFFFFFFFFu, i);
            if (j == 0xFFFFFFFFu) break;
            if (k[j] == key) {
                dup = true;
                break;
            }
            at = (at + 1) & (entries - 1);
        }
    }
    lds_sync();
    return __ballot(dup) != 0;
}

// Orders kp[0, m) by child (child_of(key) < fan), keys with even `second` first
// inside every child (a full leaf's rotation halves), through tmp[0, m).
template <typename F>
__device__ __forceinline__ void tree_partition(uint64_t *kp, uint64_t *tmp, uint32_t m, uint32_t unit, uint32_t fan,
                                               F &&child_of) {
    const uint32_t lane = lane_id();
    const unsigned long long lt = (1ull << lane) - 1;
    uint32_t evens[kMaxFanout];
#pragma unroll
    for (uint32_t c = 0; c < kMaxFanout; c++) evens[c] = 0;
    for (uint32_t j0 = 0; j0 < m; j0 += 64) {
        const bool valid = j0 + lane < m;
        const uint64_t key = valid ? kp[j0 + lane] : 0;
        const uint32_t cid = child_of(key);
        const bool even = (key & 1) == 0;
#pragma unroll
        for (uint32_t c = 0; c < kMaxFanout; c++)
            if (c < fan) evens[c] += (uint32_t)__popcll(__ballot(valid && even && cid == c));
    }
    uint32_t base_e[kMaxFanout], base_o[kMaxFanout];
#pragma unroll
    for (uint32_t c = 0; c < kMaxFanout; c++) {
        base_e[c] = c * unit;
        base_o[c] = c * unit + evens[c];
    }
    for (uint32_t j0 = 0; j0 < m; j0 += 64) {
        const bool valid = j0 + lane < m;
        const uint64_t key = valid ? kp[j0 + lane] : 0;
        const uint32_t cid = child_of(key);
        const bool even = (key & 1) == 0;
        uint32_t pos = 0;
#pragma unroll
        for (uint32_t c = 0; c < kMaxFanout; c++) {
            if (c < fan) {
                const unsigned long long me = __ballot(valid && even && cid == c);
                const unsigned long long mo = __ballot(valid && !even && cid == c);
                if (cid == c) pos = even ? base_e[c] + (uint32_t)__popcll(me & lt) : base_o[c] + (uint32_t)__popcll(mo & lt);
                base_e[c] += (uint32_t)__popcll(me);
                base_o[c] += (uint32_t)__popcll(mo);
            }
        }
        if (valid) tmp[pos] = key;
    }
    lds_sync();
    for (uint32_t i = lane; i < m; i += 64) kp[i] = tmp[i];
    lds_sync();
}

// How a wave searches a node: groups sub, sub + q, ... of the node's candidate groups.
// With q > 1 waves of a workgroup share a node: *best (LDS) is the lowest seed any of
// them has found, and a wave ends once its next group lies above it.
struct TreeShare {
    uint32_t sub, q;
    unsigned long long *best;
    __device__ __forceinline__ bool beaten(uint64_t seed) const {
        if (q == 1) return false;
        const unsigned long long b = *(volatile unsigned long long *)best;
        return seed >= uni64(b);
    }
};

// Lowest valid seed of one leaf of at least kStagedMinLeaf keys, as staged_claim with
// the keys in LDS; kNone if another wave's seed is lower.
template <bool ROT, int U, bool R64>
__device__ __forceinline__ uint64_t tree_staged(const uint64_t *kp, uint32_t m, uint32_t nl, uint2 *queue,
                                                const uint16_t *canon, const TreeShare &sh, uint64_t &work) {
    const uint32_t stride = ROT ? m : 1;
    const uint32_t k = uni(c_stage.k[m]);
    const uint32_t b = ROT && 2 * nl < m ? nl : 0;
    StageKeys sk;
    sk.load_lds(kp + b, k);
    constexpr uint32_t kGroups = 64;  // candidate indexes are relative to this wave's every 64 groups
    const uint32_t q = uni(sh.q), sub = uni(sh.sub);
    for (uint64_t unit0 = 0; unit0 * stride < kSeedLimit; unit0 += (uint64_t)kGroups * q * U * 64) {
        const uint64_t base = unit0 * stride + c_start_seed[kSeedLeaf];
        const uint32_t max_idx = kGroups * q * U * 64 - 1;
        StageQueue sq{queue, 0};
        for (uint32_t g = 0, last = 0; !last; g++) {
            const uint32_t idx0 = (g * q + sub) * U * 64;
            last = g == kGroups || sh.beaten((unit0 + idx0) * stride);
            if (!last) {
                stage_push<U, R64>(sk, base, stride, m, idx0, sq);
                work += (uint64_t)U * 64 * k;
            }
            while (last ? sq.n > 0 : sq.n >= kStagedFill) {
                work += (uint64_t)64 * (m - k);
                const uint64_t hit = stage_test<ROT, R64, kKeysLds>(kp, m, nl, k, base, stride, max_idx, sq, canon);
                if (hit != kNone) return hit + unit0 * stride;
            }
            if (last && g < kGroups) return kNone;
        }
    }
    return kSeedLimit;
}

// Lowest hit of a search by groups of U * 64 candidates; kNone if another wave's is
// lower.
template <int U, typename F>
__device__ __forceinline__ uint64_t tree_groups(uint32_t scale, uint32_t m, const TreeShare &sh, uint64_t &work, F &&group) {
    const uint32_t q = uni(sh.q);
    for (uint64_t u0 = (uint64_t)uni(sh.sub) * U * 64; u0 * scale < kSeedLimit; u0 += (uint64_t)q * U * 64) {
        if (sh.beaten(u0 * scale)) return kNone;
        work += (uint64_t)U * 64 * m;
        const uint64_t hit = group(u0);
        if (hit != kNone) return hit;
    }
    return kSeedLimit;
}

// One node of a bucket's tree: keys [off, off + m) of the bucket, seed slot, fanout-2
// depth.
struct TreeItem {
    uint16_t off, m;
    uint32_t depth;
    uint32_t slot;
};

// UL: candidates per lane of the leaves and of heavy aggregation nodes.  TEAM: a
// workgroup per bucket whose waves take the nodes of one tree depth after another
// (few buckets: more waves than one per bucket); otherwise a wave per bucket, node
// by node in preorder.
template <int UL, bool R64, bool TEAM>
__global__ __launch_bounds__(TEAM ? 512 : 256, TEAM ? 2 : 4) void k_tree(TreeArgs a) {
    extern __shared__ uint8_t s_tree[];
    // workgroup: Golomb-Rice parameters and node counts by size, increment tables,
    // least rotations, counters; then the keys, scratch, staged queues and lists
    __shared__ unsigned long long s_stat[3 * kNumKinds];
    __shared__ TreeItem s_stack[TEAM ? 1 : 4][48];
    __shared__ unsigned long long s_un, s_best[8];
    __shared__ uint32_t s_team[4];  // bucket ticket, nodes of this depth, of the next, duplicates
    if (a.stop && (uni(*a.stop) & a.stop_mask)) return;
    if (a.max_bucket && uni(*a.max_bucket) < a.min_m) return;
    const SplitParams P = a.P;
    const bool rotate = a.rotate != 0;
    uint16_t *nodes_of = (uint16_t *)s_tree;
    uint8_t *gol = s_tree + 2 * a.cap + 16;
    uint32_t *up_lut = (uint32_t *)(s_tree + ((3 * a.cap + 47) & ~15u));
    uint32_t *lo_lut = up_lut + ((P.upper + 3) & ~3u);
    uint16_t *canon = (uint16_t *)(lo_lut + ((P.lower + 3) & ~3u));
    const bool use_canon = rotate && P.leaf <= kNecklaceMax;
    uint8_t *waves = (uint8_t *)(canon + (use_canon ? 1u << P.leaf : 0));
    for (uint32_t i = threadIdx.x; i <= a.cap; i += blockDim.x) {
        gol[i] = (uint8_t)(a.memo[i] >> 27);
        nodes_of[i] = (uint16_t)a.memo[kMaxBucket + i];
    }
    for (uint32_t r = threadIdx.x; r < P.upper; r += blockDim.x) up_lut[r] = 1u << (a.up_fb * (r / P.lower));
    for (uint32_t r = threadIdx.x; r < P.lower; r += blockDim.x) lo_lut[r] = 1u << (a.lo_fb * (r / P.leaf));
    if (use_canon) {
        const uint32_t L = P.leaf, full = (1u << L) - 1;
        for (uint32_t x = threadIdx.x; x <= full; x += blockDim.x) {
            uint32_t c = x, y = x;
            for (uint32_t t = 1; t < L; t++) {
                y = ((y << 1) | (y >> (L - 1))) & full;
                c = y < c ? y : c;
            }
            canon[x] = (uint16_t)c;
        }
    }
    if (threadIdx.x < 3 * kNumKinds) s_stat[threadIdx.x] = 0;
    __syncthreads();
    const uint32_t lane = lane_id(), wid = uni(threadIdx.x >> 6), n_w = uni(blockDim.x >> 6);
    // TEAM: one set of keys and scratch, a staged queue per wave, two node lists
    uint64_t *keys = (uint64_t *)(waves + (TEAM ? 0 : (size_t)wid * (a.cap * 8 + a.scratch)));
    uint8_t *scratch = (uint8_t *)(keys + a.cap);
    uint2 *queue = (uint2 *)(TEAM ? scratch + a.scratch + (size_t)wid * a.queue : scratch);
    TreeItem *lists = (TreeItem *)(scratch + a.scratch + (size_t)n_w * a.queue);  // TEAM only
    const uint32_t list_cap = a.cap / 2 + 1;
    const uint32_t up_hi = uni(((uint32_t)(uintptr_t)up_lut >> 2) << 16), lo_hi = uni(((uint32_t)(uintptr_t)lo_lut >> 2) << 16);
    const unsigned long long t_end = a.limit_ticks ? uni64(*a.clock0) + a.limit_ticks : ~0ull;
    uint64_t ev[kNumKinds] = {0, 0, 0, 0, 0}, sd[kNumKinds] = {0, 0, 0, 0, 0}, wk[kNumKinds] = {0, 0, 0, 0, 0};
    uint64_t un = 0;  // unary bits of this wave's nodes of the bucket
    uint32_t bm = 0;  // keys of the bucket
    // Part size, parts and start seed of a split node.
    auto split_of = [&](uint32_t kind, uint32_t m, uint32_t depth, uint32_t &unit, uint32_t &fan) -> uint64_t {
        if (kind == kHigher) {
            unit = higher_split(P, m);
            fan = 2;
            return c_start_seed[depth];
        }
        unit = kind == kUpper ? P.lower : P.leaf;
        fan = (m + unit - 1) / unit;
        return c_start_seed[kind == kUpper ? kSeedUpper : kSeedLower];
    };
    // Searches one node: its lowest seed (of this wave's share).
    auto search = [&](uint32_t koff, uint32_t m, uint32_t depth, const TreeShare &sh) -> uint64_t {
        uint64_t *kp = keys + koff;
        const uint32_t kind = classify(P, m, rotate);
        uint64_t x = 0, work = 0;
        uint32_t unit = 0, fan = 0;
        if (kind == kHigher) {
            const uint64_t seed0 = split_of(kind, m, depth, unit, fan);
            const uint32_t H = (unit * 65536u + m - 1) / m;  // unit < 3000: below 2^28
            x = tree_groups<1>(1, m, sh, work, [&](uint64_t u0) { return group_higher<1, kKeysLds, R64>(kp, m, seed0, unit, H, u0); });
        } else if (kind == kUpper || kind == kLower) {
            const bool up = kind == kUpper;
            const uint64_t seed0 = split_of(kind, m, depth, unit, fan);
            const uint32_t fb = up ? a.up_fb : a.lo_fb, magic = up ? a.up_magic : a.lo_magic;
            uint32_t T = 0;
            for (uint32_t p = 0; p + 1 < fan; p++) T |= unit << (p * fb);
            const uint32_t cmask = (1u << ((fan - 1) * fb)) - 1;  // at most 31 bits
            const uint32_t hi = up ? up_hi : lo_hi;
            // UL candidates per lane from about 500 expected candidates on, on both levels
            // (1.8M keys at l = 12, b = 200, upper level one per lane 10.0 ms, this 6.1),
            // one below (a pass of UL tests 64 UL at once)
            if (UL > 1 && gol[m] >= 8)
                x = tree_groups<UL>(1, m, sh, work, [&](uint64_t u0) {
                    return group_aggr<UL, false, true, kKeysLds, R64>(kp, m, seed0, fb, magic, T, cmask, hi, 2, u0);
                });
            else
                x = tree_groups<1>(1, m, sh, work, [&](uint64_t u0) {
                    return group_aggr<1, false, true, kKeysLds, R64>(kp, m, seed0, fb, magic, T, cmask, hi, 2, u0);
                });
        } else {
            const bool odd_key = lane < m && (kp[lane < m ? lane : 0] & 1) != 0;
            const uint32_t nl = m - (uint32_t)__popcll(__ballot(odd_key));
            if (kind == kLeafRot) {
                if (m >= kStagedMinLeaf)
                    x = tree_staged<true, UL, R64>(kp, m, nl, queue, canon, sh, work);
                else
                    x = tree_groups<UL>(m, m, sh, work, [&](uint64_t u0) {
                        return group_leaf_rot<UL, kKeysLds, R64, false>(kp, m, nl, u0, canon);
                    });
            } else if (m >= kStagedMinLeaf) {
                x = tree_staged<false, UL, R64>(kp, m, 0, queue, canon, sh, work);
            } else {
                x = tree_groups<UL>(1, m, sh, work, [&](uint64_t u0) { return group_leaf_brute<UL, kKeysLds, R64>(kp, m, m, u0); });
            }
        }
#pragma unroll
        for (int k = 0; k < kNumKinds; k++) wk[k] += (uint32_t)k == kind ? work : 0;
        return x;
    };
    // Records a node's seed, orders its keys by child and hands every child of two or
    // more keys to push, right to left.
    auto finish = [&](uint32_t koff, uint32_t m, uint32_t depth, uint32_t slot, uint64_t x, auto &&push) {
        uint64_t *kp = keys + koff;
        uint64_t *tmp = (uint64_t *)scratch + (TEAM ? koff : 0);
        const uint32_t kind = classify(P, m, rotate);
        if (lane == 0) {
            a.seeds[slot] = x;
            a.node_m[slot] = (uint16_t)m;
            if (x >= kSeedLimit) atomicOr(a.err, kErrSeedLimit);
        }
        if (x >= kSeedLimit) return;
        un += (x >> gol[m]) + 1;
        const uint64_t e = kind == kLeafRot ? (x / m + 1) * m : (x + 1) * m;
        const uint64_t t = kind == kLeafRot ? e : x + 1;
#pragma unroll
        for (int k = 0; k < kNumKinds; k++) {
            ev[k] += (uint32_t)k == kind ? e : 0;
            sd[k] += (uint32_t)k == kind ? t : 0;
        }
        if (m <= P.leaf) return;
        uint32_t unit = 0, fan = 0;
        const uint64_t sa = split_of(kind, m, depth, unit, fan) + x;
        tree_partition(kp, tmp, m, unit, fan, [&](uint64_t key) -> uint32_t {
            const uint32_t r = remap_any(key + sa, m, R64);
            if (kind == kHigher) return r >= unit ? 1u : 0u;
            return __umul24(r, kind == kUpper ? a.up_magic : a.lo_magic) >> 20;  // r / unit
        });
        for (int c = (int)fan - 1; c >= 0; c--) {
            const uint32_t cs = c == (int)fan - 1 ? m - (fan - 1) * unit : unit;
            // preorder slots: the node's own, then its children's subtrees left to right
            if (cs > 1) push(TreeItem{(uint16_t)(koff + (uint32_t)c * unit), (uint16_t)cs, depth + 1,
                                      slot + 1 + (uint32_t)c * nodes_of[unit]});
        }
    };
    // A bucket that is one full leaf has not been ordered by parity yet.
    auto order_leaf_bucket = [&]() {
        if (classify(P, bm, rotate) == kLeafRot)
            tree_partition(keys, (uint64_t *)scratch, bm, bm, 1, [](uint64_t) { return 0u; });
    };
    auto past_limit = [&]() -> bool {
        if (!a.limit_ticks) return false;
        uint32_t l = 0;
        if (lane == 0) l = (unsigned long long)wall_clock64() > t_end;
        if (uni(l) && lane == 0) atomicOr(a.err, kErrTimeout);
        return uni(l) != 0;
    };
    uint64_t b = 0, b_end = 0;
    for (;;) {
        if constexpr (TEAM) {
            __syncthreads();  // the bucket before is done with its keys and lists
            if (threadIdx.x == 0) {
                s_team[0] = atomicAdd(&a.ctl[0], 1u);
                s_un = 0;
            }
            __syncthreads();
            b = uni(s_team[0]);
            if (b >= a.nb) break;
        } else {
            if (b >= b_end) {
                uint32_t t = 0;
                if (lane == 0) t = atomicAdd(&a.ctl[0], 1u);
                b = (uint64_t)uni(t) * a.batch;
                if (b >= a.nb) break;
                b_end = b + a.batch < a.nb ? b + a.batch : a.nb;
            }
        }
        const uint64_t bucket = uni64(b++);
        const uint64_t off = uni64(a.acc[bucket]);
        bm = uni((uint32_t)(a.acc[bucket + 1] - off));
        if (bm < 2 || bm >= kMaxBucket) {  // oversized buckets fail the build
            if (lane == 0) a.bits[bucket] = 0;
            continue;
        }
        if (bm < a.min_m || bm > a.max_m) continue;
        const uint32_t slot0 = uni((uint32_t)a.node_base[bucket]);
        const uint64_t fixed = uni(a.memo[bm] & 0xFFFF);
        const uint32_t entries = tree_dup_entries(a.cap);
        if constexpr (TEAM) {
            TreeItem *cur = lists, *next = lists + list_cap;
            for (uint32_t i = threadIdx.x; i < bm; i += blockDim.x) keys[i] = a.sorted[off + i];
            if (threadIdx.x == 0) cur[0] = TreeItem{0, (uint16_t)bm, 0, slot0};
            __syncthreads();
            if (wid == 0) {
                const bool dup = tree_duplicates(keys, bm, (uint32_t *)scratch, entries);
                const bool late = past_limit();
                order_leaf_bucket();
                if (lane == 0) {
                    s_team[3] = dup || late;
                    s_team[1] = 1;
                    if (dup) atomicOr(a.err, kErrDuplicateKeys);
                }
            }
            __syncthreads();
            if (uni(s_team[3])) {
                if (threadIdx.x == 0) a.bits[bucket] = 0;
                continue;
            }
            un = 0;
            for (uint32_t count = 1; count;) {
                if (threadIdx.x == 0) s_team[2] = 0;
                __syncthreads();
                auto push = [&](const TreeItem &child) {
                    if (lane == 0) next[atomicAdd(&s_team[2], 1u)] = child;
                };
                if (2 * count <= n_w) {
                    // fewer nodes than half the waves: q waves share each node
                    const uint32_t q = n_w / count, node = wid / q, sub = wid - node * q;
                    if (node < count) {
                        if (sub == 0 && lane == 0) s_best[node] = kNone;
                    }
                    __syncthreads();
                    if (node < count) {
                        const TreeItem it = cur[node];
                        const uint64_t x = search(uni(it.off), uni(it.m), uni(it.depth), TreeShare{sub, q, &s_best[node]});
                        if (lane == 0 && x != kNone) atomicMin(&s_best[node], (unsigned long long)x);
                    }
                    __syncthreads();
                    if (node < count && sub == 0) {
                        const TreeItem it = cur[node];
                        finish(uni(it.off), uni(it.m), uni(it.depth), uni(it.slot), uni64(s_best[node]), push);
                    }
                } else {
                    for (uint32_t i = wid; i < count; i += n_w) {
                        const TreeItem it = cur[i];
                        const uint64_t x = search(uni(it.off), uni(it.m), uni(it.depth), TreeShare{0, 1, nullptr});
                        finish(uni(it.off), uni(it.m), uni(it.depth), uni(it.slot), x, push);
                    }
                }
                __syncthreads();
                count = uni(s_team[2]);
                TreeItem *t = cur;
                cur = next;
                next = t;
                __syncthreads();  // every wave has read the count before it is cleared
            }
            if (lane == 0) atomicAdd(&s_un, (unsigned long long)un);
            __syncthreads();
            if (threadIdx.x == 0) a.bits[bucket] = fixed + s_un;
        } else {
            if (past_limit()) break;
            TreeItem *stack = s_stack[wid];
            for (uint32_t i = lane; i < bm; i += 64) keys[i] = a.sorted[off + i];
            lds_sync();
            if (tree_duplicates(keys, bm, (uint32_t *)scratch, entries)) {
                if (lane == 0) {
                    atomicOr(a.err, kErrDuplicateKeys);
                    a.bits[bucket] = 0;
                }
                continue;
            }
            order_leaf_bucket();
            un = 0;
            int sp = 1;
            if (lane == 0) stack[0] = TreeItem{0, (uint16_t)bm, 0, slot0};
            lds_sync();
            while (sp > 0) {
                const TreeItem it = stack[--sp];
                const uint64_t x = search(uni(it.off), uni(it.m), uni(it.depth), TreeShare{0, 1, nullptr});
                finish(uni(it.off), uni(it.m), uni(it.depth), uni(it.slot), x, [&](const TreeItem &child) {
                    if (lane == 0) stack[sp] = child;
                    sp++;
                });
                lds_sync();
            }
            if (lane == 0) a.bits[bucket] = fixed + un;
        }
    }
    if (lane == 0) {
#pragma unroll
        for (int k = 0; k < kNumKinds; k++) {
            if (ev[k]) atomicAdd(&s_stat[k], (unsigned long long)ev[k]);
            if (sd[k]) atomicAdd(&s_stat[kNumKinds + k], (unsigned long long)sd[k]);
            if (wk[k]) atomicAdd(&s_stat[2 * kNumKinds + k], (unsigned long long)wk[k]);
        }
    }
    __syncthreads();
    if (threadIdx.x < 3 * kNumKinds && s_stat[threadIdx.x])
        atomicAdd(threadIdx.x < 2 * kNumKinds ? &a.evals[threadIdx.x] : &a.work[threadIdx.x - 2 * kNumKinds],
                  s_stat[threadIdx.x]);
}

// LDS of one k_tree workgroup of `waves` waves for buckets of at most cap keys.
struct TreeLds {
    uint32_t scratch, queue;
    size_t bytes;
};
inline TreeLds tree_lds(const SplitParams &P, bool rotate, uint32_t cap, uint32_t waves, bool team) {
    uint32_t scratch = cap * 8;
    scratch = scratch > 4 * tree_dup_entries(cap) ? scratch : 4 * tree_dup_entries(cap);
    const uint32_t queue = P.leaf >= kStagedMinLeaf ? kStagedCap * 8 : 0;
    size_t b = ((3 * cap + 47) & ~15u) + 4 * (size_t)(((P.upper + 3) & ~3u) + ((P.lower + 3) & ~3u));
    if (rotate && P.leaf <= kNecklaceMax) b += (size_t)2 << P.leaf;
    if (team) return {scratch, queue, b + cap * 8 + scratch + (size_t)waves * queue + 2 * (cap / 2 + 1) * sizeof(TreeItem)};
    if (scratch < queue) scratch = queue;
    return {scratch, queue, b + (size_t)waves * (cap * 8 + scratch)};
}

}  // namespace rsa
