// svm_tree.h -- shared-state executor: many shots of one program per
// workgroup, one copy of the amplitudes per group of shots that agree on
// everything the amplitudes depend on.
//
// One shot per thread holds its xoshiro256++ state and its response
// (svm_tree_args.h): the record bits and the few other bits the walk reads,
// to which every random bit that comes up 1 adds a precomputed row.  There
// is no Pauli frame, and no opcode that only moves one.  Shots whose random
// outcomes (and frame bits at phase opcodes) agreed so far have the same
// amplitudes, bit for bit, so the team keeps one state per such group
// ("node") and sweeps all nodes as one flat array: entry i of node n at
// n 2^r + i.  An active measurement writes both outcomes' folded states of
// every node and sums both probabilities; each shot then draws its own
// outcome from its own stream, and the (node, outcome) pairs that occur
// become the next nodes.  Nothing is approximated or carried over from one
// launch to the next: a shot draws what it draws on the per-shot executors,
// against probabilities that agree to rounding (the order of a node's sums
// depends on the team and on how many nodes there are).
//
// Why.  The per-shot tiers move the whole state once or twice per
// measurement and shot and dispatch every opcode per shot.  Here a level
// with N nodes of rank r moves N 2^r entries for all the shots together,
// and N doubles at most while r falls by one: a team of 1000 shots at peak
// 16 moves about 12 x 2^16 entries instead of 1000 x 2 x 2^16, and every
// opcode is dispatched once per 64 shots.
//
// Measured on one MI355X (per call, before -> after; before: the per-shot
// tiers): 24-qubit Clifford+T, peak 10 x 20000 shots 2304 -> 55 us, peak 16 x
// 2000 1805 -> 278 us; 34 qubits, peak 25 x 64 shots 752 -> 66.5 ms; 512
// programs x 1000 shots 54.4 -> 0.64 to 0.70 ms; surface-code memories, distance
// 3 x 10^6 shots 162 -> 126 us, distance 7 (97 qubits) x 20000 7770 -> 85 us,
// distance 5 with 4 forced faults x 20000 3940 -> 210 us (135 of kernel).  With
// a frame per shot and every opcode walked (the same executor before the
// response) peak 10 took 82 us, its walk 35 of them.
// What bounds it: memories, the dependent loads of a noise event (about 1.3
// us for the slowest of 64 shots) and the draws; up to peak 12 the passes'
// fixed part, about 2 us a measurement; from peak 14 their entries (16
// instructions and 32 bytes each).  128 VGPRs, 30 to 35 of them spilled: teams
// of 1024 threads allow no more.
//
// The array work itself is planned on the host (svm_tree_plan.h): each pass
// gathers through a linear map over GF(2), so a lane's source index is the
// XOR of a per-lane part, fixed for the pass, and a uniform part that
// changes by one column between its entries.
#pragma once

#include "svm_device.h"
#include "svm_tree_args.h"
#include "svm_sweeps.h"

namespace csvm {

typedef __attribute__((address_space(3))) uint32_t tree_lds_u32;
typedef uint32_t TreeQuad __attribute__((ext_vector_type(4)));  // a group of a row

// orders one lane's LDS accesses with another's of its wavefront
CSVM_INLINE void tree_wave_fence() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// (tables that lanes index for themselves)
typedef const __attribute__((address_space(1))) TreeQuad* glb_quad;
typedef const __attribute__((address_space(1))) double* glb_f64;
typedef const __attribute__((address_space(1))) uint32_t* glb_u32;
typedef const __attribute__((address_space(1))) uint64_t* glb_u64;

template <class AmpT>
struct TreeInterp {
    typedef tree_lds_u32 lds_u32;
    typedef __attribute__((address_space(3))) TreeStage lds_stage;
    typedef __attribute__((address_space(3))) uint64_t lds_u64;
    static constexpr uint32_t G = 4;  // pairs in flight per lane: eight 16-byte loads

    uint32_t tid, lane, wave, nthreads, nwaves;
    AmpT *src, *dst;
    lds_u32 *nsrc, *nsrc2;  // node -> stored node
    lds_u32 *nch, *nch2;    // node -> choice word
    lds_u32 *flags, *flags2;
    uint32_t scale_word;    // index of the rescale flag behind the bitmaps' words
    lds_f64 *psum, *part;
    lds_stage* stage;
    uint32_t N;             // nodes
    // the next pass's words (svm_tree_args.h), loaded while the one before
    // it runs: lane b of `wa` the header, of the halves of `wa`, `wb`, `wc`
    // the columns
    uint32_t next, wa, wb, wc;
    // this thread's shot
    uint32_t node, live;
    Rng rng;
    uint32_t next_noise, discarded, reachable, dust;
    double logp;
    const uint8_t* forced;  // its forced record row (MODE_FORCED)
    lds_u32* R;             // its response: word w at R[w << 6]
    // MODE_KFAULT: its forced noise sites, then readout entries, each ascending
    lds_u32* kf;
    uint32_t kf_nn, kf_pos, kf_n, kf_rpos;  // kf null: gap sampling

    // -------------------------------------------------------------- response
    CSVM_INLINE static void add_word(lds_u32* p, uint32_t x) {
        (void)__hip_atomic_fetch_xor(p, x, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WAVEFRONT);  // one LDS instruction
    }
    // Add a row of `units` units where `on`: a few entries, against some dozen
    // words of a response.
    CSVM_INLINE void add_entries(TreeQuad e) {
        if (e.y) add_word(R + e.x, e.y);
        if (e.w) add_word(R + e.z, e.w);
    }
    CSVM_INLINE void add_row(cptr<TreeQuad> row, uint32_t units, bool on) {
        const TreeQuad e0 = row[0], e1 = row[1];
        if (!on) return;
        add_entries(e0);
        add_entries(e1);
        for (uint32_t g = 2; g < 2u * units; ++g) add_entries(row[g]);
    }
    // The same for `count` rows in turn, bit j's being fires().  A row's first
    // unit arrives while the one before it is added (its load is issued after
    // that one's wait: scalar loads are only waited for all together), and
    // entries are masked, not branched over: at a wavefront or two per SIMD a
    // taken branch costs as much as several instructions.
    template <class F>
    CSVM_INLINE void add_rows(cptr<TreeQuad> row, uint32_t units, uint32_t count, F fires) {
        TreeQuad e0 = row[0], e1 = row[1];
        for (uint32_t j = 0; j < count; ++j) {
            cptr<TreeQuad> next = row + (j + 1u < count ? 2u * units : 0u);
            asm volatile("" ::"s"(e0.x), "s"(e1.x));
            const TreeQuad n0 = next[0], n1 = next[1];
            const uint32_t m = fires() ? 0xFFFFFFFFu : 0u;
            add_word(R + e0.x, e0.y & m);
            if (e0.w) {
                add_word(R + e0.z, e0.w & m);
                add_word(R + e1.x, e1.y & m);
                add_word(R + e1.z, e1.w & m);
            }
            for (uint32_t g = 2; g < 2u * units; ++g) {
                const TreeQuad e = row[g];
                if (!e.y) break;
                add_word(R + e.x, e.y & m);
                add_word(R + e.z, e.w & m);
            }
            row = next;
            e0 = n0;
            e1 = n1;
        }
    }
    CSVM_INLINE static cptr<TreeQuad> row_at(cptr<DevProgram> P, uint32_t unit) {
        return (cptr<TreeQuad>)cp(P->lp_rows) + 2 * (size_t)unit;
    }
    CSVM_INLINE uint32_t bits(uint32_t at, uint32_t n) const { return (R[(at >> 5) << 6] >> (at & 31u)) & ((1u << n) - 1u); }

    // ----------------------------------------------------------------- noise
    // Gap sampler (svm.h:229-243)
    CSVM_INLINE void draw_next_noise(cptr<DevProgram> P, double cur) {
        const uint32_t n = P->num_sites;
        if (n == 0 || next_noise >= n) {
            next_noise = kNoNoise;
            return;
        }
        const double gap = -log(1.0 - rng_double(rng));
        next_noise = hazard_upper_bound((glb_f64)P->hazards, n, (glb_u32)P->hz_guide, P->hz_buckets, P->hz_scale, cur + gap);
    }
    // The first channel whose running sum exceeds r (pick_channel's rule and
    // first try, on TreeChan records): its row's first entry and their number.
    CSVM_INLINE static double chan_cum(TreeQuad c) { return __hiloint2double((int)c.y, (int)c.x); }
    CSVM_INLINE void pick(glb_quad ch, uint32_t n, double u, uint32_t& first, uint32_t& count) {
        const uint32_t q = (uint32_t)(u * (double)n), g = q < n ? q : n - 1u;
        const TreeQuad last = ch[n - 1u], before = ch[g > 0 ? g - 1u : 0u];
        TreeQuad c = ch[g];
        const double r = u * chan_cum(last);
        count = 0;
        if (!((g == 0 || chan_cum(before) <= r) && r < chan_cum(c))) {
            uint32_t lo = 0, hi = n;
            while (lo < hi) {
                const uint32_t mid = lo + (hi - lo) / 2;
                if (r < chan_cum(ch[mid]))
                    hi = mid;
                else
                    lo = mid + 1;
            }
            if (lo == n) return;
            c = ch[lo];
        }
        first = c.z;
        count = c.w;
    }
    // Fire the site next_noise and find the next one (svm_kernels.inl:1886-1920).
    // A chain of dependent loads bounds it, so the tables are laid out for
    // few of them, and the row's first entries are under way while the next
    // site is looked up.
    CSVM_INLINE void noise(cptr<DevProgram> P) {
        const TreeQuad t = ((glb_quad)P->lp_sites)[next_noise];
        const double u = rng_double(rng);
        uint32_t first = 0, count = 0;
        if (t.y) pick((glb_quad)P->lp_chans + t.x, t.y, u, first, count);
        glb_quad row = (glb_quad)P->lp_chan_rows + (first >> 1);
        TreeQuad e0{0, 0, 0, 0}, e1{0, 0, 0, 0};
        if (count > 0) e0 = row[0];
        if (count > 2) e1 = row[1];
        if (kf) {  // svm.h:218-225
            next_noise = kf_pos < kf_nn ? kf[kf_pos << 6] : kNoNoise;
            kf_pos++;
        } else {
            next_noise++;
            draw_next_noise(P, chan_cum(TreeQuad{t.z, t.w, 0, 0}));
        }
        for (uint32_t i = 0;;) {  // (adding zero does nothing)
            add_word(R + e0.x, e0.y);
            add_word(R + e0.z, e0.w);
            add_word(R + e1.x, e1.y);
            add_word(R + e1.z, e1.w);
            i += 4;
            if (i >= count) break;
            e0 = row[i >> 1];
            e1 = TreeQuad{0, 0, 0, 0};
            if (i + 2u < count) e1 = row[(i >> 1) + 1u];
        }
    }

    // Choose this shot's (`on`) fault set (svm.cc:435-520; with unequal
    // probabilities about 45 instructions a site, 85 us for 670 sites, where
    // looking the limits up as they are needed took 134) into its list -- room
    // for 5 k words a lane: picks, then the sparse Fisher-Yates map of at
    // most 2 k positions -- and arm the noise cursor.
    CSVM_INLINE void kfault_prepare(cptr<KfTables> T, lds_u32* list, bool on) {
        const uint32_t n = T->n, k = T->k, n_q = T->n_q;
        uint32_t m = 0;
        if (k == 0) {
        } else if (T->uniform) {
            lds_u32 *keys = list + (k << 6), *vals = list + (3u * k << 6);
            uint32_t nk = 0;
            auto find = [&](uint32_t pos) -> uint32_t {  // index in the map, or nk
                uint32_t e = 0;
                while (e < nk && keys[e << 6] != pos) ++e;
                return e;
            };
            for (uint32_t j = 0; j < k; ++j) {
                const uint32_t pick = j + (uint32_t)(rng_double(rng) * (double)(n - j));
                if (pick == j) continue;  // swap with itself
                const uint32_t nk0 = nk, ej = find(j), ep = find(pick);
                const uint32_t vj = ej < nk0 ? vals[ej << 6] : j, vp = ep < nk0 ? vals[ep << 6] : pick;
                const uint32_t sj = ej < nk0 ? ej : nk++, sp = ep < nk0 ? ep : nk++;
                keys[sj << 6] = j;  // pool[j] <- pool[pick], pool[pick] <- pool[j]
                vals[sj << 6] = vp;
                keys[sp << 6] = pick;
                vals[sp << 6] = vj;
            }
            for (uint32_t j = 0; j < k; ++j) {  // prefix pool[0..k), sorted as it is taken
                const uint32_t e = find(j), v = e < nk ? vals[e << 6] : j;
                uint32_t b = j;
                for (; b > 0 && list[(b - 1u) << 6] > v; --b) list[b << 6] = list[(b - 1u) << 6];
                list[b << 6] = v;
            }
            m = k;
        } else {
            // One draw a site until every fault is placed, against a limit that
            // depends on the faults still to place.  The limits of some sites
            // at a time are laid out for the wavefront in the rest of its
            // lists' room (128 k of them).  No branch on a hit: the site is
            // stored where the next hit's will overwrite it, and both limits
            // that the next site can have are loaded under this one's draw.
            const glb_u64 lim = (glb_u64)T->below;
            lds_u64* held = (lds_u64*)(list - lane + (k << 6));
            const uint32_t stride = k + 1u, per = (k << 7) / stride;
            uint32_t needed = on ? k : 0u;
            lds_u32* slot = list;
            for (uint32_t base = 0; base < n && __any(needed != 0u); base += per - 1u) {
                tree_wave_fence();
                for (uint32_t e = lane; e < per * stride; e += 64u)
                    if (base * stride + e < (n + 1u) * stride) held[e] = lim[base * stride + e];
                tree_wave_fence();
                const uint32_t end = n - base < per - 1u ? n : base + per - 1u;
                const lds_u64* q = held + needed;
                uint64_t p = *q;
                for (uint32_t i = base; i < end && needed; ++i) {
                    q += stride;
                    const uint64_t miss = q[0], next = q[-1];
                    const uint64_t x = rng_next(rng) >> 11;
                    *slot = i;
                    const bool hit = x < p;
                    slot += hit ? 64 : 0;
                    q -= hit ? 1 : 0;
                    needed -= hit ? 1u : 0u;
                    p = hit ? next : miss;
                }
            }
            m = k - needed;
            tree_wave_fence();
        }
        // picks are ascending: quantum sites first, then readout entries
        uint32_t nn = 0;
        while (nn < m && list[nn << 6] < n_q) ++nn;
        for (uint32_t j = nn; j < m; ++j) list[j << 6] -= n_q;
        kf = list;
        kf_nn = nn;
        kf_n = m;
        kf_rpos = nn;
        next_noise = on && nn ? list[0] : kNoNoise;
        kf_pos = 1;
    }

    // svm_internal.h:65-79
    CSVM_INLINE uint32_t sample_branch(double p0, double p1, double total) {
        const double eps = kDustEpsilon * total;
        if (p1 <= eps) {
            if (p1 > 0.0) dust++;
            return 0;
        }
        if (p0 <= eps) {
            if (p0 > 0.0) dust++;
            return 1;
        }
        const double r = rng_double(rng);
        return (r * total < p0) ? 0u : 1u;
    }
    // svm_forced_kernels.cc:43-61; false: outcome b is unreachable
    CSVM_INLINE bool forced_branch(double p0, double p1, double total, uint32_t b) {
        const double eps = kDustEpsilon * total;
        if (p1 <= eps) {
            if (p1 > 0.0) dust++;
            return b == 0;
        }
        if (p0 <= eps) {
            if (p0 > 0.0) dust++;
            return b == 1;
        }
        logp += log((b ? p1 : p0) / total);
        return true;
    }

    // ------------------------------------------------------------- splitting
    // The live shots' keys (below nkeys) become the new node numbers, in key
    // order.  Returns through `id` this shot's number and leaves N nodes.
    // A node's old tables are still readable until the caller swaps them.
    CSVM_INLINE uint32_t renumber(uint32_t key, uint32_t nkeys, uint32_t rescale) {
        const uint32_t words = (nkeys + 31u) >> 5;
        for (uint32_t w = tid; w < words; w += nthreads) flags[w] = 0u;
        if (tid == 0) flags[scale_word] = 0u;
        __syncthreads();
        if (live) {
            __hip_atomic_fetch_or(flags + (key >> 5), 1u << (key & 31u), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
            if (rescale) flags[scale_word] = 1u;
        }
        __syncthreads();
        if (words == 1u) {
            const uint32_t w = flags[0];
            N = uni((uint32_t)__popc(w));
            return (uint32_t)__popc(w & ((1u << (key & 31u)) - 1u));
        }
        uint32_t total = 0, id = 0;
        for (uint32_t base = 0; base < words; base += 64u) {
            const uint32_t v = base + lane < words ? flags[base + lane] : 0u;
            uint32_t incl = (uint32_t)__popc(v);
#pragma unroll
            for (int off = 1; off < 64; off <<= 1) {
                const uint32_t up = (uint32_t)__shfl_up((int)incl, off, 64);
                if (lane >= (uint32_t)off) incl += up;
            }
            const uint32_t at = (key >> 5) - base;  // wraps where the key lies before this block
            const uint32_t excl = incl - (uint32_t)__popc(v);
            const uint32_t e = (uint32_t)__shfl((int)excl, (int)(at & 63u), 64);
            const uint32_t w = (uint32_t)__shfl((int)v, (int)(at & 63u), 64);
            if (at < 64u) id = total + e + (uint32_t)__popc(w & ((1u << (key & 31u)) - 1u));
            total += uni((uint32_t)__shfl((int)incl, 63, 64));
        }
        N = uni(total);
        return id;
    }
    CSVM_INLINE void swap_tables() {
        lds_u32* t = nsrc;
        nsrc = nsrc2;
        nsrc2 = t;
        t = nch;
        nch = nch2;
        nch2 = t;
        t = flags;
        flags = flags2;
        flags2 = t;
    }
    // kTreeChoice: part the shots of every node by `bits` frame bits
    CSVM_INLINE void choice_split(uint32_t c, uint32_t bits, uint32_t at) {
        if (!__syncthreads_or((int)(live && c != 0u))) return;  // every bit 0: nodes and choice words stay
        const uint32_t id = renumber((node << bits) | c, N << bits, 0u);
        if (live) {
            nsrc2[id] = nsrc[node];
            nch2[id] = nch[node] | (c << at);
            node = id;
        }
        swap_tables();
    }

    // ----------------------------------------------------------------- passes
    // The words of a coordinate index (svm_tree_args.h): the source offset,
    // the written offset, the relative signs and the general-phase word.
    struct Words {
        uint32_t x, o, s, g;
        CSVM_INLINE Words operator^(const Words& w) const { return Words{x ^ w.x, o ^ w.o, s ^ w.s, g ^ w.g}; }
    };
    // The running pass: its header in scalar registers, its columns spread
    // over the wavefront's lanes.
    struct Pass {
        uint32_t type, r0, r, quarter, ngen, gen_off, sign0, ez_choices, lo;
        uint32_t wa, wb, wc;
        CSVM_INLINE static uint32_t at(uint32_t w, uint32_t i) { return (uint32_t)__builtin_amdgcn_readlane(w, i); }
        CSVM_INLINE uint32_t head(uint32_t i) const { return at(wa, i); }
        template <bool FULL>
        CSVM_INLINE Words column(uint32_t b) const {
            return Words{at(wa, 32u + b), at(wb, b), at(wb, 32u + b), FULL ? at(wc, b) : 0u};
        }
    };
    CSVM_INLINE void load_pass(cptr<DevProgram> Pg, uint32_t i) {
        const uint32_t* w = reinterpret_cast<const uint32_t*>(opaque(Pg)->tree_passes + i);
        next = i;
        wa = w[lane];
        wb = w[64u + lane];
        wc = w[128u + (lane & 31u)];
    }
    CSVM_INLINE static uint32_t odd(uint32_t i, uint32_t m) { return (uint32_t)__popc(i & m) & 1u; }
    CSVM_INLINE static double flip(double a, uint32_t sign) {
        return __longlong_as_double(__double_as_longlong(a) ^ ((long long)((unsigned long long)sign << 32)));
    }
    CSVM_INLINE static const AmpT* at(const AmpT* p, uint32_t off) {
        return (const AmpT*)((const __attribute__((address_space(std::is_same<AmpT, lds_d2>::value ? 3 : 1))) char*)p + off);
    }
    CSVM_INLINE static AmpT* at(AmpT* p, uint32_t off) { return const_cast<AmpT*>(at(const_cast<const AmpT*>(p), off)); }

    // sum over the 2^t lanes (t <= 6) that share the lane bits above t; every
    // lane of them gets it
    template <int CTRL>
    CSVM_INLINE static double dpp_add(double a) {
        const long long b = __double_as_longlong(a);
        const uint32_t lo = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)b, CTRL, 0xF, 0xF, true);
        const uint32_t hi = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(b >> 32), CTRL, 0xF, 0xF, true);
        return a + __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));
    }
    CSVM_INLINE static void lanes_sum(double& a, double& b, uint32_t t) {
        if (t >= 1u) a = dpp_add<0xB1>(a), b = dpp_add<0xB1>(b);    // quad_perm 1,0,3,2
        if (t >= 2u) a = dpp_add<0x4E>(a), b = dpp_add<0x4E>(b);    // quad_perm 2,3,0,1
        if (t >= 3u) a = dpp_add<0x141>(a), b = dpp_add<0x141>(b);  // row_half_mirror
        if (t >= 4u) a = dpp_add<0x140>(a), b = dpp_add<0x140>(b);  // row_mirror
        if (t >= 5u) a += __shfl_xor(a, 16, 64), b += __shfl_xor(b, 16, 64);
        if (t >= 6u) a += __shfl_xor(a, 32, 64), b += __shfl_xor(b, 32, 64);
    }

    // K pairs whose words (pair bit clear) are w[], `pair` those of the pair
    // bit: load, and (FULL) pending expansions and general phases.
    template <uint32_t K, bool FULL>
    CSVM_INLINE void gather(cptr<DevProgram> Pg, const Pass& q, const AmpT* sp, uint32_t ch, const Words& pair,
                            const Words (&w)[K], dv2 (&p)[K], dv2 (&h)[K]) {
        if (!FULL || q.r0 == q.r) {
#pragma unroll
            for (uint32_t e = 0; e < K; ++e) {
                p[e] = *at(sp, w[e].x);
                h[e] = *at(sp, w[e].x ^ pair.x);
            }
        } else {
#pragma unroll
            for (uint32_t e = 0; e < K; ++e) {
                p[e] = *at(sp, w[e].x & q.lo);
                h[e] = *at(sp, (w[e].x ^ pair.x) & q.lo);
            }
            if (!q.ez_choices) {
#pragma unroll
                for (uint32_t e = 0; e < K; ++e) {
                    const uint32_t a = w[e].x >> (q.r0 + 4u), b = (w[e].x ^ pair.x) >> (q.r0 + 4u);
                    p[e] = cmul(p[e], mk(stage->tab[a][0], stage->tab[a][1]));
                    h[e] = cmul(h[e], mk(stage->tab[b][0], stage->tab[b][1]));
                }
            } else {
                cptr<TreePass> T = cp(opaque(Pg)->tree_passes) + next;
                for (uint32_t b = 0; b < q.r - q.r0; ++b) {
                    const uint32_t s = q.r0 + 4u + b, cb = (pair.x >> s) & 1u;
                    const int32_t c = T->ez_choice[b];
                    const double zi = T->ez[b][1];
                    const dv2 z = mk(T->ez[b][0], (c >= 0 && ((ch >> (c & 31)) & 1u)) ? -zi : zi);
#pragma unroll
                    for (uint32_t e = 0; e < K; ++e) {
                        const uint32_t xb = (w[e].x >> s) & 1u;
                        if (xb) p[e] = cmul(p[e], z);
                        if (xb ^ cb) h[e] = cmul(h[e], z);
                    }
                }
            }
        }
        if (FULL && q.ngen) {
            cptr<TreePhase> ph = cp(opaque(Pg)->tree_phases) + q.gen_off;
            for (uint32_t j = 0; j < q.ngen; ++j) {
                const int32_t c = ph[j].choice;
                const double zi = ph[j].pi;
                const dv2 z = mk(ph[j].pr, (c >= 0 && ((ch >> (c & 31)) & 1u)) ? -zi : zi);
                const uint32_t cb = (pair.g >> j) & 1u;
#pragma unroll
                for (uint32_t e = 0; e < K; ++e) {
                    const uint32_t b = (w[e].g >> j) & 1u;
                    if (b) p[e] = cmul(p[e], z);
                    if (b ^ cb) h[e] = cmul(h[e], z);
                }
            }
        }
    }
    // what the pass makes of its pairs: writes at dp (and dh, half a state
    // on), and sums into v0, v1; i[] + il (il per lane): their coordinates
    template <uint32_t K, bool FULL>
    CSVM_INLINE void finish(cptr<DevProgram> Pg, const Pass& q, AmpT* dp, AmpT* dh, uint32_t ch, const Words (&w)[K],
                            const uint32_t (&i)[K], uint32_t il, bool ok, dv2 (&p)[K], dv2 (&h)[K], double& v0, double& v1) {
        const uint32_t type = q.type;
        if (type == TREE_INTERFERE || type == TREE_H) {
            // the relative sign goes into the additions: +-1 times h
#pragma unroll
            for (uint32_t e = 0; e < K; ++e) {
                const double sg = __hiloint2double((int)(0x3FF00000u | (w[e].s & 0x80000000u)), 0);
                dv2 s, d;
                if (q.quarter) {  // uniform: times +-i
                    s = mk(__fma_rn(h[e].y, -sg, p[e].x), __fma_rn(h[e].x, sg, p[e].y));
                    d = mk(__fma_rn(h[e].y, sg, p[e].x), __fma_rn(h[e].x, -sg, p[e].y));
                } else {
                    s = mk(__fma_rn(h[e].x, sg, p[e].x), __fma_rn(h[e].y, sg, p[e].y));
                    d = mk(__fma_rn(h[e].x, -sg, p[e].x), __fma_rn(h[e].y, -sg, p[e].y));
                }
                if (ok) {
                    *at(dp, w[e].o) = cscale(s, kInvSqrt2);
                    *at(dh, w[e].o) = cscale(d, kInvSqrt2);
                }
                v0 = __fma_rn(s.x, s.x, __fma_rn(s.y, s.y, v0));
                v1 = __fma_rn(d.x, d.x, __fma_rn(d.y, d.y, v1));
            }
            return;
        }
        if (type != TREE_COPY) {
            // (the quarter turn of a diagonal measurement's upper half is a
            // phase of the whole outcome, but U2 and EXP_VAL need it)
#pragma unroll
            for (uint32_t e = 0; e < K; ++e) {
                const uint32_t s = w[e].s & 0x80000000u;
                if (q.quarter && FULL) h[e] = mk(-h[e].y, h[e].x);
                h[e] = mk(flip(h[e].x, s), flip(h[e].y, s));
            }
        }
        if (FULL && type >= TREE_EV) {
            const uint32_t evz = q.head(12), half = 1u << (q.r - 1u);
            const bool imag = q.head(13) != 0u;
#pragma unroll
            for (uint32_t e = 0; e < K; ++e) {
                const double zl = odd(i[e] + il, evz) ? -1.0 : 1.0, zh = odd(i[e] + half + il, evz) ? -1.0 : 1.0;
                const double np = p[e].x * p[e].x + p[e].y * p[e].y, nh = h[e].x * h[e].x + h[e].y * h[e].y;
                v1 += np + nh;
                if (type == TREE_EV0) {
                    v0 += zl * np + zh * nh;
                } else {
                    const double re = h[e].x * p[e].x + h[e].y * p[e].y, im = h[e].x * p[e].y - h[e].y * p[e].x;
                    v0 += imag ? -(zl * im - zh * im) : (zl + zh) * re;
                }
            }
            return;
        }
        if (FULL && type == TREE_U2) {
            const double* m = &opaque(Pg)->u2[q.head(10)].matrices[(ch >> q.head(11)) & 3u][0][0];
            const dv2 m00 = mk(m[0], m[1]), m01 = mk(m[2], m[3]), m10 = mk(m[4], m[5]), m11 = mk(m[6], m[7]);
#pragma unroll
            for (uint32_t e = 0; e < K; ++e) {
                const dv2 a = p[e], b = h[e];
                p[e] = cadd(cmul(m00, a), cmul(m01, b));
                h[e] = cadd(cmul(m10, a), cmul(m11, b));
            }
        }
#pragma unroll
        for (uint32_t e = 0; e < K; ++e) {
            if (ok) {
                *at(dp, w[e].o) = p[e];
                *at(dh, w[e].o) = h[e];
            }
            v0 = __fma_rn(p[e].x, p[e].x, __fma_rn(p[e].y, p[e].y, v0));
            v1 = __fma_rn(h[e].x, h[e].x, __fma_rn(h[e].y, h[e].y, v1));
        }
    }
    // a times the relative turn of a quad's corner (bit 31: corner 1, ...)
    CSVM_INLINE static dv2 corner(dv2 a, const Pass& q, uint32_t s, uint32_t bit) {
        const uint32_t f = (s >> bit) << 31;
        if ((q.quarter >> bit) & 1u) a = mk(-a.y, a.x);
        return mk(flip(a.x, f), flip(a.y, f));
    }
    // U4: quads of the top two coordinate bits, one at a time per lane
    CSVM_INLINE void pass_u4(cptr<DevProgram> Pg, const Pass& q) {
        const uint32_t s = q.r - 2u, n4 = 1u << s;
        const size_t total = (size_t)N << s;
        const Words c2 = q.template column<true>(q.r - 2u), c3 = q.template column<true>(q.r - 1u);
        for (size_t f0 = (size_t)wave << 6; f0 < total; f0 += (size_t)nwaves << 6) {
            const bool in = f0 + lane < total;
            const size_t f = in ? f0 + lane : 0;  // lanes past the end repeat the first quad
            const uint32_t n = (uint32_t)(f >> s), i = (uint32_t)f & (n4 - 1u);
            Words x = {0u, 0u, q.sign0, 0u};
            for (uint32_t b = 0; b < s; ++b) {
                const Words c = q.template column<true>(b);
                if ((i >> b) & 1u) x = x ^ c;
            }
            const uint32_t ch = nch[n];
            // the pairs (bit r-2 clear, bit r-1 free) and (bit r-2 set, bit r-1 free)
            const Words w[2] = {x, x ^ c2};
            dv2 lo[2], hi[2];
            gather<2, true>(Pg, q, src + ((size_t)nsrc[n] << q.r0), ch, c3, w, lo, hi);
            lo[1] = corner(lo[1], q, x.s, 31u);
            hi[0] = corner(hi[0], q, x.s, 30u);
            hi[1] = corner(hi[1], q, x.s, 29u);
            if (in) {
                const double* m = &opaque(Pg)->u4[q.head(10)].entries[(ch >> q.head(11)) & 15u].matrix[0][0][0];
                AmpT* dp = dst + ((size_t)n << q.r);
#pragma unroll 1
                for (uint32_t row = 0; row < 4; ++row) {
                    const double* e = m + 8 * row;
                    dv2 acc = cmul(mk(e[0], e[1]), lo[0]);
                    acc = cadd(acc, cmul(mk(e[2], e[3]), lo[1]));
                    acc = cadd(acc, cmul(mk(e[4], e[5]), hi[0]));
                    acc = cadd(acc, cmul(mk(e[6], e[7]), hi[1]));
                    dp[i + row * n4] = acc;
                }
            }
        }
    }
    // A unit of a node: 2^ub wavefront steps of 64 pairs in Gray order from
    // coordinate i0 (words wu, uniform) on, K pairs per lane at a time.
    template <uint32_t K, bool FULL>
    CSVM_INLINE void unit(cptr<DevProgram> Pg, const Pass& q, const AmpT* sp, AmpT* dp, AmpT* dh, uint32_t ch,
                          const Words& pair, const Words& wl, Words wu, uint32_t i0, uint32_t steps, double& v0, double& v1) {
        for (uint32_t j0 = 0; j0 < steps; j0 += K) {
            uint32_t i[K];
            Words w[K];
#pragma unroll
            for (uint32_t e = 0; e < K; ++e) {
                if (j0 + e != 0u) {  // one coordinate bit flips
                    const uint32_t b = 6u + (uint32_t)__builtin_ctz(j0 + e);
                    i0 ^= 1u << b;
                    wu = wu ^ q.template column<FULL>(b);
                }
                i[e] = i0;
                w[e] = wl ^ wu;
            }
            dv2 p[K], h[K];
            gather<K, FULL>(Pg, q, sp, ch, pair, w, p, h);
            finish<K, FULL>(Pg, q, dp, dh, ch, w, i, lane, true, p, h, v0, v1);
        }
    }
    // The pass over nodes of 64 pairs or more: a wavefront takes a unit at a
    // time.  A node's units are dealt to 2^pb sums.
    template <uint32_t K, bool FULL>
    CSVM_INLINE void units(cptr<DevProgram> Pg, const Pass& q, const Words& pair, const Words& wl, uint32_t ub, uint32_t upn,
                           uint32_t pb) {
        const uint32_t t = q.r - 1u, steps = 1u << ub, items = N << pb, pp = 1u << pb;
        for (uint32_t item = wave; item < items; item += nwaves) {
            const uint32_t n = item >> pb;
            const AmpT* sp = src + ((size_t)uni(nsrc[n]) << q.r0);
            AmpT* dp = dst + ((size_t)n << q.r);
            AmpT* dh = dp + (1u << t);
            const uint32_t ch = uni(nch[n]);
            double v0 = 0.0, v1 = 0.0;
            Words wu = {0u, 0u, 0u, 0u};
            uint32_t before = 0;
            for (uint32_t u = item & (pp - 1u); u < upn; u += pp) {
                for (uint32_t d = u ^ before; d; d &= d - 1u)
                    wu = wu ^ q.template column<FULL>(6u + ub + (uint32_t)__builtin_ctz(d));
                before = u;
                unit<K, FULL>(Pg, q, sp, dp, dh, ch, pair, wl, wu, u << (6u + ub), steps, v0, v1);
            }
            lanes_sum(v0, v1, 6u);
            if (lane == 0u) {
                lds_f64* o = pb == 0u ? psum : part;
                o[2 * item] = v0;
                o[2 * item + 1] = v1;
            }
        }
    }

    // The next pass over every node.  Afterwards psum holds the nodes' sums
    // (pairs (v0, v1)), written states are in src, and every wavefront sees
    // both.  Returns the pass's rank and type through the arguments.
    CSVM_INLINE void pass(cptr<DevProgram> Pg, uint32_t& rank, int32_t& ev_sign) {
        Pass q;
        q.wa = wa;
        q.wb = wb;
        q.wc = wc;
        q.type = q.head(0);
        q.r0 = q.head(1);
        q.r = q.head(3);
        q.quarter = q.head(4);
        q.ngen = q.head(5);
        q.gen_off = q.head(6);
        q.sign0 = q.head(7);
        q.ez_choices = q.head(8);
        q.lo = (16u << q.r0) - 1u;
        rank = q.r;
        ev_sign = (int32_t)q.head(14);
        const uint32_t reset = q.head(9), t = q.r - 1u;
        const bool full = q.r0 != q.r || q.ngen || q.type > TREE_H;
        if (q.r0 != q.r && !q.ez_choices && tid < (1u << (q.r - q.r0))) {
            cptr<TreePass> T = cp(opaque(Pg)->tree_passes) + next;
            stage->tab[tid][0] = T->ez_tab[tid][0];
            stage->tab[tid][1] = T->ez_tab[tid][1];
        }
        __syncthreads();  // the stage, and the node tables of the last split
        uint32_t pb = 0;  // sums per node: 2^pb
        if (q.type == TREE_U4) {
            pass_u4(Pg, q);
        } else {
            const Words pair = q.template column<true>(t);
            // the part of the words that a lane's own coordinate bits give
            Words wl = {0u, 0u, q.sign0, 0u};
            const uint32_t lb = t < 6u ? t : 6u;
            for (uint32_t b = 0; b < lb; ++b) {
                const Words c = q.template column<true>(b);
                if ((lane >> b) & 1u) wl = wl ^ c;
            }
            if (t <= 6u) {
                // one pair per lane, 2^(6-t) nodes per wavefront step
                const uint32_t total = N << t, il = lane & ((1u << t) - 1u), zero[1] = {0u};
                const Words w[1] = {wl};
                for (uint32_t f0 = wave << 6; f0 < total; f0 += nwaves << 6) {
                    const bool ok = f0 + lane < total;
                    const uint32_t n = ok ? (f0 + lane) >> t : 0u;  // lanes past the end repeat node 0
                    const uint32_t ch = nch[n];
                    dv2 p[1], h[1];
                    double v0 = 0.0, v1 = 0.0;
                    AmpT* dp = dst + ((size_t)n << q.r);
                    gather<1, true>(Pg, q, src + ((size_t)nsrc[n] << q.r0), ch, pair, w, p, h);
                    finish<1, true>(Pg, q, dp, dp + (1u << t), ch, w, zero, il, ok, p, h, v0, v1);
                    lanes_sum(v0, v1, t);
                    if (ok && il == 0u) {
                        psum[2 * n] = v0;
                        psum[2 * n + 1] = v1;
                    }
                }
            } else {
                const uint32_t ub = t - 6u < 3u ? t - 6u : 3u, upn = 1u << (t - 6u - ub);
                // about kTreeParts sums for the team to work on
                while ((1u << pb) < upn && pb < 6u && (2u << pb) * N <= kTreeParts) ++pb;
                if (full || ub == 1u)
                    units<2, true>(Pg, q, pair, wl, ub, upn, pb);
                else
                    units<G, false>(Pg, q, pair, wl, ub, upn, pb);
            }
        }
        load_pass(Pg, next + 1u);  // the table ends with a spare entry
        __syncthreads();
        if (pb) {  // a node's partial sums, in order
            if (tid < N) {
                const lds_f64* o = part + ((2u * tid) << pb);
                double v0 = o[0], v1 = o[1];
                for (uint32_t j = 1; j < (1u << pb); ++j) {
                    v0 += o[2 * j];
                    v1 += o[2 * j + 1];
                }
                psum[2 * tid] = v0;
                psum[2 * tid + 1] = v1;
            }
            __syncthreads();
        }
        if (q.type < TREE_EV) {
            AmpT* w = src;
            src = dst;
            dst = w;
            if (q.type != TREE_DIAG && q.type != TREE_INTERFERE)
                for (uint32_t n = tid; n < N; n += nthreads) {
                    nsrc[n] = n;
                    if (reset) nch[n] = 0u;
                }
        }
    }

    // The measurement's shots draw (or are told) their outcomes and part.
    CSVM_INLINE void measure(cptr<TreeQuad> row, uint32_t units, uint32_t rank, uint32_t idx, bool forced_op) {
        uint32_t b = 0, need = 0;
        double pb = 0.0;
        if (live) {
            const double p0 = psum[2 * node], p1 = psum[2 * node + 1], total = p0 + p1;
            if (forced_op) {
                // the response still holds the record of outcome 0
                b = (forced[idx] ? 1u : 0u) ^ bits(idx, 1u);
                if (!forced_branch(p0, p1, total, b)) {
                    reachable = 0;
                    live = 0;
                }
            } else {
                b = sample_branch(p0, p1, total);
            }
            // svm.h:177-186 rescales the array once |gamma|, the inverse of
            // its norm, leaves [1e-100, 1e100]
            pb = b ? p1 : p0;
            need = (pb < 1e-200 && pb > 0.0) || pb > 1e200;
        }
        add_row(row, units, live && b);
        const uint32_t key = 2u * node + b, id = renumber(key, 2u * N, need);
        if (live) {
            nsrc2[id] = key;
            nch2[id] = 0u;
            node = id;
        }
        const bool rescale = uni(flags[scale_word]) != 0u;
        swap_tables();
        if (rescale) {  // a node's shots have the same pb
            __syncthreads();
            if (live) psum[node] = need ? 1.0 / sqrt(pb) : 1.0;
            __syncthreads();
            for (uint32_t n = 0; n < N; ++n) {
                const double s = unid(psum[n]);
                AmpT* a = src + ((size_t)uni(nsrc[n]) << (rank - 1u));
                if (s != 1.0)
                    for (uint32_t i = tid; i < (1u << (rank - 1u)); i += nthreads) a[i] = cscale(a[i], s);
            }
            __syncthreads();
        }
    }

    // ---------------------------------------------------------------- dispatch
    // Walks the bytecode.  Opcodes that hold barriers are run by every
    // thread, the others by the live shots.
    CSVM_INLINE void run(cptr<DevProgram> Pg, double* ev_row) {
        const uint32_t n_instr = opaque(Pg)->tree_n;
        cptr<uint64_t> code = (cptr<uint64_t>)cp(opaque(Pg)->tree_bc);
        uint64_t n0 = code[0], n1 = code[1], n2 = code[2];
        for (uint32_t pc = 0; pc < n_instr; ++pc) {
            const uint64_t w0 = n0, w1 = n1, w2 = n2;
            code = opaque(code + 4);  // (the next instruction arrives while this one runs)
            n0 = code[0];
            n1 = code[1];
            n2 = code[2];
            const uint32_t op = (uint32_t)(w0 & 0xFF), reserved = (uint32_t)(w0 >> 8) & 0xFFu;
            const uint32_t count = (uint32_t)((w0 >> 32) & 0xFFFF), i0 = (uint32_t)w1, i1 = (uint32_t)(w1 >> 32);
            const uint32_t units = (uint32_t)(w0 >> 48);
            cptr<DevProgram> P = opaque(Pg);
            if (op == kLpNoise) {
                while (next_noise >= i0 && next_noise < i1) noise(P);  // (a dead shot's index is kNoNoise)
            } else if (op == kTreeMeas || op == kTreePass || op == kTreeEv) {
                uint32_t rank = 0;
                int32_t ev_sign = 1;
                if (op != kTreeEv || w2 == 0u) pass(Pg, rank, ev_sign);
                if (op == kTreeMeas) {
                    measure(row_at(opaque(Pg), i1), units, rank, i0, reserved != 0u);
                    if (!live) next_noise = kNoNoise;
                } else if (op == kTreeEv && live && ev_row) {
                    double v = w2 == 1u ? 0.0 : 1.0;
                    if (w2 == 0u) {
                        const double den = psum[2 * node + 1];
                        v = den > 0.0 ? (double)ev_sign * psum[2 * node] / den : 0.0;
                    }
                    if (bits(i1, 1u)) v = -v;
                    v = v > 1.0 ? 1.0 : v;
                    ev_row[i0] = v < -1.0 ? -1.0 : v;
                }
            } else if (op == kLpRandom) {
                add_rows(row_at(P, i1), units, count, [&] { return live && (rng_next(rng) >> 63); });  // the draw is not below 1/2
            } else if (op == kLpReadout) {
                uint32_t r = i0;
                add_rows(row_at(P, i1), units, count, [&] {
                    bool fire = false;
                    if (live) {
                        if (kf) {
                            fire = kf_rpos < kf_n && kf[kf_rpos << 6] == r;
                            if (fire) kf_rpos++;
                        } else {
                            fire = rng_double(rng) < cp(P->ro_prob)[r];
                        }
                    }
                    ++r;
                    return fire;
                });
            } else if (op == kTreeChoice) {
                choice_split(bits(i0, reserved), reserved, (uint32_t)w2);
            } else if (op == kTreeNode) {
                const uint32_t st = bits(i1, reserved);
                const uint32_t o = reserved == 4u ? P->u4[i0].entries[st].out_state : P->u2[i0].out_states[st];
                for (uint32_t j = 0; j < reserved; ++j) add_row(row_at(P, (uint32_t)w2 + j * units), units, live && ((o >> j) & 1u));
            } else if (op == kLpPostselect) {
                if (live && bits(i0, 1u)) {
                    cptr<uint32_t> row = cp(P->lp_dense) + (size_t)i1 * P->lp_words;
                    for (uint32_t w = 0; w < P->lp_words; ++w) R[w << 6] &= row[w];
                    discarded = 1;
                    live = 0;
                    next_noise = kNoNoise;
                }
            } else if (op == kLpCoin) {
                bool one = false;
                if (live) {
                    logp += log(0.5);
                    one = (forced[i0] ? 1u : 0u) != bits(i0, 1u);
                }
                add_row(row_at(P, i1), units, one);
            } else {  // kLpStatic
                if (live && (forced[i0] ? 1u : 0u) != bits(i0, 1u)) {
                    reachable = 0;
                    live = 0;
                    next_noise = kNoNoise;
                }
            }
        }
    }
};

// Rows of n bits of a wavefront's first `shots` shots, shot f of the launch
// on, from response word w0 on: one byte a bit, or 8 bits a byte.  The rows
// are consecutive bytes, so the lanes write them 16 bytes (packed: 4 bytes)
// a step, wherever shots begin, and not each its own shot byte by byte.
CSVM_INLINE void tree_write_section(uint8_t* out, uint64_t f, uint32_t shots, uint32_t n, bool packed,
                                    const tree_lds_u32* wave_R, uint32_t w0, uint32_t lane) {
    if (!out || n == 0 || shots == 0) return;
    const tree_lds_u32* R = wave_R + (w0 << 6);
    const uint32_t row = packed ? (n + 7u) / 8u : n, total = shots * row, unit = packed ? 4u : 16u;
    uint8_t* to = out + f * row;
    const uint32_t head = (uint32_t)(reinterpret_cast<uintptr_t>(to) & (unit - 1u));
    for (uint32_t b = unit * lane; b < total + head; b += 64u * unit) {
        // bytes [lo, hi) of the section; lo is unit-aligned except at its start
        const uint32_t lo = b < head ? 0u : b - head, hi = b + unit - head < total ? b + unit - head : total;
        uint32_t s = lo / row, i = lo - s * row, acc = 0;
        for (uint32_t t = lo; t < hi;) {
            const uint32_t take = hi - t < row - i ? hi - t : row - i;
            const tree_lds_u32* col = R + s;
            if (packed) {
                const uint32_t w = i >> 2, sh = (i & 3u) * 8u;
                uint64_t x = col[w << 6];
                if (sh && (w + 1u) * 4u < row) x |= (uint64_t)col[(w + 1u) << 6] << 32;
                const uint32_t m = take < 4u ? (1u << (8u * take)) - 1u : 0xFFFFFFFFu;
                acc |= ((uint32_t)(x >> sh) & m) << (8u * (t - lo));
            } else {
                const uint32_t w = i >> 5, sh = i & 31u;
                uint64_t x = col[w << 6];
                if (sh + take > 32u) x |= (uint64_t)col[(w + 1u) << 6] << 32;
                acc |= ((uint32_t)(x >> sh) & ((1u << take) - 1u)) << (t - lo);
            }
            t += take;
            i = 0;
            ++s;
        }
        if (packed) {
            if (hi - lo == 4u)
                *reinterpret_cast<uint32_t*>(to + lo) = acc;
            else
                for (uint32_t t = lo; t < hi; ++t) to[t] = (uint8_t)(acc >> (8u * (t - lo)));
        } else if (hi - lo == 16u) {
            // bits 4j .. 4j + 3 to the bytes of word j
            TreeQuad q;
#pragma unroll
            for (uint32_t j = 0; j < 4; ++j) q[j] = (((acc >> (4u * j)) & 15u) * 0x00204081u) & 0x01010101u;
            *reinterpret_cast<TreeQuad*>(to + lo) = q;
        } else {
            for (uint32_t t = lo; t < hi; ++t) to[t] = (uint8_t)((acc >> (t - lo)) & 1u);
        }
    }
}

// What the wavefront's shots leave; s: this lane's shot within the launch,
// if `mine`, f the first lane's.
template <class S>
CSVM_INLINE void tree_write_rows(cptr<DevProgram> P, cptr<ShotArgs> A, const S& shot, uint64_t s, uint64_t f, bool mine) {
    const bool packed = (A->flags & CLIFFT_REC_PACKED) != 0;
    const uint32_t shots = (uint32_t)__builtin_popcountll(__ballot(mine));
    const uint32_t wm = lane_words(P->num_meas), wd = lane_words(P->num_det);
    cptr<uint8_t> expo = cp(P->expected_obs);
    for (uint32_t i = 0; i < P->n_expected_obs && i < P->num_obs; ++i)
        if (load_u8(expo, i)) shot.R[(wm + wd + (i >> 5)) << 6] ^= 1u << (i & 31u);
    tree_wave_fence();
    const tree_lds_u32* R = shot.R - shot.lane;
    tree_write_section(A->out_meas, f, shots, P->num_meas, packed, R, 0, shot.lane);
    tree_write_section(A->out_det, f, shots, P->num_det, packed, R, wm, shot.lane);
    tree_write_section(A->out_obs, f, shots, P->num_obs, packed, R, wm + wd, shot.lane);
    tree_wave_fence();  // (the next chunk's shots overwrite the columns)
    if (!mine) return;
    if (A->out_disc) A->out_disc[s] = (uint8_t)shot.discarded;
    if (A->mode == MODE_FORCED && A->out_logp) A->out_logp[s] = shot.reachable ? shot.logp : kUnreachable;
    if (shot.dust && A->dust_counter) atomicAdd(A->dust_counter, (unsigned long long)shot.dust);
}

template <class AmpT>
__device__ __forceinline__ void tree_range(cptr<DevProgram> Pg, cptr<ShotArgs> Ag, uint64_t c_first, uint64_t c_step,
                                           uint64_t s_lo, uint64_t s_hi, uint64_t seed, dv2* buf) {
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
    typedef TreeInterp<AmpT> Interp;
    typedef tree_lds_u32 lds_u32;
    Interp S;
    S.tid = threadIdx.x;
    S.lane = threadIdx.x & 63u;
    S.wave = uni(threadIdx.x >> 6);
    S.nthreads = blockDim.x;
    S.nwaves = blockDim.x >> 6;
    cptr<DevProgram> P = opaque(Pg);
    cptr<ShotArgs> A = opaque(Ag);
    const uint32_t chunk = A->tree_chunk, amp = A->amp_elems;
    const uint32_t words = P->lp_words, kf_words = A->mode == MODE_KFAULT ? 5u * cp(A->kf)->k : 0u;
    unsigned char* p = smem;
    AmpT *b0, *b1;
    if (std::is_same<AmpT, lds_d2>::value) {
        b0 = (AmpT*)((dv2*)p);
        b1 = b0 + amp;
        p += 32u * (size_t)amp;
    } else {
        b0 = (AmpT*)buf;
        b1 = b0 + amp;
    }
    lds_u32* tables = (lds_u32*)p;
    p += (16u * chunk + 15u) / 16u * 16u;
    S.psum = (lds_f64*)p;
    S.part = S.psum + 2 * chunk;
    p += 16u * chunk + 16u * kTreeParts;
    lds_u32* flag0 = (lds_u32*)p;
    const uint32_t fwords = tree_flag_words(chunk);
    p += (8u * fwords + 15u) / 16u * 16u;
    S.stage = (typename Interp::lds_stage*)p;
    p += sizeof(TreeStage);
    S.R = (lds_u32*)(p + (size_t)S.wave * (words + kf_words) * 256u) + S.lane;
    S.scale_word = fwords - 1u;
    for (uint64_t c = c_first;; c += c_step) {
        const uint64_t s0 = s_lo + c * chunk;
        if (s0 >= s_hi) break;
        const uint64_t s = s0 + S.tid;
        const bool mine = S.tid < chunk && s < s_hi;
        A = opaque(Ag);
        P = opaque(Pg);
        {
            cptr<uint32_t> first = cp(P->lp_dense);  // the constants
            for (uint32_t w = 0; w < words; ++w) S.R[w << 6] = first[w];
        }
        S.dust = 0;
        S.discarded = 0;
        S.reachable = 1;
        S.logp = 0.0;
        S.forced = nullptr;
        S.kf = nullptr;
        S.kf_nn = S.kf_pos = S.kf_n = S.kf_rpos = 0;
        S.next_noise = kNoNoise;
        S.load_pass(P, 0);
        S.rng = rng_for_shot(seed, A->shot_begin + s);
        S.live = mine ? 1u : 0u;
        S.node = 0;
        S.N = 1;
        S.src = b0;
        S.dst = b1;
        S.nsrc = tables;
        S.nsrc2 = tables + chunk;
        S.nch = tables + 2 * chunk;
        S.nch2 = tables + 3 * chunk;
        S.flags = flag0;
        S.flags2 = flag0 + fwords;
        double* ev_row = nullptr;
        // svm.cc:602-606: no gap draw, fault set first
        if (A->mode == MODE_KFAULT) S.kfault_prepare(cp(A->kf), S.R + (words << 6), mine);
        if (mine) {
            if (A->mode != MODE_KFAULT) {
                S.next_noise = 0;
                S.draw_next_noise(P, 0.0);
            }
            if (A->mode == MODE_FORCED) S.forced = A->forced_records + s * P->num_meas;
            const uint32_t nev = P->num_ev;
            ev_row = A->out_ev ? A->out_ev + s * nev : nullptr;
            if (ev_row)
                for (uint32_t i = 0; i < nev; ++i) ev_row[i] = 0.0;
        }
        if (S.tid == 0) {
            S.nsrc[0] = 0u;
            S.nch[0] = 0u;
            if (amp) S.src[0] = mk(1.0, 0.0);
        }
        __syncthreads();

        S.run(Pg, ev_row);

        tree_write_rows(opaque(Pg), opaque(Ag), S, s, s0 + 64u * S.wave, mine);
        __syncthreads();  // the tables and the state are rewritten by the next chunk
    }
}

}  // namespace csvm
