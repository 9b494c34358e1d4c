// swmi_device.h -- device helpers shared by the kernels: address-space views, the lcg32 parameter pairs, the
// flip rules, the union-finds in LDS and in HBM, and the decomposition of the work list into blocks.
#pragma once

#include <hip/hip_runtime.h>

#include <algorithm>
#include <type_traits>

#include "swmi_internal.h"

namespace swmi
{
    __device__ __forceinline__ uint32_t Uniform(const uint32_t v) { return __builtin_amdgcn_readfirstlane(v); }

    // The buffers are reached through pointers stored in the lattice descriptor, which the compiler sees
    // as generic (FLAT) addresses; FLAT accesses wait on both the memory and the LDS counters. Every
    // buffer access goes through a global-address-space view instead.
    template <typename T>
    using gptr = __attribute__((address_space(1))) T*;

    template <typename T>
    __device__ __forceinline__ gptr<T> Glob(T* p)
    {
        return (gptr<T>)(p);
    }

    // plain vector types (HIP's uint2/uint4 classes cannot be assigned through address-space-1 pointers)
    using u32x2 = uint32_t __attribute__((ext_vector_type(2)));
    using u32x4 = uint32_t __attribute__((ext_vector_type(4)));

    // Buffer views (raw: stride 0, byte offsets). The hardware checks a lane's offset against the view's
    // size and drops a store past it, which lets a lane opt out of a store without an exec mask.
    using Rsrc = __amdgpu_buffer_rsrc_t;
    constexpr uint32_t kNoStore = 0x80000000u;   // a lane offset past every view
    template <typename T>
    __device__ __forceinline__ Rsrc MakeRsrc(T* base, const uint32_t bytes)
    {
        return __builtin_amdgcn_make_buffer_rsrc(static_cast<void*>(base), 0, static_cast<int>(bytes), 0x00020000);
    }

    // bit `lane` of a wave-uniform mask, as a per-lane predicate (v_cndmask on the SGPR pair)
    __device__ __forceinline__ bool LaneBit(const uint64_t mask) { return __builtin_amdgcn_inverse_ballot_w64(mask); }

    // 64-bit shifts by 0..64 (a shift by 64 yields 0; the hardware would use the count modulo 64)
    __device__ __forceinline__ uint64_t Shr(const uint64_t v, const uint32_t s) { return s >= 64u ? 0ull : v >> s; }
    __device__ __forceinline__ uint64_t Shl(const uint64_t v, const uint32_t s) { return s >= 64u ? 0ull : v << s; }

    __device__ __forceinline__ uint32_t ReadLane(const uint32_t v, const uint32_t lane)
    {
        return static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(v), static_cast<int>(lane)));
    }

    // Numerical Recipes pair k of random/src/lcg32.cpp:18-24.
    __device__ __forceinline__ void ParamsOf(const uint32_t k, uint32_t& a, uint32_t& c)
    {
        const bool b0 = (k & 1u) != 0u, b1 = (k & 2u) != 0u, b2 = (k & 4u) != 0u;
        const uint32_t a01 = b0 ? 2891336453u : 1372383749u;
        const uint32_t a23 = b0 ? 32310901u : 2024337845u;
        const uint32_t c01 = b0 ? 1640531513u : 1289706101u;
        const uint32_t c23 = b0 ? 626627237u : 797082193u;
        a = b2 ? 29943829u : (b1 ? a23 : a01);
        c = b2 ? 1013904223u : (b1 ? c23 : c01);
    }

    // Offset added to the rotation at update `it` (random/src/lcg32.cpp:56-64): state[it & 63] + (it even).
    __device__ __forceinline__ uint32_t ShuffleShift(const uint32_t st, const uint32_t it)
    {
        return ReadLane(st, it & 63u) + ((it & 1u) ? 0u : 1u);
    }

    // ---- random flip rule: MurmurHash3 (Austin Appleby, public domain). The cluster with canonical root r
    // flips iff the top bit of Fmix32(r ^ key) is set; key = MurmurHash3_x86_32 of the 4-byte lcg32
    // iteration count before the sweep, seeded with the lattice seed. ----
    __device__ __forceinline__ uint32_t Fmix32(uint32_t h)
    {
        h ^= h >> 16;
        h *= 0x85EBCA6Bu;
        h ^= h >> 13;
        h *= 0xC2B2AE35u;
        h ^= h >> 16;
        return h;
    }

    __device__ __forceinline__ uint32_t FlipKey(const uint32_t seed, const uint32_t iteration)
    {
        uint32_t k = iteration * 0xCC9E2D51u;
        k = (k << 15) | (k >> 17);
        k *= 0x1B873593u;
        uint32_t h = seed ^ k;
        h = (h << 13) | (h >> 19);
        h = h * 5u + 0xE6546B64u;
        return Fmix32(h ^ 4u);
    }

    // ---- union-find in LDS. Nodes are named by their byte offset into the workgroup's parent array P
    // (so no instruction scales an index into an address); parents satisfy P[x] <= x, so roots are cluster
    // minima. ----
    __device__ __forceinline__ uint32_t* At(uint32_t* P, const uint32_t off)
    {
        return reinterpret_cast<uint32_t*>(reinterpret_cast<char*>(P) + off);
    }

    // byte offset of the LDS word p from P
    __device__ __forceinline__ uint32_t OffsetFrom(const uint32_t* P, const uint32_t* p)
    {
        return static_cast<uint32_t>(reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) const uint32_t*)p) -
                                     reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) const uint32_t*)P));
    }

    __device__ __forceinline__ uint32_t LdsLoad(const uint32_t* p)
    {
        return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    }

    // An empty asm statement that reads v: v's load completes before this point, so it cannot be sunk past a
    // later branch (an early exit) and is waited for together with the loads issued beside it.
    __device__ __forceinline__ void Issued(const uint32_t v)
    {
        asm volatile("" ::"v"(v));
    }

    __device__ __forceinline__ void Issued(const uint64_t v)
    {
        asm volatile("" ::"v"(v));
    }

    // An empty asm statement that needs the uniform value v in scalar registers here: a descriptor field read
    // this way is fetched at this point, with the others read beside it, not at its first use.
    template <typename T>
    __device__ __forceinline__ void HeldScalar(const T v)
    {
        asm volatile("" ::"s"(v));
    }

    __device__ __forceinline__ void LdsMin(uint32_t* p, const uint32_t v)
    {
        (void)__hip_atomic_fetch_min(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    }

    // Down bonds are deduplicated before any union: lanes l-1 and l lie in the same "overlap interval"
    // when they share their row run above and their row run below (mask C); only the first down bond
    // of every interval can join two different clusters. With M = C << 1 (continuation) and
    // S1 = (D << 1) & M, the positions that follow an earlier bond of the same interval are
    // S1 | (M & ((M + S1) ^ M)) (carries of S1 run through the ones of M).
    __device__ __forceinline__ uint64_t FirstBondPerInterval(const uint64_t D, const uint64_t C, const uint64_t rowstart)
    {
        const uint64_t M = (C << 1) & ~rowstart;
        const uint64_t S1 = (D << 1) & M;
        const uint64_t later = S1 | (M & ((M + S1) ^ M));
        return D & ~later;
    }

    // Union of the pairs (a, b) held by the lanes, all lanes in lockstep. Each step moves the ends that
    // are not roots up (two parents, halving the path); when both are roots the larger is linked under the
    // smaller with atomicMin, and a lost race continues with the value found (the loop of the reference
    // Merge, swendsen_wang_amd_gpu.cpp:368-401). Lanes with nothing to do hold a == b; only lanes that
    // link issue the atomic (idle lanes would all hit the same word). a and b are byte offsets into P.
    __device__ __forceinline__ void LdsUnionLockstep(uint32_t* P, uint32_t a, uint32_t b)
    {
        while (__ballot(a != b))
        {
            // lanes that are done (a == b) only read P[a]; they follow no pointer and write nothing, so
            // their a may name a node another wave has not written yet
            const bool act = a != b;
            const uint32_t pa = LdsLoad(At(P, a));
            const uint32_t pb = LdsLoad(At(P, b));
            const bool roots = (pa == a) && (pb == b);
            const bool up = act && !roots;
            const uint32_t lo = min(a, b), hi = max(a, b);
            uint32_t old = hi;
            if (act && roots)
                old = __hip_atomic_fetch_min(At(P, hi), lo, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
            const bool linked = roots && old == hi;
            // ends that are not roots move two steps up and point their node at the grandparent (path
            // halving, monotone like every write to P)
            const uint32_t ga = up ? LdsLoad(At(P, pa)) : 0u;
            const uint32_t gb = up ? LdsLoad(At(P, pb)) : 0u;
            if (up && ga != pa)
                LdsMin(At(P, a), ga);
            if (up && gb != pb)
                LdsMin(At(P, b), gb);
            if (act)
            {
                a = roots ? (linked ? hi : lo) : ga;
                b = roots ? (linked ? hi : old) : gb;
            }
        }
    }

    // One row of a 64-wide tile joins the union-find: B are its bonds to the right (inside the tile), D the bonds
    // from the row above into it, Rp the root of this lane's site in the row above (resolved when that row was
    // labelled), self this lane's node. A row run's label is the minimum of its first site and the roots its down
    // bonds reach, taken by one LDS atomic per row: the run's word of M holds the maximum of base - node, and base
    // grows from row to row by more than any node (bits 16 and up, the low 16 all ones), so what earlier rows left
    // there is smaller than anything this row writes and no row clears its words. A bond to any other root links
    // that root under the minimum with one atomicMin, and only a link that loses a race goes through the lockstep
    // union. P[self] is left at the run's label, an ancestor; returns the root of this lane's site after the row's
    // links. M: 64 words of the wave, below base at the start; spare: a word of the lane's own, the target of LDS
    // operations the lane has no use for (both as byte offsets from P: the selects below are between offsets, and P's
    // address stays in the instructions' offset fields).
    // LDS operations are what a row waits for (about 7 cycles of the CU's one pipe per operation of a wave with scattered
    // roots, and the round trip): a row takes four and one per chase step, where clearing, minimum, entry and root as
    // separate operations took eight.
    __device__ __forceinline__ uint32_t LabelRow64(uint32_t* P, const uint32_t M, const uint32_t spare, const uint32_t self,
                                                   const uint64_t B, const uint64_t D, const uint32_t Rp, const uint32_t base)
    {
        // word of this lane's row run: the number of run starts after lane 0 up to this lane
        const uint32_t Mk = M + 4u * __builtin_amdgcn_mbcnt_hi(static_cast<uint32_t>(~B >> 32),
                                                               __builtin_amdgcn_mbcnt_lo(static_cast<uint32_t>(~B), 0u));
        // a run's first lane brings its own node, a bonded lane the root above (an earlier row's node, so smaller)
        const uint32_t x = LaneBit(D) ? Rp : self;
        (void)__hip_atomic_fetch_max(At(P, LaneBit(~(B << 1) | D) ? Mk : spare), base - x, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        uint32_t root = base - LdsLoad(At(P, Mk));
        __hip_atomic_store(At(P, self), root, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        // bonds to a root other than the run's minimum link that root under it
        const uint64_t mg = D & __ballot(Rp != root);
        if (mg != 0ull)
        {
            const uint32_t old = __hip_atomic_fetch_min(At(P, LaneBit(mg) ? Rp : spare), root, __ATOMIC_RELAXED,
                                                        __HIP_MEMORY_SCOPE_WORKGROUP);
            // Rp was no longer a root (another lane linked it first): join the two trees
            const uint64_t more = mg & __ballot(old != Rp) & __ballot(old != root);
            if (more != 0ull)
            {
                const bool mo = LaneBit(more);
                LdsUnionLockstep(P, mo ? root : 0u, mo ? old : 0u);
            }
            // the run's minimum may itself have been linked under another root
            for (;;)
            {
                const uint32_t pr = LdsLoad(At(P, root));
                if (!__ballot(pr != root))
                    break;
                root = pr;
            }
        }
        return root;
    }

    // base of LabelRow64 for the k-th row a wave labels, k from 1 to 65535
    __device__ __forceinline__ uint32_t RowBase(const uint32_t k) { return (k << 16) | 0xFFFFu; }

    // ---- union-find in HBM over the roots of edge-reaching clusters, one node per slot (every block numbers
    // its edge roots densely, so a block's nodes share a few cache lines). Entry of slot c: (key << 32) | parent
    // slot, where a root's key is its site index and a non-root holds its parent's key. Links are made with
    // agent-scope 64-bit atomicMin (the 8 XCD L2s are not coherent with each other for plain stores), which
    // orders by key first: a parent's key never exceeds its child's, so a tree's root is the minimum site of
    // its component. Chase loads are relaxed atomic loads (never hoisted by the compiler); a stale value is an
    // earlier parent, still an ancestor, and every link is decided by an atomicMin that returns the true value,
    // so staleness only costs retries and longer paths. ----
    __device__ __forceinline__ uint64_t SlotEntry(const uint32_t key, const uint32_t slot)
    {
        return (static_cast<uint64_t>(key) << 32) | slot;
    }

    __device__ __forceinline__ uint64_t CachedLoad64(gptr<uint64_t> p)
    {
        return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    }

    // Loads of the merge's chases. FRESH reads the entry as it is now, past the CU's cache (agent scope);
    // otherwise the load may hit a line the CU cached earlier in the kernel. Fresh loads cost memory traffic
    // and save retries: they pay where the merge is latency-bound, i.e. where all its blocks are resident at
    // once (LaunchMerge chooses).
    template <bool FRESH>
    __device__ __forceinline__ uint64_t ChaseLoad64(gptr<uint64_t> p)
    {
        return __hip_atomic_load(p, __ATOMIC_RELAXED, FRESH ? __HIP_MEMORY_SCOPE_AGENT : __HIP_MEMORY_SCOPE_WORKGROUP);
    }

    __device__ __forceinline__ uint64_t SlotLinkMin(gptr<uint64_t> p, const uint64_t v)
    {
        return __hip_atomic_fetch_min(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }

    // Union of the clusters of slots a and b (keys ka, kb), the loop of the reference Merge
    // (swendsen_wang_amd_gpu.cpp:368-401) on slot entries. The ends start as the listed roots k_bond_label
    // wrote (entry = (own key << 32) | self), so the first link is tried at once, without chasing: when a
    // concurrent union got there first, atomicMin returns the parent found and the loop continues from it.
    // Both ends are chased together (their loads in flight at once); a start node more than one hop from its
    // root is pointed at the root (the atomic returns nothing, so the wave does not wait for it). A slot out
    // of range or a parent with a larger key can only come from a broken invariant, which is reported through
    // the lattice's error flag instead of being followed.
    template <bool FRESH>
    __device__ void SlotUnion(gptr<uint64_t> E, uint32_t a, uint32_t ka, uint32_t b, uint32_t kb, const uint32_t nslots,
                              gptr<uint32_t> err)
    {
        if (a < nslots && b < nslots && ka != kb)
        {
            if (ka > kb)
            {
                const uint32_t t = a, tk = ka;
                a = b;
                ka = kb;
                b = t;
                kb = tk;
            }
            const uint64_t old = SlotLinkMin(&E[b], SlotEntry(ka, a));
            if (old == SlotEntry(kb, b) || static_cast<uint32_t>(old) == a)
                return;
            b = static_cast<uint32_t>(old);
            kb = static_cast<uint32_t>(old >> 32);
        }
        for (;;)
        {
            if (a >= nslots || b >= nslots)
                break;
            const uint32_t a0 = a, b0 = b;
            uint64_t ea = ChaseLoad64<FRESH>(&E[a]), eb = ChaseLoad64<FRESH>(&E[b]);
            uint32_t ha = 0, hb = 0;
            bool bad = false;
            while (static_cast<uint32_t>(ea) != a || static_cast<uint32_t>(eb) != b)
            {
                const uint32_t pa = static_cast<uint32_t>(ea), qa = static_cast<uint32_t>(ea >> 32);
                const uint32_t pb = static_cast<uint32_t>(eb), qb = static_cast<uint32_t>(eb >> 32);
                if (pa >= nslots || qa > ka || pb >= nslots || qb > kb)
                {
                    bad = true;
                    break;
                }
                if (pa != a)
                {
                    a = pa;
                    ka = qa;
                    ea = ChaseLoad64<FRESH>(&E[a]);
                    ++ha;
                }
                if (pb != b)
                {
                    b = pb;
                    kb = qb;
                    eb = ChaseLoad64<FRESH>(&E[b]);
                    ++hb;
                }
            }
            if (bad)
                break;
            if (ha > 1)
                (void)SlotLinkMin(&E[a0], SlotEntry(ka, a));
            if (hb > 1)
                (void)SlotLinkMin(&E[b0], SlotEntry(kb, b));
            if (a == b)
                return;
            if (ka > kb)
            {
                const uint32_t t = a, tk = ka;
                a = b;
                ka = kb;
                b = t;
                kb = tk;
            }
            const uint64_t old = SlotLinkMin(&E[b], SlotEntry(ka, a));
            if (old == SlotEntry(kb, b))
                return;
            b = static_cast<uint32_t>(old);
            kb = static_cast<uint32_t>(old >> 32);
        }
        (void)__hip_atomic_fetch_or(err, kErrLabelRange, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }

    // Key of the canonical root (the minimum site) of the cluster of slot c, whose entry e the caller loaded;
    // c_max bounds the slots. A chase that leaves the slots or meets a parent with a larger key clears ok.
    __device__ __forceinline__ uint32_t SlotRootKey(gptr<uint64_t> E, uint32_t c, uint64_t e, const uint32_t c_max, bool& ok)
    {
        uint32_t k = static_cast<uint32_t>(e >> 32);
        while (static_cast<uint32_t>(e) != c)
        {
            const uint32_t p = static_cast<uint32_t>(e), kp = static_cast<uint32_t>(e >> 32);
            if (p >= c_max || kp > k)
            {
                ok = false;
                break;
            }
            c = p;
            k = kp;
            e = CachedLoad64(&E[c]);
        }
        return static_cast<uint32_t>(e >> 32);
    }

    // ---- work decomposition ----
    // Workgroups are dispatched round-robin over the 8 XCDs; give each XCD a contiguous range of blocks
    // so that blocks that share cache lines (spin rows, halos) meet in the same L2.
    __device__ __forceinline__ uint32_t RemapBlock(const uint32_t units)
    {
        const uint32_t per = (units + kNumXcd - 1) / kNumXcd;
        return (blockIdx.x % kNumXcd) * per + blockIdx.x / kNumXcd;
    }

    // Lattice of block b in the work list; a work list of one lattice is passed as a null pointer, which
    // saves the dependent load of the block's entry before the descriptor.
    __device__ __forceinline__ uint32_t LatticeOf(const uint32_t* __restrict__ block_lat, const uint32_t b)
    {
        return block_lat ? block_lat[b] : 0u;
    }

    struct Block
    {
        uint32_t lb;       // block index within its lattice
        uint32_t sx, sy;   // block column, block row
        uint32_t wyb;      // first wave row of the block
        uint32_t nwr;      // wave rows in the block
        uint32_t stride;   // sites between consecutive wave rows (64 * tiles_x)
        uint32_t base;     // first site of the block
    };

    __device__ __forceinline__ Block DecodeBlock(const LatDesc& d, const uint32_t b)
    {
        Block bl;
        bl.lb = b - d.block_base;
        bl.sx = bl.lb % d.tiles_x;
        bl.sy = bl.lb / d.tiles_x;
        bl.wyb = bl.sy * kWavesPerBlock * d.twr;
        bl.nwr = min(kWavesPerBlock * d.twr, d.nwr_y - bl.wyb);
        bl.stride = 64u * d.tiles_x;
        bl.base = bl.wyb * bl.stride + bl.sx * 64u;
        return bl;
    }

    __device__ __forceinline__ uint32_t BlockBase(const LatDesc& d, const uint32_t sx, const uint32_t sy)
    {
        return sy * kWavesPerBlock * d.twr * 64u * d.tiles_x + sx * 64u;
    }

    __device__ __forceinline__ uint32_t SiteOf(const uint32_t base, const uint32_t stride, const uint32_t q)
    {
        return base + (q >> 6) * stride + (q & 63u);
    }

    // ---- the flip rule (reference FlipClusters_Kernel, swendsen_wang_amd_gpu.cpp:445-467) ----
    // Row-major site index of a padded site index p (d.n0 is the row pitch, d.n0v the lattice width).
    __device__ __forceinline__ uint32_t RealSite(const LatDesc& d, const uint32_t p)
    {
        return d.n0v == d.n0 ? p : (p / d.n0) * d.n0v + p % d.n0;
    }

    // The flip rule for the cluster whose canonical root is the padded site `root`. The pitch and the width
    // are even, so a padded index and its row-major index have the same parity.
    __device__ __forceinline__ uint32_t FlipBit(const LatDesc& d, const uint32_t root, const bool random_rule, const uint32_t key)
    {
        return random_rule ? (Fmix32(RealSite(d, root) ^ key) >> 31) : (root & 1u);
    }

    // A block's flip bitmap has one bit per label index: bit q (q < qcap) for the cluster rooted at block-local
    // index q that stays inside the block, the rule applied to the root's own site; bit qcap + s for the
    // edge-reaching cluster whose root holds slot s, the rule applied to its canonical root (set by the
    // resolve). Word w of the rule part: bit j for q = 32w + j (block bases and row strides are even, so under
    // the parity rule q's parity is its site's parity).
    __device__ __forceinline__ uint32_t RuleWord(const LatDesc& d, const Block& bl, const uint32_t w, const bool random_rule,
                                                 const uint32_t key)
    {
        if (!random_rule)
            return 0xAAAAAAAAu;
        uint32_t v = 0;
        for (uint32_t j = 0; j < 32u; ++j)
            v |= FlipBit(d, SiteOf(bl.base, bl.stride, 32u * w + j), true, key) << j;
        return v;
    }

    static inline uint32_t XcdGrid(const uint32_t units) { return ((units + kNumXcd - 1) / kNumXcd) * kNumXcd; }
}
