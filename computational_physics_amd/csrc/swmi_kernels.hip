// swmi_kernels.hip -- gfx950 kernels of the Swendsen-Wang engine.
//
// One sweep of tiled lattices = three launches over the engine's block work list (all lattices of the engine at once):
//   k_bond_label  (swmi_bond.hip) per block (one workgroup of 4, 8 or 16 wavefronts): applies the previous sweep's
//                 cluster flip to each site as it loads it (label -> bit of the block's flip bitmap) and
//                 stores the flipped spin; two lcg32 draws per site; bond activation against the integer
//                 threshold on 64-bit ballot masks (scalar unit); row runs from the masks, unions in an LDS
//                 union-find (atomicMin keeps parent <= child, so roots are cluster minima); block-local
//                 uint16 labels with an edge flag; the block-edge bond bits and the block's halo spins.
//   k_merge       per block: unions across block edges by 64-bit atomicMin in a union-find in HBM over the slots
//                 of the edge-reaching clusters (two waves per block; k_merge_block with one for large launches).
//   k_resolve     per block (two waves): the block's slots are chased in that union-find, their flip bits written
//                 out and the block's halo spins flipped in place. Advances the lcg32 iteration count; the spin
//                 array waits for the next k_bond_label.
// k_join does the work of k_merge and k_resolve for lattices of few blocks, and k_resident (swmi_resident.hip) sweeps
// small lattices whole, without any of these launches. k_flip applies a pending flip to the spin array; it runs only
// before the array itself is read (downloads, checkpoints, inspection). k_observables takes a sample without storing the flip.
// Spin bytes: bit 0 is the spin, bits 3-5 hold the site's current lcg32 parameter selector, i.e. the
// index k of the Numerical Recipes pair (a_k, c_k) that lane i of its group uses after the group's
// rotations (sel0[(i + rot) & 63]). The byte is read every sweep anyway, so the generator needs no other
// per-group data except on the sweeps that rotate (one in 7.5); only those store lcg32 states.
// Reference behaviour: ising/src/swendsen_wang_amd_gpu.cpp:78-467 (four kernels per sweep) and the CPU
// labeller ising/src/swendsen_wang_cpu.cpp:13-205; the kernels here are written for wave64 CDNA4.
#include "swmi_device.h"

namespace swmi
{
    // =============================================================================================
    // k_merge: unions across block edges (reference MergeLabels_Kernel, swendsen_wang_amd_gpu.cpp:280-329)
    // =============================================================================================
    // One two-wave workgroup per block: wavefront 0 takes the right edge (one lane per lattice row),
    // wavefront 1 the down edge (one lane per column). Two waves per block keep every block of a 4096^2
    // lattice resident at once, so the latency-bound union chains of all blocks overlap.
    // Bit `lane` of `bits`: a bond from a site of this block to a site of block lb_b (first site base_b), whose
    // edge entries (ecol / erow: (label << 16) | root index q) are va and vb. Both sites belong to clusters
    // that reach their block's edge, so their labels name slots.
    // Per wave, the distinct slots of one edge's root pairs in LDS: S[p] = lattice-wide slot + 1 of local node p
    // (0: free), K[p] its key; L[p] = (key of its parent << 32) | local parent (a root holds its own key and
    // position). Inserted by open addressing over 128 positions (at most 128 slots: every insert ends).
    __device__ __forceinline__ uint32_t LocalNode(uint32_t* S, uint32_t* K, uint64_t* L, const uint32_t c, const uint32_t k, const bool want)
    {
        uint32_t p = Fmix32(c * 0x85EBCA6Bu) & 127u;
        bool open = want;
        while (__ballot(open))
        {
            if (open)
            {
                uint32_t found = 0u;
                if (__hip_atomic_compare_exchange_strong(&S[p], &found, c + 1u, __ATOMIC_RELAXED, __ATOMIC_RELAXED,
                                                         __HIP_MEMORY_SCOPE_WORKGROUP))
                {
                    K[p] = k;
                    __hip_atomic_store(&L[p], SlotEntry(k, p), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
                    open = false;
                }
                else if (found == c + 1u)
                    open = false;
                else
                    p = (p + 1u) & 127u;
            }
        }
        return p;
    }

    __device__ __forceinline__ uint64_t LocalEntry(uint64_t* L, const uint32_t p)
    {
        return __hip_atomic_load(&L[p], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    }

    template <bool FRESH, bool LOCAL>
    __device__ __forceinline__ void MergeEdge(const LatDesc& d, const Block& bl, const uint64_t bits, const uint32_t va,
                                              const uint32_t vb, const uint32_t lb_b, const uint32_t base_b, gptr<uint32_t> err,
                                              uint64_t* H, uint32_t* S, uint32_t* K, uint32_t* W)
    {
        const uint32_t lane = threadIdx.x & 63u;
        const bool bit = LaneBit(bits);
        const uint32_t slots = kWavesPerBlock * d.edge_cap;
        uint32_t ka = 0, kb = 0, ca = 0, cb = 0;
        if (bit)
        {
            const uint32_t la = va >> 16, lb = vb >> 16;
            const uint32_t sa = (la & 0x7FFFu) - d.qcap, sb = (lb & 0x7FFFu) - d.qcap;
            if (!(la & kEdgeFlag) || !(lb & kEdgeFlag) || sa >= slots || sb >= slots)
                (void)__hip_atomic_fetch_or(err, kErrLabelRange, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            ka = SiteOf(bl.base, bl.stride, va & 0xFFFFu);
            kb = SiteOf(base_b, bl.stride, vb & 0xFFFFu);
            ca = bl.lb * slots + min(sa, slots - 1u);
            cb = lb_b * slots + min(sb, slots - 1u);
        }
        // Without local unions, one lattice-wide union per distinct pair of roots (below T_c most bonds of an edge
        // join the same two clusters): the lanes insert their pairs into the wave's LDS hash set H (128 slots for
        // at most 64 pairs, linear probing, so every insert ends), and the lane whose insert lands leads the union
        // for its pair. With them, every bonded lane takes part in the local unions below, where a repeated pair
        // costs nothing.
        const uint32_t lo = min(ka, kb), hi = max(ka, kb);
        const bool want = bit && ka != kb;
        bool leader = LOCAL && want;
        if (!LOCAL && __ballot(want))
        {
            H[lane] = 0ull;
            H[64u + lane] = 0ull;
            const uint64_t key = (static_cast<uint64_t>(hi) << 32) | lo;   // hi > lo: never 0 (the empty slot)
            uint32_t slot = Fmix32(lo ^ (hi * 0x9E3779B9u)) & 127u;
            bool open = want;
            while (__ballot(open))
            {
                if (open)
                {
                    uint64_t found = 0ull;
                    if (__hip_atomic_compare_exchange_strong(&H[slot], &found, key, __ATOMIC_RELAXED, __ATOMIC_RELAXED,
                                                             __HIP_MEMORY_SCOPE_WORKGROUP))
                    {
                        leader = true;
                        open = false;
                    }
                    else if (found == key)
                        open = false;
                    else
                        slot = (slot + 1u) & 127u;
                }
            }
        }
        if constexpr (!LOCAL)
        {
            if (leader)
                SlotUnion<FRESH>(Glob(d.cpar), ca, ka, cb, kb, d.n_blocks * slots, err);
            return;
        }
        if (!__ballot(leader))
            return;
        // The pairs of one edge often share a slot (a cluster of one block meets several of its neighbour's), and
        // lanes that link the same root race on one entry of the slot union-find. So the pairs are first united in
        // LDS, over their distinct slots (H holds the local entries here), and each slot that is not its local
        // component's root is then linked under that root: one lattice-wide union per lane, no two on one slot.
        S[lane] = 0u;
        S[64u + lane] = 0u;
        uint32_t a = LocalNode(S, K, H, ca, ka, leader);
        uint32_t b = LocalNode(S, K, H, cb, kb, leader);
        bool open = leader;
        while (__ballot(open))
        {
            if (open)
            {
                uint64_t ea = LocalEntry(H, a), eb = LocalEntry(H, b);
                while (static_cast<uint32_t>(ea) != a)
                {
                    a = static_cast<uint32_t>(ea) & 127u;
                    ea = LocalEntry(H, a);
                }
                while (static_cast<uint32_t>(eb) != b)
                {
                    b = static_cast<uint32_t>(eb) & 127u;
                    eb = LocalEntry(H, b);
                }
                if (a == b)
                    open = false;
                else
                {
                    if ((ea >> 32) > (eb >> 32))   // roots hold their own keys; link the larger under the smaller
                    {
                        const uint32_t t = a;
                        a = b;
                        b = t;
                        const uint64_t te = ea;
                        ea = eb;
                        eb = te;
                    }
                    const uint64_t old = __hip_atomic_fetch_min(&H[b], SlotEntry(static_cast<uint32_t>(ea >> 32), a),
                                                                __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
                    if (old == eb)
                        open = false;
                    else   // b had been linked under old's parent (which this link may have displaced): unite with it
                        b = static_cast<uint32_t>(old) & 127u;
                }
            }
        }
        // the local nodes that are not their component's root, listed one per lane
        uint32_t item[2], root[2];
        bool has[2];
#pragma unroll
        for (uint32_t h = 0; h < 2u; ++h)
        {
            const uint32_t p = lane + 64u * h;
            uint32_t r = p;
            has[h] = false;
            if (S[p] != 0u)
            {
                uint64_t e = LocalEntry(H, r);
                while (static_cast<uint32_t>(e) != r)
                {
                    r = static_cast<uint32_t>(e) & 127u;
                    e = LocalEntry(H, r);
                }
                has[h] = r != p;
            }
            item[h] = p;
            root[h] = r;
        }
        const uint64_t f0 = __ballot(has[0]), f1 = __ballot(has[1]);
        const uint32_t n0 = static_cast<uint32_t>(__popcll(f0)), n = n0 + static_cast<uint32_t>(__popcll(f1));
        const uint32_t i0 = __builtin_amdgcn_mbcnt_hi(static_cast<uint32_t>(f0 >> 32), __builtin_amdgcn_mbcnt_lo(static_cast<uint32_t>(f0), 0u));
        const uint32_t i1 = n0 + __builtin_amdgcn_mbcnt_hi(static_cast<uint32_t>(f1 >> 32), __builtin_amdgcn_mbcnt_lo(static_cast<uint32_t>(f1), 0u));
        // at most one per local link, so at most one per pair: n <= 64
        if (has[0] && i0 < 64u)
            W[i0] = (root[0] << 8) | item[0];
        if (has[1] && i1 < 64u)
            W[i1] = (root[1] << 8) | item[1];
        if (lane < n && lane < 64u)
        {
            const uint32_t w = W[lane], p = w & 0xFFu, r = w >> 8;
            SlotUnion<FRESH>(Glob(d.cpar), S[p] - 1u, K[p], S[r] - 1u, K[r], d.n_blocks * slots, err);
        }
        if (n > 64u && lane == 0u)
            (void)__hip_atomic_fetch_or(err, kErrLabelRange, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }

    template <bool FRESH, bool LOCAL>
    __device__ __forceinline__ void MergeEdges(const LatDesc& d, const uint32_t b)
    {
        // the lattice's active flag is loaded with the edge data (an inactive lattice links nothing)
        const gptr<const uint32_t> active = Glob(static_cast<const uint32_t*>(d.state)) + kStActive;
        const Block bl = DecodeBlock(d, b);
        const gptr<uint64_t> bb = Glob(d.bbits) + kBbitWords * bl.lb;
        const uint32_t lane = threadIdx.x & 63u;
        const uint32_t w = Uniform(threadIdx.x >> 6);
        const uint32_t tw = d.tw, rpw = d.rpw, twr = d.twr;
        const gptr<uint32_t> err = Glob(d.state) + kStErr;
        __shared__ uint64_t HS[2][128];   // per wave: the hash set of root pairs (small launches) or the local entries
        __shared__ uint32_t SS[2][128], SK[2][128], SW[2][64];   // per wave: local slots, their keys, the union list

        if (w == 0)
        {
            // right edge: the block's lattice rows, 64 per pass (lane = row); bit r of word 1 + t is row
            // t * twr * rpw + r; entries from the compact edge columns, loaded with the bond words
            const uint32_t rows = bl.nwr * rpw, per_tile = twr * rpw;
            const uint32_t sx_r = (bl.sx + 1u == d.tiles_x) ? 0u : bl.sx + 1u;
            const uint32_t lb_r = bl.sy * d.tiles_x + sx_r;
            const uint32_t base_r = BlockBase(d, sx_r, bl.sy);
            const gptr<const uint32_t> ec = Glob(static_cast<const uint32_t*>(d.ecol));
            const gptr<const uint32_t> ea = ec + (2u * bl.lb + 1u) * d.ecol_stride;
            const gptr<const uint32_t> eb = ec + (2u * lb_r) * d.ecol_stride;
            const uint64_t r0 = bb[1], r1 = bb[2], r2 = bb[3], r3 = bb[4];
            for (uint32_t p0 = 0; p0 < rows; p0 += 64u)
            {
                const uint32_t row = min(p0 + lane, rows - 1u);
                const uint32_t va = ea[row], vb = eb[row];
                const uint32_t act = *active;
                Issued(r0);
                Issued(r1);
                Issued(r2);
                Issued(r3);
                Issued(va);
                Issued(vb);
                const uint32_t t = row / per_tile, r = row - t * per_tile;
                const uint64_t word = t == 0u ? r0 : (t == 1u ? r1 : (t == 2u ? r2 : r3));
                const uint64_t bits = __ballot(p0 + lane < rows && ((word >> r) & 1ull) != 0ull);
                if (bits && act != 0u)
                    MergeEdge<FRESH, LOCAL>(d, bl, bits, va, vb, lb_r, base_r, err, HS[0], SS[0], SK[0], SW[0]);
            }
        }
        else
        {
            // down edge: the lanes of the block's last lattice row (the last lattice row of its last wave row)
            // against the first lattice row of the block below (lanes 0 .. tw - 1 of its first wave row)
            const uint32_t sy_b = bl.sy + 1u == d.blocks_y ? 0u : bl.sy + 1u;
            const uint32_t lb_b = sy_b * d.tiles_x + bl.sx;
            const gptr<const uint32_t> er = Glob(static_cast<const uint32_t*>(d.erow));
            const uint32_t va = er[2u * 64u * bl.lb + 64u + lane], vb = er[2u * 64u * lb_b + (lane & (tw - 1u))];
            const uint64_t down_bits = bb[0];
            const uint32_t act = *active;
            Issued(va);
            Issued(vb);
            if (down_bits && act != 0u)
                MergeEdge<FRESH, LOCAL>(d, bl, down_bits, va, vb, lb_b, BlockBase(d, bl.sx, sy_b), err, HS[1], SS[1], SK[1], SW[1]);
        }
    }

    template <bool FRESH, bool LOCAL>
    __global__ __launch_bounds__(128) void k_merge(const LatDesc* __restrict__ descs, const uint32_t* __restrict__ block_lat,
                                                   const uint32_t total_blocks)
    {
        const uint32_t b = RemapBlock(total_blocks);
        if (b < total_blocks)
            MergeEdges<FRESH, LOCAL>(descs[LatticeOf(block_lat, b)], b);
    }

    // of one lattice whose descriptor comes with the launch
    template <bool FRESH>
    __global__ __launch_bounds__(128) void k_merge_one(const LatDesc d, const uint32_t total_blocks)
    {
        const uint32_t b = RemapBlock(total_blocks);
        if (b < total_blocks)
            MergeEdges<FRESH, false>(d, b);
    }

    // k_merge for 64-wide tiles and blocks of at most 64 rows (at most 252 boundary sites, so 252 slots): one wave per
    // block takes both of its edges. The bonded pairs are first united in LDS, in a table indexed by slot (256 entries
    // each for the block, its right and its lower neighbour: no hashing), so that pairs that share a cluster, also
    // across the two edges, cost one lattice-wide union per non-root slot and no two lanes race on one slot; a slot
    // that several lanes hold is claimed by the last of them to write its mark.
    template <bool FRESH>
    __global__ __launch_bounds__(64) void k_merge_block(const LatDesc* __restrict__ descs, const uint32_t* __restrict__ block_lat,
                                                        const uint32_t total_blocks)
    {
        constexpr uint32_t kN = 256u;
        __shared__ uint64_t L[3u * kN];   // (key of the parent << 32) | parent; later the list of unions
        const uint32_t b = RemapBlock(total_blocks);
        if (b >= total_blocks)
            return;
        const LatDesc& d = descs[LatticeOf(block_lat, b)];
        const gptr<const uint32_t> active = Glob(static_cast<const uint32_t*>(d.state)) + kStActive;
        const Block bl = DecodeBlock(d, b);
        const uint32_t lane = threadIdx.x;
        const gptr<const uint64_t> bb = Glob(static_cast<const uint64_t*>(d.bbits)) + kBbitWords * bl.lb;
        const gptr<const uint32_t> ec = Glob(static_cast<const uint32_t*>(d.ecol)), er = Glob(static_cast<const uint32_t*>(d.erow));
        const gptr<uint32_t> err = Glob(d.state) + kStErr;
        const uint32_t es = d.ecol_stride, twr = d.twr, qcap = d.qcap, slots = kWavesPerBlock * d.edge_cap;
        const uint32_t sx_r = (bl.sx + 1u == d.tiles_x) ? 0u : bl.sx + 1u, sy_b = bl.sy + 1u == d.blocks_y ? 0u : bl.sy + 1u;
        const uint32_t lb_r = bl.sy * d.tiles_x + sx_r, lb_b = sy_b * d.tiles_x + bl.sx;
        const uint32_t row = min(lane, bl.nwr - 1u);
        // pair 0: the right edge at lattice row `lane`; pair 1: the down edge at column `lane`
        uint32_t va[2], vb[2];
        va[0] = ec[(2u * bl.lb + 1u) * es + row];
        vb[0] = ec[2u * lb_r * es + row];
        va[1] = er[2u * 64u * bl.lb + 64u + lane];
        vb[1] = er[2u * 64u * lb_b + lane];
        const uint64_t right = bb[1u + row / twr], down = bb[0];
        const uint32_t act = *active;
        Issued(va[0]);
        Issued(vb[0]);
        Issued(va[1]);
        Issued(vb[1]);
        Issued(right);
        Issued(down);
        bool bit[2] = {lane < bl.nwr && ((right >> (row % twr)) & 1ull) != 0ull, ((down >> lane) & 1ull) != 0ull};
        if (act == 0u || !__ballot(bit[0] || bit[1]))
            return;

        uint32_t n[4], k[4];   // nodes and keys: a and b of pair 0, a and b of pair 1
#pragma unroll
        for (uint32_t p = 0; p < 2u; ++p)
        {
            const uint32_t region = (1u + p) * kN, base = BlockBase(d, p ? bl.sx : sx_r, p ? sy_b : bl.sy);
            const uint32_t sa = ((va[p] >> 16) & 0x7FFFu) - qcap, sb = ((vb[p] >> 16) & 0x7FFFu) - qcap;
            // both ends of a bond across an edge belong to edge-reaching clusters
            const bool good = ((va[p] >> 16) & (vb[p] >> 16) & kEdgeFlag) && sa < min(slots, kN) && sb < min(slots, kN);
            if (bit[p] && !good)
            {
                (void)__hip_atomic_fetch_or(err, kErrLabelRange, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                bit[p] = false;
            }
            n[2u * p] = bit[p] ? sa : 0u;
            n[2u * p + 1u] = bit[p] ? region + sb : 0u;
            k[2u * p] = SiteOf(bl.base, bl.stride, va[p] & 0xFFFFu);
            k[2u * p + 1u] = SiteOf(base, bl.stride, vb[p] & 0xFFFFu);
            if (bit[p])
            {
                __hip_atomic_store(&L[n[2u * p]], SlotEntry(k[2u * p], n[2u * p]), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
                __hip_atomic_store(&L[n[2u * p + 1u]], SlotEntry(k[2u * p + 1u], n[2u * p + 1u]), __ATOMIC_RELAXED,
                                   __HIP_MEMORY_SCOPE_WORKGROUP);
            }
        }
#pragma unroll
        for (uint32_t p = 0; p < 2u; ++p)
        {
            uint32_t x = n[2u * p], y = n[2u * p + 1u];
            bool open = bit[p];
            while (__ballot(open))
            {
                if (open)
                {
                    uint64_t ex = LocalEntry(L, x), ey = LocalEntry(L, y);
                    while (static_cast<uint32_t>(ex) != x || static_cast<uint32_t>(ey) != y)
                    {
                        x = static_cast<uint32_t>(ex);
                        y = static_cast<uint32_t>(ey);
                        ex = LocalEntry(L, x);
                        ey = LocalEntry(L, y);
                    }
                    if (x == y)
                        open = false;
                    else
                    {
                        // roots hold their own entries; link the larger under the smaller (a lattice one block wide or
                        // high has the same slot in two of the table's parts: equal keys, ordered by node)
                        if (ex > ey)
                        {
                            const uint32_t t = x;
                            x = y;
                            y = t;
                            const uint64_t te = ex;
                            ex = ey;
                            ey = te;
                        }
                        const uint64_t old = __hip_atomic_fetch_min(&L[y], ex, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
                        if (old == ey)
                            open = false;
                        else   // y had been linked under old's parent (which this link may have displaced): unite with it
                            y = static_cast<uint32_t>(old);
                    }
                }
            }
        }
        // the roots of the lane's nodes, chased together (a lane without a pair sits on no node: done at once)
        uint64_t e[4];
        uint32_t r[4];
#pragma unroll
        for (uint32_t i = 0; i < 4u; ++i)
        {
            r[i] = n[i];
            e[i] = bit[i >> 1] ? LocalEntry(L, n[i]) : static_cast<uint64_t>(n[i]);
        }
        for (;;)
        {
            bool moved = false;
#pragma unroll
            for (uint32_t i = 0; i < 4u; ++i)
                if (static_cast<uint32_t>(e[i]) != r[i])
                {
                    r[i] = static_cast<uint32_t>(e[i]);
                    e[i] = LocalEntry(L, r[i]);
                    moved = true;
                }
            if (!__ballot(moved))
                break;
        }
        // one lane claims each node that is not its component's root
        bool has[4];
#pragma unroll
        for (uint32_t i = 0; i < 4u; ++i)
            if (r[i] != n[i])
                __hip_atomic_store(&L[n[i]], static_cast<uint64_t>(lane * 4u + i), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
#pragma unroll
        for (uint32_t i = 0; i < 4u; ++i)
            has[i] = r[i] != n[i] && LocalEntry(L, n[i]) == static_cast<uint64_t>(lane * 4u + i);
        const auto slot_of = [&](const uint32_t node) {
            return (node < kN ? bl.lb : (node < 2u * kN ? lb_r : lb_b)) * slots + (node & (kN - 1u));
        };
        // the unions, listed one per lane: two words (slot, key) each for the node and its root. At most one per link
        // made above, so at most 128.
        uint32_t total = 0;
#pragma unroll
        for (uint32_t i = 0; i < 4u; ++i)
        {
            const uint64_t f = __ballot(has[i]);
            const uint32_t at = total + __builtin_amdgcn_mbcnt_hi(static_cast<uint32_t>(f >> 32), __builtin_amdgcn_mbcnt_lo(static_cast<uint32_t>(f), 0u));
            if (has[i] && at < 128u)
            {
                __hip_atomic_store(&L[2u * at], SlotEntry(k[i], slot_of(n[i])), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
                __hip_atomic_store(&L[2u * at + 1u], SlotEntry(static_cast<uint32_t>(e[i] >> 32), slot_of(r[i])), __ATOMIC_RELAXED,
                                   __HIP_MEMORY_SCOPE_WORKGROUP);
            }
            total += static_cast<uint32_t>(__popcll(f));
        }
        for (uint32_t i = lane; i < min(total, 128u); i += 64u)
        {
            const uint64_t x = LocalEntry(L, 2u * i), y = LocalEntry(L, 2u * i + 1u);
            SlotUnion<FRESH>(Glob(d.cpar), static_cast<uint32_t>(x), static_cast<uint32_t>(x >> 32), static_cast<uint32_t>(y),
                             static_cast<uint32_t>(y >> 32), d.n_blocks * slots, err);
        }
        if (total > 128u && lane == 0u)
            (void)__hip_atomic_fetch_or(err, kErrLabelRange, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }

    // =============================================================================================
    // k_resolve / k_flip: resolve + flip (reference ResolveLabels_Kernel / FlipClusters_Kernel,
    // swendsen_wang_amd_gpu.cpp:403-467), split into the decision (k_resolve, end of every sweep) and its
    // application to the spin array (the next sweep's k_bond_label, or k_flip before the array itself is read)
    // =============================================================================================
    // Bitmap index of a label: the root index, or qcap + slot for an edge-reaching cluster. An index outside
    // the block's range (a broken invariant) clears ok and reads bit 0.
    __device__ __forceinline__ uint32_t LabelBit(const uint32_t lab, const uint32_t qmax, const uint32_t qcap, const uint32_t slots,
                                                 bool& ok)
    {
        const uint32_t i = lab & 0x7FFFu;
        const bool good = (lab & kEdgeFlag) ? (i >= qcap && i < qcap + slots) : (i < qmax);
        if (!good)
            ok = false;
        return good ? i : 0u;
    }

    // flip bit of a site with label lab from the block's bitmap
    __device__ __forceinline__ uint32_t FlipOfLabel(const uint32_t lab, const uint32_t* fb, const uint32_t qmax, const uint32_t qcap,
                                                    const uint32_t slots, bool& ok)
    {
        const uint32_t i = LabelBit(lab, qmax, qcap, slots, ok);
        return (fb[i >> 5] >> (i & 31u)) & 1u;
    }

    // The block's edge-root slots (the dense prefix k_bond_label filled), for i in [first, total) step
    // `stride`: f(slot within the block, lattice-wide slot).
    template <typename F>
    __device__ __forceinline__ void ForBlockSlots(const LatDesc& d, const Block& bl, const uint32_t first, const uint32_t stride, F&& f)
    {
        const uint32_t slots = kWavesPerBlock * d.edge_cap;
        const uint32_t total = min(Glob(d.edge_count)[kWavesPerBlock * bl.lb], slots);
        for (uint32_t i = first; i < total; i += stride)
            f(i, slots * bl.lb + i);
    }

    // The lattice's counters at the end of the sweep that began at iteration `it`.
    __device__ __forceinline__ void AdvanceIteration(const LatDesc& d, const uint32_t it)
    {
        const gptr<uint32_t> stp = Glob(d.state);
        stp[kStApplied] = it;
        stp[kStIteration] = it + 2u;
        // a rotating sweep stored the states at which its lanes' pairs changed (last)
        if ((it + 2u) % 15u == 0u)
            Glob(d.aux)[kAuxRngIt] = it + 1u;
        else if ((it + 1u) % 15u == 0u)
            Glob(d.aux)[kAuxRngIt] = it;
    }

    // End of a sweep, per block (two waves): the slots of the block's edge-reaching clusters are chased in the
    // slot union-find, and each slot's bit becomes the flip rule applied to its canonical root; then the
    // block's flip bitmap and the flipped spins of its first column and first wave row (the halos its left
    // and upper neighbours read in the next sweep) are written out, and the lattice's counters move on:
    // applied = the iteration whose spins the array holds, iteration += 2. The spin array itself is left for
    // the next sweep to flip.
    // kMaxRows: lattice rows of the tallest block.
    template <uint32_t kMaxRows>
    __global__ __launch_bounds__(128) void k_resolve(const LatDesc* __restrict__ descs, const uint32_t* __restrict__ block_lat,
                                                     const uint32_t total_blocks)
    {
        constexpr uint32_t kThreads = 128;
        constexpr uint32_t kMaxSites = kWavesPerBlock * 64u * 64u;
        __shared__ uint32_t sw[kMaxSites / 32u];   // flip bits of the block's slots (at most one slot per site)
        const uint32_t b = RemapBlock(total_blocks);
        if (b >= total_blocks)
            return;
        const LatDesc& d = descs[LatticeOf(block_lat, b)];
        const gptr<uint32_t> stp = Glob(d.state);
        const Block bl = DecodeBlock(d, b);
        const uint32_t qmax = bl.nwr * 64u, qcap = d.qcap, slots = kWavesPerBlock * d.edge_cap;
        const gptr<const uint32_t> erow0 = Glob(static_cast<const uint32_t*>(d.erow)) + 2u * 64u * bl.lb;
        const gptr<const uint32_t> ecol0 = Glob(static_cast<const uint32_t*>(d.ecol)) + 2u * bl.lb * d.ecol_stride;
        bool ok = true;

        // halo sites: entry t < rows is the first column at lattice row t of the block, entry rows + j the
        // first wave row at lane j. Their labels and the block's slot count need only the descriptor and are
        // loaded with the lattice's counters; their spins (written into the halo by this sweep's
        // k_bond_label) follow with the first entries of the slot chases. The halo is flipped in place.
        const uint32_t rows = bl.nwr * d.rpw;
        constexpr uint32_t kHaloPer = (kMaxRows + 64u + kThreads - 1u) / kThreads;
        // (straight-line loads from a selected address, every one in range, so that they are all in flight
        // at once; hoff is the entry's offset in the halo)
        uint32_t hs[kHaloPer], hl[kHaloPer], hoff[kHaloPer];
#pragma unroll
        for (uint32_t k = 0; k < kHaloPer; ++k)
        {
            const uint32_t t = threadIdx.x + k * kThreads;
            const bool col = t < rows;
            const uint32_t j = min(t - rows, 63u);
            hoff[k] = col ? t : d.ecol_stride + j;
            hl[k] = *(col ? ecol0 + t : erow0 + j) >> 16;
        }
        const uint32_t nslot = min(Glob(d.edge_count)[kWavesPerBlock * bl.lb], slots);
        const uint32_t active = stp[kStActive], hside = stp[kStHaloSide], fkey = stp[kStFlipKey];
#pragma unroll
        for (uint32_t k = 0; k < kHaloPer; ++k)
            Issued(hl[k]);
        Issued(nslot);
        Issued(hside);
        Issued(fkey);
        if (active == 0u)
            return;
        const bool random_rule = d.flip_rule != 0u;
        const uint32_t key = random_rule ? fkey : 0u;
        const gptr<uint8_t> halo = Glob(d.halo) + (hside * d.n_blocks + bl.lb) * d.halo_stride;
        const gptr<uint64_t> E = Glob(d.cpar);
        const uint32_t c_max = d.n_blocks * slots, c0 = slots * bl.lb;
        const uint64_t e_first = threadIdx.x < nslot ? CachedLoad64(&E[c0 + threadIdx.x]) : 0ull;
#pragma unroll
        for (uint32_t k = 0; k < kHaloPer; ++k)
            hs[k] = halo[hoff[k]];
        // each slot's canonical root, one slot per lane; a wave assembles the flip bits of 64 slots per pass
        // with a ballot and writes them as whole words, into LDS for the halo flips and into the block's fbits
        // (words past the last slot are left as they were: no label names a slot past the count)
        const gptr<uint32_t> fbits_g = Glob(d.fbits) + bl.lb * d.fsw;
        const uint32_t lane = threadIdx.x & 63u, w = threadIdx.x >> 6;
        for (uint32_t s0 = 0; s0 < nslot; s0 += kThreads)
        {
            const uint32_t i = s0 + threadIdx.x;
            uint32_t bit = 0;
            if (i < nslot)
                bit = FlipBit(d, SlotRootKey(E, c0 + i, i == threadIdx.x ? e_first : CachedLoad64(&E[c0 + i]), c_max, ok),
                              random_rule, key);
            const uint64_t m = __ballot(bit != 0u);
            const uint32_t wd = (s0 + w * 64u) >> 5;
            if (lane == 0u && wd < d.fsw)
            {
                sw[wd] = static_cast<uint32_t>(m);
                fbits_g[wd] = static_cast<uint32_t>(m);
            }
            if (lane == 32u && wd + 1u < d.fsw)
            {
                sw[wd + 1u] = static_cast<uint32_t>(m >> 32);
                fbits_g[wd + 1u] = static_cast<uint32_t>(m >> 32);
            }
        }
        __syncthreads();

        // the flip of a halo site: its slot's bit, or for a cluster inside the block (a padding lane of the
        // first wave row) the rule at its root; a label out of range clears ok
        const auto halo_flip = [&](const uint32_t lab) -> uint32_t {
            const uint32_t i = lab & 0x7FFFu;
            if (lab & kEdgeFlag)
            {
                if (i < qcap || i - qcap >= nslot)
                {
                    ok = false;
                    return 0u;
                }
                return (sw[(i - qcap) >> 5] >> ((i - qcap) & 31u)) & 1u;
            }
            if (i >= qmax)
            {
                ok = false;
                return 0u;
            }
            return FlipBit(d, SiteOf(bl.base, bl.stride, i), random_rule, key);
        };
#pragma unroll
        for (uint32_t k = 0; k < kHaloPer; ++k)
        {
            const uint32_t t = threadIdx.x + k * kThreads;
            if (t < rows + 64u)
                halo[hoff[k]] = static_cast<uint8_t>((hs[k] ^ halo_flip(hl[k])) & 1u);
        }
        if (!ok)
            (void)__hip_atomic_fetch_or(stp + kStErr, kErrLabelRange, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if (bl.lb == 0 && threadIdx.x == 0)
            AdvanceIteration(d, stp[kStIteration]);
    }

    // =============================================================================================
    // k_join: k_merge and k_resolve of a lattice of few blocks, in one workgroup
    // =============================================================================================
    // For a lattice of few blocks the two kernels are launch time and chains of memory round trips. Here one workgroup of
    // 16 waves holds the whole lattice's slot union-find in LDS: node 256 * block + slot (a block
    // of 64 columns and at most 64 rows has at most 252 boundary sites, so at most 252 slots). The edges, the halo
    // labels and the counters are read in one round trip; the unions are LDS operations; the flip bits, the flipped
    // halos and every slot's root go out as k_resolve and k_merge leave them (the root directly as parent).
    // A wave takes two edges and one block, so at most 16 blocks: one CU reads about 8 KB per microsecond from the other
    // CUs' results, which bounds it (microseconds per sweep at T_c with k_merge and k_resolve / with k_join: 6 blocks
    // 17.5 / 13.9, 16 blocks 18.8 / 16.2, and with more edges per wave 24 blocks 19.3 / 20.0, 64 blocks 20.1 / 32.1).
    __global__ __launch_bounds__(1024) void k_join(const LatDesc* __restrict__ descs, const uint32_t* __restrict__ slots)
    {
        constexpr uint32_t kWaves = 16, kEdges = 2u, kNodes = 256u;
        extern __shared__ uint64_t L[];            // kNodes entries per block: (key of the parent << 32) | parent
        __shared__ uint32_t sw[kWaves * 8u];       // flip bits by node
        const LatDesc& d = descs[LatticeOf(slots, blockIdx.x)];
        const gptr<uint32_t> stp = Glob(d.state);
        const uint32_t lane = threadIdx.x & 63u, w = Uniform(threadIdx.x >> 6);
        const uint32_t tx = d.tiles_x, nb = d.n_blocks, brows = kWavesPerBlock * d.twr, stride = 64u * tx, qcap = d.qcap;
        const uint32_t bslots = kWavesPerBlock * d.edge_cap, es = d.ecol_stride;
        const gptr<const uint32_t> ec = Glob(static_cast<const uint32_t*>(d.ecol)), er = Glob(static_cast<const uint32_t*>(d.erow));
        const gptr<const uint64_t> bb = Glob(static_cast<const uint64_t*>(d.bbits));
        const gptr<const uint32_t> counts = Glob(static_cast<const uint32_t*>(d.edge_count));
        bool ok = true;
        const auto rows_of = [&](const uint32_t sy) { return min(brows, d.nwr_y - sy * brows); };

        // edge e = w + 16 k: block e / 2, its right edge (lane = row) or its down edge (lane = column)
        uint32_t va[kEdges], vb[kEdges], lbb[kEdges], base_a[kEdges], base_b[kEdges];   // base: first site of the block
        uint64_t word[kEdges];
#pragma unroll
        for (uint32_t k = 0; k < kEdges; ++k)
        {
            const uint32_t e = min(w + kWaves * k, 2u * nb - 1u), lb = e >> 1;
            const uint32_t sx = lb % tx, sy = lb / tx;
            const bool down = (e & 1u) != 0u;
            const uint32_t sx_b = down ? sx : (sx + 1u == tx ? 0u : sx + 1u), sy_b = !down ? sy : (sy + 1u == d.blocks_y ? 0u : sy + 1u);
            lbb[k] = sy_b * tx + sx_b;
            base_a[k] = sy * brows * stride + sx * 64u;
            base_b[k] = sy_b * brows * stride + sx_b * 64u;
            const uint32_t row = min(lane, rows_of(sy) - 1u);
            va[k] = *(down ? er + 128u * lb + 64u + lane : ec + (2u * lb + 1u) * es + row);
            vb[k] = *(down ? er + 128u * lbb[k] + lane : ec + 2u * lbb[k] * es + row);
            word[k] = bb[kBbitWords * lb + (down ? 0u : 1u + row / d.twr)];
        }
        // block w: its slots and its halo (first column, first row)
        const uint32_t blk = min(w, nb - 1u), blk_rows = rows_of(blk / tx);
        const uint32_t cnt = counts[kWavesPerBlock * blk];
        const uint32_t hc = ec[2u * blk * es + min(lane, blk_rows - 1u)] >> 16, hr = er[128u * blk + lane] >> 16;
        const uint32_t active = stp[kStActive], hside = stp[kStHaloSide], fkey = stp[kStFlipKey], it = stp[kStIteration];
        if (active == 0u)
            return;
        const gptr<uint8_t> halo = Glob(d.halo) + (hside * nb + blk) * d.halo_stride;
        const uint32_t sc = halo[min(lane, blk_rows - 1u)], sr = halo[es + lane];

        // every slot's node, a root keyed by its site (the edge entries of a block name all of its slots)
        const uint32_t max_slots = min(bslots, kNodes);
        const auto slot_of = [&](const uint32_t v) { return (v >> 16) - (kEdgeFlag + qcap); };   // of no slot: past them all
        const auto node_of = [&](const uint32_t lb, const uint32_t v) { return lb * kNodes + slot_of(v); };
        const auto put = [&](const uint32_t lb, const uint32_t base, const uint32_t v) {
            if (slot_of(v) < max_slots)
            {
                const uint32_t n = node_of(lb, v);
                __hip_atomic_store(&L[n], SlotEntry(SiteOf(base, stride, v & 0xFFFFu), n), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
            }
        };
#pragma unroll
        for (uint32_t k = 0; k < kEdges; ++k)
            if (w + kWaves * k < 2u * nb)
            {
                put((w + kWaves * k) >> 1, base_a[k], va[k]);
                put(lbb[k], base_b[k], vb[k]);
            }
        __syncthreads();

        // unions of the bonded pairs, one lane each (the loop of k_merge's local unions)
#pragma unroll
        for (uint32_t k = 0; k < kEdges; ++k)
        {
            const uint32_t e = w + kWaves * k;
            if (e < 2u * nb)
            {
                const uint32_t lb = e >> 1;
                const bool down = (e & 1u) != 0u;
                const uint32_t bit = down ? lane : lane % d.twr;
                bool open = ((word[k] >> bit) & 1ull) != 0ull && (down || lane < rows_of(lb / tx));
                // both ends of a bond across an edge belong to edge-reaching clusters
                if (open && max(slot_of(va[k]), slot_of(vb[k])) >= max_slots)
                {
                    ok = false;
                    open = false;
                }
                // (a lane that takes part follows only nodes written above, whose parents are such nodes)
                uint32_t a = node_of(lb, va[k]), b = node_of(lbb[k], vb[k]);
                while (__ballot(open))
                {
                    if (open)
                    {
                        uint64_t ea = LocalEntry(L, a), eb = LocalEntry(L, b);
                        while (static_cast<uint32_t>(ea) != a || static_cast<uint32_t>(eb) != b)
                        {
                            a = static_cast<uint32_t>(ea);
                            b = static_cast<uint32_t>(eb);
                            ea = LocalEntry(L, a);
                            eb = LocalEntry(L, b);
                        }
                        if (a == b)
                            open = false;
                        else
                        {
                            if ((ea >> 32) > (eb >> 32))   // roots hold their own keys; link the larger under the smaller
                            {
                                const uint32_t t = a;
                                a = b;
                                b = t;
                                const uint64_t te = ea;
                                ea = eb;
                                eb = te;
                            }
                            const uint64_t old = __hip_atomic_fetch_min(&L[b], SlotEntry(static_cast<uint32_t>(ea >> 32), a),
                                                                        __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
                            if (old == eb)
                                open = false;
                            else   // b had been linked under old's parent (which this link may have displaced): unite with it
                                b = static_cast<uint32_t>(old);
                        }
                    }
                }
            }
        }
        __syncthreads();

        const bool random_rule = d.flip_rule != 0u;
        const uint32_t key = random_rule ? fkey : 0u;
        if (w < nb)
        {
            const uint32_t nslot = Uniform(min(cnt, max_slots));
            uint32_t* const bits = sw + blk * 8u;
            // two slots per lane, their chases in flight together
            for (uint32_t s0 = 0; s0 < nslot; s0 += 128u)
            {
                uint32_t n[2];
                uint64_t e[2];
#pragma unroll
                for (uint32_t j = 0; j < 2u; ++j)
                {
                    n[j] = blk * kNodes + min(s0 + 64u * j + lane, nslot - 1u);
                    e[j] = LocalEntry(L, n[j]);
                }
                // (a node that no edge named, of a count that is too large, holds whatever the LDS held: its chase stays in
                // the table and ends by its length; roots read themselves again)
                uint32_t left = nb * kNodes;
                for (; left != 0u; --left)
                {
                    uint32_t moved = 0;
#pragma unroll
                    for (uint32_t j = 0; j < 2u; ++j)
                    {
                        const uint32_t up = min(static_cast<uint32_t>(e[j]), nb * kNodes - 1u);
                        moved |= up ^ n[j];
                        n[j] = up;
                    }
                    if (!__ballot(moved != 0u))
                        break;
#pragma unroll
                    for (uint32_t j = 0; j < 2u; ++j)
                        e[j] = LocalEntry(L, n[j]);
                }
                ok = ok && left != 0u;
#pragma unroll
                for (uint32_t j = 0; j < 2u; ++j)
                {
                    const uint32_t first = s0 + 64u * j, i = first + lane;
                    uint32_t bit = 0;
                    if (i < nslot)
                    {
                        const uint32_t root = static_cast<uint32_t>(e[j] >> 32);
                        bit = FlipBit(d, root, random_rule, key);
                        Glob(d.cpar)[bslots * blk + i] = SlotEntry(root, bslots * (n[j] / kNodes) + n[j] % kNodes);
                    }
                    const uint64_t m = __ballot(bit != 0u);
                    if (first < nslot && lane < 2u)
                    {
                        const uint32_t v = lane ? static_cast<uint32_t>(m >> 32) : static_cast<uint32_t>(m);
                        bits[(first >> 5) + lane] = v;
                        if ((first >> 5) + lane < d.fsw)
                            Glob(d.fbits)[blk * d.fsw + (first >> 5) + lane] = v;
                    }
                }
            }
            const auto flip = [&](const uint32_t lab) -> uint32_t {
                const uint32_t i = lab & 0x7FFFu;
                if (lab & kEdgeFlag)
                {
                    const uint32_t s = i - qcap;
                    if (s >= nslot)
                    {
                        ok = false;
                        return 0u;
                    }
                    return (LdsLoad(&bits[s >> 5]) >> (s & 31u)) & 1u;
                }
                if (i >= blk_rows * 64u)
                {
                    ok = false;
                    return 0u;
                }
                return FlipBit(d, SiteOf((blk / tx) * brows * stride + (blk % tx) * 64u, stride, i), random_rule, key);
            };
            if (lane < blk_rows)
                halo[lane] = static_cast<uint8_t>((sc ^ flip(hc)) & 1u);
            halo[es + lane] = static_cast<uint8_t>((sr ^ flip(hr)) & 1u);
        }
        if (!ok)
            (void)__hip_atomic_fetch_or(stp + kStErr, kErrLabelRange, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if (threadIdx.x == 0)
            AdvanceIteration(d, it);
    }

    // Applies a pending flip to the spin array (lattices without one return at once): per block (two
    // waves, every block of a 4096^2 lattice resident at once), the flip bits written by k_resolve and the
    // labels of the last sweep, four sites per lane. k_set_applied follows it.
    __global__ __launch_bounds__(128) void k_flip(const LatDesc* __restrict__ descs, const uint32_t* __restrict__ block_lat,
                                                  const uint32_t total_blocks)
    {
        constexpr uint32_t kThreads = 128;
        constexpr uint32_t kPass = kThreads / 16;   // wave rows per pass of the workgroup (16 lanes per wave row)
        constexpr uint32_t kCh = 8;                 // passes loaded together
        constexpr uint32_t kMaxSites = kWavesPerBlock * 64u * 64u;
        __shared__ uint32_t fb[2u * kMaxSites / 32u];
        const uint32_t b = RemapBlock(total_blocks);
        if (b >= total_blocks)
            return;
        const LatDesc& d = descs[LatticeOf(block_lat, b)];
        const gptr<uint32_t> stp = Glob(d.state);
        if (stp[kStApplied] == stp[kStIteration])
            return;
        const Block bl = DecodeBlock(d, b);
        const gptr<uint16_t> local = Glob(d.local);
        const gptr<uint8_t> spins = Glob(d.spins);
        const uint32_t qmax = bl.nwr * 64u, qcap = d.qcap, slots = kWavesPerBlock * d.edge_cap;
        const uint32_t sub = threadIdx.x >> 4;
        const uint32_t col = (threadIdx.x & 15u) * 4u;
        bool ok = true;

        u32x2 lv[kCh];
        uint32_t sv[kCh];
        const auto load = [&](const uint32_t r0) {
#pragma unroll
            for (uint32_t k = 0; k < kCh; ++k)
            {
                const uint32_t r = r0 + sub + k * kPass;
                lv[k] = u32x2{0u, 0u};
                sv[k] = 0u;
                if (r < bl.nwr)
                {
                    const uint32_t site = bl.base + r * bl.stride + col;
                    lv[k] = *(gptr<const u32x2>)(local + site);
                    sv[k] = *(gptr<const uint32_t>)(spins + site);
                }
            }
        };
        load(0u);
        // the edge-reaching clusters' bits from k_resolve, and the rule words of the clusters inside the block
        // (the pending flip belongs to the sweep that started at iteration `applied`)
        const gptr<const uint32_t> fbits_g = Glob(static_cast<const uint32_t*>(d.fbits)) + bl.lb * d.fsw;
        for (uint32_t i = threadIdx.x; i < d.fsw; i += kThreads)
            fb[qcap / 32u + i] = fbits_g[i];
        const bool random_rule = d.flip_rule != 0u;
        const uint32_t key = random_rule ? FlipKey(d.seed, stp[kStApplied]) : 0u;
        for (uint32_t i = threadIdx.x; i < bl.nwr * 2u; i += kThreads)
            fb[i] = RuleWord(d, bl, i, random_rule, key);
        __syncthreads();

        for (uint32_t r0 = 0;;)
        {
#pragma unroll
            for (uint32_t k = 0; k < kCh; ++k)
            {
                const uint32_t r = r0 + sub + k * kPass;
                if (r < bl.nwr)
                {
                    const uint32_t site = bl.base + r * bl.stride + col;
                    const uint32_t lab[4] = {lv[k].x & 0xFFFFu, lv[k].x >> 16, lv[k].y & 0xFFFFu, lv[k].y >> 16};
                    uint32_t flip = 0;
#pragma unroll
                    for (uint32_t e = 0; e < 4; ++e)
                        flip |= FlipOfLabel(lab[e], fb, qmax, qcap, slots, ok) << (8u * e);
                    *(gptr<uint32_t>)(spins + site) = sv[k] ^ flip;
                }
            }
            r0 += kCh * kPass;
            if (r0 >= bl.nwr)
                break;
            load(r0);
        }
        if (!ok)
            (void)__hip_atomic_fetch_or(stp + kStErr, kErrLabelRange, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }

    // After k_flip over a work list: every lattice's spin array holds its chain's state.
    __global__ __launch_bounds__(256) void k_set_applied(const LatDesc* __restrict__ descs, const uint32_t* __restrict__ block_lat,
                                                         const uint32_t total_blocks)
    {
        const uint32_t b = blockIdx.x * 256u + threadIdx.x;
        if (b >= total_blocks)
            return;
        const LatDesc& d = descs[LatticeOf(block_lat, b)];
        if (b == d.block_base)
            d.state[kStApplied] = d.state[kStIteration];
    }

    __global__ void k_set_applied_one(uint32_t* __restrict__ state)
    {
        state[kStApplied] = state[kStIteration];
    }

    // Inspection kernel: the canonical label (minimum site index) of every site, written to parent[]: the
    // canonical root of every slot of the block (kept in LDS, one word per slot), then every site's label.
    __device__ __forceinline__ void WriteLabels(const LatDesc& d, const uint32_t b)
    {
        constexpr uint32_t kPass = 16;   // wave rows per pass of the workgroup (16 lanes per wave row)
        constexpr uint32_t kCh = 4;      // passes loaded together
        extern __shared__ uint32_t R[];  // kWavesPerBlock * edge_cap entries (at most the block's sites)
        const Block bl = DecodeBlock(d, b);
        const gptr<uint32_t> L = Glob(d.parent);
        const gptr<uint16_t> local = Glob(d.local);
        const uint32_t qmax = bl.nwr * 64u, qcap = d.qcap, slots = kWavesPerBlock * d.edge_cap;
        const uint32_t sub = threadIdx.x >> 4;
        const uint32_t col = (threadIdx.x & 15u) * 4u;
        bool ok = true;
        const bool whole = Glob(static_cast<const uint32_t*>(d.aux))[kAuxWholeLabels] != 0u;

        u32x2 lv[kCh];
        const auto load = [&](const uint32_t r0) {
#pragma unroll
            for (uint32_t k = 0; k < kCh; ++k)
            {
                const uint32_t r = r0 + sub + k * kPass;
                lv[k] = u32x2{0u, 0u};
                if (r < bl.nwr)
                    lv[k] = *(gptr<const u32x2>)(local + bl.base + r * bl.stride + col);
            }
        };
        load(0u);

        // phase 1: canonical root of every slot in use
        const gptr<uint64_t> E = Glob(d.cpar);
        const uint32_t c_max = d.n_blocks * slots;
        if (!whole)
            ForBlockSlots(d, bl, threadIdx.x, 256u, [&](const uint32_t slot, const uint32_t c) { R[slot] = SlotRootKey(E, c, CachedLoad64(&E[c]), c_max, ok); });
        __syncthreads();

        // phase 2: every site's label, four sites per lane
        for (uint32_t r0 = 0;;)
        {
#pragma unroll
            for (uint32_t k = 0; k < kCh; ++k)
            {
                const uint32_t r = r0 + sub + k * kPass;
                if (r < bl.nwr)
                {
                    const uint32_t site = bl.base + r * bl.stride + col;
                    const uint32_t lab[4] = {lv[k].x & 0xFFFFu, lv[k].x >> 16, lv[k].y & 0xFFFFu, lv[k].y >> 16};
                    uint32_t root[4];
#pragma unroll
                    for (uint32_t e = 0; e < 4; ++e)
                    {
                        if (whole)   // the label is the canonical site already
                        {
                            root[e] = lab[e];
                            continue;
                        }
                        const uint32_t i = LabelBit(lab[e], qmax, qcap, slots, ok);
                        root[e] = (lab[e] & kEdgeFlag) ? R[i >= qcap ? i - qcap : 0u] : SiteOf(bl.base, bl.stride, i);
                    }
                    *(gptr<u32x4>)(L + site) = u32x4{root[0], root[1], root[2], root[3]};
                }
            }
            r0 += kCh * kPass;
            if (r0 >= bl.nwr)
                break;
            load(r0);
        }
        if (!ok)
            (void)__hip_atomic_fetch_or(Glob(d.state) + kStErr, kErrLabelRange, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }

    __global__ __launch_bounds__(256) void k_write_labels(const LatDesc* __restrict__ descs, const uint32_t* __restrict__ block_lat,
                                                          const uint32_t total_blocks)
    {
        const uint32_t b = RemapBlock(total_blocks);
        if (b < total_blocks)
            WriteLabels(descs[LatticeOf(block_lat, b)], b);
    }

    __global__ __launch_bounds__(256) void k_write_labels_one(const LatDesc d, const uint32_t total_blocks)
    {
        const uint32_t b = RemapBlock(total_blocks);
        if (b < total_blocks)
            WriteLabels(d, b);
    }

    // =============================================================================================
    // Observables: per-block partial sums of sum s(s_right + s_down) and sum s (lattice.cpp:29-67)
    // =============================================================================================
    // A conditional sample is due when the lattice has advanced since its last sample, is past its warmup
    // and sits on its own n_sep grid.
    __device__ __forceinline__ bool SampleDue(const uint32_t* st)
    {
        const uint32_t it = st[kStIteration], meas = st[kStItMeas], sep2 = st[kStSep2];
        return it > st[kStLastSample] && it > meas && sep2 != 0u && (it - meas) % sep2 == 0u;
    }

    // A flip that is still pending is applied on the way (from the labels and the flip bits, as k_bond_label does) and
    // not stored: the spin array is read once (1 byte a site, 3 with the labels of a pending flip) and left for the
    // next sweep (8192^2: 206 us per sample with k_flip, k_set_applied and three reads per spin, now 75 with the final
    // sum, 68 of them here for 3 bytes a site, 2.9 TB/s). Per wave one tile: spin masks of its rows by ballot, one per
    // lane, the neighbours by shifts and from the next lane; the row below the tile is read again by the tile above it (or comes from the halo across the block
    // edge). Summing row by row with scalar operations was bound by the scalar unit (104 us at 8192^2).
    __global__ __launch_bounds__(256) void k_observables(const LatDesc* __restrict__ descs, const uint32_t* __restrict__ block_lat,
                                                         const uint32_t total_blocks, const uint32_t sample_mode)
    {
        constexpr uint32_t kCh = 8;   // rows loaded together
        constexpr uint32_t kMaxSites = kWavesPerBlock * 64u * 64u;
        __shared__ uint32_t fb[2u * kMaxSites / 32u];
        __shared__ int32_t s_e[kWavesPerBlock], s_m[kWavesPerBlock];
        const uint32_t b = RemapBlock(total_blocks);
        if (b >= total_blocks)
            return;
        const LatDesc& d = descs[LatticeOf(block_lat, b)];
        if (sample_mode == kSampleDue && !SampleDue(d.state))
            return;
        const gptr<const uint32_t> stp = Glob(static_cast<const uint32_t*>(d.state));
        const bool pending = stp[kStApplied] != stp[kStIteration];
        const Block bl = DecodeBlock(d, b);
        const uint32_t lane = threadIdx.x & 63u;
        const uint32_t w = Uniform(threadIdx.x >> 6);
        const uint32_t r_begin = w * d.twr;
        const uint32_t nrow = bl.nwr > r_begin ? min(d.twr, bl.nwr - r_begin) : 0u;
        const bool last_wave = r_begin + nrow >= bl.nwr;
        const uint32_t pitch = d.n0, tw = d.tw, qcap = d.qcap;
        const bool lastcol = bl.sx + 1u == d.tiles_x;
        const uint64_t vmask = lastcol ? d.vlast : ~0ull;   // lanes that hold sites
        const uint32_t elane = lastcol ? d.elast : tw - 1u;  // a lattice row's last site in this tile
        uint64_t rowstart = 1;
        for (uint32_t j = tw; j < 64u; j += tw)
            rowstart |= 1ull << j;
        const uint64_t redge = rowstart << elane;
        const uint64_t low = Shr(~0ull, tw);   // lanes whose lower neighbour sits in the same wave row
        const uint32_t sx_r = lastcol ? 0u : bl.sx + 1u;
        const uint32_t sy_b = bl.sy + 1u == d.blocks_y ? 0u : bl.sy + 1u;
        const gptr<const uint8_t> spins = Glob(static_cast<const uint8_t*>(d.spins));
        const gptr<const uint16_t> local = Glob(static_cast<const uint16_t*>(d.local));
        const gptr<const uint8_t> halo = Glob(static_cast<const uint8_t*>(d.halo)) + stp[kStHaloSide] * d.n_blocks * d.halo_stride;

        if (pending)
        {
            const gptr<const uint32_t> fbits_g = Glob(static_cast<const uint32_t*>(d.fbits)) + bl.lb * d.fsw;
            for (uint32_t i = threadIdx.x; i < d.fsw; i += 256u)
                fb[qcap / 32u + i] = fbits_g[i];
            const bool random_rule = d.flip_rule != 0u;
            const uint32_t key = random_rule ? FlipKey(d.seed, stp[kStApplied]) : 0u;
            for (uint32_t i = threadIdx.x; i < bl.nwr * 2u; i += 256u)
                fb[i] = RuleWord(d, bl, i, random_rule, key);
        }
        // 64-wide tiles: lane r's hr is the spin to the right of the tile's row r (narrower ones wrap inside the row)
        uint32_t hr = 0;
        if (tw == 64u && lane < nrow)
            hr = pending ? halo[(bl.sy * d.tiles_x + sx_r) * d.halo_stride + r_begin + lane]
                         : spins[(bl.wyb + r_begin + lane) * pitch + sx_r * 64u];

        // the row below the tile: the next tile's first row, or across the block edge the halo (the flipped spins of a
        // pending flip); loaded without conditions, like the rows of a chunk, so that the loads overlap
        // (in range for every wave: the last tile and the waves past it, which own no rows in a partial block, read the
        // block's last row and do not use it)
        const uint32_t r_below = min(r_begin + nrow, bl.nwr - 1u);
        const uint32_t site_below = last_wave && !pending ? BlockBase(d, bl.sx, sy_b) + lane : bl.base + r_below * bl.stride + lane;
        const uint32_t below_sp = spins[site_below], below_lab = local[site_below];
        const uint32_t below_halo = halo[(sy_b * d.tiles_x + bl.sx) * d.halo_stride + d.ecol_stride + lane];
        __syncthreads();

        // (a label outside the block's range is a broken invariant, as in k_flip)
        const uint32_t qmax = bl.nwr * 64u, slots = kWavesPerBlock * d.edge_cap, first_slot = kEdgeFlag + qcap;
        uint64_t bad = 0;   // lanes
        const auto flip_of = [&](const uint32_t lab) {
            const uint32_t i = lab & 0x7FFFu;
            bad |= __ballot(lab >= qmax) & __ballot(lab - first_slot >= slots);
            return fb[min(i >> 5, 2u * kMaxSites / 32u - 1u)] >> (i & 31u);
        };
        const uint64_t Sbelow = __ballot((((pending ? (last_wave ? below_halo : below_sp ^ flip_of(below_lab)) : below_sp)) & 1u) != 0u);
        // lane r collects the mask of the tile's row r (nrow <= 64): the sums are then one row per lane
        uint32_t Slo = 0, Shi = 0;
        const uint32_t span = (bl.nwr - 1u) * bl.stride + 64u;
        const Rsrc rs_spins = MakeRsrc(d.spins + bl.base, span), rs_local = MakeRsrc(d.local + bl.base, span * 2u);
        const auto rows = [&](auto pending_t) {
            constexpr bool kPend = decltype(pending_t)::value;
            for (uint32_t r0 = 0; r0 < nrow; r0 += kCh)
            {
                uint32_t sp[kCh], lab[kCh];
#pragma unroll
                for (uint32_t k = 0; k < kCh; ++k)
                {
                    const uint32_t off = Uniform((r_begin + min(r0 + k, nrow - 1u)) * bl.stride);
                    sp[k] = __builtin_amdgcn_raw_buffer_load_b8(rs_spins, lane, off, 0);
                    lab[k] = kPend ? __builtin_amdgcn_raw_buffer_load_b16(rs_local, lane * 2u, off * 2u, 0) : 0u;
                }
#pragma unroll
                for (uint32_t k = 0; k < kCh; ++k)
                {
                    const uint32_t r = r0 + k;
                    if (r < nrow)
                    {
                        const uint64_t S = __ballot(((kPend ? sp[k] ^ flip_of(lab[k]) : sp[k]) & 1u) != 0u);
                        Slo = LaneBit(1ull << r) ? static_cast<uint32_t>(S) : Slo;
                        Shi = LaneBit(1ull << r) ? static_cast<uint32_t>(S >> 32) : Shi;
                    }
                }
            }
        };
        if (pending)
            rows(std::true_type{});
        else
            rows(std::false_type{});
        if (bad != 0ull && lane == 0u)
            (void)__hip_atomic_fetch_or(Glob(d.state) + kStErr, kErrLabelRange, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        int32_t e = 0, m = 0;
        {
            const uint64_t S = (static_cast<uint64_t>(Shi) << 32) | Slo;
            const bool last = lane + 1u >= nrow;
            const uint32_t dlo = __shfl_down(Slo, 1), dhi = __shfl_down(Shi, 1);
            const uint64_t Sn = last ? Sbelow : (static_cast<uint64_t>(dhi) << 32) | dlo;
            const uint64_t RS = ((S >> 1) & ~redge) | (tw == 64u ? static_cast<uint64_t>(hr & 1u) << elane : (S << elane) & redge);
            const uint64_t SD = (Shr(S, tw) & low) | Shl(Sn, 64u - tw);
            const int32_t nv = __popcll(vmask);
            if (lane < nrow)
            {
                e = 2 * (__popcll(~(S ^ RS) & vmask) + __popcll(~(S ^ SD) & vmask)) - 2 * nv;
                m = 2 * __popcll(S & vmask) - nv;
            }
        }
        for (uint32_t s = 32; s > 0; s >>= 1)
        {
            e += __shfl_down(e, s);
            m += __shfl_down(m, s);
        }
        if (lane == 0u)
        {
            s_e[w] = e;
            s_m[w] = m;
        }
        __syncthreads();
        if (threadIdx.x == 0)
        {
            d.partials[2u * bl.lb] = s_e[0] + s_e[1] + s_e[2] + s_e[3];
            d.partials[2u * bl.lb + 1u] = s_m[0] + s_m[1] + s_m[2] + s_m[3];
        }
    }

    // One workgroup per lattice: reduce the block partials (whole numbers: any order), append (E, M) to the series
    // and accumulate the FP64 moments (the only FP64 of the tiled path).
    template <uint32_t kWaves>
    __global__ __launch_bounds__(64 * kWaves) void k_finalize_samples(const LatDesc* __restrict__ descs, const uint32_t* __restrict__ slots,
                                                                      const uint32_t sample_mode)
    {
        constexpr uint32_t kThreads = 64u * kWaves, kCh = kWaves == 1u ? 1u : 8u;   // entries loaded together per thread
        __shared__ long long red_e[kWaves], red_m[kWaves];
        const LatDesc& d = descs[slots[blockIdx.x]];
        if (sample_mode == kSampleDue && !SampleDue(d.state))
            return;
        long long e = 0, m = 0;
        const gptr<const u32x2> part = (gptr<const u32x2>)(d.partials);
        const uint32_t n_blocks = d.n_blocks;
        for (uint32_t i = threadIdx.x; i < n_blocks; i += kCh * kThreads)
        {
            u32x2 v[kCh];
#pragma unroll
            for (uint32_t k = 0; k < kCh; ++k)
                v[k] = part[min(i + k * kThreads, n_blocks - 1u)];
#pragma unroll
            for (uint32_t k = 0; k < kCh; ++k)
                if (i + k * kThreads < n_blocks)
                {
                    e += static_cast<int32_t>(v[k].x);
                    m += static_cast<int32_t>(v[k].y);
                }
        }
        for (uint32_t s = 32; s > 0; s >>= 1)
        {
            e += __shfl_down(e, s);
            m += __shfl_down(m, s);
        }
        if ((threadIdx.x & 63u) == 0u)
        {
            red_e[threadIdx.x >> 6] = e;
            red_m[threadIdx.x >> 6] = m;
        }
        __syncthreads();
        if (threadIdx.x == 0)
            for (uint32_t k = 1; k < kWaves; ++k)
            {
                red_e[0] += red_e[k];
                red_m[0] += red_m[k];
            }
        if (threadIdx.x == 0)
        {
            LatState* st = reinterpret_cast<LatState*>(d.state);
            const double n = static_cast<double>(d.n0v) * static_cast<double>(d.n1);
            const double ev = -static_cast<double>(red_e[0]) / n;
            const double mv = static_cast<double>(red_m[0]) / n;
            st->moments[0] += 1.0;
            st->moments[1] += ev;
            st->moments[2] += ev * ev;
            st->moments[3] += fabs(mv);
            st->moments[4] += mv * mv;
            st->moments[5] += (mv * mv) * (mv * mv);
            if (st->n_samples < st->series_cap)
            {
                long long* series = reinterpret_cast<long long*>(d.state + kLatStateWords);
                series[2u * st->n_samples] = red_e[0];
                series[2u * st->n_samples + 1u] = red_m[0];
            }
            st->n_samples += 1u;
            st->last_sample = st->iteration;
        }
    }

    // Fresh per-lattice state: counters and moments zero, no sweep limit unless it_end says otherwise.
    __global__ __launch_bounds__(256) void k_init_state(uint32_t* __restrict__ state, uint32_t* __restrict__ aux, const uint32_t words,
                                                        const uint32_t series_cap, const uint32_t it_end, const uint32_t it_meas,
                                                        const uint32_t sep2)
    {
        if (threadIdx.x < kAuxWords)
            aux[threadIdx.x] = 0u;
        for (uint32_t i = threadIdx.x; i < words; i += blockDim.x)
        {
            uint32_t v = 0;
            if (i == 2u)
                v = series_cap;
            else if (i == kStItEnd)
                v = it_end;
            else if (i == kStActive)
                v = 1u;
            else if (i == kStItMeas)
                v = it_meas;
            else if (i == kStSep2)
                v = sep2;
            state[i] = v;
        }
    }

    __global__ void k_set_rng_current(const uint32_t* __restrict__ state, uint32_t* __restrict__ aux) { aux[kAuxRngIt] = state[kStIteration]; }

    // The states of the lattice's current iteration, for callers that read them (export, checkpoint): four sites per
    // thread, the pair of each site's selector applied once per update since. k_set_rng_current follows it.
    __global__ __launch_bounds__(256) void k_advance_rng(const uint32_t* __restrict__ spins4, u32x4* __restrict__ rng4, const uint64_t n4,
                                                         const uint32_t* __restrict__ state, const uint32_t* __restrict__ aux)
    {
        __shared__ uint32_t JA[8], JC[8];
        const uint32_t n = state[kStIteration] - aux[kAuxRngIt];
        if (n == 0u)
            return;
        if (threadIdx.x < 8u)
        {
            uint32_t a, c, ja = 1u, jc = 0u;
            ParamsOf(threadIdx.x, a, c);
            for (uint32_t i = 0; i < n; ++i)
            {
                ja *= a;
                jc = a * jc + c;
            }
            JA[threadIdx.x] = ja;
            JC[threadIdx.x] = jc;
        }
        __syncthreads();
        const uint64_t i = static_cast<uint64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
        if (i >= n4)
            return;
        const uint32_t sel = spins4[i] >> kSelShift;
        u32x4 v = rng4[i];
#pragma unroll
        for (uint32_t e = 0; e < 4u; ++e)
        {
            const uint32_t k = (sel >> (8u * e)) & 7u;
            v[e] = JA[k] * v[e] + JC[k];
        }
        rng4[i] = v;
    }

    // Schedule relative to the current iteration: `sweeps` more sweeps (0: no limit), the first `warmup` of
    // them unsampled, then a conditional sample after every n_sep-th.
    __global__ void k_set_schedule(uint32_t* __restrict__ state, const uint32_t sweeps, const uint32_t warmup, const uint32_t n_sep)
    {
        if (threadIdx.x != 0)
            return;
        const uint32_t it = state[kStIteration];
        state[kStItEnd] = sweeps ? it + 2u * sweeps : 0xFFFFFFFFu;
        state[kStItMeas] = it + 2u * warmup;
        state[kStSep2] = 2u * n_sep;
        state[kStLastSample] = it;
    }

    // =============================================================================================
    // Initialisation
    // =============================================================================================
    // LCG32_State<64>::Init (random/src/lcg32.cpp:31-49) of every group, one thread per group, with the
    // POSIX drand48 recurrence in 48-bit integer arithmetic and IEEE double products.
    // The selector of lane i (bits 1-3 of the spin byte of site 64g+i) starts as sel0[i]; run after the
    // spins are set.
    __global__ __launch_bounds__(256) void k_init_rng(uint8_t* __restrict__ spins, uint32_t* __restrict__ rng, uint64_t* __restrict__ masks,
                                                      uint32_t* __restrict__ rot, const uint32_t n_groups, const uint32_t seed)
    {
        const uint32_t g = blockIdx.x * blockDim.x + threadIdx.x;
        if (g >= n_groups)
            return;
        const uint64_t kA = 0x5DEECE66Dull, kC = 0xBull, kMask = (1ull << 48) - 1ull;
        uint64_t xs = (static_cast<uint64_t>(seed * 0x9E3779B1u + g + 1u) << 16) | 0x330Eull;
        uint64_t m0 = 0, m1 = 0, m2 = 0;
        for (uint32_t i = 0; i < 64u; ++i)
        {
            xs = (kA * xs + kC) & kMask;
            const double dr = static_cast<double>(xs) * 0x1p-48;
            const uint32_t k = static_cast<uint32_t>(__dmul_rn(1000.0, dr)) % 5u;
            m0 |= static_cast<uint64_t>(k & 1u) << i;
            m1 |= static_cast<uint64_t>((k >> 1) & 1u) << i;
            m2 |= static_cast<uint64_t>((k >> 2) & 1u) << i;
        }
        xs = (kA * xs + kC) & kMask;
        const double dr = static_cast<double>(xs) * 0x1p-48;
        uint32_t a, c;
        ParamsOf(static_cast<uint32_t>((m0 & 1ull) | ((m1 & 1ull) << 1) | ((m2 & 1ull) << 2)), a, c);
        uint32_t st = a * (static_cast<uint32_t>(__dmul_rn(4026531839.0, dr)) + 1u) + c;
        uint32_t* out = rng + static_cast<size_t>(g) * 64u;
        uint8_t* sp = spins + static_cast<size_t>(g) * 64u;
        out[0] = st;
        for (uint32_t i = 0; i < 64u; ++i)
        {
            const uint32_t k = static_cast<uint32_t>(((m0 >> i) & 1ull) | (((m1 >> i) & 1ull) << 1) | (((m2 >> i) & 1ull) << 2));
            sp[i] = static_cast<uint8_t>((sp[i] & 1u) | (k << kSelShift));
            if (i > 0)
            {
                ParamsOf(k, a, c);
                st = a * st + c;
                out[i] = st;
            }
        }
        masks[3u * g] = m0;
        masks[3u * g + 1u] = m1;
        masks[3u * g + 2u] = m2;
        rot[g] = 0;
    }

    // Hot start (ising/src/lattice.cpp:24-26): site i gets the (i+1)-th drand48 of srand48(spin_seed);
    // drand48() < 0.5 <=> bit 47 of the 48-bit state is clear. Each thread jumps ahead to its chunk. Site
    // i = y*n0v + x is stored at y*pitch + x.
    __global__ __launch_bounds__(256) void k_hot_start(uint8_t* __restrict__ spins, const uint64_t n, const uint32_t spin_seed,
                                                       const uint32_t n0v, const uint32_t pitch)
    {
        constexpr uint32_t kChunk = 64;
        const uint64_t first = (static_cast<uint64_t>(blockIdx.x) * blockDim.x + threadIdx.x) * kChunk;
        if (first >= n)
            return;
        const uint64_t kMask = (1ull << 48) - 1ull;
        // (ja, jc) = affine map x -> A x + C raised to the power `first`
        uint64_t ja = 1, jc = 0, ba = 0x5DEECE66Dull, bc = 0xBull;
        for (uint64_t e = first; e; e >>= 1)
        {
            if (e & 1ull)
            {
                ja = (ba * ja) & kMask;
                jc = (ba * jc + bc) & kMask;
            }
            bc = (ba * bc + bc) & kMask;
            ba = (ba * ba) & kMask;
        }
        uint64_t xs = (static_cast<uint64_t>(spin_seed) << 16) | 0x330Eull;
        xs = (ja * xs + jc) & kMask;
        const uint64_t end = min(n, first + kChunk);
        for (uint64_t i = first; i < end; ++i)
        {
            xs = (0x5DEECE66Dull * xs + 0xBull) & kMask;
            const uint64_t at = n0v == pitch ? i : (i / n0v) * pitch + i % n0v;
            spins[at] = static_cast<uint8_t>((xs >> 47) & 1ull);
        }
    }

    // Upload of n row-major spins: replace bit 0 of every spin byte (site i = y*n0v + x at y*pitch + x), keep
    // the lcg32 selector bits.
    __global__ __launch_bounds__(256) void k_set_spins(uint8_t* __restrict__ spins, const uint8_t* __restrict__ src, const uint64_t n,
                                                       const uint32_t n0v, const uint32_t pitch)
    {
        const uint64_t i = static_cast<uint64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
        if (i < n)
        {
            const uint64_t at = n0v == pitch ? i : (i / n0v) * pitch + i % n0v;
            spins[at] = static_cast<uint8_t>((spins[at] & 0xFEu) | (src[i] & 1u));
        }
    }

    // Download of row-major spins [first, first + n), bit 0 of the spin bytes: sixteen sites per thread where no row is
    // padded (first and n are then multiples of 64).
    __global__ __launch_bounds__(256) void k_get_spins(uint8_t* __restrict__ dst, const uint8_t* __restrict__ spins, const uint64_t first,
                                                       const uint64_t n,
                                                       const uint32_t n0v, const uint32_t pitch)
    {
        const uint64_t i = static_cast<uint64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
        if (n0v == pitch)
        {
            if (16u * i < n)
                reinterpret_cast<u32x4*>(dst)[i] = reinterpret_cast<const u32x4*>(spins + first)[i] & 0x01010101u;
        }
        else if (i < n)
            dst[i] = spins[((first + i) / n0v) * pitch + (first + i) % n0v] & 1u;
    }

    __global__ void k_set_threshold(LatDesc* __restrict__ a, LatDesc* __restrict__ b, const uint32_t threshold)
    {
        a->threshold = threshold;
        b->threshold = threshold;
    }

    __global__ __launch_bounds__(64) void k_reset_measurements(const LatDesc* __restrict__ descs, const uint32_t n)
    {
        const uint32_t i = blockIdx.x * 64u + threadIdx.x;
        if (i >= n)
            return;
        uint32_t* const state = descs[i].state;
        state[kStSamples] = 0u;
        for (uint32_t w = kStMoments; w < kLatStateWords; ++w)
            state[w] = 0u;
    }

    // Row-major bytes (n0v wide) to the padded layout (pitch wide, padding columns 0), and back.
    __global__ __launch_bounds__(256) void k_pad_bytes(uint8_t* __restrict__ dst, const uint8_t* __restrict__ src, const uint64_t np,
                                                       const uint32_t n0v, const uint32_t pitch)
    {
        const uint64_t p = static_cast<uint64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
        if (p < np)
        {
            const uint64_t x = p % pitch;
            dst[p] = x < n0v ? src[(p / pitch) * n0v + x] : 0u;
        }
    }

    // Canonical padded labels (root's padded index per padded site) to row-major labels of row-major sites.
    __global__ __launch_bounds__(256) void k_unpad_labels(uint32_t* __restrict__ dst, const uint32_t* __restrict__ src, const uint64_t n,
                                                          const uint32_t n0v, const uint32_t pitch)
    {
        const uint64_t i = static_cast<uint64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
        if (i < n)
        {
            const uint32_t root = src[(i / n0v) * pitch + i % n0v];
            dst[i] = (root / pitch) * n0v + root % pitch;
        }
    }

    __global__ __launch_bounds__(256) void k_copy(const uint4* __restrict__ src, uint4* __restrict__ dst, const uint64_t n16)
    {
        for (uint64_t i = static_cast<uint64_t>(blockIdx.x) * blockDim.x + threadIdx.x; i < n16;
             i += static_cast<uint64_t>(gridDim.x) * blockDim.x)
            dst[i] = src[i];
    }

    // =============================================================================================
    // launch wrappers
    // =============================================================================================
    // defined in swmi_bond.hip, one part per combination
    template <bool TW64, BondMode MODE>
    void LaunchBondLabelT(const LatDesc* d_desc, const uint32_t* d_block_lat, uint32_t total_blocks, uint32_t max_twr, BondForm form, bool pad,
                          hipStream_t stream);

    template <bool TW64>
    void LaunchLabelBlocksT(const LatDesc& d, uint32_t total_blocks, BondForm form, bool pad, hipStream_t stream);

    void LaunchBondLabel(const LatDesc* d_desc, const uint32_t* d_block_lat, const uint32_t total_blocks, const uint32_t max_twr,
                         const BondForm form, const bool all_tw64, const bool pad, const bool debug, hipStream_t stream)
    {
        if (debug)
        {
            if (all_tw64)
                LaunchBondLabelT<true, BondMode::kInspect>(d_desc, d_block_lat, total_blocks, max_twr, form, pad, stream);
            else
                LaunchBondLabelT<false, BondMode::kInspect>(d_desc, d_block_lat, total_blocks, max_twr, form, pad, stream);
        }
        else if (all_tw64)
            LaunchBondLabelT<true, BondMode::kSweep>(d_desc, d_block_lat, total_blocks, max_twr, form, pad, stream);
        else
            LaunchBondLabelT<false, BondMode::kSweep>(d_desc, d_block_lat, total_blocks, max_twr, form, pad, stream);
    }

    // Two-wave merge workgroups resident at once on MI355X: 256 CUs x 16 (8 waves per SIMD).
    constexpr uint32_t kOneRoundMergeBlocks = 4096;
    // Launches of at least this many blocks unite each edge's pairs in LDS before the lattice-wide unions: many
    // blocks race on the memory-side atomics there. Smaller launches see few races and only the added latency.
    // Microseconds per sweep without / with, both edges of a block in one wave (k_merge_block) at T_c: 36 blocks 19.6 /
    // 21.0, 256 blocks 21.8 / 23.4, 1024 blocks 32.6 / 33.5, 4096 blocks (with each edge's own local unions before, which
    // narrow and tall tiles keep) 67.4 / 66.9, 16384 blocks 234.8 / 224.8.
    constexpr uint32_t kLocalUnionBlocks = 4096;

    template <bool FRESH>
    void LaunchMergeAs(const LatDesc* d_desc, const uint32_t* d_block_lat, const uint32_t total_blocks, hipStream_t stream)
    {
        if (total_blocks >= kLocalUnionBlocks)
            k_merge<FRESH, true><<<XcdGrid(total_blocks), 128, 0, stream>>>(d_desc, d_block_lat, total_blocks);
        else
            k_merge<FRESH, false><<<XcdGrid(total_blocks), 128, 0, stream>>>(d_desc, d_block_lat, total_blocks);
    }

    void LaunchMerge(const LatDesc* d_desc, const uint32_t* d_block_lat, const uint32_t total_blocks, const bool all_tw64,
                     const uint32_t max_rows, hipStream_t stream)
    {
        if (all_tw64 && max_rows <= 64u && total_blocks >= kLocalUnionBlocks)
        {
            if (total_blocks <= kOneRoundMergeBlocks)
                k_merge_block<true><<<XcdGrid(total_blocks), 64, 0, stream>>>(d_desc, d_block_lat, total_blocks);
            else
                k_merge_block<false><<<XcdGrid(total_blocks), 64, 0, stream>>>(d_desc, d_block_lat, total_blocks);
            return;
        }
        if (total_blocks <= kOneRoundMergeBlocks)
            LaunchMergeAs<true>(d_desc, d_block_lat, total_blocks, stream);
        else
            LaunchMergeAs<false>(d_desc, d_block_lat, total_blocks, stream);
    }

    void LaunchResolve(const LatDesc* d_desc, const uint32_t* d_block_lat, const uint32_t total_blocks, const uint32_t max_rows,
                       hipStream_t stream)
    {
        // (a tile has at most 64 lattice rows, a block of 16-row tiles 64: one halo entry per thread instead of three)
        if (max_rows > 64u)
            k_resolve<kWavesPerBlock * 64u><<<XcdGrid(total_blocks), 128, 0, stream>>>(d_desc, d_block_lat, total_blocks);
        else
            k_resolve<64><<<XcdGrid(total_blocks), 128, 0, stream>>>(d_desc, d_block_lat, total_blocks);
    }

    void LaunchJoin(const LatDesc* d_desc, const uint32_t* d_slots, const uint32_t n_lattices, const uint32_t max_blocks, hipStream_t stream)
    {
        k_join<<<n_lattices, 1024, max_blocks * 256u * sizeof(uint64_t), stream>>>(d_desc, d_slots);
    }

    void LaunchMaterialize(const LatDesc* d_desc, const uint32_t* d_block_lat, const uint32_t total_blocks, hipStream_t stream)
    {
        k_flip<<<XcdGrid(total_blocks), 128, 0, stream>>>(d_desc, d_block_lat, total_blocks);
        k_set_applied<<<(total_blocks + 255u) / 256u, 256, 0, stream>>>(d_desc, d_block_lat, total_blocks);
    }

    void LaunchWriteLabels(const LatDesc* d_desc, const uint32_t* d_block_lat, const uint32_t total_blocks, const uint32_t max_twr,
                           hipStream_t stream)
    {
        const size_t lds = static_cast<size_t>(kWavesPerBlock) * max_twr * 64u * sizeof(uint32_t);
        k_write_labels<<<XcdGrid(total_blocks), 256, lds, stream>>>(d_desc, d_block_lat, total_blocks);
    }

    void LaunchSetApplied(uint32_t* state, hipStream_t stream) { k_set_applied_one<<<1, 1, 0, stream>>>(state); }

    void LaunchSetRngCurrent(const uint32_t* state, uint32_t* aux, hipStream_t stream)
    {
        k_set_rng_current<<<1, 1, 0, stream>>>(state, aux);
    }

    void LaunchAdvanceRng(const uint8_t* spins, uint32_t* rng, const uint64_t np, const uint32_t* state, uint32_t* aux, hipStream_t stream)
    {
        const uint64_t n4 = np / 4;   // np is a multiple of 64
        k_advance_rng<<<static_cast<uint32_t>((n4 + 255) / 256), 256, 0, stream>>>(reinterpret_cast<const uint32_t*>(spins),
                                                                                   reinterpret_cast<u32x4*>(rng), n4, state, aux);
        LaunchSetRngCurrent(state, aux, stream);
    }

    void LaunchLabelBlocks(const LatDesc& d, const BondForm form, const bool pad, hipStream_t stream)
    {
        const uint32_t g = XcdGrid(d.n_blocks);
        if (d.tw == 64u)
            LaunchLabelBlocksT<true>(d, d.n_blocks, form, pad, stream);
        else
            LaunchLabelBlocksT<false>(d, d.n_blocks, form, pad, stream);
        if (d.n_blocks <= kOneRoundMergeBlocks)
            k_merge_one<true><<<g, 128, 0, stream>>>(d, d.n_blocks);
        else
            k_merge_one<false><<<g, 128, 0, stream>>>(d, d.n_blocks);
        k_write_labels_one<<<g, 256, d.qcap * sizeof(uint32_t), stream>>>(d, d.n_blocks);
    }

    void LaunchObservables(const LatDesc* d_desc, const uint32_t* d_block_lat, const uint32_t total_blocks, const uint32_t sample_mode,
                           hipStream_t stream)
    {
        k_observables<<<XcdGrid(total_blocks), 256, 0, stream>>>(d_desc, d_block_lat, total_blocks, sample_mode);
    }

    // Lattices of at most 64 blocks take one wave: 6000 lattices of 8^2 measured every 10 sweeps take 48.8 us per sweep with
    // sixteen, 46.0 with one.
    void LaunchFinalizeSamples(const LatDesc* d_desc, const uint32_t* d_slots, const uint32_t n_lattices, const uint32_t max_blocks,
                               const uint32_t sample_mode, hipStream_t stream)
    {
        if (max_blocks <= 64u)
            k_finalize_samples<1><<<n_lattices, 64, 0, stream>>>(d_desc, d_slots, sample_mode);
        else
            k_finalize_samples<16><<<n_lattices, 1024, 0, stream>>>(d_desc, d_slots, sample_mode);
    }

    void LaunchInitState(uint32_t* state, uint32_t* aux, const uint32_t words, const uint32_t series_cap, const uint32_t it_end,
                         const uint32_t it_meas, const uint32_t sep2, hipStream_t stream)
    {
        k_init_state<<<1, 256, 0, stream>>>(state, aux, words, series_cap, it_end, it_meas, sep2);
    }

    void LaunchSetSchedule(uint32_t* state, const uint32_t sweeps, const uint32_t warmup, const uint32_t n_sep, hipStream_t stream)
    {
        k_set_schedule<<<1, 64, 0, stream>>>(state, sweeps, warmup, n_sep);
    }

    void LaunchInitRng(uint8_t* spins, uint32_t* rng, uint64_t* masks, uint32_t* rot, const uint32_t n_groups, const uint32_t seed,
                       hipStream_t stream)
    {
        k_init_rng<<<(n_groups + 255) / 256, 256, 0, stream>>>(spins, rng, masks, rot, n_groups, seed);
    }

    void LaunchSetSpins(uint8_t* spins, const uint8_t* src, const uint64_t n, const uint32_t n0v, const uint32_t pitch,
                        hipStream_t stream)
    {
        k_set_spins<<<static_cast<uint32_t>((n + 255) / 256), 256, 0, stream>>>(spins, src, n, n0v, pitch);
    }

    void LaunchGetSpins(uint8_t* dst, const uint8_t* spins, const uint64_t first, const uint64_t n, const uint32_t n0v, const uint32_t pitch,
                        hipStream_t stream)
    {
        const uint64_t threads = n0v == pitch ? n / 16u : n;
        k_get_spins<<<static_cast<uint32_t>((threads + 255) / 256), 256, 0, stream>>>(dst, spins, first, n, n0v, pitch);
    }

    void LaunchSetThreshold(LatDesc* a, LatDesc* b, const uint32_t threshold, hipStream_t stream)
    {
        k_set_threshold<<<1, 1, 0, stream>>>(a, b, threshold);
    }

    void LaunchResetMeasurements(const LatDesc* d_desc, const uint32_t n, hipStream_t stream)
    {
        k_reset_measurements<<<(n + 63u) / 64u, 64, 0, stream>>>(d_desc, n);
    }

    void LaunchPadBytes(uint8_t* dst, const uint8_t* src, const uint64_t np, const uint32_t n0v, const uint32_t pitch,
                        hipStream_t stream)
    {
        k_pad_bytes<<<static_cast<uint32_t>((np + 255) / 256), 256, 0, stream>>>(dst, src, np, n0v, pitch);
    }

    void LaunchUnpadLabels(uint32_t* dst, const uint32_t* src, const uint64_t n, const uint32_t n0v, const uint32_t pitch,
                           hipStream_t stream)
    {
        k_unpad_labels<<<static_cast<uint32_t>((n + 255) / 256), 256, 0, stream>>>(dst, src, n, n0v, pitch);
    }

    void LaunchHotStart(uint8_t* spins, const uint64_t n, const uint32_t spin_seed, const uint32_t n0v, const uint32_t pitch,
                        hipStream_t stream)
    {
        const uint64_t threads = (n + 63) / 64;
        k_hot_start<<<static_cast<uint32_t>((threads + 255) / 256), 256, 0, stream>>>(spins, n, spin_seed, n0v, pitch);
    }

    void LaunchCopy(const uint4* src, uint4* dst, const uint64_t n16, hipStream_t stream)
    {
        k_copy<<<2048, 256, 0, stream>>>(src, dst, n16);
    }
}
