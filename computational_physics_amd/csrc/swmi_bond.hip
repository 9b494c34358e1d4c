// swmi_bond.hip -- k_bond_label: bond activation and tile labelling (the first kernel of a sweep, see
// swmi_kernels.hip). Compiled once per SWMI_BOND_TW64 (64-wide tiles or narrow ones) and SWMI_BOND_MODE (a BondMode): the
// specialisations take most of the build and these parts build in parallel.
#include "swmi_device.h"

namespace swmi
{
    // =============================================================================================
    // k_bond_label
    // =============================================================================================
    // Per wavefront (tile) the rows are processed top to bottom with the loads of the next kCh rows in
    // flight together. Bonds are computed on wave-uniform 64-bit masks: S (spin up), U1/U2 (draw below
    // threshold), B (bond to the right neighbour inside the tile), D (bond to the site below).
    // 64-wide tiles keep the previous row's roots resolved in registers (Rp) and label a row with LabelRow64.
    // Narrow tiles record one union per overlap interval of consecutive rows in a per-wave LDS queue,
    // worked off 64 at a time whenever it fills.
    // Nodes of the LDS union-find are byte offsets into P. After the final find, the root of every
    // cluster that reaches the block edge carries kPFlag in its own entry, so a site's label (root index,
    // plus kEdgeFlag) is P[root] >> 2.
    // What bounds it: at 4096^2 (46.1 us, 10.5 B a site moved, 4.0 TB/s from the memory-side cache) the dependent
    // operations down a strip at eight waves per SIMD, with vector issue 50 %, the LDS pipe 48 % (a third of it bank
    // conflicts) and the scalar unit 37 % busy: 59.9 vector, 45.0 scalar and 15.7 LDS instructions per 64-site row (about 11
    // of the LDS ones in the row loop), where 81, 72 and 19.3 took 55.9 us; at 8192^2
    // (171 us, 4.1 TB/s) HBM, where a large copy reaches 5.0, and 14.6 B a site took 227; below 1024^2 the chain of LDS
    // round trips down a strip (256^2 9.6 us with 4-row strips, 14.7 with 16).
    // MODE: the sweep proper; the inspection build, in which bonds may be injected instead of generated and may be
    // recorded; or the labelling of an injected bond field alone.
    // PAD: the lattice is stored with a row pitch d.n0 above its width d.n0v; in the last tile column only
    // the lanes up to d.elast hold sites (mask d.vlast), the rest are padding: they bond to nothing, their
    // draws are unused, and the row's last site bonds across the lattice edge instead of lane tw - 1.
    // NW: waves of the workgroup, each with a strip of 4 * twr / NW wave rows of the block, at most TWR_MAX. Four
    // waves label a tile each; sixteen label a quarter tile each, which shortens the chain of dependent LDS
    // operations down a strip where a launch has too few blocks to fill the chip (LaunchBondLabelT).
    // FULL: every strip of every block has exactly TWR_MAX rows, so that the row counts are constants.
    template <uint32_t NW, uint32_t TWR_MAX, bool TW64, BondMode MODE, bool PAD, bool FULL>
    __device__ __forceinline__ void BondLabel(const LatDesc* __restrict__ descs, const uint32_t* __restrict__ block_lat,
                                              const uint32_t total_blocks)
    {
        // All loads of a chunk of rows are issued before its first store: on this hardware the memory
        // counter that a load waits on also counts the stores issued before it.
        constexpr bool DBG = MODE == BondMode::kInspect;
        constexpr uint32_t kCh = TWR_MAX < 16 ? TWR_MAX : 16;
        constexpr uint32_t kRows = TWR_MAX < 16 ? TWR_MAX : 16;   // rows resolved together at the end
        // 64-wide tiles of at most kRows rows keep their rows' roots in registers from the row loop to the labels
        constexpr bool kKeep = TW64 && TWR_MAX <= kRows;
        // and collect what the edges of the tile need as bits of scalar words
        constexpr bool kBits = kKeep && !DBG;
        constexpr uint32_t kSites = NW * TWR_MAX * 64;
        constexpr uint32_t kThreads = NW * 64u;
        constexpr uint32_t kQw = 128u;                             // per-wave LDS words of Q
        constexpr uint32_t kPFlag = 1u << 17;
        static_assert(kSites * 4u <= (1u << 16), "byte offsets must fit the 16-bit halves of a queue entry");
        static_assert((kPFlag >> 2) == kEdgeFlag, "a flagged root entry shifts into a flagged label");
        __shared__ uint32_t P[kSites];
        // per wave: 64-wide tiles keep the run minima of the current row in words 0-63 and give each lane a
        // word of its own in 64-127 (the target of LDS operations a lane has no use for, so that they need
        // no exec mask); narrow tiles keep their union queue here
        __shared__ uint32_t Q[NW * kQw];
        __shared__ uint32_t FB[2u * kSites / 32u];   // flip bits of a pending flip, by label index (root or qcap + slot)
        __shared__ uint64_t s_first_B[NW];
        // Numerical Recipes pairs (a << 32 | c: the loaded pair is the 64-bit addend of the multiply-add as it is) by
        // selector: words 0-7 one update, words 8-15 the jump from the stored states to this sweep's
        __shared__ __align__(128) uint64_t AC[16];
        __shared__ uint64_t s_right[NW == kWavesPerBlock ? 1u : kWavesPerBlock];   // bonds across the right edge, per tile
        __shared__ uint32_t s_nslot;            // slots given to the block's edge-reaching clusters

        const uint32_t b = RemapBlock(total_blocks);
        if (b >= total_blocks)
            return;
        if (threadIdx.x == 0)
            s_nslot = 0u;
        if (NW != kWavesPerBlock && threadIdx.x < kWavesPerBlock)
            s_right[threadIdx.x] = 0ull;
        const LatDesc& d = descs[LatticeOf(block_lat, b)];
        const Block bl = DecodeBlock(d, b);
        const uint32_t lane = threadIdx.x & 63u;
        const uint32_t lane4 = lane * 4u;
        const uint32_t w = Uniform(threadIdx.x >> 6);

        const uint32_t n0 = d.n0, n1 = d.n1, twr = FULL ? TWR_MAX : d.twr * kWavesPerBlock / NW;   // wave rows of a strip
        const uint32_t bnwr = FULL ? NW * TWR_MAX : bl.nwr;                                          // and of the block
        const uint32_t tw = TW64 ? 64u : d.tw, rpw = TW64 ? 1u : d.rpw;
        const uint32_t lx = lane & (tw - 1u);
        const uint32_t lrow = TW64 ? 0u : lane / tw;
        const uint32_t x = bl.sx * tw + lx;
        const bool lastcol = PAD && bl.sx + 1u == d.tiles_x;
        const uint64_t vmask = lastcol ? d.vlast : ~0ull;   // lanes that hold sites
        const uint32_t elane = lastcol ? d.elast : tw - 1u;  // lx of a lattice row's last site in this tile
        const bool rbound = lx == elane;
        const bool injected = MODE == BondMode::kLabel || (DBG && d.bond_in != nullptr);
        const uint32_t thr = d.threshold;
        const gptr<uint32_t> stp = Glob(d.state);
        const gptr<uint8_t> dump = DBG ? Glob(d.bond_dump) : nullptr;
        const gptr<uint8_t> spins = Glob(d.spins);
        const gptr<uint32_t> rotp = Glob(d.rot);
        const gptr<const uint8_t> bond_in = Glob(d.bond_in);

        const uint32_t r_begin = w * twr;
        const uint32_t nrow = FULL ? TWR_MAX : (bnwr > r_begin ? min(twr, bnwr - r_begin) : 0u);
        // buffer views of this block's part of the per-site arrays (row offsets in scalar registers, the lane
        // offset in a vector register, no per-row vector addresses)
        const uint32_t span = (bnwr - 1u) * bl.stride + 64u;   // sites from the block's first to its last
        const Rsrc rs_spins = MakeRsrc(d.spins + bl.base, span);
        const Rsrc rs_rng = MakeRsrc(d.rng + bl.base, span * 4u);
        const Rsrc rs_local = MakeRsrc(d.local + bl.base, span * 2u);
        const gptr<const uint32_t> fbits_g = Glob(static_cast<const uint32_t*>(d.fbits)) + bl.lb * d.fsw;
        const uint32_t nwaves = (bnwr + twr - 1u) / twr;
        const bool last_wave = w + 1u == nwaves;
        const uint32_t sx_r = bl.sx + 1u == d.tiles_x ? 0u : bl.sx + 1u;   // block column to the right
        const uint32_t sy_b = bl.sy + 1u == d.blocks_y ? 0u : bl.sy + 1u;   // block row below
        // the two sides of the halo array (by sweep parity)
        const gptr<const uint8_t> halo_s0 = Glob(static_cast<const uint8_t*>(d.halo));
        const gptr<const uint8_t> halo_s1 = halo_s0 + d.n_blocks * d.halo_stride;

        // Everything the block reads that needs only the descriptor is loaded together, before any of it is
        // used, so that the round trips overlap: the lattice's counters (read before this kernel stores any
        // state), the block's flip bits (they matter only under a pending flip: the edge-reaching clusters'
        // bits from k_resolve; before them in FB the rule words of the clusters inside the block, constant
        // under the parity rule) and every candidate for the spin below the tile (which one is used depends on
        // the counters). The descriptor fields these loads need are fetched first, in one batch, and the loads
        // carry no condition (in-range addresses, values unused where they do not apply), so that the compiler
        // neither fetches a field at its first use nor waits for every load at the end of a branch.
        HeldScalar(d.state);
        HeldScalar(d.aux);
        HeldScalar(d.fbits);
        HeldScalar(d.halo);
        HeldScalar(d.ecol_stride);
        HeldScalar(d.halo_stride);
        HeldScalar(d.qcap);
        HeldScalar(d.fsw);
        HeldScalar(d.n_blocks);
        const uint32_t it0 = injected ? 0u : stp[kStIteration];
        const uint32_t it_end = injected ? 0u : stp[kStItEnd];
        const uint32_t applied = injected ? 0u : stp[kStApplied];
        const uint32_t rng_it = injected ? 0u : Glob(static_cast<const uint32_t*>(d.aux))[kAuxRngIt];
        const uint32_t y_last = (bl.wyb + r_begin + (nrow > 0 ? nrow : 1u) - 1u) * rpw + lrow;
        const uint32_t y_below = nrow > 0 ? ((y_last + 1u == n1) ? 0u : y_last + 1u) : 0u;
        const uint32_t below = (r_begin + nrow) * bl.stride + lx;   // the site below the tile, inside the block
        const uint32_t below_halo = (sy_b * d.tiles_x + bl.sx) * d.halo_stride + d.ecol_stride + lx;
        const uint32_t hd_spin = MODE == BondMode::kLabel ? 0u : spins[y_below * n0 + x];
        // (the label-only pass over injected bonds has no flip bits and no halos: those loads belong to the sweep,
        // where `injected` is false at compile time)
        uint32_t fbw = 0, hd_lab = 0, hd_sv = 0, hd_h0 = 0, hd_h1 = 0;
        if (!injected)
        {
            // fsw <= 256: a block has at most 2 * 64 + 2 * kWavesPerBlock * 64 boundary sites, 4 * edge_cap / 32
            // words of slots (the engine checks the bound), so one word per thread
            fbw = fbits_g[min(static_cast<uint32_t>(threadIdx.x), d.fsw - 1u)];
            hd_lab = __builtin_amdgcn_raw_buffer_load_b16(rs_local, below * 2u, 0, 0);
            hd_sv = __builtin_amdgcn_raw_buffer_load_b8(rs_spins, below, 0, 0);
            hd_h0 = halo_s0[below_halo];
            hd_h1 = halo_s1[below_halo];
            Issued(fbw);   // not sunk into the branch that stores it
        }

        // sweep schedule: a lattice past its last sweep is left alone by the whole sweep
        const bool act = injected || it0 < it_end;
        if (bl.lb == 0 && threadIdx.x == 0)
        {
            stp[kStActive] = act ? 1u : 0u;
            if (act)
                Glob(d.aux)[kAuxWholeLabels] = 0u;
            if (act && d.flip_rule != 0u)
                stp[kStFlipKey] = FlipKey(d.seed, it0);   // an inactive lattice keeps the key of its pending flip
            if (act && !injected)
                stp[kStHaloSide] = (it0 >> 1) & 1u;
        }
        if (!act)
            return;
        // The previous sweep's flip is still pending (applied != iteration): it is applied here, each site
        // as it is loaded, from its label and the block's flip bits; the flipped spins are stored as the
        // rows are processed. That flip belongs to the sweep that started at iteration it0 - 2.
        const bool pending = !injected && applied != it0;
        const uint32_t it1 = it0 + 1u;
        const uint32_t it2 = it1 + 1u;
        const bool rot1 = !injected && (it1 % 15u == 0u);
        const bool rot2 = !injected && (it2 % 15u == 0u);
        // The stored states are those of iteration rng_it: a lane's (a, c) stays the same until the next rotation,
        // so the state after the sweep's first update is one affine step away, u1 = A st + C with (A, C) the pair
        // applied it1 - rng_it times, and the sweep needs to store no state. A rotating sweep stores the state at
        // which the pairs change (it0, or it1 when the second update rotates): at most 15 updates are jumped. Both
        // updates rotate only in the sweep in which the 32-bit update count wraps (2^32 - 1 is a multiple of 15).
        const uint32_t n_jump = min((rot1 ? it0 : it1) - rng_it, 15u);

        // halos: this sweep writes the block's first column and first wave row into its side of the halo
        // array; the other side holds the neighbours' flipped halos of the pending flip
        const uint32_t hside = (it0 >> 1) & 1u;
        const gptr<const uint8_t> halo_g = hside ? halo_s0 : halo_s1;
        const Rsrc rs_halo = MakeRsrc(d.halo + (hside * d.n_blocks + bl.lb) * d.halo_stride, d.halo_stride);
        const uint32_t hcol_off = (lx == 0u && !injected) ? lrow : kNoStore;   // first column: one lane per lattice row
        uint32_t* const Qw = Q + w * kQw;
        uint32_t* const Pl = At(P, lane4);   // this lane's entry of wave row 0
        uint32_t* const dummy = Qw + 64u + lane;
        const uint32_t run_words = OffsetFrom(P, Qw), spare = OffsetFrom(P, dummy);
        // a full queue (>= 64 entries) is worked off right away; the tail moves to the front
        const auto drain64 = [&](uint32_t& qlen) {
            const uint32_t e = Qw[lane];
            LdsUnionLockstep(P, e >> 16, e & 0xFFFFu);
            const uint32_t rem = qlen - 64u;
            const uint32_t t = Qw[64u + lane];
            if (lane < rem)
                Qw[lane] = t;
            qlen = rem;
        };

        // lane masks: first column of a lattice row, lanes with a right neighbour inside the wave row,
        // lanes whose down neighbour sits in the same wave row
        uint64_t rowstart = 1;
        if (!TW64)
            for (uint32_t j = tw; j < 64u; j += tw)
                rowstart |= 1ull << j;
        const uint64_t redge = rowstart << elane;   // the last site of every lattice row of the wave row
        const uint64_t in_right = PAD ? (vmask & ~redge) : ~redge;
        const uint64_t low = TW64 ? 0ull : ((1ull << (64u - tw)) - 1ull);
        const uint64_t lanes_below = (1ull << lane) - 1ull;

        // pending flip: the block's flip bits (loaded into FB above), one per label index (k_resolve wrote the
        // bit of every cluster: by root index, or by qcap + slot for an edge-reaching one), so a site's flip is
        // the bit at its label's index
        const uint32_t ac_at = static_cast<uint32_t>(reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) uint64_t*)AC));
        // the pair of the selector bits ks of a spin byte, in half `first` of AC (AC's alignment makes the sum an or)
        const auto pair_of = [&](const uint32_t ks, const uint32_t first) {
            static_assert(kSelMask == 7u * sizeof(uint64_t), "the selector bits are a byte offset into AC");
            return ((__attribute__((address_space(3))) const uint64_t*)static_cast<uintptr_t>(ac_at | ks))[first];
        };
        const auto flip_of = [&](const uint32_t lab) { return (LdsLoad(&FB[(lab & 0x7FFFu) >> 5]) >> (lab & 31u)) & 1u; };

        // spins below the tile (down halo), needed last but fetched first. Under a pending flip, below the
        // block the neighbour's halo holds the flipped spin; inside the block the spin and label of the site
        // below are carried across the barrier in the lane's spare LDS word (writing them there needs the
        // loaded values, so these loads complete before the wave that owns the site may store its flipped
        // spin) and flipped after it, with the block's flip bits.
        uint32_t halo_down = 0;
        const bool carry = nrow > 0 && pending && !last_wave;
        // The block's flip bits and rule words, the carried site below and the barrier that publishes them: run
        // by every wave after the loads of its first chunk of rows are issued, so that this work and the
        // barrier overlap their round trip.
        const auto meet = [&]() {
            if (!injected)
            {
                if (threadIdx.x < 8u)
                {
                    uint32_t a, c, ja = 1u, jc = 0u;
                    ParamsOf(threadIdx.x, a, c);
                    for (uint32_t i = 0; i < n_jump; ++i)
                    {
                        ja *= a;
                        jc = a * jc + c;
                    }
                    AC[threadIdx.x] = (static_cast<uint64_t>(a) << 32) | c;
                    AC[8u + threadIdx.x] = (static_cast<uint64_t>(ja) << 32) | jc;
                }
                if (threadIdx.x < d.fsw)
                    FB[d.qcap / 32u + threadIdx.x] = fbw;
                if (d.flip_rule == 0u)
                    for (uint32_t i = threadIdx.x; i < bnwr * 2u; i += kThreads)   // bl.nwr * 64 root indices, 32 per word
                        FB[i] = RuleWord(d, bl, i, false, 0u);
                else if (pending)   // the random rule's words, with the key of the pending flip's sweep
                    for (uint32_t i = threadIdx.x; i < bnwr * 2u; i += kThreads)
                        FB[i] = RuleWord(d, bl, i, true, FlipKey(d.seed, it0 - 2u));
            }
            if (nrow > 0)
            {
                if (!pending)
                    halo_down = hd_spin;
                else if (carry)
                    __hip_atomic_store(dummy, (hd_lab << 8) | (hd_sv & 0xFFu), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
                else
                    halo_down = hside ? hd_h0 : hd_h1;
            }
            __syncthreads();   // AC, FB, the carried site below
            if (carry)
            {
                const uint32_t v = LdsLoad(dummy);
                const uint32_t lab = v >> 8;
                halo_down = (v & 0xFFu) ^ flip_of(lab);
            }
        };

        uint64_t last_B = 0, last_D = 0, down_bits = 0, right_bits = 0;
        uint32_t qlen = 0;
        uint32_t Rp = 0;   // 64-wide tiles: root of this lane's site in the previous row
        uint32_t Rk[kKeep ? kRows / 2u + 1u : 1u];   // the rows' roots as they were labelled, two to a word
        if (TW64)
            Qw[lane] = 0u;   // run words of LabelRow64
        uint64_t prev_S = 0, prev_U2 = 0, prev_B = 0, prev_Ball = 0;
        uint32_t prev_site = 0;
        uint32_t colv = 0;   // 64-wide tiles: lane r collects the first-column spin of row r
        // kBits: the rows' first-column spin, last-column spin and last-column draw, the latest row in bit 0, and the
        // spins right of the tile (lane r: row r)
        uint32_t col_b = 0, s63_b = 0, u63_b = 0, hright = 0;
        const auto last_bit = [&](const uint64_t m) { return static_cast<uint32_t>(PAD ? (m >> elane) & 1ull : m >> 63); };
        {
            // the chunk loop exists twice: sweeps without a group rotation (13 in 15) carry no rotation code
            // (and twice more for the sweeps that apply a pending flip on load, the rule after any sweep)
            const auto chunks = [&](auto rotating, auto flipping) {
            constexpr bool kRot = decltype(rotating)::value;
            constexpr bool kPend = decltype(flipping)::value;
            // rows loaded together: a flip on load also keeps the labels in flight, so at most eight
            constexpr uint32_t kC = kPend && kCh > 8u ? kCh / 2u : kCh;
            // what one chunk of rows loads per lane: the spin byte, the lcg32 state and, under a pending flip,
            // the label of its site in each row; one right-halo spin and one rotation offset per row (lane i:
            // row r0 + i of the chunk)
            struct Chunk
            {
                uint32_t sp[kC], aux[kC], lab[kC], h, g_rot;
            };
            // The loads carry no condition (rows past the tile re-read its last row, values unused), so that
            // they issue back to back and their latencies overlap.
            const auto load = [&](const uint32_t r0, Chunk& c) {
                const uint32_t lrow_ch = r_begin + min(r0 + (lane % kC), nrow - 1u);
                // right halo of a 64-wide tile: under a pending flip the right neighbour's flipped first column
                c.h = 0;
                if (TW64 && !kBits)
                    c.h = pending ? halo_g[(bl.sy * d.tiles_x + sx_r) * d.halo_stride + lrow_ch]
                                  : spins[(bl.wyb + lrow_ch) * n0 + sx_r * 64u];
                // rotation offsets of the chunk's groups, needed on rotating sweeps only
                c.g_rot = kRot ? rotp[(bl.base + lrow_ch * bl.stride) >> 6] : 0u;
#pragma unroll
                for (uint32_t i = 0; i < kC; ++i)
                {
                    // row base in scalar registers, the lane offset in a vector register
                    const uint32_t wr = r_begin + min(r0 + i, nrow - 1u);
                    const uint32_t rowoff = Uniform(wr * bl.stride);
                    c.sp[i] = __builtin_amdgcn_raw_buffer_load_b8(rs_spins, lane, rowoff, 0);
                    c.aux[i] = injected ? (bond_in + bl.base + rowoff)[lane] : __builtin_amdgcn_raw_buffer_load_b32(rs_rng, lane4, rowoff * 4u, 0);
                    c.lab[i] = kPend ? __builtin_amdgcn_raw_buffer_load_b16(rs_local, lane * 2u, rowoff * 2u, 0) : 0u;
                }
            };
            const auto process = [&](const uint32_t r0, auto rc_t, Chunk& c) {
                constexpr uint32_t rc = decltype(rc_t)::value;   // r0 where the rows' roots are kept
                uint32_t(&sp)[kC] = c.sp;
                const uint32_t(&aux)[kC] = c.aux;
                const uint32_t(&lab)[kC] = c.lab;
                const uint32_t h = c.h, g_rot = c.g_rot;
                if (kPend)
                {
#pragma unroll
                    for (uint32_t i = 0; i < kC; ++i)
                        sp[i] ^= flip_of(lab[i]);
                }
                const uint64_t HR = TW64 && !kBits ? __ballot((h & 1u) != 0u) : 0ull;

#pragma unroll
                for (uint32_t i = 0; i < kC; ++i)
                {
                    const uint32_t r = r0 + i;
                    if (r < nrow)
                    {
                        const uint32_t wr = r_begin + r;
                        const uint32_t site = bl.base + wr * bl.stride + lane;
                        const uint64_t S = __ballot((sp[i] & 1u) != 0u);
                        if (kBits)
                        {
                            col_b = (col_b << 1) + (static_cast<uint32_t>(S) & 1u);
                            s63_b = (s63_b << 1) + last_bit(S);
                        }
                        else if (TW64)
                            colv = LaneBit(1ull << r) ? static_cast<uint32_t>(S) : colv;   // bit 0 of S: lane 0's spin
                        else
                            __builtin_amdgcn_raw_buffer_store_b8(static_cast<uint8_t>(sp[i] & 1u), rs_halo, hcol_off, wr * rpw, 0);
                        if (r == 0 && r_begin == 0u && !injected)
                            __builtin_amdgcn_raw_buffer_store_b8(static_cast<uint8_t>(sp[i] & 1u), rs_halo, d.ecol_stride + lane, 0, 0);
                        uint64_t Ball, U2;
                        if (!injected)
                        {
                            // two LCG32_State<64>::Update of the group of this wave row
                            // (random/src/lcg32.cpp:51-84); a rotation by `shift` moves lane
                            // (i + shift) & 63's selector to lane i
                            uint32_t ks = sp[i] & kSelMask, shift = 0;
                            const uint64_t jump = pair_of(ks, 8u);
                            uint64_t ac = pair_of(ks, 0u);
                            uint32_t u1 = static_cast<uint32_t>(jump >> 32) * aux[i] + static_cast<uint32_t>(jump);
                            if (kRot)
                            {
                                // the state jumped to is the one the rotation works on and the one stored
                                __builtin_amdgcn_raw_buffer_store_b32(u1, rs_rng, lane4, Uniform(wr * bl.stride) * 4u, 0);
                                shift = ShuffleShift(u1, rot1 ? it1 : it2) & 63u;
                                ks = static_cast<uint32_t>(__shfl(static_cast<int>(ks), static_cast<int>((lane + shift) & 63u)));
                                ac = pair_of(ks, 0u);
                                if (rot1)
                                    u1 = static_cast<uint32_t>(ac >> 32) * u1 + static_cast<uint32_t>(ac);
                                if (rot1 && rot2)   // the sweep in which the update count wraps to 0
                                {
                                    __builtin_amdgcn_raw_buffer_store_b32(u1, rs_rng, lane4, Uniform(wr * bl.stride) * 4u, 0);
                                    const uint32_t second = ShuffleShift(u1, it2) & 63u;
                                    ks = static_cast<uint32_t>(__shfl(static_cast<int>(ks), static_cast<int>((lane + second) & 63u)));
                                    ac = pair_of(ks, 0u);
                                    shift += second;
                                }
                            }
                            const uint32_t st = static_cast<uint32_t>(ac >> 32) * u1 + static_cast<uint32_t>(ac);
                            if (kRot)
                            {
                                spins[site] = static_cast<uint8_t>((sp[i] & 1u) | ks);
                                if (lane == 0)
                                    rotp[site >> 6] = (ReadLane(g_rot, i) + shift) & 63u;
                            }
                            else if (kPend)
                                __builtin_amdgcn_raw_buffer_store_b8(static_cast<uint8_t>(sp[i]), rs_spins, lane, Uniform(wr * bl.stride), 0);
                            const uint64_t U1 = __ballot(u1 < thr);
                            U2 = __ballot(st < thr);
                            // right neighbour's spin: next lane, or for a row's last site the halo (64-wide
                            // tiles) or the first column of the same lattice row (narrow tiles: one tile
                            // column)
                            uint64_t RS;
                            if (kBits)
                            {
                                RS = S >> 1;   // the last column's bond follows after the rows
                                u63_b = (u63_b << 1) + last_bit(U1);
                            }
                            else if (!PAD)
                                RS = TW64 ? ((S >> 1) | (((HR >> i) & 1ull) << 63))
                                          : (((S >> 1) & in_right) | ((S << (tw - 1u)) & ~in_right));
                            else
                                RS = TW64 ? (((S >> 1) & ~redge) | (((HR >> i) & 1ull) << elane))
                                          : (((S >> 1) & ~redge) | ((S << elane) & redge));
                            Ball = ~(S ^ RS) & U1;
                        }
                        else
                        {
                            Ball = __ballot((aux[i] & 1u) != 0u);
                            U2 = __ballot((aux[i] & 2u) != 0u);
                            if (kBits)
                                u63_b = (u63_b << 1) + last_bit(Ball);
                        }
                        if (PAD)
                        {
                            Ball &= vmask;
                            U2 &= vmask;
                        }
                        const uint64_t B = Ball & in_right;
                        const uint64_t edge = Ball & redge;
                        if (kBits)
                        {
                        }
                        else if (TW64)
                            right_bits |= (PAD ? ((edge >> elane) & 1ull) : (edge >> 63)) << r;
                        else
                            for (uint32_t j = 0; j < rpw; ++j)
                                right_bits |= ((edge >> (j * tw + elane)) & 1ull) << (r * rpw + j);
                        if (r == 0)
                            s_first_B[w] = B;

                        const uint32_t row_b = wr * 256u;   // byte offset of the wave row in P
                        if (TW64)
                        {
                            const uint64_t D = r == 0 ? 0ull : (injected ? prev_U2 : (~(prev_S ^ S) & prev_U2));
                            if (dump && r > 0)
                                dump[prev_site] = static_cast<uint8_t>((LaneBit(prev_Ball) ? 1u : 0u) | (LaneBit(D) ? 2u : 0u));
                            Rp = LabelRow64(P, run_words, spare, row_b + lane4, B, D, Rp, RowBase(r + 1u));
                            if (kKeep)
                            {
                                if (i % 2u == 0u)
                                    Rk[(rc + i) / 2u] = Rp;
                                else
                                    Rk[(rc + i) / 2u] |= Rp << 16;
                            }
                        }
                        else
                        {
                            // every site starts under the first site of its row run
                            const uint64_t below = ~B & lanes_below;
                            const uint32_t run_start = below ? 64u - static_cast<uint32_t>(__clzll(below)) : 0u;
                            *At(Pl, row_b) = row_b + run_start * 4u;
                            if (r > 0)
                            {
                                // bonds of the previous wave row to the row below: queue one union per overlap
                                // interval
                                const uint64_t SD = (Shr(prev_S, tw) & low) | Shl(S, 64u - tw);
                                const uint64_t D = injected ? prev_U2 : (~(prev_S ^ SD) & prev_U2);
                                const uint64_t tgtB = Shr(prev_B, tw) | Shl(B, 64u - tw);
                                const uint64_t K = FirstBondPerInterval(D, prev_B & tgtB, rowstart);
                                if (LaneBit(K))
                                {
                                    const uint32_t top = row_b - 256u + lane4;
                                    const uint32_t bot = (lane < 64u - tw) ? top + tw * 4u : row_b + lane4 - (64u - tw) * 4u;
                                    const uint32_t pos = qlen + __builtin_amdgcn_mbcnt_hi(static_cast<uint32_t>(K >> 32),
                                                                                         __builtin_amdgcn_mbcnt_lo(static_cast<uint32_t>(K), 0u));
                                    Qw[pos] = (top << 16) | bot;
                                }
                                qlen += static_cast<uint32_t>(__popcll(K));
                                if (qlen >= 64u)
                                    drain64(qlen);
                                if (dump)
                                    dump[prev_site] = static_cast<uint8_t>((LaneBit(prev_Ball) ? 1u : 0u) | (LaneBit(D) ? 2u : 0u));
                            }
                        }
                        if (kBits)   // the three words take this row's bits here (the compiler would keep every row's masks)
                        {
                            col_b = Uniform(col_b);
                            s63_b = Uniform(s63_b);
                            u63_b = Uniform(u63_b);
                            asm volatile("" : "+s"(col_b), "+s"(s63_b), "+s"(u63_b));
                        }
                        prev_S = S;
                        prev_U2 = U2;
                        prev_B = B;
                        prev_Ball = Ball;
                        prev_site = site;
                    }
                }
            };
            // a tile of at most kC rows is one chunk, starting at row 0; the first chunk's loads go out before
            // the barrier (a wave without rows loads nothing and only meets the others there)
            Chunk c0;
            if (nrow > 0)
                load(0u, c0);
            if (kBits && MODE != BondMode::kLabel && nrow > 0)
            {
                // right halo of the tile's rows: under a pending flip the right neighbour's flipped first column
                const uint32_t lr = r_begin + min(lane, nrow - 1u);
                hright = kPend ? halo_g[(bl.sy * d.tiles_x + sx_r) * d.halo_stride + lr] : spins[(bl.wyb + lr) * n0 + sx_r * 64u];
            }
            meet();
            if (nrow == 0)
                return;
            process(0u, std::integral_constant<uint32_t, 0>{}, c0);
            if constexpr (kKeep)
            {
                // (a chunk has kC = kRows or kRows / 2 rows: at most one more, at a row known here)
                if (TWR_MAX > kC && nrow > kC)
                {
                    Chunk c;
                    load(kC, c);
                    process(kC, std::integral_constant<uint32_t, TWR_MAX <= kC ? 0u : kC>{}, c);
                }
            }
            else
                for (uint32_t r0 = kC; r0 < (TWR_MAX <= kC ? 0u : nrow); r0 += kC)
                {
                    Chunk c;
                    load(r0, c);
                    process(r0, std::integral_constant<uint32_t, 0>{}, c);
                }
            };
            if (rot1 || rot2)
            {
                if (pending)
                    chunks(std::true_type{}, std::true_type{});
                else
                    chunks(std::true_type{}, std::false_type{});
            }
            else if (pending)
                chunks(std::false_type{}, std::true_type{});
            else
                chunks(std::false_type{}, std::false_type{});
        }
        if (nrow > 0)
        {
            if (kBits)
            {
                // row r of the words is bit nrow - 1 - r
                const uint32_t up = 32u - nrow;   // (nrow is 1 to 16)
                const uint32_t h = static_cast<uint32_t>(__ballot((hright & 1u) != 0u));
                right_bits = (MODE == BondMode::kLabel ? ~0u : ~((__brev(s63_b) >> up) ^ h)) & (__brev(u63_b) >> up);
                colv = (__brev(col_b) >> up) >> (lane & 31u);
            }
            if (NW != kWavesPerBlock && lane == 0u && right_bits != 0ull)   // read after the last barrier
                (void)__hip_atomic_fetch_or(&s_right[r_begin / d.twr], right_bits << (r_begin % d.twr), __ATOMIC_RELAXED,
                                            __HIP_MEMORY_SCOPE_WORKGROUP);
            if (TW64 && !injected)   // first column of the tile's rows (rpw == 1): one store per wave
                __builtin_amdgcn_raw_buffer_store_b8(static_cast<uint8_t>(colv & 1u), rs_halo, lane < nrow ? r_begin + lane : kNoStore, 0, 0);

            // bonds out of the last wave row: into the same wave row (tw < 64), into the next tile of the
            // block, or across the block edge
            {
                const uint32_t wr = r_begin + nrow - 1u;
                // halo spins arrive in the lanes that need them (lanes >= 64 - tw)
                const uint64_t H = __ballot((halo_down & 1u) != 0u);
                const uint64_t SD = TW64 ? H : ((Shr(prev_S, tw) & low) | (H & ~low));
                const uint64_t D = injected ? prev_U2 : (~(prev_S ^ SD) & prev_U2);
                if (!TW64)
                {
                    const uint64_t Din = D & low;
                    const uint64_t K = FirstBondPerInterval(Din, prev_B & Shr(prev_B, tw), rowstart);
                    if (LaneBit(K))
                    {
                        const uint32_t pos = qlen + __builtin_amdgcn_mbcnt_hi(static_cast<uint32_t>(K >> 32),
                                                                             __builtin_amdgcn_mbcnt_lo(static_cast<uint32_t>(K), 0u));
                        const uint32_t top = wr * 256u + lane4;
                        Qw[pos] = (top << 16) | (top + tw * 4u);
                    }
                    qlen += static_cast<uint32_t>(__popcll(K));
                    if (qlen >= 64u)
                        drain64(qlen);
                }
                if (dump)
                    dump[prev_site] = static_cast<uint8_t>((LaneBit(prev_Ball) ? 1u : 0u) | (LaneBit(D) ? 2u : 0u));
                last_B = prev_B;
                if (last_wave)
                    down_bits = D & ~low;
                else
                    last_D = D & ~low;
            }

            // the rest of the queued unions of this tile (fewer than 64)
            if (!TW64 && qlen > 0)
            {
                const uint32_t e = (lane < qlen) ? Qw[lane] : 0u;
                LdsUnionLockstep(P, e >> 16, e & 0xFFFFu);
            }
        }
        __syncthreads();

        // unions across the tile edges inside the block
        if (nrow > 0 && !last_wave)
        {
            const uint32_t wr = r_begin + nrow - 1u;
            const uint64_t Bbot = s_first_B[w + 1u];
            const uint64_t tgtB = TW64 ? Bbot : Shl(Bbot, 64u - tw);
            const bool go = LaneBit(FirstBondPerInterval(last_D, last_B & tgtB, rowstart));
            const uint32_t top = wr * 256u + lane4;
            // (64-wide tiles: from the root the last row was labelled with)
            LdsUnionLockstep(P, go ? (TW64 ? Rp : top) : 0u, go ? top + 256u - (64u - tw) * 4u : 0u);
        }
        __syncthreads();

        const uint32_t qcap = d.qcap, bslots = kWavesPerBlock * d.edge_cap;
        const Rsrc rs_cpar = MakeRsrc(d.cpar + bslots * bl.lb, bslots * 8u);
        const Rsrc rs_ecol = MakeRsrc(d.ecol + 2u * bl.lb * d.ecol_stride, 8u * d.ecol_stride);
        const Rsrc rs_erow = MakeRsrc(d.erow + 2u * 64u * bl.lb, 2u * 64u * 4u);

        // Edge marks: the lanes of m[k] flag their root[k], a site on the block edge (lanes off the edge flag their own
        // word of Q). The marks of the K vectors are issued together and return the root's entry as it was: the lane
        // that found it unflagged (the cluster's first mark) gives the cluster the next slot of the block (one LDS
        // counter, one addition per wave), writes the slot's union-find entry (a root keyed by the root's site) and
        // makes the root's entry in P kPFlag | (qcap + slot) << 2, so that after the barrier every site of the cluster
        // reads the label 0x8000 | (qcap + slot). A block has at most as many edge roots as boundary sites, within its
        // slot capacity; more would be a broken invariant, reported through the error flag.
        const auto mark = [&](const auto& root, const auto& m, const auto K_t) {
            constexpr uint32_t K = decltype(K_t)::value;
            uint32_t old[K];
            uint64_t F[K];
            uint32_t total = 0;
#pragma unroll
            for (uint32_t k = 0; k < K; ++k)
            {
                const uint32_t o = __hip_atomic_fetch_or(LaneBit(m[k]) ? At(P, root[k]) : dummy, kPFlag, __ATOMIC_RELAXED,
                                                         __HIP_MEMORY_SCOPE_WORKGROUP);
                old[k] = LaneBit(m[k]) ? o : kPFlag;
            }
#pragma unroll
            for (uint32_t k = 0; k < K; ++k)
            {
                F[k] = __ballot(old[k] < kPFlag);
                total += static_cast<uint32_t>(__popcll(F[k]));
            }
            if (total == 0u)
                return;
            uint32_t base = 0;
            if (lane == 0u)
                base = __hip_atomic_fetch_add(&s_nslot, total, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
            base = __builtin_amdgcn_readfirstlane(base);
#pragma unroll
            for (uint32_t k = 0; k < K; ++k)
            {
                const bool first = LaneBit(F[k]);
                const uint32_t pos = base + __builtin_amdgcn_mbcnt_hi(static_cast<uint32_t>(F[k] >> 32),
                                                                      __builtin_amdgcn_mbcnt_lo(static_cast<uint32_t>(F[k]), 0u));
                __hip_atomic_store(first ? At(P, root[k]) : dummy, kPFlag | ((qcap + min(pos, bslots - 1u)) << 2), __ATOMIC_RELAXED,
                                   __HIP_MEMORY_SCOPE_WORKGROUP);
                const u32x2 entry = {bslots * bl.lb + pos, SiteOf(bl.base, bl.stride, root[k] >> 2)};   // (site << 32) | slot
                __builtin_amdgcn_raw_buffer_store_b64(entry, rs_cpar, first ? pos * 8u : kNoStore, 0, 0);
                base += static_cast<uint32_t>(__popcll(F[k]));
            }
        };

        if constexpr (kKeep)
        {
            // Every site's block-local root, from the rows' roots as they were labelled, all rows of the tile in flight,
            // and the root of one more site per lane: lane i < kRows row i's first column, lane kRows + i its last, so
            // that one vector holds what the rows need for the block's edge columns.
            constexpr uint32_t kSide = kRows;
            const uint32_t srow = lane % kSide;
            const bool sides = lane < 2u * kSide && srow < nrow;
            uint32_t xs[kRows], xside = 0;
            if (nrow > 0u)
            {
#pragma unroll
                for (uint32_t i = 0; i < kRows; ++i)
                    xs[i] = i < nrow ? (i % 2u == 0u ? Rk[i / 2u] & 0xFFFFu : Rk[i / 2u] >> 16) : r_begin * 256u;
                xside = (r_begin + (sides ? srow : 0u)) * 256u + (sides && lane >= kSide ? elane * 4u : 0u);
                // two steps per round; a round ends the chase once a step moved no lane of any row. The differences are
                // summed in vector registers (17 values below 2^17 cannot wrap to zero). Parents only decrease, so a
                // chase ends within kSites steps; more rounds mean a broken forest, which is reported instead of
                // followed.
                for (uint32_t round = 0;; ++round)
                {
                    if (round * 2u > kSites)
                    {
                        if (lane == 0)
                            (void)__hip_atomic_fetch_or(stp + kStErr, kErrLabelRange, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                        break;
                    }
                    uint32_t ys[kRows];
                    const uint32_t yside = LdsLoad(At(P, xside));
                    uint32_t moved = yside ^ xside;
#pragma unroll
                    for (uint32_t i = 0; i < kRows; ++i)
                    {
                        ys[i] = LdsLoad(At(P, xs[i]));
                        moved += ys[i] ^ xs[i];
                    }
                    if (!__ballot(moved != 0u))
                        break;
                    xside = LdsLoad(At(P, yside));
                    moved = xside ^ yside;
#pragma unroll
                    for (uint32_t i = 0; i < kRows; ++i)
                    {
                        xs[i] = LdsLoad(At(P, ys[i]));
                        moved += xs[i] ^ ys[i];
                    }
                    if (!__ballot(moved != 0u))
                        break;
                }
            }
            __syncthreads();   // no chase may meet a flagged entry
            uint32_t xlast = xs[0];   // root in the tile's last row
#pragma unroll
            for (uint32_t i = 1; i < kRows; ++i)
                xlast = i + 1u == nrow ? xs[i] : xlast;
            if (nrow > 0u)
            {
                const uint32_t root[3] = {xside, xs[0], xlast};
                const uint64_t m[3] = {__ballot(sides), r_begin == 0u ? vmask : 0ull, last_wave ? vmask : 0ull};
                mark(root, m, std::integral_constant<uint32_t, 3>{});
            }
            __syncthreads();   // every slot label in place

            // labels out: the block-local labels, and (label << 16) | root index of the block's first and last column and
            // first and last wave row for the merge and the halo flips. The outputs go through buffer views of this
            // block's part of each array; a lane with nothing to store gets an offset past the view, and the hardware
            // drops that store (no exec mask).
            if (nrow > 0u)
            {
                const auto entry = [&](const uint32_t root) { return ((LdsLoad(At(P, root)) >> 2) << 16) | (root >> 2); };
                const auto emit = [&](auto full_t) {
                    constexpr bool kFull = decltype(full_t)::value;
#pragma unroll
                    for (uint32_t i = 0; i < kRows; ++i)
                        if (kFull || i < nrow)
                            __builtin_amdgcn_raw_buffer_store_b16(static_cast<uint16_t>(LdsLoad(At(P, xs[i])) >> 2), rs_local, lane * 2u,
                                                                  (r_begin + i) * bl.stride * 2u, 0);
                };
                if (nrow == kRows)
                    emit(std::true_type{});
                else
                    emit(std::false_type{});
                __builtin_amdgcn_raw_buffer_store_b32(entry(xside), rs_ecol,
                                                      sides ? ((lane >= kSide ? d.ecol_stride : 0u) + r_begin + srow) * 4u : kNoStore, 0, 0);
                if (r_begin == 0u)
                    __builtin_amdgcn_raw_buffer_store_b32(entry(xs[0]), rs_erow, lane4, 0, 0);
                if (last_wave)
                    __builtin_amdgcn_raw_buffer_store_b32(entry(xlast), rs_erow, lane4, 256u, 0);
            }
        }
        else
        {
            // every site's block-local root (kRows chases in flight per lane). A tile of at most kRows rows
            // keeps its roots in registers; taller tiles write them back into P.
            const bool one_chunk = TWR_MAX <= kRows || nrow <= kRows;
            uint32_t xs[kRows];
            // (a wave of a partial block may own no rows: its part of P was never written and is not chased)
            for (uint32_t r0 = 0; r0 < (TWR_MAX <= kRows ? (nrow > 0 ? 1u : 0u) : nrow); r0 += kRows)
            {
#pragma unroll
                for (uint32_t i = 0; i < kRows; ++i)
                    xs[i] = (r_begin + ((r0 + i < nrow) ? r0 + i : r0)) * 256u + lane4;
                // two steps per round; a round ends the chase once a step moved no lane of any row. The
                // differences are summed in vector registers (16 values below 2^17 cannot wrap to zero). Parents
                // only decrease, so a chase ends within kSites steps; more rounds mean a broken forest, which is
                // reported instead of followed.
                for (uint32_t round = 0;; ++round)
                {
                    if (round * 2u > kSites)
                    {
                        if (lane == 0)
                            (void)__hip_atomic_fetch_or(stp + kStErr, kErrLabelRange, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                        break;
                    }
                    uint32_t ys[kRows];
                    uint32_t moved = 0;
#pragma unroll
                    for (uint32_t i = 0; i < kRows; ++i)
                    {
                        ys[i] = LdsLoad(At(P, xs[i]));
                        moved += ys[i] ^ xs[i];
                    }
                    if (!__ballot(moved != 0u))
                        break;
                    moved = 0;
#pragma unroll
                    for (uint32_t i = 0; i < kRows; ++i)
                    {
                        xs[i] = LdsLoad(At(P, ys[i]));
                        moved += xs[i] ^ ys[i];
                    }
                    if (!__ballot(moved != 0u))
                        break;
                }
                if (!one_chunk)
                {
#pragma unroll
                    for (uint32_t i = 0; i < kRows; ++i)
                        if (r0 + i < nrow)
                            *At(Pl, (r_begin + r0 + i) * 256u) = xs[i];
                }
            }
            // (taller tiles: a flagged entry is a root's own, first flagged by the edge marks, later holding its
            // slot label; either way the site is its own root)
            const auto root_of = [&](const uint32_t r) {
                if (one_chunk)
                    return xs[r];
                const uint32_t v = LdsLoad(At(Pl, (r_begin + r) * 256u));
                return v >= kPFlag ? (r_begin + r) * 256u + lane4 : v;
            };
            __syncthreads();   // no chase may meet a flagged entry

            // Sites on the block edge flag their root: the edge lanes of a row are `side`, plus every lane of the block's first
            // and last lattice rows.
            const uint64_t side = TW64 ? (PAD ? (1ull | (1ull << elane)) : 0x8000000000000001ull) : __ballot(lx == 0 || rbound);
            const uint64_t top_first = r_begin == 0 ? (TW64 ? vmask : (__ballot(lrow == 0) & vmask)) : 0ull;
            const uint64_t bottom_last = last_wave ? (TW64 ? vmask : (__ballot(lrow == rpw - 1u) & vmask)) : 0ull;
            const auto mark_rows = [&](auto full_t, const uint32_t r0) {
                constexpr bool kFull = decltype(full_t)::value;
                uint32_t root[kRows];
                uint64_t m[kRows];
#pragma unroll
                for (uint32_t i = 0; i < kRows; ++i)
                {
                    const uint32_t r = r0 + i;
                    root[i] = 0u;
                    m[i] = 0ull;
                    if (kFull || r < nrow)
                    {
                        m[i] = side | (r == 0u ? top_first : 0ull) | ((kFull ? i + 1u == kRows : r + 1u == nrow) ? bottom_last : 0ull);
                        root[i] = root_of(r);
                    }
                }
                mark(root, m, std::integral_constant<uint32_t, kRows>{});
            };
            // full tiles (the rule) take the row count and the first and last row masks at compile time (16 x 65536 40.5
            // against 39.8 us per sweep)
            const bool full = TWR_MAX <= kRows && nrow == kRows;
            if (full)
                mark_rows(std::true_type{}, 0u);
            else if (one_chunk)
                mark_rows(std::false_type{}, 0u);
            else
                for (uint32_t r0 = 0; r0 < nrow; r0 += kRows)
                    mark_rows(std::false_type{}, r0);
            __syncthreads();   // every slot label in place

            // labels out, as above
            const uint32_t ecol_off = LaneBit(side) ? ((rbound ? d.ecol_stride : 0u) + r_begin * rpw + lrow) * 4u : kNoStore;
            const auto emit = [&](const uint32_t r, const uint32_t root) {
                const uint32_t wr = r_begin + r;
                const uint32_t rowoff = wr * bl.stride;   // sites from the block's first site
                const uint32_t lab = LdsLoad(At(P, root)) >> 2;
                const uint32_t e = (lab << 16) | (root >> 2);
                __builtin_amdgcn_raw_buffer_store_b16(static_cast<uint16_t>(lab), rs_local, lane * 2u, rowoff * 2u, 0);
                __builtin_amdgcn_raw_buffer_store_b32(e, rs_ecol, ecol_off, r * rpw * 4u, 0);
                if (wr == 0u)
                    __builtin_amdgcn_raw_buffer_store_b32(e, rs_erow, lane4, 0, 0);
                if (wr + 1u == bnwr)
                    __builtin_amdgcn_raw_buffer_store_b32(e, rs_erow, lane4, 256u, 0);
            };
            if (full)
            {
#pragma unroll
                for (uint32_t i = 0; i < kRows; ++i)
                    emit(i, xs[i]);
            }
            else if (one_chunk)
            {
#pragma unroll
                for (uint32_t i = 0; i < kRows; ++i)
                    if (i < nrow)
                        emit(i, xs[i]);
            }
            else
                for (uint32_t r = 0; r < nrow; ++r)
                    emit(r, root_of(r));
        }
        const gptr<uint64_t> bb = Glob(d.bbits) + kBbitWords * bl.lb;
        if (lane == 0)
        {
            if (last_wave)
                bb[0] = down_bits;
            if (NW == kWavesPerBlock)
                bb[1u + w] = right_bits;
        }
        if (NW != kWavesPerBlock && threadIdx.x < kWavesPerBlock)
            bb[1u + threadIdx.x] = s_right[threadIdx.x];
        if (threadIdx.x == 0)
        {
            const uint32_t n = LdsLoad(&s_nslot);
            Glob(d.edge_count)[kWavesPerBlock * bl.lb] = min(n, bslots);
            if (n > bslots)
                (void)__hip_atomic_fetch_or(stp + kStErr, kErrLabelRange, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
    }

    // 64-wide tiles of up to 16 rows: eight waves per SIMD (the register budget is asked for explicitly; the compiler
    // keeps the excess scalar registers in vector lanes). Narrow tiles keep the default budget (the cap would spill
    // vector registers to scratch), and taller tiles are limited by their LDS anyway.
    // NW waves per block: four take a tile each, eight and sixteen a half and a quarter of a tile.
    template <uint32_t NW, uint32_t TWR_MAX, BondMode MODE, bool PAD, bool FULL>
    __global__ __launch_bounds__(64 * NW) __attribute__((amdgpu_waves_per_eu(8, 8))) void k_bond_label(
        const LatDesc* __restrict__ descs, const uint32_t* __restrict__ block_lat, const uint32_t total_blocks)
    {
        BondLabel<NW, TWR_MAX, true, MODE, PAD, FULL>(descs, block_lat, total_blocks);
    }

    template <uint32_t TWR_MAX, bool TW64, BondMode MODE, bool PAD>
    __global__ __launch_bounds__(256) void k_bond_label_any(const LatDesc* __restrict__ descs, const uint32_t* __restrict__ block_lat,
                                                            const uint32_t total_blocks)
    {
        BondLabel<kWavesPerBlock, TWR_MAX, TW64, MODE, PAD, false>(descs, block_lat, total_blocks);
    }

    // The labelling of one bond field alone: the descriptor comes with the launch, not from memory.
    template <uint32_t NW, uint32_t TWR_MAX, bool PAD, bool FULL>
    __global__ __launch_bounds__(64 * NW) __attribute__((amdgpu_waves_per_eu(8, 8))) void k_label_blocks(const LatDesc d, const uint32_t total_blocks)
    {
        BondLabel<NW, TWR_MAX, true, BondMode::kLabel, PAD, FULL>(&d, nullptr, total_blocks);
    }

    // (TWR_MAX 8 has half the LDS and rows of 16: 2 x 2^20 at bond density 0.95 74 against 83 us, the whole call 93 and 100)
    template <uint32_t TWR_MAX, bool PAD>
    __global__ __launch_bounds__(256) void k_label_blocks_narrow(const LatDesc d, const uint32_t total_blocks)
    {
        BondLabel<kWavesPerBlock, TWR_MAX, false, BondMode::kLabel, PAD, false>(&d, nullptr, total_blocks);
    }

    // Launches of few blocks of 64-wide tiles, all of a height that four waves can share, give every block more waves:
    // sixteen up to one block per CU, eight up to three. Microseconds per sweep at T_c with 4 / 8 / 16 waves: 6 blocks
    // (128 x 192) 17.0 / 14.4 / 13.9, 16 (256^2) 19.1 / 16.5 / 16.2, 36 (384^2) 22.6 / 20.0 / 19.6, 64 (512^2) 22.9 / 20.3 /
    // 20.0, 132 (768 x 704) 23.9 / 21.3 / 20.9, 256 (1024^2) 24.7 / 22.1 / 21.8, 256 padded (1000^2) 25.2 / 22.8 / 22.4; with
    // builds of before the constant row counts 352 padded blocks (1000 x 1350) 25.4 / 23.7 / 25.1, 484 (1408^2) - / 25.5 / 26.9,
    // 676 (1664^2) 29.2 / 28.8 / -, 1024 (2048^2) 32.6 / 33.3 / 46.
    constexpr uint32_t kWideBlocks = 256;
    constexpr uint32_t kHalfBlocks = 768;
    // f(NW) with the waves per block for a launch of 64-wide tiles of at most 16 rows
    template <typename F>
    static void WithWaves(const uint32_t total_blocks, const BondForm form, F&& f)
    {
        if (form != BondForm::kAny && total_blocks <= kWideBlocks)
            f(std::integral_constant<uint32_t, 16>{});
        else if (form != BondForm::kAny && total_blocks <= kHalfBlocks)
            f(std::integral_constant<uint32_t, 8>{});
        else
            f(std::integral_constant<uint32_t, kWavesPerBlock>{});
    }

#if SWMI_BOND_MODE == 2
    // tiles of at most 16 rows
    template <bool TW64>
    void LaunchLabelBlocksT(const LatDesc& d, const uint32_t total_blocks, const BondForm form, const bool pad, hipStream_t stream)
    {
        const uint32_t g = XcdGrid(total_blocks);
        if constexpr (TW64)
            WithWaves(total_blocks, form, [&](auto nw) {
                constexpr uint32_t NW = decltype(nw)::value;
                if (pad)
                    k_label_blocks<NW, 64 / NW, true, false><<<g, 64 * NW, 0, stream>>>(d, total_blocks);
                else if (form == BondForm::kFull)
                    k_label_blocks<NW, 64 / NW, false, true><<<g, 64 * NW, 0, stream>>>(d, total_blocks);
                else
                    k_label_blocks<NW, 64 / NW, false, false><<<g, 64 * NW, 0, stream>>>(d, total_blocks);
            });
        else if (pad)
            k_label_blocks_narrow<16, true><<<g, 256, 0, stream>>>(d, total_blocks);
        else if (d.twr <= 8u)
            k_label_blocks_narrow<8, false><<<g, 256, 0, stream>>>(d, total_blocks);
        else
            k_label_blocks_narrow<16, false><<<g, 256, 0, stream>>>(d, total_blocks);
    }

    template void LaunchLabelBlocksT<SWMI_BOND_TW64>(const LatDesc&, uint32_t, BondForm, bool, hipStream_t);
#else
    // Padded lattices of more blocks run with the default register budget (seven blocks per CU) up to two rounds of
    // blocks, with eight blocks per CU above: 2209 blocks (3000^2) 51.2 against 51.7 us per sweep, 3969 (4000^2) 73.3
    // against 70.5, 15625 (8000^2) 205.1 against 205.0.
    constexpr uint32_t kPadRounds = 2u * 7u * 256u;

    template <bool TW64, BondMode MODE>
    void LaunchBondLabelT(const LatDesc* d_desc, const uint32_t* d_block_lat, const uint32_t total_blocks, const uint32_t max_twr,
                          const BondForm form, const bool pad, hipStream_t stream)
    {
        const uint32_t g = XcdGrid(total_blocks);
        const auto launch = [&](auto kernel, const uint32_t threads = 256) {
            kernel<<<g, threads, 0, stream>>>(d_desc, d_block_lat, total_blocks);
        };
        if constexpr (TW64)
        {
            if (!pad && max_twr <= 8 && (form == BondForm::kAny || total_blocks > kHalfBlocks))
                return launch(k_bond_label<kWavesPerBlock, 8, MODE, false, false>);
            if (max_twr <= 16 && (!pad || (form != BondForm::kAny && total_blocks <= kHalfBlocks) || total_blocks > kPadRounds))
                return WithWaves(total_blocks, form, [&](auto nw) {
                    constexpr uint32_t NW = decltype(nw)::value;
                    constexpr bool kSweep = MODE == BondMode::kSweep;
                    if (pad)
                        launch(k_bond_label<NW, 64 / NW, MODE, true, false>, 64 * NW);
                    else if (kSweep && form == BondForm::kFull)
                        launch(k_bond_label<NW, 64 / NW, MODE, false, kSweep>, 64 * NW);
                    else
                        launch(k_bond_label<NW, 64 / NW, MODE, false, false>, 64 * NW);
                });
        }
        if (pad)   // padded lattices: two tile-height bounds (and the small one of narrow tiles)
        {
            if (!TW64 && max_twr <= 4)
                launch(k_bond_label_any<4, false, MODE, true>);
            else if (max_twr <= 16)
                launch(k_bond_label_any<16, TW64, MODE, true>);
            else
                launch(k_bond_label_any<64, TW64, MODE, true>);
        }
        // (widths 2 and 4: microseconds per sweep with the 8-row build / this one, 2 x 65536 21.5 / 20.4, 4 x 65536 25.5 / 24.3)
        else if (!TW64 && max_twr <= 4)
            launch(k_bond_label_any<4, false, MODE, false>);
        else if (!TW64 && max_twr <= 8)
            launch(k_bond_label_any<8, false, MODE, false>);
        else if (!TW64 && max_twr <= 16)
            launch(k_bond_label_any<16, false, MODE, false>);
        else if (max_twr <= 32)
            launch(k_bond_label_any<32, TW64, MODE, false>);
        else
            launch(k_bond_label_any<64, TW64, MODE, false>);
    }

    template void LaunchBondLabelT<SWMI_BOND_TW64, static_cast<BondMode>(SWMI_BOND_MODE)>(const LatDesc*, const uint32_t*, uint32_t, uint32_t,
                                                                                       BondForm, bool, hipStream_t);
#endif
}
