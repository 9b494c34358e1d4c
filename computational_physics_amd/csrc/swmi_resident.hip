// swmi_resident.hip -- k_resident: whole sweeps of small lattices in one workgroup.
//
// A lattice of at most kResidentSites padded sites fits one workgroup: spins, lcg32 states and selectors in
// registers, the union-find over all of its sites in LDS. One launch then runs any number of sweeps with their
// samples, where the tiled path (swmi_kernels.hip) needs three launches per sweep and three more kernels per sample.
// What bounds it is the chain of dependent LDS operations per row of a wave's strip, so sixteen waves (the largest
// workgroup) share the lattice's rows: strips of at most 16 rows of one tile column (64-wide tiles) or 16 wave rows
// (narrower lattices). Microseconds per sweep at T_c, tiled / here: 32^2 24.4 / 3.8, 64^2 12.8 / 4.3, 128^2
// 13.7 / 11.6 (before the tiled path had its builds for launches of few blocks 35, 24 and 24); of the 128^2 sweep the rows take 6, the strip edges 1.3, the final roots 2, the flips 0.9, waiting the rest.
#include "swmi_device.h"

namespace swmi
{
    namespace
    {
        constexpr uint32_t kWaves = kResidentWaves;
        constexpr uint32_t kQw = 128u;   // per-wave LDS words: run minima and spare words, or the union queue
    }

    // Unions a wave collects and works off 64 at a time, all lanes in lockstep (Qw: 128 words of the wave).
    struct UnionQueue
    {
        uint32_t* P;
        uint32_t* Qw;
        uint32_t lane, len = 0;

        // the lanes of K bring the pair (a, b) of nodes
        __device__ __forceinline__ void Push(const uint64_t K, const uint32_t a, const uint32_t b)
        {
            if (LaneBit(K))
                Qw[len + __builtin_amdgcn_mbcnt_hi(static_cast<uint32_t>(K >> 32), __builtin_amdgcn_mbcnt_lo(static_cast<uint32_t>(K), 0u))] =
                    (a << 16) | b;
            len += static_cast<uint32_t>(__popcll(K));
            if (len >= 64u)
            {
                const uint32_t e = Qw[lane];
                LdsUnionLockstep(P, e >> 16, e & 0xFFFFu);
                const uint32_t rem = len - 64u;
                const uint32_t t = Qw[64u + lane];
                if (lane < rem)
                    Qw[lane] = t;
                len = rem;
            }
        }

        __device__ __forceinline__ void Finish()
        {
            if (len > 0u)
            {
                const uint32_t e = lane < len ? Qw[lane] : 0u;
                LdsUnionLockstep(P, e >> 16, e & 0xFFFFu);
                len = 0u;
            }
        }
    };

    // The roots of kR nodes per lane, two steps per round, every row of the lane in flight. Parents only decrease: a
    // chase that does not end within the sites is a broken forest, reported (false) instead of followed.
    template <uint32_t kR>
    __device__ __forceinline__ bool FindRoots(uint32_t* P, uint32_t (&xs)[kR])
    {
        for (uint32_t round = 0;; ++round)
        {
            if (round * 2u > kResidentSites)
                return false;
            uint32_t ys[kR];
            uint32_t moved = 0;
#pragma unroll
            for (uint32_t i = 0; i < kR; ++i)
            {
                ys[i] = LdsLoad(At(P, xs[i]));
                moved += ys[i] ^ xs[i];
            }
            if (!__ballot(moved != 0u))
                return true;
            moved = 0;
#pragma unroll
            for (uint32_t i = 0; i < kR; ++i)
            {
                xs[i] = LdsLoad(At(P, ys[i]));
                moved += xs[i] ^ ys[i];
            }
            if (!__ballot(moved != 0u))
                return true;
        }
    }

    __device__ __forceinline__ uint64_t Uniform64(const uint64_t v)
    {
        return (static_cast<uint64_t>(Uniform(static_cast<uint32_t>(v >> 32))) << 32) | Uniform(static_cast<uint32_t>(v));
    }

    // the first lane of the row run of `lane` in a narrow wave row with right bonds B
    __device__ __forceinline__ uint32_t RunStart(const uint64_t B, const uint32_t lane)
    {
        const uint64_t before = ~B & ((1ull << lane) - 1ull);
        return before ? 64u - static_cast<uint32_t>(__clzll(before)) : 0u;
    }

    // Narrow lattices (rows of tw < 64 sites): the unions of wave rows y0 .. y0 + nrow of `rows`, from their masks B
    // (bonds inside the row), D (down) and E (across the lattice's right edge; elane: a row's last site).
    __device__ __forceinline__ void NarrowUnions(UnionQueue& q, const uint64_t* sB, const uint64_t* sD, const uint64_t* sE, const uint32_t y0,
                                                 const uint32_t nrow, const uint32_t rows, const uint32_t tw, const uint64_t rowstart,
                                                 const uint32_t elane)
    {
        const uint32_t lane4 = q.lane * 4u;
        for (uint32_t i = 0; i < nrow; ++i)
        {
            const uint32_t y = y0 + i, yn = y + 1u == rows ? 0u : y + 1u;
            const uint64_t B = Uniform64(sB[y]), Bn = Uniform64(sB[yn]);
            const uint64_t K = FirstBondPerInterval(Uniform64(sD[y]), B & (Shr(B, tw) | Shl(Bn, 64u - tw)), rowstart);
            const uint32_t top = y * 256u + lane4;
            q.Push(K, top, q.lane < 64u - tw ? top + tw * 4u : yn * 256u + lane4 - (64u - tw) * 4u);
            q.Push(Uniform64(sE[y]), top, top - elane * 4u);
        }
        q.Finish();
    }

    // Flip of a site of the tiled path's last sweep that is still pending: the rule at the root of a cluster inside
    // its block, or the bit k_resolve wrote for the slot of an edge-reaching cluster. A label outside the block's range
    // (a broken invariant) clears ok.
    __device__ uint32_t PendingFlip(const LatDesc& d, const uint32_t wr, const uint32_t sx, const uint32_t lab, const bool random_rule,
                                    const uint32_t key, bool& ok)
    {
        const uint32_t brows = kWavesPerBlock * d.twr, sy = wr / brows;
        const uint32_t i = lab & 0x7FFFu;
        if (lab & kEdgeFlag)
        {
            const uint32_t slots = kWavesPerBlock * d.edge_cap, s = min(i - d.qcap, slots - 1u);
            ok = ok && i - d.qcap < slots;
            return (Glob(static_cast<const uint32_t*>(d.fbits))[(sy * d.tiles_x + sx) * d.fsw + (s >> 5)] >> (s & 31u)) & 1u;
        }
        ok = ok && i < min(brows, d.nwr_y - sy * brows) * 64u;
        return FlipBit(d, SiteOf(BlockBase(d, sx, sy), 64u * d.tiles_x, i), random_rule, key);
    }

    // kR: rows of a strip (the lattices of a launch need at most kR). TW64: rows of 64 sites per tile column; else a
    // wave row holds 64 / tw lattice rows. PAD: some lattice of the launch has padding columns.
    // Runs `groups` groups of `sweeps` sweeps, a sample after each group when sample_mode >= 0 (a SampleMode).
    // Per sweep: (1) every wave draws, forms the bond masks of its strip and labels it row by row; (2) unions across
    // the strips' edges; (3) every site's root, the flip, the spin masks of the next sweep. Three barriers.
    // Nodes of the union-find are the byte offsets 4 * site into P, so a cluster's root is its canonical site.
    // FULL: every wave of every lattice has exactly kR rows.
    template <uint32_t kR, bool TW64, bool PAD, bool FULL>
    __global__ __launch_bounds__(64 * kWaves) void k_resident(const LatDesc* __restrict__ descs, const uint32_t* __restrict__ slots,
                                                              const uint32_t sweeps, const uint32_t groups, const int32_t sample_mode)
    {
#include "swmi_resident_body.h"
    }

    template <uint32_t kR, bool TW64, bool PAD, bool FULL>
    __device__ __forceinline__ void ResidentOf(const LatDesc* __restrict__ descs, const uint32_t* __restrict__ slots, const uint32_t sweeps,
                                               const uint32_t groups, const int32_t sample_mode)
    {
#include "swmi_resident_body.h"
    }

    // Lattices of several kinds in one launch, so that their chains run beside each other and not one launch after
    // another: 32^2, 64^2, 128^2, 48^2 and 100^2 together 34.0 us per sweep as five launches, 12.2 as one. (The bodies have
    // LDS arrays of their own, 58 KB in all beside P: one workgroup per CU, which is all that such a launch has.)
    __global__ __launch_bounds__(64 * kWaves) void k_resident_mixed(const LatDesc* __restrict__ descs, const uint32_t* __restrict__ slots,
                                                                    const uint32_t sweeps, const uint32_t groups, const int32_t sample_mode)
    {
        const LatDesc& d = descs[slots[blockIdx.x]];
        const uint32_t strips = kWaves / d.tiles_x, rows = (d.nwr_y + strips - 1u) / strips;
        if (d.tw != 64u)
            rows <= 4u ? ResidentOf<4, false, true, false>(descs, slots, sweeps, groups, sample_mode)
                       : ResidentOf<kResidentRows, false, true, false>(descs, slots, sweeps, groups, sample_mode);
        else
            rows <= 4u ? ResidentOf<4, true, true, false>(descs, slots, sweeps, groups, sample_mode)
                       : ResidentOf<kResidentRows, true, true, false>(descs, slots, sweeps, groups, sample_mode);
    }

    // The labelling alone, of a bond field given row by row (bit 0: bond to the right, bit 1: bond down): the canonical
    // label of every site of an n0 x n1 lattice in one launch, without scratch memory. Tiled, a 128^2 field took four
    // launches (setup, labels per block, merge, labels out): 23.5 us per call, this kernel 12.9.
    template <uint32_t kR, bool TW64>
    __global__ __launch_bounds__(64 * kWaves) void k_label_whole(const WholeGeometry g, const uint8_t* __restrict__ bonds,
                                                                 uint32_t* __restrict__ labels)
    {
        extern __shared__ uint32_t P[];
        __shared__ uint32_t Q[kWaves * kQw];
        __shared__ uint64_t sB[kResidentSites / 64u];
        __shared__ uint64_t sD[TW64 ? 1u : kResidentSites / 64u];
        __shared__ uint64_t sE[TW64 ? 1u : kResidentSites / 64u];
        const uint32_t lane = threadIdx.x & 63u, lane4 = lane * 4u;
        const uint32_t w = Uniform(threadIdx.x >> 6);
        const uint32_t tx = g.tiles_x, rows = g.nwr_y;
        const uint32_t tw = TW64 ? 64u : g.tw, rpw = TW64 ? 1u : 64u / tw;
        const uint32_t nstrips = kWaves / tx, R = (rows + nstrips - 1u) / nstrips;
        const uint32_t col = w % tx, strip = w / tx, y0 = strip * R;
        const uint32_t nrow = (strip < nstrips && y0 < rows) ? min(R, rows - y0) : 0u;
        const uint32_t ybelow = y0 + nrow >= rows ? 0u : y0 + nrow;
        const uint32_t cright = col + 1u == tx ? 0u : col + 1u;
        const uint32_t g0 = y0 * tx + col;
        const bool lastcol = col + 1u == tx;
        const uint64_t vmask = lastcol ? g.vlast : ~0ull;
        const uint32_t elane = lastcol ? g.elast : tw - 1u;
        uint64_t rowstart = 1;
        if (!TW64)
            for (uint32_t j = tw; j < 64u; j += tw)
                rowstart |= 1ull << j;
        const uint64_t redge = rowstart << elane;

        // this lane's site of row i: x of its lattice row y (its index in the caller's arrays)
        const uint32_t x = col * 64u + (lane & (tw - 1u)), ly = TW64 ? 0u : lane / tw;
        const bool valid = LaneBit(vmask);
        uint32_t bt[kR];
#pragma unroll
        for (uint32_t i = 0; i < kR; ++i)
        {
            bt[i] = 0u;
            if (i < nrow && valid)
                bt[i] = bonds[((y0 + i) * rpw + ly) * g.n0 + x];
        }
        uint32_t* const Qw = Q + w * kQw;
        const uint32_t run_words = OffsetFrom(P, Qw), spare = OffsetFrom(P, Qw + 64u + lane);
        const uint32_t rowb = tx * 256u, node0 = g0 * 256u + lane4;
        Qw[lane] = 0u;
        uint32_t xs[kR], Rp = 0;
        uint64_t prev_D = 0, prev_B = 0, right_bits = 0;
#pragma unroll
        for (uint32_t i = 0; i < kR; ++i)
        {
            xs[i] = node0;
            if (i < nrow)
            {
                const uint64_t Ball = __ballot((bt[i] & 1u) != 0u), D = __ballot((bt[i] & 2u) != 0u);
                const uint64_t B = Ball & ~redge;
                const uint32_t node = node0 + i * rowb;
                if (TW64)
                {
                    right_bits |= ((Ball >> elane) & 1ull) << i;
                    Rp = LabelRow64(P, run_words, spare, node, B, i == 0u ? 0ull : prev_D, Rp, RowBase(i + 1u));
                    xs[i] = Rp;
                    if (i == 0u && lane == 0u)
                        sB[w] = B;
                }
                else
                {
                    *At(P, node) = node - lane4 + RunStart(B, lane) * 4u;
                    xs[i] = node;
                    if (lane == 0u)
                    {
                        sB[y0 + i] = B;
                        sD[y0 + i] = D;
                        sE[y0 + i] = Ball & redge;
                    }
                }
                prev_D = D;
                prev_B = B;
            }
        }
        __syncthreads();   // every node and bond mask in place
        if (nrow > 0u)
        {
            UnionQueue queue{P, Qw, lane};
            if (TW64)
            {
                const uint64_t Bn = Uniform64(sB[ybelow == 0u ? col : (strip + 1u) * tx + col]);
                queue.Push(FirstBondPerInterval(prev_D, prev_B & Bn, 1ull), Rp, (ybelow * tx + col) * 256u + lane4);
                queue.Push(right_bits, ((y0 + lane) * tx + col) * 256u + elane * 4u, ((y0 + lane) * tx + cright) * 256u);
                queue.Finish();
            }
            else
                NarrowUnions(queue, sB, sD, sE, y0, nrow, rows, tw, rowstart, elane);
        }
        __syncthreads();   // the forest is complete
        if (nrow == 0u)
            return;
        (void)FindRoots<kR>(P, xs);
        const uint32_t pitch = tx * tw;
#pragma unroll
        for (uint32_t i = 0; i < kR; ++i)
        {
            if (i < nrow && valid)
            {
                const uint32_t p = xs[i] >> 2;
                labels[((y0 + i) * rpw + ly) * g.n0 + x] = pitch == g.n0 ? p : (p / pitch) * g.n0 + p % pitch;
            }
        }
    }

    void LaunchLabelWhole(const WholeGeometry& g, const uint8_t* bonds, uint32_t* labels, hipStream_t stream)
    {
        const uint32_t strips = kWaves / g.tiles_x, rows = (g.nwr_y + strips - 1u) / strips;
        const auto launch = [&](auto kernel) {
            kernel<<<1, 64 * kWaves, g.tiles_x * g.nwr_y * 64u * sizeof(uint32_t), stream>>>(g, bonds, labels);
        };
        if (rows <= 4u)
            g.tw == 64u ? launch(k_label_whole<4, true>) : launch(k_label_whole<4, false>);
        else
            g.tw == 64u ? launch(k_label_whole<kResidentRows, true>) : launch(k_label_whole<kResidentRows, false>);
    }

    void LaunchResident(const LatDesc* d_desc, const uint32_t* d_slots, const uint32_t n_lattices, const uint32_t max_sites,
                        const uint32_t max_rows, const bool full, const bool tw64, const bool pad, const bool mixed, const uint32_t sweeps,
                        const uint32_t groups, const int32_t sample_mode, hipStream_t stream)
    {
        const auto launch = [&](auto kernel) {
            kernel<<<n_lattices, 64 * kWaves, max_sites * sizeof(uint32_t), stream>>>(d_desc, d_slots, sweeps, groups, sample_mode);
        };
        if (mixed)
            return launch(k_resident_mixed);
        const auto launch_rows = [&](auto rows) {
            constexpr uint32_t kR = decltype(rows)::value;
            if (!tw64)
                launch(k_resident<kR, false, true, false>);
            else if (pad)
                launch(k_resident<kR, true, true, false>);
            else if (full)
                launch(k_resident<kR, true, false, true>);
            else
                launch(k_resident<kR, true, false, false>);
        };
        if (max_rows <= 4u)
            launch_rows(std::integral_constant<uint32_t, 4>{});
        else
            launch_rows(std::integral_constant<uint32_t, kResidentRows>{});
    }
}
