// swmi_resident_body.h -- the body of k_resident<kR, TW64, PAD, FULL>(descs, slots, sweeps, groups, sample_mode), included by
// that kernel and by the function of the same parameters that k_resident_mixed calls (swmi_resident.hip). As an inlined
// function of its own it took ten more registers in the kernel of full 16-row strips, which then spilled: 128^2 12.0 us
// per sweep instead of 11.5.
        extern __shared__ uint32_t P[];                // one word per padded site
        __shared__ uint32_t Q[kWaves * kQw];
        __shared__ uint64_t sS[kResidentSites / 64u];  // spins of every wave row, as the sweep finds them
        __shared__ uint64_t sB[kResidentSites / 64u];  // bonds to the right inside the wave row (64-wide: strip's first row, by wave)
        __shared__ uint64_t sD[TW64 ? 1u : kResidentSites / 64u];   // narrow: down bonds of the wave row
        __shared__ uint64_t sE[TW64 ? 1u : kResidentSites / 64u];   // narrow: bonds across the lattice's right edge
        __shared__ __align__(64) uint64_t AC[8];       // Numerical Recipes pairs (a << 32 | c) by selector
        __shared__ uint64_t JAC[8];                    // the jump from the stored states to the current iteration
        __shared__ int32_t sEM[2];
        __shared__ double sMom[6];                     // written by thread 0 only
        __shared__ uint32_t sErr;

        const LatDesc& d = descs[slots[blockIdx.x]];
        const gptr<uint32_t> stp = Glob(d.state);
        const uint32_t lane = threadIdx.x & 63u, lane4 = lane * 4u;
        const uint32_t w = Uniform(threadIdx.x >> 6);
        const uint32_t tx = d.tiles_x, rows = d.nwr_y, n0 = d.n0;
        const uint32_t tw = TW64 ? 64u : d.tw, rpw = TW64 ? 1u : d.rpw;
        const uint32_t nstrips = kWaves / tx, R = (rows + nstrips - 1u) / nstrips;
        const uint32_t col = w % tx, strip = w / tx, y0 = strip * R;
        const uint32_t nrow = FULL ? kR : ((strip < nstrips && y0 < rows) ? min(R, rows - y0) : 0u);
        constexpr bool kBits = TW64 && !PAD;   // the last column's bonds follow after the rows, from two scalar words
        const uint32_t ybelow = y0 + nrow >= rows ? 0u : y0 + nrow;   // wave row below the strip
        const uint32_t gstep = tx;                                    // groups between consecutive rows of a strip
        const uint32_t g0 = y0 * tx + col;
        const uint32_t gbelow = ybelow * tx + col;
        const uint32_t cright = col + 1u == tx ? 0u : col + 1u;

        const bool lastcol = PAD && col + 1u == tx;
        const uint64_t vmask = lastcol ? d.vlast : ~0ull;
        const uint32_t elane = lastcol ? d.elast : tw - 1u;
        uint64_t rowstart = 1;
        if (!TW64)
            for (uint32_t j = tw; j < 64u; j += tw)
                rowstart |= 1ull << j;
        const uint64_t redge = rowstart << elane;
        const uint64_t in_right = vmask & ~redge;
        const uint64_t low = TW64 ? 0ull : ((1ull << (64u - tw)) - 1ull);

        uint32_t it = stp[kStIteration];
        const uint32_t it_end = stp[kStItEnd], applied = stp[kStApplied], rng_it = Glob(d.aux)[kAuxRngIt];
        const uint32_t it_meas = stp[kStItMeas], sep2 = stp[kStSep2], thr = d.threshold, seed = d.seed;
        const bool random_rule = d.flip_rule != 0u;
        uint32_t n_samples = stp[kStSamples], last_sample = stp[kStLastSample];
        const uint32_t series_cap = stp[2];
        LatState* const st_g = reinterpret_cast<LatState*>(d.state);
        if (threadIdx.x < 6u)
            sMom[threadIdx.x] = st_g->moments[threadIdx.x];
        if (threadIdx.x < 8u)
        {
            uint32_t a, c, ja = 1u, jc = 0u;
            ParamsOf(threadIdx.x, a, c);
            const uint32_t n_jump = min(it - rng_it, 15u);
            for (uint32_t i = 0; i < n_jump; ++i)
            {
                ja *= a;
                jc = a * jc + c;
            }
            AC[threadIdx.x] = (static_cast<uint64_t>(a) << 32) | c;
            JAC[threadIdx.x] = (static_cast<uint64_t>(ja) << 32) | jc;
        }
        if (threadIdx.x == 0)
        {
            sEM[0] = 0;
            sEM[1] = 0;
            sErr = 0u;
        }

        // spin bytes (spin and selector), lcg32 states and group rotations of the strip
        uint32_t sp[kR], rs[kR];
        // (buffer views: row offsets in scalar registers, no per-row vector addresses to keep)
        const uint32_t np = rows * tx * 64u;
        const Rsrc rs_spins = MakeRsrc(d.spins, np), rs_rng = MakeRsrc(d.rng, np * 4u), rs_local = MakeRsrc(d.local, np * 2u);
        const gptr<uint32_t> rotp = Glob(d.rot);
        const bool pending = applied != it;
        const uint32_t pkey = pending && random_rule ? FlipKey(seed, applied) : 0u;
        bool ok = true;
#pragma unroll
        for (uint32_t i = 0; i < kR; ++i)
        {
            sp[i] = 0u;
            rs[i] = 0u;
            if (i < nrow)
            {
                const uint32_t first = (g0 + i * gstep) * 64u;
                sp[i] = __builtin_amdgcn_raw_buffer_load_b8(rs_spins, lane, first, 0);
                rs[i] = __builtin_amdgcn_raw_buffer_load_b32(rs_rng, lane4, first * 4u, 0);
                if (pending)
                    sp[i] ^= PendingFlip(d, y0 + i, col, __builtin_amdgcn_raw_buffer_load_b16(rs_local, lane * 2u, first * 2u, 0),
                                         random_rule, pkey, ok);
            }
        }
        uint32_t grot = lane < nrow ? rotp[g0 + lane * gstep] : 0u;   // lane i: row i
        __syncthreads();   // AC, JAC, sErr
        if (!ok)
            sErr = kErrLabelRange;
#pragma unroll
        for (uint32_t i = 0; i < kR; ++i)
        {
            if (i < nrow)
            {
                const uint64_t j = JAC[(sp[i] & kSelMask) >> kSelShift];
                rs[i] = static_cast<uint32_t>(j >> 32) * rs[i] + static_cast<uint32_t>(j);
                const uint64_t S = __ballot((sp[i] & 1u) != 0u);
                if (lane == 0u)
                    sS[g0 + i * gstep] = S;
            }
        }
        __syncthreads();   // sS

        uint32_t* const Qw = Q + w * kQw;
        const uint32_t run_words = OffsetFrom(P, Qw), spare = OffsetFrom(P, Qw + 64u + lane);
        const uint32_t rowb = n0 * 4u * rpw;                // P bytes between consecutive rows of a strip
        const uint32_t node0 = g0 * 256u + lane4;           // this lane's node of the strip's first row
        const uint32_t node_below = gbelow * 256u + lane4;
        // sweeps until the schedule ends (without one the update count may wrap)
        const uint32_t last_active = it_end == 0xFFFFFFFFu ? 0xFFFFFFFFu : (it_end > it ? (it_end - it - 1u) / 2u + 1u : 0u);
        const uint32_t total = min(groups * sweeps, last_active);
        uint32_t done = 0;
        Qw[lane] = 0u;   // run words of LabelRow64

        const auto first_col = [&]() -> uint64_t {   // bit i: spin of row i's right neighbour column
            uint32_t h = 0;
            if (TW64 && lane < nrow)
                h = static_cast<uint32_t>(sS[(y0 + lane) * tx + cright]) & 1u;
            return __ballot(h != 0u);
        };
        const uint32_t ac_at = static_cast<uint32_t>(reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) uint64_t*)AC));
        const auto pair_of = [&](const uint32_t ks) {   // AC's alignment makes the address an or
            return *(__attribute__((address_space(3))) const uint64_t*)static_cast<uintptr_t>(ac_at | ks);
        };
        const auto right_of = [&](const uint64_t S, const uint64_t HR, const uint32_t i) -> uint64_t {
            if (TW64)
                return ((S >> 1) & ~redge) | (((HR >> i) & 1ull) << elane);
            return ((S >> 1) & ~redge) | ((S << elane) & redge);
        };
        UnionQueue queue{P, Qw, lane};

        const auto sweep = [&](const bool last) {
            const uint32_t it1 = it + 1u, it2 = it + 2u;
            const bool rot1 = it1 % 15u == 0u, rot2 = it2 % 15u == 0u;
            const uint64_t HR = first_col();
            const uint64_t Sbelow = nrow > 0u ? Uniform64(sS[gbelow]) : 0ull;
            uint32_t s63_b = 0, u63_b = 0;   // last column's spin and draw, the latest row in bit 0
            uint64_t right_bits = 0, prev_S = 0, prev_U2 = 0, prev_B = 0;
            uint32_t Rp = 0;
            uint32_t xs[kR];   // every row's root: as the row was labelled, later the root of the whole forest
            uint64_t Snext = nrow > 0u ? __ballot((sp[0] & 1u) != 0u) : 0ull;
#pragma unroll
            for (uint32_t i = 0; i < kR; ++i)
            {
                if (i < nrow)
                {
                    const uint64_t S = Snext;
                    if (i + 1u < kR)
                        Snext = __ballot((sp[i + 1u < kR ? i + 1u : i] & 1u) != 0u);
                    // two LCG32_State<64>::Update of the row's group (random/src/lcg32.cpp:51-84)
                    uint32_t ks = sp[i] & kSelMask, st = rs[i], shift = 0;
                    if (rot1)
                    {
                        shift = ShuffleShift(st, it1) & 63u;
                        ks = static_cast<uint32_t>(__shfl(static_cast<int>(ks), static_cast<int>((lane + shift) & 63u)));
                    }
                    uint64_t ac = pair_of(ks);
                    st = static_cast<uint32_t>(ac >> 32) * st + static_cast<uint32_t>(ac);
                    const uint64_t U1 = __ballot(st < thr);
                    if (rot2)   // (both rotate in the sweep in which the update count wraps to 0)
                    {
                        const uint32_t second = ShuffleShift(st, it2) & 63u;
                        ks = static_cast<uint32_t>(__shfl(static_cast<int>(ks), static_cast<int>((lane + second) & 63u)));
                        ac = pair_of(ks);
                        shift += second;
                    }
                    st = static_cast<uint32_t>(ac >> 32) * st + static_cast<uint32_t>(ac);
                    const uint64_t U2 = __ballot(st < thr) & vmask;
                    rs[i] = st;
                    if (rot1 || rot2)
                    {
                        sp[i] = (sp[i] & 1u) | ks;
                        grot = lane == i ? (grot + shift) & 63u : grot;
                    }
                    const uint64_t Ball = ~(S ^ (kBits ? S >> 1 : right_of(S, HR, i))) & U1 & vmask;
                    const uint64_t B = Ball & in_right;
                    const uint32_t node = node0 + i * rowb;
                    if (TW64)
                    {
                        if (kBits)
                        {
                            s63_b = Uniform((s63_b << 1) + static_cast<uint32_t>(S >> 63));
                            u63_b = Uniform((u63_b << 1) + static_cast<uint32_t>(U1 >> 63));
                            asm volatile("" : "+s"(s63_b), "+s"(u63_b));   // taken here, not kept as the rows' masks
                        }
                        else
                            right_bits |= ((Ball >> elane) & 1ull) << i;
                        const uint64_t D = i == 0u ? 0ull : (~(prev_S ^ S) & prev_U2);
                        Rp = LabelRow64(P, run_words, spare, node, B, D, Rp, RowBase(i + 1u));
                        xs[i] = Rp;
                        if (i == 0u && lane == 0u)
                            sB[w] = B;
                    }
                    else
                    {
                        // every site starts under the first site of its row run
                        *At(P, node) = node - lane4 + RunStart(B, lane) * 4u;
                        const uint64_t Sn = i + 1u < nrow ? Snext : Sbelow;
                        const uint64_t SD = (Shr(S, tw) & low) | Shl(Sn, 64u - tw);
                        if (lane == 0u)
                        {
                            sB[y0 + i] = B;
                            sD[y0 + i] = ~(S ^ SD) & U2;
                            sE[y0 + i] = Ball & redge;
                        }
                    }
                    prev_S = S;
                    prev_U2 = U2;
                    prev_B = B;
                }
            }
            if (kBits)
            {
                const uint32_t up = 32u - max(nrow, 1u);   // row i of the words is bit nrow - 1 - i
                right_bits = ~((__brev(s63_b) >> up) ^ static_cast<uint32_t>(HR)) & (__brev(u63_b) >> up);
            }
            __syncthreads();   // every node and bond mask in place

            if (nrow > 0u)
            {
                if (TW64)
                {
                    // down, into the first row of the strip below (this strip's own where it is alone in its column)
                    const uint64_t Dl = ~(prev_S ^ Sbelow) & prev_U2;
                    const uint64_t Bn = Uniform64(sB[ybelow == 0u ? col : (strip + 1u) * tx + col]);
                    queue.Push(FirstBondPerInterval(Dl, prev_B & Bn, 1ull), Rp, node_below);
                    // right, one lane per row
                    queue.Push(right_bits, ((y0 + lane) * tx + col) * 256u + elane * 4u, ((y0 + lane) * tx + cright) * 256u);
                    queue.Finish();
                    Qw[lane] = 0u;   // the queue took the run words' place
                }
                else
                    NarrowUnions(queue, sB, sD, sE, y0, nrow, rows, tw, rowstart, elane);
            }
            __syncthreads();   // the forest is complete

            if (nrow > 0u)
            {
#pragma unroll
                for (uint32_t i = 0; i < kR; ++i)
                    if (!TW64 || i >= nrow)
                        xs[i] = node0 + (i < nrow ? i : 0u) * rowb;
                if (!FindRoots<kR>(P, xs) && lane == 0u)
                    sErr = kErrLabelRange;
                // the flips; lane i collects the spin mask of row i and stores it
                uint32_t Slo = 0, Shi = 0;
                const auto flip = [&](const auto& bit_of) {
#pragma unroll
                    for (uint32_t i = 0; i < kR; ++i)
                    {
                        sp[i] ^= bit_of(xs[i] >> 2);
                        const uint64_t S = __ballot((sp[i] & 1u) != 0u);
                        Slo = LaneBit(1ull << i) ? static_cast<uint32_t>(S) : Slo;
                        Shi = LaneBit(1ull << i) ? static_cast<uint32_t>(S >> 32) : Shi;
                    }
                };
                if (random_rule)
                {
                    const uint32_t key = FlipKey(seed, it);
                    flip([&](const uint32_t root) { return FlipBit(d, root, true, key); });
                }
                else
                    flip([&](const uint32_t root) { return FlipBit(d, root, false, 0u); });
                if (lane < nrow)
                    sS[g0 + lane * gstep] = (static_cast<uint64_t>(Shi) << 32) | Slo;
                if (last)
                {
#pragma unroll
                    for (uint32_t i = 0; i < kR; ++i)
                        if (i < nrow)
                            __builtin_amdgcn_raw_buffer_store_b16(static_cast<uint16_t>(xs[i] >> 2), rs_local, lane * 2u,
                                                                  (g0 + i * gstep) * 128u, 0);
                }
            }
            it = it2;
            __syncthreads();   // sS of the new configuration; P is free
        };

        // (E, M) of the configuration, appended as k_finalize_samples does
        const auto sample = [&]() {
            if (sample_mode == static_cast<int32_t>(kSampleDue) &&
                !(it > last_sample && it > it_meas && sep2 != 0u && (it - it_meas) % sep2 == 0u))
                return;
            const uint64_t HR = first_col();
            const uint64_t Sbelow = nrow > 0u ? Uniform64(sS[gbelow]) : 0ull;
            const int32_t nv = __popcll(vmask);
            int32_t e = 0, m = 0;
            uint64_t Snext = nrow > 0u ? __ballot((sp[0] & 1u) != 0u) : 0ull;
#pragma unroll
            for (uint32_t i = 0; i < kR; ++i)
            {
                if (i < nrow)
                {
                    const uint64_t S = Snext;
                    if (i + 1u < kR)
                        Snext = __ballot((sp[i + 1u < kR ? i + 1u : i] & 1u) != 0u);
                    const uint64_t Sn = i + 1u < nrow ? Snext : Sbelow;
                    const uint64_t SD = TW64 ? Sn : ((Shr(S, tw) & low) | Shl(Sn, 64u - tw));
                    e += 2 * (__popcll(~(S ^ right_of(S, HR, i)) & vmask) + __popcll(~(S ^ SD) & vmask)) - 2 * nv;
                    m += 2 * __popcll(S & vmask) - nv;
                }
            }
            if (lane == 0u && nrow > 0u)
            {
                __hip_atomic_fetch_add(&sEM[0], e, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
                __hip_atomic_fetch_add(&sEM[1], m, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
            }
            __syncthreads();
            if (threadIdx.x == 0)
            {
                const long long E = sEM[0], M = sEM[1];
                const double n = static_cast<double>(d.n0v) * static_cast<double>(d.n1);
                const double ev = -static_cast<double>(E) / n;
                const double mv = static_cast<double>(M) / n;
                sMom[0] += 1.0;
                sMom[1] += ev;
                sMom[2] += ev * ev;
                sMom[3] += fabs(mv);
                sMom[4] += mv * mv;
                sMom[5] += (mv * mv) * (mv * mv);
                if (n_samples < series_cap)
                {
                    long long* series = reinterpret_cast<long long*>(d.state + kLatStateWords);
                    series[2u * n_samples] = E;
                    series[2u * n_samples + 1u] = M;
                }
                sEM[0] = 0;
                sEM[1] = 0;
            }
            n_samples += 1u;
            last_sample = it;
            __syncthreads();
        };

        for (uint32_t g = 0; g < groups; ++g)
        {
            for (uint32_t s = 0; s < sweeps && done < total; ++s)
            {
                ++done;
                sweep(done == total);
            }
            if (sample_mode >= 0)
                sample();
        }

        // the chain's state back to memory: no flip pending, states of the current iteration
#pragma unroll
        for (uint32_t i = 0; i < kR; ++i)
        {
            if (i < nrow && (done > 0u || pending))
            {
                const uint32_t first = (g0 + i * gstep) * 64u;
                __builtin_amdgcn_raw_buffer_store_b8(static_cast<uint8_t>(sp[i]), rs_spins, lane, first, 0);
                __builtin_amdgcn_raw_buffer_store_b32(rs[i], rs_rng, lane4, first * 4u, 0);
            }
        }
        if (done > 0u && lane < nrow)
            rotp[g0 + lane * gstep] = grot;
        if (threadIdx.x == 0)
        {
            if (sErr != 0u)
                (void)__hip_atomic_fetch_or(stp + kStErr, sErr, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            if (done > 0u || pending)
            {
                stp[kStIteration] = it;
                stp[kStApplied] = it;
                Glob(d.aux)[kAuxRngIt] = it;
            }
            if (done > 0u)
                Glob(d.aux)[kAuxWholeLabels] = 1u;
            if (sample_mode >= 0)
            {
                stp[kStSamples] = n_samples;
                stp[kStLastSample] = last_sample;
                for (uint32_t k = 0; k < 6u; ++k)
                    st_g->moments[k] = sMom[k];
            }
        }
