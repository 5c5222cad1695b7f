// msx_loop.hpp -- the slice loop of a few waves in one persistent kernel.
//
// Two sweeps per slice are two dependent launches: about 4 us each between
// the end of one and the first load of the next, for sweeps that compute 2-3
// us when a wave is small.  Here a team of work-groups stays on the GPU for a
// wave's whole loop and alternates between the two phases, the same
// transforms in the same order as row_sweep and col_sweep (same plans, same
// pointwise arithmetic: the exit waves are equal bit for bit).
//
// Between phases the team's work-groups exchange the wave through memory.
// They may run on different XCDs, whose L2 caches are not coherent with each
// other, so the wave is stored write-through and loaded past the local caches
// (device scope, kScopeDev); then no cache has to be flushed or invalidated
// and transmissions, twiddles and tables stay cached.  The barrier: every
// work-group drains its stores, publishes the phase number in a word of its
// own, and polls the words of all others with one load per lane.  Measured
// (256-thread work-groups, phases that only barrier / that also store and load
// 1 KB each): 1.2 / 2.1 us for 32 work-groups, 2.0 / 3.3 for 64, 2.3 / 4.6 for
// 128; one shared counter took 2.6 us for 64.
//
// Every wait ends: the launch is cooperative (all work-groups resident, or
// the launch fails), and a work-group that polls longer than `spin` times
// raises `status` and `dead` and leaves, after which the others run out as
// well; loops launched before the host has seen it leave at their first
// barrier.  The host then runs the call again by the sweeps.
#pragma once
#include "msx_sweep.hpp"

namespace msx {

// One wave of a job set (msx_multislice_batch): where its exit wave goes, its
// incident wave, its slices.
template <typename C> struct LoopJob {
    C* psi;
    const C* src;
    int nslice, pad;
};

template <typename C> struct LoopArgs {
    using Re = typename real_of<C>::type;
    C* psi;                 // [nb][NX][NY]: the waves, advanced in place
    const C* src;           // incident waves instead of psi (first_real)
    long long src_bstride;  // elements between waves of src (0: one for all)
    const C* trans;         // [nlayer][NX][NY]
    // layer of every slice and which propagator factors it takes, or null:
    // slice s is layer s and all take the first
    const int2* slices;
    const C *px, *py;       // propagator factors, [..][NX] and [..][NY]
    // a job set instead (psi, src, trans, slices, px, py unused): every wave
    // with its own buffers and slice count, transmission trans_tab[s nb + b]
    // and factors prop_tab[s nb + b], px then py
    const LoopJob<C>* jobs;
    const C* const* trans_tab;
    const C* const* prop_tab;
    const float *kx2, *ky2;
    float k2max;
    int blo, bhi;           // y columns in band: iy < blo and iy >= NY - bhi
    const C *twx, *twy;
    Re inv;                 // 1 / (NX NY)
    int s0, s1, nb;         // slices [s0, s1) (of a job set: 0 and each job's count)
    // first_real: slice s0 starts from real-space waves; otherwise psi holds
    // what a column sweep leaves (the inverse x transform of the spectrum).
    // first_all: slice s0 reads every y column (real-space waves, and generated
    // probes, whose columns no band limit has cleared), else those in band.
    // mixed: stop in that state, before the last inverse y transform
    int first_real, first_all, mixed;
    int team;               // work-groups per team; the grid is a multiple
    unsigned* flags;        // [teams][team] phase numbers, all at most `epoch`
    unsigned epoch;
    unsigned spin;          // polls before a wait gives up
    unsigned* dead;         // set by a wait that gave up, on the device ..
    int* status;            // .. and for the host
};

template <typename C, int NX, int NY> struct LoopShape {
    using PR = Plan<NY>;
    using PC = ColPlan<NX>;
    // threads per work-group: in FP32 tiles of at least 8 columns (64-byte row
    // pieces; 512 columns of one wave 1.02 -> 1.08x the sweeps, of 4 waves
    // 0.98 -> 1.22x); FP64 tiles of 4 are as wide, and 512 threads spill
    static constexpr int BT = sizeof(C) == 8 && 8 * PC::T > 256 ? 8 * PC::T : 256;
    static constexpr int LPW = BT / PR::T, TW = BT / PC::T;
    using LR = RowLds<PR, C>;
    using LC = ColLds<PC, C, TW>;
    static constexpr size_t tile = LC::len * sizeof(C), row = LPW * LR::len * sizeof(C);
    static constexpr bool DB = 2 * tile <= 75 * 1024;  // two work-groups per CU
    static constexpr size_t lds = row > (DB ? 2 : 1) * tile ? row : (DB ? 2 : 1) * tile;
    static constexpr int row_units = NX / LPW;  // work-groups a row phase can use
};

template <typename C, int NX, int NY>
__global__ __launch_bounds__((LoopShape<C, NX, NY>::BT)) void slice_loop_kernel(LoopArgs<C> p) {
    using Re = typename real_of<C>::type;
    using S = LoopShape<C, NX, NY>;
    using PR = typename S::PR;
    using PC = typename S::PC;
    constexpr int T = PR::T, E = NY / T, LPW = S::LPW, Tc = PC::T, Ec = NX / Tc, TW = S::TW;
    static_assert(64 % T == 0 && NX % LPW == 0 && NY % TW == 0, "rows inside a wavefront, whole units");
    extern __shared__ __align__(16) unsigned char smem_raw[];
    __shared__ int gave_up;
    C* smem = reinterpret_cast<C*>(smem_raw);
    const int tid = threadIdx.x;
    const int team = (int)blockIdx.x / p.team, m = (int)blockIdx.x % p.team, nteam = (int)gridDim.x / p.team;
    unsigned* const flags = p.flags + (size_t)team * p.team;
    const unsigned dead = __hip_atomic_load(p.dead, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);

    // row phase: line lw, position t
    const int lw = tid / T, t = tid % T;
    using LR = typename S::LR;
    const typename LR::View rlds[2] = {{smem + lw * LR::len}, {smem + lw * LR::len}};
    TwReg<PR, C> twr;
    load_twiddles<PR>(twr, t, p.twy);
    unsigned inb = 0;
#pragma unroll
    for (int e = 0; e < E; ++e) inb |= (t + e * T < p.blo || t + e * T >= NY - p.bhi ? 1u : 0u) << e;
    // column phase: column cw of a tile, position tc
    const int cw = tid % TW, tc = tid / TW;
    using LC = typename S::LC;
    const typename LC::View clds[2] = {{smem + cw}, {smem + LC::len + cw}};
    TwReg<PC, C> twc;
    load_twiddles<PC>(twc, tc, p.twx);
    float kx2[Ec];
#pragma unroll
    for (int e = 0; e < Ec; ++e) kx2[e] = p.kx2[tc + e * Tc];
    constexpr int groups = NY / TW;
    const int blo = p.blo, bhi = NY - p.bhi;
    const int gl = min((blo + TW - 1) / TW, groups), gr = max(bhi / TW, gl), ngl = gl + max(groups - gr, 0);

    constexpr int img_bytes = NX * NY * (int)sizeof(C);
    unsigned phase = p.epoch;
    // the team's barrier; `ahead` issues loads that do not depend on it.
    // False: a wait gave up, every thread of the work-group leaves.  The
    // work-group barriers order LDS only: each wavefront has waited for its
    // own stores before the first, and loads in flight stay so.
    auto sync = [&](auto&& ahead) -> bool {
        ++phase;
        __builtin_amdgcn_s_waitcnt(0);
        lds_barrier();
        if (tid == 0) __hip_atomic_store(&flags[m], phase, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        ahead();
        if (tid < 64) {
            for (int i = tid; i < p.team; i += 64) {
                unsigned n = 0;
                while ((int)(__hip_atomic_load(&flags[i], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) - phase) < 0) {
                    if (++n >= p.spin) {
                        gave_up = 1;
                        break;
                    }
                }
            }
        }
        asm volatile("" ::: "memory");
        lds_barrier();
        if (gave_up) {
            if (tid == 0) {
                __hip_atomic_store(p.dead, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                *p.status = 1;
            }
            return false;
        }
        return true;
    };

    if (tid == 0) gave_up = dead != 0;  // (read after the first barrier)
    for (int b = team; b < p.nb; b += nteam) {
        C* img = p.psi + (long long)b * NX * NY;
        const C* in0 = p.src ? p.src + b * p.src_bstride : img;
        int s1 = p.s1;
        if (p.jobs) {
            const LoopJob<C> j = p.jobs[b];
            img = j.psi;
            in0 = j.src;
            s1 = j.nslice;
        }
        img = uniform_ptr(img);
        in0 = uniform_ptr(in0);
        s1 = __builtin_amdgcn_readfirstlane(s1);
        const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(img, 0, img_bytes, kBufWord3);
        C tr[E], px[Ec];
        auto layer_of = [&](int s) -> long long { return p.slices ? p.slices[s].x : s; };
        auto prop_of = [&](int s) -> long long { return p.slices ? p.slices[s].y : 0; };
        auto load_tr = [&](int s, int u) {
            const C* q = p.jobs ? p.trans_tab[(long long)s * p.nb + b] : p.trans + layer_of(s) * (NX * NY);
            q = uniform_ptr(q) + (u * LPW + lw) * NY + t;
#pragma unroll
            for (int e = 0; e < E; ++e) tr[e] = q[e * T];
        };
        auto px_of = [&](int s) {
            return uniform_ptr(p.jobs ? p.prop_tab[(long long)s * p.nb + b] : p.px + prop_of(s) * NX);
        };
        auto load_px = [&](int s) {
            const C* q = px_of(s) + tc;
#pragma unroll
            for (int e = 0; e < Ec; ++e) px[e] = q[e * Tc];
        };
        if (m < S::row_units) load_tr(p.s0, m);
        for (int s = p.s0; s < s1; ++s) {
            const bool all = s == p.s0 && p.first_all, real = s == p.s0 && p.first_real;
            // [IFFT_y], x scaled transmission, FFT_y (row_sweep)
            for (int u = m; u < S::row_units; u += p.team) {
                const unsigned row = (unsigned)(u * LPW + lw) * NY + t;
                C a[E];
                if (all) {  // (a branch of its own: one mask for both costs 0.4 us per slice)
                    const C* q = in0 + row;
#pragma unroll
                    for (int e = 0; e < E; ++e) a[e] = q[e * T];
                } else {
#pragma unroll
                    for (int e = 0; e < E; ++e)
                        a[e] = buf_load<C, kScopeDev>(
                            rs, ((inb >> e) & 1u) ? (row + e * T) * (unsigned)sizeof(C) : kBufDrop);
                }
                if (u != m) load_tr(s, u);
                if (real) {
#pragma unroll
                    for (int e = 0; e < E; ++e) a[e] = cmul(a[e], tr[e]);
                } else {
                    fft_line<PR, -1, true>(a, t, rlds, twr);
#pragma unroll
                    for (int e = 0; e < E; ++e) a[e] = cmul(a[e], cscale(tr[e], p.inv));
                }
                fft_line<PR, 1, true>(a, t, rlds, twr);
#pragma unroll
                for (int e = 0; e < E; ++e)
                    buf_store<kScopeDev>(a[e], rs, ((inb >> e) & 1u) ? (row + e * T) * (unsigned)sizeof(C) : kBufDrop);
            }
            if (!sync([&] { load_px(s); })) return;
            auto next_tr = [&] {
                if (s + 1 < s1 && m < S::row_units) load_tr(s + 1, m);
            };
            if (m >= ngl) next_tr();
            // FFT_x, propagator and band limit, IFFT_x (col_sweep)
            const C* const py = p.jobs ? px_of(s) + NX : p.py + prop_of(s) * NY;
            for (int k = m; k < ngl; k += p.team) {
                const int g = k < gl ? k : k - gl + gr, y = g * TW + cw;
                const bool live = y < blo || y >= bhi;
                const unsigned col = (unsigned)tc * NY + (unsigned)y;
                const float ky2 = p.ky2[y];
                const C fy = py[y];
                C a[Ec];
#pragma unroll
                for (int e = 0; e < Ec; ++e)
                    a[e] = buf_load<C, kScopeDev>(rs, live ? (col + e * Tc * NY) * (unsigned)sizeof(C) : kBufDrop);
                // the next slice's transmission row, a phase before its use (a
                // new layer comes from HBM); behind the tile in issue order, so
                // that waiting for the tile does not wait for it
                if (k == m) next_tr();
                fft_line<PC, 1, false, S::DB, 0>(a, tc, clds, twc);
#pragma unroll
                for (int e = 0; e < Ec; ++e) {
                    if (kx2[e] + ky2 < p.k2max) a[e] = cmul(cmul(a[e], fy), px[e]);
                    else a[e] = mk<C>((Re)0, (Re)0);
                }
                fft_line<PC, -1, false, S::DB, PC::P - 1>(a, tc, clds, twc);
#pragma unroll
                for (int e = 0; e < Ec; ++e)
                    buf_store<kScopeDev>(a[e], rs, live ? (col + e * Tc * NY) * (unsigned)sizeof(C) : kBufDrop);
            }
            if (s + 1 == s1 && p.mixed) break;
            if (!sync([] {})) return;
        }
        if (p.mixed) {
            __syncthreads();  // the next wave's rows reuse the columns' LDS
            continue;
        }
        // the exit wave: IFFT_y, every element stored
        for (int u = m; u < S::row_units; u += p.team) {
            const unsigned row = (unsigned)(u * LPW + lw) * NY + t;
            C a[E];
#pragma unroll
            for (int e = 0; e < E; ++e)
                a[e] = buf_load<C, kScopeDev>(rs, ((inb >> e) & 1u) ? (row + e * T) * (unsigned)sizeof(C) : kBufDrop);
            fft_line<PR, -1, true>(a, t, rlds, twr);
#pragma unroll
            for (int e = 0; e < E; ++e) buf_store(cscale(a[e], p.inv), rs, (row + e * T) * (unsigned)sizeof(C));
        }
    }
}

}  // namespace msx
