// Two fused steps in one pass over the population array (k_pair), from
// the state an even AA step leaves (site y's post-collision population l in
// its own slot opp(l)) in p.f to the same form in p.f2. Included by
// lb_kernels.h.
//
// A step by itself streams 19 populations in and 19 out per site and is bound
// by that traffic (256^3 FP64: 0.89 ms, 5.7 TB/s) or, on small lattices, by
// the latency of its chain of loads and the launch. Here a workgroup holds a tile of
// columns (j,k) with a one-column rim and sweeps it along i, one plane per
// iteration:
//   first step   every column, rim included, gathers plane i from p.f and
//                collides; the results go to LDS in the storage type, so they
//                round as a store to memory would;
//   second step  the inner columns of plane i - 1 gather from LDS, collide
//                and store to p.f2.
// Only the first step of the rim is computed twice (by this tile and by its
// neighbour), so two steps move little more than one step's bytes. Results
// are bit-identical to single steps. Measured (ms per step, single / paired):
// 256^3 channel FP64 0.893 / 0.564 (a pair moves 5.46 GB past L2, 1.07 of its
// populations, as L2 catches 40% of the rims: 4.8 TB/s, 0.83 of the copy),
// FP32 0.454 / 0.299 and FP16 0.265 / 0.274 (VALU instructions issue in 75 and
// 85% of the CUs' busy cycles; FP64 35%); 512x128x128 duct FP64 0.433 / 0.295;
// 32x34x8 channel 0.0190 / 0.0044.
//
// LDS. A population with c_i = -1 is needed in the iteration it is made in,
// one with c_i = 0 in the next, one with c_i = +1 in the one after, so the
// three kinds sit in rings of 2, 2 and 3 planes (the second plane of the
// c_i = -1 ring serves bounce-back, which reads the site's own populations).
// The rest population and the two along i stay in their own column, in
// registers. That is 36 values per column: with 512 columns of 8 bytes
// 144 KiB, one workgroup per CU. The loads of the next plane are issued
// before the second step computes, so memory works during both collisions.
//
// Sparse layout (PAIR_SPARSE). The same sweep over the cells of a tile; only
// fluid sites load and store. The compact indices around come from LDS too
// (18 of them per site; the single step reads 9 bytes of codes), a ring of
// four planes, each loaded an iteration ahead. Tiles' rows start and end
// anywhere in a line: L2 joins the stores (1.80 GB written for 1.72 GB of
// populations on 384x192x192 cells of 20% solid). ms per step there, single /
// paired: FP64 0.592 / 0.458; 256x128x128 0.169 / 0.146. The indices take the
// 16 KiB of LDS that FP64's rings leave of 160.
#pragma once
#include <type_traits>

namespace lb {

// Ring slot of population l among those of its kind that cross columns.
LBD constexpr int ring_slot(int l) {
    return CI[l] < 0 ? (l < 2 ? l : l - 1)       // 0, 1, 3, 4
           : CI[l] == 0 ? (l < 9 ? l - 5 : l - 6)  // 5-8, 10-13
                        : (l < 16 ? l - 14 : l - 15);  // 14, 15, 17, 18
}
LBD constexpr bool in_ring(int l) { return l != 2 && l != REST && l != 16; }
constexpr int RING_M = 0, RING_0 = 8, RING_P = 24, RING_SLOTS = 36;

// Orders this workgroup's LDS accesses around a barrier; global loads in
// flight stay in flight.
LBD void lds_barrier() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

template <int P> LBD typename Var<P>::TC from_ts(typename Var<P>::TS v, float inv_scale) {
    if constexpr (P == LB_FP16_STORAGE) return (float)v * inv_scale;
    else return v;
}
template <int P> LBD typename Var<P>::TS to_ts(typename Var<P>::TC v, float scale) {
    if constexpr (P == LB_FP16_STORAGE) return (_Float16)(v * scale);
    else return (typename Var<P>::TS)v;
}

// Ladd's term (ladd_apply) on the moving links w of a site whose walls move
// with v: opposite links take the same product, with opposite signs, so nine
// products serve all 18.
template <class TC, int... Ls>
LBD void ladd_links(TC* f, uint32_t w, TC den, const double* v, std::integer_sequence<int, Ls...>) {
    auto pair = [&](auto link) {
        constexpr int L = decltype(link)::value, O = opp(L);
        const TC t = ladd_term<TC>(L, den, (TC)ladd_combine<L>(v));
        if (w >> link_slot(L) & 1u) f[L] += t;
        if (w >> link_slot(O) & 1u) f[O] -= t;
    };
    (pair(std::integral_constant<int, Ls>{}), ...);
}

// FEAT: what there is besides fluid, stationary walls and periodic faces:
// PAIR_MOVING (moving walls), PAIR_FULL (Zou-He faces, symmetric y / z faces,
// a per-site acceleration), or both.
template <int P, int RLX, int FEAT>
__global__ __launch_bounds__(pair_threads(P)) void k_pair(StepParams p, PairParams q) {
    using TS = typename Var<P>::TS;
    using TC = typename Var<P>::TC;
    constexpr bool SH = Var<P>::SH, FULL = (FEAT & PAIR_FULL) != 0, MOV = (FEAT & PAIR_MOVING) != 0;
    constexpr bool SP = (FEAT & PAIR_SPARSE) != 0;
    constexpr int NT = pair_threads(P), NC = pair_cells(P);
    // The gather's loads that are issued before the first step; the others
    // follow it, and have the second step's time to arrive. Measured (ms per
    // step, all 19 first / 14): FP32 256^3 0.322 / 0.300; dense FP64 256^3,
    // which waits for memory as it is, 0.566 / 0.595; with the sparse sweeps as
    // long as the dense ones, FP32 256x128x128 0.103 / 0.090 and FP64
    // 384x192x192 0.501 / 0.492.
    constexpr int FIRST = (P == LB_FP64 && !SP) || (MOV && FULL) ? Q : 14;
    auto in_part = [](int part, int l) constexpr { return part < 0 || (l < FIRST) == (part == 0); };
    __shared__ TS ring[RING_SLOTS * NT];
    __shared__ uint32_t idx[SP ? 4 * NC : 1];
    static_assert(sizeof(ring) + (SP ? sizeof(idx) : 0) <= 160 * 1024, "a CU has 160 KiB of LDS");

    // tile and chunk of this workgroup: each XCD takes a contiguous range, so
    // that neighbouring tiles, which read each other's rims, share its L2
    const uint32_t per = gridDim.x >> 3;
    const uint32_t w = (blockIdx.x & 7u) * per + (blockIdx.x >> 3);
    if (w >= q.total) return;
    const uint32_t tk = w % q.ntk, rest = w / q.ntk, tj = rest % q.ntj, ch = rest / q.ntj;
    const int k0 = (int)tk * q.TK, j0 = (int)tj * q.TJ;
    const int nx = p.d.nx, ny = p.d.ny, nz = p.d.nz;
    const int i0 = (int)ch * q.chunk, i1 = min(i0 + q.chunk, nx);

    // this thread's column, wrapped through periodic y / z faces
    const int EK = q.TK + 2 * q.hk;
    const int t = (int)threadIdx.x;
    const int jj = t / EK, kk = t - jj * EK;
    const int j = j0 - q.hj + jj, k = k0 - q.hk + kk;
    const bool pery = p.d.bc[2] == PERIODIC, perz = p.d.bc[4] == PERIODIC;
    int jw = j, kw = k;
    if (pery) jw = j < 0 ? j + ny : j >= ny ? j - ny : j;
    if (perz) kw = k < 0 ? k + nz : k >= nz ? k - nz : k;
    const bool col = jj < q.TJ + 2 * q.hj && j <= ny && k <= nz && jw >= 0 && jw < ny && kw >= 0 && kw < nz;
    if (!col) jw = kw = 0;  // addresses only; the column's mask reads as zero
    const bool inner = col && jj >= q.hj && jj < q.hj + q.TJ && kk >= q.hk && kk < q.hk + q.TK && j < ny && k < nz;
    // byte offsets of the upstream rows and of k - c_k, within a plane
    // (through a wall or a symmetric face: the column's own)
    const uint32_t rsb = (uint32_t)(p.rs * (int64_t)sizeof(TS));
    const int jl = jw > 0 ? jw - 1 : pery ? ny - 1 : 0, jh = jw < ny - 1 ? jw + 1 : pery ? 0 : ny - 1;
    const int kl = kw > 0 ? kw - 1 : perz ? nz - 1 : 0, kh = kw < nz - 1 ? kw + 1 : perz ? 0 : nz - 1;
    const uint32_t rowo[3] = {(uint32_t)jh * rsb, (uint32_t)jw * rsb, (uint32_t)jl * rsb};  // by c_j + 1
    const uint32_t ko[3] = {(uint32_t)kh * (uint32_t)sizeof(TS), (uint32_t)kw * (uint32_t)sizeof(TS),
                            (uint32_t)kl * (uint32_t)sizeof(TS)};  // by c_k + 1
    const uint32_t own = rowo[1] + ko[1];
    // the same in columns of the tile
    const int so[3] = {jw < ny - 1 || pery ? -EK : 0, 0, jw > 0 || pery ? EK : 0};
    const int sk[3] = {kw < nz - 1 || perz ? -1 : 0, 0, kw > 0 || perz ? 1 : 0};
    // symmetric faces: links of this column that a mirror sends back
    bool sy[3] = {false, false, false}, sz[3] = {false, false, false};  // by c + 1
    if (FULL) {
        sy[2] = p.d.bc[2] == SYMMETRIC && jw == 0;
        sy[0] = p.d.bc[3] == SYMMETRIC && jw == ny - 1;
        sz[2] = p.d.bc[4] == SYMMETRIC && kw == 0;
        sz[0] = p.d.bc[5] == SYMMETRIC && kw == nz - 1;
    }
    const bool mir = FULL && (sy[0] || sy[2] || sz[0] || sz[2]);

    const int64_t psb = p.ps * (int64_t)sizeof(TS);
    const int64_t plane = (int64_t)ny * rsb;
    const uint32_t cplane = (uint32_t)ny * (uint32_t)p.d.nzp;
    const uint32_t ccol = (uint32_t)jw * (uint32_t)p.d.nzp + (uint32_t)kw;
    const bool perx = p.d.bc[0] == PERIODIC;
    // lattice plane of i, or -1 outside a wall
    auto wrapx = [&](int i) -> int {
        const int w = perx ? (i < 0 ? i + nx : i >= nx ? i - nx : i) : i;
        return w >= 0 && w < nx ? w : -1;
    };
    auto mask_of = [&](int ip) -> uint32_t { return ip >= 0 && col ? p.mask[(uint32_t)ip * cplane + ccol] : 0u; };
    const TC rho0 = (TC)p.rho0;
    const TC* A = (const TC*)p.acc;
    const int64_t nq = p.nq;
    TC prm[2] = {(TC)p.prm[0], (TC)p.prm[1]};

    // The first step's gather (populations as stored) of the plane ip at F,
    // between the planes at Fl and Fh: one load per link, of a scalar base and
    // a 32-bit lane offset. Waves with bounce-back or mirrored links choose
    // each lane's offset; own populations lie beyond the plane before's from
    // the same base. Across a periodic x face, where the planes do not follow
    // each other, links along i that bounce back load again instead. (A second
    // set of loads for the other waves would not do: the compiler waits for
    // whatever may be in flight to a register before it loads it again, and
    // that counts the stores.) The asm keeps the strides from being
    // multiplied out ahead of the loop, into registers it does not have.
    TS g[Q] = {};
    auto gather = [&](auto part, const char* Fl, const char* F, const char* Fh, int ip, uint32_t m) {
        constexpr int PT = decltype(part)::value;
        const bool follow = !perx || (ip > 0 && ip < nx - 1);
        if (!(m & M_FLUID)) return;
        uint32_t sb = (uint32_t)psb, pb = (uint32_t)plane;
        asm volatile("" : "+s"(sb), "+s"(pb));
        const char* const bl = uniform_ptr(follow ? F - plane : Fl);
        const char* const bh = uniform_ptr(follow ? F : Fh);
        const char* const b0 = uniform_ptr(F);
        const uint32_t dh = follow ? pb : 0u;
        uint32_t off[Q];
#pragma unroll
        for (int l = 0; l < Q; ++l)
            off[l] = rowo[CJ[l] + 1] + ko[CK[l] + 1] + ((uint32_t)opp(l) * sb + (CI[l] < 0 ? dh : 0u));
        const bool some = __ballot((m & M_LINKS) != 0 || mir) != 0;
        if (some) {
#pragma unroll
            for (int l = 0; l < Q; ++l) {
                if (l == REST || !in_part(PT, l)) continue;
                if (FULL && (CJ[l] || CK[l])) {  // the mirrored population's slot
                    const bool y = CJ[l] && sy[CJ[l] + 1], z = CK[l] && sz[CK[l] + 1];
                    uint32_t d = 0;
                    if (y) d = (uint32_t)(l - mirror(l, 1)) * sb;
                    if (z) d = (uint32_t)(l - mirror(l, 2)) * sb;
                    if (y && z) d = (uint32_t)(l - mirror(mirror(l, 2), 1)) * sb;
                    off[l] += d;
                }
                const uint32_t mine = own + ((uint32_t)l * sb + (CI[l] > 0 && follow ? pb : 0u));
                off[l] = m & (1u << l) ? mine : off[l];
            }
        }
#pragma unroll
        for (int l = 0; l < Q; ++l)
            if (in_part(PT, l)) g[l] = *(const TS*)((CI[l] > 0 ? bl : CI[l] < 0 ? bh : b0) + off[l]);
        if (some && !follow) {
#pragma unroll
            for (int l = 0; l < Q; ++l)
                if (CI[l] != 0 && in_part(PT, l) && (m & (1u << l))) g[l] = *(const TS*)(b0 + (own + (uint32_t)l * sb));
        }
    };
    // The same in the sparse layout: the compact indices of the planes around
    // are in LDS as sp_elem gives them (a ring of four planes, I0 the plane
    // before). 32-bit element offsets reach the whole array (lb_finalize).
    const int EX = EK + 2, xc = (jj + 1) * EX + kk + 1;
    uint32_t nN = 0, nA = 0, nB = 0;  // own sp_elem in planes i + 1, i, i - 1
    auto gather_sp = [&](auto part, const uint32_t* I0, const uint32_t* I1, const uint32_t* I2, uint32_t m) {
        constexpr int PT = decltype(part)::value;
        if (!(m & M_FLUID)) return;
        uint32_t np = (uint32_t)p.ps;
        asm volatile("" : "+s"(np));
        const TS* const b = uniform_ptr((const TS*)p.f);
        nN = I1[xc];
#pragma unroll
        for (int l = 0; l < Q; ++l) {
            if (!in_part(PT, l)) continue;
            uint32_t e = (uint32_t)opp(l) * np;
            if (l == REST) {
                e += nN;
            } else {
                e += (CI[l] > 0 ? I0 : CI[l] < 0 ? I2 : I1)[xc - CJ[l] * EX - CK[l]];
                if (FULL && (CJ[l] || CK[l])) {
                    const bool y = CJ[l] && sy[CJ[l] + 1], z = CK[l] && sz[CK[l] + 1];
                    uint32_t d = 0;
                    if (y) d = (uint32_t)(l - mirror(l, 1)) * np;
                    if (z) d = (uint32_t)(l - mirror(l, 2)) * np;
                    if (y && z) d = (uint32_t)(l - mirror(mirror(l, 2), 1)) * np;
                    e += d;
                }
                const uint32_t mine = (uint32_t)l * np + nN;
                e = m & (1u << l) ? mine : e;
            }
            g[l] = b[e];
        }
    };
    // Cells of those planes that this thread keeps: clamped to the lattice
    // beyond a wall or a symmetric face, where the mirrored populations are.
    uint32_t cell[2] = {0, 0}, cv[2] = {0, 0};
    if (SP) {
#pragma unroll
        for (int e = 0; e < 2; ++e) {
            const int y = (t + e * NT) / EX, z = (t + e * NT) - y * EX;
            int cj = j0 - q.hj - 1 + y, ck = k0 - q.hk - 1 + z;
            if (pery) cj = cj < 0 ? cj + ny : cj >= ny ? cj - ny : cj;
            if (perz) ck = ck < 0 ? ck + nz : ck >= nz ? ck - nz : ck;
            cj = min(max(cj, 0), ny - 1);
            ck = min(max(ck, 0), nz - 1);
            cell[e] = (uint32_t)cj * (uint32_t)p.d.nzp + (uint32_t)ck;
        }
    }
    auto load_idx = [&](int i) {
        const uint32_t* const b = uniform_ptr(p.cidx + (uint32_t)max(wrapx(i), 0) * cplane);
#pragma unroll
        for (int e = 0; e < 2; ++e) cv[e] = b[cell[e]];
    };
    auto keep_idx = [&](int slot) {
#pragma unroll
        for (int e = 0; e < 2; ++e) idx[slot * NC + e * NT + t] = sp_elem(cv[e], p.bsh, p.bmul);
    };
    // One collision, on the streamed populations f of the site (ip, jw, kw).
    // What is loaded in a branch is waited for there: a wait behind it would
    // be for everything in flight on the other path too. Returns the density
    // as stored.
    auto site = [&](TC* f, uint32_t m, int ip, TC* vel) -> double {
        const uint32_t c = (uint32_t)ip * cplane + ccol;
        if (FULL && (m & M_ZH_ANY)) zouhe_site<TC, SH>(p, m, ip, jw, kw, rho0, f);
        TC acc[3];
#pragma unroll
        for (int a = 0; a < 3; ++a) acc[a] = (TC)p.g[a];
        if (FULL && A) {
            TC s[3] = {A[c], A[nq + c], A[2 * nq + c]};
            asm volatile("" : "+v"(s[0]), "+v"(s[1]), "+v"(s[2]));
#pragma unroll
            for (int a = 0; a < 3; ++a) acc[a] += s[a];
        }
        TC ds;
        const TC den = collide<RLX, TC, SH, P == LB_FP32_SHIFTED, true>(f, acc, prm, rho0, vel, ds);
        return SH ? p.rho0 + (double)ds : (double)den;
    };

    // Ladd's term of a moving site: its wall velocity comes from the few in q,
    // its moving links in w and, for the first step, the density rho are
    // loaded with the plane before
    double rho = 0.0, rhoN = 0.0;
    uint32_t wB = 0, wA = 0, wN = 0;  // of planes i - 1, i, i + 1
    auto load_ladd = [&](int ip, uint32_t m) {
        if (!(m & M_MOVING)) return;
        const uint32_t c = (uint32_t)ip * cplane + ccol;
        wN = q.mov[c];
        rhoN = q.rho_in[c];
    };
    auto ladd = [&](TC* f, uint32_t w, TC den) {
        double v[3] = {q.wall[0][0], q.wall[0][1], q.wall[0][2]};
#pragma unroll
        for (int e = 1; e < PAIR_WALLS; ++e)
#pragma unroll
            for (int a = 0; a < 3; ++a) v[a] = (w >> 18) == (uint32_t)e ? q.wall[e][a] : v[a];
        ladd_links(f, w, den, v, std::make_integer_sequence<int, REST>{});
    };

    // Waits for the gather's loads here rather than at their first use.
    auto arrive = [&] {
#pragma unroll
        for (int l = 0; l < Q; ++l) asm volatile("" : "+v"(g[l]));
        if (MOV) asm volatile("" : "+v"(wN), "+v"(rhoN));
        if (SP) asm volatile("" : "+v"(cv[0]), "+v"(cv[1]));
    };

    // lattice planes of i - 1, i, i + 1, their places in p.f and their masks
    int ipB = -1, ip = wrapx(i0 - 1), ipN = wrapx(i0);
    auto place = [&](int w) { return (const char*)p.f + (int64_t)max(w, 0) * plane; };
    const char *FA = place(ip), *FN = place(ipN);
    uint32_t mB = 0, mA = mask_of(ip), mN = mask_of(ipN);
    double dB = 0.0, dA = 0.0;                             // density of planes i - 1, i
    TS r0 = TS(0), m1 = TS(0), p1 = TS(0), p2 = TS(0);  // plane i - 1: rest, l = 2, l = 16; plane i - 2: l = 16
    if (MOV) load_ladd(ip, mA);
    const std::integral_constant<int, -1> all;
    const std::integral_constant<int, 0> part0;
    const std::integral_constant<int, 1> part1;
    if constexpr (SP) {
        load_idx(i0 - 2);
        keep_idx(3);
        load_idx(i0 - 1);
        keep_idx(0);
        load_idx(i0);
        keep_idx(1);
        load_idx(i0 + 1);
        keep_idx(2);
        lds_barrier();
        gather_sp(all, idx + 3 * NC, idx, idx + NC, mA);
        nA = nN;
        load_idx(i0 + 2);
        lds_barrier();
    } else {
        gather(all, place(wrapx(i0 - 2)), FA, FN, ip, mA);
    }
    arrive();
    wA = wN;
    rho = rhoN;
    int r2 = 0, r3 = 0;  // ring planes of i
    for (int i = i0 - 1; i <= i1; ++i) {
        // the next plane's loads are in flight during both collisions
        TC f[Q];
#pragma unroll
        for (int l = 0; l < Q; ++l) f[l] = from_ts<P>(g[l], p.inv_scale);
        const int ipNN = i < i1 ? wrapx(i + 2) : -1;
        const char* const FNN = place(ipNN);
        uint32_t mNN = mask_of(ipNN);
        if (MOV) load_ladd(ipN, mN);
        // the gather of plane i + 1, one part at a time
        const int s0 = i - i0 + 1;  // ring plane of i in idx
        auto load_next = [&](auto part) {
            if (i >= i1) return;
            if constexpr (SP)
                gather_sp(part, idx + (s0 & 3) * NC, idx + (s0 + 1 & 3) * NC, idx + (s0 + 2 & 3) * NC, mN);
            else
                gather(part, FA, FN, FNN, ipN, mN);
        };
        load_next(part0);
        __builtin_amdgcn_sched_barrier(0);

        // ---- first step, plane i ----
        TS s9 = TS(0), s2 = TS(0), s16 = TS(0);
        if (mA & M_FLUID) {
            TC vel[3];
            if (MOV && (mA & M_MOVING)) ladd(f, wA, (TC)rho);
            dA = site(f, mA, ip, vel);
            s9 = to_ts<P>(f[REST], p.scale);
            s2 = to_ts<P>(f[2], p.scale);
            s16 = to_ts<P>(f[16], p.scale);
        }
        lds_barrier();  // the second step's reads of the planes overwritten here are done
        TS* const wm = ring + (RING_M + 4 * r2) * NT + t;
        TS* const w0 = ring + (RING_0 + 8 * r2) * NT + t;
        TS* const wp = ring + (RING_P + 4 * r3) * NT + t;
        if (mA & M_FLUID) {
#pragma unroll
            for (int l = 0; l < Q; ++l) {
                if (!in_ring(l)) continue;
                TS* const d = CI[l] < 0 ? wm : CI[l] == 0 ? w0 : wp;
                d[ring_slot(l) * NT] = to_ts<P>(f[l], p.scale);
            }
        }
        if (SP) keep_idx(s0 + 3 & 3);
        lds_barrier();
        if (SP) load_idx(i + 4);
        load_next(part1);
        __builtin_amdgcn_sched_barrier(0);
        // ---- second step, plane i - 1 ----
        const bool second = i > i0 && inner && (mB & M_FLUID);
        TC h[Q];
        if (second) {
            const int r3a = r3 == 0 ? 2 : r3 - 1, r3b = r3 == 2 ? 0 : r3 + 1;  // planes i - 1, i - 2
            const TS* const rm = wm;                                                // c_i = -1 of plane i
            const TS* const rm1 = ring + (RING_M + 4 * (r2 ^ 1)) * NT + t;          // ... of plane i - 1
            const TS* const r01 = ring + (RING_0 + 8 * (r2 ^ 1)) * NT + t;          // c_i = 0 of plane i - 1
            const TS* const rp1 = ring + (RING_P + 4 * r3a) * NT + t;               // c_i = +1 of plane i - 1
            const TS* const rp2 = ring + (RING_P + 4 * r3b) * NT + t;               // ... of plane i - 2
            TS v[Q];
            v[REST] = r0;
            v[2] = s2;
            v[16] = p2;
            if (__ballot((mB & M_LINKS) != 0 || mir) == 0) {
#pragma unroll
                for (int l = 0; l < Q; ++l) {
                    if (!in_ring(l)) continue;
                    const TS* const b = CI[l] < 0 ? rm : CI[l] == 0 ? r01 : rp2;
                    v[l] = b[ring_slot(l) * NT - CJ[l] * EK - CK[l]];
                }
            } else {
                if (mB & (1u << 2)) v[2] = p1;
                if (mB & (1u << 16)) v[16] = m1;
#pragma unroll
                for (int l = 0; l < Q; ++l) {
                    if (!in_ring(l)) continue;
                    const TS* const b = CI[l] < 0 ? rm : CI[l] == 0 ? r01 : rp2;
                    const TS* const bo = CI[l] > 0 ? rm1 : CI[l] == 0 ? r01 : rp1;
                    const TS* a = b + (ring_slot(l) * NT - so[CJ[l] + 1] - sk[CK[l] + 1]);
                    if (FULL) {
                        const bool y = CJ[l] && sy[CJ[l] + 1], z = CK[l] && sz[CK[l] + 1];
                        int d = 0;
                        if (y) d = (ring_slot(mirror(l, 1)) - ring_slot(l)) * NT;
                        if (z) d = (ring_slot(mirror(l, 2)) - ring_slot(l)) * NT;
                        if (y && z) d = (ring_slot(mirror(mirror(l, 2), 1)) - ring_slot(l)) * NT;
                        a += d;
                    }
                    if (mB & (1u << l)) a = bo + ring_slot(opp(l)) * NT;
                    v[l] = *a;
                }
            }
            TC vel[3];
#pragma unroll
            for (int l = 0; l < Q; ++l) h[l] = from_ts<P>(v[l], p.inv_scale);
            if (MOV && (mB & M_MOVING)) ladd(h, wB, (TC)dB);
            const double den = site(h, mB, ipB, vel);
            const uint32_t c = (uint32_t)ipB * cplane + ccol;
            if (p.store_dv) {
                p.den[c] = den;
                p.vel[c] = (double)vel[0];
                p.vel[nq + c] = (double)vel[1];
                p.vel[2 * nq + c] = (double)vel[2];
            }
            if (MOV && (mB & M_MOVING)) q.rho_out[c] = den;
        }
        // Wait for the next plane's loads here, before the stores: one counter
        // covers both, and after them the wait would be for the stores too.
        arrive();
        asm volatile("" : "+v"(mNN));
        if (second) {
            // Plain stores: L2 joins the lines that two tiles share. With
            // non-temporal ones 256^3 FP64 ran 0.615 ms per step (plain 0.572
            // in the same session) and tiles that split lines 0.968 (33x12x32;
            // 0.751).
            uint64_t step = (uint64_t)psb;
            if constexpr (SP) {
                uint64_t a = (uint64_t)((TS*)p.f2 + nB);
                asm volatile("" : "+s"(step), "+v"(a));
#pragma unroll
                for (int sl = 0; sl < Q; ++sl) {
                    *(__attribute__((address_space(1))) TS*)a = to_ts<P>(h[opp(sl)], p.scale);
                    a += step;
                }
            } else {
                char* G = (char*)p.f2 + (int64_t)ipB * plane;
                uint32_t o = own;
                asm volatile("" : "+s"(step), "+v"(o));  // not multiplied out, nor widened, ahead of the loop
#pragma unroll
                for (int sl = 0; sl < Q; ++sl) {
                    *(TS*)(uniform_ptr(G) + o) = to_ts<P>(h[opp(sl)], p.scale);
                    G += step;
                }
            }
        }
        r0 = s9;
        m1 = s2;
        p2 = p1;
        p1 = s16;
        dB = dA;
        ipB = ip;
        ip = ipN;
        ipN = ipNN;
        FA = FN;
        FN = FNN;
        nB = nA;
        nA = nN;
        wB = wA;
        wA = wN;
        rho = rhoN;
        mB = mA;
        mA = mN;
        mN = mNN;
        r2 ^= 1;
        r3 = r3 == 2 ? 0 : r3 + 1;
    }
}

template <int P, int RLX, int LAYOUT>
static void launch_pair_feat(const StepParams& p, const PairParams& q, int feat, hipStream_t st) {
    const unsigned grid = (q.total + 7) / 8 * 8;
    constexpr int NT = pair_threads(P);
    if (feat == 0) k_pair<P, RLX, LAYOUT><<<grid, NT, 0, st>>>(p, q);
    else if (feat == PAIR_MOVING) k_pair<P, RLX, LAYOUT | PAIR_MOVING><<<grid, NT, 0, st>>>(p, q);
    else if (feat == PAIR_FULL) k_pair<P, RLX, LAYOUT | PAIR_FULL><<<grid, NT, 0, st>>>(p, q);
    else k_pair<P, RLX, LAYOUT | PAIR_MOVING | PAIR_FULL><<<grid, NT, 0, st>>>(p, q);
}

template <int P, int RLX>
static void launch_pair_layout(const StepParams& p, const PairParams& q, int feat, hipStream_t st) {
    if (p.cidx) launch_pair_feat<P, RLX, PAIR_SPARSE>(p, q, feat, st);
    else launch_pair_feat<P, RLX, 0>(p, q, feat, st);
}

template <int P>
void launch_pair_rlx(const StepParams& p, const PairParams& q, int rlx, int feat, hipStream_t st) {
    if (rlx == BGK) launch_pair_layout<P, BGK>(p, q, feat, st);
    else if (rlx == TRT) launch_pair_layout<P, TRT>(p, q, feat, st);
    else launch_pair_layout<P, REGUL>(p, q, feat, st);
}

}  // namespace lb
