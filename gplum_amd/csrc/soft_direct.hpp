// soft_direct.hpp -- the soft force of the functors and of MultiWalk: i-groups against lists
// that the caller gives.
//
// What bounds it: FP32 VALU issue (EP-EP about 45 instructions per pair, no reuse that a
// matrix product could take); for the small calls, latency.  A workgroup of 8 waves takes
// 2 LI i-particles: a wave is LI i-lanes times 64 / LI j-lanes, every lane holds two
// i-particles (half the LDS reads per pair, two independent chains), and the j entries are
// dealt over the 8 * 64 / LI j-lanes of the workgroup.  The partial sums of an i-particle
// thus meet inside one workgroup: no scratch memory, no atomics, a fixed order.  j entries are
// staged 512 or more at a time, the next tile's loads in flight during the pairs of this one.
// Where i-particles abound and the list is short there is nothing to deal: a workgroup of 4 waves
// then takes 256 i-particles, one per lane, and every lane the whole list (direct_wide).
// A lane takes whole quads of consecutive entries, summed in FP32 and the quads in FP64, so a
// result does not depend on the split beyond FP64 rounding: the functors and MultiWalk agree.  (Every
// pair added in FP64: 65536 x 65536 3764 us; quads: see the table at direct_min_wg.)
#pragma once
#include <type_traits>

#include "soft_kernels.hpp"

namespace gplum {

constexpr int DIRECT_BLOCK = 512;
constexpr int DIRECT_IPL = 2;                          // i-particles per lane
constexpr int DIRECT_WAVES = DIRECT_BLOCK / 64;
constexpr int DIRECT_WIDE = 256;                       // lanes, and i-particles, of a workgroup without j-lanes
static_assert(DIRECT_BLOCK >= 8 * 64, "the sums over the waves take a lane each");

// A tile of staged entries: entry k at place (k % 4) * N / 4 + k / 4, so that lanes with
// consecutive quads read consecutive places.
template <int N>
struct DirectTile {
    float4 a[N], b[N], c[N];
    __device__ static int place(int k) { return (k & 3) * (N / 4) + (k >> 2); }
};
struct DirectSums {
    double d[DIRECT_WAVES][4][64];
    int n[DIRECT_WAVES][4][64];
};

// An EP / SP entry as loaded (FP64), staged as FP32 relative to x_ref.
template <class SRC>
struct DirectEP {
    using Src = SRC;
    double x, y, z, m, ro, rs;
    int id, rk;
    __device__ void load(const Src &s, int e) { s.load(e, x, y, z, m, ro, rs, id, rk); }
    template <class TILE>
    __device__ void stage(TILE &T, int t, double x0, double y0, double z0, float) const {
        float xh, xl, yh, yl, zh, zl;
        split(x - x0, xh, xl);
        split(y - y0, yh, yl);
        split(z - z0, zh, zl);
        const float rof = (float)ro, rsf = (float)rs;
        T.a[t] = make_float4(xh, yh, zh, (float)m);
        T.b[t] = make_float4(rof * rof, (rsf * rsf) * 1.0201f, __int_as_float(id), __int_as_float(rk));
        T.c[t] = make_float4(xl, yl, zl, 0.f);
    }
};
template <class SRC, bool QUAD>
struct DirectSP {
    using Src = SRC;
    double m, x, y, z, q[6];
    __device__ void load(const Src &s, int e) { s.load(e, m, x, y, z, q); }
    template <class TILE>
    __device__ void stage(TILE &T, int t, double x0, double y0, double z0, float eps2) const {
        T.a[t] = make_float4((float)(x - x0), (float)(y - y0), (float)(z - z0), (float)m);
        if (QUAD) spj_terms(q, eps2, T.b[t], T.c[t]);
    }
};

// FP64 sums of one i-particle
struct Acc64 {
    double x = 0., y = 0., z = 0., p = 0.;
    int ngb = 0, rank = 0, idmax = ID_MAX_CLEAR, idmin = 2147483647;
};

// All entries of one list: staged tile by tile; the lane's quads of a tile: `pair(place)` for
// each entry and `fold()` at its end.
template <int BLOCK, int NJ, class J, class TILE, class PAIR, class FOLD>
__device__ inline void direct_list(const typename J::Src &src, int begin, int n, int j0, TILE &T, double x0, double y0,
                                   double z0, float eps2, PAIR pair, FOLD fold) {
    constexpr int N = sizeof(T.a) / sizeof(T.a[0]), Q = N / 4, E = N / BLOCK;
    const int t = (int)threadIdx.x;
    J next[E];
#pragma unroll
    for (int e = 0; e < E; e++)
        if (t + e * BLOCK < n) next[e].load(src, begin + t + e * BLOCK);
    for (int base = 0; base < n; base += N) {
        const int cnt = min(N, n - base);
        __syncthreads();
#pragma unroll
        for (int e = 0; e < E; e++)
            if (t + e * BLOCK < cnt) next[e].stage(T, TILE::place(t + e * BLOCK), x0, y0, z0, eps2);
        __syncthreads();
#pragma unroll
        for (int e = 0; e < E; e++) {
            const int k = base + N + t + e * BLOCK;
            if (k < n) next[e].load(src, begin + k);
        }
        int q = j0;
        for (int r = (cnt >> 2) / NJ; r > 0; r--, q += NJ) {
#pragma unroll 2
            for (int c = 0; c < 4; c++) pair(c * Q + q);
            fold();
        }
        if (4 * q < cnt) {
            for (int c = 0; c < 4; c++)
                if (4 * q + c < cnt) pair(c * Q + q);
            fold();
        }
    }
}

// LI: i-lanes of a wave, 2 i-particles each; DIRECT_WIDE: the workgroup's, one each.
// groups: one per workgroup, of at most IPL LI i-particles; nullptr: workgroup b takes the i-particles
// from IPL LI b on of `one` (ni in all, relative to the first).
constexpr int direct_block(int li) { return li == DIRECT_WIDE ? DIRECT_WIDE : DIRECT_BLOCK; }
constexpr int direct_ipl(int li) { return li == DIRECT_WIDE ? 1 : DIRECT_IPL; }
template <int MODE, int LI, class JE, class JS>
__global__ __launch_bounds__(direct_block(LI)) void k_direct_f32(const SoftGroup *__restrict__ groups, SoftGroup one, SrcEPI is,
                                                                  typename JE::Src je, typename JS::Src js, SinkForce out,
                                                                  float eps2) {
    constexpr int BLOCK = direct_block(LI), IPL = direct_ipl(LI), NJ = BLOCK / LI;
    using Tile = DirectTile<(4 * NJ > BLOCK ? 4 * NJ : BLOCK)>;                 // a quad for every j-lane
    __shared__ __align__(16) char s_mem[NJ == 1 || sizeof(Tile) > sizeof(DirectSums) ? sizeof(Tile) : sizeof(DirectSums)];
    Tile &T = *reinterpret_cast<Tile *>(s_mem);
    const int t = (int)threadIdx.x, lane = t & 63;
    const int w = __builtin_amdgcn_readfirstlane(t >> 6);
    const int il = NJ == 1 ? t : lane % LI, j0 = NJ == 1 ? 0 : w * (64 / LI) + lane / LI;
    SoftGroup G = one;
    if (groups) {
        G = groups[blockIdx.x];
    } else {
        G.i_begin = (int)blockIdx.x * (IPL * LI);
        G.ni = min(IPL * LI, one.ni - G.i_begin);
    }

    double x0, y0, z0;
    {
        double ro, rs;
        int id, rk;
        is.load(G.i_ref, x0, y0, z0, ro, rs, id, rk);
    }
    // a lane past the last i-particle computes a value that is not written
    IState I[IPL];
    Acc64 a[IPL];
#pragma unroll
    for (int u = 0; u < IPL; u++) {
        const int i = il + u * LI;
        I[u] = IState{1e18f, 1e18f, 1e18f, 0.f, 0.f, 0.f, 0.f, -1.f, -1, 0};
        if (i < G.ni) {
            double x, y, z, ro, rs;
            is.load(G.i_begin + i, x, y, z, ro, rs, I[u].id, I[u].rank);
            split(x - x0, I[u].xh, I[u].xl);
            split(y - y0, I[u].yh, I[u].yl);
            split(z - z0, I[u].zh, I[u].zl);
            const float rof = (float)ro, rsf = (float)rs;
            I[u].ro2 = rof * rof;
            I[u].rs2 = (rsf * rsf) * 1.0201f;
        }
    }
    Acc32 s[IPL];
    auto fold = [&]() {
#pragma unroll
        for (int u = 0; u < IPL; u++) {
            a[u].x += s[u].x; a[u].y += s[u].y; a[u].z += s[u].z; a[u].p += s[u].p;
            s[u] = Acc32();
        }
    };
    if (MODE & EP) {
        direct_list<BLOCK, NJ, JE>(je, G.j_begin, G.nj, j0, T, x0, y0, z0, eps2, [&](int k) {
            const float4 pj = T.a[k], aj = T.b[k], lj = T.c[k];
            bool near[IPL], any = false;
#pragma unroll
            for (int u = 0; u < IPL; u++) {
                near[u] = epep_pair(I[u], pj, aj, lj, eps2, s[u]);
                any = any || near[u];
            }
            if (__ballot(any)) {
#pragma unroll
                for (int u = 0; u < IPL; u++)
                    if (near[u]) epep_neighbour(I[u], aj, a[u].ngb, a[u].rank, a[u].idmax, a[u].idmin);
            }
        }, fold);
    }
    if (MODE & (SPQ | SPM)) {
        direct_list<BLOCK, NJ, JS>(js, G.s_begin, G.ns, j0, T, x0, y0, z0, eps2, [&](int k) {
            const float4 pj = T.a[k];
            float4 qa{}, qb{};
            if (MODE & SPQ) { qa = T.b[k]; qb = T.c[k]; }
#pragma unroll
            for (int u = 0; u < IPL; u++) epsp_pair<(MODE & SPQ) != 0>(I[u], pj, qa, qb, eps2, s[u]);
        }, fold);
    }
    if constexpr (NJ == 1) {
        if (t < G.ni)
            out.write(G.i_begin + t, a[0].x, a[0].y, a[0].z, a[0].p, a[0].ngb, a[0].rank, a[0].idmax, a[0].idmin,
                      (MODE & EP) != 0);
    } else {
        DirectSums &R = *reinterpret_cast<DirectSums *>(s_mem);
#pragma unroll
        for (int u = 0; u < IPL; u++) {
#pragma unroll
            for (int d = LI; d < 64; d <<= 1) {
                a[u].x += __shfl_xor(a[u].x, d); a[u].y += __shfl_xor(a[u].y, d);
                a[u].z += __shfl_xor(a[u].z, d); a[u].p += __shfl_xor(a[u].p, d);
                if (MODE & EP) {
                    a[u].ngb += __shfl_xor(a[u].ngb, d); a[u].rank += __shfl_xor(a[u].rank, d);
                    a[u].idmax = max(a[u].idmax, __shfl_xor(a[u].idmax, d));
                    a[u].idmin = min(a[u].idmin, __shfl_xor(a[u].idmin, d));
                }
            }
            __syncthreads();
            if (lane < LI) {
                R.d[w][0][il] = a[u].x; R.d[w][1][il] = a[u].y; R.d[w][2][il] = a[u].z; R.d[w][3][il] = a[u].p;
                R.n[w][0][il] = a[u].ngb; R.n[w][1][il] = a[u].rank; R.n[w][2][il] = a[u].idmax; R.n[w][3][il] = a[u].idmin;
            }
            __syncthreads();
            // 8 sums over the waves, one lane each
            if (t < 4 * LI) {
                const int s = t / LI;
                double v = R.d[0][s][il];
                for (int q = 1; q < DIRECT_WAVES; q++) v += R.d[q][s][il];
                R.d[0][s][il] = v;
            } else if ((MODE & EP) && t >= DIRECT_BLOCK / 2 && t < DIRECT_BLOCK / 2 + 4 * LI) {
                const int s = (t - DIRECT_BLOCK / 2) / LI;
                int v = R.n[0][s][il];
                for (int q = 1; q < DIRECT_WAVES; q++) {
                    const int x = R.n[q][s][il];
                    v = s < 2 ? v + x : s == 2 ? max(v, x) : min(v, x);
                }
                R.n[0][s][il] = v;
            }
            __syncthreads();
            if (t < LI && t + u * LI < G.ni)
                out.write(G.i_begin + t + u * LI, R.d[0][0][t], R.d[0][1][t], R.d[0][2][t], R.d[0][3][t], R.n[0][0][t],
                          R.n[0][1][t], R.n[0][2][t], R.n[0][3][t], (MODE & EP) != 0);
        }
    }
}

// LI: the most i-lanes that still leave enough workgroups (or enough for a short list, below).  More
// i-lanes mean fewer workgroups that each stage the j list, fewer workgroups mean idle CUs (256 of
// them): up to 8 i-lanes about one per CU is enough, above, where staging is under a tenth of the
// work, two (both resident).  One line for all sizes: it lies 2 % above the best split at 3001 x
// 10007 and 7 % at 20000 x 20000 below.
// EP-EP, us, LI = 2 / 4 / 8 / 16 / 32 / 64 (the chosen one starred; in brackets a workgroup of
// 256 lanes per 256 i-particles with pairs summed 32 at a time in FP32):
//   117 x 731        *7.9 / 8.4 / 8.9 / 11.3 / 16.0 / 26.7      (63.0)
//   2000 x 2000      17.3 / *13.1 / 16.1 / 22.6 / 35.8 / 64.6   (315)
//   3001 x 10007     68.4 / *59.8 / 58.6 / 90.4 / 160 / 307     (1553)
//   8192 x 8192      133 / 92.0 / *73.6 / 77.5 / 133 / 252      (1264)
//   20000 x 20000    669 / 477 / 380 / *407 / 508 / 608         (3075)
//   65536 x 65536    6647 / 4686 / 3711 / 3301 / 3179 / *3251   (10050; now 1.3 T pairs/s)
constexpr int direct_min_wg(int li) { return li <= 8 ? 240 : 500; }
// A short list takes as many i-lanes as leave its quads a j-lane each: more j-lanes only make the
// sum over them longer.  us: 8 x 32 6.6 / 6.2 / 5.4 / 5.0 / 4.7 / *4.6, 64 x 64 6.8 / 6.4 / 6.0 / 5.6 /
// *5.5 / 5.8, 120 x 120 6.9 / 6.5 / 6.2 / *5.8 / 6.7 / 8.5, 64 x 256 6.9 / 6.7 / *6.4 / 6.7 / 8.4 / 11.4,
// 60 x 500 7.2 / *7.2 / 7.5 / 8.9 / 12.4 / 18.8, 2000 x 200 10.1 / 6.9 / *6.6 / 7.1 / 7.8 / 10.6.
constexpr int DIRECT_SHORT = DIRECT_WAVES * 64 * 4;

// One i-particle per lane and no j-lanes: where the i-particles fill the chip by themselves and the
// list is too short to pay for the sums over j-lanes.  us, the rule's split above -> wide: 65536 x 8 6.8 ->
// 4.3, x 32 7.2 -> 7.8; 131072 x 8 10.9 -> 4.8, x 32 11.7 -> 8.2, x 128 20.1 -> 23.1; 262144 x 8 19.6 -> 6.5, x 128
// 35.2 -> 32.9, x 512 103 -> 118; 524288 x 128 68.8 -> 58.7, x 512 200 -> 208; 1048576 x 1 71 -> 20, x 128 133 -> 101, x 512
// 395 -> 385, x 2048 1497 -> 1506.
constexpr bool direct_wide(long long ni, long long entries) { return ni >= 1500 * (entries + 16); }

// calls f(LI) with the rule's LI; entries: of a list (the average of several); count(i-particles
// per workgroup): the workgroups of the call
template <class COUNT, class F>
void direct_lanes(long long entries, COUNT count, F f) {
    auto fits = [&](auto LI) {
        if (LI.value > 2 && LI.value * entries > DIRECT_SHORT && count(DIRECT_IPL * LI.value) < direct_min_wg(LI.value))
            return false;
        f(LI);
        return true;
    };
    fits(std::integral_constant<int, 64>()) || fits(std::integral_constant<int, 32>()) ||
        fits(std::integral_constant<int, 16>()) || fits(std::integral_constant<int, 8>()) ||
        fits(std::integral_constant<int, 4>()) || fits(std::integral_constant<int, 2>());
}

// a table of i-groups of at most 2 li i-particles each
template <int MODE, class JE, class JS>
void launch_direct_groups(int li, const SoftGroup *d_groups, int ngroups, SrcEPI is, typename JE::Src je, typename JS::Src js,
                          SinkForce out, float eps2, hipStream_t st) {
    if (ngroups <= 0) return;
    auto go = [&](auto LI) {
        if (li == LI.value)
            hipLaunchKernelGGL((k_direct_f32<MODE, LI.value, JE, JS>), dim3(ngroups), dim3(DIRECT_BLOCK), 0, st, d_groups,
                               SoftGroup{}, is, je, js, out, eps2);
    };
    go(std::integral_constant<int, 64>()); go(std::integral_constant<int, 32>()); go(std::integral_constant<int, 16>());
    go(std::integral_constant<int, 8>()); go(std::integral_constant<int, 4>()); go(std::integral_constant<int, 2>());
}

// one functor call: nj EP or SP entries
template <int MODE, class J>
void launch_direct_f32(const gplum_epi *epi, int ni, typename J::Src js, int nj, gplum_force *force, float eps2,
                       hipStream_t st) {
    SoftGroup one{};
    one.ni = ni;
    one.nj = one.ns = nj;
    auto count = [&](int per_wg) { return ceil_div(ni, per_wg); };
    auto go = [&](auto LI) {
        hipLaunchKernelGGL((k_direct_f32<MODE, LI.value, J, J>), dim3(count(direct_ipl(LI.value) * LI.value)),
                           dim3(direct_block(LI.value)), 0, st, nullptr, one, SrcEPI{epi}, js, js, SinkForce{force}, eps2);
    };
    if (direct_wide(ni, nj)) go(std::integral_constant<int, DIRECT_WIDE>());
    else direct_lanes(nj, count, go);
}

}  // namespace gplum
