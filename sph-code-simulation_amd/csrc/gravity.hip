// gravity.hip -- Barnes-Hut tree walk for self-gravity.
//
// Reference: GravityForce::calculation -> BHTree::tree_force ->
// BHNode::calc_force (src/gravity_force.cpp:52-89, src/bhtree.cpp:146-150,
// 319-393).  For particle i a node is opened when edge^2 > theta^2 d^2 or
// d^2 < edge^2, with d the minimum-image vector from r_i to the node's centre
// of mass; an opened leaf contributes Hernquist & Katz (1989) softened pair
// terms for every member j != i, an unopened node its monopole.  phi is
// assigned, acc is added to (the walk runs after FluidForce).
//
// A wavefront owns 64 consecutive particles in key order (a compact region)
// and walks the pre-ordered node array once for all of them: at each node
// every lane takes the reference's opening decision for its own particle in
// FP64; lanes that accept the node add its monopole and sit out its subtree,
// and the wave descends while any lane opens.  An opened leaf's members are
// loaded once per wave into LDS, and the lanes share the opening lanes'
// particles among themselves.  Each particle therefore interacts with exactly
// the nodes and leaf members of its own reference walk, while node records are
// wave-uniform scalar loads and member records are loaded once per wave instead
// of once per lane.  The pair and monopole terms run in the pair precision T
// with compensated sums taken in blocks of at most 16 terms.  The node range is
// cut into pieces walked by different wavefronts; their sums are added in a
// fixed order in FP64.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <climits>

#include "ctx.hpp"

namespace sphgpu {

namespace {

// order LDS accesses between the lanes of one wavefront
SPH_DEV void wave_lds_fence()
{
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

// x of the lane that a DPP control pairs with this one (all lanes active)
template <int CTRL> SPH_DEV float dpp(float x)
{
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), CTRL, 0xf, 0xf, true));
}
template <int CTRL> SPH_DEV double dpp(double x)
{
    const long long b = __double_as_longlong(x);
    const int lo = __builtin_amdgcn_update_dpp(0, (int)b, CTRL, 0xf, 0xf, true);
    const int hi = __builtin_amdgcn_update_dpp(0, (int)(b >> 32), CTRL, 0xf, 0xf, true);
    return __longlong_as_double((long long)(((unsigned long long)(unsigned)hi << 32) | (unsigned)lo));
}

// Hernquist & Katz (1989) softened potential and force factors
// (src/bhtree.cpp:319-345), epsilon = h/2: f(r, h) for the potential, g(r, h)
// for the force (acceleration = -r_ij G m g).  FP64: the reference's
// expressions.
SPH_DEV double hk_f(double r, double h)
{
    const double e = h * 0.5;
    const double u = r / e;
    if (u < 1.0) return (-0.5 * u * u * (1.0 / 3.0 - 3.0 / 20 * u * u + u * u * u / 20) + 1.4) / e;
    else if (u < 2.0) return -1.0 / (15 * r) + (-u * u * (4.0 / 3.0 - u + 0.3 * u * u - u * u * u / 30) + 1.6) / e;
    else return 1 / r;
}

SPH_DEV double hk_g(double r, double h)
{
    const double e = h * 0.5;
    const double u = r / e;
    if (u < 1.0) return (4.0 / 3.0 - 1.2 * u * u + 0.5 * u * u * u) / (e * e * e);
    else if (u < 2.0)
        return (-1.0 / 15 + 8.0 / 3 * u * u * u - 3 * u * u * u * u + 1.2 * u * u * u * u * u - u * u * u * u * u * u / 6.0) /
               (r * r * r);
    else return 1 / (r * r * r);
}

// FP32: the same polynomials with the reciprocals 1/e and 1/r formed once per
// pair side and every branch evaluated (the lanes of a wave take different
// branches for the same neighbour), selected by u
SPH_DEV void hk_fg(float r, float inv_r, float inv_e, float &f, float &g)
{
    const float u = r * inv_e;
    const float u2 = u * u, u3 = u2 * u;
    const float inv_r3 = inv_r * inv_r * inv_r;
    const float inv_e3 = inv_e * inv_e * inv_e;
    const float fa = fmaf(-0.5f * u2, fmaf(u3, 1.0f / 20.0f, fmaf(u2, -3.0f / 20.0f, 1.0f / 3.0f)), 1.4f) * inv_e;
    const float fb = fmaf(fmaf(-u2, fmaf(u3, -1.0f / 30.0f, fmaf(u2, 0.3f, 4.0f / 3.0f - u)), 1.6f), inv_e,
                          -(1.0f / 15.0f) * inv_r);
    const float ga = fmaf(0.5f, u3, fmaf(-1.2f, u2, 4.0f / 3.0f)) * inv_e3;
    const float gb = fmaf(u3, fmaf(u3, -1.0f / 6.0f, fmaf(1.2f, u2, fmaf(-3.0f, u, 8.0f / 3.0f))), -1.0f / 15.0f) * inv_r3;
    f = u < 1.0f ? fa : (u < 2.0f ? fb : inv_r);
    g = u < 1.0f ? ga : (u < 2.0f ? gb : inv_r3);
}

constexpr int kGravSideMax = 64;

template <typename T> struct GravArgs {
    int n, n_nodes;
    const double *x64[3];
    RecView<T> rv;
    const GravNode *__restrict__ node;
    double theta2, G;
    Box box;
    long long *stats;
    // the walk in 2 nside pieces: with c the node index of the wavefront's
    // particles, pieces 2k and 2k + 1 take the nodes whose distance to c in
    // pre-order is in [n_nodes k^2 / nside^2, n_nodes (k + 1)^2 / nside^2), to
    // the right and to the left; piece s writes its sums to
    // part[(4 s + c) n + i], c = phi, a_x, a_y, a_z
    int nside, ngroups;
    int bound[kGravSideMax + 1];  // n_nodes k^2 / nside^2
    const int *nbase;
    double *part;
};

// one record per node, pre-order: centre of mass, edge^2 (the reference's
// e * e), mass, member range, subtree end and signed level
__global__ void k_grav_nodes(int n_nodes, int cap, const double *__restrict__ com, const double *__restrict__ edge,
                             const double *__restrict__ mass, const int *__restrict__ start,
                             const int *__restrict__ end, const int *__restrict__ skip, const int *__restrict__ level,
                             float G, GravNode *__restrict__ out)
{
    const int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= n_nodes) return;
    GravNode g;
    g.cx = com[k];
    g.cy = com[(size_t)cap + k];
    g.cz = com[2 * (size_t)cap + k];
    g.l2 = edge[k] * edge[k];
    g.mass = mass[k];
    g.gm = G * (float)mass[k];
    g.pad = 0.0f;
    g.start = start[k];
    g.end = end[k];
    g.skip = skip[k];
    g.level = level[k];
    out[k] = g;
}

template <typename T> struct GravStage;
template <> struct GravStage<float> {
    float4 own[kWave]; // the wavefront's particles: x, y, z, 1/e_i
    float4 p[kWave];   // x, y, z, 1/e_j
    float gm[kWave];   // G m_j / 2
    int lane[kWave];   // the opening lanes, packed
};
template <> struct GravStage<double> {
    double4 own[kWave];
    double4 p[kWave];  // x, y, z, h_j
    double gm[kWave];
    int lane[kWave];
};

// minimum-image component for a periodic box, the plain difference otherwise
// (P is the box's periodic flag, fixed per launch)
template <bool P, typename T> SPH_DEV T grav_rij(T xi, T xj, const Box &b, int k)
{
    return P ? rij_axis<T>(xi, xj, b, k) : xi - xj;
}

// the 64-byte record of a node (the same for all lanes) in one scalar load; no
// kernel that reads records writes them, which the address space states
SPH_DEV GravNode load_node(const GravNode *p)
{
    typedef int I16 __attribute__((ext_vector_type(16)));
    union {
        I16 v;
        GravNode g;
    } u;
    typedef const __attribute__((address_space(4))) I16 *Constant;
    u.v = *(Constant)(unsigned long long)p;
    return u.g;
}

// Wavefronts a SIMD that the walk is compiled for (512 registers shared by
// them).  The FP32 forms are bound by latency and arithmetic together and take 8
// (64 registers), which spills 6 in open 3D (1M particles 1979 us; 7 wavefronts
// without a spill 2038) and 12 in periodic 2D (262k 381 us; without a spill
// 393).  Periodic 3D, with the image and its tie test for every pair, would
// spill 37 into the pair loop: at 8 wavefronts 205k particles took 2838 us and
// 1M 10776, at 6 (80 registers, 7 reloaded per opened leaf) 1231 and 5097, at 5
// without a spill 1314 and 5397.  FP64 fits 4 without a spill (94 registers).
template <int D, typename T, bool P> constexpr int grav_waves_per_simd()
{
    return sizeof(T) == 8 ? 4 : (P && D == 3 ? 6 : 8);
}

template <int D, typename T, bool P>
__global__ __launch_bounds__(256, (grav_waves_per_simd<D, T, P>())) void k_gravity(GravArgs<T> a)
{
    __shared__ GravStage<T> stage[4];
    GravStage<T> &st = stage[(threadIdx.x >> 6) & 3];
    const int lane = threadIdx.x & (kWave - 1);
    // Workgroups are dispatched in order and round-robin over the XCDs: each XCD
    // keeps one contiguous eighth of the particles and starts the pieces around
    // the particles themselves, the heavy ones, before the far ones (heavy
    // pieces that start last leave a long tail, and at a regular stride between
    // light ones they all land on the same shader engines: two alternating
    // halves took 5.1 ms at 1M particles at the instruction count of 3.4 ms).
    const int gx = (a.ngroups + kNumXcd - 1) / kNumXcd;  // particle groups per XCD
    const int kb = blockIdx.x / kNumXcd;
    const int seg = kb / gx;
    const int group = (blockIdx.x % kNumXcd) * gx + kb % gx;
    const int i0 = group * blockDim.x + threadIdx.x;
    if ((i0 & ~(kWave - 1)) >= a.n) return;  // whole wave beyond the particles
    const bool valid = i0 < a.n;
    const int i = valid ? i0 : a.n - 1;
    typedef typename V4T<T>::type V4;
    const V4 *__restrict__ RP = a.rv.r[R_POSH];
    const V4 *__restrict__ RV = a.rv.r[R_VELM];
    double ri[3] = {0, 0, 0};
#pragma unroll
    for (int k = 0; k < D; ++k) ri[k] = a.x64[k][i];
    {
        const V4 pi_ = RP[i];
        if constexpr (sizeof(T) == 4) st.own[lane] = make_float4(pi_.x, pi_.y, pi_.z, 2.0f / pi_.w);
        else st.own[lane] = pi_;
    }
    // half-box ties of the FP32 minimum image: the FP32 positions and their
    // difference carry at most 4 u X of rounding (X the largest coordinate
    // magnitude); 2^-18 (X + L) covers it
    float tie_band[3] = {0.f, 0.f, 0.f};
    if constexpr (P) {
#pragma unroll
        for (int k = 0; k < D; ++k) {
            const double X = fmax(fabs(a.box.lo[k]), fabs(a.box.hi[k]));
            tie_band[k] = (float)((X + a.box.range[k]) * 3.814697265625e-06);
        }
    }
    const T G = T(a.G);
    // compensated sums in blocks of at most 16 terms (fold below)
    BlockAcc<T> phi, ac[3];
    auto fold = [&]() {
        phi.fold();
#pragma unroll
        for (int k = 0; k < D; ++k) ac[k].fold();
    };
    int since_fold = 0;  // node steps since the last fold (wave-uniform)
    int inter = 0;  // of the wavefront
    // the lane takes part in the walk from node `resume` on; a lane that
    // accepted a node's monopole resumes at the node's subtree end
    int resume = valid ? 0 : INT_MAX;
    // BHNode::calc_force opening test (src/bhtree.cpp:350-358): d and d^2 to
    // the node's centre of mass, and whether this lane opens the node
    auto opens = [&](const GravNode &g, double d[3], double &d2) -> bool {
        const double cm[3] = {g.cx, g.cy, g.cz};
#pragma unroll
        for (int k = 0; k < D; ++k) {
            d[k] = grav_rij<P, double>(ri[k], cm[k], a.box, k);
            d2 = (k == 0) ? d[k] * d[k] : d2 + d[k] * d[k];
        }
        return (g.l2 > a.theta2 * d2) || (d2 < g.l2);
    };
    const int mid = min((i0 & ~(kWave - 1)) + kWave / 2, a.n - 1);
    const int here = __builtin_amdgcn_readfirstlane(a.nbase[mid]);
    const int d0 = a.bound[seg >> 1], d1 = a.bound[(seg >> 1) + 1];
    int node = (seg & 1) ? max(0, here - d1) : min(a.n_nodes, here + d0);
    const int node_end = (seg & 1) ? max(0, here - d0) : min(a.n_nodes, here + d1);
    if (node > 0 && node < node_end) {
        // a later piece: a lane that accepts an ancestor of the first node has
        // that subtree in the ancestor's piece and resumes behind it
        int anc = 0;
        while (anc != node) {
            const GravNode g = a.node[anc];
            double d[3] = {0, 0, 0}, d2 = 0.0;
            if (anc >= resume && !opens(g, d, d2)) resume = g.skip;
            // the child whose subtree holds the first node
            int ch = anc + 1, sk = a.node[ch].skip;
            while (sk <= node) {
                ch = sk;
                sk = a.node[ch].skip;
            }
            anc = ch;
        }
    }
    while (node < node_end) {
        // a lane adds at most one monopole per node step
        if (++since_fold == 16) {
            fold();
            since_fold = 0;
        }
        node = __builtin_amdgcn_readfirstlane(node);
        const GravNode g = load_node(a.node + node);
        const bool act = node >= resume;
        double d[3] = {0, 0, 0};
        double d2 = 0.0;
        bool open = false;
        // (a SIMD skips the 16 lanes of a pass that are all inactive: lanes that
        // sit out the subtree are kept out of the test, too)
        if (act) {
            open = opens(g, d, d2);
            if (!open) {
                // monopole (src/bhtree.cpp:387-392)
                const T r_inv = (sizeof(T) == 4) ? trsqrt(T(d2)) : tdiv(T(1.0), tsqrt(T(d2)));
                const T gm = sizeof(T) == 4 ? T(g.gm) : G * T(g.mass);
                const T s = gm * (r_inv * r_inv * r_inv);
                if constexpr (sizeof(T) == 4) {
                    phi.p = fmaf(-gm, r_inv, phi.p);
#pragma unroll
                    for (int k = 0; k < D; ++k) ac[k].p = fmaf(-T(d[k]), s, ac[k].p);
                } else {
                    phi.add(-(gm * r_inv));
#pragma unroll
                    for (int k = 0; k < D; ++k) ac[k].add(-(T(d[k]) * s));
                }
                resume = g.skip;
            }
        }
        const unsigned long long om = __builtin_amdgcn_ballot_w64(open);
        inter += __popcll(__builtin_amdgcn_ballot_w64(act) & ~om);
        if (om == 0ull) {
            node = g.skip;
            continue;
        }
        if (g.level < 0) {
            // opened leaf: pair terms with every member j != i
            // (src/bhtree.cpp:362-378).  A quarter of the lanes open a leaf on
            // average (of a third of the leaves at most four), so each opening
            // lane's particle is given to G = 1, 2, 4, 8 or 16 lanes that take
            // every G-th of the staged members; at most 16 terms a lane, then
            // a tree over the G lanes, then one compensated addition.  1M
            // Evrard, FP32: 3000 -> 2633 us a walk; 606k FP64: 8293 -> 5431.
            // With fused multiply-adds, counts in scalar registers, the node
            // record in one scalar load, the particles in LDS (8 waves a SIMD;
            // 6 took 2640) and idle lanes out of the test: 2335 and 5107.
            const int np = __popcll(om);
            const int lg = np > 32 ? 0 : np > 16 ? 1 : np > 8 ? 2 : np > 4 ? 3 : 4;
            const int rank = __builtin_amdgcn_mbcnt_hi((unsigned)(om >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)om, 0));
            const int chunk = lg == 1 ? 32 : kWave;
            const int slot = lane >> lg;
            for (int s0 = g.start; s0 < g.end; s0 += chunk) {
                const int cnt = min(chunk, g.end - s0);
                if (lane < cnt) {
                    const V4 pj = RP[s0 + lane];
                    const T mj = RV[s0 + lane].w;
                    if constexpr (sizeof(T) == 4) st.p[lane] = make_float4(pj.x, pj.y, pj.z, 2.0f / pj.w);
                    else st.p[lane] = pj;
                    st.gm[lane] = T(0.5) * (G * mj);
                }
                if (open) st.lane[rank] = lane;
                wave_lds_fence();
                const int src = lg == 0 ? lane : (slot < np ? st.lane[slot] : lane);
                const bool work = lg == 0 ? open : slot < np;
                const int is = (i0 & ~(kWave - 1)) + src;
                const typename V4T<T>::type own = st.own[src];
                const T xs[3] = {own.x, own.y, own.z};
                const T es = own.w;
                inter += np * cnt - __popcll(__builtin_amdgcn_ballot_w64(open && i >= s0 && i < s0 + cnt));
                // blocks of 16 terms a lane: one, unless the particles keep
                // their lanes
                for (int t0 = lane & ((1 << lg) - 1); t0 < cnt || lg != 0; t0 += 16 << lg) {
                    T bs[4] = {T(0), T(0), T(0), T(0)};
                    if (work) {
                        const int t1 = min(cnt, t0 + (16 << lg));
                        for (int t = t0; t < t1; t += 1 << lg) {
                            if (s0 + t == is) continue;
                            const typename V4T<T>::type q = st.p[t];
                            const T xj[3] = {q.x, q.y, q.z};
                            T rij[3] = {0, 0, 0};
                            T r2 = T(0);
#pragma unroll
                            for (int k = 0; k < D; ++k) rij[k] = grav_rij<P, T>(xs[k], xj[k], a.box, k);
                            if constexpr (P && sizeof(T) == 4) {
                                // a component within FP32 rounding of half the
                                // box takes its image from the FP64 positions, as
                                // the reference chooses it (the image, and with
                                // it the sign, flips there)
                                bool tie = false;
#pragma unroll
                                for (int k = 0; k < D; ++k)
                                    tie = tie || fabsf(fabsf(xs[k] - xj[k]) - 0.5f * a.box.rangef[k]) <= tie_band[k];
                                if (tie)
#pragma unroll
                                    for (int k = 0; k < D; ++k)
                                        rij[k] = (T)rij_axis<double>(a.x64[k][is], a.x64[k][s0 + t], a.box, k);
                            }
#pragma unroll
                            for (int k = 0; k < D; ++k) {
                                if (k == 0) r2 = rij[k] * rij[k];
                                else if constexpr (sizeof(T) == 4) r2 = fmaf(rij[k], rij[k], r2);
                                else r2 += rij[k] * rij[k];
                            }
                            const T gm = st.gm[t];
                            T fsum, gsum;
                            if constexpr (sizeof(T) == 4) {
                                // 1/r from one reciprocal square root, r = r^2 / r
                                // (r = 0 for coincident particles: the polynomial
                                // branch u < 1 takes no 1/r)
                                const float inv_r = trsqrt(r2);
                                const float r = r2 > 0.f ? r2 * inv_r : 0.f;
                                // beyond both softening lengths (u >= 2 on both
                                // sides, the usual case in an opened leaf) the
                                // terms are 1/r and 1/r^3; the polynomials run
                                // only when some lane of the wave has a near pair
                                const bool near = r * es < 2.0f || r * q.w < 2.0f;
                                if (__builtin_amdgcn_ballot_w64(near)) {
                                    float fi, gi, fj, gj;
                                    hk_fg(r, inv_r, es, fi, gi);
                                    hk_fg(r, inv_r, q.w, fj, gj);
                                    fsum = fi + fj;
                                    gsum = gi + gj;
                                } else {
                                    fsum = 2.0f * inv_r;
                                    gsum = 2.0f * (inv_r * inv_r * inv_r);
                                }
                            } else {
                                const T r = tsqrt(r2);
                                fsum = hk_f(r, es) + hk_f(r, q.w);
                                gsum = hk_g(r, es) + hk_g(r, q.w);
                            }
                            const T s2 = gm * gsum;
                            if constexpr (sizeof(T) == 4) {
                                bs[3] = fmaf(-gm, fsum, bs[3]);
#pragma unroll
                                for (int k = 0; k < D; ++k) bs[k] = fmaf(-rij[k], s2, bs[k]);
                            } else {
                                bs[3] -= gm * fsum;
#pragma unroll
                                for (int k = 0; k < D; ++k) bs[k] -= rij[k] * s2;
                            }
                        }
                    }
                    // sum over the particle's lanes, back to its own lane
                    if (lg != 0) {
#pragma unroll
                        for (int c = 0; c < 4; ++c) bs[c] += dpp<0xB1>(bs[c]);
                        if (lg > 1) {
#pragma unroll
                            for (int c = 0; c < 4; ++c) bs[c] += dpp<0x4E>(bs[c]);
                        }
                        if (lg > 2) {
#pragma unroll
                            for (int c = 0; c < 4; ++c) bs[c] += dpp<0x141>(bs[c]);
                        }
                        if (lg > 3) {
#pragma unroll
                            for (int c = 0; c < 4; ++c) bs[c] += dpp<0x140>(bs[c]);
                        }
#pragma unroll
                        for (int c = 0; c < 4; ++c) bs[c] = __shfl(bs[c], (rank << lg) & (kWave - 1), kWave);
                    }
                    if (open) {
                        phi.add_block(bs[3]);
#pragma unroll
                        for (int k = 0; k < D; ++k) ac[k].add_block(bs[k]);
                    }
                    if (lg != 0) break;
                }
                wave_lds_fence();
            }
        }
        ++node;
    }
    if (valid) {
        double *const q = a.part + 4 * (size_t)seg * a.n + i;
        q[0] = (double)phi.get();
#pragma unroll
        for (int k = 0; k < D; ++k) q[(size_t)(k + 1) * a.n] = (double)ac[k].get();
    }
    if (lane == 0) atomicAdd(stat_ptr(a.stats, 10), (unsigned long long)inter);
}

// the pieces' sums in a fixed order (FP64, deterministic), one thread per
// particle and component
__global__ void k_gravity_sum(int n, int nseg, const double *__restrict__ part, double *__restrict__ phi, double *ax,
                              double *ay, double *az)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x, c = blockIdx.y;
    if (i >= n) return;
    const double *const q = part + (size_t)c * n + i;
    double s = 0.0;
#pragma unroll 8
    for (int g = 0; g < nseg; ++g) s += q[4 * (size_t)g * n];
    if (c == 0) phi[i] = s;
    else (c == 1 ? ax : c == 2 ? ay : az)[i] += s;
}

// Pieces of the walk on each side of a wavefront's particles.  One wavefront
// walks the tree for 64 particles, a serial chain of a thousand node steps: 800
// us for 14k particles, whose 224 wavefronts leave most of the chip idle, and
// in larger sets the last wavefronts leave a tail.  The pre-order node range is
// therefore split until about kGravWaves wavefronts are there to be scheduled
// (8 fit a SIMD, 8192 the chip).  Evrard, FP32: 14k particles 801 -> 117 us,
// 200k 1284 -> 807 (with 16384 / 32768 / 131072 wavefronts 914 / 812 / 873), 1M
// 3603 -> 2961 (3326 / 3251 / 2911); FP64: 14k 1565 -> 318, 278k 5156 -> 4270,
// 606k 9380 -> 8293 (all with one lane a particle in opened leaves).
constexpr int kGravWaves = 65536;
int grav_sides(int n)
{
    const int waves = (n + kWave - 1) / kWave;
    return std::max(1, std::min(kGravWaves / waves / 2, kGravSideMax));
}

template <typename T> void launch_gravity(sphgpu_ctx *c, int nside, double *part)
{
    GravArgs<T> a;
    a.n = c->n;
    a.n_nodes = c->tree.n_nodes;
    for (int k = 0; k < 3; ++k) a.x64[k] = c->pos[k < c->dim ? k : 0];
    a.rv = rec_view<T>(c);
    a.node = c->tree.gnode;
    a.theta2 = c->prm.theta * c->prm.theta;
    a.G = c->prm.gravity_constant;
    a.box = c->box;
    a.stats = c->dstats;
    a.nside = nside;
    for (int k = 0; k <= nside; ++k) a.bound[k] = (int)((long long)a.n_nodes * k * k / ((long long)nside * nside));
    a.ngroups = grid_for(c->n, 256);
    a.nbase = c->tree.nbase;
    a.part = part;
    const dim3 g((a.ngroups + kNumXcd - 1) / kNumXcd * kNumXcd * 2 * nside), b(256);
#define LAUNCH(D)                                                                          \
    if (c->box.periodic) hipLaunchKernelGGL((k_gravity<D, T, true>), g, b, 0, c->stream, a); \
    else hipLaunchKernelGGL((k_gravity<D, T, false>), g, b, 0, c->stream, a);
    if (c->dim == 1) { LAUNCH(1) } else if (c->dim == 2) { LAUNCH(2) } else { LAUNCH(3) }
#undef LAUNCH
}

} // namespace

int gravity(sphgpu_ctx *c)
{
    if (!c->prm.use_gravity) return 0;
    if (!c->tree.valid) return fail(c, SPHGPU_E_STATE, "gravity needs a built tree");
    if (c->mirror_dirty) {
        int rc = refresh_mirrors(c);
        if (rc) return rc;
    }
    Tree &t = c->tree;
    if (t.gnode_cap < t.n_nodes) {
        if (t.gnode) hipFree(t.gnode);
        t.gnode = nullptr;
        t.gnode_cap = 0;
        const int cap = t.n_nodes + t.n_nodes / 4 + 64;
        if (hipMalloc((void **)&t.gnode, sizeof(GravNode) * (size_t)cap) != hipSuccess)
            return fail(c, SPHGPU_E_NOMEM, "gravity node records");
        t.gnode_cap = cap;
    }
    time_begin(c, "gravity_nodes");
    hipLaunchKernelGGL(k_grav_nodes, dim3(grid_for(t.n_nodes, 256)), dim3(256), 0, c->stream, t.n_nodes, t.node_cap,
                       t.com, t.edge, t.mass, t.start, t.end, t.skip, t.level, (float)c->prm.gravity_constant, t.gnode);
    time_end(c);
    // the pieces' sums: in the exchange's staging block, which is idle here and
    // has room for kStageSides pieces a side (the sets that take that few are the
    // large ones), else in memory of their own; without that, fewer pieces
    constexpr int kStageSides = SPHGPU_NFIELDS / 8;
    int nside = grav_sides(c->n);
    double *part = c->stage;
    if (nside > kStageSides) {
        if (!t.gpart && hipMalloc((void **)&t.gpart, sizeof(double) * 8 * (size_t)nside * c->n) != hipSuccess) {
            (void)hipGetLastError();
            t.gpart = nullptr;
            nside = kStageSides;
        } else {
            part = t.gpart;
        }
    }
    const int nseg = 2 * nside;
    time_begin(c, "gravity");
    if (c->prm.pair_precision == SPHGPU_PAIR_FP64) launch_gravity<double>(c, nside, part);
    else launch_gravity<float>(c, nside, part);
    hipLaunchKernelGGL(k_gravity_sum, dim3(grid_for(c->n, 256), c->dim + 1), dim3(256), 0, c->stream, c->n, nseg,
                       (const double *)part, c->sc[S_PHI], c->acc[0], c->acc[1], c->acc[2]);
    time_end(c);
    HIPCHK(c, hipGetLastError());
    return 0;
}

} // namespace sphgpu
