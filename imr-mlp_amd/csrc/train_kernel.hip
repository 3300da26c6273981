// Training kernels for gfx950 (fp64).
//
//   structure_reduce_kernel  per-structure energy and virial from site values
//                            (the virial when per-atom virials are given)
//   loss_kernel              weighted E/F/S loss, its adjoints dL/dE, dL/dF,
//                            dL/dS and the seven metrics, one wave per
//                            structure (Trainer_MTP::AddLossGard,
//                            train/train_mtp.cpp:3839-3996)
//   grad_kernel              coefficient gradient of
//                              G = sum_i [dLdE_c E_i + sum_j W_ij . dE_i/dr_ij]
//                              W_ij = dLdF_i - dLdF_idx(j) - dLdS_c r_ij
//                            (AccumulateEFSCombinationGard,
//                            potentials/potential_mtp.cpp:6896-6923, over
//                            accumulate_site_parameter_gradient, :3348-3550)
//   rows_reduce_kernel       ordered sum of the per-wave gradient rows
//
// The gradient kernel runs one wave per atom, like the E/F/S kernel, in
// directional form instead of forming the reference's per-pair Jacobians:
//   1. lanes over neighbours: basic moments m_b = sum_j f Y and their
//      tangents along W, q_b = sum_j W_j . grad_r(f Y), summed on the matrix
//      cores (add_dual_moments);
//   2. the product rules carry (m, Q) forward: Q_o += c (Q_l m_r + m_l Q_r);
//      then dG/dxi_s = dLdE m_map(s) + Q_map(s);
//   3. reverse rules carry (A, Gb) with seeds (xi, dLdE xi):
//      A_x += c A_o m_r,  Gb_x += c (Gb_o m_r + A_o Q_r), so at a basic
//      Gb_b = dG/dm_b and A_b = dG/dq_b;
//   4. lanes over neighbours again: with U = sum A Y, V = sum nu A Y,
//      H = sum Gb Y and Wg = sum A W.grad_u(Y) over the basics of radial
//      function mu,
//        dG/dc[ti,tj,mu,k] += alpha Q_k + beta Q'_k,
//        alpha = H - (w_u/d) V + Wg/d,  beta = w_u U,  w_u = W . u,
//      from the value and gradient of two polynomials per radial function by
//      nested Horner, summed over the neighbours of each species on the
//      matrix cores into the wave's gradient accumulator.
// Each wave accumulates over its atoms in LDS and writes one gradient row;
// the rows are summed in a fixed order, so the gradient is repeatable bit
// for bit for a given launch shape.
#include "mtp_device.hpp"

namespace mtpx {

namespace {

__global__ __launch_bounds__(kWave) void structure_reduce_kernel(const int *soff, int nconf,
                                                                 const double *site_energy,
                                                                 const double *site_virial,
                                                                 double *energy, double *stress)
{
    const int c = blockIdx.x, lane = threadIdx.x;
    if (c >= nconf)
        return;
    double e = 0.0, v[9] = {0, 0, 0, 0, 0, 0, 0, 0, 0};
    for (int i = soff[c] + lane; i < soff[c + 1]; i += kWave) {
        e += site_energy[i];
        if (site_virial)
#pragma unroll
            for (int k = 0; k < 9; ++k)
                v[k] += site_virial[9 * (size_t)i + k];
    }
    e = wave_sum(e);
#pragma unroll
    for (int k = 0; k < 9; ++k)
        v[k] = wave_sum(v[k]);
    if (lane == 0) {
        energy[c] = e;
        if (stress)
#pragma unroll
            for (int k = 0; k < 9; ++k)
                stress[9 * (size_t)c + k] = v[k];
    }
}

__global__ __launch_bounds__(kWave) void loss_kernel(LossArgs a)
{
    const int c = blockIdx.x, lane = threadIdx.x;
    if (c >= a.nconf)
        return;
    const int a0 = a.soff[c], a1 = a.soff[c + 1], N = a1 - a0;
    const int *act = a.active + 3 * c;  // energy, forces, stress terms in the loss
    double lf = 0.0, sqf = 0.0;
    for (int i = a0 + lane; i < a1; i += kWave) {
        double g0 = 0.0, g1 = 0.0, g2 = 0.0;
        if (act[1]) {
            const double w = a.wF[i];
            const double d0 = a.F[3 * (size_t)i] - a.tF[3 * (size_t)i];
            const double d1 = a.F[3 * (size_t)i + 1] - a.tF[3 * (size_t)i + 1];
            const double d2 = a.F[3 * (size_t)i + 2] - a.tF[3 * (size_t)i + 2];
            const double ff = (d0 * d0 + d1 * d1) + d2 * d2;
            lf += w * ff;
            sqf += ff;
            g0 = 2.0 * w * d0;
            g1 = 2.0 * w * d1;
            g2 = 2.0 * w * d2;
        }
        a.dLdF[3 * (size_t)i] = g0;
        a.dLdF[3 * (size_t)i + 1] = g1;
        a.dLdF[3 * (size_t)i + 2] = g2;
    }
    lf = wave_sum(lf);
    sqf = wave_sum(sqf);
    if (lane != 0)
        return;
    double ls = 0.0, sqs = 0.0, le = 0.0, sqe = 0.0, dE = 0.0;
    double dS[9] = {0, 0, 0, 0, 0, 0, 0, 0, 0};
    if (N > 0 && act[2]) {
        const double w = a.wS[c];
        for (int q = 0; q < 9; ++q) {
            const double d = a.S[9 * (size_t)c + q] - a.tS[9 * (size_t)c + q];
            sqs += d * d;
            dS[q] = 2.0 * w * d;
        }
        ls = w * sqs;
    }
    if (N > 0 && act[0]) {
        const double w = a.wE[c];
        const double d = a.E[c] - a.tE[c];
        const double ff = d * d;
        le = w * ff;
        sqe = ff / N / N;
        dE = 2.0 * w * d;
    }
    a.dLdE[c] = dE;
    for (int q = 0; q < 9; ++q)
        a.dLdS[9 * (size_t)c + q] = dS[q];
    double *row = a.metric_rows + 7 * (size_t)c;
    row[0] = (lf + ls) + le;
    row[1] = le;
    row[2] = lf;
    row[3] = ls;
    row[4] = sqe;
    row[5] = sqf;
    row[6] = sqs;
}

// Ordered column sums of a [rows][cols] array (metrics, gradient rows).  A
// workgroup takes kRowCols columns; its kRowGroups row groups each sum a
// contiguous run of rows in row order (eight loads in flight), and the
// group sums are added in group order, so the result is the same bits on
// every run.
constexpr int kRowCols = 16, kRowGroups = 16;
__global__ __launch_bounds__(256) void rows_reduce_kernel(const double *rows, int nrows, int cols,
                                                          double *out, int accumulate)
{
    __shared__ double part[kRowGroups][kRowCols];
    const int c = threadIdx.x % kRowCols, g = threadIdx.x / kRowCols;
    const int k = blockIdx.x * kRowCols + c;
    const int per = (nrows + kRowGroups - 1) / kRowGroups;
    const int r1 = min(nrows, (g + 1) * per);
    double s = 0.0;
    if (k < cols) {
        int r = g * per;
        for (; r + 8 <= r1; r += 8) {
            double v[8];
#pragma unroll
            for (int q = 0; q < 8; ++q)
                v[q] = rows[(size_t)(r + q) * cols + k];
#pragma unroll
            for (int q = 0; q < 8; ++q)
                s += v[q];
        }
        for (; r < r1; ++r)
            s += rows[(size_t)r * cols + k];
    }
    part[g][c] = s;
    __syncthreads();
    if (g == 0 && k < cols) {
        double t = part[0][c];
        for (int q = 1; q < kRowGroups; ++q)
            t += part[q][c];
        out[k] = accumulate ? out[k] + t : t;
    }
}

// ---- gradient kernel ---------------------------------------------------

// Neighbours whose five operand tables (add_dual_moments) a wave holds at a
// time, and the waves per SIMD the gradient kernel is compiled for.  With 64
// the tables take 160 registers.  At level 10, whose other phases are small
// and whose work space leaves room for two workgroups on a CU, halves of 32
// fit two waves on a SIMD: a training batch of 30,000 atoms takes 418 us
// (64 neighbours and one wave: 479; 64 and two waves: 450, with spills), one
// of 100,000 1,135 (1,355; 1,260).  Level 16 spills at two waves either way
// (30,000 atoms 920 us against 815) and is slower in halves at one wave (880).
template <class P>
struct GradShape {
    static constexpr int batch = 64, waves_per_simd = 1;
};
template <>
struct GradShape<ProfLevel10> {
    static constexpr int batch = 32, waves_per_simd = 2;
};

struct GradNbr {
    double wx, wy, wz, wu;  // W_ij and W_ij . u
};

// W_ij = dLdF_i - dLdF_idx(j) - dLdS r_ij (zero for lanes without an entry)
template <class P>
__device__ __forceinline__ GradNbr pair_weight(const DevNeighbors &nb, const TrainArgs &t,
                                               const double fi[3], const double S[9],
                                               int64_t p, bool valid, const Nbr<P::M> &q)
{
    GradNbr g{0, 0, 0, 0};
    if (valid) {
        const int j = nb.idx[p];
        double w[3];
#pragma unroll
        for (int a = 0; a < 3; ++a) {
            w[a] = fi[a] - t.dLdF[3 * (size_t)j + a];
            w[a] -= S[3 * a] * q.x;
            w[a] -= S[3 * a + 1] * q.y;
            w[a] -= S[3 * a + 2] * q.z;
        }
        g.wx = w[0];
        g.wy = w[1];
        g.wz = w[2];
        g.wu = (g.wx * q.ux + g.wy * q.uy) + g.wz * q.uz;
    }
    return g;
}

// Step 1.  With h = f' w_u and t = (f / d) (W - w_u u), the tangent of a basic
// moment is
//   q_abc = sum_j [h Y_abc + t . grad_u Y_abc]
//         = H_abc + a X_(a-1)bc + b Y_a(b-1)c + c Z_ab(c-1)
// with H, X, Y, Z the sums of h, t_x, t_y, t_z times the monomials: five
// products of neighbour values and monomials (f gives the moments), formed
// on the matrix cores as in add_moments from one transpose of the monomials,
// and the factors a, b, c applied once per atom instead of once per
// neighbour.  Sums go to the pairs {m, q} with LDS adds: tab as add_moments,
// shift (m.mono_shift, from global memory) the basic moment and factor that a
// gradient sum adds to.  The neighbours come in parts of GradShape::batch: a
// part holds its columns of the five tables in registers.
template <class P, class Tab>
__device__ __forceinline__ void add_dual_moments(const DevModel &m, double *red, const Tab &tab,
                                                 unsigned base,
                                                 const Nbr<P::M> &q, const GradNbr &g, int cnt,
                                                 int lane)
{
    constexpr int G = (P::M + 3) / 4, NB = GradShape<P>::batch, S = NB / 4;
    const double tx = (g.wx - g.wu * q.ux) * q.invd, ty = (g.wy - g.wu * q.uy) * q.invd,
                 tz = (g.wz - g.wu * q.uz) * q.invd;
    // (part p: the neighbours p NB .. p NB + NB - 1)
    auto group = [&](int grp, int part) __attribute__((always_inline)) {
        const int col = part * NB + (lane >> 4);
        // neighbour values of four radial functions: f, h, t_x, t_y, t_z
        constexpr int T = 5;
        double af[T][S];
        auto take = [&](int t0, int n) {
            wave_sync();
#pragma unroll
            for (int t = t0; t < t0 + n; ++t) {
                const double *a = red + (4 * (t - t0) + (lane & 3)) * kRedStride + col;
#pragma unroll
                for (int s = 0; s < S; ++s)
                    af[t][s] = lds_read(a + 4 * s);
            }
            wave_sync();
        };
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            const int mu = 4 * grp + k < P::M ? 4 * grp + k : P::M - 1;
            lds_write(red + k * kRedStride + lane, q.f[mu]);
            lds_write(red + (4 + k) * kRedStride + lane, q.fd[mu] * g.wu);
            lds_write(red + (8 + k) * kRedStride + lane, q.f[mu] * tx);
            lds_write(red + (12 + k) * kRedStride + lane, q.f[mu] * ty);
        }
        take(0, 4);
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            const int mu = 4 * grp + k < P::M ? 4 * grp + k : P::M - 1;
            lds_write(red + k * kRedStride + lane, q.f[mu] * tz);
        }
        take(4, 1);
        // (functions of degree 0 have no gradient sums)
        bool grads = true;
        if constexpr (P::exact)
            grads = P::nm[4 * grp] > 0;
        auto chunk = [&](int entry) __attribute__((always_inline)) {
            wave_sync();
            unsigned sh[3];
#pragma unroll
            for (int t = 0; t < 3; ++t)
                sh[t] = m.mono_shift[(3 * entry + t) * kWave + lane];
            const double *b = red + (lane & (kChunk - 1)) * kRedStride + col;
            double v[S], s0[T], s1[T];
#pragma unroll
            for (int s = 0; s < S; ++s)
                v[s] = lds_read(b + 4 * s);
#pragma unroll
            for (int t = 0; t < T; ++t)
                s0[t] = s1[t] = 0.0;
#pragma unroll
            for (int k = 0; k < S; k += 4)
                if (4 * k < cnt - part * NB) {
#pragma unroll
                    for (int s = k; s < k + 4; s += 2)
#pragma unroll
                        for (int t = 0; t < T; ++t)
                            if (t < 2 || grads) {
                                s0[t] = __builtin_amdgcn_mfma_f64_4x4x4f64(af[t][s], v[s], s0[t],
                                                                           0, 0, 0);
                                s1[t] = __builtin_amdgcn_mfma_f64_4x4x4f64(
                                    af[t][s + 1], v[s + 1], s1[t], 0, 0, 0);
                            }
                }
            const unsigned w = tab[entry * kWave + lane];
            if (w != 0xffffu) {
                lds_add(base + 16 * w, s0[0] + s1[0]);
                lds_add(base + 16 * w + 8, s0[1] + s1[1]);
            }
            if (grads)
#pragma unroll
                for (int t = 0; t < 3; ++t) {
                    const unsigned w2 = sh[t] & 0xffffu;
                    if (w2 != 0xffffu)
                        lds_add(base + 16 * w2 + 8,
                                (double)(int)(sh[t] >> 16) * (s0[2 + t] + s1[2 + t]));
                }
            wave_sync();
        };
        for_monomials<P::NUMAX>(
            q.ux, q.uy, q.uz, [&](auto E, double v) __attribute__((always_inline)) {
                constexpr int e = decltype(E)::value;
                if (mono_groups<P>(m, e / kChunk) >> grp & 1) {
                    lds_write(red + (e % kChunk) * kRedStride + lane, v);
                    if constexpr (e % kChunk == kChunk - 1 || e == mono_count(P::NUMAX) - 1)
                        chunk(mono_entry<P>(m, e / kChunk, grp));
                }
            });
    };
    auto groups = [&](int part) __attribute__((always_inline)) {
#pragma unroll
        for (int grp = 0; grp < G; ++grp)
            group(grp, part);
    };
    if constexpr (NB == kWave) {
        groups(0);
    } else {
#pragma unroll 1
        for (int part = 0; part < kWave / NB && part * NB < cnt; ++part)
            groups(part);
    }
}

// Step 4: the force polynomials' scheme (poly_grad) over the staged pairs
// {A, G}: value and gradient of the A polynomial and value of the G one.
struct PolyPair {
    PolyGrad a;
    double g;
};
template <int kCount>
struct PairStream {
    unsigned at;
    v2d buf[2][4];
    __device__ __forceinline__ void load(int block)
    {
#pragma unroll
        for (int k = 0; k < 4; ++k)
            if (4 * block + k < kCount)
                buf[block & 1][k] = ((lds_v2d)(uintptr_t)at)[4 * block + k];
    }
    __device__ __forceinline__ PairStream(const double2 *AG, double &tie)
        : at(lds_address(reinterpret_cast<const double *>(AG)))
    {
        asm volatile("" : "+v"(at), "+v"(tie));
        load(0);
    }
    __device__ __forceinline__ v2d next(int e, double &v, double &w)
    {
        if (e % 4 == 0 && e + 4 < kCount) {
            asm volatile("" : "+v"(at), "+v"(v), "+v"(w));
            load(e / 4 + 1);
        }
        return buf[(e / 4) & 1][e % 4];
    }
};
template <int N>
__device__ __forceinline__ PolyPair poly_pair(const double2 *AG, double x, double y, double z,
                                              double &tie)
{
    PairStream<mono_count(N)> c(AG, tie);
    PolyGrad g{0, 0, 0, 0};
    double h = 0;
    int e = 0;
#pragma unroll
    for (int a = N; a >= 0; --a) {
        double q = 0, qy = 0, qz = 0, qh = 0;
#pragma unroll
        for (int b = N - a; b >= 0; --b) {
            const v2d first = a < N && b == N - a ? c.next(e, g.p, h) : c.next(e, q, qh);
            double r = first.x, rz = 0, rh = first.y;
            ++e;
#pragma unroll
            for (int k = N - a - b - 1; k >= 0; --k) {
                const v2d v = c.next(e, r, rh);
                ++e;
                rz = k == N - a - b - 1 ? r : fma(rz, z, r);
                r = fma(r, z, v.x);
                rh = fma(rh, z, v.y);
            }
            if (b == N - a) {
                q = r;
                qz = rz;
                qh = rh;
            } else {
                qy = b == N - a - 1 ? q : fma(qy, y, q);
                qz = fma(qz, y, rz);
                q = fma(q, y, r);
                qh = fma(qh, y, rh);
            }
            asm volatile("" : "+v"(q), "+v"(qy), "+v"(qz), "+v"(qh));
        }
        if (a == N) {
            g = PolyGrad{q, 0, qy, qz};
            h = qh;
        } else {
            g.x = a == N - 1 ? g.p : fma(g.x, x, g.p);
            g.y = fma(g.y, x, qy);
            g.z = fma(g.z, x, qz);
            g.p = fma(g.p, x, q);
            h = fma(h, x, qh);
        }
        asm volatile("" : "+v"(g.p), "+v"(g.x), "+v"(g.y), "+v"(g.z), "+v"(h));
    }
    return PolyPair{g, h};
}
template <int N, int NMAX>
__device__ __forceinline__ PolyPair poly_pair_of(int nu, const double2 *AG, double x, double y,
                                                 double z, double &tie)
{
    if constexpr (N < NMAX)
        if (nu > N)
            return poly_pair_of<N + 1, NMAX>(nu, AG, x, y, z, tie);
    return poly_pair<N>(AG, x, y, z, tie);
}

// alpha_mu and beta_mu of one neighbour into rows mu and kMaxMu + mu of the
// transpose buffer:
//   alpha = p_G + (1 / d) (W - w_u u) . grad p_A,  beta = w_u p_A
struct RadialRows {
    double *red;
    int lane;
    double tx, ty, tz, wu, win, tie;
    __device__ __forceinline__ void put(int mu, const PolyPair &p)
    {
        const double al = fma(tx, p.a.x, fma(ty, p.a.y, fma(tz, p.a.z, p.g)));
        lds_write(red + mu * kRedStride + lane, al * win);
        lds_write(red + (kMaxMu + mu) * kRedStride + lane, wu * p.a.p * win);
    }
};
template <class P, int MU = 0, int OFF = 0>
__device__ __forceinline__ void radial_rows_exact(const double2 *AG, const Nbr<P::M> &q,
                                                  RadialRows &r)
{
    r.put(MU, poly_pair<P::nm[MU]>(AG + OFF, q.ux, q.uy, q.uz, r.tie));
    if constexpr (MU + 1 < P::M)
        radial_rows_exact<P, MU + 1, OFF + force_size(P::nm[MU])>(AG, q, r);
}

// Step 4 of one batch: the radial gradient
//   grad[tj][mu][k] += sum_j [t_j = tj] (alpha_mu Q_k + beta_mu Q'_k),
// per mu the product of four species' masked alphas (betas) with the basis
// functions on the matrix cores (rows species, columns k).
template <class P>
__device__ __forceinline__ void add_radial_gradient(const DevModel &m, double *red, int *ctype,
                                                    const double2 *AG, double *grad, int MR,
                                                    int ti, int tj, double win,
                                                    const Nbr<P::M> &q, const GradNbr &g, int cnt,
                                                    int lane)
{
    constexpr int S = kWave / 4;
    const int R = P::exact ? P::RMAX : m.R;
    double bq[2][S];
    {
        double Q[2][P::RMAX];
        radial_basis<P>(m, ti, tj, q.d, Q[0], Q[1]);
        ctype[lane] = tj;
        // (columns past the basis size hold what the buffer held: their sums
        // are not used)
        const double *b = red + (lane & (kChunk - 1)) * kRedStride + (lane >> 4);
#pragma unroll
        for (int t = 0; t < 2; ++t) {
#pragma unroll
            for (int k = 0; k < P::RMAX; ++k)
                lds_write(red + k * kRedStride + lane, Q[t][k]);
            wave_sync();
#pragma unroll
            for (int s = 0; s < S; ++s)
                bq[t][s] = lds_read(b + 4 * s);
            wave_sync();
        }
    }
    int ty[S];
#pragma unroll
    for (int s = 0; s < S; ++s)
        ty[s] = ctype[4 * s + (lane >> 4)];
    RadialRows r{red, lane, (g.wx - g.wu * q.ux) * q.invd, (g.wy - g.wu * q.uy) * q.invd,
                 (g.wz - g.wu * q.uz) * q.invd, g.wu, win, 0.0};
    if constexpr (P::exact) {
        radial_rows_exact<P>(AG, q, r);
    } else {
#pragma unroll 1
        for (int mu = 0; mu < m.M; ++mu) {
            const int nu = m.numax[mu];
            if (nu < 0) {
                r.put(mu, PolyPair{{0, 0, 0, 0}, 0});
                continue;
            }
            r.put(mu, poly_pair_of<0, P::NUMAX>(nu, AG, q.ux, q.uy, q.uz, r.tie));
            AG += force_size(nu);
        }
    }
    wave_sync();
#pragma unroll 1
    for (int mu = 0; mu < (P::exact ? P::M : m.M); ++mu) {
        const double *a = red + mu * kRedStride + (lane >> 4);
        double va[2][S];
#pragma unroll
        for (int s = 0; s < S; ++s) {
            va[0][s] = lds_read(a + 4 * s);
            va[1][s] = lds_read(a + kMaxMu * kRedStride + 4 * s);
        }
        for (int z0 = 0; z0 < m.Z; z0 += 4) {
            const int sp = z0 + (lane & 3);
            double s0 = 0.0, s1 = 0.0;
#pragma unroll
            for (int k = 0; k < S; k += 4)
                if (4 * k < cnt) {
#pragma unroll
                    for (int s = k; s < k + 4; ++s) {
                        s0 = __builtin_amdgcn_mfma_f64_4x4x4f64(ty[s] == sp ? va[0][s] : 0.0,
                                                                bq[0][s], s0, 0, 0, 0);
                        s1 = __builtin_amdgcn_mfma_f64_4x4x4f64(ty[s] == sp ? va[1][s] : 0.0,
                                                                bq[1][s], s1, 0, 0, 0);
                    }
                }
            const int so = z0 + (lane >> 4), k = lane & (kChunk - 1);
            if (so < m.Z && k < R)
                grad[(ti * m.Z + so) * MR + mu * R + k] += s0 + s1;
        }
    }
    wave_sync();
}

template <class P, bool kTabLds, int kMaxWaves>
__global__ __launch_bounds__(kWave *kMaxWaves, GradShape<P>::waves_per_simd) void grad_kernel(
    DevModel m, DevNeighbors nb, TrainArgs t)
{
    extern __shared__ double lds[];
    const int tid = threadIdx.x, lane = tid & (kWave - 1), wave = tid / kWave;
    const int nwaves = blockDim.x / kWave;
    const Shared L = shared_layout(m, lds, false);  // seeds are read from global memory
    double *ws = lds + shared_doubles(m, kTabLds, false) + (size_t)wave * m.tr_priv;
    // {value, dual} pairs: {m, Q} for the moments, {A, G} for the adjoints
    double2 *wp = reinterpret_cast<double2 *>(ws);
    double *red = ws + m.tr_red;
    double2 *AG = reinterpret_cast<double2 *>(ws + m.tr_stage);
    double *grad = ws + m.tr_grad;  // radial part of the gradient
    const int rowid = blockIdx.x * nwaves + wave;
    // species and moment part: accumulated in the wave's own gradient row
    double *grow = t.grad_rows + (size_t)rowid * m.ncoef;
    int *ctype = reinterpret_cast<int *>(ws + m.tr_ctype);

    stage_shared(m, L, kTabLds, tid, blockDim.x);
    for (int k = lane; k < m.nradial; k += kWave)
        grad[k] = 0.0;
    for (int k = m.nradial + lane; k < m.ncoef; k += kWave)
        grow[k] = 0.0;
    __syncthreads();
    using Steps = std::conditional_t<kTabLds, LdsSteps, GlobalSteps>;
    const Steps fwd_tab(kTabLds ? L.fwd_steps : m.fwd_steps, lane);
    const Steps bwd_tab(kTabLds ? L.bwd_steps : m.bwd_steps, lane);
    const MonoTab<kTabLds> mono(m, L.mono);
    const int MR = P::exact ? P::M * P::RMAX : m.M * m.R;

    for (int i = rowid; i < nb.n; i += gridDim.x * nwaves) {
        const int ti = nb.center_type[i];
        const int beg = nb.offsets[i];
        const int n = nb.offsets[i + 1] - beg;
        const int c = t.center_structure[i];
        const double se = t.dLdE[c];
        double S[9], fi[3];
#pragma unroll
        for (int k = 0; k < 9; ++k)
            S[k] = t.dLdS[9 * (size_t)c + k];
#pragma unroll
        for (int a = 0; a < 3; ++a)
            fi[a] = t.dLdF[3 * (size_t)i + a];
        for (int k = lane; k < m.K; k += kWave)
            wp[k] = double2{0.0, 0.0};
        wave_sync();

        // ---- 1. basic moments and their tangents ----------------------------
        for (int base = 0; base < n; base += kWave) {
            Nbr<P::M> q;
            const bool valid = lane < n - base;
            const int64_t p = beg + base + lane;
            load_neighbor<P>(m, nb, L.coef, ti, p, valid, q);
            const GradNbr g = pair_weight<P>(nb, t, fi, S, p, valid, q);
            add_dual_moments<P>(m, red, mono, lds_address(ws), q, g, n - base, lane);
        }
        wave_sync();
        if (lane == 0)
            for (int k = 0; k < m.ndup; ++k)
                wp[m.dup[2 * k]] = wp[m.dup[2 * k + 1]];
        // the zero slot may lie under the transpose buffer
        if (lane == 0)
            wp[m.dummy] = double2{0.0, 0.0};
        wave_sync();

        // ---- 2. rules forward with tangents; moment and species gradient ----
        run_rules<true>(fwd_tab, m.fwd_level_step, m.nfwd, ws);
        for (int s = lane; s < m.S; s += kWave) {
            const double2 x = wp[L.map[s]];
            grow[m.nradial + m.Z + s] += se * x.x + x.y;
        }
        if (lane == 0)
            grow[m.nradial + ti] += se;

        // ---- 3. reverse rules: A with seeds xi, G with seeds dLdE xi --------
        for (int k = lane; k < m.K; k += kWave) {
            const double sd = m.seed[k];
            wp[m.K4 + k] = double2{sd, se * sd};
        }
        wave_sync();
        run_rules<true>(bwd_tab, m.bwd_level_step, m.nbwd, ws);
        if (lane == 0)
            for (int k = 0; k < m.ndup; ++k) {
                const double2 v = wp[m.K4 + m.dup[2 * k]];
                double2 &t = wp[m.K4 + m.dup[2 * k + 1]];
                t = double2{t.x + v.x, t.y + v.y};
            }
        wave_sync();
        // {A, G} in the polynomials' order (the stage may lie over the moment
        // pairs, which are no longer read; the adjoint pairs are not under it)
        for (int s = lane; s < m.nforce; s += kWave) {
            const int b = L.force_basic[s];
            AG[s] = b >= 0 ? wp[m.K4 + b] : double2{0.0, 0.0};
        }
        wave_sync();

        // ---- 4. radial coefficient gradient ---------------------------------
        for (int base = 0; base < n; base += kWave) {
            Nbr<P::M> q;
            int tj;
            const bool valid = lane < n - base;
            const int64_t p = beg + base + lane;
            const double win = load_geometry<P::M, !P::exact>(m, nb, p, valid, q, tj, ti);
            const GradNbr g = pair_weight<P>(nb, t, fi, S, p, valid, q);
            add_radial_gradient<P>(m, red, ctype, AG, grad, MR, ti, tj, win, q, g, n - base, lane);
        }
        wave_sync();
    }
    // the radial part of this wave's gradient row
    for (int k = lane; k < m.nradial; k += kWave)
        grow[k] = grad[k];
}

template <class P>
struct GradWaves {
    static constexpr int value = 4;
};

template <class P>
void launch_grad_variant(const DevModel &m, const DevNeighbors &nb, const TrainArgs &t,
                         const EfsLaunch &cfg, hipStream_t s)
{
    constexpr int W = GradWaves<P>::value;
    if (cfg.lds_tables)
        hipLaunchKernelGGL((grad_kernel<P, true, W>), dim3(cfg.grid), dim3(kWave * cfg.waves),
                           cfg.lds_bytes, s, m, nb, t);
    else
        hipLaunchKernelGGL((grad_kernel<P, false, W>), dim3(cfg.grid), dim3(kWave * cfg.waves),
                           cfg.lds_bytes, s, m, nb, t);
}

}  // namespace

bool grad_configure(const DevModel &m, int n, int num_cus, size_t lds_limit, EfsLaunch &cfg)
{
    return configure_launch(m, n, num_cus, 4, lds_limit, m.tr_priv, cfg, -1, false);
}

hipError_t launch_structure_reduce(const int *soff, int nconf, const double *site_energy,
                                   const double *site_virial, double *energy, double *stress,
                                   hipStream_t s)
{
    if (nconf > 0)
        hipLaunchKernelGGL(structure_reduce_kernel, dim3(nconf), dim3(kWave), 0, s, soff, nconf,
                           site_energy, site_virial, energy, stress);
    return hipGetLastError();
}

hipError_t launch_loss(const LossArgs &a, hipStream_t s)
{
    if (a.nconf > 0)
        hipLaunchKernelGGL(loss_kernel, dim3(a.nconf), dim3(kWave), 0, s, a);
    return hipGetLastError();
}

hipError_t launch_rows_reduce(const double *rows, int nrows, int cols, double *out, bool accumulate,
                              hipStream_t s)
{
    if (cols > 0)
        hipLaunchKernelGGL(rows_reduce_kernel, dim3((cols + kRowCols - 1) / kRowCols), dim3(256),
                           0, s, rows, nrows, cols, out, accumulate ? 1 : 0);
    return hipGetLastError();
}

hipError_t launch_grad(const DevModel &m, const DevNeighbors &nb, const TrainArgs &t,
                       const EfsLaunch &cfg, hipStream_t s)
{
    switch (efs_variant(m, m.R)) {
    case 0: launch_grad_variant<ProfLevel16>(m, nb, t, cfg, s); break;
    case 1: launch_grad_variant<ProfLevel20>(m, nb, t, cfg, s); break;
    case 2: launch_grad_variant<ProfLevel10>(m, nb, t, cfg, s); break;
    case 3: launch_grad_variant<ProfSmall>(m, nb, t, cfg, s); break;
    default: launch_grad_variant<ProfGeneric>(m, nb, t, cfg, s); break;
    }
    return hipGetLastError();
}

}  // namespace mtpx
