// flux.hh -- face fluxes of the GRMHD right-hand side (reference:
// evolve.cpp:813-1068, grmhd.hh:551-970).
//
// Included by grmhd.hip after the block geometry (DevGrid, Opts, wg_pos,
// face_metric).  k_flux (UCT) and k_flux_gs (Gardiner-Stone EMFs) solve the
// faces of all three directions in one launch, one thread per face.
#pragma once

// The reconstructed variables of a face (the normal B is the face value).
enum { FQ_RHO = 0, FQ_ZX, FQ_ZY, FQ_ZZ, FQ_YE, FQ_TH, FQ_ENT, FQ_B0, FQ_B1, FQ_N };

// aux variable of reconstructed variable v of direction D
template <int D>
GHD int fq_aux(int v, int thermo) {
    constexpr int J0 = D == 0 ? 1 : 0, J1 = D == 2 ? 1 : 2;
    switch (v) {
        case FQ_RHO: return RHO_;
        case FQ_ZX: return ZVECX_;
        case FQ_ZY: return ZVECY_;
        case FQ_ZZ: return ZVECZ_;
        case FQ_YE: return YE_;
        case FQ_TH: return thermo ? PRESS_ : TEMP_;
        case FQ_ENT: return ENTROPY_;
        case FQ_B0: return BX_ + J0;
        default: return BX_ + J1;
    }
}

// Fluxes of one face of direction D from the states below (L) and above (R)
// it for UCT (compute_mhd_fluxes, grmhd.hh:774-970).  V: the HLL-averaged
// transverse transport velocities and the wave speeds.  A ring face returns
// after V.
template <typename EOS, bool FLAT, int D>
GHD void face_solve(const EOS& eos, const Opts& o, const Met& mf, const double L[FQ_N], const double R[FQ_N], double Bn,
                    bool ring, double V[4], double F[7]) {
    constexpr int J0 = D == 0 ? 1 : 0, J1 = D == 2 ? 1 : 2;
    double zl[3] = {L[FQ_ZX], L[FQ_ZY], L[FQ_ZZ]}, zr[3] = {R[FQ_ZX], R[FQ_ZY], R[FQ_ZZ]};
    double Bl[3], Br[3];
    Bl[D] = Bn; Bl[J0] = L[FQ_B0]; Bl[J1] = L[FQ_B1];
    Br[D] = Bn; Br[J0] = R[FQ_B0]; Br[J1] = R[FQ_B1];
    const double rhol = L[FQ_RHO], rhor = R[FQ_RHO];
    double pl, pr, el, er, a2l, a2r;   // a2 = rho h c_s^2
    if (o.thermo) {
        pl = eos.face_from_press(el, a2l, L[FQ_TH], rhol);
        pr = eos.face_from_press(er, a2r, R[FQ_TH], rhor);
    } else {
        pl = eos.face_from_temp(el, a2l, L[FQ_TH], rhol);
        pr = eos.face_from_temp(er, a2r, R[FQ_TH], rhor);
    }
    double ialp = 1.0, gdd = 1.0;
    if constexpr (!FLAT) {
        ialp = 1.0 / mf.alp;
        gdd = D == 0 ? mf.gi[0] : (D == 1 ? mf.gi[3] : mf.gi[5]);
    }
    double wl, wr, bl[4], br[4], b2l, b2r, vtl[3], vtr[3], cml, cpl, cmr, cpr, cmin, cmax;
    // W, b^mu and b^2 (smallb), the transport velocity, and the wave speeds:
    // with K = W^2 rho h (1 - c_s^2) and N = rho h c_s^2 + b^2 the roots of
    // the quadratic of the reference's get_cm_cp are
    //   [v K - beta N -+ alpha sqrt(N (K (g^dd - (z^d/W)^2) + N g^dd))] / (K + N),
    // one root and one reciprocal, and no difference of nearly equal terms
    // under the root.
    auto kin = [&](const double* z, const double* B, double rho, double p, double eps, double a2, double& W, double* b,
                   double& b2, double* vt, double& cm, double& cp) {
        double zlow[3], Blow[3], iW;
        lower3<FLAT>(mf.g, z[0], z[1], z[2], zlow);
        nr_sqrt(z[0] * zlow[0] + z[1] * zlow[1] + z[2] * zlow[2] + 1, W, iW);
        const double Bz = B[0] * zlow[0] + B[1] * zlow[1] + B[2] * zlow[2];
        lower3<FLAT>(mf.g, B[0], B[1], B[2], Blow);
        if constexpr (FLAT) {
            b[0] = Bz;
            for (int i = 0; i < 3; ++i) { b[1 + i] = iW * (B[i] + Bz * z[i]); vt[i] = iW * z[i]; }
        } else {
            b[0] = Bz * ialp;
            const double Wa = W * ialp;
            for (int i = 0; i < 3; ++i) {
                b[1 + i] = iW * (B[i] + Bz * (z[i] - Wa * mf.beta[i]));
                vt[i] = mf.alp * iW * z[i] - mf.beta[i];
            }
        }
        b2 = (B[0] * Blow[0] + B[1] * Blow[1] + B[2] * Blow[2] + Bz * Bz) * (iW * iW);
        const double K = W * W * (rho + eps * rho + p - a2), N = a2 + b2, vh = z[D] * iW;
        const double x = fmax(0., N * (K * (gdd - vh * vh) + N * gdd));
        double d, id, m = vt[D] * K;
        nr_sqrt(fmax(x, 1e-290), d, id);   // (x = 0: a cold, unmagnetised state)
        if constexpr (!FLAT) { m -= mf.beta[D] * N; d *= mf.alp; }
        const double i = nr_rcp(K + N), l1 = (m - d) * i, l2 = (m + d) * i;
        cm = fmin(l1, l2); cp = fmax(l1, l2);
    };
    kin(zl, Bl, rhol, pl, el, a2l, wl, bl, b2l, vtl, cml, cpl);
    kin(zr, Br, rhor, pr, er, a2r, wr, br, b2r, vtr, cmr, cpr);
    if (o.riemann == 1) {
        cmax = fmax(fmax(fabs(cml), fabs(cmr)), fmax(fabs(cpl), fabs(cpr)));
        if (fmin(rhol, rhor) < o.c_limit) cmax = fmax(cmax, mf.alp * sqrt(gdd) + fabs(mf.beta[D]));
        cmin = cmax;
    } else {
        cmin = -fmin(0., fmin(cml, cmr));
        cmax = fmax(0., fmax(cpl, cpr));
    }
    if (cmin < 1e-12 && cmax < 1e-12) { cmin = 1; cmax = 1; }
    const double ihll = nr_rcp(cmax + cmin);   // shared by the HLL fluxes of this face
    const double sg = mf.sqrtg;
    V[0] = hll_r(vtl[J0], vtr[J0], 0, 0, cmin, cmax, ihll);
    V[1] = hll_r(vtl[J1], vtr[J1], 0, 0, cmin, cmax, ihll);
    V[2] = cmin; V[3] = cmax;
    if (ring) return;
    // conserved and fluxes along D (grmhd_subexpressions.hh:97-156)
    double bsh[3];
    lower3(mf.g, mf.beta[0], mf.beta[1], mf.beta[2], bsh);
    const double ia2 = ialp * ialp;
    auto side = [&](double rho, double p, double eps, const double* z, const double* b, double b2, double w,
                    const double* vt, double ye, double ent, double U[7], double Fx[7]) {
        double S[3];
        conserved<FLAT>(mf, rho, p, eps, z, ent, w, b2, b, U[DENS_], U[TAU_], S, U[ENTROPYSTAR_]);
        U[SX_] = S[0]; U[SY_] = S[1]; U[SZ_] = S[2];
        U[YESTAR_] = ye * U[DENS_];
        const double rhoh = b2 + eps * rho + p + rho, ps = 0.5 * b2 + p;
        const double W2rh = w * w * rhoh, fD = vt[D] * U[DENS_];
        double blo[3], vlo[3];
        lower3<FLAT>(mf.g, b[1], b[2], b[3], blo);
        lower3<FLAT>(mf.g, vt[0], vt[1], vt[2], vlo);
        Fx[DENS_] = fD;
        if constexpr (FLAT) {
            Fx[TAU_] = W2rh * vt[D] - b[0] * b[1 + D] - fD;
            const double c = vt[D] * W2rh;
            for (int a = 0; a < 3; ++a)
                Fx[SX_ + a] = a == D ? -b[1 + D] * blo[a] + ps + c * vlo[a] : -b[1 + D] * blo[a] + c * vlo[a];
        } else {
            Fx[TAU_] = W2rh * vt[D] + ps * mf.beta[D] - mf.alp * mf.alp * b[0] * b[1 + D] - fD;
            const double c = vt[D] * W2rh * ia2;
            for (int a = 0; a < 3; ++a)
                Fx[SX_ + a] = mf.alp * (-b[1 + D] * (blo[a] + b[0] * bsh[a]) + (a == D ? ps : 0.0) + c * (vlo[a] + bsh[a]));
        }
        Fx[ENTROPYSTAR_] = vt[D] * U[ENTROPYSTAR_];
        Fx[YESTAR_] = ye * fD;
    };
    double Ul[7], Ur[7], Fl[7], Fr[7];
    side(rhol, pl, el, zl, bl, b2l, wl, vtl, L[FQ_YE], L[FQ_ENT], Ul, Fl);
    side(rhor, pr, er, zr, br, b2r, wr, vtr, R[FQ_YE], R[FQ_ENT], Ur, Fr);
#pragma unroll
    for (int v = 0; v < 7; ++v) F[v] = sg * hll_r(Fl[v], Fr[v], Ul[v], Ur[v], cmin, cmax, ihll);
}

// Arguments of the flux kernels.
struct FluxArgs {
    const double* aux;
    const double* mstate; int mnv;     // metric source
    const double* B[3];                // face B
    double* flux[3]; double* vbar[3];
    const double* fmc[3];              // face-metric caches or null
    // ring_own (per block, bit 2 d + side for the six block faces): when
    // given, a ring face is computed only if its ghost side lies beyond an
    // outflow face of the instance; the others are interior faces of the
    // neighbouring block, from which the edge EMFs then take them.
    // With nbr (the neighbour across each of the six block faces, in the
    // second and third RK stages, whose gathers leave the face slabs alone) a
    // full face takes a cell beyond a block face from the neighbouring
    // block's interior (normal index shifted by one block extent); beyond an
    // outflow face (no neighbour) and on ring faces, from its own ghosts,
    // which run their own c2p or copy one that does.
    const uint8_t* ring_own;
    const int32_t* nbr;
    int dir0, ndir;                    // directions of this launch: dir0 .. dir0 + ndir - 1
    int tiles, tilesr;                 // workgroups per block and direction: full faces, ring faces
};

// A double through a 32-bit byte offset from a wave-uniform base: the
// addressing form with a scalar base and one vector register, no 64-bit
// vector adds.  (One variable of one block spans less than 2^32 bytes: its
// arrays would not fit the card otherwise.)
__device__ __forceinline__ double ld_off(const double* base, uint32_t off) {
    return *reinterpret_cast<const double*>(reinterpret_cast<const char*>(base) + off);
}
// Streaming store: what the flux kernels write is read next by other kernels,
// after more than the caches hold.
__device__ __forceinline__ void st_off(double* base, uint32_t off, double v) {
    __builtin_nontemporal_store(v, reinterpret_cast<double*>(reinterpret_cast<char*>(base) + off));
}

// Between two variables: the values of the last one are formed here and not
// where they are used (sunk into the branch of the face, everything they come
// from would stay alive instead), and the next one is not interleaved with
// it (nine variables at a time need more registers than there are).
__device__ __forceinline__ void settle(double& lo, double& hi) {
    asm volatile("" : "+v"(lo), "+v"(hi));
    __builtin_amdgcn_sched_barrier(0);
}

// The transverse indices (ghosts included) of line p of direction D: the
// n0 n1 lines with both interior, or (ring) the lines with exactly one in
// the ghost layers (they feed only the transverse reconstructions of the
// edge EMFs; lines with both in the ghost layers are never read).  False where
// there is none or another block writes it.
GHD bool line_pos(const DevGrid& G, int T0, int T1, bool ring, int p, uint8_t own, bool use_own, int& b, int& c) {
    const int ng = G.ng, n0 = G.n[T0], n1 = G.n[T1];
    if (!ring) {
        udivmod(p, n0, c, b);
        b += ng; c += ng;
        return c < n1 + ng;
    }
    const int g2 = 2 * ng, nA = g2 * n1;
    int gl, side;
    if (p < nA) {                      // t0 ghost, t1 interior
        udivmod(p, g2, c, gl);
        c += ng;
        b = gl < ng ? gl : n0 + gl;
        side = 2 * T0 + (gl >= ng);
    } else {                           // t0 interior, t1 ghost
        udivmod(p - nA, n0, gl, b);
        if (gl >= g2) return false;
        b += ng;
        c = gl < ng ? gl : n1 + gl;
        side = 2 * T1 + (gl >= ng);
    }
    return !use_own || ((own >> side) & 1);
}

// Metric of face (i, j, k): the cache (only the inverse component this
// direction uses: cmcp, the LLF speed limit) or the interpolation.
template <bool FLAT, int D>
__device__ __forceinline__ void face_met(const DevGrid& G, const FluxArgs& f, double alp_ex, int64_t q, int i, int j,
                                         int k, int64_t st, Met& mf, bool& excise) {
    excise = false;
    if constexpr (FLAT) {
        mf.flat();
    } else if (f.fmc[D]) {
        const int64_t nfd = G.nface[D];
        const double* FM = f.fmc[D] + q * FMC * nfd + fidx<D>(G, i, j, k);
        for (int a = 0; a < 6; ++a) { mf.g[a] = FM[a * nfd]; mf.gi[a] = 0.0; }
        mf.gi[D == 0 ? 0 : (D == 1 ? 3 : 5)] = FM[6 * nfd];
        for (int a = 0; a < 3; ++a) mf.beta[a] = FM[(7 + a) * nfd];
        mf.alp = FM[10 * nfd];
        mf.sqrtg = FM[11 * nfd];
        excise = FM[12 * nfd] != 0.0;
    } else {
        const int64_t nc = G.ncell;
        face_metric(f.mstate + q * (int64_t)f.mnv * nc, nc, cidx(G, i, j, k), st, alp_ex, mf, excise);
    }
}

// One face of direction D: thread e of block q over its full faces, or its
// ring faces.
template <typename EOS, int REC, bool FLAT, int D>
__device__ __forceinline__ void flux_face(const DevGrid& G, const EOS& eos, const Opts& o, const FluxArgs& f, int64_t q,
                                          int e, bool ring) {
    constexpr int T0 = D == 0 ? 1 : 0, T1 = D == 2 ? 1 : 2;
    const int Rn = G.n[D] + 1, ng = G.ng, nD = G.n[D];
    int a, b, c, r;
    if (D == 1 && !ring) {
        // x, then the normal, then z
        udivmod(e, G.n[T0], r, b); udivmod(r, Rn, c, a);
        if (c >= G.n[T1]) return;
        b += ng; c += ng;
    } else {
        const int per = ring ? 2 * ng * (G.n[T0] + G.n[T1]) : G.n[T0] * G.n[T1];
        int p;
        if (D == 0) udivmod(e, Rn, p, a); else udivmod(e, per, a, p);
        if (a >= Rn || !line_pos(G, T0, T1, ring, p, (ring && f.ring_own) ? f.ring_own[q] : 0, f.ring_own != nullptr, b, c)) return;
    }
    const int m0 = ng + a;
    const int i = D == 0 ? m0 : b, j = D == 1 ? m0 : (D == 0 ? b : c), k = D == 2 ? m0 : c;
    const int64_t nc = G.ncell, nf = G.nface[D];
    const int64_t st = D == 0 ? 1 : (D == 1 ? G.N[0] : (int64_t)G.N[0] * G.N[1]);
    const double Bf = ld_off(f.B[D] + q * nf, (uint32_t)fidx<D>(G, i, j, k) * 8u);
    // (scalar registers; -1: none)
    int32_t nl = -1, nh = -1;
    if (!ring && f.nbr) {
        nl = __builtin_amdgcn_readfirstlane(f.nbr[q * 6 + 2 * D]);
        nh = __builtin_amdgcn_readfirstlane(f.nbr[q * 6 + 2 * D + 1]);
    }
    const int64_t c0 = cidx(G, i, j, k);
    const double* P[6];
    {
        // points 0 to 2 can only lie before the block, the others only beyond
        const double* own = f.aux + q * NAUX * nc + c0;
        const int64_t dl = nl < 0 ? 0 : (nl - q) * NAUX * nc + nD * st, dh = nh < 0 ? 0 : (nh - q) * NAUX * nc - nD * st;
#pragma unroll
        for (int t = 0; t < 3; ++t) P[t] = own + (t - 3) * st + (m0 + t - 3 < ng ? dl : 0);
#pragma unroll
        for (int t = 3; t < 6; ++t) P[t] = own + (t - 3) * st + (m0 + t - 3 >= nD + ng ? dh : 0);
    }
    auto load = [&](int v, double* u, uint32_t z) {
        const int64_t ov = fq_aux<D>(v, o.thermo) * nc + z;
#pragma unroll
        for (int t = 0; t < 6; ++t) u[t] = P[t][ov];
    };
    double L[FQ_N], R[FQ_N];
    {
        double u[3][6];
        bool ok = true;
        load(0, u[0], 0u);
        load(1, u[1], 0u);
#pragma unroll
        for (int v = 0; v < FQ_N; ++v) {
            if (v + 2 < FQ_N) load(v + 2, u[(v + 2) % 3], 0u);
            __builtin_amdgcn_sched_barrier(0);
            const double* w = u[v % 3];
            if (ring && (v == FQ_YE || v == FQ_ENT)) { L[v] = 0.0; R[v] = 0.0; }
            else if constexpr (REC == 0) ok = wenoz_face(w[0], w[1], w[2], w[3], w[4], w[5], L[v], R[v]) && ok;
            else recon<REC>(w[1], w[2], w[3], w[4], L[v], R[v]);
            settle(L[v], R[v]);
        }
        // Some variable's products are out of range: each such variable takes
        // the other form, by itself.  (All of them at once would give a full
        // face another rounding than the ring face that the neighbour forms of
        // it without Y_e and entropy, and the blocks' face B would part.)
        if constexpr (REC == 0)
            if (!ok) {
                uint32_t again = 0;
                asm volatile("" : "+v"(again));
#pragma unroll
                for (int v = 0; v < FQ_N; ++v) {
                    if (ring && (v == FQ_YE || v == FQ_ENT)) continue;
                    load(v, u[0], again);
                    double lo, hi;
                    if (!wenoz_face(u[0][0], u[0][1], u[0][2], u[0][3], u[0][4], u[0][5], lo, hi))
                        wenoz_face_wide(u[0][0], u[0][1], u[0][2], u[0][3], u[0][4], u[0][5], L[v], R[v]);
                    settle(L[v], R[v]);
                }
            }
    }
    Met mf;
    bool excise = false;
    face_met<FLAT, D>(G, f, o.ex.alp_ex, q, i, j, k, st, mf, excise);
    if constexpr (!FLAT)
        if (excise) {
#pragma unroll
            for (int v = 0; v < FQ_N; ++v) {
                const int64_t ov = fq_aux<D>(v, o.thermo) * nc;
                L[v] = P[2][ov]; R[v] = P[3][ov];
            }
        }
    double V[4], F[7];
    face_solve<EOS, FLAT, D>(eos, o, mf, L, R, Bf / mf.sqrtg, ring, V, F);
    const int64_t ns = G.ns;
    const uint32_t so = (uint32_t)sidx(G, i, j, k) * 8u;
    double* V0 = f.vbar[D] + q * 4 * ns;
#pragma unroll
    for (int v = 0; v < 4; ++v) st_off(V0 + v * ns, so, V[v]);
    if (ring) return;
    double* F0 = f.flux[D] + q * NHRSC * ns;
#pragma unroll
    for (int v = 0; v < NHRSC; ++v) st_off(F0 + v * ns, so, F[v]);
}

// The faces of f.ndir directions of every block, one thread per face.  The
// workgroups of a block follow each other direction by direction, plane by
// plane along z, on one XCD (wg_pos_in), then the next block's: the three
// directions read the same nine primitives, and the second and third find
// them in that XCD's L2.  Ring faces (many in the first RK stage, and in every
// stage of a forest and of a curved grid without a cached metric that agrees
// across block faces) come behind the full faces of all blocks: their threads
// are shorter.
//
// Bound by the FP64 units (about 350 us of arithmetic for 512 blocks of
// 16^3) beside the stores of fluxes and face values: 535 us per launch there
// in the RK stages that share ring faces, 725 with them (500 and 430, the
// latter without the flux stores, on a card with faster memory); one launch
// per direction over rows in the boundary's layout, which also copied its
// outer face values into the neighbours' ring slots, took 3 x 245.  (The edge
// EMFs read them from the neighbour instead: 130 MB less to write.)  A thread
// per face with nine variables one after another needs 126 VGPRs (4 waves per
// SIMD; curved 167, 3 waves: the bound of 3 keeps the hybrid EOS from 169).  A thread that walks along a line of
// faces saves the shared half of the reconstruction but keeps the stencils of
// nine variables: 230 VGPRs, 2 waves, 1.0 ms for y and 0.9 for z per three
// stages against 0.67 and 0.64 here; with the stencil read again at each step
// 1.1 and 1.0.
template <typename EOS, int REC, bool FLAT>
__global__ __launch_bounds__(256, 3) void k_flux(DevGrid G, EOS eos, Opts o, FluxArgs f) {
    const uint32_t nfull = (uint32_t)(f.tiles * f.ndir) * (uint32_t)G.nq;
    const bool ring = blockIdx.x >= nfull;
    const WgPos wp = ring ? wg_pos_in(blockIdx.x - nfull, gridDim.x - nfull, f.tilesr * f.ndir)
                          : wg_pos_in(blockIdx.x, nfull, f.tiles * f.ndir);
    int t, d;
    udivmod(wp.tile, f.ndir, t, d);
    const int e = t * (int)blockDim.x + (int)threadIdx.x;
    switch (f.dir0 + d) {
        case 0: flux_face<EOS, REC, FLAT, 0>(G, eos, o, f, wp.q, e, ring); break;
        case 1: flux_face<EOS, REC, FLAT, 1>(G, eos, o, f, wp.q, e, ring); break;
        default: flux_face<EOS, REC, FLAT, 2>(G, eos, o, f, wp.q, e, ring); break;
    }
}

// Fluxes and face EMFs for GS: face e of direction D of block q, of every face
// (FOFC widens the normal range by one face on each side; only: its correction
// pass, evolve.cpp:646-702, the tagged faces of the normal range [ng, n + ng]).
// WENO-Z is formed from the candidates, every quotient is an IEEE division and
// the wave speeds are get_cm_cp's, for the sign of the mass flux: the edge EMF
// takes a side by it, and where nothing flows (between two cells reset to the
// floor, in a stationary flow) that sign is rounding.  With k_flux's forms B
// is off by 0.2 of its largest value at single faces beside floored cells,
// which is why this path is not k_flux's.
template <typename EOS, int REC, bool FLAT, int D>
__device__ __forceinline__ void gs_face(const DevGrid& G, const EOS& eos, const Opts& o, const FluxArgs& f,
                                        const uint8_t* only, int64_t q, int e) {
    constexpr int T0 = D == 0 ? 1 : 0, T1 = D == 2 ? 1 : 2;
    const int N0 = G.N[T0], N1 = G.N[T1], Rg = G.n[D] + 1 + 2 * o.fofc;
    if (e >= Rg * N0 * N1) return;
    int a, b, c, r;
    if (D == 0) { udivmod(e, Rg, r, a); udivmod(r, N0, c, b); }
    else if (D == 1) { udivmod(e, N0, r, b); udivmod(r, Rg, c, a); }
    else { udivmod(e, N0, r, b); udivmod(r, N1, a, c); }
    a += G.ng - o.fofc;
    const int i = D == 0 ? a : b, j = D == 1 ? a : (D == 0 ? b : c), k = D == 2 ? a : c;
    if (only && (a < G.ng || a > G.ng + G.n[D] || !only[q * G.nface[D] + fidx<D>(G, i, j, k)])) return;
    const int64_t nc = G.ncell;
    const int64_t c0 = cidx(G, i, j, k);
    const int64_t st = D == 0 ? 1 : (D == 1 ? G.N[0] : (int64_t)G.N[0] * G.N[1]);
    const double* A = f.aux + q * NAUX * nc;
    Met mf;
    bool excise = false;
    face_met<FLAT, D>(G, f, o.ex.alp_ex, q, i, j, k, st, mf, excise);
    // reconstruction of RHO Z(3) YE THERMO ENT B(3)
    const int th_aux = o.thermo ? PRESS_ : TEMP_;
    const int ridx[10] = {RHO_, ZVECX_, ZVECY_, ZVECZ_, YE_, th_aux, ENTROPY_, BX_, BY_, BZ_};
    const int rloc[10] = {RHOL, ZXL, ZYL, ZZL, YEL, o.thermo ? PRESSL : TEMPL, ENTL, BXL, BYL, BZL};
    double pL[NPRIM], pR[NPRIM];
#pragma unroll
    for (int v = 0; v < 10; ++v) {
        // (the normal B component is replaced by the face value below)
        if (v == 7 + D) { pL[rloc[v]] = 0.0; pR[rloc[v]] = 0.0; continue; }
        double uL, uR;
        const double* P = A + ridx[v] * nc + c0;
        if (!FLAT && excise) { uL = P[-st]; uR = P[0]; }
        else if constexpr (REC == 0) wenoz(P[-3 * st], P[-2 * st], P[-st], P[0], P[st], P[2 * st], uL, uR);
        else recon<REC>(P[-2 * st], P[-st], P[0], P[st], uL, uR);
        pL[rloc[v]] = uL; pR[rloc[v]] = uR;
    }
    double Bn = f.B[D][q * G.nface[D] + fidx<D>(G, i, j, k)] / mf.sqrtg;
    pL[BXL + D] = Bn; pR[BXL + D] = Bn;
    unsigned ee = 0;
    if (o.thermo) {
        double h, s;
        pL[EPSL] = eos.eps_from_press(h, pL[CS2L], pL[TEMPL], s, pL[PRESSL], pL[RHOL], ee);
        pR[EPSL] = eos.eps_from_press(h, pR[CS2L], pR[TEMPL], s, pR[PRESSL], pR[RHOL], ee);
    } else {
        pL[PRESSL] = eos.press_from_temp(pL[EPSL], pL[CS2L], pL[TEMPL], pL[RHOL], ee);
        pR[PRESSL] = eos.press_from_temp(pR[EPSL], pR[CS2L], pR[TEMPL], pR[RHOL], ee);
    }
    // compute_mhd_fluxes (grmhd.hh:774-970)
    const double *zl = &pL[ZXL], *zr = &pR[ZXL], *Bl = &pL[BXL], *Br = &pR[BXL];
    double wl = lorentz<FLAT>(mf.g, zl), wr = lorentz<FLAT>(mf.g, zr);
    double bl[4], br[4], b2l, b2r;
    smallb<FLAT>(mf, Bl, zl, wl, bl, b2l);
    smallb<FLAT>(mf, Br, zr, wr, br, b2r);
    double vtl[3], vtr[3];
    vtilde(mf, zl, wl, vtl);
    vtilde(mf, zr, wr, vtr);
    double cml, cpl, cmr, cpr, cmin, cmax;
    cmcp<FLAT>(mf, pL[RHOL], pL[PRESSL], pL[EPSL], pL[CS2L], wl, b2l, vtl, D, cml, cpl);
    cmcp<FLAT>(mf, pR[RHOL], pR[PRESSL], pR[EPSL], pR[CS2L], wr, b2r, vtr, D, cmr, cpr);
    if (o.riemann == 1) {
        cmax = fmax(fmax(fabs(cml), fabs(cmr)), fmax(fabs(cpl), fabs(cpr)));
        if (fmin(pL[RHOL], pR[RHOL]) < o.c_limit) {
            double gdd = D == 0 ? mf.gi[0] : (D == 1 ? mf.gi[3] : mf.gi[5]);
            cmax = fmax(cmax, mf.alp * sqrt(gdd) + fabs(mf.beta[D]));
        }
        cmin = cmax;
    } else {
        cmin = -fmin(0., fmin(cml, cmr));
        cmax = fmax(0., fmax(cpl, cpr));
    }
    if (cmin < 1e-12 && cmax < 1e-12) { cmin = 1; cmax = 1; }
    const double ihll = 1.0 / (cmax + cmin);   // shared by the HLL fluxes of this face
    const int64_t so = sidx(G, i, j, k), ns = G.ns;
    double* V = f.vbar[D] + q * 4 * ns + so;
    double Dl, taul, Sl[3], Esl, Dr, taur, Sr[3], Esr;
    conserved<FLAT>(mf, pL[RHOL], pL[PRESSL], pL[EPSL], zl, pL[ENTL], wl, b2l, bl, Dl, taul, Sl, Esl);
    conserved<FLAT>(mf, pR[RHOL], pR[PRESSL], pR[EPSL], zr, pR[ENTL], wr, b2r, br, Dr, taur, Sr, Esr);
    // fluxes along D (grmhd_subexpressions.hh:97-156)
    double bsh[3]; lower3(mf.g, mf.beta[0], mf.beta[1], mf.beta[2], bsh);
    double ia2 = 1. / (mf.alp * mf.alp);
    double Fl[7], Fr[7];
    {
        double rhoh = b2l + pL[EPSL] * pL[RHOL] + pL[PRESSL] + pL[RHOL];
        double ps = 0.5 * b2l + pL[PRESSL];
        double W2rh = wl * wl * rhoh;
        double fD = vtl[D] * Dl;
        Fl[0] = fD;
        double blo[3]; lower3<FLAT>(mf.g, bl[1], bl[2], bl[3], blo);
        double vlo[3]; lower3<FLAT>(mf.g, vtl[0], vtl[1], vtl[2], vlo);
        if constexpr (FLAT) {
            Fl[4] = W2rh * vtl[D] - bl[0] * bl[1 + D] - fD;
            const double c = vtl[D] * W2rh;
            for (int a = 0; a < 3; ++a)
                Fl[1 + a] = a == D ? -bl[1 + D] * blo[a] + ps + c * vlo[a] : -bl[1 + D] * blo[a] + c * vlo[a];
        } else {
            Fl[4] = W2rh * vtl[D] + ps * mf.beta[D] - mf.alp * mf.alp * bl[0] * bl[1 + D] - fD;
            const double c = vtl[D] * W2rh * ia2;
            for (int a = 0; a < 3; ++a)
                Fl[1 + a] = mf.alp * (-bl[1 + D] * (blo[a] + bl[0] * bsh[a]) + (a == D ? ps : 0.0) + c * (vlo[a] + bsh[a]));
        }
        Fl[6] = vtl[D] * Esl;
        Fl[5] = pL[YEL] * fD;
    }
    {
        double rhoh = b2r + pR[EPSL] * pR[RHOL] + pR[PRESSL] + pR[RHOL];
        double ps = 0.5 * b2r + pR[PRESSL];
        double W2rh = wr * wr * rhoh;
        double fD = vtr[D] * Dr;
        Fr[0] = fD;
        double blo[3]; lower3<FLAT>(mf.g, br[1], br[2], br[3], blo);
        double vlo[3]; lower3<FLAT>(mf.g, vtr[0], vtr[1], vtr[2], vlo);
        if constexpr (FLAT) {
            Fr[4] = W2rh * vtr[D] - br[0] * br[1 + D] - fD;
            const double c = vtr[D] * W2rh;
            for (int a = 0; a < 3; ++a)
                Fr[1 + a] = a == D ? -br[1 + D] * blo[a] + ps + c * vlo[a] : -br[1 + D] * blo[a] + c * vlo[a];
        } else {
            Fr[4] = W2rh * vtr[D] + ps * mf.beta[D] - mf.alp * mf.alp * br[0] * br[1 + D] - fD;
            const double c = vtr[D] * W2rh * ia2;
            for (int a = 0; a < 3; ++a)
                Fr[1 + a] = mf.alp * (-br[1 + D] * (blo[a] + br[0] * bsh[a]) + (a == D ? ps : 0.0) + c * (vlo[a] + bsh[a]));
        }
        Fr[6] = vtr[D] * Esr;
        Fr[5] = pR[YEL] * fD;
    }
    double* F = f.flux[D] + q * NHRSC * ns + so;
    const double sg = mf.sqrtg;
    F[DENS_ * ns] = sg * hll_r(Fl[0], Fr[0], Dl, Dr, cmin, cmax, ihll);
    F[ENTROPYSTAR_ * ns] = sg * hll_r(Fl[6], Fr[6], Esl, Esr, cmin, cmax, ihll);
    F[TAU_ * ns] = sg * hll_r(Fl[4], Fr[4], taul, taur, cmin, cmax, ihll);
    F[SX_ * ns] = sg * hll_r(Fl[1], Fr[1], Sl[0], Sr[0], cmin, cmax, ihll);
    F[SY_ * ns] = sg * hll_r(Fl[2], Fr[2], Sl[1], Sr[1], cmin, cmax, ihll);
    F[SZ_ * ns] = sg * hll_r(Fl[3], Fr[3], Sl[2], Sr[2], cmin, cmax, ihll);
    F[YESTAR_ * ns] = sg * hll_r(Fl[5], Fr[5], pL[YEL] * Dl, pR[YEL] * Dr, cmin, cmax, ihll);
    {  // face EMFs (grmhd.hh:937-969)
        if (D == 0) {
            double a = -Bl[0] * vtl[2] + Bl[2] * vtl[0], b = -Br[0] * vtr[2] + Br[2] * vtr[0];
            V[0] = sg * hll_r(a, b, Bl[2], Br[2], cmin, cmax, ihll);
            a = -Bl[0] * vtl[1] + Bl[1] * vtl[0]; b = -Br[0] * vtr[1] + Br[1] * vtr[0];
            V[ns] = -sg * hll_r(a, b, Bl[1], Br[1], cmin, cmax, ihll);
        } else if (D == 1) {
            double a = -Bl[1] * vtl[2] + Bl[2] * vtl[1], b = -Br[1] * vtr[2] + Br[2] * vtr[1];
            V[0] = -sg * hll_r(a, b, Bl[2], Br[2], cmin, cmax, ihll);
            a = Bl[0] * vtl[1] - Bl[1] * vtl[0]; b = Br[0] * vtr[1] - Br[1] * vtr[0];
            V[ns] = sg * hll_r(a, b, Bl[0], Br[0], cmin, cmax, ihll);
        } else {
            double a = Bl[1] * vtl[2] - Bl[2] * vtl[1], b = Br[1] * vtr[2] - Br[2] * vtr[1];
            V[0] = sg * hll_r(a, b, Bl[1], Br[1], cmin, cmax, ihll);
            a = Bl[0] * vtl[2] - Bl[2] * vtl[0]; b = Br[0] * vtr[2] - Br[2] * vtr[0];
            V[ns] = -sg * hll_r(a, b, Bl[0], Br[0], cmin, cmax, ihll);
        }
    }
}

// The directions of a block follow each other, as in k_flux.  One launch for
// the three: torus forest 2540 -> 2411 us per step, curved 80^3 2116 -> 1995,
// 24^3 209 -> 172 against a launch per direction (2523, 2037 and 499 with
// those on three streams).
struct FaceTags { const uint8_t* d[3]; };
template <typename EOS, int REC, bool FLAT>
__global__ __launch_bounds__(256) void k_flux_gs(DevGrid G, EOS eos, Opts o, FluxArgs f, FaceTags only) {
    const WgPos wp = wg_pos(f.tiles * f.ndir);
    int t, d;
    udivmod(wp.tile, f.ndir, t, d);
    const int e = t * (int)blockDim.x + (int)threadIdx.x;
    switch (f.dir0 + d) {
        case 0: gs_face<EOS, REC, FLAT, 0>(G, eos, o, f, only.d[0], wp.q, e); break;
        case 1: gs_face<EOS, REC, FLAT, 1>(G, eos, o, f, only.d[1], wp.q, e); break;
        default: gs_face<EOS, REC, FLAT, 2>(G, eos, o, f, only.d[2], wp.q, e); break;
    }
}
