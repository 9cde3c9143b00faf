// Stage kernel for small meshes (gfx950): the same stage of a block of BE
// elements as stage_kernel, spread over four wavefronts.
//
// stage_kernel runs a block on one wavefront, whose chain of three surface
// passes, the indicator and three volume passes takes 15 (weak form) to 90 us
// (FP64, N = 4) however few blocks there are: on a mesh of fewer blocks than
// the chip has SIMDs (1024) that chain is the whole launch, and most of the
// chip waits.  Here wavefronts 0..2 take one direction each (the face fluxes
// and volume terms of its lines stay in registers), wavefront 3 computes the
// blending factor meanwhile, and the 256 threads own one node each for the
// loads, the Runge-Kutta update, the positivity check and the CFL partials.
// The terms are added to the node accumulators in the order of stage_kernel,
// a barrier apart, with the same operations: Euler results have the same bits
// in both forms; GLM-MHD sums rotated states and agrees to rounding.
#pragma once

#include "dg_stage.hpp"

namespace nemo {

constexpr int WIDE_NT = CFL_NT;

// Variable in row h of a state rotated to direction d.
__device__ __forceinline__ int rotated_row(int h, int d) {
    return (h >= 1 && h <= 3) ? 1 + (d + h - 1) % 3 : ((h >= 5 && h <= 7) ? 5 + (d + h - 5) % 3 : h);
}

template <int EQ, int M, int BE, int VOL, int SURF, typename Real, int IK>
__device__ __forceinline__ void stage_block_wide(const StageArgs<M, Real>& a, const long long blk, double* lds,
                                                 Real* s_alpha, unsigned long long* s_max, int* s_bad) {
    using Sh = StageShape<M, BE>;
    using L = StageLds<EQ, M, BE, Real>;
    using TU = typename L::TU;
    constexpr int M2 = Sh::M2, M3 = Sh::M3, NN = Sh::NN, NT = Sh::NT;
    static_assert(NN <= WIDE_NT && NT <= 64, "a node per thread, a direction's lines per wavefront");
    static_assert(L::DOUBLES >= 3 * CFL_NT, "the CFL reduction runs in the operator's LDS");
    constexpr int V = NVars<EQ>::V;
    constexpr bool COMPACT = L::COMPACT;
    double* s_p64 = lds + L::RAW_DOUBLES;
    TU (*s_u)[NN] = reinterpret_cast<TU (*)[NN]>(lds);
    Real (*s_acc)[NN] = reinterpret_cast<Real (*)[NN]>(reinterpret_cast<TU*>(lds) + V * NN);
    double (*s_u64)[NN] = reinterpret_cast<double (*)[NN]>(lds);

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const long long e0 = blk * BE;
    const long long EM3 = a.nelem * (long long)M3;
    const int nvalid = int(a.nelem - e0 < BE ? a.nelem - e0 : BE) * M3;
    const bool own = tid < nvalid;                        // this thread's node
    const long long gi0 = own ? e0 * M3 + tid : 0;        // (other threads read node 0 of element 0)
    const int sl = tid < NN ? slot<M>(tid) : 0;
    const bool lines = lane < NT;                         // lanes beyond the tile repeat line 0 and write nothing
    const int ln = lines ? lane : 0;
    const int el = ln / M2;

    double glm_alpha = 0.0;
    MhdGas<Real> mg = a.mhd;
    if constexpr (EQ == EQ_MHD) {
        mg.ch = Real(a.glm[0]);
        glm_alpha = a.glm[1];
    }

    // ---- loads: the thread's node, the line's face nodes -----------------
    double u[V], r0v[V], r1v[V];
    float r0f[V];
    const int s = a.stage;
    const bool lsrk = a.timedisc == TD_LSRK54;
    const bool update = a.rhs_out == nullptr;
#pragma unroll
    for (int h = 0; h < V; ++h) {
        u[h] = a.u_in[h * EM3 + gi0];
        r0v[h] = r1v[h] = 0.0;
        r0f[h] = 0.0f;
    }
    // The Runge-Kutta registers of the node, requested when the terms are
    // formed (their registers are free then), in time for the update behind
    // the additions.
    auto load_registers = [&]() __attribute__((always_inline)) {
        if (!update || s == 1) return;
#pragma unroll
        for (int h = 0; h < V; ++h) {
            const long long gi = h * EM3 + gi0;
            if (COMPACT && lsrk)
                r0f[h] = reinterpret_cast<const float*>(a.r0)[gi];
            else
                r0v[h] = a.r0[gi];
            if (!lsrk && s >= 3) r1v[h] = a.r1[gi];
        }
    };
    // The line of this lane in direction d = its wavefront (wavefront 3: x,
    // unused): first node n0, stride nst.
    const int d = wave < 3 ? wave : 0;
    const int line = ln - el * M2, ta = line % M, tb = line / M;
    auto first_node = [=](int k) { return k == 0 ? M * ta + M2 * tb : (k == 1 ? ta + M2 * tb : ta + M * tb); };
    auto node_stride = [](int k) { return k == 0 ? 1 : (k == 1 ? M : M2); };
    const int n0 = first_node(d), nst = node_stride(d);
    double um[V], up[V];
    const long long ec = e0 + el < a.nelem ? e0 + el : 0;
    const long long em = a.nbr[ec * 6 + 2 * d], ep = a.nbr[ec * 6 + 2 * d + 1];
    const double dx = a.delta[ec * 3 + d];
    {
        // across a mortar or boundary face the element's own face node (its
        // flux is discarded)
        const long long om = (em < 0 ? ec : em) * M3 + n0 + (em < 0 ? 0 : (M - 1) * nst);
        const long long op = (ep < 0 ? ec : ep) * M3 + n0 + (ep < 0 ? (M - 1) * nst : 0);
#pragma unroll
        for (int h = 0; h < V; ++h) {
            const int r = EQ == EQ_MHD ? rotated_row(h, d) : h;
            um[h] = a.u_in[r * EM3 + om];
            up[h] = a.u_in[r * EM3 + op];
        }
    }
    if (tid < NN) {
#pragma unroll
        for (int h = 0; h < V; ++h) s_u[h][sl] = TU(u[h]);
        if constexpr (COMPACT) s_p64[sl] = pressure64<EQ>(a.ph64, u);
    }
    if (tid < 4 * BE) s_max[tid] = 0ull;
    if (tid == 0) *s_bad = 0;
    __syncthreads();

    // ---- directions and indicator side by side ---------------------------
    // Every wavefront passes the same barriers: one after which the blending
    // factors are known and the indicator's work rows are free, then one
    // after each addition to the accumulators.
    // The code of direction d.  With ONE_COPY it is the x code on states
    // rotated to direction d at run time (D = 0, `d` a variable): row h of them
    // is variable row[h].  Otherwise D = d and nothing is rotated.
    // One copy where the code is long: three copies of the MHD passes do not
    // fit the instruction cache (HLLD, N = 3, 128 blocks: 40.9 -> 21.4 us).  The
    // Euler passes keep one per direction, whose LDS offsets are constants
    // (FP32, N = 3, 1024 blocks: 21.2 us against 24.2), and the bits of
    // stage_kernel.
    constexpr bool ONE_COPY = EQ == EQ_MHD;
    auto direction = [&](auto dtag, const int d) __attribute__((always_inline)) {
        constexpr int D = decltype(dtag)::value;
        int row[V], ns[M];
#pragma unroll
        for (int h = 0; h < V; ++h) row[h] = ONE_COPY ? rotated_row(h, d) : h;
#pragma unroll
        for (int i = 0; i < M; ++i) ns[i] = bslot<M>(el * M3, first_node(d) + i * node_stride(d));
        // the order of stage_kernel's volume passes
        constexpr bool XLAST = EQ == EQ_EULER && sizeof(Real) == 8 && VOL == VOL_EC && M <= 4;
        const int rank = XLAST ? (d + 2) % 3 : d;
        Real c[M][V], fm[V], fp[V];
        if constexpr (EQ == EQ_EULER) {
            ElemGeom geo;
            geo.nbr[2 * D] = int32_t(em);
            geo.nbr[2 * D + 1] = int32_t(ep);
            geo.dx[D] = dx;
            Real jac;
            surface_fluxes<D, M, BE, SURF, Real, TU>(a, ln, e0, s_u, s_p64, geo, um, up, fm, fp, jac);
            // the volume pass reads its nodes anew, as in stage_kernel: shared
            // with the face solves, its expressions would be contracted into
            // other FMAs (other last bits) and hold more registers
            asm volatile("" ::: "memory");
            NodeState<Real> S[M];
            Real vjac;
            volume_terms<D, M, BE, VOL, Real, TU, false>(a, ln, e0, s_u, s_p64, geo, S, c, vjac);
            __syncthreads();
            blend_fv<D, M, SURF, Real>(a, S, vjac, s_alpha[el], c);
            load_registers();
#pragma unroll
            for (int p = 0; p < 3; ++p) {
                if (p == D && lines) surface_add<D, M, BE, Real>(a, ln, s_acc, fm, fp, jac);
                __syncthreads();
            }
        } else {
            auto mortar = [&](long long slot, Real (&f)[V]) __attribute__((always_inline)) {
                const double* mf = a.mortar_flux + size_t(slot) * V * M2 + ta + M * tb;
#pragma unroll
                for (int h = 0; h < V; ++h) f[h] = Real(mf[row[h] * M2]);
            };
            MhdState<Real> S[M], Nm, Np;
#pragma unroll
            for (int i = 0; i < M; ++i) {
#pragma unroll
                for (int h = 0; h < V; ++h) S[i].u[h] = Real(s_u[row[h]][ns[i]]);
                mhd_make_state<VOL == VOL_EC>(mg, S[i]);
            }
#pragma unroll
            for (int h = 0; h < V; ++h) {
                Nm.u[h] = Real(um[h]);
                Np.u[h] = Real(up[h]);
            }
            mhd_face_fluxes<0, M, SURF, Real>(mg, S, Nm, Np, fm, fp);
            const Real jac = Real(2.0 / dx);
            if (em < 0) mortar(-em - 1, fm);
            if (ep < 0) mortar(-ep - 1, fp);
            mhd_volume_dg<0, M, VOL, Real>(a, mg, S, fm, fp, jac, c);
            __syncthreads();
            mhd_blend_fv<0, M, SURF, Real>(a, mg, S, fm, fp, jac, s_alpha[el], c);
            load_registers();
        }
#pragma unroll
        for (int p = 0; p < 3; ++p) {
            if (p == rank && lines) {
#pragma unroll
                for (int i = 0; i < M; ++i)
#pragma unroll
                    for (int h = 0; h < V; ++h) {
                        if (EQ == EQ_MHD && p == 0)
                            s_acc[row[h]][ns[i]] = c[i][h];
                        else
                            s_acc[row[h]][ns[i]] += c[i][h];
                    }
            }
            __syncthreads();
        }
    };
    if (wave < 3) {
        if (ONE_COPY)
            direction(std::integral_constant<int, 0>{}, d);
        else if (wave == 0)
            direction(std::integral_constant<int, 0>{}, 0);
        else if (wave == 1)
            direction(std::integral_constant<int, 1>{}, 1);
        else
            direction(std::integral_constant<int, 2>{}, 2);
    } else {
        if (lines) {
            Real alpha = Real(0);
            if constexpr (IK == IK_MLP) {
                alpha = indicator_mlp<EQ, M, BE, Real, TU, true>(a, lane, e0, s_u, s_acc, s_p64);
            } else if constexpr (IK == IK_STORED) {
                alpha = e0 + el < a.nelem ? Real(a.alpha_step[e0 + el]) : Real(0);
            } else if (a.indicator == IND_PP) {
                alpha = indicator_pp<EQ, M, BE, Real, TU, true>(a, lane, e0, s_u, s_acc, s_p64);
            }
            s_alpha[el] = alpha;
        }
        load_registers();
        constexpr int BARRIERS = EQ == EQ_EULER ? 7 : 4;
#pragma unroll
        for (int p = 0; p < BARRIERS; ++p) __syncthreads();
    }

    // ---- the thread's node: time derivative, probe ------------------------
    double f[V];
    if (tid < NN) {
#pragma unroll
        for (int h = 0; h < V; ++h) {
            if constexpr (!COMPACT) u[h] = s_u[h][sl];  // (not held across the passes)
            f[h] = double(s_acc[h][sl]);
            if constexpr (EQ == EQ_MHD)
                if (h == GLMP) f[h] = f[h] - glm_alpha * u[h];
        }
    }
    if (!update) {
        if (own)
#pragma unroll
            for (int h = 0; h < V; ++h) a.rhs_out[h * EM3 + gi0] = f[h];
        return;
    }
    const double dt = a.dt_run ? a.dt_run[a.block_run[blk]] : (a.dt_dev ? *a.dt_dev : a.dt);
    double st[V];
    if (own) {
#pragma unroll
        for (int h = 0; h < V; ++h) {
            const long long gi = h * EM3 + gi0;
            if (COMPACT && lsrk) {
                // FP32 register, rounded once (as in stage_block)
                const float rg = float(s == 1 ? f[h] : a.rk.lsrk_a[s - 1] * double(r0f[h]) + f[h]);
                reinterpret_cast<float*>(a.r0)[gi] = rg;
                st[h] = u[h] + a.rk.lsrk_c[s - 1] * dt * double(rg);
            } else if (lsrk) {
                st[h] = probe_lsrk(a, gi, s, dt, u[h], r0v[h], f[h]);
            } else {
                const double* k = a.rk.ssp;
                switch (s) {
                case 1: st[h] = u[h] + k[3] * dt * f[h]; a.r0[gi] = u[h]; break;
                case 2: st[h] = k[5] * r0v[h] + k[6] * u[h] + k[7] * dt * f[h]; break;
                case 3: st[h] = k[9] * r0v[h] + k[10] * u[h] + k[11] * dt * f[h]; break;
                case 4:
                    st[h] = k[13] * r0v[h] + k[14] * u[h] + k[15] * dt * f[h];
                    a.r1[gi] = r1v[h] + k[22] * dt * f[h];
                    break;
                default: st[h] = k[17] * r0v[h] + k[18] * u[h] + k[19] * dt * f[h] + r1v[h]; break;
                }
            }
        }
    }

    // ---- positivity repair -------------------------------------------------
    if (a.repair) {
        if (own && !isvalid64<EQ>(a.ph64, st)) *s_bad = 1;
        __syncthreads();  // also: the accumulators have been read
        if (*s_bad) {
            if (own)
#pragma unroll
                for (int h = 0; h < V; ++h) s_u64[h][sl] = st[h];
            __syncthreads();
            // (elements without an invalid node come back unchanged)
            if (tid < BE && e0 + tid < a.nelem) {
                double* su[V];
#pragma unroll
                for (int h = 0; h < V; ++h) su[h] = s_u64[h];
                if (!repair_element<EQ, M>(a.ph64, a.rk.w64, su, tid * M3)) *(volatile int*)a.status = 1;
            }
            __syncthreads();
            if (own)
#pragma unroll
                for (int h = 0; h < V; ++h) st[h] = s_u64[h][sl];
        }
    }

    // ---- new state; SSP register r1 takes the repaired state ---------------
    if (own) {
#pragma unroll
        for (int h = 0; h < V; ++h) {
            const long long gi = h * EM3 + gi0;
            a.u_out[gi] = st[h];
            if (!lsrk) {
                if (s == 2) a.r1[gi] = a.rk.ssp[20] * st[h];
                else if (s == 3) a.r1[gi] = r1v[h] + a.rk.ssp[21] * st[h];
            }
        }
    }

    // ---- CFL partials of the new state (last stage of a step) -------------
    if (a.cfl_part) {
        block_cfl_nodes<EQ, M, BE>(a.ph64, a.delta, e0, a.nelem, own, st, s_max, a.cfl_part + 4 * blk);
        if (a.fin.ticket) {
            __syncthreads();  // the operator's LDS is free
            cfl_last_block(a.cfl_part, int(gridDim.x), a.fin, M, reinterpret_cast<double (*)[CFL_NT]>(lds), s_bad);
        }
    }
}

// Two workgroups on a CU: left to themselves the FP64 Euler passes and the FP32
// MHD ones take 256 VGPRs and a few AGPRs, which allow one (FP32 MHD, N = 4,
// 2916 blocks: 144.7 -> 95.6 us).  FP64 GLM-MHD does not fit in 256.
template <int EQ, int M, int BE, int VOL, int SURF, typename Real, int IK = IK_RUNTIME>
__global__ __launch_bounds__(WIDE_NT) __attribute__((amdgpu_waves_per_eu(EQ == EQ_EULER || sizeof(Real) == 4 ? 2 : 1)))
void stage_kernel_wide(StageArgs<M, Real> a) {
    __shared__ __align__(16) double lds[StageLds<EQ, M, BE, Real>::DOUBLES];
    __shared__ unsigned long long s_max[4 * BE];
    __shared__ Real s_alpha[BE];
    __shared__ int s_bad;
    const long long nblocks = (a.nelem + BE - 1) / BE;
    stage_block_wide<EQ, M, BE, VOL, SURF, Real, IK>(a, xcd_block(nblocks), lds, s_alpha, s_max, &s_bad);
}

}  // namespace nemo
