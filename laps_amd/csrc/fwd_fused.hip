// fwd_fused.hip -- forward y and z passes of the fluxes with the spectral
// divergence / curl folded in, and the RK3 update folded into the z pass.
//
// Reference: calc_rhs (mhdrhs.f90:174-279), rkt (rktmod.f90:34-62),
// dealias (dealiasing.f90:70-113) and the y/z legs of
// transform_flux_real_to_fourier (fftw.f90:136-180).
//
// fnl = -(kx F_a + ky F_b + kz F_c) (k = i*k') is linear and each derivative
// factor depends only on modes the pass already knows: kx' and ky' on the y
// pass output, kz' on the z pass output. So the y pass of a divergence group
// (F_a, F_b, F_c) writes  G = -i kx' Y(F_a) - i ky' Y(F_b)  and  Y(F_c)
// (three fields in, two out; the expanding box's energy source is added to G), and the z pass
// forms fnl = Z(G) - i kz' Z(Y F_c)
// per mode, where the RK3 update, implicit diffusion and dealiasing follow in
// registers. The induction fields E are transformed as they are and -i k' x E is formed in the z
// pass (kx', ky' are constants of its column): three fields pass through memory where partial
// curls formed in the y pass took five, as the three work-groups of a column that share them run
// side by side on one XCD. The mass flux is not transformed at all (MassArgs).
// With corotating AEB, kx' and ky' both depend on (kx, ky); both are known per
// output mode of the y pass and per column of the z pass.

#include <type_traits>

#include "internal.hpp"
#include "physics_dev.hpp"

namespace laps {

// ZP: the z pass, whose blocks also carry the RHS and RK3 update. The passes use the plan of
// radices <= 8 (8 values per work-item, so a block keeps one transform's result live across
// the next at 4-5 waves per SIMD), except the FP32 y pass at 256, which runs faster on the
// two-stage radix-16x16 plan (one LDS exchange, 16 values per work-item: 2.62 against 3.15
// ms per mixed phase-shift step). On that plan the FP32 z pass ran at 2 waves per SIMD
// (236 registers) and took 2.83 ms; on the low-radix plan 2.74 ms, and 2.58 ms on its
// variant with 32 busy work-items per line and 16 columns (PlanLowW; the FP64 passes on it
// need 150-180 registers, one block per CU, or spill).
// ALT (the y pass at 256 only): the wide 8·8·4 plan with 16 columns. FP32: instead of the
// two-stage plan with 32, for launches of one chain (0.82 -> 0.79 ms per mixed 2/3-rule step;
// with the two chains of phase shift the two-stage plan is faster, 2.47 against 2.69). FP64:
// instead of PlanLow with 8, for launches of two chains, held to 128 registers (92 bytes
// spilled; 4.56 -> 4.16 ms per phase-shift step; with one chain 1.17 -> 1.18, not used)
template <typename T, int N, bool ZP, bool ALT = false>
struct FwdCfg {
    // the FP32 z pass at 256 and the ALT y passes: the 8·8·4 plan with two last-stage
    // butterflies per work-item (32 per line, none idle) and 16 columns, 128-byte rows of D
    // and Uf in FP32, 256-byte rows of the y pass in FP64
    static constexpr bool WIDE = N == 256 && (ALT || (sizeof(T) == 4 && ZP));
    using P = std::conditional_t<(sizeof(T) == 4 && N == 256 && !ZP && !ALT), Plan<N>,
                                 std::conditional_t<WIDE, PlanLowW<N>, PlanLow<N>>>;
    using I = PlanInfo<N, P>;
    // columns per block: rows of 128 bytes (8 FP64 or 16 FP32 columns), 256 bytes for the FP32
    // y pass on the two-stage plan; the FP32 z pass has 16 columns only on the wide plan (on
    // PlanLow, 1024-work-item blocks, it measured slower at 256), else 8
    static constexpr int TX = (sizeof(T) == 8) ? (WIDE ? 16 : 8) : (WIDE ? 16 : (ZP ? 8 : (N == 256 ? 32 : 16)));
    static constexpr int TPL = I::TPL;
    static constexpr int NT = TX * TPL;
    static constexpr int LS = N + 1;
    // waves per SIMD the register allocation must allow: the z passes at 256, the FP32 y pass at
    // 256 on the two-stage plan and the FP64 ALT y pass (512-thread blocks, 66-72 KB of LDS) fit
    // two blocks per CU only at <= 128 VGPRs
    static constexpr int MINW = (N == 256 && (ZP || (sizeof(T) == 4 ? !ALT : ALT))) ? 4 : 1;
    static_assert(64 % TX == 0 && (NT % 64 == 0 || 64 % NT == 0), "every wave holds whole rows of the tile");
};

// derivative factors k' (real; the spectral factor is i*k'), mhdrhs.f90:192-204; r0r = R0/R,
// formed once per work-item (the reference's (k*R0)/R per mode, within an ulp)
__device__ __forceinline__ void kprime_xy(double wx, double wy, const PhysParams& pp, double r0r, double& kx,
                                          double& ky) {
    kx = wx;
    ky = wy * r0r;
    if (pp.corot_k) {
        kx = wx * pp.cos_c + wy * pp.sin_c;
        ky = (-wx * pp.sin_c + wy * pp.cos_c) * r0r;
    }
}

template <typename T>
__device__ __forceinline__ cpx<T> mul_i(T k, cpx<T> z) { return {-k * z.y, k * z.x}; }  // (i k) z

// The RK3 update (rktmod.f90:34-62), U <- (U + c_n fnl_n + d_n fnl_{n-1}) / implicit factor, with the
// previous right-hand side folded into the state it will be added to: a substage stores
// V = U_new + d_{n+1} fnl_n, and the next one reads V in the place of both (256^3 with phase shift:
// z pass 1004 -> 932 us in FP64, 703 -> 604 in mixed precision). Where the right-hand side holds the
// state itself (expanding box, explicit dissipation: L U), U is read again in the second substage
// only: for the third, whose right-hand side is not kept, c L U is folded into V too. Within a step U
// is stored where it is read again or is the z inverse's input (FP64; the mixed step transforms its
// FP32 copy).
__device__ __forceinline__ bool rhs_holds_u(const PhysParams& pp) {
    return pp.aeb || (pp.visc && pp.visc_exp) || (pp.resis && pp.resis_exp);
}
__device__ __forceinline__ bool store_u(bool fp64, int irk, const PhysParams& pp) {
    return fp64 || irk == 2 || (irk == 0 && rhs_holds_u(pp));
}

// rho of one box: fnl = -i k'.m_hat, the RK3 update (rktmod.f90:34-62) and the dealiasing
// (dealiasing.f90:70-113) of every stored mode; work-group blk of m.nblk, nt work-items each.
template <typename T>
__device__ __forceinline__ void mass_update(const MassArgs& m, const PhysParams& pp, const Ctl* __restrict__ ctl,
                                            int blk, int nt) {
    if (ctl->status != 0) return;  // uniform over the box: the step was refused
    cpx<double>* const U = m.U + blockIdx.y * m.u_bx;
    cpx<float>* const Uf = m.Uf ? m.Uf + blockIdx.y * m.uf_bx : nullptr;
    cpx<double>* const V = m.V + blockIdx.y * m.v_bx;
    const double r0r = pp.radius0 / ctl->radius, tau = ctl->tau;
    const double c = ctl->cc[m.irk], dn = m.irk < 2 ? ctl->dd[m.irk + 1] : 0.0, cl = ctl->cc[2];
    const bool wrU = store_u(sizeof(T) == 8, m.irk, pp);
    const bool masked = pp.dealias == 1 || pp.dealias == 3;
    const unsigned n = (unsigned)m.KXP * m.CY * m.CZ;  // below 2^31 on the supported grids
    for (unsigned i = blk * nt + threadIdx.x; i < n; i += m.nblk * nt) {
        const int kx = (int)(i % m.KXP);
        if (kx >= m.KX) continue;
        const unsigned row = i / m.KXP;
        const int cy = (int)(row % m.CY), cz = (int)(row / m.CY);
        if (masked) {
            const int lim = m.tb.kzlim[cy * m.KX + kx], mz = m.tb.mz[cz];
            if (mz > lim || -mz > lim) {
                if (m.clear_outside) {
                    U[i] = cpx<double>{0.0, 0.0};
                    if (Uf) Uf[i] = cpx<float>{0.0f, 0.0f};
                }
                continue;
            }
        }
        cpx<double> mom[3];
#pragma unroll
        for (int a = 0; a < 3; ++a) {
            if constexpr (sizeof(T) == 4) {
                const cpx<float> q = Uf[(1 + a) * m.ufs + i];
                mom[a] = cpx<double>{double(q.x), double(q.y)};
            } else {
                mom[a] = U[(1 + a) * m.ufs + i];
            }
        }
        const cpx<double> base = m.irk != 0 ? V[i] : U[i];
        double kxp, kyp;
        kprime_xy(m.tb.wx[kx], m.tb.wy[cy], pp, r0r, kxp, kyp);
        const double kzp = m.tb.wz[cz] * r0r;
        const double sx = kxp * mom[0].x + kyp * mom[1].x + kzp * mom[2].x;
        const double sy = kxp * mom[0].y + kyp * mom[1].y + kzp * mom[2].y;
        cpx<double> fnl{sy, -sx};
        if (pp.aeb && m.irk != 2) {
            const cpx<double> u = m.irk != 0 ? U[i] : base;
            fnl = fnl - cpx<double>{(u.x * 2.0) / tau, (u.y * 2.0) / tau};
        }
        cpx<double> un{c * fnl.x + base.x, c * fnl.y + base.y};
        if (pp.dealias == 2) {
            const double fx = m.tb.fx[kx], fy = m.tb.fy[cy], fz = m.tb.fz[cz];
            un = {((un.x * fx) * fy) * fz, ((un.y * fx) * fy) * fz};
        }
        if (wrU) U[i] = un;
        if (Uf) Uf[i] = cpx<float>{float(un.x), float(un.y)};
        if (m.irk != 2) {
            cpx<double> vn{un.x + dn * fnl.x, un.y + dn * fnl.y};
            if (pp.aeb && m.irk == 1) vn = vn - cpx<double>{cl * ((un.x * 2.0) / tau), cl * ((un.y * 2.0) / tau)};
            store_stream(V + i, vn);
        }
    }
}

// ---------------------------------------------------------------- y pass
template <typename T, int N, bool ALT>
__global__ __launch_bounds__((FwdCfg<T, N, false, ALT>::NT), (FwdCfg<T, N, false, ALT>::MINW)) void k_yfwd_group(const cpx<T>* __restrict__ in,
                                                                 cpx<T>* __restrict__ out, YGArgs a,
                                                                 const cpx<T>* __restrict__ tw,
                                                                 const double* __restrict__ wxt,
                                                                 const double* __restrict__ wyf, PhysParams pp,
                                                                 const Ctl* __restrict__ ctl, int ntile, int nz) {
    using C = FwdCfg<T, N, false, ALT>;
    using I = typename C::I;
    // FP32: the derivative factors come from LDS tables of their y-dependent parts (below)
    constexpr bool TAB = sizeof(T) == 4;
    __shared__ cpx<T> sh[C::TX * C::LS];
    __shared__ cpx<T> stw[N];
    __shared__ double swy[TAB ? 1 : N];
    __shared__ T sax[TAB ? N : 1], say[TAB ? N : 1];
    ctl += blockIdx.y;             // batched boxes: one per grid row
    long long bid = blockIdx.x;
    const long long bpc = (long long)ntile * nz * a.ngroups;  // blocks per chain
    if (a.mass.nblk && bid >= bpc * a.nch) {
        mass_update<T>(a.mass, pp, ctl, (int)(bid - bpc * a.nch), C::NT);
        return;  // whole work-group, before any barrier
    }
    LdsTable<cpx<T>, N, C::NT> twt;
    LdsTable<double, N, C::NT> wyt;
    twt.fetch(tw);
    wyt.fetch(wyf);
    twt.put(stw);  // visible after the barrier that opens each transform
    if constexpr (!TAB) wyt.put(swy);
    const int l = threadIdx.x % C::TX, j = threadIdx.x / C::TX;
    in += blockIdx.y * a.in_bx;
    out += blockIdx.y * a.out_bx;
    if (a.nch == 2 && bid >= bpc) {
        bid -= bpc;
        in += a.in_ch;
        out += a.out_ch;
    }
    const long long lead = a.mix ? a.ngroups : 1;
    int gi = (int)(bid % lead);
    bid /= lead;
    const int tile = (int)(bid % ntile);
    bid /= ntile;
    const int z = (int)(bid % nz);
    if (!a.mix) gi = (int)(bid / nz);
    const YGroup G = a.g[gi];
    const int col = tile * C::TX + l;
    const bool valid = col < a.ncol;
    const int kx = valid ? col : 0;
    const double radius = ctl->radius;
    const double r0r = pp.radius0 / radius;  // R0/R of the wave-number scalings
    const double wx = wxt[kx];
    // derivative factors kx', ky' of output position p of this column (mhdrhs.f90:192-204).
    // FP64: the reference's expressions per mode (kprime_xy, R0/R formed once). FP32: kx' = cx + ax[p] and
    // ky' = cy + ay[p], the y-dependent parts tabulated in LDS once per block (the pass
    // rounds the factors to FP32 either way), so no factor is held in registers across
    // transforms and no FP64 quotient is formed per mode.
    T cx = T(0), cy = T(0);
    if constexpr (TAB) {
        const double rr = r0r;
#pragma unroll
        for (int i = 0; i < decltype(wyt)::PER; ++i) {
            const int t = (int)threadIdx.x + i * C::NT;
            if (t < N) {
                const double wy = wyt.r[i];
                sax[t] = pp.corot_k ? T(wy * pp.sin_c) : T(0);
                say[t] = pp.corot_k ? T(wy * pp.cos_c * rr) : T(wy * rr);
            }
        }
        cx = pp.corot_k ? T(wx * pp.cos_c) : T(wx);
        cy = pp.corot_k ? T(-wx * pp.sin_c * rr) : T(0);
    }
    auto kxy = [&](int p, T& kxv, T& kyv) {
        if constexpr (TAB) {
            kxv = cx + sax[p];
            kyv = cy + say[p];
        } else {
            double kxp, kyp;
            kprime_xy(wx, swy[p], pp, r0r, kxp, kyp);
            kxv = T(kxp);
            kyv = T(kyp);
        }
    };
    const bool stored = col < a.ncol_st;  // to the end of the last live piece of the row (kPiece)
    const int ylim = a.ylim && stored ? a.ylim[a.pieces ? col / kPiece<T> * kPiece<T> : kx] : N;
    cpx<T>* line = sh + l * C::LS;
    auto lds = [&](int p) { return line + p; };
    const cpx<T>* ib = in + (long long)z * N * a.rs + kx;
    cpx<T>* ob = out + (long long)z * a.cy * a.rs + col;

    auto fft_field = [&](int f, cpx<T>* v) {
        const cpx<T>* src = ib + f * a.in_fs;
        auto load = [&](int p) -> cpx<T> { return valid ? load_stream(src + p * a.rs) : cpx<T>{T(0), T(0)}; };
        __syncthreads();  // the LDS line may still be read by the previous transform
        return line_fft_regs<N, -1, T, typename C::P>(j, stw, load, lds, v);
    };
    auto store = [&](int f, int p, cpx<T> val) {
        const int s = pos_to_stored(p, N, a.cy);
        const int my = p <= N / 2 ? p : p - N;
        if (stored && s >= 0 && my <= ylim && -my <= ylim) store_stream(ob + f * a.out_fs + s * a.rs, val);
    };

    cpx<T> va[I::RMAX], vb[I::RMAX];
    // i k z + acc with one rounding, so that a divergence is the same bits in the one group of the large
    // form and in the groups of the split form (a box of an ensemble and the box on its own)
    auto add_i = [](T k, cpx<T> z, cpx<T> acc) {
        if constexpr (sizeof(T) == 8) return cpx<T>{fma(-k, z.y, acc.x), fma(k, z.x, acc.y)};
        else return cpx<T>{fmaf(-k, z.y, acc.x), fmaf(k, z.x, acc.y)};
    };
    if (G.kind == 3) {
        // symmetric momentum flux tensor M = (xx, xy, xz, yy, yz, zz) in in[0..5]:
        // out = -i(kx' Y M_xx + ky' Y M_xy), Y M_xz, -i(kx' Y M_xy + ky' Y M_yy), Y M_yz,
        //       -i(kx' Y M_xz + ky' Y M_yz), Y M_zz  (the x, y, z momentum divergence groups;
        // each off-diagonal component is transformed once and used by both rows)
        auto neg = [](cpx<T> z) { return cpx<T>{-z.x, -z.y}; };
        const bool h = fft_field(G.in[0], va);                                      // xx
        // the tables are visible after the transform's first barrier; FP64 keeps the
        // factors in registers (4 per work-item), FP32 reads them from the tables at each use
        constexpr int NKC = TAB ? 1 : I::RLAST;
        T kxc[NKC], kyc[NKC];
        if constexpr (!TAB) {
#pragma unroll
            for (int r = 0; r < I::RLAST; ++r) kxy(h ? j + r * I::BLAST : 0, kxc[r], kyc[r]);
        }
        auto kxr = [&](int r) -> T {
            if constexpr (TAB) return cx + sax[h ? j + r * I::BLAST : 0];
            else return kxc[r];
        };
        auto kyr = [&](int r) -> T {
            if constexpr (TAB) return cy + say[h ? j + r * I::BLAST : 0];
            else return kyc[r];
        };
#pragma unroll
        for (int r = 0; r < I::RLAST; ++r) va[r] = mul_i(kxr(r), va[r]);
        fft_field(G.in[1], vb);                                                     // xy
        if (h) {
#pragma unroll
            for (int r = 0; r < I::RLAST; ++r) {
                store(G.out[0], j + r * I::BLAST, neg(add_i(kyr(r), vb[r], va[r])));
                vb[r] = mul_i(kxr(r), vb[r]);                                       // y row, x part
            }
        }
        fft_field(G.in[3], va);                                                     // yy
        if (h) {
#pragma unroll
            for (int r = 0; r < I::RLAST; ++r) store(G.out[2], j + r * I::BLAST, neg(add_i(kyr(r), va[r], vb[r])));
        }
        fft_field(G.in[2], va);                                                     // xz
        if (h) {
#pragma unroll
            for (int r = 0; r < I::RLAST; ++r) {
                store(G.out[1], j + r * I::BLAST, va[r]);
                va[r] = mul_i(kxr(r), va[r]);                                       // z row, x part
            }
        }
        fft_field(G.in[4], vb);                                                     // yz
        if (h) {
#pragma unroll
            for (int r = 0; r < I::RLAST; ++r) {
                store(G.out[3], j + r * I::BLAST, vb[r]);
                store(G.out[4], j + r * I::BLAST, neg(add_i(kyr(r), vb[r], va[r])));
            }
        }
        fft_field(G.in[5], va);                                                     // zz
        if (h) {
#pragma unroll
            for (int r = 0; r < I::RLAST; ++r) store(G.out[5], j + r * I::BLAST, va[r]);
        }
        return;
    }
    if (G.kind == 2) {
        if (fft_field(G.in[0], va)) {
#pragma unroll
            for (int r = 0; r < I::RLAST; ++r) store(G.out[0], j + r * I::BLAST, va[r]);
        }
        return;
    }
    const bool has = fft_field(G.in[0], va);
    fft_field(G.in[1], vb);
    if (has) {
#pragma unroll
        for (int r = 0; r < I::RLAST; ++r) {
            T kx_, ky_;
            kxy(j + r * I::BLAST, kx_, ky_);
            const cpx<T> gsum = add_i(ky_, vb[r], mul_i(kx_, va[r]));
            vb[r] = cpx<T>{-gsum.x, -gsum.y};                                    // -(i kx' Ya + i ky' Yb)
        }
    }
    if (G.in[3] >= 0) {
        fft_field(G.in[3], va);                                                 // + Y(source)
#pragma unroll
        for (int r = 0; r < I::RLAST; ++r) vb[r] = vb[r] + va[r];
    }
    if (has) {
#pragma unroll
        for (int r = 0; r < I::RLAST; ++r) store(G.out[0], j + r * I::BLAST, vb[r]);
    }
    if (G.in[2] < 0) return;
    fft_field(G.in[2], va);
    if (has) {
#pragma unroll
        for (int r = 0; r < I::RLAST; ++r) store(G.out[1], j + r * I::BLAST, va[r]);  // Y(F_c)
    }
}

// ---------------------------------------------------------------- z pass + RK3
// One work-group per (equation, column tile, cy), two transforms (four with the shifted grid):
//   B_x  -i ky' Z(E_z) + i kz' Z(E_y)      momentum, energy (mass)  Z(D[f]) - i kz' Z(D[f + 1])
//   B_y   i kx' Z(E_z) - i kz' Z(E_x)
//   B_z   i ky' Z(E_x) - i kx' Z(E_y)
// The next transform's input tile is loaded into LDS while the current one is transformed (TileLoad),
// so only the first of the chain waits for memory: at 256^3 with phase shift 1056 -> 1021 us a launch
// in FP64 and 777 -> 740 in FP32, 512 x 512 x 128 FP32 520 -> 454 us (with loads at the head of each
// transform instead; neutral at 277-281 us with the 2/3 rule). With the block order below 256^3 phase
// shift FP64 takes 900 us: 3.2 GB at 3.5 TB/s, where a copy of this row pattern reaches 4.6-5: the rest
// is the first load, the update's loads and work-group turnover. The right-hand side of a mode stays in
// the registers of the work-item whose last butterfly made it, and the update follows there: adjacent
// work-items hold adjacent kx, so U and V are read and
// written in whole rows of the tile. Forming the three components of B in one work-group (three
// transforms instead of six) held 204 registers, one work-group per CU.
//
// sh: the lines of the tile between the stages, raw: the tile being loaded; two LDS arrays that the
// compiler is told do not overlap, so that it does not wait for the loads into raw at reads of sh.
template <typename T, int N, int OPT>
__device__ __forceinline__ void zfwd_body(cpx<T>* __restrict__ sh, cpx<T>* __restrict__ raw, cpx<T>* __restrict__ stw,
                                          double* __restrict__ swz, const cpx<T>* __restrict__ D,
                                          cpx<double>* __restrict__ U, cpx<double>* __restrict__ V, const ZArgs& a,
                                          const cpx<T>* __restrict__ tw, const BoxTables& tb,
                                          const double* __restrict__ wzf, const PhysParams& pp,
                                          const Ctl* __restrict__ ctl, int irk, int ntile, T scale) {
    using C = FwdCfg<T, N, true>;
    using I = typename C::I;
    constexpr int RL = I::RLAST;
    constexpr int TX = C::TX;
    using TL = TileLoad<N, TX * (int)sizeof(cpx<T>), C::NT>;
    // batched boxes: one per grid row
    ctl += blockIdx.y;
    D += blockIdx.y * a.d_bx;
    U += blockIdx.y * a.u_bx;
    V += blockIdx.y * a.v_bx;
    const cpx<T>* const Ds = a.Ds ? (const cpx<T>*)a.Ds + blockIdx.y * a.d_bx : nullptr;
    cpx<float>* const Uf = a.Uf ? a.Uf + blockIdx.y * a.uf_bx : nullptr;
    // Block -> (equation, slab sl of ntile * CY, padded to whole groups of 8). The three B equations of a
    // slab come first and side by side on one XCD (work-groups are dealt round-robin over the 8), so
    // that the reads of E they share hit its L2: block ((sl / 8) 3 + eq) 8 + sl % 8. The others follow,
    // with one chain an equation at a time (its tiles in memory order), with the two chains of phase
    // shift all equations of a slab together. At 256^3 with phase shift 909 us (FP64) and 565 (FP32),
    // against 1017-1036 and 582 an equation at a time and 940 and 587 with all equations of a slab on
    // one XCD; at 128x128x64 with the filter 57.8 us an equation at a time, 60.6 together, 61.4.
    const int neq = a.mass ? 8 : 7;
    const int nsp = (ntile * a.CY + 7) / 8 * 8;
    int eq, sl;  // eq: 0 B_z, 1 B_x, 2 B_y, 3-5 momentum, 6 energy, 7 mass
    if ((int)blockIdx.x < 3 * nsp) {
        const unsigned grp = blockIdx.x / 24;
        eq = (int)(blockIdx.x / 8 - grp * 3);
        sl = (int)(grp * 8 + (blockIdx.x & 7));
    } else {
        const int q = (int)blockIdx.x - 3 * nsp;
        eq = 3 + (Ds ? q % (neq - 3) : q / nsp);
        sl = Ds ? q / (neq - 3) : q % nsp;
    }
    if (sl >= ntile * a.CY) return;  // whole work-group, before any barrier
    const int tile = sl % ntile, cy = sl / ntile;
    const int l = threadIdx.x % TX, j = threadIdx.x / TX;
    const int col = tile * TX + l;
    const bool valid = col < a.KX;
    const int kx = valid ? col : 0;
    // Rows (kx, my) of the mask with no kept mode, by arithmetic (mask_row_dead): no table or control
    // word is waited for before the first tile's loads are issued.
    const int my = cy <= (a.CY == (int)a.mY ? a.CY / 2 : (a.CY - 1) / 2) ? cy : cy - a.CY;
    auto row_live = [&](int c) {
        return c < a.KX && (OPT != 1 || !mask_row_dead(pp.dealias, a.mX, a.mY, a.mZ, c, my));
    };
    // every wave holds all TX columns of the tile: a tile with no kept mode has nothing to
    // transform, read or write (unless the modes outside the kept set must be cleared)
    if (OPT == 1 && !a.clear_outside && __ballot(row_live(col)) == 0) return;
    // the 16 bytes of each row this work-item loads: one FP64 column or two FP32 columns of the tile
    // (columns past KX are row padding). A column with no kept mode (OPT 1) is not read, as the y pass
    // did not store it; what the tile then holds there reaches no mode that is updated.
    constexpr int CPL = 16 / (int)sizeof(cpx<T>);
    const int lc = tile * TX + TL::piece(threadIdx.x) * CPL;
    const bool on = row_live(lc) || (CPL == 2 && row_live(lc + 1));
    const long long zls = (long long)a.CY * a.rs;   // z line stride of D
    const long long mode0 = (long long)cy * a.rs + kx;
    // first and second field of the equation, with D's tile of a field
    const int v = eq == 0 ? 6 : (eq < 3 ? 3 + eq : (eq < 6 ? eq - 2 : (eq == 6 ? 7 : 0)));
    const int f1 = eq == 0 ? kDE : (eq < 3 ? kDE + 2 : (eq < 6 ? kDMom + 2 * (eq - 3) : (eq == 6 ? kDEnergy : kDMass)));
    const int f2 = eq == 1 ? kDE + 1 : (eq == 2 ? kDE : f1 + 1);
    auto fetch = [&](const cpx<T>* base, int f) {
        TL::run((const char*)(base + f * a.in_fs + (long long)cy * a.rs + tile * TX), zls * (long long)sizeof(cpx<T>),
                (char*)raw, on);
    };
    fetch(Ds ? Ds : D, f1);
    LdsTable<cpx<T>, N, C::NT> twt;
    LdsTable<double, N, C::NT> wzt;
    twt.fetch(tw);
    wzt.fetch(wzf);
    const int lim = tb.kzlim[(long long)cy * a.KX + kx];
    const double wx = tb.wx[kx], wy = tb.wy[cy];
    const double radius = ctl->radius, tau = ctl->tau;
    if (ctl->status != 0) {  // uniform over the box: the step was refused
        wait_loads();        // no load into LDS outlives the work-group
        return;
    }
    twt.put(stw);  // visible after the barrier that opens each transform
    wzt.put(swz);
    const double r0r = pp.radius0 / radius;  // R0/R of the wave-number scalings
    cpx<T>* line = sh + l * C::LS;
    auto lds = [&](int p) { return line + p; };
    cpx<T> w[I::RMAX];
    bool has = false;
    double kxd, kyd;
    kprime_xy(wx, wy, pp, r0r, kxd, kyd);
    const T kxp = T(kxd), kyp = T(kyd);
    // Z of the tile in raw, into w; `next` issues the loads of the tile after it
    auto transform = [&](auto next) {
        wait_loads();
        lds_barrier();
        if (j < I::B0) {
#pragma unroll
            for (int r = 0; r < C::P::R0; ++r) w[r] = raw[(j + r * I::B0) * TX + l];
        }
        has = line_fft_stages<N, -1, T, typename C::P>(j, stw, lds, w, next);
    };
    auto kz_at = [&](int r) -> T { return T(swz[has ? j + r * I::BLAST : 0] * r0r); };
    // phase-shift dealiasing: fnl = (Z(D) + conj(ph) Z(Ds)) / 2, ph of the output mode: the shifted
    // grid first, turned back in place, then the plain grid on top
    const cpx<double> wcb = Ds ? cmul(a.phc[kx], a.phb[cy]) : cpx<double>{1.0, 0.0};
    auto unshift = [&](cpx<T>(&acc)[RL]) {
#pragma unroll
        for (int r = 0; r < RL; ++r) {
            const cpx<double> q = cmul(a.ph[has ? j + r * I::BLAST : 0], wcb);
            acc[r] = cmul(acc[r], cpx<T>{T(q.x), T(-q.y)});
        }
    };
    const double sc = Ds ? 0.5 * double(scale) : double(scale);
    const double c = ctl->cc[irk], dn = irk < 2 ? ctl->dd[irk + 1] : 0.0, ts = ctl->ts[irk];
    const double cl = ctl->cc[2];
    const bool holds_u = rhs_holds_u(pp), rdU = irk == 1 && holds_u, wrU = store_u(sizeof(T) == 8, irk, pp);

    // the modes of this work-item: stored z row of output r, -1 outside the kept set
    auto row_of = [&](int r) -> int {
        const int p = j + r * I::BLAST;
        int cz = pos_to_stored(p, N, a.CZ);
        if constexpr (OPT == 1) {
            const int mz = p <= N / 2 ? p : p - N;
            if (mz > lim || -mz > lim) cz = -1;
        }
        return valid && j < I::BLAST ? cz : -1;
    };
    // RK3 update of variable v at this work-item's modes from its unscaled right-hand side. What it
    // starts from (U, or V after the first substage) is loaded four modes at a time: issued before the
    // last transform's LDS stages it took the registers to 150 and more (256^3 932 -> 1366 us).
    auto update = [&](const cpx<T>(&acc)[RL]) {
        const cpx<double>* src = (irk != 0 ? V : U) + v * a.ufs + mode0;
        cpx<double> base[RL];
#pragma unroll
        for (int r = 0; r < RL; ++r) {
            if (r % 4 == 0) {
#pragma unroll
                for (int q = r; q < (r + 4 < RL ? r + 4 : RL); ++q) {
                    const int cz = row_of(q);
                    base[q] = cz >= 0 ? load_stream(src + cz * zls) : cpx<double>{0.0, 0.0};
                }
            }
            const int p = j + r * I::BLAST;
            const int cz = row_of(r);
            if (cz < 0) {
                // outside the kept set the new state is zero whatever U holds there: it is not read,
                // and V there is never read
                if (OPT == 1 && a.clear_outside) {
                    const int q = pos_to_stored(p, N, a.CZ);
                    if (q >= 0) {
                        U[v * a.ufs + q * zls + mode0] = cpx<double>{0.0, 0.0};
                        if (Uf) Uf[v * a.ufs + q * zls + mode0] = cpx<float>{0.0f, 0.0f};
                    }
                }
                continue;
            }
            const long long mi = cz * zls + mode0;
            const double wz = swz[p];
            cpx<double> fnl{double(acc[r].x) * sc, double(acc[r].y) * sc};
            if (a.clos && v >= 1) fnl = fnl + a.clos[(v - 1) * a.ufs + mi];
            const double k2 = (pp.visc || pp.resis) ? ksquare(wx, wy, wz, pp, ctl, r0r) : 0.0;
            // f + L u
            auto add_linear = [&](cpx<double> f, cpx<double> u) {
                if (pp.aeb && v < 7) {
                    const double fac = (v == 2 || v == 3) ? 3.0 : (v >= 5 ? 1.0 : 2.0);
                    f = f - cpx<double>{(u.x * fac) / tau, (u.y * fac) / tau};
                }
                if (pp.visc && pp.visc_exp && v >= 1 && v <= 3)
                    f = f - cpx<double>{u.x * pp.nu * k2, u.y * pp.nu * k2};
                if (pp.resis && pp.resis_exp && v >= 4 && v <= 6 && !(pp.conserve_bg && kx == 0 && p == 0))
                    f = f - cpx<double>{u.x * pp.eta * k2, u.y * pp.eta * k2};
                return f;
            };
            if (holds_u && irk != 2) fnl = add_linear(fnl, rdU ? load_stream(U + v * a.ufs + mi) : base[r]);
            cpx<double> un{c * fnl.x + base[r].x, c * fnl.y + base[r].y};
            if (pp.visc && !pp.visc_exp && v >= 1 && v <= 3) {
                const double den = ts * k2 * pp.nu + 1.0;
                const double inv = 1.0 / den;
                un = {un.x * inv, un.y * inv};
            }
            if (pp.resis && !pp.resis_exp && v >= 4 && v <= 6) {
                const double den = ts * k2 * pp.eta + 1.0;
                const double inv = 1.0 / den;
                un = {un.x * inv, un.y * inv};
            }
            if constexpr (OPT == 2) {
                const double fx = tb.fx[kx], fy = tb.fy[cy], fz = tb.fz[cz];
                un = {((un.x * fx) * fy) * fz, ((un.y * fx) * fy) * fz};
            }
            if (wrU) store_stream(U + v * a.ufs + mi, un);
            if (Uf) store_stream(Uf + v * a.ufs + mi, cpx<float>{float(un.x), float(un.y)});
            // the next step's first substage weighs this RHS by dd(0) = 0 (rktmod.f90:40-42)
            if (irk != 2) {
                cpx<double> vn{un.x + dn * fnl.x, un.y + dn * fnl.y};
                if (rdU) {
                    const cpx<double> q = add_linear(cpx<double>{0.0, 0.0}, un);
                    vn = {vn.x + cl * q.x, vn.y + cl * q.y};
                }
                store_stream(V + v * a.ufs + mi, vn);
            }
        }
    };

    const T k1 = eq == 0 ? kyp : (eq == 1 ? -kyp : kxp);
    const T sz = eq == 1 ? T(1) : T(-1);
    cpx<T> acc[RL];
#pragma unroll
    for (int r = 0; r < RL; ++r) acc[r] = cpx<T>{T(0), T(0)};
#pragma unroll 1
    for (int ch = Ds ? 1 : 0; ch >= 0; --ch) {
        transform([&]() { fetch(ch ? Ds : D, f2); });
#pragma unroll
        for (int r = 0; r < RL; ++r) acc[r] = acc[r] + (eq < 3 ? mul_i(k1, w[r]) : w[r]);
        transform([&]() {
            if (ch) fetch(D, f1);
        });
#pragma unroll
        for (int r = 0; r < RL; ++r) acc[r] = acc[r] + mul_i(eq == 0 ? -kxp : sz * kz_at(r), w[r]);
        if (ch) unshift(acc);
    }
    if (valid && has) update(acc);
}

template <typename T, int N, int OPT>
__global__ __launch_bounds__((FwdCfg<T, N, true>::NT), (FwdCfg<T, N, true>::MINW)) void k_zfwd_rhs(const cpx<T>* __restrict__ D,
                                                               cpx<double>* __restrict__ U,
                                                               cpx<double>* __restrict__ V, ZArgs a,
                                                               const cpx<T>* __restrict__ tw, BoxTables tb,
                                                               const double* __restrict__ wzf, PhysParams pp,
                                                               const Ctl* __restrict__ ctl, int irk, int ntile,
                                                               T scale) {
    using C = FwdCfg<T, N, true>;
    __shared__ cpx<T> sh[C::TX * C::LS];
    __shared__ __align__(16) cpx<T> raw[N * C::TX];
    __shared__ cpx<T> stw[N];
    __shared__ double swz[N];
    zfwd_body<T, N, OPT>(sh, raw, stw, swz, D, U, V, a, tw, tb, wzf, pp, ctl, irk, ntile, scale);
}

// ---------------------------------------------------------------- launchers

template <typename T, int N, bool ALT>
static hipError_t do_yg_c(const cpx<T>* in, cpx<T>* out, const YGArgs& a, const cpx<T>* tw, const double* wxt,
                          const double* wyf, const PhysParams& pp, const Ctl* ctl, int nz, hipStream_t s) {
    using C = FwdCfg<T, N, false, ALT>;
    const int ntile = (a.ncol + C::TX - 1) / C::TX;
    YGArgs b = a;
    if (b.mass.nblk) {
        // one mode a work-item (one memory latency) in small boxes, four where that still fills the chip
        const long long n = (long long)b.mass.KXP * b.mass.CY * b.mass.CZ;
        const long long per = n > 4096LL * C::NT ? 4LL * C::NT : C::NT;
        b.mass.nblk = (int)((n + per - 1) / per);
    }
    const long long nblk = (long long)ntile * nz * b.ngroups * b.nch + b.mass.nblk;
    hipLaunchKernelGGL((k_yfwd_group<T, N, ALT>), dim3((unsigned)nblk, b.nbox > 1 ? b.nbox : 1), dim3(C::NT), 0, s, in,
                       out, b, tw, wxt, wyf, pp, ctl, ntile, nz);
    return hipGetLastError();
}

template <typename T, int N>
static hipError_t do_yg(const cpx<T>* in, cpx<T>* out, const YGArgs& a, const cpx<T>* tw, const double* wxt,
                        const double* wyf, const PhysParams& pp, const Ctl* ctl, int nz, hipStream_t s) {
    if constexpr (N == 256) {
        // the wide plan: FP32 launches of one chain, FP64 launches of two
        if ((a.nch == 2) == (sizeof(T) == 8)) return do_yg_c<T, N, true>(in, out, a, tw, wxt, wyf, pp, ctl, nz, s);
    }
    return do_yg_c<T, N, false>(in, out, a, tw, wxt, wyf, pp, ctl, nz, s);
}

template <typename T>
hipError_t launch_yfwd_group(int ny, const cpx<T>* in, cpx<T>* out, const YGArgs& a, const cpx<T>* tw,
                             const double* wxt, const double* wyf, const PhysParams& pp, const Ctl* ctl, int nz,
                             hipStream_t s) {
    switch (ny) {
        case 16: return do_yg<T, 16>(in, out, a, tw, wxt, wyf, pp, ctl, nz, s);
        case 32: return do_yg<T, 32>(in, out, a, tw, wxt, wyf, pp, ctl, nz, s);
        case 64: return do_yg<T, 64>(in, out, a, tw, wxt, wyf, pp, ctl, nz, s);
        case 128: return do_yg<T, 128>(in, out, a, tw, wxt, wyf, pp, ctl, nz, s);
        case 256: return do_yg<T, 256>(in, out, a, tw, wxt, wyf, pp, ctl, nz, s);
        case 512: return do_yg<T, 512>(in, out, a, tw, wxt, wyf, pp, ctl, nz, s);
        case 96: return do_yg<T, 96>(in, out, a, tw, wxt, wyf, pp, ctl, nz, s);
        default: return hipErrorInvalidValue;
    }
}

template <typename T, int N, int OPT>
static hipError_t do_zr(const cpx<T>* D, cpx<double>* U, cpx<double>* V, const ZArgs& a, const cpx<T>* tw,
                        const BoxTables& tb, const double* wzf, const PhysParams& pp, const Ctl* ctl, int irk,
                        T scale, hipStream_t s) {
    using C = FwdCfg<T, N, true>;
    const int ntile = (a.KX + C::TX - 1) / C::TX;
    const long long nblk = (a.mass ? 8LL : 7LL) * (((long long)ntile * a.CY + 7) / 8 * 8);
    hipLaunchKernelGGL((k_zfwd_rhs<T, N, OPT>), dim3((unsigned)nblk, a.nbox > 1 ? a.nbox : 1), dim3(C::NT), 0, s, D, U,
                       V, a, tw, tb, wzf, pp, ctl, irk, ntile, scale);
    return hipGetLastError();
}

template <typename T, int N>
static hipError_t do_zr_opt(const cpx<T>* D, cpx<double>* U, cpx<double>* V, const ZArgs& a, const cpx<T>* tw,
                            const BoxTables& tb, const double* wzf, const PhysParams& pp, const Ctl* ctl, int irk,
                            T scale, hipStream_t s) {
    if (pp.dealias == 1 || pp.dealias == 3) return do_zr<T, N, 1>(D, U, V, a, tw, tb, wzf, pp, ctl, irk, scale, s);
    if (pp.dealias == 2) return do_zr<T, N, 2>(D, U, V, a, tw, tb, wzf, pp, ctl, irk, scale, s);
    return do_zr<T, N, 0>(D, U, V, a, tw, tb, wzf, pp, ctl, irk, scale, s);
}

template <typename T>
hipError_t launch_zfwd_rhs(int nz, const cpx<T>* D, cpx<double>* U, cpx<double>* V, const ZArgs& a,
                           const cpx<T>* tw, const BoxTables& tb, const double* wzf, const PhysParams& pp,
                           const Ctl* ctl, int irk, T scale, hipStream_t s) {
    switch (nz) {
        case 16: return do_zr_opt<T, 16>(D, U, V, a, tw, tb, wzf, pp, ctl, irk, scale, s);
        case 32: return do_zr_opt<T, 32>(D, U, V, a, tw, tb, wzf, pp, ctl, irk, scale, s);
        case 64: return do_zr_opt<T, 64>(D, U, V, a, tw, tb, wzf, pp, ctl, irk, scale, s);
        case 128: return do_zr_opt<T, 128>(D, U, V, a, tw, tb, wzf, pp, ctl, irk, scale, s);
        case 256: return do_zr_opt<T, 256>(D, U, V, a, tw, tb, wzf, pp, ctl, irk, scale, s);
        case 512: return do_zr_opt<T, 512>(D, U, V, a, tw, tb, wzf, pp, ctl, irk, scale, s);
        case 96: return do_zr_opt<T, 96>(D, U, V, a, tw, tb, wzf, pp, ctl, irk, scale, s);
        default: return hipErrorInvalidValue;
    }
}

template hipError_t launch_yfwd_group<double>(int, const cpx<double>*, cpx<double>*, const YGArgs&,
                                              const cpx<double>*, const double*, const double*, const PhysParams&,
                                              const Ctl*, int, hipStream_t);
template hipError_t launch_yfwd_group<float>(int, const cpx<float>*, cpx<float>*, const YGArgs&, const cpx<float>*,
                                             const double*, const double*, const PhysParams&, const Ctl*, int,
                                             hipStream_t);
template hipError_t launch_zfwd_rhs<double>(int, const cpx<double>*, cpx<double>*, cpx<double>*, const ZArgs&,
                                            const cpx<double>*, const BoxTables&, const double*, const PhysParams&,
                                            const Ctl*, int, double, hipStream_t);
template hipError_t launch_zfwd_rhs<float>(int, const cpx<float>*, cpx<double>*, cpx<double>*, const ZArgs&,
                                           const cpx<float>*, const BoxTables&, const double*, const PhysParams&,
                                           const Ctl*, int, float, hipStream_t);

}  // namespace laps
