// laps_api.hip -- the C ABI of include/laps.h and the orchestration of one
// RK3 step on the device.
//
// Device data layout (one box):
//   U      [11][CZ][CY][KX] FP64 complex : spectral state uu_fourier (8) +
//                                         Hall current J_hat (3), kept box
//   Ufull  [11][nz][ny][nx/2+1] FP64     : un-dealiased spectrum of the state
//                                         handed over by laps_set_state
//   V      [8][CZ][CY][KX] FP64 complex  : within a step, the state plus the next
//                                         substage's share of the last RHS
//                                         (U + d fnl; RK3's fnl_rk folded in)
//   S      [12][nz][ny][nx] FP64 real    : real-space state uu(8)+uu_prim(4)
//                                         (the uploaded one, or materialised)
//   P1,P2  T complex                     : transform intermediates, T = FP64
//                                         or FP32 (mixed precision)
// The "kept box" holds kx < KX and the stored ky/kz rows of the modes that
// survive dealiasing: all modes for the compact filter (option 2), the
// bounding box of the 2/3 sphere for option 1. Modes outside the box are
// identically zero after every substage (dealiasing.f90:87-99), so the
// transforms read and write only the box.
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <mutex>
#include <string>
#include <vector>

#include "../../include/laps.h"
#include "host_copy.hpp"
#include "internal.hpp"

using namespace laps;

static_assert(sizeof(laps_params) == 168, "laps_params layout is part of the ABI");
static_assert(LAPS_MLP_NPARAM == laps::kClNParam && LAPS_CLOSURE_NPARAM == laps::kClNParam + laps::kClNNorm,
              "closure parameter layout");

namespace {

thread_local std::string g_err;

int fail(int code, const std::string& msg) {
    g_err = msg;
    return code;
}

#define LAPS_CK(...)                                                                               \
    do {                                                                                           \
        hipError_t e_ = (__VA_ARGS__);                                                             \
        if (e_ != hipSuccess)                                                                      \
            return fail(LAPS_EDEVICE, std::string(#__VA_ARGS__) + ": " + hipGetErrorString(e_));   \
    } while (0)

constexpr double kPiRef = 3.141592653589793;  // mhdinit.f90:7
constexpr long double kPiL = 3.141592653589793238462643383279502884L;

// exp(-2 pi i t / n), angle reduced to one octant in long double
void root(long t, long n, double& c, double& s) {
    t %= n;
    const long q8 = 8 * t, oct = q8 / n, rem = q8 - oct * n;
    const long double a = (oct % 2 == 0) ? kPiL / 4.0L * (long double)rem / (long double)n
                                         : kPiL / 4.0L * (long double)(n - rem) / (long double)n;
    const long double ca = cosl(a), sa = sinl(a);
    long double cr, sr;
    switch (oct) {
        case 0: cr = ca; sr = sa; break;
        case 1: cr = sa; sr = ca; break;
        case 2: cr = -sa; sr = ca; break;
        case 3: cr = -ca; sr = sa; break;
        case 4: cr = -ca; sr = -sa; break;
        case 5: cr = -sa; sr = -ca; break;
        case 6: cr = sa; sr = -ca; break;
        default: cr = ca; sr = -sa; break;
    }
    c = (double)cr;
    s = -(double)sr;
}

// wave_number_* (mhdinit.f90:83-111): 2*pi*m/L, m signed, Nyquist carries +n/2
double wave_number(int i, int n, double L) {
    const int m = (i <= n / 2) ? i : i - n;
    return 2 * kPiRef * (double)m / L;
}

int signed_index(int i, int n) { return (i <= n / 2) ? i : i - n; }

// dealiasing.f90:100-111
double compact_filter(double w, double L, int n, double af) {
    const double aj = (5.0 + 6.0 * af) / 8.0;
    const double bj = (1.0 + 2.0 * af) / 2.0;
    const double cj = -(1.0 - 2 * af) / 8.0;
    const double wl = w * L / n;
    return (aj + bj * cos(wl) + cj * cos(2 * wl)) / (1 + 2 * af * cos(wl));
}

bool supported_len(int n) { return n == 16 || n == 32 || n == 64 || n == 96 || n == 128 || n == 256 || n == 512; }

struct DevTables {
    double *wx = nullptr, *wy = nullptr, *wz = nullptr, *fx = nullptr, *fy = nullptr, *fz = nullptr;
    int *kzlim = nullptr, *mz = nullptr, *ylim = nullptr;
    BoxTables view() const { return BoxTables{wx, wy, wz, kzlim, ylim, fx, fy, fz, mz}; }
};

}  // namespace

// Kernel classes of the step pipeline, timed with HIP events on the
// context's stream when laps_timing_enable() is on.
enum KClass { K_ZINV, K_YINV, K_XFUSED, K_YFWD, K_ZFWD, K_CURL, K_CTL, K_XC2R, K_XR2C, K_NCLASS };
static const char* const kClassNames[K_NCLASS] = {
    "fft_z_inverse", "fft_y_inverse", "x_c2r_flux_r2c", "fft_y_fwd_divcurl", "fft_z_fwd_rhs_rk3",
    "hall_curl", "control", "fft_x_c2r", "fft_x_r2c"};

struct Timing {
    bool on = false;
    std::vector<hipEvent_t> pool;
    std::vector<std::pair<int, std::pair<hipEvent_t, hipEvent_t>>> pending;
    double ms[K_NCLASS] = {0};
    double bytes[K_NCLASS] = {0};
    long long launches[K_NCLASS] = {0};
};

struct laps_ctx {
    Timing timing;
    laps_params p{};
    int nx = 0, ny = 0, nz = 0, nxh = 0;
    long long N = 0, M = 0;
    bool mixed = false;
    hipStream_t stream = nullptr;
    Box full{}, kept{};
    DevTables tfull, tkept;
    PhysParams pp{};
    Ctl* ctl = nullptr;
    cpx<double>* twd[3] = {nullptr, nullptr, nullptr};
    cpx<float>* twf[3] = {nullptr, nullptr, nullptr};
    cpx<double>* U = nullptr;
    cpx<double>* Ufull = nullptr;
    cpx<double>* V = nullptr;
    double* S = nullptr;
    void* P1 = nullptr;
    void* P2 = nullptr;
    void* P3 = nullptr;                                   // shifted-grid y-pass output (option 3), in P2
    long long p1 = 0, p2 = 0;                             // complex elements per chain of P1, P2
    // learned closure: parameters + normalisation (FP32), features, outputs, the 12 real
    // correction fields, their spectra, and the RHS term on the full and the kept box
    // mixed precision: FP32 copy of U (8 state fields written by the z pass, 3 Hall-current
    // fields by the curl), the z-inverse input; U stays the FP64 state
    cpx<float>* Uf = nullptr;
    bool closure = false;
    float *cl_P = nullptr, *cl_X = nullptr, *cl_Y = nullptr, *cl_id = nullptr;
    double* cl_C = nullptr;
    cpx<double>*cl_A = nullptr, *cl_B = nullptr, *cl_full = nullptr, *cl_rhs = nullptr;  // A, B: FP64 scratch
    cpx<double>*phx = nullptr, *phy = nullptr, *phz = nullptr;  // e^{i pi m/n} per axis (option 3)
    cpx<double>* phyk = nullptr;                                 // phy of the kept box's stored ky
    cpx<double>* X1 = nullptr;
    cpx<double>* X2 = nullptr;
    double* Xr = nullptr;
    double* red = nullptr;
    double* dave = nullptr;
    unsigned long long* dbits = nullptr;
    std::vector<void*> allocs;
    bool have_state = false, fresh = false, materialized = false, stepped_since_set = false;
    uint64_t gen = 0;  // bumped when the kernels a step launches change (state upload, fixed dt)
    bool tuned = false;
    int plan_zinv = 0, plan_yinv = 0;  // FFT variants (plan, tile width) of the inverse z / y passes, by autotune()
    YGArgs yg{}, yg_split{};  // y forward groups of large and of small launches
    ZArgs zr{};
    double yfwd_bytes = 0, zfwd_bytes = 0;  // algorithmic elements x 2 (multiply by sizeof(T))
    // modes the dealiasing keeps, and (kx, cy) rows of the kept box holding at least one
    // (with no mask: every mode and row of the box, padding columns excluded)
    long long nkept = 0, nlive = 0;
    double fixed_dt = 0.0;
    int nblk_red = 1024;
    // batched launches of an ensemble group, set on the group's first box while one step of the
    // group is captured: n boxes whose U, Uf, V, P1, P2 sit at these element strides (in each
    // buffer's own element type) from this box's, and whose control blocks follow this box's
    struct Batch {
        int n = 1;
        long long u = 0, uf = 0, v = 0, p1 = 0, p2 = 0;
    } batch;
    // output staging (laps_stage_output): the outNNN.dat payload (nx,ny,nz,8) copied from the
    // real-space state S into pinned host memory on a stream of its own, while later steps run
    double* stage_host = nullptr;       // hipHostMalloc'd, 8 N doubles
    hipStream_t stage_stream = nullptr;
    hipEvent_t stage_ready = nullptr, stage_done = nullptr;
    bool stage_pending = false;          // a copy was queued: S is read until stage_done
    double stage_time = 0.0, stage_dt = 0.0;
    long long stage_istep = 0;

    HostCopy host;                       // copies of whole arrays to and from the caller's memory
    hipError_t to_host(void* dst, const void* src, size_t n) { return host.to_host(dst, src, n, p.device, stream); }
    hipError_t to_device(void* dst, const void* src, size_t n) {
        return host.to_device(dst, src, n, p.device, stream);
    }

    int alloc(void** ptr, size_t bytes) {
        if (bytes == 0) bytes = 16;
        hipError_t e = hipMalloc(ptr, bytes);
        if (e != hipSuccess) {
            *ptr = nullptr;
            return fail(LAPS_ENOMEM, "hipMalloc of " + std::to_string(bytes) + " bytes failed: " + hipGetErrorString(e));
        }
        allocs.push_back(*ptr);
        return LAPS_OK;
    }
    template <typename P>
    int allocn(P** ptr, size_t count) {
        return alloc((void**)ptr, count * sizeof(P));
    }
    long long kb() const { return kept.modes(); }
    int nf_in() const { return p.if_hall ? 11 : 8; }
    bool mass_flux() const { return p.dealias_option == 0; }  // the mass flux is transformed (MassArgs)
    // fluxes the x pass transforms: 6 (symmetric tensor) + 3 + 3, + 1 expanding-box source, + 3 mass
    int nf_out() const { return 12 + (p.if_aeb ? 1 : 0) + (mass_flux() ? 3 : 0); }
    int nx_slots() const { return mass_flux() ? 16 : nf_out(); }  // slots of P1 they occupy
    int nd() const { return mass_flux() ? 13 : 11; }              // y forward outputs
};

namespace {

// ------------------------------------------------------------------ setup helpers

int upload_tables(laps_ctx* c, const Box& b, bool pruned, const std::vector<int>& kzlim, DevTables& t) {
    std::vector<double> wx(b.KX), fx(b.KX), wy(b.CY), fy(b.CY), wz(b.CZ), fz(b.CZ);
    std::vector<int> mz(b.CZ);
    auto fft_index = [](int s, int cnt, int n) { return (cnt == n || s <= (cnt - 1) / 2) ? s : n - (cnt - s); };
    for (int i = 0; i < b.KX; ++i) {
        wx[i] = wave_number(i, c->nx, c->p.Lx);
        fx[i] = compact_filter(wx[i], c->p.Lx, c->nx, c->p.afx);
    }
    for (int s = 0; s < b.CY; ++s) {
        const int iy = fft_index(s, b.CY, c->ny);
        wy[s] = wave_number(iy, c->ny, c->p.Ly);
        fy[s] = compact_filter(wy[s], c->p.Ly, c->ny, c->p.afy);
    }
    for (int s = 0; s < b.CZ; ++s) {
        const int iz = fft_index(s, b.CZ, c->nz);
        wz[s] = wave_number(iz, c->nz, c->p.Lz);
        fz[s] = compact_filter(wz[s], c->p.Lz, c->nz, c->p.afz);
        mz[s] = signed_index(iz, c->nz);
    }
    std::vector<int> lim = kzlim;
    if (!pruned) lim.assign((size_t)b.KX * b.CY, c->nz);
    // per kx, the largest |my| of a row holding a kept mode (-1: none)
    std::vector<int> ylim(b.KX, -1);
    for (int s = 0; s < b.CY; ++s) {
        const int my = std::abs(signed_index(fft_index(s, b.CY, c->ny), c->ny));
        for (int i = 0; i < b.KX; ++i)
            if (lim[(size_t)s * b.KX + i] >= 0) ylim[i] = std::max(ylim[i], my);
    }
    int rc;
    if ((rc = c->allocn(&t.wx, b.KX)) || (rc = c->allocn(&t.fx, b.KX)) || (rc = c->allocn(&t.wy, b.CY)) ||
        (rc = c->allocn(&t.fy, b.CY)) || (rc = c->allocn(&t.wz, b.CZ)) || (rc = c->allocn(&t.fz, b.CZ)) ||
        (rc = c->allocn(&t.mz, b.CZ)) || (rc = c->allocn(&t.kzlim, lim.size())) || (rc = c->allocn(&t.ylim, b.KX)))
        return rc;
    LAPS_CK(hipMemcpy(t.wx, wx.data(), wx.size() * 8, hipMemcpyHostToDevice));
    LAPS_CK(hipMemcpy(t.fx, fx.data(), fx.size() * 8, hipMemcpyHostToDevice));
    LAPS_CK(hipMemcpy(t.wy, wy.data(), wy.size() * 8, hipMemcpyHostToDevice));
    LAPS_CK(hipMemcpy(t.fy, fy.data(), fy.size() * 8, hipMemcpyHostToDevice));
    LAPS_CK(hipMemcpy(t.wz, wz.data(), wz.size() * 8, hipMemcpyHostToDevice));
    LAPS_CK(hipMemcpy(t.fz, fz.data(), fz.size() * 8, hipMemcpyHostToDevice));
    LAPS_CK(hipMemcpy(t.mz, mz.data(), mz.size() * 4, hipMemcpyHostToDevice));
    LAPS_CK(hipMemcpy(t.kzlim, lim.data(), lim.size() * 4, hipMemcpyHostToDevice));
    LAPS_CK(hipMemcpy(t.ylim, ylim.data(), ylim.size() * 4, hipMemcpyHostToDevice));
    return LAPS_OK;
}

// Bounding box of the modes kept by the 2/3 rule (dealiasing.f90:87-99),
// evaluated with the reference's expression, or by phase-shift dealiasing
// (option 3, no reference counterpart: the open ellipsoid
// (mx/nx)^2 + (my/ny)^2 + (mz/nz)^2 < 2/9, tested exactly in integers), plus
// the per-column |mz| limit.
int compute_kept_box(laps_ctx* c, std::vector<int>& kzlim) {
    const int nx = c->nx, ny = c->ny, nz = c->nz, nxh = c->nxh;
    const bool shift = c->p.dealias_option == 3;
    if (c->p.dealias_option != 1 && !shift) {
        c->kept = c->full;
        c->kept.KXP = (c->full.KX + 15) / 16 * 16;
        c->nlive = (long long)c->kept.KX * c->kept.CY;
        c->nkept = c->nlive * c->kept.CZ;
        return LAPS_OK;
    }
    std::vector<double> ax(nxh), ay(ny), az(nz);
    for (int i = 0; i < nxh; ++i) { const double w = wave_number(i, nx, c->p.Lx); ax[i] = w * c->p.Lx / (2 * kPiRef * nx); }
    for (int i = 0; i < ny; ++i) { const double w = wave_number(i, ny, c->p.Ly); ay[i] = w * c->p.Ly / (2 * kPiRef * ny); }
    for (int i = 0; i < nz; ++i) { const double w = wave_number(i, nz, c->p.Lz); az[i] = w * c->p.Lz / (2 * kPiRef * nz); }
    auto keep = [&](int ix, int iy, int iz) {
        if (shift) {
            const long long X = nx, Y = ny, Z = nz, mx = ix, my = signed_index(iy, ny), mz = signed_index(iz, nz);
            return 9 * (mx * mx * Y * Y * Z * Z + my * my * X * X * Z * Z + mz * mz * X * X * Y * Y) <
                   2 * X * X * Y * Y * Z * Z;
        }
        const double r = sqrt(ax[ix] * ax[ix] + ay[iy] * ay[iy] + az[iz] * az[iz]);
        return !(r > 1. / 3.);
    };
    int kxmax = -1, kymax = 0, kzmax = 0;
    std::vector<int> col((size_t)nxh * ny, -1);
    for (int iy = 0; iy < ny; ++iy)
        for (int ix = 0; ix < nxh; ++ix) {
            int lim = -1;
            for (int iz = 0; iz < nz; ++iz)
                if (keep(ix, iy, iz)) lim = std::max(lim, std::abs(signed_index(iz, nz)));
            // the kept set of a column must be |mz| <= lim exactly
            for (int iz = 0; iz < nz; ++iz) {
                const bool inside = std::abs(signed_index(iz, nz)) <= lim;
                if (inside != keep(ix, iy, iz)) return fail(LAPS_EINVAL, "dealias mask is not a z-interval");
            }
            col[(size_t)iy * nxh + ix] = lim;
            if (lim >= 0) {
                kxmax = std::max(kxmax, ix);
                kymax = std::max(kymax, std::abs(signed_index(iy, ny)));
                kzmax = std::max(kzmax, lim);
            }
        }
    if (kxmax < 0) return fail(LAPS_EINVAL, "dealias mask keeps no mode");
    Box b;
    b.KX = kxmax + 1;
    b.KXP = (b.KX + 15) / 16 * 16;
    b.CY = std::min(2 * kymax + 1, ny);
    b.CZ = std::min(2 * kzmax + 1, nz);
    if (b.CY == ny - 1) b.CY = ny;  // keep compact rows symmetric or full
    if (b.CZ == nz - 1) b.CZ = nz;
    c->kept = b;
    kzlim.assign((size_t)b.KX * b.CY, -1);
    for (int cy = 0; cy < b.CY; ++cy) {
        const int iy = (b.CY == ny || cy <= (b.CY - 1) / 2) ? cy : ny - (b.CY - cy);
        for (int kx = 0; kx < b.KX; ++kx) kzlim[(size_t)cy * b.KX + kx] = col[(size_t)iy * nxh + kx];
    }
    // the inverse passes drop a row by an integer test of its mz = 0 mode
    // (mask_row_dead); it must never drop a row that holds a kept mode
    for (int cy = 0; cy < b.CY; ++cy) {
        const int iy = (b.CY == ny || cy <= (b.CY - 1) / 2) ? cy : ny - (b.CY - cy);
        for (int kx = 0; kx < b.KX; ++kx)
            if (kzlim[(size_t)cy * b.KX + kx] >= 0 &&
                mask_row_dead(c->p.dealias_option, nx, ny, nz, kx, signed_index(iy, ny)))
                return fail(LAPS_EINVAL, "internal: the row test of the inverse passes drops a kept mode");
    }
    c->nkept = c->nlive = 0;
    for (int lim : kzlim) {
        if (lim < 0) continue;
        ++c->nlive;
        c->nkept += std::min(2 * lim + 1, b.CZ);
    }
    return LAPS_OK;
}

// ------------------------------------------------------------------ kernel timing

hipEvent_t take_event(laps_ctx* c) {
    if (!c->timing.pool.empty()) {
        hipEvent_t e = c->timing.pool.back();
        c->timing.pool.pop_back();
        return e;
    }
    hipEvent_t e = nullptr;
    if (hipEventCreate(&e) != hipSuccess) return nullptr;
    return e;
}

// Runs `launch` (returning hipError_t); with timing on, brackets it with
// events on the context stream and books `bytes` of algorithmic traffic.
template <class F>
hipError_t timed(laps_ctx* c, int cls, double bytes, F launch) {
    if (!c->timing.on) return launch();
    hipEvent_t a = take_event(c), b = take_event(c);
    if (a) (void)hipEventRecord(a, c->stream);
    hipError_t e = launch();
    if (b) (void)hipEventRecord(b, c->stream);
    if (a && b) c->timing.pending.push_back({cls, {a, b}});
    c->timing.bytes[cls] += bytes;
    c->timing.launches[cls] += 1;
    return e;
}

// timing off while in scope (utility transforms, autotuning)
struct TimingOff {
    laps_ctx* c;
    bool was;
    explicit TimingOff(laps_ctx* cc) : c(cc), was(cc->timing.on) { c->timing.on = false; }
    ~TimingOff() { c->timing.on = was; }
};

int collect_timing(laps_ctx* c) {
    LAPS_CK(hipStreamSynchronize(c->stream));
    for (auto& pe : c->timing.pending) {
        float ms = 0.f;
        if (hipEventElapsedTime(&ms, pe.second.first, pe.second.second) == hipSuccess) c->timing.ms[pe.first] += ms;
        c->timing.pool.push_back(pe.second.first);
        c->timing.pool.push_back(pe.second.second);
    }
    c->timing.pending.clear();
    return LAPS_OK;
}

// ------------------------------------------------------------------ pipelines

template <typename T>
const cpx<T>* tw_of(laps_ctx* c, int axis);
template <>
const cpx<double>* tw_of<double>(laps_ctx* c, int axis) { return c->twd[axis]; }
template <>
const cpx<float>* tw_of<float>(laps_ctx* c, int axis) { return c->twf[axis]; }

// Columns that a pass over the rows of b stores: up to the end of the last piece (kPiece) where the rows
// are aligned, as the kept box's are. Launches that fit the memory-side cache pay for the added bytes
// and gain nothing (128x128x64 FP64, 65 -> 68 columns: x pass 45.9 -> 48.6 us, y inverse 34.2 -> 35.0), so
// the y inverse, the x and the y forward pass store so above it.
constexpr double kCacheBytes = 256e6;
template <typename T>
int stored_cols(const Box& b) {
    const int n = (b.KX + kPiece<T> - 1) / kPiece<T> * kPiece<T>;
    return b.KXP % 16 == 0 && n <= b.KXP ? n : b.KX;
}
// y inverse of `fields` fields (chains and boxes counted)
template <typename T>
int y_stored_cols(const laps_ctx* c, const Box& b, double fields) {
    return fields * c->nz * c->ny * b.KX * 2 * sizeof(T) > kCacheBytes ? stored_cols<T>(b) : b.KX;
}

// spectral box (fields with stride fs) -> real fields, unnormalised
// (transform_uu_fourier_to_real, fftw.f90:73-103)
// With dst == nullptr the x leg is left out and B holds the y-inverted rows.
// With shift, every field is sampled on the grid shifted by half a cell along
// each axis (phase-shift dealiasing): the z leg multiplies its input mode
// (mx, my, mz) by e^{i pi (mx/nx + my/ny + mz/nz)}, the shift of all three
// axes at once, as the modes are independent of each other in the y and x legs.
// With nch = 2 the z leg also writes the shifted fields as chain 1 (at A + a_ch),
// read once from src, and the y leg transforms both chains (chain 1 to B + b_ch).
template <typename T, typename TS = double>
int inv_pipeline(laps_ctx* c, const cpx<TS>* src, long long fs, const Box& b, int nf, T* dst, cpx<T>* A,
                 cpx<T>* B, int plan_z = 0, int plan_y = 0, bool shift = false, int nch = 1, long long a_ch = 0,
                 long long b_ch = 0, bool masked = false, int nbox = 1, long long src_bx = 0, long long a_bx = 0,
                 long long b_bx = 0, bool curl = false) {
    if (nch == 2 && (dst || !shift)) return fail(LAPS_EINVAL, "internal: two chains are the shifted pair");
    const long long NX = c->nx, NY = c->ny, NZ = c->nz;
    StridedArgs z{};
    if (shift) {
        z.ph = c->phz;
        z.phc = c->phx;
        z.phb = b.CY == c->ny ? c->phy : c->phyk;
    }
    const long long RS = b.KXP;
    z.ncol = b.KX; z.ncol_st = stored_cols<T>(b); z.in_cnt = b.CZ; z.out_cnt = (int)NZ;
    z.in_ls = (long long)b.CY * RS; z.out_ls = (long long)b.CY * RS;
    z.nb1 = b.CY; z.in_b1 = RS; z.out_b1 = RS;
    z.nb2 = nf; z.in_b2 = fs; z.out_b2 = NZ * b.CY * RS;
    z.nch = nch; z.out_ch = a_ch; z.pair = true;
    z.dual = nch == 2;  // the shifted chain from the plain chain's loads, in the same work-group
    z.nbox = nbox; z.in_bx = src_bx; z.out_bx = a_bx;
    if (curl) {  // the Hall current formed from B as the z pass loads it (no k_curl launch)
        const BoxTables t = c->tkept.view();
        z.curl = 1;
        z.kwx = t.wx; z.kwy = t.wy; z.kwz = t.wz;
        z.kctl = c->ctl;
        z.k_r0 = c->pp.radius0; z.k_cos = c->pp.cos_c; z.k_sin = c->pp.sin_c;
        z.k_corot = c->pp.corot_k;
    }
    // masked: src is the kept-box state after a masked substage (zero outside the kept set);
    // the mask rows with no kept mode are skipped by the z inverse and read as zero by the y
    // inverse
    const int mask = (masked && (c->p.dealias_option == 1 || c->p.dealias_option == 3)) ? c->p.dealias_option : 0;
    const double rows = mask ? (double)c->nlive : (double)b.CY * b.KX;
    if (mask) {
        z.mask = mask; z.row_role = 1; z.cy_cnt = b.CY;
        z.mX = NX; z.mY = NY; z.mZ = NZ;
    }
    // bytes: the kept rows of every stored field read once, every field written per chain (with
    // the Hall current formed here, J is not read: its B reads are those of fields 4-6)
    const double ez = (double)nf * rows, er = (double)(nf - (curl ? 3 : 0)) * rows;
    LAPS_CK(timed(c, K_ZINV, er * b.CZ * 2.0 * sizeof(TS) + ez * nch * NZ * 2.0 * sizeof(T),
                  [&] { return launch_strided<TS, T>(c->nz, +1, src, A, z, tw_of<T>(c, 2), T(1), c->stream, plan_z); }));
    StridedArgs y{};
    y.ncol = b.KX; y.ncol_st = y_stored_cols<T>(c, b, (double)nch * nbox * nf); y.in_cnt = b.CY; y.out_cnt = (int)NY;
    y.in_ls = RS; y.out_ls = RS;
    y.nb1 = (int)NZ; y.in_b1 = (long long)b.CY * RS; y.out_b1 = NY * RS;
    y.nb2 = nf; y.in_b2 = NZ * b.CY * RS; y.out_b2 = NZ * NY * RS;
    y.nch = nch; y.in_ch = a_ch; y.out_ch = b_ch;
    y.nbox = nbox; y.in_bx = a_bx; y.out_bx = b_bx;
    if (mask) {
        y.mask = mask; y.row_role = 2;
        y.mX = NX; y.mY = NY; y.mZ = NZ;
    }
    const double ey = (double)nf * NZ * 2.0 * sizeof(T);
    LAPS_CK(timed(c, K_YINV, nch * ey * (rows + (double)b.KX * NY),
                  [&] { return launch_strided<T, T>(c->ny, +1, A, B, y, tw_of<T>(c, 1), T(1), c->stream, plan_y); }));
    if (!dst) return LAPS_OK;
    XArgs x{};
    x.nrows = (long long)nf * NZ * NY; x.kx = b.KX; x.crow = RS; x.rrow = NX;
    LAPS_CK(timed(c, K_XC2R, (double)x.nrows * sizeof(T) * (2.0 * b.KX + NX),
                  [&] { return launch_x_c2r<T>(c->nx, B, dst, x, tw_of<T>(c, 0), c->stream); }));
    return LAPS_OK;
}

// real fields -> spectral box in A, normalised by 1/(nx ny nz)
// (transform_flux_real_to_fourier, mhdrhs.f90:128-172; fftw.f90:42-71).
// With src == nullptr the x leg is left out: A already holds x-transformed rows.
template <typename T>
int fwd_pipeline(laps_ctx* c, const T* src, int nf, const Box& b, cpx<T>* A, cpx<T>* B) {
    const long long NX = c->nx, NY = c->ny, NZ = c->nz;
    const long long RS = b.KXP;
    if (src) {
        XArgs x{};
        x.nrows = (long long)nf * NZ * NY; x.kx = b.KX; x.crow = RS; x.rrow = NX;
        LAPS_CK(timed(c, K_XR2C, (double)x.nrows * sizeof(T) * (2.0 * b.KX + NX),
                      [&] { return launch_x_r2c<T>(c->nx, src, A, x, tw_of<T>(c, 0), c->stream); }));
    }
    StridedArgs y{};
    y.ncol = y.ncol_st = b.KX; y.in_cnt = (int)NY; y.out_cnt = b.CY;
    y.in_ls = RS; y.out_ls = RS;
    y.nb1 = (int)NZ; y.in_b1 = NY * RS; y.out_b1 = (long long)b.CY * RS;
    y.nb2 = nf; y.in_b2 = NZ * NY * RS; y.out_b2 = NZ * b.CY * RS;
    const double ey = (double)nf * NZ * b.KX * 2.0 * sizeof(T);
    LAPS_CK(timed(c, K_YFWD, ey * (NY + b.CY),
                  [&] { return launch_strided<T, T>(c->ny, -1, A, B, y, tw_of<T>(c, 1), T(1), c->stream); }));
    StridedArgs z{};
    z.ncol = z.ncol_st = b.KX; z.in_cnt = (int)NZ; z.out_cnt = b.CZ;
    z.in_ls = (long long)b.CY * RS; z.out_ls = (long long)b.CY * RS;
    z.nb1 = b.CY; z.in_b1 = RS; z.out_b1 = RS;
    z.nb2 = nf; z.in_b2 = NZ * b.CY * RS; z.out_b2 = (long long)b.CZ * b.CY * RS;
    const T scale = T(1.0 / ((double)c->nx * (double)c->ny * (double)c->nz));
    const double ez = (double)nf * b.CY * b.KX * 2.0 * sizeof(T);
    LAPS_CK(timed(c, K_ZFWD, ez * (NZ + b.CZ),
                  [&] { return launch_strided<T, T>(c->nz, -1, B, A, z, tw_of<T>(c, 2), scale, c->stream); }));
    return LAPS_OK;
}

// The z-inverse input of a substage: the FP64 state, or its FP32 copy in mixed precision
// (the transforms round their input to FP32 at load either way).
template <typename T>
const cpx<T>* state_src(laps_ctx* c);
template <>
const cpx<double>* state_src<double>(laps_ctx* c) { return c->U; }
template <>
const cpx<float>* state_src<float>(laps_ctx* c) { return c->Uf; }

// Points per field (kept kx, all chains and boxes of the launch) below which the y forward pass runs
// its split groups. Measured in FP64, large form against split: 32^3 12.8 -> 6.6 us, 64^3 14.9 ->
// 10.7, 96x32x64 with two chains (188k points) 20.8 -> 19.5; 128x128x64 (532k) 48.4 -> 53.0,
// 256^3 348 -> 437.
constexpr long long kYSplitPoints = 1LL << 18;

// the right-hand side holds the state itself (rhs_holds_u in the kernels)
bool rhs_holds_state(const PhysParams& pp) {
    return pp.aeb || (pp.visc && pp.visc_exp) || (pp.resis && pp.resis_exp);
}

// one substage of evolve (mhd.f90:303-325): [curl J] -> z, y inverse ->
// fused x pass (C2R, fluxes, CFL, R2C) -> y, z forward -> RHS + RK3 + dealias
template <typename T>
int substage(laps_ctx* c, int irk) {
    const bool first = c->fresh && irk == 0;
    const bool hall = c->p.if_hall != 0;
    const long long KB = c->kb();
    const long long NZ = c->nz, NY = c->ny;
    cpx<T>* P1 = (cpx<T>*)c->P1;
    cpx<T>* P2 = (cpx<T>*)c->P2;
    const Box& k = c->kept;
    // batched launches (ensemble groups): every launch covers nb boxes
    const laps_ctx::Batch& bt = c->batch;
    const int nb = bt.n;
    if (nb > 1 && first) return fail(LAPS_EINVAL, "internal: the first substage is not batched");
    int rc;
    XFArgs xa{};
    xa.nbox = nb;
    xa.st_bx = bt.p2;
    xa.jb_bx = bt.p2;
    xa.out_bx = bt.p1;
    xa.nrows = NZ * NY;
    xa.npts = c->N;
    xa.S = c->S;
    xa.out = P1;
    xa.kx_o = k.KX;
    xa.rs_o = k.KXP;
    xa.fs_o = NZ * NY * k.KXP;
    xa.mass = c->mass_flux() ? 1 : 0;
    double xin;
    // phase-shift dealiasing after the first substage: the plain and the shifted grid run as
    // chains 0 and 1 of each launch of the inverse, x and y-forward passes
    const int nch = (!first && c->p.dealias_option == 3) ? 2 : 1;
    if (first) {
        // first substage: the uploaded real fields are used as they are; J
        // comes from the un-dealiased spectrum (mhd.f90:121-122, :305)
        if (hall) {
            LAPS_CK(timed(c, K_CURL, 96.0 * c->M, [&] {
                return launch_curl(c->Ufull, c->Ufull + 8 * c->M, c->M, c->full, c->tfull.view(), c->pp, c->ctl,
                                   c->stream);
            }));
            if ((rc = inv_pipeline<T>(c, c->Ufull + 8 * c->M, c->M, c->full, 3, (T*)nullptr, P1, P2))) return rc;
            xa.jb = P2;
            xa.kx_j = c->nxh;
            xa.rs_j = c->full.KXP;
            xa.fs_j = NZ * NY * c->full.KXP;
        }
        xin = 96.0 * c->N + (hall ? 3.0 * xa.nrows * c->nxh * 2 * sizeof(T) : 0.0);
    } else {
        // the Hall current J = i k' x B is formed by the z inverse from the B fields it loads
        // (StridedArgs::curl): no J is written to or read from HBM
        if ((rc = inv_pipeline<T, T>(c, state_src<T>(c), KB, k, c->nf_in(), (T*)nullptr, P1, P2, c->plan_zinv,
                                     c->plan_yinv, nch == 2, nch, c->p1, c->p2, true, nb,
                                     c->Uf ? bt.uf : bt.u, bt.p1, bt.p2, hall)))
            return rc;
        xa.nch = nch;
        xa.st_ch = c->p2;
        xa.jb_ch = c->p2;
        xa.out_ch = c->p1;
        xa.st = P2;
        xa.kx_s = k.KX;
        xa.rs_s = k.KXP;
        xa.fs_s = NZ * NY * k.KXP;
        xa.jb = P2 + 8 * xa.fs_s;
        xa.kx_j = k.KX;
        xa.rs_j = k.KXP;
        xa.fs_j = xa.fs_s;
        xin = (double)nch * c->nf_in() * xa.nrows * k.KX * 2 * sizeof(T);
    }
    if ((double)nch * nb * c->nf_out() * NZ * NY * k.KX * 2 * sizeof(T) > kCacheBytes) xa.kx_o = stored_cols<T>(k);
    const bool cfl = irk == 0 && !(c->fixed_dt > 0);
    const double xout = (double)c->nf_out() * xa.nrows * k.KX * 2 * sizeof(T);
    LAPS_CK(timed(c, K_XFUSED, xin + nch * xout, [&] {
        return launch_xfused<T>(c->nx, first, cfl, xa, tw_of<T>(c, 0), c->pp, c->ctl, c->stream);
    }));
    if (irk == 0) LAPS_CK(timed(c, K_CTL, 0.0, [&] { return launch_ctl_finalize(c->ctl, c->pp, c->stream, nb); }));
    // y forward with the x/y derivative terms folded in, then z forward + RHS + RK3 + dealias
    // small launches: the groups that transform one or two fields each (setup_forward_groups)
    YGArgs ya = k.KX * NZ * NY * nch * nb < kYSplitPoints ? c->yg_split : c->yg;
    ya.nch = nch;
    ya.pieces = (double)nch * nb * c->nd() * NZ * k.CY * k.KX * 2 * sizeof(T) > kCacheBytes;
    if (ya.pieces) ya.ncol_st = stored_cols<T>(k);
    // the groups of a tile after each other where the pass reads more than 1.1 GB: 256^3 phase shift FP32
    // 613 -> 592 us, FP64 1142 -> 1134, 512x512x128 FP32 480 -> 466, 128x512x128 phase shift FP64
    // 717 -> 657; below, a group at a time (256^3 2/3 rule FP32 180, 188 mixed; 128^3 FP64 45, 53).
    // By the box where boxes are batched: see the rule of the strided passes (do_strided_p)
    ya.mix = (double)nch * c->nf_out() * NZ * NY * k.KX * 2 * sizeof(T) > 1.1e9;
    ya.in_ch = c->p1;
    ya.out_ch = c->p2;
    ya.ylim = c->tkept.ylim;
    ya.nbox = nb;
    ya.in_bx = bt.p1;
    ya.out_bx = bt.p2;
    // bytes per mode and variable of the update: U or V read (in the second substage both where the
    // right-hand side holds the state), U, V and the FP32 copy written as store_u says
    const bool rd_u = rhs_holds_state(c->pp);
    const double state_bytes = 16.0 * (1 + (irk == 1 && rd_u ? 1 : 0) +
                                       (sizeof(T) == 8 || irk == 2 || (irk == 0 && rd_u) ? 1 : 0) +
                                       (irk < 2 ? 1 : 0)) + (c->Uf ? 8.0 : 0.0);
    double mass_bytes = 0.0;
    if (!c->mass_flux()) {
        MassArgs& m = ya.mass;
        m.KX = k.KX; m.CY = k.CY; m.CZ = k.CZ; m.KXP = k.KXP;
        m.nblk = 1;
        m.U = c->U;
        m.Uf = c->Uf;
        m.V = c->V;
        m.ufs = KB;
        m.tb = c->tkept.view();
        m.irk = irk;
        m.clear_outside = first ? 1 : 0;
        m.u_bx = bt.u;
        m.uf_bx = bt.uf;
        m.v_bx = bt.v;
        // rho or V read, m read, rho stored (see state_bytes)
        mass_bytes = (double)c->nkept * (state_bytes + 3 * 2.0 * sizeof(T));
    }
    LAPS_CK(timed(c, K_YFWD, nch * c->yfwd_bytes * sizeof(T) + mass_bytes, [&] {
        return launch_yfwd_group<T>(c->ny, P1, P2, ya, tw_of<T>(c, 1), c->tkept.wx, c->tfull.wy, c->pp, c->ctl,
                                    c->nz, c->stream);
    }));
    ZArgs za = c->zr;
    cpx<T>* P3 = (cpx<T>*)c->P3;
    if (first && c->p.dealias_option == 3) {
        // phase-shift dealiasing, first substage: the shifted grid from the full spectrum, after
        // the plain one (z-inverse input times e^{i pi m/n} of all three axes, z-forward output
        // times the conjugate); its y-pass output goes to P3
        XFArgs xs = xa;
        if ((rc = inv_pipeline<T>(c, c->Ufull, c->M, c->full, c->nf_in(), (T*)nullptr, P1, P3, 0, 0, true)))
            return rc;
        xs.kx_s = c->nxh;
        xs.rs_s = c->full.KXP;
        xs.fs_s = NZ * NY * c->full.KXP;
        xs.st = P3;
        xs.jb = P3 + 8 * xs.fs_s;
        xs.kx_j = xs.kx_s;
        xs.rs_j = xs.rs_s;
        xs.fs_j = xs.fs_s;
        const double xins = (double)c->nf_in() * xs.nrows * xs.kx_s * 2 * sizeof(T);
        LAPS_CK(timed(c, K_XFUSED, xins + xout, [&] {
            return launch_xfused<T>(c->nx, false, false, xs, tw_of<T>(c, 0), c->pp, c->ctl, c->stream);
        }));
        ya.mass.nblk = 0;  // rho is updated once
        LAPS_CK(timed(c, K_YFWD, c->yfwd_bytes * sizeof(T), [&] {
            return launch_yfwd_group<T>(c->ny, P1, P3, ya, tw_of<T>(c, 1), c->tkept.wx, c->tfull.wy, c->pp, c->ctl,
                                        c->nz, c->stream);
        }));
    }
    za.clos = c->closure ? c->cl_rhs : nullptr;
    za.Uf = c->Uf;
    za.nbox = nb;
    za.d_bx = bt.p2;
    za.u_bx = bt.u;
    za.v_bx = bt.v;
    za.uf_bx = bt.uf;
    if (c->p.dealias_option == 3) {
        // the z pass averages the right-hand sides of the two grids
        za.Ds = P3;
        za.ph = c->phz;
        za.phc = c->phx;
        za.phb = c->phyk;
    }
    const T scale = T(1.0 / ((double)c->nx * (double)c->ny * (double)c->nz));
    // kept modes only: outside the kept set nothing is read, and U is written as
    // zero only by the first substage after a state upload
    za.clear_outside = first ? 1 : 0;
    const double nv = c->mass_flux() ? 8.0 : 7.0;
    const double cleared = first ? (double)k.KX * k.CY * k.CZ - (double)c->nkept : 0.0;
    const double zb = c->zfwd_bytes * sizeof(T) * (za.Ds ? 2 : 1) + nv * (double)c->nkept * state_bytes +
                      nv * cleared * (16.0 + (c->Uf ? 8.0 : 0.0));
    LAPS_CK(timed(c, K_ZFWD, zb, [&] {
        return launch_zfwd_rhs<T>(c->nz, P2, c->U, c->V, za, tw_of<T>(c, 2), c->tkept.view(), c->tfull.wz, c->pp,
                                  c->ctl, irk, scale, c->stream);
    }));
    return LAPS_OK;
}

// Times the inverse z and y passes of the kept box in each variant (two FFT plans x two tile
// widths; events on the context stream, on the real buffers) and keeps the fastest of each.
template <typename T>
int autotune(laps_ctx* c) {
    // LAPS_FFT_PLAN = 0 or 1 fixes both plans (default tile width) instead (reproducible runs:
    // the timed choice can differ between contexts, and with it the rounding of the transforms);
    // "z,y" (two variants 0-3) fixes the z and y inverse variants separately
    if (const char* fixed = std::getenv("LAPS_FFT_PLAN")) {
        if ((fixed[0] == '0' || fixed[0] == '1') && fixed[1] == 0) {
            c->plan_zinv = c->plan_yinv = fixed[0] - '0';
            c->tuned = true;
            return LAPS_OK;
        }
        if (fixed[0] >= '0' && fixed[0] <= '3' && fixed[1] == ',' && fixed[2] >= '0' && fixed[2] <= '3' &&
            fixed[3] == 0) {
            c->plan_zinv = fixed[0] - '0';
            c->plan_yinv = fixed[2] - '0';
            c->tuned = true;
            return LAPS_OK;
        }
    }
    TimingOff off(c);
    const Box& k = c->kept;
    cpx<T>* P1 = (cpx<T>*)c->P1;
    cpx<T>* P2 = (cpx<T>*)c->P2;
    hipEvent_t e0, e1;
    LAPS_CK(hipEventCreate(&e0));
    LAPS_CK(hipEventCreate(&e1));
    constexpr int NV = 4;
    float best_zy[NV] = {0, 0, 0, 0}, best_y[NV] = {0, 0, 0, 0};  // min over repetitions
    // the launches a step makes: with phase-shift dealiasing both grids as two chains
    const int nch = c->p.dealias_option == 3 ? 2 : 1;
    const long long NY = c->ny, NZ = c->nz, RS = k.KXP;
    StridedArgs y{};
    y.ncol = k.KX; y.ncol_st = y_stored_cols<T>(c, k, (double)nch * c->nf_in()); y.in_cnt = k.CY; y.out_cnt = (int)NY;
    y.in_ls = RS; y.out_ls = RS;
    y.nb1 = (int)NZ; y.in_b1 = (long long)k.CY * RS; y.out_b1 = NY * RS;
    y.nb2 = c->nf_in(); y.in_b2 = NZ * k.CY * RS; y.out_b2 = NZ * NY * RS;
    y.nch = nch; y.in_ch = c->p1; y.out_ch = c->p2;
    if (c->p.dealias_option == 1 || c->p.dealias_option == 3) {  // as in the substage
        y.mask = c->p.dealias_option; y.row_role = 2;
        y.mX = c->nx; y.mY = NY; y.mZ = NZ;
    }
    auto time_it = [&](auto launch, float& ms) -> int {
        LAPS_CK(hipEventRecord(e0, c->stream));
        const int rc = launch();
        if (rc) return rc;
        LAPS_CK(hipEventRecord(e1, c->stream));
        LAPS_CK(hipEventSynchronize(e1));
        LAPS_CK(hipEventElapsedTime(&ms, e0, e1));
        return LAPS_OK;
    };
    for (int rep = 0; rep < 4; ++rep) {
        for (int v = 0; v < NV; ++v) {
            // z (variant v) + y (variant 0), then y alone (variant v)
            float ms_zy = 0, ms_y = 0;
            int rc = time_it([&] {
                return inv_pipeline<T, T>(c, state_src<T>(c), c->kb(), k, c->nf_in(), (T*)nullptr, P1, P2, v, 0,
                                          nch == 2, nch, c->p1, c->p2, true, 1, 0, 0, 0, c->p.if_hall != 0);
            }, ms_zy);
            if (!rc) rc = time_it([&] {
                const hipError_t he = launch_strided<T, T>(c->ny, +1, P1, P2, y, tw_of<T>(c, 1), T(1), c->stream, v);
                return he == hipSuccess ? LAPS_OK : fail(LAPS_EDEVICE, hipGetErrorString(he));
            }, ms_y);
            if (rc) {
                (void)hipEventDestroy(e0);
                (void)hipEventDestroy(e1);
                return rc;
            }
            if (rep == 0) continue;  // warm-up
            best_zy[v] = (rep == 1 || ms_zy < best_zy[v]) ? ms_zy : best_zy[v];
            best_y[v] = (rep == 1 || ms_y < best_y[v]) ? ms_y : best_y[v];
        }
    }
    // a variant other than the default only when clearly faster (3 %), so repeated runs pick
    // the same code; the z pass is compared on its own time (z + y with the y variant held at 0,
    // less that y time)
    int vz = 0, vy = 0;
    float tz = best_zy[0] - best_y[0];
    for (int v = 1; v < NV; ++v) {
        const float z = best_zy[v] - best_y[0];
        if (z < 0.97f * tz) { tz = z; vz = v; }
    }
    // the y pass is compared where a step runs it: right after the chosen z pass (its time
    // alone, on an input written long before, has ranked the variants differently)
    float best_zyv[NV] = {0, 0, 0, 0};
    for (int rep = 0; rep < 4; ++rep) {
        for (int v = 0; v < NV; ++v) {
            float ms = 0;
            const int rc = time_it([&] {
                return inv_pipeline<T, T>(c, state_src<T>(c), c->kb(), k, c->nf_in(), (T*)nullptr, P1, P2, vz, v,
                                          nch == 2, nch, c->p1, c->p2, true, 1, 0, 0, 0, c->p.if_hall != 0);
            }, ms);
            if (rc) {
                (void)hipEventDestroy(e0);
                (void)hipEventDestroy(e1);
                return rc;
            }
            if (rep == 0) continue;  // warm-up
            best_zyv[v] = (rep == 1 || ms < best_zyv[v]) ? ms : best_zyv[v];
        }
    }
    (void)hipEventDestroy(e0);
    (void)hipEventDestroy(e1);
    float ty = best_zyv[0];
    for (int v = 1; v < NV; ++v)
        if (best_zyv[v] < 0.97f * ty) { ty = best_zyv[v]; vy = v; }
    c->plan_zinv = vz;
    c->plan_yinv = vy;
    c->tuned = true;
    if (std::getenv("LAPS_TUNE_LOG")) {
        std::fprintf(stderr, "[laps] autotune %dx%dx%d %s: z inverse", c->nx, c->ny, c->nz, c->mixed ? "mixed" : "fp64");
        for (int v = 0; v < NV; ++v) std::fprintf(stderr, " %.3f", best_zy[v] - best_y[0]);
        std::fprintf(stderr, " ms -> variant %d; z + y inverse", vz);
        for (int v = 0; v < NV; ++v) std::fprintf(stderr, " %.3f", best_zyv[v]);
        std::fprintf(stderr, " ms -> y variant %d\n", vy);
    }
    return LAPS_OK;
}

int closure_step(laps_ctx* c, bool full);

template <typename T>
int one_step(laps_ctx* c) {
    int rc;
    if (c->closure && (rc = closure_step(c, false))) return rc;
    for (int irk = 0; irk < 3; ++irk)
        if ((rc = substage<T>(c, irk))) return rc;
    LAPS_CK(timed(c, K_CTL, 0.0, [&] { return launch_ctl_end(c->ctl, c->pp, c->stream, c->batch.n); }));
    c->fresh = false;
    c->materialized = false;
    return LAPS_OK;
}

// FP64 single-field utilities (set_state, materialisation, laps_fft_*)
int fwd_fp64(laps_ctx* c, const double* real, cpx<double>* out_full) {
    TimingOff off(c);
    int rc = fwd_pipeline<double>(c, real, 1, c->full, c->X1, c->X2);
    if (rc) return rc;
    if (out_full != c->X1)
        LAPS_CK(hipMemcpyAsync(out_full, c->X1, c->M * sizeof(cpx<double>), hipMemcpyDeviceToDevice, c->stream));
    return LAPS_OK;
}

int inv_fp64(laps_ctx* c, const cpx<double>* src, const Box& b, double* real) {
    TimingOff off(c);
    return inv_pipeline<double>(c, src, b.modes(), b, 1, real, c->X1, c->X2);
}

// FP64 complex fields of n elements that P1 and P2 hold (at least one, at most 8)
int p1_fields(const laps_ctx* c, long long n) {
    const long long chains = c->p.dealias_option == 3 ? 2 : 1, ts = c->mixed ? 4 : 8;
    return (int)std::max(1LL, std::min(8LL, chains * c->p1 * ts / 8 / n));
}
int p2_fields(const laps_ctx* c, long long n) {
    const long long chains = c->p.dealias_option == 3 ? 2 : 1, ts = c->mixed ? 4 : 8;
    return (int)std::max(1LL, std::min(8LL, chains * c->p2 * ts / 8 / n));
}

// A step refused by the dt < 1e-8 test (status LAPS_DT_STOP) leaves the
// state untouched; if no step was ever taken since laps_set_state, the
// uploaded arrays are still the state (mhd.f90:216-242 writes them as is).
int refresh_fresh(laps_ctx* c) {
    if (c->fresh || !c->stepped_since_set) return LAPS_OK;
    Ctl h;
    LAPS_CK(hipStreamSynchronize(c->stream));
    LAPS_CK(hipMemcpy(&h, c->ctl, sizeof(Ctl), hipMemcpyDeviceToHost));
    if (h.status != 0 && h.istep == 0) {
        c->fresh = true;
        c->materialized = true;
    }
    return LAPS_OK;
}

// S is read by a queued output copy until stage_done: work that rewrites S waits for it
int wait_stage(laps_ctx* c, bool host) {
    if (!c->stage_pending) return LAPS_OK;
    if (host) LAPS_CK(hipEventSynchronize(c->stage_done));
    else LAPS_CK(hipStreamWaitEvent(c->stream, c->stage_done, 0));
    return LAPS_OK;
}

int materialize(laps_ctx* c) {
    int rc0 = refresh_fresh(c);
    if (rc0) return rc0;
    if (c->materialized) return LAPS_OK;
    int rc;
    if ((rc = wait_stage(c, false))) return rc;
    // as many fields to a launch as the step's intermediates hold in FP64 (nothing in them outlives a
    // step): all 8 in FP64, 4 or more in mixed precision. One field to a launch, in scratch of its
    // own, the state took 161 us at 32^3 and 1.79 ms at 256^3; so, 73 us and 1.62 ms.
    TimingOff off(c);
    const Box& k = c->kept;
    const int nf = std::min(p1_fields(c, (long long)c->nz * k.CY * k.KXP), p2_fields(c, (long long)c->nz * c->ny * k.KXP));
    for (int f = 0; f < 8; f += nf)
        if ((rc = inv_pipeline<double>(c, c->U + f * c->kb(), c->kb(), k, std::min(nf, 8 - f), c->S + f * c->N,
                                       (cpx<double>*)c->P1, (cpx<double>*)c->P2, 0, 0, false, 1, 0, 0, true)))
            return rc;
    LAPS_CK(launch_prim<double>(c->S, c->S + 8 * c->N, c->N, c->p.adiabatic_index, c->stream));
    c->materialized = true;
    return LAPS_OK;
}

// Learned closure, evaluated once per step on the state at the start of the
// step: features -> network -> 12 correction fields -> their spectra -> the
// momentum, induction and energy RHS term on the kept box (held over the three
// substages; the z pass adds it).
int closure_buffers(laps_ctx* c) {
    if (c->cl_P) return LAPS_OK;
    int rc;
    if ((rc = c->allocn(&c->cl_P, kClNParam + kClNNorm)) || (rc = c->allocn(&c->cl_X, c->N * kClIn)) ||
        (rc = c->allocn(&c->cl_Y, c->N * kClOut)) || (rc = c->allocn(&c->cl_id, 2 * kClIn)) ||
        (rc = c->allocn(&c->cl_C, 12 * c->N)) ||
        (rc = c->allocn(&c->cl_A, 12 * std::max(c->M, (long long)c->nz * c->ny * c->kept.KXP))) ||
        (rc = c->allocn(&c->cl_B, 12 * std::max(c->M, (long long)c->nz * c->ny * c->kept.KXP))) ||
        (rc = c->allocn(&c->cl_full, 7 * c->M)) || (rc = c->allocn(&c->cl_rhs, 7 * c->kb())))
        return rc;
    std::vector<float> id(2 * kClIn, 0.f);
    for (int q = 0; q < kClIn; ++q) id[kClIn + q] = 1.f;
    LAPS_CK(hipMemcpy(c->cl_id, id.data(), id.size() * sizeof(float), hipMemcpyHostToDevice));
    return LAPS_OK;
}

int closure_features(laps_ctx* c, const float* norm) {
    int rc = materialize(c);
    if (rc) return rc;
    LAPS_CK(launch_cl_features(c->S, c->nx, c->ny, c->nz, c->pp.dx, c->pp.dy, c->pp.dz, norm, c->cl_X, c->stream));
    return LAPS_OK;
}

// On the kept box (the step: cl_rhs) or, for laps_closure_eval, the full spectrum (cl_full) with
// the network's outputs in cl_Y.
int closure_step(laps_ctx* c, bool full) {
    int rc = materialize(c);
    if (rc) return rc;
    LAPS_CK(launch_cl_net(c->S, c->nx, c->ny, c->nz, c->pp.dx, c->pp.dy, c->pp.dz, c->cl_P, c->p.adiabatic_index,
                          full ? c->cl_Y : nullptr, c->cl_C, c->stream));
    const Box& b = full ? c->full : c->kept;
    {
        TimingOff off(c);  // the 12 fields in one batched transform; spectra in cl_A
        if ((rc = fwd_pipeline<double>(c, c->cl_C, 12, b, c->cl_A, c->cl_B))) return rc;
    }
    LAPS_CK(launch_cl_rhs(c->cl_A, b, (full ? c->tfull : c->tkept).view(), full ? c->cl_full : c->cl_rhs, c->stream));
    return LAPS_OK;
}

// Forward-pass plan: the groups of the y pass, from the x pass's flux slots (0-5 momentum tensor xx
// xy xz yy yz zz, 6-8 E, 9-11 energy, 12 expanding-box source, 13-15 mass without dealiasing) to the
// fields of the z pass (kDMom ...). Largest groups first, so that their work-groups start first.
// In the large form the momentum tensor is one group: each component is read and transformed once
// and used in both rows, six transforms in a chain. In the split form every output field is a group
// of its own with two transforms at most, the off-diagonal components transformed again: more work,
// a third of the chain, for launches too small to fill the chip with chains.
void setup_forward_groups(laps_ctx* c) {
    const Box& k = c->kept;
    const long long NY = c->ny, NZ = c->nz;
    for (int split = 0; split < 2; ++split) {
        YGArgs y{};
        y.ncol = y.ncol_st = k.KX;  // (the substage sets ncol_st)
        y.cy = k.CY;
        y.rs = k.KXP;
        y.in_fs = NZ * NY * k.KXP;
        y.out_fs = NZ * k.CY * k.KXP;
        y.nch = 1;
        int g = 0;
        auto group = [&](int kind) -> YGroup& {
            YGroup& q = y.g[g++];
            q.kind = kind;
            for (int t = 0; t < 6; ++t) q.in[t] = q.out[t] = -1;
            return q;
        };
        auto copy = [&](int in, int out) {
            YGroup& q = group(2);
            q.in[0] = in;
            q.out[0] = out;
        };
        std::vector<std::pair<int, int>> copies;  // after the groups of two and more transforms
        auto divergence = [&](int a, int b, int d, int out, int source) {
            YGroup& q = group(0);
            q.in[0] = a;
            q.in[1] = b;
            q.in[2] = split ? -1 : d;
            q.in[3] = source;
            q.out[0] = out;
            q.out[1] = out + 1;
            if (split) copies.push_back({d, out + 1});
        };
        if (split) {
            const int row[3][3] = {{0, 1, 2}, {1, 3, 4}, {2, 4, 5}};
            for (int t = 0; t < 3; ++t) divergence(row[t][0], row[t][1], row[t][2], kDMom + 2 * t, -1);
        } else {
            YGroup& mom = group(3);
            for (int t = 0; t < 6; ++t) {
                mom.in[t] = t;
                mom.out[t] = kDMom + t;
            }
        }
        divergence(9, 10, 11, kDEnergy, c->p.if_aeb ? 12 : -1);
        if (c->mass_flux()) divergence(13, 14, 15, kDMass, -1);
        for (const auto& q : copies) copy(q.first, q.second);
        for (int t = 0; t < 3; ++t) copy(6 + t, kDE + t);
        y.ngroups = g;
        (split ? c->yg_split : c->yg) = y;
    }
    ZArgs z{};
    z.KX = k.KX; z.CY = k.CY; z.CZ = k.CZ;
    z.rs = k.KXP;
    z.in_fs = NZ * k.CY * k.KXP;
    z.ufs = k.modes();
    z.mass = c->mass_flux() ? 1 : 0;
    z.mX = c->nx; z.mY = NY; z.mZ = NZ;
    c->zr = z;
    // the y pass stores, and the z pass reads, only the (kx, cy) rows that hold a kept mode
    c->yfwd_bytes = 2.0 * NZ * ((double)c->nf_out() * NY * k.KX + (double)c->nd() * c->nlive);
    c->zfwd_bytes = 2.0 * (double)c->nlive * c->nd() * NZ;
}

PhysParams make_phys(const laps_params& p) {
    PhysParams pp{};
    pp.gamma = p.adiabatic_index;
    pp.di = p.ion_inertial_length;
    pp.nu = p.viscosity;
    pp.eta = p.resistivity;
    pp.radius0 = p.radius0;
    pp.Ur = p.if_aeb ? p.Ur0 : 0.0;  // mhd.f90:88-90
    const double ang = p.if_corotating ? p.corotating_angle : 0.0;  // AEBmod.f90:28-30
    pp.cos_c = cos(ang);
    pp.sin_c = sin(ang);
    pp.cfl = p.cfl;
    pp.fixed_dt = 0.0;
    pp.dx = p.Lx / p.nx;
    pp.dy = p.Ly / p.ny;
    pp.dz = p.Lz / p.nz;
    pp.hall = p.if_hall != 0;
    pp.aeb = p.if_aeb != 0;
    pp.corot_k = p.if_aeb && p.if_corotating;
    pp.corot_ksq = p.if_corotating != 0;
    pp.visc = p.if_visc != 0;
    pp.visc_exp = p.if_visc_exp != 0;
    pp.resis = p.if_resis != 0;
    pp.resis_exp = p.if_resis_exp != 0;
    pp.conserve_bg = p.if_conserve_background != 0;
    pp.dealias = p.dealias_option;
    return pp;
}

int reset_ctl(laps_ctx* c, double time, double dt_prev, bool ksq_updated) {
    Ctl h{};
    h.time = time;
    h.dt = 0.0;
    h.dt_prev = dt_prev;
    h.radius = c->pp.radius0 + c->pp.Ur * time;
    h.tau = h.radius / c->pp.Ur;
    h.r0r = c->pp.radius0 / h.radius;
    h.dtmin_bits = 0x7FF0000000000000ULL;
    for (int i = 0; i < kCflSlots; ++i) h.dtmin_slot[i] = 0x7FF0000000000000ULL;
    h.istep = 0;
    h.status = 0;
    h.ksq_updated = ksq_updated ? 1 : 0;
    LAPS_CK(hipMemcpy(c->ctl, &h, sizeof(Ctl), hipMemcpyHostToDevice));
    return LAPS_OK;
}

int read_ctl(laps_ctx* c, Ctl& h) {
    LAPS_CK(hipStreamSynchronize(c->stream));
    LAPS_CK(hipMemcpy(&h, c->ctl, sizeof(Ctl), hipMemcpyDeviceToHost));
    return LAPS_OK;
}

int check_ctx(laps_ctx* c, bool need_state) {
    if (!c) return fail(LAPS_EINVAL, "null context");
    if (need_state && !c->have_state) return fail(LAPS_ESTATE, "no state: call laps_set_state first");
    hipError_t e = hipSetDevice(c->p.device);
    if (e != hipSuccess) return fail(LAPS_EDEVICE, std::string("hipSetDevice: ") + hipGetErrorString(e));
    return LAPS_OK;
}

void free_all(laps_ctx* c) {
    for (auto& pe : c->timing.pending) {
        c->timing.pool.push_back(pe.second.first);
        c->timing.pool.push_back(pe.second.second);
    }
    c->timing.pending.clear();
    for (hipEvent_t e : c->timing.pool) (void)hipEventDestroy(e);
    c->timing.pool.clear();
    for (void* ptr : c->allocs) (void)hipFree(ptr);
    c->allocs.clear();
    if (c->stage_stream) (void)hipStreamSynchronize(c->stage_stream);
    if (c->stage_host) (void)hipHostFree(c->stage_host);
    c->host.release();
    if (c->stage_ready) (void)hipEventDestroy(c->stage_ready);
    if (c->stage_done) (void)hipEventDestroy(c->stage_done);
    if (c->stage_stream) (void)hipStreamDestroy(c->stage_stream);
    c->stage_host = nullptr;
    c->stage_ready = c->stage_done = nullptr;
    c->stage_stream = nullptr;
    if (c->stream) (void)hipStreamDestroy(c->stream);
    c->stream = nullptr;
}

}  // namespace

// ====================================================================== C ABI

extern "C" {

void laps_default_params(laps_params* p) {
    if (!p) return;
    std::memset(p, 0, sizeof(*p));
    p->nx = 128; p->ny = 128; p->nz = 64;
    p->precision = LAPS_FP64;
    p->Lx = p->Ly = p->Lz = 2.0 * kPiRef;
    p->adiabatic_index = 5. / 3.;
    p->cfl = 0.5;
    p->dealias_option = 2;
    p->afx = p->afy = p->afz = 0.495;
    p->radius0 = 30.0;
}

const char* laps_last_error(void) { return g_err.c_str(); }

int laps_create(const laps_params* p, laps_ctx** out) {
    if (!p || !out) return fail(LAPS_EINVAL, "null argument");
    *out = nullptr;
    if (!supported_len(p->nx) || !supported_len(p->ny) || !supported_len(p->nz))
        return fail(LAPS_EINVAL, "grid lengths must be 16, 32, 64, 96, 128, 256 or 512 per axis");
    if (p->precision != LAPS_FP64 && p->precision != LAPS_MIXED) return fail(LAPS_EINVAL, "unknown precision");
    if (p->dealias_option < 0 || p->dealias_option > 3)
        return fail(LAPS_EINVAL, "dealias_option must be 0, 1, 2 or 3");
    if (!(p->Lx > 0 && p->Ly > 0 && p->Lz > 0)) return fail(LAPS_EINVAL, "box lengths must be positive");
    int ndev = 0;
    if (hipGetDeviceCount(&ndev) != hipSuccess || ndev <= p->device || p->device < 0)
        return fail(LAPS_EDEVICE, "no HIP device " + std::to_string(p->device));
    LAPS_CK(hipSetDevice(p->device));
    laps_ctx* c = new laps_ctx();
    c->p = *p;
    c->nx = p->nx; c->ny = p->ny; c->nz = p->nz; c->nxh = p->nx / 2 + 1;
    c->N = (long long)c->nx * c->ny * c->nz;
    c->M = (long long)c->nxh * c->ny * c->nz;
    c->mixed = p->precision == LAPS_MIXED;
    c->full = Box{c->nxh, c->ny, c->nz, c->nxh};
    c->pp = make_phys(*p);
    int rc;
    auto bail = [&](int code) {
        free_all(c);
        delete c;
        return code;
    };
    if (hipStreamCreateWithFlags(&c->stream, hipStreamNonBlocking) != hipSuccess)
        return bail(fail(LAPS_EDEVICE, "hipStreamCreate failed"));
    std::vector<int> kzlim;
    if ((rc = compute_kept_box(c, kzlim))) return bail(rc);
    if ((rc = upload_tables(c, c->full, false, {}, c->tfull))) return bail(rc);
    if ((rc = upload_tables(c, c->kept, p->dealias_option == 1 || p->dealias_option == 3, kzlim, c->tkept)))
        return bail(rc);
    // twiddle tables W_n^t for the three axis lengths, FP64 and FP32
    const int lens[3] = {c->nx, c->ny, c->nz};
    for (int a = 0; a < 3; ++a) {
        const int n = lens[a];
        std::vector<cpx<double>> d(n);
        std::vector<cpx<float>> f(n);
        for (int t = 0; t < n; ++t) {
            root(t, n, d[t].x, d[t].y);
            f[t].x = (float)d[t].x;
            f[t].y = (float)d[t].y;
        }
        if ((rc = c->allocn(&c->twd[a], n)) || (rc = c->allocn(&c->twf[a], n))) return bail(rc);
        if (hipMemcpy(c->twd[a], d.data(), n * sizeof(cpx<double>), hipMemcpyHostToDevice) != hipSuccess ||
            hipMemcpy(c->twf[a], f.data(), n * sizeof(cpx<float>), hipMemcpyHostToDevice) != hipSuccess)
            return bail(fail(LAPS_EDEVICE, "twiddle upload failed"));
    }
    const long long KB = c->kb();
    const long long NX = c->nx, NY = c->ny, NZ = c->nz;
    const Box& k = c->kept;
    setup_forward_groups(c);
    const int nfi = c->nf_in(), nfo = c->nx_slots(), nd = c->nd();
    long long p1 = std::max({(long long)nfi * NZ * k.CY * k.KXP, (long long)nfo * NZ * NY * k.KXP,
                             3LL * NZ * NY * c->nxh});
    long long p2 = std::max({(long long)nfi * NZ * NY * k.KXP, (long long)nd * NZ * k.CY * k.KXP,
                             3LL * NZ * NY * c->nxh});
    const bool shift = p->dealias_option == 3;
    if (shift) {  // the shifted first substage inverts the full spectrum (11 fields) through P1 and P3
        p1 = std::max(p1, (long long)nfi * NZ * NY * c->full.KXP);
        p2 = std::max(p2, (long long)nfi * NZ * NY * c->full.KXP);
    }
    const size_t ts = c->mixed ? sizeof(float) : sizeof(double);
    // phase-shift dealiasing runs the plain and the shifted grid as two chains of one launch
    // per pass: P1 and P2 hold both, chain 1 at + p1 and + p2 (P3 = P2 + p2)
    // (chain 1 starts 5 KiB past a whole number of 64 KiB, so that the two chains' rows at the
    // same offset do not fall on the same HBM channels)
    auto chain_pad = [&](long long e) {
        const long long unit = 65536 / (2 * (long long)ts), pad = 5120 / (2 * (long long)ts);
        return (e + unit - 1) / unit * unit + pad;
    };
    p1 = chain_pad(p1);
    p2 = chain_pad(p2);
    c->p1 = p1;
    c->p2 = p2;
    const int nchain = shift ? 2 : 1;
    // FP64 single-field scratch: a full spectrum, or one kept-box field inverted along z and y
    const size_t xs = (size_t)std::max(c->M, NZ * NY * (long long)k.KXP);
    (void)NX;
    if ((rc = c->allocn(&c->ctl, 1)) || (rc = c->allocn(&c->U, 11 * KB)) || (rc = c->allocn(&c->Ufull, 11 * c->M)) ||
        (rc = c->allocn(&c->V, 8 * KB)) || (rc = c->allocn(&c->S, 12 * c->N)) ||
        (rc = c->alloc(&c->P1, nchain * p1 * 2 * ts)) || (rc = c->alloc(&c->P2, nchain * p2 * 2 * ts)) ||
        (rc = c->allocn(&c->X1, xs)) || (rc = c->allocn(&c->X2, xs)) || (rc = c->allocn(&c->Xr, c->N)) ||
        (rc = c->allocn(&c->red, (size_t)c->nblk_red * 16)) || (rc = c->allocn(&c->dave, 8)) ||
        (rc = c->allocn(&c->dbits, 1)) || (c->mixed && (rc = c->allocn(&c->Uf, 11 * KB))))
        return bail(rc);
    if (c->Uf && hipMemset(c->Uf, 0, 11 * KB * sizeof(cpx<float>)) != hipSuccess)
        return bail(fail(LAPS_EDEVICE, "clearing the FP32 state copy failed"));
    if (shift) {
        // half a cell along every axis: e^{i k delta} = e^{i pi m/n}, signed m with the +Nyquist
        // convention of the wave numbers
        // (pruned: entry i is stored row i of an axis kept as cnt rows, 0..(cnt-1)/2 and then the
        // negative modes up to n - 1)
        auto table = [&](cpx<double>** dst, int n, int cnt, bool pruned) -> int {
            std::vector<cpx<double>> h(cnt);
            for (int i = 0; i < cnt; ++i) {
                const int m = signed_index(pruned && i > (cnt - 1) / 2 ? n - (cnt - i) : i, n);
                h[i].x = cos(kPiRef * m / n);
                h[i].y = sin(kPiRef * m / n);
            }
            int r = c->allocn(dst, cnt);
            if (r) return r;
            if (hipMemcpy(*dst, h.data(), cnt * sizeof(cpx<double>), hipMemcpyHostToDevice) != hipSuccess)
                return fail(LAPS_EDEVICE, "phase table upload failed");
            return LAPS_OK;
        };
        c->P3 = (char*)c->P2 + p2 * 2 * ts;
        if ((rc = table(&c->phx, c->nx, c->nxh, false)) ||
            (rc = table(&c->phy, c->ny, c->ny, false)) || (rc = table(&c->phz, c->nz, c->nz, false)) ||
            (rc = table(&c->phyk, c->ny, k.CY, true)))
            return bail(rc);
    }
    if ((rc = reset_ctl(c, 0.0, 0.0, false))) return bail(rc);
    *out = c;
    return LAPS_OK;
}

void laps_destroy(laps_ctx* c) {
    if (!c) return;
    (void)hipSetDevice(c->p.device);
    if (c->stream) (void)hipStreamSynchronize(c->stream);
    free_all(c);
    delete c;
}

int laps_set_state(laps_ctx* c, const double* uu, const double* uu_prim) {
    int rc = check_ctx(c, false);
    if (rc) return rc;
    if (!uu || !uu_prim) return fail(LAPS_EINVAL, "null state pointer");
    LAPS_CK(hipStreamSynchronize(c->stream));
    if ((rc = wait_stage(c, true))) return rc;
    LAPS_CK(c->to_device(c->S, uu, 8 * c->N * sizeof(double)));
    LAPS_CK(c->to_device(c->S + 8 * c->N, uu_prim, 4 * c->N * sizeof(double)));
    {
        // as many fields to a launch as P1 holds in FP64 (P1 is free between steps), the result in place
        // in Ufull
        TimingOff off(c);
        const int nf = p1_fields(c, c->M);
        for (int f = 0; f < 8; f += nf)
            if ((rc = fwd_pipeline<double>(c, c->S + f * c->N, std::min(nf, 8 - f), c->full, c->Ufull + f * c->M,
                                           (cpx<double>*)c->P1)))
                return rc;
    }
    LAPS_CK(hipMemsetAsync(c->U, 0, 11 * c->kb() * sizeof(cpx<double>), c->stream));
    LAPS_CK(launch_gather_box(c->Ufull, c->U, 8, c->M, c->kb(), c->nxh, c->ny, c->nz, c->kept, c->stream));
    if (c->Uf)
        LAPS_CK(launch_convert<double, float>((const double*)c->U, (float*)c->Uf, 2 * 8 * c->kb(), c->stream));
    if ((rc = reset_ctl(c, 0.0, 0.0, false))) return rc;
    LAPS_CK(hipStreamSynchronize(c->stream));
    c->have_state = true;
    c->fresh = true;
    c->materialized = true;
    c->stepped_since_set = false;
    ++c->gen;
    return LAPS_OK;
}

int laps_set_time(laps_ctx* c, double time, double dt_prev) {
    int rc = check_ctx(c, false);
    if (rc) return rc;
    Ctl h;
    if ((rc = read_ctl(c, h))) return rc;
    h.time = time;
    h.dt_prev = dt_prev;
    h.radius = c->pp.radius0 + c->pp.Ur * time;
    h.tau = h.radius / c->pp.Ur;
    h.r0r = c->pp.radius0 / h.radius;
    h.ksq_updated = 1;  // evolve_radius calls update_ksquare (AEBmod.f90:70)
    LAPS_CK(hipMemcpy(c->ctl, &h, sizeof(Ctl), hipMemcpyHostToDevice));
    return LAPS_OK;
}

int laps_set_fixed_dt(laps_ctx* c, double dt) {
    int rc = check_ctx(c, false);
    if (rc) return rc;
    c->fixed_dt = dt > 0 ? dt : 0.0;
    c->pp.fixed_dt = c->fixed_dt;
    ++c->gen;
    return LAPS_OK;
}

int laps_step(laps_ctx* c, int nsteps) {
    int rc = check_ctx(c, true);
    if (rc) return rc;
    if (nsteps < 0) return fail(LAPS_EINVAL, "nsteps < 0");
    if (!c->tuned && nsteps > 0) {
        rc = c->mixed ? autotune<float>(c) : autotune<double>(c);
        if (rc) return rc;
    }
    for (int s = 0; s < nsteps; ++s) {
        rc = c->mixed ? one_step<float>(c) : one_step<double>(c);
        if (rc) return rc;
        c->stepped_since_set = true;
    }
    return LAPS_OK;
}

int laps_sync(laps_ctx* c) {
    int rc = check_ctx(c, false);
    if (rc) return rc;
    LAPS_CK(hipStreamSynchronize(c->stream));
    return LAPS_OK;
}

int laps_get_scalars(laps_ctx* c, double* time, double* dt, double* radius, int64_t* istep, int32_t* status) {
    int rc = check_ctx(c, false);
    if (rc) return rc;
    Ctl h;
    if ((rc = read_ctl(c, h))) return rc;
    if (time) *time = h.time;
    if (dt) *dt = h.status ? h.dt_prev : h.dt;
    if (radius) *radius = h.radius;
    if (istep) *istep = h.istep;
    if (status) *status = h.status;
    return LAPS_OK;
}

int laps_cfl(laps_ctx* c, double* dtmin_raw, double* dt_next) {
    int rc = check_ctx(c, true);
    if (rc) return rc;
    if ((rc = materialize(c))) return rc;
    LAPS_CK(launch_ctl_begin(c->ctl, c->stream));
    LAPS_CK(launch_cfl(c->S, c->S + 8 * c->N, c->N, c->pp, c->ctl, c->stream));
    Ctl h;
    if ((rc = read_ctl(c, h))) return rc;
    double raw;
    std::memcpy(&raw, &h.dtmin_bits, 8);
    double dt;
    if (c->fixed_dt > 0) {
        dt = c->fixed_dt;
    } else {
        const double dtmin = raw * c->p.cfl;
        dt = h.dt_prev;
        if (dt < 0.98 * dtmin || dt > 1.02 * dtmin) dt = dtmin;
    }
    if (dtmin_raw) *dtmin_raw = raw;
    if (dt_next) *dt_next = dt;
    return LAPS_OK;
}

int laps_get_state(laps_ctx* c, double* uu, double* uu_prim) {
    int rc = check_ctx(c, true);
    if (rc) return rc;
    if ((rc = materialize(c))) return rc;
    LAPS_CK(hipStreamSynchronize(c->stream));
    if (uu) LAPS_CK(c->to_host(uu, c->S, 8 * c->N * sizeof(double)));
    if (uu_prim) LAPS_CK(c->to_host(uu_prim, c->S + 8 * c->N, 4 * c->N * sizeof(double)));
    return LAPS_OK;
}

int laps_stage_output(laps_ctx* c, int primitive) {
    int rc = check_ctx(c, true);
    if (rc) return rc;
    if (!c->stage_host) {
        if (hipHostMalloc((void**)&c->stage_host, 8 * c->N * sizeof(double), hipHostMallocDefault) != hipSuccess) {
            c->stage_host = nullptr;
            return fail(LAPS_ENOMEM, "pinned output buffer allocation failed");
        }
        if (hipStreamCreateWithFlags(&c->stage_stream, hipStreamNonBlocking) != hipSuccess ||
            hipEventCreateWithFlags(&c->stage_ready, hipEventDisableTiming) != hipSuccess ||
            hipEventCreateWithFlags(&c->stage_done, hipEventDisableTiming) != hipSuccess)
            return fail(LAPS_EDEVICE, "output staging stream / events");
    }
    // the previous copy must have left the pinned buffer before this one overwrites it
    if ((rc = wait_stage(c, true))) return rc;
    if ((rc = materialize(c))) return rc;
    Ctl h;
    if ((rc = read_ctl(c, h))) return rc;   // the step scalars of this state (one small read)
    c->stage_time = h.time;
    c->stage_dt = h.dt;
    c->stage_istep = h.istep;
    // the payload of output_uu (mhdoutput.f90:87-117): rho, then rho u or u, B, then e or p,
    // field blocks of S = [uu(8), uu_prim(4)] copied straight into the pinned buffer
    LAPS_CK(hipEventRecord(c->stage_ready, c->stream));
    LAPS_CK(hipStreamWaitEvent(c->stage_stream, c->stage_ready, 0));
    const size_t fb = (size_t)c->N * sizeof(double);
    const double* S = c->S;
    double* H = c->stage_host;
    const long long N = c->N;
    LAPS_CK(hipMemcpyAsync(H, S, fb, hipMemcpyDeviceToHost, c->stage_stream));
    LAPS_CK(hipMemcpyAsync(H + N, primitive ? S + 8 * N : S + N, 3 * fb, hipMemcpyDeviceToHost, c->stage_stream));
    LAPS_CK(hipMemcpyAsync(H + 4 * N, S + 4 * N, 3 * fb, hipMemcpyDeviceToHost, c->stage_stream));
    LAPS_CK(hipMemcpyAsync(H + 7 * N, primitive ? S + 11 * N : S + 7 * N, fb, hipMemcpyDeviceToHost,
                           c->stage_stream));
    LAPS_CK(hipEventRecord(c->stage_done, c->stage_stream));
    c->stage_pending = true;
    return LAPS_OK;
}

int laps_staged_output(laps_ctx* c, const double** payload, double* time, double* dt, int64_t* istep) {
    int rc = check_ctx(c, false);
    if (rc) return rc;
    if (!payload) return fail(LAPS_EINVAL, "null output");
    if (!c->stage_pending) return fail(LAPS_ESTATE, "no output staged: call laps_stage_output first");
    LAPS_CK(hipEventSynchronize(c->stage_done));
    *payload = c->stage_host;
    if (time) *time = c->stage_time;
    if (dt) *dt = c->stage_dt;
    if (istep) *istep = c->stage_istep;
    return LAPS_OK;
}

int laps_get_spectral(laps_ctx* c, double* uhat) {
    int rc = check_ctx(c, true);
    if (rc) return rc;
    if (!uhat) return fail(LAPS_EINVAL, "null output");
    if ((rc = refresh_fresh(c))) return rc;
    LAPS_CK(hipStreamSynchronize(c->stream));
    if (c->fresh) {
        LAPS_CK(c->to_host(uhat, c->Ufull, 8 * c->M * sizeof(cpx<double>)));
        return LAPS_OK;
    }
    const Box& b = c->kept;
    const long long KB = c->kb();
    std::vector<cpx<double>> box((size_t)8 * KB);
    LAPS_CK(c->to_host(box.data(), c->U, box.size() * sizeof(cpx<double>)));
    cpx<double>* o = (cpx<double>*)uhat;
    std::memset(o, 0, 8 * c->M * sizeof(cpx<double>));
    for (int f = 0; f < 8; ++f)
        for (int cz = 0; cz < b.CZ; ++cz) {
            const int iz = (b.CZ == c->nz || cz <= (b.CZ - 1) / 2) ? cz : c->nz - (b.CZ - cz);
            for (int cy = 0; cy < b.CY; ++cy) {
                const int iy = (b.CY == c->ny || cy <= (b.CY - 1) / 2) ? cy : c->ny - (b.CY - cy);
                for (int kx = 0; kx < b.KX; ++kx)
                    o[f * c->M + ((long long)iz * c->ny + iy) * c->nxh + kx] =
                        box[f * KB + ((long long)cz * b.CY + cy) * b.KXP + kx];
            }
        }
    return LAPS_OK;
}

int laps_moments(laps_ctx* c, double ave[8], double var[8], double rho_u2[3]) {
    int rc = check_ctx(c, true);
    if (rc) return rc;
    if ((rc = materialize(c))) return rc;
    const int nb = c->nblk_red;
    LAPS_CK(launch_moments(c->S, c->S + 8 * c->N, c->N, c->red, nb, c->stream));
    std::vector<double> part((size_t)nb * 16);
    LAPS_CK(hipStreamSynchronize(c->stream));
    LAPS_CK(hipMemcpy(part.data(), c->red, part.size() * 8, hipMemcpyDeviceToHost));
    double s[16] = {0};
    for (int b = 0; b < nb; ++b)
        for (int k = 0; k < 16; ++k) s[k] += part[(size_t)b * 16 + k];
    double a[8];
    for (int k = 0; k < 8; ++k) {
        a[k] = s[k] / (double)c->N;
        const double sq = s[8 + k] / (double)c->N;
        if (ave) ave[k] = a[k];
        if (var) var[k] = sq - a[k] * a[k];
    }
    // second pass needs the means on the device
    LAPS_CK(hipMemcpy(c->dave, a, 8 * sizeof(double), hipMemcpyHostToDevice));
    LAPS_CK(launch_moments2(c->S, c->S + 8 * c->N, c->N, c->dave, c->red, nb, c->stream));
    const int nb2 = nb;
    std::vector<double> part2((size_t)nb2 * 3);
    LAPS_CK(hipStreamSynchronize(c->stream));
    LAPS_CK(hipMemcpy(part2.data(), c->red, part2.size() * 8, hipMemcpyDeviceToHost));
    double r[3] = {0, 0, 0};
    for (int b = 0; b < nb2; ++b)
        for (int k = 0; k < 3; ++k) r[k] += part2[(size_t)b * 3 + k];
    if (rho_u2)
        for (int k = 0; k < 3; ++k) rho_u2[k] = r[k] / (double)c->N;
    return LAPS_OK;
}

int laps_budgets(laps_ctx* c, double out[LAPS_NBUDGET]) {
    int rc = check_ctx(c, true);
    if (rc) return rc;
    if (!out) return fail(LAPS_EINVAL, "null output");
    if ((rc = materialize(c))) return rc;
    const int nb = c->nblk_red;
    LAPS_CK(launch_budget_real(c->S, c->S + 8 * c->N, c->N, c->p.adiabatic_index, c->red, nb, c->stream));
    std::vector<double> part((size_t)nb * 5);
    LAPS_CK(hipStreamSynchronize(c->stream));
    LAPS_CK(hipMemcpy(part.data(), c->red, part.size() * 8, hipMemcpyDeviceToHost));
    double r[5] = {0, 0, 0, 0, 0};
    for (int b = 0; b < nb; ++b)
        for (int k = 0; k < 5; ++k) r[k] += part[(size_t)b * 5 + k];
    for (int k = 0; k < 5; ++k) out[k] = r[k] / (double)c->N;
    if ((rc = refresh_fresh(c))) return rc;
    if (c->fresh)
        LAPS_CK(launch_budget_spec(c->Ufull, c->M, c->full, c->tfull.view(), c->pp, c->ctl, c->nx, c->red, nb,
                                   c->stream));
    else
        LAPS_CK(launch_budget_spec(c->U, c->kb(), c->kept, c->tkept.view(), c->pp, c->ctl, c->nx, c->red, nb,
                                   c->stream));
    std::vector<double> part2((size_t)nb * 2);
    LAPS_CK(hipStreamSynchronize(c->stream));
    LAPS_CK(hipMemcpy(part2.data(), c->red, part2.size() * 8, hipMemcpyDeviceToHost));
    double h[2] = {0, 0};
    for (int b = 0; b < nb; ++b)
        for (int k = 0; k < 2; ++k) h[k] += part2[(size_t)b * 2 + k];
    out[5] = h[0];
    out[6] = h[1];
    return LAPS_OK;
}

int laps_max_divb(laps_ctx* c, double* out) {
    int rc = check_ctx(c, true);
    if (rc) return rc;
    if (!out) return fail(LAPS_EINVAL, "null output");
    if ((rc = refresh_fresh(c))) return rc;
    const unsigned long long zero = 0;
    LAPS_CK(hipMemcpyAsync(c->dbits, &zero, 8, hipMemcpyHostToDevice, c->stream));
    if (c->fresh)
        LAPS_CK(launch_divb(c->Ufull, c->M, c->full, c->tfull.view(), c->pp, c->ctl, c->dbits, c->stream));
    else
        LAPS_CK(launch_divb(c->U, c->kb(), c->kept, c->tkept.view(), c->pp, c->ctl, c->dbits, c->stream));
    unsigned long long bits = 0;
    LAPS_CK(hipStreamSynchronize(c->stream));
    LAPS_CK(hipMemcpy(&bits, c->dbits, 8, hipMemcpyDeviceToHost));
    std::memcpy(out, &bits, 8);
    return LAPS_OK;
}

int laps_fft_r2c(laps_ctx* c, int nf, const double* real_in, double* spec_out) {
    int rc = check_ctx(c, false);
    if (rc) return rc;
    if (nf < 0 || (nf > 0 && (!real_in || !spec_out))) return fail(LAPS_EINVAL, "bad arguments");
    LAPS_CK(hipStreamSynchronize(c->stream));
    for (int f = 0; f < nf; ++f) {
        LAPS_CK(c->to_device(c->Xr, real_in + (size_t)f * c->N, c->N * 8));
        if ((rc = fwd_fp64(c, c->Xr, c->X1))) return rc;
        LAPS_CK(hipStreamSynchronize(c->stream));
        LAPS_CK(c->to_host(spec_out + (size_t)f * 2 * c->M, c->X1, c->M * 16));
    }
    return LAPS_OK;
}

int laps_fft_c2r(laps_ctx* c, int nf, const double* spec_in, double* real_out) {
    int rc = check_ctx(c, false);
    if (rc) return rc;
    if (nf < 0 || (nf > 0 && (!spec_in || !real_out))) return fail(LAPS_EINVAL, "bad arguments");
    LAPS_CK(hipStreamSynchronize(c->stream));
    for (int f = 0; f < nf; ++f) {
        LAPS_CK(c->to_device(c->X2, spec_in + (size_t)f * 2 * c->M, c->M * 16));
        if ((rc = inv_fp64(c, c->X2, c->full, c->Xr))) return rc;
        LAPS_CK(hipStreamSynchronize(c->stream));
        LAPS_CK(c->to_host(real_out + (size_t)f * c->N, c->Xr, c->N * 8));
    }
    return LAPS_OK;
}

int laps_timing_enable(laps_ctx* c, int enable) {
    int rc = check_ctx(c, false);
    if (rc) return rc;
    if ((rc = collect_timing(c))) return rc;
    for (int k = 0; k < K_NCLASS; ++k) {
        c->timing.ms[k] = 0.0;
        c->timing.bytes[k] = 0.0;
        c->timing.launches[k] = 0;
    }
    c->timing.on = enable != 0;
    return LAPS_OK;
}

int laps_timing_read(laps_ctx* c, int index, const char** name, double* total_ms, double* total_bytes,
                     int64_t* launches) {
    int rc = check_ctx(c, false);
    if (rc) return rc;
    if ((rc = collect_timing(c))) return rc;
    if (index < 0 || index >= K_NCLASS) {
        if (name) *name = nullptr;
        return LAPS_OK;
    }
    if (name) *name = kClassNames[index];
    if (total_ms) *total_ms = c->timing.ms[index];
    if (total_bytes) *total_bytes = c->timing.bytes[index];
    if (launches) *launches = c->timing.launches[index];
    return LAPS_OK;
}

int laps_get_stream(laps_ctx* c, void** stream) {
    int rc = check_ctx(c, false);
    if (rc) return rc;
    if (!stream) return fail(LAPS_EINVAL, "null output");
    *stream = (void*)c->stream;
    return LAPS_OK;
}

// ------------------------------------------------------------------ ensemble
//
// Independent boxes (each a full context with its own stream, buffers and
// device-side dt) advanced together. The first step after a state upload runs
// eagerly per box; after that one step of every box is captured once as a
// hipGraph, the boxes as parallel branches forked from and joined into the
// ensemble's own stream, and each further step is one launch of that graph.
// A box whose launches change (new state, fixed dt) makes the next
// laps_ens_step capture again.
struct laps_ens {
    std::vector<laps_ctx*> box;
    // launch groups: boxes with identical parameters, whose step buffers (U, Uf, V, P1, P2 and
    // the control block) sit at a fixed stride in pools of the ensemble, so that one launch per
    // kernel steps the whole group; group[g][0] is the box whose context issues the launches
    std::vector<std::vector<int>> group;
    std::vector<laps_ctx::Batch> gbatch;
    std::vector<void*> pools;
    std::vector<uint64_t> gen;         // box generations the graph was captured at
    int device = 0;
    hipStream_t origin = nullptr;
    hipEvent_t fork = nullptr, after = nullptr;  // capture fork; order after launches
    std::vector<hipEvent_t> join, before;        // capture joins; order before launches
    // graphs of 1 and of kEnsMulti steps: a launch of the latter advances every box by kEnsMulti
    // steps (each box's dt and time live on the device, so the steps need no host work between)
    hipGraph_t graph[2] = {nullptr, nullptr};
    hipGraphExec_t exec[2] = {nullptr, nullptr};
};
constexpr int kEnsMulti = 8;

static void ens_drop_graph(laps_ens* e) {
    for (int g = 0; g < 2; ++g) {
        if (e->exec[g]) (void)hipGraphExecDestroy(e->exec[g]);
        if (e->graph[g]) (void)hipGraphDestroy(e->graph[g]);
        e->exec[g] = nullptr;
        e->graph[g] = nullptr;
    }
}

// captures graph `which` (0: one step, 1: kEnsMulti steps) of every box
static int ens_capture(laps_ens* e, int which) {
    const int nst = which ? kEnsMulti : 1;
    for (laps_ctx* c : e->box)
        if (c->closure) return fail(LAPS_EINVAL, "ensemble boxes with a learned closure are stepped per box");
    for (laps_ctx* c : e->box) c->timing.on = false;
    LAPS_CK(hipStreamBeginCapture(e->origin, hipStreamCaptureModeThreadLocal));
    int rc = LAPS_OK;
    hipError_t he = hipEventRecord(e->fork, e->origin);
    for (size_t g = 0; g < e->group.size() && he == hipSuccess && rc == LAPS_OK; ++g) {
        // a group whose boxes launch alike (same plans, same dt mode) is stepped by batched
        // launches of its first box; otherwise each box is a branch of its own
        const std::vector<int>& idx = e->group[g];
        laps_ctx* c0 = e->box[idx[0]];
        bool alike = idx.size() > 1;
        for (int i : idx) {
            const laps_ctx* c = e->box[i];
            alike = alike && c->plan_zinv == c0->plan_zinv && c->plan_yinv == c0->plan_yinv &&
                    c->fixed_dt == c0->fixed_dt && !c->fresh;
        }
        for (size_t m = 0; m < (alike ? 1 : idx.size()) && he == hipSuccess && rc == LAPS_OK; ++m) {
            const int i = idx[m];
            laps_ctx* c = e->box[i];
            he = hipStreamWaitEvent(c->stream, e->fork, 0);
            if (he != hipSuccess) break;
            if (alike) c->batch = e->gbatch[g];
            for (int st = 0; st < nst && rc == LAPS_OK; ++st)
                rc = c->mixed ? one_step<float>(c) : one_step<double>(c);
            c->batch = laps_ctx::Batch{};
            if (rc) break;
            he = hipEventRecord(e->join[i], c->stream);
            if (he == hipSuccess) he = hipStreamWaitEvent(e->origin, e->join[i], 0);
        }
    }
    hipGraph_t g = nullptr;
    const hipError_t he2 = hipStreamEndCapture(e->origin, &g);
    if (rc || he != hipSuccess || he2 != hipSuccess) {
        if (g) (void)hipGraphDestroy(g);
        if (rc) return rc;
        return fail(LAPS_EDEVICE, std::string("ensemble graph capture: ") +
                                      hipGetErrorString(he != hipSuccess ? he : he2));
    }
    e->graph[which] = g;
    LAPS_CK(hipGraphInstantiate(&e->exec[which], e->graph[which], nullptr, nullptr, 0));
    return LAPS_OK;
}

// Groups the boxes of identical parameters and moves each group's step buffers into pools of
// the ensemble, box m of a group at m times a fixed stride, so that a launch of the group's
// first box with grid rows for the boxes steps them all. The boxes have no state yet: nothing
// is copied. Each box remains a full context of its own (per-box calls use its pointers).
static int ens_make_groups(laps_ens* e) {
    const int nbox = (int)e->box.size();
    std::vector<bool> taken(nbox, false);
    auto round256 = [](size_t b) { return (b + 255) / 256 * 256; };
    for (int i = 0; i < nbox; ++i) {
        if (taken[i]) continue;
        std::vector<int> idx{i};
        taken[i] = true;
        for (int j = i + 1; j < nbox; ++j)
            if (!taken[j] && std::memcmp(&e->box[i]->p, &e->box[j]->p, sizeof(laps_params)) == 0) {
                idx.push_back(j);
                taken[j] = true;
            }
        e->group.push_back(idx);
        e->gbatch.push_back(laps_ctx::Batch{});
        const int G = (int)idx.size();
        if (G < 2) continue;
        laps_ctx* c0 = e->box[i];
        const long long KB = c0->kb();
        const size_t ts = c0->mixed ? sizeof(float) : sizeof(double);
        const long long nchain = c0->p.dealias_option == 3 ? 2 : 1;
        const size_t bu = round256(11 * KB * sizeof(cpx<double>));
        const size_t buf = c0->Uf ? round256(11 * KB * sizeof(cpx<float>)) : 0;
        const size_t bv = round256(8 * KB * sizeof(cpx<double>));
        const size_t bp1 = round256(nchain * c0->p1 * 2 * ts), bp2 = round256(nchain * c0->p2 * 2 * ts);
        const size_t bctl = sizeof(Ctl);
        void *pu = nullptr, *puf = nullptr, *pv = nullptr, *pp1 = nullptr, *pp2 = nullptr, *pctl = nullptr;
        auto pool = [&](void** q, size_t bytes) -> int {
            if (bytes == 0) return LAPS_OK;
            const hipError_t he = hipMalloc(q, bytes * G);
            if (he != hipSuccess) {
                *q = nullptr;
                return fail(LAPS_ENOMEM, "ensemble pool allocation failed");
            }
            e->pools.push_back(*q);
            return LAPS_OK;
        };
        int rc;
        if ((rc = pool(&pu, bu)) || (rc = pool(&puf, buf)) || (rc = pool(&pv, bv)) || (rc = pool(&pp1, bp1)) ||
            (rc = pool(&pp2, bp2)) || (rc = pool(&pctl, bctl)))
            return rc;
        if (puf && hipMemset(puf, 0, buf * G) != hipSuccess) return fail(LAPS_EDEVICE, "clearing a pool failed");
        for (int m = 0; m < G; ++m) {
            laps_ctx* c = e->box[idx[m]];
            auto move = [&](void* old, void* fresh) {
                for (auto it = c->allocs.begin(); it != c->allocs.end(); ++it)
                    if (*it == old) {
                        (void)hipFree(old);
                        c->allocs.erase(it);
                        break;
                    }
                return fresh;
            };
            c->U = (cpx<double>*)move(c->U, (char*)pu + m * bu);
            if (c->Uf) c->Uf = (cpx<float>*)move(c->Uf, (char*)puf + m * buf);
            c->V = (cpx<double>*)move(c->V, (char*)pv + m * bv);
            c->P1 = move(c->P1, (char*)pp1 + m * bp1);
            c->P2 = move(c->P2, (char*)pp2 + m * bp2);
            if (c->P3) c->P3 = (char*)c->P2 + c->p2 * 2 * ts;
            c->ctl = (Ctl*)move(c->ctl, (char*)pctl + m * bctl);
            if ((rc = reset_ctl(c, 0.0, 0.0, false))) return rc;
        }
        laps_ctx::Batch& b = e->gbatch.back();
        b.n = G;
        b.u = (long long)(bu / sizeof(cpx<double>));
        b.uf = (long long)(buf / sizeof(cpx<float>));
        b.v = (long long)(bv / sizeof(cpx<double>));
        b.p1 = (long long)(bp1 / (2 * ts));
        b.p2 = (long long)(bp2 / (2 * ts));
    }
    return LAPS_OK;
}

int laps_ens_create(int nbox, const laps_params* params, laps_ens** out) {
    if (!out) return fail(LAPS_EINVAL, "null output");
    *out = nullptr;
    if (nbox <= 0 || !params) return fail(LAPS_EINVAL, "an ensemble needs nbox >= 1 parameter sets");
    for (int i = 1; i < nbox; ++i)
        if (params[i].device != params[0].device) return fail(LAPS_EINVAL, "ensemble boxes must share one device");
    laps_ens* e = new laps_ens();
    e->device = params[0].device;
    auto bail = [&](int rc) {
        laps_ens_destroy(e);
        return rc;
    };
    for (int i = 0; i < nbox; ++i) {
        laps_ctx* c = nullptr;
        int rc = laps_create(&params[i], &c);
        if (rc) return bail(rc);
        e->box.push_back(c);
    }
    e->gen.assign(nbox, ~0ull);
    {
        const int rc = ens_make_groups(e);
        if (rc) return bail(rc);
    }
    if (hipSetDevice(e->device) != hipSuccess || hipStreamCreateWithFlags(&e->origin, hipStreamNonBlocking) != hipSuccess ||
        hipEventCreateWithFlags(&e->fork, hipEventDisableTiming) != hipSuccess ||
        hipEventCreateWithFlags(&e->after, hipEventDisableTiming) != hipSuccess)
        return bail(fail(LAPS_EDEVICE, "ensemble stream/event creation failed"));
    e->join.assign(nbox, nullptr);
    e->before.assign(nbox, nullptr);
    for (int i = 0; i < nbox; ++i)
        if (hipEventCreateWithFlags(&e->join[i], hipEventDisableTiming) != hipSuccess ||
            hipEventCreateWithFlags(&e->before[i], hipEventDisableTiming) != hipSuccess)
            return bail(fail(LAPS_EDEVICE, "ensemble event creation failed"));
    *out = e;
    return LAPS_OK;
}

void laps_ens_destroy(laps_ens* e) {
    if (!e) return;
    (void)hipSetDevice(e->device);
    if (e->origin) (void)hipStreamSynchronize(e->origin);
    ens_drop_graph(e);
    for (hipEvent_t v : e->join)
        if (v) (void)hipEventDestroy(v);
    for (hipEvent_t v : e->before)
        if (v) (void)hipEventDestroy(v);
    if (e->fork) (void)hipEventDestroy(e->fork);
    if (e->after) (void)hipEventDestroy(e->after);
    if (e->origin) (void)hipStreamDestroy(e->origin);
    for (laps_ctx* c : e->box) laps_destroy(c);
    for (void* q : e->pools) (void)hipFree(q);  // the boxes' step buffers (no longer theirs to free)
    delete e;
}

int laps_ens_size(const laps_ens* e) { return e ? (int)e->box.size() : 0; }

int laps_ens_groups(const laps_ens* e) { return e ? (int)e->group.size() : 0; }

laps_ctx* laps_ens_box(laps_ens* e, int i) {
    if (!e || i < 0 || i >= (int)e->box.size()) return nullptr;
    return e->box[i];
}

int laps_ens_step(laps_ens* e, int nsteps) {
    if (!e) return fail(LAPS_EINVAL, "null ensemble");
    if (nsteps < 0) return fail(LAPS_EINVAL, "nsteps < 0");
    if (nsteps == 0) return LAPS_OK;
    LAPS_CK(hipSetDevice(e->device));
    for (laps_ctx* c : e->box)
        if (!c->have_state) return fail(LAPS_ESTATE, "ensemble box without state: call laps_set_state first");
    // the first step after an upload (and the plan autotune) runs eagerly, for every box alike
    bool eager = false;
    for (laps_ctx* c : e->box) eager = eager || c->fresh || !c->tuned;
    int rc;
    if (eager) {
        // the boxes of a group take the FFT plans of its first box, so that their launches
        // can be batched
        for (const std::vector<int>& idx : e->group) {
            laps_ctx* c0 = e->box[idx[0]];
            for (size_t m = 0; m < idx.size(); ++m) {
                laps_ctx* c = e->box[idx[m]];
                if (m > 0 && c0->tuned && !c->tuned) {
                    c->plan_zinv = c0->plan_zinv;
                    c->plan_yinv = c0->plan_yinv;
                    c->tuned = true;
                }
                if ((rc = laps_step(c, 1))) return rc;
            }
        }
        if (--nsteps == 0) return LAPS_OK;
    }
    bool stale = false;
    for (size_t i = 0; i < e->box.size(); ++i) stale = stale || e->gen[i] != e->box[i]->gen;
    if (stale) ens_drop_graph(e);
    // the graph's branches start after all work already queued on the box streams
    for (size_t i = 0; i < e->box.size(); ++i) {
        LAPS_CK(hipEventRecord(e->before[i], e->box[i]->stream));
        LAPS_CK(hipStreamWaitEvent(e->origin, e->before[i], 0));
    }
    const int nmulti = nsteps / kEnsMulti, nsingle = nsteps % kEnsMulti;
    for (int which = 0; which < 2; ++which) {
        if (e->exec[which] || (which ? nmulti : nsingle) == 0) continue;
        // capturing records the steps without running them; their launches are the graph's
        std::vector<bool> timing(e->box.size());
        for (size_t i = 0; i < e->box.size(); ++i) timing[i] = e->box[i]->timing.on;
        rc = ens_capture(e, which);
        for (size_t i = 0; i < e->box.size(); ++i) e->box[i]->timing.on = timing[i];
        if (rc) return rc;
    }
    for (size_t i = 0; i < e->box.size(); ++i) e->gen[i] = e->box[i]->gen;
    for (int s = 0; s < nmulti; ++s) LAPS_CK(hipGraphLaunch(e->exec[1], e->origin));
    for (int s = 0; s < nsingle; ++s) LAPS_CK(hipGraphLaunch(e->exec[0], e->origin));
    LAPS_CK(hipEventRecord(e->after, e->origin));
    for (laps_ctx* c : e->box) {
        LAPS_CK(hipStreamWaitEvent(c->stream, e->after, 0));
        c->stepped_since_set = true;
        c->fresh = false;
        c->materialized = false;
    }
    return LAPS_OK;
}

int laps_ens_sync(laps_ens* e) {
    if (!e) return fail(LAPS_EINVAL, "null ensemble");
    LAPS_CK(hipSetDevice(e->device));
    LAPS_CK(hipStreamSynchronize(e->origin));
    for (laps_ctx* c : e->box) LAPS_CK(hipStreamSynchronize(c->stream));
    return LAPS_OK;
}

// ------------------------------------------------------------------ learned closure

int laps_closure_set(laps_ctx* c, const float* params, int nparams) {
    int rc = check_ctx(c, false);
    if (rc) return rc;
    if (!params) {
        c->closure = false;
        ++c->gen;
        return LAPS_OK;
    }
    if (nparams != LAPS_CLOSURE_NPARAM) return fail(LAPS_EINVAL, "closure parameter vector has the wrong length");
    if (c->p.if_aeb) return fail(LAPS_EINVAL, "the learned closure is defined for the periodic box without AEB");
    if ((rc = closure_buffers(c))) return rc;
    LAPS_CK(hipStreamSynchronize(c->stream));
    LAPS_CK(hipMemcpy(c->cl_P, params, (size_t)nparams * sizeof(float), hipMemcpyHostToDevice));
    c->closure = true;
    ++c->gen;
    return LAPS_OK;
}

int laps_closure_features(laps_ctx* c, float* out) {
    int rc = check_ctx(c, true);
    if (rc) return rc;
    if (!out) return fail(LAPS_EINVAL, "null output");
    if ((rc = closure_buffers(c))) return rc;
    if ((rc = closure_features(c, c->cl_id))) return rc;
    LAPS_CK(hipStreamSynchronize(c->stream));
    LAPS_CK(c->to_host(out, c->cl_X, (size_t)c->N * kClIn * sizeof(float)));
    return LAPS_OK;
}

int laps_closure_filter(laps_ctx* c, int r, double* out) {
    int rc = check_ctx(c, true);
    if (rc) return rc;
    if (!out) return fail(LAPS_EINVAL, "null output");
    if (r < 1 || c->nx % r || c->ny % r || c->nz % r) return fail(LAPS_EINVAL, "the filter width must divide the grid");
    if ((rc = materialize(c))) return rc;
    // J = curl B of the current state in real space: the spectral curl (the Hall-current slots of
    // the state buffer, which every substage rewrites) and three FP64 inverse transforms
    const bool fr = c->fresh;
    cpx<double>* src = fr ? c->Ufull : c->U;
    const Box& b = fr ? c->full : c->kept;
    const long long fs = fr ? c->M : c->kb();
    const long long Nc = (c->N / r / r) / r;
    double *J = nullptr, *O = nullptr;
    if (hipMalloc(&J, 3 * c->N * sizeof(double)) != hipSuccess) return fail(LAPS_ENOMEM, "current buffer");
    if (hipMalloc(&O, kClFilt * Nc * sizeof(double)) != hipSuccess) {
        (void)hipFree(J);
        return fail(LAPS_ENOMEM, "filter output buffer");
    }
    auto done = [&](int code) {
        (void)hipStreamSynchronize(c->stream);
        (void)hipFree(J);
        (void)hipFree(O);
        return code;
    };
    hipError_t he = launch_curl(src, src + 8 * fs, fs, b, (fr ? c->tfull : c->tkept).view(), c->pp, c->ctl, c->stream);
    if (he != hipSuccess) return done(fail(LAPS_EDEVICE, hipGetErrorString(he)));
    for (int a = 0; a < 3; ++a)
        if ((rc = inv_fp64(c, src + (8 + a) * fs, b, J + a * c->N))) return done(rc);
    he = launch_cl_filter(c->S, J, c->nx, c->ny, c->nz, r, c->p.if_hall ? c->p.ion_inertial_length : 0.0, O,
                          c->stream);
    if (he == hipSuccess) he = hipStreamSynchronize(c->stream);
    if (he == hipSuccess) he = c->to_host(out, O, kClFilt * Nc * sizeof(double));
    if (he != hipSuccess) return done(fail(LAPS_EDEVICE, hipGetErrorString(he)));
    return done(LAPS_OK);
}

int laps_closure_filter_spectral(laps_ctx* c, laps_ctx* g, double* out) {
    int rc = check_ctx(c, true);
    if (rc) return rc;
    if (!g || !out) return fail(LAPS_EINVAL, "null coarse context or output");
    if (g->p.device != c->p.device) return fail(LAPS_EINVAL, "the two contexts must be on one device");
    if (g->nx > c->nx || g->ny > c->ny || g->nz > c->nz)
        return fail(LAPS_EINVAL, "the coarse grid must not be finer than the fine one");
    if ((rc = materialize(c))) return rc;
    const bool fr = c->fresh;
    cpx<double>* src = fr ? c->Ufull : c->U;
    const Box& b = fr ? c->full : c->kept;
    const long long fs = fr ? c->M : c->kb();
    const long long N = c->N, Nc = g->N, Mc = g->full.modes();
    const double di = c->p.if_hall ? c->p.ion_inertial_length : 0.0;
    // device buffers: one fine field and its spectrum, J, the filtered state (with its
    // primitives) and current on the fine grid, the 2 x 26 cut spectra, the coarse output
    std::vector<void*> bufs;
    auto get = [&](void** p, size_t bytes) -> int {
        if (hipMalloc(p, bytes) != hipSuccess) return fail(LAPS_ENOMEM, "spectral filter buffer");
        bufs.push_back(*p);
        return LAPS_OK;
    };
    double *X, *J, *Sb, *Jb, *O;
    cpx<double>*Fs, *Cs, *Tc;
    auto done = [&](int code) {
        (void)hipStreamSynchronize(c->stream);
        (void)hipStreamSynchronize(g->stream);
        for (void* p : bufs) (void)hipFree(p);
        return code;
    };
    if ((rc = get((void**)&X, N * sizeof(double))) || (rc = get((void**)&J, 3 * N * sizeof(double))) ||
        (rc = get((void**)&Sb, 12 * N * sizeof(double))) || (rc = get((void**)&Jb, 3 * N * sizeof(double))) ||
        (rc = get((void**)&Fs, c->full.modes() * sizeof(cpx<double>))) ||
        (rc = get((void**)&Cs, 2 * kClFilt * Mc * sizeof(cpx<double>))) ||
        (rc = get((void**)&Tc, Mc * sizeof(cpx<double>))) || (rc = get((void**)&O, 2 * kClFilt * Nc * sizeof(double))))
        return done(rc);
    const int nyf = c->ny, nzf = c->nz, kxpf = c->full.KXP;
    auto cut = [&](cpx<double>* C) {
        return launch_spec_cut(Fs, nyf, nzf, kxpf, C, g->nx, g->ny, g->nz, g->full.KXP, +1, c->stream);
    };
    auto uncut = [&](const cpx<double>* C, double* real) -> int {
        LAPS_CK(hipMemsetAsync(Fs, 0, c->full.modes() * sizeof(cpx<double>), c->stream));
        LAPS_CK(launch_spec_cut(Fs, nyf, nzf, kxpf, (cpx<double>*)C, g->nx, g->ny, g->nz, g->full.KXP, -1, c->stream));
        return inv_fp64(c, Fs, c->full, real);
    };
    hipError_t he = launch_curl(src, src + 8 * fs, fs, b, (fr ? c->tfull : c->tkept).view(), c->pp, c->ctl, c->stream);
    if (he != hipSuccess) return done(fail(LAPS_EDEVICE, hipGetErrorString(he)));
    for (int a = 0; a < 3; ++a)
        if ((rc = inv_fp64(c, src + (8 + a) * fs, b, J + a * N))) return done(rc);
    // the cut of each field of the fine state: C[q]
    for (int q = 0; q < kClFilt; ++q) {
        if ((he = launch_cl_point(c->S, J, N, q, di, X, c->stream)) != hipSuccess) return done(fail(LAPS_EDEVICE, hipGetErrorString(he)));
        if ((rc = fwd_fp64(c, X, Fs))) return done(rc);
        if ((he = cut(Cs + q * Mc)) != hipSuccess) return done(fail(LAPS_EDEVICE, hipGetErrorString(he)));
    }
    // the cut state and current brought back to the fine grid (exact, zero-padded), the
    // primitives of the cut state (u = cut(m) / cut(rho)), and the same fields from them: D[q]
    for (int q = 0; q < 8; ++q)
        if ((rc = uncut(Cs + q * Mc, Sb + q * N))) return done(rc);
    LAPS_CK(launch_prim<double>(Sb, Sb + 8 * N, N, c->p.adiabatic_index, c->stream));
    for (int a = 0; a < 3; ++a) {
        if ((rc = fwd_fp64(c, J + a * N, Fs))) return done(rc);
        if ((he = cut(Tc)) != hipSuccess) return done(fail(LAPS_EDEVICE, hipGetErrorString(he)));
        if ((rc = uncut(Tc, Jb + a * N))) return done(rc);
    }
    cpx<double>* Ds = Cs + kClFilt * Mc;
    for (int q = 0; q < kClFilt; ++q) {
        if ((he = launch_cl_point(Sb, Jb, N, q, di, X, c->stream)) != hipSuccess) return done(fail(LAPS_EDEVICE, hipGetErrorString(he)));
        if ((rc = fwd_fp64(c, X, Fs))) return done(rc);
        if ((he = cut(Ds + q * Mc)) != hipSuccess) return done(fail(LAPS_EDEVICE, hipGetErrorString(he)));
    }
    // to the coarse grid's points with the coarse context's transforms
    LAPS_CK(hipStreamSynchronize(c->stream));
    for (int q = 0; q < 2 * kClFilt; ++q)
        if ((rc = inv_fp64(g, Cs + q * Mc, g->full, O + q * Nc))) return done(rc);
    he = hipStreamSynchronize(g->stream);
    if (he == hipSuccess) he = c->to_host(out, O, 2 * kClFilt * Nc * sizeof(double));
    if (he != hipSuccess) return done(fail(LAPS_EDEVICE, hipGetErrorString(he)));
    return done(LAPS_OK);
}

int laps_closure_eval(laps_ctx* c, float* out, double* rhs) {
    int rc = check_ctx(c, true);
    if (rc) return rc;
    if (!c->closure) return fail(LAPS_ESTATE, "no closure set: call laps_closure_set first");
    if ((rc = closure_step(c, true))) return rc;
    LAPS_CK(hipStreamSynchronize(c->stream));
    if (out) LAPS_CK(c->to_host(out, c->cl_Y, (size_t)c->N * kClOut * sizeof(float)));
    if (rhs) LAPS_CK(c->to_host(rhs, c->cl_full, (size_t)7 * c->M * sizeof(cpx<double>)));
    return LAPS_OK;
}

// Device buffers of the stateless network calls, freed on every path.
struct MlpBufs {
    std::vector<void*> ptrs;
    int get(float** p, size_t count) {
        void* q = nullptr;
        if (hipMalloc(&q, count * sizeof(float) + 16) != hipSuccess)
            return fail(LAPS_ENOMEM, "network buffer allocation failed");
        ptrs.push_back(q);
        *p = (float*)q;
        return LAPS_OK;
    }
    ~MlpBufs() {
        for (void* q : ptrs) (void)hipFree(q);
    }
};

int laps_mlp_forward(int device, int64_t n, const float* X, const float* params, float* Y) {
    if (n <= 0 || !X || !params || !Y) return fail(LAPS_EINVAL, "bad network arguments");
    LAPS_CK(hipSetDevice(device));
    MlpBufs b;
    float *dX, *dP, *dY;
    int rc;
    if ((rc = b.get(&dX, n * kClIn)) || (rc = b.get(&dP, kClNParam)) || (rc = b.get(&dY, n * kClOut))) return rc;
    LAPS_CK(hipMemcpy(dX, X, n * kClIn * sizeof(float), hipMemcpyHostToDevice));
    LAPS_CK(hipMemcpy(dP, params, kClNParam * sizeof(float), hipMemcpyHostToDevice));
    LAPS_CK(launch_mlp_fwd(dX, n, dP, dY, nullptr));
    LAPS_CK(hipDeviceSynchronize());
    LAPS_CK(hipMemcpy(Y, dY, n * kClOut * sizeof(float), hipMemcpyDeviceToHost));
    return LAPS_OK;
}

int laps_mlp_grad(int device, int64_t n, const float* X, const float* T, const float* params, float* grad,
                  float* loss) {
    if (n <= 0 || !X || !T || !params || !grad) return fail(LAPS_EINVAL, "bad network arguments");
    LAPS_CK(hipSetDevice(device));
    MlpBufs b;
    float *dX, *dT, *dP, *dS, *dG, *dL;
    int rc;
    if ((rc = b.get(&dX, n * kClIn)) || (rc = b.get(&dT, n * kClOut)) || (rc = b.get(&dP, kClNParam)) ||
        (rc = b.get(&dS, (size_t)mlp_part_rows(n) * kClPart)) || (rc = b.get(&dG, kClNParam)) || (rc = b.get(&dL, 1)))
        return rc;
    LAPS_CK(hipMemcpy(dX, X, n * kClIn * sizeof(float), hipMemcpyHostToDevice));
    LAPS_CK(hipMemcpy(dT, T, n * kClOut * sizeof(float), hipMemcpyHostToDevice));
    LAPS_CK(hipMemcpy(dP, params, kClNParam * sizeof(float), hipMemcpyHostToDevice));
    LAPS_CK(launch_mlp_grad(dX, dT, n, dP, dS, dG, dL, nullptr));
    LAPS_CK(hipDeviceSynchronize());
    LAPS_CK(hipMemcpy(grad, dG, kClNParam * sizeof(float), hipMemcpyDeviceToHost));
    if (loss) LAPS_CK(hipMemcpy(loss, dL, sizeof(float), hipMemcpyDeviceToHost));
    return LAPS_OK;
}

// ------------------------------------------------------------------ gradient without allocation
// laps_mlp_grad_noalloc keeps the partial sums of the gradient (one row per work-group, at most
// one work-group per CU for the sample counts it takes) in one file-scope device array, so a call
// allocates nothing. Each device holds its own copy of the array; its address
// is looked up once per device (hipGetSymbolAddress, with that device current) and only that
// address is passed to kernels. Every call on a device shares the array: calls that overlap on
// one device race.
constexpr long long kNoAllocRows = LAPS_MLP_NOALLOC_MAX / 32;
constexpr long long kNoAllocFloats = kNoAllocRows * kClPart;
static __device__ __align__(256) float scratch[kNoAllocFloats];
constexpr int kNoAllocDevices = 64;

static int scratch_address(int device, float** out) {
    static std::mutex mu;
    static float* addr[kNoAllocDevices] = {};
    if (device < 0 || device >= kNoAllocDevices) return fail(LAPS_EINVAL, "laps_mlp_grad_noalloc: bad device");
    std::lock_guard<std::mutex> lock(mu);
    if (!addr[device]) {
        void* p = nullptr;
        const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (e != hipSuccess || !p)
            return fail(LAPS_EDEVICE, std::string("laps_mlp_grad_noalloc: scratch address: ") + hipGetErrorString(e));
        addr[device] = (float*)p;
    }
    *out = addr[device];
    return LAPS_OK;
}

int laps_mlp_grad_noalloc(int device, int64_t n, const float* X, const float* T, const float* params,
                          float* grad, float* loss, void* stream) {
    if (n <= 0 || n > LAPS_MLP_NOALLOC_MAX)
        return fail(LAPS_EINVAL, "laps_mlp_grad_noalloc: n = " + std::to_string((long long)n) +
                                     " outside 1.." + std::to_string(LAPS_MLP_NOALLOC_MAX));
    if (!X || !T || !params || !grad) return fail(LAPS_EINVAL, "laps_mlp_grad_noalloc: null buffer");
    LAPS_CK(hipSetDevice(device));
    float* sc = nullptr;
    int rc;
    if ((rc = scratch_address(device, &sc))) return rc;
    const hipStream_t st = (hipStream_t)stream;
    if (mlp_part_rows(n) > kNoAllocRows) return fail(LAPS_EINVAL, "internal: partial sums exceed the fixed array");
    LAPS_CK(launch_mlp_grad(X, T, n, params, sc, grad, loss, st));
    return LAPS_OK;
}

int laps_mlp_train(int device, int64_t n, const float* X, const float* T, float* params, int steps, int batch,
                   float lr, float* loss_hist) {
    if (n <= 0 || !X || !T || !params || steps < 0 || batch <= 0) return fail(LAPS_EINVAL, "bad training arguments");
    if (batch > n) batch = (int)n;
    LAPS_CK(hipSetDevice(device));
    MlpBufs b;
    float *dX, *dT, *dP, *dS, *dM, *dV, *dL;
    int rc;
    if ((rc = b.get(&dX, n * kClIn)) || (rc = b.get(&dT, n * kClOut)) || (rc = b.get(&dP, kClNParam)) ||
        (rc = b.get(&dS, (size_t)mlp_part_rows(batch) * kClPart)) || (rc = b.get(&dM, kClNParam)) ||
        (rc = b.get(&dV, kClNParam)) || (rc = b.get(&dL, steps > 0 ? steps : 1)))
        return rc;
    LAPS_CK(hipMemcpy(dX, X, n * kClIn * sizeof(float), hipMemcpyHostToDevice));
    LAPS_CK(hipMemcpy(dT, T, n * kClOut * sizeof(float), hipMemcpyHostToDevice));
    LAPS_CK(hipMemcpy(dP, params, kClNParam * sizeof(float), hipMemcpyHostToDevice));
    std::vector<float> zero(kClNParam, 0.f);
    LAPS_CK(hipMemcpy(dM, zero.data(), kClNParam * sizeof(float), hipMemcpyHostToDevice));
    LAPS_CK(hipMemcpy(dV, zero.data(), kClNParam * sizeof(float), hipMemcpyHostToDevice));
    const long long nb = n / batch;  // whole batches, taken in turn (the caller shuffles the samples)
    double b1t = 1.0, b2t = 1.0;
    for (int s = 0; s < steps; ++s) {
        const long long off = (long long)(s % nb) * batch;
        const float* xb = dX + off * kClIn;
        const float* tb = dT + off * kClOut;
        b1t *= 0.9;
        b2t *= 0.999;
        LAPS_CK(launch_mlp_train_step(xb, tb, batch, dP, dS, dM, dV, dL + s, lr, (float)b1t, (float)b2t, nullptr));
    }
    LAPS_CK(hipDeviceSynchronize());
    LAPS_CK(hipMemcpy(params, dP, kClNParam * sizeof(float), hipMemcpyDeviceToHost));
    if (loss_hist && steps > 0) LAPS_CK(hipMemcpy(loss_hist, dL, steps * sizeof(float), hipMemcpyDeviceToHost));
    return LAPS_OK;
}

}  // extern "C"
