// fields.hip -- device kernels around the pressure solve: divergence of the
// staggered velocity (RHS of MG_MODE and the continuity error), the PCG
// coefficient beta = alpha dt / rho, the MG_MODE projection, and the FAST_MODE
// source and projection of the constant-coefficient splitting (reference
// density rho0, extrapolated old pressure 2 psi^n - psi^(n-1)).
//
// Staggered layout: ux, uz hold nx*ny*nz faces (face i between cells i and i+1,
// face 0 == face nx by periodicity); uy holds nx*(ny+1)*nz faces, j = 0..ny,
// with the walls at j = 0 and j = ny.
#include <algorithm>
#include <cstring>
#include <map>
#include <mutex>

#include "fields.hpp"

namespace tbfg {

// per-axis metrics: df[i-1] = df(i), dcn[i-1] = dc(i+1), i = 1..n
struct FieldGeo {
    int nx, ny, nz;
    const double* df[3];
    const double* dcn[3];
};

struct FieldGeoOwner {
    DevBuf buf;
    FieldGeo view{};
};

static std::mutex g_geo_mu;
static std::map<std::string, std::unique_ptr<FieldGeoOwner>> g_geo_cache;

static int get_geo(const tbfg_grid_desc* g, FieldGeo& out)
{
    TBFG_TRY(validate_grid(g));
    int dev = 0;
    TBFG_HIP(hipGetDevice(&dev));
    const std::string key = grid_key(g, dev);
    std::lock_guard<std::mutex> lk(g_geo_mu);
    auto it = g_geo_cache.find(key);
    if (it == g_geo_cache.end()) {
        HostLevel L = make_level(g, 0);
        std::vector<double> h;
        size_t off[3][2];
        for (int a = 0; a < 3; ++a) {
            off[a][0] = h.size();
            for (int i = 1; i <= L.n[a]; ++i) h.push_back(L.ax[a].df(i));
            off[a][1] = h.size();
            for (int i = 1; i <= L.n[a]; ++i) h.push_back(L.ax[a].dc(i + 1));
        }
        std::unique_ptr<FieldGeoOwner> o(new FieldGeoOwner());
        TBFG_TRY(upload(o->buf, h.data(), h.size() * 8));
        o->view.nx = L.n[0];
        o->view.ny = L.n[1];
        o->view.nz = L.n[2];
        for (int a = 0; a < 3; ++a) {
            o->view.df[a] = o->buf.as<double>() + off[a][0];
            o->view.dcn[a] = o->buf.as<double>() + off[a][1];
        }
        it = g_geo_cache.emplace(key, std::move(o)).first;
    }
    out = it->second->view;
    return TBFG_OK;
}

// (i, j, k) of a thread in a row-wise launch made as a 1-D grid of
// ceil(nx / blockDim.x) * ny * nz workgroups.  Workgroups go round-robin to the 8
// XCDs, each with its own L2, so consecutive ones are renumbered to fall on one
// XCD: each XCD then works through a contiguous range of rows and planes, and the
// y and z neighbours a workgroup reads were read into that XCD's L2 by its
// neighbours (a 3-D grid numbered rows first sends neighbouring rows to different
// XCDs, and each of them fetches the shared faces from HBM again).
__device__ __forceinline__ void row_cell(int nx, int ny, int& i, int& j, int& k)
{
    const unsigned nb = gridDim.x;
    unsigned id = blockIdx.x;
    if ((nb & 7u) == 0) id = (id & 7u) * (nb >> 3) + (id >> 3);
    const unsigned gx = ((unsigned)nx + blockDim.x - 1) / blockDim.x;
    const unsigned bx = id % gx, r = id / gx;
    i = (int)(bx * blockDim.x + threadIdx.x);
    j = (int)(r % (unsigned)ny);
    k = (int)(r / (unsigned)ny);
}

__device__ __forceinline__ double div_cell(const FieldGeo& G, const double* __restrict__ ux,
                                           const double* __restrict__ uy, const double* __restrict__ uz, int i, int j,
                                           int k)
{
    const int nx = G.nx, ny = G.ny, nz = G.nz;
    const size_t c = i + (size_t)nx * (j + (size_t)ny * k);
    const size_t w = (i > 0 ? i - 1 : nx - 1) + (size_t)nx * (j + (size_t)ny * k);
    const size_t b = i + (size_t)nx * (j + (size_t)ny * (k > 0 ? k - 1 : nz - 1));
    const size_t yt = i + (size_t)nx * ((j + 1) + (size_t)(ny + 1) * k);
    const size_t yb = i + (size_t)nx * (j + (size_t)(ny + 1) * k);
    const double dx = (ux[c] - ux[w]) / G.df[0][i];
    const double dy = (uy[yt] - uy[yb]) / G.df[1][j];
    const double dz = (uz[c] - uz[b]) / G.df[2][k];
    return dx + dy + dz;
}

// poissonEqn.f90:176-188 / auxiliaryRoutines.f90:66-79
__global__ void k_divergence(FieldGeo G, const double* __restrict__ ux, const double* __restrict__ uy,
                             const double* __restrict__ uz, double* __restrict__ div)
{
    int i, j, k;
    row_cell(G.nx, G.ny, i, j, k);
    if (i >= G.nx) return;
    div[i + (size_t)G.nx * (j + (size_t)G.ny * k)] = div_cell(G, ux, uy, uz, i, j, k);
}

// auxiliaryRoutines.f90:60-82: max |div u| (the reference prints it times dt)
__global__ void k_maxdiv(FieldGeo G, const double* __restrict__ ux, const double* __restrict__ uy,
                         const double* __restrict__ uz, unsigned long long* out)
{
    int i, j, k;
    row_cell(G.nx, G.ny, i, j, k);
    double v = 0.0;
    if (i < G.nx) v = fabs(div_cell(G, ux, uy, uz, i, j, k));
    if (!(v == v)) v = __longlong_as_double(0x7ff0000000000000LL);  // NaN -> +inf
    for (int off = 32; off > 0; off >>= 1) v = fmax(v, __shfl_down(v, off, 64));
    __shared__ double wmax[16];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    if (lane == 0) wmax[wave] = v;
    __syncthreads();
    if (threadIdx.x == 0) {
        double m = 0.0;
        for (int w = 0; w < (int)((blockDim.x + 63) >> 6); ++w) m = fmax(m, wmax[w]);
        // non-negative doubles order like their bit patterns
        atomicMax(out, (unsigned long long)__double_as_longlong(m));
    }
}

// poissonEqn.f90:331-337
__global__ void k_beta(size_t n, double alpha_dt, const double* __restrict__ rho, double* __restrict__ beta)
{
    const size_t t = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t < n) beta[t] = alpha_dt / rho[t];
}

// momentumEqn.f90:806-866 (addPressureGrad) on all periodic x/z faces and the
// interior y faces (setEqnBounds, momentumEqn.f90:1134-1190).
__global__ void k_project_mg(FieldGeo G, double alpha_dt, const double* __restrict__ rho,
                             const double* __restrict__ psi, double* __restrict__ ux, double* __restrict__ uy,
                             double* __restrict__ uz)
{
    int i, j, k;
    row_cell(G.nx, G.ny, i, j, k);
    const int nx = G.nx, ny = G.ny, nz = G.nz;
    if (i >= nx) return;
    const size_t c = i + (size_t)nx * (j + (size_t)ny * k);
    const size_t e = (i + 1 < nx ? i + 1 : 0) + (size_t)nx * (j + (size_t)ny * k);
    const size_t f = i + (size_t)nx * (j + (size_t)ny * (k + 1 < nz ? k + 1 : 0));
    const double ic = 1.0 / rho[c];
    double inv = 0.5 * (1.0 / rho[e] + ic);
    ux[c] = ux[c] - alpha_dt * inv * (psi[e] - psi[c]) / G.dcn[0][i];
    inv = 0.5 * (1.0 / rho[f] + ic);
    uz[c] = uz[c] - alpha_dt * inv * (psi[f] - psi[c]) / G.dcn[2][k];
    if (j + 1 < ny) {
        const size_t n = i + (size_t)nx * ((j + 1) + (size_t)ny * k);
        const size_t yf = i + (size_t)nx * ((j + 1) + (size_t)(ny + 1) * k);
        inv = 0.5 * (1.0 / rho[n] + ic);
        uy[yf] = uy[yf] - alpha_dt * inv * (psi[n] - psi[c]) / G.dcn[1][j];
    }
}

// Old levels of the FAST splitting (poissonEqn.f90:255-301): psi^n (p1), psi^(n-1) (p2)
// and the surface-tension levels st^n, st^(n-1), three staggered components each laid
// out like the velocity.  A level, or a component, may be absent (then zero): its
// pointer is that of another array and its bit in `has` is clear, so that every load is
// unconditional (a branch around each load made the compiler wait for it there).
struct OldLevels {
    const double* p[2];     // psi^n, psi^(n-1)
    const double* st[2][3]; // st^n, st^(n-1)
    unsigned has;           // bit l: p[l]; bit 2 + 3 l + c: st[l][c]
};
// which levels a kernel reads: none, pressure, pressure and surface tension
enum { kNoLevels = 0, kPsiLevels = 1, kAllLevels = 2 };

template <int MODE>
__device__ __forceinline__ double old_psi(const OldLevels& o, int l, size_t i)
{
    if (MODE == kNoLevels) return 0.0;
    const double v = o.p[l][i];
    return (o.has >> l) & 1u ? v : 0.0;
}

template <int MODE>
__device__ __forceinline__ double old_st(const OldLevels& o, int l, int comp, size_t f)
{
    if (MODE != kAllLevels) return 0.0;
    const double v = o.st[l][comp][f];
    return (o.has >> (2 + 3 * l + comp)) & 1u ? v : 0.0;
}

// the face value G_f = (2 d psi^n - d psi^(n-1)) / dc - 2 st^n_f + st^(n-1)_f
// (poissonEqn.f90:255-301, momentumEqn.f90:1104-1121), in the reference's order of
// operations; a*, b* the values of the two levels on either side of the face
template <int MODE>
__device__ __forceinline__ double old_grad(double a1, double b1, double a2, double b2, double dc, double s1, double s2)
{
    if (MODE == kNoLevels) return 0.0;
    const double g = (2.0 * (b1 - a1) - (b2 - a2)) / dc;
    return MODE == kPsiLevels ? g : g - 2.0 * s1 + s2;
}

// Launch of the column kernels below: a thread owns the column (i, j) of a chunk of kc
// planes and marches through it, so the values of the plane before and after stay in
// registers (read once per chunk instead of once per z neighbour: at 192x128x192 a
// plane of the up to 16 arrays is 3 MB, and the z neighbours fell out of the L2), and
// the loads of the next plane are in flight while one is computed.  The in-plane
// neighbours come from the tile's own rows (L1).  Tiles of 64 x 4 columns, or 32 x 8
// where those leave fewer lanes idle; chunks for one resident round of workgroups
// (three per CU by registers: 768), since a second, partly filled one costs as much as
// a full one.  192x128x192 with every level, in a step: source 211 -> 145 us, projection
// 153 -> 139 us (their bytes at the copy rate: 96 and 118 us).
struct ColGrid {
    dim3 blk;
    unsigned nblocks;
    int tiles_x, ntiles, kc;
};

static ColGrid column_grid(int nx, int ny, int nz)
{
    ColGrid c;
    const bool wide = (nx + 63) / 64 * 64 <= (nx + 31) / 32 * 32;
    c.blk = wide ? dim3(64, 4) : dim3(32, 8);
    c.tiles_x = (int)ceil_div(nx, c.blk.x);
    c.ntiles = c.tiles_x * (int)ceil_div(ny, c.blk.y);
    const int chunks = std::max(1, std::min(nz, 768 / c.ntiles));
    c.kc = (nz + chunks - 1) / chunks;
    c.nblocks = (unsigned)c.ntiles * ceil_div(nz, c.kc);
    return c;
}

// consecutive tiles of a chunk of planes on one XCD, as row_cell
__device__ __forceinline__ void column_cell(int kc, int tiles_x, int ntiles, int nz, int& i, int& j, int& k0, int& k1)
{
    const unsigned nb = gridDim.x;
    unsigned id = blockIdx.x;
    if ((nb & 7u) == 0) id = (id & 7u) * (nb >> 3) + (id >> 3);
    const int tile = (int)(id % (unsigned)ntiles);
    k0 = (int)(id / (unsigned)ntiles) * kc;
    k1 = min(nz, k0 + kc);
    i = (tile % tiles_x) * (int)blockDim.x + (int)threadIdx.x;
    j = (tile / tiles_x) * (int)blockDim.y + (int)threadIdx.y;
}

// FAST computeSource + computeOldPressDiv with two old levels (poissonEqn.f90:193-305):
// s = rho0/(alpha dt) div u* + div[(1 - rho0 (1/rho)_f) G_f], G_f the face gradient of
// 2 psi^n - psi^(n-1) minus 2 st^n_f - st^(n-1)_f; (1/rho)_f the arithmetic face mean.
// The face after a cell reads the st values of the cell's own face index, the face
// before it those of the previous face (in y the wall faces 0 and ny included).  The
// flux and the velocity of the face after a cell in z are those of the face before the
// next one: carried along the march.
template <int MODE>
__global__ void __launch_bounds__(256)
    k_source_fast(FieldGeo G, double r_adt, double rho0, const double* __restrict__ rho,
                  const double* __restrict__ ux, const double* __restrict__ uy, const double* __restrict__ uz,
                  OldLevels o, double* __restrict__ s, int kc, int tiles_x, int ntiles)
{
    int i, j, k0, k1;
    column_cell(kc, tiles_x, ntiles, G.nz, i, j, k0, k1);
    const int nx = G.nx, ny = G.ny, nz = G.nz;
    if (i >= nx || j >= ny) return;
    const size_t plane = (size_t)nx * ny;
    const size_t oc = i + (size_t)nx * j;
    const size_t oe = (i + 1 < nx ? i + 1 : 0) + (size_t)nx * j;
    const size_t ow = (i > 0 ? i - 1 : nx - 1) + (size_t)nx * j;
    const size_t on = i + (size_t)nx * (j + 1 < ny ? j + 1 : j);  // wall ghost = the cell
    const size_t os = i + (size_t)nx * (j > 0 ? j - 1 : j);
    const double dxf = G.df[0][0], dzf = G.df[2][0], dyf = G.df[1][j];
    const double dxc = G.dcn[0][0], dzc = G.dcn[2][0];
    const double dycp = G.dcn[1][j], dycm = G.dcn[1][j > 0 ? j - 1 : 0];
    // 1 - rho0 (1/rho)_f of the face between inverses a and b
    auto weight = [&](double a, double b) { return 1.0 - rho0 * 0.5 * (b + a); };
    const size_t pb = plane * (size_t)(k0 > 0 ? k0 - 1 : nz - 1), p0 = plane * k0 + oc;
    double ic = 1.0 / rho[p0], c1 = old_psi<MODE>(o, 0, p0), c2 = old_psi<MODE>(o, 1, p0);
    double fzm = weight(1.0 / rho[pb + oc], ic) *
                 old_grad<MODE>(old_psi<MODE>(o, 0, pb + oc), c1, old_psi<MODE>(o, 1, pb + oc), c2, dzc,
                                old_st<MODE>(o, 0, 2, pb + oc), old_st<MODE>(o, 1, 2, pb + oc));
    double uzm = uz[pb + oc];
    // the loads of a plane, issued while the plane before is computed
    struct Plane {
        double rf, re, rw, rn, rs;                            // density behind the faces (z-: the plane before)
        double f1, f2, e1, e2, w1, w2, n1, n2, s1, s2;         // the two old pressures there
        double uxc, uxw, uyt, uyb, uzc;
        double x1, x2, m1, m2, t1, t2, b1, b2, z1, z2;         // surface tension: x+, x-, y+, y-, z+
    };
    auto load = [&](Plane& v, int k) {
        const size_t pk = plane * k, f = plane * (size_t)(k + 1 < nz ? k + 1 : 0) + oc;
        const size_t yt = i + (size_t)nx * ((j + 1) + (size_t)(ny + 1) * k);  // y face after the cell
        const size_t yb = yt - nx;                                             // y face before it
        const size_t c = pk + oc, e = pk + oe, w = pk + ow, n = pk + on, so = pk + os;
        v.rf = rho[f], v.re = rho[e], v.rw = rho[w], v.rn = rho[n], v.rs = rho[so];
        v.f1 = old_psi<MODE>(o, 0, f), v.f2 = old_psi<MODE>(o, 1, f);
        v.e1 = old_psi<MODE>(o, 0, e), v.e2 = old_psi<MODE>(o, 1, e);
        v.w1 = old_psi<MODE>(o, 0, w), v.w2 = old_psi<MODE>(o, 1, w);
        v.n1 = old_psi<MODE>(o, 0, n), v.n2 = old_psi<MODE>(o, 1, n);
        v.s1 = old_psi<MODE>(o, 0, so), v.s2 = old_psi<MODE>(o, 1, so);
        v.uxc = ux[c], v.uxw = ux[w], v.uyt = uy[yt], v.uyb = uy[yb], v.uzc = uz[c];
        v.x1 = old_st<MODE>(o, 0, 0, c), v.x2 = old_st<MODE>(o, 1, 0, c);
        v.m1 = old_st<MODE>(o, 0, 0, w), v.m2 = old_st<MODE>(o, 1, 0, w);
        v.t1 = old_st<MODE>(o, 0, 1, yt), v.t2 = old_st<MODE>(o, 1, 1, yt);
        v.b1 = old_st<MODE>(o, 0, 1, yb), v.b2 = old_st<MODE>(o, 1, 1, yb);
        v.z1 = old_st<MODE>(o, 0, 2, c), v.z2 = old_st<MODE>(o, 1, 2, c);
    };
    Plane v;
    load(v, k0);
    for (int k = k0; k < k1; ++k) {
        Plane nxt;
        load(nxt, min(k + 1, k1 - 1));
        __builtin_amdgcn_sched_barrier(0);
        const double div = (v.uxc - v.uxw) / dxf + (v.uyt - v.uyb) / dyf + (v.uzc - uzm) / dzf;
        const double gxp = old_grad<MODE>(c1, v.e1, c2, v.e2, dxc, v.x1, v.x2);
        const double gxm = old_grad<MODE>(v.w1, c1, v.w2, c2, dxc, v.m1, v.m2);
        const double gyp = old_grad<MODE>(c1, v.n1, c2, v.n2, dycp, v.t1, v.t2);
        const double gym = old_grad<MODE>(v.s1, c1, v.s2, c2, dycm, v.b1, v.b2);
        const double gzp = old_grad<MODE>(c1, v.f1, c2, v.f2, dzc, v.z1, v.z2);
        const double jf = 1.0 / v.rf;
        const double fzp = weight(ic, jf) * gzp;
        const double dx = (weight(1.0 / v.re, ic) * gxp - weight(1.0 / v.rw, ic) * gxm) / dxf;
        const double dy = (weight(1.0 / v.rn, ic) * gyp - weight(1.0 / v.rs, ic) * gym) / dyf;
        const double dz = (fzp - fzm) / dzf;
        s[plane * k + oc] = div * r_adt * rho0 + dx + dy + dz;
        ic = jf, c1 = v.f1, c2 = v.f2;
        fzm = fzp;
        uzm = v.uzc;
        v = nxt;
    }
}

// FAST makeVelocityDivFree + computeOldPressGrad (momentumEqn.f90:999-1127):
// u_f -= alpha dt [(1/rho0) d psi + ((1/rho)_f - 1/rho0) G_f] on the periodic x/z
// faces and the interior y faces.  The plane after a cell's is its own on the next
// step of the march.
template <int MODE>
__global__ void __launch_bounds__(256)
    k_project_fast(FieldGeo G, double alpha_dt, double rho0, const double* __restrict__ rho,
                   const double* __restrict__ psi, OldLevels o, double* __restrict__ ux, double* __restrict__ uy,
                   double* __restrict__ uz, int kc, int tiles_x, int ntiles)
{
    int i, j, k0, k1;
    column_cell(kc, tiles_x, ntiles, G.nz, i, j, k0, k1);
    const int nx = G.nx, ny = G.ny, nz = G.nz;
    if (i >= nx || j >= ny) return;
    const size_t plane = (size_t)nx * ny;
    const size_t oc = i + (size_t)nx * j;
    const size_t oe = (i + 1 < nx ? i + 1 : 0) + (size_t)nx * j;
    const size_t on = j + 1 < ny ? oc + nx : oc;
    const double dxc = G.dcn[0][0], dzc = G.dcn[2][0], dyc = G.dcn[1][j];
    const double inv0 = 1.0 / rho0;
    // the correction of a face between inverses ia, ib and pressures pa, pb, with the old levels' G_f
    auto face = [&](double ia, double ib, double pa, double pb, double g, double dc) {
        const double inv = 0.5 * (ib + ia);
        return alpha_dt * (inv0 * ((pb - pa) / dc) + (inv - inv0) * g);
    };
    const size_t p0 = plane * k0 + oc;
    double ic = 1.0 / rho[p0], pc = psi[p0], c1 = old_psi<MODE>(o, 0, p0), c2 = old_psi<MODE>(o, 1, p0);
    struct Plane {
        double rf, re, rn, pf, pe, pn, f1, f2, e1, e2, n1, n2, vx, vy, vz, x1, x2, y1, y2, z1, z2;
    };
    auto load = [&](Plane& v, int k) {
        const size_t pk = plane * k, f = plane * (size_t)(k + 1 < nz ? k + 1 : 0) + oc;
        const size_t c = pk + oc, e = pk + oe, n = pk + on;
        const size_t yf = i + (size_t)nx * ((j + 1) + (size_t)(ny + 1) * k);
        v.rf = rho[f], v.re = rho[e], v.rn = rho[n];
        v.pf = psi[f], v.pe = psi[e], v.pn = psi[n];
        v.f1 = old_psi<MODE>(o, 0, f), v.f2 = old_psi<MODE>(o, 1, f);
        v.e1 = old_psi<MODE>(o, 0, e), v.e2 = old_psi<MODE>(o, 1, e);
        v.n1 = old_psi<MODE>(o, 0, n), v.n2 = old_psi<MODE>(o, 1, n);
        v.vx = ux[c], v.vy = uy[yf], v.vz = uz[c];
        v.x1 = old_st<MODE>(o, 0, 0, c), v.x2 = old_st<MODE>(o, 1, 0, c);
        v.y1 = old_st<MODE>(o, 0, 1, yf), v.y2 = old_st<MODE>(o, 1, 1, yf);
        v.z1 = old_st<MODE>(o, 0, 2, c), v.z2 = old_st<MODE>(o, 1, 2, c);
    };
    Plane v;
    load(v, k0);
    for (int k = k0; k < k1; ++k) {
        Plane nxt;
        load(nxt, min(k + 1, k1 - 1));  // (each face belongs to one thread and plane: none is read after its update)
        __builtin_amdgcn_sched_barrier(0);
        const size_t c = plane * k + oc;
        const double jf = 1.0 / v.rf;
        ux[c] = v.vx - face(ic, 1.0 / v.re, pc, v.pe, old_grad<MODE>(c1, v.e1, c2, v.e2, dxc, v.x1, v.x2), dxc);
        uz[c] = v.vz - face(ic, jf, pc, v.pf, old_grad<MODE>(c1, v.f1, c2, v.f2, dzc, v.z1, v.z2), dzc);
        if (j + 1 < ny)
            uy[i + (size_t)nx * ((j + 1) + (size_t)(ny + 1) * k)] =
                v.vy - face(ic, 1.0 / v.rn, pc, v.pn, old_grad<MODE>(c1, v.n1, c2, v.n2, dyc, v.y1, v.y2), dyc);
        ic = jf, pc = v.pf, c1 = v.f1, c2 = v.f2;
        v = nxt;
    }
}

// updatePressure (poissonEqn.f90:374-415) + clean_st_prev_bc (:419-459) for the
// channel, one thread per face row entry: p = psi; psi2 <- psi1 <- psi
// (storeOldField); st2 <- st1 <- st (storeOldFieldV, st NULL = zero); the old st
// levels zeroed on the y wall faces (j = 0, ny).  Block row j = ny carries only
// the top wall face of the y component.  Each entry is read and written by its
// own thread, so the rotation is in place.
struct StRotate {
    const double* cur[3];
    double* l1[3];
    double* l2[3];
};

__global__ void k_update_pressure(int nx, int ny, int nz, const double* __restrict__ psi, double* __restrict__ p,
                                  double* __restrict__ psi1, double* __restrict__ psi2, StRotate st, int with_st)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    const int j = blockIdx.y;
    const int k = blockIdx.z;
    if (i >= nx) return;
    if (j < ny) {
        const size_t c = i + (size_t)nx * (j + (size_t)ny * k);
        const double v = psi[c];
        if (p) p[c] = v;
        psi2[c] = psi1[c];
        psi1[c] = v;
        if (with_st) {
            for (int a = 0; a < 3; a += 2) {
                st.l2[a][c] = st.l1[a][c];
                st.l1[a][c] = st.cur[a] ? st.cur[a][c] : 0.0;
            }
        }
    }
    if (with_st) {
        const size_t yf = i + (size_t)nx * (j + (size_t)(ny + 1) * k);
        if (j == 0 || j == ny) {
            st.l2[1][yf] = 0.0;
            st.l1[1][yf] = 0.0;
        } else {
            st.l2[1][yf] = st.l1[1][yf];
            st.l1[1][yf] = st.cur[1] ? st.cur[1][yf] : 0.0;
        }
    }
}

static dim3 row_block(int nx) { return dim3(nx >= 256 ? 256 : (unsigned)next_pow2(nx < 64 ? 64 : nx)); }

int divergence_dev(const tbfg_grid_desc* g, const double* ux, const double* uy, const double* uz, double* div,
                   void* stream)
{
    if (!ux || !uy || !uz || !div) {
        set_error("tbfg_divergence_dev: NULL argument");
        return TBFG_EINVAL;
    }
    FieldGeo G;
    TBFG_TRY(get_geo(g, G));
    dim3 blk = row_block(G.nx);
    hipLaunchKernelGGL(k_divergence, dim3(ceil_div(G.nx, blk.x) * G.ny * G.nz), blk, 0, (hipStream_t)stream, G, ux, uy,
                       uz, div);
    TBFG_HIP(hipGetLastError());
    return TBFG_OK;
}

int max_divergence_dev(const tbfg_grid_desc* g, const double* ux, const double* uy, const double* uz, double* out,
                       void* stream)
{
    if (!ux || !uy || !uz || !out) {
        set_error("tbfg_max_divergence_dev: NULL argument");
        return TBFG_EINVAL;
    }
    FieldGeo G;
    TBFG_TRY(get_geo(g, G));
    DevBuf res;
    TBFG_TRY(res.alloc(sizeof(unsigned long long)));
    hipStream_t s = (hipStream_t)stream;
    TBFG_HIP(hipMemsetAsync(res.p, 0, sizeof(unsigned long long), s));
    dim3 blk = row_block(G.nx);
    hipLaunchKernelGGL(k_maxdiv, dim3(ceil_div(G.nx, blk.x) * G.ny * G.nz), blk, 0, s, G, ux, uy, uz,
                       res.as<unsigned long long>());
    TBFG_HIP(hipGetLastError());
    unsigned long long bits = 0;
    TBFG_HIP(hipMemcpyAsync(&bits, res.p, sizeof bits, hipMemcpyDeviceToHost, s));
    TBFG_HIP(hipStreamSynchronize(s));
    double v;
    static_assert(sizeof v == sizeof bits, "64-bit double");
    std::memcpy(&v, &bits, sizeof v);
    *out = v;
    return TBFG_OK;
}

// ----------------------------------------------- continuity error without allocation
//
// The same kernel as max_divergence_dev with its scratch -- the max word and the
// per-axis metrics -- in one file-scope device array instead of a hipMalloc per call
// and the geometry cache: [max word, padding to 256 B | df, dc(i+1) of x | of y | of z].
// Each device holds its own copy; its address comes from hipGetSymbolAddress on the
// first call on that device (the array's name is not a device address in host code).
constexpr int kNoAllocMaxAxis = 4096;   // cells per axis
constexpr size_t kNoAllocHead = 32;     // doubles before the metrics
constexpr size_t kNoAllocDoubles = kNoAllocHead + 2 * 3 * (size_t)kNoAllocMaxAxis;  // 196,864 bytes
static __device__ __align__(256) double scratch[kNoAllocDoubles];

struct NoAllocScratch {
    std::mutex mu;           // held for a whole call: the call ends with its stream drained
    double* ptr = nullptr;   // this device's copy of `scratch`
};

static std::mutex g_noalloc_mu;
static std::map<int, std::unique_ptr<NoAllocScratch>> g_noalloc;  // by device

static int noalloc_scratch(int dev, NoAllocScratch** out)
{
    std::lock_guard<std::mutex> lk(g_noalloc_mu);
    std::unique_ptr<NoAllocScratch>& slot = g_noalloc[dev];
    if (!slot) {
        void* p = nullptr;
        TBFG_HIP(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
        std::unique_ptr<NoAllocScratch> d(new NoAllocScratch());
        d->ptr = static_cast<double*>(p);
        slot = std::move(d);
    }
    *out = slot.get();
    return TBFG_OK;
}

int max_divergence_noalloc_dev(const tbfg_grid_desc* g, const double* ux, const double* uy, const double* uz,
                               double* out, void* stream)
{
    if (!ux || !uy || !uz || !out) {
        set_error("tbfg_max_divergence_noalloc_dev: NULL argument");
        return TBFG_EINVAL;
    }
    TBFG_TRY(validate_grid(g));
    for (int a = 0; a < 3; ++a)
        if (g->n[a] > kNoAllocMaxAxis) {
            set_error("tbfg_max_divergence_noalloc_dev: axis %d has %d cells, at most %d fit its scratch", a,
                      g->n[a], kNoAllocMaxAxis);
            return TBFG_EINVAL;
        }
    int dev = 0;
    TBFG_HIP(hipGetDevice(&dev));
    NoAllocScratch* d = nullptr;
    TBFG_TRY(noalloc_scratch(dev, &d));
    std::lock_guard<std::mutex> lk(d->mu);

    // host image of the used part of the scratch: a zero max word, then the metrics
    // (the values get_geo uploads, so both entry points compute the same result)
    const HostLevel L = make_level(g, 0);
    std::vector<double> h(kNoAllocHead, 0.0);
    FieldGeo G;
    G.nx = L.n[0];
    G.ny = L.n[1];
    G.nz = L.n[2];
    size_t off[3][2];
    for (int a = 0; a < 3; ++a) {
        off[a][0] = h.size();
        for (int i = 1; i <= L.n[a]; ++i) h.push_back(L.ax[a].df(i));
        off[a][1] = h.size();
        for (int i = 1; i <= L.n[a]; ++i) h.push_back(L.ax[a].dc(i + 1));
    }
    for (int a = 0; a < 3; ++a) {
        G.df[a] = d->ptr + off[a][0];
        G.dcn[a] = d->ptr + off[a][1];
    }
    hipStream_t s = (hipStream_t)stream;
    unsigned long long bits = 0;
    hipError_t e = hipMemcpyAsync(d->ptr, h.data(), h.size() * sizeof(double), hipMemcpyHostToDevice, s);
    if (e == hipSuccess) {
        const dim3 blk = row_block(G.nx);
        hipLaunchKernelGGL(k_maxdiv, dim3(ceil_div(G.nx, blk.x) * G.ny * G.nz), blk, 0, s, G, ux, uy, uz,
                           reinterpret_cast<unsigned long long*>(d->ptr));
        e = hipGetLastError();
    }
    if (e == hipSuccess) e = hipMemcpyAsync(&bits, d->ptr, sizeof bits, hipMemcpyDeviceToHost, s);
    // drained on every path: `h` and `bits` live on this frame, and the next call reuses the scratch
    const hipError_t es = hipStreamSynchronize(s);
    if (e == hipSuccess) e = es;
    if (e != hipSuccess) {
        set_error("tbfg_max_divergence_noalloc_dev: %s", hipGetErrorString(e));
        return TBFG_EDEVICE;
    }
    double v;
    std::memcpy(&v, &bits, sizeof v);
    *out = v;
    return TBFG_OK;
}

int beta_dev(const tbfg_grid_desc* g, double alpha_dt, const double* rho, double* beta, void* stream)
{
    TBFG_TRY(validate_grid(g));
    if (!rho || !beta) {
        set_error("tbfg_beta_dev: NULL argument");
        return TBFG_EINVAL;
    }
    const size_t n = (size_t)g->n[0] * g->n[1] * g->n[2];
    hipLaunchKernelGGL(k_beta, dim3(ceil_div(n, 256)), dim3(256), 0, (hipStream_t)stream, n, alpha_dt, rho, beta);
    TBFG_HIP(hipGetLastError());
    return TBFG_OK;
}

// a NULL level, or a NULL component of one, is zero (`any` stands in for its address);
// mode: the levels that are there
static OldLevels old_levels(const double* psi1, const double* psi2, const double* const st1[3],
                            const double* const st2[3], const double* any_cell, const double* any_y, int& mode)
{
    OldLevels o{};
    const double* p[2] = {psi1, psi2};
    const double* const* st[2] = {st1, st2};
    for (int l = 0; l < 2; ++l) {
        o.p[l] = p[l] ? p[l] : any_cell;
        if (p[l]) o.has |= 1u << l;
        for (int c = 0; c < 3; ++c) {
            const double* a = st[l] ? st[l][c] : nullptr;
            o.st[l][c] = a ? a : (c == 1 ? any_y : any_cell);
            if (a) o.has |= 1u << (2 + 3 * l + c);
        }
    }
    mode = (o.has >> 2) ? kAllLevels : (o.has ? kPsiLevels : kNoLevels);
    return o;
}

int source_fast_dev(const tbfg_grid_desc* g, double alpha_dt, double rho0, const double* rho, const double* ux,
                    const double* uy, const double* uz, const double* psi1, const double* psi2,
                    const double* const st1[3], const double* const st2[3], double* s, void* stream)
{
    if (!rho || !ux || !uy || !uz || !s) {
        set_error("tbfg_source_fast_dev: NULL argument");
        return TBFG_EINVAL;
    }
    if (!(alpha_dt > 0.0) || !(rho0 > 0.0)) {
        set_error("tbfg_source_fast_dev: alpha_dt = %g, rho0 = %g (both must be > 0)", alpha_dt, rho0);
        return TBFG_EINVAL;
    }
    FieldGeo G;
    TBFG_TRY(get_geo(g, G));
    if (g->stretch[0] || g->stretch[2]) {
        set_error("tbfg_source_fast_dev: x and z must be uniform (FAST_MODE)");
        return TBFG_EINVAL;
    }
    int mode = 0;
    const OldLevels o = old_levels(psi1, psi2, st1, st2, rho, uy, mode);
    const ColGrid cg = column_grid(G.nx, G.ny, G.nz);
    auto k = mode == kAllLevels   ? k_source_fast<kAllLevels>
             : mode == kPsiLevels ? k_source_fast<kPsiLevels>
                                  : k_source_fast<kNoLevels>;
    hipLaunchKernelGGL(k, dim3(cg.nblocks), cg.blk, 0, (hipStream_t)stream, G, 1.0 / alpha_dt, rho0, rho, ux, uy, uz, o,
                       s, cg.kc, cg.tiles_x, cg.ntiles);
    TBFG_HIP(hipGetLastError());
    return TBFG_OK;
}

int project_fast_dev(const tbfg_grid_desc* g, double alpha_dt, double rho0, const double* rho, const double* psi,
                     const double* psi1, const double* psi2, const double* const st1[3],
                     const double* const st2[3], double* ux, double* uy, double* uz, void* stream)
{
    if (!rho || !psi || !ux || !uy || !uz) {
        set_error("tbfg_project_fast_dev: NULL argument");
        return TBFG_EINVAL;
    }
    if (!(rho0 > 0.0)) {
        set_error("tbfg_project_fast_dev: rho0 = %g (must be > 0)", rho0);
        return TBFG_EINVAL;
    }
    FieldGeo G;
    TBFG_TRY(get_geo(g, G));
    if (g->stretch[0] || g->stretch[2]) {
        set_error("tbfg_project_fast_dev: x and z must be uniform (FAST_MODE)");
        return TBFG_EINVAL;
    }
    int mode = 0;
    const OldLevels o = old_levels(psi1, psi2, st1, st2, rho, uy, mode);
    const ColGrid cg = column_grid(G.nx, G.ny, G.nz);
    auto k = mode == kAllLevels   ? k_project_fast<kAllLevels>
             : mode == kPsiLevels ? k_project_fast<kPsiLevels>
                                  : k_project_fast<kNoLevels>;
    hipLaunchKernelGGL(k, dim3(cg.nblocks), cg.blk, 0, (hipStream_t)stream, G, alpha_dt, rho0, rho, psi, o, ux, uy, uz,
                       cg.kc, cg.tiles_x, cg.ntiles);
    TBFG_HIP(hipGetLastError());
    return TBFG_OK;
}

int update_pressure_dev(const tbfg_grid_desc* g, const double* psi, double* p, double* psi1, double* psi2,
                        const double* const st[3], double* const st1[3], double* const st2[3], void* stream)
{
    TBFG_TRY(validate_grid(g));
    if (!psi || !psi1 || !psi2) {
        set_error("tbfg_update_pressure_dev: psi, psi1 and psi2 must not be NULL");
        return TBFG_EINVAL;
    }
    if ((st1 == nullptr) != (st2 == nullptr)) {
        set_error("tbfg_update_pressure_dev: st1 and st2 must both be given or both be NULL");
        return TBFG_EINVAL;
    }
    StRotate r{};
    const int with_st = st1 != nullptr;
    if (with_st) {
        for (int a = 0; a < 3; ++a) {
            if (!st1[a] || !st2[a]) {
                set_error("tbfg_update_pressure_dev: st1[%d] or st2[%d] is NULL", a, a);
                return TBFG_EINVAL;
            }
            r.cur[a] = st ? st[a] : nullptr;
            r.l1[a] = st1[a];
            r.l2[a] = st2[a];
        }
    } else if (st) {
        set_error("tbfg_update_pressure_dev: st given without st1, st2 to store it in");
        return TBFG_EINVAL;
    }
    const int nx = g->n[0], ny = g->n[1], nz = g->n[2];
    dim3 blk = row_block(nx);
    hipLaunchKernelGGL(k_update_pressure, dim3(ceil_div(nx, blk.x), ny + 1, nz), blk, 0, (hipStream_t)stream, nx, ny,
                       nz, psi, p, psi1, psi2, r, with_st);
    TBFG_HIP(hipGetLastError());
    return TBFG_OK;
}

int project_mg_dev(const tbfg_grid_desc* g, double alpha_dt, const double* rho, const double* psi, double* ux,
                   double* uy, double* uz, void* stream)
{
    if (!rho || !psi || !ux || !uy || !uz) {
        set_error("tbfg_project_mg_dev: NULL argument");
        return TBFG_EINVAL;
    }
    FieldGeo G;
    TBFG_TRY(get_geo(g, G));
    dim3 blk = row_block(G.nx);
    hipLaunchKernelGGL(k_project_mg, dim3(ceil_div(G.nx, blk.x) * G.ny * G.nz), blk, 0, (hipStream_t)stream, G,
                       alpha_dt, rho, psi, ux, uy, uz);
    TBFG_HIP(hipGetLastError());
    return TBFG_OK;
}

}  // namespace tbfg
