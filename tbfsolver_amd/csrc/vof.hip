// vof.hip -- material properties from the volume fraction on the device
// (updateMaterialProps and smoothVF, VOF.f90:197-262): two passes of
// trilinear cell -> vertex interpolation (interpolation.f90:188-226) and
// vertex -> cell averaging (:231-276) smooth c into cs, then
// rho = rho_g cs + (1 - cs) rho_l and mu likewise.  Ghost cells of c and cs
// are the periodic images in x and z and the wall row itself in y (the
// zero-gradient boundary of the volume fraction).
//
// The trilinear weights are products of one-dimensional ones, and the ghosts are
// those of each axis by itself, so a pass is T_x T_y T_z with T a three-point filter
// per axis, and both passes are the five-point filters T^2 of each axis: one kernel
// reads c once and writes cs, rho and mu, where four kernels carried the vertex
// field and cs through memory twice with eight gathered values and an FP64 division
// per vertex and cell.  The weights are formed once per grid in extended precision.
// 256x192x256: 429 -> 110 us (32 B per cell must move: 79 us at the copy rate).
#include <algorithm>
#include <map>
#include <mutex>
#include <string>

#include "fields.hpp"

namespace tbfg {

struct VofGeo {
    int nx, ny, nz;
    const double* w[3];  // five-point weights of each axis, entry 5 i + m: the value at offset m - 2 of cell i
};

struct VofGeoOwner {
    DevBuf buf;
    VofGeo view{};
};

static std::mutex g_vof_mu;
static std::map<std::string, std::unique_ptr<VofGeoOwner>> g_vof_cache;

// T^2 of one axis.  T takes cell m (1-based) from the centres m - 1, m, m + 1: the
// vertex values weigh the centre on each side by the distance to the other one, the
// cell value the vertices likewise.  On the bounded axis the offsets that fall outside
// read the wall row: the weight of a row that several offsets read is spread evenly
// over them.
static void filter_weights(const Axis& ax, bool periodic, std::vector<double>& out)
{
    using ld = long double;
    const int n = ax.n;
    std::vector<ld> a(n + 2), b(n + 2), d(n + 2);
    auto lo = [&](int v) { return ((ld)ax.c(v + 1) - (ld)ax.f(v)) / ((ld)ax.c(v + 1) - (ld)ax.c(v)); };
    for (int m = 1; m <= n; ++m) {
        const ld span = (ld)ax.f(m) - (ld)ax.f(m - 1);
        const ld cl = ((ld)ax.f(m) - (ld)ax.c(m)) / span, ch = ((ld)ax.c(m) - (ld)ax.f(m - 1)) / span;
        a[m] = cl * lo(m - 1);
        b[m] = cl * (1 - lo(m - 1)) + ch * lo(m);
        d[m] = ch * (1 - lo(m));
    }
    a[0] = a[n], b[0] = b[n], d[0] = d[n];  // (used on a periodic axis only)
    a[n + 1] = a[1], b[n + 1] = b[1], d[n + 1] = d[1];
    for (int m = 1; m <= n; ++m) {
        ld w[5] = {0, 0, 0, 0, 0};
        const ld t[3] = {a[m], b[m], d[m]};
        for (int s = 0; s < 3; ++s) {
            int r = m - 1 + s;  // the row the second application reads
            if (!periodic) r = r < 1 ? 1 : (r > n ? n : r);
            const ld u[3] = {a[r], b[r], d[r]};
            for (int q = 0; q < 3; ++q) {
                int src = r - 1 + q;
                if (!periodic) src = src < 1 ? 1 : (src > n ? n : src);
                int off = src - m + 2;
                w[off] += t[s] * u[q];
            }
        }
        if (!periodic)
            for (int wall : {1, n}) {
                int cnt = 0;
                ld sum = 0;
                auto reads = [&](int o) {
                    const int r = m + o - 2;
                    return (r < 1 ? 1 : (r > n ? n : r)) == wall;
                };
                for (int o = 0; o < 5; ++o)
                    if (reads(o)) {
                        sum += w[o];
                        ++cnt;
                    }
                for (int o = 0; o < 5 && cnt > 0; ++o)
                    if (reads(o)) w[o] = sum / cnt;
            }
        for (int o = 0; o < 5; ++o) out.push_back((double)w[o]);
    }
}

static int get_vof_geo(const tbfg_grid_desc* g, VofGeo& out)
{
    TBFG_TRY(validate_grid(g));
    int dev = 0;
    TBFG_HIP(hipGetDevice(&dev));
    const std::string key = grid_key(g, dev);
    std::lock_guard<std::mutex> lk(g_vof_mu);
    auto it = g_vof_cache.find(key);
    if (it == g_vof_cache.end()) {
        HostLevel L = make_level(g, 0);
        std::vector<double> h;
        size_t off[3];
        for (int a = 0; a < 3; ++a) {
            off[a] = h.size();
            filter_weights(L.ax[a], a != 1, h);
        }
        std::unique_ptr<VofGeoOwner> o(new VofGeoOwner());
        TBFG_TRY(upload(o->buf, h.data(), h.size() * 8));
        o->view.nx = L.n[0];
        o->view.ny = L.n[1];
        o->view.nz = L.n[2];
        for (int a = 0; a < 3; ++a) o->view.w[a] = o->buf.as<double>() + off[a];
        it = g_vof_cache.emplace(key, std::move(o)).first;
    }
    out = it->second->view;
    return TBFG_OK;
}

// cs = T^2 c on every axis and the material properties of cs.  A workgroup owns TX x
// TY columns (four consecutive rows per thread) and marches through kc planes: a
// plane of c with its two-cell ring is staged in LDS (its loads issued one plane
// ahead), filtered along x into LDS, then along y into registers, where the last five
// planes' values wait for the filter along z.  Two barriers per plane.
template <int TX>
__global__ void __launch_bounds__(256)
    k_smooth_props(VofGeo G, const double* __restrict__ c, double* __restrict__ cs, double rho_l, double rho_g,
                   double mu_l, double mu_g, double* __restrict__ rho, double* __restrict__ mu, int kc, int tiles_x,
                   int ntiles)
{
    constexpr int NT = 256, GR = NT / TX, TY = 4 * GR;
    constexpr int PX = TX + 4, PY = TY + 4, PS = PX * PY, NP = (PS + NT - 1) / NT;
    __shared__ double sC[PS];
    __shared__ double sX[PY * TX];
    const int nx = G.nx, ny = G.ny, nz = G.nz;
    unsigned id = blockIdx.x;  // consecutive tiles of a chunk on one XCD
    if ((gridDim.x & 7u) == 0) id = (id & 7u) * (gridDim.x >> 3) + (id >> 3);
    const int tile = (int)(id % (unsigned)ntiles);
    const int k0 = (int)(id / (unsigned)ntiles) * kc, k1 = min(nz, k0 + kc);
    if (k0 >= nz) return;
    const int tx0 = (tile % tiles_x) * TX, ty0 = (tile / tiles_x) * TY;
    const int x = (int)threadIdx.x % TX, g = (int)threadIdx.x / TX;
    const size_t plane = (size_t)nx * ny;
    int off[NP];
#pragma unroll
    for (int m = 0; m < NP; ++m) {
        const int t = min((int)threadIdx.x + m * NT, PS - 1);
        const int yy = t / PX, xx = t - yy * PX;
        const int j = min(max(ty0 + yy - 2, 0), ny - 1);
        const int i = (min(tx0 + xx - 2, nx + 1) + 2 * nx) % nx;
        off[m] = nx * j + i;
    }
    const int gx = min(tx0 + x, nx - 1);
    double wx[5], wy[4][5];
#pragma unroll
    for (int o = 0; o < 5; ++o) {
        wx[o] = G.w[0][5 * gx + o];
#pragma unroll
        for (int u = 0; u < 4; ++u) wy[u][o] = G.w[1][5 * min(ty0 + 4 * g + u, ny - 1) + o];
    }
    auto wrap = [&](int k) { return (k + 2 * nz) % nz; };
    double pre[NP];
    auto fetch = [&](int k) {
        const double* src = c + plane * wrap(k);
#pragma unroll
        for (int m = 0; m < NP; ++m) pre[m] = src[off[m]];
    };
    fetch(k0 - 2);
    double h[4][5];
    auto step = [&](int k, int S) {  // plane k; S: its slot among the five
#pragma unroll
        for (int m = 0; m < NP; ++m) sC[min((int)threadIdx.x + m * NT, PS - 1)] = pre[m];
        __syncthreads();
        fetch(min(k + 1, k1 + 1));
#pragma unroll
        for (int r = 0; r < PY; r += GR) {
            const int yy = r + g;
            if (PY % GR == 0 || yy < PY) {
                const double* p = sC + yy * PX + x;
                sX[yy * TX + x] = (wx[0] * p[0] + wx[4] * p[4]) + (wx[1] * p[1] + wx[3] * p[3]) + wx[2] * p[2];
            }
        }
        __syncthreads();
        double f[8];
#pragma unroll
        for (int r = 0; r < 8; ++r) f[r] = sX[(4 * g + r) * TX + x];
#pragma unroll
        for (int u = 0; u < 4; ++u)
            h[u][S] = (wy[u][0] * f[u] + wy[u][4] * f[u + 4]) + (wy[u][1] * f[u + 1] + wy[u][3] * f[u + 3]) +
                      wy[u][2] * f[u + 2];
        const int ko = k - 2;  // the plane whose five are complete
        if (ko < k0 || ko >= k1 || tx0 + x >= nx) return;
        const double* wz = G.w[2] + 5 * ko;
        const double z0 = wz[0], z1 = wz[1], z2 = wz[2], z3 = wz[3], z4 = wz[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const int j = ty0 + 4 * g + u;
            if (j >= ny) break;
            const double v = (z0 * h[u][(S + 1) % 5] + z4 * h[u][S]) + (z1 * h[u][(S + 2) % 5] + z3 * h[u][(S + 4) % 5]) +
                             z2 * h[u][(S + 3) % 5];
            const size_t o = plane * ko + (size_t)nx * j + tx0 + x;
            cs[o] = v;
            rho[o] = rho_g * v + (1.0 - v) * rho_l;
            if (mu) mu[o] = mu_g * v + (1.0 - v) * mu_l;
        }
    };
    for (int k = k0 - 2; k < k1 + 2; k += 5) {
#pragma unroll
        for (int u = 0; u < 5; ++u)
            if (k + u < k1 + 2) step(k + u, u);
    }
}

int64_t material_work_doubles(const tbfg_grid_desc* g)
{
    if (validate_grid(g) != TBFG_OK) return -1;
    return (int64_t)(g->n[0] + 1) * (g->n[1] + 1) * (g->n[2] + 1);
}

int material_props_dev(const tbfg_grid_desc* g, double rho_l, double rho_g, double mu_l, double mu_g, const double* c,
                       double* cs, double* rho, double* mu, double* work, void* stream)
{
    if (!c || !cs || !rho || !work) {
        set_error("tbfg_material_props_dev: NULL argument");
        return TBFG_EINVAL;
    }
    if (c == cs) {
        set_error("tbfg_material_props_dev: c and cs must not alias");
        return TBFG_EINVAL;
    }
    VofGeo G;
    TBFG_TRY(get_vof_geo(g, G));
    hipStream_t s = (hipStream_t)stream;
    // every cell of c is read by several workgroups: an output over c needs a copy of it
    const size_t n = (size_t)G.nx * G.ny * G.nz;
    auto over = [&](const double* a) { return a && a < c + n && c < a + n; };
    if (over(cs) || over(rho) || over(mu)) {
        TBFG_HIP(hipMemcpyAsync(work, c, n * sizeof(double), hipMemcpyDeviceToDevice, s));
        c = work;
    }
    // 64-cell rows, or 32-cell ones where they leave fewer lanes idle; chunks of planes
    // for about three workgroups per CU (four planes of each chunk are read twice)
    const bool wide = (G.nx + 63) / 64 * 64 <= (G.nx + 31) / 32 * 32;
    const int tx = wide ? 64 : 32, ty = 4 * (256 / tx);
    const int tiles_x = (G.nx + tx - 1) / tx, ntiles = tiles_x * ((G.ny + ty - 1) / ty);
    const int kc = std::min(32, std::max(4, (int)(((int64_t)G.nz * ntiles + 767) / 768)));
    const dim3 grid((unsigned)ntiles * (unsigned)((G.nz + kc - 1) / kc));
    if (wide)
        hipLaunchKernelGGL(k_smooth_props<64>, grid, dim3(256), 0, s, G, c, cs, rho_l, rho_g, mu_l, mu_g, rho, mu, kc,
                           tiles_x, ntiles);
    else
        hipLaunchKernelGGL(k_smooth_props<32>, grid, dim3(256), 0, s, G, c, cs, rho_l, rho_g, mu_l, mu_g, rho, mu, kc,
                           tiles_x, ntiles);
    TBFG_HIP(hipGetLastError());
    return TBFG_OK;
}

}  // namespace tbfg
