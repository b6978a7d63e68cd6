// Device code of the Monte Carlo passes shared by the ahead-of-time kernels
// (mj_mc.hip) and those compiled per Hamiltonian (mj_jit.hip).
#pragma once

constexpr uint32_t kMcStream = 0x4D430000u;   // counter word 3 of the Monte Carlo draws
constexpr int kMcIsing = 1;            // MJ_MC_ISING
constexpr int kMcThreads = 256;
constexpr int kMcVals = 32;

struct McState {
    double cone, cos_cone, acc, nb, rate;
};

struct McArgs {
    double *m;              // state, SoA
    int64_t np;
    int nx, ny, nz, px, py, pz;
    int p, ca, cb, color;
    int64_t nthreads;
    int n_iso, n_dm, n_gen;
    const int *o3;          // offsets (3 each), classes iso | dm | gen, no d = 0
    const double *cf;       // iso: s; dm: s, w; gen: 9
    double c0[9];           // on-site C_0 = A_0 + A_0^T
    int bmode;
    double zb[3], z[9];
    const double *bmap;
    double kT;
    uint64_t seed, sweep;
    int sampler;
    McState *st;
    double *acc_part;
    // compiled passes: acc_part counts a whole sweep (each pass adds to its
    // blocks' entries); the first pass of a sweep makes st of st_in and the
    // fold_n partials (per replica) of the sweep before, and every block of it
    // its own copy of the cone
    int first;
    const McState *st_in;
    const double *fold_part;
    int fold_n, adapt;
    double n_done, n_next;
    // replicas (parallel tempering): blockIdx.y is the replica; its state, counters,
    // partials and temperature are at these strides (kT_rep null: one temperature)
    int64_t rep_cm, rep_part;
    const double *kT_rep;
    // colour-major copy of the state used by the passes: slot of site (x, y, z) =
    // class * R * W + (y + ny z) * W + x / p, R = ny nz rows, W = ceil(nx / p)
    double *cm;
    const double *cbmap;    // per-site field map in the same order (or null)
    int64_t cs;             // component stride of cm (p R W)
    int W;
    const int *csh;         // per stencil entry: class shift (dx + a dy + b dz) mod p
    const double *cf9;      // every stencil entry as a full 3x3 block (passes)
    // rows at least the stencil reach from the y and z boundaries take the
    // neighbour slots from a table: slot + tab[x0 * ne + e] (+-W across x)
    int fast, ne;
    const int *tab;
    int ylo, yhi, zlo, zhi;
    // single-site energies
    int64_t nsites;
    const int64_t *sites;
    const double *spins;    // AoS 3 per site, or null for the current spin
    double *e_out;
    double vals[kMcVals];   // compiled kernels: the stencil's distinct values
};

__device__ __forceinline__ v3 mc_zeeman(const McArgs &a, const double *bmap, int64_t stride, int64_t i)
{
    if (a.bmode == 1) return mk3(a.zb[0], a.zb[1], a.zb[2]);
    if (a.bmode == 2) {
        const double bx = bmap[i], by = bmap[i + stride], bz = bmap[i + 2 * stride];
        return mk3((bx * a.z[0] + by * a.z[3]) + bz * a.z[6], (bx * a.z[1] + by * a.z[4]) + bz * a.z[7],
                   (bx * a.z[2] + by * a.z[5]) + bz * a.z[8]);
    }
    return mk3(0.0, 0.0, 0.0);
}

// energy of site i with spin s: s.(h + z) + s^T C_0 s / 2
__device__ __forceinline__ double mc_site_energy(const McArgs &a, v3 s, v3 h)
{
    const double *c = a.c0;
    const double qx = (c[0] * s.x + c[1] * s.y) + c[2] * s.z;
    const double qy = (c[3] * s.x + c[4] * s.y) + c[5] * s.z;
    const double qz = (c[6] * s.x + c[7] * s.y) + c[8] * s.z;
    return dot3(s, h) + 0.5 * dot3(s, mk3(qx, qy, qz));
}

// sphereft: uniform in the cap of half-angle `cone` around s (cc = cos cone)
__device__ __forceinline__ v3 mc_sphere(v3 s, double cc, double u1, double u2)
{
    const double ct = u1 + cc * (1.0 - u1);
    const double st = sqrt(1.0 - ct * ct);
    double sp, cp;
    mj_sincos2pi(u2, &sp, &cp);
    const double cti = s.z;
    const double rr = s.x * s.x + s.y * s.y;
    const double sti = sqrt(rr);
    double cpi = 1.0, spi = 0.0;
    if (!(rr < 0.00001)) {
        cpi = s.x / sqrt(rr);
        spi = s.y / sqrt(rr);
    }
    const double t = st * sp * cti + ct * sti;
    const double ny = st * cp * cpi + t * spi;
    const double nx = -(st * cp * spi) + t * cpi;
    const double nz = -(st * sp * sti) + ct * cti;
    const double ss = sqrt((nx * nx + ny * ny) + nz * nz);
    return mk3(nx / ss, ny / ss, nz / ss);
}

// acceptance counters after a sweep (s accepted of n_done), and the cone for the
// next sweep's n_next proposals (cone_update n_next times at the running rate)
__device__ __forceinline__ void mc_fold_state(McState *st, double s, double n_done, double n_next, int adapt)
{
    const double acc = st->acc + s, nb = st->nb + n_done;
    st->acc = acc;
    st->nb = nb;
    if (nb > 0.0) st->rate = acc / nb;
    if (adapt && n_next > 0.0) {
        const double pi = 3.14159265358979323846264338327950288;   // constant.f90:32
        const double rate = st->rate;
        double cone = st->cone;
        if (rate > 0.5 && cone < pi) {
            const double k = fmin(ceil((pi - cone) / 1.0e-4), n_next);
            cone = cone + k * 1.0e-4;
        } else if (rate < 0.5 && cone > 0.01) {
            const double k = fmin(ceil((cone - 0.01) / 1.0e-4), n_next);
            cone = cone - k * 1.0e-4;
        }
        st->cone = cone;
        st->cos_cone = cos(cone);
    }
}

// the new spin proposed for site i (spin s)
__device__ __forceinline__ v3 mc_propose(const McArgs &a, int rep, int64_t i, v3 s, double cc, uint32_t c[4])
{
    c[0] = (uint32_t)i;
    c[1] = (uint32_t)a.sweep;
    c[2] = (uint32_t)(a.sweep >> 32);
    c[3] = kMcStream + (uint32_t)rep;
    philox4x32_10(c, (uint32_t)a.seed, (uint32_t)(a.seed >> 32));
    const double two_m32 = 2.3283064365386962890625e-10;
    if (a.sampler == kMcIsing) return mk3(-s.x, -s.y, -s.z);
    return mc_sphere(s, cc, (double)c[0] * two_m32, (double)c[1] * two_m32);
}

// accept (MCstep.f90:70-88) on the pair field pf of the site
__device__ __forceinline__ bool mc_accept(const McArgs &a, v3 s, v3 sn, v3 pf, int64_t slot, double kT, uint32_t c2)
{
    const v3 zf = mc_zeeman(a, a.cbmap, a.cs, slot);
    const v3 h = mk3(pf.x + zf.x, pf.y + zf.y, pf.z + zf.z);
    const double de = mc_site_energy(a, sn, h) - mc_site_energy(a, s, h);
    bool acc = de < 0.0;
    if (!acc && kT > 0.0) {
        const double tmp = fmax(-de / kT, -200.0);
        acc = c2 == 0u || mj_log01((double)c2 * 2.3283064365386962890625e-10) < tmp;
    }
    return acc;
}

// One colour class, the stencil and the lattice compile-time (G of mj_jit.hip).
// The loads of a site are in flight before the proposal is computed.
template <class G>
__device__ __forceinline__ void mc_pass_body(const McArgs &a)
{
    __shared__ int cnt[kMcThreads / 64];
    __shared__ double red[kMcThreads], cone;
    const int rep = blockIdx.y;
    double *cm = a.cm + rep * a.rep_cm;
    const double kT = a.kT_rep ? a.kT_rep[rep] : a.kT;
    double cc = 0.0;
    if (a.first) {
        double v = 0.0;
        for (int i = threadIdx.x; i < a.fold_n; i += kMcThreads) v += a.fold_part[rep * a.rep_part + i];
        v = mj_block_sum(v, red, kMcThreads);
        if (threadIdx.x == 0) {
            McState st = a.st_in[rep];
            mc_fold_state(&st, v, a.n_done, a.n_next, a.adapt);
            cone = st.cos_cone;
            if (blockIdx.x == 0) a.st[rep] = st;
        }
        __syncthreads();
        cc = cone;
    } else {
        cc = a.st[rep].cos_cone;
    }
    // bands of rows stay on one XCD: its L2 holds most of their neighbours
    const int bid = mj_xcd_remap(blockIdx.x, gridDim.x);
    const int t = bid * kMcThreads + (int)threadIdx.x;
    bool acc = false;
    if (t < G::kRows * G::kW) {
        const int row = t / G::kW, jj = t % G::kW, y = row % G::kNy, z = row / G::kNy;
        const int x0 = G::first(a.color, y, z), x = x0 + jj * G::kP;
        if (x < G::kNx) {
            const int64_t slot = (int64_t)a.color * (G::kRows * G::kW) + t;
            const v3 s = mk3(cm[slot], cm[slot + a.cs], cm[slot + 2 * a.cs]);
            uint32_t c[4];
            v3 sn;
            const v3 pf = G::field(a, cm, a.color, x0, jj, x, y, z, [&]() __attribute__((always_inline)) {
                sn = mc_propose(a, rep, (int64_t)x + (int64_t)G::kNx * row, s, cc, c);
            });
            acc = mc_accept(a, s, sn, pf, slot, kT, c[2]);
            if (acc) {
                cm[slot] = sn.x;
                cm[slot + a.cs] = sn.y;
                cm[slot + 2 * a.cs] = sn.z;
            }
        }
    }
    const int n = __popcll(__ballot(acc));
    if (threadIdx.x % 64 == 0) cnt[threadIdx.x / 64] = n;
    __syncthreads();
    if (threadIdx.x == 0) {
        int v = 0;
        for (int w = 0; w < kMcThreads / 64; ++w) v += cnt[w];
        double *part = a.acc_part + rep * a.rep_part + blockIdx.x;
        *part = a.first ? (double)v : *part + (double)v;
    }
}

// E and M of every replica: per-block partials
template <class G>
__device__ __forceinline__ void mc_energy_body(const McArgs &a, double *part)
{
    __shared__ double red[kMcThreads];
    const int rep = blockIdx.y;
    const double *cm = a.cm + rep * a.rep_cm;
    const int t = (int)blockIdx.x * kMcThreads + (int)threadIdx.x;
    double v[4] = {0.0, 0.0, 0.0, 0.0};
    if (t < G::kP * G::kRows * G::kW) {
        const int k = t / (G::kRows * G::kW), rest = t % (G::kRows * G::kW);
        const int row = rest / G::kW, jj = rest % G::kW, y = row % G::kNy, z = row / G::kNy;
        const int x0 = G::first(k, y, z), x = x0 + jj * G::kP;
        if (x < G::kNx) {
            const v3 m = mk3(cm[t], cm[t + a.cs], cm[t + 2 * a.cs]);
            const v3 pf = G::field(a, cm, k, x0, jj, x, y, z, []() {});
            const v3 zf = mc_zeeman(a, a.cbmap, a.cs, t);
            v[0] = mc_site_energy(a, m, mk3(0.5 * pf.x + zf.x, 0.5 * pf.y + zf.y, 0.5 * pf.z + zf.z));
            v[1] = m.x;
            v[2] = m.y;
            v[3] = m.z;
        }
    }
    const int64_t base = ((int64_t)rep * gridDim.x + blockIdx.x) * 4;
    for (int q = 0; q < 4; ++q) {
        const double sq = mj_block_sum(v[q], red, kMcThreads);
        if (threadIdx.x == 0) part[base + q] = sq;
    }
}
