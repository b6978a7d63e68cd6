// Differentiable SIB trajectory: forward with checkpoints and the hand-written
// reverse (adjoint) step on the device.
//
// Forward step (per site i; T = 0; Mentink et al. 2010 SIB as in the plain path):
//   B(x)_i = -(sum_d C_d x_{i+d}) - Z^T b_i,   C = sum_k theta_k C^(k)
//   a1 = f (B(m) + alpha m x B(m)),  mt = cay(m, a1),  p = (m + mt)/2
//   a2 = f (B(p) + alpha p x B(p)),  m' = cay(m, a2),   f = -dt / (2 (1+alpha^2) hbar)
// with cay(m, a) = (I + [a]x)^-1 (I - [a]x) m.  Reverse of one step, given
// g' = dL/dm':
//   d cay(m,a)/dm ^T g = cay(g, -a);  d cay/da ^T g = M(-a) g x (cay(m,a) + m),
//   M(-a) g = (g + a x g + (a.g) a)/(1+|a|^2);
//   a = f (B + alpha x x B):  gB = f (ga + alpha ga x x),  gx += f alpha (B x ga);
//   B(x) field: gx += -(C * gB) (the operator is symmetric: C_{-d}^T = C_d);
//   dL/dtheta_k += sum_i gB_i . (-(C^(k) x)_i);  dL/db_i += -Z gB_i.
// Kernels of a reverse step: R1 (stage-2 site math), R2 (transpose of the
// stage-2 field + stage-1 site math), R3 (transpose of the stage-1 field); R3
// of a step and R1 of the step before it run as one kernel.
// Checkpoints every `ckpt` steps; a segment is recomputed forward (storing m_n
// and p_n) before its reverse sweep.
#include <math.h>
#include <stdlib.h>
#include <string.h>

#include <algorithm>
#include <array>
#include <vector>

#include "mj_device.h"
#include "mj_internal.h"
#include "mj_stage_body.h"   // mj_block_sum, fused_wrap
#include "mj_adj_body.h"

#define MJ_ADJ_MAXP kAdjMaxParam

__global__ void __launch_bounds__(256) k_adj_sib1(const AdjArgs a)
{
    extern __shared__ double L[];
    adj_sib1_body<AdjRt>(a, L);
}

__global__ void __launch_bounds__(256) k_adj_sib2(const AdjArgs a)
{
    extern __shared__ double L[];
    adj_sib2_body<AdjRt>(a, L);
}

__global__ void __launch_bounds__(256) k_adj_sibf(const AdjArgs a)
{
    extern __shared__ double L[];
    adj_sibf_body<AdjRt>(a, L);
}

__global__ void __launch_bounds__(256) k_adj_r1(const AdjArgs a)
{
    extern __shared__ double L[];
    adj_r1_body<AdjRt>(a, L);
}

__global__ void __launch_bounds__(256) k_adj_r3r1(const AdjArgs a)
{
    extern __shared__ double L[];
    adj_r3r1_body<AdjRt>(a, L);
}

__global__ void __launch_bounds__(256) k_adj_r2(const AdjArgs a)
{
    extern __shared__ double L[];
    adj_r2_body<AdjRt>(a, L);
}

__global__ void __launch_bounds__(256) k_adj_r3(const AdjArgs a)
{
    extern __shared__ double L[];
    adj_r3_body<AdjRt>(a, L);
}

__global__ void k_adj_bmap(const double *bext, const double *h_aos, double *bmap, int64_t n, int64_t np)
{
    int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    for (int c = 0; c < 3; ++c) bmap[i + c * np] = bext[c] + (h_aos ? h_aos[3 * i + c] : 0.0);
}

__global__ void k_adj_aos_soa(const double *in, double *out, int64_t n, int64_t np, int to_soa)
{
    int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    for (int c = 0; c < 3; ++c) {
        if (to_soa) out[i + c * np] = in[3 * i + c];
        else out[3 * i + c] = in[i + c * np];
    }
}

// ---------------------------------------------------------------------------
// host side
// ---------------------------------------------------------------------------
struct AdjState {
    int nparam = 0;
    std::vector<std::vector<int>> pofs3;          // per parameter: offsets (3 each) of unit H blocks
    std::vector<std::vector<double>> pblk;        // per parameter: 9 per offset (H_MM(i, i+d) = A)
    // device
    int *d_ofs = nullptr, *d_pstart = nullptr, *d_pofs = nullptr;
    int *d_ofs0 = nullptr;           // the total stencil in the fused step's S0 layout (null: two kernels per step)
    size_t shm_fused = 0;
    double *d_cf = nullptr, *d_pcf = nullptr;
    double *d_cls = nullptr;         // compiled kernels: the total stencil's distinct values
    hipFunction_t fn[MJ_ADJ_KERNELS] = {};   // (null: ahead-of-time)
    JitRef mod;                              // their module
    AdjStencil built;                        // what they were compiled for (lattice and tile are the context's)
    bool built_fused = false;
    double *d_bext = nullptr, *d_bmap = nullptr;
    double *ckpt = nullptr;          // ncp * 3np
    double *segm = nullptr, *segp = nullptr;   // (ckpt + 1) * 3np and ckpt * 3np
    double *g = nullptr, *gB = nullptr, *gacc = nullptr, *gpd = nullptr, *ghmap = nullptr, *ppart = nullptr;
    int nofs = 0, rx = 0, ry = 0, rz = 0, bx = 0, by = 0, bz = 0, nblocks = 0;
    int nsteps = 0, ckpt_every = 0, ncp = 0;
    double alpha = 0.0, dt = 0.0;
    std::vector<double> theta;
    int ready = 0;                   // a forward pass has run to its end with the buffers and sizes held here
    int last_valid = 0;              // segm/segp hold the last segment of the forward pass
    // graphs of one full segment (ckpt_every steps): forward recompute, reverse sweep
    hipGraphExec_t g_fwd = nullptr, g_rev = nullptr;
};

static void adj_drop_graphs(AdjState *s)
{
    if (s->g_fwd) (void)hipGraphExecDestroy(s->g_fwd);
    if (s->g_rev) (void)hipGraphExecDestroy(s->g_rev);
    s->g_fwd = s->g_rev = nullptr;
}

#define ADJ(c) ((AdjState *)(c)->adj)

static void adj_free(AdjState *s)
{
    adj_drop_graphs(s);
    int *ip[] = {s->d_ofs, s->d_pstart, s->d_pofs, s->d_ofs0};
    for (int *p : ip)
        if (p) hipFree(p);
    double *dp[] = {s->d_cf, s->d_pcf, s->d_cls, s->d_bext, s->d_bmap, s->ckpt, s->segm, s->segp,
                    s->g, s->gB, s->gacc, s->gpd, s->ghmap, s->ppart};
    for (double *p : dp)
        if (p) hipFree(p);
}

void mj_adj_destroy(mj_ctx *c)
{
    if (!c->adj) return;
    adj_free(ADJ(c));
    delete ADJ(c);
    c->adj = nullptr;
}

static inline int canon_d(int d, int n, int periodic)
{
    if (!periodic) return d;
    d %= n;
    if (d < 0) d += n;
    if (2 * d > n) d -= n;
    return d;
}

// symmetrised stencil C_d = A_d + A_{-d}^T of a list of H blocks
static void symmetrise(const mj_ctx *c, const std::vector<int> &o3, const std::vector<double> &blk,
                       std::vector<std::array<int, 3>> &offs, std::vector<std::array<double, 9>> &C)
{
    auto slot = [&](int dx, int dy, int dz) -> std::array<double, 9> & {
        std::array<int, 3> o = {dx, dy, dz};
        for (size_t k = 0; k < offs.size(); ++k)
            if (offs[k] == o) return C[k];
        offs.push_back(o);
        C.push_back({0, 0, 0, 0, 0, 0, 0, 0, 0});
        return C.back();
    };
    for (size_t k = 0; k < blk.size() / 9; ++k) {
        int d[3], md[3];
        for (int q = 0; q < 3; ++q) {
            d[q] = canon_d(o3[3 * k + q], c->dim[q], c->periodic[q]);
            md[q] = canon_d(-o3[3 * k + q], c->dim[q], c->periodic[q]);
        }
        auto &f = slot(d[0], d[1], d[2]);
        for (int q = 0; q < 9; ++q) f[q] += blk[9 * k + q];
        auto &g = slot(md[0], md[1], md[2]);
        for (int r = 0; r < 3; ++r)
            for (int q = 0; q < 3; ++q) g[3 * r + q] += blk[9 * k + 3 * q + r];
    }
}

extern "C" int mj_adjoint_setup(mj_ctx *c, int nparam, const int *nofs, const int *ofs3, const double *blocks9)
{
    if (!c || nparam < 0 || nparam > MJ_ADJ_MAXP || (nparam && (!nofs || !ofs3 || !blocks9))) {
        mj_set_error("mj_adjoint_setup: bad argument (at most 13 parameters)");
        return MJ_EINVAL;
    }
    if (!c->has_z) {
        mj_set_error("mj_adjoint_setup: register the Zeeman (B-M) term first");
        return MJ_ESTATE;
    }
    mj_adj_destroy(c);
    AdjState *s = new AdjState();
    c->adj = s;
    s->nparam = nparam;
    int pos = 0;
    for (int k = 0; k < nparam; ++k) {
        s->pofs3.emplace_back(ofs3 + 3 * pos, ofs3 + 3 * (pos + nofs[k]));
        s->pblk.emplace_back(blocks9 + 9 * pos, blocks9 + 9 * (pos + nofs[k]));
        pos += nofs[k];
    }
    return MJ_OK;
}

static void adj_args(const mj_ctx *c, const AdjState *s, AdjArgs &a)
{
    memset(&a, 0, sizeof a);
    a.nx = c->dim[0];
    a.ny = c->dim[1];
    a.nz = c->dim[2];
    a.px = c->periodic[0];
    a.py = c->periodic[1];
    a.pz = c->periodic[2];
    a.bx = s->bx;
    a.by = s->by;
    a.bz = s->bz;
    a.rx = s->rx;
    a.ry = s->ry;
    a.rz = s->rz;
    a.ntx = (a.nx + a.bx - 1) / a.bx;
    a.nty = (a.ny + a.by - 1) / a.by;
    a.nblocks = a.ntx * a.nty * ((a.nz + a.bz - 1) / a.bz);
    a.np = c->np;
    a.nofs = s->nofs;
    a.ofs = s->d_ofs;
    a.ofs0 = s->d_ofs0;
    a.cf = s->d_cf;
    a.cls = s->d_cls;
    a.nparam = s->nparam;
    a.pstart = s->d_pstart;
    a.pofs = s->d_pofs;
    a.pcf = s->d_pcf;
    for (int q = 0; q < 9; ++q) a.z[q] = c->zblk[q];
    a.bmap = s->d_bmap;
    a.alpha = s->alpha;
    a.f = -0.5 * s->dt / ((1.0 + s->alpha * s->alpha) * MJ_HBAR);
}

static int adj_launch(const AdjState *s, int kind, const AdjArgs &a, int ntiles, hipStream_t st)
{
    const int T = (a.bx + 2 * a.rx) * (a.by + 2 * a.ry) * (a.bz + 2 * a.rz);
    const int nthr = a.bx * a.by * a.bz;
    size_t shm = sizeof(double) * ((size_t)3 * T * ntiles + nthr);
    if (kind != MJ_ADJ_SIBF && shm > 65536) {
        mj_set_error("adjoint: the stencil reach needs more LDS than a workgroup has");
        return MJ_ENOTSUP;
    }
    if (kind == MJ_ADJ_SIBF) shm = s->shm_fused;
    if (s->fn[kind]) {
        AdjArgs arg = a;
        void *params[] = {&arg};
        MJ_HIP_CHECK(hipModuleLaunchKernel(s->fn[kind], (unsigned)a.nblocks, 1, 1, (unsigned)nthr, 1, 1, (unsigned)shm, st,
                                           params, nullptr));
        return MJ_OK;
    }
    void (*const aot[MJ_ADJ_KERNELS])(const AdjArgs) = {k_adj_sib1, k_adj_sib2, k_adj_sibf, k_adj_r1,
                                                        k_adj_r2,   k_adj_r3r1, k_adj_r3};
    hipLaunchKernelGGL(aot[kind], dim3(a.nblocks), dim3(nthr), shm, st, a);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) {
        return mj_hip_fail(MJ_EHIP, std::string("adjoint kernel launch: ") + hipGetErrorString(e));
    }
    return MJ_OK;
}

#define ATRY(x)                     \
    do {                            \
        int r_ = (x);               \
        if (r_ != MJ_OK) return r_; \
    } while (0)

static int adj_alloc(double **p, size_t n)
{
    if (*p) hipFree(*p);
    *p = nullptr;
    if (hipMalloc(p, sizeof(double) * std::max<size_t>(n, 1)) != hipSuccess) {
        return mj_hip_fail(MJ_ENOMEM, "adjoint: device allocation failed");
    }
    return MJ_OK;
}

// The kernels compiled for the parameter set (mj_jit_adjoint), from kJitSites
// sites on (MJ_JIT=0 never, 1 always).  The values
// of the total stencil change with theta, its structure does not: places with
// the same unit coefficients in every parameter (up to one sign) hold the same
// value, places with none hold zero.  More than 64 values, or places whose sums
// round differently, keep the ahead-of-time kernels.
static int adj_compile(mj_ctx *c, AdjState *s, const std::vector<std::array<int, 3>> &offs,
                       const std::vector<std::array<double, 9>> &C,
                       const std::vector<std::vector<std::array<int, 3>>> &poffs,
                       const std::vector<std::vector<std::array<double, 9>>> &pC)
{
    hipFunction_t had[MJ_ADJ_KERNELS];   // the last pass's: the same ones while only the values change
    for (int k = 0; k < MJ_ADJ_KERNELS; ++k) {
        had[k] = s->fn[k];
        s->fn[k] = nullptr;
    }
    const char *env = getenv("MJ_JIT");
    if ((env && env[0] == '0') || (!(env && env[0] == '1') && c->n < kJitSites)) return MJ_OK;
    AdjStencil st;
    std::vector<std::vector<double>> keys;
    std::vector<double> vals;
    for (size_t e = 0; e < offs.size(); ++e) {
        st.o3.insert(st.o3.end(), offs[e].begin(), offs[e].end());
        for (int q = 0; q < 9; ++q) {
            std::vector<double> key(s->nparam, 0.0);
            for (int k = 0; k < s->nparam; ++k)
                for (size_t j = 0; j < poffs[k].size(); ++j)
                    if (poffs[k][j] == offs[e]) key[k] = pC[k][j][q];
            double lead = 0.0;
            for (double v : key)
                if (lead == 0.0) lead = v;
            if (lead == 0.0) {
                if (C[e][q] != 0.0) return MJ_OK;
                st.cls.push_back(0);
                continue;
            }
            const double sign = lead < 0.0 ? -1.0 : 1.0;
            for (double &v : key) v = sign * v + 0.0;
            size_t i = std::find(keys.begin(), keys.end(), key) - keys.begin();
            if (i == keys.size()) {
                keys.push_back(key);
                vals.push_back(sign * C[e][q]);
            }
            if (vals[i] != sign * C[e][q]) return MJ_OK;
            st.cls.push_back((int)sign * (int)(i + 1));
        }
    }
    if (vals.size() > 64) return MJ_OK;
    for (int k = 0; k < s->nparam; ++k) {
        st.po3.emplace_back();
        st.pblk.emplace_back();
        for (size_t j = 0; j < poffs[k].size(); ++j) {
            st.po3[k].insert(st.po3[k].end(), poffs[k][j].begin(), poffs[k][j].end());
            st.pblk[k].insert(st.pblk[k].end(), pC[k][j].begin(), pC[k][j].end());
        }
    }
    const int b[3] = {s->bx, s->by, s->bz}, r[3] = {s->rx, s->ry, s->rz};
    const bool fused = s->d_ofs0 != nullptr, same = had[MJ_ADJ_R2] && s->built_fused == fused && s->built == st;
    if (!same) ATRY(adj_alloc(&s->d_cls, vals.size()));   // as many values as the structure has
    if (!vals.empty())
        MJ_HIP_CHECK(hipMemcpy(s->d_cls, vals.data(), sizeof(double) * vals.size(), hipMemcpyHostToDevice));
    if (same) {
        std::copy(had, had + MJ_ADJ_KERNELS, s->fn);
        return MJ_OK;
    }
    ATRY(mj_jit_adjoint(c, st, b, r, fused, &s->mod, s->fn));
    s->built = st;
    s->built_fused = fused;
    return MJ_OK;
}

// one forward SIB step from x_in to x_out (SoA), storing the midpoint in pbuf:
// one fused kernel when its tiles fit, else the two stage kernels
static int adj_step(mj_ctx *c, AdjState *s, const double *xin, double *pbuf, double *xout)
{
    AdjArgs a;
    adj_args(c, s, a);
    a.x = xin;
    a.out0 = pbuf;
    if (s->d_ofs0) {
        a.out1 = xout;
        return adj_launch(s, MJ_ADJ_SIBF, a, 1, c->stream);
    }
    ATRY(adj_launch(s, MJ_ADJ_SIB1, a, 1, c->stream));
    a.x = pbuf;
    a.m = xin;
    a.out0 = xout;
    return adj_launch(s, MJ_ADJ_SIB2, a, 1, c->stream);
}

// `len` steps of one segment: segm[q] -> (segp[q], segm[q+1]); a full segment
// replays the captured graph (captured on first use after each forward set-up)
static int adj_segment_fwd(mj_ctx *c, AdjState *s, int len)
{
    const size_t n3 = 3 * (size_t)c->np;
    auto enqueue = [&](int n) -> int {
        for (int q = 0; q < n; ++q) ATRY(adj_step(c, s, s->segm + n3 * q, s->segp + n3 * q, s->segm + n3 * (q + 1)));
        return MJ_OK;
    };
    if (len != s->ckpt_every) return enqueue(len);
    if (!s->g_fwd) {
        hipGraph_t g = nullptr;
        MJ_HIP_CHECK(hipStreamBeginCapture(c->stream, hipStreamCaptureModeThreadLocal));
        int rc = enqueue(len);
        hipError_t e = hipStreamEndCapture(c->stream, &g);
        if (rc != MJ_OK || e != hipSuccess) {
            if (g) (void)hipGraphDestroy(g);
            if (rc != MJ_OK) return rc;
            return mj_hip_fail(MJ_EHIP, std::string("adjoint forward capture: ") + hipGetErrorString(e));
        }
        e = hipGraphInstantiate(&s->g_fwd, g, nullptr, nullptr, 0);
        (void)hipGraphDestroy(g);
        if (e != hipSuccess) {
            s->g_fwd = nullptr;
            return mj_hip_fail(MJ_EHIP, std::string("adjoint forward graph: ") + hipGetErrorString(e));
        }
    }
    MJ_HIP_CHECK(hipGraphLaunch(s->g_fwd, c->stream));
    return MJ_OK;
}

extern "C" int mj_adjoint_forward(mj_ctx *c, const double *theta, const double *bext, const double *hmap_dev,
                                  const double *m0_dev, int nsteps, double timestep, double damping, int ckpt_every,
                                  double *mfinal_dev)
{
    if (!c || !c->adj || (!theta && ADJ(c)->nparam) || !bext || !m0_dev || !mfinal_dev || nsteps < 1 ||
        ckpt_every < 1 || !(timestep > 0.0) || !(damping >= 0.0)) {
        mj_set_error("mj_adjoint_forward: bad argument or mj_adjoint_setup not called");
        return MJ_EINVAL;
    }
    MJ_HIP_CHECK(hipSetDevice(c->device));
    AdjState *s = ADJ(c);
    s->ready = 0;
    adj_drop_graphs(s);   // their launches hold the buffers and kernels replaced below
    s->theta.assign(theta, theta + s->nparam);
    s->nsteps = nsteps;
    s->ckpt_every = ckpt_every;
    s->alpha = damping;
    s->dt = timestep;
    // total and unit stencils (symmetrised), LDS offsets for the tile
    std::vector<std::array<int, 3>> offs;
    std::vector<std::array<double, 9>> C;
    std::vector<int> all3;
    std::vector<double> allb;
    for (int k = 0; k < s->nparam; ++k) {
        all3.insert(all3.end(), s->pofs3[k].begin(), s->pofs3[k].end());
        for (size_t q = 0; q < s->pblk[k].size(); ++q) allb.push_back(theta[k] * s->pblk[k][q]);
    }
    symmetrise(c, all3, allb, offs, C);
    std::vector<std::vector<std::array<int, 3>>> poffs(s->nparam);
    std::vector<std::vector<std::array<double, 9>>> pC(s->nparam);
    for (int k = 0; k < s->nparam; ++k) symmetrise(c, s->pofs3[k], s->pblk[k], poffs[k], pC[k]);
    s->rx = s->ry = s->rz = 0;
    for (auto &o : offs) {
        s->rx = std::max(s->rx, std::abs(o[0]));
        s->ry = std::max(s->ry, std::abs(o[1]));
        s->rz = std::max(s->rz, std::abs(o[2]));
    }
    // tile: up to 256 sites, smaller (down to one wavefront) while that gives
    // fewer than 512 workgroups, so that small lattices still spread over the CUs
    {
        const int px = 1 << (int)ceil(log2((double)std::max(c->dim[0], 1)));
        const int py = 1 << (int)ceil(log2((double)std::max(c->dim[1], 1)));
        int nthr = 256;
        while (nthr > 64 && (int64_t)c->n / nthr < 512) nthr >>= 1;
        s->bx = std::min(px, nthr / 8);   // 32x8, 16x8 or 8x8
        s->by = std::max(1, std::min(nthr / s->bx, py));
        s->bz = 1;
    }
    const int sx = s->bx + 2 * s->rx, sy = s->by + 2 * s->ry;
    auto lofs = [&](const std::array<int, 3> &o) { return o[2] * sx * sy + o[1] * sx + o[0]; };
    std::vector<int> hofs;
    std::vector<double> hcf;
    for (size_t k = 0; k < offs.size(); ++k) {
        hofs.push_back(lofs(offs[k]));
        hcf.insert(hcf.end(), C[k].begin(), C[k].end());
    }
    std::vector<int> hps(1, 0), hpofs;
    std::vector<double> hpcf;
    for (int k = 0; k < s->nparam; ++k) {
        for (size_t q = 0; q < poffs[k].size(); ++q) {
            hpofs.push_back(lofs(poffs[k][q]));
            hpcf.insert(hpcf.end(), pC[k][q].begin(), pC[k][q].end());
        }
        hps.push_back((int)hpofs.size());
    }
    s->nofs = (int)hofs.size();
    int *ip[4] = {s->d_ofs, s->d_pstart, s->d_pofs, s->d_ofs0};
    for (int *p : ip)
        if (p) hipFree(p);
    s->d_ofs0 = nullptr;
    // the fused forward step (MJ_ADJ_FUSE=0: two kernels per step; the same bits)
    {
        const int s0x = s->bx + 4 * s->rx, s0y = s->by + 4 * s->ry, s0z = s->bz + 4 * s->rz;
        const size_t shm = sizeof(double) * 3 * ((size_t)s0x * s0y * s0z + (size_t)sx * sy * (s->bz + 2 * s->rz));
        const char *fe = getenv("MJ_ADJ_FUSE");
        if (shm <= 65536 && !(fe && fe[0] == '0')) {
            std::vector<int> hofs0;
            for (auto &o : offs) hofs0.push_back(o[2] * s0x * s0y + o[1] * s0x + o[0]);
            MJ_HIP_CHECK(hipMalloc(&s->d_ofs0, sizeof(int) * std::max<size_t>(1, hofs0.size())));
            if (!hofs0.empty())
                MJ_HIP_CHECK(hipMemcpy(s->d_ofs0, hofs0.data(), sizeof(int) * hofs0.size(), hipMemcpyHostToDevice));
            s->shm_fused = shm;
        }
    }
    MJ_HIP_CHECK(hipMalloc(&s->d_ofs, sizeof(int) * std::max<size_t>(1, hofs.size())));
    MJ_HIP_CHECK(hipMalloc(&s->d_pstart, sizeof(int) * hps.size()));
    MJ_HIP_CHECK(hipMalloc(&s->d_pofs, sizeof(int) * std::max<size_t>(1, hpofs.size())));
    ATRY(adj_alloc(&s->d_cf, hcf.size()));
    ATRY(adj_alloc(&s->d_pcf, hpcf.size()));
    if (!hofs.empty()) {
        MJ_HIP_CHECK(hipMemcpy(s->d_ofs, hofs.data(), sizeof(int) * hofs.size(), hipMemcpyHostToDevice));
        MJ_HIP_CHECK(hipMemcpy(s->d_cf, hcf.data(), sizeof(double) * hcf.size(), hipMemcpyHostToDevice));
    }
    MJ_HIP_CHECK(hipMemcpy(s->d_pstart, hps.data(), sizeof(int) * hps.size(), hipMemcpyHostToDevice));
    if (!hpofs.empty()) {
        MJ_HIP_CHECK(hipMemcpy(s->d_pofs, hpofs.data(), sizeof(int) * hpofs.size(), hipMemcpyHostToDevice));
        MJ_HIP_CHECK(hipMemcpy(s->d_pcf, hpcf.data(), sizeof(double) * hpcf.size(), hipMemcpyHostToDevice));
    }
    ATRY(adj_compile(c, s, offs, C, poffs, pC));
    // buffers
    const size_t n3 = 3 * (size_t)c->np;
    s->ncp = (nsteps + ckpt_every - 1) / ckpt_every;
    ATRY(adj_alloc(&s->d_bext, 3));
    ATRY(adj_alloc(&s->d_bmap, n3));
    ATRY(adj_alloc(&s->ckpt, n3 * s->ncp));
    ATRY(adj_alloc(&s->segm, n3 * (ckpt_every + 1)));
    ATRY(adj_alloc(&s->segp, n3 * ckpt_every));
    MJ_HIP_CHECK(hipMemcpy(s->d_bext, bext, sizeof(double) * 3, hipMemcpyHostToDevice));
    const unsigned nb = (unsigned)((c->n + 255) / 256);
    hipLaunchKernelGGL(k_adj_bmap, dim3(nb), dim3(256), 0, c->stream, s->d_bext, hmap_dev, s->d_bmap, c->n, c->np);
    // forward with checkpoints: segment by segment, states kept as in the recompute
    s->last_valid = 0;
    hipLaunchKernelGGL(k_adj_aos_soa, dim3(nb), dim3(256), 0, c->stream, m0_dev, s->segm, c->n, c->np, 1);
    int len = 0;
    for (int seg = 0; seg < s->ncp; ++seg) {
        len = std::min(ckpt_every, nsteps - seg * ckpt_every);
        if (seg > 0)
            MJ_HIP_CHECK(hipMemcpyAsync(s->segm, s->segm + n3 * ckpt_every, sizeof(double) * n3,
                                        hipMemcpyDeviceToDevice, c->stream));
        MJ_HIP_CHECK(hipMemcpyAsync(s->ckpt + n3 * seg, s->segm, sizeof(double) * n3, hipMemcpyDeviceToDevice,
                                    c->stream));
        ATRY(adj_segment_fwd(c, s, len));
    }
    s->last_valid = 1;
    hipLaunchKernelGGL(k_adj_aos_soa, dim3(nb), dim3(256), 0, c->stream, s->segm + n3 * len, mfinal_dev, c->n, c->np,
                       0);
    MJ_HIP_CHECK(hipStreamSynchronize(c->stream));
    s->ready = 1;
    return MJ_OK;
}

// reverse sweep over one segment (q = len-1 .. 0): R1, R2, R3 per step
static int adj_segment_rev(mj_ctx *c, AdjState *s, int len)
{
    const size_t n3 = 3 * (size_t)c->np;
    AdjArgs a0;
    adj_args(c, s, a0);
    a0.ppart = s->ppart;
    a0.ghmap = s->ghmap;
    double *gB2 = s->gB, *gB1 = s->gB + n3;
    auto enqueue = [&](int n) -> int {
        {
            AdjArgs a = a0;          // R1 of the segment's last step: stage-2 site math
            a.x = s->segp + n3 * (n - 1);
            a.m = s->segm + n3 * (n - 1);
            a.m1 = s->segm + n3 * n;
            a.gin = s->g;
            a.out0 = gB2;
            a.out1 = s->gacc;
            a.out2 = s->gpd;
            ATRY(adj_launch(s, MJ_ADJ_R1, a, 1, c->stream));
        }
        for (int q = n - 1; q >= 0; --q) {
            AdjArgs b = a0;          // R2: transpose of the stage-2 field + stage-1 site math
            b.x = gB2;
            b.m = s->segm + n3 * q;
            b.gacc_in = s->gacc;
            b.gpd_in = s->gpd;
            b.out0 = gB1;
            b.out1 = s->gacc;        // own-site read-then-write
            ATRY(adj_launch(s, MJ_ADJ_R2, b, 2, c->stream));
            if (q > 0) {             // R3 of step q + R1 of step q-1
                AdjArgs f = a0;
                f.x = gB1;
                f.x2 = s->segp + n3 * (q - 1);
                f.gacc_in = s->gacc;
                f.m = s->segm + n3 * (q - 1);
                f.m1 = s->segm + n3 * q;
                f.out0 = gB2;
                f.out1 = s->gacc;    // own-site read-then-write
                f.out2 = s->gpd;
                ATRY(adj_launch(s, MJ_ADJ_R3R1, f, 2, c->stream));
            } else {                 // R3 of the segment's first step: lambda to memory
                AdjArgs r = a0;
                r.ppart = nullptr;
                r.ghmap = nullptr;
                r.x = gB1;
                r.gacc_in = s->gacc;
                r.out0 = s->g;
                ATRY(adj_launch(s, MJ_ADJ_R3, r, 1, c->stream));
            }
        }
        return MJ_OK;
    };
    if (len != s->ckpt_every) return enqueue(len);
    if (!s->g_rev) {
        hipGraph_t g = nullptr;
        MJ_HIP_CHECK(hipStreamBeginCapture(c->stream, hipStreamCaptureModeThreadLocal));
        int rc = enqueue(len);
        hipError_t e = hipStreamEndCapture(c->stream, &g);
        if (rc != MJ_OK || e != hipSuccess) {
            if (g) (void)hipGraphDestroy(g);
            if (rc != MJ_OK) return rc;
            return mj_hip_fail(MJ_EHIP, std::string("adjoint reverse capture: ") + hipGetErrorString(e));
        }
        e = hipGraphInstantiate(&s->g_rev, g, nullptr, nullptr, 0);
        (void)hipGraphDestroy(g);
        if (e != hipSuccess) {
            s->g_rev = nullptr;
            return mj_hip_fail(MJ_EHIP, std::string("adjoint reverse graph: ") + hipGetErrorString(e));
        }
    }
    MJ_HIP_CHECK(hipGraphLaunch(s->g_rev, c->stream));
    return MJ_OK;
}

extern "C" int mj_adjoint_backward(mj_ctx *c, const double *gfinal_dev, double *gtheta, double *gbext,
                                   double *ghmap_dev, double *gm0_dev)
{
    if (!c || !c->adj || !gfinal_dev || (!gtheta && ADJ(c)->nparam) || !gbext) {
        mj_set_error("mj_adjoint_backward: bad argument or no forward pass");
        return MJ_EINVAL;
    }
    AdjState *s = ADJ(c);
    if (!s->ready) {
        mj_set_error("mj_adjoint_backward: call mj_adjoint_forward first");
        return MJ_ESTATE;
    }
    MJ_HIP_CHECK(hipSetDevice(c->device));
    const size_t n3 = 3 * (size_t)c->np;
    AdjArgs a0;
    adj_args(c, s, a0);
    const int nv = s->nparam + 3;
    if (!s->g) {   // kept until the next mj_adjoint_setup (sizes fixed per context and parameter set)
        ATRY(adj_alloc(&s->gB, 2 * n3));
        ATRY(adj_alloc(&s->gacc, n3));
        ATRY(adj_alloc(&s->gpd, n3));
        ATRY(adj_alloc(&s->ghmap, n3));
        ATRY(adj_alloc(&s->ppart, (size_t)a0.nblocks * nv));
        ATRY(adj_alloc(&s->g, n3));   // last: there only when all are
    }
    MJ_HIP_CHECK(hipMemsetAsync(s->ghmap, 0, sizeof(double) * n3, c->stream));
    MJ_HIP_CHECK(hipMemsetAsync(s->ppart, 0, sizeof(double) * a0.nblocks * nv, c->stream));
    const unsigned nb = (unsigned)((c->n + 255) / 256);
    hipLaunchKernelGGL(k_adj_aos_soa, dim3(nb), dim3(256), 0, c->stream, gfinal_dev, s->g, c->n, c->np, 1);
    for (int seg = s->ncp - 1; seg >= 0; --seg) {
        const int j0 = seg * s->ckpt_every;
        const int len = std::min(s->ckpt_every, s->nsteps - j0);
        if (!(seg == s->ncp - 1 && s->last_valid)) {   // the forward pass left the last segment in place
            MJ_HIP_CHECK(hipMemcpyAsync(s->segm, s->ckpt + n3 * seg, sizeof(double) * n3, hipMemcpyDeviceToDevice,
                                        c->stream));
            ATRY(adj_segment_fwd(c, s, len));
        }
        ATRY(adj_segment_rev(c, s, len));
    }
    s->last_valid = s->ncp == 1;
    std::vector<double> part((size_t)a0.nblocks * nv);
    MJ_HIP_CHECK(hipMemcpyAsync(part.data(), s->ppart, sizeof(double) * part.size(), hipMemcpyDeviceToHost, c->stream));
    if (ghmap_dev)
        hipLaunchKernelGGL(k_adj_aos_soa, dim3(nb), dim3(256), 0, c->stream, s->ghmap, ghmap_dev, c->n, c->np, 0);
    if (gm0_dev) hipLaunchKernelGGL(k_adj_aos_soa, dim3(nb), dim3(256), 0, c->stream, s->g, gm0_dev, c->n, c->np, 0);
    MJ_HIP_CHECK(hipStreamSynchronize(c->stream));
    for (int q = 0; q < nv; ++q) {
        double t = 0.0;
        for (int b = 0; b < a0.nblocks; ++b) t += part[(size_t)b * nv + q];
        if (q < s->nparam) gtheta[q] = t;
        else gbext[q - s->nparam] = t;
    }
    return MJ_OK;
}
