// Internal declarations shared by the library's translation units.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <memory>
#include <string>
#include <vector>

#include "../../include/matjes_hip.h"

void mj_set_error(const std::string &msg);

// a HIP call failed: the message, and the error taken off the runtime's record,
// where the next launch's check would find it again
inline int mj_hip_fail(int code, const std::string &msg)
{
    (void)hipGetLastError();
    mj_set_error(msg);
    return code;
}

#define MJ_HIP_CHECK(call)                                                                                    \
    do {                                                                                                      \
        hipError_t e_ = (call);                                                                               \
        if (e_ != hipSuccess) return mj_hip_fail(MJ_EHIP, std::string(#call) + ": " + hipGetErrorString(e_)); \
    } while (0)

#include "mj_kargs.h"

struct DipolarFFT;  // mj_fft.hip

// Pinned memory between a caller's arrays and the device, kept with its object:
// the kernels that lay a field out read and write it themselves.
struct MjHostStage {
    double *buf = nullptr;
    int64_t half = 0;                  // doubles of a chunk, whole sites
    int chunks = 0;                    // 1 (the object's fields fit in one) or 2
    hipEvent_t ev[2] = {nullptr, nullptr};
};
int mj_stage_alloc(MjHostStage &h, int64_t n3);
void mj_stage_free(MjHostStage &h);
// n sites of a field (SoA, stride np) to / from the caller's AoS array (up: 3 n <= half); |x| < eps goes out as 0.
// Both end synchronised.
int mj_download(MjHostStage &h, const double *soa, int64_t n, int64_t np, double eps, double *host, hipStream_t s);
int mj_upload(MjHostStage &h, const double *host, double *soa, int64_t n, int64_t np, hipStream_t s);
// count doubles as they are
int mj_download_flat(MjHostStage &h, const double *dev, int64_t count, double *host, hipStream_t s);

struct mj_ctx {
    MjHostStage host;
    int device = 0;
    int dim[3] = {1, 1, 1};
    int periodic[3] = {0, 0, 0};
    int dim_mode = 3;
    int64_t n = 0;      // sites
    int64_t np = 0;     // padded SoA stride
    hipStream_t stream = nullptr;

    // state buffers (SoA, 3*np doubles each)
    double *A = nullptr, *Bb = nullptr, *Db = nullptr, *Fb = nullptr, *Nb = nullptr;
    double *epart = nullptr;   // 2 x max blocks
    double *evals = nullptr;   // energies device array
    int64_t evals_cap = 0;
    int epart_cap = 0;
    int state_set = 0;

    // Hamiltonian (host accumulation)
    // each registered M-M term on its own (energy per term); mm_terms_generic
    // when a term is not translation invariant
    struct MMTerm {
        std::vector<int> ofs3;
        std::vector<double> blk9;
    };
    std::vector<MMTerm> mm_terms;
    int mm_terms_generic = 0;
    std::vector<int> st_ofs;           // 3 per entry
    std::vector<double> st_blk;        // 9 per entry (H_MM(i,i+d) blocks, summed)
    int has_mm = 0;
    int mm_generic = 0;                // 1: generic CSR path
    std::vector<int64_t> g_rows;       // generic: 0-based COO of H_MM
    std::vector<int> g_cols;
    std::vector<double> g_vals;
    double zblk[9] = {0};
    int has_z = 0;
    std::vector<double> bvec;          // B order parameter (AoS 3N) or 3
    int bmode = 0;

    // device stencil
    int *d_ofs = nullptr;
    double *d_cf = nullptr;
    int n_iso = 0, n_dm = 0, n_gen = 0;
    std::vector<int> h_ofs3;           // host copy of the classified stencil: offsets (3 each) and
    std::vector<double> h_cf;          // coefficients in the order iso | dm | gen
    std::vector<int> h_ord;            // the entries in the order every kernel sums them, by (dz, dy, dx)
    std::vector<double> h_blk;         // their 3x3 blocks in that order (KArgs::cf)
    int rx = 0, ry = 0, rz = 0;
    int bx = 0, by = 0, bz = 0;        // 0: auto
    int dirty = 1;
    double zb[3] = {0, 0, 0};
    double *d_bmap = nullptr;
    double *d_maps = nullptr;          // field maps of the time-dependent B (SoA, 3 np each)
    int nmaps = 0;
    // generic CSR (H + H^T), device
    int *d_rp = nullptr, *d_ci = nullptr;
    double *d_v = nullptr;

    DipolarFFT *dip = nullptr;
    void *jit = nullptr;               // per-Hamiltonian compiled stage kernels (mj_jit.hip)
    int use_jit = 0;                   // they run now; jit_later: once aot_launches reach kJitPays
    int jit_later = 0;
    int64_t aot_launches = 0;          // stage kernels this context has run ahead of time
    void *adj = nullptr;               // differentiable SIB trajectory (mj_adjoint.hip)
    void *mc = nullptr;                // Metropolis Monte Carlo state (mj_mc.hip)
    // graph of a chunk of steps (small lattices: one replay instead of 2 launches per step)
    hipGraphExec_t gexec = nullptr;
    std::vector<double> gkey;          // the parameters it was captured for
    uint64_t *d_step = nullptr;        // device step counter read by the replayed kernels
    double *estage = nullptr;          // energies written by one replay
    int rk_order = 4;                  // integration 4: N_order (the reference's default)
    // per-term device copies of the registered M-M terms (offsets, blocks), made
    // on first use by mj_term_mult / mj_energy_terms and kept; staging vectors
    std::vector<int *> term_ofs;
    std::vector<double *> term_blk;
    double *tm_in = nullptr, *tm_out = nullptr;
    double *Drk[6] = {};               // integration 4: D of the stages before the last (SoA)
    // the effective field of the last stage of the last step (mj_keep_last_field)
    int keep_field = 0, field_valid = 0;
    double *Lf = nullptr;
};

int mj_finalize(mj_ctx *c);   // build device-side Hamiltonian if dirty

// Objects of at least kJitSites sites run kernels compiled for their Hamiltonian
// from their first call on (stage kernels, Monte Carlo passes, the adjoint, a
// batch's fused step by the sites of all its systems); compiling takes 0.2 s for
// the field, 0.5 to 0.7 s for an integrator.  A lattice of at least kJitSmall does
// so once it has run kJitPays stage kernels ahead of time: compiled, a launch of
// 32x32 to 56x59 sites is shorter by 1.4 to 2.9 us for the field, 1.3 to 2.1 for
// Euler and 2.8 to 3.7 for a stage of Heun, SIB or Depondt (8.7 us a step -> 3.1 on
// the square lattice, 11.9 -> 4.5 on the triangular one), so that by then about the
// time of compiling would have been saved; a Hamiltonian of fewer (a field, 40 steps
// of Heun in 0.4 to 0.5 ms) would wait 500 times its own time.  The kernels give the same bits.
// MJ_JIT=0: none compiled, 1: all.
constexpr int64_t kJitSites = 4096, kJitSmall = 1024, kJitPays = 100000;

// a compiled module on its device, unloaded with its last holder
struct JitModule {
    int device = 0;
    hipModule_t mod = nullptr;
    ~JitModule();
};
using JitRef = std::shared_ptr<JitModule>;

// per-Hamiltonian stage kernels (mj_jit.hip)
int mj_jit_prepare(mj_ctx *c, int bx, int by, int bz, int nblocks, int ntx, int nty);
int mj_jit_launch(mj_ctx *c, int mode, bool noise, const KArgs &a, hipStream_t s);
int mj_jit_resolve(mj_ctx *c, int mode, bool noise);
int mj_jit_fused_ok(const mj_ctx *c);   // the fused integration-2 kernel was generated
void mj_jit_destroy(mj_ctx *c);
// kernels of the differentiable SIB trajectory for a parameter set's stencil: offsets (3 per entry) and value
// classes (9 per entry: 0 zero, +-k the k-th value or its negative), the parameters' unit stencils (offsets, blocks)
enum { MJ_ADJ_SIB1, MJ_ADJ_SIB2, MJ_ADJ_SIBF, MJ_ADJ_R1, MJ_ADJ_R2, MJ_ADJ_R3R1, MJ_ADJ_R3, MJ_ADJ_KERNELS };
struct AdjStencil {
    std::vector<int> o3, cls;
    std::vector<std::vector<int>> po3;
    std::vector<std::vector<double>> pblk;
    bool operator==(const AdjStencil &o) const
    {
        return o3 == o.o3 && cls == o.cls && po3 == o.po3 && pblk == o.pblk;
    }
};
int mj_jit_adjoint(const mj_ctx *c, const AdjStencil &st, const int b[3], const int r[3], bool fused,
                   JitRef *mod, hipFunction_t fn[MJ_ADJ_KERNELS]);
// Monte Carlo kernels of a stencil without its on-site entry (offsets o3, full blocks cf9, class shifts csh) on the
// context's lattice coloured (x + ca y + cb z) mod p; vals: the distinct coefficients, for McArgs::vals (more than
// kMcMaxVals are literals, and none returned)
constexpr int kMcMaxVals = 32;
int mj_jit_mc(const mj_ctx *c, const std::vector<int> &o3, const std::vector<double> &cf9, const std::vector<int> &csh,
              int p, int ca, int cb, JitRef *mod, hipFunction_t *pass, hipFunction_t *energy,
              std::vector<double> *vals);
// the fused step of a batch's systems of one stencil and tile (fn null: its tile does not fit in LDS)
int mj_jit_batch_fused(int device, const std::vector<int> &ofs3, const std::vector<int> &cls, int ncls, int bx, int by,
                       int rx, int ry, int rz, int mode, JitRef *mod, hipFunction_t *fn, size_t *shm);

void mj_adj_destroy(mj_ctx *c);   // mj_adjoint.hip
void mj_mc_destroy(mj_ctx *c);    // mj_mc.hip
int mj_energy_into(mj_ctx *c, double *dst_dev);   // total energy of the state into device memory (mj_api.hip)

// dipolar (mj_fft.hip)
int dip_create(mj_ctx *c, const int N_rep[3], const int periodic[3], const double *K_n);
int dip_destroy(mj_ctx *c);
int dip_clone(mj_ctx *dst, const mj_ctx *src);   // dst->dip with src's operator, buffers and plans of its own
// the grid dip_apply writes H_fft into, with its row, plane and component strides
void dip_geometry(const mj_ctx *c, const double **grid, int *dnx, int *dny, int64_t *hstride);
// H_fft of SoA state `m` into the padded real grid owned by the dipolar object;
// returns the grid pointer and geometry through KArgs fields
int dip_apply(mj_ctx *c, const double *m_soa, KArgs *ka);
