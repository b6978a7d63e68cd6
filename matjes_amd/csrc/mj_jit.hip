// Per-Hamiltonian stage kernels compiled with hipRTC on first use.
//
// The stencil of a translation-invariant Hamiltonian is known once the
// Hamiltonian is registered, so the stage kernel is specialised for it: the
// lattice and tile sizes become compile-time constants (no integer division
// in the index math, a fixed trip count for the LDS fill) and the neighbour
// sum is fully unrolled with immediate LDS offsets and the block coefficients
// as exact literals.  The kernel body is the same source as the
// ahead-of-time kernel (mj_stage_body.h) with the same summation order, so
// the two give identical results; modules are found by their source text
// (mj_modcache.h) and compiled per integrator family on first use.
#include <hip/hiprtc.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>

#include <algorithm>
#include <array>
#include <map>
#include <sstream>
#include <string>
#include <vector>

#include "mj_internal.h"
#include "mj_modcache.h"
#include "_jit_embed.h"   // kJitRngH, kJitDeviceH, kJitKargsH, kJitBodyH (generated by matjes_amd/build.py)

struct JitState {
    std::string geom;              // generated geometry + stencil source of the stage kernels
    std::map<int, JitRef> mods;    // family -> module
    hipFunction_t fn[12][2] = {};     // resolved kernels per (mode, noise)
    int nthr = 0;
    size_t shm = 0;
    // both stages of integration 2, SIB or Depondt (MODE_HEUNF, _SIBF, _DEPF) in one kernel, when the tile fits
    int fuse_ok = 0, fuse_nthr = 0, fuse_nblocks = 0;
    size_t fuse_shm = 0;
    std::string fuse_tile;         // its constants; its sums are written when a family that has it is asked for
    int fuse_spt = 1, fuse_T0 = 0, fuse_s0x = 0, fuse_s0y = 0, fuse_s1x = 0, fuse_s1y = 0, fuse_s1z = 0;
    // persistent stage-1 kernels (stage_body_persistent): direct fill, whole XCD bands
    int pers_ok = 0, nblocks = 0;
    size_t pers_shm = 0;
    hipFunction_t fnp[12] = {};
    int pers_grid[12] = {};
};

// stage-1 modes with a persistent form (no own-site operands, no thermal field)
static bool persistent_mode(int mode)
{
    return mode == MODE_HEUN1 || mode == MODE_EULER || mode == MODE_SIB1 || mode == MODE_DEP1;
}

static void hexd(std::ostringstream &o, double v)
{
    char b[64];
    snprintf(b, sizeof b, "%a", v);
    o << "(" << b << ")";
}

// family of a mode: kernels compiled together
static int family_of(int mode)
{
    switch (mode) {
    case MODE_FIELD: return 0;
    case MODE_EULER: return 1;
    case MODE_HEUN1:
    case MODE_HEUN2:
    case MODE_HEUNF: return 2;
    case MODE_SIB1:
    case MODE_SIB2:
    case MODE_SIBF: return 3;
    case MODE_RKS: return 5;
    default: return 4;
    }
}

// Entries between two scheduling barriers of an unrolled neighbour sum: without
// barriers the LDS reads of the whole stencil are in flight at once, 87 VGPRs
// to the one-site fused step of the 18-neighbour stencil instead of 63 and
// more register moves (triangular 1024x1024, Heun: 4 to 12 entries equal within
// 1%, none 1% slower)
static const int kSumGroup = 12;

// The unrolled neighbour sums of `ns` sites one above the other (1, or 2: the
// site at c and the one a row of the region above it) over LDS components of
// stride TS in a region of row length sx and plane size sxy: the neighbours
// (ofs3, 3 per entry) by (dz, dy, dx) as every kernel sums them, each read once
// and added to the sums of the sites that have it.  coef(entry, 3 row + column)
// is the coefficient's expression, empty for a zero one, which is left out:
// fma(0, m, a) returns a for every finite m and nonzero a, and the sign of an
// exactly zero sum is the only other difference (the on-site anisotropy block
// diag(0, 0, K) and interfacial DMI, D_z = 0, are mostly zeros).
template <class Coef>
static void emit_sum(std::ostringstream &g, const std::vector<int> &ofs3, const char *name, int ns, int sx, int sxy,
                     int TS, Coef coef)
{
    g << "  static __device__ __forceinline__ void " << name << "(const KArgs &a, const double *L, int c";
    for (int q = 0; q < ns; ++q) g << ", double &ax" << q << ", double &ay" << q << ", double &az" << q;
    g << ") {\n    const double *Lx = L + c, *Ly = L + " << TS << " + c, *Lz = L + " << 2 * TS << " + c;\n";
    static const char *mm[3] = {"mx", "my", "mz"}, *acc[3] = {"ax", "ay", "az"};
    struct Use {
        int site, ent;
    };
    std::map<std::array<int, 3>, std::vector<Use>> by;   // (dz, dy, dx) from site 0 -> the sites it is a neighbour of
    for (size_t k = 0; k < ofs3.size() / 3; ++k) {
        const int *o = &ofs3[3 * k];
        for (int q = 0; q < ns; ++q) by[{o[2], o[1] + q, o[0]}].push_back({q, (int)k});
    }
    int n = 0;
    for (auto &kv : by) {
        const int lofs = kv.first[0] * sxy + kv.first[1] * sx + kv.first[2];
        g << "    { const double mx = Lx[" << lofs << "], my = Ly[" << lofs << "], mz = Lz[" << lofs << "];\n";
        for (const Use &u : kv.second)
            for (int r = 0; r < 3; ++r)
                for (int q = 0; q < 3; ++q) {
                    const std::string v = coef(u.ent, 3 * r + q);
                    if (v.empty()) continue;
                    g << "      " << acc[r] << u.site << " = fma(" << v << ", " << mm[q] << ", " << acc[r] << u.site
                      << ");\n";
                }
        g << "    }\n";
        if (++n % kSumGroup == 0) g << "    __builtin_amdgcn_sched_barrier(0);\n";
    }
    g << "  }\n";
}

// offsets of a context's stencil in the order of the sum, and its coefficients as literals
static std::vector<int> sum_offsets(const mj_ctx *c)
{
    std::vector<int> o;
    for (int k : c->h_ord) o.insert(o.end(), &c->h_ofs3[3 * k], &c->h_ofs3[3 * k] + 3);
    return o;
}
static auto literal_coef(const mj_ctx *c)
{
    return [c](int ent, int q) -> std::string {
        const double v = c->h_blk[9 * ent + q];
        if (v == 0.0) return std::string();
        std::ostringstream o;
        hexd(o, v);
        return o.str();
    };
}

// the regions of a fused tile: its constants (JitFused, BatchFused) and LDS bytes
static size_t emit_fused_tile(std::ostringstream &g, int BX, int BY, int BZ, int rx, int ry, int rz, int nthr, int spt,
                              int nsub, int nb, int wide, bool dma, int &T0, bool &alias)
{
    const int s0x = BX + 4 * rx, s0y = BY + 4 * ry, s0z = BZ + 4 * rz;
    const int t0 = s0x * s0y * s0z, t1 = (BX + 2 * rx) * (BY + 2 * ry) * (BZ + 2 * rz);
    const int all = nthr + wide, rthr = wide ? wide : nthr;
    T0 = dma ? 2 * all * ((t0 / 2 + all - 1) / all) : t0;
    // S1 in S0's place while a thread holds its share of the ring in registers
    alias = t1 - BX * BY * BZ <= 2 * rthr;
    g << "  static constexpr int kBx = " << BX << ", kBy = " << BY << ", kBz = " << BZ << ", kRx = " << rx
      << ", kRy = " << ry << ", kRz = " << rz << ";\n";
    g << "  static constexpr int kFill = " << (t0 + all - 1) / all << ";   // S0 sites per thread\n";
    g << "  static constexpr int kS0x = " << s0x << ", kS0y = " << s0y << ", kS0z = " << s0z << ", kT0 = " << T0 << ";\n";
    g << "  static constexpr bool kDma = " << (dma ? "true" : "false") << ", kAlias = " << (alias ? "true" : "false")
      << ";\n";
    g << "  static constexpr int kNthrBase = " << nb << ", kNsub = " << nsub << ";\n";
    g << "  static constexpr int kSpt = " << spt << ", kNthr = " << nthr
      << ";   // sites per thread, their threads\n  static constexpr int kWide = " << wide << ", kAll = " << all
      << ";   // threads of the ring's own, all\n";
    return sizeof(double) * ((size_t)3 * T0 + (alias ? 0 : (size_t)3 * t1) + BX * BY * BZ / 64 + 1);
}

// Geometry of the fused kernels (fused_body): the tile is the stage kernels'
// tile (bx, by, bz), or two of them along y (one plane deep); regions S0 (reach
// 2R) and S1 (reach R) in LDS.  Needs whole wavefronts per stage tile and at
// most 64 KiB of LDS.  Three forms, by the number of double tiles: single
// tiles while the double ones give a CU fewer than two workgroups (a launch of
// a small lattice is the latency of one tile), double tiles with threads of
// their own (a ring of 0.41 instead of 0.69 sites per site at reach 2), and
// from six workgroups per CU on double tiles with two sites per thread, where
// the CUs are full and the neighbours read once for both sites count.  Measured,
// us per step, Heun at 10 K, single / double / pairs: triangular 384x384 8.45 /
// 9.23 / 9.71, 512x512 10.5 / 9.6 / 10.2, 724x724 19.2 / 18.5 / 18.8, 1024x1024
// 29.4 / 27.3 / 26.6, 1500x1500 62.3 / 56.9 / 54.9; square 384x384 6.2 / 7.0 /
// 7.4, 512x512 7.6 / 7.4 / 7.9, 1024x1024 19.6 / 19.1 / 19.5, 1500x1500 39.3 /
// 38.7 / 39.7 (SIB 42.4 / 39.5 / 39.4, Depondt 46.5 / 42.9 / 42.3).
// Up to one single tile per CU the ring has wavefronts of its own: a launch is
// one tile's latency, and the first stage then runs once instead of twice in
// turn (us per step, Heun at 10 K: triangular 64x64 5.34 -> 4.90, 256x256 5.88 ->
// 5.44, square 64x64 4.24 -> 4.03, 64x64x16 6.2 -> 5.4; beyond, 384x384 8.45 ->
// 8.03 but Depondt 9.2 -> 10.2, square 6.2 -> 6.4, 128x128x16 11.8 -> 12.2).
// MJ_FUSE_SPT=1 or 2 asks for single tiles or pairs, MJ_FUSE_SUB=2 for double
// tiles, MJ_FUSE_WIDE=0 or 1 against or for the ring's own wavefronts.
static void prepare_fused(const mj_ctx *c, JitState *j, int bx, int by, int bz, int ntx, int nty, int ntz)
{
    j->fuse_ok = 0;
    const int nb = bx * by * bz;
    if (nb % 64 != 0 || ntx <= 0) return;
    const int rx = c->rx, ry = c->ry, rz = c->rz;
    const char *sp = getenv("MJ_FUSE_SPT"), *su = getenv("MJ_FUSE_SUB");
    int cus = 0;
    if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, c->device) != hipSuccess) cus = 256;
    const bool pairs = bz == 1 && bx == 32 && by % 2 == 0;
    const long nwg2 = (long)ntx * ((c->dim[1] + 2 * by - 1) / (2 * by)) * ntz;
    int form = 0;   // 0: one stage tile; 1: two, threads of their own; 2: two, two sites per thread
    if (bz == 1 && nwg2 >= 2L * cus) form = pairs && nwg2 >= 6L * cus ? 2 : 1;
    if (sp) form = atoi(sp) == 2 && pairs ? 2 : 0;
    if (su && atoi(su) == 2 && bz == 1) form = 1;
    for (; form >= 0; --form) {
        const int spt = form == 2 ? 2 : 1, nsub = form ? 2 : 1;
        const int BX = bx, BY = by * nsub, BZ = bz, nthr = BX * BY * BZ / spt;
        const bool dma = bx % 2 == 0 && c->dim[0] % 2 == 0 && nthr % 64 == 0;
        std::ostringstream t;
        int T0 = 0;
        bool alias = false;
        const int nring = (BX + 2 * rx) * (BY + 2 * ry) * (BZ + 2 * rz) - BX * BY * BZ;
        const char *we = getenv("MJ_FUSE_WIDE");
        const bool few = we ? we[0] == '1' : (long)ntx * nty * ntz <= cus;
        const int wide = form == 0 && few ? std::min((nring + 63) / 64 * 64, 1024 - nthr) : 0;
        const size_t shm = emit_fused_tile(t, BX, BY, BZ, rx, ry, rz, nthr, spt, nsub, nb, wide, dma, T0, alias);
        if (shm > 65536 || nthr + wide > 1024) continue;
        const int ntyf = (c->dim[1] + BY - 1) / BY, ntzf = (c->dim[2] + BZ - 1) / BZ;
        t << "  static constexpr bool kEnergy = true;\n";
        auto cst = [&](const char *n, const char *ty, long v) {
            t << "  static __device__ __forceinline__ constexpr " << ty << " " << n << "(const KArgs &) { return " << v
              << "; }\n";
        };
        cst("nx", "int", c->dim[0]), cst("ny", "int", c->dim[1]), cst("nz", "int", c->dim[2]);
        cst("ntx", "int", ntx), cst("nty", "int", ntyf), cst("nty_base", "int", nty);
        cst("bmode", "int", c->bmode), cst("dma", "bool", dma);   // bmode: 0 no Zeeman, 1 uniform, 2 per site
        t << "  static __device__ __forceinline__ int block(const KArgs &) { return mj_xcd_remap(blockIdx.x, "
          << ntx * ntyf * ntzf << "); }\n";
        j->fuse_tile = t.str();
        j->fuse_spt = spt;
        j->fuse_T0 = T0;
        j->fuse_s0x = BX + 4 * rx;
        j->fuse_s0y = BY + 4 * ry;
        j->fuse_s1x = BX + 2 * rx;
        j->fuse_s1y = BY + 2 * ry;
        j->fuse_s1z = BZ + 2 * rz;
        j->fuse_ok = 1;
        j->fuse_nthr = nthr + wide;
        j->fuse_nblocks = ntx * ntyf * ntzf;
        j->fuse_shm = shm;
        return;
    }
}

static void emit_fused(std::ostringstream &g, const mj_ctx *c, const JitState *j)
{
    g << "struct JitFused {\n" << j->fuse_tile;
    const auto ofs3 = sum_offsets(c);
    const auto cf = literal_coef(c);
    const int xy0 = j->fuse_s0x * j->fuse_s0y, xy1 = j->fuse_s1x * j->fuse_s1y, t1 = xy1 * j->fuse_s1z;
    emit_sum(g, ofs3, "stencil0", 1, j->fuse_s0x, xy0, j->fuse_T0, cf);
    emit_sum(g, ofs3, j->fuse_spt == 2 ? "pair1" : "stencil1", j->fuse_spt, j->fuse_s1x, xy1, t1, cf);
    if (j->fuse_spt == 2) emit_sum(g, ofs3, "pair0", 2, j->fuse_s0x, xy0, j->fuse_T0, cf);
    g << "};\n";
}

int mj_jit_fused_ok(const mj_ctx *c) { return c->jit && ((const JitState *)c->jit)->fuse_ok; }

int mj_jit_prepare(mj_ctx *c, int bx, int by, int bz, int nblocks, int ntx, int nty)
{
    JitState *j = c->jit ? (JitState *)c->jit : new JitState();
    c->jit = j;
    j->mods.clear();
    for (auto &row : j->fn) row[0] = row[1] = nullptr;
    std::ostringstream g;
    const int sx = bx + 2 * c->rx, sy = by + 2 * c->ry, sz = bz + 2 * c->rz;
    const int T = sx * sy * sz;
    const int nthr = bx * by * bz;
    // direct global -> LDS tile fill: 16-byte pairs along x need even reach,
    // even tile and lattice rows and whole wavefronts; the LDS components are
    // then padded to whole trips of the workgroup
    const bool dma = c->rx % 2 == 0 && bx % 2 == 0 && c->dim[0] % 2 == 0 && nthr % 64 == 0;
    const int TS = dma ? 2 * nthr * ((T / 2 + nthr - 1) / nthr) : T;   // LDS component stride
    g << "struct JitGeom {\n";
    g << "  static constexpr int kNit = " << (T + bx * by * bz - 1) / (bx * by * bz) << ";\n";
    g << "  static constexpr bool kDma = " << (dma ? "true" : "false") << ", kCfLds = false;\n  static constexpr int kTrips = 1;\n";
    g << "  static constexpr int kT = " << TS << ";\n";
    g << "  static __device__ __forceinline__ int tstride(const KArgs &, int) { return " << TS << "; }\n";
    g << "  static constexpr int kBx = " << bx << ", kBy = " << by << ", kBz = " << bz << ", kRx = " << c->rx
      << ", kRy = " << c->ry << ", kRz = " << c->rz << ", kNx = " << c->dim[0] << ", kNy = " << c->dim[1] << ";\n";
    auto cst = [&](const char *n, long v) {
        g << "  static __device__ __forceinline__ constexpr int " << n << "(const KArgs &) { return " << v << "; }\n";
    };
    cst("bx", bx); cst("by", by); cst("bz", bz);
    cst("rx", c->rx); cst("ry", c->ry); cst("rz", c->rz);
    cst("nx", c->dim[0]); cst("ny", c->dim[1]); cst("nz", c->dim[2]);
    cst("ntx", ntx); cst("nty", nty); cst("nblocks", nblocks);
    g << "  static __device__ __forceinline__ int block(const KArgs &) { return mj_xcd_remap(blockIdx.x, " << nblocks
      << "); }\n";
    g << "  static __device__ __forceinline__ int part(const KArgs &) { return mj_xcd_remap(blockIdx.x, " << nblocks
      << "); }\n";
    emit_sum(g, sum_offsets(c), "sum", 1, sx, sx * sy, TS, literal_coef(c));
    g << "  static __device__ __forceinline__ void stencil(const KArgs &a, const double *L, int, int c, double &ax, "
         "double &ay, double &az) { sum(a, L, c, ax, ay, az); }\n};\n";
    j->nthr = nthr;
    size_t shm = (size_t)3 * TS * sizeof(double);
    if (shm < (size_t)j->nthr * sizeof(double)) shm = (size_t)j->nthr * sizeof(double);
    j->shm = shm;
    j->nblocks = nblocks;
    j->pers_ok = dma && nblocks % 8 == 0 && 3 * TS >= nthr;
    j->pers_shm = (size_t)6 * TS * sizeof(double);
    for (auto &f : j->fnp) f = nullptr;
    for (auto &g2 : j->pers_grid) g2 = 0;
    prepare_fused(c, j, bx, by, bz, ntx, nty, ntx == 0 ? 0 : nblocks / (ntx * nty));
    j->geom = g.str();
    return MJ_OK;
}

void mj_jit_destroy(mj_ctx *c)
{
    delete (JitState *)c->jit;
    c->jit = nullptr;
}

static std::string family_source(const mj_ctx *c, const JitState *j, int fam);
static std::string device_headers();

// the source of the kernels of one integrator family (for offline inspection)
std::string mj_jit_source(const mj_ctx *c, int fam)
{
    return c->jit ? device_headers() + family_source(c, (const JitState *)c->jit, fam) : std::string();
}

JitModule::~JitModule()
{
    int cur = 0;
    (void)hipGetDevice(&cur);
    (void)hipSetDevice(device);
    (void)hipDeviceSynchronize();   // its kernels are done
    (void)hipModuleUnload(mod);
    (void)hipSetDevice(cur);
}

// compiles a source and loads it on `device` (the current one)
static int compile_module(int device, const std::string &src, JitRef *out)
{
    hiprtcProgram prog;
    if (hiprtcCreateProgram(&prog, src.c_str(), "mj_stage_jit.hip", 0, nullptr, nullptr) != HIPRTC_SUCCESS) {
        mj_set_error("hiprtcCreateProgram failed");
        return MJ_EHIP;
    }
    const char *opts[] = {"--offload-arch=gfx950", "-O3", "-std=c++17", "-ffp-contract=off",
                          "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops"};
    hiprtcResult rc = hiprtcCompileProgram(prog, 8, opts);
    if (rc != HIPRTC_SUCCESS) {
        size_t ls = 0;
        hiprtcGetProgramLogSize(prog, &ls);
        std::string log(ls, ' ');
        if (ls) hiprtcGetProgramLog(prog, &log[0]);
        hiprtcDestroyProgram(&prog);
        mj_set_error("hipRTC compile of the stage kernels failed: " + log.substr(0, 2000));
        return MJ_EHIP;
    }
    size_t cs = 0;
    hiprtcGetCodeSize(prog, &cs);
    std::vector<char> code(cs);
    hiprtcGetCode(prog, code.data());
    hiprtcDestroyProgram(&prog);
    hipModule_t mod;
    hipError_t e = hipModuleLoadData(&mod, code.data());
    if (e != hipSuccess) return mj_hip_fail(MJ_EHIP, std::string("hipModuleLoadData: ") + hipGetErrorString(e));
    *out = std::make_shared<JitModule>();
    (*out)->device = device;
    (*out)->mod = mod;
    return MJ_OK;
}

// the modules of the process: 64 (some 0.1 MB each) beside those in use
static ModCache<JitModule> &modules()
{
    static auto *cache = new ModCache<JitModule>(64);   // never destroyed: the runtime ends first
    return *cache;
}

// The module of a source on a device (the caller's current one): the device
// headers, `extra` ones, and `src`, which alone says which module it is.  With
// the 80 KB of headers in the text to be built and found, the first field of a
// new object took 30 to 70 us more (64x64 and 128x128, triangular).
static int compile_source(int device, const std::string &src, const char *extra, JitRef *out)
{
    return modules().get(device, src, out,
                         [&](JitRef *m) { return compile_module(device, device_headers() + extra + "\n" + src, m); });
}

extern "C" int mj_jit_stats(int64_t *compiled, int64_t *kept)
{
    long long a = 0, b = 0;
    modules().stats(&a, &b);
    if (compiled) *compiled = a;
    if (kept) *kept = b;
    return MJ_OK;
}

static int compile_family(const mj_ctx *c, JitState *j, int fam, JitRef *out)
{
    return compile_source(c->device, family_source(c, j, fam), "", out);
}

static std::string device_headers()
{
    std::ostringstream s;
    s << "#define MJ_JIT 1\n" << kJitRngH << "\n" << kJitDeviceH << "\n" << kJitKargsH << "\n" << kJitBodyH << "\n";
    return s.str();
}

// The fused step of the systems of a batch that share a stencil's offsets and a
// tile (bx x by, 256 sites): tile, regions and neighbour sums compile-time, the
// lattices' sizes, Zeeman terms and coefficients read from the batch's tables.
// cls[9 entry + q]: 0 a coefficient that is zero in every such system, +-k the
// k-th value of a system's `ncls` (or its negative): the values stay in scalar
// registers, an operand of the fused products.
// Instruction issue bounds it, as the single lattice's step.  24 replicas of 256^2
// (18 neighbours, T > 0) and 12 more lattices of 32 to 400 a side, 2.2 M sites:
// 50 us a step, the ahead-of-time kernel (k_batch_fused: offsets and full 3x3
// blocks read in a loop, wrapped coordinates per staged site) 81 us.
int mj_jit_batch_fused(int device, const std::vector<int> &ofs3, const std::vector<int> &cls, int ncls, int bx, int by,
                       int rx, int ry, int rz, int mode, JitRef *mod, hipFunction_t *fn, size_t *shm)
{
    std::ostringstream g;
    int T0 = 0;
    bool alias = false;
    const int s0x = bx + 4 * rx, s0y = by + 4 * ry, s1x = bx + 2 * rx, s1y = by + 2 * ry;
    g << "struct BatchFused {\n";
    const bool dma = bx % 2 == 0;   // 16-byte pairs along x: no pair spans two rows of the region
    *shm = emit_fused_tile(g, bx, by, 1, rx, ry, rz, bx * by, 1, 1, bx * by, 0, dma, T0, alias);
    if (*shm > 65536) {
        *fn = nullptr;
        return MJ_OK;
    }
    g << "  static constexpr bool kEnergy = false;\n";
    auto arg = [&](const char *n, const char *ty, const char *v) {
        g << "  static __device__ __forceinline__ " << ty << " " << n << "(const KArgs &a) { return " << v << "; }\n";
    };
    arg("nx", "int", "a.nx"), arg("ny", "int", "a.ny"), arg("nz", "int", "a.nz");
    arg("ntx", "int", "a.ntx"), arg("nty", "int", "a.nty"), arg("nty_base", "int", "a.nty");
    arg("bmode", "int", "a.bmode"), arg("dma", "bool", dma ? "((a.nx | a.np) & 1) == 0" : "false"), arg("block", "int", "a.vbid");
    auto cf = [&](int ent, int q) -> std::string {
        const int k = cls[9 * ent + q];
        return k == 0 ? std::string() : std::string(k < 0 ? "-" : "") + "a.cf[" + std::to_string(abs(k) - 1) + "]";
    };
    emit_sum(g, ofs3, "stencil0", 1, s0x, s0x * s0y, T0, cf);
    emit_sum(g, ofs3, "stencil1", 1, s1x, s1x * s1y, s1x * s1y * (1 + 2 * rz), cf);
    g << "};\n";
    std::ostringstream s;
    s << g.str();
    s << "extern \"C\" __global__ void __launch_bounds__(" << bx * by
      << ") mj_batch_fused(const KArgs base, const BatchSys *__restrict__ sys, const int *__restrict__ blk2sys, "
         "const double *__restrict__ sigma, const uint64_t *__restrict__ stepp, const int *__restrict__ list, int nlist, "
         "const double *__restrict__ vals) {\n  extern __shared__ double lds[];\n"
         "  const int b = mj_xcd_remap(blockIdx.x, nlist);\n  const int gb = list ? list[b] : b;\n"
         "  const int s = blk2sys[gb];\n  KArgs a = sys_args(base, sys[s], gb, sigma[s], *stepp + base.step);\n"
         "  a.cf = vals + (int64_t)s * " << ncls << ";\n  fused_body<" << mode << ", true, BatchFused>(a, lds);\n}\n";
    const int rc = compile_source(device, s.str(), kJitBatchH, mod);
    if (rc != MJ_OK) return rc;
    const hipError_t e = hipModuleGetFunction(fn, (*mod)->mod, "mj_batch_fused");
    if (e != hipSuccess) return mj_hip_fail(MJ_EHIP, std::string("hipModuleGetFunction mj_batch_fused: ") + hipGetErrorString(e));
    return MJ_OK;
}

// The differentiable SIB trajectory's kernels for a parameter set: lattice, tile
// and stencils compile-time, the values (they change with the parameters) from
// scalar registers; terms in the order of apply_blocks, structural zeros left
// out.  Latency bounds them on the lattices they are used for (one wavefront a
// workgroup at 128^2): the halo's wraps and the table of offsets went, all of a
// workgroup's loads are in flight before its first store to LDS.  128^2, 4
// neighbours, 3 parameters: forward step 7.9 -> 4.2 us, R2 11.1 -> 4.8, R3 with
// R1 11.2 -> 4.9.
int mj_jit_adjoint(const mj_ctx *c, const AdjStencil &st, const int b[3], const int r[3], bool fused,
                   JitRef *mod, hipFunction_t fn[MJ_ADJ_KERNELS])
{
    std::ostringstream g;
    const int nthr = b[0] * b[1] * b[2];
    int s1[3], s0[3];
    for (int d = 0; d < 3; ++d) {
        s1[d] = b[d] + 2 * r[d];
        s0[d] = b[d] + 4 * r[d];
    }
    const int t1 = s1[0] * s1[1] * s1[2], t0 = s0[0] * s0[1] * s0[2], np = (int)st.po3.size();
    g << "struct AdjJit {\n  static constexpr bool kConst = true;\n  static constexpr int kTrips = "
      << (t1 + nthr - 1) / nthr << ", kTrips0 = " << (t0 + nthr - 1) / nthr << ", kMaxVals = " << np + 3 << ";\n";
    auto cst = [&](const char *n, int v) {
        g << "  static __device__ __forceinline__ constexpr int " << n << "(const AdjArgs &) { return " << v << "; }\n";
    };
    cst("nx", c->dim[0]), cst("ny", c->dim[1]), cst("nz", c->dim[2]), cst("bx", b[0]), cst("by", b[1]), cst("bz", b[2]);
    cst("rx", r[0]), cst("ry", r[1]), cst("rz", r[2]), cst("nparam", np);
    cst("ntx", (c->dim[0] + b[0] - 1) / b[0]), cst("nty", (c->dim[1] + b[1] - 1) / b[1]);
    // sum over entries (offsets o3, coefficient expressions) into name(x, y, z)
    auto emit = [&](const char *v, const std::vector<int> &o3, const int sz[3], auto coef) {
        static const char *mm[3] = {"mx", "my", "mz"}, *ac[3] = {"ax", "ay", "az"};
        g << "    { double ax = 0.0, ay = 0.0, az = 0.0;\n";
        for (size_t e = 0; e < o3.size() / 3; ++e) {
            const int l = (o3[3 * e + 2] * sz[1] + o3[3 * e + 1]) * sz[0] + o3[3 * e];
            g << "    { const double mx = L[c + " << l << "], my = L[T + c + " << l << "], mz = L[2 * T + c + " << l << "];\n";
            for (int q = 0; q < 9; ++q) {
                const std::string w = coef(e, q);
                if (!w.empty())
                    g << "      " << ac[q / 3] << " = fma(" << w << ", " << mm[q % 3] << ", " << ac[q / 3] << ");\n";
            }
            g << "    }\n";
        }
        g << "    " << v << " }\n";
    };
    auto cls = [&](size_t e, int q) -> std::string {
        const int k = st.cls[9 * e + q];
        return k == 0 ? std::string() : std::string(k < 0 ? "-" : "") + "a.cls[" + std::to_string(abs(k) - 1) + "]";
    };
    for (int h = 0; h < 2; ++h) {
        g << "  static __device__ __forceinline__ v3 " << (h ? "sum0" : "sum")
          << "(const AdjArgs &a, const double *L, int T, int c) {\n";
        emit("return mk3(ax, ay, az);", st.o3, h ? s0 : s1, cls);
        g << "  }\n";
    }
    g << "  static __device__ __forceinline__ void units(const AdjArgs &a, const double *L, int T, int c, v3 gB, double *vals) "
         "{\n";
    for (int k = 0; k < np; ++k) {
        const std::string v = "vals[" + std::to_string(k) + "] = -dot3(gB, mk3(ax, ay, az));";
        emit(v.c_str(), st.po3[k], s1, [&](size_t e, int q) -> std::string {
            const double w = st.pblk[k][9 * e + q];
            if (w == 0.0) return std::string();
            std::ostringstream o;
            hexd(o, w);
            return o.str();
        });
    }
    g << "  }\n};\n";
    std::ostringstream s;
    s << g.str();
    static const char *names[MJ_ADJ_KERNELS] = {"sib1", "sib2", "sibf", "r1", "r2", "r3r1", "r3"};
    auto want = [&](int k) { return k == MJ_ADJ_SIBF ? fused : k == MJ_ADJ_SIB1 || k == MJ_ADJ_SIB2 ? !fused : true; };
    for (int k = 0; k < MJ_ADJ_KERNELS; ++k)
        if (want(k))
            s << "extern \"C\" __global__ void __launch_bounds__(" << nthr << ") mj_adj_" << names[k]
              << "(const AdjArgs a) { extern __shared__ double lds[]; adj_" << names[k] << "_body<AdjJit>(a, lds); }\n";
    const int rc = compile_source(c->device, s.str(), kJitAdjH, mod);
    if (rc != MJ_OK) return rc;
    for (int k = 0; k < MJ_ADJ_KERNELS; ++k) {
        if (!want(k)) continue;
        const hipError_t e = hipModuleGetFunction(&fn[k], (*mod)->mod, (std::string("mj_adj_") + names[k]).c_str());
        if (e != hipSuccess) return mj_hip_fail(MJ_EHIP, std::string("hipModuleGetFunction: ") + hipGetErrorString(e));
    }
    return MJ_OK;
}

// Monte Carlo passes and replica energies: the neighbours' slots from the
// lattice's constants, the spins of 18 neighbours in flight together (the
// proposal is computed under the first ones), coefficients as operands, terms
// in the order and with the operations of mc_pair_field_cm (zero ones left out).
// Latency bounds a pass (two wavefronts per SIMD at 131072 sites): 18 neighbours
// in three trips through a table of slots took 18.2 us per class of 1024^2 (8
// classes) and 13.9 us for 8 replicas of 256^2, one trip with the addresses from
// constants 8.1 and 6.6; replica energies 34.6 -> 22.  The distinct coefficients
// (up to sign) are read into scalar registers, so that a scan over couplings
// compiles once per structure; more than 32 are literals.  Blocks of 64 and 128
// threads: 8 and 2 % slower at 1024^2, equal at 256^2.
int mj_jit_mc(const mj_ctx *c, const std::vector<int> &o3, const std::vector<double> &cf9, const std::vector<int> &csh,
              int p, int ca, int cb, JitRef *mod, hipFunction_t *pass, hipFunction_t *energy,
              std::vector<double> *vals)
{
    constexpr int kGroup = 18;
    const int nx = c->dim[0], ny = c->dim[1], nz = c->dim[2], W = (nx + p - 1) / p, ne = (int)csh.size();
    const int64_t RW = (int64_t)ny * nz * W;
    std::ostringstream g;
    g << "struct McGeom {\n  static constexpr int kNx = " << nx << ", kNy = " << ny << ", kRows = " << ny * nz
      << ", kW = " << W << ", kP = " << p << ";\n";
    g << "  static __device__ __forceinline__ int first(int k, int y, int z) {\n    int x0 = (k - " << ca << " * y - " << cb
      << " * z) % " << p << ";\n    return x0 < 0 ? x0 + " << p << " : x0;\n  }\n";
    g << "  template <class Mid> static __device__ __forceinline__ v3 field(const McArgs &a, const double *cm, int k, int x0, "
         "int jj, int x, int y, int z, Mid mid) {\n    double ax = 0.0, ay = 0.0, az = 0.0;\n";
    // column of the neighbour at dx, row offset of the one at (dy, dz); open edges: false
    std::map<int, int> dxs;
    std::map<std::array<int, 2>, int> rows;
    for (int e = 0; e < ne; ++e) {
        dxs.insert({o3[3 * e], (int)dxs.size()});
        rows.insert({{o3[3 * e + 1], o3[3 * e + 2]}, (int)rows.size()});
    }
    for (auto &kv : dxs) {
        const int dx = kv.first, i = kv.second;
        const int q0 = (dx % p + p) % p, f = (dx - q0) / p;   // dx = f p + q0
        g << "    int j" << i << " = jj + " << f << " + (x0 + " << q0 << " >= " << p << " ? 1 : 0);\n";
        g << "    const int u" << i << " = x + " << dx << "; const bool cx" << i << " = " << (c->periodic[0] ? "true" : "")
          << (c->periodic[0] ? "" : "u" + std::to_string(i) + " >= 0 && u" + std::to_string(i) + " < " + std::to_string(nx))
          << ";\n";
        if (c->periodic[0])
            g << "    j" << i << " += u" << i << " < 0 ? " << W << " : u" << i << " >= " << nx << " ? " << -W << " : 0;\n";
    }
    for (auto &kv : rows) {
        const int i = kv.second;
        auto axis = [&](const char *v, int d, int n, int per) {
            const std::string w = std::string(v) + std::to_string(i);
            g << "    int " << w << " = " << v << " + " << d << "; const bool c" << w << " = ";
            if (d == 0) g << "true;\n";
            else if (!per) g << w << " >= 0 && " << w << " < " << n << ";\n";
            else if (abs(d) <= n) g << "true; " << w << " += " << w << " < 0 ? " << n << " : " << w << " >= " << n << " ? " << -n << " : 0;\n";
            else g << "true; " << w << " = ((" << w << " % " << n << ") + " << n << ") % " << n << ";\n";
        };
        axis("y", kv.first[0], ny, c->periodic[1]);
        axis("z", kv.first[1], nz, c->periodic[2]);
        g << "    const int r" << i << " = (y" << i << " + " << ny << " * z" << i << ") * " << W << "; const bool cr" << i
          << " = cy" << i << " && cz" << i << ";\n";
    }
    vals->clear();
    auto place = [&](double v) {   // of +-v among them
        return std::find_if(vals->begin(), vals->end(), [&](double w) { return w == v || w == -v; }) - vals->begin();
    };
    for (double v : cf9)
        if (v != 0.0 && place(v) == (ptrdiff_t)vals->size()) vals->push_back(v);
    const bool literal = vals->size() > kMcMaxVals;
    if (literal) vals->clear();
    auto coef = [&](double v) {
        if (literal) {
            hexd(g, v);
        } else {
            const auto k = place(v);
            g << ((*vals)[k] == v ? "" : "-") << "a.vals[" << k << "]";
        }
    };
    auto has = [&](int e, int col) { return cf9[9 * e + col] != 0.0 || cf9[9 * e + 3 + col] != 0.0 || cf9[9 * e + 6 + col] != 0.0; };
    static const char *mm[3] = {"mx", "my", "mz"}, *acc[3] = {"ax", "ay", "az"};
    for (int e0 = 0; e0 < ne; e0 += kGroup) {
        const int e1 = std::min(ne, e0 + kGroup);
        for (int e = e0; e < e1; ++e) {
            const int *o = &o3[3 * e];
            const int i = dxs[o[0]], r = rows[{o[1], o[2]}];
            const bool open = (!c->periodic[0] && o[0]) || (!c->periodic[1] && o[1]) || (!c->periodic[2] && o[2]);
            g << "    const int k" << e << " = k + " << csh[e] << " >= " << p << " ? k + " << csh[e] - p << " : k + " << csh[e]
              << ";\n    const double *q" << e << " = cm + (int64_t)k" << e << " * " << RW << "; const bool ok" << e << " = ";
            if (open) g << "cx" << i << " && cr" << r << ";\n";
            else g << "true;\n";
            g << "    const unsigned s" << e << " = ok" << e << " ? 8u * (unsigned)(r" << r << " + j" << i << ") : 0u;\n";
            for (int d = 0; d < 3; ++d)
                if (has(e, d)) {
                    g << "    double " << mm[d] << e << " = *(const double *)((const char *)(q" << e << " + " << d
                      << " * a.cs) + s" << e << ");\n";
                }
        }
        g << "    __builtin_amdgcn_sched_barrier(0);\n";
        if (e0 == 0) g << "    mid();\n";
        for (int e = e0; e < e1; ++e) {
            const int *o = &o3[3 * e];
            const bool open = (!c->periodic[0] && o[0]) || (!c->periodic[1] && o[1]) || (!c->periodic[2] && o[2]);
            for (int d = 0; d < 3 && open; ++d)
                if (has(e, d)) g << "    " << mm[d] << e << " = ok" << e << " ? " << mm[d] << e << " : 0.0;\n";
            for (int r = 0; r < 3; ++r)
                for (int d = 0; d < 3; ++d) {
                    const double v = cf9[9 * e + 3 * r + d];
                    if (v == 0.0) continue;
                    g << "    " << acc[r] << " = fma(";
                    coef(v);
                    g << ", " << mm[d] << e << ", " << acc[r] << ");\n";
                }
        }
    }
    if (ne == 0) g << "    mid();\n";
    g << "    return mk3(ax, ay, az);\n  }\n};\n";
    std::ostringstream s;
    s << g.str();
    s << "extern \"C\" __global__ void __launch_bounds__(kMcThreads) mj_mc_pass(const McArgs a) { "
         "mc_pass_body<McGeom>(a); }\n";
    s << "extern \"C\" __global__ void __launch_bounds__(kMcThreads) mj_mc_energy(const McArgs a, double *part) { "
         "mc_energy_body<McGeom>(a, part); }\n";
    const int rc = compile_source(c->device, s.str(), kJitMcH, mod);
    if (rc != MJ_OK) return rc;
    hipError_t e = hipModuleGetFunction(pass, (*mod)->mod, "mj_mc_pass");
    if (e == hipSuccess) e = hipModuleGetFunction(energy, (*mod)->mod, "mj_mc_energy");
    if (e != hipSuccess) return mj_hip_fail(MJ_EHIP, std::string("hipModuleGetFunction: ") + hipGetErrorString(e));
    return MJ_OK;
}

static std::string family_source(const mj_ctx *c, const JitState *j, int fam)
{
    std::ostringstream s;
    s << j->geom << "\n";
    if (j->fuse_ok && fam >= 2 && fam <= 4) emit_fused(s, c, j);
    static const int fam_modes[6][3] = {{MODE_FIELD, -1, -1}, {MODE_EULER, -1, -1}, {MODE_HEUN1, MODE_HEUN2, MODE_HEUNF},
                                        {MODE_SIB1, MODE_SIB2, MODE_SIBF}, {MODE_DEP1, MODE_DEP2, MODE_DEPF},
                                        {MODE_RKS, -1, -1}};
    // occupancy hint: minimum waves per SIMD (MJ_WAVES_PER_EU), which caps VGPRs
    const char *wpe = getenv("MJ_WAVES_PER_EU");
    std::string attr;
    if (wpe && atoi(wpe) > 0) attr = " __attribute__((amdgpu_waves_per_eu(" + std::to_string(atoi(wpe)) + ")))";
    for (int q = 0; q < 3; ++q) {
        int mode = fam_modes[fam][q];
        if (mode < 0) continue;
        for (int nz = 0; nz < 2; ++nz) {
            if (mode == MODE_HEUNF || mode == MODE_SIBF || mode == MODE_DEPF) {
                if (j->fuse_ok)
                    s << "extern \"C\" __global__ void __launch_bounds__(" << j->fuse_nthr << ")" << attr
                      << " mj_stage_" << mode << "_" << nz << "(const KArgs a) { extern __shared__ double lds[]; "
                      << "fused_body<" << mode << ", " << (nz ? "true" : "false") << ", JitFused>(a, lds); }\n";
                continue;
            }
            s << "extern \"C\" __global__ void __launch_bounds__(" << j->nthr << ")" << attr << " mj_stage_" << mode << "_" << nz
              << "(const KArgs a) { extern __shared__ double lds[]; stage_body<" << mode << ", "
              << (nz ? "true" : "false") << ", JitGeom>(a, lds); }\n";
        }
        if (j->pers_ok && persistent_mode(mode))
            s << "extern \"C\" __global__ void __launch_bounds__(" << j->nthr << ")" << attr << " mj_pstage_" << mode
              << "(const KArgs a) { extern __shared__ double lds[]; stage_body_persistent<" << mode
              << ", JitGeom>(a, lds); }\n";
    }
    return s.str();
}

// compile (first use of the family) and resolve the kernel of (mode, noise)
static int jit_resolve(mj_ctx *c, int mode, bool noise, hipFunction_t *out)
{
    JitState *j = (JitState *)c->jit;
    hipFunction_t f = j->fn[mode][noise ? 1 : 0];
    if (!f) {
        int fam = family_of(mode);
        auto it = j->mods.find(fam);
        JitRef mod;
        if (it == j->mods.end()) {
            int rc = compile_family(c, j, fam, &mod);
            if (rc) return rc;
            j->mods[fam] = mod;
        } else {
            mod = it->second;
        }
        char name[64];
        snprintf(name, sizeof name, "mj_stage_%d_%d", mode, noise ? 1 : 0);
        hipError_t e = hipModuleGetFunction(&f, mod->mod, name);
        if (e != hipSuccess) return mj_hip_fail(MJ_EHIP, std::string("hipModuleGetFunction ") + name + ": " + hipGetErrorString(e));
        j->fn[mode][noise ? 1 : 0] = f;
    }
    *out = f;
    return MJ_OK;
}

static int jit_resolve_persistent(mj_ctx *c, int mode, hipFunction_t *out, int *grid);
static bool persist_enabled();

// resolve ahead of time (before a stream capture: no compilation while capturing)
int mj_jit_resolve(mj_ctx *c, int mode, bool noise)
{
    hipFunction_t f;
    int rc = jit_resolve(c, mode, noise, &f);
    JitState *j = (JitState *)c->jit;
    if (rc == MJ_OK && !noise && j->pers_ok && persistent_mode(mode) && persist_enabled()) {
        int grid = 0;
        rc = jit_resolve_persistent(c, mode, &f, &grid);
    }
    return rc;
}

// the persistent form of a stage-1 kernel (MJ_PERSIST=1), resolved with its grid:
// as many workgroups as fit on the device at once, a multiple of 8
static int jit_resolve_persistent(mj_ctx *c, int mode, hipFunction_t *out, int *grid)
{
    JitState *j = (JitState *)c->jit;
    if (!j->fnp[mode]) {
        hipFunction_t f0;
        int rc = jit_resolve(c, mode, false, &f0);   // compiles the family
        if (rc != MJ_OK) return rc;
        hipModule_t mod = j->mods[family_of(mode)]->mod;
        char name[64];
        snprintf(name, sizeof name, "mj_pstage_%d", mode);
        hipFunction_t f;
        hipError_t e = hipModuleGetFunction(&f, mod, name);
        if (e != hipSuccess) return mj_hip_fail(MJ_EHIP, std::string("hipModuleGetFunction ") + name + ": " + hipGetErrorString(e));
        int per_cu = 0, ncu = 0;
        if (hipModuleOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, f, j->nthr, j->pers_shm) != hipSuccess ||
            hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount, c->device) != hipSuccess) {
            return mj_hip_fail(MJ_EHIP, "persistent stage kernel: occupancy query failed");
        }
        int g = std::max(1, per_cu) * std::max(1, ncu);
        g = std::min(g, j->nblocks);
        g = std::max(8, g / 8 * 8);
        j->fnp[mode] = f;
        j->pers_grid[mode] = g;
    }
    *out = j->fnp[mode];
    *grid = j->pers_grid[mode];
    return MJ_OK;
}

static bool persist_enabled()
{
    const char *e = getenv("MJ_PERSIST");
    return e && e[0] == '1';
}

int mj_jit_launch(mj_ctx *c, int mode, bool noise, const KArgs &a, hipStream_t s)
{
    JitState *j = (JitState *)c->jit;
    if (!noise && j->pers_ok && persistent_mode(mode) && persist_enabled()) {
        hipFunction_t fp;
        int grid = 0;
        int rc = jit_resolve_persistent(c, mode, &fp, &grid);
        if (rc != MJ_OK) return rc;
        KArgs arg = a;
        void *params[] = {&arg};
        hipError_t e = hipModuleLaunchKernel(fp, (unsigned)grid, 1, 1, (unsigned)j->nthr, 1, 1, (unsigned)j->pers_shm, s,
                                             params, nullptr);
        if (e != hipSuccess) return mj_hip_fail(MJ_EHIP, std::string("hipModuleLaunchKernel (persistent): ") + hipGetErrorString(e));
        return MJ_OK;
    }
    hipFunction_t f;
    int rc = jit_resolve(c, mode, noise, &f);
    if (rc != MJ_OK) return rc;
    KArgs arg = a;
    void *params[] = {&arg};
    const bool fused = mode == MODE_HEUNF || mode == MODE_SIBF || mode == MODE_DEPF;
    hipError_t e = hipModuleLaunchKernel(f, (unsigned)(fused ? j->fuse_nblocks : a.nblocks), 1, 1,
                                         (unsigned)(fused ? j->fuse_nthr : j->nthr), 1, 1,
                                         (unsigned)(fused ? j->fuse_shm : j->shm), s, params, nullptr);
    if (e != hipSuccess) return mj_hip_fail(MJ_EHIP, std::string("hipModuleLaunchKernel: ") + hipGetErrorString(e));
    return MJ_OK;
}
