// Body of the fused field + integrator-stage kernel, shared by the
// ahead-of-time kernels (runtime geometry, mj_kernels.hip) and the kernels
// compiled per Hamiltonian at set-up (compile-time geometry and unrolled
// stencil, mj_jit.hip).  The geometry policy G supplies tile/lattice sizes and
// the stencil sum; both policies sum the stencil in the same order, so the two
// paths give identical results.
//
// One kernel evaluates B_eff = -dH/dm at every site of a tile and applies one
// integrator stage in registers, so a stage is one pass over HBM:
//   - the state (SoA mx|my|mz, FP64) of the tile plus a halo of the stencil
//     reach is staged in LDS (open boundaries zero-filled, periodic wrapped),
//     then every site sums its translation-invariant 3x3 blocks from LDS;
//   - Zeeman (uniform or per-site B order parameter) and the dipolar H_fft
//     (read from the FFT output grid) are added in the epilogue;
//   - the stage (reference Euler / two-half-step Heun, SIB, Depondt) and the
//     in-register Philox thermal field finish the site;
//   - optionally the energy of the stencil state is reduced per block, and
//     block 0 folds the previous kernel's per-block partials into E.
// Reference: field hamiltonian_collection.f90:433-454; stage loop
// spindynamics.f90:260-323; energy hamiltonian_collection.f90:365-400.
#pragma once

__device__ __forceinline__ bool mj_wrap_idx(int &g, int n, int periodic)
{
    if (g >= 0 && g < n) return true;
    if (!periodic) return false;
    g %= n;
    if (g < 0) g += n;
    return true;
}

// workgroups are dispatched round-robin over the 8 XCDs; give each XCD a
// contiguous band of tiles so halos are shared inside one L2
__device__ __forceinline__ int mj_xcd_remap(int bid, int nb)
{
    if ((nb & 7) != 0) return bid;
    return (bid & 7) * (nb >> 3) + (bid >> 3);
}

// The neighbour sums, complete at this point of the program.  Without it the
// compiler moves the sums' additions past the next branch of the site algebra
// and keeps every neighbour's operands in registers across it: 160 VGPRs for
// the two-site fused step of the 18-neighbour stencil, 116 with it.
__device__ __forceinline__ void mj_settle(double &ax, double &ay, double &az)
{
    asm volatile("" : "+v"(ax), "+v"(ay), "+v"(az));
}

// Deterministic block reductions.  Full wavefronts: xor butterfly inside the
// wave (every lane ends with the same value: each step adds the same two
// operands in either order), then the per-wave values in wave order; one
// barrier instead of a log2(nthr)-step tree.  Blocks that are not a multiple
// of 64 threads (tiny lattices) use a tree over LDS.  Every thread gets the
// result; `red` (nthr doubles) may be reused after the call.
template <class OP>
__device__ __forceinline__ double mj_block_reduce(double v, double *red, int nthr, OP op)
{
    const int t = threadIdx.x;
    if ((nthr & 63) == 0) {
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) v = op(v, __shfl_xor(v, o, 64));
        if ((t & 63) == 0) red[t >> 6] = v;
        __syncthreads();
        double r = red[0];
        for (int w = 1; w < (nthr >> 6); ++w) r = op(r, red[w]);
        __syncthreads();
        return r;
    }
    red[t] = v;
    __syncthreads();
    for (int s = 512; s > 0; s >>= 1) {
        if (t < s && t + s < nthr) red[t] = op(red[t], red[t + s]);
        __syncthreads();
    }
    double r = red[0];
    __syncthreads();
    return r;
}

struct MjAdd {
    __device__ __forceinline__ double operator()(double a, double b) const { return a + b; }
};
struct MjMax {
    __device__ __forceinline__ double operator()(double a, double b) const { return fmax(a, b); }
};

__device__ __forceinline__ double mj_block_sum(double v, double *red, int nthr)
{
    return mj_block_reduce(v, red, nthr, MjAdd());
}

__device__ __forceinline__ double mj_block_max(double v, double *red, int nthr)
{
    return mj_block_reduce(v, red, nthr, MjMax());
}

// runtime-geometry policy (ahead-of-time kernels)
struct RtGeom {
    static constexpr int kNit = 0;         // trips of the tile fill: known only at run time
    static constexpr bool kDma = false;    // direct global -> LDS fill (compile-time geometry only)
    static constexpr bool kCfLds = false;  // the stencil's blocks staged in LDS behind the tile,
    static constexpr int kTrips = 1;       // so many values a thread at once
    // LDS stride between the x, y, z components of the tile (the tile size here)
    static __device__ __forceinline__ int tstride(const KArgs &, int T) { return T; }
    static __device__ __forceinline__ int bx(const KArgs &a) { return a.bx; }
    static __device__ __forceinline__ int by(const KArgs &a) { return a.by; }
    static __device__ __forceinline__ int bz(const KArgs &a) { return a.bz; }
    static __device__ __forceinline__ int rx(const KArgs &a) { return a.rx; }
    static __device__ __forceinline__ int ry(const KArgs &a) { return a.ry; }
    static __device__ __forceinline__ int rz(const KArgs &a) { return a.rz; }
    static __device__ __forceinline__ int nx(const KArgs &a) { return a.nx; }
    static __device__ __forceinline__ int ny(const KArgs &a) { return a.ny; }
    static __device__ __forceinline__ int nz(const KArgs &a) { return a.nz; }
    static __device__ __forceinline__ int ntx(const KArgs &a) { return a.ntx; }
    static __device__ __forceinline__ int nty(const KArgs &a) { return a.nty; }
    static __device__ __forceinline__ int nblocks(const KArgs &a) { return a.nblocks; }
    // tile of this workgroup, and the slot of its energy partial (the tile's
    // index: partials are summed in tile order whichever workgroup made them)
    static __device__ __forceinline__ int block(const KArgs &a) { return mj_xcd_remap(blockIdx.x, a.nblocks); }
    static __device__ __forceinline__ int part(const KArgs &a) { return mj_xcd_remap(blockIdx.x, a.nblocks); }
    static __device__ __forceinline__ void stencil(const KArgs &a, const double *L, int T, int c, double &ax,
                                                   double &ay, double &az)
    {
        sum(a.n_ent, a.ofs, a.cf, L, T, c, ax, ay, az);
    }
    // every entry as a full block (a zero coefficient adds an exact zero), in
    // one loop without a test of its kind: the reads of several entries are in
    // flight together
    static __device__ __forceinline__ void sum(int n, const int *ofs, const double *cf, const double *L, int T, int c,
                                               double &ax, double &ay, double &az)
    {
#pragma unroll 4
        for (int k = 0; k < n; ++k) {
            const int j = c + ofs[k];
            const double *q = cf + 9 * k;
            const double mx = L[j], my = L[T + j], mz = L[2 * T + j];
            ax = fma(q[0], mx, ax);
            ax = fma(q[1], my, ax);
            ax = fma(q[2], mz, ax);
            ay = fma(q[3], mx, ay);
            ay = fma(q[4], my, ay);
            ay = fma(q[5], mz, ay);
            az = fma(q[6], mx, az);
            az = fma(q[7], my, az);
            az = fma(q[8], mz, az);
        }
    }
};


// The same for the ahead-of-time stage kernels, with the blocks staged in LDS
// (where the host made room for them, KArgs::cf_lds): they run on lattices of a
// few tiles, where a launch is the latency of one tile, and the blocks' way
// through a cold scalar cache came after the tile's instead of with it (32x32,
// Heun, us per step: square 11.5 -> 11.2, triangular 15.1 -> 15.3, integration 4
// 26.5 -> 25.3 and 34.6 -> 33.6).  A tile of one wavefront copies three values a
// thread: all in flight before the tile's loads, stored after them (24x24, 100
// steps, copied one after the other -> so: triangular Heun 1465 -> 1372 us, SIB
// 1448 -> 1364, square 1055 -> 1045).
struct AotGeom : RtGeom {
    static constexpr bool kCfLds = true;
    static constexpr int kTrips = 3;
    static __device__ __forceinline__ void stencil(const KArgs &a, const double *L, int T, int c, double &ax,
                                                   double &ay, double &az)
    {
        if (a.cf_lds) sum(a.n_ent, a.ofs, L + 3 * T, L, T, c, ax, ay, az);
        else sum(a.n_ent, a.ofs, a.cf, L, T, c, ax, ay, az);
    }
    // the blocks, a few values a thread, in flight before the tile's loads ...
    static __device__ __forceinline__ void load(const KArgs &a, double v[kTrips])
    {
        if (!a.cf_lds) return;
#pragma unroll
        for (int i = 0; i < kTrips; ++i) v[i] = a.cf[min((int)(threadIdx.x + i * blockDim.x), 9 * a.n_ent - 1)];
    }
    // ... and stored after them
    static __device__ __forceinline__ void store(const KArgs &a, double *L, int T, const double v[kTrips])
    {
        if (!a.cf_lds) return;
        int t = threadIdx.x;
#pragma unroll
        for (int i = 0; i < kTrips; ++i, t += blockDim.x)
            if (t < 9 * a.n_ent) L[3 * T + t] = v[i];
        for (; t < 9 * a.n_ent; t += blockDim.x) L[3 * T + t] = a.cf[t];
    }
};

// The thread's own site in a tile, and the own-site operands of the epilogue
// (issued early: their latency overlaps the tile fill or the stencil).
struct SiteCtx {
    int lx, ly, lz, gx, gy, gz;
    bool active;
    int64_t gi;
    v3 pre_aux, pre_own;
    v3 th;            // NOISE stages: the thermal field, when computed ahead of the epilogue
    uint64_t nstep;   // NOISE stages with a compile-time geometry: the step of the Philox counter
};

// The Philox thermal field of a NOISE stage needs only (seed, step, site), not
// the tile: it is computed while the tile loads are in flight, and its
// Langevin term on m0 (HEUN2, thermal_term) is formed in the epilogue.  A field
// supplied by the caller (a.noise) is read in the epilogue too
// (site_thermal_final): loads here would make the Philox path wait for the
// tile loads.
template <int MODE>
__device__ __forceinline__ v3 thermal_term(const KArgs &a, const SiteCtx &s, v3 bt)
{
    if constexpr (MODE == MODE_HEUN2) return llg_torque(mj_unit(s.pre_own).n, bt, a.alpha);
    return bt;
}

template <int MODE, bool NOISE>
__device__ __forceinline__ void site_thermal(const KArgs &a, SiteCtx &s)
{
    if constexpr (NOISE) {
        if (s.active && !a.noise) {
            const v3 g = normals3(a.seed, s.nstep, (uint32_t)s.gi);
            s.th = mk3(a.sigma * g.x, a.sigma * g.y, a.sigma * g.z);
        }
    }
}

// Epilogue: the early result (kernels with a compile-time tile fill), else the
// whole thermal part here, as the ahead-of-time kernels have no fill to overlap.
template <int MODE, class G>
__device__ __forceinline__ v3 site_thermal_final(const KArgs &a, const SiteCtx &s)
{
    const int64_t np = a.np;
    if (a.noise) return thermal_term<MODE>(a, s, mk3(a.noise[s.gi], a.noise[s.gi + np], a.noise[s.gi + 2 * np]));
    if constexpr (G::kNit > 0) {
        return thermal_term<MODE>(a, s, s.th);
    } else {
        const v3 g = normals3(a.seed, a.stepp ? *a.stepp + a.step : a.step, (uint32_t)s.gi);
        return thermal_term<MODE>(a, s, mk3(a.sigma * g.x, a.sigma * g.y, a.sigma * g.z));
    }
}

// Interior tile straight from global memory into LDS: each lane moves 16 B,
// two neighbouring sites of a tile row (tile rows and the lattice rows have
// even length and start at even sites, so a pair never straddles a row and is
// 16-byte aligned), and lands at its wave's LDS base + 16 * lane.  Every lane
// of every wave issues (the components are padded to whole trips of the
// workgroup: surplus lanes reload the last pair into the padding), so the
// code is branch-free: no join after which the compiler's waits for other
// loads would become full waits.  The loads bypass the registers; the caller
// waits for them (vmcnt) before the barrier.
template <class G>
__device__ __forceinline__ void tile_fill_direct(const KArgs &a, double *lds, int64_t base)
{
    constexpr int BX = G::kBx, BY = G::kBy, BZ = G::kBz, RX = G::kRx, RY = G::kRy, RZ = G::kRz;
    constexpr int SX = BX + 2 * RX, SY = BY + 2 * RY, SZ = BZ + 2 * RZ;
    constexpr int T = SX * SY * SZ, P = T / 2, NTHR = BX * BY * BZ, TS = G::kT;
    constexpr int NX = G::kNx, NY = G::kNy;
    static_assert(TS >= 2 * NTHR * ((P + NTHR - 1) / NTHR), "component stride must hold whole trips");
    const int64_t np = a.np;
    const int wave = (int)threadIdx.x >> 6;
#pragma unroll
    for (int p0 = 0; p0 < P; p0 += NTHR) {
        const int q = min(p0 + (int)threadIdx.x, P - 1);
        const int t = 2 * q;
        const int lx = t % SX;
        const int r = t / SX;
        const int ly = r % SY;
        const int lz = r / SY;
        const int64_t g = base + lx + (int64_t)NX * ((int64_t)ly + (int64_t)NY * lz);
        const int wfirst = __builtin_amdgcn_readfirstlane(p0 + 64 * wave);
#pragma unroll
        for (int c = 0; c < 3; ++c)
            __builtin_amdgcn_global_load_lds((const void *)(a.src + g + c * np),
                                             (__attribute__((address_space(3))) void *)(lds + c * TS + 2 * wfirst), 16,
                                             0, 0);
    }
}

// One tile of the state plus its halo into LDS: interior tiles take a
// branch-free path, boundary tiles wrap (periodic) or zero-fill (open).  With
// a compile-time trip count the loads go to registers first and the stage's
// thermal part is computed before they are stored.
template <int MODE, bool NOISE, class G>
__device__ __forceinline__ void tile_fill(const KArgs &a, double *lds, int x0, int y0, int z0, SiteCtx &st)
{
    const int BX = G::bx(a), BY = G::by(a), BZ = G::bz(a);
    const int RX = G::rx(a), RY = G::ry(a), RZ = G::rz(a);
    const int NX = G::nx(a), NY = G::ny(a), NZ = G::nz(a);
    const int SX = BX + 2 * RX, SY = BY + 2 * RY, SZ = BZ + 2 * RZ;
    const int TT = SX * SY * SZ;          // tile sites
    const int T = G::tstride(a, TT);      // LDS component stride
    const int nthr = BX * BY * BZ;
    const int64_t np = a.np;
    const bool interior = x0 - RX >= 0 && x0 + BX + RX <= NX && y0 - RY >= 0 && y0 + BY + RY <= NY &&
                          z0 - RZ >= 0 && z0 + BZ + RZ <= NZ;
    if (interior) {
        const int64_t base = (int64_t)(x0 - RX) + (int64_t)NX * ((int64_t)(y0 - RY) + (int64_t)NY * (z0 - RZ));
        if constexpr (G::kNit > 0) {
            constexpr int NIT = G::kNit;
            double vx[NIT], vy[NIT], vz[NIT];
            // unconditional loads (the last trip's surplus threads reload element
            // T-1 and store nothing): straight-line code keeps the compiler's
            // waits on the tile loads exact, so the thermal part overlaps them
#pragma unroll
            for (int it = 0; it < NIT; ++it) {
                const int t = min(threadIdx.x + it * nthr, TT - 1);
                const int lx = t % SX;
                const int r = t / SX;
                const int ly = r % SY;
                const int lz = r / SY;
                const int64_t g = base + lx + (int64_t)NX * ((int64_t)ly + (int64_t)NY * lz);
                vx[it] = a.src[g];
                vy[it] = a.src[g + np];
                vz[it] = a.src[g + 2 * np];
            }
            site_thermal<MODE, NOISE>(a, st);
#pragma unroll
            for (int it = 0; it < NIT; ++it) {
                const int t = threadIdx.x + it * nthr;
                if (t < TT) {
                    lds[t] = vx[it];
                    lds[T + t] = vy[it];
                    lds[2 * T + t] = vz[it];
                }
            }
            return;
        }
        const int nit = (TT + nthr - 1) / nthr;
        for (int it = 0; it < nit; ++it) {
            const int t = threadIdx.x + it * nthr;
            if (t >= TT) break;
            const int lx = t % SX;
            const int r = t / SX;
            const int ly = r % SY;
            const int lz = r / SY;
            const int64_t g = base + lx + (int64_t)NX * ((int64_t)ly + (int64_t)NY * lz);
            lds[t] = a.src[g];
            lds[T + t] = a.src[g + np];
            lds[2 * T + t] = a.src[g + 2 * np];
        }
    } else {
        if constexpr (G::kNit > 0) site_thermal<MODE, NOISE>(a, st);
        for (int t = threadIdx.x; t < TT; t += nthr) {
            const int lx = t % SX;
            const int r = t / SX;
            const int ly = r % SY;
            const int lz = r / SY;
            int gx = x0 + lx - RX, gy = y0 + ly - RY, gz = z0 + lz - RZ;
            double vx = 0.0, vy = 0.0, vz = 0.0;
            if (mj_wrap_idx(gx, NX, a.px) && mj_wrap_idx(gy, NY, a.py) && mj_wrap_idx(gz, NZ, a.pz)) {
                const int64_t g = (int64_t)gx + (int64_t)NX * ((int64_t)gy + (int64_t)NY * gz);
                vx = a.src[g];
                vy = a.src[g + np];
                vz = a.src[g + 2 * np];
            }
            lds[t] = vx;
            lds[T + t] = vy;
            lds[2 * T + t] = vz;
        }
    }
}

template <int MODE, bool NOISE, class G>
__device__ __forceinline__ SiteCtx site_begin(const KArgs &a, int x0, int y0, int z0, uint64_t nstep)
{
    SiteCtx s;
    const int BX = G::bx(a), BY = G::by(a);
    const int64_t np = a.np;
    s.lx = threadIdx.x % BX;
    s.ly = (threadIdx.x / BX) % BY;
    s.lz = threadIdx.x / (BX * BY);
    s.gx = x0 + s.lx;
    s.gy = y0 + s.ly;
    s.gz = z0 + s.lz;
    s.active = s.gx < G::nx(a) && s.gy < G::ny(a) && s.gz < G::nz(a);
    s.gi = s.active ? (int64_t)s.gx + (int64_t)G::nx(a) * ((int64_t)s.gy + (int64_t)G::ny(a) * s.gz) : 0;
    constexpr bool kAux = MODE == MODE_HEUN2 || MODE == MODE_DEP2;
    constexpr bool kOwn = (MODE == MODE_HEUN2 && NOISE) || MODE == MODE_SIB2 || MODE == MODE_DEP2;
    s.pre_aux = mk3(0.0, 0.0, 0.0);
    s.pre_own = mk3(0.0, 0.0, 0.0);
    s.th = mk3(0.0, 0.0, 0.0);
    s.nstep = nstep;
    // compile-time geometries load unconditionally (gi = 0 off the lattice): no
    // join that would make the thermal part wait for them
    constexpr bool kAll = G::kNit > 0;
    if constexpr (kAux && !(NOISE && G::kNit > 0)) {
        if (kAll || s.active) s.pre_aux = mk3(a.aux[s.gi], a.aux[s.gi + np], a.aux[s.gi + 2 * np]);
    }
    if constexpr (kOwn) {
        if (kAll || s.active) s.pre_own = mk3(a.own[s.gi], a.own[s.gi + np], a.own[s.gi + 2 * np]);
    }
    return s;
}

// Field at the own site from the tile in LDS, the block reductions (energy,
// max |B|: slot `part`; `fold`: this block folds the previous kernel's
// energy partials) and the integrator epilogue.
template <int MODE, bool NOISE, class G>
__device__ __forceinline__ void site_end(const KArgs &a, double *lds, const SiteCtx &st, int part, bool fold)
{
    const int BX = G::bx(a), BY = G::by(a), BZ = G::bz(a);
    const int RX = G::rx(a), RY = G::ry(a), RZ = G::rz(a);
    const int SX = BX + 2 * RX, SY = BY + 2 * RY, SZ = BZ + 2 * RZ;
    const int T = G::tstride(a, SX * SY * SZ);   // LDS component stride
    const int nthr = BX * BY * BZ;
    const int64_t np = a.np;
    const int lx = st.lx, ly = st.ly, lz = st.lz, gx = st.gx, gy = st.gy, gz = st.gz;
    const bool active = st.active;
    const int64_t gi = st.gi;
    const v3 pre_aux = st.pre_aux, pre_own = st.pre_own;
    (void)pre_aux;
    (void)pre_own;
    (void)SZ;

    double ax = 0.0, ay = 0.0, az = 0.0;   // sum_d C_d m_{i+d}  (= (H + H^T) m at i)
    v3 m;                                  // state at the own site
    if (a.use_stencil) {
        const int c = (lz + RZ) * SX * SY + (ly + RY) * SX + (lx + RX);
        m = mk3(lds[c], lds[T + c], lds[2 * T + c]);
        G::stencil(a, lds, T, c, ax, ay, az);
        mj_settle(ax, ay, az);
    } else {
        m = active ? mk3(a.src[gi], a.src[gi + np], a.src[gi + 2 * np]) : mk3(0.0, 0.0, 0.0);
        if (active) {
            ax = a.fld_in[gi];
            ay = a.fld_in[gi + np];
            az = a.fld_in[gi + 2 * np];
        }
    }

    // Zeeman: Z^T b (uniform or per site)
    double zx = 0.0, zy = 0.0, zz = 0.0;
    if (a.bmode == 1) {
        zx = a.zb[0];
        zy = a.zb[1];
        zz = a.zb[2];
    } else if (a.bmode == 3 && active) {
        double bxv = 0.0, byv = 0.0, bzv = 0.0;
        // unrolled over the at most 4 maps: constant indices into wmap keep a
        // kernel's local copy of the arguments in registers (no scratch)
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            if (k < a.nmaps) {
                const double *f = a.maps + (int64_t)k * 3 * np;
                bxv = bxv + a.wmap[3 * k] * f[gi];
                byv = byv + a.wmap[3 * k + 1] * f[gi + np];
                bzv = bzv + a.wmap[3 * k + 2] * f[gi + 2 * np];
            }
        }
        zx = (bxv * a.z[0] + byv * a.z[3]) + bzv * a.z[6];
        zy = (bxv * a.z[1] + byv * a.z[4]) + bzv * a.z[7];
        zz = (bxv * a.z[2] + byv * a.z[5]) + bzv * a.z[8];
    } else if (a.bmode == 2 && active) {
        const double bxv = a.bmap[gi], byv = a.bmap[gi + np], bzv = a.bmap[gi + 2 * np];
        zx = (bxv * a.z[0] + byv * a.z[3]) + bzv * a.z[6];
        zy = (bxv * a.z[1] + byv * a.z[4]) + bzv * a.z[7];
        zz = (bxv * a.z[2] + byv * a.z[5]) + bzv * a.z[8];
    }
    // dipolar H_fft at this site (the padded grid keeps the lattice at its origin)
    double hx = 0.0, hy = 0.0, hz = 0.0;
    if (a.hdip && active) {
        const int64_t h = (int64_t)gx + (int64_t)a.dnx * ((int64_t)gy + (int64_t)a.dny * gz);
        hx = a.hdip[h];
        hy = a.hdip[h + a.hstride];
        hz = a.hdip[h + 2 * a.hstride];
    }
    // B = -(H m + H^T m + Z^T b) - 2 H_fft      (hamiltonian_collection.f90:442-453)
    v3 B = mk3(-(ax + zx) - 2.0 * hx, -(ay + zy) - 2.0 * hy, -(az + zz) - 2.0 * hz);

    // max |B| over the block (update_time.f90:58-68: the field of the last stage, no thermal part)
    if (a.bmax_part) {
        const double nb = active ? norm3(B) : 0.0;
        __syncthreads();
        const double s = mj_block_max(nb, lds, nthr);
        if (threadIdx.x == 0) a.bmax_part[part] = s;
    }
    // energy of the stencil state: m.(H m) + b.(Z m) + m.H_fft = m.(acc/2 + Z^T b + h)
    if (a.energy) {
        double e = 0.0;
        if (active)
            e = mj_site_energy(m, mk3(ax, ay, az), mk3(zx + hx, zy + hy, zz + hz));
        __syncthreads();
        double s = mj_block_sum(e, lds, nthr);
        if (threadIdx.x == 0) a.epart[part] = s;
    }
    // block 0 folds the previous kernel's partials into E (stream order makes them complete)
    if (a.ered_in && fold) {
        __syncthreads();
        double v = 0.0;
        for (int i = threadIdx.x; i < a.n_ered; i += nthr) v += a.ered_in[i];
        double s = mj_block_sum(v, lds, nthr);
        if (threadIdx.x == 0) *a.e_out = s * a.e_scale;
    }
    if (!active) return;

    const double alpha = a.alpha;
    // the stage's effective field (no thermal term): MODE_FIELD's product, or
    // the field of a step's last stage when the host keeps it
    if (a.fld_out) {
        a.fld_out[gi] = B.x;
        a.fld_out[gi + np] = B.y;
        a.fld_out[gi + 2 * np] = B.z;
    }
    if constexpr (MODE == MODE_FIELD) {
    } else if constexpr (MODE == MODE_EULER) {
        const MjUnit u = mj_unit(m);
        // Dint = 1 D (get_Dmode_int)
        const v3 D = llg_torque(u.n, B, alpha);
        v3 o;
        if constexpr (NOISE) o = euler_step(m, u, D, a.kdt, llg_torque(u.n, site_thermal_final<MODE, G>(a, st), alpha), a.kdt);
        else o = euler_step0(m, u, D, a.kdt);
        a.dst[gi] = o.x;
        a.dst[gi + np] = o.y;
        a.dst[gi + 2 * np] = o.z;
    } else if constexpr (MODE == MODE_RKS) {
        // stage i of integration 4 (spindynamics.f90:294-318 with get_Dmode_int,
        // solver_order.f90:46-58): D_i = LLG(B(m), m); Dint = w_1 D_1 + ... + w_i D_i;
        // m' = euler(m, Dint, 0, dt_i).  Unrolled over the at most 7 earlier stages
        // (constant indices keep the argument block in registers).
        const MjUnit u = mj_unit(m);
        const v3 D = llg_torque(u.n, B, alpha);
        v3 dint = mk3(0.0, 0.0, 0.0);
#pragma unroll
        for (int k = 0; k < 7; ++k) {
            if (k < a.nprev) {
                const double *p = a.dprev[k];
                dint = fma3(a.wrk[k], mk3(p[gi], p[gi + np], p[gi + 2 * np]), dint);
            }
        }
        double wi = 0.0;
#pragma unroll
        for (int k = 0; k < 8; ++k)
            if (k == a.nprev) wi = a.wrk[k];
        const v3 o = euler_step0(m, u, fma3(wi, D, dint), a.kdt);
        if (a.dout) {
            a.dout[gi] = D.x;
            a.dout[gi + np] = D.y;
            a.dout[gi + 2 * np] = D.z;
        }
        a.dst[gi] = o.x;
        a.dst[gi + np] = o.y;
        a.dst[gi + 2 * np] = o.z;
    } else if constexpr (MODE == MODE_HEUN1) {
        // stage 1 of integration 2: D1 = LLG(B(m0), m0); m1 = euler(m0, 1*D1 + 0*D2, 0, dt/2)
        const MjUnit u = mj_unit(m);
        const v3 D = llg_torque(u.n, B, alpha);
        const v3 o = euler_step0(m, u, D, a.kdt);
        a.dst[gi] = o.x;
        a.dst[gi + np] = o.y;
        a.dst[gi + 2 * np] = o.z;
        a.aux[gi] = D.x;
        a.aux[gi + np] = D.y;
        a.aux[gi + 2 * np] = D.z;
    } else if constexpr (MODE == MODE_HEUN2) {
        // stage 2: D2 = LLG(B(m1), m1); m2 = euler(m1, 0.5 D1 + 0.5 D2, DT(m0), dt/2)
        const MjUnit u = mj_unit(m);
        // Dint = D1/2 + D2/2 (get_Dmode_int)
        const v3 d = pre_aux + llg_torque(u.n, B, alpha);
        v3 o;
        if constexpr (NOISE) {
            // Langevin term of the last stage on m0 (pre_own, site_thermal), spindynamics.f90:269-271,311
            o = euler_step(m, u, d, 0.5 * a.kdt, site_thermal_final<MODE, G>(a, st), a.kdt);
        } else {
            o = euler_step0(m, u, d, 0.5 * a.kdt);
        }
        a.dst[gi] = o.x;
        a.dst[gi + np] = o.y;
        a.dst[gi + 2 * np] = o.z;
    } else {
        if constexpr (NOISE) {
            const v3 bt = site_thermal_final<MODE, G>(a, st);
            B = mk3(B.x + bt.x, B.y + bt.y, B.z + bt.z);
        }
        if constexpr (MODE == MODE_SIB1) {
            const v3 p = cayley_mid(m, sib_vec(m, B, alpha, -0.5 * a.kdt));
            a.dst[gi] = p.x;
            a.dst[gi + np] = p.y;
            a.dst[gi + 2 * np] = p.z;
        } else if constexpr (MODE == MODE_SIB2) {
            // m is the midpoint p here
            const v3 o = cayley(pre_own, sib_vec(m, B, alpha, -0.5 * a.kdt));
            a.dst[gi] = o.x;
            a.dst[gi + np] = o.y;
            a.dst[gi + 2 * np] = o.z;
        } else if constexpr (MODE == MODE_DEP1) {
            v3 b1 = dep_field(m, B, alpha);
            v3 mt = dep_rotate(m, b1, a.kdt);
            a.dst[gi] = mt.x;
            a.dst[gi + np] = mt.y;
            a.dst[gi + 2 * np] = mt.z;
            a.aux[gi] = b1.x;
            a.aux[gi + np] = b1.y;
            a.aux[gi + 2 * np] = b1.z;
        } else if constexpr (MODE == MODE_DEP2) {
            v3 b2 = dep_field(m, B, alpha);   // m is the predictor here
            const v3 b1 = pre_aux;
            v3 ba = mk3(0.5 * (b1.x + b2.x), 0.5 * (b1.y + b2.y), 0.5 * (b1.z + b2.z));
            v3 o = dep_rotate(pre_own, ba, a.kdt);
            a.dst[gi] = o.x;
            a.dst[gi + np] = o.y;
            a.dst[gi + 2 * np] = o.z;
        }
    }
}

template <int MODE, bool NOISE, class G>
__device__ __forceinline__ void stage_body(const KArgs &a, double *lds)
{
    const int bid = G::block(a);
    const int tx = bid % G::ntx(a);
    const int tr = bid / G::ntx(a);
    const int ty = tr % G::nty(a);
    const int tz = tr / G::nty(a);
    const int x0 = tx * G::bx(a), y0 = ty * G::by(a), z0 = tz * G::bz(a);
    // interior tiles of the compile-time geometries: the tile goes straight to
    // LDS first, before any other load (the compiler does not count these loads
    // among the ones in flight, so a later wait on a register load would also
    // wait for them); the thermal field is computed while they land
    // the Philox step, read before anything is written (a scalar load)
    uint64_t nstep = 0;
    if constexpr (NOISE && G::kNit > 0) nstep = a.stepp ? *a.stepp + a.step : a.step;
    bool direct = false;
    if constexpr (G::kDma) {
        constexpr int RX = G::kRx, RY = G::kRy, RZ = G::kRz, NX = G::kNx, NY = G::kNy;
        direct = a.use_stencil && (((unsigned long long)a.src) & 15ull) == 0 && x0 - RX >= 0 &&
                 x0 + G::kBx + RX <= NX && y0 - RY >= 0 && y0 + G::kBy + RY <= NY && z0 - RZ >= 0 &&
                 z0 + G::kBz + RZ <= G::nz(a);
        if (direct)
            tile_fill_direct<G>(a, lds,
                                (int64_t)(x0 - RX) + (int64_t)NX * ((int64_t)(y0 - RY) + (int64_t)NY * (z0 - RZ)));
    }
    SiteCtx st = site_begin<MODE, NOISE, G>(a, x0, y0, z0, nstep);
    [[maybe_unused]] double cf[G::kTrips];
    if constexpr (G::kCfLds) G::load(a, cf);
    if (direct) {
        site_thermal<MODE, NOISE>(a, st);
        __builtin_amdgcn_s_waitcnt(0);   // this wave's tile loads are in LDS
    } else if (a.use_stencil) {
        tile_fill<MODE, NOISE, G>(a, lds, x0, y0, z0, st);
    } else if constexpr (G::kNit > 0) {
        site_thermal<MODE, NOISE>(a, st);
    }
    // with the thermal part computed early, the epilogue's aux operand is
    // loaded after it (fewer registers live across it)
    constexpr bool kAux = MODE == MODE_HEUN2 || MODE == MODE_DEP2;
    if constexpr (kAux && NOISE && G::kNit > 0) st.pre_aux = mk3(a.aux[st.gi], a.aux[st.gi + a.np], a.aux[st.gi + 2 * a.np]);
    if constexpr (G::kCfLds)
        G::store(a, lds, (G::bx(a) + 2 * G::rx(a)) * (G::by(a) + 2 * G::ry(a)) * (G::bz(a) + 2 * G::rz(a)), cf);
    if (a.use_stencil) __syncthreads();
    site_end<MODE, NOISE, G>(a, lds, st, G::part(a), blockIdx.x == 0);
}


// Persistent form of stage_body for stages that read nothing but their tile
// (stage 1 of the two-stage integrators; compile-time geometry with the direct
// global -> LDS fill, a whole number of tiles per XCD band).  Each workgroup
// walks its XCD's band of tiles; the next interior tile goes from HBM straight
// into the second of two LDS buffers while the current one is computed, so the
// fill latency of all but the first tile is hidden.  Same arithmetic and
// energy-partial slots (the tile index) as stage_body.
template <int MODE, class G>
__device__ __forceinline__ void stage_fill_any(const KArgs &a, double *buf, int t)
{
    constexpr int RX = G::kRx, RY = G::kRy, RZ = G::kRz, NX = G::kNx, NY = G::kNy;
    const int tx = t % G::ntx(a), tr = t / G::ntx(a), ty = tr % G::nty(a), tz = tr / G::nty(a);
    const int x0 = tx * G::kBx, y0 = ty * G::kBy, z0 = tz * G::kBz;
    const bool direct = (((unsigned long long)a.src) & 15ull) == 0 && x0 - RX >= 0 && x0 + G::kBx + RX <= NX &&
                        y0 - RY >= 0 && y0 + G::kBy + RY <= NY && z0 - RZ >= 0 && z0 + G::kBz + RZ <= G::nz(a);
    if (direct) {
        tile_fill_direct<G>(a, buf, (int64_t)(x0 - RX) + (int64_t)NX * ((int64_t)(y0 - RY) + (int64_t)NY * (z0 - RZ)));
    } else {
        SiteCtx dummy;
        dummy.active = false;
        tile_fill<MODE, false, G>(a, buf, x0, y0, z0, dummy);
    }
}

template <int MODE, class G>
__device__ __forceinline__ void stage_body_persistent(const KArgs &a, double *lds)
{
    static_assert(G::kDma, "the persistent form needs the direct LDS fill");
    static_assert(MODE == MODE_HEUN1 || MODE == MODE_EULER || MODE == MODE_SIB1 || MODE == MODE_DEP1,
                  "stages with own-site operands are not persistent");
    constexpr int TS = G::kT;
    const int per_xcd = (int)gridDim.x >> 3;          // gridDim.x is a multiple of 8
    const int band = G::nblocks(a) >> 3;              // tiles per XCD band
    const int xcd = (int)blockIdx.x & 7, slot = (int)blockIdx.x >> 3;
    double *buf0 = lds, *buf1 = lds + 3 * TS;
    int k = 0;
    int t = slot < band ? xcd * band + slot : -1;
    if (t < 0) return;                                // uniform: the whole workgroup
    stage_fill_any<MODE, G>(a, buf0, t);
    for (;;) {
        const int jn = slot + (k + 1) * per_xcd;
        const int tn = jn < band ? xcd * band + jn : -1;
        __builtin_amdgcn_s_waitcnt(0);                // this wave's tile loads (and earlier stores) done
        __syncthreads();                              // every wave's: tile t is in LDS, the other buffer is free
        double *cur = (k & 1) ? buf1 : buf0;
        double *nxt = (k & 1) ? buf0 : buf1;
        if (tn >= 0) stage_fill_any<MODE, G>(a, nxt, tn);
        const int tx = t % G::ntx(a), tr = t / G::ntx(a), ty = tr % G::nty(a), tz = tr / G::nty(a);
        SiteCtx st = site_begin<MODE, false, G>(a, tx * G::kBx, ty * G::kBy, tz * G::kBz, 0);
        site_end<MODE, false, G>(a, cur, st, t, false);
        if (tn < 0) break;
        t = tn;
        ++k;
    }
}

// ---------------------------------------------------------------------------
// Both stages of integration 2, SIB or Depondt in one kernel (geometry F of
// mj_jit.hip: compile-time tile and stencil; the lattice's sizes and the
// coefficients compile-time for one Hamiltonian, run-time for a batch).  Regions of a tile (BX x BY x BZ sites, reach R):
//   S0 = the tile plus 2R on every side: m0, staged in LDS;
//   S1 = the tile plus R: stage 1 runs on every S1 site from S0 (the tile's own
//        sites and the ring around them) and its result goes to LDS, in S0's
//        place once every thread is done with S0;
// then stage 2 runs on the tile from S1 and writes m' out of place (other tiles
// still read m0 around this one).  S1 sites outside the tile repeat stage 1 of
// the neighbouring tiles with the same arithmetic, and every operation is the
// two-kernel path's, so m' equals that path's bit for bit while HBM sees m0 in
// and m' out, 48 B per site-step.
//   integration 2: stage 1 is HEUN1 (m1, the own sites keep D1 and the Langevin
//     torque on m0), stage 2 HEUN2;
//   SIB: stage 1 the midpoint p = m + g w(m, a1), stage 2 m' = cay(m, a2(p));
//   Depondt: stage 1 rotates m about its field b1 into the predictor (the own
//     sites keep b1), stage 2 rotates m about (b1 + b2)/2.
// SIB and Depondt add the same thermal field (Philox of the site and step) in
// both stages, so their ring draws it too.
//
// What bounds it is instruction issue (84% of the cycles at 2048x2048, 424 of 633
// VALU instructions per 64 sites FP64) and the LDS
// reads of the neighbour sums, 19 entries x 24 B per evaluation of the
// triangular workload.  A thread takes kSpt = 1 site, or 2 sites one above the
// other (tiles 32 wide, two wavefront halves per pair of rows), whose sums then
// read each neighbour they share once (24 entries instead of 38); S1 in S0's
// place leaves room for twice the workgroups per CU, the ring before the own
// sites and the settled sums for their registers (106 VGPRs, 160 before); no
// site of a tile is tested for lying off the lattice, which also keeps the
// code in a few long blocks.  Heun, triangular at 10 K with the energy every
// step: 1024x1024 37.1 -> 28.3 us per step, 2048x2048 (no energy) 112.6 -> 87.
//
// Energy partials of m0 are formed per tile of the two-kernel path (by rows of
// BY / kNsub, whole wavefronts, in that path's lane order; a pair's two rows
// are one wavefront there, and adding them first is that path's first
// butterfly); workgroup 0 of the next launch folds them in that path's order
// (a fold by the last workgroup to finish would need agent-scope fences in
// every workgroup, and those write back the whole L2 on this multi-XCD part).
// ---------------------------------------------------------------------------
// Zeeman of the fused kernel: the field mode is a compile-time constant of a
// per-Hamiltonian geometry (no branch between the stencil's LDS reads and their sums)
template <class F>
__device__ __forceinline__ v3 fused_zeeman(const KArgs &a, bool live, int64_t gi)
{
    double zx = 0.0, zy = 0.0, zz = 0.0;
    const int bmode = F::bmode(a);
    if (bmode == 1) {
        zx = a.zb[0];
        zy = a.zb[1];
        zz = a.zb[2];
    } else if (bmode == 2 && live) {
        const int64_t np = a.np;
        const double bxv = a.bmap[gi], byv = a.bmap[gi + np], bzv = a.bmap[gi + 2 * np];
        zx = (bxv * a.z[0] + byv * a.z[3]) + bzv * a.z[6];
        zy = (bxv * a.z[1] + byv * a.z[4]) + bzv * a.z[7];
        zz = (bxv * a.z[2] + byv * a.z[5]) + bzv * a.z[8];
    }
    return mk3(zx, zy, zz);
}

// coordinate g of a region position wrapped on a periodic axis of n sites;
// false off an open edge.  A tile of b sites and its halo of 2r reach past the
// lattice by less than one period unless n < b + 2r (then the remainder).
__device__ __forceinline__ bool fused_wrap(int &g, int n, int b, int r, int periodic)
{
    if (n < b + 2 * r) return mj_wrap_idx(g, n, periodic);
    const bool in = g >= 0 && g < n;
    g += g < 0 ? n : g >= n ? -n : 0;
    return in || periodic;
}

// global site of a region position (lattice coordinates g*), wrapped on
// periodic axes; false off an open edge
template <class F>
__device__ __forceinline__ bool fused_site(const KArgs &a, int gx, int gy, int gz, int64_t &gi)
{
    const bool in = fused_wrap(gx, F::nx(a), F::kBx, F::kRx, a.px) & fused_wrap(gy, F::ny(a), F::kBy, F::kRy, a.py) &
                    fused_wrap(gz, F::nz(a), F::kBz, F::kRz, a.pz);
    gi = (int64_t)gx + (int64_t)F::nx(a) * ((int64_t)gy + (int64_t)F::ny(a) * gz);
    return in;
}

template <class F>
__device__ __forceinline__ void fused_s0_fill(const KArgs &a, double *L0, int x0, int y0, int z0, bool direct,
                                              v3 v[F::kFill])
{
    constexpr int SX = F::kS0x, SY = F::kS0y, SZ = F::kS0z, T0 = F::kT0, NTHR = F::kAll;
    constexpr int RX2 = 2 * F::kRx, RY2 = 2 * F::kRy, RZ2 = 2 * F::kRz;
    const int64_t np = a.np;
    if constexpr (F::kDma) {
      if (direct) {
        // interior: 16-byte pairs along x straight into LDS (tile_fill_direct)
        constexpr int P = SX * SY * SZ / 2;
        static_assert(T0 >= 2 * NTHR * ((P + NTHR - 1) / NTHR), "S0 stride must hold whole trips");
        const int64_t base =
            (int64_t)(x0 - RX2) + (int64_t)F::nx(a) * ((int64_t)(y0 - RY2) + (int64_t)F::ny(a) * (z0 - RZ2));
        const int wave = (int)threadIdx.x >> 6;
#pragma unroll
        for (int p0 = 0; p0 < P; p0 += NTHR) {
            const int q = min(p0 + (int)threadIdx.x, P - 1);
            const int t = 2 * q;
            const int lx = t % SX;
            const int r = t / SX;
            const int ly = r % SY;
            const int lz = r / SY;
            const int64_t g = base + lx + (int64_t)F::nx(a) * ((int64_t)ly + (int64_t)F::ny(a) * lz);
            const int wfirst = __builtin_amdgcn_readfirstlane(p0 + 64 * wave);
#pragma unroll
            for (int c = 0; c < 3; ++c)
                __builtin_amdgcn_global_load_lds((const void *)(a.src + g + c * np),
                                                 (__attribute__((address_space(3))) void *)(L0 + c * T0 + 2 * wfirst),
                                                 16, 0, 0);
        }
        return;
      }
    }
    (void)direct;
    // boundary tiles, and lattices whose rows do not pair up: into registers, to
    // be stored by fused_s0_store after the thermal field is drawn
#pragma unroll
    for (int it = 0; it < F::kFill; ++it) {
        const int t = min((int)threadIdx.x + it * NTHR, SX * SY * SZ - 1);
        const int lx = t % SX;
        const int r = t / SX;
        const int ly = r % SY;
        const int lz = r / SY;
        int64_t g = 0;
        const bool in = fused_site<F>(a, x0 + lx - RX2, y0 + ly - RY2, z0 + lz - RZ2, g);
        const double *p = a.src + (in ? g : 0);
        const double vx = p[0], vy = p[np], vz = p[2 * np];
        v[it] = in ? mk3(vx, vy, vz) : mk3(0.0, 0.0, 0.0);
    }
}

template <class F>
__device__ __forceinline__ void fused_s0_store(double *L0, const v3 v[F::kFill])
{
    constexpr int T = F::kS0x * F::kS0y * F::kS0z, T0 = F::kT0;
#pragma unroll
    for (int it = 0; it < F::kFill; ++it) {
        const int t = (int)threadIdx.x + it * F::kAll;
        if (t < T) {
            L0[t] = v[it].x;
            L0[T0 + t] = v[it].y;
            L0[2 * T0 + t] = v[it].z;
        }
    }
}

// S1 position of ring site k (S1 minus the tile): z slabs, then y slabs of
// the tile's planes, then x slabs of its rows
template <class F>
__device__ __forceinline__ void fused_ring_pos(int k, int &sx, int &sy, int &sz)
{
    constexpr int BX = F::kBx, BY = F::kBy, BZ = F::kBz, RX = F::kRx, RY = F::kRy, RZ = F::kRz;
    constexpr int S1X = BX + 2 * RX, S1Y = BY + 2 * RY;
    constexpr int NZS = 2 * RZ * S1X * S1Y, NYS = 2 * RY * BZ * S1X;
    if (k < NZS) {
        const int plane = k / (S1X * S1Y), rem = k % (S1X * S1Y);
        sz = plane < RZ ? plane : plane + BZ;
        sy = rem / S1X;
        sx = rem % S1X;
    } else if (k < NZS + NYS) {
        const int q = k - NZS, row = q / S1X;
        const int yy = row % (2 * RY);
        sz = RZ + row / (2 * RY);
        sy = yy < RY ? yy : yy + BY;
        sx = q % S1X;
    } else {
        const int q = k - NZS - NYS, col = q % (2 * RX), row = q / (2 * RX);
        sy = RY + row % BY;
        sz = RZ + row / BY;
        sx = col < RX ? col : col + BX;
    }
}

// What an own site carries from stage 1 to stage 2: Heun's D1 and the Langevin
// torque on m0; SIB's and Depondt's m0, thermal field and (Depondt) b1
template <int MODE>
struct FusedKeep {
    v3 p, q, r;
};

// field of the neighbour sum s
__device__ __forceinline__ v3 fused_field(v3 s, v3 z) { return mk3(-(s.x + z.x), -(s.y + z.y), -(s.z + z.z)); }

// stage 1 at a site with state m0 and neighbour sum s: the stage's result, the
// energy term of m0, what stage 2 needs of it (th: the site's thermal field)
template <int MODE, bool NOISE, class F>
__device__ __forceinline__ v3 fused_stage1(const KArgs &a, v3 m0, v3 s, int64_t gi, v3 th, FusedKeep<MODE> &k, double &e)
{
    const v3 z = fused_zeeman<F>(a, true, gi);
    v3 B = fused_field(s, z);
    e = mj_site_energy(m0, s, z);
    if constexpr (MODE == MODE_HEUNF) {
        const MjUnit u = mj_unit(m0);
        k.p = llg_torque(u.n, B, a.alpha);
        // Langevin term of the last stage on m0 (HEUN2: thermal_term)
        if constexpr (NOISE) k.q = llg_torque(u.n, th, a.alpha);
        return euler_step0(m0, u, k.p, a.kdt);   // Dint = 1 D1
    }
    if constexpr (NOISE) B = mk3(B.x + th.x, B.y + th.y, B.z + th.z);
    k.p = m0;
    k.q = th;
    if constexpr (MODE == MODE_DEPF) {
        k.r = dep_field(m0, B, a.alpha);
        return dep_rotate(m0, k.r, a.kdt);
    }
    return cayley_mid(m0, sib_vec(m0, B, a.alpha, -0.5 * a.kdt));
}

// stage 2 at an own site from the stage-1 state m and its neighbour sum s
template <int MODE, bool NOISE, class F>
__device__ __forceinline__ void fused_stage2(const KArgs &a, v3 m, v3 s, int64_t gi, const FusedKeep<MODE> &k)
{
    const int64_t np = a.np;
    v3 B = fused_field(s, fused_zeeman<F>(a, true, gi));
    if (a.fld_out) {   // the last stage's field, kept for the host
        a.fld_out[gi] = B.x;
        a.fld_out[gi + np] = B.y;
        a.fld_out[gi + 2 * np] = B.z;
    }
    v3 o;
    if constexpr (MODE == MODE_HEUNF) {
        const MjUnit u = mj_unit(m);
        const v3 d = k.p + llg_torque(u.n, B, a.alpha);   // Dint = D1/2 + D2/2
        if constexpr (NOISE) o = euler_step(m, u, d, 0.5 * a.kdt, k.q, a.kdt);
        else o = euler_step0(m, u, d, 0.5 * a.kdt);
    } else {
        if constexpr (NOISE) B = mk3(B.x + k.q.x, B.y + k.q.y, B.z + k.q.z);
        if constexpr (MODE == MODE_DEPF) {
            const v3 b2 = dep_field(m, B, a.alpha);
            o = dep_rotate(k.p, mk3(0.5 * (k.r.x + b2.x), 0.5 * (k.r.y + b2.y), 0.5 * (k.r.z + b2.z)), a.kdt);
        } else {
            o = cayley(k.p, sib_vec(m, B, a.alpha, -0.5 * a.kdt));
        }
    }
    a.dst[gi] = o.x;
    a.dst[gi + np] = o.y;
    a.dst[gi + 2 * np] = o.z;
}

// the neighbour sums of a thread's sites (one, or two one above the other)
// centred at c in LDS: REG 0 the S0 layout, 1 the S1 layout
template <int REG, class F>
__device__ __forceinline__ void fused_sums(const KArgs &a, const double *L, int c, v3 s[F::kSpt])
{
#pragma unroll
    for (int j = 0; j < F::kSpt; ++j) s[j] = mk3(0.0, 0.0, 0.0);
    if constexpr (F::kSpt == 2) {
        if constexpr (REG == 0) F::pair0(a, L, c, s[0].x, s[0].y, s[0].z, s[1].x, s[1].y, s[1].z);
        else F::pair1(a, L, c, s[0].x, s[0].y, s[0].z, s[1].x, s[1].y, s[1].z);
        mj_settle(s[1].x, s[1].y, s[1].z);
    } else {
        if constexpr (REG == 0) F::stencil0(a, L, c, s[0].x, s[0].y, s[0].z);
        else F::stencil1(a, L, c, s[0].x, s[0].y, s[0].z);
    }
    mj_settle(s[0].x, s[0].y, s[0].z);
}

template <bool NOISE>
__device__ __forceinline__ v3 fused_thermal(const KArgs &a, uint64_t nstep, int64_t gi)
{
    if constexpr (NOISE) {
        const v3 g = normals3(a.seed, nstep, (uint32_t)gi);
        return mk3(a.sigma * g.x, a.sigma * g.y, a.sigma * g.z);
    }
    return mk3(0.0, 0.0, 0.0);
}

template <int MODE, bool NOISE, class F>
__device__ __forceinline__ void fused_body(const KArgs &a, double *lds)
{
    constexpr int BX = F::kBx, BY = F::kBy, BZ = F::kBz, RX = F::kRx, RY = F::kRy, RZ = F::kRz;
    constexpr int SPT = F::kSpt, NTHR = F::kNthr, NB = F::kNthrBase, NBW = NB / 64;
    constexpr int BYT = BY / SPT;                 // rows of threads
    constexpr int S0X = F::kS0x, S0Y = F::kS0y, T0 = F::kT0;
    constexpr int S1X = BX + 2 * RX, S1Y = BY + 2 * RY, S1Z = BZ + 2 * RZ, T1 = S1X * S1Y * S1Z;
    constexpr int NRING = T1 - BX * BY * BZ;
    // threads of the ring's own (after those of the tile), or the tile's threads
    constexpr int WIDE = F::kWide, RTHR = WIDE ? WIDE : NTHR;
    constexpr int NRT = (NRING + RTHR - 1) / RTHR;   // ring sites per thread
    constexpr bool ALIAS = F::kAlias;                // S1 in S0's place
    static_assert(NB % 64 == 0 && NTHR * SPT == BX * BY * BZ, "whole wavefronts, every tile site once");
    static_assert(SPT == 1 || (SPT == 2 && BX == 32 && BZ == 1 && BYT % F::kNsub == 0 && NTHR >= NB),
                  "a pair's rows are one wavefront of the two-kernel path");
    double *L0 = lds;                                  // S0: 3 x T0
    double *L1 = ALIAS ? lds : lds + 3 * T0;           // S1: 3 x T1
    double *red = lds + 3 * T0 + (ALIAS ? 0 : 3 * T1);   // per-wave sums (BX BY BZ / 64)

    const int bid = F::block(a);
    const int tx = bid % F::ntx(a), tr = bid / F::ntx(a), ty = tr % F::nty(a), tz = tr / F::nty(a);
    const int x0 = tx * BX, y0 = ty * BY, z0 = tz * BZ;
    uint64_t nstep = 0;
    if constexpr (NOISE) nstep = a.stepp ? *a.stepp + a.step : a.step;
    const bool direct = F::dma(a) && (((unsigned long long)a.src) & 15ull) == 0 && x0 - 2 * RX >= 0 &&
                        x0 + BX + 2 * RX <= F::nx(a) && y0 - 2 * RY >= 0 && y0 + BY + 2 * RY <= F::ny(a) &&
                        z0 - 2 * RZ >= 0 && z0 + BZ + 2 * RZ <= F::nz(a);
    v3 fill[F::kFill];
    fused_s0_fill<F>(a, L0, x0, y0, z0, direct, fill);

    // S1 inside the lattice: every site of it is one of the lattice's
    const bool inside = x0 - RX >= 0 && x0 + BX + RX <= F::nx(a) && y0 - RY >= 0 && y0 + BY + RY <= F::ny(a) &&
                        z0 - RZ >= 0 && z0 + BZ + RZ <= F::nz(a);
    // index of the site at lattice coordinates (x, y, z): wrapped on periodic
    // axes, 0 off an open edge.  Stage 1 runs there all the same: S0 is zero
    // around an open edge, and a zero spin stays zero in every stage.
    auto index = [&](int x, int y, int z) -> int64_t {
        if (inside) return (int64_t)x + (int64_t)F::nx(a) * ((int64_t)y + (int64_t)F::ny(a) * z);
        int64_t g = 0;
        return fused_site<F>(a, x, y, z, g) ? g : 0;
    };

    const bool own = WIDE == 0 || (int)threadIdx.x < NTHR;   // whole wavefronts
    const int rid = WIDE == 0 ? (int)threadIdx.x : own ? NRING : (int)threadIdx.x - NTHR;
    // the thread's own sites (rows SPT ly + j); active: inside the lattice
    const int lx = threadIdx.x % BX, ly = (threadIdx.x / BX) % BYT * SPT, lz = threadIdx.x / (BX * BYT);
    const int gx = x0 + lx, gz = z0 + lz;
    bool active[SPT];
    int64_t gi[SPT];
    v3 th[SPT];
#pragma unroll
    for (int j = 0; j < SPT; ++j) {
        active[j] = false;
        gi[j] = 0;
        if (!own) continue;
        const int gy = y0 + ly + j;
        active[j] = inside || (gx < F::nx(a) && gy < F::ny(a) && gz < F::nz(a));
        gi[j] = index(gx, gy, gz);
        // the Philox thermal field while the tile lands, one site after the other
        th[j] = fused_thermal<NOISE>(a, nstep, gi[j]);
        if constexpr (NOISE) mj_settle(th[j].x, th[j].y, th[j].z);
        __builtin_amdgcn_sched_barrier(0);
    }
    if (direct) __builtin_amdgcn_s_waitcnt(0);
    else fused_s0_store<F>(L0, fill);
    __syncthreads();

    // stage 1 on the ring of S1, before the own sites: they have more to keep
    // (kept apart in the schedule: overlapping the two doubles the live registers)
    auto ring = [&](int k, int &c1) -> v3 {
        int sx, sy, sz;
        fused_ring_pos<F>(k, sx, sy, sz);
        c1 = sz * S1X * S1Y + sy * S1X + sx;
        const int c0 = (sz + RZ) * S0X * S0Y + (sy + RY) * S0X + (sx + RX);
        const int64_t gw = index(x0 - RX + sx, y0 - RY + sy, z0 - RZ + sz);
        v3 bt = mk3(0.0, 0.0, 0.0);
        if constexpr (MODE != MODE_HEUNF) bt = fused_thermal<NOISE>(a, nstep, gw);
        v3 s = mk3(0.0, 0.0, 0.0);
        F::stencil0(a, L0, c0, s.x, s.y, s.z);
        mj_settle(s.x, s.y, s.z);
        FusedKeep<MODE> drop;
        double ee;
        const v3 m = fused_stage1<MODE, NOISE && MODE != MODE_HEUNF, F>(
            a, mk3(L0[c0], L0[T0 + c0], L0[2 * T0 + c0]), s, gw, bt, drop, ee);
        return m;
    };
    v3 mr[ALIAS && NRT > 0 ? NRT : 1];
    int cr[ALIAS && NRT > 0 ? NRT : 1];
    if constexpr (ALIAS) {
#pragma unroll
        for (int r = 0; r < NRT; ++r) {
            const int k = rid + r * RTHR;
            cr[r] = -1;
            if (k < NRING) mr[r] = ring(k, cr[r]);
        }
    } else {
        for (int k = rid; k < NRING; k += RTHR) {
            int c1;
            const v3 m = ring(k, c1);
            L1[c1] = m.x;
            L1[T1 + c1] = m.y;
            L1[2 * T1 + c1] = m.z;
        }
    }
    __builtin_amdgcn_sched_barrier(0);

    // stage 1 at the own positions
    FusedKeep<MODE> keep[SPT];
    v3 m1[SPT];
    double e = 0.0;
    if (own) {
        const int c0 = (lz + 2 * RZ) * S0X * S0Y + (ly + 2 * RY) * S0X + (lx + 2 * RX);
        v3 s[SPT];
        fused_sums<0, F>(a, L0, c0, s);
#pragma unroll
        for (int j = 0; j < SPT; ++j) {
            const int c = c0 + j * S0X;
            const v3 m0 = mk3(L0[c], L0[T0 + c], L0[2 * T0 + c]);
            double ej;
            m1[j] = fused_stage1<MODE, NOISE, F>(a, m0, s[j], gi[j], th[j], keep[j], ej);
            if (!active[j]) ej = 0.0;
            e = j == 0 ? ej : e + ej;
            __builtin_amdgcn_sched_barrier(0);
        }
    }
    // energy partials of m0 (mj_block_reduce's order: wavefronts in lane order,
    // then in wave order); red[q]: wavefront q of the two-kernel path's tiles
    if (F::kEnergy && a.energy) {
        constexpr int W = 64 / SPT;
        double v = e;
#pragma unroll
        for (int o = W / 2; o > 0; o >>= 1) v = v + __shfl_xor(v, o, 64);
        if (own && threadIdx.x % W == 0) red[threadIdx.x / W] = v;
    }
    const int s1 = (lz + RZ) * S1X * S1Y + (ly + RY) * S1X + (lx + RX);
    if constexpr (ALIAS) {
        __syncthreads();   // S0 is done with
#pragma unroll
        for (int r = 0; r < NRT; ++r) {
            if (cr[r] >= 0) {
                L1[cr[r]] = mr[r].x;
                L1[T1 + cr[r]] = mr[r].y;
                L1[2 * T1 + cr[r]] = mr[r].z;
            }
        }
    }
#pragma unroll
    for (int j = 0; j < SPT; ++j) {
        if (!own) continue;
        const int c = s1 + j * S1X;
        L1[c] = m1[j].x;
        L1[T1 + c] = m1[j].y;
        L1[2 * T1 + c] = m1[j].z;
    }
    __syncthreads();
    // tile h of the two-kernel path (tx, ty * NSUB + h, tz): its wavefronts'
    // sums are red[h NBW ...]; one thread per tile adds them in order
    if (F::kEnergy && a.energy && (int)threadIdx.x < F::kNsub) {
        const int h = threadIdx.x, sub_ty = ty * F::kNsub + h;
        if (sub_ty < F::nty_base(a)) {
            double r = red[h * NBW];
            for (int w = 1; w < NBW; ++w) r = r + red[h * NBW + w];
            a.epart[tx + F::ntx(a) * (sub_ty + F::nty_base(a) * tz)] = r;
        }
    }

    // stage 2 at the own sites from S1
    __builtin_amdgcn_sched_barrier(0);
    if (own) {
        v3 s[SPT];
        fused_sums<1, F>(a, L1, s1, s);
#pragma unroll
        for (int j = 0; j < SPT; ++j) {
            if (active[j]) {
                const int c = s1 + j * S1X;
                fused_stage2<MODE, NOISE, F>(a, mk3(L1[c], L1[T1 + c], L1[2 * T1 + c]), s[j], gi[j], keep[j]);
            }
            __builtin_amdgcn_sched_barrier(0);
        }
    }

    // workgroup 0 folds the previous launch's partials (the energy of the state
    // entering the previous step) as the stage-2 kernel's block 0 folds them:
    // strided sums over its first NB threads, then their wavefronts in order
    if (F::kEnergy && a.ered_in && blockIdx.x == 0) {
        __syncthreads();
        double v = 0.0;
        if (threadIdx.x < NB)
            for (int i = threadIdx.x; i < a.n_ered; i += NB) v += a.ered_in[i];
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) v = v + __shfl_xor(v, o, 64);
        if ((threadIdx.x & 63) == 0 && threadIdx.x < NB) red[threadIdx.x >> 6] = v;
        __syncthreads();
        if (threadIdx.x == 0) {
            double r = red[0];
            for (int w = 1; w < NBW; ++w) r = r + red[w];
            *a.e_out = r * a.e_scale;
        }
    }
}
