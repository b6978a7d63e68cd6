// Device code of the differentiable SIB trajectory, shared by the
// ahead-of-time kernels (mj_adjoint.hip) and those compiled per parameter set
// (mj_jit.hip).  A geometry G gives the lattice, tile and stencils: from the
// arguments (AdjRt) or as constants.
#pragma once

struct AdjArgs {
    int nx, ny, nz, px, py, pz, bx, by, bz, rx, ry, rz, ntx, nty, nblocks;
    int64_t np;
    int nofs;
    const int *ofs;     // LDS offsets of the total stencil
    const int *ofs0;    // the same in the fused step's S0 layout (tile + 2 reach)
    const double *cf;   // 9 per offset (row-major C_d)
    const double *cls;  // compiled kernels: the stencil's distinct values
    int nparam;
    const int *pstart;  // unit stencils: entries [pstart[k], pstart[k+1]) of pofs/pcf
    const int *pofs;
    const double *pcf;
    double z[9];
    const double *bmap; // b_i (SoA)
    double alpha, f;
    // state
    const double *x;    // stencil state of the kernel (SoA)
    const double *x2;   // second stencil state (fused R3 + R1: the midpoint of the earlier step)
    const double *m;    // own-site state m_n
    const double *m1;   // own-site state m_{n+1}
    const double *gin;  // own-site input gradient
    const double *gacc_in, *gpd_in;
    double *out0, *out1, *out2;
    double *ghmap;
    double *ppart;      // [nblocks][nparam + 3]
};

constexpr int kAdjMaxParam = 13;

__device__ __forceinline__ v3 v_add(v3 a, v3 b) { return mk3(a.x + b.x, a.y + b.y, a.z + b.z); }
__device__ __forceinline__ v3 v_scale(double s, v3 a) { return mk3(s * a.x, s * a.y, s * a.z); }

// (I - [a]x + a a^T)^T ... M(-a) g = (g + a x g + (a.g) a) / (1 + |a|^2)
__device__ __forceinline__ v3 minv_t(v3 a, v3 g)
{
    const v3 w = fma3(dot3(a, g), a, cross3_add(a, g, g));
    return v_scale(mj_rcp(fma(a.z, a.z, fma(a.y, a.y, fma(a.x, a.x, 1.0)))), w);
}

__device__ __forceinline__ v3 apply_blocks(const double *L, int T, int c, int n, const int *ofs, const double *cf)
{
    double ax = 0.0, ay = 0.0, az = 0.0;
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
    return mk3(ax, ay, az);
}

// geometry from the arguments
struct AdjRt {
    static constexpr bool kConst = false;
    static constexpr int kTrips = 1, kTrips0 = 1, kMaxVals = kAdjMaxParam + 3;
#define MJ_ADJ_ARG(n) \
    static __device__ __forceinline__ int n(const AdjArgs &a) { return a.n; }
    MJ_ADJ_ARG(nx) MJ_ADJ_ARG(ny) MJ_ADJ_ARG(nz) MJ_ADJ_ARG(bx) MJ_ADJ_ARG(by) MJ_ADJ_ARG(bz) MJ_ADJ_ARG(rx)
    MJ_ADJ_ARG(ry) MJ_ADJ_ARG(rz) MJ_ADJ_ARG(ntx) MJ_ADJ_ARG(nty) MJ_ADJ_ARG(nparam)
#undef MJ_ADJ_ARG
    static __device__ __forceinline__ v3 sum(const AdjArgs &a, const double *L, int T, int c)
    {
        return apply_blocks(L, T, c, a.nofs, a.ofs, a.cf);
    }
    static __device__ __forceinline__ v3 sum0(const AdjArgs &a, const double *L, int T, int c)
    {
        return apply_blocks(L, T, c, a.nofs, a.ofs0, a.cf);
    }
    // vals[k] = -gB . (C^(k) x) of the parameters' unit stencils
    static __device__ __forceinline__ void units(const AdjArgs &a, const double *L, int T, int c, v3 gB, double *vals)
    {
        for (int k = 0; k < a.nparam; ++k)
            vals[k] = -dot3(gB, apply_blocks(L, T, c, a.pstart[k + 1] - a.pstart[k], a.pofs + a.pstart[k],
                                             a.pcf + 9 * a.pstart[k]));
    }
};

// lattice site of a region position (wrapped on periodic axes; false off an open edge)
template <class G>
__device__ __forceinline__ bool adj_site_of(const AdjArgs &a, int gx, int gy, int gz, int64_t &g)
{
    const bool in = fused_wrap(gx, G::nx(a), G::bx(a), G::rx(a), a.px) & fused_wrap(gy, G::ny(a), G::by(a), G::ry(a), a.py) &
                    fused_wrap(gz, G::nz(a), G::bz(a), G::rz(a), a.pz);
    g = (int64_t)gx + (int64_t)G::nx(a) * ((int64_t)gy + (int64_t)G::ny(a) * gz);
    return in;
}

// the tile at (x0, y0, z0) of src with a halo of H (1 or 2) times the reach
template <class G, int H>
struct AdjTile {
    v3 v[H == 1 ? G::kTrips : G::kTrips0];
    int s0, s1, T;

    static __device__ __forceinline__ v3 get(const AdjArgs &a, const double *src, int t, int s0, int s1, int x0, int y0,
                                             int z0)
    {
        const int lx = t % s0, r = t / s0, ly = r % s1, lz = r / s1;
        int64_t g = 0;
        const bool in = adj_site_of<G>(a, x0 + lx - H * G::rx(a), y0 + ly - H * G::ry(a), z0 + lz - H * G::rz(a), g);
        const double *p = src + (in ? g : 0);
        const double vx = p[0], vy = p[a.np], vz = p[2 * a.np];
        return in ? mk3(vx, vy, vz) : mk3(0.0, 0.0, 0.0);
    }
    // constants: every load in flight before the first store; else straight to LDS
    __device__ __forceinline__ void load(const AdjArgs &a, const double *src, double *L, int x0, int y0, int z0)
    {
        const int nthr = G::bx(a) * G::by(a) * G::bz(a);
        s0 = G::bx(a) + 2 * H * G::rx(a);
        s1 = G::by(a) + 2 * H * G::ry(a);
        T = s0 * s1 * (G::bz(a) + 2 * H * G::rz(a));
        if constexpr (G::kConst) {
#pragma unroll
            for (int k = 0; k < (H == 1 ? G::kTrips : G::kTrips0); ++k)
                v[k] = get(a, src, min((int)threadIdx.x + k * nthr, T - 1), s0, s1, x0, y0, z0);
        } else {
            for (int t = threadIdx.x; t < T; t += nthr) put(L, t, get(a, src, t, s0, s1, x0, y0, z0));
        }
    }
    __device__ __forceinline__ void put(double *L, int t, v3 w) const
    {
        L[t] = w.x;
        L[T + t] = w.y;
        L[2 * T + t] = w.z;
    }
    __device__ __forceinline__ void store(const AdjArgs &a, double *L) const
    {
        if constexpr (G::kConst) {
            const int nthr = G::bx(a) * G::by(a) * G::bz(a);
#pragma unroll
            for (int k = 0; k < (H == 1 ? G::kTrips : G::kTrips0); ++k)
                if ((int)threadIdx.x + k * nthr < T) put(L, (int)threadIdx.x + k * nthr, v[k]);
        }
    }
};

struct Site {
    int x0, y0, z0, lx, ly, lz, c, T;
    bool active;
    int64_t gi;
};

template <class G>
__device__ __forceinline__ Site adj_site(const AdjArgs &a)
{
    Site s;
    const int bx = G::bx(a), by = G::by(a), bz = G::bz(a), sx = bx + 2 * G::rx(a), sy = by + 2 * G::ry(a);
    const int bid = blockIdx.x;
    const int tx = bid % G::ntx(a), tr = bid / G::ntx(a), ty = tr % G::nty(a), tz = tr / G::nty(a);
    s.x0 = tx * bx;
    s.y0 = ty * by;
    s.z0 = tz * bz;
    s.lx = threadIdx.x % bx;
    s.ly = (threadIdx.x / bx) % by;
    s.lz = threadIdx.x / (bx * by);
    const int gx = s.x0 + s.lx, gy = s.y0 + s.ly, gz = s.z0 + s.lz;
    s.active = gx < G::nx(a) && gy < G::ny(a) && gz < G::nz(a);
    s.gi = s.active ? (int64_t)gx + (int64_t)G::nx(a) * ((int64_t)gy + (int64_t)G::ny(a) * gz) : 0;
    s.c = (s.lz + G::rz(a)) * sx * sy + (s.ly + G::ry(a)) * sx + (s.lx + G::rx(a));
    s.T = sx * sy * (bz + 2 * G::rz(a));
    return s;
}

__device__ __forceinline__ v3 ld3(const double *p, int64_t i, int64_t np) { return mk3(p[i], p[i + np], p[i + 2 * np]); }
__device__ __forceinline__ void st3(double *p, int64_t i, int64_t np, v3 v)
{
    p[i] = v.x;
    p[i + np] = v.y;
    p[i + 2 * np] = v.z;
}

__device__ __forceinline__ v3 zeeman_t(const AdjArgs &a, v3 b)   // Z^T b_i
{
    return mk3((b.x * a.z[0] + b.y * a.z[3]) + b.z * a.z[6], (b.x * a.z[1] + b.y * a.z[4]) + b.z * a.z[7],
               (b.x * a.z[2] + b.y * a.z[5]) + b.z * a.z[8]);
}

__device__ __forceinline__ v3 zeeman_vjp(const AdjArgs &a, v3 g)   // -Z g
{
    return mk3(-((a.z[0] * g.x + a.z[1] * g.y) + a.z[2] * g.z), -((a.z[3] * g.x + a.z[4] * g.y) + a.z[5] * g.z),
               -((a.z[6] * g.x + a.z[7] * g.y) + a.z[8] * g.z));
}

// SIB's vector a(x) = f (B + alpha x x B) of a spin with neighbour sum acc and
// field term b, B and x x B kept
struct SibVec {
    v3 B, av;
};
__device__ __forceinline__ SibVec adj_vec(const AdjArgs &a, v3 x, v3 acc, v3 b)
{
    SibVec r;
    const v3 zb = zeeman_t(a, b);
    r.B = mk3(-(acc.x + zb.x), -(acc.y + zb.y), -(acc.z + zb.z));
    r.av = v_scale(a.f, fma3(a.alpha, cross3(x, r.B), r.B));
    return r;
}

// the block's running sums, read at the kernel's start (thread q: value q)
__device__ __forceinline__ double adj_part(const AdjArgs &a, int nv)
{
    return (int)threadIdx.x < nv ? a.ppart[(size_t)blockIdx.x * nv + threadIdx.x] : 0.0;
}

// per-block deterministic sums of nparam + 3 values, accumulated into
// ppart[block][*]: every value's wavefront butterflies, one barrier, then
// thread q adds value q's wave sums in wave order (mj_block_sum's order for
// each value, without a barrier pair per value)
template <class G>
__device__ __forceinline__ void adj_reduce(const AdjArgs &a, double *red, const double *vals, double part)
{
    const int nv = G::nparam(a) + 3, nthr = G::bx(a) * G::by(a) * G::bz(a);
    __syncthreads();
    if ((nthr & 63) != 0) {
        for (int q = 0; q < nv; ++q) {
            const double t = mj_block_sum(vals[q], red, nthr);
            if (threadIdx.x == 0) a.ppart[(size_t)blockIdx.x * nv + q] += t;
        }
        return;
    }
    const int nw = nthr >> 6;
    if constexpr (G::kConst) {   // the values' butterflies side by side
        double w[G::kMaxVals];
#pragma unroll
        for (int q = 0; q < G::kMaxVals; ++q) w[q] = vals[q];
#pragma unroll
        for (int o = 32; o > 0; o >>= 1)
#pragma unroll
            for (int q = 0; q < G::kMaxVals; ++q) w[q] = w[q] + __shfl_xor(w[q], o, 64);
#pragma unroll
        for (int q = 0; q < G::kMaxVals; ++q)
            if ((threadIdx.x & 63) == 0) red[q * nw + (threadIdx.x >> 6)] = w[q];
    } else {
        for (int q = 0; q < nv; ++q) {
            double v = vals[q];
#pragma unroll
            for (int o = 32; o > 0; o >>= 1) v = v + __shfl_xor(v, o, 64);
            if ((threadIdx.x & 63) == 0) red[q * nw + (threadIdx.x >> 6)] = v;
        }
    }
    __syncthreads();
    if ((int)threadIdx.x < nv) {
        const int q = threadIdx.x;
        double r = red[q * nw];
        for (int k = 1; k < nw; ++k) r = r + red[q * nw + k];
        a.ppart[(size_t)blockIdx.x * nv + q] = part + r;
    }
}

// forward stage 1: p = (m + cay(m, a1(m)))/2
template <class G>
__device__ __forceinline__ void adj_sib1_body(const AdjArgs &a, double *L)
{
    const Site s = adj_site<G>(a);
    AdjTile<G, 1> t;
    t.load(a, a.x, L, s.x0, s.y0, s.z0);
    const v3 b = ld3(a.bmap, s.gi, a.np);
    t.store(a, L);
    __syncthreads();
    if (!s.active) return;
    const v3 m = mk3(L[s.c], L[s.T + s.c], L[2 * s.T + s.c]);
    st3(a.out0, s.gi, a.np, cayley_mid(m, adj_vec(a, m, G::sum(a, L, s.T, s.c), b).av));
}

// forward stage 2: m' = cay(m, a2(p))
template <class G>
__device__ __forceinline__ void adj_sib2_body(const AdjArgs &a, double *L)
{
    const Site s = adj_site<G>(a);
    AdjTile<G, 1> t;
    t.load(a, a.x, L, s.x0, s.y0, s.z0);
    const v3 b = ld3(a.bmap, s.gi, a.np), m = ld3(a.m, s.gi, a.np);
    t.store(a, L);
    __syncthreads();
    if (!s.active) return;
    const v3 p = mk3(L[s.c], L[s.T + s.c], L[2 * s.T + s.c]);
    st3(a.out0, s.gi, a.np, cayley(m, adj_vec(a, p, G::sum(a, L, s.T, s.c), b).av));
}

// the midpoint p of SIB's first stage at one site from the S0 tile
template <class G>
__device__ __forceinline__ v3 adj_midpoint(const AdjArgs &a, const double *L0, int T0, int c0, int64_t gi, v3 &m)
{
    const v3 b = ld3(a.bmap, gi, a.np);
    m = mk3(L0[c0], L0[T0 + c0], L0[2 * T0 + c0]);
    return cayley_mid(m, adj_vec(a, m, G::sum0(a, L0, T0, c0), b).av);
}

// a whole forward step in one kernel: the tile plus twice the reach (S0) in
// LDS, the midpoint on the tile plus the reach (S1: the tile's own sites and
// a ring repeating the neighbouring tiles' first stage with the same
// operations), the second stage on the tile.  out0 = the midpoint p (kept for
// the reverse sweep), out1 = m'; bit for bit k_adj_sib1 then k_adj_sib2.
template <class G>
__device__ __forceinline__ void adj_sibf_body(const AdjArgs &a, double *L)
{
    const int bx = G::bx(a), by = G::by(a), bz = G::bz(a), rx = G::rx(a), ry = G::ry(a), rz = G::rz(a);
    const int sx_ = bx + 2 * rx, sy_ = by + 2 * ry;
    const int s0x = bx + 4 * rx, s0y = by + 4 * ry, s0z = bz + 4 * rz, T0 = s0x * s0y * s0z;
    const int nthr = bx * by * bz;
    double *L0 = L;
    double *L1 = L + 3 * T0;
    const Site s = adj_site<G>(a);
    const int T1 = s.T;
    AdjTile<G, 2> t;
    t.load(a, a.x, L0, s.x0, s.y0, s.z0);
    const v3 b = ld3(a.bmap, s.gi, a.np);
    t.store(a, L0);
    __syncthreads();
    v3 m0 = mk3(0.0, 0.0, 0.0);
    {
        int64_t gw = 0;
        v3 p = mk3(0.0, 0.0, 0.0);
        if (adj_site_of<G>(a, s.x0 + s.lx, s.y0 + s.ly, s.z0 + s.lz, gw)) {
            const int c0 = (s.lz + 2 * rz) * s0x * s0y + (s.ly + 2 * ry) * s0x + (s.lx + 2 * rx);
            p = adj_midpoint<G>(a, L0, T0, c0, gw, m0);
        }
        L1[s.c] = p.x;
        L1[T1 + s.c] = p.y;
        L1[2 * T1 + s.c] = p.z;
    }
    // the ring of S1: z slabs, then y slabs of the tile's planes, then x slabs of its rows
    const int nzs = 2 * rz * sx_ * sy_, nys = 2 * ry * bz * sx_;
    for (int k = threadIdx.x; k < T1 - nthr; k += nthr) {
        int sx, sy, sz;
        if (k < nzs) {
            const int plane = k / (sx_ * sy_), rem = k % (sx_ * sy_);
            sz = plane < rz ? plane : plane + bz;
            sy = rem / sx_;
            sx = rem % sx_;
        } else if (k < nzs + nys) {
            const int q = k - nzs, row = q / sx_, yy = row % (2 * ry);
            sz = rz + row / (2 * ry);
            sy = yy < ry ? yy : yy + by;
            sx = q % sx_;
        } else {
            const int q = k - nzs - nys, col = q % (2 * rx), row = q / (2 * rx);
            sy = ry + row % by;
            sz = rz + row / by;
            sx = col < rx ? col : col + bx;
        }
        const int c1 = sz * sx_ * sy_ + sy * sx_ + sx;
        int64_t gw = 0;
        v3 p = mk3(0.0, 0.0, 0.0);
        if (adj_site_of<G>(a, s.x0 - rx + sx, s.y0 - ry + sy, s.z0 - rz + sz, gw)) {
            const int c0 = (sz + rz) * s0x * s0y + (sy + ry) * s0x + (sx + rx);
            v3 mm;
            p = adj_midpoint<G>(a, L0, T0, c0, gw, mm);
        }
        L1[c1] = p.x;
        L1[T1 + c1] = p.y;
        L1[2 * T1 + c1] = p.z;
    }
    __syncthreads();
    if (!s.active) return;
    const v3 p = mk3(L1[s.c], L1[T1 + s.c], L1[2 * T1 + s.c]);
    const SibVec v = adj_vec(a, p, G::sum(a, L1, T1, s.c), b);
    st3(a.out0, s.gi, a.np, p);
    st3(a.out1, s.gi, a.np, cayley(m0, v.av));
}

// own-site operands of R1, loaded ahead of the tiles' barrier
struct R1Own {
    v3 b, m, m1, g, gh;
};
__device__ __forceinline__ R1Own r1_own(const AdjArgs &a, const Site &s, const double *g)
{
    return {ld3(a.bmap, s.gi, a.np), ld3(a.m, s.gi, a.np), ld3(a.m1, s.gi, a.np), ld3(g, s.gi, a.np),
            ld3(a.ghmap, s.gi, a.np)};
}

// R1: reverse of the stage-2 site math: the midpoint tile p is in L, own.g =
// dL/dm' at the own site.  out0 = gB2, out1 = gacc (cay(g', -a2)), out2 = gp_direct
template <class G>
__device__ __forceinline__ void r1_site(const AdjArgs &a, const double *L, const Site &s, const R1Own &o, double *vals)
{
    const int T = s.T;
    const v3 p = mk3(L[s.c], L[T + s.c], L[2 * T + s.c]);
    const SibVec v = adj_vec(a, p, G::sum(a, L, T, s.c), o.b);
    const v3 gm = cayley(o.g, mk3(-v.av.x, -v.av.y, -v.av.z));
    const v3 w = minv_t(v.av, o.g);
    const v3 ga = cross3(w, v_add(o.m1, o.m));
    const v3 gB = v_scale(a.f, v_add(ga, v_scale(a.alpha, cross3(ga, p))));
    const v3 gp = v_scale(a.f * a.alpha, cross3(v.B, ga));
    st3(a.out0, s.gi, a.np, gB);
    st3(a.out1, s.gi, a.np, gm);
    st3(a.out2, s.gi, a.np, gp);
    G::units(a, L, T, s.c, gB, vals);
    const v3 gb = zeeman_vjp(a, gB);
    vals[G::nparam(a)] = gb.x;
    vals[G::nparam(a) + 1] = gb.y;
    vals[G::nparam(a) + 2] = gb.z;
    st3(a.ghmap, s.gi, a.np, v_add(o.gh, gb));
}

template <class G>
__device__ __forceinline__ void adj_r1_body(const AdjArgs &a, double *L)
{
    const Site s = adj_site<G>(a);
    double *red = L + 3 * s.T;
    AdjTile<G, 1> t;
    t.load(a, a.x, L, s.x0, s.y0, s.z0);
    const R1Own o = r1_own(a, s, a.gin);
    const double part = adj_part(a, G::nparam(a) + 3);
    t.store(a, L);
    __syncthreads();
    double vals[G::kMaxVals];
    for (int q = 0; q < G::kMaxVals; ++q) vals[q] = 0.0;
    if (s.active) r1_site<G>(a, L, s, o, vals);
    adj_reduce<G>(a, red, vals, part);
}

// R3 of step q fused with R1 of step q-1: lambda_q = gacc - C * gB1 at the own
// site (tile of gB1 in x), then the stage-2 reverse of step q-1 with
// g = lambda_q (tile of its midpoint in x2); lambda_q never goes to memory
template <class G>
__device__ __forceinline__ void adj_r3r1_body(const AdjArgs &a, double *L)
{
    const Site s = adj_site<G>(a);
    double *LP = L + 3 * s.T;
    double *red = L + 6 * s.T;
    AdjTile<G, 1> t, tp;
    t.load(a, a.x, L, s.x0, s.y0, s.z0);
    tp.load(a, a.x2, LP, s.x0, s.y0, s.z0);
    R1Own o = r1_own(a, s, a.gacc_in);
    const double part = adj_part(a, G::nparam(a) + 3);
    t.store(a, L);
    tp.store(a, LP);
    __syncthreads();
    double vals[G::kMaxVals];
    for (int q = 0; q < G::kMaxVals; ++q) vals[q] = 0.0;
    if (s.active) {
        const v3 c = G::sum(a, L, s.T, s.c);
        o.g = mk3(o.g.x - c.x, o.g.y - c.y, o.g.z - c.z);
        r1_site<G>(a, LP, s, o, vals);
    }
    adj_reduce<G>(a, red, vals, part);
}

// R2: transpose of the stage-2 field (stencil over gB2 in x) + reverse of the
// stage-1 site math (needs the stencil of m: second tile).
// gin = gB2 is x; m stencil read from a.m; gacc_in, gpd_in own.
// out0 = gB1, out1 = gacc2
template <class G>
__device__ __forceinline__ void adj_r2_body(const AdjArgs &a, double *L)
{
    const Site s = adj_site<G>(a);
    const int T = s.T;
    double *LM = L + 3 * T;
    double *red = L + 6 * T;
    AdjTile<G, 1> t, tm;
    t.load(a, a.x, L, s.x0, s.y0, s.z0);
    tm.load(a, a.m, LM, s.x0, s.y0, s.z0);
    const v3 b = ld3(a.bmap, s.gi, a.np), gacc = ld3(a.gacc_in, s.gi, a.np), gpd = ld3(a.gpd_in, s.gi, a.np);
    const v3 gh = ld3(a.ghmap, s.gi, a.np);
    const double part = adj_part(a, G::nparam(a) + 3);
    t.store(a, L);
    tm.store(a, LM);
    __syncthreads();
    double vals[G::kMaxVals];
    for (int q = 0; q < G::kMaxVals; ++q) vals[q] = 0.0;
    if (s.active) {
        const v3 tgb = G::sum(a, L, T, s.c);
        const v3 gmt = v_scale(0.5, mk3(gpd.x - tgb.x, gpd.y - tgb.y, gpd.z - tgb.z));
        v3 gm = v_add(gacc, gmt);
        const v3 m = mk3(LM[s.c], LM[T + s.c], LM[2 * T + s.c]);
        const SibVec v = adj_vec(a, m, G::sum(a, LM, T, s.c), b);
        const v3 mt = cayley(m, v.av);
        gm = v_add(gm, cayley(gmt, mk3(-v.av.x, -v.av.y, -v.av.z)));
        const v3 w = minv_t(v.av, gmt);
        const v3 ga = cross3(w, v_add(mt, m));
        const v3 gB = v_scale(a.f, v_add(ga, v_scale(a.alpha, cross3(ga, m))));
        gm = v_add(gm, v_scale(a.f * a.alpha, cross3(v.B, ga)));
        st3(a.out0, s.gi, a.np, gB);
        st3(a.out1, s.gi, a.np, gm);
        G::units(a, LM, T, s.c, gB, vals);
        const v3 gb = zeeman_vjp(a, gB);
        vals[G::nparam(a)] = gb.x;
        vals[G::nparam(a) + 1] = gb.y;
        vals[G::nparam(a) + 2] = gb.z;
        st3(a.ghmap, s.gi, a.np, v_add(gh, gb));
    }
    adj_reduce<G>(a, red, vals, part);
}

// R3: lambda_n = gacc2 - C * gB1   (x = gB1)
template <class G>
__device__ __forceinline__ void adj_r3_body(const AdjArgs &a, double *L)
{
    const Site s = adj_site<G>(a);
    AdjTile<G, 1> t;
    t.load(a, a.x, L, s.x0, s.y0, s.z0);
    const v3 g = ld3(a.gacc_in, s.gi, a.np);
    t.store(a, L);
    __syncthreads();
    if (!s.active) return;
    const v3 c = G::sum(a, L, s.T, s.c);
    st3(a.out0, s.gi, a.np, mk3(g.x - c.x, g.y - c.y, g.z - c.z));
}
