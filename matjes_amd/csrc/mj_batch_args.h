// The table entry of a batched system and a tile's kernel arguments from it,
// shared by the ahead-of-time batch kernels (mj_batch.hip) and those compiled
// per stencil (mj_jit.hip).
#pragma once

struct BatchSys {
    int nx, ny, nz, px, py, pz;
    int bx, by, bz, rx, ry, rz, sx, sy, sz, ntx, nty, ntz, nblocks, block0;
    int n_ent, ofs_off, bmode;   // ofs_off: offsets and blocks of the entries
    int ofs0_off;         // the stencil's offsets in the fused step's S0 layout (tile + 2R)
    int64_t base;
    const double *hdip;   // dipolar systems: the padded grid of H_fft (null: none), its row / plane / component strides
    int dnx, dny;
    int64_t hstride;
    double zb[3];
    double z9[9];         // the Zeeman block, for a per-site B map (bmode 2)
    double alpha, rden;   // rden = 1 / (1 + alpha^2)
    uint64_t seed;
};

// the arguments of tile gb (a tile of system S) from the batch-wide ones:
// the system's geometry, stencil, Zeeman term, damping and Philox stream, its
// slice of the state buffers, its thermal amplitude and the absolute step;
// DIP: the batch holds dipolar systems (their H_fft grids)
template <bool DIP = false>
__device__ __forceinline__ KArgs sys_args(const KArgs &base, const BatchSys &S, int gb, double sigma, uint64_t step)
{
    KArgs a = base;
    a.nx = S.nx;
    a.ny = S.ny;
    a.nz = S.nz;
    a.px = S.px;
    a.py = S.py;
    a.pz = S.pz;
    a.bx = S.bx;
    a.by = S.by;
    a.bz = S.bz;
    a.rx = S.rx;
    a.ry = S.ry;
    a.rz = S.rz;
    a.sx = S.sx;
    a.sy = S.sy;
    a.sz = S.sz;
    a.ntx = S.ntx;
    a.nty = S.nty;
    a.ntz = S.ntz;
    a.nblocks = S.nblocks;
    a.vbid = gb - S.block0;
    a.vbase = S.block0;
    a.src = base.src + S.base;
    a.own = base.own ? base.own + S.base : nullptr;
    a.dst = base.dst ? base.dst + S.base : nullptr;
    a.aux = base.aux ? base.aux + S.base : nullptr;
    a.ofs = base.ofs + S.ofs_off;
    a.cf = base.cf + 9 * S.ofs_off;
    a.n_ent = S.n_ent;
    a.bmode = S.bmode;
    a.zb[0] = S.zb[0];
    a.zb[1] = S.zb[1];
    a.zb[2] = S.zb[2];
    a.bmap = base.bmap ? base.bmap + S.base : nullptr;
#pragma unroll
    for (int k = 0; k < 9; ++k) a.z[k] = S.z9[k];
    if constexpr (DIP) {
        a.hdip = S.hdip;
        a.dnx = S.dnx;
        a.dny = S.dny;
        a.hstride = S.hstride;
    }
    a.alpha = S.alpha;
    a.kdt = base.kt * S.rden;
    a.sigma = sigma;
    a.seed = S.seed;
    a.step = step;
    return a;
}
