// gfx950 kernels of the multigrid preconditioner of the red-black CG (see MgDesc in
// tau_internal.h for the cycle and its data).
//
// The fine level's sweeps are fused pairs like k_rb_yq: one kernel forms the black values of
// x1 and leaves the red residual summed over the coarse cells (k_mg_fine<pre>), one adds the
// prolonged correction while it loads, forms the black values again and writes z with the
// partial r.z (k_mg_fine<post>).  Slot k of a red row lies in coarse cell k, so restriction and
// prolongation along x are the identity on the slots.  Coarse levels take four half-sweep
// kernels each, the levels that fit the LDS of one CU one launch together.
#include "device_common.h"

#include <algorithm>

namespace ft {

namespace {

// Smallest volume and shortest flow axis that take the cycle.  Along a short axis the Jacobi form
// needs few iterations too ((180, n, 200) along y to 1e-8: n = 16 4.8 ms against 5.7 with the
// cycle, n = 24 6.7 against 6.6, n = 32 8.2 against 7.3).  Smaller volumes would gain as well (48^3
// 6.3 -> 2.7 ms, 32^3 4.1 -> 2.0 ms), but keep the Jacobi form, by whose iteration counts the
// compaction of batch tails is pinned (24 x 40 x 96 volumes).
constexpr long long kMgMinVoxels = 96 * 1024;
constexpr int kMgMinFlow = 24;

__host__ __device__ constexpr int half_up(int n) { return (n + 1) / 2; }

// Face coefficients of a row in FP32 (positive), as k_rb_yq's LDS pairs.
__device__ __forceinline__ float mg_sum(const FacePair<float>* ftab, int code, const float (&o)[6]) {
    const int o4 = (code >> 4) & 4;
    const FacePair<float> px = ftab[(code & 3) | o4];
    const FacePair<float> py = ftab[((code >> 2) & 3) | o4];
    const FacePair<float> pz = ftab[((code >> 4) & 3) | o4];
    float acc = 0.0f;
    acc = fmaf(pz.m, o[0], acc);
    acc = fmaf(py.m, o[1], acc);
    acc = fmaf(px.m, o[2], acc);
    acc = fmaf(px.p, o[3], acc);
    acc = fmaf(py.p, o[4], acc);
    acc = fmaf(pz.p, o[5], acc);
    return acc;
}

// Fine level.  Geometry, rings and LDS planes as in k_rb_yq (columns that march z, p planes
// double-buffered, Y planes in a ring, one barrier per plane), in FP32:
//   pre:  u = x1; Y = (1/|D_b|) A_br u; G = A_rb Y on the red voxels, summed over the four red
//         voxels of each 2 x 2 x 2 coarse cell into lev[0].g.  The two planes are summed in the
//         column's register, the two rows through LDS (odd rows store, even rows add), always
//         as (row 2Y, both planes) + (row 2Y+1, both planes).
//   post: u = x1 + e of the coarse cell (added as a plane's loads are first used); z =
//         (1/|D_r|) (A_rb Y - r) into the next p's buffer; partial r.z.
template <int TY, bool POST>
__global__ __launch_bounds__(kRbTX*(TY + 3)) __attribute__((amdgpu_waves_per_eu(6))) void k_mg_fine(RbLaunch L, MgLaunch M) {
    static_assert(TY % 2 == 0, "a tile holds whole coarse cells");
    constexpr int AHEAD = 2, R = AHEAD + 2;
    constexpr int NT = kRbTX * (TY + 3);
    constexpr int PW = kRbTX + 4, PH = TY + 4;
    constexpr int YW = kRbTX + 2, YH = TY + 2;
    constexpr int NPO = 2 * PW + 2 * (TY + 2) + 4;
    static_assert(kRbTX == 64 && NPO <= 3 * 64, "one p-only point per lane of waves TY .. TY+2");
    const int slot = xcd_remap(blockIdx.x, gridDim.x);
    if (slot >= M.ntiles) return;
    const int2 tl = M.tiles[slot];
    const int v = tl.x, lt = tl.y;
    const VolState<double>* vs = L.st + v;
    if (vs->status != ST_RUNNING || !vs->mg) return;
    const RbDesc d = L.vol[v];
    const MgDesc& md = M.vol[v];
    __shared__ float tab[kTabEntries];
    __shared__ FacePair<float> ftab[8];
    __shared__ float pbuf[2][PW * PH + 1];
    __shared__ float ybuf[R][YW * YH + 1];
    __shared__ float rows[2][TY / 2][kRbTX];
    const Coef<double> c = L.coef[v];
    const Coef<float> cf{(float)c.ci0, (float)c.ci1, (float)c.ci2, (float)c.cb0, (float)c.cb1, 0.0f, 0.0f, 0.0f, 0.0f};
    for (int i = (int)threadIdx.x; i < kTabEntries; i += NT) tab[i] = M.tab[(long long)v * kTabEntries + i];
    if (threadIdx.x < 8) ftab[threadIdx.x] = face_pair(cf, (int)threadIdx.x);
    __syncthreads();
    const int k0 = (lt % md.tiles_x) * kRbTX;
    const int y0 = ((lt / md.tiles_x) % md.tiles_y) * TY;
    const int z0 = (lt / (md.tiles_x * md.tiles_y)) * md.tz;
    const int z1 = min(z0 + md.tz, d.nz);
    const bool odd = (vs->phase & 1) != 0;
    const float* X1 = L.q + d.off_c;
    const float* Rr = L.r + d.off_c;
    float* Z = L.p[odd ? 0 : 1] + d.off_c;
    const unsigned* code_r4 = reinterpret_cast<const unsigned*>(d.code_c[0]);
    const unsigned* code_b4 = reinterpret_cast<const unsigned*>(d.code_c[1]);
    const int cnx = md.lev[0].nx, cny = md.lev[0].ny;
    float* G1 = md.mem + md.lev[0].off;
    const int tid = (int)threadIdx.x, w = tid >> 6, lane = tid & 63;
    // this thread's column (slot kc, row yc)
    const bool own = w < TY;
    const bool has_col = w < TY + 2 || lane < 2 * TY;
    const int kc = w <= TY + 1 ? k0 + lane : (lane < TY ? k0 - 1 : k0 + kRbTX);
    const int yc = own ? y0 + w : (w == TY ? y0 - 1 : (w == TY + 1 ? y0 + TY : y0 + (lane % TY)));
    const bool col_pad = has_col && kc >= -1 && kc <= d.hx && yc >= -1 && yc <= d.ny;
    const bool col_box = has_col && kc >= 0 && kc < d.hx && yc >= 0 && yc < d.ny;
    const unsigned cel = col_pad ? (unsigned)(kc + 1) + (unsigned)d.px * (unsigned)(yc + 1) : 0u;
    const unsigned cel4 = cel >> 2, csh = (cel & 3u) * 8u;
    const int pdst = has_col ? (kc - k0 + 2) + (yc - y0 + 2) * PW : PW * PH;
    const int ypos = (kc - k0 + 1) + (yc - y0 + 1) * YW;
    const int ydst = has_col ? ypos : YW * YH;
    const bool ok0 = col_box && 2 * kc < d.nx, ok1 = col_box && 2 * kc + 1 < d.nx;
    const int xo0 = (2 * kc == d.nx - 1 ? 1 << 7 : 0) | (kc == 0 ? 1 << 8 : 0);
    const int xo1 = 2 * kc + 1 == d.nx - 1 ? 1 << 7 : 0;
    const bool yface = yc == 0 || yc == d.ny - 1;
    const int sb0 = (1 + yc) & 1;   // parity of the column's black voxel in even planes (red: 1 - sb0)
    const unsigned ecol = col_box ? (unsigned)kc + (unsigned)cnx * (unsigned)(yc >> 1) : 0u;
    // this thread's p-only point (lanes of waves TY .. TY+2)
    int podst = PW * PH;
    unsigned pel = 0u, epel = 0u;
    bool pok0 = false, pok1 = false;
    int psr0 = 0;   // parity of the point's red voxel in even planes
    {
        const int i = (w - TY) * 64 + lane;
        if (w >= TY && i < NPO) {
            int kk, yy;
            if (i < 2 * PW) {
                kk = k0 - 2 + i % PW;
                yy = i < PW ? y0 - 2 : y0 + TY + 1;
            } else if (i < 2 * PW + 2 * (TY + 2)) {
                const int j = i - 2 * PW;
                kk = j < TY + 2 ? k0 - 2 : k0 + kRbTX + 1;
                yy = y0 - 1 + j % (TY + 2);
            } else {
                const int j = i - 2 * PW - 2 * (TY + 2);
                kk = (j & 1) ? k0 + kRbTX : k0 - 1;
                yy = (j & 2) ? y0 + TY : y0 - 1;
            }
            podst = (kk - k0 + 2) + (yy - y0 + 2) * PW;
            if (kk >= -1 && kk <= d.hx && yy >= -1 && yy <= d.ny) pel = (unsigned)(kk + 1) + (unsigned)d.px * (unsigned)(yy + 1);
            if (kk >= 0 && kk < d.hx && yy >= 0 && yy < d.ny) {
                epel = (unsigned)kk + (unsigned)cnx * (unsigned)(yy >> 1);
                psr0 = yy & 1;
                pok0 = 2 * kk < d.nx;
                pok1 = 2 * kk + 1 < d.nx;
            }
        }
    }
    // plane zz's offset in elements (uniform); 0 outside -1 .. nz
    auto plane = [&](int zz) { return (unsigned)(zz + 1) <= (unsigned)(d.nz + 1) ? d.pp * (unsigned)(zz + 1) : 0u; };
    auto eplane = [&](int zz) {
        return (unsigned)zz < (unsigned)d.nz ? (unsigned)cnx * (unsigned)cny * (unsigned)(zz >> 1) : 0u;
    };
    // 1 / |diagonal| of a row: the table, or the formula on a y or z box face
    auto inv = [&](int code, int s, int yy, int zz, bool zface) {
        if (yface || zface)
            return -1.0f / diag_of<float>(code, box_flags(2 * kc + s, yy, zz, d.nx, d.ny, d.nz), d.primary, cf);
        return tab[code | (s ? xo1 : xo0)];
    };
    AccDD acc[1];
    acc[0].init();
    const int t0 = z0 - 1;
    float pr[R], po[R], er[R], eo[R], rr[R];
    unsigned cb[R], cr[R];
    // u of plane zz from its loads: the correction is added on the red voxels of the box
    auto finish_col = [&](int zz, float x, float e) {
        const bool ok = (((~sb0 ^ zz) & 1) ? ok1 : ok0) && (unsigned)zz < (unsigned)d.nz;
        return ok ? x + e : x;
    };
    auto finish_po = [&](int zz, float x, float e) {
        const bool ok = (((psr0 ^ zz) & 1) ? pok1 : pok0) && (unsigned)zz < (unsigned)d.nz;
        return ok ? x + e : x;
    };
    pr[R - 1] = ld(X1 + plane(t0 - 1), cel);
    if (POST) er[R - 1] = ld(G1 + eplane(t0 - 1), ecol);
    cr[R - 1] = 0;
    rr[R - 1] = 0.0f;
#pragma unroll
    for (int i = 0; i < AHEAD; ++i) {
        const unsigned o = plane(t0 + i);
        pr[i] = ld(X1 + o, cel);
        po[i] = ld(X1 + o, pel);
        if (POST) {
            er[i] = ld(G1 + eplane(t0 + i), ecol);
            eo[i] = ld(G1 + eplane(t0 + i), epel);
        }
        cb[i] = ld(code_b4 + (o >> 2), cel4);
        if (i < AHEAD - 1) {
            cr[i] = ld(code_r4 + (o >> 2), cel4);
            if (POST) rr[i] = ld(Rr + o, cel);
        }
    }
    if (POST) {
        pr[R - 1] = finish_col(t0 - 1, pr[R - 1], er[R - 1]);
        pr[0] = finish_col(t0, pr[0], er[0]);
    }
    float hold = 0.0f;   // pre: G of the pair's first plane
    auto step = [&](auto J, int t) {
        constexpr int j = decltype(J)::value;
        constexpr int jm = (j + R - 1) % R, jn = (j + 1) % R;
        {
            const unsigned o = plane(t + AHEAD), oq = plane(t + AHEAD - 1);
            pr[(j + AHEAD) % R] = ld(X1 + o, cel);
            po[(j + AHEAD) % R] = ld(X1 + o, pel);
            cb[(j + AHEAD) % R] = ld(code_b4 + (o >> 2), cel4);
            cr[(j + AHEAD - 1) % R] = ld(code_r4 + (oq >> 2), cel4);
            if (POST) {
                const unsigned eo_ = eplane(t + AHEAD);
                er[(j + AHEAD) % R] = ld(G1 + eo_, ecol);
                eo[(j + AHEAD) % R] = ld(G1 + eo_, epel);
                rr[(j + AHEAD - 1) % R] = ld(Rr + oq, cel);
            }
        }
        if (POST) pr[jn] = finish_col(t + 1, pr[jn], er[jn]);
        float* pb = pbuf[t & 1];
        pb[pdst] = pr[j];
        pb[podst] = POST ? finish_po(t, po[j], eo[j]) : po[j];
        __syncthreads();
        const int s = sb0 ^ (t & 1);
        const float* pl = pb + pdst;
        const float u[6] = {pr[jm], pl[-PW], pl[s - 1], pl[s], pl[PW], pr[jn]};
        const int code = (int)((cb[j] >> csh) & 0xffu);
        const float yv = mg_sum(ftab, code, u) * inv(code, s, yc, t, t == 0 || t == d.nz - 1);
        const float yt = ((s ? ok1 : ok0) && t >= 0 && t < d.nz) ? yv : 0.0f;
        ybuf[j][ydst] = yt;
        // red voxel of plane t - 1 (own rows; it has the parity of plane t's black one)
        const int tq = t - 1;
        const bool red = own && (s ? ok1 : ok0) && tq >= z0 && tq < z1;
        float g = 0.0f;
        if (red) {
            const float* yl = ybuf[jm] + ypos;
            const float o[6] = {ybuf[(j + R - 2) % R][ypos], yl[-YW], yl[s - 1], yl[s], yl[YW], yt};
            const int code_q = (int)((cr[jm] >> csh) & 0xffu);
            g = mg_sum(ftab, code_q, o);
            if (POST) {
                const float zv = (g - rr[jm]) * inv(code_q, s, yc, tq, tq == 0 || tq == d.nz - 1);
                st(Z + d.pp * (unsigned)(tq + 1), cel, zv);
                acc[0].add(rr[jm], zv);
            }
        }
        if (!POST) {
            const int o = tq - z0;
            if (o & 1) {   // the pair is complete: odd rows hand theirs over
                hold += g;
                if (own && (w & 1)) rows[(o >> 1) & 1][w >> 1][lane] = hold;
            } else {
                if (o >= 2 && own && !(w & 1) && ok0)   // after the barrier: the previous pair
                    st(G1 + (unsigned)cnx * (unsigned)cny * (unsigned)((tq - 2) >> 1), ecol,
                       hold + rows[((o >> 1) - 1) & 1][w >> 1][lane]);
                hold = g;
            }
        }
    };
    for (int t = t0;; t += R)
        if (ring_turn<0, R, R>(step, t, z1)) break;
    if (POST) {
        block_reduce_store<AccDD, 1, NT>(acc, M.part + 2 * ((long long)md.part_base + lt));
        return;
    }
    const int ol = z1 - 1 - z0;   // the last pair (one plane at the end of an odd volume)
    if (own && (w & 1) && !(ol & 1)) rows[(ol >> 1) & 1][w >> 1][lane] = hold;
    __syncthreads();
    if (own && !(w & 1) && ok0)
        st(G1 + (unsigned)cnx * (unsigned)cny * (unsigned)((z1 - 1) >> 1), ecol, hold + rows[(ol >> 1) & 1][w >> 1][lane]);
}

// ---- coarse levels -------------------------------------------------------------------------
// A thread takes the red or black voxel of one row of one coarse cell: four consecutive lanes
// (the cell's four rows) per cell of the next level, so the restriction sums four lanes.
struct MgLev {
    int nx, ny, nz, cx, cy;          // extents; those of the next level (x, y)
    float *g, *t, *fx, *fy, *fz, *iv;
    float* gc;                       // next level's g
};

__device__ __forceinline__ MgLev mg_lev(const MgDesc& d, int l) {
    MgLev r;
    const MgLevel& a = d.lev[l];
    r.nx = a.nx;
    r.ny = a.ny;
    r.nz = a.nz;
    r.cx = half_up(a.nx);
    r.cy = half_up(a.ny);
    r.g = d.mem + a.off;
    r.t = r.g + a.n;
    r.fx = r.t + a.n;
    r.fy = r.fx + a.n;
    r.fz = r.fy + a.n;
    r.iv = r.fz + a.n;
    r.gc = d.mem + d.lev[l + 1].off;
    return r;
}

struct MgCell {
    int x, y, z;
    unsigned i;
    bool ok;
};

// Cell of colour `colour` in row j (0..3) of coarse cell C.
__device__ __forceinline__ MgCell mg_cell(int nx, int ny, int nz, int cx, int cy, unsigned C, int j, int colour) {
    const unsigned row = C / (unsigned)cx;
    const int K = (int)(C - row * (unsigned)cx);
    const int Z = (int)(row / (unsigned)cy), Y = (int)(row - (unsigned)Z * (unsigned)cy);
    MgCell c;
    c.y = 2 * Y + (j & 1);
    c.z = 2 * Z + (j >> 1);
    c.x = 2 * K + ((colour + c.y + c.z) & 1);
    c.ok = c.x < nx && c.y < ny && c.z < nz;
    if (!c.ok) c.x = c.y = c.z = 0;   // a cell in the box: its neighbours' indices stay inside too
    c.i = (unsigned)c.x + (unsigned)nx * ((unsigned)c.y + (unsigned)ny * (unsigned)c.z);
    return c;
}

// Face coefficients and indices of the six neighbours (x-, x+, y-, y+, z-, z+); a face of the box
// has coefficient 0 and the cell itself as neighbour.
template <class LV>
__device__ __forceinline__ void mg_faces(const LV& l, const MgCell& c, float (&f)[6], unsigned (&n)[6]) {
    const unsigned sy = (unsigned)l.nx, sz = (unsigned)l.nx * (unsigned)l.ny;
    n[0] = c.x > 0 ? c.i - 1u : c.i;
    n[1] = c.x + 1 < l.nx ? c.i + 1u : c.i;
    n[2] = c.y > 0 ? c.i - sy : c.i;
    n[3] = c.y + 1 < l.ny ? c.i + sy : c.i;
    n[4] = c.z > 0 ? c.i - sz : c.i;
    n[5] = c.z + 1 < l.nz ? c.i + sz : c.i;
    f[0] = c.x > 0 ? l.fx[n[0]] : 0.0f;
    f[1] = l.fx[c.i];   // 0 at the last cell
    f[2] = c.y > 0 ? l.fy[n[2]] : 0.0f;
    f[3] = l.fy[c.i];
    f[4] = c.z > 0 ? l.fz[n[4]] : 0.0f;
    f[5] = l.fz[c.i];
}

__device__ __forceinline__ float mg_dot(const float (&f)[6], const float (&u)[6]) {
    float a = f[4] * u[4];
    a = fmaf(f[2], u[2], a);
    a = fmaf(f[0], u[0], a);
    a = fmaf(f[1], u[1], a);
    a = fmaf(f[3], u[3], a);
    return fmaf(f[5], u[5], a);
}

enum MgStep : int { MG_PRE_BLACK = 0, MG_RESTRICT, MG_POST_BLACK, MG_POST_RED };

// Half sweeps of one level:
//   pre black:  t = (g + sum c g_r iv_r) iv on black cells (red ones: g iv, never stored)
//   restrict:   next g = sum over the cell's red children of sum c t_b
//   post black: g = (g + sum c (g_r iv_r + e)) iv on black cells, e the next level's solution
//   post red:   g = (g + sum c g_b) iv on red cells (g is then the level's solution)
template <int STEP>
__global__ __launch_bounds__(kMgThreads) void k_mg_level(RbLaunch L, const MgDesc* vol, const int2* blocks, int nblk, int lev) {
    const int slot = xcd_remap(blockIdx.x, gridDim.x);
    if (slot >= nblk) return;
    const int2 b = blocks[slot];
    if (L.st[b.x].status != ST_RUNNING || !L.st[b.x].mg) return;
    const MgDesc& d = vol[b.x];
    const MgLev l = mg_lev(d, lev);
    const unsigned id = (unsigned)b.y * kMgThreads + threadIdx.x;
    const unsigned C = id >> 2, nc = (unsigned)d.lev[lev + 1].n;
    constexpr int colour = (STEP == MG_PRE_BLACK || STEP == MG_POST_BLACK) ? 1 : 0;
    MgCell c = mg_cell(l.nx, l.ny, l.nz, l.cx, l.cy, C < nc ? C : 0u, (int)(id & 3u), colour);
    c.ok = c.ok && C < nc;
    float f[6];
    unsigned n[6];
    mg_faces(l, c, f, n);
    float u[6];
    if (STEP == MG_RESTRICT) {
#pragma unroll
        for (int k = 0; k < 6; ++k) u[k] = l.t[n[k]];
        float s = 0.0f;
#pragma unroll
        for (int k = 0; k < 6; ++k) u[k] = f[k] != 0.0f ? u[k] : 0.0f;   // a box face's "neighbour" is red
        s = c.ok ? mg_dot(f, u) : 0.0f;
        s += __shfl_xor(s, 1, 64);
        s += __shfl_xor(s, 2, 64);
        if ((id & 3u) == 0u && C < nc) l.gc[C] = s;
        return;
    }
#pragma unroll
    for (int k = 0; k < 6; ++k) u[k] = l.g[n[k]];
    if (STEP != MG_POST_RED) {
        float w[6];
#pragma unroll
        for (int k = 0; k < 6; ++k) w[k] = l.iv[n[k]];
        if (STEP == MG_POST_BLACK) {
            float e[6];
            const unsigned px = (unsigned)l.cx, pxy = (unsigned)l.cx * (unsigned)l.cy;
            const unsigned cb = (unsigned)(c.y >> 1) * px + (unsigned)(c.z >> 1) * pxy;
            const unsigned base = cb + (unsigned)(c.x >> 1);
            e[0] = l.gc[c.x > 0 ? cb + (unsigned)((c.x - 1) >> 1) : base];
            e[1] = l.gc[c.x + 1 < l.nx ? cb + (unsigned)((c.x + 1) >> 1) : base];
            e[2] = l.gc[c.y > 0 && !(c.y & 1) ? base - px : base];
            e[3] = l.gc[c.y + 1 < l.ny && (c.y & 1) ? base + px : base];
            e[4] = l.gc[c.z > 0 && !(c.z & 1) ? base - pxy : base];
            e[5] = l.gc[c.z + 1 < l.nz && (c.z & 1) ? base + pxy : base];
#pragma unroll
            for (int k = 0; k < 6; ++k) u[k] = fmaf(u[k], w[k], e[k]);
        } else {
#pragma unroll
            for (int k = 0; k < 6; ++k) u[k] = u[k] * w[k];
        }
    }
    const float r = (l.g[c.i] + mg_dot(f, u)) * l.iv[c.i];
    if (!c.ok) return;
    if (STEP == MG_PRE_BLACK)
        l.t[c.i] = r;
    else
        l.g[c.i] = r;
}

// The levels from `bottom` on, one block per volume, in LDS: one V-cycle with two sweeps before
// and after each correction, down to a level of one cell, whose equation is solved.  t holds the
// iterate u.  (Two sweeps here save 3-15% of the CG's iterations at no further launches.  A second
// V-cycle on the first one's residual saves as many, but 2 B - B A B is indefinite where the
// cycle overcorrects, as in long clogged volumes.)
constexpr int kMgBottomThreads = 1024;

struct LdsLev {
    int nx, ny, nz, cx, cy, n, nc;
    float *g, *t, *fx, *fy, *fz, *iv, *gc, *tc;
};

__global__ __launch_bounds__(kMgBottomThreads) void k_mg_bottom(RbLaunch L, MgLaunch M) {
    __shared__ float sm[kMgArrays][kMgBottomCells];
    const int v = M.vols[blockIdx.x];
    if (L.st[v].status != ST_RUNNING || !L.st[v].mg) return;
    const MgDesc& d = M.vol[v];
    const int tid = (int)threadIdx.x;
    const int b = d.bottom, last = d.nlev - 1;
    // cells of a level start at its offset from the bottom level (all arrays alike)
    auto lds_off = [&](int l) { return (int)((d.lev[l].off - d.lev[b].off) / kMgArrays); };
    for (int l = b; l <= last; ++l) {
        const int n = d.lev[l].n, o = lds_off(l);
        const float* src = d.mem + d.lev[l].off;
        for (int i = tid; i < n; i += kMgBottomThreads) {
            if (l == b) sm[0][o + i] = src[i];
#pragma unroll
            for (int a = 2; a < kMgArrays; ++a) sm[a][o + i] = src[(long long)a * n + i];
        }
    }
    auto level = [&](int l) {
        LdsLev r;
        const int o = lds_off(l), oc = l < last ? lds_off(l + 1) : o;
        r.nx = d.lev[l].nx;
        r.ny = d.lev[l].ny;
        r.nz = d.lev[l].nz;
        r.cx = half_up(r.nx);
        r.cy = half_up(r.ny);
        r.n = d.lev[l].n;
        r.nc = l < last ? d.lev[l + 1].n : 0;
        r.g = sm[0] + o;
        r.t = sm[1] + o;
        r.fx = sm[2] + o;
        r.fy = sm[3] + o;
        r.fz = sm[4] + o;
        r.iv = sm[5] + o;
        r.gc = sm[0] + oc;
        r.tc = sm[1] + oc;
        return r;
    };
    // f(cell) for this thread's cells of one colour, then a barrier
    auto cells = [&](const LdsLev& q, int colour, auto f) {
        for (int id = tid; id < 4 * q.nc; id += kMgBottomThreads) {
            const MgCell c = mg_cell(q.nx, q.ny, q.nz, q.cx, q.cy, (unsigned)id >> 2, id & 3, colour);
            if (c.ok) f(c);
        }
        __syncthreads();
    };
    auto sweep = [&](const LdsLev& q, int colour) {
        cells(q, colour, [&](const MgCell& c) {
            float f[6], u[6];
            unsigned n[6];
            mg_faces(q, c, f, n);
#pragma unroll
            for (int k = 0; k < 6; ++k) u[k] = q.t[n[k]];   // a box face's coefficient is 0, t finite
            q.t[c.i] = (q.g[c.i] + mg_dot(f, u)) * q.iv[c.i];
        });
    };
    __syncthreads();
    for (int l = b; l < last; ++l) {
        const LdsLev q = level(l);
        for (int i = tid; i < q.n; i += kMgBottomThreads) q.t[i] = q.g[i] * q.iv[i];   // red sweep from zero
        __syncthreads();
        sweep(q, 1);
        sweep(q, 0);
        sweep(q, 1);
        for (int i0 = 0; i0 < 4 * q.nc; i0 += kMgBottomThreads) {   // whole waves: lanes are summed
            const int id = i0 + tid;
            float s = 0.0f;
            if (id < 4 * q.nc) {
                const MgCell c = mg_cell(q.nx, q.ny, q.nz, q.cx, q.cy, (unsigned)id >> 2, id & 3, 0);
                if (c.ok && q.iv[c.i] > 0.0f) {
                    float f[6], u[6];
                    unsigned n[6];
                    mg_faces(q, c, f, n);
#pragma unroll
                    for (int k = 0; k < 6; ++k) u[k] = q.t[n[k]];
                    s = (q.g[c.i] + mg_dot(f, u)) - q.t[c.i] / q.iv[c.i];
                }
            }
            s += __shfl_xor(s, 1, 64);
            s += __shfl_xor(s, 2, 64);
            if ((id & 3) == 0 && id < 4 * q.nc) q.gc[id >> 2] = s;
        }
        __syncthreads();
    }
    if (tid == 0) {
        const LdsLev q = level(last);
        q.t[0] = q.g[0] * q.iv[0];
    }
    __syncthreads();
    for (int l = last - 1; l >= b; --l) {
        const LdsLev q = level(l);
        cells(q, 0, [&](const MgCell& c) { q.t[c.i] += q.tc[(c.x >> 1) + q.cx * ((c.y >> 1) + q.cy * (c.z >> 1))]; });
        sweep(q, 1);
        sweep(q, 0);
        sweep(q, 1);
        sweep(q, 0);
    }
    float* out = d.mem + d.lev[b].off;
    const LdsLev q = level(b);
    for (int i = tid; i < q.n; i += kMgBottomThreads) out[i] = q.t[i];
}

// r.z of one preconditioned volume, then beta = r.z / (previous r.z).
__global__ __launch_bounds__(kFinThreads) void k_mg_fin(RbLaunch L, MgLaunch M) {
    const int v = M.vols[blockIdx.x];
    VolState<double>* s = L.st + v;
    if (s->status != ST_RUNNING || !s->mg) return;
    const MgDesc& d = M.vol[v];
    AccDD sum[1];
    sum[0].init();
    for (int i = (int)threadIdx.x; i < d.ntiles; i += kFinThreads) {
        const double* p = M.part + 2 * ((long long)d.part_base + i);
        sum[0].add2(p[0], p[1]);
    }
    __shared__ double red[2];
    block_reduce_store<AccDD, 1, kFinThreads>(sum, red);
    if (threadIdx.x == 0) {
        const double rz = red[0] + red[1];
        if (!s->first) s->beta = rz / s->absnew;
        s->absnew = rz;
    }
}

// ---- set-up --------------------------------------------------------------------------------
// Coefficient of a coarse face: the children's faces across it (sum m) in series with half of each
// side's own faces (sums l and r over the four child pairs; has = false: the side is one child
// wide), but at least kMgFaceMin of m.  Between uniform full cells this is m / 2, the coarse
// area over the coarse distance; a solid wall inside a cell, which the cell's one value cannot
// resolve, lowers it, a wall on the face raises it to m.  Without the lower bound porous media
// (paths around the wall) take up to 10x the iterations, with m / 2 throughout (8, 8, 4096)-like
// clogged volumes take 3x (184 against 59).
constexpr float kMgFaceMin = 0.4f;
__device__ __forceinline__ float mg_series(float m, float l, bool has_l, float r, bool has_r) {
    float R = 1.0f / m;
    if (has_l) R += 0.5f / l;
    if (has_r) R += 0.5f / r;
    return m > 0.0f ? fmaxf(1.0f / R, kMgFaceMin * m) : 0.0f;
}

// Coefficients of level l from the stencil codes (l = 0) or from level l - 1: the faces towards
// x+, y+, z+ and, in t, the cell's half-cell faces on the primary axis.
__global__ __launch_bounds__(kMgThreads) void k_mg_coef(RbLaunch L, MgLaunch M, int lev) {
    const int v = M.vols[blockIdx.y];
    const MgDesc& d = M.vol[v];
    if (lev >= d.nlev) return;
    const MgLevel& a = d.lev[lev];
    const RbDesc& rb = L.vol[v];
    float* g = d.mem + a.off;
    float *t = g + a.n, *fx = t + a.n, *fy = fx + a.n, *fz = fy + a.n;
    const int fn[3] = {lev ? d.lev[lev - 1].nx : rb.nx, lev ? d.lev[lev - 1].ny : rb.ny, lev ? d.lev[lev - 1].nz : rb.nz};
    const int primary = rb.primary;
    const Coef<double> c = L.coef[v];
    const float ci[3] = {(float)c.ci0, (float)c.ci1, (float)c.ci2};
    const float cb[2] = {(float)c.cb0, (float)c.cb1};
    const float* pf[3] = {nullptr, nullptr, nullptr};
    const float* pt = nullptr;
    if (lev) {
        const MgLevel& p = d.lev[lev - 1];
        const float* m = d.mem + p.off;
        pt = m + p.n;
        pf[0] = pt + p.n;
        pf[1] = pf[0] + p.n;
        pf[2] = pf[1] + p.n;
    }
    const unsigned st[3] = {1u, (unsigned)fn[0], (unsigned)fn[0] * (unsigned)fn[1]};
    // face of child fi towards + along axis q (inside the box)
    auto face = [&](unsigned fi, int q) {
        if (lev) return pf[q][fi];
        const int code = rb.code[fi];
        return ci[((code >> 6) & 1) + ((code >> (2 * q)) & 1)];
    };
    // sum of the faces towards + along q of the children at plane k (along q) of the coarse cell I
    auto sum4 = [&](const int (&I)[3], int q, int k) {
        const int u = q == 0 ? 1 : 0, w = q == 2 ? 1 : 2;
        float s = 0.0f;
        for (int j = 0; j < 4; ++j) {
            const int a0 = 2 * I[u] + (j & 1), a1 = 2 * I[w] + (j >> 1);
            if (a0 < fn[u] && a1 < fn[w]) s += face((unsigned)a0 * st[u] + (unsigned)a1 * st[w] + (unsigned)k * st[q], q);
        }
        return s;
    };
    for (unsigned i = blockIdx.x * kMgThreads + threadIdx.x; i < (unsigned)a.n; i += gridDim.x * kMgThreads) {
        const unsigned row = i / (unsigned)a.nx;
        const int I[3] = {(int)(i - row * (unsigned)a.nx), (int)(row % (unsigned)a.ny), (int)(row / (unsigned)a.ny)};
        float s[3], own[3];
#pragma unroll
        for (int q = 0; q < 3; ++q) {
            const int lo = 2 * I[q], nq = fn[q];
            own[q] = lo + 1 < nq ? sum4(I, q, lo) : 0.0f;
            s[q] = 0.0f;
            if (lo + 2 < nq) {
                const bool wide = lo + 3 < nq;   // the next cell has two children
                s[q] = mg_series(sum4(I, q, lo + 1), own[q], true, wide ? sum4(I, q, lo + 2) : 0.0f, wide);
            }
        }
        // half-cell faces at either end of the primary axis
        const int np = fn[primary], lo = 2 * I[primary];
        const float inner = primary == 0 ? own[0] : (primary == 1 ? own[1] : own[2]);
        float end[2] = {0.0f, 0.0f};
        for (int j = 0; j < 8; ++j) {
            const int x[3] = {2 * I[0] + (j & 1), 2 * I[1] + ((j >> 1) & 1), 2 * I[2] + (j >> 2)};
            if (x[0] >= fn[0] || x[1] >= fn[1] || x[2] >= fn[2]) continue;
            const int k = primary == 0 ? x[0] : (primary == 1 ? x[1] : x[2]);
            if (k != 0 && k != np - 1) continue;
            const unsigned fi = (unsigned)x[0] + (unsigned)x[1] * st[1] + (unsigned)x[2] * st[2];
            if (lev) {
                end[k == 0 ? 0 : 1] += pt[fi];   // one cell along the axis: both ends together
            } else {
                const float h = cb[(rb.code[fi] >> 6) & 1];
                if (k == 0) end[0] += h;
                if (k == np - 1) end[1] += h;
            }
        }
        const bool two = lo + 1 < np;   // two children along the axis
        g[i] = 0.0f;
        fx[i] = s[0];
        fy[i] = s[1];
        fz[i] = s[2];
        t[i] = mg_series(end[0], inner, two, 0.0f, false) + mg_series(end[1], inner, two, 0.0f, false);
    }
}

// 1 / diagonal of every level, and the fine level's FP32 table.
__global__ __launch_bounds__(kMgThreads) void k_mg_diag(RbLaunch L, MgLaunch M) {
    const int v = M.vols[blockIdx.y];
    const MgDesc& d = M.vol[v];
    const unsigned id = blockIdx.x * kMgThreads + threadIdx.x, step = gridDim.x * kMgThreads;
    for (unsigned i = id; i < (unsigned)kTabEntries; i += step)
        M.tab[(long long)v * kTabEntries + i] = (float)(-L.tab[(long long)v * 2 * kTabEntries + kTabEntries + i]);
    for (int l = 0; l < d.nlev; ++l) {
        const MgLevel& a = d.lev[l];
        const float* t = d.mem + a.off + a.n;
        const float *fx = t + a.n, *fy = fx + a.n, *fz = fy + a.n;
        float* iv = d.mem + a.off + (size_t)5 * a.n;
        for (unsigned i = id; i < (unsigned)a.n; i += step) {
            const unsigned row = i / (unsigned)a.nx;
            const int X = (int)(i - row * (unsigned)a.nx), Y = (int)(row % (unsigned)a.ny), Z = (int)(row / (unsigned)a.ny);
            float s = t[i] + fx[i] + fy[i] + fz[i];
            if (X > 0) s += fx[i - 1];
            if (Y > 0) s += fy[i - (unsigned)a.nx];
            if (Z > 0) s += fz[i - (unsigned)a.nx * (unsigned)a.ny];
            iv[i] = s > 0.0f ? 1.0f / s : 0.0f;
        }
    }
}

}  // namespace

bool mg_plan(int nx, int ny, int nz, int primary, MgDesc* d, size_t* floats) {
    *d = MgDesc{};
    *floats = 0;
    const int flow = primary == 0 ? nx : (primary == 1 ? ny : nz);
    if ((long long)nx * ny * nz < kMgMinVoxels || flow < kMgMinFlow) return false;
    int x = nx, y = ny, z = nz;
    size_t off = 0;
    while ((d->nlev == 0 || x > 1 || y > 1 || z > 1) && d->nlev < kMgLevels) {
        x = half_up(x);
        y = half_up(y);
        z = half_up(z);
        MgLevel& l = d->lev[d->nlev++];
        l.nx = x;
        l.ny = y;
        l.nz = z;
        l.n = x * y * z;
        l.off = (unsigned)off;
        off += (size_t)kMgArrays * l.n;
    }
    if (d->lev[d->nlev - 1].n != 1) return false;
    int cells = 0;
    d->bottom = d->nlev;
    while (d->bottom > 0 && cells + d->lev[d->bottom - 1].n <= kMgBottomCells) cells += d->lev[--d->bottom].n;
    const size_t elems = (size_t)rb_row_pitch(half_up(nx)) * (size_t)(ny + 2) * (size_t)(nz + 2);
    if (off > 2 * elems) return false;
    d->tiles_x = (half_up(nx) + kRbTX - 1) / kRbTX;
    d->tiles_y = (ny + kMgTY - 1) / kMgTY;
    const long long txy = (long long)d->tiles_x * d->tiles_y;
    long long tz = (long long)nz * txy / 512;   // about two blocks per CU
    tz = std::max<long long>(4, std::min<long long>(32, tz));
    d->tz = (int)(tz & ~1ll);
    d->tiles_z = (nz + d->tz - 1) / d->tz;
    d->ntiles = d->tiles_x * d->tiles_y * d->tiles_z;
    *floats = off;
    return true;
}

hipError_t mg_setup(const RbLaunch& L, const MgLaunch& M, hipStream_t s) {
    if (M.nvol <= 0) return hipSuccess;
    for (int l = 0; l < M.nlev_max; ++l)
        hipLaunchKernelGGL(k_mg_coef, dim3(l == 0 ? 512 : (l == 1 ? 64 : 8), M.nvol), dim3(kMgThreads), 0, s, L, M, l);
    hipLaunchKernelGGL(k_mg_diag, dim3(512, M.nvol), dim3(kMgThreads), 0, s, L, M);
    return hipGetLastError();
}

hipError_t mg_cycle(const RbLaunch& L, const MgLaunch& M, hipStream_t s) {
    const dim3 fb(kRbTX * (kMgTY + 3)), cb(kMgThreads);
    hipLaunchKernelGGL((k_mg_fine<kMgTY, false>), dim3(M.ntiles), fb, 0, s, L, M);
    for (int l = 0; l < M.nlev; ++l) {
        const int2* blk = M.blocks + M.blk_off[l];
        hipLaunchKernelGGL((k_mg_level<MG_PRE_BLACK>), dim3(M.nblk[l]), cb, 0, s, L, M.vol, blk, M.nblk[l], l);
        hipLaunchKernelGGL((k_mg_level<MG_RESTRICT>), dim3(M.nblk[l]), cb, 0, s, L, M.vol, blk, M.nblk[l], l);
    }
    hipLaunchKernelGGL(k_mg_bottom, dim3(M.nvol), dim3(kMgBottomThreads), 0, s, L, M);
    for (int l = M.nlev - 1; l >= 0; --l) {
        const int2* blk = M.blocks + M.blk_off[l];
        hipLaunchKernelGGL((k_mg_level<MG_POST_BLACK>), dim3(M.nblk[l]), cb, 0, s, L, M.vol, blk, M.nblk[l], l);
        hipLaunchKernelGGL((k_mg_level<MG_POST_RED>), dim3(M.nblk[l]), cb, 0, s, L, M.vol, blk, M.nblk[l], l);
    }
    hipLaunchKernelGGL((k_mg_fine<kMgTY, true>), dim3(M.ntiles), fb, 0, s, L, M);
    hipLaunchKernelGGL(k_mg_fin, dim3(M.nvol), dim3(kFinThreads), 0, s, L, M);
    return hipGetLastError();
}

}  // namespace ft
