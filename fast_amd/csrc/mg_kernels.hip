// gfx950 kernels of the multigrid preconditioner of the red-black CG (see MgDesc in
// tau_internal.h for the cycle and its data).
//
// The fine level's sweeps are fused pairs like k_rb_yq: one kernel forms the black values of
// x1 and leaves the red residual summed over the coarse cells (k_mg_fine<pre>), one adds the
// prolonged correction while it loads, forms the black values again and writes z with the
// partial r.z (k_mg_fine<post>).  Slot k of a red row lies in coarse cell k, so restriction and
// prolongation along x are the identity on the slots.  Coarse levels take one launch per half
// cycle each, the levels that fit the LDS of one CU one launch together.
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

// g1: the first level's g (pre), its solution (post).
__device__ __forceinline__ MgFine mg_fine(const MgDesc& d, bool post) {
    return MgFine{d.tiles_x, d.tiles_y, d.tz, d.part_base, d.lev[0].nx, d.lev[0].ny, d.mem + d.lev[0].off + (post ? d.lev[0].n : 0)};
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
    const MgFine md = mg_fine(M.vol[v], POST);
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
    const int cnx = md.cnx, cny = md.cny;
    float* G1 = md.g1;
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
    // Rings: u, the p-only point and the black code of planes t-1 .. t+2; the red code and r of planes
    // t-1 and t (issued first in a step, so waiting for them leaves the later loads in flight); e of
    // two plane pairs (t0 is odd, so a plane's pair is a constant of its ring index).
    float pr[R], po[R], er[2], eo[2], rr[2];
    unsigned cb[R], cr[2];
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
    if (POST) {
        er[1] = ld(G1 + eplane(t0), ecol);   // planes t0 - 1 and t0
        eo[1] = ld(G1 + eplane(t0), epel);
        er[0] = ld(G1 + eplane(t0 + 1), ecol);
        eo[0] = ld(G1 + eplane(t0 + 1), epel);
    }
    cr[1] = 0;   // q(t0 - 1) is never formed
    rr[1] = 0.0f;
#pragma unroll
    for (int i = 0; i < AHEAD; ++i) {
        const unsigned o = plane(t0 + i);
        pr[i] = ld(X1 + o, cel);
        po[i] = ld(X1 + o, pel);
        cb[i] = ld(code_b4 + (o >> 2), cel4);
    }
    if (POST) {
        pr[R - 1] = finish_col(t0 - 1, pr[R - 1], er[1]);
        pr[0] = finish_col(t0, pr[0], er[1]);
    }
    float hold = 0.0f;   // pre: G of the pair's first plane
    auto step = [&](auto J, int t) {
        constexpr int j = decltype(J)::value;
        constexpr int jm = (j + R - 1) % R, jn = (j + 1) % R;
        {
            const unsigned oq = plane(t), o = plane(t + AHEAD);
            cr[j & 1] = ld(code_r4 + (oq >> 2), cel4);
            if (POST) rr[j & 1] = ld(Rr + oq, cel);
            pr[(j + AHEAD) % R] = ld(X1 + o, cel);
            po[(j + AHEAD) % R] = ld(X1 + o, pel);
            cb[(j + AHEAD) % R] = ld(code_b4 + (o >> 2), cel4);
            if (POST && (j & 1)) {   // plane t + 2 opens a pair
                er[((j + 1) >> 1) & 1] = ld(G1 + eplane(t + AHEAD), ecol);
                eo[((j + 1) >> 1) & 1] = ld(G1 + eplane(t + AHEAD), epel);
            }
        }
        if (POST) pr[jn] = finish_col(t + 1, pr[jn], er[(j >> 1) & 1]);
        float* pb = pbuf[t & 1];
        pb[pdst] = pr[j];
        pb[podst] = POST ? finish_po(t, po[j], eo[((j + 3) >> 1) & 1]) : po[j];
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
            const int code_q = (int)((cr[(j + 1) & 1] >> csh) & 0xffu);
            g = mg_sum(ftab, code_q, o);
            if (POST) {
                const float zv = (g - rr[(j + 1) & 1]) * inv(code_q, s, yc, tq, tq == 0 || tq == d.nz - 1);
                st(Z + d.pp * (unsigned)(tq + 1), cel, zv);
                acc[0].add(rr[(j + 1) & 1], zv);
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
struct MgCell {
    int x, y, z;
    unsigned i;
    bool ok;
};

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

struct MgLevelArgs {
    const VolState<double>* st;
    const MgDesc* vol;
    const int2* blocks;
    int nblk, lev, tz;
};

struct Float2 {   // two neighbouring floats at any element
    float x, y;
};
__device__ __forceinline__ Float2 ld2(const float* p, unsigned i) {
    Float2 v;
    __builtin_memcpy(&v, p + i, sizeof(v));
    return v;
}

// One level, half a cycle per launch:
//   down: b = (g + sum c g_r iv_r) iv on the black cells (the red ones are g iv), next g = sum over the
//         cell's red children of sum c b
//   up:   b = (g + sum c (g_r iv_r + e)) iv with e the next level's solution (its t), red cells
//         (g + sum c b) iv; both are the level's solution, stored in t
// A thread takes a column of cell pairs (2k, 2k + 1) of one row and marches z; each plane of a pair has
// one red and one black cell.  Step t forms the black cells of plane t and the red ones of plane t - 1,
// which are at the same x.  LDS holds a value per pair: the red values of planes t, t + 1 and the black
// ones of planes t - 1, t.  A tile has one pair and two rows of halo on each side, where the values
// its own red cells need are formed again.  Loads take both cells of a pair, two planes ahead.
// Bound by the chain of steps at 32^3 and 64^3 cells, by loads and memory (five values a cell) beyond.
// Two launches a half cycle, one per colour with a thread per cell of that colour, took twice the
// traffic: a cycle's levels of 64^3 (one level) 15.4 -> 9.6 us in half as many launches, of 256^3
// (three) 75 -> 58 us, of 384^3 (four) 197 -> 144 us, of 24 volumes 100 -> 83 us.  With 4-byte loads
// of the cells' own faces this form took 83 us at 256^3; tiles of 24 rows and 512 threads are even.
template <bool UP>
__global__ __launch_bounds__(kMgThreads) void k_mg_level(MgLevelArgs A) {
    constexpr int TK = kMgLevTK, TY = kMgLevTY, PW = TK + 2, PH = TY + 4;
    static_assert(PW * PH <= kMgThreads && TY % 2 == 0, "a thread per pair of the tile and its halo");
    __shared__ float wbuf[2][PW * (PH + 2) + 2], bbuf[2][PW * (PH + 2) + 2];
    __shared__ float rows[2][TY / 2][TK];
    const int slot = xcd_remap(blockIdx.x, gridDim.x);
    if (slot >= A.nblk) return;
    const int2 b = A.blocks[slot];
    const MgLevel la = A.vol[b.x].lev[A.lev], lc = A.vol[b.x].lev[A.lev + 1];
    float* mem = A.vol[b.x].mem;
    if (A.st[b.x].status != ST_RUNNING || !A.st[b.x].mg) return;
    const int nx = la.nx, ny = la.ny, nz = la.nz, cx = lc.nx, cy = lc.ny;
    const unsigned nxy = (unsigned)nx * (unsigned)ny, cxy = (unsigned)cx * (unsigned)cy;
    const float* G = mem + la.off;
    float* S = mem + la.off + la.n;   // t
    const float *FX = S + la.n, *FY = FX + la.n, *FZ = FY + la.n, *IV = FZ + la.n;
    float* GC = mem + lc.off;         // next level: g (down), t (up)
    const float* E = GC + lc.n;
    const int tx = (cx + TK - 1) / TK, ty = (ny + TY - 1) / TY;
    const int k0 = (b.y % tx) * TK, y0 = ((b.y / tx) % ty) * TY, z0 = (b.y / (tx * ty)) * A.tz;
    const int z1 = min(z0 + A.tz, nz);
    const int tid = (int)threadIdx.x;
    const bool has = tid < PW * PH;
    const int ck = tid % PW, cr = tid / PW;
    const int k = k0 - 1 + ck, y = y0 - 2 + cr;
    const bool inb = has && k >= 0 && k < cx && y >= 0 && y < ny;
    const bool ok0 = inb && 2 * k < nx, ok1 = inb && 2 * k + 1 < nx;
    const bool mid = has && cr >= 1 && cr <= TY + 2;                               // black values are formed here
    const bool own = has && ck >= 1 && ck <= TK && cr >= 2 && cr < TY + 2;
    // place in LDS, with a row of padding on either side; threads without a pair write the spare place
    const int at = has ? PW + 1 + tid : PW * (PH + 2) + 1, rd = has ? at : PW + 1;
    const unsigned col = inb ? 2u * (unsigned)k + (unsigned)nx * (unsigned)y : 0u;
    const unsigned colx = inb && k > 0 ? col - 1u : 0u, coly = inb && y > 0 ? col - (unsigned)nx : 0u;
    const unsigned ccol = inb ? (unsigned)k + (unsigned)cx * (unsigned)(y >> 1) : 0u;
    auto plane = [&](int z) { return (unsigned)min(max(z, 0), nz - 1) * nxy; };
    // both cells of the pair on one plane (the second one of a row's last pair may be the next value
    // in memory: it is never used)
    struct Pair {
        Float2 g, iv, fx, fy, fz, ym;
        float xm, e;
    };
    Pair ring[4];   // planes t - 1 .. t + 2
    auto load = [&](Pair& q, int z) {
        const unsigned o = plane(z);
        q.g = ld2(G + o, col);
        q.iv = ld2(IV + o, col);
        q.fx = ld2(FX + o, col);
        q.fy = ld2(FY + o, col);
        q.fz = ld2(FZ + o, col);
        q.ym = ld2(FY + o, coly);
        q.xm = FX[o + colx];
        if (UP) q.e = E[(unsigned)(min(max(z, 0), nz - 1) >> 1) * cxy + ccol];
    };
    // by masks: a choice between two fields becomes an access with a computed address, in scratch memory
    auto pick = [](Float2 v, int s) {
        const unsigned m = 0u - (unsigned)s;
        return __uint_as_float((__float_as_uint(v.x) & ~m) | (__float_as_uint(v.y) & m));
    };
    auto ok = [&](int s) { return s ? ok1 : ok0; };
    // value of the red cell of plane z, at parity s
    auto red_value = [&](const Pair& q, int z, int s) {
        const float g = pick(q.g, s), iv = pick(q.iv, s);
        const float v = UP ? fmaf(g, iv, q.e) : g * iv;
        return ok(s) && (unsigned)z < (unsigned)nz ? v : 0.0f;
    };
    // sum of face times neighbour of the cell at parity s of plane z; zm: faces of plane z - 1
    auto dot = [&](const Pair& q, const Float2& zm, int z, int s, const float (&u)[6]) {
        const float xm = k > 0 ? q.xm : 0.0f;
        const float f[6] = {pick(Float2{xm, q.fx.x}, s), pick(q.fx, s), y > 0 ? pick(q.ym, s) : 0.0f, pick(q.fy, s),
                            z > 0 ? pick(zm, s) : 0.0f, pick(q.fz, s)};
        return mg_dot(f, u);
    };
    const int t0 = z0 - 1;
    load(ring[3], t0 - 1);
    load(ring[0], t0);
    load(ring[1], t0 + 1);
    const int sy = (1 + y) & 1;   // parity of the row's black cells in even planes
    float wm = red_value(ring[3], t0 - 1, sy ^ (t0 & 1)), w0 = red_value(ring[0], t0, 1 ^ sy ^ (t0 & 1));
    float bm = 0.0f, b1 = 0.0f;   // black values of planes t - 2 and t - 1 in this column
    float hold = 0.0f;            // down: the pair of planes' first sum
    auto step = [&](auto J, int t) {
        constexpr int j = decltype(J)::value, jm = (j + 3) % 4, jp = (j + 1) % 4, jn = (j + 2) % 4;
        const int s = sy ^ (t & 1);
        const Float2 zz = ring[jn].fz;   // plane t - 2
        load(ring[jn], t + 2);
        const float wp = red_value(ring[jp], t + 1, s);
        wbuf[t & 1][at] = w0;
        __syncthreads();
        const float* w = wbuf[t & 1] + rd;
        float bv;
        {
            const float u[6] = {w[s - 1], w[s], w[-PW], w[PW], wm, wp};
            bv = (pick(ring[j].g, s) + dot(ring[j], ring[jm].fz, t, s, u)) * pick(ring[j].iv, s);
            bv = mid && ok(s) && (unsigned)t < (unsigned)nz ? bv : 0.0f;
        }
        bbuf[t & 1][at] = bv;
        const int tq = t - 1;
        float d = 0.0f;
        if (own && ok(s) && tq >= z0) {
            const float* bl = bbuf[(t & 1) ^ 1] + rd;
            const float u[6] = {bl[s - 1], bl[s], bl[-PW], bl[PW], bm, bv};
            d = dot(ring[jm], zz, tq, s, u);
        }
        if (UP) {
            if (own && ok(s)) {
                if (t >= z0 && t < z1) S[plane(t) + col + (unsigned)s] = bv;
                if (tq >= z0) S[plane(tq) + col + (unsigned)s] = (pick(ring[jm].g, s) + d) * pick(ring[jm].iv, s);
            }
        } else if (tq >= z0) {
            const int o = tq - z0;
            if (o & 1) {   // the pair of planes is complete: odd rows hand theirs over
                hold += d;
                if (own && (cr & 1)) rows[(o >> 1) & 1][(cr - 2) >> 1][ck - 1] = hold;
            } else {
                if (o >= 2 && own && !(cr & 1) && inb)   // after the barrier: the previous pair
                    GC[(unsigned)((tq - 2) >> 1) * cxy + ccol] = hold + rows[((o >> 1) - 1) & 1][(cr - 2) >> 1][ck - 1];
                hold = d;
            }
        }
        wm = w0;
        w0 = wp;
        bm = b1;
        b1 = bv;
    };
    for (int t = t0;; t += 4)
        if (ring_turn<0, 4, 4>(step, t, z1)) break;
    if (UP) return;
    const int ol = z1 - 1 - z0;   // the last pair (one plane at the end of an odd level)
    if (own && (cr & 1) && !(ol & 1)) rows[(ol >> 1) & 1][(cr - 2) >> 1][ck - 1] = hold;
    __syncthreads();
    if (own && !(cr & 1) && inb)
        GC[(unsigned)((z1 - 1) >> 1) * cxy + ccol] = hold + rows[(ol >> 1) & 1][(cr - 2) >> 1][ck - 1];
}

// The levels from `bottom` on, one block per volume, in LDS: one V-cycle with two sweeps before
// and after each correction; the last level (at most 64 cells) is solved with its inverse.  t
// holds the iterate u.  (Two sweeps here save 3-15% of the CG's iterations at no further launches.
// A second V-cycle on the first one's residual saves as many, but 2 B - B A B is indefinite
// where the cycle overcorrects, as in long clogged volumes.)
// Bound by the chain of phases (a phase is one half sweep and a barrier, about 0.4 us): 16^3 cells
// took 26 us with levels down to one cell, integer divisions and level data read from memory in
// every phase; now eight phases a level, two levels and one product take 18 us.
constexpr int kMgBottomThreads = 1024;

struct LdsLev {
    int nx, ny, nz, cx, cy, n, nc;
    unsigned mx, my;   // ceil(2^32 / cx), ceil(2^32 / cy): exact quotients for the cells kept here
    float *g, *t, *fx, *fy, *fz, *iv, *gc, *tc;
};

__device__ __forceinline__ MgCell lds_cell(const LdsLev& q, unsigned C, int j, int colour) {
    const unsigned row = q.cx == 1 ? C : __umulhi(C, q.mx);
    const int K = (int)(C - row * (unsigned)q.cx);
    const unsigned Zu = q.cy == 1 ? row : __umulhi(row, q.my);
    const int Z = (int)Zu, Y = (int)(row - Zu * (unsigned)q.cy);
    MgCell c;
    c.y = 2 * Y + (j & 1);
    c.z = 2 * Z + (j >> 1);
    c.x = 2 * K + ((colour + c.y + c.z) & 1);
    c.ok = c.x < q.nx && c.y < q.ny && c.z < q.nz;
    c.i = (unsigned)c.x + (unsigned)q.nx * ((unsigned)c.y + (unsigned)q.ny * (unsigned)c.z);
    return c;
}

__global__ __launch_bounds__(kMgBottomThreads) void k_mg_bottom(RbLaunch L, MgLaunch M) {
    __shared__ float sm[kMgArrays][kMgBottomCells];
    __shared__ MgLevel sl[kMgLevels];
    const int v = M.vols[blockIdx.x];
    if (L.st[v].status != ST_RUNNING || !L.st[v].mg) return;
    const MgDesc& d = M.vol[v];
    const int tid = (int)threadIdx.x;
    const int b = d.bottom, last = d.nlev - 1;
    float* mem = d.mem;
    // row tid / 16 of the last level's inverse (64 x 64, padded with zeros), columns 4 (tid % 16) ..
    const float4 inv = reinterpret_cast<const float4*>(mem + d.inv_off)[tid];
    if (tid >= b && tid <= last) sl[tid] = d.lev[tid];
    __syncthreads();
    // cells of a level start at its offset from the bottom level (all arrays alike)
    const unsigned off_b = sl[b].off;
    auto lds_off = [&](int l) { return (int)((sl[l].off - off_b) / kMgArrays); };
    for (int l = b; l <= last; ++l) {
        const int n = sl[l].n, o = lds_off(l);
        const float* src = mem + sl[l].off;
        for (int i = tid; i < n; i += kMgBottomThreads) {
            if (l == b) sm[0][o + i] = src[i];
            if (l < last) {
#pragma unroll
                for (int a = 2; a < kMgArrays; ++a) sm[a][o + i] = src[(long long)a * n + i];
            }
        }
    }
    auto level = [&](int l) {
        LdsLev r;
        const int o = lds_off(l), oc = lds_off(l + 1);
        r.nx = sl[l].nx;
        r.ny = sl[l].ny;
        r.nz = sl[l].nz;
        r.cx = half_up(r.nx);
        r.cy = half_up(r.ny);
        r.mx = 0xFFFFFFFFu / (unsigned)r.cx + 1u;
        r.my = 0xFFFFFFFFu / (unsigned)r.cy + 1u;
        r.n = sl[l].n;
        r.nc = sl[l + 1].n;
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
    // f(cell) for this thread's cells of one colour
    auto cells = [&](const LdsLev& q, int colour, auto f) {
        for (int id = tid; id < 4 * q.nc; id += kMgBottomThreads) {
            const MgCell c = lds_cell(q, (unsigned)id >> 2, id & 3, colour);
            if (c.ok) f(c);
        }
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
        __syncthreads();
    };
    __syncthreads();
    for (int l = b; l < last; ++l) {
        const LdsLev q = level(l);
        // red sweep from zero and the black one after it, at once: the red values are g iv
        cells(q, 0, [&](const MgCell& c) { q.t[c.i] = q.g[c.i] * q.iv[c.i]; });
        cells(q, 1, [&](const MgCell& c) {
            float f[6], u[6];
            unsigned n[6];
            mg_faces(q, c, f, n);
#pragma unroll
            for (int k = 0; k < 6; ++k) u[k] = q.g[n[k]] * q.iv[n[k]];
            q.t[c.i] = (q.g[c.i] + mg_dot(f, u)) * q.iv[c.i];
        });
        __syncthreads();
        sweep(q, 0);
        sweep(q, 1);
        for (int i0 = 0; i0 < 4 * q.nc; i0 += kMgBottomThreads) {   // whole waves: lanes are summed
            const int id = i0 + tid;
            float s = 0.0f;
            if (id < 4 * q.nc) {
                const MgCell c = lds_cell(q, (unsigned)id >> 2, id & 3, 0);
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
    {
        const int n = sl[last].n, o = lds_off(last), c = 4 * (tid & 15);
        const float* g = sm[0] + o;
        float s = inv.x * (c < n ? g[c] : 0.0f);
        s = fmaf(inv.y, c + 1 < n ? g[c + 1] : 0.0f, s);
        s = fmaf(inv.z, c + 2 < n ? g[c + 2] : 0.0f, s);
        s = fmaf(inv.w, c + 3 < n ? g[c + 3] : 0.0f, s);
#pragma unroll
        for (int k = 1; k < 16; k <<= 1) s += __shfl_xor(s, k, 64);
        if ((tid & 15) == 0 && (tid >> 4) < n) sm[1][o + (tid >> 4)] = s;
    }
    __syncthreads();
    for (int l = last - 1; l >= b; --l) {
        const LdsLev q = level(l);
        // black sweep on u_r + e (the red sweep after it replaces u_r, so e is never added there)
        cells(q, 1, [&](const MgCell& c) {
            float f[6], u[6], e[6];
            unsigned n[6];
            mg_faces(q, c, f, n);
            const int px = q.cx, pxy = q.cx * q.cy;
            const int cb = (c.y >> 1) * px + (c.z >> 1) * pxy, base = cb + (c.x >> 1);
            e[0] = q.tc[c.x > 0 ? cb + ((c.x - 1) >> 1) : base];
            e[1] = q.tc[c.x + 1 < q.nx ? cb + ((c.x + 1) >> 1) : base];
            e[2] = q.tc[c.y > 0 && !(c.y & 1) ? base - px : base];
            e[3] = q.tc[c.y + 1 < q.ny && (c.y & 1) ? base + px : base];
            e[4] = q.tc[c.z > 0 && !(c.z & 1) ? base - pxy : base];
            e[5] = q.tc[c.z + 1 < q.nz && (c.z & 1) ? base + pxy : base];
#pragma unroll
            for (int k = 0; k < 6; ++k) u[k] = f[k] != 0.0f ? q.t[n[k]] + e[k] : 0.0f;   // not t of this cell, being written
            q.t[c.i] = (q.g[c.i] + mg_dot(f, u)) * q.iv[c.i];
        });
        __syncthreads();
        sweep(q, 0);
        sweep(q, 1);
        sweep(q, 0);
    }
    const float* u = sm[1];
    for (int i = tid; i < sl[b].n; i += kMgBottomThreads) mem[off_b + (unsigned)sl[b].n + i] = u[i];
}

// r.z of one preconditioned volume, then beta = r.z / (previous r.z).  Where mg_beta ends the cycle the passes of
// this iteration leave the volume alone; x's pending step is in the buffer the cycle did not write.
__global__ __launch_bounds__(kFinThreads) void k_mg_fin(RbLaunch L, MgLaunch M) {
    const int v = M.vols[blockIdx.x];
    VolState<double>* s = L.st + v;
    if (s->status != ST_RUNNING || !s->mg) return;
    const int ntiles = M.vol[v].ntiles, base = M.vol[v].part_base;
    AccDD sum[1];
    sum[0].init();
    for (int i = (int)threadIdx.x; i < ntiles; i += kFinThreads) {
        const double* p = M.part + 2 * ((long long)base + i);
        sum[0].add2(p[0], p[1]);
    }
    __shared__ double red[2];
    block_reduce_store<AccDD, 1, kFinThreads>(sum, red);
    if (threadIdx.x == 0) mg_beta(s, red[0] + red[1]);
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

// Coefficients of the first level from the stencil codes: the faces towards x+, y+, z+ and, in t, the
// cell's half-cell faces on the primary axis.  A code holds its voxel's and its neighbours' solid flags,
// so a cell's own faces and those towards + take its 8 children's codes, and the next cells' inner
// faces 4 codes each: 20 independent byte loads (256^3: 400 us with a loop over the faces on 512
// blocks, 43 us so).
__global__ __launch_bounds__(kMgThreads) void k_mg_coef0(RbLaunch L, MgLaunch M) {
    const int v = M.vols[blockIdx.y];
    const MgDesc& d = M.vol[v];
    const MgLevel a = d.lev[0];
    const RbDesc& rb = L.vol[v];
    const uint8_t* code = rb.code;
    float* g = d.mem + a.off;
    float *t = g + a.n, *fx = t + a.n, *fy = fx + a.n, *fz = fy + a.n;
    const int fn[3] = {rb.nx, rb.ny, rb.nz};
    const int primary = rb.primary;
    const Coef<double> c = L.coef[v];
    const float c0 = (float)c.ci0, c1 = (float)c.ci1, c2 = (float)c.ci2, b0 = (float)c.cb0, b1 = (float)c.cb1;
    const unsigned st[3] = {1u, (unsigned)fn[0], (unsigned)fn[0] * (unsigned)fn[1]};
    // face between voxels of solid flags o and n
    auto face = [&](int o, int n) { return o + n == 0 ? c0 : (o + n == 1 ? c1 : c2); };
    for (unsigned i = blockIdx.x * kMgThreads + threadIdx.x; i < (unsigned)a.n; i += gridDim.x * kMgThreads) {
        const unsigned row = i / (unsigned)a.nx;
        const int I[3] = {(int)(i - row * (unsigned)a.nx), (int)(row % (unsigned)a.ny), (int)(row / (unsigned)a.ny)};
        const unsigned o = 2u * (unsigned)I[0] + 2u * (unsigned)I[1] * st[1] + 2u * (unsigned)I[2] * st[2];
        bool two[3], next[3], wide[3];   // two children; a next cell; two children in the next cell
#pragma unroll
        for (int q = 0; q < 3; ++q) {
            two[q] = 2 * I[q] + 1 < fn[q];
            next[q] = 2 * I[q] + 2 < fn[q];
            wide[q] = 2 * I[q] + 3 < fn[q];
        }
        int ch[8];      // children (bit q of the index: upper along axis q); -1 outside the box
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            const bool in = (!(j & 1) || two[0]) && (!(j & 2) || two[1]) && (!(j & 4) || two[2]);
            const int v8 = code[in ? o + (unsigned)(j & 1) + (unsigned)((j >> 1) & 1) * st[1] + (unsigned)(j >> 2) * st[2] : o];
            ch[j] = in ? v8 : -1;
        }
        float s[3], own[3];
#pragma unroll
        for (int q = 0; q < 3; ++q) {
            const int u = q == 0 ? 1 : 0, w = q == 2 ? 1 : 2;
            float in = 0.0f, m = 0.0f, r = 0.0f;
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const int lo = ((j & 1) << u) | ((j >> 1) << w), hi = lo | (1 << q);
                const unsigned nx = o + 2u * st[q] + (unsigned)(j & 1) * st[u] + (unsigned)(j >> 1) * st[w];
                const int cn = code[next[q] && ch[lo] >= 0 ? nx : o];
                if (two[q] && ch[lo] >= 0) in += face((ch[lo] >> 6) & 1, (ch[lo] >> (2 * q)) & 1);
                if (next[q] && ch[hi] >= 0) m += face((ch[hi] >> 6) & 1, (ch[hi] >> (2 * q)) & 1);
                if (wide[q] && ch[lo] >= 0) r += face((cn >> 6) & 1, (cn >> (2 * q)) & 1);
            }
            own[q] = in;
            s[q] = next[q] ? mg_series(m, in, true, r, wide[q]) : 0.0f;
        }
        // half-cell faces at either end of the primary axis
        float end[2] = {0.0f, 0.0f};
        const int Ip = primary == 0 ? I[0] : (primary == 1 ? I[1] : I[2]), np = primary == 0 ? fn[0] : (primary == 1 ? fn[1] : fn[2]);
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            if (ch[j] < 0) continue;
            const int k = 2 * Ip + ((j >> primary) & 1);
            const float h = (ch[j] >> 6) & 1 ? b1 : b0;
            if (k == 0) end[0] += h;
            if (k == np - 1) end[1] += h;
        }
        const float inner = primary == 0 ? own[0] : (primary == 1 ? own[1] : own[2]);
        const bool tp = 2 * Ip + 1 < np;
        g[i] = 0.0f;
        fx[i] = s[0];
        fy[i] = s[1];
        fz[i] = s[2];
        t[i] = mg_series(end[0], inner, tp, 0.0f, false) + mg_series(end[1], inner, tp, 0.0f, false);
    }
}

// The same of level `lev` >= 1 from level lev - 1.
__global__ __launch_bounds__(kMgThreads) void k_mg_coef(RbLaunch L, MgLaunch M, int lev) {
    const int v = M.vols[blockIdx.y];
    const MgDesc& d = M.vol[v];
    if (lev >= d.nlev) return;
    const MgLevel a = d.lev[lev], p = d.lev[lev - 1];
    const int primary = L.vol[v].primary;
    float* g = d.mem + a.off;
    float *t = g + a.n, *fx = t + a.n, *fy = fx + a.n, *fz = fy + a.n;
    const int fn[3] = {p.nx, p.ny, p.nz};
    const float* pt = d.mem + p.off + p.n;
    const unsigned st[3] = {1u, (unsigned)fn[0], (unsigned)fn[0] * (unsigned)fn[1]};
    for (unsigned i = blockIdx.x * kMgThreads + threadIdx.x; i < (unsigned)a.n; i += gridDim.x * kMgThreads) {
        const unsigned row = i / (unsigned)a.nx;
        const int I[3] = {(int)(i - row * (unsigned)a.nx), (int)(row % (unsigned)a.ny), (int)(row / (unsigned)a.ny)};
        const unsigned o = 2u * (unsigned)I[0] + 2u * (unsigned)I[1] * st[1] + 2u * (unsigned)I[2] * st[2];
        float s[3], own[3];
#pragma unroll
        for (int q = 0; q < 3; ++q) {
            const int u = q == 0 ? 1 : 0, w = q == 2 ? 1 : 2;
            const float* f = pt + (size_t)(q + 1) * p.n;   // faces towards + along q
            const bool two = 2 * I[q] + 1 < fn[q], next = 2 * I[q] + 2 < fn[q], wide = 2 * I[q] + 3 < fn[q];
            float in = 0.0f, m = 0.0f, r = 0.0f;
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const bool ok = 2 * I[u] + (j & 1) < fn[u] && 2 * I[w] + (j >> 1) < fn[w];
                const unsigned b = o + (ok ? (unsigned)(j & 1) * st[u] + (unsigned)(j >> 1) * st[w] : 0u);
                const float f0 = f[b], f1 = f[next ? b + st[q] : b], f2 = f[wide ? b + 2u * st[q] : b];
                in += ok && two ? f0 : 0.0f;
                m += ok && next ? f1 : 0.0f;
                r += ok && wide ? f2 : 0.0f;
            }
            own[q] = in;
            s[q] = next ? mg_series(m, in, true, r, wide) : 0.0f;
        }
        // half-cell faces at either end of the primary axis (one cell along it: both ends together)
        const int Ip = primary == 0 ? I[0] : (primary == 1 ? I[1] : I[2]), np = primary == 0 ? fn[0] : (primary == 1 ? fn[1] : fn[2]);
        float end[2] = {0.0f, 0.0f};
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            const bool ok = 2 * I[0] + (j & 1) < fn[0] && 2 * I[1] + ((j >> 1) & 1) < fn[1] && 2 * I[2] + (j >> 2) < fn[2];
            const int k = 2 * Ip + ((j >> primary) & 1);
            if (!ok || (k != 0 && k != np - 1)) continue;
            end[k == 0 ? 0 : 1] += pt[o + (unsigned)(j & 1) + (unsigned)((j >> 1) & 1) * st[1] + (unsigned)(j >> 2) * st[2]];
        }
        const float inner = primary == 0 ? own[0] : (primary == 1 ? own[1] : own[2]);
        const bool tp = 2 * Ip + 1 < np;
        g[i] = 0.0f;
        fx[i] = s[0];
        fy[i] = s[1];
        fz[i] = s[2];
        t[i] = mg_series(end[0], inner, tp, 0.0f, false) + mg_series(end[1], inner, tp, 0.0f, false);
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

// Inverse of the last level's matrix (-A, at most 64 cells), by Gauss-Jordan elimination without
// pivoting (the matrix is symmetric and positive definite), stored 64 x 64 with zeros around.
// Cells cut off from both ends (a phase without conductivity) leave a pivot of rounding size: that
// row and column are left at zero, which keeps the product symmetric and positive semi-definite.
constexpr int kMgInv = 64;
__global__ __launch_bounds__(kMgBottomThreads) void k_mg_inv(MgLaunch M) {
    __shared__ double a[kMgInv][kMgInv + 1], least[kMgInv];
    const MgDesc& d = M.vol[M.vols[blockIdx.x]];
    const MgLevel q = d.lev[d.nlev - 1];
    const float* t = d.mem + q.off + q.n;
    const float *fx = t + q.n, *fy = fx + q.n, *fz = fy + q.n;
    const int tid = (int)threadIdx.x;
    for (int k = tid; k < kMgInv * kMgInv; k += kMgBottomThreads) a[k / kMgInv][k % kMgInv] = 0.0;
    __syncthreads();
    if (tid < q.n) {
        const int x = tid % q.nx, y = (tid / q.nx) % q.ny, z = tid / (q.nx * q.ny);
        double diag = t[tid];
        auto face = [&](bool has, int j, float f) {
            if (!has) return;
            a[tid][j] = -(double)f;
            diag += f;
        };
        face(x + 1 < q.nx, tid + 1, fx[tid]);
        face(x > 0, tid - 1, fx[x > 0 ? tid - 1 : tid]);
        face(y + 1 < q.ny, tid + q.nx, fy[tid]);
        face(y > 0, tid - q.nx, fy[y > 0 ? tid - q.nx : tid]);
        face(z + 1 < q.nz, tid + q.nx * q.ny, fz[tid]);
        face(z > 0, tid - q.nx * q.ny, fz[z > 0 ? tid - q.nx * q.ny : tid]);
        a[tid][tid] = diag;
        least[tid] = 1e-12 * diag;
    }
    __syncthreads();
    const int r = tid >> 4, c0 = 4 * (tid & 15);   // this thread's four elements
    for (int k = 0; k < q.n; ++k) {
        const double p = a[k][k] > least[k] ? 1.0 / a[k][k] : 0.0, f = a[r][k];
        double row[4];
#pragma unroll
        for (int m = 0; m < 4; ++m) row[m] = c0 + m == k ? p : a[k][c0 + m] * p;
        __syncthreads();
#pragma unroll
        for (int m = 0; m < 4; ++m) a[r][c0 + m] = r == k ? row[m] : (c0 + m == k ? 0.0 : a[r][c0 + m]) - f * row[m];
        __syncthreads();
    }
    float* out = d.mem + d.inv_off;
#pragma unroll
    for (int m = 0; m < 4; ++m)
        out[r * kMgInv + c0 + m] = r < q.n && c0 + m < q.n ? (float)a[r][c0 + m] : 0.0f;
}

}  // namespace

// Planes per tile of the fine passes: the fewest plane steps over the rounds of the two blocks a CU
// holds at once, over all volumes of the launch; a tile has a prologue of three planes.  Against two
// blocks per CU for each volume alone, at most 32 planes: 12 volumes of 60^3 to 129^3 11.8 -> 10.4 ms,
// 384^3 30.2 -> 29.7 ms.  The choice is within 2% of the best of a sweep over 2 .. 128 for 64^3 to 384^3.
constexpr int kMgRound = 512;
// The same for a level's tiles of four waves (four blocks on a CU).
constexpr int kMgLevRound = 1024;

bool mg_plan(int nx, int ny, int nz, int primary, MgDesc* d, size_t* floats) {
    *d = MgDesc{};
    *floats = 0;
    const int flow = primary == 0 ? nx : (primary == 1 ? ny : nz);
    if ((long long)nx * ny * nz < kMgMinVoxels || flow < kMgMinFlow) return false;
    int x = nx, y = ny, z = nz;
    size_t off = 0;
    while ((d->nlev == 0 || d->lev[d->nlev - 1].n > kMgInv) && d->nlev < kMgLevels) {
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
    if (d->lev[d->nlev - 1].n > kMgInv) return false;
    off = (off + 3) & ~(size_t)3;   // float4 rows
    d->inv_off = (unsigned)off;
    off += kMgInv * kMgInv;
    int cells = 0;
    d->bottom = d->nlev;
    while (d->bottom > 0 && cells + d->lev[d->bottom - 1].n <= kMgBottomCells) cells += d->lev[--d->bottom].n;
    const size_t elems = (size_t)rb_row_pitch(half_up(nx)) * (size_t)(ny + 2) * (size_t)(nz + 2);
    if (off > 2 * elems) return false;
    d->tiles_x = (half_up(nx) + kRbTX - 1) / kRbTX;
    d->tiles_y = (ny + kMgTY - 1) / kMgTY;
    d->nz = nz;
    *floats = off;
    return true;
}

// The planes per tile with the fewest steps over rounds of `round` blocks; count(tz), most(tz): tiles and
// planes of the deepest one.
template <class C, class D>
static int least_steps(int round, C count, D most) {
    int best = kMgLeastTz;
    long long least = 0;
    for (int tz = kMgLeastTz; tz <= 128; tz += 2) {
        const long long cost = ((count(tz) + round - 1) / round) * (most(tz) + 3);
        if (tz == kMgLeastTz || cost < least) {
            best = tz;
            least = cost;
        }
    }
    return best;
}

int mg_level_tiles(const MgLevel& l, int tz) {
    return ((half_up(l.nx) + kMgLevTK - 1) / kMgLevTK) * ((l.ny + kMgLevTY - 1) / kMgLevTY) * ((l.nz + tz - 1) / tz);
}

int mg_level_tz(const std::vector<MgLevel>& l) {
    auto count = [&](int tz) {
        long long n = 0;
        for (const MgLevel& m : l) n += mg_level_tiles(m, tz);
        return n;
    };
    auto most = [&](int tz) {
        int n = 0;
        for (const MgLevel& m : l) n = std::max(n, std::min(tz, m.nz));
        return n;
    };
    return least_steps(kMgLevRound, count, most);
}

int mg_tile(std::vector<MgDesc>& d, const std::vector<int>& vols) {
    auto count = [&](const MgDesc& m, int tz) { return (long long)m.tiles_x * m.tiles_y * ((m.nz + tz - 1) / tz); };
    auto all = [&](int tz) {
        long long n = 0;
        for (int v : vols) n += count(d[v], tz);
        return n;
    };
    auto most = [&](int tz) {
        int n = 0;
        for (int v : vols) n = std::max(n, std::min(tz, d[v].nz));
        return n;
    };
    const int best = least_steps(kMgRound, all, most);
    int tiles = 0;
    for (int v : vols) {
        MgDesc& m = d[v];
        m.tz = best;
        m.tiles_z = (m.nz + best - 1) / best;
        m.ntiles = (int)count(m, best);
        m.part_base = tiles;
        tiles += m.ntiles;
    }
    return tiles;
}

void cg_state_event(VolState<double>* s, int event, double value) {
    const bool update = s->status == ST_UPDATE || s->status == ST_FRESH;
    if (event == 0 ? !update : s->status != ST_RUNNING) return;
    const double tot[4] = {value, event == 0 ? 1.0 : -value, value, -value};
    if (event == 0)
        mixres_update(s, tot);
    else if (event == 1 && s->mg)
        mg_beta(s, value);
    else if (event == 2)
        fin_update<double, F_CG1>(s, tot);
    else if (event == 3)
        fin_update<double, F_CG2>(s, tot);
}

hipError_t mg_setup(const RbLaunch& L, const MgLaunch& M, hipStream_t s) {
    if (M.nvol <= 0) return hipSuccess;
    auto blocks = [](int cells) { return (unsigned)std::min(32768, std::max(1, (cells + kMgThreads - 1) / kMgThreads)); };
    hipLaunchKernelGGL(k_mg_coef0, dim3(blocks(M.cells[0]), M.nvol), dim3(kMgThreads), 0, s, L, M);
    for (int l = 1; l < M.nlev_max; ++l)
        hipLaunchKernelGGL(k_mg_coef, dim3(blocks(M.cells[l]), M.nvol), dim3(kMgThreads), 0, s, L, M, l);
    hipLaunchKernelGGL(k_mg_diag, dim3(blocks(M.cells[0]), M.nvol), dim3(kMgThreads), 0, s, L, M);
    hipLaunchKernelGGL(k_mg_inv, dim3(M.nvol), dim3(kMgBottomThreads), 0, s, M);
    return hipGetLastError();
}

hipError_t mg_cycle(const RbLaunch& L, const MgLaunch& M, hipStream_t s) {
    const dim3 fb(kRbTX * (kMgTY + 3)), cb(kMgThreads);
    auto args = [&](int l) {
        return MgLevelArgs{L.st, M.vol, M.blocks + M.blk_off[l], M.nblk[l], l, M.lev_tz[l]};
    };
    hipLaunchKernelGGL((k_mg_fine<kMgTY, false>), dim3(M.ntiles), fb, 0, s, L, M);
    for (int l = 0; l < M.nlev; ++l) hipLaunchKernelGGL(k_mg_level<false>, dim3(M.nblk[l]), cb, 0, s, args(l));
    hipLaunchKernelGGL(k_mg_bottom, dim3(M.nvol), dim3(kMgBottomThreads), 0, s, L, M);
    for (int l = M.nlev - 1; l >= 0; --l) hipLaunchKernelGGL(k_mg_level<true>, dim3(M.nblk[l]), cb, 0, s, args(l));
    hipLaunchKernelGGL((k_mg_fine<kMgTY, true>), dim3(M.ntiles), fb, 0, s, L, M);
    hipLaunchKernelGGL(k_mg_fin, dim3(M.nvol), dim3(kFinThreads), 0, s, L, M);
    return hipGetLastError();
}

}  // namespace ft
