// Reactive area density: marching-cubes area of the isovalue level set of a volume.
//
// Reference (`fast alpha`): getReactiveAreaDensity / getReactiveAreaDensityTensor
// (fastlib/src/volume/VolumeMeasures.cpp:294-333) -> getVolumeArea
// (fastlib/src/volume/VolumeSurface.cpp:9-36) -> ___generateTrianglesSurfaceArea
// (fastlib/src/cuda/VolumeSurface.cu:203-258), then Volume::sum of the per-voxel areas.
//
// The reference samples the volume as a linearly filtered, clamped, normalized-coordinate
// uchar texture (fastlib/src/utility/DataPtr.cpp:565-592) at the corners of every voxel
// (VolumeSurface.cu:83-103, positions i/N).  A corner sits on the midpoint between texel
// centres in every axis, so its value is the mean of the 8 voxels around it (indices clamped
// into the volume), byte/255: (sum of the 8 bytes) / 2040, which for a 0/255 volume is k/8
// exactly.  Here those corner values are built from voxel sums instead of texture reads:
// a wave keeps, for its 64x4 tile and the plane being marched, the 2x2 in-plane voxel sums
// of every lattice point (registers) and adds two consecutive planes of them into corner
// counts; lane masks classify a row of cubes from its corner counts, and the cubes that cross
// the level set are queued and triangulated by the whole wave.
//
// Two modes share the march.  MODE 0 reads the volume's bytes (one surface).  MODE 1 reads
// a byte of face bits per voxel (bit f: a pore voxel whose component touches face f; the
// boundary-connected volumes of getReactiveAreaDensityTensor) and carries the six per-face
// counts packed in nibbles, so one pass yields all six surfaces.
//
// Per cube the arithmetic is the reference's float arithmetic, operation by operation and
// without contraction (the file is built with -ffp-contract=off): positions (1/N)*i and
// (1/N)*i + 1/N, vertexInterp / lerp (VolumeSurface.cu:171-178, CudaMath.h:1134-1137),
// triangleArea = 0.5 * length(cross(v1 - v0, v2 - v0)) (VolumeSurface.cu:187-189), the
// sum of all areas in double (VolumeSurface.cu:240-255, per cube in table order, then over the
// volume).  Here the sum of the triangles is double-double with one final rounding, so it does
// not depend on the reduction tree.
#include <hip/hip_runtime.h>
#include <hipcub/hipcub.hpp>

#include <cstdint>
#include <mutex>

#include "mc_table.h"

namespace fta {

constexpr int kTX = 64, kTY = 4, kTZ = 16;   // cubes of a wave's tile (fewer planes in small volumes: mc_tz)

__constant__ uint64_t c_tri[256] = FAST_MC_TRI_WORDS;

// Double-double sum of doubles (TwoSum, then renormalise).
struct DdSum {
    double hi, lo;
    __device__ __forceinline__ void init() { hi = 0.0; lo = 0.0; }
    __device__ __forceinline__ void add2(double p, double e) {
        const double s = hi + p;
        const double v = s - hi;
        double t = (hi - (s - v)) + (p - v);
        t += lo + e;
        hi = s + t;
        lo = t - (hi - s);
    }
};

__device__ __forceinline__ void wave_combine(DdSum& a) {
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
        const double h = __shfl_xor(a.hi, off, 64);
        const double l = __shfl_xor(a.lo, off, 64);
        a.add2(h, l);
    }
}

// Face bits 0..5 of a code byte, one per nibble (bit f at 4 f).
__device__ __forceinline__ uint32_t spread6(uint32_t b) {
    const uint32_t x = (b & 7u) | (b & 0x38u) << 9;   // three bits a half
    return (x | x << 3 | x << 6) & 0x111111u;
}

// Corner coordinates of one cube: X0 = (1/nx) i, X1 = X0 + 1/nx, likewise y and z.
struct CubeGeo {
    float X0, X1, Y0, Y1, Z0, Z1;
};

// vertexInterp along one axis: the other two coordinates of the edge's end points are equal,
// so p0 + t (p1 - p0) leaves them unchanged.
__device__ __forceinline__ float lerp_axis(float iso, float fa, float fb, float A, float B) {
    if (fb == fa) return A;
    const float t = (iso - fa) / (fb - fa);
    return A + t * (B - A);
}

// Vertex on edge e (corners a -> b as in the table's edge list), by cases: used where a
// thread triangulates its own cube (the mesh export).
__device__ __forceinline__ void edge_vertex_switch(unsigned e, const float (&f)[8], const CubeGeo& g, float iso,
                                                   float& x, float& y, float& z) {
    switch (e) {
        case 0: x = lerp_axis(iso, f[0], f[1], g.X0, g.X1); y = g.Y0; z = g.Z0; break;
        case 1: x = g.X1; y = lerp_axis(iso, f[1], f[2], g.Y0, g.Y1); z = g.Z0; break;
        case 2: x = lerp_axis(iso, f[2], f[3], g.X1, g.X0); y = g.Y1; z = g.Z0; break;
        case 3: x = g.X0; y = lerp_axis(iso, f[3], f[0], g.Y1, g.Y0); z = g.Z0; break;
        case 4: x = lerp_axis(iso, f[4], f[5], g.X0, g.X1); y = g.Y0; z = g.Z1; break;
        case 5: x = g.X1; y = lerp_axis(iso, f[5], f[6], g.Y0, g.Y1); z = g.Z1; break;
        case 6: x = lerp_axis(iso, f[6], f[7], g.X1, g.X0); y = g.Y1; z = g.Z1; break;
        case 7: x = g.X0; y = lerp_axis(iso, f[7], f[4], g.Y1, g.Y0); z = g.Z1; break;
        case 8: x = g.X0; y = g.Y0; z = lerp_axis(iso, f[0], f[4], g.Z0, g.Z1); break;
        case 9: x = g.X1; y = g.Y0; z = lerp_axis(iso, f[1], f[5], g.Z0, g.Z1); break;
        case 10: x = g.X1; y = g.Y1; z = lerp_axis(iso, f[2], f[6], g.Z0, g.Z1); break;
        default: x = g.X0; y = g.Y1; z = lerp_axis(iso, f[3], f[7], g.Z0, g.Z1); break;
    }
}

struct Vert {
    float x, y, z;
};

// The vertices on the 12 edges of a cube to ev (stride kTX); t(a, b): the interpolation parameter
// from corner a to corner b.  Edges that the surface does not cut get a value that is never read.
template <class T>
__device__ __forceinline__ void cube_vertices(const CubeGeo& g, Vert* ev, T t) {
    ev[0 * kTX] = Vert{g.X0 + t(0, 1) * (g.X1 - g.X0), g.Y0, g.Z0};
    ev[1 * kTX] = Vert{g.X1, g.Y0 + t(1, 2) * (g.Y1 - g.Y0), g.Z0};
    ev[2 * kTX] = Vert{g.X1 + t(2, 3) * (g.X0 - g.X1), g.Y1, g.Z0};
    ev[3 * kTX] = Vert{g.X0, g.Y1 + t(3, 0) * (g.Y0 - g.Y1), g.Z0};
    ev[4 * kTX] = Vert{g.X0 + t(4, 5) * (g.X1 - g.X0), g.Y0, g.Z1};
    ev[5 * kTX] = Vert{g.X1, g.Y0 + t(5, 6) * (g.Y1 - g.Y0), g.Z1};
    ev[6 * kTX] = Vert{g.X1 + t(6, 7) * (g.X0 - g.X1), g.Y1, g.Z1};
    ev[7 * kTX] = Vert{g.X0, g.Y1 + t(7, 4) * (g.Y0 - g.Y1), g.Z1};
    ev[8 * kTX] = Vert{g.X0, g.Y0, g.Z0 + t(0, 4) * (g.Z1 - g.Z0)};
    ev[9 * kTX] = Vert{g.X1, g.Y0, g.Z0 + t(1, 5) * (g.Z1 - g.Z0)};
    ev[10 * kTX] = Vert{g.X1, g.Y1, g.Z0 + t(2, 6) * (g.Z1 - g.Z0)};
    ev[11 * kTX] = Vert{g.X0, g.Y1, g.Z0 + t(3, 7) * (g.Z1 - g.Z0)};
}

__device__ __forceinline__ float triangle_area(const Vert& a, const Vert& b, const Vert& c) {
    const float ux = b.x - a.x, uy = b.y - a.y, uz = b.z - a.z;
    const float vx = c.x - a.x, vy = c.y - a.y, vz = c.z - a.z;
    const float nx = uy * vz - uz * vy;
    const float ny = uz * vx - ux * vz;
    const float nz = ux * vy - uy * vx;
    return sqrtf(nx * nx + ny * ny + nz * nz) * 0.5f;
}

// Lanes below this one whose bit is set in m.
__device__ __forceinline__ int lanes_below(unsigned long long m) {
    return (int)__builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u));
}

// The value of the lane below (lane 0: `edge`) and above (lane 63: `edge`).
__device__ __forceinline__ uint32_t lane_below(uint32_t v, uint32_t edge) {
    return (uint32_t)__builtin_amdgcn_update_dpp((int)edge, (int)v, 0x138 /* wave_shr:1 */, 0xF, 0xF, false);
}
__device__ __forceinline__ uint32_t lane_above(uint32_t v, uint32_t edge) {
    return (uint32_t)__builtin_amdgcn_update_dpp((int)edge, (int)v, 0x130 /* wave_shl:1 */, 0xF, 0xF, false);
}

// One wave: cubes [x0, x0+64) x [y0, y0+4) x [k0, k0+tz), a lane per cube of a row.  Writes NS
// double-double partials (hi, lo) per wave to part[(block * NS + s) * 2].
// thr: the smallest corner count whose value (count / 2040, or / 8 for face bits) is not
// below the isovalue.  The value is monotone in the count, so "corner inside" is count < thr.
// A lane holds the counts of its cube's two corners in x on every lattice row.  Whether a cube
// has corners on both sides is decided for a row of cubes at once, on lane masks in scalar
// registers; those cubes are appended to a queue in LDS.  64 of them at a time are triangulated, so
// the float work runs on full waves: first a lane per cube puts the 12 edge vertices and its triangles'
// edges into LDS, then a lane per triangle adds its area (a cube has 1 to 5 triangles; a lane that
// walked its cube's list would wait for the longest).  Where all corner counts are multiples of
// 255 (a 0/255 volume; always with face bits) the interpolation parameters come from a table of
// the 9 x 9 pairs, made with the same float operations, instead of 12 divisions.  Nothing is
// shared between waves: there are no barriers.
// Bound by instruction issue, most of it the triangulation (a quarter of the cubes of a porous
// 256^3 volume).  A block of four waves that kept planes and corner counts in LDS, with four
// barriers a layer, took 195 us for 256^3 bytes and 303 us for the faces of 250 x 233 x 241; the
// march in registers with a lane walking its cube's triangles 143 and 240 us; this form 94 and 152 us.
template <int MODE>
__global__ __launch_bounds__(kTX) void k_mc_area(const uint8_t* __restrict__ src, int nx, int ny, int nz, int tz,
                                                 float iso, uint32_t thr, double* __restrict__ part) {
    constexpr int NS = MODE ? 6 : 1;
    constexpr int NW = MODE ? 2 : 1;           // words of a lattice row's corner pair
    constexpr int NR = kTY + 2, NL = kTY + 1;  // voxel rows and lattice rows of a plane
    constexpr int KQ = 2 * kTX - 1;            // a row appends up to 64 to at most 63
    __shared__ Vert EV[12 * kTX];              // edge vertices of the cubes being triangulated
    __shared__ uint32_t TQ[5 * kTX];           // their triangles: three edges | cube << 12 | faces << 18
    __shared__ float TT[81];                   // interpolation parameter between corner values a/8 and b/8, at 9 a + b
    __shared__ uint4 QC[KQ * NW];              // corner counts: (row, plane); MODE 0 both x in a word, MODE 1 one x each
    __shared__ uint32_t QH[KQ];                // lane | row << 6 | layer << 8

    const int lane = threadIdx.x;
    const int x0 = blockIdx.x * kTX, y0 = blockIdx.y * kTY, k0 = blockIdx.z * tz;
    const int k1 = min(k0 + tz, nz);
    const size_t sxy = (size_t)nx * (size_t)ny;
    const float sx = 1.0f / (float)nx, sy = 1.0f / (float)ny, sz = 1.0f / (float)nz;
    const unsigned xm = (unsigned)min(x0 + lane, nx - 1);
    const unsigned xe = (unsigned)(lane == kTX - 1 ? min(x0 + kTX, nx - 1) : max(x0 - 1, 0));
    const unsigned long long cols = __ballot(x0 + lane < nx);

    uint32_t vm[NR], ve[NR];                   // the plane in flight: the lane's voxels, those beside the tile
    auto load_plane = [&](int z) {
        const uint8_t* plane = src + sxy * (size_t)z;
#pragma unroll
        for (int r = 0; r < NR; ++r) {
            const uint8_t* row = plane + (size_t)nx * (size_t)min(max(y0 - 1 + r, 0), ny - 1);
            vm[r] = row[xm];
            ve[r] = row[xe];
        }
    };
    // 2x2 in-plane sums at the lattice rows, for the lane's two corners in x
    struct Pair {
        uint32_t w[NW];
    };
    auto plane_sums = [&](Pair (&t)[NL]) {
        Pair h[NR];
#pragma unroll
        for (int r = 0; r < NR; ++r) {
            const uint32_t v = MODE ? spread6(vm[r]) : vm[r], e = MODE ? spread6(ve[r]) : ve[r];
            const uint32_t lo = v + lane_below(v, e), hi = v + lane_above(v, e);
            if constexpr (MODE == 0) {
                h[r].w[0] = lo | hi << 16;
            } else {
                h[r].w[0] = lo;
                h[r].w[1] = hi;
            }
        }
#pragma unroll
        for (int r = 0; r < NL; ++r)
#pragma unroll
            for (int i = 0; i < NW; ++i) t[r].w[i] = h[r].w[i] + h[r + 1].w[i];
    };
    auto add = [](Pair (&c)[NL], const Pair (&a)[NL], const Pair (&b)[NL]) {
#pragma unroll
        for (int r = 0; r < NL; ++r)
#pragma unroll
            for (int i = 0; i < NW; ++i) c[r].w[i] = a[r].w[i] + b[r].w[i];
    };
    // Lane masks of a lattice row whose combination tells which cubes may hold a surface.
    //   MODE 0: any / all of the lane's two corners inside.
    //   MODE 1: the two corners differ; the row differs from the next one.
    struct Mask {
        unsigned long long a, b;
    };
    auto masks = [&](const Pair (&c)[NL], Mask (&m)[NL]) {
#pragma unroll
        for (int r = 0; r < NL; ++r) {
            if constexpr (MODE == 0) {
                const unsigned long long p = __ballot((c[r].w[0] & 0xFFFFu) < thr), q = __ballot(c[r].w[0] < thr << 16);
                m[r].a = p | q;
                m[r].b = p & q;
            } else {
                m[r].a = __ballot(c[r].w[0] != c[r].w[1]);
                m[r].b = r + 1 < NL ? __ballot(c[r].w[0] != c[r + 1 < NL ? r + 1 : r].w[0]) : 0ull;
            }
        }
    };

    DdSum acc[NS];
#pragma unroll
    for (int s = 0; s < NS; ++s) acc[s].init();

    DdSum whole;   // MODE 1: triangles of all six surfaces
    whole.init();
    for (int i = lane; i < 81; i += kTX) {
        const float fa = (float)(i / 9) / 8.0f, fb = (float)(i % 9) / 8.0f;
        TT[i] = fb == fa ? 0.0f : (iso - fa) / (fb - fa);
    }

    // Add the areas of the triangles of this lane's cube (corner pattern ci; ci = 0: none), whose vertices
    // are in EV, to the surfaces `faces`.  Called by all lanes.
    auto triangles = [&](unsigned ci, uint32_t faces) {
        const uint64_t w = c_tri[ci];
        const unsigned ntri = (unsigned)(w >> 60);
        const unsigned long long b0 = __ballot(ntri & 1u), b1 = __ballot(ntri & 2u), b2 = __ballot(ntri & 4u);
        const int at = lanes_below(b0) + 2 * lanes_below(b1) + 4 * lanes_below(b2);
        const int total = (int)__popcll(b0) + 2 * (int)__popcll(b1) + 4 * (int)__popcll(b2);
        const uint32_t tag = (uint32_t)lane << 12 | faces << 18;
#pragma unroll
        for (unsigned j = 0; j < 5; ++j)
            if (j < ntri) TQ[at + (int)j] = ((uint32_t)(w >> (12 * j)) & 0xFFFu) | tag;
        __syncthreads();   // one wave: orders its LDS accesses
        for (int i = lane; i < total; i += kTX) {
            const uint32_t q = TQ[i];
            const Vert* ev = EV + ((q >> 12) & 63u);
            const float area = triangle_area(ev[(q & 15u) * kTX], ev[((q >> 4) & 15u) * kTX], ev[((q >> 8) & 15u) * kTX]);
            if constexpr (MODE == 0) {
                acc[0].add2((double)area, 0.0);
            } else {
                const uint32_t fm = q >> 18;
                if (fm == 63u) {
                    whole.add2((double)area, 0.0);
                } else {
#pragma unroll
                    for (int s = 0; s < NS; ++s)
                        if ((fm >> s) & 1u) acc[s].add2((double)area, 0.0);
                }
            }
        }
        __syncthreads();
    };

    // Triangulate the cubes of queue entries q (one per lane; `has`: the lane has one).  Called by all lanes.
    auto process = [&](int q, bool has) {
        const uint32_t h = has ? QH[q] : 0u;
        CubeGeo g;
        g.Z0 = sz * (float)(k0 + (int)(h >> 8));
        g.Z1 = g.Z0 + sz;
        g.X0 = sx * (float)(x0 + (int)(h & 63u));
        g.X1 = g.X0 + sx;
        g.Y0 = sy * (float)(y0 + (int)((h >> 6) & 3u));
        g.Y1 = g.Y0 + sy;
        // corner m of the table: x of (0 1 1 0), row of (0 0 1 1), plane m / 4
        constexpr int kX[4] = {0, 1, 1, 0}, kY[4] = {0, 0, 1, 1};
        uint32_t w[NW][4] = {}, c[8];
        if (has) {
#pragma unroll
            for (int j = 0; j < NW; ++j) {
                const uint4 v = QC[q * NW + j];
                w[j][0] = v.x;
                w[j][1] = v.y;
                w[j][2] = v.z;
                w[j][3] = v.w;
            }
        }
#pragma unroll
        for (int m = 0; m < 8; ++m) {
            const int x = kX[m & 3], i = 2 * (m >> 2) + kY[m & 3];
            c[m] = MODE ? w[x * (NW - 1)][i] : (x ? w[0][i] >> 16 : w[0][i] & 0xFFFFu);
        }
        if constexpr (MODE == 0) {
            unsigned ci = 0;
            uint32_t k[8], odd = 0;
#pragma unroll
            for (int m = 0; m < 8; ++m) {
                ci |= (c[m] < thr ? 1u : 0u) << m;
                k[m] = (c[m] * 257u + 8u) >> 16;   // c / 255 where that is whole
                odd |= c[m] ^ (k[m] * 255u);
            }
            if (__ballot(odd != 0u) == 0ull) {
                cube_vertices(g, EV + lane, [&](int a, int b) { return TT[9u * k[a] + k[b]]; });
            } else {
                float f[8];
#pragma unroll
                for (int m = 0; m < 8; ++m) f[m] = (float)c[m] / 2040.0f;
                cube_vertices(g, EV + lane, [&](int a, int b) { return (iso - f[a]) / (f[b] - f[a]); });
            }
            triangles(has ? ci : 0u, 0u);
        } else {
            // faces with corners on both sides, at bit 4 f + 3: a nibble n <= 8 has n + 8 - thr >= 8
            // where n >= thr (1 <= thr <= 8; otherwise all corners are on one side)
            uint32_t any = 0, all = ~0u;
#pragma unroll
            for (int m = 0; m < 8; ++m) {
                const uint32_t o = c[m] + (8u - thr) * 0x111111u;
                any |= o;
                all &= o;
            }
            uint32_t rest = has && thr >= 1u && thr <= 8u ? any & ~all & 0x888888u : 0u;
            // faces with equal counts have the same triangles (usually all six share the pore space
            // here): one triangulation for the first of the rest and its equals
            while (__ballot(rest != 0u) != 0ull) {
                const int s4 = rest ? (__ffs((int)rest) - 1) & ~3 : 0;
                uint32_t diff = 0, k[8];
                unsigned ci = 0;
#pragma unroll
                for (int m = 0; m < 8; ++m) {
                    k[m] = (c[m] >> s4) & 15u;
                    diff |= c[m] ^ (k[m] * 0x111111u);
                    ci |= (k[m] < thr ? 1u : 0u) << m;
                }
                const uint32_t same = rest & ~(((diff & 0x777777u) + 0x777777u) | diff);
                uint32_t faces = 0;
#pragma unroll
                for (int s = 0; s < 6; ++s) faces |= (same >> (3 * s + 3)) & (1u << s);
                cube_vertices(g, EV + lane, [&](int a, int b) { return TT[9u * k[a] + k[b]]; });
                triangles(rest ? ci : 0u, faces);
                rest &= ~same;
            }
        }
    };

    // Corner counts of lattice plane k0: voxel planes k0 - 1 and k0 (clamped).
    Pair sum[NL], below[NL], above[NL];
    Mask mb[NL], ma[NL];
    load_plane(max(k0 - 1, 0));
    plane_sums(below);
    load_plane(k0);
    plane_sums(sum);
    add(below, below, sum);
    masks(below, mb);
    load_plane(min(k0 + 1, nz - 1));
    int n = 0;   // queued cubes (uniform)
    for (int k = k0; k < k1; ++k) {
        Pair next[NL];
        plane_sums(next);
        load_plane(min(k + 2, nz - 1));   // in flight while this layer is worked on
        add(above, sum, next);
        masks(above, ma);
        unsigned long long surf[kTY], some = 0ull;
#pragma unroll
        for (int r = 0; r < kTY; ++r) {
            if constexpr (MODE == 0) {
                surf[r] = (mb[r].a | mb[r + 1].a | ma[r].a | ma[r + 1].a) & ~(mb[r].b & mb[r + 1].b & ma[r].b & ma[r + 1].b);
            } else {
                surf[r] = mb[r].a | mb[r + 1].a | ma[r].a | ma[r + 1].a | mb[r].b | ma[r].b |
                          __ballot(below[r].w[0] != above[r].w[0]);
            }
            surf[r] = y0 + r < ny ? surf[r] & cols : 0ull;
            some |= surf[r];
        }
        if (some != 0ull) {
#pragma unroll
            for (int r = 0; r < kTY; ++r) {
                const unsigned long long m = surf[r];
                if (m == 0ull) continue;
                if ((m >> lane) & 1ull) {
                    const int slot = n + lanes_below(m);
#pragma unroll
                    for (int j = 0; j < NW; ++j)
                        QC[slot * NW + j] = uint4{below[r].w[j], below[r + 1].w[j], above[r].w[j], above[r + 1].w[j]};
                    QH[slot] = (uint32_t)lane | (uint32_t)r << 6 | (uint32_t)(k - k0) << 8;
                }
                n += (int)__popcll(m);
                if (n >= kTX) {
                    __syncthreads();   // one wave: orders its LDS accesses
                    n -= kTX;
                    process(n + lane, true);
                }
            }
        }
#pragma unroll
        for (int r = 0; r < NL; ++r) {
            below[r] = above[r];
            sum[r] = next[r];
            mb[r] = ma[r];
        }
    }
    __syncthreads();
    process(lane, lane < n);

    const size_t blk = ((size_t)blockIdx.z * gridDim.y + blockIdx.y) * gridDim.x + blockIdx.x;
#pragma unroll
    for (int s = 0; s < NS; ++s) {
        if constexpr (MODE == 1) acc[s].add2(whole.hi, whole.lo);
        wave_combine(acc[s]);
        if (lane == 0) {
            part[(blk * NS + s) * 2] = acc[s].hi;
            part[(blk * NS + s) * 2 + 1] = acc[s].lo;
        }
    }
}

// One block per surface: sum that surface's nblk block partials in a fixed order.
constexpr int kFinalThreads = 1024;
__global__ __launch_bounds__(kFinalThreads) void k_mc_final(const double* __restrict__ part, size_t nblk, int ns,
                                                            double* __restrict__ out) {
    __shared__ double red[kFinalThreads / 64][2];
    const int s = blockIdx.x, tid = threadIdx.x;
    DdSum a;
    a.init();
#pragma unroll 4
    for (size_t b = tid; b < nblk; b += kFinalThreads) a.add2(part[(b * ns + s) * 2], part[(b * ns + s) * 2 + 1]);
    wave_combine(a);
    if ((tid & 63) == 0) {
        red[tid >> 6][0] = a.hi;
        red[tid >> 6][1] = a.lo;
    }
    __syncthreads();
    if (tid == 0) {
        DdSum t;
        t.init();
        for (int q = 0; q < kFinalThreads / 64; ++q) t.add2(red[q][0], red[q][1]);
        out[s] = t.hi + t.lo;
    }
}

// Scratch of the allocation-free whole-volume area (fast_alpha_area_noalloc): the block
// partials (2 doubles per block of k_mc_area<0>) followed by the result (1 double).  Every
// block writes its own partial and k_mc_final writes the result, so nothing in it needs to
// start at zero.  One copy per device, held until the process ends; calls that overlap on one
// device share it.
constexpr size_t kScratchDoubles = (size_t)1 << 17;   // 1 MiB
static __device__ __align__(256) double scratch[kScratchDoubles];

size_t mc_scratch_doubles() { return kScratchDoubles; }

// Device address of `scratch` on `device` (the current device): looked up with
// hipGetSymbolAddress on the first call for that device and kept.  Host code uses only this
// address; the array's name is not a device address in host code.
hipError_t mc_scratch_address(int device, double** out) {
    constexpr int kMaxDevices = 64;
    static std::mutex mu;
    static double* addr[kMaxDevices] = {};
    if (device < 0 || device >= kMaxDevices) return hipErrorInvalidDevice;
    std::lock_guard<std::mutex> lk(mu);
    if (!addr[device]) {
        void* p = nullptr;
        const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (e != hipSuccess) return e;
        addr[device] = (double*)p;
    }
    *out = addr[device];
    return hipSuccess;
}

// Planes of a tile.  A CU holds 12 waves (their LDS), so few tall tiles end in a nearly empty round; each
// tile reads two planes more than it has.  Measured with 16, 8 and 4 planes: 400 x 300 x 350 (11550
// tiles of 16) 240, 244, 268 us a call; 256^3 (4096) 126, 116, 122; 100 x 120 x 90 (360) 57, 50, 40.
static int mc_tz(int nx, int ny, int nz) {
    const size_t n = (size_t)((nx + kTX - 1) / kTX) * (size_t)((ny + kTY - 1) / kTY) * (size_t)((nz + kTZ - 1) / kTZ);
    return n >= 8192 ? kTZ : (n >= 2048 ? kTZ / 2 : kTZ / 4);
}

// Grid of the area kernel for an nx x ny x nz volume.
dim3 mc_grid(int nx, int ny, int nz) {
    const int tz = mc_tz(nx, ny, nz);
    return dim3((unsigned)((nx + kTX - 1) / kTX), (unsigned)((ny + kTY - 1) / kTY), (unsigned)((nz + tz - 1) / tz));
}

// The grid's y and z extents stay within the launch limit (65535).
bool mc_fits(int nx, int ny, int nz) {
    const dim3 g = mc_grid(nx, ny, nz);
    return g.y <= 65535u && g.z <= 65535u;
}

size_t mc_blocks(int nx, int ny, int nz) {
    const dim3 g = mc_grid(nx, ny, nz);
    return (size_t)g.x * g.y * g.z;
}

// Areas of `src` (an nx x ny x nz volume): MODE 0 one surface of the bytes, MODE 1 six
// surfaces of face bits.  part: mc_blocks() * NS * 2 doubles; out: NS doubles (device).
hipError_t mc_area(const uint8_t* src, int nx, int ny, int nz, float iso, int faces, double* part, double* out,
                   hipStream_t s) {
    const dim3 grid = mc_grid(nx, ny, nz);
    const int tz = mc_tz(nx, ny, nz);
    const size_t nblk = mc_blocks(nx, ny, nz);
    // first count whose value is not below iso (the same float division as the kernels)
    const uint32_t maxc = faces ? 8u : 2040u;
    const float div = faces ? 8.0f : 2040.0f;
    uint32_t thr = 0;
    while (thr <= maxc && (float)thr / div < iso) ++thr;
    if (faces) {
        hipLaunchKernelGGL(k_mc_area<1>, grid, dim3(kTX), 0, s, src, nx, ny, nz, tz, iso, thr, part);
        hipLaunchKernelGGL(k_mc_final, dim3(6), dim3(kFinalThreads), 0, s, part, nblk, 6, out);
    } else {
        hipLaunchKernelGGL(k_mc_area<0>, grid, dim3(kTX), 0, s, src, nx, ny, nz, tz, iso, thr, part);
        hipLaunchKernelGGL(k_mc_final, dim3(1), dim3(kFinalThreads), 0, s, part, nblk, 1, out);
    }
    return hipGetLastError();
}

// ---------------------------------------------------------------------------------------
// Triangle mesh for the OBJ export (`fast alpha --mesh`, AlphaModule.h:145-167): the volume
// padded with one zero voxel per side (Volume::withZeroPadding), marching cubes over the
// padded grid with output positions in a box centred at the origin, spacing 1/maxDim
// (getVolumeAreaMesh, VolumeSurface.cpp:39-74; ___generateTriangles, VolumeSurface.cu:260-357).
// Triangles are emitted in linear cube order, then table order, as the reference's compaction
// by exclusive scan orders them.
// ---------------------------------------------------------------------------------------
namespace {

__global__ __launch_bounds__(256) void k_pad(const uint8_t* __restrict__ src, int nx, int ny, int nz,
                                             uint8_t* __restrict__ dst) {
    const int px = nx + 2, py = ny + 2, pz = nz + 2;
    const long long n = (long long)px * py * pz;
    for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (long long)gridDim.x * blockDim.x) {
        const int x = (int)(i % px), y = (int)((i / px) % py), z = (int)(i / ((long long)px * py));
        const bool inside = x >= 1 && x <= nx && y >= 1 && y <= ny && z >= 1 && z <= nz;
        dst[i] = inside ? src[(size_t)(x - 1) + (size_t)nx * ((size_t)(y - 1) + (size_t)ny * (size_t)(z - 1))] : 0;
    }
}

// Byte sums of the 8 clamped voxels around each corner of cube (x, y, z) of an r0 x r1 x r2 volume.
__device__ __forceinline__ void corner_sums(const uint8_t* v, int r0, int r1, int r2, int x, int y, int z,
                                            uint32_t (&c)[8]) {
    const int dx[8] = {0, 1, 1, 0, 0, 1, 1, 0}, dy[8] = {0, 0, 1, 1, 0, 0, 1, 1}, dz[8] = {0, 0, 0, 0, 1, 1, 1, 1};
#pragma unroll
    for (int m = 0; m < 8; ++m) {
        uint32_t s = 0;
#pragma unroll
        for (int k = -1; k <= 0; ++k)
#pragma unroll
            for (int j = -1; j <= 0; ++j)
#pragma unroll
                for (int i = -1; i <= 0; ++i) {
                    const int a = min(max(x + dx[m] + i, 0), r0 - 1);
                    const int b = min(max(y + dy[m] + j, 0), r1 - 1);
                    const int cc = min(max(z + dz[m] + k, 0), r2 - 1);
                    s += v[(size_t)a + (size_t)r0 * ((size_t)b + (size_t)r1 * (size_t)cc)];
                }
        c[m] = s;
    }
}

__global__ __launch_bounds__(256) void k_mesh_count(const uint8_t* __restrict__ v, int r0, int r1, int r2,
                                                    uint32_t thr, uint32_t* __restrict__ count) {
    const long long n = (long long)r0 * r1 * r2;
    for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (long long)gridDim.x * blockDim.x) {
        const int x = (int)(i % r0), y = (int)((i / r0) % r1), z = (int)(i / ((long long)r0 * r1));
        uint32_t c[8];
        corner_sums(v, r0, r1, r2, x, y, z, c);
        unsigned in = 0;
#pragma unroll
        for (int m = 0; m < 8; ++m) in |= (c[m] < thr ? 1u : 0u) << m;
        count[i] = 3u * (uint32_t)(c_tri[in] >> 60);
    }
}

// out: 6 floats per vertex (position, then the triangle's normal), at 6 * offset[cube].
__global__ __launch_bounds__(256) void k_mesh_emit(const uint8_t* __restrict__ v, int r0, int r1, int r2, float iso,
                                                   const uint32_t* __restrict__ count,
                                                   const uint64_t* __restrict__ offset, float* __restrict__ out) {
    const long long n = (long long)r0 * r1 * r2;
    const float tvs = 1.0f / (float)max(r0, max(r1, r2));   // params.dx = dy = dz = 1 / maxDim
    const float hx = 0.5f * (tvs * (float)r0), hy = 0.5f * (tvs * (float)r1), hz = 0.5f * (tvs * (float)r2);
    for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (long long)gridDim.x * blockDim.x) {
        if (count[i] == 0) continue;
        const int x = (int)(i % r0), y = (int)((i / r0) % r1), z = (int)(i / ((long long)r0 * r1));
        uint32_t c[8];
        corner_sums(v, r0, r1, r2, x, y, z, c);
        float f[8];
#pragma unroll
        for (int m = 0; m < 8; ++m) f[m] = (float)c[m] / 2040.0f;
        unsigned ci = 0;
#pragma unroll
        for (int m = 0; m < 8; ++m) ci |= (f[m] < iso ? 1u : 0u) << m;
        CubeGeo g;
        g.X0 = tvs * (float)x - hx;
        g.X1 = g.X0 + tvs;
        g.Y0 = tvs * (float)y - hy;
        g.Y1 = g.Y0 + tvs;
        g.Z0 = tvs * (float)z - hz;
        g.Z1 = g.Z0 + tvs;
        const uint64_t w = c_tri[ci];
        const int ntri = min((int)(w >> 60), (int)(count[i] / 3u));   // never beyond the space counted
        float* o = out + 6 * (size_t)offset[i];
        for (int t = 0; t < ntri; ++t) {
            float p[3][3];
#pragma unroll
            for (int q = 0; q < 3; ++q)
                edge_vertex_switch((unsigned)(w >> (4 * (3 * t + q))) & 15u, f, g, iso, p[q][0], p[q][1], p[q][2]);
            const float ux = p[1][0] - p[0][0], uy = p[1][1] - p[0][1], uz = p[1][2] - p[0][2];
            const float vx = p[2][0] - p[0][0], vy = p[2][1] - p[0][1], vz = p[2][2] - p[0][2];
            const float nxv = uy * vz - uz * vy, nyv = uz * vx - ux * vz, nzv = ux * vy - uy * vx;
            const float inv = 1.0f / sqrtf(nxv * nxv + nyv * nyv + nzv * nzv);
#pragma unroll
            for (int q = 0; q < 3; ++q) {
                float* d = o + 6 * (3 * t + q);
                d[0] = p[q][0];
                d[1] = p[q][1];
                d[2] = p[q][2];
                d[3] = nxv * inv;
                d[4] = nyv * inv;
                d[5] = nzv * inv;
            }
        }
    }
}

inline unsigned mesh_grid(long long n) {
    long long b = (n + 255) / 256;
    return (unsigned)(b > 65536 ? 65536 : (b < 1 ? 1 : b));
}

}  // namespace

// Padded volume and per-cube vertex counts.  padded: (nx+2)(ny+2)(nz+2) bytes; count: as many
// uint32.  thr as for the area kernels.
hipError_t mesh_count(const uint8_t* src, int nx, int ny, int nz, float iso, uint8_t* padded, uint32_t* count,
                      hipStream_t s) {
    const long long n = (long long)(nx + 2) * (ny + 2) * (nz + 2);
    uint32_t thr = 0;
    while (thr <= 2040u && (float)thr / 2040.0f < iso) ++thr;
    hipLaunchKernelGGL(k_pad, dim3(mesh_grid(n)), dim3(256), 0, s, src, nx, ny, nz, padded);
    hipLaunchKernelGGL(k_mesh_count, dim3(mesh_grid(n)), dim3(256), 0, s, padded, nx + 2, ny + 2, nz + 2, thr, count);
    return hipGetLastError();
}

namespace {
struct Widen {
    __host__ __device__ uint64_t operator()(uint32_t v) const { return v; }
};
}  // namespace

// Exclusive prefix sum of n per-cube counts into 64-bit offsets (hipCUB, summing in 64 bits).
// Call with tmp = nullptr for *tmp_bytes.
hipError_t mesh_scan(const uint32_t* count, uint64_t* offset, int n, void* tmp, size_t* tmp_bytes, hipStream_t s) {
    hipcub::TransformInputIterator<uint64_t, Widen, const uint32_t*> wide(count, Widen());
    return hipcub::DeviceScan::ExclusiveSum(tmp, *tmp_bytes, wide, offset, n, s);
}

hipError_t mesh_emit(const uint8_t* padded, int nx, int ny, int nz, float iso, const uint32_t* count,
                     const uint64_t* offset, float* out, hipStream_t s) {
    const long long n = (long long)(nx + 2) * (ny + 2) * (nz + 2);
    hipLaunchKernelGGL(k_mesh_emit, dim3(mesh_grid(n)), dim3(256), 0, s, padded, nx + 2, ny + 2, nz + 2, iso, count,
                       offset, out);
    return hipGetLastError();
}

}  // namespace fta
