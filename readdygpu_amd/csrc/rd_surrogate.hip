// rd_surrogate.hip -- composite external potential and its BF16 MLP surrogate.
//
// The composite is a geometry of order-one pieces (attractive disks and
// cylinders, the forms of CudaSimulation.cu:1049-1148 with any normal); a
// particle feels the piece nearest to it in energy, or the sum of all pieces
// (rd_set_composite_combine).  Evaluating it exactly
// costs one pass over every piece per particle (the reference's orderOne loop
// shape, CudaSimulation.cu:1049-1236), VALU-bound.  The surrogate is an MLP
// 3 -> 64 -> 64 -> 64 -> 3 trained on the GPU, by the kernels below, on
// gradients that the exact evaluator generates; in the step it replaces the
// exact pass.  Both passes write one float4 per sorted slot (gradient,
// energy) that the force kernel adds to the particle's gradient.
#include "rd_host.h"
#include "rd_kernels.h"
#include "rd_mlp.h"

#include <cmath>
#include <cstring>
#include <string>
#include <vector>

// ===========================================================================
// Exact composite
// ===========================================================================
struct RdPiece {
    float o[3];
    float n[3];        // unit axis
    float R;           // radius
    float hh;          // half height (0 for a disk: its energy along the axis is s^2)
    float k;
    int zaxis;         // axis is +z: cheaper projection
};                     // 40 bytes: 512 pieces and a 2 KB queue leave room for 7 workgroups per CU

__device__ __forceinline__ float piece_energy(const RdPiece& p, float x, float y, float z)
{
    float vx = x - p.o[0], vy = y - p.o[1], vz = z - p.o[2];
    float s, r2;
    if (p.zaxis) {
        s = vz;
        r2 = vx * vx + vy * vy;
    } else {
        s = vx * p.n[0] + vy * p.n[1] + vz * p.n[2];
        float qx = vx - s * p.n[0], qy = vy - s * p.n[1], qz = vz - s * p.n[2];
        r2 = qx * qx + qy * qy + qz * qz;
    }
    float dn = fmaxf(fabsf(s) - p.hh, 0.0f);
    float r = __builtin_amdgcn_sqrtf(r2);
    float dr = fmaxf(r - p.R, 0.0f);
    return 0.5f * p.k * (dn * dn + dr * dr);
}

// gradient of one piece: attractive disk / cylinder (ext_grad forms)
__device__ __forceinline__ float3 piece_grad(const RdPiece& p, float x, float y, float z)
{
    float vx = x - p.o[0], vy = y - p.o[1], vz = z - p.o[2];
    float s = vx * p.n[0] + vy * p.n[1] + vz * p.n[2];
    float qx = vx - s * p.n[0], qy = vy - s * p.n[1], qz = vz - s * p.n[2];
    float r, rinv;
    fast_len(qx * qx + qy * qy + qz * qz, &r, &rinv);
    float as = fabsf(s), sg = s > 0.0f ? 1.0f : (s < 0.0f ? -1.0f : 0.0f);
    float gn = as > p.hh ? p.k * (as - p.hh) * sg : 0.0f;
    float gx = gn * p.n[0], gy = gn * p.n[1], gz = gn * p.n[2];
    if (r > p.R) {
        float pre = p.k * (r - p.R) * rinv;
        gx += pre * qx; gy += pre * qy; gz += pre * qz;
    }
    return make_float3(gx, gy, gz);
}

#define RD_PIECES_MAX 2048

// composite at one position: energy and gradient.  SUM: the sum over every
// piece, as orderOne adds every order-one potential (CudaSimulation.cu:
// 1049-1236); otherwise the nearest piece in energy (first argmin).
template <bool SUM>
__device__ __forceinline__ float4 composite_at(const RdPiece* __restrict__ pc, int np, float x, float y, float z)
{
    if constexpr (SUM) {
        float gx = 0.f, gy = 0.f, gz = 0.f, e = 0.f;
        for (int k = 0; k < np; ++k) {
            const float3 g = piece_grad(pc[k], x, y, z);
            gx += g.x; gy += g.y; gz += g.z;
            e += piece_energy(pc[k], x, y, z);
        }
        return make_float4(gx, gy, gz, e);
    }
    float best = INFINITY;
    int kb = 0;
    for (int k = 0; k < np; ++k) {
        float e = piece_energy(pc[k], x, y, z);
        if (e < best) { best = e; kb = k; }
    }
    if (np == 0) return make_float4(0.f, 0.f, 0.f, 0.f);
    float3 g = piece_grad(pc[kb], x, y, z);
    return make_float4(g.x, g.y, g.z, best);
}

// The nearest of pieces whose axes are all +z, the same arithmetic as
// piece_energy: a[k] = origin, radius; b[k] = half height, k / 2 (in LDS).
// Bound by vector instructions (87% of the cycles): a piece is two LDS reads, of which four
// pieces' go out together, and 16 instructions and a square root, where the
// form for any axis reads ten words and branches on each piece's axis.  256
// disks, 16 crowded cytosol boxes: pass 90 -> 68 us, whole step 264 -> 240; 64
// boxes 806 -> 764.  The pieces from scalar loads: 272 (16 boxes).
__device__ __forceinline__ float4 composite_at_z(const float4* __restrict__ a, const float2* __restrict__ b,
                                                 const RdPiece* __restrict__ pieces, int np, float x, float y, float z)
{
    float best = INFINITY;
    int kb = 0;
#pragma unroll 4
    for (int k = 0; k < np; ++k) {
        const float4 o = a[k];
        const float2 h = b[k];
        const float vx = x - o.x, vy = y - o.y, vz = z - o.z;
        const float dn = fmaxf(fabsf(vz) - h.x, 0.0f);
        const float dr = fmaxf(__builtin_amdgcn_sqrtf(vx * vx + vy * vy) - o.w, 0.0f);
        const float e = h.y * (dn * dn + dr * dr);
        if (e < best) { best = e; kb = k; }
    }
    const float3 g = piece_grad(pieces[kb], x, y, z);
    return make_float4(g.x, g.y, g.z, best);
}

// ---- nearest piece by a grid of candidate lists ----
// The domain (the union of the replica boxes) is cut into cells; each cell
// lists, in index order, the pieces that can be the nearest in energy
// somewhere in it.  A point evaluates its cell's list with the arithmetic and
// the first-argmin rule of the scan over all pieces, so the result is the
// same bit for bit.
// A piece's energy is k/2 times its squared distance d, and d changes by at
// most the distance moved: with rho the half diagonal of a cell (plus a
// margin for rounding) a piece outside max(d(centre) - rho, 0) <= the least
// k/2 (d(centre) + rho)^2 over all pieces cannot be nearest.  Of the pieces
// left, those after a piece that contains the whole cell (energy 0) never
// come first.  Coplanar pieces (z axis, same plane, height and stiffness)
// share their axial term dn, so among those of the nearest piece's plane only
// the radial excess dr = max(r - R, 0) decides: one whose excess is larger
// than another's everywhere in the cell is left out, if the scan's FP32 sum
// dn^2 + dr^2 tells them apart, that is if the squared excesses differ by more
// than its rounding (far from the plane the sum absorbs dr, both energies are
// the same and the lower index wins); and so is one after a coplanar piece
// that covers the cell's whole x-y extent (a membrane of overlapping disks).
#define RD_GRID_CELLS (1 << 16)
#define RD_GRID_LIST 32          // entry 0: count (0xffff: scan all pieces), then indices
// one cell per thread, pieces in dynamic LDS
__global__ __launch_bounds__(256) void k_comp_grid(RdCompGrid g, float margin, const RdPiece* __restrict__ table,
                                                   int np, uint16_t* __restrict__ list)
{
    extern __shared__ RdPiece pieces[];
    for (int k = threadIdx.x; k < np; k += 256) pieces[k] = table[k];
    __syncthreads();
    const int c = blockIdx.x * 256 + threadIdx.x;
    if (c >= g.n[0] * g.n[1] * g.n[2]) return;
    const int ix = c % g.n[0], iy = c / g.n[0] % g.n[1], iz = c / g.n[0] / g.n[1];
    const float x = g.lo[0] + ((float)ix + 0.5f) * g.edge[0];
    const float y = g.lo[1] + ((float)iy + 0.5f) * g.edge[1];
    const float z = g.lo[2] + ((float)iz + 0.5f) * g.edge[2];
    const float exy2 = g.edge[0] * g.edge[0] + g.edge[1] * g.edge[1];
    const float rho = 0.5f * sqrtf(exy2 + g.edge[2] * g.edge[2]) + margin, rhoxy = 0.5f * sqrtf(exy2) + margin;
    auto dist = [&](const RdPiece& p, float* r_out) {        // to the disk or solid cylinder
        const float vx = x - p.o[0], vy = y - p.o[1], vz = z - p.o[2];
        float s = vz, r2 = vx * vx + vy * vy;
        if (!p.zaxis) {                                      // (the same for every lane)
            s = vx * p.n[0] + vy * p.n[1] + vz * p.n[2];
            const float qx = vx - s * p.n[0], qy = vy - s * p.n[1], qz = vz - s * p.n[2];
            r2 = qx * qx + qy * qy + qz * qz;
        }
        const float r = __builtin_amdgcn_sqrtf(r2);
        const float dn = fmaxf(fabsf(s) - p.hh, 0.0f), dr = fmaxf(r - p.R, 0.0f);
        *r_out = r;
        return __builtin_amdgcn_sqrtf(dn * dn + dr * dr);
    };
    auto coplanar = [](const RdPiece& a, const RdPiece& b) {
        return a.zaxis && b.zaxis && a.o[2] == b.o[2] && a.hh == b.hh && a.k == b.k;
    };
    float least = INFINITY, r;
    int near = 0;
#pragma unroll 4
    for (int k = 0; k < np; ++k) {
        const float d = dist(pieces[k], &r) + rho;
        const float e = 0.5f * pieces[k].k * d * d;
        if (e < least) { least = e; near = k; }
    }
    least *= 1.00001f;
    const RdPiece ref = pieces[near];
    float side = INFINITY;                       // least radial excess that the coplanar pieces reach everywhere
#pragma unroll 4
    for (int k = 0; k < np; ++k) {
        (void)dist(pieces[k], &r);
        if (coplanar(ref, pieces[k])) side = fminf(side, fmaxf(r - pieces[k].R, 0.0f) + rhoxy);
    }
    const float axial = fmaxf(fabsf(z - ref.o[2]) - ref.hh, 0.0f) + rho;     // their dn, at most
    uint16_t* out = list + (size_t)c * RD_GRID_LIST;
    int cnt = 0, cover = -1;
    for (int k = 0; k < np; ++k) {
        const RdPiece& p = pieces[k];
        const float d = fmaxf(dist(p, &r) - rho, 0.0f);
        if (!(0.5f * p.k * d * d <= least)) continue;
        // (3.6e-7 of the sum: the roundings of both sums and of their products with k / 2)
        const float a = r - p.R - rhoxy;
        if (coplanar(ref, p) && a > side && (a - side) * (a + side) > 1e-6f * (axial * axial + a * a)) continue;
        if (cover >= 0 && coplanar(p, pieces[cover])) continue;
        if (++cnt >= RD_GRID_LIST) break;
        out[cnt] = (uint16_t)k;
        if (cover < 0 && p.zaxis && r + rhoxy <= p.R) cover = k;
        const float s = (x - p.o[0]) * p.n[0] + (y - p.o[1]) * p.n[1] + (z - p.o[2]) * p.n[2];
        if (r + rho <= p.R && fabsf(s) + rho <= p.hh) break;          // contains the cell
    }
    out[0] = cnt < RD_GRID_LIST ? (uint16_t)cnt : (uint16_t)0xffff;
}

// Nearest piece at one position per lane (`act`: the lane has one; every lane
// of the wave calls it).  A lane's list is evaluated from global memory.  A
// wave with a lane that has none (a position outside the domain, a list that
// overflowed) scans all pieces, in every lane, from RD_NEAR_CHUNK pieces at a
// time in LDS of its own, which needs no barrier; the next chunk is loaded
// meanwhile.  (From global memory each piece's load is waited for, and with the
// other lanes masked the scan takes 1.7 times as long.)  2,048 pieces, 1,000
// points of which every 16th is outside: 524 us a call from global memory, 284
// so, 280 without a grid; a slab of 141 nm and 10,000 particles, where most
// lists overflow: 361, 238 and 257 us a step.
#define RD_NEAR_CHUNK 64
typedef RdPiece RdNearLds[RD_NEAR_CHUNK];
__device__ __forceinline__ float4 composite_near(const RdCompGrid& g, const RdPiece* __restrict__ pieces, int np, float x,
                                                 float y, float z, bool act, RdPiece* __restrict__ stage)
{
    const float fx = floorf((x - g.lo[0]) * g.inv[0]), fy = floorf((y - g.lo[1]) * g.inv[1]),
                fz = floorf((z - g.lo[2]) * g.inv[2]);
    const bool in = act && fx >= 0.0f && fx < (float)g.n[0] && fy >= 0.0f && fy < (float)g.n[1] && fz >= 0.0f &&
                    fz < (float)g.n[2];
    const uint4* l = reinterpret_cast<const uint4*>(
        g.list + (in ? (size_t)(((int)fz * g.n[1] + (int)fy) * g.n[0] + (int)fx) * RD_GRID_LIST : 0));
    float best = INFINITY;
    int kb = 0;
    auto test = [&](const RdPiece& p, int k) {
        const float e = piece_energy(p, x, y, z);
        if (e < best) { best = e; kb = k; }
    };
    uint4 v = make_uint4(0xffffu, 0u, 0u, 0u);
    if (in) v = l[0];                            // the count and the first seven entries
    const int cnt = (int)(v.x & 0xffffu);
    if (!__any(act && cnt == 0xffff)) {
        for (int i = 1; act && i <= cnt;) {
            const uint32_t w[4] = { v.x, v.y, v.z, v.w };
            if (i + 7 - (i & 7) < cnt) v = l[(i >> 3) + 1];
#pragma unroll
            for (int q = 0; q < 8; ++q)
                if (q >= (i & 7) && (i & ~7) + q <= cnt) {
                    const int k = (int)(w[q >> 1] >> (16 * (q & 1)) & 0xffffu);
                    test(pieces[k], k);
                }
            i = (i & ~7) + 8;
        }
    } else {
        constexpr int W = sizeof(RdPiece) / 4;   // words of a piece, and of each lane's share of a chunk
        static_assert(sizeof(RdPiece) % 4 == 0 && RD_NEAR_CHUNK == 64, "a chunk is W words of each lane");
        const uint32_t* const src = reinterpret_cast<const uint32_t*>(pieces);
        const int lane = threadIdx.x & 63, last = np * W - 1;
        uint32_t next[W];
#pragma unroll
        for (int q = 0; q < W; ++q) next[q] = src[min(q * 64 + lane, last)];
        for (int k0 = 0; k0 < np; k0 += RD_NEAR_CHUNK) {
            wave_lds_sync();                     // the last chunk has been read
#pragma unroll
            for (int q = 0; q < W; ++q) reinterpret_cast<uint32_t*>(stage)[q * 64 + lane] = next[q];
            wave_lds_sync();
#pragma unroll
            for (int q = 0; q < W; ++q) next[q] = src[min((k0 + RD_NEAR_CHUNK) * W + q * 64 + lane, last)];
            const int m = min(RD_NEAR_CHUNK, np - k0);
#pragma unroll 4
            for (int k = 0; k < m; ++k) test(stage[k], k0 + k);
        }
    }
    const float3 gr = piece_grad(pieces[kb], x, y, z);
    return make_float4(gr.x, gr.y, gr.z, best);
}

// external pass over sorted slots with the grid, for a composite on every
// type.  Bound by the lists' and pieces' load latency.  512 pieces, 500,000
// particles of the slab: 16 us (9.4 us after 100 steps, when they lie near the
// pieces) against 147 us (129) scanning all pieces from LDS; 2M: 43 against
// 503 us; 16 pieces: 5.8 against 7.8 us.  Twice the cells: 14 us, for twice the
// set-up.  When it is built and used: comp_grid.
__global__ __launch_bounds__(256) void k_composite_near(const float4* __restrict__ ps, int n, RdCompGrid g,
                                                        const RdPiece* __restrict__ pieces, int np,
                                                        float4* __restrict__ gext)
{
    __shared__ RdNearLds stage[4];
    const long s = (long)xcd_block(blockIdx.x, gridDim.x) * 256 + threadIdx.x;
    float4 p = make_float4(0.f, 0.f, 0.f, 0.f);
    if (s < n) p = ps[s];
    const float4 e = composite_near(g, pieces, np, p.x, p.y, p.z, s < n, stage[threadIdx.x >> 6]);
    if (s < n) gext[s] = e;
}

__device__ __forceinline__ void put_point(float* __restrict__ grad, float* __restrict__ energy, long i, float4 g)
{
    grad[3 * i] = g.x; grad[3 * i + 1] = g.y; grad[3 * i + 2] = g.z;
    energy[i] = g.w;
}

// at given points x[3 m]
__global__ __launch_bounds__(256) void k_composite_points_near(const float* __restrict__ x, long m, RdCompGrid g,
                                                               const RdPiece* __restrict__ pieces, int np,
                                                               float* __restrict__ grad, float* __restrict__ energy)
{
    __shared__ RdNearLds stage[4];
    const long i = (long)blockIdx.x * 256 + threadIdx.x;
    float p[3] = { 0.f, 0.f, 0.f };
    if (i < m) { p[0] = x[3 * i]; p[1] = x[3 * i + 1]; p[2] = x[3 * i + 2]; }
    const float4 e = composite_near(g, pieces, np, p[0], p[1], p[2], i < m, stage[threadIdx.x >> 6]);
    if (i < m) put_point(grad, energy, i, e);
}

// exact pass over sorted slots: gext[s] for the particles whose type is in the
// mask (other slots are left alone: the force kernel reads gext only for
// those types).  One round of resident workgroups takes chunks of 256 slots
// in turn (selected particles gather in some cells, e.g. on a membrane, so
// contiguous shares would be unbalanced), and compacts the selected ones
// into an LDS queue; whenever 256 are queued, every thread evaluates one, so
// no lane idles on an unselected particle.
// Piece table in dynamic LDS: np * sizeof(RdPiece) bytes; ALLZ: every piece's
// axis is +z.
template <bool SUM, bool ALLZ>
__global__ __launch_bounds__(256) void k_composite_slots(const float4* __restrict__ ps, int n,
                                                         const RdPiece* __restrict__ pieces, int np,
                                                         uint32_t type_mask, float4* __restrict__ gext)
{
    extern __shared__ __align__(16) RdPiece pc[];
    __shared__ uint32_t q[512];
    __shared__ int wcnt[4];
    float4* const za = reinterpret_cast<float4*>(pc);
    float2* const zb = reinterpret_cast<float2*>(za + np);
    for (int k = threadIdx.x; k < np; k += 256) {
        if constexpr (ALLZ) {
            const RdPiece p = pieces[k];
            za[k] = make_float4(p.o[0], p.o[1], p.o[2], p.R);
            zb[k] = make_float2(p.hh, 0.5f * p.k);
        } else {
            pc[k] = pieces[k];
        }
    }
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
    auto eval = [&](uint32_t s) {
        float4 p = ps[s];
        if constexpr (ALLZ) gext[s] = composite_at_z(za, zb, pieces, np, p.x, p.y, p.z);
        else gext[s] = composite_at<SUM>(pc, np, p.x, p.y, p.z);
    };
    int qn = 0;                       // queued entries (same in every thread)
    for (long base = (long)xcd_block(blockIdx.x, gridDim.x) * 256; base < n; base += (long)gridDim.x * 256) {
        const long s = base + tid;
        const bool on = s < n && ((type_mask >> w_type(ps[s].w)) & 1u);
        const uint64_t b = __ballot(on);
        if (lane == 0) wcnt[w] = __popcll(b);
        __syncthreads();
        int off = qn, tot = 0;
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            off += k < w ? wcnt[k] : 0;
            tot += wcnt[k];
        }
        if (on) q[off + lanes_below(b)] = (uint32_t)s;      // qn < 256, tot <= 256
        qn += tot;
        __syncthreads();
        if (qn >= 256) {
            eval(q[tid]);
            __syncthreads();
            if (tid < qn - 256) q[tid] = q[256 + tid];
            qn -= 256;
            __syncthreads();
        }
    }
    if (tid < qn) eval(q[tid]);
}

// exact pass when the composite acts on every type: one slot per thread
template <bool SUM>
__global__ __launch_bounds__(256) void k_composite_all(const float4* __restrict__ ps, int n,
                                                       const RdPiece* __restrict__ pieces, int np,
                                                       float4* __restrict__ gext)
{
    extern __shared__ RdPiece pc[];
    for (int k = threadIdx.x; k < np; k += 256) pc[k] = pieces[k];
    __syncthreads();
    const long s = (long)xcd_block(blockIdx.x, gridDim.x) * 256 + threadIdx.x;
    if (s >= n) return;
    const float4 p = ps[s];
    gext[s] = composite_at<SUM>(pc, np, p.x, p.y, p.z);
}

// exact evaluation at given points x[3 m]
template <bool SUM>
__global__ __launch_bounds__(256) void k_composite_points(const float* __restrict__ x, long m,
                                                          const RdPiece* __restrict__ pieces, int np,
                                                          float* __restrict__ grad, float* __restrict__ energy)
{
    extern __shared__ RdPiece pc[];
    for (int k = threadIdx.x; k < np; k += 256) pc[k] = pieces[k];
    __syncthreads();
    const long i = (long)blockIdx.x * 256 + threadIdx.x;
    if (i >= m) return;
    put_point(grad, energy, i, composite_at<SUM>(pc, np, x[3 * i], x[3 * i + 1], x[3 * i + 2]));
}

// ===========================================================================
// Training data: uniform positions in the domain, exact gradients
// ===========================================================================
__device__ __forceinline__ float u01(uint32_t b) { return (float)(b >> 8) * (1.0f / 16777216.0f); }

__device__ __forceinline__ float norm_coord(float x, float lo, float sc) { return (x - lo) * sc - 1.0f; }

// SUM: the pieces' sum; NEAR: the nearest piece by the grid; neither: by the
// scan over all pieces
template <bool SUM, bool NEAR>
__global__ __launch_bounds__(256) void k_sur_data(long m, uint64_t seed, RdMlpNorm nm, float span0, float span1,
                                                  float span2, RdCompGrid grid, const RdPiece* __restrict__ pieces,
                                                  int np,
                                                  float4* __restrict__ xn, float4* __restrict__ tg,
                                                  double* __restrict__ bsum)
{
    extern __shared__ RdPiece pc[];
    __shared__ double red[4];
    if constexpr (!NEAR) {
        for (int k = threadIdx.x; k < np; k += 256) pc[k] = pieces[k];
        __syncthreads();
    }
    const long i = (long)blockIdx.x * 256 + threadIdx.x;
    double sq = 0.0;
    uint32_t c[4] = { (uint32_t)i, (uint32_t)((uint64_t)i >> 32), 0x44415441u, 0x53555247u };
    philox4x32_10(c, (uint32_t)seed, (uint32_t)(seed >> 32));
    const float x = nm.lo[0] + u01(c[0]) * span0;
    const float y = nm.lo[1] + u01(c[1]) * span1;
    const float z = nm.lo[2] + u01(c[2]) * span2;
    float4 g;
    if constexpr (NEAR) {
        __shared__ RdNearLds stage[4];
        g = composite_near(grid, pieces, np, x, y, z, i < m, stage[threadIdx.x >> 6]);
    } else if (i < m) {
        g = composite_at<SUM>(pc, np, x, y, z);
    }
    if (i < m) {
        xn[i] = make_float4(norm_coord(x, nm.lo[0], nm.sc[0]), norm_coord(y, nm.lo[1], nm.sc[1]),
                            norm_coord(z, nm.lo[2], nm.sc[2]), 0.0f);
        tg[i] = make_float4(g.x, g.y, g.z, 0.0f);
        sq = (double)g.x * g.x + (double)g.y * g.y + (double)g.z * g.z;
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) sq += __shfl_down(sq, o, 64);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = sq;
    __syncthreads();
    if (threadIdx.x == 0) bsum[blockIdx.x] = red[0] + red[1] + red[2] + red[3];
}

// gscale = sqrt(sum / (3 m)) in a fixed order; targets divided by it
__global__ __launch_bounds__(256) void k_sur_scale_sum(const double* __restrict__ bsum, int nb, long m,
                                                       float* __restrict__ gscale)
{
    __shared__ double red[256];
    double a = 0.0;
    for (int i = threadIdx.x; i < nb; i += 256) a += bsum[i];
    red[threadIdx.x] = a;
    __syncthreads();
    if (threadIdx.x == 0) {
        double t = 0.0;
        for (int i = 0; i < 256; ++i) t += red[i];
        double gs = sqrt(t / (3.0 * (double)m));
        *gscale = gs > 0.0 ? (float)gs : 1.0f;
    }
}

__global__ __launch_bounds__(256) void k_sur_normalise(float4* __restrict__ tg, long m, const float* __restrict__ gscale)
{
    long i = (long)blockIdx.x * 256 + threadIdx.x;
    if (i >= m) return;
    float inv = 1.0f / *gscale;
    float4 g = tg[i];
    tg[i] = make_float4(g.x * inv, g.y * inv, g.z * inv, 0.0f);
}

// ===========================================================================
// Training: forward + backward of 64 samples per workgroup -> partial gradients
// ===========================================================================
struct RdTrainCtl {
    unsigned long long step;   // optimiser steps taken
    unsigned long long cur;    // the step being taken (written by k_mlp_train for k_mlp_adam)
    float loss;                // loss of the last step
    float lr, c1, c2;          // its learning rate and bias corrections
};

#define RD_TLD 72   // row stride (bf16) of the staging matrices [64][RD_TLD]
#define RD_TLF 68   // row stride (float) of the FP32 one: 4 rows apart is 16 banks apart

// one stage of the backward pass, shared by the workgroup's waves: dz and the
// layer's input in BF16 ([feature][sample]), dz in FP32
struct RdTrainStage {
    __bf16 d[64 * RD_TLD], h[64 * RD_TLD];
    float f[64 * RD_TLF];
};

// the wave's sample columns (tile wv) of a stage
__device__ __forceinline__ void stage_bf16(__bf16* S, const float (&a)[4][4], int wv, int lane)
{
    const int j = lane & 15, g = lane >> 4;
#pragma unroll
    for (int ti = 0; ti < 4; ++ti)
#pragma unroll
        for (int r = 0; r < 4; ++r) S[(ti * 16 + 4 * g + r) * RD_TLD + wv * 16 + j] = (__bf16)a[ti][r];
}

// the same of SiLU = z s
__device__ __forceinline__ void stage_product(__bf16* S, const float (&z)[4][4], const float (&s)[4][4], int wv, int lane)
{
    float h[4][4];
#pragma unroll
    for (int ti = 0; ti < 4; ++ti)
#pragma unroll
        for (int r = 0; r < 4; ++r) h[ti][r] = z[ti][r] * s[ti][r];
    stage_bf16(S, h, wv, lane);
}

__device__ __forceinline__ void stage_f32(float* S, const float (&a)[4][4], int wv, int lane)
{
    const int j = lane & 15, g = lane >> 4;
#pragma unroll
    for (int ti = 0; ti < 4; ++ti)
#pragma unroll
        for (int r = 0; r < 4; ++r) S[(ti * 16 + 4 * g + r) * RD_TLF + wv * 16 + j] = a[ti][r];
}

__device__ __forceinline__ rd_bf16x8 lds_frag(const __bf16* S, int row, int col)
{
    return *reinterpret_cast<const rd_bf16x8*>(S + row * RD_TLD + col);
}

// rows 16 ti .. 16 ti + 15 of dW[i][k] = sum_samples D[i][s] H[k][s] (64x64),
// written to out (row-major [64][64])
__device__ __forceinline__ void wgrad_rows(const RdTrainStage& S, int ti, float* __restrict__ out, int lane)
{
    const int j = lane & 15, g = lane >> 4;
    const rd_bf16x8 a0 = lds_frag(S.d, ti * 16 + j, 8 * g), a1 = lds_frag(S.d, ti * 16 + j, 32 + 8 * g);
#pragma unroll
    for (int tk = 0; tk < 4; ++tk) {
        rd_f32x4 acc = { 0.f, 0.f, 0.f, 0.f };
        acc = RD_MFMA(a0, lds_frag(S.h, tk * 16 + j, 8 * g), acc);
        acc = RD_MFMA(a1, lds_frag(S.h, tk * 16 + j, 32 + 8 * g), acc);
#pragma unroll
        for (int r = 0; r < 4; ++r) out[(ti * 16 + 4 * g + r) * 64 + tk * 16 + j] = acc[r];
    }
}

// bias gradient of features 16 ti .. 16 ti + 15: sum over the 64 samples of dz
__device__ __forceinline__ void bgrad_rows(const RdTrainStage& S, int ti, float* __restrict__ out, int lane)
{
    const int j = lane & 15, g = lane >> 4;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        const float* d = S.f + (ti * 16 + 4 * g + r) * RD_TLF + j;
        const float v = rd_sum16(d[0] + d[16] + d[32] + d[48]);
        if (j == 0) out[ti * 16 + 4 * g + r] = v;
    }
}

// dz of the layer below: (W^T dz) dsilu(z), W^T fragments wt
__device__ __forceinline__ void back64(const rd_bf16x8 (&wt)[4][2], const float (&z)[4][4], const float (&s)[4][4],
                                       float (&dz)[4][4])
{
    const rd_f32x4 zero[4] = {};
    float dh[4][4];
    rd_mlp_layer64(wt, zero, dz, dh);
#pragma unroll
    for (int b = 0; b < 4; ++b)
#pragma unroll
        for (int r = 0; r < 4; ++r) dz[b][r] = dh[b][r] * rd_dsilu(z[b][r], s[b][r]);
}

// Learning rate (cosine from lr0 to lr1 over total steps) and Adam's bias
// corrections.
struct RdSchedule {
    float lr0, lr1;
    long long total;
    float b1, b2;
};

// Samples: idx = sequential ? c : Philox(seed, step, c) mod m.  Samples at
// c >= batch (padding of the last workgroup) contribute nothing.
//
// A batch is small for the chip (8,192 samples: 128 workgroups of 64), so the
// step is bound by its chain of latencies: each of the four waves takes 16
// samples through the network and back, all weight fragments are loaded to
// registers up front, and the waves meet once per layer, at a stage in LDS
// (two, used in turn, so that one barrier per stage suffices) from which each
// wave computes a quarter of the layer's weight and bias gradients.  256
// steps of 8,192 samples with k_mlp_adam: 16 us a step, against 53 us with
// 64 samples in each wave (32 workgroups), weights staged in LDS and the step
// counter in a kernel of its own.  The sums' orders are those of that form.
// One more workgroup computes the step's schedule meanwhile.
__global__ __launch_bounds__(256) void k_mlp_train(const float4* __restrict__ xn_all, const float4* __restrict__ tn_all,
                                                   long m, uint64_t inv_m, int batch, int sequential, uint64_t seed,
                                                   const RdMlpPack* __restrict__ pk, RdTrainCtl* __restrict__ ctl,
                                                   float* __restrict__ partial, RdSchedule sch)
{
    __shared__ __align__(16) RdTrainStage stage[2];
    __shared__ float xs[3][64], rs[3][64];           // inputs and residuals of the samples
    const unsigned long long step = ctl->step;
    if (blockIdx.x == gridDim.x - 1) {
        if (threadIdx.x == 0) {
            const unsigned long long t = step + 1;
            const double ph = sch.total > 0 ? fmin(1.0, (double)(t - 1) / (double)sch.total) : 0.0;
            ctl->cur = step;
            ctl->lr = sch.lr1 + 0.5f * (sch.lr0 - sch.lr1) * (float)(1.0 + cos(3.14159265358979323846 * ph));
            ctl->c1 = 1.0f - (float)pow((double)sch.b1, (double)t);
            ctl->c2 = 1.0f - (float)pow((double)sch.b2, (double)t);
        }
        return;
    }
    const int wv = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int j = lane & 15, g = lane >> 4;
    float* out = partial + (size_t)blockIdx.x * RD_MLP_ROW;

    const int c = blockIdx.x * 64 + wv * 16 + j;
    const bool live = c < batch;
    long idx = c;
    if (!sequential) {
        uint32_t q[4] = { (uint32_t)c, (uint32_t)step, (uint32_t)(step >> 32), 0x5452414eu };
        philox4x32_10(q, (uint32_t)seed, (uint32_t)(seed >> 32));
        // x mod m from the quotient's estimate mulhi(x, 2^64 / m), at most 2 low
        const uint64_t x = (uint64_t)q[1] << 32 | q[0];
        uint64_t rem = x - __umul64hi(x, inv_m) * (uint64_t)m;
        rem -= rem >= (uint64_t)m ? (uint64_t)m : 0u;
        rem -= rem >= (uint64_t)m ? (uint64_t)m : 0u;
        idx = (long)rem;
    }
    if (!live) idx = 0;
    const float4 xa = xn_all[idx], ta = tn_all[idx];
    // the lane's weights: layer 1 (features 16 ti + 4 g + r: 12 consecutive
    // values per tile), biases, and the fragments of every layer
    rd_f32x4 w1[4][3], b1[4], b2[4], b3[4];
#pragma unroll
    for (int ti = 0; ti < 4; ++ti) {
        const int f = ti * 16 + 4 * g;
        b1[ti] = *reinterpret_cast<const rd_f32x4*>(pk->b1 + f);
        b2[ti] = *reinterpret_cast<const rd_f32x4*>(pk->b2 + f);
        b3[ti] = *reinterpret_cast<const rd_f32x4*>(pk->b3 + f);
#pragma unroll
        for (int k = 0; k < 3; ++k) w1[ti][k] = *reinterpret_cast<const rd_f32x4*>(pk->w1 + 3 * f + 4 * k);
    }
    rd_bf16x8 w2[4][2], w3[4][2], w2t[4][2], w3t[4][2], w4[2], w4t[4];
#pragma unroll
    for (int to = 0; to < 4; ++to)
#pragma unroll
        for (int kb = 0; kb < 2; ++kb) w2[to][kb] = pk->w2[to][kb][lane];
#pragma unroll
    for (int to = 0; to < 4; ++to)
#pragma unroll
        for (int kb = 0; kb < 2; ++kb) w3[to][kb] = pk->w3[to][kb][lane];
#pragma unroll
    for (int kb = 0; kb < 2; ++kb) w4[kb] = pk->w4[kb][lane];
#pragma unroll
    for (int to = 0; to < 4; ++to) w4t[to] = pk->w4t[to][lane];
#pragma unroll
    for (int to = 0; to < 4; ++to)
#pragma unroll
        for (int kb = 0; kb < 2; ++kb) w3t[to][kb] = pk->w3t[to][kb][lane];
#pragma unroll
    for (int to = 0; to < 4; ++to)
#pragma unroll
        for (int kb = 0; kb < 2; ++kb) w2t[to][kb] = pk->w2t[to][kb][lane];
    rd_f32x4 b4 = { 0.f, 0.f, 0.f, 0.f };
    if (g == 0) { b4[0] = pk->b4[0]; b4[1] = pk->b4[1]; b4[2] = pk->b4[2]; }
    const float xn[3] = { xa.x, xa.y, xa.z }, tn[3] = { ta.x, ta.y, ta.z };

    // ---- forward ----
    float z1[4][4], z2[4][4], z3[4][4], s1[4][4], s2[4][4], s3[4][4], h[4][4];
#pragma unroll
    for (int ti = 0; ti < 4; ++ti)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int k = 3 * r;
            float v = w1[ti][k / 4][k % 4] * xn[0];
            v = v + w1[ti][(k + 1) / 4][(k + 1) % 4] * xn[1];
            v = v + w1[ti][(k + 2) / 4][(k + 2) % 4] * xn[2];
            z1[ti][r] = v + b1[ti][r];
        }
    rd_mlp_silu_all(z1, s1, h);
    rd_mlp_layer64(w2, b2, h, z2);
    rd_mlp_silu_all(z2, s2, h);
    rd_mlp_layer64(w3, b3, h, z3);
    rd_mlp_silu_all(z3, s3, h);              // h = h3
    rd_f32x4 y = b4;
    y = RD_MFMA(w4[0], rd_mlp_bop(h, 0), y);
    y = RD_MFMA(w4[1], rd_mlp_bop(h, 1), y);

    // ---- residuals and dy (lanes of group 0 hold the outputs) ----
    const float sc2 = 2.0f / (float)batch;
    float dy[3];
    __bf16* const SD = stage[0].d;
    stage_bf16(stage[0].h, h, wv, lane);
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        const float r = (g == 0 && live) ? y[k] - tn[k] : 0.0f;
        dy[k] = sc2 * r;
        if (g == 0) {
            SD[k * RD_TLD + wv * 16 + j] = (__bf16)dy[k];
            rs[k][wv * 16 + j] = r;
            xs[k][wv * 16 + j] = xn[k];
        }
    }
    __syncthreads();
    // columns 16 wv .. of dW4 = dy h3^T
    {
        rd_bf16x8 a0, a1;
        if (j < 3) { a0 = lds_frag(SD, j, 8 * g); a1 = lds_frag(SD, j, 32 + 8 * g); }
        else {
#pragma unroll
            for (int t = 0; t < 8; ++t) { a0[t] = (__bf16)0.0f; a1[t] = (__bf16)0.0f; }
        }
        rd_f32x4 acc = { 0.f, 0.f, 0.f, 0.f };
        acc = RD_MFMA(a0, lds_frag(stage[0].h, wv * 16 + j, 8 * g), acc);
        acc = RD_MFMA(a1, lds_frag(stage[0].h, wv * 16 + j, 32 + 8 * g), acc);
        if (g == 0) {
#pragma unroll
            for (int r = 0; r < 3; ++r) out[RD_MLP_W4 + r * 64 + wv * 16 + j] = acc[r];
        }
    }
    // db4 and the loss
    if (wv == 0) {
        float l = 0.0f, d4[3] = { 0.0f, 0.0f, 0.0f };
        if (g == 0) {
#pragma unroll
            for (int tj = 0; tj < 4; ++tj)
#pragma unroll
                for (int k = 0; k < 3; ++k) {
                    const float r = rs[k][tj * 16 + j];
                    l += r * r;
                    d4[k] = tj == 0 ? sc2 * r : d4[k] + sc2 * r;
                }
        }
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            const float v = rd_sum16(d4[k]);
            if (lane == 0) out[RD_MLP_B4 + k] = v;
        }
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) l += __shfl_xor(l, o, 64);
        if (lane == 0) out[RD_MLP_NPARAM] = l / (float)batch;
    }

    // dz3 = (W4^T dy) dsilu: B operand = dy in lanes of group 0 (k = 0..2)
    float dz[4][4];
    {
        rd_bf16x8 b;
#pragma unroll
        for (int t = 0; t < 8; ++t) b[t] = (__bf16)((g == 0 && t < 3) ? dy[t < 3 ? t : 0] : 0.0f);
#pragma unroll
        for (int to = 0; to < 4; ++to) {
            rd_f32x4 acc = { 0.f, 0.f, 0.f, 0.f };
            acc = RD_MFMA(w4t[to], b, acc);
#pragma unroll
            for (int r = 0; r < 4; ++r) dz[to][r] = acc[r] * rd_dsilu(z3[to][r], s3[to][r]);
        }
    }
    // dW3 = dz3 h2^T
    stage_bf16(stage[1].d, dz, wv, lane);
    stage_product(stage[1].h, z2, s2, wv, lane);
    stage_f32(stage[1].f, dz, wv, lane);
    __syncthreads();
    back64(w3t, z2, s2, dz);                   // dz2
    wgrad_rows(stage[1], wv, out + RD_MLP_W3, lane);
    bgrad_rows(stage[1], wv, out + RD_MLP_B3, lane);
    // dW2 = dz2 h1^T
    stage_bf16(stage[0].d, dz, wv, lane);
    stage_product(stage[0].h, z1, s1, wv, lane);
    stage_f32(stage[0].f, dz, wv, lane);
    __syncthreads();
    back64(w2t, z1, s1, dz);                   // dz1
    wgrad_rows(stage[0], wv, out + RD_MLP_W2, lane);
    bgrad_rows(stage[0], wv, out + RD_MLP_B2, lane);
    // dW1 = dz1 xn^T in FP32 on the VALU
    stage_f32(stage[1].f, dz, wv, lane);
    __syncthreads();
    bgrad_rows(stage[1], wv, out + RD_MLP_B1, lane);
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        const float* d = stage[1].f + (wv * 16 + 4 * g + r) * RD_TLF + j;
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            float v = d[0] * xs[k][j];
            v = v + d[16] * xs[k][16 + j];
            v = v + d[32] * xs[k][32 + j];
            v = v + d[48] * xs[k][48 + j];
            v = rd_sum16(v);
            if (j == 0) out[RD_MLP_W1 + 3 * (wv * 16 + 4 * g + r) + k] = v;
        }
    }
}

// write the packed BF16 / FP32 copies of master parameter p
__device__ __forceinline__ void pack_param(RdMlpPack* __restrict__ pk, int p, float w)
{
    const __bf16 wb = (__bf16)w;
    auto put = [&](rd_bf16x8* frag, int t) { reinterpret_cast<__bf16*>(frag)[t] = wb; };
    auto kpos = [](int b, int& kb, int& g, int& t) {
        kb = (b >> 4) >> 1;
        t = 4 * ((b >> 4) & 1) + (b & 3);
        g = (b & 15) >> 2;
    };
    if (p < RD_MLP_B1) {
        pk->w1[p] = (float)wb;
        pk->w1s[p] = (float)wb * RD_MLP_NLOG2E;
        return;
    }
    if (p < RD_MLP_W2) {
        pk->b1[p - RD_MLP_B1] = w;
        pk->b1s[p - RD_MLP_B1] = w * RD_MLP_NLOG2E;
        return;
    }
    if (p < RD_MLP_B2 || (p >= RD_MLP_W3 && p < RD_MLP_B3)) {
        const bool l3 = p >= RD_MLP_W3;
        const int q = p - (l3 ? RD_MLP_W3 : RD_MLP_W2);
        const int a = q >> 6, b = q & 63;       // W[a][b]: output a, input b
        int kb, g, t;
        kpos(b, kb, g, t);
        put(l3 ? &pk->w3[a >> 4][kb][g * 16 + (a & 15)] : &pk->w2[a >> 4][kb][g * 16 + (a & 15)], t);
        kpos(a, kb, g, t);
        put(l3 ? &pk->w3t[b >> 4][kb][g * 16 + (b & 15)] : &pk->w2t[b >> 4][kb][g * 16 + (b & 15)], t);
        return;
    }
    if (p < RD_MLP_W3) {
        pk->b2[p - RD_MLP_B2] = w;
        pk->b2s[p - RD_MLP_B2] = w * RD_MLP_NLOG2E;
        return;
    }
    if (p < RD_MLP_W4) {
        pk->b3[p - RD_MLP_B3] = w;
        pk->b3s[p - RD_MLP_B3] = w * RD_MLP_NLOG2E;
        return;
    }
    if (p < RD_MLP_B4) {
        const int q = p - RD_MLP_W4, o = q >> 6, b = q & 63;
        int kb, g, t;
        kpos(b, kb, g, t);
        put(&pk->w4[kb][g * 16 + o], t);
        put(&pk->w4t[b >> 4][b & 15], o);
        reinterpret_cast<__bf16*>(&pk->w4s[kb][g * 16 + o])[t] = (__bf16)(w * RD_MLP_NLN2);
        return;
    }
    pk->b4[p - RD_MLP_B4] = w;
}

__global__ __launch_bounds__(256) void k_mlp_pack(const float* __restrict__ master, RdMlpPack* __restrict__ pk)
{
    int p = blockIdx.x * 256 + threadIdx.x;
    if (p < RD_MLP_NPARAM) pack_param(pk, p, master[p]);
}

// Sum the partial gradients in row order (deterministic), Adam step on the
// FP32 master weights, refresh the packed copies; the loss column's thread
// advances the step counter (k_mlp_train reads it, nothing here does).
__global__ __launch_bounds__(256) void k_mlp_adam(const float* __restrict__ partial, int nrow,
                                                  float* __restrict__ master, float* __restrict__ mom,
                                                  float* __restrict__ vel, RdMlpPack* __restrict__ pk,
                                                  RdTrainCtl* __restrict__ ctl, float b1, float b2, float eps,
                                                  float* __restrict__ grad_out, int apply,
                                                  float* __restrict__ loss_hist)
{
    // 32 parameters per workgroup, the partial rows split over 8 slices, the
    // slices added in a fixed order: deterministic, and enough workgroups to
    // keep the loads in flight (8 per thread at once)
    __shared__ float red[8][32];
    const int pl = threadIdx.x & 31, slice = threadIdx.x >> 5;
    const int p = blockIdx.x * 32 + pl;
    const bool sum = slice == 0 && p < RD_MLP_NPARAM;
    float m = 0.0f, v = 0.0f, w0 = 0.0f;
    if (sum && apply) { m = mom[p]; v = vel[p]; w0 = master[p]; }
    const unsigned long long cur = ctl->cur;
    const float lr = ctl->lr, c1 = ctl->c1, c2 = ctl->c2;
    float part = 0.0f;
    if (p <= RD_MLP_NPARAM) {
        const float* src = partial + p;
        int w = slice;
        for (; w + 56 < nrow; w += 64) {
            float q[8];
#pragma unroll
            for (int k = 0; k < 8; ++k) q[k] = src[(size_t)(w + 8 * k) * RD_MLP_ROW];
#pragma unroll
            for (int k = 0; k < 8; ++k) part += q[k];
        }
        for (; w < nrow; w += 8) part += src[(size_t)w * RD_MLP_ROW];
    }
    red[slice][pl] = part;
    __syncthreads();
    if (slice != 0 || p > RD_MLP_NPARAM) return;
    float gsum = 0.0f;
#pragma unroll
    for (int k = 0; k < 8; ++k) gsum += red[k][pl];
    if (p == RD_MLP_NPARAM) {        // loss column
        ctl->loss = gsum;
        if (loss_hist) loss_hist[cur] = gsum;
        if (apply) ctl->step = cur + 1;
        return;
    }
    if (grad_out) grad_out[p] = gsum;
    if (!apply) return;
    m = b1 * m + (1.0f - b1) * gsum;
    v = b2 * v + (1.0f - b2) * gsum * gsum;
    mom[p] = m;
    vel[p] = v;
    const float mh = m / c1;
    const float vh = v / c2;
    const float w = w0 - lr * mh / (sqrtf(vh) + eps);
    master[p] = w;
    pack_param(pk, p, w);
}

// ===========================================================================
// Inference
// ===========================================================================
// Persistent waves: the forward weights (A fragments, 18 KB) and layer-1
// weights and biases are staged in LDS per workgroup; the compiler keeps the
// fragments a lane uses in registers across tiles (about 210 VGPRs: 2 waves
// per SIMD, which overlap one wave's SiLU work on the VALU with the other's
// MFMAs; the MFMAs write VGPRs directly, built with
// -mllvm -amdgpu-mfma-vgpr-form, so no accumulator-register reads follow
// them).  Samples go through the network one sample tile (16 samples) at a
// time, so only one tile's activations are live, as packed BF16 B operands.
// Lane l holds sample l % 16 of the tile; outputs land in lanes 0..15.
//
// The staged copies are the pack's inference copies: layer 1 and the biases
// carry -log2(e) and W4 carries -ln 2, so every layer yields zs = -log2(e) z
// and the activation zs / (1 + 2^zs) = -log2(e) SiLU(z) feeds the next layer
// unchanged (W2 and W3 see the factor in both their input and their output);
// W4's -ln 2 removes it.  SiLU then costs 2^x, a reciprocal, an add and one
// multiply.  The inference is VALU-bound (two transcendentals per
// activation), so each VALU instruction saved counts.
struct RdMlpFwdLds {
    rd_bf16x8 w2[4][2][64], w3[4][2][64], w4[2][64];
    float w1[192], b1[64], b2[64], b3[64], b4[4];
};

// BLOCK threads stage the weights with compile-time strides (blockDim.x
// would be a load from the dispatch packet ahead of each loop), loads issued
// in two batches ahead of their LDS stores (two global latencies instead of
// one per loop iteration; one batch of everything spills registers)
template <int BLOCK>
__device__ __forceinline__ void mlp_stage(RdMlpFwdLds& L, const RdMlpPack* __restrict__ pk_g)
{
    const uint4* src = reinterpret_cast<const uint4*>(pk_g);      // w2, w3 lead the pack
    uint4* dst = reinterpret_cast<uint4*>(&L);
    constexpr int N23 = (int)(sizeof(rd_bf16x8) * (2 * 4 * 2 * 64) / 16);
    static_assert(N23 % (2 * BLOCK) == 0 && BLOCK >= 192, "staging layout");
    const int t = threadIdx.x;
    const uint4* s4 = reinterpret_cast<const uint4*>(pk_g->w4s);
    uint4* d4 = reinterpret_cast<uint4*>(L.w4);
    // batch 1: the small arrays and half of w2, w3
    uint4 v4 = make_uint4(0u, 0u, 0u, 0u);
    float v1 = 0.0f, vb1 = 0.0f, vb2 = 0.0f, vb3 = 0.0f, vb4 = 0.0f;
    if (t < 2 * 64) v4 = s4[t];
    if (t < 192) v1 = pk_g->w1s[t];
    if (t < 64) { vb1 = pk_g->b1s[t]; vb2 = pk_g->b2s[t]; vb3 = pk_g->b3s[t]; }
    if (t < 4) vb4 = pk_g->b4[t];
    constexpr int KH = N23 / (2 * BLOCK);
    for (int h = 0; h < 2; ++h) {
        uint4 v[KH];
#pragma unroll
        for (int k = 0; k < KH; ++k) v[k] = src[t + (h * KH + k) * BLOCK];
#pragma unroll
        for (int k = 0; k < KH; ++k) dst[t + (h * KH + k) * BLOCK] = v[k];
    }
    if (t < 2 * 64) d4[t] = v4;
    if (t < 192) L.w1[t] = v1;
    if (t < 64) { L.b1[t] = vb1; L.b2[t] = vb2; L.b3[t] = vb3; }
    if (t < 4) L.b4[t] = vb4;
}

// -log2(e) SiLU(z) from zs = -log2(e) z
__device__ __forceinline__ float rd_silu_l2(float zs)
{
    return zs * __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(zs));
}

// network output for this lane's sample of the tile (valid in lanes 0..15)
__device__ __forceinline__ float3 mlp_tile(const RdMlpFwdLds& L, const float (&xn)[3])
{
    const int lane = threadIdx.x & 63;
    const int g = lane >> 4;
    // layer 1 (FP32 FMAs, VALU) -> SiLU -> B operands
    rd_f32x4 z[4];
#pragma unroll
    for (int ti = 0; ti < 4; ++ti)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int f = ti * 16 + 4 * g + r;
            float v = __builtin_fmaf(L.w1[3 * f], xn[0], L.b1[f]);
            v = __builtin_fmaf(L.w1[3 * f + 1], xn[1], v);
            z[ti][r] = __builtin_fmaf(L.w1[3 * f + 2], xn[2], v);
        }
    rd_bf16x8 hb[2];
#pragma unroll
    for (int kb = 0; kb < 2; ++kb)
#pragma unroll
        for (int t = 0; t < 8; ++t) hb[kb][t] = (__bf16)rd_silu_l2(z[2 * kb + t / 4][t & 3]);
    // layers 2 and 3 (MFMA) -> SiLU
#pragma unroll
    for (int layer = 0; layer < 2; ++layer) {
        const float* bb = layer == 0 ? L.b2 : L.b3;
#pragma unroll
        for (int to = 0; to < 4; ++to) {
            rd_f32x4 acc;
#pragma unroll
            for (int r = 0; r < 4; ++r) acc[r] = bb[to * 16 + 4 * g + r];
            acc = RD_MFMA(layer == 0 ? L.w2[to][0][lane] : L.w3[to][0][lane], hb[0], acc);
            acc = RD_MFMA(layer == 0 ? L.w2[to][1][lane] : L.w3[to][1][lane], hb[1], acc);
            z[to] = acc;
        }
#pragma unroll
        for (int kb = 0; kb < 2; ++kb)
#pragma unroll
            for (int t = 0; t < 8; ++t) hb[kb][t] = (__bf16)rd_silu_l2(z[2 * kb + t / 4][t & 3]);
    }
    // layer 4 (MFMA, rows 0..2 of 16)
    rd_f32x4 acc;
#pragma unroll
    for (int r = 0; r < 4; ++r) acc[r] = (g == 0 && r < 3) ? L.b4[r] : 0.0f;
    acc = RD_MFMA(L.w4[0][lane], hb[0], acc);
    acc = RD_MFMA(L.w4[1][lane], hb[1], acc);
    return make_float3(acc[0], acc[1], acc[2]);
}

// surrogate pass over sorted slots: gext[s] = gscale * mlp(normalised position)
// for the particles whose type is in the mask (other slots are not written).
// One round of resident waves takes chunks of 64 slots in turn; a wave
// appends the selected slots of its chunk to a ring queue in LDS and runs a
// tile whenever 16 are queued; the last partial tile runs at the end.
#define RD_MLP_RING 128
__global__ __launch_bounds__(256) void k_mlp_slots(const RdMlpPack* __restrict__ pk, const float4* __restrict__ ps,
                                                   int n, RdMlpNorm nm, uint32_t type_mask,
                                                   float4* __restrict__ gext)
{
    __shared__ RdMlpFwdLds L;
    __shared__ float4 ring[4][RD_MLP_RING];              // normalised position, slot
    mlp_stage<256>(L, pk);
    __syncthreads();
    const int lane = threadIdx.x & 63, j = lane & 15;
    float4* q = ring[threadIdx.x >> 6];
    auto tile = [&](uint32_t head, int cnt) {            // cnt in 1..16 entries from head
        const bool ok = j < cnt;
        const float4 p = q[(head + (ok ? j : 0)) & (RD_MLP_RING - 1)];
        const float xn[3] = { p.x, p.y, p.z };
        const float3 y = mlp_tile(L, xn);
        if (lane < 16 && ok)
            gext[__float_as_uint(p.w)] = make_float4(y.x * nm.gscale, y.y * nm.gscale, y.z * nm.gscale, 0.f);
    };
    const long nchunks = ((long)n + 63) / 64;
    const long wpb = blockDim.x >> 6;
    const long stride = (long)gridDim.x * wpb;
    uint32_t head = 0, tail = 0;                         // tail - head <= 15 between chunks
    long c = (long)xcd_block(blockIdx.x, gridDim.x) * wpb + (threadIdx.x >> 6);
    float4 next = make_float4(0.f, 0.f, 0.f, 0.f);       // the next chunk's record, a chunk ahead
    if (c * 64 + lane < n) next = ps[c * 64 + lane];
    for (; c < nchunks; c += stride) {
        const long s = c * 64 + lane;
        const float4 p = next;
        if (s + stride * 64 < n) next = ps[s + stride * 64];
        const bool on = s < n && ((type_mask >> w_type(p.w)) & 1u);
        const uint64_t b = __ballot(on);
        if (on)
            q[(tail + lanes_below(b)) & (RD_MLP_RING - 1)] =
                make_float4(norm_coord(p.x, nm.lo[0], nm.sc[0]), norm_coord(p.y, nm.lo[1], nm.sc[1]),
                            norm_coord(p.z, nm.lo[2], nm.sc[2]), __uint_as_float((uint32_t)s));
        tail += (uint32_t)__popcll(b);
        wave_lds_sync();
#pragma unroll 1
        while (tail - head >= 16) {
            tile(head, 16);
            head += 16;
        }
        wave_lds_sync();
    }
    if (tail != head) tile(head, (int)(tail - head));
}

// inference at normalised points -> raw network output, STRIDE values per
// point in both (3, or 4 with the last one unused)
template <int STRIDE>
__global__ __launch_bounds__(256) void k_mlp_points(const RdMlpPack* __restrict__ pk, const float* __restrict__ xin,
                                                    long m, float* __restrict__ out)
{
    __shared__ RdMlpFwdLds L;
    mlp_stage<256>(L, pk);
    __syncthreads();
    const int lane = threadIdx.x & 63, j = lane & 15;
    const long ntiles = (m + 15) / 16;
    const long wpb = blockDim.x >> 6;
    const long stride = (long)gridDim.x * wpb;
    for (long t = (long)xcd_block(blockIdx.x, gridDim.x) * wpb + (threadIdx.x >> 6); t < ntiles; t += stride) {
        const long i = t * 16 + j;
        float xn[3] = { 0.f, 0.f, 0.f };
        if (i < m) {
#pragma unroll
            for (int k = 0; k < 3; ++k) xn[k] = xin[i * STRIDE + k];
        }
        const float3 y = mlp_tile(L, xn);
        if (lane < 16 && i < m) {
            out[i * STRIDE] = y.x; out[i * STRIDE + 1] = y.y; out[i * STRIDE + 2] = y.z;
        }
    }
}

// squared error of the network's outputs y (times gscale) against the exact
// gradients t, and the squared gradients, per workgroup in FP64
__global__ __launch_bounds__(256) void k_sur_error(const float4* __restrict__ t, const float4* __restrict__ y, long m,
                                                   double gscale, double* __restrict__ num, double* __restrict__ den)
{
    __shared__ double red[2][4];
    const long i = (long)blockIdx.x * 256 + threadIdx.x;
    double a = 0.0, b = 0.0;
    if (i < m) {
        const float4 g = t[i], v = y[i];
        const double ex = g.x, ey = g.y, ez = g.z;
        const double dx = v.x * gscale - ex, dy = v.y * gscale - ey, dz = v.z * gscale - ez;
        a = dx * dx + dy * dy + dz * dz;
        b = ex * ex + ey * ey + ez * ez;
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) { a += __shfl_down(a, o, 64); b += __shfl_down(b, o, 64); }
    if ((threadIdx.x & 63) == 0) { red[0][threadIdx.x >> 6] = a; red[1][threadIdx.x >> 6] = b; }
    __syncthreads();
    if (threadIdx.x == 0) {
        num[blockIdx.x] = red[0][0] + red[0][1] + red[0][2] + red[0][3];
        den[blockIdx.x] = red[1][0] + red[1][1] + red[1][2] + red[1][3];
    }
}

// ===========================================================================
// Host side
// ===========================================================================
static int sset_err(rd_system* h, int code, const std::string& m)
{
    h->err = m;
    return code;
}

#define SHIPCK(h, x)                                                                           \
    do {                                                                                       \
        hipError_t e_ = (x);                                                                   \
        if (e_ != hipSuccess)                                                                  \
            return sset_err((h), RD_EHIP, std::string(#x) + ": " + hipGetErrorString(e_));    \
    } while (0)

static inline unsigned nb256(long n) { return (unsigned)((n + 255) / 256); }
static inline size_t pieces_lds(const rd_system* h) { return sizeof(RdPiece) * (size_t)(h->npieces > 0 ? h->npieces : 1); }

void rd_host_free_surrogate(rd_system* h)
{
    void* ptrs[] = { h->d_pieces, h->d_gext, h->d_master, h->d_mom, h->d_vel, h->d_pack, h->d_ctl, h->d_partial,
                     h->d_xn, h->d_tg, h->d_gscale, h->d_sbsum, h->d_loss_hist, h->d_comp_list };
    for (void* p : ptrs)
        if (p) (void)hipFree(p);
    h->d_pieces = nullptr; h->d_gext = nullptr; h->d_master = h->d_mom = h->d_vel = nullptr;
    h->d_pack = nullptr; h->d_ctl = nullptr; h->d_partial = nullptr; h->d_xn = h->d_tg = nullptr;
    h->d_gscale = nullptr; h->d_sbsum = nullptr; h->d_loss_hist = nullptr;
    h->d_comp_list = nullptr; h->comp_grid_set = false;
    h->gext_cap = 0; h->partial_rows = 0; h->nsamples = 0; h->loss_hist_cap = 0;
}

static uint32_t all_types(const rd_system* h) { return h->nt >= 32 ? 0xffffffffu : (1u << h->nt) - 1u; }

// Grid of the nearest-piece composite over the union of the replica boxes, for
// a call that passes over the pieces `passes` times (of passes_of; 0: only a
// grid that is there is taken, RD_GRID_NOW: the caller asks for it).
// Not used, and every piece scanned, for a sum, a stiffness that is not positive
// (no nearest distance) or few pieces: on sorted slots 12 pieces win and 9 do
// not (2M slots: scan 18.5 and 16.2 us, grid 16.6 and 17.1), on points in random
// order, whose lists are read here and there, 32 and 24 (1M training points:
// scan 58.0 and 54.5 us, grid 57.5 and 56.9).
// Building the lists (k_comp_grid on the handle's stream) takes as long as 3.5
// passes save, at any number of pieces (512: 200 us for 55 us a pass; 2,048:
// 780 for 220), so it waits until more than three passes over the same pieces
// and boxes have been asked for: a program that moves its pieces for every few
// points or steps scans them (512 pieces, one point: 474 us for rd_set_composite
// and rd_composite_eval, 667 with a grid).
#define RD_GRID_SLOT_PIECES 12
#define RD_GRID_POINT_PIECES 32
#define RD_GRID_PASSES 3
// A scan takes the same time for up to about 130,000 points, which are resident
// at once, and grows from there.
static long passes_of(long points) { return 1 + (points >> 17); }

// union of the replica boxes: [axis] { low, high }
static void union_box(const rd_system* h, double (&box)[3][2])
{
    for (int d = 0; d < 3; ++d) {
        box[d][0] = h->reps.empty() ? h->prm.lattice_bounds[2 * d] : h->reps[0].lo[d];
        box[d][1] = h->reps.empty() ? h->prm.lattice_bounds[2 * d + 1] : h->reps[0].hi[d];
        for (const rd_system::Rep& r : h->reps) {
            box[d][0] = std::min(box[d][0], r.lo[d]);
            box[d][1] = std::max(box[d][1], r.hi[d]);
        }
    }
}

static int comp_grid(rd_system* h, RdCompGrid* g, long passes, int min_pieces)
{
    memset(g, 0, sizeof(*g));
    if (h->comp_sum || h->npieces < min_pieces) return RD_OK;
    double box[3][2], vol = 1.0, reach = 0.0;
    union_box(h, box);
    bool same = h->comp_grid_set;
    for (int d = 0; d < 3; ++d) {
        vol *= box[d][1] - box[d][0];
        same = same && h->comp_lo[d] == box[d][0] && h->comp_hi[d] == box[d][1];
    }
    if (same) { *g = h->comp_built; return RD_OK; }
    h->comp_passes += passes;
    if (h->comp_passes <= RD_GRID_PASSES) return RD_OK;
    // (of pieces and boxes that no grid serves, one without lists is kept)
    h->comp_grid_set = false;
    bool ok = true;
    for (const rd_pot1& p : h->comp) {
        ok = ok && p.force_const > 0.0f && std::isfinite(p.force_const) && std::isfinite(p.radius) && std::isfinite(p.height);
        for (int d = 0; d < 3; ++d) ok = ok && std::isfinite(p.origin[d]) && std::isfinite(p.normal[d]);
    }
    const double edge = std::cbrt(vol / RD_GRID_CELLS);
    long cells = 1;
    for (int d = 0; d < 3; ++d) {
        const double lo = box[d][0], hi = box[d][1];
        g->n[d] = (int)std::min(std::max((hi - lo) / edge, 1.0), (double)RD_GRID_CELLS);
        cells *= g->n[d];
        g->lo[d] = (float)lo;
        g->edge[d] = (float)((hi - lo) / g->n[d]);
        g->inv[d] = (float)(g->n[d] / (hi - lo));
        // the largest separation of a position and a piece, for the rounding margin
        for (const rd_pot1& p : h->comp)
            reach = std::max(reach, std::max(std::fabs(lo - p.origin[d]), std::fabs(hi - p.origin[d])) +
                                        std::max(std::fabs(lo), std::fabs(hi)) + std::fabs(p.radius) +
                                        std::fabs(p.height));
    }
    if (ok && cells <= 4L * RD_GRID_CELLS && reach < 1e12) {
        if (cells > h->comp_cells) {
            if (h->d_comp_list) (void)hipFree(h->d_comp_list);
            h->d_comp_list = nullptr;
            h->comp_cells = 0;
            SHIPCK(h, hipMalloc(&h->d_comp_list, sizeof(uint16_t) * RD_GRID_LIST * (size_t)cells));
            h->comp_cells = cells;
        }
        g->list = h->d_comp_list;
        hipLaunchKernelGGL(k_comp_grid, dim3((unsigned)((cells + 255) / 256)), dim3(256), pieces_lds(h), h->stream, *g,
                           (float)(1e-5 * reach), (const RdPiece*)h->d_pieces, h->npieces, h->d_comp_list);
        SHIPCK(h, hipGetLastError());
    }
    h->comp_built = *g;
    for (int d = 0; d < 3; ++d) { h->comp_lo[d] = box[d][0]; h->comp_hi[d] = box[d][1]; }
    h->comp_grid_set = true;
    h->comp_passes = 0;
    return RD_OK;
}

// persistent grid of k_mlp_points: one tile of 16 points per wave and round
static inline unsigned mlp_point_blocks(long m) { return (unsigned)std::min(((m + 15) / 16 + 3) / 4, 2048L); }

// the exact pass over the slots of some types
static auto* slots_kernel(const rd_system* h)
{
    return h->comp_sum ? k_composite_slots<true, false>
                       : (h->comp_allz ? k_composite_slots<false, true> : k_composite_slots<false, false>);
}

// external pass of the step (sorted slots -> gext)
void rd_host_launch_ext(rd_system* h)
{
    if (h->n <= 0) return;
    if (h->ext_mode == RD_EXT_SURROGATE) {
        unsigned blocks = std::min(h->ext_blocks[1] > 0 ? (unsigned)h->ext_blocks[1] : 2048u, nb256(h->n));
        hipLaunchKernelGGL(k_mlp_slots, dim3(blocks), dim3(256), 0, h->stream, (const RdMlpPack*)h->d_pack,
                           (const float4*)h->d_ps, h->n, h->mlp_norm, h->comp_mask, h->d_gext);
    } else if ((h->comp_mask & all_types(h)) == all_types(h)) {
        // (a composite on some of the types keeps the scan below: it is the
        // reference that the surrogate is trained for and timed against on
        // the cytosol's membrane, 64 replicas: scan 189 us, surrogate 91 us,
        // grid 64 us)
        if (h->comp_near.list)
            hipLaunchKernelGGL(k_composite_near, dim3(nb256(h->n)), dim3(256), 0, h->stream, h->d_ps, h->n,
                               h->comp_near, (const RdPiece*)h->d_pieces, h->npieces, h->d_gext);
        else
            hipLaunchKernelGGL(h->comp_sum ? k_composite_all<true> : k_composite_all<false>, dim3(nb256(h->n)), dim3(256),
                           pieces_lds(h), h->stream, h->d_ps, h->n, (const RdPiece*)h->d_pieces, h->npieces,
                           h->d_gext);
    } else {
        unsigned blocks = std::min(h->ext_blocks[0] > 0 ? (unsigned)h->ext_blocks[0] : 2048u, nb256(h->n));
        hipLaunchKernelGGL(slots_kernel(h), dim3(blocks), dim3(256), pieces_lds(h), h->stream, h->d_ps, h->n, (const RdPiece*)h->d_pieces, h->npieces,
                           h->comp_mask, h->d_gext);
    }
}

// before steps or gradients that make the external pass `passes` times: the
// pass takes the grid if it is there or is built now (`changed`: from now on)
int rd_host_ext_passes(rd_system* h, long passes, bool* changed)
{
    if (!h->ext_active() || h->ext_mode != RD_EXT_EXACT || (h->comp_mask & all_types(h)) != all_types(h) || h->comp_near.list)
        return RD_OK;
    const int rc = comp_grid(h, &h->comp_near, passes * passes_of(h->n), RD_GRID_SLOT_PIECES);
    if (changed) *changed = h->comp_near.list != nullptr;
    return rc;
}

// gext buffer sized for the current particle count; resident workgroups of
// the slot passes for the current piece count
int rd_host_ext_capacity(rd_system* h)
{
    if (!h->ext_active()) return RD_OK;
    h->comp_near.list = nullptr;
    const int rc = rd_host_ext_passes(h, 0, nullptr);
    if (rc) return rc;
    int per = 0;
    SHIPCK(h, hipOccupancyMaxActiveBlocksPerMultiprocessor(&per, (const void*)slots_kernel(h), 256,
                                                           pieces_lds(h)));
    h->ext_blocks[0] = std::max(per, 1) * h->ncu;
    SHIPCK(h, hipOccupancyMaxActiveBlocksPerMultiprocessor(&per, (const void*)k_mlp_slots, 256, 0));
    h->ext_blocks[1] = std::max(per, 1) * h->ncu;
    int need = h->n > 0 ? h->n : 1;
    if (need > h->gext_cap) {
        if (h->d_gext) (void)hipFree(h->d_gext);
        h->d_gext = nullptr;
        SHIPCK(h, hipMalloc(&h->d_gext, sizeof(float4) * need));
        h->gext_cap = need;
    }
    return RD_OK;
}

static void to_piece(const rd_pot1& q, RdPiece& p)
{
    memset(&p, 0, sizeof(p));
    double nn = std::sqrt((double)q.normal[0] * q.normal[0] + (double)q.normal[1] * q.normal[1] +
                          (double)q.normal[2] * q.normal[2]);
    for (int a = 0; a < 3; ++a) {
        p.o[a] = q.origin[a];
        p.n[a] = nn > 0 ? (float)(q.normal[a] / nn) : (a == 2 ? 1.0f : 0.0f);
    }
    p.R = q.radius;
    p.hh = q.type == RD_POT1_CYLINDER ? 0.5f * q.height : 0.0f;
    p.k = q.force_const;
    p.zaxis = (p.n[0] == 0.0f && p.n[1] == 0.0f && p.n[2] == 1.0f) ? 1 : 0;
}

extern "C" int rd_set_composite(rd_system* h, int n_pieces, const rd_pot1* pieces, uint32_t type_mask)
{
    if (!h || n_pieces < 0 || (n_pieces > 0 && !pieces)) return RD_EINVAL;
    if (n_pieces > RD_PIECES_MAX) return sset_err(h, RD_EINVAL, "too many composite pieces");
    static bool attr = false;
    if (!attr) {
        const int bytes = (int)(sizeof(RdPiece) * RD_PIECES_MAX);
        const void* fns[] = { (const void*)k_composite_slots<false, false>, (const void*)k_composite_slots<false, true>,
                              (const void*)k_composite_slots<true, false>, (const void*)k_composite_all<false>, (const void*)k_composite_all<true>,
                              (const void*)k_composite_points<false>, (const void*)k_composite_points<true>,
                              (const void*)k_sur_data<false, false>, (const void*)k_sur_data<true, false>,
                              (const void*)k_comp_grid };
        for (const void* f : fns) SHIPCK(h, hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, bytes));
        attr = true;
    }
    for (int i = 0; i < n_pieces; ++i) {
        const rd_pot1& q = pieces[i];
        if ((q.type != RD_POT1_DISK && q.type != RD_POT1_CYLINDER) || q.subtype != RD_SUB_ATTRACTIVE)
            return sset_err(h, RD_EINVAL, "composite pieces are attractive disks or cylinders");
    }
    SHIPCK(h, hipSetDevice(h->dev));
    std::vector<RdPiece> pc(n_pieces);
    for (int i = 0; i < n_pieces; ++i) to_piece(pieces[i], pc[i]);
    if (h->d_pieces) (void)hipFree(h->d_pieces);
    h->d_pieces = nullptr;
    if (n_pieces > 0) {
        SHIPCK(h, hipMalloc(&h->d_pieces, sizeof(RdPiece) * n_pieces));
        SHIPCK(h, hipMemcpy(h->d_pieces, pc.data(), sizeof(RdPiece) * n_pieces, hipMemcpyHostToDevice));
    }
    h->comp_grid_set = false;
    h->comp_passes = 0;
    h->comp_allz = std::all_of(pc.begin(), pc.end(), [](const RdPiece& p) { return p.zaxis != 0; });
    h->npieces = n_pieces;
    h->comp_mask = type_mask;
    h->comp.assign(pieces, pieces + n_pieces);
    h->dirty = true;
    return RD_OK;
}

extern "C" int rd_set_composite_combine(rd_system* h, int combine)
{
    if (!h || (combine != RD_COMBINE_NEAREST && combine != RD_COMBINE_SUM)) return RD_EINVAL;
    h->comp_sum = combine == RD_COMBINE_SUM;
    h->dirty = true;
    return RD_OK;
}

extern "C" int rd_set_external_mode(rd_system* h, int mode)
{
    if (!h || mode < RD_EXT_EXACT || mode > RD_EXT_SURROGATE) return RD_EINVAL;
    if (mode == RD_EXT_SURROGATE && !h->sur_ready) return sset_err(h, RD_ESTATE, "the surrogate has no weights");
    h->ext_mode = mode;
    h->dirty = true;
    return RD_OK;
}

// Points to the device, and results (a[na], then b[nb] in one device array; a
// null destination is left out) back, through pinned memory where it holds
// them; points_out waits for the stream.  Up to the smallest pinned buffer the
// results lie behind the points (at: where), beyond it they take the points'
// place, once the copy of the points is known to be done, a second wait of 10 us
// (one point of 16 pieces: 36.2 us a call with it, 26.6 without; pageable
// memory both ways, 33.8).
static hipError_t points_in(rd_system* h, float* dst, const float* src, long n, long nout, size_t* at)
{
    const size_t in = sizeof(float) * (size_t)n, both = in + sizeof(float) * (size_t)nout;
    *at = both <= RD_STAGE_MIN ? in : 0;
    char* stage = rd_host_stage(h, *at ? both : in);
    if (stage) memcpy(stage, src, in);
    return hipMemcpyAsync(dst, stage ? (const void*)stage : (const void*)src, in, hipMemcpyHostToDevice, h->stream);
}

static hipError_t points_out(rd_system* h, float* a, long na, float* b, long nb, const float* src, size_t at)
{
    hipError_t e = at ? hipSuccess : hipStreamSynchronize(h->stream);
    const size_t sa = sizeof(float) * (size_t)na, sb = sizeof(float) * (size_t)nb;
    char* stage = e == hipSuccess ? rd_host_stage(h, at + sa + sb) : nullptr;
    if (stage) stage += at;
    if (e == hipSuccess && stage) e = hipMemcpyAsync(stage, src, sa + sb, hipMemcpyDeviceToHost, h->stream);
    if (e == hipSuccess && !stage && a) e = hipMemcpyAsync(a, src, sa, hipMemcpyDeviceToHost, h->stream);
    if (e == hipSuccess && !stage && b) e = hipMemcpyAsync(b, src + na, sb, hipMemcpyDeviceToHost, h->stream);
    if (e == hipSuccess) e = hipStreamSynchronize(h->stream);
    if (e == hipSuccess && stage && a) memcpy(a, stage, sa);
    if (e == hipSuccess && stage && b) memcpy(b, stage + sa, sb);
    return e;
}

// exact composite at host points (test and data checks)
extern "C" int rd_composite_eval(rd_system* h, long m, const float* xyz, float* grad, float* energy)
{
    if (!h || m < 0 || (m > 0 && !xyz)) return RD_EINVAL;
    if (m == 0) return RD_OK;
    SHIPCK(h, hipSetDevice(h->dev));
    RdCompGrid g;
    const int rc = comp_grid(h, &g, passes_of(m), RD_GRID_POINT_PIECES);
    if (rc) return rc;
    float *dx = nullptr, *dg = nullptr;                 // positions; gradients, then energies
    SHIPCK(h, hipMalloc(&dx, sizeof(float) * 3 * m));
    hipError_t e = hipMalloc(&dg, sizeof(float) * 4 * m);
    size_t at = 0;
    if (e == hipSuccess) e = points_in(h, dx, xyz, 3 * m, 4 * m, &at);
    if (e == hipSuccess) {
        if (g.list)
            hipLaunchKernelGGL(k_composite_points_near, dim3(nb256(m)), dim3(256), 0, h->stream, dx, m, g,
                               (const RdPiece*)h->d_pieces, h->npieces, dg, dg + 3 * m);
        else
            hipLaunchKernelGGL(h->comp_sum ? k_composite_points<true> : k_composite_points<false>, dim3(nb256(m)),
                               dim3(256), pieces_lds(h), h->stream, dx, m, (const RdPiece*)h->d_pieces, h->npieces,
                               dg, dg + 3 * m);
        e = hipGetLastError();
    }
    if (e == hipSuccess) e = points_out(h, grad, 3 * m, energy, m, dg, at);
    (void)hipFree(dx);
    if (dg) (void)hipFree(dg);
    if (e != hipSuccess) return sset_err(h, RD_EHIP, std::string("composite eval: ") + hipGetErrorString(e));
    return RD_OK;
}

static int sur_alloc(rd_system* h)
{
    if (h->d_master) return RD_OK;
    SHIPCK(h, hipSetDevice(h->dev));
    SHIPCK(h, hipMalloc(&h->d_master, sizeof(float) * RD_MLP_NPARAM));
    SHIPCK(h, hipMalloc(&h->d_mom, sizeof(float) * RD_MLP_NPARAM));
    SHIPCK(h, hipMalloc(&h->d_vel, sizeof(float) * RD_MLP_NPARAM));
    SHIPCK(h, hipMalloc(&h->d_pack, sizeof(RdMlpPack)));
    SHIPCK(h, hipMalloc(&h->d_ctl, sizeof(RdTrainCtl)));
    SHIPCK(h, hipMalloc(&h->d_gscale, sizeof(float)));
    SHIPCK(h, hipMemset(h->d_pack, 0, sizeof(RdMlpPack)));    // zero padding rows of W4 / W4^T
    SHIPCK(h, hipMemset(h->d_ctl, 0, sizeof(RdTrainCtl)));
    if (!h->norm_set) {
        // default domain: the (first) box
        const double* lo = h->reps.empty() ? nullptr : h->reps[0].lo;
        for (int d = 0; d < 3; ++d) {
            double l = lo ? h->reps[0].lo[d] : h->prm.lattice_bounds[2 * d];
            double u = lo ? h->reps[0].hi[d] : h->prm.lattice_bounds[2 * d + 1];
            h->mlp_norm.lo[d] = (float)l;
            h->mlp_norm.sc[d] = (float)(2.0 / (u - l));
            h->norm_hi[d] = u;
        }
        h->mlp_norm.gscale = 1.0f;
    }
    return RD_OK;
}

static int sur_upload_master(rd_system* h, const std::vector<float>& w)
{
    SHIPCK(h, hipMemcpy(h->d_master, w.data(), sizeof(float) * RD_MLP_NPARAM, hipMemcpyHostToDevice));
    SHIPCK(h, hipMemset(h->d_mom, 0, sizeof(float) * RD_MLP_NPARAM));
    SHIPCK(h, hipMemset(h->d_vel, 0, sizeof(float) * RD_MLP_NPARAM));
    SHIPCK(h, hipMemset(h->d_ctl, 0, sizeof(RdTrainCtl)));
    hipLaunchKernelGGL(k_mlp_pack, dim3(nb256(RD_MLP_NPARAM)), dim3(256), 0, h->stream, h->d_master,
                       (RdMlpPack*)h->d_pack);
    SHIPCK(h, hipGetLastError());
    SHIPCK(h, hipStreamSynchronize(h->stream));
    h->sur_ready = true;
    return RD_OK;
}

// weights: uniform(-a, a) with a = sqrt(6 / fan_in) (He-uniform for SiLU), biases 0;
// host generator: splitmix64 of the seed
extern "C" int rd_surrogate_init(rd_system* h, uint64_t seed)
{
    if (!h) return RD_EINVAL;
    int rc = sur_alloc(h);
    if (rc) return rc;
    std::vector<float> w(RD_MLP_NPARAM, 0.0f);
    uint64_t st = seed;
    auto next = [&]() {
        uint64_t z = (st += 0x9E3779B97F4A7C15ull);
        z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
        z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
        z ^= z >> 31;
        return (double)(z >> 11) * (1.0 / 9007199254740992.0);
    };
    auto fill = [&](int off, int count, int fan_in) {
        double a = std::sqrt(6.0 / fan_in);
        for (int i = 0; i < count; ++i) w[off + i] = (float)((2.0 * next() - 1.0) * a);
    };
    fill(RD_MLP_W1, 192, 3);
    fill(RD_MLP_W2, 4096, 64);
    fill(RD_MLP_W3, 4096, 64);
    fill(RD_MLP_W4, 192, 64);
    return sur_upload_master(h, w);
}

extern "C" int rd_surrogate_set_weights(rd_system* h, const float* w)
{
    if (!h || !w) return RD_EINVAL;
    int rc = sur_alloc(h);
    if (rc) return rc;
    std::vector<float> v(w, w + RD_MLP_NPARAM);
    return sur_upload_master(h, v);
}

extern "C" int rd_surrogate_get_weights(rd_system* h, float* w)
{
    if (!h || !w) return RD_EINVAL;
    if (!h->d_master) return sset_err(h, RD_ESTATE, "no surrogate");
    SHIPCK(h, hipMemcpy(w, h->d_master, sizeof(float) * RD_MLP_NPARAM, hipMemcpyDeviceToHost));
    return RD_OK;
}

extern "C" int rd_surrogate_set_norm(rd_system* h, const double* lo, const double* hi, double gscale)
{
    if (!h || !lo || !hi || !(gscale > 0)) return RD_EINVAL;
    for (int d = 0; d < 3; ++d) {
        if (!(hi[d] > lo[d])) return RD_EINVAL;
        h->mlp_norm.lo[d] = (float)lo[d];
        h->mlp_norm.sc[d] = (float)(2.0 / (hi[d] - lo[d]));
        h->norm_hi[d] = hi[d];
    }
    h->mlp_norm.gscale = (float)gscale;
    h->norm_set = true;
    h->dirty = true;
    return RD_OK;
}

extern "C" int rd_surrogate_get_norm(rd_system* h, double* lo, double* hi, double* gscale)
{
    if (!h) return RD_EINVAL;
    for (int d = 0; d < 3; ++d) {
        if (lo) lo[d] = h->mlp_norm.lo[d];
        if (hi) hi[d] = h->norm_hi[d];
    }
    if (gscale) *gscale = h->mlp_norm.gscale;
    return RD_OK;
}

// m uniform positions in the domain (normalised) and the exact gradients there
static int launch_sur_data(rd_system* h, long m, uint64_t seed, float4* xn, float4* tg, double* bsum)
{
    const RdMlpNorm& nm = h->mlp_norm;
    float span[3];
    for (int d = 0; d < 3; ++d) span[d] = (float)(h->norm_hi[d] - nm.lo[d]);
    // Where more than a few samples fall outside the boxes nearly every wave scans
    // (a wave of 64 has all inside once in two at 1.1% outside), and no grid is
    // built for them; the scan of the grid's kernel is taken all the same.
    double box[3][2], in = 1.0;
    union_box(h, box);
    for (int d = 0; d < 3; ++d) {
        const double lo = nm.lo[d], hi = h->norm_hi[d];
        in *= std::max(0.0, std::min(hi, box[d][1]) - std::max(lo, box[d][0])) / (hi - lo);
    }
    const bool inside = in >= 0.99;
    RdCompGrid g;
    const int rc = comp_grid(h, &g, inside ? passes_of(m) : 0, RD_GRID_POINT_PIECES);
    if (rc) return rc;
    if (g.list || (!inside && !h->comp_sum && h->npieces >= RD_GRID_POINT_PIECES))
        hipLaunchKernelGGL((k_sur_data<false, true>), dim3(nb256(m)), dim3(256), 0, h->stream, m, seed, nm, span[0],
                           span[1], span[2], g, (const RdPiece*)h->d_pieces, h->npieces, xn, tg, bsum);
    else
        hipLaunchKernelGGL((h->comp_sum ? k_sur_data<true, false> : k_sur_data<false, false>), dim3(nb256(m)),
                           dim3(256), pieces_lds(h), h->stream, m, seed, nm, span[0], span[1], span[2], g,
                           (const RdPiece*)h->d_pieces, h->npieces, xn, tg, bsum);
    return RD_OK;
}

// training set: m uniform positions in the domain, exact composite gradients
// normalised by their RMS component (which becomes the output scale)
extern "C" int rd_surrogate_make_data(rd_system* h, long m, uint64_t seed, double* gscale)
{
    if (!h || m < 64) return RD_EINVAL;
    if (h->npieces <= 0) return sset_err(h, RD_ESTATE, "set the composite first");
    int rc = sur_alloc(h);
    if (rc) return rc;
    if (m > h->nsamples) {
        if (h->d_xn) (void)hipFree(h->d_xn);
        if (h->d_tg) (void)hipFree(h->d_tg);
        if (h->d_sbsum) (void)hipFree(h->d_sbsum);
        h->d_xn = h->d_tg = nullptr; h->d_sbsum = nullptr;
        SHIPCK(h, hipMalloc(&h->d_xn, sizeof(float4) * m));
        SHIPCK(h, hipMalloc(&h->d_tg, sizeof(float4) * m));
        SHIPCK(h, hipMalloc(&h->d_sbsum, sizeof(double) * nb256(m)));
    }
    h->nsamples = m;
    rc = launch_sur_data(h, m, seed, h->d_xn, h->d_tg, h->d_sbsum);
    if (rc) return rc;
    hipLaunchKernelGGL(k_sur_scale_sum, dim3(1), dim3(256), 0, h->stream, h->d_sbsum, (int)nb256(m), m, h->d_gscale);
    hipLaunchKernelGGL(k_sur_normalise, dim3(nb256(m)), dim3(256), 0, h->stream, h->d_tg, m, h->d_gscale);
    SHIPCK(h, hipGetLastError());
    float gs = 1.0f;
    SHIPCK(h, hipMemcpyAsync(&gs, h->d_gscale, sizeof(float), hipMemcpyDeviceToHost, h->stream));
    SHIPCK(h, hipStreamSynchronize(h->stream));
    h->mlp_norm.gscale = gs;
    if (gscale) *gscale = gs;
    return RD_OK;
}

static int ensure_partial(rd_system* h, int batch)
{
    const size_t rows = ((size_t)batch + 63) / 64;
    if (rows > h->partial_rows) {
        if (h->d_partial) (void)hipFree(h->d_partial);
        h->d_partial = nullptr;
        SHIPCK(h, hipMalloc(&h->d_partial, sizeof(float) * RD_MLP_ROW * rows));
        h->partial_rows = rows;
    }
    return RD_OK;
}

static void launch_train_step(rd_system* h, const float4* xn, const float4* tn, long m, int batch, int sequential,
                              uint64_t seed, const rd_train_params& tp, float* grad_out, int apply, float* loss_hist)
{
    const int rows = (batch + 63) / 64;
    const RdSchedule sch = { tp.lr, tp.lr_min, (long long)tp.steps, tp.beta1, tp.beta2 };
    hipLaunchKernelGGL(k_mlp_train, dim3(rows + 1), dim3(256), 0, h->stream, xn, tn, m,
                       ~(uint64_t)0 / (uint64_t)m, batch, sequential, seed, (const RdMlpPack*)h->d_pack,
                       (RdTrainCtl*)h->d_ctl, h->d_partial, sch);
    hipLaunchKernelGGL(k_mlp_adam, dim3((RD_MLP_NPARAM + 1 + 31) / 32), dim3(256), 0, h->stream, h->d_partial, rows,
                       h->d_master, h->d_mom, h->d_vel, (RdMlpPack*)h->d_pack, (RdTrainCtl*)h->d_ctl, tp.beta1,
                       tp.beta2, tp.eps, grad_out, apply, loss_hist);
}

// loss and gradient of one batch (no update): the gradient check entry
extern "C" int rd_surrogate_loss_grad(rd_system* h, long m, const float* xn, const float* tn, double* loss, float* grad)
{
    if (!h || m < 1 || !xn || !tn) return RD_EINVAL;
    if (!h->sur_ready) return sset_err(h, RD_ESTATE, "the surrogate has no weights");
    if (m > (1 << 22)) return sset_err(h, RD_EINVAL, "batch too large");
    int rc = ensure_partial(h, (int)m);
    if (rc) return rc;
    std::vector<float4> hx(m), ht(m);
    for (long i = 0; i < m; ++i) {
        hx[i] = make_float4(xn[3 * i], xn[3 * i + 1], xn[3 * i + 2], 0.f);
        ht[i] = make_float4(tn[3 * i], tn[3 * i + 1], tn[3 * i + 2], 0.f);
    }
    float4 *dx = nullptr, *dt = nullptr;
    float* dg = nullptr;
    SHIPCK(h, hipMalloc(&dx, sizeof(float4) * m));
    SHIPCK(h, hipMalloc(&dt, sizeof(float4) * m));
    SHIPCK(h, hipMalloc(&dg, sizeof(float) * RD_MLP_NPARAM));
    SHIPCK(h, hipMemcpyAsync(dx, hx.data(), sizeof(float4) * m, hipMemcpyHostToDevice, h->stream));
    SHIPCK(h, hipMemcpyAsync(dt, ht.data(), sizeof(float4) * m, hipMemcpyHostToDevice, h->stream));
    rd_train_params tp{};
    tp.steps = 1;
    launch_train_step(h, dx, dt, m, (int)m, 1, 0, tp, dg, 0, nullptr);
    hipError_t e = hipGetLastError();
    RdTrainCtl ctl{};
    if (e == hipSuccess && grad) e = hipMemcpyAsync(grad, dg, sizeof(float) * RD_MLP_NPARAM, hipMemcpyDeviceToHost, h->stream);
    if (e == hipSuccess) e = hipMemcpyAsync(&ctl, h->d_ctl, sizeof(ctl), hipMemcpyDeviceToHost, h->stream);
    if (e == hipSuccess) e = hipStreamSynchronize(h->stream);
    (void)hipFree(dx); (void)hipFree(dt); (void)hipFree(dg);
    if (e != hipSuccess) return sset_err(h, RD_EHIP, std::string("loss_grad: ") + hipGetErrorString(e));
    if (loss) *loss = ctl.loss;
    return RD_OK;
}

// Adam on the training set: tp.steps steps of tp.batch samples drawn with
// replacement (Philox of seed and step); loss per step into loss_curve
extern "C" int rd_surrogate_train(rd_system* h, const rd_train_params* tp, float* loss_curve)
{
    if (!h || !tp || tp->steps < 1 || tp->batch < 64 || tp->batch > (1 << 20)) return RD_EINVAL;
    if (!h->sur_ready) return sset_err(h, RD_ESTATE, "the surrogate has no weights");
    if (h->nsamples < 64) return sset_err(h, RD_ESTATE, "no training data");
    int rc = ensure_partial(h, tp->batch);
    if (rc) return rc;
    if ((size_t)tp->steps > h->loss_hist_cap) {
        if (h->d_loss_hist) (void)hipFree(h->d_loss_hist);
        h->d_loss_hist = nullptr;
        SHIPCK(h, hipMalloc(&h->d_loss_hist, sizeof(float) * tp->steps));
        h->loss_hist_cap = tp->steps;
    }
    SHIPCK(h, hipMemset(h->d_ctl, 0, sizeof(RdTrainCtl)));
    SHIPCK(h, hipMemset(h->d_mom, 0, sizeof(float) * RD_MLP_NPARAM));
    SHIPCK(h, hipMemset(h->d_vel, 0, sizeof(float) * RD_MLP_NPARAM));
    // two launches a step, 5 us of host time against 16 us on the GPU (a graph
    // of 64 steps took 0.7 ms to capture, instantiate and free)
    hipError_t e = hipSuccess;
    for (int done = 0; e == hipSuccess && done < tp->steps; ++done) {
        launch_train_step(h, h->d_xn, h->d_tg, h->nsamples, tp->batch, 0, tp->seed, *tp, nullptr, 1, h->d_loss_hist);
        e = hipGetLastError();
    }
    if (e == hipSuccess && loss_curve)
        e = hipMemcpyAsync(loss_curve, h->d_loss_hist, sizeof(float) * tp->steps, hipMemcpyDeviceToHost, h->stream);
    if (e == hipSuccess) e = hipStreamSynchronize(h->stream);
    if (e != hipSuccess) return sset_err(h, RD_EHIP, std::string("train: ") + hipGetErrorString(e));
    h->dirty = true;     // new packed weights: the captured step graphs stay valid (same buffers)
    return RD_OK;
}

// raw network outputs at normalised inputs
extern "C" int rd_surrogate_predict(rd_system* h, long m, const float* xn, float* y)
{
    if (!h || m < 0 || (m > 0 && (!xn || !y))) return RD_EINVAL;
    if (!h->sur_ready) return sset_err(h, RD_ESTATE, "the surrogate has no weights");
    if (m == 0) return RD_OK;
    float *dx = nullptr, *dout = nullptr;
    SHIPCK(h, hipMalloc(&dx, sizeof(float) * 3 * m));
    hipError_t e = hipMalloc(&dout, sizeof(float) * 3 * m);
    size_t at = 0;
    if (e == hipSuccess) e = points_in(h, dx, xn, 3 * m, 3 * m, &at);
    if (e == hipSuccess) {
        hipLaunchKernelGGL(k_mlp_points<3>, dim3(mlp_point_blocks(m)), dim3(256), 0, h->stream,
                           (const RdMlpPack*)h->d_pack, (const float*)dx, m, dout);
        e = hipGetLastError();
    }
    if (e == hipSuccess) e = points_out(h, y, 3 * m, nullptr, 0, dout, at);
    (void)hipFree(dx);
    if (dout) (void)hipFree(dout);
    if (e != hipSuccess) return sset_err(h, RD_EHIP, std::string("predict: ") + hipGetErrorString(e));
    return RD_OK;
}

// relative RMSE of the surrogate gradient against the exact composite on m
// fresh uniform samples: sqrt(sum |g_mlp - g|^2 / sum |g|^2)
extern "C" int rd_surrogate_validate(rd_system* h, long m, uint64_t seed, double* rel_rmse)
{
    if (!h || m < 64 || !rel_rmse) return RD_EINVAL;
    if (!h->sur_ready || h->npieces <= 0) return sset_err(h, RD_ESTATE, "composite and surrogate required");
    const unsigned nb = nb256(m);
    float4* d = nullptr;                             // positions, exact gradients, outputs
    double* bs = nullptr;                            // sums of each workgroup (two sets)
    SHIPCK(h, hipMalloc(&d, sizeof(float4) * 3 * m));
    hipError_t e = hipMalloc(&bs, sizeof(double) * 2 * nb);
    int rc = RD_OK;
    std::vector<double> sums(2 * (size_t)nb);
    if (e == hipSuccess) {
        float4 *dt = d + m, *dy = d + 2 * m;
        rc = launch_sur_data(h, m, seed, d, dt, bs);
        if (rc == RD_OK) {
            hipLaunchKernelGGL(k_mlp_points<4>, dim3(mlp_point_blocks(m)), dim3(256), 0, h->stream,
                               (const RdMlpPack*)h->d_pack, (const float*)d, m, (float*)dy);
            hipLaunchKernelGGL(k_sur_error, dim3(nb), dim3(256), 0, h->stream, dt, dy, m, (double)h->mlp_norm.gscale,
                               bs, bs + nb);
            e = hipGetLastError();
            if (e == hipSuccess)
                e = hipMemcpyAsync(sums.data(), bs, sizeof(double) * 2 * nb, hipMemcpyDeviceToHost, h->stream);
        }
        const hipError_t se = hipStreamSynchronize(h->stream);
        if (e == hipSuccess) e = se;
    }
    (void)hipFree(d);
    if (bs) (void)hipFree(bs);
    if (rc) return rc;
    if (e != hipSuccess) return sset_err(h, RD_EHIP, std::string("validate: ") + hipGetErrorString(e));
    double num = 0.0, den = 0.0;
    for (unsigned i = 0; i < nb; ++i) { num += sums[i]; den += sums[nb + i]; }
    *rel_rmse = den > 0 ? std::sqrt(num / den) : 0.0;
    return RD_OK;
}
