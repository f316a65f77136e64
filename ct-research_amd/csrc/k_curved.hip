// k_curved.hip - backprojection of the curved (cylindrical, equiangular)
// cone-beam FDK for gfx950 (My_toolbox/Implement_UnitedImaging_Data/
// ImplementUI.cu:80-153).
//
// The channel angle gamma = atan(u / (D - s)) and the in-plane source
// distance rho depend on (x, y, view) only, and the row coordinate
// xi = Dsd z / rho is linear in z.  A workgroup owns a tile of 16 x 16
// columns x TZ slices and loops over all views (the reference launches one
// kernel per view, ImplementUI.cu:333-339); a thread keeps its column's TZ
// sums in registers.  Per view the tile's detector footprint (a rectangle of
// channels x rows, computed once per geometry in FP64) is copied into LDS by
// the DMA path (buffer_load ... lds) while the previous view is
// interpolated from the other buffer, one barrier per view.  Per (column,
// view) a thread forms gamma, rho and the channel interpolation once; each
// voxel then costs a row coordinate, two LDS pair reads and its weight
// dbeta rho / L2^1.5.  Footprints too large for LDS read global memory.
//
// Bound by vector issue.  512 x 512 x 50 voxels, 800 views: 6.4 to 6.8 ms with
// 16 instructions and a reciprocal square root (a quarter of the rate) per
// voxel and view, and 89 per column and view shared by 10 slices; 5.2 ms with
// 13 per voxel where the footprint lies on the detector and the cone is thin,
// and about 60 per column shared by 25 slices.
#include "ctr_internal.h"

#include <algorithm>
#include <cmath>

namespace ctr {
namespace {

constexpr int kCvTX = 16, kCvTS = 16, kCvThreads = kCvTX * kCvTS;
// Floats per staged row, 96 or 128 by the footprint's channels, and per buffer
// (2 x 16 KiB of LDS per workgroup, five workgroups per CU: 42 or 32 rows)
constexpr int kCvNarrow = 96, kCvWide = 128, kCvCap = 4096;
enum { kCvEmpty = 1, kCvRowsIn = 2, kCvFits = 4 };
__host__ __device__ __forceinline__ int cv_pitch(int channels) { return channels <= kCvNarrow ? kCvNarrow : kCvWide; }
constexpr int kBufDword3 = 0x00020000;   // raw 32-bit buffer descriptor word 3 on gfx9

__device__ __forceinline__ int xcd_tile(int bid, int nwg)
{
    return (nwg & 7) == 0 ? (bid & 7) * (nwg >> 3) + (bid >> 3) : bid;
}

// Footprint of (tile, view): the channels between the extreme channel angles
// of the tile's corner columns (the level sets of gamma are rays from the
// source, so the extremes over the convex tile are at corners), and the rows
// between the extreme row coordinates xi = Dsd z / rho over the tile's slice
// range and its rho range (rho_min from the point of the tile nearest the
// source), both widened by a margin and by the bilinear neighbour.
__global__ __launch_bounds__(256) void k_curved_footprints(CurvedBpParams P, int4 *__restrict__ out)
{
    const long idx = (long)blockIdx.x * 256 + threadIdx.x;
    const long ntiles = (long)P.tiles_t * P.tiles_s * P.tiles_z;
    if (idx >= ntiles * P.nb) return;
    const int tile = (int)(idx / P.nb), b = (int)(idx % P.nb);
    const int tt = tile % P.tiles_t, rest = tile / P.tiles_t;
    const int ts = rest % P.tiles_s, tzi = rest / P.tiles_s;
    const int i_lo = tt * kCvTX, i_hi = min(i_lo + kCvTX - 1, P.nt - 1);
    const int j_lo = ts * kCvTS, j_hi = min(j_lo + kCvTS - 1, P.ns - 1);
    const int k_lo = tzi * P.tz, k_hi = k_lo + P.tz - 1;   // slices past nz too: computed, not written
    const double sb = P.view[2 * b], cb = P.view[2 * b + 1], D = P.D;
    const double x_lo = (i_lo + (double)P.off) * P.rt - P.ct, x_hi = (i_hi + (double)P.off) * P.rt - P.ct;
    const double y_lo = (j_lo + (double)P.off) * P.rs - P.cs, y_hi = (j_hi + (double)P.off) * P.rs - P.cs;
    double gmin = 1e300, gmax = -1e300, rho_max = 0.0;
    for (int c = 0; c < 4; ++c) {
        const double x = (c & 1) ? x_hi : x_lo, y = (c & 2) ? y_hi : y_lo;
        const double u = x * cb + y * sb, ds = D - (-x * sb + y * cb);
        const double gi = atan(u / ds) * P.g_scale + P.g_off;
        gmin = fmin(gmin, gi);
        gmax = fmax(gmax, gi);
        rho_max = fmax(rho_max, sqrt(u * u + ds * ds));
    }
    // the source (-D sin b, D cos b) clamped into the tile's box of column centres
    const double xs = -D * sb, ysrc = D * cb;
    const double dx = xs - fmin(fmax(xs, x_lo), x_hi), dy = ysrc - fmin(fmax(ysrc, y_lo), y_hi);
    const double rho_min = sqrt(dx * dx + dy * dy);
    const double z_lo = (k_lo + (double)P.off) * P.rz - P.cz, z_hi = (k_hi + (double)P.off) * P.rz - P.cz;
    double vmin = 1e300, vmax = -1e300;
    for (int c = 0; c < 4; ++c) {
        const double z = (c & 1) ? z_hi : z_lo, rho = (c & 2) ? rho_max : rho_min;
        const double v = (double)P.Dsd * z / rho * P.x_scale + P.x_off;
        vmin = fmin(vmin, v);
        vmax = fmax(vmax, v);
    }
    const double eu = 2e-3 + 4e-6 * fmax(fabs(gmin), fabs(gmax));
    const double ev = 2e-3 + 4e-6 * fmax(fabs(vmin), fabs(vmax));
    int flags = 0;
    if (!(gmax + eu >= 0.0 && gmin - eu < P.gmax)) flags |= kCvEmpty;   // every column skipped
    int c0 = (int)floor(fmax(gmin - eu, -1.0)), c1 = (int)floor(fmin(gmax + eu, (double)P.ng)) + 1;
    int r0 = (int)floor(fmax(vmin - ev, -1.0)), r1 = (int)floor(fmin(vmax + ev, (double)P.nx)) + 1;
    c0 = max(c0, 0);
    c1 = min(c1, P.ng - 1);
    r0 = max(r0, 0);
    r1 = min(r1, P.nx - 1);
    // at least 2 x 2 samples so that every clamped bilinear stencil is inside
    if (c1 <= c0) {
        if (c0 > 0) c0 = c1 - 1; else c1 = c0 + 1;
    }
    if (r1 <= r0) {
        if (r0 > 0) r0 = r1 - 1; else r1 = r0 + 1;
    }
    const int W = c1 - c0 + 1, H = r1 - r0 + 1;
    if (W <= kCvWide && H * cv_pitch(W) <= kCvCap) flags |= kCvFits;
    if (vmin - ev >= 0.0 && vmax + ev < P.xmax) flags |= kCvRowsIn;   // every row coordinate on the detector
    out[idx] = make_int4(c0, r0, W | (H << 16), flags);
}

// DMA copy of view b's footprint rows into buf: lane l of a wave copies
// channel c0 + l (clamped into the row) of row r into buf[r * pitch + l], and
// for footprints wider than 64 channels also c0 + 64 + l into
// buf[r * pitch + 64 + l] (as far as the pitch).  Offsets past the view read
// zero (hardware range check).
__device__ __forceinline__ void curved_issue(const float *__restrict__ filt, const CurvedBpParams &P, int b, int4 f,
                                             float *buf)
{
    if ((f.w & kCvEmpty) || !(f.w & kCvFits)) return;
    const int W = f.z & 0xffff, H = f.z >> 16, pitch = cv_pitch(W);
    const size_t view = (size_t)P.nx * P.ng;
    __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc((void *)(filt + (size_t)b * view), 0,
                                                                  (int)(view * sizeof(float)), kBufDword3);
    const int lane = (int)(threadIdx.x & 63);
    const unsigned v0 = (unsigned)min(f.x + lane, P.ng - 1) * 4u, v1 = (unsigned)min(f.x + 64 + lane, P.ng - 1) * 4u;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    for (int r = wave; r < H; r += kCvThreads / 64) {
        const unsigned roff = (unsigned)((f.y + r) * P.ng) * 4u;
        __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, buf + r * pitch, 4, v0, roff, 0, 0);
        if (W > 64 && lane < pitch - 64)
            __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, buf + r * pitch + 64, 4, v1, roff, 0, 0);
    }
}

// One column's TZ voxels of one view, every row coordinate (va + c vb) on the
// detector and z^2 / rho^2 < kCvThin: the two channels are interpolated in the
// row coordinate and weighted by wl and wr (dbeta / rho^2 times the channel
// weights) and by (1 + q)^-1.5, q = z^2 / rho^2, as its series to q^2 (the next
// term, 2.2 q^3, stays below 6e-8), with c1 and c2 the coefficients times
// 1 / rho^2 and 1 / rho^4.
constexpr float kCvThin = 0.003f;
template <int TZ>
__device__ __forceinline__ void curved_inside(const float *col, const float (&zz)[TZ], float va, float vb, float wl,
                                              float wr, float c1, float c2, float (&acc)[TZ])
{
    const char *base = reinterpret_cast<const char *>(col);
#pragma unroll
    for (int c = 0; c < TZ; ++c) {
        const float xi = fmaf((float)c, vb, va);
        const float fx = __builtin_amdgcn_fractf(xi);
        const float *q = reinterpret_cast<const float *>(base + __mul24((int)xi, kCvNarrow * 4));
        const float v0 = q[0], v1 = q[1], v2 = q[kCvNarrow], v3 = q[kCvNarrow + 1];
        const float val = fmaf(wr, fmaf(fx, v3 - v1, v1), wl * fmaf(fx, v2 - v0, v0));
        acc[c] = fmaf(val, fmaf(fmaf(c2, zz[c], c1), zz[c], 1.0f), acc[c]);
        if (c % 5 == 4) __builtin_amdgcn_sched_barrier(0);   // five voxels' reads at a time (registers)
    }
}

// Blocks of grid row s > 0 take the s-th share of `share` views and the s-th
// of the partial volumes (bp_share).
template <int TZ>
__global__ __launch_bounds__(kCvThreads, 5) void k_curved_tiled(const float *__restrict__ filt, float *__restrict__ vol,
                                                             const float *__restrict__ views, CurvedBpParams P, int share)
{
    __shared__ float lds[2][kCvCap];
    const int tile = xcd_tile(blockIdx.x, gridDim.x);
    const int tt = tile % P.tiles_t, rest = tile / P.tiles_t;
    const int ts = rest % P.tiles_s, tzi = rest / P.tiles_s;
    const int i = tt * kCvTX + (threadIdx.x & (kCvTX - 1)), j = ts * kCvTS + (threadIdx.x / kCvTX);
    const int k0 = tzi * TZ;
    const bool col_in = i < P.nt && j < P.ns;
    const float x = ((float)i + P.off) * P.rt - P.ct, y = ((float)j + P.off) * P.rs - P.cs;
    const float z0 = ((float)k0 + P.off) * P.rz - P.cz;
    float zz[TZ], acc[TZ], zmax = 0.0f;
#pragma unroll
    for (int c = 0; c < TZ; ++c) {
        const float z = ((float)(k0 + c) + P.off) * P.rz - P.cz, z2 = z * z;
        // uniform: in a scalar register
        zz[c] = __builtin_bit_cast(float, __builtin_amdgcn_readfirstlane(__builtin_bit_cast(int, z2)));
        zmax = fmaxf(zmax, z2);
        acc[c] = 0.0f;
    }
    const int ng = P.ng;
    const size_t view_elems = (size_t)P.nx * ng;
    const unsigned row_bytes = (unsigned)ng * 4u;
    const float xlast = __builtin_bit_cast(float, __builtin_bit_cast(int, P.xmax) - 1);   // largest float below xmax
    const int4 *ft = P.foot + (size_t)tile * P.nb;
    const int b0 = blockIdx.y * share, b1 = min(b0 + share, P.nb);

    int4 fn = ft[b0];
    curved_issue(filt, P, b0, fn, lds[b0 & 1]);
    for (int b = b0; b < b1; ++b) {
        const int4 f = fn;
        const float *buf = lds[b & 1];
        // this wave's copies of view b are complete; after the barrier every
        // wave's are, and no wave still reads the other buffer (view b-1)
        __builtin_amdgcn_s_waitcnt(0);
        __syncthreads();
        if (b + 1 < b1) {
            fn = ft[b + 1];
            curved_issue(filt, P, b + 1, fn, lds[(b + 1) & 1]);
        }
        if ((f.w & kCvEmpty) || !col_in) continue;
        const float sb = views[2 * b], cb = views[2 * b + 1];
        const float u = fmaf(x, cb, y * sb), s = fmaf(-x, sb, y * cb);
        // source (-D sin b, D cos b, 0): in-plane distance^2 = u^2 + (D - s)^2
        const float ds = P.D - s;
        const float rho2 = fmaf(u, u, ds * ds);
        const float tg = u * __builtin_amdgcn_rcpf(ds);
        // atan by fan_atan where every lane is inside its range, as in a usual fan
        const float gi = fmaf(__all(fabsf(tg) < kFanAtanMax) ? fan_atan(tg) : atanf(tg), P.g_scale, P.g_off);
        if (!(gi >= 0.0f && gi < P.gmax)) continue;
        const int i0 = min((int)gi, ng - 2);
        const float fg = gi - (float)i0;
        const float inv_rho = __builtin_amdgcn_rsqf(rho2), iq = inv_rho * inv_rho;
        const float xs = P.Dsd * inv_rho * P.x_scale;   // row coordinate per unit z
        const bool fits = (f.w & kCvFits) != 0;
        const int pitch = cv_pitch(f.z & 0xffff);
        const float *col = buf + (i0 - f.x) - f.y * pitch;
        if (fits && pitch == kCvNarrow && (f.w & kCvRowsIn) && __all(zmax * iq < kCvThin)) {
            const float w = P.dbeta * iq, wr = w * fg;
            curved_inside<TZ>(col, zz, fmaf(z0, xs, P.x_off), P.rz * xs, w - wr, wr, -1.5f * iq, 1.875f * iq * iq, acc);
            continue;
        }
        const float wb = P.dbeta * rho2 * inv_rho;
        // rows are clamped into the detector and out-of-range voxels get weight
        // 0; the clamped stencil lies in the footprint, whose rows reach the
        // detector edge whenever a sample leaves it.  A footprint larger than
        // an LDS buffer reads pairs from global memory (32-bit byte offsets
        // from the view's uniform base).
        const float *Fv = filt + (size_t)b * view_elems;
        float kf = (float)k0;
        asm volatile("" : "+v"(kf));   // the slices' z are formed here, not kept in registers
        auto clamped = [&](auto pairs) {
#pragma unroll
            for (int c = 0; c < TZ; ++c) {
                const float z = ((kf + (float)c) + P.off) * P.rz - P.cz;
                const float xi = fmaf(z, xs, P.x_off);
                const float xcl = __builtin_amdgcn_fmed3f(xi, 0.0f, xlast);
                const bool in = xi == xcl;
                const float fxs = __builtin_amdgcn_fractf(xcl);
                float2 p0, p1;
                pairs((int)xcl, p0, p1);
                const float a = fmaf(fg, p0.y - p0.x, p0.x);
                const float bq = fmaf(fg, p1.y - p1.x, p1.x);
                // weight dbeta rho / L2^1.5 (ImplementUI.cu:145: / L2 * dbeta / (sqrt(L2) / rho))
                const float r = __builtin_amdgcn_rsqf(fmaf(z, z, rho2));
                float w = wb * (r * r * r);
                // the weight is formed for every lane (no branch around it),
                // four voxels' reads at a time (registers)
                asm("" : "+v"(w));
                acc[c] = fmaf(fmaf(fxs, bq - a, a), in ? w : 0.0f, acc[c]);
                if (c % 4 == 3) __builtin_amdgcn_sched_barrier(0);
            }
        };
        if (fits)
            clamped([&](int j0, float2 &p0, float2 &p1) {
                const float *q = col + __mul24(j0, pitch);
                p0 = make_float2(q[0], q[1]);
                p1 = make_float2(q[pitch], q[pitch + 1]);
            });
        else
            clamped([&](int j0, float2 &p0, float2 &p1) {   // 4-byte aligned pairs
                const unsigned ob = (unsigned)(j0 * ng + i0) * 4u;
                __builtin_memcpy(&p0, reinterpret_cast<const char *>(Fv) + ob, sizeof p0);
                __builtin_memcpy(&p1, reinterpret_cast<const char *>(Fv) + (ob + row_bytes), sizeof p1);
            });
    }
    if (!col_in) return;
    vol += blockIdx.y * ((size_t)P.nt * P.ns * P.nz);
#pragma unroll
    for (int c = 0; c < TZ; ++c) {
        const int k = k0 + c;
        if (k < P.nz) {
            const size_t o = ((size_t)k * P.ns + j) * P.nt + i;
            vol[o] = P.accumulate ? vol[o] + acc[c] : acc[c];
        }
    }
}

// Staged rows of the largest footprint with tiles of tz slices, over the
// distances from the source of the columns inside the fan.
int cv_rows(const CurvedBpParams &P, int tz)
{
    const double g0 = -P.g_off / P.g_scale, g1 = (P.gmax - P.g_off) / P.g_scale;   // the end channels' angles
    const double half = std::min(std::hypot(0.5 * P.nt * P.rt, 0.5 * P.ns * P.rs),
                                 P.D * std::sin(std::min(std::max(std::fabs(g0), std::fabs(g1)), 1.57)));
    const double near = std::max(P.D - half, 1e-3 * P.D), far = P.D + half;
    int most = 0;
    for (int k0 = 0; k0 < P.nz; k0 += tz) {
        double v0 = 1e300, v1 = -1e300;
        for (int c = 0; c < 4; ++c) {
            const double z = ((c & 1 ? std::min(k0 + tz, P.nz) - 1 : k0) + (double)P.off) * P.rz - P.cz;
            const double v = P.Dsd * z / (c & 2 ? near : far) * P.x_scale + P.x_off;
            v0 = std::min(v0, v);
            v1 = std::max(v1, v);
        }
        const double lo = std::max(v0, 0.0), hi = std::min(v1 + 2.0, (double)P.nx);
        most = std::max(most, (int)std::min(std::max(hi - lo, 0.0), 1e6));
    }
    return most;
}

// Blocks that the chip holds at a time (five of 32 KiB of LDS per CU).
constexpr long kCvBlocks = 1280;

// z depth of a tile: the per-view column set-up (about 55 instructions) is
// shared by the tile's slices (about 15 each; 45 where the footprints exceed
// LDS); slices past nz are wasted work.  More than 8 slices only where tiles and
// sets of views still fill the chip: of few views a block's time is what counts
// (258 x 121 x 56, 12 views: 31 us with 8 slices, 36 us with 20; 117 x 4 x 46, 7
// views: 17 and 25 us).
int choose_tz(const CurvedBpParams &P)
{
    static const int cand[] = {4, 6, 8, 10, 12, 16, 20, 25, 32};
    const long columns = (long)((P.nt + kCvTX - 1) / kCvTX) * ((P.ns + kCvTS - 1) / kCvTS);
    int best = 8;
    long best_cost = -1;
    for (int tz : cand) {
        const long tiles_z = (P.nz + tz - 1) / tz, tiles = columns * tiles_z;
        const int share = bp_share(tiles, P.nb, (size_t)P.nt * P.ns * P.nz);
        if (tz > 8 && tiles * ((P.nb + share - 1) / share) < kCvBlocks) continue;
        const long each = cv_rows(P, tz) * kCvNarrow <= kCvCap ? 15 : 45;
        const long cost = tiles_z * (55 + each * tz);
        if (best_cost < 0 || cost < best_cost) {
            best = tz;
            best_cost = cost;
        }
    }
    return best;
}

template <int TZ>
hipError_t launch_tz(const CurvedBpParams &P, const float *filt, float *vol, int share, hipStream_t st)
{
    const dim3 grid(P.tiles_t * P.tiles_s * P.tiles_z, (P.nb + share - 1) / share);
    hipLaunchKernelGGL((k_curved_tiled<TZ>), grid, dim3(kCvThreads), 0, st, filt, vol, P.view, P, share);
    return hipGetLastError();
}

}  // namespace

size_t curved_plan(CurvedBpParams &P)
{
    P.tz = choose_tz(P);
    P.tiles_t = (P.nt + kCvTX - 1) / kCvTX;
    P.tiles_s = (P.ns + kCvTS - 1) / kCvTS;
    P.tiles_z = (P.nz + P.tz - 1) / P.tz;
    return (size_t)P.tiles_t * P.tiles_s * P.tiles_z * P.nb;
}

hipError_t launch_curved_footprints(const CurvedBpParams &P, int4 *foot, hipStream_t st)
{
    const long n = (long)P.tiles_t * P.tiles_s * P.tiles_z * P.nb;
    hipLaunchKernelGGL(k_curved_footprints, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, P, foot);
    return hipGetLastError();
}

int curved_splits(const CurvedBpParams &P)
{
    const int share = bp_share((long)P.tiles_t * P.tiles_s * P.tiles_z, P.nb, (size_t)P.nt * P.ns * P.nz);
    return (P.nb + share - 1) / share;
}

hipError_t launch_curved_bp(const CurvedBpParams &Pin, const float *filt, float *vol, float *parts, hipStream_t st)
{
    if (!Pin.foot) return hipErrorInvalidValue;
    CurvedBpParams P = Pin;
    const int splits = parts ? curved_splits(P) : 1;
    const int share = splits > 1 ? bp_share((long)P.tiles_t * P.tiles_s * P.tiles_z, P.nb, (size_t)P.nt * P.ns * P.nz) : P.nb;
    float *dst = splits > 1 ? parts : vol;
    if (splits > 1) P.accumulate = 0;
    hipError_t e = hipErrorInvalidValue;
    switch (P.tz) {
    case 4: e = launch_tz<4>(P, filt, dst, share, st); break;
    case 6: e = launch_tz<6>(P, filt, dst, share, st); break;
    case 8: e = launch_tz<8>(P, filt, dst, share, st); break;
    case 10: e = launch_tz<10>(P, filt, dst, share, st); break;
    case 12: e = launch_tz<12>(P, filt, dst, share, st); break;
    case 16: e = launch_tz<16>(P, filt, dst, share, st); break;
    case 20: e = launch_tz<20>(P, filt, dst, share, st); break;
    case 25: e = launch_tz<25>(P, filt, dst, share, st); break;
    case 32: e = launch_tz<32>(P, filt, dst, share, st); break;
    default: break;
    }
    if (e != hipSuccess || splits == 1) return e;
    return launch_sum_parts(parts, splits, (size_t)P.nt * P.ns * P.nz, vol, Pin.accumulate, st);
}

}  // namespace ctr
