// k_forward.hip - Siddon ray-driven forward projector for gfx950.
//
// One thread per ray (view, row, column); all views in one launch.  A block
// is 64 columns x 4 rows of one view, so a wavefront holds 64 neighbouring,
// nearly parallel rays that walk neighbouring voxels (shared cache lines).
//
// Per ray the entry/exit of the volume box, the first crossing of each axis
// and the crossing counts are computed in FP64 (near-parallel rays need it).
// The traversal runs in FP32: the next crossing of each axis is formed as
// first + count * step with one fma (no accumulated drift), and the axis
// whose plane comes first advances with selects rather than branches, so a
// wavefront never splits three ways.  The loop runs the FP64 setup's crossing
// count and the last segment ends at the exit parameter.  The volume is read
// through a range-checked buffer descriptor.  (The system-matrix walk keeps
// FP64 parameters: it is an export, not a hot loop.)
//
// Geometry: ProjectionCone_3D.cu:26-42 (source, end point at 2D along the
// ray through (p, xi) of the virtual isocentre detector); segment weight is
// the intersection length in mm, as the reference's :311-356.
#include "ctr_internal.h"

#include <algorithm>
#include <cmath>
#include <cstdlib>

namespace ctr {
namespace {

constexpr int kBX = 64, kBY = 4;
// detector columns per wavefront: a block covers 64 columns x 4 rows, and a
// wavefront 16 columns of all 4 rows (wave w: columns 16 w ..).  At oblique
// views the rays of one row reach the same D plane at heights that spread
// with the column, so a wider row span touches more z slices per gather:
// 16 x 4 measured 18.7 ms at 256^3 / 360 views and 257 ms at 512^3 / 720,
// 32 x 2 18.8 / 259 ms, 64 x 1 19.1 / 266 ms
constexpr int kWaveCols = 16;
static_assert(kWaveCols != 16 || (kBX == 64 && kBY == 4), "16-column wavefronts of 4 rows tile a 64 x 4 block");
static_assert(kWaveCols != 32 || (kBX == 64 && kBY % 2 == 0), "32-column wavefronts of 2 rows need an even block height");

// Column and row of this thread's ray within its block.
__device__ __forceinline__ void ray_of_thread(int &dcol, int &drow)
{
    if (kWaveCols == 32) {
        const int wave = threadIdx.y, lane = threadIdx.x;   // blockDim.x = 64: one wavefront per y
        dcol = (wave & 1) * 32 + (lane & 31);
        drow = (wave >> 1) * 2 + (lane >> 5);
    } else if (kWaveCols == 16) {
        const int wave = threadIdx.y, lane = threadIdx.x;
        dcol = wave * 16 + (lane & 15);
        drow = lane >> 4;
    } else {
        dcol = threadIdx.x;
        drow = threadIdx.y;
    }
}

struct AxisSetup {
    int i0, n;        // start index, number of plane crossings
    double next0;     // first crossing, relative to the entry parameter
    double step;      // parameter step between crossings
    int stride;       // signed index stride
};

__device__ __forceinline__ AxisSetup setup_axis(double s, double d, double lam_in, double lam_out, double r, int nvox,
                                                int stride)
{
    AxisSetup a;
    const double xin = (s + lam_in * d) / r, xout = (s + lam_out * d) / r;
    if (d > 0.0) {
        int i0 = (int)floor(xin), i1 = (int)ceil(xout) - 1;
        i0 = min(max(i0, 0), nvox - 1);
        i1 = min(max(i1, i0), nvox - 1);
        a.i0 = i0;
        a.n = i1 - i0;
        a.next0 = ((i0 + 1) * r - s) / d - lam_in;
        a.step = r / d;
        a.stride = stride;
    } else if (d < 0.0) {
        int i0 = (int)ceil(xin) - 1, i1 = (int)floor(xout);
        i0 = min(max(i0, 0), nvox - 1);
        i1 = max(min(i1, i0), 0);
        a.i0 = i0;
        a.n = i0 - i1;
        a.next0 = (i0 * r - s) / d - lam_in;
        a.step = -r / d;
        a.stride = -stride;
    } else {
        a.i0 = min(max((int)floor(xin), 0), nvox - 1);
        a.n = 0;
        a.next0 = __builtin_huge_val();
        a.step = 0.0;
        a.stride = 0;
    }
    return a;
}

constexpr int kBufDword3 = 0x00020000;   // raw 32-bit buffer descriptor word 3 on gfx9

// Slab clip of the ray s + lam*d against [0, b]; returns false on a miss.
__device__ __forceinline__ bool clip_axis(double s, double d, double b, double &lo, double &hi)
{
    if (d == 0.0) return s >= 0.0 && s < b;
    const double inv = 1.0 / d;
    const double t1 = -s * inv, t2 = (b - s) * inv;
    lo = fmax(lo, fmin(t1, t2));
    hi = fmin(hi, fmax(t1, t2));
    return true;
}

// Walk of one ray through the volume: per-axis crossings after the entry
// point, the exit parameter and the first voxel.
struct RayWalk {
    AxisSetup at, as, az;
    double lam_end;   // chord length through the volume box
    int idx0;         // first voxel (in the layout the strides describe)
};

// Set-up of ray (view ib, column ip, row ix); false on a miss.  With tr the
// t and s strides are those of a [z][t][s] copy of the volume.
__device__ __forceinline__ bool ray_walk(const RayParams &g, int ib, int ip, int ix, bool tr, RayWalk &w)
{
    const double sb = g.view[4 * ib + 0], cb = g.view[4 * ib + 1];
    const double P = g.p[ip], X = g.xi[ix];
    double st, ss, dx, dy, dz;
    if (g.parallel) {
        // foot point of the line and its unit direction (ProjectionParallel_2D.cu:22-28)
        st = 0.5 * g.bt + P * cb;
        ss = 0.5 * g.bs + P * sb;
        dx = -sb;
        dy = cb;
        dz = 0.0;
    } else {
        st = g.view[4 * ib + 2];
        ss = g.view[4 * ib + 3];
        dx = P * cb + g.D * sb;
        dy = P * sb - g.D * cb;
        dz = X;
        const double inv_n = 1.0 / sqrt(dx * dx + dy * dy + dz * dz);
        dx *= inv_n;
        dy *= inv_n;
        dz *= inv_n;
    }
    double lo = -__builtin_huge_val(), hi = __builtin_huge_val();
    bool hit = clip_axis(st, dx, g.bt, lo, hi);
    hit = clip_axis(ss, dy, g.bs, lo, hi) && hit;
    hit = clip_axis(g.sz, dz, g.bz, lo, hi) && hit;
    if (!hit || !(hi > lo)) return false;
    const int st_t = tr ? g.ns : 1, st_s = tr ? 1 : g.nt;
    w.at = setup_axis(st, dx, lo, hi, g.rt, g.nt, st_t);
    w.as = setup_axis(ss, dy, lo, hi, g.rs, g.ns, st_s);
    w.az = setup_axis(g.sz, dz, lo, hi, g.rz, g.nz, g.nt * g.ns);
    w.lam_end = hi - lo;
    w.idx0 = w.az.i0 * (g.nt * g.ns) + w.as.i0 * st_s + w.at.i0 * st_t;
    return true;
}

// Minimum / maximum of an int over the wavefront; every lane must be active.
__device__ __forceinline__ int wave_min_int(int v)
{
    for (int m = 32; m > 0; m >>= 1) v = min(v, __shfl_xor(v, m, 64));
    return v;
}
__device__ __forceinline__ int wave_max_int(int v)
{
    for (int m = 32; m > 0; m >>= 1) v = max(v, __shfl_xor(v, m, 64));
    return v;
}

// min(a, b) for finite or infinite operands as one v_med3 (no NaN quieting).
// ninf is -inf held in a register the compiler cannot see through
// (opaque_ninf): with a literal -inf it rewrites the med3 as an IEEE min and
// re-canonicalises every operand defined outside the loop on every slab.
__device__ __forceinline__ float min_nc(float a, float b, float ninf)
{
    return __builtin_amdgcn_fmed3f(a, b, ninf);
}
__device__ __forceinline__ float opaque_ninf()
{
    float v;
    asm volatile("v_mov_b32 %0, 0xff800000" : "=v"(v));
    return v;
}

__device__ __forceinline__ float load_vox(__amdgpu_buffer_rsrc_t rs, unsigned off)
{
    return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rs, off, 0, 0));
}

// One crossing at a time: the axis whose plane comes first advances (t
// before s before z on ties).  The c-th crossing of an axis is first +
// c * step, one rounding each (an accumulated next += step drifts by the
// square root of the crossing count in ulps).  Parameters are relative to
// the entry point, so they stay below the chord length.
__device__ __forceinline__ float walk_crossings(__amdgpu_buffer_rsrc_t rs, const RayWalk &w)
{
    const float inf = __builtin_huge_valf();
    const float t0 = w.at.n > 0 ? (float)w.at.next0 : inf, dt = (float)w.at.step;
    const float s0 = w.as.n > 0 ? (float)w.as.next0 : inf, ds = (float)w.as.step;
    const float z0 = w.az.n > 0 ? (float)w.az.next0 : inf, dz = (float)w.az.step;
    // byte strides; negative ones wrap, as unsigned offsets do
    const unsigned bt_st = (unsigned)w.at.stride * 4u, bs_st = (unsigned)w.as.stride * 4u,
                   bz_st = (unsigned)w.az.stride * 4u;
    float nt = t0, ns = s0, nz = z0, ct = 0.0f, cs = 0.0f, cz = 0.0f;   // crossings passed per axis
    unsigned off = (unsigned)w.idx0 * 4u;
    float lam = 0.0f, acc = 0.0f;
    // every counted crossing ends a segment; the last segment ends at the exit
    const int crossings = w.at.n + w.as.n + w.az.n;
    for (int k = 0; k < crossings; ++k) {
        const bool bt = nt <= ns && nt <= nz;
        const bool bs = !bt && ns <= nz;
        const float m = bt ? nt : (bs ? ns : nz);
        acc = fmaf(m - lam, load_vox(rs, off), acc);
        lam = m;
        off += bt ? bt_st : (bs ? bs_st : bz_st);
        ct = bt ? ct + 1.0f : ct;
        cs = bs ? cs + 1.0f : cs;
        cz = (!bt && !bs) ? cz + 1.0f : cz;
        nt = fmaf(ct, dt, t0);
        ns = fmaf(cs, ds, s0);
        nz = fmaf(cz, dz, z0);
    }
    return fmaf((float)w.lam_end - lam, load_vox(rs, off), acc);
}

// Line integral of one ray; also returns the chord length of the ray
// through the volume box (the row sum A*1 of the Siddon system matrix).
// Every lane of the wavefront must call it (valid false for lanes without a
// ray): the wavefront decides together how it walks.
//
// A wavefront holds 64 neighbouring rays of one detector row.  When, for all
// of them, the in-plane axis D that the view runs along has the shortest
// crossing step (by 0.1%, so float rounding cannot put two crossings of
// another axis between two D planes), the rays walk D's slabs in lockstep:
// at iteration u every ray is in the same absolute slab, so the wavefront's
// loads fall on a few neighbouring cache lines (one row of the layout whose
// fastest axis is the other in-plane axis).  In a slab a ray crosses each
// other axis at most once, so the slab is at most three segments: before
// the first crossing, between the two, after the second.  The segments and
// voxels are those of the one-crossing-at-a-time walk, which the other
// wavefronts run.  No crossing within rounding of the exit is taken that the
// FP64 set-up did not count, so no weighted load falls outside the volume
// (where the two layouts differ).
//
// kSkip: the second and third voxels of a slab are read only by the lanes whose
// segment there is not empty, which shortens the gathers, and four slabs are
// taken at a time where they lie on every ray.  The sums are the same bit for
// bit for finite volumes (a skipped term is 0 * v; an infinite v would make it
// NaN).  Slab by slab with all reads / kSkip, projection of 2n x 2n rays a view
// and SIRT step: 416^3, 30 views 7.8 / 5.4 and 13.0 / 11.3 ms; 256^3, 90 views
// 4.5 / 3.6 and 7.9 / 7.1 ms; 128^3, 90 views 559 / 490 and 1058 / 981 us;
// 96^3, 90 views 245 / 226 and 527 / 502 us; 80^3 155 / 154 and 396 / 391 us; 64^3 89 /
// 91 and 299 / 301 us; 32^3, 60 views 18 / 20 us, so from 2^19 voxels on.  It takes
// 72 registers (seven wavefronts per SIMD) for 51; six slabs at a time measured
// 8% more than four, masks without the blocks 2% more than neither.
constexpr int kSlabs = 4;
template <bool kSkip>
__device__ __forceinline__ float trace_ray(const float *__restrict__ vol, const RayParams &g, int ib, int ip, int ix,
                                           bool valid, float &chord)
{
    // views whose central ray runs mostly along t read the [z][t][s] copy, so
    // that the neighbouring rays of a wavefront (neighbouring p, offset in s)
    // gather from neighbouring addresses
    const bool along_t = fabs(g.view[4 * ib + 0]) > fabs(g.view[4 * ib + 1]);
    const bool tr = g.volT != nullptr && along_t;
    RayWalk w;
    const bool hit = valid && ray_walk(g, ib, ip, ix, tr, w);
    chord = hit ? (float)w.lam_end : 0.0f;

    // num_records is 32 bits: 2^30 voxels (4 GiB) saturate to 2^32 - 1, above every valid offset
    const size_t vbytes = (size_t)g.nt * g.ns * g.nz * sizeof(float);
    const unsigned nbytes = vbytes > 0xFFFFFFFFull ? 0xFFFFFFFFu : (unsigned)vbytes;
    // base and size are the same for the whole block (one view of one
    // problem); stating it keeps the descriptor in scalar registers where the
    // compiler cannot prove it (the batched kernels read them from a job
    // table).  readfirstlane returns int: each half goes through unsigned, so
    // the low half is zero-extended, not sign-extended into the high one.
    const unsigned long long base = (unsigned long long)(tr ? g.volT : vol);
    const unsigned hi = (unsigned)__builtin_amdgcn_readfirstlane((unsigned)(base >> 32));
    const unsigned lo = (unsigned)__builtin_amdgcn_readfirstlane((unsigned)base);
    const unsigned long long ubase = ((unsigned long long)hi << 32) | (unsigned long long)lo;
    __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(
        (void *)ubase, 0, (int)__builtin_amdgcn_readfirstlane(nbytes), kBufDword3);

    // lockstep slabs: D is t or s by the view, A the other in-plane axis, B = z
    const AxisSetup aD = along_t ? w.at : w.as;
    const AxisSetup aA = along_t ? w.as : w.at;
    const AxisSetup &aB = w.az;
    bool ok = true;
    if (hit) {
        const double lim = 1.001 * aD.step;
        ok = aD.stride != 0 && (aA.n == 0 || aA.step >= lim) && (aB.n == 0 || aB.step >= lim);
    }
    const unsigned long long bad = __ballot(hit && !ok);
    const unsigned long long up = __ballot(hit && aD.stride > 0), down = __ballot(hit && aD.stride < 0);
    if (bad != 0 || (up != 0 && down != 0)) return hit ? walk_crossings(rs, w) : 0.0f;

    // wavefront-relative slab index u: absolute D index istart + dir * u
    const int dir = up != 0 ? 1 : -1;
    const int first = hit ? aD.i0 : (dir > 0 ? 0x7fffffff : -0x7fffffff);
    const int istart = dir > 0 ? wave_min_int(first) : wave_max_int(first);
    // this ray's first slab, >= 0; a lane without a hit starts 2^30 slabs
    // late, so its k = u - o never enters [0, nD]
    const int o = hit ? dir * (aD.i0 - istart) : (1 << 30);
    const int uend = __builtin_amdgcn_readfirstlane(wave_max_int(hit ? o + aD.n : -1));   // uniform
    const int nD = hit ? aD.n : 0;

    const float inf = __builtin_huge_valf();
    const float D0 = hit ? (float)aD.next0 : inf, dD = hit ? (float)aD.step : 0.0f;
    const float A0 = hit && aA.n > 0 ? (float)aA.next0 : inf, dA = hit ? (float)aA.step : 0.0f;
    const float B0 = hit && aB.n > 0 ? (float)aB.next0 : inf, dB = hit ? (float)aB.step : 0.0f;
    const float lend = hit ? (float)w.lam_end : 0.0f;
    // 8 ulps below the exit: the float crossings of the FP64-counted planes
    // are within about 2 ulps of their exact values
    const float lcnt = __builtin_bit_cast(float, max(__builtin_bit_cast(int, lend) - 8, 0));
    const unsigned sD = (unsigned)aD.stride * 4u, sA = (unsigned)aA.stride * 4u, sB = (unsigned)aB.stride * 4u;
    unsigned off = hit ? (unsigned)w.idx0 * 4u : 0u;
    float pA = A0, pB = B0, cA = 0.0f, cB = 0.0f, kf = 0.0f, s = 0.0f, acc = 0.0f;
    const float ninf = opaque_ninf();
    for (int u = 0; u <= uend; ++u) {
        const int k = u - o;
        // kSlabs slabs at a time where every ray either has all of them before
        // its last counted crossing or none of them: no clamps, and their
        // gathers in flight together
        const bool none = k > nD || k + (kSlabs - 1) < 0;
        const bool all = k >= 0 && k + (kSlabs - 1) < nD && fmaf(kf + (float)(kSlabs - 1), dD, D0) <= lcnt;
        if (kSkip && __ballot(!(none || all)) == 0) {
            if (all) {
                float w1[kSlabs], w2[kSlabs], w3[kSlabs], v1[kSlabs], v2[kSlabs], v3[kSlabs];
                unsigned o1[kSlabs], o2[kSlabs], o3[kSlabs];
#pragma unroll
                for (int q = 0; q < kSlabs; ++q) {
                    const float e = fmaf(kf + (float)q, dD, D0);
                    const bool hasA = pA < e, hasB = pB < e;
                    const float p1 = min_nc(min_nc(pA, pB, ninf), e, ninf);
                    const float p2 = min_nc(__builtin_amdgcn_fmed3f(pA, pB, e), e, ninf);
                    w1[q] = p1 - s;
                    w2[q] = p2 - p1;
                    w3[q] = e - p2;
                    o1[q] = off;
                    o2[q] = off + (pA <= pB ? sA : sB);
                    o3[q] = off + (hasA ? sA : 0u) + (hasB ? sB : 0u);
                    cA = hasA ? cA + 1.0f : cA;
                    cB = hasB ? cB + 1.0f : cB;
                    pA = fmaf(cA, dA, A0);
                    pB = fmaf(cB, dB, B0);
                    off = o3[q] + sD;
                    s = e;
                }
#pragma unroll
                for (int q = 0; q < kSlabs; ++q) {
                    v1[q] = load_vox(rs, o1[q]);
                    v2[q] = v3[q] = 0.0f;
                    if (w2[q] != 0.0f) v2[q] = load_vox(rs, o2[q]);
                    if (w3[q] != 0.0f) v3[q] = load_vox(rs, o3[q]);
                }
#pragma unroll
                for (int q = 0; q < kSlabs; ++q) {
                    acc = fmaf(w1[q], v1[q], acc);
                    acc = fmaf(w2[q], v2[q], acc);
                    acc = fmaf(w3[q], v3[q], acc);
                }
                kf += (float)kSlabs;
            }
            u += kSlabs - 1;
            continue;
        }
        if ((unsigned)k > (unsigned)nD) continue;   // k outside [0, nD]
        // slab k ends at the k-th D crossing, the last one at the exit
        const float e = min_nc(fmaf(kf, dD, D0), lend, ninf);
        // crossings count up to ec: one past the last counted crossing of an
        // axis is at or beyond the exit, within rounding of it
        const float ec = min_nc(e, lcnt, ninf);
        const bool hasA = pA < ec, hasB = pB < ec;
        // p1 <= p2: the crossings inside the slab in order, ec where there is none
        const float p1 = min_nc(min_nc(pA, pB, ninf), ec, ninf);
        const float p2 = min_nc(__builtin_amdgcn_fmed3f(pA, pB, ec), ec, ninf);
        const unsigned offm = off + (pA <= pB ? sA : sB);
        const unsigned off3 = off + (hasA ? sA : 0u) + (hasB ? sB : 0u);
        const float w2 = p2 - p1, w3 = e - p2;
        acc = fmaf(p1 - s, load_vox(rs, off), acc);
        if (kSkip) {
            // the second and third voxels are read only by lanes whose
            // segment in them is not empty (a crossing inside the slab); a
            // skipped term is 0 * v, so the sum is unchanged bit for bit for
            // finite volumes (an infinite v would make that term NaN)
            float v2 = 0.0f, v3 = 0.0f;
            if (w2 != 0.0f) v2 = load_vox(rs, offm);
            if (w3 != 0.0f) v3 = load_vox(rs, off3);
            acc = fmaf(w2, v2, acc);
            acc = fmaf(w3, v3, acc);
        } else {
            acc = fmaf(w2, load_vox(rs, offm), acc);
            acc = fmaf(w3, load_vox(rs, off3), acc);
        }
        cA = hasA ? cA + 1.0f : cA;
        cB = hasB ? cB + 1.0f : cB;
        pA = fmaf(cA, dA, A0);
        pB = fmaf(cB, dB, B0);
        off = off3 + sD;
        s = e;
        kf += 1.0f;
    }
    return hit ? acc : 0.0f;
}

// Siddon system-matrix row of one ray: the voxels the walk above visits with
// a segment of positive length, in visiting order (the rows GenSysMatFan.m /
// GenSysMatCircular3D.m assemble; A x is exactly trace_ray).  kFill false
// only counts them; kFill true writes at most `limit` entries (the count).
template <bool kFill>
__device__ __forceinline__ int sysmat_row(const RayParams &g, int ib, int ip, int ix, int *__restrict__ col,
                                          float *__restrict__ val, long long limit)
{
    RayWalk w;
    if (!ray_walk(g, ib, ip, ix, false, w)) return 0;
    int idx = w.idx0, cnt = 0;
    const double inf = __builtin_huge_val();
    double nt = w.at.n > 0 ? w.at.next0 : inf;
    double ns = w.as.n > 0 ? w.as.next0 : inf;
    double nz = w.az.n > 0 ? w.az.next0 : inf;
    double lam = 0.0;
    const int total = w.at.n + w.as.n + w.az.n + 1;
    for (int k = 0; k < total; ++k) {
        const double m = fmin(fmin(nt, ns), fmin(nz, w.lam_end));
        if (m > lam) {
            if (kFill && cnt < limit) {
                col[cnt] = idx;
                val[cnt] = (float)(m - lam);
            }
            ++cnt;
        }
        lam = m;
        const bool bt = nt <= ns && nt <= nz;
        const bool bs = !bt && ns <= nz;
        idx += bt ? w.at.stride : (bs ? w.as.stride : w.az.stride);
        nt = bt ? nt + w.at.step : nt;
        ns = bs ? ns + w.as.step : ns;
        nz = (!bt && !bs) ? nz + w.az.step : nz;
    }
    return cnt;
}

__global__ __launch_bounds__(kBX *kBY) void k_sysmat_count(long long *__restrict__ counts, RayParams g)
{
    const int ip = blockIdx.x * kBX + threadIdx.x;
    const int ix = blockIdx.y * kBY + threadIdx.y;
    const int ib = blockIdx.z;
    if (ip >= g.np || ix >= g.nx) return;
    counts[((size_t)ib * g.nx + ix) * g.np + ip] = sysmat_row<false>(g, ib, ip, ix, nullptr, nullptr, 0);
}

__global__ __launch_bounds__(kBX *kBY) void k_sysmat_fill(const long long *__restrict__ row_ptr, int *__restrict__ col,
                                                         float *__restrict__ val, RayParams g)
{
    const int ip = blockIdx.x * kBX + threadIdx.x;
    const int ix = blockIdx.y * kBY + threadIdx.y;
    const int ib = blockIdx.z;
    if (ip >= g.np || ix >= g.nx) return;
    const size_t ray = ((size_t)ib * g.nx + ix) * g.np + ip;
    const long long o = row_ptr[ray];
    sysmat_row<true>(g, ib, ip, ix, col + o, val + o, row_ptr[ray + 1] - o);
}

template <bool kSkip>
__global__ __launch_bounds__(kBX *kBY, kSkip ? 7 : 8) void k_ray_fp(const float *__restrict__ vol, float *__restrict__ proj,
                                                                   RayParams g)
{
    int dcol, drow;
    ray_of_thread(dcol, drow);
    const int ip = blockIdx.x * kBX + dcol;
    const int ix = blockIdx.y * kBY + drow;
    const int ib = blockIdx.z;
    const bool valid = ip < g.np && ix < g.nx;
    float chord;
    const float acc = trace_ray<kSkip>(vol, g, ib, ip, ix, valid, chord);
    if (valid) proj[((size_t)ib * g.nx + ix) * g.np + ip] = acc;
}

__device__ __forceinline__ double wave_sum(double v)
{
    for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
    return v;
}

// SIRT residual pass: r = (b - A x) / (A 1 + 1e-9) and per-block partial sums
// of (b - A x)^2 and |b - A x| (SIRT3D.m:80-81, :87) for block (bx, by) of
// view ib; the block's pair goes to partials[2 blk].  For the cone beam r is
// stored times the ray norm, the form in which the exact adjoint reads it.
template <bool kSkip>
__device__ __forceinline__ void fp_residual_block(const float *__restrict__ vol, const float *__restrict__ b,
                                                  float *__restrict__ r, double *__restrict__ partials,
                                                  const RayParams &g, int bx, int by, int ib, size_t blk)
{
    __shared__ double red[2][kBY];
    int dcol, drow;
    ray_of_thread(dcol, drow);
    const int ip = bx * kBX + dcol;
    const int ix = by * kBY + drow;
    double e2 = 0.0, e1 = 0.0;
    const bool valid = ip < g.np && ix < g.nx;
    float chord;
    const float acc = trace_ray<kSkip>(vol, g, ib, ip, ix, valid, chord);
    if (valid) {
        const size_t ray = ((size_t)ib * g.nx + ix) * g.np + ip;
        const float e = b[ray] - acc;
        const float rr = e / (chord + 1e-9f);
        r[ray] = g.residual_norm ? rr * ray_norm((float)g.p[ip], (float)g.xi[ix], (float)g.D) : rr;
        e2 = (double)e * (double)e;
        e1 = fabs((double)e);
    }
    e2 = wave_sum(e2);
    e1 = wave_sum(e1);
    if (threadIdx.x == 0) {
        red[0][threadIdx.y] = e2;
        red[1][threadIdx.y] = e1;
    }
    __syncthreads();
    if (threadIdx.x == 0 && threadIdx.y == 0) {
        double s2 = 0.0, s1 = 0.0;
        for (int w = 0; w < kBY; ++w) {
            s2 += red[0][w];
            s1 += red[1][w];
        }
        partials[2 * blk + 0] = s2;
        partials[2 * blk + 1] = s1;
    }
}

template <bool kSkip>
__global__ __launch_bounds__(kBX *kBY, kSkip ? 7 : 8) void k_ray_fp_residual(const float *__restrict__ vol, const float *__restrict__ b,
                                                              float *__restrict__ r, double *__restrict__ partials,
                                                              RayParams g)
{
    const size_t blk = ((size_t)blockIdx.z * gridDim.y + blockIdx.y) * gridDim.x + blockIdx.x;
    fp_residual_block<kSkip>(vol, b, r, partials, g, blockIdx.x, blockIdx.y, blockIdx.z, blk);
}

// Independent problems in one launch: a flat grid over the jobs' block ranges.
__global__ __launch_bounds__(kBX *kBY) void k_ray_fp_residual_batched(const FpJob *__restrict__ jobs, int njobs)
{
    // job blockIdx.y, its block blockIdx.x; blocks past the job's grid leave at once
    const int p = blockIdx.y, local = blockIdx.x;
    const int gx = jobs[p].gx, gy = jobs[p].gy;
    if (local >= gx * gy * jobs[p].g.nb) return;
    const RayParams g = jobs[p].g;
    const int bx = local % gx, by = (local / gx) % gy, ib = local / (gx * gy);
    if (g.skip_empty)
        fp_residual_block<true>(jobs[p].vol, jobs[p].b, jobs[p].r, jobs[p].partials, g, bx, by, ib, (size_t)local);
    else
        fp_residual_block<false>(jobs[p].vol, jobs[p].b, jobs[p].r, jobs[p].partials, g, bx, by, ib, (size_t)local);
}

// ---------------------------------------------------------------------------
// 2-D images (one slice, one detector row: fan and parallel beams).  The
// crossings, segments and float operations are those of trace_ray without the
// third axis, in the same order (a residual history of SIRT shows a rounding of
// another kind at 1e-8), laid out for what a 2-D problem lacks, rays and
// wavefronts:
//   - a wavefront holds 64 neighbouring rays of the one detector row (the
//     16 x 4 layout of the cone beam would leave 48 of its lanes empty);
//   - each ray walks the slabs of the axis with its own shorter step, so it
//     meets at most one crossing of the other axis in a slab (two that coincide
//     but for rounding are taken in two slabs, the second segment a rounding
//     short) and none has to walk crossing by crossing;
//   - rays read the image or its transpose, whichever has their other axis
//     fastest, from one buffer that holds both;
//   - the weights and offsets of kFlatUnroll slabs are formed ahead of their
//     loads, so that many gathers are in flight at three wavefronts per SIMD.
// 256^2 / 360 views / 512 bins, residual pass: 144 us in the cone beam's
// kernel, 37 us here, bound by VALU issue (15 instructions a slab) and by the
// gathers' latency in turn; without the second layout, rays of the other axis
// in a wavefront cost 65 us.
// ---------------------------------------------------------------------------
constexpr int kFlatUnroll = 8, kFlatWaves = 4;

// Part `part` of `parts` of the ray's slabs (the whole ray: 0 of 1).
__device__ __forceinline__ float trace_ray_flat(const RayParams &g, int ib, int ip, bool valid, float &chord, int part = 0,
                                                int parts = 1)
{
    RayWalk w;
    const bool go = valid && ray_walk(g, ib, ip, 0, false, w);
    chord = go ? (float)w.lam_end : 0.0f;
    if (__ballot(go) == 0) return 0.0f;
    const int npix = g.nt * g.ns;
    __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc((void *)g.flat, 0, (int)((unsigned)npix * (g.flat_alone ? 4u : 8u)), kBufDword3);
    const bool lane_t = w.at.stride != 0 && (w.as.stride == 0 || w.at.step <= w.as.step);
    const AxisSetup aD = lane_t ? w.at : w.as;
    const AxisSetup aA = lane_t ? w.as : w.at;
    const int sgnD = aD.stride > 0 ? 1 : -1, sgnA = aA.stride > 0 ? 1 : (aA.stride < 0 ? -1 : 0);
    const bool swap = lane_t && !g.flat_alone;   // reads the transpose
    const unsigned sA = (unsigned)(sgnA * (lane_t && g.flat_alone ? g.nt : 1)) * 4u;
    const unsigned sD = (unsigned)(sgnD * (swap ? g.ns : (lane_t ? 1 : g.nt))) * 4u;
    const unsigned idx0 = swap ? (unsigned)(npix + w.at.i0 * g.ns + w.as.i0) : (unsigned)w.idx0;

    // trace_ray's 16 neighbouring rays that do not all have the view's axis as
    // their shorter one walk crossing by crossing, with one segment behind the
    // last counted crossing; the others cut that segment at lcnt
    const bool along_t = fabs(g.view[4 * ib + 0]) > fabs(g.view[4 * ib + 1]);
    const AxisSetup &vD = along_t ? w.at : w.as, &vA = along_t ? w.as : w.at;
    const bool odd = go && !(vD.stride != 0 && (vA.n == 0 || vA.step >= 1.001 * vD.step));
    const unsigned long long of_group = 0xffffull << (__lane_id() & 48);
    const bool one_tail = (__ballot(odd) & of_group) != 0 ||
                          ((__ballot(go && vD.stride > 0) & of_group) != 0 && (__ballot(go && vD.stride < 0) & of_group) != 0);

    // slab index relative to the first slab of the wavefront's rays of the same
    // axis and direction, so that these read one image row together
    const int kind = (lane_t ? 2 : 0) + (sgnD > 0 ? 1 : 0), from = sgnD * aD.i0;
    int istart = 0;
#pragma unroll
    for (int c = 0; c < 4; ++c) {
        const bool same = go && kind == c;
        if (__ballot(same) == 0) continue;
        const int m = wave_min_int(same ? from : 0x7fffffff);
        istart = same ? m : istart;
    }
    const int o = go ? from - istart : (1 << 30);
    const int uend = __builtin_amdgcn_readfirstlane(wave_max_int(go ? o + aD.n : -1));
    const int nD = go ? aD.n : 0;

    const float inf = __builtin_huge_valf();
    const float D0 = go ? (float)aD.next0 : inf, dD = go ? (float)aD.step : 0.0f;
    const float A0 = go && aA.n > 0 ? (float)aA.next0 : inf, dA = go ? (float)aA.step : 0.0f;
    const float lend = go ? (float)w.lam_end : 0.0f;
    const float near_end = __builtin_bit_cast(float, max(__builtin_bit_cast(int, lend) - 8, 0));
    const float lcnt = one_tail ? lend : near_end, most = one_tail ? (float)aA.n : inf;
    const int last = one_tail ? nD : -1;   // the slab that ends at the exit, whatever its plane's float parameter
    const float ninf = opaque_ninf();
    int ubegin = 0, ulast = uend;
    if (parts > 1) {   // this part's blocks of slabs
        const int blocks = uend / kFlatUnroll + 1;
        ubegin = blocks * part / parts * kFlatUnroll;
        ulast = min(uend, blocks * (part + 1) / parts * kFlatUnroll - 1);
    }
    unsigned off;
    float pA, cA, s, sum = 0.0f;
    auto begin = [&]() {   // the ray's state at slab ubegin
        off = idx0 * 4u;
        pA = A0;
        cA = s = 0.0f;
        const int k = ubegin - o;
        if (parts > 1 && go && k > 0 && k <= nD) {
            s = min_nc(fmaf((float)(k - 1), dD, D0), lend, ninf);
            if (pA < s) {   // crossings before s: a guess, and its neighbours by the walk's own comparison
                cA = fminf(fmaxf(ceilf((s - A0) / dA), 0.0f), (float)aA.n);
                if (cA > 0.0f && fmaf(cA - 1.0f, dA, A0) >= s) cA -= 1.0f;
                if (cA < (float)aA.n && fmaf(cA, dA, A0) < s) cA += 1.0f;
            }
            pA = fmaf(cA, dA, A0);
            off += (unsigned)(int)cA * sA + (unsigned)k * sD;
        }
    };
    begin();
    float w1[kFlatUnroll], w2[kFlatUnroll], v1[kFlatUnroll], v2[kFlatUnroll];
    unsigned o1[kFlatUnroll];
    for (int u = ubegin; u <= ulast; u += kFlatUnroll) {
        const int k0 = u - o;
        const float kf = (float)k0;
        // all slabs of the block lie on every ray and end before its last
        // counted crossing: no clamps, no masks
        const bool inner = k0 >= 0 && k0 + kFlatUnroll - 1 < nD && fmaf(kf + (float)(kFlatUnroll - 1), dD, D0) <= near_end;
        if (__ballot(!inner) == 0) {
#pragma unroll
            for (int q = 0; q < kFlatUnroll; ++q) {
                const float e = fmaf(kf + (float)q, dD, D0);
                const bool hasA = pA < e;
                const float p1 = min_nc(pA, e, ninf);
                w1[q] = p1 - s;
                w2[q] = e - p1;
                o1[q] = off;
                off += (hasA ? sA : 0u) + sD;
                cA = hasA ? cA + 1.0f : cA;
                pA = fmaf(cA, dA, A0);
                s = e;
            }
#pragma unroll
            for (int q = 0; q < kFlatUnroll; ++q) {
                v1[q] = load_vox(rs, o1[q]);
                v2[q] = load_vox(rs, o1[q] + sA);
            }
#pragma unroll
            for (int q = 0; q < kFlatUnroll; ++q) {
                sum = fmaf(w1[q], v1[q], sum);
                sum = fmaf(w2[q], v2[q], sum);
            }
        } else {
            // a slab outside the ray gets weights of 0 and offsets past the
            // image, which read 0; the segment behind the last counted
            // crossing, if there is one, follows its slab's other two
            float w3[kFlatUnroll];
            unsigned o2[kFlatUnroll], o3[kFlatUnroll];
#pragma unroll
            for (int q = 0; q < kFlatUnroll; ++q) {
                const bool act = go && (unsigned)(k0 + q) <= (unsigned)nD;
                const float plane = min_nc(fmaf(kf + (float)q, dD, D0), lend, ninf);
                const float e = k0 + q == last ? lend : plane;
                const float ec = min_nc(e, lcnt, ninf);
                const bool hasA = act && pA < ec && cA < most;
                const float p1 = hasA ? pA : ec;
                w1[q] = act ? p1 - s : 0.0f;
                w2[q] = act ? ec - p1 : 0.0f;
                w3[q] = act ? e - ec : 0.0f;
                o1[q] = act ? off : 0xFFFFFFFCu;
                o2[q] = act ? off + sA : 0xFFFFFFFCu;
                o3[q] = off + (hasA ? sA : 0u);
                cA = hasA ? cA + 1.0f : cA;
                pA = fmaf(cA, dA, A0);
                off = act ? o3[q] + sD : off;
                s = act ? e : s;
            }
#pragma unroll
            for (int q = 0; q < kFlatUnroll; ++q) {
                v1[q] = load_vox(rs, o1[q]);
                v2[q] = load_vox(rs, o2[q]);
            }
#pragma unroll
            for (int q = 0; q < kFlatUnroll; ++q) {
                sum = fmaf(w1[q], v1[q], sum);
                sum = fmaf(w2[q], v2[q], sum);
                if (w3[q] != 0.0f) sum = fmaf(w3[q], load_vox(rs, o3[q]), sum);
            }
        }
    }
    // the walk multiplies the pixels beside a ray by 0, and an infinite or NaN one
    // makes a NaN of it: such a ray is walked again, its own pixels only
    const bool again = !(fabsf(sum) < inf);
    if (__ballot(again) != 0) {
        begin();
        float own = 0.0f;
        for (int u = ubegin; u <= ulast; ++u) {
            const int k = u - o;
            if (!again || (unsigned)k > (unsigned)nD) continue;
            const float plane = min_nc(fmaf((float)k, dD, D0), lend, ninf);
            const float e = k == last ? lend : plane, ec = min_nc(e, lcnt, ninf);
            const bool hasA = pA < ec && cA < most;
            const float p1 = hasA ? pA : ec;
            const unsigned next = off + (hasA ? sA : 0u);
            if (p1 != s) own = fmaf(p1 - s, load_vox(rs, off), own);
            if (ec != p1) own = fmaf(ec - p1, load_vox(rs, off + sA), own);
            if (e != ec) own = fmaf(e - ec, load_vox(rs, next), own);
            cA = hasA ? cA + 1.0f : cA;
            pA = fmaf(cA, dA, A0);
            off = next + sD;
            s = e;
        }
        sum = again ? own : sum;
    }
    return sum;
}

// Wavefront `wave` of the launch: 64 columns of one view.
__device__ __forceinline__ bool flat_item(const RayParams &g, int &ib, int &ip)
{
    const int chunks = (g.np + 63) / 64;
    const long item = (long)blockIdx.x * kFlatWaves + __builtin_amdgcn_readfirstlane((int)threadIdx.y);
    ib = (int)(item / chunks);
    ip = (int)(item - (long)ib * chunks) * 64 + (int)threadIdx.x;
    return ib < g.nb;
}

__global__ __launch_bounds__(64 * kFlatWaves) void k_ray_fp_flat(float *__restrict__ proj, RayParams g)
{
    int ib, ip;
    if (!flat_item(g, ib, ip)) return;
    float chord;
    const float acc = trace_ray_flat(g, ib, ip, ip < g.np, chord);
    if (ip < g.np) proj[(size_t)ib * g.np + ip] = acc;
}

// The same for few rays: the block's wavefronts walk a share of the slabs of the
// same 64 rays each, and the shares are added in order.  A ray's walk is a chain
// of gathers' latencies that nothing hides below a few wavefronts per SIMD.
// Whole calls, a ray to one lane / split by 2 / 4 / 8 (pixels, views x bins):
//    64^2,  90 x   96   15.8 /  9.2 /  9.1 /  9.2 us
//   128^2, 180 x  192   24.5 / 16.8 / 14.6 / 14.1 us
//   256^2, 360 x  512   41.3 / 51.0 / 48.7 / 58.8 us (2880 wavefronts of rays)
//   512^2, 360 x  730  113.9 / 97.9 / 91.1 / 99.9 us (4320)
//   512^2, 720 x 1024    267 /  263 /  267 /  297 us (11520)
// 3 us of the first column's first line are the image's transpose, left out up
// to 128^2 pixels.
__global__ __launch_bounds__(64 * kFlatWaves) void k_ray_fp_flat_split(float *__restrict__ proj, RayParams g)
{
    __shared__ float part[kFlatWaves][64];
    const int chunks = (g.np + 63) / 64, ib = blockIdx.x / chunks, ip = (blockIdx.x - ib * chunks) * 64 + (int)threadIdx.x;
    const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.y);
    float chord;
    part[wave][threadIdx.x] = trace_ray_flat(g, ib, ip, ip < g.np, chord, wave, kFlatWaves);
    __syncthreads();
    if (wave != 0 || ip >= g.np) return;
    float sum = part[0][threadIdx.x];
#pragma unroll
    for (int w = 1; w < kFlatWaves; ++w) sum += part[w][threadIdx.x];
    proj[(size_t)ib * g.np + ip] = sum;
}

// The residual pass (fp_residual_block) of a 2-D problem.
__global__ __launch_bounds__(64 * kFlatWaves) void k_ray_fp_residual_flat(const float *__restrict__ b,
                                                                          float *__restrict__ r,
                                                                          double *__restrict__ partials, RayParams g)
{
    __shared__ double red[2][kFlatWaves];
    int ib, ip;
    double e2 = 0.0, e1 = 0.0;
    if (flat_item(g, ib, ip)) {
        float chord;
        const float acc = trace_ray_flat(g, ib, ip, ip < g.np, chord);
        if (ip < g.np) {
            const size_t ray = (size_t)ib * g.np + ip;
            const float e = b[ray] - acc;
            r[ray] = e / (chord + 1e-9f);
            e2 = (double)e * (double)e;
            e1 = fabs((double)e);
        }
    }
    e2 = wave_sum(e2);
    e1 = wave_sum(e1);
    if (threadIdx.x == 0) {
        red[0][threadIdx.y] = e2;
        red[1][threadIdx.y] = e1;
    }
    __syncthreads();
    if (threadIdx.x == 0 && threadIdx.y == 0) {
        double s2 = 0.0, s1 = 0.0;
        for (int w = 0; w < kFlatWaves; ++w) {
            s2 += red[0][w];
            s1 += red[1][w];
        }
        partials[2 * (size_t)blockIdx.x] = s2;
        partials[2 * (size_t)blockIdx.x + 1] = s1;
    }
}

// ---------------------------------------------------------------------------
// Cone beam by detector columns.
//
// All rays of one detector column (one view, one p) share their path through
// the (t, s) plane: seen from above they are one line.  k_ray_cells walks that
// line once in FP64 and lists the voxel columns (cells) it crosses, with the
// in-plane parameter at which each begins and its length, four cells to a
// 64-byte block.  k_ray_columns then gives a wavefront 64 neighbouring rows of
// the detector column and walks the list: a block is the same for the
// wavefront and comes through the scalar cache in one load, and a lane only
// keeps track of its slice.  The volume is read from a copy with z fastest,
// [s][t][1 + nz + 1] with a slice of zeros at both ends, so the wavefront's
// load of a cell is one run of neighbouring voxels, and a ray that leaves
// through the top or the bottom reads zeros from there on.
//
// Slices change rarely (a cone angle of 12 degrees passes a plane every five
// voxels), so a lane looks for its next z crossing once per block, or twice
// where a ray of the wavefront is steep enough to cross two planes in a block:
// each cell's length splits at the crossing, clamped into the cell, between the
// old slice and the new one.  Steeper still, the cells are taken one by one,
// each cut by as many crossings as there are.
//
// Crossing parameters and cell bounds are floats relative to the entry point,
// with one rounding each, as in the slab walk, and lengths are differences of
// them (lengths rounded one by one would sum up with a bias: 1.2e-6 instead of
// 3e-8 on a volume of ones).  Per ray and voxel column the loop issues 6.5 VALU
// instructions and two loads (the slab walk: 32 instructions and three loads
// per slab of 1.4 voxel columns).
// ---------------------------------------------------------------------------
constexpr int kColWaves = 4;

// One wavefront per detector column of view view0 + blockIdx.y: its list and
// its head.  LDS: C.stride + 1 cell parameters, then C.stride offsets.
__global__ __launch_bounds__(64) void k_ray_cells(RayParams g, ColumnLists C, int view0)
{
    extern __shared__ float cells[];
    float *sl = cells;
    unsigned *so = reinterpret_cast<unsigned *>(cells + C.stride + 1);
    const int ip = blockIdx.x, v = blockIdx.y, ib = view0 + v, lane = threadIdx.x;
    const size_t col = (size_t)v * g.np + ip;
    const double sb = g.view[4 * ib + 0], cb = g.view[4 * ib + 1], st = g.view[4 * ib + 2], ss = g.view[4 * ib + 3];
    const double P = g.p[ip];
    double dx = P * cb + g.D * sb, dy = P * sb - g.D * cb;
    const double inv_n = 1.0 / sqrt(dx * dx + dy * dy);
    dx *= inv_n;
    dy *= inv_n;
    double lo = -__builtin_huge_val(), hi = __builtin_huge_val();
    bool hit = clip_axis(st, dx, g.bt, lo, hi);
    hit = clip_axis(ss, dy, g.bs, lo, hi) && hit && hi > lo;
    if (!hit) {
        if (lane == 0) C.head[col] = ColumnHead{};
        return;
    }
    const AxisSetup at = setup_axis(st, dx, lo, hi, g.rt, g.nt, 1), as = setup_axis(ss, dy, lo, hi, g.rs, g.ns, 1);
    // slabs of the axis with the shorter step; at most one crossing of the
    // other axis in a slab, but for rounding, and any number is listed
    const bool along_t = at.stride != 0 && (as.stride == 0 || at.step <= as.step);
    const AxisSetup aD = along_t ? at : as, aA = along_t ? as : at;
    const double len = hi - lo, inv_step = aA.n > 0 ? 1.0 / aA.step : 0.0;
    const unsigned pitch = (unsigned)(g.nz + 2) * 4u;
    auto crossings_before = [&](double lam) {
        const double c = aA.n > 0 ? ceil((lam - aA.next0) * inv_step) : 0.0;
        return (int)fmin(fmax(c, 0.0), (double)aA.n);
    };
    for (int k = lane; k <= aD.n; k += 64) {
        const double l0 = k == 0 ? 0.0 : aD.next0 + (k - 1) * aD.step, l1 = aD.next0 + k * aD.step;
        const int c0 = k == 0 ? 0 : crossings_before(l0), c1 = k == aD.n ? aA.n : crossings_before(l1);
        double begin = l0;
        for (int c = c0; c <= c1; ++c) {
            const int iD = aD.i0 + aD.stride * k, iA = aA.i0 + aA.stride * c;
            sl[k + c] = (float)begin;
            so[k + c] = (unsigned)(along_t ? iA * g.nt + iD : iD * g.nt + iA) * pitch;
            begin = aA.next0 + c * aA.step;
        }
    }
    // the list ends in cells of length 0, up to an even number of blocks and one
    // more that is read ahead
    const int n = aD.n + aA.n + 1, padded = (n + 2 * kColBlock - 1) / (2 * kColBlock) * (2 * kColBlock);
    __syncthreads();
    if (lane <= padded + kColBlock - n) {
        sl[n + lane] = (float)len;
        if (lane < padded + kColBlock - n) so[n + lane] = so[n - 1];
    }
    __syncthreads();
    float longest = 0.0f, pair = 0.0f;
    unsigned *out = reinterpret_cast<unsigned *>(C.blocks + col * (C.stride / kColBlock));
    for (int e = lane; e < (padded + kColBlock) * 4; e += 64) {   // 16 words a block: l[5], d[4], off[4]
        const int q = e & 15, i = (e >> 4) * kColBlock;
        unsigned w = 0;
        if (q < 5) {
            w = __builtin_bit_cast(unsigned, sl[i + q]);
            if (q == 4) {
                longest = fmaxf(longest, sl[i + 4] - sl[i]);
                pair = fmaxf(pair, fmaxf(sl[i + 2] - sl[i], sl[i + 4] - sl[i + 2]));
            }
        } else if (q < 9) {
            w = __builtin_bit_cast(unsigned, fmaxf(sl[i + q - 4] - sl[i + q - 5], 0.0f));
        } else if (q < 13) {
            w = so[i + q - 9];
        }
        out[e] = w;
    }
    for (int m = 32; m > 0; m >>= 1) {
        longest = fmaxf(longest, __shfl_xor(longest, m, 64));
        pair = fmaxf(pair, __shfl_xor(pair, m, 64));
    }
    if (lane == 0)
        C.head[col] = ColumnHead{lo, len, 1.0 / sqrt(P * P + g.D * g.D), padded, longest * 1.0001f, pair * 1.0001f};
}

// x clamped into [0, hi]
__device__ __forceinline__ int clamp_i(int x, int hi)
{
    int r;
    asm("v_med3_i32 %0, %1, 0, %2" : "=v"(r) : "v"(x), "v"(hi));
    return r;
}

// v of the lane byte / 4 (mod 64)
__device__ __forceinline__ float lane_value(int byte, float v)
{
    return __builtin_bit_cast(float, __builtin_amdgcn_ds_bpermute(byte, __builtin_bit_cast(int, v)));
}

// v of lane i, for the whole wavefront
__device__ __forceinline__ float lane_float(float v, int i)
{
    return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), i));
}

// State of a lane on its way through the cells of a list.
struct ColumnLane {
    float Z0, dZ;   // first z crossing and the step between them
    int zb, sgn;    // first slice (bytes into a cell) and the step per crossing
};

// Sum over the blocks of a list, nb of them (even, and one more to read).
// WINDOW: the cell's 64 slices around the wavefront's rows are loaded as one
// run, a slice per lane, and handed to the rows by lane permutations; otherwise
// each row reads its own two.  The window halves the loads, whose address and
// tag work bounds the loop (7 cycles a load, 4 for 64 lanes at best): 3.0
// against 3.7 ms for 256^3 / 90 views / 512^2, the rows of a wavefront 40
// slices apart.  Where they fan out to more than 64 slices two windows would
// do, which measured 47 ms against 41 for the plain loads at 512^3 / 240 views.
template <bool WINDOW, int STEP>
__device__ __forceinline__ float column_sum(__amdgpu_buffer_rsrc_t rs, const ColumnBlock *__restrict__ blk, int nb, int top,
                                            const ColumnLane &L)
{
    // a block on its way: weights of the old and the new slice, loaded values
    struct Part {
        float w1[kColBlock], w2[kColBlock], v[kColBlock], u[kColBlock];
        int io[kColBlock / STEP], in[kColBlock / STEP];
    };
    const int lane4 = (int)__lane_id() * 4;
    float acc = 0.0f, pZ = L.Z0;
    int za = L.zb, cz = 0;
    auto load = [&](int z, unsigned cell) {
        return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rs, z, (int)cell, 0));
    };
    ColumnBlock next = blk[0];
    auto issue = [&](Part &q, int i) {
        const ColumnBlock c = next;
        next = blk[i + 1];
        constexpr int H = kColBlock / STEP;
        float p[H];
        int zo[H], zn[H];
#pragma unroll
        for (int k = 0; k < H; ++k) {
            p[k] = pZ;
            zo[k] = za;
            cz += pZ < c.l[(k + 1) * STEP] ? 1 : 0;
            pZ = fmaf((float)cz, L.dZ, L.Z0);
            zn[k] = za = clamp_i(__mul24(cz, L.sgn) + L.zb, top);
        }
        if constexpr (!WINDOW) {
#pragma unroll
            for (int j = 0; j < kColBlock; ++j) {
                q.v[j] = load(zo[j / STEP], c.off[j]);
                q.u[j] = load(zn[j / STEP], c.off[j]);
            }
        } else {
            // the wavefront's slices lie between those of its first and last
            // row, one more to either side for each step back and one for ties
            const int e0 = __builtin_amdgcn_readlane(za, 0), e1 = __builtin_amdgcn_readlane(za, 63);
            const int base = max(min(e0, e1) - 4 * (H + 1), 0);
#pragma unroll
            for (int k = 0; k < H; ++k) {
                q.io[k] = zo[k] - base;
                q.in[k] = zn[k] - base;
            }
#pragma unroll
            for (int j = 0; j < kColBlock; ++j) q.v[j] = load(lane4, c.off[j] + base);
        }
#pragma unroll
        for (int j = 0; j < kColBlock; ++j) {
            q.w1[j] = __builtin_amdgcn_fmed3f(p[j / STEP] - c.l[j], 0.0f, c.d[j]);
            q.w2[j] = c.d[j] - q.w1[j];
        }
    };
    auto sum = [&](const Part &q) {
        float v1[kColBlock], v2[kColBlock];
#pragma unroll
        for (int j = 0; j < kColBlock; ++j) {
            v1[j] = WINDOW ? lane_value(q.io[j / STEP], q.v[j]) : q.v[j];
            v2[j] = WINDOW ? lane_value(q.in[j / STEP], q.v[j]) : q.u[j];
        }
#pragma unroll
        for (int j = 0; j < kColBlock; ++j) {
            acc = fmaf(q.w1[j], v1[j], acc);
            acc = fmaf(q.w2[j], v2[j], acc);
        }
    };
    Part A, B;
    issue(A, 0);
    for (int i = 0; i < nb; i += 2) {
        issue(B, i + 1);
        sum(A);
        issue(A, min(i + 2, nb - 1));
        sum(B);
    }
    return acc;
}

// Line integrals of the 64 rows of a wavefront through the cells of detector
// column `col`.
__device__ __forceinline__ float trace_column(const RayParams &g, const ColumnHead *__restrict__ heads,
                                              const ColumnBlock *__restrict__ blocks, size_t stride, size_t col, int ip,
                                              int ix, bool valid)
{
    const ColumnHead h = heads[col];
    if (h.n == 0) return 0.0f;
    const double slope = g.xi[valid ? ix : g.nx - 1] * h.inv_rho;   // z per in-plane length
    // first slice, next plane and the step between planes
    // (divided as in setup_axis: a level ray between two slices takes the same one)
    const double zin = (g.sz + h.lo * slope) / g.rz;
    const double k0 = slope < 0.0 ? ceil(zin) - 1.0 : floor(zin);
    double z0 = __builtin_huge_val(), dz = 0.0, out = __builtin_huge_val();
    if (slope != 0.0) {
        const double inv_s = 1.0 / slope;
        z0 = ((slope > 0.0 ? k0 + 1.0 : k0) * g.rz - g.sz) * inv_s - h.lo;
        dz = g.rz * fabs(inv_s);
        out = (slope > 0.0 ? g.bz - g.sz : -g.sz) * inv_s - h.lo;
    }
    const double norm = sqrt(fma(slope, slope, 1.0));
    const bool hit = fmin(h.len, out) > 0.0;
    if (__ballot(hit) == 0) return 0.0f;
    const float Z0 = (float)z0, dZ = (float)dz;
    const int top = 4 * (g.nz + 1);   // slices 0 and nz + 1 of the copy are zeros
    const int zb = (int)fmin(fmax(4.0 * (k0 + 1.0), 0.0), (double)top), sgn = slope > 0.0 ? 4 : -4;

    const size_t vbytes = (size_t)g.nt * g.ns * (g.nz + 2) * sizeof(float);
    const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(
        (void *)g.volZ, 0, (int)(vbytes > 0xFFFFFFFFull ? 0xFFFFFFFFu : (unsigned)vbytes), kBufDword3);
    const ColumnBlock *__restrict__ blk = blocks + col * stride;
    // cell by cell: the voxels that the ray meets and no others
    auto by_cells = [&]() {
        // a ray crosses no planes behind the volume's top or bottom: it may be
        // steep enough for any number of them there (thin slices, rows far off
        // the volume)
        const int edge = slope > 0.0 ? top : 0;
        float sum = 0.0f, pZ = zb == edge ? __builtin_huge_valf() : Z0;
        int za = zb, cz = 0;
        auto load = [&](int z, unsigned cell) {
            return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rs, z, (int)cell, 0));
        };
        for (int i = 0; i < h.n; ++i) {
            const ColumnBlock &c = blk[i / kColBlock];
            const int j = i % kColBlock;
            const float l1 = c.l[j + 1];
            const unsigned cell = c.off[j];
            float l = c.l[j];
            while (pZ < l1) {
                if (pZ > l) {
                    sum = fmaf(pZ - l, load(za, cell), sum);
                    l = pZ;
                }
                ++cz;
                za = clamp_i(__mul24(cz, sgn) + zb, top);
                pZ = za == edge ? __builtin_huge_valf() : fmaf((float)cz, dZ, Z0);
            }
            if (l1 > l) sum = fmaf(l1 - l, load(za, cell), sum);
        }
        return sum;
    };
    float acc = 0.0f;
    bool again = true;
    const int nb = h.n / kColBlock;
    if (__ballot(dZ != 0.0f && dZ < h.pair) == 0) {
        // widest run of slices (bytes) between the first and the last row, the
        // outermost ones: a row's height grows with the way from the source until
        // the line leaves the box, or the row its top or bottom, where its slice
        // stays.  Rows on one side of the source plane fan out until the outer one
        // leaves; on both sides each goes on until it leaves by itself.
        const float s0 = lane_float((float)slope, 0), s1 = lane_float((float)slope, 63);
        const float reach = (float)(h.lo + h.len), half = 0.5f * (float)g.bz;
        const float r0 = fabsf(s0) * reach, r1 = fabsf(s1) * reach, outer = fmaxf(r0, r1);
        const float fan = s0 * s1 < 0.0f ? fminf(r0, half) + fminf(r1, half)
                                         : fabsf(s1 - s0) * reach * (outer > half ? half / outer : 1.0f);
        const float wide = 4.0f * (fan / (float)g.rz) + 36.0f;
        const bool narrow = wide <= 4.0f * 63.0f, gentle = __ballot(dZ != 0.0f && dZ < h.block) == 0;
        const ColumnLane lane{Z0, dZ, zb, sgn};
        if (gentle)
            acc = narrow ? column_sum<true, kColBlock>(rs, blk, nb, top, lane)
                         : column_sum<false, kColBlock>(rs, blk, nb, top, lane);
        else
            acc = narrow ? column_sum<true, kColBlock / 2>(rs, blk, nb, top, lane)
                         : column_sum<false, kColBlock / 2>(rs, blk, nb, top, lane);
        // column_sum multiplies a block's other slice by 0, and an infinite or
        // NaN voxel there makes a NaN of a ray that passes it by
        again = !(fabsf(acc) < __builtin_huge_valf());
    }
    if (__ballot(again) != 0) {
        const float sum = by_cells();
        acc = again ? sum : acc;
    }
    return hit ? acc * (float)norm : 0.0f;
}

// Workgroup -> (64 rows, view, four detector columns).  Consecutive workgroups
// go to the eight XCDs in turn; an XCD is given tiles of kColTileP x kColTileV
// (columns, views), 256 workgroups, which is what its 32 CUs hold at a time:
// neighbouring columns of neighbouring views cross the same cells, so the
// wavefronts in flight share them in the XCD's L2.  Tiles run over the columns,
// then the views, rows slowest: one band of slices at a time, which stays in the
// Infinity Cache.
constexpr int kColTileP = 16, kColTileV = 16;

struct ColumnTile {
    int p0, v, row0;   // p0 or v past the end: an empty place of a partial tile
};
__host__ __device__ __forceinline__ int column_tiles_p(const RayParams &g)
{
    return (g.np + kColWaves * kColTileP - 1) / (kColWaves * kColTileP);
}
__host__ __device__ __forceinline__ int column_tiles_v(int views) { return (views + kColTileV - 1) / kColTileV; }
__device__ __forceinline__ ColumnTile column_tile(const RayParams &g, int views)
{
    constexpr int kTile = kColTileP * kColTileV;
    const int place = blockIdx.x >> 3, tile = place / kTile * 8 + (int)(blockIdx.x & 7), in = place % kTile;
    const int tp = column_tiles_p(g), tv = column_tiles_v(views);
    const int ip = tile % tp, rest = tile / tp;
    return ColumnTile{(ip * kColTileP + in % kColTileP) * kColWaves, rest % tv * kColTileV + in / kColTileP,
                      rest / tv * 64};
}

__global__ __launch_bounds__(64 * kColWaves, 8) void k_ray_columns(float *__restrict__ out,
                                                                const ColumnHead *__restrict__ heads,
                                                                const ColumnBlock *__restrict__ blocks, RayParams g,
                                                                int stride, int view0, int views)
{
    __shared__ float sums[kColWaves][65];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const ColumnTile B = column_tile(g, views);
    const int ip = B.p0 + wave;
    float acc = 0.0f;
    const bool there = B.p0 < g.np && B.v < views && B.row0 < g.nx;
    if (there && ip < g.np) {
        const int ix = B.row0 + lane;
        acc = trace_column(g, heads, blocks, stride, (size_t)B.v * g.np + ip, ip, ix, ix < g.nx);
    }
    // the block's 64 x 4 results, four neighbouring columns of a row per four threads
    sums[wave][lane] = acc;
    __syncthreads();
    const int c = threadIdx.x % kColWaves, r = threadIdx.x / kColWaves;
    const int oc = B.p0 + c, orow = B.row0 + r;
    if (there && oc < g.np && orow < g.nx) out[((size_t)(view0 + B.v) * g.nx + orow) * g.np + oc] = sums[c][r];
}

int column_blocks(const RayParams &g, int views)
{
    const long tiles = (long)column_tiles_p(g) * column_tiles_v(views) * ((g.nx + 63) / 64);
    return (int)((tiles + 7) / 8 * 8 * kColTileP * kColTileV);
}

// Lists of C.views views at a time, then their rays.
hipError_t launch_columns(const RayParams &g, float *out, hipStream_t st)
{
    const ColumnLists &C = g.cols;
    for (int v0 = 0; v0 < g.nb; v0 += C.views) {
        const int views = g.nb - v0 < C.views ? g.nb - v0 : C.views, n = column_blocks(g, views);
        hipLaunchKernelGGL(k_ray_cells, dim3(g.np, views), dim3(64), (2 * C.stride + 1) * sizeof(float), st, g, C, v0);
        hipLaunchKernelGGL(k_ray_columns, dim3((unsigned)n), dim3(64 * kColWaves), 0, st, out, C.head, C.blocks, g,
                           C.stride / kColBlock, v0, views);
        const hipError_t e = hipGetLastError();
        if (e != hipSuccess) return e;
    }
    return hipSuccess;
}

unsigned flat_blocks(const RayParams &g)
{
    const long items = (long)((g.np + 63) / 64) * g.nb;
    return (unsigned)((items + kFlatWaves - 1) / kFlatWaves);
}

dim3 fp_grid(const RayParams &g) { return dim3((g.np + kBX - 1) / kBX, (g.nx + kBY - 1) / kBY, g.nb); }

}  // namespace

// lists of one pass (16 bytes a cell) stay in the Infinity Cache beside a band of slices
constexpr size_t kColListBytes = (size_t)256 << 20;

// Where the columns are faster than the slab walk (CTR_FP_COLUMNS = 0 / 1
// overrides).  A wavefront always pays for 64 rows, so they need about 0.7 of
// its lanes filled, and three launches and a list of the cells pay from 12000
// wavefronts and 80 slices on; the rows of a wavefront are to span less than 70
// slices at the far side (they share one run of 64), or 110 where nearly all are
// filled.  Slab walk / columns in us (nz, views x columns x rows, span):
//   324, 183 x 674 x 467, 59   11910 / 8180    269, 25 x 567 x 521, 74   1458 / 1944
//   254, 223 x 688 x 414, 57   12409 / 8869    258, 105 x 408 x 387, 87  3522 / 3783
//   150, 242 x 380 x 221, 51    1998 / 1468    119, 136 x 202 x 185, 74   582 /  466 (0.96 filled)
//   125, 25 x 358 x 156, 53      218 /  173     51, 232 x 164 x 101, 54   197 /  214
//    89, 124 x 173 x 126, 61     198 /  137     43, 290 x 121 x 60, 59    116 /  121
//   109, 350 x 288 x 132, 73    1770 / 1750     52, 139 x 186 x 69 (0.54 filled) 121 / 147
// Wider spans, all lanes filled (rows leave the volume at its top and bottom,
// and the slab walk ends there; beyond 250 slices the columns lose without limit,
// 153 / 570 us at 4100):
//    80, 60 x 300 x 128, 82    359 / 264        80, 60 x 300 x 128, 164   267 / 276
//   120, 60 x 300 x 128, 123   396 / 453       200, 60 x 300 x 256, 115   677 / 767
//   320, 90 x 300 x 384, 115  3929 / 3371      200, 60 x 300 x 256, 262   433 / 500
// Over 66 geometries of 20 to 400 slices: 0.6% slower on the mean than the
// faster of the two each time, 10% faster than the slab walk.
// The residual pass of SIRT keeps the slab walk: the history of its norms, in 64
// bits, shows the rounding of the walk's chain of sums (1e-9 to 1e-8 of a norm,
// also for 2e7 rays), and a problem's history is not to depend on the kernel.
static bool column_use(const RayParams &g, double row_pitch)
{
    if (const char *e = std::getenv("CTR_FP_COLUMNS")) return std::atoi(e) != 0;
    const size_t chunks = (g.nx + 63) / 64, waves = (size_t)g.nb * g.np * chunks;
    const double fill = (double)g.nx / (64.0 * chunks), far = g.D + 0.5 * std::hypot(g.bt, g.bs);
    const double span = 63.0 * row_pitch * far / (g.D * g.rz);
    return g.nz >= 80 && waves >= 12000 && fill >= 0.7 && span < (fill > 0.95 ? 110.0 : 70.0);
}

bool column_plan(const RayParams &g, double row_pitch, ColumnPlan &L)
{
    // 32-bit offsets into the z-fastest copy, 24-bit offsets into its columns,
    // one workgroup row per view in the list kernel
    if (g.parallel || (size_t)g.nt * g.ns * (g.nz + 2) > ((size_t)1 << 30) || g.nz > (1 << 20)) return false;
    if (!column_use(g, row_pitch)) return false;
    L.stride = (g.nt + g.ns + 1 + 2 * kColBlock - 1) / (2 * kColBlock) * (2 * kColBlock) + kColBlock;
    if (L.stride > 4096) return false;   // the list kernel's LDS
    const size_t per_view = (size_t)g.np * (L.stride / kColBlock * sizeof(ColumnBlock) + sizeof(ColumnHead));
    const size_t views = std::max<size_t>(1, kColListBytes / per_view / kColTileV) * kColTileV;
    L.views = (int)std::min<size_t>({views, (size_t)g.nb, 65535});
    L.list_bytes = (size_t)L.views * per_view + 256;
    L.vol_bytes = (size_t)g.nt * g.ns * (g.nz + 2) * sizeof(float);
    return true;
}

void column_bind(RayParams &g, const ColumnPlan &L, float *volz, void *lists)
{
    g.volZ = volz;
    g.cols.blocks = (ColumnBlock *)lists;   // 64-byte aligned, before the heads
    g.cols.head = (ColumnHead *)(g.cols.blocks + (size_t)L.views * g.np * (L.stride / kColBlock));
    g.cols.stride = L.stride;
    g.cols.views = L.views;
}

int ray_fp_blocks(const RayParams &g)
{
    if (g.flat) return (int)flat_blocks(g);
    const dim3 grid = fp_grid(g);
    return (int)(grid.x * grid.y * grid.z);
}

hipError_t launch_sysmat_count(const RayParams &g, long long *counts, hipStream_t st)
{
    hipLaunchKernelGGL(k_sysmat_count, dim3((g.np + kBX - 1) / kBX, (g.nx + kBY - 1) / kBY, g.nb), dim3(kBX, kBY), 0,
                       st, counts, g);
    return hipGetLastError();
}

hipError_t launch_sysmat_fill(const RayParams &g, const long long *row_ptr, int *col, float *val, hipStream_t st)
{
    hipLaunchKernelGGL(k_sysmat_fill, dim3((g.np + kBX - 1) / kBX, (g.nx + kBY - 1) / kBY, g.nb), dim3(kBX, kBY), 0,
                       st, row_ptr, col, val, g);
    return hipGetLastError();
}

// Where splitting the rays of a 2-D projection is faster (k_ray_fp_flat_split).
bool flat_split(const RayParams &g) { return (long)((g.np + 63) / 64) * g.nb < 6144; }

hipError_t launch_ray_fp(const RayParams &g, const float *vol, float *proj, hipStream_t st)
{
    if (g.volZ) return launch_columns(g, proj, st);
    if (g.flat && flat_split(g)) {
        hipLaunchKernelGGL(k_ray_fp_flat_split, dim3((g.np + 63) / 64 * g.nb), dim3(64, kFlatWaves), 0, st, proj, g);
        return hipGetLastError();
    }
    if (g.flat) {
        hipLaunchKernelGGL(k_ray_fp_flat, dim3(flat_blocks(g)), dim3(64, kFlatWaves), 0, st, proj, g);
        return hipGetLastError();
    }
    if (g.skip_empty) hipLaunchKernelGGL((k_ray_fp<true>), fp_grid(g), dim3(kBX, kBY), 0, st, vol, proj, g);
    else hipLaunchKernelGGL((k_ray_fp<false>), fp_grid(g), dim3(kBX, kBY), 0, st, vol, proj, g);
    return hipGetLastError();
}

hipError_t launch_ray_fp_residual(const RayParams &g, const float *vol, const float *b, float *r, double *partials,
                                  int *nblocks, hipStream_t st)
{
    if (g.flat) {
        *nblocks = (int)flat_blocks(g);
        hipLaunchKernelGGL(k_ray_fp_residual_flat, dim3(flat_blocks(g)), dim3(64, kFlatWaves), 0, st, b, r, partials, g);
        return hipGetLastError();
    }
    const dim3 grid = fp_grid(g);
    *nblocks = (int)(grid.x * grid.y * grid.z);
    if (g.skip_empty)
        hipLaunchKernelGGL((k_ray_fp_residual<true>), grid, dim3(kBX, kBY), 0, st, vol, b, r, partials, g);
    else
        hipLaunchKernelGGL((k_ray_fp_residual<false>), grid, dim3(kBX, kBY), 0, st, vol, b, r, partials, g);
    return hipGetLastError();
}

int fp_job_blocks(const RayParams &g, int *gx, int *gy)
{
    const dim3 grid = fp_grid(g);
    *gx = (int)grid.x;
    *gy = (int)grid.y;
    return (int)(grid.x * grid.y * grid.z);
}

hipError_t launch_ray_fp_residual_batched(const FpJob *jobs, int njobs, int max_blocks, hipStream_t st)
{
    hipLaunchKernelGGL(k_ray_fp_residual_batched, dim3((unsigned)max_blocks, (unsigned)njobs), dim3(kBX, kBY), 0, st,
                       jobs, njobs);
    return hipGetLastError();
}

}  // namespace ctr
